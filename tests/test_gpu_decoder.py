"""GPU parity of the decoder (Session / Model / Batch) against the oracle.

Bit-exact throughout: caches, hidden states, logits and greedy token ids.
The full decode workload (20 layers, 256 cached positions, 64 greedy tokens)
is checked against the oracle at full size; the batch workload is checked
against single-sequence GPU sessions (bit-exact) and a subset against the
oracle.
"""
import numpy as np
import pytest

import oracle
import rustyneedle_amd as rn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiny(tiny_config, tiny_weights):
    return rn.Model(tiny_config, tiny_weights), oracle.OracleModel(tiny_config, tiny_weights)


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def test_rotary_table_matches_oracle(tiny, tiny_config):
    gm, om = tiny
    cos, sin = gm.rotary_table()
    assert np.array_equal(_bits(cos), _bits(om.rope_cos))
    assert np.array_equal(_bits(sin), _bits(om.rope_sin))


def test_push_hidden_logits_and_cache(tiny, tiny_config):
    gm, om = tiny
    k, v = rn.synthetic_cache(tiny_config, 40, "push")
    gs, os_ = gm.session(64), om.session(64)
    gs.set_cache(k, v)
    os_.set_cache(k, v)
    for tok in (3, 999, 0, 512):
        gs.push(tok)
        os_.push(tok)
        assert np.array_equal(_bits(gs.hidden()), _bits(os_.hidden))
        assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))
    assert len(gs) == os_.length == 44
    gk, gv = gs.get_cache()
    assert np.array_equal(gk.view(np.uint16), os_.keys[:, :, :44])
    assert np.array_equal(gv.view(np.uint16), os_.values[:, :, :44])


def test_push_over_long_cache(tiny, tiny_config):
    """Caches longer than one pass of the fused head kernel's preloaded key
    (512) and value (320) rows, and a position that starts a new class of 32."""
    gm, om = tiny
    k, v = rn.synthetic_cache(tiny_config, 575, "long")
    gs, os_ = gm.session(640), om.session(640)
    gs.set_cache(k, v)
    os_.set_cache(k, v)
    for tok in (5, 999, 17):
        gs.push(tok)
        os_.push(tok)
        assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))


def test_push_from_empty_session(tiny):
    gm, om = tiny
    gs, os_ = gm.session(8), om.session(8)
    for tok in (1, 2):
        gs.push(tok)
        os_.push(tok)
    assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))


def test_greedy_tiny_bit_identical(tiny, tiny_config):
    gm, om = tiny
    k, v = rn.synthetic_cache(tiny_config, 100, "greedy")
    gs, os_ = gm.session(200), om.session(200)
    gs.set_cache(k, v)
    os_.set_cache(k, v)
    ids = gs.decode_greedy(17, 40)
    ref = os_.greedy(17, 40)
    assert ids.tolist() == ref.tolist()
    assert len(gs) == 140
    # the session continues exactly like the oracle's after the greedy run
    assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))


def test_greedy_equals_push_logits_argmax(tiny, tiny_config):
    """The on-device argmax of the captured step equals host argmax of logits."""
    gm, _ = tiny
    k, v = rn.synthetic_cache(tiny_config, 20, "loop")
    a, b = gm.session(64), gm.session(64)
    a.set_cache(k, v)
    b.set_cache(k, v)
    ids = a.decode_greedy(5, 12)
    tok, manual = 5, []
    for _ in range(12):
        b.push(tok)
        tok = oracle.argmax(b.logits())
        manual.append(tok)
    assert ids.tolist() == manual


def test_profile_step_matches_greedy(tiny, tiny_config):
    """The per-kernel profiling path runs the same kernels as the captured step."""
    gm, _ = tiny
    k, v = rn.synthetic_cache(tiny_config, 30, "profile")
    a, b = gm.session(64), gm.session(64)
    a.set_cache(k, v)
    b.set_cache(k, v)
    prof = a.profile_step(7, 6)
    b.decode_greedy(7, 6)
    assert len(a) == len(b) == 36
    assert np.array_equal(_bits(a.logits()), _bits(b.logits()))
    assert prof["qkv_attention"]["per_step"] == tiny_config["layers"]
    # the greedy choice is reduced by the next step's first kernel: no
    # separate argmax kernel in the step
    assert prof["logits"]["per_step"] == 1 and prof["final"]["per_step"] == 0
    assert all(p["us"] > 0 for k, p in prof.items() if k != "final")


def test_feed_prefill_bit_exact_and_equals_pushes(tiny, tiny_config):
    gm, om = tiny
    k, v = rn.synthetic_cache(tiny_config, 30, "feed")
    tokens = rn.synth_tokens(rn.SEED, "feed.tokens", tiny_config["vocab"], 70)
    gs, os_, gp = gm.session(128), om.session(128), gm.session(128)
    for s in (gs, os_, gp):
        s.set_cache(k, v)
    gs.feed(tokens)
    os_.feed(tokens)
    for t in tokens:
        gp.push(int(t))
    assert np.array_equal(_bits(gs.hidden()), _bits(os_.hidden))
    assert np.array_equal(_bits(gs.hidden()), _bits(gp.hidden()))
    assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))
    ck, cv = gs.get_cache()
    pk, pv = gp.get_cache()
    assert np.array_equal(ck.view(np.uint16), pk.view(np.uint16))
    assert np.array_equal(cv.view(np.uint16), pv.view(np.uint16))
    assert np.array_equal(ck.view(np.uint16), os_.keys[:, :, :100])


# 40 tokens: the normed products quantise their rows in their own prologue,
# gate/up on 64-column tiles, with a partial last row tile; 65: the gate/up
# input through the separate norm launch
@pytest.mark.parametrize("count", [1, 3, 4, 40, 65])
def test_feed_small_and_ragged_counts(tiny, count):
    gm, om = tiny
    tokens = (np.arange(count) * 37 + 11) % 1000
    gs, os_ = gm.session(96), om.session(96)
    gs.feed(tokens)
    os_.feed(tokens)
    assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))


@pytest.mark.parametrize("cached,count", [
    (0, 300),      # past the 256 rows one staged chunk holds
    (0, 640),      # whole 16-query tiles on the matrix instructions
    (37, 701),     # a ragged last tile behind a cached prefix
    (1600, 645),   # 2245 positions, on the tiles
    (1690, 660),   # 2350, past them
    (1664, 640),   # the longest context of the tiles, 2304 positions
    (1665, 640),   # the first past it
    (0, 1000),     # 1024 tiles of 64 x 64 in the gated product where it is 4096 rows wide
])
def test_long_feed_bit_exact(tiny_config, cached, count):
    cfg = dict(tiny_config, max_positions=2400, ffn=2048)
    weights = rn.synthetic_weights(cfg, seed=5)
    gs = rn.Model(cfg, weights).session(cached + count)
    os_ = oracle.OracleModel(cfg, weights).session(cached + count)
    if cached:
        k, v = rn.synthetic_cache(cfg, cached, "longfeed")
        gs.set_cache(k, v)
        os_.set_cache(k, v)
    tokens = rn.synth_tokens(rn.SEED, "longfeed.tokens", cfg["vocab"], count)
    oracle.set_threads(8)
    try:
        gs.feed(tokens)
        os_.feed(tokens)
        assert np.array_equal(_bits(gs.hidden()), _bits(os_.hidden))
        assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))
    finally:
        oracle.set_threads(1)
    gk, gv = gs.get_cache()
    assert np.array_equal(gk.view(np.uint16), os_.keys[:, :, :cached + count])
    assert np.array_equal(gv.view(np.uint16), os_.values[:, :, :cached + count])


@pytest.mark.parametrize("cached,count", [
    (1500, 130),   # 264 blocks where 256-row chunks leave one a CU: half chunks
    (1500, 127),   # 256 blocks: whole chunks
    (2848, 129),   # 2977 positions leave one block a CU either way: whole chunks
    (2847, 129),   # two half-chunk blocks still fit
    (6000, 49),    # too long for whole chunks beside four score rows
    (6139, 5),     # the longest context of the four-query blocks
    (6140, 5),     # a block a query past it
])
def test_feed_after_a_long_context(tiny_config, cached, count):
    cfg = dict(tiny_config, layers=1, max_positions=6200)
    weights = rn.synthetic_weights(cfg, seed=6)
    gs = rn.Model(cfg, weights).session(cached + count)
    os_ = oracle.OracleModel(cfg, weights).session(cached + count)
    k, v = rn.synthetic_cache(cfg, cached, "longcontext")
    gs.set_cache(k, v)
    os_.set_cache(k, v)
    tokens = rn.synth_tokens(rn.SEED, "longcontext.tokens", cfg["vocab"], count)
    oracle.set_threads(8)
    try:
        gs.feed(tokens)
        os_.feed(tokens)
        assert np.array_equal(_bits(gs.hidden()), _bits(os_.hidden))
        assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))
    finally:
        oracle.set_threads(1)


@pytest.mark.parametrize("tiny_sums", [False, True])
def test_long_feed_of_extreme_scores_and_values(tiny_config, tiny_sums):
    """640 tokens and more, whose products the f32 matrix instructions form, over
    cached keys that spread the scores far past the exponent's floor and values of
    zeros of both signs, subnormals and tiny magnitudes. With `tiny_sums` every
    position of weight holds zeros and the rest subnormals, so that each product of a
    weight at the floor (2^-126 and a little) and each sum is subnormal; the output
    matrix's scales bring them back beside the residual stream."""
    cached, count = 300, 704
    cfg = dict(tiny_config, layers=2, max_positions=1024)
    weights = rn.synthetic_weights(cfg, seed=8)
    rng = np.random.default_rng(8)
    k, v = rn.synthetic_cache(cfg, cached, "extreme")
    shape = (cfg["layers"], cfg["heads"])
    # pairs of opposite keys far along one dimension: one of them scores high with any query
    for i in range(16):
        far = np.zeros((*shape, 64), np.float16)
        np.put_along_axis(far, rng.integers(0, 64, (*shape, 1)), np.float16(3000.0), -1)
        k[:, :, 2 * i], k[:, :, 2 * i + 1] = far, -far
    if tiny_sums:
        v[:] = (rng.uniform(-6e-5, 6e-5, v.shape)).astype(np.float16)  # subnormal in 16 bits
        v[:, :, :32] = np.where(rng.integers(0, 2, v[:, :, :32].shape), np.float16(0.0), np.float16(-0.0))
        for layer in weights["layers"]:
            layer["qkv"][1][2 * cfg["d_model"]:] *= np.float32(1e-9)  # the fed tokens' own values: zeros and subnormals
            layer["out"][1][:] *= np.float32(1e39 / 2 ** 7)
    else:
        k[:, :, 32::3] *= np.float16(30.0)
        v[:, :, 0::4] = (rng.uniform(-1, 1, v[:, :, 0::4].shape) * 1e-7).astype(np.float16)
        v[:, :, 1::4] = np.where(rng.integers(0, 2, v[:, :, 1::4].shape), np.float16(0.0), np.float16(-0.0))
        v[:, :, 2::4] *= np.float16(6e4 / 8)
    gs = rn.Model(cfg, weights).session(cached + count)
    os_ = oracle.OracleModel(cfg, weights).session(cached + count)
    gs.set_cache(k, v)
    os_.set_cache(k, v)
    tokens = rn.synth_tokens(rn.SEED, "extreme.tokens", cfg["vocab"], count)
    oracle.set_threads(8)
    try:
        gs.feed(tokens)
        os_.feed(tokens)
    finally:
        oracle.set_threads(1)
    assert np.all(np.isfinite(os_.hidden))
    assert np.array_equal(_bits(gs.hidden()), _bits(os_.hidden))
    gk, gv = gs.get_cache()
    assert np.array_equal(gk.view(np.uint16), os_.keys[:, :, :cached + count])
    assert np.array_equal(gv.view(np.uint16), os_.values[:, :, :cached + count])


def test_clone_is_independent(tiny, tiny_config):
    gm, _ = tiny
    k, v = rn.synthetic_cache(tiny_config, 10, "clone")
    base = gm.session(32)
    base.set_cache(k, v)
    base.push(4)
    c = base.clone()
    assert len(c) == 11
    assert np.array_equal(_bits(c.logits()), _bits(base.logits()))
    c.push(9)
    base.push(9)
    assert np.array_equal(_bits(c.logits()), _bits(base.logits()))
    c.push(1)
    assert len(c) == 13 and len(base) == 12


def test_capacity_and_argument_errors(tiny):
    gm, _ = tiny
    s = gm.session(4)
    with pytest.raises(rn.RnError) as e:
        s.push(1000)  # outside the vocabulary
    assert e.value.code == rn.RN_ERR_ARGUMENT
    s.feed([1, 2, 3])
    with pytest.raises(rn.RnError) as e:
        s.decode_greedy(1, 2)
    assert e.value.code == rn.RN_ERR_CAPACITY
    s.push(5)
    with pytest.raises(rn.RnError) as e:
        s.push(5)
    assert e.value.code == rn.RN_ERR_CAPACITY
    with pytest.raises(rn.RnError) as e:
        gm.session(4).logits()
    assert e.value.code == rn.RN_ERR_STATE


def test_batch_decode_equals_sessions_and_oracle(tiny, tiny_config):
    gm, om = tiny
    count, steps = 9, 10
    lengths = rn.synth_tokens(rn.SEED, "batch.lengths", 60, count) + 1
    first = rn.synth_tokens(rn.SEED, "batch.first", tiny_config["vocab"], count)
    b = rn.Batch(gm, count, 80)
    caches = []
    for i in range(count):
        k, v = rn.synthetic_cache(tiny_config, int(lengths[i]), f"batch.{i}")
        caches.append((k, v))
        b.set_cache(i, k, v)
    ids = b.decode_greedy(first, steps)
    for i in range(count):
        s = gm.session(80)
        s.set_cache(*caches[i])
        assert ids[i].tolist() == s.decode_greedy(int(first[i]), steps).tolist(), i
        if i < 3:
            o = om.session(80)
            o.set_cache(*caches[i])
            assert ids[i].tolist() == o.greedy(int(first[i]), steps).tolist(), i


@pytest.mark.parametrize("heads_blocks,capacity", [(300, 250), (300, 300)])
def test_batch_decode_with_a_full_chip(tiny, tiny_config, heads_blocks, capacity):
    """More than 256 attention blocks, with caches of one 256-position pass and past it."""
    gm, _ = tiny
    count, steps = -(-heads_blocks // tiny_config["heads"]), 4
    lengths = rn.synth_tokens(rn.SEED, "full.lengths", capacity - steps, count) + 1
    lengths[0] = capacity - steps
    first = rn.synth_tokens(rn.SEED, "full.first", tiny_config["vocab"], count)
    k, v = rn.synthetic_cache(tiny_config, capacity, "full")
    b = rn.Batch(gm, count, capacity)
    for i, n in enumerate(lengths):
        b.set_cache(i, np.ascontiguousarray(k[:, :, :n]), np.ascontiguousarray(v[:, :, :n]))
    ids = b.decode_greedy(first, steps)
    for i in (0, 1, count // 2, count - 1):
        s = gm.session(capacity)
        s.set_cache(np.ascontiguousarray(k[:, :, :lengths[i]]), np.ascontiguousarray(v[:, :, :lengths[i]]))
        assert ids[i].tolist() == s.decode_greedy(int(first[i]), steps).tolist(), i
        assert np.array_equal(_bits(b.logits()[i]), _bits(s.logits())), i


@pytest.mark.parametrize("count,capacity,lengths", [
    (9, 384, [285, 286, 287, 288, 289, 380]),        # under 256 blocks, one pass of keys, two of values
    (9, 390, [287, 289, 382, 383, 384, 386]),        # one pass of the larger instance
    (9, 576, [382, 385, 570, 572]),
    (9, 960, [285, 383, 384, 385, 575, 576, 577, 650, 767, 768, 769, 865, 956]),  # and several of the smaller
    (33, 960, [574, 575, 576, 577, 638, 639, 640, 641, 956]),                    # over 256: several of the larger
])
def test_batch_decode_passes(tiny_config, count, capacity, lengths):
    """Lengths around the passes of every attention instance, beside short sequences."""
    cfg = dict(tiny_config, layers=1, max_positions=1024)
    gm = rn.Model(cfg, rn.synthetic_weights(cfg, seed=9))
    steps = 4
    lengths = [1, 31, 200] + lengths
    count = max(count, len(lengths))
    lengths = np.array([lengths[i % len(lengths)] for i in range(count)])
    assert lengths.max() + steps <= capacity
    first = rn.synth_tokens(rn.SEED, "passes.first", cfg["vocab"], count)
    k, v = rn.synthetic_cache(cfg, capacity, "passes")
    b = rn.Batch(gm, count, capacity)
    for i, n in enumerate(lengths):
        b.set_cache(i, np.ascontiguousarray(k[:, :, :n]), np.ascontiguousarray(v[:, :, :n]))
    ids = b.decode_greedy(first, steps)
    for i in range(min(count, 16)):
        s = gm.session(capacity)
        s.set_cache(np.ascontiguousarray(k[:, :, :lengths[i]]), np.ascontiguousarray(v[:, :, :lengths[i]]))
        assert ids[i].tolist() == s.decode_greedy(int(first[i]), steps).tolist(), (i, lengths[i])
        assert np.array_equal(_bits(b.logits()[i]), _bits(s.logits())), (i, lengths[i])


def test_full_decode_workload_bit_identical():
    """The batch-1 decode workload at full size: 20 layers, d 512, vocab 8192,
    fp16 cache pre-filled to 256, 64 greedy tokens — ids equal the oracle's."""
    cfg = dict(rn.NEEDLE_DECODER)
    w = rn.synthetic_weights(cfg)
    gm, om = rn.Model(cfg, w), oracle.OracleModel(cfg, w)
    k, v = rn.synthetic_cache(cfg, 256, "decode")
    first = int(rn.synth_tokens(rn.SEED, "decode.first", cfg["vocab"], 1)[0])
    gs = gm.session(320)
    gs.set_cache(k, v)
    ids = gs.decode_greedy(first, 64)
    oracle.set_threads(8)
    try:
        os_ = om.session(320)
        os_.set_cache(k, v)
        ref = os_.greedy(first, 64)
    finally:
        oracle.set_threads(1)
    assert ids.tolist() == ref.tolist()
    assert np.array_equal(_bits(gs.logits()), _bits(os_.logits()))


def test_synthetic_model_equals_host_weights():
    """rn_model_create_synthetic draws the same tensors as synthetic_weights."""
    cfg = dict(rn.NEEDLE_DECODER)
    cfg.update(layers=2, vocab=512)
    a = rn.Model(cfg, seed=99)
    b = rn.Model(cfg, rn.synthetic_weights(cfg, seed=99))
    sa, sb = a.session(8), b.session(8)
    sa.push(3)
    sb.push(3)
    assert np.array_equal(_bits(sa.logits()), _bits(sb.logits()))
