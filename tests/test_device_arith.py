"""The float-reciprocal division of engine.h (`rcp_u` / `divmod_u`), restated in numpy float32.

The kernels divide lane indices by a wave-uniform divisor (token row m by Tv in the QKV epilogue,
combine row R by NH * Tv and then Tv) as q = trunc(m * rcp(d)) followed by one correction step, with
rcp the hardware's v_rcp_f32 (within 1 ulp of 1 / d). The claim is that this equals integer division
for every m below 2^20. Here the reciprocal is taken as the correctly rounded 1 / d and as its two
neighbours one ulp away, which brackets v_rcp_f32's result, and the quotient and remainder are
compared with numpy's integer division over every m below 2^18 for the divisors the kernels see
(every d up to 256, the pi0.5 and MolmoAct2 token counts and their multiples by the head count) and
a spread of others up to 2^18. A planted mistake (the correction step left out) must fail.

Also the softmax over key segments of the attention that shares a token tile among two waves
(stage_catt of ma2_group.hip), restated for one query row: the fold exp2(fma(s, qscale, -m)) weighs
masked scores by the rounding error of -1e30 qscale, so a wave must leave out a segment in which no
block is its own.
"""
import numpy as np


def _divmod_float(m, d, rd, correct=True):
    q = (m.astype(np.float32) * np.float32(rd)).astype(np.int64)  # float32 product, truncated
    if correct:
        r = m - q * d
        q = np.where(r < 0, q - 1, np.where(r >= d, q + 1, q))
    return q, m - q * d


def _reciprocals(d):
    r0 = np.float32(1.0) / np.float32(d)
    return (np.nextafter(r0, np.float32(0)), r0, np.nextafter(r0, np.float32(np.inf)))


def _divisors():
    tok = [10, 30, 50, 200, 493, 968, 1018]
    ds = set(range(1, 257)) | set(tok) | {8 * t for t in tok} | {16 * t for t in tok}
    ds |= {int(x) for x in np.unique(np.geomspace(257, 1 << 18, 60).astype(np.int64))}
    return sorted(ds)


def test_divmod_u_matches_integer_division():
    m = np.arange(1 << 18, dtype=np.int64)
    for d in _divisors():
        for rd in _reciprocals(d):
            q, r = _divmod_float(m, d, rd)
            bad = np.flatnonzero((q != m // d) | (r != m % d))
            assert bad.size == 0, (d, float(rd), int(m[bad[0]]))


def test_divmod_u_needs_its_correction_step():
    m = np.arange(1 << 18, dtype=np.int64)
    wrong = 0
    for d in (3, 7, 10, 50, 968):
        for rd in _reciprocals(d):
            q, _ = _divmod_float(m, d, rd, correct=False)
            wrong += int((q != m // d).sum())
    assert wrong > 0


MASKED = np.float32(-1e30)


def _softmax_state(segments, qscale, skip=True):
    """(m, l) of one wave and query row after segments of raw scores; None: no block of it is the wave's."""
    m, l = MASKED, np.float32(0)
    for seg in segments:
        if seg is None and skip:
            continue
        x = np.full(64, MASKED) if seg is None else np.asarray(seg, np.float32)
        new = max(m, np.float32(x.max() * qscale))
        with np.errstate(over="ignore", under="ignore"):
            alpha = np.exp2(np.float64(m) - np.float64(new)).astype(np.float32)
            # fma: the product of two float32 is exact in float64
            w = np.exp2((x.astype(np.float64) * np.float64(qscale) - np.float64(new)).astype(np.float32))
            l = np.float32(l * alpha + w.sum(dtype=np.float32))
        m = new
    return m, l


def _qscale(head_dim):  # as the kernels round it: log2(e) times 1 / sqrt(head_dim), both float32
    return np.float32(1.4426950408889634) * np.float32(1.0 / np.sqrt(head_dim))


def test_segment_without_a_block_has_no_weight():
    rng = np.random.default_rng(0)
    for hd in (64, 80, 96, 128, 192, 256):
        q, keys = _qscale(hd), rng.standard_normal(64).astype(np.float32) * 8
        m, l = _softmax_state([None], q)
        assert l == 0 and np.isfinite(m)
        alone, led = _softmax_state([keys], q), _softmax_state([None, keys], q)
        assert alone == led == _softmax_state([keys, None], q), hd
        ref = np.exp2(keys.astype(np.float64) * np.float64(q))
        assert abs(np.float64(alone[1]) * np.exp2(np.float64(alone[0])) / ref.sum() - 1) < 1e-5


def test_segment_without_a_block_needs_its_skip():
    states = [_softmax_state([None], _qscale(hd), skip=False)[1] for hd in (64, 80, 96, 128, 192, 256)]
    assert np.isinf(states).any()
