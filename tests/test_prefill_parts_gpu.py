"""Prefill on the bf16 matrix cores: f32 operands as three bf16 parts.

The results against 64 bits (at most 4e-6 of the result's norm: a few f32
roundings of sums of d products and of up to T_k weights), at the edges of the
32-key and 32-row tiles and of the 16-dim steps, and for values the parts do
not hold (infinities, magnitudes near both ends of f32), which a unit computes
again in f32.
"""
import numpy as np
import pytest
import torch

import nne_testlib as T

pytestmark = pytest.mark.gpu


def attend64(q, k, v, causal, offset=0):
    g = q.shape[1] // k.shape[1]
    k, v = (np.repeat(x.astype(np.float64), g, 1) for x in (k, v))
    s = np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k) / np.sqrt(q.shape[3])
    if causal:
        s = np.where(np.arange(s.shape[3]) > np.arange(s.shape[2])[:, None] + offset, -np.inf, s)
    w = np.exp(s - s.max(-1, keepdims=True))
    return np.einsum("bhqk,bhkd->bhqd", w / w.sum(-1, keepdims=True), v)


def run(q, k, v, causal, offset=0):
    nne = T.load_package()
    dev = [torch.from_numpy(x).cuda() for x in (q, k, v)]
    o = nne.attention_forward(*dev, causal, q_offset=offset)
    torch.cuda.synchronize()
    return o.cpu().numpy()


def draw(seed, b, hq, hkv, tq, tk, d):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((b, h, t, d)).astype(np.float32)
            for h, t in ((hq, tq), (hkv, tk), (hkv, tk)))


def check64(o, ref):
    assert np.isfinite(o).all()
    assert np.linalg.norm(o - ref) <= 4e-6 * np.linalg.norm(ref)


# Enough heads for the unsplit launch, then few enough for the key split.
@pytest.mark.parametrize("heads", [(40, 20), (2, 1)])
@pytest.mark.parametrize("d", [4, 20, 32, 36, 64, 68, 100, 128])
@pytest.mark.parametrize("tq,tk,causal", [(97, 289, False), (289, 289, True), (320, 1, False),
                                          (33, 320, True), (300, 31, False)])
def test_tile_edges(heads, d, tq, tk, causal):
    q, k, v = draw(d + tq, 2, heads[0], heads[1], tq, tk, d)
    check64(run(q, k, v, causal, tk - tq), attend64(q, k, v, causal, tk - tq))


# More 32-row units than two per CU: the 8-wave kernel (at 512 dims with K and V
# in one buffer); rows that are not whole units, tails of one key, padded dims.
@pytest.mark.parametrize("d", [132, 192, 196, 256, 260, 384, 388, 512])
@pytest.mark.parametrize("hq,hkv,tq,tk,causal", [(140, 140, 97, 129, True), (140, 20, 97, 31, False),
                                                 (75, 75, 225, 225, True)])
def test_tile_edges_above_128_dims(d, hq, hkv, tq, tk, causal):
    q, k, v = draw(d + tq, 1, hq, hkv, tq, tk, d)
    check64(run(q, k, v, causal, tk - tq), attend64(q, k, v, causal, tk - tq))


# More workgroups than CUs, causal: items longest first over all heads (the heads no
# multiple of 8, the items none either), and pairs with a last round barely filled.
@pytest.mark.parametrize("d,hq,hkv,t", [(132, 301, 301, 140), (256, 270, 135, 130), (260, 300, 300, 65),
                                        (388, 61, 61, 290), (512, 66, 11, 225), (320, 42, 42, 449)])
def test_causal_items_longest_first(d, hq, hkv, t):
    q, k, v = draw(d + t, 1, hq, hkv, t, t, d)
    check64(run(q, k, v, True), attend64(q, k, v, True))


@pytest.mark.parametrize("d", [256, 512])
@pytest.mark.parametrize("qs,ks,vs", [(1.0, 1.0, 1e-37), (1e-30, 1e30, 1.0), (1e30, 1e-30, 1.0)])
def test_magnitudes_above_128_dims(d, qs, ks, vs):
    q, k, v = draw(17, 1, 140, 140, 97, 129, d)
    q[..., d // 2:] *= np.float32(qs)      # half of the dims: one wave sees them, all must know
    k[..., d // 2:] *= np.float32(ks)
    v *= np.float32(vs)
    ref = attend64(q, k, v, True, 32)
    scale = 1 / np.abs(ref).max()
    check64(run(q, k, v, True, 32).astype(np.float64) * scale, ref * scale)


@pytest.mark.parametrize("d", [256, 512])
def test_infinities_above_128_dims(d):
    q, k, v = draw(18, 1, 140, 140, 97, 129, d)
    q[:, 3] = np.abs(q[:, 3]) + np.float32(0.01)
    k[:, 3, 50] = -np.inf
    v[0, 5, 70, d - 1] = np.inf
    o = run(q, k, v, False)
    k[:, 3, 50] = -1e30
    ref = attend64(q, k, v, False)
    assert np.isposinf(o[0, 5, :, d - 1]).all()
    check64(o[0, 5, :, :d - 1], ref[0, 5, :, :d - 1])
    others = [h for h in range(140) if h != 5]
    check64(o[:, others], ref[:, others])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("qs,ks,vs", [(1.0, 1.0, 1e-37), (1.0, 1.0, 1e34), (1e-30, 1e30, 1.0),
                                      (1e30, 1e-30, 1.0), (1e-36, 1e36, 1e-36)])
def test_magnitudes_near_the_ends_of_f32(d, qs, ks, vs):
    q, k, v = draw(7, 2, 40, 20, 300, 300, d)
    q, k, v = q * np.float32(qs), k * np.float32(ks), v * np.float32(vs)
    ref = attend64(q, k, v, True)
    scale = 1 / np.abs(ref).max()      # norms of 1e34-sized values leave f32
    check64(run(q, k, v, True).astype(np.float64) * scale, ref * scale)


# One batch element takes the key split, four the unsplit launch.
@pytest.mark.parametrize("b", [1, 4])
@pytest.mark.parametrize("d", [64, 128])
def test_keys_of_minus_infinity_have_no_weight(b, d):
    q, k, v = draw(8, b, 40, 20, 300, 300, d)
    q = np.abs(q) + np.float32(0.01)      # q . k = -inf for every row
    k[:, 3, 250] = -np.inf
    k[:, 7, 5] = -np.inf
    check64(run(q, k, v, False), attend64(q, np.maximum(k, np.float32(-1e30)), v, False))


@pytest.mark.parametrize("b", [1, 4])
@pytest.mark.parametrize("d", [64, 128])
def test_nan_and_infinity_reach_the_rows_that_see_them(b, d):
    q, k, v = draw(9, b, 40, 20, 300, 300, d)
    ref = attend64(q, k, v, True)
    v[0, 2, 200, 3] = np.inf
    k[0, 4, 100, 0] = np.nan
    o = run(q, k, v, True)
    assert np.isposinf(o[0, 4:6, 200:, 3]).all()
    assert np.isnan(o[0, 8:10, 100:]).all()
    # Rows of earlier key tiles, and every other head, are as without them.
    check64(o[0, 4:6, :192], ref[0, 4:6, :192])
    check64(o[0, 8:10, :96], ref[0, 8:10, :96])
    others = [h for h in range(40) if h not in (4, 5, 8, 9)]
    check64(o[:, others], ref[:, others])


@pytest.mark.parametrize("b", [1, 4])
@pytest.mark.parametrize("d", [20, 32, 61, 128])
def test_recomputed_units_through_strided_dims(b, d):
    """Views whose dims are a row apart, where the f32 recompute loads one float at
    a time: keys of minus infinity, and a V at the top of f32's range."""
    q, k, v = draw(d, b, 40, 20, 97, 300, d)
    q = np.abs(q) + np.float32(0.01)
    k[:, 3, 250] = -np.inf
    v[:, 7] *= np.float32(1e37)
    nne = T.load_package()
    dev = [torch.from_numpy(np.ascontiguousarray(x.swapaxes(2, 3))).cuda().transpose(2, 3) for x in (q, k, v)]
    o = nne.attention_forward(*dev, True, q_offset=203)
    torch.cuda.synchronize()
    o = o.cpu().numpy().astype(np.float64)
    ref = attend64(q, np.maximum(k, np.float32(-1e30)), v, True, 203)
    for x in (o, ref):
        x[:, 14:16] *= 1e-37
    check64(o, ref)


# The last stride of the vector loads' 32-bit offsets, and the first of the scalar
# loads; few units (up to 128 dims the key split), and more than CUs.
@pytest.mark.parametrize("d,heads,st", [(64, 2, 1 << 24), (64, 2, (1 << 25) - 4), (64, 2, 1 << 25),
                                        (192, 300, (1 << 25) - 4), (192, 300, 1 << 25),
                                        (512, 300, (1 << 25) - 4)])
def test_row_strides_beyond_the_vector_loads(d, heads, st):
    """K/V rows 2^25 floats apart take the scalar-load variant."""
    tk = 40
    q, k, v = draw(10, 1, heads, 1, 64, tk, d)
    big = torch.empty(tk * st, device="cuda")
    kd, vd = (torch.as_strided(big, (1, 1, tk, d), (tk * st, tk * st, st, 1), off) for off in (0, 512))
    kd.copy_(torch.from_numpy(k))
    vd.copy_(torch.from_numpy(v))
    nne = T.load_package()
    o = nne.attention_forward(torch.from_numpy(q).cuda(), kd, vd, False)
    torch.cuda.synchronize()
    check64(o.cpu().numpy(), attend64(q, k, v, False))


@pytest.mark.parametrize("b", [1, 4])       # the key split and the unsplit launch
@pytest.mark.parametrize("d", [20, 64, 128, 192, 256, 512])
@pytest.mark.parametrize("bits", [112, 124])
def test_tiny_weights_keep_their_bits(b, d, bits):
    """Key 0 takes nearly all of the weight with a V of zeros; every other key's
    weight is about 2^-bits on V of 2^60.  The scores share their roundings, each
    at most 2^-24 of `bits`: of the scale, its log2 form, the query times it, two
    in the sum and the difference from the maximum; times ln 2 that is the error."""
    t = 300 if d <= 128 else 97
    h = 40 if d <= 128 else 140 // b
    q, k, v = draw(d + bits, b, h, h, t, t, d)
    q[..., 1:] *= np.float32(0.05)
    k[..., 1:] *= np.float32(0.05)
    q[..., 0] = 1
    k[..., 0] = -bits * np.log(2) * np.sqrt(d)
    k[..., 0, 0] = 0
    v *= np.float32(2.0**60)
    v[..., 0, :] = 0
    ref = attend64(q, k, v, False)
    o = run(q, k, v, False)
    assert np.linalg.norm(o - ref) <= 6 * bits * 2.0**-24 * np.log(2) * np.linalg.norm(ref)


@pytest.mark.parametrize("b", [1, 4])
@pytest.mark.parametrize("d", [20, 64, 128, 192, 256, 512])
@pytest.mark.parametrize("vs", [1e-35, 1e-39, 1e-42])
def test_values_below_the_normal_range(b, d, vs):
    """V and O down to the smallest subnormals, 2^-149 apart: one rounding there
    and a few of 2^-24 of the value."""
    t = 300 if d <= 128 else 97
    h = 40 if d <= 128 else 140 // b
    q, k, v = draw(d, b, h, h, t, t, d)
    v *= np.float32(vs)
    ref = attend64(q, k, v, True)
    assert (np.abs(run(q, k, v, True) - ref) <= 2.0**-149 + 1e-5 * vs).all()


@pytest.mark.parametrize("d", [32, 64, 128, 256, 512])
def test_large_scores_keep_their_differences(d):
    """Every score has 200 in common, spread over the dims.  In log2 units the
    scores lie between 2^8 and 2^9, where one f32 rounding leaves 2^-15 / sqrt(12)
    (root mean square) of a score and ln 2 times that, 6e-6, of a weight; the D/16
    sums at growing sizes come to little more, 48 at full size to four times it."""
    t, h = (300, 80) if d <= 128 else (97, 140)
    q, k, v = draw(d, 1, h, h, t, t, d)
    u = np.sign(np.random.default_rng(5).standard_normal(d)) * np.sqrt(200 / np.sqrt(d))
    q, k = q + u.astype(np.float32), k + u.astype(np.float32)
    ref = attend64(q, k, v, False)
    assert np.linalg.norm(run(q, k, v, False) - ref) <= 8e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("d", [64, 128, 256, 512])
def test_results_far_below_one_on_ordinary_values(d):
    """Peaked scores over a V of ones and zeros: the results are the weights, down
    to f32's smallest, each within 16 roundings of a score below 128 (2^-18 each,
    times ln 2)."""
    t, h = (300, 80) if d <= 128 else (97, 140)
    q, k, _ = draw(d, 1, h, h, t, t, d)
    q, k = q * np.float32(4), k * np.float32(4)
    v = np.broadcast_to(np.eye(t, d, dtype=np.float32), (1, h, t, d)).copy()
    ref = attend64(q, k, v, False)
    seen = ref > 2.0**-124
    assert (np.abs(run(q, k, v, False) - ref)[seen] <= 16 * 2.0**-18 * np.log(2) * ref[seen]).all()


@pytest.mark.parametrize("d,heads,tq", [(64, 2, 4), (128, 8, 16), (192, 2, 3), (256, 4, 16),      # split-K
                                        (64, 4, 40), (128, 20, 300), (192, 4, 70), (512, 4, 40)])
@pytest.mark.parametrize("step", [0, 4])
def test_rows_that_overlap(d, heads, tq, step):
    """K/V views whose rows are one row broadcast (row stride 0) or a window that
    moves by 4 floats."""
    tk = 90
    rng = np.random.default_rng(d + step)
    kf, vf = (rng.standard_normal(step * tk + d).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((1, heads, tq, d)).astype(np.float32)
    rows = np.arange(tk)[:, None] * step + np.arange(d)
    kd, vd = (torch.as_strided(torch.from_numpy(x).cuda(), (1, 1, tk, d), (0, 0, step, 1)) for x in (kf, vf))
    o = T.load_package().attention_forward(torch.from_numpy(q).cuda(), kd, vd, False)
    torch.cuda.synchronize()
    check64(o.cpu().numpy(), attend64(q, kf[rows][None, None], vf[rows][None, None], False))


# Few rows (split-K, were the rows in order), few units, and more units than CUs;
# the scalar loads of every kernel that takes such rows, over several key tiles.
@pytest.mark.parametrize("d,heads,tq,tk", [(64, 2, 4, 90), (128, 8, 16, 300), (64, 4, 40, 200), (128, 20, 97, 289),
                                           (192, 2, 3, 90), (256, 4, 16, 100), (132, 3, 70, 100),
                                           (192, 300, 40, 109), (256, 130, 97, 129)])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_that_run_backwards(d, heads, tq, tk, causal):
    """Negative K/V row strides through the C ABI (torch has none)."""
    import ctypes
    nne = T.load_package()
    q, k, v = draw(d + tk, 1, heads, heads, tq, tk, d)
    dev = [torch.from_numpy(x).cuda() for x in (q, k[:, :, ::-1].copy(), v[:, :, ::-1].copy())]
    o = torch.full(q.shape, float("nan"), device="cuda")
    i64 = ctypes.c_int64 * 4
    rows = i64(heads * tk * d, tk * d, -d, 1)
    last = (tk - 1) * d * 4          # row 0 of the reversed tensors
    args = []
    for t, first, st in ((dev[0], 0, None), (dev[1], last, rows), (dev[2], last, rows)):
        args += [ctypes.c_void_p(t.data_ptr() + first), i64(*t.shape), st]
    nne.check(nne.lib().nne_attention_forward(*args, ctypes.c_void_p(o.data_ptr()), None, int(causal), tk - tq,
                                              0, 0.0, None))
    torch.cuda.synchronize()
    check64(o.cpu().numpy(), attend64(q, k, v, causal, tk - tq))
