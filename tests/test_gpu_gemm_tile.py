"""Edges of the prompt-chunk GEMM (gemm_tile_kernel) and of the split-16
activation planes, through the C ABI against the CPU oracle and 64-bit sums.

Rows around the 64- and 128-row tiles, shapes that the rule between them gives
to either, row blocks that do not fill a 128-column tile, K of one quad (one
stage) and of K splits that divide unevenly. Bars as in
test_gpu_gemm.py: Q8 2e-6 of max|y|, f32 1e-5.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _proj(gh, gctx, packed, s16, n, k, x, act):
    import torch

    w = gctx.weight(packed, s16, k, n)
    try:
        xd = torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda()
        y = torch.full((x.shape[0] + 1, n), 7.0, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        gh.check(gh.lib().glacier_hip_int4_gemv(gctx.h, w, xd.data_ptr(), gh.F32, x.shape[0], None,
                                                y.data_ptr(), act, None), "int4_gemv", gctx.h)
        gctx.sync()
        y = y.cpu().numpy()
    finally:
        gh.lib().glacier_hip_int4_weight_destroy(w)
    assert np.all(y[-1] == 7.0)  # the row past the last is untouched
    return y[:-1]


@pytest.mark.parametrize("n,k", [(16, 128), (112, 640), (144, 1408), (272, 256)])
@pytest.mark.parametrize("m", [33, 63, 64, 65, 127, 128, 129, 192, 193, 257])
@pytest.mark.parametrize("act", ["q8", "f32"])
def test_tile_edges_match_oracle(gh, gctx, ora, n, k, m, act):
    packed = gh.synth_int4(n + k, 1, n * k // 2)
    s16 = gh.synth_scales_f16(n + k, 2, n * k // 32)
    s32 = s16.view(np.float16).astype(np.float32)
    x = np.random.default_rng(m + n).standard_normal((m, k)).astype(np.float32)
    got = _proj(gh, gctx, packed, s16, n, k, x, gh.ACT_Q8 if act == "q8" else gh.ACT_F32)
    fn = ora.linear_int4_q8 if act == "q8" else ora.linear_int4_f32
    want = fn(x, packed, s32, n, k, 32)
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    assert err < (2e-6 if act == "q8" else 1e-5), err


@pytest.mark.parametrize("n,k,m", [(16400, 128, 193), (16400, 256, 255), (16400, 256, 257),
                                   (16400, 640, 300), (16400, 384, 383), (4608, 3584, 250)])
@pytest.mark.parametrize("act", ["q8", "f32"])
def test_wide_outputs_match_64_bit_sums(gh, gctx, n, k, m, act):
    """Enough columns for more than one 128-row tile a CU (the last shape with
    a K split too); the same bars against 64-bit sums."""
    import torch

    packed = gh.synth_int4(n + k, 1, n * k // 2)
    s16 = gh.synth_scales_f16(n + k, 2, n * k // 32)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    got = torch.from_numpy(_proj(gh, gctx, packed, s16, n, k, x,
                                 gh.ACT_Q8 if act == "q8" else gh.ACT_F32)).cuda().double()
    xv = x.reshape(m, -1, 32)
    if act == "q8":  # group codes as the quantiser rounds them, half away from zero
        sc = np.abs(xv).max(-1, keepdims=True) / np.float32(127)
        r = xv * (np.float32(1) / sc)
        xv = np.clip(np.sign(r) * np.floor(np.abs(r) + np.float32(0.5)), -127, 127) * sc.astype(np.float64)
    u = torch.from_numpy(np.stack([packed & 15, packed >> 4], -1).reshape(n, k)).cuda()
    w = (u.double() - 7).view(n, -1, 32) * torch.from_numpy(s16.view(np.float16).reshape(n, -1, 1)).cuda().double()
    want = torch.from_numpy(xv.reshape(m, k).astype(np.float64)).cuda() @ w.view(n, k).t().contiguous()
    err = float((got - want).abs().max() / want.abs().max())
    assert err < (2e-6 if act == "q8" else 1e-5), err


@pytest.mark.parametrize("m", [3, 17, 40, 130])
def test_split16_planes_keep_f32_range(gh, gctx, m):
    """Groups of very different magnitude (1e-36 to 1e30, zeros, one large
    element among small ones): every group's contribution to 2^-20 of the sum
    of its absolute products (hi + lo holds 23 bits of every element within
    2^-17 of its group's largest, an absolute 2^-39 of it below that; f32
    sums of 32 add a few 2^-24)."""
    n, k = 32, 256
    rng = np.random.default_rng(m)
    packed = gh.synth_int4(9, 1, n * k // 2)
    s16 = gh.synth_scales_f16(9, 2, n * k // 32)
    u = np.stack([packed & 15, packed >> 4], -1).reshape(n, k).astype(np.float64) - 7
    w = u * np.repeat(s16.view(np.float16).astype(np.float64).reshape(n, k // 32), 32, 1)
    x = rng.standard_normal((m, k)).astype(np.float32)
    for i, mag in enumerate([1e-36, 1e-20, 0.0, 1.0, 1e-4, 65504.0, 1e30, 1e10]):
        live = np.zeros((m, k), np.float32)
        live[:, 32 * i:32 * i + 32] = x[:, 32 * i:32 * i + 32] * np.float32(mag)
        live[:, 32 * i] *= np.float32(1000.0 if mag < 1e20 else 1.0)
        got = _proj(gh, gctx, packed, s16, n, k, live, gh.ACT_F32)
        want = live.astype(np.float64) @ w.T
        bound = np.abs(live).astype(np.float64) @ np.abs(w).T * 2.0 ** -20 + 1e-44
        assert np.all(np.abs(got - want) <= bound), (mag, np.max(np.abs(got - want) / bound))


def test_noalloc_accepts_the_same_calls(gh, gctx):
    """The fixed scratch takes 64 f32 rows of 18944 columns and refuses 64 of
    20224 (4 MiB counted at three bytes an element), as it did with
    three-digit planes."""
    import torch

    L = gh.lib()
    for k, ok in ((18944, True), (20224, False)):
        packed = gh.synth_int4(3, 1, 16 * k // 2)
        s16 = gh.synth_scales_f16(3, 2, 16 * k // 32)
        w = gctx.weight(packed, s16, k, 16)
        x = torch.randn((64, k), device="cuda")
        y = torch.empty((64, 16), device="cuda")
        want = torch.empty_like(y)
        torch.cuda.synchronize()
        rc = L.glacier_hip_int4_gemv_noalloc(gctx.h, w, x.data_ptr(), gh.F32, 64, None,
                                             y.data_ptr(), gh.ACT_F32, None)
        gctx.sync()
        assert (rc == gh.OK) == ok, (k, rc)
        if ok:
            gh.check(L.glacier_hip_int4_gemv(gctx.h, w, x.data_ptr(), gh.F32, 64, None,
                                             want.data_ptr(), gh.ACT_F32, None), "gemv", gctx.h)
            gctx.sync()
            assert float((y - want).abs().max() / want.abs().max()) < 1e-6
        L.glacier_hip_int4_weight_destroy(w)


@pytest.mark.parametrize("m", [3, 17, 40, 130])
def test_split16_infinities_are_the_f32_product(gh, gctx, m):
    """An f32 infinity times a weight is an infinity of their signs (NaN for
    weight 0), infinities of two signs and NaN give NaN, other rows and the
    row's finite columns are untouched by it."""
    n, k = 48, 256
    packed = gh.synth_int4(19, 1, n * k // 2)
    s16 = gh.synth_scales_f16(19, 2, n * k // 32)
    u = np.stack([packed & 15, packed >> 4], -1).reshape(n, k).astype(np.float64) - 7
    w = u * np.repeat(s16.view(np.float16).astype(np.float64).reshape(n, k // 32), 32, 1)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    clean = _proj(gh, gctx, packed, s16, n, k, x, gh.ACT_F32)
    bad = x.copy()
    bad[0, 5] = np.inf
    bad[m // 2, 37] = -np.inf
    bad[m - 1, [70, 71, 200]] = [np.inf, np.inf, -np.inf]
    bad[1, 9] = np.nan
    got = _proj(gh, gctx, packed, s16, n, k, bad, gh.ACT_F32)
    with np.errstate(invalid="ignore"):
        want = (bad.astype(np.float64)[:, None, :] * w[None]).sum(-1)
    rows = {0, 1, m // 2, m - 1}
    for r in range(m):
        if r not in rows:
            assert np.array_equal(got[r], clean[r])
        else:
            assert not np.isfinite(want[r]).any()
            assert np.array_equal(got[r], want[r].astype(np.float32), equal_nan=True), r


@pytest.mark.parametrize("m", [1, 2])
def test_digit_infinities(gh, gctx, m):
    """Up to 2 rows (three-digit planes): one infinity in a group is the f32
    product too; several in a group, or a NaN, make the row NaN."""
    n, k = 48, 256
    packed = gh.synth_int4(23, 1, n * k // 2)
    s16 = gh.synth_scales_f16(23, 2, n * k // 32)
    u = np.stack([packed & 15, packed >> 4], -1).reshape(n, k).astype(np.float64) - 7
    w = u * np.repeat(s16.view(np.float16).astype(np.float64).reshape(n, k // 32), 32, 1)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    clean = _proj(gh, gctx, packed, s16, n, k, x, gh.ACT_F32)
    for at in ({37: np.inf}, {37: -np.inf}, {5: np.inf, 70: np.inf}, {5: np.inf, 200: -np.inf},
               {9: np.nan}, {9: np.nan, 11: np.inf}, {64: np.inf, 95: np.inf}):
        bad = x.copy()
        for i, v in at.items():
            bad[0, i] = v
        got = _proj(gh, gctx, packed, s16, n, k, bad, gh.ACT_F32)
        assert np.array_equal(got[1:], clean[1:])
        groups = [i // 32 for i in at]
        if len(set(groups)) < len(groups):
            assert np.isnan(got[0]).all()
        else:
            with np.errstate(invalid="ignore"):
                want = (bad[0].astype(np.float64) * w).sum(-1)
            assert np.array_equal(got[0], want.astype(np.float32), equal_nan=True), at
