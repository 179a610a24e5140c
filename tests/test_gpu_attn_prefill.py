"""Edges of the prompt-chunk attention kernel (glacier_hip_paged_attention_prefill)
against 64-bit sums: chunks around its 16-row wave tiles and 32-key stages,
every group size from 1 to 8 query heads per KV head (one row tile, or as many
as fill 4 or 8 waves), both head widths, chunks that start mid-page, scattered
pages whose unused slots hold NaN, and one row that dominates its softmax.

Bar: 2e-6 of the largest output. Scores carry f32 accumulation rounding
(|q . k| up to ~60 here: 2^-19 absolute, 3e-7 in the exponent after the
1 / sqrt(hd) factor), outputs the fp16 hi + lo split of the weights (2^-22).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS, LAYER = 3, 1


def _case(gh, gctx, Hq, Hkv, hd, pos0, T, seed):
    import torch

    g = torch.Generator().manual_seed(seed)
    end = pos0 + T
    npages = -(-end // 16)
    perm = torch.randperm(npages + 2, generator=g)
    pool = torch.full((npages + 2, LAYERS, 2, 16, Hkv * hd), float("nan"), dtype=torch.float16)
    kv = torch.randn((2, end, Hkv * hd), generator=g).half()
    for p in range(end):
        pool[perm[p // 16], LAYER, :, p % 16] = kv[:, p]
    q = 1.5 * torch.randn((T, Hq, hd), generator=g)
    q[T // 2] *= 4.0
    table = perm[:npages].to(torch.int32)
    qd, pd, td = q.reshape(T, -1).cuda(), pool.cuda(), table.cuda()
    out = torch.full((T + 1, Hq * hd), 5.0, device="cuda")
    torch.cuda.synchronize()
    gh.check(gh.lib().glacier_hip_paged_attention_prefill(
        gctx.h, qd.data_ptr(), pd.data_ptr(), td.data_ptr(), npages, pos0, T, LAYER, LAYERS, Hq, Hkv,
        hd, out.data_ptr(), None), "attention_prefill", gctx.h)
    gctx.sync()
    got = out.cpu().numpy()
    assert np.all(got[T] == 5.0)
    kvd = kv.double().view(2, end, Hkv, hd)
    want = np.empty((T, Hq, hd))
    mask = torch.arange(end)[None, :] > (pos0 + torch.arange(T))[:, None]
    for h in range(Hq):
        kh = h // (Hq // Hkv)
        sc = (q[:, h].double() @ kvd[0, :, kh].T) / np.sqrt(hd)
        want[:, h] = (torch.softmax(sc.masked_fill(mask, -np.inf), -1) @ kvd[1, :, kh]).numpy()
    err = np.max(np.abs(got[:T].reshape(T, Hq, hd) - want)) / np.max(np.abs(want))
    assert err < 2e-6, err


@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 33, 64, 97])
@pytest.mark.parametrize("pos0", [0, 1, 15, 16, 33, 47])
@pytest.mark.parametrize("hd", [64, 128])
def test_chunk_edges(gh, gctx, T, pos0, hd):
    _case(gh, gctx, 14, 2, hd, pos0, T, 100 * T + pos0)


@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("hd", [64, 128])
def test_group_sizes(gh, gctx, G, hd):
    _case(gh, gctx, 2 * G, 2, hd, 21, 150, G)


def test_more_workgroups_than_a_run(gh, gctx):
    """Over 512 workgroups (three runs of 256 in the block order)."""
    _case(gh, gctx, 40, 8, 64, 5, 1100, 7)


@pytest.mark.parametrize("G,T", [(1, 400), (1, 530), (2, 250), (2, 290), (3, 150), (4, 100), (4, 150)])
@pytest.mark.parametrize("hd", [64, 128])
def test_tiles_per_workgroup(gh, gctx, G, T, hd):
    """32 KV heads: row counts on both sides of the line (256 workgroups of
    fewest tiles) past which a workgroup takes 8 / G tiles."""
    _case(gh, gctx, 32 * G, 32, hd, 21, T, G)


def _launch(gh, gctx, q, kv, pos0, Hq, Hkv, hd):
    """q [T][Hq][hd] f32, kv [2][pos0 + T][Hkv * hd] fp16 in consecutive pages."""
    import torch

    T, end = q.shape[0], kv.shape[1]
    npages = -(-end // 16)
    pool = torch.zeros((npages, LAYERS, 2, 16, Hkv * hd), dtype=torch.float16)
    for p in range(end):
        pool[p // 16, LAYER, :, p % 16] = kv[:, p]
    qd, pd = q.reshape(T, -1).cuda(), pool.cuda()
    td = torch.arange(npages, dtype=torch.int32, device="cuda")
    out = torch.empty_like(qd)
    torch.cuda.synchronize()
    gh.check(gh.lib().glacier_hip_paged_attention_prefill(
        gctx.h, qd.data_ptr(), pd.data_ptr(), td.data_ptr(), npages, pos0, T, LAYER, LAYERS, Hq, Hkv,
        hd, out.data_ptr(), None), "attention_prefill", gctx.h)
    gctx.sync()
    return out.cpu().view(T, Hq, hd)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("G", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("pos0", [0, 5])
@pytest.mark.parametrize("bad", [20, 50, 77])
def test_infinite_v_stays_out_of_earlier_rows(gh, gctx, hd, G, pos0, bad):
    """An infinity in one position's V row reaches no 16-row tile that ends
    before that position, wherever both lie in a workgroup's rows and a
    32-key stage."""
    import torch

    T, Hkv = 130, 2
    Hq = G * Hkv
    g = torch.Generator().manual_seed(G + bad)
    kv = torch.randn((2, pos0 + T, Hkv * hd), generator=g).half()
    q = 1.5 * torch.randn((T, Hq, hd), generator=g)
    want = _launch(gh, gctx, q, kv, pos0, Hq, Hkv, hd)
    kv[1, pos0 + bad] = float("inf")
    got = _launch(gh, gctx, q, kv, pos0, Hq, Hkv, hd)
    before = bad // 16 * 16
    assert torch.equal(got[:before], want[:before])
    assert not torch.isfinite(got[bad:]).any()


@pytest.mark.parametrize("top", [50, 200])
@pytest.mark.parametrize("hd", [64, 128])
def test_growing_maxima_at_large_scores(gh, gctx, hd, top):
    """Scores that rise to `top` over the keys, so every 32-key stage raises
    the maximum of rows whose earlier keys still weigh. Only one dimension is
    nonzero and its products have 22 bits, so every q . k is exact and the
    error left is the softmax's own. Bar 1e-6: weights carry the fp16 hi + lo
    split (2^-22), the exponential (2^-23) and their exponent's rounding, which
    averages under 2^-22 over the keys that count (the nearest few e-folds); a
    rescale that does not match the rounded maxima the weights were taken from
    costs about half an ulp of 1.44 * top (3e-6 to 5e-6 here at 200)."""
    import torch

    T, Hq, Hkv = 300, 4, 2
    g = torch.Generator().manual_seed(top + hd)
    unit = top * hd ** 0.5 / 32.0  # K at which a q of 32 scores `top`
    q = torch.zeros((T, Hq, hd))
    q[:, :, 0] = (30 + 4 * torch.rand((T, Hq), generator=g)).half().float()
    kv = torch.randn((2, T, Hkv, hd), generator=g).half()
    kv[0] = 0
    rise = unit * (1 - 0.08 * (50 / top) * (T - torch.arange(T)) / 32)
    kv[0, :, :, 0] = (rise[:, None] + 0.02 * unit * (50 / top) *
                      torch.randn((T, Hkv), generator=g)).half()
    got = _launch(gh, gctx, q, kv.reshape(2, T, -1), 0, Hq, Hkv, hd).double()
    mask = torch.arange(T)[None, :] > torch.arange(T)[:, None]
    for h in range(Hq):
        K, V = kv[0, :, h // 2].double(), kv[1, :, h // 2].double()
        sc = (q[:, h].double() @ K.T) / np.sqrt(hd)
        want = torch.softmax(sc.masked_fill(mask, -np.inf), -1) @ V
        err = float((got[:, h] - want).abs().max() / want.abs().max())
        assert err < 1e-6, (h, err)
