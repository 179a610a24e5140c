"""f32-page decode attention through glacier_hip_paged_attention at the edges
of its work list: 16-position pages, 64- and 256-position items, the line at
max_ctx = 256, one and 64 lanes, group sizes 1 to 8, K / V beyond the fp16
range, unused page slots holding NaN. Against 64-bit sums; bar 1e-6 of the
largest output (f32 scores of |q . k| up to ~60: 2^-19 absolute before the
1 / sqrt(hd) factor)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS, LAYER = 2, 1


def _run(gh, gctx, ctxs, max_ctx, Hq, Hkv, hd, seed, kv_scale=1.0):
    import torch

    g = torch.Generator().manual_seed(seed)
    pages = [-(-c // 16) for c in ctxs]
    width = -(-max_ctx // 16)
    perm = torch.randperm(sum(pages) + 1, generator=g)
    pool = torch.full((sum(pages) + 1, LAYERS, 2, 16, Hkv * hd), float("nan"))
    pool[perm[-1]] = 0.0
    table = torch.full((len(ctxs), width), int(perm[-1]), dtype=torch.int32)
    q = 1.5 * torch.randn((len(ctxs), Hq, hd), generator=g) / kv_scale
    want = np.empty((len(ctxs), Hq, hd))
    at = 0
    for i, c in enumerate(ctxs):
        kv = kv_scale * torch.randn((2, c, Hkv * hd), generator=g)
        for p in range(pages[i]):
            table[i, p] = perm[at + p]
            n = min(16, c - 16 * p)
            pool[perm[at + p], LAYER, :, :n] = kv[:, 16 * p:16 * p + n]
        at += pages[i]
        k64 = kv.double().view(2, c, Hkv, hd)
        for h in range(Hq):
            kh = h // (Hq // Hkv)
            w = torch.softmax((k64[0, :, kh] @ q[i, h].double()) / np.sqrt(hd), -1)
            want[i, h] = (w @ k64[1, :, kh]).numpy()
    qd, pd, td = q.reshape(len(ctxs), -1).cuda(), pool.cuda(), table.cuda()
    cl = torch.tensor(ctxs, dtype=torch.int32, device="cuda")
    out = torch.empty_like(qd)
    torch.cuda.synchronize()
    gh.check(gh.lib().glacier_hip_paged_attention(
        gctx.h, qd.data_ptr(), pd.data_ptr(), gh.F32, td.data_ptr(), width, cl.data_ptr(), len(ctxs),
        LAYER, LAYERS, Hq, Hkv, hd, max_ctx, out.data_ptr(), None), "paged_attention", gctx.h)
    gctx.sync()
    err = np.max(np.abs(out.cpu().numpy().reshape(want.shape) - want)) / np.max(np.abs(want))
    assert err < 1e-6, err


@pytest.mark.parametrize("max_ctx", [256, 257])
@pytest.mark.parametrize("hd", [64, 128])
def test_context_edges(gh, gctx, hd, max_ctx):
    _run(gh, gctx, [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, max_ctx], max_ctx, 14, 2, hd, 3)


@pytest.mark.parametrize("ctxs", [[1], [3000], [5] * 64, list(range(1, 65)), [2000] + [7] * 20])
def test_lane_counts(gh, gctx, ctxs):
    _run(gh, gctx, ctxs, max(ctxs), 8, 2, 64, len(ctxs))


@pytest.mark.parametrize("G", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("hd", [64, 128])
def test_group_sizes(gh, gctx, G, hd):
    _run(gh, gctx, [200, 33, 300], 300, 3 * G, 3, hd, G)


@pytest.mark.parametrize("scale", [1e6, 1e-6])
def test_values_outside_the_fp16_range(gh, gctx, scale):
    _run(gh, gctx, [40, 300], 300, 8, 2, 128, 5, kv_scale=scale)


def _uniform(gh, gctx, q, k, v, hd):
    """One lane, one KV head, two query heads: q [2][hd], k and v [c][hd]."""
    import torch

    c = k.shape[0]
    pages = -(-c // 16)
    pool = torch.zeros((pages, 1, 2, 16, hd))
    for p in range(c):
        pool[p // 16, 0, 0, p % 16] = k[p]
        pool[p // 16, 0, 1, p % 16] = v[p]
    qd, pd = q.reshape(1, -1).cuda(), pool.cuda()
    td = torch.arange(pages, dtype=torch.int32, device="cuda").view(1, -1)
    cl = torch.tensor([c], dtype=torch.int32, device="cuda")
    out = torch.empty_like(qd)
    torch.cuda.synchronize()
    gh.check(gh.lib().glacier_hip_paged_attention(
        gctx.h, qd.data_ptr(), pd.data_ptr(), gh.F32, td.data_ptr(), pages, cl.data_ptr(), 1, 0, 1, 2,
        1, hd, c, out.data_ptr(), None), "paged_attention", gctx.h)
    gctx.sync()
    return out.cpu().view(2, hd)


@pytest.mark.parametrize("size", [1.0, 3e4, 1e15])
@pytest.mark.parametrize("c", [33, 300])
@pytest.mark.parametrize("hd", [64, 128])
def test_equal_scores_of_any_size_weigh_equally(gh, gctx, hd, c, size):
    """Equal K rows: the output is V's mean whatever their score is, also
    where one f32 rounding of q . k is worth many e-folds (bar: f32 sums of c
    equal weights)."""
    import torch

    for seed in range(6):
        g = torch.Generator().manual_seed(seed)
        q = size * torch.randn((2, hd), generator=g)
        k = size * torch.randn((1, hd), generator=g).repeat(c, 1)
        v = 1.0 + torch.rand((c, hd), generator=g)
        want = v.double().mean(0)
        got = _uniform(gh, gctx, q, k, v, hd).double()
        err = float((got - want).abs().max())
        assert err < 2e-6, (seed, err)


@pytest.mark.parametrize("c", [64, 300])
@pytest.mark.parametrize("hd", [64, 128])
def test_pages_of_minus_infinite_scores_weigh_nothing(gh, gctx, hd, c):
    """Whole pages whose scores overflow to -inf beside finite ones."""
    import torch

    g = torch.Generator().manual_seed(c)
    q = torch.randn((2, hd), generator=g).abs() + 1.0
    k = torch.randn((c, hd), generator=g)
    v = torch.randn((c, hd), generator=g)
    dead = torch.zeros(c, dtype=torch.bool)
    dead[16:48] = True
    if c > 128:
        dead[64:128] = True  # a whole work item
    k[dead] = -3e38
    got = _uniform(gh, gctx, q, k, v, hd).double()
    live = ~dead
    for h in range(2):
        sc = (k[live].double() @ q[h].double()) / np.sqrt(hd)
        want = torch.softmax(sc, -1) @ v[live].double()
        err = float((got[h] - want).abs().max() / want.abs().max())
        assert err < 1e-6, (h, err)


@pytest.mark.parametrize("ctx,lanes,Hkv", [(65537, 1, 2), (70000, 1, 2), (70000, 3, 1)])
def test_contexts_past_the_work_list(gh, gctx, ctx, lanes, Hkv):
    """Over 65536 positions of few KV heads (attn_decode_kernel, at most 1024
    records of a row)."""
    _run(gh, gctx, [ctx] + [37] * (lanes - 1), ctx, 2 * Hkv, Hkv, 64, 11)
