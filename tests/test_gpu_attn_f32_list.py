"""f32-page decode attention through glacier_hip_paged_attention at the edges
of its kernels: 16-position pages, the per-head kernel's passes, the work
list's 64- and 256-position items, the lines between them, one and 64 lanes,
group sizes 1 to 8, K / V beyond the fp16 range, unused page slots holding
NaN. Against 64-bit sums; bar 1e-6 of the
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
@pytest.mark.parametrize("c", [33, 300, 600])
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


@pytest.mark.parametrize("c", [64, 300, 600])
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


@pytest.mark.parametrize("hd,max_ctx", [(64, c) for c in (63, 64, 65, 128, 129, 256, 257, 511, 512, 513)] +
                         [(128, c) for c in (31, 32, 33, 64, 65, 128, 129, 255, 256, 257)])
def test_passes_of_the_per_head_kernel(gh, gctx, hd, max_ctx):
    """Contexts around a wave's positions and a pass, at max_ctx around 1, 2,
    4 and 8 passes (heads of 64: 64 positions each, 128: 32) and past them."""
    ctxs = [c for c in (1, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 63, 64, 65, 100, 128, 200, 256, 300)
            if c < max_ctx]
    _run(gh, gctx, ctxs + [max_ctx], max_ctx, 6, 3, hd, max_ctx)


@pytest.mark.parametrize("Hkv", [1, 3, 4, 7])
@pytest.mark.parametrize("lanes", [1, 2, 7, 64])
def test_pairs_over_the_xcds(gh, gctx, lanes, Hkv):
    """Rows x KV heads that do and do not fill eights."""
    _run(gh, gctx, [5 + i % 20 for i in range(lanes)], 24, 2 * Hkv, Hkv, 64, lanes)


@pytest.mark.parametrize("hd,Hq,lanes,max_ctx", [
    (64, 24, 64, 64), (64, 25, 64, 64), (64, 16, 64, 256), (64, 17, 64, 256), (64, 8, 64, 300),
    (64, 9, 64, 300), (128, 24, 64, 64), (128, 16, 64, 128), (128, 17, 64, 128), (128, 8, 64, 256),
    (128, 9, 64, 256)])
def test_workgroups_around_the_line(gh, gctx, hd, Hq, lanes, max_ctx):
    """Both sides of the workgroup count past which the work list runs."""
    _run(gh, gctx, [1 + (37 * i) % max_ctx for i in range(lanes)], max_ctx, Hq, Hq, hd, Hq)
