"""Timed cases of the text token loop: projections, attention and whole requests.

A case is a dict of plain values; its "kind" says which public entry point a
pass calls:

* "proj": one INT4 projection of m activation rows, glacier_hip_int4_gemv;
* "attn": one decode step's paged attention over several lanes,
  glacier_hip_paged_attention;
* "prompt_attn": causal attention of one lane's prompt chunk,
  glacier_hip_paged_attention_prefill;
* "request": whole requests through glacier_hip.Session: every lane is begun
  and prefilled, then all lanes decode together, fed from a fixed token list;
  the logits of the first and the last decode step come back.

Weights are Gaussian rows quantised to group-32 INT4 codes with fp16 scales,
activations Gaussian with a per-channel gain (the spread that RMSNorm'd and
SwiGLU'd activations have). All inputs come from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "glacier-engine_amd"))
import glacier_hip as gh  # noqa: E402

PAGE = 16          # positions of a KV page
KV_LAYERS = 28     # layers a page of the stand-alone attention cases holds
GEOMETRY = {       # query heads, KV heads, head_dim, model width, MLP width
    "7b": dict(heads=28, kv_heads=4, head_dim=128, dim=3584, hidden=18944),
    "05b": dict(heads=14, kv_heads=2, head_dim=64, dim=896, hidden=4864),
}
# The whole requests run a slice of the model's layers with a vocabulary cut
# in about the same proportion, so a step's time divides between layers and
# head as in the full model.
VOCAB = 20480

_state = {}


def _ctx():
    if "ctx" not in _state:
        _state["ctx"] = gh.Context(0)
        _state["stream"] = torch.cuda.Stream()
    return _state["ctx"], _state["stream"].cuda_stream


def listed():
    proj = lambda name, n, k, m, x="f32": dict(name=name, kind="proj", n=n, k=k, m=m, x=x, act="auto")  # noqa: E731
    return [
        # the smallest projection of a batch-1 token: latency and launches
        proj("qkv_05b_1_row", 1152, 896, 1),
        # the widest projection of a batch-1 token, 53% of a 7B token's weights
        proj("gate_up_7b_1_row", 37888, 3584, 1),
        # the vocabulary head of a batch-1 token (f32 activation arithmetic)
        proj("head_7b_1_row", 152064, 3584, 1),
        # a small decode batch, activations handed over in bf16
        proj("wide_8_rows_bf16", 11008, 4096, 8, "bf16"),
        # the down projection of 32 decode lanes (f32 arithmetic: wide input)
        proj("down_7b_32_rows", 3584, 18944, 32),
        # a prompt chunk through one half of gate/up
        proj("up_7b_2048_rows", 18944, 3584, 2048),
        # a prompt of odd length through down (f32 arithmetic)
        proj("down_7b_1999_rows", 3584, 18944, 1999),
        # four decode lanes of very different contexts, fp16 pages
        dict(name="attn_7b_4_lanes", kind="attn", geometry="7b", kv="f16", ctx="512,2048,4096,8192"),
        # ragged lanes of the small model, f32 pages (the reference's storage)
        dict(name="attn_05b_6_lanes_f32", kind="attn", geometry="05b", kv="f32",
             ctx="37,130,517,1030,1999,4096"),
        # the attention of a fresh 2048-token prompt
        dict(name="attn_7b_prompt_2048", kind="prompt_attn", geometry="7b", pos0=0, rows=2048),
        # one user: a 128-token prompt, then batch-1 decode
        dict(name="request_7b", kind="request", geometry="7b", layers=4, lanes=1, prompt=128,
             steps=48, kv="f16"),
        # 32 users: prompts of 20 to 99 tokens, then decode in one batch
        dict(name="lanes_7b_32", kind="request", geometry="7b", layers=2, lanes=32, prompt=60,
             steps=24, kv="f16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj"] * 6 + ["attn"] * 2 + ["prompt_attn"] * 2 + ["request"])
    if kind == "proj":
        while True:
            n, k = 16 * _log(rng, 24, 2400), 128 * _log(rng, 5, 150)
            m = rng.choice([1, 2, rng.randint(3, 16), rng.randint(17, 48), _log(rng, 49, 2048)])
            if m * n * k <= 1.2e11:
                break
        return dict(kind=kind, n=n, k=k, m=m, x=rng.choice(["f32", "f32", "bf16"]),
                    act=rng.choice(["auto", "auto", "f32"]))
    if kind == "attn":
        ctx, room = [], 14000
        for _ in range(rng.choice([1, 2, 3, 5, 8, 16, 31])):
            c = min(_log(rng, 4, 8192), room)
            if c > 0:
                ctx.append(c)
            room -= c
        return dict(kind=kind, geometry=rng.choice(["7b", "05b"]), kv=rng.choice(["f16", "f16", "f32"]),
                    ctx=",".join(str(c) for c in ctx))
    if kind == "prompt_attn":
        rows = _log(rng, 17, 2048)
        return dict(kind=kind, geometry=rng.choice(["7b", "05b"]),
                    pos0=rng.choice([0, rng.randint(1, 2048 - rows) if rows < 2048 else 0]), rows=rows)
    return dict(kind=kind, geometry=rng.choice(["7b", "05b"]), layers=rng.randint(1, 2),
                lanes=rng.choice([1, 1, 2, 3, 5, 9, 17]), prompt=_log(rng, 12, 200),
                steps=rng.randint(8, 24), kv=rng.choice(["f16", "f32"]))


# ---- inputs -------------------------------------------------------------------------
def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + what)
    return g


def _quantised(g, n, k):
    """Packed codes [n, k/2] (u8, even column in the low nibble) and fp16
    scales [n, k/32], on the GPU: Gaussian rows, codes round(w / scale) + 7."""
    packed = torch.empty((n, k // 2), dtype=torch.uint8, device="cuda")
    scales = torch.empty((n, k // 32), dtype=torch.float16, device="cuda")
    step = max(16, (1 << 26) // k)
    for r in range(0, n, step):
        w = torch.randn((min(step, n - r), k // 32, 32), generator=g, device="cuda") / math.sqrt(k)
        s = (w.abs().amax(-1, keepdim=True) / 7).half()
        u = (torch.round(w / s.float()) + 7).clamp_(0, 15).to(torch.uint8).view(-1, k)
        packed[r:r + step] = u[:, 0::2] | (u[:, 1::2] << 4)
        scales[r:r + step] = s.view(-1, k // 32)
    return packed, scales


def _dequantised(packed, scales, dtype=torch.float64):
    u = torch.stack((packed & 15, packed >> 4), -1).view(packed.shape[0], -1)
    w = (u.to(dtype) - 7).view(packed.shape[0], -1, 32) * scales.to(dtype).unsqueeze(-1)
    return w.view(packed.shape[0], -1)


def _rows(g, m, k, x):
    gain = torch.exp(0.7 * torch.randn(k, generator=g, device="cuda"))
    v = torch.randn((m, k), generator=g, device="cuda") * gain
    return v.to(torch.bfloat16) if x == "bf16" else v


def _contexts(case):
    return [int(c) for c in case["ctx"].split(",")]


def _attn_inputs(case, seed):
    """Queries, page pool [pages][layers][K, V][16][kv_heads * hd], scattered
    page table and context lengths of a decode or prompt attention case."""
    geo, g = GEOMETRY[case["geometry"]], _gen(seed, 2)
    prompt = case["kind"] == "prompt_attn"
    ctx = [case["pos0"] + case["rows"]] if prompt else _contexts(case)
    rows = case["rows"] if prompt else len(ctx)
    pages = [-(-c // PAGE) for c in ctx]
    total = sum(pages)
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros((len(ctx), max(pages)), dtype=torch.int32, device="cuda")
    at = 0
    for i, p in enumerate(pages):
        table[i, :p] = perm[at:at + p]
        at += p
    kvd = geo["kv_heads"] * geo["head_dim"]
    dt = torch.float32 if case.get("kv") == "f32" else torch.float16
    pool = torch.empty((total, KV_LAYERS, 2, PAGE, kvd), dtype=dt, device="cuda")
    pool.normal_(generator=g)
    q = 1.5 * torch.randn((rows, geo["heads"] * geo["head_dim"]), generator=g, device="cuda")
    return q, pool, table, torch.tensor(ctx, dtype=torch.int32, device="cuda")


class _Weight:
    """An uploaded INT4 weight, released with its owner."""

    def __init__(self, packed, scales, k, n):
        ctx, _ = _ctx()
        self.h = ctx.weight(packed.cpu().numpy(), scales.cpu().numpy().view(np.uint16), k, n)

    def __del__(self):
        if gh is not None and getattr(self, "h", None):
            gh.lib().glacier_hip_int4_weight_destroy(self.h)


class _Served:
    """A model slice and a session on it."""

    def __init__(self, case, seed):
        ctx, _ = _ctx()
        geo, g = GEOMETRY[case["geometry"]], _gen(seed, 3)
        D, F, hd = geo["dim"], geo["hidden"], geo["head_dim"]
        kvd = geo["kv_heads"] * hd
        cfg = dict(num_layers=case["layers"], dim=D, hidden_dim=F, num_heads=geo["heads"],
                   num_kv_heads=geo["kv_heads"], head_dim=hd, vocab_size=VOCAB, group_size=32,
                   rms_eps=1e-6, rope_theta=1e6)

        def norm():
            return (1 + 0.1 * torch.randn(D, generator=g, device="cuda")).cpu().numpy()

        def weight(n, k):
            packed, scales = _quantised(g, n, k)
            return packed.cpu().numpy(), scales.float().cpu().numpy()

        layers = []
        for _ in range(case["layers"]):
            L = dict(input_norm=norm(), post_attn_norm=norm())
            for name, n, k in (("q", D, D), ("k", kvd, D), ("v", kvd, D), ("o", D, D),
                               ("gate", F, D), ("up", F, D), ("down", D, F)):
                L["w_" + name], L["s_" + name] = weight(n, k)
            layers.append(L)
        head, head_scales = weight(VOCAB, D)
        self.session = self.model = None
        self.model = gh.Model(ctx, cfg)
        self.model.set_from_host(dict(
            layers=layers, final_norm=norm(), lm_head=head, lm_head_scales=head_scales,
            embedding=torch.randn((VOCAB, D), generator=g, device="cuda").cpu().numpy()))
        rng = np.random.default_rng(seed)
        lanes, self.steps = case["lanes"], case["steps"]
        # prompts from a third to five thirds of the nominal length, spread evenly
        span = [case["prompt"]] if lanes == 1 else \
            [max(1, round(case["prompt"] * (1 / 3 + 4 / 3 * i / (lanes - 1)))) for i in range(lanes)]
        self.prompts = [rng.integers(0, VOCAB, n).astype(np.uint32) for n in span]
        self.feed = rng.integers(0, VOCAB, (self.steps, lanes)).astype(np.uint32)
        self.lanes = list(range(lanes))
        self.session = gh.Session(self.model, max_lanes=lanes, max_positions=max(span) + self.steps + 8,
                                  kv_dtype=gh.F32 if case["kv"] == "f32" else gh.F16)

    def run(self):
        s = self.session
        for i in self.lanes:
            s.begin(i, seed=i + 1)
            s.prefill(i, self.prompts[i])
        _, first = s.step(self.lanes, self.feed[0], want_logits=True)
        for t in range(1, self.steps - 1):
            s.step(self.lanes, self.feed[t])
        _, last = s.step(self.lanes, self.feed[self.steps - 1], want_logits=True)
        return first, last

    def __del__(self):
        if getattr(self, "session", None):
            self.session.close()
        if getattr(self, "model", None):
            self.model.close()


# ---- the interface --------------------------------------------------------------------
def prepare(case, seed):
    ctx, stream = _ctx()
    if case["kind"] == "request":
        return _Served(case, seed)
    L = gh.lib()
    if case["kind"] == "proj":
        n, k, m = case["n"], case["k"], case["m"]
        w = _Weight(*_quantised(_gen(seed, 0), n, k), k, n)
        x = _rows(_gen(seed, 1), m, k, case["x"])
        y = torch.empty((m, n), dtype=torch.float32, device="cuda")
        act = {"auto": gh.ACT_AUTO, "f32": gh.ACT_F32}[case["act"]]
        args = (ctx.h, w.h, x.data_ptr(), gh.BF16 if case["x"] == "bf16" else gh.F32, m, None,
                y.data_ptr(), act, stream)
        state = (L.glacier_hip_int4_gemv, args, y, (w, x))
    else:
        geo = GEOMETRY[case["geometry"]]
        q, pool, table, lens = _attn_inputs(case, seed)
        out = torch.empty_like(q)
        shape = (KV_LAYERS - 1, KV_LAYERS, geo["heads"], geo["kv_heads"], geo["head_dim"])
        if case["kind"] == "attn":
            ctxs = _contexts(case)
            args = (ctx.h, q.data_ptr(), pool.data_ptr(), gh.F32 if case["kv"] == "f32" else gh.F16,
                    table.data_ptr(), table.shape[1], lens.data_ptr(), len(ctxs), *shape, max(ctxs),
                    out.data_ptr(), stream)
            fn = L.glacier_hip_paged_attention
        else:
            args = (ctx.h, q.data_ptr(), pool.data_ptr(), table.data_ptr(), table.shape[1],
                    case["pos0"], case["rows"], *shape, out.data_ptr(), stream)
            fn = L.glacier_hip_paged_attention_prefill
        state = (fn, args, out, (q, pool, table, lens))
    torch.cuda.synchronize()
    return state


def run(state):
    if isinstance(state, _Served):
        return state.run()
    fn, args, out, _ = state
    rc = fn(*args)
    if rc:
        gh.check(rc, "perf case", args[0])
    return out


def work(case):
    if case["kind"] == "proj":
        n, k, m = case["n"], case["k"], case["m"]
        return dict(bytes=n * k * 9 // 16 + m * k * (2 if case["x"] == "bf16" else 4) + m * n * 4,
                    flops=2 * m * n * k)
    geo = GEOMETRY[case["geometry"]]
    width, kvd = geo["heads"] * geo["head_dim"], geo["kv_heads"] * geo["head_dim"]
    if case["kind"] == "attn":
        ctx = _contexts(case)
        return dict(bytes=sum(2 * c * kvd * (4 if case["kv"] == "f32" else 2) + -(-c // PAGE) * 4
                              for c in ctx) + 2 * len(ctx) * width * 4,
                    flops=4 * sum(ctx) * width)
    if case["kind"] == "prompt_attn":
        T, end = case["rows"], case["pos0"] + case["rows"]
        return dict(bytes=2 * end * kvd * 2 + 2 * T * width * 4,
                    flops=4 * width * (T * case["pos0"] + T * (T + 1) // 2))
    D, F = geo["dim"], geo["hidden"]
    layer = D * (D + 2 * kvd) + D * D + 3 * F * D
    lanes, steps, prompt = case["lanes"], case["steps"], case["prompt"]
    passes = lanes + steps  # a prompt pass per lane, then the batched steps
    tokens = lanes * (prompt + steps)
    elem = 4 if case["kv"] == "f32" else 2
    kv = case["layers"] * 2 * kvd * elem
    attended = lanes * (prompt + steps * (prompt + steps / 2))
    return dict(bytes=passes * (case["layers"] * layer + VOCAB * D) * 9 // 16 + int(kv * attended),
                flops=2 * tokens * case["layers"] * layer + 2 * lanes * (steps + 1) * VOCAB * D)


def tolerance(case):
    if case["kind"] == "request":
        # 8-bit activation codes sit on rounding edges: another order of an
        # f32 sum moves some by one code in every layer that follows. Measured
        # with attention and O as one launch or two and with the prompt in one
        # chunk or 16-row chunks: 0.0054 at two layers, 0.0096 at four.
        return {"rel": min(0.03, 0.01 * case["layers"]), "max": 0.2}
    # f32 sums of up to 19456 exact products, or a softmax over up to 8192:
    # up to 6e-7 from the 64-bit values
    return {"rel": 2.5e-6, "max": 1e-4}


def _auto_f32(case):
    return case["act"] == "f32" or case["n"] > 65536 or case["k"] > 16384


def exact(case, seed):
    if case["kind"] == "request":
        return None  # no 64-bit value: the 8-bit activation codes round f32 values
    if case["kind"] == "proj":
        n, k, m = case["n"], case["k"], case["m"]
        packed, scales = _quantised(_gen(seed, 0), n, k)
        x = _rows(_gen(seed, 1), m, k, case["x"]).float()
        if not _auto_f32(case):  # group-32 8-bit codes, rounded half away from zero in f32
            v = x.view(m, -1, 32)
            s = v.abs().amax(-1, keepdim=True)
            s = s / torch.full_like(s, 127)  # (by a number torch multiplies with its reciprocal)
            r = v * torch.where(s == 0, torch.zeros_like(s), 1 / s)
            x = (torch.sign(r) * torch.floor(r.abs() + 0.5)).clamp_(-127, 127).double() * s.double()
            x = x.view(m, k)
        x = x.double()
        y = torch.empty((m, n), dtype=torch.float64, device="cuda")
        step = max(16, (1 << 27) // k)
        for r in range(0, n, step):
            y[:, r:r + step] = x @ _dequantised(packed[r:r + step], scales[r:r + step]).t()
        return y
    geo = GEOMETRY[case["geometry"]]
    H, Hkv, hd = geo["heads"], geo["kv_heads"], geo["head_dim"]
    G = H // Hkv
    q, pool, table, lens = _attn_inputs(case, seed)
    q = q.double().view(-1, H, hd)
    out = torch.empty_like(q)
    prompt = case["kind"] == "prompt_attn"
    for lane, c in enumerate(lens.tolist()):
        kv = pool[table[lane, :-(-c // PAGE)].long(), KV_LAYERS - 1].double()
        kv = kv.transpose(0, 1).reshape(2, -1, Hkv, hd)[:, :c]
        rows = slice(None) if prompt else slice(lane, lane + 1)
        for h in range(Hkv):
            K, V = kv[0, :, h], kv[1, :, h]
            for j in range(h * G, (h + 1) * G):
                sc = q[rows, j] @ K.t() / math.sqrt(hd)
                if prompt:
                    at = case["pos0"] + torch.arange(sc.shape[0], device="cuda")
                    sc.masked_fill_(torch.arange(c, device="cuda") > at[:, None], -math.inf)
                out[rows, j] = torch.softmax(sc, -1) @ V
    return out.view(-1, H * hd)
