"""Timed cases of the verification path, through the package's public calls.

Three kinds of single calls -- the dequant-GEMM, the attention of the verified
rows, the acceptance rule -- and two whole calls of a Llama-shaped model: the
prompt and one verify forward.  Shapes are those of the benchmark (the 7B
target: dim 4096, 32 heads, FFN 11008, vocabulary 32000; its draft: dim 2048,
16 heads, FFN 5632) and generic ones around them.  Inputs are drawn on the GPU
from the seed alone; GGUF blocks are packed here from drawn fields, so that
`exact` decodes the same fields in 64 bits without the package.
"""
import collections
import importlib.util
import math
import os
import sys

import numpy as np
import torch

PKG_DIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "universal-loader_amd")
DEV = "cuda"

# bytes per element of the GGUF types
TYPE_ID = {"f16": 1, "q4_0": 2, "q8_0": 8, "q4_k": 12, "q6_k": 14}
TYPE_BYTES = {"f16": 2.0, "q4_0": 18 / 32, "q8_0": 34 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256}

# the benchmark's target and draft; n_layers comes from the case
MODELS = {
    "target": dict(dim=4096, n_heads=32, n_kv_heads=32, ffn=11008, vocab=32000),
    "draft": dict(dim=2048, n_heads=16, n_kv_heads=16, ffn=5632, vocab=32000),
}
RMS_EPS, ROPE_BASE = 1e-5, 10000.0

DeviceSpan = collections.namedtuple("DeviceSpan", "ptr nbytes")


def _package():
    if "universal_loader_amd" in sys.modules:
        return sys.modules["universal_loader_amd"]
    spec = importlib.util.spec_from_file_location("universal_loader_amd", os.path.join(PKG_DIR, "__init__.py"),
                                                  submodule_search_locations=[PKG_DIR])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["universal_loader_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


_ctx = None


def _context():
    """One context (one stream) for the process, as a serving program keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = _package().Context(0)
    return _ctx


def listed():
    return [
        # a draft model's fused Q|K|V at one token: the smallest, most frequent linear of a step
        dict(name="gemm_draft_m1", op="gemm", type="q4_k", N=6144, K=2048, M=1),
        # the 7B down projection over five verified rows
        dict(name="gemm_down_m5", op="gemm", type="q4_0", N=4096, K=11008, M=5),
        # the LM head of a mixed-type file over six verified rows
        dict(name="gemm_head_m6", op="gemm", type="q6_k", N=32000, K=4096, M=6),
        # gate|up of the 7B target over a batch of 8 sequences of 6 rows
        dict(name="gemm_batch_m48", op="gemm", type="q4_k", N=22016, K=4096, M=48),
        # a short prompt of odd length through a square projection
        dict(name="gemm_prompt_m333", op="gemm", type="q8_0", N=4096, K=4096, M=333),
        # a 2048-token prompt through an FFN projection: the largest linear
        dict(name="gemm_prompt_m2048", op="gemm", type="q4_k", N=11008, K=4096, M=2048),
        # a chain of five verified tokens over a 4096-token cache
        dict(name="attn_chain", op="attn", H=32, Hkv=32, D=128, prefix=4096, nq=5, tree=False),
        # a 16-node draft tree, grouped-query heads, ragged prefix
        dict(name="attn_tree_gqa", op="attn", H=32, Hkv=8, D=64, prefix=1777, nq=16, tree=True),
        # a server's batch under the usual sampling options
        dict(name="accept_topk", op="accept", B=16, k=4, V=32000, temperature=0.8, top_k=40, top_p=0.9, greedy=False),
        # the whole distribution over a large vocabulary
        dict(name="accept_full", op="accept", B=16, k=8, V=128256, temperature=0.8, top_k=0, top_p=1.0, greedy=False),
        # a prompt through the first layers and the head of the 7B target
        dict(name="model_prompt", op="model", model="target", n_layers=4, pos=0, rows=1500),
        # six verified tokens behind a 2048-token prompt
        dict(name="model_verify", op="model", model="target", n_layers=4, pos=2048, rows=6),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "attn", "accept", "model"])
    if op == "gemm":
        t = rng.choice(["q4_k", "q4_k", "q4_0", "q6_k", "q8_0", "f16"])
        step = 256 if t in ("q4_k", "q6_k") else 32
        K = step * max(1, _log_int(rng, 512, 11008) // step)
        N = _log_int(rng, 256, 32000)
        if rng.random() < 0.5:  # most widths are multiples of a head
            N = max(64, N // 64 * 64)
        M = _log_int(rng, 1, 2048)
        while 2 * M * N * K > 2 * 2048 * 11008 * 4096:
            M = M // 2 + 1
        return dict(op=op, type=t, N=N, K=K, M=M)
    if op == "attn":
        D = rng.choice([64, 128])
        Hkv = rng.choice([1, 2, 4, 8, 16, 32])
        H = Hkv * rng.choice([g for g in (1, 2, 3, 4, 8) if Hkv * g <= 32])
        return dict(op=op, H=H, Hkv=Hkv, D=D, prefix=_log_int(rng, 16, 8192), nq=rng.randint(1, 16),
                    tree=rng.random() < 0.5)
    if op == "accept":
        mode = rng.choice(["full", "topk", "topk", "greedy"])
        return dict(op=op, B=rng.randint(1, 16), k=rng.randint(1, 8), V=_log_int(rng, 2000, 128256), temperature=0.8,
                    top_k=rng.randint(10, 100) if mode == "topk" else 0,
                    top_p=round(rng.uniform(0.8, 1.0), 2) if mode == "topk" else 1.0, greedy=mode == "greedy")
    if rng.random() < 0.5:
        return dict(op=op, model=rng.choice(["target", "draft"]), n_layers=rng.randint(1, 3), pos=0,
                    rows=_log_int(rng, 17, 1500))
    return dict(op=op, model=rng.choice(["target", "draft"]), n_layers=rng.randint(1, 3),
                pos=_log_int(rng, 64, 2048), rows=rng.randint(1, 16))


# ---- GGUF blocks from drawn fields -------------------------------------------


def _gen(seed, stream):
    return torch.Generator(DEV).manual_seed((seed * 1000003 + stream) & 0x7FFFFFFF)


def _halfs(x):
    """fp16 values as little-endian bytes, one trailing axis of 2."""
    return x.contiguous().view(torch.uint8).reshape(*x.shape, 2)


def _normal_ints(g, shape, std, mid, lo, hi):
    return torch.randn(shape, generator=g, device=DEV).mul_(std).add_(mid).round_().clamp_(lo, hi).to(torch.int16)


def _ints(g, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=g, device=DEV, dtype=torch.int16)


def _weight(kind, N, K, seed, stream, std=0.02, dense=False):
    """N rows of K elements of about N(0, std^2): raw GGUF bytes [N][row bytes]
    on the GPU, or with dense the float64 values those bytes stand for."""
    g = _gen(seed, stream)
    u8 = lambda x: x.to(torch.uint8)  # noqa: E731
    if kind == "f16":
        w = torch.randn((N, K), generator=g, device=DEV).mul_(std).half()
        return w.double() if dense else w.view(torch.uint8).reshape(N, -1)
    scale = lambda shape, mid: (torch.rand(shape, generator=g, device=DEV) * 0.6 + 0.7).mul_(mid).half()  # noqa: E731
    if kind in ("q4_0", "q8_0"):
        nb = K // 32
        q = _normal_ints(g, (N, nb, 32), 2.7, 8, 0, 15) if kind == "q4_0" else _normal_ints(g, (N, nb, 32), 40, 0, -127,
                                                                                           127)
        d = scale((N, nb), std / (2.7 if kind == "q4_0" else 40))
        d = torch.where(torch.rand((N, nb), generator=g, device=DEV) < 0.5, d, -d)
        if dense:
            return (q.double() - (8 if kind == "q4_0" else 0)).mul_(d.double()[..., None]).reshape(N, K)
        body = u8(q[..., :16] | (q[..., 16:] << 4)) if kind == "q4_0" else q.to(torch.int8).view(torch.uint8)
        return torch.cat([_halfs(d), body], dim=2).reshape(N, -1)
    ns = K // 256
    if kind == "q4_k":
        q = _normal_ints(g, (N, ns, 8, 32), 2.7, 7.5, 0, 15)
        sc = _ints(g, (N, ns, 8), 24, 63)
        mn = (sc + _ints(g, (N, ns, 8), -4, 4)).clamp_(0, 63)
        d = scale((N, ns), std / (2.7 * 44))
        dmin = (d.float() * 7.5).half()
        if dense:
            w = q.double().mul_((d.double()[..., None] * sc.double())[..., None])
            return w.sub_((dmin.double()[..., None] * mn.double())[..., None]).reshape(N, K)
        lo = u8(sc[..., :4] | ((sc[..., 4:] >> 4) << 6))
        mid = u8(mn[..., :4] | ((mn[..., 4:] >> 4) << 6))
        hi = u8((sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4))
        qs = u8(q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(N, ns, 128)
        return torch.cat([_halfs(d), _halfs(dmin), lo, mid, hi, qs], dim=2).reshape(N, -1)
    # q6_k: elements [half][quarter][32] of a super-block, one int8 scale per 16
    q = _normal_ints(g, (N, ns, 2, 4, 32), 10.8, 32, 0, 63)
    sc = _ints(g, (N, ns, 16), 40, 127)
    sc = torch.where(torch.rand((N, ns, 16), generator=g, device=DEV) < 0.5, sc, -sc)
    d = scale((N, ns), std / (10.8 * 84))
    if dense:
        w = (q.double() - 32).reshape(N, ns, 16, 16)
        return w.mul_((d.double()[..., None] * sc.double())[..., None]).reshape(N, K)
    ql = u8((q[:, :, :, :2] & 15) | ((q[:, :, :, 2:] & 15) << 4)).reshape(N, ns, 128)
    h = q >> 4
    qh = u8(h[:, :, :, 0] | (h[:, :, :, 1] << 2) | (h[:, :, :, 2] << 4) | (h[:, :, :, 3] << 6)).reshape(N, ns, 64)
    return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _halfs(d)], dim=2).reshape(N, -1)


# ---- inputs -------------------------------------------------------------------


def _gemm_x(case, seed):
    return torch.randn((case["M"], case["K"]), generator=_gen(seed, 900), device=DEV).half()


def _attn_in(case, seed):
    g = _gen(seed, 901)
    L = case["prefix"] + case["nq"]
    make = lambda *s: torch.randn(s, generator=g, device=DEV).half()  # noqa: E731
    q, k, v = make(case["nq"], case["H"], case["D"]), make(L, case["Hkv"], case["D"]), make(L, case["Hkv"], case["D"])
    parent = None
    if case["tree"]:
        r = np.random.default_rng(seed)
        parent = np.array([-1] + [r.integers(max(-1, i - 4), i) for i in range(1, case["nq"])], np.int32)
    return q, k, v, parent


def _model_tensors(case, seed, dense=False):
    """(name, kind, value, ne0, ne1): Q4_K matrices and embedding, fp32 norms."""
    c = MODELS[case["model"]]
    dim, ffn, D = c["dim"], c["ffn"], c["dim"] // c["n_heads"]
    mats = [("token_embd", dim, c["vocab"]), ("output", dim, c["vocab"])]
    for l in range(case["n_layers"]):
        mats += [(f"blk.{l}.attn_q", dim, dim), (f"blk.{l}.attn_k", dim, c["n_kv_heads"] * D),
                 (f"blk.{l}.attn_v", dim, c["n_kv_heads"] * D), (f"blk.{l}.attn_output", dim, dim),
                 (f"blk.{l}.ffn_gate", dim, ffn), (f"blk.{l}.ffn_up", dim, ffn), (f"blk.{l}.ffn_down", ffn, dim)]
    for i, (name, ne0, ne1) in enumerate(mats):
        yield name + ".weight", "q4_k", _weight("q4_k", ne1, ne0, seed, i, dense=dense), ne0, ne1
    norms = ["output_norm"] + [f"blk.{l}.{n}_norm" for l in range(case["n_layers"]) for n in ("attn", "ffn")]
    for i, name in enumerate(norms):
        w = 1 + 0.1 * torch.randn(dim, generator=_gen(seed, 500 + i), device=DEV)
        yield name + ".weight", "f32", w, dim, 1


def _model_tokens(case, seed):
    n = case["pos"] + case["rows"]
    return np.random.default_rng(seed).integers(0, MODELS[case["model"]]["vocab"], n).astype(np.int32)


class _ModelState:
    """A loaded model on a context of its own, with its cache filled up to pos."""

    def __init__(self, case, seed):
        pkg = _package()
        self.ctx = pkg.Context(0)
        self.model = pkg.Model(self.ctx, n_layers=case["n_layers"], max_ctx=2112, rms_eps=RMS_EPS, rope_base=ROPE_BASE,
                               **MODELS[case["model"]])
        for name, kind, w, ne0, ne1 in _model_tensors(case, seed):
            torch.cuda.synchronize()
            span = DeviceSpan(w.data_ptr(), w.numel() * w.element_size())
            self.model.set_tensor(name, 0 if kind == "f32" else TYPE_ID[kind], span, ne0, ne1)
        tokens = _model_tokens(case, seed)
        self.pos, self.tokens = case["pos"], tokens[case["pos"]:]
        if self.pos:
            self.model.forward(tokens[:self.pos], 0)

    def __del__(self):
        self.model.close()
        self.ctx.close()


def prepare(case, seed):
    if case["op"] == "model":
        return dict(op="model", m=_ModelState(case, seed))
    pkg, ctx = _package(), _context()
    if case["op"] == "gemm":
        raw = _weight(case["type"], case["N"], case["K"], seed, 0).cpu().numpy()
        wid = ctx.weight_upload(TYPE_ID[case["type"]], raw, case["N"], case["K"])
        st = dict(op="gemm", wid=wid, M=case["M"], x=_gemm_x(case, seed),
                  y=torch.empty((case["M"], case["N"]), device=DEV))
    elif case["op"] == "attn":
        q, k, v, parent = _attn_in(case, seed)
        st = dict(op="attn", q=q, k=k, v=v, parent=parent, case=case,
                  out=torch.empty((case["nq"], case["H"], case["D"]), device=DEV))
    else:
        g = _gen(seed, 902)
        B, k, V = case["B"], case["k"], case["V"]
        target = torch.randn((B, k + 1, V), generator=g, device=DEV).mul_(3)
        draft = target[:, :k] + torch.randn((B, k, V), generator=g, device=DEV)
        if case["greedy"]:
            drawn = draft.argmax(2)
        else:  # a draw from softmax(draft / temperature)
            e = torch.empty((B, k, V), device=DEV).exponential_(generator=g)
            drawn = (draft / case["temperature"] - e.log_()).argmax(2)
        st = dict(op="accept", B=B, k=k, V=V, target=target, draft=draft.contiguous(), drawn=drawn.int(),
                  u=torch.rand((B, k + 1), generator=g, device=DEV),
                  s=pkg.sampling(case["temperature"], case["top_k"], case["top_p"], case["greedy"]),
                  tokens=torch.empty((B, k + 1), dtype=torch.int32, device=DEV),
                  accepted=torch.empty(B, dtype=torch.int32, device=DEV))
    torch.cuda.synchronize()  # the context works on a stream of its own
    return st


def run(st):
    if st["op"] == "model":
        m = st["m"]
        return m.model.forward(m.tokens, m.pos, n_logits=min(16, len(m.tokens)))
    ctx = _context()
    if st["op"] == "gemm":
        ctx.verify_gemm(st["wid"], st["x"].data_ptr(), st["M"], st["y"].data_ptr())
        return st["y"]
    if st["op"] == "attn":
        c = st["case"]
        ctx.verify_attention(st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), c["prefix"], c["nq"],
                             st["parent"], c["H"], c["Hkv"], c["D"], c["D"] ** -0.5, st["out"].data_ptr())
        return st["out"]
    ctx.accept(st["s"], st["B"], st["k"], st["V"], st["target"].data_ptr(), st["draft"].data_ptr(),
               st["drawn"].data_ptr(), st["u"].data_ptr(), st["tokens"].data_ptr(), st["accepted"].data_ptr())
    return st["tokens"], st["accepted"]


def work(case):
    if case["op"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=TYPE_BYTES[case["type"]] * N * K + 2 * M * K + 4 * M * N, flops=2 * M * N * K)
    if case["op"] == "attn":
        L, H, D, nq = case["prefix"] + case["nq"], case["H"], case["D"], case["nq"]
        return dict(bytes=4 * L * case["Hkv"] * D + 6 * nq * H * D, flops=4 * nq * L * H * D)
    if case["op"] == "accept":
        n = case["B"] * (2 * case["k"] + 1) * case["V"]
        return dict(bytes=4 * n, flops=2 * n)
    c, T, pos = MODELS[case["model"]], case["rows"], case["pos"]
    dim, kv = c["dim"], c["n_kv_heads"] * (c["dim"] // c["n_heads"])
    per_layer = dim * (2 * dim + 2 * kv) + 3 * dim * c["ffn"]
    n_out = min(16, T)
    seen = T * pos + T * (T + 1) // 2  # (query, key) pairs
    layers = case["n_layers"]
    return dict(bytes=144 / 256 * (layers * per_layer + c["vocab"] * dim) + layers * 4 * (pos + T) * kv +
                T * dim * 144 / 256 + 4 * n_out * c["vocab"],
                flops=layers * (2 * T * per_layer + 4 * seen * dim) + 2 * n_out * c["vocab"] * dim)


def tolerance(case):
    if case["op"] == "gemm":
        # exact products summed in fp32 (up to 3.4e-7 from 64 bits measured); a Q6_K weight is rounded to fp16
        # where its integer part passes 2048 (1.1e-4)
        return {"rel": 4.5e-4} if case["type"] == "q6_k" else {"rel": 1.5e-6}
    if case["op"] == "attn":  # 2.8e-7 measured
        return {"rel": 1e-6}
    if case["op"] == "accept":
        return "exact"
    # the cache and the queries are fp16: another order of the fp32 sums moves some by one unit (8.5e-5 between
    # two splits of the same prompt into calls; 1.3e-3 from 64 bits on both)
    return {"rel": 3.5e-4}


# ---- 64-bit results -------------------------------------------------------------


def _attend64(q, k, v, mask, scale):
    """q [nq][H][D], k, v [L][Hkv][D], mask [nq][L] -> [nq][H][D], float64."""
    out = torch.empty_like(q)
    g = q.shape[1] // k.shape[1]
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // g].t().contiguous()).mul_(scale).masked_fill_(~mask, -math.inf)
        out[:, h] = torch.softmax(s, 1) @ v[:, h // g].contiguous()
    return out


def _model64(case, seed):
    c = MODELS[case["model"]]
    H, Hkv, D = c["n_heads"], c["n_kv_heads"], c["dim"] // c["n_heads"]
    W = {name: w for name, _, w, _, _ in _model_tensors(case, seed, dense=True)}
    tokens = torch.from_numpy(_model_tokens(case, seed)).to(DEV).long()
    T = len(tokens)
    mask = torch.ones((T, T), dtype=torch.bool, device=DEV).tril()
    pos = torch.arange(T, device=DEV, dtype=torch.float64)
    ang = pos[:, None] * ROPE_BASE ** (-2 * torch.arange(D // 2, device=DEV, dtype=torch.float64) / D)
    co, si = ang.cos()[:, None], ang.sin()[:, None]

    def norm(h, w):
        return h * torch.rsqrt((h * h).mean(1, keepdim=True) + RMS_EPS) * w.double()

    def rope(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * co - b * si, a * si + b * co], dim=3).reshape(x.shape)

    h = W["token_embd.weight"][tokens]
    for l in range(case["n_layers"]):
        w = lambda n: W[f"blk.{l}.{n}.weight"]  # noqa: E731,B023
        x = norm(h, w("attn_norm"))
        q, k = rope((x @ w("attn_q").t()).view(T, H, D)), rope((x @ w("attn_k").t()).view(T, Hkv, D))
        v = (x @ w("attn_v").t()).view(T, Hkv, D)
        h = h + _attend64(q, k, v, mask, D ** -0.5).reshape(T, H * D) @ w("attn_output").t()
        x = norm(h, w("ffn_norm"))
        gate = x @ w("ffn_gate").t()
        h = h + (torch.nn.functional.silu(gate) * (x @ w("ffn_up").t())) @ w("ffn_down").t()
    n = min(16, case["rows"])
    return (norm(h[-n:], W["output_norm.weight"]) @ W["output.weight"].t()).cpu().numpy()


def exact(case, seed):
    if case["op"] == "gemm":
        w = _weight(case["type"], case["N"], case["K"], seed, 0, dense=True)
        return _gemm_x(case, seed).double() @ w.t()
    if case["op"] == "attn":
        q, k, v, parent = _attn_in(case, seed)
        P, nq = case["prefix"], case["nq"]
        mask = torch.ones((nq, P + nq), dtype=torch.bool)
        mask[:, P:] = torch.eye(nq, dtype=torch.bool) if parent is not None else torch.ones((nq, nq)).tril().bool()
        for i in range(nq if parent is not None else 0):
            a = parent[i]
            while a >= 0:
                mask[i, P + a] = True
                a = parent[a]
        return _attend64(q.double(), k.double(), v.double(), mask.to(DEV), case["D"] ** -0.5)
    if case["op"] == "accept":
        return None  # whole numbers only
    return _model64(case, seed)
