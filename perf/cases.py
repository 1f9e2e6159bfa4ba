"""Performance cases of the dispatch library, through the entry points a
compiled Vx program calls: the routed `a @ b` (vx_plugin_dispatch_async with a
kind=matmul payload), the flash-attention forward, the int8 GEMV, and the
int8 Llama decoder.

Operands are torch tensors in HBM; the library launches on the null stream,
torch's default stream, so its work and torch's are ordered.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from vx_amd import abi
from vx_amd.decode import LlamaI8
from vx_amd.llama import LlamaConfig, rope_table
from vx_amd.runtime import DispatchLibrary, flash_attention_fwd, gemv_i8

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
DTYPE = {"f32": abi.DTYPE_F32, "bf16": abi.DTYPE_BF16, "f16": abi.DTYPE_F16}
BYTES = {"f32": 4, "bf16": 2, "f16": 2}

_lib: list[DispatchLibrary] = []


def lib() -> DispatchLibrary:
    if not _lib:
        _lib.append(DispatchLibrary())
    return _lib[0]


def listed() -> list[dict]:
    return [
        # The GEMM the framework is quoted on: bf16 4096^3, f32 result.
        gemm("gemm_bf16_4096", "bf16", "f32", 4096, 4096, 4096),
        # A Llama-2-7B up projection of a 512-token prefill chunk, bf16 kept
        # between layers.
        gemm("gemm_bf16_chunk512", "bf16", "bf16", 512, 11008, 4096),
        # The same model's square projection for a decode batch of 8 tokens.
        gemm("gemm_bf16_batch8", "bf16", "f32", 8, 4096, 4096),
        # A shape off every tile and alignment: odd rows, N and K, f16.
        gemm("gemm_f16_ragged", "f16", "f32", 1000, 777, 1111),
        # The f32 matmul a program gets without naming a type, at the largest
        # size the reference publishes a time for.
        gemm("gemm_f32_2048", "f32", "f32", 2048, 2048, 2048),
        # Training-shaped causal attention: the size the framework is quoted on.
        fa("attn_causal_2048", 4, 32, 32, 2048, 2048, 128, True),
        # The reference's attention benchmark: a 512-token prefill chunk over
        # a cache of 1536, 32 query heads on 4 KV heads.
        fa("attn_chunk512_at1536", 1, 32, 4, 512, 2048, 128, True),
        # One new token of each of 8 sequences over a cache of 4096.
        fa("attn_decode_8x4096", 8, 32, 4, 1, 4096, 128, True),
        # bs=1 weight-only linear: the smallest call of a decode step.
        gemv("gemv_i8_4096_b1", 4096, 4096, 1),
        # Greedy decode as quoted: 16-token prompt, 256 new tokens.
        generate("decode_16_256", 12, 16, 256),
        # A longer prompt and a short answer.
        generate("decode_256_64", 12, 256, 64),
        # Scoring a given text: the logits after each of its 200 tokens.
        logits("score_200", 12, 200),
    ]


def gemm(name, dtype, out, m, n, k) -> dict:
    return {"name": name, "kind": "gemm", "dtype": dtype, "out": out, "m": m, "n": n, "k": k}


def fa(name, batch, heads, kv_heads, seq_q, seq_k, head_dim, causal) -> dict:
    return {"name": name, "kind": "fa", "batch": batch, "heads": heads, "kv_heads": kv_heads,
            "seq_q": seq_q, "seq_k": seq_k, "head_dim": head_dim, "causal": causal}


def gemv(name, rows, cols, batch) -> dict:
    return {"name": name, "kind": "gemv", "rows": rows, "cols": cols, "batch": batch}


def generate(name, kv_heads, prompt, steps) -> dict:
    return {"name": name, "kind": "generate", "kv_heads": kv_heads, "prompt": prompt, "steps": steps}


def logits(name, kv_heads, tokens) -> dict:
    return {"name": name, "kind": "logits", "kv_heads": kv_heads, "tokens": tokens}


def _log(rng, lo, hi) -> int:
    """A size spread over the logarithm of its range."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _size(rng, lo, hi) -> int:
    """Half of the sizes as they come (odd ones among them), half on a grid
    that layers are usually built on."""
    v = _log(rng, lo, hi)
    if rng.random() < 0.5:
        g = 64 if v >= 512 else 8
        v = max(lo, min(hi, v // g * g))
    return v


def draw(rng) -> dict:
    kind = rng.choice(["gemm", "gemm", "gemm", "fa", "fa", "gemv", "generate", "logits"])
    if kind == "gemm":
        dtype, out = rng.choice([("bf16", "f32"), ("bf16", "bf16"), ("f16", "f32"), ("f32", "f32")])
        top = 2.0 ** 33 if dtype == "f32" else 2.0 ** 36  # no more work than the listed ones
        while True:
            hi = 4096 if dtype == "f32" else 12288
            m, n, k = _size(rng, 1, hi), _size(rng, 64, hi), _size(rng, 64, hi)
            if 2.0 ** 18 <= m * n * k <= top:
                break
        c = gemm("", dtype, out, m, n, k)
    elif kind == "fa":
        while True:
            head_dim = rng.choice([64, 128])
            kv_heads = rng.choice([1, 2, 4, 8, 12, 32])
            heads = kv_heads * rng.choice([1, 1, 4, 8])
            batch = _log(rng, 1, 16)
            causal = rng.random() < 0.7
            what = rng.choice(["square", "chunk", "decode"])
            seq_k = _size(rng, 16, 8192)
            seq_q = {"square": seq_k, "chunk": min(seq_k, _size(rng, 16, 512)), "decode": 1}[what]
            flops = 4.0 * batch * heads * seq_q * seq_k * head_dim
            if heads <= 64 and flops <= 2.7e11 and batch * kv_heads * seq_k * head_dim <= 2 ** 28:
                break
        c = fa("", batch, heads, kv_heads, seq_q, seq_k, head_dim, causal)
    elif kind == "gemv":
        cols = 16 * _log(rng, 16, 1024)
        c = gemv("", _size(rng, 256, 32000), cols, rng.choice([1, 1, 2, 4, 8, rng.randint(1, 16)]))
    elif kind == "generate":
        prompt, steps = _log(rng, 1, 256), _log(rng, 1, 64)
        c = generate("", rng.choice([12, 4]), prompt, steps)
    else:
        c = logits("", rng.choice([12, 4]), _log(rng, 1, 256))
    c.pop("name")
    return c


def _config(case) -> LlamaConfig:
    """The decoder of the decode benchmark (dim 768, 12 layers, SwiGLU 2048,
    vocabulary 32000), with all or a third of the KV heads."""
    return LlamaConfig(n_kv_heads=case["kv_heads"])


_rope: dict = {}


def _model(cfg: LlamaConfig, gen) -> dict[str, np.ndarray]:
    """The int8 model of N(0, 0.02) weights, quantised per row as
    vx_amd.llama.make_model does, with the numbers drawn on the GPU."""
    d, h, kv, L = cfg.dim, cfg.hidden_dim, cfg.kv_dim, cfg.n_layers
    out = {}

    def put(name, *shape):
        w = torch.randn(shape, generator=gen, device="cuda") * 0.02
        s = w.abs().amax(dim=-1) / 127.0
        out[f"{name}_q"] = torch.round(w / s[..., None]).clamp_(-127, 127).to(torch.int8).cpu().numpy()
        out[f"{name}_s"] = s.cpu().numpy()

    put("tok", cfg.vocab_size, d)
    for name, rows, cols in (("wq", d, d), ("wk", kv, d), ("wv", kv, d), ("wo", d, d), ("w1", h, d),
                             ("w2", d, h), ("w3", h, d)):
        put(name, L, rows, cols)
    out["rms_att"], out["rms_ffn"] = np.ones((L, d), np.float32), np.ones((L, d), np.float32)
    out["rms_final"] = np.ones(d, np.float32)
    if cfg not in _rope:
        _rope[cfg] = rope_table(cfg)
    out["rope"] = _rope[cfg]
    return out


class _Model(LlamaI8):
    def __del__(self):
        self.close()


class _Call:
    """A routed matmul's call site as a compiled program holds it: the
    payload is a constant, the descriptors and the argument array are on the
    stack."""

    def __init__(self, a, b, c, in_dtype, out_dtype):
        args = abi.CallArgs()
        args.memref(abi.Descriptor(a.data_ptr(), a.shape), in_dtype).scalar(0, abi.KIND_I64)
        args.memref(abi.Descriptor(b.data_ptr(), b.shape), in_dtype).scalar(1, abi.KIND_I64)
        args.scalar(0.0, abi.KIND_F32).memref(abi.Descriptor(c.data_ptr(), c.shape), out_dtype)
        payload = abi.matmul_payload()
        self.payload = ctypes.create_string_buffer(payload, len(payload))
        self.size = len(payload)
        self.keep = args
        self.argv, self.tags, self.n = args.arrays()
        self.fn = lib().lib.vx_plugin_dispatch_async

    def __call__(self):
        self.fn(self.payload, self.size, self.argv, self.tags, self.n)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _gemm_inputs(case, seed):
    g, dt = _gen(seed), TORCH[case["dtype"]]
    m, n, k = case["m"], case["n"], case["k"]
    if case["dtype"] == "f32":
        a = torch.rand((m, k), generator=g, device="cuda") * 2 - 1
        b = torch.rand((k, n), generator=g, device="cuda") * 2 - 1
        return a, b
    a = torch.randn((m, k), generator=g, device="cuda")
    b = torch.randn((k, n), generator=g, device="cuda") * k ** -0.5
    return a.to(dt), b.to(dt)


def _fa_inputs(case, seed):
    g, d = _gen(seed), case["head_dim"]

    def normal(heads, seq):
        return torch.randn((case["batch"], heads, seq, d), generator=g, device="cuda").to(torch.bfloat16)

    return (normal(case["heads"], case["seq_q"]), normal(case["kv_heads"], case["seq_k"]),
            normal(case["kv_heads"], case["seq_k"]))


def _gemv_inputs(case, seed):
    g = _gen(seed)
    w = torch.randint(-127, 128, (case["rows"], case["cols"]), generator=g, device="cuda", dtype=torch.int8)
    s = torch.rand(case["rows"], generator=g, device="cuda") * 0.009 + 0.001
    x = torch.randn((case["batch"], case["cols"]), generator=g, device="cuda").to(torch.bfloat16)
    return w, s, x


def _tokens(case, seed):
    rng = np.random.default_rng(seed)
    n = case["prompt"] if case["kind"] == "generate" else case["tokens"]
    return rng.integers(0, _config(case).vocab_size, size=n, dtype=np.int32)


def prepare(case, seed):
    st = {"case": case}
    kind = case["kind"]
    if kind == "gemm":
        a, b = _gemm_inputs(case, seed)
        c = torch.empty((case["m"], case["n"]), device="cuda", dtype=TORCH[case["out"]])
        st.update(a=a, b=b, c=c, call=_Call(a, b, c, DTYPE[case["dtype"]], DTYPE[case["out"]]))
    elif kind == "fa":
        q, k, v = _fa_inputs(case, seed)
        lse = torch.empty(q.shape[:3], device="cuda", dtype=torch.float32)
        st.update(q=q, k=k, v=v, o=torch.empty_like(q), lse=lse)
    elif kind == "gemv":
        w, s, x = _gemv_inputs(case, seed)
        st.update(w=w, s=s, x=x, y=torch.empty((case["batch"], case["rows"]), device="cuda"))
    else:
        cfg = _config(case)
        st.update(model=_Model(lib(), cfg, _model(cfg, _gen(seed))), tokens=_tokens(case, seed))
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemm":
        st["call"]()
        return st["c"]
    if kind == "fa":
        rc = flash_attention_fwd(lib(), st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(),
                                 st["o"].data_ptr(), st["lse"].data_ptr(), case["batch"], case["heads"],
                                 case["kv_heads"], case["seq_q"], case["seq_k"], case["head_dim"],
                                 case["head_dim"] ** -0.5, case["causal"])
        if rc != 0:
            raise RuntimeError(f"flash attention returned {rc}")
        return {"o": st["o"], "lse": st["lse"]}
    if kind == "gemv":
        rc = gemv_i8(lib(), st["w"].data_ptr(), st["s"].data_ptr(), st["x"].data_ptr(), st["y"].data_ptr(),
                     case["rows"], case["cols"], case["batch"])
        if rc != 0:
            raise RuntimeError(f"gemv returned {rc}")
        return st["y"]
    if kind == "generate":
        tokens, margin = st["model"].generate(st["tokens"], case["steps"])
        return {"tokens": tokens, "margin": margin}
    return st["model"].logits(st["tokens"])


def work(case) -> dict:
    kind = case["kind"]
    if kind == "gemm":
        m, n, k, e = case["m"], case["n"], case["k"], BYTES[case["dtype"]]
        return {"bytes": e * (m * k + k * n) + BYTES[case["out"]] * m * n, "flops": 2.0 * m * n * k}
    if kind == "fa":
        b, h, hk, sq, sk, d = (case[x] for x in ("batch", "heads", "kv_heads", "seq_q", "seq_k", "head_dim"))
        seen = sq * sk if not case["causal"] else sq * (sk - sq) + sq * (sq + 1) // 2
        return {"bytes": 2 * b * d * (2 * h * sq + 2 * hk * sk) + 4 * b * h * sq, "flops": 4.0 * b * h * seen * d}
    if kind == "gemv":
        r, c, b = case["rows"], case["cols"], case["batch"]
        return {"bytes": r * c + 4 * r + b * (2 * c + 4 * r), "flops": 2.0 * r * c * b}
    # The decoder: each new token waits for the one before it and reads every
    # weight; the tokens that are given (the prompt, the scored text) can
    # share one reading. All read the keys and values before them.
    cfg = _config(case)
    given = case["prompt"] if kind == "generate" else case["tokens"]
    after = case["steps"] - 1 if kind == "generate" else 0
    heads = given if kind == "logits" else 1  # positions the classifier is needed for
    classifier = cfg.vocab_size * cfg.dim
    layers = cfg.int8_weight_bytes() - classifier
    kv = 2 * cfg.n_layers * cfg.kv_dim * 4
    pos = given + after
    nbytes = (1 + after) * (layers + classifier) + kv * pos
    nbytes += sum(kv * p for p in range(given, pos))
    if kind == "logits":
        nbytes += 4 * given * cfg.vocab_size
    flops = 2.0 * pos * layers + 2.0 * (heads + after) * classifier
    flops += 4.0 * cfg.n_layers * cfg.dim * pos * (pos + 1) / 2
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "gemm":
        # f32 sums of K terms in another order (4e-7 to 1.1e-6 from the 64-bit
        # result, most at the longest K); a 16-bit result adds its one
        # rounding (1.7e-3).
        return {"rel": 1e-5, "max": 1e-4} if case["out"] == "f32" else {"rel": 7e-3, "max": 4e-2}
    if kind == "fa":
        return {"rel": 1e-2, "max": 0.1}  # probabilities and the output in bf16 (2.1e-3 to 2.5e-3)
    if kind == "gemv":
        return {"rel": 2e-6, "max": 2e-5}  # f32 sums of exact products (7e-8 at batch 1)
    if kind == "generate":
        # margins are differences of two logits (1.6e-6); a near tie may fall the other way
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    return {"rel": 4e-6, "max": 4e-5}  # 12 layers of f32 sums (4e-7)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        a, b = _gemm_inputs(case, seed)
        return a.double() @ b.double()
    if kind == "fa":
        return _fa_exact(case, seed)
    if kind == "gemv":
        w, s, x = _gemv_inputs(case, seed)
        return (x.double() @ w.double().T) * s.double()
    return _llama_exact(case, seed)


def _fa_exact(case, seed):
    q, k, v = (t.double() for t in _fa_inputs(case, seed))
    sq, sk = case["seq_q"], case["seq_k"]
    group = case["heads"] // case["kv_heads"]
    o, lse = torch.empty_like(q), torch.empty(q.shape[:3], device="cuda", dtype=torch.float64)
    hide = None
    if case["causal"]:
        i = torch.arange(sq, device="cuda")[:, None] + (sk - sq)
        hide = torch.arange(sk, device="cuda")[None, :] > i
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            s = (q[b, h] @ k[b, h // group].T.contiguous()) * case["head_dim"] ** -0.5
            if hide is not None:
                s.masked_fill_(hide, -math.inf)
            lse[b, h] = torch.logsumexp(s, dim=-1)
            o[b, h] = torch.exp(s - lse[b, h][:, None]) @ v[b, h // group]
    return {"o": o, "lse": lse}


def _llama_exact(case, seed):
    """The decoder in 64 bits: the given tokens together, then greedily one
    by one."""
    cfg = _config(case)
    w = _model(cfg, _gen(seed))
    hs, heads, kv_heads = cfg.head_size, cfg.n_heads, cfg.n_kv_heads

    def mat(name, layer=None):
        q, s = w[f"{name}_q"], w[f"{name}_s"]
        q, s = (q, s) if layer is None else (q[layer], s[layer])
        return torch.from_numpy(q).cuda().double() * torch.from_numpy(s).cuda().double()[:, None]

    tok = mat("tok")
    layers = [{n: mat(n, l) for n in ("wq", "wk", "wv", "wo", "w1", "w2", "w3")} for l in range(cfg.n_layers)]
    rope = torch.from_numpy(w["rope"]).cuda().double()
    cache = [[None, None] for _ in layers]

    def norm(x):  # the norm weights are 1
        return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + 1e-5)

    def rotate(x, p0):  # [T, heads, hs] at positions p0 ...
        c, s = rope[p0:p0 + x.shape[0], None, :, 0], rope[p0:p0 + x.shape[0], None, :, 1]
        e, o = x[..., 0::2], x[..., 1::2]
        return torch.stack((e * c - o * s, e * s + o * c), dim=-1).flatten(-2)

    def forward(ids, p0):
        x = tok[ids]
        T = x.shape[0]
        for kv, m in zip(cache, layers):
            y = norm(x)
            q = rotate((y @ m["wq"].T).view(T, heads, hs), p0)
            k = rotate((y @ m["wk"].T).view(T, kv_heads, hs), p0)
            v = (y @ m["wv"].T).view(T, kv_heads, hs)
            kv[0] = k if kv[0] is None else torch.cat((kv[0], k))
            kv[1] = v if kv[1] is None else torch.cat((kv[1], v))
            kk = kv[0].repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1).contiguous()
            vv = kv[1].repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1).contiguous()
            s = (q.transpose(0, 1).contiguous() @ kk.transpose(1, 2).contiguous()) * hs ** -0.5
            hide = torch.arange(kk.shape[1], device="cuda")[None, :] > torch.arange(T, device="cuda")[:, None] + p0
            p = torch.softmax(s.masked_fill(hide, -math.inf), dim=-1)
            x = x + (p @ vv).transpose(0, 1).reshape(T, cfg.dim) @ m["wo"].T
            y = norm(x)
            x = x + (torch.nn.functional.silu(y @ m["w1"].T) * (y @ m["w3"].T)) @ m["w2"].T
        return norm(x)

    ids = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda()
    if case["kind"] == "logits":
        return forward(ids, 0) @ tok.T
    x, p, margin = forward(ids, 0)[-1:], len(ids), []
    while True:
        top = torch.topk((x @ tok.T)[0], 2)
        margin.append(top.values[0] - top.values[1])
        if len(margin) == case["steps"]:
            return {"tokens": None, "margin": torch.stack(margin)}
        x, p = forward(top.indices[:1], p), p + 1
