"""The work that a user of this library has it do, one case per entry point:
the decode step's matvecs, their batched forms (speculative verify, prompts),
the prefill GEMM, one layer's attention over a KV cache, the IBF v5 INT4 and
product-quantised matvecs with the top-K head, and two whole calls on a
decoder of a few layers.

Sizes are those of the decoder shapes in libinferbit_amd.ibf (TinyLlama-1.1B:
hidden 2048, MLP 5632, 32/4 heads of 64; Mistral-7B: hidden 4096, MLP 14336,
32/8 heads of 128; vocabulary 32000) in the listed cases, and any size between
in the drawn ones.  Weights are N(0, 0.02) quantized per row (or per group) on
the GPU, activations N(0, 1) with a few large channels as behind an rmsnorm."""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

import libinferbit_amd as L
from libinferbit_amd import ibf
from libinferbit_amd.model import Model

DEV = "cuda:0"
VOCAB = 32000

# decoders of a few layers at the widths of the two benchmark shapes
DECODERS = {
    "tinyllama": dict(ibf.TINYLLAMA, num_layers=4),
    "mistral": dict(ibf.MISTRAL, num_layers=2),
}


def listed():
    return [
        # the smallest call: an INT8 projection of the small decoder, bound by latency and the launch
        dict(name="matvec-int8-2048x2048", kind="matvec", M=2048, N=2048, bits=8),
        # the headline: an INT4 MLP matrix of the large decoder, batch 1
        dict(name="matvec-int4-14336x4096", kind="matvec", M=14336, N=4096, bits=4),
        # the decode form of INT4 tensors, int8 activations quantized in front: the down projection
        dict(name="w4a8-4096x14336", kind="w4a8", M=4096, N=14336),
        # the same tensors for 16 positions at once, as a speculative verify issues them
        dict(name="w4a8-batch16-14336x4096", kind="w4a8_batch", M=14336, N=4096, B=16),
        # an INT8 attention projection for 8 positions
        dict(name="int8-batch8-4096x4096", kind="int8_batch", M=4096, N=4096, B=8),
        # a 512-token prompt through one MLP matrix: the largest call, bound by the matrix cores
        dict(name="gemm-512x4096x14336", kind="gemm", M=14336, N=4096, B=512),
        # one layer's cache write and attention at 4096 cached positions, INT8 cache
        dict(name="attn-int8-4096", kind="attn", heads=32, kv=8, hd=128, T=4096, bits=8),
        # a two-level product-quantised projection as the v5 session runs it by default
        dict(name="pq2-4096x14336", kind="pq", M=4096, C=896, levels=2, K2=256, outliers=0, variant="streaming"),
        # the v5 greedy / top-k sampling head over the whole vocabulary
        dict(name="pq-head-32000x4096-k50", kind="pq_head", M=VOCAB, C=256, levels=2, K2=256, k_top=50),
        # an IBF v5 INT4 group-scaled matrix with AWQ scales and fp16 outliers for 8 positions
        dict(name="int4g-batch8-14336x4096", kind="int4g", M=14336, N=4096, G=128, awq=True, K_out=8, B=8),
        # a whole call: logits behind a 32-token prompt, bit-identical mode (the default)
        dict(name="prompt32-tinyllama", kind="prompt", decoder="tinyllama", T=0, B=32),
        # a whole call: 8 drafted positions verified behind 1024 cached ones
        dict(name="verify8-mistral-1024", kind="verify", decoder="mistral", T=1024, B=8),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _rows(rng, lo=256, hi=14336):
    m = int(_log(rng, lo, hi))
    return max(lo, m // 16 * 16) if rng.random() < 0.5 else m


def _cols(rng, step, lo=512, hi=14336):
    s = max(step, rng.choice((4, 64, 128, 256, 512)))
    return min(hi // s * s, max((lo + s - 1) // s * s, int(_log(rng, lo, hi)) // s * s))


def draw(rng):
    kind = rng.choice(("matvec", "w4a8", "w4a8_batch", "int8_batch", "gemm", "attn", "pq", "pq_head", "int4g", "prompt",
                       "verify"))
    if kind == "matvec":
        return dict(kind=kind, M=_rows(rng), N=_cols(rng, 4), bits=rng.choice((8, 4, 2)))
    if kind == "w4a8":
        return dict(kind=kind, M=_rows(rng), N=_cols(rng, 32))
    if kind == "w4a8_batch":
        return dict(kind=kind, M=_rows(rng), N=_cols(rng, 128) // 128 * 128, B=rng.randint(1, 32))
    if kind == "int8_batch":
        return dict(kind=kind, M=_rows(rng, hi=8192), N=_cols(rng, 32, hi=8192), B=rng.randint(1, 32))
    if kind == "gemm":
        return dict(kind=kind, M=_rows(rng, 512), N=_cols(rng, 64, hi=4096), B=int(_log(rng, 33, 513)))
    if kind == "attn":
        heads, kv, hd = rng.choice(((32, 8, 128), (32, 4, 64), (32, 32, 128), (16, 2, 64)))
        return dict(kind=kind, heads=heads, kv=kv, hd=hd, T=int(_log(rng, 16, 8000)), bits=rng.choice((8, 8, 32, 4)))
    if kind == "pq":
        levels = rng.choice((1, 2, 2))
        return dict(kind=kind, M=_rows(rng, hi=8192), C=int(_log(rng, 64, 897)), levels=levels,
                    K2=rng.choice((256, 64, 16)) if levels == 2 else 0, outliers=rng.choice((0, 0, 16, 128)),
                    variant=rng.choice(("streaming", "streaming", "skip", "sparse", "l1_only")))
    if kind == "pq_head":
        levels = rng.choice((1, 2))
        return dict(kind=kind, M=int(_log(rng, 4096, VOCAB + 1)), C=rng.choice((64, 128, 160, 256)), levels=levels,
                    K2=256 if levels == 2 else 0, k_top=rng.choice((8, 40, 50, 100)))
    if kind == "int4g":
        G = rng.choice((128, 128, 128, 64, 32))
        return dict(kind=kind, M=_rows(rng), N=_cols(rng, 128) // 128 * 128, G=G, awq=rng.random() < 0.5,
                    K_out=rng.choice((0, 4, 8, 20)), B=rng.choice((1, rng.randint(2, 16), rng.randint(2, 32))))
    decoder = rng.choice(("tinyllama", "mistral"))
    if kind == "prompt":
        return dict(kind=kind, decoder=decoder, T=rng.choice((0, int(_log(rng, 16, 1024)))), B=int(_log(rng, 1, 100)))
    return dict(kind=kind, decoder=decoder, T=int(_log(rng, 16, 2000)), B=rng.randint(2, 16))


# ── inputs ────────────────────────────────────────────────────────────────


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _acts(g, *shape):
    """N(0, 1) with about one channel in 128 eight times as large, the same channels for every position."""
    x = torch.randn(*shape, generator=g, device=DEV)
    big = (torch.rand(shape[-1], generator=g, device=DEV) < 1 / 128).float()
    return x * (1 + 7 * big)


def _weights(g, bits, M, N):
    """N(0, 0.02) rows quantized by the per-row rules of the v1 file: packed codes, fp16 scales."""
    w = torch.empty(M, N * bits // 8, dtype=torch.uint8, device=DEV)
    s = torch.empty(M, dtype=torch.float16, device=DEV)
    for r in range(0, M, 4096):
        a = torch.randn(min(4096, M - r), N, generator=g, device=DEV) * 0.02
        if bits == 2:
            th = 0.7 * a.abs().mean(1, keepdim=True)
            keep = a.abs() > th
            sc = (a.abs() * keep).sum(1, keepdim=True) / keep.sum(1, keepdim=True).clamp(min=1)
            q = (1 + keep * a.sign()).to(torch.uint8).view(-1, N // 4, 4)
            p = q[:, :, 0] | q[:, :, 1] << 2 | q[:, :, 2] << 4 | q[:, :, 3] << 6
        else:
            top = 127 if bits == 8 else 7
            sc = a.abs().amax(1, keepdim=True) / top
            q = (a / sc).round().clamp(-top, top)
            if bits == 8:
                p = q.to(torch.int8).view(torch.uint8)
            else:
                q = (q + 8).to(torch.uint8).view(-1, N // 2, 2)
                p = q[:, :, 0] | q[:, :, 1] << 4
        w[r:r + a.shape[0]] = p
        s[r:r + a.shape[0]] = sc.squeeze(1).half()
    return w, s


def _dense(w, s, bits, M, N):
    """The matrix that the packed codes and scales stand for, in 64 bits."""
    if bits == 8:
        q = w.view(torch.int8).double()
    elif bits == 4:
        q = torch.stack((w & 15, w >> 4), 2).view(M, N).double() - 8
    else:
        q = torch.stack((w & 3, (w >> 2) & 3, (w >> 4) & 3, w >> 6), 2).view(M, N).double() - 1
    return q * s.double()[:, None]


def _over(a, n):
    """a / n rounded once (a number as divisor is turned into a product with its reciprocal)."""
    return a / torch.full_like(a, float(n))


def _quant_act(x):
    """The per-128-group int8 rule of the W4A8 form: codes and scales, in 32 bits as it is defined."""
    B, N = x.shape
    G = (N + 127) // 128
    p = torch.zeros(B, G * 128, device=DEV)
    p[:, :N] = x
    p = p.view(B, G, 128)
    sc = _over(p.abs().amax(2), 127)
    t = p * (1.0 / sc)[:, :, None]
    q = torch.trunc(t + torch.where(p >= 0, 0.5, -0.5)).clamp(-127, 127)
    return q.to(torch.int8).view(B, G * 128)[:, :N].contiguous(), sc.contiguous()


def _f16bits(a):
    return np.asarray(a, np.float16).view(np.uint16)


def _pq_tensor(case, seed):
    """A product-quantised matrix in the file's layout: 16-column chunks, 256 codewords a side."""
    r = np.random.default_rng(seed)
    M, C, K, K2 = case["M"], case["C"], 256, case["K2"]
    n_out = case.get("outliers", 0)
    t = dict(M=M, N=16 * C + n_out, G=16, K=K, n_levels=case["levels"], n_outlier=n_out, C=C, K_l2=K2)
    for s in "lr":
        t["cb1" + s] = _f16bits(r.standard_normal((K, 8)) * 0.02)
        t["i1" + s] = np.frombuffer(r.bytes(M * C), np.uint8).reshape(M, C)
        if case["levels"] == 2:
            t["cb2" + s] = _f16bits(r.standard_normal((K2, 8)) * 0.005)
            i2 = np.frombuffer(r.bytes(M * C), np.uint8).reshape(M, C) & np.uint8(K2 - 1)
            t["i2" + s] = i2
            if K2 == 16:
                p = np.zeros((M, C + (C & 1)), np.uint8)
                p[:, :C] = i2
                t["i2" + s] = p[:, 0::2] | p[:, 1::2] << 4
    t["row_scale"] = _f16bits(1 + 0.1 * r.standard_normal(M))
    if n_out:
        t["ocols"] = np.sort(r.choice(t["N"], n_out, replace=False)).astype(np.int32)
        t["oside"] = r.integers(-127, 128, (M, n_out), dtype=np.int8)
        t["oscale"] = _f16bits(r.uniform(0.5, 1.5, n_out) * 3e-4)
    return t


def _pq_x(case, seed, t):
    """Activations of a product-quantised projection, some chunks of them quiet."""
    x = _acts(_gen(seed), t["N"])
    quiet = torch.rand(t["N"] // 16 + 1, generator=_gen(seed + 1), device=DEV) < 0.1
    return x * torch.where(quiet.repeat_interleave(16)[:t["N"]], 1e-4, 1.0)


def _int4g(case, seed):
    """Group-scaled INT4 codes of N(0, 0.02) rows; the K_out largest weights of a row kept in fp16 beside them."""
    g = _gen(seed)
    M, N, G, K = case["M"], case["N"], case["G"], case["K_out"]
    q = np.empty((M, N // 2), np.uint8)
    s = np.empty((M, N // G), np.uint16)
    idx, val = np.empty((M, K), np.uint16), np.empty((M, K), np.uint16)
    for r in range(0, M, 4096):
        a = torch.randn(min(4096, M - r), N, generator=g, device=DEV) * 0.02
        n = a.shape[0]
        if K:
            i = a.abs().topk(K, 1).indices
            idx[r:r + n] = i.cpu().numpy().astype(np.uint16)
            val[r:r + n] = a.gather(1, i).half().cpu().numpy().view(np.uint16)
            a.scatter_(1, i, 0.0)
        v = a.view(n, N // G, G)
        sc = (v.abs().amax(2, keepdim=True) / 7).half()
        c = ((v / sc.float()).round().clamp(-8, 7) + 8).to(torch.uint8).view(n, N // 2, 2)
        q[r:r + n] = (c[:, :, 0] | c[:, :, 1] << 4).cpu().numpy()
        s[r:r + n] = sc.squeeze(2).cpu().numpy().view(np.uint16)
    t = dict(q=q, s=s)
    if case["awq"]:
        t["inv_act"] = torch.exp(0.3 * torch.randn(N, generator=g, device=DEV)).cpu().numpy()
    if K:
        t.update(outl_idx=idx, outl_val=val)
    return t, _acts(g, case["B"], N)


def _kv_fill(g, T, kv, hd, bits):
    """An empty cache of T rows and the fp32 K and V to be written into it."""
    row = kv * hd
    shape = (T, row) if bits in (32, 8) else (T, kv * hd // 2)
    dt = torch.float32 if bits == 32 else torch.int8 if bits == 8 else torch.uint8
    data = [torch.zeros(shape, dtype=dt, device=DEV) for _ in "kv"]
    sc = [torch.zeros(T, kv, device=DEV) if bits < 16 else None for _ in "kv"]
    return data, sc, [torch.randn(T, row, generator=g, device=DEV) for _ in "kv"]


def _decoder(case, seed):
    cfg = DECODERS[case["decoder"]]
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "m.ibf")
        ibf.write_synthetic(path, cfg, seed=seed)
        m = Model(path)
    r = np.random.default_rng(seed)
    if case["T"]:
        shape = (cfg["num_layers"], case["T"], cfg["num_kv_heads"] * cfg["head_dim"])
        m.kv_prefill(*(r.standard_normal(shape, np.float32) for _ in "kv"))
    return dict(model=m, T=case["T"], tokens=r.integers(0, VOCAB, case["B"]).astype(np.int32))


def prepare(case, seed):
    L.ops.init(0)
    kind, g = case["kind"], _gen(seed)
    if kind in ("prompt", "verify"):
        return dict(case=case, **_decoder(case, seed))
    if kind == "attn":
        data, sc, kv = _kv_fill(g, case["T"], case["kv"], case["hd"], case["bits"])
        for t in range(case["T"] - 1):   # the positions decoded so far
            L.ops.kv_cache_write(*data, *sc, t, kv[0][t], kv[1][t], case["kv"], case["hd"], case["bits"])
        q = torch.randn(case["heads"] * case["hd"], generator=g, device=DEV)
        return dict(case=case, data=data, sc=sc, q=q, k=kv[0][-1].clone(), v=kv[1][-1].clone(), out=torch.empty_like(q))
    if kind in ("pq", "pq_head"):
        t = _pq_tensor(case, seed)
        return dict(case=case, t=L.ops.PqDeviceTensor(t), x=_pq_x(case, seed, t), out=torch.empty(case["M"], device=DEV))
    if kind == "int4g":
        t, x = _int4g(case, seed)
        return dict(case=case, t=L.ops.Int4gDeviceTensor(t), x=x, out=torch.empty(case["B"], case["M"], device=DEV))
    M, N, B = case["M"], case["N"], case.get("B", 1)
    bits = case.get("bits", 4 if kind.startswith("w4a8") else 8)
    w, s = _weights(g, bits, M, N)
    st = dict(case=case, w=w, s=s, x=_acts(g, B, N), out=torch.empty(B, M, device=DEV))
    if kind == "w4a8":
        st.update(q=torch.empty(N, dtype=torch.int8, device=DEV), sa=torch.empty((N + 127) // 128, device=DEV))
    elif kind == "w4a8_batch":
        st["q"], st["sa"] = _quant_act(st["x"])
    elif kind == "gemm":
        st["ws"] = torch.empty(L.lib().ibh_gemm_int8_workspace_bytes(N, B), dtype=torch.uint8, device=DEV)
    return st


# ── one pass ──────────────────────────────────────────────────────────────

VARIANTS = {"streaming": (0, 0.0, 0.0), "l1_only": (1, 0.0, 0.0), "sparse": (3, 0.0, 1e-2)}


def run(st):
    c, ops = st["case"], L.ops
    kind = c["kind"]
    if kind == "matvec":
        ops.parallel_matmul(st["out"], st["w"], st["s"], st["x"], c["M"], c["N"], c["bits"])
    elif kind == "w4a8":
        ops.matmul_w4a8_x(st["out"], st["w"], st["s"], st["x"], c["M"], c["N"], st["q"], st["sa"])
    elif kind == "w4a8_batch":
        ops.matmul_w4a8_batch(st["out"], st["w"], st["s"], st["q"], st["sa"], c["M"], c["N"], c["B"], c["M"])
    elif kind == "int8_batch":
        ops.matmul_int8_batch(st["out"], st["w"], st["s"], st["x"], c["M"], c["N"], c["B"], c["M"])
    elif kind == "gemm":
        ops.gemm_int8(st["out"], st["w"], st["s"], st["x"], c["M"], c["N"], c["B"], c["M"], st["ws"])
    elif kind == "attn":
        pos = c["T"] - 1
        ops.kv_cache_write(*st["data"], *st["sc"], pos, st["k"], st["v"], c["kv"], c["hd"], c["bits"])
        ops.attn_decode(st["out"], st["q"], *st["data"], *st["sc"], pos, c["heads"], c["kv"], c["hd"], c["bits"])
        return [st["out"], *st["data"], *(s for s in st["sc"] if s is not None)]
    elif kind == "pq":
        if c["variant"] == "skip":
            st["t"].matmul(st["x"], st["out"])
        else:
            st["t"].matmul_policy(st["x"], st["out"], *VARIANTS[c["variant"]])
    elif kind == "pq_head":
        return list(st["t"].lm_head_topk(st["x"], c["k_top"]))
    elif kind == "int4g":
        if c["B"] == 1:
            st["t"].matmul(st["x"][0], st["out"][0])
        else:
            st["t"].matmul_batched(st["x"], st["out"])
    else:
        m = st["model"]
        y = m.forward(st["tokens"]) if kind == "prompt" else m.forward_positions(st["tokens"])
        m.kv_truncate(st["T"])
        return y
    return st["out"]


# ── what a pass cannot do without ─────────────────────────────────────────


def work(case):
    kind = case["kind"]
    if kind == "attn":
        T, kv, hd, bits = case["T"], case["kv"], case["hd"], case["bits"]
        row = kv * hd * bits // 8 + (4 * kv if bits < 16 else 0)
        return {"bytes": 2 * T * row + 8 * (case["heads"] + kv) * hd, "flops": 4.0 * T * case["heads"] * hd}
    if kind in ("pq", "pq_head"):
        M, C, K2 = case["M"], case["C"], case["K2"]
        n_out = case.get("outliers", 0)
        l2 = case["levels"] == 2 and case.get("variant") != "l1_only"
        books = 2 * 256 * 16 + (2 * K2 * 16 if l2 else 0)
        rows = 2.0 * C * (1 + (0 if not l2 or kind == "pq_head" else 0.5 if K2 == 16 else 1)) + 2 + n_out
        b = M * rows + books + 4 * (16 * C + n_out) + (8 * case["k_top"] if kind == "pq_head" else 4 * M)
        return {"bytes": b, "flops": M * C * (4.0 if l2 else 2.0) + 2.0 * books * C}
    if kind == "int4g":
        M, N, B = case["M"], case["N"], case["B"]
        b = M * N // 2 + 2 * M * (N // case["G"]) + 4 * M * case["K_out"] + (4 * N if case["awq"] else 0)
        return {"bytes": b + 4 * B * (N + M), "flops": 2.0 * B * M * N}
    if kind in ("prompt", "verify"):
        cfg, B, T = DECODERS[case["decoder"]], case["B"], case["T"]
        H, I, nl = cfg["hidden_size"], cfg["intermediate_size"], cfg["num_layers"]
        KV = cfg["num_kv_heads"] * cfg["head_dim"]
        attn, mlp = H * (H + 2 * KV), H * H + 3 * H * I          # INT8 q/k/v; INT4 o and MLP
        row = KV * cfg["kv_bits"] // 8
        heads = VOCAB * H * (1 if kind == "prompt" else B)
        b = nl * (attn + mlp // 2 + 2 * row * (T + B)) + VOCAB * H + 4 * VOCAB * (1 if kind == "prompt" else B)
        return {"bytes": b, "flops": 2.0 * (B * nl * (attn + mlp) + heads) + 4.0 * nl * H * B * (T + B / 2)}
    M, N, B = case["M"], case["N"], case.get("B", 1)
    bits = case.get("bits", 4 if kind.startswith("w4a8") else 8)
    x = N + 4 * ((N + 127) // 128) if kind == "w4a8_batch" else 4 * N
    return {"bytes": M * N * bits // 8 + 2 * M + B * (x + 4 * M), "flops": 2.0 * B * M * N}


def tolerance(case):
    kind = case["kind"]
    if kind in ("w4a8", "w4a8_batch", "prompt", "verify"):
        return "exact"      # integer sums folded in a fixed order; the whole calls run in the bit-identical mode
    if kind == "pq_head":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.01}
    # 32-bit sums in another order, activations to about 2^-21 of the largest one (up to 8e-6 from 64 bits was
    # measured); cache codes are whole values and stay
    return {"rel": 2e-5, "max": 2e-4}


# ── the same in 64 bits ───────────────────────────────────────────────────


def _pq_dense(t, levels):
    """[M, 16 C] in 64 bits, the row scale applied."""
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in t.items()
           if isinstance(v, np.ndarray) and v.dtype == np.uint8}
    book = {k: torch.from_numpy(v.view(np.float16).astype(np.float64)).to(DEV) for k, v in t.items()
            if k.startswith("cb")}
    M, C = t["M"], t["C"]
    w = torch.empty(M, C, 16, dtype=torch.float64, device=DEV)
    for h, s in enumerate("lr"):
        v = book["cb1" + s][dev["i1" + s].long()]
        if levels == 2:
            i2 = dev["i2" + s]
            if t["K_l2"] == 16:
                i2 = torch.stack((i2 & 15, i2 >> 4), 2).view(M, -1)[:, :C]
            v = v + book["cb2" + s][i2.long()]
        w[:, :, 8 * h:8 * h + 8] = v
    return w.view(M, 16 * C) * torch.from_numpy(t["row_scale"].view(np.float16).astype(np.float64)).to(DEV)[:, None]


def _pq_exact(case, seed):
    t = _pq_tensor(case, seed)
    x = _pq_x(case, seed, t).double()
    inner = torch.ones(t["N"], dtype=torch.bool, device=DEV)
    y = torch.zeros(case["M"], dtype=torch.float64, device=DEV)
    if t["n_outlier"]:
        oc = torch.from_numpy(t["ocols"]).to(DEV).long()
        inner[oc] = False
        osc = torch.from_numpy(t["oscale"].view(np.float16).astype(np.float64)).to(DEV)
        xo = osc * x[oc]
        if t["n_outlier"] >= 32:            # from 32 columns on their activations are int8 codes of one scale, as defined
            xo = (x[oc].float() * osc.float())
            meta = _over(xo.abs().max(), 127)
            u = xo * (1.0 / meta)
            xo = torch.trunc(u + torch.where(u >= 0, 0.5, -0.5)).clamp(-128, 127).double() * meta.double()
        y += torch.from_numpy(t["oside"]).to(DEV).double() @ xo
    xi = x[inner].view(-1, 16).clone()
    top = xi.abs().amax(1)
    if case.get("variant") == "skip":       # chunks below a hundredth of the largest activation
        xi[top.float() < (0.01 * xi.abs().max().float())] = 0
    elif case.get("variant") == "sparse":
        xi[top.float() <= VARIANTS["sparse"][2]] = 0
    xi = xi.view(-1)
    if case["kind"] == "pq":
        return y + _pq_dense(t, 1 if case["variant"] == "l1_only" else case["levels"]) @ xi
    best = (_pq_dense(t, 1) @ xi).topk(case["k_top"]).indices
    full = (_pq_dense(t, case["levels"])[best] @ xi).sort(descending=True)
    return [full.values, best[full.indices].to(torch.int32)]


def _attn_exact(case, seed):
    g = _gen(seed)
    T, kv, hd, nh, bits = (case[k] for k in ("T", "kv", "hd", "heads", "bits"))
    _, _, fill = _kv_fill(g, T, kv, hd, bits)
    q = torch.randn(nh * hd, generator=g, device=DEV).double().view(kv, nh // kv, hd)
    codes, scales, vals = [], [], []
    for a in (f.view(T, kv, hd) for f in fill):
        if bits == 32:
            codes.append(a.reshape(T, -1).double())
            vals.append(a.double())
            continue
        top = 127 if bits == 8 else 7
        sc = _over(a.abs().amax(2), top).clamp(min=1e-8)
        t = a * (1.0 / sc)[:, :, None]
        c = torch.trunc(t + torch.where(t >= 0, 0.5, -0.5)).clamp(-top, top)
        codes.append(None)
        scales.append(sc.double())
        vals.append(c.double() * sc.double()[:, :, None])
    p = torch.softmax((torch.matmul(q, vals[0].permute(1, 2, 0).contiguous())) / math.sqrt(hd), 2)
    out = torch.matmul(p, vals[1].permute(1, 0, 2).contiguous()).reshape(-1)
    return [out, *codes, *scales]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prompt", "verify"):
        return None     # int8 activation codes follow the 32-bit sums in front of them: 64 bits give other codes
    if kind in ("pq", "pq_head"):
        return _pq_exact(case, seed)
    if kind == "attn":
        return _attn_exact(case, seed)
    if kind == "int4g":
        t, x = _int4g(case, seed)
        M, N, G = case["M"], case["N"], case["G"]
        q, s = torch.from_numpy(t["q"]).to(DEV), torch.from_numpy(t["s"].view(np.float16)).to(DEV).double()
        w = (torch.stack((q & 15, q >> 4), 2).view(M, N // G, G).double() - 8).mul_(s[:, :, None]).view(M, N)
        if case["K_out"]:
            w.scatter_add_(1, torch.from_numpy(t["outl_idx"].astype(np.int64)).to(DEV),
                           torch.from_numpy(t["outl_val"].view(np.float16).astype(np.float64)).to(DEV))
        x = x.double()
        if case["awq"]:
            x = x * torch.from_numpy(t["inv_act"]).to(DEV).double()
        return x @ w.t().contiguous()
    g = _gen(seed)
    M, N, B = case["M"], case["N"], case.get("B", 1)
    bits = case.get("bits", 4 if kind.startswith("w4a8") else 8)
    w, s = _weights(g, bits, M, N)
    x = _acts(g, B, N)
    if kind.startswith("w4a8"):
        q, sa = _quant_act(x)
        x = q.double() * sa.double().repeat_interleave(128, 1)[:, :N]
    return x.double() @ _dense(w, s, bits, M, N).t().contiguous()
