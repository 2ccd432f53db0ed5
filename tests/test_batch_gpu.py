"""Batched-position kernels: the INT8 batch chains against the oracle bit for
bit (through the dispatch-table entry that runs them, at tile edges,
remainders and every slots-per-wavefront form)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def table():
    import libinferbit_amd as L
    L.ops.init(0)
    P, I = C.c_void_p, C.c_int
    names = ("matmul_int4", "matmul_int8", "matmul_int2", "rmsnorm", "rope", "softmax", "silu_mul", "matmul_w4a8",
             "matmul_w4a8_batch", "matmul_int8_batch")

    class Kernels(C.Structure):
        _fields_ = [(n, P) for n in names]

    k = Kernels()
    L.lib().ib_init_kernels_hip(C.byref(k))
    return {"matmul_int8_batch": C.CFUNCTYPE(None, P, P, P, P, I, I, I, I)(k.matmul_int8_batch),
            "matmul_int8": C.CFUNCTYPE(None, P, P, P, P, I, I)(k.matmul_int8)}


# M, N, B, M_stride: one row and column block; partial row and column tiles;
# 1, 2 and 4 slots per wavefront (4: 8192 rows x 32); N % 16 != 0 (one chain per thread)
@pytest.mark.parametrize("M,N,B,ms", [(1, 16, 1, 1), (64, 128, 8, 64), (65, 144, 3, 70), (200, 400, 32, 203),
                                      (1000, 2048, 17, 1000), (4096, 144, 32, 4096), (8192, 272, 31, 8192),
                                      (8192, 128, 32, 8195), (33, 100, 5, 33)])
def test_int8_batch_chains_bit_exact(table, oracle_lib, M, N, B, ms):
    print(f"case int8 chains M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(-127, 128, (M, N), dtype=np.int8)
    s = (r.random(M) * 0.01 + 1e-4).astype(np.float32)
    x = r.standard_normal((B, N)).astype(np.float32)
    want = oracle_lib.matmul_int8_batch(w, s, x, ms)
    out = np.full((B - 1) * ms + M, 7.0, np.float32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    table["matmul_int8_batch"](p(out), p(w), p(s), p(x), M, N, B, ms)
    want = np.asarray(want).reshape(-1)
    for b in range(B):
        np.testing.assert_array_equal(out[b * ms:b * ms + M].view(np.uint32), want[b * ms:b * ms + M].view(np.uint32))
        assert (out[b * ms + M:(b + 1) * ms] == 7.0).all()


# rows that end inside a 128-column group, at every columns-per-pass form
@pytest.mark.parametrize("M,N,B", [(48, 192, 5), (33, 160, 16), (100, 1056, 9), (17, 96, 32), (64, 416, 4), (20, 32, 6)])
def test_w4a8_batch_ragged_groups_bit_exact(oracle_lib, M, N, B):
    import torch

    import libinferbit_amd as L
    L.ops.init(0)
    print(f"case w4a8 batch ragged M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(0, 256, (M, N // 2), dtype=np.uint8)
    s = (r.random(M) * 0.01 + 1e-3).astype(np.float16)
    qx = r.integers(-127, 128, (B, N), dtype=np.int8)
    sa = (r.random((B, (N + 127) // 128)) * 0.02 + 1e-3).astype(np.float32)
    out = torch.empty(B * M, device="cuda")
    L.ops.matmul_w4a8_batch(out, torch.from_numpy(w).cuda(), torch.from_numpy(s.view(np.int16)).cuda(),
                            torch.from_numpy(qx).cuda(), torch.from_numpy(sa).cuda(), M, N, B, M)
    want = oracle_lib.matmul_w4a8_batch(w, s.astype(np.float32), qx, sa).reshape(-1)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


PROMPT_MODELS = {
    "int8kv": dict(kv_bits=8),
    "fp32kv": dict(kv_bits=32),
    "int4kv": dict(kv_bits=4, num_kv_heads=4),
    "mlp_int2": dict(kv_bits=8, bits=dict(gate_proj=2, up_proj=2, down_proj=2)),
    "all_int8": dict(kv_bits=8, bits=dict(o_proj=8, gate_proj=8, up_proj=8, down_proj=8)),
    "all_int4": dict(kv_bits=32, bits=dict(q_proj=4, k_proj=4, v_proj=4, token_embedding=4, head=4)),
    "mixed_qkv": dict(kv_bits=8, bits=dict(q_proj=8, k_proj=4, v_proj=8)),
    "hd128": dict(kv_bits=8, hidden_size=512, num_heads=4, num_kv_heads=1, head_dim=128),
    "ragged": dict(kv_bits=8, hidden_size=192, num_heads=3, num_kv_heads=1, intermediate_size=320),
}


def _add_masks(path, inter, keep):
    """Append a sparsity mask to every layer of an IBF file: a share of `keep`
    of the MLP rows active, other rows in each layer."""
    import json

    from libinferbit_amd import ibf
    raw = open(path, "rb").read()
    n = int(np.frombuffer(raw[8:16], np.uint32)[1])
    head, data = json.loads(raw[32:32 + n]), raw[ibf._align(32 + n):]
    for i, layer in enumerate(head["layers"]):
        data += bytes(ibf._align(len(data)) - len(data))
        layer["sparsity_mask"] = {"offset": len(data), "size": inter}
        data += (np.random.default_rng(i).random(inter) < keep).astype(np.uint8).tobytes()
    head["data"]["weight_data_size"] = len(data)
    js = json.dumps(head, separators=(",", ":")).encode()
    with open(path, "wb") as f:
        f.write(raw[:8] + np.array([1, len(js), 0], np.uint32).tobytes() + bytes(12) + js)
        f.write(bytes(ibf._align(32 + len(js)) - 32 - len(js)) + data)


@pytest.mark.parametrize("name", list(PROMPT_MODELS))
def test_prompt_equals_single_steps(tmp_path, name):
    """A prompt in batched passes leaves the logits, the cache and the greedy
    stream of single steps, bit for bit (exact mode): prompts of one pass, of
    several, with a short last one, and behind cached positions."""
    from libinferbit_amd import ibf
    from libinferbit_amd.model import Model
    spec = dict(PROMPT_MODELS[name])
    bits = spec.pop("bits", None)
    cfg = dict(ibf.TINYLLAMA, num_layers=2, hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64,
               intermediate_size=512, vocab_size=1000, max_context_length=200)
    cfg.update(spec)
    path = str(tmp_path / "m.ibf")
    ibf.write_synthetic(path, cfg, seed=31, bits=bits)
    toks = np.random.default_rng(7).integers(0, 1000, 130).astype(np.int32)
    one, many = Model(path), Model(path)
    at = 0
    for n in (3, 33, 1, 70, 2, 16):
        print(f"case prompt {name} {at}+{n}", flush=True)
        for t in toks[at:at + n]:
            a = one.forward([t])
        b = many.forward(toks[at:at + n])
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
        at += n
    assert one.kv_length() == many.kv_length() == at
    # the caches are the same: so is what follows from them
    np.testing.assert_array_equal(one.forward_positions(toks[:5]).view(np.uint32),
                                  many.forward_positions(toks[:5]).view(np.uint32))
    one.kv_clear()
    many.kv_clear()
    for t in toks[:39]:
        one.forward([t])
    np.testing.assert_array_equal(one.generate(toks[39:40], 9), many.generate(toks[:40], 9))
    one.close()
    many.close()


# both folds (tall matrices hand the sum on, others gather), 1 and 2 column
# tiles, codes in LDS and (2048 x 5632 at 17 columns and more) from L2; a last
# row tile and a last group that are not whole
@pytest.mark.parametrize("M,N,B", [(6001, 2048, 5), (6001, 2048, 32), (8200, 4096, 16), (8200, 4096, 17), (4099, 2080, 9),
                                   (2048, 2048, 9), (1003, 2048, 16), (1024, 4096, 17), (2048, 5632, 31),
                                   (500, 6176, 20), (14336, 4096, 8), (5632, 6144, 12), (40, 64, 17)])
def test_w4a8_batch_columns_bit_exact(oracle_lib, M, N, B):
    import torch

    import libinferbit_amd as L
    L.ops.init(0)
    print(f"case w4a8 columns M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(0, 256, (M, N // 2), dtype=np.uint8)
    s = (r.random(M) * 0.01 + 1e-3).astype(np.float16)
    qx = r.integers(-127, 128, (B, N), dtype=np.int8)
    sa = (r.random((B, (N + 127) // 128)) * 0.02 + 1e-3).astype(np.float32)
    ms = M + 3
    out = torch.full(((B - 1) * ms + M,), 7.0, device="cuda")
    L.ops.matmul_w4a8_batch(out, torch.from_numpy(w).cuda(), torch.from_numpy(s.view(np.int16)).cuda(),
                            torch.from_numpy(qx).cuda(), torch.from_numpy(sa).cuda(), M, N, B, ms)
    got = out.cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(min(M, 40)), np.arange(max(0, M - 40), M), r.integers(0, M, 200)]))
    want = oracle_lib.matmul_w4a8_batch(np.ascontiguousarray(w[rows]), s[rows].astype(np.float32), qx, sa).reshape(B, -1)
    for b in range(B):
        np.testing.assert_array_equal(got[b * ms + rows].view(np.uint32), want[b].view(np.uint32))
        assert (got[b * ms + M:(b + 1) * ms] == 7.0).all()


# the last column count of one kernel and the first of the other, for the rules
# by groups, by row tiles per block and by a badly filled last round of blocks
@pytest.mark.parametrize("M,N,B", [(70, 256, 8), (70, 256, 9), (1003, 512, 16), (1003, 512, 17), (1003, 896, 16),
                                   (1003, 896, 17), (100, 1152, 8), (100, 1152, 9), (4100, 4096, 10), (4100, 4096, 11),
                                   (4100, 8192, 5), (4100, 8192, 6), (9000, 2560, 8), (9000, 2560, 9), (9216, 8192, 10),
                                   (9216, 8192, 11), (20000, 2048, 9), (20000, 2048, 10), (70, 288, 5), (70, 288, 4)])
def test_w4a8_batch_handover_bit_exact(oracle_lib, M, N, B):
    test_w4a8_batch_columns_bit_exact(oracle_lib, M, N, B)


# M, N, B, M_stride: part-filled row tiles and column tiles, one and two row
# tiles per wavefront, rows that end inside a 128-column group or are shorter
# than the wavefronts' split, both column-tile forms
@pytest.mark.parametrize("M,N,B,ms", [(1, 16, 2, 1), (17, 144, 3, 20), (4100, 1040, 16, 4100), (4113, 4080, 9, 4113),
                                      (100, 8192, 17, 100), (4112, 656, 32, 4120)])
def test_int8_batch_digits(M, N, B, ms):
    """Fast INT8 batch against float64.  An element keeps at most max|group| *
    2^-29 of error (a digit unit), the group's sum 2^-23, each of the fp32 sums
    (N / 128 / 8 in a wavefront, 8 over them) 2^-24 of its partial: bounded by 2^-24 * (N / 1024 + 13) of sum |w| * max|group|."""
    import torch
    import libinferbit_amd as L
    L.ops.init(0)
    print(f"case int8 digits M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(-127, 128, (M, N), dtype=np.int8)
    s = (r.random(M) * 0.01 + 1e-4).astype(np.float32)
    x = r.standard_normal((B, N)).astype(np.float32)
    x[0] *= np.float32(2.0) ** r.integers(-40, 30, N).astype(np.float32)
    x[1] = 0
    out = torch.full(((B - 1) * ms + M,), 7.0, device="cuda")
    g = lambda a: torch.from_numpy(a).cuda()
    L.ops.matmul_int8_batch(out, g(w), g(s), g(x), M, N, B, ms)
    got = out.cpu().numpy()
    pad = -N % 128
    gm = np.abs(np.pad(x, ((0, 0), (0, pad)))).reshape(B, -1, 128).max(2).repeat(128, 1)[:, :N].astype(np.float64)
    for b in range(B):
        y = got[b * ms:b * ms + M].astype(np.float64)
        want = (w.astype(np.float64) @ x[b].astype(np.float64)) * s
        bound = 2.0 ** -24 * (N / 1024 + 13) * (np.abs(w.astype(np.float64)) @ gm[b]) * s
        assert (np.abs(y - want) <= bound).all()
        assert (got[b * ms + M:(b + 1) * ms] == 7.0).all()
    # Inf and NaN stay in their own column and come out as in an fp32 sum
    x[0, N // 2], x[B - 1, N - 1] = np.inf, np.nan
    clean = got.copy()
    L.ops.matmul_int8_batch(out, g(w), g(s), g(x), M, N, B, ms)
    got = out.cpu().numpy()
    y, wm = got[:M], w[:, N // 2]
    assert (y[wm > 0] == np.inf).all() and (y[wm < 0] == -np.inf).all() and np.isnan(y[wm == 0]).all()
    assert np.isnan(got[(B - 1) * ms:]).all()
    np.testing.assert_array_equal(got[ms:(B - 1) * ms], clean[ms:(B - 1) * ms])


def _int8_batch(w, s, x, ms=None):
    import torch
    import libinferbit_amd as L
    L.ops.init(0)
    B, N = x.shape
    M = w.shape[0]
    out = torch.empty(B * M, device="cuda")
    g = lambda a: torch.from_numpy(a).cuda()
    L.ops.matmul_int8_batch(out, g(w), g(s), g(x), M, N, B, M)
    return out.cpu().numpy().reshape(B, M).astype(np.float64)


# one column and several; rows on both sides of the split over row tiles
@pytest.mark.parametrize("M,N,B", [(4096, 4096, 1), (100, 14336, 1), (300, 2048, 2), (4112, 1040, 8), (64, 8192, 32)])
def test_int8_batch_small_beside_large(M, N, B):
    """An element far below its group's largest keeps its bits: rows whose
    weights on the large channels are 0, against float64.  A group's x is held
    to 2^-29 of its largest (30 bits and sign, truncated); its integer sum is
    rounded twice and each fp32 partial sum once (N / 1024 + 8 of them) to
    2^-24, the row scale once more."""
    print(f"case int8 range M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(-127, 128, (M, N), dtype=np.int8)
    s = (r.random(M) * 0.01 + 1e-4).astype(np.float32)
    x = r.standard_normal((B, N)).astype(np.float32)
    big = r.random(N) < 1 / 128
    x[:, big] *= np.float32(2.0 ** 14)
    w[: M // 2, big] = 0
    got = _int8_batch(w, s, x)
    gm = np.abs(np.pad(x, ((0, 0), (0, -N % 128)))).reshape(B, -1, 128).max(2).repeat(128, 1)[:, :N].astype(np.float64)
    a = np.abs(w.astype(np.float64))
    for b in range(B):
        want = (w.astype(np.float64) @ x[b].astype(np.float64)) * s
        bound = (2.0 ** -29 * (a @ gm[b]) + 2.0 ** -24 * (N / 1024 + 12) * (a @ np.abs(x[b]).astype(np.float64))) * s
        assert (np.abs(got[b] - want) <= bound).all()


# two to four columns on either side of the rows and lengths where the vector
# form hands over to the digits
@pytest.mark.parametrize("M,N,B", [(1024, 4096, 3), (1025, 4096, 3), (1024, 2064, 4), (256, 4112, 4), (257, 4112, 4),
                                   (256, 4096, 4), (2049, 1024, 2), (2049, 1040, 2), (3, 14336, 3)])
def test_int8_batch_few_columns(M, N, B):
    """Both forms against float64: a lane's chain of N / 64 products, rounded
    up, and six folds, each to 2^-24 of its partial sum (the digits' bound is
    smaller), the row scale once more."""
    print(f"case int8 few columns M={M} N={N} B={B}", flush=True)
    r = np.random.default_rng(M + N + B)
    w = r.integers(-128, 128, (M, N), dtype=np.int8)
    s = (r.random(M) * 0.01 + 1e-4).astype(np.float32)
    x = r.standard_normal((B, N)).astype(np.float32)
    got = _int8_batch(w, s, x)
    for b in range(B):
        want = (w.astype(np.float64) @ x[b].astype(np.float64)) * s
        bound = 2.0 ** -24 * (N / 64 + 16 + 7) * (np.abs(w.astype(np.float64)) @ np.abs(x[b]).astype(np.float64)) * s
        assert (np.abs(got[b] - want) <= bound).all()


def test_int8_batch_tiny_x():
    """Groups of subnormal and just normal numbers, exactly held."""
    r = np.random.default_rng(5)
    w = r.integers(-127, 128, (40, 512), dtype=np.int8)
    x = (r.integers(-(1 << 22), 1 << 22, (3, 512)) * 2.0 ** -149).astype(np.float32)
    got = _int8_batch(w, np.ones(40, np.float32), x)
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    assert (np.abs(got - want) <= 2.0 ** -24 * 8 * (np.abs(x).astype(np.float64) @ np.abs(w.T.astype(np.float64)))).all()


def test_int8_batch_long_rows():
    """Columns whose offsets pass 32 bits of bytes together."""
    import torch
    import libinferbit_amd as L
    L.ops.init(0)
    M, N, B = 2, (1 << 25) + 16, 32
    print(f"case int8 long rows N={N} B={B}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    w = torch.randint(-127, 128, (M, N), dtype=torch.int8, device="cuda", generator=g)
    x = torch.randn(B, N, device="cuda", generator=g)
    out = torch.empty(B, M, device="cuda")
    L.ops.matmul_int8_batch(out, w, torch.ones(M, device="cuda"), x, M, N, B, M)
    for b in range(B):
        want = (w.double() * x[b].double()).sum(1)
        # sums of 2^25 / 1024 + 8 fp32 steps in 8 wavefronts, each within 2^-24 of the partial sum
        assert ((out[b].double() - want).abs() <= 2.0 ** -24 * N / 128 * 8 * want.abs().clamp(min=73 * N ** 0.5)).all()


@pytest.mark.parametrize("keep", [0.5, 0.9])                  # the sparse row path, and above its limit of 80 %
@pytest.mark.parametrize("bits", [None, dict(gate_proj=8, up_proj=8, down_proj=8)])
def test_prompt_with_sparsity_masks(tmp_path, keep, bits):
    """Prompts through layers with a sparsity mask: the logits, the cache and
    what follows of single steps, bit for bit, and other ones than unmasked."""
    from libinferbit_amd import ibf
    from libinferbit_amd.model import Model
    cfg = dict(ibf.TINYLLAMA, num_layers=2, hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64,
               intermediate_size=512, vocab_size=1000, max_context_length=200, kv_bits=8)
    path = str(tmp_path / "m.ibf")
    ibf.write_synthetic(path, cfg, seed=31, bits=bits)
    plain = Model(path)
    _add_masks(path, 512, keep)
    one, many = Model(path), Model(path)
    toks = np.random.default_rng(7).integers(0, 1000, 60).astype(np.int32)
    print(f"case prompt mask {keep} {bits}", flush=True)
    at = 0
    for n in (7, 33):
        for t in toks[at:at + n]:
            a = one.forward([t])
        b = many.forward(toks[at:at + n])
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
        assert not np.array_equal(plain.forward(toks[at:at + n]), b)
        at += n
    np.testing.assert_array_equal(one.forward_positions(toks[:5]).view(np.uint32),
                                  many.forward_positions(toks[:5]).view(np.uint32))


@pytest.mark.parametrize("w4a8", [False, True])
@pytest.mark.parametrize("name", ["int8kv", "all_int8", "all_int4", "mixed_qkv"])
def test_fast_prompt_near_single_steps(tmp_path, monkeypatch, name, w4a8):
    """Fast mode: a prompt's projections run on the batch kernels, so its
    logits differ from single steps by fp32 rounding (1e-4 of the largest, as
    fast and exact mode do), and with int8 activation codes by the codes that
    such rounding moves by one (up to 1/127 of a group's largest, a few in a
    thousand: 2e-2 at this width)."""
    from libinferbit_amd import ibf
    from libinferbit_amd.model import Model
    monkeypatch.setenv("IB_W4A8", "1" if w4a8 else "0")
    spec = dict(PROMPT_MODELS[name])
    bits = spec.pop("bits", None)
    cfg = dict(ibf.TINYLLAMA, num_layers=2, hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64,
               intermediate_size=512, vocab_size=1000, max_context_length=200)
    cfg.update(spec)
    path = str(tmp_path / "m.ibf")
    ibf.write_synthetic(path, cfg, seed=31, bits=bits)
    one, many = Model(path), Model(path)
    one.set_exact(False)
    many.set_exact(False)
    toks = np.random.default_rng(7).integers(0, 1000, 60).astype(np.int32)
    print(f"case fast prompt {name} w4a8={w4a8}", flush=True)
    at = 0
    for n in (3, 33, 16):
        for t in toks[at:at + n]:
            a = one.forward([t])
        b = many.forward(toks[at:at + n])
        d = np.abs(a.astype(np.float64) - b).max() / np.abs(a).max()
        print(f"  {n}: {d:.2e}", flush=True)
        assert d <= (2e-2 if w4a8 else 1e-4)
        at += n


# decoders of real widths, whose launches take the forms of many row blocks: 8
# slots a block of the fused INT8 chains (40 row blocks and more), the W4A8 fold
# handed on between wavefronts, and columns that do not fit LDS
@pytest.mark.parametrize("I,bits", [(5632, None), (5600, None), (5600, dict(o_proj=8, gate_proj=8, up_proj=8, down_proj=8))])
def test_wide_prompt_equals_single_steps(tmp_path, I, bits):
    from libinferbit_amd import ibf
    from libinferbit_amd.model import Model
    cfg = dict(ibf.TINYLLAMA, num_layers=2, intermediate_size=I, vocab_size=1000, max_context_length=200)
    path = str(tmp_path / "m.ibf")
    ibf.write_synthetic(path, cfg, seed=31, bits=bits)
    toks = np.random.default_rng(7).integers(0, 1000, 100).astype(np.int32)
    one, many = Model(path), Model(path)
    at = 0
    for n in (32, 25, 31, 7):
        print(f"case wide prompt {I} {bits} {at}+{n}", flush=True)
        for t in toks[at:at + n]:
            a = one.forward([t])
        b = many.forward(toks[at:at + n])
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
        at += n
    np.testing.assert_array_equal(one.forward_positions(toks[:5]).view(np.uint32),
                                  many.forward_positions(toks[:5]).view(np.uint32))


class _Mat(C.Structure):                                       # MatDesc (ibh_common.h)
    _fields_ = [("out", C.c_void_p), ("w", C.c_void_p), ("s", C.c_void_p), ("M", C.c_int)]


def _internal(name, *args):
    """A C++ launcher of the library that only its own files call."""
    import libinferbit_amd as L
    f = getattr(L.lib(), name)
    f.restype, f.argtypes = C.c_int, args
    return f


# rows of 1 to 3 matrices, columns, slots: partial row blocks, 4 and 8 slots a
# block with a remainder, a last tile of 16 columns
@pytest.mark.parametrize("Ms,N,B", [((2000, 300, 260), 2048, 31), ((2000, 300, 260), 272, 7), ((2560,), 1040, 25),
                                    ((4100,), 400, 17), ((70, 64), 16, 3), ((1,), 144, 1)])
def test_fused_int8_chains_bit_exact(table, Ms, N, B):
    """The prompt's INT8 products against the one-vector exact kernel, bit for
    bit: normal numbers, subnormal ones, and sums that cancel to nothing."""
    import torch

    import libinferbit_amd as L
    launch = _internal("_Z27ibh_launch_int8_batch_exactPKN3ibh7MatDescEiiPKfiibP12ihipStream_ti", C.c_void_p, C.c_int,
                       C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_bool, C.c_void_p, C.c_int)
    r = np.random.default_rng(sum(Ms) + N + B)
    ws = [r.integers(-127, 128, (M, N), dtype=np.int8) for M in Ms]
    ss = [(r.random(M) * 0.01 + 1e-4).astype(np.float32) for M in Ms]
    x = r.standard_normal((B, N)).astype(np.float32)
    x[B // 3] *= np.float32(2.0) ** -135                       # products and sums subnormal or lost
    x[2 * B // 3] *= np.float32(2.0) ** r.integers(-149, 100, N).astype(np.float32)
    h = N // 32 * 16
    for w in ws:                                               # a chain's second half takes its first away again
        w[::2, h:2 * h] = -w[::2, :h]
    x[B - 1, h:2 * h] = x[B - 1, :h]
    dw = [torch.from_numpy(w).cuda() for w in ws]
    ds = [torch.from_numpy(s).cuda() for s in ss]
    dx = torch.from_numpy(x).cuda()
    out = [torch.full((B, M), 7.0, device="cuda") for M in Ms]
    d = (_Mat * len(Ms))(*[_Mat(o.data_ptr(), w.data_ptr(), s.data_ptr(), M) for o, w, s, M in zip(out, dw, ds, Ms)])
    print(f"case fused chains {Ms} N={N} B={B}", flush=True)
    assert launch(C.addressof(d), len(Ms), 1, dx.data_ptr(), N, B, True, torch.cuda.current_stream().cuda_stream, 0) == 0
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    for o, w, s, M in zip(out, ws, ss, Ms):
        got = o.cpu().numpy()
        for b in range(B):
            want = np.empty(M, np.float32)
            table["matmul_int8"](p(want), p(w), p(s), p(np.ascontiguousarray(x[b])), M, N)
            np.testing.assert_array_equal(got[b].view(np.uint32), want.view(np.uint32))


# the fused fold handed on (tall), gathered, with codes from L2, and rows that
# end inside a group; 2 matrices in a launch
@pytest.mark.parametrize("Ms,N,B", [((8200,), 4096, 9), ((8200,), 4096, 17), ((5632, 5632), 2048, 32), ((2048,), 5632, 31),
                                    ((1000, 500), 6176, 20), ((500,), 2080, 9), ((40,), 64, 17), ((1003,), 2048, 16)])
def test_fused_w4a8_columns_bit_exact(Ms, N, B):
    """The prompt's W4A8 products against the one-vector product, bit for bit."""
    import torch

    import libinferbit_amd as L
    L.ops.init(0)
    launch = _internal("_Z21ibh_launch_w4a8_batchPKN3ibh7MatDescEiiPKaPKfiibP12ihipStream_ti", C.c_void_p, C.c_int, C.c_int,
                       C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_bool, C.c_void_p, C.c_int)
    r = np.random.default_rng(sum(Ms) + N + B)
    g = lambda a: torch.from_numpy(a).cuda()
    dw = [g(r.integers(0, 256, (M, N // 2), dtype=np.uint8)) for M in Ms]
    ds = [g((r.random(M) * 0.01 + 1e-3).astype(np.float16)) for M in Ms]
    q = g(r.integers(-127, 128, (B, N), dtype=np.int8))
    sa = g((r.random((B, (N + 127) // 128)) * 0.02 + 1e-3).astype(np.float32))
    out = [torch.full((B, M), 7.0, device="cuda") for M in Ms]
    d = (_Mat * len(Ms))(*[_Mat(o.data_ptr(), w.data_ptr(), s.data_ptr(), M) for o, w, s, M in zip(out, dw, ds, Ms)])
    print(f"case fused w4a8 {Ms} N={N} B={B}", flush=True)
    assert launch(C.addressof(d), len(Ms), 0, q.data_ptr(), sa.data_ptr(), N, B, True,
                  torch.cuda.current_stream().cuda_stream, 0) == 1
    for o, w, s, M in zip(out, dw, ds, Ms):
        y = torch.empty(M, device="cuda")
        for b in range(B):
            L.ops.parallel_matmul_w4a8(y, w, s, q[b].contiguous(), sa[b].contiguous(), M, N)
            assert torch.equal(o[b].view(torch.int32), y.view(torch.int32))
