"""GPU parity of the PQ LUT matvec against the reference-written golden
vectors and the oracle.  The chunk sum is associated differently from the
CPU's serial loop: bar max|y_gpu - y_cpu| / max|y_cpu| <= 1e-4."""
import numpy as np
import pytest
import torch

from conftest import load_golden, pq_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import libinferbit_amd as L
    L.ops.init(0)
    return L.ops


def run(ops, t, x):
    d = ops.PqDeviceTensor(t)
    out = torch.empty(t["M"], device="cuda")
    d.matmul(torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda(), out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def relerr(a, b):
    return float(np.abs(a.astype(np.float64) - b).max() / np.abs(b).max())


@pytest.mark.parametrize("name", ["l1", "l2p16", "l2u8", "l2u16", "out8", "out40"])
def test_pq_golden(ops, name):
    print(f"case pq {name}", flush=True)
    t = pq_case(load_golden("pq.npz"), name)
    assert relerr(run(ops, t, t["x"]), t["y"]) <= 1e-4
    assert relerr(run(ops, t, t["xs"]), t["ys"]) <= 1e-4       # chunk-skipping case


def test_pq_mistral_ffn_shape(ops, oracle_lib):
    """M=4096, N=14336, G=16, K=256, one level, no outliers."""
    from gen_golden import make_pq
    rng = np.random.default_rng(5)
    t = make_pq(rng, 4096, 896, 16, 256, 1, 0, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    assert relerr(run(ops, t, x), oracle_lib.pq_matmul(t, x)) <= 1e-4


def test_pq_zero_input(ops, oracle_lib):
    from gen_golden import make_pq
    t = make_pq(np.random.default_rng(1), 64, 16, 16, 256, 1, 0, 8)
    x = np.zeros(t["N"], np.float32)
    np.testing.assert_array_equal(run(ops, t, x), oracle_lib.pq_matmul(t, x))


def run_streaming(ops, t, x):
    d = ops.PqDeviceTensor(t)
    out = torch.empty(t["M"], device="cuda")
    d.matmul_streaming(torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda(), out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("name", ["l1", "l2p16", "l2u8", "l2u16", "out8", "out40", "g4", "g32", "g4l2"])
def test_pq_streaming_golden(ops, name):
    """ib_pq_matmul_fp32_streaming_cached (the PQ session's default): no chunk skipping."""
    print(f"case pq streaming {name}", flush=True)
    d = load_golden("pqs.npz")
    src = d if f"{name}.M" in d.files else load_golden("pq.npz")
    t = pq_case(src, name)
    assert relerr(run_streaming(ops, t, t["x"]), d[f"{name}.y"]) <= 1e-4
    if f"{name}.ys" in d.files:
        assert relerr(run_streaming(ops, t, t["xs"]), d[f"{name}.ys"]) <= 1e-4


def test_pq_streaming_mistral_shape(ops, oracle_lib):
    from gen_golden import make_pq
    rng = np.random.default_rng(6)
    t = make_pq(rng, 4096, 896, 16, 256, 1, 0, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    x[: t["N"] // 3] *= 1e-3
    assert relerr(run_streaming(ops, t, x), oracle_lib.pq_matmul_streaming(t, x)) <= 1e-4


def test_pq_streaming_rejects_wide_chunks(ops):
    from gen_golden import make_pq
    from libinferbit_amd import IbhError
    t = make_pq(np.random.default_rng(1), 16, 4, 64, 16, 1, 0, 0)
    with pytest.raises(IbhError):
        run_streaming(ops, t, np.zeros(t["N"], np.float32))


def run_q8lut(ops, t, x):
    d = ops.PqDeviceTensor(t)
    out = torch.empty(t["M"], device="cuda")
    d.matmul_q8lut(torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda(), out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("name", ["l1", "l2", "out8", "out40l2", "g4", "g32", "g6"])
def test_pq_q8lut_golden(ops, name):
    """ib_pq_matmul_fp32_q8lut: the int8 codes equal the reference's, the
    gather sums in another order."""
    print(f"case pq q8lut {name}", flush=True)
    d = load_golden("pqq8.npz")
    t = pq_case(d, name)
    assert relerr(run_q8lut(ops, t, t["x"]), d[f"{name}.y"]) <= 1e-4


def test_pq_q8lut_mistral_shape(ops, oracle_lib):
    from gen_golden import make_pq
    rng = np.random.default_rng(61)
    t = make_pq(rng, 4096, 896, 16, 256, 2, 256, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    assert relerr(run_q8lut(ops, t, x), oracle_lib.pq_matmul_q8lut(t, x)) <= 1e-4


def test_pq_q8lut_rejects_unreadable_level2(ops):
    from gen_golden import make_pq
    from libinferbit_amd import IbhError
    t = make_pq(np.random.default_rng(2), 16, 4, 16, 64, 2, 256, 0)     # K_l2 != K
    with pytest.raises(IbhError):
        run_q8lut(ops, t, np.zeros(t["N"], np.float32))


PQV_NAMES = ["l1", "l2p16", "l2u8", "l2u16", "out8", "out40", "pyr16", "pyr8"]
PQV_POLICIES = {"l1only": (1, 0.0, 0.0), "l2skip05": (2, 0.5, 0.0), "l2skip5": (2, 5.0, 0.0),
                "sparse": (3, 0.0, 1e-2), "int8": (4, 0.0, 0.0)}


def run_policy(ops, t, x, v, st, at):
    d = ops.PqDeviceTensor(t)
    out = torch.empty(t["M"], device="cuda")
    d.matmul_policy(torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda(), out, v, st, at)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("name", PQV_NAMES)
@pytest.mark.parametrize("pol", list(PQV_POLICIES))
def test_pq_policy_golden(ops, name, pol):
    """The PQ session's policy variants against the reference's outputs."""
    print(f"case pq policy {name} {pol}", flush=True)
    d = load_golden("pqv.npz")
    src = d if f"{name}.M" in d.files else load_golden("pq.npz")
    t = pq_case(src, name)
    v, st, at = PQV_POLICIES[pol]
    assert relerr(run_policy(ops, t, t["x"], v, st, at), d[f"{name}.{pol}.y"]) <= 1e-4
    assert relerr(run_policy(ops, t, t["xs"], v, st, at), d[f"{name}.{pol}.ys"]) <= 1e-4


@pytest.mark.parametrize("v,st,at", [(1, 0, 0), (2, 0.5, 0), (3, 0, 1e-3), (4, 0, 0)])
def test_pq_policy_mistral_shape(ops, oracle_lib, v, st, at):
    from gen_golden import make_pq
    print(f"case pq policy mistral v={v}", flush=True)
    rng = np.random.default_rng(8)
    t = make_pq(rng, 4096, 896, 16, 256, 2, 256, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    x[: t["N"] // 3] *= 1e-4
    assert relerr(run_policy(ops, t, x, v, st, at), oracle_lib.pq_matmul_variant(t, x, v, st, at)) <= 1e-4


@pytest.mark.parametrize("name,k", [("head1", 1), ("head1", 8), ("head1", 40), ("head2", 3), ("head2", 64),
                                    ("small", 12)])
def test_pq_lm_head_topk_golden(ops, name, k):
    print(f"case pq topk {name} k={k}", flush=True)
    d = load_golden("pqtopk.npz")
    t = pq_case(d, name)
    lg, ids = ops.PqDeviceTensor(t).lm_head_topk(torch.from_numpy(t["x"]).cuda(), k)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(ids.cpu().numpy(), d[f"{name}.k{k}.ids"])
    want = d[f"{name}.k{k}.logits"]
    assert float(np.abs(lg.cpu().numpy().astype(np.float64) - want).max() / np.abs(want).max()) <= 1e-4


def test_pq_lm_head_topk_vocab_shape(ops, oracle_lib):
    """A 32000-row head (Llama vocabulary) over hidden 4096, two levels."""
    from gen_golden import make_pq
    rng = np.random.default_rng(12)
    t = make_pq(rng, 32000, 256, 16, 256, 2, 256, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    want_lg, want_ids = oracle_lib.pq_lm_head_topk(t, x, 50)
    lg, ids = ops.PqDeviceTensor(t).lm_head_topk(torch.from_numpy(x).cuda(), 50)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(ids.cpu().numpy(), want_ids)
    assert float(np.abs(lg.cpu().numpy().astype(np.float64) - want_lg).max() / np.abs(want_lg).max()) <= 1e-4


@pytest.mark.parametrize("k", [1, 8, 16, 17])
def test_pq_lm_head_topk_two_pass(ops, oracle_lib, k):
    """Heads of 4096 rows and more with K <= 16 select in two passes (each
    block of 1024 rows keeps its K best, then one block selects among the
    candidates); K = 17 takes the one-pass select.  Ids equal the oracle's,
    also with many exactly tied rows (duplicated index rows)."""
    from gen_golden import make_pq
    rng = np.random.default_rng(100 + k)
    t = make_pq(rng, 32000, 64, 16, 64, 1, 0, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    d = ops.PqDeviceTensor(t)
    want_lg, want_ids = oracle_lib.pq_lm_head_topk(t, x, k)
    lg, ids = d.lm_head_topk(torch.from_numpy(x).cuda(), k)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(ids.cpu().numpy(), want_ids)
    assert float(np.abs(lg.cpu().numpy().astype(np.float64) - want_lg).max() / np.abs(want_lg).max()) <= 1e-4
    # ties: the best row copied into rows spread over several blocks
    best = int(want_ids[0])
    t2 = dict(t)
    for key in ("i1l", "i1r"):
        a = np.array(t[key])
        for r in (5, 3000, 17001, 31999):
            a[r] = a[best]
        t2[key] = a
    rs = np.array(t["row_scale"])
    for r in (5, 3000, 17001, 31999):
        rs[r] = rs[best]
    t2["row_scale"] = rs
    want_lg2, want_ids2 = oracle_lib.pq_lm_head_topk(t2, x, k)
    lg2, ids2 = ops.PqDeviceTensor(t2).lm_head_topk(torch.from_numpy(x).cuda(), k)
    torch.cuda.synchronize()
    got = ids2.cpu().numpy()
    # equal refined logits: the oracle keeps the reference's heap order, the
    # GPU row order; compare as sets per equal value and the values exactly
    assert sorted(got.tolist()) == sorted(want_ids2.tolist())
    assert float(np.abs(lg2.cpu().numpy().astype(np.float64) - want_lg2).max() / np.abs(want_lg2).max()) <= 1e-4


@pytest.mark.parametrize("heavy", [False, True])
@pytest.mark.parametrize("shape", [(4096, 896, 16, 256, 0), (300, 130, 16, 256, 0), (1000, 64, 8, 128, 40),
                                   (257, 200, 4, 64, 8), (513, 97, 16, 256, 33)])
def test_pq_one_launch_matches_three_kernels(ops, oracle_lib, shape, heavy):
    """The one-launch kernel (tables on the matrix cores, per-row fixed-point
    words) against the three-kernel path and the oracle, on ragged row
    tiles and slabs, with and without outliers, x N(0,1) and heavy-tailed
    (Student t, 1.5 dof: the fixed-point scale follows max|x|); each call
    twice, so the words' reset between calls is exercised."""
    from gen_golden import make_pq
    M, C, G, K, no = shape
    print(f"case pq one-launch {shape} heavy={heavy}", flush=True)
    rng = np.random.default_rng(M + C)
    t = make_pq(rng, M, C, G, K, 1, 0, no)
    x = (rng.standard_t(1.5, t["N"]) if heavy else rng.standard_normal(t["N"])).astype(np.float32)
    ref = oracle_lib.pq_matmul(t, x)
    lib = ops.lib()
    try:
        lib.ibh_pq_set_fused(0)
        three = run(ops, t, x)
    finally:
        lib.ibh_pq_set_fused(1)
    one = run(ops, t, x)
    again = run(ops, t, x)
    np.testing.assert_array_equal(one, again)
    assert relerr(one, ref) <= 1e-4
    assert relerr(one, three) <= 1e-5


def test_pq_one_launch_nonfinite_x(ops, oracle_lib):
    """A non-finite x on the one-launch path: every row NaN (the CPU gives
    +-Inf or NaN there), and the next finite call is right again."""
    from gen_golden import make_pq
    rng = np.random.default_rng(11)
    t = make_pq(rng, 4096, 896, 16, 256, 1, 0, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    for bad in (np.inf, np.nan):
        xb = x.copy()
        xb[123] = bad
        y = run(ops, t, xb)
        assert np.isnan(y).all()
        assert not np.isfinite(oracle_lib.pq_matmul(t, xb)).all()
    assert relerr(run(ops, t, x), oracle_lib.pq_matmul(t, x)) <= 1e-4


def test_pq_workspace_needs_stamp(ops, oracle_lib):
    """A caller workspace that ibh_pq_workspace_init did not prepare: NaN rows
    and IBH_DEVERR_PQ_WS, never a silent sum into unknown words; prepared,
    the same memory gives the right result."""
    import ctypes
    from gen_golden import make_pq
    rng = np.random.default_rng(12)
    t = make_pq(rng, 4096, 896, 16, 256, 1, 0, 0)
    x = rng.standard_normal(t["N"]).astype(np.float32)
    d = ops.PqDeviceTensor(t)
    lib = ops.lib()
    assert lib.ibh_device_errors(1) == 0
    ws = torch.full((d.ws.numel(),), 7, dtype=torch.uint8, device="cuda")   # garbage, no stamp
    xd = torch.from_numpy(x).cuda()
    out = torch.empty(t["M"], device="cuda")
    assert lib.ibh_pq_matmul(ctypes.byref(d.s), xd.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), None) == 0
    torch.cuda.synchronize()
    assert torch.isnan(out).all()
    assert lib.ibh_device_errors(1) == 2
    assert lib.ibh_device_errors(0) == 0
    assert lib.ibh_pq_workspace_init(ws.data_ptr(), ws.numel(), None) == 0
    assert lib.ibh_pq_matmul(ctypes.byref(d.s), xd.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), None) == 0
    torch.cuda.synchronize()
    assert relerr(out.cpu().numpy(), oracle_lib.pq_matmul(t, x)) <= 1e-4
    assert lib.ibh_device_errors(0) == 0


def _fused(ops, on):
    import libinferbit_amd as L
    L.lib().ibh_pq_set_fused(int(on))


# M, C, G, K, K2, outliers: whole and partial row tiles and slabs, odd chunk
# counts (byte-wise indices), packed 4-bit and byte level-2 indices, codebooks
# that are not whole 32-code tiles, short half-chunks, both outlier rules
TWO_LEVEL = [(512, 32, 16, 256, 256, 0), (700, 33, 16, 256, 256, 8), (1, 1, 16, 256, 16, 0), (513, 95, 16, 256, 16, 40),
             (300, 64, 16, 256, 64, 0), (1025, 160, 16, 100, 100, 0), (257, 48, 8, 64, 16, 4), (100, 31, 6, 16, 16, 0),
             (64, 896, 16, 256, 256, 128), (600, 64, 4, 33, 256, 0), (4700, 864, 4, 16, 16, 4)]


@pytest.mark.parametrize("M,C,G,K,K2,no", TWO_LEVEL)
def test_two_level_one_launch_matches_three(ops, M, C, G, K, K2, no):
    """The one-launch kernel on two-level tensors against the three-kernel
    path: every chunk rule, and non-finite x value for value."""
    from gen_golden import make_pq
    t = make_pq(np.random.default_rng(M + C), M, C, G, K, 2, K2, no)
    d = ops.PqDeviceTensor(t)
    x = torch.randn(t["N"], generator=torch.Generator().manual_seed(C)) * 0.7
    x[torch.rand(t["N"], generator=torch.Generator().manual_seed(M)) < 0.3] *= 1e-4
    big = x.clone()
    big[: t["N"] // 2] *= 1e30
    inf, nan = x.clone(), x.clone()
    inf[t["N"] // 3] = float("inf")
    nan[t["N"] // 3] = float("nan")
    out = torch.empty(M, device="cuda")
    try:
        for name, v in (("plain", x), ("tiny", x * 1e-36), ("big", big), ("inf", inf), ("nan", nan)):
            for pol in (None, (0, 0.0, 0.0), (3, 0.0, 1e-2)):
                print(f"case two-level {M}x{C} G={G} K={K}/{K2} no={no} {name} {pol}", flush=True)
                got = []
                for on in (1, 0):
                    _fused(ops, on)
                    for _ in range(2):
                        if pol is None:
                            d.matmul(v.cuda(), out)
                        else:
                            d.matmul_policy(v.cuda(), out, *pol)
                    got.append(out.cpu().numpy().astype(np.float64))
                fin = np.isfinite(got[1])
                assert np.array_equal(fin, np.isfinite(got[0])) and np.array_equal(np.isnan(got[1]), np.isnan(got[0]))
                assert np.array_equal(got[0][~fin & ~np.isnan(got[1])], got[1][~fin & ~np.isnan(got[1])])
                if fin.any():
                    # fp32 sums of up to 2 * 2 * 896 terms in two orders
                    assert np.abs(got[0] - got[1])[fin].max() <= 2e-6 * max(np.abs(got[1][fin]).max(), 1e-37)
    finally:
        _fused(ops, 1)


@pytest.mark.parametrize("M,k", [(256, 256), (300, 50), (1025, 256), (1024, 1), (33000, 8), (33000, 256), (2000, 257)])
def test_pq_lm_head_topk_pick(ops, oracle_lib, M, k):
    """The candidate selection at the edges of a thread's share, of the
    one-read span (32768) and of its K limit; all logits equal (lowest rows)."""
    from gen_golden import make_pq
    print(f"case topk pick M={M} k={k}", flush=True)
    t = make_pq(np.random.default_rng(M + k), M, 24, 16, 256, 2, 64, 0)
    x = np.random.default_rng(k).standard_normal(t["N"]).astype(np.float32)
    d = ops.PqDeviceTensor(t)
    lg, ids = d.lm_head_topk(torch.from_numpy(x).cuda(), k)
    want_lg, want_ids = oracle_lib.pq_lm_head_topk(t, x, k)
    got = ids.cpu().numpy()
    # the rows selected are the same; two may change places only where their
    # logits are closer than the rounding of two fp32 sums of 24 * 32 terms
    # (2 * sqrt(768) * 2^-24 of the largest)
    np.testing.assert_array_equal(np.sort(got), np.sort(want_ids))
    by_row = dict(zip(want_ids.tolist(), want_lg.tolist()))
    moved = got != want_ids
    assert np.abs(np.array([by_row[i] for i in got[moved].tolist()]) - want_lg[moved]).max(initial=0) \
        <= 2 * 768 ** 0.5 * 2.0 ** -24 * np.abs(want_lg).max()
    assert relerr(lg.cpu().numpy(), want_lg) <= 1e-5
    lg, ids = d.lm_head_topk(torch.zeros(t["N"], device="cuda"), k)
    np.testing.assert_array_equal(ids.cpu().numpy(), np.arange(k))


def test_two_level_unprepared_workspace(ops):
    """Two-level calls on a workspace that ibh_pq_workspace_init did not
    prepare keep giving the product (they never needed the row words)."""
    import ctypes

    import libinferbit_amd as L
    from gen_golden import make_pq
    t = make_pq(np.random.default_rng(77), 300, 70, 16, 256, 2, 64, 8)
    d = ops.PqDeviceTensor(t)
    x = torch.randn(t["N"], generator=torch.Generator().manual_seed(3)).cuda()
    want, out = torch.empty(300, device="cuda"), torch.empty(300, device="cuda")
    d.matmul(x, want)
    ws = torch.full((d.ws.numel(),), 0x5A, dtype=torch.uint8, device="cuda")
    L._lib.check(L.lib().ibh_pq_matmul(ctypes.byref(d.s), x.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(),
                                       torch.cuda.current_stream().cuda_stream), "ibh_pq_matmul")
    assert relerr(out.cpu().numpy(), want.cpu().numpy()) <= 2e-6   # two orders of the same fp32 terms


@pytest.mark.parametrize("book", ["cb1l", "cb1r", "cb2l", "cb2r"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("M,C,K2", [(600, 70, 256), (520, 96, 16)])
def test_two_level_nonfinite_codeword(ops, M, C, K2, book, bad):
    """A NaN or Inf codeword reaches the rows that use it, and no others, as in
    the three-kernel path; the workspace stays good for the next call."""
    from gen_golden import make_pq
    print(f"case two-level codeword {M}x{C} K2={K2} {book} {bad}", flush=True)
    t = make_pq(np.random.default_rng(M + K2), M, C, 16, 256, 2, K2, 0)
    if K2 == 16:
        for i in ("i2l", "i2r"):                      # packed codes: every other row does without code 3
            lo, hi = t[i][::2] & 15, t[i][::2] >> 4
            t[i][::2] = np.where(lo == 3, 4, lo) | np.where(hi == 3, 4, hi) << 4
    x = torch.randn(t["N"], generator=torch.Generator().manual_seed(C)).cuda()
    good = ops.PqDeviceTensor(t)
    cb = t[book].copy().view(np.float16).reshape(-1, 8)
    cb[3, 5] = bad
    d = ops.PqDeviceTensor({**t, book: cb.reshape(-1).view(np.uint16)})
    d.ws = good.ws
    out, want = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    good.matmul_streaming(x, want)
    clean = want.clone()
    try:
        _fused(ops, 0)
        d.matmul_streaming(x, want)
    finally:
        _fused(ops, 1)
    for _ in range(2):
        d.matmul_streaming(x, out)
        g, w = out.cpu().numpy(), want.cpu().numpy()
        assert 0 < np.isfinite(w).sum() < M
        np.testing.assert_array_equal(np.isnan(g), np.isnan(w))
        np.testing.assert_array_equal(g[np.isinf(w)], w[np.isinf(w)])
        fin = np.isfinite(w)
        # fp32 sums of 4 * 96 entries in two orders
        assert np.abs(g - w)[fin].max() <= 2e-6 * np.abs(w[fin]).max()
    good.matmul_streaming(x, out)
    assert torch.equal(out, clean)


# fewer than 16 index bytes in all, and rows whose slabs hold 16-byte pieces
@pytest.mark.parametrize("M,C,K2", [(1, 1, 0), (3, 5, 256), (7, 1, 16), (200, 64, 0), (200, 64, 256), (200, 64, 16)])
def test_pq_operands_at_any_address(ops, oracle_lib, M, C, K2):
    """Indices at odd addresses, codebooks at 2-byte and x at 4-byte ones: the
    same rows as from aligned operands, and those the oracle's."""
    from gen_golden import make_pq
    print(f"case pq addresses {M}x{C} K2={K2}", flush=True)
    t = make_pq(np.random.default_rng(M + C), M, C, 16, 256, 2 if K2 else 1, K2, 0)
    x = np.random.default_rng(C).standard_normal(t["N"]).astype(np.float32)
    d, e = ops.PqDeviceTensor(t), ops.PqDeviceTensor(t)
    for k, f in ops.PqDeviceTensor._MAP.items():
        if t.get(k) is None:
            continue
        raw = np.ascontiguousarray(t[k]).view(np.uint8).reshape(-1)
        off = t[k].dtype.itemsize
        b = torch.zeros(raw.size + off, dtype=torch.uint8, device="cuda")
        b[off:] = torch.from_numpy(raw.copy()).cuda()
        e.keep.append(b)
        setattr(e.s, f, b.data_ptr() + off)
    xb = torch.zeros(t["N"] + 1, device="cuda")
    xb[1:] = torch.from_numpy(x).cuda()
    a, b = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    d.matmul(torch.from_numpy(x).cuda(), a)
    e.matmul(xb[1:], b)
    assert torch.equal(a, b)
    assert relerr(a.cpu().numpy(), oracle_lib.pq_matmul(t, x)) <= 1e-4


@pytest.mark.parametrize("M,C,G,K,K2,no", TWO_LEVEL + [(40, 2016, 16, 256, 256, 0), (1100, 700, 8, 64, 16, 8)])
def test_two_level_direct_rows(ops, M, C, G, K, K2, no):
    """The sums that need neither tables nor row words (a workspace that was
    not prepared, a non-finite or tiny x) are the three-kernel path's bit for bit."""
    import ctypes

    import libinferbit_amd as L
    from gen_golden import make_pq
    print(f"case two-level direct {M}x{C} G={G} K={K}/{K2} no={no}", flush=True)
    t = make_pq(np.random.default_rng(M + C), M, C, G, K, 2, K2, no)
    d = ops.PqDeviceTensor(t)
    x = torch.randn(t["N"], generator=torch.Generator().manual_seed(C))
    x[torch.rand(t["N"], generator=torch.Generator().manual_seed(M)) < 0.3] *= 1e-4
    inf = x.clone()
    inf[t["N"] // 3] = float("inf")
    tiny = x * 2.0 ** -127                    # rows and table entries are subnormal
    raw = torch.full((d.ws.numel(),), 0x5A, dtype=torch.uint8, device="cuda")
    out, want = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    for v, ws in ((x, raw), (inf, d.ws), (tiny, d.ws)):
        for skip in (True, False):
            v = v.cuda()
            try:
                _fused(ops, 0)
                d.matmul(v, want) if skip else d.matmul_streaming(v, want)
            finally:
                _fused(ops, 1)
            f = L.lib().ibh_pq_matmul if skip else L.lib().ibh_pq_matmul_streaming
            out.fill_(7.0)
            L._lib.check(f(ctypes.byref(d.s), v.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(),
                           torch.cuda.current_stream().cuda_stream), "two-level direct")
            if C > 32 or ws is d.ws:      # one slab needs no words: the tables serve it
                np.testing.assert_array_equal(out.cpu().numpy(), want.cpu().numpy())
            else:
                assert (out - want).abs().max() <= 2e-6 * want.abs().max()
    assert L.lib().ibh_device_errors(0) == 0


# a slab's last 16-byte pieces: whole, part-filled, reaching into the slab or
# row before, of odd rows whose packed codes start a half-byte later
@pytest.mark.parametrize("K2", [0, 16, 64])
@pytest.mark.parametrize("C", [15, 16, 17, 18, 30, 31, 32, 34, 47, 49, 63, 79, 94, 95])
def test_pq_ragged_chunk_counts(ops, oracle_lib, C, K2):
    from gen_golden import make_pq
    print(f"case pq ragged C={C} K2={K2}", flush=True)
    M = 70
    t = make_pq(np.random.default_rng(C + K2), M, C, 16, 256, 2 if K2 else 1, K2, 5)
    x = np.random.default_rng(C).standard_normal(t["N"]).astype(np.float32)
    x[:: 3] *= 1e-4
    d = ops.PqDeviceTensor(t)
    v = torch.from_numpy(x).cuda()
    a, b = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    for f in (d.matmul, d.matmul_streaming):
        f(v, a)
        try:
            _fused(ops, 0)
            f(v, b)
        finally:
            _fused(ops, 1)
        # fp32 sums of up to 4 * 95 entries in two orders, entries of 23 bits of x
        assert (a - b).abs().max() <= 1e-6 * b.abs().max()


# slabs of 32 chunks: the large channel's own, others, a ragged last one; x read
# as float4s (G = 16) and element by element (95 chunks of 6)
@pytest.mark.parametrize("M,C,G,K2", [(520, 96, 16, 0), (520, 96, 16, 16), (520, 96, 16, 256), (1100, 95, 6, 64),
                                      (300, 20, 16, 0)])
def test_pq_rows_without_the_large_channel(ops, M, C, G, K2):
    """A channel 2^32 times the others: rows whose codewords are 0 there keep
    the bits of the others."""
    from gen_golden import make_pq
    print(f"case pq large channel {M}x{C} G={G} K2={K2}", flush=True)
    K, hf, big = 256, G // 2, 3
    rng = np.random.default_rng(M + C + K2)
    t = make_pq(rng, M, C, G, K, 2 if K2 else 1, K2, 0)
    books = [("cb1l", "cb1r", "i1l", "i1r")] + ([("cb2l", "cb2r", "i2l", "i2r")] if K2 else [])
    x = rng.standard_normal(C * G).astype(np.float32)
    x[big * G + 1] = 2.0 ** 32
    want, size = np.zeros(M), np.zeros(M)
    for names in books:
        for side, (cb, ix) in enumerate(zip(names[:2], names[2:])):
            t[cb] = t[cb].copy()
            t[ix] = t[ix].copy()
            words = t[cb].reshape(-1, hf)
            words[0] = 0
            idx = t[ix].reshape(M, -1)
            if ix[1] == "2" and K2 == 16:
                codes = np.stack([idx & 15, idx >> 4], -1).reshape(M, -1)[:, :C]
                if side == 0:
                    idx[:, big // 2] &= 15                  # chunk 3: the high half
                    codes[:, big] = 0
            else:
                codes = idx
                if side == 0:
                    idx[:, big] = 0
            tab = np.einsum("kh,ch->ck", words.view(np.float16).astype(np.float64),
                            x.astype(np.float64).reshape(C, 2, hf)[:, side])
            terms = tab[np.arange(C)[None], codes]
            want += terms.sum(1)
            size += np.abs(np.einsum("kh,ch->ck", np.abs(words.view(np.float16).astype(np.float64)),
                                     np.abs(x.astype(np.float64)).reshape(C, 2, hf)[:, side])[np.arange(C)[None], codes]).sum(1)
    scale = t["row_scale"].view(np.float16).astype(np.float64)
    d = ops.PqDeviceTensor(t)
    out = torch.empty(M, device="cuda")
    d.matmul_streaming(torch.from_numpy(x).cuda(), out)
    got = out.cpu().numpy().astype(np.float64)
    # x to 2^-22 of each element (down to 2^-17 of its 8), chains of up to 16 + 16
    # fp32 adds of 2^-24 each
    assert (np.abs(got - want * scale) <= 2.0 ** -18 * size * np.abs(scale)).all()
