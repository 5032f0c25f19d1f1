"""The few-row MFMA matmul (csrc/skinny.hip) at the edges of its tiles, row counts and K splits, against the oracle.

Every (waves, tiles) choice of its dispatch is reached by the number of 16-row weight tiles per compute unit; the row counts
are the edges of the 16- and 32-row passes, K the fewest superblocks, an odd count and more superblocks than waves.  Q6_K
weights also start 2 bytes past a dword.  Bounds: assert_parity's (rel 1e-3 of the largest output; per element 1e-5 of the
sum of |terms|, what f32 reordering moves)."""
import numpy as np
import pytest

import oracle as O
import qmm
from helpers import acts, assert_parity, terms, weights

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a, pad=0):
    """The array's bytes on the GPU, `pad` bytes past an aligned start, nothing readable assumed behind them."""
    a = np.ascontiguousarray(a).reshape(-1).view(np.uint8)
    t = torch.zeros(a.size + pad, dtype=torch.uint8, device="cuda")
    t[pad:] = torch.from_numpy(a).cuda()
    return t[pad:]


def silu(v):
    v = np.asarray(v, np.float64)
    return v / (1.0 + np.exp(-v))


@pytest.fixture(scope="module")
def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("gtype", [O.Q4K, O.Q6K])
@pytest.mark.parametrize("per_cu,extra,k", [(0, 5, 2304), (0, 21, 256), (1, 3, 768), (2, 9, 256), (4, 17, 256),
                                            (6, 1, 256)])
def test_rows_over_tile_counts(gtype, per_cu, extra, k, cus):
    rng = np.random.default_rng(7000 + per_cu + k)
    n = 16 * per_cu * cus + extra
    wq = O.quantize(gtype, weights(rng, n, k))
    wd = dev(wq, 2 if gtype == O.Q6K else 0)
    for b in (3, 16, 17, 32):
        x = acts(rng, b, k)
        x[b - 1] = 0.0  # a row of zero blocks
        got = qmm.qmatmul_decode(gtype, wd, torch.from_numpy(x).cuda(), n).cpu().numpy()
        term = terms(gtype, x, wq, n) if n < 1000 else None
        assert_parity(got, O.matmul(gtype, x, wq, n), term, what=f"{gtype} n={n} k={k} b={b}")


@pytest.mark.parametrize("gtype", [O.Q4K, O.Q6K])
@pytest.mark.parametrize("per_cu,extra,k", [(0, 19, 1280), (3, 7, 256)])
def test_glu_rows_over_tile_counts(gtype, per_cu, extra, k, cus):
    """Gate and up start at different offsets within a dword (Q6_K)."""
    rng = np.random.default_rng(7100 + per_cu + k)
    n = 16 * per_cu * cus + extra
    g, u = (O.quantize(gtype, weights(rng, n, k)) for _ in range(2))
    gd, ud = dev(g, 2 if gtype == O.Q6K else 0), dev(u)
    for b in (3, 16, 17, 32):
        x = acts(rng, b, k)
        vy, kp = qmm.quantize_decode(gtype, torch.from_numpy(x).cuda())
        got = qmm.mmvq_fused_glu(gtype, gd, ud, vy, k, n, b, kp).cpu().numpy()
        want = silu(O.matmul(gtype, x, g, n)) * O.matmul(gtype, x, u, n)
        assert_parity(got, want, what=f"glu {gtype} n={n} k={k} b={b}")


ROWS16 = [O.Q8_0, O.Q4_0, O.Q5_0, O.Q5K]  # the types that take up to 16 rows


@pytest.mark.parametrize("gtype", ROWS16)
@pytest.mark.parametrize("per_cu,extra,k", [(0, 5, 2304), (0, 21, 256), (1, 3, 768), (2, 9, 256), (4, 17, 256)])
def test_sixteen_row_types_over_tile_counts(gtype, per_cu, extra, k, cus):
    """Both sides of the row counts from which the kernel takes over, weights that start on a dword only, and all output
    types (f16 / bf16 within their rounding of the f32 result)."""
    rng = np.random.default_rng(7400 + per_cu + k)
    n = 16 * per_cu * cus + extra
    wq = O.quantize(gtype, weights(rng, n, k))
    wd = dev(wq, 0 if gtype == O.Q5K else 4)
    for b in (3, 5, 9, 16):
        x = acts(rng, b, k)
        x[b - 1] = 0.0
        got = qmm.qmatmul_decode(gtype, wd, torch.from_numpy(x).cuda(), n)
        term = terms(gtype, x, wq, n) if n < 1000 else None
        assert_parity(got.cpu().numpy(), O.matmul(gtype, x, wq, n), term, what=f"{gtype} n={n} k={k} b={b}")
        vy, kp = qmm.quantize_decode(gtype, torch.from_numpy(x).cuda())
        for dt in (torch.float16, torch.bfloat16):
            assert torch.equal(qmm.mmvq(gtype, wd, vy, k, n, b, kp, out_dtype=dt), got.to(dt))


@pytest.mark.parametrize("gtype", ROWS16[:3])
@pytest.mark.parametrize("n,k", [(19, 1280), (4101, 256)])
def test_fused_forms_of_32_value_types(gtype, n, k):
    rng = np.random.default_rng(7500 + n)
    g, u, v = (O.quantize(gtype, weights(rng, n - 3 * i, k)) for i in range(3))
    for b in (2, 3, 5, 8, 16):
        x = acts(rng, b, k)
        vy, kp = qmm.quantize_decode(gtype, torch.from_numpy(x).cuda())
        n1 = n - 3  # the up rows past n1 are the next matrix's: not read
        got = qmm.mmvq_fused_glu(gtype, dev(g), dev(u), vy, k, n1, b, kp).cpu().numpy()
        want = silu(O.matmul(gtype, x, g, n)[:, :n1]) * O.matmul(gtype, x, u, n1)
        assert_parity(got, want, what=f"glu {gtype} n={n1} b={b}")
        qkv = qmm.mmvq_fused_qkv(gtype, dev(g), dev(u), dev(v), vy, k, n, n - 3, n - 6, b, kp)
        for o, w, m in zip(qkv, (g, u, v), (n, n - 3, n - 6)):
            assert_parity(o.cpu().numpy(), O.matmul(gtype, x, w, m), what=f"qkv {gtype} n={m} b={b}")


@pytest.mark.parametrize("gtype", [O.Q4K, O.Q6K])
@pytest.mark.parametrize("counts", [(0, 1, 16, 17, 33, 5), (3, 0, 2), (70, 1, 0, 16)])
def test_grouped_rows_per_expert(gtype, counts):
    """Experts of no, few, 16, 17 and more than 32 rows (several passes), over both Q8_K tile layouts."""
    rng = np.random.default_rng(7200 + len(counts))
    n, k, e, total = 83, 1280, len(counts), sum(counts)
    assert total <= 32 * e  # the few-row kernel's share of the grouped entry
    ws = [O.quantize(gtype, weights(rng, n, k)) for _ in range(e)]
    wd = dev(np.concatenate(ws), 2 if gtype == O.Q6K else 0)
    ids = np.repeat(np.arange(e), counts)
    rng.shuffle(ids)
    x = acts(rng, total, k)
    bounds, tok, _, counts_d, _ = qmm.moe_dispatch(torch.from_numpy(ids.astype(np.int32)).cuda(), e, 1)
    want = np.stack([O.matmul(gtype, x[i:i + 1], ws[ids[i]], n)[0] for i in range(total)])
    for q8k in ([False, True] if gtype == O.Q4K else [False]):
        y, _ = qmm.quantize_prefill(gtype, torch.from_numpy(x).cuda(), ids=tok, q8k=q8k)
        out = torch.full((total, n), float("nan"), device="cuda")
        qmm.mmq_moe(gtype, wd, y, tok, bounds, e, k, n, total, int(counts_d.max().item()), out, q8k=q8k)
        assert_parity(out.cpu().numpy(), want, what=f"grouped {gtype} {counts} q8k={q8k}")


@pytest.mark.parametrize("gtype", [O.Q4K, O.Q6K])
@pytest.mark.parametrize("counts", [(0, 1, 16, 17, 33, 5), (70, 30, 12, 16)])
def test_grouped_glu(gtype, counts):
    """launch_mmq_gguf_<t>_moe_glu (few rows an expert, and enough on average for its wider tiles) in the experts' row
    order, gate and up at different offsets within a dword (Q6_K); above 32 rows an expert it launches nothing."""
    rng = np.random.default_rng(7300 + len(counts))
    n, k, e, total = 83, 768, len(counts), sum(counts)
    gs, us = ([O.quantize(gtype, weights(rng, n, k)) for _ in range(e)] for _ in range(2))
    gd, ud = dev(np.concatenate(gs), 2 if gtype == O.Q6K else 0), dev(np.concatenate(us))
    x = acts(rng, total, k)
    bounds = torch.tensor(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), device="cuda")
    y, _ = qmm.quantize_prefill(gtype, torch.from_numpy(x).cuda())
    out = torch.full((total, n), float("nan"), device="cuda")
    fn = getattr(qmm.lib(), f"launch_mmq_gguf_{qmm.tname(gtype)}_moe_glu")
    args = [qmm._ptr(gd), qmm._ptr(ud), qmm._ptr(y), qmm._ptr(bounds), qmm._ptr(out), k, n, total, k // 256, n]
    assert fn(*args, 1, 0, qmm._stream()) == (0 if total > 32 else 1)
    if total <= 32 * e:
        out.fill_(float("nan"))
        assert fn(*args, e, 0, qmm._stream()) == 1
        qmm.check()
        ex = np.repeat(np.arange(e), counts)
        want = np.stack([silu(O.matmul(gtype, x[i:i + 1], gs[ex[i]], n)[0]) * O.matmul(gtype, x[i:i + 1], us[ex[i]], n)[0]
                         for i in range(total)])
        assert_parity(out.cpu().numpy(), want, what=f"grouped glu {gtype} {counts}")
    assert fn(*args, e, 9, qmm._stream()) == -1 and qmm.last_error()
    qmm.lib().qmm_clear_error()


# The wide prefill tiles (256 weight rows x 64 or 128 activation rows): ragged in both, an odd number of superblocks, Q6_K
# 2 bytes past a dword; sizes at which the dispatch's model takes them (several rounds of the other forms' tiles)
WIDE = [(O.Q4K, 14113, 1280, 333, True), (O.Q4K, 14113, 1280, 333, False), (O.Q5K, 14113, 1280, 333, True),
        (O.Q5K, 9999, 768, 260, False), (O.Q6K, 14113, 1280, 333, False), (O.Q6K, 14113, 1280, 61, False),
        (O.IQ4XS, 14113, 1280, 333, False)]


@pytest.mark.parametrize("gtype,n,k,m,q8k", WIDE)
def test_wide_prefill_tiles(gtype, n, k, m, q8k):
    rng = np.random.default_rng(7400 + m + k)
    if gtype == O.IQ4XS:
        wq = rng.integers(0, 256, n * k // 256 * 136, dtype=np.uint8)
        wq.reshape(-1, 136)[:, :2] = (rng.uniform(0.5, 1.5, n * k // 256) * 0.002).astype(np.float16).view(
            np.uint8).reshape(-1, 2)
    else:
        wq = O.quantize(gtype, weights(rng, n, k))
    wd = dev(wq, 2 if gtype == O.Q6K else 0)
    x = acts(rng, m, k)
    x[m - 1] = 0.0
    want = O.matmul(gtype, x, wq, n)
    xd = torch.from_numpy(x).cuda()
    got = qmm.qmatmul_prefill(gtype, wd, xd, n, q8k=q8k)
    assert_parity(got.cpu().numpy(), want, what=f"wide {gtype} n={n} k={k} m={m}")
    half = qmm.qmatmul_prefill(gtype, wd, xd, n, out_dtype=torch.bfloat16, q8k=q8k)
    assert torch.equal(half.view(torch.int16), got.to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("gtype,n,k,m", [(O.Q6K, 4001, 7168, 300), (O.Q5K, 1000, 7168, 500)])
def test_wide_prefill_split_k(gtype, n, k, m):
    """Wide tiles over more planes than the reference's fixup buffer holds, through QMatMul::forward, twice: the same bits
    whichever split finishes first."""
    import ctypes
    rng = np.random.default_rng(7500 + m)
    wq = O.quantize(gtype, weights(rng, n, k))
    x = acts(rng, m, k)
    H = qmm.host()
    h = ctypes.c_void_p()
    assert H.qmm_qtensor_from_data(gtype, wq.ctypes.data, wq.size, 1, n, k, 0, ctypes.byref(h)) == 0
    try:
        xd = torch.from_numpy(x).cuda()
        outs = [torch.full((m, n), float("nan"), device="cuda") for _ in range(2)]
        for o in outs:
            assert H.qmm_qmatmul_forward(h, xd.data_ptr(), 0, m, o.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream) == 0, H.qmm_host_last_error()
        torch.cuda.synchronize()
    finally:
        H.qmm_qtensor_free(h)
    assert torch.equal(outs[0], outs[1])
    assert_parity(outs[0].cpu().numpy(), O.matmul(gtype, x, wq, n), what=f"split wide {gtype} n={n} k={k} m={m}")


@pytest.mark.parametrize("gtype", ROWS16[:3])
@pytest.mark.parametrize("n,k,m", [(16583, 1280, 90), (16583, 1280, 121), (16640, 256, 96), (4019, 14336, 470)])
def test_prefill_tiles_of_32_value_types(gtype, n, k, m):
    """96- and 128-row activation tiles with ragged rows and weight rows (more weight tiles than half the compute units),
    and the shape where K is split; both activation layouts.  A prime count of distinct weight rows repeats, so that a
    misplaced tile shows.  f16 output is the f32 one rounded."""
    rng = np.random.default_rng(7600 + n + m)
    u = 67
    wq = O.quantize(gtype, weights(rng, u, k))
    rows = np.arange(n) % u
    wd = dev(np.ascontiguousarray(wq).reshape(-1).view(np.uint8).reshape(u, -1)[rows])
    x = acts(rng, m, k)
    xd = torch.from_numpy(x).cuda()
    y, _ = qmm.quantize_prefill(gtype, xd)
    got = qmm.mmq(gtype, wd, y, k, n, m)
    assert_parity(got.cpu().numpy(), O.matmul(gtype, x, wq, u)[:, rows], what=f"{gtype} {n}x{k} m={m}")
    assert torch.equal(qmm.mmq(gtype, wd, y, k, n, m, out_dtype=torch.float16), got.half())
    y, _ = qmm.quantize_prefill(gtype, xd, q8_1=True)
    got = qmm.mmq(gtype, wd, y, k, n, m, q8_1=True)
    one = qmm.mmq(gtype, wd, y, k, n, m, q8_1=True, tmp_fixup=False)  # K in one piece
    assert (got - one).abs().max() <= 1e-5 * one.abs().max()
