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
