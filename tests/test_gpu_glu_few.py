"""Gate / up / GLU at 2-32 columns in one few-column launch (hip_qmm_mul_mat_glu
on matrices of at least 4096 rows and 12M weights) against the two products and
the GLU kernel run one by one.  The products' own kernels sum K in other orders,
so gate and up agree within 1e-6 of max; swiglu's slope is at most 1.1 and the
product of two such factors gives 4e-6 of max |out| with both at their maxima."""
import numpy as np
import pytest

import oracle_lib as O
from cases import acts, max_err_scaled, weights_q

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TYPES = {"Q4_K": O.TYPE_Q4_K, "Q5_K": O.TYPE_Q5_K, "Q6_K": O.TYPE_Q6_K, "Q8_0": O.TYPE_Q8_0,
         "Q4_0": O.TYPE_Q4_0, "IQ4_XS": O.TYPE_IQ4_XS}


def _weights(t, nrows, K, idx):
    """nrows quantized rows: a base of 512, repeated with its rows rolled."""
    base = weights_q(t, 512, K, idx)
    w = np.concatenate([np.roll(base, 7 * i, axis=0) for i in range((nrows + 511) // 512)])[:nrows]
    return torch.from_numpy(np.ascontiguousarray(w)).cuda()


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("nrows,K,ncols", [
    (6147, 2048, 2), (6147, 2048, 3), (6147, 2048, 4), (6147, 2048, 8),  # the packed MFMA form; 3 rows in the last tile
    (6147, 2048, 9), (6147, 2048, 16),                   # one column tile
    (12300, 2048, 17), (5152, 2560, 17), (5152, 2560, 32),  # two column tiles; 5152 x 2560: an odd ring of 10 steps
    (4096, 4096, 13),                                    # 128 workgroups, two K halves
])
def test_glu_few_columns(tname, nrows, K, ncols):
    import ggml_hip as G
    t = TYPES[tname]
    # every case runs the one launch but the first columns of some types, and beyond 16
    # columns Q6_K, Q8_0 and, from 8 MiB of weights on, Q4_0 (the fused MMQ tile)
    other = "unfused" if ncols < {"Q6_K": 3, "Q4_0": 3, "IQ4_XS": 4}.get(tname, 2) else "few"
    if ncols > 16 and (tname in ("Q6_K", "Q8_0") or (tname, nrows) == ("Q4_0", 12300)):
        other = "tile"
    assert G.kernel("mul_mat_glu", tname, K, nrows, ncols) == other
    w, wg = _weights(t, nrows, K, 0), _weights(t, nrows, K, 1)
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    out = torch.full((ncols, nrows + 5), float("nan"), device="cuda")
    got = G.mul_mat_glu(tname, w, wg, x, out=out[:, :nrows]).cpu().numpy()
    assert np.isnan(out[:, nrows:].cpu().numpy()).all()
    want = G.glu_f32(G.mul_mat(tname, wg, x), G.mul_mat(tname, w, x), "SWIGLU").cpu().numpy()
    assert max_err_scaled(got, want) < 4e-6, max_err_scaled(got, want)


@pytest.mark.parametrize("tname,nrows,K,ncols", [
    ("Q4_K", 4096, 8192, 4), ("Q4_K", 4096, 8192, 13), ("Q4_K", 4096, 8192, 24), ("Q5_K", 4096, 8192, 6),
    ("Q5_K", 4096, 8192, 13), ("Q6_K", 4096, 8192, 6), ("Q6_K", 4096, 8192, 13), ("Q8_0", 4096, 8192, 13),
    ("Q4_0", 4096, 8192, 13), ("IQ4_XS", 4096, 8192, 13), ("IQ4_XS", 4096, 8192, 24),
])
def test_glu_few_columns_precision(tname, nrows, K, ncols):
    """REGLU against the f64 gate and up: max(gate, 0) * up is off by the two sums'
    relative errors, each below 2.75 f32 half-ulps as the whole-K sums' are, and by the
    product's own rounding: sqrt(2 * 2.75^2 + 1) = 4.02 half-ulps in the 2-norm (plain
    sums measured 4.1-5.2 at 13 columns of Q4_K, Q5_K, Q8_0 and Q4_0, these 1.4-3.3)."""
    import ggml_hip as G
    t = TYPES[tname]
    assert G.kernel("mul_mat_glu", tname, K, nrows, ncols) == "few"
    w, wg = _weights(t, nrows, K, 0), _weights(t, nrows, K, 1)
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    got = G.mul_mat_glu(tname, w, wg, x, "REGLU").cpu().numpy()[:, :512].astype(np.float64)
    y = G.quantize_q8_1(x, K).cpu().numpy()
    up, gate = (O.mul_mat_q8_1_f64(t, weights_q(t, 512, K, i), 512, K, y, ncols) for i in (0, 1))
    want = np.maximum(gate, 0.0) * up
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel < 4.02 * 2.0 ** -24, rel * 2.0 ** 24


@pytest.mark.parametrize("op", ["REGLU", "GEGLU", "SWIGLU_OAI", "SWIGLU_CLAMP"])
def test_glu_few_columns_ops(op):
    """Every GLU op in the epilogue: the sums are the plain few-column kernel's of
    an unsplit grid (14336 rows, 5 columns: two K halves there, one ring here), so
    only rounding separates them; GEGLU rounds its gate to f16 (one f16 step on
    the few gates that cross)."""
    import ggml_hip as G
    nrows, K, ncols = 14336, 1024, 5
    assert G.kernel("mul_mat_glu", "Q4_K", K, nrows, ncols) == "few"
    w, wg = _weights(O.TYPE_Q4_K, nrows, K, 0), _weights(O.TYPE_Q4_K, nrows, K, 1)
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    got = G.mul_mat_glu("Q4_K", w, wg, x, op).cpu().numpy()
    want = G.glu_f32(G.mul_mat("Q4_K", wg, x), G.mul_mat("Q4_K", w, x), op).cpu().numpy()
    assert max_err_scaled(got, want) < (2e-3 if op == "GEGLU" else 8e-6), max_err_scaled(got, want)


def test_glu_few_columns_unaligned_rows_stay_unfused():
    """Rows the few-column kernel does not take run as before: the two products and
    the GLU, bit for bit."""
    import ggml_hip as G
    nrows, K, ncols = 6144, 2048, 6
    ws = []
    for i in (0, 1):
        w = _weights(O.TYPE_Q8_0, nrows, K, i)
        buf = torch.zeros(w.numel() + 16, dtype=torch.uint8, device="cuda")
        v = buf[2:2 + w.numel()].view(w.shape)
        v.copy_(w)
        ws.append(v)
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    got = G.mul_mat_glu("Q8_0", ws[0], ws[1], x).cpu().numpy()
    want = G.glu_f32(G.mul_mat("Q8_0", ws[1], x), G.mul_mat("Q8_0", ws[0], x), "SWIGLU").cpu().numpy()
    np.testing.assert_array_equal(got, want)
