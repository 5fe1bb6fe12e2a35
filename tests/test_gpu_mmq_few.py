"""The few-column GEMM whose 16-row workgroups hold all of K (at most 12224 rows and
64 Mi weights, up to 32 columns; Q6_K 16), against the f64 Q8_1 formula at the edges
of its tiles and K parts.  Each output sums exact integer dots with f32 scales: at
most 8 terms a K step, 256 weights, then the steps and a tree of 8 parts, so the error
is below (8 + K / 256 / 8 + 8) f32 half-ulps of the sum of |terms|, which is under 8
times max |out| for these inputs: 24 * 6e-8 * 8 = 1.2e-5 at most; the shared gate of
2e-6 of max |out| holds for the random signs."""
import numpy as np
import pytest

import oracle_lib as O
from cases import acts, max_err_scaled, weights_q

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F64_TOL = 2e-6
TYPES = {"Q4_K": O.TYPE_Q4_K, "Q5_K": O.TYPE_Q5_K, "Q6_K": O.TYPE_Q6_K, "Q8_0": O.TYPE_Q8_0,
         "Q4_0": O.TYPE_Q4_0, "IQ4_XS": O.TYPE_IQ4_XS}


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("nrows,K,ncols", [
    (1, 2048, 1), (15, 2048, 2), (16, 2048, 8), (17, 2048, 9),  # one workgroup and one row more; a step a wave
    (333, 4096, 7), (333, 6144, 16), (33, 6144, 17), (33, 6144, 32),  # 3 steps a wave; column tiles
    (1537, 6144, 16), (1537, 6144, 17), (1537, 6144, 32),  # 3 steps a wave where a step has more work (Q6_K, two tiles)
    (65, 512, 5), (65, 1536, 13), (65, 2560, 31),  # fewer steps than waves; uneven parts
])
def test_few_whole_k(tname, nrows, K, ncols):
    import ggml_hip as G
    t = TYPES[tname]
    # beside it: 33 rows of 3 steps of two column tiles and 333 of Q6_K (64-row workgroups), and the
    # tile for Q6_K above 16 columns or on rows of K % 2048 (not 16-byte aligned), for Q8_0 from 8 MiB on
    beside = "few" if (nrows, K) == (33, 6144) or (tname, nrows, K) == ("Q6_K", 333, 6144) else "few whole K"
    if tname == "Q6_K" and (ncols > 16 or K % 2048) or tname == "Q8_0" and nrows == 1537 and ncols > 16:
        beside = "tile"
    assert G.kernel("mmq", tname, K, nrows, ncols) == beside
    wq = weights_q(t, nrows, K)
    w_d = torch.from_numpy(np.array(wq)).cuda()
    x_d = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    qs, ds = G.quantize_q8_1_planar(x_d)
    out = torch.full((ncols + 1, nrows + 3), float("nan"), device="cuda")
    got = G.mmq(tname, w_d, K, qs, ds, out=out[:ncols, :nrows]).cpu().numpy()
    assert np.isnan(out[:, nrows:].cpu().numpy()).all() and np.isnan(out[ncols].cpu().numpy()).all()
    again = G.mmq(tname, w_d, K, qs, ds).cpu().numpy()
    np.testing.assert_array_equal(got, again)
    ideal = O.mul_mat_q8_1_f64(t, wq, nrows, K, G.quantize_q8_1(x_d, K).cpu().numpy(), ncols)
    assert max_err_scaled(got, ideal) < F64_TOL, max_err_scaled(got, ideal)


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("ncols", [6, 13])
def test_few_whole_k_precision(tname, ncols):
    """Four steps a wave add no error that grows with the steps: below 2.75 f32 half-ulps
    of the result's norm (a step's blocks, its min term and the result each round once;
    plain sums measured 3.2 at 6 columns of Q4_K)."""
    import ggml_hip as G
    nrows, K = 2048, 8192
    t = TYPES[tname]
    wq = weights_q(t, nrows, K)
    w_d = torch.from_numpy(np.array(wq)).cuda()
    x_d = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    qs, ds = G.quantize_q8_1_planar(x_d)
    got = G.mmq(tname, w_d, K, qs, ds).cpu().numpy().astype(np.float64)
    ideal = O.mul_mat_q8_1_f64(t, wq, nrows, K, G.quantize_q8_1(x_d, K).cpu().numpy(), ncols)
    rel = np.linalg.norm(got - ideal) / np.linalg.norm(ideal)
    assert rel < 2.75 * 2.0 ** -24, rel * 2.0 ** 24


@pytest.mark.parametrize("nrows", [12224, 12225])
@pytest.mark.parametrize("K", [512, 1024])
@pytest.mark.parametrize("ncols", [3, 13, 24])
def test_few_row_limit(nrows, K, ncols):
    """The last rows each form takes: 16-row workgroups up to 12224 (from 4 steps on
    and with one column tile), 64-row above."""
    import ggml_hip as G
    whole_k = nrows == 12224 and K == 1024 and ncols <= 16
    assert G.kernel("mmq", "Q5_K", K, nrows, ncols) == ("few whole K" if whole_k else "few")
    wq = weights_q(O.TYPE_Q5_K, nrows, K)
    w_d = torch.from_numpy(np.array(wq)).cuda()
    x_d = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    qs, ds = G.quantize_q8_1_planar(x_d)
    got = G.mmq("Q5_K", w_d, K, qs, ds).cpu().numpy()
    ideal = O.mul_mat_q8_1_f64(O.TYPE_Q5_K, wq, nrows, K, G.quantize_q8_1(x_d, K).cpu().numpy(), ncols)
    assert max_err_scaled(got, ideal) < F64_TOL, max_err_scaled(got, ideal)


def _op(G, tname, w_d, K, x_d):
    """hip_qmm_mul_mat with exactly the workspace that it asks for."""
    import ctypes
    ncols, nrows = x_d.shape[0], w_d.shape[0]
    out = torch.full((ncols, nrows + 3), float("nan"), device="cuda")
    ws = torch.empty(G.workspace_size(tname, K, ncols, nrows), dtype=torch.uint8, device="cuda")
    e = G.lib().hip_qmm_mul_mat(TYPES[tname], G._ptr(w_d), K, nrows, w_d.stride(0), G._ptr(x_d), ncols, x_d.stride(0),
                                G._ptr(out), nrows + 3, G._ptr(ws), ctypes.c_size_t(ws.numel()), G._stream())
    assert e == 0, e
    assert np.isnan(out[:, nrows:].cpu().numpy()).all()
    return out[:, :nrows].cpu().numpy()


# 3-8 columns: the least count that each row and K band sends to the few-column GEMM, and one
# fewer or the GEMV's shapes beside them
@pytest.mark.parametrize("tname,nrows,K,ncols,few", [
    ("Q4_K", 6144, 1024, 3, 1), ("Q4_K", 4097, 1024, 5, 1), ("Q4_K", 4097, 1024, 4, 0), ("Q4_K", 2049, 4096, 7, 1),
    ("Q4_K", 2048, 4096, 7, 0), ("Q5_K", 4097, 1024, 4, 1), ("Q5_K", 4097, 768, 8, 0), ("Q5_K", 4096, 1024, 4, 0), ("Q5_K", 4096, 1024, 5, 1), ("Q5_K", 2050, 8192, 5, 1), ("Q5_K", 2050, 2048, 8, 0),
    ("Q6_K", 6150, 2048, 4, 1), ("Q6_K", 2050, 4096, 5, 1), ("Q8_0", 4100, 1024, 5, 1), ("Q8_0", 4100, 1024, 4, 0),
    ("Q4_0", 6144, 1024, 8, 1), ("Q4_0", 6144, 1024, 7, 0), ("IQ4_XS", 4100, 1024, 6, 1), ("IQ4_XS", 2050, 4096, 7, 1),
    ("Q8_0", 4100, 2048, 17, 1), ("Q4_0", 4100, 4096, 24, 0), ("Q8_0", 4096, 4096, 32, 1),  # whole K, the tile
])
def test_op_route(tname, nrows, K, ncols, few):
    import ggml_hip as G
    t = TYPES[tname]
    wq = weights_q(t, nrows, K)
    w_d = torch.from_numpy(np.array(wq)).cuda()
    x_d = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    assert G.kernel("mul_mat", tname, K, nrows, ncols) == (
        "few whole K" if few else "gemv" if ncols <= 8 else "tile")
    got = _op(G, tname, w_d, K, x_d)
    qs, ds = G.quantize_q8_1_planar(x_d)
    gemm = G.mmq(tname, w_d, K, qs, ds).cpu().numpy()
    assert np.array_equal(got, gemm) == bool(few or ncols > 8)
    ideal = O.mul_mat_q8_1_f64(t, wq, nrows, K, G.quantize_q8_1(x_d, K).cpu().numpy(), ncols)
    assert max_err_scaled(got, ideal) < F64_TOL, max_err_scaled(got, ideal)
