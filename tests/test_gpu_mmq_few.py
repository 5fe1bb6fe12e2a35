"""The few-column GEMM whose 16-row workgroups hold all of K (at most 12224 rows and
64 Mi weights, up to 32 columns; Q6_K 16), against the f64 Q8_1 formula at the edges
of its tiles and K parts.  Each output sums exact integer dots with f32 scales: at
most 8 terms a K step, 256 weights, then the steps and 8 parts in order, so the error
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
    (65, 512, 5), (65, 1536, 13), (65, 2560, 31),  # fewer steps than waves; uneven parts
])
def test_few_whole_k(tname, nrows, K, ncols):
    import ggml_hip as G
    t = TYPES[tname]
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


@pytest.mark.parametrize("nrows", [12224, 12225])
@pytest.mark.parametrize("ncols", [3, 13, 24])
def test_few_row_limit(nrows, ncols):
    """The last rows each form takes: 16-row workgroups up to 12224, 64-row above."""
    import ggml_hip as G
    K = 512
    wq = weights_q(O.TYPE_Q5_K, nrows, K)
    w_d = torch.from_numpy(np.array(wq)).cuda()
    x_d = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    qs, ds = G.quantize_q8_1_planar(x_d)
    got = G.mmq("Q5_K", w_d, K, qs, ds).cpu().numpy()
    ideal = O.mul_mat_q8_1_f64(O.TYPE_Q5_K, wq, nrows, K, G.quantize_q8_1(x_d, K).cpu().numpy(), ncols)
    assert max_err_scaled(got, ideal) < F64_TOL, max_err_scaled(got, ideal)
