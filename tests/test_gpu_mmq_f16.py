"""The f16 GEMM of large Q4_K / Q5_K / Q6_K grids (mmq_f16.hip) against the int8
MMQ and the f64 formula.

hip_qmm_mul_mat takes it when the workspace holds the columns' panels
(hip_qmm_mul_mat_workspace_preferred); with the required workspace the same call
runs the int8 kernels.  The block products are exact in both.  Unsplit Q4_K and
Q5_K sums run in the same order, so the outputs are equal bit for bit; Q6_K's two
scale groups of a block are added before the f32 sum, and K splits differ, so
those agree within f32 rounding: 1e-6 of max |out| (sums of up to 56 super-blocks
at 2^-24 each)."""
import numpy as np
import pytest

import oracle_lib as O
from cases import acts, max_err_scaled, weights_q

torch = pytest.importorskip("torch")

F64_TOL = 2e-6
TYPES = {"Q4_K": O.TYPE_Q4_K, "Q5_K": O.TYPE_Q5_K, "Q6_K": O.TYPE_Q6_K}


def test_preferred_workspace_without_a_device():
    """The panels are asked for only where the f16 GEMM runs: K-quants with mins
    or Q6_K, K a multiple of 256, more than 32 columns; never less than the
    required workspace."""
    import ggml_hip as G
    L = G.lib()
    for t in (2, 8, 12, 13, 14, 23):
        for K in (256, 768, 4096, 4128, 14336):
            for nrows in (1, 300, 4096, 14336):
                for n in (1, 8, 32, 33, 200, 513, 2048, 65535):
                    need = L.hip_qmm_mul_mat_workspace_size(t, K, nrows, n)
                    pref = L.hip_qmm_mul_mat_workspace_preferred(t, K, nrows, n)
                    gneed = L.hip_qmm_mul_mat_glu_workspace_size(t, K, nrows, n)
                    gpref = L.hip_qmm_mul_mat_glu_workspace_preferred(t, K, nrows, n)
                    assert pref >= need and gpref >= gneed
                    if t not in (12, 13, 14) or K % 256 or n <= 32:
                        assert pref == need and gpref == gneed
    assert L.hip_qmm_mul_mat_workspace_preferred(12, 4096, 14336, 512) == 16 * 16 * 18432


def _weights(t, nrows, K, idx=0):
    """Quantized rows: a base of at most 1024 rows, repeated with its rows rolled."""
    base = weights_q(t, min(nrows, 1024), K, idx)
    w = np.concatenate([np.roll(base, 17 * i, axis=0) for i in range((nrows + 1023) // 1024)])[:nrows]
    return np.ascontiguousarray(w)


def _op(G, t, w, x, out, ws):
    n, K = x.shape
    rc = G.lib().hip_qmm_mul_mat(t, w.data_ptr(), K, w.shape[0], w.stride(0), x.data_ptr(), n, x.stride(0),
                                 out.data_ptr(), out.stride(0), ws.data_ptr(), ws.numel(),
                                 torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("tname,nrows,K,ncols", [
    ("Q4_K", 14333, 1024, 2045),  # three rounds of 256 x 128 tiles, 128 more as quarter tiles; ragged rows, columns
    ("Q5_K", 14333, 1024, 2045),
    ("Q4_K", 6150, 2048, 1025),   # one column in the last column tile
    ("Q5_K", 6401, 768, 1100),    # an odd number of super-blocks; one row in the last row tile
    ("Q4_K", 14336, 1024, 512),   # one partly filled round
    ("Q4_K", 4096, 14336, 512),   # K split
    ("Q6_K", 10493, 512, 1019),   # a round, then 72 as quarter tiles
    ("Q6_K", 2100, 256, 400),     # one super-block
    ("Q6_K", 6401, 768, 300),
    ("Q6_K", 4096, 8192, 512),    # 256 x 128 tiles, K split
    ("Q6_K", 1030, 4096, 512),    # 128 x 64 tiles, K split
    ("Q6_K", 2100, 512, 333),     # 128 x 64 tiles, unsplit
])
def test_f16_route_matches_int8(tname, nrows, K, ncols):
    import ggml_hip as G
    t, L = TYPES[tname], G.lib()
    need = L.hip_qmm_mul_mat_workspace_size(t, K, nrows, ncols)
    pref = L.hip_qmm_mul_mat_workspace_preferred(t, K, nrows, ncols)
    assert pref > need  # the f16 route takes it
    wq = _weights(t, nrows, K)
    w_d = torch.from_numpy(wq).cuda()
    # columns 8 floats apart from their neighbours' ends, outputs 3: strides of the views, not the shapes
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    xs = torch.full((ncols, K + 8), float("nan"), device="cuda")
    xs[:, :K] = x
    out = torch.full((ncols, nrows + 3), float("nan"), device="cuda")
    ws = torch.full((pref,), 255, dtype=torch.uint8, device="cuda")  # scratch left as NaN patterns
    got = _op(G, t, w_d, xs[:, :K], out[:, :nrows], ws).cpu().numpy()
    assert np.isnan(out[:, nrows:].cpu().numpy()).all()
    int8 = _op(G, t, w_d, x, torch.empty((ncols, nrows), device="cuda"), ws[:need]).cpu().numpy()
    panels = K // 256 * ((ncols + 127) // 128 * 4) * 18432
    if tname != "Q6_K" and L.hip_qmm_mmq_split_k(t, K, nrows, ncols) == 1 and pref == panels:
        np.testing.assert_array_equal(got, int8)
    assert max_err_scaled(got, int8) < 1e-6
    np.testing.assert_array_equal(G.mul_mat(tname, w_d, x).cpu().numpy(), got)  # the wrapper prefers it too
    rows = np.r_[0:40, nrows // 2:nrows // 2 + 40, nrows - 40:nrows]
    y = G.quantize_q8_1(x, K).cpu().numpy()
    ideal = O.mul_mat_q8_1_f64(t, wq[rows], len(rows), K, y, ncols)
    assert max_err_scaled(got[:, rows], ideal) < F64_TOL


@pytest.mark.gpu
def test_f16_route_leaves_unaligned_columns_to_int8():
    """Columns not 16-byte aligned cannot be read as float4: the int8 kernels run."""
    import ggml_hip as G
    nrows, K, ncols, t = 6150, 2048, 1025, O.TYPE_Q4_K
    pref = G.lib().hip_qmm_mul_mat_workspace_preferred(t, K, nrows, ncols)
    w_d = torch.from_numpy(_weights(t, nrows, K)).cuda()
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    buf = torch.zeros(ncols * K + 1, device="cuda")
    xu = buf[1:].view(ncols, K)
    xu.copy_(x)
    ws = torch.empty(pref, dtype=torch.uint8, device="cuda")
    a = _op(G, t, w_d, xu, torch.empty((ncols, nrows), device="cuda"), ws)
    b = _op(G, t, w_d, x, torch.empty((ncols, nrows), device="cuda"), ws)
    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("tname,nrows,K,ncols", [("Q4_K", 7165, 1024, 2045), ("Q5_K", 6150, 2048, 1024),
                                                 ("Q6_K", 1030, 512, 333), ("Q6_K", 5250, 512, 1019)])
def test_f16_glu_matches_int8(tname, nrows, K, ncols):
    """Gate / up / GLU: 128 output rows per wide tile (64 per narrow or quarter
    tile); equal to the int8 fused kernel bit for bit for Q4_K and Q5_K."""
    import ggml_hip as G
    t, L = TYPES[tname], G.lib()
    need = L.hip_qmm_mul_mat_glu_workspace_size(t, K, nrows, ncols)
    assert L.hip_qmm_mul_mat_glu_workspace_preferred(t, K, nrows, ncols) > need
    w, wg = (torch.from_numpy(_weights(t, nrows, K, i)).cuda() for i in (0, 1))
    x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
    got = G.mul_mat_glu(tname, w, wg, x).cpu().numpy()
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    int8 = G.mul_mat_glu(tname, w, wg, x, workspace=ws).cpu().numpy()
    if tname == "Q6_K":
        assert max_err_scaled(got, int8) < 2e-6
    else:
        np.testing.assert_array_equal(got, int8)


@pytest.mark.gpu
def test_f16_route_under_graph_capture():
    """The route's launches replay: panels, tiles and K-split partials are
    rewritten on every replay."""
    import ggml_hip as G
    cases = [("Q6_K", 1030, 4096, 512), ("Q4_K", 6150, 2048, 1025)]
    ins = []
    for tname, nrows, K, ncols in cases:
        w = torch.from_numpy(_weights(TYPES[tname], nrows, K)).cuda()
        x = torch.from_numpy(np.array(acts(ncols, K))).cuda()
        ins.append((tname, w, x))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        outs = [G.mul_mat(*a) for a in ins]
    for rep in range(3):
        for _, _, x in ins:
            x.mul_(-0.5)
        want = [G.mul_mat(*a) for a in ins]
        for o in outs:
            o.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        for o, v in zip(outs, want):
            np.testing.assert_array_equal(o.cpu().numpy(), v.cpu().numpy(), err_msg=f"replay {rep}")
