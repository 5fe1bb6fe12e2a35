"""Activations and weight scales at the ends of f16 against the f64 Q8_1 formula.

A Q8_1 block whose 32 activations sum past 65504 has an infinite s next to a finite
d.  Only the types with mins (Q4_K, Q5_K) use s, so the others' results are finite
and stay within the shared gate of 2e-6 of max |out|; an infinite s or weight scale
that the formula does use gives the formula's infinity."""
import numpy as np
import pytest

import oracle_lib as O
from cases import acts, max_err_scaled, weights_q

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F64_TOL = 2e-6
NO_MINS = {"Q6_K": O.TYPE_Q6_K, "Q8_0": O.TYPE_Q8_0, "Q4_0": O.TYPE_Q4_0, "IQ4_XS": O.TYPE_IQ4_XS}
MINS = {"Q4_K": O.TYPE_Q4_K, "Q5_K": O.TYPE_Q5_K}


def _weights(t, nrows, K, idx=0):
    """nrows quantized rows: a base of at most 512, repeated with its rows rolled."""
    base = weights_q(t, min(nrows, 512), K, idx)
    w = np.concatenate([np.roll(base, 7 * i, axis=0) for i in range((nrows + 511) // 512)])[:nrows]
    return np.ascontiguousarray(w)


def _overflowing(ncols, K):
    """N(0, 1) columns in which every third block of 32, from another one in each
    column, is 3000 throughout: its sum of 96000 is past f16."""
    x = np.array(acts(ncols, K))
    for c in range(ncols):
        x[c].reshape(-1, 32)[c % 3::3] = 3000.0
    return x


def _ideal(G, t, w, x_d):
    K = x_d.shape[1]
    with np.errstate(invalid="ignore", over="ignore"):
        return O.mul_mat_q8_1_f64(t, w, len(w), K, G.quantize_q8_1(x_d, K).cpu().numpy(), len(x_d))


# the routes of a few columns: 16-row workgroups with all of K, 64-row ones (12300
# rows), up to 8 columns, one and two tiles of 16
@pytest.mark.parametrize("tname", list(NO_MINS))
@pytest.mark.parametrize("nrows,K,ncols", [(333, 4096, 5), (5120, 4096, 8), (333, 2048, 13), (333, 2048, 24),
                                           (12300, 512, 4), (12300, 512, 13), (12300, 512, 24)])
def test_few_columns_overflowing_block_sums(tname, nrows, K, ncols):
    import ggml_hip as G
    t = NO_MINS[tname]
    w = _weights(t, nrows, K)
    w_d = torch.from_numpy(w).cuda()
    x_d = torch.from_numpy(_overflowing(ncols, K)).cuda()
    rows = np.r_[0:min(nrows, 100), max(nrows - 100, 0):nrows]
    ideal = _ideal(G, t, w[rows], x_d)
    assert np.isfinite(ideal).all()
    qs, ds = G.quantize_q8_1_planar(x_d)
    for got in (G.mmq(tname, w_d, K, qs, ds), G.mul_mat(tname, w_d, x_d)):
        assert torch.isfinite(got).all()
        assert max_err_scaled(got.cpu().numpy()[:, rows], ideal) < F64_TOL


@pytest.mark.parametrize("tname,ncols", [(t, n) for t in NO_MINS for n in (4, 8, 13)] + [("Q4_0", 24), ("IQ4_XS", 24)])
def test_glu_few_columns_overflowing_block_sums(tname, ncols):
    """REGLU: max(gate, 0) * up, off by at most the two products' errors times the
    other factor."""
    import ggml_hip as G
    t, nrows, K = NO_MINS[tname], 6147, 2048
    w, wg = _weights(t, nrows, K, 0), _weights(t, nrows, K, 1)
    x_d = torch.from_numpy(_overflowing(ncols, K)).cuda()
    got = G.mul_mat_glu(tname, torch.from_numpy(w).cuda(), torch.from_numpy(wg).cuda(), x_d, "REGLU")
    assert torch.isfinite(got).all()
    rows = np.r_[0:100, nrows - 100:nrows]
    up, gate = _ideal(G, t, w[rows], x_d), _ideal(G, t, wg[rows], x_d)
    bound = 2 * F64_TOL * np.abs(up).max() * np.abs(gate).max()
    assert np.abs(got.cpu().numpy()[:, rows] - np.maximum(gate, 0.0) * up).max() < bound


# the MMQ tiles: an op's own Q8_1 copy leaves s out for these types
@pytest.mark.parametrize("tname", list(NO_MINS))
@pytest.mark.parametrize("nrows,K,ncols", [(333, 2048, 40), (1030, 4096, 200)])
def test_tiles_overflowing_block_sums(tname, nrows, K, ncols):
    import ggml_hip as G
    t = NO_MINS[tname]
    w = _weights(t, nrows, K)
    x = _overflowing(ncols, K)
    w_d, x_d = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    xu = torch.empty(ncols * K + 1, device="cuda")[1:].view(ncols, K)  # not 16-byte aligned: the plain quantizer
    xu.copy_(x_d)
    rows = np.r_[0:100, nrows - 100:nrows]
    ideal = _ideal(G, t, w[rows], x_d)
    for got in (G.mul_mat(tname, w_d, x_d), G.mul_mat(tname, w_d, xu)):
        assert torch.isfinite(got).all()
        assert max_err_scaled(got.cpu().numpy()[:, rows], ideal) < F64_TOL
    gated = G.mul_mat_glu(tname, w_d, torch.from_numpy(_weights(t, nrows, K, 1)).cuda(), x_d, "REGLU")
    assert torch.isfinite(gated).all()


@pytest.mark.parametrize("tname", list(NO_MINS))
def test_mul_mat_id_overflowing_block_sums(tname):
    import ggml_hip as G
    from cases import mul_mat_id_f64, route_top_k
    t, n_as, nrows, K, n_tokens = NO_MINS[tname], 4, 96, 1024, 40
    w = np.stack([weights_q(t, nrows, K, i) for i in range(n_as)])
    x = _overflowing(n_tokens, K)
    ids = route_top_k(n_tokens, n_as, 2)[0]
    w_d, ids_d = torch.from_numpy(w).cuda(), torch.from_numpy(ids).cuda()
    xu = torch.empty(n_tokens * K + 1, device="cuda")[1:].view(n_tokens, 1, K)  # not 16-byte aligned
    xu.copy_(torch.from_numpy(x).view(n_tokens, 1, K))
    x_d = xu.clone()
    ideal = mul_mat_id_f64(t, w, nrows, K, G.quantize_q8_1(x_d.view(n_tokens, K), K).cpu().numpy(), 1, ids)
    for v in (x_d, xu):
        got = G.mul_mat_id(tname, w_d, v, ids_d)
        assert torch.isfinite(got).all()
        assert max_err_scaled(got.cpu().numpy(), ideal) < F64_TOL
    assert torch.isfinite(G.mul_mat_id_glu(tname, w_d, w_d, x_d, ids_d, "REGLU")).all()


# up to 8 columns an infinite s of Q4_K / Q5_K times its mins is the formula's -inf
@pytest.mark.parametrize("tname", list(MINS))
@pytest.mark.parametrize("nrows,K,ncols", [(12300, 512, 4), (12300, 512, 8), (6147, 1024, 8), (333, 4096, 5)])
def test_few_columns_infinite_min_term(tname, nrows, K, ncols):
    import ggml_hip as G
    t = MINS[tname]
    w = _weights(t, nrows, K)
    x = np.array(acts(ncols, K))
    x[1::3, 32 * 3:32 * 4] = 3000.0  # a block of columns 1, 4, ..
    x_d = torch.from_numpy(x).cuda()
    qs, ds = G.quantize_q8_1_planar(x_d)
    got = G.mmq(tname, torch.from_numpy(w).cuda(), K, qs, ds).cpu().numpy()[:, :200]
    ideal = _ideal(G, t, w[:200], x_d)
    inf = np.isneginf(ideal)
    assert inf[1::3].mean() > 0.9 and not inf[0::3].any()
    assert np.isneginf(got[inf]).all()
    keep = ~inf.any(axis=1)
    assert max_err_scaled(got[keep], ideal[keep]) < F64_TOL


def _infinite_block(tname, w, row, sb):
    """256 weights of a row: an infinite f16 scale, positive codes and sub-block
    scales, no min."""
    nb = {"Q8_0": 34, "Q4_0": 18}.get(tname)
    if nb:
        blk = w[row, sb * 8 * nb:(sb * 8 + 1) * nb]
        blk[:2] = (0x00, 0x7C)
        blk[2:] = 0x7F if tname == "Q8_0" else 0xFF
        return
    size = O.BLOCK[O.TYPE_IDS[tname]][1]
    blk = w[row, sb * size:(sb + 1) * size]
    blk[:] = 0xFF  # largest codes
    if tname == "Q6_K":
        blk[192:208], blk[208:210] = 1, (0x00, 0x7C)
    elif tname == "IQ4_XS":
        blk[:2] = (0x00, 0x7C)
    else:
        blk[:4], blk[4:16] = (0x00, 0x7C, 0x00, 0x00), 0x11


# whole-K (333 rows, 5 / 13 / 24 columns) and fused sums, which keep their rounding
# errors, and the 64-row workgroups' plain ones
@pytest.mark.parametrize("tname", list(NO_MINS) + list(MINS))
@pytest.mark.parametrize("nrows,K,ncols", [(333, 4096, 5), (333, 4096, 13), (333, 4096, 24), (12300, 512, 5)])
def test_few_columns_infinite_weight_scale(tname, nrows, K, ncols):
    import ggml_hip as G
    t = O.TYPE_IDS[tname]
    w = _weights(t, nrows, K)
    rows = [3, nrows - 1]
    for i, r in enumerate(rows):
        _infinite_block(tname, w, r, i)
    x = np.abs(np.array(acts(ncols, K))) + 0.1
    x[1::2] *= -1.0  # columns 1, 3, ..: -inf
    x_d = torch.from_numpy(x).cuda()
    pick = np.r_[0:100, nrows - 100:nrows]
    ideal = _ideal(G, t, w[pick], x_d)
    qs, ds = G.quantize_q8_1_planar(x_d)
    got = G.mmq(tname, torch.from_numpy(w).cuda(), K, qs, ds).cpu().numpy()[:, pick]
    bad = np.isin(pick, rows)
    assert np.isposinf(ideal[0::2][:, bad]).all() and np.isneginf(ideal[1::2][:, bad]).all()
    np.testing.assert_array_equal(got[:, bad], ideal[:, bad])
    assert max_err_scaled(got[:, ~bad], ideal[:, ~bad]) < F64_TOL


@pytest.mark.parametrize("ncols", [5, 13])
def test_glu_few_columns_infinite_weight_scale(ncols):
    """REGLU of an infinite gate and a positive finite up."""
    import ggml_hip as G
    t, nrows, K = O.TYPE_Q8_0, 6147, 2048
    w, wg = _weights(t, nrows, K, 0), _weights(t, nrows, K, 1)
    _infinite_block("Q8_0", wg, 3, 0)
    x = np.abs(np.array(acts(ncols, K))) + 0.1
    x_d = torch.from_numpy(x).cuda()
    w_d, wg_d = torch.from_numpy(w).cuda(), torch.from_numpy(wg).cuda()
    up = _ideal(G, t, w[:8], x_d)
    got = G.mul_mat_glu("Q8_0", w_d, wg_d, x_d, "REGLU").cpu().numpy()
    np.testing.assert_array_equal(got[:, 3], np.copysign(np.inf, up[:, 3]))
    assert np.isfinite(np.delete(got, 3, axis=1)).all()
