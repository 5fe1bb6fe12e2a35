"""hip_qmm_mul_mat_noalloc runs the kernel that hip_qmm_mul_mat runs with the preferred
workspace, also where that is larger than the 32 MiB that bound the required one."""
import pathlib
import random
import re

import numpy as np
import pytest

import oracle_lib as O
from cases import acts, weights_q
from test_zz_no_alloc import SCRATCH_BYTES, _lib

torch = pytest.importorskip("torch")


def test_noalloc_array_holds_every_preferred_workspace():
    """Without a device: whatever is accepted finds the workspace with which
    hip_qmm_mul_mat runs its fastest kernel, so both run the same one."""
    G, L = _lib()
    header = (pathlib.Path(__file__).resolve().parents[1] / "include" / "ggml_hip_qmm.h").read_text()
    sizes = dict(re.findall(r"#define (HIP_QMM_NOALLOC_\w+) \((\d+)u << 20\)", header))
    array = int(sizes["HIP_QMM_NOALLOC_ARRAY_BYTES"]) << 20
    assert int(sizes["HIP_QMM_NOALLOC_SCRATCH_BYTES"]) << 20 == SCRATCH_BYTES
    rng, above = random.Random(0), 0
    for _ in range(200000):
        t = rng.choice((12, 13, 14))
        K = 256 * max(1, round(2 ** rng.uniform(0, 12)))
        n = min(65535, round(2 ** rng.uniform(5, 16)) + rng.choice((-1, 0, 1)))
        M = round(2 ** rng.uniform(5, 18))
        if L.hip_qmm_mul_mat_workspace_size(t, K, M, n) <= SCRATCH_BYTES:
            pref = L.hip_qmm_mul_mat_workspace_preferred(t, K, M, n)
            assert pref <= array, (t, K, M, n, pref)
            above += pref > SCRATCH_BYTES
    assert above > 1000


@pytest.mark.gpu
@pytest.mark.parametrize("tname,nrows,K,T", [("Q6_K", 4096, 8192, 512), ("Q4_K", 4096, 14336, 512)])
def test_noalloc_runs_the_preferred_kernel(tname, nrows, K, T):
    """A shape whose preferred workspace is over 32 MiB."""
    G, L = _lib()
    t = O.TYPE_IDS[tname]
    assert L.hip_qmm_mul_mat_workspace_size(t, K, nrows, T) <= SCRATCH_BYTES
    assert L.hip_qmm_mul_mat_workspace_preferred(t, K, nrows, T) > SCRATCH_BYTES
    w_d = torch.from_numpy(np.tile(weights_q(t, 512, K), (nrows // 512, 1))).cuda()
    x_d = torch.from_numpy(np.array(acts(T, K))).cuda()
    out = torch.full((T, nrows), float("nan"), device="cuda")
    e = L.hip_qmm_mul_mat_noalloc(t, G._ptr(w_d), K, nrows, w_d.stride(0), G._ptr(x_d), T, K, G._ptr(out), nrows,
                                  G._stream())
    assert e == 0
    assert torch.equal(out, G.mul_mat(tname, w_d, x_d))
