"""What hip_qmm_mul_mat hands to hip_qmm_mmq as its scratch lies inside the caller's
workspace, down to the required size.  Without a device: in a process of its own, a shim
loaded first stands in for the quantizer and for hip_qmm_mmq and prints the scratch it
is given."""
import subprocess
import sys

import ggml_hip as G

SHIM = r"""
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
namespace { uintptr_t base; size_t total; }
int qmm_quantize_planar(const float *, int64_t, int64_t, int64_t, int8_t *qs, void *, uint32_t, struct ihipStream_t *) {
    base = (uintptr_t)qs;
    return 0;
}
extern "C" int hip_qmm_mmq(int, const void *, int64_t, int64_t, int64_t, const int8_t *, const void *, int64_t, float *,
                           int64_t, void *ws, size_t size, void *) {
    printf("%lld %llu\n", ws ? (long long)((uintptr_t)ws - base) : -1, (unsigned long long)size);
    fflush(stdout);
    return 0;
}
"""

CALL = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
L = ctypes.CDLL(sys.argv[1])
L.hip_qmm_mul_mat_workspace_size.restype = ctypes.c_size_t
i64, vp = ctypes.c_int64, ctypes.c_void_p
for line in sys.argv[3:]:
    t, nrows, K, n, extra, rs = (int(v) for v in line.split(","))
    need = L.hip_qmm_mul_mat_workspace_size(t, i64(K), i64(nrows), i64(n))
    size = need + extra
    # addresses that nothing reads: both kernels are stand-ins
    e = L.hip_qmm_mul_mat(t, vp(1 << 20), i64(K), i64(nrows), i64(rs), vp(1 << 21), i64(n), i64(K), vp(1 << 22),
                          i64(nrows), vp(1 << 23), ctypes.c_size_t(size), None)
    print("call", e, size, flush=True)
"""


def test_scratch_lies_inside_the_workspace(tmp_path):
    src, shim = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(shim), str(src)], check=True)
    # (type, rows, K, columns, bytes above the required workspace, row bytes): few-column calls
    # without partials, whose required size is not a multiple of 256, and one with partials
    cases = [(13, 4097, 1024, 5, 0, 704), (13, 4097, 1024, 5, 127, 704), (13, 4097, 1024, 5, 128, 704),
             (12, 6144, 1024, 3, 0, 576), (12, 300, 14336, 24, 0, 8064), (14, 6150, 2048, 4, 0, 1680)]
    args = [str(G.LIB_PATH), str(shim)] + [",".join(map(str, c)) for c in cases]
    out = subprocess.run([sys.executable, "-c", CALL] + args, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    lines = [v.split() for v in out.stdout.splitlines()]
    assert len(lines) == 2 * len(cases), out.stdout
    for c, (off, size), call in zip(cases, lines[0::2], lines[1::2]):
        assert call[:2] == ["call", "0"], c
        off, size, total = int(off), int(size), int(call[2])
        assert size == 0 if off < 0 else off + size <= total, (c, off, size, total)
