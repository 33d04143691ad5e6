"""What kd_mm_run would launch, without a GPU: kd_mm_host.cpp compiled with
launchers that record their arguments in place of the kernels'."""
import ctypes
import functools
import os
import subprocess
import tempfile
from collections import namedtuple

import kd_fa
import kd_mm

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "kd_mm_host.cpp"
static int32_t got[6];
static hipError_t record(int kernel, int tile, const kdfa::MmArgs &a) {
    const int32_t v[] = {kernel, tile, a.tiles_m, a.tiles_n, a.n_blocks, a.cols};
    for (int i = 0; i < 6; ++i) got[i] = v[i];
    return hipSuccess;
}
namespace kdfa {
int device_gfx950() { return KD_FA_OK; }
hipError_t launch_dequant(const DqArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_mm(const MmArgs &a, int tile, bool, hipStream_t) { return record(0, tile, a); }
hipError_t launch_mm_ksplit(const MmArgs &a, int tile, bool, hipStream_t) { return record(1, tile, a); }
hipError_t launch_mm_skinny(const MmArgs &a, bool, hipStream_t) { return record(2, 0, a); }
}
extern "C" const int32_t *recorded() { return got; }
"""

Plan = namedtuple("Plan", "kernel tile tiles_m tiles_n n_blocks cols")
KERNELS = ("mm_bf16", "mm_ksplit", "mm_skinny")


@functools.lru_cache(maxsize=None)
def _host():
    d = tempfile.mkdtemp()
    src, out = os.path.join(d, "plan.cpp"), os.path.join(d, "plan.so")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O1", "-fPIC", "--offload-arch=gfx950", "-shared",
                    "-I", os.path.join(ROOT, "kandinsky.cpp_amd", "csrc"), src, "-o", out], check=True, capture_output=True)
    lib = ctypes.CDLL(out)
    lib.recorded.restype = ctypes.POINTER(ctypes.c_int32)
    lib.kd_mm_run.argtypes = [ctypes.POINTER(kd_mm.KdMmDesc), ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
    return lib


def _view(t, rows, cols, size, kind, row_bytes):
    t.type = kind
    for i, (ne, nb) in enumerate([(cols, size), (rows, row_bytes), (1, row_bytes * rows), (1, row_bytes * rows)]):
        t.ne[i], t.nb[i] = ne, nb
    t.data = 1 << 20   # not read


def plan(M, N, K, x_f32=True):
    """The launch of a BF16-weight call of M tokens, N outputs and K inputs."""
    d = kd_mm.KdMmDesc()
    _view(d.w, N, K, 2, kd_mm.TYPE_BF16, 2 * K)
    _view(d.x, M, K, 4 if x_f32 else 2, kd_mm.TYPE_F32 if x_f32 else kd_mm.TYPE_BF16, (4 if x_f32 else 2) * K)
    _view(d.dst, M, N, 4, kd_mm.TYPE_F32, 4 * N)
    lib = _host()
    st = lib.kd_mm_run(ctypes.byref(d), None, 0, None)
    assert st == kd_fa.OK, st
    v = lib.recorded()
    return Plan(KERNELS[v[0]], *(v[i] for i in range(1, 6)))
