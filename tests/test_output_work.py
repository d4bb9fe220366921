"""Workspaces that RecviewOutputStage keeps between calls (CPU, against stand-ins for HIP)."""
import ctypes as C
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r'''
// host-only stand-ins for the HIP calls of rv_output.cpp, counting what is held
#include <cstdlib>
#include "rv_internal.h"
static int held = 0;
extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = std::malloc(n); held++; return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { *p = std::calloc(1, n); held++; return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); held--; return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); held--; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
int stub_held() { return held; }
void stub_reset(int dev) { rv::free_output_works(dev); }
}
namespace rv {
bool hip_ok(hipError_t e, const char*) { return e == hipSuccess; }
void set_message(const std::string&) {}
void launch_output_stage_parts(const void*, int, int, int, uint16_t*, void*, void*, hipStream_t) {}
}
'''


def test_kept_workspaces_are_given_back(tmp_path):
    """RecviewOutputStage keeps one workspace over calls in turn, and both its device and
    its pinned host memory are free again before a reset of their device."""
    csrc = os.path.join(ROOT, "recview_amd", "csrc")
    (tmp_path / "stub.cpp").write_text(STUB)
    so = tmp_path / "stub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-Wl,-Bsymbolic",
                    "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                    os.path.join(csrc, "rv_output.cpp"), str(tmp_path / "stub.cpp"), "-o", str(so)], check=True)
    L = C.CDLL(str(so))
    L.RecviewOutputStage.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_double, C.c_int, C.c_void_p, C.c_void_p,
                                     C.c_void_p, C.c_void_p]
    for _ in range(3):
        assert L.RecviewOutputStage(1, 1, 8, 4.0, 2, 1, None, None, None) == 0
        assert L.stub_held() == 2
    L.stub_reset(1)
    assert L.stub_held() == 2                          # another device's
    L.stub_reset(0)
    assert L.stub_held() == 0
