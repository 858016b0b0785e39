"""CPU test of mc_align.cpp's sharpness entry point on a stand-in for the HIP
runtime that records asynchronous copies from host memory until the stream is
synchronised: after a failed allocation or launch none may be pending, since the
host vectors they read are freed or written again by the next call."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

HARNESS = r"""
#include "mc_kernels.h"
#include "mc_abi.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
static int pending = 0, mallocs_left = -1;
static bool launch_fails = false;
extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { pending = 0; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  if (mallocs_left == 0) return hipErrorOutOfMemory;
  if (mallocs_left > 0) mallocs_left--;
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { pending++; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}
namespace mc {
hipError_t launch_padded_to_spec(const float2*, int, float2*, hipStream_t) { return hipSuccess; }
size_t sharp_part_elems(int nframes, int) { return nframes + 1; }
hipError_t launch_sharpness(const float2*, size_t, int, int, const double2*, float2*, const float*, double2*,
                            double2* out, hipStream_t) {
  if (launch_fails) return hipErrorInvalidValue;
  out[0] = make_double2(0, 0);
  return hipSuccess;
}
}
int main() {
  const int n = 64, F = 3;
  std::vector<float> spec((size_t)F * n * (n + 2));
  const double shift[2 * F] = {};
  double J;
  int bad = 0;
  // the k-th allocation of the call fails, then the launch, then nothing
  for (int k = 0; k < 7; k++) {
    mc_context c;
    if (mc_context_create(0, &c) || mc_set_spectra(c, spec.data(), n, F)) return 90;
    mallocs_left = k < 4 ? k : -1;
    launch_fails = k == 4;
    const int rc = mc_sharpness(c, shift, 100.f, &J, nullptr);
    mallocs_left = -1;
    printf("%d: rc %d, %d pending\n", k, rc, pending);
    if ((rc != 0) != (k < 5) || pending) bad = 1;
    mc_context_destroy(c);
  }
  return bad;
}
"""


def test_failed_sharpness_leaves_no_copy_pending(tmp_path):
    if not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime.h")):
        pytest.skip("HIP headers not available")
    src = tmp_path / "harness.cpp"
    src.write_text(HARNESS)
    csrc = os.path.join(ROOT, "motioncorr1exp_amd", "csrc")
    exe = tmp_path / "harness"
    # entry points that the harness does not call stay unresolved
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I", csrc, "-I",
                        os.path.join(ROOT, "include"), "-isystem", os.path.join(ROCM, "include"), str(src),
                        os.path.join(csrc, "mc_align.cpp"), "-o", str(exe), "-no-pie", "-Wl,-z,lazy",
                        "-Wl,--unresolved-symbols=ignore-all"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
