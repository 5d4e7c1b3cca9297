"""The evidence downloads after a compute_evidence that ran out of device memory: b2ctrain_amd/csrc/b2c/evidence.cpp,
compiled for the host against a stand-in of the few runtime calls it makes, whose allocations fail on demand and whose
kernels check their buffers. Each allocation of a second, larger pass fails in turn; the downloads that follow must
stay inside the buffers there are."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "b2ctrain_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

STAND_IN = r"""
#include <cstring>
#include <map>
#include <new>
#include "b2c/evidence.h"

static std::map<void*, size_t> blocks;
static int until_failure = -1;  // allocations that still succeed; negative: all
static bool overrun = false;

static void reach(const void* p, size_t bytes) {
  const auto b = blocks.find(const_cast<void*>(p));
  if (b == blocks.end() || b->second < bytes) overrun = true;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  if (until_failure == 0) return hipErrorOutOfMemory;
  if (until_failure > 0) until_failure--;
  *p = malloc(bytes);
  blocks[*p] = bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) { blocks.erase(p); free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  reach(s, n);
  if (!overrun) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
int b2c_hip_fill_u32(uint32_t* d, uint32_t v, size_t n, hipStream_t) { for (size_t i = 0; i < n; i++) d[i] = v; return 0; }
int b2c_hip_evidence_export(int n, const float* in, float* out, hipStream_t) {
  reach(in, (size_t)n * B2C_EVIDENCE_STRIDE * 4);
  reach(out, (size_t)n * 7 * 4);
  return 0;
}
int b2c_hip_label_export(int n, const float* in, float* out, hipStream_t) {
  reach(in, (size_t)n * B2C_LABEL_BINS * 4);
  reach(out, (size_t)n * 2 * 4);
  return 0;
}
}

int main() {
  alignas(b2c::RenderCtx) static unsigned char ctx_bytes[sizeof(b2c::RenderCtx)];  // no view: never looked at
  auto& ctx = *reinterpret_cast<b2c::RenderCtx*>(ctx_bytes);
  b2c::Model& m = *new b2c::Model;
  b2c::EvidenceParams cfg;
  cfg.export_labels = true;
  const std::vector<b2c::ViewGPU> views;
  const std::vector<b2c::Camera> cams;
  int failed = 0;
  for (int k = 0; k < 5; k++) {  // evidence and its rows, the view's sums, labels and their rows
    m.n = 100 << (2 * k);
    b2c::compute_evidence(ctx, m, views, cams, cfg, nullptr);
    m.n *= 2;
    until_failure = k;
    try {
      b2c::compute_evidence(ctx, m, views, cams, cfg, nullptr);
    } catch (const std::runtime_error&) {
      failed++;
    }
    until_failure = -1;
    std::vector<float> out((size_t)m.n * 7, 1.f);
    b2c::download_evidence(m, out.data(), nullptr);
    b2c::download_labels(m, out.data(), nullptr);
    if (overrun) {
      printf("a download reached past its buffer after allocation %d failed\n", k);
      return 1;
    }
  }
  printf("passes that ran out of memory: %d\n", failed);
  return failed == 5 ? 0 : 2;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="needs a host compiler and the HIP headers")
def test_downloads_after_an_allocation_failed(tmp_path):
    src, exe = tmp_path / "stand_in.cpp", tmp_path / "stand_in"
    src.write_text(STAND_IN)
    subprocess.check_call(["g++", "-std=c++20", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                           f"-I{ROOT}/include", f"-I{CSRC}", f"-I{CSRC}/kernels", str(src),
                           os.path.join(CSRC, "b2c", "evidence.cpp"), "-Wl,--unresolved-symbols=ignore-all",
                           "-o", str(exe)])
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
