"""A backend's memory outlives sp_backend_destroy while a ticket names it: backend/Backend.cpp over a HIP runtime of host
stubs whose commands are complete at once, built with the host's address sanitizer. No GPU."""
import os
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIP = pathlib.Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "include"

STUBS = r"""
#include "splash_hip.h"
#include "backend/KernelRegistry.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
namespace {
template <class T> hipError_t handle(T *out) { *out = reinterpret_cast<T>(std::malloc(1)); return hipSuccess; }
template <class T> hipError_t freed(T h) { std::free(reinterpret_cast<void *>(h)); return hipSuccess; }
int calls = 0, failing = -1;   // the event record that fails
}
extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) { std::memset(p, 0, sizeof *p); return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return freed(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return freed(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return freed(e); }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return freed(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return ++calls == failing ? hipErrorInvalidValue : hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipLaunchHostFunc(hipStream_t, hipHostFn_t f, void *user) { f(user); return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = 1 << 30; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) { *d = p; return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
}
#define OK(call) do { if ((call) != SP_OK) { std::printf("line %d\n", __LINE__); return 1; } } while (0)
int main(int, char **argv) {
  const bool buffers = std::strchr(argv[1], 'b'), recorded = std::strchr(argv[1], 'r'), fails = std::strchr(argv[1], 'f');
  splash::hipbackend::registerKernel({"stub", [](const splash::hipbackend::LaunchArgs &) { return hipSuccess; }, 1, 4});
  sp_backend *backend = nullptr;
  OK(sp_backend_create(0, 0, &backend));
  sp_buffer *buffer = nullptr;
  uint32_t word = 0;
  sp_dispatch d{};
  if (buffers) {
    OK(sp_buffer_alloc(backend, 64, SP_STORAGE_PRIVATE, "buffer", &buffer));
    d.kernel = "stub"; d.buffer_count = 1; d.buffers = &buffer; d.params = &word; d.params_bytes = 4;
    for (int i = 0; i < 3; ++i) d.grid[i] = d.block[i] = 1;
  }
  for (int before = 0; before < 3; ++before) {   // the events of finished commands are there for the last one
    sp_ticket *ticket = nullptr;
    OK(sp_submit(backend, &d, buffers, nullptr, nullptr, &ticket));
    OK(sp_ticket_wait(ticket, nullptr, nullptr));
  }
  sp_ticket *ticket = nullptr;
  sp_command *command = nullptr;
  if (recorded) OK(sp_command_create(backend, &d, 1, &command));
  if (fails) failing = calls + 2;
  const sp_status status = recorded ? sp_command_submit(command, nullptr, nullptr, &ticket) : sp_submit(backend, &d, buffers, nullptr, nullptr, &ticket);
  if ((status != SP_OK) != fails) return 2;
  if (command) sp_command_release(command);
  if (buffer) sp_buffer_release(buffer);
  sp_backend_destroy(backend);
  if (ticket) OK(sp_ticket_wait(ticket, nullptr, nullptr));
  std::puts("done");
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not (HIP / "hip" / "hip_runtime.h").exists():
        pytest.skip("no host compiler or no HIP headers")
    folder = tmp_path_factory.mktemp("backend")
    (folder / "stubs.cpp").write_text(STUBS)
    out = folder / "program"
    build = ["g++", "-std=c++20", "-O1", "-g", "-w", "-fsanitize=address", "-static-libasan", "-D__HIP_PLATFORM_AMD__", f"-I{HIP}",
             f"-I{ROOT / 'include'}", f"-I{ROOT / 'splash_amd' / 'csrc'}", str(folder / "stubs.cpp"),
             str(ROOT / "splash_amd" / "csrc" / "backend" / "Backend.cpp"), "-o", str(out), "-pthread"]
    subprocess.run(build, check=True, timeout=240)
    return out


# b: a dispatch with a buffer, whose last name the ticket holds; r: recorded; f: a submission that fails; none: no dispatch
@pytest.mark.parametrize("what", ["-", "b", "br", "bf", "brf", "f"])
def test_a_ticket_keeps_its_backend(program, what):
    run = subprocess.run([str(program), what], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout.strip() == "done", run.stdout + run.stderr[-4000:]
