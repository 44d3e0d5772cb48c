"""The op layer on the host alone: csrc/ops.cpp compiled against a stand-in HIP runtime of several devices and
launchers that only note what they were called with."""
import ctypes
import os
import subprocess

import pytest

from svod_amd import ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STAND_IN = r"""
#include <hip/hip_runtime_api.h>
#include <cstring>
#include "kernels.h"
static int current = 0, launched_on = -1;
// Stream 0x1000 + n is of device n.
extern "C" {
int current_device() { return current; }
int last_launch() { const int on = launched_on; launched_on = -1; return on; }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) {
  if ((uintptr_t)s < 0x1000) return hipErrorInvalidHandle;
  *d = (int)((uintptr_t)s - 0x1000);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "?"; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
// Device 2 has no kernels.
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) { std::strcpy(p->gcnArchName, d == 2 ? "gfx90a" : "gfx950"); return hipSuccess; }
}
namespace svodk {
static hipError_t noted() { launched_on = current; return hipSuccess; }
hipError_t launch_heads(const HeadsArgs &, hipStream_t) { return noted(); }
hipError_t launch_norm(const NormArgs &, hipStream_t) { return noted(); }
hipError_t launch_linear(const LinearArgs &, hipStream_t) { return noted(); }
hipError_t launch_attention(const AttnArgs &, hipStream_t) { return noted(); }
hipError_t launch_combine(const CombineArgs &, hipStream_t) { return noted(); }
hipError_t launch_order_rows(const void *, int32_t, int32_t, int32_t, int32_t *, hipStream_t) { return noted(); }
hipError_t split_scratch(void **ptr, int64_t *bytes) { *ptr = nullptr; *bytes = 0; return hipSuccess; }
bool heads_supports(int32_t) { return true; }
bool norm_supports(int64_t) { return true; }
bool linear_supports(int64_t, int64_t) { return true; }
bool linear_turns(int32_t) { return true; }
bool attention_supports(int32_t) { return true; }
bool attention_decodes(const AttnArgs &, int32_t) { return false; }
int32_t attention_decode_limit() { return 0; }
void attention_decode_rows(int32_t) {}
void attention_stream_slots(int32_t) {}
uint32_t next_queue_set() { return 0; }
LinearTile linear_tile_of(int64_t, int64_t, int64_t, int, int) { return kTile128x128; }
int linear_tile(int32_t) { return 0; }
const char *linear_config(const LinearArgs &) { return ""; }
const char *attention_config(const AttnArgs &) { return ""; }
}  // namespace svodk
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("host")
    source, built = where / "stand_in.cpp", where / "host.so"
    source.write_text(STAND_IN)
    csrc = os.path.join(ROOT, "svod_amd", "csrc")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
                    "-Wl,-Bsymbolic", f"-I{csrc}", "-I/opt/rocm/include", os.path.join(csrc, "ops.cpp"), str(source), "-o", str(built)],
                   check=True, capture_output=True)
    return ctypes.CDLL(str(built))


def desc(at, *shape, dtype=0):
    return ctypes.byref(ops._Tensor(at, dtype, len(shape), (ctypes.c_int64 * 4)(*shape)))


def calls(lib):
    q = [desc(at, 2, 8, 4, 64) for at in (0x10000, 0x20000, 0x30000, 0x40000)]
    rows = [desc(at, 2, 8, 256) for at in (0x10000, 0x20000, 0x30000, 0x40000)]
    w, wide, none = desc(0x50000, 256), desc(0x60000, 256, 256), ctypes.c_void_p()
    attn, eps = ops._Attn(), ctypes.c_double(1e-6)
    return {
        "attention": lambda s: lib.svodk_attention(*q[:3], ctypes.byref(attn), q[3], s),
        "attention_packed": lambda s: lib.svodk_attention_packed(desc(0x10000, 2, 8, 12 * 64), 4, 4, ctypes.byref(attn), q[3], s),
        "heads": lambda s: lib.svodk_heads(desc(0x10000, 2, 8, 12 * 64), ctypes.byref(ops._Qkv(heads=4, kv_heads=4, head_dim=64, eps=1e-6)),
                                           *q[1:], s),
        "linear": lambda s: lib.svodk_linear(rows[0], wide, ctypes.byref(ops._Linear()), rows[1], s),
        "rms_norm": lambda s: lib.svodk_rms_norm(rows[0], w, eps, 0, rows[1], s),
        "add_layer_norm": lambda s: lib.svodk_add_layer_norm(rows[0], rows[1], w, none, eps, 0, rows[2], rows[3], s),
        "order_rows": lambda s: lib.svodk_order_rows(desc(0x10000, 8, dtype=3), desc(0x20000, 8, dtype=3), s),
    }


@pytest.mark.parametrize("name", ["attention", "attention_packed", "heads", "linear", "rms_norm", "add_layer_norm", "order_rows"])
def test_a_call_runs_on_its_streams_device(lib, name):
    call = calls(lib)[name]
    for stream, on in ((0x1000, 0), (0x1003, 3), (0, 0), (2, 0), (0x1001, 1)):
        assert call(ctypes.c_void_p(stream)) == 0
        assert lib.last_launch() == on, hex(stream)
        assert lib.current_device() == 0  # the caller's device is the caller's again
    assert call(ctypes.c_void_p(0x1002)) == 1 and lib.last_launch() == -1 and lib.current_device() == 0  # Fallback::Target
