"""csrc/include/chronos_lds.h on the host: a kernel's LDS attribute is set once on every device that launches it, and again where setting it failed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = r"""
#pragma once
enum hipError_t { hipSuccess, hipErrorUnknown };
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize };
extern int device, calls;
extern const void* last;
extern hipError_t get, set;
inline hipError_t hipGetDevice(int* d) { if (get == hipSuccess) *d = device; return get; }
inline hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int) { last = f; ++calls; return set; }
"""
MAIN = r"""
#include "chronos_lds.h"
#include <cstdio>
int device = 0, calls = 0;
const void* last = nullptr;
hipError_t get = hipSuccess, set = hipSuccess;
template <int N> void kern(int) {}
#define ASK(N, want) do { calls = 0; chronos::lds_limit<kern<N>>(1000); if (calls != want || (want && last != (const void*)kern<N>)) { std::printf("line %d: %d\n", __LINE__, calls); return 1; } } while (0)
int main() {
    ASK(0, 1); ASK(0, 0);
    ASK(1, 1); ASK(1, 0);               // a kernel of the same type is another one
    device = 1; ASK(0, 1); ASK(0, 0); ASK(1, 1);
    device = 0; ASK(0, 0); ASK(1, 0);
    device = 63; ASK(0, 1); ASK(0, 0);
    device = 64; ASK(0, 1); ASK(0, 1);  // no bit for it
    device = 2; set = hipErrorUnknown; ASK(0, 1); ASK(0, 1);
    set = hipSuccess; ASK(0, 1); ASK(0, 0);
    get = hipErrorUnknown; ASK(0, 1);
    std::puts("ok");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_once_per_kernel_and_device(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime_api.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(tmp_path), "-I", os.path.join(ROOT, "csrc", "include"), str(tmp_path / "main.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout


def test_launches_that_ask_for_it_keep_it_by_device():
    """The recurrences' chunks, the experts and the joined products: no attribute set once per process."""
    for name in ("hybrid/chunk_scan.hip", "hybrid/gla_scan.hip", "hybrid/moe_grouped.hip"):
        with open(os.path.join(ROOT, "csrc", name)) as f:
            text = f.read()
        assert "hipFuncSetAttribute" not in text and "lds_limit<" in text, name
