"""Control-plane parity with LeanStream's own runtime (CPU).

tests/golden/runtime_trace.cpp drives ExecutionQueue, WeightManager (through a manual
IOBackend), KernelSelector and Runtime/LayerStep through scripted scenarios and prints a
canonical trace: queue words, ready_indices in publication order, every descriptor, every
return code and every IOBackend call. tests/golden/runtime_trace.txt is that trace produced
by LeanStream's runtime sources compiled into oracle/_ref (tests/golden/make_runtime_trace.sh).
This repository's runtime must reproduce it line for line: descriptors, publication order
and queue state are bit-exact requirements.
"""
import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
GOLDEN = ROOT / "tests" / "golden" / "runtime_trace.txt"
DRIVER = ROOT / "tests" / "golden" / "runtime_trace.cpp"
RUNTIME = ["execution_queue.cpp", "kernel_selector.cpp", "weight_manager.cpp", "runtime.cpp"]


def _build(tmp_path, name, sources, extra=()):
    exe = tmp_path / name
    cmd = ["g++", "-O1", "-std=c++17", "-UNDEBUG", f"-I{ROOT / 'include'}", *map(str, sources), *extra, "-lpthread",
           "-o", str(exe)]
    subprocess.run(cmd, check=True, capture_output=True)
    return exe


def _first_difference(a, b):
    for i, (x, y) in enumerate(zip(a, b)):
        if x != y:
            return i, x, y
    return min(len(a), len(b)), None, None


def test_runtime_reproduces_reference_trace(tmp_path):
    exe = _build(tmp_path, "trace_mine", [DRIVER] + [ROOT / "leanstream_amd" / "csrc" / "runtime" / f for f in RUNTIME])
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()
    want = GOLDEN.read_text().splitlines()
    i, got_line, want_line = _first_difference(out, want)
    assert out == want, f"first difference at line {i + 1}: got {got_line!r}, reference {want_line!r}"
    assert want[-1] == "== end" and len(want) > 100


def test_golden_trace_is_current_with_the_reference_build():
    """Where LeanStream's sources are present (not on GPU test machines), the committed fixture
    must still be what the reference runtime prints."""
    ref = ROOT / "oracle" / "_ref" / "runtime_trace_ref"
    if not Path(os.environ.get("LEANSTREAM_REFERENCE", "/root/reference"), "src", "runtime").is_dir():
        pytest.skip("reference sources not present")
    if not ref.is_file():
        subprocess.run(["make", "-s", "-C", str(ROOT / "oracle"), "ref-trace"], check=True, capture_output=True)
    out = subprocess.run([str(ref)], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()
    assert out == GOLDEN.read_text().splitlines()


SELECTOR_ALLOC = r'''
#include "leanstream/kernel_selector.h"
#include <cstdio>
#include <cstdlib>
#include <new>
static unsigned long allocations = 0;
void* operator new(size_t n) { ++allocations; if (void* p = std::malloc(n ? n : 1)) return p; throw std::bad_alloc(); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
using namespace leanstream::runtime;
int main() {
    uint8_t lut[4 * 8];
    for (int i = 0; i < 32; ++i) lut[i] = (uint8_t)(i % 7);   // ids 5, 6 are out of the catalog
    KernelSelector s({lut, 4, 8});
    unsigned long sum = 0, before = allocations;
    for (int r = 0; r < 20000; ++r)
        for (uint32_t l = 0; l < 5; ++l)
            for (uint32_t b = 0; b < 9; ++b) {
                sum += s.select(l, b) + s.plan({l, b}).candidate.workers;
                sum += quantize_io_load(r, 20000, 8);
            }
    std::printf("%lu %lu\n", allocations - before, sum);
    return allocations == before ? 0 : 1;
}
'''


def test_kernel_selection_is_allocation_free(tmp_path):
    """kernel_selector_test.cpp:44-50: selection and planning never allocate."""
    src = tmp_path / "alloc.cpp"
    src.write_text(SELECTOR_ALLOC)
    exe = _build(tmp_path, "alloc", [src, ROOT / "leanstream_amd" / "csrc" / "runtime" / "kernel_selector.cpp"])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split()[0] == "0"
