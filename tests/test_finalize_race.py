"""A read that ends while its layer is being finalized (CPU).

A completion before finalize publishes nothing: finalize publishes what is READY by then. The
transport's READY store and its look at the phase, against finalize's store of the phase and its look
at READY, must not both pass each other, or the group is published by neither and the layer's
consumer waits for it until its bound.
"""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
RUNTIME = [ROOT / "leanstream_amd" / "csrc" / "runtime" / f for f in ("execution_queue.cpp", "weight_manager.cpp")]


def test_every_group_is_published_once(tmp_path):
    exe = tmp_path / "finalize_race"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "golden" / "finalize_race.cpp"),
                    *map(str, RUNTIME), "-lpthread", "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe), "500000"], check=True, capture_output=True, text=True, timeout=110).stdout
    assert out.split() == ["layers", "500000", "unpublished", "0", "failed", "0"], out
