"""No kernel of the library keeps registers in scratch memory (CPU; read from the metadata that the
compiler stores beside each kernel of the library built here).

The persistent kernels run two waves a SIMD at up to 256 registers: what does not fit goes to
scratch, where every wave writes and reads it again, and the results do not show it.
"""
import re

from leanstream_amd import _native

SYMBOL = re.compile(rb"\.symbol(?:[\xa0-\xbf]|\xd9.|\xda..)([\w$.]+)\.kd", re.S)   # msgpack string


def number(data, at):
    """The msgpack unsigned integer at `at`."""
    if data[at] < 0x80:
        return data[at]
    width = {0xCC: 1, 0xCD: 2, 0xCE: 4, 0xCF: 8}[data[at]]
    return int.from_bytes(data[at + 1:at + 1 + width], "big")


def kernels():
    """{kernel: (scratch bytes a lane, spilled vector registers)}; a kernel's keys are sorted."""
    data = _native.LIBRARY_PATH.read_bytes()
    out = {}
    for m in re.finditer(rb"\.private_segment_fixed_size", data):
        spills = data.index(b".vgpr_spill_count", m.end())
        name = SYMBOL.search(data, m.end(), spills)[1].decode()
        out[name] = number(data, m.end()), number(data, spills + len(b".vgpr_spill_count"))
    return out


def test_no_kernel_spills():
    found = kernels()
    for family in ("fused_layer_kernel", "stage_a_kernel", "stage_b_kernel", "chain_kernel", "dense_gate_up_kernel",
                   "dense_down_kernel", "dense_reduce_kernel"):
        assert any(family in name for name in found), family
    assert {name: v for name, v in found.items() if any(v)} == {}
