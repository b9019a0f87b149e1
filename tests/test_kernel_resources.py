"""What the pivot panels' kernels take of the hardware, from the metadata of the built library: the panel is held in
registers, so a register in scratch memory (a spill, an array indexed by a variable, a called function's frame)
defeats it, and it must not come back unnoticed."""
import os
import re

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparsedirectsolver.jl_amd", "csrc",
                   "libsds_hip.so")


def _kernels():
    data = open(LIB, "rb").read()
    out = {}
    for at in re.finditer(b"amdhsa.kernels", data):
        u = msgpack.Unpacker(raw=False, strict_map_key=False)
        u.feed(data[at.start() - 2:at.start() + (1 << 20)])  # (the map's and the key's header bytes before the name)
        for k in u.unpack()["amdhsa.kernels"]:
            out[k[".name"]] = k
    return out


@pytest.mark.skipif(not os.path.exists(LIB), reason="the library is not built")
@pytest.mark.parametrize("kernel,classes", [("k_ldlt_panel", 8), ("k_lu_panel", 8)])
def test_pivot_panels_use_no_scratch_memory(kernel, classes):
    found = {n: k for n, k in _kernels().items() if kernel + "I" in n}
    assert len(found) == classes
    for name, k in found.items():
        assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_spill_count"] == 0, (name, k)
        assert not k.get(".uses_dynamic_stack", False), name
