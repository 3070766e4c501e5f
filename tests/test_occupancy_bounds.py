"""The autotuner's variants with a minimum of waves per SIMD can have that many:
registers (512 per lane and SIMD, allotted by eights) and LDS (160 KB a CU)
of each such kernel, from the metadata that the compiler leaves in the
library, allow the bound its name states."""
import os
import re
import struct

import pytest

from dynearthsol_amd import lib

msgpack = pytest.importorskip("msgpack")
pytestmark = pytest.mark.skipif(not os.path.exists(lib.LIB_PATH), reason="library not built")

# mangled template arguments: dimension, staged, waves (A, E, where it has a bound); dimension, waves, staged (C)
BOUNDED = [re.compile(r"8k_pass_[ae]ILi[23]ELb[01]ELi(\d+)E"), re.compile(r"8k_pass_cILi[23]ELi(\d+)E"),
           re.compile(r"14k_pass_c_mixedILi[23]ELi(\d+)E")]


def _kernels():
    blob = open(lib.LIB_PATH, "rb").read()
    for m in re.finditer(rb"AMDGPU\0\0", blob):        # ELF note: name size, description size, type, name, description
        name, size, kind = struct.unpack("<III", blob[m.start() - 12:m.start()])
        if name == 7 and kind == 32:
            yield from msgpack.unpackb(blob[m.end():m.end() + size])["amdhsa.kernels"]


def test_variants_reach_their_waves_per_simd():
    seen = set()
    for k in _kernels():
        bound = next((int(m.group(1)) for m in (p.search(k[".name"]) for p in BOUNDED) if m), None)
        if bound is None:
            continue
        assert k[".max_flat_workgroup_size"] == 256      # a wave per SIMD and block
        waves = min(512 // max(-(-k[".vgpr_count"] // 8) * 8, 1), 8)
        blocks = 163840 // max(k[".group_segment_fixed_size"], 1)
        print(k[".name"], "bound", bound, "registers allow", waves, "LDS", blocks)
        assert min(waves, blocks) >= bound, k[".name"]
        seen.add(bound)
    assert {1, 2, 3, 4, 6} <= seen, seen
