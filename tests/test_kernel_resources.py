"""Workgroups per CU that the registers of the built kernels allow, where the
schedule and its tuner count on them (tune.diag_slots, choose_kinds): read from
the metadata of libmfdag.so's own code objects, no GPU needed.  A gfx950 SIMD
has 512 vector registers per lane (a 256-thread workgroup puts one wave on each
of the four), a CU 160 KB of LDS."""
import struct

import msgpack
import pytest

import mfdag
from mfdag import tune


def kernels():
    """{mangled name: (vector registers, LDS bytes)} of every kernel."""
    with open(mfdag.LIB_PATH, "rb") as f:
        b = f.read()
    out, at = {}, b.find(b"\x7fELF", 1)
    while at > 0:
        if struct.unpack_from("<H", b, at + 18)[0] == 224:  # EM_AMDGPU
            table, = struct.unpack_from("<Q", b, at + 40)
            size, count = struct.unpack_from("<HH", b, at + 58)
            for h in range(at + table, at + table + size * count, size):
                if struct.unpack_from("<I", b, h + 4)[0] != 7:  # SHT_NOTE
                    continue
                q = at + struct.unpack_from("<Q", b, h + 24)[0]
                name, desc, kind = struct.unpack_from("<III", b, q)
                if kind != 32:  # NT_AMDGPU_METADATA
                    continue
                q += 12 + (name + 3) // 4 * 4
                for k in msgpack.unpackb(b[q:q + desc])["amdhsa.kernels"]:
                    out[k[".name"]] = (k[".vgpr_count"], k[".group_segment_fixed_size"])
        at = b.find(b"\x7fELF", at + 1)
    return out


def per_cu(name, elem_bytes):
    """Workgroups of each matching kernel per CU."""
    tag = f"{len(name)}{name}I{'d' if elem_bytes == 8 else 'f'}"
    found = [v for k, v in kernels().items() if tag in k]
    assert found, name
    return [min(512 // ((regs + 7) // 8 * 8), 163840 // lds) for regs, lds in found]


@pytest.mark.parametrize("elem_bytes", [8, 4])
def test_workgroups_per_cu(elem_bytes):
    many = tune.diag_slots(elem_bytes, tune.APART_DIAG) // tune.CUS
    assert all(w >= many for w in per_cu("k_diag", elem_bytes) + per_cu("k_small_front", elem_bytes))
    assert all(w >= tune.diag_slots(elem_bytes) // tune.CUS for w in per_cu("k_upd_diag", elem_bytes))
    # choose_kinds: two medium fronts per CU
    assert all(w >= 2 for w in per_cu("k_front_wg", elem_bytes))
