"""CPU check of the built library: kernels that hide latency behind each other's
waves keep the registers that leave room for those waves.  Reads the kernel
descriptions (AMDGPU metadata note) of the code objects in libastrea_hip.so."""
import os
import re
import struct

import msgpack
import pytest

from astrea_amd import _lib as L


def _kernels():
    data = open(L.LIB_PATH, "rb").read()
    out = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        base = m.start()
        (count,) = struct.unpack_from("<Q", data, base + 24)
        at = base + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + n]
            at += 24 + n
            if b"gfx950" in name and size:
                out.update(_notes(data[base + off:base + off + size]))
    return out


def _notes(elf):
    (phoff,), (phnum,) = struct.unpack_from("<Q", elf, 32), struct.unpack_from("<H", elf, 56)
    for k in range(phnum):
        kind, _, start, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + 56 * k)
        at = start
        while kind == 4 and at < start + size:  # PT_NOTE
            n, d, tag = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (n + 3 & ~3)
            if tag == 32:  # NT_AMDGPU_METADATA
                for kernel in msgpack.unpackb(elf[desc:desc + d])["amdhsa.kernels"]:
                    yield kernel[".name"], kernel
            at = desc + (d + 3 & ~3)


# (reconstruction kernel, components, reconstructions, solvers or sweeps, waves per SIMD)
HYDRO1, HYDRO2, MHD2, ALL = 0x13, 0x17, 0x77, 0xFF
PLM, PPM, WENO3, WENO5, WENO7 = 1, 2, 3, 4, 5
LLF, HLLC, HLLD = 0, 1, 2
ROOM = [("recon2d", HYDRO2, (WENO3, WENO5, WENO7), (0, 1), 4), ("recon2d", MHD2, (WENO3, WENO5, WENO7), (0, 1), 3),
        ("sweep1d", HYDRO1, (WENO3, WENO5, WENO7), (LLF, HLLC), 4), ("sweep1d", ALL, (WENO3, WENO5), (LLF, HLLC), 3),
        ("sweep1d", ALL, (WENO7,), (LLF, HLLC), 2), ("sweep1d", ALL, (PLM, WENO3), (HLLD,), 3)]


@pytest.mark.parametrize("kernel,mask,recons,last,waves", ROOM, ids=str)
def test_registers_leave_room_for_the_waves(kernel, mask, recons, last, waves):
    if not os.path.exists(L.LIB_PATH):
        pytest.skip("library not built (run python -m astrea_amd._build)")
    found = 0
    for name, k in _kernels().items():
        m = re.match(rf"_ZN2ah14{kernel}_kernelIdLi{mask}ELi(\d)ELi(\d)ELi\d+E(?:Li\d+E)?Lb0E", name)
        if not m or int(m[1]) not in recons or int(m[2]) not in last:
            continue
        found += 1
        used = k[".vgpr_count"]  # accumulation registers included: one file of 512 per lane, in eights
        assert 512 // (used + 7 & ~7) >= waves and k[".vgpr_spill_count"] == 0, (name, used, k[".vgpr_spill_count"])
    assert found >= len(recons) * len(last)


@pytest.mark.parametrize("recon", [PPM, WENO5])
def test_hlld_of_many_tubes_leaves_room_for_three_waves(recon):
    """The 1D HLLD sweep that a launch of more than two workgroups per CU takes
    has the general divisions, whose registers leave room for a third wave."""
    if not os.path.exists(L.LIB_PATH):
        pytest.skip("library not built (run python -m astrea_amd._build)")
    found = [k for name, k in _kernels().items()
             if re.match(rf"_ZN2ah14sweep1d_kernelIdLi{ALL}ELi{recon}ELi{HLLD}ELi\d+ELb0ELi0ELb0E", name)]
    assert len(found) == 1
    assert 512 // (found[0][".vgpr_count"] + 7 & ~7) >= 3 and found[0][".vgpr_spill_count"] == 0


def test_2d_flux_tiles_of_hllc_leave_room_for_three_waves():
    """The 2D HLLC flux tiles of FP64 hydrodynamics, whose LDS lets three
    workgroups share a CU, keep the registers for it."""
    if not os.path.exists(L.LIB_PATH):
        pytest.skip("library not built (run python -m astrea_amd._build)")
    found = {name: k for name, k in _kernels().items()
             if re.match(rf"_ZN2ah13flux2d_kernelIdLi{HYDRO2}ELi({LLF}|{HLLC})ELi[012]ELi[01]ELi16ELi10ELb0ELi256ELin1E", name)}
    assert len(found) == 12
    for name, k in found.items():
        assert 512 // (k[".vgpr_count"] + 7 & ~7) >= 3 and k[".vgpr_spill_count"] == 0, (name, k[".vgpr_count"])
