"""Kernels of the built library: none that its dispatch never launches, and what
their layout and registers are meant to give."""
import os
import re
import subprocess

import pytest

import test_isa_store_form as isa

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lattice-qcd-rs_amd", "lqcd",
                   "liblqcd_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def symbols(code_objects, part):
    """Kernel symbols that contain `part`."""
    for path in code_objects:
        for s in re.findall(rb"_ZN4lqcd\w+", path.read_bytes()):
            s = s.decode()
            if part in s and not s.endswith("kd"):
                yield s


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
@pytest.mark.parametrize("kernel", ["k_gauss_start", "k_gauss_links"])
def test_transports_are_built_for_the_dimensions_that_take_them(kernel):
    """gauss_uses_transports: not D = 3."""
    data = open(LIB, "rb").read()
    name = f"{len(kernel)}{kernel}ILi%dE".encode()
    assert [d for d in (2, 3, 4) if name % d in data] == [2, 4]


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    tmp, paths = tmp_path_factory.mktemp("co"), []
    for k, o in enumerate(isa.gfx950_code_objects(open(LIB, "rb").read())):
        paths.append(tmp / f"co{k}.elf")
        paths[-1].write_bytes(o)
    return paths


def kernel_object(code_objects, symbol):
    found = [p for p in code_objects if symbol.encode() in p.read_bytes()]
    assert len(found) == 1, (symbol, found)
    return str(found[0])


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(isa.OBJDUMP)),
                    reason="library not built or llvm-objdump absent")
def test_f32_normalisation_reads_the_two_columns_it_needs(code_objects):
    """Columns 0 and 1 are three 16-byte words of an f32 link (fields.hpp)."""
    symbol = next(s for s in symbols(code_objects, "k_reunitarizeIf"))
    out = subprocess.run([isa.OBJDUMP, "-d", "--mcpu=gfx950", f"--disassemble-symbols={symbol}",
                          kernel_object(code_objects, symbol)], capture_output=True, text=True, check=True).stdout
    loads = re.findall(r"buffer_load_dword(x\d)?", out)
    assert loads == ["x4"] * 3


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(READELF)),
                    reason="library not built or llvm-readelf absent")
@pytest.mark.parametrize("kernel", ["k_drift", "k_reunitarize", "k_links_from_aos", "k_links_to_aos"])
def test_link_kernels_hold_their_matrices_in_registers(code_objects, kernel):
    """No LDS and no scratch: a matrix that the compiler leaves in memory costs
    the small lattices two thirds of their time."""
    n = 0
    for path in code_objects:
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for entry in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
            symbol = re.search(r"\.symbol:\s+(\S+)", entry).group(1)
            if f"{len(kernel)}{kernel}I" not in symbol:
                continue
            n += 1
            assert int(re.search(r"\.group_segment_fixed_size:\s+(\d+)", entry).group(1)) == 0, symbol
            assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", entry).group(1)) == 0, symbol
    assert n > 0
