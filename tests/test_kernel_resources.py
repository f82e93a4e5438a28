"""Registers and record loads of the tiled FP64 kernels, from the object file
of this build (no GPU): what their occupancy and latency rest on, which a
change elsewhere in the shared headers can take away without a word."""
import re
import subprocess
from pathlib import Path

import pytest

LLVM = Path("/opt/rocm/llvm/bin")
OBJ = Path(__file__).resolve().parents[1] / "rc_amd" / "_obj" / "rcg_tiled.o"


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    if not OBJ.exists():
        pytest.skip("no object file of this build")
    d = tmp_path_factory.mktemp("code")
    o = d / OBJ.name
    o.write_bytes(OBJ.read_bytes())
    subprocess.run([LLVM / "llvm-objdump", "--offloading", o.name], cwd=d, check=True,
                   capture_output=True)
    return next(d.glob("*gfx950"))


def kernels(code):
    """{name: (SGPRs, VGPRs)} of the code object's metadata."""
    text = subprocess.run([LLVM / "llvm-readelf", "--notes", code], check=True,
                          capture_output=True, text=True).stdout
    out = {}
    for part in text.split(".agpr_count")[1:]:
        get = lambda key: re.search(key + r":\s+(\S+)", part).group(1)  # noqa: E731
        out[get(r"\.name")] = int(get(r"\.sgpr_count")), int(get(r"\.vgpr_count"))
    return out


@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("kernel", ["k_grid_tiles_f64", "k_degrid_tiles_f64"])
def test_eight_workgroups_a_cu(code, kernel, tile):
    """Eight workgroups of four wavefronts: at most 64 VGPRs and 96 SGPRs (an
    allocation of 112 leaves room for seven)."""
    (sgpr, vgpr), = [v for n, v in kernels(code).items() if f"{kernel}ILi{tile}E" in n]
    assert sgpr <= 96 and vgpr <= 64


@pytest.mark.parametrize("tile", [16, 32, 64])
def test_records_by_the_scalar_path(code, tile):
    """The FP64 degridder's vector loads are the item's range (two or three),
    the tile's cells and the taps: no record words among them."""
    name, = [n for n in kernels(code) if f"k_degrid_tiles_f64ILi{tile}E" in n]
    name = name.removesuffix(".kd")
    text = subprocess.run([LLVM / "llvm-objdump", "-d", f"--disassemble-symbols={name}", code],
                          check=True, capture_output=True, text=True).stdout
    loads = re.findall(r"\bglobal_load_\w+", text)
    assert loads.count("global_load_dwordx4") == 2
    assert 4 <= len(loads) <= 5
