"""What a handle asks of the device, checked on the CPU: the library's HIP
calls go to the stand-ins of tests/host/handle_check.c, which run no kernels."""
import os
import subprocess

import pytest

import pvof

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "parties-vof-ibm_amd")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    pvof.load_lib()                                   # builds it if nothing is there
    out, so = str(tmp_path_factory.mktemp("handle") / "handle_check"), os.path.join(PKG, "_build")
    subprocess.run(["gcc", "-O1", "-std=gnu99", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-rdynamic", "-o", out,
                    os.path.join(HERE, "host", "handle_check.c"), "-L" + so, "-lparties_vof", "-Wl,-rpath," + so,
                    "-Wl,-rpath-link,/opt/rocm/lib", "-Wl,--allow-shlib-undefined"], check=True, capture_output=True)
    return out


def check(exe, *args):
    r = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return {k: int(v) for k, v in (line.split() for line in r.stdout.splitlines())}


# odd and even numbers of rows, pitches of an odd and an even number of lines
SIZES = [(8, 8), (96, 96), (768, 491), (88, 56), (64, 33), (9, 13), (256, 128)]


@pytest.mark.parametrize("nx,ny", SIZES)
def test_fields_start_on_a_line(exe, nx, ny):
    """Cell (0, 0) of every field, which kernels read in pairs of doubles."""
    assert check(exe, "layout", nx, ny)["field"] == 0


@pytest.mark.parametrize("nx,ny", [s for s in SIZES if s[0] % 16 == 0])
def test_row_tables_start_on_a_pair(exe, nx, ny):
    """Cosines and twiddles of the row transforms, read in pairs of doubles."""
    got = check(exe, "layout", nx, ny)
    assert got["rtx"] == 0 and got["wx"] == 0


# bottoms of an even number of cells and of an odd one (88 x 56 -> 11 x 7, 18 x 26 -> 9 x 13), the grid
# itself the bottom, and three levels above it
@pytest.mark.parametrize("nx,ny", [(8, 8), (13, 15), (18, 26), (88, 56), (96, 96), (176, 112), (512, 256)])
def test_multigrid_arrays_start_on_a_pair(exe, nx, ny):
    got = check(exe, "layout", nx, ny)
    assert got["level"] == 0 and got["H"] == 0 and got["r2"] == 0


# the longest rows (powers of two and 2^a 3^b), whose padded transforms take more than 64 KiB, and the
# longest that do not
@pytest.mark.parametrize("nx,large", [(4096, 1), (3888, 1), (3456, 0), (2048, 0), (16, 0)])
def test_row_transforms_are_allowed_their_lds(exe, nx, large):
    got = check(exe, "lds", nx, 9)
    assert (got["large"] > 0) == bool(large) and got["refused"] == 0


# part of one staging buffer, several
@pytest.mark.parametrize("nx,ny", [(8, 8), (1000, 700)])
def test_transfers_are_complete_on_return(exe, nx, ny):
    """Setting and reading a field leave nothing queued, whether the array is
    on the host (staged) or on the device (a strided copy)."""
    got = check(exe, "transfers", nx, ny)
    got.pop("pinned")
    assert got == dict(set=0, get=0, device_set=0, device_get=0, wrong=0)


@pytest.mark.parametrize("nx,ny", [(8, 8), (96, 96), (505, 505), (1000, 700)])
def test_transfers_pin_no_more_than_they_stage(exe, nx, ny):
    """Two buffers of a field, or of 2 MiB where a field is larger."""
    assert check(exe, "transfers", nx, ny)["pinned"] <= 2 * min(8 * (nx + 7) * (ny + 7), 2 << 20)
