"""Host-checkable parts of the wide kernels (``csrc/ace_wide.hpp``), on the CPU:
the exact soft moments' fixed point and the launch geometry."""

from __future__ import annotations

import ctypes
import re
import struct
import subprocess
from pathlib import Path

import pytest
import torch

from ace_kernels import _lib
from ace_kernels.common import bin_tables

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "ace-kernels_amd" / "csrc"
MAX_LDS = 160 * 1024


@pytest.fixture(scope="module")
def lib(tmp_path_factory) -> ctypes.CDLL:
    out = tmp_path_factory.mktemp("wide") / "libwide.so"
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-std=c++17", "-ffp-contract=off", "-mfma", f"-I{CSRC}",
                    str(HERE / "wide_harness.cpp"), "-o", str(out)], check=True, capture_output=True)
    lib = ctypes.CDLL(str(out))
    ll = ctypes.c_longlong
    lib.check_exact_moments.restype = ll
    lib.check_exact_moments.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_double,
                                        ctypes.c_int]
    lib.wide_geometry.argtypes = [ll, ll, ll, *[ctypes.c_int] * 6, ctypes.POINTER(ll)]
    lib.exact_shift.argtypes = [ll, ctypes.c_int]
    lib.soft_forward_wide.argtypes = [ll, ll, ll, *[ctypes.c_int] * 3]
    return lib


def _half_edges(k: int) -> torch.Tensor:
    return bin_tables(k, True, torch.device("cpu"))[0]


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 10, 15, 16, 17, 20, 31, 32, 33, 50, 64, 100, 127, 128, 129, 255, 256,
                               257, 300, 511, 512])
def test_exact_moments(lib, k) -> None:
    """The offset of every probability is exact in float32, an integer from
    half-bin 1 on, and below 1.2 2^24: its square below 2^50.6."""
    table = _half_edges(k)
    assert lib.check_exact_moments(table.data_ptr(), k, 64, 4999, 1.2 * 2 ** 24, 0) == 0


def test_a_base_with_too_many_bits_fails(lib) -> None:
    """An odd base: h w is no float32 for the upper half-bins, or p 2^m - h w
    needs more than 24 bits."""
    table = _half_edges(20)
    assert lib.check_exact_moments(table.data_ptr(), 20, 64, 4999, 1.2 * 2 ** 24, 1) > 0


def test_shifts(lib) -> None:
    """A batch index's sums of u^2 (below 1.2^2 2^48) and of half-bin 0's
    2^16 u (below 2^40) stay inside int64 after their shift."""
    for bits in range(0, 41):
        n = (1 << bits) - 1
        assert n * 1.2 ** 2 * 2 ** 48 / 2 ** lib.exact_shift(n, 0) < 2 ** 63
        assert n * 2 ** 40 / 2 ** lib.exact_shift(n, 1) < 2 ** 63
        # and no bit of the squares is dropped that could stay
        shift = lib.exact_shift(n, 0)
        assert shift == 0 or (n + 1) * 1.2 ** 2 * 2 ** 48 / 2 ** (shift - 1) > 2 ** 63


@pytest.mark.parametrize("soft", [0, 1])
@pytest.mark.parametrize("labels", [0, 1])
@pytest.mark.parametrize("elem", [2, 4])
@pytest.mark.parametrize("backward", [0, 1])
def test_geometry(lib, soft, labels, elem, backward) -> None:
    """Every channel count has a variant that holds it; no copy counts more
    voxels than its field; the tiles cover the row; the LDS of both kernels at
    20 bins fits; and the workspace holds the final sums of every replica."""
    out = (ctypes.c_longlong * 9)()
    for c in range(1, 65):
        for n in (0, 1, 255, 256, 257, 20001, 128 ** 3):
            for k in (1, 20, 50, 512):
                for b, bg in ((1, 1), (3, 0)):
                    lib.wide_geometry(b, c, n, k, soft, bg, labels, elem, backward, out)
                    cmax, vec, copies, steps, lds_fwd, lds_bwd, tiles, ws_bytes, count = out
                    if k <= 20:
                        assert lds_fwd <= MAX_LDS - 16 and lds_bwd <= MAX_LDS
                    words = (10 if labels else 11) if soft else (2 if labels else 3)
                    assert ws_bytes >= b * words * (c - (1 - bg if c > 1 else 0)) * k * 8
                    assert c <= cmax <= max(c + 1, 1.46 * c) and vec in (1, 2, 4)
                    assert copies in (1, 2, 4, 8) and steps >= 1
                    assert count <= (4095 if soft else 2047), (c, n, k, count)
                    assert tiles * 256 * vec * steps >= n


@pytest.mark.parametrize("channels,bins,voxels,elem,most", [
    (14, 50, 143_312, 4, 512), (14, 100, 70_602, 4, 256), (20, 50, 250_047, 2, 512), (24, 50, 83_248, 2, 256),
    (24, 50, 499_280, 2, 768)])
def test_soft_backward_whole_rounds(lib, channels, bins, voxels, elem, most) -> None:
    """The half-bin coefficients leave room for one or two blocks of these
    soft gradients per CU: their blocks are no few more than a whole number of
    rounds."""
    out = (ctypes.c_longlong * 9)()
    lib.wide_geometry(1, channels, voxels, bins, 1, 1, 1, elem, 1, out)
    lds, tiles = out[5], out[6]
    round_ = 256 * (160 * 1024 // lds)
    assert round_ in (256, 512) and tiles <= most and most % round_ == 0


# measured on MI355X: (batch, channels, voxels, bins, labels), the kernel that was
# faster by a tenth or more
GENERIC_FASTER = [
    (1, 5, 198_476, 50, 1), (1, 8, 250_047, 32, 1), (1, 8, 250_047, 50, 1), (1, 8, 499_280, 100, 1),
    (16, 8, 8000, 50, 1), (1, 10, 198_476, 50, 1), (1, 12, 83_248, 50, 1), (1, 12, 166_375, 100, 1),
    (1, 3, 666_072, 100, 0), (1, 4, 499_280, 100, 0), (1, 5, 198_476, 50, 0), (2, 8, 29_791, 50, 0),
    (1, 8, 250_047, 100, 0), (1, 12, 166_375, 50, 0), (1, 16, 62_400, 50, 0)]
WIDE_FASTER = [
    (1, 5, 198_476, 20, 1), (2, 5, 1_376_256, 20, 1), (1, 8, 499_280, 20, 1), (1, 8, 2_000_376, 50, 1),
    (2, 8, 576, 10, 1), (1, 10, 796_000, 50, 1), (1, 14, 287_496, 50, 1), (1, 17, 59_582, 50, 1),
    (1, 24, 83_248, 50, 1), (1, 32, 125_000, 32, 1), (2, 4, 1_003_520, 20, 0), (1, 3, 2_666_000, 50, 0),
    (1, 6, 1_331_000, 20, 0), (1, 8, 1_000_000, 20, 0), (1, 1, 4_000_000, 20, 0), (1, 12, 333_270, 20, 0)]


def test_soft_forward_takes_the_faster_kernel(lib) -> None:
    for b, c, n, k, labels in GENERIC_FASTER:
        assert not lib.soft_forward_wide(b, c, n, k, 1, labels), (b, c, n, k, labels)
    for b, c, n, k, labels in WIDE_FASTER:
        assert lib.soft_forward_wide(b, c, n, k, 1, labels), (b, c, n, k, labels)


def test_soft_forward_rule_above_some_size(lib) -> None:
    """From some size on the wide kernel takes every larger problem of up to 50
    bins, and above 16 channels every problem."""
    for c in (1, 2, 3, 4, 5, 8, 9, 12, 16, 17, 40, 64):
        for k in (1, 10, 20, 50):
            wide = [lib.soft_forward_wide(1, c, 4 ** i, k, 1, 0) for i in range(1, 15)]
            assert wide[-1] and (c <= 16 or all(wide)), (c, k, wide)
            # a problem too small for many blocks may be wide too
            assert sum(a != b for a, b in zip(wide, wide[1:])) <= 2, (c, k, wide)


def _spills(path: Path) -> dict:
    """Kernel name -> vector registers spilled, from the metadata of the code
    objects in the built library."""
    msgpack = pytest.importorskip("msgpack")
    data = path.read_bytes()
    magic, out, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (at := data.find(magic, at)) >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, length = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" not in target or not size:
                continue
            elf = data[at + off:at + off + size]
            table, = struct.unpack_from("<Q", elf, 0x28)
            entry, count = struct.unpack_from("<HH", elf, 0x3a)
            for h in range(table, table + entry * count, entry):
                if struct.unpack_from("<I", elf, h + 4)[0] != 7:  # SHT_NOTE
                    continue
                note, = struct.unpack_from("<Q", elf, h + 0x18)
                name, desc, kind = struct.unpack_from("<III", elf, note)
                start = note + 12 + (name + 3) // 4 * 4
                assert kind == 32  # NT_AMDGPU_METADATA
                for k in msgpack.unpackb(elf[start:start + desc])["amdhsa.kernels"]:
                    out[k[".name"]] = k[".vgpr_spill_count"]
        at += len(magic)
    return out


def test_label_kernels_up_to_24_channels_do_not_spill() -> None:
    """Two tiles in flight stay in vector registers for class labels, both
    binnings and directions, but for a handful of registers."""
    kernel = re.compile(r"(fwd|bwd)_kernel_wideI\w+?Li(\d+)ELi\d+ELi\d+ELb([01])ELb1E")
    found = 0
    for name, spilled in _spills(_lib.LIB_PATH).items():
        m = kernel.search(name)
        if m and int(m.group(2)) <= 24:
            found += 1
            assert spilled <= 16, (name, spilled)
    assert found == 15 * 3 * 2 * 2  # variants x element types x binnings x directions
