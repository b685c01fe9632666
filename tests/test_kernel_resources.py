"""What the compiler gave the kernels of ``libimhip.so``, from the metadata of its code objects: registers and
private memory decide how many wavefronts a SIMD holds, and neither shows in a result."""

import os
import re
import struct

import pytest

from instantmimic_amd import build

msgpack = pytest.importorskip("msgpack")

_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
_NOTES, _AMDGPU_METADATA = 7, 32  # section and note types


def _kernels_of(elf: bytes):
    sections, (size, count) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        _, kind, _, _, at, _ = struct.unpack_from("<IIQQQQ", elf, sections + i * size)
        if kind == _NOTES:
            name, words, note = struct.unpack_from("<III", elf, at)
            if note == _AMDGPU_METADATA:
                start = at + 12 + -(-name // 4) * 4
                yield from msgpack.unpackb(elf[start : start + words], strict_map_key=False)["amdhsa.kernels"]


@pytest.fixture(scope="module")
def kernels():
    """{mangled name: metadata} of the library's gfx950 kernels."""
    with open(build.LIB, "rb") as f:
        lib = f.read()
    found, at = {}, lib.find(_MAGIC)
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", lib, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", lib, entry)
            if size and b"gfx950" in lib[entry + 24 : entry + 24 + length]:
                found.update((k[".name"], k) for k in _kernels_of(lib[at + offset : at + offset + size]))
            entry += 24 + length
        at = lib.find(_MAGIC, at + 1)
    return found


def _wavefronts(kernel) -> int:
    """Wavefronts that a SIMD's 512 registers a lane hold, handed out by eights."""
    return 512 // (-(-kernel[".vgpr_count"] // 8) * 8)


def test_start_of_a_solve_does_not_pay_for_the_wide_form(kernels):
    """Up to 64 dofs the launch needs 72 registers a lane, beyond 124: in one kernel every model had the four
    wavefronts per SIMD of the wide form."""
    starts = [k for n, k in kernels.items() if "newton_init_context_kernel" in n]
    assert max(map(_wavefronts, starts)) >= 5 and all(k[".private_segment_fixed_size"] == 0 for k in starts)


def test_resident_loops_stay_within_the_private_memory_they_are_admitted_with(kernels):
    """A resident kernel beyond the limit is left out at run time without a word, and its batches take a slower one."""
    with open(os.path.join(build.CSRC, "newton_solve.hip")) as f:
        limit = int(re.search(r"kResidentPrivate = (\d+);", f.read())[1])
    private = {n: k[".private_segment_fixed_size"] for n, k in kernels.items() if re.search(r"newton_(sparse|dense_tile|dense_wave)_resident_kernel", n)}
    assert len(private) == 22 and max(private.values()) <= limit <= 2 * max(private.values())


def test_kept_muscle_entries_stay_in_registers(kernels):
    """Up to four kept entries a thread (with six, six values are parked); sums that read ahead of their additions took
    twelve to twenty bytes of private memory a lane."""
    kept = [k for n, k in kernels.items() if re.search(r"muscle_world_kernelILi\dELi\d+ELi[24]E", n)]
    assert len(kept) == 12 and all(k[".private_segment_fixed_size"] == 0 for k in kept)


def test_line_search_with_eight_rows_a_lane_keeps_four_wavefronts(kernels):
    """Up to 256 rows: 128 registers a lane; a shorter form for the rows without friction beside the other took 131."""
    (search,) = [k for n, k in kernels.items() if "newton_linesearch_kernelILi8E" in n]
    assert _wavefronts(search) >= 4 and search[".private_segment_fixed_size"] == 0
