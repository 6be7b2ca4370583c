"""Register and scratch use of kernels whose speed rests on it, from the metadata
the compiler wrote into the library's gfx950 code object.

The loss passes of 1024^2 run two workgroups of 16 wavefronts on a CU only with 64
vector registers or fewer and half the LDS: with 65, the gradient pass of 16 fields
takes 133 us instead of 95. The pass with the loss has to hold two transforms of
eight values and a sum in double there and spills a little.
"""
import re
import struct

import msgpack
import pytest

from s_spi_spring_amd import hipcore


def code_object_kernels():
    blob = open(hipcore.LIB_PATH, "rb").read()
    out = {}
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    assert at >= 0, "no uncompressed offload bundle in the library"
    count = struct.unpack_from("<Q", blob, at + 24)[0]
    p = at + 32
    for _ in range(count):
        off, size, idlen = struct.unpack_from("<QQQ", blob, p)
        ident = blob[p + 24:p + 24 + idlen].decode()
        p += 24 + idlen
        if "gfx950" not in ident:
            continue
        elf = blob[at + off:at + off + size]
        shoff, = struct.unpack_from("<Q", elf, 40)
        shentsize, shnum = struct.unpack_from("<HH", elf, 58)
        for i in range(shnum):
            kind, _, _, s_off, s_size = struct.unpack_from("<IQQQQ", elf, shoff + i * shentsize + 4)
            if kind != 7:       # SHT_NOTE
                continue
            q, end = s_off, s_off + s_size
            while q < end:
                namesz, descsz, ntype = struct.unpack_from("<III", elf, q)
                d = q + 12 + (namesz + 3) // 4 * 4
                if ntype == 32:     # NT_AMDGPU_METADATA
                    for k in msgpack.unpackb(elf[d:d + descsz])["amdhsa.kernels"]:
                        out[k[".name"]] = k
                q = d + (descsz + 3) // 4 * 4
    return out


@pytest.fixture(scope="module")
def kernels():
    return code_object_kernels()


def named(kernels, pattern):
    found = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert found, pattern
    return found


def test_loss_passes_of_1024_run_two_workgroups_on_a_cu(kernels):
    for name, k in named(kernels, r"k_col_lossILi1024ELi0ELb").items():
        scratch = k[".private_segment_fixed_size"]
        assert k[".vgpr_count"] <= 64 and scratch <= (32 if "ELb1E" in name else 0), (name, k[".vgpr_count"], scratch)
        assert 2 * k[".group_segment_fixed_size"] <= 160 * 1024, name


SIZES = [64, 128, 256, 384, 512, 768, 1024, 2048]


def test_every_column_variant_has_its_own_passes(kernels):
    """A variant that a caller sets runs its own kernels, not another variant's in its place."""
    for n in SIZES:
        steps = any(hipcore.row_variant_recomputes_state(n, r) for r in range(hipcore.variant_counts(n)[1]))
        for v in range(hipcore.variant_counts(n)[0]):
            named(kernels, rf"5k_colILi{n}ELi0ELi{v}EE")
            for mode in range(3 if steps else 0):
                named(kernels, rf"10k_col_stepILi{n}ELi{mode}ELi{v}EE")


def test_compiled_choice_of_the_iteration_passes_spills_nothing(kernels):
    for n in SIZES[2:]:
        col, row = hipcore.default_variants(n)
        for name, k in named(kernels, rf"(10k_col_stepILi{n}ELi[01]ELi{col}EE|12k_row_listedILi{n}ELi\dELi{row}EE)").items():
            # 2048^2: 32 values of 8 bytes, field and state, in 128 registers
            assert k[".private_segment_fixed_size"] <= (64 if n == 2048 else 0), (name, k[".private_segment_fixed_size"])


def test_on_chip_blocks_spill_little(kernels):
    for name, k in named(kernels, r"k_iter_fusedILi(64|128)").items():
        assert k[".private_segment_fixed_size"] <= 16, (name, k[".private_segment_fixed_size"])
