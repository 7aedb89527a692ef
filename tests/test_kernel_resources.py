"""What the compiled kernels hold on a compute unit: registers, scratch memory and workgroups side by side, read off what the compiler
wrote beside each kernel of the built libraries.  A change that costs a kernel a workgroup or makes it spill shows here."""
import re
import struct

import pytest

from deliverance_amd.kernels import build

msgpack = pytest.importorskip("msgpack")

LDS = 160 * 1024                 # bytes of a compute unit
LANES, REGISTERS = 64, 512       # of a wavefront; vector registers of a SIMD, four SIMDs a compute unit


def _code_objects(blob):
    """The gfx950 code objects of a library (each a bundle of one entry a target: offset, size, name)."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", -1
    while (at := blob.find(magic, at + 1)) >= 0:
        n, q = struct.unpack_from("<Q", blob, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", blob, q)
            if b"gfx950" in blob[q + 24:q + 24 + length]:
                yield blob[at + offset:at + offset + size]
            q += 24 + length


def _notes(elf):
    """The kernels' descriptions in an ELF file's note sections."""
    table = struct.unpack_from("<Q", elf, 40)[0]
    entry, n = struct.unpack_from("<HH", elf, 58)
    for i in range(n):
        kind, = struct.unpack_from("<I", elf, table + i * entry + 4)
        if kind == 7:
            offset, = struct.unpack_from("<Q", elf, table + i * entry + 24)
            name, size, _ = struct.unpack_from("<III", elf, offset)
            yield from msgpack.unpackb(elf[offset + 12 + (name + 3) // 4 * 4:][:size])["amdhsa.kernels"]


def resources(unit, kernel):
    """Template arguments -> (workgroups a compute unit, scratch bytes a lane) of the kernels of this name."""
    try:
        build.build(only=[unit], verbose=False)
    except build.KernelLibraryError as e:
        pytest.skip(str(e))
    with open(build.unit_path(unit), "rb") as f:
        blob = f.read()
    found = {}
    for elf in _code_objects(blob):
        for k in _notes(elf):
            m = re.match(r"_Z\d+%s((?:I(?:L[a-z]\d+E)+E)?)" % kernel, k[".name"])
            if m:
                waves = -(-k[".max_flat_workgroup_size"] // LANES)
                a_simd = min(8, REGISTERS // (-(-max(1, k[".vgpr_count"]) // 8) * 8))
                fit = min(4 * a_simd // waves, LDS // max(1, k[".group_segment_fixed_size"]))
                found[tuple(int(x) for x in re.findall(r"L[a-z](\d+)E", m[1]))] = (fit, k[".private_segment_fixed_size"])
    assert found, f"{kernel} is not in {unit}"
    return found


@pytest.mark.parametrize("unit", ["attn_decode", "attn_decode_rel"])
def test_decode_attention_fits_side_by_side_and_does_not_spill(unit):
    """Three workgroups of 8 wavefronts a compute unit for head sizes up to 32, two up to 64; no scratch memory up to a head size of 128, and above, where two
    pieces of keys and all results fill the registers, no more than a few numbers a lane."""
    found = resources(unit, unit + "_kernel")
    assert {a[:2] for a in found} == {(1, 16), (2, 16), (1, 8), (2, 8), (4, 8), (8, 8)}
    for (dk, waves, split), (workgroups, scratch) in found.items():
        assert workgroups >= ({1: 3, 2: 2}.get(dk, 1) if waves == 8 else 1), (dk, waves, split)
        assert scratch <= (60 if dk == 8 else 0), (dk, waves, split)


def test_prefill_attention_fits_side_by_side_and_does_not_spill():
    """The form for long steps (4 row blocks, no phases): three workgroups a compute unit at head sizes of 48 and 64 where q is asked for first, two with a
    bias at 80; head sizes of 240 and 256 spill what their results leave no room for and no more."""
    found = resources("attn_prefill", "attn_prefill_kernel")
    late = {a[:4] for a in found if a[4]}
    assert late == {(4, 4, 1, 0), (4, 4, 1, 1)}
    for (d16, blocks, phases, table, q_late), (workgroups, scratch) in found.items():
        if (blocks, phases) == (4, 1):
            assert workgroups >= (3 if d16 in (3, 4) and table and not q_late else 2 if d16 <= 4 else 1), (d16, table, q_late)
            assert scratch <= {15: 44, 16: 208}.get(d16, 0), (d16, table, q_late)
    for (d16, blocks, phases, table, q_late), (workgroups, scratch) in resources("attn_prefill_rel", "attn_prefill_rel_kernel").items():
        if (blocks, phases) == (4, 1):
            assert workgroups >= (2 if d16 <= 5 else 1) and scratch == 0, (d16, table, q_late)


def test_norm_and_product_of_few_rows_run_side_by_side():
    """gemm_ln_quads: steps whose launch is up to two workgroups a compute unit have them side by side (a wide workgroup alone would leave half of them for a
    second round); no scratch memory; every kernel that is compiled is one that some call asks for.  Which kernel a row goes to does not hang on the columns, but for 5 to 8
    rows with K from 641 to 1,024."""
    from deliverance_amd.kernels import ops
    found = resources("gemm_fused", "gemm_ln_quads_kernel")
    lib, asked = ops._lib(), set()
    columns = (1, 4, 8, 256, 768, 1024, 1500, 2304, 3072, 4096, 4800, 5120, 6144, 6400, 7168, 8192, 8193, 9600, 10240, 10241, 12800, 14336, 14337, 15360, 16384, 50257)
    for M in (1, 4, 5, 8):
        for K in range(8, 2049, 8):
            for dtype in (ops.F32, ops.BF16):
                cols = [lib.da_gemm_bf16_ln_choice(M, N, K, dtype) for N in columns]
                assert all(cols) or not any(cols) or (M > 4 and 640 < K <= 1024)
                for N, c in zip(columns, cols):
                    if not c:
                        continue
                    form = ((1 if M <= 4 else 2), -(-c // 4), *((4, 1) if K <= 512 else (4, 2) if K <= 1024 else (6, 2) if K <= 1536 else (8, 2)), int(dtype == ops.BF16))
                    asked.add(form)
                    workgroups, scratch = found[form]
                    assert scratch == 0 and c <= 32
                    if lib.da_can_fuse_ln(M, K, N) and 256 < -(-N // c) <= 512:
                        assert workgroups >= 2, (M, K, N, c, dtype)
    assert asked == set(found)
