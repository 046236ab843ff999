"""Properties of the prefill and the wave-specialized kernel that hold only if the compiler leaves its memory operations as they are written: they are read off the
gfx950 instructions of the library that this tree builds.  No GPU is needed."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "fp6_llm_amd", "libfp6mi.so")
OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump") or "") if os.path.exists(p)), None)

pytestmark = pytest.mark.skipif(OBJDUMP is None, reason="needs llvm-objdump of the ROCm compiler")


def code_objects(data):
    """The gfx950 ELF images in a shared library: every translation unit brings one bundle (magic, count, then per entry
    offset, size, length of the target's name, name)."""
    magic, pos = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (pos := data.find(magic, pos)) >= 0:
        at = pos + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, pos + len(magic))[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            if data[at + 24:at + 24 + length].endswith(b"gfx950") and size:
                yield data[pos + offset:pos + offset + size]
            at += 24 + length
        pos += len(magic)


def instructions(tmp_path_factory, kernel):
    """{symbol: [instruction, ...]} of every instance of a kernel."""
    kernels = {}
    with open(LIBRARY, "rb") as f:
        images = list(code_objects(f.read()))
    for i, image in enumerate(images):
        path = tmp_path_factory.mktemp("elf") / ("%d.elf" % i)
        path.write_bytes(image)
        table = subprocess.run([OBJDUMP, "-t", str(path)], capture_output=True, text=True, check=True).stdout
        names = sorted({line.split()[-1] for line in table.splitlines() if kernel in line and "." not in line.split()[-1]})
        if not names:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", "--disassemble-symbols=" + ",".join(names), str(path)],
                              capture_output=True, text=True, check=True).stdout
        name = None
        for line in text.splitlines():
            head = re.match(r"(?:[0-9a-f]+ )?<(\S+)>:$", line.strip())
            if head:
                name = head.group(1) if head.group(1) in names else name   # (a label inside a kernel stays part of it)
                kernels.setdefault(name, [])
                continue
            code = line.split("//")[0].strip()
            if name and code:
                kernels[name].append(code)
    return kernels


@pytest.fixture(scope="module")
def prefill_kernels(tmp_path_factory):
    """{symbol: [instruction, ...]} of every gemm_prefill instance."""
    kernels = instructions(tmp_path_factory, "gemm_prefill")
    assert len(kernels) == 8, sorted(kernels)   # four formats, with and without group exponents
    return kernels


def is_transfer(code):
    return code.startswith("buffer_load") and code.endswith(" lds")


def is_vector_memory(code):
    return re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", code) is not None


def test_prefill_transfers_have_their_whole_offset_range_checked(prefill_kernels):
    """A position beyond K reads as zero because its offset lies beyond the buffer's size.  The hardware compares the vector offset
    with the size less the scalar offset; a scalar offset larger than the size (one row in the buffer and K % 256 == 64) would
    leave that to the sign of a difference."""
    for name, code in prefill_kernels.items():
        transfers = [c for c in code if is_transfer(c)]
        assert len(transfers) == 24, name       # eight ahead of the loop, eight for each half block
        for c in transfers:
            scalar_offset = re.match(r"buffer_load_dwordx4 v\d+, s\[\d+:\d+\], (\S+) offen( offset:\d+)? lds$", c)
            assert scalar_offset and scalar_offset.group(1) == "0", (name, c)


def test_prefill_waits_cover_every_transfer(prefill_kernels):
    """Before the barrier of a half block a wavefront waits until all but the last n of its vector memory operations are done, n
    being the number of weight loads it issues after its last transfer.  Were there fewer of those, for instance because two had
    been merged, the wait would leave transfers open."""
    for name, code in prefill_kernels.items():
        counted = 0
        for i, c in enumerate(code):
            wait = re.match(r"s_waitcnt vmcnt\((\d+)\)", c)
            if not wait or int(wait.group(1)) == 0 or code[i + 1] != "s_barrier":
                continue
            counted += 1
            last = max(j for j in range(i) if is_transfer(code[j]))
            between = code[last + 1:i]
            assert not any(b.startswith(("s_cbranch", "s_branch", "s_setpc")) for b in between), name
            assert sum(is_vector_memory(b) for b in between) >= int(wait.group(1)), (name, c)
            first = max((j for j in range(last) if code[j] == "s_barrier"), default=0)
            assert sum(is_transfer(b) for b in code[first:i]) >= 8, name
        assert counted == 2, (name, counted)    # one for each half block


def test_wide_kernel_waits_cover_every_transfer(tmp_path_factory):
    """As for the prefill kernel: a chunk's barrier waits until all but the last n vector memory operations are done, n being the weight loads issued after
    the chunk's last transfer."""
    kernels = instructions(tmp_path_factory, "gemm_wide")
    assert len(kernels) == 48, sorted(kernels)   # four formats, with and without group exponents, six tiles
    for name, code in kernels.items():
        FM, GS, NT, RT, WK = map(int, re.search(r"gemm_wideILi(\d+)ELb([01])ELi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
        loads = RT * ((1 if FM == 21 else 2) + GS)
        counted = 0
        for i, c in enumerate(code):
            wait = re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", c)
            if not wait or int(wait.group(1)) != loads or code[i + 1] != "s_barrier":
                continue
            counted += 1
            last = max(j for j in range(i) if is_transfer(code[j]))
            between = code[last + 1:i]
            assert not any(b.startswith(("s_cbranch", "s_branch", "s_setpc")) for b in between), name
            assert sum(is_vector_memory(b) and not b.startswith("scratch") for b in between) >= int(wait.group(1)), (name, c)
            first = max(j for j in range(last) if code[j] == "s_barrier")
            assert sum(is_transfer(b) for b in code[first:i]) == NT, (name, i)
        assert counted == 2 * WK, (name, counted)


def test_span_kernel_waits_cover_every_transfer(tmp_path_factory):
    """The wide kernel's waits at the widths in between, where the transfers of a chunk do not divide evenly over the half steps."""
    kernels = instructions(tmp_path_factory, "gemm_span")
    assert len(kernels) == 48, sorted(kernels)   # four formats, with and without group exponents, six tiles
    for name, code in kernels.items():
        FM, GS, NT, RT, WK = map(int, re.search(r"gemm_spanILi(\d+)ELb([01])ELi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
        loads = RT * ((1 if FM == 21 else 2) + GS)
        counted = 0
        for i, c in enumerate(code):
            wait = re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", c)
            if not wait or int(wait.group(1)) != loads or code[i + 1] != "s_barrier":
                continue
            counted += 1
            last = max(j for j in range(i) if is_transfer(code[j]))
            between = code[last + 1:i]
            assert not any(b.startswith(("s_cbranch", "s_branch", "s_setpc")) for b in between), name
            assert sum(is_vector_memory(b) and not b.startswith("scratch") for b in between) >= loads, (name, c)
            first = max(j for j in range(last) if code[j] == "s_barrier")
            assert sum(is_transfer(b) for b in code[first:i]) == NT, (name, i)
        assert counted == 2 * WK, (name, counted)


def test_wave_specialized_kernels_of_128_rows_hold_no_exponents_in_registers(tmp_path_factory):
    """The loading wavefronts bring the group exponents of 128 rows as far ahead as the weights.  Loads of the arithmetic wavefronts (one 16-bit load a
    row tile and K block) were waited for at the barrier of every block, which made what the ring has under way no use."""
    kernels = {n: code for n, code in instructions(tmp_path_factory, "gemm_ws").items() if re.search(r"gemm_wsILi\d+ELb1ELi\d+ELi\d+ELi4E", n)}
    assert len(kernels) == 16, sorted(kernels)   # four formats, tiles of 48, 64, 80 and 96 columns
    for name, code in kernels.items():
        assert any(c.startswith("global_load_lds_ushort") for c in code), name
        assert not any(re.match(r"(global|flat|buffer)_load_[us]short", c) for c in code), name


def test_quantizer_chooses_its_arithmetic_before_a_block(tmp_path_factory):
    """quant_fused holds both arithmetics at each place where it converts a block (two strings each).  The general one once followed the fast one in a pass
    of its own, so that a row with a subnormal scale had its tile read and converted twice.  Registers that do not suffice go to scratch memory in the
    general one alone: between two conversions of the fast one there is no scratch access."""
    kernels = instructions(tmp_path_factory, "quant_fused")
    assert len(kernels) == 24, sorted(kernels)   # four formats, three types of weights, with and without group exponents
    for name, code in kernels.items():
        conversions = [i for i, c in enumerate(code) if c.startswith("v_cvt_scalef32_2xpk16")]
        places = 3 if "ILi" in name and re.search(r"ELi8ELi2E", name) and "EfLb" in name else 4   # two blocks in registers, one in LDS (16-bit weights), the others
        assert len(conversions) == places * 2 * 2, (name, len(conversions))
        scratch = [i for i, c in enumerate(code) if c.startswith("scratch")]
        assert len(scratch) <= 8, name
        for i in scratch:   # the conversion that follows a store or stands around a reload has the general arithmetic's clamps ahead of it
            after = next(j for j in conversions if j > i)
            before = max([j for j in conversions if j < i], default=max(0, after - 400))
            assert sum(c.startswith("v_min") for c in code[before:after]) >= 16, (name, i)


def test_tile_kernel_without_a_bias_holds_no_code_for_one(tmp_path_factory):
    """A branch in the epilogue that no launch without a bias takes cost gemm_tile a register or two, some instances spills, and 0.2 to 0.5 % of a call of 5 us: the
    bias has instances of its own, with one load more for every row tile."""
    kernels = instructions(tmp_path_factory, "gemm_tile")
    loads = {}
    for name, code in kernels.items():
        shape = re.search(r"gemm_tileI((?:L\w\d+E)+)Lb([01])EE", name)
        loads.setdefault(shape.group(1), {})[int(shape.group(2))] = sum(c.startswith(("global_load", "buffer_load", "flat_load")) for c in code)
    assert len(loads) == 26 * 2 * 4
    for shape, n in loads.items():
        RT = int(re.findall(r"Li(\d+)E", shape)[2])
        assert n[1] - n[0] == RT, (shape, n)


def test_dequantizer_writes_a_block_to_lds_before_it_reads_other_lanes_rows(tmp_path_factory):
    """dequant_native's lanes read back rows that other lanes of their wavefront wrote.  The source says so with a fence between the two (without one the order would rest on
    the compiler not telling a lane's own addresses apart), and every write stands ahead of every read in the built code."""
    with open(os.path.join(ROOT, "fp6_llm_amd", "csrc", "fp6mi_gemm.hip")) as f:
        body = re.search(r"void dequant_native\(.*?\n}\n", f.read(), re.S).group(0)
    write, read = body.index("reinterpret_cast<v8h *>(mine"), body.index("reinterpret_cast<const v4u *>(mine")
    order = [body.find(text, write) for text in ('__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront")', "__builtin_amdgcn_wave_barrier()", '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront")')]
    assert [write] + order + [read] == sorted([write] + order + [read])
    kernels = instructions(tmp_path_factory, "dequant_native")
    assert len(kernels) == 8, sorted(kernels)   # four formats, with and without group exponents
    for name, code in kernels.items():
        writes, reads = ([i for i, c in enumerate(code) if c.startswith(op)] for op in ("ds_write", "ds_read"))
        assert len(writes) >= 8 and len(reads) >= 8 and max(writes) < min(reads), name


def test_dequantizer_keeps_what_the_last_level_cache_holds(tmp_path_factory):
    """What dequant_native writes is read next.  Its outputs go past the caches only where they are larger than the memory-side cache; the others are written through to it."""
    for name, code in instructions(tmp_path_factory, "dequant_native").items():
        stores = [c for c in code if re.match(r"(buffer|global)_store_dwordx4", c)]
        assert sum(c.startswith("buffer") and c.endswith(" sc1") for c in stores) == 8 and sum(c.startswith("global") and c.endswith(" nt") for c in stores) == 8 and len(stores) == 16, (name, stores)
