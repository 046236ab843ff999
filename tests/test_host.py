"""CPU-side product code (libfp6mi.so through the C ABI and the Python API) against the oracle and the golden fixtures.
No GPU compute is called here; the library must load and export every symbol that include/fp6mi.h declares."""
import ctypes
import decimal
import fractions
import glob
import hashlib
import json
import os
import re
import subprocess
import sys

import numpy as np
import pytest
import torch

import oracle
import fp6_llm_amd as fp6
from fp6_llm_amd import _lib, quant, synth

FORMATS = [(3, 2), (2, 2), (2, 3), (2, 1)]
BLOCK_BYTES = {6: 3072, 5: 2560, 4: 2048}   # native layout: bytes of a 16-row x 256-column block, by bit width
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _problem(seed, OC, IC, E, M):
    raw, sc, _ = synth.uniform_problem(seed, OC, IC, 1, E, M)
    return raw, sc


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "fp6mi.h")).read()
    declared = set(re.findall(r"\b(fp6mi_[a-z0-9_]+)\s*\(", header))
    assert declared and declared == set(_lib.EXPORTED)
    L = _lib.lib()
    for name in declared:
        assert hasattr(L, name), name
    assert L.fp6mi_version() >= 100
    assert b"success" in L.fp6mi_error_string(0)


def test_golden_prepack_fixtures(golden_dir):
    for f in sorted(glob.glob(os.path.join(golden_dir, "prepack_e*_*.npz"))):
        E, M = (int(v) for v in re.search(r"prepack_e(\d)m(\d)_", f).groups())
        z = np.load(f)
        raw = np.ascontiguousarray(z["raw"])
        OC, IC = raw.shape[0], raw.shape[1] * 32 // (1 + E + M)
        got = np.empty_like(raw)   # through the C ABI: the Python wrapper keeps the reference's OC % 256 rule
        assert _lib.lib().fp6mi_prepack_ref(E, M, got.ctypes.data, raw.ctypes.data, OC, IC) == 0
        assert got.tobytes() == z["packed"].tobytes(), f


@pytest.mark.parametrize("E,M", FORMATS)
def test_prepack_hash_at_benchmark_size(golden_dir, E, M):
    """Config 2 size (4096x4096): bytes identical to what the reference's prepacker produced (committed SHA-256)."""
    ref = json.load(open(os.path.join(golden_dir, "prepack_hashes.json")))["e%dm%d_4096x4096_seed2001" % (E, M)]
    raw = quant.pack_raw(synth.uniform_codes(2001, 4096, 4096, E, M), E, M)
    assert hashlib.sha256(raw.tobytes()).hexdigest() == ref["raw_sha256"]
    packed = fp6.weight_prepacking_eXmY_cpu(E, M, torch.from_numpy(raw)).numpy()
    assert hashlib.sha256(packed.tobytes()).hexdigest() == ref["packed_sha256"]


@pytest.mark.parametrize("E,M", FORMATS)
@pytest.mark.parametrize("OC,IC", [(256, 64), (256, 320), (512, 1024)])
def test_prepack_dequant_native_against_oracle(E, M, OC, IC):
    raw, sc = _problem(OC + IC, OC, IC, E, M)
    t = torch.from_numpy(raw)
    packed = fp6.weight_prepacking_eXmY_cpu(E, M, t)
    assert packed.shape == t.shape and packed.dtype == torch.int32
    assert packed.numpy().tobytes() == oracle.prepack(raw, E, M).tobytes()
    dq = fp6.weight_dequant_eXmY_cpu(E, M, t, torch.from_numpy(sc)).numpy()
    assert dq.shape == (OC, IC)
    assert (dq.view(np.uint16) == oracle.dequant(raw, sc, E, M).view(np.uint16)).all()
    # native layout: same bits by both routes, and a lossless round trip
    nat = fp6.weight_prepacking_native_cpu(E, M, t)
    assert nat.numel() * 4 == fp6.native_bytes(E, M, OC, IC) == (OC // 16) * ((IC + 255) // 256) * BLOCK_BYTES[1 + E + M]
    assert torch.equal(nat, fp6.to_native(packed, E, M))
    L = _lib.lib()
    back = np.empty_like(raw)
    assert L.fp6mi_unpack_native(E, M, back.ctypes.data, nat.data_ptr(), OC, IC) == 0 and (back == raw).all()
    back2 = np.empty_like(raw)
    assert L.fp6mi_unpack_ref(E, M, back2.ctypes.data, packed.data_ptr(), OC, IC) == 0 and (back2 == raw).all()


def test_fp6_wrappers_are_the_e3m2_case():
    raw, sc = _problem(1, 256, 128, 3, 2)
    t, s = torch.from_numpy(raw), torch.from_numpy(sc)
    assert torch.equal(fp6.weight_prepacking_cpu(t), fp6.weight_prepacking_eXmY_cpu(3, 2, t))
    assert torch.equal(fp6.weight_dequant_cpu(t, s), fp6.weight_dequant_eXmY_cpu(3, 2, t, s))


@pytest.mark.parametrize("E,M", FORMATS)
def test_native_fp6_lane_image_is_the_hardware_operand(E, M):
    """Layout spot check written from the layout's definition, not from the packer: row 16R+m, K block U, lane m+16q,
    code index ci = 8s+j  <->  column 256U + 32s + 8q + j."""
    x = 1 + E + M
    OC, IC = 32, 512
    codes = synth.uniform_codes(42, OC, IC, E, M)
    nat = fp6.weight_prepacking_native_cpu(E, M, torch.from_numpy(quant.pack_raw(codes, E, M))).numpy().view(np.uint32)
    bb = BLOCK_BYTES[x] // 4
    for (R, U, lane) in [(0, 0, 0), (1, 1, 37), (0, 1, 63), (1, 0, 16)]:
        m, q = lane % 16, lane // 16
        blk = nat[(R * 2 + U) * bb:(R * 2 + U + 1) * bb]
        want = [codes[16 * R + m, 256 * U + 32 * s + 8 * q + j] for s in range(8) for j in range(8)]
        if x == 4:
            d = [blk[(i // 4) * 256 + lane * 4 + i % 4] for i in range(8)]
            # four stored dwords per string; dwords five and six of the 6-bit string sit in the two fixed-zero low bits of the fields
            P, Q, R = 0xC30C30C3, 0x30C30C30, 0x0C30C30C
            for h in range(2):
                S = [int(d[4 * h + k]) for k in range(4)]
                D = [S[0] & ~P, S[1] & ~Q, S[2] & ~R, S[3] & ~P, (S[0] & P) | (S[2] & R), (S[1] & Q) | (S[3] & P)]
                big = sum(D[w] << (32 * w) for w in range(6))
                fields = [(big >> (6 * i)) & 63 for i in range(32)]
                assert all(f & 3 == 0 for f in fields)                 # the two bits appended below the mantissa
                assert [f >> 2 for f in fields] == [int(v) for v in want[32 * h:32 * h + 32]]
        elif x == 6:
            d = [blk[(i // 4) * 256 + lane * 4 + i % 4] for i in range(12)]
            for h in range(2):
                big = sum(int(d[6 * h + w]) << (32 * w) for w in range(6))
                got = [(big >> (6 * i)) & 63 for i in range(32)]
                assert got == [int(v) for v in want[32 * h:32 * h + 32]]
        else:
            d = [blk[(i // 4) * 256 + lane * 4 + i % 4] for i in range(8)] + [blk[512 + lane * 2 + i] for i in range(2)]
            # five stored dwords per string; the sixth dword of the 6-bit string sits in the fixed-zero bit of every field
            A, B, C = 0x10410410, 0x04104104, 0x41041041
            for h in range(2):
                S = [int(d[4 * h + k]) for k in range(4)] + [int(d[8 + h])]
                D = [S[0] & ~A, S[1] & ~B, S[2] & ~C, S[3] & ~A, S[4] & ~B,
                     (S[0] & A) | (S[1] & B) | ((((S[2] & C) | (S[3] & A) | (S[4] & B)) << 1) & 0xFFFFFFFF)]
                big = sum(D[w] << (32 * w) for w in range(6))
                fields = [(big >> (6 * i)) & 63 for i in range(32)]
                assert all((f >> 4) & 1 == 0 for f in fields)          # the inserted exponent bit
                got = [(f & 15) | ((f >> 5) << 4) for f in fields]
                assert got == [int(v) for v in want[32 * h:32 * h + 32]]


def test_prepack_in_place_and_padding_is_zero():
    E, M = 3, 2
    raw, _ = _problem(9, 256, 320, E, M)
    L = _lib.lib()
    buf = raw.copy()
    assert L.fp6mi_prepack_ref(E, M, buf.ctypes.data, buf.ctypes.data, 256, 320) == 0
    assert buf.tobytes() == oracle.prepack(raw, E, M).tobytes()
    # K = 320 is padded to 512 in the native layout: the padded columns hold code 0
    nat = fp6.weight_prepacking_native_cpu(E, M, torch.from_numpy(raw))
    wide = np.zeros((256, 512), np.uint8)
    wide[:, :320] = quant.unpack_raw(raw, E, M)
    assert torch.equal(nat, fp6.weight_prepacking_native_cpu(E, M, torch.from_numpy(quant.pack_raw(wide, E, M))))


def test_error_codes_instead_of_aborts():
    L = _lib.lib()
    buf = np.zeros(1 << 16, np.uint8)
    p = buf.ctypes.data
    assert L.fp6mi_prepack_ref(4, 3, p, p, 64, 64) == -1                      # unsupported format (reference: exit(-1))
    assert L.fp6mi_prepack_ref(3, 2, p, p, 32, 64) == -2                      # M % 64 (reference: assert)
    assert L.fp6mi_prepack_ref(3, 2, p, p, 64, 96) == -2                      # K % 64
    assert L.fp6mi_prepack_ref(3, 2, None, p, 64, 64) == -3
    assert L.fp6mi_dequant(1, 2, p, p, 64, 64, p) == -1
    assert L.fp6mi_native_bytes(3, 2, 24, 64) == 0
    assert L.fp6mi_prepack_native(3, 2, p, p, 64, 64) == -2                   # may not alias
    # GEMM argument checks happen on the host before anything is launched
    assert L.fp6mi_linear_native(3, 2, None, p, p, p, p, 100, 1, 64, None, 1) == -2      # M % 256
    assert L.fp6mi_linear_native(3, 2, None, p, p, p, p, 256, 0, 64, None, 1) == -2      # N == 0
    assert L.fp6mi_linear_native(3, 2, None, p, p, p, p, 256, 1, 96, None, 1) == -2      # K % 64
    assert L.fp6mi_linear_native(5, 2, None, p, p, p, p, 256, 1, 64, None, 1) == -1
    assert L.fp6mi_linear_native(3, 2, None, p, p, p, p, 256, 1, 64, None, 2) == -4      # splitK without workspace
    assert L.fp6mi_linear_native(3, 2, None, p, p, p, p, 256, 1, 64, None, 0) == -5
    assert L.fp6mi_linear_native(3, 2, None, None, p, p, p, 256, 1, 64, None, 1) == -3
    assert L.fp6mi_linear_native(3, 2, None, p + 4, p, p, p, 256, 1, 64, None, 1) == -6  # alignment
    assert L.fp6mi_linear_native(3, 2, None, p, p + 1, p, p, 256, 1, 64, None, 1) == -6  # scales are halfs: 2-byte alignment
    for code in (-1, -2, -3, -4, -5, -6, -7, -8):
        assert len(L.fp6mi_error_string(code)) > 8
    assert L.fp6mi_workspace_bytes(256, 8, 1) == 0 and L.fp6mi_workspace_bytes(256, 8, 3) == 3 * 256 * 8 * 4


def test_python_api_argument_errors():
    t = torch.zeros((256, 12), dtype=torch.int32)
    with pytest.raises(ValueError):
        fp6.weight_prepacking_cpu(torch.zeros((100, 12), dtype=torch.int32))      # OC % 256
    with pytest.raises(ValueError):
        fp6.weight_prepacking_cpu(torch.zeros((256, 13), dtype=torch.int32))      # width not a multiple of x
    with pytest.raises(ValueError):
        fp6.weight_prepacking_cpu(t.to(torch.int64))
    with pytest.raises(ValueError):
        fp6.weight_prepacking_eXmY_cpu(4, 3, t)
    with pytest.raises(ValueError):
        fp6.weight_dequant_cpu(t, torch.ones(100, dtype=torch.float16))
    with pytest.raises(ValueError):
        fp6.linear_forward_cuda(torch.zeros(1, 64, dtype=torch.float16), t, torch.ones(256, dtype=torch.float16), 1)  # not on GPU


def test_drop_in_call_refuses_the_same_arguments_with_and_without_the_extension(monkeypatch):
    """The drop-in call checks its arguments in the extension where that is built: what is refused, and with which words, is what the
    Python checks say.  (On the CPU every call ends at the latest at the weights, which have to be on the GPU.)"""
    if fp6._ext is None:
        pytest.skip("the torch extension is not built")
    w, x, sc = torch.zeros(256, 12, dtype=torch.int32), torch.zeros(3, 64, dtype=torch.float16), torch.ones(256, dtype=torch.float16)
    calls = [(3, 2, x, w, sc), (3, 2, w, sc, x), (2, 2, x, w, sc), (2, 1, sc, x, w), (4, 3, x, w, sc), (2, 3, x[:, :32], w, sc), (3, 2, x.float(), w, sc),
             (3, 2, x, w, sc.float()), (3, 2, x, w.long(), sc), (3, 2, x, w, w), (3, 2, x, x, sc), (3, 2, x, w, x), (3, 2, x[0], w, sc), (3, 2, x, w, sc[None, None]),
             (3, 2, x, w[0], sc), (3, 2, x, w[0, 0], sc), (3, 2, x, w[:, :11], sc), (3, 2, x, w.t(), sc), (3, 2, x, None, sc), (3, 2, x, w.numpy(), sc)]
    for call in calls:
        said = []
        for ext in (fp6._ext, None):
            monkeypatch.setattr(fp6, "_ext", ext)
            with pytest.raises(Exception) as e:
                fp6.linear_forward_eXmY_cuda(*call)
            said.append((type(e.value), str(e.value)))
        monkeypatch.undo()
        assert said[0] == said[1], call


def test_an_extension_of_an_older_tree_is_not_used():
    """An extension built before the drop-in call moved into it has no linear_forward_any_order: the package then takes its ctypes path."""
    code = ("import sys, types\n"
            "old = sys.modules['fp6_llm_amd._fp6mi_torch'] = types.ModuleType('fp6_llm_amd._fp6mi_torch')\n"
            "old.linear_forward_native = old.clear_workspaces = old.clear_twins = lambda *a: None\n"
            "import torch, fp6_llm_amd as fp6\n"
            "w, x, sc = torch.zeros(256, 12, dtype=torch.int32), torch.zeros(3, 64).half(), torch.ones(256).half()\n"
            "try:\n    fp6.linear_forward_cuda(x, w, sc)\n"
            "except ValueError as e:\n    assert str(e) == 'weights must be on the GPU', e\n"
            "fp6.clear_caches()\n"
            "assert fp6._ext is None\n")
    env = {k: v for k, v in os.environ.items() if k != "FP6MI_NO_TORCH_EXT"}
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT, env=env)


def test_reference_heuristic_is_kept_verbatim():
    for args in [(4096, 8, 108), (11008, 8, 108), (8192, 512, 256), (256, 1, 108), (28672, 32, 108), (4096, 8, 256)]:
        assert fp6.HeuristicFuntion_SplitK(*args) == oracle.heuristic_splitk(*args)
        assert fp6.Num_Wave(args[0], args[1], 3, args[2]) == pytest.approx(oracle.num_wave(args[0], args[1], 3, args[2]))


def test_mi355x_heuristic_prefers_no_split_when_rows_fill_the_chip():
    for (M, N, K) in [(4096, 8, 4096), (11008, 8, 4096), (8192, 16, 8192), (28672, 8, 8192), (8192, 512, 8192)]:
        assert fp6.heuristic_splitk_mi355x(M, N, K) == 1
    # batches above 16 tile the rows in blocks of 64..256: K is cut to make up the missing parallelism, into 2, 3, 4, 6 or 8
    # pieces and never into more pieces than there are 256-column K blocks
    for (M, N, K) in [(8192, 32, 8192), (28672, 32, 8192), (8192, 64, 8192), (4096, 32, 11008), (10240, 32, 8192), (4096, 128, 512)]:
        s = fp6.heuristic_splitk_mi355x(M, N, K)
        assert s in (1, 2, 3, 4, 6, 8) and s <= (K + 255) // 256, (M, N, K, s)
    assert fp6.heuristic_splitk_mi355x(8192, 32, 8192) > 1          # 64 row blocks alone leave three quarters of the CUs idle
    s = fp6.heuristic_splitk_mi355x(256, 8, 28672)      # 16 row tiles cannot occupy 256 CUs: splitting K pays
    assert 2 <= s <= 64
    assert fp6.heuristic_splitk_mi355x(256, 1, 1024) == 1  # too little work to pay for a second launch


def test_rule_based_heuristic_for_other_cu_counts():
    """With a CU count that has no measured table the cost rules decide; known answers of those rules for a 304-CU part."""
    assert fp6.heuristic_splitk_mi355x(4096, 8, 4096, 304) == 1
    assert fp6.heuristic_splitk_mi355x(8192, 512, 8192, 304) == 1
    for (M, N, K) in [(8192, 32, 8192), (28672, 32, 8192), (8192, 64, 8192)]:
        s = fp6.heuristic_splitk_mi355x(M, N, K, 304)
        assert s in (1, 2, 4, 8)
    assert fp6.heuristic_splitk_mi355x(8192, 32, 8192, 304) >= fp6.heuristic_splitk_mi355x(28672, 32, 8192, 304)


def test_compiled_launch_shape_lists_match_the_kernel_source():
    from fp6_llm_amd import tune
    src = open(os.path.join(os.path.dirname(fp6.__file__), "csrc", "fp6mi_gemm.hip")).read()
    stream = {(0, int(a), int(b), 1, int(c)) for a, b, c in re.findall(r"FP6MI_CASE\((\d+), (\d+), (\d+)\)", src)}
    tile_src, ws_src = src.split("c.kind == 2")    # the wave-specialized shapes are listed after those of the tile kernel
    tile = {(1, int(a), int(b), int(c), int(d)) for a, b, c, d in re.findall(r"FP6MI_CASE\((\d+), (\d+), (\d+), (\d+)\)", tile_src)}
    ws = {(2, int(a), int(b), int(c), int(d)) for a, b, c, d in re.findall(r"FP6MI_CASE\((\d+), (\d+), (\d+), (\d+)\)", ws_src)}
    assert stream == set(tune.COMPILED_STREAM) and tile == set(tune.COMPILED_TILE) and ws == set(tune.COMPILED_WS)
    assert set(tune.STREAM_SMALL + tune.STREAM_WIDE) <= stream and set(tune.TILE) <= tile


def test_measured_table_holds_only_compiled_shapes_and_query_launch_follows_it():
    from fp6_llm_amd import tune
    compiled = set(tune.COMPILED_STREAM + tune.COMPILED_TILE + tune.COMPILED_WS)
    inc = open(tune.INC_PATH).read()
    entries = re.findall(r"^\{(\d+),(\d+),(\d+),(\d+),\{(.*)\}\},$", inc, flags=re.M)
    L = _lib.lib()
    shape = (ctypes.c_int * 5)()
    for xb, m256, k64, n, cells in entries:
        E, Mb = {6: (3, 2), 5: (2, 2), 4: (2, 1)}[int(xb)]
        OC, IC, BS = int(m256) * 256, int(k64) * 64, int(n)
        for i, cell in enumerate(re.findall(r"\{([\d,]+)\}", cells)):
            v = tuple(int(t) for t in cell.split(","))
            if v[0] == 255:
                continue
            assert v[:5] in compiled, (xb, OC, IC, BS, v)
            assert v[0] == 0 or OC % tune.tile_rows(v[:5]) == 0      # (the stream kernel's last workgroup holds what is left of the row tiles)
            assert L.fp6mi_query_table(E, Mb, OC, BS, IC, tune.SPLITS[i], shape) == 0
            assert tuple(shape) == v[:5], (xb, OC, IC, BS, tune.SPLITS[i], tuple(shape), v)
            assert L.fp6mi_query_launch(E, Mb, OC, BS, IC, tune.SPLITS[i], shape) == 0
            wide = BS > 96 and shape[0] == 2 and shape[3] == 4 and shape[4] <= 2
            assert (wide or tuple(shape) == v[:5]) and L.fp6mi_launch_source(E, Mb, OC, BS, IC, tune.SPLITS[i]) == (2 if wide else 0)
    # any legal problem gets a compiled shape that divides its rows, measured neighbour or not
    for (OC, IC, BS, sk) in [(256, 64, 1, 1), (768, 1088, 3, 2), (4352, 4160, 8, 1), (9984, 3008, 40, 3), (65536, 16384, 700, 1), (512, 64, 17, 1)]:
        for (E, Mb) in FORMATS:
            assert L.fp6mi_query_launch(E, Mb, OC, BS, IC, sk, shape) == 0
            assert tuple(shape) in compiled and (shape[0] == 0 or OC % tune.tile_rows(tuple(shape)) == 0), (OC, IC, BS, sk, tuple(shape))
    assert L.fp6mi_query_launch(3, 2, 100, 1, 64, 1, shape) == -2 and L.fp6mi_query_launch(4, 3, 256, 1, 64, 1, shape) == -1


@pytest.mark.parametrize("OC,IC,N,splitK,prefill", [
    (4608, 4544, 777, 1, True),        # 252 workgroups of 128 x 128 (one round) against 126 of 256 x 128
    (4608, 4544, 777, 2, False),       # a split keeps the measured shapes
    (28672, 8192, 384, 1, True),       # 672 (three rounds) against 336 (two, of twice the length)
    (28672, 8192, 512, 1, False),      # a measured problem keeps its measured shape
    (8192, 8192, 4000, 1, False),      # long prompt whose rows are a power of two apart
    (8192, 8192, 100, 1, False),       # one column block
    (15616, 2560, 3854, 1, False),     # long prompt, 15 half rounds for 16
    (3328, 11904, 3495, 1, True),      # long prompt, 3 for 4
    (256, 1 << 21, 4096, 1, False),    # K beyond the kernel's 32-bit offsets
    (2816, 5504, 6934, 1, False),      # longer prompts than 4096: 1.12 of the time before, 5 half rounds for 6
    (5888, 9280, 4841, 1, False),      # 1.10, 7 for 8
    (2304, 1600, 12360, 1, True),      # but short rows: 0.93
    (7936, 15104, 3537, 1, False),     # long rows from N 3072 on, 7 for 8: 1.03
    (2816, 10816, 3634, 1, True),      # a quarter fewer: 0.98
    (2816, 14528, 4049, 1, False),     # the same close to N 4096: 1.01
    (12032, 64, 343, 1, False),        # one round of 256 x 128, two half as long: 1.03, with group exponents 1.08
    (17920, 6016, 218, 1, False),      # the same: 1.07, with group exponents 1.16
    (26624, 192, 824, 1, False),       # six half rounds for six: 1.10
    (27648, 192, 1548, 1, False),      # 11 half rounds for 12, but little K: 1.05, with group exponents 1.10
    (30208, 320, 1724, 1, True),       # from K 320 on (13 for 14): 0.87, 0.90
    (2304, 5888, 1520, 1, True),       # one half round for two: 0.66
])
def test_prefill_kernel_rule(OC, IC, N, splitK, prefill):
    shape = (ctypes.c_int * 5)()
    assert _lib.lib().fp6mi_query_table(3, 2, OC, N, IC, splitK, shape) >= 0
    assert (tuple(shape) == (2, 8, 4, 2, 2)) == prefill, tuple(shape)


@pytest.mark.parametrize("E,M", FORMATS)
def test_quantizer(E, M):
    x = 1 + E + M
    mags = quant.magnitudes(E, M)
    assert (mags == np.abs(oracle.value_table(E, M)[: 1 << (x - 1)])).all()
    allc = np.arange(1 << x, dtype=np.uint8)
    vals = oracle.value_table(E, M)
    q = quant.quantize_codes(vals, E, M)
    assert (q == allc).all()                                       # exact values map to their own code (incl. -0)
    assert quant.quantize_codes(np.array([1e9, -1e9]), E, M).tolist() == [(1 << (x - 1)) - 1, (1 << x) - 1]  # clamp
    mid = (mags[:-1] + mags[1:]) / 2
    tie = quant.quantize_codes(mid, E, M)
    assert (tie % 2 == 0).all()                                    # ties go to the even code
    v = np.linspace(-mags[-1], mags[-1], 4001)
    assert (np.diff(vals[quant.quantize_codes(v, E, M)]) >= 0).all()  # monotone
    assert (np.abs(vals[quant.quantize_codes(v, E, M)] - v) <= np.diff(mags).max() / 2 + 1e-12).all()
    w = synth.normal(5, (64, 128))
    codes, scale = quant.quantize_rowwise(w, E, M)
    assert scale.dtype == np.float16 and codes.max() < (1 << x)
    deq = quant.dequantize_codes(codes, scale, E, M)
    assert np.abs(deq - w).max() <= np.abs(w).max() / mags[-1] * np.diff(mags).max() * 0.51
    raw = quant.pack_raw(codes, E, M)
    assert (quant.unpack_raw(raw, E, M) == codes).all() and (oracle.unpack_codes(raw, E, M) == codes).all()


def _awkward_weights(seed, OC, IC):
    """Gaussian weights with what a quantizer gets wrong: zero rows, a row whose scale is an fp16 subnormal, a huge row,
    negative zeros, exact ties of the scaled grid, and NaN / +-Inf entries."""
    w = synth.normal(seed, (OC, IC)).astype(np.float32)
    w[1, :] = 0.0
    w[2, :] *= 1e-7
    w[3, :] *= 3000.0
    w[4, ::3] = -0.0
    w[5, :] = 0.0
    w[5, 0] = 28.0
    w[5, 1:65] = np.arange(64, dtype=np.float32) * 0.4375
    w[6, :] = -w[5, :]
    w[7, 3] = np.nan
    w[7, 4] = np.inf
    w[7, 5] = -np.inf
    return w


@pytest.mark.parametrize("E,M", FORMATS)
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_host_quantizer_equals_the_exact_definition(E, M, dtype):
    """quant.quantize_rowwise / quantize_groupwise (float64 quotients, searchsorted) against the oracle's definition in exact
    arithmetic: same scales, same codes, same group exponents."""
    with np.errstate(over="ignore"):
        w = _awkward_weights(61, 64, 320).astype(dtype)
    codes, sc = quant.quantize_rowwise(w, E, M)
    c0, s0 = oracle.quantize_from_definition(w, E, M)
    assert np.array_equal(sc.view(np.uint16), s0.view(np.uint16)) and np.array_equal(codes, c0)
    spread = np.exp(np.random.default_rng(5).normal(0, 2.0, (64, 3))).repeat(128, axis=1)[:, :320]
    spread[:8] = 1.0
    with np.errstate(over="ignore", invalid="ignore"):
        wg = (w.astype(np.float64) * spread).astype(dtype)
    codes, sc, ex = quant.quantize_groupwise(wg, E, M)
    c0, s0, e0 = oracle.quantize_grouped_from_definition(wg, E, M)
    assert np.array_equal(sc.view(np.uint16), s0.view(np.uint16)) and np.array_equal(ex, e0) and np.array_equal(codes, c0)


def test_native_weight_file_round_trip(tmp_path):
    from fp6_llm_amd import module
    raw, sc = _problem(21, 256, 320, 2, 2)
    nat = fp6.weight_prepacking_native_cpu(2, 2, torch.from_numpy(raw))
    path = str(tmp_path / "w.fp6mi")
    module.save_native(path, nat, torch.from_numpy(sc), 2, 2, 256, 320)
    nat2, sc2, hdr = module.load_native(path)
    assert torch.equal(nat, nat2) and (sc2.numpy() == sc).all() and hdr["in_features"] == 320 and hdr["exponent"] == 2
    with open(path, "r+b") as f:
        f.truncate(4000)
    with pytest.raises(ValueError):
        module.load_native(path)
    with open(path, "wb") as f:
        f.write(b"not a weight file")
    with pytest.raises(ValueError):
        module.load_native(path)


# ------------------------------------------------------------------------------------------------ per-group exponents
def _grouped_problem(seed, OC, IC, E, M):
    """Gaussian weights whose groups of 128 columns differ in magnitude by powers of e, so that the exponents vary."""
    rng = np.random.default_rng(seed)
    spread = np.exp(rng.normal(0, 1.5, (OC, (IC + 127) // 128))).repeat(128, axis=1)[:, :IC]
    return synth.normal(seed, (OC, IC)) * spread


@pytest.mark.parametrize("E,M", FORMATS)
def test_groupwise_quantizer(E, M):
    OC, IC = 64, 320   # the last group has 64 columns
    w = _grouped_problem(31, OC, IC, E, M)
    codes, sc, ex = quant.quantize_groupwise(w, E, M)
    top = quant.max_value(E, M)
    assert ex.dtype == np.uint8 and ex.shape == (OC, 3) and ex.min() >= 112 and ex.max() == 127 and len(np.unique(ex)) > 3
    _, sc_row = quant.quantize_rowwise(w, E, M)
    assert (sc == sc_row).all()                                  # the row scale is the row-wise one
    for g in range(3):
        blockmax = np.abs(w[:, 128 * g:128 * g + 128]).max(axis=1) / sc.astype(np.float64)
        f = np.exp2(ex[:, g].astype(np.float64) - 127)
        # the group fits under its factor (the row's largest group only up to the rounding of the fp16 row scale, like row-wise) ...
        assert ((blockmax <= top * f) | ((ex[:, g] == 127) & (blockmax <= top * (1 + 2.0 ** -10)))).all()
        assert ((blockmax > top * f / 2) | (ex[:, g] == 112)).all()   # ... and would not fit under half of it
    deq = quant.dequantize_grouped(codes, sc, ex, E, M)
    rw_codes, _ = quant.quantize_rowwise(w, E, M)
    assert np.abs(deq - w).mean() < np.abs(quant.dequantize_codes(rw_codes, sc, E, M) - w).mean()
    # weights without spread between groups of a row's own maximum group keep factor 1 there
    assert (ex.max(axis=1) == 127).all()
    # a zero matrix: scale 1, any exponent, all codes zero magnitude
    c0, s0, e0 = quant.quantize_groupwise(np.zeros((16, 128)), E, M)
    assert (s0 == 1).all() and (c0 & ((1 << (E + M)) - 1) == 0).all() and e0.shape == (16, 1)


@pytest.mark.parametrize("E,M", FORMATS)
def test_grouped_dequant_and_exponent_packing(E, M):
    OC, IC = 64, 320
    codes, sc, ex = quant.quantize_groupwise(_grouped_problem(32, OC, IC, E, M), E, M)
    raw = torch.from_numpy(quant.pack_raw(codes, E, M))
    dq = fp6.weight_dequant_grouped_cpu(E, M, raw, torch.from_numpy(sc), torch.from_numpy(ex)).numpy()
    assert (dq.view(np.uint16) == oracle.dequant_grouped_from_definition(codes, sc, ex, E, M).view(np.uint16)).all()
    ones = torch.full((OC, 3), 127, dtype=torch.uint8)               # factor 1 everywhere = the reference's dequantizer
    assert torch.equal(fp6.weight_dequant_grouped_cpu(E, M, raw, torch.from_numpy(sc), ones),
                       fp6.weight_dequant_eXmY_cpu(E, M, raw, torch.from_numpy(sc)))
    # packed order, from its definition: [row tile][K block][row in tile][half]; halves beyond IC hold 127
    nat = fp6.pack_group_exps(torch.from_numpy(ex), OC, IC).numpy()
    assert nat.size == fp6.group_exps_bytes(OC, IC) == (OC // 16) * 2 * 32
    for (R, U, m, h) in [(0, 0, 0, 0), (3, 0, 15, 1), (2, 1, 7, 0), (1, 1, 9, 1)]:
        want = ex[16 * R + m, 2 * U + h] if 2 * U + h < 3 else 127
        assert nat[((R * 2 + U) * 16 + m) * 2 + h] == want
    with pytest.raises(ValueError):
        fp6.pack_group_exps(torch.from_numpy(ex[:, :2].copy()), OC, IC)


def test_grouped_weight_file_and_fused_layers(tmp_path):
    from fp6_llm_amd import module
    E, M = 2, 1
    ws = [torch.from_numpy(_grouped_problem(40 + i, oc, 384, E, M)).float() for i, oc in enumerate((256, 512))]
    parts = [module.FPxLinear.from_float(w, E, M, group_scales=True) for w in ws]
    whole = module.FPxLinear.from_float(torch.cat(ws), E, M, group_scales=True)
    fused = module.FPxLinear.fused(parts)
    assert fused.group_exps is not None and torch.equal(fused.group_exps, whole.group_exps)
    assert torch.equal(fused.weight_native, whole.weight_native) and torch.equal(fused.scales, whole.scales)
    with pytest.raises(ValueError):
        module.FPxLinear.fused([parts[0], module.FPxLinear.from_float(ws[1], E, M)])
    # a layer built empty with group_scales=True takes the state of a quantized one
    blank = module.FPxLinear(384, 768, E, M, group_scales=True)
    assert (blank.group_exps == 127).all()
    blank.load_state_dict(whole.state_dict())
    assert torch.equal(blank.group_exps, whole.group_exps) and torch.equal(blank.weight_native, whole.weight_native)
    assert "group_exps" not in module.FPxLinear(384, 768, E, M).state_dict()
    path = str(tmp_path / "g.fp6mi")
    module.save_native(path, whole.weight_native, whole.scales, E, M, 768, 384, whole.group_exps)
    nat2, sc2, hdr = module.load_native(path)
    assert torch.equal(nat2, whole.weight_native) and torch.equal(sc2, whole.scales) and torch.equal(hdr["group_exps"], whole.group_exps)
    module.save_native(path, whole.weight_native, whole.scales, E, M, 768, 384)
    assert "group_exps" not in module.load_native(path)[2]


def test_module_construction_routes_agree():
    from fp6_llm_amd import module
    raw, sc = _problem(22, 256, 128, 3, 2)
    t, s = torch.from_numpy(raw), torch.from_numpy(sc)
    a = module.FPxLinear.from_raw(t, s)
    b = module.FPxLinear.from_prepacked(fp6.weight_prepacking_cpu(t), s)
    assert torch.equal(a.weight_native, b.weight_native) and torch.equal(a.scales, b.scales)
    w = torch.from_numpy(synth.normal(3, (256, 128))).float()
    c = module.FPxLinear.from_float(w)
    codes, scales = quant.quantize_rowwise(w.numpy(), 3, 2)
    assert torch.equal(c.weight_native, fp6.weight_prepacking_native_cpu(3, 2, torch.from_numpy(quant.pack_raw(codes, 3, 2))))
    with pytest.raises(ValueError):
        module.FPxLinear(100, 256)


def test_split_heuristic_per_format():
    L = _lib.lib()
    for (M, N, K) in [(4096, 8, 4096), (8192, 32, 8192), (256, 8, 28672), (17920, 32, 6656), (1024, 300, 2048)]:
        assert L.fp6mi_heuristic_splitk_format(3, 2, M, N, K, 256) == L.fp6mi_heuristic_splitk(M, N, K, 256)
        assert L.fp6mi_heuristic_splitk_format(2, 3, M, N, K, 256) == L.fp6mi_heuristic_splitk(M, N, K, 256)   # same bytes, same table
        for (E, Mb) in FORMATS:
            s = fp6.heuristic_splitk_mi355x(M, N, K, EXPONENT=E, MANTISSA=Mb)
            assert 1 <= s <= 64 and s <= (K + 255) // 256


def test_fused_layers_are_the_concatenation():
    """Fusing layers over one input = quantizing the row-concatenated weight: native tiles are stored row tile after row tile."""
    from fp6_llm_amd import module
    for (E, M) in FORMATS:
        ws = [torch.from_numpy(synth.normal(61 + i, (oc, 320))).float() for i, oc in enumerate((256, 512, 256))]
        bs = [torch.from_numpy(synth.normal(71 + i, (w.shape[0],))).half() for i, w in enumerate(ws)]
        parts = [module.FPxLinear.from_float(w, E, M, bias=b) for w, b in zip(ws, bs)]
        fused = module.FPxLinear.fused(parts)
        whole = module.FPxLinear.from_float(torch.cat(ws), E, M, bias=torch.cat(bs))
        assert fused.out_features == 1024 and fused.in_features == 320
        assert torch.equal(fused.weight_native, whole.weight_native)
        assert torch.equal(fused.scales, whole.scales) and torch.equal(fused.bias, whole.bias)
    with pytest.raises(ValueError):
        module.FPxLinear.fused([module.FPxLinear.from_float(ws[0], 3, 2), module.FPxLinear.from_float(ws[0], 2, 2)])


def test_e2m2_code_read_as_e3m2_is_a_quarter_of_its_value():
    """What the FP5 native layout relies on: inserting a zero above the two exponent bits of an e2m2 code gives the e3m2
    code of exactly a quarter of its value, for all 32 codes (subnormals and signed zeros included)."""
    v5, v6 = oracle.value_table(2, 2), oracle.value_table(3, 2)
    for code in range(32):
        field = (code & 15) | ((code >> 4) << 5)
        assert v6[field] * 4.0 == v5[code] and np.signbit(v6[field]) == np.signbit(v5[code])


def test_e2m1_code_with_two_zeros_appended_is_the_e2m3_code_of_its_value():
    """What the FP4 native layout relies on: an e2m1 code shifted left by two bits is the e2m3 code of the same value, for all
    16 codes (the subnormal and the signed zeros included)."""
    v4, v6 = oracle.value_table(2, 1), oracle.value_table(2, 3)
    for code in range(16):
        assert v6[code << 2] == v4[code] and np.signbit(v6[code << 2]) == np.signbit(v4[code])


def test_bench_refuses_more_than_one_gpu_and_lists_the_benchmark_configurations():
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert res.returncode != 0 and "ONE GPU" in res.stderr
    sys.path.insert(0, root)
    import bench
    assert bench.WORKLOADS[bench.HEADLINE] == (3, 2, 4096, 4096, 8)
    # every shape of the five benchmark configurations is a workload: 4096^2 at 1/8/16, the two 7B MLP shapes at 8/32, the three
    # 70B shapes at 32, and 8192^2 at ten batch sizes in both formats
    assert len([w for w in bench.WORKLOADS if w.startswith(("fp6_", "fp5_"))]) == 3 + 4 + 3 + 20
    assert bench.weight_bytes(3, 2, 4096, 4096) == 12582912 and bench.algorithmic_bytes(3, 2, 4096, 4096, 8) == 12722176


def test_tuner_candidates_and_table_emission(tmp_path, monkeypatch):
    from fp6_llm_amd import tune
    compiled = set(tune.COMPILED_STREAM + tune.COMPILED_TILE + tune.COMPILED_WS)
    for (OC, IC, BS) in [(256, 64, 1), (4096, 4096, 8), (4096, 4096, 17), (11008, 4096, 64), (768, 2048, 512), (8192, 8192, 2048)]:
        cands = list(tune.candidates(OC, IC, BS))
        assert cands, (OC, IC, BS)
        for cfg, sk in cands:
            ragged = cfg[0] == 0                       # the stream kernel's last workgroup holds what is left of the row tiles
            assert cfg in compiled and (ragged or OC % tune.tile_rows(cfg) == 0) and 1 <= sk <= (IC + 255) // 256
            assert cfg[0] != 0 or BS <= 64 or (BS <= 128 and OC <= 2560)     # the stream kernel is a candidate up to four column blocks, eight on short matrices
            assert cfg[0] == 0 or BS > 16
    src = tmp_path / "t.jsonl"
    src.write_text(json.dumps({"E": 3, "M": 2, "OC": 512, "IC": 1024, "BS": 8, "best": {"1": [[0, 1, 1, 1, 8], 3.21], "4": [[0, 1, 2, 1, 4], 4.0]}}) + "\n")
    monkeypatch.setattr(tune, "INC_PATH", str(tmp_path / "out.inc"))
    tune.main(["emit", str(src)])
    lines = [l for l in (tmp_path / "out.inc").read_text().splitlines() if l.startswith("{")]
    assert lines == ["{6,2,16,8,{{0,1,1,1,8,160},{255,0,0,0,0,0},{255,0,0,0,0,0},{0,1,2,1,4,200},{255,0,0,0,0,0},{255,0,0,0,0,0}}},"]


# ------------------------------------------------------------------------------------------------ randomized round trips
def test_packers_round_trip_on_random_shapes_and_bits():
    """Property check with hypothesis: for any supported format, any legal shape and any bit pattern, the reference layout and
    the native layout both unpack to the raw tensor they were packed from, both routes to the native layout agree, and the
    host prepacker equals the oracle's."""
    from hypothesis import given, settings, strategies as st

    @settings(max_examples=40, deadline=None)
    @given(fmt=st.sampled_from(FORMATS), tiles=st.integers(1, 3), kblocks=st.integers(1, 9), seed=st.integers(0, 2 ** 31 - 1))
    def check(fmt, tiles, kblocks, seed):
        E, M = fmt
        x = 1 + E + M
        OC, IC = 64 * tiles, 64 * kblocks
        raw = np.random.default_rng(seed).integers(0, 2 ** 32, size=(OC, IC // 32 * x), dtype=np.uint64).astype(np.uint32).view(np.int32)
        L = _lib.lib()
        packed, back = np.empty_like(raw), np.empty_like(raw)
        assert L.fp6mi_prepack_ref(E, M, packed.ctypes.data, raw.ctypes.data, OC, IC) == 0
        assert packed.tobytes() == oracle.prepack(raw, E, M).tobytes()
        assert L.fp6mi_unpack_ref(E, M, back.ctypes.data, packed.ctypes.data, OC, IC) == 0 and (back == raw).all()
        nat = np.empty(fp6.native_bytes(E, M, OC, IC), np.uint8)
        nat2 = np.empty_like(nat)
        assert L.fp6mi_prepack_native(E, M, nat.ctypes.data, raw.ctypes.data, OC, IC) == 0
        assert L.fp6mi_relayout_ref_to_native(E, M, nat2.ctypes.data, packed.ctypes.data, OC, IC) == 0 and (nat == nat2).all()
        back[:] = 0
        assert L.fp6mi_unpack_native(E, M, back.ctypes.data, nat.ctypes.data, OC, IC) == 0 and (back == raw).all()

    check()



def test_host_code_and_oracle_are_clean_under_asan_and_ubsan():
    """Builds tests/sanitize (the engine's CPU functions + the oracle with AddressSanitizer and UBSan, ROCm's clang) and runs its
    driver over every format, cut K blocks, in-place packing and the grouped dequantizer."""
    import shutil
    import subprocess
    d = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize")
    if not os.path.exists("/opt/rocm/llvm/bin/clang++") or not shutil.which("make") or not os.path.isdir(d):
        pytest.skip("needs ROCm's clang and make")
    res = subprocess.run(["make", "-C", d, "-B", "run"], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0 and "clean under ASan + UBSan" in res.stdout, res.stdout[-2000:] + res.stderr[-2000:]


def test_the_reference_package_name_imports_the_same_functions():
    """`import fp6_llm` (the reference's package name, fp6_llm/__init__.py:1) gives the engine's functions under the reference's names."""
    import fp6_llm
    for name in ["linear_forward_cuda", "weight_prepacking_cpu", "weight_dequant_cpu", "linear_forward_eXmY_cuda", "weight_prepacking_eXmY_cpu",
                 "weight_dequant_eXmY_cpu", "Num_Wave", "HeuristicFuntion_SplitK"]:
        assert getattr(fp6_llm, name) is getattr(fp6, name)


def test_launch_source_tells_measured_from_carried_over_from_rules():
    L = _lib.lib()
    assert L.fp6mi_launch_source(3, 2, 4096, 8, 4096, 1) == 0          # in the table
    assert L.fp6mi_launch_source(3, 2, 4096, 7, 4096, 1) == 0          # the next larger measured batch of a measured matrix
    assert L.fp6mi_launch_source(3, 2, 4352, 8, 4160, 1) == 1          # neighbours within a factor 1.5
    assert L.fp6mi_launch_source(3, 2, 256, 8, 64, 1) == 2               # far from every measured problem
    assert L.fp6mi_launch_source(3, 2, 4096, 8, 4096, 5) == 2          # a split the table does not hold
    assert L.fp6mi_launch_source(4, 3, 4096, 8, 4096, 1) == -1 and L.fp6mi_launch_source(3, 2, 100, 8, 4096, 1) == -2
    assert b"library version" in L.fp6mi_tuning_info()


def test_launch_source_of_problems_the_prefill_rule_takes():
    """The prefill kernel is in no row of the table: where it runs, a rule has put it there, also on a measured matrix."""
    L = _lib.lib()
    shape = (ctypes.c_int * 5)()
    for OC, IC, N, prefill in ((28672, 8192, 384, True), (28672, 8192, 512, False), (22016, 4096, 511, True), (4608, 4544, 777, True)):
        assert (L.fp6mi_query_table(3, 2, OC, N, IC, 1, shape) == 2) == prefill
        assert (tuple(shape) == (2, 8, 4, 2, 2)) == prefill


def test_wide_kernel_takes_the_place_of_larger_tiles():
    """fp6mi_query_kernel is what a call launches: the table's shape or the rules' up to 96 columns, where K is beyond the wide kernel's 32-bit offsets and where
    the problem is small; a compiled shape that divides the rows everywhere."""
    from fp6_llm_amd import tune
    L = _lib.lib()
    base, shape = (ctypes.c_int * 5)(), (ctypes.c_int * 5)()
    compiled = set(tune.COMPILED_STREAM + tune.COMPILED_TILE + tune.COMPILED_WS)
    rng = np.random.default_rng(11)
    seen = set()
    for _ in range(2000):
        E, M = FORMATS[rng.integers(len(FORMATS))]
        OC, IC, N = 256 * int(2 ** rng.uniform(0, 7.5)), 64 * int(2 ** rng.uniform(0, 9)), int(2 ** rng.uniform(0, 13.5))
        for splitK in {1, int(rng.integers(1, 12)), fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M)}:
            for grouped in (0, 1):
                source = L.fp6mi_query_table(E, M, OC, N, IC, splitK, base)
                assert source >= 0 and L.fp6mi_query_kernel(E, M, OC, N, IC, splitK, grouped, shape) == 0
                s = tuple(shape)
                wide = s[0] == 2 and s[3] == 4 and s[4] <= 2
                assert s in compiled and (s[0] == 0 or OC % tune.tile_rows(s) == 0)
                assert (wide and N > 96 and splitK <= (IC + 255) // 256) or s == tuple(base)
                if not grouped:   # the other two queries say the same
                    assert L.fp6mi_query_launch(E, M, OC, N, IC, splitK, base) == 0 and tuple(base) == s
                    assert L.fp6mi_launch_source(E, M, OC, N, IC, splitK) == (2 if wide else source)
                seen.add(s)
    assert {(2, 8, 4, 4, 1), (2, 8, 4, 4, 2), (2, 6, 4, 4, 1), (2, 8, 2, 4, 2), (2, 6, 2, 4, 2), (2, 4, 2, 4, 2)} <= seen
    for OC, IC, N, wide in ((8192, 8192, 96, False), (1536, 1216, 258, False), (28672, 8192, 2048, True), (8192, 1 << 21, 2048, False)):
        assert L.fp6mi_query_kernel(3, 2, OC, N, IC, 1, 0, shape) == 0 and (shape[0] == 2 and shape[3] == 4 and shape[4] <= 2) == wide
    assert L.fp6mi_query_kernel(3, 2, 100, 1, 64, 1, 0, shape) == -2 and L.fp6mi_query_kernel(4, 3, 256, 1, 64, 1, 0, shape) == -1


def test_every_matrix_of_the_table_is_measured_at_every_batch():
    """A matrix with no row at a batch is answered from its neighbours there: 9216 x 9216 in FP5 was cut into four at 257 to 320 columns, where it and
    each of its neighbours are fastest unsplit (and four pieces do not fit the static workspace)."""
    inc = open(os.path.join(os.path.dirname(fp6.__file__), "csrc", "fp6mi_tuning.inc")).read()
    rows = {tuple(map(int, r)) for r in re.findall(r"^\{(\d+),(\d+),(\d+),(\d+),\{\{", inc, re.M)}
    matrices, batches = {r[1:3] for r in rows}, {r[3] for r in rows}
    assert len(rows) == 3 * len(matrices) * len(batches)
    for N in range(257, 321):
        assert fp6.heuristic_splitk_mi355x(9216, N, 9216, EXPONENT=2, MANTISSA=2) == 1, N


@pytest.mark.parametrize("E,M,OC,IC,N", [(2, 1, 1280, 2304, 113), (2, 2, 1536, 1408, 47), (2, 3, 1280, 2048, 126), (2, 3, 2048, 3136, 255), (3, 2, 2048, 3456, 231),
                                         (2, 3, 3328, 1600, 71), (2, 2, 1536, 2752, 173), (2, 1, 1792, 7424, 39), (2, 2, 2048, 6528, 45)])
def test_a_short_matrix_is_not_cut_because_a_longer_one_nearly_would_be(E, M, OC, IC, N):
    """Matrices off the table whose neighbours there have more columns and gain little by a split, or nothing: a split's second launch and its partial sums
    do not shrink with K, and measured on the GPU these are 5-53 % slower in the three to eight pieces they were cut into."""
    assert fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M) == 1


def test_cpp_torch_entry_points_carry_the_reference_names():
    """The torch extension defines the reference's six C++ functions (fp6_llm/csrc/fp6_linear.cuh:50-90) and binds them under the
    reference's Python names (fp6_llm/csrc/pybind.cpp:8-15); the CPU ones must give the oracle's bytes."""
    ext = pytest.importorskip("fp6_llm_amd._fp6mi_torch")
    for name in ("linear_forward_cuda", "weight_prepacking_cpu", "weight_dequant_cpu", "linear_forward_eXmY_cuda", "weight_prepacking_eXmY_cpu",
                 "weight_dequant_eXmY_cpu"):
        assert callable(getattr(ext, name))
    header = open(os.path.join(os.path.dirname(fp6.__file__), "csrc", "fp6_linear_torch.h")).read()
    for name in ("fp6_linear_forward_cuda", "fp_eXmY_linear_forward_cuda", "weight_matrix_prepacking_cpu", "weight_matrix_prepacking_fp_eXmY_cpu",
                 "weight_matrix_dequant_cpu", "weight_matrix_dequant_fp_eXmY_cpu"):
        assert name in header
    for (E, M) in FORMATS:
        raw, sc, _ = synth.uniform_problem(70 + E + M, 256, 320, 1, E, M)
        packed = ext.weight_prepacking_eXmY_cpu(E, M, torch.from_numpy(raw))
        assert packed.numpy().tobytes() == oracle.prepack(raw, E, M).tobytes()
        deq = ext.weight_dequant_eXmY_cpu(E, M, torch.from_numpy(raw), torch.from_numpy(sc))
        assert (deq.numpy().view(np.uint16) == oracle.dequant(raw, sc, E, M).view(np.uint16)).all()
    raw, sc, _ = synth.uniform_problem(71, 256, 320, 1, 3, 2)
    assert torch.equal(ext.weight_prepacking_cpu(torch.from_numpy(raw)), fp6.weight_prepacking_cpu(torch.from_numpy(raw)))
    assert torch.equal(ext.weight_dequant_cpu(torch.from_numpy(raw), torch.from_numpy(sc)), fp6.weight_dequant_cpu(torch.from_numpy(raw), torch.from_numpy(sc)))
    with pytest.raises(ValueError):
        ext.weight_prepacking_cpu(torch.zeros((100, 12), dtype=torch.int32))           # OC % 256 (the reference asserts)
    with pytest.raises(ValueError):
        ext.weight_prepacking_eXmY_cpu(4, 3, torch.zeros((256, 16), dtype=torch.int32))  # a format nobody has
    with pytest.raises(ValueError):
        ext.weight_dequant_cpu(torch.zeros((256, 12), dtype=torch.int32), torch.zeros(255, dtype=torch.float16))


def test_which_biases_the_kernels_add():
    """A plain fp16 vector beside the input; whatever autograd, a transform or another type has a part in stays a torch addition."""
    from torch.autograd import forward_ad
    from fp6_llm_amd.module import FPxLinear
    layer, x = FPxLinear(64, 256), torch.zeros(1, 64, dtype=torch.float16)
    assert not layer._bias_in_kernel(x)   # none
    half = torch.ones(256, dtype=torch.float16)
    for bias, want in ((half, True), (half.float(), False), (half[:1], False), (torch.ones(512, dtype=torch.float16)[::2], False), (half[None], False)):
        layer.bias = bias
        assert layer._bias_in_kernel(x) is want
    layer.bias = half.clone().requires_grad_()
    assert not layer._bias_in_kernel(x)
    with torch.no_grad():
        assert layer._bias_in_kernel(x)
    layer.bias = half
    with forward_ad.dual_level():
        assert not layer._bias_in_kernel(x)
    seen = []
    torch.func.vmap(lambda z: (z, seen.append(layer._bias_in_kernel(x)))[0])(torch.zeros(2))
    assert seen == [False]


@pytest.mark.parametrize("above,rows,library", [("auto", 3072, False), ("auto", 32767, False), ("auto", 32768, True), (3072, 3072, True), (3072, 3071, False), (None, 32768, False)])
def test_which_route_a_long_prompt_takes(monkeypatch, above, rows, library):
    """dequant_above: "auto" keeps the mixed-input kernels up to 32768 rows, a number of the user's own is taken as it stands, also when it is set later."""
    import copy
    from fp6_llm_amd import module
    monkeypatch.setattr(module, "weight_dequant_native_cuda", lambda *a: torch.full((256, 64), 2.0, dtype=torch.float16))
    monkeypatch.setattr(module, "linear_forward_native", lambda E, M, x, *a: torch.full((x.shape[0], 256), -1.0, dtype=torch.float16))
    layer = module.FPxLinear(64, 256, dequant_above=above)
    later = module.FPxLinear(64, 256)
    later.dequant_above = 3072 if above == 3072 else layer.dequant_above
    x = torch.ones(rows, 64, dtype=torch.float16)
    for l in (layer, later, copy.deepcopy(layer)):
        assert float(l(x)[0, 0]) == (128.0 if library else -1.0)


def _long_prompt_stubs(monkeypatch):
    """FPxLinear's two routes without a GPU: the kernels answer -1 and are no part of any graph, dequantized weights are all 2."""
    from fp6_llm_amd import module
    monkeypatch.setattr(module, "weight_dequant_native_cuda", lambda *a: torch.full((256, 64), 2.0, dtype=torch.float16))
    monkeypatch.setattr(module, "linear_forward_native", lambda E, M, x, *a: torch.full((x.shape[0], 256), -1.0, dtype=torch.float16))
    return module


@pytest.mark.parametrize("bias", [False, True])
def test_long_prompts_that_something_follows_keep_the_library_route(monkeypatch, bias):
    """From 3072 rows on an input that is differentiated (backward, forward mode, torch.func), mapped over, traced, seen by a dispatch mode or a subclass, cast by
    autocast or off a 16-byte boundary goes through torch.nn.functional.linear, as it always did."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    module = _long_prompt_stubs(monkeypatch)
    layer = module.FPxLinear(64, 256, bias=torch.ones(256, dtype=torch.float16) if bias else None)
    want, kernels = 128.0 + bias, -1.0 + bias
    monkeypatch.setattr(module.FPxLinear, "_bias_in_kernel", lambda self, x2: False)
    x = torch.ones(3072, 64, dtype=torch.float16)
    assert float(layer(x)[0, 0]) == kernels and float(layer(x[:, None, :])[0, 0, 0]) == kernels

    g = x.clone().requires_grad_()
    (g.sum() + layer(g).sum(dtype=torch.float32)).backward()
    assert torch.equal(g.grad, torch.full_like(x, 513.0))                     # 1 + 256 * 2
    f = torch.ones(3072, 64, requires_grad=True)                              # (float32: cast to fp16 on the way in)
    layer(f).sum(dtype=torch.float32).backward()
    assert torch.equal(f.grad, torch.full_like(f, 512.0))
    with torch.no_grad():
        assert float(layer(g)[0, 0]) == kernels
    with forward_ad.dual_level():
        y = forward_ad.unpack_dual(layer(forward_ad.make_dual(x, x)))
        assert float(y.tangent[0, 0]) == 128.0 and float(y.primal[0, 0]) == want
    assert float(torch.func.vmap(layer)(x[None])[0, 0, 0]) == want
    assert float(torch.func.grad(lambda z: layer(z).sum(dtype=torch.float32))(x)[0, 0]) == 512.0
    traced = torch.jit.trace(layer.forward, (x,), check_trace=False)
    assert float(traced(2 * x)[0, 0]) == 256.0 + bias

    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))
    with Seen():
        assert float(layer(x)[0, 0]) == want
    assert any("mm" in n for n in Seen.names)

    class Sub(torch.Tensor):
        pass
    assert type(layer(x.as_subclass(Sub))) is Sub
    with torch.autocast("cpu", torch.bfloat16):
        y = layer(x)
    assert float(y[0, 0]) == want and (y.dtype == torch.bfloat16 or bias)
    off = torch.ones(3072 * 64 + 1, dtype=torch.float16)[1:].view(3072, 64)
    assert off.data_ptr() % 16 and float(layer(off)[0, 0]) == want
    neg = torch._neg_view(x)
    assert float(layer(neg)[0, 0]) == -128.0 + bias


def test_a_torch_without_the_private_names_keeps_the_torch_operations(monkeypatch):
    """Whether a transform or a mode is active is asked by names of torch's own that another version may lack: then nothing is passed by."""
    module = _long_prompt_stubs(monkeypatch)
    layer, x = module.FPxLinear(64, 256, bias=torch.ones(256, dtype=torch.float16)), torch.ones(3072, 64, dtype=torch.float16)
    assert layer._bias_in_kernel(x) and layer._kernels_take(x)
    for owner, name in ((module, "_peek_transform"), (module, "_dispatch_modes")):
        with monkeypatch.context() as m:
            m.setattr(owner, name, None)
            assert not layer._bias_in_kernel(x) and not layer._kernels_take(x) and float(layer(x)[0, 0]) == 129.0
    with monkeypatch.context() as m:
        m.delattr(torch.autograd.forward_ad, "_current_level")
        assert not layer._bias_in_kernel(x) and not layer._kernels_take(x) and float(layer(x)[0, 0]) == 129.0


def test_dequant_above_says_what_it_does(monkeypatch):
    """The number that is read is the number of rows from which weights are dequantized: "auto" reads PREFILL_CROSSOVER, which a subclass may lower, or 3072
    where the wide tiles do not run; whole modules pickled before it was a property keep their route."""
    import copy
    import pickle
    import types
    module = _long_prompt_stubs(monkeypatch)
    x = torch.ones(33000, 64, dtype=torch.float16)

    def library_from(layer, rows):
        assert layer.dequant_above == rows
        assert float(layer(x[:rows])[0, 0]) == 128.0 and float(layer(x[:rows - 1])[0, 0]) == -1.0
    def layer_is_auto(layer):   # what requires a gradient still gets it
        return layer(x[:3072].clone().requires_grad_()).requires_grad
    plain = module.FPxLinear(64, 256)
    assert plain.dequant_above == module.FPxLinear.PREFILL_CROSSOVER
    for layer in (plain, copy.deepcopy(plain), pickle.loads(pickle.dumps(plain))):
        library_from(layer, 32768)
    for rows in (7, 3072, 32768):
        library_from(module.FPxLinear(64, 256, dequant_above=rows), rows)
        plain.dequant_above = rows
        library_from(plain, rows)
    assert not layer_is_auto(plain)
    for auto in ("auto", module.FPxLinear(64, 256).dequant_above):
        plain.dequant_above = auto
        library_from(plain, 32768)
        assert layer_is_auto(plain)
    plain.dequant_above = None
    assert plain.dequant_above is None and float(plain(x)[0, 0]) == -1.0

    for rows in (100, 3072, 5000):
        monkeypatch.setattr(module.FPxLinear, "PREFILL_CROSSOVER", rows)
        library_from(module.FPxLinear(64, 256), rows)
    monkeypatch.setattr(module.FPxLinear, "PREFILL_CROSSOVER", 32768)
    monkeypatch.setattr(module.FPxLinear, "_wide_tiles", lambda self, device: False)
    library_from(module.FPxLinear(64, 256), 3072)
    monkeypatch.undo()
    _long_prompt_stubs(monkeypatch)
    part = module.FPxLinear(64, 256)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: types.SimpleNamespace(multi_processor_count=32))
    assert not part._wide_tiles(torch.device("cuda:0")) and part._wide_tiles(torch.device("cpu"))
    assert not module.FPxLinear((1 << 20) + 64, 256)._wide_tiles(torch.device("cpu"))

    # the state of a whole module as earlier versions pickled it
    for held, rows in ((3072, 3072), (module._AutoRows(3072), 32768), (512, 512)):
        state = {k: v for k, v in module.FPxLinear(64, 256).__dict__.items() if k not in ("_auto", "_rows")}
        old = module.FPxLinear.__new__(module.FPxLinear)
        old.__setstate__(dict(state, dequant_above=held))
        library_from(old, rows)


def test_a_split_for_decoding_is_not_taken_for_long_prompts(monkeypatch):
    """split_k=4 of 28672 features would keep 15 GB of partial sums for 32767 rows; under "auto" long prompts take the heuristic's split, as they took none
    before they ran on the kernels.  With a threshold of the user's own, or none, the split holds for all rows that the kernels get."""
    module = _long_prompt_stubs(monkeypatch)
    splits = []
    monkeypatch.setattr(module, "linear_forward_native", lambda E, M, x, w, s, OC, sk, *a: (splits.append(sk), torch.zeros(x.shape[0], OC, dtype=torch.float16))[1])
    monkeypatch.setattr(module, "heuristic_splitk_mi355x", lambda *a: 77)
    x = torch.ones(32767, 64, dtype=torch.float16)
    for above, rows, want in (("auto", 1, 4), ("auto", 3071, 4), ("auto", 3072, 77), ("auto", 32767, 77), (None, 3072, 4), (4000, 3999, 4)):
        module.FPxLinear(64, 256, split_k=4, dequant_above=above)(x[:rows])
        assert splits.pop() == want, (above, rows)


def test_a_call_reads_every_buffer_once(monkeypatch):
    """A read of a buffer is a call of nn.Module.__getattr__, half a microsecond beside kernels of four: a forward pass without a bias takes four."""
    module = _long_prompt_stubs(monkeypatch)
    layer, x, names = module.FPxLinear(64, 256), torch.ones(8, 64, dtype=torch.float16), []
    layer(x)
    found = torch.nn.Module.__getattr__
    monkeypatch.setattr(module.FPxLinear, "__getattr__", lambda self, name: (names.append(name), found(self, name))[1], raising=False)
    layer(x)
    assert sorted(names) == ["bias", "group_exps", "scales", "weight_native"]


def test_a_split_of_the_heuristics_is_launched_by_what_it_was_chosen_for():
    """From 97 columns on the heuristic's split is launched by gemm_wide or by the table's shape for that very split; the rules launch one only where the table
    holds no split of the problem.  1024x8192 N 600 was cut in three for gemm_wide and launched with a tile of the rules, whose time nothing had compared."""
    L = _lib.lib()
    shape = (ctypes.c_int * 5)()
    rng = np.random.default_rng(12)
    problems = [(3, 2, 1024, 8192, 600), (3, 2, 1024, 8192, 800), (3, 2, 2048, 8192, 500), (3, 2, 1280, 2624, 525)]
    for _ in range(4000):
        problems.append((*FORMATS[rng.integers(len(FORMATS))], 256 * int(2 ** rng.uniform(0, 7)), 64 * int(2 ** rng.uniform(0, 9)), int(2 ** rng.uniform(6.6, 12))))
    cut = 0
    for E, M, OC, IC, N in problems:
        split = fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M)
        for grouped in (0, 1):
            assert L.fp6mi_query_kernel(E, M, OC, N, IC, split, grouped, shape) == 0
            if shape[0] == 2 and ((shape[3] == 4 and shape[4] <= 2) or shape[3] == 2):   # gemm_wide, or gemm_prefill in the place of a shape of the table's
                cut += split > 1
                continue
            if L.fp6mi_query_table(E, M, OC, N, IC, split, None) == 2:
                assert all(L.fp6mi_query_table(E, M, OC, N, IC, s, None) == 2 for s in (1, 2, 3, 4, 6, 8)), (E, M, OC, IC, N, split, tuple(shape))
    assert cut > 100


def test_splits_stay_within_the_workspaces_they_are_chosen_for():
    """Where gemm_wide took the table's place the heuristic asked for up to 370 MB of partial sums, and ordinary prompts for more than the static workspace holds
    (which the table had left uncut).  The C heuristic's splits fit that one, but for the few that the table itself holds; Python's stay under 96 MiB, and are
    also taken by the workspace that the C answer fits into."""
    L = _lib.lib()
    static = L.fp6mi_static_workspace_bytes()
    for OC, IC, N in ((8192, 28672, 512), (8192, 8192, 600), (5120, 8192, 800), (4096, 14336, 700), (5120, 21952, 896), (6912, 27712, 257), (1280, 24384, 1117)):
        for E, M in ((3, 2), (2, 2)):
            assert L.fp6mi_workspace_bytes(OC, N, L.fp6mi_heuristic_splitk_format(E, M, OC, N, IC, 256)) <= static, (OC, IC, N)
    for OC, IC, N in ((13568, 24704, 364), (12800, 28288, 365), (12544, 25664, 355)):   # the table's choice once its times are scaled to N, not before
        assert L.fp6mi_workspace_bytes(OC, N, L.fp6mi_heuristic_splitk(OC, N, IC, 256)) <= static, (OC, IC, N)
    rng = np.random.default_rng(13)
    most, beyond, fewer = 0, 0, 0
    for _ in range(20000):
        E, M = FORMATS[rng.integers(len(FORMATS))]
        OC, IC, N = 256 * int(2 ** rng.uniform(0, 6.8)), 64 * int(2 ** rng.uniform(2, 8.8)), int(2 ** rng.uniform(6.6, 15))
        c, py = L.fp6mi_heuristic_splitk_format(E, M, OC, N, IC, 256), fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M)
        most, beyond = max(most, L.fp6mi_workspace_bytes(OC, N, py)), beyond + (L.fp6mi_workspace_bytes(OC, N, c) > static)
        fewer += c != py
        assert c == py or L.fp6mi_workspace_bytes(OC, N, py) > static or c > py
        assert c == L.fp6mi_heuristic_splitk_within(E, M, OC, N, IC, 256, static)
    assert most <= fp6.SPLIT_WORKSPACE_BYTES and beyond <= 20000 // 100 and fewer > 100


@pytest.mark.parametrize("E,M,OC,IC,N,grouped,wide", [
    (2, 2, 1024, 6144, 1848, 0, False), (2, 1, 2560, 19904, 3224, 0, False), (2, 2, 1536, 14336, 691, 0, False), (3, 2, 1024, 16000, 774, 0, False),
    (2, 2, 768, 5504, 2310, 0, False), (2, 2, 1792, 28288, 807, 1, False), (2, 2, 2048, 2304, 616, 0, False),   # 1.11 to 1.24 with 64-column tiles
    (3, 2, 5632, 256, 325, 0, False), (2, 1, 512, 256, 2951, 0, False), (3, 2, 21504, 384, 172, 1, False), (3, 2, 14336, 512, 220, 0, False),         # 1.05 to 1.22 with little K
    (3, 2, 4608, 2816, 545, 0, True), (3, 2, 512, 8960, 2877, 0, True), (3, 2, 5632, 4096, 1000, 0, True), (3, 2, 4096, 960, 609, 0, True),
    (2, 2, 28672, 512, 500, 0, True)])
def test_where_the_wide_kernel_does_not_pay(E, M, OC, IC, N, grouped, wide):
    """Problems on which gemm_wide took 1.05 to 1.24 of the time of the shape whose place it took, unsplit, and some beside them where it takes less."""
    shape = (ctypes.c_int * 5)()
    assert _lib.lib().fp6mi_query_kernel(E, M, OC, N, IC, 1, grouped, shape) == 0
    assert (shape[0] == 2 and shape[3] == 4 and shape[4] <= 2) == wide, tuple(shape)


@pytest.mark.parametrize("OC,IC,N,shape", [
    (1280, 1216, 21, (0, 1, 1, 1, 8)), (4096, 1152, 20, (0, 1, 2, 1, 8)), (2304, 1152, 70, (0, 1, 3, 1, 8)), (4096, 1152, 33, (0, 1, 2, 1, 8)), (4096, 1152, 49, (0, 1, 2, 1, 8)), (4096, 1152, 65, (0, 1, 2, 1, 4)),
    (4096, 1152, 96, (0, 1, 2, 1, 4)), (4096, 320, 32, (0, 1, 1, 1, 4)), (4096, 320, 48, (0, 1, 2, 1, 4)), (4096, 768, 128, (0, 1, 2, 1, 4)), (768, 1344, 256, (0, 1, 3, 1, 8)),
    (4096, 1152, 97, None), (4096, 320, 129, None), (4096, 256, 20, None), (4096, 1024, 24, None)])   # more outputs, a single K block, four of them: tiles
def test_little_k_takes_the_stream_kernel_unsplit(OC, IC, N, shape):
    """Up to K 1408 the rules never split, and give few outputs to the stream kernel; its shapes on both sides of each line."""
    got = (ctypes.c_int * 5)()
    assert fp6.heuristic_splitk_mi355x(OC, N, IC) == 1
    assert _lib.lib().fp6mi_query_table(3, 2, OC, N, IC, 1, got) == 2
    assert tuple(got) == shape if shape else got[0] == 1


@pytest.mark.parametrize("OC,IC,N,split", [(2048, 3264, 6, False), (1536, 3840, 2, False), (2304, 2176, 13, False), (2048, 2304, 26, False), (2560, 7744, 2, False), (9216, 1408, 24, False),
                                           (1536, 28096, 13, True), (1280, 28288, 1, True), (4864, 9536, 25, True), (5120, 14784, 13, True), (1792, 22464, 3, True)])
def test_small_batches_are_split_for_long_rows_only(OC, IC, N, split):
    """Matrices off the table: measured, the first are 0.64 to 0.95 of the time uncut, the others 1.2 to 1.7."""
    assert (fp6.heuristic_splitk_mi355x(OC, N, IC) > 1) == split


class _OnGpu:
    """A CPU tensor that says it is on the GPU, for checks that come before the first use of a device."""

    def __init__(self, t):
        self._t, self.device = t, torch.device("cuda", 0)

    def __getattr__(self, name):
        return getattr(self._t, name)


@pytest.mark.parametrize("OC,IC", [(16, 64), (256, 320)])
def test_dequantizer_refuses_scales_and_weights_it_would_read_wrongly(OC, IC, monkeypatch):
    """Fewer scales than rows would be read out of range, other types and strided codes as other values: refused before anything is allocated or launched."""
    monkeypatch.setattr(fp6, "_ext", None)
    for E, M in fp6.FORMATS:
        native, scales = torch.zeros(fp6.native_bytes(E, M, OC, IC) // 4, dtype=torch.int32), torch.ones(OC, dtype=torch.float16)
        strided = torch.zeros(2 * native.numel(), dtype=torch.int32)[::2]
        for w, s in ((native, scales[:-1]), (native, scales[:0]), (native, scales[0]), (native, scales.float()), (native, scales.bfloat16()), (strided, scales)):
            with pytest.raises(ValueError):
                fp6.weight_dequant_native_cuda(E, M, _OnGpu(w), _OnGpu(s), OC, IC)


class _Whole:
    def __init__(self, index):
        if index:
            self.__class__ = type("Index", (), {"__index__": lambda _: 256})
        else:
            self.__class__ = type("Int", (), {"__int__": lambda _: 256, "__float__": lambda _: 256.0})


@pytest.mark.parametrize("value", [256, True, 0, -1, 2 ** 63 - 1, 2 ** 63, -2 ** 70, 256.0, "256", None, 1j, np.int64(256), np.uint8(3), np.float32(256), np.float16(256), np.float64(256),
                                   np.array(256), np.array(256.0), np.array([2, 3]), fractions.Fraction(256), decimal.Decimal(256), torch.tensor(256), torch.tensor(256.0), torch.tensor([2, 3]),
                                   torch.tensor(256).half(), float("nan"), np.float32("nan"), _Whole(True), _Whole(False)], ids=lambda v: type(v).__name__ + " " + str(v)[:12])
def test_positional_call_takes_the_numbers_that_the_dispatcher_takes(value):
    """Formats, rows and splits given as whole numbers of any kind: one entry point gets as far as the other (here to the first check, of tensors that are not on a GPU), or raises the same."""
    if fp6._ext is None:
        pytest.skip("the extension is not built")
    x, w, s = torch.zeros(1, 256, dtype=torch.float16), torch.zeros(fp6.native_bytes(3, 2, 256, 256) // 4, dtype=torch.int32), torch.ones(256, dtype=torch.float16)
    for at in (0, 1, 5, 6):
        args = [3, 2, x, w, s, 256, 1, None, None, None, None]
        args[at] = value
        ended = []
        for call in (fp6._ext.linear_forward_native, fp6._ext.linear_forward_positional):
            with pytest.raises(Exception) as e:
                call(*args)
            ended.append((e.type, str(e.value) if e.type is ValueError else ""))
        assert ended[0] == ended[1], at


@pytest.mark.parametrize("whole", [3, np.int64(3), np.uint8(3), torch.tensor(3), np.array(3)], ids=lambda v: type(v).__name__)
@pytest.mark.parametrize("broken", [3.0, np.float32(3), np.float32(3.7), torch.tensor(3.7), fractions.Fraction(7, 2), "3", None], ids=lambda v: type(v).__name__ + str(v)[:12])
def test_weight_preparation_takes_whole_numbers_only(whole, broken):
    """The extension's entry points, like the Python path behind them, refuse a format or a size that is no integer instead of cutting its fraction off.  (A tensor that is
    not on a GPU ends a call whose numbers are taken with None.)"""
    if fp6._ext is None:
        pytest.skip("the extension is not built")
    t = torch.zeros(256, 12, dtype=torch.int32)
    calls = [lambda v: fp6._ext.to_native(t, v, 2), lambda v: fp6._ext.to_native(t, 3, v), lambda v: fp6._ext.weight_quantize_native(v, 2, t, False),
             lambda v: fp6._ext.weight_quantize_native(3, v, t, False), lambda v: fp6._ext.weight_dequant_native(v, 2, t, t, 256, 64, None),
             lambda v: fp6._ext.weight_dequant_native(3, v, t, t, 256, 64, None), lambda v: fp6._ext.weight_dequant_native(3, 2, t, t, v, 64, None),
             lambda v: fp6._ext.weight_dequant_native(3, 2, t, t, 256, v, None)]
    for call in calls:
        assert call(whole) is None
        with pytest.raises(TypeError):
            call(broken)


@pytest.mark.parametrize("E,M,OC,IC,N,split,shape", [
    (2, 3, 2560, 1856, 789, 1, (2, 5, 2, 4, 2)), (3, 2, 2048, 2624, 1219, 1, (2, 5, 2, 4, 2)), (3, 2, 2048, 2432, 1218, 1, (2, 5, 2, 4, 2)), (2, 1, 6400, 11136, 202, 4, (2, 8, 4, 4, 2)),
    (2, 3, 3584, 12480, 411, 4, (2, 8, 4, 4, 2))])
def test_a_tile_of_gemm_span_that_is_not_ahead_by_enough_leaves_the_place_to_gemm_wide(E, M, OC, IC, N, split, shape):
    """Where gemm_span's tile is expected to be the fastest, but not by the margin that it is held to against the table, gemm_wide's own fastest is asked, which is held to less; if that
    passes, the span tile, which is ahead of it, is launched at that split.  Measured, us, the table's shape that was taken instead, gemm_wide's and this one: 17.4, 14.7 and 13.8; 22.5,
    20.0 and 19.0; 21.0, 18.0 and 17.2; 47.7 (uncut) and 40.7; 51.0 (in two) and 48.7."""
    got = (ctypes.c_int * 5)()
    assert fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M) == split
    assert _lib.lib().fp6mi_query_kernel(E, M, OC, N, IC, split, 0, got) == 0 and tuple(got) == shape


W64, W96, W128, T96, T128 = (2, 4, 2, 4, 2), (2, 6, 2, 4, 2), (2, 8, 2, 4, 2), (2, 6, 4, 4, 1), (2, 8, 4, 4, 2)   # gemm_wide: 64-128 columns; 256 rows
S48, S80, S112, S80T, S96T, S112T = (2, 3, 2, 4, 2), (2, 5, 2, 4, 2), (2, 7, 2, 4, 2), (2, 5, 4, 4, 2), (2, 6, 4, 4, 2), (2, 7, 4, 4, 2)   # gemm_span


@pytest.mark.parametrize("E,M,OC,IC,N,grouped,split,shape", [
    # from K 1024
    (2, 2, 2560, 960, 1926, 0, 1, T96), (2, 2, 2560, 1024, 1926, 0, 1, S80T), (2, 1, 8192, 960, 440, 0, 1, W64), (2, 1, 8192, 1024, 440, 0, 1, S112),
    # 128 x 48 up to N 600, 128 x 112 uncut without group exponents up to 1400, the others up to 3072
    (3, 2, 1536, 11328, 601, 0, 1, W64), (3, 2, 2304, 3584, 600, 0, 1, S48), (3, 2, 2304, 3584, 601, 0, 1, W64), (2, 1, 2304, 4992, 1400, 0, 1, S112), (2, 1, 2304, 4992, 1401, 0, 1, W128), (2, 1, 2304, 4992, 1401, 1, 1, S112),
    (2, 2, 2048, 2176, 3072, 0, 1, S96T), (2, 2, 2048, 2176, 3073, 0, 1, T128),
    # 128 x 112 uncut with K from 8192: not where the last round is less than seven eighths full, with group exponents not near 128 x 96; a last round from three quarters on counts 3 % more
    (2, 2, 2560, 8128, 1225, 0, 1, S112), (2, 2, 2560, 8192, 1225, 0, 1, W128), (3, 2, 5632, 20800, 408, 1, 1, W96), (2, 2, 3328, 8128, 784, 1, 1, S112), (2, 2, 3328, 8192, 784, 1, 1, W96), (2, 2, 6912, 11008, 409, 1, 1, S112), (2, 1, 3328, 6144, 784, 0, 1, S112), (2, 1, 3328, 6144, 785, 0, 1, W96),
    (3, 2, 2048, 2176, 1635, 0, 1, W128),
    # 256 x 80 uncut, more columns than rows, K from 4096: not near 128 x 128 (1.11, 1.10 and 1.07 of its time), but where another tile of gemm_span is ahead of that (0.94 of its)
    (3, 2, 1536, 14976, 2641, 0, 1, W128), (2, 2, 1792, 11520, 2304, 0, 1, W128), (2, 1, 1792, 7552, 2223, 0, 1, W128), (3, 2, 2048, 4096, 2552, 0, 1, S80T), (2, 3, 1536, 16448, 2161, 0, 1, W128),
    # 128 x 48 in a single round against the table's shapes, K of a piece from 4096
    (3, 2, 1280, 8064, 195, 0, 2, S48), (3, 2, 1280, 8192, 195, 0, 2, (1, 2, 1, 4, 4)), (2, 3, 2048, 4032, 579, 0, 1, S48), (2, 3, 2048, 4096, 579, 0, 1, (2, 4, 2, 4, 4)),
    (2, 2, 2816, 18304, 326, 1, 1, (2, 4, 2, 4, 4)), (2, 2, 2048, 26816, 582, 0, 1, (2, 4, 2, 4, 4))])
def test_where_gemm_span_is_launched(E, M, OC, IC, N, grouped, split, shape):
    """The shapes on both sides of each line of span_margin and wide_replaces."""
    got = (ctypes.c_int * 5)()
    assert _lib.lib().fp6mi_query_kernel(E, M, OC, N, IC, split, grouped, got) == 0 and tuple(got) == shape


@pytest.mark.parametrize("E,M,OC,IC,N,split,shape", [
    # uncut tiles of 128 rows, and 128 x 112 in pieces, decide no split: measured, us, uncut and this one 52.8 and 45.7, 66.8 and 59.2, 55.5 and 49.3, 92.4 and 83.5 (with 256 x 128), 46.8 and 42.8
    (2, 3, 3328, 8640, 585, 3, T128), (3, 2, 4352, 11200, 543, 3, T128), (2, 2, 5120, 9152, 451, 3, T128), (3, 2, 3584, 12800, 945, 2, S112T), (2, 2, 9984, 7488, 216, 3, T128),
    # where the others answer with the same split they are launched
    (2, 2, 4608, 4544, 777, 1, S112), (3, 2, 8192, 4992, 445, 1, S112), (2, 1, 20736, 4992, 142, 1, S48),
    # those of 256 rows decide splits, uncut 256 x 80 up to K 20480
    (3, 2, 17408, 7168, 196, 1, S80T), (2, 2, 4864, 5632, 1067, 1, S96T), (2, 3, 2816, 20480, 1552, 1, S80T), (2, 3, 2816, 20544, 1552, 3, (2, 8, 4, 4, 1))])
def test_which_tiles_of_gemm_span_choose_a_split(E, M, OC, IC, N, split, shape):
    got = (ctypes.c_int * 5)()
    assert fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M) == split
    assert _lib.lib().fp6mi_query_kernel(E, M, OC, N, IC, split, 0, got) == 0 and tuple(got) == shape


@pytest.mark.parametrize("E,M,OC,IC,N,shape", [
    # 5 bits: beyond 128 columns no second round of two row tiles on eight wavefronts; three tiles where they fill one, four wavefronts beyond four outputs' tiles a CU, other formats as before
    (2, 2, 512, 1280, 256, (0, 1, 2, 1, 8)), (2, 2, 512, 1280, 257, (0, 1, 3, 1, 8)), (2, 2, 512, 1280, 385, (1, 2, 1, 4, 4)), (3, 2, 512, 1280, 385, (0, 1, 2, 1, 8)), (2, 1, 512, 1280, 385, (0, 1, 2, 1, 8)),
    (2, 2, 1280, 1152, 144, (0, 1, 3, 1, 8)), (2, 2, 1280, 1152, 145, (1, 2, 1, 4, 4)), (2, 2, 2048, 1280, 128, (0, 1, 2, 1, 8)), (2, 2, 2048, 1280, 129, (0, 1, 2, 1, 4)), (2, 2, 2560, 1216, 78, (0, 1, 2, 1, 8)),
    # K 1344 is the rules' whatever M and N are, K 1408 is in the table's reach
    (3, 2, 1280, 1344, 200, (0, 1, 2, 1, 4)), (3, 2, 28672, 1344, 17, (1, 2, 2, 4, 2)), (3, 2, 1280, 1408, 200, None), (3, 2, 4096, 1408, 24, None)])
def test_little_k_by_format_and_where_the_table_begins(E, M, OC, IC, N, shape):
    got = (ctypes.c_int * 5)()
    source = _lib.lib().fp6mi_query_table(E, M, OC, N, IC, 1, got)
    if shape:
        assert source == 2 and tuple(got) == shape and fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M) == 1
    else:
        assert source == 1


def test_a_module_finds_buffers_parameters_and_submodules():
    """FPxLinear looks for a buffer before nn.Module does, and finds and refuses what nn.Module does: with and without a bias, before __init__, copied, pickled, with its buffers
    replaced or taken out, and as a subclass with parameters and modules of its own."""
    import copy
    import pickle

    from fp6_llm_amd import module

    class Wrapped(module.FPxLinear):
        def __init__(self):
            super().__init__(64, 256, bias=torch.ones(256, dtype=torch.float16))
            self.gain = torch.nn.Parameter(torch.ones(3))
            self.inner = torch.nn.Linear(2, 2)

        @property
        def broken(self):
            raise AttributeError("broken has no value")

    plain, wrapped = module.FPxLinear(64, 256), Wrapped()
    assert plain.bias is None and plain.group_exps is None and wrapped.bias is wrapped._buffers["bias"] and wrapped.gain is wrapped._parameters["gain"] and wrapped.inner is wrapped._modules["inner"]
    for m in (plain, wrapped):
        assert m.scales is m._buffers["scales"] and m.weight_native is m._buffers["weight_native"]
        for name in ("nothing", "_buffer", "weight"):
            with pytest.raises(AttributeError, match=name):
                getattr(m, name)
            assert not hasattr(m, name)
    with pytest.raises(AttributeError):
        wrapped.broken
    bare = module.FPxLinear.__new__(module.FPxLinear)   # before nn.Module has made its dictionaries
    for name in ("_buffers", "scales", "training_steps"):
        with pytest.raises(AttributeError):
            getattr(bare, name)
    for other in (copy.deepcopy(plain), copy.copy(plain), pickle.loads(pickle.dumps(plain))):
        assert torch.equal(other.scales, plain.scales) and other.bias is None and list(other.state_dict()) == list(plain.state_dict())
    plain.scales = torch.full_like(plain.scales, 2.0)
    assert plain.scales is plain._buffers["scales"] and (plain.scales == 2).all()
    swapped = torch.zeros_like(plain.scales)
    got = torch.func.functional_call(_Reads(plain), {"layer.scales": swapped}, ())
    assert got is swapped and plain.scales is not swapped
    del plain.scales
    with pytest.raises(AttributeError, match="scales"):
        plain.scales


class _Reads(torch.nn.Module):
    def __init__(self, layer):
        super().__init__()
        self.layer = layer

    def forward(self):
        return self.layer.scales


@pytest.mark.parametrize("E,M,OC,IC,N,split,shape", [
    (2, 2, 2048, 14144, 21, 8, (1, 2, 1, 4, 4)), (3, 2, 2304, 7360, 18, 6, (1, 2, 1, 4, 4)), (3, 2, 2304, 6784, 24, 6, (1, 2, 1, 4, 4)), (2, 1, 2048, 19264, 25, 8, (1, 2, 1, 4, 4)),
    (2, 2, 2048, 14144, 16, 4, (0, 1, 2, 1, 8)), (2, 2, 2048, 2176, 21, 1, (0, 1, 1, 1, 4))])   # up to 16 columns, and uncut, it is the stream kernel's
def test_a_cut_stream_kernel_does_not_replace_a_cut_tile_kernel(E, M, OC, IC, N, split, shape):
    """17 to 32 columns, matrices off the table: measured, us, in three or four pieces of the stream kernel and here, 12.1 and 10.0, 10.3 and 9.0, 10.7 and 9.2."""
    got = (ctypes.c_int * 5)()
    assert fp6.heuristic_splitk_mi355x(OC, N, IC, EXPONENT=E, MANTISSA=M) == split
    assert _lib.lib().fp6mi_query_kernel(E, M, OC, N, IC, split, 0, got) == 0 and tuple(got) == shape
