"""Host-side checks that need no GPU: the C-ABI library loads, exports what include/fcr.h
declares, rejects bad arguments before touching the device, and the Python entry point mirrors
the reference's validation (flash_colreduce/flash.py:354-364)."""
import ctypes
import os
import re

import pytest
import torch

import flash_colreduce_amd as fca
from flash_colreduce_amd import _lib
from oracle.colreduce_oracle import colreduce_ref
from tests import _inputs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "fcr.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fcr_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    names = _declared_symbols()
    assert {"fcr_version", "fcr_last_error", "fcr_lse_bytes", "fcr_row_lse", "fcr_col_reduce",
            "fcr_col_reduce_sum_max", "fcr_pack_f32", "fcr_colreduce", "fcr_colreduce_static",
            "fcr_colreduce_to", "fcr_topk_mask", "fcr_topk_mask_ws", "fcr_topk_mask_typed", "fcr_topk_bytes", "fcr_set_option",
            "fcr_colreduce_status", "fcr_colreduce_sum_max", "fcr_colreduce_sum_max_to", "fcr_workspace_bytes",
            "fcr_colreduce_ws"} <= set(names)
    for name in names:
        assert hasattr(lib, name), name


def test_version_and_sizes():
    lib = _lib.load()
    assert lib.fcr_version() == 320
    assert lib.fcr_lse_bytes(2, 3, 5, 7, 64) == 2 * 3 * 5 * 4
    assert lib.fcr_lse_bytes(1, 32, 8192, 8192, 128) == 32 * 8192 * 4      # enough row tiles: no scratch
    assert lib.fcr_lse_bytes(1, 32, 512, 16384, 128) == 32 * 512 * 4 * 9   # 8 key ranges + the result
    # few queries, many keys (256 CUs assumed without a device): the result, two sets of 64-bit slots for
    # one workgroup per CU of 128 rows, and the status line
    assert lib.fcr_lse_bytes(1, 32, 128, 4096, 128) == (32 * 128 + 2 * 2 * 256 * 128 + 32) * 4
    assert lib.fcr_lse_bytes(-1, 3, 5, 7, 8) == 0 and lib.fcr_lse_bytes(1, 3, 0, 7, 8) == 0


def test_row_sweep_scratch_covers_every_row_width():
    """fcr_lse_bytes does not know the row width: it is the most that any number of 64-byte steps of a row asks for
    (the tile height, hence the number of key ranges, depends on it), restated here for 256 CUs and more than 128 queries."""
    import random
    lib = _lib.load()
    if torch.cuda.is_available():
        pytest.skip("the sizes are restated for the 256 CUs that the library assumes without a device")
    rng = random.Random(5)

    def swept(m, rows):
        rem = m % rows
        return m // rows * rows + min((rem + 31) // 32, 4) * (rows // 4)

    def splits(bh, m, n, ksteps):
        chunks, pairs2 = (n + 63) // 64, bh * ((m + 255) // 256)
        one = (ksteps > 4 or swept(m, 128) * (100 + 3 * ksteps) < swept(m, 256) * 100 or
               (pairs2 < 256 and n <= 1024) or 256 <= pairs2 < 512)
        wgs = bh * ((m + (128 if one else 256) - 1) // (128 if one else 256))
        return 1 if wgs >= 256 or chunks < 16 else max(1, min(512 // wgs, chunks // 4, 64))

    for _ in range(3000):
        b, h, m, n = rng.randint(1, 4), rng.randint(1, 40), int(2 ** rng.uniform(7.1, 13)), int(2 ** rng.uniform(6, 18))
        most = max(splits(b * h, m, n, ks) for ks in range(1, 17))
        assert lib.fcr_lse_bytes(b, h, m, n, 64) == 4 * b * h * m * (1 + most if most > 1 else 1), (b, h, m, n)


def test_workspace_size_of_one_query():
    """One query asks for its scores and key ranges behind fcr_lse_bytes, for every row width the kernels take; for
    any other width (which the call then rejects) and for more queries it is fcr_lse_bytes."""
    lib = _lib.load()
    for dtype, limit, step in ((0, 512, 8), (1, 512, 8), (2, 256, 4)):
        for d in range(step, limit + 1, step):
            assert lib.fcr_workspace_bytes(dtype, 2, 3, 1, 1000, d) >= lib.fcr_lse_bytes(2, 3, 1, 1000, d) + 4 * 6 * 1000
        for d in (limit + step, 2 * limit, 1 << 20, 1 << 30, (1 << 31) - 1, step - 1, 0, -step):
            assert lib.fcr_workspace_bytes(dtype, 2, 3, 1, 1000, d) == lib.fcr_lse_bytes(2, 3, 1, 1000, d)
        assert lib.fcr_workspace_bytes(dtype, 2, 3, 2, 1000, 64) == lib.fcr_lse_bytes(2, 3, 2, 1000, 64)
        assert lib.fcr_workspace_bytes(dtype, 2, 3, 1, 0, 64) == 0
    assert lib.fcr_workspace_bytes(3, 2, 3, 1, 1000, 64) == lib.fcr_lse_bytes(2, 3, 1, 1000, 64)


def _call(lib, fn, **over):
    a = dict(q=16, k=32, lse=48, out=64, dtype=0, B=1, H=1, M=8, N=8, D=64,
             qs=(512, 512, 64, 1), ks=(512, 512, 64, 1), scale=0.125, red=0, causal=0)
    a.update(over)
    qs = _lib.strides4(a["qs"]) if a["qs"] is not None else None
    ks = _lib.strides4(a["ks"]) if a["ks"] is not None else None
    common = (a["dtype"], a["B"], a["H"], a["M"], a["N"], a["D"], qs, ks, a["scale"])
    if fn == "row_lse":
        return lib.fcr_row_lse(a["q"], a["k"], a["lse"], *common, a["causal"], None)
    if fn == "col_reduce":
        return lib.fcr_col_reduce(a["q"], a["k"], a["lse"], a["out"], *common, a["red"], a["causal"], None)
    if fn == "colreduce_to":
        return lib.fcr_colreduce_to(a["q"], a["k"], a["out"], a.get("out_dtype", 0), a["lse"], *common, a["red"],
                                    a["causal"], None)
    if fn == "colreduce_sum_max":
        return lib.fcr_colreduce_sum_max(a["q"], a["k"], a["out"], a.get("out_max", 80), a["lse"], *common, a["causal"],
                                         None)
    if fn == "colreduce_ws":   # no room in the workspace unless a case says so: every other error comes before that one
        return lib.fcr_colreduce_ws(a["q"], a["k"], a["out"], a.get("out_max"), a.get("out_dtype", 0), a["lse"],
                                    a.get("ws_bytes", 0), *common, a["red"], a["causal"], None)
    return lib.fcr_colreduce(a["q"], a["k"], a["out"], a["lse"], *common, a["red"], a["causal"], None)


@pytest.mark.parametrize("fn", ["row_lse", "col_reduce", "colreduce", "colreduce_to", "colreduce_sum_max", "colreduce_ws"])
def test_c_abi_rejects_bad_arguments_without_a_device(fn):
    """Every rejection happens before the first HIP call, so fake pointers are safe here."""
    lib = _lib.load()
    cases = [
        (dict(q=None), -1), (dict(k=None), -1), (dict(lse=None), -1), (dict(qs=None), -1),
        (dict(dtype=3), -2), (dict(dtype=-1), -2),
        (dict(B=0), -3), (dict(M=0), -3), (dict(N=-4), -3), (dict(D=0), -3), (dict(D=12), -3),
        (dict(D=520), -3), (dict(D=516), -3), (dict(M=(1 << 30) + 1), -3),
        (dict(D=1 << 30), -3), (dict(dtype=2, D=(1 << 30) + 64), -3),          # D times the element size passes 2^31, 2^32
        (dict(dtype=2, D=260), -3), (dict(dtype=2, D=6), -3),                 # fp32: a multiple of 4, at most 256
        (dict(dtype=2, D=64, qs=(512, 512, 66, 1)), -4),                       # fp32: strides in multiples of 4
        (dict(qs=(512, 512, 64, 2)), -4), (dict(ks=(512, 512, 60, 1)), -4), (dict(q=18), -4),
        (dict(H=2, ks=(512, -512, 64, 1)), -4), (dict(B=2, qs=(-512, 512, 64, 1)), -4),
        (dict(H=2, qs=(512, 4, 64, 1)), -4),                                   # head stride not a multiple of 16 bytes
        (dict(B=1 << 12, H=1 << 12), -3),                                      # 2^24 workgroups: more threads than a launch may have
        (dict(qs=(512, 512, 0, 1)), -4), (dict(ks=(512, 512, 32, 1)), -4),   # overlapping rows
        (dict(scale=float("inf")), -6), (dict(scale=float("nan")), -6),
    ]
    if fn == "colreduce_to":   # takes the mean as a third reduction, and a result type
        cases += [(dict(out=None), -1), (dict(red=3), -5), (dict(red=-1), -5), (dict(out_dtype=3), -2),
                  (dict(out_dtype=-1), -2)]
    elif fn == "colreduce_ws":
        cases += [(dict(out=None), -1), (dict(red=3), -5), (dict(red=1, out_max=80), -5), (dict(out_dtype=3), -2),
                  (dict(lse=52), -4), (dict(B=1 << 12, H=1 << 12, M=1), -3), (dict(M=1), -7), (dict(ws_bytes=31), -7),
                  (dict(dtype=2, M=1, N=1000, ks=(64000, 64000, 64, 1), ws_bytes=3), -7)]
    elif fn == "colreduce_sum_max":
        cases += [(dict(out=None), -1), (dict(out_max=None), -1)]
    elif fn != "row_lse":
        cases += [(dict(out=None), -1), (dict(red=2), -5), (dict(red=-1), -5)]
    for over, code in cases:
        assert _call(lib, fn, **over) == code, over
        assert lib.fcr_last_error() != b""
    with pytest.raises(_lib.FcrError) as e:
        _lib.check(_call(lib, fn, D=12))
    assert e.value.code == -3 and "multiple of 8" in str(e.value)


def test_options_and_status_reject_bad_arguments_without_a_device():
    lib = _lib.load()
    assert lib.fcr_set_option(99, 1) == -3
    assert lib.fcr_set_option(_lib.OPT_WAIT_POLLS, -5) == -3
    assert lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1) == 0 and lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 1 << 20) == 0
    assert lib.fcr_colreduce_status(None, 0, 1, 1, 8, 8, 64, None) == -1
    assert lib.fcr_colreduce_status(16, 0, 1, 1, 0, 8, 64, None) == -3
    # problems that never take the single sweep have nothing to report: no device is asked
    assert lib.fcr_colreduce_status(16, 0, 1, 1, 512, 512, 64, None) == 0      # more than 128 queries
    assert lib.fcr_colreduce_status(16, 2, 1, 1, 64, 4096, 64, None) == 0      # fp32 operands
    assert lib.fcr_colreduce_status(16, 0, 1, 1, 64, 512, 64, None) == 0       # fewer than 1024 keys


def test_pack_f32_rejects_bad_arguments_without_a_device():
    lib = _lib.load()
    assert lib.fcr_pack_f32(None, 16, 4, 8, 3, 0, None) == -1
    assert lib.fcr_pack_f32(16, None, 4, 8, 3, 0, None) == -1
    assert lib.fcr_pack_f32(16, 32, 0, 8, 3, 0, None) == -3
    assert lib.fcr_pack_f32(16, 32, 4, 8, 2, 0, None) == -3      # terms must be 1 or 3
    assert lib.fcr_pack_f32(16, 32, 4, 88, 3, 0, None) == -3     # 3 * 88 > 256
    assert lib.fcr_pack_f32(16, 32, 4, 264, 1, 0, None) == -3


def test_python_entry_validation_matches_reference_messages():
    q = torch.zeros(1, 2, 4, 8, dtype=torch.float16)
    k = torch.zeros(1, 2, 6, 8, dtype=torch.float16)
    with pytest.raises(ValueError, match="must be on CUDA device"):
        fca.flash_colreduce(q, k, "sum")
    with pytest.raises(ValueError, match="must be on CUDA device"):
        fca.flash_colreduce(q, k, "bogus")  # device is checked first, as in the reference


def test_naive_colreduce_matches_oracle_on_config1():
    """Configuration 1 of the benchmark set: the CPU-runnable fp32 case, non-causal, all three reductions."""
    q, k = _inputs.config1()
    for red in ("sum", "mean", "max"):
        got = fca.naive_colreduce(q, k, red)
        assert got.shape == (1, 2, 256) and got.dtype == torch.float32
        want = colreduce_ref(q, k, red, compute_dtype=torch.float64).float()
        torch.testing.assert_close(got, want, rtol=2e-3, atol=1e-5)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n", [(5, 9), (9, 5), (6, 6)])
def test_naive_colreduce_matches_oracle_small(m, n, causal):
    q, k = _inputs.randn_pair(2, 3, m, n, 12, seed=m + n, dtype=torch.float32)
    for red in ("sum", "mean", "max"):
        got = fca.naive_colreduce(q, k, red, is_causal=causal, scale=0.3)
        want = colreduce_ref(q, k, red, causal, scale=0.3, compute_dtype=torch.float64).float()
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-7)
    with pytest.raises(ValueError, match="Invalid reduction"):
        fca.naive_colreduce(q, k, "median")


def test_native_host_path_leaves_the_rest_to_python():
    """Without a device nothing is for the native path: tensors on the host, other objects, wrong counts of arguments."""
    host = _lib.host()
    x = torch.zeros(1, 1, 2, 8)
    assert host.reduce(x, x, "sum", False, None, None, False) is None
    assert host.reduce(x, None, "sum", False, None, None, False) is None
    assert host.reduce(x, x, ["sum"], False, None, None, True) is None
    assert host.keep(x, 1, False) is None and host.keep("x", 1, False) is None
    with pytest.raises(TypeError):
        host.reduce(x, x)
    with pytest.raises(TypeError):
        host.keep(x)


def test_topk_scratch_is_what_the_type_can_use():
    lib = _lib.load()
    for rows in (1, 32, 1000):
        for n in (1, 32768, 32769, 65536, 65537, 1 << 20):
            plain = lib.fcr_topk_bytes(rows, n)
            assert lib.fcr_topk_bytes_typed(_lib.DTYPE_F32, rows, n) == plain and (plain > 0) == (n > 32768)
            for dtype in (_lib.DTYPE_F16, _lib.DTYPE_BF16):
                assert lib.fcr_topk_bytes_typed(dtype, rows, n) == (plain if n > 65536 else 0)
    assert lib.fcr_topk_bytes_typed(3, 32, 100000) == 0 and lib.fcr_topk_bytes_typed(_lib.DTYPE_F32, 0, 100000) == 0


def test_without_the_native_host_path_calls_go_through_python(monkeypatch):
    """_host.so missing, or built against another torch: a warning, and nothing is refused."""
    import sys
    from flash_colreduce_amd import flash as F
    monkeypatch.delattr(fca, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "flash_colreduce_amd._host", None)
    monkeypatch.setattr(F, "_native", None)
    with pytest.warns(RuntimeWarning, match="_host.so cannot be loaded"):
        host = F._host()
    x = torch.zeros(1, 1, 2, 8)
    assert F._host() is host and host.reduce(x, x, "sum", False, None, None, False) is None and host.keep(x, 1, False) is None


@pytest.fixture(scope="module")
def f32_tiles(tmp_path_factory):
    """The tile rules of the fp32 sweeps (csrc/f32_tiles.h), compiled for the host: (waves, groups) of both sweeps."""
    import subprocess
    where = tmp_path_factory.mktemp("tiles")
    (where / "t.cpp").write_text('#include "f32_tiles.h"\n'
                                 'static int code(fcr_tiles::F32Tile t) { return t.waves * 16 + t.groups; }\n'
                                 'extern "C" int col(int ks, int both, int m, int n, long long bh, int causal, int cus) {\n'
                                 '  return code(fcr_tiles::f32_col_tile(ks, both, m, n, bh, causal, cus)); }\n'
                                 'extern "C" int row(int m, int n, long long bh, int causal, int cus) {\n'
                                 '  return code(fcr_tiles::f32_row_tile(m, n, bh, causal, cus)); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flash_colreduce_amd", "csrc"),
                    str(where / "t.cpp"), "-o", str(where / "t.so")], check=True)
    lib = ctypes.CDLL(str(where / "t.so"))
    lib.col.argtypes = [ctypes.c_int] * 4 + [ctypes.c_longlong] + [ctypes.c_int] * 2
    lib.row.argtypes = [ctypes.c_int] * 2 + [ctypes.c_longlong] + [ctypes.c_int] * 2
    return (lambda *a: divmod(lib.col(*a), 16)), (lambda *a: divmod(lib.row(*a), 16))


@pytest.mark.parametrize("rows", [1, 64, 65, 128, 129, 256, 257, 300, 384, 385, 512, 513, 1000, 4097])
def test_fp32_launches_stay_below_the_runtime_limit(f32_tiles, rows):
    """Whatever passes the argument check (fewer than 2^24 tiles of 128 rows) is launched with fewer than 2^32 threads."""
    col, row = f32_tiles
    per = (rows + 127) // 128
    for bh in {2 ** e + i for e in range(24) for i in (-1, 0, 1)} | {(2 ** 24 - 1) // per}:
        if bh < 1 or bh * per >= 2 ** 24:
            continue
        for causal in (0, 1):
            tiles = [row(rows, other, bh, causal, 256) for other in (64, 2000)]
            tiles += [col(ks, both, other, rows, bh, causal, 256) for ks in (1, 4, 8) for both in (0, 1) for other in (5, 128, 300, 2000)]
            for waves, groups in tiles:
                assert (waves, groups) in ((4, 1), (4, 2), (8, 1), (8, 2))
                height = 16 * waves * groups
                assert bh * ((rows + height - 1) // height) * 64 * waves < 2 ** 32, (bh, causal, waves, groups)


def test_fp32_tiles_with_the_mask(f32_tiles):
    """One to two 128-row tiles per CU with the mask: eight waves where the sweeps differ in length, four where most are whole or short."""
    col, row = f32_tiles
    for m, n, bh, waves in ((1500, 1500, 40, 8), (1000, 1400, 40, 8), (1400, 1000, 40, 8), (1000, 1900, 30, 4), (481, 2000, 20, 4), (512, 700, 60, 4)):
        assert col(4, 0, m, n, bh, 1, 256)[0] == waves, (m, n)
    for m, n, bh, waves in ((1500, 1500, 33, 8), (1000, 1400, 33, 8), (1000, 1900, 33, 4), (2000, 700, 24, 4)):
        assert row(m, n, bh, 1, 256)[0] == waves, (m, n)
    assert col(4, 0, 2000, 2000, 20, 0, 256) == (8, 2) and col(4, 0, 2000, 2000, 48, 1, 256) == (8, 2)   # no mask; three per CU
    assert col(2, 1, 12, 15478, 2, 0, 256) == (4, 2) and col(8, 1, 128, 1024, 32, 1, 256) == (8, 1)


def test_which_calls_have_room_for_the_word_of_both_sweeps():
    """fcr_workspace_bytes holds a status word for 16-bit problems whose sweeps share a launch (with the mask or without), restated for 256 CUs
    at shapes on both sides of the rule's cuts: those on the second side lose by it, or gain nothing."""
    lib = _lib.load()
    if torch.cuda.is_available():
        pytest.skip("the rule is restated for the 256 CUs that the library assumes without a device")
    more = lambda h, m, n, d, dtype=0: lib.fcr_workspace_bytes(dtype, 1, h, m, n, d) - lib.fcr_lse_bytes(1, h, m, n, d)
    for shape in ((32, 2048, 2048, 256), (11, 4078, 4078, 128), (27, 2240, 2240, 128), (155, 1538, 1538, 128), (3, 700, 700, 128), (24, 2893, 2893, 128),
                  (10, 1895, 1895, 256), (18, 7902, 7902, 64), (60, 1000, 1000, 128), (2, 1000, 1100, 128), (250, 520, 1500, 128)):
        assert 0 < more(*shape) <= 512 and 0 < more(*shape, 1) <= 512 and more(*shape, 2) == 0, shape
    for shape in ((4, 128, 700, 128), (32, 512, 32768, 128), (68, 1090, 8104, 128), (300, 2000, 2000, 256), (216, 1562, 1562, 256), (1, 6891, 8176, 32),
                  (1, 7061, 7061, 32), (246, 314, 8281, 96), (80, 570, 570, 48), (85, 601, 601, 32), (60, 800, 800, 96), (72, 670, 670, 80)):
        assert more(*shape) == 0, shape
