"""GPU parity: libfcr (through flash_colreduce / the C ABI) against the CPU oracle on the same
seeded inputs.  Tolerances are those of the headline metric: rtol 2e-3 / atol 1e-5 for sum and mean,
2e-3 relative for max, checked on the kernel's fp32 result."""
import math

import pytest
import torch

import flash_colreduce_amd as fca
from oracle.colreduce_oracle import colreduce_ref, row_lse2_ref
from tests import _inputs

pytestmark = pytest.mark.gpu
REDUCTIONS = ["sum", "mean", "max"]


def check(got: torch.Tensor, want: torch.Tensor, reduction: str, what=""):
    got = got.detach().float().cpu()
    want = want.float()
    assert got.shape == want.shape, (got.shape, want.shape)
    assert torch.isfinite(got).all(), what
    if reduction == "max":
        rel = ((got - want).abs() / want.abs().clamp_min(1e-30)).max().item()
        assert rel <= 2e-3, f"{what} max: relative error {rel:.3e}"
    else:
        torch.testing.assert_close(got, want, rtol=2e-3, atol=1e-5, msg=lambda m: f"{what} {reduction}: {m}")


def run_all(q, k, causal, scale=None, what="", reductions=REDUCTIONS, chunk_rows=4096):
    qd, kd = q.cuda(), k.cuda()
    for red in reductions:
        got = fca.flash_colreduce(qd, kd, red, is_causal=causal, scale=scale, out_dtype=torch.float32)
        want = colreduce_ref(q, k, red, causal, scale=scale, chunk_rows=chunk_rows)
        check(got, want, red, f"{what} causal={causal}")


# --- the reference's own grid (tests/test_correctness.py:8-13), all fp16 ----------------------
@pytest.mark.parametrize("is_causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 48, 72])
@pytest.mark.parametrize("m,n", [(128, 128), (131, 131), (128, 1024), (131, 1027)])
@pytest.mark.parametrize("h", [8, 13])
@pytest.mark.parametrize("b", [1, 4, 7])
def test_reference_grid(b, h, m, n, d, is_causal):
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=0)
    run_all(q, k, is_causal, what=f"b{b} h{h} m{m} n{n} d{d}")


@pytest.mark.parametrize("is_causal", [False, True])
@pytest.mark.parametrize("reduction", REDUCTIONS)
@pytest.mark.parametrize("m,n,d", [(128, 128, 64), (131, 1027, 72), (128, 1024, 48)])
def test_reference_tolerance_on_native_dtype(m, n, d, reduction, is_causal):
    """The reference's assertion as written (tests/test_correctness.py:29-32): fp16 result against
    the materialising implementation run in fp16 on the same device, atol = rtol = 1e-3."""
    q, k = _inputs.randn_pair(4, 8, m, n, d, seed=0)
    q, k = q.cuda(), k.cuda()
    output = fca.flash_colreduce(q, k, reduction=reduction, is_causal=is_causal)
    target = fca.naive_colreduce(q, k, reduction=reduction, is_causal=is_causal)
    assert output.dtype == torch.float16 and output.shape == (4, 8, n)
    torch.testing.assert_close(output, target, atol=1e-3, rtol=1e-3)


# --- the benchmark set's five configurations ---------------------------------------------------------------
def test_config1_rounded_to_fp16():
    """Config 1 is the fp32 CPU case; the device path takes 16-bit inputs, so the kernel is fed
    the fp16 rounding of the same tensors and compared with the oracle on those."""
    q, k = _inputs.config1()
    run_all(q.half(), k.half(), False, what="config1")


def test_config1_fp32():
    """Config 1 as given: fp32 operands, multiplied as two fp16 parts (D = 64).  The device result
    is good far beyond the metric's tolerance; 1e-5 would fail with any 16-bit rounding of the operands."""
    q, k = _inputs.config1()
    qd, kd = q.cuda(), k.cuda()
    for red in REDUCTIONS:
        got = fca.flash_colreduce(qd, kd, red)
        assert got.dtype == torch.float32 and got.shape == (1, 2, 256)
        want = colreduce_ref(q, k, red, compute_dtype=torch.float64).float()
        check(got, want, red, "config1 fp32")
        torch.testing.assert_close(got.cpu(), want, rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [(100, 260, 20), (257, 300, 80), (64, 500, 128), (300, 300, 100), (33, 700, 6),
                                   (130, 140, 200), (300, 420, 132), (64, 1000, 256), (257, 129, 252),
                                   (40, 3000, 160)])
def test_fp32_operands(m, n, d, causal):
    """fp32 inputs keep their precision for every D up to 256: held to 1e-5, which no 16-bit rounding of
    the operands meets (D = 6 is zero padded to 8; rows of more than 512 bytes take the 1 KiB ring)."""
    q, k = _inputs.randn_pair(2, 2, m, n, d, seed=d, dtype=torch.float32)
    qd, kd = q.cuda(), k.cuda()
    for red in REDUCTIONS:
        got = fca.flash_colreduce(qd, kd, red, is_causal=causal, scale=0.11)
        want = colreduce_ref(q, k, red, causal, scale=0.11, compute_dtype=torch.float64).float()
        assert got.dtype == torch.float32
        check(got, want, red, f"fp32 d{d}")
        torch.testing.assert_close(got.cpu(), want, rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("terms,d,rtol", [(3, 80, 2e-5), (3, 20, 2e-5), (1, 200, 5e-3)])
def test_fp32_operands_packed_for_the_16_bit_matrix_instructions(terms, d, rtol):
    """fcr_pack_f32 + FCR_DTYPE_F16 through the C ABI: the faster, less exact way to feed fp32 operands
    (three fp16 segments give products to about 2^-22, one segment is a single rounding to fp16)."""
    from flash_colreduce_amd import _lib, flash as F
    b, h, m, n = 2, 2, 130, 700
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=terms + d, dtype=torch.float32)
    qp, kp = F.pack_f32(q.cuda(), False, terms), F.pack_f32(k.cuda(), True, terms)
    lib = _lib.load()
    out = torch.empty(b * h, n, device="cuda")
    lse = torch.empty(lib.fcr_lse_bytes(b, h, m, n, qp.shape[3]) // 4, device="cuda")
    _lib.check(lib.fcr_colreduce(qp.data_ptr(), kp.data_ptr(), out.data_ptr(), lse.data_ptr(), _lib.DTYPE_F16, b, h, m, n,
                                 qp.shape[3], _lib.strides4(qp.stride()), _lib.strides4(kp.stride()), 0.11,
                                 _lib.REDUCE_SUM, 1, torch.cuda.current_stream().cuda_stream))
    want = colreduce_ref(q, k, "sum", True, scale=0.11, compute_dtype=torch.float64).float()
    torch.testing.assert_close(out.view(b, h, n).cpu(), want, rtol=rtol, atol=1e-7)


@pytest.mark.parametrize("d", [64, 192])
def test_fp32_operands_beyond_the_fp16_range(d):
    """fp32 keeps its range: queries of magnitude 3e5 (an fp16 rounding would give inf and NaN results)
    with a scale that brings the scores back to order one, and keys of magnitude 1e-7."""
    b, h, m, n = 1, 3, 200, 333
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=77, dtype=torch.float32)
    for fq, fk in ((3e5, 1.0), (1.0, 1e-7), (2e4, 2e4)):
        qq, kk = q * fq, k * fk
        scale = 0.125 / (fq * fk)
        for red, causal in (("sum", True), ("max", False), ("mean", True)):
            got = fca.flash_colreduce(qq.cuda(), kk.cuda(), red, is_causal=causal, scale=scale)
            want = colreduce_ref(qq, kk, red, causal, scale=scale, compute_dtype=torch.float64).float()
            check(got, want, red, f"fp32 range {fq} {fk}")


def test_config2():
    q, k = _inputs.config2()
    run_all(q, k, False, what="config2")


def test_config3():
    q, k = _inputs.config3()
    run_all(q, k, True, what="config3")


def _full_size(q, k, reductions, oracle_heads, what):
    """Full-size run: every head on the GPU, the oracle on a few heads, and properties that
    hold at any size on all heads (rows of a softmax add to one; 0 < max <= 1; mean <= max)."""
    m, n = q.shape[2], k.shape[2]
    qd, kd = q.cuda(), k.cuda()
    outs = {r: fca.flash_colreduce(qd, kd, r, is_causal=True, out_dtype=torch.float32) for r in reductions}
    for r, got in outs.items():
        want = colreduce_ref(q[:, oracle_heads], k[:, oracle_heads], r, True)
        check(got[:, oracle_heads], want, r, f"{what} heads {oracle_heads}")
    if "sum" in outs or "mean" in outs:
        if "sum" in outs:
            s = outs["sum"].double()
        else:
            cnt = torch.arange(n, 0, -1, device="cuda", dtype=torch.float64) if m == n else None
            s = outs["mean"].double() * cnt
        total = s.sum(-1).cpu()
        torch.testing.assert_close(total, torch.full_like(total, float(m)), rtol=1e-4, atol=0)
    if "max" in outs:
        mx = outs["max"]
        assert (mx > 0).all() and (mx <= 1 + 1e-6).all()
        # causal, M == N: only the last query sees the last key, so max == sum == mean there
        if "mean" in outs:
            assert (outs["mean"] <= mx * (1 + 1e-5)).all()
            torch.testing.assert_close(outs["mean"][..., -1], mx[..., -1], rtol=1e-5, atol=0)


def test_config4_full_size():
    q, k = _inputs.config4()
    _full_size(q, k, ["sum"], [0, 10, 21, 31], "config4")


def test_config5_full_size():
    q, k = _inputs.config5()
    _full_size(q, k, ["mean", "max"], [0, 9, 17, 31], "config5")


def test_headline_shape_fp16():
    q, k = _inputs.headline()
    _full_size(q, k, ["sum"], [0, 5, 18, 31], "headline")


# --- beyond the reference's grid ----------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [
    (1, 1, 8), (1, 77, 16), (77, 1, 24), (2, 300, 128), (300, 2, 128), (257, 255, 128),
    (64, 64, 128), (513, 513, 96), (1000, 40, 40), (40, 1000, 20), (333, 777, 104), (700, 300, 56),
])
def test_ragged_shapes(m, n, d, causal, dtype):
    """M > N (offset clamps to 0), single rows/columns, D that needs zero padding, both dtypes."""
    q, k = _inputs.randn_pair(2, 3, m, n, d, seed=m * 7 + n, dtype=dtype)
    run_all(q, k, causal, what=f"m{m} n{n} d{d} {dtype}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [(300, 420, 136), (257, 129, 192), (130, 1000, 256), (64, 64, 200),
                                   (1, 700, 250), (520, 520, 144)])
def test_head_dims_above_128(m, n, d, causal, dtype):
    """D in (128, 256]: one resident 32-row block per wave, 128-row tiles."""
    q, k = _inputs.randn_pair(1, 3, m, n, d, seed=d + m, dtype=dtype)
    run_all(q, k, causal, what=f"m{m} n{n} d{d} {dtype}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [(300, 420, 264), (257, 129, 320), (130, 1000, 512), (64, 64, 400),
                                   (1, 700, 500), (520, 520, 384), (40, 3000, 512), (200, 200, 257), (90, 300, 449)])
def test_head_dims_above_256(m, n, d, causal, dtype):
    """D in (256, 512] for 16-bit elements: rows of up to 1 KiB, 9 to 16 k-steps, one workgroup per CU
    (the reference pads such a D to 512 and runs it when it fits, flash.py:368-373); every k-step count,
    D that is no multiple of 8 (padded by the host), few queries against many keys (split row sweep)."""
    q, k = _inputs.randn_pair(1, 3, m, n, d, seed=d + m, dtype=dtype)
    run_all(q, k, causal, what=f"m{m} n{n} d{d} {dtype}")


def test_every_k_step_count_of_long_16_bit_rows():
    for d in range(264, 513, 32):     # 264, 296, ..: 9 to 16 k-steps of 32 elements
        q, k = _inputs.randn_pair(2, 2, 150, 333, d, seed=d)
        run_all(q.half(), k.half(), True, what=f"d{d}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,m,n,d", [(1, 4, 40, 5000, 64), (1, 32, 128, 4096, 128), (1, 1, 300, 3001, 128),
                                       (2, 3, 1, 2048, 32), (1, 2, 257, 1100, 72)])
def test_few_queries_many_keys(b, h, m, n, d, causal):
    """Shapes where the row kernel splits the keys of a tile over several workgroups and a second
    small kernel merges the partial log-sum-exps."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=n + m)
    qd, kd = q.cuda(), k.cuda()
    got = fca.row_lse2(qd, kd, is_causal=causal).double().cpu()
    torch.testing.assert_close(got, row_lse2_ref(q, k, causal), rtol=0, atol=3e-4)
    run_all(q, k, causal, what=f"split b{b} h{h} m{m} n{n} d{d}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,m,n,d", [
    (103, 10, 32, 40, 8),      # one tile per (b,h): 1030 pairs, more than one launch group either way
    (5, 68, 700, 520, 16),     # three row tiles, 340 pairs: last group is partial
    (5, 8, 64, 4096, 32),      # split keys, 40 pairs in groups of 16 without the mask
    (3, 23, 520, 300, 8),      # 69 pairs, not a multiple of 8
])
def test_many_heads_in_launch_groups(b, h, m, n, d, causal):
    """(b,h) pairs are launched in groups; cover more pairs than one group holds, partial last groups
    and pair counts that are not multiples of 8, for both kernels and the split-key row sweep."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=b * h + m)
    run_all(q, k, causal, what=f"groups b{b} h{h} m{m} n{n} d{d}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [
    (1, 1, 8), (1, 4100, 128), (16, 64, 64), (17, 65, 72), (63, 200, 128), (64, 1100, 128), (64, 10, 32),
    (33, 4097, 96), (64, 6000, 128), (8, 2048, 16), (64, 129, 136),
])
def test_at_most_64_queries(m, n, d, causal, dtype):
    """Few query rows against few or many keys: the row sweep keeps one 32-row block per wave and the
    waves without any query only help staging; the causal diagonal is the last M keys.  Also the fused
    sum+max form."""
    q, k = _inputs.randn_pair(2, 5, m, n, d, seed=m + 3 * n + d, dtype=dtype)
    run_all(q, k, causal, what=f"small m{m} n{n} d{d} {dtype}")
    got = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ("sum", "max"), is_causal=causal, out_dtype=torch.float32)
    check(got[0], colreduce_ref(q, k, "sum", causal), "sum", f"small fused m{m} n{n} d{d}")
    check(got[1], colreduce_ref(q, k, "max", causal), "max", f"small fused m{m} n{n} d{d}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,m,n,d", [
    (4, 16, 64, 4100, 128),    # 64 pairs x 4 key ranges
    (2, 130, 33, 1030, 64),    # one range per pair, a ragged last chunk, padded query groups
    (4, 40, 1, 2048, 16),      # a single query
    (6, 50, 64, 1100, 72),     # D not a multiple of 32
    (1, 8, 17, 40000, 32),     # many ranges per pair
    (4, 16, 128, 4100, 128),   # eight resident query groups
    (4, 70, 97, 1030, 48),     # eight groups, the last two partly / wholly padding
])
def test_few_queries_with_streamed_keys(b, h, m, n, d, causal, dtype):
    """At most 128 queries, D <= 128 and enough (b,h) pairs x keys to fill the chip: the column
    sweep with the queries resident in every wave and the keys streamed in ranges; sum, mean, max and
    the fused sum+max form.  With the mask the diagonal is the last M keys."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=b * h + m + n, dtype=dtype)
    run_all(q, k, causal, what=f"streamed keys b{b} h{h} m{m} n{n} d{d} {dtype}")
    got = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ("sum", "max"), is_causal=causal, out_dtype=torch.float32)
    check(got[0], colreduce_ref(q, k, "sum", causal), "sum", "streamed keys fused")
    check(got[1], colreduce_ref(q, k, "max", causal), "max", "streamed keys fused")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,m,n,d", [
    (1, 32, 2048, 2048, 128),   # 256 workgroups of 256 rows either way: both sweeps take 128-row tiles
    (4, 16, 300, 1100, 64),     # only the column sweep is in that range
    (2, 8, 8192, 520, 32),      # only the row sweep is; M > N
    (1, 16, 8192, 8192, 16),    # exactly two per CU: finer tiles with the mask only
    (1, 32, 512, 2880, 128),    # 384 column workgroups of 256 keys: finer tiles without the mask too
])
def test_between_one_and_two_workgroups_per_cu(b, h, m, n, d, causal):
    """Launches that would put between one and two 256-row workgroups on a CU use 128-row tiles (at
    exactly one or two per CU depending on the sweep and the mask)."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=m + n + d)
    run_all(q, k, causal, what=f"finer tiles b{b} h{h} m{m} n{n} d{d}", reductions=("sum", "max"))


@pytest.mark.parametrize("b,h,m,n,d", [(1, 33, 1100, 1100, 64), (2, 16, 2048, 2048, 32), (3, 11, 1900, 2100, 136),
                                       (1, 40, 1537, 1500, 128), (1, 7, 9000, 9000, 16)])
def test_causal_launches_that_are_on_the_chip_at_once(b, h, m, n, d):
    """One to two workgroups per CU with the mask: the second half of the tiles is dealt in reverse.  Every tile
    of every head is still taken once (heads that do and do not divide the CU count)."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=m + d)
    run_all(q, k, True, what=f"{b}x{h} {m}x{n}x{d}", reductions=["sum", "max"])


@pytest.mark.parametrize("b,h,m,n,d", [(1, 71, 1900, 1850, 16), (1, 67, 1100, 1100, 32), (5, 7, 1100, 1090, 256), (1, 33, 2048, 2050, 136)])
def test_causal_launches_of_two_to_four_workgroups_per_cu(b, h, m, n, d):
    """The second workgroup of every CU dealt backwards and a third helping behind it: 256-row and 128-row tiles, heads that do
    not divide the eight dies, numbers of workgroups that are no multiple of eight."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=m + d)
    run_all(q, k, True, what=f"{b}x{h} {m}x{n}x{d}", reductions=["sum", "max"])


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,m,n,d", [(1, 2, 256, 256, 64), (1, 1, 2, 65, 4), (2, 3, 65, 63, 72), (1, 4, 191, 961, 128),
                                       (1, 8, 960, 960, 132), (1, 128, 64, 128, 16), (1, 129, 64, 128, 32),
                                       (1, 8, 1000, 2048, 256)])
def test_fp32_tiles_of_64_rows(b, h, m, n, d, causal):
    """fp32 launches that leave CUs idle take 64-row tiles: remainders of a tile, of a wave's 16 rows and of a chunk,
    M > N, both sides of the split row sweep, the most and one more than the most workgroups of the rule."""
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=m + n, dtype=torch.float32)
    run_all(q, k, causal, what=f"fp32 {b}x{h} {m}x{n}x{d}")
    s, mx = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ["sum", "max"], is_causal=causal)
    check(s.cpu(), colreduce_ref(q, k, "sum", causal), "sum", "fp32 pair")
    check(mx.cpu(), colreduce_ref(q, k, "max", causal), "max", "fp32 pair")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(2, 256, 256, 64), (3, 65, 63, 72), (4, 191, 960, 128), (1, 700, 333, 256)])
def test_fp32_tiles_of_64_rows_give_the_bits_of_taller_ones(h, m, n, d, causal):
    """The same heads alone (64-row tiles) and among as many copies as fill the chip (128 rows or more): each row and each
    column is added up in the same order whatever the tile."""
    q, k = (x.cuda() for x in _inputs.randn_pair(1, h, m, n, d, seed=m + n, dtype=torch.float32))
    copies = 512 // h
    qs, ks = q.repeat(copies, 1, 1, 1), k.repeat(copies, 1, 1, 1)
    assert torch.equal(fca.row_lse2(q, k, causal)[0], fca.row_lse2(qs, ks, causal)[-1])
    for red in REDUCTIONS:
        assert torch.equal(fca.flash_colreduce(q, k, red, causal)[0], fca.flash_colreduce(qs, ks, red, causal)[-1]), red


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(129, 300, 1000, 32), (12, 547, 2661, 64), (33, 200, 2000, 64), (130, 150, 1024, 64), (176, 140, 1024, 64),
                                     (12, 200, 2661, 128), (13, 200, 2661, 128)])
def test_sums_and_maxima_tile_heights(h, m, n, d, causal):
    """Both sides of the rule that gives the column tiles of sums and maxima together one or two key blocks per wave: one k-step,
    two with at most one, about two and a half and 2.75 workgroups of 256 keys per CU, 128-key tiles that just fit the CUs."""
    q, k = _inputs.randn_pair(1, h, m, n, d, seed=n + d)
    s, mx = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ["sum", "max"], is_causal=causal, out_dtype=torch.float32)
    check(s, colreduce_ref(q, k, "sum", causal), "sum", "pair")
    check(mx, colreduce_ref(q, k, "max", causal), "max", "pair")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,h,m,n,d", [(torch.float16, 2, 70, 99, 16), (torch.bfloat16, 2, 200, 333, 64), (torch.float16, 4, 300, 2100, 256),
                                           (torch.bfloat16, 1, 65, 130, 512), (torch.float16, 32, 70, 4096, 64), (torch.bfloat16, 64, 1, 8192, 128),
                                           (torch.float16, 32, 33, 2048, 128), (torch.float16, 2, 128, 64, 32)])
def test_key_that_no_query_counts_beside_rows_of_padding(dtype, h, m, n, d, causal):
    """Keys whose scores are -inf against every query: their columns are 0 in sums and maxima, with query counts that fill no
    tile too, in the column kernels of the two-kernel path."""
    q, k = (x.to(dtype) for x in _inputs.randn_pair(1, h, m, n, d, seed=m + n, dtype=torch.float32))
    q, k = q.clone(), k.clone()
    q[..., 3] = -q[..., 3].abs() - 0.1
    dead = [0, n // 2, n - 1] if not causal else [n // 2]   # (queries that see an infinite key only have no softmax)
    k[:, :, dead, 3] = float("inf")
    keep = torch.tensor([j for j in range(n) if j not in dead])
    c = max(n - m, 0)
    vis = (torch.arange(m)[:, None] + c >= torch.arange(n)[None]) if causal else torch.ones(m, n, dtype=torch.bool)
    s = torch.matmul(q[0].double(), k[0][:, keep].double().transpose(1, 2).contiguous()) * d ** -0.5
    p = torch.softmax(s.masked_fill(~vis[:, keep], -math.inf), -1)
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    try:
        for single in (0, 1):
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, single)
            for red, w in (("sum", p.sum(1)), ("max", p.amax(1))):
                got = fca.flash_colreduce(q.cuda(), k.cuda(), red, is_causal=causal, out_dtype=torch.float32).cpu()
                assert (got[0][:, dead] == 0).all(), (red, single)
                torch.testing.assert_close(got[0][:, keep], w.float(), rtol=2e-5, atol=1e-7)
    finally:
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(2, 65, 63, 4), (3, 129, 1100, 12), (8, 960, 960, 16), (8, 961, 961, 20), (140, 130, 257, 28),
                                     (300, 255, 70, 8), (2, 1000, 5000, 16), (40, 2000, 300, 28)])
def test_fp32_rows_shorter_than_32(h, m, n, d, causal):
    """D < 32 on the fp32 instructions: tiles of 64, 128 and 256 rows with ragged ends, the split row sweep, one and two k-steps.
    At most 28 products round a score by 2^-19 of their sum of magnitudes, a few tens: 1e-5 as for the other fp32 tests."""
    q, k = _inputs.randn_pair(1, h, m, n, d, seed=h + d, dtype=torch.float32)
    s, mx = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ["sum", "max"], is_causal=causal)
    for red, pair in (("sum", s), ("mean", None), ("max", mx)):
        want = colreduce_ref(q, k, red, causal, compute_dtype=torch.float64).float()
        for got in (fca.flash_colreduce(q.cuda(), k.cuda(), red, is_causal=causal), pair):
            if got is not None:
                torch.testing.assert_close(got.cpu(), want, rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(130, 257, 300, 36), (180, 300, 257, 96), (130, 257, 300, 256), (9, 511, 700, 128),
                                     (1, 65, 33, 32), (3, 129, 1100, 28)])
def test_fp32_split_tiles(h, m, n, d, causal):
    """fp32 rows as two fp16 parts: tiles of 256, 128 and 64 rows with ragged ends, more than one and more than two 128-row tiles
    per CU (which the mask treats differently), D that ends inside eight values, both sides of D = 32.  Probabilities carry
    the error of the scores (N(0,1) operands: 2^-21 of a sum of |q_d k_d| / sqrt(D) of ten or less, hardly ever all of it one
    way), and a sum that of its additions: 1e-5 as for the other fp32 tests."""
    q, k = _inputs.randn_pair(1, h, m, n, d, seed=h + d, dtype=torch.float32)
    s, mx = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ["sum", "max"], is_causal=causal)
    for red, pair in (("sum", s), ("mean", None), ("max", mx)):
        want = colreduce_ref(q, k, red, causal, compute_dtype=torch.float64).float()
        for got in (fca.flash_colreduce(q.cuda(), k.cuda(), red, is_causal=causal), pair):
            if got is not None:
                torch.testing.assert_close(got.cpu(), want, rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("d", [24, 32, 128, 256])
def test_fp32_split_rows_of_any_magnitude(d):
    """Every row is scaled by its own power of two (test_fp32_operands_near_the_ends_of_the_range has the ends), and the spread
    inside a row does not matter.  A score is off by at most 2^-21 of |q||k| per product (2^-23 for each operand, 2^-22 for the
    product of the lower parts) and by the roundings of its sum, at most 2^-24 of the running sum in each of up to 24 matrix
    instructions; signs vary, so running sums stay below a third of the sum of |q_d k_d|, which makes it 2^-21 too.  A log-sum-exp
    is off by at most 2^-20 of the row's largest sum of |q_d k_d|, and by two units in the last place of a value between 8 and 16 (log2 of 300 keys), 2^-19, for its own rounding: a logarithm and
    the additions that merge four partial results."""
    m, n = 260, 300
    g = torch.Generator().manual_seed(d)
    q = torch.randn(1, 2, m, d, generator=g) * torch.exp(3 * torch.randn(1, 2, m, d, generator=g)) * 2.0 ** -10
    k = torch.randn(1, 2, n, d, generator=g) * torch.exp(3 * torch.randn(1, 2, n, d, generator=g)) * 2.0 ** -10
    k[0, 0] *= (2.0 ** (torch.arange(n) % 40 - 20).float())[:, None]
    q[0, 1] *= (2.0 ** (torch.arange(m) % 40 - 20).float())[:, None]
    k[0, 1, 5] = 0.0
    k[0, 1, 6] *= 2.0 ** -130
    for up, down in ((1.0, 1.0), (2.0 ** 70, 2.0 ** -70), (2.0 ** -80, 2.0 ** 80)):
        qq, kk = q * up, k * down
        got = fca.row_lse2(qq.cuda(), kk.cuda(), scale=0.1).cpu().double()
        size = torch.matmul(qq.double().abs(), kk.double().abs().transpose(2, 3)) * (0.1 * 1.4427)
        err = (got - row_lse2_ref(qq, kk, False, scale=0.1).double()).abs()
        assert (err <= 2.0 ** -20 * size.amax(-1) + 2.0 ** -19).all(), (up, (err / (size.amax(-1) + 2)).max())


@pytest.mark.parametrize("exponent", [-125, -120, -115, -110, -100, 88, 100, 103, 104, 106, 108, 110, 112, 115, 120, 124])
@pytest.mark.parametrize("m,n,d", [(70, 300, 128), (300, 1100, 64), (260, 130, 256), (130, 70, 24)])
def test_fp32_operands_near_the_ends_of_the_range(m, n, d, exponent):
    """Finite keys and queries whose magnitudes make up for each other: the results are those of the same operands at
    magnitude one.  A power of two changes no bit of a product; a denormal element (2^-125 N(0,1) holds some) is held to
    2^-149, which is 2^-23 of it or more, so there the bound is the one of scores that are off by 2^-22 each."""
    q, k = _inputs.randn_pair(1, 2, m, n, d, seed=m + d, dtype=torch.float32)
    if exponent < 0:
        k = (k * 2.0 ** exponent) * 2.0 ** -exponent   # the bits a denormal loses
    else:
        q = (q * 2.0 ** -exponent) * 2.0 ** exponent
    big, small = k * 2.0 ** exponent, q * 2.0 ** -exponent
    assert torch.isfinite(big).all() and torch.isfinite(small).all()
    for red in REDUCTIONS:
        got = fca.flash_colreduce(small.cuda(), big.cuda(), red)
        assert torch.isfinite(got).all(), red
        torch.testing.assert_close(got.cpu(), colreduce_ref(q, k, red, False, compute_dtype=torch.float64).float(), rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("d", [16, 32, 128, 256])
def test_fp32_scores_of_one_product(d):
    """One non-zero product per score: 2^-21 of it at most (2^-23 for each operand, 2^-22 for the product of the lower parts; D < 32:
    one rounding), and 2^-23 for the scale and the sum; random mantissas and those that lose the most."""
    g = torch.Generator().manual_seed(d)
    bh, m = 96, 70
    q, k = torch.zeros(1, bh, m, d), torch.zeros(1, bh, 1, d)
    at = torch.randint(0, d, (bh,), generator=g)
    q[0, torch.arange(bh), :, at] = torch.randn(bh, m, generator=g)
    k[0, torch.arange(bh), 0, at] = torch.randn(bh, generator=g)
    for i, (x, y) in enumerate(((1 + 2.0 ** -11, 1 + 2.0 ** -11), (1 + 2.0 ** -11 - 2.0 ** -13,) * 2, (2 - 2.0 ** -23,) * 2,
                                (1 + 2.0 ** -11 - 2.0 ** -23, 1 + 2.0 ** -11 + 2.0 ** -23))):
        q[0, i, :, at[i]], k[0, i, 0, at[i]] = x, -y
    want = (q.double() * k.double()).sum(-1) * 1.4426950408889634
    err = (fca.row_lse2(q.cuda(), k.cuda(), scale=1.0).cpu().double() - want).abs()
    assert (err <= (2.0 ** -21 + 2.0 ** -23) * want.abs()).all(), (err / want.abs()).max()


@pytest.mark.parametrize("d", [16, 64, 256])
def test_fp32_large_scores_of_two_products(d):
    """Scores of 60 from two products each.  An exponent of 2 is off by 2^-21 of its size (as above) and 2^-23 for the roundings of
    sum, scale and log-sum-exp, a probability by ln 2 times twice that (its own score and the row's sum)."""
    g = torch.Generator().manual_seed(d)
    q, k = torch.zeros(1, 4, 300, d), torch.zeros(1, 4, 500, d)
    for at in (5, 9):
        q[..., at] = 7 + torch.randn(1, 4, 300, generator=g).abs()
        k[..., at] = 4 + 0.1 * torch.randn(1, 4, 500, generator=g)
    size = (torch.matmul(q.double(), k.double().transpose(2, 3)) * 1.4427).max().item()
    rtol = 0.6932 * 2 * (2.0 ** -21 + 2.0 ** -23) * size
    for red in ("sum", "max"):
        want = colreduce_ref(q, k, red, False, scale=1.0, compute_dtype=torch.float64).float()
        torch.testing.assert_close(fca.flash_colreduce(q.cuda(), k.cuda(), red, scale=1.0).cpu(), want, rtol=rtol, atol=1e-8)


@pytest.mark.parametrize("side", ["query", "key"])
@pytest.mark.parametrize("exponent", [6, 10, 14, 18, 22, 26, 30, 60, 90])
@pytest.mark.parametrize("h,m,n,d", [(2, 260, 300, 128), (1, 70, 1100, 64), (140, 257, 130, 256), (2, 300, 70, 36)])
def test_fp32_channel_that_only_one_side_uses(h, m, n, d, exponent, side):
    """A channel of 2^exponent in the rows of one operand (in every third row, so that tiles and chunks hold both kinds),
    zero in the other's: it takes part in no score, and the others keep their precision.  A score in the exponent of 2
    is off by 2^-21 of its sum of |q_d k_d|, by the rounding of that sum (under 2^-21 of it for the up to 16 terms of size that it
    has) and by 2^-20 (four times the 2^-22 that the parts of small elements may lose); log2 of up to 1100 rounds to 2^-20 at most."""
    q, k = _inputs.randn_pair(1, h, m, n, d, seed=m + d, dtype=torch.float32)
    q, k = q.clone(), k.clone()
    (q if side == "query" else k)[:, :, ::3, 5] = 2.0 ** exponent
    (k if side == "query" else q)[..., 5] = 0.0
    size = torch.matmul(q.double().abs(), k.double().abs().transpose(2, 3)).amax(-1) * (d ** -0.5 * 1.4427)
    err = (fca.row_lse2(q.cuda(), k.cuda()).cpu().double() - row_lse2_ref(q, k, False).double()).abs()
    assert (err <= 2.0 ** -20 * size + 2.0 ** -20 + 2.0 ** -20).all(), err.max()
    for red in ("sum", "max"):
        want = colreduce_ref(q, k, red, False, compute_dtype=torch.float64).float()
        torch.testing.assert_close(fca.flash_colreduce(q.cuda(), k.cuda(), red).cpu(), want, rtol=1e-5, atol=1e-8)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(2, 200, 333, 64), (5, 130, 129, 128), (2, 300, 2100, 256), (140, 257, 130, 40), (2, 70, 99, 28)])
def test_fp32_rows_without_a_scale(h, m, n, d, causal):
    """Infinities: a key whose scores are -inf against every query counts for nothing, alone in its chunk, and with an
    infinite query as well; the rest of its chunk and of its tile is as if it were not there.  A NaN query leaves NaN on the
    columns it sees and nowhere else."""
    q, k = _inputs.randn_pair(1, h, m, n, d, seed=m, dtype=torch.float32)
    q, k = q.clone(), k.clone()
    q[..., 3] = -q[..., 3].abs() - 0.1
    dead = [0, n // 2, n - 1] if not causal else [n // 2]
    k[:, 0, dead, 3] = float("inf")
    keep = torch.tensor([j for j in range(n) if j not in dead])
    c = max(n - m, 0)
    vis = (torch.arange(m)[:, None] + c >= torch.arange(n)[None]) if causal else torch.ones(m, n, dtype=torch.bool)
    s = (torch.matmul(q[0, 0].double(), k[0, 0, keep].double().T) * d ** -0.5).masked_fill(~vis[:, keep], -math.inf)
    want = torch.softmax(s, -1)
    for red in ("sum", "max"):
        got = fca.flash_colreduce(q.cuda(), k.cuda(), red, is_causal=causal).cpu()
        assert (got[0, 0, dead] == 0).all()
        w = want.sum(0) if red == "sum" else want.amax(0)
        torch.testing.assert_close(got[0, 0, keep], w.float(), rtol=1e-5, atol=1e-8)
        other = colreduce_ref(q[:, 1:], k[:, 1:], red, causal, compute_dtype=torch.float64).float()
        torch.testing.assert_close(got[:, 1:], other, rtol=1e-5, atol=1e-8)
    q[0, 1, m // 2, 1] = float("nan")
    got = fca.flash_colreduce(q.cuda(), k.cuda(), "sum", is_causal=causal).cpu()
    assert torch.equal(torch.isnan(got[0, 1]), vis[m // 2]) and not torch.isnan(got[0, 0]).any()


@pytest.mark.parametrize("m", [100, 128, 300, 384, 600])
def test_row_sweep_block_choice(m):
    """Query counts for which the row sweep keeps one 32-row block per wave (M <= 128 and ragged M
    such as 300, 384, 600) next to ones that keep two; the last tile has waves without any query."""
    q, k = _inputs.randn_pair(1, 6, m, 1500, 128, seed=m)
    for causal in (False, True):
        got = fca.row_lse2(q.cuda(), k.cuda(), is_causal=causal).double().cpu()
        torch.testing.assert_close(got, row_lse2_ref(q, k, causal), rtol=0, atol=3e-4)
        run_all(q, k, causal, what=f"row blocks m{m}", reductions=("sum",))


def test_key_operand_beyond_4_gib():
    """One head whose keys take more than 4 GiB: row offsets inside an operand exceed 32 bits and the
    buffer views are clamped; the last columns lie past that mark.  Relative check only (the sums are
    far below the absolute tolerance)."""
    n, d = (1 << 24) + 77, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    k = torch.randn(1, 1, n, d, device="cuda", dtype=torch.float16, generator=g)
    q = torch.randn(1, 1, 4, d, device="cuda", dtype=torch.float16, generator=g)
    qc, kc = q.cpu(), k.cpu()
    for causal in (False, True):
        got_s, got_m = fca.flash_colreduce_multi(q, k, ("sum", "max"), is_causal=causal, out_dtype=torch.float32)
        for got, red in ((got_s, "sum"), (got_m, "max")):
            want = colreduce_ref(qc, kc, red, causal, chunk_rows=16)
            torch.testing.assert_close(got.cpu(), want, rtol=2e-3, atol=0, msg=lambda m: f"{red} causal={causal}: {m}")


# --- the single sweep for few queries against many keys (keys read once) -------------------------------------
def _c_abi_colreduce(q, k, red, causal, scale=None):
    """fcr_colreduce through ctypes on device tensors; returns (out [B,H,N] fp32, lse [B,H,M] fp32, status)."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    b, h, m, d = q.shape
    n = k.shape[2]
    out = torch.empty(b * h, n, device="cuda")
    lse = torch.empty(lib.fcr_lse_bytes(b, h, m, n, d) // 4, device="cuda")
    dt = {torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}[q.dtype]
    _lib.check(lib.fcr_colreduce(q.data_ptr(), k.data_ptr(), out.data_ptr(), lse.data_ptr(), dt, b, h, m, n, d,
                                 _lib.strides4(q.stride()), _lib.strides4(k.stride()),
                                 float(scale if scale is not None else 1 / math.sqrt(d)),
                                 _lib.REDUCE_MAX if red == "max" else _lib.REDUCE_SUM, int(causal), None))
    status = lib.fcr_colreduce_status(lse.data_ptr(), dt, b, h, m, n, d, None)
    return out.view(b, h, n), lse[: b * h * m].view(b, h, m), status


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,m,n,d", [
    (1, 2, 64, 1024, 128),     # the smallest problem that takes the single sweep: one workgroup per pair
    (1, 3, 64, 16384, 128),    # teams of 16 workgroups
    (2, 3, 128, 4096, 128),    # two query halves, teams of 8
    (3, 5, 40, 3001, 64),      # ragged queries and keys, a partial last chunk
    (1, 2, 100, 5000, 72),     # two halves, the second ragged; D not a multiple of 32
    (2, 7, 17, 2100, 16),      # rows of 32 bytes
    (1, 1, 1, 70000, 128),     # one query, 69 workgroups on one pair
    (40, 16, 64, 2048, 32),    # 640 pairs for 128 teams: five rounds per workgroup
    (40, 16, 16, 8192, 64),    # at most 32 queries: two groups of queries per wave, 2048 keys per workgroup and pair
    (8, 32, 32, 8192, 128),    # the same with all 32 rows
    (64, 8, 7, 4100, 128),     # a ragged third workgroup
    (300, 4, 9, 1500, 32),     # a single workgroup per pair sweeping less than its share
    (3, 5, 20, 9000, 72),      # ragged everything
])
def test_single_sweep(b, h, m, n, d, causal, dtype):
    """At most 128 queries against at least 1024 keys: one sweep over the keys computes the row statistics
    and the columns (col_fused_kernel).  Sum, mean and max against the oracle through the operator; the
    row statistics and the status word through the C ABI; and the two-kernel path on the same inputs."""
    from flash_colreduce_amd import _lib
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=b + h + m + n, dtype=dtype)
    qd, kd = q.cuda(), k.cuda()
    what = f"single sweep b{b} h{h} m{m} n{n} d{d} {dtype}"
    run_all(q, k, causal, what=what)
    got, lse, status = _c_abi_colreduce(qd, kd, "sum", causal)
    assert status == 0
    torch.testing.assert_close(lse.double().cpu(), row_lse2_ref(q, k, causal), rtol=0, atol=3e-4)
    lib = _lib.load()
    lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 0)
    try:
        two, lse2, _ = _c_abi_colreduce(qd, kd, "sum", causal)
    finally:
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
    torch.testing.assert_close(got, two, rtol=2e-5, atol=1e-7)
    torch.testing.assert_close(lse, lse2, rtol=0, atol=2e-5)
    assert torch.equal(got, _c_abi_colreduce(qd, kd, "sum", causal)[0])   # no atomic adds: repeatable bit for bit
    # sums and maxima from the same single sweep (fcr_colreduce_sum_max)
    both_sum, both_max = fca.flash_colreduce_multi(qd, kd, ["sum", "max"], is_causal=causal, out_dtype=torch.float32)
    check(both_sum.cpu(), colreduce_ref(q, k, "sum", causal), "sum", what + " both")
    check(both_max.cpu(), colreduce_ref(q, k, "max", causal), "max", what + " both")
    torch.testing.assert_close(both_sum, got, rtol=2e-5, atol=1e-7)
    # (the team's partial values are merged by half as many waves, in another order: equal to rounding)
    torch.testing.assert_close(both_max.view(b, h, n), _c_abi_colreduce(qd, kd, "max", causal)[0], rtol=2e-5, atol=0)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,n,d,dtype", [
    (1, 1, 1, 8, torch.float16),          # one key, one granule per row
    (2, 3, 31, 16, torch.bfloat16),       # less than a step of a wave
    (1, 2, 257, 24, torch.float16),       # three granules on four lanes
    (3, 5, 1025, 72, torch.bfloat16),     # nine granules on sixteen lanes, one column past a workgroup's
    (2, 4, 4097, 128, torch.float16),     # more than one key range per pair
    (1, 3, 1000, 200, torch.bfloat16),    # 32 lanes per row
    (1, 2, 333, 512, torch.float16),      # 64 lanes per row
    (2, 2, 600, 4, torch.float32), (1, 3, 2049, 80, torch.float32), (1, 2, 777, 256, torch.float32),
    (1, 1, 70001, 64, torch.float16),     # more key ranges than lanes in the merge
])
def test_one_query(b, h, n, d, dtype, causal):
    """One query row (one_query_*_kernel): every lanes-per-row, ragged lengths, both layouts; the row statistics and
    the status word of its workspace; and the other path through the C ABI."""
    from flash_colreduce_amd import _lib
    from flash_colreduce_amd.flash import _DTYPES as DT
    q, k = _inputs.randn_pair(b, h, 1, n, d, seed=n + d, dtype=dtype)
    what = f"one query b{b} h{h} n{n} d{d} {dtype}"
    qd, kd = q.cuda(), k.cuda()
    kt = kd.transpose(1, 2).contiguous().transpose(1, 2)   # token-major memory seen as heads
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    nbytes = lib.fcr_workspace_bytes(DT[dtype], b, h, 1, n, d)
    assert nbytes >= lib.fcr_lse_bytes(b, h, 1, n, d) + 4 * b * h * n
    for red in REDUCTIONS:
        want = colreduce_ref(q, k, red, causal)
        got = fca.flash_colreduce(qd, kd, red, is_causal=causal, out_dtype=torch.float32)
        check(got.cpu(), want, red, what)
        assert torch.equal(got, fca.flash_colreduce(qd, kt, red, is_causal=causal, out_dtype=torch.float32))
        assert torch.equal(fca.flash_colreduce(qd, kd, red, is_causal=causal), got.to(dtype))   # (means divide by one)
        if red == "mean":
            continue
        ws = torch.full((nbytes // 4,), float("nan"), device="cuda")
        one, other = (torch.empty(b, h, n, device="cuda") for _ in range(2))
        code = _lib.REDUCE_MAX if red == "max" else _lib.REDUCE_SUM
        common = (DT[dtype], b, h, 1, n, d, _lib.strides4(qd.stride()), _lib.strides4(kd.stride()), d ** -0.5, code,
                  int(causal), stream)
        _lib.check(lib.fcr_colreduce_ws(qd.data_ptr(), kd.data_ptr(), one.data_ptr(), None, _lib.DTYPE_F32,
                                        ws.data_ptr(), nbytes, *common))
        assert torch.equal(one, got)
        torch.testing.assert_close(ws[: b * h].view(b, h, 1).double().cpu(), row_lse2_ref(q, k, causal), rtol=0, atol=3e-4)
        assert lib.fcr_colreduce_status(ws.data_ptr(), DT[dtype], b, h, 1, n, d, stream) == 0
        _lib.check(lib.fcr_colreduce_ws(qd.data_ptr(), kd.data_ptr(), other.data_ptr(), None, _lib.DTYPE_F32,
                                        ws.data_ptr(), lib.fcr_lse_bytes(b, h, 1, n, d), *common))
        torch.testing.assert_close(other, one, rtol=2e-5, atol=1e-7)


def _one_query_ref(q, k):
    """softmax rows of one query per pair in float64, batch entry by batch entry on the device; and their base-2 statistics."""
    p, stat = [], []
    for b in range(q.shape[0]):
        s = (q[b].double() * k[b].double()).sum(-1) / math.sqrt(q.shape[3])
        p.append(torch.softmax(s, -1))
        stat.append(torch.logsumexp(s, -1, keepdim=True) / math.log(2))
    return torch.stack(p), torch.stack(stat)


@pytest.mark.parametrize("b,h,n,d,dtype", [
    (1, 1, 16384, 64, torch.float16),    # 64 key ranges: every wave of the second launch merges all of them
    (1, 2, 16385, 64, torch.float16),    # 65: the waves share them, the last one holds one key
    (1, 1, 65537, 64, torch.float16),    # 257: more than one per thread
    (1, 1100, 1025, 256, torch.float32),   # more steps than there is room for: ranges of two steps, the last one of one key
    (8, 150, 1000, 256, torch.float32),    # the same, the last range of two steps as well, its second one partial
    (32, 1024, 70, 512, torch.float16),    # one range of three steps, the last one partial (keys shared by the batch)
])
def test_one_query_ranges(b, h, n, d, dtype):
    """One query whose keys are cut into as many ranges as the merge treats differently, or into ranges of several steps
    of a workgroup: scores that grow along the keys, so that the running maximum changes in every step."""
    g = torch.Generator(device="cuda").manual_seed(n)
    q = torch.randn(b, h, 1, d, device="cuda", generator=g)
    k = torch.randn(1 if n == 70 else b, h, n, d, device="cuda", generator=g)
    k += q[:k.shape[0]] * torch.linspace(0, 8.0 / math.sqrt(d), n, device="cuda").view(1, 1, n, 1)
    q, k = q.to(dtype), k.to(dtype).expand(b, h, n, d)
    want, stat = _one_query_ref(q, k)
    s, m = fca.flash_colreduce_multi(q, k, ["sum", "max"], is_causal=True, out_dtype=torch.float32)
    for got in (s, m, fca.flash_colreduce(q, k, "sum", out_dtype=torch.float32)):
        # products of up to 150 in base 2, 2^-24 per addition, eight or sixteen lanes' partial sums: below 1e-4 of a probability
        torch.testing.assert_close(got.double(), want, rtol=1e-4, atol=1e-30)
    from flash_colreduce_amd import _lib
    from flash_colreduce_amd.flash import _DTYPES as DT
    lib = _lib.load()
    nbytes = lib.fcr_workspace_bytes(DT[dtype], b, h, 1, n, d)
    ws, out = torch.full((nbytes // 4,), float("nan"), device="cuda"), torch.empty(b, h, n, device="cuda")
    _lib.check(lib.fcr_colreduce_ws(q.data_ptr(), k.data_ptr(), out.data_ptr(), None, _lib.DTYPE_F32, ws.data_ptr(), nbytes,
                                    DT[dtype], b, h, 1, n, d, _lib.strides4(q.stride()), _lib.strides4(k.stride()), d ** -0.5,
                                    _lib.REDUCE_SUM, 1, torch.cuda.current_stream().cuda_stream))
    torch.testing.assert_close(ws[: b * h].view(b, h, 1).double(), stat, rtol=0, atol=1e-4)


@pytest.mark.parametrize("shared", ["batch", "heads", "both"])
@pytest.mark.parametrize("b,h,n,d,dtype", [
    (3, 5, 1025, 72, torch.bfloat16), (2, 2, 777, 256, torch.float32), (8, 1, 300, 64, torch.float16),
    (7, 8, 16500, 128, torch.bfloat16),   # more keys than the L2s hold, fewer batch entries than XCDs
    (8, 8, 16384, 128, torch.bfloat16),   # as many as the L2s hold
    (8, 8, 16385, 128, torch.bfloat16), (11, 3, 30011, 256, torch.float16), (9, 8, 9001, 128, torch.float32),   # more
])
def test_one_query_shared_keys(b, h, n, d, dtype, shared):
    """One query against keys that the batch, the heads or both share by a stride of zero: whatever the order of the
    workgroups and the way the keys are loaded, the bits of the same keys held once per pair."""
    g = torch.Generator(device="cuda").manual_seed(n + d)
    q = torch.randn(b, h, 1, d, device="cuda", generator=g, dtype=dtype)
    k = torch.randn(1 if shared != "heads" else b, 1 if shared != "batch" else h, n, d, device="cuda", generator=g, dtype=dtype)
    k = k.expand(b, h, n, d)
    whole = k.contiguous()
    for red in REDUCTIONS:
        got = fca.flash_colreduce(q, k, red, is_causal=True, out_dtype=torch.float32)
        assert torch.equal(got, fca.flash_colreduce(q, whole, red, is_causal=True, out_dtype=torch.float32)), red
    p = torch.softmax((q[-1].double() * whole[-1].double()).sum(-1) / math.sqrt(d), -1)
    check(fca.flash_colreduce(q, k, "sum", out_dtype=torch.float32)[-1], p.cpu(), "sum", f"shared by {shared}")


# one launch and two: the largest number of keys of either limit and one more, the most pairs and one more, every number of lanes per row
@pytest.mark.parametrize("b,h,n,d,dtype", [(1, 8, 1024, 128, torch.bfloat16), (1, 8, 1025, 128, torch.bfloat16), (1, 130, 4096, 128, torch.float16),
                                           (1, 130, 4097, 128, torch.float16), (4, 64, 500, 64, torch.float16), (1, 257, 500, 64, torch.float16),
                                           (1, 3, 8192, 8, torch.float16), (1, 3, 8193, 8, torch.float16), (2, 2, 33, 16, torch.bfloat16),
                                           (1, 5, 255, 256, torch.float32), (1, 5, 1, 72, torch.bfloat16), (2, 70, 700, 40, torch.float32),
                                           (1, 2, 513, 512, torch.float16),
                                           # rows that fill half of their lanes: few pairs, more, and a quarter of the chip's
                                           (1, 4, 512, 136, torch.float16), (1, 4, 513, 136, torch.float16), (1, 20, 768, 136, torch.bfloat16),
                                           (1, 20, 769, 136, torch.bfloat16), (1, 64, 963, 136, torch.float16), (1, 64, 964, 136, torch.float16)])
def test_one_query_in_one_launch(b, h, n, d, dtype):
    """Against 64 bits: a probability is good to the rounding of its score (2^4: 2^-20) and of the sum."""
    g = torch.Generator(device="cuda").manual_seed(n + d)
    q, k = (torch.randn(b, h, r, d, device="cuda", generator=g).to(dtype) for r in (1, n))
    want, _ = _columns_f64(q, k, False)
    for causal in (False, True):
        for red in REDUCTIONS:
            assert _rel(fca.flash_colreduce(q, k, red, causal, out_dtype=torch.float32), want) <= 1e-5
    s, m = fca.flash_colreduce_multi(q, k, ["sum", "max"], out_dtype=torch.float32)
    assert torch.equal(s, m)
    k[0, 1 % h, n // 2, 0] = float("nan")
    s = fca.flash_colreduce(q, k, "sum", out_dtype=torch.float32)
    assert s[0, 1 % h].isnan().all() and s.isnan().sum().item() == n


# The bound is the mean error of the two launches on such inputs (standard error over 60 calls 0.004e-7); adding up the sixteen waves of the
# one launch one after the other gave 1.411e-7 and 1.282e-7, scaling each once gives 1.312e-7 and 1.164e-7.
@pytest.mark.parametrize("dtype,bound", [(torch.float16, 1.330e-7), (torch.bfloat16, 1.186e-7)])
def test_one_query_in_one_launch_is_no_less_exact_than_two(dtype, bound):
    errors = []
    for seed in range(32):
        g = torch.Generator(device="cuda").manual_seed(1000 + seed)
        q = torch.randn((1, 256, 1, 128), generator=g, device="cuda").to(dtype)
        k = torch.randn((1, 256, 1000, 128), generator=g, device="cuda").to(dtype)
        want = ((k.double() * q.double()).sum(-1) * 128**-0.5).softmax(-1)
        got = fca.flash_colreduce(q, k, "sum", out_dtype=torch.float32).double()
        errors.append(((got - want).norm() / want.norm()).item())
    assert sum(errors) / len(errors) <= bound


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_row_lse2_of_one_query_keeps_no_score_array(dtype):
    """The row statistics are a view of the row sweep's buffer, which has no room for the scores that one query's
    column reduction keeps: 4 bytes per key would live as long as the (B, H, 1) result."""
    from flash_colreduce_amd import _lib
    b, h, n, d = 2, 3, 40000, 64
    q, k = _inputs.randn_pair(b, h, 1, n, d, seed=8, dtype=dtype)
    lse = fca.row_lse2(q.cuda(), k.cuda())
    torch.testing.assert_close(lse.double().cpu(), row_lse2_ref(q, k), rtol=0, atol=3e-4)
    assert lse.untyped_storage().nbytes() == _lib.load().fcr_lse_bytes(b, h, 1, n, d) < 4 * b * h * n


def test_one_query_under_graph_capture():
    """One query recorded into a HIP graph: every replay on new inputs, with eager calls between them, gives the eager bits."""
    b, h, n, d = 3, 5, 5003, 128
    q0, k0 = _inputs.randn_pair(b, h, 1, n, d, seed=40, dtype=torch.bfloat16)
    qs, ks = q0.cuda(), k0.cuda()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fca.flash_colreduce_multi(qs, ks, ["mean", "max"], True)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fca.flash_colreduce_multi(qs, ks, ["mean", "max"], True)
    for seed in (41, 42, 43):
        q1, k1 = _inputs.randn_pair(b, h, 1, n, d, seed=seed, dtype=torch.bfloat16)
        qs.copy_(q1)
        ks.copy_(k1)
        graph.replay()
        torch.cuda.synchronize()
        got = [x.clone() for x in out]
        eager = fca.flash_colreduce_multi(qs, ks, ["mean", "max"], True)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, eager)), seed
        # the result is rounded to bf16: half a unit of 2^-8
        torch.testing.assert_close(got[1].float().cpu(), colreduce_ref(q1, k1, "max", True).float(), rtol=2.0 ** -8, atol=1e-7)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_one_query_non_finite(dtype):
    """One query: a NaN or +inf score makes the sums of its row NaN and its maxima 0, -inf scores count nothing (a row
    of nothing else is a NaN row), scores far from zero keep their softmax."""
    h, n, d = 6, 3000, 64
    q, k = _inputs.randn_pair(1, h, 1, n, d, seed=12, dtype=torch.float32)
    q[..., 0] = 1.0
    k[0, 0, 2000, 5] = float("nan")
    k[0, 1, 7, 0] = float("inf")
    k[0, 2, 100:2900, 0] = -float("inf")
    k[0, 3, :, 0] = -float("inf")
    k[0, 4] *= 30.0
    q, k = q.to(dtype), k.to(dtype)
    s, m = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ["sum", "max"], is_causal=True, out_dtype=torch.float32)
    bad = [0, 1, 3]
    assert torch.isnan(s[0, bad]).all() and (m[0, bad] == 0).all()
    good = [2, 4, 5]
    p = torch.softmax((q.double() @ k.double().transpose(2, 3))[0, good, 0] / math.sqrt(d), -1)
    for got in (s, m):
        # scaled |q||k| sums of up to 150 at 2^-24 per term, added up eight at a time: below 1e-4 of a probability
        torch.testing.assert_close(got[0, good].double().cpu(), p, rtol=1e-4, atol=1e-30)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m", [64, 128])
def test_single_sweep_scores_far_from_zero(m, causal):
    """Row sums of 2^score that overflow or vanish in fp32 (an enormous aligned key late in the sweep, rows
    whose scores are all around -190, unscaled scores): the workgroup sweeps its keys a second time keeping
    the scores and reduces them maximum first."""
    b, h, n, d = 1, 3, 4096, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=9)
    q, k = q.float(), k.float()
    k[:, 0, 3000] = 40.0 * q[:, 0, 50]
    k[:, 0, 3001] = -40.0 * q[:, 0, 50]
    k[:, 1] = -3.0 * q[:, 1, :1] + 0.1 * k[:, 1]
    k[:, 1, 3500:] *= 0.0
    for scale in (None, 1.0):
        run_all(q.half(), k.half(), causal, scale=scale, what=f"single sweep, far scores, m{m} scale={scale}")


@pytest.mark.parametrize("causal", [False, True])
def test_single_sweep_nan_and_inf_inputs(causal):
    """As test_nan_and_inf_inputs, on a shape that takes the single sweep: NaN rows make the columns they
    see NaN and leave the others alone; the maxima are compared where no NaN row looks."""
    b, h, m, n, d = 1, 4, 100, 2600, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=56)
    q, k = q.clone(), k.clone()
    q[0, 0, 70, 5] = float("nan")
    q[0, 1, 20, 3] = float("inf")
    k[0, 2, 1000, 7] = float("-inf")
    c = max(n - m, 0)
    scores = torch.einsum("bhmd,bhnd->bhmn", q.float(), k.float())
    vis = (torch.arange(m)[:, None] + c >= torch.arange(n)[None, :]) if causal else torch.ones(m, n, dtype=torch.bool)
    bad = ((torch.isnan(scores) | (scores == float("inf"))) & vis).any(-1)
    assert bad[0, 0].sum() == 1 and bad[0, 1].sum() == 1 and bad[0, 2].sum() > 10 and not bad[0, 3].any()
    nan_cols = (bad[..., None] & vis).any(-2)
    q_clean = torch.where(bad[..., None], torch.zeros_like(q), q)
    k_clean = torch.nan_to_num(k, neginf=0.0)
    qd, kd = q.cuda(), k.cuda()
    for red in REDUCTIONS:
        got = fca.flash_colreduce(qd, kd, red, is_causal=causal, out_dtype=torch.float32).cpu()
        want = colreduce_ref(q_clean, k_clean, red, causal)
        if red != "max":
            assert torch.equal(torch.isnan(got), nan_cols), red
        ok = ~nan_cols
        ok[0, 2] = False
        if causal:
            assert ok[0, 0].any() and ok[0, 1].any()
        check(got[ok], want[ok], red, f"single sweep, columns no NaN row sees, causal={causal}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m", [3, 20, 40, 100])
def test_single_sweep_rows_of_padding_meet_a_non_finite_key(m, causal):
    """Fewer queries than a workgroup holds rows for: the rows of padding are rows of zeros, which the fast form
    of the sweep leaves in place.  A key with an infinite element turns their scores into NaN (0 * inf); the
    sweep notices and hides them the slow way.  Here every real query is positive where the key is -inf, so
    the key's scores are -inf, its column is exactly 0 and every other column is untouched."""
    b, h, n, d = 2, 3, 3000, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=91 + m)
    q, k = q.half().clone(), k.half().clone()
    q[..., 7] = q[..., 7].abs() + 0.5
    k[0, 1, 1234, 7] = float("-inf")
    k[1, 2, n - 1, 7] = float("-inf")
    for red in REDUCTIONS:
        got = fca.flash_colreduce(q.cuda(), k.cuda(), red, is_causal=causal, out_dtype=torch.float32).cpu()
        assert not torch.isnan(got).any(), red
        assert got[0, 1, 1234] == 0 and got[1, 2, n - 1] == 0
        check(got, colreduce_ref(q, k, red, causal), red, f"padding rows m{m} {red}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [(100, 1030, 64), (128, 1537, 128), (65, 1024 + 448, 32), (40, 1100, 128), (64, 2049, 64), (20, 2100, 128),
                                   (2, 4100, 96)])
def test_single_sweep_chunks_past_the_last_key(m, n, d, causal):
    """The last workgroup of a team holds whole chunks past the last key, from one to all but one of them: left out in the
    first sweep, and hidden in the second one (scores far from zero) and where maxima are asked for."""
    q, k = _inputs.randn_pair(2, 3, m, n, d, seed=n)
    run_all(q, k, causal, what=f"{m}x{n}x{d}")
    run_all(q * 40, k, causal, what=f"{m}x{n}x{d} far from zero")


@pytest.mark.parametrize("m,n", [(60, 3000), (7, 1030)])
def test_single_sweep_in_a_workspace_of_8_byte_alignment(m, n):
    """The calls without a size take a workspace at any multiple of 8 bytes: the slots are cleared there too, to their last word and no further."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    h, d = 5, 64
    q, k = (torch.randn(1, h, r, d, device="cuda").half() for r in (m, n))
    want, _ = _columns_f64(q, k, True)
    size = lib.fcr_lse_bytes(1, h, m, n, d) // 4
    for start in (2, 4):
        ws = torch.full((size + 8,), 1.0, device="cuda")
        lse = ws[start : start + size]
        assert lse.data_ptr() % 16 == 8 * (start % 4 == 2)
        out = torch.empty(1, h, n, device="cuda")
        _lib.check(lib.fcr_colreduce(q.data_ptr(), k.data_ptr(), out.data_ptr(), lse.data_ptr(), _lib.DTYPE_F16, 1, h, m, n, d,
                                     _lib.strides4(q.stride()), _lib.strides4(k.stride()), d ** -0.5, _lib.REDUCE_SUM, 1,
                                     torch.cuda.current_stream().cuda_stream))
        assert lib.fcr_colreduce_status(lse.data_ptr(), _lib.DTYPE_F16, 1, h, m, n, d, None) == 0
        assert _rel(out, want) <= 1e-5
        assert (ws[:start] == 1).all() and (ws[start + size :] == 1).all()


def test_single_sweep_bounded_wait():
    """The wait for the team is bounded from the host: with a limit of zero polls a workgroup whose partners
    have not all published gives up at once, stores NaN for its columns of that pair, sets the status word
    and goes on; every workgroup ends normally.  What is not NaN is right, the status says whether anything
    is, and the next call with the usual limit is clean."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    b, h, m, n, d = 4, 16, 64, 8192, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=5)
    qd, kd = q.cuda(), k.cuda()
    want = colreduce_ref(q, k, "sum", True)
    assert lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 0) == 0
    try:
        got, _, status = _c_abi_colreduce(qd, kd, "sum", True)
    finally:
        assert lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 1 << 20) == 0
    got = got.cpu()
    gave_up = torch.isnan(got)
    assert status == (_lib.E_WAIT if gave_up.any() else 0), (status, int(gave_up.sum()))
    if status:
        assert b"gave up waiting" in lib.fcr_last_error()
    torch.testing.assert_close(got[~gave_up], want[~gave_up], rtol=2e-3, atol=1e-5)
    got, _, status = _c_abi_colreduce(qd, kd, "sum", True)
    assert status == 0
    check(got, want, "sum", "after the limit is restored")
    assert lib.fcr_set_option(7, 1) == -3 and lib.fcr_set_option(_lib.OPT_WAIT_POLLS, -1) == -3


# pairs in several rounds: at most 32 queries in workgroups of four waves (two per CU) where they are faster on 256 CUs (`four`), else of eight;
# one workgroup per team (1024 keys), several and many, keys that fill no step, no batch and no chunk, both edges of the query groups
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d,dtype,four", [
    (300, 20, 1100, 64, torch.float16, False), (60, 32, 5001, 128, torch.bfloat16, True), (520, 2, 1024, 40, torch.float16, True),
    (20, 17, 20000, 96, torch.float16, True), (60, 33, 5001, 128, torch.float16, False), (150, 31, 2049, 128, torch.bfloat16, True),
    (128, 32, 8192, 128, torch.bfloat16, True), (128, 2, 4100, 96, torch.float16, True), (64, 16, 8191, 128, torch.float16, True),
    (150, 17, 2048, 32, torch.bfloat16, True), (10, 31, 33000, 64, torch.float16, True), (32, 9, 16384, 32, torch.bfloat16, False)])
def test_single_sweep_in_rounds(h, m, n, d, dtype, four, causal):
    """Against 64 bits (see test_few_keys for the bound), then scores far from zero, NaN rows and infinite keys against the two kernels."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:   # the slots of that form need room behind what every form needs
        code = {torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}[dtype]
        assert (lib.fcr_workspace_bytes(code, 2, h, m, n, d) > lib.fcr_lse_bytes(2, h, m, n, d)) == four
    g = torch.Generator(device="cuda").manual_seed(h + n)
    q, k = (torch.randn(2, h, r, d, device="cuda", generator=g).to(dtype) for r in (m, n))
    sums, most = _columns_f64(q, k, causal)
    assert _rel(fca.flash_colreduce(q, k, "sum", causal, out_dtype=torch.float32), sums) <= 1e-5
    s2, m2 = fca.flash_colreduce_multi(q, k, ["sum", "max"], causal, out_dtype=torch.float32)
    assert _rel(s2, sums) <= 1e-5 and _rel(m2, most) <= 1e-5
    q[0, 1] *= 30
    k[0, 2, n // 2] *= 60
    q[1, 3, m - 1, 0] = float("nan")
    k[1, 4, n // 3, 0] = float("inf")
    for red in ("sum", "max"):
        got = {}
        for option in (1, 0):
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
            try:
                got[option] = fca.flash_colreduce(q, k, red, causal, out_dtype=torch.float32)
            finally:
                lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
        assert torch.equal(got[1].isnan(), got[0].isnan()), red
        torch.testing.assert_close(got[1], got[0], rtol=2e-4, atol=1e-6, equal_nan=True)   # scores of 2^9: 2^-15 each


def test_single_sweep_in_rounds_bounded_wait():
    """As test_single_sweep_bounded_wait, in workgroups of four waves."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    q, k = (torch.randn(2, 60, r, 64, device="cuda").half() for r in (30, 8192))
    ws, out = torch.empty(_lib_workspace(q, k), device="cuda"), torch.empty(120, 8192, device="cuda")
    assert 4 * ws.numel() > lib.fcr_lse_bytes(2, 60, 30, 8192, 64)
    want, _ = _columns_f64(q, k, True)
    want = want.view(120, 8192)
    for polls in (0, 1 << 20):
        assert lib.fcr_set_option(_lib.OPT_WAIT_POLLS, polls) == 0
        try:
            _ws_call(q, k, out, ws, True)
            status = lib.fcr_colreduce_status(ws.data_ptr(), _lib.DTYPE_F16, 2, 60, 30, 8192, 64, torch.cuda.current_stream().cuda_stream)
        finally:
            assert lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 1 << 20) == 0
        gave_up = torch.isnan(out)
        assert status == (_lib.E_WAIT if gave_up.any() else 0) and not (polls and status)
        torch.testing.assert_close(out[~gave_up], want[~gave_up].float(), rtol=1e-4, atol=1e-6)


def test_single_sweeps_on_two_streams_are_chained():
    """A single sweep expects the whole chip (its workgroups wait for each other), so the library chains the
    single sweeps that a process issues on different streams with an event: calls issued alternately on two
    streams, with no host synchronisation between them, all give the results of the calls made alone."""
    qa, ka = _inputs.randn_pair(2, 8, 64, 8192, 128, seed=5, dtype=torch.float16)
    qb, kb = _inputs.randn_pair(1, 16, 128, 4096, 64, seed=6, dtype=torch.bfloat16)
    qa, ka, qb, kb = qa.cuda(), ka.cuda(), qb.cuda(), kb.cuda()
    want_a = fca.flash_colreduce(qa, ka, "sum", is_causal=True)
    want_b = fca.flash_colreduce(qb, kb, "max", is_causal=False)
    check(want_a.float().cpu(), colreduce_ref(qa.cpu(), ka.cpu(), "sum", True), "sum", "alone")
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    got = []
    for _ in range(25):
        with torch.cuda.stream(sa):
            got.append((want_a, fca.flash_colreduce(qa, ka, "sum", is_causal=True)))
        with torch.cuda.stream(sb):
            got.append((want_b, fca.flash_colreduce(qb, kb, "max", is_causal=False)))
    torch.cuda.synchronize()
    for want, out in got:
        assert torch.equal(out, want)


def test_single_sweep_under_graph_capture():
    """The single sweep (a small kernel that clears the slots, then the sweep) captured and replayed."""
    b, h, m, n, d = 2, 8, 64, 4096, 128
    qs = torch.zeros(b, h, m, d, device="cuda", dtype=torch.float16)
    ks = torch.zeros(b, h, n, d, device="cuda", dtype=torch.float16)
    q0, k0 = _inputs.randn_pair(b, h, m, n, d, seed=31)
    qs.copy_(q0)
    ks.copy_(k0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fca.flash_colreduce(qs, ks, "mean", True, out_dtype=torch.float32)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fca.flash_colreduce(qs, ks, "mean", True, out_dtype=torch.float32)
    for seed in (32, 33, 34):
        q1, k1 = _inputs.randn_pair(b, h, m, n, d, seed=seed)
        qs.copy_(q1)
        ks.copy_(k1)
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        eager = fca.flash_colreduce(qs, ks, "mean", True, out_dtype=torch.float32)
        torch.cuda.synchronize()
        assert torch.equal(got, eager), seed
        check(got, colreduce_ref(q1, k1, "mean", True), "mean", f"single sweep, graph replay seed {seed}")


@pytest.mark.parametrize("causal", [False, True])
def test_explicit_and_negative_scale(causal):
    q, k = _inputs.randn_pair(1, 4, 200, 333, 64, seed=21)
    for scale in (0.05, 1.0 / 3.0, -0.125, 0.0):
        run_all(q, k, causal, scale=scale, what=f"scale={scale}")


@pytest.mark.parametrize("causal", [False, True])
def test_strided_inputs(causal):
    """[B,M,H,D] storage viewed as [B,H,M,D], a slice with a storage offset, and a layout that
    forces a copy (d stride 2)."""
    g = torch.Generator().manual_seed(5)
    b, h, m, n, d = 2, 5, 150, 290, 64
    q_store = torch.randn(b, m, h, d, generator=g).half()
    k_store = torch.randn(b, n + 16, h, 2 * d, generator=g).half()
    q = q_store.permute(0, 2, 1, 3)
    k = k_store.permute(0, 2, 1, 3)[:, :, 8:8 + n, d:]
    assert not q.is_contiguous() and not k.is_contiguous()
    run_all(q, k, causal, what="permuted+sliced")
    k2 = torch.randn(b, h, n, 2 * d, generator=g).half()[..., ::2]
    assert k2.stride(3) == 2
    run_all(q, k2, causal, what="d-stride 2")
    # contiguous but starting 2 bytes off a 16-byte boundary
    flat = torch.randn(b * h * n * d + 1, generator=g).half().cuda()
    k3 = flat[1:].view(b, h, n, d)
    assert k3.is_contiguous() and k3.data_ptr() % 16 != 0
    got = fca.flash_colreduce(q.cuda(), k3, "sum", is_causal=causal, out_dtype=torch.float32)
    check(got, colreduce_ref(q, k3.cpu(), "sum", causal), "sum", "misaligned base")


@pytest.mark.parametrize("causal", [False, True])
def test_expanded_operands(causal):
    """Operands whose rows overlap in memory (expand() gives a row stride of 0): the library's buffer
    views cannot describe them, so the host copies; one query repeated M times, one key repeated N
    times, and a batch/head broadcast (stride 0 on those dimensions is addressed directly)."""
    b, h, m, n, d = 2, 3, 70, 200, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=61)
    qd, kd = q.cuda(), k.cuda()

    def run(qx, kx, what):  # expanded on the device: a host-to-device copy would make them dense
        assert qx.is_cuda and kx.is_cuda
        for red in REDUCTIONS:
            got = fca.flash_colreduce(qx, kx, red, is_causal=causal, out_dtype=torch.float32)
            check(got, colreduce_ref(qx.cpu(), kx.cpu(), red, causal), red, what)

    q1 = qd[:, :, :1].expand(b, h, m, d)
    assert q1.stride(2) == 0
    run(q1, kd, "expanded query rows")
    k1 = kd[:, :, 3:4].expand(b, h, n, d)
    run(qd, k1, "expanded key rows")
    kb = kd[:1, :1].expand(b, h, n, d)
    assert kb.stride(0) == 0 and kb.stride(1) == 0
    run(qd, kb, "key broadcast over batch and heads")
    # through the C ABI the overlapping rows are rejected, not misread
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    out = torch.empty(b * h, n, device="cuda")
    lse = torch.empty(lib.fcr_lse_bytes(b, h, m, n, d) // 4, device="cuda")
    rc = lib.fcr_colreduce(q1.data_ptr(), kd.data_ptr(), out.data_ptr(), lse.data_ptr(), _lib.DTYPE_F16, b, h, m, n, d,
                           _lib.strides4(q1.stride()), _lib.strides4(kd.stride()), 0.125, 0, int(causal), None)
    assert rc == -4 and b"row stride" in lib.fcr_last_error()


@pytest.mark.parametrize("causal", [False, True])
def test_single_row_with_any_row_stride(causal):
    """One query row or one key row whose row stride is smaller than D (a slice of an expanded tensor keeps
    stride 0; torch reports arbitrary strides for dimensions of size one): the stride of a single row is
    never used, through the operator and through the C ABI alike."""
    from flash_colreduce_amd import _lib
    b, h, d = 2, 3, 64
    q, k = _inputs.randn_pair(b, h, 40, 700, d, seed=77)
    qd, kd = q.cuda(), k.cuda()
    q1 = qd[:, :, 7:8].expand(b, h, 5, d)[:, :, :1]       # M = 1, row stride 0
    k1 = kd[:, :, 9:10].expand(b, h, 6, d)[:, :, :1]      # N = 1, row stride 0
    assert q1.stride(2) == 0 and k1.stride(2) == 0
    lib = _lib.load()
    for qx, kx in ((q1, kd), (qd, k1), (q1, k1)):
        m, n = qx.shape[2], kx.shape[2]
        for red in REDUCTIONS:
            got = fca.flash_colreduce(qx, kx, red, is_causal=causal, out_dtype=torch.float32)
            check(got, colreduce_ref(qx.cpu(), kx.cpu(), red, causal), red, f"m{m} n{n}")
        out = torch.empty(b * h, n, device="cuda")
        lse = torch.empty(lib.fcr_lse_bytes(b, h, m, n, d) // 4, device="cuda")
        _lib.check(lib.fcr_colreduce(qx.data_ptr(), kx.data_ptr(), out.data_ptr(), lse.data_ptr(), _lib.DTYPE_F16, b, h,
                                     m, n, d, _lib.strides4(qx.stride()), _lib.strides4(kx.stride()), 0.125, 0,
                                     int(causal), None))
        check(out.view(b, h, n), colreduce_ref(qx.cpu(), kx.cpu(), "sum", causal), "sum", f"C ABI m{m} n{n}")


@pytest.mark.parametrize("causal", [False, True])
def test_score_jumps_renormalise(causal):
    """Scores that jump by far more than 64 binades in the middle of the sweep, and rows whose
    scores are all hugely negative: exercises the renormalisation of the running row sum."""
    b, h, m, n, d = 1, 2, 96, 640, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=9)
    q = q.float()
    k = k.float()
    k[:, 0, 300] = 40.0 * q[:, 0, 50]          # one enormous aligned key, late
    k[:, 0, 301] = -40.0 * q[:, 0, 50]         # and an enormously negative one
    k[:, 1, :, :] = -3.0 * q[:, 1, :1, :] + 0.1 * k[:, 1]   # all scores of row 0 around -190
    k[:, 1, 500:] *= 0.0
    run_all(q.half(), k.half(), causal, what="jumps")
    run_all(q.half(), k.half(), causal, scale=1.0, what="jumps scale 1")


@pytest.mark.parametrize("causal", [False, True])
def test_nan_and_inf_inputs(causal):
    """Non-finite inputs.  A row of scores with a NaN or a +inf (inf - inf in the softmax) is a NaN row:
    every column it may see gets a NaN sum and mean, as in the materialising reference (naive.py:19-28).
    Columns hidden from every such row are untouched (the reference's materialised softmax makes the
    hidden entries of a NaN row NaN as well, naive.py:24-25; its kernel, like this one, never visits
    them, flash.py:198-207), as are rows and (b,h) pairs without one.  The column maximum follows IEEE
    maxNum (a NaN operand is dropped, like the Triton max at flash.py:123-124), so 'max' is compared on
    the columns no NaN row sees (test_max_leaves_nan_rows_out checks it on the others)."""
    b, h, m, n, d = 1, 4, 150, 260, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=55)
    q = q.clone()
    k = k.clone()
    q[0, 0, 70, 5] = float("nan")          # head 0: a NaN in query 70
    q[0, 1, 20, 3] = float("inf")          # head 1: an infinity in query 20 (scores +inf and -inf)
    k[0, 2, 100, 7] = float("-inf")        # head 2: an infinity in key 100: +inf scores for queries with q[7] < 0
    c = max(n - m, 0)
    scores = torch.einsum("bhmd,bhnd->bhmn", q.float(), k.float())
    vis = (torch.arange(m)[:, None] + c >= torch.arange(n)[None, :]) if causal else torch.ones(m, n, dtype=torch.bool)
    bad = ((torch.isnan(scores) | (scores == float("inf"))) & vis).any(-1)          # [b, h, m]: NaN rows
    assert bad[0, 0].sum() == 1 and bad[0, 1].sum() == 1 and bad[0, 2].sum() > 10 and not bad[0, 3].any()
    nan_cols = (bad[..., None] & vis).any(-2)                                          # [b, h, n]
    q_clean = torch.where(bad[..., None], torch.zeros_like(q), q)   # a zero row adds nothing to columns it cannot see
    k_clean = torch.nan_to_num(k, neginf=0.0)
    qd, kd = q.cuda(), k.cuda()
    for red in REDUCTIONS:
        got = fca.flash_colreduce(qd, kd, red, is_causal=causal, out_dtype=torch.float32).cpu()
        want = colreduce_ref(q_clean, k_clean, red, causal)
        if red != "max":
            assert torch.equal(torch.isnan(got), nan_cols), red
        ok = ~nan_cols
        ok[0, 2] = False     # head 2: the key with the infinity changes every row that sees it
        if causal:
            assert ok[0, 0].any() and ok[0, 1].any()
        check(got[ok], want[ok], red, f"columns no NaN row sees, causal={causal}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n", [(150, 260), (300, 3000), (64, 700), (100, 900), (64, 2048), (128, 4096)])
def test_max_leaves_nan_rows_out(m, n, causal):
    """The column maximum of a column that a NaN row sees is the maximum over the other rows that see it,
    and 0 when there is none: a NaN is dropped by the maximum (IEEE maxNum), as in the reference's kernel
    (tl.max and tl.atomic_max, flash.py:123-124,262-273), not propagated as by the materialising reference
    (naive.py:36-37).  Every column kernel (resident keys, streamed keys, single sweep, sum and max from
    one sweep), checked ON the columns the NaN rows see, against a float64 softmax written out here."""
    b, h, d = 1, 3, 64
    q, k = _inputs.randn_pair(b, h, m, n, d, seed=77 + m)
    q, k = q.half().clone(), k.half().clone()
    q[0, 0, m // 2, 5] = float("nan")       # head 0: one NaN row in the middle
    q[0, 1, m - 1, 0] = float("nan")        # head 1: the last row, the only one that sees the last column when causal
    q[0, 1, 3, 1] = float("inf")            #         and a row with +inf and -inf scores
    k[0, 2, n - 5, 7] = float("-inf")       # head 2: a key that gives +inf, -inf scores
    c = max(n - m, 0)
    vis = (torch.arange(m)[:, None] + c >= torch.arange(n)[None, :]) if causal else torch.ones(m, n, dtype=torch.bool)
    s = torch.einsum("bhmd,bhnd->bhmn", q.double(), k.double()) / math.sqrt(d)
    s = torch.where(vis, s, torch.full_like(s, float("-inf")))
    bad = (torch.isnan(s) | (s == float("inf"))).any(-1)                     # [b, h, m]
    p = torch.softmax(torch.where(bad[..., None], torch.zeros_like(s), s), dim=-1)
    p = torch.where(vis, p, torch.zeros_like(p))
    want_max = torch.where(bad[..., None], torch.zeros_like(p), p).amax(-2)
    nan_cols = (bad[..., None] & vis).any(-2)
    want_sum = torch.where(nan_cols, torch.full_like(want_max, float("nan")),
                           torch.where(bad[..., None], torch.zeros_like(p), p).sum(-2))
    assert bad[0, 0].sum() == 1 and bad[0, 1].sum() == 2 and bad[0, 2].sum() >= 1
    if causal:
        assert want_max[0, 1, -1] == 0    # no row left for the last column
    qd, kd = q.cuda(), k.cuda()
    got = fca.flash_colreduce(qd, kd, "max", is_causal=causal, out_dtype=torch.float32).cpu()
    assert not torch.isnan(got).any()
    torch.testing.assert_close(got.double(), want_max, rtol=2e-3, atol=1e-30)
    both_sum, both_max = fca.flash_colreduce_multi(qd, kd, ["sum", "max"], is_causal=causal, out_dtype=torch.float32)
    torch.testing.assert_close(both_max.cpu().double(), want_max, rtol=2e-3, atol=1e-30)
    torch.testing.assert_close(both_sum.cpu().double(), want_sum, rtol=2e-3, atol=1e-5, equal_nan=True)


def test_heavy_hitter_columns_small():
    q, k = _inputs.config4(heads=2, n=1024)
    run_all(q, k, True, what="config4-small")
    q, k = _inputs.config5(heads=2, n=1536)
    run_all(q, k, True, what="config5-small")


@pytest.mark.parametrize("causal", [False, True])
def test_row_lse2(causal):
    q, k = _inputs.randn_pair(2, 3, 300, 520, 80, seed=13)
    got = fca.row_lse2(q.cuda(), k.cuda(), is_causal=causal).double().cpu()
    want = row_lse2_ref(q, k, causal)
    assert got.shape == (2, 3, 300)
    torch.testing.assert_close(got, want, rtol=0, atol=2e-5 * 12)


def test_key_shift_invariance_bf16_inputs():
    """Adding one vector to every key of a head only shifts each row's scores (config 5's
    perturbation); exact in real arithmetic, so checked in fp16 where the shift is representable."""
    q, k = _inputs.randn_pair(1, 2, 256, 384, 64, seed=31)
    k = (k.float() * 4).round() / 4
    shift = torch.tensor([0.5, -0.25] * 32).view(1, 1, 1, 64)
    a = fca.flash_colreduce(q.cuda(), k.half().cuda(), "sum", True, out_dtype=torch.float32)
    b = fca.flash_colreduce(q.cuda(), (k + shift).half().cuda(), "sum", True, out_dtype=torch.float32)
    torch.testing.assert_close(a, b, rtol=2e-3, atol=1e-5)


def test_deterministic_and_stream_safe():
    """No atomics: results are bitwise repeatable, also on a side stream."""
    q, k = _inputs.randn_pair(2, 4, 700, 900, 128, seed=17)
    q, k = q.cuda(), k.cuda()
    ref = {r: fca.flash_colreduce(q, k, r, True, out_dtype=torch.float32) for r in REDUCTIONS}
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        again = {r: fca.flash_colreduce(q, k, r, True, out_dtype=torch.float32) for r in REDUCTIONS}
    s.synchronize()
    for r in REDUCTIONS:
        assert torch.equal(ref[r], again[r]), r


def test_output_dtype_and_mean_epilogue():
    q, k = _inputs.randn_pair(1, 2, 64, 200, 32, seed=3, dtype=torch.bfloat16)
    q, k = q.cuda(), k.cuda()
    out = fca.flash_colreduce(q, k, "mean", True)
    assert out.dtype == torch.bfloat16 and out.shape == (1, 2, 200)
    s = fca.flash_colreduce(q, k, "sum", True)
    div = torch.cat([torch.full((136,), 64.0), torch.arange(64, 0, -1).float()]).cuda()
    torch.testing.assert_close(out, (s / div.to(torch.bfloat16)), rtol=0, atol=0)


@pytest.mark.parametrize("res_dtype", [None, torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d,dtype", [(300, 5000, 64, torch.bfloat16),     # counts that bf16 and fp16 round
                                         (700, 300, 128, torch.float16),     # more queries than keys
                                         (40, 9000, 128, torch.float16),     # the few-queries column sweep
                                         (1, 77, 32, torch.bfloat16), (513, 513, 72, torch.float16)])
def test_cast_and_mean_in_the_kernel_repeat_the_torch_steps(m, n, d, dtype, causal, res_dtype):
    """The column kernel's typed store against the reference's own sequence of torch operations
    (flash.py:308 cast, 377-384 in-place divisions) applied to the fp32 result of the C ABI: bit for bit."""
    from flash_colreduce_amd import flash as F
    q, k = _inputs.randn_pair(2, 3, m, n, d, seed=m + n, dtype=dtype)
    q, k = q.cuda(), k.cuda()
    want_dtype = dtype if res_dtype is None else res_dtype
    for red in REDUCTIONS:
        got = fca.flash_colreduce(q, k, red, is_causal=causal, out_dtype=res_dtype)
        (acc,), _ = F._launch(q, k, ["max" if red == "max" else "sum"], causal, None)
        scores = acc.view(2, 3, n).to(want_dtype)
        if red == "mean":
            if causal:
                c = max(n - m, 0)
                scores[..., :c] /= m
                scores[..., c:] /= torch.arange(n - c, 0, -1, device=q.device)
            else:
                scores /= m
        assert got.dtype == want_dtype and got.shape == (2, 3, n)
        assert torch.equal(got, scores), (red, (got.float() - scores.float()).abs().max().item())


@pytest.mark.parametrize("causal", [False, True])
def test_multi_reduction_shares_the_row_pass(causal):
    q, k = _inputs.randn_pair(2, 3, 300, 450, 64, seed=8, dtype=torch.bfloat16)
    qd, kd = q.cuda(), k.cuda()
    outs = fca.flash_colreduce_multi(qd, kd, ["mean", "max", "sum", "mean"], is_causal=causal,
                                     out_dtype=torch.float32)
    assert len(outs) == 4
    for red, got in zip(["mean", "max", "sum", "mean"], outs):
        one = fca.flash_colreduce(qd, kd, red, is_causal=causal, out_dtype=torch.float32)
        if red == "max":
            assert torch.equal(got, one)  # a maximum does not depend on the tiling
        else:
            torch.testing.assert_close(got, one, rtol=1e-5, atol=1e-7)
        check(got, colreduce_ref(q, k, red, causal), red, "multi")
    only_sums = fca.flash_colreduce_multi(qd, kd, ["sum", "mean"], is_causal=causal, out_dtype=torch.float32)
    assert torch.equal(only_sums[0], fca.flash_colreduce(qd, kd, "sum", is_causal=causal, out_dtype=torch.float32))
    with pytest.raises(ValueError, match="Invalid reduction: median"):
        fca.flash_colreduce_multi(qd, kd, ["sum", "median"])
    with pytest.raises(ValueError, match="at least one"):
        fca.flash_colreduce_multi(qd, kd, [])


@pytest.mark.parametrize("res_dtype", [None, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d,dtype", [(300, 5000, 64, torch.bfloat16), (64, 4096, 128, torch.float16),
                                         (100, 2000, 32, torch.bfloat16), (700, 300, 128, torch.float16)])
def test_sum_or_mean_with_max_finished_in_the_kernel(m, n, d, dtype, causal, res_dtype):
    """'sum' or 'mean' together with 'max' is one call of fcr_colreduce_sum_max_to (two kernels, or the single
    sweep): both results leave it in the result type, the means divided as flash.py:377-384 does.  Held to
    the torch sequence on the same call's fp32 sums bit for bit, and to the one-reduction calls."""
    q, k = _inputs.randn_pair(2, 3, m, n, d, seed=m + n, dtype=dtype)
    qd, kd = q.cuda(), k.cuda()
    rt = dtype if res_dtype is None else res_dtype
    s32, x32 = fca.flash_colreduce_multi(qd, kd, ["sum", "max"], is_causal=causal, out_dtype=torch.float32)
    check(s32.cpu(), colreduce_ref(q, k, "sum", causal), "sum", "pair")
    check(x32.cpu(), colreduce_ref(q, k, "max", causal), "max", "pair")
    for red in ("sum", "mean"):
        got, mx = fca.flash_colreduce_multi(qd, kd, [red, "max"], is_causal=causal, out_dtype=res_dtype)
        assert got.dtype == rt and mx.dtype == rt and got.shape == (2, 3, n) and mx.shape == (2, 3, n)
        want = s32.to(rt)
        if red == "mean":
            c = max(n - m, 0) if causal else n
            want[..., :c] /= m
            if c < n:
                want[..., c:] /= torch.arange(n - c, 0, -1, device="cuda")
        assert torch.equal(got, want), red
        assert torch.equal(mx, x32.to(rt))
        one = fca.flash_colreduce(qd, kd, red, is_causal=causal, out_dtype=res_dtype)
        torch.testing.assert_close(got.float(), one.float(), rtol=2e-5 if rt == torch.float32 else 1e-2, atol=1e-7)
    twice = fca.flash_colreduce_multi(qd, kd, ["max", "mean", "max"], is_causal=causal)
    assert torch.equal(twice[0], twice[2]) and twice[0].data_ptr() != twice[2].data_ptr()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [(1, 1, 8), (131, 1027, 72), (700, 300, 128), (40, 1000, 24), (300, 420, 200),
                                   (1024, 1024, 128)])
def test_sum_and_max_from_one_sweep(m, n, d, causal, dtype):
    q, k = _inputs.randn_pair(2, 2, m, n, d, seed=m + n + d, dtype=dtype)
    s, mx, mean = fca.flash_colreduce_multi(q.cuda(), k.cuda(), ["sum", "max", "mean"], is_causal=causal,
                                            out_dtype=torch.float32)
    check(s, colreduce_ref(q, k, "sum", causal), "sum", "fused")
    check(mx, colreduce_ref(q, k, "max", causal), "max", "fused")
    check(mean, colreduce_ref(q, k, "mean", causal), "mean", "fused")


@pytest.mark.parametrize("n,k", [(1, 1), (5, 2), (256, 100), (257, 256), (1000, 0), (1000, 1000), (1000, 1500),
                                 (4099, 1024), (8192, 2048), (8200, 8199), (32768, 8192), (32769, 1), (40000, 5000),
                                 (70001, 0), (70001, 69000), (131072, 200)])
def test_topk_keep_mask(n, k):
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n + k)
    vals = torch.rand(6, n, generator=g)
    vals[1] = (vals[1] * 8).floor() / 8          # heavy ties
    vals[2] = 0.25                                # all equal
    vals[3] = -vals[3]                            # negatives
    vals[4, ::3] = 0.0
    vals[4, 1::3] = -0.0
    mask, thr = fca.topk_keep_mask(vals.cuda().view(2, 3, n), k, return_threshold=True)
    assert mask.dtype == torch.bool and mask.shape == (2, 3, n) and thr.shape == (2, 3)
    want = topk_mask_ref(vals.numpy(), k)
    assert (mask.view(6, n).cpu().numpy() == want).all()
    if 0 < k <= n:
        kth = torch.sort(vals, dim=1, descending=True).values[:, k - 1]
        assert torch.equal(thr.view(6).cpu(), kth)


@pytest.mark.parametrize("rows,n,k", [(5, 32769, 5), (5, 40000, 39999), (5, 70001, 1234), (5, 262144, 65536),
                                      (5, 300007, 100000),
                                      (128, 65537, 3000), (64, 131072, 131000)])   # 32 keys per thread
def test_topk_long_rows_with_and_without_scratch(rows, n, k):
    """Rows of more than 32768 columns: spread over workgroups when the caller brings scratch
    (fcr_topk_mask_ws), one workgroup per row otherwise (fcr_topk_mask); both against the oracle."""
    from flash_colreduce_amd import _lib
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n)
    vals = torch.randn(rows, n, generator=g)
    vals[1] = (vals[1] * 4).round() / 4           # heavy ties, both signs
    vals[2] = 1.5                                 # all equal: the lowest k columns win
    vals[3, : n // 2] = vals[3, n // 2: n // 2 * 2]   # every value of the first half twice
    want = topk_mask_ref(vals.numpy(), k)
    kth = torch.sort(vals, dim=1, descending=True).values[:, k - 1]
    lib = _lib.load()
    dev = vals.cuda()
    stream = torch.cuda.current_stream().cuda_stream
    nbytes = lib.fcr_topk_bytes(rows, n)
    assert nbytes > 0 and lib.fcr_topk_bytes(rows, 32768) == 0
    ws = torch.full((nbytes,), 0xAB, device="cuda", dtype=torch.uint8)   # the scratch need not be cleared
    for use_ws in (True, False):
        mask = torch.full((rows, n), 7, device="cuda", dtype=torch.uint8)
        thr = torch.empty(rows, device="cuda")
        if use_ws:
            _lib.check(lib.fcr_topk_mask_ws(dev.data_ptr(), mask.data_ptr(), thr.data_ptr(), rows, n, k, ws.data_ptr(),
                                            nbytes, stream))
        else:
            _lib.check(lib.fcr_topk_mask(dev.data_ptr(), mask.data_ptr(), thr.data_ptr(), rows, n, k, stream))
        assert (mask.cpu().numpy() == want).all(), use_ws
        assert torch.equal(thr.cpu(), kth), use_ws


def test_topk_takes_the_operator_result_as_it_comes():
    """fp16 / bf16 scores, as flash_colreduce returns them for 16-bit operands: same mask as for their fp32 values."""
    from oracle.colreduce_oracle import topk_mask_ref
    q, k = _inputs.randn_pair(1, 3, 200, 3000, 64, seed=21, dtype=torch.bfloat16)
    scores = fca.flash_colreduce(q.cuda(), k.cuda(), "sum", is_causal=True)
    assert scores.dtype == torch.bfloat16
    mask = fca.topk_keep_mask(scores, 500)
    want = topk_mask_ref(scores.float().cpu().view(3, 3000).numpy(), 500)
    assert (mask.view(3, 3000).cpu().numpy() == want).all()
    with pytest.raises(ValueError):
        fca.topk_keep_mask(scores.to(torch.float64), 5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(1, 1), (7, 3), (1000, 100), (1027, 1000), (8192, 2048), (8190, 17), (32768, 5000),
                                 (32770, 300), (70001, 20000), (300004, 1000)])
def test_topk_reads_16_bit_rows(n, k, dtype):
    """16-bit score rows are read by the kernels themselves (every kernel of the selection, rows that do and
    do not start on 8-byte boundaries): heavy ties, as 16-bit values have them, against the oracle on the
    widened values; the threshold is the k-th largest value, widened."""
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(7 * n + k)
    vals = torch.randn(5, n, generator=g).to(dtype)
    vals[1] = (torch.rand(n, generator=g) * 4).to(dtype)          # a few hundred distinct values
    vals[2] = 0.5
    vals[3, ::2] = -0.0
    vals[3, 1::2] = 0.0
    mask, thr = fca.topk_keep_mask(vals.cuda(), k, return_threshold=True)
    want = topk_mask_ref(vals.float().numpy(), k)
    assert (mask.cpu().numpy() == want).all()
    kth = torch.sort(vals.float(), dim=1, descending=True).values[:, k - 1]
    assert thr.dtype == torch.float32 and torch.equal(thr.cpu() + 0.0, kth + 0.0)   # + 0.0: -0 and +0 are one value


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [100, 5000, 20000, 40000, 70001])
def test_topk_orders_nans_above_everything(n, dtype):
    """A NaN of either sign ranks above +inf, NaNs tie (lower column first): every kernel of the selection
    against the oracle; the threshold is a NaN exactly when the k-th largest entry is one."""
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n)
    vals = torch.randn(4, n, generator=g).to(dtype)
    nan = float("nan")
    vals[0, [3, n // 2, n - 1]] = nan
    vals[0, 7] = float("inf")
    vals[1, 5] = -nan
    vals[1, 50] = nan
    vals[2, ::3] = nan                                   # a third of the row
    vals[3] = nan                                        # the whole row
    vals[3, 10] = 1.0
    lib_rows = vals.cuda()
    for k in (1, 2, 3, 4, 5, n // 3, n // 2, n - 1, n):
        mask, thr = fca.topk_keep_mask(lib_rows, k, return_threshold=True)
        want = topk_mask_ref(vals.float().numpy(), k)
        assert (mask.cpu().numpy() == want).all(), k
        nans = torch.isnan(vals.float()).sum(1)
        assert torch.equal(torch.isnan(thr.cpu()), nans >= k), k


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("n", [63, 2047, 2048, 2049, 8191, 8193, 32761, 32768])
def test_topk_narrowing(n, dtype):
    """Rows that end the narrowing in each of its ways, at the edges of the three workgroup sizes: spread scores
    (ranked after the first count), one value in most columns, two neighbouring values, values packed into one bin
    of the first count by a far outlier on either side, everything equal; bases that are not 16-byte aligned."""
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n)
    r = torch.randn(7, n, generator=g)
    r[1] = torch.where(r[1] < 1, torch.zeros(n), r[1])
    r[2] = torch.where(r[2] < 0, torch.full((n,), 0.5), torch.full((n,), 0.5 + 2.0 ** -11))
    r[3] = 1 + r[3].abs() * 1e-3
    r[3, n // 2] = 6e4
    r[4] = 1 + r[4].abs() * 1e-3
    r[4, n // 3] = -6e4
    r[5] = -3.25
    r[6] = float("nan")
    r[6, : n // 2] = -float("inf")
    r = r.to(dtype)
    dev = r.cuda()   # rows of an odd number of elements: their bases have every alignment
    for k in (1, n // 4, n // 2 + 1, n - 1, n):
        mask, thr = fca.topk_keep_mask(dev, k, return_threshold=True)
        want = topk_mask_ref(r.float().numpy(), k)
        assert (mask.cpu().numpy() == want).all(), (n, k, dtype)
        torch.testing.assert_close(thr.cpu(), r.float().sort(dim=1, descending=True).values[:, k - 1], rtol=0, atol=0,
                                   equal_nan=True)   # (a NaN sorts above +inf)


@pytest.mark.parametrize("n,c", [(1100, 127), (2048, 128), (2048, 129), (4666, 126), (8192, 130), (8193, 255), (20000, 256),
                                 (32768, 257), (32768, 600)])
def test_topk_bins_of_many_keys(n, c):
    """A first bin that holds c keys, on both sides of the number that is ranked at once (128, or 256 in rows of more than
    8192 columns), with the k-th largest at its top, inside it and at its end: c equal values, c values in
    neighbouring floats, and both kinds in one bin.  Mask and threshold."""
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n + c)
    base = torch.linspace(2.0, 4.0, n).repeat(3, 1)       # neighbours 2^23 / n floats apart
    at = n // 2
    base[:, at: at + c] = 3.0
    steps = torch.arange(c) * 2.0 ** -22                  # neighbouring floats; a bin takes 2^13 (up to 2048 columns 2^15)
    base[1, at: at + c] += steps
    base[2, at: at + c] += torch.where(torch.arange(c) < c // 2, torch.zeros(c), steps)
    rows = base[:, torch.randperm(n, generator=g)].contiguous()
    above = int((base[0] > 3.0).sum())
    for k in (above - 1, above + 1, above + c // 2, above + c - 1, above + c + 1):
        mask, thr = fca.topk_keep_mask(rows.cuda(), k, return_threshold=True)
        assert (mask.cpu().numpy() == topk_mask_ref(rows.numpy(), k)).all(), (n, c, k)
        assert torch.equal(thr.cpu(), rows.sort(dim=1, descending=True).values[:, k - 1]), (n, c, k)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [9, 2040, 2048, 2049, 8192, 8199, 16384, 16391, 32768, 32775, 65536, 65537])
def test_topk_16_bit_rows_of_any_bits(n, dtype):
    """16-bit rows at the edges of the workgroups that hold them, bases of every 2-byte alignment: every bit pattern (infinities,
    NaNs, denormals, both zeros), one value in most columns, a bin of a few values, all equal to the largest key (NaN).  Mask and
    threshold are exact."""
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n)
    r = torch.randint(-32768, 32768, (5, n), generator=g, dtype=torch.int32).to(torch.int16).view(dtype)
    r[1] = torch.randn(n, generator=g).exp().to(dtype)
    r[2] = torch.where(r[1].float() < 3, torch.ones(()), r[1].float()).to(dtype)
    r[3] = (1 + torch.randint(0, 5, (n,), generator=g) * 2.0 ** -7).to(dtype)
    r[3, n // 2] = float("inf")
    r[4] = float("nan")
    dev = r.cuda()
    for k in (1, n // 4 + 1, n // 2, n - 1, n):
        mask, thr = fca.topk_keep_mask(dev, k, return_threshold=True)
        assert (mask.cpu().numpy() == topk_mask_ref(r.float().numpy(), k)).all(), (n, k)
        kth = r.float().sort(dim=1, descending=True).values[:, k - 1]
        torch.testing.assert_close(thr.cpu() + 0.0, kth + 0.0, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 17, 511, 513, 2050, 8193, 20011])
def test_topk_16_bit_rows_without_signs(n, dtype):
    """Waves whose columns are all at least zero take their keys from the bits: such rows, all zeros, denormals and infinities, and
    rows of which one wave alone holds a negative number, a negative zero or a NaN.  Exact."""
    from oracle.colreduce_oracle import topk_mask_ref
    g = torch.Generator().manual_seed(n)
    r = torch.rand(7, n, generator=g).mul(4).exp().to(dtype)
    r[1] = 0
    r[2] = torch.randint(0, 40, (n,), generator=g, dtype=torch.int32).to(torch.int16).view(dtype)
    r[3, n // 2] = float("inf")
    r[4, n - 1] = -1
    r[5, 0] = -0.0
    r[6, n // 3] = float("nan")
    dev = r.cuda()
    for k in sorted({1, (n + 3) // 4, n}):
        mask, thr = fca.topk_keep_mask(dev, k, return_threshold=True)
        assert (mask.cpu().numpy() == topk_mask_ref(r.float().numpy(), k)).all(), (n, k)
        kth = r.float().sort(dim=1, descending=True).values[:, k - 1]
        torch.testing.assert_close(thr.cpu() + 0.0, kth + 0.0, rtol=0, atol=0, equal_nan=True)


def test_topk_on_reduced_columns():
    from oracle.colreduce_oracle import topk_mask_ref
    q, k = _inputs.config4(heads=4, n=2048)
    s = fca.flash_colreduce(q.cuda(), k.cuda(), "sum", is_causal=True, out_dtype=torch.float32)
    mask = fca.topk_keep_mask(s, 512)
    assert (mask.sum(-1) == 512).all()
    assert (mask.view(4, 2048).cpu().numpy() == topk_mask_ref(s.view(4, 2048).cpu().numpy(), 512)).all()
    assert mask[..., 0].all()   # the sink column is always kept


def test_random_shapes_against_oracle():
    """Seeded sweep over shapes, dtypes, masks, scales and layouts that no other test names."""
    import random
    rng = random.Random(20240607)
    for case in range(60):
        b, h = rng.randint(1, 3), rng.randint(1, 5)
        m = rng.choice([1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 100, 127, 129, 255, 257, 400, 513, 700])
        n = rng.choice([1, 3, 16, 17, 32, 63, 65, 128, 130, 255, 256, 257, 300, 511, 640, 1025, 2100])
        d = rng.choice([8, 16, 24, 32, 40, 64, 72, 96, 100, 128, 136, 160, 192, 256])
        dtype = rng.choice([torch.float16, torch.bfloat16])
        causal = rng.random() < 0.5
        scale = rng.choice([None, None, 0.07, 0.3])
        q, k = _inputs.randn_pair(b, h, m, n, d, seed=1000 + case, dtype=dtype)
        if rng.random() < 0.3:  # [B, rows, H, D] storage
            q = q.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
            k = k.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
        reds = rng.sample(REDUCTIONS, rng.randint(1, 3))
        what = f"case {case}: b{b} h{h} m{m} n{n} d{d} {dtype} causal={causal} scale={scale} {reds}"
        outs = fca.flash_colreduce_multi(q.cuda(), k.cuda(), reds, is_causal=causal, scale=scale,
                                         out_dtype=torch.float32)
        for red, got in zip(reds, outs):
            check(got, colreduce_ref(q, k, red, causal, scale=scale), red, what)


def test_random_decode_shapes_and_fp32_against_oracle():
    """Second seeded sweep: few queries against many keys (single sweep and its neighbours on either side of
    its limits: 128 queries, 1024 keys, rows of 256 bytes) and fp32 operands of any shape."""
    import random
    rng = random.Random(977)
    for case in range(60):
        b, h = rng.randint(1, 2), rng.randint(1, 6)
        if case % 3 == 2:
            dtype = torch.float32
            m = rng.choice([1, 5, 64, 100, 129, 300])
            n = rng.choice([7, 130, 513, 1500, 2600])
            d = rng.choice([4, 12, 64, 100, 128, 200, 256])
        else:
            dtype = rng.choice([torch.float16, torch.bfloat16])
            m = rng.choice([1, 2, 16, 33, 63, 64, 65, 100, 127, 128, 129, 140])
            n = rng.choice([960, 1023, 1024, 1025, 1100, 2047, 2049, 3000, 4097, 7000, 9001])
            d = rng.choice([8, 32, 64, 72, 128, 136])
        causal = rng.random() < 0.5
        scale = rng.choice([None, None, 0.05, 0.4])
        q, k = _inputs.randn_pair(b, h, m, n, d, seed=5000 + case, dtype=dtype)
        if rng.random() < 0.3:  # [B, rows, H, D] storage
            q = q.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
            k = k.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
        reds = rng.sample(REDUCTIONS, rng.randint(1, 3))
        what = f"case {case}: b{b} h{h} m{m} n{n} d{d} {dtype} causal={causal} scale={scale} {reds}"
        for red in reds:   # one call per reduction: the calls that may take the single sweep
            got = fca.flash_colreduce(q.cuda(), k.cuda(), red, is_causal=causal, scale=scale, out_dtype=torch.float32)
            check(got, colreduce_ref(q, k, red, causal, scale=scale), red, what)


def _columns_f64(q, k, causal, scale=None):
    """Column sums and maxima in 64 bits on the device (q, k: (B,H,.,D) on the GPU)."""
    q, k = q.double(), k.double()
    m, n = q.shape[2], k.shape[2]
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * (q.shape[3] ** -0.5 if scale is None else scale)
    if causal:
        hidden = torch.arange(n, device=q.device)[None] > torch.arange(m, device=q.device)[:, None] + max(n - m, 0)
        s = s.masked_fill(hidden, float("-inf"))
    p = s.softmax(-1)
    return p.sum(2), p.amax(2)


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


# keys around what a wave's groups and the forms hold (16, 128, 256, 512), one more than the most; queries around a chunk (16, 32)
# and a split; pairs that share workgroups (few) and that do not
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d,dtype", [
    (1, 2, 1, 8, torch.float16), (3, 31, 15, 64, torch.bfloat16), (2, 33, 129, 128, torch.float16), (130, 64, 128, 72, torch.bfloat16),
    (300, 17, 127, 128, torch.float16), (5, 300, 256, 128, torch.float16), (260, 70, 250, 96, torch.bfloat16), (2, 257, 257, 64, torch.float16),
    (20, 512, 512, 128, torch.bfloat16), (140, 100, 511, 128, torch.float16), (70, 320, 300, 40, torch.float16), (300, 40, 512, 32, torch.float16),
    (2, 5000, 200, 128, torch.float16), (3, 100, 256, 256, torch.bfloat16), (260, 33, 130, 192, torch.float16), (4, 65, 257, 256, torch.float16),
    (4, 90, 513, 128, torch.float16), (64, 1, 200, 128, torch.float16), (300, 15, 16, 136, torch.bfloat16),
    # long calls on both sides of the line that leaves them to the two kernels
    (150, 255, 300, 64, torch.float16), (150, 257, 300, 64, torch.float16), (256, 500, 500, 64, torch.bfloat16), (70, 520, 300, 32, torch.float16),
    (160, 1500, 141, 8, torch.float16), (160, 1537, 141, 8, torch.bfloat16), (150, 790, 400, 96, torch.float16), (70, 1000, 3, 64, torch.float16)])
def test_few_keys(h, m, n, d, dtype, causal):
    """Pairs whose keys fit a workgroup's registers: sums, maxima, both at once and the row statistics, against 64 bits.  A score of
    magnitude 2^4 is rounded to 2^-20, so a probability is good to 2^-19 and a few 1e-6 in the norm; 1e-5 leaves room for
    the order of the sums."""
    g = torch.Generator(device="cuda").manual_seed(h + m + n)
    q, k = (torch.randn(2, h, r, d, device="cuda", generator=g).to(dtype) for r in (m, n))
    sums, most = _columns_f64(q, k, causal)
    got = fca.flash_colreduce(q, k, "sum", causal, out_dtype=torch.float32)
    assert torch.isfinite(got).all() and _rel(got, sums) <= 1e-5
    mx = fca.flash_colreduce(q, k, "max", causal, out_dtype=torch.float32)
    assert _rel(mx, most) <= 1e-5
    s2, m2 = fca.flash_colreduce_multi(q, k, ["sum", "max"], causal, out_dtype=torch.float32)
    assert _rel(s2, sums) <= 1e-5 and _rel(m2, most) <= 1e-5
    ws = torch.empty(_lib_workspace(q, k), device="cuda")
    out = torch.empty(2 * h, n, device="cuda")
    _ws_call(q, k, out, ws, causal)
    torch.testing.assert_close(ws[: 2 * h * m].view(2, h, m), fca.row_lse2(q, k, causal), rtol=1e-5, atol=1e-5)
    assert torch.equal(out.view(2, h, n), got)


@pytest.mark.parametrize("h,m,n,d", [(2, 100, 1025, 128), (3, 128, 1600, 64), (70, 65, 2048 + 64, 128), (2, 64, 2049, 64), (3, 33, 2100, 128),
                                     (80, 40, 4096 + 39, 96), (300, 30, 1024 + 3, 128), (9, 32, 3072 + 31, 64)])
def test_single_sweep_rows_that_see_none_of_the_last_keys(h, m, n, d):
    """Causal, and the last workgroup of a team has fewer keys than there are queries: the first rows see none of them, which is a sum of 0 and
    no reason to sweep again.  Every form of the sweep (65 to 128, 33 to 64, up to 32 queries with eight and four waves), against 64 bits (see
    test_few_keys for the bound); a NaN query in such a row against the two kernels."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(n + m)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).bfloat16() for r in (m, n))
    sums, most = _columns_f64(q, k, True)
    got = [fca.flash_colreduce(q, k, red, True, out_dtype=torch.float32) for red in ("sum", "max")]
    got += fca.flash_colreduce_multi(q, k, ["sum", "max"], True, out_dtype=torch.float32)
    for x, want in zip(got, (sums, most, sums, most)):
        assert torch.isfinite(x).all() and _rel(x, want) <= 1e-5
    q[:, 0, 0, 0] = float("nan")
    for red in ("sum", "max"):
        both = []
        for option in (1, 0):
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
            try:
                both.append(fca.flash_colreduce(q, k, red, True, out_dtype=torch.float32))
            finally:
                lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
        torch.testing.assert_close(both[0], both[1], rtol=1e-4, atol=1e-6, equal_nan=True)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(3, 33, 1500, 64), (2, 63, 2111, 128), (70, 65, 1111, 128), (3, 127, 1024, 96), (3, 128, 1100, 64),
                                     (80, 17, 4100, 128), (300, 31, 1030, 128)])
def test_single_sweep_hidden_scores_beside_odd_rows(h, m, n, d, causal):
    """What the mask hides and rows of padding (query counts that fill no tile) are told apart by their values unless some row's are not finite: keys of
    both signs of infinity and NaN, which rows of padding meet as NaN, and NaN queries, in sums, maxima and both, in every form of the sweep, against the
    two kernels: NaN in the same columns, the others the same to rounding."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(n + m)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).half() for r in (m, n))
    cases = []
    for value in (float("inf"), float("-inf"), float("nan")):
        bad = k.clone()
        bad[:, 0, n // 2, 1] = value
        bad[:, -1, n - 1, 0] = value
        cases += [(q, bad)]
    same_sign = q.clone()
    same_sign[..., 1] = -same_sign[..., 1].abs() - 0.1   # (every score of the infinite key is -inf)
    dead = k.clone()
    dead[:, :, n // 2, 1] = float("inf")
    bad_q = q.clone()
    bad_q[:, 0, m // 2, 0] = float("nan")
    cases += [(same_sign, dead), (bad_q, k), (bad_q, dead)]
    for at, (x, y) in enumerate(cases):
        got = {}
        for option in (1, 0):
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
            try:
                got[option] = [fca.flash_colreduce(x, y, red, causal, out_dtype=torch.float32) for red in ("sum", "max")]
                got[option] += fca.flash_colreduce_multi(x, y, ["sum", "max"], causal, out_dtype=torch.float32)
            finally:
                lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
        for a, b in zip(got[1], got[0]):
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-6, equal_nan=True, msg=lambda t: f"case {at}: {t}")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(2, 100, 1024, 128), (3, 128, 1100, 64), (30, 65, 2049, 128), (100, 70, 1600, 64), (129, 128, 1025, 96), (2, 64, 2100, 128),
                                     (1, 33, 65536, 64), (40, 40, 3000, 96), (100, 48, 1025, 128), (300, 60, 1200, 128), (300, 20, 2900, 128), (7, 32, 5000, 64)])
def test_single_sweep_keys_dealt_evenly(h, m, n, d, causal):
    """Keys dealt to as few workgroups as can hold them and, in one round, to as many as there are CUs for: two steps each, one more or
    less in the last, ragged chunks, in every form of the sweep; against 64 bits (see test_few_keys for the bound)."""
    g = torch.Generator(device="cuda").manual_seed(n + m)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).half() for r in (m, n))
    sums, most = _columns_f64(q, k, causal)
    got = [fca.flash_colreduce(q, k, red, causal, out_dtype=torch.float32) for red in ("sum", "max")]
    got += fca.flash_colreduce_multi(q, k, ["sum", "max"], causal, out_dtype=torch.float32)
    for x, want in zip(got, (sums, most, sums, most)):
        assert torch.isfinite(x).all() and _rel(x, want) <= 1e-5


def _lib_workspace(q, k):
    from flash_colreduce_amd import _lib
    b, h, m, d = q.shape
    return _lib.load().fcr_workspace_bytes({torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}[q.dtype], b, h, m, k.shape[2], d) // 4


def _ws_call(q, k, out, ws, causal, scale=None):
    from flash_colreduce_amd import _lib
    b, h, m, d = q.shape
    code = {torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}[q.dtype]
    _lib.check(_lib.load().fcr_colreduce_ws(
        q.data_ptr(), k.data_ptr(), out.data_ptr(), None, _lib.DTYPE_F32, ws.data_ptr(), 4 * ws.numel(), code, b, h, m, k.shape[2], d,
        _lib.strides4(q.stride()), _lib.strides4(k.stride()), d ** -0.5 if scale is None else scale, _lib.REDUCE_SUM, int(causal),
        torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(2, 100, 100, 64), (3, 70, 300, 128), (300, 40, 200, 128), (2, 65, 250, 256)])
def test_few_keys_scores_that_the_plain_sums_do_not_take(h, m, n, d, causal):
    """Against the two kernels where 2^score leaves the range of a sum, scales of any sign, layouts, rows and keys that are not finite:
    the same columns are NaN, the others agree to what scores of magnitude 2^9 (2^-15 each) leave."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(h + n)

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    q, k = rand(1, h, m, d), rand(1, h, n, d)
    far_q, far_k, jump = q.clone(), k.clone(), k.clone()
    far_q[:, :, m // 2:] *= 40
    far_k[:, :, ::3] -= 6 * q[:, :, :1]
    jump[:, :, n // 2] *= 60
    bad_q, bad_k, low_k = q.clone(), k.clone(), k.clone()
    bad_q[:, 0, m // 3, 0] = float("nan")
    bad_q[:, -1, m - 1, 1] = float("inf")
    bad_k[:, 0, n // 2, 0] = float("inf")
    low_k[:, :, 1:, :] = 0
    low_k[:, :, 0, 0] = float("-inf")
    cases = [(q, k, None), (far_q, k, None), (q, far_k, None), (q, jump, None), (bad_q, k, None), (q, bad_k, None), (q.abs(), low_k, None),
             (q, k, 0.0), (q, k, -0.3), (q.transpose(2, 1).contiguous().transpose(2, 1), k[:, :1].expand(1, h, n, d), None),
             (q, k, None), (q, k, None)]
    for at, (x, y, scale) in enumerate(cases):
        x, y = x.half(), y.half()
        if at == 9:      # keys that the heads share by a stride of zero (a conversion would make each head its own)
            y = k[:, :1].half().expand(1, h, n, d)
        elif at == 10:   # padded key rows
            y = torch.nn.functional.pad(y, (0, 8))[..., :d]
        elif at == 11:   # token-major keys
            y = y.transpose(1, 2).contiguous().transpose(1, 2)
        assert y.stride(2) == {10: d + 8, 11: h * d}.get(at, d)
        for red in ("sum", "max"):
            got = {}
            for option in (1, 0):
                lib.fcr_set_option(0, option)
                try:
                    got[option] = fca.flash_colreduce(x, y, red, causal, scale, out_dtype=torch.float32)
                finally:
                    lib.fcr_set_option(0, 1)
            assert torch.equal(got[1].isnan(), got[0].isnan()), (at, red)
            torch.testing.assert_close(got[1], got[0], rtol=2e-4, atol=1e-6, equal_nan=True, msg=lambda t: f"case {at} {red}: {t}")


@pytest.mark.parametrize("dtype,level", [(torch.bfloat16, 20), (torch.bfloat16, 30), (torch.float16, 30)])
def test_few_keys_far_scores_round_once(dtype, level):
    """Rows whose scores lie far below zero together, which the plain sums do not take: product * scale less the row's lse is rounded once,
    as in the two kernels, so the errors against 64 bits are no larger than theirs.  (Rounded twice one of the errors of each case is
    0.4 to 4 % larger; these 6144 columns of 70 rows leave less than 1 % between two orders of summation.)"""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    h, m, n, d = 24, 70, 256, 192
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g) for r in (m, n))
    o = torch.randn(1, h, 1, d, device="cuda", generator=g)
    o *= level ** 0.5 * d ** 0.25 / o.norm(dim=-1, keepdim=True)
    q, k = (q + o).to(dtype), (k - o).to(dtype)   # scores around -level
    sums, most = _columns_f64(q, k, True)
    err = {}
    for option in (1, 0):
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
        try:
            err[option] = [_rel(fca.flash_colreduce(q, k, red, True, out_dtype=torch.float32), want)
                           for red, want in (("sum", sums), ("max", most))]
        finally:
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
    assert all(now <= 1.003 * two for now, two in zip(err[1], err[0])), err


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d,scale", [(2, 100, 100, 64, None), (300, 97, 130, 128, None), (3, 300, 256, 96, -0.1), (300, 70, 512, 64, None),
                                           (2, 1000, 300, 128, None), (2, 65, 250, 256, None), (260, 49, 120, 192, -0.07)])
def test_few_keys_from_a_far_row_on(h, m, n, d, scale, causal):
    """Rows whose scores lie around -30, which the plain sums do not take, from the first row on, from one inside a chunk, from the first of a chunk,
    in the last row only and in one row alone: what is left of a workgroup's chunks is then formed the other way.  Scores of magnitude
    2^6 are rounded to 2^-18, those of products of 30 * sqrt(d) in fp32 sums to about the same: 2e-5 in the norm holds both."""
    g = torch.Generator(device="cuda").manual_seed(h + m + d)
    q0, k = (torch.randn(1, h, r, d, device="cuda", generator=g) for r in (m, n))
    o = torch.randn(1, h, 1, d, device="cuda", generator=g)
    o *= (30 / (d ** -0.5 if scale is None else -scale)) ** 0.5 / o.norm(dim=-1, keepdim=True)
    if scale is not None:
        k = -k
    k = k - o if scale is None else k + o
    k = k.half()
    for rows in (slice(0, m), slice(m // 2, m), slice(m // 3, m // 3 + 1), slice(32, 64), slice(m - 1, m)):
        q = q0.clone()
        q[:, :, rows] += o if scale is None else -o
        q = q.half()
        sums, most = _columns_f64(q, k, causal, scale)
        got = [fca.flash_colreduce(q, k, red, causal, scale, out_dtype=torch.float32) for red in ("sum", "max")]
        both = fca.flash_colreduce_multi(q, k, ["sum", "max"], causal, scale, out_dtype=torch.float32)
        for x, want in ((got[0], sums), (got[1], most), (both[0], sums), (both[1], most)):
            assert _rel(x, want) <= 2e-5, rows
        ws, out = torch.empty(_lib_workspace(q, k), device="cuda"), torch.empty(h, n, device="cuda")
        _ws_call(q, k, out, ws, causal, scale)
        torch.testing.assert_close(ws[: h * m].view(1, h, m), fca.row_lse2(q, k, causal, scale), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("m,n,d", [(40, 40, 64), (20, 200, 128), (33, 250, 256), (16, 500, 64)])
def test_few_keys_small_probabilities_of_small_sums(m, n, d, causal):
    """Rows whose sum of 2^score is between 2^-20 and 1 with keys whose 2^score fp32 cannot hold, though their probabilities of 2^-118 to
    2^-126 it can: bf16 and fp32 results keep them, as the two kernels do.  The exponents are integers here and the sums short, so a
    probability is good to the rounding of an lse of magnitude 2^3 and of a score of 2^7 (2^-18 together)."""
    q = torch.zeros(1, 3, m, d, device="cuda", dtype=torch.float16)
    k = torch.zeros(1, 3, n, d, device="cuda", dtype=torch.float16)
    q[..., 0] = 1
    k[..., 0] = -math.floor(math.log2(n)) - 4        # 2^-4 to 2^-3 in a row that sees every key
    k[:, :, 1::7, 0] = -126 - torch.arange(1, 4, device="cuda").repeat(n)[: len(range(1, n, 7))].half()
    want, most = _columns_f64(q, k, causal, math.log(2))
    assert ((want > 0) & (want < 2.0 ** -110)).any()
    got = fca.flash_colreduce(q, k, "sum", causal, math.log(2), out_dtype=torch.float32)
    two = fca.flash_colreduce_multi(q, k, ["sum", "max"], causal, math.log(2), out_dtype=torch.float32)
    for x, y in ((got, want), (two[0], want), (two[1], most)):
        assert ((x.double() - y).abs() <= 2.0 ** -17 * y).all(), ((x.double() - y) / y).abs().max()
    low = fca.flash_colreduce(q.bfloat16(), k.bfloat16(), "sum", causal, math.log(2))
    assert ((low.double() - want).abs() <= 2.0 ** -8 * want).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [
    (1, 2, 1, 32), (3, 31, 15, 64), (2, 33, 129, 128), (300, 65, 128, 72), (5, 300, 256, 128), (2, 257, 255, 60), (20, 200, 200, 40),
    (2, 1000, 17, 96), (9, 1056, 33, 128), (3, 5000, 250, 64), (3, 100, 256, 256), (4, 16, 130, 192), (150, 49, 250, 160), (260, 15, 127, 224), (2, 256, 256, 64),
    # on both sides of the lines that leave long calls, and more keys, to the two kernels
    (128, 257, 256, 32), (2, 224, 200, 32), (130, 520, 40, 64), (130, 512, 200, 64), (260, 1100, 30, 64), (260, 1500, 20, 36), (4, 90, 257, 64)])
def test_few_keys_f32(h, m, n, d, causal):
    """fp32 pairs whose keys fit a workgroup's registers: sums, maxima, both and the row statistics against 64 bits, to the 1e-5 that fp32
    operands are held to everywhere, and no further off than 1.15 times the two kernels (their own spread between shapes) in any of them."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(h + m + n)
    q, k = (torch.randn(2, h, r, d, device="cuda", generator=g) for r in (m, n))
    sums, most = _columns_f64(q, k, causal)
    err = {}
    for option in (1, 0):
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
        try:
            one = [fca.flash_colreduce(q, k, red, causal) for red in ("sum", "max")]
            two = fca.flash_colreduce_multi(q, k, ["sum", "max"], causal)
            ws = torch.empty(lib.fcr_workspace_bytes(_lib.DTYPE_F32, 2, h, m, n, d) // 4, device="cuda")
            out = torch.empty(2 * h, n, device="cuda")
            _lib.check(lib.fcr_colreduce_ws(
                q.data_ptr(), k.data_ptr(), out.data_ptr(), None, _lib.DTYPE_F32, ws.data_ptr(), 4 * ws.numel(), _lib.DTYPE_F32, 2, h, m, n, d,
                _lib.strides4(q.stride()), _lib.strides4(k.stride()), d ** -0.5, _lib.REDUCE_SUM, int(causal), torch.cuda.current_stream().cuda_stream))
        finally:
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
        torch.testing.assert_close(ws[: 2 * h * m].view(2, h, m), fca.row_lse2(q, k, causal), rtol=1e-5, atol=1e-5)
        assert torch.equal(out.view(2, h, n), one[0])
        err[option] = [_rel(x, want) for x, want in ((one[0], sums), (one[1], most), (two[0], sums), (two[1], most))]
    for now, before in zip(err[1], err[0]):
        assert now <= 1e-5 and now <= max(1.15 * before, 1.2e-7), err


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(2, 70, 70, 64), (3, 100, 250, 128), (300, 40, 100, 32), (2, 65, 250, 256)])
def test_few_keys_f32_special_rows(h, m, n, d, causal):
    """fp32 rows that the parts do not take (not finite, from 2^104 on, elements of 600 on both sides), scores far from zero, scales of any
    sign, token-major and padded layouts: NaN in the columns of the two kernels, the others the same to what scores of magnitude 2^9 leave."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(m + n)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g) for r in (m, n))
    cases = [(q, k, None), (q, k, 0.0), (q, k, -0.2), (q * 30, k, 1.0 / d ** 0.5), (q + 5, k - 5, None), (torch.zeros_like(q), k, None)]
    for value in (float("nan"), float("inf"), float("-inf")):
        bad_q, bad_k = q.clone(), k.clone()
        bad_q[:, 0, m // 3, 1] = value
        bad_k[:, -1, n // 2, 0] = value
        cases += [(bad_q, k, None), (q, bad_k, None), (bad_q, bad_k, -0.1)]
    big_q, big_k = q.clone(), k.clone()
    big_q[:, :, m - 1] *= 2.0 ** 110
    big_k[:, 0, n - 1] *= 2.0 ** 105
    cases += [(big_q, k, 2.0 ** -110), (q, big_k, 2.0 ** -106)]
    one_q, one_k = q.clone(), k.clone()
    one_q[:, :, 5:7, 0] = 600.0   # (past 300 on both sides, with scores below 2^9)
    one_k[:, :, :3, 1] = 600.0
    cases += [(one_q, one_k, None)]
    wide = torch.randn(1, n, h, d + 4, device="cuda", generator=g)[..., :d].transpose(1, 2)
    cases += [(q.transpose(1, 2).contiguous().transpose(1, 2), wide, None)]
    for at, (x, y, scale) in enumerate(cases):
        for red in ("sum", "max", "pair"):
            got = {}
            for option in (1, 0):
                lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
                try:
                    got[option] = (torch.stack(list(fca.flash_colreduce_multi(x, y, ["sum", "max"], causal, scale))) if red == "pair"
                                   else fca.flash_colreduce(x, y, red, causal, scale))
                finally:
                    lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
            assert torch.equal(got[1].isnan(), got[0].isnan()), (at, red)
            torch.testing.assert_close(got[1], got[0], rtol=2e-4, atol=1e-6, equal_nan=True, msg=lambda t: f"case {at} {red}: {t}")


@pytest.mark.parametrize("h,m,n,d", [(1, 500, 250, 64), (3, 130, 70, 64), (1, 1023, 200, 128), (2, 700, 100, 256), (5, 97, 129, 40), (1, 66, 256, 192)])
def test_few_keys_f32_bits_do_not_depend_on_the_number_of_pairs(h, m, n, d):
    """Shared pairs, whose columns a second launch adds up, pairs of one workgroup each and pairs in several rounds, in the ranges of
    queries that sizes alone set."""
    q, k = (x.cuda() for x in _inputs.randn_pair(1, h, m, n, d, seed=m + n, dtype=torch.float32))
    for copies in (60 // h, 600 // h):
        qs, ks = q.repeat(copies, 1, 1, 1), k.repeat(copies, 1, 1, 1)
        for red in REDUCTIONS:
            assert torch.equal(fca.flash_colreduce(q, k, red, True)[0], fca.flash_colreduce(qs, ks, red, True)[-1]), (red, copies)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_few_keys_under_graph_capture(dtype):
    """Shared pairs (two launches) in a captured graph, replayed with other contents and eager calls between."""
    q, k = (torch.randn(1, 4, r, 64, device="cuda").to(dtype) for r in (300, 200))
    fca.flash_colreduce(q, k, "mean", True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fca.flash_colreduce(q, k, "mean", True)
    for _ in range(4):
        q.copy_(torch.randn(q.shape, device="cuda"))
        k.copy_(torch.randn(k.shape, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, fca.flash_colreduce(q, k, "mean", True))


def test_hip_graph_capture_and_replay():
    """The whole call (torch allocations, both kernels, cast) captured in a graph and replayed with
    new contents in the static inputs; every replay must equal the eager result for those contents."""
    b, h, m, n, d = 1, 4, 300, 500, 64
    qs = torch.zeros(b, h, m, d, device="cuda", dtype=torch.float16)
    ks = torch.zeros(b, h, n, d, device="cuda", dtype=torch.float16)
    q0, k0 = _inputs.randn_pair(b, h, m, n, d, seed=77)
    qs.copy_(q0)
    ks.copy_(k0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # warm up outside the capture
        fca.flash_colreduce_multi(qs, ks, ["sum", "max"], True, out_dtype=torch.float32)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        s_out, m_out = fca.flash_colreduce_multi(qs, ks, ["sum", "max"], True, out_dtype=torch.float32)
        one = fca.flash_colreduce(qs, ks, "mean", True, out_dtype=torch.float32)
    for seed in (78, 79, 80):
        q1, k1 = _inputs.randn_pair(b, h, m, n, d, seed=seed)
        qs.copy_(q1)
        ks.copy_(k1)
        graph.replay()
        torch.cuda.synchronize()
        got = (s_out.clone(), m_out.clone(), one.clone())
        es, em = fca.flash_colreduce_multi(qs, ks, ["sum", "max"], True, out_dtype=torch.float32)
        e1 = fca.flash_colreduce(qs, ks, "mean", True, out_dtype=torch.float32)
        torch.cuda.synchronize()
        assert torch.equal(got[0], es) and torch.equal(got[1], em) and torch.equal(got[2], e1), seed
        check(got[0], colreduce_ref(q1, k1, "sum", True), "sum", f"graph replay seed {seed}")


def test_graph_capture_of_a_causal_mean_never_seen_before():
    """The causal mean divisor is built on the device by every call.  Capture a causal mean whose
    divisor length was never used in this process, call eagerly BEFORE the first replay, then capture a
    second graph with the same length and replay only that one: each result must be the oracle's."""
    b, h, m, n, d = 1, 3, 211, 347, 32      # divisor length 211, used by no other test
    qc, kc = _inputs.randn_pair(b, h, m, n, d, seed=91)
    q, k = qc.cuda(), kc.cuda()
    want = colreduce_ref(qc, kc, "mean", True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # warm up the kernels, but not the mean epilogue
        fca.flash_colreduce(q, k, "sum", True, out_dtype=torch.float32)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g1 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g1):
        out1 = fca.flash_colreduce(q, k, "mean", True, out_dtype=torch.float32)
    eager = fca.flash_colreduce(q, k, "mean", True, out_dtype=torch.float32)   # before any replay
    torch.cuda.synchronize()
    check(eager, want, "mean", "eager call between capture and first replay")
    g2 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g2):
        out2 = fca.flash_colreduce(q, k, "mean", True, out_dtype=torch.float32)
    g2.replay()                                                                  # g1 never replayed so far
    torch.cuda.synchronize()
    check(out2, want, "mean", "second graph replayed alone")
    assert torch.equal(out2, eager)
    g1.replay()
    torch.cuda.synchronize()
    assert torch.equal(out1, eager)


def test_launcher_stub_of_the_integration_notes():
    """The ctypes launcher shown to maintainers (the first python block of section 2 of the integration
    notes) is executed as written, against the built library, and must reproduce flash_colreduce."""
    import os
    import re
    from flash_colreduce_amd import _lib
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    text = open(os.path.join(root, "INTEGRATION.md")).read()
    section = text[text.index("## 2."):]
    code = re.search(r"```python\n(.*?)```", section, flags=re.S).group(1)
    code = code.replace("/path/to/libfcr.so", _lib.LIB_PATH)
    scope = {}
    exec(compile(code, "INTEGRATION.md", "exec"), scope)
    for dtype in (torch.float16, torch.bfloat16, torch.float32):   # the three element types the reference's tl.dot takes
        q, k = _inputs.randn_pair(2, 3, 130, 1000, 64, seed=4, dtype=dtype)
        qd, kd = q.cuda(), k.cuda()
        for red, causal in (("sum", True), ("max", False)):
            got = scope["_flash_colreduce"](qd, kd, red, causal, 0.125)
            assert got.dtype == dtype and got.shape == (2, 3, 1000)
            assert torch.equal(got, fca.flash_colreduce(qd, kd, red, is_causal=causal, scale=0.125))


def test_plain_c_caller_of_the_c_abi():
    """tests/c_abi/check.c: hipMalloc, fcr_colreduce, closed forms; no Python or torch in that process."""
    import os
    import subprocess
    from flash_colreduce_amd import build as fcr_build
    from flash_colreduce_amd import _lib
    header = os.path.join(fcr_build.INCLUDE, "fcr.h")
    newest = max(os.path.getmtime(f) for f in (fcr_build.C_CHECK_SRC, header, _lib.LIB_PATH))
    if not os.path.exists(fcr_build.C_CHECK_BIN) or os.path.getmtime(fcr_build.C_CHECK_BIN) < newest:
        fcr_build.build_c_check(verbose=False)   # never a binary older than its source, the header or the library
    done = subprocess.run([fcr_build.C_CHECK_BIN], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.strip() == "ok", (done.returncode, done.stdout, done.stderr)


class _NeverNative:
    """Stands in for the native host path and answers nothing."""
    def reduce(self, *a):
        return None

    def keep(self, *a):
        return None


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_native_host_path_gives_what_the_general_one_gives(dtype, monkeypatch):
    """Layouts, result types, scales and orders: the native path and the Python one run the same launches, so results
    are equal bit for bit; what would need a copy, a message or another device is left to the Python one."""
    from flash_colreduce_amd import flash as F
    b, h, m, n, d = 2, 3, 70, 1100, 64
    g = torch.Generator(device="cuda").manual_seed(5)

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g).to(dtype)

    q, k = rand(b, h, m, d), rand(b, h, n, d)
    qt, kt = rand(b, m, h, d).transpose(1, 2), rand(b, n, h, d).transpose(1, 2)
    odd = rand(b, h, m, d + 3)[..., :d]                        # rows off their alignment: copied
    cases = [(q, k, True), (qt, kt, True), (qt, k, True), (q[:1], k[:1], True), (q[:, :, :1], k, True), (q, k[:, :, 5:905], True),
             (q, k[:1].expand(b, h, n, d), True), (q.as_strided((1, 1, 1, d), (7, 3, 5, 1)), k[:1, :1], True), (odd, k, False),
             (q.expand(b, h, m, d)[:, :, :1].expand(b, h, m, d), k, False), (rand(b, h, m, 20)[..., :18], rand(b, h, n, 20)[..., :18], False),
             (q.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2), k, False)]
    calls = []
    for x, y, native in cases:
        assert (F._host().reduce(x, y, "sum", False, None, None, False) is not None) == native
        for red, causal, scale, out in (("sum", True, None, None), ("mean", 1, 0.3, torch.float32), ("max", False, -0.2, torch.bfloat16)):
            calls.append(lambda x=x, y=y, red=red, causal=causal, scale=scale, out=out: fca.flash_colreduce(x, y, red, causal, scale, out_dtype=out))
        for reds in (["sum", "max"], ("max", "mean"), ["max", "max"], ["mean", "sum"], ["max"], ["sum", "max", "sum"]):
            calls.append(lambda x=x, y=y, reds=reds: fca.flash_colreduce_multi(x, y, reds, is_causal=True))
    s = rand(b, h, n)
    for scores in (s, s[0], s[0, 0], s[:, :, ::2], s.float(), s.permute(2, 0, 1), rand(3, 1, 70000)):
        for kk in (0, 5, scores.shape[-1], -3, True):
            calls.append(lambda scores=scores, kk=kk: fca.topk_keep_mask(scores, kk, return_threshold=kk != 5))

    def flat(r):
        return list(r) if isinstance(r, tuple) else [r]

    native = [flat(c()) for c in calls]
    monkeypatch.setattr(F, "_native", _NeverNative())
    for c, got in zip(calls, native):
        want = flat(c())
        assert len(want) == len(got)
        for x, y in zip(got, want):
            assert x.shape == y.shape and x.dtype == y.dtype and x.is_contiguous()
            assert torch.equal(torch.nan_to_num(x.float(), nan=7.5), torch.nan_to_num(y.float(), nan=7.5))


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("dtype,n,scratch", [(torch.float16, 50000, False), (torch.bfloat16, 65536, False), (torch.float16, 65544, True),
                                             (torch.float32, 50000, True)])
def test_topk_allocates_no_scratch_that_no_kernel_reads(dtype, n, scratch, native, monkeypatch):
    from flash_colreduce_amd import flash as F
    if not native:
        monkeypatch.setattr(F, "_native", _NeverNative())
    s = torch.rand(4, n, device="cuda").to(dtype)
    fca.topk_keep_mask(s, 100)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    mask = fca.topk_keep_mask(s, 100)
    extra = torch.cuda.max_memory_allocated() - before
    assert (extra > 4 * n + 4096) == scratch and mask.sum().item() == 400


def test_native_host_path_under_capture_streams_and_modes():
    """Allocations and launches go where torch's would: into a captured graph (replayed with other contents and eager calls between),
    on the caller's stream, out of inference mode; a refused argument of the library raises its error."""
    from flash_colreduce_amd import _lib
    q, k = (x.cuda() for x in _inputs.randn_pair(1, 4, 90, 300, 64, seed=1))
    q2, k2 = (x.cuda() for x in _inputs.randn_pair(1, 4, 90, 300, 64, seed=2))
    want = [fca.flash_colreduce(a, c, "mean", True) for a, c in ((q, k), (q2, k2))]
    masks = [fca.topk_keep_mask(w, 30) for w in want]
    qs, ks = q.clone(), k.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fca.flash_colreduce(qs, ks, "mean", True)
        mask = fca.topk_keep_mask(out, 30)
    for i in (1, 0, 1):
        qs.copy_((q, q2)[i])
        ks.copy_((k, k2)[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[i]) and torch.equal(mask, masks[i])
        assert torch.equal(fca.flash_colreduce(q, k, "mean", True), want[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(2_000_000)
        late = q.clone()
        assert torch.equal(fca.flash_colreduce(late, k, "mean", True), want[0])
    with torch.inference_mode():
        r = fca.flash_colreduce(q, k, "mean", True)
        assert r.is_inference() and torch.equal(r, want[0])
    assert not fca.flash_colreduce(q.clone().requires_grad_(), k, "mean", True).requires_grad
    with pytest.raises(_lib.FcrError):
        fca.flash_colreduce(q, k, "sum", scale=float("inf"))


def test_python_errors_on_device():
    q = torch.zeros(1, 2, 4, 8, dtype=torch.float16, device="cuda")
    k = torch.zeros(1, 2, 6, 8, dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError, match="Head dimension must be <= 512"):
        fca.flash_colreduce(torch.zeros(1, 1, 4, 513, dtype=torch.float16, device="cuda"),
                            torch.zeros(1, 1, 4, 513, dtype=torch.float16, device="cuda"), "sum")
    with pytest.raises(ValueError, match="Head dimension must be <= 256"):
        fca.flash_colreduce(torch.zeros(1, 1, 4, 260, device="cuda"), torch.zeros(1, 1, 4, 260, device="cuda"), "sum")
    with pytest.raises(ValueError, match="Invalid reduction: median"):
        fca.flash_colreduce(q, k, "median")
    with pytest.raises(ValueError, match="same batch size, number of heads, and head dimension"):
        fca.flash_colreduce(q, k[:, :1], "sum")
    with pytest.raises(ValueError, match="float16, bfloat16 or float32"):
        fca.flash_colreduce(q.double(), k.double(), "sum")
    with pytest.raises(ValueError, match="float16, bfloat16 or float32"):
        fca.flash_colreduce(q.float(), k, "sum")
    # zero queries see no key: every column is 1/N
    out = fca.flash_colreduce(q, k, "max", out_dtype=torch.float32)
    torch.testing.assert_close(out, torch.full((1, 2, 6), 1 / 6, device="cuda"))
    assert fca.flash_colreduce(q[:, :, :0], k, "sum").shape == (1, 2, 6)
    assert fca.flash_colreduce(q, k[:, :, :0], "sum").shape == (1, 2, 0)


@pytest.mark.parametrize("h,m,n,d,dtype,causal", [
    (3, 700, 700, 128, torch.float16, True), (2, 900, 640, 128, torch.bfloat16, True), (3, 600, 850, 128, torch.float16, True),
    (1, 513, 513, 104, torch.float16, True), (60, 1000, 1000, 128, torch.bfloat16, True), (240, 520, 520, 128, torch.float16, True),
    (5, 1101, 1101, 64, torch.float16, True), (270, 520, 521, 48, torch.bfloat16, True), (4, 640, 640, 24, torch.float16, True),
    (9, 777, 777, 96, torch.bfloat16, True), (100, 1000, 1000, 80, torch.float16, True), (3, 530, 530, 256, torch.float16, True),
    (2, 1200, 1200, 200, torch.bfloat16, True), (1, 641, 600, 136, torch.float16, True),
    (130, 600, 600, 128, torch.float16, False), (250, 530, 530, 128, torch.bfloat16, False), (100, 530, 540, 128, torch.float16, False),
    (130, 600, 600, 64, torch.bfloat16, False), (130, 576, 600, 160, torch.float16, False), (240, 600, 1500, 72, torch.float16, False)])
def test_both_sweeps_in_one_launch(h, m, n, d, dtype, causal):
    """Every tile size of the launch that holds both sweeps, ragged tiles and chunks, more and fewer keys than queries: sums, maxima,
    both and the row statistics, against 64 bits (see test_few_keys for the bound) and, where the row sweep of the two launches is not
    split, bit for bit against those."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(h + m + n)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).to(dtype) for r in (m, n))
    sums, most = _columns_f64(q, k, causal)
    got = {}
    for option in (1, 0):
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
        try:
            one = [fca.flash_colreduce(q, k, red, causal, out_dtype=torch.float32) for red in ("sum", "max")]
            pair = fca.flash_colreduce_multi(q, k, ["sum", "max"], causal, out_dtype=torch.float32)
            ws, out = torch.empty(_lib_workspace(q, k), device="cuda"), torch.empty(h, n, device="cuda")
            _ws_call(q, k, out, ws, causal)
            got[option] = [*one, *pair, ws[: h * m].clone(), out.view(1, h, n)]
        finally:
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
    for x, want in zip(got[1], (sums, most, sums, most, None, sums)):
        assert want is None or (torch.isfinite(x).all() and _rel(x, want) <= 1e-5)
    same = h * ((m + 255) // 256) >= 256 and m > 256   # no row sweep of these is split
    for x, y in zip(got[1], got[0]):
        assert torch.equal(x, y) if same else torch.allclose(x, y, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("h,m,n,d", [(3, 700, 700, 128), (60, 1000, 1000, 128), (5, 1100, 1100, 64), (2, 600, 600, 256)])
def test_both_sweeps_in_one_launch_special_rows(h, m, n, d):
    """Rows and keys that are not finite, scores of exactly zero (an lse of 0 for the row that sees one key), scales of any sign:
    NaN in the same columns as with two launches, the others the same to rounding."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(h + n)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).half() for r in (m, n))
    bad_q, bad_k, zero = q.clone(), k.clone(), torch.zeros_like(q)
    bad_q[:, 0, m // 3, 0] = float("nan")
    bad_q[:, -1, m - 1, 1] = float("inf")
    bad_k[:, 0, n // 2, 0] = float("-inf")
    for x, y, scale in ((bad_q, k, None), (q, bad_k, None), (zero, k, None), (q, k, 0.0), (q, k, -0.3)):
        for red in ("sum", "max"):
            got = {}
            for option in (1, 0):
                lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
                try:
                    got[option] = fca.flash_colreduce(x, y, red, True, scale, out_dtype=torch.float32)
                finally:
                    lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
            torch.testing.assert_close(got[1], got[0], rtol=1e-4, atol=1e-6, equal_nan=True)


@pytest.mark.parametrize("reduction", ["sum", "max", "pair"])
def test_both_sweeps_wait_is_bounded(reduction):
    """With no polls allowed the column sweeps, which all start beside the row sweeps here, give up: the kernel ends, the
    columns are NaN, and the next call is right."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    q, k = (x.cuda() for x in _inputs.randn_pair(1, 4, 1200, 1200, 128, seed=5, dtype=torch.float16))
    call = lambda: (fca.flash_colreduce_multi(q, k, ["sum", "max"], True) if reduction == "pair" else [fca.flash_colreduce(q, k, reduction, True)])
    want = call()
    lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 0)
    try:
        assert all(x.isnan().any() for x in call())
    finally:
        lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 1 << 20)
    for x, y in zip(call(), want):
        assert torch.isfinite(x).all() and torch.equal(x, y)


def test_both_sweeps_under_graph_capture():
    """A captured call takes the two launches, whose replays wait for nothing beside them: replays on new operands, with eager calls and
    synchronizations between them, give the bits of two launches and the eager result to rounding."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    q, k = (x.cuda() for x in _inputs.randn_pair(2, 6, 900, 900, 128, seed=3, dtype=torch.bfloat16))
    fca.flash_colreduce(q, k, "sum", True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fca.flash_colreduce(q, k, "sum", True, out_dtype=torch.float32)
    for step in range(4):
        q.copy_(torch.randn_like(q))
        graph.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(out, fca.flash_colreduce(q, k, "sum", True, out_dtype=torch.float32), rtol=1e-5, atol=1e-6)
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 0)
        try:
            assert torch.equal(out, fca.flash_colreduce(q, k, "sum", True, out_dtype=torch.float32)), step
        finally:
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)


def test_launches_that_wait_on_two_streams():
    """Both sweeps in one launch and single sweeps, issued in turn on two streams without a wait between them: the host chains them, and every
    result is the one of a call by itself."""
    shapes = [(6, 900, 900, 128), (32, 100, 4096, 128), (3, 1100, 1100, 64), (64, 64, 8192, 128)]
    ops = [tuple(torch.randn(1, h, r, d, device="cuda").half() for r in (m, n)) for h, m, n, d in shapes]
    want = [fca.flash_colreduce(q, k, "sum", True) for q, k in ops]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = []
    for step in range(12):
        for i, (q, k) in enumerate(ops):
            with torch.cuda.stream(streams[(step + i) % 2]):
                got.append((i, fca.flash_colreduce(q, k, "sum", True)))
    torch.cuda.synchronize()
    assert all(torch.equal(x, want[i]) for i, x in got)


def test_both_sweeps_wait_for_no_other_stream():
    """A call that holds both sweeps in one launch runs while a stream on which the one before it was issued is busy with
    something else: nothing of that stream is waited for."""
    q, k = (x.cuda() for x in _inputs.randn_pair(1, 3, 700, 700, 128, seed=4, dtype=torch.float16))
    want = fca.flash_colreduce(q, k, "sum", True)
    first = torch.cuda.Stream()
    one = torch.ones(1, device="cuda")
    beside = None
    for _ in range(8):   # a stream that runs beside the first one (they share hardware queues)
        other = torch.cuda.Stream()
        with torch.cuda.stream(other):
            fca.flash_colreduce(q, k, "sum", True), one + one
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            torch.cuda._sleep(50_000_000)
            busy = torch.cuda.Event()
            busy.record()
        with torch.cuda.stream(other):
            one + one
        other.synchronize()
        if not busy.query():
            beside = other
            break
    torch.cuda.synchronize()
    assert beside is not None
    with torch.cuda.stream(first):
        fca.flash_colreduce(q, k, "sum", True)
        torch.cuda._sleep(50_000_000)
        busy = torch.cuda.Event()
        busy.record()
    with torch.cuda.stream(beside):
        got = fca.flash_colreduce(q, k, "sum", True)
    beside.synchronize()
    assert not busy.query()
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_prefill_beside_a_captured_decode():
    """Eager calls that hold both sweeps in one launch on one stream, replays of a graph that holds a single sweep on another, with no
    wait between the two streams: every result is that of a call by itself, again after synchronizations and with calls in between."""
    g = torch.Generator(device="cuda").manual_seed(11)
    make = lambda h, m, n, d: tuple(torch.randn(1, h, r, d, device="cuda", generator=g).half() for r in (m, n))
    decode = make(64, 64, 8192, 128)
    prefills = [make(12, 1100, 1100, 128), make(60, 1000, 1000, 128), make(3, 700, 700, 256), make(40, 1500, 1500, 64)]
    want = [fca.flash_colreduce(q, k, "sum", True) for q, k in (decode, *prefills)]
    graph, left, right = torch.cuda.CUDAGraph(), torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.graph(graph):
        out = fca.flash_colreduce(*decode, "sum", True)
    torch.cuda.synchronize()
    for rounds in (1, 4, 8):
        got = []
        for step in range(rounds):
            with torch.cuda.stream(left):
                graph.replay()
                got.append((0, out.clone()))
            with torch.cuda.stream(right):
                got += [(1 + i, fca.flash_colreduce(q, k, "sum", True)) for i, (q, k) in enumerate(prefills)]
        torch.cuda.synchronize()
        assert all(torch.equal(x, want[i]) for i, x in got)
        assert torch.equal(fca.flash_colreduce(*prefills[0], "sum", True), want[1])


def _decode_call(q, k, out, ws, stream):
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    _, h, m, d = q.shape
    _lib.check(lib.fcr_colreduce(q.data_ptr(), k.data_ptr(), out.data_ptr(), ws.data_ptr(), _lib.DTYPE_F16, 1, h, m, k.shape[2], d,
                                 _lib.strides4(q.stride()), _lib.strides4(k.stride()), d ** -0.5, 0, 1, stream))


def test_single_sweeps_take_the_two_kernels_where_nothing_orders_them():
    """While the stream of the last single sweep is being captured, nothing can be recorded behind what it was given before: a call on another
    stream then takes the two kernels (their bits, and a status of 0 whatever the scratch held), and the single sweep again afterwards."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    h, m, n, d = 64, 64, 8192, 128
    g = torch.Generator(device="cuda").manual_seed(9)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).half() for r in (m, n))
    floats = lib.fcr_lse_bytes(1, h, m, n, d) // 4
    ws, side_ws = (torch.empty(floats, device="cuda") for _ in range(2))
    out, side_out = (torch.empty(h, n, device="cuda") for _ in range(2))
    main, side = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    want = {}
    for option in (0, 1):
        lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, option)
        try:
            _decode_call(q, k, out, ws, main.cuda_stream)
            main.synchronize()
            want[option] = out.clone()
        finally:
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
    assert not torch.equal(want[0], want[1])
    _decode_call(q, k, out, ws, main.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    side_ws.fill_(-1.0)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=main, capture_error_mode="relaxed"):
        _decode_call(q, k, out, ws, main.cuda_stream)
        _decode_call(q, k, side_out, side_ws, side.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(side_out, want[0])
    assert lib.fcr_colreduce_status(side_ws.data_ptr(), _lib.DTYPE_F16, 1, h, m, n, d, side.cuda_stream) == 0
    _decode_call(q, k, side_out, side_ws, side.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(side_out, want[1])
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want[1])


def test_single_sweeps_on_the_streams_of_several_threads():
    """hipStreamPerThread is one handle for a stream of every thread: single sweeps that threads issue on theirs are kept apart, among
    themselves and from those on an ordinary stream, and every result is right."""
    import threading
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    per_thread = 2   # hipStreamPerThread
    h, m, n, d = 64, 64, 8192, 128
    g = torch.Generator(device="cuda").manual_seed(10)
    q, k = (torch.randn(1, h, r, d, device="cuda", generator=g).half() for r in (m, n))
    floats = lib.fcr_lse_bytes(1, h, m, n, d) // 4
    streams = [per_thread, per_thread, torch.cuda.Stream().cuda_stream]
    ws = [torch.empty(floats, device="cuda") for _ in range(4)]
    out = [torch.zeros(h, n, device="cuda") for _ in range(4)]
    _decode_call(q, k, out[3], ws[3], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    errors = []

    def run(i):
        try:
            for _ in range(6):
                _decode_call(q, k, out[i], ws[i], streams[i])
        except Exception as e:
            errors.append(e)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    assert all(torch.equal(x, out[3]) for x in out[:3])


def test_both_sweeps_report_a_wait_that_gave_up():
    """fcr_colreduce_ws_status says so after the call whose columns are NaN, and 0 after any other call on that workspace: the next one, one in two
    launches, one on a workspace whose word was never written, one without room for the word."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    h, m, d = 4, 1200, 128
    q, k = (x.cuda() for x in _inputs.randn_pair(1, h, m, m, d, seed=5, dtype=torch.float16))
    ws, out = torch.full((_lib_workspace(q, k),), -1.0, device="cuda"), torch.empty(h, m, device="cuda")
    least = lib.fcr_lse_bytes(1, h, m, m, d) // 4
    assert ws.numel() > least
    state = lambda w: lib.fcr_colreduce_ws_status(w.data_ptr(), 4 * w.numel(), _lib.DTYPE_F16, 1, h, m, m, d, torch.cuda.current_stream().cuda_stream)

    def call(w, causal, options=()):
        for option, value in options:
            lib.fcr_set_option(option, value)
        try:
            _ws_call(q, k, out, w, causal)
        finally:
            lib.fcr_set_option(_lib.OPT_WAIT_POLLS, 1 << 20)
            lib.fcr_set_option(_lib.OPT_SINGLE_SWEEP, 1)
        return state(w)
    no_polls, two_launches = [(_lib.OPT_WAIT_POLLS, 0)], [(_lib.OPT_SINGLE_SWEEP, 0)]
    assert call(ws, True, two_launches) == 0     # first of all: nothing else has cleared the word
    for after in ((True, ()), (True, two_launches), (False, ())):
        assert call(ws, True, no_polls) == -8 and out.isnan().any()
        assert call(ws, *after) == 0 and out.isfinite().all()
    assert call(ws[:least], True, no_polls) == 0 and out.isnan().any()
    assert lib.fcr_colreduce_ws_status(None, 1 << 20, 0, 1, 1, 8, 8, 64, None) == -1


@pytest.mark.parametrize("h,m,n,d,dtype,causal", [
    (300, 520, 900, 64, torch.float16, True), (250, 520, 1500, 128, torch.bfloat16, True), (64, 700, 1100, 256, torch.float16, True),
    (170, 700, 1400, 72, torch.float16, True), (128, 1000, 1530, 40, torch.bfloat16, True), (40, 1025, 1800, 200, torch.float16, True),
    (60, 1000, 1000, 80, torch.bfloat16, True), (62, 1000, 1030, 128, torch.float16, True), (27, 2240, 2240, 128, torch.float16, True),
    (155, 1538, 1538, 128, torch.bfloat16, True), (50, 1100, 1010, 96, torch.float16, True), (140, 560, 520, 160, torch.bfloat16, False),
    (250, 520, 1500, 104, torch.float16, False), (90, 1000, 900, 128, torch.bfloat16, False)])
def test_both_sweeps_share_a_launch(h, m, n, d, dtype, causal):
    """The same for calls whose sweeps share a launch by the library's own word (the workspace has room for its status), so that two launches are
    not compared with themselves: more keys than queries behind the mask, every pair of tile sizes, several rounds."""
    from flash_colreduce_amd import _lib
    lib = _lib.load()
    dt = {torch.float16: _lib.DTYPE_F16, torch.bfloat16: _lib.DTYPE_BF16}[dtype]
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:   # (the shapes are chosen for that)
        assert lib.fcr_workspace_bytes(dt, 1, h, m, n, d) > lib.fcr_lse_bytes(1, h, m, n, d)
    test_both_sweeps_in_one_launch(h, m, n, d, dtype, causal)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,m,n,d", [(1, 100, 29647, 64), (1, 2, 63379, 96), (2, 128, 20001, 128), (3, 33, 33000, 64), (1, 64, 40000, 128)])
def test_single_sweep_teams_of_one_to_three_pairs(h, m, n, d, causal):
    """Long caches of few pairs, whose teams stop growing at 64 members: the last of them with few keys, ragged chunks."""
    test_single_sweep_keys_dealt_evenly(h, m, n, d, causal)
