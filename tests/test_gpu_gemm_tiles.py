"""The edge GEMM tiles (256×256 down to 32×128) and their K ranges against the oracle, at the sizes where they can go
wrong: one row, one past and one short of a tile, k tails of one vector, ranges of unequal length, both layouts of
each operand, dual GEMMs finished from partial sums.

Tolerances: a sum of n products in f32, in any order, is off by at most n·2^-23 of the sum of their magnitudes |A|·|B| (each
addition rounds or truncates; products of 16- and 8-bit values are exact), and a bf16 result by 2^-8 of itself on both
sides: every element is held to that bound. The fp8 instruction adds 64 products at a time, aligned to the largest of
them and cut there (measured: off by 2^-16.5 of |A|·|B| at 77 products): cut at 2^-19 of the largest, the 64 lose at most
2^-13 of it. Integers exactly."""
import re

import numpy as np
import pytest

from edge_programs import dot
from helpers import check, oracle_outputs, run_pjrt
from oracle import stablehlo as sh
from ryft_amd import configs, pjrt

pytestmark = pytest.mark.gpu


def check_elements(got_raw, prog, ins, k, name):
    """Every element of a dot within its bound of the oracle's; returns the largest error relative to the bound."""
    (want, dt), = oracle_outputs(prog, ins)
    if dt not in sh.FLOAT:
        return check(got_raw, (want, dt), 0.0, name)
    def magnitude(x):
        bits = {1: 0x7F, 2: 0x7FFF, 4: 0x7FFFFFFF}[x.data.itemsize]
        u = x.data.view(f"u{x.data.itemsize}")
        return configs.HostInput((u & u.dtype.type(bits)).view(x.data.dtype), x.type, x.dims)
    (mags, _), = oracle_outputs(prog, [magnitude(x) for x in ins])
    got = sh.from_raw(got_raw, dt)
    assert got.shape == want.shape and np.isfinite(got).all(), name
    bound = k * 2.0 ** -23 * 1.01 * mags  # (1.01: the oracle's own rounding of the magnitudes and the products of roundings)
    if all(x.type == pjrt.BufferType.F8E4M3FN for x in ins):
        bound = bound + 2.0 ** -13 * mags
    if dt == "bf16":
        bound = bound + 2.0 ** -7 * 1.01 * np.abs(want)
    ratio = np.abs(got - want) / np.maximum(bound, 1e-300)
    worst = np.unravel_index(np.argmax(ratio), ratio.shape)
    assert ratio[worst] <= 1, f"{name}: element {worst} is {got[worst]}, not {want[worst]} (bound {bound[worst]:.2e})"
    return float(ratio[worst])

def _contracted(prog, ins):
    return ins[0].dims[int(re.search(r"contracting_dims = \[(\d+)\]", prog).group(1))]


CASES = [
    # (program, tile, split over K)
    (dot("bf16_one_row", (1, 4096), (4096, 1032), "bf16", "f32", [1], [0], seed=31), "32x128", True),
    (dot("bf16_33_rows", (33, 1096), (1096, 2056), "bf16", "f32", [1], [0], seed=32), None, False),
    (dot("bf16_64_tiles", (1000, 1000), (1000, 1000), "bf16", "f32", [1], [0], seed=33), "64x64", False),
    (dot("bf16_k_contiguous_both", (65, 2056), (1031, 2056), "bf16", "f32", [1], [1], seed=34), None, False),
    (dot("bf16_m_contiguous_tail", (1001, 136), (1001, 264), "bf16", "f32", [0], [0], seed=35), None, True),
    (dot("bf16_128_tiles", (2000, 520), (520, 4088), "bf16", "f32", [1], [0], seed=36), "128x128", False),
    (dot("bf16_256_tiles", (136, 4088), (136, 4088), "bf16", "f32", [0], [0], seed=37), "256x256", False),
    (dot("bf16_256_tiles_k_contiguous_b", (72, 4096), (4088, 72), "bf16", "f32", [0], [1], seed=38), "256x256", False),
    (dot("i8_one_row", (1, 4096), (4096, 2064), "i8", "i32", [1], [0], seed=39), "32x128", True),
    (dot("i8_rows_of_tiles", (129, 528), (528, 1040), "i8", "i32", [1], [0], seed=40), None, False),
    (dot("i8_k_contiguous_both", (250, 1040), (263, 1040), "i8", "i32", [1], [1], seed=41), None, False),
    (dot("i8_m_contiguous", (528, 272), (528, 144), "i8", "i32", [0], [0], seed=42), None, False),
    (dot("f32_ranges", (33, 1000), (1000, 264), "f32", "f32", [1], [0], seed=43), "64x64", True),
    (dot("f16_tail", (130, 264), (264, 136), "f16", "f32", [1], [0], seed=44), "128x128", False),
    (dot("fp8_tail", (130, 272), (272, 144), "f8E4M3FN", "f32", [1], [0], seed=45), "128x128", False),
    (dot("bf16_partial_chunks", (70, 200), (200, 1000 - 4), "bf16", "f32", [1], [0], out_convert="bf16", seed=48), None, False),
    (dot("bf16_result_of_ranges", (17, 4096), (4096, 520), "bf16", "f32", [1], [0], out_convert="bf16", seed=49), None, True),
    (dot("bf16_result_m_contiguous", (136, 4088), (136, 1032), "bf16", "f32", [0], [0], out_convert="bf16", seed=50), None, False),
    (dot("f16_result_tail", (130, 264), (264, 140), "f16", "f32", [1], [0], out_convert="bf16", seed=59), None, False),
    (dot("fp8_m_contiguous", (272, 144), (272, 144), "f8E4M3FN", "f32", [0], [0], seed=46), "128x128", False),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0][0] for c in CASES])
def test_gemm_tiles(gpu_client, case):
    (name, prog, ins), tile, split = case
    outs, exe = run_pjrt(gpu_client, prog, ins)
    plan = exe.describe_plan()
    assert "_edge_" in plan and (tile is None or f"tile={tile}" in plan), plan
    assert not split or "splits=" in plan, plan
    err = check_elements(outs[0], prog, ins, _contracted(prog, ins), name)
    again, _ = run_pjrt(gpu_client, prog, ins, executable=exe)
    assert (outs[0] == again[0]).all()
    print(f"[tiles] {name} {plan.splitlines()[-1].split('tile=')[1].split(' flops')[0]} error {err:.2f} of the bound", flush=True)


# operands whose rows the loads cannot read, copied into padded rows first: the copy keeps the layout of a
# free-contiguous operand and transposes a K-contiguous one, in blocks of 64 × 64 and vectors of 16 bytes
PACKED = [dot("bf16_both_transposed", (67, 1001), (129, 1001), "bf16", "f32", [1], [1], seed=51),
          dot("bf16_lhs_transposed_rhs_rows", (3, 65, 63), (3, 63, 71), "bf16", "f32", [2], [1], [0], [0], seed=52),
          dot("bf16_free_contiguous", (130, 67), (130, 201), "bf16", "f32", [0], [0], seed=53),
          dot("i8_odd", (17, 333), (333, 31), "i8", "i32", [1], [0], seed=54),
          dot("i8_odd_transposed", (65, 130), (129, 130), "i8", "i32", [1], [1], seed=55),
          dot("f32_odd", (65, 131), (131, 67), "f32", "f32", [1], [0], seed=56),
          dot("fp8_odd", (33, 77), (77, 19), "f8E4M3FN", "f32", [1], [0], seed=57),
          dot("bf16_f8_odd", (5, 72), (72, 999), "bf16", "f32", [1], [0], rhs_dt="f8E4M3FN", seed=58)]


@pytest.mark.parametrize("case", PACKED, ids=[c[0] for c in PACKED])
def test_unaligned_operands(gpu_client, case):
    name, prog, ins = case
    outs, exe = run_pjrt(gpu_client, prog, ins)
    assert "dot_operand_copy" in exe.describe_plan() and "generic" not in exe.describe_plan()
    check_elements(outs[0], prog, ins, _contracted(prog, ins), name)


@pytest.mark.parametrize("kw", [dict(m=1, d=1024, f=2048), dict(m=16, d=2048, f=1040), dict(m=33, d=1040, f=2048),
                                dict(m=77, d=1280, f=2048), dict(m=130, d=512, f=528)])
def test_swiglu_of_few_rows(gpu_client, kw):
    # the dual gate / up GEMM and the down projection of a few rows: 32-row tiles, partial sums of both accumulators
    w = configs.c5_swiglu_fp8(**kw)
    outs, exe = run_pjrt(gpu_client, w.program, w.inputs)
    assert "gemm_bf16f8_mfma_dual_edge" in exe.describe_plan()
    # three bf16 roundings in a row (norm, SwiGLU product, result), on both sides
    err = check(outs[0], oracle_outputs(w.program, w.inputs)[0], 3 * 2.0 ** -8, str(kw))
    again, _ = run_pjrt(gpu_client, w.program, w.inputs, executable=exe)
    assert (outs[0] == again[0]).all()
    print(f"[tiles] swiglu {kw} error {err:.2e}", flush=True)


def test_infinities_past_the_last_k_stay_out(gpu_client):
    """A partial last k-tile reads the last valid k again and zeroes it: an infinity there is multiplied once, not by
    the zeros of the padding (0 · inf would turn the result into NaN)."""
    for spec in (((9, 72), (72, 24), [1], [0]), ((72, 16), (72, 24), [0], [0]), ((9, 72), (25, 72), [1], [1])):
        name, prog, ins = dot("inf_tail", spec[0], spec[1], "bf16", "f32", spec[2], spec[3], seed=47)
        last = [slice(None)] * 2
        last[spec[3][0]] = -1
        ins[1].data[tuple(last)] = 0x7F80  # +inf at k = 71
        outs, exe = run_pjrt(gpu_client, prog, ins)
        (want, dt), = oracle_outputs(prog, ins)
        got = sh.from_raw(outs[0], dt)
        assert np.isinf(want).all() and (got == want).all()


@pytest.mark.parametrize("dt,out", [("bf16", "f32"), ("i8", "i32"), ("f32", "f32")])
def test_empty_contraction(gpu_client, dt, out):
    name, prog, ins = dot("k0", (16, 0), (0, 24), dt, out, [1], [0])
    outs, exe = run_pjrt(gpu_client, prog, ins)
    assert "gemm_generic" in exe.describe_plan() and outs[0].shape == (16, 24) and not outs[0].any()


def test_timings_name_the_tile_that_ran(gpu_client):
    for spec, label in (((1000, 1000, 1000), "gemm_bf16_mfma_edge_64x64"), ((1, 4096, 1032), "gemm_bf16_mfma_edge_32x128_splitk16")):
        m, k, n = spec
        name, prog, ins = dot("timed", (m, k), (k, n), "bf16", "f32", [1], [0], seed=60)
        _, exe = run_pjrt(gpu_client, prog, ins)
        gpu_client.set_kernel_timing(True)
        run_pjrt(gpu_client, prog, ins, executable=exe)
        timing = gpu_client.kernel_timing()
        gpu_client.set_kernel_timing(False)
        assert list(timing) == [label], timing


def test_operand_of_more_chunks_than_32_bits_count(gpu_client):
    """34.4 GB of int8 whose rows the loads cannot read: the copy indexes its 2^31 + 2^20 vectors of 16 bytes in 64 bits.
    The operand, (7k + 3f) mod 64, is computed on the device; one-hot rows pick its first, middle and last rows."""
    K, F = 1 << 20, 32769
    t = lambda e: f"tensor<{K}x{F}x{e}>"
    src = f"""module {{
  func.func @main() -> {t("i8")} {{
    %0 = stablehlo.iota dim = 0 : {t("i32")}
    %1 = stablehlo.iota dim = 1 : {t("i32")}
    %c = stablehlo.constant dense<7> : {t("i32")}
    %d = stablehlo.constant dense<3> : {t("i32")}
    %m = stablehlo.constant dense<63> : {t("i32")}
    %2 = stablehlo.multiply %0, %c : {t("i32")}
    %3 = stablehlo.multiply %1, %d : {t("i32")}
    %4 = stablehlo.add %2, %3 : {t("i32")}
    %5 = stablehlo.and %4, %m : {t("i32")}
    %6 = stablehlo.convert %5 : ({t("i32")}) -> {t("i8")}
    return %6 : {t("i8")}
  }}
}}"""
    made = gpu_client.compile(pjrt.Program.mlir(src)).execute([[]])[0]
    made.done.await_()
    rows = [0, 1, K // 2, K - 2, K - 1]
    a = np.zeros((len(rows), K), np.int8)
    a[np.arange(len(rows)), rows] = 1
    lt, ot = f"tensor<{len(rows)}x{K}xi8>", f"tensor<{len(rows)}x{F}xi32>"
    exe = gpu_client.compile(pjrt.Program.mlir(f"""module {{
  func.func @main(%arg0: {lt}, %arg1: {t("i8")}) -> {ot} {{
    %0 = stablehlo.dot_general %arg0, %arg1, contracting_dims = [1] x [0] : ({lt}, {t("i8")}) -> {ot}
    return %0 : {ot}
  }}
}}"""))
    assert "dot_operand_copy" in exe.describe_plan() and "gemm_i8_mfma_edge" in exe.describe_plan(), exe.describe_plan()
    out = exe.execute([[gpu_client.buffer(a, pjrt.BufferType.S8, a.shape), made.outputs[0]]])[0]
    out.done.await_()
    want = (7 * np.array(rows)[:, None] + 3 * np.arange(F)) & 63
    assert np.array_equal(out.outputs[0].to_numpy(), want)
