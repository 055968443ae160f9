"""Attention of any query and key count against the oracle: the 128-query kernel's edges (lengths around its blocks of
128 queries and 64 keys, ranges of keys merged in-kernel) and the few-queries kernel (rows per load, iterations and key
ranges that do not divide the cache).

Tolerance: the probabilities and the result are rounded to bf16 (2^-9 relative each, on both sides), so two correct
results differ by at most 4 · 2^-9 = 2^-7 normwise."""
import re

import numpy as np
import pytest

from helpers import oracle_outputs, run_pjrt
from oracle import stablehlo as sh
from ryft_amd import configs

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -7

EDGE = [dict(s=9, d=64), dict(s=63, d=64), dict(s=65, d=128), dict(s=127, d=128), dict(s=129, d=64), dict(s=300, d=128),
        dict(b=2, h=4, s=200, d=64), dict(s=100, sk=65, d=128, mask=None), dict(s=130, sk=1, d=64, mask=None),
        dict(s=128, sk=64 * 8 + 1, d=128, mask=None), dict(s=5, sk=1030, d=64, mask=None),
        # causal (key <= query) with keys that no query sees, and with queries past the last key
        dict(s=70, sk=200, d=64), dict(s=100, sk=1000, d=128), dict(s=200, sk=70, d=128), dict(s=300, sk=2, d=64)]
DECODE = [dict(s=1, sk=1, d=64, mask=None), dict(s=1, sk=127, d=128, mask=None), dict(s=1, sk=129, d=128, mask=None),
          dict(s=2, sk=1025, d=64, mask=None), dict(s=3, sk=2050, d=128, mask=None), dict(s=4, sk=255, d=64, mask=None),
          dict(s=4, d=128), dict(b=2, h=3, s=1, sk=3000, d=64, mask=None), dict(s=4, sk=2, d=64),
          dict(s=2, sk=9, d=128), dict(s=3, sk=1030, d=64)]


def _run(gpu_client, kw, kernel, edit=None):
    w = configs.c4_causal_attention(**{**dict(b=1, h=2), **kw})
    if edit:
        edit(w)
    outs, exe = run_pjrt(gpu_client, w.program, w.inputs)
    assert kernel in exe.describe_plan()
    again, _ = run_pjrt(gpu_client, w.program, w.inputs)
    assert np.array_equal(outs[0], again[0])
    (want, dt), = oracle_outputs(w.program, w.inputs)
    return sh.from_raw(outs[0], dt), want


@pytest.mark.parametrize("kernel,kw", [("attention_edge", k) for k in EDGE] + [("attention_decode", k) for k in DECODE])
def test_attention_lengths(gpu_client, kernel, kw):
    got, want = _run(gpu_client, kw, kernel)
    err = sh.rel_error(got, want)
    print(f"[attention] {kernel} {kw} error {err:.2e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("kernel,kw", [("attention_edge", dict(s=70, d=64)), ("attention_edge", dict(s=9, sk=65, d=128, mask=None)),
                                       ("attention_decode", dict(s=1, sk=65, d=64, mask=None))])
def test_attention_infinity_in_the_last_value_row(gpu_client, kernel, kw):
    """Rows that the kernels read past the last key must not reach the result: an infinity in the last value row stays
    an infinity where that key is visible."""
    def edit(w):
        w.inputs[2].data[..., -1, 0] = 0x7F80  # bf16 +inf
    got, want = _run(gpu_client, kw, kernel, edit)
    seen = np.isposinf(want[..., 0])  # (a masked infinity is 0 · inf = NaN in the oracle; the kernels skip the key)
    assert seen.any() and np.all(np.isposinf(got[..., 0][seen]))
    assert sh.rel_error(got[..., 1:], want[..., 1:]) <= TOL


@pytest.mark.parametrize("kernel,kw", [("attention_edge", dict(s=9, sk=65, d=64, mask=None)),
                                       ("attention_decode", dict(s=1, sk=600, d=64, mask=None))])
def test_attention_all_scores_minus_infinity(gpu_client, kernel, kw):
    def edit(w):
        w.inputs[0].data[...] = 0x3F80  # q = 1
        w.inputs[1].data[...] = 0xFF80  # k = -inf
    got, want = _run(gpu_client, kw, kernel, edit)
    assert np.all(np.isnan(want)) and np.all(np.isnan(got))


def _rewrite(w, heads=None, kv_heads=None, f32=False):
    """The program with operands handed over as [b, s, h, d] (`heads`: which of q, k, v), keys and values of fewer heads
    broadcast to all of them, or the f32 result of the second product."""
    types = [re.search(rf"%arg{i}: (tensor<\S+>)", w.program).group(1) for i in range(3)]
    body, ops = w.program, ""
    for i, (x, t) in enumerate(zip(w.inputs, types)):
        b, h, s, d = x.dims
        if heads and heads[i]:
            x.data = np.ascontiguousarray(x.data.transpose(0, 2, 1, 3))
            x.dims, op = (b, s, h, d), "transpose %arg{i}, dims = [0, 2, 1, 3]"
        elif kv_heads and i:
            x.data = np.ascontiguousarray(x.data[:, :kv_heads])
            x.dims, op = (b, kv_heads, s, d), "broadcast_in_dim %arg{i}, dims = [0, 1, 2, 3]"
        else:
            continue
        given = "tensor<" + "x".join(map(str, x.dims)) + "xbf16>"
        body = re.sub(rf"(?<!: )%arg{i}(?!:)", f"%in{i}", body).replace(f"%arg{i}: {t}", f"%arg{i}: {given}")
        ops += f"    %in{i} = stablehlo.{op.format(i=i)} : ({given}) -> {t}\n"
    body = body.replace(" {\n    %0", " {\n" + ops + "    %0", 1)
    if f32:
        body = re.sub(r"    %18 = .*\n", "", body).replace("return %18 : " + types[0], "return %17 : " + types[0].replace("bf16", "f32"))
        body = body.replace(f"-> {types[0]} {{", f"-> {types[0].replace('bf16', 'f32')} {{", 1)
    w.program = body


@pytest.mark.parametrize("kernel,kw", [("attention_edge", dict(b=2, h=4, s=130, d=64)),
                                       ("attention_edge", dict(b=2, h=4, s=100, sk=1000, d=128, mask=None)),
                                       ("attention_decode", dict(b=2, h=4, s=3, sk=700, d=128, mask=None))])
@pytest.mark.parametrize("edit", [dict(heads=(1, 1, 1)), dict(heads=(1, 0, 1)), dict(kv_heads=1), dict(f32=True)],
                         ids=["bshd", "q_and_v_bshd", "one_kv_head", "f32_result"])
def test_attention_operand_layouts(gpu_client, kernel, kw, edit):
    got, want = _run(gpu_client, kw, kernel, lambda w: _rewrite(w, **edit))
    err = sh.rel_error(got, want)
    print(f"[attention] {kernel} {kw} {edit} error {err:.2e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("nan", [0x7FC0, 0xFFC0])  # either sign: the block maximum is taken over integers
@pytest.mark.parametrize("kernel,kw,key", [("attention_edge", dict(s=150, d=64), 100),
                                           ("attention_edge", dict(s=9, sk=700, d=128, mask=None), 650),
                                           ("attention_decode", dict(s=4, d=128), 2),
                                           ("attention_decode", dict(s=1, sk=700, d=64, mask=None), 650)])
def test_attention_nan_score(gpu_client, kernel, kw, key, nan):
    """A NaN in one key row makes every query that sees the key NaN and no other."""
    def edit(w):
        w.inputs[1].data[0, 0, key, 5] = nan
    got, want = _run(gpu_client, kw, kernel, edit)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any() and not np.isnan(want).all()
    rest = ~np.isnan(want)
    assert np.max(np.abs(got[rest] - want[rest])) <= TOL * np.max(np.abs(want[rest]))
