"""Attention of any query and key count against the oracle: the 128-query kernel's edges (lengths around its blocks of
128 queries and 64 keys, ranges of keys merged in-kernel) and the few-queries kernel (rows per load, iterations and key
ranges that do not divide the cache).

Tolerance: the probabilities and the result are rounded to bf16 (2^-9 relative each, on both sides), so two correct
results differ by at most 4 · 2^-9 = 2^-7 normwise."""
import numpy as np
import pytest

from helpers import oracle_outputs, run_pjrt
from oracle import stablehlo as sh
from ryft_amd import configs

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -7

EDGE = [dict(s=9, d=64), dict(s=63, d=64), dict(s=65, d=128), dict(s=127, d=128), dict(s=129, d=64), dict(s=300, d=128),
        dict(b=2, h=4, s=200, d=64), dict(s=100, sk=65, d=128, mask=None), dict(s=130, sk=1, d=64, mask=None),
        dict(s=128, sk=64 * 8 + 1, d=128, mask=None), dict(s=5, sk=1030, d=64, mask=None)]
DECODE = [dict(s=1, sk=1, d=64, mask=None), dict(s=1, sk=127, d=128, mask=None), dict(s=1, sk=129, d=128, mask=None),
          dict(s=2, sk=1025, d=64, mask=None), dict(s=3, sk=2050, d=128, mask=None), dict(s=4, sk=255, d=64, mask=None),
          dict(s=4, d=128), dict(b=2, h=3, s=1, sk=3000, d=64, mask=None)]


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
