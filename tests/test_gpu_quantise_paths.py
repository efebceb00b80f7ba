"""The row tail's refined products (csrc/prefill_stack.hip with_quotient, csrc/common.hpp
srq_index) against the divisions they stand for, where the two could part: rows whose norm is
zero, infinite or NaN, and steps at and past the ends of the range that takes the products.
"""
import numpy as np
import pytest
import torch

from slang_amd import _lib
from slang_amd.decoder import rows_tail

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("x_q,q2", [(0.0625, 0.03125), (0.0, 0.0), (0.07, 1e-20), (1e20, 0.05)])
def test_rows_tail_of_zero_infinite_and_ordinary_rows(x_q, q2):
    """Row 0: a zero residual and zero output (norm sqrt(eps)); row 1: an infinite output value;
    row 2: an infinite residual; row 3: NaN; the rest ordinary. Against the same arithmetic in
    torch float32: NaN and infinities in the same places, finite values within the f32 bound of
    the two row sums (1e-5 of the row's values) and the operand within one step of it."""
    print(f"rows_tail x_q {x_q} q2 {q2}", flush=True)
    rng = np.random.default_rng(5)
    n, eps = 1536, np.float32(1e-6)
    hid = rng.standard_normal((9, n)).astype(np.float32)
    x16 = (rng.standard_normal((9, n)) * 3).astype(np.float16)
    hid[0], x16[0] = 0, 0
    x16[1, 5] = np.inf
    hid[2, 7] = np.inf
    hid[3, 9] = np.nan
    w1, w2 = ((1 + 0.1 * rng.standard_normal(n)).astype(np.float32) for _ in range(2))
    t = lambda v: torch.from_numpy(v.copy()).to(DEV)  # noqa: E731
    h = t(hid)
    y = rows_tail(h, t(x16), x_q=x_q, w1=t(w1), mult=0.75, mode=_lib.TAIL_NORM, w2=t(w2), q2=q2)
    srq = lambda v, s: np.fmin(np.fmax(np.round(v / np.float32(s)), -128), 127) * np.float32(s) if s else v  # noqa: E731
    rms = lambda v: np.sqrt((v.astype(np.float64) ** 2).mean(1, keepdims=True).astype(np.float32) + eps)  # noqa: E731
    with np.errstate(all="ignore"):
        d = srq(x16.astype(np.float32), x_q)
        want = (hid + d / rms(d) * w1) * np.float32(0.75)
        got = h.cpu().numpy()
        z = srq(got / rms(got) * w2, q2)
    assert np.array_equal(np.isnan(want), np.isnan(got)) and np.array_equal(np.isinf(want), np.isinf(got))
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= 1e-5 * (1 + np.abs(want[ok]))).all()
    g = y.float().cpu().numpy()
    assert np.array_equal(np.isnan(z), np.isnan(g))
    ok = np.isfinite(z) & (np.abs(z) < 60000)
    assert (np.abs(g[ok] - z[ok]) <= q2 * 1.001 + 1e-3 * np.abs(z[ok]) + 1e-7).all()
