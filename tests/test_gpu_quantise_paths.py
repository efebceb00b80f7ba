"""The row tail's refined products (csrc/prefill_stack.hip with_quotient, csrc/common.hpp
srq_index) against the divisions they stand for, where the two could part: rows whose norm is
zero, infinite or NaN, steps at and past the ends of the range that takes the products, and, bit
for bit, values at and beside the ties and rows whose sum of squares is exact in any order.
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


def bits16(v):
    return v.astype(np.float16).view(np.uint16)


def srq32(v, step):
    """f32: rint of an IEEE division, the product rounded once."""
    s = np.float32(step)
    with np.errstate(all="ignore"):
        return (np.fmin(np.fmax(np.rint(v / s), -128), 127).astype(np.float32) * s) if step else v


STEPS = [0.02, 0.0137, 0.3330001, 1e-6, 2.0 ** -40, 2.0 ** 40, 1e-14, 1e14, 0.0]


@pytest.mark.parametrize("step", STEPS)
def test_operand_codes_at_the_ties(step):
    """TAIL_SRQ without an addend, so no row sum enters: values at every tie of the step's grid and
    one ulp either side, past both ends, and whole steps. The operand equals the division's."""
    print(f"rows_tail ties step {step}", flush=True)
    s = np.float32(step or 0.02)
    tie = ((np.arange(-140, 141) + 0.5).astype(np.float32) * s).astype(np.float32)
    v = np.concatenate([tie, np.nextafter(tie, np.float32(np.inf)), np.nextafter(tie, np.float32(-np.inf)),
                        np.arange(-140, 141).astype(np.float32) * s, np.float32([0.0, -0.0, 1e30, -1e30, np.inf, -np.inf])])
    hid = np.resize(v, (3, 1536)).astype(np.float32)
    h = torch.from_numpy(hid.copy()).to(DEV)
    y = rows_tail(h, mode=_lib.TAIL_SRQ, q2=step).cpu().numpy()
    with np.errstate(over="ignore"):
        assert np.array_equal(y.view(np.uint16), bits16(srq32(hid, step)))


@pytest.mark.parametrize("n", [520, 1536, 4096])
@pytest.mark.parametrize("step", [0.02, 0.0137, 0.3330001, 1e-14])
def test_row_quotients_equal_the_divisions(n, step):
    """Rows of whole numbers up to 60, whose sums of squares every order gives exactly (60^2 4096 <
    2^24): the norm is the same f32 as here, so x / norm, the products behind it and the operand's
    codes have to be those of the divisions, bit for bit. First without an addend (the operand's
    norm), then with one on a zero residual (the addend's norm; no sum behind it that an fma
    could round otherwise)."""
    print(f"rows_tail quotients n {n} step {step}", flush=True)
    rng = np.random.default_rng(n)
    eps = np.float32(1e-6)
    x = rng.integers(-60, 61, (37, n)).astype(np.float32)
    w1, w2 = ((1 + 0.3 * rng.standard_normal(n)).astype(np.float32) for _ in range(2))
    t = lambda v: torch.from_numpy(v.copy()).to(DEV)  # noqa: E731
    norm = np.sqrt((x * x).sum(1, dtype=np.float64).astype(np.float32)[:, None] / np.float32(n) + eps)
    z = (x / norm) * w2
    for mode, want in ((_lib.TAIL_NORM, z), (_lib.TAIL_NORM16, z.astype(np.float16).astype(np.float32))):
        y = rows_tail(t(x), mode=mode, w2=t(w2), q2=step, eps=float(eps)).cpu().numpy()
        assert np.array_equal(y.view(np.uint16), bits16(srq32(want, step))), f"mode {mode}"
    h = torch.zeros(37, n, device=DEV)
    rows_tail(h, t(x.astype(np.float16)), x_q=1.0, w1=t(w1), mult=0.75, eps=float(eps))
    assert np.array_equal(h.cpu().numpy(), (x / norm) * w1 * np.float32(0.75))
