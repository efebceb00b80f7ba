"""The pieces that a prefill cuts long rows into (g4a_prefill's key split) against the same call
on the smallest workspace, which runs uncut. Sizes at the ends of the plan: one piece a block
beside blocks of two, shares that differ by a tile, the last block of one row, the largest number
of pieces, two and three rounds of workgroups, and a window. Both forms round P to f16 against
their own running maximum, so they agree within |d| <= 2e-3 + 1e-2 |ref|, the bound that either
meets against the oracle."""
import numpy as np
import pytest
import torch

import slang_amd as sa
from helpers import contract_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("S,start,hd,kvH,window,q_hilo", [
    (160, 0, 256, 2, 0, False),  # 3 tiles: the last block alone is cut, 2 tiles and 1
    (97, 0, 512, 1, 0, False),  # 4 tiles are one piece: not cut, as the next
    (97, 0, 256, 2, 0, False),
    (97, 160, 512, 1, 0, False),
    (300, 0, 512, 1, 0, False),
    (1500, 0, 256, 2, 0, False),  # one round of 4 pieces a block
    (1537, 0, 256, 2, 0, True),
    (1900, 1100, 512, 1, 0, False),  # two rounds, shares of 18 and 19 tiles
    (2047, 0, 512, 1, 0, True),
    (3001, 0, 256, 2, 0, False),  # the last block is one row past a full one
    (33, 4000, 256, 1, 0, False),  # few long blocks
    (601, 70, 512, 1, 512, False),
    (601, 0, 256, 2, 512, True),
])
def test_pieces_match_uncut(S, start, hd, kvH, window, q_hilo):
    g = torch.Generator().manual_seed(S + start)
    cfg = sa.AttnConfig(8, kvH, hd, window)
    q = torch.randn(S, 8, hd, generator=g).to(DEV)
    k, v = (torch.randn(start + S, kvH, hd, generator=g).to(DEV).half() for _ in range(2))
    k *= hd ** -0.5  # scores of order 1: every key counts
    cos, sin = (torch.as_tensor(x).to(DEV) for x in sa.rope_tables(np.arange(start, start + S), hd, 1e6))
    uncut_bytes = 0 if hd == 256 else -(-S * 8 * hd * 2 // 256) * 256 * (1 + q_hilo)  # q in f16
    cut = sa.prefill_ws_bytes(S, start, cfg, q_hilo=q_hilo) > uncut_bytes
    assert cut == (start + S > 97), "this call should be cut" if not cut else "this call should not be cut"
    ws = sa.Workspace(DEV)
    got = [sa.prefill(q, k, v, start, cfg, q_gain=torch.ones(hd, device=DEV), rope_cos=cos, rope_sin=sin,
                      out_dtype=torch.float32, q_hilo=q_hilo, workspace=ws, split=s).cpu().numpy()
           for s in (True, False)]
    contract_close(got[0], got[1], f"S={S}+{start} hd={hd} kvH={kvH} W={window}")


def attend64(q, k, v, start, window):
    """q [S][nH][hd] (normalised, rotated) at positions start.., causal, windowed, in float64."""
    S, nH, _ = q.shape
    key, at = torch.arange(start + S, device=DEV), start + torch.arange(S, device=DEV)[:, None]
    ok = (key[None] <= at) & ((key[None] > at - window) if window else True)
    outs = [torch.softmax((q[:, h] @ k[:, h * k.shape[1] // nH].double().T).masked_fill(~ok, -float("inf")), -1)
            @ v[:, h * k.shape[1] // nH].double() for h in range(nH)]
    return torch.stack(outs, 1)


@pytest.mark.parametrize("S,start,hd,kvH,window,q_hilo", [
    (1900, 1100, 256, 1, 512, False), (1900, 1100, 256, 1, 512, True), (1500, 0, 256, 2, 0, False), (1500, 0, 256, 2, 0, True),
    (1000, 1000, 256, 4, 0, False), (1000, 1000, 256, 8, 0, True), (1000, 1000, 512, 1, 0, False), (1001, 1000, 512, 1, 0, True),
    (1900, 1100, 512, 1, 512, False), (600, 3000, 512, 1, 512, True), (999, 1000, 512, 4, 0, False), (1000, 1000, 512, 8, 0, False)])
def test_few_pieces_lose_no_precision(S, start, hd, kvH, window, q_hilo):
    """Where the plan cuts long rows into few pieces, their partials hold 24 bits: the error of an
    f32 output against float64 is the uncut call's, within 10 % (P rounds to f16 against another
    running maximum). f16 partials of n pieces would add 2^-11 / sqrt(3 n) or so of the values,
    1.2 times the uncut error and more at these sizes."""
    print(f"pieces S {S} start {start} hd {hd} kvH {kvH} W {window} q_hilo {q_hilo}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(S + start)
    cfg = sa.AttnConfig(8, kvH, hd, window)
    q16_bytes = (1 + q_hilo) * S * 8 * hd * 2
    assert sa.prefill_ws_bytes(S, start, cfg, q_hilo=q_hilo) > 1.5 * q16_bytes, "this call should be cut"
    q = torch.randn(S, 8, hd, device=DEV, generator=g)
    k, v = (torch.randn(start + S, kvH, hd, device=DEV, generator=g).half() for _ in range(2))
    q64 = q.double() / torch.sqrt((q.double() ** 2).mean(-1, keepdim=True) + 1e-6)
    ref = attend64(q64 if q_hilo else q64.half().double(), k, v, start, window)
    err = [float((sa.prefill(q, k, v, start, cfg, q_gain=torch.ones(hd, device=DEV), out_dtype=torch.float32, q_hilo=q_hilo,
                             workspace=sa.Workspace(DEV), split=s).double() - ref).norm() / ref.norm()) for s in (True, False)]
    print(f"split {err[0]:.3e} uncut {err[1]:.3e}", flush=True)
    assert err[0] <= 1.1 * err[1], f"split {err[0]:.2e}, uncut {err[1]:.2e}"


def test_split_off_runs_uncut_on_a_grown_workspace():
    """split=False after a call that grew the workspace to the split's size gives the uncut call's
    values, bit for bit, not the split's."""
    g = torch.Generator(device=DEV).manual_seed(3)
    cfg = sa.AttnConfig(8, 1, 512)
    q = torch.randn(600, 8, 512, device=DEV, generator=g)
    k, v = (torch.randn(600, 1, 512, device=DEV, generator=g).half() for _ in range(2))
    ws = sa.Workspace(DEV)
    run = lambda w, s: sa.prefill(q, k, v, 0, cfg, q_gain=torch.ones(512, device=DEV), workspace=w, split=s)  # noqa: E731
    cut, uncut = run(ws, True), run(sa.Workspace(DEV), False)
    assert not torch.equal(cut, uncut)
    assert torch.equal(run(ws, False), uncut)
