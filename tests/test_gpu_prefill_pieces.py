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
    (97, 0, 256, 2, 0, False),  # 2 tiles: the longest block alone is cut
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
    ws = sa.Workspace(DEV)
    got = [sa.prefill(q, k, v, start, cfg, q_gain=torch.ones(hd, device=DEV), rope_cos=cos, rope_sin=sin,
                      out_dtype=torch.float32, q_hilo=q_hilo, workspace=ws, split=s).cpu().numpy()
           for s in (True, False)]
    contract_close(got[0], got[1], f"S={S}+{start} hd={hd} kvH={kvH} W={window}")
