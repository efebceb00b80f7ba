"""Every form in which one sequence may be given to decode() -- q, the caches and out with or
without the sequence dimension, the length as a number, a list, an array or a device tensor --
gives the same bytes, and forms that do not match stay refused."""
import numpy as np
import pytest
import torch

import slang_amd as sa

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n", [1, 37, 40])
def test_one_sequence_forms(n):
    g = torch.Generator().manual_seed(n)
    q = torch.randn(8, 256, generator=g).to(DEV)
    k, v = (torch.randn(40, 2, 256, generator=g).to(DEV).half() for _ in range(2))
    cfg, ws = sa.AttnConfig(8, 2, 256), sa.Workspace(DEV)
    ref = sa.decode(q, k, v, np.array([n]), cfg, workspace=ws)
    assert ref.shape == q.shape
    for length in (n, [n], (n,), np.int32(n), torch.tensor([n], dtype=torch.int32, device=DEV)):
        for q1, k1, v1 in ((q, k, v), (q[None], k[None], v[None]), (q[None], k, v[None]), (q, k[None], v)):
            got = sa.decode(q1, k1, v1, length, cfg, workspace=ws, max_key_len=n)
            assert got.shape == q1.shape
            assert torch.equal(got.view_as(ref), ref)
    for out in (torch.empty(8, 256, device=DEV), torch.empty(1, 8, 256, device=DEV)):
        got = sa.decode(q, k, v, n, cfg, workspace=ws, out=out)
        assert got.shape == q.shape and got.data_ptr() == out.data_ptr() and torch.equal(got, ref)


def test_mismatched_forms_are_refused():
    q, k = torch.zeros(8, 256, device=DEV), torch.zeros(40, 2, 256, device=DEV, dtype=torch.float16)
    cfg, ws = sa.AttnConfig(8, 2, 256), sa.Workspace(DEV)
    for q1, k1, v1, length in ((q, k, k, 41), (q, k, k, 0), (q, k, k, [3, 3]), (q, k, k[:39], 3),
                               (q, k[:, :1], k[:, :1], 3), (q[:7], k, k, 3), (q, k, k.float(), 3),
                               (q[None].expand(2, 8, 256), k, k, [3, 3]), (q, k[::2], k[::2], 3)):
        with pytest.raises(ValueError):
            sa.decode(q1, k1, v1, length, cfg, workspace=ws)
