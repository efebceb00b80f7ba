"""g4a_gemm16 / g4a_gemm16_ws / g4a_gemm16_geglu at the edges of every output tile the launch
plan can take (csrc/gemm_plan.hpp kTiles): ragged tokens and outputs, one k-stage, fewer stages than
the pipeline holds, grouped matrices whose last tiles are partly empty, and a split with the
smallest tiles. Products against float64 (on the GPU, the operands being f16 exactly):

    |got - f16(ref)| <= one f16 ulp of ref + K 2^-24 sum|a w|

the f32 accumulation bound in any order, plus the f16 rounding of a value that far off. The
gate/up form must equal g4a_gemm16 followed by g4a_geglu16, which divides, code for code.
"""
import numpy as np
import pytest
import torch

import slang_amd as sa
from slang_amd.decoder import geglu16

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(M, K, ns, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(M, K, device=DEV, generator=g).half()
    return a, [(0.05 * torch.randn(n, K, device=DEV, generator=g)).half() for n in ns]


def srq_of_f16(step):
    """[65536] f32: srq(f32(v), step) of the f16 v of each bit pattern, by an IEEE f32 division."""
    v = np.arange(65536, dtype=np.uint16).view(np.float16).astype(np.float32)
    s = np.float32(step)
    with np.errstate(all="ignore"):
        return torch.from_numpy(np.clip(np.rint(v / s), -128, 127).astype(np.float32) * s if step else v).to(DEV)


def close(got, a, w, what):
    ref = a.double() @ w.double().T
    mag = a.double().abs() @ w.double().abs().T
    r16 = ref.half().double()
    ulp = torch.clamp(2.0 ** (torch.floor(torch.log2(ref.abs().clamp_min(2.0 ** -14))) - 10), min=2.0 ** -24)
    bad = (got.double() - r16).abs() > ulp + a.shape[1] * 2.0 ** -24 * mag
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} products off"


# Which tile a shape runs on is the plan's choice: test_gemm_plan.py holds that these lists reach
# all of them, each with a ragged last tile.
SHAPES = [(2047, 64, (24576,)), (2040, 192, (12288, 12160)), (1000, 128, (24448,)), (2047, 128, (4096, 512, 512)),
          (1893, 192, (3072,)), (1893, 64, (2048, 384, 640)), (1024, 320, (2048, 512)), (513, 64, (4096,)),
          (1, 64, (128,)), (65, 448, (384, 128)), (63, 128, (24576,)),
          (1893, 320, (12288, 12160)), (4000, 320, (4096,)), (1893, 512, (4096, 512, 512)), (1893, 640, (2048, 512)),
          (1500, 640, (2048, 384, 640)), (513, 1536, (4096,)), (700, 1536, (2048, 384, 640)), (65, 2048, (384, 128)),
          (1, 2048, (128,)), (1, 128, (128,))]
SPLIT_SHAPES = [(77, 4096, (128, 384)), (1, 8192, (128,)), (1000, 12288, (1536,)), (130, 6144, (1536,)), (40, 1024, (128,)),
                (200, 1344, (256,)), (300, 2048, (1536,)), (1, 1536, (256,)), (700, 6144, (1536,)),
                (200, 16384, (2048, 256, 256)), (77, 16384, (384, 128)), (65, 12288, (1536,))]
GEGLU_SHAPES = [(2047, 64, 12288), (1000, 128, 12224), (1893, 192, 1536), (1024, 320, 1216), (65, 64, 64),
                (1893, 320, 12224), (300, 1088, 12224), (1893, 640, 1216), (1000, 1536, 1216), (65, 2048, 64), (65, 448, 64)]


@pytest.mark.parametrize("M,K,ns", SHAPES)
def test_every_tile_matches_float64(M, K, ns):
    print(f"gemm16 M {M} K {K} n {ns}", flush=True)
    a, ws = operands(M, K, ns, M + K)
    outs = [torch.full((M + 2, n), 7.0, device=DEV, dtype=torch.float16) for n in ns]
    sa.gemm16(a, [(w, o[:M], None) for w, o in zip(ws, outs)])
    for i, (w, o) in enumerate(zip(ws, outs)):
        close(o[:M], a, w, f"matrix {i}")
        assert (o[M:] == 7.0).all(), "stores past M"
    # the q path: srq of the same f16 products, exactly, at a power of two, steps that have f16 values
    # at their ties, and outside the range that the refined products take (0, 1e-14)
    q = torch.full((M + 2, ns[0]), 7.0, device=DEV)
    bits = outs[0][:M].view(torch.int16).int() & 0xFFFF
    for step in (0.03125, 7 / 256, 13 / 1024, 0.0, 1e-14):
        sa.gemm16(a, [(ws[0], q[:M], step)])
        assert torch.equal(q[:M], srq_of_f16(step)[bits]), f"step {step}"
        assert (q[M:] == 7.0).all(), "stores past M"


@pytest.mark.parametrize("step", [7 / 256, 13 / 1024, 41 / 2048, 0.0137, 0.3330001, 1e-6, 1e-14, 1e14, 0.0])
def test_q_path_of_every_f16_value(step):
    """Every finite f16 value as a product of the q path. The first steps put f16 values at ties that
    x (1 / step), rounded, takes to the wrong side 78, 22 and 8 times."""
    print(f"q path every f16 step {step}", flush=True)
    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.float16)
    v = torch.where(torch.isfinite(v), v, torch.zeros(())).half().to(DEV)
    q = torch.empty(64, 1024, device=DEV)
    sa.gemm16(torch.eye(64, device=DEV).half(), [(v.view(1024, 64), q, step)])
    assert torch.equal(q.T, srq_of_f16(step)[v.view(torch.int16).int() & 0xFFFF].view(1024, 64))


@pytest.mark.parametrize("M,K,ns", SPLIT_SHAPES)
def test_split_tiles_match_float64_and_repeat(M, K, ns):
    print(f"gemm16 split M {M} K {K} n {ns}", flush=True)
    a, ws = operands(M, K, ns, M + K)
    outs = [torch.full((M + 2, n), 7.0, device=DEV, dtype=torch.float16) for n in ns]
    mats = [(w, o[:M], None) for w, o in zip(ws, outs)]
    gws = sa.GemmWorkspace()
    gws.get(sa.gemm16_ws_bytes(M, K, ns))
    parts = gws.buf[sa._lib.GEMM_TICKET_BYTES:].fill_(0xFF)  # stale partials are NaN and must not be read
    sa.gemm16(a, mats, gws)
    assert (parts != 0xFF).any(), "this product should split K"
    first = [o.clone() for o in outs]
    sa.gemm16(a, mats, gws)
    for i, (w, o, f) in enumerate(zip(ws, outs, first)):
        assert torch.equal(o, f), "a repeat call differs"
        close(o[:M], a, w, f"matrix {i}")
        assert (o[M:] == 7.0).all(), "stores past M"
    assert not gws.buf[:sa._lib.GEMM_TICKET_BYTES].any(), "tickets left non-zero"


def gelu_table(step):
    v = (np.arange(256) - 128).astype(np.float64) * step
    return torch.from_numpy((0.5 * v * (1 + np.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))).astype(np.float32)).to(DEV)


def geglu_pair(a, wg, wu, gq, uq, oq, lut):
    M, n = a.shape[0], wg.shape[0]
    out = torch.full((M + 2, n), 7.0, device=DEV, dtype=torch.float16)
    sa.gemm16_geglu(a, wg, wu, gq, uq, oq, out=out[:M], gelu_lut=lut)
    g, u = (torch.empty(M, n, device=DEV, dtype=torch.float16) for _ in range(2))
    for w, o in ((wg, g), (wu, u)):
        pad = torch.zeros(-n % 128, a.shape[1], device=DEV, dtype=torch.float16)
        full = torch.empty(M, n + len(pad), device=DEV, dtype=torch.float16)
        sa.gemm16(a, [(torch.cat([w, pad]), full, None)])
        o.copy_(full[:, :n])
    assert (out[M:] == 7.0).all(), "stores past M"
    return out[:M], geglu16(g, u, gq, uq, oq, gelu_lut=lut)


@pytest.mark.parametrize("M,K,n", GEGLU_SHAPES)
@pytest.mark.parametrize("table", [True, False])
def test_geglu_tiles_equal_the_divided_form(M, K, n, table):
    print(f"gemm16_geglu M {M} K {K} n {n} table {table}", flush=True)
    a, (wg, wu) = operands(M, K, (n, n), M + n)
    got, want = geglu_pair(a, wg, wu, 0.013, 0.021, 0.0073, gelu_table(0.013) if table else None)
    assert torch.equal(got, want), f"{int((got != want).sum())} codes differ"


@pytest.mark.parametrize("step", [0.02, 0.0137, 0.3330001, 1e-6, 1e-14, 1e14])
@pytest.mark.parametrize("scale", [1.0, 2.0])
def test_geglu_codes_of_every_f16_value(step, scale):
    """Every finite f16 value as a gate and as an up product (scale 2: the largest overflow to
    f16 infinities), at steps the epilogue quantises by refined products and, at the two last,
    by division: the codes equal the divided form's."""
    print(f"geglu every f16 step {step} scale {scale}", flush=True)
    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.float16)
    v = torch.where(torch.isfinite(v), v, torch.zeros(())).half().to(DEV)
    a = (scale * torch.eye(64, device=DEV)).half()
    wg, wu = v.view(1024, 64), v.view(1024, 64).flip(0).contiguous()
    lut = gelu_table(0.02) + 0.25 * torch.sign(gelu_table(0.02))
    for w1, w2, steps in ((wg, wu, (step, 0.02, 0.05)), (wu, wg, (0.02, step, 0.05)), (wg, wg, (0.02, 0.02, step))):
        got, want = geglu_pair(a, w1, w2, *steps, lut)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), f"{int((got != want).sum())} codes differ"
