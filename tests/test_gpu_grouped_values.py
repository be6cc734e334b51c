"""The grouped decode's value products at their edges: infinite and NaN values
(the 16-bit forms split a probability into terms, an empty one of which times an
infinity is NaN where the probability's own product is infinite) and logits far
past the exponent range of a float32 maximum."""

import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "int4-kv-cache-quantization-cuda-triton-pallas_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

pytestmark = pytest.mark.gpu

SHAPES = [(64, 2, "float16"), (64, 8, "bfloat16"), (128, 2, "bfloat16"), (128, 4, "float16"),
          (128, 8, "float16"), (128, 8, "float32"), (256, 2, "bfloat16"), (256, 4, "float16"),
          (256, 4, "float32")]


def _inputs(D, rep, vdtype, lens):
    import torch
    from flash_decode_int4 import ops
    g = torch.Generator("cuda").manual_seed(D + rep)
    B, H, T = len(lens), 2, max(lens)
    cols = -(-T // 16)
    pt = torch.randperm(B * cols, device="cuda", generator=g).to(torch.int32).view(B, cols)
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    kp = torch.zeros(B * cols, H, 16, D // 2, dtype=torch.uint8, device="cuda")
    s = torch.zeros(B, H, -(-T // 128), D, device="cuda")
    z = torch.zeros_like(s)
    ops.quantize_int4_paged(torch.randn(B, H, T, D, device="cuda", generator=g), sl, pt, kp, s, z)
    v = torch.randn(B * cols, H, 16, D, device="cuda", generator=g).to(getattr(torch, vdtype))
    q = torch.randn(B, H * rep, D, device="cuda", generator=g) * (2.0 / D ** 0.5)
    return ops, q, kp, v, s, z, pt, sl


@pytest.mark.parametrize("D,rep,vdtype", SHAPES)
def test_infinite_and_nan_values(D, rep, vdtype):
    import torch
    from flash_decode_int4 import capi
    ops, q, kp, v, s, z, pt, sl = _inputs(D, rep, vdtype, [700, 133])
    v[pt[0, 3].item(), 0, 4, 7] = float("inf")
    v[pt[0, 20].item(), 1, 15, D - 1] = -float("inf")
    v[pt[0, 7].item(), 1, 0, 2] = float("nan")
    v[pt[1, 8].item(), 0, 4, 9] = float("inf")      # the last valid row of a partial chunk
    a = ops.flash_decode_paged(q, kp, v, s, z, pt, sl)
    with capi.tuning(decode_vector_only=1):
        b = ops.flash_decode_paged(q, kp, v, s, z, pt, sl)
    assert torch.isinf(b).any() and torch.isnan(b).any()
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.isinf(a), torch.isinf(b))
    assert torch.equal(a[torch.isinf(b)], b[torch.isinf(b)])
    # Both are float32 sums of at most 700 products: 2e-6 as between the two
    # kernels on finite values.
    f = torch.isfinite(b)
    assert (a[f] - b[f]).abs().max().item() < 2e-6


@pytest.mark.parametrize("D,rep,vdtype", SHAPES)
@pytest.mark.parametrize("scale", [1e5, 1e9, 1e18])
def test_huge_logits(D, rep, vdtype, scale):
    """Logits of 1e5 and beyond are far apart, so the softmax is one row: the
    grouped kernel picks the row the per-head kernel (double maxima) picks."""
    import torch
    from flash_decode_int4 import capi
    ops, q, kp, v, s, z, pt, sl = _inputs(D, rep, vdtype, [300, 17])
    a = ops.flash_decode_paged(q * scale, kp, v, s, z, pt, sl)
    with capi.tuning(decode_heads_per_wg=1):
        b = ops.flash_decode_paged(q * scale, kp, v, s, z, pt, sl)
    assert (a - b).abs().max().item() < 2e-6
