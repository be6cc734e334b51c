"""The split merge around its rounds of eight: any split count, splits that hold
no rows, and values of empty splits that are never read."""

import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "int4-kv-cache-quantization-cuda-triton-pallas_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("splits", [1, 2, 7, 8, 9, 16, 17, 64])
def test_merge_of_given_partials(D, splits):
    """Partials of known maxima, sums and values against float64; every third
    split is empty (maximum -inf) and holds NaN values, one head has no rows."""
    import torch
    from flash_decode_int4._lib import load_binding
    C = load_binding()
    B, H = 2, 3
    g = torch.Generator("cuda").manual_seed(D + splits)
    n = B * H * splits
    acc = torch.randn(B, H, splits, D, device="cuda", generator=g)
    m = torch.randn(B, H, splits, device="cuda", generator=g).double() * 5
    l = torch.rand(B, H, splits, device="cuda", generator=g).double() + 0.5
    l = l.float().double()
    empty = torch.zeros(B, H, splits, dtype=torch.bool, device="cuda")
    empty[:, :, 1::3] = True
    empty[1, 2] = True
    m[empty] = -float("inf")
    l[empty] = 0.0
    acc[empty] = float("nan")
    buf = torch.zeros(int(C.decode_partials_bytes(B, H, D, splits)), dtype=torch.uint8,
                      device="cuda")
    buf[:n * D * 4].view(torch.float32).copy_(acc.flatten())
    off = (n * D * 4 + 255) // 256 * 256
    buf[off:off + n * 16].view(torch.float64).copy_(torch.stack([m, l], -1).flatten())
    out = C.merge_splits(buf, B, H, D, splits)
    w = torch.where(empty, 0.0, torch.exp(m - m.amax(-1, keepdim=True).clamp(min=-1e300)))
    want = (w[..., None] * torch.nan_to_num(acc.double())).sum(2)
    want = want / (w * l).sum(-1, keepdim=True).clamp(min=1e-10)
    # Each weight is a hardware exponential (1 ulp, argument rounded to 2^-24 of at
    # most 60); sums of at most 64 float32 terms.
    assert torch.equal(out[1, 2], torch.zeros_like(out[1, 2]))
    assert (out - want).abs().max().item() < 2e-5 * want.abs().max().item()


@pytest.mark.parametrize("D", [64, 128, 256])
def test_merge_of_partials_at_any_alignment(D):
    """fdi4_merge_splits takes partials that start at any element."""
    import torch
    from flash_decode_int4 import capi
    lib = capi.load()
    B, H, S = 2, 2, 5
    g = torch.Generator("cuda").manual_seed(D)
    acc = torch.randn(B * H * S * D + 3, device="cuda", generator=g)
    ml = torch.rand(B * H * S * 2 + 1, device="cuda", generator=g, dtype=torch.float64) + 0.5
    outs = []
    for a, m in ((acc[3:], ml[1:]), (acc[3:].clone(), ml[1:].clone())):
        out = torch.empty(B, H, D, device="cuda")
        capi.check(lib.fdi4_merge_splits(a.data_ptr(), m.data_ptr(), B, H, D, S, out.data_ptr(),
                                         out.stride(0), out.stride(1),
                                         torch.cuda.current_stream().cuda_stream), "merge")
        outs.append(out)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("bad", ["nan", "inf", "-inf"])
@pytest.mark.parametrize("splits", [1, 2, 9])
@pytest.mark.parametrize("rep,vector,vdtype", [(1, 0, "float32"), (4, 0, "float32"),
                                               (4, 0, "float16"), (4, 1, "float32")])
def test_non_finite_query(rep, vector, vdtype, splits, bad):
    """A NaN or infinite query element makes its head's output NaN in every kernel
    and at every split count (a split of NaN logits has the maximum of an empty
    one, -inf, but not its sum); the other heads keep theirs."""
    import torch
    from flash_decode_int4 import capi, ops
    B, H, D, T = 2, 2, 128, 700
    g = torch.Generator("cuda").manual_seed(splits)
    cols = -(-T // 16)
    pt = torch.randperm(B * cols, device="cuda", generator=g).to(torch.int32).view(B, cols)
    sl = torch.tensor([T, 130], dtype=torch.int32, device="cuda")
    kp = torch.zeros(B * cols, H, 16, D // 2, dtype=torch.uint8, device="cuda")
    s = torch.zeros(B, H, -(-T // 128), D, device="cuda")
    z = torch.zeros_like(s)
    ops.quantize_int4_paged(torch.randn(B, H, T, D, device="cuda", generator=g), sl, pt, kp, s, z)
    v = torch.randn(B * cols, H, 16, D, device="cuda", generator=g).to(getattr(torch, vdtype))
    q = torch.randn(B, H * rep, D, device="cuda", generator=g) * (2.0 / D ** 0.5)
    qb = q.clone()
    qb[0, 1, 3] = float(bad)
    qb[1, 0, D - 1] = float(bad)
    with capi.tuning(decode_vector_only=vector):
        good = ops.flash_decode_paged(q, kp, v, s, z, pt, sl, num_splits=splits)
        out = ops.flash_decode_paged(qb, kp, v, s, z, pt, sl, num_splits=splits)
    hit = torch.zeros(B, H * rep, dtype=torch.bool, device="cuda")
    hit[0, 1] = hit[1, 0] = True
    assert torch.isnan(out[hit]).all()
    # The same sums, or (float16) those of the float32 products: 700 terms.
    assert (out[~hit] - good[~hit]).abs().max().item() < 2e-6
