"""fdi4_decode_paged_noalloc with an automatic split count whose partials are
larger than the static array: fewer splits, the same result."""

import ctypes
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "int4-kv-cache-quantization-cuda-triton-pallas_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,rep,D,rows", [(1, 4, 1, 64, 600), (300, 32, 4, 256, 16000),
                                            (65, 4, 2, 128, 20000), (33, 8, 4, 256, 16000)])
def test_automatic_count_fits(B, H, rep, D, rows):
    """Counts that fit (1 and 10 splits), one that is cut to 1 (from 2) and one cut
    to several (13, 13.6 MB). All sequences read the same few pages, so that long
    tables need little memory; lengths differ."""
    import torch
    from flash_decode_int4 import capi, ops
    lib = capi.load()
    g = torch.Generator("cuda").manual_seed(B)
    P, cols = 8, -(-rows // 16)
    kp = torch.randint(0, 256, (P, H, 16, D // 2), device="cuda", generator=g, dtype=torch.uint8)
    v = torch.randn(P, H, 16, D, device="cuda", generator=g)
    G = -(-cols // 8)
    s = (torch.rand(1, H, 1, D, device="cuda", generator=g) * 0.1).expand(B, H, G, D)
    z = torch.zeros(1, H, 1, D, device="cuda").expand(B, H, G, D)
    pt = torch.randint(0, P, (1, cols), device="cuda", generator=g,
                       dtype=torch.int32).expand(B, cols)
    sl = torch.randint(1, 200, (B,), device="cuda", generator=g, dtype=torch.int32)
    sl[0] = rows
    q = torch.randn(B, H * rep, D, device="cuda", generator=g) / D ** 0.5
    out = torch.empty_like(q)
    cache = capi.PagedCache(
        k_pages=kp.data_ptr(), k_page_stride=kp.stride(0), k_head_stride=kp.stride(1),
        k_row_stride=kp.stride(2), v_pages=v.data_ptr(), v_dtype=capi.V_F32,
        v_page_stride=v.stride(0), v_head_stride=v.stride(1), v_row_stride=v.stride(2),
        k_scale=s.data_ptr(), k_zp=z.data_ptr(), s_head_stride=s.stride(1),
        page_table=pt.data_ptr(), seq_lens=sl.data_ptr(), num_kv_heads=H, head_dim=D,
        page_rows=16, pages_per_group=8, max_pages=cols, num_pages=P)
    capi.check(lib.fdi4_decode_paged_noalloc(
        q.data_ptr(), B, H * rep, q.stride(0), q.stride(1), ctypes.byref(cache), out.data_ptr(),
        out.stride(0), out.stride(1), 0, torch.cuda.current_stream().cuda_stream), "noalloc")
    ref = ops.flash_decode_paged(q, kp, v, s, z, pt, sl, 128, num_splits=1)
    # The same float32 sums with other splits.
    assert (out - ref).abs().max().item() < 5e-6
