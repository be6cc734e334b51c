"""The decode's split count over shapes (host arithmetic, no GPU): bounded, and
every split holds chunks, enough for each wave of its workgroup."""

import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "int4-kv-cache-quantization-cuda-triton-pallas_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from flash_decode_int4 import capi  # noqa: E402


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("v_dtype", [capi.V_F32, capi.V_F16, capi.V_BF16])
@pytest.mark.parametrize("kv_heads,rep", [(1, 1), (8, 1), (32, 1), (2, 2), (8, 4), (4, 8), (3, 3),
                                          (1, 32)])
def test_split_count(head_dim, v_dtype, kv_heads, rep):
    lib = capi.load()
    hq = kv_heads * rep
    for batch in (1, 3, 17, 48, 300):
        for rows in (1, 16, 250, 2048, 16000, 200000):
            for page_rows in (1, 16, 256):
                pages = -(-rows // page_rows)
                cache = capi.PagedCache(max_pages=pages, page_rows=page_rows,
                                        num_kv_heads=kv_heads, head_dim=head_dim,
                                        v_dtype=v_dtype, pages_per_group=max(1, 256 // page_rows))
                chunks = pages * -(-page_rows // 16)
                s = lib.fdi4_decode_num_splits(batch, hq, cache)
                assert 1 <= s <= 64
                if s == 1:
                    continue
                per_split = -(-chunks // s)
                assert -(-chunks // per_split) == s
                # A chunk for each wave with grouped heads (two or more a
                # workgroup), four without.
                grouped = rep % 2 == 0
                one_a_simd = (not grouped and head_dim == 128 and v_dtype == capi.V_F32
                              and batch * hq * 4 <= 2048)
                waves = 8 if chunks >= 32 and not one_a_simd else 4
                if grouped and head_dim == 256:
                    waves = 4
                assert per_split >= waves * (1 if grouped else 4)


@pytest.mark.parametrize("batch,heads,head_dim,rows", [(2, 16, 256, 5000), (5, 16, 256, 2000),
                                                       (1, 8, 128, 20000)])
def test_groups_longer_than_any_sequence(batch, heads, head_dim, rows):
    """One scale group over the whole sequence, however many pages it is said to
    have (their chunks do not fit 32 bits from 2^27 pages of 256 rows up)."""
    lib = capi.load()
    counts = set()
    for pages in (1 << 20, (1 << 28) + 1, (1 << 31) - 1):
        cache = capi.PagedCache(max_pages=-(-rows // 256), page_rows=256, num_kv_heads=heads,
                                head_dim=head_dim, v_dtype=capi.V_F32, pages_per_group=pages)
        counts.add(lib.fdi4_decode_num_splits(batch, heads, cache))
    assert len(counts) == 1
