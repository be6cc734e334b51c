"""The calls whose time matters to a user of this framework, as measurable cases.

Each case is one call (or one short run of calls) through the public entry
points: the paged decode over every value type and head layout, the serving
step, the prefill of a sequence cache, the two key quantizers, and the
reference's shared-stream attention call. ``listed()`` gives the fixed cases,
``draw(rng)`` more of the same ranges.

Inputs are synthetic and made from the seed alone, on the GPU: keys and values
N(0, 1), queries N(0, 1) * 2 / sqrt(D) (the kernels apply no softmax scale, so
a caller scales the query; the logits then spread as a trained layer's do).
Sequence lengths belong to the case and not to the seed, so that a case's work
is a number.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "int4-kv-cache-quantization-cuda-triton-pallas_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from flash_decode_int4 import ops  # noqa: E402
from flash_decode_int4.vllm_integration import INT4PagedSequenceCache  # noqa: E402

_DT = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _decode(name, batch, kv_heads, q_heads, head_dim, tokens, ragged=False, values="float32",
            query="float32", page_rows=16, group_rows=128):
    return dict(name=name, kind="decode", batch=batch, kv_heads=kv_heads, q_heads=q_heads,
                head_dim=head_dim, tokens=tokens, ragged=ragged, values=values, query=query,
                page_rows=page_rows, group_rows=group_rows)


def _step(name, batch, kv_heads, q_heads, head_dim, tokens, steps, ragged=False,
          values="float32", query="float32"):
    return dict(name=name, kind="step", batch=batch, kv_heads=kv_heads, q_heads=q_heads,
                head_dim=head_dim, tokens=tokens, steps=steps, ragged=ragged, values=values,
                query=query, page_rows=16, group_rows=128)


def listed():
    return [
        # The smallest call: one short sequence, four heads (latency, launches).
        _decode("decode_small", 1, 4, 4, 64, 512),
        # The benchmark's headline: one query per head, float32 values.
        _decode("decode_mha_f32", 8, 32, 32, 128, 2048),
        # The same cache as a 16-bit model holds it (float16 values and queries).
        _decode("decode_mha_f16", 8, 32, 32, 128, 2048, values="float16", query="float16"),
        # A large batch of sequences of every length up to 8192 (continuous batching).
        _decode("decode_ragged_f32", 32, 32, 32, 128, 8192, ragged=True),
        # Grouped query heads over long contexts, bfloat16: a current chat model's layer.
        _decode("decode_gqa_bf16", 8, 8, 32, 128, 8192, values="bfloat16", query="bfloat16"),
        # The widest head, grouped, at an odd length.
        _decode("decode_gqa_d256_bf16", 4, 4, 16, 256, 4095, values="bfloat16",
                query="bfloat16"),
        # Sixteen tokens of a serving loop: append, attend, advance (one query per head).
        _step("step_mha_f32", 8, 32, 32, 128, 1984, 16),
        # The same with eight query heads per kv-head, 16-bit, ragged lengths.
        _step("step_gqa_f16", 16, 8, 64, 128, 4096, 16, ragged=True, values="float16",
              query="float16"),
        # Prompts entering the cache: keys quantized, values paged, open groups staged.
        dict(name="prefill_bf16", kind="prefill", batch=8, kv_heads=8, q_heads=8, head_dim=128,
             tokens=2048, ragged=True, values="bfloat16", query="bfloat16", page_rows=16,
             group_rows=128),
        # The grouped key quantizer alone at the headline's size.
        dict(name="quantize_paged", kind="quantize_paged", batch=8, kv_heads=32, q_heads=32,
             head_dim=128, tokens=2048, ragged=False, values="float32", query="float32",
             page_rows=16, group_rows=128),
        # The reference's own quantizer call: one scale group over all rows.
        dict(name="quantize_rows", kind="quantize_rows", rows=32768, channels=128),
        # The reference's own attention call: every query over one stream of pages.
        dict(name="shared_stream", kind="shared", batch=8, q_heads=32, head_dim=128, pages=8,
             page_rows=256, last_rows=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over the listed ranges (log-uniform, odd ones among
    them), every value type, head layout and page size in use."""
    most = max(work(c)["bytes"] for c in listed())
    while True:
        kind = rng.choice(["decode"] * 5 + ["step"] * 2 + ["prefill", "quantize_paged",
                                                           "quantize_rows", "shared"])
        if kind == "quantize_rows":
            case = dict(kind=kind, rows=_log_int(rng, 100, 40000),
                        channels=rng.choice([64, 128, 128, 256, 100, 1024]))
        elif kind == "shared":
            rows = rng.choice([16, 64, 256])
            case = dict(kind=kind, batch=_log_int(rng, 1, 16), q_heads=rng.choice([8, 16, 32]),
                        head_dim=rng.choice([64, 80, 128, 256]),
                        pages=_log_int(rng, 2, 4096 // rows), page_rows=rows,
                        last_rows=rng.randint(1, rows))
        else:
            kv = rng.choice([1, 2, 4, 8, 8, 16, 32])
            per = rng.choice([1, 1, 2, 4, 4, 8]) if kv <= 16 else 1
            values = rng.choice(["float32", "float16", "bfloat16"])
            case = dict(kind=kind, batch=_log_int(rng, 1, 48), kv_heads=kv, q_heads=kv * per,
                        head_dim=rng.choice([64, 128, 128, 256]),
                        tokens=_log_int(rng, 200, 16000), ragged=rng.random() < 0.5,
                        values=values, query=rng.choice([values, "float32"]), page_rows=16,
                        group_rows=128)
            if kind == "step":
                case["steps"] = 16
                case["tokens"] = min(case["tokens"], 6000)
            if kind in ("decode", "quantize_paged"):
                case["page_rows"] = rng.choice([16, 16, 16, 32, 8])
                case["group_rows"] = rng.choice([128, 128, 64, 256])
        if work(case)["bytes"] <= most / {"step": 2, "prefill": 16}.get(kind, 1):
            return case


def _lengths(case):
    """int64 [B] lengths before the call; a step's segment stays in one scale group."""
    B, T, G = case["batch"], case["tokens"], case["group_rows"]
    if case["ragged"]:
        rng = np.random.RandomState(B * 7919 + T)
        lens = rng.randint(max(1, T // 64), T + 1, size=B)
    else:
        lens = np.full(B, T)
    lens = lens.astype(np.int64)
    n = case.get("steps", 0)
    if n:
        off = lens % G
        lens -= np.maximum(off + n - G, 0)
    return lens


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _queries(g, case, *lead):
    D = case["head_dim"]
    q = torch.randn(*lead, case["q_heads"], D, generator=g, device="cuda") * (2.0 / math.sqrt(D))
    return q.to(_DT[case["query"]])


def _decode_inputs(case, seed):
    """Dense keys, paged values, query, random page table and lengths."""
    g = _gen(seed)
    B, H, D, R = case["batch"], case["kv_heads"], case["head_dim"], case["page_rows"]
    lens = _lengths(case)
    T = int(lens.max())
    pages = -(-lens // R)
    P, cols = int(pages.sum()), int(pages.max())
    perm = torch.randperm(P, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(B, cols, dtype=torch.int32, device="cuda")
    at = 0
    for b in range(B):
        n = int(pages[b])
        table[b, :n] = perm[at:at + n]
        at += n
    q = _queries(g, case, B)
    k = _randn(g, B, H, T, D)
    return dict(k=k, q=q, table=table, lens=torch.as_tensor(lens, dtype=torch.int32).cuda(),
                n=lens, P=P, T=T, g=g)


def _values(case, x):
    return _randn(x["g"], x["P"], case["kv_heads"], case["page_rows"], case["head_dim"],
                  dtype=_DT[case["values"]])


def _cache_inputs(case, seed):
    """A step's or a prefill's dense prompt, and the new tokens."""
    g = _gen(seed)
    B, H, D = case["batch"], case["kv_heads"], case["head_dim"]
    lens = _lengths(case)
    T = int(lens.max())
    vdt = _DT[case["values"]]
    x = dict(n=lens, T=T, k=_randn(g, B, H, T, D), v=_randn(g, B, H, T, D, dtype=vdt))
    n = case.get("steps", 0)
    if n:
        x["k_new"] = _randn(g, n, B, H, D)
        x["v_new"] = _randn(g, n, B, H, D, dtype=vdt)
        x["q"] = _queries(g, case, n, B)
    return x


def _shared_inputs(case, seed):
    """The reference benchmark's shape of input: NumPy pages of a shared stream."""
    rng = np.random.RandomState(seed % (2 ** 32))
    B, H, D, nb, R = (case["batch"], case["q_heads"], case["head_dim"], case["pages"],
                      case["page_rows"])
    q = (rng.randn(B, H, D) * (2.0 / math.sqrt(D))).astype(np.float32)
    kq, s, z, v = [], [], [], []
    for i in range(nb):
        rows = R if i < nb - 1 else case["last_rows"]
        k = rng.randn(rows, D).astype(np.float32)
        mn, mx = k.min(0), k.max(0)
        sc = np.maximum(mx - mn, np.float32(1e-8)) / np.float32(15)
        kq.append(np.clip(np.round((k - mn) / sc), 0, 15).astype(np.uint8))
        s.append(sc)
        z.append((-mn / sc).astype(np.float32))
        v.append(rng.randn(rows, D).astype(np.float32))
    return q, kq, s, z, v


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

def _paged_outputs(case, x):
    B, H, D, R, G = (case["batch"], case["kv_heads"], case["head_dim"], case["page_rows"],
                     case["group_rows"])
    groups = -(-x["table"].shape[1] * R // G)
    kp = torch.zeros(x["P"], H, R, D // 2, dtype=torch.uint8, device="cuda")
    s = torch.zeros(B, H, groups, D, device="cuda")
    return kp, s, torch.zeros_like(s)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "quantize_rows":
        return dict(kind=kind, kv=_randn(_gen(seed), case["rows"], case["channels"]))
    if kind == "shared":
        return dict(kind=kind, call=ops.prepare_flash_decode_hip(*_shared_inputs(case, seed)))
    if kind in ("decode", "quantize_paged"):
        x = _decode_inputs(case, seed)
        kp, s, z = _paged_outputs(case, x)
        st = dict(kind=kind, group_rows=case["group_rows"], kp=kp, s=s, z=z, table=x["table"],
                  lens=x["lens"])
        if kind == "quantize_paged":
            st["k"] = x["k"]
            return st
        ops.quantize_int4_paged(x["k"], x["lens"], x["table"], kp, s, z, case["group_rows"])
        st["q"] = x["q"]
        x["k"] = None
        st["v"] = _values(case, x)
        return st
    x = _cache_inputs(case, seed)
    n = case.get("steps", 0)
    R = case["page_rows"]
    cache = INT4PagedSequenceCache(
        int((-(-(x["n"] + n) // R)).sum()), case["kv_heads"], case["head_dim"], case["batch"],
        x["T"] + n, R, case["group_rows"], case["values"])
    st = dict(kind=kind, cache=cache)
    if kind == "prefill":
        st.update(k=x["k"], v=x["v"], lens=x["n"])
        return st
    cache.prefill(x["k"], x["v"], x["n"])
    cache.reserve(case["batch"], n)
    st.update(steps=n, batch=case["batch"], start=cache.seq_lens.clone(), k_new=x["k_new"],
              v_new=x["v_new"], q=x["q"])
    return st


def run(st):
    kind = st["kind"]
    if kind == "decode":
        return ops.flash_decode_paged(st["q"], st["kp"], st["v"], st["s"], st["z"], st["table"],
                                      st["lens"], st["group_rows"])
    if kind == "quantize_paged":
        ops.quantize_int4_paged(st["k"], st["lens"], st["table"], st["kp"], st["s"], st["z"],
                                st["group_rows"])
        return st["kp"], st["s"], st["z"]
    if kind == "quantize_rows":
        return ops.quantize_int4(st["kv"])
    if kind == "shared":
        return st["call"].run()
    cache = st["cache"]
    if kind == "prefill":
        cache.prefill(st["k"], st["v"], st["lens"])
        return dict(k_pages=cache.k_pages, v_pages=cache.v_pages, k_scale=cache.k_scale,
                    k_zp=cache.k_zp, table=cache.page_table, lens=cache.seq_lens,
                    stage=cache.k_stage)
    # A segment of a serving loop from the same prompt each time (a rejected
    # draft's tokens are taken back by setting the lengths): reserve, then steps.
    cache.seq_lens.copy_(st["start"])
    cache.reserve(st["batch"], st["steps"])
    out = [cache.step(st["k_new"][i], st["v_new"][i], st["q"][i]) for i in range(st["steps"])]
    return dict(out=out, k_pages=cache.k_pages, v_pages=cache.v_pages, k_scale=cache.k_scale,
                k_zp=cache.k_zp, lens=cache.seq_lens, stage=cache.k_stage)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far outputs may be off
# ---------------------------------------------------------------------------

def _size(dt):
    return 4 if dt == "float32" else 2


def _attend_bytes(case, lens):
    H, Hq, D, R, G = (case["kv_heads"], case["q_heads"], case["head_dim"], case["page_rows"],
                      case["group_rows"])
    n = 0
    for t in lens:
        t = int(t)
        n += H * (t * D // 2 + t * D * _size(case["values"]) + -(-t // G) * D * 8)
        n += -(-t // R) * 4 + 4
    return n + 2 * len(lens) * Hq * D * _size(case["query"])


def _quantize_bytes(case, lens):
    H, D, R, G = case["kv_heads"], case["head_dim"], case["page_rows"], case["group_rows"]
    return sum(H * (int(t) * D * 4 + int(t) * D // 2 + -(-int(t) // G) * D * 8)
               + -(-int(t) // R) * 4 for t in lens)


def work(case):
    kind = case["kind"]
    if kind == "quantize_rows":
        r, c = case["rows"], case["channels"]
        return dict(bytes=r * c * 5 + 8 * c, flops=6 * r * c)
    if kind == "shared":
        rows = (case["pages"] - 1) * case["page_rows"] + case["last_rows"]
        D, BH = case["head_dim"], case["batch"] * case["q_heads"]
        return dict(bytes=rows * (D // 2 + 4 * D) + case["pages"] * (8 * D + 4) + 8 * BH * D,
                    flops=4 * BH * rows * D)
    lens = _lengths(case)
    H, Hq, D = case["kv_heads"], case["q_heads"], case["head_dim"]
    if kind == "decode":
        return dict(bytes=_attend_bytes(case, lens), flops=4 * Hq * D * int(lens.sum()))
    if kind == "quantize_paged":
        return dict(bytes=_quantize_bytes(case, lens), flops=6 * H * D * int(lens.sum()))
    if kind == "prefill":
        stage = int((lens % case["group_rows"]).sum()) * H * D * 4
        return dict(bytes=_quantize_bytes(case, lens) + stage
                    + 2 * int(lens.sum()) * H * D * _size(case["values"]),
                    flops=6 * H * D * int(lens.sum()))
    nbytes = flops = 0
    for i in range(case["steps"]):
        n = lens + i + 1
        open_rows = int((n - (n - 1) // case["group_rows"] * case["group_rows"]).sum())
        nbytes += _attend_bytes(case, n) + case["batch"] * H * D * (8 + 2 * _size(case["values"]))
        nbytes += open_rows * H * D * 4 + open_rows * H * D // 2 + case["batch"] * H * D * 8
        flops += 4 * Hq * D * int(n.sum())
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """Quantized keys, scales and moved values are bit-exact by contract. An
    attention output is a float32 sum, rounded once to the query's type: about
    four times its measured distance from exact() (up to 3.1e-7, 2.1e-4 and
    1.7e-3 for float32, float16 and bfloat16 outputs)."""
    if case["kind"] in ("prefill", "quantize_paged", "quantize_rows"):
        return "exact"
    return dict(rel={"float32": 1.5e-6, "float16": 8e-4, "bfloat16": 7e-3}[
        case.get("query", "float32")])


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _group_codes(k, G):
    """float32 keys [H, T, D] -> bins (float64), scale and zero-point (float32)
    [H, groups, D] of groups of G rows, one IEEE float32 operation each."""
    bins = torch.empty(k.shape, dtype=torch.float64, device=k.device)
    ss, zs = [], []
    fifteen = torch.full((), 15.0, device=k.device)
    for g0 in range(0, k.shape[1], G):
        x = k[:, g0:g0 + G]
        mn, mx = x.amin(1), x.amax(1)
        s = torch.clamp(mx - mn, min=1e-8) / fifteen
        bins[:, g0:g0 + G] = torch.round((x - mn[:, None]) / s[:, None]).clamp(0, 15).double()
        ss.append(s)
        zs.append(-mn / s)
    return bins, torch.stack(ss, 1), torch.stack(zs, 1)


def _scales64(k, G):
    """float64 scale and zero-point of every group of keys [H, T, D]."""
    ss, zs = [], []
    for g0 in range(0, k.shape[1], G):
        x = k[:, g0:g0 + G].double()
        mn, mx = x.amin(1), x.amax(1)
        s = torch.clamp(mx - mn, min=float(np.float32(1e-8))) / 15.0
        ss.append(s)
        zs.append(-mn / s)
    return torch.stack(ss, 1), torch.stack(zs, 1)


def _attend64(q, kd, v):
    """q [Hq, D], kd and v [H, T, D], all float64 -> [Hq, D]."""
    H = kd.shape[0]
    q = q.reshape(H, -1, q.shape[-1])
    w = torch.softmax(torch.bmm(q, kd.transpose(1, 2).contiguous()), dim=-1)
    return torch.bmm(w, v).reshape(-1, q.shape[-1])


def _dequant64(k, G):
    bins, s, z = _group_codes(k, G)
    T = k.shape[1]
    s = s.double().repeat_interleave(G, 1)[:, :T]
    z = z.double().repeat_interleave(G, 1)[:, :T]
    return (bins - z) * s


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize_rows":
        k = _randn(_gen(seed), case["rows"], case["channels"])
        s, z = _scales64(k[None], case["rows"])
        return None, s[0, 0], z[0, 0]
    if kind == "shared":
        q, kq, s, z, v = _shared_inputs(case, seed)
        k = np.concatenate([(a.astype(np.float64) - zz.astype(np.float64)) * ss.astype(np.float64)
                            for a, ss, zz in zip(kq, s, z)])
        lg = q.astype(np.float64) @ k.T
        w = np.exp(lg - lg.max(-1, keepdims=True))
        return (w / w.sum(-1, keepdims=True)) @ np.concatenate(v).astype(np.float64)
    G, R = case["group_rows"], case["page_rows"]
    B, H, D = case["batch"], case["kv_heads"], case["head_dim"]
    if kind in ("decode", "quantize_paged"):
        x = _decode_inputs(case, seed)
        if kind == "quantize_paged":
            _, s, z = _paged_outputs(case, x)
            s, z = s.double(), z.double()
            for b in range(B):
                n = int(x["n"][b])
                sb, zb = _scales64(x["k"][b, :, :n], G)
                s[b, :, :sb.shape[1]], z[b, :, :sb.shape[1]] = sb, zb
            return None, s, z
        v = _values(case, x)
        out = []
        for b in range(B):
            n = int(x["n"][b])
            pages = x["table"][b, :-(-n // R)].long()
            vb = v[pages].permute(1, 0, 2, 3).reshape(H, -1, D)[:, :n].double()
            out.append(_attend64(x["q"][b].double(), _dequant64(x["k"][b, :, :n], G), vb))
        return torch.stack(out)
    x = _cache_inputs(case, seed)
    if kind == "prefill":
        cols = -(-x["T"] // R)
        s = torch.zeros(B, H, -(-cols * R // G), D, dtype=torch.float64, device="cuda")
        z = torch.zeros_like(s)
        for b in range(B):
            n = int(x["n"][b])
            sb, zb = _scales64(x["k"][b, :, :n], G)
            s[b, :, :sb.shape[1]], z[b, :, :sb.shape[1]] = sb, zb
        return dict(k_pages=None, v_pages=None, k_scale=s, k_zp=z, table=None, lens=None,
                    stage=None)
    outs = [[] for _ in range(case["steps"])]
    for b in range(B):
        n = int(x["n"][b])
        k = torch.cat([x["k"][b, :, :n], x["k_new"][:, b].transpose(0, 1)], 1)
        v = torch.cat([x["v"][b, :, :n], x["v_new"][:, b].transpose(0, 1)], 1).double()
        o = n // G * G   # the closed groups stay; the open one is quantized again each step
        closed = _dequant64(k[:, :o], G) if o else v[:, :0]
        for i in range(case["steps"]):
            kd = torch.cat([closed, _dequant64(k[:, o:n + i + 1], G)], 1)
            outs[i].append(_attend64(x["q"][i, b].double(), kd, v[:, :n + i + 1]))
    return dict(out=[torch.stack(o) for o in outs], k_pages=None, v_pages=None, k_scale=None,
                k_zp=None, lens=None, stage=None)
