"""Performance cases of the full-attention library: the calls a serving program
makes for one Qwen3.5/3.6 attention layer, over the sizes it makes them with.

Kinds (each runs public entry points of ``supersonic_amd.kernel_ffi``):

* ``decode``       one ``fused_decode`` step of a batch (bf16 or fp8 cache, contiguous or paged)
* ``layer_kernel`` one decode layer as the persistent kernel (``decode_layer``)
* ``layer_step``   one decode layer as separate calls: projections, decode, output projection
* ``prefill``      one ``fused_prefill`` chunk, with or without a cached prefix
* ``proj``         the projections of a chunk alone (``qkv_proj`` and ``o_proj_residual``)
* ``layer_chunk``  one prefill layer: projections, ``fused_prefill``, output projection
* ``mixed``        one ``fused_mixed`` step: a prefill chunk and a decode batch together
* ``dropin``       the reference's prefill attention symbol, as its Rust crate calls it

Head shapes are those of the repository's tests and benchmark: 8/2 heads
(hidden 1024), 16/4 (hidden 4096) and 16/2 (hidden 2048), head size 256, 64
rotary dims.  Lengths go from 16 tokens to 32768 a sequence, batches from 1 to
32 sequences, chunks from 16 to 8192 tokens.
"""
from __future__ import annotations

import math
import random

import torch

from supersonic_amd import kernel_ffi as K

D, ROT, THETA, EPS = 256, 64, 1.0e7, 1e-6
PAGE = 64
HIDDEN = {(8, 2): 1024, (16, 4): 4096, (16, 2): 2048}
HEADS = sorted(HIDDEN)
DEV = "cuda:0"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a single chat on the smallest model: the launch-bound end of decode
        dict(name="decode_single", kind="decode", batch=1, hq=8, hkv=2, lo=2048, hi=2048, fp8=False, paged=False),
        # the benchmark's headline: 8 long contexts
        dict(name="decode_long", kind="decode", batch=8, hq=16, hkv=4, lo=32768, hi=32768, fp8=False, paged=False),
        # ragged batch over an fp8 cache
        dict(name="decode_fp8", kind="decode", batch=16, hq=16, hkv=4, lo=1024, hi=16384, fp8=True, paged=False),
        # a whole decode layer of the smallest model in one launch
        dict(name="layer_kernel", kind="layer_kernel", batch=1, hq=8, hkv=2, lo=2048, hi=2048, fp8=False,
             paged=False),
        # an ordinary serving step: 32 ragged sequences of one paged cache through one layer
        dict(name="layer_step", kind="layer_step", batch=32, hq=16, hkv=4, lo=200, hi=4000, fp8=False, paged=True,
             rope=False),
        # the next turn of a chat: a short chunk behind a long cached prefix
        dict(name="prefill_turn", kind="prefill", rows=333, start=7001, hq=16, hkv=2, fp8=False, paged=True),
        # the benchmark's long prompt
        dict(name="prefill_long", kind="prefill", rows=4096, start=0, hq=16, hkv=4, fp8=False, paged=False),
        # a later chunk of a long prompt over an fp8 cache
        dict(name="prefill_fp8", kind="prefill", rows=4096, start=4096, hq=16, hkv=4, fp8=True, paged=False),
        # an ordinary prompt through a whole layer
        dict(name="layer_prompt", kind="layer_chunk", rows=1000, start=0, hq=16, hkv=4, fp8=False, paged=False),
        # the reference's attention symbol on a medium prompt of the smallest model
        dict(name="dropin_prompt", kind="dropin", rows=700, start=0, hq=8, hkv=2, dtype="bf16"),
        # the projections of a full chunk
        dict(name="proj_chunk", kind="proj", rows=4096, hq=16, hkv=4),
        # chunked-prefill batching: a full chunk beside 32 ragged decodes of the same paged cache
        dict(name="mixed_step", kind="mixed", rows=8192, start=0, batch=32, hq=16, hkv=2, lo=512, hi=16384, fp8=False,
             paged=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        c = _draw(rng)
        if work(c)["flops"] <= 5e11:  # the largest listed case has 5.5e11
            return c


def _draw(rng):
    kind = rng.choices(["decode", "layer_kernel", "layer_step", "prefill", "proj", "layer_chunk", "mixed", "dropin"],
                       [6, 2, 5, 6, 4, 3, 2, 2])[0]
    hq, hkv = rng.choice(HEADS)
    c = dict(kind=kind, hq=hq, hkv=hkv)
    if kind in ("decode", "layer_kernel", "layer_step", "mixed"):
        c["batch"] = _log_int(rng, 1, 32)
        if kind == "layer_kernel":  # at most 4 query heads a kv head, batch * attention width <= 32768, batch <= 16
            hq, hkv = c["hq"], c["hkv"] = rng.choice([(8, 2), (16, 4)])
            c["batch"] = _log_int(rng, 1, min(16, 32768 // (hq * D)))
        # at most 262144 cached tokens in all
        c["hi"] = _log_int(rng, 16, min(32768, 262144 // c["batch"]))
        c["lo"] = c["hi"] if rng.random() < 0.3 else max(16, c["hi"] // rng.choice([2, 4, 16]))
        c["fp8"] = rng.random() < 0.35
        c["paged"] = rng.random() < 0.5
        if kind == "layer_step":
            c["rope"] = rng.random() < 0.4
            c["fp8"] = c["fp8"] and not c["rope"]  # qkv_proj_rope appends to bf16 caches
    if kind in ("prefill", "layer_chunk", "mixed", "dropin"):
        c["rows"] = _log_int(rng, 16, 8192)
        c["start"] = _log_int(rng, 16, 16384) if rng.random() < 0.6 else 0
        if kind == "dropin":
            c["dtype"] = rng.choice(["bf16", "f16"])
        elif kind != "mixed":
            c["fp8"] = rng.random() < 0.35
            c["paged"] = rng.random() < 0.5
    if kind == "mixed":
        c["paged"] = True
    if kind == "proj":
        c["rows"] = _log_int(rng, 1, 8192)
    return c


# ----------------------------------------------------------------- the inputs
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def randn(self, *shape, std=1.0, dtype=torch.bfloat16):
        t = torch.randn(*shape, generator=self.g, device=DEV, dtype=dtype)
        return t.mul_(std) if std != 1.0 else t


def _lens(case, seed):
    """Cached tokens of each sequence before the step (positions of the new tokens): the case sets the lengths (and with
    them the cache's size), the seed which sequence has which."""
    r = random.Random(case["batch"] * 1000003 + case["lo"] * 7919 + case["hi"])
    lens = [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    random.Random(int(seed) + 17).shuffle(lens)
    return lens


def _tables(n):
    inv = THETA ** (-torch.arange(0, ROT, 2, device=DEV, dtype=torch.float64) / ROT)
    ang = torch.arange(n, device=DEV, dtype=torch.float64)[:, None] * inv
    return ang.cos().float().bfloat16(), ang.sin().float().bfloat16()


def _to_fp8(x):
    """Rows of x as e4m3 codes with their absmax scales."""
    sc = (x.float().abs().amax(-1) / 448.0).clamp_min(1e-12)
    codes = (x.float() / sc[..., None]).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    return codes, sc


def _cache(g, lens, hkv, fp8, paged, seed):
    """A cache that holds lens[b] tokens of sequence b."""
    if paged:
        per = [(n + PAGE - 1) // PAGE for n in lens]
        pages = sum(per)
        order = list(range(pages))
        random.Random(int(seed) + 3).shuffle(order)
        table, at = [], 0
        for p in per:
            table.append(order[at:at + p] + [0] * (max(per) - p))
            at += p
        shape = (pages, hkv, PAGE, D)
        bt = torch.tensor(table, dtype=torch.int32, device=DEV)
    else:
        shape = (len(lens), hkv, max(lens), D)
        bt = None
    k, v = g.randn(*shape), g.randn(*shape)
    if not fp8:
        return K.KvCache(k, v, block_table=bt)
    (kc, ks), (vc, vs) = _to_fp8(k), _to_fp8(v)
    return K.KvCache(kc, vc, ks, vs, block_table=bt)


def _zeros(n):
    return torch.zeros(max(int(n), 1), dtype=torch.uint8, device=DEV)


def _bf16(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device=DEV)


def prepare(case, seed):
    g = _Gen(seed)
    kind, hq, hkv = case["kind"], case["hq"], case["hkv"]
    hid = HIDDEN[(hq, hkv)]
    fp8, paged = case.get("fp8", False), case.get("paged", False)
    s = dict(case=case, kind=kind, hq=hq, hkv=hkv, shape=dict(q_heads=hq, kv_heads=hkv, head_dim=D, rotary_dim=ROT))
    rows, start = case.get("rows", 0), case.get("start", 0)
    s["qw"], s["kw"] = g.randn(D, std=0.1), g.randn(D, std=0.1)

    if kind == "dropin":
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
        L = start + rows
        s["q"] = g.randn(1, hq, rows, D, dtype=dt)
        s["k"], s["v"] = g.randn(1, hkv, L, D, dtype=dt), g.randn(1, hkv, L, D, dtype=dt)
        s["out"] = torch.empty(1, hq, rows, D, dtype=torch.float32, device=DEV)
        return s

    decode = kind in ("decode", "layer_kernel", "layer_step", "mixed")
    lens = _lens(case, seed) if decode else []
    s["lens"] = lens
    held = [n + 1 for n in lens]
    if kind in ("prefill", "layer_chunk"):
        held = [start + rows]
    elif kind == "mixed":
        held = [start + rows] + held
    if held:
        s["cos"], s["sin"] = _tables(max(held))
        s["cache"] = _cache(g, held, hkv, fp8, paged, seed)
    if decode:
        B = len(lens)
        s["pos"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        s["max_len"] = max(lens) + 1
    n = rows if kind in ("prefill", "layer_chunk", "proj") else (len(lens) if decode else 0)

    # weights of the layer
    if kind in ("layer_kernel", "layer_step", "layer_chunk", "proj"):
        s["nw"] = g.randn(hid, std=0.1)
        s["wq"] = g.randn(hq * 2 * D, hid, std=hid ** -0.5)
        s["wk"], s["wv"] = g.randn(hkv * D, hid, std=hid ** -0.5), g.randn(hkv * D, hid, std=hid ** -0.5)
        s["wo"] = g.randn(hid, hq * D, std=(hq * D) ** -0.5)
        s["residual"] = g.randn(n, hid)  # what the layer before hands over
        s["hidden"] = torch.empty_like(s["residual"])
    if kind in ("layer_step", "layer_chunk", "proj"):
        s["q_proj"], s["k_new"], s["v_new"] = _bf16(n, hq * 2 * D), _bf16(n, hkv * D), _bf16(n, hkv * D)
        s["ws_o"] = _zeros(K.o_proj_workspace_size(n, hid, hq * D))
        if case.get("rope"):
            s["q"], s["gate"] = _bf16(n, hq * D), _bf16(n, hq * D)
            s["kv_lens"] = s["pos"] + 1
            s["ws_qkv"] = _zeros(K.qkv_proj_rope_workspace_size(n, hid, hq, hkv, D))
        else:
            s["ws_qkv"] = _zeros(K.qkv_proj_workspace_size(n, hid, hq * 2 * D, hkv * D))
    if kind in ("decode", "prefill", "mixed"):
        s["q_proj"] = g.randn(n, hq * 2 * D)
        s["k_new"], s["v_new"] = g.randn(n, hkv * D), g.randn(n, hkv * D)
    if kind == "proj":
        s["attn"] = g.randn(n, hq * D)
    elif kind != "layer_kernel":
        s["attn"] = _bf16(n, hq * D)

    if kind in ("decode", "layer_step"):
        s["ws"] = _zeros(K.decode_workspace_size(len(lens), hq, hkv, D, s["max_len"]))
    elif kind == "layer_kernel":
        s["ws"] = _zeros(K.decode_layer_workspace_size(len(lens), hid, hq, hkv, D, s["max_len"]))
    elif kind in ("prefill", "layer_chunk"):
        s["ws"] = _zeros(K.prefill_workspace_size(fp8, hkv, D, rows, start))
    elif kind == "mixed":
        cache = s["cache"]
        bt = cache.block_table
        mine = K.KvCache(cache.k, cache.v, cache.k_scale, cache.v_scale, bt[:1].contiguous())
        theirs = K.KvCache(cache.k, cache.v, cache.k_scale, cache.v_scale, bt[1:].contiguous())
        s["chunk"] = dict(q_proj=g.randn(rows, hq * 2 * D), k_new=g.randn(rows, hkv * D), v_new=g.randn(rows, hkv * D),
                          cache=mine, out=_bf16(rows, hq * D), chunk_start=start)
        s["decode"] = dict(q_proj=s["q_proj"], k_new=s["k_new"], v_new=s["v_new"], positions=s["pos"], cache=theirs,
                           out=s["attn"], max_kv_len=s["max_len"])
        s["ws"] = _zeros(K.mixed_workspace_size(fp8, hq, hkv, D, s["chunk"], s["decode"]))
    return s


# ------------------------------------------------------------------- one pass
def _kv(cache):
    r = dict(k=cache.k, v=cache.v)
    if cache.k_scale is not None:
        r.update(ks=cache.k_scale, vs=cache.v_scale)
    return r


def run(s):
    kind, shape = s["kind"], s["shape"]
    if kind == "decode":
        K.fused_decode(0, s["q_proj"], s["k_new"], s["v_new"], s["qw"], s["kw"], s["cos"], s["sin"], s["pos"],
                       s["cache"], s["attn"], max_kv_len=s["max_len"], eps=EPS, workspace=s["ws"], **shape)
        return dict(out=s["attn"], **_kv(s["cache"]))
    if kind == "prefill":
        K.fused_prefill(0, s["q_proj"], s["k_new"], s["v_new"], s["qw"], s["kw"], s["cos"], s["sin"], s["cache"],
                        s["attn"], chunk_start=s["case"]["start"], eps=EPS, workspace=s["ws"], **shape)
        return dict(out=s["attn"], **_kv(s["cache"]))
    if kind == "mixed":
        K.fused_mixed(0, s["qw"], s["kw"], s["cos"], s["sin"], chunk=s["chunk"], decode=s["decode"], eps=EPS,
                      workspace=s["ws"], **shape)
        return dict(chunk=s["chunk"]["out"], out=s["attn"], **_kv(s["cache"]))
    if kind == "dropin":
        q, k = s["q"], s["k"]
        K.full_attention_prefill(0, K.ScalarType.BF16 if q.dtype == torch.bfloat16 else K.ScalarType.F16, 1, s["hq"],
                                 s["hkv"], q.shape[2], k.shape[2], D, D ** -0.5, s["case"]["start"], q, k, s["v"],
                                 s["out"])
        return dict(out=s["out"])
    # the layers and the projections: the residual stream arrives in the layer's own buffer
    s["hidden"].copy_(s["residual"])
    if kind == "layer_kernel":
        K.decode_layer(0, s["hidden"], s["nw"], s["wq"], s["wk"], s["wv"], s["qw"], s["kw"], s["wo"], s["cos"],
                       s["sin"], s["pos"], s["cache"], s["ws"], max_kv_len=s["max_len"], eps=EPS, qk_eps=EPS, **shape)
        return dict(hidden=s["hidden"], **_kv(s["cache"]))
    if s["case"].get("rope"):
        K.qkv_proj_rope(0, s["hidden"], s["nw"], s["wq"], s["wk"], s["wv"], s["qw"], s["kw"], s["cos"], s["sin"],
                        s["pos"], s["q"], s["gate"], s["k_new"], s["v_new"], eps=EPS, qk_eps=EPS, cache=s["cache"],
                        workspace=s["ws_qkv"], **shape)
        K.decode_attend(0, s["q"], s["kv_lens"], s["cache"], s["attn"], q_heads=s["hq"], kv_heads=s["hkv"], head_dim=D,
                        max_kv_len=s["max_len"], gate=s["gate"], workspace=s["ws"])
    else:
        K.qkv_proj(0, s["hidden"], s["nw"], s["wq"], s["wk"], s["wv"], s["q_proj"], s["k_new"], s["v_new"], eps=EPS,
                   workspace=s["ws_qkv"])
        if kind == "layer_step":
            K.fused_decode(0, s["q_proj"], s["k_new"], s["v_new"], s["qw"], s["kw"], s["cos"], s["sin"], s["pos"],
                           s["cache"], s["attn"], max_kv_len=s["max_len"], eps=EPS, workspace=s["ws"], **shape)
        elif kind == "layer_chunk":
            K.fused_prefill(0, s["q_proj"], s["k_new"], s["v_new"], s["qw"], s["kw"], s["cos"], s["sin"], s["cache"],
                            s["attn"], chunk_start=s["case"]["start"], eps=EPS, workspace=s["ws"], **shape)
    K.o_proj_residual(0, s["attn"], s["wo"], s["hidden"], workspace=s["ws_o"])
    out = dict(hidden=s["hidden"], k_new=s["k_new"], v_new=s["v_new"])
    if kind == "proj":
        return dict(out, q_proj=s["q_proj"])
    return dict(out, attn=s["attn"], **_kv(s["cache"]))


# ------------------------------------------------------- what a pass must move
def work(case):
    kind, hq, hkv = case["kind"], case["hq"], case["hkv"]
    hid = HIDDEN[(hq, hkv)]
    rows, start = case.get("rows", 0), case.get("start", 0)
    fp8 = case.get("fp8", False)
    tok = 2 * hkv * ((D + 4) if fp8 else 2 * D)       # one cached token's K and V
    new = 2 * hkv * D * 2                              # one new token's K and V
    nbytes = flops = 0.0
    if kind == "dropin":
        L = start + rows
        return dict(bytes=float(rows * hq * D * 6 + L * new), flops=4.0 * hq * D * rows * (start + (rows + 1) / 2))
    if kind in ("decode", "layer_kernel", "layer_step", "mixed"):
        B, mean = case["batch"], (case["lo"] + case["hi"]) / 2.0
        flops += 4.0 * hq * D * B * (mean + 1)
        nbytes += B * (mean * tok + tok)
        nbytes += B * (hq * D * 2 * 3 + new)           # q and gate in, output out, new K and V in
    if kind in ("prefill", "layer_chunk", "mixed"):
        flops += 4.0 * hq * D * rows * (start + (rows + 1) / 2)
        nbytes += start * tok + rows * (tok + hq * D * 2 * 3 + new)
    if kind in ("layer_kernel", "layer_step", "layer_chunk", "proj"):
        n = rows if kind in ("layer_chunk", "proj") else case["batch"]
        nw = hid * (3 * hq * D + 2 * hkv * D)
        flops += 2.0 * n * nw
        nbytes += 2.0 * nw + n * hid * 4               # the weights, the residual stream in and out
        if kind == "proj":
            nbytes += n * (hq * D * 6 + new)           # q, gate, k, v out, the attention's output in
        else:                                          # inside a layer these need not reach memory
            nbytes -= n * (hq * D * 6 + new)
    return dict(bytes=float(nbytes), flops=float(flops))


def tolerance(case):
    """bf16 outputs of bf16 products with fp32 accumulation.  Two runs of one decode (its blocks are claimed in another
    order, so the bf16 weights round against another running maximum) differ by 0.0027 (largest value 0.014 of the rms),
    and every path is 0.002 to 0.005 from the 64-bit result.  ``differ``: e4m3 codes of values that a rounding error
    takes across a tie."""
    if case["kind"] == "proj":
        return dict(rel=4e-3, max=0.03)
    if case["kind"] == "dropin":  # fp32 outputs of 16-bit weights, 0.0012 from the 64-bit result
        return dict(rel=5e-3, max=0.04)
    return dict(rel=1e-2, max=0.08, differ=2e-3)


# --------------------------------------------------------- the result in 64 bits
def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + w.double())


def _rope(x, cos, sin):
    """x [n, heads, D] at positions whose table rows are cos, sin [n, ROT / 2]."""
    h = ROT // 2
    a, b, c, s = x[..., :h], x[..., h:ROT], cos.double()[:, None], sin.double()[:, None]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., ROT:]], -1)


def _rows64(cache, b, n):
    """The first n cached rows of sequence b: K and V [hkv, n, D]."""
    got = []
    for x, sc in ((cache.k, cache.k_scale), (cache.v, cache.v_scale)):
        if cache.block_table is None:
            x, sc = x[b, :, :n], None if sc is None else sc[b, :, :n]
        else:
            p = cache.block_table[b, :(n + PAGE - 1) // PAGE].long()
            x = x[p].transpose(0, 1).reshape(x.shape[1], -1, D)[:, :n]
            sc = None if sc is None else sc[p].transpose(0, 1).reshape(sc.shape[1], -1)[:, :n]
        x = x.double() if sc is None else x.contiguous().view(torch.float8_e4m3fn).float().double() * sc.double()[..., None]
        got.append(x)
    return got


def _put(cache, r, b, at, k, v):
    """Rows k, v [hkv, n, D] at tokens at .. of sequence b, in the 64-bit copies r of the cache."""
    n = k.shape[1]
    t = torch.arange(at, at + n, device=DEV)
    if cache.block_table is None:
        where = (torch.full_like(t, b), t)
    else:
        where = (cache.block_table[b].long()[t // PAGE], t % PAGE)
    if cache.k_scale is None:
        r["k"][where[0], :, where[1]] = k.transpose(0, 1)
        r["v"][where[0], :, where[1]] = v.transpose(0, 1)
    else:
        r["ks"][where[0], :, where[1]] = (k.abs().amax(-1) / 448.0).clamp_min(1e-12).transpose(0, 1)
        r["vs"][where[0], :, where[1]] = (v.abs().amax(-1) / 448.0).clamp_min(1e-12).transpose(0, 1)


def _attend(q, k, v, first):
    """Row i of q [n, hq, D] over the keys 0 .. first + i of k, v [hkv, L, D]."""
    n, hq = q.shape[:2]
    hkv, L = k.shape[:2]
    out = torch.empty_like(q)
    last = first + torch.arange(n, device=DEV)
    keys = torch.arange(L, device=DEV)
    step = max(1, (1 << 26) // max(L, 1))
    for h in range(hq):
        kh, vh = k[h // (hq // hkv)], v[h // (hq // hkv)]
        for i in range(0, n, step):
            sc = (q[i:i + step, h] @ kh.t()) * D ** -0.5
            sc.masked_fill_(keys[None] > last[i:i + step, None], -math.inf)
            out[i:i + step, h] = torch.softmax(sc, -1) @ vh
    return out


def _decode64(s, cache, q_proj, k_new, v_new, r, first=0):
    """The decode batch's output [B, hq * D]; r gets the appended rows."""
    hq, hkv, B = s["hq"], s["hkv"], len(s["lens"])
    qg = q_proj.double().view(B, hq, 2, D)
    pos = s["pos"].long()
    q = _rope(_norm(qg[:, :, 0], s["qw"]), s["cos"][pos], s["sin"][pos])
    kn = _rope(_norm(k_new.double().view(B, hkv, D), s["kw"]), s["cos"][pos], s["sin"][pos])
    vn = v_new.double().view(B, hkv, D)
    out = torch.empty(B, hq, D, dtype=torch.float64, device=DEV)
    for b, n in enumerate(s["lens"]):
        k, v = _rows64(cache, b, n)
        k, v = torch.cat([k, kn[b][:, None]], 1), torch.cat([v, vn[b][:, None]], 1)
        out[b] = _attend(q[b:b + 1], k, v, n)[0]
        _put(cache, r, b, n, kn[b][:, None], vn[b][:, None])
    return (out * torch.sigmoid(qg[:, :, 1])).reshape(B, hq * D)


def _prefill64(s, cache, q_proj, k_new, v_new, start, r):
    hq, hkv, n = s["hq"], s["hkv"], q_proj.shape[0]
    qg = q_proj.double().view(n, hq, 2, D)
    cos, sin = s["cos"][start:start + n], s["sin"][start:start + n]
    q = _rope(_norm(qg[:, :, 0], s["qw"]), cos, sin)
    kn = _rope(_norm(k_new.double().view(n, hkv, D), s["kw"]), cos, sin).transpose(0, 1)
    vn = v_new.double().view(n, hkv, D).transpose(0, 1)
    k, v = _rows64(cache, 0, start)
    out = _attend(q, torch.cat([k, kn], 1), torch.cat([v, vn], 1), start)
    _put(cache, r, 0, start, kn, vn)
    return (out * torch.sigmoid(qg[:, :, 1])).reshape(n, hq * D)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "dropin":
        q, k, v = s["q"][0].double().transpose(0, 1), s["k"][0].double(), s["v"][0].double()
        return dict(out=_attend(q, k, v, case["start"]).transpose(0, 1)[None])
    r = {}
    if "cache" in s:
        cache = s["cache"]
        r = dict(k=cache.k.double(), v=cache.v.double()) if cache.k_scale is None else \
            dict(k=None, v=None, ks=cache.k_scale.double(), vs=cache.v_scale.double())
    if kind == "decode":
        return dict(r, out=_decode64(s, cache, s["q_proj"], s["k_new"], s["v_new"], r))
    if kind == "prefill":
        return dict(r, out=_prefill64(s, cache, s["q_proj"], s["k_new"], s["v_new"], case["start"], r))
    if kind == "mixed":
        c = s["chunk"]
        chunk = _prefill64(s, c["cache"], c["q_proj"], c["k_new"], c["v_new"], case["start"], r)
        out = _decode64(s, s["decode"]["cache"], s["q_proj"], s["k_new"], s["v_new"], r)
        return dict(r, chunk=chunk, out=out)
    x = _norm(s["residual"].double(), s["nw"])
    q_proj, k_new, v_new = (x @ s[w].double().t() for w in ("wq", "wk", "wv"))
    attn = s.get("attn")
    if kind == "proj":
        attn = attn.double()
    elif kind == "layer_chunk":
        attn = _prefill64(s, cache, q_proj, k_new, v_new, case["start"], r)
    else:
        attn = _decode64(s, cache, q_proj, k_new, v_new, r)
    hidden = s["residual"].double() + attn @ s["wo"].double().t()
    if kind == "layer_kernel":
        return dict(r, hidden=hidden)
    if case.get("rope"):  # qkv_proj_rope hands out k as the cache holds it
        pos = s["pos"].long()
        n, hkv = len(s["lens"]), case["hkv"]
        k_new = _rope(_norm(k_new.view(n, hkv, D), s["kw"]), s["cos"][pos], s["sin"][pos]).reshape(n, hkv * D)
    out = dict(hidden=hidden, k_new=k_new, v_new=v_new)
    if kind == "proj":
        return dict(out, q_proj=q_proj)
    return dict(out, attn=attn, **r)
