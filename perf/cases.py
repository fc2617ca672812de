"""The work a serving program has this library do, as timed cases.

Every case is one pass through the package's public entry points on inputs
that a program holds in GPU memory: cache writers (prefill, ragged prompts,
decode-step appends), the paged decode (one call, a whole captured step, the
split records of a context-parallel rank), the KV4/FP8 NZ decode and the
codec leaves. Sizes are the configurations that the benchmark and the tests
use, and their neighbourhood.

  listed()            the named cases
  draw(rng)           another case of the same ranges
  prepare(case, seed) inputs, caches, workspaces and captured graphs
  run(state)          one pass; its outputs
  work(case)          the bytes and operations a pass cannot do without
  tolerance(case)     how far two correct implementations may differ
  exact(case, seed)   the floating outputs in 64 bits, in plain torch
"""
from __future__ import annotations

import importlib
import math

import torch

tq4 = importlib.import_module("ascend-micro-harness_amd")
DEV = "cuda"
STRIP = 16
KV4_GAIN = 2.9832882881  # levels of the KV4/FP8 cache per unit of its scale


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # One sequence being generated: the latency of a single decode call.
        dict(name="decode_1x4096", kind="decode", batch=1, heads=32, kv_heads=8, head_size=128,
             page=16, lo=4096, hi=4096, stage=1, rotated=False),
        # A serving batch of unequal contexts, the largest decode.
        dict(name="decode_64_ragged", kind="decode", batch=64, heads=32, kv_heads=8,
             head_size=128, page=16, lo=512, hi=8192, stage=1, rotated=False),
        # One very long context.
        dict(name="decode_1x65536", kind="decode", batch=1, heads=32, kv_heads=8, head_size=128,
             page=16, lo=65536, hi=65536, stage=1, rotated=False),
        # A small batch's token step, several layers, captured as a serving
        # loop captures it: append the token, then attend, per layer.
        dict(name="step_8x8_layers", kind="step", layers=8, batch=8, heads=32, kv_heads=8,
             head_size=128, page=16, lo=300, hi=3001, stage=1),
        # A context-parallel rank: the split records, and their combine; wide
        # heads, a full GQA group and large pages.
        dict(name="partials_d256", kind="partials", batch=4, heads=32, kv_heads=2,
             head_size=256, page=128, lo=1055, hi=8192, splits=8),
        # A long prompt through the whole-strip writer, and a short INT8 one.
        dict(name="prefill_bf16_16384", kind="prefill", dtype="bf16", tokens=16384, kv_heads=8,
             head_size=128, page=16),
        dict(name="prefill_a8_1024", kind="prefill", dtype="int8", tokens=1024, kv_heads=8,
             head_size=128, page=16),
        # The decode step's append of one token per sequence.
        dict(name="append_64", kind="append", tokens=64, kv_heads=8, head_size=128, page=16),
        # A batch of prompt chunks of uneven lengths that begin anywhere in a page.
        dict(name="chunks_8_ragged", kind="chunks", requests=8, lo=17, hi=2048, kv_heads=8,
             head_size=128, page=16),
        # The KV4/FP8 cache: one request over pre-rotated FP32 queries, and a
        # batch over raw BF16 ones.
        dict(name="nz_1x4096", kind="nz", batch=1, heads=16, kv_heads=1, page=128, lo=4096,
             hi=4096, raw=False, element="fp16", stage=0),
        dict(name="nz_32x8192", kind="nz", batch=32, heads=64, kv_heads=4, page=128, lo=8192,
             hi=8192, raw=True, element="bf16", stage=1),
        # The RMS codec's writer.
        dict(name="codec_rms_4096", kind="codec", codec="rms", dtype="bf16", tokens=4096,
             kv_heads=8, head_size=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_KINDS = ("decode", "decode", "decode", "step", "partials", "prefill", "append", "chunks", "nz",
          "codec")


def _draw_once(rng):
    kind = rng.choice(_KINDS)
    d = rng.choice((64, 128, 128, 256))
    page = rng.choice((16, 16, 32, 64, 128))
    hkv = rng.choice((1, 2, 4, 8, 8))
    if kind in ("decode", "step", "partials"):
        group = rng.choice((1, 2, 3, 4, 4, 5, 7, 8, 16))
        hi = _log(rng, 33, 65536 if kind == "decode" else 8192)
        lo = hi if rng.random() < 0.3 else max(1, int(hi * rng.uniform(0.05, 0.95)))
        batch = _log(rng, 1, 64 if kind == "decode" else 16)
        c = dict(kind=kind, batch=batch, heads=hkv * group, kv_heads=hkv, head_size=d, page=page,
                 lo=lo, hi=hi)
        if kind == "decode":
            c.update(stage=rng.choice((0, 1, 1, 2)), rotated=rng.random() < 0.2)
        elif kind == "step":
            c.update(layers=rng.choice((2, 4, 8)), stage=1)
        else:
            c.update(splits=rng.choice((1, 2, 3, 4, 8, 16)))
        return c
    if kind == "prefill":
        return dict(kind=kind, dtype=rng.choice(("bf16", "int8")),
                    tokens=STRIP * _log(rng, 1, 1024), kv_heads=hkv, head_size=d, page=page)
    if kind == "append":
        return dict(kind=kind, tokens=_log(rng, 1, 1024), kv_heads=hkv, head_size=d, page=page)
    if kind == "chunks":
        hi = _log(rng, 2, 2048)
        return dict(kind=kind, requests=_log(rng, 1, 32), lo=max(1, int(hi * rng.uniform(0, 1))),
                    hi=hi, kv_heads=hkv, head_size=d, page=page)
    if kind == "nz":
        hkv = rng.choice((1, 2, 4))
        hi = _log(rng, 65, 16384)
        raw = rng.random() < 0.5
        return dict(kind=kind, batch=_log(rng, 1, 32), heads=hkv * rng.choice((1, 4, 8, 16, 20)),
                    kv_heads=hkv, page=rng.choice((64, 128, 256)), lo=max(1, hi - _log(rng, 1, hi)),
                    hi=hi, raw=raw, element=rng.choice(("fp16", "bf16")),
                    stage=rng.choice((0, 1, 2)) if raw else 0)
    codec = rng.choice(("rms", "rms", "lloyd", "icdf"))
    if codec == "rms":
        return dict(kind=kind, codec=codec, dtype=rng.choice(("bf16", "fp16")),
                    tokens=_log(rng, 1, 16384), kv_heads=hkv, head_size=d)
    if codec == "lloyd":
        return dict(kind=kind, codec=codec, bits=rng.choice((2, 4)), mode=rng.choice((0, 2, 4)),
                    count=8 * _log(rng, 128, 1 << 20))
    return dict(kind=kind, codec=codec, dtype=rng.choice(("bf16", "fp16")),
                count=1024 * _log(rng, 1, 1 << 14))


# what a drawn case may cost: the largest listed case's bytes, or, for the
# token-granular writers, the listed one's tokens x heads
_BYTES_MAX = 330e6
_CHUNK_ROWS_MAX = 8 * 1032 * 8


def draw(rng):
    names = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        c = _draw_once(rng)
        if c in names or work(c)["bytes"] > _BYTES_MAX:
            continue
        if c["kind"] == "chunks" and sum(_lens(c, c["requests"])) * c["kv_heads"] > _CHUNK_ROWS_MAX:
            continue
        return c


# ------------------------------------------------------------------- inputs
def _lens(case, n):
    """n lengths spread evenly over [lo, hi] (the seed only permutes them)."""
    lo, hi = case["lo"], case["hi"]
    return [hi] if n == 1 else [lo + (hi - lo) * i // (n - 1) for i in range(n)]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 12345)
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, device=DEV, generator=g).to(dtype)


def _signs(g, d):
    return (torch.randint(0, 2, (d,), device=DEV, generator=g) * 2 - 1).to(torch.float32)


def _perm(g, n):
    return torch.randperm(n, device=DEV, generator=g).to(torch.int32)


def _permuted_lens(case, g):
    n = case["batch"]
    order = torch.randperm(n, device=DEV, generator=g).tolist()
    lens = _lens(case, n)
    return [lens[i] for i in order]


def _tables(g, lens, page):
    """(block tables [n][max pages], pages in the pool): every sequence's
    pages at random places of one shared pool."""
    need = [(c + page - 1) // page for c in lens]
    pool = sum(need) + 1
    perm = _perm(g, pool).cpu()
    tab = torch.zeros((len(lens), max(need)), dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tab[b, :n] = perm[at:at + n]
        at += n
    return tab.to(DEV), pool


def _pack(codes):
    """Signed 4-bit codes (int8, last dim even) to bytes, low nibble first."""
    c = codes.view(torch.uint8)
    return (c[..., 0::2] & 15 | (c[..., 1::2] << 4)).view(torch.int8)


def _quantise(y, dim):
    """The cache's quantiser over `dim`: codes and exponent of rotated values
    (scale = 2^(e-2) / sqrt(d))."""
    e = torch.frexp(y.abs().amax(dim, keepdim=True))[1] - 1
    codes = torch.clamp(torch.round(torch.ldexp(y, 2 - e)), -8, 7)
    return codes.to(torch.int8), e.squeeze(dim)


def _filled_cache(g, pool, hkv, page, d):
    """A cache as the writers leave it after N(0,1) keys and values (the
    rotation of a normal vector is normal with d times the variance)."""
    rows = pool * hkv * page
    kc = torch.empty(rows * d // 2, dtype=torch.int8, device=DEV)
    vc = torch.empty_like(kc)
    sc = torch.empty(2 * rows, dtype=torch.float32, device=DEV)
    step = max(STRIP, (1 << 25) // d // STRIP * STRIP)
    isl = 1.0 / math.sqrt(d)
    for r0 in range(0, rows, step):
        n = min(step, rows - r0)
        codes, e = _quantise(_randn(g, n, d) * math.sqrt(d), 1)
        kc[r0 * d // 2:(r0 + n) * d // 2] = _pack(codes).view(-1)
        sc[r0:r0 + n] = torch.ldexp(torch.full_like(e, isl, dtype=torch.float32), e - 2)
        codes, e = _quantise(_randn(g, n // STRIP, d, STRIP) * math.sqrt(d), 1)
        vc[r0 * d // 2:(r0 + n) * d // 2] = _pack(codes).view(-1)
        sc[rows + r0:rows + r0 + n] = torch.ldexp(
            torch.full_like(e, isl, dtype=torch.float32), e - 2).view(-1)
    return kc, vc, sc


def _decode_inputs(case, g, layers=1):
    """Lengths, tables, caches and queries of a decode-shaped case."""
    hkv, page, d = case["kv_heads"], case["page"], case["head_size"]
    lens = _permuted_lens(case, g)
    tab, pool = _tables(g, lens, page)
    s = dict(case=case, lens=lens, tables=tab, pool=pool, signs=_signs(g, d),
             ctx=torch.tensor(lens, dtype=torch.int32, device=DEV))
    caches = [_filled_cache(g, pool, hkv, page, d) for _ in range(layers)]
    shape = (layers, case["batch"])
    s["q"] = _randn(g, *shape, case["heads"], d, dtype=torch.bfloat16)
    if layers > 1 or case["kind"] == "step":
        s["caches"] = [torch.stack(c) for c in zip(*caches)]
        s["k"] = _randn(g, *shape, hkv, d, dtype=torch.bfloat16)
        s["v"] = _randn(g, *shape, hkv, d, dtype=torch.bfloat16)
        last = [n - 1 for n in lens]
        at = torch.tensor(last, device=DEV)
        pages = tab.gather(1, (at // page)[:, None])[:, 0]
        s["slots"] = (pages * page + at % page).to(torch.int32)
    else:
        s["caches"] = list(caches[0])
        s["q"] = s["q"][0].contiguous()
        if case.get("stage") == 2:
            s["gate"] = _randn(g, case["batch"], case["heads"], d)
    return s


def _run_step(s):
    """One token step over the layers, as torch operators."""
    c, outs = s["case"], []
    ops = torch.ops.tq4
    kc, vc, sc = s["caches"]
    for i in range(c["layers"]):
        ops.reshape_scatter(s["k"][i], s["v"][i], kc[i], vc[i], sc[i], s["slots"], s["signs"],
                            None, c["page"], 0.0)
        outs.append(ops.paged_attention(
            s["q"][i], kc[i], vc[i], sc[i], s["tables"], s["ctx"], s["signs"], s["ws"], None,
            c["kv_heads"], c["page"], s["splits"], 0.0, 0.0, c["stage"], False))
    return outs


def _nz_inputs(case, g):
    hkv, page, n = case["kv_heads"], case["page"], case["batch"]
    lens = _permuted_lens(case, g)
    tab, pool = _tables(g, lens, page)
    rows = pool * page
    # levels of N(0,1) vectors at an RMS scale near one
    codes = torch.clamp(torch.floor(torch.randn(
        (2, rows * hkv * 256), device=DEV, generator=g) * KV4_GAIN), -8, 7).to(torch.int8)
    packed = _pack(codes).view(torch.uint8)
    s = dict(case=case, lens=lens, tables=tab, pool=pool, key=packed[0].contiguous(),
             value=packed[1].contiguous(),
             scales=torch.rand((rows, 8), device=DEV, generator=g) * 0.5 + 0.75,
             ctx=torch.tensor(lens, dtype=torch.int32, device=DEV))
    elem = torch.bfloat16 if case["element"] == "bf16" else torch.float16
    s["q"] = _randn(g, n, case["heads"], 256, dtype=elem if case["raw"] else torch.float32)
    s["elem"] = elem
    if case["raw"]:
        s["signs"] = _signs(g, 256)
        s["q_rot"] = torch.empty(s["q"].shape, dtype=torch.float32, device=DEV)
        s["gate"] = _randn(g, *s["q"].shape, dtype=elem) if case["stage"] == 2 else None
    return s


def _empty_cache(pool, hkv, page, d):
    rows = pool * hkv * page
    return [torch.zeros(rows * d // 2, dtype=torch.int8, device=DEV),
            torch.zeros(rows * d // 2, dtype=torch.int8, device=DEV),
            torch.zeros(2 * rows, dtype=torch.float32, device=DEV)]


def _writer_inputs(case, g):
    """Rows, slots and the pool of the prefill, append and chunks cases."""
    hkv, page, d, kind = case["kv_heads"], case["page"], case["head_size"], case["kind"]
    s = dict(case=case, signs=_signs(g, d))
    if kind == "prefill":
        n = case["tokens"]
        tab, pool = _tables(g, [n], page)
        at = torch.arange(n, device=DEV)
        s["slots"] = (tab[0][at // page] * page + at % page).to(torch.int32)
        s["caches"] = _empty_cache(pool, hkv, page, d)
    elif kind == "append":  # each token somewhere in a page of its own sequence
        n = case["tokens"]
        pool = n + 1
        off = torch.randint(0, page, (n,), device=DEV, generator=g)
        s["slots"] = (_perm(g, pool)[:n] * page + off).to(torch.int32)
        s["caches"] = list(_filled_cache(g, pool, hkv, page, d))
    else:  # chunks: each begins behind a cached prefix of 0 .. 3 strips' tokens
        r = case["requests"]
        lens = _lens(case, r)
        lens = [lens[i] for i in torch.randperm(r, device=DEV, generator=g).tolist()]
        begin = torch.randint(0, 48, (r,), device=DEV, generator=g).tolist()
        tab, pool = _tables(g, [47 + c for c in lens], page)
        slots, cu = [], [0]
        for i, (b, c) in enumerate(zip(begin, lens)):
            at = torch.arange(b, b + c, device=DEV)
            slots.append(tab[i][at // page] * page + at % page)
            cu.append(cu[-1] + c)
        n = cu[-1]
        s["slots"] = torch.cat(slots).to(torch.int32)
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device=DEV)
        s["caches"] = list(_filled_cache(g, pool, hkv, page, d))
    s["pool"] = pool
    if case.get("dtype") == "int8":
        s["k"], s["v"] = (torch.randint(-127, 128, (n, hkv, d), device=DEV, generator=g,
                                        dtype=torch.int8) for _ in range(2))
    else:
        s["k"], s["v"] = (_randn(g, n, hkv, d, dtype=torch.bfloat16) for _ in range(2))
    return s


def _codec_inputs(case, g):
    s = dict(case=case)
    half = torch.bfloat16 if case.get("dtype") == "bf16" else torch.float16
    if case["codec"] == "rms":
        n, hkv, d = case["tokens"], case["kv_heads"], case["head_size"]
        pool = (n + STRIP - 1) // STRIP + 1
        slots = pool * STRIP
        s.update(signs=_signs(g, d), slots=_perm(g, slots)[:n].contiguous(), pool=pool,
                 k=_randn(g, n, hkv, d, dtype=half), v=_randn(g, n, hkv, d, dtype=half),
                 kc=torch.zeros(slots * hkv * d // 2, dtype=torch.int8, device=DEV),
                 vc=torch.zeros(slots * hkv * d // 2, dtype=torch.int8, device=DEV),
                 sc=torch.zeros(slots * tq4.rms_scale_slot_floats(hkv), dtype=torch.float32,
                                device=DEV))
    elif case["codec"] == "icdf":
        s["x"] = _randn(g, case["count"], dtype=half)
    elif case["mode"] == 4:
        s["x"] = torch.randint(0, 256, (case["count"] * case["bits"] // 8,), device=DEV,
                               generator=g, dtype=torch.uint8)
    else:
        s["x"] = _randn(g, case["count"])
    return s


def _inputs(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("decode", "partials"):
        return _decode_inputs(case, g)
    if kind == "step":
        return _decode_inputs(case, g, case["layers"])
    if kind == "nz":
        return _nz_inputs(case, g)
    if kind == "codec":
        return _codec_inputs(case, g)
    return _writer_inputs(case, g)


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind in ("decode", "step"):
        # a server holds the lengths on the host when it plans the step
        k = tq4.auto_splits(case["batch"], case["kv_heads"], s["tables"].shape[1], case["page"],
                            context_lens=s["lens"])
        s["splits"] = k
        s["ws"] = tq4.decode_workspace(case["batch"], case["heads"], case["kv_heads"],
                                       case["head_size"], k)
    if kind == "step":
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _run_step(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["outs"] = _run_step(s)
    if kind == "nz":
        s["ws"] = tq4.torch_ops.kv4fp8_workspace_for(s["q"], case["kv_heads"], s["tables"],
                                                     case["page"], s["pool"])
    return s


# ---------------------------------------------------------------- one pass
def _record_parts(rec):
    """The records' fields on their own (an empty split's m is -3e38)."""
    return {"m": rec[..., 0], "l": rec[..., 1], "acc": rec[..., 4:]}


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "decode":
        kc, vc, sc = s["caches"]
        return tq4.paged_decode(
            s["q"], kc, vc, sc, s["tables"], s["ctx"], s["signs"], c["kv_heads"], c["page"],
            s["pool"], workspace=s["ws"], gate=s.get("gate"), num_splits=s["splits"],
            output_stage=c["stage"], flags=tq4.TQ4_DECODE_QUERY_ROTATED if c["rotated"] else 0)
    if kind == "step":
        s["graph"].replay()
        return {"out": s["outs"], "caches": s["caches"]}
    if kind == "partials":
        kc, vc, sc = s["caches"]
        rec = tq4.paged_decode_partials(
            s["q"], kc, vc, sc, s["tables"], s["ctx"], s["signs"], c["kv_heads"], c["page"],
            s["pool"], c["splits"])
        out = tq4.splitk_combine(rec, s["signs"], c["batch"], c["heads"], c["head_size"],
                                 c["splits"])
        return {**_record_parts(rec), "out": out}
    if kind == "prefill":
        write = (tq4.reshape_and_cache_a8 if c["dtype"] == "int8" else tq4.reshape_and_cache_bf16)
        write(s["k"], s["v"], *s["caches"], s["slots"], pi_signs=s["signs"],
              num_blocks=s["pool"], block_size=c["page"])
        return s["caches"]
    if kind in ("append", "chunks"):
        tq4.reshape_scatter(s["k"], s["v"], *s["caches"], s["slots"], s["signs"],
                            cu_seqlens=s.get("cu"), num_blocks=s["pool"], block_size=c["page"])
        return s["caches"]
    if kind == "nz":
        elem = s["elem"]
        if c["raw"]:
            out = tq4.kv4fp8_decode_raw_query(
                s["q"], s["signs"], s["key"], s["value"], s["scales"], s["tables"], s["ctx"],
                c["kv_heads"], c["page"], s["pool"], gate=s["gate"], output_stage=c["stage"],
                query_out=s["q_rot"], workspace=s["ws"])
            return {"out": out, "q_rot": s["q_rot"]}
        return {"out": tq4.kv4fp8_decode(
            s["q"], s["key"], s["value"], s["scales"], s["tables"], s["ctx"], c["kv_heads"],
            c["page"], s["pool"], out_dtype=elem, workspace=s["ws"])}
    if c["codec"] == "rms":
        tq4.rms_reshape_and_cache(s["k"], s["v"], s["kc"], s["vc"], s["sc"], s["slots"],
                                  s["signs"], num_blocks=s["pool"], block_size=STRIP)
        return {"key": s["kc"], "value": s["vc"], "scale": s["sc"]}
    if c["codec"] == "icdf":
        return {"codes": tq4.icdf_quantize(s["x"])}
    dst, codes = tq4.lloydmax_quantize(s["x"], bits=c["bits"], mode=c["mode"])
    return {"dst": dst} if c["mode"] == 4 else {"dst": dst, "codes": codes}


# ------------------------------------------------------- what a pass must do
def _append_bytes(rows, tokens, d, in_bytes):
    """Writer traffic of `rows` (token, kv head) pairs: both planes read,
    their codes and scales written, a slot per token."""
    return rows * (2 * d * in_bytes + d + 8) + tokens * 4


def work(case):
    kind = case["kind"]
    if kind in ("decode", "step", "partials", "nz"):
        n, hq, hkv, page = case["batch"], case["heads"], case["kv_heads"], case["page"]
        lens = _lens(case, n)
        total = sum(lens)
        tables = 4 * sum((c + page - 1) // page for c in lens) + 4 * n
        if kind == "nz":
            q = 2 if case["raw"] else 4
            nbytes = (total * hkv * (256 + 8) + tables + n * hq * 256 * (q + 2) +
                      (n * hq * 256 * 4 if case["raw"] else 0) +
                      (n * hq * 256 * 2 if case["stage"] == 2 else 0))
            return dict(bytes=nbytes, flops=4 * total * hq * 256)
        d = case["head_size"]
        nbytes = total * hkv * (d + 8) + tables + 2 * n * hq * d * 2
        flops = 4 * total * hq * d
        if kind == "decode" and case["stage"] == 2:
            nbytes += n * hq * d * 4
        if kind == "partials":
            nbytes += n * hq * case["splits"] * (d + 4) * 4  # the records are a result
        if kind == "step":
            L = case["layers"]
            nbytes = L * (nbytes + _append_bytes(n * hkv, n, d, 2))
            flops = L * (flops + n * hkv * 2 * d * int(math.log2(d)))
        return dict(bytes=nbytes, flops=flops)
    if kind == "codec" and case["codec"] != "rms":
        n = case["count"]
        if case["codec"] == "icdf":
            return dict(bytes=n * 2 + n // 2, flops=4 * n)
        return dict(bytes=n * 4 + n * case["bits"] // 8 + (0 if case["mode"] == 4 else n * 4),
                    flops=4 * n)
    hkv, d = case["kv_heads"], case["head_size"]
    tokens = sum(_lens(case, case["requests"])) if kind == "chunks" else case["tokens"]
    rows = tokens * hkv
    flops = rows * 2 * d * (int(math.log2(d)) + 3)
    if kind == "codec":
        return dict(bytes=rows * 5 * d + tokens * (4 * ((2 * hkv + 7) // 8 * 8) + 4), flops=flops)
    return dict(bytes=_append_bytes(rows, tokens, d, 1 if case.get("dtype") == "int8" else 2),
                flops=flops)


def tolerance(case):
    kind = case["kind"]
    # Measured against the 64-bit results: 1.7e-3 for every BF16 output (its
    # rounding alone), 2.1e-4 for FP16 ones, 3.5e-4 for the partial records
    # (FP16 operands). A BF16 value may be a unit (2^-8) off, an FP8 operand
    # may fall on the other side of its rounding boundary.
    if kind == "nz":
        return ({"rel": 7e-3, "max": 5e-2} if case["element"] == "bf16" else
                {"rel": 1e-3, "max": 2e-2})
    if kind in ("decode", "step", "partials"):
        return {"rel": 7e-3, "max": 3e-2}
    return "exact"  # bytes, and scales and centroids whose bits are the contract


# ------------------------------------------------------------- in 64 bits
def _hadamard(n):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _rotation(signs):
    """M = (H_{d/32} x I_32) diag(signs) (I_{d/32} x H_32), as a matrix."""
    d, s = signs.numel(), signs.double()
    eye = lambda n: torch.eye(n, dtype=torch.float64, device=DEV)  # noqa: E731
    return torch.kron(_hadamard(d // 32), eye(32)) @ (s[:, None] * torch.kron(eye(d // 32),
                                                                            _hadamard(32)))


def _codes(packed, shape):
    b = packed.view(torch.uint8)
    lo, hi = (b & 15).to(torch.int8), (b >> 4).to(torch.int8)
    c = torch.stack([lo, hi], -1).view(*shape)
    return torch.where(c > 7, c - 16, c).double()


def _sequence(caches, pages, n, pool, hkv, page, d):
    """Keys and values [kv heads][n][d] of a sequence, in the rotated basis."""
    kc, vc, sc = caches
    p = pages[:(n + page - 1) // page].long()
    m = p.numel()
    k = _codes(kc.view(pool, -1)[p], (m, hkv, page, d))
    v = _codes(vc.view(pool, -1)[p], (m, hkv, page // STRIP, d, STRIP))
    v = v.permute(0, 1, 2, 4, 3).reshape(m, hkv, page, d)
    ks, vs = sc.view(2, pool, hkv, page)[:, p].double()
    k, v = k * ks[..., None], v * vs[..., None]
    return [x.transpose(0, 1).reshape(hkv, m * page, d)[:, :n].contiguous() for x in (k, v)]


def _stage(ctx, m, stage, gate, isl):
    """The output stages on rows [..., d] of the rotated basis."""
    if stage >= 1:
        ctx = ctx @ m * isl
        if stage == 2:
            ctx = ctx / (1.0 + torch.exp(-gate.double()))
    return ctx


def _exact_decode(case, s, caches, q, replace=None):
    """Decode outputs [n][heads][d]; `replace`: (keys, values) [n][kv heads][d]
    of each sequence's last token, in place of what the cache holds."""
    hkv, page, d = case["kv_heads"], case["page"], case["head_size"]
    group, isl = case["heads"] // hkv, 1.0 / math.sqrt(d)
    m = _rotation(s["signs"])
    rotated = case.get("rotated", False)
    qr = q.double() if rotated else q.double() @ m.T * isl
    outs, records = [], []
    for b, n in enumerate(s["lens"]):
        k, v = _sequence(caches, s["tables"][b], n, s["pool"], hkv, page, d)
        if replace is not None:
            k[:, n - 1], v[:, n - 1] = replace[0][b], replace[1][b]
        qs = qr[b].view(hkv, group, d)
        sc = torch.matmul(k, qs.transpose(1, 2).contiguous()) * isl  # [hkv][n][group]
        if case["kind"] == "partials":
            records.append(_exact_records(case, s, sc, v))
        p = torch.softmax(sc, 1).transpose(1, 2).contiguous()
        outs.append(torch.matmul(p, v).view(case["heads"], d))
    gate = s.get("gate")
    out = _stage(torch.stack(outs), m, case.get("stage", 1), gate, isl)
    return out, records


def _exact_records(case, s, sc, v):
    """[heads][splits][d + 4] records (m, l, 0, 0, acc) of one sequence."""
    hkv, page, d, splits = case["kv_heads"], case["page"], case["head_size"], case["splits"]
    group = case["heads"] // hkv
    width = -(-s["tables"].shape[1] // splits) * page
    rec = torch.zeros((hkv, group, splits, d + 4), dtype=torch.float64, device=DEV)
    rec[..., 0] = -3e38
    for k in range(splits):
        part = sc[:, k * width:(k + 1) * width]
        if part.shape[1] == 0:
            continue
        mx = part.amax(1)  # [hkv][group]
        p = torch.exp(part - mx[:, None])
        rec[:, :, k, 0] = mx
        rec[:, :, k, 1] = p.sum(1)
        rec[:, :, k, 4:] = torch.matmul(p.transpose(1, 2).contiguous(),
                                        v[:, k * width:(k + 1) * width])
    return rec.view(case["heads"], splits, d + 4)


def _fp8(x):
    return x.float().to(torch.float8_e4m3fn).double()


def _exact_nz(case, s):
    """The KV4/FP8 operator in 64 bits: its FP8 operands (queries per row,
    probabilities per 64-row tile) are part of its definition, all else exact."""
    hkv, page, n_heads = case["kv_heads"], case["page"], case["heads"]
    group, scale = n_heads // hkv, 1.0 / 16.0
    q = s["q"].double()
    pi = None
    if case["raw"]:
        sg = s["signs"].double()
        pi = sg[:, None] * _hadamard(256) * sg[None, :] / 16.0
        q = q @ pi.T
    q_scale = 448.0 / (q.abs().amax(-1, keepdim=True) + 1e-20)
    q8 = _fp8(q * q_scale)
    outs = []
    for b, n in enumerate(s["lens"]):
        tiles = (n + 63) // 64
        pages = s["tables"][b, :(n + page - 1) // page].long()

        def rows(packed):
            # [page][tile][head][column group][row][byte] -> [head][row][channel]
            x = packed.view(-1, page // 64, hkv, 4, 64, 32)[pages].permute(2, 0, 1, 4, 3, 5)
            x = x.reshape(hkv, pages.numel() * page, 128)[:, :tiles * 64]
            c = torch.cat([x & 15, x >> 4], -1).to(torch.int8)
            return torch.where(c > 7, c - 16, c).double() + 0.5

        k, v = rows(s["key"]), rows(s["value"])
        sl = s["scales"].view(-1, page, 8)[pages].view(-1, 8)[:tiles * 64].double()
        ks, vs = sl[:, :hkv].T / KV4_GAIN, sl[:, hkv:2 * hkv].T / KV4_GAIN
        qb = q8[b].view(hkv, group, 256)
        logits = torch.matmul(qb, k.transpose(1, 2).contiguous()) * (ks * scale)[:, None]
        logits = logits / q_scale[b].view(hkv, group, 1)
        logits[:, :, n:] = -math.inf
        mx = logits.amax(-1, keepdim=True)
        p = torch.exp(logits - mx)
        total = p.sum(-1, keepdim=True)
        pv = (p * vs[:, None]).view(hkv, group, tiles, 64)
        pv = torch.nan_to_num(pv)
        tile_max = pv.amax(-1, keepdim=True)
        up = 448.0 / torch.clamp(tile_max, min=1e-300)
        p8 = (_fp8(pv * up) / up).view(hkv, group, tiles * 64)
        outs.append((torch.matmul(p8, v) / total).view(n_heads, 256))
    out = torch.stack(outs)
    if case["raw"]:
        if case["stage"] >= 1:
            out = out @ pi.T
        if case["stage"] == 2:
            out = out / (1.0 + torch.exp(-s["gate"].double().clamp(min=-80.0)))
        return {"out": out, "q_rot": q}
    return {"out": out}


def _written_scales(case, s, floor):
    """The scale planes a TQ4 writer leaves, in 64 bits."""
    hkv, page, d = case["kv_heads"], case["page"], case["head_size"]
    m = _rotation(s["signs"])
    sc = s["caches"][2].double().view(2, s["pool"], hkv, page)
    slots = s["slots"].long()
    for plane, x in enumerate((s["k"], s["v"])):
        a = torch.matmul(x.double(), m.T.contiguous()).abs().amax(-1).clamp(min=floor)
        scale = torch.exp2(torch.frexp(a)[1].double() - 3) / math.sqrt(d)
        sc[plane, slots // page, :, slots % page] = scale
    return sc.view(-1)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind in ("decode", "partials"):
        out, records = _exact_decode(case, s, s["caches"], s["q"])
        if kind == "decode":
            return out
        return {**_record_parts(torch.stack(records)), "out": out}
    if kind == "step":
        d, m = case["head_size"], _rotation(s["signs"])
        outs = []
        for i in range(case["layers"]):
            last = []
            for x in (s["k"][i], s["v"][i]):
                codes, e = _quantise(x.double() @ m.T, -1)
                last.append(codes.double() * torch.exp2(e.double() - 2)[..., None] / math.sqrt(d))
            outs.append(_exact_decode(case, s, [c[i] for c in s["caches"]], s["q"][i], last)[0])
        return {"out": outs, "caches": [None, None, None]}
    if kind == "nz":
        return _exact_nz(case, s)
    if kind == "codec":
        if case["codec"] != "rms":
            return None
        hkv, d = case["kv_heads"], case["head_size"]
        sc = s["sc"].double().view(-1, tq4.rms_scale_slot_floats(hkv))
        rows = torch.cat([s["k"], s["v"]], 1).double()
        sc[s["slots"].long(), :2 * hkv] = rows.norm(dim=-1) / math.sqrt(d) + 1e-20
        return {"key": None, "value": None, "scale": sc.view(-1)}
    return [None, None, _written_scales(case, s, 1.0 if kind == "prefill" else 0.0)]
