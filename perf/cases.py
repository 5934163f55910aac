"""The performance cases of the codec: what a serving program has it do, through
its public entry points, over the sizes, types and options that occur.

A program stores KV-cache values (BF16 pages on the GPU -> compressed streams
on the GPU, sizes and bounds on the host) and restores them (streams -> pages
in the paged layout).  The families of cases, each in both directions:

``page``    one fp32 page through ``compress`` / ``decompress``: one-page jobs
            and every segment that the batched paths decline, in the wrapper's
            encoding mode (plain is the connector's default)
``pages32`` a list of equal fp32 pages through ``compress_batch_fixed`` /
            ``decompress_batch``
``blocks``  whole BF16 KV blocks [2, layers, tokens, heads, dim] through
            ``compress_batch_fixed_bf16`` / ``decompress_batch_fixed_bf16_scatter``
            into other page slots (one or more destinations a page)
``layer``   K and V of one layer over a whole context, as two long segments
            (``compress_batch_fixed_bf16`` / ``decompress_batch_fixed_bf16``)
``mixed``   a job with a bound per layer group: the grouped layer-indexed store
            and restore, through the C ABI with tables built once, as a native
            serving loop and bench.py call it
``ragged``  BF16 segments of any length at any 2-byte address

Every stream byte, size, bound and restored value is reproducible bit for bit,
so every tolerance is "exact".
"""

from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(
    REPO,
    "reducing-pcie-bottlenecks-for-llm-serving-with-cuszp-compressed-kv-cache-transfer_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import cuszp_wrapper_cpp as cpp  # noqa: E402
import kv_synth  # noqa: E402
import kvszp  # noqa: E402

MODES = {"fixed": cpp.MODE_FIXED, "plain": cpp.MODE_PLAIN, "outlier": cpp.MODE_OUTLIER}

# Values of the largest case: 2048 blocks of [2, 28, 16, 4, 128].
MOST_VALUES = 2048 * 458752


def listed():
    return [
        # One evicted block of a 28-layer, 2-head model as an fp32 segment in
        # the default mode: the smallest job, one call per block.
        {"name": "page_plain_store", "family": "page", "way": "store", "mode": "plain",
         "n": 229376, "eps": 1e-4, "relative": True},
        {"name": "page_plain_restore", "family": "page", "way": "restore", "mode": "plain",
         "n": 229376, "eps": 1e-4, "relative": True},
        # A job of 64 such blocks held in fp32.
        {"name": "pages32_store", "family": "pages32", "way": "store", "pages": 64,
         "n": 229376, "eps": 1e-4, "relative": True},
        {"name": "pages32_restore", "family": "pages32", "way": "restore", "pages": 64,
         "n": 229376, "eps": 1e-4, "relative": True},
        # Eight running requests each fill a block during decode.
        {"name": "blocks_decode_store", "family": "blocks", "way": "store", "pages": 8,
         "layers": 28, "tokens": 16, "heads": 2, "dim": 128, "eps": 1e-4,
         "relative": True, "values": "gauss", "dests": 1},
        # One layer of a 32K context with 8 heads: segments of 32 Mi values.
        {"name": "layer_32k_store", "family": "layer", "way": "store", "tokens": 32768,
         "heads": 8, "dim": 128, "eps": 1e-4, "relative": True},
        # One layer of a 4K context with 2 heads, fetched ahead of its use.
        {"name": "layer_4k_restore", "family": "layer", "way": "restore", "tokens": 4096,
         "heads": 2, "dim": 128, "eps": 1e-4, "relative": True},
        # A 4K prompt of a 28-layer, 2-head model: 256 blocks, 21 layers at
        # REL 1e-4 and 7 at 1e-5 (bench.py's default workload).
        {"name": "mixed_4k_store", "family": "mixed", "way": "store", "pages": 256,
         "layers": 28, "tokens": 16, "heads": 2, "dim": 128},
        {"name": "mixed_4k_restore", "family": "mixed", "way": "restore", "pages": 256,
         "layers": 28, "tokens": 16, "heads": 2, "dim": 128},
        # 256 segments of an odd length, one behind the other.
        {"name": "ragged_store", "family": "ragged", "way": "store", "pages": 256,
         "n": 100003, "eps": 1e-4, "relative": True},
        {"name": "ragged_restore", "family": "ragged", "way": "restore", "pages": 256,
         "n": 100003, "eps": 1e-4, "relative": True},
        # A 32K prompt of a 28-layer, 4-head model out and back into other
        # page slots: the largest job.
        {"name": "blocks_32k_step", "family": "blocks", "way": "step", "pages": 2048,
         "layers": 28, "tokens": 16, "heads": 4, "dim": 128, "eps": 1e-5,
         "relative": True, "values": "rope", "dests": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["page", "pages32", "blocks", "blocks", "layer", "mixed", "mixed",
                         "ragged"])
    case = {"family": family, "way": rng.choice(["store", "restore"])}
    if family == "mixed":
        case.update(pages=_log(rng, 4, 600), layers=rng.randint(8, 48),
                    tokens=rng.choice([8, 16, 32]), heads=rng.randint(1, 8),
                    dim=rng.choice([64, 80, 96, 128]))
    else:
        case.update(eps=rng.choice([1e-3, 1e-4, 1e-5]), relative=rng.random() < 0.8)
    if family == "page":
        case.update(mode=rng.choice(["plain", "plain", "outlier", "fixed"]),
                    n=_log(rng, 4096, 1 << 20))
    elif family == "pages32":
        case.update(pages=_log(rng, 2, 200), n=_log(rng, 8192, 1 << 18))
    elif family == "blocks":
        case.update(pages=_log(rng, 1, 1000), layers=rng.randint(2, 48),
                    tokens=rng.choice([8, 16, 32]), heads=rng.randint(1, 8),
                    dim=rng.choice([64, 80, 96, 128]),
                    values=rng.choice(["gauss", "rope", "stress"]),
                    dests=rng.choice([1, 1, 2, 4]))
    elif family == "layer":
        case.update(tokens=_log(rng, 500, 32768), heads=rng.randint(1, 8), dim=128)
    elif family == "ragged":
        case.update(pages=_log(rng, 4, 400), n=_log(rng, 1000, 300000) | 1)
    while _segments(case) * _values(case) > MOST_VALUES // 2:
        case["pages"] = case["pages"] // 2
    return case


def _values(case):
    """Values of one page or segment."""
    if case["family"] in ("blocks", "mixed"):
        return 2 * case["layers"] * case["tokens"] * case["heads"] * case["dim"]
    if case["family"] == "layer":
        return case["tokens"] * case["heads"] * case["dim"]
    return case["n"]


def _segments(case):
    """Pages or segments of one pass."""
    return {"page": 1, "layer": 2}.get(case["family"]) or case["pages"]


# ---- inputs -----------------------------------------------------------------

def _inputs(case, seed):
    """The values to store: [segments, values of a segment], BF16 or fp32."""
    family = case["family"]
    if family in ("blocks", "mixed"):
        shape = kv_synth.KVShape(case["layers"], case["heads"], case["dim"],
                                 case["pages"] * case["tokens"], case["tokens"])
        values = case.get("values", "gauss")
        if values == "rope":
            return kv_synth.rope_kv(shape, seed, "cuda")
        pages = kv_synth.paged_kv(shape, seed, "cuda")
        if values == "stress":
            # a tenth of the blocks padding, a tenth with heavy tails
            g = torch.Generator().manual_seed(seed)
            kind = torch.rand(case["pages"], generator=g)
            for i in (kind < 0.1).nonzero().flatten().tolist():
                pages[i].zero_()
            g = torch.Generator("cuda").manual_seed(seed)
            for i in ((kind >= 0.1) & (kind < 0.2)).nonzero().flatten().tolist():
                chi = torch.randn(2, pages.shape[1], generator=g, device="cuda")
                pages[i] /= (chi.square().sum(0) / 2).sqrt().clamp_min(1e-3).to(torch.bfloat16)
        return pages
    if family == "layer":
        shape = kv_synth.KVShape(1, case["heads"], case["dim"], case["tokens"])
        k, v = kv_synth.layer_kv(shape, 0, seed, "cuda")
        return torch.stack([k.reshape(-1), v.reshape(-1)])
    # Segments of any length: per-channel scales over 256 channels, four in
    # 128 of them large, as in the K and V of a layer.
    g = torch.Generator("cuda").manual_seed(seed)
    sigma = torch.exp(0.5 * torch.randn(256, generator=g, device="cuda"))
    sigma[torch.randperm(128, generator=g, device="cuda")[:4]] *= 15.0
    count = _segments(case) * case["n"]
    z = torch.randn(-(-count // 256), 256, generator=g, device="cuda") * sigma
    # BF16 cache values, widened for the fp32 entry points
    z = z.to(torch.bfloat16).flatten()[:count].view(_segments(case), case["n"])
    return z if family == "ragged" else z.float()


def _groups(case):
    """(bound, layers) of a mixed job: the profile of the 28-layer model, and
    every fourth layer at the smaller bound otherwise."""
    if case["layers"] == 28:
        return kv_synth.mixed_bound_groups()
    return kv_synth.mixed_bound_groups(case["layers"], range(0, case["layers"], 4))


_WRAPPERS: dict = {}


def _wrapper(mode="fixed", relative=True):
    """The codec object that a program makes once and keeps."""
    key = (mode, relative)
    if key not in _WRAPPERS:
        cfg = cpp.CompressionConfig(1e-4, relative, cpp.DIM_1D, MODES[mode], cpp.TYPE_FLOAT)
        _WRAPPERS[key] = cpp.CuSZpWrapper(cfg, 0)
    return _WRAPPERS[key]


def _buffers(counts):
    """One compressed buffer per segment of `counts` values, as slices of one
    zeroed slab: the capacity the API asks for, 512-byte steps."""
    caps = []
    for n in counts:
        blocks = -(-n // 32)
        worst = 1024 * -(-n // 32768) + 136 * blocks
        caps.append(-(-max(8 * n, worst) // 512) * 512)
    slab = torch.zeros(sum(caps), dtype=torch.uint8, device="cuda")
    return slab, list(slab.split(caps))


def _packed(wrapper, buffers, sizes):
    """The streams as a restore finds them: one slab, 8-byte-aligned offsets."""
    slab = torch.zeros(sum(-(-s // 8) * 8 for s in sizes), dtype=torch.uint8, device="cuda")
    ok, offsets, _ = wrapper.pack_payloads([b[:s] for b, s in zip(buffers, sizes)], slab)
    assert ok
    return [slab[o:o + s] for o, s in zip(offsets, sizes)]


def _mixed_tables(case, pages):
    """The requests of a mixed job, group by group, as C arrays."""
    groups = _groups(case)
    per_layer = case["tokens"] * case["heads"] * case["dim"]
    counts = [2 * len(layers) * per_layer for _, layers in groups for _ in range(case["pages"])]
    index = [torch.tensor(layers, dtype=torch.long, device="cuda") for _, layers in groups]
    rows = [p.data_ptr() for p in pages] * len(groups)
    return {
        "counts": counts, "index": index, "per_layer": per_layer, "batch": len(counts),
        "groups": len(groups), "pages": pages, "page_table": kvszp.ptr_array(rows),
        "eps": kvszp.f32_array([b for b, _ in groups for _ in range(case["pages"])]),
        "index_table": kvszp.ptr_array([t.data_ptr() for t in index]),
        "selected": kvszp.size_array([len(layers) for _, layers in groups]),
        "group_sizes": kvszp.size_array([case["pages"]] * len(groups)),
        "sizes": (ctypes.c_uint64 * len(counts))(), "bounds": (ctypes.c_float * len(counts))(),
        "ctx": _wrapper()._ctx, "layers": case["layers"],
    }


def _mixed_store(t):
    kvszp.check(t["ctx"].compress_indexed_groups(
        t["page_table"], t["stream_table"], t["caps"], t["index_table"], t["selected"],
        t["group_sizes"], t["groups"], 2, t["layers"], t["per_layer"], t["eps"], t["batch"],
        torch.cuda.current_stream().cuda_stream, t["sizes"], t["bounds"]))


# ---- one case ----------------------------------------------------------------

def _stored(case, pages):
    """State of a store: inputs, buffers and the wrapper."""
    if case["family"] == "mixed":
        t = _mixed_tables(case, pages)
        slab, buffers = _buffers(t["counts"])
        return dict(t, case=case, slab=slab, buffers=buffers,
                    stream_table=kvszp.ptr_array([b.data_ptr() for b in buffers]),
                    caps=kvszp.u64_array([b.numel() for b in buffers]))
    slab, buffers = _buffers([pages.shape[1]] * pages.shape[0])
    w = _wrapper(case.get("mode", "fixed"), case["relative"])
    return {"case": case, "w": w, "pages": list(pages), "slab": slab, "buffers": buffers,
            "eps": [case["eps"]] * pages.shape[0]}


def prepare(case, seed):
    pages = _inputs(case, seed)
    st = _stored(case, pages)
    st["out"] = None
    if case["way"] == "store":
        return st
    family = case["family"]
    if family == "mixed":
        _mixed_store(st)
        st["streams"] = _packed(_wrapper(), st["buffers"], list(st["sizes"]))
        out = torch.zeros_like(pages)
        back = _mixed_tables(case, out)
        back.update(case=case, out=out, streams=st["streams"],
                    sizes=kvszp.u64_array(list(st["sizes"])),
                    bounds=kvszp.f32_array(list(st["bounds"])),
                    stream_table=kvszp.ptr_array([s.data_ptr() for s in st["streams"]]))
        return back
    st["out"] = torch.zeros_like(pages)
    if family == "blocks":
        # other slots of the cache; `dests` pieces of a block lie apart
        g = torch.Generator().manual_seed(seed + 17)
        pieces = list(st["out"].view(pages.shape[0] * case["dests"], -1))
        st["to"] = [pieces[i] for i in torch.randperm(len(pieces), generator=g).tolist()]
    elif family in ("page", "pages32"):
        st["to"] = list(st["out"])
    if case["way"] == "restore":
        done = _store(st)
        st["sizes"] = [int(s) for s in done["sizes"]]
        st["bounds"] = [float(b) for b in done["bounds"]]
        st["streams"] = _packed(_wrapper(), st["buffers"], st["sizes"])
        st["pages"] = st["slab"] = st["buffers"] = None
    return st


def _store(st):
    family = st["case"]["family"]
    if family == "mixed":
        _mixed_store(st)
        return {"sizes": np.frombuffer(st["sizes"], np.int64),
                "bounds": np.frombuffer(st["bounds"], np.float32), "streams": st["slab"]}
    if family == "page":
        ok, _, size, bound = st["w"].compress(st["pages"][0], st["buffers"][0], st["eps"][0])
        sizes, bounds = [size], [bound]
    elif family == "pages32":
        ok, sizes, bounds = st["w"].compress_batch_fixed(st["pages"], st["buffers"], st["eps"])
    else:
        ok, sizes, bounds = st["w"].compress_batch_fixed_bf16(st["pages"], st["buffers"],
                                                              st["eps"])
    assert ok
    st["sizes"], st["bounds"] = sizes, bounds
    return {"sizes": np.array(sizes, np.int64), "bounds": np.array(bounds, np.float32),
            "streams": st["slab"]}


def _restore(st):
    case = st["case"]
    family = case["family"]
    if family == "mixed":
        kvszp.check(st["ctx"].decompress_indexed_scatter_groups(
            st["stream_table"], st["sizes"], st["bounds"], st["batch"], st["page_table"],
            st["index_table"], st["selected"], st["group_sizes"], st["groups"], 2,
            st["layers"], st["per_layer"], torch.cuda.current_stream().cuda_stream))
        return st["out"]
    streams = st.get("streams") or st["buffers"]
    n = st["out"].shape[1]
    if family == "page":
        ok = st["w"].decompress(streams[0], st["sizes"][0], st["to"][0], st["bounds"][0])
    elif family == "pages32":
        ok = st["w"].decompress_batch(streams, st["sizes"], st["to"], st["bounds"])
    elif family == "blocks":
        ok = st["w"].decompress_batch_fixed_bf16_scatter(
            streams, st["sizes"], st["to"], n, case["dests"], n // case["dests"], st["bounds"])
    else:
        ok = st["w"].decompress_batch_fixed_bf16(streams, st["sizes"], st["out"], n,
                                                 st["bounds"])
    assert ok
    return st["out"]


def run(st):
    way = st["case"]["way"]
    if way == "store":
        return _store(st)
    if way == "restore":
        return {"values": _restore(st)}
    out = _store(st)
    out["values"] = _restore(st)
    return out


# ---- what a pass needs, and what it gives --------------------------------------

def work(case):
    """Each value read (written) once, each stream byte written (read) once.
    Stream bytes of a value, measured on these values: a header byte and a
    sign word per 32 values, and 5 to 12 planes by the bound."""
    values = _segments(case) * _values(case)
    per_stream = {1e-3: 0.66, 1e-4: 1.07, 1e-5: 1.37}
    if case["family"] == "mixed":
        stream = 1.15
    elif not case["relative"]:
        stream = {1e-3: 1.6, 1e-4: 1.9, 1e-5: 2.3}[case["eps"]]
    else:
        stream = per_stream[case["eps"]]
    wide = 4 if case["family"] in ("page", "pages32") else 2
    passes = 2 if case["way"] == "step" else 1
    return {"bytes": passes * values * (wide + stream), "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Bounds and restored values in 64 bits; sizes and stream bytes have no
    such value (they follow the 32-bit quantizer)."""
    pages = _inputs(case, seed)
    if case["family"] == "mixed":
        per_layer = case["tokens"] * case["heads"] * case["dim"]
        parts = [(b, pages.view(pages.shape[0], 2, case["layers"], per_layer), list(layers))
                 for b, layers in _groups(case)]
    else:
        parts = [(case["eps"], pages.view(pages.shape[0], 1, 1, -1), [0])]
    bounds, values = [], None
    want_values = case["way"] != "store"
    if want_values:
        values = torch.empty(parts[0][1].shape, dtype=torch.float64, device="cuda")
    for eps, view, layers in parts:
        eps = float(np.float32(eps))
        for i in range(view.shape[0]):
            x = view[i][:, layers].double()
            eb = eps
            if case.get("relative", True):
                eb = eps * max(float(x.max() - x.min()), float(np.float32(1e-6)))
            bounds.append(eb)
            if want_values:
                q = (x / (2 * eb) + 0.5).floor_().clamp_(-2147483647, 2147483647)
                values[i][:, layers] = q * (2 * eb)
    if want_values:
        values = values.view(pages.shape)
        if case["family"] == "blocks":
            g = torch.Generator().manual_seed(seed + 17)
            order = torch.randperm(pages.shape[0] * case["dests"], generator=g)
            out = torch.empty_like(values)
            out.view(len(order), -1)[order.cuda()] = values.view(len(order), -1)
            values = out
    stored = {"sizes": None, "bounds": np.array(bounds), "streams": None}
    if case["way"] == "store":
        return stored
    if case["way"] == "restore":
        return {"values": values}
    return dict(stored, values=values)
