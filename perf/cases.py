"""The performance cases of the FP8 + Huffman and AWQ int4 + Huffman weight paths.

A user of this framework decodes weights (one call a weight, one plan launch a
layer or a pipeline stage) and builds sidecars (one call a weight). The cases
run each of these through the public entry points: the ``MPServe_cuda`` ops,
``DecodePlan`` and ``AwqDecodePlan``, from the smallest weight to the layers and
the stage that a serving program decodes at once.

Every path is lossless integer work, so every tolerance is ``"exact"``.

A case is a dict of plain values:

``kind``      what one pass is:
              ``fp8_op``      huffman_decode_fp8 on a weight that is decoded again and again
                              (a serving loop: the op keeps that weight's plan);
              ``fp8_once``    huffman_decode_fp8 on a weight that is decoded once (a loader);
              ``fp8_plan``    one DecodePlan launch over many weights;
              ``fp8_encode``  huffman_build_fp8_decode_tables of one weight;
              ``awq_op``, ``awq_plan``, ``awq_encode``: the same for the AWQ int4 variants.
``n``, ``m``  shape of the weight (ops and builders).
``k``         substreams a bucket (threads_per_block).
``block``     FP8: 0 for one scale a row, else the side of the square scale blocks.
``group``     AWQ: columns a quantisation group (by-scale sidecar); 0 for one
              scale a row and the row-bucket sidecar.
``outliers``  share of elements at +-8 sigma (their keys need ESC codes).
``hidden``, ``kv``, ``ffn``, ``layers``, ``vocab``: plans: widths of the layers'
              seven linear weights, and an output head of vocab x hidden (0: none).
"""
from __future__ import annotations

import torch

import MPServe_cuda
from mpserve_amd.awq import AwqDecodePlan
from mpserve_amd.decode import DecodePlan, sidecar_decode_args

DEVICE = "cuda"
FP8_MAX = 448.0


def _op(kind, n, m, k, block=0, group=0, outliers=0.0):
    return {"kind": kind, "n": n, "m": m, "k": k, "block": block, "group": group, "outliers": outliers}


def _plan(kind, hidden, kv, ffn, layers, vocab, k, group=0, outliers=0.0):
    return {"kind": kind, "hidden": hidden, "kv": kv, "ffn": ffn, "layers": layers, "vocab": vocab, "k": k,
            "group": group, "outliers": outliers}


def listed():
    return [
        # The smallest weight that fills a row of substreams: the call's own latency counts.
        dict(_op("fp8_op", 256, 1024, 1024), name="fp8_op_smallest"),
        # A loader that decodes each weight once, a k or v projection of an 8B layer: no plan exists yet.
        dict(_op("fp8_once", 1024, 4096, 1024), name="fp8_once_kv"),
        # A weight whose columns are no multiple of the substreams (widths that are not powers of two).
        dict(_op("fp8_op", 3001, 5000, 1024), name="fp8_op_ragged"),
        # A checkpoint with 128 x 128 scale blocks, one attention projection.
        dict(_op("fp8_op", 4096, 4096, 1024, block=128), name="fp8_op_block128"),
        # One 8B decoder layer, decoded as a serving engine does before the layer's products.
        dict(_plan("fp8_plan", 4096, 1024, 14336, 1, 0, 1024), name="fp8_layer8b"),
        # One 70B decoder layer whose weights have outliers (ESC codes).
        dict(_plan("fp8_plan", 8192, 1024, 28672, 1, 0, 1024, outliers=1e-3), name="fp8_layer70b_esc"),
        # The last of four pipeline stages of an 8B model: eight layers and the output head.
        dict(_plan("fp8_plan", 4096, 1024, 14336, 8, 128256, 1024), name="fp8_stage8b"),
        # Offline compression: the smallest weight of a layer at the builder's default of 256 substreams,
        dict(_op("fp8_encode", 1024, 4096, 256), name="fp8_encode_kv"),
        # and the largest, at the compressor's default of 1024.
        dict(_op("fp8_encode", 14336, 4096, 1024), name="fp8_encode_gate"),
        # One 8B layer from an AWQ int4 checkpoint with 128-column groups.
        dict(_plan("awq_plan", 4096, 1024, 14336, 1, 0, 1024, group=128), name="awq_layer8b"),
        # One AWQ projection with a scale a row, at the builder's default of 256 substreams.
        dict(_op("awq_op", 4096, 4096, 256), name="awq_op_rows"),
        # Offline compression of one AWQ projection.
        dict(_op("awq_encode", 4096, 4096, 1024, group=128), name="awq_encode_q"),
    ]


def _log_between(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.choice(["fp8_op", "fp8_op", "fp8_once", "fp8_plan", "fp8_encode", "fp8_encode", "awq_op", "awq_plan",
                       "awq_encode"])
    k = rng.choice([256, 512, 1024, 1024])
    if kind in ("fp8_plan", "awq_plan"):
        hidden = 128 * int(_log_between(rng, 4, 48))
        kv = max(128, hidden // rng.choice([1, 2, 4, 8]) // 128 * 128)
        ffn = max(128, int(hidden * rng.choice([2.5, 2.75, 3.5])) // 128 * 128)
        awq = kind == "awq_plan"
        return _plan(kind, hidden, kv, ffn, rng.choice([1, 1, 2]), 0, k, group=rng.choice([128, 128, 0]) if awq else 0,
                     outliers=0.0 if awq else rng.choice([0.0, 0.0, 1e-3]))
    n = int(_log_between(rng, 64, 14336))
    m = int(_log_between(rng, 256, 14336))
    while n * m > 58_000_000:
        n = (n + 1) // 2
    form = rng.choice(["odd", "ragged", "even", "even"])  # columns: any, a multiple of 8, a multiple of 1024 (256 below it)
    if form == "ragged":
        m = max(8, m // 8 * 8)
    elif form == "even":
        m = m // 1024 * 1024 if m >= 1024 else m // 256 * 256
    block = group = 0
    outliers = 0.0
    if kind.startswith("fp8"):
        if rng.random() < 0.25:
            block = 128
            n, m = max(1, n // 128) * 128, max(2, m // 128) * 128
        elif rng.random() < 0.3:
            outliers = 1e-3
    elif rng.random() < 0.6:
        group = rng.choice([128, 128, 64])
        m = max(1, m // group) * group
    return _op(kind, n, m, k, block=block, group=group, outliers=outliers)


# --------------------------------------------------------------------------- inputs
def _shapes(case):
    """(n, m) of every weight of the case, in order."""
    if "hidden" not in case:
        return [(case["n"], case["m"])]
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    layer = [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f)]
    head = [(case["vocab"], h)] if case["vocab"] else []
    return layer * case["layers"] + head


def _weight(n, m, outliers, seed):
    """A BF16 weight as trained models have them: normal, with (optionally) rare outliers of 8 sigma."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    sigma = 0.015 if outliers else 0.02
    w = torch.randn((n, m), generator=g, device=DEVICE).mul_(sigma)
    if outliers:
        u = torch.rand((n, m), generator=g, device=DEVICE)
        w = torch.where(u < outliers, torch.where(u < 0.5 * outliers, -8.0 * sigma, 8.0 * sigma), w)
    return w.to(torch.bfloat16)


def _fp8(w, block):
    """(e4m3 bytes, 16-bit scale keys): absmax / 448 of a row or of a block, keyed by its FP16 bits."""
    n, m = w.shape
    f = w.float()
    if block:
        t = f.view(n // block, block, m // block, block)
        s = t.abs().amax(dim=(1, 3)) / FP8_MAX
        q = t / s[:, None, :, None]
    else:
        s = f.abs().amax(dim=1) / FP8_MAX
        q = f / s[:, None]
    q = q.clamp_(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn).view(torch.uint8).reshape(n, m)
    return q.contiguous(), s.to(torch.float16).view(torch.uint16)


def _int4(w, group):
    """(int4 values 0..15, BF16 scale bits): absmax / 7 of a group or of a row, zero point 8."""
    n, m = w.shape
    f = w.float().view(n, m // group, group) if group else w.float().view(n, 1, m)
    s = (f.abs().amax(dim=2) / 7.0).to(torch.bfloat16)
    q = (torch.round(f / s.float()[:, :, None]) + 8).clamp_(0, 15).to(torch.uint8).reshape(n, m)
    key = s.view(torch.uint16)
    return q.contiguous(), key.contiguous() if group else key.reshape(n).contiguous()


def _build(case, w, q, key):
    if case["kind"].startswith("fp8"):
        return MPServe_cuda.huffman_build_fp8_decode_tables(w, q, key, 7, case["k"])
    if case["group"]:
        return MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables_by_scale(w, q, key, 11, case["k"], 1024)
    return MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables(w, q, key, 11, case["k"])


# what a program keeps of a sidecar to decode with it
_KEEP = ("bitstream_u64", "decode_syms_u16", "decode_lens_u8", "bucket_table_i32", "bucket_col_start_i32",
         "bucket_col_len_i32", "bucket_row_offsets_i32", "row_indices_i32", "bucket_thread_startbit_u32",
         "bucket_bit_base_i64", "bucket_group_offsets_i32", "group_rows_i32", "group_col_start_i32", "shape_nmkg_i64")


def _awq_args(q, sc, group):
    n, m = q.shape
    if group:
        return (q, sc["bitstream_u64"], sc["decode_syms_u16"], sc["decode_lens_u8"], sc["bucket_table_i32"],
                sc["bucket_group_offsets_i32"], sc["group_rows_i32"], sc["group_col_start_i32"],
                sc["bucket_thread_startbit_u32"], sc["bucket_bit_base_i64"], n, m, 11, group)
    return (q, sc["bitstream_u64"], sc["decode_syms_u16"], sc["decode_lens_u8"], sc["bucket_table_i32"],
            sc["bucket_col_start_i32"], sc["bucket_col_len_i32"], sc["bucket_row_offsets_i32"], sc["row_indices_i32"],
            sc["bucket_thread_startbit_u32"], sc["bucket_bit_base_i64"], n, m, 11)


def _arena_bytes(case):
    """Room for any sidecar of the case: about 100 scales occur (a bucket holds at most 128 rows, or 1024 groups, of
    one scale); 400 are allowed for."""
    n, m, k = case["n"], case["m"], case["k"]
    fp8 = case["kind"].startswith("fp8")
    if case["block"]:
        buckets = (n // 128) * (m // 128)
    else:
        buckets = min(n * m, 400) + (n * (m // case["group"]) // 1024 if case["group"] else n // 128)
    tables = 400 * (256 * 196 if fp8 else 16 * 5124)
    return 2 * n * m + tables + buckets * (4 * (k + 1) + 4096) + 16 * n * max(1, m // 64)


def prepare(case, seed):
    kind = case["kind"]
    quantise = (lambda w: _fp8(w, case.get("block", 0))) if kind.startswith("fp8") else (lambda w: _int4(w, case["group"]))
    items = []
    for i, (n, m) in enumerate(_shapes(case)):
        w = _weight(n, m, case["outliers"], seed * 1009 + i)
        q, key = quantise(w)
        if kind.endswith("encode"):
            arena = torch.zeros(_arena_bytes(case), dtype=torch.uint8, device=DEVICE)
            return {"kind": kind, "args": (w, q, key), "case": case, "arena": arena}
        sc = _build(case, w, q, key)
        out = torch.empty((n, m), dtype=torch.bfloat16, device=DEVICE)
        items.append((q, {x: sc[x] for x in _KEEP if x in sc}, out))
    if kind == "fp8_plan":
        return {"kind": kind, "plan": DecodePlan(items)}
    if kind == "awq_plan":
        return {"kind": kind, "plan": AwqDecodePlan(items)}
    q, sc, out = items[0]
    args = _awq_args(q, sc, case["group"]) if kind == "awq_op" else sidecar_decode_args(q, sc)
    return {"kind": kind, "args": args, "out": out, "by_scale": bool(case["group"])}


def run(state):
    kind = state["kind"]
    if kind.endswith("plan"):
        return list(state["plan"].decode())
    if kind.endswith("encode"):
        # a compressor lays a weight's sidecar tensors into one buffer, as they go into the file
        sc = _build(state["case"], *state["args"])
        parts = [t.reshape(-1).view(torch.uint8) for t in sc.values()]
        torch.cat(parts, out=state["arena"][:sum(p.numel() for p in parts)])
        return state["arena"]
    if kind == "awq_op":
        op = (MPServe_cuda.huffman_decode_awq_int4_bucket_by_scale if state["by_scale"]
              else MPServe_cuda.huffman_decode_awq_int4_bucket)
        return op(*state["args"], out=state["out"])
    if kind == "fp8_once":
        MPServe_cuda.clear_decode_plans()  # the op has not met this weight
    return MPServe_cuda.huffman_decode_fp8(*state["args"], out=state["out"])


def work(case):
    """Bytes: the low-bit values, the coded symbols, the code tables and the BF16 weights, each once. A normal
    weight codes in about 4 bits an element (FP8; 230 tables a scale, about 80 distinct row or block scales) or
    7.2 bits (AWQ; 16 tables a scale, about 160 distinct group scales)."""
    fp8 = case["kind"].startswith("fp8")
    total = 0
    for n, m in _shapes(case):
        if fp8:
            b = case.get("block", 0)
            scales = 1 if case["outliers"] else min(80, (n // b) * (m // b) if b else n)
            total += n * m * (1 + 0.5 + 2) + scales * 230 * 192
        else:
            scales = min(160, n * m // case["group"] if case["group"] else n)
            total += n * m * (1 + 0.9 + 2) + scales * 16 * 3072
        # a builder reads the weight and the low-bit values and writes the coded symbols and the tables: the same bytes
    return {"bytes": int(total), "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The decode is lossless: its result is the weight itself. The row-bucket AWQ coding is not (an element
    equal to its key's escape symbol is lost), and a builder's outputs are codes and tables, whole numbers."""
    kind = case["kind"]
    if kind.endswith("encode") or (kind.startswith("awq") and not case["group"]):
        return None
    ws = [_weight(n, m, case["outliers"], seed * 1009 + i).double() for i, (n, m) in enumerate(_shapes(case))]
    return ws if kind.endswith("plan") else ws[0]
