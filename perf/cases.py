"""The measured work of this library: restoring tensors from their encoded planes and encoding them, through the
entry points of ``ptwm_amd.api``, in the formats that programs keep weights in.

A case is one call (a pass) of one program:

- ``decode``: a compressed model, layer or tensor lies in HBM and is restored into HBM through
  ``hardware_backend_dispatch_decode_cuda`` with its decode plan.  Plane CRC-32s are in the plan and checked by the
  call, as the container decode does by default (crates/ptwm-core/src/container.rs:2154-2159), unless the case says
  otherwise.  The tensor hash (XXH64, serial by its definition) is computed on host cores from a copy of the restored
  bytes; that option is bound by the copy to the host and is not among the cases.
- ``encode``: tensors in HBM are split and coded into a buffer in HBM, through ``encode_tensors_cuda`` (several
  tensors), ``encode_tensor_cuda`` (one) or ``encode_tensor_ref_cuda`` (the reference's own plane formats).

The library's formats are ``huff_ilv`` and ``rans_ilv``; ``reference`` stands for the reference's Huffman and rANS
planes, in chunks (256 KiB is its default compression chunk) or as one payload a plane.
"""
import math

import numpy as np
import torch

from ptwm_amd import api, ids, plan

DEVICE = "cuda:0"
HUFFMAN, RANS = 1, 3  # codec wire ids (crates/ptwm-core/src/codec.rs:7-9)

# By tensor kind: the chain that a container gives it, and its planes' codecs in the reference's formats (the exponent
# plane of fp32 takes rANS, every other plane Huffman).
CHAIN = {"bf16": plan.CHAIN_IEEE16_SPLIT2, "fp32": plan.CHAIN_IEEE32_SPLIT4, "e4m3": plan.CHAIN_E4M3_NIBBLE,
         "fp4": plan.CHAIN_NIBBLE_SPLIT, "e8m0": plan.CHAIN_PASSTHROUGH}
REFERENCE = {"bf16": [HUFFMAN, HUFFMAN], "fp32": [HUFFMAN, HUFFMAN, HUFFMAN, RANS], "e4m3": [HUFFMAN, HUFFMAN],
             "fp4": [HUFFMAN, HUFFMAN], "e8m0": [HUFFMAN]}
BYTES = {"bf16": 2, "fp32": 4, "e4m3": 1, "mxfp4": 1}

# Encoded bytes over raw bytes of the distributions below (they hardly depend on the size).
RATIO = {("huff_ilv", "bf16"): 0.684, ("huff_ilv", "fp32"): 0.844, ("huff_ilv", "e4m3"): 0.856,
         ("huff_ilv", "mxfp4"): 0.963, ("rans_ilv", "bf16"): 0.666, ("rans_ilv", "fp32"): 0.831,
         ("rans_ilv", "e4m3"): 0.831, ("rans_ilv", "mxfp4"): 0.958, ("reference", "bf16"): 0.678,
         ("reference", "fp32"): 0.830, ("reference", "e4m3"): 0.847, ("reference", "mxfp4"): 0.963}


def case(op, codec, dtype, rows, cols, name=None, layers=0, chunk=0, crc=True):
    """`rows` x `cols` is one tensor's shape; with `layers`, the feed-forward and hidden sizes of that many decoder
    layers."""
    c = {"op": op, "codec": codec, "dtype": dtype, "rows": rows, "cols": cols, "layers": layers, "chunk": chunk,
         "crc": crc}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # Random access to the smallest tensor of a model, a norm weight of 4096 values: latency and launches.
        case("decode", "huff_ilv", "bf16", 1, 4096, "decode norm weight"),
        # Random access to a small matrix.
        case("decode", "huff_ilv", "bf16", 1024, 1024, "decode bf16 1024x1024"),
        # Loading a model: four layers of the Llama-3-8B-shaped model (36 tensors, 1.74 GB) in one call.
        case("decode", "huff_ilv", "bf16", 14336, 4096, "decode bf16 4 layers", layers=4),
        # An fp8 checkpoint's large matrix.
        case("decode", "huff_ilv", "e4m3", 8192, 8192, "decode e4m3 8192x8192"),
        # An fp32 tensor in the denser of the library's two formats.
        case("decode", "rans_ilv", "fp32", 4096, 4096, "decode fp32 4096x4096 rans"),
        # MXFP4 weights with their block scales, two tensors in one call, not verified (a reload of checked bytes).
        case("decode", "huff_ilv", "mxfp4", 14336, 2048, "decode mxfp4 14336x2048", crc=False),
        # Writing a model: two layers in one batched call.
        case("encode", "huff_ilv", "bf16", 14336, 4096, "encode bf16 2 layers", layers=2),
        # Writing one fp8 tensor of odd sizes in the denser format.
        case("encode", "rans_ilv", "e4m3", 5001, 3333, "encode e4m3 5001x3333 rans"),
        # A layer of a bf16 model that the reference wrote, in its default chunks.
        case("decode", "reference", "bf16", 14336, 4096, "decode reference bf16 layer", layers=1, chunk=256 << 10),
        # An fp32 tensor that the reference wrote with a rANS exponent plane.
        case("decode", "reference", "fp32", 4096, 4096, "decode reference fp32", chunk=256 << 10),
        # An fp8 tensor that the reference wrote with one payload a plane.
        case("decode", "reference", "e4m3", 8192, 8192, "decode reference e4m3"),
        # Writing an fp32 tensor for the reference to read.
        case("encode", "reference", "fp32", 4096, 4096, "encode reference fp32", chunk=256 << 10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "decode", "encode"])
    codec = rng.choice(["huff_ilv", "huff_ilv", "rans_ilv", "reference"])
    dtype = rng.choice(["bf16", "bf16", "fp32", "e4m3", "mxfp4"])
    chunk = 0
    if codec == "reference":  # a rANS plane comes in chunks, another one may come whole
        chunk = rng.choice([64, 128, 256, 512]) << 10
        if dtype != "fp32" and rng.random() < 0.4:
            chunk = 0
    crc = rng.random() < 0.75
    if dtype == "bf16" and rng.random() < 0.4:
        hidden = 128 * rng.randint(4, 32)
        inner = hidden * 7 // 2
        most = 1 if codec == "reference" else 4 if op == "decode" else 2
        return case(op, codec, dtype, inner, hidden, layers=rng.randint(1, most), chunk=chunk, crc=crc)
    most = 32 << 20 if dtype == "mxfp4" else 64 << 20
    n = _log_int(rng, 4096, most // BYTES[dtype])
    cols = min(n, _log_int(rng, 64, 16384))
    if dtype == "mxfp4":
        cols = max(16, cols // 16 * 16)  # a scale for every 32 values, 16 bytes
    return case(op, codec, dtype, max(1, n // cols), cols, chunk=chunk, crc=crc)


def _shapes(c):
    """(kind, shape) of every tensor of a case."""
    if c["layers"]:
        inner, hidden = c["rows"], c["cols"]
        layer = [(hidden, hidden), (hidden // 4, hidden), (hidden // 4, hidden), (hidden, hidden), (inner, hidden),
                 (inner, hidden), (hidden, inner), (hidden,), (hidden,)]
        return [("bf16", s) for _ in range(c["layers"]) for s in layer]
    if c["dtype"] == "mxfp4":
        return [("fp4", (c["rows"], c["cols"])), ("e8m0", (c["rows"], c["cols"] // 16))]
    return [(c["dtype"], (c["rows"], c["cols"]))]


def _tensor(kind, shape, g):
    """The raw bytes of one tensor: weights are N(0, 0.02), norm weights 1 +- 0.01."""
    if kind == "bf16" and (len(shape) == 1 or shape[0] == 1):
        t = (1 + 0.01 * (2 * torch.rand(shape, generator=g, device=DEVICE) - 1)).to(torch.bfloat16)
    elif kind == "bf16":
        t = (torch.randn(shape, generator=g, device=DEVICE) * 0.02).to(torch.bfloat16)
    elif kind == "fp32":  # one value in a hundred an outlier
        t = torch.randn(shape, generator=g, device=DEVICE) * 0.02
        t = torch.where(torch.rand(shape, generator=g, device=DEVICE) < 0.01, t * 50, t)
    elif kind == "e4m3":  # rows scaled to the type's range
        t = torch.randn(shape, generator=g, device=DEVICE)
        t = (t / t.abs().amax(1, keepdim=True) * 448).to(torch.float8_e4m3fn)
    elif kind == "fp4":  # two nearly uniform codes a byte
        t = torch.randint(0, 256, shape, generator=g, device=DEVICE, dtype=torch.uint8)
    else:  # block scale exponents
        t = torch.round(torch.randn(shape, generator=g, device=DEVICE) * 1.5 - 6) + 127
        t = t.clamp(0, 255).to(torch.uint8)
    return t.contiguous().view(torch.uint8).reshape(-1)


def _encode_all(c, items, out):
    """Every tensor's planes in `out`, and the plan that restores the tensors at 256-byte boundaries."""
    if c["codec"] != "reference":
        used, state = api.encode_tensors_cuda([(CHAIN[k], t) for k, t in items], out, 0, codec=c["codec"])
        return used, plan.decode_plan(state)
    at = restored = 0
    plans = []
    for kind, t in items:
        used, state = api.encode_tensor_ref_cuda(CHAIN[kind], REFERENCE[kind], c["chunk"], t, out[at:], 0)
        p = plan.decode_plan(state)[0]
        p.out_offset = restored
        for q in p.planes:
            q.payload_offset += at
        plans.append(p)
        at = (at + used + 255) // 256 * 256
        restored = (restored + t.numel() + 255) // 256 * 256
    return at, plans


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    items = [(kind, _tensor(kind, shape, g)) for kind, shape in _shapes(case)]
    raw = sum(t.numel() for _, t in items)
    out = torch.zeros(raw + raw // 16 + 65536 * len(items) + (1 << 20), dtype=torch.uint8, device=DEVICE)
    if case["op"] == "encode":
        return {"case": case, "items": items, "out": out}
    used, plans = _encode_all(case, items, out)
    if case["crc"]:
        for (kind, t), p in zip(items, plans):
            for q, crc in zip(p.planes, api.plane_crc32_cuda(CHAIN[kind], t, 0)):
                q.crc32 = crc
    restored = plans[-1].out_offset + plans[-1].out_len
    return {"case": case, "planes": out[:used].clone(), "plan": plan.encode_plan(plans),
            "out": torch.zeros(restored, dtype=torch.uint8, device=DEVICE)}


def run(state):
    c = state["case"]
    if c["op"] == "decode":
        api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL, state["plan"],
                                                  state["planes"], state["out"], 0)
        return state["out"]
    items, out = state["items"], state["out"]
    if c["codec"] == "reference":
        at, plans = 0, []
        for kind, t in items:
            used, p = api.encode_tensor_ref_cuda(CHAIN[kind], REFERENCE[kind], c["chunk"], t, out[at:], 0)
            at = (at + used + 255) // 256 * 256
            plans.append(p)
        used, p = at, b"".join(plans)
    elif len(items) == 1:
        used, p = api.encode_tensor_cuda(CHAIN[items[0][0]], items[0][1], out, 0, codec=c["codec"])
    else:
        used, p = api.encode_tensors_cuda([(CHAIN[k], t) for k, t in items], out, 0, codec=c["codec"])
    return {"planes": out, "used": used, "plan": np.frombuffer(p, np.uint8)}  # the buffer is zero past `used`


def work(case):
    raw = sum(math.prod(shape) * BYTES.get(kind, 1) for kind, shape in _shapes(case))
    return {"bytes": raw * (1 + RATIO[case["codec"], case["dtype"]]), "flops": 0}


def tolerance(case):
    return "exact"  # bytes in, bytes out
