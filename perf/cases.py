"""What the speed of this library is measured on: the calls that an archiver of quantized models makes
while it packs and extracts, over the sizes, types and options it makes them with.

  regrow     a tensor's quantization regrown from its base weights (every file of a pack and of an
             extract, every tensor: most of the device time of both)
  dequant    a quantized tensor widened to float32 (a seed that other files are regrown from)
  qr_encode  the residual of a regrown tensor coded against the file's own bytes (pack)
  qr_decode  the same read back (extract)
  r2_decode  BF16 base tensors decoded into device memory (the start of every extract)

Tensors are resident on the device, as the pack and the extract hold them; where a path takes host
data by its nature (coded streams, tables) it is host data here too.
"""
import math

import numpy as np
import torch

from seedpack_amd import device as dev
from seedpack_amd import qr, r2
from seedpack_amd.gpuquant import GPUQuant, quantize_into
from seedpack_amd.requant import BY_NAME, NEED_IMATRIX, QFUN

QUANTS = sorted(BY_NAME)
LATTICE = {"IQ2_XXS", "IQ2_XS", "IQ2_S", "IQ3_XXS", "IQ3_S", "IQ1_S", "IQ1_M"}
LEGACY = {"Q8_0", "Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q2_0"}
DEQUANT = ["Q8_0", "Q4_0", "Q4_K", "Q6_K"]           # the types that serve as seeds most often
SRC = {"bf16": (np.uint16, 2), "f16": (np.float16, 2), "f32": (np.float32, 4)}


# ------------------------------------------------------------------------------------------ the cases

def listed():
    def regrow(name, quant, rows, cols, imatrix=True, src="bf16", dist="normal"):
        return {"name": name, "op": "regrow", "quant": quant, "rows": rows, "cols": cols, "imatrix": imatrix,
                "src": src, "dist": dist}

    return [
        # a small model's key projection: the call is over before the device is full
        regrow("q4_k-small", "Q4_K", 256, 1024),
        # the most common quant on a large feed-forward matrix
        regrow("q4_k-ffn", "Q4_K", 12288, 4096),
        # the embedding / output of a Q4_K_M file: its largest tensor
        regrow("q6_k-embedding", "Q6_K", 151936, 1024),
        # the largest 8-bit tensor, without an importance matrix
        regrow("q8_0-embedding", "Q8_0", 151936, 1024, imatrix=False),
        # a non-linear 4-bit attention projection
        regrow("iq4_xs-attn", "IQ4_XS", 4096, 4096, dist="student"),
        # low-bit lattice quants: the slowest regrowths of an archive
        regrow("iq2_xs-ffn", "IQ2_XS", 4096, 12288, dist="student"),
        regrow("iq3_xxs-ragged", "IQ3_XXS", 2053, 3584, dist="student"),
        regrow("iq1_s-attn", "IQ1_S", 4096, 4096, dist="student"),
        # a 6-bit embedding widened to be the seed of other files
        {"name": "dequant-q6_k", "op": "dequant", "quant": "Q6_K", "rows": 151936, "cols": 1024},
        # residual coding, one batch of one tensor: a lattice type and a K-quant
        {"name": "qr_encode-iq2_xs", "op": "qr_encode", "quant": "IQ2_XS", "rows": 4096, "cols": 4096, "changed": 0.01},
        {"name": "qr_decode-q4_k", "op": "qr_decode", "quant": "Q4_K", "rows": 12288, "cols": 4096, "changed": 0.01},
        # the attention matrices of one block of the base
        {"name": "r2_decode-attn", "op": "r2_decode", "rows": 4096, "cols": 4096, "kv": 1024},
    ]


def _shape(rng, least, most, step, cols_most=16384):
    """rows and columns of a matrix of about least..most weights (even over the logarithm): columns a
    multiple of step, rows anything"""
    n = math.exp(rng.uniform(math.log(least), math.log(most)))
    cols = step * rng.randint(1, max(1, cols_most // step))
    while cols > n / 4 and cols > step:
        cols = step * max(1, cols // (2 * step))
    return max(1, int(n // cols)), cols


def draw(rng):
    op = rng.choices(["regrow", "dequant", "qr_encode", "qr_decode", "r2_decode"], [70, 8, 8, 8, 6])[0]
    if op == "regrow":
        quant = rng.choice(QUANTS)
        qk = QFUN[BY_NAME[quant]][1]
        rows, cols = _shape(rng, 1 << (21 if quant in LEGACY else 18), 40e6 if quant in LATTICE else 120e6, qk)
        return {"op": op, "quant": quant, "rows": rows, "cols": cols,
                "imatrix": BY_NAME[quant] in NEED_IMATRIX or rng.random() < 0.85,
                "src": rng.choices(["bf16", "f16", "f32"], [80, 10, 10])[0], "dist": rng.choice(["normal", "student"])}
    if op == "dequant":
        quant = rng.choice(DEQUANT)
        rows, cols = _shape(rng, 1 << 22, 120e6, QFUN[BY_NAME[quant]][1])
        return {"op": op, "quant": quant, "rows": rows, "cols": cols}
    if op == "r2_decode":
        rows, cols = _shape(rng, 1 << 20, 10e6, 64, 8192)
        return {"op": op, "rows": rows, "cols": cols, "kv": max(1, rows // rng.choice([1, 2, 4, 8]))}
    quant = rng.choice(QUANTS)
    rows, cols = _shape(rng, 1 << 19, 14e6 if quant in LATTICE else 40e6, QFUN[BY_NAME[quant]][1])
    return {"op": op, "quant": quant, "rows": rows, "cols": cols, "changed": rng.choice([0.002, 0.01, 0.03])}


# ------------------------------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weights(g, rows, cols, dist):
    """float32 weights: N(0, 0.02) with a few outliers, or Student-t (5 degrees of freedom)"""
    n = rows * cols
    x = torch.randn(n, generator=g, device="cuda")
    if dist == "student":
        chi = torch.zeros(n, device="cuda")
        for _ in range(5):
            chi += torch.randn(n, generator=g, device="cuda").square_()
        return x.div_(chi.div_(5).sqrt_()).mul_(0.015 * math.sqrt(3 / 5))
    x.mul_(0.02)
    hit = torch.rand(n, generator=g, device="cuda") < 1e-3
    return torch.where(hit, torch.randn(n, generator=g, device="cuda") * 0.2, x)


def _stored(x, src):
    return x.to({"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[src])


def _importance(g, cols):
    return torch.randn(cols, generator=g, device="cuda").exp_()


def _array(t, dtype):
    """the library's view of a tensor's memory"""
    return dev.DeviceArray(t.numel() * t.element_size() // np.dtype(dtype).itemsize, dtype, ptr=t.data_ptr(), owner=t)


class _Memory:
    """a DeviceArray's bytes as torch takes them over (the array stays alive with the tensor)"""

    def __init__(self, a, dtype="|u1"):
        self.array = a
        self.__cuda_array_interface__ = {"shape": (a.nbytes,), "typestr": dtype, "data": (a.ptr, False), "version": 2}


def _tensor(a):
    return torch.as_tensor(_Memory(a), device="cuda")


def _blocks(g, quant, n):
    """n random blocks of a type: any codes, fp16 scales of the size real tensors have"""
    bs = QFUN[BY_NAME[quant]][2]
    b = torch.randint(256, (n, bs), generator=g, device="cuda", dtype=torch.uint8)
    at = {"Q8_0": [0], "Q4_0": [0], "Q4_K": [0, 2], "Q6_K": [208]}[quant]
    for o in at:
        d = (torch.rand(n, generator=g, device="cuda") * 4e-3 + 1e-4).half()
        b[:, o:o + 2] = d.view(torch.uint8).reshape(n, 2)
    return b


def prepare(case, seed):
    op, g = case["op"], _generator(seed)
    rows, cols = case["rows"], case["cols"]
    if op == "r2_decode":
        kv = case["kv"]
        shapes = [("attn_q", rows, cols), ("attn_k", kv, cols), ("attn_v", kv, cols), ("attn_output", rows, cols)]
        parts = [_stored(_weights(g, r, c, "normal"), "bf16") for _, r, c in shapes]
        at, tensors = 0, []
        for (name, r, c), w in zip(shapes, parts):
            tensors.append(("blk.0.%s.weight" % name, at, 2 * r * c, c))
            at += 2 * r * c
        layout = r2.layout_of(tensors, at)
        file = torch.cat(parts).view(torch.uint8)
        torch.cuda.synchronize()
        coded = r2.BF16v2().compress(_array(file, np.uint8), layout)
        return {"op": op, "codec": r2.BF16v2(), "parts": {k: coded[k] for k in ("meta", "side", "tables", "lens", "stream")}}
    T = BY_NAME[case["quant"]]
    _, qk, bs = QFUN[T]
    n = rows * cols
    if op == "dequant":
        blocks = _blocks(g, case["quant"], n // qk)
        out = torch.empty(n, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        return {"op": op, "gq": GPUQuant(), "type": T, "cols": cols, "src": _array(blocks, np.uint8), "out": out,
                "dst": _array(out, np.float32)}
    src = case.get("src", "bf16")
    w = _stored(_weights(g, rows, cols, case.get("dist", "student")), src)
    imx = _importance(g, cols) if case.get("imatrix", True) else None
    out = torch.empty(n // qk * bs, dtype=torch.uint8, device="cuda")
    s = {"op": op, "type": T, "cols": cols, "src": _array(w, SRC[src][0]), "out": out, "dst": _array(out, np.uint8),
         "imx": None if imx is None else _array(imx, np.float32)}
    torch.cuda.synchronize()
    if op == "regrow":
        return s
    # the file: the regrown tensor with one byte changed in some of its blocks
    quantize_into(T, s["src"], cols, s["dst"], s["imx"])
    torch.cuda.synchronize()
    file = out.clone().view(-1, bs)
    hit = torch.nonzero(torch.rand(len(file), generator=g, device="cuda") < case["changed"]).reshape(-1)
    file[hit, torch.randint(bs, (len(hit),), generator=g, device="cuda")] ^= 0x21
    torch.cuda.synchronize()
    s["file"] = _array(file, np.uint8)
    s["seed"] = _array(w, np.uint8)
    s["where"] = (0, 30, cols, 0 if T in qr.GRID_TYPES else -1)
    # room for the coded stream: the changed blocks twice over and 64 bytes a segment
    s["coded"] = np.empty(int(2 * case["changed"] * file.numel()) + 64 * (n // 16384 + 64), np.uint8)
    if op == "qr_decode":
        p = qr.encode_parts(T, [(s["file"], s["dst"]) + s["where"]], s["seed"], s["imx"])
        s["parts"] = (p["freq"], p["used"], p["lens"], p["stream"].tobytes())
    return s


# ------------------------------------------------------------------------------------------ one pass

def run(s):
    op = s["op"]
    if op == "regrow":
        quantize_into(s["type"], s["src"], s["cols"], s["dst"], s["imx"])
        return s["out"]
    if op == "dequant":
        s["gq"].dequantize(s["type"], s["src"], s["cols"], out=s["dst"])
        return s["out"]
    if op == "qr_encode":
        p = qr.encode_parts(s["type"], [(s["file"], s["dst"]) + s["where"]], s["seed"], s["imx"])
        # the frequencies follow from the counts; the stream's length is the data's, its room the case's
        s["coded"][:len(p["stream"])] = p["stream"]
        s["coded"][len(p["stream"]):] = 0
        return {"counts": p["counts"], "lens": p["lens"], "stream": s["coded"]}
    if op == "qr_decode":
        return _tensor(qr.decode_parts(s["type"], *s["parts"], [(s["dst"],) + s["where"]], s["seed"], s["imx"]))
    return _tensor(s["codec"].decompress(s["parts"], device=True))


# ------------------------------------------------------------------------------------------ its work

# float operations per weight that the quantizers' definitions ask for with an importance matrix: each
# trial scale rounds every weight and forms its sums (and, where a min is fitted, the error of the fit);
# a lattice trial also measures the listed neighbours of the groups that fall off the grid
TRIAL = {"Q2_K": 37 * 15, "Q4_K": 37 * 15, "Q5_K": 37 * 15, "Q4_1": 37 * 15, "Q5_1": 37 * 15, "Q3_K": 19 * 8,
         "Q6_K": 19 * 8, "Q4_0": 19 * 8, "Q5_0": 19 * 8, "IQ4_XS": 16 * 13, "IQ4_NL": 16 * 13, "IQ2_XXS": 14 * 100,
         "IQ2_XS": 20 * 100, "IQ2_S": 20 * 40, "IQ3_XXS": 32 * 50, "IQ3_S": 20 * 70, "IQ1_S": 1000, "IQ1_M": 1000}


def work(case):
    op, n = case["op"], case["rows"] * case["cols"]
    if op == "r2_decode":
        n = 2 * (case["rows"] + case["kv"]) * case["cols"]
        return {"bytes": 3.3 * n, "flops": 0}            # coded to about 0.65 of 2 bytes, 2 bytes written
    _, qk, bs = QFUN[BY_NAME[case["quant"]]]
    blocks = n // qk * bs
    if op == "dequant":
        return {"bytes": blocks + 4 * n, "flops": 2 * n}
    if op == "regrow":
        imx = 4 * case["cols"] if case["imatrix"] else 0
        return {"bytes": SRC[case["src"]][1] * n + blocks + imx, "flops": TRIAL.get(case["quant"], 4) * n}
    # the prediction and the file, and of the base and the model only what the changed blocks need
    return {"bytes": 2 * blocks + 2 * n * case["changed"], "flops": 0}


def tolerance(case):
    return "exact"        # bytes, and for dequant the one rounding of each product: identical on both sides


# ------------------------------------------------------------------------------------------ in 64 bits

def exact(case, seed):
    """dequant's values from the blocks' definitions, in float64; the other paths give bytes"""
    if case["op"] != "dequant":
        return None
    quant, n = case["quant"], case["rows"] * case["cols"]
    b = _blocks(_generator(seed), quant, n // QFUN[BY_NAME[quant]][1])
    f16 = lambda o: b[:, o:o + 2].contiguous().view(torch.float16).double()            # (blocks, 1)
    if quant == "Q8_0":
        x = f16(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif quant == "Q4_0":
        q = b[:, 2:].int()
        x = f16(0) * (torch.cat([q & 15, q >> 4], 1) - 8).double()
    elif quant == "Q4_K":
        s, q = b[:, 4:16].int(), b[:, 16:].int().view(-1, 4, 32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        x = (f16(0) * sc.double())[:, :, None] * q - (f16(2) * mn.double())[:, :, None]
    else:
        lo, hi = b[:, :128].int().view(-1, 2, 2, 32), b[:, 128:192].int().view(-1, 2, 1, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        lo = torch.cat([lo & 15, lo >> 4], 2)                                           # (blocks, half, quarter, 32)
        hi = torch.cat([hi & 3, hi >> 2 & 3, hi >> 4 & 3, hi >> 6], 2)
        q = ((lo | hi << 4) - 32).double().view(-1, 16, 16)
        x = (f16(208) * sc)[:, :, None] * q
    return x.reshape(-1)
