"""Checkpoints that the generator does not write, made from one that it does: other
shapes, other metadata, tensors scaled."""
import json
import struct

import numpy as np


def read(path):
    """(metadata, {name: array}) of a safetensors file of F32 and I64 tensors."""
    b = open(path, "rb").read()
    (n,) = struct.unpack("<Q", b[:8])
    head = json.loads(b[8:8 + n])
    meta = head.pop("__metadata__")
    kind = {"F32": "<f4", "I64": "<i8"}
    return meta, {k: np.frombuffer(b, kind[v["dtype"]], int(np.prod(v["shape"])), 8 + n + v["data_offsets"][0])
                  .reshape(v["shape"]).copy() for k, v in head.items()}


def write(path, meta, tensors):
    head, data, at = {"__metadata__": meta}, [], 0
    for k, a in tensors.items():
        kind = {"f": "F32", "i": "I64"}[a.dtype.kind]
        a = np.ascontiguousarray(a)
        head[k] = {"dtype": kind, "shape": list(a.shape), "data_offsets": [at, at + a.nbytes]}
        data.append(a.tobytes())
        at += a.nbytes
    hj = json.dumps(head, separators=(",", ":")).encode()
    hj += b" " * (-(8 + len(hj)) % 8)
    with open(path, "wb") as f:
        f.write(struct.pack("<Q", len(hj)) + hj + b"".join(data))
    return str(path)


def edited(src, dst, edit):
    """dst: the checkpoint src after edit(metadata, tensors)."""
    meta, t = read(src)
    edit(meta, t)
    return write(dst, meta, t)


def compress_ratio(ratio, seed=0):
    """An edit that gives every CAB the width embed / ratio."""
    def edit(meta, t):
        meta["compress_ratio"] = str(ratio)
        c = int(meta["embed_dim"])
        w = c // ratio
        rng = np.random.default_rng(seed)

        def n(*s):
            return rng.standard_normal(s, dtype=np.float32) * np.float32(0.02)
        for k in [k for k in t if k.endswith(".conv_block.cab.0.weight")]:
            p = k[:-len("0.weight")]
            t[p + "0.weight"], t[p + "0.bias"], t[p + "2.weight"] = n(w, c, 3, 3), n(w), n(c, w, 3, 3)
    return edit
