"""Measured workloads of causal_conv1d_fn, each one pass through the package's public entry point.

A case is a dict of plain values:
  name     its name (listed cases only)
  kind     "infer" (autograd off) or "train" (forward, then the gradients of every differentiable
           input for a given upstream gradient)
  B, T, D, W   batch, seqlen, dim (channels), filter width
  dtype    of x, out, the upstream gradient and the states; weight and bias are fp32
  bias, silu   bias on / silu activation on
  states   "infer": initial_states given and final_states returned, as a streaming program hands
           them from call to call; "train": initial_states given, their gradient returned
  packed   seq_idx of packed sequences: segments of 64 to 4096 rows, the last 5 % of a row padding
  pitch    channels of the tensor x is a channel slice of, from channel c0 (0: x is contiguous)
  graph    the pass is captured in a graph once and replayed, as a program does whose step is
           shorter than the host's work for it
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "causal-conv1d-triton_amd"))

from causal_conv1d_triton import causal_conv1d_fn  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ESIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


def _case(name, kind, B, T, D, W=4, dtype="bf16", bias=True, silu=True, states=False, packed=False,
          pitch=0, c0=0, graph=False):
    c = dict(kind=kind, B=B, T=T, D=D, W=W, dtype=dtype, bias=bias, silu=silu, states=states,
             packed=packed, pitch=pitch, c0=c0, graph=graph)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One generated token of a serving batch, the states carried from step to step.
        _case("decode", "infer", 16, 1, 2048, states=True),
        # Chunked prefill of the same server: 256 tokens per call.
        _case("chunk", "infer", 16, 256, 2048, states=True),
        # Long-context prefill without states.
        _case("prefill", "infer", 4, 32768, 1024),
        # A short training step called as it stands, where host work and launches count.
        _case("train_short", "train", 4, 512, 1024),
        # A middle-sized captured step in fp16, filter only (no bias, no activation), ragged length.
        _case("train_mid_fp16", "train", 4, 2047, 1024, dtype="fp16", bias=False, silu=False,
              graph=True),
        # The benchmark shape, captured as bench.py captures it.
        _case("train_bench", "train", 4, 8192, 1024, graph=True),
        # Mamba-2 2.7B's convolution: x is the xBC slice of the in_proj output (z, xBC, dt).
        _case("train_inproj", "train", 8, 4096, 5376, pitch=10576, c0=5120),
        # Packed variable-length training with a wider filter and learned initial states.
        _case("train_packed_w7", "train", 4, 16384, 4096, W=7, states=True, packed=True),
        # Channel counts and lengths that no access width divides.
        _case("train_odd", "train", 4, 5001, 1501),
        # Full-precision training.
        _case("train_fp32", "train", 4, 4096, 2048, dtype="fp32"),
        # Filters wider than the usual four taps.
        _case("train_w16", "train", 4, 8192, 1024, W=16, graph=True),
        # A long filter, past the widths compiled one by one.
        _case("train_w64", "train", 2, 4096, 1024, W=64, graph=True),
    ]


# Elements of x that no drawn case exceeds, by width: the listed cases of the widths.
def _most_elements(W):
    return 8 << 20 if W > 32 else 32 << 20 if W > 8 else 128 << 20


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["infer", "train", "train"])
    W = rng.choice([4, 4, 4, 4, rng.randint(2, 8), rng.randint(2, 8), rng.randint(9, 32), log(33, 128)])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    # Channels: usually a multiple of 64, else any number.
    D = 64 * log(4, 84) if rng.random() < 0.65 else log(64, 5376)
    # Lengths: decode steps, or from short chunks to long contexts, any number of rows.
    T = 1 if kind == "infer" and rng.random() < 0.2 else log(16, 32768)
    most = _most_elements(W) // (2 if dtype == "fp32" else 1)
    T = max(1, min(T, most // D))
    B = max(1, min(log(1, 32), most // (T * D)))
    packed = kind == "train" and T >= 512 and rng.random() < 0.2
    pitch, c0 = 0, 0
    if rng.random() < 0.2:  # a slice of a projection's output
        extra = log(1, 330)
        pitch, c0 = D + 16 * extra, 16 * rng.randint(0, extra)
    return _case(None, kind, B, T, D, W, dtype, bias=rng.random() < 0.8, silu=rng.random() < 0.8,
                 states=rng.random() < 0.4, packed=packed, pitch=pitch, c0=c0,
                 graph=kind == "train" and rng.random() < 0.5)


def _packed_ids(rng, B, T):
    ids = np.empty((B, T), np.int32)
    for b in range(B):
        t = n = 0
        while t < T:
            length = int(rng.integers(64, 4097))
            ids[b, t:t + length] = n
            t += length
            n += 1
        ids[b, T - T // 20:] = -1
    return ids


def _inputs(case, seed):
    """x ~ N(0, 1), weight ~ N(0, 1 / W), bias ~ N(0, 1), states and upstream gradient ~ N(0, 1)."""
    B, T, D, W = case["B"], case["T"], case["D"], case["W"]
    dt = DTYPES[case["dtype"]]
    g = torch.Generator(DEV).manual_seed(seed)
    train = case["kind"] == "train"

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)

    if case["pitch"]:
        wide = normal(B, T, case["pitch"], dtype=dt)
        x = wide[..., case["c0"]:case["c0"] + D]
    else:
        x = normal(B, T, D, dtype=dt)
    s = {"x": x.detach(), "w": normal(D, W) / math.sqrt(W), "b": normal(D) if case["bias"] else None,
         "init": normal(B, W - 1, D, dtype=dt) if case["states"] else None,
         "dy": normal(B, T, D, dtype=dt) if train else None, "seq": None}
    if case["packed"]:
        s["seq"] = torch.from_numpy(_packed_ids(np.random.default_rng(seed), B, T)).to(DEV)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["act"] = "silu" if case["silu"] else None
    s["train"], s["graph"] = case["kind"] == "train", None
    s["wrt"] = []
    if s["train"]:
        s["wrt"] = [s[k].requires_grad_(True) for k in ("x", "w", "b", "init") if s[k] is not None]
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(s)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            s["outs"] = _pass(s)
        s["graph"] = graph
    return s


def _pass(s):
    if not s["train"]:
        with torch.no_grad():
            return causal_conv1d_fn(s["x"], s["w"], s["b"], initial_states=s["init"],
                                    return_final_states=s["init"] is not None, activation=s["act"])
    out = causal_conv1d_fn(s["x"], s["w"], s["b"], seq_idx=s["seq"], initial_states=s["init"],
                           activation=s["act"])
    return (out.detach(),) + torch.autograd.grad(out, s["wrt"], s["dy"])


def run(s):
    if s["graph"] is None:
        return _pass(s)
    s["graph"].replay()
    return s["outs"]


def work(case):
    """Every input read once, every output written once; two operations per tap and element in the
    forward, and in the backward for the gradient of x and for that of the weight."""
    B, T, D, W = case["B"], case["T"], case["D"], case["W"]
    n, state, e = B * T * D, B * (W - 1) * D, ESIZE[case["dtype"]]
    params = D * (W + (1 if case["bias"] else 0)) * 4
    train = case["kind"] == "train"
    tensors = 4 if train else 2  # x and out; with the upstream gradient and the gradient of x
    byts = tensors * n * e + params * (2 if train else 1)
    if case["states"]:
        byts += 2 * state * e
    if case["packed"]:
        byts += 4 * B * T
    return {"bytes": byts, "flops": 2 * W * n * (3 if train else 1)}


def tolerance(case):
    """About four times the largest relative error against exact() that the path shows: the rounding
    of out and of the gradient of x to their dtype (bf16 1.7e-3, fp16 2.1e-4), in fp32 the sums (up to 2.4e-7, more for other orders of them)."""
    return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 2e-6}[case["dtype"]]}


def exact(case, seed):
    """The pass in 64 bits: a sum of shifted products, masked where the sequence ids differ, and the
    same sums for the gradients."""
    s = _inputs(case, seed)
    B, T, D, W = case["B"], case["T"], case["D"], case["W"]
    P, train = W - 1, case["kind"] == "train"
    w = s["w"].double()
    outs, dxs, dinits, finals = [], [], [], []
    dw = torch.zeros(D, W, dtype=torch.float64, device=DEV)
    db = torch.zeros(D, dtype=torch.float64, device=DEV)
    for i in range(B):  # one batch row at a time: 64-bit copies of all of them need not fit
        x = s["x"][i].detach().double()
        head = s["init"][i].detach().double() if s["init"] is not None else x.new_zeros(P, D)
        xx = torch.cat([head, x])
        ids = None
        if s["seq"] is not None:
            seq = s["seq"][i]
            first = seq[:1] if s["init"] is not None else torch.full_like(seq[:1], -1)
            ids = torch.cat([first.expand(P), seq])
        masks = [None if ids is None else (ids[k:k + T] == seq).double()[:, None] for k in range(W)]

        z = x.new_zeros(T, D)
        for k in range(W):
            z += w[:, k] * xx[k:k + T] if ids is None else w[:, k] * xx[k:k + T] * masks[k]
        if s["b"] is not None:
            z += s["b"].double()
        pad = None if ids is None else (seq < 0)[:, None]
        if pad is not None:
            z.masked_fill_(pad, 0.0)
        sig = torch.sigmoid(z) if case["silu"] else None
        outs.append(z * sig if case["silu"] else z)
        if s["init"] is not None:
            finals.append(xx[T:])
        if not train:
            continue
        g = s["dy"][i].double()
        if case["silu"]:
            g = g * sig * (1 + z * (1 - sig))
        if pad is not None:
            g = g.masked_fill(pad, 0.0)
        dxx = x.new_zeros(T + P, D)
        for k in range(W):
            gm = g if ids is None else g * masks[k]
            dxx[k:k + T] += w[:, k] * gm
            dw[:, k] += (gm * xx[k:k + T]).sum(0)
        db += g.sum(0)
        dxs.append(dxx[P:])
        dinits.append(dxx[:P])
    out = torch.stack(outs)
    if not train:
        return (out, torch.stack(finals)) if s["init"] is not None else out
    grads = [torch.stack(dxs), dw]
    if s["b"] is not None:
        grads.append(db)
    if s["init"] is not None:
        grads.append(torch.stack(dinits))
    return (out, *grads)
