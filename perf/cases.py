"""What the speed of this library is measured on: the calls a program that runs a quantised sparse-MoE model makes, through the
package's public entry points.

A case is a dict of plain values.  Families (`"kind"`):

  linear  QMatMul: one resident quantised matrix, the attention and output projections around the MoE block.
  moe     SparseMoeBlock on activations that are resident in HBM.
  stack   stack_forward: the MoE blocks of consecutive layers, y = x + moe(rms_norm(x)) each, as one call.
  host    SparseMoeBlock on host arrays, what candle's CustomOp1::cpu_fwd hands over (its Device has no HIP variant).

Weights are N(0, 0.02) quantised on the GPU with the library's QTensor::quantize, activations N(0, 1), the router f32
N(0, 0.02); everything follows from the seed.
"""
import math

import numpy as np
import torch

import candle_amd

DTYPES = {"q4_0": (candle_amd.GGML_Q4_0, 32, 18), "q8_0": (candle_amd.GGML_Q8_0, 32, 34), "q4_k": (candle_amd.GGML_Q4K, 256, 144),
          "q5_k": (candle_amd.GGML_Q5K, 256, 176), "q6_k": (candle_amd.GGML_Q6K, 256, 210)}

# layer shapes of the benchmark and of the tests
SHAPES = {
    "mixtral": dict(hidden=4096, ffn=14336, experts=8, top_k=2, shared=0),    # Mixtral-8x7B
    "small": dict(hidden=1024, ffn=3584, experts=8, top_k=2, shared=0),       # a quarter of its width
    "fine": dict(hidden=2048, ffn=1408, experts=60, top_k=4, shared=5632),    # Qwen-MoE: many small experts, one always on
}
# router logit biases under which top-2 of eight gives expert loads that follow Zipf(1): what a prompt of one topic does
ZIPF_BIAS = (0.0, -1.158, -1.581, -1.845, -2.033, -2.186, -2.299, -2.398)

RMS_EPS = 1e-5

# projections of the Mixtral shape: q / o, the grouped k / v, the output head
LINEARS = ((4096, 4096), (1024, 4096), (32000, 4096))


def _linear(dtype, n, k, tokens):
    return {"kind": "linear", "dtype": dtype, "n": n, "k": k, "tokens": tokens}


def _moe(kind, shape, dtype, tokens, down=None, skewed=False, layers=1):
    return {"kind": kind, "shape": shape, "dtype": dtype, "down": down or dtype, "tokens": tokens, "skewed": skewed, "layers": layers}


def listed():
    cases = [
        # one sequence being decoded: an attention projection, the smallest call there is
        ("linear_decode_1", _linear("q4_k", 4096, 4096, 1)),
        # the output head of a decode batch, Q6_K as Q4_K_M files store it
        ("head_decode_32", _linear("q6_k", 32000, 4096, 32)),
        # the same attention projection for a prompt of a length that fits no tile
        ("linear_prefill_777", _linear("q4_k", 4096, 4096, 777)),
        # a small Q4_0 layer, a handful of tokens: launches and latency
        ("small_decode_16", _moe("moe", "small", "q4_0", 16)),
        # Mixtral, decode: one sequence, a served batch, a large served batch
        ("decode_1", _moe("moe", "mixtral", "q4_k", 1)),
        ("decode_32", _moe("moe", "mixtral", "q4_k", 32)),
        ("decode_64", _moe("moe", "mixtral", "q4_k", 64)),
        # a chunk of a prompt together with decoding sequences, in the mixed types of a Q4_K_M file
        ("chunk_301", _moe("moe", "mixtral", "q4_k", 301, down="q6_k")),
        # a long prompt whose tokens crowd on a few experts
        ("prefill_4096", _moe("moe", "mixtral", "q4_k", 4096, skewed=True)),
        # many small Q8_0 experts with an always-on one, a short prompt
        ("fine_prefill_512", _moe("moe", "fine", "q8_0", 512)),
        # consecutive layers of one decode step: every layer's weights come from HBM
        ("stack_decode_32", _moe("stack", "mixtral", "q4_k", 32, layers=4)),
        # the drop-in op: a batch that arrives from and returns to host memory
        ("host_100", _moe("host", "mixtral", "q4_k", 100)),
    ]
    return [dict(c, name=name) for name, c in cases]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "moe", "moe", "moe", "moe", "small", "fine", "fine", "stack", "host"))
    if kind == "linear":
        n, k = rng.choice(LINEARS)
        # the head sees one row per sequence, the attention projections every token of a prompt
        return _linear(rng.choice(("q4_k", "q5_k", "q6_k", "q8_0")), n, k, _log_int(rng, 1, 128 if n == 32000 else 4096))
    if kind == "moe":
        dtype, down = rng.choice((("q4_k", "q4_k"), ("q4_k", "q6_k"), ("q5_k", "q5_k"), ("q5_k", "q6_k"), ("q6_k", "q6_k")))
        return _moe("moe", "mixtral", dtype, _log_int(rng, 1, 3000), down=down, skewed=rng.random() < 0.3)
    if kind == "small":
        return _moe("moe", "small", rng.choice(("q4_0", "q4_k")), _log_int(rng, 1, 1000))
    if kind == "fine":
        return _moe("moe", "fine", "q8_0", _log_int(rng, 1, 2000))
    if kind == "stack":
        return _moe("stack", "mixtral", "q4_k", _log_int(rng, 1, 64), layers=rng.randint(2, 4))
    return _moe("host", "mixtral", "q4_k", _log_int(rng, 1, 600))


def _blocks(gen, dtype, rows, cols):
    """The bytes of a quantised [rows, cols] matrix, on the host, as a file loader holds them."""
    x = torch.randn((rows, cols), generator=gen, device="cuda") * 0.02
    return candle_amd.quantize_weights(DTYPES[dtype][0], x).cpu().numpy()


def _vector(gen, shape, std=0.02, mean=0.0):
    return (mean + std * torch.randn(shape, generator=gen, device="cuda")).cpu().numpy()


def _weights(gen, case):
    """One layer's weights on the host: matrices as quantised bytes, vectors as f32."""
    s = SHAPES[case["shape"]]
    H, F, E, Fs = s["hidden"], s["ffn"], s["experts"], s["shared"]
    dt, down = case["dtype"], case["down"]
    w = {}
    if Fs:
        w.update(shared_w1=_blocks(gen, dt, Fs, H), shared_w3=_blocks(gen, dt, Fs, H), shared_w2=_blocks(gen, down, H, Fs),
                 shared_gate=_vector(gen, (H,)))
    if case["skewed"]:
        w.update(gate_bias=np.array(ZIPF_BIAS, dtype=np.float32))
    if case["kind"] == "stack":
        w.update(rms_alpha=_vector(gen, (H,), 0.1, 1.0))
    w.update(w1=[_blocks(gen, dt, F, H) for _ in range(E)])
    w.update(w3=[_blocks(gen, dt, F, H) for _ in range(E)])
    w.update(w2=[_blocks(gen, down, H, F) for _ in range(E)])
    w.update(gate=_vector(gen, (E, H)))
    return w


def _layer(gen, case):
    s = SHAPES[case["shape"]]
    w = _weights(gen, case)
    kw = {}
    if s["shared"]:
        kw.update(shared_ffn=s["shared"], shared_w1=w["shared_w1"], shared_w3=w["shared_w3"], shared_w2=w["shared_w2"],
                  shared_gate=w["shared_gate"])
    if case["skewed"]:
        kw.update(gate_bias=w["gate_bias"])
    if case["kind"] == "stack":
        kw.update(rms_alpha=w["rms_alpha"], rms_eps=RMS_EPS)
    return candle_amd.SparseMoeBlock(s["hidden"], s["ffn"], s["experts"], s["top_k"], DTYPES[case["dtype"]][0], w["gate"], w["w1"], w["w3"],
                                     w["w2"], ggml_dtype_down=DTYPES[case["down"]][0], **kw)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    T = case["tokens"]
    if case["kind"] == "linear":
        n, k = case["n"], case["k"]
        lin = candle_amd.QMatMul(DTYPES[case["dtype"]][0], _blocks(gen, case["dtype"], n, k), n, k)
        return {"kind": "linear", "lin": lin, "x": torch.randn((T, k), generator=gen, device="cuda")}
    layers = [_layer(gen, case) for _ in range(case["layers"])]
    x = torch.randn((T, SHAPES[case["shape"]]["hidden"]), generator=gen, device="cuda")
    return {"kind": case["kind"], "layers": layers, "x": x.cpu().numpy() if case["kind"] == "host" else x}


def run(state):
    if state["kind"] == "linear":
        return state["lin"].forward(state["x"])
    if state["kind"] == "stack":
        return candle_amd.stack_forward(state["layers"], state["x"])
    return state["layers"][0].forward(state["x"])


def work(case):
    T = case["tokens"]
    if case["kind"] == "linear":
        _, be, bb = DTYPES[case["dtype"]]
        n, k = case["n"], case["k"]
        return {"bytes": n * k // be * bb + 4 * T * (n + k), "flops": 2 * T * n * k}
    s = SHAPES[case["shape"]]
    H, F, E, top_k, Fs = s["hidden"], s["ffn"], s["experts"], s["top_k"], s["shared"]
    per_weight = lambda name: DTYPES[name][2] / DTYPES[name][1]
    matrix_bytes = H * (2 * per_weight(case["dtype"]) + per_weight(case["down"]))   # of w1, w3 and w2, per unit of the ffn size
    active = E * (1.0 - (1.0 - top_k / E) ** T)   # experts that uniform routing reaches
    weights = matrix_bytes * (active * F + Fs)
    router = 4 * H * (E + (1 if Fs else 0))
    ops = 2 * T * 3 * H * (top_k * F + Fs) + 2 * T * H * E
    return {"bytes": case["layers"] * int(weights + router) + 2 * 4 * T * H, "flops": case["layers"] * ops}


def tolerance(case):
    # Integer dot products are exact; what is left are the f32 sums over blocks.  Against the same product in 64 bits a
    # projection shows 1.7e-7 (2-norm) and 6.4e-7 (largest difference over the rms).
    if case["kind"] == "linear":
        return {"rel": 1e-6, "max": 3e-6}
    # Inside a layer the intermediate is quantised to 8 bits again, where a last-bit difference moves a value by one step
    # now and then.  Against a model with 64-bit sums, and between the kernels that sum in different orders: 1.1e-4 and
    # 3.4e-3 over batches; a single token, where one step weighs more, 3.1e-4.  Steps weigh sqrt(14336 / ffn) times as much
    # in narrower layers.
    if case["kind"] != "stack":
        widen = math.sqrt(14336.0 / SHAPES[case["shape"]]["ffn"])
        return {"rel": widen * (1.2e-3 if case["tokens"] < 32 else 4.5e-4), "max": widen * 1.4e-2}
    # The next layer quantises that difference again: four layers summed in another order differ by 5.8e-3 and 3.1e-2.
    return {"rel": 2.4e-2, "max": 1.3e-1}


# What `run` returns, in 64 bits: the blocks decoded, activations quantised to 8 bits as the quantised products of GGML do
# (that is part of the result, not an approximation of it), everything else in double precision.
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _k_scales(b):
    """The eight 6-bit scales and minimums of Q4_K and Q5_K blocks, from their twelve bytes."""
    b = b.int()
    lo, mid, hi = b[:, 0:4], b[:, 4:8], b[:, 8:12]
    return torch.cat((lo & 63, (hi & 15) | (lo >> 6 << 4)), 1).double(), torch.cat((mid & 63, (hi >> 4) | (mid >> 6 << 4)), 1).double()


def _decode(dtype, raw, rows, cols):
    _, _, size = DTYPES[dtype]
    b = torch.from_numpy(np.ascontiguousarray(raw).view(np.uint8).reshape(-1, size)).cuda()
    if dtype == "q8_0":
        x = _f16(b[:, :2]) * b[:, 2:].view(torch.int8).double()
    elif dtype == "q4_0":
        q = b[:, 2:]
        x = _f16(b[:, :2]) * (torch.cat((q & 15, q >> 4), 1).double() - 8)
    elif dtype == "q6_k":
        lo, hi, sc = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32), b[:, 192:208].view(torch.int8).double()
        q = torch.cat((lo & 15, lo >> 4), 2) | (torch.cat([hi >> s & 3 for s in (0, 2, 4, 6)], 2) << 4)
        x = ((q.reshape(-1, 16, 16).double() - 32) * sc[:, :, None]).reshape(-1, 256) * _f16(b[:, 208:210])
    else:
        sc, mn = _k_scales(b[:, 4:16])
        q = b[:, size - 128:].reshape(-1, 4, 1, 32)
        q = torch.cat((q & 15, q >> 4), 2).reshape(-1, 8, 32)
        if dtype == "q5_k":
            q = q | (torch.stack([b[:, 16:48] >> s & 1 for s in range(8)], 1) << 4)
        x = (_f16(b[:, :2]) * sc)[:, :, None] * q.double() - (_f16(b[:, 2:4]) * mn)[:, :, None]
    return x.reshape(rows, cols)


def _quantised(dtype, x):
    """The rows as the quantised product sees them: blocks of 256 (Q8_K) beside K-quants, of 32 (Q8_0) beside the others."""
    n = DTYPES[dtype][1]
    v = x.float().reshape(-1, n)
    amax, at = v.abs().max(1, keepdim=True)
    if n == 256:
        inv = -128.0 / v.gather(1, at)
        d = 1.0 / inv
    else:
        d = amax / 127.0
        inv = 1.0 / d
        d = d.half()
    t = (v * inv).double()
    q = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return torch.where(amax > 0, q.clamp(-128, 127) * d.double(), 0.0).reshape(x.shape)


def _expert(case, x, ffn, w1, w3, w2):
    H = x.shape[1]
    xq = _quantised(case["dtype"], x)
    a, b = xq @ _decode(case["dtype"], w1, ffn, H).T, xq @ _decode(case["dtype"], w3, ffn, H).T
    h = a * torch.sigmoid(a) * b
    # One layer: the intermediate stays in 64 bits.  Rounded to 8 bits as the layer does, its last bits decide which step a
    # value takes, and an equally good sum in another order is 1e-7 off by luck or 1e-4.  In a stack the steps of the layers
    # before are part of what a layer reads.
    return (_quantised(case["down"], h) if case["kind"] == "stack" else h) @ _decode(case["down"], w2, H, ffn).T


def _block64(case, w, x):
    s = SHAPES[case["shape"]]
    vec = lambda name: torch.from_numpy(w[name]).cuda().double()
    xs = x
    if "rms_alpha" in w:
        xs = (x / (x.square().mean(1, keepdim=True) + RMS_EPS).sqrt() * vec("rms_alpha")).float().double()   # an f32 row in the model
    probs = torch.softmax(xs @ vec("gate").T + (vec("gate_bias") if "gate_bias" in w else 0.0), 1)
    top, idx = probs.topk(s["top_k"], 1)
    top = top / top.sum(1, keepdim=True)
    y = x.clone() if "rms_alpha" in w else torch.zeros_like(x)
    for e in range(s["experts"]):
        t, r = (idx == e).nonzero(as_tuple=True)
        if len(t):
            y.index_add_(0, t, top[t, r, None] * _expert(case, xs[t], s["ffn"], w["w1"][e], w["w3"][e], w["w2"][e]))
    if s["shared"]:
        y += torch.sigmoid(xs @ vec("shared_gate"))[:, None] * _expert(case, xs, s["shared"], w["shared_w1"], w["shared_w3"], w["shared_w2"])
    return y


def exact(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    T = case["tokens"]
    if case["kind"] == "linear":
        n, k = case["n"], case["k"]
        w = _decode(case["dtype"], _blocks(gen, case["dtype"], n, k), n, k)
        return _quantised(case["dtype"], torch.randn((T, k), generator=gen, device="cuda")) @ w.T
    layers = [_weights(gen, case) for _ in range(case["layers"])]
    x = torch.randn((T, SHAPES[case["shape"]]["hidden"]), generator=gen, device="cuda").double()
    for w in layers:
        x = _block64(case, w, x)
    return x.cpu().numpy() if case["kind"] == "host" else x
