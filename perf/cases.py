"""Performance cases of the scan library: what a program that uses it calls.

listed() gives the fixed cases, draw(rng) another one of the same ranges.
prepare(case, seed) makes what the program has before the call (device
buffers, a handle, a captured graph, host arrays for the cost model),
run(state) is one pass through the public entry points, work(case) the bytes
and operations that pass cannot do without, and exact(case, seed) its result
from plain torch or numpy in 64 bits.

uint32 data lives in int32 tensors (the library scans the bits, mod 2^32).
"""
import math

import numpy as np
import torch

import gpuprefixsums_amd as gps
import gpuprefixsums_amd.torch_ops  # noqa: F401  (registers torch.ops.gps.*)
from gpuprefixsums_amd.tuner.model import GpuMlp

DEVICE = "cuda"

# The values a pass scans: byte counts, small integers, or every uint32 (the
# sums wrap); normal floats, or BF16 spread over eight decades with random sign.
BYTE, SMALL, FULL = 8, 10, 32
NORMAL, DECADES = "normal", "decades"


def listed():
    return [
        # A few hundred bins or per-block counts in a latency-bound loop.
        dict(name="scan_1k", kind="scan", algo="csdl", n=1021, inclusive=True, bits=BYTE, shift=0, stall=0),
        # Stream-compaction offsets of a million flags or counts.
        dict(name="scan_1m_exclusive", kind="scan", algo="csdl", n=1 << 20, inclusive=False, bits=BYTE, shift=0,
             stall=0),
        # A slice x[1:] of a larger array, of no round length.
        dict(name="scan_12m_slice", kind="scan", algo="csdl", n=12_345_677, inclusive=True, bits=FULL, shift=1,
             stall=0),
        # The benchmark's headline: 1 GiB in, 1 GiB out.
        dict(name="scan_256m", kind="scan", algo="csdl", n=1 << 28, inclusive=True, bits=FULL, shift=0, stall=0),
        # The same under emulated deadlock: every 7th tile withholds its word.
        dict(name="fallback_256m_stall7", kind="scan", algo="csdldf", n=1 << 28, inclusive=True, bits=FULL, shift=0,
             stall=7),
        # The reference's second algorithm, on a length past a power of two.
        dict(name="rts_67m", kind="scan", algo="rts", n=(1 << 26) + 5, inclusive=True, bits=FULL, shift=0, stall=0),
        # Four counters per element (uint4 structs), each scanned on its own.
        dict(name="struct_1m_exclusive", kind="struct", n=1_000_003, inclusive=False, bits=FULL),
        # Compensated floating-point scans: a large one through a handle and
        # an ordinary one through the PyTorch operator.
        dict(name="f32_128m", kind="fp", api="handle", n=1 << 27, dtype="f32", values=NORMAL),
        dict(name="bf16_3m_op", kind="fp", api="op", n=3_000_017, dtype="bf16", values=DECADES),
        # The benchmark's ragged batch, replayed from a captured graph.
        dict(name="segmented_51m_graph", kind="segmented", api="graph", n=50_934_930, segments=4096, dtype="u32",
             inclusive=False),
        # Many short sequences (about 128 elements each) through the operator.
        dict(name="segmented_f32_2m_op", kind="segmented", api="op", n=2_097_169, segments=16384, dtype="f32",
             inclusive=True),
        # Epochs of the tuner's cost model on its own training-set size.
        dict(name="cost_model_epochs", kind="train", batch=18_808, features=18, hidden=64, epochs=20),
    ]


def draw(rng):
    kind = rng.choices(["scan", "struct", "fp", "segmented", "train"], [6, 2, 3, 4, 1])[0]
    if kind == "scan":
        algo = rng.choices(["csdl", "rts", "csdldf"], [4, 1, 1])[0]
        return dict(kind="scan", algo=algo, n=_log_uniform(rng, 10, 27.9), inclusive=rng.random() < 0.5,
                    bits=rng.choice([BYTE, FULL]), shift=rng.choice([0, 0, 0, 1, 2, 3]),
                    stall=rng.choice([0, 7, 8]) if algo == "csdldf" else 0)
    if kind == "struct":
        return dict(kind="struct", n=_log_uniform(rng, 10, 25.9), inclusive=rng.random() < 0.5, bits=FULL)
    if kind == "fp":
        dtype = rng.choice(["f32", "bf16"])
        return dict(kind="fp", api=rng.choice(["handle", "op"]), n=_log_uniform(rng, 10, 27), dtype=dtype,
                    values=NORMAL if dtype == "f32" else DECADES)
    if kind == "segmented":
        dtype = rng.choice(["u32", "u32", "f32", "bf16"])
        return dict(kind="segmented", api=rng.choice(["handle", "op", "graph"] if dtype == "u32" else ["handle", "op"]),
                    n=_log_uniform(rng, 12, 26), segments=_log_uniform(rng, 0, 14), dtype=dtype,
                    inclusive=dtype != "u32" or rng.random() < 0.5)
    return dict(kind="train", batch=_log_uniform(rng, 9, 14.2), features=rng.randint(6, 32),
                hidden=rng.choice([32, 48, 64, 64, 96]), epochs=rng.randint(4, 12))


def _log_uniform(rng, lo, hi):
    return int(round(2.0 ** rng.uniform(lo, hi)))


# ---- inputs -----------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _integers(n, bits, seed):
    lo, hi = (-(1 << 31), 1 << 31) if bits == FULL else (0, 1 << bits)
    return torch.randint(lo, hi, (n,), dtype=torch.int32, device=DEVICE, generator=_generator(seed))


def _floats(n, dtype, values, seed):
    g = _generator(seed)
    if values == NORMAL:
        x = torch.randn(n, device=DEVICE, generator=g)
    else:
        x = torch.pow(10.0, torch.rand(n, device=DEVICE, generator=g) * 8.0 - 4.0)
        x *= torch.randint(0, 2, (n,), device=DEVICE, generator=g) * 2 - 1
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _offsets(n, segments, seed):
    """Log-normal segment lengths (sigma 1.5), scaled to end at n."""
    rng = np.random.default_rng(seed)
    ends = np.cumsum(np.exp(1.5 * rng.standard_normal(segments)))
    off = np.concatenate([[0], np.rint(ends * (n / ends[-1]))]).astype(np.int64)
    off[-1] = n
    return torch.from_numpy(off).to(DEVICE)


def _scan_input(case, seed):
    """The scanned tensor: a slice `shift` elements into its buffer."""
    return _integers(case["n"] + case["shift"], case["bits"], seed)[case["shift"]:]


def _segmented_input(case, seed):
    if case["dtype"] == "u32":
        x = _integers(case["n"], SMALL, seed)
    else:
        x = _floats(case["n"], case["dtype"], NORMAL, seed)
    return x, _offsets(case["n"], case["segments"], seed)


def _training_set(case, seed):
    """Standardised features, targets with the features' scale, He-uniform
    weights and zero biases: what the cost model's fit starts from."""
    rng = np.random.default_rng(seed)
    B, D, H = case["batch"], case["features"], case["hidden"]
    x = rng.standard_normal((B, D)).astype(np.float32)
    t = (x[:, 0] + np.abs(x[:, 1]) - 0.5 * x[:, 2] * x[:, 3] + 0.1 * rng.standard_normal(B)).astype(np.float32)
    w = [rng.uniform(-1, 1, (H, D)) * math.sqrt(6.0 / D), np.zeros(H), rng.uniform(-1, 1, (H, H)) * math.sqrt(6.0 / H),
         np.zeros(H), rng.uniform(-1, 1, H) * math.sqrt(6.0 / H), np.zeros(1)]
    return x, t, np.concatenate([a.ravel() for a in w]).astype(np.float32)


LEARNING_RATE, WEIGHT_DECAY = 3e-3, 1e-5


# ---- one pass ---------------------------------------------------------------

ALGOS = {"csdl": gps.ALGO_CSDL, "rts": gps.ALGO_RTS, "csdldf": gps.ALGO_CSDLDF}


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case=case)
    if kind == "scan":
        state["x"] = _scan_input(case, seed)
        state["out"] = torch.empty(case["n"], dtype=torch.int32, device=DEVICE)
        state["handle"] = gps.ScanHandle(ALGOS[case["algo"]], case["n"], stall_period=case["stall"])
    elif kind == "struct":
        state["x"] = _integers(4 * case["n"], case["bits"], seed)
        state["out"] = torch.empty(4 * case["n"], dtype=torch.int32, device=DEVICE)
        state["handle"] = gps.ScanHandle(gps.ALGO_CSDL, case["n"])
    elif kind == "fp":
        state["x"] = _floats(case["n"], case["dtype"], case["values"], seed)
        if case["api"] == "handle":
            state["out"] = torch.empty(case["n"], dtype=torch.float32, device=DEVICE)
            state["handle"] = gps.ScanHandle(gps.ALGO_CSDL, case["n"])
    elif kind == "segmented":
        state["x"], state["offsets"] = _segmented_input(case, seed)
        if case["api"] != "op":
            out_type = torch.int32 if case["dtype"] == "u32" else torch.float32
            state["out"] = torch.empty(case["n"], dtype=out_type, device=DEVICE)
            state["handle"] = gps.ScanHandle(gps.ALGO_CSDL, case["n"])
        if case["api"] == "graph":
            state["graph"] = state["handle"].segmented_graph(state["x"], state["out"], state["offsets"],
                                                             case["segments"], case["n"], case["inclusive"])
    else:
        state["x"], state["t"], state["params"] = _training_set(case, seed)
        state["model"] = GpuMlp(case["features"], case["hidden"], case["batch"])
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "scan":
        state["handle"].scan(state["x"], state["out"], inclusive=case["inclusive"])
        return state["out"]
    if kind == "struct":
        state["handle"].scan_u32x4(state["x"], state["out"], case["n"], inclusive=case["inclusive"])
        return state["out"]
    if kind == "fp":
        if case["api"] == "op":
            return torch.ops.gps.cumsum(state["x"])
        if case["dtype"] == "bf16":
            state["handle"].inclusive_bf16_f32(state["x"], state["out"])
        else:
            state["handle"].inclusive_f32(state["x"], state["out"])
        return state["out"]
    if kind == "segmented":
        if case["api"] == "op":
            return torch.ops.gps.segmented_cumsum(state["x"], state["offsets"], case["inclusive"])
        if case["api"] == "graph":
            state["graph"].launch(torch.cuda.current_stream())
        elif case["dtype"] == "u32":
            state["handle"].segmented(state["x"], state["out"], state["offsets"], case["segments"], case["n"],
                                      case["inclusive"])
        else:
            state["handle"].segmented_fp(state["x"], state["out"], state["offsets"], case["segments"], case["n"],
                                         bf16=case["dtype"] == "bf16")
        return state["out"]
    model = state["model"]
    model.set_params(state["params"])
    curve = model.train(state["x"], state["t"], case["epochs"], LEARNING_RATE, WEIGHT_DECAY)
    return {"curve": curve, "params": model.get_params()}


# ---- what a pass cannot do without -------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "train":
        B, D, H, epochs = case["batch"], case["features"], case["hidden"], case["epochs"]
        count = H * D + H * H + 3 * H + 1
        # Per sample: forward, weight gradients, and the gradient into both
        # hidden layers (none into the input).
        flops = 2 * B * (2 * (D * H + H * H + H) + H * H + H)
        return {"bytes": 4 * (B * D + B + 2 * count + epochs), "flops": epochs * (flops + 10 * count)}
    n = case["n"]
    if kind == "struct":
        return {"bytes": 32 * n, "flops": 4 * n}
    element = 6 if case.get("dtype") == "bf16" else 8
    return {"bytes": element * n + (8 * (case["segments"] + 1) if kind == "segmented" else 0), "flops": n}


# ---- the same results in 64 bits ----------------------------------------------

def _wrapped(x, inclusive, dim=0):
    """Scan mod 2^32 of an int32 tensor's bits, as int32."""
    wide = x.to(torch.int64) & 0xFFFFFFFF
    s = torch.cumsum(wide, dim)
    return (s if inclusive else s - wide).to(torch.int32)


def _restarted(x, offsets, inclusive):
    """64-bit scan of x that restarts at every offset."""
    s = torch.cumsum(x, 0)
    before = torch.cat([s.new_zeros(1), s])[offsets[:-1]]
    s -= torch.repeat_interleave(before, offsets[1:] - offsets[:-1])
    return s if inclusive else s - x


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        return _wrapped(_scan_input(case, seed), case["inclusive"])
    if kind == "struct":
        x = _integers(4 * case["n"], case["bits"], seed)
        return _wrapped(x.view(-1, 4), case["inclusive"]).view(-1)
    if kind == "fp":
        return torch.cumsum(_floats(case["n"], case["dtype"], case["values"], seed).to(torch.float64), 0)
    if kind == "segmented":
        x, offsets = _segmented_input(case, seed)
        if case["dtype"] == "u32":
            return _restarted(x.to(torch.int64), offsets, case["inclusive"]).to(torch.int32)
        return _restarted(x.to(torch.float64), offsets, True)
    return _train_64(case, seed)


def _train_64(case, seed):
    """Full-batch AdamW on the three-layer perceptron, in numpy doubles."""
    x, t, p = (a.astype(np.float64) for a in _training_set(case, seed))
    B, D, H = case["batch"], case["features"], case["hidden"]
    cuts = np.cumsum([H * D, H, H * H, H, H])
    m, v = np.zeros_like(p), np.zeros_like(p)
    curve = np.zeros(case["epochs"])
    for step in range(1, case["epochs"] + 1):
        W1, b1, W2, b2, W3, b3 = np.split(p, cuts)
        W1, W2 = W1.reshape(H, D), W2.reshape(H, H)
        z1 = x @ W1.T + b1
        a1 = np.maximum(z1, 0.0)
        z2 = a1 @ W2.T + b2
        a2 = np.maximum(z2, 0.0)
        d = a2 @ W3 + b3 - t
        curve[step - 1] = np.mean(d * d)
        dy = 2.0 * d / B
        dz2 = np.outer(dy, W3) * (z2 > 0)
        dz1 = (dz2 @ W2) * (z1 > 0)
        g = np.concatenate([(dz1.T @ x).ravel(), dz1.sum(0), (dz2.T @ a1).ravel(), dz2.sum(0), a2.T @ dy, [dy.sum()]])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        update = (m / (1.0 - 0.9 ** step)) / (np.sqrt(v / (1.0 - 0.999 ** step)) + 1e-8)
        p = p - LEARNING_RATE * (update + WEIGHT_DECAY * p)
    return {"curve": curve, "params": p}
