"""The work that a program using this library has it do, as measurable cases.

A mixture-of-experts layer serves a model in four ways, and the cases cover
each over its real range, through the public entry points of
gotransformers_amd (device buffers are torch tensors):

  layer  one MoE forward over device-resident fp32 rows (forward_device), from
         a single generated token to a long prefill, with the expert path
         chosen by the library or the fp32-accuracy path asked for;
  stack  the MoE half of several consecutive blocks, x <- x + MoE(RMSNorm(x)),
         over a device-resident residual stream (stack_forward_device);
  host   the layer's host call as the Go package makes it for every Forward:
         float64 rows in and out, then the cached routing state;
  train  one optimizer step's worth of low-rank adapter training: a few
         micro-batches of forward and backward through the host calls, then
         every adapter's accumulated gradients read back.

The layer shapes are the ones the benchmark and the tests run: d=1024 E=16
k=2 h=2048 Int8; d=1024 E=64+1 shared k=6 h=512 FP4; d=2048 E=128 k=8 h=768
Int8 with skewed routing; d=2048 E=64+1 k=4 h=1024 FP4; d=256 E=8 k=2 h=512
Float32; and a layer of ragged widths with clamped SwiGLU.
"""
import math

import numpy as np
import torch

import gotransformers_amd as gt

PRECISIONS = {"int8": gt.INT8, "fp4": gt.FP4, "fp32": gt.FLOAT32}
PATHS = {"auto": gt.PATH_AUTO, "fp32": gt.PATH_FP32}
POOL_ROWS = 1024
FP4_VALUES = np.array([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0])
NORM_EPS = 1e-6

SHAPES = {
    "small": dict(d=256, h=512, E=8, S=0, k=2, prec="fp32", zipf=0.0, clamp=0.0),
    "wide": dict(d=1024, h=2048, E=16, S=0, k=2, prec="int8", zipf=0.0, clamp=0.0),
    "many": dict(d=1024, h=512, E=64, S=1, k=6, prec="fp4", zipf=0.0, clamp=0.0),
    "skewed": dict(d=2048, h=768, E=128, S=0, k=8, prec="int8", zipf=0.6, clamp=0.0),
    "block": dict(d=2048, h=1024, E=64, S=1, k=4, prec="fp4", zipf=0.0, clamp=0.0),
    "ragged": dict(d=1000, h=1201, E=14, S=2, k=3, prec="int8", zipf=0.0, clamp=2.0),
}


def _case(kind, shape, T, layers=1, path="auto", hashed=False, rank=0, micro=1, **changes):
    c = dict(SHAPES[shape], kind=kind, T=T, layers=layers, path=path, hashed=hashed, rank=rank, micro=micro)
    c.update(changes)
    return c


def listed():
    cases = {
        # one generated token: launches and latency
        "decode_int8_t1": _case("layer", "wide", 1),
        # a decode batch of 32 sequences
        "decode_int8_t32": _case("layer", "wide", 32),
        # an odd decode batch near the end of the range the library calls decode
        "decode_fp4_t113": _case("layer", "block", 113),
        # decode through consecutive blocks, their weights far larger than any cache
        "decode_stack_fp4_t64": _case("stack", "block", 64, layers=8),
        # the Go package's Forward during batched decode
        "host_int8_t24": _case("host", "wide", 24),
        # Float32 experts with the accurate path asked for, as a numerics check does
        "accurate_f32_t128": _case("layer", "small", 128, path="fp32"),
        # a short prompt, or decode and prompt chunks batched together
        "chunk_fp4_t333": _case("layer", "block", 333),
        # ragged widths, clamped SwiGLU, two shared experts
        "ragged_int8_t777": _case("layer", "ragged", 777),
        # prefill over many small experts
        "prefill_fp4_t4096": _case("layer", "many", 4096),
        # a long prefill whose routing is skewed
        "prefill_int8_t16384": _case("layer", "skewed", 16384),
        # a prefill chunk through consecutive blocks
        "prefill_stack_fp4_t8192": _case("stack", "block", 8192, layers=3),
        # adapter training with gradient accumulation
        "train_fp4_t512": _case("train", "many", 512, rank=16, micro=4),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    what = rng.choice(["decode", "decode", "decode_stack", "host", "accurate", "chunk", "prefill", "prefill_stack",
                       "train"])
    hashed = rng.random() < 0.15
    clamp = 3.0 if rng.random() < 0.2 else 0.0
    if what == "decode":
        shape = rng.choice(["wide", "many", "skewed", "block", "ragged"])
        return _case("layer", shape, log_int(1, {"wide": 64, "ragged": 37}.get(shape, 128)), hashed=hashed,
                     clamp=clamp, prec=rng.choice(["int8", "fp4"]))
    if what == "decode_stack":
        return _case("stack", rng.choice(["wide", "block"]), log_int(1, 64), layers=rng.randint(2, 8),
                     prec=rng.choice(["int8", "fp4"]))
    if what == "host":
        return _case("host", rng.choice(["wide", "many", "block", "ragged"]), log_int(1, 1024), hashed=hashed,
                     clamp=clamp)
    if what == "accurate":
        return _case("layer", rng.choice(["small", "wide", "many", "ragged"]), log_int(65, 1024), path="fp32",
                     prec=rng.choice(["fp32", "int8", "fp4"]))
    if what == "chunk":
        return _case("layer", rng.choice(["wide", "many", "block", "ragged"]), log_int(130, 1024), hashed=hashed,
                     clamp=clamp, prec=rng.choice(["int8", "fp4"]))
    if what == "prefill":
        shape = rng.choice(["wide", "many", "skewed", "block", "ragged"])
        return _case("layer", shape, log_int(1024, 16384 if shape == "skewed" else 8192),
                     prec=rng.choice(["int8", "fp4"]))
    if what == "prefill_stack":
        return _case("stack", "block", log_int(512, 8192), layers=rng.randint(2, 3))
    shape = rng.choice(["small", "wide", "many"])
    return _case("train", shape, log_int(16, 512), rank=rng.choice([4, 8, 16]),
                 micro=rng.randint(1, 2 if shape == "many" else 4))


# --------------------------------------------------------------------------
# weights and inputs, from the seed alone
# --------------------------------------------------------------------------

def _rng(case, seed, what):
    key = [seed, case["d"], case["h"], case["E"], case["k"], case["S"], case["T"], case["layers"], case["rank"], what]
    return np.random.default_rng(key)


def _encode(prec, w):
    """Rows of w in the reference's storage: per-16-value blocks, absmax/127
    (Int8) or absmax/6 (FP4, even value in the low nibble) scales."""
    rows, width = w.shape
    if prec == "fp32":
        return w.astype(np.float32), None
    blocks = -(-width // 16)
    padded = np.zeros((rows, blocks * 16), np.float32)
    padded[:, :width] = w
    b = padded.reshape(rows, blocks, 16)
    scale = np.abs(b).max(axis=2) / np.float32(127.0 if prec == "int8" else 6.0)
    scale = np.where(scale == 0, np.float32(1), scale).astype(np.float32)
    q = b / scale[:, :, None]
    if prec == "int8":
        codes = np.clip(np.rint(q), -127, 127).astype(np.int8).reshape(rows, -1)[:, :width]
        return np.ascontiguousarray(codes), scale
    mids = (FP4_VALUES[1:] + FP4_VALUES[:-1]) / 2
    m = np.searchsorted(mids.astype(np.float32), np.abs(q)).astype(np.uint8)
    m |= np.where(q < 0, 8, 0).astype(np.uint8)
    m = m.reshape(rows, -1)
    return np.ascontiguousarray(m[:, 0::2] | (m[:, 1::2] << 4))[:, :(width + 1) // 2].copy(), scale


class _Rows:
    """One matrix as gtmoe_rows takes it."""

    def __init__(self, prec, rows, width, values, scales):
        self.precision, self.rows, self.width, self.values, self.scales = PRECISIONS[prec], rows, width, values, scales


def _matrices(case, seed, layer):
    """The expert matrices of one layer: an iterator over ((kind, index,
    which), rows, biases).  Every matrix takes its rows in its own order from
    a pool of N(0, 0.02) rows, its block scales varied row by row."""
    rng = _rng(case, seed, 100 + layer)
    d, h = case["d"], case["h"]
    pools = {w: _encode(case["prec"], rng.standard_normal((POOL_ROWS, w), dtype=np.float32) * np.float32(0.02))
             for w in {d, h}}
    for kind, count in (("shared", case["S"]), ("routed", case["E"])):
        for i in range(count):
            for which, rows, width in (("gate", h, d), ("up", h, d), ("down", d, h)):
                values, scales = pools[width]
                pick = np.concatenate([rng.permutation(POOL_ROWS) for _ in range(-(-rows // POOL_ROWS))])[:rows]
                sc = None
                if scales is not None:
                    sc = scales[pick] * rng.uniform(0.7, 1.4, (rows, 1)).astype(np.float32)
                yield (kind, i, which), _Rows(case["prec"], rows, width, values[pick], sc), \
                    rng.standard_normal(rows) * 0.01


def _router(case, seed, layer):
    rng = _rng(case, seed, 200 + layer)
    w = (rng.standard_normal((case["E"], case["d"])) * 0.02).astype(np.float32)
    b = rng.standard_normal(case["E"]) * 0.01
    if case["zipf"]:
        p = 1.0 / np.arange(1, case["E"] + 1) ** 1.2
        b[rng.permutation(case["E"])] += case["zipf"] * np.log(p / p[0])
    return w, b


def _norm(case, seed, layer):
    return _rng(case, seed, 300 + layer).uniform(0.8, 1.2, case["d"])


def _inputs(case, seed, micro=0):
    """Token rows (activations after a norm: unit variance) and token ids."""
    rng = _rng(case, seed, 400 + micro)
    return (rng.standard_normal((case["T"], case["d"])).astype(np.float32),
            rng.integers(0, 50000, case["T"]))


def _output_gradients(case, seed, micro):
    return _rng(case, seed, 500 + micro).standard_normal((case["T"], case["d"])) * 1e-2


def _adapter_keys(case):
    for kind, count in (("shared", case["S"]), ("routed", case["E"])):
        for i in range(count):
            for which in ("gate", "up", "down"):
                yield kind, i, which
    yield "router", 0, None


def _adapter_shape(case, which):
    """(inputs, outputs) of the layer an adapter sits on; which None: the router."""
    return {"gate": (case["d"], case["h"]), "up": (case["d"], case["h"]), "down": (case["h"], case["d"]),
            None: (case["d"], case["E"])}[which]


def _adapters(case, seed):
    """Adapters some steps into training: (Down, Up) per layer."""
    rng = _rng(case, seed, 600)
    for key in _adapter_keys(case):
        inputs, outputs = _adapter_shape(case, key[2])
        r = min(case["rank"], inputs, outputs)
        yield key, rng.uniform(-1, 1, (r, inputs)) / math.sqrt(inputs), rng.standard_normal((outputs, r)) * 0.01


# --------------------------------------------------------------------------
# what a program holds, and one pass
# --------------------------------------------------------------------------

_context = None


def _open():
    global _context
    if _context is None:
        _context = gt.Context(0)
    return _context


class _State:
    def __init__(self, case):
        self.case = case
        self.layers = []

    def __del__(self):
        for m in self.layers:
            m.destroy()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def prepare(case, seed):
    st = _State(case)
    for layer in range(case["layers"]):
        m = gt.MixtureOfExperts(_open(), case["d"], case["h"], case["S"], case["E"], case["k"],
                                PRECISIONS[case["prec"]], case["clamp"], case["hashed"])
        st.layers.append(m)
        for (kind, i, which), rows, biases in _matrices(case, seed, layer):
            m.upload(kind, i, which, rows, biases)
        if not case["hashed"]:
            w, b = _router(case, seed, layer)
            m.upload_router(_Rows("fp32", case["E"], case["d"], w, None), b)
        if case["kind"] == "stack":
            m.set_norm_weights(_norm(case, seed, layer))
    x, ids = _inputs(case, seed)
    st.path = PATHS[case["path"]]
    if case["kind"] in ("layer", "stack"):
        st.x0 = torch.from_numpy(x).cuda()
        st.ids = torch.from_numpy(ids).cuda() if case["hashed"] else None
        st.ids_ptr = st.ids.data_ptr() if case["hashed"] else None
        st.y = torch.empty_like(st.x0)
    elif case["kind"] == "host":
        st.x = x.astype(np.float64)
        st.ids = ids if case["hashed"] else None
    else:
        m = st.layers[0]
        m.add_adapters(case["rank"], 2.0 * case["rank"])
        for key, down, up in _adapters(case, seed):
            m.set_adapter(*key, down, up)
        st.x = [_inputs(case, seed, i)[0].astype(np.float64) for i in range(case["micro"])]
        st.g = [_output_gradients(case, seed, i) for i in range(case["micro"])]
        # the optimizer's flat gradient vector: each adapter's Down and Up in turn
        st.grads = np.zeros(sum(dn.size + up.size for _, dn, up in _adapters(case, seed)))
    return st


def _read_gradients(case, m, flat):
    """Every adapter's gradients into the optimizer's vector, in place."""
    lib, at = gt.library(), flat.ctypes.data
    for kind, i, which in _adapter_keys(case):
        inputs, outputs = _adapter_shape(case, which)
        r = min(case["rank"], inputs, outputs)
        role = gt.ROLE_ROUTER if kind == "router" else gt.ROLES[(kind, which)]
        m.ctx.check(lib.gtmoe_layer_adapter_gradients(m.handle, role, i, at, at + 8 * r * inputs))
        at += 8 * r * (inputs + outputs)


def run(state):
    c, kind = state.case, state.case["kind"]
    if kind == "layer":
        state.layers[0].forward_device(c["T"], state.x0.data_ptr(), state.y.data_ptr(), state.ids_ptr, state.path,
                                       _stream())
        return state.y
    if kind == "stack":
        state.y.copy_(state.x0)
        gt.stack_forward_device(state.layers, c["T"], state.y.data_ptr(), None, state.path, _stream())
        return state.y
    m = state.layers[0]
    if kind == "host":
        y = m.forward(state.x, state.ids)
        r = m.last_routing()
        return {"y": y, "gates": r.gates, "chosen": r.chosen, "load": r.load}
    m.zero_adapter_gradients()
    out = {"y": [], "dx": [], "grads": state.grads}
    for x, g in zip(state.x, state.g):
        out["y"].append(m.forward(x))
        out["dx"].append(m.backward(g))
    _read_gradients(c, m, state.grads)
    return out


# --------------------------------------------------------------------------
# bounds
# --------------------------------------------------------------------------

def work(case):
    T, d, h, E, k, S = (case[n] for n in ("T", "d", "h", "E", "k", "S"))
    per_value = {"int8": 1.0, "fp4": 0.5, "fp32": 4.0}[case["prec"]] + (0.0 if case["prec"] == "fp32" else 0.25)
    active = S + E * (1.0 - (1.0 - k / E) ** T)
    weights = active * 3 * d * h * per_value + E * d * 4
    flops = 2.0 * T * ((S + k) * 3 * d * h + E * d)
    if case["kind"] == "train":
        P, R = T * (S + k), case["rank"]
        adapters = R * ((S + E) * 3 * (d + h) + d + E)
        lora = 3 * 2.0 * R * (P * 3 * (d + h) + T * (d + E))
        return {"bytes": weights + adapters * (4 + 8) + case["micro"] * T * d * 8 * 4,
                "flops": case["micro"] * (2 * flops + lora)}
    rows = 2 * T * d * (8 if case["kind"] == "host" else 4)
    if case["kind"] == "host":
        rows += T * k * 12 + E * 4
    return {"bytes": case["layers"] * weights + rows, "flops": case["layers"] * flops}


def _fp32_experts(case):
    few = case["T"] * case["k"] <= 8 * case["E"]
    return case["kind"] == "train" or case["path"] == "fp32" or few


def tolerance(case):
    """About four times the distance from 64-bit arithmetic.  Accurate path
    (and training): fp32 sums over tokens kept to 16 significant bits,
    5e-6 to 7e-6.  Otherwise bf16 operands with fp32 sums, 4.4e-3; through a
    stack also tokens whose k-th and next expert are nearly tied and change
    places, 1.7e-2 over three blocks."""
    if _fp32_experts(case):
        return {"rel": 3e-5, "differ": 0.02}
    return {"rel": 1.5e-2 if case["layers"] == 1 else 6e-2, "differ": 0.02}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------

def _decode64(rows):
    v = torch.from_numpy(rows.values).cuda()
    if rows.scales is None:
        return v.double()
    s = torch.from_numpy(rows.scales).cuda().double()
    if rows.precision == gt.FP4:
        table = torch.from_numpy(np.concatenate([FP4_VALUES, -FP4_VALUES])).cuda()
        v = torch.stack([table[(v & 15).long()], table[(v >> 4).long()]], dim=2).reshape(rows.rows, -1)
        v = v[:, :rows.width]
    return v.double() * s.repeat_interleave(16, dim=1)[:, :rows.width]


def _route64(case, logits, ids):
    E, k = case["E"], case["k"]
    if case["hashed"]:
        first = (ids.astype(np.uint64) * np.uint64(2654435761) + np.uint64(12345)) % np.uint64(E)
        chosen = (torch.from_numpy(first.astype(np.int64)).cuda()[:, None] + torch.arange(k, device="cuda")) % E
        return chosen, torch.full((len(ids), k), 1.0 / k, dtype=torch.float64, device="cuda")
    affinity = torch.sqrt(torch.nn.functional.softplus(logits, threshold=1e9))
    chosen = affinity.topk(k, dim=1).indices.sort(dim=1).values
    gates = affinity.gather(1, chosen)
    return chosen, gates / gates.sum(dim=1, keepdim=True)


def _layer64(case, seed, layer, x, ids, adapters=None):
    """One layer over rows x; adapters: key -> (Down, Up) tensors."""
    def linear(v, key, w, b):
        y = v @ w.T
        if adapters is not None:
            down, up = adapters[key]
            y = y + (2.0 * case["rank"] / down.shape[0]) * ((v @ down.T) @ up.T)
        return y + torch.from_numpy(b).cuda()

    logits = None
    if not case["hashed"]:
        w, b = _router(case, seed, layer)
        logits = linear(x, ("router", 0, None), torch.from_numpy(w).cuda().double(), b)
    chosen, gates = _route64(case, logits, ids)
    y = torch.zeros_like(x)
    expert = {}
    for key, rows, biases in _matrices(case, seed, layer):
        expert[key[2]] = (key, _decode64(rows), biases)
        if key[2] != "down":
            continue
        if key[0] == "shared":
            tokens, weight = slice(None), 1.0
        else:
            tokens, slot = torch.nonzero(chosen == key[1], as_tuple=True)
            weight = gates[tokens, slot][:, None]
        v = x[tokens]
        gate, up = linear(v, *expert["gate"]), linear(v, *expert["up"])
        if case["clamp"]:
            gate, up = gate.clamp(max=case["clamp"]), up.clamp(-case["clamp"], case["clamp"])
        out = linear(torch.nn.functional.silu(gate) * up, *expert["down"]) * weight
        y = y + out if key[0] == "shared" else y.index_add(0, tokens, out)
    return y, chosen, gates


def _train64(case, seed):
    adapters = {key: tuple(torch.from_numpy(a.astype(np.float32)).cuda().double().requires_grad_() for a in (dn, up))
                for key, dn, up in _adapters(case, seed)}
    out = {"y": [], "dx": []}
    for i in range(case["micro"]):
        x = torch.from_numpy(_inputs(case, seed, i)[0]).cuda().double().requires_grad_()
        y, _, _ = _layer64(case, seed, 0, x, None, adapters)
        y.backward(torch.from_numpy(_output_gradients(case, seed, i)).cuda())
        out["y"].append(y.detach().cpu().numpy())
        out["dx"].append(x.grad.cpu().numpy())
    out["grads"] = np.concatenate([np.zeros(a.numel()) if a.grad is None else a.grad.flatten().cpu().numpy()
                                   for key in _adapter_keys(case) for a in adapters[key]])
    return out


def exact(case, seed):
    if case["kind"] == "train":
        return _train64(case, seed)
    rows, ids = _inputs(case, seed)
    x = torch.from_numpy(rows).cuda().double()
    if case["kind"] == "stack":
        for layer in range(case["layers"]):
            norm = torch.from_numpy(_norm(case, seed, layer)).cuda()
            v = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + NORM_EPS) * norm
            x = x + _layer64(case, seed, layer, v, ids)[0]
        return x
    y, chosen, gates = _layer64(case, seed, 0, x, ids)
    if case["kind"] == "layer":
        return y
    return {"y": y.cpu().numpy(), "gates": gates.cpu().numpy(), "chosen": chosen.int().cpu().numpy(),
            "load": torch.bincount(chosen.flatten(), minlength=case["E"]).int().cpu().numpy()}
