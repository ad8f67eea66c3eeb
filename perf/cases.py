"""Performance cases: the work that users of ojasx_amd have it do, through its entry points.

* ``linear``: one ``E8LatticeLinear`` forward call, from a single token to a prefill of
  thousands of rows, in every bitrate, with bias, LoRA adapter and Hadamard rotation;
* ``train``: the same layer's forward and backward (gradients of x, adapter and bias);
* ``stack``: the grouped decode GEMV over the linears of a decoder stack, one launch;
* ``step``: the E8 launches of one decode step of a decoder (fused q/k/v with rank-8
  adapters on q and v, o, fused gate/up, down, lm_head), replayed from a captured graph;
* ``encode``: packing of weight matrices, as a model conversion does it layer by layer;
* ``moment``: an optimizer's E8-packed first moment, unpacked and packed again.

Packed weights are made here with plain torch from N(0, 0.02) matrices (0.1% of the
entries of an ``encode`` case are +-8 sigma outliers), so inputs do not depend on the
package's own encoder.
"""

import math
import os
import sys

import torch

_PKG = os.path.abspath("ojasx-open-source-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ojasx_amd  # noqa: E402
from ojasx_amd import optim_state  # noqa: E402
from ojasx_amd.grouped import GroupedGemv, stack_jobs  # noqa: E402

DEV = torch.device("cuda:0")
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
CODE_BYTES = {1.0: 1 / 8, 1.5: 3 / 16, 2.0: 1 / 4}  # per weight


def listed():
    def lin(name, kind, bitrate, gs, m, n, k, dtype, bias=False, rank=0, hadamard=False):
        return {"name": name, "kind": kind, "bitrate": bitrate, "gs": gs, "m": m, "n": n, "k": k,
                "dtype": dtype, "bias": bias, "rank": rank, "hadamard": hadamard}

    def stack(name, bitrate, gs, m, layers):
        return {"name": name, "kind": "stack", "bitrate": bitrate, "gs": gs, "m": m,
                "layers": layers, "hidden": 4096, "kv": 1024, "ffn": 14336, "dtype": "bf16"}

    return [
        # one projection called eagerly on one token: the smallest call, where latency and
        # the host's work per call count
        lin("token_linear", "linear", 1.5, 32, 1, 4096, 4096, "bf16"),
        # the same layer left in torch's default dtype: fp32 activations on one token
        lin("token_linear_fp32", "linear", 1.5, 32, 1, 4096, 4096, "fp32"),
        # a batch between decode and prefill through a layer converted with from_linear's
        # defaults (2 bits, group size 8, bias); ragged rows and columns
        lin("batch_default_fp16", "linear", 2.0, 8, 77, 4100, 3072, "fp16", bias=True),
        # the largest prefill: 8192 tokens through the gate / up projection
        lin("prefill_8192", "linear", 1.5, 32, 8192, 14336, 4096, "bf16"),
        # a decode step at batch 4: the launches of 8 decoder layers and the lm_head
        {"name": "decode_step", "kind": "step", "bitrate": 1.5, "gs": 32, "m": 4, "layers": 8,
         "hidden": 4096, "kv": 1024, "ffn": 14336, "vocab": 128256, "rank": 8, "dtype": "bf16"},
        # weight streaming at its plainest: every linear of a 32-layer decoder in one launch,
        # for one token, for a batch of 16, and in the default bitrate for a batch of 4
        stack("stack_token", 1.5, 32, 1, 32),
        stack("stack_batch16", 1.5, 32, 16, 32),
        stack("stack_2bit_batch4", 2.0, 32, 4, 16),
        # fine-tuning: forward and backward of a projection with a rank-8 adapter, ternary
        # group 64, over 2048 tokens in bf16 ...
        lin("train_lora", "train", 1.5, 64, 2048, 4096, 4096, "bf16", rank=8),
        # ... and one sequence of 16 tokens in fp32 through gate / up
        lin("train_lora_fp32", "train", 1.5, 64, 16, 14336, 4096, "fp32", rank=8),
        # conversion of one fp16 weight matrix
        {"name": "encode_fp16", "kind": "encode", "bitrate": 1.5, "gs": 32, "n": 14336, "k": 4096,
         "dtype": "fp16"},
        # an optimizer step's traffic with an E8-packed moment
        {"name": "moment", "kind": "moment", "n": 4096, "k": 4096, "dtype": "fp32"},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def mult(lo, hi, unit):
        return max(1, log(lo, hi) // unit) * unit

    def gs_of(bitrate):
        return rng.choice([16, 32, 32, 64]) if bitrate == 1.5 else rng.choice([8, 16, 32, 64])

    kind = rng.choice(["linear"] * 5 + ["train"] * 2 + ["stack", "step", "encode", "moment"])
    bitrate = rng.choice([1.5, 1.5, 2.0, 1.0])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind in ("linear", "train"):
        gs = gs_of(bitrate)
        # widths are mostly multiples of 256, some of 64 and a few of the group size only
        unit = rng.choice([1024, 256, 256, 64, 64, gs])
        k = mult(256, 14336, unit)
        n = rng.choice([mult(256, 14336, 64), mult(256, 14336, 64), log(256, 14336)])
        m = log(1, 8192)
        if dtype == "fp32" or k % 64 or (kind == "train" and n % 64):
            m = log(1, 64)
        while m * n * k > 8192 * 4096 * 4096:
            m //= 2
        return {"kind": kind, "bitrate": bitrate, "gs": gs, "m": m, "n": n, "k": k,
                "dtype": dtype, "bias": rng.random() < 0.4, "rank": rng.choice([0, 0, 8, 16]),
                "hadamard": rng.random() < 0.15 and k % 32 == 0}
    if kind in ("stack", "step"):
        hidden = mult(1024, 4096, 256)
        case = {"kind": kind, "bitrate": bitrate, "gs": 32 if bitrate == 1.5 else gs_of(bitrate),
                "m": rng.choice([1, 2, 4, rng.randint(1, 16)]), "layers": rng.randint(2, 16),
                "hidden": hidden, "kv": mult(hidden // 8, hidden, 64),
                "ffn": mult(hidden * 2, min(hidden * 4, 14336), 256),
                "dtype": "fp16" if dtype == "fp16" else "bf16"}
        if kind == "step":
            case["layers"] = rng.randint(1, 6)
            case["vocab"] = log(16384, 128256)
            case["rank"] = rng.choice([0, 8, 8, 16])
        return case
    n, k = log(256, 14336), log(256, 4096)
    if kind == "encode":
        k = rng.choice([mult(256, 4096, 64), mult(256, 4096, 64), k])
        gs = rng.choice([16, 32, 64, 128]) if bitrate == 1.5 else rng.choice([8, 16, 32, 64])
        return {"kind": kind, "bitrate": bitrate, "gs": gs, "n": n, "k": k, "dtype": dtype}
    return {"kind": "moment", "n": n, "k": k, "dtype": "fp32"}


# ------------------------------------------------------------------ packed weights

def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * (salt + 1) + seed)


def _root_table():
    rows = []
    for i in range(8):
        for j in range(i + 1, 8):
            for a in (-2, 2):
                for b in (-2, 2):
                    r = [0] * 8
                    r[i], r[j] = a, b
                    rows.append(r)
    for p in range(256):
        r = [1 if (p >> (7 - t)) & 1 else -1 for t in range(8)]
        if r.count(-1) % 2 == 0:
            rows.append(r)
    for i in range(8):
        for a in (-2, 2):
            r = [0] * 8
            r[i] = a
            rows.append(r)
    return torch.tensor(rows, dtype=torch.float32, device=DEV)


def _even(q, v, alt):
    """Moves the coordinate that costs least of every 8-vector whose sum is odd."""
    pen = (alt - v).square_().sub_((q - v).square_())
    at = pen.argmin(dim=1, keepdim=True)
    odd = (q.sum(dim=1, keepdim=True) % 2) != 0
    return q.scatter(1, at, torch.where(odd, alt.gather(1, at), q.gather(1, at)))


def _packed(bitrate, n, k, gs, gen):
    """Codes and fp16 scales of an N(0, 0.02) matrix [n, k], groups along the flat matrix."""
    pad = -(n * k) % gs
    w = torch.randn(n * k + pad, generator=gen, device=DEV) * 0.02
    if pad:
        w[n * k:] = 0
    groups = w.view(-1, gs)
    scales = (groups.norm(dim=1) / math.sqrt(gs) + 1e-8).half()
    v = (groups / scales.float()[:, None]).view(-1, 8)
    if bitrate == 1.5:
        q = v.round().clamp_(-1, 1)
        q = _even(q, v, torch.where(q != 0, torch.zeros_like(q), torch.where(v < 0, -1.0, 1.0)))
        powers = torch.tensor([3 ** i for i in range(8)], dtype=torch.float32, device=DEV)
        # (not a matrix-vector product: over more than 2^24 rows the library's is wrong)
        code = ((q + 1) * powers).sum(dim=1).to(torch.int32) // 2
        pair = code[0::2] | (code[1::2] << 12)
        packed = torch.stack([pair & 255, (pair >> 8) & 255, pair >> 16], dim=1)
    elif bitrate == 2.0:
        x = v - 0.5
        q = x.round().clamp_(-2, 1)
        q = _even(q, x, torch.where(x > q, q + 1, q - 1).clamp_(-2, 1))
        c = (q + 2).to(torch.int32).view(-1, 4)
        packed = c[:, 0] | (c[:, 1] << 2) | (c[:, 2] << 4) | (c[:, 3] << 6)
    else:
        table = _root_table()
        unit = (table / table.norm(dim=1, keepdim=True)).t().contiguous()
        code = torch.cat([(part @ unit).argmax(dim=1) for part in v.split(1 << 20)])
        q = table[code].view(-1, gs)
        scales = ((groups * q).sum(dim=1) / q.square().sum(dim=1)).half()
        packed = code
    return packed.reshape(-1).to(torch.uint8), scales


def _dense(bitrate, packed, scales, n, k, gs, dtype):
    """The weights a layer in `dtype` holds, as 64-bit values."""
    b = packed.to(torch.int32)
    if bitrate == 1.5:
        b = b.view(-1, 3)
        pair = b[:, 0] | (b[:, 1] << 8) | (b[:, 2] << 16)
        raw = torch.stack([pair & 4095, pair >> 12], dim=1).view(-1, 1) * 2
        powers = torch.tensor([3 ** i for i in range(8)], dtype=torch.int32, device=DEV)
        q = (raw // powers) % 3 - 1
    elif bitrate == 2.0:
        shifts = torch.tensor([0, 2, 4, 6], dtype=torch.int32, device=DEV)
        q = ((b[:, None] >> shifts) & 3) - 1.5
    else:
        q = _root_table()[b]
    w = q.reshape(-1, gs).to(dtype) * scales.to(dtype)[:, None]
    return w.reshape(-1)[: n * k].view(n, k).double()


def _rows(m, k, dtype, gen, scale=1.0):
    return (torch.randn(m, k, generator=gen, device=DEV) * scale).to(dtype)


def _layer_data(case, n, k, bias, rank, gen):
    dt = DTYPES[case["dtype"]]
    d = {"n": n, "k": k}
    d["packed"], d["scales"] = _packed(case["bitrate"], n, k, case["gs"], gen)
    d["bias"] = _rows(1, n, dt, gen, 0.1).view(n) if bias else None
    d["a"] = _rows(k, rank, dt, gen, 0.02) if rank else None
    d["b"] = _rows(rank, n, dt, gen, 0.02) if rank else None
    return d


def _layer(case, d, hadamard=False):
    rank = 0 if d["a"] is None else d["a"].shape[1]
    layer = ojasx_amd.E8LatticeLinear(d["k"], d["n"], bias=d["bias"] is not None, rank=rank,
                                      group_size=case["gs"], bitrate=case["bitrate"],
                                      use_hadamard=hadamard, device=DEV,
                                      dtype=DTYPES[case["dtype"]])
    with torch.no_grad():
        layer.packed_weight.copy_(d["packed"])
        layer.block_scales.copy_(d["scales"])
        if d["bias"] is not None:
            layer.bias.copy_(d["bias"])
        if rank:
            layer.lora_A.copy_(d["a"])
            layer.lora_B.copy_(d["b"])
    return layer


def _linear_data(case, seed):
    gen = _gen(seed)
    d = _layer_data(case, case["n"], case["k"], case["bias"], case["rank"], gen)
    dt = DTYPES[case["dtype"]]
    x = _rows(case["m"], case["k"], dt, gen)
    gy = _rows(case["m"], case["n"], dt, gen, 0.02) if case["kind"] == "train" else None
    return d, x, gy


def _stack_shapes(case):
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f)]


def _stack_data(case, seed):
    gen = _gen(seed)
    dt = DTYPES[case["dtype"]]
    xs = {k: _rows(case["m"], k, dt, gen) for k in sorted({case["hidden"], case["ffn"]})}
    linears = []
    for _ in range(case["layers"]):
        for n, k in _stack_shapes(case):
            packed, scales = _packed(case["bitrate"], n, k, case["gs"], gen)
            linears.append({"packed": packed, "scales": scales, "N": n, "K": k})
    return xs, linears


def _step_data(case, seed):
    gen = _gen(seed)
    dt = DTYPES[case["dtype"]]
    x = _rows(case["m"], case["hidden"], dt, gen, 0.5)
    act = _rows(case["m"], case["ffn"], dt, gen, 0.5)
    layers = []
    for _ in range(case["layers"]):
        ranks = [case["rank"], 0, case["rank"], 0, 0, 0, 0]  # adapters on q and v
        layers.append([_layer_data(case, n, k, False, r, gen)
                       for (n, k), r in zip(_stack_shapes(case), ranks)])
    head = _layer_data(case, case["vocab"], case["hidden"], False, 0, gen)
    return x, act, layers, head


def _encode_data(case, seed):
    gen = _gen(seed)
    w = torch.randn(case["n"], case["k"], generator=gen, device=DEV) * 0.02
    far = torch.rand(case["n"], case["k"], generator=gen, device=DEV) < 1e-3
    sign = torch.where(w < 0, -0.16, 0.16)
    return torch.where(far, sign, w).to(DTYPES[case["dtype"]])


def _moment_data(case, seed):
    gen = _gen(seed)
    packed, scales = _packed(2.0, 1, case["n"] * case["k"] + -(case["n"] * case["k"]) % 32, 32, gen)
    moment = torch.randn(case["n"], case["k"], generator=gen, device=DEV) * 1e-3
    return packed, scales, moment


# ------------------------------------------------------------------ the passes

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear", "train"):
        d, x, gy = _linear_data(case, seed)
        layer = _layer(case, d, case["hadamard"])
        state = {"kind": kind, "layer": layer, "x": x}
        if kind == "linear":
            layer.requires_grad_(False)
        else:
            state["x"] = x.requires_grad_(True)
            state["gy"] = gy
            state["wrt"] = [x] + [p for p in (layer.lora_A, layer.lora_B, layer.bias)
                                  if p is not None]
        return state
    if kind == "stack":
        xs, linears = _stack_data(case, seed)
        dt = DTYPES[case["dtype"]]
        # one output buffer per decoder layer, the linears' [m, n] results one after another
        per = [case["m"] * n for n, _ in _stack_shapes(case)]
        outs = [torch.empty(sum(per), dtype=dt, device=DEV) for _ in range(case["layers"])]
        ys = [y for out in outs for y in out.split(per)]
        keep = [t for l in linears for t in (l["packed"], l["scales"])] + list(xs.values())
        plan = GroupedGemv(stack_jobs(linears, xs, ys), case["m"], dt, DEV, keep=keep,
                           bitrate=case["bitrate"], group_size=case["gs"])
        return {"kind": kind, "plan": plan, "outs": outs}
    if kind == "step":
        return _prepare_step(case, seed)
    if kind == "encode":
        packer = {1.0: ojasx_amd.RootE8LatticePacker, 1.5: ojasx_amd.TernaryE8LatticePacker,
                  2.0: ojasx_amd.E8LatticePacker}[case["bitrate"]]
        return {"kind": kind, "packer": packer, "gs": case["gs"], "w": _encode_data(case, seed)}
    packed, scales, moment = _moment_data(case, seed)
    old = {"exp_avg_packed": packed, "exp_avg_scales": scales,
           "exp_avg_padded_rows": packed.numel() * 4 // 32}
    return {"kind": kind, "old": old, "moment": moment}


def _prepare_step(case, seed):
    x, act, data, head_data = _step_data(case, seed)
    dt = DTYPES[case["dtype"]]
    layers = []
    for q, k, v, o, gate, up, down in [[_layer(case, d).requires_grad_(False) for d in ds]
                                       for ds in data]:
        layers.append((GroupedGemv.fused([q, k, v], case["m"], dt), o,
                       GroupedGemv.fused([gate, up], case["m"], dt), down))
    head = _layer(case, head_data).requires_grad_(False)

    def step():
        out = []
        for qkv, o, gate_up, down in layers:
            out += [qkv(x), o(x), gate_up(x), down(act)]
        return out + [head(x)]

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = step()
    return {"kind": "step", "graph": graph, "out": out, "keep": (x, act, layers, head)}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "train":
        y = state["layer"](state["x"])
        return [y.detach()] + list(torch.autograd.grad(y, state["wrt"], state["gy"]))
    if kind == "stack":
        state["plan"]()
        return state["outs"]
    if kind == "step":
        state["graph"].replay()
        return state["out"]
    if kind == "encode":
        packed, scales, _ = state["packer"].pack(state["w"], group_size=state["gs"])
        return [packed, scales]
    moment = state["moment"]
    dense = optim_state.unpack_exp_avg(state["old"], moment.shape, torch.float32)
    new = {}
    optim_state.pack_exp_avg(new, moment, True, torch.float32)
    return [dense, new["exp_avg_packed"], new["exp_avg_scales"]]


# ------------------------------------------------------------------ 64-bit results

def _fwht32(x):
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    for _ in range(5):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((x.reshape(-1, 32) @ h) / math.sqrt(32)).reshape(x.shape)


def _apply(case, d, x, scaling=0.0):
    w = _dense(case["bitrate"], d["packed"], d["scales"], d["n"], d["k"], case["gs"],
               DTYPES[case["dtype"]])
    y = x.double() @ w.t()
    if d["a"] is not None:
        y += scaling * ((x.double() @ d["a"].double()) @ d["b"].double())
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "train"):
        d, x, gy = _linear_data(case, seed)
        w = _dense(case["bitrate"], d["packed"], d["scales"], d["n"], d["k"], case["gs"],
                   DTYPES[case["dtype"]])
        x = x.double()
        y = (_fwht32(x) if case["hadamard"] else x) @ w.t()
        if d["bias"] is not None:
            y += d["bias"].double()
        if case["rank"]:
            s, a, b = 16.0 / case["rank"], d["a"].double(), d["b"].double()
            y += s * ((x @ a) @ b)
        if kind == "linear":
            return y
        gy = gy.double()
        gx = gy @ w
        if case["hadamard"]:
            gx = _fwht32(gx)
        out = [y, gx]
        if case["rank"]:
            gyb = gy @ b.t()
            gx += s * (gyb @ a.t())
            out += [s * (x.t() @ gyb), s * ((x @ a).t() @ gy)]
        if d["bias"] is not None:
            out.append(gy.sum(dim=0))
        return out
    if kind == "stack":
        xs, linears = _stack_data(case, seed)
        ys = [_apply(case, {"packed": l["packed"], "scales": l["scales"], "n": l["N"],
                            "k": l["K"], "a": None}, xs[l["K"]]).view(-1) for l in linears]
        return [torch.cat(ys[i:i + 7]) for i in range(0, len(ys), 7)]
    if kind == "step":
        x, act, layers, head = _step_data(case, seed)
        s = 16.0 / case["rank"] if case["rank"] else 0.0
        out = []
        for q, k, v, o, gate, up, down in layers:
            out += [torch.cat([_apply(case, d, x, s) for d in (q, k, v)], 1), _apply(case, o, x),
                    torch.cat([_apply(case, d, x) for d in (gate, up)], 1),
                    _apply(case, down, act)]
        return out + [_apply(case, head, x)]
    if kind == "encode":
        return None  # codes: whole numbers with the packer's own rounding and ties
    packed, scales, moment = _moment_data(case, seed)
    w = _dense(2.0, packed, scales, 1, packed.numel() * 4, 32, torch.float32)
    return [w.view(-1)[: moment.numel()].view(moment.shape), None, None]


# ------------------------------------------------------------------ bytes, operations, bounds

def _layer_work(case, m, n, k, rank=0, x_read=True):
    e = SIZE[case["dtype"]]
    weights = n * k * CODE_BYTES[case["bitrate"]] + n * k / case["gs"] * 2
    nbytes = weights + rank * (n + k) * e + m * n * e + (m * k * e if x_read else 0)
    return {"bytes": nbytes, "flops": 2.0 * m * (n * k + rank * (n + k))}


def _sum(parts):
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def work(case):
    kind = case["kind"]
    if kind in ("linear", "train"):
        m, n, k, r = case["m"], case["n"], case["k"], case["rank"]
        parts = [_layer_work(case, m, n, k, r)]
        if case["bias"]:
            parts.append({"bytes": n * SIZE[case["dtype"]], "flops": m * n})
        if kind == "train":  # the weights' codes again, gy in, gradients out
            e = SIZE[case["dtype"]]
            parts.append(_layer_work(case, m, n, k, r))
            parts.append({"bytes": (r * (n + k) + (n if case["bias"] else 0)) * e,
                          "flops": 2.0 * m * r * (n + k)})
        return _sum(parts)
    if kind in ("stack", "step"):
        per = []
        for i, (n, k) in enumerate(_stack_shapes(case)):
            r = case.get("rank", 0) if i in (0, 2) else 0
            per.append(_layer_work(case, case["m"], n, k, r, x_read=False))
        parts = per * case["layers"]
        parts.append({"bytes": case["m"] * (case["hidden"] + case["ffn"]) * SIZE[case["dtype"]],
                      "flops": 0})
        if kind == "step":
            parts.append(_layer_work(case, case["m"], case["vocab"], case["hidden"],
                                     x_read=False))
        return _sum(parts)
    numel = case["n"] * case["k"]
    if kind == "encode":
        out = numel * CODE_BYTES[case["bitrate"]] + numel / case["gs"] * 2
        return {"bytes": numel * SIZE[case["dtype"]] + out, "flops": 0}
    packed = numel / 4 + numel / 32 * 2
    return {"bytes": 2 * (numel * 4 + packed), "flops": 0}


def tolerance(case):
    if case["kind"] in ("encode", "moment"):
        return "exact"
    # about four times what exact() shows: 1.7e-3 (one rounding of an fp32 sum) to 2.5e-3 in
    # bf16, 2.1e-4 to 2.5e-4 in fp16, 1.7e-6 in fp32
    rel = {"bf16": 1e-2, "fp16": 1e-3, "fp32": 7e-6}[case["dtype"]]
    # a Hadamard rotation rounds each of its five stages to the dtype: 5e-3 and 6e-4
    return {"rel": 2 * rel if case.get("hadamard") and case["dtype"] != "fp32" else rel}
