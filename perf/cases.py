"""The work that a program using the MoE engine has it do, as measurable cases.

Every case runs through gyrodx.engine.Engine, in one of the four ways a program calls it:

  step     one decode step of a served model: gm_forward_decode_noalloc for every MoE layer of the
           step, between device tensors, captured once in a HIP graph and replayed
  layer    gm_forward: one MoE layer on host rows, the result back in host memory
  stack    gm_forward_stack: x <- x + MoE_l(RMSNorm_l(x)) through a list of layers, host rows in and out
  resident gm_run_stack over tokens uploaded once, then gm_read_outputs

Shapes are this repository's own: hidden 2048 / 256 experts / top-8 / F 512 in TQ2_T (its benchmark),
the mixed-quant layer with a bf16 shared expert of width 1024, and hidden 2560 / F 640 / top-10 (the
real model's experts). A deep stack lists its distinct layers several times over, since laying out a
whole model's weights would take longer than the passes. Prefill stacks stay a few layers deep:
further down, tokens near a routing tie take other experts after any change of rounding. Weights, routers and tokens follow
gyrodx.synth's distributions: uniform trellis bytes, block scales of random sign in [2^-8, 2^-3),
N(0, 0.02) routers (with a Zipf(1.1) bias where `zipf` says so), N(0, 1) tokens.
"""
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT / "gyro-dx_amd"))

from gyrodx import synth  # noqa: E402
from gyrodx.engine import PATH_DECODE, PATH_PREFILL, Engine  # noqa: E402

BF16, Q8_0 = 30, 8  # GGML types of a shared expert's rows

BASE = dict(E=2048, F=512, NE=256, U=8, type=144, SF=0, sh_type=BF16, zipf=False)
CODER = dict(BASE, E=2560, F=640, NE=256, U=10)


def listed():
    return [
        # The smallest call a program can make: one token through one layer, host to host.
        dict(BASE, name="layer_decode_1", call="layer", n=1, layers=1, depth=1),
        # A token and a batch of eight through four layers of a served model.
        dict(BASE, name="step_decode_1", call="step", n=1, layers=4, depth=4),
        dict(BASE, name="step_decode_8", call="step", n=8, layers=4, depth=4),
        # Layers whose experts mix all eight Gyro types, with the shared expert; an odd batch.
        dict(BASE, name="step_decode_mixed_3", call="step", n=3, layers=3, depth=3, type=0, SF=1024),
        # The real model's experts with its Q8_0 shared expert, two sequences.
        dict(CODER, name="step_decode_coder_2", call="step", n=2, layers=3, depth=3, SF=640, sh_type=Q8_0),
        # Single-stream generation through a model's MoE layers.
        dict(BASE, name="stack_decode_1", call="stack", n=1, layers=4, depth=12),
        # A short prompt, or a batch of sequences past the decode path's eight.
        dict(BASE, name="stack_prefill_37", call="stack", n=37, layers=4, depth=4),
        # A prompt chunk through one layer whose caller keeps its activations on the host.
        dict(BASE, name="layer_prefill_300", call="layer", n=300, layers=1, depth=1, prefill=True),
        # The benchmark's prompt size (one short of the round number) with its skewed router.
        dict(BASE, name="stack_prefill_1023_zipf", call="stack", n=1023, layers=3, depth=6, zipf=True),
        # Mixed types and the shared expert at the benchmark's mixed prompt size.
        dict(BASE, name="stack_prefill_mixed_509", call="stack", n=509, layers=2, depth=2, type=0, SF=1024),
        # The real model's experts in a 64-step type.
        dict(CODER, name="stack_prefill_coder_777", call="stack", n=777, layers=2, depth=2, type=148),
        # The largest call: 32,768 token slots.
        dict(BASE, name="resident_prefill_4096", call="resident", n=4096, layers=2, depth=4),
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))

    shape = rng.choice(["base", "base", "coder", "other"])
    c = dict(CODER if shape == "coder" else BASE)
    if shape == "other":
        c.update(E=256 * rng.randint(4, 12), F=128 * rng.randint(2, 6), NE=rng.choice([64, 96, 128, 192, 256]),
                 U=rng.choice([2, 4, 6, 8, 10, 16]))
    c["type"] = rng.choice([144, 144, 144, 145, 147, 148, 151, 0])
    c["zipf"] = rng.random() < 0.4
    if rng.random() < 0.4:
        c.update(SF=64 * rng.randint(4, 16), sh_type=rng.choice([BF16, Q8_0]))
    call = rng.choice(["layer", "layer", "step", "stack", "stack", "resident"])
    decode = call == "step" or rng.random() < 0.3
    c["call"] = call
    c["layers"] = 1 if call == "layer" else rng.randint(1, 3)
    c["depth"] = c["layers"] * rng.randint(1, 3) if decode and call != "step" and call != "layer" else c["layers"]
    c["n"] = rng.randint(1, 8) if decode else log_int(9, 32768 // max(c["U"], 12))
    if not decode:
        c["prefill"] = True
    return c


def is_prefill(c):
    return bool(c.get("prefill")) or c["n"] > 8


# ---- inputs ------------------------------------------------------------------------------------

def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1009 + stream)
    return g


def _types(c, seed, l):
    if c["type"]:
        return np.full((c["NE"], 3), c["type"], np.uint32)
    rng = np.random.default_rng([seed, l, 1])
    return rng.choice(np.array(sorted(synth.TYPES), np.uint32), size=(c["NE"], 3))


def _blocks(c, seed, l, p, t, count):
    """`count` matrices of projection p in Gyro type t: uint8 [count, rows, blocks, block bytes] on the GPU."""
    rows, cols = (c["F"], c["E"]) if p < 2 else (c["E"], c["F"])
    shape = (count, rows, cols // 128)
    g = _gen(seed, 1000 + 100 * l + 10 * p + (t - 144))
    raw = torch.randint(0, 256, shape + (synth.TYPES[t][2],), dtype=torch.uint8, device="cuda", generator=g)
    # Block scale: sign random, exponent field 7..11, mantissa uniform.
    half = torch.randint(0, 1024, shape, device="cuda", generator=g, dtype=torch.int32)
    half += torch.randint(7, 12, shape, device="cuda", generator=g, dtype=torch.int32) << 10
    half += torch.randint(0, 2, shape, device="cuda", generator=g, dtype=torch.int32) << 15
    raw[..., 0] = (half & 255).to(torch.uint8)
    raw[..., 1] = (half >> 8).to(torch.uint8)
    return raw


def _normal(shape, seed, stream, scale):
    return torch.randn(shape, device="cuda", generator=_gen(seed, stream), dtype=torch.float32) * scale


def _signs(n, seed, stream):
    return (torch.randint(0, 2, (n,), device="cuda", generator=_gen(seed, stream)) * 2 - 1).float()


def _zipf(c, seed, l):
    pmf = np.arange(1, c["NE"] + 1, dtype=np.float64) ** -1.1
    bias = np.empty(c["NE"])
    bias[np.random.default_rng([seed, l, 2]).permutation(c["NE"])] = np.log(pmf / pmf.sum())
    return bias.astype(np.float32)


def _small(c, seed, l):
    """Everything of layer l but the experts, on the GPU: router, bias, signs, norm, shared expert."""
    s, E, F, SF = 100 * l, c["E"], c["F"], c["SF"]
    d = dict(router=_normal((c["NE"], E), seed, s + 1, 0.02), gate_signs=_signs(E, seed, s + 2),
             down_signs=_signs(F, seed, s + 3), norm=1 + _normal((E,), seed, s + 4, 0.1),
             bias=torch.from_numpy(_zipf(c, seed, l)).cuda() if c["zipf"] else None)
    if SF:
        d["shared"] = [_normal(sh, seed, s + 5 + i, 0.02) for i, sh in enumerate(((SF, E), (SF, E), (E, SF)))]
        d["shared_gate"] = _normal((E,), seed, s + 8, 0.02)
    return d


def _make_layer(c, seed, l):
    d, NE = _small(c, seed, l), c["NE"]
    types = _types(c, seed, l)
    mats = []
    for p in range(3):
        mine = [None] * NE
        for t in np.unique(types[:, p]):
            where = np.flatnonzero(types[:, p] == t)
            raw = _blocks(c, seed, l, p, int(t), len(where)).flatten(2).cpu().numpy()
            for i, e in enumerate(where):
                mine[e] = raw[i]
        mats.append(mine)
    host = lambda t: None if t is None else t.cpu().numpy()  # noqa: E731
    layer = synth.Layer(E=c["E"], F=c["F"], n_expert=NE, n_used=c["U"], types=types, gate=mats[0], up=mats[1],
                        down=mats[2], router=host(d["router"]), router_bias=host(d["bias"]),
                        gate_signs=host(d["gate_signs"]), down_signs=host(d["down_signs"]),
                        norm_weight=host(d["norm"]))
    if c["SF"]:
        layer.SF, layer.sh_type, layer.sh_gate_inp = c["SF"], c["sh_type"], host(d["shared_gate"])
        if c["sh_type"] == BF16:
            rows = [w.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16) for w in d["shared"]]
        else:
            rows = [synth.q8_0_quantize(host(w)) for w in d["shared"]]
        layer.sh_gate, layer.sh_up, layer.sh_down = rows
    return layer


def _tokens(c, seed):
    """A step's layers get rows of their own (the attention before each makes them); the others one set."""
    return _normal((c["depth"], c["n"], c["E"]) if c["call"] == "step" else (c["n"], c["E"]), seed, 9, 1.0)


def prepare(case, seed):
    c = case
    path = PATH_PREFILL if is_prefill(c) else PATH_DECODE
    # An engine is made for the calls that a program will send it, not for the one at hand.
    eng = Engine(max_tok=8 if c["call"] == "step" else 64 if path == PATH_DECODE else 1024 if c["n"] <= 1024 else 4096)
    ids = [eng.add_layer(_make_layer(c, seed, l)) for l in range(c["layers"])]
    order = [ids[i % len(ids)] for i in range(c["depth"])]
    x = _tokens(c, seed)
    s = dict(call=c["call"], path=path, n=c["n"], order=order)
    if c["call"] == "step":
        out = torch.empty_like(x)

        def step():
            stream = torch.cuda.current_stream().cuda_stream
            for i, l in enumerate(order):
                eng.forward_decode_noalloc(l, x[i].data_ptr(), c["n"], out[i].data_ptr(), stream)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        s.update(graph=graph, x=x, out=out)
    else:
        s["x"] = x.cpu().numpy()
        if c["call"] == "resident":
            eng.set_tokens(s["x"])
    s["engine"] = eng
    return s


def run(state):
    s = state
    if s["call"] == "step":
        s["graph"].replay()
        return s["out"]
    if s["call"] == "layer":
        return s["engine"].forward(s["order"][0], s["x"], s["path"])
    if s["call"] == "stack":
        return s["engine"].forward_stack(s["order"], s["x"], s["path"])
    s["engine"].run_stack(s["path"], s["n"], 1, s["order"])
    return s["engine"].read_outputs(s["n"])


# ---- what a pass cannot do without ----------------------------------------------------------------

def _distinct(c):
    """Experts that n tokens of such a router choose, per layer."""
    rng = np.random.default_rng(5)
    logits = rng.standard_normal((c["n"], c["NE"])) * (0.02 * c["E"] ** 0.5)
    if c["zipf"]:
        logits = logits + _zipf(c, 0, 0)
    return len(np.unique(np.argpartition(-logits, c["U"] - 1, axis=1)[:, :c["U"]]))


def work(case):
    c = case
    E, F, n = c["E"], c["F"], c["n"]
    block = synth.TYPES[c["type"]][2] if c["type"] else np.mean([t[2] for t in synth.TYPES.values()])
    sh_byte = 2 if c["sh_type"] == BF16 else 34 / 32
    used = _distinct(c)
    per_layer = used * 3 * E * F / 128 * block + c["NE"] * E * 4 + 3 * E * c["SF"] * sh_byte
    # A list that names a layer again reads its weights again: other layers' weights lie between.
    ends = 2 * n * E * 4 * (c["depth"] if c["call"] == "step" else 1)
    flops = c["depth"] * n * (2 * E * c["NE"] + 6 * E * F * c["U"] + 6 * E * c["SF"])
    return {"bytes": float(c["depth"] * per_layer + ends), "flops": float(flops)}


def tolerance(case):
    """About four times the distance to exact(). Decode keeps everything in 32 bits (a layer 3e-7 to
    6e-7 off, 12 layers 1.4e-6). Prefill multiplies binary16 weights and activations (a layer
    5.5e-4 off). In a prefill stack a token whose last chosen expert and the next one are near a tie
    takes the other one after any change of rounding in a layer before, and its row then differs by
    that expert's share: 0.01 to 0.04 over the rows."""
    c = case
    if not is_prefill(c):
        return {"rel": 2e-6 if c["depth"] == 1 or c["call"] == "step" else 8e-6, "max": 1e-4}
    if c["depth"] == 1:
        return {"rel": 2.2e-3, "max": 0.05}
    return {"rel": 0.03, "max": 0.95}


# ---- the same in 64 bits --------------------------------------------------------------------------

def _decode(raw, t):
    """Gyro blocks uint8 [rows, blocks, block bytes] of type t as float64 [rows, blocks * 128]."""
    k, steps, bb = synth.TYPES[t]
    book = torch.from_numpy(np.fromfile(ROOT / "gyro-dx_amd" / "data" / "gyro_codebook.f16", np.float16)).cuda()
    pairs = book.double().view(2048, 2)
    rows, nblk, _ = raw.shape
    scale = raw[..., :2].contiguous().view(torch.float16).double()
    stream = raw[..., 2:].long()
    nb = bb - 2
    if t == 144:  # the byte before a step's own is the state's high byte
        state = (stream.roll(1, -1) << 8) | stream
    else:  # 16 bits of the circular little-endian stream at bit (steps - 1 - step) k
        off = (steps - 1 - torch.arange(steps, device=raw.device)) * k
        b = off >> 3
        word = stream[..., b] | (stream[..., (b + 1) % nb] << 8) | (stream[..., (b + 2) % nb] << 16)
        state = word >> (off & 7)
    h = ((state & 0x7FFF) * 0x9E3779B1) & 0xFFFFFFFF
    v = pairs[h >> 21]
    if steps == 32:
        v = torch.cat([v, pairs[(h >> 10) & 0x7FF]], -1)
    return (v.reshape(rows, nblk, 128) * scale).reshape(rows, nblk * 128)


def _rotate(x, signs):
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((x * signs.double()).view(-1, 128) @ (h / 128 ** 0.5)).view(x.shape)


def _silu(v):
    return v / (1 + torch.exp(-v))


def _moe64(c, seed, l, x):
    d, types = _small(c, seed, l), _types(c, seed, l)
    logits = x @ d["router"].double().T
    if d["bias"] is not None:
        logits = logits + d["bias"].double()
    w, ids = torch.topk(torch.softmax(logits, -1), c["U"], dim=-1)
    w = w / w.sum(-1, keepdim=True)
    xh = _rotate(x, d["gate_signs"])
    chosen = set(ids.unique().tolist())
    out = torch.zeros_like(x)
    mats = [{}, {}, {}]
    for p in range(3):
        for t in np.unique(types[:, p]):
            where = np.flatnonzero(types[:, p] == t)
            raw = _blocks(c, seed, l, p, int(t), len(where))
            for i, e in enumerate(where):
                mats[p][int(e)] = (raw[i], int(t))
    for e in sorted(chosen):
        tok, k = (ids == e).nonzero(as_tuple=True)
        gate, up, down = (_decode(*mats[p][e]) for p in range(3))
        a = _silu(xh[tok] @ gate.T) * (xh[tok] @ up.T)
        out.index_add_(0, tok, (_rotate(a, d["down_signs"]) @ down.T) * w[tok, k, None])
    if c["SF"]:
        if c["sh_type"] == BF16:
            sg, su, sd = (m.to(torch.bfloat16).double() for m in d["shared"])
        else:
            sg, su, sd = (_q8_values(m) for m in d["shared"])
        gate = torch.sigmoid(x @ d["shared_gate"].double())
        out += ((_silu(x @ sg.T) * (x @ su.T)) @ sd.T) * gate[:, None]
    return out


def _q8_values(w):
    """What rows hold once stored as 32-value blocks of a binary16 scale and int8 values."""
    q = torch.from_numpy(synth.q8_0_quantize(w.cpu().numpy())).view(w.shape[0], w.shape[1] // 32, 34).cuda()
    d = q[..., :2].contiguous().view(torch.float16).double()
    return (d * q[..., 2:].contiguous().view(torch.int8).double()).view(w.shape)


def exact(case, seed):
    c = case
    x = _tokens(c, seed).double()
    if c["call"] == "step":
        return torch.stack([_moe64(c, seed, i % c["layers"], x[i]) for i in range(c["depth"])])
    if c["call"] == "layer":
        return _moe64(c, seed, 0, x)
    for i in range(c["depth"]):
        l = i % c["layers"]
        norm = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * _small(c, seed, l)["norm"].double()
        x = x + _moe64(c, seed, l, norm)
    return x
