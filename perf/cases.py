"""The work this backend is used for, as cases that can be timed and checked.

Three kinds of case, all through the Python binding's public entry points:

* ``layer``: one transformer layer's seven products (q, k, v, o of hidden x
  hidden, gate and up of ffn x hidden, down of hidden x ffn), captured once
  in a HIP graph and replayed, as a serving loop does. A single token goes
  through ``compute`` (which quantizes inside), a batch quantizes each input
  once and calls ``mul_mat`` for the products that share it.
* ``product``: one eager call, as a script or a test harness makes it:
  ``compute`` from fp32 activations, or ``mul_mat`` on activations that are
  quantized already.
* ``weights``: the device weight quantizers, as at model load.

Inputs are made on the GPU in plain torch; the formats are decoded again in
plain torch (64 bits) for the exact results.
"""
import importlib
import math

import torch

pkg = importlib.import_module("qgemm-perf-framework-ng_amd")

TYPES = {"q4_0": pkg.Q4_0, "q4_K": pkg.Q4_K, "iq2_xxs": pkg.IQ2_XXS}
QK = {"q4_0": 32, "q4_K": 256, "iq2_xxs": 256}
WEIGHT_BYTES = {"q4_0": 18, "q4_K": 144, "iq2_xxs": 66}
ACT_BYTES = {"q4_0": 34, "q4_K": 292, "iq2_xxs": 292}

# Macs of the largest listed product (2048 x 11008 x 4096): drawn cases stay below it.
MOST_MACS = 2048 * 11008 * 4096


def listed():
    return [
        # The smallest call a program makes: one token, one projection, eager.
        {"name": "call_q4_0_1", "kind": "product", "type": "q4_0", "m": 1, "n": 4096, "k": 4096, "entry": "compute"},
        # Single-token decode through a 4096-wide layer.
        {"name": "layer_q4_0_1", "kind": "layer", "type": "q4_0", "m": 1, "hidden": 4096, "ffn": 11008},
        # The same with the 2-bit format, whose table lookups cost more than its bytes.
        {"name": "layer_iq2_xxs_1", "kind": "layer", "type": "iq2_xxs", "m": 1, "hidden": 4096, "ffn": 14336},
        # A decode batch.
        {"name": "layer_iq2_xxs_16", "kind": "layer", "type": "iq2_xxs", "m": 16, "hidden": 4096, "ffn": 11008},
        # A larger, odd decode batch.
        {"name": "layer_q4_0_37", "kind": "layer", "type": "q4_0", "m": 37, "hidden": 4096, "ffn": 11008},
        # Decode with many users, or a short prompt.
        {"name": "layer_q4_K_100", "kind": "layer", "type": "q4_K", "m": 100, "hidden": 4096, "ffn": 11008},
        # A prompt of ordinary length through a small (1536-wide) model's layer.
        {"name": "layer_q4_0_480", "kind": "layer", "type": "q4_0", "m": 480, "hidden": 1536, "ffn": 4096},
        # The same in q4_K with a ragged prompt length.
        {"name": "layer_q4_K_333", "kind": "layer", "type": "q4_K", "m": 333, "hidden": 1536, "ffn": 4096},
        # A prompt of 512 tokens through one 4096-wide projection.
        {"name": "product_iq2_xxs_512", "kind": "product", "type": "iq2_xxs", "m": 512, "n": 4096, "k": 4096,
         "entry": "compute"},
        # A long prompt through the FFN's up projection: the largest.
        {"name": "product_q4_0_2048", "kind": "product", "type": "q4_0", "m": 2048, "n": 11008, "k": 4096,
         "entry": "mul_mat"},
        # A long prompt through the FFN's down projection, from fp32.
        {"name": "product_q4_K_2048", "kind": "product", "type": "q4_K", "m": 2048, "n": 4096, "k": 11008,
         "entry": "compute"},
        # Model load: one FFN matrix quantized on the device.
        {"name": "weights_q4_K", "kind": "weights", "type": "q4_K", "n": 11008, "k": 4096},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "product", "product", "weights"])
    qtype = rng.choice(["q4_0", "q4_K", "iq2_xxs"])
    if kind == "weights":
        return {"kind": kind, "type": rng.choice(["q4_0", "q4_K"]), "n": _log_int(rng, 64, 11008),
                "k": 256 * _log_int(rng, 1, 43)}
    if kind == "layer":
        hidden, ffn = 256 * _log_int(rng, 4, 20), 256 * _log_int(rng, 8, 56)
        m = _log_int(rng, 1, min(512, MOST_MACS // (4 * hidden * hidden + 3 * hidden * ffn)))
        return {"kind": kind, "type": qtype, "m": m, "hidden": hidden, "ffn": ffn}
    n = _log_int(rng, 32, 16384)
    k = 128 * _log_int(rng, 2, 112) if qtype == "q4_0" else 256 * _log_int(rng, 1, 56)
    m = _log_int(rng, 1, min(2048, MOST_MACS // (n * k)))
    return {"kind": kind, "type": qtype, "m": m, "n": n, "k": k, "entry": rng.choice(["compute", "mul_mat"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _activation(g, m, k):
    """Normal activations with a few large channels, as a layer's inputs have them."""
    x = torch.randn((m, k), generator=g, device="cuda")
    channels = torch.randint(0, k, (max(1, k // 512),), generator=g, device="cuda")
    x[:, channels] *= 8.0
    return x


def _half_bytes(d):
    """fp16 scales as a trailing axis of two bytes."""
    return d.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _weight_q4_0(g, n, k):
    """Normal weights in q4_0 blocks: the value of largest magnitude becomes -8."""
    x = torch.randn((n, k // 32, 32), generator=g, device="cuda")
    top = x.gather(2, x.abs().argmax(2, keepdim=True))
    d = top / -8.0
    q = (x / d + 8.5).to(torch.int32).clamp_(0, 15).to(torch.uint8)
    qs = q[..., :16] | (q[..., 16:] << 4)
    return torch.cat([_half_bytes(d.squeeze(2)), qs], 2).reshape(n, -1)


def _weight_q4_K(g, n, k):
    """Normal weights in q4_K super-blocks: a 6-bit scale and minimum per 32 values."""
    x = torch.randn((n, k // 256, 8, 32), generator=g, device="cuda")
    low = x.amin(3).clamp_(max=0.0)
    scale = (x.amax(3) - low) / 15.0
    d = (scale.amax(2) / 63.0).to(torch.float16)
    dmin = (-low.amin(2) / 63.0).to(torch.float16)
    s = (scale / d.float().unsqueeze(2)).round().clamp_(1, 63)
    m = (-low / dmin.float().unsqueeze(2).clamp_min(1e-7)).round().clamp_(0, 63)
    step, base = d.float().unsqueeze(2) * s, dmin.float().unsqueeze(2) * m
    q = ((x + base.unsqueeze(3)) / step.unsqueeze(3)).round().clamp_(0, 15).to(torch.uint8)
    qs = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(n, k // 256, 128)
    s, m = s.to(torch.uint8), m.to(torch.uint8)
    packed = torch.cat([s[..., :4] | ((s[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                        (s[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], 2)
    return torch.cat([_half_bytes(d), _half_bytes(dmin), packed, qs], 2).reshape(n, -1)


def _weight_iq2_xxs(g, n, k):
    """Random grid and sign indices and sub-block scales, block scales in [0.001, 0.01)."""
    d = torch.rand((n, k // 256), generator=g, device="cuda") * 0.009 + 0.001
    body = torch.randint(0, 256, (n, k // 256, 64), generator=g, device="cuda", dtype=torch.uint8)
    return torch.cat([_half_bytes(d), body], 2).reshape(n, -1)


_WEIGHT = {"q4_0": _weight_q4_0, "q4_K": _weight_q4_K, "iq2_xxs": _weight_iq2_xxs}


def _layer_shapes(case):
    """(input, n, k) of the seven products; inputs 0..3 feed q/k/v, o, gate/up and down."""
    h, f = case["hidden"], case["ffn"]
    return [(0, h, h), (0, h, h), (0, h, h), (1, h, h), (2, f, h), (2, f, h), (3, h, f)]


def _inputs(case, seed):
    """(activations, weights): the weights belong to the products in order."""
    g = _generator(seed)
    kind, m = case["kind"], case.get("m")
    if kind == "weights":
        return [torch.randn((case["n"], case["k"]), generator=g, device="cuda")], []
    if kind == "product":
        return [_activation(g, m, case["k"])], [_WEIGHT[case["type"]](g, case["n"], case["k"])]
    h, f = case["hidden"], case["ffn"]
    acts = [_activation(g, m, k) for k in (h, h, h, f)]
    return acts, [_WEIGHT[case["type"]](g, n, k) for _, n, k in _layer_shapes(case)]


def _layer_pass(s):
    t, m = s["type"], s["m"]
    if m == 1:
        for (i, n, _), w, out, ws in zip(s["shapes"], s["weights"], s["outs"], s["ws"]):
            pkg.compute(t, s["acts"][i], w, n, out=out, workspace=ws)
        return
    for x, q in zip(s["acts"], s["quantized"]):
        pkg.quantize_activation(t, x, out=q)
    for (i, n, k), w, out in zip(s["shapes"], s["weights"], s["outs"]):
        pkg.mul_mat(t, w, s["quantized"][i], m, n, k, out=out)


def prepare(case, seed):
    acts, weights = _inputs(case, seed)
    kind = case["kind"]
    s = {"kind": kind, "type": TYPES[case["type"]], "acts": acts, "weights": weights}
    if kind == "weights":
        return s
    pkg.device_check()
    m = s["m"] = case["m"]
    if kind == "product":
        n, k = s["n"], s["k"] = case["n"], case["k"]
        s["entry"] = case["entry"]
        s["out"] = torch.empty((m, n), device="cuda")
        if case["entry"] == "mul_mat":
            s["quantized"] = pkg.quantize_activation(s["type"], acts[0])
        else:
            s["ws"] = _workspace(case["type"], m, k)
        return s
    s["shapes"] = _layer_shapes(case)
    s["outs"] = [torch.empty((m, n), device="cuda") for _, n, _ in s["shapes"]]
    if m == 1:
        s["ws"] = [_workspace(case["type"], m, k) for _, _, k in s["shapes"]]
    else:
        s["quantized"] = [_workspace(case["type"], m, x.shape[1]) for x in acts]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _layer_pass(s)
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"], stream=stream):
        _layer_pass(s)
    return s


def _workspace(name, m, k):
    return torch.empty((m, k // QK[name] * ACT_BYTES[name]), dtype=torch.uint8, device="cuda")


def run(state):
    kind = state["kind"]
    if kind == "layer":
        state["graph"].replay()
        return state["outs"]
    if kind == "weights":
        return pkg.quantize_weights_gpu(state["type"], state["acts"][0])
    if state["entry"] == "compute":
        return pkg.compute(state["type"], state["acts"][0], state["weights"][0], state["n"], out=state["out"],
                           workspace=state["ws"])
    return pkg.mul_mat(state["type"], state["weights"][0], state["quantized"], state["m"], state["n"], state["k"],
                       out=state["out"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what it must return
# ---------------------------------------------------------------------------

def work(case):
    t, kind = case["type"], case["kind"]
    if kind == "weights":
        values = case["n"] * case["k"]
        return {"bytes": values * 4 + values // QK[t] * WEIGHT_BYTES[t], "flops": 0}
    m = case["m"]
    shapes = [(0, case["n"], case["k"])] if kind == "product" else _layer_shapes(case)
    inputs = {i: k for i, _, k in shapes}
    if kind == "product" and case["entry"] == "mul_mat":
        read = m * (case["k"] // QK[t]) * ACT_BYTES[t]
    else:
        read = sum(m * k * 4 for k in inputs.values())
    read += sum(n * (k // QK[t]) * WEIGHT_BYTES[t] for _, n, k in shapes)
    return {"bytes": read + sum(m * n * 4 for _, n, _ in shapes), "flops": sum(2 * m * n * k for _, n, k in shapes)}


def tolerance(case):
    if case["kind"] == "weights":
        return "exact"
    # fp32 sums over k / 32 or k / 256 exact integer block sums: measured up to
    # 2.1e-7 and 1.8e-6 from 64 bits (2048 x 11008 x 4096)
    return {"rel": 1e-6, "max": 8e-6}


_GRID = (
    0x0000, 0x0002, 0x0005, 0x0008, 0x000a, 0x0011, 0x0014, 0x0020, 0x0022, 0x0028, 0x002a, 0x0041, 0x0044, 0x0050,
    0x0058, 0x0061, 0x0064, 0x0080, 0x0082, 0x008a, 0x00a2, 0x0101, 0x0104, 0x0110, 0x0115, 0x0140, 0x0184, 0x0198,
    0x0200, 0x0202, 0x0222, 0x0282, 0x0401, 0x0404, 0x0410, 0x0421, 0x0424, 0x0440, 0x0442, 0x0448, 0x0460, 0x0481,
    0x0484, 0x0490, 0x04a4, 0x0500, 0x0502, 0x0508, 0x0520, 0x0546, 0x0569, 0x0580, 0x0591, 0x0609, 0x0610, 0x0640,
    0x0684, 0x06a4, 0x0800, 0x0805, 0x0808, 0x0814, 0x0828, 0x0841, 0x0844, 0x0850, 0x0852, 0x0888, 0x0904, 0x0940,
    0x0a02, 0x0a14, 0x1001, 0x1004, 0x1010, 0x1021, 0x1040, 0x1060, 0x1084, 0x1090, 0x1095, 0x1100, 0x1108, 0x1120,
    0x1150, 0x115a, 0x1180, 0x1224, 0x1245, 0x1400, 0x1408, 0x1420, 0x1425, 0x1449, 0x1480, 0x1518, 0x1562, 0x1600,
    0x1616, 0x1801, 0x1804, 0x1810, 0x1840, 0x1881, 0x1900, 0x1905, 0x19a0, 0x1a51, 0x2000, 0x2002, 0x200a, 0x2044,
    0x2061, 0x2080, 0x2082, 0x2129, 0x2148, 0x2200, 0x2202, 0x2401, 0x2404, 0x2410, 0x2440, 0x2456, 0x2500, 0x2541,
    0x2564, 0x2690, 0x2808, 0x2820, 0x2894, 0x2a44, 0x4001, 0x4004, 0x4010, 0x4018, 0x4021, 0x4024, 0x4040, 0x4048,
    0x4056, 0x4060, 0x4081, 0x4084, 0x4090, 0x4100, 0x4120, 0x4161, 0x4180, 0x4185, 0x4201, 0x4210, 0x4248, 0x4256,
    0x4268, 0x4400, 0x4408, 0x4420, 0x4480, 0x4499, 0x4512, 0x4524, 0x4600, 0x4801, 0x4804, 0x4810, 0x4840, 0x4845,
    0x4900, 0x4958, 0x4961, 0x4982, 0x4a45, 0x4a90, 0x5000, 0x5008, 0x5011, 0x5019, 0x5020, 0x5080, 0x5088, 0x5104,
    0x5142, 0x51a4, 0x5291, 0x5490, 0x5492, 0x550a, 0x5601, 0x5654, 0x5800, 0x5811, 0x5819, 0x5864, 0x5940, 0x5a08,
    0x6004, 0x6010, 0x6040, 0x6068, 0x6100, 0x6155, 0x6218, 0x6260, 0x6400, 0x6405, 0x6510, 0x6512, 0x6584, 0x6842,
    0x8000, 0x8002, 0x800a, 0x8041, 0x8082, 0x8104, 0x8118, 0x8140, 0x8211, 0x8401, 0x8404, 0x8410, 0x8415, 0x8440,
    0x8460, 0x8500, 0x8546, 0x8594, 0x8609, 0x8640, 0x8660, 0x8802, 0x8904, 0x8a11, 0x9004, 0x9010, 0x9024, 0x9040,
    0x90a1, 0x9116, 0x9180, 0x9245, 0x9400, 0x9422, 0x9444, 0x9551, 0x9881, 0x9920, 0xa002, 0xa050, 0xa085, 0xa109,
    0xa200, 0xa418, 0xa850, 0xa904)


def _half(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).squeeze(-1).double()


def _decode(name, w, k):
    """Weight blocks (n, bytes) -> float64 (n, k)."""
    n = w.shape[0]
    b = w.view(n, k // QK[name], WEIGHT_BYTES[name])
    d = _half(b, 0)
    if name == "q4_0":
        qs = b[..., 2:]
        q = torch.cat([qs & 15, qs >> 4], 2).double() - 8.0
        return (q * d.unsqueeze(2)).reshape(n, k)
    if name == "q4_K":
        dmin, p, qs = _half(b, 2), b[..., 4:16], b[..., 16:].reshape(n, -1, 4, 32)
        s = torch.cat([p[..., :4] & 63, (p[..., 8:] & 15) | ((p[..., :4] >> 6) << 4)], 2).double()
        m = torch.cat([p[..., 4:8] & 63, (p[..., 8:] >> 4) | ((p[..., 4:8] >> 6) << 4)], 2).double()
        q = torch.stack([qs & 15, qs >> 4], 3).reshape(n, -1, 8, 32).double()
        return (q * (s * d.unsqueeze(2)).unsqueeze(3) - (m * dmin.unsqueeze(2)).unsqueeze(3)).reshape(n, k)
    sub = b[..., 2:].reshape(n, -1, 8, 8).to(torch.int64)
    codes = torch.tensor(_GRID, device=w.device)
    lanes = torch.arange(8, device=w.device)
    magnitude = torch.tensor([8.0, 25.0, 43.0, 0.0], dtype=torch.float64, device=w.device)
    values = magnitude[(codes.unsqueeze(1) >> (2 * lanes)) & 3][sub[..., :4]]  # (n, blocks, 8, 4, 8)
    word = sub[..., 4] | (sub[..., 5] << 8) | (sub[..., 6] << 16) | (sub[..., 7] << 24)
    index = (word.unsqueeze(-1) >> (7 * torch.arange(4, device=w.device))) & 127
    bits = (index.unsqueeze(-1) >> lanes) & 1
    bits[..., 7] = bits.sum(-1) & 1
    scale = 0.125 * d.unsqueeze(2) * (2 * (word >> 28) + 1).double()
    return (values * (1 - 2 * bits) * scale.unsqueeze(-1).unsqueeze(-1)).reshape(n, k)


def _quantized(name, x):
    """The values q8_0 (blocks of 32, fp16 scale) or q8_K (256, fp32 scale) gives x, in 64 bits."""
    block = QK[name]
    v = x.reshape(x.shape[0], -1, block)
    d = v.abs().amax(2, keepdim=True) / torch.full((), 127.0, device=x.device)
    inverse = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    t = (v * inverse).double()
    q = torch.sign(t) * torch.floor(t.abs() + 0.5)
    d = d.to(torch.float16).double() if name == "q4_0" else d.double()
    return (q * d).reshape(x.shape)


def exact(case, seed):
    if case["kind"] == "weights":
        return None
    acts, weights = _inputs(case, seed)
    name = case["type"]
    acts = [_quantized(name, x) for x in acts]
    if case["kind"] == "product":
        return acts[0] @ _decode(name, weights[0], case["k"]).T
    return [acts[i] @ _decode(name, w, k).T for (i, _, k), w in zip(_layer_shapes(case), weights)]
