"""What a user of the library has it do, as cases that can be timed: the quantized projections of a
decoding or prefilling decoder, dense and mixture-of-experts, through the public Python entry points.

A case is a dict of plain values; `prepare` makes what a program holds before the call (resident
weights, activations, output buffers), `run` is one pass.  The families:

  qkv      one token's q/k/v projections in one call: the smallest work, launch latency counts
  layers   one token through whole decoder layers' projections (q/k/v, o, SwiGLU FFN)
  head     the output projection through the host-buffer seam: the sampler wants the logits on the host
  batch    a batch of decoding sequences (2 .. 40 rows): the weights' bytes count
  prefill  a prompt's rows through one matrix, or gate and up over one batch
  moe      router, expert FFN and combine of a mixture-of-experts layer, one token or a prompt
"""
import math

import torch

import frink_amd as fa

DEVICE = "cuda:0"
KINDS = {"Q4_K": fa.Q4_K, "Q5_K": fa.Q5_K, "Q6_K": fa.Q6_K, "Q8_0": fa.Q8_0, "MXFP4": fa.MXFP4}


def listed():
    return [
        # decode of one token, Llama-3-8B shapes in a Q4_K_M file: the attention's three projections alone ...
        {"name": "decode_qkv", "family": "qkv", "kind": "Q4_K", "hidden": 4096, "kv": 1024},
        # ... and two whole layers of it (down projections in Q6_K)
        {"name": "decode_layers", "family": "layers", "kind": "Q4_K", "down": "Q6_K", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "layers": 2},
        # the output head of a 32000-token vocabulary, from host buffers to host buffers
        {"name": "head_from_host", "family": "head", "kind": "Q6_K", "rows": 32000, "cols": 4096},
        # eight sequences decoding together: gate or up
        {"name": "batch_8", "family": "batch", "kind": "Q4_K", "batch": 8, "rows": 14336, "cols": 4096},
        # an odd number of sequences, Llama-2-7B's down projection (43 blocks a row)
        {"name": "batch_13_ragged", "family": "batch", "kind": "Q6_K", "batch": 13, "rows": 4096, "cols": 11008},
        # a 512-token prompt chunk: gate and up over one quantization, then the down projection
        {"name": "prefill_gate_up", "family": "prefill", "kind": "Q4_K", "batch": 512, "rows": 14336, "cols": 4096, "pair": True},
        {"name": "prefill_down", "family": "prefill", "kind": "Q6_K", "batch": 512, "rows": 4096, "cols": 14336, "pair": False},
        # a short prompt that fills no tile, the kind a Q5_K_M file holds most of
        {"name": "prefill_ragged", "family": "prefill", "kind": "Q5_K", "batch": 197, "rows": 11008, "cols": 4096, "pair": False},
        # a long prompt through a Q8_0 model's down projection
        {"name": "prefill_long", "family": "prefill", "kind": "Q8_0", "batch": 2048, "rows": 4096, "cols": 14336, "pair": False},
        # a layer of 128 experts, top-8, in a Q4_K_M file: one token, and a prompt chunk
        {"name": "moe_decode", "family": "moe", "kind": "Q4_K", "down": "Q6_K", "tokens": 1, "experts": 128, "top_k": 8,
         "hidden": 2048, "ffn": 768},
        {"name": "moe_prefill", "family": "moe", "kind": "Q4_K", "down": "Q6_K", "tokens": 512, "experts": 128, "top_k": 8,
         "hidden": 2048, "ffn": 768},
        # a layer of 32 MXFP4 experts, top-4 (gpt-oss-20b's shape), a prompt chunk
        {"name": "moe_mxfp4", "family": "moe", "kind": "MXFP4", "down": "MXFP4", "tokens": 512, "experts": 32, "top_k": 4,
         "hidden": 2880, "ffn": 2880},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    family = rng.choice(("qkv", "layers", "head", "batch", "prefill", "prefill", "moe", "moe"))

    def width(low, high):
        return 256 * rng.randint(low // 256, high // 256)

    if family == "qkv":
        hidden = width(2048, 8192)
        return {"family": family, "kind": rng.choice(("Q4_K", "Q5_K", "Q6_K", "Q8_0")), "hidden": hidden,
                "kv": hidden // rng.choice((1, 4, 8))}
    if family == "layers":
        kind, down = rng.choice((("Q4_K", "Q4_K"), ("Q4_K", "Q6_K"), ("Q5_K", "Q6_K"), ("Q8_0", "Q8_0")))
        hidden = width(2048, 4096)
        return {"family": family, "kind": kind, "down": down, "hidden": hidden, "kv": hidden // rng.choice((1, 4, 8)),
                "ffn": width(5632, 14336), "layers": 1 if kind == "Q8_0" else rng.randint(1, 2)}
    if family == "head":
        return {"family": family, "kind": rng.choice(("Q6_K", "Q8_0")), "rows": _log_int(rng, 8000, 40000), "cols": width(2048, 5120)}
    if family == "batch":
        return {"family": family, "kind": rng.choice(("Q4_K", "Q5_K", "Q6_K", "Q8_0")), "batch": _log_int(rng, 2, 40),
                "rows": _log_int(rng, 1024, 14336), "cols": width(2048, 14336)}
    if family == "prefill":
        kind = rng.choice(("Q4_K", "Q5_K", "Q6_K", "Q8_0"))
        cols, rows = width(2048, 14336), _log_int(rng, 1024, 14336)
        most = min(2048, (2048 * 4096 * 14336) // (2 * rows * cols))
        return {"family": family, "kind": kind, "batch": _log_int(rng, 48, most), "rows": rows, "cols": cols,
                "pair": kind in ("Q4_K", "Q5_K") and rng.random() < 0.5}
    if rng.random() < 0.33:
        return {"family": family, "kind": "MXFP4", "down": "MXFP4", "tokens": _log_int(rng, 1, 768), "experts": rng.choice((8, 16, 32)),
                "top_k": rng.choice((2, 4)), "hidden": 32 * rng.randint(32, 90), "ffn": 32 * rng.randint(32, 90)}
    experts, hidden = rng.choice((16, 60, 64, 128)), width(1024, 2560)
    widest = 256 * min(6, 128 * 2048 * 768 // (experts * hidden * 256))
    return {"family": family, "kind": "Q4_K", "down": rng.choice(("Q4_K", "Q6_K")), "tokens": _log_int(rng, 1, 1024),
            "experts": experts, "top_k": rng.choice((2, 4, 6, 8)), "hidden": hidden, "ffn": width(512, widest)}


# ---- inputs ----

def _codes(gen, shape, mid, spread, top):
    """Quantization codes 0 .. top as encoded normal weights have them."""
    z = torch.randn(shape, generator=gen, device=DEVICE)
    return z.mul_(spread).add_(mid).round_().clamp_(0, top).to(torch.uint8)


def _f16(gen, n, low, high):
    v = torch.rand(n, 1, generator=gen, device=DEVICE) * (high - low) + low
    return v.to(torch.float16).view(torch.uint8)


def _six_bit_scales(gen, n):
    """The 12 packed bytes of a K-quant super-block's eight 6-bit scales and eight 6-bit mins; the largest of each is
    near the top of the range, the others not far below."""
    s = torch.randint(36, 64, (n, 16), generator=gen, device=DEVICE, dtype=torch.uint8)
    sc, m = s[:, :8], s[:, 8:]
    return torch.cat((sc[:, :4] | (sc[:, 4:] >> 4 << 6), m[:, :4] | (m[:, 4:] >> 4 << 6),
                      (sc[:, 4:] & 15) | (m[:, 4:] & 15) << 4), 1)


def _blocks(kind, rows, cols, gen):
    """GGUF block bytes of a rows x cols matrix of weights of about N(0, 0.02): the codes, scales and offsets that the
    kind's encoder gives such weights, drawn directly."""
    n = rows * cols // fa.BLOCK[KINDS[kind]][1]
    if kind == "Q4_K":
        c = _codes(gen, (n, 4, 2, 32), 7.5, 3.6, 15)
        parts = (_f16(gen, n, 0.8e-4, 1.2e-4), _f16(gen, n, 0.7e-3, 0.9e-3), _six_bit_scales(gen, n),
                 (c[:, :, 0] | c[:, :, 1] << 4).reshape(n, 128))
    elif kind == "Q5_K":
        c = _codes(gen, (n, 8, 32), 15.5, 7.4, 31)
        high = torch.zeros((n, 32), dtype=torch.uint8, device=DEVICE)
        for j in range(8):
            high |= c[:, j] >> 4 << j
        low = (c & 15).view(n, 4, 2, 32)
        parts = (_f16(gen, n, 0.4e-4, 0.6e-4), _f16(gen, n, 0.7e-3, 0.9e-3), _six_bit_scales(gen, n), high,
                 (low[:, :, 0] | low[:, :, 1] << 4).reshape(n, 128))
    elif kind == "Q6_K":
        c = _codes(gen, (n, 2, 4, 32), 32.0, 15.0, 63)
        low, high = c & 15, c >> 4
        scale = torch.randint(70, 128, (n, 16), generator=gen, device=DEVICE, dtype=torch.int16)
        sign = torch.randint(0, 2, (n, 16), generator=gen, device=DEVICE, dtype=torch.int16) * 2 - 1
        parts = ((low[:, :, :2] | low[:, :, 2:] << 4).reshape(n, 128),
                 (high[:, :, 0] | high[:, :, 1] << 2 | high[:, :, 2] << 4 | high[:, :, 3] << 6).reshape(n, 64),
                 (scale * sign).to(torch.int8).view(torch.uint8), _f16(gen, n, 1.0e-5, 1.6e-5))
    elif kind == "Q8_0":
        q = torch.randn((n, 32), generator=gen, device=DEVICE).mul_(58.0).round_().clamp_(-127, 127).to(torch.int8)
        parts = (_f16(gen, n, 3e-4, 4e-4), q.view(torch.uint8))
    else:  # MXFP4: an E8M0 scale, then 32 E2M1 codes (a sign over a magnitude code)
        z = torch.randn((n, 2, 16), generator=gen, device=DEVICE)
        c = (z.abs() * 2.7).round_().clamp_(0, 7).to(torch.uint8) | (z < 0).to(torch.uint8) << 3
        e = torch.randint(118, 122, (n, 1), generator=gen, device=DEVICE, dtype=torch.uint8)
        parts = (e, c[:, 0] | c[:, 1] << 4)
    return torch.cat(parts, 1).reshape(-1)


def _weights(kind, rows, cols, gen):
    return fa.Weights.from_device(KINDS[kind], _blocks(kind, rows, cols, gen), rows, cols)


def _activations(gen, rows, cols):
    """Normalised hidden states: N(0, 1), a few channels eight times as large."""
    x = torch.randn((rows, cols), generator=gen, device=DEVICE)
    x[:, torch.randint(0, cols, (max(1, cols // 512),), generator=gen, device=DEVICE)] *= 8.0
    return x


def _out(*shape):
    return torch.empty(shape, dtype=torch.float32, device=DEVICE)


def prepare(case, seed):
    gen = torch.Generator(DEVICE)
    gen.manual_seed(seed)
    family = case["family"]
    s = {"family": family}
    if family == "qkv":
        h, kv = case["hidden"], case["kv"]
        s["w"] = [_weights(case["kind"], r, h, gen) for r in (h, kv, kv)]
        s["x"] = _activations(gen, 1, h)[0]
        s["y"] = [_out(r) for r in (h, kv, kv)]
    elif family == "layers":
        h, kv, ffn, kind = case["hidden"], case["kv"], case["ffn"], case["kind"]
        s["layers"] = []
        for _ in range(case["layers"]):
            s["layers"].append({
                "qkv": [_weights(kind, r, h, gen) for r in (h, kv, kv)], "o": _weights(kind, h, h, gen),
                "gate": _weights(kind, ffn, h, gen), "up": _weights(kind, ffn, h, gen), "down": _weights(case["down"], h, ffn, gen),
                # the attention and the norms between the projections are not the library's: their results come as inputs
                "x_attn": _activations(gen, 1, h)[0], "x_o": _activations(gen, 1, h)[0], "x_ffn": _activations(gen, 1, h)[0],
                "y_qkv": [_out(r) for r in (h, kv, kv)], "y_o": _out(h), "y_ffn": _out(h)})
    elif family == "head":
        s["kind"], s["rows"] = KINDS[case["kind"]], case["rows"]
        s["data"] = _blocks(case["kind"], case["rows"], case["cols"], gen).cpu().numpy()
        s["row_bytes"] = s["data"].size // case["rows"]
        s["resident"] = fa.Weights.from_host(s["kind"], s["data"], case["rows"], case["cols"])  # uploaded once, when the model loads
        s["x"] = _activations(gen, 1, case["cols"])[0].cpu().numpy()
    elif family in ("batch", "prefill"):
        rows, cols, m = case["rows"], case["cols"], case["batch"]
        s["w"] = [_weights(case["kind"], rows, cols, gen) for _ in range(2 if case.get("pair") else 1)]
        s["x"] = _activations(gen, m, cols)
        s["y"] = [_out(m, rows) for _ in s["w"]]
    else:
        e, h, ffn, t = case["experts"], case["hidden"], case["ffn"], case["tokens"]
        s["gate"], s["up"] = _weights(case["kind"], e * ffn, h, gen), _weights(case["kind"], e * ffn, h, gen)
        s["down"] = _weights(case["down"], e * h, ffn, gen)
        s["x"] = _activations(gen, t, h)
        s["logits"] = torch.randn((t, e), generator=gen, device=DEVICE)
        s["experts"], s["top_k"], s["y"] = e, case["top_k"], _out(t, h)
    return s


def run(s):
    family = s["family"]
    if family == "qkv":
        return fa.gemv_multi(s["w"], s["x"], outs=s["y"])
    if family == "layers":
        for l in s["layers"]:
            fa.gemv_multi(l["qkv"], l["x_attn"], outs=l["y_qkv"])
            l["o"].gemv(l["x_o"], out=l["y_o"])
            fa.ffn_swiglu(l["gate"], l["up"], l["down"], l["x_ffn"], out=l["y_ffn"])
        return [l["y_qkv"] + [l["y_o"], l["y_ffn"]] for l in s["layers"]]
    if family == "head":
        return fa.launch_matvec(s["kind"], s["data"], s["x"], s["rows"], s["row_bytes"])
    if family in ("batch", "prefill"):
        if len(s["w"]) == 2:
            return fa.gemm_pair(s["w"][0], s["w"][1], s["x"], outs=s["y"])
        return s["w"][0].gemm(s["x"], out=s["y"][0])
    ids, weights = fa.route_top_k_softmax(s["logits"], s["top_k"], True)
    return fa.moe_ffn(s["gate"], s["up"], s["down"], s["experts"], s["x"], ids, weights, out=s["y"]), ids, weights


# ---- what a pass cannot do without ----

def _matrix(kind, rows, cols):
    size, elems = fa.BLOCK[KINDS[kind]]
    return rows * (cols // elems) * size


def work(case):
    family = case["family"]
    if family == "qkv":
        h, out = case["hidden"], case["hidden"] + 2 * case["kv"]
        return {"bytes": _matrix(case["kind"], out, h) + 4 * (h + out), "flops": 2 * out * h}
    if family == "layers":
        h, kv, ffn = case["hidden"], case["kv"], case["ffn"]
        rows = h + 2 * kv + h + 2 * ffn
        one = _matrix(case["kind"], rows, h) + _matrix(case["down"], h, ffn) + 4 * (3 * h + h + 2 * kv + h + h)
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 2 * (rows * h + h * ffn)}
    if family == "head":
        return {"bytes": _matrix(case["kind"], case["rows"], case["cols"]) + 4 * (case["rows"] + case["cols"]),
                "flops": 2 * case["rows"] * case["cols"]}
    if family in ("batch", "prefill"):
        n, m, rows, cols = 2 if case.get("pair") else 1, case["batch"], case["rows"], case["cols"]
        return {"bytes": n * _matrix(case["kind"], rows, cols) + 4 * m * (cols + n * rows), "flops": n * 2 * m * rows * cols}
    e, k, h, ffn, t = case["experts"], case["top_k"], case["hidden"], case["ffn"], case["tokens"]
    visited = e * (1.0 - (1.0 - k / e) ** t)  # the experts that independent routings of t tokens are expected to reach
    expert = 2 * _matrix(case["kind"], ffn, h) + _matrix(case["down"], h, ffn)
    return {"bytes": visited * expert + 4 * t * (2 * h + e + 2 * k), "flops": 2 * t * k * 3 * h * ffn}


def tolerance(case):
    """One projection multiplies exactly quantized activations, so two correct implementations differ by the order of
    their f32 sums: against 64-bit sums of the same products 0.7e-7 to 1.8e-7 was seen for the K-quants and up to 3.8e-7
    for Q8_0, which adds 448 scaled blocks of 14336 columns.  Where a result is quantized again (the SwiGLU in front of a
    down projection), a last-bit difference now and then moves one value to the next level: up to 1.6e-4 of an output row
    was seen for one token of a mixture-of-experts layer, whose intermediate is short, and less for long ones."""
    if case["family"] == "moe":
        return {"rel": 6e-4}
    if case["family"] == "layers":
        return {"rel": 4e-4}
    return {"rel": 1.5e-6}
