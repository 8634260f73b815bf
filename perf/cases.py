"""Performance cases: the calls a user of this package makes, over the sizes they are made at.

Training side: the bulk nearest-neighbour quantizer under both score rules, the per-matrix requantize of a
training step, the fused optimiser step with its requantize.  Packing side: the pack-time quantizer, the
18-bit codec with the fp16 reconstruction.  Inference side: one packed linear at one token and at 64, a
decoder block over a whole prompt, the INT8 head over a prompt, and KV-cached generation of the whole
model at batch 1 and 16.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same ranges; ``prepare`` makes what a
program holds before the call, ``run`` is one pass through the public entry points, ``exact`` the float64
values of the outputs that have one (plain torch / numpy, the codebook built here).
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from pollux_amd import castor, optim, pack
from pollux_amd.model import GraphDecoder, KVCache, PackedBlock, PackedPolluxModel, PolluxConfig
from pollux_amd.packed import PackedH24Linear, PackedInt8Linear, dequantize_h24

DEV = "cuda"
CODES = 196_561
SQRT2 = math.sqrt(2.0)


def listed() -> list[dict]:
    return [
        # re-quantizing a 403M-parameter model's weights in one call (the bulk throughput workload)
        {"name": "quantize_bulk", "kind": "quantize", "mode": "bf16", "rows": 209_715, "cols": 1920},
        # the same search under fp32 scores (the semantics of the GPU training path), one up-projection
        {"name": "quantize_fp32_scores", "kind": "quantize", "mode": "fp32", "rows": 7680, "cols": 1920},
        # one small training matrix, as a step requantizes it: launches and latency count
        {"name": "requantize_1152", "kind": "requantize", "rows": 1152, "cols": 1152},
        # an optimiser step of one d=1920 layer's six matrices, with their requantize and packed codes
        {"name": "train_step_1920", "kind": "train", "d": 1920},
        # packing one trained up-projection for a checkpoint
        {"name": "pack_layer_7680x1920", "kind": "pack", "rows": 7680, "cols": 1920},
        # writing, re-reading and expanding a bulk of codes: encode, decode, fp16 weights
        {"name": "codec_bulk", "kind": "codec", "rows": 209_712, "cols": 1920},
        # the smallest inference call: one token through one packed linear
        {"name": "linear_1_token", "kind": "linear", "out": 7680, "in": 1920, "tokens": 1, "dtype": "bf16"},
        # a small batch or short prompt through one packed linear
        {"name": "linear_64_tokens", "kind": "linear", "out": 1920, "in": 7680, "tokens": 64, "dtype": "bf16"},
        # a decoder block over a prompt of the model's full context
        {"name": "block_prompt_1024", "kind": "block", "heads": 80, "batch": 1, "tokens": 1024},
        # logits of every position of a prompt (scoring a text)
        {"name": "head_256_tokens", "kind": "head", "vocab": 50_688, "d": 1920, "tokens": 256},
        # generation by one user: a prompt, then tokens one by one
        {"name": "generate_batch_1", "kind": "generate", "layers": 18, "heads": 80, "vocab": 50_688, "batch": 1,
         "prompt": 64, "new": 16},
        # generation for 16 users at once, ragged prompt length
        {"name": "generate_batch_16", "kind": "generate", "layers": 18, "heads": 80, "vocab": 50_688, "batch": 16,
         "prompt": 57, "new": 16},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["quantize", "requantize", "train", "pack", "codec", "linear", "linear", "block", "head",
                       "generate"])
    c: dict = {"kind": kind}
    if kind == "quantize":
        c["mode"] = rng.choice(["bf16", "bf16", "fp32"])
        c["rows"], c["cols"] = _log(rng, 1, 200_000 if c["mode"] == "bf16" else 9000), 24 * rng.randint(1, 80)
    elif kind in ("requantize", "pack"):
        c["rows"], c["cols"] = _log(rng, 8, 7680), 24 * _log(rng, 1, 320)
    elif kind == "train":
        c["d"] = 24 * rng.randint(2, 80)
    elif kind == "codec":
        c["rows"], c["cols"] = _log(rng, 1, 200_000), 24 * rng.randint(1, 80)
    elif kind == "linear":
        c["out"], c["in"] = _log(rng, 24, 7680), 24 * _log(rng, 4, 320)
        c["tokens"], c["dtype"] = _log(rng, 1, 1024), rng.choice(["bf16", "fp32"])
    elif kind == "block":
        c["heads"], c["batch"] = rng.randint(4, 80), rng.randint(1, 4)
        c["tokens"] = _log(rng, 2, 1024 // c["batch"])
    elif kind == "head":
        c["vocab"], c["d"], c["tokens"] = 24 * _log(rng, 20, 2112), 48 * rng.randint(4, 40), _log(rng, 1, 256)
    else:
        c["layers"], c["heads"], c["vocab"] = rng.randint(1, 18), rng.randint(8, 80), 24 * _log(rng, 40, 2112)
        c["batch"], c["prompt"], c["new"] = rng.randint(1, 16), _log(rng, 2, 64), rng.randint(2, 16)
    return c


# ---------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _weight(rows: int, cols: int, g: torch.Generator) -> torch.Tensor:
    return torch.randn(rows, cols, generator=g, device=DEV) * 0.02


def _indices(n: int, g: torch.Generator) -> torch.Tensor:
    return torch.randint(0, CODES, (n,), generator=g, device=DEV, dtype=torch.int32)


def _sigma16(rows: int, g: torch.Generator) -> torch.Tensor:
    return (torch.rand(rows, generator=g, device=DEV) * 0.045 + 0.005).half()


def _fill_linear(layer: PackedH24Linear, g: torch.Generator) -> torch.Tensor:
    """Random codes and row scales into a packed layer; returns the codes."""
    idx = _indices(layer.num_atoms, g)
    layer.packed_weights.copy_(castor.pack_indices(idx))
    layer.sigma_rows.copy_(_sigma16(layer.out_features, g))
    return idx


def _fill_int8(layer, rows: int, cols: int, g: torch.Generator) -> None:
    layer.weight_int8.copy_(torch.randint(-127, 128, (rows, cols), generator=g, device=DEV, dtype=torch.int8))
    layer.mu_rows.copy_((torch.rand(rows, generator=g, device=DEV) * 0.1 + 0.01).half())


def _norm_weight(n: int, g: torch.Generator) -> torch.Tensor:
    return 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _fill_block(block: PackedBlock, g: torch.Generator) -> list[torch.Tensor]:
    with torch.no_grad():
        for ln in (block.ln1, block.ln2, block.attn.q_ln, block.attn.k_ln):
            ln.weight.copy_(_norm_weight(ln.weight.numel(), g))
    a, m = block.attn, block.mlp
    return [_fill_linear(l, g) for l in (a.q_proj, a.k_proj, a.v_proj, a.o_proj, m.fc1, m.fc2)]


def _config(case: dict) -> PolluxConfig:
    return PolluxConfig(n_layers=case.get("layers", 1), n_heads=case["heads"], n_embd=24 * case["heads"],
                        vocab_size=case.get("vocab", 96), tokenizer_vocab_size=case.get("vocab", 96))


def _train_shapes(d: int) -> list[tuple[int, int]]:
    return [(d, d)] * 4 + [(4 * d, d), (d, 4 * d)]


# Late in the cool-down: the weights hardly move over many passes on one state, so every pass sees them as
# training leaves them.
HEAT, STEP = 2e-4, 10_000


def prepare(case: dict, seed: int) -> dict:
    g, kind = _gen(seed), case["kind"]
    s: dict = {"case": case}
    if kind == "quantize":
        n = case["rows"] * case["cols"] // 24
        if case["mode"] == "fp32":  # lattice coordinates of normalised weights
            s["x"] = torch.randn(n, 24, generator=g, device=DEV) * SQRT2
        else:  # directions uniform on the sphere, radius U(0, 2) * sqrt(32)
            x = torch.randn(n, 24, generator=g, device=DEV)
            r = torch.rand(n, 1, generator=g, device=DEV) * (2.0 * math.sqrt(32.0))
            s["x"] = x.mul_(r / x.norm(dim=1, keepdim=True))
    elif kind in ("requantize", "pack"):
        s["w"] = _weight(case["rows"], case["cols"], g)
    elif kind == "train":
        s["params"] = []
        for rows, cols in _train_shapes(case["d"]):
            lat = _weight(rows, cols, g)
            grad = torch.randn(rows, cols, generator=g, device=DEV) * 1e-3
            m = torch.randn(rows, cols, generator=g, device=DEV) * 3e-4
            v = (torch.randn(rows, cols, generator=g, device=DEV) * 1e-3).square_().add_(1e-7)
            s["params"].append((lat.clone(), grad, m, v, lat))
        s["heat"] = torch.tensor(HEAT, device=DEV)
        s["step"] = torch.tensor(STEP, device=DEV)
        s["inertia"] = optim.width_inertia(case["d"])
    elif kind == "codec":
        s["idx"] = _indices(case["rows"] * case["cols"] // 24, g)
        s["sigma"] = _sigma16(case["rows"], g)
    elif kind == "linear":
        with torch.device(DEV):
            s["layer"] = PackedH24Linear(case["in"], case["out"])
        s["idx"] = _fill_linear(s["layer"], g)
        x = torch.randn(case["tokens"], case["in"], generator=g, device=DEV)
        s["x"] = x.bfloat16() if case["dtype"] == "bf16" else x
    elif kind == "block":
        cfg = _config(case)
        with torch.device(DEV):
            s["block"] = PackedBlock(cfg).eval()
        s["idx"] = _fill_block(s["block"], g)
        shape = (case["batch"], case["heads"], case["tokens"], 24)
        s["cache"] = KVCache([torch.zeros(shape, device=DEV)], [torch.zeros(shape, device=DEV)])
        s["x"] = torch.randn(case["batch"], case["tokens"], 24 * case["heads"], generator=g, device=DEV)
    elif kind == "head":
        with torch.device(DEV):
            s["layer"] = PackedInt8Linear(case["d"], case["vocab"])
        _fill_int8(s["layer"], case["vocab"], case["d"], g)
        s["norm"] = _norm_weight(case["d"], g)
        s["x"] = torch.randn(1, case["tokens"], case["d"], generator=g, device=DEV)
    else:
        cfg = _config(case)
        with torch.device("meta"):
            model = PackedPolluxModel(cfg)
        s["model"] = model = model.to_empty(device=DEV).eval()
        with torch.no_grad():
            model.pos_emb.weight.copy_(torch.randn(model.pos_emb.weight.shape, generator=g, device=DEV) * 0.02)
            model.ln_f.weight.copy_(_norm_weight(24 * case["heads"], g))
        for part in (model.tok_emb, model.head):
            _fill_int8(part, case["vocab"], 24 * case["heads"], g)
        s["idx"] = [_fill_block(b, g) for b in model.blocks]
        ids = torch.randint(0, case["vocab"], (case["batch"], case["prompt"] + case["new"]), generator=g, device=DEV)
        s["ids"] = ids
        s["decoder"] = GraphDecoder(model, batch=case["batch"])
        s["decoder"].prefill(ids[:, :case["prompt"]])  # captures its graphs, once per program
    return s


@torch.no_grad()
def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "quantize":
        return castor.quantize_indices(s["x"], mode=case["mode"])
    if kind == "requantize":
        return castor.requantize_h24(s["w"], mode="bf16")
    if kind == "pack":
        return pack.quantize_h24_layer(s["w"])
    if kind == "train":
        scalars = optim.step_scalars(s["heat"], s["step"], s["inertia"], DEV)
        norms, codes = optim.pollux_h24_step_many_(s["params"], heat=s["heat"], step=s["step"],
                                                   width_inertia=s["inertia"], mode="bf16", return_codes=True,
                                                   scalars=scalars)
        return [{"p": p, "m": m, "v": v, "latent": lat, "norm": n, "packed": k["packed"], "sigma": k["sigma"]}
                for (p, _, m, v, lat), n, k in zip(s["params"], norms, codes)]
    if kind == "codec":
        packed = castor.pack_indices(s["idx"])
        return {"packed": packed, "indices": castor.unpack_indices(packed, s["idx"].numel()),
                "weight": dequantize_h24(packed, s["sigma"], case["rows"], case["cols"])}
    if kind == "linear":
        return s["layer"](s["x"])
    if kind == "block":
        s["cache"].length = 0
        return {"y": s["block"](s["x"], s["cache"], 0), "k": s["cache"].k[0], "v": s["cache"].v[0]}
    if kind == "head":
        return s["layer"](s["x"], norm=(s["norm"], 1e-8))
    dec, t, ids = s["decoder"], case["prompt"], s["ids"]
    logits = [dec.prefill(ids[:, :t])]
    for i in range(case["new"]):  # the next token of each sequence is the caller's choice
        logits.append(dec.decode(ids[:, t + i]).clone())
    return torch.stack(logits)


# ---------------------------------------------------------------- what a pass cannot do without


def _linear_bytes(out: int, inn: int) -> float:
    return 2.25 * out * inn / 24 + 2 * out


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("quantize", "requantize", "pack", "codec"):
        el = case["rows"] * case["cols"]
        n = el // 24
        # the sums over 2,048 Golay sign patterns and 759 octads that order the 196,560 codes
        nn = 2.0 * 24 * (2048 + 759) * n
        if kind == "quantize":
            return {"bytes": 4.0 * el + 4 * n, "flops": nn}
        if kind == "requantize":
            return {"bytes": 8.0 * el + 6.25 * n + 4 * case["rows"], "flops": nn}
        if kind == "pack":
            return {"bytes": 4.0 * el + 2.25 * n + 2 * case["rows"], "flops": nn}
        return {"bytes": n * (4 + 2.25 + 2.25 + 8 + 2.25 + 48) + 2 * case["rows"], "flops": 0.0}
    if kind == "train":
        el = sum(r * c for r, c in _train_shapes(case["d"]))
        return {"bytes": el * 32.0 + 2.25 * el / 24, "flops": 2.0 * (2048 + 759) * el}
    if kind == "linear":
        sz = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": _linear_bytes(case["out"], case["in"]) + sz * case["tokens"] * (case["out"] + case["in"]),
                "flops": 2.0 * case["tokens"] * case["out"] * case["in"]}
    if kind == "head":
        return {"bytes": float(case["vocab"] * (case["d"] + 2) + 4 * case["tokens"] * (case["vocab"] + case["d"])),
                "flops": 2.0 * case["tokens"] * case["vocab"] * case["d"]}
    d = 24 * case["heads"]
    block = 6 * _linear_bytes(2 * d, d)
    if kind == "block":
        t, b = case["tokens"], case["batch"]
        return {"bytes": block + 16.0 * b * t * d, "flops": b * t * (24.0 * d * d + 2.0 * t * d)}
    # generate: one pass over the prompt, then one position per new token; every step reads every weight
    b, p, new, L, v = case["batch"], case["prompt"], case["new"], case["layers"], case["vocab"]
    kv = 8.0 * b * d * L * (p + sum(p + i + 1 for i in range(new)))
    return {"bytes": (new + 1) * (L * block + v * (d + 2) + 4.0 * b * v) + kv,
            "flops": b * (L * 24.0 * d * d * (p + new) + 2.0 * d * v * (new + 1)
                          + 2.0 * L * d * (p * p + sum(2.0 * (p + i + 1) for i in range(new))))}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "codec":
        return "exact"
    if kind in ("quantize", "requantize", "train"):
        # codes: an atom within an fp32 rounding of a tie may take the other code; scales, moments and
        # weights: fp32 sums and elementwise steps (measured up to 1.6e-7 from the float64 values)
        return {"rel": 1e-6, "max": 1e-5, "differ": 5e-5}
    if kind == "pack":
        # fp16 row scales: another summation order moves one in some thousand by an ulp
        return {"rel": 1e-4, "max": 1e-3, "differ": 5e-5}
    if kind == "linear" and case["dtype"] == "bf16":
        # fp32 sums (1e-7 apart) rounded to bf16: one value in some ten thousand takes the neighbouring one
        return {"rel": 2e-4, "max": 1e-2}
    if kind == "generate":
        return {"rel": 2e-6, "max": 8e-5}  # whole model; measured 3.2e-7 from float64
    return {"rel": 1.5e-6, "max": 6e-5}  # fp32 sums of up to 7,680 terms; measured 1.4e-7 to 3.2e-7


# ---------------------------------------------------------------- float64 values


@functools.lru_cache(maxsize=1)
def _codebook_int8() -> np.ndarray:
    """The 196,561 codes as raw integers: origin, then the minimal vectors in lexicographic order."""
    words = []
    for msg in range(4096):  # extended Golay code, generator x^11 + x^9 + x^7 + x^6 + x^5 + x + 1
        rem = msg << 11
        for bit in range(22, 10, -1):
            if rem >> bit & 1:
                rem ^= 0xAE3 << (bit - 11)
        w = msg << 11 | rem
        words.append(w | (bin(w).count("1") & 1) << 23)
    bits = ((np.array(words)[:, None] >> np.arange(24)) & 1).astype(np.int8)
    rows = []
    for i in range(24):
        for j in range(i + 1, 24):
            two = np.zeros((4, 24), np.int8)
            two[:, i], two[:, j] = [-4, -4, 4, 4], [-4, 4, -4, 4]
            rows.append(two)
    signs = np.array([[1 - 2 * (k >> b & 1) for b in range(8)] for k in range(256)], np.int8)
    signs = signs[(signs < 0).sum(1) % 2 == 0]
    for o in bits[bits.sum(1) == 8]:
        eight = np.zeros((128, 24), np.int8)
        eight[:, np.flatnonzero(o)] = 2 * signs
        rows.append(eight)
    for p in range(24):
        odd = 1 - 2 * bits
        odd[:, p] = -3
        rows.append(odd)
    raw = np.concatenate(rows)
    raw = raw[np.lexsort(raw.T[::-1])]
    return np.concatenate([np.zeros((1, 24), np.int8), raw])


@functools.lru_cache(maxsize=1)
def _codebook16() -> torch.Tensor:
    table = _codebook_int8().astype(np.float32) * np.float32(1.0 / math.sqrt(8.0))
    return torch.from_numpy(table).to(DEV).half()


def _dense16(idx: torch.Tensor, sigma: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    """The stored fp16 weight that a packed layer stands for."""
    c = _codebook16()[idx.long()].view(rows, cols)
    return (c * sigma.view(-1, 1)) * float(1.0 / SQRT2)


def _dense_layer(layer: PackedH24Linear, idx: torch.Tensor) -> torch.Tensor:
    return _dense16(idx, layer.sigma_rows, layer.out_features, layer.in_features).double()


def _int8_dense(layer) -> torch.Tensor:
    step = layer.mu_rows.float() * float(np.float32(1.0) / np.float32(127.0))
    return (layer.weight_int8.half() * step.half().unsqueeze(-1)).double()


def _norm64(x: torch.Tensor, w: torch.Tensor, eps: float = 1e-8) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _block64(block: PackedBlock, idx: list[torch.Tensor], x: torch.Tensor):
    """(output, keys, values) of a decoder block over whole sequences."""
    b, t, d = x.shape
    a, m = block.attn, block.mlp
    layers = (a.q_proj, a.k_proj, a.v_proj, a.o_proj, m.fc1, m.fc2)

    def mul(i, v):
        return v @ _dense_layer(layers[i], idx[i]).T

    n = _norm64(x, block.ln1.weight)
    q, k, v = (mul(i, n).view(b, t, d // 24, 24).transpose(1, 2).contiguous() for i in range(3))
    q, k = _norm64(q, a.q_ln.weight), _norm64(k, a.k_ln.weight)
    mask = torch.ones(t, t, dtype=torch.bool, device=x.device).triu(1)
    out = torch.empty_like(q)
    for i in range(b):
        s = (q[i] @ k[i].transpose(1, 2).contiguous()) / math.sqrt(24.0)
        out[i] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[i]
    x = x + mul(3, out.transpose(1, 2).reshape(b, t, d))
    h = torch.nn.functional.gelu(mul(4, _norm64(x, block.ln2.weight)))
    return x + mul(5, h), k, v


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "quantize":
        return None  # whole numbers
    s = prepare(case, seed)
    if kind in ("requantize", "pack"):
        rms = (s["w"].double().square().mean(1) + 1e-8).sqrt()
        if kind == "pack":
            return (None, rms * math.sqrt(12.0))
        return {"sigma": rms, "indices": None, "packed": None, "weight": None}
    if kind == "train":
        gamma = 0.065771
        b1, b2 = 1.0 - math.sqrt(gamma), 1.0 - gamma
        cap = (SQRT2 - 1.0) / 2.0 / SQRT2
        scale = HEAT * gamma / SQRT2 / s["inertia"]
        out = []
        for _, grad, m, v, lat in s["params"]:
            gr = grad.double()
            m64 = m.double() * b1 + (1 - b1) * gr
            v64 = v.double() * b2 + (1 - b2) * gr * gr
            st = -scale * (m64 / (1 - b1 ** (STEP + 1))) / ((v64 / (1 - b2 ** (STEP + 1))).sqrt() + 1e-8)
            norm = st.view(-1, 24).norm(dim=1, keepdim=True)
            st = (st.view(-1, 24) * (cap / norm.clamp_min(1e-8)).clamp(max=1.0)).view_as(st)
            lat64 = lat.double() * (1.0 - HEAT * gamma ** 2) + st
            out.append({"p": None, "m": m64, "v": v64, "latent": lat64, "norm": st.norm(), "packed": None,
                        "sigma": (lat64.square().mean(1) + 1e-8).sqrt()})
        return out
    if kind == "codec":
        table = torch.from_numpy(_codebook_int8()).to(DEV)
        w = table[s["idx"].long()].double().view(case["rows"], case["cols"])
        w.mul_(s["sigma"].double().view(-1, 1) / 4.0)  # 1 / sqrt 8 / sqrt 2
        return {"packed": None, "indices": None, "weight": w}
    if kind == "linear":
        return s["x"].double() @ _dense_layer(s["layer"], s["idx"]).T
    if kind == "block":
        y, k, v = _block64(s["block"], s["idx"], s["x"].double())
        return {"y": y, "k": k, "v": v}
    if kind == "head":
        return _norm64(s["x"].double(), s["norm"]) @ _int8_dense(s["layer"]).T
    model, t, n = s["model"], case["prompt"], case["new"]
    emb = _int8_dense(model.tok_emb)
    x = emb[s["ids"]] + model.pos_emb.weight[:t + n].double()
    del emb
    for block, idx in zip(model.blocks, s["idx"]):
        x = _block64(block, idx, x)[0]
    y = _norm64(x[:, t - 1:], model.ln_f.weight)
    w = _int8_dense(model.head)
    return torch.stack([y[:, i].contiguous() @ w.T for i in range(n + 1)])
