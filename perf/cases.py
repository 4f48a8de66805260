"""Performance cases of the SDXL attention path on one MI355X.

Each case is one call that a program makes through the public entry points of ``sdxl_hip``: the
attention of the UNet, of the text encoders and of the VAE, the attention sublayers of a transformer
block, and the per-request projection of the text context. The listed cases are points of the ranges
that ``draw`` samples; sizes are image-token counts of square and non-square latents (multiples of no
tile), the text encoders' 77 tokens, and generic lengths for the masked and fallback calls.
"""
import math
import os
import sys

import torch

_PACKAGE_DIR = os.path.join(os.getcwd(), "sdxl-end2end_amd")
if _PACKAGE_DIR not in sys.path:
    sys.path.insert(0, _PACKAGE_DIR)

import sdxl_hip  # noqa: E402

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
_DEVICE = "cuda:0"


# ------------------------------------------------------------------------------------ the cases
def _attention(batch, heads, q_seq, k_seq, head_dim=64, dtype="f16", causal=False, mask=False, packed=False):
    return {"kind": "attention", "batch": batch, "heads": heads, "q_seq": q_seq, "k_seq": k_seq,
            "head_dim": head_dim, "dtype": dtype, "causal": causal, "mask": mask, "packed": packed}


def _self_sublayer(batch, seq, heads, weights, activations):
    return {"kind": "self_sublayer", "batch": batch, "seq": seq, "heads": heads, "weights": weights,
            "activations": activations}


def _cross_sublayer(batch, seq, heads, context, weights, activations):
    return {"kind": "cross_sublayer", "batch": batch, "seq": seq, "heads": heads, "context": context,
            "weights": weights, "activations": activations}


def _context_projection(batch, context, channels, width, weights):
    return {"kind": "context_projection", "batch": batch, "context": context, "channels": channels,
            "width": width, "weights": weights}


def listed():
    cases = {
        # A text encoder's causal self-attention: the smallest call, all latency.
        "text_causal_77": _attention(2, 12, 77, 77, causal=True),
        # Level-2 self-attention of a non-square image (26 x 38 latent tokens): ragged rows and keys, bf16.
        "self_l2_ragged_988": _attention(2, 20, 988, 988, dtype="bf16"),
        # Level-1 self-attention of a 1024 x 1024 image with guidance (batch 2): the UNet's dominant call.
        "self_l1_4096": _attention(2, 10, 4096, 4096),
        # Level-1 cross-attention against the 77 text tokens, two non-square images with guidance.
        "cross_l1_77": _attention(4, 10, 3840, 77),
        # A padded batch of longer prompts in a causal encoder: key mask and causal limit together.
        "masked_causal_1500": _attention(2, 16, 1500, 1500, causal=True, mask=True),
        # The VAE's single-head FP32 attention: a 512 x 512 image and a 1024 x 1024 one (the largest call).
        "vae_f32_4096": _attention(1, 1, 4096, 4096, head_dim=512, dtype="f32"),
        "vae_f32_16384": _attention(1, 1, 16384, 16384, head_dim=512, dtype="f32"),
        # The UNet's level-2 attention run wholly in FP32 (an upcast pipeline): outside the 16-bit kernels.
        "self_f32_1024": _attention(1, 20, 1024, 1024, dtype="f32"),
        # The self-attention sublayer of a level-1 block, E4M3 weights.
        "self_sublayer_l1": _self_sublayer(2, 4096, 10, "e4m3", "f16"),
        # The same of a level-2 block with E4M3 activations as well.
        "self_sublayer_l2_fp8": _self_sublayer(2, 1024, 20, "e4m3", "e4m3"),
        # The cross-attention sublayer of a level-2 block, fp16 weights.
        "cross_sublayer_l2": _cross_sublayer(2, 1024, 20, 77, "f16", "f16"),
        # K | V of the text context, once per request and block.
        "context_projection": _context_projection(2, 77, 2048, 1280, "f16"),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    family = rng.choice(("self", "self", "cross", "text", "vae", "fallback", "self_sublayer", "cross_sublayer",
                         "context_projection"))
    if family == "self":  # image tokens, either level, up to a 1024 x 1024 image's guided batch
        batch, heads = rng.choice((1, 2, 4)), rng.choice((10, 20))
        seq = _log_int(rng, 200, 4200 // (2 if batch * heads > 40 else 1))
        return _attention(batch, heads, seq, seq, dtype=rng.choice(("f16", "bf16")), packed=rng.random() < 0.5)
    if family == "cross":
        batch, heads = rng.choice((1, 2, 4)), rng.choice((10, 20))
        return _attention(batch, heads, _log_int(rng, 200, 4200), rng.choice((77, 77, 154, rng.randint(1, 231))),
                          dtype=rng.choice(("f16", "bf16")))
    if family == "text":
        seq = rng.choice((77, _log_int(rng, 20, 2000)))
        return _attention(rng.choice((1, 2, 4)), rng.choice((12, 16, 20)), seq, seq, dtype=rng.choice(("f16", "bf16")),
                          causal=rng.random() < 0.7, mask=rng.random() < 0.6)
    if family == "vae":
        seq = _log_int(rng, 500, 16384)
        return _attention(2 if seq < 4000 and rng.random() < 0.3 else 1, 1, seq, seq, head_dim=512, dtype="f32")
    if family == "fallback":
        dtype = rng.choice(("f32", "f32", "f16", "bf16"))
        head_dim = rng.choice((16, 40, 64, 80, 128, 160, rng.randint(8, 200)))
        if dtype != "f32" and head_dim == 64:
            head_dim = 80
        seq = _log_int(rng, 77, 1200)
        return _attention(rng.choice((1, 2)), rng.randint(2, 12), seq, rng.choice((seq, 77)), head_dim, dtype,
                          causal=rng.random() < 0.2, mask=rng.random() < 0.3)
    weights = rng.choice(("f16", "e4m3"))
    if family == "context_projection":
        return _context_projection(rng.choice((1, 2, 4)), rng.choice((77, 154, rng.randint(1, 231))),
                                   rng.choice((768, 1280, 2048)), rng.choice((640, 1280)), weights)
    activations = rng.choice(("f16", "e4m3")) if weights == "e4m3" else "f16"
    heads = rng.choice((10, 20))
    batch, seq = rng.choice((1, 2, 4)), _log_int(rng, 200, 4200 if heads == 10 else 1100)
    if family == "self_sublayer":
        return _self_sublayer(batch, seq, heads, weights, activations)
    return _cross_sublayer(batch, seq, heads, rng.choice((77, 77, rng.randint(1, 154))), weights, activations)


# ------------------------------------------------------------------------------------ the inputs
def _pack_e4m3(rows):
    """Codes and fp32 scales of the library's row rule: amax / 448, nearest even."""
    rows = rows.float()
    amax = rows.abs().amax(dim=-1, keepdim=True)
    scale = torch.where(amax > 0, (amax / 448.0).clamp_min(1e-12), torch.ones_like(amax))
    codes = (rows / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return codes.view(torch.uint8), scale.squeeze(-1).contiguous()


def _inputs(case, seed):
    gen = torch.Generator(device=_DEVICE)
    gen.manual_seed(seed)

    def normal(*shape, std=1.0, mean=0.0, dtype=torch.float16):
        return (torch.randn(*shape, generator=gen, device=_DEVICE, dtype=torch.float32) * std + mean).to(dtype)

    if case["kind"] == "attention":
        dtype = _DTYPES[case["dtype"]]
        batch, q_seq, k_seq = case["batch"], case["q_seq"], case["k_seq"]
        width = case["heads"] * case["head_dim"]
        if case["packed"]:  # q | k | v as one projection leaves them
            query, key, value = normal(batch, q_seq, 3 * width, dtype=dtype).split(width, dim=-1)
        else:
            query = normal(batch, q_seq, width, dtype=dtype)
            key, value = (normal(batch, k_seq, width, dtype=dtype) for _ in range(2))
        key_mask = None
        if case["mask"]:  # padding at the end of each sequence, at least one token kept
            kept = torch.randint(k_seq // 2, k_seq + 1, (batch, 1), generator=gen, device=_DEVICE).clamp_min(1)
            key_mask = (torch.arange(k_seq, device=_DEVICE)[None, :] < kept).to(torch.int32)
        return {"query": query, "key": key, "value": value, "key_mask": key_mask}

    def weight(rows, cols):
        w = normal(rows, cols, std=cols ** -0.5)
        return _pack_e4m3(w) if case["weights"] == "e4m3" else (w, None)

    if case["kind"] == "context_projection":
        w, scale = weight(2 * case["width"], case["channels"])
        return {"context": normal(case["batch"], case["context"], case["channels"]), "w_kv": w, "w_kv_scale": scale}

    width = case["heads"] * 64
    data = {"x": normal(case["batch"], case["seq"], width), "gamma": normal(width, std=0.1, mean=1.0),
            "beta": normal(width, std=0.1), "w_out": normal(width, width, std=width ** -0.5),
            "b_out": normal(width, std=0.1)}
    data["w_in"], data["w_in_scale"] = weight(3 * width if case["kind"] == "self_sublayer" else width, width)
    if case["kind"] == "cross_sublayer":
        data["kv"] = normal(case["batch"], case["context"], 2 * width)
    return data


def prepare(case, seed):
    state = _inputs(case, seed)
    state["case"] = case
    if case["kind"].endswith("_sublayer"):  # the workspace that a program keeps over its blocks and steps
        rows, width = case["batch"] * case["seq"], case["heads"] * 64
        bytes_per_value = 8 if case["kind"] == "self_sublayer" else 4
        state["workspace"] = torch.empty(rows * width * bytes_per_value, dtype=torch.uint8, device=_DEVICE)
    return state


# ------------------------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    if case["kind"] == "attention":
        return sdxl_hip.attention(state["query"], state["key"], state["value"], case["heads"],
                                  causal=case["causal"], key_mask=state["key_mask"])
    if case["kind"] == "context_projection":
        return sdxl_hip.project_context_kv(state["context"], state["w_kv"], state["w_kv_scale"])
    fp8 = case["activations"] == "e4m3"
    if case["kind"] == "self_sublayer":
        return sdxl_hip.attn_sublayer(state["x"], state["gamma"], state["beta"], state["w_in"], state["w_in_scale"],
                                      state["w_out"], state["b_out"], case["heads"], workspace=state["workspace"],
                                      fp8_activations=fp8)
    return sdxl_hip.cross_attn_sublayer(state["x"], state["gamma"], state["beta"], state["w_in"],
                                        state["w_in_scale"], state["kv"], state["w_out"], state["b_out"],
                                        case["heads"], workspace=state["workspace"], fp8_activations=fp8)


# ------------------------------------------------------------------------------------ its work
def _attention_flops(case):
    q_seq, k_seq = case["q_seq"], case["k_seq"]
    pairs = q_seq * k_seq
    if case["causal"]:  # key j <= query i
        full = max(0, q_seq - k_seq)
        ramp = q_seq - full
        pairs = ramp * (ramp + 1) // 2 + full * k_seq
    return 4.0 * case["batch"] * case["heads"] * case["head_dim"] * pairs


def work(case):
    batch = case["batch"]
    if case["kind"] == "attention":
        elem = 4 if case["dtype"] == "f32" else 2
        width = case["heads"] * case["head_dim"]
        traffic = elem * batch * width * 2 * (case["q_seq"] + case["k_seq"])
        if case["mask"]:
            traffic += 4 * batch * case["k_seq"]
        return {"bytes": float(traffic), "flops": _attention_flops(case)}
    w_elem = 1 if case["weights"] == "e4m3" else 2
    if case["kind"] == "context_projection":
        rows, cols, depth = batch * case["context"], 2 * case["width"], case["channels"]
        traffic = 2 * rows * depth + w_elem * cols * depth + 2 * rows * cols
        return {"bytes": float(traffic), "flops": 2.0 * rows * cols * depth}
    rows, width = batch * case["seq"], case["heads"] * 64
    if case["kind"] == "self_sublayer":
        keys, in_cols, extra = case["seq"], 3 * width, 0
    else:
        keys, in_cols, extra = case["context"], width, 2 * batch * case["context"] * 2 * width
    traffic = 2 * 2 * rows * width + w_elem * in_cols * width + 2 * width * width + 2 * 3 * width + extra
    flops = 2.0 * rows * width * (in_cols + width) + 4.0 * rows * keys * width
    return {"bytes": float(traffic), "flops": flops}


def tolerance(case):
    # About four times the distance from 64 bits measured over these ranges: f16 2.9e-4, bf16 2.3e-3,
    # f32 2.3e-6, projections and sublayers 2.2e-4 (E4M3 activations: room for rounding ties besides).
    if case["kind"] == "attention":
        return {"rel": {"f16": 1.2e-3, "bf16": 1e-2, "f32": 1e-5}[case["dtype"]]}
    if case["kind"] == "context_projection":
        return {"rel": 1e-3}
    return {"rel": 2e-3 if case["activations"] == "e4m3" else 1e-3}


# ------------------------------------------------------------------------------------ in 64 bits
def _exact_attention(query, key, value, heads, causal=False, key_mask=None):
    batch, q_seq, width = query.shape
    k_seq, dim = key.shape[1], width // heads
    out = torch.zeros(batch, q_seq, width, dtype=torch.float64, device=query.device)
    rows = max(1, (1 << 27) // k_seq)  # at most 1 GiB of scores at a time
    for b in range(batch):
        for h in range(heads):
            cols = slice(h * dim, (h + 1) * dim)
            k64, v64 = key[b, :, cols].double(), value[b, :, cols].double()
            for first in range(0, q_seq, rows):
                scores = query[b, first:first + rows, cols].double() @ k64.t() / math.sqrt(dim)
                if key_mask is not None:
                    scores.masked_fill_(key_mask[b][None, :] == 0, -math.inf)
                if causal:
                    i = torch.arange(first, first + scores.shape[0], device=query.device)[:, None]
                    scores.masked_fill_(torch.arange(k_seq, device=query.device)[None, :] > i, -math.inf)
                out[b, first:first + rows, cols] = torch.softmax(scores, dim=-1) @ v64
    return out


def _dequantised(w, scale):
    if scale is None:
        return w.double()
    return w.view(torch.float8_e4m3fn).double() * scale.double()[:, None]


def exact(case, seed):
    data = _inputs(case, seed)
    if case["kind"] == "attention":
        return _exact_attention(data["query"], data["key"], data["value"], case["heads"], case["causal"],
                                data["key_mask"])
    if case["kind"] == "context_projection":
        return data["context"].double() @ _dequantised(data["w_kv"], data["w_kv_scale"]).t()
    x = data["x"].double()
    centred = x - x.mean(dim=-1, keepdim=True)
    normed = centred / torch.sqrt(centred.square().mean(dim=-1, keepdim=True) + 1e-5)
    normed = normed * data["gamma"].double() + data["beta"].double()
    if case["activations"] == "e4m3":  # the option's own rounding of the activations
        codes, scale = _pack_e4m3(normed)
        normed = codes.view(torch.float8_e4m3fn).double() * scale.double()[..., None]
    projected = normed @ _dequantised(data["w_in"], data["w_in_scale"]).t()
    if case["kind"] == "self_sublayer":
        query, key, value = projected.chunk(3, dim=-1)
    else:
        query, (key, value) = projected, data["kv"].chunk(2, dim=-1)
    attended = _exact_attention(query, key, value, case["heads"])
    return x + attended @ data["w_out"].double().t() + data["b_out"].double()
