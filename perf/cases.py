"""The work that a user of nestedtensor_amd has it do, as measurable cases.

Six kinds of pass, each through the package's public entry points:

  collate   a list of token-id tensors -> nested tensor -> (padded ids, mask)
  pad       packed sequences -> padded tensor -> packed again, by value or by length
  images    a list of ragged images -> nested tensor -> (padded, mask) -> nested again
  mha       one nested multi-head attention layer (self- or cross-attention)
  encoder   token ids -> embedding -> one transformer encoder layer -> padded output
  conv      ragged feature maps through two 1x1 convolutions, row-major and
            channels-last storage

Every case is a plain dict; the lengths of a batch follow from the case alone, the
values and the order of the batch from the seed.
"""

import math
import random

import torch
import torch.nn.functional as F

import nestedtensor_amd as nt

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i64": torch.int64}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "i64": 8}
DEVICE = "cuda"


def listed():
    return [
        # A serving or training loop's collate step: a small batch of token ids becomes
        # a padded tensor and its mask.  Next to no data: launches and host work.
        dict(name="collate_ids", kind="collate", dtype="i64", batch=64, spread="uniform", low=8, high=128, lengths=11),
        # Activations of a small model handed to dense code and taken back (fp32, pad value 0).
        dict(name="pad_small_f32", kind="pad", dtype="f32", batch=64, spread="uniform", low=1, high=128, width=256,
             back="value", lengths=1010),
        # A chunk of a large corpus of hidden states: 512 sequences, 4.3 GB packed, padded
        # and un-padded again from the known lengths.  Bound by memory.
        dict(name="pad_large_f16", kind="pad", dtype="f16", batch=512, spread="uniform", low=1, high=2048, width=4096,
             back="length", lengths=1014),
        # A detection batch: sixteen fp32 images of different sizes, batched with a mask and
        # split up again.
        dict(name="images_f32", kind="images", dtype="f32", batch=16, channels=3, low=480, high=1024, lengths=1011),
        # Online serving: four short sequences arrive as separate tensors, one attention
        # layer, padded result.  A new nested size on every pass, next to no arithmetic.
        dict(name="mha_serve_f16", kind="mha", form="serve", dtype="f16", batch=4, spread="uniform", low=8, high=64,
             heads=8, head_dim=64, lengths=3),
        # A BERT-base sized self-attention layer, fp16.
        dict(name="mha_base_f16", kind="mha", form="self", dtype="f16", batch=32, spread="uniform", low=32, high=512,
             heads=12, head_dim=64, lengths=1012),
        # Many sequences, most of them short (high raggedness), bf16.
        dict(name="mha_ragged_bf16", kind="mha", form="bt", dtype="bf16", batch=128, spread="exp", low=8, high=512,
             heads=16, head_dim=64, lengths=1013),
        # A wide layer on long documents: arithmetic-bound.
        dict(name="mha_long_f16", kind="mha", form="self", dtype="f16", batch=16, spread="uniform", low=256, high=2048,
             heads=16, head_dim=128, lengths=1015),
        # The BERT-base layer in single precision.
        dict(name="mha_base_f32", kind="mha", form="self", dtype="f32", batch=32, spread="uniform", low=32, high=512,
             heads=12, head_dim=64, lengths=1012),
        # A decoder's cross-attention: 100 queries per sequence against a ragged memory.
        dict(name="mha_cross_f16", kind="mha", form="cross", dtype="f16", batch=32, spread="uniform", low=256,
             high=1024, queries=100, heads=8, head_dim=64, lengths=1016),
        # A whole encoder layer from token ids to a padded result, fp16, a new batch on
        # every pass.
        dict(name="encoder_base_f16", kind="encoder", dtype="f16", batch=32, spread="uniform", low=32, high=512,
             heads=12, head_dim=64, vocab=30522, lengths=1012),
        # The 1x1 convolutions of a bottleneck block on ragged feature maps.
        dict(name="conv_maps_f16", kind="conv", dtype="f16", batch=16, channels=64, inner=256, low=120, high=256,
             lengths=1011),
    ]


def _log_int(rng, low, high):
    """An integer spread evenly over the logarithm of [low, high]."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case of the ranges above."""
    while True:
        case = _draw_once(rng)
        w = work(case)
        # no drawn case costs more than the largest listed one; fp32 products run at a
        # sixteenth of the rate of fp16 ones
        if w["bytes"] <= 8e9 and w["flops"] * (16 if case["dtype"] == "f32" else 1) <= 8e11:
            return case


def _draw_once(rng):
    kind = rng.choice(("collate", "pad", "pad", "images", "mha", "mha", "mha", "encoder", "conv"))
    case = dict(kind=kind, lengths=rng.randrange(1, 1 << 20))
    if kind == "collate":
        high = _log_int(rng, 16, 1024)
        case.update(dtype="i64", batch=_log_int(rng, 2, 256), spread="uniform", low=rng.randint(1, high), high=high)
    elif kind == "pad":
        high = _log_int(rng, 8, 2048)
        back = rng.choice(("value", "length"))
        case.update(dtype=rng.choice(("f32", "f16", "bf16")), batch=_log_int(rng, 4, 512),
                    spread=rng.choice(("uniform", "exp")), low=1, high=high, width=_log_int(rng, 16, 4096), back=back)
    elif kind == "images":
        high = _log_int(rng, 64, 1024)
        case.update(dtype=rng.choice(("f32", "f16")), batch=_log_int(rng, 2, 32), channels=rng.choice((1, 3)),
                    low=max(32, high // 2), high=high)
    elif kind in ("mha", "encoder"):
        head_dim = rng.choice((32, 64, 64, 128))
        heads = rng.randint(2, 2048 // head_dim if head_dim == 128 else 16)
        high = _log_int(rng, 16, 2048)
        case.update(dtype=rng.choice(("f16", "bf16", "f32")) if kind == "mha" else rng.choice(("f16", "bf16")),
                    batch=_log_int(rng, 1, 256), spread=rng.choice(("uniform", "exp")), low=max(1, high // 16),
                    high=high, heads=heads, head_dim=head_dim)
        if kind == "encoder":
            case.update(vocab=30522)
        else:
            case.update(form=rng.choice(("serve", "self", "bt", "cross")))
            if case["form"] == "cross":
                case.update(queries=_log_int(rng, 8, 512))
    else:
        high = _log_int(rng, 32, 320)
        case.update(dtype=rng.choice(("f16", "bf16")), batch=_log_int(rng, 2, 32), channels=rng.choice((32, 64, 128)),
                    inner=rng.choice((64, 128, 256)), low=max(16, high // 2), high=high)
    return case


def _lengths(case):
    """The lengths of the batch, at least one of them the longest allowed."""
    rng = random.Random(case["lengths"])
    low, high = case["low"], case["high"]
    if case.get("spread") == "exp":
        # truncated exponential: most sequences are short
        mean = low + (high - low) * 0.18
        out = [max(low, min(high, int(round(rng.expovariate(1.0 / mean))))) for _ in range(case["batch"])]
    else:
        out = [rng.randint(low, high) for _ in range(case["batch"])]
    out[0] = high
    return out


def _extents(case):
    """(H, W) of a batch of images, at least one of the largest height and one of the largest width."""
    rng = random.Random(case["lengths"])
    out = [[rng.randint(case["low"], case["high"]) for _ in range(2)] for _ in range(case["batch"])]
    out[0][0] = out[-1][1] = case["high"]
    return out


def _normal(shape, dtype, gen, scale=1.0):
    return torch.randn(shape, device=DEVICE, dtype=dtype, generator=gen).mul_(scale)


def prepare(case, seed):
    gen = torch.Generator(DEVICE).manual_seed(seed)
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    shuffle = random.Random(seed).shuffle
    state = dict(case=case, dtype=dtype)
    if kind in ("images", "conv"):
        extents = _extents(case)
        shuffle(extents)
        maps = [torch.rand((case["channels"], h, w), device=DEVICE, generator=gen).to(dtype) for h, w in extents]
        if kind == "images":
            state["images"] = maps
        else:
            c, n = case["channels"], case["inner"]
            state["maps"] = nt.nested_tensor(maps, dtype=dtype, device=DEVICE)
            state["expand"] = _normal((n, c, 1, 1), dtype, gen, c ** -0.5)
            state["reduce"] = _normal((c, n, 1, 1), dtype, gen, n ** -0.5)
        return state
    lengths = _lengths(case)
    shuffle(lengths)
    total = sum(lengths)
    if kind in ("collate", "encoder"):
        ids = torch.randint(0, case.get("vocab", 30522), (total,), device=DEVICE, generator=gen)
        state["ids"] = [t.clone() for t in ids.split(lengths)]
        if kind == "collate":
            return state
    elif kind == "pad":
        # an exact zero would be read as padding when the rows are taken back by value
        flat = _normal((total, case["width"]), dtype, gen)
        if case["back"] == "value":
            flat.masked_fill_(flat == 0, 0.5)
        state["packed"] = nt.nested_tensor(list(flat.split(lengths)), dtype=dtype, device=DEVICE)
        return state
    E, H = case["heads"] * case["head_dim"], case["heads"]
    state["attention"] = dict(
        heads=H, head_dim=case["head_dim"], scaling=case["head_dim"] ** -0.5,
        w_in=_normal((3 * E, E), dtype, gen, 0.02), b_in=_normal((3 * E,), dtype, gen, 0.02),
        w_out=_normal((E, E), dtype, gen, 0.02), b_out=_normal((E,), dtype, gen, 0.02))
    if kind == "encoder":
        state["table"] = _normal((case["vocab"], E), dtype, gen)
        state["w1"], state["b1"] = _normal((4 * E, E), dtype, gen, 0.02), _normal((4 * E,), dtype, gen, 0.02)
        state["w2"], state["b2"] = _normal((E, 4 * E), dtype, gen, 0.02), _normal((E,), dtype, gen, 0.02)
        for k in ("1", "2"):
            state["gain" + k] = 1 + _normal((E,), dtype, gen, 0.1)
            state["shift" + k] = _normal((E,), dtype, gen, 0.1)
        return state
    tokens = [t.clone() for t in _normal((total, E), dtype, gen).split(lengths)]
    if case["form"] == "serve":
        state["tokens"] = tokens
        layer = torch.nn.MultiheadAttention(E, H, device=DEVICE, dtype=dtype).eval()
        p = state["attention"]
        for param, value in ((layer.in_proj_weight, p["w_in"]), (layer.in_proj_bias, p["b_in"]),
                             (layer.out_proj.weight, p["w_out"]), (layer.out_proj.bias, p["b_out"])):
            param.data.copy_(value)
            param.requires_grad_(False)
        state["layer"] = layer
        return state
    state["memory"] = nt.nested_tensor(tokens, dtype=dtype, device=DEVICE)
    if case["form"] == "cross":
        queries = _normal((case["batch"], case["queries"], E), dtype, gen)
        state["query"] = nt.nested_tensor(list(queries), dtype=dtype, device=DEVICE)
    else:
        state["query"] = state["memory"]
    return state


def _attention(state, query, memory, op=None):
    p = state["attention"]
    op = op or torch.ops.nestedtensor.min_mha
    return op(p["heads"], p["head_dim"], 0.0, False, query, memory, memory, p["w_in"], p["b_in"], p["scaling"],
              p["w_out"], p["b_out"])


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


def _run_collate(state, case):
    ids = nt.nested_tensor(state["ids"], dtype=torch.int64, device=DEVICE)
    return ids.to_tensor_mask()


def _run_pad(state, case):
    packed = state["packed"]
    padded = packed.to_padded_tensor(0)
    if case["back"] == "value":
        again = nt.nested_tensor_from_padded_tensor(padded, padding=0)
    else:
        again = nt.from_padded_tensor(padded, packed)
    return padded, again._impl.buffer, again._impl.sizes


def _run_images(state, case):
    images = nt.nested_tensor(state["images"], dtype=state["dtype"], device=DEVICE)
    data, mask = images.to_tensor_mask()
    again = nt.nested_tensor_from_tensor_mask(data, mask)
    return data, mask, again._impl.buffer, again._impl.sizes


def _run_mha(state, case):
    if case["form"] == "serve":
        x = nt.nested_tensor(state["tokens"], dtype=state["dtype"], device=DEVICE)
        return state["layer"](x, x, x, need_weights=False)[0].to_padded_tensor(0)
    op = torch.ops.nestedtensor.bt_min_mha if case["form"] == "bt" else None
    return _attention(state, state["query"], state["memory"], op)._impl.buffer


def _run_encoder(state, case):
    E = case["heads"] * case["head_dim"]
    ids = nt.nested_tensor(state["ids"], dtype=torch.int64, device=DEVICE)
    x = F.embedding(ids, state["table"])
    x = F.layer_norm(x + _attention(state, x, x), (E,), state["gain1"], state["shift1"])
    y = F.linear(nt.linear_act(x, state["w1"], state["b1"], "gelu"), state["w2"], state["b2"])
    return F.layer_norm(x + y, (E,), state["gain2"], state["shift2"]).to_padded_tensor(0)


def _run_conv(state, case):
    wide = F.relu(torch.conv2d(state["maps"], state["expand"]))
    narrow = torch.conv2d(wide.contiguous(memory_format=torch.channels_last), state["reduce"])
    return narrow.contiguous()._impl.buffer


_RUN = dict(collate=_run_collate, pad=_run_pad, images=_run_images, mha=_run_mha, encoder=_run_encoder, conv=_run_conv)


def work(case):
    kind, eb, B = case["kind"], BYTES[case["dtype"]], case["batch"]
    if kind in ("images", "conv"):
        pixels = sum(h * w for h, w in _extents(case))
        c = case["channels"]
        if kind == "conv":
            n = case["inner"]
            return {"bytes": 2 * pixels * c * eb + 2 * c * n * eb, "flops": 4 * pixels * c * n}
        padded = B * c * case["high"] ** 2
        # packed: images read, buffer written; padded: buffer read, tensor and mask written;
        # back: tensor and mask read where they hold data, buffer written
        return {"bytes": 5 * pixels * c * eb + padded * (eb + 2), "flops": 0}
    lengths = _lengths(case)
    total = sum(lengths)
    if kind == "collate":
        return {"bytes": 2 * total * eb + total * eb + B * max(lengths) * (eb + 1), "flops": 0}
    if kind == "pad":
        valid, padded = total * case["width"] * eb, B * max(lengths) * case["width"] * eb
        # taken back by value the whole padded tensor has to be read, by length its rows only
        return {"bytes": valid + padded + (padded if case["back"] == "value" else valid) + valid, "flops": 0}
    E = case["heads"] * case["head_dim"]
    if kind == "encoder":
        return {"bytes": total * (8 + E * eb) + 12 * E * E * eb + B * max(lengths) * E * eb,
                "flops": 24 * total * E * E + 4 * E * sum(n * n for n in lengths)}
    if case["form"] == "cross":
        queries = B * case["queries"]
        return {"bytes": (2 * queries + total) * E * eb + 4 * E * E * eb,
                "flops": 4 * queries * E * E + 4 * total * E * E + 4 * E * case["queries"] * total}
    out = B * max(lengths) * E * eb if case["form"] == "serve" else total * E * eb
    return {"bytes": total * E * eb + out + 4 * E * E * eb,
            "flops": 8 * total * E * E + 4 * E * sum(n * n for n in lengths)}


def tolerance(case):
    if case["kind"] in ("collate", "pad", "images"):
        return "exact"
    # four times what the path differs from the same computation in 64 bits (2-norm: 4.3e-4 in
    # fp16, 3.4e-3 in bf16, 9e-7 in fp32; largest: 3.6e-3, 4.3e-2 and 8e-6)
    return {"f16": {"rel": 1.7e-3, "max": 1.5e-2}, "bf16": {"rel": 1.3e-2, "max": 0.17},
            "f32": {"rel": 4e-6, "max": 4e-5}}[case["dtype"]]
