"""The encoder calls that this repository's speed is judged by.

A pass is one call of an encoder's public `forward(modality, adapter_name, batch)`, as Eric's executor makes it for a
batch of requests: every model family, images and videos, one small image up to a full batch, bf16 and fp8 weights,
patches already on the device (what `Worker.upload` leaves there), fp32 patches in host memory (what the reference's
executor hands over) and frames as decoded.  Values are synthetic: N(0, 0.02) weights of the checkpoints' shapes, N(0, 1)
patches, U(-1, 1) SigLIP pixels, random bytes for photographs.

A server loads a checkpoint once and then meets new inputs: `prepare` keeps one model per family in this process (its
weights do not depend on the seed) and makes the batch from the seed.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from cornserve_amd.eric.api import Modality
from cornserve_amd.eric.frames import target_size
from cornserve_amd.eric.models.gemma3 import Gemma3VisionEncoder
from cornserve_amd.eric.models.llava_onevision import LlavaOneVisionEncoder, anyres_grid_shape
from cornserve_amd.eric.models.qwen2_5_vl import Qwen2_5_VisionTransformer
from cornserve_amd.eric.models.qwen2_vl import Qwen2VisionTransformer
from cornserve_amd.eric.models.qwen3_vl import Qwen3_VisionTransformer

PHOTO_BUDGET = (56 * 56, 14 * 14 * 4 * 1280)     # the image processor's default pixel budget


def listed() -> list[dict]:
    return [
        # one thumbnail or icon in a chat turn: the least work a request can carry, all latency
        {"name": "q25_thumbnail", "model": "qwen2_5_vl", "input": "device", "items": "1x112x168"},
        # one ordinary image alone: an interactive request while the queue is short
        {"name": "q25_one_image", "model": "qwen2_5_vl", "input": "device", "items": "1x448x448"},
        # one photograph straight from the decoder (host bytes; resize, normalisation and patch layout run on the GPU)
        {"name": "q25_photo", "model": "qwen2_5_vl", "input": "photo", "items": "1x1080x1920"},
        # eight equal images: the headline batch
        {"name": "q25_batch", "model": "qwen2_5_vl", "input": "device", "items": "1x448x448*8"},
        # sixteen images of every shape (sides uniform from 224 to 1344, seeded): a full batch of mixed traffic
        {"name": "q25_ragged", "model": "qwen2_5_vl", "input": "device", "items": _mixed_items(16, 224, 1344, 28, 4)},
        # fp8 weights on video: two clips of 16 frames
        {"name": "q25_fp8_videos", "model": "qwen2_5_vl_fp8", "input": "device", "items": "16x336x588*2"},
        # fp8 weights on one scanned page, sides that are not multiples of a window
        {"name": "q25_fp8_page", "model": "qwen2_5_vl_fp8", "input": "device", "items": "1x1036x756"},
        # two images of odd shapes in host memory, as the reference's executor hands them over
        {"name": "q2_host_pair", "model": "qwen2_vl", "input": "host", "items": "1x420x644,1x336x476"},
        # a small mixed batch of the newest family, with its deepstack outputs
        {"name": "q3_mixed", "model": "qwen3_vl", "input": "device", "items": "1x512x512,1x736x416,1x1056x800,1x288x640"},
        # one image of the fixed-size family, and a batch of them
        {"name": "gemma_one", "model": "gemma3", "input": "device", "items": "1x896x896"},
        {"name": "gemma_batch", "model": "gemma3", "input": "device", "items": "1x896x896*4"},
        # an image cut into tiles and merged into one sequence
        {"name": "llava_image", "model": "llava_ov", "input": "device", "items": "1x768x1152"},
    ]


def draw(rng) -> dict:
    kind = rng.choice(("qwen2_5_vl", "qwen2_5_vl", "qwen2_5_vl_fp8", "qwen2_vl", "qwen3_vl", "gemma3", "llava_ov"))
    if kind == "gemma3":
        n = rng.randint(1, 6)
        return {"model": kind, "input": rng.choice(("device", "host")), "items": f"1x896x896*{n}"}
    if kind == "llava_ov":
        if rng.random() < 0.3:
            return {"model": kind, "input": "device", "items": f"{rng.randint(2, 24)}x384x384"}
        n = rng.randint(1, 3)
        return {"model": kind, "input": "device",
                "items": ",".join(f"1x{rng.randint(200, 1600)}x{rng.randint(200, 1600)}" for _ in range(n))}
    if kind == "qwen2_5_vl" and rng.random() < 0.15:
        return {"model": kind, "input": "photo", "items": f"1x{rng.randint(120, 2400)}x{rng.randint(120, 2400)}"}
    factor = 32 if kind == "qwen3_vl" else 28
    patches = math.exp(rng.uniform(math.log(64), math.log(28000)))     # of the whole batch
    video = rng.random() < 0.25 and patches > 1000
    items, left = [], patches
    while left > 0 and len(items) < 16:
        share = min(left, 9000.0, max(16.0, patches * rng.uniform(0.1, 1.0)))
        frames = 2 * rng.randint(1, 8) if video else 1
        units = share / 4 / max(1, frames // 2)                        # merged units of one frame
        h = max(2, round(math.sqrt(units) * math.exp(rng.uniform(-0.5, 0.5))))
        w = max(2, round(units / h))
        items.append(f"{frames}x{h * factor}x{w * factor}")
        left -= max(1, frames // 2) * h * w * 4
    return {"model": kind, "input": rng.choice(("device", "device", "host")), "items": ",".join(items)}


# ---- batches ------------------------------------------------------------------------------------------------------
def _mixed_items(n: int, lo: int, hi: int, factor: int, seed: int) -> str:
    """n image sizes, sides spread over the multiples of `factor` in [lo, hi] by a fixed congruential sequence."""
    x, sides = seed, []
    for _ in range(2 * n):
        x = (x * 1103515245 + 12345) % 2**31
        sides.append((lo // factor + (x >> 16) % (hi // factor - lo // factor + 1)) * factor)
    return ",".join(f"1x{h}x{w}" for h, w in zip(sides[::2], sides[1::2]))


def _items(case: dict) -> list[tuple[int, int, int]]:
    """(frames, height, width) of every item."""
    out = []
    for part in case["items"].split(","):
        size, _, count = part.partition("*")
        out += [tuple(int(v) for v in size.split("x"))] * int(count or 1)
    return out


def _grids(case: dict) -> list[tuple[int, int, int]]:
    """(t, h, w) in patches of every item of a Qwen batch."""
    patch = 16 if case["model"] == "qwen3_vl" else 14
    grids = []
    for t, h, w in _items(case):
        if case["input"] == "photo":
            h, w = target_size(h, w, 28, *PHOTO_BUDGET)
        grids.append(((t + 1) // 2, h // patch, w // patch))
    return grids


def _tiles(case: dict) -> list[int]:
    """384-pixel tiles of every item of a LLaVA-OneVision batch (a video: its frames)."""
    cfg = _llava_config()
    if _items(case)[0][0] > 1:
        return [t for t, _, _ in _items(case)]
    return [1 + math.prod(anyres_grid_shape((h, w), cfg.image_grid_pinpoints, 384)) for _, h, w in _items(case)]


def _batch(case: dict, seed: int) -> tuple[Modality, dict]:
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = case["input"] == "host"

    def pixels(shape: tuple, lo: float | None = None) -> torch.Tensor:
        if lo is None:
            x = torch.randn(shape, generator=gen, device="cuda")
        else:
            x = torch.rand(shape, generator=gen, device="cuda") * -2 * lo + lo
        return x.cpu() if host else x.to(torch.bfloat16)

    if case["model"] == "gemma3":
        n = len(_items(case))
        return Modality.IMAGE, {"pixel_values": [pixels((1, 3, 896, 896), -1.0) for _ in range(n)],
                                "num_crops": [torch.zeros(1, dtype=torch.int64) for _ in range(n)]}
    if case["model"] == "llava_ov":
        px = [pixels((n, 3, 384, 384), -1.0) for n in _tiles(case)]
        if _items(case)[0][0] > 1:
            return Modality.VIDEO, {"pixel_values_videos": px}
        return Modality.IMAGE, {"pixel_values": px, "image_sizes": [torch.tensor([h, w]) for _, h, w in _items(case)]}
    if case["input"] == "photo":
        frames = [torch.randint(0, 256, (t, h, w, 3), dtype=torch.uint8, generator=gen, device="cuda").cpu()
                  for t, h, w in _items(case)]
        return Modality.IMAGE, {"raw_frames": frames, "raw_frames_budget": [torch.tensor(PHOTO_BUDGET) for _ in frames]}
    patch = 16 if case["model"] == "qwen3_vl" else 14
    px = [pixels((t * h * w, 3 * 2 * patch * patch)) for t, h, w in _grids(case)]
    grid = [torch.tensor([g], dtype=torch.int64) for g in _grids(case)]
    if _items(case)[0][0] > 1:
        return Modality.VIDEO, {"pixel_values_videos": px, "video_grid_thw": grid}
    return Modality.IMAGE, {"pixel_values": px, "image_grid_thw": grid}


# ---- models -------------------------------------------------------------------------------------------------------
def _siglip_config(image_size: int, layers: int) -> SimpleNamespace:
    return SimpleNamespace(hidden_size=1152, intermediate_size=4304, num_hidden_layers=layers, num_attention_heads=16,
                           num_channels=3, image_size=image_size, patch_size=14, layer_norm_eps=1e-6,
                           hidden_act="gelu_pytorch_tanh", attention_dropout=0.0, vision_use_head=False)


def _llava_config() -> SimpleNamespace:
    return SimpleNamespace(
        vision_config=_siglip_config(384, 26), text_config=SimpleNamespace(hidden_size=3584), vision_feature_layer=-1,
        vision_feature_select_strategy="full", projector_hidden_act="gelu", multimodal_projector_bias=True,
        image_grid_pinpoints=[[384 * i, 384 * j] for i in range(1, 7) for j in range(1, 7)],
        vision_aspect_ratio="anyres_max_9", model_type="llava_onevision")


def _new_model(kind: str):
    if kind in ("qwen2_5_vl", "qwen2_5_vl_fp8"):
        vc = SimpleNamespace(depth=32, hidden_size=1280, intermediate_size=3420, num_heads=16, in_channels=3, patch_size=14,
                             temporal_patch_size=2, spatial_merge_size=2, window_size=112, out_hidden_size=3584,
                             fullatt_block_indexes=[7, 15, 23, 31], hidden_act="silu")
        return Qwen2_5_VisionTransformer(SimpleNamespace(vision_config=vc),
                                         weight_format="fp8_e4m3" if kind.endswith("fp8") else "bf16")
    if kind == "qwen2_vl":
        vc = SimpleNamespace(depth=32, embed_dim=1280, hidden_size=3584, num_heads=16, mlp_ratio=4.0, in_channels=3,
                             patch_size=14, temporal_patch_size=2, spatial_merge_size=2)
        return Qwen2VisionTransformer(SimpleNamespace(vision_config=vc, rms_norm_eps=1e-6))
    if kind == "qwen3_vl":
        vc = SimpleNamespace(depth=27, hidden_size=1152, intermediate_size=4304, num_heads=16, in_channels=3, patch_size=16,
                             temporal_patch_size=2, spatial_merge_size=2, out_hidden_size=4096, num_position_embeddings=2304,
                             deepstack_visual_indexes=[8, 16, 24], hidden_act="gelu_pytorch_tanh")
        return Qwen3_VisionTransformer(SimpleNamespace(vision_config=vc))
    if kind == "gemma3":
        cfg = SimpleNamespace(vision_config=_siglip_config(896, 27), text_config=SimpleNamespace(hidden_size=2560),
                              mm_tokens_per_image=256, model_type="gemma3")
        model = Gemma3VisionEncoder(cfg)
        model.multi_modal_projector.make_adapter("a", cfg)
        return model
    return LlavaOneVisionEncoder(_llava_config())


_models: dict = {}


def _model(kind: str):
    if kind not in _models:
        with torch.device("cuda"):
            was = torch.get_default_dtype()
            torch.set_default_dtype(torch.bfloat16)
            try:
                model = _new_model(kind)
            finally:
                torch.set_default_dtype(was)
        model = model.to(device="cuda", dtype=torch.bfloat16).eval()
        gen = torch.Generator(device="cuda").manual_seed(1)
        modules = [model, *(model.multi_modal_projector.adapters.values() if kind == "gemma3" else ())]
        with torch.no_grad():
            for name, p in (np_ for m in modules for np_ in m.named_parameters()):
                p.copy_(torch.randn(p.shape, generator=gen, device="cuda") * 0.02)
                # (the projector norm of the fixed-size family has a zero-centred scale)
                if ("norm" in name or "ln_q" in name) and name.endswith("weight") and "soft_emb" not in name:
                    p.add_(1.0)
        _models[kind] = model
    return _models[kind]


# ---- what is measured ---------------------------------------------------------------------------------------------
def prepare(case: dict, seed: int) -> dict:
    modality, batch = _batch(case, seed)
    return {"model": _model(case["model"]), "modality": modality, "batch": batch}


def run(state: dict) -> list[torch.Tensor]:
    return state["model"](state["modality"], "a", state["batch"])


def work(case: dict) -> dict:
    """Weights, inputs and outputs once each; multiply-adds of the linear layers and of attention, two operations each."""
    kind = case["model"]
    if kind in ("gemma3", "llava_ov"):
        E, inter, patch_in = 1152, 4304, 3 * 14 * 14
        per, layers = (4096, 27) if kind == "gemma3" else (729, 26)
        tiles = len(_items(case)) if kind == "gemma3" else sum(_tiles(case))
        rows = tiles * per
        block, attn = 4 * E * E + 2 * E * inter, 4.0 * rows * per * E * layers
        if kind == "gemma3":
            out_rows, width, head = tiles * 256, 2560, 1152 * 2560
            head_flops = 2.0 * out_rows * head
        else:
            out_rows, width, head = rows, 3584, 1152 * 3584 + 3584 * 3584
            head_flops = 2.0 * rows * head
        weights = 2.0 * (layers * block + patch_in * E + head)
        in_bytes = tiles * 3.0 * (896 if kind == "gemma3" else 384) ** 2 * (4 if case["input"] == "host" else 2)
        flops = 2.0 * rows * (patch_in * E + layers * block) + attn + head_flops
        return {"bytes": weights + in_bytes + 2.0 * out_rows * width, "flops": flops}
    grids = _grids(case)
    L = sum(t * h * w for t, h, w in grids)
    frame_pairs = sum(t * float(h * w) ** 2 for t, h, w in grids)          # query-key pairs inside frames
    if kind == "qwen3_vl":
        E, inter, depth, width, patch_in, mergers = 1152, 2 * 4304, 27, 4096, 3 * 2 * 16 * 16, 4
        pairs = depth * frame_pairs
    elif kind == "qwen2_vl":
        E, inter, depth, width, patch_in, mergers = 1280, 2 * 5120, 32, 3584, 1176, 1
        pairs = depth * frame_pairs
    else:
        E, inter, depth, width, patch_in, mergers = 1280, 3 * 3420, 32, 3584, 1176, 1
        pairs = 4 * frame_pairs
        for t, h, w in grids:                                              # 28 blocks attend inside 8 x 8 windows
            sq = lambda n: (n // 8) * 64 + (n % 8) ** 2                    # noqa: E731
            pairs += 28.0 * t * sq(h) * sq(w)
    block = 4 * E * E + E * inter
    merger = (4 * E) ** 2 + 4 * E * width
    weights = (1.0 if kind.endswith("fp8") else 2.0) * (depth * block + mergers * merger) + 2.0 * patch_in * E
    if case["input"] == "photo":
        in_bytes = float(sum(t * h * w * 3 for t, h, w in _items(case)))
    else:
        in_bytes = L * patch_in * (4.0 if case["input"] == "host" else 2.0)
    flops = 2.0 * L * (patch_in * E + depth * block) + 2.0 * (L / 4) * mergers * merger + 4.0 * E * pairs
    return {"bytes": weights + in_bytes + 2.0 * (L / 4) * width * mergers, "flops": flops}


def tolerance(case: dict) -> dict:
    """bf16 activations through 26 to 32 blocks.  Evaluations that differ only in where they round (norms folded into the
    GEMMs or on their own, one launch or three for a window block) are this far apart at most, times about four: relative
    error 1.3e-2 and largest difference 7e-2 with the Qwen families and with LLaVA-OneVision, 5e-3 and 2.3e-2 with SigLIP's
    4096 tokens (3e-2 is the most that is stated for any)."""
    return {"rel": 0.02, "max": 0.1} if case["model"] == "gemma3" else {"rel": 0.03, "max": 0.28}
