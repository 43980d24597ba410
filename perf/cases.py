"""What is timed when the speed of this library is followed: the attention calls, prepared-key calls and whole attention
blocks that a denoising step makes of it, through the public entry points, from one image to the longest clip.

A case is a dict of plain values:

  kind      "attention"  ``attention(q, k, v)``: the K/V pass and the attention kernel, one call
            "prepared"   ``attention_prepared`` of new queries against text keys prepared once (the later denoising steps)
            "block"      ``PikaH3AttnProcessor(fused_projections=True)``: AdaLN -> to_q/to_k/to_v (+ LoRA) -> attention ->
                         to_out.0 (+ LoRA), gate and residual
  frames, rows_h, rows_w, audio, text    a packed document: latent frames x patch grid, audio latents (two channels), text
                         rows; ``frames`` 0: no grid, the call has ``sq`` rows and no rotation unless ``rope`` says otherwise
  sq, sk    query and key rows of calls without a grid (``sk`` 0: self-attention)
  shortest  valid keys of the shortest entry of the batch, the others spread evenly up to ``sk`` (0: no key mask)
  rope      0 none, 1 interleaved pairs, 2 half-split pairs
  fp8       "" bf16, "absmax" or "pow2": fp8 QK^T with that scale rule
  sparse    64 x 64 tile map: two latent frames around plus this share of random tiles (0: dense)
"""
import math
from types import SimpleNamespace

import torch

import pika_h3_flex_amd as pk

D = 128
EPS = 1e-6


def _case(kind, **kw):
    c = dict(kind=kind, batch=1, heads=24, frames=0, rows_h=0, rows_w=0, audio=0, text=0, sq=0, sk=0, shortest=0, rope=0,
             fp8="", sparse=0.0)
    c.update(kw)
    return c


def _named(name, kind, **kw):
    return dict(_case(kind, **kw), name=name)


def listed():
    clip = dict(frames=37, rows_h=15, rows_w=26, audio=200, rope=1)     # 480p, five seconds: 14,830 rows and the prompt
    full = dict(frames=31, rows_h=30, rows_w=52, rope=1)                # 480p benchmark layer: 48,360 rows
    return [
        # one small call with nothing around it: the plumbing configuration, where launches and host time count
        _named("plumbing", "attention", heads=4, sq=1024),
        # a few short sequences padded to one length
        _named("batch-padded", "attention", batch=3, heads=8, sq=777, shortest=300, rope=2),
        # the ordinary document of the default request: prompt, stereo audio and five seconds of video
        _named("clip", "attention", **clip, text=512),
        # the headline layer, and the same with fp8 QK^T
        _named("480p", "attention", **full),
        _named("480p-fp8", "attention", **full, fp8="absmax"),
        # the longest clip at the larger size
        _named("768p", "attention", frames=31, rows_h=48, rows_w=84, rope=1),
        # the block-sparse layer at the headline size, and on an ordinary document in fp8 with power-of-two scales
        _named("480p-sparse", "attention", **full, sparse=0.10),
        _named("clip-sparse-fp8", "attention", **clip, text=77, fp8="pow2", sparse=0.10),
        # text cross-attention of a joint video and audio layer: every step's call, keys prepared in the call
        _named("cross", "attention", sq=49640, sk=512, shortest=302),
        # the later denoising steps of a clip against a long prompt whose keys are already prepared
        _named("cross-prepared", "prepared", sq=14830, sk=2048, shortest=1531),
        # the attention half of a block: a single image (one latent frame and a short prompt), and the ordinary clip
        _named("block-image", "block", frames=1, rows_h=24, rows_w=42, text=77, rope=1),
        _named("block-clip", "block", **clip, text=512),
    ]


_LARGEST = 4.0 * 124992.0 ** 2 * D * 24     # attention operations of the largest listed case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_document(rng, most):
    """A packed document of at most ``most`` rows: grids of the resolution tiers and their aspect ratios."""
    while True:
        rows_h, rows_w = rng.choice([(15, 26), (26, 15), (20, 20), (17, 23), (24, 42), (42, 24), (30, 52), (32, 32), (48, 84)])
        frames = _log(rng, 1, 107)
        audio = rng.choice([0, _log(rng, 5, 640)])
        text = rng.choice([0, rng.randint(1, 77), _log(rng, 77, 2048)])
        if 256 <= frames * rows_h * rows_w + 2 * audio + text <= most:
            return dict(frames=frames, rows_h=rows_h, rows_w=rows_w, audio=audio, text=text)


def draw(rng):
    which = rng.choice(["small", "small", "dense", "dense", "sparse", "cross", "prepared", "block"])
    if which == "small":
        batch, sq = rng.randint(1, 4), _log(rng, 64, 3000)
        masked = rng.random() < 0.5
        return _case("attention", batch=batch, heads=rng.choice([1, 2, 3, 4, 8, 16, 24]), sq=sq,
                     shortest=rng.randint(1, sq) if masked else 0, rope=rng.choice([0, 1, 2]),
                     fp8="" if masked else rng.choice(["", "", "absmax", "pow2"]))
    if which == "dense":
        return _case("attention", **_draw_document(rng, 120000), rope=rng.choice([1, 1, 2]), fp8=rng.choice(["", "", "absmax", "pow2"]))
    if which == "sparse":
        return _case("attention", **_draw_document(rng, 60000), rope=1, fp8=rng.choice(["", "absmax", "pow2"]),
                     sparse=rng.choice([0.05, 0.10, 0.20]))
    if which in ("cross", "prepared"):
        sk = rng.choice([rng.randint(16, 256), 512, rng.randint(256, 2048)])
        return _case("attention" if which == "cross" else "prepared", batch=rng.choice([1, 1, 2]), sq=_log(rng, 256, 60000), sk=sk,
                     shortest=rng.choice([0, rng.randint(min(16, sk), sk)]))
    return _case("block", **_draw_document(rng, 50000), rope=1, fp8=rng.choice(["", "", "absmax", "pow2"]),
                 sparse=rng.choice([0.0, 0.0, 0.0, 0.10]))


# ---------------------------------------------------------------------------------------------------------------------
def _layout(case):
    return pk.packing.build_layout(num_text_tokens=case["text"], num_latent_frames=case["frames"], latent_height=2 * case["rows_h"],
                                   latent_width=2 * case["rows_w"], num_audio_latents=case["audio"])


def _sizes(case):
    sq = (case["frames"] * case["rows_h"] * case["rows_w"] + 2 * case["audio"] + case["text"]) if case["frames"] else case["sq"]
    return sq, case["sk"] or sq


def _valid(case):
    """Valid keys of every entry of the batch."""
    _, sk = _sizes(case)
    n, b = case["shortest"] or sk, case["batch"]
    return [n + (sk - n) * i // max(1, b - 1) for i in range(b)]


_kept = {}   # kept tiles of a map, by what it depends on: work() asks for no more than the count


def _tile_map(case):
    lay = _layout(case)
    return pk.packing.packed_window_tile_map(lay, window_frames=2, global_fraction=case["sparse"], seed=0)


def _attended(case):
    """(query, key) pairs of one head."""
    sq, sk = _sizes(case)
    if not case["sparse"]:
        return sq * sum(_valid(case))
    key = tuple(case[k] for k in ("frames", "rows_h", "rows_w", "audio", "text", "sparse"))
    if key not in _kept:
        rows = torch.full((-(-sq // 64),), 64, dtype=torch.int64)
        rows[-1] = sq - 64 * (len(rows) - 1)
        m = _tile_map(case).to(torch.int64)
        _kept[key] = int((rows[:, None] * m * rows[None, :]).sum())
    return _kept[key]


def _rows(shape, gen, std=1.0):
    """Normal values in bf16, as a projection of normalised hidden states leaves them."""
    out = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        part = flat[i:i + (1 << 28)]
        part.copy_(torch.randn(part.shape, generator=gen, device="cuda").mul_(std))
    return out


def _norm_weight(gen):
    return 1.0 + 0.1 * torch.randn((D,), generator=gen, device="cuda")


class _LoraLinear:
    """A linear layer with one rank-128 adapter beside it, in the form adapters are injected in."""

    def __init__(self, n, k, gen):
        self.base_layer = torch.nn.Linear(k, n, device="cuda", dtype=torch.bfloat16)
        self.lora_A = {"default": torch.nn.Linear(k, 128, bias=False, device="cuda", dtype=torch.bfloat16)}
        self.lora_B = {"default": torch.nn.Linear(128, n, bias=False, device="cuda", dtype=torch.bfloat16)}
        self.scaling = {"default": 0.5}
        with torch.no_grad():
            for lin in (self.base_layer, self.lora_A["default"], self.lora_B["default"]):
                lin.weight.copy_(_rows(tuple(lin.weight.shape), gen, 0.02))
            self.base_layer.bias.copy_(_rows((n,), gen, 0.02))


def _prepare_block(case, gen):
    S, _ = _sizes(case)
    H = case["heads"]
    C = H * D
    attn = SimpleNamespace(heads=H, to_q=_LoraLinear(C, C, gen), to_k=_LoraLinear(C, C, gen), to_v=_LoraLinear(C, C, gen),
                           to_out=[_LoraLinear(C, C, gen)],
                           norm_q=SimpleNamespace(weight=_norm_weight(gen), eps=EPS), norm_k=SimpleNamespace(weight=_norm_weight(gen), eps=EPS))
    proc = pk.PikaH3AttnProcessor(fused_projections=True, rope_mode=case["rope"], fp8_qk=_fp8(case))
    proc.packed_weights(attn)
    x = _rows((1, S, C), gen)
    shift, scale, gate = (_rows((3, C), gen, 0.2) for _ in range(3))    # three timestep groups
    index = (torch.arange(S, device="cuda") * 3 // S).to(torch.int32)
    call = dict(position_ids=_layout(case).position_ids.to("cuda"), rope_key="document", gate=gate, gate_index=index, residual=x,
                adaln=dict(shift=shift, scale=scale, row_index=index, norm="layer", eps=EPS))
    if case["sparse"]:
        call["block_mask"] = pk.BlockMask.from_dense(_tile_map(case), device="cuda")
    return SimpleNamespace(kind="block", proc=proc, attn=attn, x=x, call=call)


def _fp8(case):
    return {"": False, "absmax": True, "pow2": "pow2"}[case["fp8"]]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    if case["kind"] == "block":
        return _prepare_block(case, gen)
    sq, sk = _sizes(case)
    B, H = case["batch"], case["heads"]
    q = _rows((B, sq, H * D), gen, 1.1).view(B, sq, H, D)     # hidden states N(0, 1) through weights of spread 0.02: spread 1.1
    k = _rows((B, sk, H * D), gen, 1.1).view(B, sk, H, D)
    v = _rows((B, sk, H * D), gen, 1.1).view(B, sk, H, D)
    q_opts = dict(q_norm_weight=_norm_weight(gen))
    k_opts = dict(k_norm_weight=_norm_weight(gen), norm_eps=EPS, fp8_qk=_fp8(case))
    if case["rope"]:
        if case["frames"]:
            pos = _layout(case).position_ids.to("cuda")
        else:
            pos = pk.video_position_ids(sq, 1, 1).to("cuda")
        tables = pk.rope_tables(pos)
        q_opts.update(rope_q=tables)
        k_opts.update(rope_mode=case["rope"], rope_k=tables)
    if case["shortest"]:
        valid = torch.tensor(_valid(case), device="cuda")
        k_opts.update(key_mask=torch.arange(sk, device="cuda")[None, :] < valid[:, None])
    if case["kind"] == "prepared":
        return SimpleNamespace(kind="prepared", q=q, kv=pk.prepare_kv(k, v, **k_opts), opts=q_opts)
    opts = dict(q_opts, **k_opts)
    if case["sparse"]:
        opts.update(block_mask=pk.BlockMask.from_dense(_tile_map(case), device="cuda"))
    return SimpleNamespace(kind="attention", q=q, k=k, v=v, opts=opts)


@torch.no_grad()
def run(state):
    if state.kind == "block":
        return state.proc(state.attn, state.x, **state.call)
    if state.kind == "prepared":
        return pk.attention_prepared(state.q, state.kv, **state.opts)
    return pk.attention(state.q, state.k, state.v, **state.opts)


def work(case):
    sq, sk = _sizes(case)
    B, H = case["batch"], case["heads"]
    C = H * D
    flops = 4.0 * _attended(case) * D * H
    if case["kind"] == "block":
        # hidden states in (the residual is the same rows), result out; four weight matrices with their adapters
        weights = 4 * (C * C + 2 * C * 128)
        return {"bytes": 2.0 * (2 * sq * C + weights) + 8.0 * sq * (D // 2),
                "flops": flops + 2.0 * sq * weights}
    keys = sum(_valid(case))
    bytes_ = 2.0 * C * (2 * B * sq + 2 * keys)
    if case["rope"]:
        bytes_ += 8.0 * (D // 2) * sq
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Four times the distance of the outputs from the same path in float64 (attention in bf16: 3.3e-3, largest single
    difference 2.2e-2; with fp8 operands, against the quantised operands in float64: 2.4e-3 and 1.8e-2; a block, whose
    result is dominated by the residual: 1.6e-3 and 5.5e-3)."""
    if case["kind"] == "block":
        return {"rel": 6.5e-3, "max": 2.2e-2}
    return {"rel": 1e-2, "max": 7.5e-2} if case["fp8"] else {"rel": 1.3e-2, "max": 9e-2}
