"""GPU parity of the projection entry points (pkh3_pack_*, pkh3_adaln_modulate, pkh3_qkv_proj, pkh3_out_proj)
against the float64 oracle (oracle/projection_oracle.py), through the C ABI.

bf16 bar of the path: max-abs <= 2e-2 and cosine >= 0.9999 against float64 on tensors of unit scale; the fp8 /
block-sparse attention variants keep their cosine >= 0.995 bar.  The operand-image layout is checked against its
documented index formula, written out here independently of the kernels."""
import pytest
import torch

from tests import test_attention_forms as forms

pytestmark = pytest.mark.gpu

D = 128


def _r(*shape, seed=0, std=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std


def _unpack(buf, rows, K):
    """Operand images -> matrix: image (rb, ks) holds rows 16*rb..+15; lane 16*g + c carries elements
    32*ks + 8*g + 0..7 of row 16*rb + c."""
    img = buf.view(torch.bfloat16).view(-1, K // 32, 4, 16, 8)      # [rb, ks, g, c, j]
    return img.permute(0, 3, 1, 2, 4).reshape(-1, K)[:rows]


def _head_perm_source(rho):
    """Source row (inside its 128-row head) of image row ``rho``: 16*fb + 4*g + i <- 32*(fb//2) + 8*g + 4*(fb%2) + i."""
    fb, g, i = rho // 16, (rho // 4) % 4, rho % 4
    return 32 * (fb // 2) + 8 * g + 4 * (fb % 2) + i


def test_pack_layout_matches_its_index_formula():
    from pika_h3_flex_amd import projections as P

    x = _r(70, 96, seed=1).to(torch.bfloat16).cuda()
    buf = P.pack_rows(x)
    assert buf.numel() == 256 * 96 * 2                                # rows padded to 256
    torch.cuda.synchronize()
    full = _unpack(buf, 256, 96)
    assert torch.equal(full[:70].cpu(), x.cpu()) and float(full[70:].float().abs().sum()) == 0.0
    # a strided source (a column slice of a wider matrix)
    wide = _r(40, 200, seed=2).to(torch.bfloat16).cuda()
    assert torch.equal(_unpack(P.pack_rows(wide[:, 8:104]), 40, 96).cpu(), wide[:, 8:104].cpu())
    # weights: identity order for a V projection, permuted inside every 128-row head otherwise
    w = _r(256, 64, seed=3).to(torch.bfloat16).cuda()
    assert torch.equal(_unpack(P.pack_weight(w, head_perm=False), 256, 64).cpu(), w.cpu())
    got = _unpack(P.pack_weight(w, head_perm=True), 256, 64).cpu()
    src = torch.tensor([128 * (r // 128) + _head_perm_source(r % 128) for r in range(256)])
    assert sorted(src.tolist()) == list(range(256))                   # a permutation
    assert torch.equal(got, w.cpu()[src])


@pytest.mark.parametrize("norm", ["layer", "rms"])
def test_adaln_modulate_matches_oracle(norm):
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    S, K, T = 333, 3072, 4
    x = (_r(S, K, seed=4) * 2 + 0.3).to(torch.bfloat16)
    shift, scale = _r(T, K, seed=5, std=0.3).to(torch.bfloat16), _r(T, K, seed=6, std=0.3).to(torch.bfloat16)
    idx = torch.randint(0, T, (S,), generator=torch.Generator().manual_seed(7)).to(torch.int32)
    img = P.adaln_modulate(x.cuda(), shift=shift.cuda(), scale=scale.cuda(), row_index=idx.cuda(), norm=norm)
    torch.cuda.synchronize()
    got = _unpack(img, S, K).cpu()
    ref = PO.adaln_modulate(x, shift=shift, scale=scale, row_index=idx, norm=norm)
    err, cos = AO.max_abs_and_cosine(got, ref)
    print(f"adaln {norm}: max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert cos >= 0.99999 and float(((got.double() - ref).abs() / (ref.abs() + 1.0)).max()) <= 2.0 ** -8   # one bf16 rounding
    # without tables: the bare norm; without an index: table row 0
    bare = _unpack(P.adaln_modulate(x.cuda(), norm=norm), S, K).cpu()
    assert AO.max_abs_and_cosine(bare, PO.adaln_modulate(x, norm=norm))[1] >= 0.99999
    row0 = _unpack(P.adaln_modulate(x.cuda(), shift=shift.cuda(), scale=scale.cuda(), norm=norm), S, K).cpu()
    assert AO.max_abs_and_cosine(row0, PO.adaln_modulate(x, shift=shift, scale=scale, norm=norm))[1] >= 0.99999


@pytest.mark.parametrize("norm", ["layer", "rms"])
@pytest.mark.parametrize("S,K", [(1, 32), (16, 512), (9, 544), (17, 1024), (24, 1056), (40, 1536), (23, 1568), (8, 2048), (31, 2080), (33, 2560), (15, 2592),
                                 (48, 3104), (7, 3584), (25, 3616), (64, 4064), (39, 4096)])
def test_adaln_modulate_of_every_row_length(S, K, norm):
    """A wave holds one to eight pieces a lane, the last of them partly or wholly there; rows up to the next 16 are zeros.  Either table
    may be missing.  One bf16 rounding of the value (2^-9 of it) and float32 statistics: 2^-8 covers both."""
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    x = (_r(S, K, seed=21) * 2 + 0.3).to(torch.bfloat16)
    tables = dict(shift=_r(3, K, seed=22, std=0.3).to(torch.bfloat16), scale=_r(3, K, seed=23, std=0.3).to(torch.bfloat16))
    idx = torch.arange(S).remainder(3).to(torch.int32)
    padded = -(-S // 16) * 16
    for names in ((), ("shift",), ("scale",), ("shift", "scale")):
        opts = {n: tables[n] for n in names}
        img = P.adaln_modulate(x.cuda(), **{n: t.cuda() for n, t in opts.items()}, **(dict(row_index=idx.cuda()) if names else {}), norm=norm)
        got = _unpack(img, padded, K).cpu()
        ref = PO.adaln_modulate(x, **opts, **(dict(row_index=idx) if names else {}), norm=norm)
        assert float(((got[:S].double() - ref).abs() / (ref.abs() + 1.0)).max()) <= 2.0 ** -8
        assert torch.count_nonzero(got[S:]) == 0


def test_adaln_layer_norm_of_rows_with_a_large_common_offset():
    """Rows whose mean is large against their spread (massive-activation channels): the variance must come from the
    distances to the mean, not from E[x^2] - mean^2, which cancels in float32.  x = 0.25 * randn + 50 (bf16 grid step
    0.25 at 50, so the spread is a few grid steps).  Also a constant row with eps = 0: zeros, not NaN."""
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    S, K = 200, 3072
    x = (_r(S, K, seed=14) * 0.25 + 50.0).to(torch.bfloat16)
    img = P.adaln_modulate(x.cuda(), norm="layer", eps=1e-6)
    torch.cuda.synchronize()
    got = _unpack(img, S, K).cpu()
    ref = PO.adaln_modulate(x, norm="layer", eps=1e-6)
    err, cos = AO.max_abs_and_cosine(got, ref)
    print(f"adaln layer norm, offset rows: max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert cos >= 0.99999 and float(((got.double() - ref).abs() / (ref.abs() + 1.0)).max()) <= 2.0 ** -8
    const = torch.full((16, K), 3.0, dtype=torch.bfloat16)
    out = _unpack(P.adaln_modulate(const.cuda(), norm="layer", eps=0.0), 16, K).cpu()
    assert torch.count_nonzero(out) == 0 and torch.isfinite(out.float()).all()


def _linear(n, k, seed, lora=True, bias=True):
    d = dict(weight=_r(n, k, seed=seed, std=k ** -0.5).to(torch.bfloat16))
    if bias:
        d["bias"] = _r(n, seed=seed + 1, std=0.1)
    if lora:
        d.update(lora_a=_r(128, k, seed=seed + 2, std=k ** -0.5).to(torch.bfloat16),
                 lora_b=_r(n, 128, seed=seed + 3, std=0.05).to(torch.bfloat16), lora_scale=0.5)
    return d


def _packed(d, head_perm=True):
    from pika_h3_flex_amd.projections import PackedLinear

    return PackedLinear.from_weights(d["weight"].cuda(), d["bias"].cuda() if "bias" in d else None,
                                     lora_a=d["lora_a"].cuda() if "lora_a" in d else None,
                                     lora_b=d["lora_b"].cuda() if "lora_b" in d else None,
                                     lora_scale=d.get("lora_scale", 1.0), head_perm=head_perm)


@pytest.mark.parametrize("S,H,variant", [
    (300, 2, "bf16"), (777, 3, "bf16"), (64, 1, "bf16"), (1000, 2, "no_lora"), (520, 2, "fp8"), (700, 2, "sparse"),
    (450, 3, "rope_half"), (520, 2, "fp8_pow2"),
])
def test_qkv_projection_feeds_attention(S, H, variant):
    """to_q/to_k/to_v (+LoRA, bias) with the K-side norm + rotation and the K/V layout in the GEMM epilogue, then the
    attention kernel on the prepared workspace: Q against lora_linear, O against the oracle's composition."""
    import pika_h3_flex_amd as pk
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    C = H * D
    lora = variant != "no_lora"
    x = _r(S, C, seed=10).to(torch.bfloat16)
    lin = {n: _linear(C, C, 20 + 10 * i, lora=lora, bias=(n != "k")) for i, n in enumerate(("q", "k", "v"))}
    wq, wk = 1.0 + 0.1 * _r(D, seed=50), 1.0 + 0.1 * _r(D, seed=51)
    pos = torch.cat([pk.video_position_ids(1, 1, S - 20), pk.audio_position_ids(10)], 0)
    mode = pk.ROPE_HALF if variant == "rope_half" else pk.ROPE_INTERLEAVED
    opts = dict(q_norm_weight=wq.cuda(), k_norm_weight=wk.cuda(), rope_mode=mode, rope_q=pk.rope_tables(pos.cuda()))
    ref_opts = dict(q_norm_weight=wq, k_norm_weight=wk, rope_mode=mode, rope_q=AO.rope_tables(pos))
    if variant == "fp8":
        opts.update(fp8_qk=True)
        ref_opts.update(fp8_qk=True)
    if variant == "fp8_pow2":   # the K epilogue of the GEMM forms the power-of-two scales
        opts.update(fp8_qk="pow2")
        ref_opts.update(fp8_qk="pow2")
    if variant == "sparse":
        n = (S + 63) // 64
        tm = (torch.rand((n, n), generator=torch.Generator().manual_seed(3)) < 0.5) | torch.eye(n, dtype=torch.bool)
        opts.update(block_mask=pk.BlockMask.from_dense(tm, device="cuda"))
        ref_opts.update(tile_map=tm)
    out, q = P.qkv_attention(P.pack_rows(x.cuda()), S, _packed(lin["q"]), _packed(lin["k"]), _packed(lin["v"], head_perm=False),
                             heads=H, return_q=True, **opts)
    torch.cuda.synchronize()
    q_ref = PO.lora_linear(x, **lin["q"]).view(1, S, H, D)
    err, cos = AO.max_abs_and_cosine(q.cpu(), q_ref)
    print(f"[{variant} S={S} H={H}] Q: max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert err <= 2e-2 and cos >= 0.9999
    # attention on bf16-rounded Q, K, V (what the product stores between its kernels; K is rounded after norm+rope
    # inside the epilogue instead, which the bf16 bar absorbs)
    r = lambda t: t.to(torch.bfloat16)
    k_ref, v_ref = (PO.lora_linear(x, **lin[n]).view(1, S, H, D) for n in ("k", "v"))
    o_ref = AO.reference_layer(r(q_ref), r(k_ref), r(v_ref), **ref_opts)
    err, cos = AO.max_abs_and_cosine(out.cpu(), o_ref)
    print(f"[{variant} S={S} H={H}] O: max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert torch.isfinite(out.float()).all()
    if variant.startswith("fp8"):
        assert cos >= 0.995
    else:
        assert err <= 2e-2 and cos >= 0.9999
    # and against the unfused route on the same Q, K, V (torch GEMM -> K/V pass -> same attention kernel)
    unfused = pk.attention(r(q_ref).cuda(), r(k_ref).cuda(), r(v_ref).cuda(), **opts)
    torch.cuda.synchronize()
    err, cos = AO.max_abs_and_cosine(out.cpu(), unfused.cpu())
    assert cos >= (0.995 if variant.startswith("fp8") else 0.9999)


@pytest.mark.parametrize("S,N,K,lora,extras", [(300, 256, 256, True, True), (1000, 384, 256, False, True), (65, 128, 512, True, False),
                                                 # the ring of four slots: even and odd numbers of chunks, a last token alone in its tile
                                                 (129, 3072, 1536, False, True), (130, 2944, 1568, True, False), (705, 1152, 1600, True, True)])
def test_out_projection_with_gate_and_residual(S, N, K, lora, extras):
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    o = _r(S, K, seed=60).to(torch.bfloat16)
    lin = _linear(N, K, 61, lora=lora)
    T = 3
    gate = _r(T, N, seed=70, std=0.5).to(torch.bfloat16)
    idx = torch.randint(0, T, (S,), generator=torch.Generator().manual_seed(71)).to(torch.int32)
    res = _r(S, N, seed=72).to(torch.bfloat16)
    kw = dict(gate=gate.cuda(), row_index=idx.cuda(), residual=res.cuda()) if extras else {}
    y = P.out_proj(o.cuda(), _packed(lin), **kw)
    torch.cuda.synchronize()
    ref = PO.lora_linear(o, **lin)
    if extras:
        ref = res.double() + gate.double()[idx.long()] * ref
    err, cos = AO.max_abs_and_cosine(y.cpu(), ref)
    print(f"out_proj S={S} N={N} K={K} lora={lora}: max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert err <= 2e-2 * max(1.0, float(ref.abs().max())) and cos >= 0.9999


# The GEMM's four workgroup heights (64, 128, 192, 256 tokens; chosen by tokens x feature tiles) on both sides of their edges,
# an odd number of k-chunks (K = 96 + the adapter's 128) and an even one.
@pytest.mark.parametrize("S,H,K,fp8,mode", [
    (31, 1, 96, False, 1), (129, 2, 128, True, 2), (449, 3, 96, True, 1),          # 64 tokens
    (3585, 24, 96, False, 1), (3713, 24, 128, True, 2), (3600, 23, 96, "pow2", 1),  # 128 tokens
    (1025, 24, 96, False, 2), (1279, 24, 128, True, 1), (1088, 23, 96, False, 0),   # 192 tokens
    (1153, 24, 96, True, 1), (1121, 23, 128, "pow2", 2), (1152, 24, 128, False, 1),   # (key tiles of one wave and shared by two)
    (1345, 24, 96, False, 2), (1536, 24, 128, True, 1), (1409, 23, 96, "pow2", 0),   # 256 tokens
])
def test_gemm_forms_of_the_qkv_projection(S, H, K, fp8, mode):
    """Q against float32 torch, and the attention output against the same kernel fed with torch's K and V through the
    separate K/V pass: every token and head, so a wrong 16-token block of any epilogue shows."""
    import pika_h3_flex_amd as pk
    from oracle import attention_oracle as AO
    from pika_h3_flex_amd import projections as P

    x = _r(S, K, seed=1).to(torch.bfloat16).cuda()
    lin = {n: _linear(H * D, K, 20 + 10 * i, bias=(n != "k")) for i, n in enumerate(("q", "k", "v"))}
    opts = dict(q_norm_weight=(1 + 0.1 * _r(D, seed=2)).cuda(), k_norm_weight=(1 + 0.1 * _r(D, seed=3)).cuda(), fp8_qk=fp8)
    if mode:
        opts.update(rope_mode=mode, rope_q=pk.rope_tables(pk.video_position_ids(1, 1, S).cuda()))
    out, q = P.qkv_attention(P.pack_rows(x), S, _packed(lin["q"]), _packed(lin["k"]), _packed(lin["v"], head_perm=False),
                             heads=H, return_q=True, **opts)

    def layer(d):
        y = x.float() @ d["weight"].cuda().float().t() + d["lora_scale"] * (x.float() @ d["lora_a"].cuda().float().t()) @ d["lora_b"].cuda().float().t()
        return (y + d["bias"].cuda() if "bias" in d else y).view(1, S, H, D)

    ref = {n: layer(d) for n, d in lin.items()}
    want = pk.attention(*(ref[n].to(torch.bfloat16) for n in ("q", "k", "v")), **opts)
    torch.cuda.synchronize()
    err, cos = AO.max_abs_and_cosine(q.cpu(), ref["q"].cpu())
    # per row and head: bf16 rounding of Q, K, V and P moves a row's direction by less than 1e-3 (fp8: another K rounding
    # flips e4m3 steps, relative 2^-4 each, on a share of the 128 products)
    rows = torch.nn.functional.cosine_similarity(out.float(), want.float(), dim=-1).min().item()
    print(f"S={S} H={H} K={K} fp8={fp8} mode={mode}: Q max_abs={err:.3e} cos={cos:.8f}; O worst row cos={rows:.6f}", flush=True)
    assert err <= 2e-2 * max(1.0, float(ref["q"].abs().max())) and cos >= 0.9999
    assert rows >= (0.99 if fp8 else 0.999)


@pytest.mark.parametrize("S,H,variant", [(1, 1, "dense"), (31, 3, "dense"), (129, 2, "dense"), (449, 3, "dense"), (129, 2, "fp8"),
                                         (31, 32, "sparse"), (31, 2, "sparse"), (257, 32, "sparse"), (449, 2, "sparse_pow2"),
                                         (641, 24, "dense"), (3585, 24, "dense"), (1025, 24, "sparse"), (1089, 24, "dense"),
                                         (1345, 24, "sparse")])
def test_qkv_projection_writes_whole_key_tiles(S, H, variant):
    """S % 64 in 1 .. 32: the second half of the last K/V record holds no key.  The kernels that walk whole 64-key tiles still
    multiply its V images (by probabilities of 0), so the projection has to write it whatever the workspace held before: here
    NaN in every byte pair.  All workgroup heights of the GEMM; the long-key and the 8-wave block-sparse kernels."""
    import pika_h3_flex_amd as pk
    from pika_h3_flex_amd import projections as P

    K = 96
    x = _r(S, K, seed=1).to(torch.bfloat16).cuda()
    packed = [_packed(_linear(H * D, K, 20 + 10 * i, bias=False), head_perm=i < 2) for i in range(3)]
    opts = dict(q_norm_weight=torch.ones(D).cuda(), k_norm_weight=torch.ones(D).cuda(), long_key_kernel=True)
    if variant.startswith("sparse"):
        n = (S + 63) // 64
        keep = (torch.rand((n, n), generator=torch.Generator().manual_seed(2)) < 0.5) | torch.eye(n, dtype=torch.bool)
        keep[:, n - 1] = True
        opts["block_mask"] = pk.BlockMask.from_dense(keep, device="cuda")
    opts["fp8_qk"] = {"fp8": True, "sparse_pow2": "pow2"}.get(variant, False)
    outs = []
    for fill in (0x00, 0xFF):
        made = []

        def workspace(device, nbytes):
            made.append(torch.full((nbytes,), fill, dtype=torch.uint8, device=device))
            return made[0]

        outs.append(P.qkv_attention(P.pack_rows(x), S, *packed, heads=H, workspace=workspace, **opts))
    torch.cuda.synchronize()
    print(f"S={S} H={H} {variant}: {int(torch.isnan(outs[1].float()).sum())} NaN", flush=True)
    assert torch.isfinite(outs[1].float()).all() and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("S,N", [(65, 256), (1471, 3072), (1537, 2944), (3583, 3072), (3649, 2944), (2881, 3072), (3263, 2944)])
@pytest.mark.parametrize("gate,residual", [(True, True), (True, False), (False, True), (False, False)])
def test_gemm_forms_of_the_out_projection(S, N, gate, residual):
    """The four workgroup heights of the row-major epilogue with each of its four combinations, every row."""
    from pika_h3_flex_amd import projections as P

    K = 96
    o = _r(S, K, seed=5).to(torch.bfloat16).cuda()
    lin = _linear(N, K, 6)
    g = _r(3, N, seed=7, std=0.5).to(torch.bfloat16).cuda()
    idx = (torch.arange(S) * 3 // S).to(torch.int32).cuda()
    res = _r(S, N, seed=8).to(torch.bfloat16).cuda()
    y = P.out_proj(o, _packed(lin), **(dict(gate=g, row_index=idx) if gate else {}), **(dict(residual=res) if residual else {}))
    w = {n: t.cuda().float() for n, t in lin.items() if torch.is_tensor(t)}
    ref = o.float() @ w["weight"].t() + w["bias"] + lin["lora_scale"] * (o.float() @ w["lora_a"].t()) @ w["lora_b"].t()
    if gate:
        ref = ref * g.float()[idx.long()]
    if residual:
        ref = ref + res.float()
    torch.cuda.synchronize()
    # one bf16 rounding of the result (at most 2^-8 of its size), and that of the 128 down-projected values (size 0.5,
    # rounding 2^-9 of it each, through weights of 0.05 and a gate of at most 2.5: spread 8e-4, times six)
    err = (y.float() - ref).abs()
    print(f"out_proj S={S} N={N} gate={gate} residual={residual}: max_abs={err.max().item():.3e}", flush=True)
    assert bool((err <= ref.abs() / 256 + 5e-3).all())


@pytest.mark.parametrize("S,K", [(1, 32), (31, 96), (33, 256), (65, 288), (300, 2080), (1085, 3072), (12289, 64)])
def test_forms_of_the_down_projection(S, K):
    """The adapter's path alone (the layer's own weight is zero): fewer k-chunks than the eight waves that share them, shares of
    unequal length, shares that are not whole groups of four, a lone row; the last case takes the large-call form."""
    from pika_h3_flex_amd import projections as P

    o = _r(S, K, seed=11).to(torch.bfloat16).cuda()
    lin = _linear(128, K, 12, bias=False)
    lin["weight"] = torch.zeros_like(lin["weight"])
    y = P.out_proj(o, _packed(lin))
    xa = lin["lora_scale"] * (o.float() @ lin["lora_a"].cuda().float().t())
    b = lin["lora_b"].cuda().float()
    ref = xa @ b.t()
    torch.cuda.synchronize()
    # the bf16 rounding of the result (2^-8 of its size at most) and of the 128 down-projected values, at most 2^-8 of each:
    # six times the spread of their sum
    bound = ref.abs() / 256 + 6.0 / 256 * ((xa * xa) @ (b * b).t()).sqrt()
    err = (y.float() - ref).abs()
    print(f"down-projection S={S} K={K}: worst {(err / bound).max().item():.3f} of the bound", flush=True)
    assert bool((err <= bound).all())


@pytest.mark.parametrize("S", [1, 17, 40, 300, 12290])
def test_down_projected_rows_past_the_end_are_zero(S):
    """Image rows past S are unwritten memory when the attention kernel left the activations (here NaN): the down-projected rows
    they give are zeros all the same, in the thin and in the large-call form (the last size)."""
    import ctypes as C

    from pika_h3_flex_amd import _lib
    from pika_h3_flex_amd import projections as P

    K = 96
    lin = _packed(_linear(128, K, 12))
    img = P.pack_rows(_r(S, K, seed=11).to(torch.bfloat16).cuda())
    cells = img.view(torch.bfloat16).view(-1, K // 32, 4, 16, 8)               # [16-row block, k-step, g, row, j]
    rows = torch.arange(cells.shape[0] * 16, device="cuda").view(-1, 1, 1, 16, 1)
    cells.masked_fill_(rows >= S, float("nan"))
    scratch = torch.full((P.packed_bytes(S, 128),), 0xFF, dtype=torch.uint8, device="cuda")
    y = torch.empty((S, 128), dtype=torch.bfloat16, device="cuda")
    a = _lib.OutArgs()
    a.o_img, a.S, a.K, a.N = img.data_ptr(), S, K, 128
    a.proj = lin.c_struct()
    a.y, a.y_stride = y.data_ptr(), 128
    a.lora_workspace, a.lora_workspace_bytes = scratch.data_ptr(), scratch.numel()
    _lib.check(_lib.load().pkh3_out_proj(C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert torch.isfinite(y.float()).all()
    tail = _unpack(scratch, (S + 15) // 16 * 16, 128)[S:]
    assert torch.count_nonzero(tail) == 0 and torch.isfinite(tail.float()).all()


@pytest.mark.parametrize("S,adapters", [(16640, "shared"), (16449, "shared"), (11008, "separate"), (33280, "out")])
def test_down_projections_of_192_token_tiles_stay_in_their_workspace(S, adapters):
    """Calls whose down-projections take tiles of 192 tokens on 256 CUs, the last one past the padded rows of the workspace (but for
    16,449 rows): what lies behind it is left alone, and the adapters' results are right to the last row."""
    import ctypes as C

    from pika_h3_flex_amd import _lib, ops
    from pika_h3_flex_amd import projections as P

    K, n = 64, 1 if adapters == "out" else 3
    lins = [dict(_linear(128, K, 12 + 10 * i, bias=False), lora_scale=0.5) for i in range(n)]
    for d in lins:
        d["weight"] = torch.zeros_like(d["weight"])                            # the adapters alone
    packed = [_packed(d, head_perm=i < 2) for i, d in enumerate(lins)]
    assert adapters != "shared" or P.PackedLinear.share_adapter_buffer(*packed)
    x = _r(S, K, seed=11).to(torch.bfloat16).cuda()
    img = P.pack_rows(x)
    need, guard = P.packed_bytes(S, 128 * n), 256 * 1024
    around = torch.full((need + 2 * guard,), 0xA5, dtype=torch.uint8, device="cuda")
    lws = around[guard:guard + need]
    y = torch.empty((1, S, 1, D), dtype=torch.bfloat16, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if n == 1:
        a = _lib.OutArgs()
        a.o_img, a.S, a.K, a.N = img.data_ptr(), S, K, 128
        a.proj = packed[0].c_struct()
        a.y, a.y_stride = y.data_ptr(), 128
        a.lora_workspace, a.lora_workspace_bytes = lws.data_ptr(), need
        _lib.check(_lib.load().pkh3_out_proj(C.byref(a), stream))
    else:
        args, keep = ops.fill_args(y, None, None, torch.empty_like(y), kv_prepared=True)
        ws = torch.empty(ops.workspace_bytes(args), dtype=torch.uint8, device="cuda")
        args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
        a = _lib.QkvArgs()
        a.x_img, a.S, a.K = img.data_ptr(), S, K
        a.q, a.k, a.v = (p.c_struct() for p in packed)
        a.lora_workspace, a.lora_workspace_bytes = lws.data_ptr(), need
        _lib.check(_lib.load().pkh3_qkv_proj(C.byref(a), C.byref(args), stream))
    torch.cuda.synchronize()
    assert bool((around[:guard] == 0xA5).all()) and bool((around[guard + need:] == 0xA5).all())
    rows = _unpack(lws, (S + 15) // 16 * 16, 128 * n).view(-1, n, 128)
    assert torch.count_nonzero(rows[S:]) == 0
    for i, d in enumerate(lins):
        xa = d["lora_scale"] * (x.float() @ d["lora_a"].cuda().float().t())
        # one rounding to bf16 (at most 2^-8 of the value) of a sum of 64 products in float32
        assert bool(((rows[:S, i].float() - xa).abs() <= xa.abs() / 256 + 1e-5).all())
    b = lins[0]["lora_b"].cuda().float()
    xa = lins[0]["lora_scale"] * (x.float() @ lins[0]["lora_a"].cuda().float().t())
    # (as in test_forms_of_the_down_projection)
    bound = (xa @ b.t()).abs() / 256 + 6.0 / 256 * ((xa * xa) @ (b * b).t()).sqrt()
    assert bool(((y.view(S, 128).float() - xa @ b.t()).abs() <= bound).all())


@pytest.mark.parametrize("S,H", [(300, 2), (1000, 3), (257, 1)])
def test_adapters_in_one_buffer_give_the_same_bits(S, H):
    """``PackedLinear.share_adapter_buffer`` lays the three down-projection images one behind the other, and
    ``pkh3_qkv_proj`` then runs them as one three-head target: the same products in the same order, so Q and the
    attention output carry the bits of the call with separate buffers.  Layers with different scales, or one without
    an adapter, are left alone."""
    import pika_h3_flex_amd as pk
    from pika_h3_flex_amd import projections as P

    C = H * D
    x = _r(S, C, seed=90).to(torch.bfloat16)
    lin = {n: _linear(C, C, 91 + 10 * i, lora=True, bias=True) for i, n in enumerate(("q", "k", "v"))}
    pos = pk.video_position_ids(1, 1, S)
    opts = dict(q_norm_weight=torch.ones(D).cuda(), k_norm_weight=torch.ones(D).cuda(), rope_mode=pk.ROPE_INTERLEAVED,
                rope_q=pk.rope_tables(pos.cuda()))
    x_img = P.pack_rows(x.cuda())
    apart = [_packed(lin["q"]), _packed(lin["k"]), _packed(lin["v"], head_perm=False)]
    out0, q0 = P.qkv_attention(x_img, S, *apart, heads=H, return_q=True, **opts)
    shared = [_packed(lin["q"]), _packed(lin["k"]), _packed(lin["v"], head_perm=False)]
    assert P.PackedLinear.share_adapter_buffer(*shared)
    base = shared[0].lora_a_img.data_ptr()
    step = 8 * (C // 32) * 1024
    assert [t.lora_a_img.data_ptr() - base for t in shared] == [0, step, 2 * step]
    out1, q1 = P.qkv_attention(x_img, S, *shared, heads=H, return_q=True, **opts)
    torch.cuda.synchronize()
    assert torch.equal(q0, q1) and torch.equal(out0, out1)
    odd = [_packed(lin["q"]), _packed(lin["k"]), _packed(lin["v"], head_perm=False)]
    odd[1].lora_scale = 0.25
    assert not P.PackedLinear.share_adapter_buffer(*odd)
    none = [_packed(lin["q"]), _packed(dict(lin["k"], lora_a=None, lora_b=None)) if False else _packed({n: t for n, t in lin["k"].items() if not n.startswith("lora")}),
            _packed(lin["v"], head_perm=False)]
    assert not P.PackedLinear.share_adapter_buffer(*none)


@pytest.mark.parametrize("rank", [128, 16])
def test_merged_adapter_is_the_same_layer(rank):
    """``merge_adapter=True`` folds the adapter into the weight when it is packed (any rank): the layer then carries no
    adapter images, and its output meets the same bar against the float64 layer as the unmerged one; the two differ
    from each other by bf16 rounding only (measured and printed)."""
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    S, N, K = 700, 256, 384
    x = _r(S, K, seed=80).to(torch.bfloat16)
    lin = _linear(N, K, 81, lora=False)
    lin.update(lora_a=_r(rank, K, seed=83, std=K ** -0.5).to(torch.bfloat16), lora_b=_r(N, rank, seed=84, std=0.05).to(torch.bfloat16),
               lora_scale=0.5)
    dev = {n: (t.cuda() if torch.is_tensor(t) else t) for n, t in lin.items()}
    merged = P.PackedLinear.from_weights(dev["weight"], dev["bias"], lora_a=dev["lora_a"], lora_b=dev["lora_b"],
                                         lora_scale=dev["lora_scale"], merge_adapter=True)
    assert merged.lora_a_img is None and merged.lora_b_img is None
    y_merged = P.out_proj(x.cuda(), merged)
    ref = PO.lora_linear(x, **lin)
    err, cos = AO.max_abs_and_cosine(y_merged.cpu(), ref)
    print(f"merged adapter (rank {rank}) vs float64 layer: max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert err <= 2e-2 * max(1.0, float(ref.abs().max())) and cos >= 0.9999
    if rank == 128:
        y_apart = P.out_proj(x.cuda(), _packed(lin))
        e2, c2 = AO.max_abs_and_cosine(y_merged.cpu(), y_apart.cpu())
        print(f"merged vs unmerged: max_abs={e2:.3e} cos={c2:.8f}", flush=True)
        assert c2 >= 0.9999
    else:
        with pytest.raises(ValueError):
            _packed(lin)          # unmerged adapters run at rank 128 only


def test_attention_block_at_480p_shapes():
    """The whole attention half of a block at the benchmark's size (S = 48,360, hidden 3072, 24 heads, LoRA rank 128 on
    all four projections): modulate -> fused QKV -> attention -> to_out with gate and residual, against the float64
    oracle run on the card for every row."""
    import pika_h3_flex_amd as pk
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    S, H = 48360, 24
    C = H * D
    dev = "cuda"
    x = _r(S, C, seed=80).to(torch.bfloat16).to(dev)
    lin = {n: {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in _linear(C, C, 90 + 10 * i).items()}
           for i, n in enumerate(("q", "k", "v", "out"))}
    T = 3
    shift, scale, gate = (_r(T, C, seed=s, std=0.2).to(torch.bfloat16).to(dev) for s in (130, 131, 132))
    pos = pk.video_position_ids(31, 30, 52).to(dev)
    idx = (torch.arange(S) * T // S).to(torch.int32).to(dev)
    ones = torch.ones(D, device=dev)
    x_img = P.adaln_modulate(x, shift=shift, scale=scale, row_index=idx, norm="layer")
    packed = {n: PackedLinear_from(lin[n], head_perm=(n != "v")) for n in lin}
    out = P.qkv_attention(x_img, S, packed["q"], packed["k"], packed["v"], heads=H, q_norm_weight=ones, k_norm_weight=ones,
                          rope_mode=pk.ROPE_INTERLEAVED, rope_q=pk.rope_tables(pos))
    y = P.out_proj(out.view(S, C), packed["out"], gate=gate, row_index=idx, residual=x)
    torch.cuda.synchronize()
    ref = PO.attention_block(x, lin, heads=H, shift=shift, scale=scale, gate=gate, row_index=idx, norm="layer",
                             q_norm_weight=ones, k_norm_weight=ones, rope_mode=AO.ROPE_INTERLEAVED, rope_q=AO.rope_tables(pos))
    err_o, cos_o = AO.max_abs_and_cosine(out.view(S, C), ref["o"])
    err_y, cos_y = AO.max_abs_and_cosine(y, ref["y"])
    print(f"480p block: O max_abs={err_o:.3e} cos={cos_o:.8f}; y max_abs={err_y:.3e} cos={cos_y:.8f}", flush=True)
    assert torch.isfinite(y.float()).all()
    assert err_o <= 2e-2 and cos_o >= 0.9999
    assert err_y <= 2e-2 * max(1.0, float(ref["y"].abs().max())) and cos_y >= 0.9999


def PackedLinear_from(d, head_perm=True):
    from pika_h3_flex_amd.projections import PackedLinear

    return PackedLinear.from_weights(d["weight"], d.get("bias"), lora_a=d.get("lora_a"), lora_b=d.get("lora_b"),
                                     lora_scale=d.get("lora_scale", 1.0), head_perm=head_perm)


class _LoraLinear(torch.nn.Module):
    """What PEFT's ``add_adapter`` leaves on a target (src/pika_h3/core/loader.py:36-37): the base layer plus
    ``lora_A`` / ``lora_B`` / ``scaling`` per adapter name, applied as base(x) + scaling * B(A(x))."""

    def __init__(self, n_in, n_out, rank=128, alpha=64, bias=True):
        super().__init__()
        self.base_layer = torch.nn.Linear(n_in, n_out, bias=bias)
        self.lora_A = torch.nn.ModuleDict({"default": torch.nn.Linear(n_in, rank, bias=False)})
        self.lora_B = torch.nn.ModuleDict({"default": torch.nn.Linear(rank, n_out, bias=False)})
        self.scaling = {"default": alpha / rank}
        torch.nn.init.normal_(self.lora_B["default"].weight, std=0.05)

    def forward(self, x):
        return self.base_layer(x) + self.scaling["default"] * self.lora_B["default"](self.lora_A["default"](x))


class _Attn(torch.nn.Module):
    def __init__(self, hidden, heads, lora):
        super().__init__()
        self.heads = heads
        mk = (lambda: _LoraLinear(hidden, hidden)) if lora else (lambda: torch.nn.Linear(hidden, hidden))
        self.to_q, self.to_k, self.to_v = mk(), mk(), mk()
        self.to_out = torch.nn.ModuleList([mk(), torch.nn.Identity()])
        self.norm_q = torch.nn.RMSNorm(hidden // heads, eps=1e-6)
        self.norm_k = torch.nn.RMSNorm(hidden // heads, eps=1e-6)


@pytest.mark.parametrize("lora", [False, True])
def test_processor_with_fused_projections(lora):
    """The processor with the library's projections (packed from the module, LoRA wrapper included) against the same
    processor on the module's own torch GEMMs, and the block extras (AdaLN, gate, residual) against the oracle."""
    import pika_h3_flex_amd as pk
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO

    torch.manual_seed(5)
    H, hidden, S = 3, 384, 410
    attn = _Attn(hidden, H, lora).cuda().to(torch.bfloat16)
    x = torch.randn((1, S, hidden), device="cuda", dtype=torch.bfloat16)
    pos = torch.cat([pk.video_position_ids(2, 10, 20), pk.audio_position_ids(5)], 0).cuda()
    plain, fused = pk.PikaH3AttnProcessor(), pk.PikaH3AttnProcessor(fused_projections=True)
    with torch.no_grad():
        y0 = plain(attn, x, position_ids=pos)
        y1 = fused(attn, x, position_ids=pos)
    torch.cuda.synchronize()
    err, cos = AO.max_abs_and_cosine(y1.cpu(), y0.cpu())
    print(f"fused vs torch projections (lora={lora}): max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert y1.shape == x.shape and err <= 3e-2 and cos >= 0.9999
    assert fused.packed_weights(attn) is fused.packed_weights(attn)          # packed once
    # block extras against the oracle
    T = 2
    shift, scale, gate = (torch.randn((T, hidden), device="cuda").mul(0.2).to(torch.bfloat16) for _ in range(3))
    idx = (torch.arange(S, device="cuda") % T).to(torch.int32)
    with torch.no_grad():
        y2 = fused(attn, x, position_ids=pos, adaln=dict(shift=shift, scale=scale, row_index=idx, norm="layer"),
                   gate=gate, gate_index=idx, residual=x)
    torch.cuda.synchronize()

    def lin_of(mod):
        base = getattr(mod, "base_layer", mod)
        d = dict(weight=base.weight.detach().cpu(), bias=base.bias.detach().float().cpu())
        if lora:
            d.update(lora_a=mod.lora_A["default"].weight.detach().cpu(), lora_b=mod.lora_B["default"].weight.detach().cpu(),
                     lora_scale=mod.scaling["default"])
        return d

    lin = {"q": lin_of(attn.to_q), "k": lin_of(attn.to_k), "v": lin_of(attn.to_v), "out": lin_of(attn.to_out[0])}
    ref = PO.attention_block(x[0].cpu(), lin, heads=H, shift=shift.cpu(), scale=scale.cpu(), gate=gate.cpu(), row_index=idx.cpu(),
                             q_norm_weight=attn.norm_q.weight.detach().float().cpu(), k_norm_weight=attn.norm_k.weight.detach().float().cpu(),
                             rope_mode=AO.ROPE_INTERLEAVED, rope_q=AO.rope_tables(pos.cpu()))
    err, cos = AO.max_abs_and_cosine(y2[0].cpu(), ref["y"])
    print(f"fused block with AdaLN, gate, residual (lora={lora}): max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert err <= 2e-2 * max(1.0, float(ref["y"].abs().max())) and cos >= 0.9999
    with pytest.raises(ValueError):
        plain(attn, x, position_ids=pos, gate=gate)


def test_rope_cache_tells_two_grids_of_equal_length_apart():
    """Two geometries with the same token count (landscape and portrait), allocated one after the other as the
    reference builds a fresh layout per forward: each call must see its own tables."""
    import pika_h3_flex_amd as pk

    torch.manual_seed(6)
    H, hidden = 2, 256
    attn = _Attn(hidden, H, False).cuda().to(torch.bfloat16)
    S = 6 * 10
    x = torch.randn((1, S, hidden), device="cuda", dtype=torch.bfloat16)
    proc, fresh = pk.PikaH3AttnProcessor(), pk.PikaH3AttnProcessor()
    outs = []
    for hp, wp in ((6, 10), (10, 6)):
        pos = pk.video_position_ids(1, hp, wp).cuda()          # same S, same allocator slot once the first is freed
        with torch.no_grad():
            outs.append((proc(attn, x, position_ids=pos), pk.PikaH3AttnProcessor()(attn, x, position_ids=pos)))
        del pos
    torch.cuda.synchronize()
    for got, want in outs:
        assert torch.equal(got, want)
    assert not torch.equal(outs[0][0], outs[1][0])
    # an in-place edit of a cached grid is seen as a new grid; a caller-supplied key short-cuts the identity check
    pos = pk.video_position_ids(1, 6, 10).cuda()
    with torch.no_grad():
        a = proc(attn, x, position_ids=pos)
        pos[:, 2] += 3.0
        pos[:, 1] *= 2.0
        b = proc(attn, x, position_ids=pos)
        c = fresh(attn, x, position_ids=pos)
        d = proc(attn, x, position_ids=pos, rope_key=("landscape", 6, 10, "edited"))
    torch.cuda.synchronize()
    assert torch.equal(b, c) and torch.equal(d, c) and not torch.equal(a, b)


def test_document_kwargs_drive_the_fused_block():
    """From one request's latents to an attention block: the wrapper-side kwargs (position grid, per-row timestep
    index; src/pika_h3/core/wrapper.py:96-205) feed the processor's RoPE tables and its AdaLN / gate gathers, checked
    against the float64 block on the same document."""
    import pika_h3_flex_amd as pk
    from pika_h3_flex_amd import packing as P
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO

    g = torch.Generator().manual_seed(11)
    F, LH, LW, T, L = 3, 12, 20, 9, 7
    video, audio = torch.randn(1, F, 24, LH, LW, generator=g), torch.randn(1, T, 64, generator=g)
    cond = {"prompt_embeds": torch.randn(L, 32, generator=g), "text_token_tags": torch.ones(L, dtype=torch.long),
            "keyframes": [{"anchor": "first", "latents": torch.randn(1, 1, 24, LH, LW, generator=g)}]}
    mi, _, _, ncv, nca = P.prepare_document(video.cuda(), audio.cuda(), cond, 0.7, 0.4, generator=None)
    pos, tidx, times = mi["position_ids"], mi["timestep_indices"], mi["timestep"]
    S = pos.shape[0]
    assert S == L + 60 + 2 * T + F * 60 and tidx.shape == (S,) and times.numel() == 3 and (ncv, nca) == (60, 0)
    assert pos.is_cuda and tidx.is_cuda and tidx.dtype == torch.int32

    torch.manual_seed(12)
    H, hidden = 2, 256
    attn = _Attn(hidden, H, True).cuda().to(torch.bfloat16)
    x = torch.randn((1, S, hidden), device="cuda", dtype=torch.bfloat16)      # the packed hidden states of the block
    K = times.numel()
    # the block's modulation tables from a time embedding per row time, the way the patched module forms them
    # (float32 SiLU, then the linear layer; patches/0001-h3-adaln-fp32.patch:126-133): six tables of K rows
    from pika_h3_flex_amd import projections as PR
    temb = torch.randn((K, 64), device="cuda").to(torch.bfloat16)
    mod_w = torch.randn((6 * hidden, 64), device="cuda").mul(0.03).to(torch.bfloat16)
    mod_b = torch.randn(6 * hidden, device="cuda").mul(0.05).to(torch.bfloat16)
    shift, scale, gate, _, _, _ = PR.modulation_tables(temb, mod_w, mod_b, hidden)
    want = PO.modulation_tables(temb.cpu(), mod_w.cpu(), mod_b.cpu(), hidden)
    for got_t, want_t in zip((shift, scale, gate), want):
        assert float((got_t.cpu().double() - want_t).abs().max()) <= 2.0 ** -7 * max(1.0, float(want_t.abs().max()))
    assert torch.equal(PR.modulation_row_index(tidx), tidx)
    proc = pk.PikaH3AttnProcessor(fused_projections=True)
    with torch.no_grad():
        y = proc(attn, x, position_ids=pos, adaln=dict(shift=shift, scale=scale, row_index=tidx, norm="layer"),
                 gate=gate, gate_index=tidx, residual=x)
    torch.cuda.synchronize()

    def lin_of(mod):
        return dict(weight=mod.base_layer.weight.detach().cpu(), bias=mod.base_layer.bias.detach().float().cpu(),
                    lora_a=mod.lora_A["default"].weight.detach().cpu(), lora_b=mod.lora_B["default"].weight.detach().cpu(),
                    lora_scale=mod.scaling["default"])

    lin = {"q": lin_of(attn.to_q), "k": lin_of(attn.to_k), "v": lin_of(attn.to_v), "out": lin_of(attn.to_out[0])}
    ref = PO.attention_block(x[0].cpu(), lin, heads=H, shift=shift.cpu(), scale=scale.cpu(), gate=gate.cpu(), row_index=tidx.cpu(),
                             q_norm_weight=attn.norm_q.weight.detach().float().cpu(), k_norm_weight=attn.norm_k.weight.detach().float().cpu(),
                             rope_mode=AO.ROPE_INTERLEAVED, rope_q=AO.rope_tables(pos.cpu()))
    err, cos = AO.max_abs_and_cosine(y[0].cpu(), ref["y"])
    print(f"document -> fused block: S={S}, {K} row times, max_abs={err:.3e} cos={cos:.8f}", flush=True)
    assert err <= 2e-2 * max(1.0, float(ref["y"].abs().max())) and cos >= 0.9999
    # the keyframe rows and the frame they pin share a grid, so with equal inputs they would rotate alike: spot-check the layout
    vi = mi["video_indices"]
    assert torch.equal(pos[vi[:60], 1:], pos[vi[60:120], 1:]) and float(pos[vi[:60], 0].abs().sum()) == 0.0


@pytest.mark.parametrize("S,H,variant", [(300, 2, "dense"), (1000, 3, "fp8"), (777, 2, "sparse"), (777, 2, "sparse_long"),
                                         (130, 1, "narrow"), (1085, 24, "short"), (1085, 24, "short_fp8"),
                                         (4200, 24, "shared"), (4200, 24, "shared_fp8")])
def test_attention_writes_the_out_projection_images(S, H, variant):
    """With PKH3_FLAG_O_IMAGES the attention epilogue writes what pkh3_pack_rows would make of its row-major output:
    the same bytes for every image row that exists, in every form of the kernel (long, short-key, narrow, shared last round, block-sparse in both)."""
    import pika_h3_flex_amd as pk
    from pika_h3_flex_amd import projections as P

    sparse, fp8, long_form = "sparse" in variant, "fp8" in variant, variant in ("dense", "sparse_long")
    want_form = {"sparse": forms.NARROW, "sparse_long": forms.SPARSE, "narrow": forms.NARROW, "fp8": forms.NARROW, "short": forms.SHORT,
                 "short_fp8": forms.SHORT}.get(variant, forms.LONG)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert forms.form(1, H, S, S, sparse=sparse, fp8=fp8, long_key_kernel=long_form, cus=cus) == want_form

    g = torch.Generator().manual_seed(21)
    q, k, v = (torch.randn((1, S, H, 128), generator=g).to(torch.bfloat16).cuda() for _ in range(3))
    w = (1.0 + 0.1 * torch.randn(128, generator=g)).cuda()
    pos = (torch.rand((S, 3), generator=g, dtype=torch.float64) * 20).cuda()
    opts = dict(q_norm_weight=w, k_norm_weight=w, rope_mode=pk.ROPE_INTERLEAVED, rope_q=pk.rope_tables(pos))
    if fp8:
        opts["fp8_qk"] = True
    # "shared": 264 query tiles on a 256-CU part: whole rounds, then the last 8 tiles shared out two ways
    if sparse:
        nt = (S + 63) // 64
        keep = torch.rand((nt, nt), generator=g) < 0.5
        keep |= torch.eye(nt, dtype=torch.bool)
        opts["block_mask"] = pk.BlockMask.from_dense(keep.cuda())
    opts["long_key_kernel"] = long_form
    rows = pk.attention(q, k, v, **opts)
    want = P.pack_rows(rows.view(S, H * 128))
    img = torch.full((P.packed_bytes(S, H * 128),), 0xAB, dtype=torch.uint8, device="cuda")
    got = pk.attention(q, k, v, out=img, out_images=True, **opts)
    torch.cuda.synchronize()
    assert got is img
    live = ((S + 31) // 32) * 2 * (H * 128 // 32) * 1024        # bytes of the 32-row blocks that hold rows
    assert torch.equal(img[:live], want[:live])
    assert bool((img[live:] == 0xAB).all())                     # blocks past the last row are left alone
    with pytest.raises(ValueError):
        pk.attention(q.expand(2, -1, -1, -1), k.expand(2, -1, -1, -1), v.expand(2, -1, -1, -1), out=img, out_images=True, **opts)


@pytest.mark.parametrize("seed", [1, 2])
def test_random_projection_combinations(seed):
    """Seeded sweep over what the fixed cases above leave out: row counts around the 16-row image and the 256-row tile
    (1, 2, 15..17, 255..257 ...), an activation width different from heads x 128, adapters and biases on some of the
    three targets only, both output forms of the attention call, each followed by the out-projection."""
    import random

    import pika_h3_flex_amd as pk
    from oracle import attention_oracle as AO
    from oracle import projection_oracle as PO
    from pika_h3_flex_amd import projections as P

    rng = random.Random(seed)
    for case in range(20):
        S = rng.choice([1, 2, 15, 16, 17, 31, 33, 47, 63, 64, 65, 255, 256, 257, 300, 511, 513, 777, 1030])
        H, K = rng.choice([1, 2, 3]), rng.choice([32, 96, 128, 256, 384, 544])
        C = H * D
        variant = rng.choice(["bf16", "bf16", "fp8", "sparse", "norope", "half"])
        base = 100000 * seed + 1000 * case
        x = _r(S, K, seed=base + 900).to(torch.bfloat16)
        lin = {n: _linear(C, K, base + 10 * i, lora=rng.random() < 0.6, bias=rng.random() < 0.6) for i, n in enumerate("qkv")}
        wq, wk = 1.0 + 0.1 * _r(D, seed=50), 1.0 + 0.1 * _r(D, seed=51)
        opts, ref_opts = dict(q_norm_weight=wq.cuda(), k_norm_weight=wk.cuda()), dict(q_norm_weight=wq, k_norm_weight=wk)
        if variant != "norope":
            pos = torch.rand((S, 3), generator=torch.Generator().manual_seed(base), dtype=torch.float64) * 20
            mode = pk.ROPE_HALF if variant == "half" else pk.ROPE_INTERLEAVED
            opts.update(rope_mode=mode, rope_q=pk.rope_tables(pos.cuda()))
            ref_opts.update(rope_mode=mode, rope_q=AO.rope_tables(pos))
        if variant == "fp8":
            opts.update(fp8_qk=True)
            ref_opts.update(fp8_qk=True)
        if variant == "sparse":
            n = (S + 63) // 64
            tm = (torch.rand((n, n), generator=torch.Generator().manual_seed(base + 3)) < 0.5) | torch.eye(n, dtype=torch.bool)
            opts.update(block_mask=pk.BlockMask.from_dense(tm, device="cuda"))
            ref_opts.update(tile_map=tm)
        as_images = rng.random() < 0.5
        out, q = P.qkv_attention(P.pack_rows(x.cuda()), S, _packed(lin["q"]), _packed(lin["k"]), _packed(lin["v"], head_perm=False),
                                 heads=H, return_q=True, out_images=as_images, **opts)
        n_out = rng.choice([128, 256, 384])
        lo = _linear(n_out, C, base + 500, lora=rng.random() < 0.5, bias=rng.random() < 0.5)
        q_ref, k_ref, v_ref = (PO.lora_linear(x, **lin[n]).view(1, S, H, D) for n in "qkv")
        r = lambda t: t.to(torch.bfloat16)
        o_ref = AO.reference_layer(r(q_ref), r(k_ref), r(v_ref), **ref_opts)
        if as_images:
            y = P.out_proj(None, _packed(lo), o_img=out, rows=S)
            y_ref = PO.lora_linear(r(o_ref).view(S, C), **lo)
            err_o, cos_o = 0.0, 1.0  # O is checked through y
        else:
            y = P.out_proj(out.view(S, C), _packed(lo))
            y_ref = PO.lora_linear(out.cpu().view(S, C), **lo)
            err_o, cos_o = AO.max_abs_and_cosine(out.cpu(), o_ref)
        torch.cuda.synchronize()
        err_q, cos_q = AO.max_abs_and_cosine(q.cpu(), q_ref)
        err_y, cos_y = AO.max_abs_and_cosine(y.cpu(), y_ref)
        label = (f"seed {seed} case {case}: S={S} H={H} K={K} {variant} images={as_images} N_out={n_out} "
                 f"lora={['lora_a' in lin[n] for n in 'qkv']} bias={['bias' in lin[n] for n in 'qkv']}: "
                 f"Q {err_q:.2e}/{cos_q:.6f} O {err_o:.2e}/{cos_o:.6f} y {err_y:.2e}/{cos_y:.6f}")
        print(label, flush=True)
        assert torch.isfinite(y.float()).all(), label
        fp8 = variant == "fp8"
        assert err_q <= 2e-2 and cos_q >= 0.9999, label
        assert cos_o >= (0.995 if fp8 else 0.9999) and (fp8 or err_o <= 2e-2), label
        assert cos_y >= (0.995 if fp8 and as_images else 0.9999), label


def test_fused_block_replays_from_a_hip_graph():
    """modulate -> q/k/v (+LoRA) -> attention -> to_out (+LoRA, gate, residual) captured into one HIP graph: the
    library clears its reduction slots with a fill kernel and launches kernels only, so every replay on fresh
    inputs, with eager work and synchronisation in between, must give the bits of the eager calls."""
    import pika_h3_flex_amd as pk
    from pika_h3_flex_amd import projections as P

    S, H = 700, 2
    C = H * D
    dev = "cuda"
    lin = {n: _packed(_linear(C, C, 300 + 10 * i), head_perm=(n != "v")) for i, n in enumerate("qkv")}
    lo = _packed(_linear(C, C, 340))
    T = 3
    shift, scale = (_r(T, C, seed=350 + i, std=0.3).to(torch.bfloat16).to(dev) for i in range(2))
    gate = _r(T, C, seed=352, std=0.5).to(torch.bfloat16).to(dev)
    idx = torch.randint(0, T, (S,), generator=torch.Generator().manual_seed(353)).to(torch.int32).to(dev)
    w = torch.ones(D, device=dev)
    pos = torch.rand((S, 3), generator=torch.Generator().manual_seed(354), dtype=torch.float64) * 20
    opts = dict(q_norm_weight=w, k_norm_weight=w, rope_mode=pk.ROPE_INTERLEAVED, rope_q=pk.rope_tables(pos.to(dev)))

    def block(x):
        x_img = P.adaln_modulate(x, shift=shift, scale=scale, row_index=idx)
        o_img = P.qkv_attention(x_img, S, lin["q"], lin["k"], lin["v"], heads=H, out_images=True, **opts)
        return P.out_proj(None, lo, gate=gate, row_index=idx, residual=x, o_img=o_img, rows=S)

    x_buf = _r(S, C, seed=360).to(torch.bfloat16).to(dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        block(x_buf)  # warm-up outside the capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_buf = block(x_buf)
    for rep in range(4):
        fresh = _r(S, C, seed=370 + rep).to(torch.bfloat16).to(dev)
        eager = block(fresh).clone()
        torch.cuda.synchronize()
        x_buf.copy_(fresh)
        y_buf.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.isfinite(y_buf.float()).all()
        assert torch.equal(y_buf, eager), f"replay {rep} differs from the eager calls"
