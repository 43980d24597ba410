"""GPU parity: the HIP path, called through the C ABI, against the float64 oracle on the same
seeded inputs.  Tolerance for the bf16 paths (from the benchmark contract): max-abs <= 2e-2 and
cosine >= 0.9999 versus the float64/fp32 reference."""
import math

import pytest
import torch

from tests import test_attention_forms as forms

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-2
MIN_COS = 0.9999


def _oracle():
    from oracle import attention_oracle as O

    return O


def _rand(shape, gen, std=1.0):
    return (torch.randn(shape, generator=gen, dtype=torch.float32) * std).to(torch.bfloat16)


def _form(*call, **opts):
    """The form of the attention kernel the call takes on this part."""
    return forms.form(*call, cus=torch.cuda.get_device_properties(0).multi_processor_count, **opts)


def _run_and_check(B, Sq, Sk, H, *, seed=0, norm=True, rope_mode=0, mask=None, std=1.0, min_cos=MIN_COS,
                   max_abs=MAX_ABS, weight_random=False, weight_scale=1.0, bf16_operands=False, fp8=False, scale=None,
                   batch_pad=0):
    """``fp8``: the fp8 QK^T path against the oracle's fake-quant emulation (cosine >= 0.995 by contract, held to
    0.9995).  ``scale``: softmax scale other than 1/sqrt(D).  ``batch_pad``: extra elements between the batch entries
    of q, k, v and the output, so the batch stride is not S*H*D."""
    import pika_h3_flex_amd as pk

    O = _oracle()
    D = 128
    gen = torch.Generator().manual_seed(seed)
    q, k, v = _rand((B, Sq, H, D), gen, std), _rand((B, Sk, H, D), gen, std), _rand((B, Sk, H, D), gen)
    qw = kw = None
    if norm:
        if weight_random:
            qw = 1.0 + 0.2 * torch.randn(D, generator=gen)
            kw = 1.0 + 0.2 * torch.randn(D, generator=gen)
        else:
            qw, kw = torch.ones(D), torch.ones(D)
        qw = qw * weight_scale
    rope_q = rope_k = None
    if rope_mode:
        posq = torch.rand((Sq, 3), generator=gen, dtype=torch.float64) * torch.tensor([30.0, 29.0, 51.0], dtype=torch.float64)
        posk = posq if Sq == Sk else torch.rand((Sk, 3), generator=gen, dtype=torch.float64) * 40.0
        rope_q = O.rope_tables(posq)
        rope_k = O.rope_tables(posk)
    ref = O.reference_layer(q, k, v, q_norm_weight=qw, k_norm_weight=kw, rope_q=rope_q, rope_k=rope_k,
                            rope_mode=rope_mode, key_mask=mask, bf16_operands=bf16_operands, fp8_qk=fp8, scale=scale)
    dev = "cuda"
    f32 = lambda t: None if t is None else t.to(torch.float32).contiguous().to(dev)
    opts = dict(q_norm_weight=f32(qw), k_norm_weight=f32(kw), norm_eps=1e-6, rope_mode=rope_mode, fp8_qk=fp8,
                softmax_scale=scale)
    if fp8:
        min_cos = 0.9995
    if rope_mode:
        opts.update(rope_q=(f32(rope_q[0]), f32(rope_q[1])), rope_k=(f32(rope_k[0]), f32(rope_k[1])))
    if mask is not None:
        opts.update(key_mask=mask.to(dev))
    # small calls take the narrow or the short-key form of the kernel: check the long-key form on the same inputs too
    def on_device(t):
        """[B, S, H, D] on the card; with batch_pad as a view into a wider buffer, so the batch stride is S*H*D + pad"""
        if not batch_pad:
            return t.to(dev)
        Bt, St = t.shape[0], t.shape[1]
        buf = torch.full((Bt, St * H * D + batch_pad), float("nan"), dtype=torch.bfloat16, device=dev)
        view = buf[:, :St * H * D].view(Bt, St, H, D)
        view.copy_(t)
        assert view.stride(0) == St * H * D + batch_pad
        return view

    for long_form in (True, False):
        o_buf = on_device(torch.zeros_like(q)) if batch_pad else None
        out = pk.attention(on_device(q), on_device(k), on_device(v), long_key_kernel=long_form, out=o_buf, **opts)
        torch.cuda.synchronize()
        out = out.cpu()
        assert torch.isfinite(out.float()).all()
        err, cos = O.max_abs_and_cosine(out, ref)
        print(f"B={B} Sq={Sq} Sk={Sk} H={H} rope={rope_mode} mask={mask is not None} long_form={long_form}: "
              f"max_abs={err:.3e} cos={cos:.7f}", flush=True)
        assert err <= max_abs and cos >= min_cos
    return out, ref


def test_plumbing_config():
    """B=1, H=4, S=1024, D=128, N(0,1) inputs, QK-RMSNorm (eps 1e-6, unit weight), no mask."""
    _run_and_check(1, 1024, 1024, 4, seed=1)


@pytest.mark.parametrize("S", [1, 7, 64, 65, 200, 257, 1000])
def test_ragged_lengths(S):
    _run_and_check(1, S, S, 2, seed=S)


@pytest.mark.parametrize("Sq,Sk", [(5, 300), (300, 5), (513, 129), (64, 4096)])
def test_rectangular(Sq, Sk):
    _run_and_check(1, Sq, Sk, 3, seed=Sq + Sk)


@pytest.mark.parametrize("fp8", [False, "pow2", True])
@pytest.mark.parametrize("B,Sq,Sk,H", [(1, 1, 97, 1), (1, 31, 129, 3), (2, 33, 255, 2), (1, 64, 1025, 2), (1, 65, 96, 5), (1, 97, 3000, 3),
                                       (1, 641, 1089, 24)])
def test_few_query_blocks(B, Sq, Sk, H, fp8):
    """Calls whose 32-query blocks hardly outnumber the CUs: key counts around whole half tiles (some of the four waves with
    one half tile more than others, the last one partial), a lone query, halves of a 64-query fp8 scale block beyond the end, and
    two blocks per CU (the last).  All of them in the narrow form.  Bounded and running-maximum softmax."""
    assert _form(B, H, Sq, Sk, fp8=fp8) == forms.NARROW
    _run_and_check(B, Sq, Sk, H, seed=Sq + Sk, weight_random=True, fp8=fp8)
    if not fp8:
        _run_and_check(B, Sq, Sk, H, seed=Sq + Sk, weight_scale=4.0, bf16_operands=True)


@pytest.mark.parametrize("B,H,Sq,Sk,masked,fp8", [(*call, fp8) for call in forms.SHORT_KEY_CALLS for fp8 in ((False,) if call[4] else (False, "pow2", True))])
def test_short_key_form(B, H, Sq, Sk, masked, fp8):
    """Ragged ends of queries and keys, one to three workgroups per CU, up to and beyond 16 key tiles; scattered key masks with a batch
    entry that has no key at all.  Bounded and running-maximum softmax."""
    assert _form(B, H, Sq, Sk, masked=masked, fp8=fp8) == forms.SHORT
    mask = None
    if masked:
        mask = torch.rand((B, Sk), generator=torch.Generator().manual_seed(Sk)) < 0.6
        mask[1] = False
    _run_and_check(B, Sq, Sk, H, seed=Sq + Sk, mask=mask, weight_random=True, fp8=fp8, rope_mode=1 + Sk % 2)
    # fp8 at weight 4: an element that float32 and float64 round to neighbouring e4m3 values (1/8 apart at most; |q'| <= 16, |k'| <= 4)
    # moves a logit by up to 0.088 * 16 * 4 / 8 = 0.7, a probability by up to a quarter of that, and an output by that much of
    # the distance of two values of V (<= 8): 1.4 at most, 0.35 for one of twice the usual size (q' 8, k' 2)
    _run_and_check(B, Sq, Sk, H, seed=Sq + Sk, mask=mask, weight_scale=4.0, bf16_operands=not fp8, fp8=fp8, max_abs=0.35 if fp8 else MAX_ABS)


@pytest.mark.parametrize("scale", [1.0, 6.0])
@pytest.mark.parametrize("B,H,Sq,Sk,rope,valid", [
    (1, 1030, 70, 1100, 0, None),           # a unit a head: every round belongs to another one, one of three groups has work
    (1, 32, 4229, 500, 0, None),            # whole rounds, some of one and two groups, a unit that holds rows of one wave only
    (2, 24, 3072, 512, 0, None),            # nothing partial but a head's last round
    (1, 24, 6500, 1024, 0, None),           # 51 units a head: the last of one goes to the run before
    (1, 24, 5600, 2496, 0, None), (1, 24, 5600, 2497, 1, None),   # the most tiles
    (1, 345, 300, 1025, 1, None), (1, 516, 200, 1088, 2, None),   # 17 tiles and rotation, the last one of one key and whole
    (3, 144, 1025, 600, 0, (0, 1, 400)),    # masked: no key, one, some
    (6, 60, 1250, 640, 0, (64, 65, 128, 129, 500, 640)),          # one to ten tiles
    (70, 4, 500, 1100, 0, tuple(75 * i % 1101 for i in range(70))), (530, 1, 200, 1100, 0, tuple(75 * i % 1101 for i in range(530))), (2, 24, 2900, 2500, 1, (64, 2500)),   # shared out by the entries' keys
])
def test_relay_form(B, H, Sq, Sk, rope, valid, scale):
    """Dense calls of more than four 128-query units a CU against 8 to 40 key tiles: a workgroup goes from unit to unit.  At scale 6
    (the norm weights of the queries) the running maximum; against the oracle with operands rounded as the kernel's are.
    Strided queries and outputs, prepared keys, the output in the queries' place and as operand images, and no norm at all."""
    import pika_h3_flex_amd as pk
    from pika_h3_flex_amd import projections as P

    O = _oracle()
    assert _form(B, H, Sq, Sk, rope=rope, masked=valid is not None) == forms.RELAY
    gen = torch.Generator(device="cuda").manual_seed(Sq + Sk)
    rows = lambda S, std=1.0: (torch.randn((B, S, H, 128), generator=gen, device="cuda") * std).to(torch.bfloat16)
    wide = torch.empty((B, Sq, H, 136), dtype=torch.bfloat16, device="cuda")
    q, k, v = wide[..., :128], rows(Sk), rows(Sk)
    q.copy_(rows(Sq))
    w = [1.0 + 0.2 * torch.randn(128, generator=gen, device="cuda") for _ in range(2)]
    opts = dict(q_norm_weight=w[0] * scale, k_norm_weight=w[1])
    ref = dict(opts, bf16_operands=scale > 1)
    if rope:
        tabs = [O.rope_tables(torch.rand((S, 3), generator=gen, dtype=torch.float64, device="cuda") * 40) for S in (Sq, Sk)]
        f32 = [tuple(t.float().contiguous() for t in pair) for pair in tabs]
        opts.update(rope_mode=rope, rope_q=f32[0], rope_k=f32[1])
        ref.update(rope_mode=rope, rope_q=tabs[0], rope_k=tabs[1])
    if valid:
        mask = torch.stack([torch.randperm(Sk, generator=gen, device="cuda") < n for n in valid])
        opts.update(key_mask=mask)
        ref.update(key_mask=mask)
    want = torch.cat([O.reference_layer(q[:, i:i + 256], k, v, **{**ref, **({"rope_q": tuple(t[i:i + 256] for t in tabs[0])} if rope else {})})
                      for i in range(0, Sq, 256)], dim=1)
    out = pk.attention(q, k, v, **opts)
    err, cos = O.max_abs_and_cosine(out, want)
    print(f"B={B} H={H} {Sq} x {Sk} rope={rope} valid={valid} scale={scale}: max_abs={err:.3e} cos={cos:.7f}", flush=True)
    # (at scale 6 a query may keep little more than one key: its numerator and the output are rounded by up to 2^-8 of the largest value each)
    assert err <= (MAX_ABS if scale == 1.0 else 2.0 ** -7 * float(v.abs().max())) and cos >= MIN_COS
    k_opts = {n: o for n, o in opts.items() if n in ("k_norm_weight", "rope_mode", "rope_k", "key_mask")}
    kv = pk.prepare_kv(k, v, **k_opts)
    assert torch.equal(pk.attention_prepared(q, kv, **{n: o for n, o in opts.items() if n not in k_opts}), out)
    if B == 1 and H <= 32:
        img = torch.full((P.packed_bytes(Sq, H * 128),), 0xAB, dtype=torch.uint8, device="cuda")
        pk.attention(q, k, v, out=img, out_images=True, **opts)
        live = ((Sq + 31) // 32) * 2 * (H * 128 // 32) * 1024
        assert torch.equal(img[:live], P.pack_rows(out.view(Sq, H * 128))[:live]) and bool((img[live:] == 0xAB).all())
    assert torch.equal(pk.attention(q, k, v, out=q, **opts), out)
    if scale == 1.0 and not rope:
        del opts["q_norm_weight"], ref["q_norm_weight"]
        ref["bf16_operands"] = True
        q.copy_(rows(Sq, 0.5))
        want = torch.cat([O.reference_layer(q[:, i:i + 256], k, v, **ref) for i in range(0, Sq, 256)], dim=1)
        err, cos = O.max_abs_and_cosine(pk.attention(q, k, v, **opts), want)
        assert err <= MAX_ABS and cos >= MIN_COS


@pytest.mark.parametrize("valid", [0, 1, 33, 64, 230])
def test_few_query_blocks_masked(valid):
    """Fewer valid keys than the waves of a workgroup have shares for, none among them, and running-maximum softmax with
    empty shares."""
    mask = torch.zeros((2, 300), dtype=torch.bool)
    mask[0, 300 - valid:] = True
    mask[1, ::2] = True
    _run_and_check(2, 77, 300, 2, seed=valid, mask=mask, weight_random=True)
    _run_and_check(2, 77, 300, 2, seed=valid, mask=mask, weight_scale=4.0, bf16_operands=True)


@pytest.mark.parametrize("H,Sq,Sk,valid", [(24, 200, 400, (96, 97, 0)), (24, 200, 400, (1, 32, 33)), (24, 500, 2040, (1312, 1345, 1)),
                                           (24, 500, 2040, (2040, 1311, 1313))])
def test_masked_calls_of_few_and_many_valid_keys(H, Sq, Sk, valid):
    """Batch entries on both sides of the number of valid keys below which a masked call of few query blocks is walked like the
    short-key form (4 half tiles at the first size, 42 at the second), each by its own count, in one launch."""
    mask = torch.zeros((3, Sk), dtype=torch.bool)
    gen = torch.Generator().manual_seed(sum(valid))
    for b, n in enumerate(valid):
        mask[b, torch.randperm(Sk, generator=gen)[:n]] = True
    _run_and_check(3, Sq, Sk, H, seed=sum(valid), mask=mask, weight_random=True)


@pytest.mark.parametrize("first,last", [(128, 192), (0, 64), (96, 160), (384, 512)])
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("H", [1, 180])
def test_runs_of_keys_with_logits_of_minus_infinity(first, last, sparse, H):
    """Keys first .. last - 1 have an element of -inf against positive query elements: their logits are -inf and they weigh
    nothing, also where they are the first keys, or all the keys, that one of the waves sharing the keys out walks (one head:
    a wave takes 128 of the 512 keys; 180 heads: one wave walks them all)."""
    import pika_h3_flex_amd as pk

    O = _oracle()
    gen = torch.Generator().manual_seed(first + H)
    q, k, v = _rand((1, 80, H, 128), gen), _rand((1, 512, H, 128), gen), _rand((1, 512, H, 128), gen)
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, first:last, :, 0] = -math.inf
    opts = dict(block_mask=pk.BlockMask.from_dense(torch.ones((2, 8), dtype=torch.bool), device="cuda")) if sparse else {}
    mask = torch.ones((1, 512), dtype=torch.bool)
    mask[:, first:last] = False
    ref = O.reference_layer(q, torch.nan_to_num(k, neginf=0.0), v, key_mask=mask)
    for long_form in (False, True):
        out = pk.attention(q.cuda(), k.cuda(), v.cuda(), long_key_kernel=long_form, **opts)
        torch.cuda.synchronize()
        assert torch.isfinite(out.float()).all(), long_form
        err, cos = O.max_abs_and_cosine(out.cpu(), ref)
        print(f"-inf keys {first}..{last - 1} sparse={sparse} H={H} long_form={long_form}: max_abs={err:.3e} cos={cos:.7f}", flush=True)
        assert err <= MAX_ABS and cos >= MIN_COS


@pytest.mark.parametrize("first,last", [(448, 512), (384, 512), (500, 505), (0, 64), (96, 160), (0, 448)])
@pytest.mark.parametrize("Sk", [505, 512])
def test_runs_of_keys_with_logits_of_minus_infinity_in_the_relay_form(first, last, Sk):
    """As above where a workgroup goes from unit to unit: it takes a head's last tile first (with fewer keys than the tile has places, or all),
    so that runs which end there leave the first sums without a finite logit."""
    import pika_h3_flex_amd as pk

    O = _oracle()
    H, Sq, last = 24, 5600, min(last, Sk)
    assert _form(1, H, Sq, Sk) == forms.RELAY
    gen = torch.Generator(device="cuda").manual_seed(first + Sk)
    q, k, v = (torch.randn((1, S, H, 128), generator=gen, device="cuda").to(torch.bfloat16) for S in (Sq, Sk, Sk))
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, first:last, :, 0] = -math.inf
    mask = torch.ones((1, Sk), dtype=torch.bool, device="cuda")
    mask[:, first:last] = False
    out = pk.attention(q, k, v)
    assert torch.isfinite(out.float()).all()
    want = torch.cat([O.reference_layer(q[:, i:i + 256], torch.nan_to_num(k, neginf=0.0), v, key_mask=mask) for i in range(0, Sq, 256)], dim=1)
    err, cos = O.max_abs_and_cosine(out, want)
    assert err <= MAX_ABS and cos >= MIN_COS


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("Sq,Sk", [(5, 300), (300, 5), (513, 129), (200, 2100)])
def test_rectangular_with_rope_and_separate_tables(Sq, Sk, mode, fp8):
    """Sq != Sk with rotation: the queries and the keys carry position grids of their own (distinct cos/sin tables);
    both pairings, bf16 and fp8, both forms of the dense kernel (long_key_kernel on and off inside the helper)."""
    _run_and_check(1, Sq, Sk, 2, seed=7 * Sq + Sk + mode, rope_mode=mode, weight_random=True, fp8=fp8)


@pytest.mark.parametrize("B,H,Sk,mode,fp8,masked", [(1, 7, 17901, 1, False, False), (1, 7, 17901, 2, True, False), (2, 5, 17900, 0, False, True)])
def test_kv_pass_walks_several_heads(B, H, Sk, mode, fp8, masked):
    """Key sets long enough that a workgroup of the K/V pass takes several heads one after the other (here 3, the last
    group with fewer), with a partial last tile, and through a scattered key mask."""
    gen = torch.Generator().manual_seed(Sk + mode)
    mask = (torch.rand((B, Sk), generator=gen) < 0.4) if masked else None
    _run_and_check(B, 40, Sk, H, seed=31 + mode, rope_mode=mode, weight_random=True, fp8=fp8, mask=mask)


@pytest.mark.parametrize("fp8", [False, True, "pow2"])
@pytest.mark.parametrize("std", [1.0, 8.0])   # bounded logits; logits that take the running maximum
@pytest.mark.parametrize("Sk", [1, 32, 33, 64, 95, 128, 129, 160, 191, 225, 513])
def test_pipelined_short_key_form_at_every_end(Sk, std, fp8):
    """Two short-key workgroups per CU and fewer: passes work on two halves at once, the last one or two of them on what is there."""
    import pika_h3_flex_amd as pk

    H, Sq = 24, 1061
    assert _form(1, H, Sq, Sk, fp8=fp8) == forms.SHORT
    gen = torch.Generator().manual_seed(Sk)
    q, k, v = (_rand((1, n, H, 128), gen, s).cuda() for n, s in ((Sq, std), (Sk, 1.0), (Sk, 1.0)))
    got = pk.attention(q, k, v, fp8_qk=fp8).float()
    want = pk.attention(q, k, v, fp8_qk=fp8, long_key_kernel=True).float()
    # the same weights, rounded to bf16 at bases that may differ (2^-9 of each, in both), and both results rounded (2^-9):
    # the weights sum to 1, so at most 4 * 2^-9 of the largest value
    assert torch.isfinite(got).all() and (got - want).abs().max() <= 4 * 2 ** -9 * v.float().abs().max()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("scale", [0.05, 0.2])
def test_softmax_scale_other_than_default(scale, fp8):
    """softmax_scale reaches the logits (bf16: folded into the Q operand; fp8: into the dequantisation factor).
    0.2 with unit-weight QK-RMSNorm bounds the logits by 37 in log2 units: still the bounded-logit path."""
    _run_and_check(1, 300, 420, 2, seed=int(scale * 100), rope_mode=1, scale=scale, fp8=fp8)


def test_softmax_scale_on_the_running_max_path():
    """scale 0.2 and norm weight x4: logit bound 148 in log2 units, far beyond the limit of the bounded-logit path."""
    _run_and_check(1, 333, 333, 2, seed=21, rope_mode=2, scale=0.2, weight_scale=4.0, bf16_operands=True)


@pytest.mark.parametrize("H,Sq,Sk,at,sparse,long_key,fp8", [
    (1, 64, 70, 69, False, False, False), (2, 40, 9000, 8999, False, False, False), (1, 64, 8193, 8192, False, False, "pow2"),   # narrow form
    (24, 1085, 1085, 1084, False, False, False), (24, 1085, 1085, 33, False, False, True),   # short-key form
    (1, 400, 9000, 8193, False, True, False), (1, 64, 16500, 16499, False, True, True),      # long form
    (2, 300, 9000, 8999, True, True, False), (1, 64, 130, 129, True, False, False),          # block-sparse, 8 waves and narrow
    (1, 33, 140001, 140000, False, False, False), (1, 33, 140001, 131071, False, False, "pow2"), (1, 33, 140001, 32769, False, False, False),
    (2, 33, 140001, 131072, False, True, False),   # norms of more keys than one trip to memory fetches
])
def test_one_key_of_a_large_norm_wherever_it_lies(H, Sq, Sk, at, sparse, long_key, fp8):
    """The softmax runs without a maximum where the largest key norm allows it: a key of a logit of 260 (base 2) anywhere, in
    a short last half tile or behind the first 256 halves, has to be seen.  Every query then attends to it alone."""
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(Sk + at)
    q = (1.0 + 0.01 * torch.randn((1, Sq, H, 128), generator=gen)).to("cuda", torch.bfloat16)
    k = (0.01 * torch.randn((1, Sk, H, 128), generator=gen)).to("cuda", torch.bfloat16)
    v = torch.randn((1, Sk, H, 128), generator=gen).to("cuda", torch.bfloat16)
    k[:, at] = 16.0
    opts = {"long_key_kernel": long_key, "fp8_qk": fp8}
    if sparse:
        opts["block_mask"] = pk.BlockMask.from_dense(torch.ones((-(-Sq // 64), -(-Sk // 64)), dtype=torch.bool), device="cuda")
    kv = pk.prepare_kv(k, v, fp8_qk=opts.pop("fp8_qk"), block_sparse=sparse, q_rows=Sq)
    for out in (pk.attention(q, k, v, fp8_qk=fp8, **opts), pk.attention_prepared(q, kv, **opts)):
        assert torch.equal(out, v[:, at:at + 1].expand_as(out))   # the other weights are below 2^-200 of this one


@pytest.mark.parametrize("fp8", [False, True, "pow2"])
@pytest.mark.parametrize("H,S,sparse", [(4, 1000, False), (2, 777, True), (200, 127, False), (24, 1500, True), (24, 4200, False)])
def test_output_in_the_place_of_the_queries(H, S, sparse, fp8):
    """out = q gives what a buffer of its own gives, in every form (narrow, short-key, long with a shared last round, 8-wave)."""
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(S)
    q, k, v = (_rand((1, S, H, 128), gen).cuda() for _ in range(3))
    w = (1.0 + 0.2 * torch.randn(128, generator=gen)).cuda()
    opts = dict(q_norm_weight=w, k_norm_weight=w, fp8_qk=fp8)
    if sparse:
        n = (S + 63) // 64
        opts["block_mask"] = pk.BlockMask.from_dense((torch.rand((n, n), generator=gen) < 0.5) | torch.eye(n, dtype=torch.bool), device="cuda")
    want = pk.attention(q, k, v, **opts)
    got = q.clone()
    assert pk.attention(got, k, v, out=got, **opts) is got
    torch.cuda.synchronize()
    same = _form(1, H, S, S, sparse=sparse, fp8=fp8) == _form(1, H, S, S, sparse=sparse, fp8=fp8, in_place=True)
    err, cos = _oracle().max_abs_and_cosine(got.cpu(), want.cpu())
    print(f"out = q: H={H} S={S} sparse={sparse} fp8={fp8}: same form {same}, max_abs={err:.3e} cos={cos:.7f}", flush=True)
    # another form adds the same products in another order: a bf16 step of the output at most
    assert torch.equal(got, want) if same else err <= 2.0 ** -6 * max(1.0, float(want.float().abs().max())) and cos >= 0.99999


def test_batch_stride_is_not_the_dense_one():
    """B = 3 with 264 stray elements between batch entries of q, k, v and the output (batch stride != S*H*D)."""
    _run_and_check(3, 130, 200, 2, seed=19, rope_mode=1, batch_pad=264)


@pytest.mark.parametrize("fp8", [False, True])
def test_zero_rows_with_norm_eps_zero(fp8):
    """norm_eps = 0 and an all-zero Q row and K row: the normalised rows are zeros (not 0 * inf), so the zero query
    attends uniformly (its output is the mean of V) and the zero key gets logit 0 from every query; no NaN anywhere.
    Checked against the oracle evaluated with zero rows replaced the same way."""
    import pika_h3_flex_amd as pk

    O = _oracle()
    gen = torch.Generator().manual_seed(123)
    B, Sq, Sk, H, D = 1, 150, 200, 2, 128
    q, k, v = _rand((B, Sq, H, D), gen), _rand((B, Sk, H, D), gen), _rand((B, Sk, H, D), gen)
    q[0, 17] = 0
    q[0, 149, 1] = 0
    k[0, 5] = 0
    k[0, 199, 0] = 0
    w = torch.ones(D)
    pos_q = torch.rand((Sq, 3), generator=gen, dtype=torch.float64) * 20
    pos_k = torch.rand((Sk, 3), generator=gen, dtype=torch.float64) * 20
    tq, tk = O.rope_tables(pos_q), O.rope_tables(pos_k)
    # the oracle's rms_norm gives 0 * inf = NaN on a zero row at eps = 0; the defined result is a zero row, which a
    # vanishing eps reproduces exactly for the zero rows and to 1e-30 relative for the others
    ref = O.reference_layer(q, k, v, q_norm_weight=w, k_norm_weight=w, norm_eps=1e-30, rope_q=tq, rope_k=tk, rope_mode=1,
                            fp8_qk=fp8)
    assert torch.isfinite(ref).all()
    f32 = lambda t: t.float().contiguous().cuda()
    for long_form in (False, True):
        out = pk.attention(q.cuda(), k.cuda(), v.cuda(), q_norm_weight=w.cuda(), k_norm_weight=w.cuda(), norm_eps=0.0,
                           rope_mode=1, rope_q=(f32(tq[0]), f32(tq[1])), rope_k=(f32(tk[0]), f32(tk[1])), fp8_qk=fp8,
                           long_key_kernel=long_form)
        torch.cuda.synchronize()
        out = out.cpu()
        assert torch.isfinite(out.float()).all()
        err, cos = O.max_abs_and_cosine(out, ref)
        print(f"eps=0 zero rows fp8={fp8} long_form={long_form}: max_abs={err:.3e} cos={cos:.7f}", flush=True)
        assert err <= MAX_ABS and cos >= (0.9995 if fp8 else MIN_COS)
        # the zero query row: uniform attention
        mean_v = v.double().mean(dim=1)  # [B, H, D]
        assert float((out[0, 17].double() - mean_v[0]).abs().max()) <= 1e-2


def test_batch_and_heads():
    _run_and_check(3, 130, 130, 5, seed=9)


@pytest.mark.parametrize("mode", [1, 2])
def test_rope_modes(mode):
    _run_and_check(1, 333, 333, 2, seed=40 + mode, rope_mode=mode, weight_random=True)


def test_no_norm_small_logits():
    _run_and_check(1, 256, 256, 2, seed=5, norm=False, std=0.3)


def test_key_mask_suffix_and_scattered():
    gen = torch.Generator().manual_seed(77)
    B, Sk = 2, 512
    mask = torch.zeros((B, Sk), dtype=torch.bool)
    mask[0, :137] = True                              # suffix padding
    mask[1] = torch.rand(Sk, generator=gen) < 0.4     # scattered
    _run_and_check(B, 200, Sk, 2, seed=6, mask=mask)


@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int64])
@pytest.mark.parametrize("Sk", [1, 64, 255, 257, 4096, 4097])
def test_key_masks_compacted_by_the_kv_pass_and_before_it(Sk, dtype):
    """Up to 4,096 keys the K/V pass finds the valid ones itself.  What lies in masked keys and values is never read as a number, and
    the valid ones are taken in order: the same bits as the call on them alone."""
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(Sk)
    q, k, v = (_rand((2, n, 3, 128), gen).cuda() for n in (70, Sk, Sk))
    keep = torch.rand((2, Sk), generator=gen) < 0.6
    keep[:, -1] = True
    n = int(keep.sum(1).min())
    for b in range(2):   # as many in both entries, so that one unmasked call has them all
        extra = keep[b].nonzero()[:-1, 0]
        keep[b, extra[torch.randperm(len(extra), generator=gen)[:int(keep[b].sum()) - n]]] = False
    keep = keep.cuda()
    ks, vs = (torch.stack([x[b, keep[b]] for b in range(2)]) for x in (k, v))
    k[~keep], v[~keep] = float("nan"), float("inf")
    mask = keep if dtype == torch.bool else keep.to(dtype) * 3
    got = pk.attention(q, k, v, key_mask=mask, long_key_kernel=True)
    assert torch.equal(got, pk.attention(q, ks, vs, long_key_kernel=True))
    other = pk.attention(q, k, v, key_mask=mask)
    assert (other.float() - got.float()).abs().max() <= 2 ** -7 * got.float().abs().max()   # sums in another order, rounded to bf16


@pytest.mark.parametrize("B,H,Sk", [(15, 4, 1000), (16, 4, 1000), (40, 3, 700), (17, 8, 4096)])   # the K/V pass reads the mask in the first only
def test_key_masks_of_many_entries(B, H, Sk):
    """One launch makes the lists of valid keys where the K/V pass has too many workgroups to look for them itself: every entry has the
    bits of a call of its own."""
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(B)
    q, k, v = (_rand((B, n, H, 128), gen).cuda() for n in (33, Sk, Sk))
    keep = (torch.rand((B, Sk), generator=gen) < torch.linspace(0.0, 1.0, B)[:, None]).cuda()   # from no key to all of them
    k[~keep], v[~keep] = float("nan"), float("inf")
    got = pk.attention(q, k, v, key_mask=keep, long_key_kernel=True)
    assert torch.equal(got, pk.attention_prepared(q, pk.prepare_kv(k, v, key_mask=keep, q_rows=33), long_key_kernel=True))
    for b in range(B):
        own = pk.attention(*(x[b:b + 1] for x in (q, k, v)), key_mask=keep[b:b + 1], long_key_kernel=True)
        assert torch.equal(got[b:b + 1], own) and torch.isfinite(own.float()).all()


def test_key_mask_all_valid_equals_no_mask():
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(3)
    q, k, v = (_rand((1, 100, 2, 128), gen).cuda() for _ in range(3))
    a = pk.attention(q, k, v)
    b = pk.attention(q, k, v, key_mask=torch.ones((1, 100), dtype=torch.bool, device="cuda"))
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_fully_masked_rows_are_zero():
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(4)
    q, k, v = (_rand((1, 70, 2, 128), gen).cuda() for _ in range(3))
    out = pk.attention(q, k, v, key_mask=torch.zeros((1, 70), dtype=torch.bool, device="cuda"))
    torch.cuda.synchronize()
    assert torch.count_nonzero(out) == 0


def test_strided_views_no_copy():
    """q/k/v as column slices of one fused [B, S, 3*H*D] projection output."""
    import pika_h3_flex_amd as pk

    O = _oracle()
    gen = torch.Generator().manual_seed(12)
    B, S, H, D = 1, 150, 3, 128
    qkv = _rand((B, S, 3 * H * D), gen)
    q, k, v = (qkv[..., i * H * D:(i + 1) * H * D].view(B, S, H, D) for i in range(3))
    ref = O.reference_layer(q, k, v)
    g = qkv.cuda()
    qg, kg, vg = (g[..., i * H * D:(i + 1) * H * D].view(B, S, H, D) for i in range(3))
    assert not qg.is_contiguous()
    out = pk.attention(qg, kg, vg)
    torch.cuda.synchronize()
    err, cos = O.max_abs_and_cosine(out.cpu(), ref)
    assert err <= MAX_ABS and cos >= MIN_COS


def test_rope_tables_kernel():
    import pika_h3_flex_amd as pk

    O = _oracle()
    from pika_h3_flex_amd.layout import audio_position_ids, video_position_ids

    pos = torch.cat([video_position_ids(5, 6, 7), audio_position_ids(40)], 0)
    cos, sin = pk.rope_tables(pos.cuda())
    rc, rs = O.rope_tables(pos)
    torch.cuda.synchronize()
    assert (cos.cpu().double() - rc).abs().max() < 1e-6
    assert (sin.cpu().double() - rs).abs().max() < 1e-6


# The kernel replaces the running max by a per-query logit bound |q_i| * max_j |k_j| * scale * log2(e) when that
# bound is at most 48; unit-weight QK-RMSNorm gives 16.3.  The cases below push the bound above the limit
# (norm weight x4 -> 65; un-normed N(0, 2^2) rows -> 65) so the running-max softmax path runs.  Logits are then
# +-45, where rounding Q' and K' to bf16 (which every bf16 matrix unit does) alone moves the softmax weights by
# more than the bf16 tolerance, so the oracle rounds its operands the same way (bf16_operands).
@pytest.mark.parametrize("S", [64, 200, 1000])
def test_large_logits_take_the_running_max_path(S):
    _run_and_check(1, S, S, 2, seed=300 + S, weight_scale=4.0, rope_mode=1, bf16_operands=True)


def test_large_logits_no_norm():
    _run_and_check(1, 300, 300, 2, seed=77, norm=False, std=2.0, bf16_operands=True)


def test_large_logits_with_key_mask():
    gen = torch.Generator().manual_seed(5)
    mask = torch.rand((2, 333), generator=gen) < 0.5
    _run_and_check(2, 150, 333, 2, seed=78, mask=mask, weight_scale=4.0, bf16_operands=True)


def test_both_softmax_forms_against_the_oracle_on_one_draw():
    """One seed, two regimes: unit norm weights (logit bound 16.3: the bounded-logit softmax, no running maximum)
    and weights x4 (bound 65: the running-max softmax).  Each is held to the oracle on its own inputs; the library
    has no switch that forces one form onto the other's inputs, so the two forms are never run on identical logits
    here -- `test_same_logits_through_both_softmax_forms` does that through the norm weights."""
    out_small, _ = _run_and_check(1, 500, 500, 2, seed=11, weight_scale=1.0)
    out_big, _ = _run_and_check(1, 500, 500, 2, seed=11, weight_scale=4.0, bf16_operands=True)
    assert not torch.equal(out_small, out_big)


def test_same_logits_through_both_softmax_forms():
    """The same logits through both softmax forms.  The kernel picks the form from the bound |q'| * max_j |k'_j| * scale
    (bounded-logit form up to 48 in log2 units).  The queries here are zero in their last 8 head-dim elements, and one
    extra key row is non-zero only there: its logit is exactly 0 for every query whatever its size, but its norm sets
    max|k'|.  With the extra row all zero the bound is 16 and the bounded-logit form runs; with 300 in those 8
    elements the bound is beyond 1000 and the running-max form runs -- on identical logits and values.  Both are held
    to the oracle and must agree with each other to the rounding of the bf16 output."""
    import pika_h3_flex_amd as pk

    O = _oracle()
    gen = torch.Generator().manual_seed(29)
    B, S, H, D = 1, 400, 2, 128
    q, k, v = _rand((B, S, H, D), gen), _rand((B, S + 1, H, D), gen), _rand((B, S + 1, H, D), gen)
    q[..., 120:] = 0
    k[:, S] = 0
    k_big = k.clone()
    k_big[:, S, :, 120:] = 300.0
    w = torch.ones(D)
    ref = O.reference_layer(q, k, v, q_norm_weight=w)
    assert float((ref - O.reference_layer(q, k_big, v, q_norm_weight=w)).abs().max()) == 0.0  # the oracle sees no difference
    for long_form in (False, True):
        bounded = pk.attention(q.cuda(), k.cuda(), v.cuda(), q_norm_weight=w.cuda(), long_key_kernel=long_form)
        running = pk.attention(q.cuda(), k_big.cuda(), v.cuda(), q_norm_weight=w.cuda(), long_key_kernel=long_form)
        torch.cuda.synchronize()
        e1, c1 = O.max_abs_and_cosine(bounded.cpu(), ref)
        e2, c2 = O.max_abs_and_cosine(running.cpu(), ref)
        e12, c12 = O.max_abs_and_cosine(bounded.cpu(), running.cpu())
        print(f"long_form={long_form}: bounded vs oracle {e1:.3e}/{c1:.7f}; running-max vs oracle {e2:.3e}/{c2:.7f}; "
              f"between them {e12:.3e}/{c12:.7f}", flush=True)
        assert e1 <= MAX_ABS and c1 >= MIN_COS and e2 <= MAX_ABS and c2 >= MIN_COS
        assert e12 <= 8e-3 and c12 >= 0.99999


@pytest.mark.parametrize("variant", ["dense_rope_mask", "sparse_fp8", "long_dense_shared_last_round"])
def test_hip_graph_replays_match_eager(variant):
    """The layer call allocates nothing and only launches kernels on the caller's stream, so it can be captured
    into a HIP graph.  Every replay, with fresh inputs in the captured buffers and eager work in between, must
    give the bits of an eager call on the same inputs."""
    import pika_h3_flex_amd as pk

    B, S, H, D = 1, 333, 2, 128
    if variant == "long_dense_shared_last_round":
        S, H = 4200, 24  # 264 query tiles on a 256-CU part: the counter fill, then one launch whose last 8 tiles are shared two ways
    gen = torch.Generator().manual_seed(91)
    dev = "cuda"
    q, k, v = (_rand((B, S, H, D), gen).to(dev) for _ in range(3))
    w = torch.ones(D, device=dev)
    opts = dict(q_norm_weight=w, k_norm_weight=w)
    if variant == "dense_rope_mask":
        pos = torch.rand((S, 3), generator=gen, dtype=torch.float64) * 20.0
        cos, sin = pk.rope_tables(pos.to(dev))
        mask = (torch.rand((B, S), generator=gen) < 0.7).to(dev)
        opts.update(rope_mode=1, rope_q=(cos, sin), key_mask=mask)
    elif variant == "long_dense_shared_last_round":
        pass
    else:
        tm = torch.rand((6, 6), generator=gen) < 0.5
        tm |= torch.eye(6, dtype=torch.bool)
        opts.update(block_mask=pk.BlockMask.from_dense(tm, device=dev), fp8_qk=True)
    out = torch.empty_like(q)
    ws = torch.empty(1 << 27, dtype=torch.uint8, device=dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        pk.attention(q, k, v, out=out, workspace=ws, **opts)  # warm-up outside the capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pk.attention(q, k, v, out=out, workspace=ws, **opts)
    for rep in range(4):
        fresh = [_rand((B, S, H, D), gen).to(dev) for _ in range(3)]
        eager = pk.attention(*fresh, **opts).clone()
        torch.cuda.synchronize()
        for dst, src in zip((q, k, v), fresh):
            dst.copy_(src)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep} differs from the eager call"


@pytest.mark.parametrize("variant", ["cross_masked", "rope_fp8", "long_keys", "block_sparse"])
def test_prepared_keys_serve_several_calls(variant):
    """pkh3_kv_prepare once, then attention calls with different queries (and query counts) on the prepared
    workspace: each must give the bits of the ordinary call on the same q, k, v."""
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(17)
    dev = "cuda"
    B, H, D = (2, 2, 128) if variant == "cross_masked" else (1, 3, 128)
    Sk = {"cross_masked": 100, "rope_fp8": 333, "long_keys": 1500, "block_sparse": 700}[variant]
    k, v = (_rand((B, Sk, H, D), gen).to(dev) for _ in range(2))
    wq = (1.0 + 0.1 * torch.randn(D, generator=gen)).to(dev)
    wk = (1.0 + 0.1 * torch.randn(D, generator=gen)).to(dev)
    k_opts = dict(k_norm_weight=wk)
    if variant == "cross_masked":
        k_opts.update(key_mask=(torch.rand((B, Sk), generator=gen) < 0.6).to(dev))
    tabs_k = None
    if variant == "rope_fp8":
        tabs_k = pk.rope_tables((torch.rand((Sk, 3), generator=gen, dtype=torch.float64) * 20).to(dev))
        k_opts.update(rope_mode=pk.ROPE_INTERLEAVED, rope_k=tabs_k, fp8_qk=True)
    kv = pk.prepare_kv(k, v, q_rows=700, block_sparse=(variant == "block_sparse"), **k_opts)
    for Sq in (77, 700, 300):
        q = _rand((B, Sq, H, D), gen).to(dev)
        q_opts = dict(q_norm_weight=wq)
        if variant == "block_sparse":  # every call brings its own tile map
            tm = torch.rand(((Sq + 63) // 64, (Sk + 63) // 64), generator=gen) < 0.5
            q_opts.update(block_mask=pk.BlockMask.from_dense(tm, device=dev))
        if variant == "rope_fp8":
            q_opts.update(rope_q=pk.rope_tables((torch.rand((Sq, 3), generator=gen, dtype=torch.float64) * 20).to(dev)))
        got = pk.attention_prepared(q, kv, **q_opts)
        want = pk.attention(q, k, v, **k_opts, **q_opts)
        torch.cuda.synchronize()
        assert torch.isfinite(got.float()).all()
        assert torch.equal(got, want), f"{variant} Sq={Sq}: prepared keys give different bits"
    with pytest.raises(ValueError, match="K-side"):
        pk.attention_prepared(q, kv, k_norm_weight=wk, **q_opts)
    with pytest.raises(ValueError, match="heads"):
        pk.attention_prepared(_rand((B, Sq, H + 1, D), gen).to(dev), kv, **q_opts)


@pytest.mark.parametrize("B,H,Sq,Sk,fp8", [
    (1, 1, 64, 64, False),       # one entry beside two workgroups of tiles
    (3, 2, 257, 190, True),       # entries ride once, not once per batch; the last one holds one row-block of four
    (2, 1, 4097, 130, True),      # more entries than tiles
    (1, 1, 70, 64 * 8192 + 65, False),  # key tiles past one round of the masks
])
def test_tile_lists_made_beside_the_kv_pass(B, H, Sq, Sk, fp8):
    """Direct calls make the tile lists in the K/V pass's launch, calls on prepared keys in a launch of their own: the same bits."""
    import pika_h3_flex_amd as pk

    gen = torch.Generator().manual_seed(Sq + Sk)
    q, k, v = (_rand((B, n, H, 128), gen).cuda() for n in (Sq, Sk, Sk))
    nq, nk = -(-Sq // 64), -(-Sk // 64)
    tiles = torch.rand((nq, nk), generator=gen) < 0.4
    tiles[:, 0] = tiles[:, -1] = True
    bm = pk.BlockMask.from_dense(tiles, device="cuda")
    opts = dict(fp8_qk=fp8)
    kv = pk.prepare_kv(k, v, q_rows=Sq, block_sparse=True, **opts)
    want = pk.attention_prepared(q, kv, block_mask=bm)
    assert torch.isfinite(want.float()).all()
    assert torch.equal(pk.attention(q, k, v, block_mask=bm, **opts), want)


def test_prepared_keys_workspace_holds_dense_and_block_sparse_calls():
    """Keys prepared with ``block_sparse=True`` at a size where long dense calls bring scratch of their own (the partial
    results of a shared last round): the workspace must hold either kind of call, and both must give the bits of the
    direct calls."""
    import pika_h3_flex_amd as pk

    B, S, H, D = 1, 1500, 24, 128
    gen = torch.Generator().manual_seed(17)
    dev = "cuda"
    q, k, v = (_rand((B, S, H, D), gen).to(dev) for _ in range(3))
    w = torch.ones(D, device=dev)
    kv = pk.prepare_kv(k, v, q_rows=S, block_sparse=True, k_norm_weight=w)
    nt = (S + 63) // 64
    tm = (torch.rand((nt, nt), generator=gen) < 0.4) | torch.eye(nt, dtype=torch.bool)
    bm = pk.BlockMask.from_dense(tm, device=dev)
    dense = pk.attention_prepared(q, kv, q_norm_weight=w)
    sparse = pk.attention_prepared(q, kv, q_norm_weight=w, block_mask=bm)
    torch.cuda.synchronize()
    assert torch.equal(dense, pk.attention(q, k, v, q_norm_weight=w, k_norm_weight=w))
    assert torch.equal(sparse, pk.attention(q, k, v, q_norm_weight=w, k_norm_weight=w, block_mask=bm))
