"""Which form of the attention kernel a call takes on a part of 256 CUs: the dispatch rule alone, no GPU needed."""
import ctypes as C

import pytest

from pika_h3_flex_amd import _lib

# Dense calls of the short-key form (B, H, Sq, Sk, key mask), with one, two and three of its workgroups on a CU, on at most and on more than
# 16 key tiles; the GPU tests run them against the oracle.
SHORT_KEY_CALLS = [(1, 64, 250, 97, False), (1, 200, 127, 700, False), (1, 200, 128, 1089, False), (1, 150, 250, 1100, False),
                   (1, 260, 129, 1057, False), (2, 130, 100, 700, True), (2, 130, 97, 1100, True)]

LONG, SHORT, NARROW, SPARSE, RELAY = _lib.FORM_LONG, _lib.FORM_SHORT, _lib.FORM_NARROW, _lib.FORM_SPARSE, _lib.FORM_RELAY


def form(B, H, Sq, Sk, *, sparse=False, masked=False, fp8=False, long_key_kernel=False, in_place=False, rope=0, cus=256):
    a = _lib.AttnArgs()
    a.B, a.H, a.Sq, a.Sk, a.D = B, H, Sq, Sk, 128
    a.flags = ((_lib.FLAG_FP8_QK if fp8 else 0) | (_lib.FLAG_FP8_POW2_SCALES if fp8 == "pow2" else 0)
               | (_lib.FLAG_LONG_KEY_KERNEL if long_key_kernel else 0))
    a.rope_mode = rope
    if in_place:
        a.q = a.o = 0x10000   # (as the rest, never dereferenced here)
    if sparse:
        a.blk_row_ptr = a.blk_col_idx = 0x10000   # never dereferenced here
    if masked:
        a.key_mask = 0x10000
    got = _lib.load_bench().pkh3_attn_form(C.byref(a), cus)
    _lib.check(min(got, 0))
    return got


@pytest.mark.parametrize("fp8", [False, True, "pow2"])
@pytest.mark.parametrize("B,H,Sq,Sk,want", [
    (1, 1, 1, 1, NARROW), (1, 24, 641, 641, NARROW), (1, 24, 900, 900, NARROW), (1, 24, 1085, 1085, NARROW),
    (1, 24, 1344, 1344, NARROW), (1, 8, 4096, 4096, NARROW), (2, 4, 4096, 300, NARROW),          # 32-query blocks up to four per CU
    (1, 24, 1345, 1345, SPARSE), (1, 10, 4096, 3040, SPARSE), (1, 8, 4097, 64, SPARSE), (1, 24, 48360, 48360, SPARSE),
    (1, 10, 4096, 3041, "fp8"), (1, 10, 4097, 4097, SPARSE),                                     # of many keys in fp8: up to five
])
def test_block_sparse_calls_go_by_their_query_blocks(B, H, Sq, Sk, want, fp8):
    if want == "fp8":
        want = NARROW if fp8 else SPARSE
    assert form(B, H, Sq, Sk, sparse=True, fp8=fp8) == want
    assert form(B, H, Sq, Sk, sparse=True, fp8=fp8, long_key_kernel=True) == SPARSE


def test_masked_calls_go_by_the_padded_keys():
    """(The valid ones are counted on the device: test_masked_calls_of_few_and_many_valid_keys in the GPU tests runs these.)"""
    assert form(3, 24, 200, 400, masked=True) == form(3, 24, 500, 2040, masked=True) == NARROW
    assert form(3, 8, 777, 777, masked=True) == SHORT and form(1, 24, 49640, 512, masked=True) == form(2, 24, 14830, 2560, masked=True) == RELAY


@pytest.mark.parametrize("B,H,Sq,Sk,masked", SHORT_KEY_CALLS)
def test_calls_of_the_short_key_form(B, H, Sq, Sk, masked):
    for fp8 in (False,) if masked else (False, True, "pow2"):
        assert form(B, H, Sq, Sk, masked=masked, fp8=fp8) == SHORT
        assert form(B, H, Sq, Sk, masked=masked, fp8=fp8, long_key_kernel=True) == LONG


@pytest.mark.parametrize("B,H,Sq,Sk,want", [
    (1, 4, 1024, 1024, NARROW), (1, 24, 641, 1089, NARROW), (1, 24, 1085, 1085, SHORT),   # a small call; the attention of one image
    (1, 24, 3008, 3008, LONG), (1, 24, 4000, 4000, SHORT),   # three short-key workgroups per CU; long ones: 192 and 264 on 256 CUs
    (1, 24, 49640, 512, RELAY), (1, 24, 14830, 1024, RELAY), (1, 24, 14830, 1025, RELAY), (1, 24, 48360, 48360, LONG),
])
def test_dense_calls_go_by_their_workgroups_and_keys(B, H, Sq, Sk, want):
    assert form(B, H, Sq, Sk) == want


@pytest.mark.parametrize("B,H,Sq,Sk,want,rotated", [
    (1, 24, 49640, 448, SHORT, SHORT), (1, 24, 49640, 449, RELAY, SHORT), (1, 24, 49640, 1024, RELAY, SHORT),   # 7 | 8 .. 16 | 17 .. 40 | 41 tiles
    (1, 24, 49640, 1025, RELAY, RELAY), (1, 24, 49640, 2560, RELAY, RELAY), (1, 24, 49640, 2561, LONG, LONG),
    (1, 32, 4096, 1024, SHORT, SHORT), (1, 32, 4096, 1025, LONG, LONG), (1, 33, 4096, 1025, RELAY, RELAY),       # four units a CU and 32 more
    (1, 28, 16384, 1024, RELAY, SHORT), (1, 28, 16385, 1024, RELAY, SHORT),                                       # (masked: 14 units a CU and 28 more)
    (1, 24, 6500, 512, RELAY, SHORT), (4, 2, 18000, 1024, RELAY, SHORT),                                          # whole heads for eight XCDs
    (1, 31, 5248, 832, SHORT, SHORT), (1, 31, 5248, 1088, RELAY, RELAY), (1, 31, 6912, 1024, RELAY, SHORT),       # ... and not, below and above 6.5 a CU
    (1, 208, 1024, 1024, SHORT, SHORT), (1, 319, 1024, 1024, SHORT, SHORT), (1, 321, 1024, 1024, RELAY, SHORT),   # heads of eight units: ten a CU
    (1, 185, 1152, 1024, RELAY, SHORT), (1, 184, 1152, 1024, RELAY, SHORT), (1, 183, 1152, 1024, SHORT, SHORT),   # ... of nine
    (1, 256, 3456, 1792, RELAY, RELAY), (1, 256, 3456, 1793, LONG, LONG), (1, 256, 3328, 1793, LONG, LONG),       # 7,168 tiles of all heads
    (1, 256, 1280, 1793, RELAY, RELAY), (4, 100, 396, 1395, RELAY, RELAY),                                        # ... and blocks of 384 rows not full
])
def test_calls_of_the_relay_form(B, H, Sq, Sk, want, rotated):
    few = Sk <= 1024 and B * H * ((Sq + 127) // 128) <= 14 * 256
    assert form(B, H, Sq, Sk) == form(B, H, Sq, Sk, in_place=True) == want
    assert form(B, H, Sq, Sk, masked=True) == (SHORT if few else want)
    assert form(B, H, Sq, Sk, rope=1) == form(B, H, Sq, Sk, rope=2) == rotated
    assert form(B, H, Sq, Sk, fp8=True) in (SHORT, LONG) and form(B, H, Sq, Sk, fp8="pow2") in (SHORT, LONG)
    assert form(B, H, Sq, Sk, long_key_kernel=True) == LONG and form(B, H, Sq, Sk, sparse=True) == SPARSE
    assert form(B, H, Sq, Sk, cus=7) in (SHORT, LONG)


@pytest.mark.parametrize("Sq", [33, 64, 1000])
@pytest.mark.parametrize("fp8", [True, "pow2"])
def test_fp8_calls_in_place_are_not_narrow(Sq, fp8):
    """A narrow workgroup reads 64 queries for their scale and writes 32: out = q would be a race between neighbours."""
    assert form(1, 4, Sq, Sq, fp8=fp8) == form(1, 4, Sq, Sq, sparse=True, fp8=fp8) == form(1, 4, Sq, Sq, in_place=True) == NARROW
    assert form(1, 4, Sq, Sq, fp8=fp8, in_place=True) == SHORT
    assert form(1, 4, Sq, Sq, sparse=True, fp8=fp8, in_place=True) == SPARSE


def test_form_of_a_bad_call_is_an_error():
    with pytest.raises(_lib.Pkh3Error):
        form(0, 1, 1, 1)
