"""Which form of the attention kernel a call takes on a part of 256 CUs: the dispatch rule alone, no GPU needed."""
import ctypes as C

import pytest

from pika_h3_flex_amd import _lib

LONG, SHORT, NARROW, SPARSE = _lib.FORM_LONG, _lib.FORM_SHORT, _lib.FORM_NARROW, _lib.FORM_SPARSE


def form(B, H, Sq, Sk, *, sparse=False, masked=False, fp8=False, long_key_kernel=False, cus=256):
    a = _lib.AttnArgs()
    a.B, a.H, a.Sq, a.Sk, a.D = B, H, Sq, Sk, 128
    a.flags = ((_lib.FLAG_FP8_QK if fp8 else 0) | (_lib.FLAG_FP8_POW2_SCALES if fp8 == "pow2" else 0)
               | (_lib.FLAG_LONG_KEY_KERNEL if long_key_kernel else 0))
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
    assert form(3, 8, 777, 777, masked=True) == SHORT and form(1, 24, 49640, 512, masked=True) == SHORT


def test_form_of_a_bad_call_is_an_error():
    with pytest.raises(_lib.Pkh3Error):
        form(0, 1, 1, 1)
