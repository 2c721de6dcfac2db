"""What the planner of the attention launches decides, on the CPU: pointers are made up, nothing is launched."""
import ctypes as C

import pytest

import jittorinfer_amd.capi as J

BF16, F16, Q8_0 = J.MLA_TYPE_BF16, J.MLA_TYPE_F16, J.MLA_TYPE_Q8_0


def _args(n_seq, n_tok, n_head, keys, kv_type=BF16, paged=True, mask_width=0, dv=512, flags=0, n_splits=0):
    """The argument block of a launch over `keys` cells per sequence; mask_width 0: no mask."""
    a = J.MlaAttnArgs()
    a.n_seq, a.n_head, a.n_tok, a.dk, a.dv = n_seq, n_head, n_tok, 576, dv
    a.q_type, a.kv_type, a.flags, a.scale, a.n_splits = J.MLA_TYPE_F32, kv_type, flags, 0.07, n_splits
    a.q, a.kv, a.dst = 1 << 20, 1 << 30, 1 << 31
    a.q_nb2, a.q_nb1, a.q_nb3 = 2304, 2304 * n_head, 2304 * n_head * n_tok
    a.kv_nb1, a.dst_nb1 = J.ROW_BYTES[kv_type], dv * 4
    if paged:
        a.bt_stride = (keys + 127) // 128
        a.n_kv, a.block_table, a.seq_lens = n_seq * a.bt_stride * 128, 1 << 20, 1 << 20
    else:
        a.n_kv, a.kv_nb3 = keys, a.kv_nb1 * keys if n_seq > 1 else 0
    if mask_width:
        a.mask, a.mask_nb1, a.mask_ne0 = 1 << 20, mask_width * 2, mask_width
    return a


def _plan(*args, **kw):
    info = J.MlaPlanInfo()
    a = _args(*args, **kw)
    assert J.library().mla_attn_plan(C.byref(a), C.byref(info)) == 0
    return info


def _workspace(*args, **kw):
    a = _args(*args, **kw)
    return J.library().mla_attn_workspace_size(C.byref(a))


@pytest.mark.parametrize("kv_type", [BF16, F16, Q8_0])
@pytest.mark.parametrize("n_seq,n_tok,n_head", [(1, 9, 16), (2, 9, 16), (1, 64, 128), (3, 2, 16)])
def test_a_mask_narrower_than_a_contiguous_cache_is_the_general_kernel_s(kv_type, n_seq, n_tok, n_head):
    """It multiplies the cells as they are, with both halves of the probabilities, and keeps small partials in f32."""
    assert _plan(n_seq, n_tok, n_head, 4096, kv_type, paged=False, mask_width=2048).variant == 0
    assert _plan(n_seq, n_tok, n_head, 4096, kv_type, paged=False, mask_width=4096).variant == 2
    assert _plan(n_seq, n_tok, n_head, 4096, kv_type, paged=False, mask_width=8192).variant == 2
    assert _workspace(n_seq, n_tok, n_head, 4096, kv_type, paged=False, mask_width=2048) <= J.MLA_ATTN_STATIC_WORKSPACE_MAX


@pytest.mark.parametrize("kv_type", [BF16, F16])
@pytest.mark.parametrize("n_seq,n_tok,n_head,dv,n_pages", [(256, 1, 128, 576, 66), (4, 1661, 48, 576, 265), (278, 1, 24, 512, 128)])
def test_narrow_masks_over_many_pages_gain_no_f16_partial_rows(kv_type, n_seq, n_tok, n_head, dv, n_pages):
    """Where the general kernel has whole rows or f32 partials.  With fewer pages the pipelined kernel has too, and takes them."""
    assert _plan(n_seq, n_tok, n_head, n_pages * 128, kv_type, mask_width=n_pages * 128 - 32, dv=dv).variant == 0
    assert _plan(n_seq, n_tok, n_head, 20 * 128, kv_type, mask_width=20 * 128 - 32, dv=dv).variant == 2


@pytest.mark.parametrize("kv_type", [BF16, F16, Q8_0])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("n_tok,n_head", [(1, 16), (2, 16), (4, 16), (1, 64), (1, 96), (3, 1), (1, 97), (1, 128), (1, 130), (3, 48)])
def test_a_tail_only_where_the_kernel_has_a_build_for_it(kv_type, paged, n_tok, n_head):
    """300 masked sequences: 44 row blocks (or 88 of the two-block ones) beyond whole rounds of 256.  Column-split programs and Q8_0 tiles."""
    n_blocks = 300 * ((n_tok * n_head + 127) // 128)
    has_build = kv_type == Q8_0 or n_tok * n_head > 96
    assert (_plan(300, n_tok, n_head, 2048, kv_type, paged=paged, mask_width=2048).n_workgroups > n_blocks) == has_build


@pytest.mark.parametrize("kv_type", [BF16, F16, Q8_0])
@pytest.mark.parametrize("n_tok", [257, 300, 356, 384, 464, 470, 480, 490, 511, 1000])
def test_a_tail_s_partial_rows_are_bounded(kv_type, n_tok):
    """A prompt chunk of n_tok row blocks behind 65536 cells: the tail adds at most 128 MB (and (m, l) pairs) to what the launch takes without."""
    kw = dict(paged=False, mask_width=65536)
    more = _workspace(1, n_tok, 128, 65536, kv_type, **kw) - _workspace(1, n_tok, 128, 65536, kv_type, flags=J.MLA_FLAG_UNIFORM_SPLITS, **kw)
    assert 0 <= more <= (128 << 20) + 512 * 128 * 8 + 512


def test_a_launch_of_many_rounds_has_no_tail():
    for n_tok, tail in ((256 + 40, True), (11 * 256 + 40, True), (12 * 256 + 40, False), (20 * 256 + 40, False)):
        assert (_plan(1, n_tok, 128, 8192, F16, paged=False, mask_width=8192).n_workgroups > n_tok) == tail


@pytest.mark.parametrize("n_seq,n_tok,n_head,keys,paged", [(73, 2, 24, 24352, False), (157, 3, 16, 11904, True), (66, 1, 48, 18176, True), (2, 17, 16, 16896, False)])
def test_more_splits_of_a_masked_launch_keep_f32_partials(n_seq, n_tok, n_head, keys, paged):
    """Where as many splits as give every CU a workgroup have f32 partials, the splits taken instead have too."""
    kw = dict(paged=paged, mask_width=keys)
    splits, rows = _plan(n_seq, n_tok, n_head, keys, F16, **kw).n_splits, n_tok * n_head
    assert splits > 1 and _workspace(n_seq, n_tok, n_head, keys, F16, **kw) >= n_seq * splits * rows * 512 * 4
@pytest.mark.parametrize("n_seq,n_tok,n_head,kv_type", [(1, 2, 64, BF16), (2, 8, 16, BF16), (1, 8, 16, Q8_0), (1, 4, 128, F16), (7, 1, 128, BF16)])
def test_few_tokens_behind_a_long_context_fill_the_chip(n_seq, n_tok, n_head, kv_type):
    """Masked row blocks over pages: 32 workgroups each leave most CUs idle."""
    blocks = n_seq * ((n_tok * n_head + 127) // 128)
    assert 128 <= _plan(n_seq, n_tok, n_head, 65536, kv_type, mask_width=65536).n_workgroups <= 256 + blocks
    assert _plan(n_seq, n_tok, n_head, 2048, kv_type, mask_width=2048).n_workgroups == 16 * blocks   # a page each
