"""Launch shapes at the edges of the dispatch rules of the attention kernels, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import util as U
from tests.test_edge_gpu import _want
from tests.test_parity_gpu import _plan_variant, _run

pytestmark = pytest.mark.gpu


def _causal_mask(n_new, lens_max, width):
    """f16 bits [n_new, width]: new token t sees keys up to lens_max - n_new + t."""
    return np.where(np.arange(width)[None, :] > lens_max - n_new + np.arange(n_new)[:, None], -np.inf, 0.0).astype(np.float16).view(np.uint16)


@pytest.mark.parametrize("k_type", [O.TYPE_BF16, O.TYPE_F16, O.TYPE_Q8_0])
@pytest.mark.parametrize("n_head,n_new,n_old,width", [(16, 9, 150, 160), (128, 3, 157, 160), (48, 5, 288, 320), (16, 2, 129, 96)])
def test_mask_rows_narrower_than_the_block_table(gpu, k_type, n_head, n_new, n_old, width):
    """Paged prompt chunks whose mask rows end before the last page does (and, in the last case, before the sequences do: the keys
    past the rows' end count as masked) run on the pipelined kernel."""
    rng = np.random.default_rng(n_head + n_new + width)
    lens = [n_old + n_new, n_old + n_new - 1]
    pool, bt, seqs = U.make_paged(rng, lens, k_type, q8_scale=1.0 / 32 if k_type == O.TYPE_Q8_0 else None)
    q = rng.standard_normal((2, n_head, n_new, 576)).astype(np.float32)
    mask = _causal_mask(n_new, max(lens), width)
    assert width < bt.shape[1] * 128
    assert _plan_variant(gpu, q, pool, k_type, mask, bt, lens, scale=U.SCALE) == 2
    got = _run(gpu, q, pool, k_type, mask=mask, bt=bt, lens=lens, scale=U.SCALE)
    print(U.check(got[..., :512], _want(q, [s[:width] for s in seqs], k_type, mask), "narrow mask rows"))


@pytest.mark.parametrize("k_type", [O.TYPE_BF16, O.TYPE_F16])
@pytest.mark.parametrize("n_head,n_new", [(43, 3), (80, 2), (24, 8), (32, 7), (16, 17)])   # 129, 160, 192, 224, 272 rows
@pytest.mark.parametrize("masked", [False, True])
def test_row_blocks_of_which_the_last_is_not_full(gpu, k_type, n_head, n_new, masked):
    """Two or three row blocks, 1 to 96 rows in the last: waves without rows beside blocks of 128."""
    rng = np.random.default_rng(n_head * n_new)
    n_kv = 224
    q = rng.standard_normal((2, n_head, n_new, 576)).astype(np.float32)
    k = U.encode_kv(rng.standard_normal((2, n_kv, 576)).astype(np.float32), k_type)
    mask = _causal_mask(n_new, n_kv, n_kv) if masked else None
    got = _run(gpu, q, k, k_type, mask=mask, scale=U.SCALE)
    print(U.check(got[..., :512], _want(q, list(k), k_type, mask), "last row block not full"))


@pytest.mark.parametrize("k_type", [O.TYPE_BF16, O.TYPE_F16, O.TYPE_Q8_0])
@pytest.mark.parametrize("n_seq,n_head,n_new,n_old,dv", [(1, 128, 257, 350, 512), (1, 128, 290, 352, 576), (1, 48, 693, 300, 512), (3, 16, 691, 250, 512)])
def test_row_blocks_left_over_from_whole_rounds_are_split(gpu, k_type, n_seq, n_head, n_new, n_old, dv):
    """257, 290, 260 and 3 x 87 row blocks: the 1, 34, 4 and 5 beyond 256 are split over several workgroups each (paged, several sequences
    of different lengths: the tail lies in the last one).  One token of the tail sees no key: NaN rows.  Checked on sampled rows, the
    tail's among them, and everywhere against the launch that does not split (same arithmetic but for the merge: f16 or f32 partials,
    within the tolerance of the oracle)."""
    import torch
    import jittorinfer_amd as J
    rng = np.random.default_rng(n_new + n_seq)
    lens = [n_old + n_new - 40 * b for b in range(n_seq)]
    q8s = 1.0 / 32 if k_type == O.TYPE_Q8_0 else None
    width = (max(lens) + 127) // 128 * 128 if n_seq > 1 else (max(lens) + 31) // 32 * 32
    q = rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)
    if n_seq > 1:
        pool, bt, seqs = U.make_paged(rng, lens, k_type, q8_scale=q8s)
        kw = dict(bt=bt, lens=lens)
    else:
        pool = U.encode_kv(rng.standard_normal((1, width, 576)).astype(np.float32), k_type, q8_scale=q8s)
        seqs, kw = [pool[0]], {}
    mask = _causal_mask(n_new, max(lens), width).copy()
    mask[n_new - 1] = 0xfc00
    tq = torch.from_numpy(q).to(gpu)
    pkw = dict(mask=torch.from_numpy(mask.view(np.float16)).to(gpu), scale=U.SCALE)
    if n_seq > 1:
        pkw.update(block_table=torch.from_numpy(bt).to(gpu), seq_lens=torch.tensor(lens, dtype=torch.int32, device=gpu))
    tp = torch.from_numpy(pool.view(np.int16) if pool.dtype == np.uint16 else pool).to(gpu)
    n_items = n_seq * ((n_head * n_new + 127) // 128)
    info = J.plan(tq, tp, k_type, dv=dv, **pkw)
    assert info["variant"] == 2 and info["n_splits"] == 1 and info["n_workgroups"] > n_items > 256, info
    assert J.plan(tq, tp, k_type, dv=dv, flags=J.MLA_FLAG_UNIFORM_SPLITS, **pkw)["n_workgroups"] == n_items
    got = _run(gpu, q, pool, k_type, dv=dv, mask=mask, scale=U.SCALE, **kw)[..., :dv]
    one = _run(gpu, q, pool, k_type, dv=dv, mask=mask, scale=U.SCALE, flags=J.MLA_FLAG_UNIFORM_SPLITS, **kw)[..., :dv]
    print(U.check(got, one, "split against unsplit"))
    for b in range(n_seq):
        for t in (0, n_new // 2, n_new - 3, n_new - 2, n_new - 1):
            want = (O.flash_attn_ext_f64 if k_type == O.TYPE_F16 else O.flash_attn_ext)(
                q[b:b + 1, :, t:t + 1], seqs[b][None, :width], k_type, dv=dv, mask=np.ascontiguousarray(mask[t:t + 1, :len(seqs[b])]), scale=U.SCALE)
            print(b, t, U.check(got[b:b + 1, t:t + 1], want, "sequence %d token %d" % (b, t)))


@pytest.mark.parametrize("k_type", [O.TYPE_BF16, O.TYPE_F16])
@pytest.mark.parametrize("n_head,groups", [(34, 2), (64, 2), (66, 2), (96, 2), (100, 4), (128, 4), (128, 2), (35, 1)])
@pytest.mark.parametrize("paged", [False, True])
def test_heads_of_a_short_decode_step_in_groups(gpu, k_type, n_head, groups, paged):
    """More than 32 heads over few keys: groups of up to 32 (or 64) heads as sequences of their own on the same keys, Q with strides that
    are not packed; ragged lengths with an empty sequence, the balanced page schedule and single pages; both passes of a 576-wide V."""
    import torch
    import jittorinfer_amd as J
    rng = np.random.default_rng(n_head + groups)
    if groups == 2 and n_head > 64:
        lens = [2500, 900, 33, 1700] if paged else [2500] * 4      # too many tiles for groups of 32
    else:
        lens = [0, 129, 300, 31, 640, 1] if paged else [416] * 3
    n_seq = len(lens)
    if paged:
        pool, bt, seqs = U.make_paged(rng, np.maximum(lens, 1), k_type)
        seqs = [s[:l] for s, l in zip(seqs, lens)]
        kw = dict(bt=bt, lens=lens)
        pkw = dict(block_table=torch.from_numpy(bt).to(gpu), seq_lens=torch.tensor(lens, dtype=torch.int32, device=gpu))
    else:
        pool = U.encode_kv(rng.standard_normal((n_seq, lens[0], 576)).astype(np.float32), k_type)
        seqs, kw, pkw = list(pool), {}, {}
    q = rng.standard_normal((n_seq, n_head, 1, 576)).astype(np.float32)
    info = J.plan(torch.from_numpy(q).to(gpu), torch.from_numpy(pool.view(np.int16)).to(gpu), k_type, dv=512, scale=U.SCALE, **pkw)
    assert info["variant"] == 2 and (info["balanced"] == 1 or info["n_workgroups"] == groups * n_seq * info["n_splits"]), info
    for dv in (512, 576):
        got = _run(gpu, q, pool, k_type, dv=dv, scale=U.SCALE, **kw)[..., :dv]
        for b in range(n_seq):
            if len(seqs[b]) == 0:
                assert np.isnan(got[b]).all()
            else:
                want = (O.flash_attn_ext_f64 if k_type == O.TYPE_F16 else O.flash_attn_ext)(q[b:b + 1], seqs[b][None], k_type, dv=dv, scale=U.SCALE)
                print(dv, b, U.check(got[b:b + 1], want, "sequence %d" % b))
    tq = torch.from_numpy(np.ascontiguousarray(q.transpose(1, 0, 2, 3))).to(gpu).permute(1, 0, 2, 3)   # [head][sequence] in memory
    tp = torch.from_numpy(pool.view(np.int16)).to(gpu)
    a = J.ggml_flash_attn_ext(tq, tp, k_type, dv=512, scale=U.SCALE, **pkw)[..., :512]
    b = J.ggml_flash_attn_ext(torch.from_numpy(q).to(gpu), tp, k_type, dv=512, scale=U.SCALE, **pkw)[..., :512]
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


def test_narrow_mask_rows_of_bf16_cells_keep_both_halves_of_the_probabilities(gpu):
    """Probabilities as hi + lo bf16 halves carry 16 bits (errors of 2^-18 on average), one f16 probability 11 (2^-13, 1.4e-4 in relative L2
    over a row): 3e-5 lies between.  And cells beyond the range of f16 are multiplied as they are."""
    rng = np.random.default_rng(3)
    n_head, n_new, width = 16, 9, 160
    lens = [n_new + 150, n_new + 149]
    for big in (False, True):
        pool, bt, seqs = U.make_paged(rng, lens, O.TYPE_BF16)
        q = rng.standard_normal((2, n_head, n_new, 576)).astype(np.float32)
        if big:   # value columns 500 .. 511 of every cell at 2^20 and above; Q is 0 there
            for x in (pool, *seqs):
                x[..., 500:512] = (x[..., 500:512] & 0x807f) | 0x4980
            q[..., 500:512] = 0
        mask = _causal_mask(n_new, max(lens), width)
        got = _run(gpu, q, pool, O.TYPE_BF16, mask=mask, bt=bt, lens=lens, scale=U.SCALE)[..., :512]
        want = _want(q, [s[:width] for s in seqs], O.TYPE_BF16, mask)
        print(U.check(got, want, "narrow mask rows", max_abs=2.0 ** 21 if big else 2e-4, rel_l2=3e-5))


@pytest.mark.parametrize("n_seq,n_new,width,paged", [(1, 290, 640, False), (2, 288, 31968, True)])
def test_static_scratch_takes_what_fits_without_the_rows_that_only_save_time(gpu, n_seq, n_new, width, paged):
    """290 row blocks whose tail's partial rows do not fit the fixed scratch beside the operand image, and 2 x 36 behind narrow mask rows whose
    seven splits do not: both run, as the launch that needs neither."""
    import ctypes as C
    import torch
    import jittorinfer_amd as J
    lib = J.library()
    rng = np.random.default_rng(n_new)
    n_head = 16 if paged else 128
    lens = [width - 3] * n_seq
    q = torch.from_numpy(rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)).to(gpu)
    if paged:
        pool, bt, _ = U.make_paged(rng, lens, O.TYPE_F16)
        kw = dict(block_table=torch.from_numpy(bt).to(gpu), seq_lens=torch.tensor(lens, dtype=torch.int32, device=gpu))
    else:
        pool, kw = U.encode_kv(rng.standard_normal((1, width, 576)).astype(np.float32), O.TYPE_F16), {}
    k = torch.from_numpy(pool.view(np.int16)).to(gpu)
    mask = torch.from_numpy(_causal_mask(n_new, width - 3, width).view(np.float16)).to(gpu)
    out = torch.full((n_seq, n_new, n_head, 512), float("nan"), dtype=torch.float32, device=gpu)
    a, _, keep = J.capi.make_args(q, k, J.MLA_TYPE_F16, dv=512, scale=U.SCALE, mask=mask, out=out, **kw)
    assert lib.mla_attn_workspace_size(C.byref(a)) > J.capi.MLA_ATTN_STATIC_WORKSPACE_MAX
    a.workspace, a.workspace_size = None, 0
    assert lib.mla_attn_launch_static(C.byref(a), C.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)) == 0
    want = J.ggml_flash_attn_ext(q, k, J.MLA_TYPE_F16, dv=512, scale=U.SCALE, mask=mask, flags=J.MLA_FLAG_UNIFORM_SPLITS, **kw)
    torch.cuda.synchronize()
    print(U.check(out.cpu().numpy(), want.cpu().numpy()[..., :512], "fixed scratch"))


@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("n_seq", [1, 2])
def test_narrow_mask_rows_over_a_contiguous_cache_keep_both_halves_too(gpu, n_seq, big):
    """The same bound for a cache without a block table (640 cells, mask rows of 544), with cells inside and beyond f16's range."""
    rng = np.random.default_rng(n_seq)
    n_head, n_new, n_kv, width = 16, 9, 640, 544
    k = U.encode_kv(rng.standard_normal((n_seq, n_kv, 576)).astype(np.float32), O.TYPE_BF16)
    q = rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)
    if big:
        k[..., 500:512] = (k[..., 500:512] & 0x807f) | 0x4980
        q[..., 500:512] = 0
    mask = _causal_mask(n_new, width - 7, width)
    got = _run(gpu, q, k, O.TYPE_BF16, mask=mask, scale=U.SCALE)[..., :512]
    want = _want(q, [s[:width] for s in k], O.TYPE_BF16, mask)
    print(U.check(got, want, "narrow mask rows, contiguous", max_abs=2.0 ** 21 if big else 2e-4, rel_l2=3e-5))


@pytest.mark.parametrize("n_seq,n_new,n_head,dv,n_pages", [(256, 1, 128, 576, 66), (278, 1, 24, 512, 128)])
def test_narrow_mask_rows_over_many_pages_keep_f32_rows(gpu, n_seq, n_new, n_head, dv, n_pages):
    """More pages than a split of the pipelined kernel can list: its splits would leave f16 partial rows (2^-12 of each, 1e-4 over a
    row) where the general kernel has whole rows or f32 partials.  One pool of pages that all the sequences share; bf16 cells and
    probabilities as hi + lo halves: 3e-5 as above."""
    rng = np.random.default_rng(n_head + dv)
    width = n_pages * 128 - 32
    lens = [int(x) for x in rng.integers(width - 200, width, n_seq)]
    k = U.encode_kv(rng.standard_normal((n_pages * 128, 576)).astype(np.float32), O.TYPE_BF16)
    bt = np.stack([rng.permutation(n_pages) for _ in range(n_seq)]).astype(np.int32)
    q = rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)
    mask = _causal_mask(n_new, width, width)
    got = _run(gpu, q, k, O.TYPE_BF16, dv=dv, mask=mask, bt=bt, lens=lens, scale=U.SCALE)[..., :dv]
    for b in (0, n_seq // 2, n_seq - 1):
        cells = np.concatenate([k[p * 128:(p + 1) * 128] for p in bt[b]])[:lens[b]]
        want = O.flash_attn_ext(q[b:b + 1], cells[None], O.TYPE_BF16, dv=dv, mask=np.ascontiguousarray(mask[:, :lens[b]]), scale=U.SCALE)
        print(U.check(got[b:b + 1], want, "sequence %d" % b, rel_l2=3e-5))


@pytest.mark.parametrize("k_type", [O.TYPE_BF16, O.TYPE_F16, O.TYPE_Q8_0])
@pytest.mark.parametrize("n_seq,n_head,n_new,paged", [(300, 16, 1, True), (288, 16, 4, False), (300, 64, 1, True), (300, 96, 1, False), (300, 97, 1, True), (260, 48, 3, True)])
def test_more_masked_sequences_than_workgroups(gpu, k_type, n_seq, n_head, n_new, paged):
    """More than 256 masked sequences of 16 to 144 rows: those beyond whole rounds of workgroups are split where the program of their
    rows has a build for it (Q8_0 cells, more than 96 rows), and have a workgroup each where it does not."""
    rng = np.random.default_rng(n_seq + n_head)
    n_kv = 768
    q8s = 1.0 / 32 if k_type == O.TYPE_Q8_0 else None
    q = rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)
    mask = _causal_mask(n_new, n_kv, n_kv)
    if paged:   # one pool of pages that all the sequences share
        k = U.encode_kv(rng.standard_normal((9 * 128, 576)).astype(np.float32), k_type, q8_scale=q8s)
        bt = np.stack([rng.permutation(9)[:n_kv // 128] for _ in range(n_seq)]).astype(np.int32)
        lens = [n_kv - b % 100 for b in range(n_seq)]
        cells = lambda b: np.concatenate([k[p * 128:(p + 1) * 128] for p in bt[b]])[:lens[b]]
        kw = dict(bt=bt, lens=lens)
    else:
        k = U.encode_kv(rng.standard_normal((n_seq, n_kv, 576)).astype(np.float32), k_type, q8_scale=q8s)
        cells, kw = (lambda b: k[b]), {}
    got = _run(gpu, q, k, k_type, mask=mask, scale=U.SCALE, **kw)[..., :512]
    for b in (0, 255, 256, n_seq - 1):
        print(b, U.check(got[b:b + 1], _want(q[b:b + 1], [cells(b)], k_type, mask), "sequence %d" % b))


@pytest.mark.parametrize("k_type,n_seq,n_new,n_head,n_pages,width", [
    (O.TYPE_Q8_0, 1, 381, 64, 75, 9504),      # 48 MB less 3 KB of partial rows on the general kernel: no room for mask extents
    (O.TYPE_F16, 157, 3, 16, 93, 93 * 128),   # three splits in f16 fit, the two that fill the chip in f32 do not
])
def test_static_scratch_takes_what_only_the_smallest_plan_fits(gpu, k_type, n_seq, n_new, n_head, n_pages, width):
    import ctypes as C
    import torch
    import jittorinfer_amd as J
    rng = np.random.default_rng(n_new)
    q = torch.from_numpy(rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)).to(gpu)
    pool = U.encode_kv(rng.standard_normal((n_pages * 128, 576)).astype(np.float32), k_type, q8_scale=1.0 / 32 if k_type == O.TYPE_Q8_0 else None)
    k = torch.from_numpy(pool.view(np.int16) if pool.dtype == np.uint16 else pool).to(gpu)
    bt = np.stack([rng.permutation(n_pages) for _ in range(n_seq)]).astype(np.int32)   # (one pool of pages that all the sequences share)
    kw = dict(block_table=torch.from_numpy(bt).to(gpu), seq_lens=torch.full((n_seq,), width - 3, dtype=torch.int32, device=gpu))
    mask = torch.from_numpy(_causal_mask(n_new, width - 3, width).view(np.float16)).to(gpu)
    out = torch.full((n_seq, n_new, n_head, 512), float("nan"), dtype=torch.float32, device=gpu)
    a, _, keep = J.capi.make_args(q, k, k_type, dv=512, scale=U.SCALE, mask=mask, out=out, **kw)
    assert a.workspace_size > J.capi.MLA_ATTN_STATIC_WORKSPACE_MAX
    a.workspace, a.workspace_size = None, 0
    assert J.library().mla_attn_launch_static(C.byref(a), C.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)) == 0
    want = J.ggml_flash_attn_ext(q, k, k_type, dv=512, scale=U.SCALE, mask=mask, **kw)
    torch.cuda.synchronize()
    print(U.check(out.cpu().numpy(), want.cpu().numpy()[..., :512], "fixed scratch"))


@pytest.mark.parametrize("k_type", [O.TYPE_BF16, O.TYPE_F16])
@pytest.mark.parametrize("n_seq,n_head,n_new,n_kv", [(96, 16, 33, 288), (96, 16, 33, 1056), (128, 48, 3, 288), (128, 48, 3, 1056)])   # 528 and 144 rows
@pytest.mark.parametrize("masked", [False, True])
def test_unsplit_row_blocks_of_which_the_last_is_not_full(gpu, k_type, n_seq, n_head, n_new, n_kv, masked):
    """A workgroup per row block; f16 cells stay on the row-split program without a mask, over more than 1024 cells and up to 512 rows.  (The
    sequences share one cache: their stride is 0.)"""
    import torch
    import jittorinfer_amd as J
    rng = np.random.default_rng(n_head * n_kv)
    q = rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)
    k = U.encode_kv(rng.standard_normal((1, n_kv, 576)).astype(np.float32), k_type)
    mask = _causal_mask(n_new, n_kv, n_kv) if masked else None
    kw = dict(mask=torch.from_numpy(mask.view(np.float16)).to(gpu)) if masked else {}
    assert J.plan(torch.from_numpy(q).to(gpu), torch.from_numpy(k.view(np.int16)).to(gpu), k_type, scale=U.SCALE, **kw)["n_splits"] == 1
    got = _run(gpu, q, k, k_type, mask=mask, scale=U.SCALE)[..., :512]
    for b in (0, n_seq - 1):
        print(b, U.check(got[b:b + 1], _want(q[b:b + 1], [k[0]], k_type, mask), "sequence %d" % b))


@pytest.mark.parametrize("n_seq,n_head,n_new", [(8, 16, 10), (31, 16, 10), (32, 16, 10)])   # 16, 62 and 64 row blocks
def test_one_page_of_f16_keys_behind_a_mask(gpu, n_seq, n_head, n_new):
    """Two row blocks per sequence, the second of 32 rows: the row-split program below 64 row blocks, the column-split one from there on."""
    rng = np.random.default_rng(n_seq)
    q = rng.standard_normal((n_seq, n_head, n_new, 576)).astype(np.float32)
    k = U.encode_kv(rng.standard_normal((n_seq, 128, 576)).astype(np.float32), O.TYPE_F16)
    mask = _causal_mask(n_new, 128, 128)
    print(U.check(_run(gpu, q, k, O.TYPE_F16, mask=mask, scale=U.SCALE)[..., :512], _want(q, list(k), O.TYPE_F16, mask), "one page"))


def test_static_scratch_takes_a_chunk_behind_a_mask_narrower_than_its_cache(gpu):
    """25600 rows over a contiguous cache: the f16 partial rows of two splits do not fit the fixed scratch, whole rows need none."""
    import ctypes as C
    import torch
    import jittorinfer_amd as J
    rng = np.random.default_rng(17)
    n_new, n_head, n_kv, width = 200, 128, 1024, 992
    q = torch.from_numpy(rng.standard_normal((1, n_head, n_new, 576)).astype(np.float32)).to(gpu)
    k = torch.from_numpy(U.encode_kv(rng.standard_normal((1, n_kv, 576)).astype(np.float32), O.TYPE_BF16).view(np.int16)).to(gpu)
    mask = torch.from_numpy(_causal_mask(n_new, width - 5, width).view(np.float16)).to(gpu)
    out = torch.full((1, n_new, n_head, 512), float("nan"), dtype=torch.float32, device=gpu)
    a, _, keep = J.capi.make_args(q, k, O.TYPE_BF16, dv=512, scale=U.SCALE, mask=mask, out=out)
    assert a.workspace_size > J.capi.MLA_ATTN_STATIC_WORKSPACE_MAX
    a.workspace, a.workspace_size = None, 0
    assert J.library().mla_attn_launch_static(C.byref(a), C.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)) == 0
    want = J.ggml_flash_attn_ext(q, k, O.TYPE_BF16, dv=512, scale=U.SCALE, mask=mask)
    torch.cuda.synchronize()
    print(U.check(out.cpu().numpy(), want.cpu().numpy()[..., :512], "fixed scratch"))
