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
