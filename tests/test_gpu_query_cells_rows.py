"""Head groups around the 8 rows up to which the per-position cell-list kernel packs two
blocks into a tile, with 2, 4 and 8 waves a list (the positions choose them)."""
import pytest

import kvdata as KD
from gpu_util import dev, say
from test_gpu_cells import _oracle_per_position, _query_lists, check, query_cells_dev_attn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [5, 200, 500])
@pytest.mark.parametrize("nh", [2, 14, 16, 18])
def test_query_cells_dev_head_groups(gpu, oracle, nh, T):
    """Groups of 1, 7, 8 and 9 rows against the oracle, within the bound that the other
    query-cell tests use (float rounding of ~1000 weighted terms)."""
    K = gpu
    n_rows, n_cells = 2000, 100
    pos0 = n_rows - T - 3
    lists = _query_lists(60 + nh, n_rows, pos0, T, n_cells)
    kc = KD.make_cache(KD.kv_rows(60 + nh, 0, KD.K_KIND, n_rows, outliers=True), n_rows)
    vc = KD.make_cache(KD.kv_rows(60 + nh, 0, KD.V_KIND, n_rows, outliers=True), n_rows)
    q = KD.q_rows(60 + nh, 1, T, nh)[0]
    say(f"query cells (device counts) nh={nh} T={T}")
    got, flags = query_cells_dev_attn(K, q, dev(kc), dev(vc), n_rows, lists, pos0)
    assert flags == 0
    check(got, _oracle_per_position(q, kc, vc, lists, pos0))
