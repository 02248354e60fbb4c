"""Block selection of many queries (the tiled score kernel, from 9 queries on) against the
same queries in calls of at most 8 (the other score kernel, itself tested against the
oracle): the dot products, the sums over heads and the biased scores are the same bits, so
the selected blocks and cells are the same, in the same order."""
import numpy as np
import pytest
import torch

import qwfn_state as S
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_heads", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("T,nb", [(9, 33), (65, 130), (130, 1009), (257, 5003), (512, 16520)])
def test_many_queries_as_few(gpu, n_heads, T, nb):
    """One to eight heads (powers of two and between); queries past a workgroup's 32 to 256 and
    short of it; blocks that end within a tile of 16, one and several tiles a wave. The
    workspace behind the scores' padding is not written."""
    k, ratio = min(nb, 60), 4
    rng = np.random.default_rng(T + n_heads)
    pool = dev(rng.standard_normal((nb, 128)).astype(np.float16).view(np.uint16))
    q = dev(rng.standard_normal((T, n_heads, 128)).astype(np.float32))
    bias = dev(np.where(rng.random((T, nb)) < 0.2, -np.inf, rng.standard_normal((T, nb))).astype(np.float32))
    blk = dev(rng.permutation(nb * ratio).astype(np.int32).reshape(nb, ratio))
    n_ws = T * ((nb + 63) // 64 * 64)
    ws = torch.full((n_ws * 4 + 4096,), 0x5A, dtype=torch.uint8, device="cuda")

    def select(a, b, w=None):
        cells = torch.full((b - a, k * ratio), -1, dtype=torch.int32, device="cuda")
        top = torch.full((b - a, k), -1, dtype=torch.int32, device="cuda")
        S.qsa_select_cells(pool, q[a:b].contiguous(), bias[a:b].contiguous(), k, blk, ratio, cells, top, ws=w)
        return host(cells), host(top)

    say(f"selection of {T} queries x {n_heads} heads over {nb} blocks")
    cells, top = select(0, T, ws)
    assert (host(ws)[n_ws * 4:] == 0x5A).all()
    for a in sorted({0, 8 * (T // 16), max(0, T - 8)}):
        c, t = select(a, min(a + 8, T))
        np.testing.assert_array_equal(top[a:a + 8], t)
        np.testing.assert_array_equal(cells[a:a + 8], c)
