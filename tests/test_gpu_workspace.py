"""Prefill calls with the workspace of a longer block over more keys: the split
count is not monotone in either, so a call whose own plan needs more takes
fewer splits. Each against the call with its own workspace, within the float
rounding of another split count."""
import ctypes

import numpy as np
import pytest
import torch

import kvdata as KD
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


# blocks and key counts below the largest, those whose own plan needs more among them (24 heads: 256 queries at
# 640 keys 31.7 MB against 25.4 at 1024, and 250 at 700 29.7; 800 of 64 heads are one split)
@pytest.mark.parametrize("T_max,nh,n_max,shapes", [(256, 24, 1024, ((256, 640), (256, 1023), (256, 300), (200, 1024), (250, 700), (40, 1024))),
                                                   (128, 24, 2048, ((128, 1216), (128, 513), (100, 2048), (64, 2000), (37, 2048))),
                                                   (800, 64, 400, ((800, 300), (512, 400), (100, 333), (9, 400)))])
def test_workspace_of_the_largest_shape(gpu, T_max, nh, n_max, shapes):
    K = gpu
    kc, vc = (KD.make_cache(KD.kv_rows(T_max, 0, kind, n_max), n_max) for kind in (KD.K_KIND, KD.V_KIND))
    kd, vd = dev(kc), dev(vc)
    qd = dev(KD.q_rows(T_max, 0, T_max, nh)[0][None].astype(np.float32))
    views = lambda T, n: (K.q_view(qd[:, :T]), K.cache_attn_view(kd, n, 2), K.cache_attn_view(vd, n, 2))
    size = lambda T, n: K.fattn_workspace_size(*views(T, n), None)
    largest = size(T_max, n_max)
    assert any(size(T, n) - largest > 0 for T, n in shapes)
    ws = torch.empty(largest, dtype=torch.uint8, device="cuda")
    for T, n in shapes:
        say(f"workspace of {T_max} x {n_max} ({largest} bytes): {T} x {nh} heads at {n} keys, its own {size(T, n)}")
        out = [torch.full((1, T, nh, 256), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
        ws.fill_(0xA5)
        K.flash_attn_ext(*views(T, n), None, 1 / 16, K.out_view(out[0]), ws=ws)
        own = torch.empty(size(T, n), dtype=torch.uint8, device="cuda")
        K.flash_attn_ext(*views(T, n), None, 1 / 16, K.out_view(out[1]), ws=own)
        a, b = host(out[0]), host(out[1])
        assert np.abs(a - b).max() <= 2e-5       # as the noalloc form with fewer splits
    # below the smallest workspace there is no plan
    qv, kv, vv = views(T_max, n_max)
    r = ctypes.byref
    o = K.out_view(torch.empty((1, T_max, nh, 256), device="cuda"))
    assert K.load().qwfn_flash_attn_ext_q8_0(r(qv), r(kv), r(vv), None, 1 / 16, 0.0, 0.0, r(o), 1, ws.data_ptr(), 255, None) == K.ENOMEM
