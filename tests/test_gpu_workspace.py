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


def test_images_in_the_workspace_of_the_largest_shape(gpu):
    """336 queries ask for more partials than 512 at the same depth; in the workspace of 512 they still get images,
    over fewer splits."""
    K = gpu
    nh, n = 16, 16384
    kc, vc = (KD.make_cache(KD.kv_rows(5, 0, kind, n), n) for kind in (KD.K_KIND, KD.V_KIND))
    kd, vd = dev(kc), dev(vc)
    qd = dev(KD.q_rows(5, 0, 512, nh)[0][None].astype(np.float32))
    kv, vv = K.cache_attn_view(kd, n, 2), K.cache_attn_view(vd, n, 2)
    size = lambda T: K.fattn_workspace_size(K.q_view(qd[:, :T]), kv, vv, None)
    assert size(336) > size(512)
    outs = []
    for nb in (size(512), size(336)):
        say(f"336 x {nh} heads at {n} keys in {nb} bytes")
        out = torch.full((1, 336, nh, 256), float("nan"), dtype=torch.float32, device="cuda")
        ws = torch.full((nb,), 0xA5, dtype=torch.uint8, device="cuda")
        K.flash_attn_ext(K.q_view(qd[:, :336]), kv, vv, None, 1 / 16, K.out_view(out), ws=ws)
        assert K.last_kernel() == "k_fa_pre<false, true>"
        outs.append(host(out))
    assert np.abs(outs[0] - outs[1]).max() <= 2e-5


def test_noalloc_with_images(gpu):
    """A prefill whose partials and images both fit the library's scratch: the plan and the bits of the call with a
    workspace of that size; one whose images do not fit with the plan's partials is planned within the scratch."""
    K = gpu
    L, r = K.load(), ctypes.byref
    for T, nh, n, splits in ((60, 32, 2000, 0), (100, 16, 1300, 2), (128, 16, 8192, 0)):
        kc, vc = (KD.make_cache(KD.kv_rows(T, 0, kind, n), n) for kind in (KD.K_KIND, KD.V_KIND))
        kd, vd, qd = dev(kc), dev(vc), dev(KD.q_rows(T, 0, T, nh)[0][None].astype(np.float32))
        qv, kv, vv = K.q_view(qd), K.cache_attn_view(kd, n, 2), K.cache_attn_view(vd, n, 2)
        L.qwfn_fattn_force_splits(splits)
        try:
            say(f"noalloc {T} x {nh} heads at {n} keys, splits {splits or 'planned'}")
            need = K.fattn_workspace_size(qv, kv, vv, None)
            ws = torch.empty(need, dtype=torch.uint8, device="cuda")
            a, b = (torch.full((1, T, nh, 256), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2))
            K.check(L.qwfn_flash_attn_ext_q8_0(r(qv), r(kv), r(vv), None, 1 / 16, 0.0, 0.0, r(K.out_view(a)), 1, ws.data_ptr(),
                                               need, None))
            name = K.last_kernel()
            K.check(L.qwfn_flash_attn_ext_q8_0_noalloc(r(qv), r(kv), r(vv), None, 1 / 16, 0.0, 0.0, r(K.out_view(b)), 1, None))
        finally:
            L.qwfn_fattn_force_splits(0)
        if splits:
            assert name == K.last_kernel() == "k_fa_pre<false, true>" and need <= 16 << 20
        if need <= 16 << 20:
            np.testing.assert_array_equal(host(a), host(b))
        else:
            assert np.abs(host(a) - host(b)).max() <= 2e-5
