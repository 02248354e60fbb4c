"""k_fa_pre over chunk images (the K/V rows of a prefill converted once, by a
launch of its own, into the call's workspace) against the same kernel
converting each chunk itself, which a workspace that holds the split partials
only selects: the arithmetic is the same, so the results are the same bits.
Against the oracle within 1e-4 (as test_gpu_prefill.py), on a few positions."""
import ctypes

import numpy as np
import pytest
import torch

import kvdata as KD
from gpu_util import dev, host, say
from oracle import oracle as O

pytestmark = pytest.mark.gpu
IMAGE = 51200        # bytes of a 64-key chunk's image, one KV head


def _partials(nh_kv, ns, R):
    """Workspace bytes of the split partials: O rows and (max, sum) pairs, 256-byte sections."""
    if ns == 1:
        return 256
    up = lambda x: (x + 255) // 256 * 256
    n = nh_kv * ns * R
    return up(up(n * 1024) + n * 8)


def _run(K, qv, kv, vv, mv, T, nh, ws_bytes, gate=None):
    out = torch.full((1, T, nh, 256), float("nan"), dtype=torch.float32, device="cuda")
    ws = torch.full((ws_bytes,), 0xA5, dtype=torch.uint8, device="cuda")
    if gate is not None:
        K.flash_attn_ext_gated(qv, kv, vv, mv, 1 / 16, K.out_view(out), gate, ws=ws)
    else:
        K.flash_attn_ext(qv, kv, vv, mv, 1 / 16, K.out_view(out), ws=ws)
    return host(out)[0], K.last_kernel()


# whole and partial last chunks (one key, 63, none missing), 8 / 12 / 4 heads a KV head, 1 and 2 splits (9 chunks a
# split at least), masked and not, K and V as halves of one buffer's rows
@pytest.mark.parametrize("T,nh,n_kv,splits,masked,paired", [(100, 16, 577, 1, True, False), (100, 16, 640, 1, False, False),
                                                            (90, 24, 639, 1, True, True), (52, 32, 1217, 2, True, False),
                                                            (200, 8, 1153, 2, True, False), (85, 16, 1280, 2, False, True)])
def test_images_same_bits(gpu, oracle, T, nh, n_kv, splits, masked, paired):
    K = gpu
    nh_kv = 2
    kc, vc = (KD.make_cache(KD.kv_rows(T, 0, kind, n_kv, outliers=True), n_kv) for kind in (KD.K_KIND, KD.V_KIND))
    q = KD.q_rows(T, 0, T, nh)[0]
    qd = dev(q[None].astype(np.float32))
    if paired:
        both = dev(np.concatenate([kc, vc], axis=1))
        kv, vv = (K.tensor(both.data_ptr() + off, K.TYPE_Q8_0, (256, n_kv, nh_kv, 1), (34, 1088, 272, n_kv * 1088))
                  for off in (0, 544))
    else:
        kd, vd = dev(kc), dev(vc)
        kv, vv = K.cache_attn_view(kd, n_kv, nh_kv), K.cache_attn_view(vd, n_kv, nh_kv)
    mask = O.causal_mask(T, n_kv - T) if masked else None
    md = dev(mask.view(np.float16)) if masked else None
    mv = K.mask_view(md) if masked else None
    qv = K.q_view(qd)
    gate = dev(KD.normal(T, 9, KD.Q_KIND, T * nh * 256).reshape(1, T, nh, 256))
    K.load().qwfn_fattn_force_splits(splits)
    try:
        need = K.fattn_workspace_size(qv, kv, vv, mv)
        base = _partials(nh_kv, splits, T * nh // nh_kv)
        assert need == base + nh_kv * -(-n_kv // 64) * IMAGE
        say(f"images T={T} heads {nh} n_kv={n_kv} splits={splits} masked={masked}")
        a, name = _run(K, qv, kv, vv, mv, T, nh, need)
        assert name == f"k_fa_pre<{'true' if masked else 'false'}, true>"
        say("the partials' workspace: no images")
        b, name = _run(K, qv, kv, vv, mv, T, nh, need - 1)
        assert name == f"k_fa_pre<{'true' if masked else 'false'}>"
        c, name = _run(K, qv, kv, vv, mv, T, nh, base)
        assert name == f"k_fa_pre<{'true' if masked else 'false'}>"
        g, _ = _run(K, qv, kv, vv, mv, T, nh, need, gate)
        if base > 256:
            r = ctypes.byref
            ws = torch.empty(base, dtype=torch.uint8, device="cuda")
            assert K.load().qwfn_flash_attn_ext_q8_0(r(qv), r(kv), r(vv), r(mv) if masked else None, 1 / 16, 0.0, 0.0,
                                                     r(K.out_view(torch.empty((1, T, nh, 256), device="cuda"))), 1,
                                                     ws.data_ptr(), base - 256, None) == K.ENOMEM
    finally:
        K.load().qwfn_fattn_force_splits(0)
    np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(a, c)
    np.testing.assert_allclose(g, a / (1 + np.exp(-host(gate)[0].astype(np.float64))), rtol=3e-6, atol=1e-7)
    toks = [0, T // 2, T - 1]
    for t in toks:
        vis = n_kv - T + t + 1 if masked else n_kv
        ref = KD.oracle_attn(q[t:t + 1], kc, vc, vis, nh_kv, None, 1 / 16)[0]
        mx, mean = KD.err_stats(a[t], ref)
        print(f"  position {t}: max abs {mx:.3e} mean abs {mean:.3e}", flush=True)
        assert mx <= 1e-4


def test_images_capture(gpu, oracle):
    """The call with images in a HIP graph, replayed: each replay the eager result."""
    K = gpu
    T, nh, n_kv = 100, 16, 700
    kc, vc = (KD.make_cache(KD.kv_rows(7, 0, kind, n_kv), n_kv) for kind in (KD.K_KIND, KD.V_KIND))
    qd, kd, vd = dev(KD.q_rows(7, 0, T, nh)[0][None].astype(np.float32)), dev(kc), dev(vc)
    qv, kv, vv = K.q_view(qd), K.cache_attn_view(kd, n_kv, 2), K.cache_attn_view(vd, n_kv, 2)
    md = dev(O.causal_mask(T, n_kv - T).view(np.float16))
    mv = K.mask_view(md)
    out = torch.zeros((1, T, nh, 256), dtype=torch.float32, device="cuda")
    K.load().qwfn_fattn_force_splits(1)
    try:
        ws = torch.empty(K.fattn_workspace_size(qv, kv, vv, mv), dtype=torch.uint8, device="cuda")
        say("images under capture")
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            K.flash_attn_ext(qv, kv, vv, mv, 1 / 16, K.out_view(out), ws=ws)
            st.synchronize()
            eager = host(out).copy()
            assert K.last_kernel() == "k_fa_pre<true, true>"
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=st):
                K.flash_attn_ext(qv, kv, vv, mv, 1 / 16, K.out_view(out), ws=ws)
        for _ in range(3):
            out.zero_()
            ws.zero_()
            g.replay()
            np.testing.assert_array_equal(host(out), eager)
            K.flash_attn_ext(qv, kv, vv, mv, 1 / 16, K.out_view(out), ws=ws)
            np.testing.assert_array_equal(host(out), eager)
    finally:
        K.load().qwfn_fattn_force_splits(0)
