"""The merge of a prefill's key splits (k_fa_pre, 2 to 16 of them) at each of its sizes
and beside them, where rows see no key of some splits or no key at all, gated and not,
with an output that is 16-byte aligned and one that is not."""
import numpy as np
import pytest
import torch

import kvdata as KD
from gpu_util import dev, host, say
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,n_kv", [(2, 1100), (3, 1100), (4, 1100), (5, 1100), (8, 1000), (9, 1100), (16, 1000)])
def test_merge_of_prefill_splits(gpu, oracle, ns, n_kv):
    """Position t of 150 sees keys 0 .. 7 t (none: position 149, masked whole), so the splits
    after 7 t hold nothing for it. Against the oracle within 1e-4 (as test_gpu_prefill.py)."""
    K = gpu
    T, nh, nh_kv = 150, 16, 2
    kc, vc = (KD.make_cache(KD.kv_rows(ns, 0, kind, n_kv, outliers=True), n_kv) for kind in (KD.K_KIND, KD.V_KIND))
    q = KD.q_rows(ns, 0, T, nh)[0]
    mask = np.full((T, n_kv), O.F16_NEG_INF, dtype=np.uint16)
    for t in range(T - 1):
        mask[t, :7 * t + 1] = 0
    qd, md = dev(q[None].astype(np.float32)), dev(mask.view(np.float16))
    kd, vd = dev(kc), dev(vc)
    qv, kv, vv, mv = K.q_view(qd), K.cache_attn_view(kd, n_kv, nh_kv), K.cache_attn_view(vd, n_kv, nh_kv), K.mask_view(md)
    gate = dev(KD.normal(ns, 9, KD.Q_KIND, T * nh * 256).reshape(1, T, nh, 256))
    outs = []
    K.load().qwfn_fattn_force_splits(ns)
    try:
        ws = torch.full((K.fattn_workspace_size(qv, kv, vv, mv),), 0xA5, dtype=torch.uint8, device="cuda")
        for off, g in ((0, None), (1, None), (0, gate)):
            say(f"prefill merge, {ns} splits, output offset {off}, gate {g is not None}")
            buf = torch.full((T * nh * 256 + 4,), float("nan"), dtype=torch.float32, device="cuda")
            ov = K.out_view(buf[off:off + T * nh * 256].view(1, T, nh, 256))
            if g is None:
                K.flash_attn_ext(qv, kv, vv, mv, 1 / 16, ov, ws=ws)
            else:
                K.flash_attn_ext_gated(qv, kv, vv, mv, 1 / 16, ov, g, ws=ws)
            assert K.last_kernel().startswith("k_fa_pre<true")
            outs.append(host(buf)[off:off + T * nh * 256].reshape(T, nh, 256))
    finally:
        K.load().qwfn_fattn_force_splits(0)
    a, b, g = outs
    np.testing.assert_array_equal(a, b)
    np.testing.assert_allclose(g, a / (1 + np.exp(-host(gate)[0].astype(np.float64))), rtol=3e-6, atol=1e-7)
    assert not a[T - 1].any()
    for t in (0, 1, 9, 10, 75, 148):
        ref = KD.oracle_attn(q[t:t + 1], kc, vc, min(n_kv, 7 * t + 1), nh_kv, None, 1 / 16)[0]
        mx, mean = KD.err_stats(a[t], ref)
        print(f"  position {t}: max abs {mx:.3e} mean abs {mean:.3e}", flush=True)
        assert mx <= 1e-4
