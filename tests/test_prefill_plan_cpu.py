"""The planner of the prefill attention (key splits and chunk images), read off
the workspace it asks for; no GPU."""
import ctypes

import pytest

import qwfn_kv as K

FAKE = 0x7F0000000000
IMAGE = 51200        # bytes of a 64-key chunk's image, one KV head


def workspace(T, nh, n_kv, B=1, nh_kv=2):
    q = K.tensor(FAKE, K.TYPE_F32, (256, T, nh, B), (4, nh * 1024, 1024, T * nh * 1024))
    k = K.tensor(FAKE, K.TYPE_Q8_0, (256, n_kv, nh_kv, B), (34, nh_kv * 272, 272, n_kv * nh_kv * 272))
    r = ctypes.byref
    return K.load().qwfn_fattn_workspace_size(r(q), r(k), r(k), None)


def expected(T, nh, n_kv, B, splits, images, nh_kv=2):
    up = lambda x: (x + 255) // 256 * 256
    n = B * splits * T * nh                       # partial rows of all KV heads
    base = up(up(n * 1024) + n * 8) if splits > 1 else 256
    return base + (nh_kv * -(-n_kv // 64) * IMAGE if images else 0)


# Attention op in us, the choice and what it was measured against: images that save less than their launch takes
# (256 x 16 at 4096: 8 splits without 67.6, 7 with 73.8; 128 x 16 at 8192: 16 without 70.4, 15 with 74.5;
# 100 x 16 at 8192: 16 without 66.8, 15 with 73.1), and images where they pay (512 x 16 at 16384: 321, without
# 368; 512 x 24 at 4096: 5 splits 160, 3 202, without 237)
@pytest.mark.parametrize("T,nh,n_kv,splits,images", [(256, 16, 4096, 8, False), (128, 16, 8192, 16, False),
                                                     (100, 16, 8192, 16, False), (512, 16, 16384, 4, True),
                                                     (512, 24, 4096, 5, True)])
def test_prefill_plan(T, nh, n_kv, splits, images):
    assert workspace(T, nh, n_kv) == expected(T, nh, n_kv, 1, splits, images)


# A batch makes no images, so its chunks have one price (before and after, us: 128 x 16 at 4096, 2 sequences, 7
# splits 75.4, 8 67.4; 512 x 24 at 2048, 2, 2 splits 210, 4 190; 200 x 24 at 4096, 4, 3 splits 277, 5 265)
@pytest.mark.parametrize("T,nh,n_kv,B,splits", [(128, 16, 4096, 2, 8), (512, 24, 2048, 2, 4), (200, 24, 4096, 4, 5)])
def test_prefill_plan_batch(T, nh, n_kv, B, splits):
    assert workspace(T, nh, n_kv, B) == expected(T, nh, n_kv, B, splits, False)


# What the splits' partials cost (before and after, us): cheap while the L2s hold them (256 x 32 at 256 keys on 8 KV
# heads: one split 39.8, two 28.9; 256 x 16 at 256, 2 sequences: 40.4, 28.8; 256 x 24 at 513: 3 splits 38.6, 5 34.3),
# dear beyond 16 splits, where the other merge reads them (64 x 24 at 8192 on 4 KV heads: 19 splits 69.3, 16 67.1;
# 128 x 24 at 65536: 32 splits 541, 10 516)
@pytest.mark.parametrize("T,nh,n_kv,B,nh_kv,splits,images", [(256, 32, 256, 1, 8, 2, False), (256, 16, 256, 2, 2, 2, False),
                                                             (256, 24, 513, 1, 2, 5, False), (64, 24, 8192, 1, 4, 16, False),
                                                             (128, 24, 65536, 1, 2, 10, True)])
def test_prefill_plan_partials(T, nh, n_kv, B, nh_kv, splits, images):
    assert workspace(T, nh, n_kv, B, nh_kv) == expected(T, nh, n_kv, B, splits, images, nh_kv)
