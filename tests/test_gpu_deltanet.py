"""GPU parity of the Gated DeltaNet recurrent update with in-kernel rollback
snapshots (qwfn_graph.cpp:240-278, :208-238) against the oracle's gated delta
rule, at the model's shapes (16 key heads, 48 value heads of 128; q, k, v read
as the views of one [T, 10240] conv output, as the reference's
deltanet_conv_qkv takes them). Tolerance: the kernel's column sums run in 8
partial sums where the oracle sums in order, so outputs and states agree to
float rounding (2e-5 relative, 1e-6 absolute). Also: T tokens in one launch
equal T launches of one token, and snapshot s equals the final state of a
launch over T - s tokens."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, say
from oracle import oracle as O

pytestmark = pytest.mark.gpu
NK, NV, D, CONV = 16, 48, 128, 10240


def _inputs(seed, T):
    rng = np.random.default_rng(seed)
    conv = rng.standard_normal((T, CONV)).astype(np.float32)
    qk = conv[:, :2 * NK * D].reshape(T, 2, NK, D)
    qk /= np.linalg.norm(qk, axis=-1, keepdims=True)             # the l2 norm of deltanet_conv_qkv
    conv[:, :2 * NK * D] = qk.reshape(T, -1)
    g = -rng.uniform(0.0, 1.5, (T, NV)).astype(np.float32)
    beta = rng.uniform(0.0, 1.0, (T, NV)).astype(np.float32)
    s0 = (rng.standard_normal((NV, D, D)) * 0.05).astype(np.float32)
    return conv, g, beta, s0


def _views(conv):
    T = conv.shape[0]
    q = conv[:, :NK * D].reshape(T, NK, D)
    k = conv[:, NK * D:2 * NK * D].reshape(T, NK, D)
    v = conv[:, 2 * NK * D:].reshape(T, NV, D)
    return q, k, v


def _run(K, conv_d, g_d, beta_d, state_d, T, n_snap):
    out = torch.zeros((T, NV, D), dtype=torch.float32, device="cuda")
    snap = torch.zeros((max(n_snap, 1), NV, D, D), dtype=torch.float32, device="cuda")
    K.gated_delta_net(conv_d[:, :NK * D], conv_d[:, NK * D:2 * NK * D], conv_d[:, 2 * NK * D:], g_d, beta_d, state_d,
                      out, NK, snap if n_snap else None, n_snap)
    return out, snap


# the kernel loads the inputs of 4 tokens at a time: 5 and 9 tokens end in a
# partial group, and 8 snapshots of 9 tokens are taken inside earlier groups
@pytest.mark.parametrize("T,n_snap", [(1, 0), (3, 2), (4, 3), (5, 4), (9, 8), (16, 3)])
def test_gated_delta_net_matches_oracle(gpu, oracle, T, n_snap):
    K = gpu
    conv, g, beta, s0 = _inputs(T, T)
    conv_d, g_d, beta_d, state_d = dev(conv), dev(g), dev(beta), dev(s0)
    say(f"gated_delta_net T={T} n_snap={n_snap}")
    out, snap = _run(K, conv_d, g_d, beta_d, state_d, T, n_snap)
    q, k, v = _views(conv)
    r_out, r_st, r_snap = O.gated_delta_net(q, k, v, g, beta, s0, n_snap=n_snap)
    np.testing.assert_allclose(host(out), r_out, rtol=2e-5, atol=1e-6)
    np.testing.assert_allclose(host(state_d), r_st, rtol=2e-5, atol=1e-6)
    if n_snap:
        np.testing.assert_allclose(host(snap)[:n_snap], r_snap, rtol=2e-5, atol=1e-6)


def test_gated_delta_net_chaining_and_snapshots(gpu, oracle):
    K = gpu
    T = 4
    conv, g, beta, s0 = _inputs(99, T)
    conv_d, g_d, beta_d = dev(conv), dev(g), dev(beta)
    say("gated_delta_net: one launch of 4 tokens")
    st_all = dev(s0)
    out_all, snap = _run(K, conv_d, g_d, beta_d, st_all, T, T - 1)
    say("gated_delta_net: four launches of one token")
    st_one = dev(s0)
    outs = []
    states = []
    for t in range(T):
        o, _ = _run(K, conv_d[t:t + 1], g_d[t:t + 1], beta_d[t:t + 1], st_one, 1, 0)
        outs.append(host(o)[0])
        states.append(host(st_one).copy())
    np.testing.assert_array_equal(host(out_all), np.stack(outs))
    np.testing.assert_array_equal(host(st_all), states[-1])
    for s in range(1, T):
        np.testing.assert_array_equal(host(snap)[s - 1], states[T - 1 - s])


def _rule64(q, k, v, g, beta, s0):
    """The recurrence in float64: q, k [T, n_k, d]; v [T, n_v, d]; returns out, the states after each token."""
    T, nk, d = q.shape
    nv = v.shape[1]
    st, out, states = s0.astype(np.float64), np.zeros((T, nv, d)), []
    q, k = (np.repeat(x.astype(np.float64), nv // nk, axis=1) for x in (q, k))
    for t in range(T):
        st = st * np.exp(g[t].astype(np.float64))[:, None, None]
        dl = (v[t].astype(np.float64) - np.einsum("hrc,hr->hc", st, k[t])) * beta[t].astype(np.float64)[:, None]
        st = st + k[t][:, :, None] * dl[:, None, :]
        out[t] = np.einsum("hrc,hr->hc", st, q[t]) / np.sqrt(d)
        states.append(st)
    return out, states


def _small(seed, T, nk, nv):
    rng = np.random.default_rng(seed)
    qk = rng.standard_normal((2, T, nk, D))
    qk = (qk / np.linalg.norm(qk, axis=-1, keepdims=True)).astype(np.float32)
    v = rng.standard_normal((T, nv, D)).astype(np.float32)
    # a head of long memory, one of short
    g = (-rng.uniform(0.0, 1.0, (T, nv)) * np.geomspace(0.01, 1.5, nv)).astype(np.float32)
    beta = rng.uniform(0.0, 1.0, (T, nv)).astype(np.float32)
    s0 = (rng.standard_normal((nv, D, D)) * 0.05).astype(np.float32)
    return qk[0], qk[1], v, g, beta, s0


def _call(K, q, k, v, g, beta, s0, n_snap=0, pad=0):
    """pad: extra floats per token in the q, k and v rows (strided views)."""
    T, nk, _ = q.shape
    nv = v.shape[1]
    rows = [np.concatenate([x.reshape(T, -1), np.full((T, pad), np.nan, np.float32)], axis=1) for x in (q, k, v)]
    qd, kd, vd = (dev(x)[:, :x.shape[1] - pad] for x in rows)
    st = dev(s0)
    out = torch.full((T, nv, D), 7.0, dtype=torch.float32, device="cuda")
    snap = torch.zeros((max(n_snap, 1), nv, D, D), dtype=torch.float32, device="cuda")
    K.gated_delta_net(qd, kd, vd, dev(g), dev(beta), st, out, nk, snap if n_snap else None, n_snap)
    return host(out), host(st), host(snap)


# chunks of 16 tokens in groups of 64 from 12 tokens on: partial chunks and groups, one and several groups, grids that are and are
# not a multiple of the 8 XCDs (4 blocks a value head), a last chunk of one token, snapshots behind the chunks
@pytest.mark.parametrize("T,nk,nv,n_snap,pad", [(11, 1, 2, 0, 0), (12, 1, 3, 0, 4), (15, 2, 2, 0, 0), (16, 1, 2, 0, 8), (17, 1, 1, 0, 0),
                                                (63, 1, 3, 0, 4), (64, 2, 4, 0, 0), (65, 1, 2, 0, 0), (129, 1, 3, 0, 12),
                                                (200, 2, 6, 0, 0), (16, 1, 3, 3, 0), (70, 1, 2, 5, 4)])
def test_gated_delta_net_chunks(gpu, T, nk, nv, n_snap, pad):
    """Against float64: a token's sums have 128 terms and a state remembers at most T tokens, so the 2-norm error
    stays within 4 sqrt(128 + T) 2^-24 of the result (5e-6 at T 200; 5e-7 seen at T 512)."""
    q, k, v, g, beta, s0 = _small(T, T, nk, nv)
    say(f"gated_delta_net chunks T={T} heads {nk}/{nv} snapshots {n_snap}")
    out, st, snap = _call(gpu, q, k, v, g, beta, s0, n_snap, pad)
    r_out, states = _rule64(q, k, v, g, beta, s0)
    tol = 4 * np.sqrt(128 + T) * 2.0 ** -24
    for name, a, b in [("out", out, r_out), ("state", st, states[-1])] + \
            [(f"snap {s}", snap[s - 1], states[T - 1 - s]) for s in range(1, n_snap + 1)]:
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"  {name} {err:.2e}", flush=True)
        assert err <= tol, name


def test_gated_delta_net_chunks_not_finite(gpu):
    """A decay of 0 forgets the state exactly; a value that is not finite reaches its own column from its token
    on, a key every column of its heads, a query its own outputs, and nothing before them."""
    T, nk, nv = 80, 2, 4
    q, k, v, g, beta, s0 = _small(3, T, nk, nv)
    g[37, 1] = -np.inf
    say("gated_delta_net chunks with a decay of 0")
    out, st, _ = _call(gpu, q, k, v, g, beta, s0)
    r_out, states = _rule64(q, k, v, g, beta, s0)
    tol = 4 * np.sqrt(128 + T) * 2.0 ** -24
    assert np.linalg.norm(out - r_out) <= tol * np.linalg.norm(r_out)
    assert np.linalg.norm(st - states[-1]) <= tol * np.linalg.norm(states[-1])
    v2, k2, q2 = v.copy(), k.copy(), q.copy()
    v2[21, 0, 5] = np.inf                    # value head 0, column 5
    k2[42, 1, 9] = np.nan                    # key head 1: value heads 2 and 3
    q2[10, 0, 3] = np.inf                    # key head 0, token 10 only: value heads 0 and 1
    say("gated_delta_net chunks with values that are not finite")
    out2, st2, _ = _call(gpu, q2, k2, v2, g, beta, s0)
    bad = np.zeros(out.shape, bool)
    bad[21:, 0, 5] = True
    bad[42:, 2:] = True
    bad[10, :2] = True
    assert not np.isfinite(out2[bad]).any()
    np.testing.assert_array_equal(out2[~bad], out[~bad])
    badst = np.zeros(st.shape, bool)
    badst[0, :, 5] = True
    badst[2:] = True
    assert not np.isfinite(st2[badst]).any()
    np.testing.assert_array_equal(st2[~badst], st[~badst])


def test_gated_delta_net_chunks_overflow(gpu):
    """Finite inputs whose d overflows at token 23 of a column (a value near the largest float at token 20, the key
    of 23 opposite to 20's): that column is not finite from token 23 on, everything before it and every other column
    is what it is without the overflow."""
    T, nk, nv = 40, 1, 2
    q, k, v, g, beta, s0 = _small(5, T, nk, nv)
    g[:], beta[20:24] = 0.0, 1.0
    k[23] = -k[20]
    v[20, 1, 7] = 3.0e38
    r_out, _ = _rule64(q, k, v, g, beta, s0)
    v2 = v.copy()
    v2[23, 1, 7] = 3.0e38                    # d = 3e38 - (-1) 3e38
    say("gated_delta_net chunks with a d that overflows")
    out, st, _ = _call(gpu, q, k, v2, g, beta, s0)
    assert not np.isfinite(out[23:, 1, 7]).any() and not np.isfinite(st[1, :, 7]).any()
    for sl in (slice(0, 20), slice(20, 23)):     # each at the scale of its own values
        np.testing.assert_allclose(out[sl, 1, 7], r_out[sl, 1, 7], rtol=0, atol=1e-5 * np.abs(r_out[sl, 1, 7]).max())
    v2[:, 1, 7] = 0.0
    out0, st0, _ = _call(gpu, q, k, v2, g, beta, s0)
    other = np.ones(out.shape, bool)
    other[:, 1, 7] = False
    np.testing.assert_array_equal(out[other], out0[other])
    others = np.ones(st.shape, bool)
    others[1, :, 7] = False
    np.testing.assert_array_equal(st[others], st0[others])


@pytest.mark.parametrize("T", [16, 64, 150])
def test_gated_delta_net_correlated_keys(gpu, T):
    """Keys and queries around one direction (mean cosine 0.7), beta near 1, long memory: the chunked outputs are
    differences of larger products there. Both forms against float64 within the bound of the other chunk tests
    (2-norm, of it 3.5e-7 seen in chunks and 1.1e-7 token by token); calls of 8 tokens, which stay token by token,
    agree with the one call to the sum of the two errors and not to the bit."""
    nk, nv = 2, 4
    rng = np.random.default_rng(T)
    q, k, v, g, beta, s0 = _small(T, T, nk, nv)
    q, k = (x + 1.7 * c / np.sqrt(D) for x, c in zip((q, k), rng.standard_normal((1, nk, D))[None].repeat(2, 0)))
    q, k = ((x / np.linalg.norm(x, axis=-1, keepdims=True)).astype(np.float32) for x in (q, k))
    assert np.mean(np.einsum("tkd,skd->kts", k, k)) > 0.6
    g, beta = (g * 0.03).astype(np.float32), (0.9 + 0.1 * beta).astype(np.float32)
    r_out, states = _rule64(q, k, v, g, beta, s0)
    say(f"gated_delta_net correlated keys T={T}, in chunks")
    out, st, _ = _call(gpu, q, k, v, g, beta, s0)
    say("the same in calls of 8 tokens")
    s1, parts = s0, []
    for t in range(0, T, 8):
        o, s1, _ = _call(gpu, *(x[t:t + 8] for x in (q, k, v, g, beta)), s1)
        parts.append(o)
    out1 = np.concatenate(parts)
    tol = 4 * np.sqrt(128 + T) * 2.0 ** -24
    for name, a, b, ref in (("out", out, out1, r_out), ("state", st, s1, states[-1])):
        ea, eb, eab = (np.linalg.norm(x) / np.linalg.norm(ref) for x in (a - ref, b - ref, a - b))
        print(f"  {name}: chunks {ea:.2e}, tokens {eb:.2e}, between them {eab:.2e}", flush=True)
        assert ea <= tol and eb <= tol and eab <= ea + eb + 1e-7
