"""GPU accept, statistics, greedy verify and tree walk at the edges of their
kernels: vocabularies around a chunk (4096) and around 64 and 128 chunks,
masked logits, maxima and temperatures on both sides of the range in which
the chunk kernels take their reduced exponential, equal draft and target rows
(a residual of exactly zero), and trees around the sizes at which the
statistics' parent filter (1024 nodes) and the walk's LDS state (4096) end."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ih():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import inferno_hip
    assert inferno_hip.quant_kernels_available(), inferno_hip._lib.last_error()
    return inferno_hip


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("V", [1, 3, 4095, 4096, 4097, 4096 * 64 + 1, 4096 * 128 + 5])
@pytest.mark.parametrize("scale,shift,T", [(3.0, 0.0, 0.8), (3.0, 2.0 ** 20 - 40, 1.0), (3.0, 2.0 ** 20 + 40, 1.0),
                                           (2e5, 0.0, 0.7), (3e-19, 0.0, 2.0 ** -61)])
def test_statistics_and_draws(ih, V, scale, shift, T):
    """zmax is the exact maximum of the fp32 quotients and zsum within 2^-21
    of the fp64 sum (each entry's exponential errs by at most ~2^-22; the
    result is rounded to fp32); the accept equals the oracle's."""
    rng = np.random.default_rng(V % 9973)
    S, k = 6, 2
    L = (rng.standard_normal((S, k + 1, V)) * scale + shift * T).astype(np.float32)
    if V > 3:
        L[0, :, rng.integers(0, V, V // 2)] = -np.inf  # a masked vocabulary
        L[1, :, -1] = L[1].max(-1) + np.float32(scale)  # the last entry the largest
    zm, zs = (a.cpu().numpy() for a in ih.softmax_stats(_dev(L.reshape(-1, V)), T))
    z = (L.reshape(-1, V) / np.float32(T)).astype(np.float64)
    assert np.array_equal(zm, z.max(-1).astype(np.float32))
    ref = np.exp(z - z.max(-1, keepdims=True)).sum(-1)
    assert np.all(np.abs(zs / ref - 1) <= 2.0 ** -21)
    Ld = L[:, :k] + (rng.standard_normal((S, k, V)) * 0.5 * scale).astype(np.float32)
    draft = rng.integers(0, V, (S, k)).astype(np.int32)
    ua = rng.random((S, k)).astype(np.float32)
    ur, ub = rng.random(S).astype(np.float32), rng.random(S).astype(np.float32)
    ur[2] = 0.0
    for mode in (0, 1):
        tok, n = ih.spec_accept(_dev(L), _dev(Ld), _dev(draft), T, _dev(ua), _dev(ur), _dev(ub), mode=mode)
        tok, n = tok.cpu().numpy(), n.cpu().numpy()
        for s in range(S):
            rt, rn = O.spec_accept(L[s], Ld[s], draft[s], T, ua[s], float(ur[s]), float(ub[s]), mode)
            assert rn == n[s] and tok[s, :len(rt)].tolist() == rt.tolist(), (mode, s, n[s], rn, tok[s], rt)


@pytest.mark.parametrize("V", [4097, 300001])
def test_equal_rows_leave_no_residual(ih, V):
    """A rejected draft whose target and draft rows are equal: every p - q is
    exactly 0, so the draw is from p (standard mode)."""
    rng = np.random.default_rng(V)
    L = (rng.standard_normal((4, 3, V)) * 2).astype(np.float32)
    draft = rng.integers(0, V, (4, 2)).astype(np.int32)
    ua = np.full((4, 2), 1.0, np.float32)  # u < ratio fails at ratio 1
    ur, ub = rng.random(4).astype(np.float32), rng.random(4).astype(np.float32)
    tok, n = ih.spec_accept(_dev(L), _dev(L[:, :2].copy()), _dev(draft), 0.9, _dev(ua), _dev(ur), _dev(ub))
    for s in range(4):
        rt, rn = O.spec_accept(L[s], L[s, :2], draft[s], 0.9, ua[s], float(ur[s]), float(ub[s]), 0)
        assert rn == 0 == int(n[s]) and int(tok[s, 0]) == int(rt[0]), (s, tok[s], rt)


@pytest.mark.parametrize("V", [1, 4095, 4097, 4096 * 64 + 1])
def test_greedy_edges(ih, V):
    rng = np.random.default_rng(V)
    S, k = 5, 9
    L = rng.integers(0, 50, (S, k + 1, V)).astype(np.float32)  # (ties everywhere)
    draft = L[:, :k].argmax(-1).astype(np.int32)
    for s in range(1, S):
        draft[s, 2 * s] = (draft[s, 2 * s] + 1) % max(V, 2)
    n, a = (t.cpu().numpy() for t in ih.greedy_verify(_dev(L), _dev(draft)))
    for s in range(S):
        rn, ra = O.greedy_verify(L[s], draft[s])
        assert rn == n[s] and np.array_equal(ra, a[s]), s


@pytest.mark.parametrize("n", [1, 2, 1024, 1025, 4096, 4097])
@pytest.mark.parametrize("shape", ["chain", "wide", "random"])
def test_tree_sizes(ih, n, shape):
    rng = np.random.default_rng(n)
    V = 24
    par = np.array([0] + [i - 1 if shape == "chain" else 0 if shape == "wide" else int(rng.integers(max(0, i - 40), i))
                          for i in range(1, n)], np.int32)
    Lt = (rng.standard_normal((n, V))).astype(np.float32)
    Ld = Lt.copy() if shape == "chain" else (Lt + 0.3 * rng.standard_normal((n, V))).astype(np.float32)
    tok = rng.integers(0, V, n).astype(np.int32)
    u = (rng.random(n) * 0.9).astype(np.float32)
    if shape == "chain":
        u[n * 3 // 4:] = 1.0  # (ratio 1 everywhere: accepted up to there)
    path = ih.tree_accept(_dev(Lt), _dev(Ld), _dev(tok), _dev(par), 1.0, _dev(u)).cpu().numpy()
    assert np.array_equal(path, O.tree_accept(Lt, Ld, tok, par, 1.0, u))


@pytest.mark.parametrize("node,parent", [(1, -1), (1, 1), (63, 64), (63, 10 ** 6)])
def test_tree_malformed_parent(ih, node, parent):
    """A malformed parent anywhere, also of a leaf that no row belongs to, is reported."""
    par = np.array([0] + [(i - 1) // 4 for i in range(1, 64)], np.int32)
    par[node] = parent
    L = np.zeros((64, 32), np.float32)
    with pytest.raises(ValueError):
        ih.tree_accept(_dev(L), _dev(L), _dev(np.zeros(64, np.int32)), _dev(par), 1.0, _dev(np.zeros(64, np.float32)))


@pytest.mark.parametrize("mode,V,steps", [(0, 4 * 4096, 64), (0, 4 * 4096, 65), (0, 4 * 4096 - 7, 129),
                                          (1, 4 * 4096, 32), (1, 4 * 4096, 33), (0, 3, 257), (1, 5000, 300)])
@pytest.mark.parametrize("top_k", [0, 5])
def test_batch_equals_single_steps(ih, mode, V, steps, top_k):
    """More than 256 chunk-sum workgroups take the decision in a launch of its
    own: the tokens of a batch on either side are those of its steps one by
    one, also for an invalid draft id, k's edges and a pre-drawn bonus."""
    rng = np.random.default_rng(steps * 11 + V)
    k = 3
    t = (2.0 * rng.standard_normal((steps, k + 1, V))).astype(np.float32)
    d = (t[:, :k] + 0.7 * rng.standard_normal((steps, k, V))).astype(np.float32)
    x = d.argmax(-1).astype(np.int32)
    x[1, 1] = V  # invalid
    u = [_dev(rng.random(s).astype(np.float32)) for s in ((steps, k), steps, steps)]
    t, d, x = _dev(t), _dev(d), _dev(x)
    kw = dict(mode=mode, top_k=min(top_k, V))
    tok, n = (a.cpu().numpy() for a in ih.spec_accept(t, d, x, 0.9, *u, **kw))
    for s in range(steps):
        o = slice(s, s + 1)
        tok1, n1 = (a.cpu().numpy() for a in ih.spec_accept(t[o], d[o], x[o], 0.9, *(v[o] for v in u), **kw))
        assert n[s] == n1[0], (s, n[s], n1[0])
        m = n[s] + 1 + (mode == 1 and n[s] == k - 1)
        assert np.array_equal(tok[s, :m], tok1[0, :m]), (s, tok[s], tok1[0])
    assert n[1] == -1 or n[1] == 0
