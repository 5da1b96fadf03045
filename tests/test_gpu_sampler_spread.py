"""GPU: the spread sampler's thresholds at the edges of its kernels: rounds of
4096 logits, candidate lists of 336 entries a round and longer (rows whose
entries crowd one bucket overflow them, and a bucket of more than 4096 entries
is refined over the row, by parts of it first), the cut that leaves entries out
of the histograms (top-k up to 256) with the threshold near the row's maximum
and past the last bucket's start, ties at the threshold, masked and unaligned
rows. Top-k tokens equal the one-workgroup kernel's; top-p and
min-p draws equal the oracle's except where u lies within 1e-5 (the sum of
the fp32 probabilities' relative errors) of a step of its cumulative
distribution."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [5, 337, 4095, 4096, 4097, 8190, 70001]
KINDS = ["gauss", "lm", "flat", "few", "masked"]


@pytest.fixture(scope="module")
def ih():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import inferno_hip
    assert inferno_hip.quant_kernels_available(), inferno_hip._lib.last_error()
    return inferno_hip


def _rows(kind, rows, V):
    rng = np.random.default_rng(V * 7 + (KINDS + ["wide", "crowded"]).index(kind))
    if kind == "lm":  # a language model's: falling with the rank
        L = -1.6 * np.log(rng.permuted(np.tile(np.arange(1.0, V + 1), (rows, 1)), axis=1)) + 0.5 * rng.standard_normal((rows, V))
    elif kind == "flat":  # one bucket holds every entry, values distinct
        L = 0.01 * rng.standard_normal((rows, V))
    elif kind == "few":  # ties everywhere
        L = rng.integers(0, 6, (rows, V)) * 0.5
    elif kind in ("wide", "crowded"):  # a threshold past the lists, in every round or in the first
        L = 2.0 * rng.standard_normal((rows, V))
        if kind == "crowded":
            L = -np.sort(-L, axis=1)
    else:
        L = 3.0 * rng.standard_normal((rows, V))
        if kind == "masked":
            L[rng.random((rows, V)) < 0.7] = -np.inf
            L[:, V // 2] = 4.0
    return L.astype(np.float32)


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("V", SIZES)
@pytest.mark.parametrize("kind", KINDS)
def test_topk(ih, kind, V):
    rows = 5
    L = _rows(kind, rows, V)
    d = _dev(L)
    rng = np.random.default_rng(V)
    for k in (1, 2, 40, 64, 65, 256, 257, 1000, 4096):
        if k >= V:
            continue
        for kw in (dict(top_k=k), dict(top_k=k, top_p=0.9), dict(top_k=k, top_p=0.95, min_p=0.02)):
            u = _dev(rng.random(rows).astype(np.float32))
            a = ih.softmax_sample(d, u, temperature=0.8, **kw).cpu().numpy()
            b = ih.softmax_sample(d, u, temperature=0.8, spread=False, **kw).cpu().numpy()
            assert np.array_equal(a, b), (k, kw, a, b)


@pytest.mark.parametrize("V", [4200, 5000, 6000, 8292, 17384, 50257])
@pytest.mark.parametrize("k", [20, 40, 100, 200, 256])
def test_topk_outlier(ih, V, k):
    """One logit 45 above the rest (z = L / T), in the first, a middle or the
    short last round: the threshold lies in the last bucket, which every round
    with a cut shares, and rounds whose counted entries pass the list are read
    from the row. The uniforms are spread over the mass below the outlier too
    (an outlier in the last round has every other candidate before it)."""
    rows = 24
    rng = np.random.default_rng(V + k)
    for sd in (0.05, 0.2, 1.0):
        for T in (0.1, 0.3, 1.0):
            for at in (1, V // 2, V - 100):
                z = sd * rng.standard_normal(V)
                z[at] = z.max() + 45.0
                L = _dev(np.tile((T * z).astype(np.float32), (rows, 1)))
                e = np.exp(z - z[at])
                below = np.sort(e)[::-1][1:k].sum()  # the other candidates' mass
                u = np.append(below * rng.random(rows - 4), [1e-30, 1e-7, 0.5, 1 - 2.0 ** -24]).astype(np.float32)
                a = ih.softmax_sample(L, _dev(u), temperature=T, top_k=k).cpu().numpy()
                b = ih.softmax_sample(L, _dev(u), temperature=T, top_k=k, spread=False).cpu().numpy()
                assert np.array_equal(a, b), (sd, T, at, a, b)
                assert b[-2] == at


@pytest.mark.parametrize("V", [4097, 9000, 12289, 30000, 98305])
@pytest.mark.parametrize("at", ["first", "last", "spread"])
def test_topk_crowded(ih, V, at):
    """Candidates crowded into the first or the last rounds, or even: a round
    passes any list (its entries come from the row, beside rounds with none),
    the lists of rows of 3 rounds and more are the longer ones for the larger
    k, and the last round is short. Values distinct and in runs of equals."""
    rows = 6
    rng = np.random.default_rng(V)
    z = 2.0 * rng.standard_normal((rows, V))
    if at != "spread":
        z = np.sort(z, axis=1) if at == "last" else -np.sort(-z, axis=1)
    z[3:] = np.round(4 * z[3:]) / 4
    d = _dev(z.astype(np.float32))
    for k in (90, 300, 700, 1500, 3000, 4096):
        if k < V:
            u = _dev(rng.random(rows).astype(np.float32))
            a = ih.softmax_sample(d, u, top_k=k).cpu().numpy()
            b = ih.softmax_sample(d, u, top_k=k, spread=False).cpu().numpy()
            assert np.array_equal(a, b), (k, a, b)


@pytest.mark.parametrize("V", SIZES)
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("kw", [dict(top_p=0.5), dict(top_p=0.95), dict(top_p=0.99985), dict(top_p=0.99995),
                                dict(top_p=0.9, min_p=0.05), dict(min_p=0.05), dict(), dict(top_p=1e-6)],
                         ids=lambda kw: ",".join(f"{k}={v}" for k, v in kw.items()) or "plain")
def test_mass_draws(ih, kind, V, kw):
    _mass_draws(ih, kind, V, kw)


def _mass_draws(ih, kind, V, kw, rows=8):
    L = _rows(kind, rows, V)
    us = np.random.default_rng(V + 1).random(rows).astype(np.float32)
    us[0] = np.float32(1 - 2.0 ** -24)
    got = ih.softmax_sample(_dev(L), _dev(us), temperature=0.9, **kw).cpu().numpy()
    for r in range(rows):
        p = O.sample_dist(L[r], temperature=0.9, **kw).astype(np.float64)
        c = np.cumsum(p)
        g, want = int(got[r]), O.softmax_sample(L[r], float(us[r]), temperature=0.9, **kw)
        if g == want:
            continue
        edge = 1.0
        if kw.get("top_p", 1.0) < 1.0:
            q = np.sort(O.sample_dist(L[r], temperature=0.9).astype(np.float64))[::-1]
            edge = np.min(np.abs(np.cumsum(q) - kw["top_p"]))
        before = c[g - 1] if g else 0.0
        assert edge < 1e-5 or (before - 1e-5 <= us[r] <= c[g] + 1e-5), (r, g, want, us[r], before, c[g])


@pytest.mark.parametrize("V", [4095, 9000, 30000, 70001])
@pytest.mark.parametrize("kind", ["wide", "crowded"])
@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_p=0.9, min_p=0.02)],
                         ids=lambda kw: ",".join(f"{k}={v}" for k, v in kw.items()))
@pytest.mark.parametrize("rows", [8, 32, 40])  # 16, 8 and 1 workgroups a row
def test_mass_draws_past_lists(ih, kind, V, kw, rows):
    _mass_draws(ih, kind, V, kw, rows)


@pytest.mark.parametrize("V", [4096, 12300])
@pytest.mark.parametrize("width", [2.0, 30.0, 60.0])
def test_mass_histograms(ih, V, width):
    """The buckets a top-p threshold is found in, as chunk_hist_kernel leaves
    them in the workspace (rows of 4104 bytes a round: statistics, then a slot
    whose first 2048 bytes are uint64 buckets mass << 13 | count, the mass of
    bucket b in 2^-x, x = 31 + floor(46 (b - 1) / 256)): each holds its entries'
    exp(z - m) to the relative error of one fp32 exponential at |z - m| <= 32:
    2^-20 / 32 of the difference's rounding, 2^-19 of the product's with
    log2 e, times ln 2, log2 e's own and the hardware's last place: 3e-6."""
    import torch
    n = -(-V // 4096)
    z = (width * np.random.default_rng(V).random(V)).astype(np.float32)
    ws = torch.zeros(ih.sampler.sample_ws_bytes(1, V), dtype=torch.uint8, device="cuda")
    ih.softmax_sample(_dev(z[None]), _dev(np.array([0.5], np.float32)), top_p=0.9, ws=ws)
    slots = ws.cpu().numpy()[8 * n:8 * n + 4096 * n].reshape(n, 4096)
    for c in range(n):
        x = z[4096 * c:4096 * (c + 1)]
        q = np.floor(x * np.float32(8)).astype(int)
        b = np.minimum(q.max() - q, 255)
        h = slots[c, :2048].view(np.uint64)
        assert np.array_equal(h & np.uint64(8191), np.bincount(b, minlength=256))
        mass = (h >> np.uint64(13)).astype(float) * 2.0 ** -(31.0 + (46 * (np.arange(256) - 1) >> 8))
        want = np.bincount(b, weights=np.exp(x.astype(float) - float(x.max())), minlength=256)
        live = want[:255] > 0
        assert np.max(np.abs(mass[:255][live] / want[:255][live] - 1)) < 3e-6
