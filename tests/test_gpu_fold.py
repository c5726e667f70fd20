"""Coset evaluation through the folded spectrum (qsft_fold_*) on the GPU,
every sample against the direct sum a_s w^{<M_c l + d_p, k_s>} in FP64.

Tolerances (max-abs over max |value|): the terms and bin sums are FP64, the
inverse transform has at most b q-point stages, so FP64 is within 1e-12 and
FP32, with b log2(q) <= 16 rounded additions of partial sums no larger than
sum |a_s|, within 2e-6 of the largest sample.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from qsft_amd import device as dv

# whole-row kernels (q = 4, b in {4, 6}) with rows that do not fill the last
# workgroup; one tile, several tiles and several passes of the others (b = 7,
# q = 2 b = 13, q = 20 b = 4), the generic radix (q = 7, 50, 64), one to four
# digit blocks; supports around the 16-, 64- and 2048-wide blocks of the prep
CASES = [(4, 10, 4, 100, 3, 11), (4, 50, 6, 1000, 2, 21), (4, 64, 6, 65, 1, 17), (4, 100, 7, 2049, 2, 33),
         (4, 9, 5, 64, 3, 10), (4, 20, 2, 16, 2, 5), (2, 8, 1, 1, 1, 9), (2, 30, 13, 63, 2, 16), (3, 67, 7, 777, 2, 19),
         (20, 16, 3, 2000, 2, 7), (20, 12, 4, 300, 1, 2), (5, 130, 4, 129, 2, 15), (7, 200, 3, 500, 2, 4),
         (50, 11, 2, 33, 1, 3), (64, 256, 2, 17, 2, 3), (4, 12, 3, 5000, 1, 12), (2, 40, 6, 0, 2, 3)]


def _inputs(q, n, b, S, C, P, seed, loc=None):
    g = np.random.default_rng(seed)
    Ms = [g.integers(0, q, size=(n, b)) for _ in range(C)]
    Ds = [g.integers(0, q, size=(P, n)) for _ in range(C)]
    loc = g.integers(0, q, size=(n, S)) if loc is None else loc
    a = g.uniform(1, 10, S) * np.exp(2j * np.pi * g.uniform(size=S))
    return Ms, Ds, loc, a


def _direct(q, b, Ms, Ds, loc, a):
    w = np.exp(2j * np.pi * np.arange(q) / q)
    lq = (np.arange(q ** b)[:, None] // q ** np.arange(b - 1, -1, -1)) % q
    out = []
    for M, D in zip(Ms, Ds):
        A = w[(lq @ ((M.T @ loc) % q)) % q]                        # (Q, S)
        out.append((A @ (a[:, None] * w[((D @ loc) % q).T])).T)
    return np.stack(out)


def _run(q, n, b, Ms, Ds, loc, a, precision):
    dev, n_pad = dv.current_device(), dv.n_pad_of(n)
    x = dv.evaluate_cosets(q, n, b, dv.Mt_tensor(Ms, b, n_pad, dev), dv.D_tensor(Ds, n_pad, dev),
                           dv.digits_tensor(loc.T, n_pad, dev), dv.strengths_tensor(a, precision, dev), precision)
    return x.cpu().numpy()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("q,n,b,S,C,P", CASES)
def test_fold_matches_direct_sum(q, n, b, S, C, P, precision, tol):
    print(f"fold q={q} n={n} b={b} S={S} C={C} P={P} {precision}", flush=True)
    Ms, Ds, loc, a = _inputs(q, n, b, S, C, P, seed=q * 97 + n + S)
    x = _run(q, n, b, Ms, Ds, loc, a, precision)
    ref = _direct(q, b, Ms, Ds, loc, a)
    assert x.shape == ref.shape
    assert np.max(np.abs(x - ref)) <= tol * max(np.max(np.abs(ref)), 1e-300)
    assert np.array_equal(x, _run(q, n, b, Ms, Ds, loc, a, precision))     # the same bits on every run


@pytest.mark.parametrize("q,b,S", [(4, 6, 1500), (4, 4, 300), (3, 5, 700), (2, 13, 400)])
def test_fold_of_crowded_bins(q, b, S):
    """Runs that span 64-term blocks and the waves' shares: every support in
    one bin, or in the bins of two values of the last digit."""
    print(f"fold crowded q={q} b={b} S={S}", flush=True)
    n, C, P = b + 6, 2, 3
    g = np.random.default_rng(S)
    loc = g.integers(0, q, size=(n, S))
    loc[:b] = 0                                                    # M picks the first b digits
    Ms, Ds, _, a = _inputs(q, n, b, S, C, P, 5, loc)
    for c in range(C):
        Ms[c][:] = 0
        Ms[c][:b] = np.eye(b, dtype=int)
    for crowd in (loc, np.where((np.arange(n) == b - 1)[:, None], np.arange(S)[None, :] % 2, loc)):
        x = _run(q, n, b, Ms, Ds, crowd, a, "fp64")
        ref = _direct(q, b, Ms, Ds, crowd, a)
        assert np.max(np.abs(x - ref)) <= 1e-12 * np.max(np.abs(ref))
