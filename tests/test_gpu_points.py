"""Explicit query points with q in {2, 3, 4}: the exact integer form against sums in 80-bit floats, and
against the w-table form where a coefficient is not finite."""
import numpy as np
import pytest
import torch

from qsft_amd import _lib as L
from qsft_amd import device as dv
from qsft_amd import kernels as K

pytestmark = pytest.mark.gpu


def _reference(q, pts, locq, a):
    """cos and sin sums of every query in 80-bit floats: x = c + i z, and the sizes of its parts."""
    E = (pts.astype(np.int64) @ locq.astype(np.int64)) % q
    half = np.sqrt(np.longdouble(3)) / 2
    cos = {2: [1, -1], 3: [1, -.5, -.5], 4: [1, 0, -1, 0]}[q]
    sin = {2: [0, 0], 3: [0, half, -half], 4: [0, 1, 0, -1]}[q]
    cos, sin = np.array(cos, dtype=np.longdouble)[E], np.array(sin, dtype=np.longdouble)[E]
    re, im = a.real.astype(np.longdouble), a.imag.astype(np.longdouble)
    cr, ci, sr, si = cos @ re, cos @ im, sin @ re, sin @ im
    return cr - si, ci + sr, np.abs(cr) + np.abs(si), np.abs(ci) + np.abs(sr)


CASES = [(4, 50, 1, 1), (4, 50, 64, 64), (2, 20, 65, 63), (3, 64, 63, 65), (3, 65, 257, 130), (4, 129, 255, 129),
         (2, 200, 1000, 191), (4, 256, 320, 257), (3, 256, 16, 40), (4, 8, 4000, 1001), (2, 3, 0, 70)]


@pytest.mark.parametrize("q,n,S,N", CASES)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("spread", [1, 12])
def test_points_integer_sums(q, n, S, N, precision, spread):
    """One rounding of the result (a few of the parts at q = 3), 2^-63 of the largest component per term."""
    print(f"points q={q} n={n} S={S} N={N} {precision} spread={spread}", flush=True)
    rng = np.random.default_rng(q * 1000 + S + N)
    locq = rng.integers(0, q, size=(n, S))
    a = rng.normal(size=S) * 10.0 ** rng.uniform(-spread, spread, S) + 1j * rng.normal(size=S)
    pts = rng.integers(0, q, size=(N, n))
    dev, n_pad = dv.current_device(), dv.n_pad_of(n)
    at = dv.strengths_tensor(a, precision, dev)
    a = at.cpu().numpy().astype(np.complex128)
    x = dv.evaluate_points(q, n, dv.digits_tensor(pts, n_pad, dev), dv.digits_tensor(locq.T, n_pad, dev), at,
                           precision).cpu().numpy().astype(np.complex128)
    re, im, pr, pi = _reference(q, pts, locq, a)
    top = max(np.abs(a.real).max(initial=0), np.abs(a.imag).max(initial=0))
    per_term = 2 * S * 2.0 ** -63 * top                          # fixed point, and the reference's own sums
    eps = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    for got, ref, parts in ((x.real, re, pr), (x.imag, im, pi)):
        bound = 2 * eps * np.abs(ref) + 4 * 2.0 ** -53 * parts * (q == 3) + per_term
        assert (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("q", [2, 3, 4])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_points_not_finite(q, bad):
    """A coefficient that is not finite comes out as the table form gives it, bit for bit."""
    rng = np.random.default_rng(q)
    n, S, N = 70, 150, 130
    dev, n_pad = dv.current_device(), dv.n_pad_of(n)
    a = rng.normal(size=S) + 1j * rng.normal(size=S)
    a[77] = complex(1.0, bad)
    m = dv.digits_tensor(rng.integers(0, q, size=(N, n)), n_pad, dev)
    k = dv.digits_tensor(rng.integers(0, q, size=(S, n)), n_pad, dev)
    at = dv.strengths_tensor(a, "fp64", dev)
    got = dv.evaluate_points(q, n, m, k, at, "fp64")
    ref = torch.empty_like(got)
    K.EvalPoints([dict(q=q, n=n, S=S, m=m, K=k, a=at, x=ref)], L.QSFT_F64, table=True).launch()
    np.testing.assert_array_equal(got.cpu().numpy(), ref.cpu().numpy())


def test_points_mixed_launch():
    """Instances of both forms, several digit widths and sizes in one call."""
    rng = np.random.default_rng(5)
    dev, items, refs = dv.current_device(), [], []
    for q, n, S, N in [(4, 50, 100, 200), (20, 30, 40, 77), (3, 50, 7, 129), (2, 130, 300, 65), (7, 50, 10, 64)]:
        n_pad = dv.n_pad_of(n)
        pts, locq = rng.integers(0, q, size=(N, n)), rng.integers(0, q, size=(n, S))
        a = rng.normal(size=S) + 1j * rng.normal(size=S)
        items.append(dict(q=q, n=n, S=S, m=dv.digits_tensor(pts, n_pad, dev), K=dv.digits_tensor(locq.T, n_pad, dev),
                          a=dv.strengths_tensor(a, "fp64", dev),
                          x=torch.empty(N, dtype=torch.complex128, device=dev)))
        refs.append(np.exp(2j * np.pi * ((pts @ locq) % q) / q) @ a)
    K.eval_points(items, L.QSFT_F64)
    for it, ref in zip(items, refs):
        assert np.abs(it["x"].cpu().numpy() - ref).max() <= 1e-13 * np.abs(ref).max() * 10
