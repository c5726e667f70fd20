"""Explicit query points with q in {2, 3, 4}: the exact integer form against sums in 80-bit floats, and
against the w-table form where a coefficient is not finite."""
from decimal import Decimal, localcontext
from fractions import Fraction

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


def _exact(q, pts, locq, a):
    """(re, im, sizes of the parts that meet) of every query in rational numbers, sqrt(3) to 100 digits."""
    with localcontext() as ctx:
        ctx.prec = 100
        half = Fraction(Decimal(3).sqrt()) / 2
    cos = {2: [1, -1], 3: [2, -1, -1], 4: [1, 0, -1, 0]}[q]
    sin = {2: [0, 0], 3: [0, 1, -1], 4: [0, 1, 0, -1]}[q]
    unit = Fraction(1, 2 ** 1074)                                 # of which every component is a whole number
    ct, st = (Fraction(1, 2), half) if q == 3 else (1, 1)
    E = (pts.astype(np.int64) @ locq.astype(np.int64)) % q
    re, im = ([int(Fraction(float(v)) / unit) for v in part] for part in (a.real, a.imag))
    out = []
    for row in E.tolist():
        cr, ci = (ct * unit * sum(cos[e] * v for e, v in zip(row, part)) for part in (re, im))
        sr, si = (st * unit * sum(sin[e] * v for e, v in zip(row, part)) for part in (re, im))
        out.append((cr - si, ci + sr, abs(cr) + abs(si), abs(ci) + abs(sr)))
    return out


def _strengths(kind, S, precision, rng):
    """Components of one size, one part far below the other, or spread over many decades."""
    re, im = rng.normal(size=S), rng.normal(size=S)
    if kind == "small im":
        im = im * 1e-25
    if kind == "small re":
        re = re * 1e-18
    if kind == "decades":
        re, im = re * 10.0 ** rng.uniform(-9, 9, S), im * 10.0 ** rng.uniform(-9, 9, S)
    if kind == "many decades":
        re, im = re * 10.0 ** rng.uniform(-24, 24, S), im * 10.0 ** rng.uniform(-24, 24, S)
    if kind == "cancelling":                                      # large terms that cancel in pairs, small ones left
        re[: S // 2 * 2: 2], im[: S // 2 * 2: 2] = 1e9 * re[: S // 2 * 2: 2], 1e9 * im[: S // 2 * 2: 2]
        re[1::2], im[1::2] = -re[: S // 2 * 2: 2], -im[: S // 2 * 2: 2]
        re[-1], im[-1] = 1e-7, 3e-8
    if kind == "whole":
        re, im = np.rint(re * 8), np.zeros(S)
    if kind == "subnormal":
        least = 5e-324 if precision == "fp64" else 2.0 ** -149
        re, im = np.rint(re * 9) * least, np.rint(im * 9) * least
    return re + 1j * im


@pytest.mark.parametrize("q", [2, 3, 4])
@pytest.mark.parametrize("n,S,N", [(50, 1, 3), (64, 64, 70), (65, 66, 33), (140, 131, 65), (250, 40, 17)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["plain", "small im", "small re", "decades", "cancelling", "whole", "subnormal",
                                  "many decades"])
def test_points_every_component_in_full(q, n, S, N, precision, kind):
    """Each component is the exact sum, rounded once: within half a unit of its own last place, whatever the sizes
    of the others. q = 3: and 2^-90 of the two sums that meet in it."""
    print(f"points in full q={q} n={n} S={S} N={N} {precision} {kind}", flush=True)
    rng = np.random.default_rng(q * 100 + S)
    locq, pts = rng.integers(0, q, size=(n, S)), rng.integers(0, q, size=(N, n))
    if kind == "cancelling":
        locq[:, 1::2] = locq[:, : S // 2 * 2: 2]
    dev, n_pad = dv.current_device(), dv.n_pad_of(n)
    at = dv.strengths_tensor(_strengths(kind, S, precision, rng), precision, dev)
    a = at.cpu().numpy().astype(np.complex128)
    x = dv.evaluate_points(q, n, dv.digits_tensor(pts, n_pad, dev), dv.digits_tensor(locq.T, n_pad, dev), at,
                           precision).cpu().numpy().astype(np.complex128)
    half_ulp = Fraction(1, 2 ** 53) if precision == "fp64" else Fraction(1, 2 ** 24)
    tiny = Fraction(1, 2 ** 1075) if precision == "fp64" else Fraction(1, 2 ** 150)   # half the smallest number
    for got, (re, im, pr, pi) in zip(x, _exact(q, pts, locq, a)):
        for g, ref, parts in ((got.real, re, pr), (got.imag, im, pi)):
            bound = max(half_ulp * abs(ref) * (1 + Fraction(1, 10 ** 6)), tiny if q == 3 else 0)
            assert abs(Fraction(float(g)) - ref) <= bound + (parts / 2 ** 90 if q == 3 else 0), (g, float(ref))


@pytest.mark.parametrize("q", [2, 3, 4])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_points_of_too_wide_a_range_by_the_table(q, precision):
    """Components that four limbs do not span (one part of q = 2 is enough) come out as the table form gives them."""
    rng = np.random.default_rng(q)
    n, S, N = 70, 150, 130
    dev, n_pad = dv.current_device(), dv.n_pad_of(n)
    a = rng.normal(size=S) * 10.0 ** rng.uniform(-18, 18, S) + 1j * rng.normal(size=S)
    a[:2] = [1e-37 / 3, 2e38]
    m = dv.digits_tensor(rng.integers(0, q, size=(N, n)), n_pad, dev)
    k = dv.digits_tensor(rng.integers(0, q, size=(S, n)), n_pad, dev)
    at = dv.strengths_tensor(a, precision, dev)
    got = dv.evaluate_points(q, n, m, k, at, precision)
    ref = torch.empty_like(got)
    K.EvalPoints([dict(q=q, n=n, S=S, m=m, K=k, a=at, x=ref)], dv.PRECISIONS[precision][0], table=True).launch()
    np.testing.assert_array_equal(got.cpu().numpy(), ref.cpu().numpy())
