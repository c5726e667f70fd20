"""Host tables of the drop-in transform: key tuples, row order and the form of the delay rows, each against
the general routine that it stands in for."""
import numpy as np
import pytest
import torch

from qsft_amd import kernels as K
from qsft_amd.utils import digit_tuples, lex_order, sort_qary_vecs


@pytest.mark.parametrize("q,n,m", [(2, 8, 200), (4, 50, 1000), (127, 3, 300), (3, 1, 3), (20, 5, 1), (5, 4, 0)])
def test_keys_and_order(q, n, m):
    rng = np.random.default_rng(q + n)
    rows = rng.permutation(np.unique(rng.integers(0, q, size=(m, n)), axis=0).reshape(-1, n))
    keys = digit_tuples(rows)
    assert keys == [tuple(r) for r in rows]
    assert all(type(d) is np.int64 for key in keys for d in key)
    if len(rows):
        np.testing.assert_array_equal(rows[lex_order(rows)], sort_qary_vecs(rows))


def _forms(q, n, C, R, rng):
    """Delay rows [C][R (n + 1)][n] of every form: one per group or shared, +1 / -1 steps, arbitrary."""
    step = np.eye(n + 1, n, -1, dtype=int)
    for sign in (1, -1):
        base = rng.integers(0, q, size=(C, R, 1, n))
        yield ((base + sign * step) % q).reshape(C, -1, n)
        yield np.repeat(((base[:1] + sign * step) % q).reshape(1, -1, n), C, axis=0)
    mixed = ((rng.integers(0, q, size=(C, R, 1, n)) + step) % q).reshape(C, -1, n)
    mixed[-1, -1, 0] = (mixed[-1, -1, 0] + 1) % q                     # one digit off in the last group
    yield mixed
    yield rng.integers(0, q, size=(C, R * (n + 1), n))


@pytest.mark.parametrize("q,n,C,R", [(2, 5, 3, 2), (3, 4, 1, 1), (4, 50, 3, 2), (20, 7, 2, 1), (4, 3, 2, 65)])
@pytest.mark.parametrize("p1", ["rows", "other"])
def test_delay_form_as_on_the_device(q, n, C, R, p1):
    rng = np.random.default_rng(q * n + C)
    p1 = n + 1 if p1 == "rows" else n
    for rows in _forms(q, n, C, R, rng):
        D = np.zeros((C, rows.shape[1], n + 3), np.int8)
        D[:, :, :n] = rows
        it = dict(C=C, q=q, n=n, p1=p1, D=torch.from_numpy(D))
        assert K.peel_flags(dict(it, **K.delay_form(D, q, n, p1))) == K.peel_flags(it)
        D[0, 0, n] = 1                                               # a digit in the padding
        it["D"] = torch.from_numpy(D)
        assert K.peel_flags(dict(it, **K.delay_form(D, q, n, p1))) == K.peel_flags(it)
