"""Coset evaluation through the folded spectrum (qsft_fold_*) on the GPU,
every sample against the direct sum a_s w^{<M_c l + d_p, k_s>} in FP64.

Tolerances (max-abs over max |value|): the terms and bin sums are FP64, the
inverse transform has at most b q-point stages, so FP64 is within 1e-12 and
FP32, with b log2(q) <= 16 rounded additions of partial sums no larger than
sum |a_s|, within 2e-6 of the largest sample.
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from qsft_amd import _lib as L
    from qsft_amd import device as dv
    from qsft_amd import kernels as K

# whole-row kernels (q = 4, b = 4..7, the last in FP32 only) with rows that do
# not fill the last workgroup and phases beyond their LDS buffer (S = 5000, 9000); one tile, several tiles and several passes of the others (b = 7,
# q = 2 b = 13, q = 20 b = 4), the generic radix (q = 7, 50, 64), one to four
# digit blocks; supports around the 16-, 64- and 2048-wide blocks of the prep
CASES = [(4, 10, 4, 100, 3, 11), (4, 50, 6, 1000, 2, 21), (4, 64, 6, 65, 1, 17), (4, 100, 7, 2049, 2, 33),
         (4, 9, 5, 64, 3, 10), (4, 20, 2, 16, 2, 5), (2, 8, 1, 1, 1, 9), (2, 30, 13, 63, 2, 16), (3, 67, 7, 777, 2, 19),
         (20, 16, 3, 2000, 2, 7), (20, 12, 4, 300, 1, 2), (5, 130, 4, 129, 2, 15), (7, 200, 3, 500, 2, 4),
         (50, 11, 2, 33, 1, 3), (64, 256, 2, 17, 2, 3), (4, 12, 3, 5000, 1, 12), (2, 40, 6, 0, 2, 3),
         (4, 30, 5, 700, 2, 13), (4, 33, 6, 5000, 1, 3), (4, 70, 7, 9000, 1, 2), (4, 8, 7, 0, 1, 2), (2, 60, 14, 500, 1, 3),
         (5, 20, 6, 900, 2, 3)]


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


def _item(q, n, b, Ms, Ds, loc, a, precision):
    dev, n_pad = dv.current_device(), dv.n_pad_of(n)
    dt = torch.complex64 if precision == "fp32" else torch.complex128
    return dict(q=q, n=n, b=b, C=len(Ms), P=Ds[0].shape[0], S=loc.shape[1], Mt=dv.Mt_tensor(Ms, b, n_pad, dev),
                D=dv.D_tensor(Ds, n_pad, dev), K=dv.digits_tensor(loc.T, n_pad, dev),
                a=dv.strengths_tensor(a, "fp64", dev),
                x=torch.empty((len(Ms), Ds[0].shape[0], q ** b), dtype=dt, device=dev))


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("q,n,b,S,C,P", [c for c in CASES if c[3] > 0])
def test_fold_with_the_sub_transform_in_the_same_launch(q, n, b, S, C, P, precision, tol):
    """transform=True: rows come out as their sub-transforms, after the passes
    left to Dft where they are more than one tile. A sample's error is at most tol of the largest sample and
    independent of its neighbours', so the error of a mean of q^b of them is
    that over sqrt(q^b), times 6 for the largest of all values, and as much
    again for the forward transform's own rounding."""
    print(f"fold + sub-DFT q={q} n={n} b={b} S={S} C={C} P={P} {precision}", flush=True)
    Ms, Ds, loc, a = _inputs(q, n, b, S, C, P, seed=q * 97 + n + S)
    it = _item(q, n, b, Ms, Ds, loc, a, precision)
    ev = K.EvalFold([it], L.QSFT_F32 if precision == "fp32" else L.QSFT_F64, transform=True)
    ev.launch()
    assert bool(ev.rest) == (q ** b * (8 if precision == "fp32" else 16) * (1 if q in (2, 3, 4, 5, 20) else 2) > 147456)
    K.Dft(ev.rest, L.QSFT_F32 if precision == "fp32" else L.QSFT_F64).launch()
    got, ref = it["x"].cpu().numpy(), _direct(q, b, Ms, Ds, loc, a)
    bound = tol * np.max(np.abs(ref)) * 12 / q ** (b / 2)
    ref = np.fft.fftn(ref.reshape(C, P, *[q] * b), axes=range(2, 2 + b)).reshape(C, P, -1) / q ** b
    assert np.max(np.abs(got - ref)) <= bound


@pytest.mark.parametrize("b,count", [(4, 15), (4, 29), (5, 29), (6, 15), (6, 29)])
def test_fold_of_many_rows_gives_the_bits_of_one_instance(b, count):
    """Launches of 4096 and 8192 rows and more give a workgroup two or four sets
    of rows of a group (P = 101 leaves the last one short): the same bits."""
    print(f"fold many rows b={b} count={count}", flush=True)
    g = [_inputs(4, 50, b, 300 + 40 * i, 3, 101, seed=i) for i in range(count)]
    items = [_item(4, 50, b, *x, "fp32") for x in g]
    assert sum(it["C"] * it["P"] for it in items) >= (4096 if count == 15 else 8192)
    K.EvalFold(items, L.QSFT_F32).launch()
    for i in (0, count // 2, count - 1):
        alone = _item(4, 50, b, *g[i], "fp32")
        K.EvalFold([alone], L.QSFT_F32).launch()
        assert torch.equal(torch.view_as_real(alone["x"]), torch.view_as_real(items[i]["x"]))


def test_fold_gives_the_same_bits_alone_and_beside_larger_rows():
    """A launch's workgroup size follows its largest tile: q = 2 and q = 3
    instances with crowded bins alone and beside rows of up to 128 KiB."""
    print("fold alone and beside larger rows", flush=True)
    shapes = [(2, 6, 1500), (2, 10, 700), (2, 14, 300), (3, 4, 1000), (3, 8, 200), (20, 2, 3000), (20, 3, 500)]
    g = [(q, b, _inputs(q, 20, b, S, 2, 5, seed=S)) for q, b, S in shapes]
    items = [_item(q, 20, b, *x, "fp32") for q, b, x in g]
    K.EvalFold(items, L.QSFT_F32, transform=True).launch()
    for (q, b, x), it in zip(g, items):
        alone = _item(q, 20, b, *x, "fp32")
        K.EvalFold([alone], L.QSFT_F32, transform=True).launch()
        assert torch.equal(torch.view_as_real(alone["x"]), torch.view_as_real(it["x"])), (q, b)


BAD = [complex(np.inf, 0), complex(0, -np.inf), complex(-np.inf, 2), complex(np.inf, np.inf), complex(np.nan, 1),
       complex(2, np.nan)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("q,n,b,S", [(2, 9, 5, 30), (2, 20, 14, 70), (3, 7, 4, 65), (4, 9, 3, 30), (4, 20, 4, 100),
                                     (4, 20, 5, 300), (4, 9, 6, 40), (4, 9, 7, 40), (5, 9, 3, 30), (20, 5, 2, 33),
                                     (20, 6, 4, 20), (7, 9, 2, 30), (50, 4, 2, 20)])
def test_fold_of_strengths_that_are_not_finite(q, n, b, S, precision):
    """One such strength, or several, makes every sample what the sum over all supports makes it: an infinity of
    the same sign or a NaN. Sub-transforms, sums over such samples, are NaN throughout."""
    print(f"fold not finite q={q} n={n} b={b} S={S} {precision}", flush=True)
    code = L.QSFT_F32 if precision == "fp32" else L.QSFT_F64
    for bad in [[v] for v in BAD] + [[BAD[0], BAD[1]], [BAD[0], -BAD[0], BAD[2]], BAD]:
        Ms, Ds, loc, a = _inputs(q, n, b, S, 2, 3, seed=S)
        a[np.random.default_rng(b).permutation(S)[:len(bad)]] = bad
        it = _item(q, n, b, Ms, Ds, loc, a, precision)
        it["a"] = dv.strengths_tensor(a, precision, dv.current_device())
        K.EvalFold([it], code).launch()
        ref = dict(it, x=torch.empty_like(it["x"]))
        K.EvalCosets([ref], code).launch()
        np.testing.assert_array_equal(torch.view_as_real(it["x"]).cpu().numpy(),
                                      torch.view_as_real(ref["x"]).cpu().numpy())
        ev = K.EvalFold([it], code, transform=True)
        ev.launch()
        K.Dft(ev.rest, code).launch()
        assert torch.isnan(torch.view_as_real(it["x"])).all()


@pytest.mark.parametrize("q,b", [(2, 6), (2, 13), (4, 3), (4, 4), (4, 5), (4, 6), (4, 7)])
@pytest.mark.parametrize("S", [64, 65, 300, 1500, 5000])
def test_fold_rounds_a_crowded_bin_once(q, b, S):
    """Every support in one bin, FP32: a sample is the bin's sum turned by a power of w, exact for q = 2 and 4, so
    each part of it is within half a unit of its last place of the sum of its terms (taken in FP64 here: 2^-53 of
    the sizes of at most S terms each time one is added)."""
    print(f"fold one bin q={q} b={b} S={S}", flush=True)
    n, C, P = b + 5, 2, 3
    Ms, Ds, loc, a = _inputs(q, n, b, S, C, P, S)
    loc[:b] = loc[:b, :1]                                          # M picks the first b digits: one bin
    for M in Ms:
        M[:] = 0
        M[:b] = np.eye(b, dtype=int)
    a = a.astype(np.complex64).astype(np.complex128)
    x = _run(q, n, b, Ms, Ds, loc, a, "fp32")
    w = np.array([1, 1j, -1, -1j])[::4 // q]
    lq = (np.arange(q ** b)[:, None] // q ** np.arange(b - 1, -1, -1)) % q
    turn = w[(lq @ loc[:b, 0]) % q]
    for c in range(C):
        ref = (w[(Ds[c] @ loc) % q] @ a)[:, None] * turn[None, :]
        for got, want in ((x[c].real, ref.real), (x[c].imag, ref.imag)):
            assert (np.abs(got - want) <= 2.0 ** -24 * (1 + 1e-6) * np.abs(want) + S * 2.0 ** -53 * np.abs(a).sum()).all()


def _scheduled(it, precision, transform, s):
    """EvalFold of one instance (and the passes left to Dft) on the schedule of the DftDesc s."""
    code, dev = (L.QSFT_F32 if precision == "fp32" else L.QSFT_F64), dv.current_device()
    q, b, C, P, S = (it[k] for k in ("q", "b", "C", "P", "S"))
    nbytes = L.lib.qsft_fold_workspace_bytes(q, b, C, P, S, 0)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    d = L.FoldDesc()
    L.check(L.lib.qsft_fold_bind(ctypes.byref(d), q, it["n"], b, C, P, S, it["Mt"].shape[-1], 0, code, L.QSFT_F64,
                                 int(transform), C * P, *(it[k].data_ptr() for k in ("Mt", "D", "K", "a", "x")),
                                 ws.data_ptr(), nbytes))
    assert d.rpw == 0                                              # a shape of the tile kernel
    d.n_pass = s.n_pass
    for p in range(s.n_pass):
        d.pass_d0[p], d.pass_d1[p], d.pass_ti[p], d.pass_ta[p] = s.pass_d0[p], s.pass_d1[p], s.pass_ti[p], s.pass_ta[p]
        d.pass_blocks[p] = s.pass_blocks[p]
        d.pass_lds[p] = L.lib.qsft_dft_lds_bytes(ctypes.byref(s), p, code)
        assert 0 < d.pass_lds[p] <= 65536
    d.tile_bins = q ** (b - s.pass_d0[0]) * s.pass_ta[0]
    d.tiles = q ** b // d.tile_bins
    pb, rb = ctypes.c_int(), ctypes.c_int()
    assert L.lib.qsft_fold_blocks(ctypes.byref(d), ctypes.byref(pb), ctypes.byref(rb)) == 0
    blocks = [[pb.value], [rb.value]] + [[d.pass_blocks[p]] for p in range(d.n_pass)]
    buf, dptr, pres, tots = K.pack([d], blocks, dev)
    st = K.stream_handle()
    L.check(L.lib.qsft_fold_prep(dptr, pres[0], pres[1], 1, tots[0], tots[1], st))
    for p in range(d.n_pass):
        L.check(L.lib.qsft_fold_rows(dptr, pres[2 + p], 1, tots[2 + p], p, code | (q << 8), d.pass_lds[p], st))
    if transform and d.n_pass > 1:
        r = L.DftDesc()
        L.check(L.lib.qsft_fold_rest(ctypes.byref(d), ctypes.byref(r)))
        K.Dft([dict(q=q, b=b, rows=r.rows, inp=it["x"], out=it["x"], desc=r)], code).launch()
    torch.cuda.synchronize()                                       # buf and ws are released


@pytest.mark.parametrize("transform", [False, True])
@pytest.mark.parametrize("q,b,precision", [(20, 4, "fp32"), (20, 3, "fp32"), (20, 3, "fp64"), (2, 16, "fp32"),
                                           (3, 10, "fp64"), (4, 8, "fp32"), (5, 6, "fp64"), (7, 5, "fp32"),
                                           (11, 3, "fp64")])
def test_fold_gives_the_same_bits_on_every_schedule(q, b, precision, transform):
    """Samples and sub-transforms do not depend on how the axes are grouped into passes."""
    print(f"fold schedules q={q} b={b} {precision} transform={transform}", flush=True)
    code = L.QSFT_F32 if precision == "fp32" else L.QSFT_F64
    x = _inputs(q, 20, b, 150, 1, 3, seed=q + b)
    first, groups = None, set()
    for cand in range(400):
        s = L.DftDesc(q=q, b=b, rows=3, in_stride=1, in_row_stride=q ** b)
        if L.lib.qsft_dft_plan_candidate(ctypes.byref(s), code, cand) != L.QSFT_OK:
            break
        split = tuple(s.pass_d0[p] for p in range(s.n_pass))
        if split in groups or s.n_pass > 1 and len(groups) >= 8:
            continue
        if L.lib.qsft_dft_lds_bytes(ctypes.byref(s), 0, code) > 65536:
            continue
        groups.add(split)
        it = _item(q, 20, b, *x, precision)
        _scheduled(it, precision, transform, s)
        bits = torch.view_as_real(it["x"])
        first = bits if first is None else first
        assert torch.equal(bits, first), split
    assert len(groups) >= 2


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("b,S", [(4, 256), (4, 257), (4, 3000), (5, 1600), (5, 1601), (5, 4097)])
def test_fold_on_both_sides_of_the_line_between_its_row_kernels(b, S, precision, tol):
    """q = 4: samples and sub-transforms where the whole-row kernel ends and the tile kernel begins, the two beside
    each other in one launch, each with the bits it has alone (bounds as above)."""
    print(f"fold line b={b} S={S} {precision}", flush=True)
    code = L.QSFT_F32 if precision == "fp32" else L.QSFT_F64
    x = _inputs(4, 21, b, S, 2, 7, seed=S)
    few = _inputs(4, 21, b, 50, 2, 7, seed=S)
    ref = _direct(4, b, *x)
    for transform in (False, True):
        items = [_item(4, 21, b, *v, precision) for v in (few, x, few)]
        K.EvalFold(items, code, transform=transform).launch()
        bound, want = tol * np.max(np.abs(ref)), ref
        if transform:
            want = np.fft.fftn(ref.reshape(2, 7, *[4] * b), axes=range(2, 2 + b)).reshape(2, 7, -1) / 4 ** b
            bound *= 12 / 4 ** (b / 2)
        assert np.max(np.abs(items[1]["x"].cpu().numpy() - want)) <= bound
        for it, v in zip(items, (few, x, few)):
            alone = _item(4, 21, b, *v, precision)
            K.EvalFold([alone], code, transform=transform).launch()
            assert torch.equal(torch.view_as_real(alone["x"]), torch.view_as_real(it["x"]))


def _unaligned(t):
    """The same values in a view that starts one element into its storage."""
    v = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return v.copy_(t)


@pytest.mark.parametrize("q,b", [(4, 4), (3, 3)])
def test_fold_reads_views_that_start_anywhere_at_every_launch(q, b):
    """Mt, D, K and complex64 a that are not 16-byte aligned, changed between the launches of one EvalFold."""
    print(f"fold unaligned views q={q} b={b}", flush=True)
    first, second = (_item(q, 13, b, *_inputs(q, 13, b, 37, 2, 5, seed=s), "fp32") for s in (1, 2))
    want = []
    for it in (first, second):
        it["a"] = it["a"].to(torch.complex64)
        K.EvalFold([it], L.QSFT_F32).launch()
        want.append(it["x"].clone())
        x = dv.evaluate_cosets(q, 13, b, *(_unaligned(it[k]) for k in ("Mt", "D", "K", "a")), "fp32")
        assert torch.equal(torch.view_as_real(x), torch.view_as_real(want[-1]))
    views = dict(first, **{k: _unaligned(first[k]) for k in ("Mt", "D", "K", "a")})
    assert all(views[k].data_ptr() % 16 for k in ("Mt", "D", "K", "a"))
    ev = K.EvalFold([views], L.QSFT_F32)
    for it, x in zip((first, second, first), (want[0], want[1], want[0])):
        for k in ("Mt", "D", "K", "a"):
            views[k].copy_(it[k])
        ev.launch()
        assert torch.equal(torch.view_as_real(views["x"]), torch.view_as_real(x))


@pytest.mark.parametrize("q,b,S", [(2, 3, 8193), (2, 1, 12289), (3, 7, 8200), (4, 4, 10240), (4, 6, 16385), (20, 4, 8250),
                                   (2, 16, 9000), (7, 5, 8193), (4, 7, 67000)])
def test_fold_ranks_many_supports_in_two_steps(q, b, S):
    """More than 8192 supports are ranked within chunks of 2048 and by a search in the others: the bits of the one-step
    ranking, alone and in a launch with few supports, for bins of many supports of all chunks and for several tiles."""
    print(f"fold two-step ranks q={q} b={b} S={S}", flush=True)
    x = _inputs(q, 17, b, S, 2, 3, seed=S)
    few = _inputs(q, 17, b, 70, 2, 3, seed=1)
    it, small = _item(q, 17, b, *x, "fp64"), _item(q, 17, b, *few, "fp64")
    ev = K.EvalFold([small, it], L.QSFT_F64)
    assert ev.chunks
    ev.launch()
    got, got_small = it["x"].clone(), small["x"].clone()
    if S * q ** b < 10 ** 7:
        ref = _direct(q, b, *x)
        assert np.max(np.abs(got.cpu().numpy() - ref)) <= 1e-12 * np.max(np.abs(ref))
    nbytes = L.lib.qsft_fold_workspace_bytes(q, b, 2, 3, S, 0)
    for one_step in (True, False):
        it["x"].fill_(0)
        if one_step:
            d = L.FoldDesc()
            ws = torch.empty(nbytes, dtype=torch.uint8, device=it["x"].device)
            L.check(L.lib.qsft_fold_bind(ctypes.byref(d), q, 17, b, 2, 3, S, it["Mt"].shape[-1], 0, L.QSFT_F64, L.QSFT_F64,
                                         0, 6, *(it[k].data_ptr() for k in ("Mt", "D", "K", "a", "x")), ws.data_ptr(),
                                         nbytes))
            assert not d.chunk
            pb, rb = ctypes.c_int(), ctypes.c_int()
            assert L.lib.qsft_fold_blocks(ctypes.byref(d), ctypes.byref(pb), ctypes.byref(rb)) == 0
            buf, dptr, pres, tots = K.pack([d], [[pb.value], [rb.value]] + [[d.pass_blocks[p]] for p in range(d.n_pass)],
                                           it["x"].device)
            st = K.stream_handle()
            L.check(L.lib.qsft_fold_prep(dptr, pres[0], pres[1], 1, tots[0], tots[1], st))
            for p in range(d.n_pass):
                L.check(L.lib.qsft_fold_rows(dptr, pres[2 + p], 1, tots[2 + p], p,
                                             L.QSFT_F64 | (q << 8) | ((b << 16) if d.rpw else 0), d.pass_lds[p], st))
            torch.cuda.synchronize()
        else:
            K.eval_fold(q, 17, b, *(it[k] for k in ("Mt", "D", "K", "a", "x")))
        assert torch.equal(torch.view_as_real(it["x"]), torch.view_as_real(got))
    K.EvalFold([small], L.QSFT_F64).launch()
    assert torch.equal(torch.view_as_real(small["x"]), torch.view_as_real(got_small))
