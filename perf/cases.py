"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is a dict of plain values. `listed()` gives the fixed cases, `draw(rng)` further ones of the same ranges,
`prepare(case, seed)` what a user's program holds before the call (inputs on the GPU, signals, plans, a server),
`run(state)` one pass through the public entry points, `work(case)` the bytes and operations the pass cannot do
without, `exact(case, seed)` the results in 64 bits where they have a closed form.

Kinds of case, by the entry point they call:

* "samples"    `qsft_amd.device.evaluate_cosets`: the samples of a sparse signal on C x P cosets (query generation
               and evaluation), the front end of every synthetic signal, FP32 and FP64.
* "subdft"     `qsft_amd.device.subtransform`: batched [q]*b transforms of stored samples.
* "heldout"    `qsft_amd.device.evaluate_points`: a recovered spectrum predicted at random held-out queries.
* "decode"     `qsft_amd.kernels.Assemble` + `PeelBatch`: working transforms with noise, then detection and peeling
               of a batch of stored sub-transforms in FP64.
* "transform"  the drop-in call of the reference's scripts: `SyntheticSubsampledSignal(...)`, then
               `QSFT(...).transform(signal, report=True, sort=True)`, one instance in FP64.
* "served"     `qsft_amd.serving.Server`: requests submitted and drained, FP32 samples with FP64 peeling.
"""
import math

import numpy as np
import torch

from qsft_amd import _lib as L
from qsft_amd import device as dv
from qsft_amd import kernels
from qsft_amd.engine import TransformSpec
from qsft_amd.qsft import QSFT
from qsft_amd.serving import Server
from qsft_amd.synthetic_signal import SyntheticSubsampledSignal

BINS_MIN, BINS_MAX = 64, 16384                      # q^b of single workloads: 4^4 .. 4^7, 20^3, 3^8, 2^12
HBM_BUDGET = 64 << 30


def listed():
    return [
        # the smallest call: the plain configuration (noiseless, identity delays) through the drop-in classes,
        # as an interactive script or a unit test makes it; latency and launches count
        dict(name="transform_k0_fp64", kind="transform", q=4, n=10, S=100, b=4, C=3, R=1, method="identity", snr=None),
        # the plain single-instance FP64 path at the headline size, 10 dB, nso detection
        dict(name="transform_k1_fp64", kind="transform", q=4, n=50, S=1000, b=6, C=3, R=2, method="nso", snr=10.0),
        # samples of one headline-size signal in FP64 (what a signal's constructor spends its time on)
        dict(name="samples_k1_fp64", kind="samples", q=4, n=50, S=1000, b=6, C=3, P=102, precision="fp64"),
        # the protein alphabet in FP32
        dict(name="samples_q20_fp32", kind="samples", q=20, n=16, S=2000, b=3, C=3, P=34, precision="fp32"),
        # ragged sizes: q = 3, two digit blocks, odd S and P
        dict(name="samples_q3_odd_fp64", kind="samples", q=3, n=67, S=777, b=7, C=2, P=131, precision="fp64"),
        # sub-transforms of a batch of 32 headline-size signals, FP32: larger than the caches
        dict(name="subdft_q4_fp32", kind="subdft", q=4, b=6, rows=9792, stride=1, precision="fp32"),
        # radix 20 in FP64, one signal
        dict(name="subdft_q20_fp64", kind="subdft", q=20, b=3, rows=102, stride=1, precision="fp64"),
        # held-out scoring of a recovered spectrum (1000 coefficients)
        dict(name="heldout_q4_fp64", kind="heldout", q=4, n=50, S=1000, N=100003, precision="fp64"),
        # detection and peeling of 8 stored headline-size transforms, fresh device noise, FP64
        dict(name="decode_k1_fp64", kind="decode", q=4, n=50, S=1000, b=6, C=3, R=2, snr=10.0, count=8),
        # one request at the headline size: serving latency with nothing else on the GPU
        dict(name="served_k1_one", kind="served", mix="k1", count=1, large=0, snr=20.0),
        # a full batch of distinct requests at the headline size: serving throughput
        dict(name="served_k1_32", kind="served", mix="k1", count=32, large=0, snr=20.0),
        # the serving mix: uneven requests (q in {2, 3, 4, 20}, n 8..64, S 10..2000, 5..30 dB) and one large job
        # (q = 4, n = 100, S = 5000, b = 7)
        dict(name="served_mix_20", kind="served", mix="k3", count=20, large=1, shapes=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, most_rows=256):
    """(q, b, n, R) with q^b in the workloads' range and R (n + 1) <= most_rows."""
    q = rng.choice([2, 3, 4, 4, 4, 5, 20])
    bs = [b for b in range(2, 16) if BINS_MIN <= q ** b <= BINS_MAX]
    b = rng.choice(bs)
    R = rng.choice([1, 2, 2])
    n = rng.randint(max(8, b), min(110, most_rows // R - 1))
    return q, b, n, R


def draw(rng):
    """One more case of the ranges the listed ones stand for; none costs more than the largest of those."""
    while True:
        c = _draw(rng)
        if work(c)["bytes"] <= max(work(x)["bytes"] for x in listed()):
            return c


def _draw(rng):
    kind = rng.choice(["samples", "samples", "subdft", "subdft", "heldout", "decode", "transform", "served", "served"])
    if kind == "samples":
        q, b, n, R = _shape(rng)
        S = min(_log(rng, 10, 5000), q ** n // 8)
        return dict(kind=kind, q=q, n=n, S=S, b=b, C=rng.randint(1, 4), P=R * (n + 1),
                    precision=rng.choice(["fp32", "fp64"]))
    if kind == "subdft":
        q, b, _, _ = _shape(rng)
        precision = rng.choice(["fp32", "fp64"])
        most = (9792 * 4096 // 2) // q ** b                     # samples of the largest listed case, in FP64
        rows = _log(rng, 11, max(12, most))
        stride = rng.choice([1, 1, 1, q])                          # a smaller b of the same stored samples
        return dict(kind=kind, q=q, b=b, rows=max(1, rows // stride), stride=stride, precision=precision)
    if kind == "heldout":
        q, _, n, _ = _shape(rng)
        S = min(_log(rng, 10, 4000), q ** n // 8)
        return dict(kind=kind, q=q, n=n, S=S, N=_log(rng, 1000, 2e8 / max(S, 1000)), precision="fp64")
    if kind == "served":
        if rng.random() < 0.5:
            return dict(kind=kind, mix="k1", count=_log(rng, 1, 32), large=0, snr=rng.choice([20.0, 25.0, 30.0]))
        return dict(kind=kind, mix="k3", count=_log(rng, 2, 19), large=rng.randint(0, 1), shapes=rng.randint(2, 10 ** 6))
    # one instance or a few, a load at which three groups peel: S between a fiftieth and a third of the bins
    q, b, n, R = _shape(rng)
    S = min(_log(rng, max(8, q ** b // 50), max(9, q ** b // 3)), 5000, q ** n // 8)
    snr = rng.choice([10.0, 20.0, 30.0])
    if kind == "decode":
        return dict(kind=kind, q=q, n=n, S=S, b=b, C=3, R=2 if 2 * (n + 1) <= 256 else 1, snr=snr,
                    count=_log(rng, 1, 8) if q ** b <= 4096 else 1)
    method = rng.choice(["nso", "nso", "identity"])
    return dict(kind=kind, q=q, n=n, S=S, b=b, C=3, R=R if method == "nso" else 1, method=method,
                snr=snr if method == "nso" else None)


# ------------------------------------------------------------------ inputs


def _support(g, q, n, S):
    """Distinct uniform support digits (n, S) and strengths |a| ~ U[1, 10], phase ~ U[0, 2 pi)."""
    loc = g.integers(0, q, size=(n, S))
    while True:
        _, first = np.unique(loc, axis=1, return_index=True)
        if first.size == S:
            break
        dup = np.setdiff1d(np.arange(S), first)
        loc[:, dup] = g.integers(0, q, size=(n, dup.size))
    return loc, g.uniform(1, 10, S) * np.exp(2j * np.pi * g.uniform(size=S))


def _delays(g, q, n, R, method="nso"):
    src = np.vstack([np.zeros((1, n), int), np.eye(n, dtype=int)])
    if method == "identity":
        return src
    return np.vstack([(g.integers(0, q, n) - src) % q for _ in range(R)])


def _noise_sd(a, snr):
    return 0.0 if snr is None else float(np.sqrt(np.sum(np.abs(a) ** 2) / 10 ** (snr / 10)))


def _instance(c, g):
    """Support, strengths, group matrices and delay rows of one instance."""
    loc, a = _support(g, c["q"], c["n"], c["S"])
    Ms = [g.integers(0, c["q"], size=(c["n"], c["b"])) for _ in range(c["C"])]
    if "P" in c:
        D = _delays(g, c["q"], c["n"], -(-c["P"] // (c["n"] + 1)))[:c["P"]]
    else:
        D = _delays(g, c["q"], c["n"], c["R"], c.get("method", "nso"))
    return loc, a, Ms, D


def _spec(q, n, S, b, snr, g):
    loc, a = _support(g, q, n, S)
    Ms = [g.integers(0, q, size=(n, b)) for _ in range(3)]
    sp = TransformSpec(q=q, n=n, b=b, C=3, R=2, locq=loc.astype(np.int8), strengths=a, Ms=Ms, D=_delays(g, q, n, 2),
                       noise_sd=_noise_sd(a, snr), method="nso", seed=int(g.integers(0, 2 ** 62)))
    sp.wire()                                                      # the request's payload, as a client sends it
    return sp


def _served_shapes(c):
    """(q, n, S, b, snr) of the case's requests."""
    if c["mix"] == "k1":
        return [(4, 50, 1000, 6, c["snr"])] * c["count"]
    g = np.random.default_rng(c["shapes"])
    out = [(4, 100, 5000, 7, float(g.uniform(5, 30)))] * c["large"]
    while len(out) < c["count"]:
        q, n = int(g.choice([2, 3, 4, 20])), int(g.integers(8, 65))
        S = max(2, min(int(np.exp(g.uniform(np.log(10), np.log(2000)))), q ** n // 8))
        out.append((q, n, S, int(np.ceil(np.log(S) / np.log(q))) + 1, float(g.uniform(5, 30))))
    return out


def _aliased(q, b, Ms, D, loc, a):
    """Sub-transforms in closed form, complex128 [C][P][q^b]: U[c][p][j] = sum over M_c^T k = j of a_k w^<d_p, k>."""
    w = np.exp(2j * np.pi * np.arange(q) / q)
    terms = a[None, :] * w[(D @ loc) % q]
    place = q ** np.arange(b - 1, -1, -1)
    U = np.zeros((len(Ms), D.shape[0], q ** b), complex)
    for c, M in enumerate(Ms):
        np.add.at(U[c].T, place @ ((M.T @ loc) % q), terms.T)
    return U


def _complex(gen, shape, dtype):
    real = torch.float32 if dtype == torch.complex64 else torch.float64
    return torch.view_as_complex(torch.randn(*shape, 2, generator=gen, device=gen.device, dtype=real))


def _table(k, values, S):
    """Recovered rows in a table of fixed size (zeros past the rows found), as a client stores uneven answers."""
    keys = np.zeros((2 * S + 64, k.shape[1]), np.int8)
    vals = np.zeros(2 * S + 64, values.dtype)
    keys[:len(k)] = k
    vals[:len(k)] = values
    return keys, vals


def prepare(case, seed):
    c, g = case, np.random.default_rng(seed)
    dev = dv.current_device()
    kind = c["kind"]
    if kind == "samples":
        loc, a, Ms, D = _instance(c, g)
        n_pad = dv.n_pad_of(c["n"])
        return dict(c, args=(c["q"], c["n"], c["b"], dv.Mt_tensor(Ms, c["b"], n_pad, dev),
                             dv.D_tensor([D] * c["C"], n_pad, dev), dv.digits_tensor(loc.T, n_pad, dev),
                             dv.strengths_tensor(a, c["precision"], dev), c["precision"]))
    if kind == "subdft":
        gen = torch.Generator(device=dev).manual_seed(seed)
        dt = torch.complex64 if c["precision"] == "fp32" else torch.complex128
        return dict(c, x=_complex(gen, (c["rows"], c["q"] ** c["b"] * c["stride"]), dt))
    if kind == "heldout":
        loc, a = _support(g, c["q"], c["n"], c["S"])
        n_pad = dv.n_pad_of(c["n"])
        m = g.integers(0, c["q"], size=(c["N"], c["n"]), dtype=np.int8)
        return dict(c, args=(c["q"], c["n"], dv.digits_tensor(m, n_pad, dev), dv.digits_tensor(loc.T, n_pad, dev),
                             dv.strengths_tensor(a, c["precision"], dev), c["precision"]))
    if kind == "decode":
        asm, peel, keep = [], [], []
        q, n, b, C, R = (c[k] for k in ("q", "n", "b", "C", "R"))
        n_pad, Q, p1 = dv.n_pad_of(n), q ** b, n + 1
        for _ in range(c["count"]):
            loc, a, Ms, D = _instance(c, g)
            sd = _noise_sd(a, c["snr"])
            src = torch.from_numpy(_aliased(q, b, Ms, D, loc, a)).to(dev)
            U = torch.empty((C, Q, R * p1), dtype=torch.complex128, device=dev)
            asm.append(dict(Q=Q, C=C, R=R, p1=p1, src=src, src_rows=R * p1, gsel=list(range(C)), rsel=list(range(R)),
                            U=U, bin_major=True, sigma=sd / Q ** 0.5, seed=int(g.integers(0, 2 ** 62))))
            peel.append(dict(q=q, n=n, b=b, C=C, P=R * p1, p1=p1, method=L.QSFT_DETECT_NSO1,
                             cutoff=1e-9 + 1.5 * sd ** 2 / Q, Mt=dv.Mt_tensor(Ms, b, n_pad, dev),
                             D=dv.D_tensor([D] * C, n_pad, dev), U=U, shared_d=True))
            keep.append(src)
        return dict(c, asm=kernels.Assemble(asm), peel=kernels.PeelBatch(peel), keep=(keep, asm, peel))
    if kind == "transform":
        loc, a = _support(g, c["q"], c["n"], c["S"])
        channel = "nso" if c["method"] == "nso" else "identity"
        query_args = dict(query_method="complex", num_subsample=c["C"], b=c["b"], delays_method_source="identity",
                          delays_method_channel=channel, num_repeat=c["R"], subsampling_method="qsft")
        qsft = QSFT(num_subsample=c["C"], num_repeat=c["R"], b=c["b"], reconstruct_method_source="identity",
                    reconstruct_method_channel=channel)
        signal = dict(signal_w=dict(zip(map(tuple, loc.T), a)), locq=loc, strengths=a, n=c["n"], q=c["q"],
                      noise_sd=_noise_sd(a, c["snr"]), noise_mode="device", noise_seed=seed)
        return dict(c, signal=signal, query_args=query_args, qsft=qsft, seed=seed % 2 ** 32)
    specs = [_spec(*s, g) for s in _served_shapes(c)]
    return dict(c, specs=specs, server=Server(hbm_budget=HBM_BUDGET, max_batch=64, max_inflight=2))


def run(state):
    kind = state["kind"]
    if kind == "samples":
        return dv.evaluate_cosets(*state["args"])
    if kind == "subdft":
        return dv.subtransform(state["x"], state["q"], state["b"], in_stride=state["stride"],
                               precision=state["precision"])
    if kind == "heldout":
        return dv.evaluate_points(*state["args"])
    if kind == "decode":
        state["asm"].launch()
        state["peel"].run(fuse_from=3)
        rows = state["peel"].results(with_info=False)
        return [_table(k, values, state["S"]) for k, values, _, _ in rows]
    if kind == "transform":
        np.random.seed(state["seed"])                              # M, D and the group order, as a script seeds them
        signal = SyntheticSubsampledSignal(query_args=dict(state["query_args"]), **state["signal"])
        rep = state["qsft"].transform(signal, report=True, sort=True)
        keys = np.array(rep["locations"])
        return _table(keys, np.array([rep["gwht"][tuple(k)] for k in keys]), state["S"])
    server = state["server"]
    reqs = [server.submit(sp) for sp in state["specs"]]
    server.drain()
    server.completed.clear()                                       # delivered: a long-lived server does not keep them
    # The rows of every request. The engine samples in FP32, so its coefficients carry FP32 accuracy (two FP32
    # evaluators of the same samples differ by 7e-8 to 1.1e-7 in them); they are kept as complex64.
    rows = [(r.result.k, r.result.values.astype(np.complex64)) for r in reqs]
    if state["mix"] == "k1":                                       # 20 dB and above: every request recovers all S
        return rows
    return [_table(k, values, r.spec.S) for (k, values), r in zip(rows, reqs)]


# -------------------------------------------------------- work and exact values


def _sample_work(q, n, S, b, C, P, itemsize):
    """Samples of C x P cosets: inputs in, samples out. The q^b samples of a coset are the inverse q-ary transform of
    the S terms folded into its q^b bins: one complex multiply-add per term and 5 Q log2 Q operations."""
    Q = q ** b
    return {"bytes": C * P * Q * itemsize + S * (n + itemsize) + C * b * n + P * n,
            "flops": C * P * (8.0 * S + 5.0 * Q * math.log2(Q))}


def _pass_work(q, n, S, b, C, P, itemsize):
    """A whole transform: the samples written, read and transformed once, the support and its values out."""
    w = _sample_work(q, n, S, b, C, P, itemsize)
    Q = q ** b
    return {"bytes": w["bytes"] + C * P * Q * itemsize + S * (n + 16),
            "flops": w["flops"] + C * P * 5.0 * Q * math.log2(Q)}


def work(case):
    c = case
    kind = c["kind"]
    if kind == "samples":
        return _sample_work(c["q"], c["n"], c["S"], c["b"], c["C"], c["P"], 8 if c["precision"] == "fp32" else 16)
    if kind == "subdft":
        Q, size = c["q"] ** c["b"], 8 if c["precision"] == "fp32" else 16
        return {"bytes": 2 * c["rows"] * Q * size, "flops": c["rows"] * 5.0 * Q * math.log2(Q)}
    if kind == "heldout":
        return {"bytes": c["N"] * (c["n"] + 16) + c["S"] * (c["n"] + 16), "flops": 8.0 * c["N"] * c["S"]}
    if kind == "decode":
        cells = c["C"] * c["R"] * (c["n"] + 1) * c["q"] ** c["b"]
        return {"bytes": c["count"] * (16 * cells + c["S"] * (c["n"] + 16)), "flops": c["count"] * 8.0 * cells}
    if kind == "transform":
        return _pass_work(c["q"], c["n"], c["S"], c["b"], c["C"], c["R"] * (c["n"] + 1), 16)
    total = {"bytes": 0.0, "flops": 0.0}
    for q, n, S, b, _ in _served_shapes(c):
        w = _pass_work(q, n, S, b, 3, 2 * (n + 1), 8)
        total = {k: total[k] + w[k] for k in total}
    return total


def _phases(A, B, q):
    """(A @ B) mod q of integer digits, exact in float64, as int64."""
    return torch.remainder(A.double() @ B.double(), q).long()


def exact(case, seed):
    c, g = case, np.random.default_rng(seed)
    dev = torch.device("cuda")
    kind = c["kind"]
    if kind == "subdft":
        x = prepare(case, seed)["x"].to(torch.complex128)[:, ::c["stride"]]
        q, b, rows = c["q"], c["b"], c["rows"]
        r = torch.arange(q, device=dev, dtype=torch.float64)
        ang = -2 * math.pi * torch.remainder(r[:, None] * r[None, :], q) / q
        F = torch.complex(torch.cos(ang), torch.sin(ang))
        for t in range(b):                                         # one axis at a time
            x = torch.matmul(F, x.reshape(rows * q ** t, q, q ** (b - 1 - t)))
        return x.reshape(rows, q ** b) / q ** b
    if kind in ("samples", "heldout"):
        q = c["q"]
        ang = 2 * math.pi * torch.arange(q, device=dev, dtype=torch.float64) / q
        w = torch.complex(torch.cos(ang), torch.sin(ang))
    if kind == "heldout":
        loc, a = _support(g, q, c["n"], c["S"])
        m = torch.from_numpy(g.integers(0, q, size=(c["N"], c["n"]), dtype=np.int8)).to(dev)
        loc, a = torch.from_numpy(loc).to(dev), torch.from_numpy(a).to(dev)
        return torch.cat([w[_phases(part, loc, q)] @ a for part in m.split(20000)])
    if kind == "samples":
        loc, a, Ms, D = _instance(c, g)
        loc, a, D = torch.from_numpy(loc).to(dev), torch.from_numpy(a).to(dev), torch.from_numpy(D).to(dev)
        if c["precision"] == "fp32":
            a = a.to(torch.complex64).to(torch.complex128)         # the strengths that the call is given
        Q, b = q ** c["b"], c["b"]
        place = q ** torch.arange(b - 1, -1, -1, device=dev)
        lq = (torch.arange(Q, device=dev)[:, None] // place) % q   # (Q, b) digits of l, most significant first
        B = a * w[_phases(D, loc, q)]                              # (P, S)
        out = []
        for M in Ms:                                               # <M l + d, k> = <l, M^T k> + <d, k> (mod q)
            kM = _phases(torch.from_numpy(M.T.copy()).to(dev), loc, q)
            out.append(torch.cat([B @ w[_phases(part, kM, q)].T for part in lq.split(2048)], dim=1))
        return torch.stack(out)
    if kind == "transform" and c["snr"] is None:
        loc, a = _support(g, c["q"], c["n"], c["S"])               # noiseless: the planted spectrum, keys sorted
        return None, _table(loc.T, a[np.lexsort(loc[::-1])], c["S"])[1]
    return None                                                    # noisy decodes have no closed form
