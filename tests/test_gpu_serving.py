"""The serving loop on the GPU: the native batch runtime gives the engine's
rows; every request's result is the same alone and in the mix; admission by
HBM footprint rejects what can never fit and queues what does not fit yet."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from qsft_amd import _lib as L
    from qsft_amd import engine as E
    from qsft_amd import kernels as K
    from qsft_amd import serving as SV


def _rows(k, v):
    return [tuple(int(x) for x in r) for r in k], np.ascontiguousarray(v, dtype=np.complex128)


def _bits(v):
    return np.ascontiguousarray(v, dtype=np.complex128).view(np.float64)


def _k3_mix(count, rng, large=0.0):
    """K3 recipe: q in {2, 3, 4, 20}, n in [8, 64], S log-uniform in [10, 2000]
    (at most q^n / 8), b = ceil(log_q S) + 1, C = 3, NSO R = 2, SNR U[5, 30] dB;
    a `large` share of q = 4, n = 100, S = 5000, b = 7 jobs."""
    specs = []
    for _ in range(count):
        if rng.uniform() < large:
            specs.append(E.random_spec(4, 100, 5000, 7, 3, 2, float(rng.uniform(5, 30)), rng=rng))
            continue
        q = int(rng.choice([2, 3, 4, 20]))
        n = int(rng.integers(8, 65))
        S = int(np.exp(rng.uniform(np.log(10), np.log(2000))))
        S = max(2, min(S, q ** n // 8))
        b = int(np.ceil(np.log(S) / np.log(q))) + 1
        specs.append(E.random_spec(q, n, S, b, 3, 2, float(rng.uniform(5, 30)), rng=rng))
    return specs


def test_runtime_batch_equals_engine_batch():
    """One native-runtime batch (ordered pack) against the Python engine's
    batch on the same inputs and noise: the same rows, bits and order."""
    rng = np.random.default_rng(3)
    specs = [E.random_spec(4, 50, 1000, 6, 3, 2, snr, rng=rng) for snr in (3.0, 10.0, None)]
    specs += [E.random_spec(20, 16, 300, 3, 3, 2, 20.0, rng=rng), E.random_spec(3, 20, 90, 4, 3, 2, 15.0, rng=rng),
              E.random_spec(2, 70, 60, 7, 3, 2, 12.0, rng=rng),                      # P = 142
              E.random_spec(4, 12, 100, 4, 3, 1, None, rng=rng, method="identity")]
    print("runtime vs engine", flush=True)
    dev = torch.device("cuda", torch.cuda.current_device())
    sb = SV.ServedBatch(specs, dev)
    sb.launch(seed_offset=6)
    sb.wait()
    got = sb.results()
    ref = E.Batch(specs, precision="fp32")
    ref.launch(seed_offset=6)
    want = ref.results()
    for i, (g, (k, v, order, _)) in enumerate(zip(got, want)):
        kg, vg = _rows(g.k, g.values)
        kw, vw = _rows(k, v)
        assert kg == kw, i
        assert np.array_equal(_bits(vg), _bits(vw)), i
        assert np.array_equal(np.asarray(g.order), order), i
    # a relaunch with another seed offset draws fresh noise; the same offset repeats the bits
    sb.launch(seed_offset=7)
    sb.wait()
    again = sb.results()
    assert any(not np.array_equal(a.values, b.values) for a, b in zip(again[:2], got[:2]))
    sb.launch(seed_offset=6)
    sb.wait()
    for a, b in zip(sb.results(), got):
        assert np.array_equal(_bits(a.values), _bits(b.values))
    # the noiseless requests recover their planted spectrum
    for i in (2, 6):
        d = got[i].to_dict()
        truth = {tuple(int(x) for x in c): a for c, a in zip(specs[i].locq.T, specs[i].strengths)}
        assert set(d) == set(truth)
        assert max(abs(d[k] - truth[k]) / abs(truth[k]) for k in truth) < 1e-5


def test_each_result_is_the_same_alone_and_in_the_mix():
    """40 requests of the K3 mix plus one large job arrive together and are
    served in continuous batches (at most 16 per batch, two batches on the GPU
    at once). Each request's rows equal those of the request served alone
    (same noise seed): same keys in the same order, values within 1e-12."""
    rng = np.random.default_rng(44)
    specs = _k3_mix(40, rng) + [E.random_spec(4, 100, 5000, 7, 3, 2, 10.0, rng=rng)]
    print("served mix of", len(specs), flush=True)
    srv = SV.Server(hbm_budget=40 << 30, max_batch=16, max_inflight=2)
    reqs = [srv.submit(sp) for sp in specs]
    srv.drain()
    assert srv.batches >= 3
    dev = torch.device("cuda", torch.cuda.current_device())
    for i, (sp, r) in enumerate(zip(specs, reqs)):
        alone = SV.ServedBatch([sp], dev)
        alone.launch()
        alone.wait()
        a, = alone.results()
        kg, vg = _rows(r.result.k, r.result.values)
        ka, va = _rows(a.k, a.values)
        assert kg == ka, (i, sp.q, sp.n, sp.b, sp.S)
        assert np.all(np.abs(vg - va) <= 1e-12 * np.abs(va)), i
        alone.free()
    lat = SV.latency_summary(reqs)
    print(f"{srv.batches} batches, latency p50 {lat['p50_ms']:.2f} ms p99 {lat['p99_ms']:.2f} ms", flush=True)


def test_admission_rejects_oversize_and_queues_under_a_small_budget():
    rng = np.random.default_rng(45)
    small = [E.random_spec(4, 30, 200, 5, 3, 2, 15.0, rng=rng) for _ in range(9)]
    fp = SV.footprint(small[0])
    budget = int(2.5 * fp)                                   # two such requests at a time
    srv = SV.Server(hbm_budget=budget, max_batch=8, max_inflight=2)
    big = E.random_spec(4, 50, 1000, 6, 3, 2, 10.0, rng=rng)
    assert SV.footprint(big) > budget
    with pytest.raises(SV.AdmissionError):
        srv.submit(big)
    reqs = [srv.submit(sp) for sp in small]
    peak = 0
    while not srv.idle():
        srv.poll()
        peak = max(peak, srv.used)
        assert srv.used <= budget
    assert all(r.result is not None for r in reqs)
    assert srv.batches >= 5                                    # at most two requests per batch fit
    print(f"budget {budget} bytes, peak {peak}, {srv.batches} batches", flush=True)
    dev = torch.device("cuda", torch.cuda.current_device())
    for sp, r in zip(small, reqs):
        alone = SV.ServedBatch([sp], dev)
        alone.launch()
        alone.wait()
        a, = alone.results()
        assert _rows(r.result.k, r.result.values)[0] == _rows(a.k, a.values)[0]


def test_open_loop_poisson_arrivals_complete():
    """Poisson arrivals replayed against the clock: every request completes,
    latencies are measured from arrival, noiseless requests are exact."""
    rng = np.random.default_rng(46)
    specs = _k3_mix(60, rng)
    for sp in specs[:10]:
        sp.noise_sd = 0.0
    arrivals = np.cumsum(rng.exponential(1.0 / 2000.0, size=len(specs)))
    srv = SV.Server(hbm_budget=40 << 30, max_batch=32, max_inflight=2)
    reqs = srv.run_open_loop(arrivals, specs)
    assert len(reqs) == len(specs) and all(r.result is not None for r in reqs)
    assert all(r.t_done >= r.t_submit for r in reqs)
    for sp, r in zip(specs[:10], reqs[:10]):
        d = r.result.to_dict()
        truth = {tuple(int(x) for x in c): a for c, a in zip(sp.locq.T, sp.strengths)}
        assert set(d) <= set(truth)
        for k, v in d.items():
            assert abs(v - truth[k]) <= 1e-4 * abs(truth[k])
    lat = SV.latency_summary(reqs)
    print(f"open loop: {srv.batches} batches, p50 {lat['p50_ms']:.2f} ms p99 {lat['p99_ms']:.2f} ms", flush=True)


def _copy(results):
    return [(np.array(r.k), np.ascontiguousarray(r.values).copy(), np.array(r.order)) for r in results]


def test_graph_replay_matches_eager_launches():
    """The batch pipeline captured as a hipGraph (stage launches, fused
    peeling tail, finalize and ordered pack on the tail stream): replay k
    gives the bits of an eager launch with seed offset k, for three replays
    with eager work and synchronisations between them."""
    rng = np.random.default_rng(47)
    specs = _k3_mix(24, rng) + [E.random_spec(4, 50, 1000, 6, 3, 2, 10.0, rng=rng) for _ in range(2)]
    dev = torch.device("cuda", torch.cuda.current_device())
    s1, t1, s2, t2 = (torch.cuda.Stream(device=dev) for _ in range(4))
    g = SV.ServedBatch(specs, dev, stream=s1, tail_stream=t1)
    g.launch(seed_offset=0)
    g.wait()
    g.capture()
    eager = SV.ServedBatch(specs, dev, stream=s2, tail_stream=t2)
    for k in (1, 2, 3):
        print("replay", k, flush=True)
        g.replay()
        g.wait()
        got = _copy(g.results())
        eager.launch(seed_offset=k)
        eager.wait()
        want = _copy(eager.results())
        torch.ones(1 << 20, device=dev).sum().item()              # other eager work between replays
        for i, (a, b) in enumerate(zip(got, want)):
            assert np.array_equal(a[0], b[0]), (k, i)
            assert np.array_equal(a[1].view(np.float64), b[1].view(np.float64)), (k, i)
            assert np.array_equal(a[2], b[2]), (k, i)


def test_k3_256_uneven_instances_in_one_batch():
    """256 instances of the K3 mix in one set of launches (one launch per
    stage and kernel variant): every instance gives the rows it gives alone,
    and noiseless copies of 32 of the shapes recover only true keys with
    their exact values, and 95 % of all planted keys."""
    rng = np.random.default_rng(48)
    specs = _k3_mix(256, rng)
    print("K3 x256:", sorted({(s.q, s.b) for s in specs}), flush=True)
    dev = torch.device("cuda", torch.cuda.current_device())
    mix = SV.ServedBatch(specs, dev)
    mix.launch(seed_offset=9)
    mix.wait()
    got = _copy(mix.results())
    for i, sp in enumerate(specs):
        alone = SV.ServedBatch([sp], dev)
        alone.launch(seed_offset=9)
        alone.wait()
        (k, v, o), = _copy(alone.results())
        assert np.array_equal(got[i][0], k), (i, sp.q, sp.n, sp.b, sp.S)
        assert np.all(np.abs(got[i][1] - v) <= 1e-12 * np.abs(v)), i
        alone.free()
    clean = [E.TransformSpec(**{**{k: v for k, v in s.__dict__.items() if not k.startswith("_")}, "noise_sd": 0.0})
             for s in specs[:32]]
    bt = SV.ServedBatch(clean, dev)
    bt.launch()
    bt.wait()
    found = planted = 0
    for r, sp in zip(bt.results(), clean):
        truth = {tuple(int(x) for x in c): a for c, a in zip(sp.locq.T, sp.strengths)}
        for key, val in r.to_dict().items():
            assert key in truth, (sp.q, sp.n, sp.S, sp.b)
            assert abs(val - truth[key]) <= 1e-4 * abs(truth[key])
        found += len(r.k)
        planted += sp.S
    print(f"noiseless K3 copies: {found} of {planted} keys", flush=True)
    assert found >= 0.95 * planted


def test_tune_leaves_shapes_with_whole_rows_alone():
    """The evaluation transforms whole rows of up to 144 KiB itself: there is nothing to measure for them."""
    print("tune whole rows", flush=True)
    rng = np.random.default_rng(8)
    specs = [E.random_spec(5, 12, 20, 5, 1, 1, 20.0, rng=rng), E.random_spec(4, 12, 20, 5, 1, 1, 20.0, rng=rng),
             E.random_spec(3, 12, 20, 10, 1, 1, 20.0, rng=rng)]
    SV.Server(hbm_budget=1 << 40).tune(specs)
    assert [K.dft_schedule(sp.q, sp.b, L.QSFT_F32)[1] for sp in specs] == [False, False, True]


def test_a_request_of_many_supports_equals_the_engine():
    """More than 8192 supports (ranked in two steps) beside few, in the native runtime and in the engine: the same rows."""
    print("runtime vs engine, many supports", flush=True)
    rng = np.random.default_rng(13)
    specs = [E.random_spec(4, 40, 8300, 7, 2, 1, None, rng=rng, method="identity"),
             E.random_spec(4, 12, 100, 4, 3, 1, None, rng=rng, method="identity")]
    sb = SV.ServedBatch(specs, torch.device("cuda", torch.cuda.current_device()))
    sb.launch(seed_offset=0)
    sb.wait()
    ref = E.Batch(specs, precision="fp32")
    ref.launch(seed_offset=0)
    for g, (k, v, order, _) in zip(sb.results(), ref.results()):
        assert len(k) > 0 and _rows(g.k, g.values)[0] == _rows(k, v)[0]
        assert np.array_equal(_bits(g.values), _bits(v)) and np.array_equal(np.asarray(g.order), order)
