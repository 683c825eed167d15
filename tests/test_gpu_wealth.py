"""GPU parity: wealth-exchange program against the oracle.

Integer wealth, the Gini/mean records and the float32 positions are
bit-exact (normal()'s erf_inv calls the shared abm_math.h log1p on both
sides)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

MODES = [O.MODE_ORIGINAL, O.MODE_PARTITIONABLE]


@pytest.fixture(scope="module")
def wealth():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from jaxabm_amd.programs import wealth

    return wealth


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n,steps,seed", [(1000, 100, 0), (2, 10, 1), (3000, 20, 5), (1025, 7, 9),
                                          (1023, 12, 4)])
def test_wealth_matches_oracle(wealth, mode, n, steps, seed):
    eng = wealth.WealthEngine(n, seed=seed, mode=mode)
    x, y, w, rng = O.wealth_init(n, seed, mode)
    np.testing.assert_array_equal(eng.x.cpu().numpy(), x)
    np.testing.assert_array_equal(eng.w.cpu().numpy(), w)
    mean, gini = eng.run(steps)
    om, og = O.wealth_run(x, y, w, rng, steps, mode)
    np.testing.assert_array_equal(eng.w.cpu().numpy(), w)
    np.testing.assert_array_equal(mean, om)
    np.testing.assert_array_equal(gini, og)
    np.testing.assert_array_equal(eng.rng, rng)
    np.testing.assert_array_equal(eng.x.cpu().numpy(), x)
    np.testing.assert_array_equal(eng.y.cpu().numpy(), y)


def test_wealth_batch_equals_alone(wealth):
    """A batched launch gives each instance exactly its solo results."""
    sizes, seeds, steps = [1000, 5000, 37, 2048], [0, 1, 2, 3], [30, 12, 50, 25]
    solo = [wealth.WealthEngine(n, seed=s).run(k) for n, s, k in zip(sizes, seeds, steps)]
    engines = [wealth.WealthEngine(n, seed=s) for n, s in zip(sizes, seeds)]
    mixed = wealth.run_batch(engines, steps)
    for (m1, g1), (m2, g2) in zip(solo, mixed):
        np.testing.assert_array_equal(m1, m2)
        np.testing.assert_array_equal(g1, g2)


def _run_raw(wealth, eng, steps, max_n, draws=False):
    """One instance through abm_wealth_run_batch with an explicit max_n, with
    or without the precomputed-draw buffer."""
    import torch
    from jaxabm_amd._lib import check, lib, ptr, stream_handle

    keys = eng.key_table(steps)
    mean = torch.empty(steps, dtype=torch.float32, device=eng.device)
    gini = torch.empty(steps, dtype=torch.float32, device=eng.device)
    buf = eng.draw_buffer(steps) if draws else None
    desc = torch.from_numpy(eng.descriptor(keys, steps, mean, gini, buf).view(np.uint8)).to(eng.device)
    check(lib().abm_wealth_run_batch(ptr(desc), 1, max_n, eng.mode, stream_handle()), "run")
    return mean.cpu().numpy(), gini.cpu().numpy()


@pytest.mark.parametrize("draws", [False, True])
@pytest.mark.parametrize("n,max_n", [(1000, 0), (1000, 500), (5000, 8000), (8000, 8000),
                                     (300, 100)])
def test_wealth_lds_and_global_paths_agree(wealth, n, max_n, draws):
    """Every path gives identical records and state: draws computed in the
    run or grid-wide before it; with a draw buffer, the exchange apart from walk
    and records, or the whole instance in one workgroup above the table's limit;
    LDS-resident runs (n <= max_n <= 8000) and global-buffer runs (max_n = 0,
    or an instance above max_n)."""
    steps = 40
    a = wealth.WealthEngine(n, seed=3)
    b = wealth.WealthEngine(n, seed=3)
    ma, ga = a.run(steps)                     # precomputed draws, max_n = n
    mb, gb = _run_raw(wealth, b, steps, max_n, draws)
    np.testing.assert_array_equal(ma, mb)
    np.testing.assert_array_equal(ga, gb)
    for t in ("w", "x", "y"):
        np.testing.assert_array_equal(getattr(a, t).cpu().numpy(), getattr(b, t).cpu().numpy())


def test_wealth_global_path_matches_oracle(wealth):
    """An instance above the LDS capacity, without a draw buffer, runs on its
    global buffers."""
    n, steps = 9000, 8
    eng = wealth.WealthEngine(n, seed=11)
    x, y, w, rng = O.wealth_init(n, 11, eng.mode)
    mean, gini = _run_raw(wealth, eng, steps, n)
    om, og = O.wealth_run(x, y, w, rng, steps, eng.mode)
    np.testing.assert_array_equal(eng.w.cpu().numpy(), w)
    np.testing.assert_array_equal(mean, om)
    np.testing.assert_array_equal(gini, og)


@pytest.mark.parametrize("n,steps,seed", [(8001, 30, 1), (50_000, 40, 2), (300_000, 12, 3)])
def test_grid_path_matches_oracle_and_one_workgroup_run(wealth, monkeypatch, n, steps, seed):
    """WealthEngine.run with each step spread over the GPU (abm_wealth_run_grid),
    from the smallest size that may take it: the oracle's records and state, and
    the same bits as the one-workgroup run of the batch entry point."""
    import os

    monkeypatch.setattr(wealth, "EXCHANGE_MAX_AGENTS", wealth.GRID_MIN_AGENTS)
    eng = wealth.WealthEngine(n, seed=seed)
    assert n > wealth.GRID_MIN_AGENTS
    mean, gini = eng.run(steps)
    x, y, w, rng = O.wealth_init(n, seed, O.MODE_PARTITIONABLE)
    om, og = O.wealth_run_threads(x, y, w, rng, steps, max(1, min(16, os.cpu_count() or 1)),
                                  O.MODE_PARTITIONABLE)
    np.testing.assert_array_equal(mean, om)
    np.testing.assert_array_equal(gini, og)
    np.testing.assert_array_equal(eng.w.cpu().numpy(), w)
    np.testing.assert_array_equal(eng.x.cpu().numpy(), x)
    np.testing.assert_array_equal(eng.y.cpu().numpy(), y)
    one = wealth.WealthEngine(n, seed=seed)
    m2, g2 = _run_raw(wealth, one, steps, 0, draws=True)
    np.testing.assert_array_equal(m2, mean)
    np.testing.assert_array_equal(g2, gini)


def test_grid_path_wealth_above_the_lds_bins(wealth, monkeypatch):
    """A state where one agent holds 5,000 units (total wealth 15,000 <= n,
    the histogram's range): wealth values past the grid path's per-workgroup
    LDS bins go to the global histogram directly; the records and state equal
    the oracle's from the same state."""
    import os

    import torch

    n, steps, seed = 20_000, 25, 5
    monkeypatch.setattr(wealth, "EXCHANGE_MAX_AGENTS", wealth.GRID_MIN_AGENTS)
    eng = wealth.WealthEngine(n, seed=seed)
    x, y, w, rng = O.wealth_init(n, seed, O.MODE_PARTITIONABLE)
    w[:] = 0
    w[20:10020] = 1
    w[7] = 5000
    eng.w.copy_(torch.from_numpy(w.copy()).to(eng.w.device))
    mean, gini = eng.run(steps)
    om, og = O.wealth_run_threads(x, y, w, rng, steps, max(1, min(16, os.cpu_count() or 1)),
                                  O.MODE_PARTITIONABLE)
    assert w.max() > 1024
    np.testing.assert_array_equal(mean, om)
    np.testing.assert_array_equal(gini, og)
    np.testing.assert_array_equal(eng.w.cpu().numpy(), w)


# one agent more or less than a thread's share, the widest 32-bit and the
# packed increment arrays, the largest instance the exchange kernel takes;
# step counts around the load-ahead distances and the 256 record workgroups
@pytest.mark.parametrize("n,steps", [(2, 1), (63, 2), (64, 7), (65, 8), (1023, 9), (1024, 17),
                                     (1025, 300), (2049, 3), (6145, 5), (10241, 4), (20480, 6),
                                     (20481, 6), (39999, 3), (40000, 4), (40001, 2)])
def test_exchange_run_matches_oracle_at_its_edges(wealth, n, steps):
    import os

    for mode in (O.MODE_PARTITIONABLE, O.MODE_ORIGINAL):
        eng = wealth.WealthEngine(n, seed=n, mode=mode)
        mean, gini = _run_raw(wealth, eng, steps, n, draws=True)
        x, y, w, rng = O.wealth_init(n, n, mode)
        om, og = O.wealth_run_threads(x, y, w, rng, steps,
                                      max(1, min(16, os.cpu_count() or 1)), mode)
        np.testing.assert_array_equal(mean, om)
        np.testing.assert_array_equal(gini, og)
        np.testing.assert_array_equal(eng.w.cpu().numpy(), w)
        np.testing.assert_array_equal(eng.x.cpu().numpy(), x)
        np.testing.assert_array_equal(eng.y.cpu().numpy(), y)


def test_batch_of_split_and_whole_runs(wealth):
    """One table with instances of uneven sizes, with and without a draw
    buffer, and steps 0: each as its own run."""
    import torch

    from jaxabm_amd._lib import check, lib, ptr, stream_handle

    sizes = [(3000, 12, True), (900, 30, False), (1, 0, None), (40, 5, True), (2999, 12, False)]
    sizes = [(max(n, 2), s, d) for n, s, d in sizes]
    engs = [wealth.WealthEngine(n, seed=i) for i, (n, _, _) in enumerate(sizes)]
    keep, descs, outs = [], [], []
    for e, (n, s, d) in zip(engs, sizes):
        keys = e.key_table(s)
        mean = torch.empty(max(s, 1), dtype=torch.float32, device=e.device)
        gini = torch.empty(max(s, 1), dtype=torch.float32, device=e.device)
        buf = e.draw_buffer(s) if d or d is None else None
        keep += [keys, buf]
        descs.append(e.descriptor(keys, s, mean, gini, buf))
        outs.append((mean, gini))
    table = torch.from_numpy(np.concatenate(descs).view(np.uint8)).cuda()
    check(lib().abm_wealth_run_batch(ptr(table), len(engs), 3000, engs[0].mode, stream_handle()),
          "run")
    for i, (e, (n, s, _), (mean, gini)) in enumerate(zip(engs, sizes, outs)):
        x, y, w, rng = O.wealth_init(n, i, e.mode)
        om, og = O.wealth_run(x, y, w, rng, s, e.mode)
        np.testing.assert_array_equal(mean.cpu().numpy()[:s], om[:s])
        np.testing.assert_array_equal(gini.cpu().numpy()[:s], og[:s])
        for a, b in ((e.w, w), (e.x, x), (e.y, y)):
            np.testing.assert_array_equal(a.cpu().numpy(), b)


def _run_grid(eng, steps, scratch):
    import torch

    from jaxabm_amd._lib import WEALTH_GRID_ACC_WORDS, check, lib, ptr, stream_handle

    keys = eng.key_table(steps)
    mean = torch.empty(steps, dtype=torch.float32, device=eng.device)
    gini = torch.empty(steps, dtype=torch.float32, device=eng.device)
    acc = torch.empty(WEALTH_GRID_ACC_WORDS, dtype=torch.int32, device=eng.device)
    buf = eng.draw_buffer(1).fill_(-1) if scratch else None
    host = eng.descriptor(keys, steps, mean, gini, buf)
    check(lib().abm_wealth_run_grid(host.ctypes.data, ptr(acc), eng.mode, stream_handle()), "run")
    return mean.cpu().numpy(), gini.cpu().numpy()


# below, at and above the smallest instance that takes one launch per step, one
# and two tiles of agents a workgroup; wealth above the LDS bins
@pytest.mark.parametrize("n,steps,rich", [(1032, 5, 0), (1033, 6, 0), (1280, 1, 0), (20_000, 25, 5000),
                                          (2 * 256 * 4096 + 3, 3, 0)])
@pytest.mark.parametrize("scratch", [False, True])
def test_grid_run_one_and_two_launches_match_oracle(wealth, n, steps, rich, scratch):
    import os

    import torch

    for mode in (O.MODE_PARTITIONABLE, O.MODE_ORIGINAL):
        eng = wealth.WealthEngine(n, seed=9, mode=mode)
        x, y, w, rng = O.wealth_init(n, 9, mode)
        if rich:
            w[:] = 0
            w[20:10020] = 1
            w[7] = rich
            eng.w.copy_(torch.from_numpy(w.copy()).to(eng.w.device))
        mean, gini = _run_grid(eng, steps, scratch)
        om, og = O.wealth_run_threads(x, y, w, rng, steps,
                                      max(1, min(16, os.cpu_count() or 1)), mode)
        assert not rich or w.max() > 1024
        np.testing.assert_array_equal(mean, om)
        np.testing.assert_array_equal(gini, og)
        for a, b in ((eng.w, w), (eng.x, x), (eng.y, y)):
            np.testing.assert_array_equal(a.cpu().numpy(), b)
        assert not eng.inc.any() and not eng.hist.any()   # left zero for the next run


def test_engine_routes_give_the_same_bits(wealth, monkeypatch):
    """The exchange run and the run over the whole GPU of one engine size."""
    n, steps = 12_001, 9
    a, b = wealth.WealthEngine(n, seed=4), wealth.WealthEngine(n, seed=4)
    ra = a.run(steps)
    monkeypatch.setattr(wealth, "DRAW_BUFFER_MAX_BYTES", 12 * n * steps - 1)
    rb = b.run(steps)
    for u, v in zip(ra, rb):
        np.testing.assert_array_equal(u, v)
    for t in ("w", "x", "y"):
        np.testing.assert_array_equal(getattr(a, t).cpu().numpy(), getattr(b, t).cpu().numpy())


@pytest.mark.parametrize("n,max_n", [(37, 0), (1000, 1000), (3000, 3000), (40_000, 40_000)])
def test_batch_instance_of_no_steps(wealth, n, max_n):
    """An instance of 0 steps has no row of draws: its buffer, here the end of a
    live one, is not read, and its state and the other instance are untouched."""
    import torch

    from jaxabm_amd._lib import check, lib, ptr, stream_handle

    idle, a, b = (wealth.WealthEngine(m, seed=6) for m in (n, 50, 50))
    want = b.run(4)
    keys, rec, draws = a.key_table(4), torch.empty(2, 4, device="cuda"), a.draw_buffer(4)
    d0 = idle.descriptor(keys, 0, rec[0], rec[1], draws)
    d0["draws"] = draws.data_ptr() + 4 * draws.numel()
    before = [getattr(idle, t).clone() for t in ("x", "y", "w")]
    table = torch.from_numpy(np.concatenate(
        [d0, a.descriptor(keys, 4, rec[0], rec[1], draws)]).view(np.uint8)).to("cuda")
    check(lib().abm_wealth_run_batch(ptr(table), 2, max_n, a.mode, stream_handle()), "run")
    for t, was in zip(("x", "y", "w"), before):
        assert torch.equal(getattr(idle, t), was)
    for got, w in zip(rec.cpu().numpy(), want):
        np.testing.assert_array_equal(got, w)


def test_batch_of_more_instances_than_a_grid_has_rows(wealth):
    """65,537 instances of one seed: each one's records and state are the
    engine's."""
    import torch

    from jaxabm_amd._lib import WEALTH_INST, check, lib, ptr, stream_handle

    B, n, steps = 65_537, 5, 3
    eng = wealth.WealthEngine(n, seed=8)
    x, y, w = (t.repeat(B) for t in (eng.x, eng.y, eng.w))
    inc = torch.zeros(B * n, dtype=torch.int32, device="cuda")
    hist = torch.zeros(B * (n + 1), dtype=torch.int32, device="cuda")
    keys = eng.key_table(steps)
    rec = torch.empty(2, B * steps, device="cuda")
    draws = torch.empty(B * steps * 3 * n, dtype=torch.int32, device="cuda")
    d, k = np.zeros(B, WEALTH_INST), np.arange(B, dtype=np.uint64)
    d["n"], d["steps"], d["keys"] = n, steps, keys.data_ptr()
    for name, t, each in (("x", x, n), ("y", y, n), ("w", w, n), ("inc", inc, n),
                          ("hist", hist, n + 1), ("mean_out", rec[0], steps),
                          ("gini_out", rec[1], steps), ("draws", draws, steps * 3 * n)):
        d[name] = t.data_ptr() + 4 * each * k
    table = torch.from_numpy(d.view(np.uint8)).to("cuda")
    check(lib().abm_wealth_run_batch(ptr(table), B, n, eng.mode, stream_handle()), "run")
    eng.rng = wealth.WealthEngine(n, seed=8).rng   # key_table moved it on
    mean, gini = eng.run(steps)
    for got, want in ((rec[0], mean), (rec[1], gini)):
        assert torch.equal(got.view(B, steps), torch.from_numpy(want.copy()).cuda().expand(B, steps))
    for got, want in ((x, eng.x), (y, eng.y), (w, eng.w)):
        assert torch.equal(got.view(B, n), want.expand(B, n))


def test_records_of_a_large_batch_match_oracle(wealth):
    """Instances around the sizes that a wavefront records alone (64 and 512
    values a round of loads, 1,024 agents at most), so many that a workgroup and
    its wavefronts take several steps each."""
    sizes, steps = [2, 63, 64, 65, 511, 512, 513, 1023, 1024, 1025], 130
    engines = [wealth.WealthEngine(n, seed=n) for _ in range(60) for n in sizes]
    records = wealth.run_batch(engines, [steps] * len(engines))
    for k, n in enumerate(sizes):
        x, y, w, rng = O.wealth_init(n, n, engines[0].mode)
        om, og = O.wealth_run(x, y, w, rng, steps, engines[0].mode)
        for e, (mean, gini) in list(zip(engines, records))[k::len(sizes)]:
            np.testing.assert_array_equal(mean, om)
            np.testing.assert_array_equal(gini, og)
            np.testing.assert_array_equal(e.w.cpu().numpy(), w)


@pytest.mark.parametrize("n", [32_768, 32_769])
def test_engine_on_both_sides_of_the_exchange_limit(wealth, n):
    """The largest engine that runs its exchange in one workgroup (32 agents a
    thread), and the first that spreads its steps over the GPU."""
    eng = wealth.WealthEngine(n, seed=5)
    assert (n > wealth.EXCHANGE_MAX_AGENTS) == (n == 32_769)
    mean, gini = eng.run(7)
    x, y, w, rng = O.wealth_init(n, 5, eng.mode)
    om, og = O.wealth_run(x, y, w, rng, 7, eng.mode)
    np.testing.assert_array_equal(mean, om)
    np.testing.assert_array_equal(gini, og)
    for a, b in ((eng.w, w), (eng.x, x), (eng.y, y)):
        np.testing.assert_array_equal(a.cpu().numpy(), b)
