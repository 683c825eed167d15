"""GPU parity: network SIR program against the oracle, bit-exact."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

MODES = [O.MODE_ORIGINAL, O.MODE_PARTITIONABLE]


@pytest.fixture(scope="module")
def sir():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from jaxabm_amd.programs import sir

    return sir


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n,m,steps,beta,gamma,seed", [
    (2000, 4, 60, 0.05, 0.1, 0),
    (5000, 2, 40, 0.3, 0.05, 3),
    (3000, 80, 25, 0.02, 0.2, 1),   # dense rows: every row is heavy
    (1000, 4, 30, 0.0, 0.1, 2),     # beta = 0: no new infection
    (1000, 4, 30, 1.0, 0.0, 2),     # beta = 1, gamma = 0
    (2000, 3, 300, 0.02, 0.01, 5),  # > 256 steps: risk marks wrap around
])
def test_sir_matches_oracle(sir, mode, n, m, steps, beta, gamma, seed):
    row_ptr, col = O.ba_csr(n, m, graph_seed=seed + 100)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), beta=beta, gamma=gamma,
                               n_seed_infected=10, seed=seed, mode=mode)
    st, rng = O.sir_init(n, 10, seed, mode)
    np.testing.assert_array_equal(eng.state_host(), st)
    np.testing.assert_array_equal(eng.rng, rng)
    want = O.sir_run(row_ptr, col, st, rng, beta, gamma, steps, mode)
    got = eng.run(steps)
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(eng.state_host(), st)
    np.testing.assert_array_equal(eng.rng, rng)
    assert (got.sum(axis=1) == n).all()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n,m,steps,beta,gamma,seed", [
    # chunks of 8192 agents (the maximum tile): tiles with many rows to scan
    # take the CSR sweep (one and two rounds), tiles of more than 65535 CSR
    # entries take worklists with row_ptr from global memory, and worklist
    # overflow in those makes each thread scan its own rows
    (100_000, 4, 40, 0.3, 0.1, 11),
    (40_000, 2, 40, 0.5, 0.05, 12),
    (20_000, 4, 60, 0.1, 0.1, 14),
    (3000, 80, 20, 0.02, 0.2, 13),   # one tile of 467k entries, all rows heavy
])
def test_sir_tile_paths_match_oracle(sir, mode, n, m, steps, beta, gamma, seed):
    row_ptr, col = O.ba_csr(n, m, graph_seed=seed + 100)
    n0 = max(10, n // 50)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), beta=beta, gamma=gamma,
                               n_seed_infected=n0, seed=seed, mode=mode, chunk_cost=1 << 40)
    assert eng.n_chunks == -(-n // 8192)
    st, rng = O.sir_init(n, n0, seed, mode)
    want = O.sir_run(row_ptr, col, st, rng, beta, gamma, steps, mode)
    got = eng.run(steps)
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(eng.state_host(), st)
    assert want[:, 1].max() > n // 4   # the epidemic reaches most tiles


@pytest.mark.parametrize("mode", MODES)
def test_sir_two_runs_continue(sir, mode):
    """A second run() continues from the current state (jaxabm/model.py:227-235)."""
    n = 3000
    row_ptr, col = O.ba_csr(n, 4, graph_seed=9)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), n_seed_infected=20, seed=4, mode=mode)
    st, rng = O.sir_init(n, 20, 4, mode)
    a = eng.run(13)
    b = eng.run(17)
    want = O.sir_run(row_ptr, col, st, rng, 0.05, 0.1, 30, mode)
    np.testing.assert_array_equal(np.concatenate([a, b]), want)


@pytest.mark.parametrize("mode", MODES)
def test_sir_full_size_matches_oracle(sir, mode):
    """The measured workload itself -- 1M-agent BA(m=4), 365 steps, 100 seed
    infections -- bit for bit against the oracle (its OpenMP path over the
    agents of each step, the same results as its serial path): every step's
    S/I/R counts and the final state; plus the invariants S + I + R = N, S
    never grows, R never shrinks."""
    import json
    import os

    from jaxabm_amd import network as N

    n, m = 1_000_000, 4
    # the graph the bench measures: the product's builder, checksummed
    row_ptr, col = N.ba_csr(n, m, graph_seed=0)
    gold = json.load(open(os.path.join(os.path.dirname(__file__), "golden",
                                       "sir_ba1M_m4_365steps.json")))
    assert N.csr_checksum(row_ptr, col) == gold["csr_sha256"]
    orp, ocol = O.ba_csr(n, m, graph_seed=0)
    np.testing.assert_array_equal(row_ptr, orp)
    np.testing.assert_array_equal(col, ocol)
    assert row_ptr[-1] == 2 * m * (n - m)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), seed=0, mode=mode)
    st, rng = O.sir_init(n, 100, 0, mode)
    threads = max(1, min(16, os.cpu_count() or 1))
    want = O.sir_run_threads(orp, ocol, st, rng, 0.05, 0.1, 365, threads, mode)
    got = np.concatenate([eng.run(12), eng.run(365 - 12)])   # a run continues the state
    np.testing.assert_array_equal(got, want)
    name = "partitionable" if mode == O.MODE_PARTITIONABLE else "original"
    np.testing.assert_array_equal(got, np.array(gold["counts"][name], np.int32))
    np.testing.assert_array_equal(eng.state_host(), st)
    assert (got.sum(axis=1) == n).all()
    assert (np.diff(got[:, 0]) <= 0).all()   # S never grows
    assert (np.diff(got[:, 2]) >= 0).all()   # R never shrinks
    assert got[-1, 1] == 0 and got[-1, 2] > n // 2


def test_seed_refuses_bad_chunk_tables(sir):
    """abm_sir_seed validates the chunk table the step kernel assumes (0 to
    n, ascending, 64-aligned inner boundaries, at most one tile per chunk)
    before launching anything."""
    import ctypes as C

    import torch

    from jaxabm_amd._lib import AbmError, SirGraph, check, lib, ptr, stream_handle

    n = 1000
    row_ptr, col = O.ba_csr(n, 4, graph_seed=2)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), n_seed_infected=5, seed=0)
    perm = torch.arange(n, dtype=torch.int32, device="cuda")
    for bad in ([0, 500, 1000], [0, 512, 999], [0, 1000, 512], [64, 1000]):
        cp = torch.tensor(bad, dtype=torch.int32, device="cuda")
        g = SirGraph(n, eng.graph.nnz, eng.graph.row_ptr.data_ptr(), eng.graph.col.data_ptr(),
                     cp.data_ptr(), len(bad) - 1)
        rc = lib().abm_sir_seed(C.byref(g), ptr(perm), 5, ptr(eng.state), ptr(eng.mark),
                                ptr(eng.bitmaps), 0, stream_handle())
        with pytest.raises(AbmError, match="chunk_ptr"):
            check(rc, "abm_sir_seed")


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("steps", [1, 31, 32, 33, 47, 48, 49, 130])
@pytest.mark.parametrize("n0,gamma", [(0, 0.5), (30, 0.5), (30, 0.02)])
def test_settling_run_equals_oracle_and_continues(sir, mode, steps, n0, gamma):
    """A run that stops launching once nobody is infected: the oracle's counts,
    state and key, also when another run continues it; one that stays infected
    launches every step."""
    n, beta = 1500, 0.01
    row_ptr, col = O.ba_csr(n, 3, graph_seed=4)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), beta=beta, gamma=gamma,
                               n_seed_infected=n0, seed=8, mode=mode)
    st, rng = O.sir_init(n, n0, 8, mode)
    for part in (steps, 40):
        want = O.sir_run(row_ptr, col, st, rng, beta, gamma, part, mode)
        got = eng.run(part)
        np.testing.assert_array_equal(got, want)
        np.testing.assert_array_equal(eng.state_host(), st)
        np.testing.assert_array_equal(eng.rng, rng)
        dead = np.flatnonzero(want[:, 1] == 0)
        if len(dead):   # launched up to two groups of 8 past the first that found none
            assert min(part, dead[0] + 1) <= eng.steps_launched <= min(part, dead[0] + 2 + 16)
        else:
            assert eng.steps_launched == part


def test_rows_at_the_end_of_the_entry_array(sir):
    """Rows of every length up to the wide loads' eight entries as the last
    rows of the array, where a wide load would pass its end."""
    for tail in range(1, 10):
        n = 200 + tail
        rng = np.random.default_rng(tail)
        # node n - 1 has `tail` neighbours; the others form a ring
        src = np.r_[np.arange(n - 1), np.full(tail, n - 1)]
        dst = np.r_[(np.arange(n - 1) + 1) % (n - 1), rng.choice(n - 1, tail, replace=False)]
        from jaxabm_amd.network import csr_undirected

        row_ptr, col = csr_undirected(n, src.astype(np.int32), dst.astype(np.int32))
        assert row_ptr[n] - row_ptr[n - 1] == tail
        eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), beta=0.6, gamma=0.1,
                                   n_seed_infected=60, seed=tail)
        st, key = O.sir_init(n, 60, tail, O.MODE_PARTITIONABLE)
        want = O.sir_run(row_ptr, col, st, key, 0.6, 0.1, 20, O.MODE_PARTITIONABLE)
        np.testing.assert_array_equal(eng.run(20), want)
        np.testing.assert_array_equal(eng.state_host(), st)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("chunk_cost", [1, 3000, 1 << 40])
def test_heavy_row_units_and_light_groups(sir, mode, chunk_cost):
    """150 hubs (more than one batch of 64) of degrees around multiples of 64
    beside light rows whose number at risk passes the group limits: tiles of 64
    agents up to one tile of all, equal to the oracle at every step."""
    n, steps, n0 = 6000, 60, 3
    rs = np.random.default_rng(11)
    adj = [set() for _ in range(n)]
    degrees = [33, 63, 64, 65, 127, 128, 129, 192, 600]
    for h in range(150):
        for u in rs.choice(np.arange(150, n), degrees[h % len(degrees)], replace=False):
            adj[h].add(int(u))
            adj[int(u)].add(h)
    for v in range(150, n - 1):   # a path: nobody is out of reach
        adj[v].add(v + 1)
        adj[v + 1].add(v)
    row_ptr = np.concatenate([[0], np.cumsum([len(a) for a in adj])]).astype(np.int32)
    col = np.concatenate([np.sort(np.fromiter(a, np.int32)) for a in adj]).astype(np.int32)
    eng = sir.SIRNetworkEngine(n, csr=(row_ptr, col), beta=0.03, gamma=0.05, n_seed_infected=n0,
                               seed=6, mode=mode, chunk_cost=chunk_cost)
    st, rng = O.sir_init(n, n0, 6, mode)
    want = O.sir_run(row_ptr, col, st, rng, 0.03, 0.05, steps, mode)
    np.testing.assert_array_equal(eng.run(steps), want)
    np.testing.assert_array_equal(eng.state_host(), st)
    assert want[:, 1].max() > n // 4
