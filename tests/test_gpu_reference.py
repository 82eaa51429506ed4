"""GPU parity of the reference-semantics annealer and the FP64 energy kernel.

The GPU chain draws from the same Philox counters as the oracle, so its
trajectories are compared with or_anneal_fields state for state; the law of
the chain is compared with the literal restatement of sa::anneal on
independent streams (hit rate against the exhaustive ground state).
"""
import json
import os
import subprocess

import numpy as np
import pytest

import onesolver_amd
import oracle
from conftest import GOLDEN
from qubo_io import load_qubo

pytestmark = pytest.mark.gpu


def _kats():
    with open(os.path.join(GOLDEN, "kat", "expected.json")) as f:
        return [(os.path.join(GOLDEN, "kat", e["file"]), e["energy"]) for e in json.load(f)]


@pytest.mark.parametrize("n,count", [(1, 3), (5, 10), (28, 1000), (100, 300), (1000, 70)])
def test_energy_fp64_matches_oracle(ctx, n, count):
    rng = np.random.default_rng(n)
    q = rng.uniform(-1, 1, (n, n))
    q = (q + q.T) / 2
    st = rng.integers(0, 2, (count, n)).astype(np.uint8)
    got = ctx.energy_fp64(q, st)
    ref = oracle.energy(q, st)
    scale = np.abs(q).sum() + 1.0
    assert np.all(np.abs(got - ref) <= 1e-12 * scale)


@pytest.mark.parametrize("n,counts", [(1, (1, 65)), (8, (64, 70000)), (57, (257,)),
                                      (64, (65600,)), (65, (1, 15, 16, 17, 8193)),
                                      (66, (31, 33)), (67, (32,)), (68, (16,)), (95, (8, 8192)),
                                      (96, (17,)), (97, (16,)), (127, (33,)), (128, (8200,)),
                                      (129, (4097,)), (161, (40,)), (260, (2753,))])
def test_energy_tiles_match_oracle(ctx, n, counts):
    """Edges of the energy kernels' tiles (states by 16 and 32, columns by 16
    and 128, the last 4 and 32 of k) and of their choice.  Whole numbers below
    2^20: every partial sum is exact, so the energies are equal."""
    rng = np.random.default_rng(n)
    q = np.triu(rng.integers(-(1 << 20), 1 << 20, (n, n))).astype(np.float64)
    q = q + np.triu(q, 1).T
    for count in counts:
        print(f"[gpu] energy tiles n={n} count={count}", flush=True)
        st = rng.integers(0, 2, (count, n)).astype(np.uint8)
        assert np.array_equal(ctx.energy_fp64(q, st), oracle.energy(q, st)), count


def _energy_in_the_kernels_order(q, x):
    """0.5 sum_j x_j (Y_j + q_jj) with Y = x q summed over k ascending (products by
    0 or 1 are exact), then columns 16 apart, the tree over 16, 128 columns at a
    time: every addition the one that the energy kernel documents."""
    n = q.shape[0]
    y = np.zeros((len(x), n))
    for k in range(n):
        y += x[:, k, None] * q[k]
    term = y + np.diag(q)
    e = np.zeros(len(x))
    for c0 in range(0, n, 128):
        s = np.zeros((len(x), 16))
        for c in range(c0, min(c0 + 128, n)):
            s[:, c % 16] = np.where(x[:, c] > 0, s[:, c % 16] + term[:, c], s[:, c % 16])
        for o in (1, 2, 4, 8):
            s = s + s[:, np.arange(16) ^ o]
        e = e + 0.5 * s[:, 0]
    return e


@pytest.mark.parametrize("n,count", [(65, 40), (127, 33), (128, 17), (129, 64), (300, 50),
                                     (515, 20), (1024, 16), (200, 9000)])
def test_energy_sums_are_in_the_documented_order(ctx, n, count):
    """Coefficients of many magnitudes, where another order of the sums shows in
    the last bits: equal bit for bit to the documented one."""
    rng = np.random.default_rng(n)
    q = np.triu(rng.normal(size=(n, n)) * 10.0 ** rng.uniform(-6, 6, (n, n)))
    q = q + np.triu(q, 1).T
    st = rng.integers(0, 2, (count, n)).astype(np.uint8)
    print(f"[gpu] energy order n={n} count={count}", flush=True)
    want = _energy_in_the_kernels_order(q, st.astype(np.float64))
    assert np.array_equal(ctx.energy_fp64(q, st), want)
    # the coefficients do tell orders apart
    assert (want != 0.5 * ((st @ q + np.diag(q)) * st).sum(1)).any()


@pytest.mark.parametrize("n,count", [(7, 100), (28, 300), (57, 257), (64, 65600)])
def test_small_energies_are_the_references_sum(ctx, n, count):
    """n <= 64: the reference's loop over i, then j >= i, bit for bit."""
    rng = np.random.default_rng(n)
    q = np.triu(rng.normal(size=(n, n)) * 10.0 ** rng.uniform(-6, 6, (n, n)))
    q = q + np.triu(q, 1).T
    st = rng.integers(0, 2, (count, n)).astype(np.uint8)
    print(f"[gpu] small energies n={n} count={count}", flush=True)
    e, x = np.zeros(count), st.astype(np.float64)
    for i in range(n):
        for j in range(i, n):
            e += q[i, j] * (x[:, i] * x[:, j])
    assert np.array_equal(ctx.energy_fp64(q, st), e)


@pytest.mark.parametrize("path,ground", _kats())
def test_reference_anneal_matches_oracle_chain_on_kats(ctx, path, ground):
    q = load_qubo(path)
    n = q.shape[0]
    beta = oracle.geometric_schedule(0.1, 10.0, 500)
    print(f"[gpu] reference anneal {os.path.basename(path)} n={n}", flush=True)
    best, be, states, energies = ctx.anneal_reference(q, beta, 128, seed=1234)
    s_or, e_or = oracle.anneal(q, n, beta, 128, seed=1234)
    assert (states == s_or).all()
    assert np.allclose(energies, oracle.energy(q, states), rtol=0, atol=1e-12)
    assert np.allclose(energies, e_or, rtol=0, atol=1e-12)
    assert abs(be - ground) < 1e-12  # every KAT is solved
    i = int(np.argmin(energies))
    assert (best == states[i]).all()


def test_reference_anneal_config1_chain_and_hit_rate(ctx):
    """Config 1: N=28 dense, geometric 0.1->1.0, 1000 iterations, 1024 tries."""
    q = load_qubo(os.path.join(GOLDEN, "c1_dense28.qubo"))
    with open(os.path.join(GOLDEN, "c1_ground.json")) as f:
        ground = json.load(f)["energy"]
    beta = oracle.geometric_schedule(0.1, 1.0, 1000)
    best, be, states, energies = ctx.anneal_reference(q, beta, 1024, seed=1234)
    # (1) FP64 energies of every returned state equal the reference energy function
    ref_e = oracle.energy(q, states)
    assert np.all(np.abs(energies - ref_e) <= 1e-9 * np.abs(ref_e))
    # (2) same chains as the oracle on the same streams
    s_or, _ = oracle.anneal(q, 28, beta, 1024, seed=1234)
    assert (states == s_or).all(axis=1).mean() >= 0.999
    # (3) law: per-replica ground-state hit rate vs the literal restatement on
    #     independent streams (replicas 4096.. of the same seed), binomial CI
    s_lit, e_lit = oracle.anneal(q, 28, beta, 1024, seed=1234, first_replica=4096, literal=True)
    tol = 1e-9 * abs(ground)
    k_gpu = int(np.sum(energies <= ground + tol))
    k_ref = int(np.sum(e_lit <= ground + tol))
    p = (k_gpu + k_ref) / 2048
    se = np.sqrt(p * (1 - p) * (2 / 1024)) + 1e-12
    print(f"[gpu] C1 hit rate gpu={k_gpu}/1024 ref={k_ref}/1024", flush=True)
    assert abs(k_gpu - k_ref) / 1024 <= 1.96 * se + 1.0 / 1024
    assert be >= ground - tol


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 512, 513, 1025, 2048, 2049])
def test_reference_anneal_windows_match_oracle_chain(ctx, n):
    """Sizes at the edges of the fields a lane holds, attempt counts that are
    no multiple of the 64 taken together, three attempts per beta, and betas
    for which the test on -b ln u does not hold (0, negative, infinite): the
    oracle's chains bit for bit (integer Q, so every field is exact)."""
    rng = np.random.default_rng(n)
    q = np.triu(rng.integers(-3, 4, (n, n)).astype(np.float64))
    q = q + np.triu(q, 1).T
    scale = max(1.0, np.sqrt(n) / 2)
    beta = np.concatenate([np.geomspace(0.3, 3.0, 40) * scale, [0.0, -1.0, np.inf, 1e-300],
                           np.geomspace(3.0, 0.5, 21) * scale])
    print(f"[gpu] reference windows n={n}", flush=True)
    tries = 70 if n <= 1025 else 20
    best, be, states, energies = ctx.anneal_reference(q, beta, tries, sweeps_per_beta=3, seed=77)
    s_or, e_or = oracle.anneal(q, n, beta, tries, sweeps_per_beta=3, seed=77)
    assert (states == s_or).all()
    assert np.array_equal(energies, e_or)
    assert be == e_or.min() and (best == s_or[int(np.argmin(e_or))]).all()


@pytest.mark.parametrize("n", [64, 65, 640, 767, 768])
def test_reference_anneal_many_tries_match_oracle_chain(ctx, n):
    """Both sides of the numbers of tries and spins at which another kernel takes
    the chains: a try's chain does not depend on the others, so the runs agree, and
    with the oracle bit for bit (integer Q)."""
    rng = np.random.default_rng(n)
    q = np.triu(rng.integers(-3, 4, (n, n)).astype(np.float64))
    q = q + np.triu(q, 1).T
    beta = np.geomspace(0.5, 2.0, 70) * np.sqrt(n)
    s_or, e_or = oracle.anneal(q, n, beta, 2049 if n < 100 else 64, seed=7)
    last = None
    for tries in (2048, 2049):
        print(f"[gpu] reference n={n} tries={tries}", flush=True)
        best, be, states, energies = ctx.anneal_reference(q, beta, tries, seed=7)
        k = min(tries, len(e_or))
        assert (states[:k] == s_or[:k]).all() and np.array_equal(energies[:k], e_or[:k])
        i = int(np.argmin(energies))
        assert be == energies[i] and (best == states[i]).all()
        if last is not None:
            assert (states[:2048] == last[0]).all() and np.array_equal(energies[:2048], last[1])
        last = states, energies


def test_reference_anneal_large_n_uses_global_fields(ctx):
    rng = np.random.default_rng(5)
    n = 4100  # above the LDS-resident field limit
    q = np.zeros((n, n))
    idx = rng.integers(0, n, (3 * n, 2))
    for i, j in idx:
        if i != j:
            q[i, j] = q[j, i] = rng.integers(-2, 3)
    q[np.arange(n), np.arange(n)] = rng.integers(-2, 3, n)
    beta = oracle.geometric_schedule(0.1, 2.0, 200)
    _, be, states, energies = ctx.anneal_reference(q, beta, 4)
    s_or, e_or = oracle.anneal(q, n, beta, 4)
    assert (states == s_or).all()
    assert np.array_equal(energies, oracle.energy(q, states))


def test_small_n_energies_follow_the_reference_order_bit_for_bit(ctx):
    """n <= 64: the FP64 energies are summed in the reference's order (one
    accumulator over the upper triangle, row by row, annealing.hpp:31-40), so
    on real-valued Q they equal the oracle's bit for bit, through
    os_energy_fp64 and through the energies reference mode returns."""
    rng = np.random.default_rng(17)
    for n in (5, 28, 33, 64):
        q = np.triu(rng.uniform(-1.0, 1.0, (n, n)))
        q = q + np.triu(q, 1).T
        print(f"[gpu] small-n energies n={n}", flush=True)
        states = rng.integers(0, 2, (300, n)).astype(np.uint8)
        assert np.array_equal(ctx.energy_fp64(q, states), oracle.energy(q, states))
        beta = oracle.geometric_schedule(0.1, 1.0, 50)
        _, _, st, en = ctx.anneal_reference(q, beta, 64)
        assert np.array_equal(en, oracle.energy(q, st))


def test_reference_anneal_rejects_bad_arguments(ctx):
    with pytest.raises(onesolver_amd.InvalidArgument):
        ctx.anneal_reference(np.zeros((3, 3)), np.ones(5), 0)


def test_cli_gpu_device_end_to_end(tmp_path):
    out = tmp_path / "r.csv"
    r = subprocess.run([onesolver_amd.CLI_PATH, "--input",
                        os.path.join(GOLDEN, "examples", "csp13.qubo"), "--output", str(out),
                        "--device-type", "gpu", "--num-iter", "2000", "--num-tries", "256",
                        "--beta-max", "5"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert "Using device: " in r.stdout
    head, row = out.read_text().splitlines()
    assert head.endswith(",energy")
    assert float(row.split(",")[-1]) == -32.0


def test_reference_anneal_published_runs_band(ctx):
    """The GPU's reference-mode chains against the reference's published
    runs (benchmarks/annealing/results/128/001.csv, beta 0.1 -> 10 as a
    temperature): every published best-of-10 energy lies inside the 0.5-99.5%
    band of the GPU's best-of-10 over 2000 blocks of independent replicas."""
    import published_band as pb
    from qubo_io import published_grid

    n = 128
    q = load_qubo(os.path.join(GOLDEN, "chimera", f"{n}_001.qubo"))
    pts = pb.published_points(published_grid(n))
    cells = [("linear", 1000), ("geometric", 500), ("geometric", 1000)]

    def sample(kind, it, count):
        beta = pb.schedule(oracle, kind, it)
        print(f"[gpu] reference anneal n={n} {kind} {it} x {count}", flush=True)
        _, _, states, e = ctx.anneal_reference(q, beta, count, seed=2024)
        assert np.all(np.abs(e - oracle.energy(q, states)) <= 1e-9 * np.abs(e))
        return e

    pits = pb.point_pits(sample, pts, cells, (10,), 2000)
    ok, outside, mean = pb.band_verdict(pits)
    print(f"[gpu] published band: mean PIT {mean:.3f} {pits}", flush=True)
    assert ok, (outside, mean)
