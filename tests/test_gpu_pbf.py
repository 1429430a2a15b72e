"""GPU parity of the position based fluids step against the oracle.

The GPU path fuses the reference's kernels (see csrc/pbf.hip) but keeps every particle's
summation order, so positions, velocities, densities, lambdas, predicted positions and the
grid are compared for exact equality after every step.  The bar of the task is 1e-5
relative over 10 steps; exact equality is stricter.
"""
import ctypes
import hashlib
import json
import os
import time

import numpy as np
import pytest

from helpers import _eq, compare_pbf, log, make_pbf_pair
from realtimeparticles_amd import capi, scenes

pytestmark = pytest.mark.gpu


def small_scene(seed=1, lattice=(24, 16, 16)):
    return scenes.dam_break(lattice, (4, 2, 2), (40, 20, 20), seed=seed, name="pbf-small")


def test_pbf_65k_ten_substeps_bit_exact():
    sc = scenes.pbf_scene("pbf-65k")
    gpu, orc = make_pbf_pair(sc, iters=4)
    for step in range(1, 11):
        log(f"pbf-65k step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


@pytest.mark.parametrize("iters", [0, 1, 2, 3])
def test_pbf_iteration_counts(iters):
    sc = small_scene(seed=2)
    gpu, orc = make_pbf_pair(sc, iters=iters)
    for step in range(1, 6):
        log(f"iters={iters} step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


@pytest.mark.parametrize("variant", [
    dict(isVorticityConfEnabled=0),
    dict(isArtPressureEnabled=0),
    dict(artPressureExp=1),
    dict(artPressureExp=0),
    # the reference's own defaults (Fluids.hpp:17-32) in their own box/grid scale
    dict(restDensity=450.0, timeStep=0.01, artPressureRadius=0.006, artPressureCoeff=0.001,
         vorticityConfCoeff=0.0004, xsphViscosityCoeff=0.0001),
])
def test_pbf_parameter_variants(variant):
    sc = small_scene(seed=3)
    gpu, orc = make_pbf_pair(sc, iters=2, gravity=9.81, **variant)
    for step in range(1, 6):
        log(f"variant {variant} step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


@pytest.mark.parametrize("flags", [0, 13, 29, 64, 76])
def test_graph_replay_equals_direct_launches(flags):
    """flags 13: XCD blocks, thread order and survivor lists inside the captured graphs; 29:
    the same with the brick thread order; 64 and 76: the quad passes, alone and with thread
    order and lists."""
    sc = small_scene(seed=4)
    a, _ = make_pbf_pair(sc, iters=4)
    b, _ = make_pbf_pair(sc, iters=4)
    a.set_tuning(64, flags, 0, 16)
    b.use_graph(False)
    for rep in range(3):
        log(f"graph replay {rep}")
        a.update(4)   # two graph launches of two substeps
        for _ in range(4):
            b.update(1)
        pa, va = a.read_state()
        pb, vb = b.read_state()
        _eq(pa, pb, f"pos after replay {rep}")
        _eq(va, vb, f"vel after replay {rep}")
    a.update(3)       # one graph launch + one direct substep
    b.update(3)
    _eq(a.read_state()[0], b.read_state()[0], "pos after odd count")
    a.update(2)       # graph recaptured for the new buffer parity
    b.update(2)
    _eq(a.read_state()[0], b.read_state()[0], "pos after recapture")
    a.close()
    b.close()


@pytest.mark.parametrize("flags", [13, 29, 76])
def test_graph_replay_with_odd_thread_order_calls(flags):
    """Three Jacobi iterations: a substep orders the threads three times, so a direct substep
    leaves the thread order's count tables the other way round from the graph's capture; the
    graph must be captured again before its next replay.  Graph and direct runs alternate and
    every state equals a direct-only run's."""
    sc = small_scene(seed=9)
    a, _ = make_pbf_pair(sc, iters=3)
    b, _ = make_pbf_pair(sc, iters=3)
    a.set_tuning(64, flags, 0, 16)
    b.set_tuning(64, flags, 0, 16)
    b.use_graph(False)
    for rep, k in enumerate((2, 1, 2, 3, 4, 1, 1, 2)):
        log(f"odd thread-order calls, flags {flags}, update({k})")
        a.update(k)
        for _ in range(k):
            b.update(1)
        pa, va = a.read_state()
        pb, vb = b.read_state()
        _eq(pa, pb, f"pos after update({k}) #{rep}")
        _eq(va, vb, f"vel after update({k}) #{rep}")
    a.close()
    b.close()


@pytest.mark.parametrize("flags,sort_bits", [(0, 0), (13, 0), (0, 7), (13, 10), (13, 11), (29, 9),
                                             (76, 0), (92, 9)])
def test_nb_particles_change_keeps_reference_sort(flags, sort_bits):
    # Model::setNbParticles (Model.hpp:106) does not reset the grid: the keys of particles
    # that left the active range stay in the reference's whole-buffer sort.  flags 13: the
    # thread order's and survivor lists' sizes follow the count.  sort_bits: the digit width
    # of the sort over the stale-tail keys (up to 2 NC + maxN).
    sc = small_scene(seed=5)
    gpu, orc = make_pbf_pair(sc, iters=2)
    gpu.set_tuning(128, flags, sort_bits, 16)
    gpu.update(1)
    orc.step(1)
    compare_pbf(gpu, orc, sc.n, 1)
    n2 = sc.n - 1000
    gpu.set_nb_particles(n2)
    orc.s.n = n2
    for step in range(2, 5):
        log(f"shrunk step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, n2, step)
    gpu.set_nb_particles(sc.n)
    orc.s.n = sc.n
    gpu.update(1)
    orc.step(1)
    compare_pbf(gpu, orc, sc.n, 5)
    gpu.close()


def test_density_error_metric():
    sc = small_scene(seed=6)
    gpu, orc = make_pbf_pair(sc, iters=4)
    gpu.update(3)
    orc.step(3)
    e = gpu.density_error()
    rel = orc.density[: sc.n].astype(np.float64) / np.float32(sc.rest_density) - 1.0
    assert e[0] == pytest.approx(np.abs(rel).max(), rel=1e-5)
    assert e[1] == pytest.approx(np.abs(rel).mean(), rel=1e-4)
    assert e[2] == pytest.approx(max(rel.max(), 0.0), rel=1e-5, abs=1e-7)
    gpu.close()


def test_pause_and_profiling():
    sc = small_scene(seed=7)
    gpu, _ = make_pbf_pair(sc, iters=2)
    p0, _ = gpu.read_state()
    gpu.pause(True)
    gpu.update(3)
    _eq(gpu.read_state()[0], p0, "paused state")
    gpu.pause(False)
    gpu.enable_profiling(True)
    gpu.update(2)
    prof = gpu.profile()
    assert prof["pbf_density_lambda"][0] == 4 and prof["pbf_correct"][0] == 4
    assert prof["radix_sort"][0] == 2 and prof["pbf_xsph"][0] == 2
    assert all(ms >= 0 for _, ms in prof.values())
    gpu.close()


def test_errors_are_reported():
    sc = small_scene(seed=8)
    gpu, _ = make_pbf_pair(sc, iters=1)
    with pytest.raises(capi.RtpError, match="exceeds"):
        gpu.set_nb_particles(sc.max_n + 1)
    with pytest.raises(capi.RtpError):
        gpu.load_state(np.zeros((sc.max_n + 1, 4), np.float32), np.zeros((sc.max_n + 1, 4), np.float32))
    gpu.close()


def test_checkpoint_restore_replays_identically():
    sc = small_scene(seed=9)
    gpu, _ = make_pbf_pair(sc, iters=3)
    gpu.update(3)
    gpu.save_checkpoint()
    gpu.update(1)
    gpu.update(2)
    pa, va = gpu.read_state()
    ka, ia, sa = gpu.read_grid()
    for rep in range(2):
        gpu.restore_checkpoint()
        gpu.update(3)
        pb, vb = gpu.read_state()
        _eq(pb, pa, f"pos after restore {rep}")
        _eq(vb, va, f"vel after restore {rep}")
        kb, ib, sb = gpu.read_grid()
        _eq(kb, ka, f"keys after restore {rep}")
        _eq(sb, sa, f"startEnd after restore {rep}")
    # restoring across a particle-count change puts the count back as well
    gpu.restore_checkpoint()
    gpu.set_nb_particles(sc.n - 100)
    gpu.restore_checkpoint()
    assert gpu.read_nb_particles() == sc.n
    gpu.update(3)
    _eq(gpu.read_state()[0], pa, "pos after restore over a count change")
    gpu.close()


@pytest.mark.parametrize("block,flags,queue,sort_bits", [
    (256, 2, 16, 0), (128, 2, 24, 7), (64, 3, 48, 0), (192, 1, 64, 10), (256, 3, 16, 11),
    (256, 0, 64, 0), (128, 0, 8, 8), (64, 4, 64, 0), (128, 6, 32, 9), (256, 7, 16, 0),
    (192, 5, 40, 4), (64, 13, 16, 10), (256, 8, 8, 0), (128, 12, 24, 11), (64, 15, 12, 7),
    (64, 13, 16, 5), (128, 13, 16, 6), (64, 29, 16, 10), (256, 20, 24, 0), (128, 31, 12, 8),
    (64, 64, 16, 0), (128, 68, 16, 10), (256, 72, 8, 0), (64, 76, 16, 9), (64, 92, 16, 10),
    (128, 84, 24, 7)])
@pytest.mark.parametrize("mapping", ["literal", "stable"])
def test_launch_shapes_do_not_change_bits(block, flags, queue, sort_bits, mapping):
    """XCD-contiguous block order, LDS wave tiles, thread re-ordering by current cell (in
    cell-index or brick order), the survivor-queue depth, replayed survivor lists, the quad
    passes (four lanes per particle, terms added in walk order) and the sort's digit width
    change where candidates are read from, which thread handles a particle and when the
    neighbour bodies run -- never which candidates or in which order."""
    sc = scenes.dam_break((48, 24, 24), (4, 2, 2), (40, 20, 20), seed=6)
    prm = sc.params(mapping)
    gpu, orc = make_pbf_pair(sc, iters=3, **{k: v for k, v in prm.items()})
    gpu.set_tuning(block, flags, sort_bits, queue)
    for step in range(1, 5):
        log(f"block {block} flags {flags} queue {queue} bits {sort_bits} {mapping} step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()



@pytest.mark.parametrize("block,queue,flags", [(256, 8, 0), (64, 64, 0), (128, 48, 0),
                                               (64, 16, 13), (256, 12, 8), (64, 16, 29),
                                               (64, 16, 64), (64, 16, 72), (64, 16, 92)])
def test_overfull_cell_keeps_bits(block, queue, flags):
    """20,000 particles in one cell (the cap iterates 101 of them) and 50 in the next cell
    of its column: the walks through them are no longer back-to-back ranges, and survivor
    queues of every depth drain in the reference's order.  A clump around a corner of eight
    capped cells gives particles more survivors than a recorded list holds: they walk again
    instead of replaying."""
    sc = scenes.dam_break((16, 16, 16), (4, 2, 2), (40, 20, 20), seed=8, extra=0)
    rng = np.random.default_rng(5)
    k = 20000
    dense = np.zeros((k, 4), np.float32)
    # inside cell (8, 8, 8) of the 40 x 20 x 20 grid (cell size 0.1, walls at -2/-1/-1)
    dense[:, 0] = -2.0 + 0.8 + 0.1 * rng.random(k, dtype=np.float32) * 0.98 + 0.001
    dense[:, 1] = -1.0 + 0.8 + 0.1 * rng.random(k, dtype=np.float32) * 0.98 + 0.001
    dense[:, 2] = -1.0 + 0.8 + 0.1 * rng.random(k, dtype=np.float32) * 0.98 + 0.001
    # and 50 in the next cell of the same column, (8, 8, 9): ranges after the capped cell
    # start 20,000 indices past its start
    nxt = np.zeros((50, 4), np.float32)
    nxt[:, :3] = dense[:50, :3]
    nxt[:, 2] += np.float32(0.1)
    # and 4,000 within 0.02 of the corner (0, 0.4, 0.4) that cells (19..20, 13..14, 13..14)
    # share: all eight are capped, so each of these particles has over 800 survivors, more
    # than a recorded list holds
    ball = np.zeros((4000, 4), np.float32)
    d = rng.normal(size=(4000, 3))
    d *= 0.02 * rng.random((4000, 1)) ** (1.0 / 3.0) / np.linalg.norm(d, axis=1, keepdims=True)
    ball[:, :3] = np.array([0.0, 0.4, 0.4]) + d
    sc.pos = np.concatenate([sc.pos, dense, nxt, ball])
    sc.vel = np.zeros_like(sc.pos)
    sc.n = sc.pos.shape[0]
    sc.max_n = (sc.n + 511) // 512 * 512 + 512
    gpu, orc = make_pbf_pair(sc, iters=2, **sc.params("stable"))
    gpu.set_tuning(block, flags, 0, queue)
    for step in range(1, 3):
        log(f"overfull cell, block {block}, queue {queue}, flags {flags}, step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


def _trace():
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "pbf65k_trace.json")
    with open(path) as f:
        return json.load(f)


def _digest(a: np.ndarray) -> str:
    return hashlib.sha256(np.ascontiguousarray(a, np.float32).tobytes()).hexdigest()


def _density_error(density: np.ndarray, rho0: float) -> list:
    rel = density.astype(np.float64) / np.float64(np.float32(rho0)) - 1.0
    return [float(np.abs(rel).max()), float(np.abs(rel).mean()), float(max(rel.max(), 0.0))]


@pytest.mark.parametrize("mapping", ["literal", "stable"])
def test_pbf_65k_long_run(mapping):
    """The 64x32x32 dam break (4 iterations) for 300 frames (600 substeps) against the
    oracle's run of the same scene (tests/golden/pbf65k_trace.json, written by
    tests/golden/make_pbf65k_trace.py):
    - graph replay at a tuned launch shape: every field against the live oracle for the first
      30 substeps, then the SHA-256 of positions and velocities against the oracle's every
      30 substeps up to 600;
    - direct launches at the default shape: max, mean and compression-only |rho/rho0 - 1| of
      the last Jacobi iteration's density after every one of the 600 substeps within 1e-4 of
      the oracle's (the full-run bar; the run is bit-exact, so they are equal), and the final
      state equal to the graph run's."""
    trace = _trace()[mapping]
    sc = scenes.pbf_scene("pbf-65k")
    prm = sc.params(mapping)
    assert trace["params"] == {k: prm[k] for k in trace["params"]}
    gpu, orc = make_pbf_pair(sc, iters=4, **prm)
    gpu.set_tuning(64, capi.LAUNCH_RESORT | capi.LAUNCH_XCD_MAP | capi.LAUNCH_NB_LIST, 0, 16)
    gpu.save_checkpoint()
    for step in range(1, 31):
        gpu.update(1)
        orc.step(1)
        if step % 10 == 0:
            log(f"pbf-65k {mapping} step {step} against the oracle")
            compare_pbf(gpu, orc, sc.n, step)
    hashes = {h["substep"]: h for h in trace["state_sha256"]}
    done = 30
    while done < 600:
        pos, vel = gpu.read_state()
        want = hashes[done]
        assert _digest(pos) == want["pos"] and _digest(vel) == want["vel"], \
            f"{mapping}: state after substep {done} differs from the oracle's run"
        gpu.update(30)
        done += 30
    a_pos, a_vel = gpu.read_state()
    assert _digest(a_pos) == hashes[600]["pos"] and _digest(a_vel) == hashes[600]["vel"], \
        f"{mapping}: state after substep 600 differs from the oracle's run"
    log(f"pbf-65k {mapping}: graph run equals the oracle's at every 30th substep")
    assert np.all(a_pos[:, 3] == 0.0) and np.all(a_vel[:, 3] == 0.0)

    gpu.restore_checkpoint()
    gpu.use_graph(False)
    gpu.set_tuning(256, 0, 0, 24)
    rho0 = prm["restDensity"]
    worst = 0.0
    for step in range(1, 601):
        gpu.update(1)
        got = _density_error(gpu.read_field(capi.FIELD_DENSITY, sc.n), rho0)
        want = trace["density_error"][step - 1]
        dev = max(abs(g - w) for g, w in zip(got, want))
        worst = max(worst, dev)
        assert dev <= 1e-4, f"{mapping} substep {step}: density error {got} vs oracle {want}"
    log(f"pbf-65k {mapping}: density-error trace within {worst:.3g} of the oracle over 600 "
        f"substeps (last {trace['density_error'][-1]})")
    b_pos, b_vel = gpu.read_state()
    _eq(b_pos, a_pos, "600 substeps, graph + tuned launches vs direct default launches (pos)")
    _eq(b_vel, a_vel, "600 substeps, graph + tuned launches vs direct default launches (vel)")
    gpu.close()


@pytest.mark.parametrize("flags", [capi.LAUNCH_QUAD,
                                   capi.LAUNCH_QUAD | capi.LAUNCH_RESORT | capi.LAUNCH_NB_LIST])
@pytest.mark.parametrize("mapping", ["literal", "stable"])
def test_pbf_65k_quad_passes_follow_oracle_trace(mapping, flags):
    """The 64x32x32 dam break with the quad passes (graph replay, 600 substeps): the SHA-256
    of positions and velocities against the oracle's run every 30 substeps."""
    trace = _trace()[mapping]
    sc = scenes.pbf_scene("pbf-65k")
    prm = sc.params(mapping)
    gpu, _ = make_pbf_pair(sc, iters=4, **prm)
    gpu.set_tuning(64, flags, 0, 16)
    hashes = {h["substep"]: h for h in trace["state_sha256"]}
    done = 0
    while done < 600:
        gpu.update(30)
        done += 30
        log(f"pbf-65k quad {mapping} flags {flags} substep {done}")
        pos, vel = gpu.read_state()
        want = hashes[done]
        assert _digest(pos) == want["pos"] and _digest(vel) == want["vel"], \
            f"{mapping}: state after substep {done} differs from the oracle's run"
    gpu.close()


def test_short_math_general_lanes_keep_bits():
    """Neighbour pairs that send single lanes down the general correctly rounded forms inside
    the short ones: squared distances in (0, 2^-96) (pairs 1e-16 and 1e-20 apart, next to
    the x = 0 plane) and gradient numerators in (0, 2^-90) (pairs 0.05 apart whose x or z
    differ by 1e-33 or 1e-35), placed among ordinary lattice particles so that their waves
    also run the short forms.  Every field against the oracle, bit for bit."""
    sc = scenes.dam_break((16, 16, 16), (4, 2, 2), (40, 20, 20), seed=12, extra=0)
    special = np.array([
        [1e-16, 0.3, 0.3, 0], [2e-16, 0.3, 0.3, 0],          # d2 = 1e-32
        [1e-20, 0.3, 0.5, 0], [2e-20, 0.3, 0.5, 0],          # d2 = 1e-40 (denormal)
        [1e-33, 0.4, 0.4, 0], [0.0, 0.45, 0.4, 0],           # dx = 1e-33
        [0.6, 0.4, 1e-35, 0], [0.6, 0.45, 0.0, 0],           # dz = 1e-35
        [0.62, 0.41, 0.01, 0], [0.63, 0.42, 0.02, 0],        # ordinary neighbours of the above
        [1e-30, 0.35, 0.31, 0], [-1e-30, 0.33, 0.29, 0],
    ], np.float32)
    sc.pos = np.concatenate([sc.pos, special])
    sc.vel = np.zeros_like(sc.pos)
    sc.n = sc.pos.shape[0]
    sc.max_n = (sc.n + 511) // 512 * 512 + 512
    for mapping in ("stable", "literal"):
        gpu, orc = make_pbf_pair(sc, iters=3, **sc.params(mapping))
        for step in range(1, 4):
            log(f"general lanes, {mapping}, step {step}")
            gpu.update(1)
            orc.step(1)
            compare_pbf(gpu, orc, sc.n, step)
        gpu.close()


@pytest.mark.parametrize("flags,queue", [(0, 8), (8, 8), (13, 16), (29, 24), (64, 16), (72, 16)])
@pytest.mark.parametrize("n", [1, 3, 61, 127, 1000])
def test_checked_pairs_in_lists_keep_bits(flags, queue, n):
    """Pairs that the unchecked terms of a replayed survivor list would get wrong, in models down
    to one particle (the first few survivors of a list, the last partial wave): coincident
    particles, distances within a few ulp of h on either side, a squared distance in (0, 2^-52),
    numerators in (0, 2^-90), and a plane of equal z, whose zero numerators need no check."""
    h = 0.1
    rng = np.random.default_rng(n)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = 0.25 * rng.random((n, 3), dtype=np.float32) + np.float32(0.05)
    pos[: n // 3, 2] = np.float32(0.15)
    k = n // 8
    pos[k: 2 * k, :3] = pos[:k, :3]  # coincident
    pos[2 * k: 3 * k, :3] = pos[:k, :3]
    pos[2 * k: 3 * k, 0] += np.float32(h) * (1 + np.arange(-(k // 2), k - k // 2, dtype=np.float32) * np.float32(2.0 ** -23))
    if n > 8:
        pos[-1, :3], pos[-2, :3] = (1e-9, 0.2, 0.2), (2e-9, 0.2, 0.2)
        pos[-3, :3], pos[-4, :3] = (1e-33, 0.1, 0.2), (0.0, 0.15, 0.2)
    sc = scenes.dam_break((4, 4, 4), (4, 2, 2), (40, 20, 20), seed=1)
    sc.pos, sc.vel, sc.n, sc.max_n = pos, np.zeros_like(pos), n, 1024
    for mapping in ("stable", "literal"):
        gpu, orc = make_pbf_pair(sc, iters=2, **sc.params(mapping))
        gpu.set_tuning(64, flags, 0, queue)
        for step in range(1, 4):
            log(f"checked pairs, n {n}, flags {flags}, {mapping}, step {step}")
            gpu.update(1)
            orc.step(1)
            compare_pbf(gpu, orc, sc.n, step)
        gpu.close()


@pytest.mark.parametrize("flags", [0, 2, 8, 13, 64, 72])
@pytest.mark.parametrize("mapping", ["stable", "literal"])
def test_pairs_whose_squared_distance_underflows(flags, mapping):
    """Particles apart by less than 2^-75, as they can be near coordinate 0: the squared distance is
    0 and the reference's gradient with it, though the differences are not; walked and replayed."""
    rng = np.random.default_rng(7)
    n = 60
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = 0.25 * rng.random((n, 3), dtype=np.float32) - np.float32(0.1)
    for k, d in enumerate([(1e-24, 0, 0), (2e-23, 0, 0), (0, 0, -1e-24), (1e-30, 0, 2e-23), (1e-38, 0, 1e-40)]):
        pos[2 * k, 0] = pos[2 * k, 2] = 0.0
        pos[2 * k + 1, :3] = pos[2 * k, :3] + np.array(d, np.float32)
    sc = scenes.dam_break((4, 4, 4), (4, 2, 2), (40, 20, 20), seed=1)
    sc.pos, sc.vel, sc.n, sc.max_n = pos, np.zeros_like(pos), n, 1024
    gpu, orc = make_pbf_pair(sc, iters=2, **sc.params(mapping))
    gpu.set_tuning(64, flags, 0, 16)
    for step in range(1, 4):
        log(f"underflowing pairs, flags {flags}, {mapping}, step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


@pytest.mark.parametrize("res", [(2, 2, 2), (5, 3, 2), (4, 2, 3), (3, 4, 5)])
@pytest.mark.parametrize("flags", [0, 2, 8, 13, 64, 72])
def test_grids_that_wrap_in_every_column(flags, res):
    """Grids of two to five cells a side: most columns wrap, so their cells are not one index range
    (and with two cells a side two of them are the same cell), in the one-lane walks' column table
    and in the quads' ranges."""
    rng = np.random.default_rng(sum(res))
    n = 40 * res[0] * res[1] * res[2] // 4
    box = tuple(np.float32(r * 0.1) for r in res)
    sc = scenes.dam_break((4, 4, 4), (4, 2, 2), (40, 20, 20), seed=1)
    sc.box, sc.res, sc.n, sc.max_n = tuple(float(b) for b in box), res, n, 1024
    sc.pos = np.zeros((n, 4), np.float32)
    sc.pos[:, :3] = (rng.random((n, 3), dtype=np.float32) - np.float32(0.5)) * np.array(box, np.float32)
    sc.vel = np.zeros_like(sc.pos)
    gpu, orc = make_pbf_pair(sc, iters=2, **sc.params("stable"))
    gpu.set_tuning(64, flags, 0, 16)
    gpu.save_checkpoint()
    gpu.update(1)
    gpu.restore_checkpoint()
    for step in range(1, 4):
        log(f"wrapping grid {res}, flags {flags}, step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


@pytest.mark.parametrize("flags", [0, 2, 8, 13, 29])
def test_column_table_only_up_to_eight_cells_a_particle(flags):
    """2,000 particles on 16,000 cells, the most the column table serves, then 1,999, whose one-lane
    walks merge the columns' cells themselves."""
    sc = scenes.dam_break((20, 10, 10), (4, 2, 2), (40, 20, 20), seed=3, extra=48)
    gpu, orc = make_pbf_pair(sc, iters=2, **sc.params("stable"))
    gpu.set_tuning(64, flags, 0, 16)
    gpu.enable_profiling(True)
    for n in (2000, 1999):
        gpu.set_nb_particles(n)
        orc.s.n = n
        gpu.reset_profile()
        for step in range(1, 4):
            log(f"column table, n {n}, flags {flags}, step {step}")
            gpu.update(1)
            orc.step(1)
            compare_pbf(gpu, orc, n, step)
        assert gpu.profile().get("pbf_columns", (0, 0))[0] == (3 if n == 2000 else 0)
    gpu.close()


@pytest.mark.parametrize("box", [(0.2, 0.1, 0.1), (800.0, 400.0, 400.0)])
def test_general_forms_outside_short_range(box):
    """Effect radius h = 0.005 and h = 20, outside [2^-7, 2^4] where the short correctly
    rounded forms are enabled: every body takes the general sequences."""
    sc = scenes.dam_break((16, 16, 16), box, (40, 20, 20), seed=13)
    gpu, orc = make_pbf_pair(sc, iters=2, **sc.params("stable"))
    for step in range(1, 4):
        log(f"h = {box[0] / 40}, step {step}")
        gpu.update(1)
        orc.step(1)
        compare_pbf(gpu, orc, sc.n, step)
    gpu.close()


@pytest.mark.parametrize("flags", [0, 13, 29, 76])
def test_bad_state_matches_oracle(flags):
    """NaN and +-inf coordinates, a NaN velocity, particles outside the walls and exactly on
    +-W in a dam break: the hash aliases and clamps them (grid.cl:14-38), the first clamp
    turns NaN positions into the lower wall, far and NaN neighbours take the exact
    expressions -- every field against the oracle, bit for bit (NaN compares equal)."""
    sc = scenes.dam_break((16, 16, 16), (4, 2, 2), (40, 20, 20), seed=14, extra=0)
    bad = np.array([
        [np.nan, 0.2, 0.2, 0], [0.3, np.inf, 0.2, 0], [0.3, 0.2, -np.inf, 0],
        [2.5, 0.1, 0.1, 0], [0.1, -1.3, 0.1, 0], [0.1, 0.1, 1.7, 0],
        [2.0, 0.5, 0.5, 0], [-2.0, 0.5, 0.5, 0], [0.5, 1.0, -1.0, 0],
        [0.31, 0.21, 0.21, 0], [0.32, 0.22, 0.2, 0], [1.95, 0.12, 0.1, 0],
    ], np.float32)
    vel = np.zeros_like(bad)
    vel[9, :3] = np.nan
    sc.pos = np.concatenate([sc.pos, bad])
    sc.vel = np.concatenate([sc.vel, vel])
    sc.n = sc.pos.shape[0]
    sc.max_n = (sc.n + 511) // 512 * 512 + 512
    for mapping in ("stable", "literal"):
        gpu, orc = make_pbf_pair(sc, iters=2, **sc.params(mapping))
        gpu.set_tuning(64, flags, 0, 16)
        for step in range(1, 4):
            log(f"bad state, flags {flags}, {mapping}, step {step}")
            gpu.update(1)
            orc.step(1)
            compare_pbf(gpu, orc, sc.n, step)
        gpu.close()


def _hip():
    """The HIP runtime that the library runs on."""
    capi.lib()
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))


def _memory():
    """Free and total device memory in bytes."""
    free, every = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(every)) == 0
    return free.value, every.value


def _used(make):
    """A new model and the device memory its creation took."""
    free = _memory()[0]
    m = make()
    return m, free - _memory()[0]


def test_default_lists_are_bounded_and_given_back():
    """The survivor lists of the default shape (1 KiB a particle): freed by a tuning without them and
    with the model, a 64th of the device's memory at most over all models."""
    n, lists = 1 << 18, 1 << 28

    def make():
        return capi.Fluids(n, 1000, (2.0, 1.0, 1.0), (20, 10, 10))
    m, took = _used(make)
    assert took > lists
    free = _memory()[0]
    m.set_tuning(64, capi.LAUNCH_QUAD, 0, 16)
    t = time.monotonic()  # freed memory may count as free a little later
    while _memory()[0] - free < lists and time.monotonic() - t < 2.0:
        time.sleep(0.01)
    assert _memory()[0] - free >= lists
    m.close()
    models = []
    while len(models) < 64:
        m, took = _used(make)
        models.append(m)
        if took < lists:
            break
    log(f"{len(models) - 1} models with default lists")
    assert took < lists and 1 < len(models) and (len(models) - 1) * lists <= _memory()[1] // 64
    models.pop(0).close()
    m, took = _used(make)
    assert took > lists
    for k in models + [m]:
        k.close()


def test_models_created_with_little_memory_free_walk_with_the_same_bits():
    sc = small_scene(seed=9)
    sc.max_n = 1 << 17
    free, every = _memory()
    if free < 0.6 * every:
        pytest.skip("another program holds the device's memory")

    def make():
        m = capi.Fluids(sc.max_n, sc.n, sc.box, sc.res, gravity=sc.gravity)
        m.set_params(**sc.params("stable"))
        return m
    with_lists, took = _used(make)
    assert took > sc.max_n * 1024
    hold = ctypes.c_void_p()
    assert _hip().hipMalloc(ctypes.byref(hold), ctypes.c_size_t(int(free - 0.49 * every))) == 0
    walks, took = _used(make)
    assert took < sc.max_n * 1024
    for m in (with_lists, walks):
        m.load_state(sc.pos, sc.vel)
        m.update(3)
    for a, b in zip(with_lists.read_state(), walks.read_state()):
        _eq(a, b, "state without lists")
    with_lists.close()
    walks.close()
    assert _hip().hipFree(hold) == 0
