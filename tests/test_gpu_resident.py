"""The resident sweep (one workgroup, many substeps per launch) against the CPU
oracle and the two-pass kernels, which setLaunchShape pins.

All results are whole numbers, so every comparison is exact.  Sizes are chosen
around the workgroup's rounds: a species of 64 and 65 members (one wave and
two), 1024 and 1025 (one round and two), 4864 and 4865 (the largest that runs
resident alone and the first that does not), and 5120 and 5121 (the same for
a batch replica)."""
import numpy as np
import pytest

import oracle
import pscbfm_amd as P
from helpers import GOLDEN, chains, make_updater, oracle_for, ordered_chains, stage_updater, stars

pytestmark = pytest.mark.gpu

KINDS = [P.LATTICE_BIT, P.LATTICE_U8]


def _dimers(box, n):
    """n ordered dimers: two species of exactly n members."""
    return ordered_chains(box, n, 2)


SYSTEMS = {
    "one_wave": lambda: _dimers((32, 32, 32), 64),
    "two_waves": lambda: _dimers((32, 32, 32), 65),
    "one_round": lambda: _dimers((64, 32, 32), 1024),
    "two_rounds": lambda: _dimers((64, 32, 32), 1025),
    "five_rounds": lambda: _dimers((64, 64, 64), 4864),
    "too_large": lambda: _dimers((64, 64, 64), 4865),
    "smallest_box": lambda: chains((8, 8, 8), 2, 5, seed=3),
    "flat_box": lambda: chains((64, 16, 8), 9, 21, seed=4),
    "network": lambda: stars((64, 64, 64), 60, 4, 7, seed=5),
    "eight_arms": lambda: stars((64, 32, 64), 40, 8, 6, seed=6),
    "lone_monomers": lambda: chains((32, 32, 32), 100, 1, seed=7),
}


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_resident_equals_oracle_and_two_pass(name, kind):
    s = SYSTEMS[name]()
    print(f"{name}: {s.n} monomers, kind {kind}", flush=True)
    cells = int(np.prod(s.box))
    seen = []
    for shape, spatial in (((0, 0), None), ((0, 0), True), ((0, 0), False), ((256, 2), None)):
        u = make_updater(s, 11, kind, block=shape[0], slots=shape[1], spatial=spatial)
        colors = u.colors(s.n)
        logs = [u.run(m, log=True)[1] for m in (1, 70, 3)]  # the second crosses 64 substeps
        seen.append((np.concatenate(logs), u.getPositions(s.n), u.downloadLattice(cells), u.proposalBits(),
                     u.counters()))
        u.cleanup()
    o = oracle_for(s, colors, 11)
    _, olog = o.run(0, 74 * (int(colors.max()) + 1))
    assert np.array_equal(seen[0][0], olog) and np.array_equal(seen[0][1], o.xyz)
    for other in seen[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(seen[0], other))


@pytest.mark.parametrize("kind", KINDS)
def test_both_paths_continue_each_other(kind):
    """Resident, two-pass and eager runs of one handle follow one trajectory:
    each leaves the buffers the other expects, whatever the substeps' parity."""
    s = chains((32, 64, 32), 60, 13, seed=8)
    u = make_updater(s, 21, kind)
    colors = u.colors(s.n)
    nc = int(colors.max()) + 1
    logs = []
    plan = [(3, (0, 0), False), (2, (128, 1), False), (1, (0, 0), False), (4, (0, 0), True), (2, (256, 2), False),
            (5, (0, 0), False)]
    for m, shape, profile in plan:
        u.setLaunchShape(*shape)
        logs.append(u.run(m, log=True, profile=profile)[1])
        u.setLaunchShape(0, 0)
    o = oracle_for(s, colors, 21)
    _, olog = o.run(0, 17 * nc)
    assert np.array_equal(np.concatenate(logs), olog)
    assert np.array_equal(u.getPositions(s.n), o.xyz)
    u.cleanup()


def test_r250_draws_and_the_launch_limit():
    """Explicit draws, and a run longer than one launch covers."""
    s = chains((32, 32, 32), 20, 16, seed=9)
    u = make_updater(s, 1)
    u.loadR250SeedFile(GOLDEN / "resultNormPscBFM.seeds", 2)
    u.setDrawChunk(300)
    colors = u.colors(s.n)
    nc = int(colors.max()) + 1
    mcs = 4200 // nc + 1
    _, log = u.run(mcs, log=True)
    r = oracle.R250.from_seed_file(GOLDEN / "resultNormPscBFM.seeds")
    r.rand32(), r.rand32()
    o = oracle_for(s, colors, 0)
    o.draws = r.substep_draws(mcs * nc, nc)
    _, olog = o.run(0, mcs * nc)
    assert np.array_equal(log, olog) and np.array_equal(u.getPositions(s.n), o.xyz)
    u.cleanup()

    v = make_updater(s, 5)
    w = make_updater(s, 5, block=256, slots=2)
    (sv, _), (sw, _) = v.run(4200), w.run(4200)
    assert (sv.accepted, sv.attempted, sv.substeps) == (sw.accepted, sw.attempted, sw.substeps)
    assert sv.substeps > 4096 and np.array_equal(v.getPositions(s.n), w.getPositions(s.n))
    v.cleanup()
    w.cleanup()


def test_tuned_small_system_stays_exact():
    """The autotuner's choice does not pin a small system to the two-pass kernels' results only."""
    s = chains((32, 32, 32), 24, 16, seed=10)
    a, b = make_updater(s, 3), make_updater(s, 3, block=64, slots=1)
    a.autotune(2)
    a.run(20)
    b.run(20)
    assert np.array_equal(a.getPositions(s.n), b.getPositions(s.n))
    a.cleanup()
    b.cleanup()


def _batch_systems():
    """Replicas of every path: resident always (up to 5120 members), resident
    only beside long two-pass work (beyond), too large for LDS, and one whose
    monomers without bonds the resident sweep does not take."""
    return [chains((32, 32, 32), 24, 16, seed=1), _dimers((64, 64, 64), 5120), _dimers((64, 64, 64), 5121), ordered_chains((64, 64, 64), 800, 16),
            stars((64, 64, 32), 30, 4, 9, seed=2), chains((128, 64, 128), 100, 50, seed=3),
            chains((32, 32, 32), 80, 1, seed=4), chains((16, 64, 32), 30, 11, seed=5),
            chains((128, 128, 64), 20, 40, seed=6)]


@pytest.mark.parametrize("kind", KINDS)
def test_batch_paths_equal_runs_alone(kind):
    systems = _batch_systems()
    batch = P.Batch(0, len(systems), kind)
    ids = [batch.add(stage_updater(s, 30 + i, kind)) for i, s in enumerate(systems)]
    for m, block in ((5, 0), (3, 128), (66, 0), (2, 64)):  # automatic paths, then all on two passes, twice
        batch.set_perform_block(block)
        batch.run(m)
    batch.remove(ids[0])
    batch.set_perform_block(0)
    batch.run(4)
    for i, (rid, s) in enumerate(zip(ids, systems)):
        if i == 0:
            continue
        u = make_updater(s, 30 + i, kind, block=256, slots=2)
        st, _ = u.run(80)
        assert np.array_equal(batch.positions(rid, s.n), u.getPositions(s.n)), i
        assert batch.info(rid).accepted == st.accepted and batch.info(rid).substeps == u.counters()[0]
        u.cleanup()


def test_batch_with_more_replicas_than_compute_units():
    """Small replicas share compute units in small workgroups beside full ones."""
    small = chains((16, 16, 16), 4, 12, seed=1)
    large = ordered_chains((64, 64, 64), 150, 16)
    staged = [(small, 100 + i) for i in range(270)] + [(large, 50), (large, 51)]
    batch = P.Batch(0, len(staged))
    ids = [batch.add(stage_updater(s, seed)) for s, seed in staged]
    batch.run(9)
    for k in (0, 1, 135, 269, 270, 271):
        s, seed = staged[k]
        u = make_updater(s, seed, block=64, slots=1)
        u.run(9)
        assert np.array_equal(batch.positions(ids[k], s.n), u.getPositions(s.n)), k
        u.cleanup()


@pytest.mark.parametrize("kind", KINDS)
def test_batch_pass_two_wider_and_narrower_than_its_lists(kind):
    """Pass-2 workgroups of 64 to 256 threads over lists of 64 and of 512 entries, filled past the first round."""
    s = ordered_chains((64, 64, 64), 800, 16)
    u = make_updater(s, 9, kind, block=256, slots=2)
    u.run(12)
    for block, slots, perform in ((64, 1, 256), (64, 1, 64), (256, 2, 64), (256, 2, 256)):
        batch = P.Batch(0, 2, kind, block, slots)
        rid = batch.add(stage_updater(s, 9, kind))
        batch.set_perform_block(perform)
        batch.run(12)
        assert np.array_equal(batch.positions(rid, s.n), u.getPositions(s.n)), (block, slots, perform)
    u.cleanup()


def test_batch_after_a_large_replica_leaves():
    """The tiles that stay close up: results do not depend on where they were."""
    large, small = ordered_chains((128, 128, 128), 3000, 32), [chains((128, 64, 128), 100, 50, seed=k) for k in (3, 4)]
    batch = P.Batch(0, 3)
    ids = [batch.add(stage_updater(s, 60 + i)) for i, s in enumerate([small[0], large, small[1]])]
    batch.run(5)
    batch.remove(ids[1])
    batch.run(7)
    for rid, s, seed in ((ids[0], small[0], 60), (ids[2], small[1], 62)):
        u = make_updater(s, seed)
        st, _ = u.run(12)
        assert np.array_equal(batch.positions(rid, s.n), u.getPositions(s.n))
        assert batch.info(rid).accepted == st.accepted
        u.cleanup()
