"""The resident sweep at its limits: LDS that is nearly full, lattices much larger
than their systems, calls of a few sweeps, and batches of every build."""
import numpy as np
import pytest

import pscbfm_amd as P
from helpers import Sys, chains, make_updater, oracle_for, ordered_chains, stage_updater, stars

pytestmark = pytest.mark.gpu

KINDS = [P.LATTICE_BIT, P.LATTICE_U8]

# 131072 bytes of LDS for the two lattices of 128 x 64 x 64, 4 per slot for up to
# 7400 monomers, and 2240 of tables: 161 of 160 * 1024 bytes at 3700 dimers.
SYSTEMS = {
    "chain_in_a_large_box": lambda: chains((128, 64, 64), 1, 128, seed=3),
    "monomer_pair_in_a_large_box": lambda: chains((64, 64, 128), 1, 2, seed=4),
    "nearly_full_lds": lambda: ordered_chains((128, 64, 64), 3700, 2),
    "smallest_box": lambda: chains((8, 8, 8), 1, 2, seed=5),
    "flat_box": lambda: chains((8, 512, 8), 12, 15, seed=6),
}


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_short_calls_equal_the_oracle(name, kind):
    s = SYSTEMS[name]()
    print(f"{name}: {s.n} monomers, kind {kind}", flush=True)
    u = make_updater(s, 17, kind)
    colors = u.colors(s.n)
    logs = [u.run(m, log=True)[1] for m in (1, 2, 10, 1)]
    x, lattice = u.getPositions(s.n), u.downloadLattice(int(np.prod(s.box)))
    steps = sum(map(len, logs))
    bits = u.proposalBits()
    u.cleanup()
    o = oracle_for(s, colors, 17)
    _, olog = o.run(0, steps)
    assert np.array_equal(np.concatenate(logs), olog) and np.array_equal(x, o.xyz)
    want = np.zeros(lattice.size, lattice.dtype)
    want[[P.zcurve_encode(s.box, *c) for c in x % np.array(s.box)]] = 1
    assert np.array_equal(lattice, want)
    assert bits[steps & 1] == 0 and bits[(steps - 1) & 1] >= olog[-1]


@pytest.mark.parametrize("kind", KINDS)
def test_one_sweep_in_a_large_box_takes_no_longer_than_two_passes(kind):
    """A launch loads and stores the whole lattice.  One load at a time, by the
    one wave that a chain needs, took 2.4 (bit) and 4 (byte lattice) times the two
    passes of a sweep; the bound of 1.5 leaves the measurement's spread to it."""
    s = SYSTEMS["chain_in_a_large_box"]()
    ms = {}
    for shape in ((0, 0), (64, 1)):
        u = make_updater(s, 5, kind, block=shape[0], slots=shape[1])
        ms[shape] = min(u.run(1)[0].gpu_ms for _ in range(30))
        u.cleanup()
    print({k: f"{v * 1e3:.1f} us" for k, v in ms.items()}, flush=True)
    assert ms[(0, 0)] < 1.5 * ms[(64, 1)]


def _branched(n):
    """n dimers, closely packed in part of 64^3, with one monomer bonded to its six
    neighbours in the packing: degrees 1, 2 and 6."""
    s = ordered_chains((64, 64, 64), 32 * 32 * 21 // 2, 2)
    s = Sys(s.box, s.xyz[:2 * n], P.chain_bonds(n, 2))
    at = {tuple(c): i for i, c in enumerate(s.xyz % 64)}
    bonded = {frozenset(b) for b in s.bonds.tolist()}
    steps = [(2, 0, 0), (-2, 0, 0), (0, 2, 0), (0, -2, 0), (0, 0, 3), (0, 0, -3)]
    for i, c in enumerate(s.xyz % 64):
        near = [at.get(tuple((c + d) % 64)) for d in steps]
        if None not in near:
            extra = [(i, j) for j in near if frozenset((i, j)) not in bonded]
            return Sys(s.box, s.xyz, np.concatenate([s.bonds, np.array(extra, s.bonds.dtype)]))
    raise AssertionError("no monomer with six neighbours")


def _builds():
    """Replicas of every resident build of a batch (up to 4096, 5120 and 8192
    members; up to two, four and eight bonds), some only resident beside long
    two-pass work, and that work; the last stays on two passes beside it."""
    return [chains((32, 32, 32), 24, 16, seed=1), ordered_chains((64, 64, 64), 4097, 2),
            ordered_chains((64, 64, 64), 5200, 2), stars((64, 64, 64), 60, 4, 7, seed=5),
            stars((64, 64, 64), 380, 4, 9, seed=1), stars((64, 64, 64), 430, 4, 9, seed=1),
            stars((64, 32, 64), 40, 8, 6, seed=6), _branched(4200), _branched(6000),
            ordered_chains((256, 256, 128), 100000, 2)]


@pytest.mark.parametrize("kind", KINDS)
def test_batch_of_every_build_equals_runs_alone(kind):
    systems = _builds()
    batch = P.Batch(0, len(systems), kind)
    ids = [batch.add(stage_updater(s, 40 + i, kind)) for i, s in enumerate(systems)]
    for m in (1, 40):
        batch.run(m)
    for i, (rid, s) in enumerate(zip(ids, systems)):
        u = make_updater(s, 40 + i, kind, block=256, slots=2)
        st, _ = u.run(41)
        assert np.array_equal(batch.positions(rid, s.n), u.getPositions(s.n)), i
        assert batch.info(rid).accepted == st.accepted, i
        u.cleanup()


@pytest.mark.parametrize("kind", KINDS)
def test_a_branched_replica_does_not_slow_the_others(kind):
    """Eight replicas of 5000 members, alone and beside a small star of eight
    arms.  With one build for all of them the star doubled the time of a sweep;
    beside it, on a compute unit of its own, it costs nothing, and the bound
    of 1.3 leaves the measurement's spread to it."""
    large, star = ordered_chains((64, 64, 64), 5000, 2), stars((32, 32, 32), 5, 8, 7, 1)
    ms = []
    for systems in ([large] * 8, [large] * 8 + [star]):
        batch = P.Batch(0, len(systems), kind)
        for i, s in enumerate(systems):
            batch.add(stage_updater(s, 7 + i, kind))
        batch.run(20)
        ms.append(min(batch.run(100) for _ in range(8)))
    print([f"{v * 10:.2f} us per sweep" for v in ms], flush=True)
    assert ms[1] < 1.3 * ms[0]
