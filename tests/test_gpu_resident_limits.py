"""The resident sweep at its limits: LDS that is nearly full, lattices much larger
than their systems, and calls of a few sweeps."""
import numpy as np
import pytest

import pscbfm_amd as P
from helpers import chains, make_updater, oracle_for, ordered_chains

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
