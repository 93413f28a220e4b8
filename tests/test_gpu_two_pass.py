"""The two-pass kernels on systems small enough to run resident: a stated launch
shape keeps them on two passes.  Eager launches, the allocation-free run, explicit
draws in graphs, and the accepted log from running totals, against the oracle."""
import numpy as np
import pytest

import oracle
import pscbfm_amd as P
from helpers import GOLDEN, chains, gpu_vs_oracle, make_updater, oracle_for, ordered_chains, stars

pytestmark = pytest.mark.gpu

KINDS = [P.LATTICE_BIT, P.LATTICE_U8]
SHAPES = [(256, 2), (64, 1)]
SEEDS = GOLDEN / "resultNormPscBFM.seeds"


def _r250_oracle(s, colors, substeps):
    r = oracle.R250.from_seed_file(SEEDS)
    r.rand32(), r.rand32()
    o = oracle_for(s, colors, 0)
    o.draws = r.substep_draws(substeps, int(colors.max()) + 1)
    return o, o.run(0, substeps)[1]


@pytest.mark.parametrize("block,slots", SHAPES)
@pytest.mark.parametrize("kind", KINDS)
def test_eager_launches_and_graphs_equal_the_oracle(kind, block, slots):
    s = chains((64, 64, 64), 40, 64, seed=11)
    for use_graph, parts in ((False, (1, 7, 16)), (True, (24,)), (True, (3, 21))):
        gx, glog, ox, olog = gpu_vs_oracle(s, seed=5, n_mcs=24, kind=kind, chunks=parts, use_graph=use_graph, block=block,
                                           slots=slots)
        assert np.array_equal(glog, olog) and np.array_equal(gx, ox)


@pytest.mark.parametrize("block,slots", SHAPES)
@pytest.mark.parametrize("kind", KINDS)
def test_runs_without_allocation(kind, block, slots):
    """Two systems in a row share the scratch; runs with and without a log continue one trajectory."""
    for s, seed, plan in ((chains((64, 64, 64), 40, 64, seed=11), 5, ((30, True), (3, False), (9, True))),
                          (chains((32, 32, 32), 12, 16, seed=4), 9, ((7, True), (2, True)))):
        u = make_updater(s, seed, kind, block=block, slots=slots)
        colors = u.colors(s.n)
        nc = int(colors.max()) + 1
        o, at = oracle_for(s, colors, seed), 0
        for m, log in plan:
            st, glog = u.runNoAlloc(m, log=log)
            _, olog = o.run(at, m * nc)
            at += m * nc
            assert st.accepted == int(olog.sum())
            if log:
                assert np.array_equal(glog, olog)
        assert np.array_equal(u.getPositions(s.n), o.xyz)
        u.cleanup()


@pytest.mark.parametrize("block,slots", SHAPES)
@pytest.mark.parametrize("kind", KINDS)
def test_explicit_draws_in_graphs_and_over_draw_chunks(kind, block, slots):
    """One table and tables of a few sweeps, in graphs of many substeps, eagerly
    and without allocation: log and coordinates are the oracle's."""
    s = chains((32, 32, 32), 20, 16, seed=7)
    for chunk, how in ((0, "graph"), (5, "graph"), (50, "graph"), (14, "eager"), (0, "noalloc")):
        u = make_updater(s, 42, kind, block=block, slots=slots)
        u.loadR250SeedFile(SEEDS, 2)
        u.setDrawChunk(chunk)
        colors = u.colors(s.n)
        logs = []
        for m in (23, 41):
            logs.append(u.runNoAlloc(m, log=True)[1] if how == "noalloc" else u.run(m, log=True, use_graph=how == "graph")[1])
        o, olog = _r250_oracle(s, colors, 64 * (int(colors.max()) + 1))
        assert np.array_equal(np.concatenate(logs), olog), (chunk, how)
        assert np.array_equal(u.getPositions(s.n), o.xyz), (chunk, how)
        u.cleanup()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("name", ["chains", "network", "automatic_shape"])
def test_log_over_bulk_graph_replays(name, kind):
    """More than two bulk graphs of 256 substeps and a rest, after unlogged runs
    and after another shape with more totals: every entry is the oracle's."""
    s = {"chains": lambda: chains((32, 64, 32), 60, 13, seed=8), "network": lambda: stars((64, 64, 64), 30, 4, 9, seed=2),
         "automatic_shape": lambda: ordered_chains((64, 64, 64), 4900, 2)}[name]()  # one size up from the resident ones
    u = make_updater(s, 21, kind)
    colors = u.colors(s.n)
    nc = int(colors.max()) + 1
    plan = [(4, (64, 1), False), (6, (256, 4), False), (640 // nc + 3, (128, 2), True), (5, (64, 1), False),
            (300 // nc, (256, 2), True)]
    o, at = oracle_for(s, colors, 21), 0
    for m, shape, log in plan:
        if name != "automatic_shape":
            u.setLaunchShape(*shape)
        st, glog = u.run(m, log=log)
        _, olog = o.run(at, m * nc)
        at += m * nc
        assert st.accepted == int(olog.sum())
        if log:
            assert glog.size == m * nc and np.array_equal(glog, olog)
    assert np.array_equal(u.getPositions(s.n), o.xyz)
    u.cleanup()
