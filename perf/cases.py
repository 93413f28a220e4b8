"""Performance cases of the scBFM sweep: what its users have it do.

A pass is one call of the simulation loop's body: advance a system (or a
batch, or a stream of jobs) by its save interval and take the coordinates, as
the command-line simulator, the replica runs and the request loop do.  The
systems are this repository's own workloads (linear-chain melts, crosslinked
stars, the replica mix) from a few hundred monomers to the 512^3 melt.

Every output is a whole number (coordinates, accepted counts), defined bit
for bit by the input and the draws, so there is no rounding to measure and
`exact` has no values to give.
"""
from __future__ import annotations

import numpy as np

import pscbfm_amd as P
from pscbfm_amd import workloads as W

LATTICES = {"bit": P.LATTICE_BIT, "u8": P.LATTICE_U8}

# Sweeps that take an ordered packing to a melt before anything is timed.
RELAX_MCS = 1000

# Integer operations of one attempted move: two 6-step hashes, the direction,
# the target and its nine-cell front plane, and (each) a bond lookup.
OPS_PER_MOVE = 60
OPS_PER_BOND = 8

# Typical acceptance of a move, for the bytes an accepted one writes.
ACCEPTANCE = 0.15

# Largest drawn system and monomer-sweeps: those of the 512^3 melt.
MAX_MONOMER_SWEEPS = 32768 * 256 * 1000


def chains(name, box, length, phi, lattice, mcs, ordered, draws="counter", log=False):
    return {"name": name, "kind": "chains", "x": box[0], "y": box[1], "z": box[2], "length": length, "phi": phi,
            "lattice": lattice, "mcs": mcs, "ordered": ordered, "draws": draws, "log": log}


def listed():
    return [
        # a first short call on a small system, as a test or an interactive
        # session makes: launches and host work count, not throughput
        chains("chains_32_short", (32, 32, 32), 16, 0.094, "bit", 100, False),
        # a small hydrogel on the reference's own draw stream, in its byte
        # lattice
        {"name": "stars_64_r250_u8", "kind": "stars", "x": 64, "y": 64, "z": 64, "stars": 29, "arm": 5,
         "lattice": "u8", "mcs": 500, "draws": "r250"},
        # a single-chain-dynamics run: a moderate box, an odd chain length
        chains("chains_64", (64, 64, 64), 37, 0.3, "bit", 1000, False),
        # a film in a non-cubic box, byte lattice, with its per-substep log
        chains("film_256x128x64_u8", (256, 128, 64), 100, 0.25, "u8", 500, False, log=True),
        # the usual melt of a production study on one card
        chains("melt_128", (128, 128, 128), 64, 0.5, "bit", 1000, True),
        # the larger melt in the reference's byte lattice
        chains("melt_256_u8", (256, 256, 256), 128, 0.5, "u8", 500, True),
        # frequent snapshots: 20 sweeps between reads of a million coordinates
        chains("melt_256_snapshots", (256, 256, 256), 128, 0.5, "bit", 20, True),
        # the headline melt, 8.39 million monomers
        chains("melt_512", (512, 512, 512), 256, 0.5, "bit", 1000, True),
        # the dense star network: branched, four species, 1.5 million monomers
        {"name": "network_256", "kind": "network", "x": 256, "y": 256, "z": 256, "stars": 12800, "arm": 29,
         "lattice": "bit", "mcs": 1000},
        # an ensemble of independent systems in one batch
        {"name": "batch_mix_256", "kind": "batch", "replicas": 256, "edges": "32,64,128", "mix": 42,
         "lattice": "bit", "mcs": 2000},
        # an ensemble of small systems in the byte lattice
        {"name": "batch_small_u8", "kind": "batch", "replicas": 96, "edges": "32,64", "mix": 7,
         "lattice": "u8", "mcs": 1000},
        # requests served: staged systems submitted at once, results collected
        {"name": "serve_48", "kind": "serve", "replicas": 48, "edges": "32,64,128", "mix": 11,
         "lattice": "bit", "mcs": 1000},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["chains", "chains", "chains", "stars", "batch", "serve"])
    lattice = rng.choice(["bit", "bit", "u8"])
    if kind == "chains":
        box = [2 ** rng.randint(5, 8) for _ in range(3)]
        if rng.random() < 0.25:
            box = [2 ** rng.randint(7, 9) for _ in range(3)]
        ordered = rng.random() < 0.5
        phi = 0.5 if ordered else round(rng.uniform(0.05, 0.4), 3)
        length = rng.choice([16, 32, 64, 128]) if ordered else _log_uniform(rng, 5, 256)
        monomers = phi * box[0] * box[1] * box[2] / 8
        mcs = max(1, min(_log_uniform(rng, 20, 1000), int(MAX_MONOMER_SWEEPS / monomers)))
        c = chains("", box, length, phi, lattice, mcs, ordered, rng.choice(["counter", "counter", "r250"]),
                   rng.random() < 0.3)
        del c["name"]
        return c
    if kind == "stars":
        edge = 2 ** rng.randint(6, 7)
        return {"kind": "stars", "x": edge, "y": edge, "z": 2 ** rng.randint(6, 7), "stars": _log_uniform(rng, 10, 200),
                "arm": rng.randint(3, 30), "lattice": lattice, "mcs": _log_uniform(rng, 50, 1000),
                "draws": rng.choice(["counter", "r250"])}
    return {"kind": kind, "replicas": _log_uniform(rng, 4, 256) if kind == "batch" else _log_uniform(rng, 4, 60),
            "edges": rng.choice(["32,64", "32,64,128"]), "mix": rng.randrange(1 << 20), "lattice": lattice,
            "mcs": _log_uniform(rng, 100, 1000)}


def _chain_count(case):
    return max(1, int(case["phi"] * case["x"] * case["y"] * case["z"] / (8 * case["length"])))


def _specs(case, seed):
    """The replica mix of the case, its growth and sweep seeds from `seed`."""
    edges = tuple(int(e) for e in case["edges"].split(","))
    specs = W.replica_specs(case["replicas"], case["mix"], edges)
    rng = np.random.default_rng([seed, case["mix"]])
    for s in specs:
        s.seed = int(rng.integers(1, 2 ** 63))
    return specs


def _chain_system(case, seed):
    box = (case["x"], case["y"], case["z"])
    n_chains, length = _chain_count(case), case["length"]
    if case["ordered"]:
        xyz = P.gen_linear_chains_ordered(box, n_chains, length)
    else:
        xyz = W.build_chains(W.ReplicaSpec(box, length, case["phi"], n_chains, seed)).xyz
    # both directions of every bond, grouped by monomer
    ids = np.arange(n_chains * length, dtype=np.uint32).reshape(n_chains, length)
    pairs = np.empty((n_chains, 2 * (length - 1), 2), dtype=np.uint32)
    pairs[:, 0::2, 0] = ids[:, :-1]
    pairs[:, 0::2, 1] = ids[:, 1:]
    pairs[:, 1::2, 0] = ids[:, 1:]
    pairs[:, 1::2, 1] = ids[:, :-1]
    return box, xyz, pairs.reshape(-1, 2)


def _updater(case, seed, box, xyz, pairs):
    """An initialized updater, in the call order of the C++ class's users."""
    u = P.UpdaterGPUScBFM_AB_Type()
    u.setGpu(0)
    u.setPeriodicity(True, True, True)
    u.setNrOfAllMonomers(len(xyz))
    u.setMonomerCoordinatesBulk(xyz)
    u.setConnectivityBulk(pairs)
    u.setLatticeSize(*box)
    forbidden = W.standard_forbidden()
    for dx in range(-4, 4):
        for dy in range(-4, 4):
            for dz in range(-4, 4):
                u.copyBondSet(dx, dy, dz, bool(forbidden[(dx & 7) | ((dy & 7) << 3) | ((dz & 7) << 6)]))
    u.setSeed(seed)
    u.setLatticeKind(LATTICES[case["lattice"]])
    u.setCheckOnInitialize(False)
    u.initialize()
    return u


def prepare(case, seed):
    if case["kind"] in ("batch", "serve"):
        kind = LATTICES[case["lattice"]]
        staged = [W.stage(r, kind) for r in W.build_replicas(_specs(case, seed))]
        counts = [s.n_monomers for s in _specs(case, seed)]
        state = {"case": case, "staged": staged, "counts": counts}
        if case["kind"] == "serve":
            state["server"] = P.Server(hbm_budget=64 << 30, tile_capacity=1 << 14, replica_capacity=256,
                                       lattice_kind=kind)
        else:
            state["batch"] = P.Batch(0, len(staged), kind)
            state["ids"] = [state["batch"].add(u) for u in staged]
        return state
    if case["kind"] == "network":
        sd = W.dense_network(seed, W.relax_on_gpu(LATTICES[case["lattice"]]), (case["x"], case["y"], case["z"]),
                             case["stars"], case["arm"])
        u = W.stage(sd, LATTICES[case["lattice"]], initialize=True)
        return {"case": case, "updater": u, "n": sd.n}
    if case["kind"] == "stars":
        box = (case["x"], case["y"], case["z"])
        xyz, bonds = P.gen_star_network(box, case["stars"], 4, case["arm"], seed)
        pairs = W.directed_pairs(len(xyz), bonds)
    else:
        box, xyz, pairs = _chain_system(case, seed)
    u = _updater(case, seed, box, xyz, pairs)
    if case.get("ordered"):
        u.setReadBack(False)
        u.runSimulationOnGPU(RELAX_MCS)
        u.setReadBack(True)
    if case.get("draws") == "r250":
        u.setR250State(np.random.default_rng(seed).integers(0, 1 << 32, 250, dtype=np.uint32))
    return {"case": case, "updater": u, "n": len(xyz)}


def run(state):
    case = state["case"]
    if case["kind"] == "serve":
        server = state["server"]
        jobs = [server.submit(u, case["mcs"]) for u in state["staged"]]
        out = []
        for job, n in zip(jobs, state["counts"]):
            server.wait(job)
            out.append(server.result(job, n))
            server.release(job)
        return out
    if case["kind"] == "batch":
        batch, ids = state["batch"], state["ids"]
        batch.run(case["mcs"])
        xyz = batch.positions_many(ids, state["counts"])
        accepted = np.array([batch.info(i).accepted for i in ids], dtype=np.int64)
        return [np.concatenate(xyz), accepted]
    u = state["updater"]
    if case.get("log"):
        stats, log = u.run(case["mcs"], log=True)
        return [u.getPositions(state["n"]), stats.accepted, log.astype(np.int64)]
    u.runSimulationOnGPU(case["mcs"])
    return [u.getPositions(state["n"]), u.lastRunStats().accepted]


def work(case):
    """Bytes and integer operations of one pass.  An attempted move reads its
    monomer's code, its partners' numbers and codes and nine lattice cells; an
    accepted one writes its code and two cells; the coordinates are written
    once."""
    if case["kind"] in ("batch", "serve"):
        n = sum(s.n_monomers for s in _specs(case, 0))
        bonds = 2.0
    elif case["kind"] == "chains":
        n = _chain_count(case) * case["length"]
        bonds = 2.0 * (case["length"] - 1) / case["length"]
    else:
        n = case["stars"] * (1 + 4 * case["arm"])
        bonds = 2.0
    cell = 1.0 if case["lattice"] == "u8" else 0.125
    moves = float(n) * case["mcs"]
    per_move = 4 + 8 * bonds + 9 * cell + ACCEPTANCE * (4 + 2 * cell)
    return {"bytes": moves * per_move + 12.0 * n, "flops": moves * (OPS_PER_MOVE + OPS_PER_BOND * bonds)}


def exact(case, seed):
    """Outputs are whole numbers: no rounding, so no value in more bits."""
    return None
