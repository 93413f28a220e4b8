// gfx950 kernels of the colored two-pass scBFM sweep.
//
// Pass 1 (check):   CRITICAL.cu:298-374  kernelSimulationScBFMCheckSpecies
// Pass 2 (perform): CRITICAL.cu:376-411  kernelSimulationScBFMPerformSpeciesAndApply
// Proposal clear:   CRITICAL.cu:561-573  (here folded into pass 1 or 2, other parity)
//
// Design (wave64, CDNA4):
//  * positions are Z-curve codes, so the own lattice cell is the code itself
//    and every neighbouring cell is a masked add on one axis' bits;
//  * the forbidden-bond table is a 512-bit mask in LDS, indexed by the
//    Z-order bond key of two codes;
//  * both passes are bound by the lines their gathers touch and, up to some
//    hundred thousand members, by dependent round trips, more than by bandwidth:
//    a pass-1 thread handles SLOTS monomers and issues their loads in batches
//    (own codes, draw keys and partner ids; then partner codes and the front
//    plane, or the plane after the bond test: kBondsFirst); the 3x3 front plane
//    is read as at most four 64-bit words;
//  * a species' slots may be in the Z-curve order of the starting corners,
//    so that a wave's members and their partners and lattice words lie
//    close together; each slot's key is the inner move hash of the member's
//    rank in the reference's order, which keys its draw either way;
//  * pass 1 compacts the surviving proposals of its workgroup into a list
//    (wave ballot + LDS counter; the order inside a list is irrelevant
//    because the result of a substep does not depend on processing order),
//    and pass 2 walks those lists densely;
//  * the proposal lattice is 1 bit per cell and double-buffered by substep
//    parity: pass 1 of substep t sets bits in buffer t&1, pass 2 of substep t
//    reads it, and pass 1 or pass 2 of substep t zeroes buffer (t+1)&1 (last
//    read by pass 2 of substep t-1, next written by pass 1 of substep t+1);
//  * the occupancy lattice is updated with plain byte stores (no atomics):
//    device-scope atomics are executed beyond the per-XCD L2 and cost a
//    memory transaction each;
//  * workgroup w runs on XCD w%8: a single system renumbers workgroups so
//    each XCD takes one contiguous eighth of the species; a batch's tile
//    table keeps a small replica's workgroups on one XCD and spreads a large
//    one over all eight;
//  * the species and kernel seed of a substep come from the device state:
//    the counter draw of (seed, substep), or an explicit draw table (R250
//    mode), so launches carry no per-substep host data.
#include "kernels.h"
#include "sweep_device.h"

namespace pscbfm {

namespace {

// Logical workgroup id: consecutive ids on the same XCD.
__device__ __forceinline__ uint32_t xcd_block(uint32_t nb) {  // nb: a multiple of 8 (grid_for)
    return (blockIdx.x & 7u) * (nb >> 3) + (blockIdx.x >> 3);
}

// A list entry as one 64-bit word: low = species-local index | direction
// << kDirShift, high = old code.
__device__ __forceinline__ uint64_t pack_entry(uint32_t x, uint32_t y) { return uint64_t(x) | (uint64_t(y) << 32); }

// List entry: x = species-local index | direction << 29, y = old code.
constexpr uint32_t kDirShift = 29;

// Zeroes slice lb of nb of the proposal buffer of the other parity, 16 bytes
// per thread and step: pass 2 of substep t-1 was its last reader and pass 1
// of substep t+1 is its next writer, so either pass of substep t may do it
// (LaunchShape::clearPass).  In pass 1 the stores go out ahead of its loads
// and stream while its waves wait on them and compute the bond test; in
// pass 2 they overlap the list walk.
__device__ __forceinline__ void clear_other_parity(const SysDesc& d, uint64_t t, uint32_t lb, uint32_t nb) {
    const gptr<uint64_t> prev = (gptr<uint64_t>)(d.proposal.global() + size_t((t + 1u) & 1u) * d.latWords);
    const uint32_t quads = d.latWords >> 2;
    const uint32_t per = (quads + nb - 1) / nb;
    const uint32_t q0 = lb * per;
    const uint32_t q1 = min(q0 + per, quads);
    for (uint32_t q = q0 + threadIdx.x; q < q1; q += blockDim.x) {
        prev[2 * size_t(q)] = 0u;
        prev[2 * size_t(q) + 1] = 0u;
    }
}

// Pass 1 of substep t for logical workgroup lb of nb of one system.  The
// survivors go to `list` (capacity SLOTS * blockDim), their number to *count.
// With `clear` it also zeroes slice lb of nb of the other parity's proposals.
// What bounds it, 512^3 melt (2 x 4.2 million members): lines that its loads
// touch, about 230 per 64 members at one a cycle and compute unit, and vector
// issue behind that.  A quarter fewer vector instructions (move geometry from LDS
// tables) left 38.1 us per substep at 38.3, and fewer, wider loads were slower
// because a lane's neighbours then held other members: two consecutive members
// per lane 41.0, exchanged between half waves 39.7, key and partners side by side
// in one record 38.5 (dense star network 11.2 against 10.65).
// KEYED: the system's slots are in spatial order and each slot's draw key is
// read from its `key` piece; else the key is the hash of the slot index.  A
// compile-time choice: as a runtime branch between the load and the hash
// inside the load batch, the compiler's wait for the loaded key also lands on
// the hashing path, which then waits for every load issued before it.
struct CheckLds {
    uint32_t forbidden[16];
    uint32_t count;
};

template <int LAT, int SLOTS, int MAXDEG, bool KEYED>
__device__ __forceinline__ void check_body(const SysDesc& d, uint64_t t, SubstepDraw draw, uint32_t lb, uint32_t nb,
                                           bool clear, gptr<uint64_t> list, gptr<uint32_t> count,
                                           CheckLds& lds) {
    if (clear) clear_other_parity(d, t, lb, nb);
    const ColorInfo ci = load_color(d.colors.global(), draw.species);
    const gptr<uint32_t> proposal = d.proposal.global();

    // The bond table goes to LDS after the gathers below are issued, and the
    // barrier that publishes it stands in front of the bond test.  A barrier
    // ahead of the gathers held every wave's loads back by the table's round
    // trip.  Its words are loaded by a lane each, before the gathers: as scalar
    // loads they were moved down to where one lane stored them, and the barrier
    // waited for them there (us per substep, 128^3 melt 6.2 and 6.1, 256^3 uint8
    // 12.4 and 12.2).
    uint32_t forbidden = 0;
    if (threadIdx.x < 16u) forbidden = d.bondMask.global()[threadIdx.x];

    const uint32_t B = blockDim.x;
    const uint32_t base = lb * (SLOTS * B);
    const gptr<const uint32_t> posAll = (gptr<const uint32_t>)d.pos.global();
    const gptr<const uint32_t> pos = posAll + ci.slotOffset;
    const gptr<const uint32_t> nbr = d.nbr.global();
    // Inner hash of each member's species-local index in the reference's
    // order, the key of its draw: read from the slot's key when the slots
    // are in spatial order, else the hash of the slot index itself.
    const gptr<const uint32_t> keys = d.key.global() + ci.slotOffset;
    // Partner ids: the bit-lattice kernel reads the full matrix rows; the
    // uint8-lattice kernel, whose plane words cost more traffic, reads the
    // 16-bit codes (half the bytes) and the full matrix only for escapes.
    const gptr<const uint32_t> ids = d.ids.global() + ci.idsOffset;
    uint32_t rb[MAXDEG];
#pragma unroll
    for (int r = 0; r < MAXDEG; ++r)
        rb[r] = LAT == kLatticeU8 ? ((cptr<uint32_t>)d.rowBase.global())[draw.species * kMaxConnectivity + uint32_t(r)] : 0u;
    const gptr<const uint64_t> lattice = (gptr<const uint64_t>)d.lattice.global();
    const AxisMasks masks = axis_masks(d);

    // The load phase is branch-free: lanes without a monomer load the first
    // one's and discard it, and a monomer with fewer bonds than others tests its
    // first one again, so every load of a thread sits in one basic block and all
    // of them are in flight together.  Offsets are 32-bit: a monomer takes eight
    // of at most 2^32 cells.  (With a "no partner" choice per row and 64-bit indices the 512^3 melt
    // took 38.6 us per substep against 38.1, the uint8 film 6.28 against 6.21.)
    // First batch of loads: own codes and partner ids.
    uint32_t j[SLOTS], m[SLOTS], hj[SLOTS], partner[SLOTS][MAXDEG];
    bool live[SLOTS], free[SLOTS];  // free: no bond to test
    gptr<const uint32_t> row[MAXDEG];
#pragma unroll
    for (int r = 0; r < MAXDEG; ++r)  // past the species' rows: the first one again
        row[r] = ci.maxDegree == 0u ? pos : nbr + ci.nbrOffset + (uint32_t(r) < ci.maxDegree ? size_t(r) * ci.nbrPitch : 0u);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        j[s] = base + uint32_t(s) * B + threadIdx.x;
        live[s] = j[s] < ci.count;
        const uint32_t jj = live[s] ? j[s] : 0u;  // count > 0 for every species
        m[s] = at(pos, 4u * jj);
        if constexpr (KEYED)
            hj[s] = at(keys, 4u * jj);
        else
            hj[s] = move_hash(jj);
        if constexpr (LAT == kLatticeU8) {
#pragma unroll
            for (int q = 0; q < MAXDEG / 2; ++q) {
                const bool have = uint32_t(q) < ci.idWords;  // the same for every lane
                const uint32_t w = ids[have ? size_t(jj) * ci.idWords + uint32_t(q) : 0u];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int r = 2 * q + h;
                    const int32_t v = int32_t(int16_t(uint16_t(h ? (w >> 16) : (w & 0xFFFFu))));
                    uint32_t id = rb[r] + jj + uint32_t(v);
                    // an escape is read only for a real row of this species, so the index stays in its matrix
                    if (have && v == kIdEscape && uint32_t(r) < ci.maxDegree)
                        id = nbr[ci.nbrOffset + size_t(r) * ci.nbrPitch + jj];
                    const bool has = have && v != kIdNone && uint32_t(r) < ci.maxDegree;
                    if (r == 0) {
                        free[s] = !has;
                        partner[s][r] = id;
                    } else {
                        partner[s][r] = has ? id : partner[s][0];
                    }
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < MAXDEG; ++r) partner[s][r] = at(row[r], 4u * jj);
            free[s] = ci.maxDegree == 0u || partner[s][0] == kNoNeighbor;
        }
    }
    // Second batch: partner codes and the front plane.  CRITICAL.cu:322-323: the
    // draw is keyed by the species-local index in the reference's order.
    // The plane words of moves that fail the bond test are not needed.  It pays
    // to wait for the test and read them for the others only on the byte lattice
    // (eight times the plane bytes), with more than two bonds (more moves fail)
    // and with several members per thread (large systems); else, a chain of round
    // trips being all that counts, the reads go out with the partners'.  us per
    // substep, together against bonds first: 256^3 melt, uint8 13.9 against 13.2;
    // dense star network 10.9 against 10.6; 512^3 melt, bit 38.3 against 38.0; 128^3
    // melt 5.84 against 6.08.
    constexpr bool kBondsFirst = LAT == kLatticeU8 || MAXDEG > 2 || SLOTS > 1;
    constexpr int kShift = LAT == kLatticeU8 ? 3 : 6;
    uint32_t partnerCode[SLOTS][MAXDEG];
    Dir dir[SLOTS];
    Move mv[SLOTS];
    PlaneWords front[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        dir[s] = dir_of_hash(move_hash(hj[s] ^ draw.seed));
        mv[s] = make_move<kShift>(m[s], dir[s], masks);
#pragma unroll
        for (int r = 0; r < MAXDEG; ++r)
            partnerCode[s][r] = at(posAll, 4u * min(partner[s][r], d.nSlots - 1u));  // a valid slot whatever was read
        if constexpr (!kBondsFirst) front[s] = plane_words(lattice, mv[s]);
    }
    if (threadIdx.x < 16u) lds.forbidden[threadIdx.x] = forbidden;
    if (threadIdx.x == 0) lds.count = 0;
    __syncthreads();
    bool ok[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        uint32_t bad = 0;
#pragma unroll
        for (int r = 0; r < MAXDEG; ++r) {
            const uint32_t key = bond_key(partnerCode[s][r], mv[s].to);
            // With the plane words still to come, the first bond's test is best left to the
            // lanes that have one (us per substep, dense star network 10.67 and 10.59).
            if (!kBondsFirst || r > 0 || !free[s]) bad |= lds.forbidden[key >> 5] >> (key & 31u);
        }
        ok[s] = live[s] && (free[s] || !(bad & 1u));
    }
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        if constexpr (kBondsFirst) {
            if (ok[s]) ok[s] = !plane_any<kShift>(lattice, m[s], dir[s], mv[s]);
        } else {
            ok[s] = ok[s] && !plane_any<kShift>(front[s], m[s], dir[s]);
        }
    }

    // Mark targets and append survivors to this workgroup's list: one LDS
    // counter update per wave for all its slots.
    const gptr<uint32_t> T = proposal + size_t(t & 1u) * d.latWords;
    const uint32_t lane = threadIdx.x & 63u;
    uint64_t mask[SLOTS];
    uint32_t before[SLOTS], total = 0;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        mask[s] = __ballot(ok[s]);
        before[s] = total;
        total += uint32_t(__popcll(mask[s]));
    }
    uint32_t waveBase = 0;
    if (lane == 0 && total != 0) waveBase = atomicAdd(&lds.count, total);
    waveBase = uint32_t(__builtin_amdgcn_readfirstlane(int32_t(waveBase)));
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        if (ok[s]) {
            __hip_atomic_fetch_or(&T[mv[s].to >> 5], 1u << (mv[s].to & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            list[waveBase + before[s] + lane_rank(mask[s])] = pack_entry(j[s] | (dir[s].number() << kDirShift), m[s]);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) *count = lds.count;
}

// Sum over the wave of small per-lane counts, bit by bit with ballots and
// scalar popcounts (a uniform loop over the bits any lane has set).
__device__ __forceinline__ uint32_t wave_sum_small(uint32_t v) {
    uint32_t total = 0;
    for (uint32_t b = 0; b < 32u && __ballot((v >> b) != 0u) != 0u; ++b)
        total += uint32_t(__popcll(__ballot(((v >> b) & 1u) != 0u))) << b;
    return total;
}

// A wave's running total of accepted moves: entry `wave` of those of its
// workgroup, read at the start of pass 2 and written at its end, so that the
// kernel ends without an atomic (which is executed beyond the L2: us per
// substep with atomics and without, 128^3 melt 7.0 and 6.7, 256^3 11.1 and 10.8,
// 512^3 39.3 and 38.6).  Only a finer launch shape than the entries
// were sized for shares one entry per workgroup, with atomics.
struct AcceptedTotal {
    gptr<uint64_t> entry;
    uint64_t before;
    bool own;
};
__device__ __forceinline__ AcceptedTotal accepted_total(const Launch& L, const SysDesc& d, uint32_t workgroup,
                                                        uint32_t workgroups) {
    const uint32_t waves = blockDim.x >> 6;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int32_t(threadIdx.x >> 6)));
    AcceptedTotal a;
    a.own = workgroups * waves <= d.accEntries;
    a.entry = L.acceptedByBlock + (a.own ? workgroup * waves + wave : workgroup);
    a.before = *a.entry;
    return a;
}
__device__ __forceinline__ void add_accepted(const AcceptedTotal& a, uint32_t accepted) {
    const uint32_t total = wave_sum_small(accepted);
    if ((threadIdx.x & 63u) == 0u && total != 0u) {
        if (a.own)
            *a.entry = a.before + total;
        else
            __hip_atomic_fetch_add(a.entry, uint64_t(total), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The accepted log.  A count per wave and substep, added to the substep's
// entry, had hundreds of atomics on one address end pass 2 (9.5 instead of 6.7
// us per substep for 32768 members).  Instead pass 1 of a single system has one
// workgroup more, which sums the waves' running totals and writes the sum,
// modulo 2^32, as the entry of the substep before; the last substep's is written
// by k_log_last.  The host takes differences.  Without a log that workgroup
// ends at once: runs with and without one replay the same graphs, and the
// launch takes no longer for it (128^3 melt 6.05 and 6.04 us per substep without and
// with it, chains of 37 on 64^3 5.84 either way).
__device__ __forceinline__ void log_totals(gptr<const uint64_t> totals, uint32_t n, gptr<uint32_t> log, uint64_t entry,
                                           uint64_t capacity) {
    if (entry >= capacity) return;
    uint32_t sum = 0;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) sum += uint32_t(totals[i]);
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) sum += uint32_t(__shfl_xor(int(sum), w, 64));
    if ((threadIdx.x & 63u) == 0u)
        __hip_atomic_fetch_add(&log[entry], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The log's entry of the substep before the one that offset k serves.
__device__ __forceinline__ void log_before(gptr<const DevState> st, uint32_t k, uint32_t totals) {
    const uint64_t t = st->substep + k;
    if (st->log != nullptr && t <= st->stopAt)
        log_totals((gptr<const uint64_t>)st->acceptedByBlock, totals, (gptr<uint32_t>)st->log, t - 1u - st->logFirst,
                   st->logCapacity);
}

// Applies an accepted move of the monomer in `slot` from code m in
// direction dir (pass 2, CRITICAL.cu:400-408): its position, the occupancy
// of the old and new corner, and the periodic image counter on a wrap.
template <int LAT>
__device__ __forceinline__ void apply_move(const SysDesc& d, gptr<uint32_t> pos, gptr<uint8_t> lat, uint32_t slot,
                                           uint32_t m, const Dir& dir, const AxisMasks& mask, const Move& mv) {
    pos[slot] = mv.to;
    if (LAT == kLatticeU8) {
        lat[m] = 0;
        lat[mv.to] = 1;
    } else {
        // Byte b of the bit lattice holds the aligned 2x2x2 block of cells
        // 8b..8b+7 (the low three code bits are the lowest bit of x, y and
        // z).  Two corners in one block would overlap, and an accepted move's
        // old and new corner cannot share a block with any other monomer's
        // old or new corner, so every byte touched here has exactly one
        // writer and its new value is known: 0 for the vacated block, the
        // single new bit for the entered one.
        const uint32_t bFrom = m >> 3, bTo = mv.to >> 3;
        if (bFrom != bTo) lat[bFrom] = 0;
        lat[bTo] = uint8_t(1u << (mv.to & 7u));
    }
    if (wraps(m, dir, mask)) {
        const gptr<int32_t> img = dir.x ? d.imgX.global() : (dir.z ? d.imgZ.global() : d.imgY.global());
        img[slot] += dir.plus ? 1 : -1;
    }
}

// Pass 2 of substep t over one pass-1 list of `count` entries, the thread's
// first of them loaded.  The accepted count is added to the totals of workgroup
// `owner` of nb.  With `clear` it also zeroes slice lb of nb of the other
// parity's proposals.
template <int LAT>
__device__ __forceinline__ void perform_body(const SysDesc& d, const Launch& L, uint32_t lb, uint32_t nb, bool clear,
                                             gptr<const uint64_t> list, uint32_t count, uint64_t e, uint32_t owner) {
    const uint64_t t = L.t;
    const SubstepDraw draw = L.draw;
    const ColorInfo ci = load_color(d.colors.global(), draw.species);
    const uint32_t B = blockDim.x;
    const AcceptedTotal total = accepted_total(L, d, owner, nb);

    if (clear) clear_other_parity(d, t, lb, nb);

    const AxisMasks masks = axis_masks(d);
    const gptr<const uint64_t> T64 =
        (gptr<const uint64_t>)(d.proposal.global() + size_t(t & 1u) * d.latWords);
    const gptr<uint32_t> pos = d.pos.global();
    const gptr<uint8_t> lat = d.lattice.global();

    // The list is compacted, so about a fifth of its capacity is filled: walk
    // only the entries that exist, one per thread and round.  The first round
    // stands alone: as the loop's first it waited for every load before it, the
    // running total's too (us per substep, 128^3 melt 6.03 and 5.83, dense star
    // network 10.95 and 10.65).
    uint32_t accepted = 0;
    auto resolve = [&](uint64_t entry) {
        const uint32_t jj = uint32_t(entry) & ((1u << kDirShift) - 1u);
        const Dir dir = dir_of_number(uint32_t(entry) >> kDirShift);
        const uint32_t m = uint32_t(entry >> 32);
        const Move mv = make_move<6>(m, dir, masks);
        if (plane_any<6>(T64, m, dir, mv)) return;
        apply_move<LAT>(d, pos, lat, ci.slotOffset + jj, m, dir, masks, mv);
        ++accepted;
    };
    if (threadIdx.x < count) resolve(e);
    for (uint32_t idx = threadIdx.x + B; idx < count; idx += B) resolve(list[idx]);
    add_accepted(total, accepted);
}

// A list's length by a vector load, so that it is in flight with the state
// (mbcnt of no lanes is 0: an address per lane; as a scalar load it was issued
// behind the wait for the state).
__device__ __forceinline__ uint32_t list_count(gptr<const uint32_t> count) {
    return uint32_t(__builtin_amdgcn_readfirstlane(int32_t(count[__builtin_amdgcn_mbcnt_lo(0u, 0u)])));
}

// ---- single system ----------------------------------------------------------------
template <int LAT, int SLOTS, int MAXDEG, bool KEYED>
__global__ __launch_bounds__(256) void k_check(SysDesc d, uint32_t k, uint32_t clear, uint32_t nb,
                                                                     uint32_t totals) {
    __shared__ CheckLds lds;
    if (blockIdx.x >= nb) {  // the log's own workgroup
        log_before(d.state.global(), k, totals);
        return;
    }
    Launch L;
    if (!begin_substep(d, k, Early{}, L)) return;
    const uint32_t lb = xcd_block(nb);
    check_body<LAT, SLOTS, MAXDEG, KEYED>(d, L.t, L.draw, lb, nb, clear != 0u,
                                   (gptr<uint64_t>)d.list.global() + size_t(lb) * (SLOTS * blockDim.x),
                                   d.listCount.global() + lb, lds);
}

// After the last substep of a logged run (the state's counter stands past it).
__global__ __launch_bounds__(256) void k_log_last(const DevState* state, uint32_t totals) {
    log_before((gptr<const DevState>)state, 0u, totals);
}

template <int LAT>
__global__ __launch_bounds__(256) void k_perform(SysDesc d, uint32_t k, uint32_t listStride, uint32_t clear) {
    const uint32_t lb = xcd_block(gridDim.x);  // same numbering as pass 1: list lb
    const gptr<const uint64_t> list = (gptr<const uint64_t>)d.list.global() + size_t(lb) * listStride;
    Launch L;
    if (!begin_substep(d, k, early_of(d, false), L)) return;
    const uint32_t count = ((cptr<uint32_t>)d.listCount.global())[lb];
    const uint64_t e = threadIdx.x < count ? list[threadIdx.x] : 0u;
    perform_body<LAT>(d, L, lb, gridDim.x, clear != 0u, list, count, e, blockIdx.x);
}

// Pass 2 of a single system with several lists per workgroup: each group
// of `group` threads (whole waves) walks one pass-1 list, DEPTH entries per
// thread at a time.  Workgroup q runs on XCD q % 8 and takes lists of that
// XCD's share (the lists its pass-1 workgroups wrote, whose lines that XCD's
// L2 holds).  The list count and a thread's first entries do not depend on
// the state, so they load with it: the walk then waits for two round trips,
// the state with the list, then the proposal words of DEPTH moves at once.
template <int LAT, int DEPTH>
__global__ __launch_bounds__(256) void k_perform_lists(SysDesc d, uint32_t k, uint32_t listStride,
                                                       uint32_t listsPerXcd, uint32_t group, uint32_t clear) {
    const uint32_t xcd = blockIdx.x & 7u, local = blockIdx.x >> 3;
    const uint32_t gi = threadIdx.x / group, lane = threadIdx.x - gi * group;
    const uint32_t li = local * (blockDim.x / group) + gi;
    const bool haveList = li < listsPerXcd;
    const uint32_t lst = xcd * listsPerXcd + (haveList ? li : 0u);
    const gptr<const uint64_t> list = (gptr<const uint64_t>)d.list.global() + size_t(lst) * listStride;
    uint32_t count = d.listCount.global()[lst];
    uint64_t e[DEPTH];
#pragma unroll
    for (int r = 0; r < DEPTH; ++r) e[r] = list[min(lane + uint32_t(r) * group, listStride - 1u)];
    Launch L;
    if (!begin_substep(d, k, early_of(d, false), L)) return;
    if (!haveList) count = 0;
    const AcceptedTotal total = accepted_total(L, d, blockIdx.x, gridDim.x);
    const uint64_t t = L.t;
    const uint32_t slotOffset =
        ((gptr<const uint32_t>)(d.colors.global() + L.draw.species))[offsetof(ColorInfo, slotOffset) / 4];
    if (clear) clear_other_parity(d, t, blockIdx.x, gridDim.x);
    const AxisMasks masks = axis_masks(d);
    const gptr<const uint64_t> T64 =
        (gptr<const uint64_t>)(d.proposal.global() + size_t(t & 1u) * d.latWords);
    const gptr<uint32_t> pos = d.pos.global();
    const gptr<uint8_t> lat = d.lattice.global();

    uint32_t accepted = 0;
    for (uint32_t base = 0; base < count; base += DEPTH * group) {  // count is the same for a whole wave
        if (base != 0) {
#pragma unroll
            for (int r = 0; r < DEPTH; ++r) e[r] = list[min(base + lane + uint32_t(r) * group, listStride - 1u)];
        }
        // Entries past the count are stale: their lanes test the plane of
        // code 0 (in bounds) and drop the result.
        Move mv[DEPTH];
        Dir dir[DEPTH];
        bool hit[DEPTH], valid[DEPTH];
#pragma unroll
        for (int r = 0; r < DEPTH; ++r) {
            valid[r] = base + lane + uint32_t(r) * group < count;
            const uint32_t m = valid[r] ? uint32_t(e[r] >> 32) : 0u;
            dir[r] = dir_of_number(valid[r] ? uint32_t(e[r]) >> kDirShift : 0u);
            mv[r] = make_move<6>(m, dir[r], masks);
            hit[r] = plane_any<6>(T64, m, dir[r], mv[r]);
        }
#pragma unroll
        for (int r = 0; r < DEPTH; ++r) {
            if (!valid[r] || hit[r]) continue;
            const uint32_t jj = uint32_t(e[r]) & ((1u << kDirShift) - 1u);
            apply_move<LAT>(d, pos, lat, slotOffset + jj, uint32_t(e[r] >> 32), dir[r], masks, mv[r]);
            ++accepted;
        }
    }
    add_accepted(total, accepted);
}

// ---- batch of replicas ---------------------------------------------------------------
// Workgroup w serves tiles[w]: chunk `chunk` of `chunks` of replica `replica`.
// Lists are indexed by w, accepted counts by (replica, chunk).
// A workgroup of a few waves spends its time on round trips that depend on each
// other: tile; state, descriptor and (pass 2) list together; species; monomers.
// With the state behind the descriptor, and the list behind the state, the mix
// of 256 systems took 111.0 ms for 2000 sweeps and 96 small byte-lattice systems
// 14.7 for 1000; so 107.7 and 13.6.  (A single system's descriptor comes with
// the launch, and its list is read behind the state: ahead of it the dense star
// network took 10.84 us per substep against 10.65.)
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
struct TileRef {
    uint32_t replica, chunk, chunks, nColors;
    gptr<DevState> state;
    uint64_t seed;
};
__device__ __forceinline__ TileRef load_tile(const Tile* tiles, uint32_t w) {
    const u32x8 v = *(cptr<u32x8>)(const u32x8*)(tiles + w);
    return {v[0], v[1], v[2], v[3], (gptr<DevState>)(uintptr_t(join64(v[4], v[5]))), join64(v[6], v[7])};
}

template <int LAT, int SLOTS, int MAXDEG>
__global__ __launch_bounds__(256) void k_check_batch(const SysDesc* __restrict__ descs, const Tile* __restrict__ tiles,
                                                     uint2* lists, uint32_t* listCounts, uint32_t k) {
    __shared__ CheckLds lds;
    const TileRef tile = load_tile(tiles, blockIdx.x);
    // never null: named here so that they are loaded with the table's address
    if (tile.replica == kNoReplica || descs == nullptr || lists == nullptr || listCounts == nullptr) return;
    const SysDesc& d = descs[tile.replica];
    Launch L;
    if (!begin_substep(tile.state, tile.seed, tile.nColors, k, early_of(d, true), L)) return;
    const gptr<uint64_t> list = global_ptr(reinterpret_cast<uint64_t*>(lists)) + size_t(blockIdx.x) * (SLOTS * blockDim.x);
    // The proposals are cleared here (the mix of 256 systems, whose small ones
    // run resident: 108.8 against 112.3 ms for 2000 sweeps with the clear in
    // pass 2).  Replicas of either slot order share a launch: one uniform
    // branch per workgroup.
    if (d.keyed != 0u)
        check_body<LAT, SLOTS, MAXDEG, true>(d, L.t, L.draw, tile.chunk, tile.chunks, true, list,
                                             global_ptr(listCounts) + blockIdx.x, lds);
    else
        check_body<LAT, SLOTS, MAXDEG, false>(d, L.t, L.draw, tile.chunk, tile.chunks, true, list,
                                              global_ptr(listCounts) + blockIdx.x, lds);
}

template <int LAT>
__global__ __launch_bounds__(256) void k_perform_batch(const SysDesc* __restrict__ descs,
                                                       const Tile* __restrict__ tiles, const uint2* lists,
                                                       const uint32_t* listCounts, uint32_t k, uint32_t listStride) {
    const TileRef tile = load_tile(tiles, blockIdx.x);
    // never null: named here so that they are loaded with the table's address
    if (tile.replica == kNoReplica || descs == nullptr || lists == nullptr || listCounts == nullptr) return;
    const SysDesc& d = descs[tile.replica];
    const gptr<const uint64_t> list = global_ptr(reinterpret_cast<const uint64_t*>(lists)) + size_t(blockIdx.x) * listStride;
    Early early = early_of(d, false);
    early.count = list_count(global_ptr(listCounts) + blockIdx.x);
    early.entry = list[min(threadIdx.x, listStride - 1u)];  // past the count: dropped
    Launch L;
    if (!begin_substep(tile.state, tile.seed, tile.nColors, k, early, L)) return;
    perform_body<LAT>(d, L, tile.chunk, tile.chunks, false, list, early.count, early.entry, tile.chunk);
}

__global__ void k_advance(DevState* st, uint32_t count) {
    if (blockIdx.x == 0 && threadIdx.x == 0)
        atomicAdd(reinterpret_cast<unsigned long long*>(&st->substep), (unsigned long long)count);
}

// Every live replica of the two-pass kernels: substep = min(substep + count, stopAt).
__global__ void k_advance_batch(const SysDesc* descs, uint32_t nDescs, uint32_t count) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nDescs || descs[r].resident != 0u) return;
    const gptr<DevState> st = descs[r].state.global();
    if (st == nullptr) return;
    const uint64_t next = st->substep + count;
    st->substep = next < st->stopAt ? next : (st->substep > st->stopAt ? st->substep : st->stopAt);
}

__global__ void k_set_stops(const SysDesc* descs, uint32_t nDescs, const uint64_t* stops) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nDescs) return;
    const gptr<DevState> st = descs[r].state.global();
    if (st == nullptr) return;
    st->stopAt = stops[r];
}

// One workgroup per replica sums its per-workgroup accepted counters.
__global__ void k_gather_state(const SysDesc* descs, uint32_t nDescs, uint64_t* out) {
    __shared__ uint64_t part[256];
    const uint32_t r = blockIdx.x;
    if (r >= nDescs) return;
    const gptr<const DevState> st = descs[r].state.global();
    uint64_t sum = 0;
    if (st != nullptr)
        for (uint32_t i = threadIdx.x; i < descs[r].accEntries; i += blockDim.x) sum += global_ptr(st->acceptedByBlock)[i];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t w = blockDim.x / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[3 * r + 0] = st ? st->substep : 0;
        out[3 * r + 1] = st ? st->stopAt : 0;
        out[3 * r + 2] = part[0];
    }
}

// The bits of m selected by `mask`, packed from bit 0 up (mask is the same
// for every lane, so the loop is uniform).
__device__ __forceinline__ uint32_t compact_bits(uint32_t m, uint32_t mask) {
    uint32_t v = 0, k = 0;
    while (mask != 0u) {
        const uint32_t b = uint32_t(__builtin_ctz(mask));
        v |= ((m >> b) & 1u) << k;
        ++k;
        mask &= mask - 1u;
    }
    return v;
}

// Unfolded corner of the monomer in slot s: the code's axis bits plus the
// image counter times the box edge, written to out[0..2].
__device__ __forceinline__ void unfold_slot(gptr<const uint32_t> pos, const gptr<const int32_t> img[3],
                                            const uint32_t mask[3], uint32_t s, gptr<int32_t> out) {
    const uint32_t m = pos[s];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int32_t edge = int32_t(1u << __builtin_popcount(mask[a]));
        out[a] = int32_t(compact_bits(m, mask[a])) + img[a][s] * edge;
    }
}

__global__ void k_unfold(SysDesc d, const uint32_t* __restrict__ slotOf, uint32_t n, int32_t* __restrict__ xyz) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const gptr<const int32_t> img[3] = {d.imgX.global(), d.imgY.global(), d.imgZ.global()};
    const uint32_t mask[3] = {d.mask[0], d.mask[1], d.mask[2]};
    unfold_slot(d.pos.global(), img, mask, global_ptr(slotOf)[i], global_ptr(xyz) + 3 * size_t(i));
}

// Several monomer ranges of several systems in one launch: workgroup b
// serves the last job whose firstBlock is at most b (jobs in order of
// firstBlock, the first at 0), monomers first + (b - firstBlock) * blockDim
// + threadIdx of that job, written as records out + ... of xyz.
__global__ __launch_bounds__(256) void k_unfold_jobs(const UnfoldJob* __restrict__ jobs, uint32_t nJobs,
                                                     int32_t* __restrict__ xyz) {
    const uint32_t b = blockIdx.x;
    uint32_t lo = 0, hi = nJobs;
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].firstBlock <= b) lo = mid;
        else hi = mid;
    }
    const UnfoldJob& J = jobs[lo];
    const uint32_t i = (b - J.firstBlock) * blockDim.x + threadIdx.x;
    if (i >= J.count) return;
    const gptr<const int32_t> img[3] = {global_ptr(J.img[0]), global_ptr(J.img[1]), global_ptr(J.img[2])};
    const uint32_t mask[3] = {J.mask[0], J.mask[1], J.mask[2]};
    unfold_slot(global_ptr(J.pos), img, mask, global_ptr(J.slotOf)[J.first + i],
                global_ptr(xyz) + 3 * (J.out + i));
}

__global__ void k_wait() {
    for (int i = 0; i < 32; ++i) __builtin_amdgcn_s_sleep(127);  // 127 * 64 cycles each
}

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += uint64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

// Plain streaming copy: the reference point that scales the HBM byte
// counters of a profiler run (it reads and writes exactly n*16 bytes).
__global__ void k_copy_u4(const uint4* __restrict__ src, uint4* __restrict__ dst, uint64_t n) {
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        dst[i] = src[i];
}

// ---- template dispatch ------------------------------------------------------------------
template <int LAT, int SLOTS, int MAXDEG>
void check_launch(const SysDesc& d, const BatchLaunch* b, uint32_t k, const LaunchShape& s, hipStream_t st) {
    const dim3 blk(s.block);
    if (b)
        hipLaunchKernelGGL((k_check_batch<LAT, SLOTS, MAXDEG>), dim3(b->tiles), blk, 0, st, b->descs, b->tileTable,
                           b->lists, b->listCounts, k);
    else if (d.keyed != 0u)
        hipLaunchKernelGGL((k_check<LAT, SLOTS, MAXDEG, true>), dim3(s.grid + 1u), blk, 0, st, d, k,
                           uint32_t(s.clearPass == 1u), s.grid, s.totals);
    else
        hipLaunchKernelGGL((k_check<LAT, SLOTS, MAXDEG, false>), dim3(s.grid + 1u), blk, 0, st, d, k,
                           uint32_t(s.clearPass == 1u), s.grid, s.totals);
}

template <int LAT, int SLOTS>
void check_by_degree(const SysDesc& d, const BatchLaunch* b, uint32_t k, const LaunchShape& s, hipStream_t st) {
    const uint32_t deg = b ? b->maxDegree : d.maxDegree;
    if (deg <= 2)
        check_launch<LAT, SLOTS, 2>(d, b, k, s, st);
    else if (deg <= 4)
        check_launch<LAT, SLOTS, 4>(d, b, k, s, st);
    else
        check_launch<LAT, SLOTS, 8>(d, b, k, s, st);
}

template <int LAT>
void check_by_slots(const SysDesc& d, const BatchLaunch* b, uint32_t k, const LaunchShape& s, hipStream_t st) {
    switch (s.slots) {
        case 1: check_by_degree<LAT, 1>(d, b, k, s, st); break;
        case 2: check_by_degree<LAT, 2>(d, b, k, s, st); break;
        default: check_by_degree<LAT, 4>(d, b, k, s, st); break;
    }
}

template <int LAT>
void perform_launch(const SysDesc& d, const BatchLaunch* b, uint32_t k, const LaunchShape& s, hipStream_t st) {
    const dim3 blk(s.passTwoBlock());
    if (b)
        hipLaunchKernelGGL((k_perform_batch<LAT>), dim3(b->tiles), blk, 0, st, b->descs, b->tileTable, b->lists,
                           b->listCounts, k, s.listStride());
    else if (s.listGroup == 0)
        hipLaunchKernelGGL((k_perform<LAT>), dim3(s.grid), blk, 0, st, d, k, s.listStride(),
                           uint32_t(s.clearPass != 1u));
    else if (s.listDepth >= 4)
        hipLaunchKernelGGL((k_perform_lists<LAT, 4>), dim3(s.passTwoGrid()), blk, 0, st, d, k, s.listStride(),
                           s.listsPerXcd(), s.listGroup, uint32_t(s.clearPass != 1u));
    else
        hipLaunchKernelGGL((k_perform_lists<LAT, 1>), dim3(s.passTwoGrid()), blk, 0, st, d, k, s.listStride(),
                           s.listsPerXcd(), s.listGroup, uint32_t(s.clearPass != 1u));
}

}  // namespace

hipError_t launch_check(const SysDesc& d, uint32_t k, const LaunchShape& s, hipStream_t st) {
    if (d.latticeKind == kLatticeU8)
        check_by_slots<kLatticeU8>(d, nullptr, k, s, st);
    else
        check_by_slots<kLatticeBit>(d, nullptr, k, s, st);
    return hipGetLastError();
}

hipError_t launch_perform(const SysDesc& d, uint32_t k, const LaunchShape& s, hipStream_t st) {
    if (d.latticeKind == kLatticeU8)
        perform_launch<kLatticeU8>(d, nullptr, k, s, st);
    else
        perform_launch<kLatticeBit>(d, nullptr, k, s, st);
    return hipGetLastError();
}

hipError_t launch_check_batch(const BatchLaunch& b, uint32_t k, const LaunchShape& s, hipStream_t st) {
    const SysDesc none{};
    if (b.latticeKind == kLatticeU8)
        check_by_slots<kLatticeU8>(none, &b, k, s, st);
    else
        check_by_slots<kLatticeBit>(none, &b, k, s, st);
    return hipGetLastError();
}

hipError_t launch_perform_batch(const BatchLaunch& b, uint32_t k, const LaunchShape& s, hipStream_t st) {
    const SysDesc none{};
    if (b.latticeKind == kLatticeU8)
        perform_launch<kLatticeU8>(none, &b, k, s, st);
    else
        perform_launch<kLatticeBit>(none, &b, k, s, st);
    return hipGetLastError();
}

hipError_t launch_advance(DevState* state, uint32_t count, hipStream_t st) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, st, state, count);
    return hipGetLastError();
}

hipError_t launch_advance_batch(const SysDesc* descs, uint32_t nDescs, uint32_t count, hipStream_t st) {
    if (nDescs == 0) return hipSuccess;
    hipLaunchKernelGGL(k_advance_batch, dim3((nDescs + 255) / 256), dim3(256), 0, st, descs, nDescs, count);
    return hipGetLastError();
}

hipError_t launch_set_stops(const SysDesc* descs, uint32_t nDescs, const uint64_t* stops, hipStream_t st) {
    if (nDescs == 0) return hipSuccess;
    hipLaunchKernelGGL(k_set_stops, dim3((nDescs + 255) / 256), dim3(256), 0, st, descs, nDescs, stops);
    return hipGetLastError();
}

hipError_t launch_gather_state(const SysDesc* descs, uint32_t nDescs, uint64_t* out, hipStream_t st) {
    if (nDescs == 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_state, dim3(nDescs), dim3(256), 0, st, descs, nDescs, out);
    return hipGetLastError();
}

hipError_t launch_unfold(const SysDesc& d, const uint32_t* slotOf, uint32_t n, int32_t* xyz, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unfold, dim3((n + 255) / 256), dim3(256), 0, st, d, slotOf, n, xyz);
    return hipGetLastError();
}

hipError_t launch_unfold_jobs(const UnfoldJob* jobs, uint32_t nJobs, uint32_t blocks, int32_t* xyz, hipStream_t st) {
    if (nJobs == 0 || blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unfold_jobs, dim3(blocks), dim3(kUnfoldBlock), 0, st, jobs, nJobs, xyz);
    return hipGetLastError();
}

hipError_t launch_log_last(const DevState* state, const LaunchShape& s, hipStream_t st) {
    hipLaunchKernelGGL(k_log_last, dim3(1), dim3(256), 0, st, state, s.totals);
    return hipGetLastError();
}

hipError_t launch_wait(hipStream_t st) {
    hipLaunchKernelGGL(k_wait, dim3(1), dim3(64), 0, st);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t st) {
    if (n == 0) return hipSuccess;
    uint64_t g = (n + 255) / 256;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(k_fill_u32, dim3(uint32_t(g)), dim3(256), 0, st, p, n, v);
    return hipGetLastError();
}

hipError_t launch_copy_u4(const void* src, void* dst, uint64_t n16, hipStream_t st) {
    if (n16 == 0) return hipSuccess;
    uint64_t g = (n16 + 255) / 256;
    if (g > 1u << 20) g = 1u << 20;
    hipLaunchKernelGGL(k_copy_u4, dim3(uint32_t(g)), dim3(256), 0, st, static_cast<const uint4*>(src),
                       static_cast<uint4*>(dst), n16);
    return hipGetLastError();
}

}  // namespace pscbfm
