// Resident sweep: one workgroup holds a whole small system in LDS and runs
// many substeps in one launch.
//
// A substep of the two-pass kernels (kernels.hip) is two launches, 6 to 7 us
// on a system of any size up to some hundred thousand monomers, nearly all of
// it the kernel boundaries and the round trips of a few dependent loads.  Here
// the boundary between the passes is a workgroup barrier and the gathers are
// LDS reads, so a substep costs what its vector instructions cost on one
// compute unit: 0.9 us for 192 members of the drawn species (two passes: 5.1),
// 1.1 to 1.25 for 512 (5.8), 3.2 for 2500, 4.8 for 4000 and 5.5 for 4800 (5.9), in a
// batch 5.9 for 5000: vector issue on one compute unit (150 instructions per 64
// members; when it was 7% more, 192 members took 1.09 us instead of 1.01).
//
// LDS: the occupancy lattice and one proposal lattice (1 bit per cell, Z-curve
// order, whatever lattice kind the system has in memory), the code of every
// slot and the bond table as bytes.  Draw keys and partner ids stay in memory;
// those of the next substep are read while this one's moves are resolved.
//
// Thread i handles members i + k*blockDim of the drawn species, k < ROUNDS, in
// registers from the draw to the resolution: the second pass tests the same
// plane cells with the same masks, on the proposal lattice.  (Compacting the
// moves that pass the bond test, and the survivors, into per-wave lists cost
// more than the idle lanes: 3.85 against 2.78 us per substep for 1850 members,
// 7.24 against 6.19 for 4921.)  What depends on the direction alone, and the
// plane's cells, are LDS tables: LDS has cycles to spare, the vector units not.
//
// The system's buffers in memory are as if the two-pass kernels had run: codes,
// images, lattice, accepted counts, log and both proposal buffers.
#include <algorithm>

#include "kernels.h"
#include "sweep_device.h"

namespace pscbfm {

namespace {

// Largest species of a system on its own, by lattice and bonds per member: us per
// substep, resident against two passes, on 64^3 (byte lattice in brackets).  Up to
// two bonds: 4088 members 4.8 and 5.8 (4.8 and 6.1), 4800 5.5 and 5.9 (5.4 and 6.2),
// 5000 5.75 and 5.7 (5.65 and 6.1).  Up to four: 4317 5.9 and 6.1 (5.7 and 6.4),
// 4687 6.2 and 6.0 (6.0 and 6.3), 4810 (6.0 and 6.45).  More: 2614 5.0 and 6.2 (4.8
// and 6.7), 3267 6.25 and 6.2 (6.0 and 6.6), 3594 6.6 and 6.1 (6.3 and 6.6), 4084 7.3
// and 6.2 (7.0 and 6.75).
uint32_t resident_alone(const SysDesc& d) {
    const bool bytes = d.latticeKind == kLatticeU8;
    if (d.maxDegree <= 2u) return 4864u;
    if (d.maxDegree <= 4u) return bytes ? 4864u : 4480u;
    return bytes ? 3776u : 3200u;
}
// Of a batch replica of up to two bonds whatever else the batch holds: with
// 5120 members 5.7 us per substep (byte lattice 5.6), where a batch of one to
// four such two-pass replicas takes 6.0 to 6.2 (6.2 to 6.6).
constexpr uint32_t kResidentInBatch = 5120;

// LDS addresses.  The kernels have no static LDS, so their dynamic LDS starts
// at address 0; plain numbers let the compiler put the fixed parts into the
// instructions' offset fields.
constexpr uint32_t kBond = 0;                  // 512 bytes by bond key
// Six direction records: masks of the axis, of u and of v, the step in dilated
// form; two steps, one in u, one in v, the cells of the words of u-1.
constexpr uint32_t kDirs = kBond + 512;
constexpr uint32_t kPlanes = kDirs + 6 * 32;   // plane cells by axis and low six code bits
constexpr uint32_t kLat = kPlanes + 192 * 8;   // occupancy, then proposals, then codes of the slots
static_assert(kLat % 16 == 0, "16-byte LDS accesses");

template <class T>
using lptr = __attribute__((address_space(3))) T*;
template <class T>
__device__ __forceinline__ lptr<T> lds(uint32_t address) {
    return (lptr<T>)(uintptr_t)address;
}

// A move from its draw to its resolution.
struct Held {
    uint32_t to, record;          // new corner; LDS address of the direction record
    uint32_t q00, q02, q20, q22;  // bytes to the 64-cell words of the front plane
    uint32_t low, high;           // its cells in a word
};

// Whether a cell of the plane is set in the lattice at LDS address `words`
// (plane_any of sweep_device.h).
__device__ __forceinline__ bool held_any(uint32_t words, const Held& h, uint32_t su, bool z) {
    const uint64_t w00 = *lds<const uint64_t>(words + h.q00), w02 = *lds<const uint64_t>(words + h.q02);
    const uint64_t w20 = *lds<const uint64_t>(words + h.q20), w22 = *lds<const uint64_t>(words + h.q22);
    return merged_any(w00, w02, w20, w22, PlaneMask{h.low, h.high, su, z ? 0xFFFF0000u : 0u, z ? 0xFFFF0000u : ~0u});
}

__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t lane) {
    return uint32_t(__builtin_amdgcn_readlane(int32_t(v), int32_t(lane)));
}

// Words that are the same for every lane, in scalar registers: in a function that
// is no kernel the compiler keeps what it loads from memory that is written in
// vector ones (four-arm stars of 580 members: 2.10 us per substep, so 2.01).
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int32_t(v))); }
__device__ __forceinline__ u32x4 uniform(u32x4 v) { return u32x4{uniform(v.x), uniform(v.y), uniform(v.z), uniform(v.w)}; }

// A substep's draw and its species' record, the same for every lane.
struct Substep {
    uint32_t seed, slotOffset, count, nbrOffset, pitch, degree;
};

// The next 64 substeps, one in each lane.
struct Ahead {
    uint32_t seed = 0, slotOffset = 0, count = 0, nbrOffset = 0, pitch = 0, degree = 0;
    __device__ __forceinline__ void fill(const SysDesc& d, uint64_t t, gptr<const uint64_t> table, uint64_t drawBase) {
        SubstepDraw draw;
        if (table == nullptr) {
            draw = substep_draw(d.seed, t, d.nColors);
        } else {
            const uint64_t e = table[t - drawBase];
            draw.species = uint32_t(e);
            draw.seed = uint32_t(e >> 32);
        }
        const ColorInfo ci = load_color(d.colors.global(), draw.species);
        seed = draw.seed;
        slotOffset = ci.slotOffset;
        count = ci.count;
        nbrOffset = ci.nbrOffset;
        pitch = ci.nbrPitch;
        degree = ci.maxDegree;
    }
    __device__ __forceinline__ Substep at(uint32_t i) const {
        return {lane_value(seed, i),      lane_value(slotOffset, i), lane_value(count, i),
                lane_value(nbrOffset, i), lane_value(pitch, i),      lane_value(degree, i)};
    }
};

// Draw keys and partner ids of a thread's members.  A lane past the species
// reads its last member's and drops the move.  A row past the species' degree
// is its first one again, as the matrix repeats the first bond of a monomer with
// fewer than others (every monomer of a resident system has one).  Without
// keys in memory the key is that of the member's index, the same for every
// substep.
template <int ROUNDS, int MAXDEG>
struct Static {
    uint32_t key[ROUNDS], id[ROUNDS][MAXDEG];
    __device__ __forceinline__ void load(const SysDesc& d, const Substep& s) {
        const gptr<const uint32_t> keys = (gptr<const uint32_t>)d.key.global() + s.slotOffset;
        const bool keyed = d.keyed != 0u;
        gptr<const uint32_t> row[MAXDEG];
#pragma unroll
        for (uint32_t r = 0; r < uint32_t(MAXDEG); ++r)
            row[r] = (gptr<const uint32_t>)d.nbr.global() + s.nbrOffset + (r < s.degree ? r * s.pitch : 0u);
#pragma unroll
        for (uint32_t k = 0; k < uint32_t(ROUNDS); ++k) {
            const uint32_t o = 4u * min(threadIdx.x + k * blockDim.x, s.count - 1u);
            if (keyed) key[k] = at(keys, o);
#pragma unroll
            for (int r = 0; r < MAXDEG; ++r) id[k][r] = at(row[r], o);
        }
    }
};

// Copies items 0..n-1, thread by thread, N loads in flight per thread: one at a
// time, the copies at a launch's ends were a chain of round trips (a call of one
// sweep, a chain of 128 in 128 x 64 x 64: 56.6 us, on the byte lattice 94.7; so,
// and with the threads that resident_block adds, 9.8 and 21.9; two passes 23).
template <int N, class Load, class Store>
__device__ __forceinline__ void in_batches(uint32_t n, Load load, Store store) {
    for (uint32_t first = 0; first < n; first += N * blockDim.x) {
        decltype(load(0u)) v[N];
#pragma unroll
        for (uint32_t q = 0; q < uint32_t(N); ++q)
            if (first + q * blockDim.x < n) v[q] = load(min(first + q * blockDim.x + threadIdx.x, n - 1u));
#pragma unroll
        for (uint32_t q = 0; q < uint32_t(N); ++q) {
            const uint32_t i = first + q * blockDim.x + threadIdx.x;
            if (i < n) store(i, v[q]);
        }
    }
}

// 16 cells of the byte lattice and of a bit lattice: four 0/1 bytes times 2^24 +
// 2^17 + 2^10 + 2^3 have their bits side by side in bits 24..27.
__device__ __forceinline__ uint32_t pack_cells(u32x4 cells) {
    uint32_t v = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) v |= ((((cells[q] & 0x01010101u) * 0x01020408u) >> 24) & 15u) << (4u * q);
    return v;
}
__device__ __forceinline__ u32x4 unpack_cells(uint32_t v) {
    u32x4 cells;
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) cells[q] = (((v >> (4u * q)) & 15u) * 0x00204081u) & 0x01010101u;
    return cells;
}

template <int ROUNDS, int MAXDEG, bool IN_KERNEL>
__device__ __forceinline__ void resident_body(const SysDesc& d, uint32_t substeps) {
    const uint32_t B = blockDim.x, tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave64 = uint32_t(__builtin_amdgcn_readfirstlane(int32_t(tid & ~63u)));
    const uint32_t latWords = d.latWords;
    const uint32_t sProp = kLat + 4u * latWords, sPos = sProp + 4u * latWords;

    const gptr<const u32x4> w = (gptr<const u32x4>)d.state.global();
    auto word = [&](int i) { return IN_KERNEL ? w[i] : uniform(w[i]); };
    const u32x4 w0 = word(0), w1 = word(1), w2 = word(2), w3 = word(3);  // DevState field order
    const uint64_t t0 = join64(w0.x, w0.y), stopAt = join64(w0.z, w0.w);
    if (t0 >= stopAt || substeps == 0u) return;
    const uint32_t n = uint32_t(min(uint64_t(substeps), stopAt - t0));
    const gptr<const uint64_t> table = (gptr<const uint64_t>)(uintptr_t(join64(w1.x, w1.y)));
    const uint64_t drawBase = join64(w1.z, w1.w);
    const gptr<uint32_t> log = (gptr<uint32_t>)(uintptr_t(join64(w2.x, w2.y)));
    const uint64_t logFirst = join64(w2.z, w2.w), logCapacity = join64(w3.x, w3.y);
    const gptr<uint64_t> accepted = (gptr<uint64_t>)(uintptr_t(join64(w3.z, w3.w)));

    // Load.
    const gptr<uint32_t> posAll = d.pos.global();
    if (d.latticeKind == kLatticeU8)
        in_batches<4>(latWords * 2u, [&](uint32_t i) { return ((gptr<const u32x4>)d.lattice.global())[i]; },
                      [&](uint32_t i, u32x4 v) { *lds<uint16_t>(kLat + 2u * i) = uint16_t(pack_cells(v)); });
    else
        in_batches<4>(latWords / 4u, [&](uint32_t i) { return ((gptr<const u32x4>)d.lattice.global())[i]; },
                      [&](uint32_t i, u32x4 v) { *lds<u32x4>(kLat + 16u * i) = v; });
    in_batches<4>(d.nSlots, [&](uint32_t i) { return posAll[i]; },
                  [&](uint32_t i, uint32_t v) { *lds<uint32_t>(sPos + 4u * i) = v; });
    for (uint32_t i = tid; i < 512u; i += B)
        *lds<uint8_t>(kBond + i) = uint8_t((d.bondMask.global()[i >> 5] >> (i & 31u)) & 1u);
    const AxisMasks masks = axis_masks(d);
    for (uint32_t i = tid; i < 6u; i += B) {
        const Dir dir = dir_of_number(i);
        const uint32_t Ma = dir.x ? masks.x : (dir.z ? masks.z : masks.y), oneA = dir.x ? 1u : (dir.z ? 4u : 2u);
        *lds<u32x4>(kDirs + 32u * i) =
            u32x4{Ma, dir.x ? masks.y : masks.x, dir.z ? masks.y : masks.z, dir.plus ? oneA : Ma};
        *lds<u32x4>(kDirs + 32u * i + 16u) = u32x4{dir.plus ? oneA << 3 : Ma ^ oneA, dir.x ? 2u : 1u, dir.z ? 2u : 4u,
                                                   dir.x ? 0xFFFF0000u : 0xFF00FF00u};
    }
    for (uint32_t i = tid; i < 192u; i += B) {
        const PlaneMask p = plane_mask(i & 63u, dir_of_number(2u * (i >> 6)));
        *lds<uint64_t>(kPlanes + 8u * i) = join64(p.low, p.high);
    }
    uint64_t total = 0;

    // Few values per thread: read one substep ahead.  Else at the substep's
    // start, ahead of the clear and its barrier.
    constexpr bool kReadAhead = ROUNDS * (1 + MAXDEG) <= 12;
    Ahead ahead;
    ahead.fill(d, t0 + min(lane, n - 1u), table, drawBase);
    Substep s = ahead.at(0);
    Static<ROUNDS, MAXDEG> st;
#pragma unroll
    for (uint32_t k = 0; k < uint32_t(ROUNDS); ++k) st.key[k] = move_hash(tid + k * B);
    if constexpr (kReadAhead) st.load(d, s);

    for (uint32_t step = 0; step < n; ++step) {
        if constexpr (!kReadAhead) st.load(d, s);
        // The last substep's proposals: read before the barrier that ended it.
        for (uint32_t i = tid; i < latWords / 4u; i += B) *lds<u32x4>(sProp + 16u * i) = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();

        Held held[ROUNDS];
        uint32_t ok = 0;  // bit k: the move of round k stands
#pragma unroll
        for (uint32_t k = 0; k < uint32_t(ROUNDS); ++k) {
            if (wave64 + k * B >= s.count) break;  // the same for the whole wave
            const uint32_t j = tid + k * B, jj = min(j, s.count - 1u);
            Held& h = held[k];
            const uint32_t m = *lds<uint32_t>(sPos + 4u * (s.slotOffset + jj));
            uint32_t code[MAXDEG];
#pragma unroll
            for (uint32_t r = 0; r < uint32_t(MAXDEG); ++r) code[r] = *lds<uint32_t>(sPos + 4u * st.id[k][r]);
            const uint32_t rn = move_hash(st.key[k] ^ s.seed);
            const Dir dir = dir_of_hash(rn);
            const uint32_t axis = dir.x ? 0u : (dir.z ? 128u : 64u);
            h.record = axis | (rn & 1u) << 5;
            const u32x4 ra = *lds<const u32x4>(kDirs + h.record), rb = *lds<const u32x4>(kDirs + h.record + 16u);
            const uint64_t cells = *lds<const uint64_t>(kPlanes + 8u * (axis | (m & 63u)));
            h.low = uint32_t(cells);
            h.high = uint32_t(cells >> 32);
            const uint32_t ta = m | ~ra.x, tu = m | ~ra.y, tv = m | ~ra.z;
            h.to = (m & ~ra.x) | ((ta + ra.w) & ra.x);
            uint32_t bad = 0;
#pragma unroll
            for (int r = 0; r < MAXDEG; ++r) bad |= *lds<const uint8_t>(kBond + bond_key(code[r], h.to));
            const uint32_t fa = (ta + rb.x) & ra.x & ~63u;
            const uint32_t u0 = fa | ((tu + ra.y) & ra.y & ~63u), u2 = fa | ((tu + rb.y) & ra.y & ~63u);
            const uint32_t v0 = (tv + ra.z) & ra.z & ~63u, v2 = (tv + rb.z) & ra.z & ~63u;
            h.q00 = (u0 | v0) >> 3;
            h.q02 = (u0 | v2) >> 3;
            h.q20 = (u2 | v0) >> 3;
            h.q22 = (u2 | v2) >> 3;
            const bool blocked = held_any(kLat, h, rb.w, dir.z);
            if (j < s.count && bad == 0u && !blocked) {
                ok |= 1u << k;
                atomicOr((uint32_t*)lds<uint32_t>(sProp + 4u * (h.to >> 5)), 1u << (h.to & 31u));
            }
        }

        const uint32_t slot0 = s.slotOffset + tid;
        if (step + 1u < n) {
            if (((step + 1u) & 63u) == 0u) ahead.fill(d, t0 + min(step + 1u + lane, n - 1u), table, drawBase);
            s = ahead.at((step + 1u) & 63u);
            if constexpr (kReadAhead) st.load(d, s);
        }
        __syncthreads();

        uint32_t moved = 0;
#pragma unroll
        for (uint32_t k = 0; k < uint32_t(ROUNDS); ++k) {
            const Held& h = held[k];
            bool go = (ok >> k & 1u) != 0u;
            if (__ballot(go) == 0u) continue;
            if (go) {
                go = !held_any(sProp, h, h.record < 64u ? 0xFFFF0000u : 0xFF00FF00u, h.record >= 128u);
                if (go) {
                    const uint32_t slot = slot0 + k * B, m = *lds<uint32_t>(sPos + 4u * slot);
                    *lds<uint32_t>(sPos + 4u * slot) = h.to;
                    // one writer per byte, as in apply_move (kernels.hip)
                    const uint32_t bFrom = m >> 3, bTo = h.to >> 3;
                    if (bFrom != bTo) *lds<uint8_t>(kLat + bFrom) = 0;
                    *lds<uint8_t>(kLat + bTo) = uint8_t(1u << (h.to & 7u));
                    // a step up has the larger code unless it wraps, a step down the smaller
                    const bool plus = (h.record & 32u) != 0u;
                    if ((h.to > m) != plus) {
                        const gptr<int32_t> img = h.record < 64u    ? d.imgX.global()
                                                  : h.record < 128u ? d.imgY.global()
                                                                    : d.imgZ.global();
                        __hip_atomic_fetch_add(&img[slot], plus ? 1 : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            }
            moved += uint32_t(__popcll(__ballot(go)));
        }
        total += moved;
        if (log != nullptr && lane == 0u && moved != 0u) {
            const uint64_t idx = t0 + step - logFirst;
            if (idx < logCapacity)
                __hip_atomic_fetch_add(&log[idx], moved, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
    }

    // Store.
    if (lane == 0u && total != 0u)
        __hip_atomic_fetch_add(&accepted[0], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    in_batches<2>(d.nSlots, [&](uint32_t i) { return *lds<uint32_t>(sPos + 4u * i); },
                  [&](uint32_t i, uint32_t v) { posAll[i] = v; });
    if (d.latticeKind == kLatticeU8)
        in_batches<2>(latWords * 2u, [&](uint32_t i) { return uint32_t(*lds<uint16_t>(kLat + 2u * i)); },
                      [&](uint32_t i, uint32_t v) { ((gptr<u32x4>)d.lattice.global())[i] = unpack_cells(v); });
    else
        in_batches<2>(latWords / 4u, [&](uint32_t i) { return *lds<u32x4>(kLat + 16u * i); },
                      [&](uint32_t i, u32x4 v) { ((gptr<u32x4>)d.lattice.global())[i] = v; });
    const gptr<u32x4> marks = (gptr<u32x4>)d.proposal.global();
    const uint32_t last = uint32_t((t0 + n - 1u) & 1u), quads = latWords / 4u;
    in_batches<2>(quads, [&](uint32_t i) { return *lds<u32x4>(sProp + 16u * i); },
                  [&](uint32_t i, u32x4 v) {
                      marks[last * quads + i] = v;
                      marks[(last ^ 1u) * quads + i] = u32x4{0u, 0u, 0u, 0u};
                  });
    if (tid == 0u) d.state.global()->substep = t0 + n;
}

// Members per thread of the batch builds.
__host__ __device__ __forceinline__ uint32_t batch_rounds(uint32_t members, uint32_t block) {
    return members <= 4u * block ? 4u : (members <= 5u * block ? 5u : 8u);
}

template <int ROUNDS, int MAXDEG>
__global__ __launch_bounds__(1024) void k_resident(SysDesc d, uint32_t substeps) {
    resident_body<ROUNDS, MAXDEG, true>(d, substeps);
}

// A function of its own per build, so that each has the registers it needs and
// no others; its arguments, the same for every lane, go back to scalar registers.
template <int ROUNDS, int MAXDEG>
__device__ __attribute__((noinline)) void resident_build(const SysDesc* desc, uint32_t substeps) {
    const uint64_t p = uint64_t(uintptr_t(desc));
    const uint64_t u = join64(uniform(uint32_t(p)), uniform(uint32_t(p >> 32)));
    resident_body<ROUNDS, MAXDEG, false>(*(const SysDesc*)(cptr<SysDesc>)uintptr_t(u), uniform(substeps));
}

template <int ROUNDS>
__device__ __forceinline__ void resident_of_degree(const SysDesc* desc, uint32_t substeps) {
    if (desc->maxDegree <= 2u)
        resident_build<ROUNDS, 2>(desc, substeps);
    else if (desc->maxDegree <= 4u)
        resident_build<ROUNDS, 4>(desc, substeps);
    else
        resident_build<ROUNDS, 8>(desc, substeps);
}

// Replicas of one build.
template <int ROUNDS, int MAXDEG>
__global__ __launch_bounds__(1024) void k_resident_batch(const SysDesc* __restrict__ descs,
                                                         const uint32_t* __restrict__ ids, uint32_t substeps) {
    resident_body<ROUNDS, MAXDEG, true>(descs[ids[blockIdx.x]], substeps);
}

// Replicas of several builds, each swept by its own.  Eight replicas of 5000
// members and a small eight-arm star, us per sweep: 26.1 with all of them on the
// build that holds both, 11.9 so, 11.8 without the star.
__global__ __launch_bounds__(1024) void k_resident_mix(const SysDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ ids, uint32_t substeps) {
    const SysDesc* desc = descs + ids[blockIdx.x];
    const uint32_t rounds = batch_rounds(desc->maxColorCount, blockDim.x);
    if (rounds == 4u)
        resident_of_degree<4>(desc, substeps);
    else if (rounds == 5u)
        resident_of_degree<5>(desc, substeps);
    else if (desc->maxDegree <= 2u)
        resident_build<8, 2>(desc, substeps);
    else
        resident_build<8, 4>(desc, substeps);
}

using ResidentKernel = void (*)(SysDesc, uint32_t);
template <int ROUNDS>
ResidentKernel resident_by_degree(uint32_t maxDegree) {
    return maxDegree <= 2u ? k_resident<ROUNDS, 2> : (maxDegree <= 4u ? k_resident<ROUNDS, 4> : k_resident<ROUNDS, 8>);
}
ResidentKernel resident_kernel(uint32_t rounds, uint32_t maxDegree) {
    if (rounds <= 1u) return resident_by_degree<1>(maxDegree);
    if (rounds <= 2u) return resident_by_degree<2>(maxDegree);
    if (rounds <= 3u) return resident_by_degree<3>(maxDegree);
    if (rounds <= 4u) return resident_by_degree<4>(maxDegree);
    return maxDegree <= 2u ? k_resident<5, 2> : k_resident<5, 4>;  // more bonds: at most four (resident_alone)
}
using ResidentBatchKernel = void (*)(const SysDesc*, const uint32_t*, uint32_t);
template <int ROUNDS>
ResidentBatchKernel resident_batch_by_degree(uint32_t maxDegree) {
    return maxDegree <= 2u ? k_resident_batch<ROUNDS, 2>
                           : (maxDegree <= 4u ? k_resident_batch<ROUNDS, 4> : k_resident_batch<ROUNDS, 8>);
}
ResidentBatchKernel resident_batch_kernel(const ResidentClass& c) {
    if (c.mixed) return k_resident_mix;
    if (c.rounds == 4u) return resident_batch_by_degree<4>(c.maxDegree);
    if (c.rounds == 5u) return resident_batch_by_degree<5>(c.maxDegree);
    return c.maxDegree <= 2u ? k_resident_batch<8, 2> : k_resident_batch<8, 4>;
}

// Dynamic LDS beyond 64 KiB is asked for per kernel and device, ahead of every
// launch that takes it: a device reset may forget it.
hipError_t allow_lds(const void* kernel, uint64_t bytes) {
    if (bytes <= 64u * 1024u) return hipSuccess;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(kResidentLds));
}

}  // namespace

uint64_t resident_lds_bytes(const SysDesc& d) {
    return kLat + 8ull * d.latWords + 4ull * ((uint64_t(d.nSlots) + 3u) & ~3ull);
}

uint32_t resident_block(const SysDesc& d) {
    if (d.maxColorCount == 0u || d.maxColorCount > resident_alone(d) || d.lone != 0u) return 0u;
    // A thread per member, but no fewer than one per 16 bytes of the lattice, up
    // to 512: every substep clears the proposals, every launch loads and stores
    // all.  One chain of 128, us per substep with 64, 256, 512 and 1024 threads:
    // 32^3 0.81, 0.77, 0.77 and 0.78; 64^3 1.64, 0.96, 0.91 and 0.92; 128 x 64 x 64
    // 2.60, 1.21, 1.08 and 1.09 (a call of one sweep 21.9, 10.9, 9.5 and 9.5).
    const uint32_t lanes = std::min(d.latWords / 4u, 512u);
    const uint32_t block = std::min((std::max(d.maxColorCount, lanes) + 63u) / 64u * 64u, 1024u);
    return resident_lds_bytes(d) <= kResidentLds ? block : 0u;
}

hipError_t launch_resident(const SysDesc& d, uint32_t substeps, uint32_t block, hipStream_t st) {
    const ResidentKernel kernel = resident_kernel((d.maxColorCount + block - 1u) / block, d.maxDegree);
    const hipError_t err = allow_lds(reinterpret_cast<const void*>(kernel), resident_lds_bytes(d));
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(block), uint32_t(resident_lds_bytes(d)), st, d, substeps);
    return hipGetLastError();
}

// Eight members per thread with more than four bonds do not fit the registers
// (62 spilled; 13 us per substep for 5000 members).
bool resident_fits(const SysDesc& d) {
    return d.maxColorCount != 0u && d.maxColorCount <= (d.maxDegree <= 4u ? 8u : 5u) * 1024u && d.lone == 0u &&
           resident_lds_bytes(d) <= kResidentLds;
}

// Measured, us per substep by members: up to two bonds 3840 4.3, 5120 5.7, 6400
// 7.2, 7680 8.3; up to four 4317 5.85, 4934 6.6, 5304 (eight members per thread,
// 18 registers spilled) 8.0; more 3267 6.3, 4084 7.3, 4574 8.1.
double resident_substep_us(const SysDesc& d) {
    double perMember = 1.1e-3;
    if (d.maxDegree > 4u)
        perMember = 1.55e-3;
    else if (d.maxDegree > 2u)
        perMember = d.maxColorCount <= 5u * 1024u ? 1.25e-3 : 1.35e-3;
    return 1.0 + perMember * double(d.maxColorCount);
}
// More bonds: up to the same time.  Four two-pass replicas take 6.5 us per substep
// with up to four bonds (byte lattice 6.9), 6.8 (7.4) with more.
bool resident_always(const SysDesc& d) {
    SysDesc chain{};
    chain.maxDegree = 2u;
    chain.maxColorCount = kResidentInBatch;
    return resident_substep_us(d) <= resident_substep_us(chain);
}

void add_to_class(ResidentClass& c, const SysDesc& d) {
    const uint32_t rounds = batch_rounds(d.maxColorCount, c.block), degree = d.maxDegree <= 2u ? 2u : (d.maxDegree <= 4u ? 4u : 8u);
    c.mixed = c.mixed || (c.count != 0u && (rounds != c.rounds || degree != c.maxDegree));
    c.rounds = rounds;
    c.maxDegree = degree;
    c.lds = std::max(c.lds, uint32_t(resident_lds_bytes(d)));
    ++c.count;
}

hipError_t launch_resident_batch(const SysDesc* descs, const uint32_t* ids, const ResidentClass& c, uint32_t substeps,
                                 hipStream_t st) {
    if (c.count == 0u) return hipSuccess;
    const ResidentBatchKernel kernel = resident_batch_kernel(c);
    const hipError_t err = allow_lds(reinterpret_cast<const void*>(kernel), c.lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(kernel, dim3(c.count), dim3(c.block), c.lds, st, descs, ids + c.first, substeps);
    return hipGetLastError();
}

}  // namespace pscbfm
