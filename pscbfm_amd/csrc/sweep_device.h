// Device-side pieces that the sweep kernels share: the state of a launch, a
// move's direction and geometry, and the test of its front plane.
#pragma once

#include "kernels.h"

namespace pscbfm {

namespace {

// Every device buffer is reached through a global-address-space pointer.
// The batch kernels read their buffer pointers from a descriptor table in
// memory, which leaves the compiler generic (FLAT) pointers: on gfx950 the
// waits it then places before using FLAT-loaded gather results proved
// insufficient under load (a few lanes consumed words that had not arrived;
// a full s_waitcnt after the gathers removed the divergence).  GLOBAL
// instructions, which the single-system kernels always get, are tracked by
// the vector-memory counter alone.
template <class T>
__device__ __forceinline__ gptr<T> global_ptr(T* p) {
    return (gptr<T>)p;
}

// What a sweep launch reads from its system's state, taken as four 16-byte
// loads of the whole 64-byte record before any branch, so that the start of
// every workgroup waits for one round trip: the substep it serves (device
// counter + k), the stop point, the draw source and the per-substep log and
// accepted-count pointers.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Launch {
    uint64_t t;
    SubstepDraw draw;
    gptr<uint32_t> log;
    uint64_t logFirst, logCapacity;
    gptr<uint64_t> acceptedByBlock;
};

__device__ __forceinline__ uint64_t join64(uint32_t lo, uint32_t hi) { return uint64_t(lo) | (uint64_t(hi) << 32); }

// What a kernel loads ahead of its branch on the state, and waits for with the
// state.  The compiler moves such loads behind the branch, a round trip later;
// as operands of an empty statement between the state's loads and the branch
// they stay in front of it.
struct Early {
    uint32_t count = 0;  // pass 2: length of the list and the thread's first entry
    uint64_t entry = 0;
    // a field of each line of the descriptor
    gptr<const ColorInfo> colors = nullptr;
    gptr<const uint32_t> key = nullptr;
    uint32_t mask = 0;
};
__device__ __forceinline__ Early early_of(const SysDesc& d, bool key) {
    Early e;
    e.colors = d.colors.global();
    if (key) e.key = d.key.global();
    e.mask = d.mask[0];
    return e;
}

// False when substep t is at or past the stop point.  Else fills `out`, whose
// pointers the host checked (DeviceSystem::writeState); the
// draw is entry t - drawBase of the explicit table when the state holds one,
// else the counter draw of (seed, t).
__device__ __forceinline__ bool begin_substep(gptr<const DevState> state, uint64_t seed, uint32_t nColors, uint32_t k,
                                              const Early& early, Launch& out) {
    const cptr<u32x4> w = (cptr<u32x4>)state;
    const u32x4 w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];  // DevState field order
    uint64_t t = join64(w0.x, w0.y);
    asm volatile("" : "+s"(t) : "v"(early.count), "v"(early.entry), "s"(early.colors), "s"(early.key), "s"(early.mask),
                 "s"(seed), "s"(nColors), "s"(k), "s"(w1.x), "s"(w2.x), "s"(w3.x));
    t += k;
    if (t >= join64(w0.z, w0.w)) return false;
    out.t = t;
    const uint64_t table = join64(w1.x, w1.y);
    if (table == 0u) {
        out.draw = substep_draw(seed, t, nColors);
    } else {
        // every lane reads the same entry: keep the draw in scalar registers
        const uint64_t e = global_ptr(reinterpret_cast<const uint64_t*>(uintptr_t(table)))[t - join64(w1.z, w1.w)];
        out.draw.species = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(e));
        out.draw.seed = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(e >> 32));
    }
    out.log = (gptr<uint32_t>)(uintptr_t(join64(w2.x, w2.y)));
    out.logFirst = join64(w2.z, w2.w);
    out.logCapacity = join64(w3.x, w3.y);
    out.acceptedByBlock = (gptr<uint64_t>)(uintptr_t(join64(w3.z, w3.w)));
    return true;
}

__device__ __forceinline__ bool begin_substep(const SysDesc& d, uint32_t k, const Early& early, Launch& out) {
    return begin_substep(d.state.global(), d.seed, d.nColors, k, early, out);
}

// Species record, read word by word.
__device__ __forceinline__ ColorInfo load_color(gptr<const ColorInfo> colors, uint32_t species) {
    const cptr<uint32_t> w = (cptr<uint32_t>)(colors + species);
    ColorInfo c{};
    c.slotOffset = w[offsetof(ColorInfo, slotOffset) / 4];
    c.count = w[offsetof(ColorInfo, count) / 4];
    c.nbrOffset = w[offsetof(ColorInfo, nbrOffset) / 4];
    c.nbrPitch = w[offsetof(ColorInfo, nbrPitch) / 4];
    c.maxDegree = w[offsetof(ColorInfo, maxDegree) / 4];
    c.idsOffset = w[offsetof(ColorInfo, idsOffset) / 4];
    c.idWords = w[offsetof(ColorInfo, idWords) / 4];
    return c;
}

// The Z-curve masks of x, y and z as values in scalar registers.  Passing
// the descriptor's array instead lets the compiler turn the per-lane choice
// of an axis into a per-lane load from the argument segment, one more
// dependent round trip in front of the lattice reads.
struct AxisMasks {
    uint32_t x, y, z;
};
__device__ __forceinline__ AxisMasks axis_masks(const SysDesc& d) {
    AxisMasks m;
    m.x = uint32_t(__builtin_amdgcn_readfirstlane(d.mask[0]));
    m.y = uint32_t(__builtin_amdgcn_readfirstlane(d.mask[1]));
    m.z = uint32_t(__builtin_amdgcn_readfirstlane(d.mask[2]));
    return m;
}

// A move's axis and sign.  Direction d: 0:-x 1:+x 2:-y 3:+y 4:-z 5:+z
// (UpdaterGPUScBFM_AB_Type.cu:534-545); two flags name the axis.
struct Dir {
    bool x, z;  // axis x, axis z (else y)
    bool plus;
    __device__ __forceinline__ uint32_t number() const { return (x ? 0u : (z ? 4u : 2u)) + (plus ? 1u : 0u); }
};
__device__ __forceinline__ Dir dir_of_number(uint32_t d) { return {d < 2u, d >= 4u, (d & 1u) != 0u}; }
// Direction rn % 6 of a hash (CRITICAL.cu:321-323).  rn % 6 is
// 2 * ((rn >> 1) % 3) + (rn & 1).  h = rn >> 1 is the sum t of its low 16 and
// its other bits modulo 3 (2^16 = 1 modulo 3), t < 2^17, and t % 3 is read off
// the fraction t / 3: with c = ceil(2^25 / 3), 128 t c modulo 2^32 is
// r / 3 of the range plus less than 2^24, for t = 3q + r.  One full-rate 24-bit
// multiply and two compares, whose results are the axis flags themselves.
__device__ __forceinline__ Dir dir_of_hash(uint32_t rn) {
    uint32_t t = ((rn >> 17) + ((rn >> 1) & 0xFFFFu)) << 7;
    asm("" : "+v"(t));  // else the shift moves to the constant, which then needs a quarter-rate 32-bit multiply
    const uint32_t f = __umul24(t, 0xAAAAABu);
    return {f < 0x55555555u, f >= 0xAAAAAAAAu, (rn & 1u) != 0u};
}

struct Move {
    uint32_t to;                  // code of the new corner
    uint32_t c00, c02, c20, c22;  // bytes to the words with the corner cells of the 3x3 plane in front: (u-1, v-1),
                                  // (u-1, v+1), (u+1, v-1), (u+1, v+1)
};

// Front plane: p + 2 e_d + a e_u + b e_v, a,b in {-1,0,1} (CRITICAL.cu:62-176),
// with (u, v) = (y, z), (x, z), (x, y) for a move along x, y, z.  The lowest
// code bits of x, y and z are bits 0, 1 and 2, their second bits 3, 4 and 5.
// The words hold 2^SHIFT cells in eight bytes: a cell's word is its code
// without the low SHIFT bits, at that code >> (SHIFT - 3) in bytes.
template <int SHIFT>
__device__ __forceinline__ Move make_move(uint32_t m, const Dir& d, const AxisMasks& mask) {
    const uint32_t Ma = d.x ? mask.x : (d.z ? mask.z : mask.y);
    const uint32_t Mu = d.x ? mask.y : mask.x;
    const uint32_t Mv = d.z ? mask.y : mask.z;
    const uint32_t oneA = d.x ? 1u : (d.z ? 4u : 2u);
    const uint32_t oneU = d.x ? 2u : 1u, oneV = d.z ? 2u : 4u;
    const uint32_t step1 = d.plus ? oneA : Ma;              // +1 or -1 in dilated form
    const uint32_t step2 = d.plus ? oneA << 3 : Ma ^ oneA;  // +2 or -2
    Move mv;
    const uint32_t ta = m | ~Ma, tu = m | ~Mu, tv = m | ~Mv;
    mv.to = (m & ~Ma) | ((ta + step1) & Ma);
    constexpr uint32_t words = ~((1u << SHIFT) - 1u);
    const uint32_t fa = (ta + step2) & Ma & words;
    const uint32_t u0 = (tu + Mu) & Mu & words, u2 = (tu + oneU) & Mu & words;
    const uint32_t v0 = (tv + Mv) & Mv & words, v2 = (tv + oneV) & Mv & words;
    mv.c00 = (fa | u0 | v0) >> (SHIFT - 3);
    mv.c02 = (fa | u0 | v2) >> (SHIFT - 3);
    mv.c20 = (fa | u2 | v0) >> (SHIFT - 3);
    mv.c22 = (fa | u2 | v2) >> (SHIFT - 3);
    return mv;
}

// Whether the axis coordinate of a move crosses the periodic boundary.
__device__ __forceinline__ bool wraps(uint32_t m, const Dir& d, const AxisMasks& mask) {
    const uint32_t Ma = d.x ? mask.x : (d.z ? mask.z : mask.y);
    return (m & Ma) == (d.plus ? Ma : 0u);
}

// All ones when bit b of m is set, else 0.
__device__ __forceinline__ uint32_t spread_bit(uint32_t m, uint32_t b) {
    return uint32_t(__builtin_amdgcn_sbfe(int32_t(m), b, 1));
}

// Whether any of the nine front-plane cells is set, read as 64-bit words.
// The low code bits interleave x, y and z, so a 64-bit word of the 1-bit
// lattice (64 cells, SHIFT 6) is an aligned 4x4x4 block and one of the byte
// lattice (8 cells, SHIFT 3) an aligned 2x2x2 block.  In either case the 3x3
// plane touches at most four words, those of its corner cells, and four
// 8-byte gathers replace nine narrow ones.
//
// The cells are picked from the words with masks, in 32-bit halves.  (Nine
// 64-bit shifts, one per cell, took 65 VALU instructions per move; this takes
// about 35.)
//  * 4x4x4 words: the plane's own coordinate is a +- 2, the same residue
//    modulo 4 for both signs, and its transverse coordinates are all residues
//    but that of u + 2 (v + 2).  So with E_k = the cells whose coordinate k
//    has the residue of m's plus 2, the plane is E_a & ~E_u & ~E_v.  A cell of
//    residue 2 or 3 in u lies in the word of u-1, one of residue 0 or 1 in
//    that of u+1 (where the two differ), so the words are merged by constant
//    masks of the second coordinate bit: first over v, then over u.
//  * 2x2x2 words: the plane has the residue of a; the word of u-1 holds only
//    residue 1 of the plane when u is even, that of u+1 only residue 0 when u
//    is odd, and both residues otherwise.
struct PlaneMask {
    uint32_t low, high;      // cells of the plane in the halves of a word
    uint32_t u, vLow, vHigh; // cells of the words of u-1 (v-1), against u+1 (v+1)
};
// 4x4x4 words.
__device__ __forceinline__ PlaneMask plane_mask(uint32_t m, const Dir& d) {
    const uint32_t sx = spread_bit(m, 0), sy = spread_bit(m, 1), sz = spread_bit(m, 2);
    const uint32_t tx = spread_bit(m, 3), ty = spread_bit(m, 4), tz = spread_bit(m, 5);
    // E_x and E_y are alike in both halves; E_z's second bit is the half itself
    const uint32_t ex = (0x55555555u ^ sx) & (0xFF00FF00u ^ tx);
    const uint32_t ey = (0x33333333u ^ sy) & (0xFFFF0000u ^ ty);
    const uint32_t ez = 0x0F0F0F0Fu ^ sz;
    const uint32_t nx = d.x ? 0u : ~0u, nz = d.z ? 0u : ~0u, ny = d.x || d.z ? ~0u : 0u;
    const uint32_t exy = (ex ^ nx) & (ey ^ ny);
    PlaneMask p;
    p.low = ((ez & tz) ^ nz) & exy;
    p.high = ((ez & ~tz) ^ nz) & exy;
    p.u = d.x ? 0xFFFF0000u : 0xFF00FF00u;
    p.vLow = d.z ? 0xFFFF0000u : 0u;
    p.vHigh = d.z ? 0xFFFF0000u : ~0u;
    return p;
}
__device__ __forceinline__ bool merged_any(uint64_t w00, uint64_t w02, uint64_t w20, uint64_t w22, const PlaneMask& p) {
    auto pick = [](uint32_t s, uint32_t a, uint32_t b) { return (a & s) | (b & ~s); };
    const uint32_t low = pick(p.u, pick(p.vLow, uint32_t(w00), uint32_t(w02)), pick(p.vLow, uint32_t(w20), uint32_t(w22)));
    const uint32_t high = pick(p.u, pick(p.vHigh, uint32_t(w00 >> 32), uint32_t(w02 >> 32)),
                               pick(p.vHigh, uint32_t(w20 >> 32), uint32_t(w22 >> 32)));
    return ((low & p.low) | (high & p.high)) != 0u;
}
// The element `bytes` behind a base that is the same for every lane, by a 32-bit offset
// (an index scaled in 64 bits costs three or four instructions more).
template <class T>
__device__ __forceinline__ T at(gptr<const T> base, uint32_t bytes) {
    return *(gptr<const T>)((gptr<const char>)base + bytes);
}
struct PlaneWords {
    uint64_t w00, w02, w20, w22;
};
__device__ __forceinline__ PlaneWords plane_words(gptr<const uint64_t> words, const Move& mv) {
    return {at(words, mv.c00), at(words, mv.c02), at(words, mv.c20), at(words, mv.c22)};
}
// Either kind of words.
template <int SHIFT>
__device__ __forceinline__ bool plane_any(const PlaneWords& p, uint32_t m, const Dir& d) {
    const uint64_t w00 = p.w00, w02 = p.w02, w20 = p.w20, w22 = p.w22;
    if constexpr (SHIFT == 6) {
        return merged_any(w00, w02, w20, w22, plane_mask(m, d));
    } else {
        const uint32_t a0 = uint32_t(w00), a1 = uint32_t(w00 >> 32), b0 = uint32_t(w02), b1 = uint32_t(w02 >> 32);
        const uint32_t c0 = uint32_t(w20), c1 = uint32_t(w20 >> 32), e0 = uint32_t(w22), e1 = uint32_t(w22 >> 32);
        const uint32_t sx = spread_bit(m, 0), sy = spread_bit(m, 1), sz = spread_bit(m, 2);
        const uint32_t lx = 0xFF00FF00u | sx, hx = ~(0xFF00FF00u & sx);
        const uint32_t ly = 0xFFFF0000u | sy, hy = ~(0xFFFF0000u & sy);
        const uint32_t ul = d.x ? ly : lx, uh = d.x ? hy : hx;
        const uint32_t vl0 = d.z ? ly : sz, vl1 = d.z ? ly : ~0u;
        const uint32_t vh0 = d.z ? hy : ~0u, vh1 = d.z ? hy : ~sz;
        const uint32_t pxy = d.x ? 0x00FF00FFu ^ sx : 0x0000FFFFu ^ sy;
        const uint32_t plane0 = d.z ? ~sz : pxy, plane1 = d.z ? sz : pxy;
        const uint32_t any0 = (((a0 & vl0) | (b0 & vh0)) & ul) | (((c0 & vl0) | (e0 & vh0)) & uh);
        const uint32_t any1 = (((a1 & vl1) | (b1 & vh1)) & ul) | (((c1 & vl1) | (e1 & vh1)) & uh);
        return ((any0 & plane0) | (any1 & plane1)) != 0u;
    }
}

template <int SHIFT>
__device__ __forceinline__ bool plane_any(gptr<const uint64_t> words, uint32_t m, const Dir& d, const Move& mv) {
    return plane_any<SHIFT>(plane_words(words, mv), m, d);
}

// Rank of this lane among the lanes of its wave whose bit is set in `mask`.
__device__ __forceinline__ uint32_t lane_rank(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}

}  // namespace

}  // namespace pscbfm
