// Multispin core of the Ising colour passes (sc, bcc, fcc): 32 sites of a row
// per 32-bit word, bit j of every word below being position i0 + j.
//
// A site's flip is accepted when dE <= 0, or else when its 32-bit draw k is
// below ceil(exp(-dE/T) * 2^32) (the reference's `u < exp(-dE/T)`,
// src/integrator.rs:127-134, with u quantised to 2^-32).  With g absent
// neighbour slots and p = Z - g present, dE depends on the site's bit b and
// on a, the number of present neighbours equal to it.  The passes form a in
// bit planes (carry-save adders over the neighbour words) and decide() takes
// it from there:
//   - the host lists, per g and a, the classes (b, a) that are not always
//     accepted with their threshold's high byte (ChainDev::plan; at h = 0 in
//     a ferromagnet one slot for each a > Z / 2).  A listed class's site mask
//     is one or two bit operations on the planes of a, and adds the byte's
//     eight bits to eight threshold planes: each site then has its own
//     threshold byte, bit k in plane k;
//   - one bit-serial comparison (eight v_bitop3 from the least significant
//     bit) of the draws' high bytes, also in planes, with the threshold
//     planes gives every listed site below its threshold, eight more those
//     equal to it.  Per listed class that is 10 operations and 16 in all; a
//     comparison of its own for each class took 19 per class (the sc pass of
//     256^3 x 3 with three classes: 57 operations a word against 46);
//   - sites whose high byte ties the threshold's (2^-8) are settled by the
//     low 24 bits of their draw: they leave a record (slot by ballot) in the
//     wave's LDS queue, and once the wave has finished its planes one lane
//     per record draws them, stores the settled word and corrects the sums.
//     The result equals comparing the full 32-bit draws.
//
// The draws' high bytes: sc slices the two Philox calls of a word by bit (bit
// k of site j's byte is bit j of word k), so the calls' words are the planes.
// bcc and fcc take whole bytes (byte pos & 3 of word (pos & 15) >> 2 of the
// call of pos >> 4); draw_planes() transposes a word's 32 bytes into planes:
// 64 operations per 32 sites, and everything after them is as in sc.  (The
// byte-wise decision this replaced, four sites per register, took 24 lane
// instructions a site on bcc 160^3 x 3 at tile 2 and 25 to 28 on fcc 128^3 x
// 3, against 12 and 13 to 15.)
#pragma once

#include "vg_device.hpp"

namespace vg {

// Boundaries of a pass's chains.  kPeriodic: periodic along every axis, where
// no slot is absent and every boundary term folds away; a launch takes it when
// all its chains are.  (The planes hold one bit per site whatever the chain's
// spin kind.)
enum IsingMode : uint32_t { kOpen = 1, kPeriodic = 2 };

constexpr uint32_t kWaves = kBlock / 64;
constexpr uint32_t kTieRows = 128;  // tie records per wave (one per word with ties)
// A record: row, first position, edge, tie mask, site bits, count planes (3 or
// 4), lower-colour count planes (fcc: up to 4).
constexpr uint32_t kTieHead = 5;

// Bitwise function of three words given by its truth table: bit i of TT is
// the result for (a, b, c) = (i >> 2 & 1, i >> 1 & 1, i & 1).  One v_bitop3.
template <uint32_t TT>
__device__ __forceinline__ uint32_t bop3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, TT);
}
constexpr uint32_t kXor3 = 0x96;  // a ^ b ^ c
constexpr uint32_t kMaj3 = 0xE8;  // at least two of a, b, c
constexpr uint32_t kSel = 0xE4;   // c ? a : b

// A word of a plane; kNoRow reads 0.
__device__ __forceinline__ uint32_t load_word(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
}

// One position of a row: byte offset of its word, and its bit there.
struct XPos {
    uint32_t off, sh;
};
__device__ __forceinline__ XPos xpos(uint32_t i) { return XPos{(i >> 5) << 2, i & 31u}; }

// The high bytes of the draws of a word's 32 sites (ca, cb: the Philox calls
// of its two halves; site 4k + m is byte m of word k of ca, cb) as planes:
// bit s of d[p] is bit p of site s's byte.  Seen as a 256-bit array indexed by
// (word k2 k1 k0, byte m1 m0, bit p2 p1 p0), each step exchanges one index
// bit of the word with one of the position in the word: m1 and m0 by byte
// permutes, then p2, p1, p0 by shifts of 4, 2 and 1 under a mask.
__device__ __forceinline__ void draw_planes(const U4& ca, const U4& cb, uint32_t d[8]) {
    const uint32_t w[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
    uint32_t x[8], y[8], z[8], v[8];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {  // word bit 2 <-> halfword
        x[k] = __builtin_amdgcn_perm(w[k + 4], w[k], 0x05040100u);
        x[k + 4] = __builtin_amdgcn_perm(w[k + 4], w[k], 0x07060302u);
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; k += (k & 1u) ? 3u : 1u) {  // word bit 1 <-> byte: k = 0,1,4,5
        y[k] = __builtin_amdgcn_perm(x[k + 2], x[k], 0x06020400u);
        y[k + 2] = __builtin_amdgcn_perm(x[k + 2], x[k], 0x07030501u);
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; k += 2) {  // word bit 0 <-> nibble
        z[k] = bop3<kSel>(y[k], y[k + 1] << 4, 0x0F0F0F0Fu);
        z[k + 1] = bop3<kSel>(y[k] >> 4, y[k + 1], 0x0F0F0F0Fu);
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {  // word bit 2 <-> bit pair
        v[k] = bop3<kSel>(z[k], z[k + 4] << 2, 0x33333333u);
        v[k + 4] = bop3<kSel>(z[k] >> 2, z[k + 4], 0x33333333u);
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; k += (k & 1u) ? 3u : 1u) {  // word bit 1 <-> bit
        z[k] = bop3<kSel>(v[k], v[k + 2] << 1, 0x55555555u);
        z[k + 2] = bop3<kSel>(v[k] >> 1, v[k + 2], 0x55555555u);
    }
    // word index now (p1, p0, p2)
#pragma unroll
    for (uint32_t p = 0; p < 8; ++p) d[p] = z[((p >> 1) & 1u) * 4u + (p & 1u) * 2u + (p >> 2)];
}

// Planes of a count 0..Z.
template <uint32_t Z>
constexpr uint32_t kPlanes = Z == 6 ? 3u : 4u;

// Sites whose count (planes a) is N.
template <uint32_t Z, uint32_t N>
__device__ __forceinline__ uint32_t count_is(const uint32_t* a) {
    if constexpr (kPlanes<Z> == 3) return bop3<(1u << N)>(a[2], a[1], a[0]);
    const uint32_t hi = bop3<(1u << (N >> 1))>(a[3], a[2], a[1]);
    return (N & 1u) ? hi & a[0] : hi & ~a[0];
}

// The threshold byte of one plan slot (bits 0-7 the byte, 8 covers b = 0, 9
// covers b = 1) into the threshold planes of its sites.
__device__ __forceinline__ void plan_slot(uint32_t slot, uint32_t e, uint32_t o, uint32_t no,
                                          uint32_t t[8], uint32_t& listed) {
    const uint32_t cover = (slot >> 8) & 3u;
    uint32_t m = e;
    if (cover != 3u) {  // a scalar branch (the asm keeps it one)
        m &= cover == 2u ? o : no;
        asm volatile("" : "+v"(m));
    }
    listed |= m;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) t[k] |= m & (0u - ((slot >> k) & 1u));
}

template <uint32_t Z, uint32_t N>
__device__ __forceinline__ void plan_counts(const uint32_t* pw, const uint32_t* a, uint32_t o,
                                            uint32_t no, uint32_t t[8], uint32_t& listed) {
    if (pw[N]) {
        const uint32_t e = count_is<Z, N>(a);
        plan_slot(pw[N], e, o, no, t, listed);
        if (pw[N] >> 16) plan_slot(pw[N] >> 16, e, o, no, t, listed);
    }
    if constexpr (N > 0) plan_counts<Z, N - 1>(pw, a, o, no, t, listed);
}

// Decision of the sites in `live` under the plan pw (one absent count): the
// accepted sites (ties excluded) and the tied ones.  A listed class whose
// threshold is zero may tie too; its tie is then never accepted.
template <uint32_t Z>
__device__ __forceinline__ void decide(const uint32_t* plan, const uint32_t* a, uint32_t o,
                                       uint32_t no, const uint32_t d[8], uint32_t live,
                                       uint32_t& acc, uint32_t& tie) {
    // The plan's words, loaded together.  The empty asm statements keep the
    // compiler from computing every slot's bit masks ahead of the z march
    // (eight registers a slot: it spilled them into vector lanes).
    uint32_t pw[Z + 1];
#pragma unroll
    for (uint32_t k = 0; k <= Z; ++k) pw[k] = plan[k];
#pragma unroll
    for (uint32_t k = 0; k <= Z; ++k) asm volatile("" : "+s"(pw[k]));
    uint32_t t[8] = {0, 0, 0, 0, 0, 0, 0, 0}, listed = 0;
    plan_counts<Z, Z>(pw, a, o, no, t, listed);
    // d < t bit-serially from the least significant bit: at bit k,
    // lt = (~d & t) | (~(d ^ t) & lt)
    uint32_t lt = 0u, eq = listed & live;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) lt = bop3<0x8E>(d[k], t[k], lt);
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) eq = bop3<0x90>(eq, d[k], t[k]);  // eq & ~(d ^ t)
    acc = bop3<0xB0>(live, listed, lt);  // live & ~(listed & ~lt)
    tie = eq;
}

// The plan of a ferromagnet without a field (ChainDev::plain, g = 0): the
// classes a > Z / 2 are listed, one threshold byte for both bits, and no
// other.  sm[i] holds the byte of a = Z / 2 + 1 + i as eight whole-word masks
// in vector registers; a listed site's threshold plane k is then a choice
// among the masks k by the planes of a (2, 3 or 5 selections), with no class
// masks, scalar bit extractions or branches.  An instruction of a wave takes
// 8 cycles to the next whatever its kind, so the scalar work of the general
// plan costs as much as its vector work: sc 256^3 x 3 (three waves a SIMD)
// 8.2 us a pass with the general plan, 7.2 with this one.  (The same with
// masks for each bit, for chains in a field, took 64 to 112 registers and
// with them the occupancy of every chain: sc 1024^3 84 -> 95 us, and the
// mixed scan in fields 12.3 -> 13.7 us; those take the general plan.)
template <uint32_t Z>
__device__ __forceinline__ void decide_plain(const uint32_t (*sm)[8], const uint32_t* a,
                                             const uint32_t d[8], uint32_t live, uint32_t& acc,
                                             uint32_t& tie) {
    uint32_t listed;
    if constexpr (Z == 6)
        listed = a[2];  // 4, 5, 6
    else if constexpr (Z == 8)
        listed = bop3<0xF8>(a[3], a[2], a[1] | a[0]);  // 8, or 5..7
    else
        listed = bop3<0xF8>(a[3], a[2], a[1] & a[0]);  // 8..12, or 7
    uint32_t lt = 0u, eq = listed & live;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        uint32_t t;
        if constexpr (Z == 6) {
            t = bop3<kSel>(sm[2][k], bop3<kSel>(sm[1][k], sm[0][k], a[0]), a[1]);
        } else if constexpr (Z == 8) {
            const uint32_t t67 = bop3<kSel>(sm[2][k], sm[1][k], a[0]);
            t = bop3<kSel>(sm[3][k], bop3<kSel>(t67, sm[0][k], a[1]), a[3]);
        } else {
            const uint32_t t89 = bop3<kSel>(sm[2][k], sm[1][k], a[0]);
            const uint32_t tab = bop3<kSel>(sm[4][k], sm[3][k], a[0]);
            const uint32_t t8b = bop3<kSel>(tab, t89, a[1]);
            t = bop3<kSel>(bop3<kSel>(sm[5][k], t8b, a[2]), sm[0][k], a[3]);
        }
        lt = bop3<0x8E>(d[k], t, lt);
        eq = bop3<0x90>(eq, d[k], t);
    }
    acc = bop3<0xB0>(live, listed, lt);
    tie = eq;
}

// Draws before loads: the draws do not wait for a plane's loads, but left to
// itself the compiler puts uses of the loads, and with them the wait, first.
// Empty asm statements keep their order: draws, then the loaded words (each
// `arrived` one).
__device__ __forceinline__ void keep_draws(uint32_t d[8]) {
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) asm volatile("" : "+v"(d[j]));
}
__device__ __forceinline__ uint32_t arrived(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Low 24 bits of a tied draw decide: accept iff they are below the low 24
// bits of the threshold.  The draw of position pos is word pos & 3 of the
// call (pos >> 2, row, sweep, purpose IsingB).
__device__ __forceinline__ bool tie_accept(const uint32_t* thr, uint32_t bj, uint32_t S,
                                           uint32_t pos, uint32_t row, uint64_t t, uint32_t colour,
                                           uint32_t k0, uint32_t k1) {
    const U4 rb = philox(U4{pos >> 2, row, (uint32_t)t, ctr_w(t, kIsingB, colour)}, k0, k1);
    return (u4_word(rb, pos & 3u) >> 8) < (thr[bj * kThrS + S] & 0xFFFFFFu);
}

// What the boundaries do to a word's sites: g absent slots at every site,
// ge more at position xe (32: none).  Bonds to lower colours (fcc): pl
// present ones, me fewer at xe.
struct Edge {
    uint32_t g, ge, xe, pl, me;
};

// Settles the tied sites tm of one word: site j has bit b = bit j of ob and
// aligned count a (planes), so u = a (b = 1) or p - a (b = 0) up neighbours
// and class S = 2u + g.  Returns the accepted flips; dm, db collect their
// magnetisation and bond changes.  BOND: 0 none, 1 all neighbours are of
// lower colours, 2 their up count is in the planes l.
template <uint32_t Z, uint32_t BOND>
__device__ __forceinline__ uint32_t settle(const uint32_t* thr, uint32_t tm, const uint32_t* a,
                                           const uint32_t* l, uint32_t ob, const Edge& ed,
                                           uint32_t i0, uint32_t row, uint64_t t, uint32_t colour,
                                           bool bonds, uint32_t k0, uint32_t k1, int32_t& dm,
                                           int32_t& db) {
    uint32_t flips = 0;
    while (tm) {
        const uint32_t j = __builtin_ctz(tm);
        tm &= tm - 1u;
        const uint32_t bj = (ob >> j) & 1u;
        uint32_t av = 0;
#pragma unroll
        for (uint32_t k = 0; k < kPlanes<Z>; ++k) av |= ((a[k] >> j) & 1u) << k;
        const bool edge = j == ed.xe;
        const uint32_t g = ed.g + (edge ? ed.ge : 0u);
        const uint32_t S = 2u * (bj ? av : Z - g - av) + g;
        if (tie_accept(thr, bj, S, i0 + j, row, t, colour, k0, k1)) {
            flips |= 1u << j;
            const int32_t ds = 2 - 4 * (int32_t)bj;
            dm += ds;
            if (BOND == 1 && bonds) db += ds * ((int32_t)S - (int32_t)Z);
            if (BOND == 2) {
                uint32_t lv = 0;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) lv |= ((l[k] >> j) & 1u) << k;
                db += ds * (2 * (int32_t)lv - (int32_t)(ed.pl - (edge ? ed.me : 0u)));
            }
        }
    }
    return flips;
}

// Record words of a pass: its count planes, and lower-colour planes where the
// bonds need their own (BOND = 2).
template <uint32_t Z, uint32_t BOND>
constexpr uint32_t kRecWords = kTieHead + kPlanes<Z> + (BOND == 2 ? 4u : 0u);

// The descriptor fields of a pass and its place in the work.
struct PassHead {
    uint64_t t, off[4];
    uint32_t k0, k1, ly, lz, w, pitch, pbc, segs, segs_m, segs_s, ly_m, ly_s, plane, items;
    bool rnd;
    bool plain;      // ChainDev::plain
    bool active;     // the workgroup belongs to a chain that runs this sweep
    uint32_t block;  // logical workgroup
    uint32_t local;  // work item in the chain
    bool go;         // this lane has an item
    uint32_t seg, y, zc;  // its segment, row in the plane and z chunk
};

// The chain of logical workgroup b (clamped to the work): from the block ->
// chain map, or, when every chain has the same number of workgroups, by
// dividing by it -- multiply by m and shift (opts bits 16-21), m = 0 for the
// map.  A wave's start is a chain of scalar loads; this takes one out.
__device__ __forceinline__ const ChainDev& pass_chain(const ChainDev* __restrict__ chains,
                                                      const uint32_t* __restrict__ block_chain,
                                                      uint32_t b, uint32_t total_blocks,
                                                      uint32_t opts, uint32_t m) {
    const uint32_t bc = min(b, total_blocks - 1u);
    return chains[m ? fast_div(bc, m, (opts >> 16) & 63u) : block_chain[bc]];
}

// Workgroups past the work (the grid is a multiple of 8) and chains that run
// fewer sweeps in this block do nothing; they are not sent away at the start
// so that the descriptor's leading fields (all but the tables) are loaded in
// one batch: a pass is short, and a chain of dependent loads at its start is
// a good part of it.  Items in natural order: segments of a row, rows y of a
// z chunk, chunks; rows y and y+1 of one plane are neighbours in memory and
// in the grid.
__device__ __forceinline__ PassHead pass_head(const ChainDev& C, uint32_t b, uint32_t total_blocks,
                                              uint32_t s) {
    constexpr uint32_t kHead = offsetof(ChainDev, thr) / 4u;
    uint32_t hd[kHead];
#pragma unroll
    for (uint32_t k = 0; k < kHead; ++k) hd[k] = reinterpret_cast<const uint32_t*>(&C)[k];
#define VG_FIELD(f) hd[offsetof(ChainDev, f) / 4u]
#define VG_FIELD64(f) \
    (((uint64_t)hd[offsetof(ChainDev, f) / 4u + 1u] << 32) | hd[offsetof(ChainDev, f) / 4u])
    PassHead h;
    h.active = b < total_blocks && s < VG_FIELD(limit);
    h.t = VG_FIELD64(sweep0) + s;
    h.k0 = hd[offsetof(ChainDev, seed) / 4u];
    h.k1 = hd[offsetof(ChainDev, seed) / 4u + 1u];
    h.off[0] = VG_FIELD64(off[0]);
    h.off[1] = VG_FIELD64(off[1]);
    h.off[2] = VG_FIELD64(off[2]);
    h.off[3] = VG_FIELD64(off[3]);
    h.plane = (uint32_t)VG_FIELD64(plane);  // below 4 GiB (checked on the host)
    h.ly = VG_FIELD(ly);
    h.lz = VG_FIELD(lz);
    h.w = VG_FIELD(w);
    h.pitch = VG_FIELD(pitch);
    h.pbc = VG_FIELD(pbc);
    h.items = VG_FIELD(items);
    h.segs = VG_FIELD(segs);
    h.segs_m = VG_FIELD(segs_m);
    h.segs_s = VG_FIELD(segs_s);
    h.ly_m = VG_FIELD(ly_m);
    h.ly_s = VG_FIELD(ly_s);
    h.rnd = VG_FIELD(proposal) != 0;
    h.plain = VG_FIELD(plain) != 0;
    h.block = b;
    h.local = (b - VG_FIELD(block0)) * kBlock + threadIdx.x;
#undef VG_FIELD
#undef VG_FIELD64
    h.go = h.active && h.local < h.items;
    const uint32_t r = fast_div(h.local, h.segs_m, h.segs_s);
    h.seg = h.local - r * h.segs;
    h.zc = fast_div(r, h.ly_m, h.ly_s);
    h.y = r - h.zc * h.ly;
    return h;
}

// A wave's march: what the planes of one pass share.
template <uint32_t Z, uint32_t BOND, uint32_t MODE>
struct March {
    static constexpr bool PER = MODE == kPeriodic;
    static constexpr uint32_t NP = kPlanes<Z>;
    static constexpr uint32_t NREC = kRecWords<Z, BOND>;

    const ChainDev& C;
    uint32_t qcap, colour, k0, k1;
    uint64_t t;
    bool rnd, bonds;  // bonds: this pass adds its bonds
    uint32_t sm[Z / 2][8];  // masks of a plain plan
    uint32_t pw[Z + 1];     // the plan of the wave's absent count
    // the lane's segment: its first position, valid positions and their mask
    uint32_t i0, nvalid, vmask;
    uint32_t nrec = 0;  // records queued by this wave, as counted by this lane
    int32_t m_part = 0, b_part = 0;
    // running popcounts: up sites; count planes over valid and over flipped
    // (BOND 1) or up (BOND 2) sites
    uint32_t ups = 0, sv[4] = {0, 0, 0, 0}, sf[4] = {0, 0, 0, 0}, nf = 0;

    __device__ __forceinline__ March(const ChainDev& chain, const PassHead& h, uint32_t opts,
                                     uint32_t c, bool with_bonds)
        : C(chain), qcap(min((opts >> 8) & 0xFFu, kTieRows)), colour(c),
          k0(h.k0), k1(h.k1), t(h.t), rnd(h.rnd), bonds(with_bonds), i0(h.seg * kIsingSeg),
          nvalid(min(kIsingSeg, h.w - i0)),
          vmask(nvalid >= 32u ? 0xFFFFFFFFu : (1u << nvalid) - 1u) {}

    // The masks of a plain plan (decide_plain).
    __device__ __forceinline__ void load_masks() {
#pragma unroll
        for (uint32_t i = 0; i < Z / 2; ++i) {
            uint32_t w = C.plan[0][Z / 2 + 1 + i];
            asm volatile("" : "+v"(w));
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                sm[i][k] = (uint32_t)__builtin_amdgcn_sbfe((int)w, k, 1);
                asm volatile("" : "+v"(sm[i][k]));
            }
        }
    }

    // The threshold table for the sites at an open x end, a copy per wave
    // (2 * kThrS <= 64 words; the wave's own LDS operations are in order).
    __device__ __forceinline__ void load_thresholds(uint32_t* thr) {
        if constexpr (!PER) {
            const uint32_t lane = threadIdx.x & 63u;
            if (lane < 2u * kThrS) thr[lane] = (&C.thr[0][0])[lane];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }

    // The absent count of the wave's words when it is one and the same for
    // every site, with its plan's words loaded ahead of the draws and the
    // plane's loads; kMixed otherwise.
    static constexpr uint32_t kMixed = ~0u;
    template <bool PLAIN>
    __device__ __forceinline__ uint32_t wave_absent(const Edge& ed) {
        uint32_t g = 0u;
        if constexpr (!PER) {
            g = (uint32_t)__builtin_amdgcn_readfirstlane((int)ed.g);
            if (__ballot(ed.g != g || ed.xe < 32u)) return kMixed;
        }
        if (!PLAIN || g != 0u) {
#pragma unroll
            for (uint32_t k = 0; k <= Z; ++k) pw[k] = C.plan[g][k];
        }
        return g;
    }

    // One word: bits o, aligned count planes a, lower-colour up-count planes l
    // (BOND 2), draw planes d, edge ed.  Stores the new word at `off` and
    // adds to the sums.
    // own: the own plane; q: the wave's tie queue; thr: the wave's threshold table
    // (load_thresholds); g: wave_absent(ed).  PLAIN: the plan of g = 0 is
    // plain.
    template <bool PLAIN>
    __device__ __forceinline__ void word(__amdgpu_buffer_rsrc_t own, uint32_t (*q)[NREC],
                                         const uint32_t* thr, uint32_t g,
                                         uint32_t o, const uint32_t* a, const uint32_t* l,
                                         const uint32_t d[8], const Edge& ed, uint32_t off,
                                         uint32_t row) {
        const uint32_t no = ~o;
        uint32_t live = vmask;
        if (rnd) {
            // Spin::rand proposes Up when its draw is below 1/2
            // (state.rs:76-84): proposal bit 0 -> Up.  A proposal equal to
            // the current spin changes nothing.
            const U4 rp = philox(U4{i0 >> 7, row, (uint32_t)t, ctr_w(t, kIsingProposal, colour)},
                                 k0, k1);
            const uint32_t wsel = (i0 >> 5) & 3u;
            const uint32_t lo = wsel & 1u ? rp.y : rp.x, hi = wsel & 1u ? rp.w : rp.z;
            live &= ~((wsel & 2u ? hi : lo) ^ o);
        }
        uint32_t acc, tie, eb = 0;
        if constexpr (!PER) eb = ed.xe < 32u ? 1u << ed.xe : 0u;
        if (PLAIN && g == 0u) {
            decide_plain<Z>(sm, a, d, live, acc, tie);
        } else if (g != kMixed) {
            decide<Z>(pw, a, o, no, d, live, acc, tie);
        } else {
            // One decision for each absent count in the wave, the sites at xe
            // apart: one lane each, from the threshold table.
            acc = 0;
            tie = 0;
            uint64_t left = __ballot(true);
            while (left) {
                const uint32_t gi = (uint32_t)__builtin_amdgcn_readlane(
                    (int)ed.g, (uint32_t)__builtin_ctzll(left));
                uint32_t ag, tg;
                const uint32_t lg = ed.g == gi ? live : 0u;
                if (PLAIN && gi == 0u)
                    decide_plain<Z>(sm, a, d, lg, ag, tg);
                else
                    decide<Z>(C.plan[gi], a, o, no, d, lg, ag, tg);
                acc |= ag;
                tie |= tg;
                left &= ~__ballot(ed.g == gi);
            }
            if (__ballot(eb != 0u)) {
                const uint32_t xe = ed.xe & 31u, gx = ed.g + ed.ge;
                uint32_t av = 0, r8 = 0;
#pragma unroll
                for (uint32_t k = 0; k < NP; ++k) av |= ((a[k] >> xe) & 1u) << k;
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) r8 |= ((d[k] >> xe) & 1u) << k;
                const uint32_t bj = (o >> xe) & 1u;
                const uint32_t S = 2u * (bj ? av : Z - gx - av) + gx;
                const bool always = ((bj ? C.always[1] : C.always[0]) >> (S & 31u)) & 1u;
                const uint32_t th = eb ? thr[bj * kThrS + S] >> 24 : 0u;
                const uint32_t ex = eb & live;
                acc = (acc & ~eb) | (always || r8 < th ? ex : 0u);
                tie = (tie & ~eb) | (!always && r8 == th ? ex : 0u);
            }
        }

        // Words with ties leave one record each in the wave's queue (their
        // tied sites keep their bits in the store below); slots by ballot.
        // When the queue is full, this lane settles them now.
        const uint64_t has = __ballot(tie != 0);
        if (has) {
            if (tie) {
                const uint32_t slot =
                    nrec + __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32),
                                                     __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
                if (slot < qcap) {
                    uint32_t* rec = q[slot];
                    rec[0] = row;
                    rec[1] = i0;
                    if constexpr (!PER)
                        rec[2] = ed.g | (ed.ge << 4) | (ed.xe << 8) | (ed.pl << 16) | (ed.me << 20);
                    rec[3] = tie;
                    rec[4] = o ^ acc;
#pragma unroll
                    for (uint32_t k = 0; k < NP; ++k) rec[kTieHead + k] = a[k];
                    if constexpr (BOND == 2) {
#pragma unroll
                        for (uint32_t k = 0; k < 4; ++k) rec[kTieHead + NP + k] = l[k];
                    }
                } else {
                    // (rare: a wave marching 8 planes near T_c queues a few
                    // dozen records against 128 slots); the sums below see
                    // the settled flips
                    int32_t dm = 0, db = 0;
                    acc |= settle<Z, BOND>(&C.thr[0][0], tie, a, l, o, ed, i0, row, t, colour,
                                           bonds, k0, k1, dm, db);
                }
            }
            nrec += __builtin_popcountll(has);
        }
        const uint32_t n = o ^ acc;
        if (acc) __builtin_amdgcn_raw_buffer_store_b32(n, own, off, 0, 0);
        const uint32_t nv = n & vmask;
        ups += __popc(nv);
        if (BOND == 1 && bonds) {
            // sum over the word's sites of s_j * (sum of its present
            // neighbours' spins) = 2a' - p, a' the count aligned with the new
            // bit: a for kept sites, p - a for flipped ones
#pragma unroll
            for (uint32_t k = 0; k < NP; ++k) {
                sv[k] += __popc(a[k] & vmask);
                sf[k] += __popc(a[k] & acc);
            }
            if constexpr (PER) {
                nf += __popc(acc);
            } else {
                const int32_t fl = (int32_t)__popc(acc);
                const int32_t xf = (acc & eb) ? 1 : 0, xk = (vmask & ~acc & eb) ? 1 : 0;
                b_part += ((int32_t)ed.g - (int32_t)Z) * ((int32_t)nvalid - 2 * fl) +
                          (int32_t)ed.ge * (xk - xf);
            }
        }
        if (BOND == 2) {
            // sum of s_j (2 l_j - pl) over the new spins, l the up neighbours
            // of lower colours and pl the present ones (fewer at xe)
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                sv[k] += __popc(l[k] & vmask);
                sf[k] += __popc(l[k] & nv);
            }
            if constexpr (!PER) {
                b_part -= (int32_t)ed.pl * (2 * (int32_t)__popc(nv) - (int32_t)nvalid);
                if (eb & vmask) b_part += (nv & eb) ? (int32_t)ed.me : -(int32_t)ed.me;
            }
        }
    }

    // Folds the running popcounts of nk planes into the sums.  pl: present
    // lower neighbours of every site (kPeriodic, BOND 2).
    __device__ __forceinline__ void fold(uint32_t nk, uint32_t pl) {
        const int32_t sites = (int32_t)(nk * nvalid);
        m_part += 2 * (int32_t)ups - sites;
        const int32_t v = (int32_t)(sv[0] + 2u * sv[1] + 4u * sv[2] + 8u * sv[3]);
        const int32_t f = (int32_t)(sf[0] + 2u * sf[1] + 4u * sf[2] + 8u * sf[3]);
        if (BOND == 1 && bonds) {
            b_part += 2 * v - 4 * f;
            if constexpr (PER) b_part -= (int32_t)Z * (sites - 2 * (int32_t)nf);
        }
        if (BOND == 2) {
            b_part += 4 * f - 2 * v;
            if constexpr (PER) b_part -= (int32_t)pl * (2 * (int32_t)ups - sites);
        }
    }

    // Settles the wave's queued ties: one lane per record draws the low 24
    // bits of each tied site, stores the settled word and corrects the sums.
    // The wave's own row stores must land first.  nrec grows by ballot counts
    // among the lanes still marching, and a lane that stops (last z chunk) or
    // never started (past the chain's items) stops counting: the lanes
    // marching longest saw every record, so the wave's maximum is the count,
    // the same for every lane.  pl: present lower neighbours of every site
    // (kPeriodic, BOND 2).
    __device__ __forceinline__ void settle_queue(__amdgpu_buffer_rsrc_t own, uint32_t (*q)[NREC],
                                                 uint32_t pitch, uint32_t pl) {
        const uint32_t nq = min(wave_max(nrec), qcap);
        if (!nq) return;
        __builtin_amdgcn_s_waitcnt(0);
        for (uint32_t e = threadIdx.x & 63u; e < nq; e += 64) {
            const uint32_t* rec = q[e];
            const uint32_t row = rec[0], p0 = rec[1];
            Edge ed{0u, 0u, 32u, pl, 0u};
            if constexpr (!PER) {
                const uint32_t w = rec[2];
                ed = Edge{w & 15u, (w >> 4) & 15u, (w >> 8) & 63u, (w >> 16) & 15u, (w >> 20) & 15u};
            }
            uint32_t a[NP], l[4] = {0, 0, 0, 0};
#pragma unroll
            for (uint32_t k = 0; k < NP; ++k) a[k] = rec[kTieHead + k];
            if constexpr (BOND == 2) {
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) l[k] = rec[kTieHead + NP + k];
            }
            const uint32_t bits = rec[4];
            const uint32_t flips = settle<Z, BOND>(&C.thr[0][0], rec[3], a, l, bits, ed, p0, row, t,
                                                   colour, bonds, k0, k1, m_part, b_part);
            // the owner stored the word with the tied sites unchanged
            if (flips)
                __builtin_amdgcn_raw_buffer_store_b32(bits ^ flips, own, row * pitch + (p0 >> 3), 0, 0);
        }
    }

    // The wave's sums to its partials (from lane 63, which has the totals).
    __device__ __forceinline__ void partials(int32_t* __restrict__ out, uint64_t pass_block,
                                             bool active) {
        m_part = wave_total(m_part);
        if (BOND != 0 && bonds) b_part = wave_total(b_part);
        if (active && (threadIdx.x & 63u) == 63u) {
            int32_t* p = out + pass_block * (2u * kWaves) + 2u * (threadIdx.x >> 6);
            p[0] = m_part;
            p[1] = BOND != 0 && bonds ? b_part : 0;
        }
    }
};

// Sum of two counts 0..2 or 0..4 held in planes (x0 + 2 x1 [+ 4 x2]).
__device__ __forceinline__ void add_pairs(uint32_t x0, uint32_t x1, uint32_t y0, uint32_t y1,
                                          uint32_t s[3]) {  // 0..2 + 0..2
    const uint32_t c = x0 & y0;
    s[0] = x0 ^ y0;
    s[1] = bop3<kXor3>(x1, y1, c);
    s[2] = bop3<kMaj3>(x1, y1, c);
}
__device__ __forceinline__ void add_quads(const uint32_t x[3], const uint32_t y[3],
                                          uint32_t s[4]) {  // 0..4 + 0..4
    const uint32_t c0 = x[0] & y[0];
    s[0] = x[0] ^ y[0];
    s[1] = bop3<kXor3>(x[1], y[1], c0);
    const uint32_t c1 = bop3<kMaj3>(x[1], y[1], c0);
    s[2] = bop3<kXor3>(x[2], y[2], c1);
    s[3] = bop3<kMaj3>(x[2], y[2], c1);
}

// Aligned count a of the up count u (planes): u where the site is Up, p - u
// where it is Down, p the present neighbours (p at every site, pe at the
// sites in eb).  Bitwise subtraction with borrows.
__device__ __forceinline__ void align_present(const uint32_t u[4], uint32_t o, uint32_t p,
                                              uint32_t pe, uint32_t eb, uint32_t a[4]) {
    uint32_t br = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t pk = bop3<kSel>(0u - ((pe >> k) & 1u), 0u - ((p >> k) & 1u), eb);
        const uint32_t diff = bop3<kXor3>(pk, u[k], br);
        br = bop3<0x8E>(pk, u[k], br);  // (~p & u) | (~(p ^ u) & br)
        a[k] = bop3<kSel>(u[k], diff, o);
    }
}
// The same for p = Z at every site: 8 - u, 12 - u in closed form.
template <uint32_t Z>
__device__ __forceinline__ void align_all(const uint32_t u[4], uint32_t o, uint32_t a[4]) {
    const uint32_t t = u[1] | u[0];
    a[0] = u[0];
    a[1] = bop3<0xB4>(u[1], u[0], o);  // o ? u1 : u1 ^ u0
    if constexpr (Z == 8) {
        a[2] = bop3<0xB4>(u[2], t, o);  // o ? u2 : u2 ^ t
        const uint32_t any = bop3<0xFE>(u[3], u[2], t);
        a[3] = bop3<kSel>(u[3], ~any, o);  // 8 - u >= 8 only for u = 0
    } else {
        a[2] = bop3<0xE1>(u[2], t, o);  // o ? u2 : ~(u2 ^ t)
        const uint32_t big = bop3<0xF8>(u[3], u[2], t);  // u3 | (u2 & t): u >= 5
        a[3] = bop3<kSel>(u[3], ~big, o);
    }
}

// Sums the pass partials of one chain's sweep s over its ncol colour passes
// into its record: record = {bond, 0, 0, mag, 0} (int64).  A pass adds the
// bonds to lower colours only (none in colour 0), so each bond counts once.
// One workgroup's work, of 256 or 1024 threads.
__device__ __forceinline__ void reduce_sweep(const ChainDev& C,
                                             const int32_t* __restrict__ partials,
                                             uint32_t total_blocks, uint32_t ncol, uint32_t nsw,
                                             uint32_t s, int64_t* __restrict__ records) {
    __shared__ int64_t red[2][16];
    const uint32_t block = blockDim.x;  // 256, or 1024 where a chain has many workgroups
    if (s >= C.limit) return;  // this chain ran fewer sweeps in the block
    int64_t mm = 0, bb = 0;
    // Four workgroups' partials at a time, in 16-byte loads, by 1024 threads where
    // there are many: one workgroup sums a chain's sweep, and with 256 threads and
    // eight loads one after the other that was 22 us for sc 1024^3, now 8.8.
    constexpr uint32_t kAhead = 4;
    static_assert(kWaves == 4, "a workgroup's partials are two 16-byte words");
    for (uint32_t c = 0; c < ncol; ++c) {
        const int4* const from = reinterpret_cast<const int4*>(partials) +
                                 ((uint64_t)(s * ncol + c) * total_blocks + C.block0) * 2u;
        for (uint32_t k = threadIdx.x; k < C.nblocks; k += kAhead * block) {
            int4 v[kAhead][2];
#pragma unroll
            for (uint32_t j = 0; j < kAhead; ++j) {
                const uint32_t at = min(k + j * block, C.nblocks - 1u);
                v[j][0] = from[2u * at];
                v[j][1] = from[2u * at + 1u];
            }
#pragma unroll
            for (uint32_t j = 0; j < kAhead; ++j) {
                if (k + j * block >= C.nblocks) break;
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h) {
                    mm += (int64_t)v[j][h].x + v[j][h].z;
                    bb += (int64_t)v[j][h].y + v[j][h].w;
                }
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mm += __shfl_xor(mm, o, 64);
        bb += __shfl_xor(bb, o, 64);
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) {
        red[0][wave] = mm;
        red[1][wave] = bb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t m = 0, bo = 0;
        for (uint32_t k = 0; k < block / 64; ++k) {
            m += red[0][k];
            bo += red[1][k];
        }
        int64_t* r = records + ((uint64_t)C.slot * nsw + s) * 5u;
        r[0] = bo;
        r[1] = 0;
        r[2] = 0;
        r[3] = m;
        r[4] = 0;
    }
}

}  // namespace vg
