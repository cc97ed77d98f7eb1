// Wolff single-cluster steps for int8 Ising chains on sc, bcc and fcc
// lattices (reference WolffIntegrator::step, src/integrator.rs:146-230).
//
// One step picks a seed site, grows the cluster over bonds between equal
// spins that are active with probability p = 1 - exp(-2J/T), and flips it;
// the field plays no part, as in the reference.  Randomness is keyed by the
// step and the bond, not drawn in visiting order: the seed site is
// floor(r64 * N / 2^64) for r64 = words 0,1 of Philox(0, 0, step, w(step,
// seed)), and a bond is active iff word 0 of Philox(lo, slot, step, w(step,
// bond)) is below ceil(p 2^32), (lo, slot) being its endpoint with the lower
// site id and that endpoint's neighbour slot.  The cluster is then the seed's
// connected component over active bonds, whatever order a parallel search
// visits it in, so the result is deterministic and the CPU oracle
// reproduces it.
//
// Layout (natural site order): spins int8 +-1 at off[0], a uint32 visit
// stamp per site at off[1], the cluster queue (uint32 site ids) at off[2].
// One workgroup runs all steps of one chain's sweep block: it sums the bonds
// and the magnetization once, then per step searches level by level (the
// queue holds the levels back to back), flips the cluster, and updates the
// sums by the cluster's size and the spins across its boundary.
//
// What bounds a step is the latency of its levels, each a chain of LDS reads,
// one Philox call and a workgroup barrier: a level of a few hundred sites is
// far below what a CU can do.  So a level's work is split as finely as it
// goes, one (site, neighbour slot) pair per thread over 1024 threads, and
// takes one barrier (the append counters rotate over three words, so none is
// reset while a slow wave may still read it).  A wave alone on its SIMD
// issues an instruction every 8 cycles, four waves one every 4 or fewer
// between them.  64 chains of 32^3 at T_c, 40 steps from the ordered side:
// 11.3 ms with 256 threads that took a site and its z slots in turn and three
// barriers a level, 2.86 ms now; one chain of 8^3, 20 steps: 0.88 and 0.25
// ms; one of 96^3 (global memory), 10 steps: 15.3 and 4.9 ms.
#include "vg_device.hpp"

namespace vg {

namespace {

// fcc sublattice half-cell offsets along x, y, z as 3-bit masks.
__device__ __forceinline__ uint32_t fcc_bits(uint32_t s) {
    return s == 0 ? 0u : (s == 1 ? 6u : (s == 2 ? 5u : 3u));
}

struct WolffGeom {
    uint32_t lx, ly, lz, pbc, lx_m, lx_s, ly_m, ly_s;
};

// Coordinate v + d (d in {-1, 0, +1}) along an axis of length n; -1 when it
// leaves an open axis.
__device__ __forceinline__ int32_t wolff_axis(uint32_t v, int d, uint32_t n, bool periodic) {
    const int32_t b = (int32_t)v + d;
    if (b >= 0 && b < (int32_t)n) return b;
    if (!periodic) return -1;
    return b < 0 ? (int32_t)n - 1 : 0;
}

// Neighbour site of `i` through slot k, or -1: sc -x,+x,-y,+y,-z,+z;
// bcc slots (dz, dy, dx), dx fastest, towards cells c -+ d; fcc 4 slots per
// other sublattice b (ascending), (d1, d2) over the two axes where the
// sublattices differ, d1 fastest.  The order of the oracle's neighbour lists.
template <uint32_t KIND>
__device__ __forceinline__ int32_t wolff_nb(const WolffGeom& g, uint32_t i, uint32_t k) {
    constexpr uint32_t sh = KIND;  // sites per cell: 1, 2, 4
    const uint32_t cell = i >> sh, a = i & ((1u << sh) - 1u);
    const uint32_t yz = fast_div(cell, g.lx_m, g.lx_s);
    const uint32_t z = fast_div(yz, g.ly_m, g.ly_s);
    const uint32_t x = cell - yz * g.lx, y = yz - z * g.ly;
    int dx, dy, dz;
    uint32_t b = 0;
    if (KIND == 0) {
        const int d = (k & 1u) ? 1 : -1;
        dx = (k >> 1) == 0 ? d : 0;
        dy = (k >> 1) == 1 ? d : 0;
        dz = (k >> 1) == 2 ? d : 0;
    } else if (KIND == 1) {
        const int sg = a == 0 ? -1 : 1;
        dx = sg * (int)(k & 1u);
        dy = sg * (int)((k >> 1) & 1u);
        dz = sg * (int)((k >> 2) & 1u);
        b = 1u - a;
    } else {
        const uint32_t r = k >> 2;
        b = r + (r >= a ? 1u : 0u);
        const uint32_t ba = fcc_bits(a), bb = fcc_bits(b), diff = ba ^ bb;
        const uint32_t e1 = (diff & 1u) ? 0u : 1u;  // lower differing axis
        const uint32_t e2 = (diff & 4u) ? 2u : 1u;  // higher differing axis
        const int d1 = (int)(k & 1u), d2 = (int)((k >> 1) & 1u);
        const auto step = [&](uint32_t e) {
            const int d = (e == e1 ? d1 : 0) + (e == e2 ? d2 : 0);
            return ((bb >> e) & 1u) > ((ba >> e) & 1u) ? -d : d;
        };
        dx = step(0);
        dy = step(1);
        dz = step(2);
    }
    const int32_t qx = wolff_axis(x, dx, g.lx, g.pbc & 1u);
    const int32_t qy = wolff_axis(y, dy, g.ly, g.pbc & 2u);
    const int32_t qz = wolff_axis(z, dz, g.lz, g.pbc & 4u);
    if ((qx | qy | qz) < 0) return -1;
    return (int32_t)((((uint32_t)qx + g.lx * ((uint32_t)qy + g.ly * (uint32_t)qz)) << sh) + b);
}

// The slot of the neighbour's list that holds the same bond.
template <uint32_t KIND>
__device__ __forceinline__ uint32_t wolff_back(uint32_t i, uint32_t k) {
    if (KIND == 0) return k ^ 1u;
    if (KIND == 1) return k;
    const uint32_t a = i & 3u, r = k >> 2, b = r + (r >= a ? 1u : 0u);
    return 4u * (a - (a > b ? 1u : 0u)) + (k & 3u);
}

// Whether slot k of site i is the one that counts its bond in a sum over all
// sites and slots (each bond is in both ends' lists): sc the + slots, bcc the
// corner sites, fcc the lower sublattice.
template <uint32_t KIND>
__device__ __forceinline__ bool wolff_counts(uint32_t i, uint32_t k) {
    if (KIND == 0) return k & 1u;
    if (KIND == 1) return (i & 1u) == 0u;
    return (k >> 2) >= (i & 3u);  // the other sublattice is above i's
}

constexpr uint32_t kWolffWaves = kWolffBlock / 64;

__device__ __forceinline__ void wolff_sum2(int64_t& x, int64_t& y, int64_t (*red)[kWolffWaves]) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        x += __shfl_xor(x, o, 64);
        y += __shfl_xor(y, o, 64);
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) {
        red[0][wave] = x;
        red[1][wave] = y;
    }
    __syncthreads();
    x = 0;
    y = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWolffWaves; ++w) {
        x += red[0][w];
        y += red[1][w];
    }
}

// Spins and visit marks of a chain of more than kWolffLdsSites sites: int8
// spins, stamps (the step's number + 1) and queue in global memory; a claim
// is an exchange of the stamp.
struct WolffGlobal {
    using Pairs = uint64_t;  // counts of (site, slot) pairs
    int8_t* spin;
    uint32_t* stamp;
    uint32_t* queue;
    uint32_t sv;  // this step's stamp
    __device__ __forceinline__ bool up(uint32_t i) const { return spin[i] > 0; }
    // a stale stamp only costs a draw (the exchange decides) or, after the
    // search, is avoided by reading past L1
    __device__ __forceinline__ bool seen(uint32_t i) const { return stamp[i] == sv; }
    __device__ __forceinline__ bool member(uint32_t i) const {
        return __hip_atomic_load(&stamp[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == sv;
    }
    __device__ __forceinline__ bool claim(uint32_t i) { return atomicExch(&stamp[i], sv) != sv; }
    __device__ __forceinline__ uint32_t qget(uint32_t q) const { return queue[q]; }
    __device__ __forceinline__ void qput(uint32_t q, uint32_t v) { queue[q] = v; }
};

// A chain of at most kWolffLdsSites sites: one spin bit (set = Up) and one
// visit bit per site in LDS; a claim is an LDS atomic OR whose old word tells
// whether this thread set the bit.  The queue's first kWolffLdsQueue entries
// are in LDS too, the rest in global memory.
struct WolffLds {
    using Pairs = uint32_t;
    uint32_t* ub;
    uint32_t* vis;
    uint32_t* lq;
    uint32_t* queue;
    __device__ __forceinline__ bool up(uint32_t i) const { return (ub[i >> 5] >> (i & 31u)) & 1u; }
    __device__ __forceinline__ bool seen(uint32_t i) const {
        return (vis[i >> 5] >> (i & 31u)) & 1u;
    }
    __device__ __forceinline__ bool member(uint32_t i) const { return seen(i); }
    __device__ __forceinline__ bool claim(uint32_t i) {
        const uint32_t m = 1u << (i & 31u);
        return (atomicOr(&vis[i >> 5], m) & m) == 0u;
    }
    __device__ __forceinline__ uint32_t qget(uint32_t q) const {
        return q < kWolffLdsQueue ? lq[q] : queue[q];
    }
    __device__ __forceinline__ void qput(uint32_t q, uint32_t v) {
        if (q < kWolffLdsQueue)
            lq[q] = v;
        else
            queue[q] = v;
    }
};

// The cluster of step t: claims it, leaves its sites in the queue and returns
// their number; `ref` is its spin.  cnt: three LDS counters, zero on entry
// (a barrier behind) and left so.  Every thread of the workgroup calls this.
template <uint32_t KIND, class M>
__device__ __forceinline__ uint32_t wolff_grow(const ChainDev& C, const WolffGeom& g, M& mem,
                                               uint64_t t, uint32_t* cnt, bool& ref) {
    constexpr uint32_t Z = KIND == 0 ? 6u : (KIND == 1 ? 8u : 12u);
    const uint32_t tid = threadIdx.x;
    const uint32_t k0 = (uint32_t)C.seed, k1 = (uint32_t)(C.seed >> 32);
    const uint32_t thr = C.wolff_thr, all = C.wolff_all;
    const uint32_t wb = ctr_w(t, kWolffBond, 0u);
    // every thread draws the seed site; one claims it
    const U4 r = philox(U4{0u, 0u, (uint32_t)t, ctr_w(t, kWolffSeed, 0u)}, k0, k1);
    const uint64_t r64 = (uint64_t)r.x | ((uint64_t)r.y << 32);
    const uint32_t src = (uint32_t)__umul64hi(r64, C.nsites);
    ref = mem.up(src);
    if (tid == 0) {
        mem.claim(src);
        mem.qput(0u, src);
    }
    __syncthreads();
    uint32_t head = 0, tail = 1, level = 0;  // level counts mod 3
    while (head < tail) {  // tail <= n (one claim per site)
        const uint32_t next = level == 2u ? 0u : level + 1u;
        // the next level's counter: last read two levels ago, a barrier back
        if (tid == 0) cnt[next] = 0u;
        const typename M::Pairs pairs = (typename M::Pairs)(tail - head) * Z;
        for (typename M::Pairs e = tid; e < pairs; e += kWolffBlock) {
            const uint32_t q = (uint32_t)(e / Z), k = (uint32_t)(e - (typename M::Pairs)q * Z);
            const uint32_t i = mem.qget(head + q);
            const int32_t jj = wolff_nb<KIND>(g, i, k);
            if (jj < 0 || (uint32_t)jj == i) continue;
            const uint32_t j = (uint32_t)jj;
            if (mem.up(j) != ref || mem.seen(j)) continue;
            const bool low = i < j;
            const uint32_t lo = low ? i : j, ls = low ? k : wolff_back<KIND>(i, k);
            const U4 d = philox(U4{lo, ls, (uint32_t)t, wb}, k0, k1);
            if ((all || d.x < thr) && mem.claim(j)) mem.qput(tail + atomicAdd(&cnt[level], 1u), j);
        }
        __syncthreads();
        head = tail;
        tail += cnt[level];
        level = next;
    }
    // the last level added nothing: its counter and the next one are zero,
    // the third is cleared here (its readers passed the barrier above)
    if (tid == 0) cnt[level == 2u ? 0u : level + 1u] = 0u;
    return tail;
}

// Sum over the cluster's boundary of the spins outside it, this thread's
// share (the neighbours outside keep their spins while the cluster flips).
template <uint32_t KIND, class M>
__device__ __forceinline__ int64_t wolff_across(const WolffGeom& g, const M& mem, uint32_t tail) {
    constexpr uint32_t Z = KIND == 0 ? 6u : (KIND == 1 ? 8u : 12u);
    int64_t across = 0;
    const typename M::Pairs pairs = (typename M::Pairs)tail * Z;
    for (typename M::Pairs e = threadIdx.x; e < pairs; e += kWolffBlock) {
        const uint32_t q = (uint32_t)(e / Z), k = (uint32_t)(e - (typename M::Pairs)q * Z);
        const uint32_t i = mem.qget(q);
        const int32_t jj = wolff_nb<KIND>(g, i, k);
        if (jj < 0 || (uint32_t)jj == i) continue;
        if (!mem.member((uint32_t)jj)) across += mem.up((uint32_t)jj) ? 1 : -1;
    }
    return across;
}

// This thread's share of the chain's bond sum and magnetization.
template <uint32_t KIND, class M>
__device__ __forceinline__ void wolff_sums(const WolffGeom& g, const M& mem, uint32_t n,
                                           int64_t& bond, int64_t& mag) {
    constexpr uint32_t Z = KIND == 0 ? 6u : (KIND == 1 ? 8u : 12u);
    bond = 0;
    mag = 0;
    for (uint32_t i = threadIdx.x; i < n; i += kWolffBlock) {
        const bool up = mem.up(i);
        mag += up ? 1 : -1;
#pragma unroll
        for (uint32_t k = 0; k < Z; ++k) {
            if (!wolff_counts<KIND>(i, k)) continue;
            const int32_t j = wolff_nb<KIND>(g, i, k);
            if (j >= 0 && (uint32_t)j != i) bond += mem.up((uint32_t)j) == up ? 1 : -1;
        }
    }
}

__device__ __forceinline__ WolffGeom wolff_geom(const ChainDev& C) {
    return WolffGeom{C.lx, C.ly, C.lz, C.pbc, C.lx_m, C.lx_s, C.ly_m, C.ly_s};
}

__device__ __forceinline__ void wolff_record(const ChainDev& C, int64_t* records, uint32_t nsw,
                                             uint32_t s, int64_t bond, int64_t mag) {
    int64_t* r = records + ((uint64_t)C.slot * nsw + s) * 5u;
    r[0] = bond;
    r[1] = 0;
    r[2] = 0;
    r[3] = mag;
    r[4] = 0;
}

}  // namespace

// grid = (chains): block b runs min(nsw, limit) steps of chain b and writes
// its records {bond, 0, 0, mag, 0} per step.  Chains of another lattice kind
// and those of at most kWolffLdsSites sites are left to the other kernels.
template <uint32_t KIND>
__global__ __launch_bounds__(kWolffBlock) void wolff_run(const ChainDev* __restrict__ chains,
                                                         uint8_t* __restrict__ arena, uint32_t nsw,
                                                         int64_t* __restrict__ records) {
    __shared__ uint32_t cnt[3];
    __shared__ int64_t red[2][kWolffWaves];
    const ChainDev& C = chains[blockIdx.x];
    const uint32_t steps = min(nsw, C.limit);
    // uniform over the workgroup
    if (steps == 0 || C.kind != KIND || C.nsites <= kWolffLdsSites) return;
    WolffGlobal mem{reinterpret_cast<int8_t*>(arena + C.off[0]),
                    reinterpret_cast<uint32_t*>(arena + C.off[1]),
                    reinterpret_cast<uint32_t*>(arena + C.off[2]), 0u};
    const uint32_t n = (uint32_t)C.nsites, tid = threadIdx.x;
    const WolffGeom g = wolff_geom(C);
    if (tid < 3u) cnt[tid] = 0u;
    for (uint32_t i = tid; i < n; i += kWolffBlock) mem.stamp[i] = 0u;
    int64_t bond, mag;
    wolff_sums<KIND>(g, mem, n, bond, mag);
    wolff_sum2(bond, mag, red);

    for (uint32_t s = 0; s < steps; ++s) {
        mem.sv = s + 1u;
        __syncthreads();  // the previous step's flips and queue reads are done
        bool ref;
        const uint32_t tail = wolff_grow<KIND>(C, g, mem, C.sweep0 + s, cnt, ref);
        int64_t across = wolff_across<KIND>(g, mem, tail), dummy = 0;
        for (uint32_t q = tid; q < tail; q += kWolffBlock)
            mem.spin[mem.qget(q)] = ref ? (int8_t)-1 : (int8_t)1;
        wolff_sum2(across, dummy, red);
        const int64_t sref = ref ? 1 : -1;
        bond += -2 * sref * across;
        mag += -2 * sref * (int64_t)tail;
        if (tid == 0) wolff_record(C, records, nsw, s, bond, mag);
    }
}

// The same steps with the chain's spins and visit marks in LDS, for chains
// of at most kWolffLdsSites sites.  Spins are packed from the int8 array at
// the start of the sweep block and written back at its end; a step's cluster
// is flipped word by word (spins ^= visits), which also clears the visits.
// Dynamic LDS: 2 * ceil(n / 32) + kWolffLdsQueue words for the largest chain
// n of the launch.
template <uint32_t KIND>
__global__ __launch_bounds__(kWolffBlock) void wolff_run_lds(const ChainDev* __restrict__ chains,
                                                             uint8_t* __restrict__ arena,
                                                             uint32_t nsw,
                                                             int64_t* __restrict__ records) {
    extern __shared__ uint32_t lds_bits[];
    __shared__ uint32_t cnt[3];
    __shared__ int64_t red[2][kWolffWaves];
    const ChainDev& C = chains[blockIdx.x];
    const uint32_t steps = min(nsw, C.limit);
    // uniform over the workgroup
    if (steps == 0 || C.kind != KIND || C.nsites > kWolffLdsSites) return;
    int8_t* const spin = reinterpret_cast<int8_t*>(arena + C.off[0]);
    const uint32_t n = (uint32_t)C.nsites, tid = threadIdx.x;
    const uint32_t nw = (n + 31u) >> 5;
    WolffLds mem{lds_bits, lds_bits + nw, lds_bits + 2u * nw,
                 reinterpret_cast<uint32_t*>(arena + C.off[2])};
    const WolffGeom g = wolff_geom(C);

    // Pack the spins (each wave 64 sites per round, one byte per lane, a
    // ballot for the two words) and clear the visit bits.
    if (tid < 3u) cnt[tid] = 0u;
    const uint32_t lane = tid & 63u;
    for (uint32_t base = (tid >> 6) * 64u; base < nw * 32u; base += kWolffBlock) {
        const uint32_t i = base + lane;
        const uint64_t m = __ballot(i < n && spin[i] > 0);
        if (lane == 0) {
            mem.ub[base >> 5] = (uint32_t)m;
            mem.vis[base >> 5] = 0u;
            if ((base >> 5) + 1u < nw) {
                mem.ub[(base >> 5) + 1u] = (uint32_t)(m >> 32);
                mem.vis[(base >> 5) + 1u] = 0u;
            }
        }
    }
    __syncthreads();
    int64_t bond, mag;
    wolff_sums<KIND>(g, mem, n, bond, mag);
    wolff_sum2(bond, mag, red);

    for (uint32_t s = 0; s < steps; ++s) {
        __syncthreads();  // the previous step's flips and queue reads are done
        bool ref;
        const uint32_t tail = wolff_grow<KIND>(C, g, mem, C.sweep0 + s, cnt, ref);
        int64_t across = wolff_across<KIND>(g, mem, tail), dummy = 0;
        wolff_sum2(across, dummy, red);  // every bit read is done after it
        for (uint32_t w = tid; w < nw; w += kWolffBlock) {
            mem.ub[w] ^= mem.vis[w];
            mem.vis[w] = 0u;
        }
        const int64_t sref = ref ? 1 : -1;
        bond += -2 * sref * across;
        mag += -2 * sref * (int64_t)tail;
        if (tid == 0) wolff_record(C, records, nsw, s, bond, mag);
    }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kWolffBlock) spin[i] = mem.up(i) ? (int8_t)1 : (int8_t)-1;
}

#define VG_WOLFF(KIND)                                                                         \
    template __global__ void wolff_run<KIND>(const ChainDev*, uint8_t*, uint32_t, int64_t*);   \
    template __global__ void wolff_run_lds<KIND>(const ChainDev*, uint8_t*, uint32_t, int64_t*);
VG_WOLFF(0)
VG_WOLFF(1)
VG_WOLFF(2)
#undef VG_WOLFF

// Random initial state in natural order, the same draws as the colour-split
// kernels: site n at (colour c, row, position i) is Up iff word (i & 3) of
// Philox(i >> 2, row, 0, w(0, init, c)) is below 2^31.
__global__ void wolff_init(const ChainDev* __restrict__ chain, uint8_t* __restrict__ arena) {
    const ChainDev& C = *chain;
    const uint64_t n = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= C.nsites) return;
    uint32_t c, row, i;
    if (C.kind == 0) {
        const uint32_t x = (uint32_t)(n % C.lx), y = (uint32_t)((n / C.lx) % C.ly);
        const uint32_t zz = (uint32_t)(n / ((uint64_t)C.lx * C.ly));
        c = (x + y + zz) & 1u;
        row = y + C.ly * zz;
        i = x >> 1;
    } else {
        const uint32_t sh = C.kind == 1 ? 1u : 2u;
        const uint64_t cell = n >> sh;
        const uint32_t x = (uint32_t)(cell % C.lx), y = (uint32_t)((cell / C.lx) % C.ly);
        const uint32_t zz = (uint32_t)(cell / ((uint64_t)C.lx * C.ly));
        c = (uint32_t)(n & ((1u << sh) - 1u));
        row = y + C.ly * zz;
        i = x;
    }
    const U4 r = philox(U4{i >> 2, row, 0u, ctr_w(0, kIsingInit, c)}, (uint32_t)C.seed,
                        (uint32_t)(C.seed >> 32));
    reinterpret_cast<int8_t*>(arena + C.off[0])[n] = (u4_word(r, i & 3u) >> 31) == 0 ? 1 : -1;
}

}  // namespace vg
