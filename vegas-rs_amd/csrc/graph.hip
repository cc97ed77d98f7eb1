// Colour-class sweeps of chains whose exchange is an arbitrary sparse matrix
// J: Exchange::new(CsMat<f64>) of the reference (src/energy.rs:170-172),
// with e_i = -sum_j J_ij s_i.s_j over row i (energy.rs:194-206) inside the
// Metropolis step of MetropolisFlipIntegrator / MetropolisIntegrator
// (src/integrator.rs:66-138).
//
// The host colours the symmetrised pattern greedily and stores the sites of
// a chain sorted by (colour, id); a colour class has no two sites that share
// a nonzero, so one pass updates a class all at once, one thread per site.
// Each position's merged row lists its neighbours (ascending site id) with
// a = J_ij and w = J_ij + J_ji for neighbours of lower colour (0 otherwise):
// h = sum a_j s_j is the field of the move, and s_i.(sum w_j s_j) after the
// move is the site's share of sum_{i != j} J_ij s_i.s_j, every pair counted
// at its higher-coloured end when both spins are final for the sweep.
//
// Ising: f64, every operation rounded on its own (no contraction), the
// acceptance `dE <= 0 or u < exp(-dE/T)` with u the 32-bit draw times
// 2^-32 and the engine's own exp (exp_f64_nonpos).  Heisenberg: the fp32
// update of the lattice passes with the couplings inside h.  Draws are keyed
// by the site id, so the CPU restatement reproduces every bit.
//
// Memory: each site reads its row (4 + 2 x 8 bytes per entry for Ising, 4 +
// 2 x 4 for Heisenberg) and its neighbours' spins by gather; this path is
// for generality (any lattice or coupling set), the stencil passes are the
// fast path for sc, bcc and fcc.
#include <type_traits>

#include "heis_common.hpp"

namespace vg {

// Row entries gathered at once: their neighbours, couplings and then spins are
// in flight together, so a row of up to eight entries waits for memory twice
// and not twice an entry.  (Past the row's end the last entry is read again and
// not added.)  A pass of 64 workgroups is one wave a SIMD and as long as its
// chain of waits: +-1 couplings on a 32^3 cubic lattice 5.6 us a pass with a
// loop over single entries and 64-bit shuffles for the sums, now 4.4; what is
// left is the launch, the descriptor, entries, spins, the f64 arithmetic and
// the sums, one after the other.
constexpr uint32_t kGather = 8;
// Ising rows all of at most this many entries take so many at once: reading the last
// one again costs what eight do.  us a pass, a loop over entries, eight and two at
// once: 200000 sites in pairs 4.9, 5.0, 4.1; a ring of 2^20 11.2, 10.9, 7.8.
constexpr uint32_t kShort = 2;

// What a pass's wave needs of its chain, loaded in one batch before anything
// is decided: field by field where each is used, the scalar loads were a chain
// of six waits at the start of a pass that lasts a few thousand cycles.  The
// class starts come with it from the descriptor; the arena's table serves
// colours past those that fit there.
struct GraphHead {
    uint64_t off[4], goff[2], seed, t, nsites;
    uint32_t p;  // the lane's position
    uint32_t proposal, w;
    bool go;     // a site of this class, in a sweep that the chain runs
};

__device__ __forceinline__ GraphHead graph_head(const ChainDev& C, const uint8_t* arena,
                                                uint32_t colour, uint32_t s, uint32_t b) {
    const uint32_t* const held = &C.plan[0][0];
    const uint32_t at = min(colour, kGraphStarts - 2u);
    uint32_t first = held[at], end = held[at + 1u], limit = C.limit, ncol = C.ncol;
    uint32_t block0 = C.block0;
    uint64_t starts = C.goff[2];
    GraphHead h{{C.off[0], C.off[1], C.off[2], C.off[3]}, {C.goff[0], C.goff[1]},
                C.seed,  C.sweep0 + s, C.nsites, 0u, C.proposal, C.w, false};
    first = loaded(first);
    end = loaded(end);
    limit = loaded(limit);
    ncol = loaded(ncol);
    block0 = loaded(block0);
    starts = loaded(starts);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) h.off[k] = loaded(h.off[k]);
    h.goff[0] = loaded(h.goff[0]);
    h.goff[1] = loaded(h.goff[1]);
    h.seed = loaded(h.seed);
    h.t = loaded(h.t);
    h.nsites = loaded(h.nsites);
    h.proposal = loaded(h.proposal);
    h.w = loaded(h.w);
    if (colour > kGraphStarts - 2u && colour < ncol) {
        const uint32_t* const cst = reinterpret_cast<const uint32_t*>(arena + starts);
        first = cst[colour];
        end = cst[colour + 1u];
    }
    h.p = first + (b - block0) * kBlock + threadIdx.x;
    h.go = s < limit && colour < ncol && h.p < end;
    return h;
}

__global__ __launch_bounds__(256) void graph_ising_pass(const ChainDev* __restrict__ chains,
                                                        const uint32_t* __restrict__ block_chain,
                                                        uint8_t* __restrict__ arena,
                                                        int64_t* __restrict__ partials,
                                                        uint32_t colour, uint32_t s,
                                                        uint32_t total_blocks, uint32_t npass) {
    const uint32_t b = blockIdx.x;
    const ChainDev& C = chains[block_chain ? block_chain[b] : 0u];
    const GraphHead H = graph_head(C, arena, colour, s, b);
    const double ghm = __longlong_as_double((long long)loaded((uint64_t)__double_as_longlong(C.ghm)));
    const double ghz = __longlong_as_double((long long)loaded((uint64_t)__double_as_longlong(C.ghz)));
    const double gbeta = __longlong_as_double((long long)loaded((uint64_t)__double_as_longlong(C.gbeta)));
    bool up = false, site_here = false;
    int64_t bsum = 0;
    const uint32_t p = H.p;
    const uint64_t t = H.t;
    if (H.go) {
        uint8_t* spin = arena + H.off[0];
        const uint32_t* ptr = reinterpret_cast<const uint32_t*>(arena + H.off[1]);
        const uint32_t* nbr = reinterpret_cast<const uint32_t*>(arena + H.off[2]);
        const double* a = reinterpret_cast<const double*>(arena + H.off[3]);
        const double* w = reinterpret_cast<const double*>(arena + H.goff[0]);
        const uint32_t site = reinterpret_cast<const uint32_t*>(arena + H.goff[1])[p];
        const U4 r = philox(U4{site, 0u, (uint32_t)t, ctr_w(t, kGraphIsing, 0)},
                            (uint32_t)H.seed, (uint32_t)(H.seed >> 32));
        double sv = spin[p] ? 1.0 : -1.0;
        // Spin::rand proposes Up when its draw is below 1/2 (state.rs:76-84);
        // a proposal equal to the current spin changes nothing.
        const bool change = H.proposal == 0 || ((r.y < 0x80000000u) ? 1.0 : -1.0) != sv;
        double h = 0.0, hb = 0.0;
        uint32_t e0 = p * H.w, e1 = e0 + H.w;  // H.w = 0: rows of different lengths
        if (!H.w) {
            e0 = ptr[p];
            e1 = ptr[p + 1];
        }
        const auto gather = [&](auto width) {
            constexpr uint32_t N = decltype(width)::value;
            for (; e0 < e1; e0 += N) {
                uint32_t j[N], bj[N];
                double aj[N], wj[N];
#pragma unroll
                for (uint32_t k = 0; k < N; ++k) {
                    const uint32_t e = min(e0 + k, e1 - 1u);
                    j[k] = nbr[e];
                    aj[k] = a[e];
                    wj[k] = w[e];
                }
#pragma unroll
                for (uint32_t k = 0; k < N; ++k) bj[k] = spin[j[k]];
#pragma unroll
                for (uint32_t k = 0; k < N; ++k) {
                    const double sj = bj[k] ? 1.0 : -1.0;
                    const double hk = __dadd_rn(h, __dmul_rn(aj[k], sj));
                    const double hbk = __dadd_rn(hb, __dmul_rn(wj[k], sj));
                    h = e0 + k < e1 ? hk : h;
                    hb = e0 + k < e1 ? hbk : hb;
                }
            }
        };
        if (H.w - 1u < kShort)
            gather(std::integral_constant<uint32_t, kShort>{});
        else
            gather(std::integral_constant<uint32_t, kGather>{});
        // The decision is computed without branches and applied by one
        // select: written as `if (dE <= 0 || u < p) flip`, the accept
        // block has two predecessors, and hipcc for gfx950 (ROCm 7.2)
        // kept the old spin on the second path (the optimised IR is
        // right).  exp is evaluated for every site; its argument is
        // clamped to <= 0, which changes nothing where it is used
        // (dE > 0).
        const double dE = __dsub_rn(__dmul_rn(__dmul_rn(2.0, sv), h),
                                    __dmul_rn(__dmul_rn(__dmul_rn(2.0, ghm), ghz), sv));
        const double pr = exp_f64_nonpos(fmin(-__dmul_rn(dE, gbeta), 0.0));
        const bool accept =
            change & ((dE <= 0.0) | (__dmul_rn((double)r.x, 0x1p-32) < pr));
        if (accept) spin[p] = sv > 0.0 ? 0 : 1;
        sv = accept ? -sv : sv;
        up = sv > 0.0;
        site_here = true;
        bsum = __double2ll_rn(__dmul_rn(__dmul_rn(sv, hb), 134217728.0));
    }
    // {bond, 0, 0, magnetisation, 0}
    const int64_t mag = 2 * (int64_t)__builtin_popcountll(__ballot(up)) -
                        (int64_t)__builtin_popcountll(__ballot(site_here));
    const int64_t sums[5] = {wave_sum_any(bsum), 0, 0, mag, 0};
    heis_block_partials(sums, partials, colour, npass, s, total_blocks, b);
}

__global__ __launch_bounds__(256) void graph_heis_pass(const ChainDev* __restrict__ chains,
                                                       const uint32_t* __restrict__ block_chain,
                                                       uint8_t* __restrict__ arena,
                                                       int64_t* __restrict__ partials,
                                                       uint32_t colour, uint32_t s,
                                                       uint32_t total_blocks, uint32_t npass) {
    const uint32_t b = blockIdx.x;
    const ChainDev& C = chains[block_chain ? block_chain[b] : 0u];
    const GraphHead H = graph_head(C, arena, colour, s, b);
    int32_t s32[4] = {0, 0, 0, 0};
    int64_t bsum = 0;
    const uint32_t p = H.p;
    const uint64_t t = H.t;
    if (H.go) {
        float* xs = reinterpret_cast<float*>(arena + H.off[0]);
        float* ys = xs + H.nsites;
        float* zs = ys + H.nsites;
        const uint32_t* ptr = reinterpret_cast<const uint32_t*>(arena + H.off[1]);
        const uint32_t* nbr = reinterpret_cast<const uint32_t*>(arena + H.off[2]);
        const float* a = reinterpret_cast<const float*>(arena + H.off[3]);
        const float* w = reinterpret_cast<const float*>(arena + H.goff[0]);
        const uint32_t site = reinterpret_cast<const uint32_t*>(arena + H.goff[1])[p];
        float h[3] = {0.0f, 0.0f, 0.0f}, hb[3] = {0.0f, 0.0f, 0.0f};
        uint32_t e0 = p * H.w, e1 = e0 + H.w;  // H.w = 0: rows of different lengths
        if (!H.w) {
            e0 = ptr[p];
            e1 = ptr[p + 1];
        }
        for (; e0 < e1; e0 += kGather) {
            uint32_t j[kGather];
            float aj[kGather], wj[kGather], sj[kGather][3];
#pragma unroll
            for (uint32_t k = 0; k < kGather; ++k) {
                const uint32_t e = min(e0 + k, e1 - 1u);
                j[k] = nbr[e];
                aj[k] = a[e];
                wj[k] = w[e];
            }
#pragma unroll
            for (uint32_t k = 0; k < kGather; ++k) {
                sj[k][0] = xs[j[k]];
                sj[k][1] = ys[j[k]];
                sj[k][2] = zs[j[k]];
            }
#pragma unroll
            for (uint32_t k = 0; k < kGather; ++k) {
                if (e0 + k >= e1) break;
#pragma unroll
                for (uint32_t c = 0; c < 3; ++c) {
                    h[c] = fa(h[c], fm(aj[k], sj[k][c]));
                    hb[c] = fa(hb[c], fm(wj[k], sj[k][c]));
                }
            }
        }
        const float o[3] = {xs[p], ys[p], zs[p]};
        float u, pr[3];
        if (H.proposal) {
            if (!proposal_first(H.seed, site, 0u, t, 0u, u, pr)) proposal_rest(H.seed, site, 0u, t, 0u, pr);
        } else {
            const U4 fw = philox(U4{site, 0u, (uint32_t)t, ctr_w(t, kHeisStream, 0)},
                                 (uint32_t)H.seed, (uint32_t)(H.seed >> 32));
            u = unit24(fw.x);
            pr[0] = -o[0];
            pr[1] = -o[1];
            pr[2] = -o[2];
        }
        float n[3];
        heis_update(C, false, o, h, hb, u, pr, n, s32, bsum);
        // the bond share can exceed the int32 fixed-point range of the
        // lattice sums when couplings are large: 64-bit conversion
        bsum = (int64_t)__float2ll_rn(fm(dot3(n[0], n[1], n[2], hb[0], hb[1], hb[2]), kFixScale));
        xs[p] = n[0];
        ys[p] = n[1];
        zs[p] = n[2];
    }
    heis_partials(s32, bsum, partials, colour, npass, s, total_blocks, b);
}

// Initial states (State::rand_with_size, src/state.rs:260-262) keyed by the
// site id: Ising Up iff word 0 of Philox(site, 0, 0, w(0, graph-init, 0)) is
// below 2^31; Heisenberg by Marsaglia's method on the calls
// Philox(site, 0, k, w(0, heis-init, 0)), two tries per call, (0,0,1) after
// 64 calls.  One thread per position.
__global__ void graph_ising_init(const ChainDev* __restrict__ chain, uint8_t* __restrict__ arena) {
    const ChainDev& C = *chain;
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= C.nsites) return;
    const uint32_t site = reinterpret_cast<const uint32_t*>(arena + C.goff[1])[p];
    const U4 r = philox(U4{site, 0u, 0u, ctr_w(0, kGraphInit, 0)}, (uint32_t)C.seed,
                        (uint32_t)(C.seed >> 32));
    arena[C.off[0] + p] = r.x < 0x80000000u ? 1 : 0;
}

__global__ void graph_heis_init(const ChainDev* __restrict__ chain, uint8_t* __restrict__ arena) {
    const ChainDev& C = *chain;
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= C.nsites) return;
    const uint32_t site = reinterpret_cast<const uint32_t*>(arena + C.goff[1])[p];
    float sx = 0.0f, sy = 0.0f, sz = 1.0f;
    for (uint32_t k = 0; k < kHeisInitMaxCalls; ++k) {
        const U4 r = philox(U4{site, 0u, k, ctr_w(0, kHeisInit, 0)}, (uint32_t)C.seed,
                            (uint32_t)(C.seed >> 32));
        bool done = false;
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) {
            const float x1 = sym24(u4_word(r, 2 * q));
            const float x2 = sym24(u4_word(r, 2 * q + 1));
            const float qq = fa(fm(x1, x1), fm(x2, x2));
            if (!done && qq < 1.0f) {
                const float root = sqrt_rn(fs(1.0f, qq));
                sx = fm(fm(2.0f, x1), root);
                sy = fm(fm(2.0f, x2), root);
                sz = fs(1.0f, fm(2.0f, qq));
                done = true;
            }
        }
        if (done) break;
    }
    float* xs = reinterpret_cast<float*>(arena + C.off[0]);
    xs[p] = sx;
    xs[C.nsites + p] = sy;
    xs[2 * C.nsites + p] = sz;
}

}  // namespace vg
