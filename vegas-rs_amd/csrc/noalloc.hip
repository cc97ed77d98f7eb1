// vg_run_sums_noalloc: the sweeps of vg_batch_run_sums for one Ising chain
// on caller-owned device buffers, allocating nothing.
//
// A batch allocates its arena, descriptors, block map, pass partials and
// records when it is created.  Here the caller brings the spins (in the
// batch arena's colour-plane layout) and the output sums; the descriptor,
// the block -> chain map and the pass partials live in `scratch`, a
// file-scope device array of kScratchBytes that every GPU the library runs
// on holds until the process ends.  Host code reaches a device's copy only
// through the address hipGetSymbolAddress returns for it (kept per device):
// the array's name in host code is a host-side stand-in, not a device
// address.  The descriptor reaches the scratch through a kernel argument,
// so a call makes no host-to-device copy either.  Calls on one GPU share its
// scratch, and everything a call reads there it has written first, so
// nothing needs clearing; calls that overlap on one GPU race.
#include <mutex>

#include "engine.hpp"

namespace vg {

constexpr uint64_t kScratchBytes = 16ull << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr uint64_t kScratchDesc = 0;      // ChainDev
constexpr uint64_t kScratchMap = 4096;    // block -> chain map (all 0)
static_assert(sizeof(ChainDev) <= kScratchMap, "descriptor slot too small");

// Writes the chain's descriptor and the block -> chain map into the scratch.
__global__ void noalloc_setup(ChainDev d, ChainDev* __restrict__ out,
                              uint32_t* __restrict__ block_chain, uint32_t nblocks) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *out = d;
    if (i < nblocks) block_chain[i] = 0;
}

// The caller's int8 planes, one byte of 0/1 per position, to one bit per
// position in place, and back.  A row's bits take the first eighth of its
// bytes, so that a row is one wave's own work: `rows` of 64 lanes hold one row
// of at most 64 segments (32 positions: 32 bytes, one word) or several, and a
// longer row is walked in chunks of 64 segments.  A chunk's loads end before
// its stores start (each word is made of its own bytes, and the lanes of a
// wave load together); chunk c's words lie in [256c, 256c + 256), below the
// bytes [2048c', ...) of every later chunk c', so packing walks upwards and
// unpacking downwards.  Only whole segments are touched, and their padding is
// zero before and after.
//
// One read and one write of the bytes for any number of sweeps: passes that
// worked on the bytes instead read and wrote eight times as much, packed every
// row they read and unpacked every row they wrote.  us a sweep, 60 sweeps a
// call: sc 64^3 18.5 on bytes, 8.9 in bits; bcc 120^3 16.2, 9.6; fcc 100^3
// with open z 35.8, 20.8.  (The one loss: a call of a single sweep over a chain
// past the caches pays the conversion alone, sc 512^3 97 us, now 111; from two
// sweeps on it gains.)
template <bool PACK>
__global__ __launch_bounds__(kBlock) void noalloc_bits(const ChainDev* __restrict__ chain,
                                                       uint8_t* __restrict__ spins) {
    const ChainDev& C = *chain;
    const uint32_t lane = threadIdx.x & 63u, segs = C.segs;
    const uint32_t per_wave = segs < 64u ? 64u / segs : 1u;  // rows
    const uint64_t wave = (uint64_t)blockIdx.x * (kBlock / 64u) + (threadIdx.x >> 6);
    const uint64_t at = wave * per_wave + (segs < 64u ? lane / segs : 0u);
    if (segs < 64u && lane >= per_wave * segs) return;
    if (at >= (uint64_t)C.ncol * C.rows) return;
    const uint32_t colour = (uint32_t)(at / C.rows), row = (uint32_t)(at % C.rows);
    uint8_t* const base = spins + C.off[colour] + (uint64_t)row * C.pitch;
    const uint32_t first = segs < 64u ? lane % segs : lane;
    const uint32_t chunks = (segs + 63u) / 64u;
    for (uint32_t k = 0; k < chunks; ++k) {
        const uint32_t seg = first + 64u * (PACK ? k : chunks - 1u - k);
        if (seg >= segs) continue;
        u32x4* const bytes = reinterpret_cast<u32x4*>(base + 32u * seg);
        uint32_t* const word = reinterpret_cast<uint32_t*>(base + 4u * seg);
        if (PACK) {
            const u32x4 a = bytes[0], b = bytes[1];
            uint32_t v = 0;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)  // four bytes of 0/1 -> four bits
                v |= (((a[j] & 0x01010101u) * 0x10204080u) >> 28) << (4u * j) |
                     (((b[j] & 0x01010101u) * 0x10204080u) >> 28) << (16u + 4u * j);
            *word = v;
        } else {
            const uint32_t v = *word;
            u32x4 a, b;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                a[j] = (((v >> (4u * j)) & 15u) * 0x00204081u) & 0x01010101u;
                b[j] = (((v >> (16u + 4u * j)) & 15u) * 0x00204081u) & 0x01010101u;
            }
            bytes[0] = a;
            bytes[1] = b;
        }
    }
}

}  // namespace vg

namespace vgi {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint8_t* g_scratch[kMaxDevices] = {};

// Device address of the current device's scratch, looked up once per device.
int scratch_of(int device, uint8_t** out) {
    if (device < 0 || device >= kMaxDevices)
        return fail(VG_ERR_INVALID_ARGUMENT, "device %d out of range", device);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(vg::scratch));
        if (e != hipSuccess || !p)
            return fail(VG_ERR_DEVICE, "hipGetSymbolAddress(scratch) failed: %s",
                        hipGetErrorString(e));
        g_scratch[device] = static_cast<uint8_t*>(p);
    }
    *out = g_scratch[device];
    return VG_OK;
}

}  // namespace
}  // namespace vgi

using namespace vgi;

extern "C" int vg_run_sums_noalloc(const vg_chain_desc* desc, double temperature,
                                   double field_magnitude, const double field_orientation[3],
                                   uint64_t sweep0, uint64_t sweeps, void* spins, int64_t* sums,
                                   void* stream) {
    if (!desc) return fail(VG_ERR_INVALID_ARGUMENT, "null descriptor");
    int rc = validate_desc(*desc);
    if (rc) return rc;
    const int g = group_of(*desc);
    if (!is_zmarch(g))
        return fail(VG_ERR_NOT_IMPLEMENTED,
                    "the allocation-free sweeps take Metropolis Ising chains (int8 or bit-packed) "
                    "on sc, bcc or fcc lattices");
    if (std::isnan(temperature) || std::isnan(field_magnitude))
        return fail(VG_ERR_INVALID_ARGUMENT, "NaN thermostat parameter");
    if (sweep0 >> 56 || sweeps > (1ull << 56) - sweep0)
        return fail(VG_ERR_INVALID_ARGUMENT, "sweep counter would pass 2^56");
    if (sweeps == 0) return VG_OK;
    if (!spins || !sums) return fail(VG_ERR_INVALID_ARGUMENT, "null spins or sums");

    // Thermostat and descriptor as a one-chain batch would hold them.
    ChainHost ch;
    ch.desc = *desc;
    ch.n_sites = sites_of(desc->lattice);
    ch.group = g;
    ch.byte_planes = desc->spin == VG_SPIN_ISING;
    ch.temperature = temperature < DBL_EPSILON ? DBL_EPSILON : temperature;
    ch.field_mag = field_magnitude;
    if (field_orientation)
        for (int k = 0; k < 3; ++k) ch.field_dir[k] = field_orientation[k];
    ChainDev d;
    rc = init_chain_dev(ch, g, 0, d);
    if (rc) return rc;
    const uint64_t plane_bytes = round_up(d.plane, 256);
    for (uint32_t c = 0; c < d.ncol; ++c) d.off[c] = c * plane_bytes;
    const uint32_t tile = default_tile(&d, 1);
    d.nzc = (d.lz + tile - 1) / tile;
    const uint64_t items = (uint64_t)d.nzc * d.ly * d.segs;
    if (items > 0x7FFFFFFFull - vg::kBlock)
        return fail(VG_ERR_INVALID_ARGUMENT, "chain too large");
    d.items = (uint32_t)items;
    d.nblocks = (uint32_t)((items + vg::kBlock - 1) / vg::kBlock);
    d.block0 = 0;

    // Scratch layout: descriptor, block map, then as many sweeps' pass
    // partials as fit (8 int32 per workgroup, colour and sweep).
    const uint64_t map_end = vg::kScratchMap + 4ull * d.nblocks;
    const uint64_t part_off = round_up(map_end, 256);
    const uint64_t per_sweep = (uint64_t)d.ncol * d.nblocks * 8u * 4u;
    // A chain is charged for items of four planes, and on bcc and fcc of 16
    // positions, whatever the layout above takes (never more but for chains
    // far from the limit).
    const uint64_t segs = g == kIsingSc ? d.segs : (d.w + 15) / 16;
    const uint64_t blocks =
        ((uint64_t)((d.lz + 3) / 4) * d.ly * segs + vg::kBlock - 1) / vg::kBlock;
    const uint64_t charged = std::max(
        round_up(vg::kScratchMap + 4ull * blocks, 256) + (uint64_t)d.ncol * blocks * 8u * 4u,
        part_off + per_sweep);
    if (charged > vg::kScratchBytes)
        return fail(VG_ERR_INVALID_ARGUMENT,
                    "chain of %llu sites needs %llu bytes of scratch per sweep; the scratch "
                    "holds %llu",
                    (unsigned long long)ch.n_sites, (unsigned long long)charged,
                    (unsigned long long)vg::kScratchBytes);
    const uint64_t chunk = std::min<uint64_t>((vg::kScratchBytes - part_off) / per_sweep, 4096);

    int device = 0;
    VG_HIP(hipGetDevice(&device));
    uint8_t* base = nullptr;
    rc = scratch_of(device, &base);
    if (rc) return rc;
    Group G;  // views of the scratch and the caller's spins; owns nothing
    G.d_chains = reinterpret_cast<ChainDev*>(base + vg::kScratchDesc);
    G.d_block_chain = reinterpret_cast<uint32_t*>(base + vg::kScratchMap);
    G.partials = base + part_off;
    G.arena = spins;
    G.tile = tile;
    G.total_blocks = d.nblocks;
    magic_div(d.nblocks, G.chain_m, G.chain_s);
    G.grid = (uint32_t)round_up(d.nblocks, vg::kNumXcd);
    G.mode = (d.pbc & 7u) == 7u ? 2u : 1u;
    G.prio = all_resident(g, G, tile, G.grid) ? 1u : 0u;
    G.tie_cap = 128;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint64_t rows_per_block = (vg::kBlock / 64u) * (d.segs < 64u ? 64u / d.segs : 1u);
    const dim3 convert((uint32_t)(((uint64_t)d.ncol * d.rows + rows_per_block - 1) / rows_per_block));
    // An error from before the call, and one of the set-up or the packing: the
    // caller's planes are as they were.  After that a failure still unpacks them.
    VG_HIP(hipGetLastError());
    hipError_t e = hipSuccess;
    for (uint64_t done = 0; done < sweeps && e == hipSuccess;) {
        const uint32_t nsw = (uint32_t)std::min<uint64_t>(chunk, sweeps - done);
        d.sweep0 = sweep0 + done;
        hipLaunchKernelGGL(vg::noalloc_setup, dim3((d.nblocks + 255) / 256), dim3(256), 0, st, d,
                           G.d_chains, G.d_block_chain, d.nblocks);
        if (done == 0) VG_HIP(hipGetLastError());
        if (ch.byte_planes && done == 0) {
            hipLaunchKernelGGL(vg::noalloc_bits<true>, convert, dim3(vg::kBlock), 0, st,
                               G.d_chains, static_cast<uint8_t*>(spins));
            VG_HIP(hipGetLastError());
        }
        for (uint32_t s = 0; s < nsw; ++s)
            for (uint32_t c = 0; c < d.ncol; ++c) launch_zmarch_pass(G, g, st, c, s);
        hipLaunchKernelGGL(vg::ising_reduce, dim3(1, nsw), dim3(reduce_block(G.total_blocks)), 0,
                           st, G.d_chains,
                           (const int32_t*)G.partials, G.total_blocks, d.ncol, nsw,
                           sums + 5 * done);
        e = hipGetLastError();
        done += nsw;
    }
    if (ch.byte_planes) {
        hipLaunchKernelGGL(vg::noalloc_bits<false>, convert, dim3(vg::kBlock), 0, st, G.d_chains,
                           static_cast<uint8_t*>(spins));
        if (e == hipSuccess) e = hipGetLastError();
    }
    if (e != hipSuccess)
        return fail(e == hipErrorOutOfMemory ? VG_ERR_OUT_OF_MEMORY : VG_ERR_DEVICE,
                    "launching the sweeps: %s", hipGetErrorString(e));
    return VG_OK;
}
