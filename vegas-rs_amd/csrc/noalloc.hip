// vg_run_sums_noalloc: the sweeps of vg_batch_run_sums for one Ising chain
// on caller-owned device buffers, allocating nothing.
//
// A batch allocates its arena, descriptors, block map, pass partials and
// records when it is created.  Here the caller brings the spins (in the
// batch arena's colour-plane layout) and the output sums; the descriptor,
// the block -> chain map, the pass partials and the bits of int8 planes live
// in `scratch`, a file-scope device array of kScratchBytes + kPlaneBytes that
// every GPU the library runs on holds until the process ends.  Host code
// reaches a device's copy only
// through the address hipGetSymbolAddress returns for it (kept per device):
// the array's name in host code is a host-side stand-in, not a device
// address.  The descriptor reaches the scratch through a kernel argument,
// so a call makes no host-to-device copy either.  Calls on one GPU share its
// scratch, and everything a call reads there it has written first, so
// nothing needs clearing; calls that overlap on one GPU race.
#include <mutex>

#include "engine.hpp"
#include "ising_word.hpp"

namespace vg {

constexpr uint64_t kScratchBytes = 16ull << 20;
constexpr uint64_t kPlaneBytes = 40ull << 20;  // the planes of an int8 chain, as bits
static __device__ __align__(256) uint8_t scratch[kScratchBytes + kPlaneBytes];

constexpr uint64_t kScratchDesc = 0;      // ChainDev
constexpr uint64_t kScratchMap = 4096;    // block -> chain map (all 0)
static_assert(sizeof(ChainDev) <= kScratchMap, "descriptor slot too small");

// Planes of int8 chains, one byte of 0/1 per position, are packed to one bit per
// position before the first sweep and unpacked after the last, whatever the
// number of sweeps: passes on the bytes read and wrote eight times as much,
// packed every row they read and unpacked every row they wrote.
//
// Chains whose bits fit kPlaneBytes are packed into the scratch: dense rows for
// the passes, and the caller's planes are written once, with the result.  The
// conversions are parts of launches that are made anyway, of noalloc_setup and
// noalloc_finish: a kernel of its own for each costs 2 us and more, which one sweep
// does not earn back.  A lane converts sixteen positions: 16 bytes on the one side
// and 2 on the other, both whole lines of a wave.  us a call of one sweep, by
// passes on bytes, with the bits in place and with the bits here: sc 128^3 37,
// 34, 31; 256^3 39, 51, 39; 512^3 98, 112, 86; bcc 200^3 40, 49, 45; fcc 200^3
// 73, 82, 71; of two sweeps sc 256^3 60, 64, 53; 512^3 172, 147, 113.  (The one
// loss to the bytes, some 16 million sites of bcc in a single sweep, is the last
// launch: 17 MB written after the bits' loads, 11 us beside 3.5 for sums alone.)
// In units of one, two and eight sixteens a lane: the same within 2%.
struct ByteRows {
    uint64_t plane, bit_plane;  // bytes from colour to colour, of the one and the other
    uint32_t pitch, bit_pitch;  // bytes from row to row
    uint32_t units;             // sixteens of positions of a colour
    uint32_t segs, segs_m, segs_s;
    uint32_t blocks;            // workgroups that convert one colour
};
constexpr uint32_t kUnits = 4;  // sixteens a lane

// The part of workgroup b (of `block` threads) in the conversion.  (The geometry
// comes with the launch: read from the descriptor it is one more wait.)
template <bool PACK>
__device__ __forceinline__ void convert_planes(const ByteRows& R, uint32_t ncol, uint32_t b,
                                               uint32_t block, uint8_t* __restrict__ bits,
                                               uint8_t* __restrict__ bytes) {
    const uint32_t colour = b / R.blocks;
    if (colour >= ncol) return;
    const uint32_t first = (b - colour * R.blocks) * (kUnits * block) + threadIdx.x;
    const __amdgpu_buffer_rsrc_t wide = plane_rsrc(
        reinterpret_cast<const uint8_t*>(uniform64((uint64_t)(bytes + colour * R.plane))),
        (uint32_t)R.plane);
    uint8_t* const narrow = bits + colour * R.bit_plane;
    u32x4 v[kUnits];
    uint16_t h[kUnits];
    uint32_t at[kUnits], out[kUnits];
#pragma unroll
    for (uint32_t j = 0; j < kUnits; ++j) {
        const uint32_t u = min(first + j * block, R.units - 1u), word = u >> 1;
        const uint32_t row = fast_div(word, R.segs_m, R.segs_s), seg = word - row * R.segs;
        at[j] = row * R.pitch + 32u * seg + 16u * (u & 1u);
        out[j] = row * R.bit_pitch + 4u * seg + 2u * (u & 1u);
        if (PACK)
            v[j] = bload16(wide, at[j]);
        else
            h[j] = *reinterpret_cast<const uint16_t*>(narrow + out[j]);
    }
#pragma unroll
    for (uint32_t j = 0; j < kUnits; ++j) {
        if (first + j * block >= R.units) break;
        if (PACK) {
            uint32_t m = 0;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)  // four bytes of 0/1 -> four bits
                m |= (((v[j][k] & 0x01010101u) * 0x10204080u) >> 28) << (4u * k);
            *reinterpret_cast<uint16_t*>(narrow + out[j]) = (uint16_t)m;
        } else {
            u32x4 w;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                w[k] = (((h[j] >> (4u * k)) & 15u) * 0x00204081u) & 0x01010101u;
            // written through the caches (sc1): nothing else of the call reads
            // them, and lines left dirty are written when the launch ends
            __builtin_amdgcn_raw_buffer_store_b128(w, wide, at[j], 0, 16);
        }
    }
}

// Writes the chain's descriptor and the block -> chain map into the scratch and,
// with PACK, the caller's planes as bits.
template <bool PACK>
__global__ __launch_bounds__(256) void noalloc_setup(ChainDev d, ByteRows R,
                                                     ChainDev* __restrict__ out,
                                                     uint32_t* __restrict__ block_chain,
                                                     uint8_t* __restrict__ bits,
                                                     uint8_t* __restrict__ bytes) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *out = d;
    if (i < d.nblocks) block_chain[i] = 0;
    if (PACK) convert_planes<true>(R, d.ncol, blockIdx.x, 256u, bits, bytes);
}

// The last sums of a call, a sweep a workgroup as ising_reduce does, and beside
// them the planes back to bytes.
__global__ __launch_bounds__(1024) void noalloc_finish(const ChainDev* __restrict__ chain, ByteRows R,
                                                    const int32_t* __restrict__ partials,
                                                    uint32_t total_blocks, uint32_t ncol,
                                                    uint32_t nsw, int64_t* __restrict__ records,
                                                    uint8_t* __restrict__ bits,
                                                    uint8_t* __restrict__ bytes) {
    if (blockIdx.x < nsw)
        reduce_sweep(*chain, partials, total_blocks, ncol, nsw, blockIdx.x, records);
    else
        convert_planes<false>(R, ncol, blockIdx.x - nsw, blockDim.x, bits, bytes);
}

// Larger chains: bytes to bits in place, and back.  A row's bits take the first
// eighth of its bytes, so that a row is one wave's own work: `rows` of 64 lanes hold one row
// of at most 64 segments (32 positions: 32 bytes, one word) or several, and a
// longer row is walked in chunks of 64 segments.  A chunk's loads end before
// its stores start (each word is made of its own bytes, and the lanes of a
// wave load together); chunk c's words lie in [256c, 256c + 256), below the
// bytes [2048c', ...) of every later chunk c', so packing walks upwards and
// unpacking downwards.  Only whole segments are touched, and their padding is
// zero before and after.
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
    ch.temperature = temperature < DBL_EPSILON ? DBL_EPSILON : temperature;
    ch.field_mag = field_magnitude;
    if (field_orientation)
        for (int k = 0; k < 3; ++k) ch.field_dir[k] = field_orientation[k];
    ChainDev d;
    rc = init_chain_dev(ch, g, 0, d);
    if (rc) return rc;
    // int8 planes: bits in the scratch where those fit, else in place
    const bool bytes = desc->spin == VG_SPIN_ISING;
    const bool dense = bytes && (uint64_t)d.ncol * round_up(d.plane, 256) <= vg::kPlaneBytes;
    if (bytes && !dense) {
        ch.byte_planes = true;
        rc = init_chain_dev(ch, g, 0, d);
        if (rc) return rc;
    }
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
    uint8_t* const bits = dense ? base + vg::kScratchBytes : static_cast<uint8_t*>(spins);
    G.arena = bits;
    G.tile = tile;
    G.total_blocks = d.nblocks;
    magic_div(d.nblocks, G.chain_m, G.chain_s);
    G.grid = (uint32_t)round_up(d.nblocks, vg::kNumXcd);
    G.mode = (d.pbc & 7u) == 7u ? 2u : 1u;
    G.prio = all_resident(g, G, tile, G.grid) ? 1u : 0u;
    G.tie_cap = 128;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* const planes = static_cast<uint8_t*>(spins);
    const uint32_t threads = reduce_block(G.total_blocks);
    const uint32_t units = 2u * d.rows * d.segs;
    const auto rows = [&](uint32_t block) {  // of byte planes, converted by workgroups of `block`
        return vg::ByteRows{round_up(byte_plane(d), 256), plane_bytes, (uint32_t)round_up(d.w, 64),
                            d.pitch, units, d.segs, d.segs_m, d.segs_s,
                            (units + vg::kUnits * block - 1) / (vg::kUnits * block)};
    };
    const vg::ByteRows packed = rows(256), unpacked = rows(threads);
    const uint64_t rows_per_block = (vg::kBlock / 64u) * (d.segs < 64u ? 64u / d.segs : 1u);
    const dim3 in_place((uint32_t)(((uint64_t)d.ncol * d.rows + rows_per_block - 1) / rows_per_block));
    // An error from before the call, and one of the set-up or the packing: the
    // caller's planes are as they were.  After that a failure still unpacks them.
    VG_HIP(hipGetLastError());
    hipError_t e = hipSuccess;
    for (uint64_t done = 0; done < sweeps && e == hipSuccess;) {
        const uint32_t nsw = (uint32_t)std::min<uint64_t>(chunk, sweeps - done);
        d.sweep0 = sweep0 + done;
        const uint32_t setup = (d.nblocks + 255) / 256;
        if (dense && done == 0)
            hipLaunchKernelGGL(vg::noalloc_setup<true>,
                               dim3(std::max(setup, d.ncol * packed.blocks)), dim3(256), 0, st, d,
                               packed, G.d_chains, G.d_block_chain, bits, planes);
        else
            hipLaunchKernelGGL(vg::noalloc_setup<false>, dim3(setup), dim3(256), 0, st, d, packed,
                               G.d_chains, G.d_block_chain, bits, planes);
        if (done == 0) VG_HIP(hipGetLastError());
        if (ch.byte_planes && done == 0) {
            hipLaunchKernelGGL(vg::noalloc_bits<true>, in_place, dim3(vg::kBlock), 0, st,
                               G.d_chains, planes);
            VG_HIP(hipGetLastError());
        }
        for (uint32_t s = 0; s < nsw; ++s)
            for (uint32_t c = 0; c < d.ncol; ++c) launch_zmarch_pass(G, g, st, c, s);
        if (dense && done + nsw == sweeps)
            hipLaunchKernelGGL(vg::noalloc_finish, dim3(nsw + d.ncol * unpacked.blocks), dim3(threads),
                               0, st, G.d_chains, unpacked, (const int32_t*)G.partials,
                               G.total_blocks, d.ncol, nsw, sums + 5 * done, bits, planes);
        else
            hipLaunchKernelGGL(vg::ising_reduce, dim3(1, nsw), dim3(threads), 0, st, G.d_chains,
                               (const int32_t*)G.partials, G.total_blocks, d.ncol, nsw,
                               sums + 5 * done);
        e = hipGetLastError();
        done += nsw;
        if (dense && e != hipSuccess && done < sweeps)  // the state that the launches reached
            hipLaunchKernelGGL(vg::noalloc_finish, dim3(d.ncol * unpacked.blocks), dim3(threads), 0, st,
                               G.d_chains, unpacked, (const int32_t*)G.partials, G.total_blocks,
                               d.ncol, 0u, sums, bits, planes);
    }
    if (ch.byte_planes) {
        hipLaunchKernelGGL(vg::noalloc_bits<false>, in_place, dim3(vg::kBlock), 0, st, G.d_chains,
                           planes);
        if (e == hipSuccess) e = hipGetLastError();
    }
    if (e != hipSuccess)
        return fail(e == hipErrorOutOfMemory ? VG_ERR_OUT_OF_MEMORY : VG_ERR_DEVICE,
                    "launching the sweeps: %s", hipGetErrorString(e));
    return VG_OK;
}
