// Internal interface of the engine shared by the C ABI (capi.hip) and the
// job server (server.hip): chain and group bookkeeping, descriptor upload,
// work layout, the sweep-block driver and the host side of the observables.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/vegas_hip.h"
#include "vg_device.hpp"

namespace vg {
// sc pass args: (chains, block -> chain map, arena, partials, colour, sweep,
// total blocks, grid, options, magic of the blocks per chain or 0).
template <uint32_t K, uint32_t MODE>
__global__ void ising_sc_pass(const ChainDev*, const uint32_t*, uint8_t*, int32_t*, uint32_t,
                              uint32_t, uint32_t, uint32_t, uint32_t, uint32_t);
__global__ void ising_reduce(const ChainDev*, const int32_t*, uint32_t, uint32_t, uint32_t,
                             int64_t*);
__global__ void ising_init(const ChainDev*, uint8_t*);
__global__ void ising_scatter(const ChainDev*, uint8_t*, const int8_t*);
__global__ void ising_gather(const ChainDev*, const uint8_t*, int8_t*, uint64_t);
template <uint32_t S>
__global__ void heis_sc_pass(const ChainDev*, const uint32_t*, float*, int64_t*, uint32_t,
                             uint32_t, uint32_t, uint32_t);
// bcc and fcc passes: one instantiation per colour A (sublattice), args as
// the sc pass's without the colour.
template <uint32_t A, uint32_t K, uint32_t MODE>
__global__ void ising_bcc_pass(const ChainDev*, const uint32_t*, uint8_t*, int32_t*, uint32_t,
                               uint32_t, uint32_t, uint32_t, uint32_t);
template <uint32_t S>
__global__ void heis_bcc_pass(const ChainDev*, const uint32_t*, float*, int64_t*, uint32_t,
                              uint32_t, uint32_t, uint32_t);
__global__ void heis_reduce(const ChainDev*, const int64_t*, uint32_t, uint32_t, uint32_t,
                            int64_t*);
template <uint32_t A, uint32_t K, uint32_t MODE>
__global__ void ising_fcc_pass(const ChainDev*, const uint32_t*, uint8_t*, int32_t*, uint32_t,
                               uint32_t, uint32_t, uint32_t, uint32_t);
// One instantiation per colour A, args (chains, block -> chain map, arena,
// partials, sweep, total blocks, grid).
template <uint32_t A, uint32_t S>
__global__ void heis_fcc_pass(const ChainDev*, const uint32_t*, float*, int64_t*, uint32_t,
                              uint32_t, uint32_t);
// Sweep blocks of small chains, one workgroup a chain.  Z: coordination
// number; R: sites of a colour per lane; SOLO: at most 64, one wave's.
template <uint32_t Z, uint32_t R, bool SOLO>
__global__ void ising_resident(const ChainDev*, uint8_t*, uint32_t, uint32_t, int64_t*);
// Heisenberg: the draws of sweeps s0 .. of a block, and the sweeps on them.
__global__ void heis_draws(const ChainDev*, uint32_t, uint32_t, uint32_t, float4*);
template <uint32_t Z, uint32_t R, bool WIDE>
__global__ void heis_resident(const ChainDev*, float*, uint32_t, uint32_t, uint32_t,
                              const float4*, uint32_t, int64_t*);
// Wolff steps of the chains of one lattice kind (0 sc, 1 bcc, 2 fcc).
template <uint32_t KIND>
__global__ void wolff_run(const ChainDev*, uint8_t*, uint32_t, int64_t*);
template <uint32_t KIND>
__global__ void wolff_run_lds(const ChainDev*, uint8_t*, uint32_t, int64_t*);
__global__ void wolff_init(const ChainDev*, uint8_t*);
__global__ void heis_clear(const ChainDev*, float*);
__global__ void heis_init(const ChainDev*, float*);
__global__ void heis_scatter(const ChainDev*, float*, const double*, uint64_t);
__global__ void heis_gather(const ChainDev*, const float*, double*, uint64_t);
__global__ void zero_i64(int64_t*, uint64_t);
__global__ void copy_words(const uint32_t*, uint32_t*, uint32_t);
__global__ void set_sweeps(const uint64_t*, ChainDev*, uint32_t);
// Graph chains (an arbitrary exchange matrix): one pass per colour class,
// args (chains, block -> chain map, arena, partials, colour, sweep, total
// blocks, passes per sweep); initial states.
__global__ void graph_ising_pass(const ChainDev*, const uint32_t*, uint8_t*, int64_t*, uint32_t,
                                 uint32_t, uint32_t, uint32_t);
__global__ void graph_heis_pass(const ChainDev*, const uint32_t*, uint8_t*, int64_t*, uint32_t,
                                uint32_t, uint32_t, uint32_t);
__global__ void graph_ising_init(const ChainDev*, uint8_t*);
__global__ void graph_heis_init(const ChainDev*, uint8_t*);
}  // namespace vg

using vg::ChainDev;

namespace vgi {

// Thread-local message of the last failure (vg_last_error) and a setter
// that returns the status code.
extern thread_local std::string g_error;
int fail(int code, const char* fmt, ...);

#define VG_HIP(call)                                                                      \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(e_ == hipErrorOutOfMemory ? VG_ERR_OUT_OF_MEMORY : VG_ERR_DEVICE, \
                        "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__,  \
                        __LINE__);                                                        \
    } while (0)

inline uint64_t round_up(uint64_t v, uint64_t m) { return (v + m - 1) / m * m; }

// Best-effort cleanup: errors there cannot be reported to anyone.
inline void quiet(hipError_t) {}

// Kernel groups: chains of one group share an arena and one pass kernel.
enum GroupKind {
    kIsingSc = 0,  // Ising lattice groups: both Ising spin kinds, one bit per site
    kHeisSc = 1,
    kIsingBcc = 2,
    kHeisBcc = 3,
    kIsingFcc = 4,
    kHeisFcc = 5,
    kIsingWolff = 6,  // Wolff cluster steps, any lattice, natural site order
    kIsingGraph = 7,  // arbitrary exchange matrix, int8 Ising, colour classes
    kHeisGraph = 8,   // arbitrary exchange matrix, fp32 Heisenberg
    kNumGroups = 9
};

inline bool is_ising(int g) {
    return g == kIsingSc || g == kIsingBcc || g == kIsingFcc || g == kIsingWolff ||
           g == kIsingGraph;
}
// Groups of chains whose exchange is a matrix (VG_LATTICE_GRAPH).
inline bool is_graph(int g) { return g == kIsingGraph || g == kHeisGraph; }
// Ising lattice groups: planes of one bit per site, a pass that marches a
// tile of z planes per work item.
inline bool is_zmarch(int g) { return g == kIsingSc || g == kIsingBcc || g == kIsingFcc; }
constexpr int kZmarchGroups[] = {kIsingSc, kIsingBcc, kIsingFcc};
// Colours (planes, passes per sweep) of a lattice group's chains; Wolff
// chains have no colour passes; graph groups keep theirs in Group::npass.
inline uint32_t colours_of(int g) {
    return g == kIsingWolff || is_graph(g)
               ? 0u
               : (g == kIsingFcc || g == kHeisFcc ? 4u : 2u);
}

inline int group_of(const vg_chain_desc& d) {
    const int k = d.lattice.kind;
    if (k == VG_LATTICE_GRAPH) return d.spin == VG_SPIN_HEISENBERG ? kHeisGraph : kIsingGraph;
    if (d.proposal == VG_PROPOSAL_WOLFF) return kIsingWolff;
    if (d.spin == VG_SPIN_HEISENBERG)
        return k == VG_LATTICE_FCC ? kHeisFcc : (k == VG_LATTICE_BCC ? kHeisBcc : kHeisSc);
    return k == VG_LATTICE_FCC ? kIsingFcc : (k == VG_LATTICE_BCC ? kIsingBcc : kIsingSc);
}

// Sites of a lattice of lx*ly*lz cells: 1 (sc), 2 (bcc) or 4 (fcc) per cell.
inline uint64_t sites_of(const vg_lattice& L) {
    const uint64_t cells = (uint64_t)L.lx * L.ly * L.lz;
    return L.kind == VG_LATTICE_SC ? cells : (L.kind == VG_LATTICE_BCC ? 2 * cells : 4 * cells);
}

struct Group {
    std::vector<uint32_t> members;  // batch chain indices
    std::vector<ChainDev> host;     // descriptors, uploaded each sweep block
    // What d_chains holds: descriptors as in host (`stale`: or not, whatever sets
    // anything in host but sweep0 says so), with these sweep0
    bool stale = true;
    std::vector<uint64_t> sent_sweeps;
    ChainDev* d_chains = nullptr;
    ChainDev* h_staging = nullptr;  // pinned copy used for the upload
    ChainDev* h_staging2 = nullptr;  // second one, for the block after (batches)
    uint32_t* d_block_chain = nullptr;
    uint32_t block_chain_cap = 0;
    uint32_t tile = 4;  // Ising sc/bcc/fcc: z planes per work item (template parameter)
    // Ising sc/bcc/fcc: the pass's form (vg::IsingMode), with every chain
    // periodic along every axis or not
    uint32_t mode = 1;
    uint32_t total_blocks = 0;
    uint32_t grid = 0;  // total_blocks rounded up to a multiple of 8
    // division by the blocks per chain when every chain of the group has the
    // same number (a pass then finds a block's chain without the map), else 0
    uint32_t chain_m = 0, chain_s = 0;
    uint32_t prio = 0;  // z-marching Ising passes: every workgroup resident at once (wave priorities on)
    // z-marching Ising passes: tie records a wave may queue (at most 128)
    uint32_t tie_cap = 128;
    // Ising sc/bcc/fcc: the caller has set the tile
    bool tile_set = false;
    // Lattice groups: sites of a colour per lane of the resident kernel that
    // runs the group's sweep blocks, 0 when colour passes do
    uint32_t resident = 0;
    // Heisenberg lattice groups: positions per work item (template parameter)
    uint32_t item = 4;
    uint32_t npass = 0;     // graph groups: passes per sweep (the most colours of a member)
    void* arena = nullptr;
    uint64_t arena_bytes = 0;
    void* partials = nullptr;  // [sweep][colour][block][quantity]
    uint64_t partial_bytes_per_sweep = 0;
    // Resident Heisenberg chains: workspace for the draws of draw_sweeps
    // sweeps, draw_stride of them a sweep and chain (the largest chain's sites)
    float4* draws = nullptr;
    uint32_t draw_sweeps = 0, draw_stride = 0;
    bool wide = false;  // resident Heisenberg chains: a member's terms may pass 2 (long_terms)
    // Capacities of d_chains / h_staging (descriptors) and of partials
    // (bytes), for batches whose membership changes (the job server).
    uint32_t chains_cap = 0;
    uint64_t partial_cap = 0;
    bool shared_arena = false;  // arena is owned by someone else (the server's pool)
};

struct ChainHost {
    vg_chain_desc desc;
    uint64_t n_sites = 0;
    uint64_t sweeps = 0;
    double temperature = 2.8;  // Thermostat::new(2.8, Field::zero()) of input.rs:274
    double field_mag = 0.0;
    double field_dir[3] = {0.0, 0.0, 1.0};
    int group = 0;
    uint32_t index = 0;  // index in its group
    // Chains of resident Heisenberg groups: the largest squared length of a spin
    // set by the caller since the last random state (drawn spins have length 1)
    double spin2 = 1.0;
    // The planes are the caller's, with rows of one byte per site (the
    // allocation-free entry point, which keeps a row's bits at its start).
    bool byte_planes = false;
    // Graph chains: sum of the matrix's diagonal (a constant -J_ii in every
    // e_i) and the position of each site in the colour-sorted order.
    double diag = 0.0;
    std::vector<uint32_t> graph_pos;
};

// Passes per sweep of group g.
inline uint32_t passes_of(const Group& G, int g) { return is_graph(g) ? G.npass : colours_of(g); }

}  // namespace vgi

struct vg_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
};

struct vg_batch {
    vg_ctx* ctx = nullptr;
    std::vector<vgi::ChainHost> chains;
    vgi::Group groups[vgi::kNumGroups];
    uint32_t max_block_sweeps = 256;
    int64_t* d_records = nullptr;  // [chain][sweep][5]
    int64_t* h_records = nullptr;  // pinned; batches: h_records2 and io behind them
    int64_t* h_records2 = nullptr;  // for the block after (batches)
    // Every chain runs every sweep of a block, so that the kernels write every
    // record (not in the job server, whose chains stop within a block).
    bool whole_blocks = false;
    // For the states of small chains, at most kIoBytes
    static constexpr uint64_t kIoBytes = 4 << 20;
    void* io = nullptr;
    uint64_t io_bytes = 0;
    // Held while io is used, and while descriptors are compared and sent: states
    // of one batch may be read from several threads.
    std::mutex io_mu, send_mu;
    bool use_graph = false;
    std::map<uint32_t, hipGraphExec_t> graphs;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipEvent_t ev2 = nullptr, ev3 = nullptr;  // the same, for the block after
    hipEvent_t done[2] = {nullptr, nullptr};  // records of a block are on the host
    // Second stream of a sweep block with passes of several groups, and the
    // events that part it from the context's stream and join it again.
    hipStream_t side = nullptr;
    hipEvent_t parted = nullptr, joined = nullptr;
    double last_ms = 0.0;
    // Per-launch timing of the colour-pass kernels (plain launches only).
    bool timing = false;
    std::vector<hipEvent_t> pass_events;  // start/stop pairs
    uint32_t pass_events_used = 0;
    double pass_ms[vgi::kNumGroups] = {};
    uint64_t pass_launches[vgi::kNumGroups] = {};
};

namespace vgi {

// A graph chain's matrix prepared for the graph passes (graph_host.hip).
struct GraphBuild {
    uint32_t ncol = 0;                  // colour classes
    uint32_t max_class = 0;             // sites of the largest class
    std::vector<uint32_t> cstart;       // class starts, ncol + 1 (positions)
    std::vector<uint32_t> site_of_pos;  // positions sorted by (colour, site id)
    std::vector<uint32_t> pos_of_site;
    std::vector<uint32_t> ptr, nbr;     // merged rows by position; neighbours as positions
    std::vector<double> a, w;           // J_ij; J_ij + J_ji for lower-colour neighbours, else 0
    double diag = 0.0;                  // sum of the diagonal entries
};
int build_graph(const vg_csr& m, GraphBuild& out);

// m, s with n / d == (n * m) >> s for every n < 2^31.
void magic_div(uint32_t d, uint32_t& m, uint32_t& s);
int validate_desc(const vg_chain_desc& d);
int coordination(int kind);
void refresh_params(vg_batch* B, uint32_t i);
// Acceptance tables (Ising) or fp32 parameters (Heisenberg) of a chain's
// current thermostat.
void ising_thresholds(const ChainHost& ch, ChainDev& d);
void heis_params(const ChainHost& ch, ChainDev& d);
int free_batch(vg_batch* B);
// Random initial state (State::rand_with_size) of an Ising lattice chain.
void launch_ising_init(const Group& G, const ChainDev& d, const ChainDev* dp, hipStream_t st);
uint32_t quantities(int group);
uint32_t quantity_bytes(int group);
// Copies group g's descriptors to the device through pinned staging buffer
// `slot` (0, or 1 for the second buffer of a batch).
int upload_descriptors(vg_batch* B, int g, int slot = 0);
int layout_work(vg_batch* B, int g, uint32_t tile);
// Whether `grid` workgroups of group g's z-marching pass at this tile are all
// resident at once (the falling wave priorities are used only then).
bool all_resident(int g, const Group& G, uint32_t tile, uint32_t grid);
void launch_zmarch_pass(const Group& G, int g, hipStream_t st, uint32_t c, uint32_t s);
// Threads of ising_reduce for a group of `blocks` pass workgroups.
inline uint32_t reduce_block(uint32_t blocks) { return blocks > 1024 ? 1024u : vg::kBlock; }
// A block of nsw sweeps on the batch's stream, its records to `records`.
int enqueue_block(vg_batch* B, uint32_t nsw, int64_t* records);
// The batch's second stream, for chains in several groups; without one (none can
// be made) every group runs on the first.
void make_side_stream(vg_batch* B);
void free_side_stream(vg_batch* B);
// The same to the device's records, or, where the caller has a pinned buffer
// for them (direct) and no graph is replayed, straight there.
int launch_block(vg_batch* B, uint32_t nsw, int64_t* direct = nullptr);
double sums_scale(int spin);
void observables(const ChainHost& ch, const vg_sweep_sums& r, double* E, double* M);
// Geometry and parameters of chain `ch` as member `slot` of group g (sizes,
// magic divisors, acceptance tables); the plane offsets are set by the caller.
int init_chain_dev(const ChainHost& ch, int g, uint32_t slot, ChainDev& d);
// The tile an Ising lattice group of n chains starts with.
uint32_t default_tile(const ChainDev* chains, size_t n);
// Elements (bytes for Ising, floats for Heisenberg) of one colour of a chain.
uint64_t colour_elems(int g, const ChainDev& d);
// Bytes of one colour plane of an Ising chain at one byte per site: what an
// int8 chain is charged for and limited by.
inline uint64_t byte_plane(const ChainDev& d) {
    return (uint64_t)d.rows * round_up(d.w, 64);
}
// Bytes of one element in group g's arena.
inline uint64_t elem_bytes(int g) { return is_ising(g) || is_graph(g) ? 1 : 4; }

}  // namespace vgi
