// Internal declarations shared by the host engine (pdfxc_host.cpp) and the
// kernels (pdfxc_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/pdfxc.h"

namespace pdfxc {

// precision modes: every non-FP64 mode keeps the split structures and runs the
// K pass on bf16 slices; the rho pass is split only in SPLIT_BF16 / SPLIT_BF16X3
inline bool prec_split_rho(int p) { return p == PDFXC_SPLIT_BF16 || p == PDFXC_SPLIT_BF16X3 || p == PDFXC_SPLIT_BFP; }
// the K pass in FP16 hi + lo with per-slab column exponents (PDFXC_SPLIT_K_F16)
inline bool prec_k_f16(int p) { return p == PDFXC_SPLIT_K_F16; }
// the K pass's slices: bf16 hi + lo, FP16 hi + lo, else bf16 hi + mid + lo
inline int prec_slices(int p) { return (p == PDFXC_SPLIT_BF16 || p == PDFXC_SPLIT_K_F16) ? 2 : 3; }
// the rho pass in block floating point: 4 slices with shared exponents (PDFXC_SPLIT_BFP)
inline bool prec_bfp(int p) { return p == PDFXC_SPLIT_BFP; }
constexpr int kBfpPlanes = 4;
constexpr int kRhoFp64Class = 16;  // split rho launch classes from here on: FP64 k_rho class - kRhoFp64Class
// bf16 elements of one molecule's P slices (and, in block FP, its row exponents after the planes)
inline int64_t psplit_elems(int p, int n) {
    const int64_t nc = (n + 7) / 8 * 8;
    if (prec_bfp(p)) return (kBfpPlanes * (int64_t)n * nc + 2 * (int64_t)n + 7) / 8 * 8;
    return (int64_t)prec_slices(p) * n * nc;
}


constexpr int kBlockPts = 128;  // grid points per block (rows of the MFMA tiles)
constexpr int kColPad = 16;     // AO columns of a block are padded to a multiple of this
constexpr int kMaxPrim = 16;
constexpr double kPi = 3.14159265358979323846;

// One shell = the 2l+1 consecutive AOs that share a centre and primitives.
struct Shell {
    int first_ao;  // global index of the first AO
    int l;         // 0 s, 1 p, 2 d
    int nprim;
    double center[3];
    double exps[kMaxPrim];   // ascending
    double coefs[kMaxPrim];  // normalised
};

constexpr int kMaxDynLds = 160 * 1024 - 16 * 1024;  // dynamic LDS ceiling per workgroup (gfx950: 160 KiB total)

// Device-side view of one grid block.
struct BlockDesc {
    int pt_begin;     // first slot (block-sorted order; every block owns 128 slots)
    int npts;         // real points (<= 128); slots npts..127 have weight 0
    int shell_begin;  // offset into the block-shell list
    int nshell;
    int nao;          // screened AO columns N_b
    int ldn;          // N_b padded to a multiple of kColPad
    int col_begin;    // offset into the block-AO-index list
    int ldp;          // AO count of the block's molecule: leading dimension of its P and K
    int64_t poff;     // offset of the molecule's dense P and K in the P / K buffers
    int64_t psoff;    // offset of the molecule's P slices (split precision)
};

// Split-precision column layout of a block: nchunk 4-aligned runs of AO
// positions in the split order (chunk ids in the chunk list from
// chunk_begin), ldnp = 4 nchunk rounded up to 32.
struct SplitBlock {
    int chunk_begin, nchunk, ldnp, pad;
};

// K pass work unit of k_kmat: 1 to kKGroupMax blocks, neighbours in the point
// bisection, on the union of their shells; all of them but the last full.
constexpr int kKGroupMax = 2;
// Units of two blocks: on grids with at least kKUnitsPerCu of them per CU;
// where the union has at most kKWiderPct % more AOs than the two have on
// average (phi and V of the union are evaluated at the points of both); and
// where its workgroup shape has a unit for every CU (a shape is a launch of its
// own, and one of a few units takes as long as its longest).  K pass, ms, of
// single blocks, all pairs, pairs up to 15 % wider, and those of shapes with a
// unit per CU:
//   blocks (units of two per CU)          single    all    15 %   15 %, filled
//   14,000 (27.4)   10-residue helix       5.50    4.48    4.57      4.58
//    8,500 (16.7)   10 residues            3.51    2.88    2.85      2.84
//    5,300 (10.3)   10 residues            2.29    2.01    1.93      1.90
//    5,200 (10.1)    5 residues            1.66    1.44    1.43      1.42
//   14,000 (27.3)   23 waters              1.16    1.18    1.06      1.02
//    8,400 (16.5)   23 waters              0.76    0.85    0.73      0.68
//    5,200 (10.2)   23 waters              0.52    0.68    0.64      0.48
//    5,200 (10.2)    8 waters              0.256   0.257   0.245     0.243
//    3,200           8 waters              0.234   0.240
//    2,800 (UKS)    12 waters              0.42    0.75
// (79,000 blocks of 30 residues: 37.0 single, 28.1 all pairs; limits of 10 %
// and 30 % are within 2 % of this, two or more units per CU up to 8 % slower).
constexpr int kKUnitsPerCu = 10, kKWiderPct = 15;
// An item has at most kKPatches patches of tiles.
// K items of a workgroup shape join the next wider one below kKJoinPerCu items
// per CU where that has items, and below kKWidenPerCu where it has none (12
// waves take a narrow unit in less time than 4, and CUs are idle).  K pass, us,
// with a launch for every shape, and joined:
//     40 blocks, 187 AOs at most     202     67      235 blocks, 8 waters (13 AOs)  34   34
//     40 blocks, 304                 232    103       40 blocks, 8 waters           66   37
//    313 blocks, 294                 277    207       40 blocks, 96 AOs             59   34
//  2,344 blocks, 185                 657    468    4,688 blocks, 23 waters         562  504
//  4,688 blocks, 284                1477   1297    7,813 blocks, 23 waters         686  682
// (joined at any number: 562 -> 543 and 686 -> 592 in the last two; at 4 items
// per CU: 657 -> 597, 1477 -> 1380.  Widened at 4: 36 -> 50 for 313 blocks.)
constexpr int kKPatches = 36, kKJoinPerCu = 16, kKWidenPerCu = 1;
// Size of the widest shape's items below kKSizePerCu items per CU: an item
// takes about 1.8 us a patch, and for the production of phi and V that every
// item of a block repeats as much as kKCostPerCol patches a column.
constexpr int kKSizePerCu = 4;
constexpr double kKCostPerCol = 0.09;
struct KBlock {
    int slot[kKGroupMax];  // first slot of every block
    int npts;              // real points of all of them
    int shell_begin, nshell, nao, ldn, col_begin;  // as in BlockDesc
    int ldp, pad;
    int64_t poff;
};

// One k_kmat work item: lower 2 x 2 tile patches [t0, t1) of a KBlock, row-major,
// on its first ncols columns and nsh shells, in slabs of ps points.
struct KWork {
    int block, t0, t1, ncols, nsh, ps;
};
// k_kmat workgroup shapes (4, 8 and 12 waves) and the dynamic LDS with which
// 3, 2 and 1 of them share a CU's 160 KiB (under 2 KiB of static LDS each,
// granules of 1280)
constexpr int kKmatClasses = 3;
constexpr size_t kKmatLds[kKmatClasses] = {50 * 1024, 77 * 1024, 157 * 1024};

// A launch of one kernel instantiation over a contiguous range of a work list.
struct LaunchRange {
    int cls;     // template instantiation
    int offset;  // first work item
    int count;   // work items (blocks for k_rho, KWork for k_kmat)
    size_t lds;  // dynamic LDS bytes
};

// A split K pass work unit: 1 to kMaxGroup spatially adjacent blocks
// (siblings of the point bisection) whose K contributions are summed in
// registers on the union of their AO columns before one scatter into K.
constexpr int kMaxGroup = 8;
constexpr int kMaxMaskWords = 32;  // union shells per group <= 32 x 32
struct KGroup {
    int sub_begin;    // the group's blocks: kg_blocks[sub_begin .. + nsub)
    int nsub;
    int shell_begin;  // union shells: kg_shells (global ids, ascending), kg_shell_col, kg_sorder
    int nshell;
    int col_begin;    // union columns: kg_cols (global AO index, ascending)
    int nao;
    int mask_begin;   // kg_masks: nsub x nword words; bit k of block j = union shell k kept by block j
    int nword;
    int ldp;          // P / K leading dimension (the molecule's AO count)
    int pad;
    int64_t poff;     // offset of the molecule's dense P and K
};

// A k_kmat_split item: lower 2 x 2 tile patches [q0, q1) of a group's union
// in column-major order (patch column Q, then rows P >= Q); its slabs hold
// the union columns [c0, c1) (c0 = 32 Q(q0), c1 = 32 Tp), which the union
// shells k0 .. nshell - 1 cover; nbuf slab buffers (1 or 2).
struct KGWork {
    int group, q0, q1, c0, c1, k0, nbuf, pad;
};

// A radial shell of a generated grid: n raw points from `first` on, directions
// (x, y, z, weight) from dir_begin on.
struct RawShell {
    double r, w, center[3];
    int64_t first;
    int dir_begin, n, atom, pad;
};

// What block screening needs of a shell: it is dropped from a block whose
// box lies further than cut, or where exp0 d^2 > 30 (cls: rank of (l, nprim)).
struct ScreenShell {
    double center[3];
    double exp0, cut;
    int l, first_ao, cls, pad;
};

struct DeviceShell {
    double cx, cy, cz;
    int l, nprim;
    int first_ao;
    int pad;
    double exps[kMaxPrim];
    double coefs[kMaxPrim];
};

// Device buffers of one context's grids and workspaces, kept from one grid to
// the next: 18 allocations and as many frees took 4 of the 26 ms of a new
// FINE grid of a 20-residue helix and half of a small density call.  All use
// is on the context's stream, whose work ends before a buffer changes hands.
// At most kPoolKeep bytes are ever kept unused (give frees what is over, the
// largest first), they give way to the context's other allocations
// (release_reserve) and go with the context.  A buffer serves requests down to
// four fifths of its size (and 64 KiB less): a grid holds its buffers for long.
// Several threads may take and give: a grid may be read (pdfxc_get_grid_rows)
// while another thread builds.
constexpr size_t kPoolKeep = (size_t)512 << 20;
class DevicePool {
public:
    ~DevicePool() {
        for (const Buf& b : bufs_) (void)hipFree(b.p);
    }
    hipError_t take(void** p, size_t bytes) {
        std::lock_guard<std::mutex> lock(mu_);
        Buf* best = nullptr;
        for (Buf& b : bufs_)
            if (!b.used && b.cap >= bytes && b.cap <= bytes + bytes / 4 + 65536 && (!best || b.cap < best->cap))
                best = &b;
        if (best) {
            idle_ -= best->cap;
        } else {
            // up to an eighth more than asked for, so that the next geometry's sizes fit
            size_t step = 256;
            while (step * 16 <= bytes) step *= 2;
            const size_t cap = (bytes + step - 1) / step * step;
            void* q = nullptr;
            hipError_t e = hipMalloc(&q, cap);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                trim_locked(0);
                e = hipMalloc(&q, cap);
            }
            if (e != hipSuccess) {
                (void)hipGetLastError();  // the caller has the error; the next launch is not to find it
                return e;
            }
            bufs_.push_back(Buf{q, cap, false});
            best = &bufs_.back();
        }
        best->used = true;
        *p = best->p;
        return hipSuccess;
    }
    bool give(void* p) {  // false: not one of this pool's
        std::lock_guard<std::mutex> lock(mu_);
        for (Buf& b : bufs_)
            if (b.p == p) {
                b.used = false;
                idle_ += b.cap;
                if (idle_ > kPoolKeep) trim_locked(kPoolKeep);
                return true;
            }
        return false;
    }
    void trim(size_t keep) {  // frees unused buffers, the largest first, until at most `keep` bytes are left
        std::lock_guard<std::mutex> lock(mu_);
        trim_locked(keep);
    }

private:
    struct Buf {
        void* p;
        size_t cap;
        bool used;
    };
    void trim_locked(size_t keep) {
        std::sort(bufs_.begin(), bufs_.end(), [](const Buf& a, const Buf& b) { return a.cap < b.cap; });
        while (idle_ > keep) {
            size_t i = bufs_.size();
            while (bufs_[i - 1].used) --i;
            (void)hipFree(bufs_[i - 1].p);
            idle_ -= bufs_[i - 1].cap;
            bufs_.erase(bufs_.begin() + (i - 1));
        }
    }

    std::mutex mu_;
    std::vector<Buf> bufs_;
    size_t idle_ = 0;  // bytes of the buffers not in use
};

struct Context {
    pdfxc_opts opts;
    DevicePool pool;
    bool rho_only = false;      // points for densities alone: no K work, no point terms
    // the points of density_at_points, kept between calls (probe_mu) while its
    // matrices take no more than kPoolKeep; its own way back to this context
    Context* probe = nullptr;
    Context* probe_of = nullptr;
    std::mutex probe_mu;
    pdfxc_tuning tune{0, 96, 0, 24, 4, 2, 0.0};  // launch shapes (pdfxc_set_tuning / pdfxc_autotune)
    int n_aos = 0;
    std::vector<Shell> shells;
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[6] = {};

    // grid in caller order: x, y, z, w columns on the device; host copies only
    // where a caller needs them (ensure_host_grid; host_mu while they are made:
    // batches on several threads may share contexts)
    std::mutex host_mu;
    int64_t n_pts = 0;
    double* d_grid = nullptr;
    std::vector<double> gx, gy, gz, gw;
    std::vector<int> gen_atom;  // atom of each point when pdfxc_generate_grid made the grid
    int grid_partition = 0;     // partition weights of a generated grid (PDFXC_PARTITION_*)
    int grid_size_adjust = 1;   // ... and its Becke size adjustments

    // blocks
    std::vector<BlockDesc> blocks;     // launch order (descending cost)
    // host copies of the block lists and slots, made by ensure_host_lists and
    // ensure_host_slots (a batch's are its own)
    int64_t n_block_shells = 0, n_block_cols = 0;  // those of the K units of several blocks included
    std::vector<KBlock> kblocks;       // units of k_kmat, in launch order
    std::vector<int> block_shells;     // global shell ids per block
    std::vector<int> block_cols;       // global AO index per block column
    std::vector<int> block_shell_col;  // local first column of each block shell
    std::vector<int> block_sorder;     // local shells of each block ordered by (l, nprim)
    std::vector<int64_t> slot_of_point;  // caller point -> slot (block*128 + k)
    std::vector<LaunchRange> rho_launches, kmat_launches;
    double flops = 0.0;
    double mean_nao = 0.0;
    int max_nao = 0;

    // device buffers
    DeviceShell* d_shells = nullptr;
    double* d_shrec = nullptr;  // per shell: cx, cy, cz, l + 4 nprim, (exp, coef) x maxprim
    int rec_stride = 0;
    double* d_pts = nullptr;  // 4 x n_slots SoA: x, y, z, w
    int64_t n_slots = 0;
    char* d_lists = nullptr;  // a context's slots, blocks, units and their lists (a batch has a buffer for each)
    char* d_work = nullptr;   // its rho and K work lists
    int* d_slot_of_point = nullptr;
    BlockDesc* d_blocks = nullptr;
    KBlock* d_kblocks = nullptr;
    int* d_block_shells = nullptr;
    int* d_block_cols = nullptr;
    int* d_block_shell_col = nullptr;
    int* d_block_sorder = nullptr;
    int* d_rho_work = nullptr;    // block indices grouped by k_rho class
    void* d_k_work = nullptr;     // KWork items grouped by k_kmat class
    double* d_coef = nullptr;     // per slot: (w vrho / 2, cx, cy, cz)
    double* d_rho = nullptr;      // per slot: rho, grad rho (4)
    double* d_rho_b = nullptr;    // UKS: beta rho, grad rho per slot (allocated by the first UKS build)
    double* d_coef_b = nullptr;   // UKS: beta point terms
    double* d_eblock = nullptr;   // per 256 slots: energy, then w rho of each spin (k_xc_points partial sums)
    double* d_P = nullptr;        // dense N x N
    double* d_K = nullptr;        // dense N x N
    double* d_P2 = nullptr;       // UKS host entry points: beta P and K (allocated on first use)
    double* d_K2 = nullptr;
    double* d_E = nullptr;        // 1 double
    double* d_packed = nullptr;   // host entry points: packed P in, packed K and E, integrated densities out
    double* h_pinned = nullptr;   // its pinned staging (packed_doubles(N) values)
    int whole_density = 0;        // spins whose integrated density the running build sums (0: none)
    int whole_spins = 0;         // spins of the last host build on this grid, 0 when there is none
    double n_whole[2] = {0.0, 0.0};  // its integrated rho_alpha and rho_beta (0 after an RKS build)

    // split precision (opts.precision != PDFXC_FP64)
    int split_nc = 0;                   // N rounded up to 8: row length of the P slices
    std::vector<int> split_perm;        // split AO order: position -> AO (each atom's shells diffuse first)
    int* d_perm = nullptr;
    std::vector<SplitBlock> sblocks;
    std::vector<int> chunks;            // per block: chunk ids (split-order AO position / 4), ascending
    std::vector<int> sshell_col;        // per block shell: local column in the chunk layout
    std::vector<LaunchRange> srho_launches, sk_launches;
    unsigned short* d_Ps = nullptr;     // S x N x split_nc bf16 slices of P in the split AO order
    SplitBlock* d_sblocks = nullptr;
    int* d_chunks = nullptr;
    int* d_sshell_col = nullptr;
    int* d_srho_work = nullptr;
    // split K pass groups (pdfxc_tuning.split_k_group blocks each) and their items
    std::vector<KGroup> kgroups;
    std::vector<int> kg_blocks, kg_shells, kg_shell_col, kg_sorder, kg_cols;
    std::vector<unsigned> kg_masks;
    KGroup* d_kgroups = nullptr;
    int* d_kg_blocks = nullptr;
    int* d_kg_shells = nullptr;
    int* d_kg_shell_col = nullptr;
    int* d_kg_sorder = nullptr;
    int* d_kg_cols = nullptr;
    unsigned* d_kg_masks = nullptr;
    KGWork* d_kg_work = nullptr;        // items of k_kmat_split
    std::vector<LaunchRange> k_fp64_launches;  // k_kmat items of blocks too wide for k_kmat_split
    int64_t n_k_fp64_blocks = 0;

    int rho_accumulate = 0;             // update mode: the rho kernels add rho[dP] to d_rho

    // persistent launches: work-queue counters of one build sequence (zeroed
    // by a fill kernel when the sequence starts), the next free one, and the
    // device's compute units
    int* d_queue = nullptr;             // kMaxQueues counters
    int n_queue_used = 0;
    bool queue_open = false;            // begin_queues ran for the current sequence
    int n_cu = 0;

    // host copies of the device work lists (d_rho_work, d_k_work, d_srho_work, d_sk_work)
    std::vector<int> h_rho_work, h_srho_work;
    std::vector<KWork> h_k_work;
    std::vector<KGWork> h_kg_work;

    // batches: P slices made per molecule (empty for one molecule)
    struct PsplitJob {
        int64_t poff, psoff;
        int perm_off, n;
    };
    std::vector<PsplitJob> psplit_jobs;

    double last_build_ms = 0.0;
    double last_kernel_ms[4] = {0, 0, 0, 0};
};

constexpr int kMaxQueues = 64;  // persistent launches per build sequence

// packed P or K of two spins, then E_xc and the two integrated densities
inline size_t packed_doubles(int n) { return (size_t)n * (n + 1) + 3; }

// error helpers
void set_error(const std::string& msg);
int hip_fail(hipError_t e, const char* what);

#define PDFXC_HIP(call)                                          \
    do {                                                         \
        hipError_t e_ = (call);                                  \
        if (e_ != hipSuccess) return ::pdfxc::hip_fail(e_, #call); \
    } while (0)

// device memory for the length of a call, from the context's pool
int context_take(Context& c, void** p, size_t bytes);
void context_give(Context& c, void* p);

// host copies of a context's grid, block lists and slots (no-ops once made)
int ensure_host_grid(Context& c);
int ensure_host_lists(Context& c);
int ensure_host_slots(Context& c);

// Grids of up to kHostPts points that came from the host stay there as well, and
// are read there (60,000 points: 34 us, about 150 by rows from the device); up to
// kHostCut points the host cuts them into blocks, and up to kHostRho points it
// puts rho in order (a build of 8 waters with rho: 11 us more than without for
// 1,000 points, 60 for 20,000, either way, against 47 and 55 by the device).
constexpr int64_t kHostPts = 65536, kHostCut = 6144, kHostRho = 16384;
void partition_points(const Context& c, std::vector<int>& order);

// (rho, grad rho) of nspin spins from their slots to rows of 4 nspin in the
// caller's order, and of one spin from such rows of 4 to its slots
int rho_to_host(Context& c, int nspin, const double* const* d_slots, double* rows);
int rho_from_host(Context& c, const double* rows, double* d_slots);

// grid blocks (pdfxc_blocks.hip)
// d_order: the points of block b are d_order[128 b ..); synchronises s
int device_partition(int64_t n, const double* d_grid, int* d_order, hipStream_t s, DevicePool& pool);
// lowers *d_first to the first point with a non-finite value
int device_check_finite(int64_t n, const double* d_grid, unsigned long long* d_first, hipStream_t s);
// generated grids: raw points, first kept point of every shell (d_first[ns]: their number), kept points
int launch_raw_points(int ns, const RawShell* d_shells, const double* d_dirs, double* d_pts, double* d_w, int* d_atom,
                      hipStream_t s);
int launch_keep_count(int ns, const RawShell* d_shells, const double* d_w, double cutoff, long long* d_first,
                      hipStream_t s);
int launch_keep_write(int ns, const RawShell* d_shells, const double* d_pts, const double* d_w, double cutoff,
                      const long long* d_first, int64_t n, double* d_grid, hipStream_t s);
int launch_grid_rows(int64_t first, int64_t n, int64_t stride, const double* d_grid, double* d_rows, hipStream_t s);
int launch_screen_blocks(int nb, int64_t n, const double* d_grid, const int* d_order, int nsh,
                         const ScreenShell* d_shells, int nw, unsigned long long* d_masks, int* d_counts,
                         hipStream_t s);
int launch_fill_blocks(Context& c, const int* d_order, const int* d_leaf, int nw, int ncls,
                       const ScreenShell* d_shells, const unsigned long long* d_masks);
// shells of blocks [g per, (g + 1) per) together: masks, (shells, AOs) counts, lists of c.kblocks
int launch_group_masks(int nb, int per, int nsh, const ScreenShell* d_shells, int nw,
                       const unsigned long long* d_masks, unsigned long long* d_gmasks, int* d_gcounts, hipStream_t s);
int launch_fill_groups(Context& c, int n, const int* d_group, int nw, int ncls, const ScreenShell* d_shells,
                       const unsigned long long* d_gmasks);
int launch_item_shells(Context& c, int n, const KWork* d_work, int* d_nsh);
// four values per point between the slots and n points of the caller's order from `first` on (its row stride and offset)
int launch_gather_points(Context& c, int64_t first, int64_t n, const double* d_slots, double* d_pts, int stride, int off);
int launch_gather_density(Context& c, const double* d_slots, double* d_out, bool grad);  // rho [n] | grad [n][3]
int launch_scatter_points(Context& c, int64_t first, int64_t n, const double* d_pts, double* d_slots);
int launch_scatter_atoms(Context& c, const int* d_atom, int* d_slot_atom);
int launch_points_to_grid(int64_t n, const double* d_xyz, double* d_grid, hipStream_t s);

// kernel launchers (pdfxc_kernels.hip)
int launch_rho(Context& c, const LaunchRange& r);
int rho_points_per_workgroup(int cls);
// dynamic LDS the 64-point k_rho class of ldn <= 256 blocks may take: 160 KiB
// less the kernel's static LDS, read from the code object
int rho64_max_dyn_lds(size_t* out);
int launch_xc_points(Context& c, int xc_type, double* d_ewf = nullptr);
int launch_kmat(Context& c, const LaunchRange& r);
int configure_kernels();
int launch_energy_sum(Context& c, double* dE);
// packed lower triangle -> dense symmetric dP, dK (if given) cleared; lower triangle of dK -> packed
int launch_unpack(int N, const double* d_packed, double* dP, double* dK, hipStream_t s);
int launch_pack(int N, const double* dK, double* d_packed, hipStream_t s);
int launch_zero(double* d, int64_t n, hipStream_t s);
// start a build sequence's persistent launches: zero the counters on the stream
int begin_queues(Context& c);
// kernel families of pdfxc_tuning.persistent (bit mask)
constexpr int kQueueRho = 1, kQueueK = 2;
// grid and queue of a launch of n_items work items of a kernel family whose
// persistent instantiation keeps `per_cu` workgroups resident per compute
// unit: a persistent launch of the resident workgroups over the next counter
// when the items exceed them (and the sequence's counters are open and the
// family's bit of tune.persistent is set), else one workgroup per item of the
// plain instantiation (queue = nullptr)
int* launch_queue(Context& c, int kind, int n_items, int per_cu, unsigned* grid);
// workgroups of `kernel` resident per compute unit at `threads` and `lds` bytes
// of dynamic LDS (at least 1)
template <typename Kernel>
inline int resident_per_cu(Kernel kernel, int threads, size_t lds) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reinterpret_cast<const void*>(kernel), threads, lds) !=
        hipSuccess) {
        (void)hipGetLastError();
        nb = 1;
    }
    return nb > 0 ? nb : 1;
}
int launch_energy_sums(Context& c, const int* d_bounds, int n_mol, double* dE);  // one E per molecule
int launch_xc_points_uks(Context& c, int xc_type);
int ensure_beta_buffers(Context* c);  // UKS beta rho / point-term buffers, zeroed when first made
int launch_eval_functional_uks(int xc_type, int64_t n, const double* d_in, double* d_out, hipStream_t s);
int launch_eval_functional(int xc_type, int64_t n, const double* d_in, double* d_out, hipStream_t s);
// pdfxc_eval_functional through the library's own device staging (no allocation)
int eval_functional_noalloc(int xc_type, int64_t n, const double* in, double* out);
int launch_eval_aos_points(const Context& c, int64_t n, const double* d_xyz, double* d_out,
                           hipStream_t s);
int launch_becke(const double* d_atoms, int n_atoms, int64_t n, const double* d_pts,
                 const int* d_atom_of_pt, double* d_w, int partition, hipStream_t s);
int launch_mfma_selftest(double* d_out, hipStream_t s);
// split precision (pdfxc_split.hip)
int split_points_per_workgroup(int cls);
// block-FP rho classes 0, 1, 2: 64, 32, 16 points per workgroup, blocks of at
// most 256, 384, 512 chunked columns; the dynamic LDS a class may take
int bfp_points_per_workgroup(int cls);
int bfp_max_columns(int cls);
int bfp_max_dyn_lds(int cls, size_t* out);
int launch_split_rho(Context& c);   // P slices + k_rho_split
int launch_split_kmat(Context& c);  // k_kmat_split
int split_kmat_max_dyn_lds(int S, size_t* out);
int launch_mfma_split_selftest(float* d_out, hipStream_t s);
constexpr int kNear = 16;  // entries per atom of a near-atom table
// XC nuclear gradient (pdfxc_grad.hip); d_gacc: functional term [3 n_atoms] then weight term [3 n_atoms]
int launch_grad_fn(Context& c, const LaunchRange& r, const int* d_shell_atom, const int* d_slot_atom,
                   int n_atoms, double* d_gacc);
// d_near: near_atoms() of the molecule
int launch_grad_w(Context& c, const double* d_atoms, const int* d_near, int n_atoms, const int* d_slot_atom,
                  const double* d_ewf, double* d_gacc, int partition);
int launch_copy(const double* src, double* dst, int64_t n, hipStream_t s);

}  // namespace pdfxc
