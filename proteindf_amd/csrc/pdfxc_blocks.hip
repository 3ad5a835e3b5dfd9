// Grid blocks on the device: the recursive bisection of the points, the AO
// screening of every block and the block lists, so that a new grid (a new
// geometry, the points of a density plot) costs no host pass over its points.
//
// The bisection cuts a node of n > 128 points along the widest extent of its
// bounding box, at the element of rank 128 floor(ceil(n / 128) / 2) in the
// order (coordinate, point index).  The cut ranks depend on n alone, so the
// tree (node ranges, chunks of every level) is known before the points are
// looked at, and block b is the run [128 b, 128 b + 128) of the final order.
//   nodes of more than kNodeMax points, a level at a time over the whole chip:
//     k_part_box    bounding boxes (one atomic per chunk of 4096 points and side)
//     k_part_hist   radix selection of the cut's key, 8 bits per launch: 8
//                   launches for the coordinate and 4 for the index that
//                   breaks ties (grids are full of equal coordinates)
//     k_part_split  points to the two sides (their order within a side is
//                   left open: the last cuts order every block)
//   k_part_leaf   nodes of at most kNodeMax points: one workgroup takes a
//                 node's points into LDS and does all its cuts there, each by
//                 a bitonic sort of 16-bit positions
// Then one wave per block: k_screen_blocks (box, shells kept, as a bit mask)
// and k_fill_blocks (the mask expanded into the block lists, the slots).
// The passes of the upper levels stream the points from HBM / L2; 1.5 million
// points take 9 levels.  On the host the same cuts (std::nth_element over an
// index array), the screening and the lists took 185, 104 and 78 ms for those
// 1.5 million points in 11,900 blocks, against 1.9, 0.06 and 0.16 ms here.
// (Grids of few points and the split precision modes take the host's cuts, see
// partition_points.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "pdfxc_internal.hpp"
#include "pdfxc_partition.hpp"

namespace pdfxc {

namespace {

static_assert(kLeafPts == kBlockPts, "a leaf of the bisection is a block");
constexpr int kPasses = 12;     // 8-bit digits: 8 of the coordinate's key, 4 of the index

struct PartState {  // per node
    unsigned long long box[6];  // ordered keys: min of 3 dimensions, then max
    unsigned long long prefix[kPasses + 1];
    unsigned int iprefix[kPasses + 1];
    int rank[kPasses + 1];
    int cursor[2];
};
struct PartBuf {
    double* v[3];
    int* idx;
};

// order-preserving 64-bit key of a double (-0 as +0, as the comparison has it)
__device__ inline unsigned long long key_of(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x + 0.0);
    return (b >> 63) ? ~b : b | 0x8000000000000000ull;
}
__device__ inline double of_key(unsigned long long k) {
    return __longlong_as_double((long long)((k >> 63) ? k & 0x7fffffffffffffffull : ~k));
}

__device__ inline int widest(const double* mn, const double* mx) {
    int dim = 0;
    for (int d = 1; d < 3; ++d)
        if (mx[d] - mn[d] > mx[dim] - mn[dim]) dim = d;
    return dim;
}
__device__ inline int state_dim(const PartState& s) {
    double mn[3], mx[3];
    for (int d = 0; d < 3; ++d) {
        mn[d] = of_key(s.box[d]);
        mx[d] = of_key(s.box[3 + d]);
    }
    return widest(mn, mx);
}

__global__ __launch_bounds__(256) void k_part_start(int64_t n, const double* __restrict__ grid, PartBuf b) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    for (int d = 0; d < 3; ++d) b.v[d][i] = grid[d * n + i];
    b.idx[i] = (int)i;
}

__global__ __launch_bounds__(256) void k_part_init(const PartNode* __restrict__ nodes, PartState* __restrict__ st,
                                                   unsigned int* __restrict__ hist) {
    const int node = blockIdx.x, t = threadIdx.x;
    for (int p = 0; p < kPasses; ++p) hist[((int64_t)node * kPasses + p) * 256 + t] = 0u;
    if (t < 6) st[node].box[t] = t < 3 ? ~0ull : 0ull;
    if (t == 0) {
        const PartNode N = nodes[node];
        st[node].prefix[0] = 0ull;
        st[node].iprefix[0] = 0u;
        st[node].rank[0] = N.mid - N.lo;
        st[node].cursor[0] = N.lo;
        st[node].cursor[1] = N.mid;
    }
}

__global__ __launch_bounds__(256) void k_part_box(const PartChunk* __restrict__ chunks, PartBuf b,
                                                  PartState* __restrict__ st) {
    __shared__ unsigned long long s_k[6];
    const PartChunk C = chunks[blockIdx.x];
    const int t = threadIdx.x;
    if (t < 6) s_k[t] = t < 3 ? ~0ull : 0ull;
    __syncthreads();
    for (int d = 0; d < 3; ++d) {
        unsigned long long mn = ~0ull, mx = 0ull;
        each_point(C, t, [&](int i) {
            const unsigned long long k = key_of(b.v[d][i]);
            mn = k < mn ? k : mn;
            mx = k > mx ? k : mx;
        });
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long a = __shfl_xor(mn, off), c = __shfl_xor(mx, off);
            mn = a < mn ? a : mn;
            mx = c > mx ? c : mx;
        }
        if ((t & 63) == 0) {
            atomicMin(&s_k[d], mn);
            atomicMax(&s_k[3 + d], mx);
        }
    }
    __syncthreads();
    if (t < 3) atomicMin(&st[C.node].box[t], s_k[t]);
    else if (t < 6) atomicMax(&st[C.node].box[t], s_k[t]);
}

// the state after pass p - 1's histogram: the digit that holds the rank
// (computed by every workgroup of the node; 256 threads)
__device__ inline void part_pick(int p, const PartState& st, const unsigned int* __restrict__ hist,
                                 unsigned long long* prefix, unsigned int* iprefix, int* rank) {
    __shared__ int s_w[4];
    __shared__ unsigned long long s_prefix;
    __shared__ unsigned int s_iprefix;
    __shared__ int s_rank;
    const int t = threadIdx.x;
    if (p == 0) {
        *prefix = st.prefix[0];
        *iprefix = st.iprefix[0];
        *rank = st.rank[0];
        return;
    }
    const int h = (int)hist[(p - 1) * 256 + t];
    int inc = h;
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(inc, off);
        if ((t & 63) >= off) inc += u;
    }
    if ((t & 63) == 63) s_w[t >> 6] = inc;
    __syncthreads();
    for (int w = 0; w < (t >> 6); ++w) inc += s_w[w];
    const int k = st.rank[p - 1];
    if (inc - h <= k && k < inc) {
        s_rank = k - (inc - h);
        s_prefix = p <= 8 ? (st.prefix[p - 1] << 8) | (unsigned long long)t : st.prefix[p - 1];
        s_iprefix = p <= 8 ? 0u : (st.iprefix[p - 1] << 8) | (unsigned int)t;
    }
    __syncthreads();
    *prefix = s_prefix;
    *iprefix = s_iprefix;
    *rank = s_rank;
}

__global__ __launch_bounds__(256) void k_part_hist(int p, const PartChunk* __restrict__ chunks,
                                                   const PartNode* __restrict__ nodes, PartBuf b,
                                                   PartState* __restrict__ st, unsigned int* __restrict__ hist) {
    __shared__ unsigned int s_h[256];
    const PartChunk C = chunks[blockIdx.x];
    const int t = threadIdx.x;
    unsigned int* nh = hist + (int64_t)C.node * kPasses * 256;
    s_h[t] = 0u;
    unsigned long long prefix;
    unsigned int iprefix;
    int rank;
    part_pick(p, st[C.node], nh, &prefix, &iprefix, &rank);
    if (p > 0 && t == 0 && C.lo == nodes[C.node].lo) {
        st[C.node].prefix[p] = prefix;
        st[C.node].iprefix[p] = iprefix;
        st[C.node].rank[p] = rank;
    }
    __syncthreads();
    const double* v = b.v[state_dim(st[C.node])];
    each_point(C, t, [&](int i) {
        const unsigned long long k = key_of(v[i]);
        if (p < 8) {
            if (p == 0 || (k >> (64 - 8 * p)) == prefix) atomicAdd(&s_h[(k >> (56 - 8 * p)) & 255u], 1u);
        } else if (k == prefix) {
            const unsigned int ix = (unsigned int)b.idx[i];
            const int q = p - 8;
            if (q == 0 || (ix >> (32 - 8 * q)) == iprefix) atomicAdd(&s_h[(ix >> (24 - 8 * q)) & 255u], 1u);
        }
    });
    __syncthreads();
    if (s_h[t]) atomicAdd(&nh[p * 256 + t], s_h[t]);
}

__global__ __launch_bounds__(256) void k_part_split(const PartChunk* __restrict__ chunks, PartBuf src, PartBuf dst,
                                                    PartState* __restrict__ st,
                                                    const unsigned int* __restrict__ hist) {
    __shared__ int s_cnt[4], s_base[2];
    const PartChunk C = chunks[blockIdx.x];
    const int t = threadIdx.x, wave = t >> 6;
    unsigned long long prefix;
    unsigned int iprefix;
    int rank;
    part_pick(kPasses, st[C.node], hist + (int64_t)C.node * kPasses * 256, &prefix, &iprefix, &rank);
    const double* v = src.v[state_dim(st[C.node])];
    const int n = C.hi - C.lo;
    // which of this thread's points go left: those below the cut's (coordinate, index)
    unsigned int left = 0u;
    int nleft = 0;
    for (int r = 0; r < kChunk / 256; ++r) {
        const int j = r * 256 + t;  // within the chunk
        bool l = false;
        if (j < n) {
            const int i = C.lo + j;
            const unsigned long long k = key_of(v[i]);
            l = k < prefix || (k == prefix && (unsigned int)src.idx[i] < iprefix);
        }
        left |= (l ? 1u : 0u) << r;
        nleft += __popcll(__ballot(l));
    }
    if ((t & 63) == 0) s_cnt[wave] = nleft;
    __syncthreads();
    if (t == 0) {
        const int tot = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
        s_base[0] = atomicAdd(&st[C.node].cursor[0], tot);
        s_base[1] = atomicAdd(&st[C.node].cursor[1], n - tot);
    }
    __syncthreads();
    // wave w's share of the two runs
    int lb = s_base[0], rb = s_base[1];
    for (int w = 0; w < wave; ++w) {
        lb += s_cnt[w];
        int mine = 0;  // points of wave w in this chunk
        for (int r = 0; r < kChunk / 256; ++r) mine += max(0, min(64, n - (r * 256 + w * 64)));
        rb += mine - s_cnt[w];
    }
    const unsigned long long below = (1ull << (t & 63)) - 1ull;
    for (int r = 0; r < kChunk / 256; ++r) {
        const int j = r * 256 + t;
        const bool in = j < n, l = (left >> r) & 1u;
        const unsigned long long ml = __ballot(in && l), mr = __ballot(in && !l);
        if (in) {
            const int i = C.lo + j;
            const int o = l ? lb + __popcll(ml & below) : rb + __popcll(mr & below);
            dst.v[0][o] = src.v[0][i];
            dst.v[1][o] = src.v[1][i];
            dst.v[2][o] = src.v[2][i];
            dst.idx[o] = src.idx[i];
        }
        lb += __popcll(ml);
        rb += __popcll(mr);
    }
}

// All cuts of a node of at most kNodeMax points: 16 waves share the node's
// current segments; each segment is sorted along its widest extent (bitonic
// network whose comparators all put the smaller element first, so positions
// past the segment's end act as the largest elements and are never touched),
// which makes the cut at any rank a cut of the run.
__global__ __launch_bounds__(1024) void k_part_leaf(const LeafNode* __restrict__ nodes, PartBuf b0, PartBuf b1,
                                                    int* __restrict__ order) {
    extern __shared__ double s_leaf[];  // x, y, z [kNodeMax] | index [kNodeMax] | positions [kNodeMax]
    int* s_idx = reinterpret_cast<int*>(s_leaf + 3 * kNodeMax);
    unsigned short* s_ord = reinterpret_cast<unsigned short*>(s_idx + kNodeMax);
    __shared__ int s_lo[33], s_dim[32];
    __shared__ unsigned long long s_box[16][6];
    const LeafNode L = nodes[blockIdx.x];
    const PartBuf src = L.buf ? b1 : b0;
    const int n = L.hi - L.lo;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    for (int i = t; i < n; i += 1024) {
        for (int d = 0; d < 3; ++d) s_leaf[d * kNodeMax + i] = src.v[d][L.lo + i];
        s_idx[i] = src.idx[L.lo + i];
        s_ord[i] = (unsigned short)i;
    }
    int nseg = 1;
    if (t == 0) {
        s_lo[0] = 0;
        s_lo[1] = n;
    }
    __syncthreads();
    for (int level = 0; level < 5; ++level) {
        // segments at this level: nseg = 2^level ranges (a range of at most 128 points is done)
        int longest = 0;
        for (int q = 0; q < nseg; ++q) longest = max(longest, s_lo[q + 1] - s_lo[q]);
        if (longest <= kBlockPts) break;  // uniform
        const int wps = 16 / nseg;  // waves per segment
        const int seg = wave / wps, sw = wave - seg * wps;
        const int lo = s_lo[seg], len = s_lo[seg + 1] - lo;
        const bool cut = len > kBlockPts;
        // widest extent of the segment
        for (int d = 0; d < 3; ++d) {
            unsigned long long mn = ~0ull, mx = 0ull;
            for (int i = sw * 64 + lane; i < len; i += wps * 64) {
                const unsigned long long k = key_of(s_leaf[d * kNodeMax + s_ord[lo + i]]);
                mn = k < mn ? k : mn;
                mx = k > mx ? k : mx;
            }
            for (int off = 32; off > 0; off >>= 1) {
                const unsigned long long a = __shfl_xor(mn, off), c = __shfl_xor(mx, off);
                mn = a < mn ? a : mn;
                mx = c > mx ? c : mx;
            }
            if (lane == 0) {
                s_box[wave][d] = mn;
                s_box[wave][3 + d] = mx;
            }
        }
        __syncthreads();
        if (sw == 0 && lane == 0) {
            double mn[3], mx[3];
            for (int d = 0; d < 3; ++d) {
                unsigned long long a = s_box[wave][d], c = s_box[wave][3 + d];
                for (int w = 1; w < wps; ++w) {
                    a = min(a, s_box[wave + w][d]);
                    c = max(c, s_box[wave + w][3 + d]);
                }
                mn[d] = of_key(a);
                mx[d] = of_key(c);
            }
            s_dim[seg] = widest(mn, mx);
        }
        __syncthreads();
        const double* v = s_leaf + s_dim[seg] * kNodeMax;
        int top = 1;
        while (top < longest) top <<= 1;
        for (int k = 2; k <= top; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                if (cut)
                    for (int c = sw * 64 + lane; c < (top >> 1); c += wps * 64) {
                        // comparator c of this stage: the first stage of a merge mirrors within runs of k
                        const int base = (c / j) * (2 * j), q = c % j;
                        const int a = base + q, e = (j == (k >> 1)) ? base + 2 * j - 1 - q : a + j;
                        if (e < len) {
                            const int pa = s_ord[lo + a], pe = s_ord[lo + e];
                            const double va = v[pa], ve = v[pe];
                            if (ve < va || (ve == va && s_idx[pe] < s_idx[pa])) {
                                s_ord[lo + a] = (unsigned short)pe;
                                s_ord[lo + e] = (unsigned short)pa;
                            }
                        }
                    }
                __syncthreads();
            }
        // cut every segment; a done segment is followed by an empty one
        int nl = 0, nh = 0;
        if (t < nseg) {
            const int l0 = s_lo[t], l1 = s_lo[t + 1], m = l1 - l0;
            nl = l0;
            nh = m > kBlockPts ? l0 + ((m + kBlockPts - 1) / kBlockPts / 2) * kBlockPts : l1;
        }
        __syncthreads();
        if (t < nseg) {
            s_lo[2 * t] = nl;
            s_lo[2 * t + 1] = nh;
        }
        if (t == 0) s_lo[2 * nseg] = n;
        nseg *= 2;
        __syncthreads();
    }
    for (int i = t; i < n; i += 1024) order[L.lo + i] = s_idx[s_ord[i]];
}

// Raw points of a generated grid, one workgroup per radial shell: the rotated
// directions of its rule times its radius, around its atom.  Plain products
// and sums, as a host compiler forms them.
__global__ __launch_bounds__(256) void k_raw_points(const RawShell* __restrict__ shells, const double* __restrict__ dirs,
                                                    double* __restrict__ pts, double* __restrict__ w,
                                                    int* __restrict__ atom) {
#pragma clang fp contract(off)
    const RawShell S = shells[blockIdx.x];
    for (int k = threadIdx.x; k < S.n; k += 256) {
        const double* d = dirs + 4 * (int64_t)(S.dir_begin + k);
        const int64_t i = S.first + k;
        for (int q = 0; q < 3; ++q) pts[3 * i + q] = d[q] * S.r + S.center[q];
        w[i] = d[3] * S.w;
        atom[i] = S.atom;
    }
}

// Points of every shell whose weight passes the screen.
__global__ __launch_bounds__(256) void k_keep_count(const RawShell* __restrict__ shells, const double* __restrict__ w,
                                                    double cutoff, long long* __restrict__ counts) {
    __shared__ int s_n[4];
    const RawShell S = shells[blockIdx.x];
    int n = 0;
    for (int k = threadIdx.x; k < S.n; k += 256) n += fabs(w[S.first + k]) > cutoff;
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off);
    if ((threadIdx.x & 63) == 0) s_n[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}

// v[0 .. n] to its exclusive prefix sums, v[n] the total (one workgroup)
__global__ __launch_bounds__(1024) void k_scan(int n, long long* __restrict__ v) {
    __shared__ long long s_part[1024];
    const int t = threadIdx.x, per = (n + 1023) / 1024;
    const int b = min(n, t * per), e = min(n, b + per);
    long long sum = 0;
    for (int i = b; i < e; ++i) sum += v[i];
    s_part[t] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const long long a = t >= off ? s_part[t - off] : 0;
        __syncthreads();
        s_part[t] += a;
        __syncthreads();
    }
    long long run = s_part[t] - sum;
    for (int i = b; i < e; ++i) {
        const long long c = v[i];
        v[i] = run;
        run += c;
    }
    if (t == 1023) v[n] = s_part[t];
}

// The kept points in their order, as grid columns (n of them).
__global__ __launch_bounds__(256) void k_keep_write(const RawShell* __restrict__ shells, const double* __restrict__ pts,
                                                    const double* __restrict__ w, double cutoff,
                                                    const long long* __restrict__ first, int64_t n,
                                                    double* __restrict__ grid) {
    __shared__ int s_n[4];
    const RawShell S = shells[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t at = first[blockIdx.x];
    for (int k0 = 0; k0 < S.n; k0 += 256) {
        const int k = k0 + threadIdx.x;
        const int64_t i = S.first + k;
        const double wi = k < S.n ? w[i] : 0.0;
        const bool keep = k < S.n && fabs(wi) > cutoff;
        const unsigned long long m = __ballot(keep);
        if (lane == 0) s_n[wave] = __popcll(m);
        __syncthreads();
        int64_t to = at + __popcll(m & ((1ull << lane) - 1ull));
        for (int q = 0; q < 4; ++q) {
            if (q < wave) to += s_n[q];
            at += s_n[q];
        }
        if (keep) {
            for (int q = 0; q < 3; ++q) grid[q * n + to] = pts[3 * i + q];
            grid[3 * n + to] = wi;
        }
        __syncthreads();
    }
}

// points [first, first + n) of the grid columns (stride apart) to rows (x, y, z, w)
__global__ __launch_bounds__(256) void k_grid_rows(int64_t first, int64_t n, int64_t stride,
                                                   const double* __restrict__ grid, double* __restrict__ rows) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < 4 * n) rows[t] = grid[(t & 3) * stride + first + (t >> 2)];
}

// First point with a value that is not finite (n when there is none).
__global__ __launch_bounds__(256) void k_check_finite(int64_t n, const double* __restrict__ grid,
                                                      unsigned long long* __restrict__ first) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    bool bad = false;
    for (int q = 0; q < 4; ++q) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(grid[q * n + i]);
        bad = bad || ((b >> 52) & 0x7ff) == 0x7ff;
    }
    if (bad) atomicMin(first, (unsigned long long)i);
}

// Shells a block keeps (one wave per block): a shell survives when the nearest
// point of the block's bounding box lies within its cut-off distances (the
// reference's alpha r^2 <= 30 of its most diffuse primitive, and the ao_screen
// bound).  Plain products and sums, as a host compiler forms them: a block's
// list does not hang on the contraction of d^2.
__global__ __launch_bounds__(256) void k_screen_blocks(int nb, int64_t n, const double* __restrict__ grid,
                                                       const int* __restrict__ order, int nsh,
                                                       const ScreenShell* __restrict__ shells, int nw,
                                                       unsigned long long* __restrict__ masks,
                                                       int* __restrict__ counts) {
#pragma clang fp contract(off)
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b >= nb) return;
    const int lo = b * kBlockPts, hi = (int)min((int64_t)lo + kBlockPts, n);
    double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
    for (int i = lo + lane; i < hi; i += 64) {
        const int p = order[i];
        for (int d = 0; d < 3; ++d) {
            const double v = grid[d * n + p];
            mn[d] = fmin(mn[d], v);
            mx[d] = fmax(mx[d], v);
        }
    }
    for (int off = 32; off > 0; off >>= 1)
        for (int d = 0; d < 3; ++d) {
            mn[d] = fmin(mn[d], __shfl_xor(mn[d], off));
            mx[d] = fmax(mx[d], __shfl_xor(mx[d], off));
        }
    int nshell = 0, nao = 0;
    for (int w = 0; w < nw; ++w) {
        const int s = w * 64 + lane;
        bool keep = false;
        int l = 0;
        if (s < nsh) {
            const ScreenShell S = shells[s];
            double d2 = 0.0;
            for (int d = 0; d < 3; ++d) {
                const double e = fmax(0.0, fmax(mn[d] - S.center[d], S.center[d] - mx[d]));
                d2 = d2 + e * e;
            }
            // distance to the box, shrunk by a relative 1e-12 for rounding
            const double dmin = sqrt(d2) * (1.0 - 1e-12);
            keep = !(S.exp0 * dmin * dmin > 30.0) && dmin <= S.cut;
            l = S.l;
        }
        const unsigned long long m = __ballot(keep);
        nshell += __popcll(m);
        nao += __popcll(m) + 2 * __popcll(__ballot(keep && l == 1)) + 4 * __popcll(__ballot(keep && l == 2));
        if (lane == 0) masks[(int64_t)b * nw + w] = m;
    }
    if (lane == 0) {
        counts[2 * b] = nshell;
        counts[2 * b + 1] = nao;
    }
}

// Lists of one shell mask (by one wave): kept shells in ascending order with
// their columns, and their order by (l, nprim) class.
__device__ __forceinline__ void fill_lists(const unsigned long long* mask, int shell_begin, int col_begin, int nw, int ncls,
                                           const ScreenShell* __restrict__ shells, int* __restrict__ bshells,
                                           int* __restrict__ bshell_col, int* __restrict__ bcols,
                                           int* __restrict__ bsorder) {
    const int lane = threadIdx.x & 63;
    const unsigned long long below = (1ull << lane) - 1ull;
    int pos0 = 0, col0 = 0;
    for (int w = 0; w < nw; ++w) {
        const unsigned long long m = mask[w];
        const bool keep = (m >> lane) & 1ull;
        const int s = w * 64 + lane;
        int l = 0, first = 0;
        if (keep) {
            l = shells[s].l;
            first = shells[s].first_ao;
        }
        const unsigned long long m1 = __ballot(keep && l == 1), m2 = __ballot(keep && l == 2);
        if (keep) {
            const int pos = pos0 + __popcll(m & below);
            const int col = col0 + __popcll(m & below) + 2 * __popcll(m1 & below) + 4 * __popcll(m2 & below);
            bshells[shell_begin + pos] = s;
            bshell_col[shell_begin + pos] = col;
            for (int q = 0; q < 2 * l + 1; ++q) bcols[col_begin + col + q] = first + q;
        }
        pos0 += __popcll(m);
        col0 += __popcll(m) + 2 * __popcll(m1) + 4 * __popcll(m2);
    }
    int out = 0;
    for (int c = 0; c < ncls; ++c) {
        pos0 = 0;
        for (int w = 0; w < nw; ++w) {
            const unsigned long long m = mask[w];
            const bool keep = ((m >> lane) & 1ull) && shells[w * 64 + lane].cls == c;
            const unsigned long long mc = __ballot(keep);
            if (keep) bsorder[shell_begin + out + __popcll(mc & below)] = pos0 + __popcll(m & below);
            out += __popcll(mc);
            pos0 += __popcll(m);
        }
    }
}

// The lists and slots of every block (one wave per block, in launch order; a
// partial block repeats its last point with weight 0).
__global__ __launch_bounds__(256) void k_fill_blocks(int nb, int64_t n, int64_t n_slots, const double* __restrict__ grid,
                                                     const int* __restrict__ order, const int* __restrict__ leaf,
                                                     const BlockDesc* __restrict__ blocks, int nw, int ncls,
                                                     const ScreenShell* __restrict__ shells,
                                                     const unsigned long long* __restrict__ masks,
                                                     int* __restrict__ bshells, int* __restrict__ bshell_col,
                                                     int* __restrict__ bcols, int* __restrict__ bsorder,
                                                     double* __restrict__ pts, int* __restrict__ slot_of_point) {
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b >= nb) return;
    const BlockDesc B = blocks[b];
    const int lf = leaf[b];
    fill_lists(masks + (int64_t)lf * nw, B.shell_begin, B.col_begin, nw, ncls, shells, bshells, bshell_col, bcols,
               bsorder);
    for (int k = lane; k < kBlockPts; k += 64) {
        const int p = order[lf * kBlockPts + min(k, B.npts - 1)];
        const int64_t slot = (int64_t)b * kBlockPts + k;
        pts[slot] = grid[p];
        pts[n_slots + slot] = grid[n + p];
        pts[2 * n_slots + slot] = grid[2 * n + p];
        pts[3 * n_slots + slot] = k < B.npts ? grid[3 * n + p] : 0.0;
        if (k < B.npts) slot_of_point[p] = (int)slot;
    }
}

// Shells of `per` neighbouring leaves together (one wave per group): the union
// of their masks and its shell and AO counts.
__global__ __launch_bounds__(256) void k_group_masks(int nb, int per, int nsh, const ScreenShell* __restrict__ shells,
                                                     int nw, const unsigned long long* __restrict__ masks,
                                                     unsigned long long* __restrict__ gmasks, int* __restrict__ counts) {
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l0 = g * per, l1 = min(nb, l0 + per);
    if (l0 >= nb) return;
    int nshell = 0, nao = 0;
    for (int w = 0; w < nw; ++w) {
        unsigned long long m = 0;
        for (int lf = l0; lf < l1; ++lf) m |= masks[(int64_t)lf * nw + w];
        const int s = w * 64 + lane;
        const bool keep = s < nsh && ((m >> lane) & 1ull);
        const int l = keep ? shells[s].l : 0;
        nshell += __popcll(m);
        nao += __popcll(m) + 2 * __popcll(__ballot(keep && l == 1)) + 4 * __popcll(__ballot(keep && l == 2));
        if (lane == 0) gmasks[(int64_t)g * nw + w] = m;
    }
    if (lane == 0) {
        counts[2 * g] = nshell;
        counts[2 * g + 1] = nao;
    }
}

// The lists of the K units that hold several blocks: group[u] >= 0 is the mask
// of unit u (one wave per unit; the others have the lists of their block).
__global__ __launch_bounds__(256) void k_fill_groups(int n, const int* __restrict__ group,
                                                     const KBlock* __restrict__ units, int nw, int ncls,
                                                     const ScreenShell* __restrict__ shells,
                                                     const unsigned long long* __restrict__ gmasks,
                                                     int* __restrict__ bshells, int* __restrict__ bshell_col,
                                                     int* __restrict__ bcols, int* __restrict__ bsorder) {
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= n || group[u] < 0) return;
    fill_lists(gmasks + (int64_t)group[u] * nw, units[u].shell_begin, units[u].col_begin, nw, ncls, shells, bshells,
               bshell_col, bcols, bsorder);
}

// shells of each K item: those whose first column lies below the item's columns
__global__ __launch_bounds__(256) void k_item_shells(int n, const KWork* __restrict__ work,
                                                     const KBlock* __restrict__ units,
                                                     const int* __restrict__ bshell_col, int* __restrict__ nsh) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const KBlock& B = units[work[i].block];
    int lo = 0, hi = B.nshell;
    while (lo < hi) {
        const int m = (lo + hi) / 2;
        if (bshell_col[B.shell_begin + m] < work[i].ncols) lo = m + 1;
        else hi = m;
    }
    nsh[i] = lo;
}

// per-point data (w doubles each) between the caller's order and the slots
__global__ __launch_bounds__(256) void k_gather_points(int64_t n, const int* __restrict__ slot_of_point,
                                                       const double* __restrict__ src, double* __restrict__ dst,
                                                       int stride, int off) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 4 * n) return;
    const int64_t p = t >> 2;
    const int q = (int)(t & 3);
    dst[stride * p + off + q] = src[4 * (int64_t)slot_of_point[p] + q];
}
// rho alone, or rho and the rows of its gradient: dst = rho [n] | grad [n][3]
__global__ __launch_bounds__(256) void k_gather_density(int64_t n, const int* __restrict__ slot_of_point,
                                                        const double* __restrict__ src, double* __restrict__ dst,
                                                        int grad) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    const double* r = src + 4 * (int64_t)slot_of_point[p];
    dst[p] = r[0];
    if (grad)
        for (int d = 0; d < 3; ++d) dst[n + 3 * p + d] = r[1 + d];
}
__global__ __launch_bounds__(256) void k_scatter_points(int64_t n, const int* __restrict__ slot_of_point,
                                                        const double* __restrict__ src, double* __restrict__ dst) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 4 * n) return;
    dst[4 * (int64_t)slot_of_point[t >> 2] + (t & 3)] = src[t];
}
__global__ __launch_bounds__(256) void k_scatter_atoms(int64_t n, const int* __restrict__ slot_of_point,
                                                       const int* __restrict__ atom, int* __restrict__ dst) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p < n) dst[slot_of_point[p]] = atom[p];
}
// points (x, y, z rows) to the columns of a grid of unit weights
__global__ __launch_bounds__(256) void k_points_to_grid(int64_t n, const double* __restrict__ xyz,
                                                        double* __restrict__ grid) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 4 * n) return;
    const int64_t q = t / n, p = t - q * n;
    grid[t] = q < 3 ? xyz[3 * p + q] : 1.0;
}

int check(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, what);
    return PDFXC_OK;
}
unsigned blocks256(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

int device_partition(int64_t n64, const double* d_grid, int* d_order, hipStream_t s, DevicePool& pool) {
    const int n = (int)n64;
    const PartTree tree = part_tree(n);
    const auto& [nodes, chunks, node_off, chunk_off, leaves, most] = tree;
    const int levels = (int)node_off.size() - 1;
    // one workspace: two point buffers | states | histograms | tables
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t b_v = up(sizeof(double) * (size_t)n), b_i = up(sizeof(int) * (size_t)n);
    const size_t b_st = up(sizeof(PartState) * most), b_h = up(sizeof(unsigned int) * most * kPasses * 256);
    const size_t b_n = up(sizeof(PartNode) * nodes.size()), b_c = up(sizeof(PartChunk) * chunks.size());
    const size_t b_l = up(sizeof(LeafNode) * leaves.size());
    const int nbuf = levels > 0 ? 2 : 1;
    void* taken = nullptr;
    const size_t total = nbuf * (3 * b_v + b_i) + b_st + b_h + b_n + b_c + b_l;
    hipError_t e = pool.take(&taken, total);
    char* ws = static_cast<char*>(taken);
    if (e != hipSuccess) {
        set_error("block partition: hipMalloc of " + std::to_string(total) + " bytes: " + hipGetErrorString(e));
        return PDFXC_ERR_MEMORY;
    }
    PartBuf buf[2];
    char* q = ws;
    for (int k = 0; k < 2; ++k) {
        if (k == 1 && nbuf == 1) {
            buf[1] = buf[0];
            break;
        }
        for (int d = 0; d < 3; ++d, q += b_v) buf[k].v[d] = reinterpret_cast<double*>(q);
        buf[k].idx = reinterpret_cast<int*>(q);
        q += b_i;
    }
    PartState* st = reinterpret_cast<PartState*>(q);
    unsigned int* hist = reinterpret_cast<unsigned int*>(q + b_st);
    PartNode* d_nodes = reinterpret_cast<PartNode*>(q + b_st + b_h);
    PartChunk* d_chunks = reinterpret_cast<PartChunk*>(q + b_st + b_h + b_n);
    LeafNode* d_leaves = reinterpret_cast<LeafNode*>(q + b_st + b_h + b_n + b_c);
    auto copy = [&](void* d, const void* h, size_t bytes) {
        if (e == hipSuccess && bytes) e = hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s);
    };
    copy(d_nodes, nodes.data(), sizeof(PartNode) * nodes.size());
    copy(d_chunks, chunks.data(), sizeof(PartChunk) * chunks.size());
    copy(d_leaves, leaves.data(), sizeof(LeafNode) * leaves.size());
    int rc = e == hipSuccess ? PDFXC_OK : hip_fail(e, "block partition: tables");
    if (rc == PDFXC_OK) {
        hipLaunchKernelGGL(k_part_start, dim3(blocks256(n)), dim3(256), 0, s, (int64_t)n, d_grid, buf[0]);
        for (int L = 0; L < levels; ++L) {
            const PartNode* nd = d_nodes + node_off[L];
            const PartChunk* ch = d_chunks + chunk_off[L];
            const dim3 gn((unsigned)(node_off[L + 1] - node_off[L])), gc((unsigned)(chunk_off[L + 1] - chunk_off[L]));
            hipLaunchKernelGGL(k_part_init, gn, dim3(256), 0, s, nd, st, hist);
            hipLaunchKernelGGL(k_part_box, gc, dim3(256), 0, s, ch, buf[L & 1], st);
            for (int p = 0; p < kPasses; ++p)
                hipLaunchKernelGGL(k_part_hist, gc, dim3(256), 0, s, p, ch, nd, buf[L & 1], st, hist);
            hipLaunchKernelGGL(k_part_split, gc, dim3(256), 0, s, ch, buf[L & 1], buf[(L + 1) & 1], st, hist);
        }
        const size_t lds = (3 * sizeof(double) + sizeof(int) + sizeof(unsigned short)) * kNodeMax;
        hipLaunchKernelGGL(k_part_leaf, dim3((unsigned)leaves.size()), dim3(1024), lds, s, d_leaves, buf[0], buf[1],
                           d_order);
        rc = check("block partition");
    }
    e = hipStreamSynchronize(s);  // the workspace and the host tables end here
    pool.give(ws);
    if (rc == PDFXC_OK && e != hipSuccess) rc = hip_fail(e, "block partition");
    return rc;
}

int launch_raw_points(int ns, const RawShell* d_shells, const double* d_dirs, double* d_pts, double* d_w, int* d_atom,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_raw_points, dim3(ns), dim3(256), 0, s, d_shells, d_dirs, d_pts, d_w, d_atom);
    return check("k_raw_points");
}

int launch_keep_count(int ns, const RawShell* d_shells, const double* d_w, double cutoff, long long* d_first,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_keep_count, dim3(ns), dim3(256), 0, s, d_shells, d_w, cutoff, d_first);
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, ns, d_first);
    return check("k_keep_count");
}

int launch_keep_write(int ns, const RawShell* d_shells, const double* d_pts, const double* d_w, double cutoff,
                      const long long* d_first, int64_t n, double* d_grid, hipStream_t s) {
    hipLaunchKernelGGL(k_keep_write, dim3(ns), dim3(256), 0, s, d_shells, d_pts, d_w, cutoff, d_first, n, d_grid);
    return check("k_keep_write");
}

int launch_grid_rows(int64_t first, int64_t n, int64_t stride, const double* d_grid, double* d_rows, hipStream_t s) {
    hipLaunchKernelGGL(k_grid_rows, dim3(blocks256(4 * n)), dim3(256), 0, s, first, n, stride, d_grid, d_rows);
    return check("k_grid_rows");
}

int device_check_finite(int64_t n, const double* d_grid, unsigned long long* d_first, hipStream_t s) {
    hipLaunchKernelGGL(k_check_finite, dim3(blocks256(n)), dim3(256), 0, s, n, d_grid, d_first);
    return check("k_check_finite");
}

int launch_screen_blocks(int nb, int64_t n, const double* d_grid, const int* d_order, int nsh,
                         const ScreenShell* d_shells, int nw, unsigned long long* d_masks, int* d_counts,
                         hipStream_t s) {
    hipLaunchKernelGGL(k_screen_blocks, dim3((nb + 3) / 4), dim3(256), 0, s, nb, n, d_grid, d_order, nsh, d_shells, nw,
                       d_masks, d_counts);
    return check("k_screen_blocks");
}

int launch_fill_blocks(Context& c, const int* d_order, const int* d_leaf, int nw, int ncls,
                       const ScreenShell* d_shells, const unsigned long long* d_masks) {
    const int nb = (int)c.blocks.size();
    hipLaunchKernelGGL(k_fill_blocks, dim3((nb + 3) / 4), dim3(256), 0, c.stream, nb, c.n_pts, c.n_slots, c.d_grid,
                       d_order, d_leaf, c.d_blocks, nw, ncls, d_shells, d_masks, c.d_block_shells, c.d_block_shell_col,
                       c.d_block_cols, c.d_block_sorder, c.d_pts, c.d_slot_of_point);
    return check("k_fill_blocks");
}

int launch_group_masks(int nb, int per, int nsh, const ScreenShell* d_shells, int nw,
                       const unsigned long long* d_masks, unsigned long long* d_gmasks, int* d_gcounts, hipStream_t s) {
    const int ng = (nb + per - 1) / per;
    hipLaunchKernelGGL(k_group_masks, dim3((ng + 3) / 4), dim3(256), 0, s, nb, per, nsh, d_shells, nw, d_masks, d_gmasks,
                       d_gcounts);
    return check("k_group_masks");
}

int launch_fill_groups(Context& c, int n, const int* d_group, int nw, int ncls, const ScreenShell* d_shells,
                       const unsigned long long* d_gmasks) {
    hipLaunchKernelGGL(k_fill_groups, dim3((n + 3) / 4), dim3(256), 0, c.stream, n, d_group, c.d_kblocks, nw, ncls,
                       d_shells, d_gmasks, c.d_block_shells, c.d_block_shell_col, c.d_block_cols, c.d_block_sorder);
    return check("k_fill_groups");
}

int launch_item_shells(Context& c, int n, const KWork* d_work, int* d_nsh) {
    if (n <= 0) return PDFXC_OK;
    hipLaunchKernelGGL(k_item_shells, dim3(blocks256(n)), dim3(256), 0, c.stream, n, d_work, c.d_kblocks,
                       c.d_block_shell_col, d_nsh);
    return check("k_item_shells");
}

int launch_gather_points(Context& c, int64_t first, int64_t n, const double* d_slots, double* d_pts, int stride, int off) {
    hipLaunchKernelGGL(k_gather_points, dim3(blocks256(4 * n)), dim3(256), 0, c.stream, n, c.d_slot_of_point + first,
                       d_slots, d_pts, stride, off);
    return check("k_gather_points");
}

int launch_gather_density(Context& c, const double* d_slots, double* d_out, bool grad) {
    hipLaunchKernelGGL(k_gather_density, dim3(blocks256(c.n_pts)), dim3(256), 0, c.stream, c.n_pts, c.d_slot_of_point,
                       d_slots, d_out, grad ? 1 : 0);
    return check("k_gather_density");
}

int launch_scatter_points(Context& c, int64_t first, int64_t n, const double* d_pts, double* d_slots) {
    hipLaunchKernelGGL(k_scatter_points, dim3(blocks256(4 * n)), dim3(256), 0, c.stream, n, c.d_slot_of_point + first,
                       d_pts, d_slots);
    return check("k_scatter_points");
}

int launch_scatter_atoms(Context& c, const int* d_atom, int* d_slot_atom) {
    hipLaunchKernelGGL(k_scatter_atoms, dim3(blocks256(c.n_pts)), dim3(256), 0, c.stream, c.n_pts, c.d_slot_of_point, d_atom,
                       d_slot_atom);
    return check("k_scatter_atoms");
}

int launch_points_to_grid(int64_t n, const double* d_xyz, double* d_grid, hipStream_t s) {
    hipLaunchKernelGGL(k_points_to_grid, dim3(blocks256(4 * n)), dim3(256), 0, s, n, d_xyz, d_grid);
    return check("k_points_to_grid");
}

}  // namespace pdfxc
