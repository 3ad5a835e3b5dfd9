// Checks of the engine's host code against the stand-in HIP runtime, one per
// argument; exit status 0 when it holds.
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "pdfxc_internal.hpp"
#include "pdfxc_partition.hpp"

extern "C" {
size_t fake_live_bytes();
void fake_limit(size_t bytes);
void fake_fail_copy(int after);
void fake_slow_copy(int ms);
long long fake_misplaced();
}

namespace {

using namespace pdfxc;

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            std::printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #x); \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

pdfxc_ctx* context(int n_aos = 1) {
    const std::vector<double> centre(3 * (size_t)n_aos, 0.0), ones((size_t)n_aos, 1.0);
    const std::vector<int> type((size_t)n_aos, 0), nprim((size_t)n_aos, 1);
    pdfxc_opts o;
    pdfxc_default_opts(&o);
    pdfxc_ctx* ctx = nullptr;
    CHECK(pdfxc_ctx_create(&ctx, n_aos, centre.data(), type.data(), nprim.data(), ones.data(), ones.data(), 1, &o) ==
          PDFXC_OK);
    return ctx;
}

std::vector<double> column(int64_t n, double first) {
    std::vector<double> v((size_t)n);
    for (int64_t i = 0; i < n; ++i) v[i] = first + 1e-3 * i;
    return v;
}

void set_grid(pdfxc_ctx* ctx, int64_t n) {
    const std::vector<double> x = column(n, 1.0), y = column(n, 2.0), z = column(n, 3.0), w = column(n, 4.0);
    CHECK(pdfxc_set_grid(ctx, n, x.data(), y.data(), z.data(), w.data()) == PDFXC_OK);
}

bool host_grid_is_right(const Context& c) {
    return c.gx == column(c.n_pts, 1.0) && c.gy == column(c.n_pts, 2.0) && c.gz == column(c.n_pts, 3.0) &&
           c.gw == column(c.n_pts, 4.0);
}

// no buffer is given to two threads at once
void pool_threads() {
    DevicePool pool;
    bool ok[4] = {true, true, true, true};
    std::vector<std::thread> threads;
    for (int k = 0; k < 4; ++k)
        threads.emplace_back([&, k] {
            for (int i = 0; i < 20000; ++i) {
                int* p[3] = {};
                for (int q = 0; q < 3; ++q) {
                    void* v = nullptr;
                    if (pool.take(&v, 4096 << ((i + q) % 4)) != hipSuccess) ok[k] = false;
                    p[q] = static_cast<int*>(v);
                    *p[q] = 4 * i + k;
                }
                for (int* v : p) {
                    ok[k] = ok[k] && *v == 4 * i + k;
                    pool.give(v);
                }
            }
        });
    for (auto& t : threads) t.join();
    for (bool b : ok) CHECK(b);
}

// two threads that need a context's host copies both return with whole ones
void host_copy_threads() {
    pdfxc_ctx* ctx = context();
    Context& c = *reinterpret_cast<Context*>(ctx);
    set_grid(ctx, 70000);
    fake_slow_copy(50);
    bool ok[2] = {};
    auto work = [&](int k) { ok[k] = ensure_host_grid(c) == PDFXC_OK && host_grid_is_right(c); };
    std::thread first(work, 0);
    std::this_thread::sleep_for(std::chrono::milliseconds(175));  // into the last of four copies
    std::thread second(work, 1);
    first.join();
    second.join();
    CHECK(ok[0] && ok[1]);
    fake_slow_copy(0);
    pdfxc_ctx_destroy(ctx);
}

// the grid's rows need no device memory that is not there, and no current device
void grid_rows() {
    pdfxc_ctx* ctx = context();
    const int64_t n = 70000;
    set_grid(ctx, n);
    int device = -1;
    CHECK(hipSetDevice(1) == hipSuccess);
    std::vector<double> rows(4 * n);
    CHECK(pdfxc_get_grid_rows(ctx, rows.data()) == PDFXC_OK);
    CHECK(fake_misplaced() == 0);
    CHECK(hipGetDevice(&device) == hipSuccess && device == 1);
    CHECK(hipSetDevice(0) == hipSuccess);
    reinterpret_cast<Context*>(ctx)->pool.trim(0);
    fake_limit(fake_live_bytes());
    CHECK(pdfxc_get_grid_rows(ctx, rows.data()) == PDFXC_OK);
    const Context& c = *reinterpret_cast<Context*>(ctx);
    CHECK(ensure_host_grid(*reinterpret_cast<Context*>(ctx)) == PDFXC_OK && host_grid_is_right(c));
    for (int64_t i = 0; i < n; ++i)
        CHECK(rows[4 * i] == c.gx[i] && rows[4 * i + 1] == c.gy[i] && rows[4 * i + 2] == c.gz[i] &&
              rows[4 * i + 3] == c.gw[i]);
    fake_limit(~(size_t)0);
    pdfxc_ctx_destroy(ctx);
}

// what a pool holds beyond the buffers in use stays bounded at every moment,
// and a buffer is not given for a quarter of its size
void pool_bound() {
    const size_t mib = (size_t)1 << 20;
    DevicePool pool;
    std::vector<void*> p(6);
    size_t used = 0;
    for (void*& v : p) CHECK(pool.take(&v, 200 * mib) == hipSuccess);
    used = fake_live_bytes();
    const size_t each = used / p.size();
    for (void* v : p) {
        pool.give(v);
        used -= each;
        CHECK(fake_live_bytes() <= used + kPoolKeep);
    }
    const size_t before = fake_live_bytes();
    void* v = nullptr;
    CHECK(pool.take(&v, 120 * mib) == hipSuccess);
    CHECK(fake_live_bytes() > before);  // not one of 200 MiB
    pool.give(v);
    CHECK(fake_live_bytes() <= kPoolKeep);
}

// buffers in reserve give way to every allocation of the context: the second
// spin's, rho in the caller's order, a batch's, a file's, a density's
void reserve_gives_way() {
    pdfxc_ctx* ctx = context();
    Context& c = *reinterpret_cast<Context*>(ctx);
    const int64_t n = 100000;
    double P = 1.0, K = 0.0, E = 0.0, x[3] = {0.0, 0.0, 0.0}, rho = 0.0;
    std::vector<double> out(8 * n);
    auto full = [&](size_t reserve) {  // nothing free but `reserve` bytes kept by the pool
        void* v = nullptr;
        fake_limit(~(size_t)0);
        c.pool.trim(0);
        CHECK(c.pool.take(&v, reserve) == hipSuccess);
        c.pool.give(v);
        fake_limit(fake_live_bytes());
    };
    set_grid(ctx, n);
    full(2 * 4 * sizeof(double) * (n + kBlockPts) + 4096);
    CHECK(pdfxc_build_uks(ctx, PDFXC_SVWN, &P, &P, &K, &K, &E, nullptr) == PDFXC_OK);
    full(8 * sizeof(double) * n);
    CHECK(pdfxc_build_uks(ctx, PDFXC_SVWN, &P, &P, &K, &K, &E, out.data()) == PDFXC_OK);
    full(4 * sizeof(double) * n);
    CHECK(pdfxc_save_grid_matrix(ctx, "/dev/null", 4) == PDFXC_OK);
    std::vector<double> phi(n);
    full(sizeof(double) * 7 * n);
    CHECK(pdfxc_eval_aos(ctx, n, out.data(), phi.data(), nullptr, nullptr, nullptr) == PDFXC_OK);
    full((size_t)64 << 20);
    pdfxc_batch* batch = nullptr;
    CHECK(pdfxc_batch_create(&batch, 1, &ctx) == PDFXC_OK);
    pdfxc_batch_destroy(batch);
    full((size_t)8 << 20);
    CHECK(pdfxc_density_at_points(ctx, &P, 1, x, &rho, nullptr) == PDFXC_OK);
    // the kept context of the densities gives way too
    fake_limit(~(size_t)0);
    CHECK(pdfxc_density_at_points(ctx, &P, n, out.data(), phi.data(), nullptr) == PDFXC_OK);
    CHECK(c.probe != nullptr);
    c.pool.trim(0);
    fake_limit(fake_live_bytes());
    CHECK(pdfxc_eval_aos(ctx, 1000, out.data(), phi.data(), nullptr, nullptr, nullptr) == PDFXC_OK);
    fake_limit(~(size_t)0);
    pdfxc_ctx_destroy(ctx);
    CHECK(fake_live_bytes() == 0);
}

// rho goes to the host and back without device memory of its own
void rho_without_memory() {
    pdfxc_ctx* ctx = context();
    Context& c = *reinterpret_cast<Context*>(ctx);
    const int64_t n = 70000;
    double P = 1.0, K = 0.0, E = 0.0;
    std::vector<double> out(8 * n), mat(13 * n);
    set_grid(ctx, n);
    CHECK(pdfxc_build_uks(ctx, PDFXC_SVWN, &P, &P, &K, &K, &E, nullptr) == PDFXC_OK);
    // point p in slot n - 1 - p; rho of slot s: 8 s + 0 .. 3 and, beta, + 4 .. 7
    std::vector<int> slots((size_t)n);
    for (int64_t i = 0; i < n; ++i) slots[i] = (int)(n - 1 - i);
    CHECK(hipMemcpy(c.d_slot_of_point, slots.data(), n * sizeof(int), hipMemcpyHostToDevice) == hipSuccess);
    for (int64_t s = 0; s < n; ++s)
        for (int q = 0; q < 4; ++q) {
            c.d_rho[4 * s + q] = 8 * s + q;
            c.d_rho_b[4 * s + q] = 8 * s + 4 + q;
        }
    c.pool.trim(0);
    fake_limit(fake_live_bytes());
    CHECK(pdfxc_build_uks(ctx, PDFXC_SVWN, &P, &P, &K, &K, &E, out.data()) == PDFXC_OK);
    for (int64_t i = 0; i < n; ++i)
        for (int q = 0; q < 8; ++q) CHECK(out[8 * i + q] == 8 * (n - 1 - i) + q);
    char path[] = "/tmp/pdfxc_rho_XXXXXX";
    const int fd = mkstemp(path);
    CHECK(fd >= 0);
    close(fd);
    CHECK(pdfxc_save_grid_matrix(ctx, path, 8) == PDFXC_OK);
    CHECK(pdfxc_load_general_matrix(path, n, 13, mat.data()) == PDFXC_OK);
    unlink(path);
    for (int64_t i = 0; i < n; ++i)
        for (int q = 0; q < 8; ++q) CHECK(mat[(5 + q) * n + i] == out[8 * i + q]);
    std::fill(c.d_rho, c.d_rho + 4 * c.n_slots, -1.0);
    std::vector<double> alpha(4 * n);
    for (int64_t i = 0; i < n; ++i)
        for (int q = 0; q < 4; ++q) alpha[4 * i + q] = out[8 * i + q];
    CHECK(rho_from_host(c, alpha.data(), c.d_rho) == PDFXC_OK);
    for (int64_t s = 0; s < c.n_slots; ++s)
        for (int q = 0; q < 4; ++q) CHECK(c.d_rho[4 * s + q] == (s < n ? 8 * s + q : 0.0));
    fake_limit(~(size_t)0);
    pdfxc_ctx_destroy(ctx);
    CHECK(fake_live_bytes() == 0);
}

// a small grid is read from the host alone, and its blocks are those of the cuts'
// definition: every node sorted along its widest extent by (coordinate, index)
void small_grids() {
    unsigned seed = 1;
    for (int64_t n : {(int64_t)1, (int64_t)128, (int64_t)129, (int64_t)300, (int64_t)2049, kHostCut}) {
        pdfxc_ctx* ctx = context();  // its buffers are new: no kernel writes the block counts
        Context& c = *reinterpret_cast<Context*>(ctx);
        std::vector<double> col[4];
        for (auto& v : col)
            for (int64_t i = 0; i < n; ++i) {
                seed = seed * 1664525u + 1013904223u;
                v.push_back((double)((int)(seed >> 24) - 128) * 0.25);  // many equal coordinates
            }
        CHECK(pdfxc_set_grid(ctx, n, col[0].data(), col[1].data(), col[2].data(), col[3].data()) == PDFXC_OK);
        fake_fail_copy(0);
        std::vector<double> rows(4 * n), x((size_t)n);
        CHECK(pdfxc_get_grid_rows(ctx, rows.data()) == PDFXC_OK);
        CHECK(pdfxc_get_grid(ctx, x.data(), nullptr, nullptr, nullptr) == PDFXC_OK && x == col[0]);
        fake_fail_copy(-1);
        for (int64_t i = 0; i < n; ++i)
            for (int q = 0; q < 4; ++q) CHECK(rows[4 * i + q] == col[q][i]);
        std::vector<int> order, want((size_t)n);
        partition_points(c, order);
        for (int64_t i = 0; i < n; ++i) want[i] = (int)i;
        std::vector<std::pair<int, int>> nodes{{0, (int)n}};
        while (!nodes.empty()) {
            const auto [lo, hi] = nodes.back();
            nodes.pop_back();
            if (hi - lo <= kBlockPts) continue;
            int dim = 0;
            double widest = -1.0;
            for (int d = 0; d < 3; ++d) {
                double mn = 1e300, mx = -1e300;
                for (int k = lo; k < hi; ++k) {
                    mn = std::min(mn, col[d][want[k]]);
                    mx = std::max(mx, col[d][want[k]]);
                }
                if (mx - mn > widest) {
                    widest = mx - mn;
                    dim = d;
                }
            }
            std::sort(want.begin() + lo, want.begin() + hi, [&](int p, int q) {
                return col[dim][p] < col[dim][q] || (col[dim][p] == col[dim][q] && p < q);
            });
            const int mid = lo + ((hi - lo + kBlockPts - 1) / kBlockPts / 2) * kBlockPts;
            nodes.push_back({lo, mid});
            nodes.push_back({mid, hi});
        }
        for (int64_t b = 0; b < n; b += kBlockPts) {  // a block's points, in any order
            const int64_t e = std::min<int64_t>(n, b + kBlockPts);
            std::sort(order.begin() + b, order.begin() + e);
            std::sort(want.begin() + b, want.begin() + e);
        }
        CHECK(order == want);
        std::vector<int> seen((size_t)c.n_slots, 0);
        CHECK((int64_t)c.slot_of_point.size() == n);
        for (int64_t s : c.slot_of_point) CHECK(s >= 0 && s < c.n_slots && seen[s]++ == 0);
        pdfxc_ctx_destroy(ctx);
    }
    CHECK(fake_live_bytes() == 0);
}

// the context that densities keep holds no matrices beyond the pool's bound
void density_keeps_little() {
    const int n = 4800;  // three matrices of 4800 x 4800 are 553 MB
    pdfxc_ctx* ctx = context(n);
    const std::vector<double> P((size_t)n * (n + 1) / 2, 0.0), x(3000, 0.5);
    std::vector<double> rho(1000);
    const size_t before = fake_live_bytes();
    CHECK(pdfxc_density_at_points(ctx, P.data(), 1000, x.data(), rho.data(), nullptr) == PDFXC_OK);
    CHECK(fake_live_bytes() <= before + kPoolKeep);
    pdfxc_ctx_destroy(ctx);
    CHECK(fake_live_bytes() == 0);
}

// a copy that fails leaves no half-made host copies behind
void failed_copies() {
    pdfxc_ctx* ctx = context();
    Context& c = *reinterpret_cast<Context*>(ctx);
    for (int k = 0; k < 4; ++k) {
        set_grid(ctx, 70000 + k);
        fake_fail_copy(k);
        CHECK(ensure_host_grid(c) == PDFXC_ERR_HIP);
        fake_fail_copy(-1);
        CHECK(ensure_host_grid(c) == PDFXC_OK && host_grid_is_right(c));
    }
    const std::vector<int> want{3, 1, 4, 1, 5};
    int* lists[4] = {c.d_block_shells, c.d_block_cols, c.d_block_shell_col, c.d_block_sorder};
    for (int* d : lists) CHECK(hipMemcpy(d, want.data(), 5 * sizeof(int), hipMemcpyHostToDevice) == hipSuccess);
    for (int k = 0; k < 4; ++k) {
        c.n_block_shells = c.n_block_cols = 5;
        c.block_shells.clear();
        c.block_cols.clear();
        c.block_shell_col.clear();
        c.block_sorder.clear();
        fake_fail_copy(k);
        CHECK(ensure_host_lists(c) == PDFXC_ERR_HIP);
        fake_fail_copy(-1);
        CHECK(ensure_host_lists(c) == PDFXC_OK);
        CHECK(c.block_shells == want && c.block_cols == want && c.block_shell_col == want && c.block_sorder == want);
    }
    pdfxc_ctx_destroy(ctx);
}

// the bisection's tree for every number of points a grid may have: each level's
// chunks cover its nodes, the leaves cover the points, threads take each once
void part_tree_sizes() {
    for (int64_t n : {(int64_t)1, (int64_t)128, (int64_t)4096, (int64_t)4097, (int64_t)8193, (int64_t)1000077,
                      ((int64_t)1 << 31) - 128}) {
        const PartTree T = part_tree(n);
        int64_t covered = 0;
        std::vector<LeafNode> leaves = T.leaves;
        std::sort(leaves.begin(), leaves.end(), [](const LeafNode& a, const LeafNode& b) { return a.lo < b.lo; });
        for (const LeafNode& L : leaves) {
            CHECK(L.lo == covered && L.hi > L.lo && L.hi - L.lo <= kNodeMax);
            covered = L.hi;
        }
        CHECK(covered == n);
        for (size_t level = 0; level + 1 < T.node_off.size(); ++level) {
            int c = T.chunk_off[level];
            for (int k = T.node_off[level]; k < T.node_off[level + 1]; ++k) {
                const PartNode& N = T.nodes[k];
                CHECK(N.lo < N.mid && N.mid < N.hi && (N.mid - N.lo) % kLeafPts == 0);
                int64_t at = N.lo;
                for (; c < T.chunk_off[level + 1] && T.chunks[c].node == k - T.node_off[level]; ++c) {
                    CHECK(T.chunks[c].lo == at && T.chunks[c].hi > at && T.chunks[c].hi - at <= kChunk);
                    at = T.chunks[c].hi;
                }
                CHECK(at == N.hi);
            }
            CHECK(c == T.chunk_off[level + 1]);
        }
        if (T.chunks.empty()) continue;
        const PartChunk& last = T.chunks.back();
        std::vector<int> times((size_t)(last.hi - last.lo), 0);
        for (int t = 0; t < kPartThreads; ++t)
            each_point(last, t, [&](int i) {
                CHECK(i >= last.lo && i < last.hi);
                ++times[i - last.lo];
            });
        for (int k : times) CHECK(k == 1);
    }
}

}  // namespace

int main(int argc, char** argv) {
    struct {
        const char* name;
        void (*run)();
    } const checks[] = {{"pool_threads", pool_threads}, {"host_copy_threads", host_copy_threads}, {"grid_rows", grid_rows},
                  {"pool_bound", pool_bound},     {"reserve_gives_way", reserve_gives_way},
                  {"density_keeps_little", density_keeps_little}, {"failed_copies", failed_copies},
                  {"part_tree_sizes", part_tree_sizes}, {"rho_without_memory", rho_without_memory},
                  {"small_grids", small_grids}};
    for (const auto& k : checks)
        if (argc == 2 && !std::strcmp(argv[1], k.name)) {
            k.run();
            return 0;
        }
    std::printf("no such check\n");
    return 2;
}
