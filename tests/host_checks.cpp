// Checks of the engine's host code against the stand-in HIP runtime, one per
// argument; exit status 0 when it holds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "pdfxc_internal.hpp"

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

pdfxc_ctx* context() {
    const double centre[3] = {0.0, 0.0, 0.0}, exps[1] = {1.0}, coefs[1] = {1.0};
    const int type = 0, nprim = 1;
    pdfxc_opts o;
    pdfxc_default_opts(&o);
    pdfxc_ctx* ctx = nullptr;
    CHECK(pdfxc_ctx_create(&ctx, 1, centre, &type, &nprim, exps, coefs, 1, &o) == PDFXC_OK);
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
    set_grid(ctx, 1000);
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
    const int64_t n = 3000;
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

}  // namespace

int main(int argc, char** argv) {
    struct {
        const char* name;
        void (*run)();
    } const checks[] = {{"pool_threads", pool_threads}, {"host_copy_threads", host_copy_threads}, {"grid_rows", grid_rows}};
    for (const auto& k : checks)
        if (argc == 2 && !std::strcmp(argv[1], k.name)) {
            k.run();
            return 0;
        }
    std::printf("no such check\n");
    return 2;
}
