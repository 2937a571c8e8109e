// A HIP runtime of host memory for tests of the library's host side without a
// GPU: the program defines the runtime calls libcurafft.so makes (they take
// precedence over libamdhip64's), counts and checks allocations, logs kernel
// launches by name and runs no kernel.  With every kernel skipped the
// coordinate ranges read back as range6 was when the context's memory for them
// was allocated: zero, for which a W-stacking call plans the fewest planes of its
// kernel, unless a scenario sets it.
//
//   host_runtime LIB SCENARIO
//
// prints one "name value" pair per line for the test to check.
#include <dlfcn.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace {

struct Alloc {
    size_t bytes;
    uint32_t id;
    bool host;
};
std::mutex mtx;
std::map<char *, Alloc> live;
std::map<const void *, std::string> kernels;
std::vector<std::string> launches;
size_t used = 0, peak = 0, total = (size_t)1 << 40;
uint32_t next_id = 1;
int bad_frees = 0, bad_copies = 0, allocs = 0;
// hipMalloc of exactly this size fails fail_times times
size_t fail_size = 0;
int fail_times = 0;
bool fail_new = false;  // operator new throws, but for what this program itself needs
struct OwnMemory {
    bool was = fail_new;
    OwnMemory() { fail_new = false; }
    ~OwnMemory() { fail_new = was; }
};
double range6[6];       // w, u and v: least and largest

// p lies in a live allocation with `bytes` to go
bool holds(const void *p, size_t bytes)
{
    auto it = live.upper_bound((char *)p);
    if (it == live.begin()) return false;
    --it;
    return (char *)p + bytes <= it->first + it->second.bytes;
}

hipError_t take(void **p, size_t bytes, bool host)
{
    std::lock_guard<std::mutex> lock(mtx);
    OwnMemory own;
    if (!host) {
        if (bytes == fail_size && fail_times > 0) {
            fail_times--;
            return hipErrorOutOfMemory;
        }
        if (used + bytes > total) return hipErrorOutOfMemory;
        allocs++;
    }
    // (untouched pages of calloc cost nothing)
    char *q = (char *)std::calloc(1, bytes);
    if (!q) return hipErrorOutOfMemory;
    live[q] = Alloc{bytes, next_id++, host};
    if (!host) used += bytes;
    peak = used > peak ? used : peak;
    *p = q;
    return hipSuccess;
}

hipError_t give(void *p)
{
    std::lock_guard<std::mutex> lock(mtx);
    if (!p) return hipSuccess;
    auto it = live.find((char *)p);
    if (it == live.end()) {
        bad_frees++;
        return hipErrorInvalidValue;
    }
    if (!it->second.host) used -= it->second.bytes;
    live.erase(it);
    std::free(p);
    return hipSuccess;
}

hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind)
{
    std::lock_guard<std::mutex> lock(mtx);
    const bool to = kind != hipMemcpyDeviceToHost, from = kind != hipMemcpyHostToDevice;
    if ((to && !holds(dst, bytes)) || (from && !holds(src, bytes))) {
        bad_copies++;
        return hipErrorInvalidValue;
    }
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}

// launches of kernels whose name holds `part`
int launched(const char *part)
{
    int n = 0;
    for (const std::string &s : launches) n += s.find(part) != std::string::npos;
    return n;
}

}  // namespace

void *operator new(size_t n)
{
    void *p = fail_new ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {

void **__hipRegisterFatBinary(const void *)
{
    static void *handle[1];
    return handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    cfg_grid = g;
    cfg_block = b;
    cfg_lds = lds;
    cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = cfg_grid;
    *b = cfg_block;
    *lds = cfg_lds;
    *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t)
{
    OwnMemory own;
    launches.push_back(kernels[f]);
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) { return take(p, n, false); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    const hipError_t e = take(p, n, true);
    if (e == hipSuccess && n == sizeof range6) std::memcpy(*p, range6, n);
    return e;
}
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return copy(d, s, n, k); }
hipError_t hipMemGetInfo(size_t *fr, size_t *tot)
{
    *fr = total - used;
    *tot = total;
    return hipSuccess;
}
hipError_t hipDeviceTotalMem(size_t *n, hipDevice_t)
{
    *n = total;
    return hipSuccess;
}
hipError_t hipPointerGetAttribute(void *data, hipPointer_attribute what, hipDeviceptr_t p)
{
    std::lock_guard<std::mutex> lock(mtx);
    auto it = live.find((char *)p);
    if (it == live.end() || what != HIP_POINTER_ATTRIBUTE_BUFFER_ID) return hipErrorInvalidValue;
    *(uint32_t *)data = it->second.id;
    return hipSuccess;
}
// every allocation is gone; the next one of the size may get its address
hipError_t hipDeviceReset(void)
{
    std::lock_guard<std::mutex> lock(mtx);
    for (auto &a : live) std::free(a.first);
    live.clear();
    used = 0;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

}  // extern "C"

namespace {

using Host = int (*)(int, int, int, double, double, double *, double *, double *, double *, double, double, int);
using HostF = int (*)(int, int, int, float, float, float *, float *, float *, float *, float, float, int);

struct Lib {
    void *h;
    template <typename F>
    F sym(const char *name) const
    {
        F f = (F)dlsym(h, name);
        if (!f) {
            std::fprintf(stderr, "%s\n", dlerror());
            std::exit(3);
        }
        return f;
    }
    // ms2dirty_1 / ms2dirtyf_1 of nrow zero rows onto nx x ny pixels
    int image(int nrow, int nx, int ny, double eps = 1e-5) const
    {
        std::vector<double> uvw(3 * (size_t)nrow), vis(2 * (size_t)nrow), img(2 * (size_t)nx * ny);
        auto f = sym<int (*)(int, int, int, double, double, double *, double *, double *, double, double, int)>(
            "ms2dirty_1");
        return f(nrow, nx, ny, 1.0, 1e9, uvw.data(), vis.data(), img.data(), eps, 2.0, -1);
    }
    int nufft(int M, int n) const
    {
        std::vector<double> x(M), c(2 * (size_t)M), k(2 * (size_t)n * n);
        auto f = sym<int (*)(int, const double *, const double *, const double *, int, int, double *, double, double)>(
            "nufft2d1");
        return f(M, x.data(), x.data(), c.data(), n, n, k.data(), 1e-5, 2.0);
    }
    int imagef(int nrow, int nx, int ny, float eps = 1e-5f) const
    {
        std::vector<float> uvw(3 * (size_t)nrow), vis(2 * (size_t)nrow), img(2 * (size_t)nx * ny);
        auto f = sym<int (*)(int, int, int, float, float, float *, float *, float *, float, float, int)>(
            "ms2dirtyf_1");
        return f(nrow, nx, ny, 1.f, 1e9f, uvw.data(), vis.data(), img.data(), eps, 2.f, -1);
    }
};

void show(const char *name, long long v) { std::printf("%s %lld\n", name, v); }

// the number of twiddle tables a call of this shape builds
int tables(const Lib &L, int nx, int ny, bool single, const char *name)
{
    launches.clear();
    const int ier = single ? L.imagef(10, nx, ny) : L.image(10, nx, ny);
    show((std::string(name) + "_ier").c_str(), ier);
    const int n = launched("twiddles");
    show((std::string(name) + "_tables").c_str(), n);
    return n;
}

// A table whose memory is gone, or that was filled in another precision, is
// built again: 64 x 64 pixels give 128-point tables of 2 KB (complex128), 100
// pixels 200-point ones of 3200 bytes.
void twiddle_tags(const Lib &L)
{
    tables(L, 64, 64, false, "first");
    tables(L, 64, 64, false, "again");
    fail_size = 3200;  // the row table of the larger call, also when it is tried again
    fail_times = 100;
    tables(L, 64, 100, false, "failed");
    fail_times = 0;
    tables(L, 64, 64, false, "after_row");
    // the column table fails once the row table of the new precision is there:
    // complex64 tables of 960 points take 7680 bytes
    tables(L, 480, 64, true, "single");
    fail_size = 15360;
    fail_times = 100;
    tables(L, 480, 64, false, "failed_column");
    fail_times = 0;
    tables(L, 480, 64, true, "single_again");
}

// the same in a context, whose buffers outlive a failed call
void context_tags(const Lib &L)
{
    const auto create = L.sym<int (*)(void **, void *)>("cg_ctx_create");
    const auto fft = L.sym<int (*)(void *, int, void *, int, int, int, int)>("cg_fft2d_dev");
    void *ctx = nullptr, *data = nullptr;
    show("ier", create(&ctx, nullptr));
    (void)take(&data, 1 << 20, false);
    auto run = [&](const char *name, int prec, int n2, int n1) {
        launches.clear();
        show((std::string(name) + "_ier").c_str(), fft(ctx, prec, data, 1, n2, n1, 1));
        show((std::string(name) + "_tables").c_str(), launched("twiddles"));
    };
    run("first", 1, 128, 128);
    run("again", 1, 128, 128);
    fail_size = 3200;
    fail_times = 100;
    run("failed", 1, 128, 200);
    run("after_row", 1, 128, 128);
    run("single", 0, 240, 128);
    fail_size = 3840;
    run("failed_column", 1, 240, 128);
    run("single_again", 0, 240, 128);
    fail_times = 0;
    L.sym<int (*)(void *)>("cg_ctx_destroy")(ctx);
    (void)give(data);
    show("left", (long long)used);
}

// What an earlier call left must not take the room of a later one: with a
// device that just holds the later call, it runs as on an idle device.
void surplus(const Lib &L)
{
    const auto release = L.sym<int (*)()>("cg_host_release");
    show("alone_ier", L.nufft(2000, 256));
    release();
    const size_t need = peak;
    show("before_ier", L.image(10, 16, 16));
    show("kept", used > 0);
    total = need;  // not a byte to spare
    show("after_ier", L.nufft(2000, 256));
    release();
    // the least device memory that holds a call's whole grid
    int whole = 0;
    for (total = (size_t)256 << 20; !whole; total += (size_t)1 << 20) {
        launches.clear();
        const int ier = L.image(10, 512, 512);
        whole = ier == 0 && launched("k_grid_sparse") == 1;
        release();
    }
    show("many_ier", L.nufft(200000, 64));
    show("many_kept", used > ((size_t)8 << 20));
    launches.clear();
    show("whole_ier", L.image(10, 512, 512));
    show("slabs", launched("k_grid_sparse"));
}

// ms2dirty on a context with gridding tiles of a given edge, 40 x 36 pixels
void tile_edges(const Lib &L)
{
    const auto create = L.sym<int (*)(void **, void *)>("cg_ctx_create");
    const auto option = L.sym<int (*)(void *, const char *, int)>("cg_ctx_set_option");
    const auto run = L.sym<int (*)(void *, int, int, int, int, double, double, const void *, int, const void *,
                                   const void *, int, void *, double, double, int)>("cg_ms2dirty_dev");
    void *uvw = nullptr, *vis = nullptr, *img = nullptr;
    (void)take(&uvw, 24 * 50, false);
    (void)take(&vis, 16 * 50, false);
    (void)take(&img, 16 * 40 * 36, false);
    for (const int tile : {0, 1, 2, 3, 5, 8, 12})
        for (const int kw : {4, 9, 10, 13}) {
            void *ctx = nullptr;
            (void)create(&ctx, nullptr);
            option(ctx, "tile_grid", tile);
            launches.clear();
            const int ier = run(ctx, 1, 50, 40, 36, 5.0, 1e9, uvw, 1, vis, nullptr, 1, img, std::pow(10.0, 1 - kw) * 1.01, 2.0, -1);
            show(("tile" + std::to_string(tile) + "_kw" + std::to_string(kw)).c_str(), ier);
            L.sym<int (*)(void *)>("cg_ctx_destroy")(ctx);
        }
}

// ms2dirty calls by whether crowded regions may go to k_grid
void crowded_rule(const Lib &L)
{
    const auto create = L.sym<int (*)(void **, void *)>("cg_ctx_create");
    const auto option = L.sym<int (*)(void *, const char *, int)>("cg_ctx_set_option");
    const auto run = L.sym<int (*)(void *, int, int, int, int, double, double, const void *, int, const void *,
                                   const void *, int, void *, double, double, int)>("cg_ms2dirty_dev");
    const int most = 50000;
    void *uvw = nullptr, *vis = nullptr, *img = nullptr;
    (void)take(&uvw, (size_t)24 * most, false);
    (void)take(&vis, (size_t)16 * most, false);
    (void)take(&img, (size_t)16 * 64 * 64, false);
    auto call = [&](const char *name, int prec, int rows, int nx, int kw, int tile, int dense) {
        void *ctx = nullptr;
        (void)create(&ctx, nullptr);
        option(ctx, "tile_grid", tile);
        option(ctx, "dense_min", dense);
        launches.clear();
        const int ier = run(ctx, prec, rows, nx, nx, 5.0, 1e9, uvw, 1, vis, nullptr, prec, img,
                            std::pow(10.0, 1 - kw) * 1.01, 2.0, -1);
        show(name, ier ? -ier : launched("6k_gridI"));
        L.sym<int (*)(void *)>("cg_ctx_destroy")(ctx);
    };
    call("narrow", 1, 1000, 64, 4, 8, 64);
    call("few_rows", 1, 50, 64, 4, 8, 64);
    call("width8_tile8", 1, most, 64, 8, 8, 64);
    call("width8_tile2", 1, most, 25, 8, 8, 64);
    call("width13", 1, most, 25, 13, 8, 64);
    call("few_rows_wide", 1, 400, 25, 8, 8, 64);
    call("odd_tile", 1, 1000, 60, 4, 12, 64);
    call("dense", 0, most, 64, 4, 8, 64);
    call("no_dense", 0, most, 64, 4, 8, 0);
    call("late_dense", 0, most, 64, 4, 8, 100000);
    // some 22 and 56 planes (w, u and v in metres)
    for (int windows : {2, 4})
        for (int kw : {3, 4, 5, 6, 7}) {
            const double w = windows == 2 ? 620 : 2000, uv = 95;
            const double r[6] = {-w, w, -uv, uv, -uv, uv};
            std::memcpy(range6, r, sizeof r);
            for (int prec : {0, 1}) {
                const std::string name = "p" + std::to_string(prec) + "_windows" + std::to_string(windows) + "_kw" +
                                         std::to_string(kw);
                call(name.c_str(), prec, most, 64, kw, 8, 0);
            }
        }
}

// dirty2ms calls by whether tiles with few points are read straight from the planes
void degrid_rule(const Lib &L)
{
    const auto create = L.sym<int (*)(void **, void *)>("cg_ctx_create");
    const auto option = L.sym<int (*)(void *, const char *, int)>("cg_ctx_set_option");
    const auto run = L.sym<int (*)(void *, int, int, int, int, double, double, const void *, int, void *,
                                   const void *, int, const void *, double, double, int)>("cg_dirty2ms_dev");
    const int most = 130 * 4096;
    void *uvw = nullptr, *vis = nullptr, *img = nullptr;
    (void)take(&uvw, (size_t)24 * most, false);
    (void)take(&vis, (size_t)16 * most, false);
    (void)take(&img, (size_t)16 * 64 * 64, false);
    auto call = [&](int tile, int kw, double w, int per) {
        const double r[6] = {-w, w, -108, 108, -108, 108};  // u and v reach the whole grid
        std::memcpy(range6, r, sizeof r);
        void *ctx = nullptr;
        (void)create(&ctx, nullptr);
        option(ctx, "tile_degrid", tile);
        launches.clear();
        const int ier = run(ctx, 1, per * (128 / tile) * (128 / tile), 64, 64, 5.0, 1e9, uvw, 1, vis, nullptr, 1,
                            img, std::pow(10.0, 1 - kw) * 1.01, 2.0, -1);
        show(("tile" + std::to_string(tile) + "_kw" + std::to_string(kw) + "_w" + std::to_string((int)w) + "_" +
              std::to_string(per)).c_str(), ier ? -ier : launched("k_degrid_direct"));
        L.sym<int (*)(void *)>("cg_ctx_destroy")(ctx);
    };
    // the fewest planes, about 30 and about 110
    for (double w : {10., 620., 4000.})
        for (int tile : {2, 4, 8, 16})
            for (int kw : {4, 6, 9, 13})
                for (int per : {10, 25, 40, 70, 90, 120, 130}) call(tile, kw, w, per);
}

// the column steps of complex128 transforms: steps on the prefetching kernel
void column_rule(const Lib &L)
{
    const auto create = L.sym<int (*)(void **, void *)>("cg_ctx_create");
    const auto fft = L.sym<int (*)(void *, int, void *, int, int, int, int)>("cg_fft2d_dev");
    void *ctx = nullptr, *data = nullptr;
    (void)create(&ctx, nullptr);
    (void)take(&data, (size_t)4 << 30, false);
    const int shapes[][4] = {{1, 1, 1024, 1024}, {1, 16, 2048, 1024}, {1, 16, 2048, 2048}, {1, 17, 4096, 2048},
                             {1, 16, 8192, 2048}, {1, 1, 1000, 1024}, {0, 1, 1024, 1024}};
    for (const auto &s : shapes) {
        launches.clear();
        const int ier = fft(ctx, s[0], data, s[1], s[2], s[3], 1);
        char name[64];
        std::snprintf(name, sizeof name, "p%d_%dx%dx%d", s[0], s[1], s[2], s[3]);
        show(name, ier ? -ier : launched("k_fft_cols_step_pf"));
    }
    L.sym<int (*)(void *)>("cg_ctx_destroy")(ctx);
}

// what two calls leave allocated
void kept_bytes(const Lib &L)
{
    show("ier", L.image(1000, 64, 64));
    show("kept", (long long)used);
    show("second_ier", L.image(1000, 100, 64));
    show("second_kept", (long long)used);
}

// After a device reset the kept buffers are gone: nothing may write to them,
// free them or take their addresses, now another's, for its own.
void device_reset(const Lib &L)
{
    show("before_ier", L.image(1000, 64, 64));
    show("kept", used > 0);
    (void)hipDeviceReset();
    std::vector<void *> others;
    for (const size_t bytes : {(size_t)1 << 12, (size_t)24000, (size_t)16000, (size_t)1 << 20}) {
        others.push_back(nullptr);
        (void)take(&others.back(), bytes, false);
    }
    const size_t held = used;
    show("after_ier", L.image(1000, 64, 64));
    (void)hipDeviceReset();
    const int ier = L.sym<int (*)()>("cg_host_release")();
    show("release_ier", ier);
    show("left", (long long)used);
    // a reset with another's memory at every kept address
    show("again_ier", L.image(1000, 64, 64));
    std::vector<std::pair<char *, Alloc>> was(live.begin(), live.end());
    for (auto &a : was) live[a.first].id = next_id++;
    show("moved_ier", L.image(1000, 64, 64));
    int lost = 0;
    for (auto &a : was) lost += !live.count(a.first);
    show("others_freed", lost);
    show("held", held > 0);
}

// the release itself needs no host memory
void release_without_heap(const Lib &L)
{
    show("ier", L.image(100, 64, 64));
    show("kept", used > 0);
    const auto release = L.sym<int (*)()>("cg_host_release");
    fail_new = true;
    const int ier = release();
    fail_new = false;
    show("release_ier", ier);
    show("left", (long long)used);
    show("allocations_left", (long long)live.size());
}

// nufft2d1 calls by whether the gridder takes the tiles from a list
void list_rule(const Lib &L)
{
    const auto create = L.sym<int (*)(void **, void *)>("cg_ctx_create");
    const auto run = L.sym<int (*)(void *, int, int, int, const void *, const void *, void *, int, int, void *, double,
                                   double)>("cg_nufft2d_dev");
    void *x = nullptr, *f = nullptr;
    (void)take(&x, (size_t)16 * 2000000, false);
    (void)take(&f, (size_t)16 * 2700 * 2700, false);
    for (int prec : {0, 1})
        for (int n : {256, 1024, 1500, 2048, 2700})
            for (int m : {30000, 1000000}) {
                void *ctx = nullptr;
                (void)create(&ctx, nullptr);
                launches.clear();
                const int ier = run(ctx, 1, prec, m, x, x, x, n, n, f, 1e-5, 2.0);
                show(("p" + std::to_string(prec) + "_" + std::to_string(n) + "_" + std::to_string(m)).c_str(),
                     ier ? -ier : launched("k_need_tiles"));
                L.sym<int (*)(void *)>("cg_ctx_destroy")(ctx);
            }
}

// transforms of lengths seen for the first time, without host memory to keep
// their plans, then with it
void plans_without_heap(const Lib &L)
{
    void *ctx = nullptr, *data = nullptr;
    L.sym<int (*)(void **, void *)>("cg_ctx_create")(&ctx, nullptr);
    (void)take(&data, (size_t)16 * 1000 * 900, false);
    const auto fft = L.sym<int (*)(void *, int, void *, int, int, int, int)>("cg_fft2d_dev");
    for (const bool none : {true, false})
        for (int prec : {0, 1}) {
            launches.clear();
            fail_new = none;
            const int ier = fft(ctx, prec, data, 1, 900, 1000, 1);
            fail_new = false;
            const std::string name = std::string(none ? "none" : "some") + std::to_string(prec);
            show((name + "_ier").c_str(), ier);
            show((name + "_rows").c_str(), launched("k_fft_rows_mix"));
            show((name + "_cols").c_str(), launched("k_fft_cols_mix"));
        }
}

}  // namespace

int main(int argc, char **argv)
{
    if (argc != 3) return 2;
    Lib L{dlopen(argv[1], RTLD_NOW | RTLD_GLOBAL)};
    if (!L.h) {
        std::fprintf(stderr, "%s\n", dlerror());
        return 3;
    }
    const std::string what = argv[2];
    if (what == "twiddle_tags") twiddle_tags(L);
    else if (what == "release_without_heap") release_without_heap(L);
    else if (what == "context_tags") context_tags(L);
    else if (what == "device_reset") device_reset(L);
    else if (what == "kept_bytes") kept_bytes(L);
    else if (what == "tile_edges") tile_edges(L);
    else if (what == "crowded_rule") crowded_rule(L);
    else if (what == "degrid_rule") degrid_rule(L);
    else if (what == "list_rule") list_rule(L);
    else if (what == "plans_without_heap") plans_without_heap(L);
    else if (what == "column_rule") column_rule(L);
    else if (what == "surplus") surplus(L);
    else return 2;
    show("bad_frees", bad_frees);
    show("bad_copies", bad_copies);
    return 0;
}
