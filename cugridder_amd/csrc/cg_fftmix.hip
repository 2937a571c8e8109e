// Row and column passes for lengths 2^a 3^b 5^c without a compile-time plan
// (cg_fft.hip has the powers of two): Stockham passes whose radices are chosen
// at run time (mix_plan), one function body per radix.
//
// Each thread owns whole butterflies: the first pass loads its inputs from HBM
// straight into registers, the last stores from them, so a length of R1 R2 R3
// goes through LDS twice (6250 = 25 x 25 x 10; a plan of radices up to 8 takes
// it through six times).  Index divisions are multiplications by reciprocals.
// Masked rows and columns, dead columns and dead frequencies are neither read
// nor written.
#include <algorithm>
#include <mutex>
#include <new>
#include <unordered_map>

#include "cg_fft.hpp"
#include "cg_fftmix.hpp"

namespace cg {

namespace {

// x / d for 0 <= x < 2^15, d < 2^15: m = floor(2^32 / d) + 1
__host__ __device__ inline uint32_t div_magic(int d) { return (uint32_t)(0xffffffffu / (uint32_t)d) + 1u; }
__device__ __forceinline__ int div_by(int x, int d, uint32_t m) { return d == 1 ? x : (int)__umulhi((uint32_t)x, m); }

constexpr int kMixMaxThreads = 704;

// butterflies of radix r a thread takes per pass: about EPT elements
__host__ __device__ constexpr int mix_per_thread(int ept, int r) { return ept / r > 0 ? ept / r : 1; }
constexpr int kRowEpt32 = 32, kRowEpt64 = 16, kColEpt = 16;

// complex128 radices above 16 do not fit the registers
template <typename T>
constexpr int mix_max_radix() { return sizeof(T) == 4 ? 25 : 16; }

constexpr int kRadices[] = {25, 20, 16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};

// the cheapest product of radices for `nb` transforms of length n on at most
// kMixMaxThreads threads: a pass costs its trip through LDS and barriers
// (four units an element), its butterfly's arithmetic (log2 of the radix) and
// the lanes it leaves idle
struct MixSearch {
    int n, nb, ept, rmax;
    MixPlan best{};
    double cost = 1e30;
    int rad[16];
    int threads(int k) const
    {
        int t = 64;
        for (int s = 0; s < k; s++) {
            const int f = nb * (n / rad[s]), per = mix_per_thread(ept, rad[s]);
            t = std::max(t, ((f + per - 1) / per + 63) / 64 * 64);
        }
        return t;
    }
    void go(int rest, int from, int k)
    {
        if (rest == 1) {
            const int t = threads(k);
            if (t > kMixMaxThreads) return;
            double c = 0;
            for (int s = 0; s < k; s++) {
                const int f = nb * (n / rad[s]), per = (f + t - 1) / t;
                c += (4.0 + std::log2((double)rad[s])) * t * per * rad[s] / ((double)nb * n);
            }
            if (c < cost) {
                cost = c;
                best.ns = k;
                best.threads = t;
                std::copy(rad, rad + k, best.rad);
            }
            return;
        }
        if (k == kMixStages) return;
        for (int i = from; i < (int)(sizeof(kRadices) / sizeof(int)); i++) {
            if (kRadices[i] > rmax || rest % kRadices[i]) continue;
            rad[k] = kRadices[i];
            go(rest / kRadices[i], i, k + 1);
        }
    }
};

MixPlan search_plan(int n, int nb, int ept, int rmax)
{
    MixSearch S{n, nb, ept, rmax};
    if (n > 1) S.go(n, 0, 0);
    MixPlan P = S.best;
    P.n = n;
    P.nb = nb;
    if (P.ns == 0) return P;
    // an odd radix first: its outputs, stored R apart in LDS, fall on
    // different banks
    for (int s = 0; s < P.ns; s++)
        if (P.rad[s] & 1) {
            std::rotate(P.rad, P.rad + s, P.rad + s + 1);
            break;
        }
    int p = 1, off = 0;
    for (int s = 0; s < P.ns; s++) {
        P.p[s] = p;
        P.mp[s] = div_magic(p);
        P.tn[s] = n / P.rad[s];
        P.mt[s] = div_magic(P.tn[s]);
        P.st[s] = P.tn[s] / p;
        P.tw[s] = off;
        if (s) off += p * (P.rad[s] - 1);
        p *= P.rad[s];
    }
    return P;
}

// plans are searched once per length; without memory to keep one, on every call
MixPlan cached_plan(int n, int nb, int ept, int rmax)
{
    static std::mutex m;
    static std::unordered_map<uint64_t, MixPlan> plans;
    const uint64_t key = ((uint64_t)n << 32) | ((uint64_t)nb << 16) | ((uint64_t)ept << 8) | rmax;
    std::lock_guard<std::mutex> lock(m);
    auto it = plans.find(key);
    if (it != plans.end()) return it->second;
    const MixPlan P = search_plan(n, nb, ept, rmax);
    try {
        plans.emplace(key, P);
    } catch (const std::bad_alloc &) {
    }
    return P;
}

// rows per workgroup: short rows are transformed together, about 4096
// elements, at most 32 rows (a bit each in the kernel)
int rows_per_group(int n) { return std::min(32, std::max(1, 4096 / n)); }

template <typename T>
MixPlan row_plan(int n)
{
    return cached_plan(n, rows_per_group(n), sizeof(T) == 4 ? kRowEpt32 : kRowEpt64, mix_max_radix<T>());
}
template <typename T>
size_t row_lds(const MixPlan &P)
{
    const size_t e = (size_t)P.nb * P.n;
    return (e + (P.rad[0] & 1 ? 0 : e >> 5)) * sizeof(cx_t<T>);
}

template <typename F>
__device__ __forceinline__ void with_radix(int r, F &&f)
{
    switch (r) {
    case 25: f(std::integral_constant<int, 25>{}); break;
    case 20: f(std::integral_constant<int, 20>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    case 15: f(std::integral_constant<int, 15>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    default: break;
    }
}
template <typename T, typename F>
__device__ __forceinline__ void with_mix_radix(int r, F &&f)
{
    with_radix(r, [&](auto RC) {
        if constexpr (decltype(RC)::value <= mix_max_radix<T>()) f(RC);
    });
}

}  // namespace

// Rows: persistent workgroups over groups of P.nb rows.  tw: the table of
// launch_row_twiddles, pass s reading w_n^(r kk n / (p R)) at P.tw[s] +
// (r - 1) p + kk, consecutive in kk as the lanes are.  Rows with mask 0 are
// zero on input (dir > 0) or unread on output (dir < 0), as are the columns x
// with rowmask[n2 + x] = 0.
template <typename T, int DIR>
__global__ __launch_bounds__(768) void k_fft_rows_mix(cx_t<T> *data, int64_t nrows, MixPlan P,
                                                      const cx_t<T> *__restrict__ tw, Live live,
                                                      const uint8_t *__restrict__ rowmask, int n2)
{
    constexpr int EPT = sizeof(T) == 4 ? kRowEpt32 : kRowEpt64;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx_t<T> *buf = reinterpret_cast<cx_t<T> *>(smem_raw);
    const int n = P.n, nt = blockDim.x, last = P.ns - 1;
    const int sh = P.rad[0] & 1 ? 31 : 5;  // LDS padding, see row_lds
    auto pos = [&](int x) { return x + (x >> sh); };
    // bit k R + r: element r of the thread's butterfly k is read in the
    // first pass / stored in the last one, the same in every group
    uint32_t inbits = 0, outbits = 0;
    {
        auto want = [&](int x, bool column_mask) {
            return column_mask ? !rowmask || rowmask[n2 + x] != 0 : live(x);
        };
        auto bits = [&](int s, bool column_mask) {
            uint32_t w = 0;
            const int R = P.rad[s], per = mix_per_thread(EPT, R), tn = P.tn[s];
            for (int k = 0; k < per; k++) {
                const int q = threadIdx.x + k * nt;
                if (q >= P.nb * tn) break;
                const int i = q - div_by(q, tn, P.mt[s]) * tn;
                for (int r = 0; r < R; r++)
                    if (want(i + r * tn, column_mask)) w |= 1u << (k * R + r);
            }
            return w;
        };
        // (the last pass's output stride p is n / R, the first's input stride)
        inbits = bits(0, DIR > 0);
        outbits = bits(last, DIR < 0);
    }
    const int64_t ngroups = (nrows + P.nb - 1) / P.nb;
    for (int64_t g = blockIdx.x; g < ngroups; g += gridDim.x) {
        const int64_t row0 = g * P.nb;
        cx_t<T> *base = data + row0 * n;
        const int nrow = (int)min((int64_t)P.nb, nrows - row0);
        // rows of the group that take part
        uint32_t on = 0xffffffffu >> (32 - nrow);
        if (rowmask) {
            const int r0 = (int)(row0 % n2), lane = threadIdx.x & 63;
            on = (uint32_t)__ballot(lane < nrow && rowmask[(r0 + lane) % n2] != 0);
            if (!on) continue;  // the same in every wave
        }
        for (int s = 0; s <= last; s++) {
            with_mix_radix<T>(P.rad[s], [&](auto RC) {
                constexpr int R = decltype(RC)::value, K = mix_per_thread(EPT, R);
                const int tn = P.tn[s], p = P.p[s], nbf = P.nb * tn;
                cx_t<T> u[K][R];
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int q = threadIdx.x + k * nt;
                    if (q >= nbf) continue;
                    const int b = P.nb == 1 ? 0 : div_by(q, tn, P.mt[s]);
                    const int i = q - b * tn;
                    if (s == 0) {
                        const bool rd = (on >> b) & 1u;
                        const cx_t<T> *src = base + (int64_t)b * n + i;
#pragma unroll
                        for (int r = 0; r < R; r++)
                            u[k][r] = rd && ((inbits >> (k * R + r)) & 1u) ? src[r * tn] : mkc((T)0, (T)0);
                    } else {
                        const int kk = i - div_by(i, p, P.mp[s]) * p;
                        const cx_t<T> *t = tw + P.tw[s] + kk;
                        const int x = b * n + i;
#pragma unroll
                        for (int r = 0; r < R; r++) u[k][r] = buf[pos(x + r * tn)];
#pragma unroll
                        for (int r = 1; r < R; r++) {
                            cx_t<T> w = t[(r - 1) * p];
                            if (DIR < 0) w.y = -w.y;
                            u[k][r] = cmul<T>(u[k][r], w);
                        }
                    }
                }
                // every read of the previous pass (of the previous group's
                // last one for s = 0) precedes the writes
                lds_barrier();
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int q = threadIdx.x + k * nt;
                    if (q >= nbf) continue;
                    dft_small<T, R, DIR>(u[k]);
                    const int b = P.nb == 1 ? 0 : div_by(q, tn, P.mt[s]);
                    const int i = q - b * tn;
                    if (s == last) {
                        if ((on >> b) & 1u) {
                            cx_t<T> *dst = base + (int64_t)b * n + i;
#pragma unroll
                            for (int r = 0; r < R; r++)
                                if ((outbits >> (k * R + r)) & 1u) dst[r * tn] = u[k][r];
                        }
                    } else {
                        const int kk = i - div_by(i, p, P.mp[s]) * p;
                        const int x = b * n + (i - kk) * R + kk;
#pragma unroll
                        for (int r = 0; r < R; r++) buf[pos(x + r * p)] = u[k][r];
                    }
                }
                if (s != last) lds_barrier();
            });
        }
    }
}

// Columns: blocks of CB = 2^P.cbsh adjacent live columns, element e of column
// b at e CB + b in LDS.  A sub-transform j of length L = P.n reads and writes
// rows j sj + e se; twmode 1 multiplies output e by w^(j e) after the
// transform, 2 input e before it, w = e^(dir 2 pi i / n2) (tw2: the table of
// n2).  UNI: 64 columns, so that a wave works on one butterfly index and the
// twiddles are scalar loads.  mode_in / mode_out: 1 skips the rows with mask 0,
// 2 the frequencies j + nsub e in [spec_a, spec_b).
template <typename T, int DIR, bool UNI>
__global__ __launch_bounds__(768) void k_fft_cols_mix(cx_t<T> *data, int n2, int n1, MixPlan P, int cbsh,
                                                      int se, int sj, int nsub, int batch, int twmode,
                                                      const cx_t<T> *__restrict__ tw2, Live live,
                                                      const uint8_t *__restrict__ rowmask, int mode_in,
                                                      int mode_out, int spec_a, int spec_b)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx_t<T> *buf = reinterpret_cast<cx_t<T> *>(smem_raw);
    const int CB = UNI ? 64 : 1 << cbsh, bsh = UNI ? 6 : cbsh;
    const int nt = blockDim.x, last = P.ns - 1, ts = n2 / P.n;
    const int nlive = live.count(n1);
    const int nx = (nlive + CB - 1) >> bsh;
    const int64_t ntile = (int64_t)nx * nsub * batch;
    const int b = threadIdx.x & (CB - 1);  // nt is a multiple of CB
    // complex128 forward: the mask of a tile's rows as a bit per element, loaded a
    // tile ahead by the lanes of each wave.  A byte waited for before each load
    // of a row took the first step of a call (4096 x 2048 x 194) from 11.2 to
    // 16.2 ms.  Not in complex64, where the wider code costs a wave per SIMD (16
    // channels on 3000 x 2500 cells: 0.68 ms the call, so 0.88), and not in the
    // inverse step, which only stores by the mask (ragged 4800 x 6250: 3.02 ms,
    // so 3.24).
    constexpr bool BITS = DIR > 0 && sizeof(T) == 8;
    uint8_t ahead[4] = {};
    auto row_bytes = [&](int64_t t) {
        if (!BITS || mode_in != 1 || t >= ntile) return;
        const int j = (int)(t / nx % nsub);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const int e = 64 * w + (threadIdx.x & 63);
            ahead[w] = e < P.n ? rowmask[j * sj + e * se] : 0;
        }
    };
    row_bytes(blockIdx.x);
    for (int64_t t = blockIdx.x; t < ntile; t += gridDim.x) {
        uint64_t rows[4];
#pragma unroll
        for (int w = 0; w < 4; w++) rows[w] = __ballot(ahead[w] != 0);
        row_bytes(t + gridDim.x);
        const int x = (int)(t % nx);
        const int64_t rest = t / nx;
        const int j = (int)(rest % nsub);
        const int c = x * CB + b;
        const bool cok = c < nlive;
        cx_t<T> *pl = data + (size_t)(rest / nsub) * n2 * n1 + (cok ? live.at(c) : 0);
        auto skip = [&](int mode, int row, int e) -> bool {
            if (mode == 1) {
                if (!BITS) return rowmask[row] == 0;
                const uint64_t w = e < 128 ? (e < 64 ? rows[0] : rows[1]) : (e < 192 ? rows[2] : rows[3]);
                return !((w >> (e & 63)) & 1);
            }
            const int k = j + nsub * e;
            return mode == 2 && k >= spec_a && k < spec_b;
        };
        for (int s = 0; s <= last; s++) {
            with_mix_radix<T>(P.rad[s], [&](auto RC) {
                constexpr int R = decltype(RC)::value, K = mix_per_thread(kColEpt, R);
                const int tn = P.tn[s], p = P.p[s];
                auto index = [&](int k) -> int {
                    const int i = ((int)threadIdx.x + k * nt) >> bsh;
                    return UNI ? __builtin_amdgcn_readfirstlane(i) : i;
                };
                cx_t<T> u[K][R];
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int i = index(k);
                    if (i >= tn) continue;
                    if (s == 0) {
                        if constexpr (BITS) {
                            // a skipped row reads the plane's first one and is
                            // cleared once every load is on its way
                            uint32_t on = 0;
#pragma unroll
                            for (int r = 0; r < R; r++)
                                if (!skip(mode_in, 0, i + r * tn)) on |= 1u << r;
#pragma unroll
                            for (int r = 0; r < R; r++) {
                                const size_t row = (size_t)(j * sj + (i + r * tn) * se);
                                u[k][r] = pl[row * n1 * ((on >> r) & 1u)];
                            }
#pragma unroll
                            for (int r = 0; r < R; r++)
                                if (!((on >> r) & 1u)) u[k][r] = mkc((T)0, (T)0);
                        } else {
#pragma unroll
                            for (int r = 0; r < R; r++) {
                                const int e = i + r * tn, row = j * sj + e * se;
                                u[k][r] = cok && !skip(mode_in, row, e) ? pl[(size_t)row * n1] : mkc((T)0, (T)0);
                            }
                        }
                        if (twmode == 2) {
#pragma unroll
                            for (int r = 0; r < R; r++) {
                                cx_t<T> w = tw2[j * (i + r * tn)];
                                if (DIR < 0) w.y = -w.y;
                                u[k][r] = cmul<T>(u[k][r], w);
                            }
                        }
                    } else {
                        const int kk = i - div_by(i, p, P.mp[s]) * p;
                        const int step = kk * ts * P.st[s];
#pragma unroll
                        for (int r = 0; r < R; r++) u[k][r] = buf[((i + r * tn) << bsh) + b];
#pragma unroll
                        for (int r = 1; r < R; r++) {
                            cx_t<T> w = tw2[r * step];
                            if (DIR < 0) w.y = -w.y;
                            u[k][r] = cmul<T>(u[k][r], w);
                        }
                    }
                }
                lds_barrier();
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const int i = index(k);
                    if (i >= tn) continue;
                    dft_small<T, R, DIR>(u[k]);
                    if (s == last) {
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            const int e = i + r * tn, row = j * sj + e * se;
                            if (!cok || skip(mode_out, row, e)) continue;
                            cx_t<T> v = u[k][r];
                            if (twmode == 1) {
                                cx_t<T> w = tw2[j * e];
                                if (DIR < 0) w.y = -w.y;
                                v = cmul<T>(v, w);
                            }
                            pl[(size_t)row * n1] = v;
                        }
                    } else {
                        const int kk = i - div_by(i, p, P.mp[s]) * p;
                        const int x0 = (i - kk) * R + kk;
#pragma unroll
                        for (int r = 0; r < R; r++) buf[((x0 + r * p) << bsh) + b] = u[k][r];
                    }
                }
                if (s != last) lds_barrier();
            });
        }
    }
}

// the twiddle table of a mixed-radix row plan (see k_fft_rows_mix)
template <typename T>
__global__ __launch_bounds__(256) void k_mix_twiddles(cx_t<T> *tw, MixPlan P)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    for (int s = 1; s < P.ns; s++) {
        const int o = t - P.tw[s], p = P.p[s], R = P.rad[s];
        if (o < 0 || o >= p * (R - 1)) continue;
        const int r = o / p + 1, kk = o - (r - 1) * p;
        double sv, cv;
        sincospi(2.0 * (double)((int64_t)r * kk * P.st[s]) / (double)P.n, &sv, &cv);
        tw[t] = mkc((T)cv, (T)sv);
    }
}

template <typename T>
bool fft_rows_mix_supported(int n)
{
    if (n == 1) return true;
    if (n < 1 || n > 16384) return false;
    const MixPlan P = row_plan<T>(n);
    return P.ns > 0 && row_lds<T>(P) <= 163840;
}

template <typename T>
int launch_mix_twiddles(cx_t<T> *tw, int n, hipStream_t s)
{
    if (n <= 1) return CG_OK;
    hipLaunchKernelGGL(k_mix_twiddles<T>, dim3((n + 255) / 256), dim3(256), 0, s, tw, row_plan<T>(n));
    CG_HIP(hipGetLastError());
    return CG_OK;
}

template <typename T>
int launch_fft_rows_mix(cx_t<T> *data, int64_t nrows, int n, int dir, const cx_t<T> *tw, int live_a,
                        int live_b, const uint8_t *rowmask, int n2, hipStream_t s)
{
    if (n <= 1 || nrows <= 0) return CG_OK;
    if (!fft_rows_mix_supported<T>(n)) return CG_ERR_SIZE;
    const MixPlan P = row_plan<T>(n);
    const size_t lds = row_lds<T>(P);
    const void *fn = dir > 0 ? (const void *)k_fft_rows_mix<T, 1> : (const void *)k_fft_rows_mix<T, -1>;
    if (lds > 65536)
        CG_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int per_cu = std::min(std::max<int>(1, (int)(163840 / lds)), std::max(1, 2048 / P.threads));
    const unsigned grid = (unsigned)std::min<int64_t>((nrows + P.nb - 1) / P.nb, (int64_t)256 * per_cu);
    const Live live{live_a, live_b};
    if (dir > 0)
        hipLaunchKernelGGL((k_fft_rows_mix<T, 1>), dim3(grid), dim3(P.threads), lds, s, data, nrows, P, tw,
                           live, rowmask, n2);
    else
        hipLaunchKernelGGL((k_fft_rows_mix<T, -1>), dim3(grid), dim3(P.threads), lds, s, data, nrows, P, tw,
                           live, rowmask, n2);
    CG_HIP(hipGetLastError());
    return CG_OK;
}

bool fft_cols_mix_supported(int L)
{
    for (int f : {2, 3, 5})
        while (L > 1 && L % f == 0) L /= f;
    return L == 1;
}

template <typename T>
int launch_fft_cols_mix(cx_t<T> *data, int batch, int n2, int n1, int L, int dir, int se, int sj,
                        int nsub, int twmode, const cx_t<T> *tw2, int live_a, int live_b,
                        const uint8_t *rowmask, int mode_in, int mode_out, int spec_a, int spec_b,
                        hipStream_t s)
{
    const Live live{live_a, live_b};
    const int nlive = live.count(n1), elem = (int)sizeof(cx_t<T>);
    if (L < 2 || L > 256 || nlive <= 0 || batch <= 0) return CG_ERR_SIZE;
    // 64 columns unless the block would leave one workgroup on a CU, or most
    // of its lanes idle
    int sh = 6;
    while (sh > 3 && ((int64_t)L * elem << sh) > 81920) sh--;
    while (sh > 3 && (1 << (sh - 1)) >= nlive) sh--;
    MixPlan P;
    for (;; sh--) {
        P = cached_plan(L, 1 << sh, kColEpt, mix_max_radix<T>());
        if (P.ns > 0) break;
        if (sh == 0) return CG_ERR_SIZE;
    }
    const size_t lds = ((size_t)L << sh) * elem;
    auto go = [&](auto kern) -> int {
        if (lds > 65536)
            CG_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds));
        const int64_t ntile = (int64_t)((nlive + (1 << sh) - 1) >> sh) * nsub * batch;
        const int per_cu = std::max(1, std::min((int)(163840 / lds), 2048 / P.threads));
        const unsigned grid = (unsigned)std::min<int64_t>(ntile, (int64_t)256 * 4 * per_cu);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(P.threads), lds, s, data, n2, n1, P, sh, se, sj, nsub,
                           batch, twmode, tw2, live, rowmask, rowmask || mode_in != 1 ? mode_in : 0,
                           rowmask || mode_out != 1 ? mode_out : 0, spec_a, spec_b);
        CG_HIP(hipGetLastError());
        return CG_OK;
    };
    if (sh == 6) return dir > 0 ? go(k_fft_cols_mix<T, 1, true>) : go(k_fft_cols_mix<T, -1, true>);
    return dir > 0 ? go(k_fft_cols_mix<T, 1, false>) : go(k_fft_cols_mix<T, -1, false>);
}

#define CG_INST(T)                                                                                          \
    template bool fft_rows_mix_supported<T>(int);                                                           \
    template int launch_mix_twiddles<T>(cx_t<T> *, int, hipStream_t);                                       \
    template int launch_fft_rows_mix<T>(cx_t<T> *, int64_t, int, int, const cx_t<T> *, int, int,            \
                                        const uint8_t *, int, hipStream_t);                                 \
    template int launch_fft_cols_mix<T>(cx_t<T> *, int, int, int, int, int, int, int, int, int,             \
                                        const cx_t<T> *, int, int, const uint8_t *, int, int, int, int,     \
                                        hipStream_t);
CG_INST(float)
CG_INST(double)
#undef CG_INST

}  // namespace cg
