// Mixed-radix row and column passes (cg_fftmix.hip).
#pragma once
#include "cg_internal.hpp"

namespace cg {

constexpr int kMixStages = 8;

// Stockham passes s < ns of nb transforms of length n on `threads` threads:
// radix rad[s] after p[s] = rad[0] .. rad[s - 1], tn[s] = n / rad[s],
// st[s] = tn[s] / p[s]; mp, mt divide by p and tn; tw[s] is the pass's first entry in the twiddle table
struct MixPlan {
    int n, nb, ns, threads;
    int rad[kMixStages], p[kMixStages], tn[kMixStages], st[kMixStages], tw[kMixStages];
    uint32_t mp[kMixStages], mt[kMixStages];
};

template <typename T>
bool fft_rows_mix_supported(int n);
// the twiddle table (n entries) of launch_fft_rows_mix
template <typename T>
int launch_mix_twiddles(cx_t<T> *tw, int n, hipStream_t s);
template <typename T>
int launch_fft_rows_mix(cx_t<T> *data, int64_t nrows, int n, int dir, const cx_t<T> *tw, int live_a,
                        int live_b, const uint8_t *rowmask, int n2, hipStream_t s);
// L is 2^a 3^b 5^c
bool fft_cols_mix_supported(int L);
// transforms of length L <= 256 along n2 (see k_fft_cols_mix)
template <typename T>
int launch_fft_cols_mix(cx_t<T> *data, int batch, int n2, int n1, int L, int dir, int se, int sj,
                        int nsub, int twmode, const cx_t<T> *tw2, int live_a, int live_b,
                        const uint8_t *rowmask, int mode_in, int mode_out, int spec_a, int spec_b,
                        hipStream_t s);

}  // namespace cg
