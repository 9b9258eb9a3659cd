// Builds wide column-ordered tiles (wide_kernel's layout) on the device from
// a plan's row-ordered arrays: one workgroup per tile sorts (column, position
// in tile) in LDS with a bitonic network, cuts the order into runs of up to 64
// entries, and writes keys, values and the runs' base columns.  (R-MAT 2^20,
// 16.8M entries: the host sort of the narrower column-ordered tiles takes
// about 70 ms with 16 threads.)
#include "plan.hpp"

namespace spd {

constexpr int SORT_TPB = 1024;
constexpr uint32_t SORT_MAX = 16384;  // entries per tile: 128 KB of 8-byte sort keys

template <typename V>
__global__ __launch_bounds__(SORT_TPB) void wide_sort_kernel(const uint32_t *__restrict__ cind, const V *__restrict__ vals,
                                                             uint32_t nnz, uint32_t entries, uint32_t words,
                                                             uint32_t pbits, uint32_t ce, uint32_t cpt,
                                                             uint32_t *__restrict__ key, V *__restrict__ val,
                                                             uint32_t *__restrict__ base, uint32_t *__restrict__ flag) {
    __shared__ uint64_t s[SORT_MAX];
    __shared__ uint32_t s_run[SORT_MAX / 64 + 1];  // first entry of each run
    __shared__ uint32_t s_nrun;
    const size_t j0 = (size_t)blockIdx.x * entries, w0 = (size_t)blockIdx.x * words;
    const uint32_t nb = (uint32_t)min((size_t)entries, nnz - j0), span = 1u << (32 - pbits);
    const uint32_t G = wide_groups(nb, words);  // groups in use, as wide_kernel counts them
    uint32_t n2 = 256;
    while (n2 < nb) n2 <<= 1;
    for (uint32_t k = threadIdx.x; k < n2; k += SORT_TPB) s[k] = k < nb ? ((uint64_t)cind[j0 + k] << 32) | k : ~0ull;
    __syncthreads();
    for (uint32_t size = 2; size <= n2; size <<= 1)
        for (uint32_t st = size >> 1; st > 0; st >>= 1) {
            for (uint32_t p = threadIdx.x; p < n2 / 2; p += SORT_TPB) {
                const uint32_t i = 2 * p - (p & (st - 1)), j = i + st;  // pairs st apart
                const uint64_t a = s[i], b = s[j];
                if ((a > b) == ((i & size) == 0)) {
                    s[i] = b;
                    s[j] = a;
                }
            }
            __syncthreads();
        }
    if (threadIdx.x == 0) {
        uint32_t n = 0, k = 0;
        while (k < nb && n < 4 * G) {
            s_run[n++] = k;
            const uint32_t c = (uint32_t)(s[k] >> 32), e = min(k + 64, nb);
            if ((uint32_t)(s[e - 1] >> 32) - c < span) {
                k = e;
            } else {
                do k++;
                while ((uint32_t)(s[k] >> 32) - c < span);
            }
        }
        if (k < nb) *flag = 1;
        s_run[n] = k;
        s_nrun = n;
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < 256 * G; w += SORT_TPB) {
        // word w of the tile: entry `lane` of run i G + g; runs past the last repeat it
        const uint32_t g = w / 256, lane = w % 256 / 4, run = min(w % 4 * G + g, s_nrun - 1);
        const uint32_t k0 = s_run[run], k = min(k0 + lane, s_run[run + 1] - 1);
        const uint32_t b = (uint32_t)(s[k0] >> 32), pos = (uint32_t)s[k];
        if (lane == 0) base[w0 / 64 + g * 4 + w % 4] = b;
        key[w0 + w] = ((uint32_t)(s[k] >> 32) - b) << pbits | wide_slot(pos, ce, cpt);
        val[w0 + w] = vals[j0 + pos];
    }
}

}  // namespace spd

int launch_wide_sort(hipStream_t s, const uint32_t *cind, const void *vals, size_t sv, uint32_t nnz, uint32_t entries,
                     uint32_t words, uint32_t pbits, uint32_t ipt, size_t sa, uint32_t *key, void *val, uint32_t *base,
                     uint32_t *flag) {
    if (entries > words || words > spd::SORT_MAX || words % 256 || entries % 256 || nnz == 0 || entries == 0) return SP_ERR_ARG;
    const uint32_t ce = 16 / (uint32_t)sa, cpt = ipt / ce;
    int rc = launch_fill_zero(s, flag, 4);
    if (rc) return rc;
    const dim3 grid((unsigned)(((uint64_t)nnz + entries - 1) / entries)), block(spd::SORT_TPB);
#define SPD_SORT(V) hipLaunchKernelGGL(spd::wide_sort_kernel<V>, grid, block, 0, s, cind, (const V *)vals, nnz, entries, words, pbits, ce, cpt, key, (V *)val, base, flag)
    switch (sv) {
    case 1: SPD_SORT(uint8_t); break;
    case 2: SPD_SORT(uint16_t); break;
    case 4: SPD_SORT(uint32_t); break;
    default: SPD_SORT(uint64_t); break;
    }
#undef SPD_SORT
    if (hipGetLastError() != hipSuccess) return SP_ERR_HIP;
    uint32_t over = 0;
    SP_HIP_TRY(hipMemcpyAsync(&over, flag, 4, hipMemcpyDeviceToHost, s));
    SP_HIP_TRY(hipStreamSynchronize(s));
    return over ? SP_ERR_RANGE : SP_OK;
}
