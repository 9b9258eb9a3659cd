// Variant-selector MLP: in -> h1 -> h2 -> out with ReLU between layers.
// Weights are used in BF16 (round-to-nearest-even copies of FP32 master
// weights), activations and accumulation are FP32.  Training runs on the
// GPU with these kernels: dense forward, masked-MSE loss gradient, ReLU
// backward, weight / input gradients, and Adam on the FP32 masters.  All
// reductions have a fixed order (no atomics), so training is reproducible.
// No counterpart in the reference.
#include <math.h>
#include <string.h>

#include <vector>

#include "plan.hpp"

namespace {

constexpr int TB = 16;  // output tile edge of the dense kernels

__host__ __device__ inline uint16_t f2bf(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return (uint16_t)((u >> 16) | 0x40);  // NaN
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

// out[b][o] = act(sum_i in[b][i] * W[o][i] + bias[o]); pre keeps the sum.
__global__ void dense_fwd(const float *__restrict__ in, const uint16_t *__restrict__ W,
                          const float *__restrict__ bias, float *__restrict__ pre, float *__restrict__ out, int B,
                          int I, int O, int relu) {
    __shared__ float s_in[TB][TB + 1];
    __shared__ float s_w[TB][TB + 1];
    const int tx = threadIdx.x % TB, ty = threadIdx.x / TB;
    const int b = blockIdx.y * TB + ty, o = blockIdx.x * TB + tx;
    float acc = 0.f;
    for (int i0 = 0; i0 < I; i0 += TB) {
        const int bi = blockIdx.y * TB + ty, ii = i0 + tx;
        s_in[ty][tx] = (bi < B && ii < I) ? in[(size_t)bi * I + ii] : 0.f;
        const int wo = blockIdx.x * TB + ty;
        s_w[ty][tx] = (wo < O && ii < I) ? bf2f(W[(size_t)wo * I + ii]) : 0.f;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TB; k++) acc = __builtin_fmaf(s_in[ty][k], s_w[tx][k], acc);
        __syncthreads();
    }
    if (b < B && o < O) {
        const float v = acc + bias[o];
        if (pre) pre[(size_t)b * O + o] = v;
        out[(size_t)b * O + o] = (relu && v < 0.f) ? 0.f : v;
    }
}

// dY = 2 M^2 (Y - T) / count; per-block partial loss sums (fixed order).
__global__ void mse_grad(const float *__restrict__ Y, const float *__restrict__ T, const float *__restrict__ M,
                         float *__restrict__ dY, float *__restrict__ partial, int n, float inv_count) {
    __shared__ float s[256];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (i < n) {
        const float m = M ? M[i] : 1.f;
        const float d = (Y[i] - T[i]) * m;
        dY[i] = 2.f * d * m * inv_count;
        l = d * d;
    }
    s[threadIdx.x] = l;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

__global__ void relu_bwd(float *__restrict__ d, const float *__restrict__ pre, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && pre[i] <= 0.f) d[i] = 0.f;
}

// dW[o][i] = sum_b dOut[b][o] in[b][i]; db[o] = sum_b dOut[b][o] (column i == I).
__global__ void dense_bwd_w(const float *__restrict__ dOut, const float *__restrict__ in, float *__restrict__ dW,
                            float *__restrict__ db, int B, int I, int O) {
    const int o = blockIdx.y, i = blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= O || i > I) return;
    float acc = 0.f;
    if (i < I) {
        for (int b = 0; b < B; b++) acc = __builtin_fmaf(dOut[(size_t)b * O + o], in[(size_t)b * I + i], acc);
        dW[(size_t)o * I + i] = acc;
    } else {
        for (int b = 0; b < B; b++) acc += dOut[(size_t)b * O + o];
        db[o] = acc;
    }
}

// dIn[b][i] = sum_o dOut[b][o] W[o][i] (the BF16 weights used forward).
__global__ void dense_bwd_x(const float *__restrict__ dOut, const uint16_t *__restrict__ W, float *__restrict__ dIn,
                            int B, int I, int O) {
    const int b = blockIdx.y, i = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B || i >= I) return;
    float acc = 0.f;
    for (int o = 0; o < O; o++) acc = __builtin_fmaf(dOut[(size_t)b * O + o], bf2f(W[(size_t)o * I + i]), acc);
    dIn[(size_t)b * I + i] = acc;
}

// Loss and gradient of one mini-batch in two kernels, for layer widths that are multiples of 8
// (16-byte weight loads) and at most MAXW.  A mini-batch is 1 to 4 MFLOP: what costs is the chain
// of launches and copies, not the arithmetic (batch 64 through the layer kernels above, eleven
// launches and five copies: 157 us).
//
// mlp_sample: a workgroup takes ROWS samples through the forward pass, the loss gradient and the
// input gradients, activations in LDS.  It reads the samples where the caller has them (pinned
// host memory: once, 0.5 KB per sample) and leaves what the weight gradients need in device
// memory.  mlp_weights: a workgroup takes 8 outputs x 64 inputs of one layer's weight gradient
// over all samples (LDS tiles of 64 samples), or 256 of the loss terms; the gradient goes to
// device memory (for Adam) and, when asked for, straight to pinned host memory.  Every sum runs
// in the order of the layer kernels, so the results have the same bits.
constexpr int ROWS = 2, SPT = 128, MAXW = 256;  // samples per workgroup, threads per sample

struct MlpArgs {
    int B, in, h1, h2, out;
    const float *x, *t, *m;   // the batch (m may be null: all ones)
    const float *p;           // FP32 parameters (biases)
    const uint16_t *pb;       // BF16 weights
    int off[6];
    float *xc, *a1, *a2, *d1, *d2, *d3, *l;  // kept for the weight gradients (xc: copy of x, or null)
    float *g, *hg, *part;     // gradient (device; host or null), loss partial sums
    float inv_count;
};

// out[o] = act(W[o] . in + bias[o]) for one sample by SPT threads
__device__ __forceinline__ void sample_dense(const float *s_in, int I, const uint16_t *__restrict__ W,
                                             const float *__restrict__ bias, float *s_out, int O, bool relu, int lane) {
    for (int o = lane; o < O; o += SPT) {
        float acc = 0.f;
#pragma unroll 4
        for (int i = 0; i < I; i += 8) {
            const uint4 w = *(const uint4 *)(W + (size_t)o * I + i);
            const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                acc = __builtin_fmaf(s_in[i + 2 * k], __builtin_bit_cast(float, ww[k] << 16), acc);
                acc = __builtin_fmaf(s_in[i + 2 * k + 1], __builtin_bit_cast(float, ww[k] & 0xFFFF0000u), acc);
            }
        }
        const float v = acc + bias[o];
        s_out[o] = (relu && v < 0.f) ? 0.f : v;
    }
}

// dIn[i] = sum_o dOut[o] W[o][i] where the activation is positive
__device__ __forceinline__ void sample_dense_bwd(const float *s_d, int O, const uint16_t *__restrict__ W, int I,
                                                 const float *s_act, float *s_din, int lane) {
    for (int i = lane; i < I; i += SPT) {
        float acc = 0.f;
#pragma unroll 16
        for (int o = 0; o < O; o++) acc = __builtin_fmaf(s_d[o], bf2f(W[(size_t)o * I + i]), acc);
        s_din[i] = s_act[i] <= 0.f ? 0.f : acc;
    }
}

__global__ __launch_bounds__(ROWS * SPT) void mlp_sample(MlpArgs a) {
    __shared__ __align__(16) float s_x[ROWS][MAXW], s_a1[ROWS][MAXW], s_a2[ROWS][MAXW], s_y[ROWS][MAXW];
    __shared__ __align__(16) float s_d[ROWS][MAXW], s_e[ROWS][MAXW];
    const int lane = threadIdx.x % SPT, r = threadIdx.x / SPT, b = blockIdx.x * ROWS + r;
    const bool in = b < a.B;  // (a sample past the batch computes on zeros and stores nothing)
    for (int i = lane; i < a.in; i += SPT) {
        const float v = in ? a.x[(size_t)b * a.in + i] : 0.f;
        s_x[r][i] = v;
        if (in && a.xc) a.xc[(size_t)b * a.in + i] = v;
    }
    // the targets' way over the bus runs beside the forward pass
    float t[MAXW / SPT], m[MAXW / SPT];
#pragma unroll
    for (int k = 0; k < MAXW / SPT; k++) {
        const int o = lane + k * SPT;
        const bool ok = in && o < a.out;
        t[k] = ok ? a.t[(size_t)b * a.out + o] : 0.f;
        m[k] = ok && a.m ? a.m[(size_t)b * a.out + o] : 1.f;
    }
    __syncthreads();
    sample_dense(s_x[r], a.in, a.pb + a.off[0], a.p + a.off[1], s_a1[r], a.h1, true, lane);
    __syncthreads();
    sample_dense(s_a1[r], a.h1, a.pb + a.off[2], a.p + a.off[3], s_a2[r], a.h2, true, lane);
    __syncthreads();
    sample_dense(s_a2[r], a.h2, a.pb + a.off[4], a.p + a.off[5], s_y[r], a.out, false, lane);
#pragma unroll
    for (int k = 0; k < MAXW / SPT; k++) {  // (each thread takes the outputs that it has formed)
        const int o = lane + k * SPT;
        if (o < a.out) {
            const float d = (s_y[r][o] - t[k]) * m[k];
            const float dy = 2.f * d * m[k] * a.inv_count;
            s_d[r][o] = dy;
            if (in) {
                a.d3[(size_t)b * a.out + o] = dy;
                a.l[(size_t)b * a.out + o] = d * d;
            }
        }
    }
    __syncthreads();
    sample_dense_bwd(s_d[r], a.out, a.pb + a.off[4], a.h2, s_a2[r], s_e[r], lane);
    __syncthreads();
    sample_dense_bwd(s_e[r], a.h2, a.pb + a.off[2], a.h1, s_a1[r], s_d[r], lane);
    if (!in) return;
    for (int i = lane; i < a.h1; i += SPT) {  // (each thread's own elements)
        a.a1[(size_t)b * a.h1 + i] = s_a1[r][i];
        a.d1[(size_t)b * a.h1 + i] = s_d[r][i];
    }
    for (int i = lane; i < a.h2; i += SPT) {
        a.a2[(size_t)b * a.h2 + i] = s_a2[r][i];
        a.d2[(size_t)b * a.h2 + i] = s_e[r][i];
    }
}

constexpr int WO = 8, WI = 64, WB = 64;  // outputs, inputs and samples of a weight-gradient tile

__host__ __device__ inline int weight_tiles(int I, int O) { return ((O + WO - 1) / WO) * ((I + WI - 1) / WI); }

__global__ __launch_bounds__(256) void mlp_weights(MlpArgs a, const float *__restrict__ x) {
    __shared__ float s_in[WB][WI], s_d[WB][WO];
    const int tid = threadIdx.x;
    int tile = blockIdx.x, I = a.in, O = a.h1, ow = a.off[0], ob = a.off[1];
    const float *dOut = a.d1, *in = x;
    const int n1 = weight_tiles(a.in, a.h1), n2 = weight_tiles(a.h1, a.h2), n3 = weight_tiles(a.h2, a.out);
    if (tile >= n1 + n2 + n3) {  // loss terms
        float *const s = &s_in[0][0];
        const int i = (tile - n1 - n2 - n3) * 256 + tid;
        s[tid] = i < a.B * a.out ? a.l[i] : 0.f;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (tid < w) s[tid] += s[tid + w];
            __syncthreads();
        }
        if (tid == 0) a.part[tile - n1 - n2 - n3] = s[0];
        return;
    }
    if (tile >= n1 + n2) {
        tile -= n1 + n2;
        I = a.h2; O = a.out; ow = a.off[4]; ob = a.off[5]; dOut = a.d3; in = a.a2;
    } else if (tile >= n1) {
        tile -= n1;
        I = a.h1; O = a.h2; ow = a.off[2]; ob = a.off[3]; dOut = a.d2; in = a.a1;
    }
    const int ti = (I + WI - 1) / WI, i0 = tile % ti * WI, o0 = tile / ti * WO;
    const int i = tid % WI, og = tid / WI * 2;
    float acc[2] = {0.f, 0.f}, accb = 0.f;
    for (int b0 = 0; b0 < a.B; b0 += WB) {
        const int nb = min(WB, a.B - b0);
#pragma unroll
        for (int k = 0; k < WB * WI / 256; k++) {
            const int b = tid / WI + k * (256 / WI);
            s_in[b][i] = b < nb && i0 + i < I ? in[(size_t)(b0 + b) * I + i0 + i] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < WB * WO / 256; k++) {
            const int b = tid / WO + k * (256 / WO), o = tid % WO;
            s_d[b][o] = b < nb && o0 + o < O ? dOut[(size_t)(b0 + b) * O + o0 + o] : 0.f;
        }
        __syncthreads();
#pragma unroll 8
        for (int b = 0; b < nb; b++) {
            const float v = s_in[b][i];
            acc[0] = __builtin_fmaf(s_d[b][og], v, acc[0]);
            acc[1] = __builtin_fmaf(s_d[b][og + 1], v, acc[1]);
        }
        if (i0 == 0 && tid < WO)
            for (int b = 0; b < nb; b++) accb += s_d[b][tid];
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int o = o0 + og + k;
        if (o < O && i0 + i < I) {
            const size_t at = (size_t)ow + (size_t)o * I + i0 + i;
            a.g[at] = acc[k];
            if (a.hg) a.hg[at] = acc[k];
        }
    }
    if (i0 == 0 && tid < WO && o0 + tid < O) {
        a.g[ob + o0 + tid] = accb;
        if (a.hg) a.hg[ob + o0 + tid] = accb;
    }
}

__global__ void adam_step(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                          float *__restrict__ v, uint16_t *__restrict__ pb, int n, float lr, float b1, float b2,
                          float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float upd = lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    const float np = p[i] - upd;
    p[i] = np;
    if (pb) pb[i] = f2bf(np);
}

__global__ void to_bf16(const float *__restrict__ p, uint16_t *__restrict__ pb, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) pb[i] = f2bf(p[i]);
}

}  // namespace

struct sp_mlp {
    sp_ctx *ctx = nullptr;
    int in = 0, h1 = 0, h2 = 0, out = 0;
    int np = 0;             // parameter count
    int off[6] = {0};       // W1 b1 W2 b2 W3 b3 offsets
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // FP32 masters, grads, Adam moments
    uint16_t *pb = nullptr;  // BF16 copy (weights used forward)
    int step = 0;
    // activations for a batch
    int cap = 0;
    float *x = nullptr, *a1 = nullptr, *z1 = nullptr, *a2 = nullptr, *z2 = nullptr, *y = nullptr;
    float *t = nullptr, *msk = nullptr, *d3 = nullptr, *d2 = nullptr, *d1 = nullptr, *part = nullptr, *l = nullptr;
    // pinned host memory of the two-kernel path: x, t and mask of a batch in (calls that hand over
    // a batch: hcap samples); gradient and loss partial sums out (ncap floats)
    float *hx = nullptr, *hg = nullptr;
    int hcap = 0;
    size_t ncap = 0;
    // widths that the two-kernel path takes (16-byte weight loads at every row)
    bool two() const {
        return in % 8 == 0 && h1 % 8 == 0 && h2 % 8 == 0 && in <= MAXW && h1 <= MAXW && h2 <= MAXW && out <= MAXW;
    }
};

static int mlp_alloc(float **p, size_t n) { return hipMalloc((void **)p, (n ? n : 1) * sizeof(float)) == hipSuccess ? SP_OK : SP_ERR_NOMEM; }

static int mlp_reserve(sp_mlp *m, int B) {
    if (B <= m->cap) return SP_OK;
    float **bufs[] = {&m->x, &m->a1, &m->z1, &m->a2, &m->z2, &m->y, &m->t, &m->msk, &m->d3, &m->d2, &m->d1, &m->part, &m->l};
    m->cap = 0;
    for (float **b : bufs)
        if (*b) { (void)hipFree(*b); *b = nullptr; }
    const size_t n[] = {(size_t)B * m->in, (size_t)B * m->h1, (size_t)B * m->h1, (size_t)B * m->h2, (size_t)B * m->h2,
                        (size_t)B * m->out, (size_t)B * m->out, (size_t)B * m->out, (size_t)B * m->out,
                        (size_t)B * m->h2, (size_t)B * m->h1, (size_t)B * m->out / 256 + 2, (size_t)B * m->out};
    for (int i = 0; i < 13; i++)
        if (mlp_alloc(bufs[i], n[i])) return SP_ERR_NOMEM;
    m->cap = B;
    return SP_OK;
}

// Pinned memory is slow to make: only gradients ask for it, and prediction for none.
static int mlp_pin(float **p, size_t n) {
    if (*p) (void)hipHostFree(*p);
    *p = nullptr;
    if (hipHostMalloc((void **)p, n * sizeof(float)) == hipSuccess) return SP_OK;
    (void)hipGetLastError();  // reported here
    return SP_ERR_NOMEM;
}
static int mlp_pin_in(sp_mlp *m, int B) {
    if (B <= m->hcap) return SP_OK;
    m->hcap = 0;
    if (int rc = mlp_pin(&m->hx, (size_t)B * (m->in + 2 * m->out))) return rc;
    m->hcap = B;
    return SP_OK;
}
static int mlp_pin_out(sp_mlp *m, int B) {
    const size_t n = (size_t)m->np + (size_t)B * m->out / 256 + 2;
    if (n <= m->ncap) return SP_OK;
    m->ncap = 0;
    if (int rc = mlp_pin(&m->hg, n)) return rc;
    m->ncap = n;
    return SP_OK;
}

extern "C" int sp_mlp_create(sp_ctx *ctx, int in, int h1, int h2, int out, uint64_t seed, sp_mlp **res) {
    if (!ctx || in <= 0 || h1 <= 0 || h2 <= 0 || out <= 0 || !res) return SP_ERR_ARG;
    (void)hipSetDevice(ctx->device);
    sp_mlp *m = new sp_mlp();
    m->ctx = ctx;
    m->in = in; m->h1 = h1; m->h2 = h2; m->out = out;
    const int sizes[6] = {h1 * in, h1, h2 * h1, h2, out * h2, out};
    for (int i = 0; i < 6; i++) { m->off[i] = m->np; m->np += sizes[i]; }
    if (mlp_alloc(&m->p, m->np) || mlp_alloc(&m->g, m->np) || mlp_alloc(&m->m, m->np) || mlp_alloc(&m->v, m->np) ||
        hipMalloc((void **)&m->pb, (size_t)m->np * 2) != hipSuccess) {
        sp_mlp_destroy(m);
        return SP_ERR_NOMEM;
    }
    // He-uniform initialisation from the project PRNG, zero biases
    std::vector<float> h(m->np, 0.f);
    sp_rng r;
    sp_rng_seed(&r, seed);
    const int fan[3] = {in, h1, h2};
    for (int l = 0; l < 3; l++) {
        const float lim = sqrtf(6.f / (float)fan[l]);
        for (int i = 0; i < sizes[2 * l]; i++) h[m->off[2 * l] + i] = (float)((2.0 * sp_rng_uniform(&r) - 1.0) * lim);
    }
    int rc = sp_mlp_set_params(m, h.data(), (size_t)m->np);
    if (!rc) {
        (void)hipMemset(m->m, 0, (size_t)m->np * 4);
        (void)hipMemset(m->v, 0, (size_t)m->np * 4);
    }
    if (rc) { sp_mlp_destroy(m); return rc; }
    *res = m;
    return SP_OK;
}

extern "C" int sp_mlp_destroy(sp_mlp *m) {
    if (!m) return SP_ERR_ARG;
    float *bufs[] = {m->p, m->g, m->m, m->v, m->x, m->a1, m->z1, m->a2, m->z2, m->y, m->t, m->msk, m->d3, m->d2, m->d1, m->part, m->l};
    for (float *b : bufs)
        if (b) (void)hipFree(b);
    for (float *b : {m->hx, m->hg})
        if (b) (void)hipHostFree(b);
    if (m->pb) (void)hipFree(m->pb);
    delete m;
    return SP_OK;
}

extern "C" size_t sp_mlp_num_params(const sp_mlp *m) { return m ? (size_t)m->np : 0; }

extern "C" int sp_mlp_set_params(sp_mlp *m, const float *host, size_t n) {
    if (!m || !host || n != (size_t)m->np) return SP_ERR_ARG;
    SP_HIP_TRY(hipMemcpy(m->p, host, n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(to_bf16, dim3((m->np + 255) / 256), dim3(256), 0, m->ctx->stream, m->p, m->pb, m->np);
    SP_HIP_TRY(hipStreamSynchronize(m->ctx->stream));
    m->step = 0;
    return SP_OK;
}

extern "C" int sp_mlp_get_params(sp_mlp *m, float *host, size_t n) {
    if (!m || !host || n != (size_t)m->np) return SP_ERR_ARG;
    SP_HIP_TRY(hipStreamSynchronize(m->ctx->stream));
    SP_HIP_TRY(hipMemcpy(host, m->p, n * 4, hipMemcpyDeviceToHost));
    return SP_OK;
}

static int forward_dev(sp_mlp *m, int B) {
    hipStream_t s = m->ctx->stream;
    const dim3 blk(TB * TB);
    auto grid = [&](int O) { return dim3((O + TB - 1) / TB, (B + TB - 1) / TB); };
    hipLaunchKernelGGL(dense_fwd, grid(m->h1), blk, 0, s, m->x, m->pb + m->off[0], m->p + m->off[1], m->z1, m->a1, B, m->in, m->h1, 1);
    hipLaunchKernelGGL(dense_fwd, grid(m->h2), blk, 0, s, m->a1, m->pb + m->off[2], m->p + m->off[3], m->z2, m->a2, B, m->h1, m->h2, 1);
    hipLaunchKernelGGL(dense_fwd, grid(m->out), blk, 0, s, m->a2, m->pb + m->off[4], m->p + m->off[5], (float *)nullptr, m->y, B, m->h2, m->out, 0);
    return hipGetLastError() == hipSuccess ? SP_OK : SP_ERR_HIP;
}

extern "C" int sp_mlp_predict(sp_mlp *m, const float *X, int B, float *Y) {
    if (!m || !X || !Y || B <= 0) return SP_ERR_ARG;
    int rc = mlp_reserve(m, B);
    if (rc) return rc;
    SP_HIP_TRY(hipMemcpyAsync(m->x, X, (size_t)B * m->in * 4, hipMemcpyHostToDevice, m->ctx->stream));
    if ((rc = forward_dev(m, B))) return rc;
    SP_HIP_TRY(hipMemcpyAsync(Y, m->y, (size_t)B * m->out * 4, hipMemcpyDeviceToHost, m->ctx->stream));
    SP_HIP_TRY(hipStreamSynchronize(m->ctx->stream));
    return SP_OK;
}

static float mean_loss(const float *part, int nb, int ny) {
    double l = 0;
    for (int i = 0; i < nb; i++) l += part[i];
    return (float)(l / ny);
}

// Loss and gradient of the batch at x, t, msk (device or pinned host memory; msk may be null) in
// two kernels; waits for them.  The gradient stays in m->g and is copied to `grad` if given.
static int loss_grad_two(sp_mlp *m, int B, const float *x, const float *t, const float *msk, float *loss, float *grad) {
    if (int rc = mlp_pin_out(m, B)) return rc;
    hipStream_t s = m->ctx->stream;
    const int ny = B * m->out, nb = (ny + 255) / 256;
    MlpArgs a{B, m->in, m->h1, m->h2, m->out, x, t, msk, m->p, m->pb, {}, x == m->x ? nullptr : m->x, m->a1, m->a2,
              m->d1, m->d2, m->d3, m->l, m->g, grad ? m->hg : nullptr, m->hg + m->np, 1.f / (float)ny};
    for (int i = 0; i < 6; i++) a.off[i] = m->off[i];
    const int tiles = weight_tiles(m->in, m->h1) + weight_tiles(m->h1, m->h2) + weight_tiles(m->h2, m->out);
    hipLaunchKernelGGL(mlp_sample, dim3((B + ROWS - 1) / ROWS), dim3(ROWS * SPT), 0, s, a);
    hipLaunchKernelGGL(mlp_weights, dim3(tiles + nb), dim3(256), 0, s, a, (const float *)m->x);
    if (hipGetLastError() != hipSuccess) return SP_ERR_HIP;
    SP_HIP_TRY(hipStreamSynchronize(s));
    if (loss) *loss = mean_loss(m->hg + m->np, nb, ny);
    if (grad) memcpy(grad, m->hg, (size_t)m->np * 4);
    return SP_OK;
}

// Forward + masked-MSE backward for one batch already in m->x / m->t / m->msk.
static int loss_grad_dev(sp_mlp *m, int B, float *loss) {
    if (m->two()) return loss_grad_two(m, B, m->x, m->t, m->msk, loss, nullptr);
    hipStream_t s = m->ctx->stream;
    int rc = forward_dev(m, B);
    if (rc) return rc;
    const int ny = B * m->out, nb = (ny + 255) / 256;
    hipLaunchKernelGGL(mse_grad, dim3(nb), dim3(256), 0, s, m->y, m->t, m->msk, m->d3, m->part, ny, 1.f / (float)ny);
    // layer 3
    hipLaunchKernelGGL(dense_bwd_w, dim3((m->h2 + 1 + 63) / 64, m->out), dim3(64), 0, s, m->d3, m->a2, m->g + m->off[4], m->g + m->off[5], B, m->h2, m->out);
    hipLaunchKernelGGL(dense_bwd_x, dim3((m->h2 + 63) / 64, B), dim3(64), 0, s, m->d3, m->pb + m->off[4], m->d2, B, m->h2, m->out);
    hipLaunchKernelGGL(relu_bwd, dim3((B * m->h2 + 255) / 256), dim3(256), 0, s, m->d2, m->z2, B * m->h2);
    // layer 2
    hipLaunchKernelGGL(dense_bwd_w, dim3((m->h1 + 1 + 63) / 64, m->h2), dim3(64), 0, s, m->d2, m->a1, m->g + m->off[2], m->g + m->off[3], B, m->h1, m->h2);
    hipLaunchKernelGGL(dense_bwd_x, dim3((m->h1 + 63) / 64, B), dim3(64), 0, s, m->d2, m->pb + m->off[2], m->d1, B, m->h1, m->h2);
    hipLaunchKernelGGL(relu_bwd, dim3((B * m->h1 + 255) / 256), dim3(256), 0, s, m->d1, m->z1, B * m->h1);
    // layer 1
    hipLaunchKernelGGL(dense_bwd_w, dim3((m->in + 1 + 63) / 64, m->h1), dim3(64), 0, s, m->d1, m->x, m->g + m->off[0], m->g + m->off[1], B, m->in, m->h1);
    if (hipGetLastError() != hipSuccess) return SP_ERR_HIP;
    if (loss) {
        std::vector<float> part(nb);
        SP_HIP_TRY(hipMemcpyAsync(part.data(), m->part, (size_t)nb * 4, hipMemcpyDeviceToHost, s));
        SP_HIP_TRY(hipStreamSynchronize(s));
        *loss = mean_loss(part.data(), nb, ny);
    }
    return SP_OK;
}

extern "C" int sp_mlp_loss_grad(sp_mlp *m, const float *X, const float *T, const float *M, int B, float *loss,
                                float *grad) {
    if (!m || !X || !T || B <= 0) return SP_ERR_ARG;
    int rc = mlp_reserve(m, B);
    if (rc) return rc;
    hipStream_t s = m->ctx->stream;
    if (m->two()) {  // the kernels read the batch from pinned memory (every call ends with a wait)
        if ((rc = mlp_pin_in(m, B))) return rc;
        float *const hx = m->hx, *const ht = hx + (size_t)B * m->in, *const hm = ht + (size_t)B * m->out;
        memcpy(hx, X, (size_t)B * m->in * 4);
        memcpy(ht, T, (size_t)B * m->out * 4);
        if (M) memcpy(hm, M, (size_t)B * m->out * 4);
        return loss_grad_two(m, B, hx, ht, M ? hm : nullptr, loss, grad);
    }
    SP_HIP_TRY(hipMemcpyAsync(m->x, X, (size_t)B * m->in * 4, hipMemcpyHostToDevice, s));
    SP_HIP_TRY(hipMemcpyAsync(m->t, T, (size_t)B * m->out * 4, hipMemcpyHostToDevice, s));
    if (M) SP_HIP_TRY(hipMemcpyAsync(m->msk, M, (size_t)B * m->out * 4, hipMemcpyHostToDevice, s));
    else {
        std::vector<float> ones((size_t)B * m->out, 1.f);
        SP_HIP_TRY(hipMemcpyAsync(m->msk, ones.data(), ones.size() * 4, hipMemcpyHostToDevice, s));
        SP_HIP_TRY(hipStreamSynchronize(s));
    }
    if ((rc = loss_grad_dev(m, B, loss))) return rc;
    if (grad) {
        SP_HIP_TRY(hipMemcpyAsync(grad, m->g, (size_t)m->np * 4, hipMemcpyDeviceToHost, s));
        SP_HIP_TRY(hipStreamSynchronize(s));
    }
    return SP_OK;
}

extern "C" int sp_mlp_adam(sp_mlp *m, float lr, float b1, float b2, float eps) {
    if (!m) return SP_ERR_ARG;
    m->step++;
    const float c1 = 1.f - powf(b1, (float)m->step), c2 = 1.f - powf(b2, (float)m->step);
    hipLaunchKernelGGL(adam_step, dim3((m->np + 255) / 256), dim3(256), 0, m->ctx->stream, m->p, m->g, m->m, m->v, m->pb,
                       m->np, lr, b1, b2, eps, c1, c2);
    return hipGetLastError() == hipSuccess ? SP_OK : SP_ERR_HIP;
}

// Mini-batch Adam over n samples for `epochs`, shuffled with the project
// PRNG; returns the mean loss of the last epoch.
extern "C" int sp_mlp_train(sp_mlp *m, const float *X, const float *T, const float *M, int n, int epochs,
                            int batch, float lr, uint64_t seed, float *final_loss) {
    if (!m || !X || !T || n <= 0 || epochs <= 0 || batch <= 0) return SP_ERR_ARG;
    const int B = batch < n ? batch : n;
    int rc = mlp_reserve(m, B);
    if (rc) return rc;
    std::vector<int> order(n);
    for (int i = 0; i < n; i++) order[i] = i;
    std::vector<float> bx((size_t)B * m->in), bt((size_t)B * m->out), bm((size_t)B * m->out);
    sp_rng r;
    sp_rng_seed(&r, seed);
    hipStream_t s = m->ctx->stream;
    double last = 0;
    for (int e = 0; e < epochs; e++) {
        for (int i = n - 1; i > 0; i--) {
            const int j = (int)(((__uint128_t)sp_rng_next(&r) * (uint64_t)(i + 1)) >> 64);
            std::swap(order[i], order[j]);
        }
        double tot = 0;
        int nbatch = 0;
        for (int s0 = 0; s0 + B <= n; s0 += B) {
            for (int q = 0; q < B; q++) {
                const int src = order[s0 + q];
                memcpy(&bx[(size_t)q * m->in], X + (size_t)src * m->in, (size_t)m->in * 4);
                memcpy(&bt[(size_t)q * m->out], T + (size_t)src * m->out, (size_t)m->out * 4);
                if (M) memcpy(&bm[(size_t)q * m->out], M + (size_t)src * m->out, (size_t)m->out * 4);
                else for (int o = 0; o < m->out; o++) bm[(size_t)q * m->out + o] = 1.f;
            }
            SP_HIP_TRY(hipMemcpyAsync(m->x, bx.data(), bx.size() * 4, hipMemcpyHostToDevice, s));
            SP_HIP_TRY(hipMemcpyAsync(m->t, bt.data(), bt.size() * 4, hipMemcpyHostToDevice, s));
            SP_HIP_TRY(hipMemcpyAsync(m->msk, bm.data(), bm.size() * 4, hipMemcpyHostToDevice, s));
            float l = 0;
            if ((rc = loss_grad_dev(m, B, &l))) return rc;
            if ((rc = sp_mlp_adam(m, lr, 0.9f, 0.999f, 1e-8f))) return rc;
            tot += l;
            nbatch++;
        }
        last = nbatch ? tot / nbatch : 0;
    }
    SP_HIP_TRY(hipStreamSynchronize(s));
    if (final_loss) *final_loss = (float)last;
    return SP_OK;
}
