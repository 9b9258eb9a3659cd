// Conjugate gradient on a plan's matrix: the iterative-solver caller that
// reuses one plan (and its tuned kernel) for every iteration.  Dot products
// reduce in a fixed order (per-block partial sums, then their sum, which every
// block of the next kernel forms for itself), so iterates are run-to-run
// identical.  The scalars stay on the device and the device stops the solve:
// an iteration is the SpMV and three kernels, without a synchronisation.  No
// counterpart in the reference.
#include <math.h>

#include "plan.hpp"

namespace {

constexpr int RB = 256;      // reduction block
constexpr int RGRID = 1024;  // partial sums per dot product
constexpr int AHEAD = 2;     // iterations queued beyond the last one known to be done

// What the kernels of a solve share.  The kernels of iteration it read slot it % 2 of rr and stop;
// cg_turn, the last of them, writes the other slot.  So no thread reads a word that the same kernel
// writes, and all threads of a kernel take the same side of a test of stop (barriers lie behind it).
struct CgState {
    double rr[2];  // r.r at the start of iteration it
    double bb, pq;
    int stop[2];   // at the start of iteration it: 0 running, 1 ended (converged or maxit), 2 not positive definite
};

// Where the host reads a solve's progress while it runs (pinned host memory).
struct CgNote {
    int it, stop;
    double rr, bb;
};

// Sum over the block's RB threads, as a tree of halves (the same pairs whatever the width of a
// step: two through LDS, the rest inside the first wave), handed to every thread.
__device__ __forceinline__ double block_sum(double acc, double *s) {
    const int t = threadIdx.x;
    s[t] = acc;
    __syncthreads();
    if (t < 128) s[t] += s[t + 128];
    __syncthreads();
    if (t < 64) {
        double v = s[t] + s[t + 64];
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w, 64);
        if (t == 0) s[0] = v;
    }
    __syncthreads();
    const double v = s[0];
    __syncthreads();  // s may be used again
    return v;
}

// The RGRID partial sums of a dot product, added by every block for itself: 8 KB from the L2 in
// place of a launch of its own.
__device__ __forceinline__ double sum_partials(const double *__restrict__ part, double *s) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < RGRID; i += RB) acc += part[i];
    return block_sum(acc, s);
}

__device__ __forceinline__ void tell(CgNote *note, int it, int stop, double rr, double bb) {
    note->rr = rr;
    note->bb = bb;
    __hip_atomic_store(&note->stop, stop, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&note->it, it, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ bool converged(double rr, double bb, double rtol) {
    const double bn = bb > 0 ? sqrt(bb) : 1.0;
    return !(sqrt(rr) / bn > rtol);
}

// r = b - r (r holds A x on entry); p = r; partial sums of b.b and r.r
template <typename T>
__global__ __launch_bounds__(RB) void cg_start(const T *__restrict__ b, T *__restrict__ r, T *__restrict__ p, uint64_t n,
                                               double *__restrict__ part_b, double *__restrict__ part_r) {
    __shared__ double s[RB];
    double sb = 0.0, sr = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * RB) {
        const T w = b[i], v = w - r[i];
        r[i] = v;
        p[i] = v;
        sb += (double)w * (double)w;
        sr += (double)v * (double)v;
    }
    sb = block_sum(sb, s);
    sr = block_sum(sr, s);
    if (threadIdx.x == 0) {
        part_b[blockIdx.x] = sb;
        part_r[blockIdx.x] = sr;
    }
}

__global__ __launch_bounds__(RB) void cg_begin(const double *__restrict__ part_b, const double *__restrict__ part_r,
                                               CgState *__restrict__ st, CgNote *__restrict__ note, double rtol,
                                               int maxit) {
    __shared__ double s[RB];
    const double bb = sum_partials(part_b, s), rr = sum_partials(part_r, s);
    if (threadIdx.x == 0) {
        st->bb = bb;
        st->rr[0] = rr;
        const int stop = maxit <= 0 || converged(rr, bb, rtol);
        st->stop[0] = stop;
        tell(note, 0, stop, rr, bb);
    }
}

// partial sums of p.q
template <typename T>
__global__ __launch_bounds__(RB) void cg_dot(const T *__restrict__ a, const T *__restrict__ b, uint64_t n,
                                             double *__restrict__ part, const CgState *__restrict__ st, int it) {
    __shared__ double s[RB];
    if (st->stop[it & 1]) return;
    double acc = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * RB)
        acc += (double)a[i] * (double)b[i];
    acc = block_sum(acc, s);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// alpha = r.r / p.q; x += alpha p; r -= alpha q; partial sums of the new r.r
template <typename T>
__global__ __launch_bounds__(RB) void cg_step(T *__restrict__ x, T *__restrict__ r, const T *__restrict__ p,
                                              const T *__restrict__ q, uint64_t n, const double *__restrict__ part_pq,
                                              double *__restrict__ part_r, CgState *__restrict__ st, int it) {
    __shared__ double s[RB];
    if (st->stop[it & 1]) return;
    const double pq = sum_partials(part_pq, s);
    if (blockIdx.x == 0 && threadIdx.x == 0) st->pq = pq;  // (read by cg_turn)
    if (!(pq > 0)) return;  // not positive definite: cg_turn stops the solve
    const T alpha = (T)(st->rr[it & 1] / pq);
    double acc = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * RB) {
        x[i] = x[i] + alpha * p[i];
        const T v = r[i] - alpha * q[i];
        r[i] = v;
        acc += (double)v * (double)v;
    }
    acc = block_sum(acc, s);
    if (threadIdx.x == 0) part_r[blockIdx.x] = acc;
}

// beta = new r.r / old r.r; p = r + beta p; block 0 counts the iteration and hands the state on to
// the next one's slot, also when the solve has stopped.
template <typename T>
__global__ __launch_bounds__(RB) void cg_turn(T *__restrict__ p, const T *__restrict__ r, uint64_t n,
                                              const double *__restrict__ part_r, CgState *__restrict__ st,
                                              CgNote *__restrict__ note, double rtol, int it, int maxit) {
    __shared__ double s[RB];
    const int ended = st->stop[it & 1];
    int *const next = &st->stop[(it + 1) & 1];
    if (ended) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *next = ended;
        return;
    }
    const double pq = st->pq, rr = st->rr[it & 1];
    if (!(pq > 0)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *next = 2;
            tell(note, it, 2, rr, st->bb);
        }
        return;
    }
    const double rr1 = sum_partials(part_r, s);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const double bb = st->bb;
        const int stop = it + 1 >= maxit || converged(rr1, bb, rtol);
        st->rr[(it + 1) & 1] = rr1;
        *next = stop;
        tell(note, it + 1, stop, rr1, bb);
    }
    const T beta = (T)(rr1 / rr);
    for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * RB)
        p[i] = r[i] + beta * p[i];
}

// Waits until the solve has done `want` iterations or stopped; false when the stream failed or
// ran out of work first.
bool await_note(CgNote *note, int want, hipStream_t s) {
    for (uint32_t spin = 1;; spin++) {
        if (__atomic_load_n(&note->it, __ATOMIC_ACQUIRE) >= want || __atomic_load_n(&note->stop, __ATOMIC_ACQUIRE))
            return true;
        if (spin % 4096 == 0 && hipStreamQuery(s) != hipErrorNotReady)
            return __atomic_load_n(&note->it, __ATOMIC_ACQUIRE) >= want || __atomic_load_n(&note->stop, __ATOMIC_ACQUIRE);
    }
}

template <typename T>
int cg_t(sp_plan *A, const T *b, T *x, int maxit, double rtol, int *iters, double *relres) {
    hipStream_t s = A->ctx->stream;
    const uint64_t n = A->nrows, vec = (n * sizeof(T) + 255) / 256 * 256;
    // r, p, q, three arrays of partial sums and the state.  The plan keeps them for its next
    // solve; a solve that finds them in use, or a plan with a memory cap, takes its own.
    const uint64_t bytes = 3 * vec + 3 * RGRID * sizeof(double) + 256;
    CgBuf own, *buf = &own;
    const bool kept = !A->opts.mem_cap_bytes && !A->cg_busy.exchange(true);
    if (kept) buf = &A->cg;
    auto done = [&](int rc) {
        if (kept) A->cg_busy.store(false);
        else own.release();
        return rc;
    };
    if (!buf->dev && (hipMalloc(&buf->dev, bytes) != hipSuccess ||
                      hipHostMalloc(&buf->note, sizeof(CgNote)) != hipSuccess)) {
        (void)hipGetLastError();  // reported here
        buf->release();
        return done(SP_ERR_NOMEM);
    }
    if (kept) A->cg_bytes.store(bytes);
    char *d = (char *)buf->dev;
    T *r = (T *)d, *p = (T *)(d + vec), *q = (T *)(d + 2 * vec);
    double *part_pq = (double *)(d + 3 * vec), *part_r = part_pq + RGRID, *part_b = part_r + RGRID;
    CgState *st = (CgState *)(part_b + RGRID);
    CgNote *note = (CgNote *)buf->note;
    note->it = -1;
    note->stop = 0;
    note->rr = note->bb = 0;
    const dim3 g(RGRID), t(RB);
    int rc = sp_spmv(A, x, r);
    if (!rc) {
        hipLaunchKernelGGL(cg_start<T>, g, t, 0, s, b, r, p, n, part_b, part_r);
        hipLaunchKernelGGL(cg_begin, dim3(1), t, 0, s, part_b, part_r, st, note, rtol, maxit);
        if (hipGetLastError() != hipSuccess) rc = SP_ERR_HIP;
    }
    // The host stays AHEAD iterations in front of the device, which decides by itself when to
    // stop: what is queued behind the last iteration only multiplies p once more.
    for (int it = 0; it < maxit && !rc; it++) {
        if (it >= AHEAD && !await_note(note, it - AHEAD, s)) { rc = SP_ERR_HIP; break; }
        if (__atomic_load_n(&note->stop, __ATOMIC_ACQUIRE)) break;
        if ((rc = sp_spmv(A, p, q))) break;
        hipLaunchKernelGGL(cg_dot<T>, g, t, 0, s, p, q, n, part_pq, st, it);
        hipLaunchKernelGGL(cg_step<T>, g, t, 0, s, x, r, p, q, n, part_pq, part_r, st, it);
        hipLaunchKernelGGL(cg_turn<T>, g, t, 0, s, p, r, n, part_r, st, note, rtol, it, maxit);
        if (hipGetLastError() != hipSuccess) rc = SP_ERR_HIP;
    }
    if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = SP_ERR_HIP;
    const int it = note->it > 0 ? note->it : 0;
    if (!rc && note->stop == 2) rc = SP_ERR_STATE;
    if (relres && note->it >= 0) *relres = sqrt(note->rr) / (note->bb > 0 ? sqrt(note->bb) : 1.0);
    if (iters) *iters = it;
    return done(rc);
}

}  // namespace

extern "C" int sp_cg(sp_plan *A, const void *b, void *x, int maxit, double rtol, int *iters, double *relres) {
    if (!A || !b || !x || maxit < 0 || !(rtol >= 0)) return SP_ERR_ARG;
    if (A->nrows != A->ncols) return SP_ERR_ARG;
    (void)hipSetDevice(A->ctx->device);
    switch (A->dtype) {
    case SP_F32: return cg_t<float>(A, (const float *)b, (float *)x, maxit, rtol, iters, relres);
    case SP_F64: return cg_t<double>(A, (const double *)b, (double *)x, maxit, rtol, iters, relres);
    default: return SP_ERR_UNSUPPORTED;
    }
}
