/*
 * k_io.hip — the host boundary of a call as kernels of its own stream (gfx950):
 * inputs read from, and results written to, pinned host memory.
 *
 * A copy queued beside the step's graph is a submission and a blit launch of its
 * own, and the stream synchronise after it waits for an interrupt's worth of
 * host time.  Read and written by kernels inside the graph, with one flag word
 * per work-group that the host polls, a step of 13 launches whose call makes
 * two copies in and two out took 470 us instead of 500 in a model of it (22 us
 * less for the copies, 8 less for the wait).
 *
 * A work-group's stores to host memory have completed before its flag is
 * released at system scope, so a host that has seen the flag sees the data.
 */
#include "k_common.h"
#include "lm_internal.h"

#define IT 256

/* tokens and positions of B rows, and the call's number, from the call block */
__global__ void __launch_bounds__(IT) k_step_in(const int *__restrict__ call, int *__restrict__ seq,
                                               int *__restrict__ tok, int *__restrict__ pos, int B)
{
    const int t = threadIdx.x;
    if (t < B) {
        tok[t] = call[LM_CALL_TOK + t];
        pos[t] = call[LM_CALL_POS + t];
    }
    if (t == IT - 1) *seq = call[0];
}

__global__ void __launch_bounds__(IT) k_rows_in(const int *__restrict__ h, int *__restrict__ d, int n)
{
    const int i = blockIdx.x * IT + threadIdx.x;
    if (i < n) d[i] = h[i];
}

/* The call's number into this work-group's flag, once its stores have landed:
 * every wave waits for its own (to host memory, which the L2 does not hold),
 * then thread 0 releases at system scope.  One such release per work-group:
 * each is also an L2 write-back. */
__device__ __forceinline__ void raise_flag(int *flags, int seq)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(flags + (size_t)blockIdx.x * LM_FLAG_STRIDE, seq, __ATOMIC_RELEASE,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

/* n floats (src 16-byte aligned, or NULL with n 0) to dst, work-group w the
 * elements [w, w + 1) * LM_GIVE_PER(n, work-groups); work-group 0 also the hand-off flag, the
 * prefill overflow flag and B ids to the header. */
__global__ void __launch_bounds__(IT) k_give(const float *__restrict__ src, float *__restrict__ dst, size_t n,
                                            const int *__restrict__ err, const int *__restrict__ ovf,
                                            const int *__restrict__ tok, int B, int *__restrict__ hdr,
                                            const int *__restrict__ seqp, int seqv, int *flags)
{
    const size_t per = LM_GIVE_PER(n, gridDim.x), a = per * blockIdx.x;
    const size_t b = a + per < n ? a + per : n;
    if (a < b) {
        const size_t b4 = a + ((b - a) & ~(size_t)3);   /* (a is a multiple of 4) */
        for (size_t i = a + 4 * threadIdx.x; i < b4; i += 4 * IT)
            *(float4 *)(dst + i) = *(const float4 *)(src + i);
        if (threadIdx.x < b - b4) dst[b4 + threadIdx.x] = src[b4 + threadIdx.x];
    }
    if (blockIdx.x == 0) {
        if ((int)threadIdx.x < B) hdr[LM_HDR_TOK + threadIdx.x] = tok[threadIdx.x];
        if (threadIdx.x == 0) {
            if (err) hdr[LM_HDR_ERR] = *err;
            /* read back over the bus, behind the store that may have set it */
            if (ovf) hdr[LM_HDR_OVF] = *(const volatile int *)ovf;
        }
    }
    raise_flag(flags, seqp ? *seqp : seqv);
}

/* The ids of steps t0 .. t0+nt-1 of an n-step greedy run of B rows that has
 * ended (pos advanced by n): out[(t - t0)*B + b]; work-group w the elements
 * [w, w + 1) * LM_GIVE_PER of nt*B. */
__global__ void __launch_bounds__(IT) k_give_ids(const int *__restrict__ hist, int stride,
                                                const int *__restrict__ pos, int B, int n, int t0, int nt,
                                                int *__restrict__ out, const int *__restrict__ err,
                                                int *__restrict__ hdr, int seqv, int *flags)
{
    const size_t tot = (size_t)nt * B, per = LM_GIVE_PER(tot, gridDim.x), a = per * blockIdx.x;
    const size_t e = a + per < tot ? a + per : tot;
    for (size_t i = a + threadIdx.x; i < e; i += IT) {
        const int t = (int)(i / B), b = (int)(i - (size_t)t * B);
        out[i] = hist[(size_t)b * stride + pos[b] - n + 1 + t0 + t];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) hdr[LM_HDR_ERR] = *err;
    raise_flag(flags, seqv);
}

extern "C" int lmk_step_in(hipStream_t s, const int *call, int *seq, int *tok, int *pos, int B)
{
    if (B < 1 || B > LM_CALL_ROWS || !call || !seq || !tok || !pos) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_step_in, dim3(1), dim3(IT), 0, s, call, seq, tok, pos, B);
    return hipGetLastError();
}

extern "C" int lmk_rows_in(hipStream_t s, const int *h, int *d, int n)
{
    if (n < 1 || !h || !d) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_rows_in, dim3((n + IT - 1) / IT), dim3(IT), 0, s, h, d, n);
    return hipGetLastError();
}

extern "C" int lmk_give(hipStream_t s, const float *src, float *dst, size_t n, int wgs, const int *err,
                        const int *ovf, const int *tok, int B, int *hdr, const int *seqp, int seqv,
                        int *flags)
{
    if (wgs < 1 || wgs > LM_GIVE_WGS || (n && (!src || !dst)) || B < 0 || B > LM_CALL_ROWS || (B && !tok) ||
        !hdr || !flags)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_give, dim3(wgs), dim3(IT), 0, s, src, dst, n, err, ovf, tok, B, hdr, seqp, seqv, flags);
    return hipGetLastError();
}

extern "C" int lmk_give_ids(hipStream_t s, const int *hist, int stride, const int *pos, int B, int n, int t0,
                            int nt, int *out, int wgs, const int *err, int *hdr, int seqv, int *flags)
{
    if (wgs < 1 || wgs > LM_GIVE_WGS || B < 1 || nt < 1 || t0 < 0 || t0 + nt > n || !hist || !pos || !out ||
        !err || !hdr || !flags)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_give_ids, dim3(wgs), dim3(IT), 0, s, hist, stride, pos, B, n, t0, nt, out, err, hdr,
                       seqv, flags);
    return hipGetLastError();
}
