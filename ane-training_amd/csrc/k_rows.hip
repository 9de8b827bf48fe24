/*
 * k_rows.hip — the projections of up to 64 rows (decode batches above 4, short
 * prompts) with their norm, rotation, residual and gate in one launch each
 * (gfx950, v_mfma_f32_16x16x32_f16, fp32 accumulation).
 *
 *   k_rows<QKV>   xn = rmsnorm(x) * gain (layer 0: of the embedding rows, which
 *                 become x); [Wq; Wk; Wv] xn; RoPE; q to memory, k and v to the
 *                 cache                       (forward.h:46-53, 55-70, 108-128)
 *   k_rows<RES>   x += W a                    (Wo, W2; forward.h:134-136, 157-159)
 *   k_rows<GATE>  xn = rmsnorm(x) * gain; g = silu(W1 xn) * (W3 xn)
 *                                             (forward.h:46-53, 139-151)
 *
 * Bound by latency, not by bytes: a layer of Stories holds 14 MB of weights and
 * each of these launches 1-6 MB, a few microseconds' worth even from HBM, while
 * a launch of any size takes about 3.  So the row norms and the partials of
 * K-split GEMMs go: five launches a layer instead of seven.  A work-group takes
 * 16 rows and 16-64 columns; its KW waves each own a K chunk of both.  The rows
 * are loaded whole (a wave two rows, full lines), normalised and rounded once
 * into LDS; the weights go from memory straight into MFMA fragments, in flight
 * while the norm runs; the KW partial tiles meet in LDS, in wave order.
 *
 * Per launch alone, replayed from a graph over 24 layers' weights (us; before:
 * the row norm's launch and the K-split or K-grouped tiled GEMM):
 *   Stories, 64 rows   QKV 5.5 (3.2 + 4.6)  Wo 3.2 (4.1)  W1/W3 6.0 (3.2 + 5.7)
 *                      W2 4.8 (4.7); the attention after it 10.0-11.5 (12.7),
 *                      with whole q rows to read instead of partials to add
 *   Stories, 41 rows   QKV 4.8 (3.1 + 6.8)  Wo 3.2 (3.6)  W1/W3 5.9 (3.1 + 5.5)  W2 4.7 (4.2)
 * Rows read in fragment order instead (each load half of each of 16 lines):
 * QKV 6.6-9.7, W2 5.8.  Whole calls: a 41-token prompt 448 -> 368 us, a
 * 64-row decode step 517 -> 464 us (12 layers).
 *
 * MFMA lane layout: lane l holds A[l % 16][8 * (l / 16) .. +8] and
 * B[8 * (l / 16) .. +8][l % 16] (= W[n0 + l % 16][k ..]); accumulator element i
 * is C[4 * (l / 16) + i][l % 16].
 */
#include "k_common.h"
#include "lm_internal.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

enum { ROWS_QKV = 0, ROWS_RES = 1, ROWS_GATE = 2 };

struct RowsArgs {
    const u16 *W;           /* [N, K] fp16 */
    int M;
    float *x;               /* residual rows [M, D]: input of the norm, or += (RES) */
    int D;                  /* RES: row width of x */
    const u16 *a16;         /* RES: operand rows [M, K] fp16 */
    const float *gain;      /* QKV, GATE: norm gain [K] */
    const u16 *emb;         /* QKV: embedding [V, K] (layer 0) or NULL */
    const int *tok;
    u16 *g;                 /* GATE: [M, F] fp16 */
    int F;
    float *q;               /* QKV: [M, NQ] */
    void *kc, *vc;
    int kv_f32, NQ, NKV, hd, lghd, Hkv, max_seq;
    const int *slot, *pos;
    const float *rc, *rs;   /* RoPE tables */
};

/* A work-group: 16 rows (tile blockIdx.y) by NT tiles of 16 columns (GATE: NT/2
 * blocks of 16 W1 rows and their 16 W3 rows); KW waves, each K / KW of the sum. */
template <int K, int KW, int NT, int E>
__global__ void __launch_bounds__(64 * KW) k_rows(RowsArgs a)
{
    constexpr bool NORM = E != ROWS_RES;
    constexpr int KS = K / KW / 32;                     /* MFMA steps per wave */
    constexpr int NL = NT * 16 + 4;                     /* padded row of a partial tile */
    constexpr int PR = E == ROWS_GATE ? NT * 4 : NT * 8;   /* output pairs per row */
    constexpr int AL = K + 8;                           /* padded row of the normalised operand */
    constexpr int RW = 16 / KW, C4 = K / 256;           /* rows per wave, float4 groups per lane */
    static_assert(K % (KW * 32) == 0 && KS >= 1, "K chunks");
    static_assert(16 * PR <= 64 * KW, "an output item per thread");
    static_assert(RW >= 1 && 16 % KW == 0 && K % 256 == 0, "whole rows per wave");
    static_assert(E != ROWS_GATE || NT % 2 == 0, "W1 and W3 tiles");
    __shared__ __attribute__((aligned(16))) float red[KW][16][NL];
    __shared__ __attribute__((aligned(16))) u16 as[16 * AL];
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * NT * 16, m0 = blockIdx.y * 16;
    const int k0 = wv * (K / KW) + g * 8;

    /* this thread's output item: row ir, columns n, n + 1 (GATE: gates n/2 ..);
     * what it needs besides the product is loaded first */
    const int ir = tid / PR, p = tid % PR;
    const bool mine = tid < 16 * PR && m0 + ir < a.M;
    const int row = mine ? m0 + ir : 0;
    const int n = n0 + 2 * p;
    float2 xo = make_float2(0.f, 0.f);
    int ps = 0, sl = 0;
    float rcos = 1.f, rsin = 0.f;
    const bool isq = n < a.NQ, rot = n < a.NQ + a.NKV;
    const int nn = isq ? n : (rot ? n - a.NQ : n - a.NQ - a.NKV);
    if constexpr (E == ROWS_RES) xo = *(const float2 *)(a.x + (size_t)row * a.D + n);
    if constexpr (E == ROWS_QKV) {
        ps = a.pos[row];
        sl = a.slot[row];
    }

    f16x8 av[KS];
    uint4 w[KS][NT];
    auto load_w = [&]() {
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                w[s][j] = *(const uint4 *)(a.W + (size_t)(n0 + j * 16 + c16) * K + k0 + s * 32);
    };
    if constexpr (!NORM) {
        /* the operand rows through LDS as well: whole lines per load, where a
         * fragment's load takes half of each of 16 lines */
        constexpr int NC = RW * K / 512;      /* 16-byte chunks per lane */
        u32x4 t[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int ch = c * 64 + lane, r = wv * RW + ch / (K / 8);
            t[c] = *(const u32x4 *)(a.a16 + (size_t)min(m0 + r, a.M - 1) * K + ch % (K / 8) * 8);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_w();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int ch = c * 64 + lane, r = wv * RW + ch / (K / 8);
            *(u32x4 *)&as[r * AL + ch % (K / 8) * 8] = t[c];
        }
    } else {
        /* wave wv normalises rows wv * RW .. of the tile into LDS, a lane the
         * columns c*256 + 4*lane ..+3, as k_rownorm does */
        float4 xv[RW][C4], gv[C4];
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const int r = min(m0 + wv * RW + i, a.M - 1);
            if (E == ROWS_QKV && a.emb) {
                const u16 *er = a.emb + (size_t)a.tok[r] * K + 4 * lane;
#pragma unroll
                for (int c = 0; c < C4; c++) {
                    const uint2 h = *(const uint2 *)(er + c * 256);
                    const f16x2 u = __builtin_bit_cast(f16x2, h.x), v = __builtin_bit_cast(f16x2, h.y);
                    xv[i][c] = make_float4((float)u.x, (float)u.y, (float)v.x, (float)v.y);
                }
            } else {
                const float *xr = a.x + (size_t)r * K + 4 * lane;
#pragma unroll
                for (int c = 0; c < C4; c++) xv[i][c] = *(const float4 *)(xr + c * 256);
            }
        }
#pragma unroll
        for (int c = 0; c < C4; c++) gv[c] = *(const float4 *)(a.gain + 4 * lane + c * 256);
        /* the weights after the rows: loads retire in issue order, so the norm
         * runs while the weights are still arriving */
        __builtin_amdgcn_sched_barrier(0);
        load_w();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (E == ROWS_QKV) {
            if (rot) {
                const int ti = ps * (a.hd >> 1) + ((nn & (a.hd - 1)) >> 1);
                rcos = a.rc[ti];
                rsin = a.rs[ti];
            }
        }
#pragma unroll
        for (int i = 0; i < RW; i++) {
            float ss = 0.f;
#pragma unroll
            for (int c = 0; c < C4; c++) {
                ss = fmaf(xv[i][c].x, xv[i][c].x, ss); ss = fmaf(xv[i][c].y, xv[i][c].y, ss);
                ss = fmaf(xv[i][c].z, xv[i][c].z, ss); ss = fmaf(xv[i][c].w, xv[i][c].w, ss);
            }
            ss = wave_sum(ss);
            const float rs = 1.0f / sqrtf(ss / K + 1e-5f);
            const int r = wv * RW + i;
#pragma unroll
            for (int c = 0; c < C4; c++) {
                const float4 v = xv[i][c], q = gv[c];
                *(uint2 *)&as[r * AL + c * 256 + 4 * lane] =
                    make_uint2((unsigned)f2h(v.x * rs * q.x) | ((unsigned)f2h(v.y * rs * q.y) << 16),
                               (unsigned)f2h(v.z * rs * q.z) | ((unsigned)f2h(v.w * rs * q.w) << 16));
            }
            if (E == ROWS_QKV && a.emb && blockIdx.x == 0 && m0 + r < a.M) {
                float *xr = a.x + (size_t)(m0 + r) * K + 4 * lane;   /* layer 0: x takes the embedding rows */
#pragma unroll
                for (int c = 0; c < C4; c++) *(float4 *)(xr + c * 256) = xv[i][c];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; s++) av[s] = __builtin_bit_cast(f16x8, *(const uint4 *)&as[c16 * AL + k0 + s * 32]);

    f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = (f32x4){};
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int j = 0; j < NT; j++)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[s], __builtin_bit_cast(f16x8, w[s][j]), acc[j],
                                                            0, 0, 0);
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[wv][4 * g + i][j * 16 + c16] = acc[j][i];
    __syncthreads();
    if (!mine) return;
    /* (GATE: pair p of block b = p / 8 at columns 32b + 2(p % 8), its W3 16 on) */
    const int col = E == ROWS_GATE ? 32 * (p / 8) + 2 * (p % 8) : 2 * p;
    float2 v = make_float2(0.f, 0.f), v3 = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < KW; i++) {
        const float2 t = *(const float2 *)&red[i][ir][col];
        v.x += t.x;
        v.y += t.y;
        if constexpr (E == ROWS_GATE) {
            const float2 u = *(const float2 *)&red[i][ir][col + 16];
            v3.x += u.x;
            v3.y += u.y;
        }
    }
    if constexpr (E == ROWS_RES) {
        *(float2 *)(a.x + (size_t)row * a.D + n) = make_float2(xo.x + v.x, xo.y + v.y);
    } else if constexpr (E == ROWS_GATE) {
        /* sigmoid with the hardware exp2 and reciprocal, as the tiled GEMM's gate */
        const float s0 = v.x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-v.x * 1.4426950408889634f));
        const float s1 = v.y * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-v.y * 1.4426950408889634f));
        *(unsigned *)(a.g + (size_t)row * a.F + n0 / 2 + 2 * p) =
            (unsigned)f2h(s0 * v3.x) | ((unsigned)f2h(s1 * v3.y) << 16);
    } else {
        const int h = nn >> a.lghd, d = nn & (a.hd - 1);
        const float o0 = rot ? fmaf(v.x, rcos, -(v.y * rsin)) : v.x;   /* forward.h:64 */
        const float o1 = rot ? fmaf(v.x, rsin, v.y * rcos) : v.y;      /* forward.h:65 */
        if (isq) {
            *(float2 *)(a.q + (size_t)row * a.NQ + n) = make_float2(o0, o1);
        } else {
            const size_t off = (((size_t)sl * a.Hkv + h) * a.max_seq + ps) * a.hd + d;
            void *dst = rot ? a.kc : a.vc;
            if (a.kv_f32) *(float2 *)((float *)dst + off) = make_float2(o0, o1);
            else *(unsigned *)((u16 *)dst + off) = (unsigned)f2h(o0) | ((unsigned)f2h(o1) << 16);
        }
    }
}

/* ============================== launchers =================================== */

template <int K, int KW, int NT, int E>
static int launch_nt(hipStream_t s, const RowsArgs &a, int N)
{
    hipLaunchKernelGGL((k_rows<K, KW, NT, E>), dim3(N / (16 * NT), (a.M + 15) / 16), dim3(64 * KW), 0, s, a);
    return hipGetLastError();
}

/* Columns per work-group: the fewest that leave no CU more than one
 * work-group (a second one on a CU costs as much again: Stories QKV at 41
 * rows 5.5 us with 432 work-groups, 4.8 with 216; at 64 rows 6.7 with 576,
 * 6.6 with 288, 5.5 with 192), else the most. */
template <int K, int KW, int E>
static int launch_rows(hipStream_t s, const RowsArgs &a, int N)
{
    const int tiles = N / 16 * ((a.M + 15) / 16);
    if constexpr (E == ROWS_GATE) {
        return tiles <= 512 || N % 64 ? launch_nt<K, KW, 2, E>(s, a, N) : launch_nt<K, KW, 4, E>(s, a, N);
    } else if constexpr (E == ROWS_QKV) {
        if (tiles <= 256 || N % 32) return launch_nt<K, KW, 1, E>(s, a, N);
        if (tiles <= 512 || N % 48) return launch_nt<K, KW, 2, E>(s, a, N);
        return launch_nt<K, KW, 3, E>(s, a, N);
    } else {
        return launch_nt<K, KW, 1, E>(s, a, N);
    }
}

template <int E>
static int launch_rows_k(hipStream_t s, const RowsArgs &a, int N, int K)
{
    switch (K) {
    case 256: return launch_rows<256, 8, E>(s, a, N);
    case 512: return launch_rows<512, 8, E>(s, a, N);
    case 768: return launch_rows<768, 8, E>(s, a, N);
    case 1024: return launch_rows<1024, 8, E>(s, a, N);
    case 2048:
        if constexpr (E == ROWS_RES) return launch_rows<2048, 8, E>(s, a, N);
        return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
}

extern "C" int lmk_rows_qkv(hipStream_t s, float *x, const uint16_t *emb, const int *tok,
                            const float *gain, const uint16_t *wqkv, int D, int M, int NQ, int NKV,
                            int hd, const float *rope_cos, const float *rope_sin, const int *pos,
                            const int *slot, float *q, void *kc, void *vc, int kv_f32, int max_seq)
{
    if (M < 1 || M > 64 || !x || (emb && !tok) || !gain || !wqkv || !pos || !slot || !q || !kc || !vc ||
        (hd != 64 && hd != 128) || NQ % hd || NKV % hd || NKV < hd)
        return hipErrorInvalidValue;
    RowsArgs a = {};
    a.W = (const u16 *)wqkv; a.M = M; a.x = x; a.D = D; a.gain = gain; a.emb = (const u16 *)emb; a.tok = tok;
    a.q = q; a.kc = kc; a.vc = vc; a.kv_f32 = kv_f32; a.NQ = NQ; a.NKV = NKV; a.hd = hd;
    a.lghd = __builtin_ctz((unsigned)hd); a.Hkv = NKV / hd; a.max_seq = max_seq;
    a.slot = slot; a.pos = pos; a.rc = rope_cos; a.rs = rope_sin;
    return launch_rows_k<ROWS_QKV>(s, a, NQ + 2 * NKV, D);
}

extern "C" int lmk_rows_res(hipStream_t s, const uint16_t *a16, const uint16_t *W, int D, int K, int M,
                            float *x)
{
    if (M < 1 || M > 64 || D < 16 || D % 16 || !a16 || !W || !x) return hipErrorInvalidValue;
    RowsArgs a = {};
    a.W = (const u16 *)W; a.M = M; a.x = x; a.D = D; a.a16 = (const u16 *)a16;
    return launch_rows_k<ROWS_RES>(s, a, D, K);
}

extern "C" int lmk_rows_gate(hipStream_t s, const float *x, const float *gain, const uint16_t *w13,
                             int D, int F, int M, uint16_t *g)
{
    if (M < 1 || M > 64 || F < LMK_GATE_BLOCK || F % LMK_GATE_BLOCK || !x || !gain || !w13 || !g)
        return hipErrorInvalidValue;
    RowsArgs a = {};
    a.W = (const u16 *)w13; a.M = M; a.x = (float *)x; a.D = D; a.gain = gain; a.g = (u16 *)g; a.F = F;
    return launch_rows_k<ROWS_GATE>(s, a, 2 * F, D);
}
