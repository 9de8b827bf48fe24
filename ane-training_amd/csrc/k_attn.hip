/*
 * k_attn.hip — causal prefill attention on MFMA (gfx950).
 *
 * Rows of a prefill chunk come in whole sequences of S consecutive rows with
 * consecutive positions.  Keys are visited in tiles of 64 positions, 0 ..
 * (last query position of the block); a wave owning 32 queries updates its
 * online softmax with each tile (forward.h:72-99, scores in log2 units):
 *   S^T = K Q^T * (log2 e / sqrt(hd))   32x32x16 f16 MFMAs, fp32 accumulation;
 *                                       keys after the query's position masked
 *   m' = max_key S if it exceeds m by more than 8, else m;
 *   P = 2^(S - m'); l = l*2^(m - m') + sum_key P;
 *   O^T = O^T*2^(m - m') + V^T P^T      P and V rounded to fp16 for the MFMA
 * and out = O / l, in fp16 (the operand of the Wo GEMM).  Any m' at or below
 * the true maximum gives the same O / l; keeping m unless it falls 8 behind
 * bounds P by 2^8 and skips the rescale of O on most tiles.  Only tiles that
 * hold a key after some query of the wave are masked.
 *
 * Computing the transposed scores puts one query in each accumulator column, so
 * lane l holds 32 of the tile's 64 scores of query l % 32 (lane l ^ 32 the other
 * 32): the softmax needs one cross-lane exchange per tile, and the accumulator
 * already has the layout of the B operand of the V^T P^T product, up to an order
 * of the 16 keys of each MFMA step.  That order is undone by storing V^T in LDS
 * with bits 2 and 3 of the key index swapped; V^T rows are XOR-swizzled in
 * 16-byte units so that neither the transposing writes nor the fragment reads
 * conflict in the LDS banks.
 *
 * Two kernels share that per-tile step:
 *   k_attn_prefill_blk    64 or 128 queries per work-group, 32 per wave; all
 *                         waves share each staged key tile, and where there are
 *                         more waves than query groups they take a step's tiles
 *                         in halves and merge at the end.  Least K/V traffic:
 *                         for many blocks.
 *   k_attn_prefill_split  32 queries per work-group; the four waves split the
 *                         key tiles round-robin, each staging its own, and merge
 *                         their (m, l, O) through LDS.  The last query block waits
 *                         for a quarter of its tiles: for few blocks (short
 *                         prompts), where the work-group count is the limit.
 */
#include "k_common.h"
#include "lm_internal.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));

#define AT 256          /* threads per work-group (4 waves) */
#define NW 4            /* waves per work-group */
#define BKV 64          /* keys per tile */

__device__ __forceinline__ f32x16 mfma32h(uint4 a, uint4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

/* 8 cache elements -> 8 fp16 */
__device__ __forceinline__ uint4 kv8_f16(const u16 *p) { return *(const uint4 *)p; }
__device__ __forceinline__ uint4 kv8_f16(const float *p)
{
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    f16x8 h;
    h[0] = (_Float16)a.x; h[1] = (_Float16)a.y; h[2] = (_Float16)a.z; h[3] = (_Float16)a.w;
    h[4] = (_Float16)b.x; h[5] = (_Float16)b.y; h[6] = (_Float16)b.z; h[7] = (_Float16)b.w;
    return __builtin_bit_cast(uint4, h);
}

/* LDS column of key k of a tile in V^T: bits 2 and 3 swapped, so that the 8 keys
 * lane l contributes to an MFMA step (4 from each of two groups of 8) are
 * contiguous.  The map is its own inverse. */
__device__ __forceinline__ int vperm(int k) { return (k & ~12) | ((k & 4) << 1) | ((k >> 1) & 4); }

/* V^T tile: row d (a head dim) holds the tile's BKV keys in vperm order as 16-byte
 * units; unit u of row d sits in slot u ^ vswz(d).  The 8 rows that one 16-byte
 * fragment read serves per LDS cycle (d .. d+7) and the 8 rows d0 + j, d0 = 0, 8,
 * .. 56 that one staging write serves then fall in 8 different slots: no bank
 * conflicts on either side. */
__device__ __forceinline__ int vswz(int d) { return (d ^ (d >> 3)) & 7; }
__device__ __forceinline__ int vt_off(int d, int col) { return d * BKV + (((col >> 3) ^ vswz(d)) << 3) + (col & 7); }

/* Staging unit `pr` (0 .. BKV/2 * HD/8 - 1) of a tile: dims d0 .. d0+7 of the keys
 * in V^T columns pk and pk+1 (keys vperm(pk), vperm(pk) + 1: pk is even and vperm
 * keeps bit 0).  Consecutive units take the 8 dim groups of one column pair, then
 * the next pair: one wave's 32-lane half covers 4 pairs of one 16-byte unit. */
template <int HD>
__device__ __forceinline__ void pair_of(int pr, int &pk, int &d0)
{
    pk = ((pr >> 3) & (BKV / 2 - 1)) * 2;
    d0 = ((pr & 7) + (pr / (BKV / 2 * 8)) * 8) * 8;
}

/* Store one staging unit: K rows of KLD halves (two 16-byte writes), V^T in the
 * swizzled layout (8 dword writes, each the two keys of one dim). */
template <int KLD>
__device__ __forceinline__ void stage_pair(u16 *sk, u16 *svt, int pk, int d0, uint4 ka, uint4 kb,
                                           uint4 va, uint4 vb)
{
    const int key = vperm(pk);
    *(uint4 *)(&sk[key * KLD + d0]) = ka;
    *(uint4 *)(&sk[(key + 1) * KLD + d0]) = kb;
    const unsigned wa[4] = {va.x, va.y, va.z, va.w}, wb[4] = {vb.x, vb.y, vb.z, vb.w};
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const unsigned a = wa[j >> 1], b = wb[j >> 1];
        const unsigned w = (j & 1) ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
        *(unsigned *)(&svt[vt_off(d0 + j, pk)]) = w;
    }
}

/* The running maximum m of a query is raised only when a tile's maximum exceeds
 * it by more than this (log2 units), so P = 2^(S - m) <= 2^8 stays well inside
 * fp16 and the rescale of O and l is skipped for most tiles. */
#define M_SLACK 8.0f

/* Online-softmax update of one wave's 32 queries (lane l: query l % 32 at
 * position qp) with the staged tile of keys k0 .. k0+63 (K rows, V^T).  MASK:
 * the tile holds keys after some query's position (wave-uniform choice). */
template <int HD, int KLD, bool MASK>
__device__ __forceinline__ void tile_update(const u16 *sk, const u16 *svt, const uint4 (&qb16)[HD / 16],
                                            int k0, int qp, float scale, f32x16 (&o)[HD / 32],
                                            float &mrow, float &lrow)
{
    constexpr int KS = HD / 16, DT = HD / 32;
    const int lane = threadIdx.x & 63, g = lane >> 5;
    /* S^T tiles: rows = keys nt*32 + (0..31), columns = the wave's queries */
    f32x16 sacc[2];
#pragma unroll
    for (int nt = 0; nt < 2; nt++) {
        sacc[nt] = (f32x16){};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const uint4 ka = *(const uint4 *)(&sk[(nt * 32 + (lane & 31)) * KLD + ks * 16 + g * 8]);
            sacc[nt] = mfma32h(ka, qb16[ks], sacc[nt]);
        }
    }
    /* element i of tile nt is key k0 + nt*32 + 8*(i/4) + 4*g + i%4; the maximum
     * is taken over the raw dot products (scale > 0) */
    float mx = -INFINITY;
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if constexpr (MASK) {
                const int key = k0 + nt * 32 + 8 * (i >> 2) + 4 * g + (i & 3);
                if (key > qp) sacc[nt][i] = -INFINITY;
            }
            mx = fmaxf(mx, sacc[nt][i]);
        }
    mx = fmaxf(mx, xor32_f(mx)) * scale;
    /* a query with every key so far masked keeps m = -inf (and O = l = 0), also
     * where another query of the wave raises its own */
    const bool raise = mx > mrow + M_SLACK;
    if (__builtin_amdgcn_ballot_w64(raise)) {     /* wave-uniform */
        const float mn = raise ? mx : mrow;
        const float corr = raise ? __builtin_amdgcn_exp2f(mrow - mn) : 1.f;   /* 0 from m = -inf */
        lrow *= corr;
#pragma unroll
        for (int j = 0; j < DT; j++) o[j] *= corr;
        mrow = mn;
    }
    const float sub = mrow == -INFINITY ? 0.f : mrow;
    float ls = 0.f;
    uint4 pb[2][2];
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            f16x8 hv;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float e = __builtin_amdgcn_exp2f(fmaf(sacc[nt][8 * hh + j], scale, -sub));
                ls += e;
                hv[j] = (_Float16)e;
            }
            pb[nt][hh] = __builtin_bit_cast(uint4, hv);
        }
    lrow += ls;                                /* per-lane partial row sum */
    /* O^T += V^T P^T over the 4 steps of 16 keys */
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int hh = 0; hh < 2; hh++)
#pragma unroll
            for (int j = 0; j < DT; j++) {
                const uint4 va = *(const uint4 *)(&svt[vt_off(j * 32 + (lane & 31), nt * 32 + hh * 16 + g * 8)]);
                o[j] = mfma32h(va, pb[nt][hh], o[j]);
            }
}

/* Q^T fragments (B operand) of a wave: query row `row` (fp32 q [rows, NQ]),
 * dims ks*16 + 8*(l/32) .. +8 of head h */
template <int HD>
__device__ __forceinline__ void load_q(const float *q, size_t row, int NQ, int h, uint4 (&qb16)[HD / 16])
{
    const float *qs = q + row * NQ + h * HD + ((threadIdx.x & 63) >> 5) * 8;
#pragma unroll
    for (int ks = 0; ks < HD / 16; ks++) qb16[ks] = kv8_f16(qs + ks * 16);
}

/* Head, sequence and query block of work-group id of nqb * nseq * H.  It runs
 * on XCD id % 8: heads fastest, neighbouring heads (one kv head's) on one XCD
 * where the count allows, so that an XCD's L2 holds the K and V of few heads;
 * a prompt's longest blocks first, so that the short ones fill the end. */
__device__ __forceinline__ void block_of(int id, int nqb, int nseq, int H, int &h, int &seq, int &qb)
{
    const int bi = small_div(id, H), hi = id - bi * H;
    h = H % 8 == 0 ? (hi & 7) * (H >> 3) + (hi >> 3) : hi;
    const int qr = small_div(bi, nseq);
    seq = bi - qr * nseq;
    qb = nqb - 1 - qr;
}

/* ---- 64- and 128-query blocks, shared tiles --------------------------------- */

/* W waves, QG of them along the block's queries (32 each), KG = W / QG along its
 * keys: a step stages KG consecutive key tiles, wave (qg, kg) takes tile kg of
 * them for the 32 queries of group qg, and with KG = 2 the two halves'
 * (m, l, O) meet in LDS at the end.  What bounds it is the longest chain of
 * dependent tiles and each tile's latency (MFMA, exp2, MFMA, barrier): the last
 * block of a prompt walks all its key tiles.  One 1900-token prompt in
 * 128-query blocks has fewer work-groups than CUs and lasts as long as 30
 * tiles in turn; KG 2 halves the chain.  us per launch at 1900: hd 128, 16
 * heads, four waves of 128 queries 70, eight waves KG 2 53; hd 64, 12 heads, 35.5
 * against 25.8 with 64-query blocks KG 2. */
template <int HD, typename KT, int QG, int W>
__global__ void __launch_bounds__(64 * W, W == 8 || QG == 2 ? 2 : 1) k_attn_prefill_blk(
    const float *__restrict__ q, const KT *__restrict__ kc, const KT *__restrict__ vc,
    const int *__restrict__ pos, const int *__restrict__ slot, int S, int nseq, int nqb, int H, int Hkv,
    int max_seq, u16 *__restrict__ out)
{
    constexpr int KG = W / QG, BQ = 32 * QG, NT = 64 * W;
    constexpr int KLD = HD + 8;          /* K tile row stride (halves)   */
    constexpr int DT = HD / 32;          /* 32-dim row tiles of O^T      */
    constexpr int UPT = BKV * HD / 16, PPT = KG * UPT / NT;   /* staging units per tile; per thread and step */
    constexpr int NB = 2;
    constexpr int TS = BKV * KLD + HD * BKV;      /* halves of one tile's K and V^T */
    constexpr int MLD = HD + 1;                   /* merge row stride (floats) */
    static_assert(PPT >= 1 && KG * UPT % NT == 0 && (UPT % NT == 0 || NT % UPT == 0), "staging shape");
    static_assert(KG == 1 || NB * KG * TS * 2 >= (QG * 32 * MLD + 2 * QG * 32) * 4, "merge area fits the staging area");
    __shared__ __attribute__((aligned(16))) u16 stg[NB][KG * TS];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qg = wave % QG, kg = wave / QG;
    int h, seq, qb;
    block_of(blockIdx.x, nqb, nseq, H, h, seq, qb);
    const int kvh = small_div(h, small_div(H, Hkv));
    const int NQ = H * HD;
    const int row0 = seq * S + qb * BQ;           /* first row of the block       */
    const int nrows = min(BQ, S - qb * BQ);       /* valid rows of the block      */
    const int p0 = pos[row0];                     /* position of the block's row 0 */
    const int cs = slot[row0];
    const size_t cbase = ((size_t)cs * Hkv + kvh) * max_seq * HD;
    /* scores are kept in log2 units: exp(x) = exp2(x * log2 e) */
    const float scale = 1.4426950408889634f / sqrtf((float)HD);
    const int last_pos = p0 + nrows - 1;          /* last query position of the block */
    const int nsteps = (last_pos / BKV + KG) / KG;

    /* K / V of one step: thread t stages units t + i*AT (two keys, 8 dims each:
     * [0] key, [1] key + 1; KG = 2: the first half of the units is tile 0's);
     * keys past the block's last position repeat it (they are masked for every
     * query that reads them).  Two register sets: step t sits in set t % 2 from
     * its fetch (two steps ahead of its use) until it is stored to LDS; one
     * set, one step ahead, at KG 2. */
    constexpr int NSET = KG == 1 ? 2 : 1;
    uint4 rk0[PPT][2], rv0[PPT][2], rk1[NSET == 2 ? PPT : 1][2], rv1[NSET == 2 ? PPT : 1][2];
    auto fetch = [&](int st, auto &rk, auto &rv) {
#pragma unroll
        for (int i = 0; i < PPT; i++) {
            int pk, d0;
            pair_of<HD>((tid + i * NT) % UPT, pk, d0);
            const int key = (st * KG + (tid + i * NT) / UPT) * BKV + vperm(pk);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const size_t off = cbase + (size_t)min(key + e, last_pos) * HD + d0;
                rk[i][e] = kv8_f16(kc + off);
                rv[i][e] = kv8_f16(vc + off);
            }
        }
    };
    auto stash = [&](int b, const auto &rk, const auto &rv) {
#pragma unroll
        for (int i = 0; i < PPT; i++) {
            int pk, d0;
            pair_of<HD>((tid + i * NT) % UPT, pk, d0);
            u16 *t = stg[b] + (tid + i * NT) / UPT * TS;
            stage_pair<KLD>(t, t + BKV * KLD, pk, d0, rk[i][0], rk[i][1], rv[i][0], rv[i][1]);
        }
    };
    fetch(0, rk0, rv0);
    if constexpr (NSET == 2) fetch(1, rk1, rv1);   /* past the last step: the last position again, unused */

    /* this wave's queries: block rows wr0 .. wr0+31; lane l takes row wr0 + l%32 */
    const int wr0 = qg * 32;
    const bool wave_active = wr0 < nrows;
    const int wave_first = p0 + wr0, wave_last = p0 + min(wr0 + 31, nrows - 1);
    const int qrow = wr0 + (lane & 31);
    const int qp = p0 + qrow;                     /* this lane's query position */
    uint4 qb16[HD / 16];
    load_q<HD>(q, (size_t)(row0 + min(qrow, nrows - 1)), NQ, h, qb16);
    f32x16 o[DT];
#pragma unroll
    for (int j = 0; j < DT; j++) o[j] = (f32x16){};
    float mrow = -INFINITY, lrow = 0.f;

    auto compute = [&](int st, int b) {
        const int k0 = (st * KG + kg) * BKV;
        const u16 *t = stg[b] + kg * TS;
        if (wave_active && k0 <= wave_last) {     /* wave-uniform */
            /* every key visible to every query (at hd 128 the two forms side by
             * side spill 60 registers, the masked one alone none) */
            if (HD == 64 && k0 + BKV - 1 <= wave_first)
                tile_update<HD, KLD, false>(t, t + BKV * KLD, qb16, k0, qp, scale, o, mrow, lrow);
            else
                tile_update<HD, KLD, true>(t, t + BKV * KLD, qb16, k0, qp, scale, o, mrow, lrow);
        }
    };
    stash(0, rk0, rv0);
    __syncthreads();
    if constexpr (NSET == 2) {
        /* step t: fetch step t+2 into the set step t left (unconditionally, so
         * the compiler waits only for the older set), compute t, store t+1 */
        auto body = [&](int st, auto &rka, auto &rva, const auto &rkb, const auto &rvb) {
            const int b = st & 1;
            fetch(st + 2, rka, rva);
            compute(st, b);
            if (st + 1 < nsteps) stash(b ^ 1, rkb, rvb);
            __syncthreads();
        };
        for (int st = 0; st < nsteps; st += 2) {
            body(st, rk0, rv0, rk1, rv1);
            if (st + 1 < nsteps) body(st + 1, rk1, rv1, rk0, rv0);
        }
    } else {
        for (int st = 0; st < nsteps; st++) {
            if (st + 1 < nsteps) fetch(st + 1, rk0, rv0);
            compute(st, st & 1);
            if (st + 1 < nsteps) stash((st + 1) & 1, rk0, rv0);
            __syncthreads();
        }
    }
    /* finish the row sum across the lane pair: element i of o[j] is dim
     * j*32 + 8*(i/4) + 4*g + i%4 of query l%32 */
    float l = lrow + xor32_f(lrow);
    if constexpr (KG == 2) {
        /* the upper key half's (m, l, O) through LDS (every wave is past its
         * last read of the staging area) */
        float *mo = (float *)&stg[0][0], *mm = mo + QG * 32 * MLD, *ml = mm + QG * 32;
        if (kg == 1) {
            if (g == 0) {
                mm[qrow] = mrow;
                ml[qrow] = l;
            }
#pragma unroll
            for (int j = 0; j < DT; j++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    mo[qrow * MLD + j * 32 + 8 * (i >> 2) + 4 * g + (i & 3)] = o[j][i];
        }
        __syncthreads();
        if (kg == 1) return;
        const float m1 = mm[qrow], M = fmaxf(mrow, m1);   /* (this half holds key 0: m is finite) */
        const float f0 = __builtin_amdgcn_exp2f(mrow - M);
        const float f1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - M);
        l = fmaf(ml[qrow], f1, l * f0);
#pragma unroll
        for (int j = 0; j < DT; j++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                o[j][i] = fmaf(mo[qrow * MLD + j * 32 + 8 * (i >> 2) + 4 * g + (i & 3)], f1, o[j][i] * f0);
    }
    if (!wave_active) return;
    if (qrow < nrows) {
        const float inv = 1.0f / l;
        u16 *op = out + (size_t)(row0 + qrow) * NQ + h * HD;
#pragma unroll
        for (int j = 0; j < DT; j++)
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const unsigned lo = (unsigned)f2h(o[j][4 * i4] * inv) |
                                    ((unsigned)f2h(o[j][4 * i4 + 1] * inv) << 16);
                const unsigned hi = (unsigned)f2h(o[j][4 * i4 + 2] * inv) |
                                    ((unsigned)f2h(o[j][4 * i4 + 3] * inv) << 16);
                *(uint2 *)(op + j * 32 + 8 * i4 + 4 * g) = make_uint2(lo, hi);
            }
    }
}

/* ---- 32-query blocks, key tiles split across the waves ---------------------- */

#define BQS 32          /* query rows per work-group */

template <int HD, typename KT>
__global__ void __launch_bounds__(AT) k_attn_prefill_split(
    const float *__restrict__ q, const KT *__restrict__ kc, const KT *__restrict__ vc,
    const int *__restrict__ pos, const int *__restrict__ slot, int S, int nseq, int nqb, int H, int Hkv,
    int max_seq, u16 *__restrict__ out)
{
    constexpr int KLD = HD + 8;          /* K tile row stride (halves)   */
    constexpr int KS = HD / 16;          /* MFMA k-steps over head dims  */
    constexpr int DT = HD / 32;          /* 32-dim row tiles of O^T      */
    constexpr int PPL = BKV * HD / 16 / 64;  /* staging units per lane (one wave stages a tile) */
    constexpr bool PREF = HD == 64 && sizeof(KT) == 2;   /* next tile in registers */
    constexpr int STAGE = BKV * KLD + HD * BKV;          /* halves of one wave's K and V^T */
    static_assert(BKV * HD / 8 % 256 == 0, "staging shape");
    constexpr int MLD = HD + 1;                          /* merge row stride (floats) */
    static_assert(NW * STAGE * 2 >= (NW * BQS * MLD + 2 * NW * BQS) * 4, "merge area fits the staging area");
    __shared__ __attribute__((aligned(16))) u16 stg[NW * STAGE];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int h, seq, qb;
    block_of(blockIdx.x, nqb, nseq, H, h, seq, qb);
    const int kvh = small_div(h, small_div(H, Hkv));
    const int NQ = H * HD;
    const int row0 = seq * S + qb * BQS;           /* first row of the block       */
    const int nrows = min(BQS, S - qb * BQS);       /* valid rows of the block      */
    const int p0 = pos[row0];                     /* position of the block's row 0 */
    const int cs = slot[row0];
    const size_t cbase = ((size_t)cs * Hkv + kvh) * max_seq * HD;
    /* scores are kept in log2 units: exp(x) = exp2(x * log2 e) */
    const float scale = 1.4426950408889634f / sqrtf((float)HD);
    const int last_pos = p0 + nrows - 1;          /* last query position of the block */
    const int ntiles = last_pos / BKV + 1;
    u16 *sk = stg + wave * STAGE, *svt = sk + BKV * KLD;

    /* K / V of one tile for this wave: lane l stages units l + i*64 (two keys, 8
     * dims each); keys past the block's last position repeat it (masked for
     * every query that reads them) */
    auto load = [&](int kt, int i, uint4 (&k8)[2], uint4 (&v8)[2]) {
        int pk, d0;
        pair_of<HD>(lane + i * 64, pk, d0);
        const int key = kt * BKV + vperm(pk);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const size_t off = cbase + (size_t)min(key + e, last_pos) * HD + d0;
            k8[e] = kv8_f16(kc + off);
            v8[e] = kv8_f16(vc + off);
        }
    };
    auto put = [&](int i, const uint4 (&k8)[2], const uint4 (&v8)[2]) {
        int pk, d0;
        pair_of<HD>(lane + i * 64, pk, d0);
        stage_pair<KLD>(sk, svt, pk, d0, k8[0], k8[1], v8[0], v8[1]);
    };
    /* hd 64 with an fp16 cache: the whole next tile is held in registers while
     * the current one computes; otherwise a tile is staged 2 units at a time */
    constexpr int RC = PREF ? PPL : 1;
    uint4 rk[RC][2], rv[RC][2];
    auto fetch = [&](int kt) {
#pragma unroll
        for (int i = 0; i < RC; i++) load(kt, i, rk[i], rv[i]);
    };
    auto stage = [&](int kt) {
        if constexpr (PREF) {
#pragma unroll
            for (int i = 0; i < PPL; i++) put(i, rk[i], rv[i]);
        } else {
#pragma unroll
            for (int i0 = 0; i0 < PPL; i0 += 2) {
                uint4 k4[2][2], v4[2][2];
#pragma unroll
                for (int i = 0; i < 2; i++) load(kt, i0 + i, k4[i], v4[i]);
#pragma unroll
                for (int i = 0; i < 2; i++) put(i0 + i, k4[i], v4[i]);
            }
        }
    };
    if (PREF && wave < ntiles) fetch(wave);       /* wave-uniform */

    /* lane l takes query row l%32 of the block */
    const int qrow = lane & 31;
    const int qp = p0 + qrow;                     /* this lane's query position */
    uint4 qb16[KS];
    load_q<HD>(q, (size_t)(row0 + min(qrow, nrows - 1)), NQ, h, qb16);
    f32x16 o[DT];
#pragma unroll
    for (int j = 0; j < DT; j++) o[j] = (f32x16){};
    float mrow = -INFINITY, lrow = 0.f;

    for (int kt = wave; kt < ntiles; kt += NW) {  /* wave-uniform */
        stage(kt);
        __builtin_amdgcn_s_waitcnt(0xc07f);       /* lgkmcnt(0): the wave's LDS writes landed */
        __builtin_amdgcn_wave_barrier();
        if (PREF && kt + NW < ntiles) fetch(kt + NW);
        if (kt * BKV + BKV - 1 <= p0)             /* wave-uniform: no key after any query */
            tile_update<HD, KLD, false>(sk, svt, qb16, kt * BKV, qp, scale, o, mrow, lrow);
        else
            tile_update<HD, KLD, true>(sk, svt, qb16, kt * BKV, qp, scale, o, mrow, lrow);
        __builtin_amdgcn_wave_barrier();           /* the tile's reads precede the next stash */
    }
    /* merge the four waves: each writes (m, l, O) of its 32 queries; element i of
     * o[j] is dim j*32 + 8*(i/4) + 4*g + i%4 of query l%32 */
    const float lsum = lrow + xor32_f(lrow);
    __syncthreads();                               /* every wave is done with its staging area */
    float *mo = (float *)stg;                      /* [NW][BQS][MLD] outputs */
    float *mm = mo + NW * BQS * MLD, *ml = mm + NW * BQS;
    if (g == 0) {
        mm[wave * BQS + qrow] = mrow;
        ml[wave * BQS + qrow] = lsum;
    }
#pragma unroll
    for (int j = 0; j < DT; j++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            mo[(wave * BQS + qrow) * MLD + j * 32 + 8 * (i >> 2) + 4 * g + (i & 3)] = o[j][i];
    __syncthreads();
    /* thread t: query t / 8, dims (t % 8) * HD/8 .. +HD/8 */
    constexpr int DPT = HD / 8;
    const int r = tid >> 3, d0 = (tid & 7) * DPT;
    if (r < nrows) {
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; w++) M = fmaxf(M, mm[w * BQS + r]);
        float wgt[NW], L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float mw = mm[w * BQS + r];
            wgt[w] = mw == -INFINITY ? 0.f : exp2f(mw - M);
            L = fmaf(ml[w * BQS + r], wgt[w], L);
        }
        const float inv = 1.0f / L;
        u16 *op = out + (size_t)(row0 + r) * NQ + h * HD + d0;
#pragma unroll
        for (int d = 0; d < DPT; d += 2) {
            float a = 0.f, bsum = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) {
                a = fmaf(mo[(w * BQS + r) * MLD + d0 + d], wgt[w], a);
                bsum = fmaf(mo[(w * BQS + r) * MLD + d0 + d + 1], wgt[w], bsum);
            }
            *(unsigned *)(op + d) = (unsigned)f2h(a * inv) | ((unsigned)f2h(bsum * inv) << 16);
        }
    }
}

/* ---- the sequences' last rows ------------------------------------------------ */

/* Work-group i copies sequence i's last residual row and query row: all that
 * the last layer's attention, Wo and FFN owe a caller that wants the last
 * rows' logits.  Latency bound (one round trip, n * (D + NQ) * 4 bytes). */
__global__ void __launch_bounds__(AT) k_last_rows(const float *__restrict__ x, const float *__restrict__ q,
                                                 int D, int NQ, int S, float *__restrict__ xo,
                                                 float *__restrict__ qo)
{
    const size_t i = blockIdx.x, row = i * S + S - 1;
    for (int c = 4 * threadIdx.x; c < D; c += 4 * AT)
        *(float4 *)(xo + i * D + c) = *(const float4 *)(x + row * D + c);
    for (int c = 4 * threadIdx.x; c < NQ; c += 4 * AT)
        *(float4 *)(qo + i * NQ + c) = *(const float4 *)(q + row * NQ + c);
}

extern "C" int lmk_last_rows(hipStream_t s, const float *x, const float *q, int D, int NQ, int S, int n,
                             float *xo, float *qo)
{
    if (D < 4 || D % 4 || NQ < 4 || NQ % 4 || S < 1 || n < 1 || !x || !q || !xo || !qo)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_last_rows, dim3(n), dim3(AT), 0, s, x, q, D, NQ, S, xo, qo);
    return hipGetLastError();
}

/* Whether the 32-query kernel (split) is taken rather than the shared-tile one:
 * up to a number of its work-groups, nseq * H * ceil(S / 32).  All of them run at
 * once up to 512 at hd 64 (two a CU) and 256 at hd 128 (one), each a quarter of
 * its block's tiles long; beyond that they queue, and the shared kernel stages a
 * tile once for more queries, but its last block walks half of its sequence's
 * tiles in turn, so that long sequences stay with the split kernel longer.
 * Sequences of up to 64 rows end in one tile: the other waves would idle.  us
 * per launch, split / shared (work-groups):
 *   hd 64     1 x 1300, 12 heads (492) 14.2 / 17.6    1 x 1900 (720) 22.0 / 23.9
 *             1 x 1500, 16 heads (752) 20.1 / 20.0    1 x 1900 (960) 25.9 / 24.1
 *             2 x 559 (576) 10.5 / 10.7               2 x 639 (640) 12.2 / 11.1
 *             3 x 400, 12 heads (468) 7.7 / 8.4       3 x 600 (684) 13.0 / 11.4
 *             8 x 128, 16 heads (512) 6.0 / 6.5       10 x 128 (640) 8.5 / 6.6
 *             16 x 64, 12 heads (384) 5.5 / 4.8       8 x 64 (192) 4.8 / 4.6
 *   fp32      2 x 559 (576) 11.8 / 12.9               2 x 639 (640) 13.6 / 13.3
 *             1 x 1900 (960) 32.3 / 30.2              3 x 400 (624) 12.7 / 10.8
 *   hd 128    1 x 640 (320) 14.9 / 20.3               1 x 1000 (512) 24.1 / 26.9
 *   16 heads  1 x 1152 (576) 32.2 / 29.7              1 x 1900 (960) 63.6 / 44.6
 *             2 x 384 (384) 14.9 / 15.7               2 x 450 (480) 17.7 / 16.2
 *             4 x 128 (256) 7.8 / 10.7                6 x 128 (384) 13.5 / 10.9
 *   fp32      1 x 512 (256) 17.2 / 20.0               1 x 600 (304) 22.6 / 21.7
 *             2 x 384 (384) 20.6 / 17.5               8 x 64 (256) 10.4 / 8.3 */
extern "C" int lmk_attn_takes_split(int hd, int kv_f32, int H, int nseq, int S)
{
    const int one = hd == 64 ? 512 : 256;
    const long wgs = (long)((S + BQS - 1) / BQS) * nseq * H;
    if (S <= 64) return wgs <= one / 2;
    if (S <= 256 || (hd == 128 && kv_f32)) return wgs <= one;
    return wgs <= (hd == 64 ? one + 11 * (S - 256) / 50 : 290 + 63 * S / 256);
}

extern "C" int lmk_attn_prefill(hipStream_t s, const float *q, const void *kc, const void *vc,
                                int kv_f32, const int *pos, const int *slot, int S, int nseq,
                                int H, int Hkv, int hd, int max_seq, uint16_t *out)
{
    if (S < 1 || nseq < 1 || H < 1 || Hkv < 1 || H % Hkv || !pos || !slot) return hipErrorInvalidValue;
    if (hd != 64 && hd != 128) return hipErrorInvalidValue;
    /* (block_of divides by small_div: ids below 2^20, divisors below 2^12) */
    if ((long)((S + BQS - 1) / BQS) * nseq * H >= 1 << 20 || nseq >= 1 << 12 || H >= 1 << 12)
        return hipErrorInvalidValue;
    if (!lmk_attn_takes_split(hd, kv_f32, H, nseq, S)) {
        /* hd 128: eight waves, two key tiles a step (two waves a SIMD); hd 64:
         * 64-query blocks of four waves, two key tiles a step, unless the
         * sequences are short (20 x 90 rows, 16 heads: 10.2 us against 8.8 with
         * 128-query blocks, which then stage each tile once) */
#define LAUNCH_APV(HD_, KT_, QG_, W_)                                                                      \
    do {                                                                                                   \
        const int nqb = (S + 32 * QG_ - 1) / (32 * QG_);   /* blocks of the kernel's own 32 * QG queries */ \
        hipLaunchKernelGGL((k_attn_prefill_blk<HD_, KT_, QG_, W_>), dim3(nqb * nseq * H), dim3(64 * W_), 0, s, q, \
                           (const KT_ *)kc, (const KT_ *)vc, pos, slot, S, nseq, nqb, H, Hkv, max_seq, out);      \
    } while (0)
#define LAUNCH_AP(HD_, KT_)                                      \
    do {                                                         \
        if constexpr (HD_ == 128) LAUNCH_APV(HD_, KT_, 4, 8);    \
        else if (S > 128) LAUNCH_APV(HD_, KT_, 2, 4);            \
        else LAUNCH_APV(HD_, KT_, 4, 4);                         \
    } while (0)
        if (hd == 64 && kv_f32) LAUNCH_AP(64, float);
        else if (hd == 64) LAUNCH_AP(64, u16);
        else if (kv_f32) LAUNCH_AP(128, float);
        else LAUNCH_AP(128, u16);
#undef LAUNCH_AP
#undef LAUNCH_APV
    } else {
        const int nqb = (S + BQS - 1) / BQS;
        dim3 grid(nqb * nseq * H);
#define LAUNCH_AP(HD_, KT_)                                                                        \
    hipLaunchKernelGGL((k_attn_prefill_split<HD_, KT_>), grid, dim3(AT), 0, s, q, (const KT_ *)kc, \
                       (const KT_ *)vc, pos, slot, S, nseq, nqb, H, Hkv, max_seq, out)
        if (hd == 64 && kv_f32) LAUNCH_AP(64, float);
        else if (hd == 64) LAUNCH_AP(64, u16);
        else if (kv_f32) LAUNCH_AP(128, float);
        else LAUNCH_AP(128, u16);
#undef LAUNCH_AP
    }
    return hipGetLastError();
}
