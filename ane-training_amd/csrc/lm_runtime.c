/*
 * lm_runtime.c — the C-ABI runtime of the Stories token loop (C99 over the HIP
 * C runtime API).  It owns device memory, the stream, the per-batch decode
 * graphs and the host-facing entry points of stories_lm.h; every kernel is
 * reached through the lmk_* launchers of the HIP translation units.
 *
 * Device layout (all row-major, W[out, in]):
 *   layer block l (one allocation for all layers, layer after layer):
 *     Wqkv [NQ + 2*NKV, D]   Wq rows, then Wk rows, then Wv rows
 *     Wo   [D, NQ]
 *     W13  [2F, D]           W1/W3 rows interleaved in blocks of 16
 *     W2   [D, F]
 *   embed [V, D], wcls [V, D] (the embedding itself when tied)   fp16
 *   rms_att [L, D], rms_ffn [L, D], rms_final [D]                  fp32
 *   RoPE cos/sin [max_seq, hd/2]                                   fp32
 *   K/V cache, per layer [max_batch][Hkv][max_seq][hd]             fp16
 *   residual x [rows, D], q [rows, NQ], gate g [rows, F],
 *   logits [rows, V]                                               fp32
 */
#include "lm_internal.h"

#include <limits.h>
#include <omp.h>
#include <pthread.h>
#include <sched.h>
#include <semaphore.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define HIPCHK(call)                                                                 \
    do {                                                                             \
        hipError_t e_ = (call);                                                      \
        if (e_ != hipSuccess) {                                                      \
            fprintf(stderr, "stories_lm: %s failed at %s:%d: %s\n", #call, __FILE__, \
                    __LINE__, hipGetErrorString(e_));                                \
            return LM_ERR_HIP;                                                       \
        }                                                                            \
    } while (0)

#define MAX_GEMV_B 4
#define GIVE_MIN_FLOATS ((size_t)1 << 20)   /* least staging of results: two 2 MiB segments */
/* What a queued decode step takes in and gives back: a call's step with its
 * logits or with the ids alone, and the steps of a greedy run (one, or
 * GRAPH_STEPS), whose inputs and ids the run moves itself. */
enum { STEP_LOGITS, STEP_IDS, STEP_GREEDY, STEP_GREEDY_N, STEP_KINDS };
#define CTX_CLASSES 4      /* context lengths the decode attention is launched for (ctx_class) */

/* A call's results on their way from the staging to the caller's memory: n
 * floats in segments of seg, segment i through half i & 1 of the staging under
 * number seq0 + i.  Threads t < nt take every nt'th share of each segment as it
 * lands; prog[t]: segments that t has done.  Thread 0 is the caller; the others
 * are the handle's own, made at its first large result: they sleep on `go`
 * between calls. */
#define CREW_MAX 4
typedef struct {
    LMModel *m;
    float *dst;                 /* NULL: only wait */
    size_t n, seg, nseg;
    int seq0, nt;
    int issued, rc, prog[CREW_MAX];
    int hands, quit;            /* threads beside the caller's */
    struct CrewHand { void *crew; int t; sem_t go; pthread_t id; } hand[CREW_MAX - 1];
} Crew;

struct LMModel {
    Config cfg;                 /* vocab_size positive */
    int untied;
    int D, F, L, H, Hkv, hd, NQ, NKV, V;
    int max_batch, max_seq, max_rows;
    int cls_nblk;
    size_t layer_elems, off_wo, off_w13, off_w2;
    hipStream_t stream;
    hipEvent_t ev0, ev1;
    hipEvent_t ev_hand;         /* end of this handle's last hand-off launches */
    /* weights */
    uint16_t *d_layers, *d_embed, *d_wcls;
    float *d_rms_att, *d_rms_ffn, *d_rms_final;
    float *d_rope_cos, *d_rope_sin;
    /* cache + activations */
    void *d_kc, *d_vc;
    size_t kv_layer_elems;
    int kv_f32;                 /* cache element: 0 = binary16, 1 = fp32 */
    /* per-row activations, max_rows rows (decode rows, or a prefill chunk) */
    float *d_x, *d_q, *d_attn, *d_g, *d_logits;
    float *d_ss;                /* per-row sums of squares of x, D/32 per row  */
    float *d_part;              /* partials of K-split GEMMs, Wo/W2 products    */
    uint16_t *d_g16;            /* gate rows in fp16 (input of the W2 GEMM)    */
    uint16_t *d_xn16, *d_a16;   /* normalised rows / attention rows in fp16    */
    LMArgPart *d_amax;
    int *d_rin;                 /* prefill rows of a chunk of R: tokens, positions, slots
                                 * (R ints each, back to back), then, for the last rows'
                                 * logits, the sequences' last positions and slots
                                 * (k_rows_in reads them from h_rin)                 */
    int *h_rin;                 /* their pinned host staging (same layout); with all
                                 * logits the device writes R floats of loss terms
                                 * after the slots (lm_prefill_loss)                 */
    int *dh_rin;                /* its device address                               */
    /* per-slot greedy state */
    int *d_tok, *d_pos, *d_hist, *d_slot_id;
    /* batch 1-4 chain: QKV, attention (fuse_qa >= 1), Wo (>= 2) and the FFN
     * (3 at one row, 4 at every batch; chain_level) in one launch, handing q,
     * k, v, the head outputs, x and the gate over through tagged words; the
     * decode-step count that tags them; the flag a hand-off wait that gives up
     * sets, and the polls before one does */
    int fuse_qa;
    int prefill_fold;           /* LM_OPT_PREFILL_FOLD */
    int fold_off;               /* the folded norm is off for the rows being redone */
    int *d_ovf;                 /* device address of ovf_slot: RESNORM's overflow flag */
    int layer_wgs;              /* whole-layer work-groups per CU at most (0: no cap) */
    unsigned long long *d_tagged;
    unsigned long long *d_cls_tw;     /* the classifier's argmax partials as tagged words (level 3) */
    unsigned *d_epoch;
    int *d_err;
    /* pinned host staging: results (give_floats floats, at least max_batch
     * rows of logits); the call block, the header and the flags of k_io.hip
     * in one block, with their device addresses */
    float *h_logits, *dh_logits;
    size_t give_floats;
    int *h_io;                  /* (lm_profile_chain) and RESNORM's overflow flag */
    int *h_call, *h_hdr, *h_flag, *dh_call, *dh_hdr, *dh_flag;
    int *d_seq;                 /* number of the call whose step is running */
    int seq;
    /* captured decode graphs by kind of step (greedy feedback stays on the
     * device) and context class: [max_batch + 1][kind][class] */
    hipGraphExec_t (*step_graph)[STEP_KINDS][CTX_CLASSES];
    /* captured prefill chunks (the layers and the classifier) of shapes.graph */
    hipGraphExec_t pgraph[LM_SHAPE_GRAPHS];
    LMShapes shapes;
    Crew crew;
    int use_graph;
    int ctx_cls;                /* context class of the decode step being queued */
};

static int g_init_status = 1; /* 1 = not attempted */

const char *lm_strerror(int status)
{
    switch (status) {
    case LM_OK: return "ok";
    case LM_ERR_NO_DEVICE: return "no HIP device";
    case LM_ERR_NOT_GFX950: return "device is not gfx950";
    case LM_ERR_INVALID: return "invalid argument";
    case LM_ERR_OOM: return "out of memory";
    case LM_ERR_HIP: return "HIP runtime error";
    case LM_ERR_IO: return "I/O error";
    case LM_ERR_FORMAT: return "bad or truncated weight file";
    case LM_ERR_RANGE: return "token, position, slot or length out of range";
    case LM_ERR_UNSUPPORTED: return "shape not supported by the kernels";
    case LM_ERR_NOT_INIT: return "lm_init not called or failed";
    default: return "unknown status";
    }
}

/* The device checks run once per process (pthread_once), so concurrent first
 * calls from several threads neither race on the status nor repeat the
 * setup; every call returns the one recorded status. */
static pthread_once_t g_init_once = PTHREAD_ONCE_INIT;

static void init_once(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n < 1) {
        fprintf(stderr, "stories_lm: no HIP device visible\n");
        g_init_status = LM_ERR_NO_DEVICE;
        return;
    }
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, 0) != hipSuccess) {
        g_init_status = LM_ERR_NO_DEVICE;
        return;
    }
    if (strncmp(p.gcnArchName, "gfx950", 6) != 0) {
        fprintf(stderr, "stories_lm: device 0 is %s, kernels are built for gfx950\n",
                p.gcnArchName);
        g_init_status = LM_ERR_NOT_GFX950;
        return;
    }
    if (hipSetDevice(0) != hipSuccess) {
        g_init_status = LM_ERR_NO_DEVICE;
        return;
    }
    if (lmk_noalloc_setup() != hipSuccess) {
        fprintf(stderr, "stories_lm: lookup of the static scratch's device address failed\n");
        g_init_status = LM_ERR_HIP;
        return;
    }
    g_init_status = LM_OK;
}

int lm_init(void)
{
    if (pthread_once(&g_init_once, init_once) != 0) return LM_ERR_NOT_INIT;
    return g_init_status;
}

int lm_device_info(LMDeviceInfo *out)
{
    if (!out) return LM_ERR_INVALID;
    int rc = lm_init();
    if (rc) return rc;
    hipDeviceProp_t p;
    HIPCHK(hipGetDeviceProperties(&p, 0));
    memset(out, 0, sizeof(*out));
    snprintf(out->name, sizeof(out->name), "%.63s", p.name);
    snprintf(out->arch, sizeof(out->arch), "%.31s", p.gcnArchName);
    out->compute_units = p.multiProcessorCount;
    out->clock_khz = p.clockRate;
    out->l2_bytes = p.l2CacheSize;
    out->total_mem = p.totalGlobalMem;
    return LM_OK;
}

/* ------------------------------------------------------------------------- */
/* creation                                                                   */
/* ------------------------------------------------------------------------- */

static int dev_alloc(void **p, size_t bytes)
{
    *p = NULL;
    if (bytes == 0) return LM_OK;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        fprintf(stderr, "stories_lm: hipMalloc(%zu) failed: %s\n", bytes, hipGetErrorString(e));
        *p = NULL;
        return LM_ERR_OOM;
    }
    return LM_OK;
}

/* Pinned host memory and its device address. */
static int host_alloc(void **h, void **d, size_t bytes)
{
    if (hipHostMalloc(h, bytes, 0) != hipSuccess) {
        fprintf(stderr, "stories_lm: hipHostMalloc(%zu) failed\n", bytes);
        *h = NULL;
        return LM_ERR_OOM;
    }
    return hipHostGetDevicePointer(d, *h, 0) == hipSuccess ? LM_OK : LM_ERR_HIP;
}

/* Copy n elements of tensor src (fp32 or fp16) as fp16 into dst (host). */
static void to_f16(const void *src, LMDType dt, size_t off, size_t n, uint16_t *dst)
{
    if (dt == LM_DTYPE_F16)
        memcpy(dst, (const uint16_t *)src + off, n * 2);
    else
        lm_f32_to_f16((const float *)src + off, dst, n);
}

static void to_f32(const void *src, LMDType dt, size_t off, size_t n, float *dst)
{
    if (dt == LM_DTYPE_F32)
        memcpy(dst, (const float *)src + off, n * 4);
    else
        lm_f16_to_f32((const uint16_t *)src + off, dst, n);
}

/* Where the host weights come from: one contiguous block per tensor
 * (LMWeights) or per-layer pointer arrays (LMLayerWeights). */
typedef struct {
    LMDType dtype;
    const void *embed, *rms_final, *wcls;   /* wcls NULL: tied */
    const LMWeights *flat;
    const LMLayerWeights *per;
} WSrc;

static const void *const *per_layer_array(const LMLayerWeights *w, int t)
{
    switch (t) {
    case LMH_T_RMS_ATT: return w->rms_att_w;
    case LMH_T_WQ: return w->wq;
    case LMH_T_WK: return w->wk;
    case LMH_T_WV: return w->wv;
    case LMH_T_WO: return w->wo;
    case LMH_T_RMS_FFN: return w->rms_ffn_w;
    case LMH_T_W1: return w->w1;
    case LMH_T_W2: return w->w2;
    case LMH_T_W3: return w->w3;
    default: return NULL;
    }
}

/* Layer l's tensor t (n elements per layer) in the source's element type. */
static const void *src_layer(const WSrc *ws, int t, size_t l, size_t n)
{
    if (ws->per) return per_layer_array(ws->per, t)[l];
    const char *base = (const char *)lmh_weights_ptr(ws->flat, t);
    return base + l * n * (ws->dtype == LM_DTYPE_F16 ? 2 : 4);
}

static int upload_weights(LMModel *m, const WSrc *w)
{
    const size_t D = m->D, F = m->F, NQ = m->NQ, NKV = m->NKV, V = m->V, L = m->L;
    const size_t GB = LMK_GATE_BLOCK;
    const LMDType dt = w->dtype;
    uint16_t *stage = (uint16_t *)malloc(m->layer_elems * 2);
    float *nf = (float *)malloc(L * D * 4);
    if (!stage || !nf) { free(stage); free(nf); return LM_ERR_OOM; }
    int rc = LM_OK;
    for (size_t l = 0; l < L && rc == LM_OK; l++) {
        uint16_t *p = stage;
        to_f16(src_layer(w, LMH_T_WQ, l, NQ * D), dt, 0, NQ * D, p);    p += NQ * D;
        to_f16(src_layer(w, LMH_T_WK, l, NKV * D), dt, 0, NKV * D, p);  p += NKV * D;
        to_f16(src_layer(w, LMH_T_WV, l, NKV * D), dt, 0, NKV * D, p);  p += NKV * D;
        to_f16(src_layer(w, LMH_T_WO, l, D * NQ), dt, 0, D * NQ, p);    p += D * NQ;
        const void *w1 = src_layer(w, LMH_T_W1, l, F * D), *w3 = src_layer(w, LMH_T_W3, l, F * D);
        for (size_t j = 0; j < F / GB; j++) {
            to_f16(w1, dt, j * GB * D, GB * D, p); p += GB * D;
            to_f16(w3, dt, j * GB * D, GB * D, p); p += GB * D;
        }
        to_f16(src_layer(w, LMH_T_W2, l, D * F), dt, 0, D * F, p);
        if (hipMemcpy(m->d_layers + l * m->layer_elems, stage, m->layer_elems * 2,
                      hipMemcpyHostToDevice) != hipSuccess)
            rc = LM_ERR_HIP;
    }
    free(stage);
    if (rc == LM_OK) {
        uint16_t *e16 = (uint16_t *)malloc(V * D * 2);
        if (!e16) rc = LM_ERR_OOM;
        if (rc == LM_OK) {
            to_f16(w->embed, dt, 0, V * D, e16);
            if (hipMemcpy(m->d_embed, e16, V * D * 2, hipMemcpyHostToDevice) != hipSuccess)
                rc = LM_ERR_HIP;
            if (rc == LM_OK && m->untied) {
                to_f16(w->wcls, dt, 0, V * D, e16);
                if (hipMemcpy(m->d_wcls, e16, V * D * 2, hipMemcpyHostToDevice) != hipSuccess)
                    rc = LM_ERR_HIP;
            }
        }
        free(e16);
    }
    if (rc == LM_OK) {
        for (size_t l = 0; l < L; l++) to_f32(src_layer(w, LMH_T_RMS_ATT, l, D), dt, 0, D, nf + l * D);
        if (hipMemcpy(m->d_rms_att, nf, L * D * 4, hipMemcpyHostToDevice) != hipSuccess) rc = LM_ERR_HIP;
        for (size_t l = 0; l < L; l++) to_f32(src_layer(w, LMH_T_RMS_FFN, l, D), dt, 0, D, nf + l * D);
        if (rc == LM_OK && hipMemcpy(m->d_rms_ffn, nf, L * D * 4, hipMemcpyHostToDevice) != hipSuccess)
            rc = LM_ERR_HIP;
        to_f32(w->rms_final, dt, 0, D, nf);
        if (rc == LM_OK && hipMemcpy(m->d_rms_final, nf, D * 4, hipMemcpyHostToDevice) != hipSuccess)
            rc = LM_ERR_HIP;
    }
    free(nf);
    return rc;
}

static size_t kv_bytes(const LMModel *m)
{
    return (size_t)m->L * m->kv_layer_elems * (m->kv_f32 ? 4 : 2);
}

/* (Re)allocate the K/V cache in the current element type, zero-filled. */
static int alloc_kv(LMModel *m)
{
    if (m->d_kc) { hipFree(m->d_kc); m->d_kc = NULL; }
    if (m->d_vc) { hipFree(m->d_vc); m->d_vc = NULL; }
    int st = dev_alloc(&m->d_kc, kv_bytes(m));
    if (!st) st = dev_alloc(&m->d_vc, kv_bytes(m));
    if (st) return st;
    if (hipMemset(m->d_kc, 0, kv_bytes(m)) != hipSuccess ||
        hipMemset(m->d_vc, 0, kv_bytes(m)) != hipSuccess)
        return LM_ERR_HIP;
    return LM_OK;
}

static void crew_end(Crew *c);

static void drop_graphs(LMModel *m)
{
    for (int i = 0; i < LM_SHAPE_GRAPHS; i++) {
        if (m->pgraph[i]) hipGraphExecDestroy(m->pgraph[i]);
        m->pgraph[i] = NULL;
        m->shapes.graph[i].used = 0;
    }
    if (!m->step_graph) return;
    for (int b = 0; b <= m->max_batch; b++)
        for (int k = 0; k < STEP_KINDS * CTX_CLASSES; k++) {
            hipGraphExec_t *ge = &m->step_graph[b][k / CTX_CLASSES][k % CTX_CLASSES];
            if (*ge) {
                hipGraphExecDestroy(*ge);
                *ge = NULL;
            }
        }
}

static void free_rows(LMModel *m)
{
    void *dev[] = {m->d_x, m->d_q, m->d_attn, m->d_g, m->d_logits, m->d_ss, m->d_part, m->d_g16,
                   m->d_xn16, m->d_a16, m->d_amax, m->d_rin};
    for (size_t i = 0; i < sizeof(dev) / sizeof(dev[0]); i++)
        if (dev[i]) hipFree(dev[i]);
    if (m->h_rin) hipHostFree(m->h_rin);
    m->d_x = m->d_q = m->d_attn = m->d_g = m->d_logits = m->d_ss = m->d_part = NULL;
    m->d_g16 = m->d_xn16 = m->d_a16 = NULL;
    m->d_amax = NULL;
    m->d_rin = m->h_rin = m->dh_rin = NULL;
    m->max_rows = 0;
}

/* (Re)allocate the per-row activation buffers for R rows.  Captured graphs
 * hold the old addresses, so they are dropped. */
static int alloc_rows(LMModel *m, int R)
{
    if (m->stream && hipStreamSynchronize(m->stream) != hipSuccess) return LM_ERR_HIP;
    drop_graphs(m);
    free_rows(m);
    const size_t r = (size_t)R, D = m->D, F = m->F, NQ = m->NQ, V = m->V;
    int st;
    if ((st = dev_alloc((void **)&m->d_x, r * D * 4))) return st;
    if ((st = dev_alloc((void **)&m->d_q, r * NQ * 4))) return st;
    if ((st = dev_alloc((void **)&m->d_attn, r * NQ * 4))) return st;
    if ((st = dev_alloc((void **)&m->d_g, r * F * 4))) return st;
    if ((st = dev_alloc((void **)&m->d_g16, r * F * 2))) return st;
    if ((st = dev_alloc((void **)&m->d_xn16, r * D * 2))) return st;
    if ((st = dev_alloc((void **)&m->d_a16, r * NQ * 2))) return st;
    if ((st = dev_alloc((void **)&m->d_logits, r * V * 4))) return st;
    if ((st = dev_alloc((void **)&m->d_ss, r * (D / 32) * 4))) return st;
    {
        /* K-split partials (widest: QKV of decode rows), or one [R, D] product
         * of prefill rows */
        const size_t w = NQ + 2 * (size_t)m->NKV > D ? NQ + 2 * (size_t)m->NKV : D;
        const size_t rd = r < 64 ? r : 64;
        size_t n = LMK_MAX_SPLIT * rd * w;
        if (r > 64 && LMK_MAX_ROW_SPLIT * r * w > n) n = LMK_MAX_ROW_SPLIT * r * w;
        if (r * D > n) n = r * D;
        if ((st = dev_alloc((void **)&m->d_part, n * 4))) return st;
    }
    if ((st = dev_alloc((void **)&m->d_amax, r * m->cls_nblk * sizeof(LMArgPart)))) return st;
    /* tokens, positions and slots of a chunk's rows, then up to as many ints more */
    if ((st = dev_alloc((void **)&m->d_rin, 4 * r * 4))) return st;
    if ((st = host_alloc((void **)&m->h_rin, (void **)&m->dh_rin, 4 * r * 4))) return st;
    m->max_rows = R;
    return LM_OK;
}

static int supported_k(int k)
{
    return k == 256 || k == 512 || k == 768 || k == 1024 || k == 2048 || k == 5632;
}

static LMModel *create_model(const Config *cfg, const WSrc *w, int max_batch, int max_seq,
                             int *status);

LMModel *lm_create(const Config *cfg, const LMWeights *w, int max_batch, int max_seq, int *status)
{
    int st = LM_OK;
    if (!cfg || !w || max_batch < 1 || max_seq < 1 ||
        (w->dtype != LM_DTYPE_F32 && w->dtype != LM_DTYPE_F16))
        st = LM_ERR_INVALID;
    for (int t = 0; t < LMH_NTENSORS - 1 && st == LM_OK; t++)
        if (!lmh_weights_ptr(w, t)) {
            fprintf(stderr, "stories_lm: weight tensor %d is NULL\n", t);
            st = LM_ERR_INVALID;
        }
    if (st != LM_OK) {
        if (status) *status = st;
        fprintf(stderr, "stories_lm: lm_create failed: %s\n", lm_strerror(st));
        return NULL;
    }
    const WSrc ws = {w->dtype, w->token_embedding, w->rms_final_w,
                     lmh_weights_untied(w) ? w->wcls : NULL, w, NULL};
    return create_model(cfg, &ws, max_batch, max_seq, status);
}

LMModel *lm_create_layers(const Config *cfg, const LMLayerWeights *w, int max_batch, int max_seq,
                          int *status)
{
    int st = LM_OK;
    if (!cfg || !w || max_batch < 1 || max_seq < 1 || cfg->n_layers < 1 ||
        (w->dtype != LM_DTYPE_F32 && w->dtype != LM_DTYPE_F16) || !w->token_embedding ||
        !w->rms_final_w)
        st = LM_ERR_INVALID;
    for (int t = LMH_T_RMS_ATT; t <= LMH_T_W3 && st == LM_OK; t++) {
        const void *const *a = per_layer_array(w, t);
        if (!a) {
            fprintf(stderr, "stories_lm: per-layer weight array %d is NULL\n", t);
            st = LM_ERR_INVALID;
        }
        for (int l = 0; a && l < cfg->n_layers && st == LM_OK; l++)
            if (!a[l]) {
                fprintf(stderr, "stories_lm: weight tensor %d of layer %d is NULL\n", t, l);
                st = LM_ERR_INVALID;
            }
    }
    if (st != LM_OK) {
        if (status) *status = st;
        fprintf(stderr, "stories_lm: lm_create_layers failed: %s\n", lm_strerror(st));
        return NULL;
    }
    const WSrc ws = {w->dtype, w->token_embedding, w->rms_final_w,
                     w->wcls && w->wcls != w->token_embedding ? w->wcls : NULL, NULL, w};
    return create_model(cfg, &ws, max_batch, max_seq, status);
}

static LMModel *create_model(const Config *cfg, const WSrc *w, int max_batch, int max_seq,
                             int *status)
{
    int st = LM_OK;
    LMModel *m = NULL;
#define FAIL(code)      \
    do {                \
        st = (code);    \
        goto fail;      \
    } while (0)
    if ((st = lm_init()) != LM_OK) goto fail;
    if ((st = lmh_check_config(cfg)) != LM_OK) {
        fprintf(stderr, "stories_lm: inconsistent Config\n");
        goto fail;
    }
    m = (LMModel *)calloc(1, sizeof(LMModel));
    if (!m) FAIL(LM_ERR_OOM);
    m->cfg = *cfg;
    m->V = cfg->vocab_size < 0 ? -cfg->vocab_size : cfg->vocab_size;
    m->cfg.vocab_size = m->V;
    m->untied = w->wcls != NULL;
    m->D = cfg->dim; m->F = cfg->hidden_dim; m->L = cfg->n_layers;
    m->H = cfg->n_heads; m->Hkv = cfg->n_kv_heads;
    m->hd = m->D / m->H;
    m->NQ = m->H * m->hd;
    m->NKV = m->Hkv * m->hd;
    if ((m->hd != 64 && m->hd != 128) || !supported_k(m->D) || m->D == 5632 || !supported_k(m->F)) {
        fprintf(stderr, "stories_lm: unsupported shape dim=%d hidden=%d head_dim=%d "
                "(need head_dim 64/128, dim in {256,512,768,1024,2048}, hidden also 5632)\n",
                m->D, m->F, m->hd);
        FAIL(LM_ERR_UNSUPPORTED);
    }
    if (max_seq > (1 << 16) || max_batch > 4096) FAIL(LM_ERR_RANGE);
    m->max_batch = max_batch;
    m->max_seq = max_seq;
    m->cls_nblk = lmk_cls_nblk(m->V);
    m->use_graph = 1;

    const size_t D = m->D, F = m->F, NQ = m->NQ, NKV = m->NKV, V = m->V, L = m->L;
    m->off_wo = (NQ + 2 * NKV) * D;
    m->off_w13 = m->off_wo + D * NQ;
    m->off_w2 = m->off_w13 + 2 * F * D;
    m->layer_elems = m->off_w2 + D * F;
    m->kv_layer_elems = (size_t)max_batch * m->Hkv * max_seq * m->hd;
    const size_t NB = (size_t)max_batch;
    m->step_graph = (hipGraphExec_t(*)[STEP_KINDS][CTX_CLASSES])calloc(NB + 1, sizeof(*m->step_graph));
    if (!m->step_graph) FAIL(LM_ERR_OOM);

    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) FAIL(LM_ERR_HIP);
    if (hipEventCreate(&m->ev0) != hipSuccess || hipEventCreate(&m->ev1) != hipSuccess ||
        hipEventCreateWithFlags(&m->ev_hand, hipEventDisableTiming) != hipSuccess)
        FAIL(LM_ERR_HIP);
    if ((st = dev_alloc((void **)&m->d_layers, L * m->layer_elems * 2))) goto fail;
    if ((st = dev_alloc((void **)&m->d_embed, V * D * 2))) goto fail;
    if (m->untied) {
        if ((st = dev_alloc((void **)&m->d_wcls, V * D * 2))) goto fail;
    } else {
        m->d_wcls = m->d_embed;
    }
    if ((st = dev_alloc((void **)&m->d_rms_att, L * D * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_rms_ffn, L * D * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_rms_final, D * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_rope_cos, (size_t)max_seq * m->hd / 2 * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_rope_sin, (size_t)max_seq * m->hd / 2 * 4))) goto fail;
    if ((st = alloc_kv(m))) goto fail;
    if ((st = alloc_rows(m, max_batch))) goto fail;
    if ((st = dev_alloc((void **)&m->d_tok, NB * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_pos, NB * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_slot_id, NB * 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_hist, (size_t)max_batch * (max_seq + 1) * 4))) goto fail;
    const size_t ntag = LM_TAG_WORDS(NQ, NKV, D, F);
    if ((st = dev_alloc((void **)&m->d_tagged, ntag * 8))) goto fail;
    const size_t ncls = (size_t)2 * LM_TAG_B * m->cls_nblk;
    if ((st = dev_alloc((void **)&m->d_cls_tw, ncls * 8))) goto fail;
    if ((st = dev_alloc((void **)&m->d_epoch, 4))) goto fail;
    if ((st = dev_alloc((void **)&m->d_err, 8))) goto fail;   /* flag, wait limit (us) */
    if (hipMemset(m->d_tagged, 0, ntag * 8) != hipSuccess || hipMemset(m->d_cls_tw, 0, ncls * 8) != hipSuccess ||
        hipMemset(m->d_epoch, 0, 4) != hipSuccess || hipMemset(m->d_err, 0, 4) != hipSuccess)
        FAIL(LM_ERR_HIP);
    {
        const int lim_us = LM_HANDOFF_US;
        if (hipMemcpy(m->d_err + 1, &lim_us, 4, hipMemcpyHostToDevice) != hipSuccess) FAIL(LM_ERR_HIP);
    }
    m->fuse_qa = 3;
    m->layer_wgs = 2;
    m->prefill_fold = 1;
    m->give_floats = NB * V > GIVE_MIN_FLOATS ? NB * V : GIVE_MIN_FLOATS;
    if ((st = host_alloc((void **)&m->h_logits, (void **)&m->dh_logits, m->give_floats * 4))) goto fail;
    {
        const size_t nflag = (size_t)2 * LM_GIVE_WGS * LM_FLAG_STRIDE, nint = LM_CALL_INTS + LM_HDR_INTS + 32;
        if ((st = host_alloc((void **)&m->h_flag, (void **)&m->dh_flag, (nflag + nint) * 4))) goto fail;
        memset(m->h_flag, 0, (nflag + nint) * 4);
        m->h_call = m->h_flag + nflag;
        m->dh_call = m->dh_flag + nflag;
        m->h_hdr = m->h_call + (LM_CALL_INTS + 15) / 16 * 16;
        m->dh_hdr = m->dh_call + (LM_CALL_INTS + 15) / 16 * 16;
    }
    if ((st = dev_alloc((void **)&m->d_seq, 4))) goto fail;
    if (hipHostMalloc((void **)&m->h_io, (size_t)4 * (max_batch + 1) * 4, 0) != hipSuccess) FAIL(LM_ERR_OOM);
    memset(m->h_io, 0, (size_t)4 * (max_batch + 1) * 4);
    /* RESNORM's overflow flag: the int after the hand-off flag's slot, written
     * by the device only when a prefill row overflows */
    if (hipHostGetDevicePointer((void **)&m->d_ovf, m->h_io + 4 * (size_t)max_batch + 1, 0) != hipSuccess)
        FAIL(LM_ERR_HIP);

    if ((st = upload_weights(m, w))) goto fail;
    {
        size_t n = (size_t)max_seq * m->hd / 2;
        float *c = (float *)malloc(n * 4), *s = (float *)malloc(n * 4);
        if (!c || !s) { free(c); free(s); FAIL(LM_ERR_OOM); }
        lm_rope_table(max_seq, m->hd, c, s);
        hipError_t e1 = hipMemcpy(m->d_rope_cos, c, n * 4, hipMemcpyHostToDevice);
        hipError_t e2 = hipMemcpy(m->d_rope_sin, s, n * 4, hipMemcpyHostToDevice);
        free(c); free(s);
        if (e1 != hipSuccess || e2 != hipSuccess) FAIL(LM_ERR_HIP);
    }
    if (hipMemset(m->d_hist, 0, (size_t)max_batch * (max_seq + 1) * 4) != hipSuccess ||
        hipMemset(m->d_pos, 0, NB * 4) != hipSuccess || hipMemset(m->d_tok, 0, NB * 4) != hipSuccess)
        FAIL(LM_ERR_HIP);
    {
        int *ids = (int *)malloc(NB * 4);
        if (!ids) FAIL(LM_ERR_OOM);
        for (int b = 0; b < max_batch; b++) ids[b] = b;
        hipError_t e = hipMemcpy(m->d_slot_id, ids, NB * 4, hipMemcpyHostToDevice);
        free(ids);
        if (e != hipSuccess) FAIL(LM_ERR_HIP);
    }
    if (hipDeviceSynchronize() != hipSuccess) FAIL(LM_ERR_HIP);
    if (status) *status = LM_OK;
    return m;
fail:
    if (status) *status = st;
    if (st != LM_OK) fprintf(stderr, "stories_lm: lm_create failed: %s\n", lm_strerror(st));
    lm_free(m);
    return NULL;
#undef FAIL
}

LMModel *lm_load_llama2c(const char *path, int max_batch, int max_seq, int *status)
{
    if (!path) {
        if (status) *status = LM_ERR_INVALID;
        return NULL;
    }
    Config cfg;
    int untied = 0;
    float *data = NULL;
    int rc = lmh_read_llama2c(path, &cfg, &untied, &data);
    if (rc) {
        if (status) *status = rc;
        return NULL;
    }
    LMWeights w;
    lm_weights_view(&cfg, LM_DTYPE_F32, data, untied, &w);
    LMModel *m = lm_create(&cfg, &w, max_batch, max_seq, status);
    free(data);
    return m;
}

LMModel *lm_load_blzt(const char *path, int max_batch, int max_seq, int *status)
{
    if (!path) {
        if (status) *status = LM_ERR_INVALID;
        return NULL;
    }
    Config cfg;
    float *data = NULL;
    int rc = lmh_read_blzt(path, &cfg, &data);
    if (rc) {
        if (status) *status = rc;
        return NULL;
    }
    LMWeights w;
    lm_weights_view(&cfg, LM_DTYPE_F32, data, 0, &w);
    LMModel *m = lm_create(&cfg, &w, max_batch, max_seq, status);
    free(data);
    return m;
}

/* Launches that hold hand-off waits (the batch 1-4 decode chain at fusion
 * levels 1-4) rely on in-order dispatch of their own work-groups on each XCD:
 * a launch's lowest unfinished work-group always finds its producers done or
 * running.  Two such launches of different handles in flight at once could
 * each hold the slots the other's lowest pending work-group needs.  So their
 * launches are ordered on the device: under g_hand_mu, a handle's stream first
 * waits for the last hand-off launches any other handle enqueued (g_hand_last),
 * then enqueues its own and records ev_hand, which becomes g_hand_last.  The
 * rest of the work of distinct handles (prefill, batched decode, copies) still
 * runs concurrently. */
static pthread_mutex_t g_hand_mu = PTHREAD_MUTEX_INITIALIZER;
static LMModel *g_hand_owner;   /* handle whose ev_hand g_hand_last is */

static int handoff_enter(LMModel *m)
{
    pthread_mutex_lock(&g_hand_mu);
    if (g_hand_owner && g_hand_owner != m &&
        hipStreamWaitEvent(m->stream, g_hand_owner->ev_hand, 0) != hipSuccess) {
        pthread_mutex_unlock(&g_hand_mu);
        fprintf(stderr, "stories_lm: hipStreamWaitEvent on another handle's decode failed\n");
        return LM_ERR_HIP;
    }
    return LM_OK;
}

/* rc: the status of what was enqueued since handoff_enter (passed through) */
static int handoff_leave(LMModel *m, int rc)
{
    if (hipEventRecord(m->ev_hand, m->stream) == hipSuccess) {
        g_hand_owner = m;
    } else {
        g_hand_owner = NULL;   /* nothing later waits on an unrecorded event */
        if (rc == LM_OK) rc = LM_ERR_HIP;
    }
    pthread_mutex_unlock(&g_hand_mu);
    return rc;
}

/* A handle being freed (its stream already synchronised) leaves the chain. */
static void handoff_forget(LMModel *m)
{
    pthread_mutex_lock(&g_hand_mu);
    if (g_hand_owner == m) g_hand_owner = NULL;
    pthread_mutex_unlock(&g_hand_mu);
}

void lm_free(LMModel *m)
{
    if (!m) return;
    if (m->stream) hipStreamSynchronize(m->stream);
    crew_end(&m->crew);
    handoff_forget(m);
    drop_graphs(m);
    free(m->step_graph);
    free_rows(m);
    void *dev[] = {m->d_layers, m->d_embed, m->untied ? m->d_wcls : NULL, m->d_rms_att,
                   m->d_rms_ffn, m->d_rms_final, m->d_rope_cos, m->d_rope_sin, m->d_kc,
                   m->d_vc, m->d_tok, m->d_pos, m->d_hist, m->d_slot_id, m->d_tagged, m->d_cls_tw, m->d_epoch,
                   m->d_err, m->d_seq};
    for (size_t i = 0; i < sizeof(dev) / sizeof(dev[0]); i++)
        if (dev[i]) hipFree(dev[i]);
    if (m->h_logits) hipHostFree(m->h_logits);
    if (m->h_io) hipHostFree(m->h_io);
    if (m->h_flag) hipHostFree(m->h_flag);
    if (m->ev0) hipEventDestroy(m->ev0);
    if (m->ev1) hipEventDestroy(m->ev1);
    if (m->ev_hand) hipEventDestroy(m->ev_hand);
    if (m->stream) hipStreamDestroy(m->stream);
    free(m);
}

int lm_get_config(const LMModel *m, Config *out)
{
    if (!m || !out) return LM_ERR_INVALID;
    *out = m->cfg;
    return LM_OK;
}

int lm_set_option(LMModel *m, int option, int value)
{
    if (!m) return LM_ERR_INVALID;
    switch (option) {
    case LM_OPT_USE_GRAPH:
        m->use_graph = value ? 1 : 0;
        return LM_OK;
    case LM_OPT_FUSE_QKV_ATTN:
        if (value < 0 || value > 4) return LM_ERR_INVALID;
        if (value == m->fuse_qa) return LM_OK;
        HIPCHK(hipStreamSynchronize(m->stream));
        drop_graphs(m);
        m->fuse_qa = value;
        return LM_OK;
    case LM_OPT_LAYER_WGS:
        if (value < 0 || value > 4) return LM_ERR_INVALID;
        if (value == m->layer_wgs) return LM_OK;
        HIPCHK(hipStreamSynchronize(m->stream));
        drop_graphs(m);
        m->layer_wgs = value;
        return LM_OK;
    case LM_OPT_PREFILL_FOLD:
        if (value != 0 && value != 1) return LM_ERR_INVALID;
        if (value == m->prefill_fold) return LM_OK;
        HIPCHK(hipStreamSynchronize(m->stream));
        drop_graphs(m);
        m->prefill_fold = value;
        return LM_OK;
    case LM_OPT_HANDOFF_US:
        if (value < 1) return LM_ERR_INVALID;
        HIPCHK(hipStreamSynchronize(m->stream));
        HIPCHK(hipMemcpy(m->d_err + 1, &value, 4, hipMemcpyHostToDevice));
        return LM_OK;
    case LM_OPT_HANDOFF_ABORT:
        /* raise the give-up flag from the host: every hand-off wait of the
         * next call ends at once (the kernels still run to their end) and
         * the call reports LM_ERR_HIP, then clears the flag */
        if (value != 1) return LM_ERR_INVALID;
        HIPCHK(hipStreamSynchronize(m->stream));
        HIPCHK(hipMemcpy(m->d_err, &value, 4, hipMemcpyHostToDevice));
        return LM_OK;
    case LM_OPT_KV_F32:
        if ((value ? 1 : 0) == m->kv_f32) return LM_OK;
        HIPCHK(hipStreamSynchronize(m->stream));
        drop_graphs(m);
        m->kv_f32 = value ? 1 : 0;
        return alloc_kv(m);
    default:
        return LM_ERR_INVALID;
    }
}

/* ------------------------------------------------------------------------- */
/* decode step                                                                */
/* ------------------------------------------------------------------------- */

#define KCHK(call)                                                                    \
    do {                                                                              \
        int e_ = (call);                                                              \
        if (e_ != 0) {                                                                \
            fprintf(stderr, "stories_lm: launch %s failed: %s\n", #call,              \
                    hipGetErrorString((hipError_t)e_));                               \
            return LM_ERR_HIP;                                                        \
        }                                                                             \
    } while (0)

/* The decode chain's fusion level for B rows: fuse_qa, where 3 takes the
 * whole-layer launch for one row only (B = 2 and 4 ran faster at level 2:
 * 203 and 281 us/step against 207 and 385) and 4 takes it for every batch;
 * the whole-layer launch is built only for the (dim, hidden) pairs and
 * batches lmk_layer_fusable names, and level 2 runs elsewhere. */
static int chain_level(const LMModel *m, int B)
{
    int lvl = m->fuse_qa;
    if (lvl == 3 && B > 1) lvl = 2;
    if (lvl == 4) lvl = 3;
    return lvl == 3 && !lmk_layer_fusable(m->D, m->F, B) ? 2 : lvl;
}

/* Context class of batch 1-4 decode rows whose largest position is p: class 0
 * up to 512 cached positions, then one more per doubling (the last for any
 * more).  From class 1 the chain splits a head's positions over attn_split
 * work-groups, so that each of their waves has at most two tiles of 32, which
 * it holds before its wait for q, k, v.  One work-group per head stays up to
 * 512: with two, the whole-layer launch of Stories measured 12.6 against 12.1
 * us at 350 positions and 12.6 against 12.8 at 500 (the merge costs one more
 * hand-off), while 1900 positions took 23.6 us unsplit and 14.3 split over 8.
 * The class is fixed when a graph is captured, so each has its own graph; where
 * no form of the chain splits (levels 0 and 1, the whole-layer launch of more
 * rows than one, the MFMA path) every length is class 0. */
static int ctx_class(int p)
{
    int c = 0;
    while (c < CTX_CLASSES - 1 && p > (512 << c)) c++;
    return c;
}

static int ctx_class_rows(const LMModel *m, const int *pos, int B, int more)
{
    int p = 0;
    const int lvl = B <= MAX_GEMV_B ? chain_level(m, B) : 0;
    if (lvl < 2 || (lvl > 2 && B > 1)) return 0;
    for (int b = 0; b < B; b++)
        if (pos[b] > p) p = pos[b];
    return ctx_class(p + more);
}

/* Work-groups per head of a context class: 1, 4, 8, 16. */
static int attn_split(int cls) { return cls ? 2 << cls : 1; }

/* Whether kernel family fam runs inside another family's launch at fusion
 * level lvl (the QKV launch; at level 3 the argmax inside the classifier's). */
static int fam_inside(int fam, int lvl)
{
    return (fam == LM_KERN_ATTN && lvl >= 1) || (fam == LM_KERN_WO && lvl >= 2) ||
           ((fam == LM_KERN_W13 || fam == LM_KERN_W2 || fam == LM_KERN_ARGMAX) && lvl >= 3);
}

/* Queue the kernel of family `fam` (LM_KERN_*) of layer l for rows 0..B-1
 * (nothing for a family that runs inside the QKV launch). */
static int enqueue_kernel(LMModel *m, int B, int fam, int l, float *logits)
{
    const int lvl = chain_level(m, B);
    if (fam_inside(fam, lvl)) return LM_OK;
    hipStream_t s = m->stream;
    const int D = m->D, F = m->F;
    const uint16_t *lw = m->d_layers + (size_t)l * m->layer_elems;
    const size_t kvo = (size_t)l * m->kv_layer_elems * (m->kv_f32 ? 4 : 2);
    void *kc = (char *)m->d_kc + kvo, *vc = (char *)m->d_vc + kvo;
    switch (fam) {
    case LM_KERN_QKV:
        if (lvl)   /* with the attention of every head (Wo from level 2, the FFN at 3) */
            KCHK(lmk_qkv_attn(s, m->d_x, l == 0 ? m->d_embed : NULL, m->d_tok,
                              m->d_rms_att + (size_t)l * D, lw, D, m->NQ, m->NKV, m->hd,
                              m->d_rope_cos, m->d_rope_sin, m->d_pos, B, kc, vc, m->kv_f32,
                              m->max_seq, m->H, m->d_tagged, m->d_epoch, l, m->L, m->d_err,
                              m->d_attn, lvl >= 2 ? lw + m->off_wo : NULL,
                              m->d_rms_ffn + (size_t)l * D, lvl == 3 ? lw + m->off_w13 : NULL,
                              lw + m->off_w2, F, m->layer_wgs, attn_split(m->ctx_cls)));
        else
            KCHK(lmk_qkv_rope(s, m->d_x, l == 0 ? m->d_embed : NULL, m->d_tok,
                              m->d_rms_att + (size_t)l * D, lw, D, m->NQ, m->NKV, m->hd,
                              m->d_rope_cos, m->d_rope_sin, m->d_pos, B, m->d_q, kc, vc, m->kv_f32,
                              m->max_seq));
        break;
    case LM_KERN_ATTN:
        KCHK(lmk_attn_decode(s, m->d_q, kc, vc, m->kv_f32, m->d_pos, NULL, B, m->H, m->Hkv,
                             m->hd, m->max_seq, m->d_attn, NULL));
        break;
    case LM_KERN_WO:
        KCHK(lmk_wo_residual(s, m->d_attn, lw + m->off_wo, D, B, m->d_x));
        break;
    case LM_KERN_W13:
        KCHK(lmk_ffn13(s, m->d_x, m->d_rms_ffn + (size_t)l * D, lw + m->off_w13, D, F, B, m->d_g));
        break;
    case LM_KERN_W2:
        KCHK(lmk_w2_residual(s, m->d_g, lw + m->off_w2, D, F, B, m->d_x));
        break;
    case LM_KERN_CLS:
        KCHK(lmk_cls(s, m->d_x, m->d_rms_final, m->d_wcls, D, m->V, B, logits, m->d_amax,
                     lvl == 3 ? m->d_cls_tw : NULL, m->d_epoch, m->d_tok, m->d_pos, m->d_hist,
                     m->max_seq + 1, m->d_err));
        break;
    case LM_KERN_ARGMAX:
        KCHK(lmk_argmax_final(s, m->d_amax, m->cls_nblk, B, m->d_tok, m->d_pos, m->d_hist,
                              m->max_seq + 1, m->d_epoch));
        break;
    default:
        return LM_ERR_INVALID;
    }
    return LM_OK;
}

/* Queue one decode step for rows 0..B-1 (tokens in d_tok, positions in d_pos);
 * logits go to `logits` (device, B x V, may be NULL), the argmax to d_tok, and
 * the history/position advance to d_hist/d_pos. */
static int enqueue_decode_gemv(LMModel *m, int B, float *logits)
{
    static const int fams[5] = {LM_KERN_QKV, LM_KERN_ATTN, LM_KERN_WO, LM_KERN_W13, LM_KERN_W2};
    int rc;
    for (int l = 0; l < m->L; l++)
        for (int f = 0; f < 5; f++)
            if ((rc = enqueue_kernel(m, B, fams[f], l, NULL))) return rc;
    if ((rc = enqueue_kernel(m, B, LM_KERN_CLS, 0, logits))) return rc;
    return enqueue_kernel(m, B, LM_KERN_ARGMAX, 0, NULL);
}

/* ------------------------------------------------------------------------- */
/* MFMA path: prefill rows and decode batches above MAX_GEMV_B                 */
/* ------------------------------------------------------------------------- */

/* Largest decode batch of the MFMA decode step (one 64-row tile). */
#define MAX_GEMM_B 64
/* Rows per prefill chunk (whole sequences). */
#define PREFILL_ROWS 2048

/* Whether M rows take the fused projections of k_rows.hip: up to 64 rows of
 * models up to 1024 wide.  Each work-group there reads its 16 rows whole, which
 * at width 2048 (131 KB of x beside 64 KB of weights) costs more than the
 * launches it saves: QKV + gate 10.3 + 13.0 us at 12 rows against 3.7 + 8.4 +
 * 3.7 + 12.5 for the row norms and tiled GEMMs, W2 (K 5632) 12.5 against 6. */
static int rows_fused(const LMModel *m, int M) { return M <= 64 && m->D <= 1024 && m->F <= 2048; }

/* Queue the layers for M rows (row r: token tok[r], position pos[r], cache slot
 * slot[r]; the K/V of every row is appended to the cache before attention, so
 * rows of one sequence attend causally to each other; seq_rows > 1: the rows
 * are whole sequences of seq_rows rows, attended by the MFMA prefill kernel,
 * else one row per slot, by the decode kernel), then the final rmsnorm +
 * classifier of the rows: logits to `logits` (decode: may be NULL) and, for
 * decode rows, the argmax partials to d_amax.  last (prefill, seq_rows > 1):
 * the logits of each sequence's last row only.  The last layer then owes every
 * row its K and V but nothing after them: once QKV has run, the last rows'
 * q and residual are gathered (k_last_rows), attended by the decode kernel,
 * and only they go on through Wo, the FFN and the classifier; their positions
 * and slots are in lpos and lslot. */
static int enqueue_rows(LMModel *m, int M, int seq_rows, const int *tok, const int *pos,
                        const int *slot, float *logits, const int *lpos, const int *lslot)
{
    hipStream_t s = m->stream;
    const int D = m->D, F = m->F, NQ = m->NQ, NKV = m->NKV, NQKV = NQ + 2 * NKV;
    const int last = lpos != NULL;
    float *x = m->d_x;
    size_t sx = (size_t)M * D;   /* split stride of a [M, D] partial */
    /* Wo and W2 write their product, not x: into d_part as fp32 (decode rows
     * (M <= 64) run these narrow projections K-split, one partial per split),
     * and the row norm that next reads x adds it (the residual add).  Only
     * unsplit decode rows keep the residual add in the GEMM epilogue. */
    int dec = M <= 64;
    const int ns_qkv = dec && seq_rows == 1 ? lmk_pick_split(M, NQKV, D) : 1;
    int ns_wo = lmk_pick_split(M, D, NQ);
    int ns_w2 = lmk_pick_split(M, D, F);
    int sep_wo = !dec || ns_wo > 1, sep_w2 = !dec || ns_w2 > 1;
    /* Beyond 64 rows, an unsplit Wo or W2 folds the row norm that follows it
     * into the GEMMs: it adds its product to x and writes u = fp16(x * gain)
     * and the sums of squares of x per 32 columns (RESNORM), and the GEMM that
     * reads u scales its product rows by 1/sqrt(mean(x^2) + 1e-5), which
     * distributes over the row's dot products.  That saves the row-norm
     * launch and the product's round trip through memory.  K-split
     * projections keep the row norm, which adds their partials (an unsplit
     * 2048-row W2 took 20 us against 14 + 5.6 for the split and the norm);
     * so do layer 0 (embedding) and the classifier.  Only prefill rows fold
     * (LM_OPT_PREFILL_FOLD): u is rounded to fp16 before the row is
     * normalised, and a prefill chunk whose u overflows is redone with the
     * row norm apart (run_prefill); decode rows have no such retry. */
    const int may_fold = seq_rows > 1 && m->prefill_fold && !m->fold_off && D % 128 == 0 && D / 32 <= 64;
    int fold_wo = may_fold && !dec && ns_wo == 1, fold_w2 = may_fold && !dec && ns_w2 == 1;
    int rs_next = 0;                   /* x's norm is pending in u for QKV */
    const float *pend = NULL;          /* W2 partials not yet added to x */
    int pend_ns = 0;
    int fused = rows_fused(m, M);      /* (also once the last rows are alone) */
    LMEpilogue ep;
    for (int l = 0; l < m->L; l++) {
        const uint16_t *lw = m->d_layers + (size_t)l * m->layer_elems;
        const size_t kvo = (size_t)l * m->kv_layer_elems * (m->kv_f32 ? 4 : 2);
        void *kc = (char *)m->d_kc + kvo, *vc = (char *)m->d_vc + kvo;
        const float *rs = rs_next ? m->d_ss : NULL;   /* u's row scale */
        if (!rs && !fused)
            KCHK(lmk_rownorm(s, m->d_x, D, M, l == 0 ? m->d_embed : NULL, tok, pend, pend_ns, sx,
                             m->d_rms_att + (size_t)l * D, m->d_xn16));
        pend = NULL;
        pend_ns = 0;
        const int split_qkv = ns_qkv > 1 && !fused;
        if (fused) {
            KCHK(lmk_rows_qkv(s, x, l == 0 ? m->d_embed : NULL, tok, m->d_rms_att + (size_t)l * D, lw, D,
                              M, NQ, NKV, m->hd, m->d_rope_cos, m->d_rope_sin, pos, slot, m->d_q, kc, vc,
                              m->kv_f32, m->max_seq));
        } else if (split_qkv) {
            /* decode rows, too few column tiles to fill the CUs: K-split QKV;
             * the attention kernel sums the partials, applies RoPE and appends
             * K/V itself */
            KCHK(lmk_gemm_split(s, m->d_xn16, D, lw, M, NQKV, D, ns_qkv, m->d_part));
            KCHK(lmk_attn_decode_part(s, m->d_part, (size_t)M * NQKV, ns_qkv, NQ, NKV, pos, slot, M,
                                      m->H, m->Hkv, m->hd, m->max_seq, m->d_rope_cos,
                                      m->d_rope_sin, kc, vc, m->kv_f32, m->d_a16));
        } else {
            /* QKV with RoPE and the K/V append in the GEMM epilogue (staged
             * through LDS and stored row-contiguously) */
            memset(&ep, 0, sizeof(ep));
            ep.q = m->d_q; ep.kc = kc; ep.vc = vc; ep.kv_f32 = m->kv_f32;
            ep.NQ = NQ; ep.NKV = NKV; ep.hd = m->hd; ep.Hkv = m->Hkv; ep.max_seq = m->max_seq;
            ep.slot = slot; ep.pos = pos; ep.rope_cos = m->d_rope_cos; ep.rope_sin = m->d_rope_sin;
            ep.rs_ss = rs; ep.nss = D / 32;
            KCHK(lmk_gemm(s, m->d_xn16, D, lw, M, NQKV, D, LMK_EPI_QKV, &ep));
        }
        if (split_qkv) {
        } else if (last && l == m->L - 1) {
            /* from here on the sequences' last rows alone, in d_attn (which
             * holds no prefill rows otherwise): residual, then q */
            const int n = M / seq_rows;
            x = m->d_attn;
            float *lq = x + (size_t)n * D;
            KCHK(lmk_last_rows(s, m->d_x, m->d_q, D, NQ, seq_rows, n, x, lq));
            M = n;
            sx = (size_t)M * D;
            dec = M <= 64;
            fused = rows_fused(m, M);
            ns_wo = lmk_pick_split(M, D, NQ);
            ns_w2 = lmk_pick_split(M, D, F);
            sep_wo = !dec || ns_wo > 1;
            sep_w2 = !dec || ns_w2 > 1;
            fold_wo = may_fold && !dec && ns_wo == 1;
            fold_w2 = may_fold && !dec && ns_w2 == 1;
            KCHK(lmk_attn_decode(s, lq, kc, vc, m->kv_f32, lpos, lslot, M, m->H, m->Hkv, m->hd,
                                 m->max_seq, NULL, m->d_a16));
        } else if (seq_rows > 1) {
            KCHK(lmk_attn_prefill(s, m->d_q, kc, vc, m->kv_f32, pos, slot, seq_rows,
                                  M / seq_rows, m->H, m->Hkv, m->hd, m->max_seq, m->d_a16));
        } else {
            KCHK(lmk_attn_decode(s, m->d_q, kc, vc, m->kv_f32, pos, slot, M, m->H, m->Hkv, m->hd,
                                 m->max_seq, NULL, m->d_a16));
        }
        if (fused) {   /* the rest of the layer in three launches */
            KCHK(lmk_rows_res(s, m->d_a16, lw + m->off_wo, D, NQ, M, x));
            KCHK(lmk_rows_gate(s, x, m->d_rms_ffn + (size_t)l * D, lw + m->off_w13, D, F, M, m->d_g16));
            KCHK(lmk_rows_res(s, m->d_g16, lw + m->off_w2, D, F, M, x));
            continue;
        }
        if (fold_wo) {
            memset(&ep, 0, sizeof(ep));
            ep.out = x; ep.ldc = D;
            ep.gain = m->d_rms_ffn + (size_t)l * D; ep.u = m->d_xn16; ep.ss = m->d_ss; ep.nss = D / 32;
            ep.ovf = m->d_ovf;
            KCHK(lmk_gemm(s, m->d_a16, NQ, lw + m->off_wo, M, D, NQ, LMK_EPI_RESNORM, &ep));
        } else if (sep_wo) {
            if (ns_wo > 1) {
                KCHK(lmk_gemm_split(s, m->d_a16, NQ, lw + m->off_wo, M, D, NQ, ns_wo, m->d_part));
            } else {
                memset(&ep, 0, sizeof(ep));
                ep.out = m->d_part; ep.ldc = D;
                KCHK(lmk_gemm(s, m->d_a16, NQ, lw + m->off_wo, M, D, NQ, LMK_EPI_STORE, &ep));
            }
            KCHK(lmk_rownorm(s, x, D, M, NULL, NULL, m->d_part, ns_wo, sx,
                             m->d_rms_ffn + (size_t)l * D, m->d_xn16));
        } else {
            memset(&ep, 0, sizeof(ep));
            ep.out = x; ep.ldc = D;
            KCHK(lmk_gemm(s, m->d_a16, NQ, lw + m->off_wo, M, D, NQ, LMK_EPI_RESID, &ep));
            KCHK(lmk_rownorm(s, x, D, M, NULL, NULL, NULL, 0, 0,
                             m->d_rms_ffn + (size_t)l * D, m->d_xn16));
        }
        memset(&ep, 0, sizeof(ep));
        ep.g = m->d_g16; ep.F = F;
        if (fold_wo) { ep.rs_ss = m->d_ss; ep.nss = D / 32; }
        KCHK(lmk_gemm(s, m->d_xn16, D, lw + m->off_w13, M, 2 * F, D, LMK_EPI_GATE, &ep));
        rs_next = fold_w2 && l + 1 < m->L;
        if (fold_w2) {
            memset(&ep, 0, sizeof(ep));
            ep.out = x; ep.ldc = D;
            if (l + 1 < m->L) {   /* u of the next layer's attention norm */
                ep.gain = m->d_rms_att + (size_t)(l + 1) * D; ep.u = m->d_xn16; ep.ss = m->d_ss;
                ep.nss = D / 32; ep.ovf = m->d_ovf;
            }
            KCHK(lmk_gemm(s, m->d_g16, F, lw + m->off_w2, M, D, F,
                          l + 1 < m->L ? LMK_EPI_RESNORM : LMK_EPI_RESID, &ep));
        } else if (sep_w2) {
            if (ns_w2 > 1) {
                KCHK(lmk_gemm_split(s, m->d_g16, F, lw + m->off_w2, M, D, F, ns_w2, m->d_part));
            } else {
                memset(&ep, 0, sizeof(ep));
                ep.out = m->d_part; ep.ldc = D;
                KCHK(lmk_gemm(s, m->d_g16, F, lw + m->off_w2, M, D, F, LMK_EPI_STORE, &ep));
            }
            pend = m->d_part;
            pend_ns = ns_w2;
        } else {
            memset(&ep, 0, sizeof(ep));
            ep.out = x; ep.ldc = D;
            KCHK(lmk_gemm(s, m->d_g16, F, lw + m->off_w2, M, D, F, LMK_EPI_RESID, &ep));
        }
    }
    KCHK(lmk_rownorm(s, x, D, M, NULL, NULL, pend, pend_ns, sx, m->d_rms_final, m->d_xn16));
    memset(&ep, 0, sizeof(ep));
    ep.out = logits; ep.ldc = m->V; ep.stream_out = 1;
    if (seq_rows > 1) {   /* prefill: logits only */
        KCHK(lmk_gemm(s, m->d_xn16, D, m->d_wcls, M, m->V, D, LMK_EPI_STORE, &ep));
    } else {              /* decode: argmax partials for the greedy step (+ logits) */
        ep.part = m->d_amax;
        KCHK(lmk_gemm(s, m->d_xn16, D, m->d_wcls, M, m->V, D, LMK_EPI_ARGMAX, &ep));
    }
    return LM_OK;
}

/* One greedy decode step of rows 0..B-1 on the MFMA path (slot b = row b). */
static int enqueue_decode_gemm(LMModel *m, int B, float *logits)
{
    int rc = enqueue_rows(m, B, 1, m->d_tok, m->d_pos, m->d_slot_id, logits, NULL, NULL);
    if (rc) return rc;
    KCHK(lmk_argmax_final(m->stream, m->d_amax, m->cls_nblk, B, m->d_tok, m->d_pos, m->d_hist,
                          m->max_seq + 1, NULL));
    return LM_OK;
}

static int enqueue_decode(LMModel *m, int B, float *logits)
{
    return B <= MAX_GEMV_B ? enqueue_decode_gemv(m, B, logits) : enqueue_decode_gemm(m, B, logits);
}

/* Greedy steps captured per multi-step graph. */
#define GRAPH_STEPS 16

/* Work-groups that give n floats to the host: 4 KiB each, as many as there
 * are flags. */
static int give_wgs(size_t n)
{
    const size_t w = (n + 1023) / 1024;
    return w < 1 ? 1 : w > LM_GIVE_WGS ? LM_GIVE_WGS : (int)w;
}

/* Queue the decode steps of `kind` for rows 0..B-1.  Single steps write the
 * logits to d_logits; multi-step runs only feed the argmax forward. */
static int enqueue_kind(LMModel *m, int B, int kind)
{
    const int call = kind == STEP_LOGITS || kind == STEP_IDS;
    const size_t n = kind == STEP_LOGITS ? (size_t)B * m->V : 0;
    int rc = LM_OK;
    if (call) KCHK(lmk_step_in(m->stream, m->dh_call, m->d_seq, m->d_tok, m->d_pos, B));
    for (int t = 0; t < (kind == STEP_GREEDY_N ? GRAPH_STEPS : 1) && rc == LM_OK; t++)
        rc = enqueue_decode(m, B, kind == STEP_GREEDY_N ? NULL : m->d_logits);
    if (rc || !call) return rc;
    KCHK(lmk_give(m->stream, n ? m->d_logits : NULL, m->dh_logits, n, give_wgs(n), m->d_err, NULL, m->d_tok, B,
                  m->dh_hdr, m->d_seq, 0, m->dh_flag));
    return LM_OK;
}

static int capture_begin(LMModel *m)
{
    HIPCHK(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
    return LM_OK;
}

/* rc: the status of what was queued since capture_begin */
static int capture_end(LMModel *m, int rc, hipGraphExec_t *ge)
{
    hipGraph_t g = NULL;
    hipError_t e = hipStreamEndCapture(m->stream, &g);
    if (rc == LM_OK && e == hipSuccess) e = hipGraphInstantiateWithFlags(ge, g, 0);
    if (g) hipGraphDestroy(g);
    if (rc != LM_OK) return rc;
    HIPCHK(e);
    return LM_OK;
}

/* Run the decode steps of `kind` of rows 0..B-1: launched directly the first
 * time, and captured while the device is busy with them, replayed from then
 * on.  Captured before its launch, a handle's first step kept the device
 * waiting for it: one row of Stories 335 -> 216 us (168 from the second on),
 * three rows 558 -> 378, 32 rows of the 2048-wide model 522 -> 387, a 17-step
 * greedy run 3243 -> 2688. */
static int enqueue_decode_steps(LMModel *m, int B, int kind)
{
    hipGraphExec_t *ge = &m->step_graph[B][kind][m->ctx_cls];
    if (m->use_graph && *ge) {
        HIPCHK(hipGraphLaunch(*ge, m->stream));
        return LM_OK;
    }
    int rc = enqueue_kind(m, B, kind);
    if (rc || !m->use_graph) return rc;
    if ((rc = capture_begin(m))) return rc;
    return capture_end(m, enqueue_kind(m, B, kind), ge);
}

/* Whether the decode step of B rows holds hand-off waits (the batch 1-4
 * chain with QKV and attention in one launch, levels 1-4). */
static int step_waits(const LMModel *m, int B)
{
    return B <= MAX_GEMV_B && chain_level(m, B) >= 1;
}

static int run_decode_steps(LMModel *m, int B, int kind, int cls)
{
    m->ctx_cls = cls;
    if (!step_waits(m, B)) return enqueue_decode_steps(m, B, kind);
    int rc = handoff_enter(m);
    if (rc) return rc;
    return handoff_leave(m, enqueue_decode_steps(m, B, kind));
}

static int check_batch(int B)
{
    if (B <= MAX_GEMM_B) return LM_OK;
    fprintf(stderr, "stories_lm: decode batch %d > %d not supported\n", B, MAX_GEMM_B);
    return LM_ERR_UNSUPPORTED;
}

/* The next call number (never 0 but at a wrap of 2^32; the flags start at 0). */
static int next_seq(LMModel *m) { return m->seq = (int)((unsigned)m->seq + 1u); }

/* Wait until flag k of set `set` carries `seq`: the share of that work-group
 * of a give kernel has landed.  Polled, since a stream synchronise returns
 * about 8 us later; now and then the stream is asked, so that work that ended
 * without raising the flag (a failed launch) ends the wait as well. */
static int wait_flag(LMModel *m, int set, int k, int seq)
{
    const int *f = m->h_flag + ((size_t)set * LM_GIVE_WGS + k) * LM_FLAG_STRIDE;
    for (unsigned spin = 1; __atomic_load_n(f, __ATOMIC_ACQUIRE) != seq; spin++) {
        __builtin_ia32_pause();
        if (spin & 4095) continue;
        const hipError_t e = hipStreamQuery(m->stream);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();   /* (not an error of a launch to come) */
            sched_yield();
            continue;
        }
        if (e == hipSuccess && __atomic_load_n(f, __ATOMIC_ACQUIRE) == seq) break;
        fprintf(stderr, "stories_lm: results did not arrive: %s\n", hipGetErrorString(e));
        return LM_ERR_HIP;
    }
    return LM_OK;
}

static size_t crew_len(const Crew *c, size_t i) { return (i + 1) * c->seg < c->n ? c->seg : c->n - i * c->seg; }

static void crew_take(Crew *c, int t, size_t i)
{
    const size_t len = crew_len(c, i);
    const int wgs = give_wgs(len);
    const size_t per = LM_GIVE_PER(len, wgs);
    const float *src = c->m->h_logits + (i & 1) * c->seg;
    for (int k = t; k < wgs && __atomic_load_n(&c->rc, __ATOMIC_RELAXED) == LM_OK; k += c->nt) {
        const int st = wait_flag(c->m, (int)(i & 1), k, (int)((unsigned)c->seq0 + (unsigned)i));
        const size_t a = per * k, e = a + per < len ? a + per : len;
        if (st) __atomic_store_n(&c->rc, st, __ATOMIC_RELAXED);
        else if (c->dst && a < e) memcpy(c->dst + i * c->seg + a, src + a, (e - a) * 4);
    }
    __atomic_store_n(&c->prog[t], (int)i + 1, __ATOMIC_RELEASE);
}

/* Spin until *p >= want (0) or the crew has failed (its status). */
static int crew_wait(Crew *c, const int *p, int want)
{
    for (unsigned spin = 1; __atomic_load_n(p, __ATOMIC_ACQUIRE) < want; spin++) {
        const int rc = __atomic_load_n(&c->rc, __ATOMIC_RELAXED);
        if (rc) return rc;
        __builtin_ia32_pause();
        if (!(spin & 4095)) sched_yield();
    }
    return LM_OK;
}

static void *crew_hand(void *arg)
{
    struct CrewHand *h = (struct CrewHand *)arg;
    Crew *c = (Crew *)h->crew;
    for (;;) {
        while (sem_wait(&h->go) != 0) { }   /* (EINTR) */
        if (c->quit) return NULL;
        for (size_t i = 0; i < c->nseg && crew_wait(c, &c->issued, (int)i + 1) == LM_OK; i++)
            crew_take(c, h->t, i);
        __atomic_store_n(&c->prog[h->t], INT_MAX, __ATOMIC_RELEASE);   /* done with this call */
    }
}

/* The handle's threads, as many as could be made (up to CREW_MAX - 1). */
static int crew_hands(Crew *c)
{
    const int want = omp_get_max_threads() < CREW_MAX ? omp_get_max_threads() - 1 : CREW_MAX - 1;
    while (c->hands < want) {
        struct CrewHand *h = &c->hand[c->hands];
        h->crew = c;
        h->t = c->hands + 1;
        if (sem_init(&h->go, 0, 0) != 0) break;
        if (pthread_create(&h->id, NULL, crew_hand, h) != 0) {
            sem_destroy(&h->go);
            break;
        }
        c->hands++;
    }
    return c->hands < want ? c->hands : want;
}

static void crew_end(Crew *c)
{
    c->quit = 1;
    for (int i = 0; i < c->hands; i++) {
        sem_post(&c->hand[i].go);
        pthread_join(c->hand[i].id, NULL);
        sem_destroy(&c->hand[i].go);
    }
    c->hands = 0;
}

/* n floats of results to the caller's dst (NULL: only wait for them): with src,
 * of device memory (complete on the stream), given to the staging in segments
 * of half of it, one crossing the bus while the host copies the other; without,
 * one segment whose give kernel is queued already under number seq0.  The
 * header comes with them.  From 1 MiB on with up to three more threads (one
 * thread copies 32 MiB to fresh pages in 1.0 ms, four in 0.2-0.5, while they
 * cross the bus in 0.58), which sleep until the first share has landed. */
static int collect(LMModel *m, const float *src, float *dst, size_t n, int seq0)
{
    const size_t half = m->give_floats / 2 & ~(size_t)3;
    Crew *c = &m->crew;
    c->m = m;
    c->dst = dst;
    c->n = c->seg = n;
    c->nseg = 1;
    c->seq0 = seq0;
    if (src) {
        c->seg = half < ((size_t)1 << 19) ? half : (size_t)1 << 19;
        c->nseg = (n + c->seg - 1) / c->seg;
        c->seq0 = (int)((unsigned)m->seq + 1u);
    }
    c->nt = 1 + (dst && n >= ((size_t)1 << 18) ? crew_hands(c) : 0);
    c->rc = LM_OK;
    c->issued = 0;
    for (int t = 0; t < c->nt; t++) c->prog[t] = 0;
    int rc = LM_OK, called = 0;
    for (size_t i = 0; i < c->nseg + 1 && rc == LM_OK; i++) {
        if (i < c->nseg) {   /* segment i into half i & 1, which segment i - 2 has left */
            for (int t = 1; t < c->nt && rc == LM_OK; t++) rc = crew_wait(c, &c->prog[t], (int)i - 1);
            const size_t len = crew_len(c, i);
            if (rc == LM_OK && src &&
                lmk_give(m->stream, src + i * c->seg, m->dh_logits + (i & 1) * c->seg, len, give_wgs(len), NULL,
                         m->d_ovf, NULL, 0, m->dh_hdr, NULL, next_seq(m),
                         m->dh_flag + (i & 1) * LM_GIVE_WGS * LM_FLAG_STRIDE) != hipSuccess)
                rc = LM_ERR_HIP;
            if (rc == LM_OK) __atomic_store_n(&c->issued, (int)i + 1, __ATOMIC_RELEASE);
        }
        if (i > 0 && rc == LM_OK) {
            if (c->nt > 1 && !called && (rc = wait_flag(m, 0, 0, c->seq0)) == LM_OK) {
                called = 1;
                for (int t = 1; t < c->nt; t++) sem_post(&c->hand[t - 1].go);
            }
            if (rc == LM_OK) {
                crew_take(c, 0, i - 1);
                rc = __atomic_load_n(&c->rc, __ATOMIC_RELAXED);
            }
        }
    }
    if (rc != LM_OK) __atomic_store_n(&c->rc, rc, __ATOMIC_RELAXED);
    for (int t = 1; called && t < c->nt; t++)
        while (__atomic_load_n(&c->prog[t], __ATOMIC_ACQUIRE) != INT_MAX) __builtin_ia32_pause();
    return __atomic_load_n(&c->rc, __ATOMIC_RELAXED);
}

/* The hand-off flag of the fused launches, as a call's results brought it. */
static int check_err(LMModel *m, int err)
{
    if (!err) return LM_OK;
    fprintf(stderr, "stories_lm: a hand-off wait inside a fused launch gave up (results invalid)\n");
    HIPCHK(hipStreamSynchronize(m->stream));
    /* Once a wait has given up, every wait of the launch ends early, so the
     * argmax reducer can advance the step count while classifier work-groups
     * dispatched before it have yet to read it; their words then carry the
     * tags of the next step.  Clear every hand-off word (tag 0 matches no
     * step) with the flag, on the model's stream, before the next call. */
    HIPCHK(hipMemsetAsync(m->d_tagged, 0, LM_TAG_WORDS(m->NQ, m->NKV, m->D, m->F) * 8, m->stream));
    HIPCHK(hipMemsetAsync(m->d_cls_tw, 0, (size_t)2 * LM_TAG_B * m->cls_nblk * 8, m->stream));
    HIPCHK(hipMemsetAsync(m->d_err, 0, 4, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    return LM_ERR_HIP;
}

static int check_tok_pos(const LMModel *m, const int *tokens, const int *pos, int B)
{
    for (int b = 0; b < B; b++) {
        if (tokens[b] < 0 || tokens[b] >= m->V) {
            fprintf(stderr, "stories_lm: token %d out of range [0,%d)\n", tokens[b], m->V);
            return LM_ERR_RANGE;
        }
        if (pos[b] < 0 || pos[b] >= m->max_seq) {
            fprintf(stderr, "stories_lm: position %d out of range [0,%d)\n", pos[b], m->max_seq);
            return LM_ERR_RANGE;
        }
    }
    return LM_OK;
}

/* One decode step of a call: its inputs into the call block, the step, its
 * logits (logits, B x V, may be NULL: staged in h_logits) and header. */
static int step_call(LMModel *m, const int *tokens, const int *pos, int B, int kind, float *logits)
{
    memcpy(m->h_call + LM_CALL_TOK, tokens, (size_t)B * 4);
    memcpy(m->h_call + LM_CALL_POS, pos, (size_t)B * 4);
    const int seq = next_seq(m);
    __atomic_store_n(m->h_call, seq, __ATOMIC_RELEASE);
    const size_t n = kind == STEP_LOGITS ? (size_t)B * m->V : 0;
    int rc = run_decode_steps(m, B, kind, ctx_class_rows(m, pos, B, 0));
    if (rc == LM_OK) rc = collect(m, NULL, logits, n, seq);
    if (rc != LM_OK) {
        (void)hipStreamSynchronize(m->stream);   /* the call block is free again */
        return rc;
    }
    return check_err(m, m->h_hdr[LM_HDR_ERR]);
}

int lm_forward_batch(LMModel *m, const int *tokens, const int *pos, int B, float *logits, int *argmax)
{
    if (!m || !tokens || !pos || B < 1) return LM_ERR_INVALID;
    if (B > m->max_batch) return LM_ERR_RANGE;
    int rc = check_tok_pos(m, tokens, pos, B);
    if (rc || (rc = check_batch(B))) return rc;
    if ((rc = step_call(m, tokens, pos, B, logits ? STEP_LOGITS : STEP_IDS, logits))) return rc;
    if (argmax) memcpy(argmax, m->h_hdr + LM_HDR_TOK, (size_t)B * 4);
    return LM_OK;
}

const float *lm_forward(LMModel *m, int token, int pos)
{
    if (!m) {
        fprintf(stderr, "stories_lm: lm_forward on NULL handle\n");
        return NULL;
    }
    if (check_tok_pos(m, &token, &pos, 1)) return NULL;
    return step_call(m, &token, &pos, 1, STEP_LOGITS, NULL) ? NULL : m->h_logits;
}

int lm_generate_greedy(LMModel *m, int B, const int *first_tokens, const int *pos0, int n_steps,
                       int *out_tokens)
{
    if (!m || !first_tokens || !pos0 || !out_tokens || B < 1 || n_steps < 0) return LM_ERR_INVALID;
    if (B > m->max_batch) return LM_ERR_RANGE;
    int rc = check_tok_pos(m, first_tokens, pos0, B);
    if (rc) return rc;
    for (int b = 0; b < B; b++)
        if (pos0[b] + n_steps > m->max_seq) {
            fprintf(stderr, "stories_lm: pos0 %d + %d steps exceeds max_seq %d\n", pos0[b], n_steps,
                    m->max_seq);
            return LM_ERR_RANGE;
        }
    if (n_steps == 0) return LM_OK;
    if ((rc = check_batch(B))) return rc;
    memcpy(m->h_call + LM_CALL_TOK, first_tokens, (size_t)B * 4);
    memcpy(m->h_call + LM_CALL_POS, pos0, (size_t)B * 4);
    __atomic_store_n(m->h_call, next_seq(m), __ATOMIC_RELEASE);
    KCHK(lmk_step_in(m->stream, m->dh_call, m->d_seq, m->d_tok, m->d_pos, B));
    int t = 0;
    for (; t + GRAPH_STEPS <= n_steps && rc == LM_OK; t += GRAPH_STEPS)
        rc = run_decode_steps(m, B, STEP_GREEDY_N, ctx_class_rows(m, pos0, B, t + GRAPH_STEPS - 1));
    for (; t < n_steps && rc == LM_OK; t++)
        rc = run_decode_steps(m, B, STEP_GREEDY, ctx_class_rows(m, pos0, B, t));
    /* the ids, as many steps at a time as the staging holds */
    const int seg = m->give_floats / B < (size_t)n_steps ? (int)(m->give_floats / B) : n_steps;
    for (int t0 = 0; t0 < n_steps && rc == LM_OK; t0 += seg) {
        const int nt = t0 + seg < n_steps ? seg : n_steps - t0, wgs = give_wgs((size_t)nt * B), seq = next_seq(m);
        if (lmk_give_ids(m->stream, m->d_hist, m->max_seq + 1, m->d_pos, B, n_steps, t0, nt,
                         (int *)m->dh_logits, wgs, m->d_err, m->dh_hdr, seq, m->dh_flag) != hipSuccess)
            rc = LM_ERR_HIP;
        else rc = collect(m, NULL, (float *)out_tokens + (size_t)t0 * B, (size_t)nt * B, seq);
    }
    if (rc != LM_OK) {
        (void)hipStreamSynchronize(m->stream);
        return rc;
    }
    return check_err(m, m->h_hdr[LM_HDR_ERR]);
}

/* Queue the layers of a prefill chunk of R rows (sequences of S rows; tokens,
 * positions and slots, R ints each, read from h_rin into d_rin) and the
 * classifier into d_logits, of every row with `all`, else of each sequence's
 * last row (positions and slots after the rows', R/S ints each). */
static int enqueue_prefill(LMModel *m, int R, int S, int all)
{
    const int *tok = m->d_rin, *pos = m->d_rin + R, *slot = m->d_rin + 2 * (size_t)R;
    const int *lpos = all ? NULL : m->d_rin + 3 * (size_t)R, *lslot = all ? NULL : lpos + R / S;
    KCHK(lmk_rows_in(m->stream, m->dh_rin, m->d_rin, 3 * R + (all ? 0 : 2 * (R / S))));
    return enqueue_rows(m, R, S, tok, pos, slot, m->d_logits, lpos, lslot);
}

/* Run a prefill chunk: launched directly, or replayed from a captured graph of
 * its shape, as lmh_shape_use says; captured behind a direct launch, while the
 * device is busy with it (a shape's second call 484 -> 344-499 us at 41 tokens
 * of Stories, 1532 -> 1299 at 8 x 256).  us a call, prompts of 30 to 52 tokens
 * through Stories, 3 / 6 / 12 lengths in rotation: 301 / 307 / 311 (replays
 * alone 301, direct launches 311); graphs replaced round robin 303 / 413 / 415. */
static int run_rows(LMModel *m, int R, int S, int all)
{
    int k = 0;
    /* (the graphs hold the folded form) */
    const int how = m->use_graph && !m->fold_off ? lmh_shape_use(&m->shapes, R, S, all, &k) : LM_SHAPE_DIRECT;
    if (how == LM_SHAPE_REPLAY) {
        HIPCHK(hipGraphLaunch(m->pgraph[k], m->stream));
        return LM_OK;
    }
    int rc = enqueue_prefill(m, R, S, all);
    if (how == LM_SHAPE_DIRECT) return rc;
    if (m->pgraph[k]) hipGraphExecDestroy(m->pgraph[k]);
    m->pgraph[k] = NULL;
    if (rc == LM_OK) rc = capture_begin(m);
    if (rc == LM_OK) rc = capture_end(m, enqueue_prefill(m, R, S, all), &m->pgraph[k]);
    if (rc != LM_OK) m->shapes.graph[k].used = 0;   /* (the entry is this shape's already) */
    return rc;
}

/* Causal forward of nseq sequences of S tokens (sequence i: slot slots[i],
 * positions pos0[i] .. pos0[i]+S-1, positions below pos0[i] already cached)
 * on the MFMA path, in chunks of whole sequences.  logits_mode LM_LOGITS_ALL:
 * every row's logits; LM_LOGITS_LAST: the last row of each sequence.  Host
 * `logits` (may be NULL) receives them in sequence order; the last chunk's
 * logits stay in d_logits. */
static int run_prefill(LMModel *m, int nseq, const int *slots, const int *pos0, const int *tokens,
                       int S, int logits_mode, float *logits, float *loss)
{
    const int V = m->V;
    unsigned char *seen = (unsigned char *)calloc((size_t)m->max_batch, 1);
    if (!seen) return LM_ERR_OOM;
    for (int i = 0; i < nseq; i++) {
        if (slots[i] < 0 || slots[i] >= m->max_batch || pos0[i] < 0 || pos0[i] + S > m->max_seq) {
            fprintf(stderr, "stories_lm: prefill sequence %d: slot %d / positions %d..%d out of "
                    "range (max_batch %d, max_seq %d)\n", i, slots[i], pos0[i], pos0[i] + S - 1,
                    m->max_batch, m->max_seq);
            free(seen);
            return LM_ERR_RANGE;
        }
        /* two sequences in one slot would write the same cache rows */
        if (seen[slots[i]]++) {
            fprintf(stderr, "stories_lm: prefill: slot %d given to more than one sequence\n",
                    slots[i]);
            free(seen);
            return LM_ERR_INVALID;
        }
        for (int t = 0; t < S; t++)
            if (tokens[(size_t)i * S + t] < 0 || tokens[(size_t)i * S + t] >= V) {
                fprintf(stderr, "stories_lm: prefill token %d out of range [0,%d)\n",
                        tokens[(size_t)i * S + t], V);
                free(seen);
                return LM_ERR_RANGE;
            }
    }
    free(seen);
    const int cs = S >= PREFILL_ROWS ? 1 : PREFILL_ROWS / S;   /* sequences per chunk */
    const int chunk_rows = (nseq < cs ? nseq : cs) * S;
    int rc;
    if (chunk_rows > m->max_rows && (rc = alloc_rows(m, chunk_rows))) return rc;
    int *h = m->h_rin;   /* pinned; each chunk ends with its results at the host */
    rc = LM_OK;
    for (int i0 = 0; i0 < nseq && rc == LM_OK; i0 += cs) {
        const int n = nseq - i0 < cs ? nseq - i0 : cs;
        const int R = n * S;
        for (int i = 0; i < n; i++)
            for (int t = 0; t < S; t++) {
                const int r = i * S + t;
                h[r] = tokens[(size_t)(i0 + i) * S + t];
                h[R + r] = pos0[i0 + i] + t;
                h[2 * R + r] = slots[i0 + i];
            }
        const int all = logits_mode == LM_LOGITS_ALL || S == 1;   /* (one row: the last) */
        if (!all)
            for (int i = 0; i < n; i++) {   /* (2n <= R: S >= 2) */
                h[3 * (size_t)R + i] = pos0[i0 + i] + S - 1;
                h[3 * (size_t)R + n + i] = slots[i0 + i];
            }
        /* pass 1 only when pass 0's folded norm overflowed fp16 (its u is
         * x * gain before the row is normalised): the same rows again with
         * the row norm apart, rewriting the same cache entries */
        for (int pass = 0; pass < 2 && rc == LM_OK; pass++) {
            rc = run_rows(m, R, S, all);
            /* the chunk's loss terms, straight to the staging, before the next
             * chunk reuses d_logits */
            if (rc == LM_OK && loss &&
                lmk_row_logprob(m->stream, m->d_logits, V, m->d_rin, S, R,
                                (float *)(m->dh_rin + 3 * (size_t)R)) != hipSuccess)
                rc = LM_ERR_HIP;
            const size_t rows = logits_mode == LM_LOGITS_ALL ? (size_t)R : (size_t)n;
            const size_t row0 = logits_mode == LM_LOGITS_ALL ? (size_t)i0 * S : (size_t)i0;
            volatile int *ovf = m->h_io + 4 * (size_t)m->max_batch + 1;
            if (rc == LM_OK && logits) {
                rc = collect(m, m->d_logits, logits + row0 * V, rows * V, 0);
                if (rc == LM_OK) *ovf = m->h_hdr[LM_HDR_OVF];
            }
            if (rc == LM_OK && (!logits || loss) && hipStreamSynchronize(m->stream) != hipSuccess)
                rc = LM_ERR_HIP;
            if (rc != LM_OK || !*ovf) break;
            *ovf = 0;
            m->fold_off = 1;
        }
        m->fold_off = 0;
        if (rc == LM_OK && loss) {
            /* mean over each sequence, summed in the reference's order
             * (forward.h:174-183: loss -= log_prob; loss / (S-1)) */
            const float *lp = (const float *)(h + 3 * (size_t)R);
            for (int i = 0; i < n; i++) {
                float acc = 0.f;
                for (int t = 0; t < S - 1; t++) acc -= lp[(size_t)i * S + t];
                loss[i0 + i] = acc / (S - 1);
            }
        }
    }
    /* after a failure, let the copy out of the staging buffer finish before
     * a later call refills it */
    if (rc != LM_OK) (void)hipStreamSynchronize(m->stream);
    return rc;
}

int lm_prefill(LMModel *m, int slot, int pos0, const int *tokens, int S, float *logits)
{
    if (!m || !tokens || S < 1) return LM_ERR_INVALID;
    if (slot < 0 || slot >= m->max_batch || pos0 < 0 || pos0 + S > m->max_seq) return LM_ERR_RANGE;
    return run_prefill(m, 1, &slot, &pos0, tokens, S, LM_LOGITS_ALL, logits, NULL);
}

static int prefill_from_zero(LMModel *m, int nseq, const int *slots, const int *tokens, int S,
                             int logits_mode, float *logits, float *loss)
{
    int *sl = (int *)malloc((size_t)nseq * 2 * sizeof(int));
    if (!sl) return LM_ERR_OOM;
    for (int i = 0; i < nseq; i++) {
        sl[i] = slots ? slots[i] : i;
        sl[nseq + i] = 0;
    }
    int rc = run_prefill(m, nseq, sl, sl + nseq, tokens, S, logits_mode, logits, loss);
    free(sl);
    return rc;
}

int lm_prefill_batch(LMModel *m, int nseq, const int *slots, const int *tokens, int S,
                     int logits_mode, float *logits)
{
    if (!m || !tokens || nseq < 1 || S < 1 ||
        (logits_mode != LM_LOGITS_ALL && logits_mode != LM_LOGITS_LAST))
        return LM_ERR_INVALID;
    return prefill_from_zero(m, nseq, slots, tokens, S, logits_mode, logits, NULL);
}

int lm_prefill_loss(LMModel *m, int nseq, const int *slots, const int *tokens, int S, float *logits,
                    float *loss)
{
    if (!m || !tokens || !loss || nseq < 1 || S < 2) return LM_ERR_INVALID;
    if (m->V % 4) {   /* the loss kernel reads each logit row as 16-byte groups */
        fprintf(stderr, "stories_lm: lm_prefill_loss: vocab_size %d is not a multiple of 4\n", m->V);
        return LM_ERR_UNSUPPORTED;
    }
    return prefill_from_zero(m, nseq, slots, tokens, S, LM_LOGITS_ALL, logits, loss);
}

int lm_read_logits(LMModel *m, int row0, int nrows, float *dst)
{
    if (!m || !dst || row0 < 0 || nrows < 0) return LM_ERR_INVALID;
    if (row0 + nrows > m->max_rows) return LM_ERR_RANGE;
    HIPCHK(hipStreamSynchronize(m->stream));
    HIPCHK(hipMemcpy(dst, m->d_logits + (size_t)row0 * m->V, (size_t)nrows * m->V * 4,
                     hipMemcpyDeviceToHost));
    return LM_OK;
}

/* ------------------------------------------------------------------------- */
/* timing                                                                     */
/* ------------------------------------------------------------------------- */

int lm_sync(LMModel *m)
{
    if (!m) return LM_ERR_INVALID;
    HIPCHK(hipStreamSynchronize(m->stream));
    return LM_OK;
}

int lm_timer_begin(LMModel *m)
{
    if (!m) return LM_ERR_INVALID;
    HIPCHK(hipEventRecord(m->ev0, m->stream));
    return LM_OK;
}

int lm_timer_end(LMModel *m, float *ms)
{
    if (!m || !ms) return LM_ERR_INVALID;
    HIPCHK(hipEventRecord(m->ev1, m->stream));
    HIPCHK(hipEventSynchronize(m->ev1));
    HIPCHK(hipEventElapsedTime(ms, m->ev0, m->ev1));
    return LM_OK;
}

/* Diagnostics: run the DPP reduction self-test (no model needed). */
int lm_selftest_reduce(const float *in64, float *out4)
{
    if (!in64 || !out4) return LM_ERR_INVALID;
    int rc = lm_init();
    if (rc) return rc;
    float *d = NULL;
    HIPCHK(hipMalloc((void **)&d, 68 * 4));
    hipError_t e = hipMemcpy(d, in64, 64 * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = (hipError_t)lmk_selftest_reduce(0, d, d + 64);
    if (e == hipSuccess) e = hipMemcpy(out4, d + 64, 16, hipMemcpyDeviceToHost);
    hipFree(d);
    HIPCHK(e);
    return LM_OK;
}

int lm_profile_chain(LMModel *m, int B, const int *tokens, const int *pos, int steps,
                     float *us_per_launch, int *launches_per_step)
{
    static const int fams[5] = {LM_KERN_QKV, LM_KERN_ATTN, LM_KERN_WO, LM_KERN_W13, LM_KERN_W2};
    if (!m || !tokens || !pos || !us_per_launch || B < 1 || steps < 1) return LM_ERR_INVALID;
    if (B > m->max_batch) return LM_ERR_RANGE;
    if (B > MAX_GEMV_B) return LM_ERR_UNSUPPORTED;
    int rc = check_tok_pos(m, tokens, pos, B);
    if (rc) return rc;
    for (int b = 0; b < B; b++)
        if (pos[b] + steps + 1 > m->max_seq) return LM_ERR_RANGE;
    const int lvl = chain_level(m, B), waits = step_waits(m, B);
    m->ctx_cls = ctx_class_rows(m, pos, B, steps);
    /* the launches of one step, in order: (family, layer) */
    const int nmax = 5 * m->L + 2;
    int *kf = (int *)calloc((size_t)nmax, sizeof(int)), *kl = (int *)calloc((size_t)nmax, sizeof(int));
    int nk = 0;
    if (!kf || !kl) rc = LM_ERR_OOM;
    for (int l = 0; l < m->L && rc == LM_OK; l++)
        for (int f = 0; f < 5; f++)
            if (!fam_inside(fams[f], lvl)) { kf[nk] = fams[f]; kl[nk++] = l; }   /* else inside QKV's */
    for (int f = LM_KERN_CLS; f <= LM_KERN_ARGMAX && rc == LM_OK; f++)
        if (!fam_inside(f, lvl)) { kf[nk] = f; kl[nk++] = 0; }   /* else inside the classifier's */
    /* Each run of consecutive launches of one family (at level 3 the L
     * whole-layer launches, then the classifier) is timed by one event pair,
     * the first launch's start to the last one's end, with no event between
     * them, so the launches meet each other as in the greedy loop's graphs;
     * the run's time is shared equally among its launches.  Steps are queued
     * back to back in runs of GRAPH_STEPS, as those graphs run them (the argmax
     * feeds each step's token to the next on the device); the stream is
     * synchronised and the events read once per run of steps. */
    int nrun = 0;
    for (int i = 0; i < nk; i++) nrun += i == 0 || kf[i] != kf[i - 1];
    const int chunk = GRAPH_STEPS;
    const size_t nev = 2 * (size_t)nrun * chunk;
    hipEvent_t *ev = (hipEvent_t *)calloc(nev, sizeof(hipEvent_t));
    double sum[LM_KERN_COUNT] = {0};
    int cnt[LM_KERN_COUNT] = {0};
    if (!ev) rc = LM_ERR_OOM;
    for (size_t i = 0; i < nev && rc == LM_OK; i++)
        if (hipEventCreate(&ev[i]) != hipSuccess) rc = LM_ERR_HIP;
    int *hio = m->h_io;
    if (rc == LM_OK) {
        memcpy(hio, tokens, B * 4);
        memcpy(hio + B, pos, B * 4);
        if (hipMemcpyAsync(m->d_tok, hio, B * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
            hipMemcpyAsync(m->d_pos, hio + B, B * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess)
            rc = LM_ERR_HIP;
    }
    for (int st0 = 0; st0 <= steps && rc == LM_OK; st0 += chunk) {   /* step 0 untimed */
        const int nst = steps + 1 - st0 < chunk ? steps + 1 - st0 : chunk;
        if (waits && (rc = handoff_enter(m))) break;
        for (int t = 0, r = 0; t < nst && rc == LM_OK; t++)
            for (int i = 0; i < nk && rc == LM_OK; i++) {
                const int first = i == 0 || kf[i] != kf[i - 1], last = i == nk - 1 || kf[i + 1] != kf[i];
                if (first || last)
                    lmk_time_next(first ? ev[2 * r] : NULL, last ? ev[2 * r + 1] : NULL);
                rc = enqueue_kernel(m, B, kf[i], kl[i], NULL);
                r += last;
            }
        if (waits) rc = handoff_leave(m, rc);
        if (rc == LM_OK && hipStreamSynchronize(m->stream) != hipSuccess) rc = LM_ERR_HIP;
        for (int t = 0, r = 0; t < nst && rc == LM_OK; t++)
            for (int i = 0, len = 0; i < nk && rc == LM_OK; i++) {
                len++;
                if (!(i == nk - 1 || kf[i + 1] != kf[i])) continue;
                float ms = 0.f;
                if (hipEventElapsedTime(&ms, ev[2 * r], ev[2 * r + 1]) != hipSuccess) rc = LM_ERR_HIP;
                if (st0 + t > 0) {
                    sum[kf[i]] += ms;
                    cnt[kf[i]] += len;
                }
                r++;
                len = 0;
            }
    }
    for (int f = 0; f < LM_KERN_COUNT; f++) {
        us_per_launch[f] = cnt[f] ? (float)(sum[f] * 1e3 / cnt[f]) : 0.f;
        if (launches_per_step)
            launches_per_step[f] = fam_inside(f, lvl)                            ? 0
                                   : f == LM_KERN_CLS || f == LM_KERN_ARGMAX ? 1
                                                                             : m->L;
    }
    for (size_t i = 0; ev && i < nev; i++)
        if (ev[i]) hipEventDestroy(ev[i]);
    free(ev);
    free(kf);
    free(kl);
    if (rc == LM_OK)
        HIPCHK(hipMemcpyAsync(m->d_pos, hio + B, B * 4, hipMemcpyHostToDevice, m->stream));
    int *err = hio + 4 * (size_t)m->max_batch;
    if (rc == LM_OK && hipMemcpyAsync(err, m->d_err, 4, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
        rc = LM_ERR_HIP;
    HIPCHK(hipStreamSynchronize(m->stream));
    if (rc == LM_OK) rc = check_err(m, *err);
    return rc;
}

/* Diagnostics: one MFMA GEMM C = A W^T on caller data (plain store epilogue
 * with argmax partials).  A is fp16 bits [M, K] (a_f32 == 0) or fp32 [M, K];
 * W fp16 bits [N, K]; C fp32 [M, N]; part (may be NULL) [M, ceil(N/32)]. */
int lm_selftest_gemm(int M, int N, int K, int a_f32, const void *A, const uint16_t *W, float *C,
                     LMArgPartHost *part)
{
    if (M < 1 || N < 1 || K < 64 || K % 64 || !A || !W || !C) return LM_ERR_INVALID;
    int rc = lm_init();
    if (rc) return rc;
    const size_t asz = (size_t)M * K * 2, wsz = (size_t)N * K * 2;
    const size_t csz = (size_t)M * N * 4, np = (size_t)M * ((N + 31) / 32);
    uint16_t *a16 = NULL;
    if (a_f32) {   /* the kernels take fp16 operands: round on the host (RNE) */
        a16 = (uint16_t *)malloc(asz);
        if (!a16) return LM_ERR_OOM;
        lm_f32_to_f16((const float *)A, a16, (size_t)M * K);
        A = a16;
    }
    void *dA = NULL, *dW = NULL, *dC = NULL, *dP = NULL;
    hipError_t e = hipMalloc(&dA, asz);
    if (e == hipSuccess) e = hipMalloc(&dW, wsz);
    if (e == hipSuccess) e = hipMalloc(&dC, csz);
    if (e == hipSuccess) e = hipMalloc(&dP, np * sizeof(LMArgPart));
    if (e == hipSuccess) e = hipMemcpy(dA, A, asz, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dW, W, wsz, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(dC, 0xFF, csz);
    if (e == hipSuccess) {
        LMEpilogue ep;
        memset(&ep, 0, sizeof(ep));
        ep.out = (float *)dC; ep.ldc = N; ep.part = (LMArgPart *)dP;
        e = (hipError_t)lmk_gemm(0, (const uint16_t *)dA, K, (const uint16_t *)dW, M, N, K,
                                 LMK_EPI_ARGMAX, &ep);
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(C, dC, csz, hipMemcpyDeviceToHost);
    if (e == hipSuccess && part) e = hipMemcpy(part, dP, np * sizeof(LMArgPart), hipMemcpyDeviceToHost);
    hipFree(dA); hipFree(dW); hipFree(dC); hipFree(dP);
    free(a16);
    HIPCHK(e);
    return LM_OK;
}

int lm_selftest_gemm_split(int M, int N, int K, int nsplit, const uint16_t *A, const uint16_t *W,
                           float *parts)
{
    if (M < 1 || M > 4096 || N < 1 || K < 64 || K % 64 || !A || !W || !parts) return LM_ERR_INVALID;
    if (nsplit == 0) nsplit = lmk_pick_split(M, N, K);
    if (nsplit < 1 || nsplit > LMK_MAX_SPLIT || K % (64 * nsplit)) return LM_ERR_INVALID;
    int rc = lm_init();
    if (rc) return rc;
    const size_t asz = (size_t)M * K * 2, wsz = (size_t)N * K * 2;
    const size_t psz = (size_t)nsplit * M * N * 4;
    void *dA = NULL, *dW = NULL, *dP = NULL;
    hipError_t e = hipMalloc(&dA, asz);
    if (e == hipSuccess) e = hipMalloc(&dW, wsz);
    if (e == hipSuccess) e = hipMalloc(&dP, psz);
    if (e == hipSuccess) e = hipMemcpy(dA, A, asz, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dW, W, wsz, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(dP, 0xFF, psz);
    if (e == hipSuccess)
        e = (hipError_t)lmk_gemm_split(0, (const uint16_t *)dA, K, (const uint16_t *)dW, M, N, K,
                                       nsplit, (float *)dP);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(parts, dP, psz, hipMemcpyDeviceToHost);
    hipFree(dA); hipFree(dW); hipFree(dP);
    HIPCHK(e);
    return nsplit;
}

int lm_selftest_gemm_gate(int M, int N, int K, const uint16_t *A, const uint16_t *W, uint16_t *g)
{
    if (M < 1 || N < 2 * LMK_GATE_BLOCK || N % (2 * LMK_GATE_BLOCK) || K < 64 || K % 64 || !A || !W || !g)
        return LM_ERR_INVALID;
    int rc = lm_init();
    if (rc) return rc;
    const int F = N / 2;
    const size_t asz = (size_t)M * K * 2, wsz = (size_t)N * K * 2, gsz = (size_t)M * F * 2;
    void *dA = NULL, *dW = NULL, *dG = NULL;
    hipError_t e = hipMalloc(&dA, asz);
    if (e == hipSuccess) e = hipMalloc(&dW, wsz);
    if (e == hipSuccess) e = hipMalloc(&dG, gsz);
    if (e == hipSuccess) e = hipMemcpy(dA, A, asz, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dW, W, wsz, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(dG, 0xFF, gsz);
    if (e == hipSuccess) {
        LMEpilogue ep;
        memset(&ep, 0, sizeof(ep));
        ep.g = (uint16_t *)dG; ep.F = F;
        e = (hipError_t)lmk_gemm(0, (const uint16_t *)dA, K, (const uint16_t *)dW, M, N, K, LMK_EPI_GATE, &ep);
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(g, dG, gsz, hipMemcpyDeviceToHost);
    hipFree(dA); hipFree(dW); hipFree(dG);
    HIPCHK(e);
    return LM_OK;
}

int lm_gemm_split_count(int M, int N, int K)
{
    if (M < 1 || N < 1 || K < 64 || K % 64) return LM_ERR_INVALID;
    return lmk_pick_split(M, N, K);
}
