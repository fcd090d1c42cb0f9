/*
 * engine.c -- C11 host engine over libg4hip.so (see engine.h).
 *
 * Structure follows thamada/Gemma4.c gemma4-4b/cpu-blas/main.c: the GGUF
 * reader and metadata defaults of parse_gguf (main.c:841-966), the tensor
 * names of load_weights (main.c:1328-1400), the layer routing helpers
 * (main.c:716-746), forward() (main.c:1838-2029) and the greedy branch of
 * generate() (main.c:2335-2488).  Arithmetic is done only by the HIP library.
 */
#define _POSIX_C_SOURCE 200809L
#include "engine.h"

#include <fcntl.h>
#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <time.h>
#include <unistd.h>

#include "../../include/g4hip.h"

#define E_N_LAYER_KV 24      /* main.c:77: layers 0..23 store KV; the tail reads 22/23 */
#define E_MAX_LAYERS 256

enum { GV_U8 = 0, GV_I8, GV_U16, GV_I16, GV_U32, GV_I32, GV_F32, GV_BOOL, GV_STR, GV_ARR, GV_U64, GV_I64, GV_F64 };

static char g_err[512];

const char *g4e_last_error(void) { return g_err; }

static int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

/* a failed g4_* call: keep the library's message */
static int lib_fail(int rc, const char *what) {
    snprintf(g_err, sizeof g_err, "%s: %s", what, g4_last_error());
    return rc;
}
#define CK(call)                                   \
    do {                                           \
        int rc_ = (call);                          \
        if (rc_) return lib_fail(rc_, #call);      \
    } while (0)

typedef struct {
    void *p;     /* device */
    int type, n, d;
    void *img;   /* device fp16 image for the batched prefill GEMM (Q4_K / Q5_K), or NULL */
} Tensor;

typedef struct {
    int dim, hidden, n_layers, n_heads, n_kv, vocab, max_seq, ple_dim, window;
    int swa_pattern, hd_swa, hd_full, rot_swa, rot_full, eos;
    float theta, theta_swa, eps, softcap;
    int swa[E_MAX_LAYERS];
    int has_swa_list;
} Config;

/* sampling settings of generate (main.c:2335-2341, 2408-2430) */
typedef struct {
    float temp, topp, penalty;
    int topk, last_n;
} SampleCfg;

struct g4e_model {
    Config c;
    /* weights (HBM) */
    Tensor embd, ple_tok, ple_proj;
    float *ple_proj_norm, *rope_freqs, *norm_out;
    float *attn_norm[E_MAX_LAYERS], *post_attn_norm[E_MAX_LAYERS], *ffn_norm[E_MAX_LAYERS];
    float *post_ffw_norm[E_MAX_LAYERS], *q_norm[E_MAX_LAYERS], *k_norm[E_MAX_LAYERS];
    float *post_norm[E_MAX_LAYERS], *out_scale[E_MAX_LAYERS];
    Tensor wq[E_MAX_LAYERS], wk[E_MAX_LAYERS], wv[E_MAX_LAYERS], wo[E_MAX_LAYERS];
    Tensor gate[E_MAX_LAYERS], up[E_MAX_LAYERS], down[E_MAX_LAYERS];
    Tensor inp_gate[E_MAX_LAYERS], proj[E_MAX_LAYERS];
    /* state (HBM) */
    float *x, *xb2, *hb, *q, *k, *v, *q_out, *ple, *ple_ctx, *ple_gate, *logits;
    float *hb2;              /* FFN up output when gate and up do not share the fused kernel */
    float *x_alt;            /* second residual-stream buffer (fused prologues write the other one) */
    float *ybuf;             /* PLE projection output, read by the next residual step */
    float *x_last;           /* buffer holding the residual stream after the last step */
    void *q8;
    float *kc[E_N_LAYER_KV], *vc[E_N_LAYER_KV];
    int kv_ring[E_N_LAYER_KV];
    float *attn_part;
    float *rope_tab;         /* (cos, sin) per pair: [rot_swa/2] then [rot_full/2] */
    int G_swa, G_full;
    void *ple_pairs;         /* g4_mm_ple_gate_proj's (value, step) pairs, one region per layer */
    size_t ple_pairs_stride;
    uint32_t *ple_seq;       /* the decode step's sequence word (advanced by the step's first launch) */
    int *dstep;              /* [0] token, [1] pos, [2] argmax / sampled token, [3] tokens in gen_hist,
                              * [4..5] the sampler's xorshift64* state */
    void *argmax_part;
    int *hstep;              /* pinned host mirror of dstep */
    void *stream;
    void *graph;             /* captured greedy decode step */
    void *sgraph;            /* captured sampled decode step ... */
    SampleCfg sgraph_cfg;    /* ... and the settings baked into it */
    int *gen_hist;           /* tokens generated by g4e_generate (repetition penalty history) */
    int gen_n;               /* host count of gen_hist entries written through g4e_gen_step */
    void *sample_part;
    /* prompt chunks (allocated on first use for pf_cap tokens; rows of the
     * chunk are contiguous) */
    int pf_cap, pf_Gmax;
    int pf_chunk;            /* tokens per prompt chunk; 0: generate prefills token by token */
    int *pf_tok;
    float *pf_x, *pf_xb2, *pf_q, *pf_k, *pf_v, *pf_ao, *pf_o, *pf_g, *pf_u, *pf_h, *pf_d, *pf_ig, *pf_pg, *pf_y;
    float *pf_ub;   /* per-block terms of the PLE gate GEMM: dim/256 slices of M x ple_dim */
    float *pf_ple, *pf_ctx, *pf_tab_swa, *pf_tab_full, *pf_part;
    void *pf_q8, *pf_q8a, *pf_q8p;
    void *pf_xs;                 /* split fp16 activations of the Q6_K GEMMs */
    int pf_xs_n;                 /* the widest row it holds */
    float *pf_kch[3], *pf_vch[3];   /* chunk K/V: [0] scratch, [1] donor 22, [2] donor 23 */
    /* host */
    int trace;
    float *layer_x;          /* host copy of dtr_x after a traced step */
    uint8_t *layer_q8;       /* host copy of dtr_q8 as BlockQ8_K structs */
    float *dtr_x;            /* device: (n_layers + 1) x dim layer inputs of the last traced step */
    void *dtr_q8;            /* device: n_layers x G4E_Q8_SLOTS Q8_K vectors of G4E_Q8_SLOT_ELEMS */
    void *allocs[4096];
    int n_allocs;
    int poison;              /* fill byte of new device buffers (G4E_POISON), -1: none */
    int f32_matmul;          /* Q4_K/Q5_K through mm_quant_rows (the reference's --f32-matmul) */
    int no_img;              /* prefill GEMMs on the quantized tensors instead of fp16 images */
    int dump_at, dump_now;   /* --dump-hidden-at position, -1: off; this step records */
    float *dstats;           /* device: (2 n_layers + 1) x (sum, l2, max) of the last dump */
    float *dfp;              /* device: layer-0 fingerprints of the last dump, G4E_FP_TAGS x 7 */
    float *dfp_k;            /* device: scratch K row for the pre-RoPE fingerprint */
    int fp_have[G4E_FP_TAGS];
};

/* ---- routing, main.c:716-746 ------------------------------------------------ */
static int is_swa(const Config *c, int l) {
    if (c->has_swa_list) return c->swa[l];
    if (c->swa_pattern <= 0) return 0;
    return (l % c->swa_pattern) < (c->swa_pattern - 1);
}
static int layer_hd(const Config *c, int l) { return is_swa(c, l) ? c->hd_swa : c->hd_full; }
static int layer_has_kv(int l) { return l < E_N_LAYER_KV; }
static int kv_source(const Config *c, int l) { return layer_has_kv(l) ? l : (is_swa(c, l) ? 22 : 23); }
static int is_kq45(int t) { return t == G4_Q4_K || t == G4_Q5_K; }

/* ---- GGUF reader (main.c:782-966) ------------------------------------------ */
typedef struct { const uint8_t *d; uint64_t p, n; int bad; } Rd;

static int need(Rd *r, uint64_t k) {
    if (r->bad || r->p + k > r->n) { r->bad = 1; return 0; }
    return 1;
}
static uint32_t ru32(Rd *r) { uint32_t v = 0; if (need(r, 4)) memcpy(&v, r->d + r->p, 4); r->p += 4; return v; }
static uint64_t ru64(Rd *r) { uint64_t v = 0; if (need(r, 8)) memcpy(&v, r->d + r->p, 8); r->p += 8; return v; }
static float rf32(Rd *r) { float v = 0; if (need(r, 4)) memcpy(&v, r->d + r->p, 4); r->p += 4; return v; }
static const char *rstr(Rd *r, uint64_t *len) {
    uint64_t n = ru64(r);
    const char *s = (const char *)r->d + r->p;
    if (!need(r, n)) n = 0;
    r->p += n;
    *len = n;
    return s;
}
static void skip(Rd *r, uint32_t t, int depth) {
    if (r->bad || depth > 4) { r->bad = 1; return; }
    switch (t) {
    case GV_U8: case GV_I8: case GV_BOOL: r->p += 1; break;
    case GV_U16: case GV_I16: r->p += 2; break;
    case GV_U32: case GV_I32: case GV_F32: r->p += 4; break;
    case GV_U64: case GV_I64: case GV_F64: r->p += 8; break;
    case GV_STR: { uint64_t n = ru64(r); r->p += n; break; }
    case GV_ARR: {
        uint32_t at = ru32(r);
        uint64_t al = ru64(r);
        if (at == GV_STR || at == GV_ARR) {
            for (uint64_t i = 0; i < al && !r->bad; i++) skip(r, at, depth + 1);
        } else {
            static const int sz[13] = {1, 1, 2, 2, 4, 4, 4, 1, 0, 0, 8, 8, 8};
            if (at > GV_F64) { r->bad = 1; break; }
            r->p += al * (uint64_t)sz[at];
        }
        break;
    }
    default: r->bad = 1;
    }
    if (r->p > r->n) r->bad = 1;
}
static int64_t rint_val(Rd *r, uint32_t t) {
    int64_t v = 0;
    switch (t) {
    case GV_U8: case GV_BOOL: if (need(r, 1)) v = r->d[r->p]; r->p += 1; break;
    case GV_I8: if (need(r, 1)) v = (int8_t)r->d[r->p]; r->p += 1; break;
    case GV_U16: { uint16_t x = 0; if (need(r, 2)) memcpy(&x, r->d + r->p, 2); r->p += 2; v = x; break; }
    case GV_I16: { int16_t x = 0; if (need(r, 2)) memcpy(&x, r->d + r->p, 2); r->p += 2; v = x; break; }
    case GV_U32: v = ru32(r); break;
    case GV_I32: v = (int32_t)ru32(r); break;
    case GV_U64: v = (int64_t)ru64(r); break;
    case GV_I64: v = (int64_t)ru64(r); break;
    case GV_F32: v = (int64_t)rf32(r); break;
    case GV_F64: { double x = 0; if (need(r, 8)) memcpy(&x, r->d + r->p, 8); r->p += 8; v = (int64_t)x; break; }
    default: skip(r, t, 0);
    }
    return v;
}
static float rfloat_val(Rd *r, uint32_t t) {
    switch (t) {
    case GV_F32: return rf32(r);
    case GV_F64: { double x = 0; if (need(r, 8)) memcpy(&x, r->d + r->p, 8); r->p += 8; return (float)x; }
    case GV_U32: return (float)ru32(r);
    case GV_I32: return (float)(int32_t)ru32(r);
    case GV_U64: return (float)ru64(r);
    case GV_I64: return (float)(int64_t)ru64(r);
    default: skip(r, t, 0); return 0.0f;
    }
}
static int key_is(const char *k, uint64_t kl, const char *lit) { return kl == strlen(lit) && !memcmp(k, lit, kl); }

typedef struct {
    const char *name;
    uint64_t nlen, off;
    uint64_t ne[4];
    int n_dims, type;
} TInfo;

/* ---- device allocation bookkeeping ----------------------------------------- */
static int dalloc(g4e_model *m, void **p, size_t bytes) {
    if (m->n_allocs >= (int)(sizeof m->allocs / sizeof m->allocs[0])) return fail(G4_ERR_NOMEM, "too many allocations");
    CK(g4_malloc(p, bytes ? bytes : 1));
    m->allocs[m->n_allocs++] = *p;
    if (m->poison >= 0) CK(g4_memset(*p, m->poison, bytes ? bytes : 1));
    return 0;
}

/* dalloc for memory the engine can do without: 0 and a pointer, or nonzero
 * and NULL with no error recorded */
static int dalloc_opt(g4e_model *m, void **p, size_t bytes) {
    *p = NULL;
    if (m->n_allocs >= (int)(sizeof m->allocs / sizeof m->allocs[0]) || g4_malloc(p, bytes ? bytes : 1)) {
        *p = NULL;
        return 1;
    }
    m->allocs[m->n_allocs++] = *p;
    return 0;
}

static size_t tensor_bytes(int type, uint64_t n, uint64_t d) {
    return g4_tensor_bytes(type, (int)n, (int)d);
}

static const TInfo *find_t(const TInfo *ti, int nt, const char *name) {
    const size_t L = strlen(name);
    for (int i = 0; i < nt; i++)
        if (ti[i].nlen == L && !memcmp(ti[i].name, name, L)) return &ti[i];
    return NULL;
}

/* upload one tensor; matrices [ne1 rows x ne0] of K-quant types go through the
 * planar layout, everything else is copied verbatim. */
static int upload(g4e_model *m, const uint8_t *base, const TInfo *t, Tensor *out) {
    const uint64_t n = t->ne[0], d = t->n_dims > 1 ? t->ne[1] : 1;
    if (t->n_dims > 2 || n == 0 || d == 0 || n > 0x7fffffff || d > 0x7fffffff)
        return fail(G4_ERR_FORMAT, "tensor %.*s: unsupported shape", (int)t->nlen, t->name);
    const size_t bytes = tensor_bytes(t->type, n, d);
    if (!bytes) return fail(G4_ERR_TYPE, "tensor %.*s: unsupported type %d or shape", (int)t->nlen, t->name, t->type);
    int rc = dalloc(m, &out->p, bytes);
    if (rc) return rc;
    out->type = t->type;
    out->n = (int)n;
    out->d = (int)d;
    const uint8_t *src = base + t->off;
    if (t->type == G4_Q4_K || t->type == G4_Q5_K || t->type == G4_Q6_K) CK(g4_upload_quant(out->p, src, t->type, (int)n, (int)d));
    else CK(g4_memcpy_h2d(out->p, src, bytes));
    return 0;
}

/* parse_gguf (main.c:841-966): metadata with the reference's defaults, the
 * tensor table, and the data offset.  Host only. */
typedef struct {
    TInfo *ti;
    uint64_t nt;
    const uint8_t *base;
} Image;

static int parse(const uint8_t *data, size_t size, int max_seq, Config *c, Image *img) {
    Rd r = {data, 0, size, 0};
    memset(c, 0, sizeof *c);
    img->ti = NULL;
    if (size < 24 || ru32(&r) != 0x46554747u) return fail(G4_ERR_FORMAT, "Error: invalid GGUF magic");
    (void)ru32(&r);
    const uint64_t n_tensors = ru64(&r), n_kv = ru64(&r);
    /* defaults, main.c:854-871 */
    c->theta = 1e6f; c->theta_swa = 10000.0f; c->eps = 1e-6f; c->max_seq = 8192; c->swa_pattern = 6;
    c->hd_swa = 256; c->hd_full = 512; c->rot_swa = 256; c->rot_full = 512; c->ple_dim = 256;
    c->window = 512; c->softcap = 30.0f; c->eos = 106;
    uint32_t alignment = 32;
    for (uint64_t i = 0; i < n_kv && !r.bad; i++) {
        uint64_t kl;
        const char *k = rstr(&r, &kl);
        const uint32_t vt = ru32(&r);
#define KI(lit, field) else if (key_is(k, kl, lit)) field = (int)rint_val(&r, vt)
#define KF(lit, field) else if (key_is(k, kl, lit)) field = rfloat_val(&r, vt)
        if (key_is(k, kl, "general.alignment")) alignment = (uint32_t)rint_val(&r, vt);
        KI("gemma4.embedding_length", c->dim);
        KI("gemma4.feed_forward_length", c->hidden);
        KI("gemma4.block_count", c->n_layers);
        KI("gemma4.attention.head_count", c->n_heads);
        KI("gemma4.attention.head_count_kv", c->n_kv);
        KI("gemma4.attention.key_length_swa", c->hd_swa);
        KI("gemma4.attention.key_length", c->hd_full);
        KI("gemma4.rope.dimension_count_swa", c->rot_swa);
        KI("gemma4.rope.dimension_count", c->rot_full);
        KF("gemma4.attention.layer_norm_rms_epsilon", c->eps);
        KF("gemma4.rope.freq_base", c->theta);
        KF("gemma4.rope.freq_base_swa", c->theta_swa);
        KI("gemma4.attention.sliding_window", c->window);
        KI("gemma4.embedding_length_per_layer_input", c->ple_dim);
        KF("gemma4.final_logit_softcapping", c->softcap);
        KI("gemma4.context_length", c->max_seq);
        KI("tokenizer.ggml.eos_token_id", c->eos);
        else if (key_is(k, kl, "gemma4.attention.sliding_window_pattern") && vt == GV_ARR) {
            const uint32_t et = ru32(&r);
            const uint64_t n = ru64(&r);
            if (n > 0 && n <= E_MAX_LAYERS && et != GV_STR && et != GV_ARR) {
                for (uint64_t j = 0; j < n; j++) c->swa[j] = rint_val(&r, et) ? 1 : 0;
                c->has_swa_list = 1;
            } else {
                for (uint64_t j = 0; j < n && !r.bad; j++) skip(&r, et, 1);
            }
        } else if (key_is(k, kl, "tokenizer.ggml.tokens") && vt == GV_ARR) {
            /* vocab_size = the length of the token list (main.c:922-931) */
            (void)ru32(&r);
            const uint64_t n = ru64(&r);
            c->vocab = (int)n;
            for (uint64_t j = 0; j < n && !r.bad; j++) { uint64_t sl; (void)rstr(&r, &sl); }
        } else {
            skip(&r, vt, 0);
        }
#undef KI
#undef KF
    }
    if (r.bad) return fail(G4_ERR_FORMAT, "truncated GGUF metadata");
    if (n_tensors > 100000) return fail(G4_ERR_FORMAT, "implausible tensor count %llu", (unsigned long long)n_tensors);
    TInfo *ti = (TInfo *)calloc(n_tensors ? n_tensors : 1, sizeof(TInfo));
    if (!ti) return fail(G4_ERR_NOMEM, "out of host memory");
    for (uint64_t i = 0; i < n_tensors && !r.bad; i++) {
        ti[i].name = rstr(&r, &ti[i].nlen);
        ti[i].n_dims = (int)ru32(&r);
        if (ti[i].n_dims < 1 || ti[i].n_dims > 4) { r.bad = 1; break; }
        for (int dd = 0; dd < ti[i].n_dims; dd++) ti[i].ne[dd] = ru64(&r);
        ti[i].type = (int)ru32(&r);
        ti[i].off = ru64(&r);
    }
    if (r.bad || alignment == 0) { free(ti); return fail(G4_ERR_FORMAT, "truncated GGUF tensor table"); }
    const uint64_t doff = (r.p + (alignment - 1)) & ~(uint64_t)(alignment - 1);
    for (uint64_t i = 0; i < n_tensors; i++) {
        const uint64_t n = ti[i].ne[0], d = ti[i].n_dims > 1 ? ti[i].ne[1] : 1;
        size_t b = tensor_bytes(ti[i].type, n, d);
        if (b == 0) b = (size_t)n * d;    /* unknown types are rejected only if used */
        if (doff + ti[i].off + b > size) { free(ti); return fail(G4_ERR_FORMAT, "tensor data past the end of the file"); }
    }
    if (max_seq > 0) c->max_seq = max_seq;
    if (c->n_layers <= 0 || c->n_layers > E_MAX_LAYERS || c->dim <= 0 || c->hidden <= 0 || c->n_heads <= 0 ||
        c->n_kv <= 0 || c->vocab <= 0 || c->max_seq <= 0 || c->n_heads % c->n_kv || c->ple_dim <= 0) {
        free(ti);
        return fail(G4_ERR_FORMAT, "bad model config (layers %d dim %d heads %d kv %d vocab %d)", c->n_layers, c->dim,
                    c->n_heads, c->n_kv, c->vocab);
    }
    img->ti = ti;
    img->nt = n_tensors;
    img->base = data + doff;
    return 0;
}

/* shape/type checks of everything load_weights binds (main.c:1328-1400);
 * the reference trusts the file, the device kernels do not. */
static int check_t(const Image *im, const char *name, const int *types, int ntypes, uint64_t n, uint64_t d,
                   int optional) {
    const TInfo *t = find_t(im->ti, (int)im->nt, name);
    if (!t) return optional ? 0 : fail(G4_ERR_FORMAT, "Error: missing tensor %s", name);
    int ok = 0;
    for (int i = 0; i < ntypes; i++) ok |= t->type == types[i];
    if (!ok) return fail(G4_ERR_TYPE, "Unsupported tensor type %d for %s", t->type, name);
    const uint64_t tn = t->ne[0], td = t->n_dims > 1 ? t->ne[1] : 1;
    if (t->n_dims > 2 || tn != n || td != d)
        return fail(G4_ERR_FORMAT, "%s: shape [%llu x %llu], expected [%llu x %llu]", name, (unsigned long long)tn,
                    (unsigned long long)td, (unsigned long long)n, (unsigned long long)d);
    if ((t->type == G4_Q4_K || t->type == G4_Q5_K || t->type == G4_Q6_K) && n % 256)
        return fail(G4_ERR_FORMAT, "%s: row length %llu not a multiple of 256", name, (unsigned long long)n);
    /* the dense GEMVs stream 16-byte chunks of a row held in LDS */
    if (d > 1 && (t->type == G4_F16 || t->type == G4_BF16 || t->type == G4_F32) &&
        (n % (t->type == G4_F32 ? 4 : 8) || n > 16384))
        return fail(G4_ERR_FORMAT, "%s: dense row length %llu unsupported", name, (unsigned long long)n);
    return 0;
}

static int validate(const Config *c, const Image *im) {
    /* every matrix goes through mm() (main.c:1669-1694), every table through
     * emb_lookup (main.c:1696-1723; the token table also through mm() for the
     * tied LM head), with the types as found in the file */
    static const int F32T[] = {G4_F32};
    static const int MAT[] = {G4_Q4_K, G4_Q5_K, G4_Q6_K, G4_BF16, G4_F16, G4_F32};
    static const int EMB[] = {G4_Q4_K, G4_Q5_K, G4_Q6_K, G4_F16, G4_F32};
    const int L = c->n_layers;
    char name[128];
    int rc;
    if (c->hd_swa != 256 && c->hd_swa != 512) return fail(G4_ERR_FORMAT, "head_dim_swa %d unsupported", c->hd_swa);
    if (c->hd_full != 256 && c->hd_full != 512) return fail(G4_ERR_FORMAT, "head_dim %d unsupported", c->hd_full);
    if (c->n_heads / c->n_kv > 8) return fail(G4_ERR_FORMAT, "n_heads/n_kv > 8 unsupported");
    if (c->dim % 256 || c->ple_dim % 256) return fail(G4_ERR_FORMAT, "dim/ple_dim must be multiples of 256");
    if (c->n_layers > E_N_LAYER_KV && c->n_layers < 24) return fail(G4_ERR_FORMAT, "layer count");
    if (c->n_layers > E_N_LAYER_KV && (is_swa(c, 22) != 1 || is_swa(c, 23) != 0))
        return fail(G4_ERR_FORMAT, "shared-KV donors 22/23 must be sliding/full layers (main.c:743-746)");
    if ((rc = check_t(im, "token_embd.weight", EMB, 5, c->dim, c->vocab, 0)) ||
        (rc = check_t(im, "per_layer_token_embd.weight", EMB, 5, (uint64_t)c->ple_dim * L, c->vocab, 0)) ||
        (rc = check_t(im, "per_layer_model_proj.weight", MAT, 6, c->dim, (uint64_t)c->ple_dim * L, 0)) ||
        (rc = check_t(im, "per_layer_proj_norm.weight", F32T, 1, c->ple_dim, 1, 0)) ||
        (rc = check_t(im, "output_norm.weight", F32T, 1, c->dim, 1, 0)) ||
        (rc = check_t(im, "rope_freqs.weight", F32T, 1, c->rot_full / 2, 1, 1)))
        return rc;
    for (int l = 0; l < L; l++) {
        const uint64_t hd = layer_hd(c, l), qd = c->n_heads * hd, kvd = c->n_kv * hd;
#define CT(suffix, types, nt_, n_, d_, opt)                                        \
        snprintf(name, sizeof name, "blk.%d." suffix, l);                          \
        if ((rc = check_t(im, name, types, nt_, n_, d_, opt))) return rc;
        CT("attn_norm.weight", F32T, 1, c->dim, 1, 0);
        CT("post_attention_norm.weight", F32T, 1, c->dim, 1, 0);
        CT("attn_q_norm.weight", F32T, 1, hd, 1, 0);
        CT("attn_k_norm.weight", F32T, 1, hd, 1, 0);
        CT("attn_q.weight", MAT, 6, c->dim, qd, 0);
        if (layer_has_kv(l)) {
            CT("attn_k.weight", MAT, 6, c->dim, kvd, 0);
            CT("attn_v.weight", MAT, 6, c->dim, kvd, 0);
        }
        CT("attn_output.weight", MAT, 6, qd, c->dim, 0);
        CT("ffn_norm.weight", F32T, 1, c->dim, 1, 0);
        CT("post_ffw_norm.weight", F32T, 1, c->dim, 1, 0);
        CT("ffn_gate.weight", MAT, 6, c->dim, c->hidden, 0);
        CT("ffn_up.weight", MAT, 6, c->dim, c->hidden, 0);
        CT("ffn_down.weight", MAT, 6, c->hidden, c->dim, 0);
        CT("inp_gate.weight", MAT, 6, c->dim, c->ple_dim, 0);
        CT("proj.weight", MAT, 6, c->ple_dim, c->dim, 0);
        CT("post_norm.weight", F32T, 1, c->dim, 1, 0);
        CT("layer_output_scale.weight", F32T, 1, 1, 1, 1);
#undef CT
    }
    return 0;
}

/* ---- model file verification --------------------------------------------
 * SHA-256 (FIPS 180-4) of a file and the `sha256sum --check` of the model
 * download (gemma4-4b/Makefile `model` target, design.md:107-117).  The round
 * constants are the first 32 fractional bits of the cube roots of the first
 * 64 primes, the initial hash those of the square roots of the first 8,
 * computed here from their definition. */
static void sha256_consts(uint32_t K[64], uint32_t H0[8]) {
    int n = 0;
    for (int p = 2; n < 64; p++) {
        int prime = 1;
        for (int q = 2; q * q <= p; q++)
            if (p % q == 0) { prime = 0; break; }
        if (!prime) continue;
        const double c = cbrt((double)p), r = sqrt((double)p);
        K[n] = (uint32_t)((c - floor(c)) * 4294967296.0);
        if (n < 8) H0[n] = (uint32_t)((r - floor(r)) * 4294967296.0);
        n++;
    }
}

#define ROR32(x, k) (((x) >> (k)) | ((x) << (32 - (k))))

static void sha256_block(uint32_t h[8], const uint32_t K[64], const uint8_t *b) {
    uint32_t w[64];
    for (int i = 0; i < 16; i++)
        w[i] = (uint32_t)b[4 * i] << 24 | (uint32_t)b[4 * i + 1] << 16 | (uint32_t)b[4 * i + 2] << 8 | b[4 * i + 3];
    for (int i = 16; i < 64; i++) {
        const uint32_t s0 = ROR32(w[i - 15], 7) ^ ROR32(w[i - 15], 18) ^ (w[i - 15] >> 3);
        const uint32_t s1 = ROR32(w[i - 2], 17) ^ ROR32(w[i - 2], 19) ^ (w[i - 2] >> 10);
        w[i] = w[i - 16] + s0 + w[i - 7] + s1;
    }
    uint32_t a = h[0], bb = h[1], c = h[2], d = h[3], e = h[4], f = h[5], g = h[6], hh = h[7];
    for (int i = 0; i < 64; i++) {
        const uint32_t t1 = hh + (ROR32(e, 6) ^ ROR32(e, 11) ^ ROR32(e, 25)) + ((e & f) ^ (~e & g)) + K[i] + w[i];
        const uint32_t t2 = (ROR32(a, 2) ^ ROR32(a, 13) ^ ROR32(a, 22)) + ((a & bb) ^ (a & c) ^ (bb & c));
        hh = g; g = f; f = e; e = d + t1; d = c; c = bb; bb = a; a = t1 + t2;
    }
    h[0] += a; h[1] += bb; h[2] += c; h[3] += d; h[4] += e; h[5] += f; h[6] += g; h[7] += hh;
}

int g4e_sha256_file(const char *path, char hex[65]) {
    if (!path || !hex) return fail(G4_ERR_ARG, "g4e_sha256_file: null pointer");
    FILE *fp = fopen(path, "rb");
    if (!fp) return fail(G4_ERR_ARG, "Error: cannot open %s", path);
    uint32_t K[64], h[8];
    sha256_consts(K, h);
    enum { CHUNK = 1 << 20 };
    uint8_t *buf = (uint8_t *)malloc(CHUNK + 128);
    if (!buf) { fclose(fp); return fail(G4_ERR_NOMEM, "out of host memory"); }
    uint64_t total = 0;
    size_t got;
    int err = 0;
    while ((got = fread(buf, 1, CHUNK, fp)) == CHUNK) {
        for (size_t o = 0; o < CHUNK; o += 64) sha256_block(h, K, buf + o);
        total += CHUNK;
    }
    if (ferror(fp)) err = 1;
    fclose(fp);
    if (err) { free(buf); return fail(G4_ERR_FORMAT, "Error: reading %s failed", path); }
    /* the tail, 0x80, zeros, the bit length (big-endian): one or two blocks */
    total += got;
    const size_t full = got / 64 * 64;
    for (size_t o = 0; o < full; o += 64) sha256_block(h, K, buf + o);
    const size_t rest = got - full;
    uint8_t tail[128] = {0};
    memcpy(tail, buf + full, rest);
    tail[rest] = 0x80;
    const size_t tl = rest < 56 ? 64 : 128;
    const uint64_t bits = total * 8;
    for (int i = 0; i < 8; i++) tail[tl - 1 - i] = (uint8_t)(bits >> (8 * i));
    for (size_t o = 0; o < tl; o += 64) sha256_block(h, K, tail + o);
    free(buf);
    for (int i = 0; i < 8; i++) snprintf(hex + 8 * i, 9, "%08x", h[i]);
    return 0;
}

int g4e_check_sha256sum(const char *path, const char *sumfile) {
    if (!path || !sumfile) return fail(G4_ERR_ARG, "g4e_check_sha256sum: null pointer");
    const char *base = strrchr(path, '/');
    base = base ? base + 1 : path;
    FILE *fp = fopen(sumfile, "r");
    if (!fp) return fail(G4_ERR_ARG, "Error: cannot open %s", sumfile);
    char line[1024], want[65] = {0};
    int found = 0;
    while (fgets(line, sizeof line, fp)) {
        /* "<64 hex>  <name>" or "<64 hex> *<name>" (sha256sum's text / binary marks) */
        size_t len = strcspn(line, "\r\n");
        line[len] = 0;
        if (len < 66 || line[64] != ' ') continue;
        const char *name = line + 65;
        if (*name == ' ' || *name == '*') name++;
        if (strcmp(name, base)) continue;
        memcpy(want, line, 64);
        for (int i = 0; i < 64; i++) want[i] = (char)((want[i] >= 'A' && want[i] <= 'F') ? want[i] - 'A' + 'a' : want[i]);
        found = 1;
        break;
    }
    fclose(fp);
    if (!found) return fail(G4_ERR_FORMAT, "%s: no checksum line for %s", sumfile, base);
    char got[65];
    int rc = g4e_sha256_file(path, got);
    if (rc) return rc;
    if (memcmp(got, want, 64)) return fail(G4_ERR_FORMAT, "%s: FAILED (sha256 %s, expected %s)", base, got, want);
    return 0;
}

int g4e_check_image(const void *data, size_t size, int max_seq, int out[9]) {
    Config c;
    Image im;
    if (!data) return fail(G4_ERR_ARG, "g4e_check_image: null pointer");
    int rc = parse((const uint8_t *)data, size, max_seq, &c, &im);
    if (rc) return rc;
    rc = validate(&c, &im);
    free(im.ti);
    if (rc == 0 && out) {
        const int v[9] = {c.dim, c.hidden, c.n_layers, c.n_heads, c.n_kv, c.vocab, c.max_seq, c.ple_dim, c.window};
        memcpy(out, v, sizeof v);
    }
    return rc;
}

/* time chunks of the decode attention for a window capacity: about 32
 * positions per workgroup at full capacity, 1..128 chunks (more only if a
 * chunk would exceed 1024 positions) */
static int attn_chunks(int cap) {
    int G = (cap + 31) / 32;
    if (G < 1) G = 1;
    if (G > 128) G = 128;
    while ((cap + G - 1) / G > 1024) G++;
    return G;
}

/* load_weights (upload to HBM) + alloc_state (main.c:1328-1423) */
static int load(g4e_model *m, const Image *im) {
    const Config *c = &m->c;
    const int L = c->n_layers;
    char name[128];
    int rc;
#define UP(nm, dst)                                                                       \
    do {                                                                                  \
        const TInfo *t_ = find_t(im->ti, (int)im->nt, nm);                                \
        if (t_ && (rc = upload(m, im->base, t_, &(dst)))) return rc;                      \
    } while (0)
#define UPF(nm, dst)                                                                      \
    do {                                                                                  \
        Tensor tt_ = {0};                                                                 \
        UP(nm, tt_);                                                                      \
        dst = (float *)tt_.p;                                                             \
    } while (0)
    UP("token_embd.weight", m->embd);
    UP("per_layer_token_embd.weight", m->ple_tok);
    UP("per_layer_model_proj.weight", m->ple_proj);
    UPF("per_layer_proj_norm.weight", m->ple_proj_norm);
    UPF("output_norm.weight", m->norm_out);
    UPF("rope_freqs.weight", m->rope_freqs);
    for (int l = 0; l < L; l++) {
#define LT(suffix, dst) snprintf(name, sizeof name, "blk.%d." suffix, l); UP(name, dst);
#define LF(suffix, dst) snprintf(name, sizeof name, "blk.%d." suffix, l); UPF(name, dst);
        LF("attn_norm.weight", m->attn_norm[l]);
        LF("post_attention_norm.weight", m->post_attn_norm[l]);
        LF("attn_q_norm.weight", m->q_norm[l]);
        LF("attn_k_norm.weight", m->k_norm[l]);
        LT("attn_q.weight", m->wq[l]);
        if (layer_has_kv(l)) {
            LT("attn_k.weight", m->wk[l]);
            LT("attn_v.weight", m->wv[l]);
        }
        LT("attn_output.weight", m->wo[l]);
        LF("ffn_norm.weight", m->ffn_norm[l]);
        LF("post_ffw_norm.weight", m->post_ffw_norm[l]);
        LT("ffn_gate.weight", m->gate[l]);
        LT("ffn_up.weight", m->up[l]);
        LT("ffn_down.weight", m->down[l]);
        LT("inp_gate.weight", m->inp_gate[l]);
        LT("proj.weight", m->proj[l]);
        LF("post_norm.weight", m->post_norm[l]);
        LF("layer_output_scale.weight", m->out_scale[l]);
#undef LT
#undef LF
    }
#undef UP
#undef UPF

    /* alloc_state, in HBM */
    const int hdmax = c->hd_full > c->hd_swa ? c->hd_full : c->hd_swa;
    const int qmax = c->n_heads * hdmax, kvmax = c->n_kv * hdmax;
    int q8n = c->hidden > qmax ? c->hidden : qmax;
    if (c->dim > q8n) q8n = c->dim;
    q8n = (q8n + 255) / 256 * 256;
    void *p;
#define DA(field, bytes) if ((rc = dalloc(m, &p, (size_t)(bytes)))) return rc; field = p;
    DA(m->x, (size_t)c->dim * 4);
    DA(m->x_alt, (size_t)c->dim * 4);
    DA(m->ybuf, (size_t)c->dim * 4);
    m->x_last = m->x;
    DA(m->xb2, (size_t)c->dim * 4);
    DA(m->hb, (size_t)c->hidden * 4);
    DA(m->hb2, (size_t)c->hidden * 4);
    DA(m->dstats, (size_t)(2 * L + 1) * 3 * 4);
    DA(m->dfp, (size_t)G4E_FP_TAGS * 7 * 4);
    DA(m->dfp_k, (size_t)c->n_kv * (c->hd_full > c->hd_swa ? c->hd_full : c->hd_swa) * 4);
    DA(m->q, (size_t)qmax * 4);
    DA(m->k, (size_t)kvmax * 4);
    DA(m->v, (size_t)kvmax * 4);
    DA(m->q_out, (size_t)qmax * 4);
    DA(m->ple, (size_t)c->ple_dim * L * 4);
    DA(m->ple_ctx, (size_t)c->ple_dim * L * 4);
    DA(m->ple_gate, (size_t)c->ple_dim * 4);
    DA(m->logits, (size_t)c->vocab * 4);
    DA(m->q8, g4_q8K_bytes(q8n));
    DA(m->dstep, 64);
    DA(m->argmax_part, g4_mm_argmax_part_bytes(c->vocab));
    DA(m->gen_hist, (size_t)c->max_seq * 4);
    DA(m->sample_part, g4_sample_part_bytes(c->vocab));
    /* the PLE gate -> projection hand-off (zeroed once; the sequence word
     * only grows, so no earlier step's pairs ever count).  G4E_PLE_FUSED=0:
     * separate launches */
    const char *pf = getenv("G4E_PLE_FUSED");
    if (!(pf && atoi(pf) == 0) && c->ple_dim > 0) {
        m->ple_pairs_stride = (g4_ple_pairs_bytes(c->ple_dim) + 255) / 256 * 256;
        DA(m->ple_pairs, m->ple_pairs_stride * L);
        CK(g4_memset(m->ple_pairs, 0, m->ple_pairs_stride * L));
        DA(m->ple_seq, 256);
        CK(g4_memset(m->ple_seq, 0, 256));
    }
    /* KV: sliding-window layers keep a ring of `window` slots, full layers
     * max_seq slots; row stride = n_kv * head_dim of the layer */
    for (int l = 0; l < L && l < E_N_LAYER_KV; l++) {
        const int kvd = c->n_kv * layer_hd(c, l);
        int slots = c->max_seq, ring = 0;
        if (is_swa(c, l) && c->window > 0 && c->window < c->max_seq) { slots = c->window; ring = c->window; }
        DA(m->kc[l], (size_t)slots * kvd * 4);
        DA(m->vc[l], (size_t)slots * kvd * 4);
        m->kv_ring[l] = ring;
    }
    /* attention partials: chunk counts fixed from capacity (<= 1024 positions
     * per chunk) so that one captured graph serves every position */
    const int cap_swa = c->window > 0 && c->window < c->max_seq ? c->window : c->max_seq;
    m->G_swa = attn_chunks(cap_swa);
    m->G_full = attn_chunks(c->max_seq);
    /* G4E_ATTN_CHUNKS_SWA=<n>: time chunks of the sliding layers' decode
     * attention (a tuning knob; the same results within the attention bar) */
    const char *gs = getenv("G4E_ATTN_CHUNKS_SWA");
    if (gs && atoi(gs) >= 1 && atoi(gs) <= 128 && (cap_swa + atoi(gs) - 1) / atoi(gs) <= 1024) m->G_swa = atoi(gs);
    /* G4E_ATTN_CHUNKS_FULL=<n>: the same for the global layers */
    const char *gf = getenv("G4E_ATTN_CHUNKS_FULL");
    if (gf && atoi(gf) >= 1 && atoi(gf) <= 128 && (c->max_seq + atoi(gf) - 1) / atoi(gf) <= 1024) m->G_full = atoi(gf);
    const int Gmax = m->G_full > m->G_swa ? m->G_full : m->G_swa;
    DA(m->attn_part, g4_attn_part_bytes(c->n_heads, hdmax, Gmax));
#undef DA
    if ((rc = dalloc(m, &p, (size_t)(c->rot_swa / 2 + c->rot_full / 2) * 8))) return rc;
    m->rope_tab = p;
    CK(g4_host_alloc((void **)&m->hstep, 64));
    memset(m->hstep, 0, 64);
    return 0;
}

static int open_image(const uint8_t *data, size_t size, int max_seq, g4e_model *m) {
    Image im;
    int rc = parse(data, size, max_seq, &m->c, &im);
    if (rc) return rc;
    rc = validate(&m->c, &im);
    if (rc == 0) rc = load(m, &im);
    free(im.ti);
    return rc;
}

int g4e_open_image(const void *data, size_t size, int max_seq, int device, g4e_model **out) {
    if (!data || !out) return fail(G4_ERR_ARG, "g4e_open_image: null pointer");
    *out = NULL;
    CK(g4_init(device));
    g4e_model *m = (g4e_model *)calloc(1, sizeof *m);
    if (!m) return fail(G4_ERR_NOMEM, "out of host memory");
    int rc = g4_stream_create(&m->stream);
    if (rc) { free(m); return lib_fail(rc, "g4_stream_create"); }
    g4_set_stream(m->stream);
    /* G4E_POISON=<byte>: fill every device buffer with that byte when it is
     * allocated (0xff: NaN floats), so that a read of memory no kernel has
     * written shows in the results */
    const char *poison = getenv("G4E_POISON");
    m->poison = poison && *poison ? (int)(strtol(poison, NULL, 0) & 0xff) : -1;
    /* G4E_PREFILL_IMAGES=0: no fp16 weight images (the prompt's batched GEMMs
     * then decode the K-quant blocks in the kernel: slower, same results) */
    const char *imgs = getenv("G4E_PREFILL_IMAGES");
    m->no_img = imgs && *imgs == '0';
    m->pf_chunk = G4E_PREFILL_CHUNK;
    m->dump_at = -1;
    rc = open_image((const uint8_t *)data, size, max_seq, m);
    if (rc == 0) rc = g4_sync() ? lib_fail(G4_ERR_HIP, "g4_sync") : 0;
    if (rc) { g4e_close(m); return rc; }
    *out = m;
    return 0;
}

int g4e_open_file(const char *path, int max_seq, int device, g4e_model **out) {
    if (!path || !out) return fail(G4_ERR_ARG, "g4e_open_file: null pointer");
    const int fd = open(path, O_RDONLY);
    if (fd < 0) return fail(G4_ERR_ARG, "Error: cannot open %s", path);
    struct stat st;
    if (fstat(fd, &st) != 0) { close(fd); return fail(G4_ERR_ARG, "Error: cannot stat %s", path); }
    void *p = mmap(NULL, (size_t)st.st_size, PROT_READ, MAP_PRIVATE, fd, 0);
    close(fd);
    if (p == MAP_FAILED) return fail(G4_ERR_NOMEM, "Error: mmap failed");
    const int rc = g4e_open_image(p, (size_t)st.st_size, max_seq, device, out);
    munmap(p, (size_t)st.st_size);
    return rc;
}

void g4e_close(g4e_model *m) {
    if (!m) return;
    g4_set_stream(m->stream);
    g4_sync();
    if (m->graph) g4_graph_destroy(m->graph);
    if (m->sgraph) g4_graph_destroy(m->sgraph);
    for (int i = 0; i < m->n_allocs; i++) g4_free(m->allocs[i]);
    if (m->hstep) g4_host_free(m->hstep);
    g4_set_stream(NULL);
    if (m->stream) g4_stream_destroy(m->stream);
    free(m->layer_x);
    free(m->layer_q8);
    free(m);
}

void g4e_config(const g4e_model *m, int out[9]) {
    const Config *c = &m->c;
    const int v[9] = {c->dim, c->hidden, c->n_layers, c->n_heads, c->n_kv, c->vocab, c->max_seq, c->ple_dim, c->window};
    memcpy(out, v, sizeof v);
}

/* ---- the step, main.c:1838-2029 ------------------------------------------ */

/* mm(o, x, w, n, d, type, q8, q8_ready), main.c:1669-1694 */
static int mm(g4e_model *m, float *o, const float *x, const Tensor *w, int q8_ready) {
    if (m->f32_matmul && is_kq45(w->type)) CK(g4_mm_quant_rows(o, x, w->p, w->n, w->d, w->type));
    else CK(g4_mm(o, x, w->p, w->n, w->d, w->type, m->q8, q8_ready));
    return 0;
}

/* Enqueue one forward step; token and position are read from m->dstep, so the
 * same sequence of launches is valid for every position (graph capture). */
/* a Q4_K/Q5_K GEMV that can take the residual step + norm + Q8_K as its
 * prologue (g4_mm_residual_q8) */
/* does mm() take this matrix through Q8_K activations (main.c:1676-1685)? */
static int q8t(const g4e_model *m, int t) { return is_kq45(t) && !m->f32_matmul; }

static int trace_pull(g4e_model *m);

/* dump_kv_fingerprint (main.c:1829-1836) of a device vector: hidden_stats
 * and its first four values, into tag t of the layer-0 record */
static int fp_tag(g4e_model *m, int t, const float *v, int n) {
    CK(g4_hidden_stats(v, n, m->dfp + 7 * t));
    CK(g4_memcpy_d2d_async(m->dfp + 7 * t + 3, v, (size_t)(n < 4 ? n : 4) * 4));
    m->fp_have[t] = 1;
    return 0;
}
/* K before RoPE: k_norm applied to a copy of the projection (main.c:1895) */
static int fp_k_pre_rope(g4e_model *m, const float *k) {
    const int hd = layer_hd(&m->c, 0), kvd = m->c.n_kv * hd;
    CK(g4_memcpy_d2d_async(m->dfp_k, k, (size_t)kvd * 4));
    CK(g4_rmsnorm_head_inplace(m->dfp_k, m->k_norm[0], m->c.n_kv, hd, m->c.eps));
    return fp_tag(m, G4E_FP_K_PRE_ROPE, m->dfp_k, kvd);
}
/* the cache row of layer 0 that holds position p, or NULL once a ring has
 * overwritten it (the reference's flat cache keeps every position) */
static const float *kc0_row(const g4e_model *m, int p, int pos) {
    const int kvd = m->c.n_kv * layer_hd(&m->c, 0), ring = m->kv_ring[0];
    if (ring > 0 && pos - p >= ring) return NULL;
    return m->kc[0] + (size_t)(ring > 0 ? p % ring : p) * kvd;
}

/* Traced steps: the Q8_K activation of quantization point `slot` of layer
 * l, re-quantized from the stored fp32 vector vec[n] (the fused kernels
 * quantize the same values in registers; the quantization is deterministic),
 * for the matrices that take Q8_K inputs. */
static int trace_q8(g4e_model *m, int l, int slot, const float *vec, int n, int type) {
    if (!m->trace || !q8t(m, type) || n % 256 || n > G4E_Q8_SLOT_ELEMS) return 0;
    uint8_t *dst = (uint8_t *)m->dtr_q8 + ((size_t)l * G4E_Q8_SLOTS + slot) * g4_q8K_bytes(G4E_Q8_SLOT_ELEMS);
    return g4_quantize_row_q8_K(vec, dst, n);
}

static int pro_ok(const g4e_model *m, const Tensor *w) {
    const int nb = m->c.dim / 256;
    return q8t(m, w->type) && m->c.dim % 256 == 0 && (nb == 8 || nb == 10 || nb == 16);
}

/* g4_mm_ple_gate_proj's shape: n = 2560, a 256-wide PLE, K-quant gate and
 * projection, and the step's sequence word advanced by the first launch */
static int ple_fused_ok(const g4e_model *m, int l) {
    const Config *c = &m->c;
    return m->ple_pairs && m->ple_seq && c->dim == 2560 && c->ple_dim == 256 && q8t(m, m->inp_gate[l].type) &&
           q8t(m, m->proj[l].type) && m->ple_proj.type == G4_BF16 && (int)m->ple_proj.n == c->dim;
}

/* Enqueue one forward step; token and position are read from m->dstep, so the
 * same sequence of launches is valid for every position (graph capture).
 * The residual stream lives in two buffers: a GEMV whose prologue performs
 * a residual step reads one and writes the other (its workgroups run
 * concurrently); single-workgroup steps update it in place. */
static int enqueue_step(g4e_model *m, int lm_mode) {
    const Config *c = &m->c;
    const int dim = c->dim, L = c->n_layers, pd = c->ple_dim;
    const int *dtok = m->dstep, *dpos = m->dstep + 1;
    float *x = m->x, *xo = m->x_alt;
    /* emb_lookup * sqrt(dim) (main.c:1849-1854) with the (cos, sin) tables of
     * both RoPE variants at this position (main.c:1725-1742) in one launch,
     * then build_ple (main.c:1747-1778) */
    float *tab_swa = m->rope_tab, *tab_full = m->rope_tab + c->rot_swa;
    if (m->ple_proj.type == G4_BF16 && (int)m->ple_proj.n == dim && dim % 8 == 0 && dim <= 4096) {
        /* with the bf16 context projection of build_ple (main.c:1749-1750)
         * in the same launch, on the same row (one launch fewer per step:
         * 2.1045 -> 2.1005 ms) */
        CK(g4_emb_lookup_rope_ple(x, m->embd.p, m->embd.type, m->embd.d, dtok, dim, sqrtf((float)dim), dpos, tab_swa,
                                  c->rot_swa, c->theta_swa, NULL, tab_full, c->rot_full, c->theta, m->rope_freqs, 1.0f,
                                  m->ple_ctx, m->ple_proj.p, (int)m->ple_proj.d, m->ple_seq));
    } else {
        CK(g4_emb_lookup_rope(x, m->embd.p, m->embd.type, m->embd.d, dtok, dim, sqrtf((float)dim), dpos, tab_swa,
                              c->rot_swa, c->theta_swa, NULL, tab_full, c->rot_full, c->theta, m->rope_freqs, 1.0f));
        CK(g4_mm(m->ple_ctx, x, m->ple_proj.p, m->ple_proj.n, m->ple_proj.d, m->ple_proj.type, m->q8, 0));
    }
    CK(g4_ple_finish(m->ple, m->ple_ctx, m->ple_tok.p, m->ple_tok.type, m->ple_tok.d, m->ple_proj_norm, dtok, 0, pd, L,
                     sqrtf((float)pd), 1.0f / sqrtf((float)dim), 1.0f / sqrtf(2.0f), c->eps));
    if (m->trace) CK(g4_memcpy_d2d_async(m->dtr_x, x, (size_t)dim * 4));
    /* --dump-hidden-at (main.c:1857-1862, 1964-1969, 2005-2010): rows after
     * the embedding, after each attention residual, at each layer's end */
    if (m->dump_now) CK(g4_hidden_stats(x, dim, m->dstats));
    for (int l = 0; l < L; l++) {
        const int hd = layer_hd(c, l), swa = is_swa(c, l);
        const int n_rot = swa ? c->rot_swa : c->rot_full;
        const int q8_att = q8t(m, m->wq[l].type);
        /* the previous layer's post_norm + residual + out_scale (main.c:1995-2003;
         * none before layer 0), this layer's attn_norm + Q8_K (main.c:1878-1884),
         * then Q, K, V on that one Q8_K of xb2 (main.c:1883-1892) */
        const float *y = l ? m->ybuf : NULL, *w_post = l ? m->post_norm[l - 1] : NULL;
        const float *osc = l ? m->out_scale[l - 1] : NULL;
        int rc;
        const int src = kv_source(c, l), has_kv = layer_has_kv(l);
        /* K rides in the Q launch when it has Q's type, and V with them when it
         * is Q6_K (fp32 path on the normed vector) */
        const int k_pair = has_kv && pro_ok(m, &m->wq[l]) && m->wk[l].type == m->wq[l].type;
        const int v_too = k_pair && m->wv[l].type == G4_Q6_K;
        if (v_too) {
            CK(g4_mm_residual_q8_qkv(m->q, m->wq[l].p, m->wq[l].d, m->k, m->wk[l].p, m->wk[l].d, m->v, m->wv[l].p,
                                     m->wv[l].d, m->wv[l].type, m->wq[l].n, m->wq[l].type, x, y ? xo : x, y, w_post, osc,
                                     m->attn_norm[l], m->xb2, m->q8, c->eps));
            if (y) { float *t = x; x = xo; xo = t; }
        } else if (k_pair) {
            CK(g4_mm_residual_q8_pair(m->q, m->wq[l].p, m->wq[l].d, m->k, m->wk[l].p, m->wk[l].d, m->wq[l].n,
                                      m->wq[l].type, x, y ? xo : x, y, w_post, osc, m->attn_norm[l], m->xb2, m->q8, 0,
                                      c->eps));
            if (y) { float *t = x; x = xo; xo = t; }
        } else if (pro_ok(m, &m->wq[l])) {
            CK(g4_mm_residual_q8(m->q, m->wq[l].p, NULL, m->wq[l].n, m->wq[l].d, m->wq[l].type, NULL, x, y ? xo : x, y,
                                 w_post, osc, m->attn_norm[l], m->xb2, m->q8, 0, c->eps));
            if (y) { float *t = x; x = xo; xo = t; }
        } else {
            CK(g4_residual_norm(x, y, w_post, osc, m->attn_norm[l], m->xb2, q8_att ? m->q8 : NULL, 0, dim, c->eps));
            if ((rc = mm(m, m->q, m->xb2, &m->wq[l], q8_att))) return rc;
        }
        if (m->trace && l > 0) CK(g4_memcpy_d2d_async(m->dtr_x + (size_t)l * dim, x, (size_t)dim * 4));
        if (m->dump_now && l == 0) {
            memset(m->fp_have, 0, sizeof m->fp_have);
            CK(fp_tag(m, G4E_FP_ATTN_NORM, m->xb2, dim));
        }
        CK(trace_q8(m, l, G4E_Q8_SLOT_ATTN, m->xb2, dim, m->wq[l].type));
        if (m->dump_now && l > 0) CK(g4_hidden_stats(x, dim, m->dstats + 3 * (2 * l)));
        if (has_kv) {
            if (!q8_att && (q8t(m, m->wk[l].type) || q8t(m, m->wv[l].type)))
                CK(g4_quantize_row_q8_K(m->xb2, m->q8, dim));
            if (!k_pair && (rc = mm(m, m->k, m->xb2, &m->wk[l], 1))) return rc;
            if (!v_too && (rc = mm(m, m->v, m->xb2, &m->wv[l], 1))) return rc;
        }
        if (m->dump_now && l == 0 && has_kv) {
            CK(fp_tag(m, G4E_FP_K_PRE_NORM, m->k, c->n_kv * hd));
            CK(fp_k_pre_rope(m, m->k));
        }
        /* q_norm + RoPE, K/V norm + RoPE + append (main.c:1886-1904) and the
         * attention over the source layer's cache (main.c:1909-1950, attn_scale
         * 1.0) in one launch pair */
        const int o_q8 = q8t(m, m->wo[l].type);
        const int G_att = swa ? m->G_swa : m->G_full;
        /* the chunk partials merged in the O GEMV's prologue (g4_mm_attn_merge)
         * on the sliding layers: one launch fewer per layer, the same bits.
         * Not on the global layers (head_dim 512): at the E4B shape with 16
         * chunks their merge prologue (1024-thread workgroups over 4096
         * inputs, 80 of them) made the step 25 us slower than the separate
         * merge and O GEMV with 32 chunks */
        const int o_merge = o_q8 && hd == 256 && G_att <= G4_MERGE_MAX_CHUNKS &&
                            (c->n_heads == 8 || c->n_heads == 16);
        const int keep_qout = !o_merge || m->trace || m->dump_now;
        CK(g4_attn_decode_fused(m->q, m->q_norm[l], has_kv ? m->k : NULL, has_kv ? m->v : NULL,
                                has_kv ? m->k_norm[l] : NULL, has_kv ? m->kc[l] : NULL, has_kv ? m->vc[l] : NULL,
                                m->kc[src], m->vc[src], c->n_kv * layer_hd(c, src), m->kv_ring[src], dpos,
                                swa ? c->window : 0, c->n_heads, c->n_kv, hd, n_rot, swa ? tab_swa : tab_full, c->eps,
                                1.0f, G_att, m->attn_part, o_merge ? NULL : m->q_out, o_q8 && !o_merge ? m->q8 : NULL));
        if (o_merge)
            CK(g4_mm_attn_merge(m->xb2, m->wo[l].p, m->wo[l].n, m->wo[l].d, m->wo[l].type, m->attn_part, G_att,
                                c->n_heads, hd, keep_qout ? m->q_out : NULL, NULL));
        CK(trace_q8(m, l, G4E_Q8_SLOT_O, m->q_out, c->n_heads * hd, m->wo[l].type));
        if (m->dump_now && l == 0) {
            const int p = m->dump_at, kvd = c->n_kv * hd;
            if (has_kv) CK(fp_tag(m, G4E_FP_K_STORE, kc0_row(m, p, p), kvd));
            const float *r0 = kc0_row(m, 0, p);
            if (r0) CK(fp_tag(m, G4E_FP_K_READ0, r0, kvd));
            if (p > 0) CK(fp_tag(m, G4E_FP_K_READN, kc0_row(m, p, p), kvd));
            CK(fp_tag(m, G4E_FP_Q_OUT, m->q_out, c->n_heads * hd));
        }
        if (!o_merge && (rc = mm(m, m->xb2, m->q_out, &m->wo[l], o_q8))) return rc;
        /* post_attention_norm + residual, then ffn_norm + Q8_K (main.c:1960-1975)
         * and gelu(gate) * up (main.c:1976-1980) */
        const int q8_ffn = q8t(m, m->gate[l].type) || q8t(m, m->up[l].type);
        if (q8t(m, m->gate[l].type) && m->gate[l].type == m->up[l].type && pro_ok(m, &m->gate[l])) {
            /* the residual step as the prologue of every workgroup of the
             * gate|up GEMV (one wave per Q8_K block); the normed vector and
             * its Q8_K are stored only for a trace (hb2: xb2 holds y) */
            const int keep = m->trace || m->dump_now;
            CK(g4_mm_residual_q8(m->hb, m->gate[l].p, m->up[l].p, dim, c->hidden, m->gate[l].type, NULL, x, xo, m->xb2,
                                 m->post_attn_norm[l], NULL, m->ffn_norm[l], keep ? m->hb2 : NULL,
                                 keep ? m->q8 : NULL, 0, c->eps));
            float *t = x; x = xo; xo = t;
            if (m->dump_now) CK(g4_hidden_stats(x, dim, m->dstats + 3 * (1 + 2 * l)));
            CK(trace_q8(m, l, G4E_Q8_SLOT_FFN, m->hb2, dim, m->gate[l].type));
        } else {
            CK(g4_residual_norm(x, m->xb2, m->post_attn_norm[l], NULL, m->ffn_norm[l], m->xb2, q8_ffn ? m->q8 : NULL, 0,
                                dim, c->eps));
            if (m->dump_now) CK(g4_hidden_stats(x, dim, m->dstats + 3 * (1 + 2 * l)));
            CK(trace_q8(m, l, G4E_Q8_SLOT_FFN, m->xb2, dim, m->gate[l].type));
            if (q8t(m, m->gate[l].type) && m->gate[l].type == m->up[l].type) {
                CK(g4_mm_gate_up_gelu(m->hb, m->gate[l].p, m->up[l].p, dim, c->hidden, m->gate[l].type, m->q8));
            } else {
                if ((rc = mm(m, m->hb, m->xb2, &m->gate[l], 1)) || (rc = mm(m, m->hb2, m->xb2, &m->up[l], 1))) return rc;
                CK(g4_gelu_mul_rows(m->hb, m->hb, m->hb2, c->hidden, 1, c->hidden));
            }
        }
        /* down (main.c:1981) */
        if ((rc = mm(m, m->xb2, m->hb, &m->down[l], 0))) return rc;
        /* post_ffw_norm + residual, Q8_K of x (main.c:1982-1988) and the
         * inp_gate GEMV with gelu * ple[l] in its epilogue (main.c:1988-1993) */
        if (ple_fused_ok(m, l) && !m->trace && !m->dump_now) {
            /* with proj (main.c:1994) in the same launch: the gate values
             * reach the projection's workgroups as (value, step) pairs */
            CK(g4_mm_ple_gate_proj(m->ybuf, m->proj[l].p, m->proj[l].type, (int)m->proj[l].d, m->inp_gate[l].p,
                                   m->inp_gate[l].type, dim, pd, m->ple + (size_t)l * pd, x, xo, m->xb2,
                                   m->post_ffw_norm[l], c->eps, (uint8_t *)m->ple_pairs + (size_t)l * m->ple_pairs_stride,
                                   m->ple_seq));
            float *t = x; x = xo; xo = t;
            continue;
        }
        if (pro_ok(m, &m->inp_gate[l])) {
            CK(g4_mm_residual_q8(m->ple_gate, m->inp_gate[l].p, NULL, dim, pd, m->inp_gate[l].type, m->ple + (size_t)l * pd, x,
                                 xo, m->xb2, m->post_ffw_norm[l], NULL, NULL, NULL, NULL, 1, c->eps));
            float *t = x; x = xo; xo = t;
        } else {
            const int q8_ig = q8t(m, m->inp_gate[l].type);
            CK(g4_residual_norm(x, m->xb2, m->post_ffw_norm[l], NULL, NULL, NULL, q8_ig ? m->q8 : NULL, 1, dim, c->eps));
            if (q8_ig) {
                CK(g4_mm_quant_dot_rows_gelu_mul(m->ple_gate, m->inp_gate[l].p, dim, pd, m->inp_gate[l].type, m->q8,
                                                 m->ple + (size_t)l * pd));
            } else {
                if ((rc = mm(m, m->ple_gate, x, &m->inp_gate[l], 0))) return rc;
                CK(g4_gelu_mul_quant(m->ple_gate, m->ple + (size_t)l * pd, pd, NULL));
            }
        }
        CK(trace_q8(m, l, G4E_Q8_SLOT_INP_GATE, x, dim, m->inp_gate[l].type));
        CK(trace_q8(m, l, G4E_Q8_SLOT_PROJ, m->ple_gate, pd, m->proj[l].type));
        /* proj (main.c:1994): mm() quantizes its 256-wide input inside the GEMV;
         * its residual step runs in the next layer's Q launch */
        if ((rc = mm(m, m->ybuf, m->ple_gate, &m->proj[l], 0))) return rc;
    }
    /* the last layer's post_norm + residual + out_scale and the final norm
     * (main.c:1995-2003, 2021) */
    CK(g4_residual_norm(x, m->ybuf, m->post_norm[L - 1], m->out_scale[L - 1], lm_mode ? m->norm_out : NULL,
                        lm_mode ? m->xb2 : NULL, NULL, 0, dim, c->eps));
    if (m->trace) CK(g4_memcpy_d2d_async(m->dtr_x + (size_t)L * dim, x, (size_t)dim * 4));
    if (m->dump_now) CK(g4_hidden_stats(x, dim, m->dstats + 3 * (2 * L)));
    m->x_last = x;
    if (lm_mode == 0) return 0;
    /* lm_mode 2, the greedy step: logits_tied and the first-index argmax in
     * one pass (main.c:1570-1667 / 1784-1786 when there is no soft-cap; with
     * one, the argmax of the soft-capped logits of main.c:1788-1795,
     * 2045-2049 -- the same token), which also stores the token as the next
     * input and advances the position */
    if (lm_mode == 2) {
        CK(g4_mm_argmax_row(m->xb2, m->embd.p, dim, c->vocab, m->embd.type, m->q8, c->softcap, m->logits,
                            m->argmax_part, m->dstep + 2, m->dstep, m->dstep + 1));
        return 0;
    }
    /* logits_tied (main.c:1780-1796): the embedding rows times the final-normed
     * hidden (kept in xb2), soft-cap; fused for a Q6_K table */
    if (m->embd.type == G4_Q6_K) {
        CK(g4_mm_quant_rows_softcap(m->logits, m->xb2, m->embd.p, dim, c->vocab, m->embd.type, c->softcap));
    } else {
        int rc = mm(m, m->logits, m->xb2, &m->embd, 0);
        if (rc) return rc;
        if (c->softcap > 0.0f) CK(g4_softcap(m->logits, c->vocab, c->softcap));
    }
    return 0;
}

/* ---------------------------------------------------------------------------
 * Prompt chunks: the forward() of m consecutive prompt tokens with lm_mode 0
 * (main.c:2366-2384 runs them one at a time), layer by layer over all m
 * tokens: the Q4_K/Q5_K projections through the batched GEMM (per-block
 * integer sums exact, fp32 fold in another order: within 1e-5 of the decode
 * GEMV's outputs, and the same bits for a token in any chunking), norms and
 * residual steps through the rows
 * forms of the decode step's kernels (same thread layout, so the same bits
 * per row), attention over m query rows.  A sliding-window ring cannot hold
 * every query's window while the chunk's own positions are appended, so each
 * storing layer writes its chunk's K/V to a chunk buffer, the attention reads
 * positions >= p0 from there and earlier ones from the cache, and the chunk
 * is appended to the cache afterwards (for the shared-KV donors 22 and 23
 * after the last layer, when their readers are done).  Only the KV caches
 * carry over to the next token, as in the reference.
 * ------------------------------------------------------------------------- */
static int pf_alloc(g4e_model *m, int cap) {
    const Config *c = &m->c;
    const int L = c->n_layers, pd = c->ple_dim;
    const int hdmax = c->hd_full > c->hd_swa ? c->hd_full : c->hd_swa;
    const int qmax = c->n_heads * hdmax, kvmax = c->n_kv * hdmax;
    int q8n = c->hidden > qmax ? c->hidden : qmax;
    if (c->dim > q8n) q8n = c->dim;
    q8n = (q8n + 255) / 256 * 256;
    const size_t M = (size_t)cap;
    int rc;
    void *p;
    m->pf_Gmax = (c->max_seq + 1023) / 1024;
    if (m->pf_Gmax < 16) m->pf_Gmax = 16;
#define PA(field, bytes) if ((rc = dalloc(m, &p, (size_t)(bytes)))) return rc; field = p;
    PA(m->pf_tok, M * 4);
    PA(m->pf_x, M * c->dim * 4);
    PA(m->pf_xb2, M * c->dim * 4);
    PA(m->pf_q, M * qmax * 4);
    PA(m->pf_k, M * kvmax * 4);
    PA(m->pf_v, M * kvmax * 4);
    PA(m->pf_ao, M * qmax * 4);
    PA(m->pf_o, M * c->dim * 4);
    PA(m->pf_g, M * c->hidden * 4);
    PA(m->pf_u, M * c->hidden * 4);
    PA(m->pf_h, M * c->hidden * 4);
    PA(m->pf_d, M * c->dim * 4);
    PA(m->pf_ig, M * pd * 4);
    PA(m->pf_pg, M * pd * 4);
    PA(m->pf_ub, (size_t)(c->dim / 256) * M * pd * 4);
    PA(m->pf_y, M * c->dim * 4);
    PA(m->pf_ple, M * L * pd * 4);
    PA(m->pf_ctx, M * L * pd * 4);
    PA(m->pf_tab_swa, M * (size_t)(c->rot_swa / 2) * 8);
    PA(m->pf_tab_full, M * (size_t)(c->rot_full / 2) * 8);
    PA(m->pf_part, M * g4_attn_part_bytes(c->n_heads, hdmax, m->pf_Gmax));
    PA(m->pf_q8, M * g4_q8K_row_stride(q8n));
    PA(m->pf_q8a, M * g4_q8K_row_stride((qmax + 255) / 256 * 256));
    PA(m->pf_q8p, M * g4_q8K_row_stride((pd + 255) / 256 * 256));
    PA(m->pf_xs, g4_split_rows_bytes(q8n, (int)M));
    m->pf_xs_n = q8n;
    for (int i = 0; i < 3; i++) {
        PA(m->pf_kch[i], M * kvmax * 4);
        PA(m->pf_vch[i], M * kvmax * 4);
    }
#undef PA
    /* fp16 images of the FFN gate and up matrices (Q4_K / Q5_K) for the chunk
     * GEMMs: built once, on the first prompt chunk, so decode-only use does
     * not hold them.  (The 2560-row matrices measured the same on images as
     * on the quantized tensors, with cold weights: O 19.2, Q|K 24.9 against
     * 25.4, proj 6.2 against 6.0 us at 511 tokens; gate|up 102 against 116.)
     * They are an optimisation with the same results: when HBM cannot hold
     * them, the matrices left without one take the quantized-tensor GEMM. */
    if (!m->no_img && !m->f32_matmul) {
        for (int l = 0; l < L && !m->no_img; l++) {
            Tensor *ts[2] = {&m->gate[l], &m->up[l]};
            for (int k = 0; k < 2; k++) {
                Tensor *t = ts[k];
                const size_t b = t->p && is_kq45(t->type) ? g4_kq_image_bytes(t->n, t->d) : 0;
                if (!b || t->img) continue;
                if (dalloc_opt(m, &t->img, b)) {
                    m->no_img = 1;   /* out of device memory: no more images */
                    break;
                }
                CK(g4_kq_image(t->img, t->p, t->n, t->d, t->type));
            }
        }
    }
    m->pf_cap = cap;
    return 0;
}

/* chunk K/V buffer of layer l (storing layers) */
static int pf_slot(int l) { return l == 22 ? 1 : l == 23 ? 2 : 0; }

/* the batched GEMM of a Q4_K / Q5_K matrix on M Q8_K rows: on its fp16 image
 * when it has one (same results) */
static int kq_batch(g4e_model *m, float *o, const Tensor *w, const void *q8, int M) {
    (void)m;
    if (w->img)
        return g4_mm_batch_img(o, w->img, q8, w->n, w->d, M, w->type) ? lib_fail(G4_ERR_HIP, "g4_mm_batch_img") : 0;
    return g4_mm_batch_q8(o, w->p, q8, w->n, w->d, M, w->type) ? lib_fail(G4_ERR_HIP, "g4_mm_batch_q8") : 0;
}

/* mm over the chunk's rows: K-quant through the batched GEMM on the Q8_K rows
 * (q8_ready: already quantized by the preceding residual step), the other
 * types per token */
static int mm_rows(g4e_model *m, float *o, const float *x, const Tensor *w, int M, int q8_ready) {
    if (m->f32_matmul && is_kq45(w->type)) {
        for (int z = 0; z < M; z++)
            CK(g4_mm_quant_rows(o + (size_t)z * w->d, x + (size_t)z * w->n, w->p, w->n, w->d, w->type));
        return 0;
    }
    if (q8t(m, w->type) && q8_ready) return kq_batch(m, o, w, m->pf_q8, M);
    if (w->type == G4_Q6_K && w->n % 256 == 0 && w->n <= m->pf_xs_n) {
        CK(g4_split_rows_f16(x, m->pf_xs, w->n, M));
        CK(g4_mm_batch_split(o, w->p, m->pf_xs, w->n, w->d, M, w->type));
        return 0;
    }
    if (w->type == G4_BF16 && w->n % 256 == 0)
        return g4_mm_batch_bf16_f32(o, x, w->p, w->n, w->d, M) ? lib_fail(G4_ERR_HIP, "g4_mm_batch_bf16_f32") : 0;
    return g4_mm_batch(o, x, w->p, w->n, w->d, M, w->type, m->pf_q8) ? lib_fail(G4_ERR_HIP, "g4_mm_batch") : 0;
}

/* the same as mm_rows for two or three matrices over the same Q8_K rows:
 * one launch when they share the K-quant type (gate and up; Q and K) */
static int mm_rows_multi(g4e_model *m, float *const *o, const Tensor *const *w, int nw, int M) {
    int same = !m->f32_matmul && is_kq45(w[0]->type);
    for (int k = 1; k < nw; k++) same = same && w[k]->type == w[0]->type && w[k]->n == w[0]->n;
    if (!same) {
        for (int k = 0; k < nw; k++) CK(mm_rows(m, o[k], NULL, w[k], M, 1));
        return 0;
    }
    const void *wp[3], *ip[3];
    int d[3], imgs = 1;
    for (int k = 0; k < nw; k++) {
        wp[k] = w[k]->p;
        ip[k] = w[k]->img;
        d[k] = w[k]->d;
        imgs = imgs && w[k]->img;
    }
    if (imgs)
        return g4_mm_batch_img_multi(o, ip, d, nw, m->pf_q8, w[0]->n, M, w[0]->type)
                   ? lib_fail(G4_ERR_HIP, "g4_mm_batch_img_multi")
                   : 0;
    return g4_mm_batch_q8_multi(o, wp, d, nw, m->pf_q8, w[0]->n, M, w[0]->type) ? lib_fail(G4_ERR_HIP, "g4_mm_batch_q8_multi") : 0;
}

/* One prompt chunk of M tokens at positions p0..p0+M-1, layer by layer.
 * trace (optional, host): each layer's input rows go to trace[(l*ntot + t0 +
 * z)*dim] and the last layer's output to l = n_layers; ntot is the whole
 * prompt's length and t0 this chunk's first row. */
/* q8trace (optional, host): the Q8_K rows of each quantization point, as
 * BlockQ8_K structs at [l][t0 + z][slot][G4E_Q8_SLOT_ELEMS / 256]; staged
 * through q8stage (M * G4E_Q8_SLOT_ELEMS / 256 blocks) */
typedef struct { uint8_t *out, *stage; int ntot, t0, M; } Q8Trace;

static int pf_trace_q8(g4e_model *m, const Q8Trace *qt, int l, int slot, const void *rows, int n, int type) {
    if (!qt || !q8t(m, type) || n % 256 || n > G4E_Q8_SLOT_ELEMS) return 0;
    CK(g4_download_q8K_rows(rows, qt->stage, n, qt->M));
    const size_t row = (size_t)(n / 256) * 292, slot_b = (size_t)(G4E_Q8_SLOT_ELEMS / 256) * 292;
    for (int z = 0; z < qt->M; z++)
        memcpy(qt->out + (((size_t)l * qt->ntot + qt->t0 + z) * G4E_Q8_SLOTS + slot) * slot_b, qt->stage + z * row, row);
    return 0;
}

static int enqueue_prefill_chunk(g4e_model *m, int p0, int M, float *trace, int ntot, int t0, const Q8Trace *qt) {
    const Config *c = &m->c;
    const int dim = c->dim, L = c->n_layers, pd = c->ple_dim;
    int rc;
    CK(g4_emb_lookup_rows(m->pf_x, m->embd.p, m->embd.type, m->embd.d, m->pf_tok, M, dim, sqrtf((float)dim)));
    /* the --dump-hidden-at row of this chunk, if any */
    const float *dump_row = m->dump_at >= p0 && m->dump_at < p0 + M ? m->pf_x + (size_t)(m->dump_at - p0) * dim : NULL;
    if (dump_row) CK(g4_hidden_stats(dump_row, dim, m->dstats));
    if ((rc = mm_rows(m, m->pf_ctx, m->pf_x, &m->ple_proj, M, 0))) return rc;
    CK(g4_ple_finish_rows(m->pf_ple, m->pf_ctx, m->ple_tok.p, m->ple_tok.type, m->ple_tok.d, m->ple_proj_norm,
                          m->pf_tok, M, pd, L, sqrtf((float)pd), 1.0f / sqrtf((float)dim), 1.0f / sqrtf(2.0f), c->eps));
    CK(g4_rope_table_rows(m->pf_tab_swa, p0, M, c->rot_swa, c->theta_swa, 1.0f, NULL));
    CK(g4_rope_table_rows(m->pf_tab_full, p0, M, c->rot_full, c->theta, 1.0f, m->rope_freqs));
    for (int l = 0; l < L; l++) {
        const int hd = layer_hd(c, l), swa = is_swa(c, l);
        const int n_rot = swa ? c->rot_swa : c->rot_full;
        const int src = kv_source(c, l), has_kv = layer_has_kv(l);
        const int kvd = c->n_kv * hd, kvd_src = c->n_kv * layer_hd(c, src);
        const int q8_att = q8t(m, m->wq[l].type);
        /* residual step of the previous layer + attn_norm (+ Q8_K rows) */
        CK(g4_residual_norm_rows(m->pf_x, l ? m->pf_y : NULL, l ? m->post_norm[l - 1] : NULL,
                                 l ? m->out_scale[l - 1] : NULL, m->attn_norm[l], m->pf_xb2, q8_att ? m->pf_q8 : NULL, 0,
                                 dim, c->eps, M, pro_ok(m, &m->wq[l])));
        if (trace) CK(g4_memcpy_d2h(trace + ((size_t)l * ntot + t0) * dim, m->pf_x, (size_t)M * dim * 4));
        if (q8_att) CK(pf_trace_q8(m, qt, l, G4E_Q8_SLOT_ATTN, m->pf_q8, dim, m->wq[l].type));
        if (dump_row && l > 0) CK(g4_hidden_stats(dump_row, dim, m->dstats + 3 * (2 * l)));
        const int q8k = has_kv && q8t(m, m->wk[l].type) && q8_att;
        if (q8k && m->wk[l].type == m->wq[l].type) {
            float *o2[2] = {m->pf_q, m->pf_k};
            const Tensor *w2[2] = {&m->wq[l], &m->wk[l]};
            if ((rc = mm_rows_multi(m, o2, w2, 2, M))) return rc;
        } else {
            if ((rc = mm_rows(m, m->pf_q, m->pf_xb2, &m->wq[l], M, q8_att))) return rc;
            if (has_kv && (rc = mm_rows(m, m->pf_k, m->pf_xb2, &m->wk[l], M, q8k))) return rc;
        }
        float *kch = NULL, *vch = NULL;
        if (has_kv) {
            const int q8v = q8t(m, m->wv[l].type) && q8_att;
            if ((rc = mm_rows(m, m->pf_v, m->pf_xb2, &m->wv[l], M, q8v))) return rc;
            kch = m->pf_kch[pf_slot(l)];
            vch = m->pf_vch[pf_slot(l)];
        }
        const int fp_row = dump_row && l == 0 ? m->dump_at - p0 : -1;
        if (fp_row >= 0) {
            memset(m->fp_have, 0, sizeof m->fp_have);
            CK(fp_tag(m, G4E_FP_ATTN_NORM, m->pf_xb2 + (size_t)fp_row * dim, dim));
            if (has_kv) {
                CK(fp_tag(m, G4E_FP_K_PRE_NORM, m->pf_k + (size_t)fp_row * kvd, kvd));
                CK(fp_k_pre_rope(m, m->pf_k + (size_t)fp_row * kvd));
            }
        }
        CK(g4_qkv_post_rows(m->pf_q, m->q_norm[l], has_kv ? m->pf_k : NULL, has_kv ? m->pf_v : NULL,
                            has_kv ? m->k_norm[l] : NULL, kch, vch, kvd, swa ? m->pf_tab_swa : m->pf_tab_full, M,
                            c->n_heads, c->n_kv, hd, n_rot, c->eps));
        /* attention over the query rows; chunks of <= 128 positions */
        const int window = swa ? c->window : 0;
        const int nmax = window > 0 && window < p0 + M ? window : p0 + M;
        int G = (nmax + 127) / 128;
        if (G > m->pf_Gmax) G = m->pf_Gmax;
        const int o_q8 = q8t(m, m->wo[l].type);
        CK(g4_attn_decode_rows(m->pf_q, m->kc[src], m->vc[src], m->pf_kch[pf_slot(src)], m->pf_vch[pf_slot(src)],
                               kvd_src, m->kv_ring[src], p0, M, window, c->n_heads, c->n_kv, hd, 1.0f, G, m->pf_part,
                               m->pf_ao, o_q8 ? m->pf_q8a : NULL));
        if (o_q8) CK(pf_trace_q8(m, qt, l, G4E_Q8_SLOT_O, m->pf_q8a, c->n_heads * hd, m->wo[l].type));
        if (fp_row >= 0) {
            /* this chunk's K rows are in kch; earlier positions in the cache */
            if (has_kv) CK(fp_tag(m, G4E_FP_K_STORE, kch + (size_t)fp_row * kvd, kvd));
            const float *r0 = p0 == 0 && has_kv ? kch : kc0_row(m, 0, p0 - 1);
            if (r0) CK(fp_tag(m, G4E_FP_K_READ0, r0, kvd));
            if (m->dump_at > 0 && has_kv) CK(fp_tag(m, G4E_FP_K_READN, kch + (size_t)fp_row * kvd, kvd));
            CK(fp_tag(m, G4E_FP_Q_OUT, m->pf_ao + (size_t)fp_row * c->n_heads * hd, c->n_heads * hd));
        }
        if (has_kv && pf_slot(l) == 0) CK(g4_kv_store_rows(m->kc[l], m->vc[l], kch, vch, kvd, m->kv_ring[l], p0, M, kvd));
        if (o_q8) {
            if ((rc = kq_batch(m, m->pf_o, &m->wo[l], m->pf_q8a, M))) return rc;
        } else if ((rc = mm_rows(m, m->pf_o, m->pf_ao, &m->wo[l], M, 0))) {
            return rc;
        }
        /* post_attention_norm + residual, ffn_norm + Q8_K rows; gelu(gate) * up; down */
        const int q8_ffn = q8t(m, m->gate[l].type);
        CK(g4_residual_norm_rows(m->pf_x, m->pf_o, m->post_attn_norm[l], NULL, m->ffn_norm[l], m->pf_xb2,
                                 q8_ffn ? m->pf_q8 : NULL, 0, dim, c->eps, M, 0));
        if (dump_row) CK(g4_hidden_stats(dump_row, dim, m->dstats + 3 * (1 + 2 * l)));
        if (q8_ffn) CK(pf_trace_q8(m, qt, l, G4E_Q8_SLOT_FFN, m->pf_q8, dim, m->gate[l].type));
        if (q8_ffn && m->up[l].type == m->gate[l].type) {
            float *o2[2] = {m->pf_g, m->pf_u};
            const Tensor *w2[2] = {&m->gate[l], &m->up[l]};
            if ((rc = mm_rows_multi(m, o2, w2, 2, M))) return rc;
        } else {
            if ((rc = mm_rows(m, m->pf_g, m->pf_xb2, &m->gate[l], M, q8_ffn))) return rc;
            if ((rc = mm_rows(m, m->pf_u, m->pf_xb2, &m->up[l], M, q8_ffn && q8t(m, m->up[l].type)))) return rc;
        }
        const Tensor *wd = &m->down[l];
        const int hsplit = wd->type == G4_Q6_K && !m->f32_matmul && wd->n == c->hidden && wd->n <= m->pf_xs_n &&
                           (wd->n == 2048 || wd->n == 4096 || wd->n == 8192 || wd->n == 10240 || wd->n == 12288 ||
                            wd->n == 16384);
        if (hsplit) {
            /* gelu(gate) * up straight into the split rows of the Q6_K down GEMM */
            CK(g4_gelu_mul_split_rows(m->pf_g, m->pf_u, c->hidden, m->pf_xs, c->hidden, M));
            CK(g4_mm_batch_split(m->pf_d, wd->p, m->pf_xs, wd->n, wd->d, M, wd->type));
        } else {
            CK(g4_gelu_mul_rows(m->pf_h, m->pf_g, m->pf_u, c->hidden, M, c->hidden));
            if ((rc = mm_rows(m, m->pf_d, m->pf_h, wd, M, 0))) return rc;
        }
        /* post_ffw_norm + residual, Q8_K rows of x; PLE gate and projection */
        const int q8_ig = q8t(m, m->inp_gate[l].type);
        CK(g4_residual_norm_rows(m->pf_x, m->pf_d, m->post_ffw_norm[l], NULL, NULL, NULL, q8_ig ? m->pf_q8 : NULL, 1,
                                 dim, c->eps, M, pro_ok(m, &m->inp_gate[l])));
        if (q8_ig) CK(pf_trace_q8(m, qt, l, G4E_Q8_SLOT_INP_GATE, m->pf_q8, dim, m->inp_gate[l].type));
        const int q8_pj = q8t(m, m->proj[l].type);
        if (q8_ig && pd <= 1024 && pd % 256 == 0 && dim % 256 == 0) {
            /* the gate GEMM split by K block (ten blocks in series per
             * workgroup otherwise, for 256 rows), then one pass that folds the
             * blocks, applies gelu * ple and writes the projection's Q8_K rows */
            CK(g4_mm_batch_q8_blocks(m->pf_ub, m->inp_gate[l].p, m->pf_q8, dim, pd, M, m->inp_gate[l].type));
            CK(g4_fold_gelu_mul_q8(m->pf_ub, m->pf_q8, dim, m->pf_ple + (size_t)l * pd, L * pd, m->pf_pg,
                                   q8_pj ? m->pf_q8p : NULL, pd, M));
        } else {
            if ((rc = mm_rows(m, m->pf_ig, m->pf_x, &m->inp_gate[l], M, q8_ig))) return rc;
            CK(g4_gelu_mul_rows(m->pf_pg, m->pf_ig, m->pf_ple + (size_t)l * pd, pd, M, L * pd));
            if (q8_pj) CK(g4_quantize_rows_q8_K(m->pf_pg, m->pf_q8p, pd, M));
        }
        if (q8_pj) {
            CK(pf_trace_q8(m, qt, l, G4E_Q8_SLOT_PROJ, m->pf_q8p, pd, m->proj[l].type));
            if ((rc = kq_batch(m, m->pf_y, &m->proj[l], m->pf_q8p, M))) return rc;
        } else if ((rc = mm_rows(m, m->pf_y, m->pf_pg, &m->proj[l], M, 0))) {
            return rc;
        }
    }
    if (trace || dump_row) {
        CK(g4_residual_norm_rows(m->pf_x, m->pf_y, m->post_norm[L - 1], m->out_scale[L - 1], NULL, NULL, NULL, 0, dim,
                                 c->eps, M, 0));
        if (trace) CK(g4_memcpy_d2h(trace + ((size_t)L * ntot + t0) * dim, m->pf_x, (size_t)M * dim * 4));
        if (dump_row) CK(g4_hidden_stats(dump_row, dim, m->dstats + 3 * (2 * L)));
    }
    /* the shared-KV donors' chunks, now that their readers are done */
    for (int l = 22; l <= 23 && l < L; l++)
        if (layer_has_kv(l)) {
            const int kvd = c->n_kv * layer_hd(c, l);
            CK(g4_kv_store_rows(m->kc[l], m->vc[l], m->pf_kch[pf_slot(l)], m->pf_vch[pf_slot(l)], kvd, m->kv_ring[l],
                                p0, M, kvd));
        }
    return 0;
}

int g4e_prefill_trace_q8(g4e_model *m, const int *tokens, int n, int pos0, float *trace, void *q8trace) {
    if (!m || !tokens || n < 0 || pos0 < 0) return fail(G4_ERR_ARG, "g4e_prefill: bad arguments");
    if (pos0 + n > m->c.max_seq) return fail(G4_ERR_ARG, "g4e_prefill: positions past max_seq");
    g4_set_stream(m->stream);
    int rc = 0;
    /* chunk buffers: sized by the first call, up to 512 tokens; longer
     * prompts run in chunks of that size */
    const int want = m->pf_chunk > 0 ? m->pf_chunk : G4E_PREFILL_CHUNK;
    if (m->pf_cap == 0 && n > 0 && (rc = pf_alloc(m, want < m->c.max_seq ? want : m->c.max_seq))) return rc;
    const int chunk = want < m->pf_cap ? want : m->pf_cap;
    Q8Trace qt = {(uint8_t *)q8trace, NULL, n, 0, 0};
    if (q8trace) {
        memset(q8trace, 0, (size_t)m->c.n_layers * n * G4E_Q8_SLOTS * (G4E_Q8_SLOT_ELEMS / 256) * 292);
        qt.stage = (uint8_t *)malloc((size_t)chunk * (G4E_Q8_SLOT_ELEMS / 256) * 292);
        if (!qt.stage) return fail(G4_ERR_NOMEM, "out of host memory");
    }
    for (int t0 = 0; t0 < n && rc == 0; t0 += chunk) {
        const int M = n - t0 < chunk ? n - t0 : chunk;
        qt.t0 = t0;
        qt.M = M;
        if ((rc = g4_memcpy_h2d(m->pf_tok, tokens + t0, (size_t)M * 4))) rc = lib_fail(rc, "g4_memcpy_h2d");
        else rc = enqueue_prefill_chunk(m, pos0 + t0, M, trace, n, t0, q8trace ? &qt : NULL);
    }
    free(qt.stage);
    if (rc) return rc;
    CK(g4_sync());
    return 0;
}

int g4e_prefill_trace(g4e_model *m, const int *tokens, int n, int pos0, float *trace) {
    return g4e_prefill_trace_q8(m, tokens, n, pos0, trace, NULL);
}

int g4e_prefill(g4e_model *m, const int *tokens, int n, int pos0) { return g4e_prefill_trace(m, tokens, n, pos0, NULL); }

int g4e_kv_info(const g4e_model *m, int layer, int out[2]) {
    if (!m || !out || layer < 0 || layer >= m->c.n_layers || !layer_has_kv(layer))
        return fail(G4_ERR_ARG, "g4e_kv_info: layer %d stores no KV", layer);
    const int ring = m->kv_ring[layer];
    out[0] = m->c.n_kv * layer_hd(&m->c, layer);
    out[1] = ring > 0 ? ring : m->c.max_seq;
    return 0;
}

int g4e_read_kv(g4e_model *m, int layer, int slot0, int nslots, float *k, float *v) {
    int info[2], rc;
    if ((rc = g4e_kv_info(m, layer, info))) return rc;
    if (slot0 < 0 || nslots < 0 || slot0 + nslots > info[1] || !k || !v) return fail(G4_ERR_ARG, "g4e_read_kv: bad range");
    g4_set_stream(m->stream);
    CK(g4_sync());
    CK(g4_memcpy_d2h(k, m->kc[layer] + (size_t)slot0 * info[0], (size_t)nslots * info[0] * 4));
    CK(g4_memcpy_d2h(v, m->vc[layer] + (size_t)slot0 * info[0], (size_t)nslots * info[0] * 4));
    return 0;
}

int g4e_set_dump_hidden_at(g4e_model *m, int pos) {
    if (!m) return fail(G4_ERR_ARG, "g4e_set_dump_hidden_at: null model");
    m->dump_at = pos >= 0 ? pos : -1;
    m->dump_now = 0;
    return 0;
}

int g4e_hidden_stats(g4e_model *m, float *out) {
    if (!m || !out) return fail(G4_ERR_ARG, "g4e_hidden_stats: null pointer");
    g4_set_stream(m->stream);
    CK(g4_sync());
    CK(g4_memcpy_d2h(out, m->dstats, (size_t)(2 * m->c.n_layers + 1) * 3 * 4));
    return 0;
}

int g4e_set_f32_matmul(g4e_model *m, int on) {
    if (!m) return fail(G4_ERR_ARG, "g4e_set_f32_matmul: null model");
    if (m->f32_matmul == (on != 0)) return 0;
    /* the captured steps took the other route */
    if (m->graph) { g4_graph_destroy(m->graph); m->graph = NULL; }
    if (m->sgraph) { g4_graph_destroy(m->sgraph); m->sgraph = NULL; }
    m->f32_matmul = on != 0;
    return 0;
}

int g4e_set_prefill_chunk(g4e_model *m, int tokens) {
    if (!m || tokens < 0 || tokens > G4E_PREFILL_CHUNK)
        return fail(G4_ERR_ARG, "g4e_set_prefill_chunk: %d tokens (0..%d)", tokens, G4E_PREFILL_CHUNK);
    if (m->pf_cap > 0 && tokens > m->pf_cap)
        return fail(G4_ERR_STATE, "g4e_set_prefill_chunk: chunk buffers hold %d tokens", m->pf_cap);
    m->pf_chunk = tokens;
    return 0;
}

static int set_step(g4e_model *m, int token, int pos) {
    const Config *c = &m->c;
    if (token < 0 || token >= c->vocab) return fail(G4_ERR_ARG, "token %d out of range", token);
    if (pos < 0 || pos >= c->max_seq) return fail(G4_ERR_ARG, "pos %d out of range (max_seq %d)", pos, c->max_seq);
    CK(g4_store_i32x2(m->dstep, token, pos));
    m->dump_now = m->dump_at >= 0 && pos == m->dump_at;
    return 0;
}

int g4e_forward(g4e_model *m, int token, int pos, int lm_mode) {
    if (!m) return fail(G4_ERR_ARG, "null model");
    g4_set_stream(m->stream);
    int rc = set_step(m, token, pos);
    if (rc) return rc;
    rc = enqueue_step(m, lm_mode);
    if (rc) return rc;
    CK(g4_sync());
    return trace_pull(m);
}

int g4e_read_logits(g4e_model *m, float *host) {
    g4_set_stream(m->stream);
    CK(g4_memcpy_d2h(host, m->logits, (size_t)m->c.vocab * 4));
    return 0;
}

int g4e_read_x(g4e_model *m, float *host) {
    g4_set_stream(m->stream);
    CK(g4_memcpy_d2h(host, m->x_last, (size_t)m->c.dim * 4));
    return 0;
}

int g4e_argmax(g4e_model *m, int *tok) {
    g4_set_stream(m->stream);
    CK(g4_argmax(m->logits, m->c.vocab, m->dstep + 2, m->argmax_part, NULL, NULL));
    CK(g4_memcpy_d2h(tok, m->dstep + 2, 4));
    return 0;
}

static size_t q8_trace_blocks(const g4e_model *m) { return (size_t)m->c.n_layers * G4E_Q8_SLOTS * (G4E_Q8_SLOT_ELEMS / 256); }

int g4e_set_trace(g4e_model *m, int on) {
    if (!m) return fail(G4_ERR_ARG, "g4e_set_trace: null model");
    on = on != 0;
    if (on && !m->layer_x) {
        const size_t nx = (size_t)(m->c.n_layers + 1) * m->c.dim;
        m->layer_x = (float *)calloc(nx, sizeof(float));
        m->layer_q8 = (uint8_t *)calloc(q8_trace_blocks(m), 292);
        if (!m->layer_x || !m->layer_q8) return fail(G4_ERR_NOMEM, "out of host memory");
        g4_set_stream(m->stream);
        void *p;
        int rc;
        if ((rc = dalloc(m, &p, nx * 4))) return rc;
        m->dtr_x = p;
        const size_t qb = (size_t)m->c.n_layers * G4E_Q8_SLOTS * g4_q8K_bytes(G4E_Q8_SLOT_ELEMS);
        if ((rc = dalloc(m, &p, qb))) return rc;
        CK(g4_memset(p, 0, qb));
        m->dtr_q8 = p;
    }
    if (on != m->trace) {
        /* captured steps carry the trace copies, or do not */
        if (m->graph) { g4_graph_destroy(m->graph); m->graph = NULL; }
        if (m->sgraph) { g4_graph_destroy(m->sgraph); m->sgraph = NULL; }
    }
    m->trace = on;
    return 0;
}

/* after a traced step has completed: device trace -> host copies */
static int trace_pull(g4e_model *m) {
    if (!m->trace) return 0;
    const int L = m->c.n_layers;
    CK(g4_memcpy_d2h(m->layer_x, m->dtr_x, (size_t)(L + 1) * m->c.dim * 4));
    const size_t sb = g4_q8K_bytes(G4E_Q8_SLOT_ELEMS), hb = (size_t)(G4E_Q8_SLOT_ELEMS / 256) * 292;
    for (int l = 0; l < L; l++) {
        /* each vector in the device layout of its own length */
        const Tensor *w[G4E_Q8_SLOTS] = {&m->wq[l], &m->wo[l], &m->gate[l], &m->inp_gate[l], &m->proj[l]};
        const int n[G4E_Q8_SLOTS] = {m->c.dim, m->c.n_heads * layer_hd(&m->c, l), m->c.dim, m->c.dim, m->c.ple_dim};
        for (int s = 0; s < G4E_Q8_SLOTS; s++) {
            if (!q8t(m, w[s]->type) || n[s] % 256 || n[s] > G4E_Q8_SLOT_ELEMS) continue;
            const size_t i = (size_t)l * G4E_Q8_SLOTS + s;
            CK(g4_download_q8K((const uint8_t *)m->dtr_q8 + i * sb, m->layer_q8 + i * hb, n[s]));
        }
    }
    return 0;
}

const float *g4e_layer_x(const g4e_model *m) { return m->layer_x; }
const void *g4e_layer_q8(const g4e_model *m) { return m->layer_q8; }

/* One greedy decode step as launches: forward with the LM head and argmax
 * (lm_mode 2), which also stores the token as the next input and advances
 * the position. */
static int enqueue_greedy_step(g4e_model *m) { return enqueue_step(m, 2); }

static int ensure_graph(g4e_model *m) {
    if (m->graph) return 0;
    m->dump_now = 0;
    CK(g4_graph_begin());
    int rc = enqueue_greedy_step(m);
    void *g = NULL;
    const int rc2 = g4_graph_end(&g);
    if (rc) return rc;
    if (rc2) return lib_fail(rc2, "g4_graph_end");
    m->graph = g;
    return 0;
}

static double now_s(void) {
    struct timespec t;
    clock_gettime(CLOCK_MONOTONIC, &t);
    return (double)t.tv_sec + (double)t.tv_nsec * 1e-9;
}

int g4e_decode_steps(g4e_model *m, int token, int pos0, int steps, int use_graph, int *out, double *sec) {
    if (!m || steps < 0) return fail(G4_ERR_ARG, "g4e_decode_steps: bad arguments");
    if (pos0 + steps > m->c.max_seq) return fail(G4_ERR_ARG, "decode past max_seq");
    g4_set_stream(m->stream);
    int rc = set_step(m, token, pos0);
    if (rc) return rc;
    m->dump_now = 0;   /* positions advance on the device: the timed loop records nothing */
    if (use_graph && (rc = ensure_graph(m))) return rc;
    CK(g4_sync());
    const double t0 = now_s();
    for (int s = 0; s < steps; s++) {
        if (use_graph) CK(g4_graph_launch(m->graph));
        else if ((rc = enqueue_greedy_step(m))) return rc;
        if (out) {
            CK(g4_memcpy_d2h_async(&m->hstep[2], m->dstep + 2, 4));
            CK(g4_sync());
            out[s] = m->hstep[2];
        }
    }
    CK(g4_sync());
    if (sec) *sec = now_s() - t0;
    return trace_pull(m);
}

/* One sampled decode step as launches: forward with logits, then the device
 * sampler (repetition penalty over gen_hist, sample_token), which stores the
 * token as the next input, appends it to gen_hist and advances the position. */
static int enqueue_sampled_step(g4e_model *m, const SampleCfg *sc) {
    int rc = enqueue_step(m, 1);
    if (rc) return rc;
    CK(g4_sample(m->logits, m->c.vocab, sc->temp, sc->topp, sc->topk, sc->penalty, sc->last_n, m->gen_hist,
                 m->dstep + 3, m->c.max_seq, (unsigned long long *)(m->dstep + 4), m->sample_part, m->dstep + 2,
                 m->dstep, m->dstep + 1));
    return 0;
}

static int ensure_sgraph(g4e_model *m, const SampleCfg *sc) {
    if (m->sgraph && !memcmp(&m->sgraph_cfg, sc, sizeof *sc)) return 0;
    if (m->sgraph) {
        g4_graph_destroy(m->sgraph);
        m->sgraph = NULL;
    }
    m->dump_now = 0;
    CK(g4_graph_begin());
    int rc = enqueue_sampled_step(m, sc);
    void *g = NULL;
    const int rc2 = g4_graph_end(&g);
    if (rc) return rc;
    if (rc2) return lib_fail(rc2, "g4_graph_end");
    m->sgraph = g;
    m->sgraph_cfg = *sc;
    return 0;
}

/* generate (main.c:2335-2488) without text: prompt, then decode steps until
 * max_new tokens or eos.  sc NULL: greedy through the argmax kernel. */
static int generate_impl(g4e_model *m, const int *prompt, int n_prompt, int max_new, int *out_tokens,
                         double *prefill_sec, double *decode_sec, int use_graph, const SampleCfg *sc) {
    g4_set_stream(m->stream);
    if (m->dump_at >= 0) use_graph = 0;   /* the dump position is known on the host only */
    const double t0 = now_s();
    int gen = 0, rc;
    /* prefill: lm_mode 0 except for the last prompt token (main.c:2366-2384),
     * in prompt chunks or token by token */
    if (m->pf_chunk > 0) {
        const int np = n_prompt - 1 < m->c.max_seq ? n_prompt - 1 : m->c.max_seq;
        if (np > 0 && (rc = g4e_prefill(m, prompt, np, 0))) return -rc;
    } else {
        for (int pos = 0; pos < n_prompt - 1; pos++) {
            if (pos >= m->c.max_seq) return gen;
            if ((rc = set_step(m, prompt[pos], pos)) || (rc = enqueue_step(m, 0))) return -rc;
        }
    }
    const int last = n_prompt - 1;
    if (last >= m->c.max_seq) return gen;
    if ((rc = set_step(m, prompt[last], last))) return -rc;
    if (use_graph && (rc = sc ? ensure_sgraph(m, sc) : ensure_graph(m))) return -rc;
    if (g4_sync()) return -lib_fail(G4_ERR_HIP, "g4_sync");
    const double t1 = now_s();
    if (prefill_sec) *prefill_sec = t1 - t0;
    /* decode: each step computes the logits of the current token and the
     * sampled (or argmax) token becomes the next input (main.c:2404-2435) */
    void *graph = sc ? m->sgraph : m->graph;
    for (int pos = last; pos < n_prompt + max_new - 1 && pos < m->c.max_seq; pos++) {
        m->dump_now = m->dump_at >= 0 && pos == m->dump_at;
        if (use_graph) rc = g4_graph_launch(graph) ? lib_fail(G4_ERR_HIP, "g4_graph_launch") : 0;
        else rc = sc ? enqueue_sampled_step(m, sc) : enqueue_greedy_step(m);
        if (rc) return -rc;
        if (g4_memcpy_d2h_async(&m->hstep[2], m->dstep + 2, 4) || g4_sync()) return -lib_fail(G4_ERR_HIP, "readback");
        const int next = m->hstep[2];
        if (next == m->c.eos) break;
        out_tokens[gen++] = next;
    }
    if (decode_sec) *decode_sec = now_s() - t1;
    return gen;
}

int g4e_generate_greedy(g4e_model *m, const int *prompt, int n_prompt, int max_new, int *out_tokens,
                        double *prefill_sec, double *decode_sec, int use_graph) {
    if (!m || !prompt || n_prompt <= 0 || max_new < 0) return -fail(G4_ERR_ARG, "g4e_generate_greedy: bad arguments");
    return generate_impl(m, prompt, n_prompt, max_new, out_tokens, prefill_sec, decode_sec, use_graph, NULL);
}

int g4e_generate(g4e_model *m, const int *prompt, int n_prompt, int max_new, float temp, float topp, int topk,
                 float penalty, int penalty_last_n, uint64_t seed, int *out_tokens, double *prefill_sec,
                 double *decode_sec, int use_graph) {
    if (!m || !prompt || n_prompt <= 0 || max_new < 0) return -fail(G4_ERR_ARG, "g4e_generate: bad arguments");
    if (topk < 1 || topk > 64 || topk > m->c.vocab)
        return -fail(G4_ERR_ARG, "g4e_generate: top-k %d not in 1..64", topk);
    g4_set_stream(m->stream);
    /* rng = seed ? seed : 1 (main.c:2341); no tokens generated yet */
    const uint64_t st = seed ? seed : 1;
    int rc;
    if ((rc = g4_store_i32x2(m->dstep + 2, 0, 0)) || (rc = g4_store_i32x2(m->dstep + 4, (int)(uint32_t)st,
                                                                          (int)(uint32_t)(st >> 32))))
        return -lib_fail(rc, "g4_store_i32x2");
    const SampleCfg sc = {temp, topp, penalty, topk, penalty_last_n};
    return generate_impl(m, prompt, n_prompt, max_new, out_tokens, prefill_sec, decode_sec, use_graph, &sc);
}

int g4e_decode_steps_sampled(g4e_model *m, int token, int pos0, int steps, float temp, float topp, int topk,
                             float penalty, int penalty_last_n, uint64_t seed, int use_graph, int *out, double *sec) {
    if (!m || steps < 0) return fail(G4_ERR_ARG, "g4e_decode_steps_sampled: bad arguments");
    if (pos0 + steps > m->c.max_seq) return fail(G4_ERR_ARG, "decode past max_seq");
    if (topk < 1 || topk > 64 || topk > m->c.vocab) return fail(G4_ERR_ARG, "top-k %d not in 1..64", topk);
    g4_set_stream(m->stream);
    const uint64_t st = seed ? seed : 1;
    CK(g4_store_i32x2(m->dstep + 2, 0, 0));
    CK(g4_store_i32x2(m->dstep + 4, (int)(uint32_t)st, (int)(uint32_t)(st >> 32)));
    int rc = set_step(m, token, pos0);
    if (rc) return rc;
    m->dump_now = 0;
    const SampleCfg sc = {temp, topp, penalty, topk, penalty_last_n};
    if (use_graph && (rc = ensure_sgraph(m, &sc))) return rc;
    CK(g4_sync());
    const double t0 = now_s();
    for (int s = 0; s < steps; s++) {
        if (use_graph) CK(g4_graph_launch(m->sgraph));
        else if ((rc = enqueue_sampled_step(m, &sc))) return rc;
        if (out) {
            CK(g4_memcpy_d2h_async(&m->hstep[2], m->dstep + 2, 4));
            CK(g4_sync());
            out[s] = m->hstep[2];
        }
    }
    CK(g4_sync());
    if (sec) *sec = now_s() - t0;
    return 0;
}

/* ---- step-by-step generation (the reference's generate loop with host
 * decisions between steps: forced tokens, the thinking budget, logit dumps) */
int g4e_gen_begin(g4e_model *m, uint64_t seed) {
    if (!m) return fail(G4_ERR_ARG, "g4e_gen_begin: null model");
    g4_set_stream(m->stream);
    const uint64_t st = seed ? seed : 1;            /* rng = seed ? seed : 1 (main.c:2341) */
    CK(g4_store_i32x2(m->dstep + 2, 0, 0));
    CK(g4_store_i32x2(m->dstep + 4, (int)(uint32_t)st, (int)(uint32_t)(st >> 32)));
    m->gen_n = 0;
    return 0;
}

int g4e_gen_step(g4e_model *m, int token, int pos, float temp, float topp, int topk, float penalty, int penalty_last_n,
                 int forced, int use_graph, int *next) {
    if (!m || !next) return fail(G4_ERR_ARG, "g4e_gen_step: null pointer");
    if (topk < 1 || topk > 64 || topk > m->c.vocab) return fail(G4_ERR_ARG, "top-k %d not in 1..64", topk);
    if (forced >= m->c.vocab) return fail(G4_ERR_ARG, "forced token %d out of range", forced);
    if (m->gen_n >= m->c.max_seq) return fail(G4_ERR_STATE, "g4e_gen_step: generated-token history is full");
    g4_set_stream(m->stream);
    int rc = set_step(m, token, pos);
    if (rc) return rc;
    if (forced >= 0) {
        /* the host's token: no draw, the history takes it (main.c:2416-2427) */
        if ((rc = enqueue_step(m, 1))) return rc;
        CK(g4_memcpy_h2d(m->gen_hist + m->gen_n, &forced, 4));
        CK(g4_store_i32x2(m->dstep + 2, forced, m->gen_n + 1));
        CK(g4_sync());
        *next = forced;
        m->gen_n++;
        return trace_pull(m);
    }
    if (m->dump_now) use_graph = 0;                 /* the dump records from eager launches */
    const SampleCfg sc = {temp, topp, penalty, topk, penalty_last_n};
    if (use_graph) {
        if ((rc = ensure_sgraph(m, &sc))) return rc;
        CK(g4_graph_launch(m->sgraph));
    } else if ((rc = enqueue_sampled_step(m, &sc))) {
        return rc;
    }
    CK(g4_memcpy_d2h_async(&m->hstep[2], m->dstep + 2, 4));
    CK(g4_sync());
    *next = m->hstep[2];
    m->gen_n++;
    return trace_pull(m);
}

int g4e_kv_fingerprint(g4e_model *m, float *out, int *have) {
    if (!m || !out || !have) return fail(G4_ERR_ARG, "g4e_kv_fingerprint: null pointer");
    g4_set_stream(m->stream);
    CK(g4_sync());
    CK(g4_memcpy_d2h(out, m->dfp, (size_t)G4E_FP_TAGS * 7 * 4));
    memcpy(have, m->fp_have, sizeof m->fp_have);
    return 0;
}
