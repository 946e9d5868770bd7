/* mia_gpu_model_prefill's one-time set-up with device allocations that fail,
 * without a GPU: the model source itself over stand-ins of the calls it
 * makes (test_prefill_setup.py compiles and runs this; what the rest of the
 * file calls stays unresolved and is not reached). Exit status 0, or the
 * number of the check that failed. */
#include "model_gpu.c"

static int mallocs, fail_at, live, attention_calls, bad_calls;

void *mhip_malloc(mhip_ctx *c, size_t bytes) {
    (void)c;
    if (++mallocs == fail_at) return NULL;
    live++;
    return malloc(bytes);
}
int mhip_free(mhip_ctx *c, void *p) {
    (void)c;
    if (p) live--;
    free(p);
    return 0;
}
const char *mhip_error(const mhip_ctx *c) {
    (void)c;
    return "stand-in";
}
int mhip_sync(mhip_ctx *c) {
    (void)c;
    return 0;
}
int mhip_dequantize_q8(mhip_ctx *c, const void *d_q, float *d_y, int n) {
    (void)c;
    (void)d_q;
    (void)n;
    bad_calls += !d_y;
    return 0;
}
size_t mhip_attention_batch_scratch_bytes(const mhip_attn_dims *s, int n, int max_seq) {
    return (size_t)s->dim * (size_t)(n + max_seq);
}
size_t mhip_attention_pack_bytes(const mhip_attn_dims *s) { return (size_t)s->dim; }
int mhip_attention_pack(mhip_ctx *c, const mhip_attn_dims *s, const void *wq, const void *wk,
                        const void *wv, const void *wo, void *pack) {
    (void)c, (void)s, (void)wq, (void)wk, (void)wv, (void)wo;
    return pack ? 0 : -1;
}
int mhip_attention_batch(mhip_ctx *c, const mhip_attn_dims *s, const float *norm, const void *wq,
                         const void *wk, const void *wv, const void *wo, const float *qn,
                         const float *kn, const double *rope, float *kc, float *vc, int pos, int n,
                         int max_seq, float *x, const void *pack, void *scratch, int flags) {
    (void)c, (void)s, (void)norm, (void)wq, (void)wk, (void)wv, (void)wo, (void)qn, (void)kn;
    (void)rope, (void)kc, (void)vc, (void)pos, (void)n, (void)max_seq, (void)pack, (void)flags;
    attention_calls++;
    bad_calls += !x || !scratch;
    return 0;
}
int mia_moe_layer_dev(mia_moe *m, int layer, float *d_x, int T, const float *d_bias) {
    (void)m, (void)layer, (void)T, (void)d_bias;
    bad_calls += !d_x;
    return 0;
}
/* (hidden symbols have to be there; not reached) */
void mia_moe_get_tensors(const mia_moe *m, mia_moe_tensors *t) { (void)m, (void)t; }
uint64_t mia_dense_walk(const mia_file_info *h, int layer, mia_layer_offsets *lo, uint64_t *embd,
                        uint64_t *onorm, uint64_t *out) {
    (void)h, (void)layer, (void)lo, (void)embd, (void)onorm, (void)out;
    return 0;
}

int main(void) {
    static mia_layer_offsets lo[2];
    const int tokens[3] = {0, 1, 2};
    /* allocation 1 is the residuals, 2 the attention scratch, 3 the pack
     * (without which the vector rows run) */
    static const int order[] = {2, 1, 3};
    for (int i = 0; i < 3; i++) {
        const int k = order[i];
        mia_gpu_model m;
        memset(&m, 0, sizeof m);
        m.info.dim = 64;
        m.info.n_layers = 2;
        m.info.n_heads = 2;
        m.info.n_kv_heads = 1;
        m.info.head_dim = 32;
        m.info.vocab = 8;
        m.info.n_active = 2;
        m.max_seq = 16;
        m.ad = (mhip_attn_dims){64, 2, 1, 32, 1e-6f};
        m.lo = lo;
        attention_calls = bad_calls = live = 0;
        for (int call = 0; call < 3; call++) {
            mallocs = 0;
            fail_at = call < 2 ? k : 0; /* two calls without memory, then one with */
            const int rc = mia_gpu_model_prefill(&m, tokens, 3, 0);
            const int want = call < 2 && k < 3 ? -1 : 0;
            if (rc != want) return 10 * k + call + 1;
            if (bad_calls) return 10 * k + call + 4;
            if (rc && attention_calls) return 10 * k + call + 7;
            if (call == 1 && k < 3 && live) return 100 + k;
        }
        if (attention_calls != (k < 3 ? 2 : 6)) return 200 + k;
    }
    return 0;
}
