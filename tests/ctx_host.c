/* A context's host memory over its calls, on the CPU (tests/test_ctx_host.py): gw_forward.c itself with the HIP runtime and the
 * kernels' launchers replaced. Device and pinned memory come from a list that gives no address out twice, so a block that is
 * freed twice, or handed to a copy after its free, is seen. Prints "ok", or the first fault. */
#include "../gwenedeg_amd/csrc/gw_forward.c"

static struct { uint8_t *p; size_t n; int live; } blk[4096];
static int nblk;

static void fault(const char *what) {
    printf("%s\n", what);
    fflush(stdout);
    _Exit(1);
}

static hipError_t take(void **p, size_t n) {
    if (nblk == 4096) fault("too many allocations");
    blk[nblk].p = calloc(n ? n : 1, 1), blk[nblk].n = n, blk[nblk].live = 1;
    *p = blk[nblk++].p;
    return hipSuccess;
}

static hipError_t give(void *p) { /* (the memory itself is kept) */
    for (int i = 0; i < nblk; i++)
        if (blk[i].p == p) {
            if (!blk[i].live) fault("freed twice");
            blk[i].live = 0;
            return hipSuccess;
        }
    fault("freed, never allocated");
    return hipSuccess;
}

static void used(const void *p, size_t n, const char *what) {
    for (int i = 0; i < nblk; i++)
        if ((const uint8_t *)p >= blk[i].p && (const uint8_t *)p + n <= blk[i].p + blk[i].n) {
            if (!blk[i].live) fault(what);
            return;
        }
    fault(what);
}

hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned int flags) { return (void)flags, take(p, n); }
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind kind, hipStream_t st) {
    (void)kind, (void)st;
    used(s, n, "a copy from memory that is not allocated");
    used(d, n, "a copy into memory that is not allocated");
    memcpy(d, s, n);
    return hipSuccess;
}
int gw_k_copy_out(float *dst, const float *src, size_t n, hipStream_t s) {
    (void)s;
    used(src, n * 4, "logits from memory that is not allocated");
    used(dst, n * 4, "logits into memory that is not allocated");
    return 0;
}

#define MUST(x) do { if ((x) != RQ_OK) fault(#x); } while (0)

int main(void) {
    GwLayer layer = { 0 };
    RqModel m = { 0 };
    m.has_weights = 1, m.dim = 256, m.hidden = 256, m.n_layers = 1, m.n_heads = 2, m.n_kv_heads = 1, m.head_dim = 128, m.vocab = 64;
    m.seq_len = 256, m.embd.type = GW_Q8_0, m.layer = &layer;
    int e, tok[8], ids[4] = { 1, 2, 3, 4 };
    float out[4 * 64];
    RqCtx *c = rq_ctx_new(&m, 4, 256, &e);
    RqSeq *s = rq_seq_new(&m, 256, RQ_KV_F16, &e);
    if (!c || !s) fault("no context or sequence");
    /* greedy steps, batches whose rows grow (the logits' staging with them), greedy steps again (the same and more) */
    MUST(gw_decode_greedy(c, s, 1, 4, tok));
    for (int rows = 1; rows <= 4; rows++) {
        RqSegment sg = { s, ids, rows, RQ_LOGITS_ALL, NULL, NULL };
        MUST(rq_forward_batch(c, &sg, 1, out, NULL));
        MUST(gw_decode_greedy(c, s, 1, rows, tok));
    }
    MUST(gw_decode_greedy(c, s, 1, 8, tok));
    rq_seq_free(s);
    rq_ctx_free(c);
    for (int i = 0; i < nblk; i++)
        if (blk[i].live) fault("not freed");
    printf("ok\n");
    return 0;
}
