/* host_runtime_check.c -- the host runtime (fastface.c) over a stand-in for
 * the device: memory is host memory, kernels do nothing, and every stream,
 * event, graph and copy call is a line on stdout.  test_host_runtime.py
 * builds it with the library's host sources and reads the lines; no GPU is
 * involved.
 *
 *   host_runtime_check <weights.ffw> <op_scales.bin> <op_scales_v2.bin> <scenario>
 *
 * A "launch" or "record" or "wait" line may be made to fail: fail_at counts
 * the calls of `fail_what` down to the one that returns an error. */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "fastface.h"
#include "fastface_kernels.h"

static const char* fail_what = "";
static int fail_at = 0;                 /* 1: the next such call fails */
static int fails(const char* what)
{
    return fail_at > 0 && !strcmp(what, fail_what) && --fail_at == 0 ? FFK_ERR_HIP : FFK_OK;
}

/* handles: small numbers, by kind */
static int n_streams, n_events, n_graphs;
static int id(const void* h) { return h ? *(const int*)h : -1; }
static void* handle(int* n) { int* h = malloc(sizeof *h); *h = (*n)++; return h; }

static void* pinned[16];
static size_t pinned_size[16];
static int n_pinned;
static int is_pinned(const void* p)
{
    for (int i = 0; i < n_pinned; i++)
        if (pinned[i] && (const char*)p >= (char*)pinned[i] && (const char*)p < (char*)pinned[i] + pinned_size[i]) return 1;
    return 0;
}
static void* pin(size_t bytes)
{
    void* p = calloc(1, bytes ? bytes : 1);
    if (n_pinned < 16) { pinned[n_pinned] = p; pinned_size[n_pinned++] = bytes; }
    return p;
}

int ffk_device_count(void) { return 1; }
void* ffk_malloc(size_t bytes) { return calloc(1, bytes ? bytes : 1); }
int ffk_free(void* p) { if (p) printf("free\n"); free(p); return 0; }
void* ffk_host_alloc(size_t bytes) { return pin(bytes); }
void* ffk_host_alloc_coherent(size_t bytes) { return pin(bytes); }
int ffk_host_free(void* p)
{
    for (int i = 0; i < n_pinned; i++) if (pinned[i] == p) pinned[i] = NULL;
    free(p);
    return 0;
}
int ffk_memcpy_h2d(void* d, const void* h, size_t n, void* s)
{
    printf("h2d %zu pinned %d stream %d\n", n, is_pinned(h), id(s));
    memcpy(d, h, n);
    return 0;
}
int ffk_memcpy_d2h(void* h, const void* d, size_t n, void* s)
{
    printf("d2h %zu pinned %d stream %d\n", n, is_pinned(h), id(s));
    memcpy(h, d, n);
    return 0;
}
int ffk_zero(void* d, size_t n, void* s) { memset(d, 0, n); return 0; }
int ffk_stream_create(void** s) { *s = handle(&n_streams); return 0; }
int ffk_stream_destroy(void* s) { free(s); return 0; }
int ffk_stream_sync(void* s) { printf("stream_sync %d\n", id(s)); return 0; }
int ffk_event_create(void** e) { *e = handle(&n_events); return 0; }
int ffk_event_destroy(void* e) { free(e); return 0; }
int ffk_event_record(void* e, void* s)
{
    const int rc = fails("record");
    printf("record %d stream %d%s\n", id(e), id(s), rc ? " FAILED" : "");
    return rc;
}
int ffk_event_sync(void* e) { printf("event_sync %d\n", id(e)); return 0; }
int ffk_stream_wait_event(void* s, void* e)
{
    const int rc = fails("wait");
    printf("wait %d stream %d%s\n", id(e), id(s), rc ? " FAILED" : "");
    return rc;
}
int ffk_graph_begin(void* s) { printf("capture %d\n", id(s)); return 0; }
int ffk_graph_end(void* s, void** g) { *g = handle(&n_graphs); return 0; }
int ffk_graph_launch(void* g, void* s)
{
    const int rc = fails("launch");
    printf("launch %d stream %d%s\n", id(g), id(s), rc ? " FAILED" : "");
    return rc;
}
int ffk_graph_destroy(void* g) { if (g) printf("graph_destroy %d\n", id(g)); free(g); return 0; }
int ffk_conv(const ffk_conv_desc* d, void* s) { return 0; }
int ffk_conv_s2_shortcut(const ffk_conv_desc* c, const ffk_conv_desc* sc, void* s) { return 1; }
int ffk_fc(const ffk_fc_desc* d, void* s) { return 0; }

static float* faces(int n) { return calloc((size_t)n * FASTFACE_INPUT_N, sizeof(float)); }

int main(int argc, char** argv)
{
    if (argc < 5) return 2;
    const char* sc = argv[4];
    setvbuf(stdout, NULL, _IOLBF, 0);
    FastFace* ff = fastface_create_with_scales(argv[1], argv[2], argv[3]);
    if (!ff) return 3;
    enum { MAX = 40 };
    float* in = faces(MAX);
    float* out = calloc(MAX * FASTFACE_OUTPUT_N, sizeof(float));
    void* mine;
    ffk_stream_create(&mine);
    printf("context %d mine %d\n", id(fastface_stream(ff)), id(mine));
#define STEP(...) do { printf("call "); printf(__VA_ARGS__); printf("\n"); } while (0)
#define DEVICE(n) do { STEP("device %d", n); printf("rc %d\n", fastface_embed_batch_device(ff, in, n, out, mine)); } while (0)
#define HOST(n) do { STEP("host %d", n); printf("rc %d\n", fastface_embed_batch(ff, in, n, out)); } while (0)
    if (!strncmp(sc, "half-fails-", 11)) {      /* <what>-<count> in the second of two split calls */
        fastface_reserve(ff, MAX);
        DEVICE(30);
        const char* dash = strrchr(sc, '-');
        static char what[16];
        snprintf(what, sizeof what, "%.*s", (int)(dash - (sc + 11)), sc + 11);
        fail_what = what;
        fail_at = atoi(dash + 1);
        DEVICE(30);
        STEP("reserve");
        printf("rc %d\n", fastface_reserve(ff, MAX + 1));
    } else if (!strcmp(sc, "sizes")) {          /* the same buffers, different batches, no wait by the caller */
        fastface_reserve(ff, MAX);
        DEVICE(8); DEVICE(8); DEVICE(5); DEVICE(36); DEVICE(37); DEVICE(37); DEVICE(8);
    } else if (!strcmp(sc, "host")) {           /* host batches around the pinned buffer's sizes */
        fastface_reserve(ff, MAX);
        HOST(1); HOST(8); HOST(2); HOST(1); HOST(8); HOST(9); HOST(1); HOST(2);
        STEP("host 7 rgb8");
        printf("rc %d\n", fastface_embed_batch_rgb8(ff, (const uint8_t*)in, 7, out));
    } else {
        fprintf(stderr, "unknown scenario %s\n", sc);
        return 2;
    }
    STEP("destroy");
    fastface_destroy(ff);
    free(in); free(out);
    return 0;
}
