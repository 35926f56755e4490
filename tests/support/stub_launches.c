/* Stand-ins for the kernel launchers and the HIP calls of csrc/layer.c: each
 * launcher appends its name to a log, so the route that a layer call takes can
 * be read without a device. Device memory is host memory here. */
#include "lh_internal.h"
#include "lh_layer.h"

#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

char stub_log[4096];
int stub_chained;   /* what lh_attention_chained reports */

static int record(const char *name)
{
    const size_t used = strlen(stub_log);
    snprintf(stub_log + used, sizeof stub_log - used, "%s%s", used ? " " : "", name);
    return 0;
}

static int record_kind(const char *name, int kind)
{
    char text[64];
    snprintf(text, sizeof text, "%s:%d", name, kind);
    return record(text);
}

/* The parameter lists are those of lh_internal.h; the values are not used. */
#pragma GCC diagnostic ignored "-Wunused-parameter"

int lh_launch_matvec(int kind, int lookup, const void *W, float scale, const float *x, float *y,
    const float *residual, uint32_t rows, uint32_t cols, uint32_t tokens, hipStream_t s)
{
    return record_kind("matvec", kind);
}

int lh_launch_qkv_rope(int strategy, const void *Wqkv, float sq, float sk, float sv,
    const float *gamma, const float *x, const lh_step_params *params, uint32_t count,
    float *q, float *kcache_layer, float *vcache_layer, uint32_t capacity, hipStream_t s)
{
    return record_kind("qkv_rope", strategy);
}

int lh_launch_gateup_silu(int strategy, const void *Wgate, const void *Wup, float sg, float su,
    const float *gamma, const float *x, uint32_t count, float *gated, hipStream_t s)
{
    return record_kind("gateup_silu", strategy);
}

int lh_launch_norm_tile(const float *x, const float *gamma, float *xt, uint32_t count,
    hipStream_t s)
{
    return record("norm_tile");
}

int lh_launch_attention_tiles(const float *q, const float *kcache_layer,
    const float *vcache_layer, uint32_t length, uint32_t count, uint32_t capacity, float *PM,
    float *PT, float *PA, float *xt, hipStream_t s)
{
    return record("attention_tiles");
}

int lh_launch_qkv_tile(int resident, const void *Wqkv, float sq, float sk, float sv,
    const float *xt, const lh_step_params *params, uint32_t count, float *q, float *kcache_layer,
    float *vcache_layer, uint32_t capacity, hipStream_t s)
{
    return record_kind("qkv_tile", resident);
}

int lh_launch_gateup_tile(int resident, const void *Wgate, const void *Wup, float sg, float su,
    const float *xt, uint32_t count, float *gated_xt, hipStream_t s)
{
    return record_kind("gateup_tile", resident);
}

int lh_launch_residual_tile(int resident, const void *W, float scale, uint32_t cols,
    const float *xt, uint32_t count, float *x, hipStream_t s)
{
    return record_kind("residual_tile", resident);
}

int lh_launch_head(const uint16_t *E, const float *gamma, const float *xrow, float *logits,
    uint32_t *nonfinite, hipStream_t s)
{
    return record("head");
}

int lh_launch_rmsnorm(const float *gamma, const float *x, float *out, uint32_t width,
    uint32_t tokens, hipStream_t s)
{
    return record("rmsnorm");
}

int lh_launch_attention(const float *q, const float *kcache_layer, const float *vcache_layer,
    const lh_step_params *params, uint32_t length, uint32_t count, uint32_t capacity, float *PM,
    float *PT, float *PA, unsigned long long *arrive, unsigned long long *bflags,
    unsigned long long epoch, int fault, float *out, hipStream_t s)
{
    return record("attention");
}

int lh_attention_chained(uint32_t length)
{
    return stub_chained;
}

int lh_launch_qkv_attention(int lookup, const uint8_t *Wqkv, float sq, float sk, float sv,
    const float *gamma, const float *x, const lh_step_params *params, uint32_t length, float *q,
    float *kcache_layer, float *vcache_layer, uint32_t capacity, float *PM, float *PT, float *PA,
    unsigned long long *arrive, unsigned long long *flags, unsigned long long *bflags,
    unsigned long long epoch, int fault, float *out, hipStream_t s)
{
    return record_kind("qkv_attention", lookup);
}

int lh_attention_xcd_probe(uint32_t *d_words, size_t words, int *ok, hipStream_t s)
{
    *ok = 1;
    return 0;
}

int lh_launch_attention_mfma(const float *q, const float *kcache_layer, const float *vcache_layer,
    const lh_step_params *params, uint32_t length, uint32_t count, uint32_t capacity, float *PM,
    float *PT, float *PA, float *out, uint16_t *xs, uint32_t xs_tokens, float *xs_scale,
    hipStream_t s)
{
    return record("attention_mfma");
}

int lh_launch_embed(const uint16_t *E, const lh_step_params *params, uint32_t count, float *x,
    hipStream_t s)
{
    return record("embed");
}

int lh_launch_step_embed(const uint16_t *E, const float *yarn, int32_t id, uint32_t length,
    float qfactor, lh_step_params *params, float *x, hipStream_t s)
{
    return record("step_embed");
}

int lh_launch_silu_mul(const float *gate, const float *up, float *out, size_t n, hipStream_t s)
{
    return record("silu_mul");
}

int lh_launch_rope_append(const float *q_raw, const float *k_raw, const float *v_raw,
    const lh_step_params *params, uint32_t count, float *q, float *kcache_layer,
    float *vcache_layer, uint32_t capacity, hipStream_t s)
{
    return record("rope_append");
}

int lh_layer_forward_mfma(const lh_layer_weights *w, float *d_x, float *d_keys, float *d_values,
    lh_workspace *ws, int input_split, const float *next_norm, hipStream_t s)
{
    return record("layer_mfma");
}

void lh_set_error(const char *format, ...)
{
    va_list args;
    va_start(args, format);
    vfprintf(stderr, format, args);
    va_end(args);
}

hipError_t lh_dev_malloc(void **ptr, size_t bytes)
{
    *ptr = calloc(1, bytes);
    return *ptr ? hipSuccess : hipErrorOutOfMemory;
}

hipError_t lh_host_malloc(void **ptr, size_t bytes, unsigned flags)
{
    return lh_dev_malloc(ptr, bytes);
}

void lh_dev_free(void *ptr)
{
    free(ptr);
}

void lh_host_free(void *ptr)
{
    free(ptr);
}

int lh_yarn(uint32_t position, float cosine[128], float sine[128])
{
    memset(cosine, 0, 128 * sizeof(float));
    memset(sine, 0, 128 * sizeof(float));
    return 0;
}

float lh_query_factor(uint32_t position)
{
    return 1.0f;
}

hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind)
{
    memcpy(dst, src, bytes);
    return hipSuccess;
}

hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind,
    hipStream_t s)
{
    return hipMemcpy(dst, src, bytes, kind);
}

hipError_t hipMemset(void *dst, int value, size_t bytes)
{
    memset(dst, value, bytes);
    return hipSuccess;
}

hipError_t hipStreamSynchronize(hipStream_t s)
{
    return hipSuccess;
}

hipError_t hipGetLastError(void)
{
    return hipSuccess;
}

const char *hipGetErrorString(hipError_t error)
{
    return "";
}
