/* gpu_attention where the card has no room for the workspace: gpu_hip.c with
 * a workspace that is never granted and kernel launches that only count.
 * Prints the context's error before and after the call, one a line, and the
 * launches of the two kernels. */
#include "../ornith-flight_amd/csrc/host/gpu_hip.c"

static int n_plain, n_mma;

void *orn_ws_get(gpu_context *ctx, size_t bytes)
{
    orn_set_err(ctx, ORN_ENOMEM, "workspace allocation of %zu bytes failed", bytes);
    return NULL;
}

size_t ornk_attention_mma_ws(int seq, int hd) { return (size_t)seq * hd * 4; }

int ornk_attention_mma(float *out, const float *Q, const float *K, const float *V, int seq, int hd,
                       float scale, void *ws, hipStream_t s)
{
    return ++n_mma, hipSuccess;
}

int ornk_attention(float *out, const float *Q, const float *K, const float *V, int seq, int hd,
                   float scale, hipStream_t s)
{
    return ++n_plain, hipSuccess;
}

hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return hipSuccess; }

int main(void)
{
    static gpu_context ctx;
    static float data[64 * 64];
    gpu_buffer b = {data, NULL, sizeof data, 0};
    for (int earlier = 0; earlier < 2; ++earlier) {
        ctx.err[0] = 0;
        if (earlier) orn_set_err(&ctx, ORN_EINVAL, "an earlier call's error");
        printf("%s\n", ctx.err);
        gpu_attention(&ctx, &b, &b, &b, &b, 64, 64);
        printf("%s\n", ctx.err);
    }
    printf("%d %d\n", n_plain, n_mma);
    return 0;
}
