// Prefill GEMMs (batches above 8): which kernel takes a batch.
#include "formats.h"
#include "kernels.h"

namespace fy {

// Both kernels split the activations into fp16 pieces (pieces.h), of the
// batch rounded up to 64 tokens. Q6_K's workspace keeps the size of int8
// digits, 136 bytes per 32 columns of the batch rounded up to 32 tokens: its
// pieces take 4 cols + cols / 8 + 4 of the 4.25 cols bytes per token.
size_t prefill_workspace(unsigned type, int cols, int batch)
{
    if (type != Q6_K) return prefill_f16_workspace(cols, batch);
    const size_t np = ((size_t)batch + 31) / 32 * 32;
    return (size_t)(cols / 32) * 136 * np;
}

const char *prefill_kernel(unsigned type) { return type == Q6_K ? "prefill_mfma" : "prefill_f16"; }

hipError_t launch_prefill(unsigned type, const uint8_t *w, const float *x, float *y, int rows, int cols, int batch,
    int whole, void *workspace, hipStream_t s)
{
    const int pad = type == Q6_K ? 32 : 64, np = (int)(((long)batch + pad - 1) / pad * pad);
    if (prefill_tile_supported(type, rows, cols, whole))
        return launch_prefill_tile(type, w, x, y, rows, cols, batch, whole, workspace, np, s);
    return launch_prefill_f16(type, w, x, y, rows, cols, batch, whole, workspace, s);
}

}  // namespace fy
