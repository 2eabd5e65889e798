// A row's LayerNorm statistics from its 64-column chunks'.
#pragma once

#include <hip/hip_runtime.h>

namespace raya {

// From the chunks' (c, r = sum (x - c), s = sum (x - c)^2), in f64 as ops::layer_norm keeps its
// statistics (crates/raya-core/src/ops.rs:51-74): a chunk's mean is c + r / 64 and its sum of
// squared deviations s - r^2 / 64; the chunks combine as Chan et al.'s pairwise update.
// Returns (mean_hi, mean_lo, 1 / sqrt(var + eps), 0) with var the biased variance and
// mean_hi + mean_lo the f64 mean to 48 bits.
__device__ __forceinline__ float4 row_norm(const float4 *st, int chunks, float eps) {
    double mean = 0.0;
    for (int c = 0; c < chunks; ++c) mean += (double)st[c].x + (double)st[c].y * (1.0 / 64.0);
    mean /= chunks;
    double m2 = 0.0;
    for (int c = 0; c < chunks; ++c) {
        const double r = st[c].y, cm = (double)st[c].x + r * (1.0 / 64.0);
        const double dm = cm - mean;
        m2 += ((double)st[c].z - r * r * (1.0 / 64.0)) + 64.0 * dm * dm;
    }
    const double var = fmax(m2, 0.0) / (64.0 * chunks);
    const float hi = (float)mean;
    return make_float4(hi, (float)(mean - (double)hi), (float)(1.0 / sqrt(var + (double)eps)), 0.0f);
}

}  // namespace raya
