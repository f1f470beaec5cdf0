// Where a grid kernel's samples come from (points a caller hands over, or the
// rays of a training batch) and how the scatter reads their feature gradients.
#pragma once

#include "grid.hpp"
#include "sampler.hpp"

namespace nect {

// ----------------------------------------------------------- position sources

template <int D>
struct PointSource {
    const float *x;
    int64_t n;
    int64_t stride;
    // 0: no such slot, 1: live slot without a sample, 2: sample.
    __device__ __forceinline__ int get(int64_t s, float (&p)[D]) const {
        if (s >= n) return 0;
        const float *r = x + s * stride;
#pragma unroll
        for (int d = 0; d < D; ++d) p[d] = r[d];
        return 2;
    }
};

// Samples of the fused training path: slot 32*tile + j of the tile list.
template <int D>
struct RaySource {
    const NectRay *rays;
    const int32_t *tile_offsets;
    const int32_t *tile_ray;
    const int32_t *n_tiles;
    float t;  // 4th coordinate (time) for D == 4
    __device__ __forceinline__ int get(int64_t slot, float (&p)[D]) const {
        const int64_t tile = slot / kTile;
        if (tile >= n_tiles[0]) return 0;
        const int r = tile_ray[tile];
        const int i = (int)(tile - tile_offsets[r]) * kTile + (int)(slot % kTile);
        const NectRay d = rays[r];
        float q[3];
        const bool ok = ray_sample(d, i, q);
#pragma unroll
        for (int k = 0; k < D && k < 3; ++k) p[k] = q[k];
        if (D == 4) p[D - 1] = t;
        return ok ? 2 : 1;
    }
};

// dL/dfeatures as the grouped scatter reads it: rows of `stride` elements of
// `dtype` (NECT_F32, NECT_F16 or NECT_BF16), each value multiplied by *scale
// when scale is set (a 16-bit network backward's scaled gradient and the
// reciprocal of its power-of-two scale: the products are exact, so the values
// equal those of the unscaled float32 copy, which is then never written).
struct DoutView {
    const void *p;
    int64_t stride;
    int32_t dtype;
    const float *scale;
};

__device__ __forceinline__ float dout_at(const DoutView &d, float sc, int64_t i) {
    if (d.dtype == NECT_F16) return (float)static_cast<const _Float16 *>(d.p)[i] * sc;
    if (d.dtype == NECT_BF16) return to_f32(static_cast<const bf16_t *>(d.p)[i]) * sc;
    return static_cast<const float *>(d.p)[i] * sc;
}

// The grid input of a sample at (z, y, x) = q and time t under the column map.
template <int D>
__device__ __forceinline__ void place_sample(uint32_t cmap, const float (&q)[3], float t, float (&p)[D]) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const uint32_t k = ((cmap >> (2 * d)) & 3u) ^ (uint32_t)d;
        p[d] = k == 0 ? q[0] : (k == 1 ? q[1] : (k == 2 ? q[2] : t));
    }
}

}  // namespace nect
