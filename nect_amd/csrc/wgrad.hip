// Weight gradient of a wide network layer: dW[i][j] += scale * sum_k dZ[k][i] * H[k][j]
// over the samples k -- a GEMM whose output is small (at most a few hundred rows
// and columns) and whose reduction runs over millions of samples.  Library GEMMs
// parallelise such shapes over the output and leave most of the device idle;
// here the samples are split: each workgroup reduces one chunk of samples for
// one 128 x 128 output tile on MFMA and adds its partial tile to dW with float
// atomics (16 consecutive floats of a row per 64-byte request).
//
// Reading both operands once bounds it: 2.5 M samples of 128 x 128, 1.28 GB, in 227 us.  The operands are staged in LDS as
// they lie in memory, by 16-byte loads, and turned by the LDS reads (ds_read_b64_tr_b16); two workgroups per CU take one
// chunk each, since every chunk costs a tile of atomics.  Before, 2-byte loads turned the operands on the way into LDS, in
// 4096 chunks: 390 us; 300000 samples of 128 x 128 94 -> 50 us, of 128 x 384 297 -> 91.
#include <algorithm>

#include "mlp_bwd.hpp"

namespace nect {

constexpr int kWgTile = 128;                 // output tile (rows and columns)
constexpr int kWgSteps = 32;                 // samples staged per step
constexpr int kWgPitch = kWgTile + 32;       // LDS row (elements): four rows of 32 columns on different banks
// Chunks over the device: two workgroups per CU (1024 chunks, four per CU: 240 us, and 71 with 300000 samples)
constexpr int64_t kWgGroups = 512;
constexpr int kWgLoads = kWgSteps * kWgTile / 8 / 256;   // 16-byte pieces of a stage per thread

typedef short i16x4 __attribute__((ext_vector_type(4)));

// A step's 32 samples of the tile's columns (zero outside the matrix) as they lie in memory: thread t takes the columns
// 8 (t % 16) .. +7 of samples t / 16 and t / 16 + 16.  p: its first piece; left: samples of the chunk from that row on;
// cols: columns of the matrix from that one on.  VEC: rows are 16-byte aligned.  The loads (wg_load) and the LDS stores
// (wg_store) are separate so that the next step's loads are in flight while this one's products run.
template <typename T, bool VEC>
__device__ __forceinline__ void wg_load(uint4 (&r)[kWgLoads], const T *__restrict__ p, int64_t ldx, int left, int cols) {
#pragma unroll
    for (int u = 0; u < kWgLoads; ++u) {
        r[u] = uint4{0, 0, 0, 0};
        if (16 * u >= left) continue;
        const T *q = p + 16 * u * ldx;
        if (VEC && cols >= 8) {
            r[u] = *reinterpret_cast<const uint4 *>(q);
        } else if (cols > 0) {
            T e[8];
#pragma unroll
            for (int m = 0; m < 8; ++m) e[m] = m < cols ? q[m] : zero_of<T>();
            __builtin_memcpy(&r[u], e, sizeof(uint4));
        }
    }
}

template <typename T>
__device__ __forceinline__ void wg_store(T *lds, const uint4 (&r)[kWgLoads]) {
#pragma unroll
    for (int u = 0; u < kWgLoads; ++u)
        *reinterpret_cast<uint4 *>(lds + (threadIdx.x / 16 + 16 * u) * kWgPitch + 8 * (threadIdx.x % 16)) = r[u];
}

// MFMA operand of columns c .. c+31 and samples k .. k+15 of a stage: lane l holds column c + l % 32 and eight of the
// samples, four from k + 4 (l / 32) and four from k + 8 + 4 (l / 32) (the other operand holds the same).  The LDS read
// turns them: of sixteen lanes, lane i reads columns 4 (i % 4) .. +3 of row i / 4 and receives column i of the four rows.
template <typename T>
__device__ __forceinline__ typename MF<T>::frag wg_frag(const T *lds, int k, int c, int lane) {
    const int i = lane & 15, g = lane >> 4;
    const T *p = lds + (k + 4 * (g >> 1) + i / 4) * kWgPitch + c + 16 * (g & 1) + 4 * (i % 4);
    using L = __attribute__((address_space(3))) i16x4;
    i16x4 v[2];
    v[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)p);
    v[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)(p + 8 * kWgPitch));
    typename MF<T>::frag f;
    __builtin_memcpy(&f, v, sizeof(f));
    return f;
}

template <typename T, bool VEC>
__global__ __launch_bounds__(256, 2) void k_wgrad(const T *__restrict__ A, int64_t lda, const T *__restrict__ B,
                                               int64_t ldb, int64_t K, int m, int n, int64_t chunk, float scale,
                                               float *__restrict__ C, int64_t ldc) {
    __shared__ __align__(16) T stage[2][2][kWgSteps * kWgPitch];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int s = lane & 31, h = lane >> 5;
    const int wm = wave >> 1, wn = wave & 1;  // the wave's 64 x 64 quarter of the tile
    const int i0 = blockIdx.y * kWgTile, j0 = blockIdx.z * kWgTile;
    const int64_t kb = (int64_t)blockIdx.x * chunk;
    const int64_t ke = kb + chunk < K ? kb + chunk : K;
    f32x16 acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[p][q] = f32x16{};
    const int tr = threadIdx.x / 16, tc = 8 * (threadIdx.x % 16);
    const T *pa = A + (kb + tr) * lda + i0 + tc, *pb = B + (kb + tr) * ldb + j0 + tc;
    const int ca = m - i0 - tc, cb = n - j0 - tc;
    int left = (int)(ke - kb);
    uint4 ra[kWgLoads], rb[kWgLoads];
    wg_load<T, VEC>(ra, pa, lda, left - tr, ca);
    wg_load<T, VEC>(rb, pb, ldb, left - tr, cb);
    for (int buf = 0; left > 0; left -= kWgSteps, buf ^= 1) {
        T *TA = stage[buf][0], *TB = stage[buf][1];
        wg_store<T>(TA, ra);
        wg_store<T>(TB, rb);
        // one barrier per step: the buffer written next was read before this one
        __syncthreads();
        pa += kWgSteps * lda;
        pb += kWgSteps * ldb;
        wg_load<T, VEC>(ra, pa, lda, left - kWgSteps - tr, ca);
        wg_load<T, VEC>(rb, pb, ldb, left - kWgSteps - tr, cb);
#pragma unroll
        for (int kk = 0; kk < kWgSteps; kk += 16) {
            typename MF<T>::frag fa[2], fb[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                fa[p] = wg_frag<T>(TA, kk, 64 * wm + 32 * p, lane);
                fb[p] = wg_frag<T>(TB, kk, 64 * wn + 32 * p, lane);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q) acc[p][q] = MF<T>::mma(fa[p], fb[q], acc[p][q]);
        }
    }
    // accumulator register j of lane (s, h): row acc_row(j, h), column s of its 32 x 32 block
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int col = j0 + 64 * wn + 32 * q + s;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int row = i0 + 64 * wm + 32 * p + acc_row(j, h);
                if (row < m && col < n) unsafeAtomicAdd(C + (int64_t)row * ldc + col, scale * acc[p][q][j]);
            }
        }
}

template <typename T>
static void launch_wgrad(dim3 grid, hipStream_t st, const void *dz, int64_t ld_dz, const void *h, int64_t ld_h, int64_t K,
                         int m, int n, int64_t chunk, float scale, float *dw, int64_t ld_dw) {
    const bool vec = (uintptr_t)dz % 16 == 0 && (uintptr_t)h % 16 == 0 && ld_dz % 8 == 0 && ld_h % 8 == 0;
    if (vec)
        hipLaunchKernelGGL((k_wgrad<T, true>), grid, dim3(256), 0, st, (const T *)dz, ld_dz, (const T *)h, ld_h, K, m, n,
                           chunk, scale, dw, ld_dw);
    else
        hipLaunchKernelGGL((k_wgrad<T, false>), grid, dim3(256), 0, st, (const T *)dz, ld_dz, (const T *)h, ld_h, K, m, n,
                           chunk, scale, dw, ld_dw);
}

}  // namespace nect

using namespace nect;

extern "C" int32_t nect_wgrad(int32_t dtype, const void *dz, int64_t ld_dz, const void *h, int64_t ld_h,
                              int64_t n_samples, int32_t n_out, int32_t n_in, float scale, float *dw, int64_t ld_dw,
                              void *stream) {
    clear_error();
    NECT_REQUIRE(dtype == NECT_F16 || dtype == NECT_BF16, "dtype must be NECT_F16 or NECT_BF16");
    NECT_REQUIRE(n_samples >= 0 && n_out >= 1 && n_in >= 1, "bad sizes");
    NECT_REQUIRE(ld_dz >= n_out && ld_h >= n_in && ld_dw >= n_in, "leading dimensions smaller than the rows");
    if (n_samples == 0) return 0;
    NECT_REQUIRE(dz && h && dw, "NULL pointer");
    const int64_t mt = (n_out + kWgTile - 1) / kWgTile, nt = (n_in + kWgTile - 1) / kWgTile;
    NECT_REQUIRE(mt <= 65535 && nt <= 65535, "output too large");
    // about kWgGroups workgroups over the device, at least 256 samples each, whole steps
    int64_t chunk = (n_samples * mt * nt + kWgGroups - 1) / kWgGroups;
    chunk = std::clamp<int64_t>((chunk + kWgSteps - 1) / kWgSteps * kWgSteps, 256, (int64_t)1 << 30);
    const int64_t chunks = (n_samples + chunk - 1) / chunk;
    NECT_REQUIRE(chunks < ((int64_t)1 << 31), "too many samples");
    const dim3 grid((unsigned)chunks, (unsigned)mt, (unsigned)nt);
    const hipStream_t st = as_stream(stream);
    if (dtype == NECT_F16)
        launch_wgrad<_Float16>(grid, st, dz, ld_dz, h, ld_h, n_samples, n_out, n_in, chunk, scale, dw, ld_dw);
    else
        launch_wgrad<bf16_t>(grid, st, dz, ld_dz, h, ld_h, n_samples, n_out, n_in, chunk, scale, dw, ld_dw);
    return check_launch("k_wgrad");
}
