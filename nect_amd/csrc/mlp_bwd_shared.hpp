// Backward pass of the fused MLP for networks whose weight gradients exceed one
// wave's registers: 16-bit weights, one output, a piecewise-linear activation and
// more hidden layers or inputs than k_mlp_backward_twin takes.
//
// As there, a wave forms each product of its tile in both operand orders, so that
// dZ and A come out with a neuron per lane and samples in the registers.  The four
// waves of a workgroup stage these operands in LDS as they are (16 bytes per lane)
// and each adds up its own blocks of dW over the four tiles: one block of every
// hidden layer, one or two of the first.  W^T is read from the staged W by LDS
// transpose reads.  Bound, as k_mlp_backward_twin, by its vector instructions and the
// one wave per SIMD that hides no latency, and by two barriers per layer.
//
// 2^21 samples, FP16 LeakyReLU, k_mlp_backward -> this kernel, ms: six layers and 76
// inputs 2.80 -> 1.51; 32 inputs and five, six, seven layers 1.08 -> 0.86, 1.63 -> 1.06,
// 3.92 -> 1.58; 128 inputs and one, two layers 1.70 -> 0.61, 1.97 -> 0.75.
#pragma once

#include "mlp_bwd_twin.hpp"

namespace nect {

// LDS image of a workgroup (byte offsets); a wave's scratch: dZ and A of a layer (1 KiB per 32 neurons x 16 samples), its
// inputs turned, dL/dz of the output as in TwinLds.
template <typename T, int H, int NQ0>
struct SharedLds {
    static constexpr int E = (int)sizeof(T);
    static constexpr int PT = 32 * NQ0;
    static constexpr int SP = PT + 16 / E, SW = kWidth + 16 / E, ST = kTile + 16 / E;
    static constexpr int w0 = 0;
    static constexpr int wh = w0 + kWidth * SP * E;
    static constexpr int wo = wh + (H - 1) * kWidth * SW * E;
    static constexpr int scratch = wo + kWidth * 4;
    static constexpr int dz = 0, in = 4096, xt = 8192;     // within a wave's scratch
    static constexpr int go = xt + PT * ST * E;
    static constexpr int per_wave = go + 2 * kTile * 4;
    static constexpr int cmap = scratch + kTwinWaves * per_wave;
    static constexpr int total = cmap + PT * 4;
};

// MFMA operand of W^T: lane l holds column c + l % 32 of rows r + 4 (l / 32) .. +3 and r + 8 + 4 (l / 32) .. +3 of M.  Of
// sixteen lanes, lane i reads four columns of row i / 4 and receives column i of the four rows.  PERM: M's columns are
// staged in the order perm64<8>.
template <typename T, bool PERM>
__device__ __forceinline__ typename Chunk<T>::type turned(const T *M, int stride, int r, int c, int lane) {
    const int i = lane & 15, g = lane >> 4, u = i & 3;
    const T *p = M + (r + 4 * (g >> 1) + i / 4) * stride + c + 16 * (g & 1) + (PERM ? 8 * (u & 1) + 4 * (u >> 1) : 4 * u);
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    using L = __attribute__((address_space(3))) i16x4;
    i16x4 v[2];
    v[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)p);
    v[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)(p + 8 * stride));
    typename Chunk<T>::type f;
    __builtin_memcpy(&f, v, sizeof(f));
    return f;
}

template <typename T, int H, int NQ0, bool RELU>
__global__ __launch_bounds__(64 * kTwinWaves, 1) void k_mlp_backward_shared(MlpArgs a) {
    using C = Chunk<T>;
    using chunk = typename C::type;
    using L = SharedLds<T, H, NQ0>;
    constexpr int V = C::V, N = 16 / V;        // chunks per 16 values
    constexpr int NT = 16 * NQ0 / V;           // chunks of a lane half's inputs, at most
    constexpr int PT = L::PT, SP = L::SP, SW = L::SW, ST = L::ST;
    extern __shared__ __align__(16) char smem[];
    T *w0 = reinterpret_cast<T *>(smem + L::w0), *wh = reinterpret_cast<T *>(smem + L::wh);
    float *wo = reinterpret_cast<float *>(smem + L::wo);
    int *cmap = reinterpret_cast<int *>(smem + L::cmap);
    const int P = a.d.n_input_padded, half = P / 2;   // half h of the lanes takes the input columns half * h ..
    {
        const T *W = static_cast<const T *>(a.w);
        for (int e = threadIdx.x; e < kWidth * PT; e += blockDim.x) {
            const int o = e / PT, c = e % PT;
            w0[o * SP + c] = c < P ? W[o * P + in_col(a, c)] : zero_of<T>();
        }
        for (int k = 1; k < H; ++k) {
            const T *Wk = W + w_off_hidden(a.d, k);
            for (int e = threadIdx.x; e < kWidth * kWidth; e += blockDim.x) {
                const int o = e >> 6, pos = e & 63;
                wh[((k - 1) * kWidth + o) * SW + pos] = Wk[o * kWidth + perm64<V>(pos)];
            }
        }
        if (threadIdx.x < kWidth) wo[threadIdx.x] = to_f32(W[w_off_out(a.d) + threadIdx.x]);
        for (int i = threadIdx.x; i < PT; i += blockDim.x) cmap[i] = i < P ? in_col(a, i) : -1;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s0 = lane & 31, h0 = lane >> 5;
    char *mine = smem + L::scratch + wave * L::per_wave;
    T *XT = reinterpret_cast<T *>(mine + L::xt);                  // [input column][sample]
    float *go_row = reinterpret_cast<float *>(mine + L::go);
    for (int i = P; i < PT; ++i)
        if (lane < ST) XT[i * ST + lane] = zero_of<T>();
    __syncthreads();

    const float loss_scale = a.loss_scale_dev ? a.loss_scale_dev[0] : a.loss_scale;
    const float out_scale = a.grad_scale / loss_scale;
    const float slope = act_pwl_slope(a.d.activation);
    // a lane's inputs as pieces of 8 bytes: rows so aligned, or planes of half a chunk or of whole chunks
    const int vpp = a.x_vpp;
    const bool pieces = vpp ? vpp == V / 2 || vpp % V == 0
                            : ((uintptr_t)a.x | (uintptr_t)(a.x_stride * sizeof(T))) % 8 == 0 && a.d.n_input % (V / 2) == 0;
    const bool padded = a.d.n_input < P;   // the last piece or pieces lie past the inputs
    const int64_t second = vpp == V / 2 ? a.x_plane : V / 2;
    int64_t xoff[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int col = h0 * half + t * V;
        xoff[t] = pieces && vpp ? (col / vpp) * a.x_plane + col % vpp : col;
    }

    // dW of the wave's blocks: of hidden layer k its rows 32 (wave / 2) .. and columns 32 (wave % 2) .., of the first layer
    // rows 32 (wave % 2) .. and columns 32 (wave / 2) .., 64 + 32 (wave / 2) ..
    f32x16 acc[H + 1];
#pragma unroll
    for (int k = 0; k <= H; ++k) acc[k] = f32x16{};
    constexpr int N0 = NQ0 > 2 ? 2 : 1;
    float dwo[2] = {0.0f, 0.0f};

    const int64_t n_tiles = tile_bound(a);
    const int64_t step = (int64_t)gridDim.x * kTwinWaves;
    const auto put = [&](int at, int p, const chunk (&v)[N]) {
#pragma unroll
        for (int c = 0; c < N; ++c)
            *reinterpret_cast<u32x4 *>(mine + at + ((2 * p + c) * 64 + lane) * 16) = __builtin_bit_cast(u32x4, v[c]);
    };
    const auto staged = [&](int t, int at, int p, int c) {
        return __builtin_bit_cast(
            chunk, *reinterpret_cast<const u32x4 *>(smem + L::scratch + t * L::per_wave + at + ((2 * p + c) * 64 + lane) * 16));
    };
    chunk x[NT];
    float dy = 0.0f;
    // rows past the end read the last one, a tile past the last one that one; their dL/dz is zero.  (Not the rows between
    // the count on the device and a.n: they may never have been written, and zero times what they hold is not zero where
    // that is not finite.)
    const auto fetch = [&](int64_t tile) {
        const int64_t row = min(min(tile, n_tiles - 1) * kTile + s0, a.n - 1);
        const T *xr = input_row<T>(a, row);
        if (pieces) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (t * V >= half) continue;
                T e[V];
                const T *x0 = xr + xoff[t], *x1 = x0 + second;
                if (!padded) {
                    __builtin_memcpy(e, __builtin_assume_aligned(x0, 8), 8);
                    __builtin_memcpy(e + V / 2, __builtin_assume_aligned(x1, 8), 8);
                } else {
                    const int left = a.d.n_input - (h0 * half + t * V);
                    uint2 v[2] = {{0, 0}, {0, 0}};
                    if (left > 0) v[0] = *reinterpret_cast<const uint2 *>(x0);
                    if (left > V / 2) v[1] = *reinterpret_cast<const uint2 *>(x1);
                    __builtin_memcpy(e, v, sizeof(e));
                }
                x[t] = C::from(e);
            }
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (t * V < half) x[t] = twin_input<T>(a, xr, h0 * half + t * V);
        }
        dy = a.dy[row * a.dy_stride];
    };
    // the waves of a workgroup stay together; one past the last tile works on dL/dz = 0
    int64_t tile = (int64_t)blockIdx.x * kTwinWaves + wave;
    if (tile - wave < n_tiles) fetch(tile);
    for (; tile - wave < n_tiles; tile += step) {
        // the LDS addresses are formed where they are used rather than hoisted across the loop
        int s = s0, h = h0;
        __asm__ volatile("" : "+v"(s), "+v"(h) : : "memory");

        // ---- forward: z1 a sample per lane, z2 a neuron per lane
        f32x16 z1[2] = {}, z2[2] = {};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (t * V >= half) break;
            const int col = h * half + t * V;
            T e[V];
            __builtin_memcpy(e, &x[t], sizeof(e));
#pragma unroll
            for (int m = 0; m < V; ++m) XT[(col + m) * ST + s] = e[m];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const chunk w = C::load(w0 + (32 * p + s) * SP + col);
                z1[p] = C::mma(w, x[t], z1[p]);
                z2[p] = C::mma(x[t], w, z2[p]);
            }
        }
        const float dy_now = dy;
        chunk a1[H > 1 ? H - 1 : 1][2][N], a2[H > 1 ? H - 1 : 1][2][N];
#pragma unroll
        for (int k = 1; k < H; ++k) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                twin_act16<T, RELU>(z1[p], slope, a1[k - 1][p]);
                twin_act16<T, RELU>(z2[p], slope, a2[k - 1][p]);
                z1[p] = f32x16{};
                z2[p] = f32x16{};
            }
            __builtin_amdgcn_sched_barrier(0);
            const T *Wk = wh + (k - 1) * kWidth * SW;
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int c = 0; c < N; ++c)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const chunk w = C::load(Wk + (32 * q + s) * SW + 32 * p + 2 * V * c + V * h);
                        z1[q] = C::mma(w, a1[k - 1][p][c], z1[q]);
                        z2[q] = C::mma(a1[k - 1][p][c], w, z2[q]);
                    }
        }

        __builtin_amdgcn_sched_barrier(0);
        // ---- output: its gradient to every sample's lane and, through LDS, to the registers of z2's samples
        float zo = 0.0f;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                z1[p][j] = twin_act<RELU>(z1[p][j], slope);   // from here on act(z): its sign is all that z is needed for
                zo = fmaf(wo[32 * p + acc_row(j, h)], z1[p][j], zo);
            }
        zo += __shfl_xor(zo, 32);
        const float go = dy_now * loss_scale * act_bwd_inline(a.d.output_activation, zo);
        const bool rv = tile < n_tiles && tile * kTile + s < a.n;
        // (the next tile's inputs, in flight during the backward products)
        if (tile - wave + step < n_tiles) fetch(tile + step);
        if (h == 0) {
            go_row[s] = rv ? go : 0.0f;
            go_row[kTile + s] = rv ? to_f32(from_f32<T>(go)) : 0.0f;
        }
        wave_lds_sync();
        __builtin_amdgcn_sched_barrier(0);
        chunk g1[2][N], g2[2][N];
        {
            const float gs = rv ? go : 0.0f;
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int c = 0; c < N; ++c) {
                    float v[V], z[V];
#pragma unroll
                    for (int m = 0; m < V; ++m) {
                        v[m] = as_float32(wo[32 * p + acc_row(V * c + m, h)] * gs);
                        z[m] = z1[p][V * c + m];
                    }
                    g1[p][c] = twin_mask<T, RELU>(v, z, slope);
                }
#pragma unroll
            for (int c = 0; c < N; ++c) {
                float go2[V], gt2[V];
#pragma unroll
                for (int m = 0; m < V; m += 4) {
                    const float *at = go_row + acc_row(V * c + m, h);
                    *reinterpret_cast<f32x4 *>(go2 + m) = *reinterpret_cast<const f32x4 *>(at);
                    *reinterpret_cast<f32x4 *>(gt2 + m) = *reinterpret_cast<const f32x4 *>(at + kTile);
                }
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const float w = wo[32 * p + s];
                    float v[V], z[V];
#pragma unroll
                    for (int m = 0; m < V; ++m) {
                        v[m] = as_float32(w * go2[m]);
                        z[m] = twin_act<RELU>(z2[p][V * c + m], slope);
                    }
                    // (the operands of a weight gradient are rounded to T, here as in the other layers)
                    const chunk az = C::pack(z);
#pragma unroll
                    for (int m = 0; m < V; ++m) dwo[p] = fmaf(gt2[m], to_f32(C::get(az, m)), dwo[p]);
                    g2[p][c] = twin_mask<T, RELU>(v, z, slope);
                }
            }
        }

        // ---- hidden layers H-1 .. 1
#pragma unroll
        for (int k = H - 1; k >= 1; --k) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                put(L::dz, p, g2[p]);
                put(L::in, p, a2[k - 1][p]);
            }
            lds_barrier();
#pragma unroll
            for (int t = 0; t < kTwinWaves; ++t)
#pragma unroll
                for (int c = 0; c < N; ++c)
                    acc[k] = C::mma(staged(t, L::dz, wave >> 1, c), staged(t, L::in, wave & 1, c), acc[k]);
            __builtin_amdgcn_sched_barrier(0);
            const T *Wk = wh + (k - 1) * kWidth * SW;
            chunk n1[2][N];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                f32x16 d1 = {}, d2 = {};
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int c = 0; c < N; ++c) {
                        const chunk w = turned<T, true>(Wk, SW, 32 * p + 16 * c, 32 * q, 32 * h + s);
                        d1 = C::mma(w, g1[p][c], d1);
                        d2 = C::mma(g1[p][c], w, d2);
                    }
                twin_mask16<T, RELU>(d1, a1[k - 1][q], slope, n1[q]);
                twin_mask16<T, RELU>(d2, a2[k - 1][q], slope, g2[q]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int c = 0; c < N; ++c) g1[q][c] = n1[q][c];
            lds_barrier();
        }

        // ---- first layer
#pragma unroll
        for (int p = 0; p < 2; ++p) put(L::dz, p, g2[p]);
        lds_barrier();
#pragma unroll
        for (int u = 0; u < N0; ++u) {
            const int q = 2 * u + (wave >> 1);
            if (q >= NQ0) continue;
#pragma unroll
            for (int t = 0; t < kTwinWaves; ++t)
#pragma unroll
                for (int c = 0; c < N; ++c) {
                    T e[V];
                    const T *xt = reinterpret_cast<const T *>(smem + L::scratch + t * L::per_wave + L::xt) +
                                  (32 * q + s) * ST + 16 * c + 4 * h;
                    __builtin_memcpy(e, __builtin_assume_aligned(xt, 8), 8);
                    __builtin_memcpy(e + 4, __builtin_assume_aligned(xt + 8, 8), 8);
                    f32x16 &sum = acc[u == 0 ? 0 : H];
                    sum = C::mma(staged(t, L::dz, wave & 1, c), C::from(e), sum);
                }
        }
        if (a.dx && tile < n_tiles) {
#pragma unroll
            for (int q = 0; q < NQ0; ++q) {
                f32x16 d = {};
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int c = 0; c < N; ++c)
                        d = C::mma(g1[p][c], turned<T, false>(w0, SP, 32 * p + 16 * c, 32 * q, 32 * h + s), d);
                // a column per lane: a store writes whole stretches of two samples' rows
                const int col = cmap[32 * q + s];
                float *dxr = a.dx + tile * kTile * a.dx_stride + col;
                if (col >= 0 && col < a.d.n_input) {
                    if ((tile + 1) * kTile <= a.n) {
#pragma unroll
                        for (int j = 0; j < 16; ++j) dxr[acc_row(j, h) * a.dx_stride] = d[j] * out_scale;
                    } else {
#pragma unroll
                        for (int j = 0; j < 16; ++j)
                            if (tile * kTile + acc_row(j, h) < a.n) dxr[acc_row(j, h) * a.dx_stride] = d[j] * out_scale;
                    }
                }
            }
        }
        lds_barrier();
    }

    // ---- the workgroup's partial weight gradients (every parameter of the slot is written once)
    float *out = a.ws + (int64_t)blockIdx.x * a.d.n_params;
#pragma unroll
    for (int k = 1; k < H; ++k) {
        float *o = out + w_off_hidden(a.d, k) + 32 * (wave >> 1) * kWidth + 32 * (wave & 1) + s0;
#pragma unroll
        for (int j = 0; j < 16; ++j) o[acc_row(j, h0) * kWidth] = acc[k][j];
    }
#pragma unroll
    for (int u = 0; u < N0; ++u) {
        const int i = 32 * (2 * u + (wave >> 1)) + s0;
        if (i >= P || i >= PT) continue;
        float *o = out + cmap[i] + 32 * (wave & 1) * P;
#pragma unroll
        for (int j = 0; j < 16; ++j) o[acc_row(j, h0) * P] = acc[u == 0 ? 0 : H][j];
    }
    float *wsum = reinterpret_cast<float *>(smem + L::scratch);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        dwo[p] += __shfl_xor(dwo[p], 32);
        if (h0 == 0) wsum[wave * kWidth + 32 * p + s0] = dwo[p];
    }
    lds_barrier();
    for (int i = threadIdx.x; i < 16 * kWidth; i += blockDim.x)
        out[w_off_out(a.d) + i] = i < kWidth ? (wsum[i] + wsum[kWidth + i]) + (wsum[2 * kWidth + i] + wsum[3 * kWidth + i])
                                             : 0.0f;   // output rows past the first: padding
}

// Whether the network takes k_mlp_backward_shared (of those that twin_suits leaves).
inline bool shared_suits(const NectMlpDesc &d, int32_t dtype) {
    return dtype != NECT_F32 && d.n_output == 1 && act_is_pwl(d.activation) && !twin_suits(d, dtype);
}

// Launchers, one per weight dtype; each returns 0 or records an error.  workgroups: rows of ws.
int32_t launch_mlp_backward_shared_f16(const MlpArgs &a, unsigned workgroups, hipStream_t st);
int32_t launch_mlp_backward_shared_bf16(const MlpArgs &a, unsigned workgroups, hipStream_t st);

template <typename T, int H, int NQ0, bool RELU>
int32_t launch_mlp_backward_shared_as(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    constexpr size_t bytes = SharedLds<T, H, NQ0>::total;
    static_assert(bytes <= kLdsLimit, "LDS image too large");
    return launch_with_lds(k_mlp_backward_shared<T, H, NQ0, RELU>, workgroups, 64 * kTwinWaves, bytes, st, a,
                           "k_mlp_backward_shared");
}

// Depths H0..H1 (the LDS limit on a network leaves at most seven layers); up to four layers only inputs of more than 64.
template <typename T, bool RELU, int H0, int H1>
int32_t launch_mlp_backward_shared(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    if constexpr (H0 <= H1) {
        if (a.d.n_hidden_layers == H0) {
            const int NQ0 = (a.d.n_input_padded + 31) / 32;
            if (NQ0 == 4) return launch_mlp_backward_shared_as<T, H0, 4, RELU>(a, workgroups, st);
            if (NQ0 == 3) return launch_mlp_backward_shared_as<T, H0, 3, RELU>(a, workgroups, st);
            if constexpr (H0 > 4) {
                if (NQ0 == 2) return launch_mlp_backward_shared_as<T, H0, 2, RELU>(a, workgroups, st);
                return launch_mlp_backward_shared_as<T, H0, 1, RELU>(a, workgroups, st);
            }
        }
        return launch_mlp_backward_shared<T, RELU, H0 + 1, H1>(a, workgroups, st);
    } else {
        set_error("k_mlp_backward_shared: no instantiation for this network");
        return 1;
    }
}

}  // namespace nect
