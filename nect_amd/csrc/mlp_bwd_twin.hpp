// Backward pass of the fused MLP whose weight gradients stay in the registers of
// one wave: networks with one output, a piecewise-linear hidden activation, up to
// 64 inputs and four hidden layers (float32: three).
//
// A weight gradient dW = dZ^T A sums over the samples, so both operands need the
// samples along K, while the layer products leave the samples on the lanes:
// k_mlp_backward turns every layer's dZ and A in LDS, one 16-bit store per value,
// with two barriers per layer.  Here a wave forms each layer product twice, with
// its operands in either order: the accumulators of W A^T hold a sample per lane
// and neurons in their registers (the next layer's operand), those of A W^T a
// neuron per lane and samples in their registers -- the operands of dW, with no
// turning, no barrier and no other wave.  The weight fragments are read from LDS
// once for both.  The doubled products are cheap where the matrix cores were
// mostly idle (9 % busy with two hidden layers in 16-bit, 20 % in float32); what
// bound k_mlp_backward there were 1547 vector instructions per tile of 32 samples
// (41 % busy) and waits (45 %), in float32 two waves per CU.  What bounds this
// kernel: the vector instructions, about 1000 per tile, and with them the chain of
// products of the one or two waves per SIMD that its accumulators leave room for.
//
// 2^21 samples, k_mlp_backward -> this kernel, ms: 32 inputs, FP16, ReLU, 1, 2, 3 and
// 4 hidden layers 0.36 -> 0.14, 0.40 -> 0.31, 0.81 -> 0.39, 0.94 -> 0.68 (LeakyReLU
// 0.18, 0.35, 0.44, 0.79); 64 inputs 0.67 -> 0.24, 0.86 -> 0.39, 1.21 -> 0.53,
// 1.33 -> 1.18; FP32, 32 inputs, 1 to 3 layers 1.56 -> 0.39, 2.44 -> 1.02,
// 3.38 -> 1.87.  (With five layers the accumulators exceed the register file; four
// spill some already.  Beyond: k_mlp_backward_shared.)
#pragma once

#include "mlp_bwd.hpp"

namespace nect {

// Chunk: 16 bytes of K values of one lane, one MFMA of 16-bit operands or four of
// float32.  The weight columns are staged in its order (perm64<V>).
template <typename T>
struct Chunk {
    static constexpr int V = 8;
    using type = typename MF<T>::frag;
    __device__ static __forceinline__ f32x16 mma(const type &a, const type &b, f32x16 c) { return MF<T>::mma(a, b, c); }
    __device__ static __forceinline__ type load(const T *p) { return MF<T>::load(p); }
    __device__ static __forceinline__ type pack(const float *v) { return MF<T>::pack(v); }
    __device__ static __forceinline__ T get(const type &c, int m) {
        T e[V];
        __builtin_memcpy(e, &c, sizeof(e));
        return e[m];
    }
    __device__ static __forceinline__ type from(const T *e) {
        type f;
        __builtin_memcpy(&f, e, sizeof(f));
        return f;
    }
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <>
struct Chunk<float> {
    static constexpr int V = 4;
    using type = f32x4;
    __device__ static __forceinline__ f32x16 mma(const type &a, const type &b, f32x16 c) {
#pragma unroll
        for (int m = 0; m < 4; ++m) c = MF<float>::mma(a[m], b[m], c);
        return c;
    }
    __device__ static __forceinline__ type load(const float *p) { return *reinterpret_cast<const type *>(p); }
    __device__ static __forceinline__ type pack(const float *v) { return type{v[0], v[1], v[2], v[3]}; }
    __device__ static __forceinline__ float get(const type &c, int m) { return c[m]; }
    __device__ static __forceinline__ type from(const float *e) { return pack(e); }
};

// V input elements of a row in general: p is the row's first element (of plane 0), zero past n_input.
template <typename T>
__device__ __forceinline__ typename Chunk<T>::type twin_input(const MlpArgs &a, const T *p, int col) {
    constexpr int V = Chunk<T>::V;
    T e[V];
    __asm__ volatile("" : "+v"(col));   // the elements' offsets are formed here, not kept across the caller's loop
#pragma unroll
    for (int m = 0; m < V; ++m) {
        const int i = col + m;
        e[m] = zero_of<T>();
        if (i < a.d.n_input) e[m] = p[a.x_vpp ? (i / a.x_vpp) * a.x_plane + i % a.x_vpp : i];
    }
    return Chunk<T>::from(e);
}

constexpr int kTwinWaves = 4;   // per workgroup

// Hidden weight-gradient blocks of a network (the output layer's gradient takes two registers).
__host__ __device__ constexpr int twin_blocks(int H, int NQ0) { return 4 * (H - 1) + 2 * NQ0; }

// act(z) of a piecewise-linear activation.
template <bool RELU>
__device__ __forceinline__ float twin_act(float z, float slope) {
    if constexpr (RELU) return __builtin_amdgcn_fmed3f(z, 0.0f, __builtin_inff());   // NaN: 0
    else return fmaxf(z, slope * z);   // 0 < slope <= 1
}

// 16 accumulator values as chunks, through the activation.
template <typename T, bool RELU>
__device__ __forceinline__ void twin_act16(const f32x16 &z, float slope, typename Chunk<T>::type (&o)[16 / Chunk<T>::V]) {
    constexpr int V = Chunk<T>::V;
#pragma unroll
    for (int c = 0; c < 16 / V; ++c) {
        float v[V];
#pragma unroll
        for (int m = 0; m < V; ++m) v[m] = twin_act<RELU>(z[V * c + m], slope);
        o[c] = Chunk<T>::pack(v);
    }
}

// A product as rounded to float32: its conversion to float16 is not folded into it (v_fma_mixlo_f16 rounds once).
__device__ __forceinline__ float as_float32(float v) {
    __asm__("" : "+v"(v));
    return v;
}

// v where the signed 16-bit halves of `a` are positive, else slope * v (RELU: 0), as a chunk of 16-bit values.  Whole
// halves of packed results are chosen: 0 - a, saturated, is negative where a > 0, and v_perm_b32 spreads its sign over
// the half -- no comparison per value, and half the registers of one.
template <typename T, bool RELU>
__device__ __forceinline__ typename Chunk<T>::type twin_choose(const float (&v)[8], const u32x4 &a, float slope) {
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    const u32x4 g = __builtin_bit_cast(u32x4, Chunk<T>::pack(v));
    u32x4 below = {0, 0, 0, 0};
    if constexpr (!RELU) {
        float b[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) b[m] = as_float32(v[m] * slope);
        below = __builtin_bit_cast(u32x4, Chunk<T>::pack(b));
    }
    u32x4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const i16x2 zero = {0, 0};
        const uint32_t word = a[k];   // (a bit cast of a vector's element itself takes element 0)
        const i16x2 minus = __builtin_elementwise_sub_sat(zero, __builtin_bit_cast(i16x2, word));
        const uint32_t m = __builtin_bit_cast(uint32_t, minus);
        const uint32_t on = __builtin_amdgcn_perm(m, m, 0x09090808u);
        r[k] = (g[k] & on) | (below[k] & ~on);
    }
    return __builtin_bit_cast(typename Chunk<T>::type, r);
}

// v * act'(z) as a chunk, from V values act(z).
template <typename T, bool RELU>
__device__ __forceinline__ typename Chunk<T>::type twin_mask(float (&v)[Chunk<T>::V], const float (&z)[Chunk<T>::V],
                                                             float slope) {
    constexpr int V = Chunk<T>::V;
    if constexpr (V == 8) {
        u32x4 top;   // the upper halves of the float32 values: their signs, and not zero from 2^-133 on
#pragma unroll
        for (int k = 0; k < 4; ++k) top[k] = __builtin_amdgcn_perm(__float_as_uint(z[2 * k + 1]), __float_as_uint(z[2 * k]), 0x07060302u);
        return twin_choose<T, RELU>(v, top, slope);
    } else {
#pragma unroll
        for (int m = 0; m < V; ++m) v[m] = z[m] > 0.0f ? v[m] : (RELU ? 0.0f : slope * v[m]);
        return Chunk<T>::pack(v);
    }
}

// d * act'(z) as chunks, the sign of z read from act(z) (the activation is increasing and act(0) = 0).
template <typename T, bool RELU>
__device__ __forceinline__ void twin_mask16(const f32x16 &d, const typename Chunk<T>::type (&act)[16 / Chunk<T>::V],
                                            float slope, typename Chunk<T>::type (&o)[16 / Chunk<T>::V]) {
    constexpr int V = Chunk<T>::V;
#pragma unroll
    for (int c = 0; c < 16 / V; ++c) {
        float v[V];
#pragma unroll
        for (int m = 0; m < V; ++m) v[m] = d[V * c + m];
        if constexpr (V == 8) {
            o[c] = twin_choose<T, RELU>(v, __builtin_bit_cast(u32x4, act[c]), slope);
        } else {
            float z[V];
#pragma unroll
            for (int m = 0; m < V; ++m) z[m] = act[c][m];
            o[c] = twin_mask<T, RELU>(v, z, slope);
        }
    }
}

// LDS image of a workgroup (byte offsets): the weights, rows padded by 16 bytes and W0 to whole blocks of 32 inputs; per
// wave its inputs turned (PT rows of 32 samples) and dL/dz of the output (float32, and rounded to T); and the row-layout
// column of each input.  The parameter gradient is summed over the waves in place of what precedes the columns.
template <typename T, int H, int NQ0>
struct TwinLds {
    static constexpr int E = (int)sizeof(T);
    static constexpr int PT = 32 * NQ0;
    static constexpr int SP = PT + 16 / E, SW = kWidth + 16 / E, ST = kTile + 16 / E;
    static constexpr int w0 = 0;
    static constexpr int wh = w0 + kWidth * SP * E;
    static constexpr int w0t = wh + (H - 1) * kWidth * SW * E;
    static constexpr int wht = w0t + PT * SW * E;
    static constexpr int wo = wht + (H - 1) * kWidth * SW * E;
    static constexpr int scratch = wo + kWidth * 4;
    static constexpr int go = PT * ST * E;                 // within a wave's scratch
    static constexpr int per_wave = go + 2 * kTile * 4;
    static constexpr int end = scratch + kTwinWaves * per_wave;
    static constexpr int grads = 4 * (kWidth * PT + (H - 1) * kWidth * kWidth + 16 * kWidth);
    static constexpr int cmap = end > grads ? end : grads;
    static constexpr int total = cmap + PT * 4;
};

// Whether the network takes k_mlp_backward_twin.
inline bool twin_suits(const NectMlpDesc &d, int32_t dtype) {
    const int H = d.n_hidden_layers, NQ0 = (d.n_input_padded + 31) / 32;
    return d.n_output == 1 && act_is_pwl(d.activation) && NQ0 <= 2 && H <= (dtype == NECT_F32 ? 3 : 4);
}

// Waves per SIMD (workgroups per CU): the accumulators of two hidden layers and 32 inputs leave room for two with a ReLU
// (0.31 ms; with one 0.33), of one layer with the others, whose slope costs registers (two layers 0.42; one wave 0.34);
// with 64 inputs and two layers two waves would spill (0.63 ms; one 0.38).
__host__ __device__ constexpr int twin_per_simd(int elem_bytes, int H, int NQ0, bool relu) {
    return elem_bytes == 2 && twin_blocks(H, NQ0) <= (relu ? 6 : 4) ? 2 : 1;
}
inline int twin_per_simd(int elem_bytes, const NectMlpDesc &d) {
    return twin_per_simd(elem_bytes, d.n_hidden_layers, (d.n_input_padded + 31) / 32, d.activation == NECT_ACT_RELU);
}

// NP: the padded inputs in sixteens.
template <typename T, int H, int NP, bool RELU>
__global__ __launch_bounds__(64 * kTwinWaves, twin_per_simd((int)sizeof(T), H, (NP + 1) / 2, RELU)) void k_mlp_backward_twin(MlpArgs a) {
    using C = Chunk<T>;
    using chunk = typename C::type;
    constexpr int NQ0 = (NP + 1) / 2, P = 16 * NP;
    using L = TwinLds<T, H, NQ0>;
    constexpr int V = C::V, N = 16 / V;        // chunks per 16 values
    constexpr int half = 8 * NP;               // inputs of a lane half: half h takes columns half * h ..
    constexpr int NT = half / V;
    constexpr int PT = L::PT, SP = L::SP, SW = L::SW, ST = L::ST;
    extern __shared__ __align__(16) char smem[];
    T *w0 = reinterpret_cast<T *>(smem + L::w0), *wh = reinterpret_cast<T *>(smem + L::wh);
    T *w0t = reinterpret_cast<T *>(smem + L::w0t), *wht = reinterpret_cast<T *>(smem + L::wht);
    float *wo = reinterpret_cast<float *>(smem + L::wo);
    int *cmap = reinterpret_cast<int *>(smem + L::cmap);
    {
        const T *W = static_cast<const T *>(a.w);
        for (int e = threadIdx.x; e < kWidth * PT; e += blockDim.x) {
            const int o = e / PT, c = e % PT;
            w0[o * SP + c] = c < P ? W[o * P + in_col(a, c)] : zero_of<T>();
        }
        for (int e = threadIdx.x; e < PT * kWidth; e += blockDim.x) {
            const int i = e >> 6, pos = e & 63;
            w0t[i * SW + pos] = i < P ? W[perm64<V>(pos) * P + in_col(a, i)] : zero_of<T>();
        }
        for (int k = 1; k < H; ++k) {
            const T *Wk = W + w_off_hidden(a.d, k);
            for (int e = threadIdx.x; e < kWidth * kWidth; e += blockDim.x) {
                const int o = e >> 6, pos = e & 63;
                wh[((k - 1) * kWidth + o) * SW + pos] = Wk[o * kWidth + perm64<V>(pos)];
                wht[((k - 1) * kWidth + o) * SW + pos] = Wk[perm64<V>(pos) * kWidth + o];
            }
        }
        if (threadIdx.x < kWidth) wo[threadIdx.x] = to_f32(W[w_off_out(a.d) + threadIdx.x]);
        for (int i = threadIdx.x; i < PT; i += blockDim.x) cmap[i] = i < P ? in_col(a, i) : -1;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s0 = lane & 31, h0 = lane >> 5;
    char *mine = smem + L::scratch + wave * L::per_wave;
    T *XT = reinterpret_cast<T *>(mine);                    // [input column][sample]
    float *go_row = reinterpret_cast<float *>(mine + L::go);
    for (int i = P; i < PT; ++i)
        if (lane < ST) XT[i * ST + lane] = zero_of<T>();
    __syncthreads();

    const float loss_scale = a.loss_scale_dev ? a.loss_scale_dev[0] : a.loss_scale;
    const float out_scale = a.grad_scale / loss_scale;
    const float slope = act_pwl_slope(a.d.activation);
    // a lane's inputs as pieces of 8 bytes: whole rows, or planes of half a chunk or of whole chunks
    const int vpp = a.x_vpp;
    const bool pieces = (vpp ? vpp == V / 2 || vpp % V == 0 : a.x_vec && a.d.n_input == P);
    const int64_t second = vpp == V / 2 ? a.x_plane : V / 2;
    int64_t xoff[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int col = h0 * half + t * V;
        xoff[t] = pieces && vpp ? (col / vpp) * a.x_plane + col % vpp : col;
    }

    f32x16 acc[H][2][2];       // [layer][p][q], layer 0: q < NQ0
#pragma unroll
    for (int k = 0; k < H; ++k)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q) acc[k][p][q] = f32x16{};
    float dwo[2] = {0.0f, 0.0f};

    const int64_t n_tiles = tile_bound(a);
    const int64_t step = (int64_t)gridDim.x * kTwinWaves;
    chunk x[NT];
    float dy = 0.0f;
    // rows past the end read the last one; their dL/dz is zero
    const auto fetch = [&](int64_t tile) {
        const int64_t row = min(tile * kTile + s0, a.n - 1);
        const T *xr = input_row<T>(a, row);
        if (pieces) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                T e[V];
                __builtin_memcpy(e, __builtin_assume_aligned(xr + xoff[t], 8), 8);
                __builtin_memcpy(e + V / 2, __builtin_assume_aligned(xr + xoff[t] + second, 8), 8);
                x[t] = C::from(e);
            }
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) x[t] = twin_input<T>(a, xr, h0 * half + t * V);
        }
        dy = a.dy[row * a.dy_stride];
    };
    int64_t tile = (int64_t)blockIdx.x * kTwinWaves + wave;
    if (tile < n_tiles) fetch(tile);
    for (; tile < n_tiles; tile += step) {
        // the LDS addresses are formed where they are used rather than hoisted across the loop
        int s = s0, h = h0;
        __asm__ volatile("" : "+v"(s), "+v"(h) : : "memory");

        // ---- forward: z1 a sample per lane, z2 a neuron per lane
        f32x16 z1[2] = {}, z2[2] = {};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
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
        const bool rv = tile * kTile + s < a.n;
        // (the next tile's inputs, in flight during the backward products)
        if (tile + step < n_tiles) fetch(tile + step);
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
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int c = 0; c < N; ++c) acc[k][p][q] = C::mma(g2[p][c], a2[k - 1][q][c], acc[k][p][q]);
            __builtin_amdgcn_sched_barrier(0);
            const T *WT = wht + (k - 1) * kWidth * SW;
            chunk n1[2][N];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                f32x16 d1 = {}, d2 = {};
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int c = 0; c < N; ++c) {
                        const chunk w = C::load(WT + (32 * q + s) * SW + 32 * p + 2 * V * c + V * h);
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
        }

        __builtin_amdgcn_sched_barrier(0);
        // ---- first layer
#pragma unroll
        for (int q = 0; q < NQ0; ++q) {
#pragma unroll
            for (int c = 0; c < N; ++c) {
                T e[V];
                const T *xt = XT + (32 * q + s) * ST + (V == 8 ? 16 * c : 8 * c) + 4 * h;
                // chunk c of lane half h: samples R(V c .. V c + V - 1, h), four in a row
                __builtin_memcpy(e, __builtin_assume_aligned(xt, 4 * sizeof(T)), 4 * sizeof(T));
                if constexpr (V == 8) __builtin_memcpy(e + 4, __builtin_assume_aligned(xt + 8, 4 * sizeof(T)), 4 * sizeof(T));
                const chunk xc = C::from(e);
#pragma unroll
                for (int p = 0; p < 2; ++p) acc[0][p][q] = C::mma(g2[p][c], xc, acc[0][p][q]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (a.dx) {
#pragma unroll
            for (int q = 0; q < NQ0; ++q) {
                f32x16 d = {};
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int c = 0; c < N; ++c)
                        d = C::mma(g1[p][c], C::load(w0t + (32 * q + s) * SW + 32 * p + 2 * V * c + V * h), d);
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
    }

    // ---- the workgroup's partial weight gradients: its waves' sums in LDS, in a fixed order, then one slot
#pragma unroll
    for (int p = 0; p < 2; ++p) dwo[p] += __shfl_xor(dwo[p], 32);
    __syncthreads();
    float *sum = reinterpret_cast<float *>(smem);
    const int off_out = (int)w_off_out(a.d);
    // in turn t, wave w adds its accumulators of every fourth block, from block (w + t) % 4 on
    for (int turn = 0; turn < kTwinWaves; ++turn) {
        const int part = (wave + turn) % kTwinWaves;
        const bool first = turn == 0;
#pragma unroll
        for (int k = 0; k < H; ++k)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < (k == 0 ? NQ0 : 2); ++q) {
                    if ((4 * k + 2 * p + q) % kTwinWaves != part) continue;
                    const int i = 32 * q + s0;
                    if (k == 0 && i >= P) continue;
                    const int width = k == 0 ? P : kWidth;
                    float *o = sum + (k == 0 ? cmap[i] : (int)w_off_hidden(a.d, k) + i) + 32 * p * width;
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        float *at = o + acc_row(j, h0) * width;
                        *at = first ? acc[k][p][q][j] : *at + acc[k][p][q][j];
                    }
                }
        if (h0 == 0 && part == 0) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                float *at = sum + off_out + 32 * p + s0;
                *at = first ? dwo[p] : *at + dwo[p];
            }
        }
        __syncthreads();
    }
    float *out = a.ws + (int64_t)blockIdx.x * a.d.n_params;
    for (int i = threadIdx.x; i < (int)a.d.n_params; i += blockDim.x)
        out[i] = i < off_out + kWidth ? sum[i] : 0.0f;   // output rows past the first: padding
}

// Launchers, one per weight dtype; each returns 0 or records an error.  workgroups: rows of ws.
int32_t launch_mlp_backward_twin_f16(const MlpArgs &a, unsigned workgroups, hipStream_t st);
int32_t launch_mlp_backward_twin_bf16(const MlpArgs &a, unsigned workgroups, hipStream_t st);
int32_t launch_mlp_backward_twin_f32(const MlpArgs &a, unsigned workgroups, hipStream_t st);

template <typename T, int H, int NP>
int32_t launch_mlp_backward_twin_as(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    constexpr size_t bytes = TwinLds<T, H, (NP + 1) / 2>::total;
    static_assert(bytes <= kLdsLimit, "LDS image too large");
    return a.d.activation == NECT_ACT_RELU
               ? launch_with_lds(k_mlp_backward_twin<T, H, NP, true>, workgroups, 64 * kTwinWaves, bytes, st, a, "k_mlp_backward_twin")
               : launch_with_lds(k_mlp_backward_twin<T, H, NP, false>, workgroups, 64 * kTwinWaves, bytes, st, a, "k_mlp_backward_twin");
}

template <typename T, int H0, int H1>
int32_t launch_mlp_backward_twin(const MlpArgs &a, unsigned workgroups, hipStream_t st) {
    if constexpr (H0 <= H1) {
        if (a.d.n_hidden_layers == H0) {
            switch (a.d.n_input_padded / 16) {
                case 1: return launch_mlp_backward_twin_as<T, H0, 1>(a, workgroups, st);
                case 2: return launch_mlp_backward_twin_as<T, H0, 2>(a, workgroups, st);
                case 3: return launch_mlp_backward_twin_as<T, H0, 3>(a, workgroups, st);
                default: return launch_mlp_backward_twin_as<T, H0, 4>(a, workgroups, st);
            }
        }
        return launch_mlp_backward_twin<T, H0 + 1, H1>(a, workgroups, st);
    } else {
        set_error("k_mlp_backward_twin: no instantiation for this depth");
        return 1;
    }
}

}  // namespace nect
