// The real-space half of an FNO layer in one kernel (bfloat16 operands, FP32
// accumulation on the MFMA units): inverse x transform, channel mixing, bias and
// GELU of one row y of one sample, and from the new activations still in LDS the
// forward x transform of the next layer or the projection head.
//
// As separate products each of these reads or writes the whole activation field:
// at batch 16, 256^2, width 64 the inverse x transform stored 268 MB of FP32 for
// the mixing to read back, the mixing's result was read again by the next x
// transform, and the projection's 128 hidden channels (537 MB of FP32) were stored
// and read once.  Here a layer reads 134 MB of activations (the first one the
// 4 MB input field, lifting it in place) and writes 134 MB (the last one 4 MB).
// Network step at batch 16: 2.79 -> 0.83 ms (a layer 105 us for 285 MB, 2.7 TB/s,
// the projecting one 179 us; they were 88 to 313 us per product, four products a
// layer).  Bound by the vector units: the GELU, its operands' conversions and the
// transposes through LDS; the products take a tenth.
//
// The products are the GEMMs of gemm.hip in the same order of summation (32x32x16
// MFMA, k ascending), and training evaluates the same GELU, so what it keeps has the
// bits of the separate products.  Inference evaluates gelu_fast (within 4e-8 of Phi,
// like erff), so its activations differ from training's where that moves a rounding
// to bfloat16, and orders the projection's final sum over hidden channels differently.
//
// A workgroup of four wavefronts holds the row's c x n activations: Vt[x][i]
// (k = channel contiguous, the mixing's operand), O[o][x] (k = x contiguous, the
// x transform's).  Widths up to 64, rows up to 256 and 2 MX up to 32 are padded
// with zeros to the MFMA tile; other shapes run on the separate products.
#include "fno_layer.h"

namespace tara {

namespace {

typedef __bf16 __attribute__((ext_vector_type(8))) v8bf;
typedef float __attribute__((ext_vector_type(16))) v16f;

__device__ __forceinline__ uint16_t to_bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (uint16_t)((u >> 16) | 0x40);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// Two floats rounded to bfloat16 (nearest even), the first in the low half.
__device__ __forceinline__ uint32_t to_bf2(float a, float b)
{
    typedef float __attribute__((ext_vector_type(2))) v2f;
    typedef __bf16 __attribute__((ext_vector_type(2))) v2bf;
    const v2f f = {a, b};
    const v2bf h = __builtin_convertvector(f, v2bf);
    return __builtin_bit_cast(uint32_t, h);
}

// gelu(v) = v Phi(v) in its library form, for what training keeps in FP32.
__device__ __forceinline__ float gelu(float v) { return 0.5f * v * (1.f + erff(v * 0.70710678118654752f)); }

// gelu for inference.  Phi(-x) = 2^-(1 + x P(x)) for x >= 0, P a degree-9 fit of
// (-log2(2 Phi(-x)))/x on [0, 6.5] (iteratively reweighted least squares on
// Chebyshev nodes, weighted by the absolute error of Phi): within 4.0e-8 of Phi
// evaluated in FP32, where 0.5 (1 + erff) is within 6e-8.  No branch: erff's two
// ranges cost about 70 instructions a value, and a layer evaluates 67 million, the
// projection 134 million; this costs 17 (projecting layer at batch 16 311 ->
// 221 us).
__device__ __forceinline__ float gelu_fast(float v)
{
    const float x = fabsf(v);
    float p = 4.283852561570711e-08f;
    p = fmaf(p, x, -1.1479279464765568e-06f);
    p = fmaf(p, x, 1.3412854059424717e-05f);
    p = fmaf(p, x, -8.738827455090359e-05f);
    p = fmaf(p, x, 0.00030743979732505977f);
    p = fmaf(p, x, -4.0233320760307834e-05f);
    p = fmaf(p, x, -0.006915317382663488f);
    p = fmaf(p, x, 0.05242950841784477f);
    p = fmaf(p, x, 0.4592222571372986f);
    p = fmaf(p, x, 1.151104211807251f);
    float q = __builtin_amdgcn_exp2f(fmaf(-p, x, -1.f));  // Phi(-x)
    q = x < 6.5f ? q : 0.f;                               // 4e-11 there
    return v * (v >= 0.f ? 1.f - q : q);
}

__device__ __forceinline__ v16f zero16()
{
    v16f a;
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = 0.f;
    return a;
}

constexpr int NX = 256;  // padded row length
constexpr int QP = 32;   // padded 2 MX

// lane l of a 32x32x16 operand: row (or column) l % 32, k = 8 (l / 32) .. +7
template <int CT>
struct Tile {
    static constexpr int CP = 32 * CT;
    static constexpr int VS = CP + 8;  // row strides (elements): 16-byte aligned, 8 lanes on distinct banks
    static constexpr int OS = NX + 8;
    static constexpr int VT = NX * VS, O = CP * OS;  // elements
    uint16_t* vt;
    uint16_t* o;
};

// Vt[x][i] = the lift of the row: bf16(wl[i] (om[x] / sig) + bl[i]), 0 past c.
template <int CT>
__device__ __forceinline__ void lift_vt(const FnoLayerArgs& a, const Tile<CT>& s, int b, int y)
{
    // a pixel per thread (rows of at most 64 or 128 pixels: 4 or 2 threads per
    // pixel, a part of the channels each), the weights uniform
    const int w = a.n > 128 ? 256 : a.n > 64 ? 128 : 64;
    const int x = threadIdx.x % w, g = __builtin_amdgcn_readfirstlane(threadIdx.x / w), ng = 256 / w;
    if (x >= a.n) return;
    const float r = a.om[(size_t)b * a.n * a.n + (size_t)y * a.n + x] / a.sig[b];
    for (int i0 = 8 * g; i0 < Tile<CT>::CP; i0 += 8 * ng) {
        float h[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) h[k] = i0 + k < a.c ? a.wl[i0 + k] * r + a.bl[i0 + k] : 0.f;
        *reinterpret_cast<uint4*>(&s.vt[x * Tile<CT>::VS + i0]) =
            make_uint4(to_bf2(h[0], h[1]), to_bf2(h[2], h[3]), to_bf2(h[4], h[5]), to_bf2(h[6], h[7]));
    }
}

// Vt[x][i] = v[b][i][y][x]: blocks of 8 channels x 8 pixels transposed in
// registers; the channel blocks of a pixel block on neighbouring lanes, so that a
// wave reads 128-byte runs of each channel and stores 128-byte runs of Vt.
template <int CT>
__device__ __forceinline__ void load_vt(const FnoLayerArgs& a, const Tile<CT>& s, int b, int y)
{
    constexpr int IB = Tile<CT>::CP / 8;
    const size_t np = (size_t)a.n * a.n;
    for (int u = threadIdx.x; u < IB * (a.n / 8); u += 256) {
        const int i0 = (u % IB) * 8, x0 = (u / IB) * 8;
        uint32_t r[8][4];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            uint4 q = make_uint4(0, 0, 0, 0);
            if (i0 + k < a.c)
                q = *reinterpret_cast<const uint4*>(a.v + ((size_t)b * a.c + i0 + k) * np + (size_t)y * a.n + x0);
            r[k][0] = q.x;
            r[k][1] = q.y;
            r[k][2] = q.z;
            r[k][3] = q.w;
        }
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            const uint32_t sel = x % 2 ? 0x07060302u : 0x05040100u;  // the high or low halves of a pair
            uint4 q;
            q.x = __builtin_amdgcn_perm(r[1][x / 2], r[0][x / 2], sel);
            q.y = __builtin_amdgcn_perm(r[3][x / 2], r[2][x / 2], sel);
            q.z = __builtin_amdgcn_perm(r[5][x / 2], r[4][x / 2], sel);
            q.w = __builtin_amdgcn_perm(r[7][x / 2], r[6][x / 2], sel);
            *reinterpret_cast<uint4*>(&s.vt[(x0 + x) * Tile<CT>::VS + i0]) = q;
        }
    }
}

// T1[y][q][b c + o] = sum_x FxT[q][x] O[o][x]; wave w < CT takes channels 32 w ..
template <int CT>
__device__ __forceinline__ void x_transform(const FnoLayerArgs& a, const Tile<CT>& s, int b, int y)
{
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    if (wave >= CT) return;
    const int l = lane % 32, kh = 8 * (lane / 32);
    v16f acc = zero16();
    for (int k = 0; k < a.n; k += 16) {
        const v8bf fa = *reinterpret_cast<const v8bf*>(a.fx + l * NX + k + kh);
        const v8bf fb = *reinterpret_cast<const v8bf*>(&s.o[(32 * wave + l) * Tile<CT>::OS + k + kh]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc, 0, 0, 0);
    }
    const int o = 32 * wave + l;
    const size_t F = (size_t)a.nb * a.c;
    if (o >= a.c) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int q = 8 * (i / 4) + 4 * (lane / 32) + i % 4;
        if (q < a.q2) a.t1[((size_t)y * a.q2 + q) * F + (size_t)b * a.c + o] = to_bf(acc[i]);
    }
}

// O[o][x] past the row (its x-transform weights are zero; it must be finite).
template <int CT>
__device__ __forceinline__ void zero_o_tail(const FnoLayerArgs& a, const Tile<CT>& s)
{
    const int k1 = (a.n + 15) / 16 * 16;
    for (int u = threadIdx.x; u < Tile<CT>::CP * (k1 - a.n); u += 256)
        s.o[(u / (k1 - a.n)) * Tile<CT>::OS + a.n + u % (k1 - a.n)] = 0;
}

template <int CT>
__global__ __launch_bounds__(256) void k_fno_lift_x(FnoLayerArgs a)
{
    __shared__ __align__(16) uint16_t lds[Tile<CT>::O];
    const Tile<CT> s{nullptr, lds};
    const int y = blockIdx.x, b = blockIdx.y;
    const float sig = a.sig[b];
    // two pixels of a channel per thread and store: channels over the wavefronts,
    // which makes the weights uniform; a lane's pixels stay the same
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const float* row = a.om + (size_t)b * a.n * a.n + (size_t)y * a.n;
    for (int x = 2 * lane; x < a.n; x += 128) {
        const float r0 = row[x] / sig, r1 = row[x + 1] / sig;
#pragma unroll 8
        for (int o = wave; o < Tile<CT>::CP; o += 4) {
            const float w = o < a.c ? a.wl[o] : 0.f, c = o < a.c ? a.bl[o] : 0.f;
            *reinterpret_cast<uint32_t*>(&s.o[o * Tile<CT>::OS + x]) = to_bf2(w * r0 + c, w * r1 + c);
        }
    }
    zero_o_tail<CT>(a, s);
    __syncthreads();
    x_transform<CT>(a, s, b, y);
}

// ZV: rows of z are 16-byte aligned.
template <int CT, bool FIRST, bool LAST, bool TRAIN, bool ZV>
__global__ __launch_bounds__(256, TRAIN ? 2 : 3) void k_fno_layer(FnoLayerArgs a)
{
    using S = Tile<CT>;
    // inference: O takes Vt's place once every wavefront has done its mixing (its
    // results wait in registers), which lets three workgroups share a CU instead of
    // two (layer at batch 16 122 -> 105 us); the projection needs Vt only
    constexpr bool SWAP = !LAST && !TRAIN;
    constexpr int LDS = TRAIN ? S::VT + S::O : S::VT > S::O ? S::VT : S::O;
    __shared__ __align__(16) uint16_t lds[LDS];
    const S s{lds, TRAIN ? lds + S::VT : lds};
    const int y = blockIdx.x, b = blockIdx.y;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int l = lane % 32, lh = lane / 32, kh = 8 * lh;
    const size_t np = (size_t)a.n * a.n;
    // inverse x transform's operand: z rows of this y, 2 MX padded to 32
    v8bf fz[CT][2];
#pragma unroll
    for (int r = 0; r < CT; ++r) {
        const int o = 32 * r + l;
        const uint16_t* zr = a.z + (((size_t)b * a.c + (o < a.c ? o : 0)) * a.n + y) * a.q2;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            uint16_t h[8];
            const int q0 = 16 * k + kh;
            if (ZV) {
                uint4 q = make_uint4(0, 0, 0, 0);
                if (o < a.c && q0 < a.q2) q = *reinterpret_cast<const uint4*>(zr + q0);
                __builtin_memcpy(h, &q, 16);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) h[i] = o < a.c && q0 + i < a.q2 ? zr[q0 + i] : 0;
            }
            __builtin_memcpy(&fz[r][k], h, 16);
        }
    }
    if constexpr (FIRST)
        lift_vt<CT>(a, s, b, y);
    else
        load_vt<CT>(a, s, b, y);
    if constexpr (TRAIN) zero_o_tail<CT>(a, s);
    __syncthreads();
    // Result registers: SWAP row x = 8 (i / 4) + 4 lh + i % 4, column o = l (four
    // consecutive pixels of one channel: one 8-byte store to O, one bias per lane);
    // else row o, column x = l (training: runs of 32 pixels to memory; projection:
    // four consecutive channels to Vt).
    float bias[CT];
    uint2 keep[2][CT][4];  // SWAP: this wavefront's two column tiles, packed
#pragma unroll
    for (int r = 0; r < CT; ++r) bias[r] = SWAP && 32 * r + l < a.c ? a.bias[32 * r + l] : 0.f;
#pragma unroll
    for (int h2 = 0; h2 < NX / 128; ++h2) {
        const int ct = wave + 4 * h2;
        if (32 * ct >= a.n) continue;
        const int x = 32 * ct + l;
        v16f acc[CT];
#pragma unroll
        for (int r = 0; r < CT; ++r) {
            // kv = inverse x transform; acc = W v; then acc + kv + bias
            v16f kv = zero16();
            acc[r] = zero16();
#pragma unroll
            for (int k = 0; k < QP / 16; ++k) {
                const v8bf h = *reinterpret_cast<const v8bf*>(a.hxt + x * QP + 16 * k + kh);
                kv = __builtin_amdgcn_mfma_f32_32x32x16_bf16(SWAP ? h : fz[r][k], SWAP ? fz[r][k] : h, kv, 0, 0, 0);
            }
#pragma unroll
            for (int k = 0; k < S::CP; k += 16) {
                const v8bf w = *reinterpret_cast<const v8bf*>(a.w + (32 * r + l) * S::CP + k + kh);
                const v8bf v = *reinterpret_cast<const v8bf*>(&s.vt[x * S::VS + k + kh]);
                acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(SWAP ? v : w, SWAP ? w : v, acc[r], 0, 0, 0);
            }
            if constexpr (SWAP) {
#pragma unroll
                for (int i = 0; i < 16; i += 4) {
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[j] = (acc[r][i + j] + kv[i + j]) + bias[r];
                        if (a.act) v[j] = gelu_fast(v[j]);
                    }
                    keep[h2][r][i / 4] = make_uint2(to_bf2(v[0], v[1]), to_bf2(v[2], v[3]));
                }
                continue;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int o = 32 * r + 8 * (i / 4) + 4 * lh + i % 4;
                const bool in = o < a.c && x < a.n;
                float v = acc[r][i] + kv[i];
                if (o < a.c) v += a.bias[o];
                const size_t q = ((size_t)b * a.c + o) * np + (size_t)y * a.n + x;
                if (TRAIN && in) a.pre[q] = v;
                if (a.act) v = TRAIN ? gelu(v) : gelu_fast(v);
                if (TRAIN && in) a.v32[q] = v;
                acc[r][i] = v;
            }
        }
        if constexpr (LAST) {
            // the projection's operand: this wave's own rows of Vt, k = channel
#pragma unroll
            for (int r = 0; r < CT; ++r)
#pragma unroll
                for (int i = 0; i < 16; i += 4)
                    *reinterpret_cast<uint2*>(&s.vt[x * S::VS + 32 * r + 8 * (i / 4) + 4 * lh]) =
                        make_uint2(to_bf2(acc[r][i], acc[r][i + 1]), to_bf2(acc[r][i + 2], acc[r][i + 3]));
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float sum = 0.f;
#pragma unroll 1
            for (int j0 = 0; j0 < 2 * a.c; j0 += 32) {
                // padded copies of b1 and w2, row j = 8 (i / 4) + 4 lh + i % 4
                float4 b1[4], w2[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    b1[i] = *reinterpret_cast<const float4*>(a.b1 + j0 + 8 * i + 4 * lh);
                    w2[i] = *reinterpret_cast<const float4*>(a.w2 + j0 + 8 * i + 4 * lh);
                }
                v16f h = zero16();
#pragma unroll
                for (int k = 0; k < S::CP; k += 16)
                    h = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        *reinterpret_cast<const v8bf*>(a.w1 + (j0 + l) * S::CP + k + kh),
                        *reinterpret_cast<const v8bf*>(&s.vt[x * S::VS + k + kh]), h, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sum += w2[i].x * gelu_fast(h[4 * i] + b1[i].x);
                    sum += w2[i].y * gelu_fast(h[4 * i + 1] + b1[i].y);
                    sum += w2[i].z * gelu_fast(h[4 * i + 2] + b1[i].z);
                    sum += w2[i].w * gelu_fast(h[4 * i + 3] + b1[i].w);
                }
            }
            sum += __shfl_xor(sum, 32);
            if (lh == 0 && x < a.n) {
                const size_t q = (size_t)b * np + (size_t)y * a.n + x;
                a.out[q] = a.om[q] + a.sig[b] * (sum + a.b2[0]);
            }
        } else if (TRAIN && x < a.n) {
#pragma unroll
            for (int r = 0; r < CT; ++r)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    s.o[(32 * r + 8 * (i / 4) + 4 * lh + i % 4) * S::OS + x] = to_bf(acc[r][i]);
        }
    }
    if constexpr (SWAP) {
        __syncthreads();  // Vt has been read
        zero_o_tail<CT>(a, s);
#pragma unroll
        for (int h2 = 0; h2 < NX / 128; ++h2)
#pragma unroll
            for (int r = 0; r < CT; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int x0 = 32 * (wave + 4 * h2) + 8 * i + 4 * lh;
                    if (x0 < a.n) *reinterpret_cast<uint2*>(&s.o[(32 * r + l) * S::OS + x0]) = keep[h2][r][i];
                }
    }
    if constexpr (!LAST) {
        __syncthreads();
        if (a.vn)
            for (int u = threadIdx.x; u < a.c * (a.n / 8); u += 256) {
                const int o = u / (a.n / 8), x0 = (u % (a.n / 8)) * 8;
                *reinterpret_cast<uint4*>(a.vn + ((size_t)b * a.c + o) * np + (size_t)y * a.n + x0) =
                    *reinterpret_cast<const uint4*>(&s.o[o * S::OS + x0]);
            }
        if (a.t1) x_transform<CT>(a, s, b, y);
    }
}

// All padded copies in one launch (a launch each cost a training step of a small
// network 20 to 50 of its 400 to 800 us): the layers' and the projection's matrices,
// then the projection's two vectors.
__global__ void k_fno_pad(FnoPadArgs a)
{
    const int cp = a.cp, h = 2 * cp;
    const size_t nm = (size_t)(a.layers + 2) * cp * cp;  // W of every layer, W1
    const size_t u = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (u < nm) {
        const size_t nw = (size_t)a.layers * cp * cp;
        const int l = (int)(u / (cp * cp)), k = (int)(u % cp);
        const int r = u < nw ? (int)(u / cp % cp) : (int)((u - nw) / cp);  // row, of C or 2 C
        const float* w = u < nw ? a.w + (size_t)l * a.c * a.c : a.w1;
        const uint16_t v = k < a.c && r < (u < nw ? a.c : 2 * a.c) ? to_bf(w[r * a.c + k]) : 0;
        if (u < nw)
            a.wp[u] = v;
        else
            a.w1p[u - nw] = v;
    } else if (u < nm + 2 * h) {
        const int q = (int)(u - nm), j = q % h;
        const float v = j < 2 * a.c ? (q < h ? a.b1 : a.w2)[j] : 0.f;
        (q < h ? a.b1p : a.w2p)[j] = v;
    }
}

template <int CT, bool FIRST, bool LAST, bool TRAIN>
void launch_layer(const FnoLayerArgs& a, hipStream_t st)
{
    const dim3 g(a.n, a.nb);
    if (a.q2 % 8 == 0)
        hipLaunchKernelGGL((k_fno_layer<CT, FIRST, LAST, TRAIN, true>), g, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((k_fno_layer<CT, FIRST, LAST, TRAIN, false>), g, dim3(256), 0, st, a);
}

template <int CT>
int launch_layer_ct(const FnoLayerArgs& a, hipStream_t st)
{
    const bool first = !a.v, last = a.out != nullptr, train = a.pre != nullptr;
    TARA_CHECK(!(last && train), TARA_ERR_ARG, "fno: the fused projection keeps nothing for training");
    if (train)
        first ? launch_layer<CT, true, false, true>(a, st) : launch_layer<CT, false, false, true>(a, st);
    else if (last)
        first ? launch_layer<CT, true, true, false>(a, st) : launch_layer<CT, false, true, false>(a, st);
    else
        first ? launch_layer<CT, true, false, false>(a, st) : launch_layer<CT, false, false, false>(a, st);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

}  // namespace

bool fno_fused_ok(int n, int c, int q2) { return n <= NX && n % 8 == 0 && c <= 64 && q2 <= QP; }

int fno_pad(int c) { return c <= 32 ? 32 : 64; }

int fno_lift_x(const FnoLayerArgs& a, hipStream_t st)
{
    TARA_CHECK(fno_fused_ok(a.n, a.c, a.q2) && a.nb <= 65535, TARA_ERR_ARG, "fno: shape does not fit the fused layer");
    if (a.c <= 32)
        hipLaunchKernelGGL(k_fno_lift_x<1>, dim3(a.n, a.nb), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(k_fno_lift_x<2>, dim3(a.n, a.nb), dim3(256), 0, st, a);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

int fno_layer(const FnoLayerArgs& a, hipStream_t st)
{
    TARA_CHECK(fno_fused_ok(a.n, a.c, a.q2) && a.nb <= 65535, TARA_ERR_ARG, "fno: shape does not fit the fused layer");
    return a.c <= 32 ? launch_layer_ct<1>(a, st) : launch_layer_ct<2>(a, st);
}

int fno_pad_weights(const FnoPadArgs& a, hipStream_t st)
{
    const size_t n = (size_t)(a.layers + 2) * a.cp * a.cp + 4 * a.cp;
    hipLaunchKernelGGL(k_fno_pad, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
    TARA_HIP(hipGetLastError());
    return TARA_OK;
}

}  // namespace tara
