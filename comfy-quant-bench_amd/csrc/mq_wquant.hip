// Offline weight quantizer (the converter side of the path): rotate each weight row by H_hblock and
// quantize it to one of the GEMMs' weight formats.
//
// The rotation is the activation quantizer's (mq_rotate.h: one wavefront per 1024-column chunk, each
// lane 16 consecutive columns, the pinned radix-4 FWHT of
// experiments/qwen21-kernel/kernels/g64_quant.cu:68-86 in registers and an LDS transpose). The group
// formats need nothing across chunks (a 64-column group is four lanes of one 16-lane row), so every
// wave takes one chunk of one row and nothing waits at a barrier; the row formats give a row to the
// four waves of a workgroup, NCH chunks each, which combine the row's maximum through LDS. The formats:
//   U4_ASYM_G64  lo = min(min w, 0), hi = max(max w, 0), s = fp16((hi - lo) / 15),
//                z = clamp(rne(-lo / s), 0, 15), q = clamp(rne(w / s) + z, 0, 15); s = 0 -> q = z = 0
//   I4_SYM_G64   s = fp16(max |w| / 7), q = clamp(rne(w / s), -7, 7); s = 0 -> q = 0
//   I4_ROW       s = max(max |w|, 1e-10) / 7,   q = clamp(rne(w / s), -7, 7)
//   I8_ROW       s = max(max |w|, 1e-10) / 127, q = clamp(rne(w / s), -127, 127)
// where w is the rotated weight (the group formats are the configs' schemes, with the min / max code
// choice of custom_nodes/comfy-lowbit-loader/formats.py:131-149 and the symmetric form of
// tools/svdquant_probe.py:105-115; the row formats are tools/gptq_w4a4.py:197-203 and
// tools/_formats.py:128-167). Scales are IEEE quotients (div_limit, checked for every
// float). Codes and zero-points take the activation quantizer's product with the reciprocal and its
// exact division wherever that product lies near a half-integer (quant16's argument: |w / s| < 128,
// here at most 127 or, for an fp16 scale rounded down in its subnormal range, 23), so they are the
// IEEE quotient's.
//
// What bounds it: HBM, 2.5 bytes per bf16 weight. At N = 12288, K = 3072 (96 MB): 22.4 us (26.5 with a
// conversion, a compare and a shift per code and IEEE divisions per lane, when the VALU set it); one
// workgroup per row with the row in LDS, a barrier per butterfly stage, one thread per group and
// an IEEE division per weight took 142 us.
#include "mq_device.h"
#include <algorithm>
#include "mq_internal.h"
#include "mq_rotate.h"

#pragma clang fp contract(off)

namespace mq {
namespace {

constexpr int kWaves = 4;   // wavefronts per workgroup

// 16 consecutive weights of type DT at element i of w, as fp32; vec: 16-byte loads (the host has
// checked the base and the row stride), else element by element.
template <int DT>
__device__ __forceinline__ void load16(const void* w, int64_t i, bool vec, float (&v)[16]) {
    if constexpr (DT == kDtF32) {
        const float* p = static_cast<const float*>(w) + i;
        if (vec) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 f = *reinterpret_cast<const float4*>(p + 4 * j);
                v[4 * j] = f.x;
                v[4 * j + 1] = f.y;
                v[4 * j + 2] = f.z;
                v[4 * j + 3] = f.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = p[j];
        }
    } else {
        const uint16_t* p = static_cast<const uint16_t*>(w) + i;
        uint32_t h[8];
        if (vec) {
            const uint4 a = *reinterpret_cast<const uint4*>(p), b = *reinterpret_cast<const uint4*>(p + 8);
            h[0] = a.x; h[1] = a.y; h[2] = a.z; h[3] = a.w;
            h[4] = b.x; h[5] = b.y; h[6] = b.z; h[7] = b.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) h[j] = p[2 * j] | static_cast<uint32_t>(p[2 * j + 1]) << 16;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v[2 * j] = DT == kDtF16 ? f16lo(h[j]) : bf16lo(h[j]);
            v[2 * j + 1] = DT == kDtF16 ? f16hi(h[j]) : bf16hi(h[j]);
        }
    }
}

// rotate_chunk_lds with the Hadamard block chosen at run time (wave-uniform).
__device__ __forceinline__ void rotate(float (&v)[16], const LdsTranspose& tr, int hblock) {
    if (hblock >= 16) {
        stage_reg<0>(v);
        stage_reg<2>(v);
    }
    if (hblock >= 64) {
        tr(v);
        stage_reg<0>(v);
        if (hblock >= 256) stage_reg<2>(v);
        tr(v);
    }
}

// kMagic + rne(v / s) of N values, for |v / s| < 128 and r = recip_row(s) (0 where every code is to be
// 0): the rounded product, or the IEEE quotient's rounding where the product lies near a half-integer
// (quant16). The integer sits in the low mantissa bits (two's complement), where the codes are clamped,
// shifted by the zero-point (both exact) and packed from, with no conversion.
template <int N>
__device__ __forceinline__ void round_magic(const float (&v)[N], float r, float s, float (&m)[N]) {
    float dmax = 0.0f;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        m[j] = __builtin_fmaf(v[j], r, kMagic);
        dmax = __builtin_fmaxf(dmax, __builtin_fabsf(__builtin_fmaf(v[j], r, -(m[j] - kMagic))));
    }
    if (dmax > kTieWindow) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (__builtin_fabsf(__builtin_fmaf(v[j], r, -(m[j] - kMagic))) > kTieWindow)
                m[j] = kMagic + __builtin_rintf(v[j] / s);
    }
}
// kMagic + clamp(n, lo, hi) of kMagic + n; NaN gives lo, as fmin(fmax(NaN, lo), hi) does.
__device__ __forceinline__ float clamp_magic(float m, float lo, float hi) {
    return __builtin_amdgcn_fmed3f(m, kMagic + lo, kMagic + hi);
}

// The low bytes of four dwords as one, in order.
__device__ __forceinline__ uint32_t low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_amdgcn_perm(b, a, 0x0c0c0400u) | __builtin_amdgcn_perm(d, c, 0x04000c0cu);
}
// 8 codes (magic-biased) as the nibbles of a dword, 4 codes as its bytes.
template <bool SIGNED>
__device__ __forceinline__ uint32_t nibbles8(const float* m) {
    uint32_t t[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t even = __float_as_uint(m[2 * e]), odd = __float_as_uint(m[2 * e + 1]);
        t[e] = (odd << 4) | (SIGNED ? even & 0xfu : even);   // (an unsigned code's low byte is the code)
    }
    return low_bytes(t[0], t[1], t[2], t[3]);
}
__device__ __forceinline__ uint32_t bytes4(const float* m) {
    return low_bytes(__float_as_uint(m[0]), __float_as_uint(m[1]), __float_as_uint(m[2]), __float_as_uint(m[3]));
}
// 8 bytes of packed codes at p (4-byte aligned; wide: 8-byte aligned)
__device__ __forceinline__ void store8(uint8_t* p, uint32_t lo, uint32_t hi, bool wide) {
    if (wide) {
        *reinterpret_cast<uint2*>(p) = uint2{lo, hi};
    } else {
        *reinterpret_cast<uint32_t*>(p) = lo;
        *reinterpret_cast<uint32_t*>(p + 4) = hi;
    }
}

// Group formats: wave u of the grid takes chunk u % chunks of row u / chunks. nonfinite (or null) is
// set to 1 where a group's scale is not finite.
template <int DT, int FMT>
__global__ void __launch_bounds__(64 * kWaves)
wquant_group_kernel(const void* __restrict__ w, int64_t ldw, int64_t N, int K, int chunks, int hblock, bool vec,
                    uint8_t* __restrict__ q, int64_t ldq, bool wide, uint16_t* __restrict__ scale, int64_t ld_scale,
                    uint8_t* __restrict__ zero, int64_t ld_zero, int* nonfinite) {
    static_assert(FMT == 0 || FMT == 1, "U4_ASYM_G64, I4_SYM_G64");
    __shared__ __attribute__((aligned(16))) float tr_lds[kWaves * kTrWave];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int seg = (lane >> 2) + 16 * (lane & 3);
    float* tb = tr_lds + wave * kTrWave + (lane & 3) * kTrG;
    const LdsTranspose tr{tb + (lane >> 2), tb + (lane >> 2) * kTrS};
    for (int64_t unit = static_cast<int64_t>(blockIdx.x) * kWaves + wave; unit < N * chunks;
         unit += static_cast<int64_t>(gridDim.x) * kWaves) {
        const int64_t row = unit / chunks;
        const int col = static_cast<int>(unit % chunks) * 1024 + 16 * seg;
        const bool in = col < K;   // lanes past the row work on its first columns and store nothing
        float v[16];
        load16<DT>(w, row * ldw + (in ? col : 0), vec, v);
        rotate(v, tr, hblock);

        // the group's extremes: 16 values here, then the four lanes that differ in lane bits 2 and 3
        [[maybe_unused]] float lo = 0.0f;
        _Float16 h;
        if constexpr (FMT == 0) {
            float mn = v[0], mx = v[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) {
                mn = __builtin_fminf(mn, v[e]);
                mx = __builtin_fmaxf(mx, v[e]);
            }
            mn = __builtin_fminf(mn, dpp_mov<kRowRor4>(mn));
            mx = __builtin_fmaxf(mx, dpp_mov<kRowRor4>(mx));
            mn = __builtin_fminf(mn, dpp_mov<kRowRor8>(mn));
            mx = __builtin_fmaxf(mx, dpp_mov<kRowRor8>(mx));
            lo = __builtin_fminf(mn, 0.0f);
            h = static_cast<_Float16>(div_limit<15>(__builtin_fmaxf(mx, 0.0f) - lo));
        } else {
            float am = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e) am = __builtin_fmaxf(am, __builtin_fabsf(v[e]));
            am = __builtin_fmaxf(am, dpp_mov<kRowRor4>(am));
            am = __builtin_fmaxf(am, dpp_mov<kRowRor8>(am));
            h = static_cast<_Float16>(div_limit<7>(am));
        }
        const float s = static_cast<float>(h);
        const float r = s == 0.0f ? 0.0f : recip_row(s);   // (a scale of 0: codes and zero-point 0)
        float z = 0.0f, c[16];
        if constexpr (FMT == 0) {
            const float t[1] = {-lo};
            float m[1];
            round_magic(t, r, s, m);
            z = clamp_magic(m[0], 0.0f, 15.0f) - kMagic;
        }
        round_magic(v, r, s, c);
        // (a NaN weight gets the lower bound: 0 where the scale is 0, as every other code of that group)
        const float lim = s == 0.0f ? 0.0f : 7.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            c[e] = FMT == 0 ? clamp_magic(c[e] + z, 0.0f, 15.0f) : clamp_magic(c[e], -lim, lim);
        if (in) store8(q + row * ldq + col / 2, nibbles8<FMT == 1>(c), nibbles8<FMT == 1>(c + 8), wide);
        const bool lead = in && (lane & 12) == 0;   // one lane per group, of column col
        if (lead) {
            scale[row * ld_scale + col / 64] = __builtin_bit_cast(uint16_t, h);
            if (nonfinite && !(s < __builtin_inff())) *nonfinite = 1;
        }
        if constexpr (FMT == 0) {
            // two groups per byte: the odd one sits 16 lanes on (absent past an odd number of groups)
            const int zi = in ? static_cast<int>(z) : 0;
            const int z1 = __shfl_xor(zi, 16, 64);
            if (lead && (lane & 16) == 0) zero[row * ld_zero + col / 128] = static_cast<uint8_t>(zi | (z1 << 4));
        }
    }
}

// Row formats: one workgroup per row, wave i its chunks i, i + 4, ...
template <int DT, int FMT, int NCH>
__global__ void __launch_bounds__(64 * kWaves)
wquant_row_kernel(const void* __restrict__ w, int64_t ldw, int K, int hblock, bool vec, uint8_t* __restrict__ q,
                  int64_t ldq, bool wide, float* __restrict__ scale) {
    static_assert(FMT == 2 || FMT == 3, "I4_ROW, I8_ROW");
    __shared__ __attribute__((aligned(16))) float tr_lds[kWaves * kTrWave];
    __shared__ float red[kWaves];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row = blockIdx.x;
    const int seg = (lane >> 2) + 16 * (lane & 3);
    float* tb = tr_lds + wave * kTrWave + (lane & 3) * kTrG;
    const LdsTranspose tr{tb + (lane >> 2), tb + (lane >> 2) * kTrS};
    float v[NCH][16], am = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int col = (i * kWaves + wave) * 1024 + 16 * seg;
        load16<DT>(w, row * ldw + (col < K ? col : 0), vec, v[i]);
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        rotate(v[i], tr, hblock);
        if ((i * kWaves + wave) * 1024 + 16 * seg < K)
#pragma unroll
            for (int e = 0; e < 16; ++e) am = __builtin_fmaxf(am, __builtin_fabsf(v[i][e]));
    }
    am = wave_max_nonneg(am);
    if (lane == 0) red[wave] = am;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) am = __builtin_fmaxf(am, red[i]);
    constexpr float L = FMT == 2 ? 7.0f : 127.0f;
    const float s = __builtin_fmaxf(am, 1e-10f) / L, r = recip_row(s);
    if (threadIdx.x == 0) scale[row] = s;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int col = (i * kWaves + wave) * 1024 + 16 * seg;
        if (col >= K) continue;
        float c[16];
        round_magic(v[i], r, s, c);
#pragma unroll
        for (int e = 0; e < 16; ++e) c[e] = clamp_magic(c[e], -L, L);
        if constexpr (FMT == 2) {
            store8(q + row * ldq + col / 2, nibbles8<true>(c), nibbles8<true>(c + 8), wide);
        } else if (wide) {
            *reinterpret_cast<uint4*>(q + row * ldq + col) = uint4{bytes4(c), bytes4(c + 4), bytes4(c + 8), bytes4(c + 12)};
        } else {
            *reinterpret_cast<uint2*>(q + row * ldq + col) = uint2{bytes4(c), bytes4(c + 4)};
            *reinterpret_cast<uint2*>(q + row * ldq + col + 8) = uint2{bytes4(c + 8), bytes4(c + 12)};
        }
    }
}

bool aligned_rows(const void* p, int64_t stride_bytes, int64_t n) {
    return reinterpret_cast<uintptr_t>(p) % n == 0 && stride_bytes % n == 0;
}

template <int DT, int FMT>
int launch_fmt(const void* w, int64_t ldw, int64_t N, int64_t K, int hblock, void* q, int64_t ldq, void* scale,
               int64_t ld_scale, void* zero, int64_t ld_zero, int* nonfinite, hipStream_t stream) {
    const bool vec = aligned_rows(w, ldw * (DT == kDtF32 ? 4 : 2), 16);
    const bool wide = aligned_rows(q, ldq, FMT == 3 ? 16 : 8);
    const int chunks = static_cast<int>((K + 1023) / 1024);
    auto* qb = static_cast<uint8_t*>(q);
    if constexpr (FMT <= 1) {
        const int64_t blocks = std::min<int64_t>((N * chunks + kWaves - 1) / kWaves, int64_t(1) << 22);
        hipLaunchKernelGGL((wquant_group_kernel<DT, FMT>), dim3(static_cast<unsigned>(blocks)), dim3(64 * kWaves), 0,
                           stream, w, ldw, N, static_cast<int>(K), chunks, hblock, vec, qb, ldq, wide,
                           static_cast<uint16_t*>(scale), ld_scale, static_cast<uint8_t*>(zero), ld_zero, nonfinite);
    } else {
        const dim3 grid(static_cast<unsigned>(N)), block(64 * kWaves);
        auto* sc = static_cast<float*>(scale);
#define MQ_WQ(NCH)                                                                                            \
    hipLaunchKernelGGL((wquant_row_kernel<DT, FMT, NCH>), grid, block, 0, stream, w, ldw, static_cast<int>(K), \
                       hblock, vec, qb, ldq, wide, sc)
        if (chunks <= kWaves) MQ_WQ(1);
        else if (chunks <= 2 * kWaves) MQ_WQ(2);
        else if (chunks <= 4 * kWaves) MQ_WQ(4);
        else MQ_WQ(8);   // K <= 32768
#undef MQ_WQ
    }
    return launch_status("quantize_weight");
}

template <int DT>
int launch_dt(const void* w, int64_t ldw, int64_t N, int64_t K, int hblock, int format, void* q, int64_t ldq,
              void* scale, int64_t ld_scale, void* zero, int64_t ld_zero, int* nonfinite, hipStream_t stream) {
    switch (format) {
        case 0: return launch_fmt<DT, 0>(w, ldw, N, K, hblock, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, stream);
        case 1: return launch_fmt<DT, 1>(w, ldw, N, K, hblock, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, stream);
        case 2: return launch_fmt<DT, 2>(w, ldw, N, K, hblock, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, stream);
        case 3: return launch_fmt<DT, 3>(w, ldw, N, K, hblock, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, stream);
        default: break;
    }
    set_error("quantize_weight: unknown format %d", format);
    return -1;
}

// int8 weights [N, K] (row stride ldw) to 16-row tiles [ceil(N / 16)][K / 64][16][64]: one thread
// per 16-byte unit u of the output, u = ((band * G + g) * 16 + row) * 4 + chunk; rows past N get 0.
__global__ void __launch_bounds__(256) tile16_kernel(const uint8_t* w, int64_t ldw, int64_t N, int64_t K,
                                                    uint8_t* out) {
    const int64_t G = K / 64, units = (N + 15) / 16 * 16 * (K / 16);
    for (int64_t u = blockIdx.x * int64_t(256) + threadIdx.x; u < units; u += int64_t(gridDim.x) * 256) {
        const int64_t chunk = u & 3, row = (u >> 2) & 15, g = (u >> 6) % G, band = (u >> 6) / G;
        const int64_t n = band * 16 + row;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (n < N) v = *reinterpret_cast<const uint4*>(w + n * ldw + g * 64 + chunk * 16);
        *reinterpret_cast<uint4*>(out + u * 16) = v;
    }
}

// Packed 4-bit weights [N, K/2] (row stride ldw bytes) expanded to int8 in the same 16-row tiles. One
// wavefront per tile (band, K group g), a lane per row and 16-column chunk (8 packed bytes in, 16 out);
// value v = q - z (uint4 with zero-point nibble z of group g) or the signed nibble, then by layout: 0
// (the group GEMM's int8 activation layout) negated in odd groups, 2 (its x16 int4 layout) 16 * v for
// signed weights, 3 (row scale) v as it is. Four values at a time, as the wide GEMM unpacks packed
// weights: (q + 0x80 - z) ^ 0x80 per byte, or (0x80 + z - q) ^ 0x80 negated, without inter-byte carries,
// and two byte permutes back to k order: about two operations a value where the value at a time it
// replaces, bound by its VALU work, took six and two 64-bit divisions a thread (the expansion is under 2 GiB, so
// the tiles count in 32 bits and the division is one per wave). expand_w4_weight, calls back to back, with the scales' launch below:
// [12288, 3072] uint4 15.9 us (22.9 before; its 60 MB take 12 at the rate of a large copy), [3072, 14336] 16.8
// (25.9); row-scale [3072, 12288] 10.0 (17.6).
enum ExpandKind : int { kExpandU4 = 0, kExpandI4 = 1, kExpandI4x16 = 2 };
template <int KIND>
__global__ void __launch_bounds__(64 * kWaves)
expand_w4_kernel(const uint8_t* __restrict__ qw, int64_t ldw, const uint8_t* __restrict__ wz, int64_t ldwz, int64_t N,
                 int G, bool alternate, uint8_t* __restrict__ out) {
    const int lane = threadIdx.x & 63, chunk = lane & 3;
    const int tiles = static_cast<int>((N + 15) / 16) * G;
    const int t = blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (t < tiles) {
        const int band = t / G, g = t - band * G;
        const int64_t n = static_cast<int64_t>(band) * 16 + (lane >> 2);
        uint32_t o[4] = {0u, 0u, 0u, 0u};
        if (n < N) {
            const uint2 w2 = *reinterpret_cast<const uint2*>(qw + n * ldw + g * 32 + chunk * 8);
            uint32_t z = 8u;
            if constexpr (KIND == kExpandU4) z = (wz[n * ldwz + (g >> 1)] >> (4 * (g & 1))) & 15u;
            const bool neg = alternate && (g & 1);
            const uint32_t zz = z * 0x01010101u;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t w = h ? w2.y : w2.x, lo, hi;
                if constexpr (KIND == kExpandI4x16) {
                    lo = (w << 4) & 0xf0f0f0f0u;
                    hi = w & 0xf0f0f0f0u;
                } else {
                    if constexpr (KIND == kExpandI4) w ^= 0x88888888u;   // v + 8
                    lo = w & 0x0f0f0f0fu;
                    hi = (w >> 4) & 0x0f0f0f0fu;
                    if (neg) {
                        lo = ((0x80808080u | zz) - lo) ^ 0x80808080u;
                        hi = ((0x80808080u | zz) - hi) ^ 0x80808080u;
                    } else {
                        lo = (lo + (0x80808080u - zz)) ^ 0x80808080u;
                        hi = (hi + (0x80808080u - zz)) ^ 0x80808080u;
                    }
                }
                o[2 * h] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
                o[2 * h + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
            }
        }
        *reinterpret_cast<uint4*>(out + static_cast<int64_t>(t) * 1024 + lane * 16) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// fp16 group scales [N, G] (row stride ldws) as the expanded-weight group GEMM's lanes load them:
// dword [g][c][u] (u fastest, ld dwords per [g][c]) = ws[32 u + c, g] | ws[32 u + 16 + c, g] << 16,
// zero for columns past N and groups past G; G4 groups in all (G rounded up to four). A thread takes four
// groups of one (c, u): eight consecutive bytes of each of its two rows (one cache line, where a thread per
// group fetched the line again), and stores that run along u.
__global__ void __launch_bounds__(256) expand_scales_kernel(const uint16_t* __restrict__ ws, int64_t ldws, int64_t N,
                                                           int G, int ld, uint32_t* __restrict__ out) {
    const int ublocks = (ld + 255) / 256;
    const int cg = blockIdx.x / ublocks, c = cg & 15, g0 = cg / 16 * 4;
    const int u = (blockIdx.x - cg * ublocks) * 256 + threadIdx.x;
    if (u >= ld) return;
    const int64_t n0 = 32 * static_cast<int64_t>(u) + c, n1 = n0 + 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int g = g0 + i;
        uint32_t v = 0u;
        if (g < G) {
            if (n0 < N) v = ws[n0 * ldws + g];
            if (n1 < N) v |= static_cast<uint32_t>(ws[n1 * ldws + g]) << 16;
        }
        out[(static_cast<int64_t>(g) * 16 + c) * ld + u] = v;
    }
}

}  // namespace

int launch_expand_scales_w4(const uint16_t* ws, int64_t ldws, int64_t N, int64_t K, uint32_t* out,
                            hipStream_t stream) {
    // One block index over (four groups, c, 256 u): G runs past a grid's 65535 in y and z for one long row. The
    // expansion is under 2 GiB, which keeps the threads under 2^31.
    const int64_t G = K / 64, ld = scale_pair_ld(N), blocks = (G + 3) / 4 * 16 * ((ld + 255) / 256);
    hipLaunchKernelGGL(expand_scales_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, ws, ldws, N,
                       static_cast<int>(G), static_cast<int>(ld), out);
    return launch_status("expand_scales_w4");
}

int launch_expand_weight_w4(const uint8_t* qw, int64_t ldw, const uint8_t* wz, int64_t ldwz, int64_t N, int64_t K,
                            int layout, uint8_t* out, hipStream_t stream) {
    const int G = static_cast<int>(K / 64);
    const int64_t tiles = (N + 15) / 16 * G;
    const dim3 grid(static_cast<unsigned>((tiles + kWaves - 1) / kWaves));   // tiles < 2 GiB / 1 KiB
    const bool alternate = layout == 0;
#define MQ_EX(KIND) \
    hipLaunchKernelGGL(expand_w4_kernel<KIND>, grid, dim3(64 * kWaves), 0, stream, qw, ldw, wz, ldwz, N, G, alternate, out)
    if (wz) MQ_EX(kExpandU4);
    else if (layout == 2) MQ_EX(kExpandI4x16);
    else MQ_EX(kExpandI4);
#undef MQ_EX
    return launch_status("expand_weight_w4");
}

int launch_tile_weight_i8(const uint8_t* w, int64_t ldw, int64_t N, int64_t K, uint8_t* out, hipStream_t stream) {
    const int64_t units = (N + 15) / 16 * 16 * (K / 16);
    const int64_t blocks = std::min<int64_t>((units + 255) / 256, 65536);
    hipLaunchKernelGGL(tile16_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, w, ldw, N, K, out);
    return launch_status("tile_weight_i8");
}

int launch_quantize_weight(const void* w, int dtype, int64_t N, int64_t K, int64_t ldw, int hblock, int format,
                           void* q, int64_t ldq, void* scale, int64_t ld_scale, void* zero, int64_t ld_zero,
                           int* nonfinite, hipStream_t st) {
    switch (dtype) {
        case 0: return launch_dt<0>(w, ldw, N, K, hblock, format, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, st);
        case 1: return launch_dt<1>(w, ldw, N, K, hblock, format, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, st);
        case 2: return launch_dt<2>(w, ldw, N, K, hblock, format, q, ldq, scale, ld_scale, zero, ld_zero, nonfinite, st);
        default: break;
    }
    set_error("quantize_weight: unknown dtype %d", dtype);
    return -1;
}

}  // namespace mq
