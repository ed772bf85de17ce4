// Load-time decode of comfy-kitchen's shipped asym_w4a8_int8 weights (4-bit codebook indices,
// fp8 e4m3fn per-group scales s_rel, per-row s_channel) to an int8 weight whose per-row scale is
// the stored s_channel, the form the int8 row-scale GEMM takes. comfy-kitchen finishes a decoded
// W4A8 weight as dequantize_int8_convrot_weight_dtype(int8_weight, s_channel, ...)
// (patches/comfy_kitchen_w4a8_dequant_fused.patch:15-18): the int8 weight's row scale is s_channel
// unchanged, so level * s_rel is already in int8 units and
//
//   t[n,k]  = fp32(level(code[n,k]) * fp8(s_rel[n, k / gs]))   level = codebook[code], or the
//                                                               signed nibble without a codebook
//   q8[n,k] = clamp(rne(t[n,k]), -127, 127)                     (0 where t is NaN)
//   row_scale[n] = s_channel[n]
//
// The output is rows [N, ldq8], or the int8 GEMM's 16-row tiles [ceil(N / 16)][K / 64][16][64]
// (MQ_W8_TILE16), so that a loader that keeps the tiles writes them at once instead of writing rows and
// tiling them in a second pass. A thread makes 16 consecutive k of one row (8 packed bytes in, 16
// bytes out; one scale where the group is 16 or more), a wavefront one tile, or 1024 columns of a row.
//
// What bounds it: HBM, 1.5 bytes per weight and the scales. N = 12288, K = 3072 to tiles (59 MB at group 16),
// calls back to back: 15.4-15.6 us a call at groups of 16, 32, 48, 64 and 128 (16.4 with an integer
// division per lane for the group index, GroupIndex below); to rows 16.1-16.4 (17.3). (One workgroup per row,
// eight k per thread step with an integer division and a scale byte load per weight, took 47.1 us to
// rows, and the tiling pass 11.6 more.)
#include <algorithm>

#include "mq_device.h"
#include "mq_internal.h"

#pragma clang fp contract(off)

namespace mq {
namespace {

constexpr int kWaves = 4;   // wavefronts per workgroup

// OCP fp8 e4m3fn -> fp32, exact (bias 7; e = 0 subnormal; S.1111.111 NaN, no infinities).
__device__ __forceinline__ float fp8_e4m3fn(uint32_t b) {
    const uint32_t e = (b >> 3) & 0xfu, m = b & 7u;
    float v;
    if (e == 0) v = static_cast<float>(m) * 0x1p-9f;
    else v = __uint_as_float(((e + 120u) << 23) | (m << 20));
    if (e == 0xfu && m == 7u) v = __builtin_nanf("");
    return (b & 0x80u) ? -v : v;
}

// k / gs for a column k that is a multiple of 16 and a group size of 16 d, without a division (gs is a
// run-time value, and an integer division a dozen instructions a lane): with u = k / 16 < 2^26,
// l = ceil(log2 d) and m = ceil(2^(26 + l) / d) = (2^(26 + l) + e) / d, e < d <= 2^l, the excess of
// u m / 2^(26 + l) over u / d is u e / (d 2^(26 + l)) < 1 / d, so its floor is u / d's. As one high product:
// (2 u) (32 m) / 2^32 = u m / 2^26, and m < 2^27 keeps 32 m in 32 bits (d < 2^26). The same work for every gs.
struct GroupIndex {
    uint32_t mul;
    int shift;
    __device__ __forceinline__ uint32_t operator()(int k) const {
        return __umulhi(static_cast<uint32_t>(k) >> 3, mul) >> shift;
    }
};
GroupIndex group_index(int gs) {
    const uint64_t d = static_cast<uint64_t>(std::max(gs / 16, 1));   // (groups under 16 are not indexed this way)
    int l = 0;
    while ((uint64_t(1) << l) < d) ++l;
    return {static_cast<uint32_t>(((uint64_t(1) << (26 + l)) + d - 1) / d) << 5, l};
}

// Units of 64 threads (one wavefront): tile t = band * (K / 64) + g, lane = (row, 16-column chunk); or,
// to rows, the part'th 1024 columns of a row. SPU: scales per 16 columns (1: group_size >= 16).
template <bool TILE, int SPU>
__global__ void __launch_bounds__(64 * kWaves)
decode_kernel(const uint8_t* __restrict__ qdata, int64_t ldq, const uint8_t* __restrict__ s_rel, int64_t lds,
              const float* __restrict__ s_channel, const float* __restrict__ codebook, GroupIndex group, int64_t N, int K,
              int8_t* __restrict__ q8, int64_t ldq8, float* __restrict__ row_scale) {
    __shared__ float lev[16];
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < 16) lev[tid] = codebook ? codebook[tid] : static_cast<float>(tid >= 8 ? tid - 16 : tid);
    __syncthreads();
    const uint32_t per = TILE ? K / 64 : (K + 1023) / 1024;   // units per band of 16 rows, or per row
    const int64_t units = (TILE ? (N + 15) / 16 : N) * per;
    const bool q_wide = ldq % 8 == 0 && reinterpret_cast<uintptr_t>(qdata) % 8 == 0;
    const bool o_wide = TILE || (ldq8 % 16 == 0 && reinterpret_cast<uintptr_t>(q8) % 16 == 0);
    for (int64_t u = static_cast<int64_t>(blockIdx.x) * kWaves + __builtin_amdgcn_readfirstlane(tid >> 6); u < units;
         u += static_cast<int64_t>(gridDim.x) * kWaves) {
        const int64_t major = u / per;
        const int part = static_cast<int>(u - major * per);
        const int64_t n = TILE ? major * 16 + (lane >> 2) : major;
        const int k = TILE ? part * 64 + (lane & 3) * 16 : part * 1024 + lane * 16;
        if (!TILE && k >= K) continue;
        uint32_t out[4] = {0u, 0u, 0u, 0u};
        if (n < N) {
            const uint8_t* qp = qdata + n * ldq + k / 2;
            uint32_t w[2];
            if (q_wide) {
                const uint2 v = *reinterpret_cast<const uint2*>(qp);
                w[0] = v.x;
                w[1] = v.y;
            } else {
                w[0] = *reinterpret_cast<const uint32_t*>(qp);
                w[1] = *reinterpret_cast<const uint32_t*>(qp + 4);
            }
            float s[SPU];
#pragma unroll
            for (int j = 0; j < SPU; ++j)
                s[j] = fp8_e4m3fn(s_rel[n * lds + (SPU > 1 ? k / (16 / SPU) + j : group(k))]);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float t = lev[(w[i >> 3] >> (4 * (i & 7))) & 0xfu] * s[i * SPU / 16];
                const float c = __builtin_fminf(__builtin_fmaxf(t, -127.0f), 127.0f) + kMagic;   // rne of the clamped t
                const uint32_t byte = t != t ? 0u : __float_as_uint(c) & 0xffu;
                out[i >> 2] |= byte << (8 * (i & 3));
            }
            if (TILE ? part == 0 && (lane & 3) == 0 : k == 0) row_scale[n] = s_channel[n];
        }
        int8_t* dst = TILE ? q8 + u * 1024 + lane * 16 : q8 + n * ldq8 + k;
        if (o_wide) {
            *reinterpret_cast<uint4*>(dst) = uint4{out[0], out[1], out[2], out[3]};
        } else {
            *reinterpret_cast<uint2*>(dst) = uint2{out[0], out[1]};
            *reinterpret_cast<uint2*>(dst + 8) = uint2{out[2], out[3]};
        }
    }
}

}  // namespace

int launch_decode_w4a8_codebook(const uint8_t* qdata, int64_t ldq, const uint8_t* s_rel, int64_t lds,
                                const float* s_channel, const float* codebook, int group_size, int64_t N,
                                int64_t K, int8_t* q8, int64_t ldq8, float* row_scale, bool tile, hipStream_t stream) {
    const int64_t units = tile ? (N + 15) / 16 * (K / 64) : N * ((K + 1023) / 1024);
    const dim3 grid(static_cast<unsigned>(std::min<int64_t>((units + kWaves - 1) / kWaves, int64_t(1) << 22)));
#define MQ_DC(TILE, SPU)                                                                                           \
    hipLaunchKernelGGL((decode_kernel<TILE, SPU>), grid, dim3(64 * kWaves), 0, stream, qdata, ldq, s_rel, lds,      \
                       s_channel, codebook, group_index(group_size), N, static_cast<int>(K), q8, ldq8, row_scale)
    if (group_size >= 16) {
        if (tile) MQ_DC(true, 1);
        else MQ_DC(false, 1);
    } else if (group_size == 8) {
        if (tile) MQ_DC(true, 2);
        else MQ_DC(false, 2);
    } else {   // 4
        if (tile) MQ_DC(true, 4);
        else MQ_DC(false, 4);
    }
#undef MQ_DC
    return launch_status("decode_w4a8_codebook");
}

}  // namespace mq
