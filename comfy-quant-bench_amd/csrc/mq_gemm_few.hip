// Quantized GEMM for a few activation rows (5 <= M <= 128, or fewer that are too long for the GEMV's LDS: a
// text prompt's tokens, a small batch of modulation vectors) with the scaled epilogues, GroupScale and
// RowScale.
//
// What bounds it: at these sizes the product is a read of the weights (4.7 MB packed at
// N = K = 3072) with far too few output tiles to fill 256 compute units, so the work is split along
// K inside the workgroup instead of over large output tiles: a workgroup owns 16 CB output columns
// and all rows (up to 16 MB of them), its W waves take contiguous slices of K, and the W partial
// sums of every output are added in LDS in wave order (deterministic; for RowScale exact int32 sums).
// Nothing is staged through LDS before that: the weights stream from HBM straight into registers,
// every byte once, and the activation codes, which all workgroups share and the L2 holds, are read
// as MFMA fragments (in the 16-row tile layout the whole linears write, a fragment is one
// contiguous 1 KB load).
//
// K is walked in spans of two 64-column groups. A packed weight row's span is 64 bytes: lane quad
// q (lanes 16 q .. 16 q + 15) of a column loads bytes 16 q .. 16 q + 15, and two
// v_permlane32_swap turn the quads' halves into one register pair per group: quads 0 to 3 then hold
// the group's 16-column chunks 0, 2, 1, 3, the order in which the activation fragments are read.
// int8 weights (rows, or 16-row tiles) are one 16-byte load per group and quad in natural order.
//
// Measured, whole linears (rotate + quantize included), against the 128 x 128-tile kernels these rows
// ran on before (one 4-wave workgroup per 128 columns; 16-row int8 tiles on the wide kernel's 128
// tile), us: W4A4 77 x 3072 x 3072 72.6 -> 11.0; W4A8 16 x 18432 x 3072 66.6 -> 15.5 and 77 x 3072 x
// 12288 254.9 -> 27.9; W8A8 8 x 3072 x 3072 15.9 -> 7.4 and 77 x 3072 x 12288 51.2 -> 25.6. Large W8A8
// products stay on the wide kernel (gemm_runs_few).
//
// The per-group scale step is the exact one: int32 partial, converted, one fp32 fma. The VALU is
// idle at these sizes (it is the loads' latency that counts), so nothing is gained by the wide
// kernel's seeded accumulators here. Signed int4 weights enter as 16 * v (two masks per dword), the
// activation layout 16 * q comes negated in odd groups: both factors are powers of two and leave
// through the group scale (or an exact shift of the int32 sum).
#include "mq_device.h"
#include "mq_internal.h"

namespace mq {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// 8 packed 4-bit weights (one dword) -> 8 int8 operands in k order. uint4: q - z, four bytes at a
// time ((v + (0x80 - z)) ^ 0x80, c holds 0x80 - z per byte); signed int4: 16 * v.
template <WKind WK>
__device__ __forceinline__ void unpack(uint32_t w, uint32_t c, int& o0, int& o1) {
    uint32_t lo, hi;
    if constexpr (WK == WKind::U4Asym) {
        lo = ((w & 0x0f0f0f0fu) + c) ^ 0x80808080u;
        hi = (((w >> 4) & 0x0f0f0f0fu) + c) ^ 0x80808080u;
    } else {
        lo = (w << 4) & 0xf0f0f0f0u;
        hi = w & 0xf0f0f0f0u;
    }
    o0 = static_cast<int>(__builtin_amdgcn_perm(hi, lo, 0x05010400u));
    o1 = static_cast<int>(__builtin_amdgcn_perm(hi, lo, 0x07030602u));
}

// MB blocks of 16 rows, CB blocks of 16 columns, W waves.
template <WKind WK, Epi EPI, int MB, int CB, int W>
__global__ void __launch_bounds__(64 * W) gemm_few_kernel(GemmArgs a) {
    static_assert(EPI == Epi::GroupScale || EPI == Epi::RowScale, "scaled epilogues");
    constexpr bool kPacked = WK != WKind::I8;
    constexpr bool kGroup = EPI == Epi::GroupScale;
    __shared__ v4i red[W * MB * CB * 64];
    __shared__ float row_s[16 * MB], col_b[16 * CB], col_s[16 * CB];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * (16 * CB);
    const int M = static_cast<int>(a.M);
    const int G = static_cast<int>(a.K / 64), S = (G + 1) / 2;
    // this wave's spans
    const int per = (S + W - 1) / W;
    const int s_begin = min(wave * per, S), s_end = min(s_begin + per, S);

    // The epilogue's inputs (row scales; column scales and bias), loaded ahead of everything else.
    static_assert(16 * MB + 16 * CB <= 64 * W, "one thread per row and column");
    float e_s = 0.0f, e_b = 0.0f;
    if (tid < 16 * MB) {
        if (tid < M) e_s = a.sa[tid];
    } else if (tid < 16 * MB + 16 * CB) {
        const int64_t n = n0 + (tid - 16 * MB);
        if (n < a.N) {
            if constexpr (!kGroup) e_s = a.ws32[n];
            if (a.bias) e_b = load_as_f32(a.bias, a.bias_dtype, n);
        }
    }

    // Every load is from an address inside its operand: columns past N read column N - 1, rows past M
    // row M - 1 (of the tile layout: the rows its last band holds), and the half span past an odd
    // number of groups the row's last group. What they bring is not used: such outputs are not
    // stored, such groups not multiplied. Addresses are a wave-uniform base and a 32-bit lane offset
    // (gemm_runs_few bounds the strides).
    uint32_t woff[CB], zoff[CB], soff[CB], aoff[MB];
    const uint8_t* wbase = a.qw;
    if (kPacked || !a.wtile) wbase += n0 * a.ldw;
    else wbase += (n0 >> 4) * G * 1024;
    const uint8_t* zbase = WK == WKind::U4Asym ? a.wz + n0 * a.ldwz : nullptr;
    const uint16_t* sbase = kGroup ? a.ws16 + n0 * a.ldws : nullptr;
    const int last_c = a.N - n0 < 16 * CB ? static_cast<int>(a.N - n0) - 1 : 16 * CB - 1;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        const uint32_t c = min(16 * cb + fr, last_c);
        if (kPacked || !a.wtile) woff[cb] = c * static_cast<uint32_t>(a.ldw) + fq * 16;
        else woff[cb] = (c >> 4) * G * 1024 + (c & 15) * 64 + fq * 16;
        zoff[cb] = WK == WKind::U4Asym ? c * static_cast<uint32_t>(a.ldwz) : 0u;
        soff[cb] = kGroup ? c * static_cast<uint32_t>(a.ldws) : 0u;
    }
    const int wstep = a.wtile ? 1024 : 64;   // int8: bytes from one group to the next
    const int ac = kPacked ? (fq & 1) * 2 + (fq >> 1) : fq;   // 16-column chunk of the group this quad multiplies
#pragma unroll
    for (int i = 0; i < MB; ++i)
        aoff[i] = (a.atile ? min(i, (M - 1) >> 4) * G * 1024 + fr * 64
                           : static_cast<uint32_t>(min(16 * i + fr, M - 1)) * static_cast<uint32_t>(a.lda)) + ac * 16;
    const int astep = a.atile ? 1024 : 64;

    // Scales and zero-points of four spans at a time: quad q of a column loads those of span s4 + q (one
    // dword of two fp16 scales, one byte of two zero-points), and span s4 + u's are read from quad u
    // when it is multiplied. A load per span and column would touch the same 16 cache lines four
    // times over and occupied the address unit longer than the weights do (M = 16, N = 18432,
    // K = 3072: 23.1 -> 17.8 us for the linear).
    const bool s_pair = (a.ldws & 1) == 0 && (reinterpret_cast<uintptr_t>(a.ws16) & 3) == 0 && 2 * S == G;
    uint32_t sq[2][CB], zq[2][CB];
    auto load_sz = [&](int set, int s4) {
        const uint32_t s = min(s4 + fq, s_end - 1);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            if constexpr (WK == WKind::U4Asym) zq[set][cb] = zbase[zoff[cb] + s];
            // (the pair past an odd number of groups: the row's last scale again)
            const uint32_t o = soff[cb] + 2 * s;
            if (s_pair) sq[set][cb] = *reinterpret_cast<const uint32_t*>(sbase + o);
            else sq[set][cb] = sbase[o] | static_cast<uint32_t>(sbase[min(o + 1, soff[cb] + G - 1)]) << 16;
        }
    };
    v4i wb[CB][kPacked ? 1 : 2], fa[2][MB];
    auto load = [&](int s) {
        const int g0 = 2 * s, g1 = min(2 * s + 1, G - 1);
        const uint32_t back = kPacked && g0 == g1 && fq >= 2 ? 32u : 0u;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            if constexpr (kPacked) {
                wb[cb][0] = *reinterpret_cast<const v4i*>(wbase + 64 * s + (woff[cb] - back));
            } else {
                wb[cb][0] = *reinterpret_cast<const v4i*>(wbase + g0 * wstep + woff[cb]);
                wb[cb][1] = *reinterpret_cast<const v4i*>(wbase + g1 * wstep + woff[cb]);
            }
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            fa[0][i] = *reinterpret_cast<const v4i*>(a.qa + g0 * astep + aoff[i]);
            fa[1][i] = *reinterpret_cast<const v4i*>(a.qa + g1 * astep + aoff[i]);
        }
    };

    f4 acc[MB][CB];
    v4i acci[MB][CB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            acc[i][cb] = f4{0.0f, 0.0f, 0.0f, 0.0f};
            acci[i][cb] = v4i{0, 0, 0, 0};
        }

    if (s_begin < s_end) {
        if constexpr (kGroup) load_sz(0, s_begin);
        load(s_begin);
    }
    for (int s0 = s_begin; s0 < s_end; s0 += 8) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int s = s0 + t, set = t >> 2;
            if (s >= s_end) break;
            if constexpr (kGroup)
                if ((t & 3) == 0 && s + 4 < s_end) load_sz(set ^ 1, s + 4);
            v4i b[CB][2];
            float sc[CB][2];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                if constexpr (kGroup) {
                    const uint32_t sp = __builtin_amdgcn_ds_bpermute((16 * (t & 3) + fr) * 4, static_cast<int>(sq[set][cb]));
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        sc[cb][h] = f16_bits_to_f32(static_cast<uint16_t>(sp >> (16 * h)));
                        if constexpr (WK == WKind::I4Sym) sc[cb][h] *= 0.0625f;
                        if (a.act_mode == 2) sc[cb][h] *= h ? -0.0625f : 0.0625f;
                    }
                }
                if constexpr (kPacked) {
                    const v4i w = wb[cb][0];
                    const auto p = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
                    const auto q = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
                    uint32_t z = 0u;
                    if constexpr (WK == WKind::U4Asym)
                        z = __builtin_amdgcn_ds_bpermute((16 * (t & 3) + fr) * 4, static_cast<int>(zq[set][cb]));
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint32_t c = 0x80808080u - ((z >> (4 * h)) & 0xfu) * 0x01010101u;
                        int o[4];
                        unpack<WK>(p[h], c, o[0], o[1]);
                        unpack<WK>(q[h], c, o[2], o[3]);
                        b[cb][h] = v4i{o[0], o[1], o[2], o[3]};
                    }
                } else {
                    b[cb][0] = wb[cb][0];
                    b[cb][1] = wb[cb][1];
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (2 * s + h >= G) break;   // an odd number of groups: nothing in the last half
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) {
                        if constexpr (kGroup) {
                            const v4i p = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[h][i], b[cb][h], v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                acc[i][cb][r] = __builtin_fmaf(static_cast<float>(p[r]), sc[cb][h], acc[i][cb][r]);
                        } else {
                            acci[i][cb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[h][i], b[cb][h], acci[i][cb], 0, 0, 0);
                        }
                    }
            }
            if (s + 1 < s_end) load(s + 1);
        }
    }

    // Each wave's sums, a lane's four rows as one 16-byte word (conflict-free), then the W sums of
    // every output in wave order.
    if (tid < 16 * MB) {
        row_s[tid] = e_s;
    } else if (tid < 16 * MB + 16 * CB) {
        col_s[tid - 16 * MB] = e_s;
        col_b[tid - 16 * MB] = e_b;
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            red[(wave * MB * CB + i * CB + cb) * 64 + lane] = kGroup ? __builtin_bit_cast(v4i, acc[i][cb]) : acci[i][cb];
    __syncthreads();
    for (int idx = tid; idx < MB * CB * 64; idx += 64 * W) {
        const int blk = idx >> 6, ln = idx & 63;
        const int lc = (blk % CB) * 16 + (ln & 15);
        const int64_t col = n0 + lc;
        const int row0 = (blk / CB) * 16 + 4 * (ln >> 4);
        if (col >= a.N || row0 >= M) continue;
        f4 t = {0.0f, 0.0f, 0.0f, 0.0f};
        v4i ti = {0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const v4i v = red[w * MB * CB * 64 + idx];
            if constexpr (kGroup) t += __builtin_bit_cast(f4, v);
            else ti += v;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (row0 + r >= M) break;
            const float sa = row_s[row0 + r];
            float y;
            if constexpr (kGroup) y = t[r] * sa + col_b[lc];
            else y = static_cast<float>(WK == WKind::I4Sym ? ti[r] >> 4 : ti[r]) * sa * col_s[lc] + col_b[lc];   // >> 4: exact
            store_from_f32(a.y, a.y_dtype, (row0 + r) * a.ldy + col, y);
        }
    }
}

template <WKind WK, Epi EPI, int MB, int CB, int W>
int launch_few(const GemmArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL((gemm_few_kernel<WK, EPI, MB, CB, W>), dim3(static_cast<unsigned>((a.N + 16 * CB - 1) / (16 * CB))),
                       dim3(64 * W), 0, stream, a);
    return launch_status("gemm_few");
}

// Columns per workgroup, by what gives every compute unit a workgroup: 16 up to N = 4096 (one round
// of 8-wave workgroups, each wave the shortest slice of K), 32 above it, which halves the reads of
// the activations (row scale, M = 77, K = 3072, linears: N = 4608 15.3 -> 12.5 us, N = 8192 16.2 ->
// 13.4 us; N = 3072 10.7 -> 12.0 us, so not there). Row-scale products of 33-80 rows and N > 8192 take
// 64 columns and four waves (M = 77, N = 12288: 20.6 us with 32 columns, 16.7 us); the group-scale
// ones, whose scale step keeps the VALU busy, are no faster that way (22.4 and 24.2 us).
template <WKind WK, Epi EPI, int MB>
int launch_cols(const GemmArgs& a, hipStream_t stream) {
    const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
    const int64_t blocks = (a.N + 15) / 16;
    if (blocks <= cus) return launch_few<WK, EPI, MB, 1, 8>(a, stream);
    if constexpr (EPI == Epi::RowScale && MB >= 3 && MB <= 5)
        if (blocks > 2 * cus) return launch_few<WK, EPI, MB, 4, 4>(a, stream);
    return launch_few<WK, EPI, MB, 2, 8>(a, stream);
}

template <WKind WK, Epi EPI>
int launch_rows(const GemmArgs& a, hipStream_t stream) {
    switch ((a.M + 15) / 16) {
        case 1: return launch_cols<WK, EPI, 1>(a, stream);
        case 2: return launch_cols<WK, EPI, 2>(a, stream);
        case 3: return launch_cols<WK, EPI, 3>(a, stream);
        case 4: return launch_cols<WK, EPI, 4>(a, stream);
        case 5: return launch_cols<WK, EPI, 5>(a, stream);
        case 6: return launch_cols<WK, EPI, 6>(a, stream);
        default: return launch_cols<WK, EPI, 8>(a, stream);
    }
}

}  // namespace

int launch_gemm_few(const GemmArgs& a, WKind wk, Epi epi, hipStream_t stream) {
    if (epi == Epi::GroupScale && wk == WKind::U4Asym) return launch_rows<WKind::U4Asym, Epi::GroupScale>(a, stream);
    if (epi == Epi::GroupScale && wk == WKind::I4Sym) return launch_rows<WKind::I4Sym, Epi::GroupScale>(a, stream);
    if (epi == Epi::RowScale && wk == WKind::I4Sym) return launch_rows<WKind::I4Sym, Epi::RowScale>(a, stream);
    if (epi == Epi::RowScale && wk == WKind::I8) return launch_rows<WKind::I8, Epi::RowScale>(a, stream);
    set_error("gemm_few: unsupported weight kind / epilogue combination");
    return -2;
}

}  // namespace mq
