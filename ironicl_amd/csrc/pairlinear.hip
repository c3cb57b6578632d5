// 512- and 1,024-deep products of the ICL stage on FP16 pairs (common.hpp):
// out = epilogue(A W^T + b), A either rows as they are (attention outputs, the
// FFN's hidden layer, normalized rows) or 512-wide rows LayerNormed in the
// prologue (the FFN's first product, the decoder's).
//
// A workgroup of four waves takes 16 RG rows x 64 CB columns. Its waves first load
// the rows (a wave per 4 RG rows, every load in flight at once), LayerNorm
// them or find each row's scale, and leave them in LDS as pairs in operand
// order; then wave w runs its CB blocks of 16 columns over the whole depth on
// v_mfma_f32_16x16x32_f16, the weights as the A operand, straight from their
// packed fragments in L2 four steps ahead. In the result, lane (m, g) =
// (lane % 16, lane / 16) holds row m's columns 4 g .. 4 g + 3, one 16-byte store.
// hi.hi products and the two small ones go to separate accumulators, so two
// chains run per row group.
//
// Scales: each row of a weight matrix by a power of two set when it is packed
// (an output's error is then that of its own terms), LayerNormed
// rows by one from the LayerNorm's weights (a value is at most sqrt(512) times
// the largest weight plus the largest bias), other rows each by its largest.
//
// Workgroups take their tiles XCD by XCD, columns fastest: a band of rows is
// read into one L2 and the weights (at most 4 MB as pairs) stay there.
#include "common.hpp"

#include <algorithm>
#include <cmath>

namespace irx {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kAhead = 4;  // weight fragments in flight, in 32-deep steps

template <int K, int RG, int CB, int EPI, bool LN>
__global__ __launch_bounds__(256) void pair_linear_kernel(PairLinear p, int col_groups, int per_xcd, int count) {
    constexpr int ROWS = 16 * RG, STRIDE = K / 2 + 4;  // words per LDS row: K halves and 16 bytes of padding
    constexpr int S = K / 512, STEPS = K / 32;
    __shared__ __attribute__((aligned(16))) float hi[ROWS * STRIDE], lo[ROWS * STRIDE];
    __shared__ float row_inv[ROWS];
    const int t = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (t >= count) return;
    const int cg = t % col_groups;
    const long long row0 = (long long)(t / col_groups) * ROWS;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, g = lane >> 4;

    // This wave's weight fragments, the first steps' in flight over the prologue.
    const float *pk = p.w.pack + (size_t)(cg * 4 + w) * CB * STEPS * 512 + lane * 4;
    u32x4 wh[kAhead], wl[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        wh[i] = *reinterpret_cast<const u32x4 *>(pk + i * 512);
        wl[i] = *reinterpret_cast<const u32x4 *>(pk + i * 512 + 256);
    }

    // Rows 4 RG w + i: lane (kb, gl) = (lane / 4, lane % 4) takes slots e of
    // k-blocks kb + 16 s, column 32 (kb + 16 s) + 16 (e / 4) + 4 gl + e % 4.
    {
        const int kb = lane >> 2, gl = lane & 3;
        f32x4 x[4 * RG][S][2];
#pragma unroll
        for (int i = 0; i < 4 * RG; ++i) {
            const long long r = min(row0 + 4 * RG * w + i, (long long)p.m - 1);
            const float *src = p.x + r * p.ldx + 32 * kb + 4 * gl;
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int h = 0; h < 2; ++h) x[i][s][h] = *reinterpret_cast<const f32x4 *>(src + 512 * s + 16 * h);
        }
        f32x4 lw[2], lb[2];
        if constexpr (LN) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                lw[h] = *reinterpret_cast<const f32x4 *>(p.lnw + 32 * kb + 16 * h + 4 * gl);
                lb[h] = *reinterpret_cast<const f32x4 *>(p.lnb + 32 * kb + 16 * h + 4 * gl);
            }
        }
#pragma unroll
        for (int i = 0; i < 4 * RG; ++i) {
            float scale;
            if constexpr (LN) {
                const f32x4 a = x[i][0][0] + x[i][0][1];
                const float mean = wave_sum((a[0] + a[1]) + (a[2] + a[3])) / (float)K;
                float sq = 0.f;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        x[i][0][h][e] -= mean;
                        sq = fmaf(x[i][0][h][e], x[i][0][h][e], sq);
                    }
                const float rstd = 1.0f / sqrtf(wave_sum(sq) / (float)K + 1e-5f);
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[i][0][h][e] = x[i][0][h][e] * rstd * lw[h][e] + lb[h][e];
                scale = p.w.ln_scale;
            } else {
                float m = 0.f;
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(x[i][s][h][e]));
                const int ex = pair_exponent(wave_max(m));
                scale = pow2(ex);
                if (lane == 0) row_inv[4 * RG * w + i] = pow2(-ex);
            }
#pragma unroll
            for (int s = 0; s < S; ++s) {
                float y[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = x[i][s][e >> 2][e & 3] * scale;
                half8 h, l;
                pair8(y, h, l);
                const int at = (4 * RG * w + i) * STRIDE + ((kb + 16 * s) * 4 + gl) * 4;
                *reinterpret_cast<half8 *>(&hi[at]) = h;
                *reinterpret_cast<half8 *>(&lo[at]) = l;
            }
        }
    }
    __syncthreads();

#pragma unroll 1
    for (int cb = 0; cb < CB; ++cb, pk += STEPS * 512) {
        f32x4 big[RG], small[RG];
#pragma unroll
        for (int r = 0; r < RG; ++r) big[r] = small[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < STEPS; ++kb) {
            const half8 ah = as_half8(wh[kb % kAhead]), al = as_half8(wl[kb % kAhead]);
            half8 bh[RG], bl[RG];
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                const int at = (16 * r + m16) * STRIDE + (kb * 4 + g) * 4;
                bh[r] = *reinterpret_cast<const half8 *>(&hi[at]);
                bl[r] = *reinterpret_cast<const half8 *>(&lo[at]);
            }
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                small[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh[r], small[r], 0, 0, 0);
                big[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bh[r], big[r], 0, 0, 0);
                small[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl[r], small[r], 0, 0, 0);
            }
            if (kb + kAhead < STEPS || cb + 1 < CB) {
                wh[kb % kAhead] = *reinterpret_cast<const u32x4 *>(pk + (kb + kAhead) * 512);
                wl[kb % kAhead] = *reinterpret_cast<const u32x4 *>(pk + (kb + kAhead) * 512 + 256);
            }
            __builtin_amdgcn_sched_barrier(0);  // keeps each load this far ahead of its use
        }

        const int col = 64 * CB * cg + 16 * (CB * w + cb) + 4 * g;
        const f32x4 bias = *reinterpret_cast<const f32x4 *>(p.bias + col);
        const f32x4 w_inv = *reinterpret_cast<const f32x4 *>(p.w.row_inv + col);
        const OutMap &o = p.out;
        const int seg = col / o.col_seg, plane = seg / o.heads, head = seg - plane * o.heads;
        const long long coff = plane * o.plane_stride + head * o.head_stride + (col - seg * o.col_seg);
#pragma unroll
        for (int r = 0; r < RG; ++r) {
            const long long row = row0 + 16 * r + m16;
            if (row >= p.m) continue;
            const float inv = LN ? p.w.ln_inv : row_inv[16 * r + m16];
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = fmaf((big[r][e] + small[r][e]) * w_inv[e], inv, bias[e]);
                if constexpr (EPI == kEpiGelu) v[e] = gelu_erf(v[e]);
            }
            if constexpr (EPI == kEpiResidual) v += *reinterpret_cast<const f32x4 *>(p.residual + row * p.ldr + col);
            const long long grp = row / o.rows_per_group;
            *reinterpret_cast<f32x4 *>(p.c + grp * o.group_stride + (row - grp * o.rows_per_group) * o.ldc + coff) = v;
        }
    }
}

// A thread per (16-column block, 32-deep step, lane) of a [n, k] matrix: the
// lane's eight values, hi then (1 KB further) lo parts.
__global__ __launch_bounds__(256) void pair_pack_kernel(const float *w, int k, long long lanes, const float *row_inv,
                                                        float *out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= lanes) return;
    const int lane = (int)(i & 63), steps = k / 32;
    const long long frag = i >> 6, cb = frag / steps;
    const float *src = w + (cb * 16 + (lane & 15)) * k + (frag - cb * steps) * 32 + 4 * (lane >> 4);
    const f32x4 a = *reinterpret_cast<const f32x4 *>(src), b = *reinterpret_cast<const f32x4 *>(src + 16);
    const float scale = 1.0f / row_inv[cb * 16 + (lane & 15)];
    float y[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = a[e] * scale, y[4 + e] = b[e] * scale;
    half8 h, l;
    pair8(y, h, l);
    *reinterpret_cast<half8 *>(out + frag * 512 + lane * 4) = h;
    *reinterpret_cast<half8 *>(out + frag * 512 + 256 + lane * 4) = l;
}

// A wave per row: the inverse of the power of two that brings the row's
// largest magnitude into [2^13, 2^14) (1 for zeros).
__global__ __launch_bounds__(256) void pair_rows_kernel(const float *w, int n, int k, float *row_inv) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    float m = 0.f;
    for (int i = lane; i < k; i += 64) m = fmaxf(m, fabsf(w[(long long)row * k + i]));
    m = wave_max(m);
    const int e = m > 0.f ? pair_exponent(m) : 0;
    if (lane == 0) row_inv[row] = pow2(-e);
}

float largest_magnitude(const float *w, size_t count) {
    unsigned largest = 0;
    for (size_t i = 0; i < count; ++i) {
        const unsigned bits = __builtin_bit_cast(unsigned, w[i]) & 0x7fffffffu;
        largest = std::max(largest, bits);
    }
    return __builtin_bit_cast(float, largest);
}

}  // namespace

int pair_scale_exponent(double largest, int top) {
    if (!(largest > 0.0)) return 0;
    return std::max(-126, std::min(126, top - 1 - std::ilogb(largest)));
}

PairW pair_pack(const float *w, int n, int k, const float *lnw, const float *lnb, float *out, hipStream_t stream) {
    if (n % 16 || k % 512) fail(3, "pair_pack: unsupported shape");
    float *row_inv = out + (size_t)n * k;
    PairW p;
    p.pack = out, p.row_inv = row_inv;
    if (lnw) {
        const int el = pair_scale_exponent(22.7 * largest_magnitude(lnw, k) + largest_magnitude(lnb, k), 15);
        p.ln_scale = std::ldexp(1.f, el), p.ln_inv = std::ldexp(1.f, -el);
    }
    const long long lanes = (long long)n / 16 * (k / 32) * 64;
    hipLaunchKernelGGL(pair_rows_kernel, dim3(ceil_div((size_t)n, 4)), dim3(256), 0, stream, w, n, k, row_inv);
    hipLaunchKernelGGL(pair_pack_kernel, dim3((unsigned)ceil_div(lanes, 256LL)), dim3(256), 0, stream, w, k, lanes,
                       row_inv, out);
    IRX_HIP(hipGetLastError());
    return p;
}

void pair_linear(const PairLinear &a, hipStream_t stream) {
    if (a.m <= 0) return;
    const bool ln = a.lnw != nullptr;
    auto aligned = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (!a.x || !a.c || !a.w.pack || !a.w.row_inv || !a.bias || a.n % 64 || (a.k != 512 && a.k != 1024) || (ln && (a.k != 512 || !a.lnb)) ||
        (a.epilogue == kEpiResidual && !a.residual) || a.out.col_seg % 4)
        fail(3, "pair_linear: unsupported arguments");
    if ((a.ldx & 3) || (a.ldr & 3) || (a.out.ldc & 3) || (a.out.head_stride & 3) || (a.out.plane_stride & 3) ||
        (a.out.group_stride & 3) || !aligned(a.x) || !aligned(a.c) || !aligned(a.w.pack) || !aligned(a.w.row_inv) || !aligned(a.bias) ||
        !aligned(a.residual) || !aligned(a.lnw) || !aligned(a.lnb))
        fail(3, "pair_linear: rows must be 16-byte aligned");
    const double m = a.m, n = a.n, k = a.k;
    KernelTimer timer(kFamGemm, stream, 2.0 * m * n * k,
                      4.0 * (m * k + n * k + m * n + (a.epilogue == kEpiResidual ? m * n : 0.0)));
    // 32 rows a workgroup once that fills the chip (half the weight reads of
    // 16; at depth 1,024 the rows' pairs take the LDS of 16), and 256 columns
    // rather than 64 once that leaves two workgroups a CU: the prologue, several
    // times a 64-column product's time, is then paid by a fourth of them.
    // Repeated launches alone, us, of 512 -> 1,024 with LayerNorm: 16 / 32 rows at
    // 512 rows (256 workgroups) 9.2 / 11.0, at 1,000 13.5 / 13.7, at 8,192 62.8 /
    // 49.9; 64 / 256 columns at 1,000 rows (128 workgroups of 256) 13.7 / 18.6, at
    // 2,048 (256) 23.9 / 20.2, at 4,096 (512) 44.2 / 26.8. Lines one doubling
    // higher for the rows and lower for the columns look better by these, but in
    // place, beside another stream or on weights not yet in L2, they lose: 1,024 rows
    // against 10,000 x 100 at auto 2,228 us here and 2,334 so, a 2,048-row build 3.52
    // and 3.62 ms (3,000 rows 4.63 and 4.56).
    const long long cus = std::max(1, a.compute_units);
    const int rg = a.k == 512 && (long long)ceil_div(a.m, 32) * (a.n / 64) >= cus ? 2 : 1;
    const long long groups = ceil_div(a.m, 16 * rg);
    const bool wide = (rg == 2 || a.k == 1024) && a.n % 256 == 0 && groups * (a.n / 256) >= 2 * cus;
    const int cgs = a.n / (wide ? 256 : 64);
    const long long count = groups * cgs, per_xcd = (count + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffLL) fail(3, "pair_linear: too many rows");
    auto go = [&]<int K, int RG, int CB, bool LN>() {
        const dim3 grid((unsigned)(per_xcd * 8)), block(256);
        if (a.epilogue == kEpiNone)
            hipLaunchKernelGGL((pair_linear_kernel<K, RG, CB, kEpiNone, LN>), grid, block, 0, stream, a, cgs, (int)per_xcd, (int)count);
        else if (a.epilogue == kEpiGelu)
            hipLaunchKernelGGL((pair_linear_kernel<K, RG, CB, kEpiGelu, LN>), grid, block, 0, stream, a, cgs, (int)per_xcd, (int)count);
        else
            hipLaunchKernelGGL((pair_linear_kernel<K, RG, CB, kEpiResidual, LN>), grid, block, 0, stream, a, cgs, (int)per_xcd, (int)count);
        IRX_HIP(hipGetLastError());
    };
    auto width = [&]<int K, int RG, bool LN>() {
        if (wide)
            go.template operator()<K, RG, 4, LN>();
        else
            go.template operator()<K, RG, 1, LN>();
    };
    if (a.k == 1024)
        width.template operator()<1024, 1, false>();
    else if (ln && rg == 2)
        width.template operator()<512, 2, true>();
    else if (ln)
        go.template operator()<512, 1, 1, true>();
    else if (rg == 2)
        width.template operator()<512, 2, false>();
    else
        go.template operator()<512, 1, 1, false>();
}

}  // namespace irx
