// Fused tail of a 128-wide transformer block on gfx950 matrix cores.
//
// The post-attention half of every column and row block (cpu.rs:1555-1601):
//   s1    = state + (att Wo^T + bo)
//   state = s1 + (gelu(LN2(s1) W1^T + b1) W2^T + b2)
// as one kernel instead of four launches (out-projection, LayerNorm, FFN up,
// FFN down), so s1, LN2(s1) and the 256-wide hidden layer never leave
// registers.
//
// Each wave owns 16 rows for the whole chain. Products are computed
// transposed, D = W X^T, on v_mfma_f32_16x16x32_f16 with both operands as FP16
// pairs (common.hpp): the weights are the A operand and the rows the B
// operand. In D, lane (m, g) = (lane % 16, lane / 16) holds row m's features
// 16 b + 4 g + r in register r of block b. The next product's B operand, for
// the 32 features of blocks 2 kb and 2 kb + 1, is the lane's eight of them:
// slot e is feature 32 kb + 16 (e / 4) + 4 g + e % 4, and the A operand's slots
// are packed the same way, so the chain runs without moving data between
// lanes. The same per-lane layout is used to load att and state and to store
// the result.
//
// Scales. Each row of a weight matrix is packed times a power of two that
// brings its largest into [2^13, 2^14). LayerNormed rows are bounded by sqrt(128) times
// the weights' largest plus the biases', the hidden layer by its weights' row
// norms, so their scales are fixed when the weights are packed; attention
// outputs, which can come from an imported cache, are scaled by row.
//
// The weights are packed once (tail128_pack) into A-operand fragments, 1 KB
// per 16 x 32 block of hi or lo parts, lane after lane, in the order the kernel
// consumes them: ten 32 KB chunks (Wo in two, then per 32-unit slice of the
// hidden layer the W1 rows and W2 columns it touches). A workgroup streams
// each chunk as two 16 KB halves (an out-projection k-block, or a slice's W1
// rows then its W2 columns) through two 16 KB LDS buffers with direct global ->
// LDS loads, so
// three workgroups share a CU; every LDS read is one 16-byte read per lane
// of consecutive addresses (no bank conflicts).
#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace irx {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kChunkFloats = 8192;  // 32 KB: the packing unit
constexpr int kChunks = 10;
// Chunks stream through LDS in halves of 16 KB (two 16 KB buffers), so a
// workgroup takes 32 KB and three fit a CU.
constexpr int kHalfFloats = kChunkFloats / 2;
constexpr int kHalves = 2 * kChunks;
constexpr int kTailWaves = 4;
constexpr int kTailRows = 16 * kTailWaves;  // rows per workgroup

__device__ __forceinline__ void wait_vm() {
    // vmcnt(0); expcnt and lgkmcnt left at their maxima (no wait).
    __builtin_amdgcn_s_waitcnt(0x0F70);
}

__device__ __forceinline__ f32x4 mfma(float a, float b, const f32x4 &acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

// An operand of 32 k-slots as an FP16 pair.
struct Pair {
    half8 h, l;
};

// acc += W X over 32 k-slots for N output blocks, each accumulator's products
// in the same order in every kernel (the small-pass forms repeat the bits).
template <int N>
__device__ __forceinline__ void pair_mfma(const Pair (&w)[N], const Pair &x, f32x4 (&acc)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[i].l, x.h, acc[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[i].h, x.l, acc[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[i].h, x.h, acc[i], 0, 0, 0);
}

// The fragments (hi, then lo 1 KB further) at `f`, the lane's base.
__device__ __forceinline__ Pair pair_at(const float *f) {
    return {as_half8(*reinterpret_cast<const u32x4 *>(f)), as_half8(*reinterpret_cast<const u32x4 *>(f + 256))};
}

// acc[0..7] += eight output blocks' fragments at `frag` times x, four at a
// time (all eight in flight take registers the kernels need).
__device__ __forceinline__ void pair_blocks(const float *frag, const Pair &x, f32x4 *acc) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        Pair f[4];
        f32x4 a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = pair_at(frag + (4 * half + i) * 512), a[i] = acc[4 * half + i];
        pair_mfma<4>(f, x, a);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[4 * half + i] = a[i];
    }
}

// The lane's features of blocks 2 kb and 2 kb + 1, times `scale`.
__device__ __forceinline__ Pair pair_of(const f32x4 &a, const f32x4 &b, float scale) {
    float y[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = a[e] * scale, y[4 + e] = b[e] * scale;
    Pair p;
    pair8(y, p.h, p.l);
    return p;
}

// The exponent that brings the row's largest of x (over the row's four lanes)
// into [2^13, 2^14).
__device__ __forceinline__ int row_exponent(const f32x4 (&x)[8]) {
    float m = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(x[b][e]));
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    return pair_exponent(m);
}

// Words of scales after a pack's fragments. Tail: LN2's scale and the hidden
// layer's, then per output the inverse of its product's scale: out-projection
// (weights only: attention outputs are scaled by row), W1, W2. Head: LN1's
// scale, then per output the inverse.
constexpr size_t kTailScales = 10 * 8192;
enum { kTailLn = 0, kTailHid = 1, kTailOutInv = 16, kTailLnInv = kTailOutInv + 128, kTailHidInv = kTailLnInv + 256 };
enum { kHeadLn = 0, kHeadInv = 16 };
static_assert(kTailHidInv + 128 <= (int)kPackScales && kHeadInv + 384 <= (int)kPackScales);

__device__ __forceinline__ f32x4 lds4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

// The chain after a 128-wide block's attention (cpu.rs:1555-1601): x holds
// the row's attention output and s1 its state, in the per-wave layout above;
// the packed weights arrive as half-chunks h0 .. h0 + 19 from next(h), which
// returns the lane's base in the half's LDS buffer. The new state goes to
// out (the lane's first feature, 4 g) when the row is live.
template <class Next>
__device__ __forceinline__ void tail_chain(f32x4 (&x)[8], f32x4 (&s1)[8], Next &&next, int h0, const Tail128 &t,
                                           float *out, bool live, int g) {
    const float *sc = t.pack + kTailScales;
    f32x4 acc[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Out-projection: half-chunk hc holds 32-wide k-block hc's fragments of the
    // eight output blocks.
    const int ea = row_exponent(x);
    const float a_scale = pow2(ea), a_inv = pow2(-ea);
    Pair xp[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) xp[kb] = pair_of(x[2 * kb], x[2 * kb + 1], a_scale);
#pragma unroll
    for (int hc = 0; hc < 4; ++hc) {
        const float *frag = next(h0 + hc);
        pair_blocks(frag, xp[hc], acc);
    }

    // s1 = state + (acc + bo), then LN2 over the row's 128 features, held by
    // lanes m, m + 16, m + 32, m + 48.
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const f32x4 bo = *reinterpret_cast<const f32x4 *>(t.bo + 16 * b + 4 * g);
        const f32x4 wi = lds4(sc + kTailOutInv + 16 * b + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s1[b][e] = s1[b][e] + __builtin_fmaf(acc[b][e] * wi[e], a_inv, bo[e]);
            sum += s1[b][e];
        }
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float mean = sum / 128.f;
    float sq = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float d = s1[b][e] - mean;
            sq = fmaf(d, d, sq);
        }
    sq += __shfl_xor(sq, 16, 64);
    sq += __shfl_xor(sq, 32, 64);
    const float rstd = 1.0f / sqrtf(sq / 128.f + 1e-5f);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const f32x4 w = *reinterpret_cast<const f32x4 *>(t.n2w + 16 * b + 4 * g);
        const f32x4 bb = *reinterpret_cast<const f32x4 *>(t.n2b + 16 * b + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = (s1[b][e] - mean) * rstd * w[e] + bb[e];
        acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // FFN, 32 hidden units per slice c: h = gelu(W1 x + b1) for units 32 c +
    // 16 hb + 4 g + e from half-chunk 4 + 2 c (even and odd k-blocks in
    // separate accumulators, four independent chains), then acc += W2 h from
    // half-chunk 5 + 2 c.
    const float ln_scale = sc[kTailLn], hid_scale = sc[kTailHid];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) xp[kb] = pair_of(x[2 * kb], x[2 * kb + 1], ln_scale);
#pragma unroll 1
    for (int c = 0; c < 8; ++c) {
        const float *frag = next(h0 + 4 + 2 * c);
        f32x4 h[2][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const Pair f[2] = {pair_at(frag + (kb * 2) * 512), pair_at(frag + (kb * 2 + 1) * 512)};
            pair_mfma<2>(f, xp[kb], h[kb & 1]);
        }
        f32x4 hg[2];
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const f32x4 b1 = *reinterpret_cast<const f32x4 *>(t.b1 + 32 * c + 16 * hb + 4 * g);
            const f32x4 wi = lds4(sc + kTailLnInv + 32 * c + 16 * hb + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                hg[hb][e] = gelu_erf(__builtin_fmaf(h[0][hb][e] + h[1][hb][e], wi[e], b1[e]));
        }
        const Pair hp = pair_of(hg[0], hg[1], hid_scale);
        const float *frag2 = next(h0 + 5 + 2 * c);
        pair_blocks(frag2, hp, acc);
    }

    if (!live) return;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const f32x4 b2 = *reinterpret_cast<const f32x4 *>(t.b2 + 16 * b + 4 * g);
        const f32x4 wi = lds4(sc + kTailHidInv + 16 * b + 4 * g);
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(acc[b][e], wi[e], b2[e]) + s1[b][e];
        *reinterpret_cast<f32x4 *>(out + 16 * b) = v;
    }
}

__global__ __launch_bounds__(256, 3) void tail128_kernel(Tail128 p) {
    __shared__ __attribute__((aligned(16))) float buf[2][kHalfFloats];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, g = lane >> 4;
    const long long row = (long long)blockIdx.x * kTailRows + wv * 16 + m16;
    const bool live = row < p.m;
    const long long r = live ? row : p.m - 1;

    // Half-chunk hc (16 KB) goes to buffer hc % 2; wave w moves its 1 KB
    // blocks 4 w .. 4 w + 3.
    auto issue = [&](int hc) {
        const float *src = p.pack + (long long)hc * kHalfFloats + (4 * wv) * 256 + lane * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_global_load_lds(src + i * 256, (lds_void *)&buf[hc & 1][(4 * wv + i) * 256], 16, 0, 0);
    };
    // Before half-chunk hc is read: its loads done, every wave past the
    // previous one (whose buffer the next half-chunk then overwrites).
    auto next = [&](int hc) {
        wait_vm();
        __syncthreads();
        if (hc + 1 < kHalves) issue(hc + 1);
        return &buf[hc & 1][lane * 4];
    };
    issue(0);

    // x: row m's features 16 kb + 4 g + e (att now, LN2(s1) later).
    f32x4 x[8], s1[8];
    const float *att = p.att + r * p.lda + 4 * g;
    const float *st = p.state + r * p.ldx + 4 * g;
#pragma unroll
    for (int b = 0; b < 8; ++b) x[b] = *reinterpret_cast<const f32x4 *>(att + 16 * b);
#pragma unroll
    for (int b = 0; b < 8; ++b) s1[b] = *reinterpret_cast<const f32x4 *>(st + 16 * b);
    tail_chain(x, s1, next, 0, p, p.state + r * p.ldx + 4 * g, live, g);
}

// A cached column block in one kernel: 64 rows of one column per workgroup,
// wave w carrying rows 16 w .. 16 w + 15 through LN1, the query projection
// (head128's order), the attention of its 8 heads to the column's 128 cached
// inducing keys and values (the 16-wide attention kernel's exact softmax and
// order) and tail128's chain, so q and the attention output never leave
// registers. 32 half-chunks of 16 KB stream through two LDS buffers: 0..3 the
// query rows' fragments, 4..11 head h's keys (fragment order, 8 KB) and values
// (8 KB: per 16-key block, four planes of 64 lanes, lane (d, g) of plane r
// holding key 16 kb + 4 g + r's dim d, gathered by 4-byte loads from the
// cache's [key][16] rows), 12..31 tail128's pack. Workgroups of one XCD take
// consecutive units, so a column's tiles share its K/V in one L2. Three
// workgroups share a CU (168 registers, as tail128; the compiler keeps a few
// values of the prologue in scratch until the epilogue): at two, the
// build's 3.2M-row blocks ran 6% slower than the three launches.
constexpr int kColumnHalves = 32;

__global__ __launch_bounds__(256, 3) void column_block_kernel(ColumnBlock p, int tiles, int per_xcd) {
    __shared__ __attribute__((aligned(16))) float buf[2][kHalfFloats];
    const int unit = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (unit >= p.cols * tiles) return;  // workgroup-uniform, before any barrier
    const int col = unit / tiles, tile = unit - col * tiles;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, g = lane >> 4;
    const long long row = (long long)tile * kTailRows + wv * 16 + m16;
    const bool live = row < p.rows;
    const long long r = live ? row : p.rows - 1;
    float *xrow = p.state + ((long long)col * p.rows + r) * 128 + 4 * g;
    const long long coff = (long long)(col / p.group) * p.group_stride + (long long)(col % p.group) * kColumnCache;
    const float *kcol = p.k + coff, *vcol = p.v + coff;

    auto issue = [&](int h) {
        float *dst = buf[h & 1];
        if (h < 4 || h >= 12) {
            const float *src = (h < 4 ? p.qpack + h * kHalfFloats : p.pack + (h - 12) * kHalfFloats) + (4 * wv) * 256 +
                               lane * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                __builtin_amdgcn_global_load_lds(src + i * 256, (lds_void *)&dst[(4 * wv + i) * 256], 16, 0, 0);
        } else {
            // Head h - 4: wave w moves key blocks 2 w and 2 w + 1.
            const float *kh = kcol + (h - 4) * (kInducing * kColumnHead), *vh = vcol + (h - 4) * (kInducing * kColumnHead);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int kb = 2 * wv + i;
                __builtin_amdgcn_global_load_lds(kh + (16 * kb + m16) * 16 + 4 * g, (lds_void *)&dst[kb * 256], 16, 0, 0);
#pragma unroll
                for (int rr = 0; rr < 4; ++rr)
                    __builtin_amdgcn_global_load_lds(vh + (16 * kb + 4 * g + rr) * 16 + m16,
                                                     (lds_void *)&dst[2048 + (kb * 4 + rr) * 64], 4, 0, 0);
            }
        }
    };
    // Half h's buffer once its loads are done and every wave is past half
    // h - 1 (whose buffer half h + 1 then overwrites).
    auto next = [&](int h) {
        wait_vm();
        __syncthreads();
        if (h + 1 < kColumnHalves) issue(h + 1);
        return &buf[h & 1][0];
    };
    issue(0);

    // The rows' states (kept for the residual) and LN1, as head128.
    f32x4 s1[8], x[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) s1[b] = *reinterpret_cast<const f32x4 *>(xrow + 16 * b);
    {
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < 8; ++b) sum += (s1[b][0] + s1[b][1]) + (s1[b][2] + s1[b][3]);
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        const float mean = sum / 128.f;
        float sq = 0.f;
#pragma unroll
        for (int b = 0; b < 8; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = s1[b][e] - mean;
                sq = fmaf(d, d, sq);
            }
        sq += __shfl_xor(sq, 16, 64);
        sq += __shfl_xor(sq, 32, 64);
        const float rstd = 1.0f / sqrtf(sq / 128.f + 1e-5f);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const f32x4 w = *reinterpret_cast<const f32x4 *>(p.lnw + 16 * b + 4 * g);
            const f32x4 bb = *reinterpret_cast<const f32x4 *>(p.lnb + 16 * b + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[b][e] = (s1[b][e] - mean) * rstd * w[e] + bb[e];
        }
    }

    // q: lane (m, g) holds head h's dims 4 g .. 4 g + 3 of row m in q[h],
    // scaled into the exp2 domain (1 / sqrt(16) = 0.25).
    const float *qsc = p.qpack + head128_pack_floats(128) - kPackScales;
    const float ln_scale = qsc[kHeadLn];
    f32x4 q[8];
#pragma unroll
    for (int ob = 0; ob < 8; ++ob) q[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const Pair xp = pair_of(x[2 * c], x[2 * c + 1], ln_scale);
        const float *frag = next(c) + lane * 4;
        pair_blocks(frag, xp, q);
    }
    const float scale = 0.25f * kLog2e;
#pragma unroll
    for (int ob = 0; ob < 8; ++ob) {
        const f32x4 qb = *reinterpret_cast<const f32x4 *>(p.qb + 16 * ob + 4 * g);
        const f32x4 wi = lds4(qsc + kHeadInv + 16 * ob + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) q[ob][e] = __builtin_fmaf(q[ob][e], wi[e], qb[e]) * scale;
    }

    // Per head: S^T = K Q^T (lane (m, g) holds keys 16 kb + 4 g + r of row
    // m), the exact softmax over the 128 keys, O^T = V^T P^T, which leaves
    // head h's output in tail128's layout for feature block h.
    f32x4 att[8];
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const float *hb = next(4 + h);
        f32x4 s[8];
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) {
            const f32x4 kf = lds4(hb + kb * 256 + lane * 4);
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 4; ++st) acc = mfma(kf[st], q[h][st], acc);
            s[kb] = acc;
        }
        float m = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) m = fmaxf(m, fmaxf(fmaxf(s[kb][0], s[kb][1]), fmaxf(s[kb][2], s[kb][3])));
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        float l = 0.f;
#pragma unroll
        for (int kb = 0; kb < 8; ++kb)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                s[kb][rr] = __builtin_amdgcn_exp2f(s[kb][rr] - m);
                l += s[kb][rr];
            }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        const float inv = 1.0f / l;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) {
            const float *vp = hb + 2048 + kb * 256 + lane;
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) o = mfma(vp[rr * 64], s[kb][rr], o);
        }
        att[h] = o * inv;
    }

    Tail128 t{};
    t.pack = p.pack, t.bo = p.bo, t.n2w = p.n2w, t.n2b = p.n2b, t.b1 = p.b1, t.b2 = p.b2;
    tail_chain(att, s1, [&](int h) { return next(h) + lane * 4; }, 12, t, xrow, live, g);
}

// The same tail for small passes (a few thousand rows or fewer), where
// tail128's 64-row workgroups would leave most CUs idle and each wave would
// carry its rows through all 320 products alone: one workgroup per 16 rows,
// wave w producing output blocks 2 w and 2 w + 1 (of the out-projection and
// of the FFN's second layer) and hidden slices 2 w and 2 w + 1. The waves
// swap s1 and the GELU layer through LDS; every wave takes LN2 of the whole
// rows itself. Fragments are read from the tail128 pack in global memory
// (320 KB, shared by every workgroup through L2), each wave's W1 fragments
// issued with its first loads. Every accumulator takes its products in
// tail128's order, so the results are tail128's bit for bit.
// tail128_rows16's chain from the out-projection on, for wave w of a
// workgroup of 16 rows: x holds the lane's row's attention output (all eight
// blocks), s1 its state's blocks 2 w and 2 w + 1, fo and f1 the wave's Wo and
// W1 fragments; s1s and hs are the workgroup's LDS exchange buffers, pk the
// lane's base in the tail128 pack. The new state's blocks 2 w, 2 w + 1 go to
// out (the lane's first feature, 4 g) when the row is live.
constexpr int kRows16S1Stride = 132, kRows16HidStride = 260;

__device__ __forceinline__ void rows16_chain(const Tail128 &t, const f32x4 (&x)[8], f32x4 (&s1)[2],
                                             const Pair (&fo)[4][2], const Pair (&f1)[2][4][2], float *s1s,
                                             float *hs, const float *pk, int w, int m16, int g, float *out,
                                             bool live) {
    constexpr int kS1Stride = kRows16S1Stride, kHidStride = kRows16HidStride;
    const float *sc = t.pack + kTailScales;
    auto w2_frag = [&](int c, int ob) { return pair_at(pk + (2 + c) * kChunkFloats + 4096 + ob * 512); };
    f32x4 xn[8];
    // Out-projection of output blocks 2 w + j; s1 = state + (acc + bo) to LDS.
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    const int ea = row_exponent(x);
    const float a_scale = pow2(ea), a_inv = pow2(-ea);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) pair_mfma<2>(fo[kb], pair_of(x[2 * kb], x[2 * kb + 1], a_scale), acc);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c0 = 16 * (2 * w + j) + 4 * g;
        const f32x4 bo = *reinterpret_cast<const f32x4 *>(t.bo + c0);
        const f32x4 wi = lds4(sc + kTailOutInv + c0);
#pragma unroll
        for (int e = 0; e < 4; ++e) s1[j][e] = s1[j][e] + __builtin_fmaf(acc[j][e] * wi[e], a_inv, bo[e]);
        *reinterpret_cast<f32x4 *>(&s1s[m16 * kS1Stride + c0]) = s1[j];
    }
    __syncthreads();

    // LN2 of the 16 rows (as tail128: row m's features over lanes m, m + 16,
    // m + 32, m + 48).
#pragma unroll
    for (int b = 0; b < 8; ++b) xn[b] = *reinterpret_cast<const f32x4 *>(&s1s[m16 * kS1Stride + 16 * b + 4 * g]);
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum += xn[b][e];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float mean = sum / 128.f;
    float sq = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float d = xn[b][e] - mean;
            sq = fmaf(d, d, sq);
        }
    sq += __shfl_xor(sq, 16, 64);
    sq += __shfl_xor(sq, 32, 64);
    const float rstd = 1.0f / sqrtf(sq / 128.f + 1e-5f);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const f32x4 nw = *reinterpret_cast<const f32x4 *>(t.n2w + 16 * b + 4 * g);
        const f32x4 nb = *reinterpret_cast<const f32x4 *>(t.n2b + 16 * b + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) xn[b][e] = (xn[b][e] - mean) * rstd * nw[e] + nb[e];
    }

    // Hidden slices c = 2 w + sl: gelu(W1 x + b1) to LDS.
    const float ln_scale = sc[kTailLn], hid_scale = sc[kTailHid];
    Pair xp[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) xp[kb] = pair_of(xn[2 * kb], xn[2 * kb + 1], ln_scale);
#pragma unroll
    for (int sl = 0; sl < 2; ++sl) {
        const int c = 2 * w + sl;
        f32x4 h[2][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) pair_mfma<2>(f1[sl][kb], xp[kb], h[kb & 1]);
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const f32x4 b1 = *reinterpret_cast<const f32x4 *>(t.b1 + 32 * c + 16 * hb + 4 * g);
            const f32x4 wi = lds4(sc + kTailLnInv + 32 * c + 16 * hb + 4 * g);
            f32x4 hg;
#pragma unroll
            for (int e = 0; e < 4; ++e) hg[e] = gelu_erf(__builtin_fmaf(h[0][hb][e] + h[1][hb][e], wi[e], b1[e]));
            *reinterpret_cast<f32x4 *>(&hs[m16 * kHidStride + 32 * c + 16 * hb + 4 * g]) = hg;
        }
    }
    // This wave's W2 fragments (output blocks 2 w + j), in flight over the barrier.
    Pair f2[8][2];
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) f2[c][ob] = w2_frag(c, 2 * w + ob);
    __syncthreads();

    // FFN down over the 256 hidden units, slice by slice as tail128 does.
    f32x4 acc2[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float *hv = &hs[m16 * kHidStride + 32 * c + 4 * g];
        pair_mfma<2>(f2[c], pair_of(lds4(hv), lds4(hv + 16), hid_scale), acc2);
    }
    if (!live) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c0 = 16 * (2 * w + j);
        const f32x4 b2 = *reinterpret_cast<const f32x4 *>(t.b2 + c0 + 4 * g);
        const f32x4 wi = lds4(sc + kTailHidInv + c0 + 4 * g);
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(acc2[j][e], wi[e], b2[e]) + s1[j][e];
        *reinterpret_cast<f32x4 *>(out + c0) = v;
    }
}

__global__ __launch_bounds__(256) void tail128_rows16_kernel(Tail128 p) {
    constexpr int kS1Stride = kRows16S1Stride, kHidStride = kRows16HidStride;
    __shared__ __attribute__((aligned(16))) float s1s[16 * kS1Stride];
    __shared__ __attribute__((aligned(16))) float hs[16 * kHidStride];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, g = lane >> 4;
    const long long row = (long long)blockIdx.x * 16 + m16;
    const bool live = row < p.m;
    const long long r = live ? row : p.m - 1;
    const float *pk = p.pack + lane * 4;
    Pair fo[4][2];
    f32x4 x[8], s1[2];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 2; ++j) fo[kb][j] = pair_at(pk + (kb * 8 + 2 * w + j) * 512);
    const float *att = p.att + r * p.lda + 4 * g;
#pragma unroll
    for (int b = 0; b < 8; ++b) x[b] = *reinterpret_cast<const f32x4 *>(att + 16 * b);
    const float *st = p.state + r * p.ldx + 4 * g;
#pragma unroll
    for (int j = 0; j < 2; ++j) s1[j] = *reinterpret_cast<const f32x4 *>(st + 16 * (2 * w + j));
    Pair f1[2][4][2];
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) f1[sl][kb][hb] = pair_at(pk + (2 + 2 * w + sl) * kChunkFloats + (kb * 2 + hb) * 512);

    rows16_chain(p, x, s1, fo, f1, s1s, hs, pk, w, m16, g, p.state + r * p.ldx + 4 * g, live);
}

// The cached column block for small passes: one workgroup per 16 rows of
// one column, wave w taking query heads and output blocks 2 w and 2 w + 1
// (tail128_rows16's split). Every wave takes LN1 of the whole rows; its
// query fragments, its heads' keys (fragment order) and values (lane (d, g)
// value r of key block kb = key 16 kb + 4 g + r's dim d) come straight from
// global memory, all issued with its first loads, and the tail's Wo and W1
// fragments follow while the attention runs. The attention outputs meet in
// LDS for the out-projection; from there on this is tail128_rows16. The
// arithmetic is column_block_kernel's, so the results are its bits.
__global__ __launch_bounds__(256) void column_block_rows16_kernel(ColumnBlock p, int groups) {
    constexpr int kS1Stride = kRows16S1Stride, kHidStride = kRows16HidStride;
    __shared__ __attribute__((aligned(16))) float as[16 * kS1Stride];
    __shared__ __attribute__((aligned(16))) float s1s[16 * kS1Stride];
    __shared__ __attribute__((aligned(16))) float hs[16 * kHidStride];
    const int unit = blockIdx.x;
    const int col = unit / groups, grp = unit - col * groups;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, g = lane >> 4;
    const long long row = (long long)grp * 16 + m16;
    const bool live = row < p.rows;
    const long long r = live ? row : p.rows - 1;
    float *xrow = p.state + ((long long)col * p.rows + r) * 128 + 4 * g;
    const long long coff = (long long)(col / p.group) * p.group_stride + (long long)(col % p.group) * kColumnCache;
    const float *kh = p.k + coff + (2 * w) * (kInducing * kColumnHead);
    const float *vh = p.v + coff + (2 * w) * (kInducing * kColumnHead);
    const float *qk = p.qpack + lane * 4, *pk = p.pack + lane * 4;

    f32x4 x[8], kf[2][8];
    Pair fq[4][2];
    float vv[2][8][4];
#pragma unroll
    for (int b = 0; b < 8; ++b) x[b] = *reinterpret_cast<const f32x4 *>(xrow + 16 * b);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 2; ++j) fq[kb][j] = pair_at(qk + (kb * 8 + 2 * w + j) * 512);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) {
            kf[j][kb] = *reinterpret_cast<const f32x4 *>(kh + j * 2048 + (16 * kb + m16) * 16 + 4 * g);
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) vv[j][kb][rr] = vh[j * 2048 + (16 * kb + 4 * g + rr) * 16 + m16];
        }

    // LN1 over the rows, as head128.
    {
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < 8; ++b) sum += (x[b][0] + x[b][1]) + (x[b][2] + x[b][3]);
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        const float mean = sum / 128.f;
        float sq = 0.f;
#pragma unroll
        for (int b = 0; b < 8; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = x[b][e] - mean;
                sq = fmaf(d, d, sq);
            }
        sq += __shfl_xor(sq, 16, 64);
        sq += __shfl_xor(sq, 32, 64);
        const float rstd = 1.0f / sqrtf(sq / 128.f + 1e-5f);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const f32x4 lw = *reinterpret_cast<const f32x4 *>(p.lnw + 16 * b + 4 * g);
            const f32x4 lb = *reinterpret_cast<const f32x4 *>(p.lnb + 16 * b + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[b][e] = (x[b][e] - mean) * rstd * lw[e] + lb[e];
        }
    }
    f32x4 q[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    const float *qsc = p.qpack + head128_pack_floats(128) - kPackScales;
    const float q_scale = qsc[kHeadLn];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) pair_mfma<2>(fq[kb], pair_of(x[2 * kb], x[2 * kb + 1], q_scale), q);
    const float scale = 0.25f * kLog2e;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const f32x4 qb = *reinterpret_cast<const f32x4 *>(p.qb + 16 * (2 * w + j) + 4 * g);
        const f32x4 wi = lds4(qsc + kHeadInv + 16 * (2 * w + j) + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) q[j][e] = __builtin_fmaf(q[j][e], wi[e], qb[e]) * scale;
    }

    // The tail's fragments for this wave and its state blocks, in flight
    // during the attention.
    Pair fo[4][2], f1[2][4][2];
    f32x4 s1[2];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 2; ++j) fo[kb][j] = pair_at(pk + (kb * 8 + 2 * w + j) * 512);
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) f1[sl][kb][hb] = pair_at(pk + (2 + 2 * w + sl) * kChunkFloats + (kb * 2 + hb) * 512);
#pragma unroll
    for (int j = 0; j < 2; ++j) s1[j] = *reinterpret_cast<const f32x4 *>(xrow + 16 * (2 * w + j));

    // Heads 2 w + j, as column_block_kernel.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        f32x4 s[8];
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 4; ++st) acc = mfma(kf[j][kb][st], q[j][st], acc);
            s[kb] = acc;
        }
        float m = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) m = fmaxf(m, fmaxf(fmaxf(s[kb][0], s[kb][1]), fmaxf(s[kb][2], s[kb][3])));
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        float l = 0.f;
#pragma unroll
        for (int kb = 0; kb < 8; ++kb)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                s[kb][rr] = __builtin_amdgcn_exp2f(s[kb][rr] - m);
                l += s[kb][rr];
            }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        const float inv = 1.0f / l;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 8; ++kb)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) o = mfma(vv[j][kb][rr], s[kb][rr], o);
        *reinterpret_cast<f32x4 *>(&as[m16 * kS1Stride + 16 * (2 * w + j) + 4 * g]) = o * inv;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 8; ++b) x[b] = *reinterpret_cast<const f32x4 *>(&as[m16 * kS1Stride + 16 * b + 4 * g]);
    Tail128 t{};
    t.pack = p.pack, t.bo = p.bo, t.n2w = p.n2w, t.n2b = p.n2b, t.b1 = p.b1, t.b2 = p.b2;
    rows16_chain(t, x, s1, fo, f1, s1s, hs, pk, w, m16, g, xrow, live);
}

// The head of a 128-wide block: y = LN1(x) W^T + b over 16 NB outputs,
// written row-major; the same per-wave layout as tail128, the fragments of W
// in (k-block, output block) order streamed through the same LDS buffers.
template <int NB>
__global__ __launch_bounds__(256, 3) void head128_kernel(Head128 p) {
    // 16 KB halves of the packed chunks, as tail128 streams them: 32 KB of LDS
    // per workgroup, so three (four at 8 and 16 output blocks, whose
    // registers allow it) share a CU.
    __shared__ __attribute__((aligned(16))) float buf[2][kHalfFloats];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, g = lane >> 4;
    const long long row = (long long)blockIdx.x * kTailRows + wv * 16 + m16;
    const bool live = row < p.m;
    const long long r = live ? row : p.m - 1;
    auto issue = [&](int hc) {
        // A short last half still moves 16 KB: the pack is padded to whole chunks.
        const float *src = p.pack + (long long)hc * kHalfFloats + (4 * wv) * 256 + lane * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_global_load_lds(src + i * 256, (lds_void *)&buf[hc & 1][(4 * wv + i) * 256], 16, 0, 0);
    };
    issue(0);

    f32x4 x[8];
    const float *xr = p.x + r * p.ldx + 4 * g;
#pragma unroll
    for (int b = 0; b < 8; ++b) x[b] = *reinterpret_cast<const f32x4 *>(xr + 16 * b);
    // LN1 over the row's 128 features (lanes m, m + 16, m + 32, m + 48).
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b) sum += (x[b][0] + x[b][1]) + (x[b][2] + x[b][3]);
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float mean = sum / 128.f;
    float sq = 0.f;
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float d = x[b][e] - mean;
            sq = fmaf(d, d, sq);
        }
    sq += __shfl_xor(sq, 16, 64);
    sq += __shfl_xor(sq, 32, 64);
    const float rstd = 1.0f / sqrtf(sq / 128.f + 1e-5f);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const f32x4 w = *reinterpret_cast<const f32x4 *>(p.lnw + 16 * b + 4 * g);
        const f32x4 bb = *reinterpret_cast<const f32x4 *>(p.lnb + 16 * b + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = (x[b][e] - mean) * rstd * w[e] + bb[e];
    }

    const float *sc = p.pack + head128_pack_floats(16 * NB) - kPackScales;
    const float ln_scale = sc[kHeadLn];
    Pair xp[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) xp[kb] = pair_of(x[2 * kb], x[2 * kb + 1], ln_scale);
    f32x4 acc[NB];
#pragma unroll
    for (int ob = 0; ob < NB; ++ob) acc[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Half c holds the pairs of eight (k-block, output block) fragments.
#pragma unroll
    for (int c = 0; c < NB / 2; ++c) {
        wait_vm();
        __syncthreads();
        if (c + 1 < NB / 2) issue(c + 1);
        const float *frag = &buf[c & 1][lane * 4];
        const int kb = 8 * c / NB, ob0 = 8 * c % NB;
        pair_blocks(frag, xp[kb], &acc[ob0]);
    }
    if (!live) return;
    float *out = p.out + row * p.ldo + 4 * g;
#pragma unroll
    for (int ob = 0; ob < NB; ++ob) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(p.b + 16 * ob + 4 * g);
        const f32x4 wi = lds4(sc + kHeadInv + 16 * ob + 4 * g);
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(acc[ob][e], wi[e], b[e]);
        *reinterpret_cast<f32x4 *>(out + 16 * ob) = v;
    }
}

// Fragment pair (rows r0.., columns c0 .. c0 + 31) of a row-major [.., ld]
// matrix, row r times 2^e[r]: lane (n, g) = (l % 16, l / 16) slot e holds row r0 + n,
// column c0 + 16 (e / 4) + 4 g + e % 4; 1 KB of hi parts, then of lo parts.
void pack_pair(const float *w, int ld, int r0, int c0, const std::vector<int> &e2, float *dst) {
    _Float16 *hi = reinterpret_cast<_Float16 *>(dst), *lo = reinterpret_cast<_Float16 *>(dst + 256);
    for (int l = 0; l < 64; ++l)
        for (int e = 0; e < 8; ++e) {
            const int r = r0 + (l & 15);
            const float x = std::ldexp(w[(long long)r * ld + c0 + 16 * (e >> 2) + 4 * (l >> 4) + (e & 3)], e2[r]);
            const _Float16 h = (_Float16)x;
            hi[l * 8 + e] = h;
            lo[l * 8 + e] = (_Float16)(x - (float)h);
        }
}

// The rows' exponents; `with` is that of the operand they multiply, whose sum
// with each stays a float's.
std::vector<int> row_exponents(const float *w, int rows, int ld, int with = 0) {
    std::vector<int> e(rows);
    for (int r = 0; r < rows; ++r) {
        float largest = 0.f;
        for (int i = 0; i < ld; ++i) largest = std::max(largest, std::fabs(w[(long long)r * ld + i]));
        e[r] = std::max(-126 - with, std::min(126 - with, pair_scale_exponent(largest, 14)));
    }
    return e;
}
// The bound of a LayerNormed row's values: at most sqrt(128) of deviation.
int ln_exponent(const float *w, const float *b) {
    float lw = 0.f, lb = 0.f;
    for (int i = 0; i < 128; ++i) lw = std::max(lw, std::fabs(w[i])), lb = std::max(lb, std::fabs(b[i]));
    return pair_scale_exponent(11.5 * lw + lb, 15);
}

}  // namespace

void head128_pack(const float *lnw, const float *lnb, const float *w, int outputs, float *out) {
    const int nb = outputs / 16;
    std::fill(out, out + head128_pack_floats(outputs), 0.f);
    const int el = ln_exponent(lnw, lnb);
    const std::vector<int> ew = row_exponents(w, outputs, 128, el);
    for (int kb = 0; kb < 4; ++kb)
        for (int ob = 0; ob < nb; ++ob)
            pack_pair(w, 128, 16 * ob, 32 * kb, ew, out + (size_t)(kb * nb + ob) * 512);
    float *sc = out + head128_pack_floats(outputs) - kPackScales;
    sc[kHeadLn] = std::ldexp(1.f, el);
    for (int r = 0; r < outputs; ++r) sc[kHeadInv + r] = std::ldexp(1.f, -el - ew[r]);
}

void head128(const Head128 &h, hipStream_t stream) {
    if (h.m <= 0) return;
    if (!h.x || !h.out || !h.pack || !h.lnw || !h.lnb || !h.b || (h.nb != 8 && h.nb != 16 && h.nb != 24))
        fail(3, "head128: unsupported arguments");
    if ((h.ldx & 3) || (h.ldo & 3) || (reinterpret_cast<uintptr_t>(h.x) & 15) ||
        (reinterpret_cast<uintptr_t>(h.out) & 15) || (reinterpret_cast<uintptr_t>(h.pack) & 15))
        fail(3, "head128: rows must be 16-byte aligned");
    const double m = (double)h.m, n = 16.0 * h.nb;
    KernelTimer timer(kFamGemm, stream, 2.0 * m * 128.0 * n, 4.0 * m * (128.0 + n) + 4.0 * 128.0 * n);
    const dim3 grid((unsigned)ceil_div(h.m, (long long)kTailRows)), block(256);
    if (h.nb == 8)
        hipLaunchKernelGGL(head128_kernel<8>, grid, block, 0, stream, h);
    else if (h.nb == 16)
        hipLaunchKernelGGL(head128_kernel<16>, grid, block, 0, stream, h);
    else
        hipLaunchKernelGGL(head128_kernel<24>, grid, block, 0, stream, h);
    IRX_HIP(hipGetLastError());
}

void tail128_pack(const float *wo, const float *n2w, const float *n2b, const float *w1, const float *b1,
                  const float *w2, float *out) {
    std::fill(out, out + kTail128PackFloats, 0.f);
    // A hidden unit: at most sqrt(128) times the norm of its weights times
    // LN2's, plus what the biases give it; its GELU is no larger.
    double hidden = 0.0;
    for (int u = 0; u < 256; ++u) {
        double norm = 0.0, bias = b1[u];
        for (int i = 0; i < 128; ++i) {
            const double a = (double)w1[u * 128 + i] * n2w[i];
            norm += a * a, bias += (double)w1[u * 128 + i] * n2b[i];
        }
        hidden = std::max(hidden, 11.5 * std::sqrt(norm) + std::fabs(bias));
    }
    const int el = ln_exponent(n2w, n2b), eh = pair_scale_exponent(hidden, 15);
    const std::vector<int> so = row_exponents(wo, 128, 128), s1 = row_exponents(w1, 256, 128, el);
    const std::vector<int> s2 = row_exponents(w2, 128, 256, eh);
    for (int kb = 0; kb < 4; ++kb)
        for (int ob = 0; ob < 8; ++ob) pack_pair(wo, 128, 16 * ob, 32 * kb, so, out + (kb * 8 + ob) * 512);
    for (int c = 0; c < 8; ++c) {
        float *chunk = out + (2 + c) * kChunkFloats;
        for (int kb = 0; kb < 4; ++kb)
            for (int hb = 0; hb < 2; ++hb) pack_pair(w1, 128, 32 * c + 16 * hb, 32 * kb, s1, chunk + (kb * 2 + hb) * 512);
        for (int ob = 0; ob < 8; ++ob) pack_pair(w2, 256, 16 * ob, 32 * c, s2, chunk + 4096 + ob * 512);
    }
    float *sc = out + kTailScales;
    sc[kTailLn] = std::ldexp(1.f, el), sc[kTailHid] = std::ldexp(1.f, eh);
    for (int r = 0; r < 128; ++r)
        sc[kTailOutInv + r] = std::ldexp(1.f, -so[r]), sc[kTailHidInv + r] = std::ldexp(1.f, -eh - s2[r]);
    for (int r = 0; r < 256; ++r) sc[kTailLnInv + r] = std::ldexp(1.f, -el - s1[r]);
}

void tail128(const Tail128 &t, hipStream_t stream, bool rows16) {
    if (t.m <= 0) return;
    if (!t.att || !t.state || !t.pack || !t.bo || !t.n2w || !t.n2b || !t.b1 || !t.b2)
        fail(3, "tail128: missing tensor");
    if ((t.lda & 3) || (t.ldx & 3) || (reinterpret_cast<uintptr_t>(t.att) & 15) ||
        (reinterpret_cast<uintptr_t>(t.state) & 15) || (reinterpret_cast<uintptr_t>(t.pack) & 15))
        fail(3, "tail128: rows must be 16-byte aligned");
    const double m = (double)t.m;
    // Products 2 m (128*128 + 2 * 128*256); bytes: att and state in, state out, weights.
    KernelTimer timer(kFamGemm, stream, m * 2.0 * (128.0 * 128 + 2 * 128.0 * 256), m * 128 * 4 * 3.0 + kTail128PackFloats * 4.0);
    if (rows16)
        hipLaunchKernelGGL(tail128_rows16_kernel, dim3((unsigned)ceil_div(t.m, 16LL)), dim3(256), 0, stream, t);
    else
        hipLaunchKernelGGL(tail128_kernel, dim3((unsigned)ceil_div(t.m, (long long)kTailRows)), dim3(256), 0, stream, t);
    IRX_HIP(hipGetLastError());
}

void column_block(const ColumnBlock &c, hipStream_t stream, bool rows16) {
    if (c.cols <= 0 || c.rows <= 0) return;
    if (!c.state || !c.k || !c.v || !c.lnw || !c.lnb || !c.qpack || !c.qb || !c.pack || !c.bo || !c.n2w || !c.n2b ||
        !c.b1 || !c.b2 || c.group <= 0)
        fail(3, "column_block: missing tensor");
    if ((reinterpret_cast<uintptr_t>(c.state) & 15) || (reinterpret_cast<uintptr_t>(c.k) & 15) ||
        (reinterpret_cast<uintptr_t>(c.v) & 15) || (reinterpret_cast<uintptr_t>(c.qpack) & 15) ||
        (reinterpret_cast<uintptr_t>(c.pack) & 15) || (c.group_stride & 3))
        fail(3, "column_block: operands must be 16-byte aligned");
    const long long tiles = (c.rows + kTailRows - 1) / kTailRows, units = tiles * c.cols;
    const long long per_xcd = (units + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffLL) fail(3, "column_block: too many rows");
    const double m = (double)c.cols * (double)c.rows;
    // q, attention (scores and values over 128 keys x 8 heads of 16), the tail.
    const double flops = m * 2.0 * (128.0 * 128 + 2.0 * 128 * 128 + 128.0 * 128 + 2 * 128.0 * 256);
    KernelTimer timer(kFamGemm, stream, flops, m * 128 * 4 * 2.0 + (double)c.cols * kColumnCache * 8.0);
    if (rows16) {
        const long long groups = (c.rows + 15) / 16;
        if (groups * c.cols > 0x7fffffffLL) fail(3, "column_block: too many rows");
        hipLaunchKernelGGL(column_block_rows16_kernel, dim3((unsigned)(groups * c.cols)), dim3(256), 0, stream, c,
                           (int)groups);
    } else {
        hipLaunchKernelGGL(column_block_kernel, dim3((unsigned)(per_xcd * 8)), dim3(256), 0, stream, c, (int)tiles,
                           (int)per_xcd);
    }
    IRX_HIP(hipGetLastError());
}

}  // namespace irx
