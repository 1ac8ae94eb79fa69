// Many-row path of the FASTQUANT RWKV-4 forward pass: a prompt (T tokens of one
// sequence; reference agnostic/backends/opt.py:61-76 with T > 1,
// modules/matmul.py:56-57,86-94) or a batch (B independent sequences, one token
// each).  Rows are tokens; every matrix product is a GEMM on the matrix cores.
//
// Arithmetic.  Exactly the single-token kernel's: each row of
// xs = fp32(x * range) is rewritten as 32-bit fixed point q = round(xs / S),
// S a power of two chosen per row so that |q| <= 2^30, and split into four
// signed base-256 digits.  The digit rows (4 per token) are the A operand and
// the weights, stored as code - 128 in 1 KiB blocks of 16 columns x 64 rows
// ("M16"), the B operand of v_mfma_i32_16x16x64_i8.  Integer sums are exact and
// independent of tiling and of any split of the contraction, so a prompt
// processed here gives the same products as the same tokens fed one at a time.
// (The reference rounds this product to bfloat16, matmul.py:57; nothing here
// is rounded below float32 class.)
//
// Digit rows are stored in fragment order: for M-tile mt (tokens 4mt..4mt+3) and
// contraction block kb (rows 64kb..64kb+63) one 1 KiB fragment whose lane
// 16g + m holds bytes k = 64kb + 16g + i (i < 16) of digit row m = 4*(t % 4) + d;
// a wavefront loads a fragment with one coalesced 16-byte-per-lane request and
// hands it to the matrix instruction unchanged.
#include "rwkv_rows.h"

#include <algorithm>
#include <type_traits>

namespace rwkv {

namespace {

constexpr int kRT = 256;           // threads of the row kernels
constexpr int kRW = kRT / 64;

typedef int v4i __attribute__((ext_vector_type(4)));

// Sums and maxima over a wavefront without the LDS crossbar (a butterfly of 64-bit shuffles is twelve dependent trips
// through LDS; the row kernels are chains of such reductions).  Every lane ends with the same value.  The sum is that of the
// butterfly, lanes 32, 16, 8, 4, 2, 1 apart in this order: its last bit reaches the logits, and with them the texts of a
// seeded sampler.  Halves and rows of 16 lanes change places by permlane swaps, and inside a row DPP rotations stand for the
// butterfly's steps, since what lanes 8 and then 4 apart have just added up repeats with that period.
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp32(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false)); }
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140, kDppRor4 = 0x124, kDppRor8 = 0x128;
__device__ __forceinline__ double wsum(double v) {
    {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    v += dpp64<kDppRor8>(v);
    v += dpp64<kDppRor4>(v);
    v += dpp64<kDppXor2>(v);
    return v + dpp64<kDppXor1>(v);
}
__device__ __forceinline__ float wmaxf(float v) {
    v = fmaxf(v, dpp32<kDppXor1>(v));
    v = fmaxf(v, dpp32<kDppXor2>(v));
    v = fmaxf(v, dpp32<kDppHalfMirror>(v));
    v = fmaxf(v, dpp32<kDppMirror>(v));
    const int i = __float_as_int(v);
    return fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(i, 0)), __int_as_float(__builtin_amdgcn_readlane(i, 16))),
                 fmaxf(__int_as_float(__builtin_amdgcn_readlane(i, 32)), __int_as_float(__builtin_amdgcn_readlane(i, 48))));
}

// Sum of N values per thread over the workgroup (fixed order), broadcast.
template <int N>
__device__ __forceinline__ void rsum(double (&v)[N], double *red /*[N*kRW]*/) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double s = wsum(v[i]);
        if (lane == 0) red[i * kRW + wave] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kRW; ++w) s += red[i * kRW + w];
        v[i] = s;
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// x[t] = ln0(emb[token[t]])          (emb.py:9, opt.py:63-64)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kRT)
rows_embed_kernel(const int64_t *__restrict__ tokens, int V, int C, const float *__restrict__ emb,
                  const double *__restrict__ w, const double *__restrict__ b, double *__restrict__ x) {
    __shared__ double red[2 * kRW];
    const int t = blockIdx.x;
    int64_t tok = tokens[t];
    if (tok < 0) tok = 0;
    if (tok >= V) tok = V - 1;
    const float *e = emb + (size_t)tok * C;
    double s[1] = {0.0};
    for (int c = threadIdx.x; c < C; c += kRT) s[0] += (double)e[c];
    rsum<1>(s, red);
    const double mean = s[0] / (double)C;
    double q[1] = {0.0};
    for (int c = threadIdx.x; c < C; c += kRT) { const double d = (double)e[c] - mean; q[0] += d * d; }
    rsum<1>(q, red);
    const double sd = sqrt(q[0] / (double)C + 1e-5);
    for (int c = threadIdx.x; c < C; c += kRT) x[(size_t)t * C + c] = w[c] * (((double)e[c] - mean) / sd) + b[c];
}

// ---------------------------------------------------------------------------
// Fixed-point digits of four consecutive values of a row (columns c0..c0+3 of token t), written into
// the row's fragments; returns the sum of the four fixed-point values.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double emit_quad(const float (&x4)[4], double invS, int c0, int t, int KB,
                                            signed char *dig) {
    // q = sum_k d_k 256^k with signed digits d_k in [-128, 127]  <=>  q + 0x80808080 has the unsigned bytes
    // d_k + 128, and b - 128 is b ^ 0x80 as a signed byte: two instructions give all four digits of a value.
    unsigned u[4];
    double qsum = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = __double2int_rn((double)x4[i] * invS);
        qsum += (double)q;
        u[i] = ((unsigned)q + 0x80808080u) ^ 0x80808080u;
    }
    // 4 x 4 byte transpose: one dword per digit plane, most significant first
    const unsigned x0 = __builtin_amdgcn_perm(u[1], u[0], 0x05010400u), x1 = __builtin_amdgcn_perm(u[1], u[0], 0x07030602u);
    const unsigned y0 = __builtin_amdgcn_perm(u[3], u[2], 0x05010400u), y1 = __builtin_amdgcn_perm(u[3], u[2], 0x07030602u);
    const unsigned pl[4] = {__builtin_amdgcn_perm(y1, x1, 0x07060302u), __builtin_amdgcn_perm(y1, x1, 0x05040100u),
                            __builtin_amdgcn_perm(y0, x0, 0x07060302u), __builtin_amdgcn_perm(y0, x0, 0x05040100u)};
    const int mt = t >> 2, m0 = (t & 3) * 4;
    const int kb = c0 >> 6, g = (c0 & 63) >> 4, j = (c0 & 15) >> 2;
    // The four lanes j = 0..3 that hold the 16 channels of one fragment slot transpose their 4 x 4 dwords
    // (two exchanges, with the neighbour and with the lane two further): lane j ends up with digit plane j of all 16
    // channels and writes it with ONE 16-byte store; the four lanes together fill a whole 64-byte line.  (Four
    // 4-byte stores per lane into four different lines cost the quantisers a third of their time.)  Callers
    // guarantee whole groups of four lanes: c0 = 4 * (a multiple-of-4-aligned lane index), widths multiples of 16.
    unsigned a4[4] = {pl[0], pl[1], pl[2], pl[3]};
    {
        const bool odd = j & 1;
        const unsigned s0 = odd ? a4[0] : a4[1], s1 = odd ? a4[2] : a4[3];
        const unsigned r0 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)s0, 0xB1, 0xf, 0xf, false);
        const unsigned r1 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)s1, 0xB1, 0xf, 0xf, false);
        if (odd) { a4[0] = r0; a4[2] = r1; } else { a4[1] = r0; a4[3] = r1; }
        const bool hi = j & 2;
        const unsigned t0 = hi ? a4[0] : a4[2], t1 = hi ? a4[1] : a4[3];
        const unsigned q0 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)t0, 0x4E, 0xf, 0xf, false);
        const unsigned q1 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)t1, 0x4E, 0xf, 0xf, false);
        if (hi) { a4[0] = q0; a4[1] = q1; } else { a4[2] = q0; a4[3] = q1; }
    }
    signed char *slot = dig + ((size_t)mt * KB + kb) * 1024 + (16 * g + m0 + j) * 16;
    *reinterpret_cast<uint4 *>(slot) = make_uint4(a4[0], a4[1], a4[2], a4[3]);
    return qsum;
}

// Power-of-two scale of a row whose largest |xs| is amax: |xs / S| <= 2^30.
__device__ __forceinline__ void row_scale(float amax, double &S, double &invS) {
    S = 0.0; invS = 0.0;
    if (amax > 0.f && amax < INFINITY) {
        int e;
        frexpf(amax, &e);                  // amax = f * 2^e, f in [0.5, 1)  =>  |xs| < 2^e
        S = ldexp(1.0, e - 30);
        invS = ldexp(1.0, 30 - e);
    }
}

// ---------------------------------------------------------------------------
// LayerNorm + token shift + time mix + row quantiser      (layernorm.py:15-20, block.py:58-67,82-91,
// matmul.py:59-62,131-133)
//   xy = ln(x[t]);  prev = sequence ? (t == 0 ? prev0 : ln(x[t-1])) : prev0[t];
//   mix_m[t] = xy * mu_m + prev * (1 - mu_m), quantised for matrix m; the newest xy becomes the shift state.
// NM == 0: LayerNorm only, one output (the head's ln_out).
// One workgroup per row; a thread keeps its NSEG groups of four channels in registers from the one
// read of x to the digits, so the mixed rows never travel through memory.
// ---------------------------------------------------------------------------
// Element (t, j) of a product handed on unfinished: the slices added up (integers: exact in any order), then
// y = S_t * tot + 128 * S_t * sum q_t + zp_t as in rows_finish_kernel.
__device__ __forceinline__ double deferred_y(const RowsDeferred &d, int t, long long tot) {
    const double S = d.S[t], sq = 128.0 * (S * d.qs[t]), zp = d.zp[t];
    return d.apart ? S * (double)tot + sq + zp : S * (double)tot + (sq + zp);
}
// The slices are requested together, of exactly so many and behind one branch for all that a thread adds up: a loop over a run-time count
// would wait for every slice before asking for the next, and a branch for each value would keep their loads apart.
template <int SLICES>
__device__ __forceinline__ long long slices_sum1(const long long *tp, size_t slice) {
    long long u[SLICES], tot = 0;
#pragma unroll
    for (int z = 0; z < SLICES; ++z) u[z] = tp[(size_t)z * slice];
#pragma unroll
    for (int z = 0; z < SLICES; ++z) tot += u[z];
    return tot;
}
template <int SLICES>
__device__ __forceinline__ void slices_sum4(const long long *tp, size_t slice, long long (&tot)[4]) {
    longlong2 u[SLICES][2];
#pragma unroll
    for (int z = 0; z < SLICES; ++z) {
        const long long *q = tp + (size_t)z * slice;
        u[z][0] = *reinterpret_cast<const longlong2 *>(q); u[z][1] = *reinterpret_cast<const longlong2 *>(q + 2);
    }
    tot[0] = tot[1] = tot[2] = tot[3] = 0;
#pragma unroll
    for (int z = 0; z < SLICES; ++z) { tot[0] += u[z][0].x; tot[1] += u[z][0].y; tot[2] += u[z][1].x; tot[3] += u[z][1].y; }
}
// F(count), the count a constant, for each of the counts that slices may have.
static_assert(kRowsDeferSlices == 6, "the counts below");
template <typename F>
__device__ __forceinline__ void with_slices(int slices, F &&f) {
    if (slices == 2) f(std::integral_constant<int, 2>());
    else if (slices == 3) f(std::integral_constant<int, 3>());
    else if (slices == 4) f(std::integral_constant<int, 4>());
    else if (slices == 5) f(std::integral_constant<int, 5>());
    else f(std::integral_constant<int, 6>());
}

struct LnQuantArgs {
    int C, R, sequence;
    const double *x;            // [R, C]
    RowsDeferred add;           // few-row form: x += this product first (and the row before, whose LayerNorm is needed), stored to x_out (tot null: none)
    double *x_out;              // null: nobody reads x again
    double *shift_out;          // few-row form of batch rows, [R, C]: the newest xy rows go here instead of to shift_dst (null: to shift_dst)
    const double *commit_src;   // few-row form or sequence: [R, C] rows (sequence: one) an earlier launch left aside (null: none) ...
    double *commit_dst;         // ... copied to commit_dst + row * prev_stride
    const double *ln_w, *ln_b;  // [C]
    const double *mu;           // [NM, C]
    const double *prev0;        // sequence: [C]; batch: row t at prev0 + t * prev_stride
    double *shift_dst;          // sequence: [C] aside (written by row R-1, while row 0 reads the state); batch: row t at shift_dst + t * prev_stride
    int64_t prev_stride;
    const float *range[3];      // per output: the matrix's per-input-channel range / offset
    const double *offset[3];
    signed char *dig[3];        // per output: fragments [ceil(R/4)][C/64][1024] and the row constants
    double *S[3], *qs[3], *zp[3];
};

constexpr int kLnMaxWidth = 6144;       // widest row the LayerNorm kernels hold in registers

// Sum of N values per thread over the kLW wavefronts of the workgroup (fixed order), broadcast.
template <int N, int kLW>
__device__ __forceinline__ void lsum(double (&v)[N], double *red /*[N*kLW]*/) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double s = wsum(v[i]);
        if (lane == 0) red[i * kLW + wave] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kLW; ++w) s += red[i * kLW + w];
        v[i] = s;
    }
    __syncthreads();
}

// Sum of N values per thread over the nw <= 8 wavefronts of the workgroup (fixed order, that of lsum), broadcast; red[N * 8]
// is used by no other reduction, so one barrier does.
__device__ __forceinline__ double row16_sum(double v) {
    v += dpp64<kDppXor1>(v);
    v += dpp64<kDppXor2>(v);
    v += dpp64<kDppHalfMirror>(v);
    return v + dpp64<kDppMirror>(v);
}
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp32<kDppXor1>(v));
    v = fmaxf(v, dpp32<kDppXor2>(v));
    v = fmaxf(v, dpp32<kDppHalfMirror>(v));
    return fmaxf(v, dpp32<kDppMirror>(v));
}
template <int N>
__device__ __forceinline__ void bsum(double (&v)[N], double *red, int nw) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double s = wsum(v[i]);
        if (lane == 0) red[i * 8 + wave] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < 8; ++w) s += w < nw ? red[i * 8 + w] : 0.0;
        v[i] = s;
    }
}
__device__ __forceinline__ void ld4(double (&v)[4], const double *p) {
    const double2 a = *reinterpret_cast<const double2 *>(p), b = *reinterpret_cast<const double2 *>(p + 2);
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ __forceinline__ void ld4(float (&v)[4], const float *p) {
    const float4 a = *reinterpret_cast<const float4 *>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}

__device__ __forceinline__ void st4(double *p, const double (&v)[4]) {
    *reinterpret_cast<double2 *>(p) = make_double2(v[0], v[1]);
    *reinterpret_cast<double2 *>(p + 2) = make_double2(v[2], v[3]);
}

// The same for fewer than kRowsDeferMax rows, where one row's chain of dependent steps is the whole kernel.  Most of it is
// instruction fetch: a launch begins with cold instruction caches and runs straight through code it uses once, so the three
// mixes are not unrolled into one workgroup but go to workgroups of their own (blockIdx.y), which take the row's statistics
// each for themselves.  A thread per group of four channels, at most 512 (the sums' order: wider rows give a thread two or three
// groups, 2048 channels apart), all loads requested before the first reduction.
//
// The workgroups of a row may not write what the others still read.  So the row's new x (a residual update that a split
// product left pending is applied here) goes to x_out, another buffer than x, and its newest shift row to shift_out; the next
// launch of this kernel copies that one into the state (commit).
//
// 8 rows of 2560 channels, three / two mixes: 6.9 / 7.4 us, 32 rows of 5120 15.2 / 14.8 us (one workgroup of 512 threads for
// the row and all its mixes: 11.1 / 9.7 and 19.6 / 15.4; the same with every parameter vector requested ahead: no faster).
constexpr int kLnRowThreads = 512;
template <int NSEG, int SLICES>
__device__ __forceinline__ void add_pending(const RowsDeferred &d, int t, int c, int step, int C, double *x_out, double (&xv)[NSEG][4]) {
    const bool gated = d.op == ROW_GATE_ADD;
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        const int c0 = c + g * step;
        if (c0 < C) {
            long long tot[4];
            float gt[4] = {0.f, 0.f, 0.f, 0.f};
            slices_sum4<SLICES>(d.tot + (size_t)t * d.ldd + c0, d.slice, tot);
            if (gated) ld4(gt, d.gate + (size_t)t * C + c0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double y = deferred_y(d, t, tot[i]), f = gated ? (double)sigmoid_f32(gt[i]) : 1.0;
                if (d.fused) xv[g][i] = fma(y, f, xv[g][i]);
                else xv[g][i] += gated ? y * f : y;
            }
            if (x_out) st4(x_out + c0, xv[g]);
        }
    }
}
// TWO: no more than 128 registers, so that two workgroups of five to eight wavefronts fit a compute unit, for grids of more than one to each.  (Of up
// to 2048 channels it takes 132 otherwise, and the second waits for the first: us a launch of 86 / 127 rows of 1088 channels 8.2 / 9.4, with 128 7.5 /
// 8.5, of 2048 11.6 / 12.8 and 11.1 / 12.4.  Smaller grids lose 0.1 to 0.3 us to the registers that go to scratch memory.)
template <bool MIX, int NSEG, bool TWO = false>
__global__ void __launch_bounds__(kLnRowThreads, TWO ? 4 : 2) rows_ln_mix_quant_row_kernel(const LnQuantArgs a) {
    __shared__ double red0[2 * 8], red1[2 * 8], red2[8], red3[8];
    __shared__ float redf[16];
    const int t = blockIdx.x, m = blockIdx.y, C = a.C, tid = threadIdx.x, nt = blockDim.x, nw = nt >> 6, lane = tid & 63;
    const bool need_prev = MIX && a.sequence && t > 0;
    const double *xr = a.x + (size_t)t * C;
    const double *pr = !MIX ? xr : need_prev ? xr - C : a.sequence ? a.prev0 : a.prev0 + (size_t)t * a.prev_stride;
    const double *mur = MIX ? a.mu + (size_t)m * C : nullptr;
    const float *range = m == 0 ? a.range[0] : m == 1 ? a.range[1] : a.range[2];
    const double *offset = m == 0 ? a.offset[0] : m == 1 ? a.offset[1] : a.offset[2];
    double xv[NSEG][4], pv[NSEG][4], lw[NSEG][4], lb[NSEG][4], mu[NSEG][4], of[NSEG][4];
    float rg[NSEG][4];
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        const int c0 = 4 * (tid + g * nt);
        if (c0 < C) {
            ld4(xv[g], xr + c0);
            if (MIX) ld4(pv[g], pr + c0);
            ld4(lw[g], a.ln_w + c0);
            ld4(lb[g], a.ln_b + c0);
            if (MIX) ld4(mu[g], mur + c0);
            ld4(rg[g], range + c0);
            ld4(of[g], offset + c0);
            if (a.commit_src && m == 0 && (!a.sequence || t == 0)) {
                double v[4];
                ld4(v, a.commit_src + (size_t)t * C + c0);
                st4(a.commit_dst + (size_t)t * a.prev_stride + c0, v);
            }
        }
    }
    if (a.add.tot) {
        // The product before this kernel was handed on unfinished: x += y (block.py:80) or x += y * sigmoid(r)
        // (block.py:95-100), as rows_finish_kernel would have done.
        const int c = 4 * tid, step = 4 * nt;
        double *xo = a.x_out && m == 0 ? a.x_out + (size_t)t * C : nullptr;
        with_slices(a.add.slices, [&](auto count) {
            add_pending<NSEG, decltype(count)::value>(a.add, t, c, step, C, xo, xv);
            if (NSEG == 1 && need_prev) add_pending<NSEG, decltype(count)::value>(a.add, t - 1, c, step, C, nullptr, pv);
        });
    }
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        if (4 * (tid + g * nt) < C) {
#pragma unroll
            for (int i = 0; i < 4; ++i) { s[0] += xv[g][i]; if (MIX) s[1] += pv[g][i]; }
        }
    }
    bsum<2>(s, red0, nw);
    const double mean = s[0] / (double)C, meanp = s[1] / (double)C;
    double q[2] = {0.0, 0.0};
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        if (4 * (tid + g * nt) < C) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double d = xv[g][i] - mean;
                q[0] += d * d;
                if (MIX) { const double dp = pv[g][i] - meanp; q[1] += dp * dp; }
            }
        }
    }
    bsum<2>(q, red1, nw);
    const double rsd = 1.0 / sqrt(q[0] / (double)C + 1e-5), rsdp = MIX ? 1.0 / sqrt(q[1] / (double)C + 1e-5) : 0.0;
    float xs[NSEG][4];
    float amax = 0.f;
    double z[1] = {0.0};
    double *sh = !MIX || m != 0 ? nullptr : a.shift_out ? a.shift_out + (size_t)t * C : t == a.R - 1 ? a.shift_dst : nullptr;
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        const int c0 = 4 * (tid + g * nt);
        if (c0 < C) {
            double xy[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                xy[i] = lw[g][i] * ((xv[g][i] - mean) * rsd) + lb[g][i];
                double v = xy[i];
                if (MIX) {
                    const double prev = need_prev ? lw[g][i] * ((pv[g][i] - meanp) * rsdp) + lb[g][i] : pv[g][i];
                    v = xy[i] * mu[g][i] + prev * (1.0 - mu[g][i]);
                }
                xs[g][i] = (float)(v * (double)rg[g][i]);
                amax = fmaxf(amax, fabsf(xs[g][i]));
                z[0] += v * of[g][i];
            }
            if (sh) st4(sh + c0, xy);
        }
    }
    amax = wmaxf(amax);
    if (lane == 0) redf[tid >> 6] = amax;
    bsum<1>(z, red2, nw);                       // (its barrier also publishes redf)
    double S, invS, qsum[1] = {0.0};
    row_scale(row16_max((lane & 15) < nw ? redf[lane & 15] : 0.f), S, invS);
    signed char *dig = m == 0 ? a.dig[0] : m == 1 ? a.dig[1] : a.dig[2];
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        const int c0 = 4 * (tid + g * nt);
        if (c0 < C) qsum[0] += emit_quad(xs[g], invS, c0, t, C >> 6, dig);
    }
    bsum<1>(qsum, red3, nw);
    if (tid == 0) {
        (m == 0 ? a.S[0] : m == 1 ? a.S[1] : a.S[2])[t] = S;
        (m == 0 ? a.qs[0] : m == 1 ? a.qs[1] : a.qs[2])[t] = qsum[0];
        (m == 0 ? a.zp[0] : m == 1 ? a.zp[1] : a.zp[2])[t] = z[0];
    }
}

template <int NM, int NSEG, int kLT>
__global__ void __launch_bounds__(kLT) rows_ln_mix_quant_kernel(const LnQuantArgs a) {
    constexpr int m0 = 0;
#include "rwkv_rows_ln_body.inc"
}
// The same for so few rows that at most two workgroups share a compute unit: twice the registers, so that the
// parameter vectors of all of a thread's channels can be on their way at once instead of one group after the other.
template <int NM, int NSEG, int kLT>
__global__ void __launch_bounds__(kLT) __attribute__((amdgpu_waves_per_eu(1, 2))) rows_ln_mix_quant_few_kernel(const LnQuantArgs a) {
    constexpr int m0 = 0;
#include "rwkv_rows_ln_body.inc"
}
// The same with a workgroup to each mix of a row (blockIdx.y): up to 256 rows of a sequence leave a compute unit one row, four
// wavefronts that wait for its parameter vectors one group of channels after the other, of all mixes in turn.  Two or three times
// the wavefronts for the same waits, and the statistics, a few additions, done again.  Bound: those dependent loads.  Not for
// batches, whose shift rows are replaced in place: a workgroup may not write what the others of its row still read.  With the
// quantiser below, prompts of 256 tokens, before / now: 10 layers of 5120 4321 / 4049 us, 16 of 4096 4813 / 4474, 24 of 2560
// 4215 / 4057, 24 of 1024 2037 / 1998; of 150 tokens 24 of 2560 3879 / 3741.
template <int NSEG, int kLT>
__global__ void __launch_bounds__(kLT) __attribute__((amdgpu_waves_per_eu(1, 3))) rows_ln_mix_quant_split_kernel(const LnQuantArgs a) {
    constexpr int NM = 1;
    const int m0 = blockIdx.y;
#include "rwkv_rows_ln_body.inc"
}

// ---------------------------------------------------------------------------
// Row quantiser: xs = fp32(v * range), S from the row's max |xs|, digits in
// fragment order, zero-point term sum v * offset and sum q   (matmul.py:59-62,131-133).
// ---------------------------------------------------------------------------
struct QuantArgs {
    int K;                      // contraction length, multiple of 64
    const void *in;             // [R, K] float64, or float32 (the kernels' TIn): what the WKV kernels and the relu^2 tail write
    const float *range;         // [K]
    const double *offset;       // [K]
    signed char *dig;           // fragments [ceil(R/4)][K/64][1024]
    double *S, *qs, *zp;        // [R]
};

// Two / four consecutive values of a float64 or float32 row as float64.
__device__ __forceinline__ double2 row_ld2(const double *p) { return *reinterpret_cast<const double2 *>(p); }
__device__ __forceinline__ double2 row_ld2(const float *p) { const float2 f = *reinterpret_cast<const float2 *>(p); return make_double2((double)f.x, (double)f.y); }
__device__ __forceinline__ void row_ld4(const double *p, double2 &a, double2 &b) { a = row_ld2(p); b = row_ld2(p + 2); }
__device__ __forceinline__ void row_ld4(const float *p, double2 &a, double2 &b) {
    const float4 f = *reinterpret_cast<const float4 *>(p);
    a = make_double2((double)f.x, (double)f.y); b = make_double2((double)f.z, (double)f.w);
}

// kQuantSeg: 16-element segments a thread keeps in registers (rows up to 16 * kRT * kQuantSeg long in one
// read): 3 covers 12288 with registers to spare for four workgroups per compute unit, 5 covers 20480.
template <int kQuantSeg, typename TIn>
__global__ void __launch_bounds__(kRT) rows_quant_kernel(const QuantArgs a) {
    __shared__ double red[2 * kRW];
    __shared__ float redf[kRW];
    const int t = blockIdx.x, K = a.K;
    const TIn *row = static_cast<const TIn *>(a.in) + (size_t)t * K;
    // The thread that will write a 16-element group of digits reads it once: xs stays in registers
    // between the pass that finds the row's scale and the pass that forms the digits (longer rows
    // fall back to a second read).
    float xs[kQuantSeg][16];
    const bool fits = K <= kQuantSeg * 16 * kRT;
    float amax = 0.f;
    double z[1] = {0.0};
    if (fits) {
#pragma unroll
        for (int s = 0; s < kQuantSeg; ++s) {
            const int c0 = (threadIdx.x + s * kRT) * 16;
            if (c0 < K) {
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    const double2 v = row_ld2(row + c0 + i);
                    const float2 r = *reinterpret_cast<const float2 *>(a.range + c0 + i);
                    const double2 o = *reinterpret_cast<const double2 *>(a.offset + c0 + i);
                    xs[s][i] = (float)(v.x * (double)r.x);
                    xs[s][i + 1] = (float)(v.y * (double)r.y);
                    amax = fmaxf(amax, fmaxf(fabsf(xs[s][i]), fabsf(xs[s][i + 1])));
                    z[0] += v.x * o.x;
                    z[0] += v.y * o.y;
                }
            }
        }
    } else {
        for (int c = threadIdx.x; c < K; c += kRT) {
            const double v = (double)row[c];
            amax = fmaxf(amax, fabsf((float)(v * (double)a.range[c])));
            z[0] += v * a.offset[c];
        }
    }
    amax = wmaxf(amax);
    if ((threadIdx.x & 63) == 0) redf[threadIdx.x >> 6] = amax;
    rsum<1>(z, red);                       // (its barriers also publish redf)
    amax = redf[0];
#pragma unroll
    for (int w = 1; w < kRW; ++w) amax = fmaxf(amax, redf[w]);
    double S, invS;
    row_scale(amax, S, invS);
    const int KB = K >> 6;
    const int mt = t >> 2, m0 = (t & 3) * 4;
    double qsum[1] = {0.0};
    auto emit = [&](int c0, const float (&x16)[16]) {
        unsigned pl[4][4];
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int j = 0; j < 4; ++j) pl[d][j] = 0u;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            int q = __double2int_rn((double)x16[i] * invS);
            qsum[0] += (double)q;
            const int d3 = (int)(signed char)(q & 0xff); q = (q - d3) >> 8;
            const int d2 = (int)(signed char)(q & 0xff); q = (q - d2) >> 8;
            const int d1 = (int)(signed char)(q & 0xff); q = (q - d1) >> 8;
            const int sh = 8 * (i & 3);
            pl[0][i >> 2] |= (unsigned)(q & 0xff) << sh;
            pl[1][i >> 2] |= (unsigned)(d1 & 0xff) << sh;
            pl[2][i >> 2] |= (unsigned)(d2 & 0xff) << sh;
            pl[3][i >> 2] |= (unsigned)(d3 & 0xff) << sh;
        }
        const int kb = c0 >> 6, g = (c0 & 63) >> 4;
        signed char *frag = a.dig + ((size_t)mt * KB + kb) * 1024;
#pragma unroll
        for (int d = 0; d < 4; ++d)
            *reinterpret_cast<uint4 *>(frag + (16 * g + m0 + d) * 16) = make_uint4(pl[d][0], pl[d][1], pl[d][2], pl[d][3]);
    };
    if (fits) {
#pragma unroll
        for (int s = 0; s < kQuantSeg; ++s) {
            const int c0 = (threadIdx.x + s * kRT) * 16;
            if (c0 < K) emit(c0, xs[s]);
        }
    } else {
        for (int c0 = threadIdx.x * 16; c0 < K; c0 += kRT * 16) {
            float x16[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) x16[i] = (float)((double)row[c0 + i] * (double)a.range[c0 + i]);
            emit(c0, x16);
        }
    }
    rsum<1>(qsum, red);
    if (threadIdx.x == 0) { a.S[t] = S; a.qs[t] = qsum[0]; a.zp[t] = z[0]; }
}

// The same quantiser with a thread owning groups of four values (NSEG of them, 4 * kRT * NSEG values per row in
// one read): every thread of the workgroup has work whatever the row length, and few registers are held.
template <int NSEG, typename TIn>
__global__ void __launch_bounds__(kRT) rows_quant4_kernel(const QuantArgs a) {
    __shared__ double red[2 * kRW];
    __shared__ float redf[kRW];
    const int t = blockIdx.x, K = a.K, tid = threadIdx.x;
    const TIn *row = static_cast<const TIn *>(a.in) + (size_t)t * K;
    float xs[NSEG][4];
    float amax = 0.f;
    double z[1] = {0.0};
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        const int c0 = 4 * (tid + g * kRT);
        if (c0 < K) {
            double2 v0, v1;
            row_ld4(row + c0, v0, v1);
            const float4 r = *reinterpret_cast<const float4 *>(a.range + c0);
            const double2 o0 = *reinterpret_cast<const double2 *>(a.offset + c0), o1 = *reinterpret_cast<const double2 *>(a.offset + c0 + 2);
            xs[g][0] = (float)(v0.x * (double)r.x); xs[g][1] = (float)(v0.y * (double)r.y);
            xs[g][2] = (float)(v1.x * (double)r.z); xs[g][3] = (float)(v1.y * (double)r.w);
            amax = fmaxf(fmaxf(amax, fmaxf(fabsf(xs[g][0]), fabsf(xs[g][1]))), fmaxf(fabsf(xs[g][2]), fabsf(xs[g][3])));
            z[0] += v0.x * o0.x; z[0] += v0.y * o0.y; z[0] += v1.x * o1.x; z[0] += v1.y * o1.y;
        }
    }
    amax = wmaxf(amax);
    if ((tid & 63) == 0) redf[tid >> 6] = amax;
    rsum<1>(z, red);                       // (its barriers also publish redf)
    amax = redf[0];
#pragma unroll
    for (int w = 1; w < kRW; ++w) amax = fmaxf(amax, redf[w]);
    double S, invS;
    row_scale(amax, S, invS);
    const int KB = K >> 6;
    double qsum[1] = {0.0};
#pragma unroll
    for (int g = 0; g < NSEG; ++g) {
        const int c0 = 4 * (tid + g * kRT);
        if (c0 < K) qsum[0] += emit_quad(xs[g], invS, c0, t, KB, a.dig);
    }
    rsum<1>(qsum, red);
    if (tid == 0) { a.S[t] = S; a.qs[t] = qsum[0]; a.zp[t] = z[0]; }
}

// Long rows, too few of them to fill the device with workgroups of 256 threads: four threads for each one of the kernel above, with
// a quarter of its groups each (NP consecutive ones), so that four times the loads are on their way from a compute unit that has
// a row or two.  Bound: those loads.  The sums are in that kernel's order, the bits its own.  256 rows of 20480 / 16384 values, caches warm:
// 13.8 / 11.4 us by the kernel above, 10.7 / 8.5 by this.
template <int NP, typename TIn>
__global__ void __launch_bounds__(4 * kRT) rows_quant_long_kernel(const QuantArgs a) {
    __shared__ double zs[kRT], red0[8], red1[4 * kRW];
    __shared__ float redf[4 * kRW];
    const int t = blockIdx.x, K = a.K, tid = threadIdx.x, part = tid / kRT, col = tid % kRT, wave = tid >> 6, lane = tid & 63;
    const TIn *row = static_cast<const TIn *>(a.in) + (size_t)t * K;
    TIn v[NP][4];
    float r[NP][4];
    double o[NP][4];
#pragma unroll
    for (int g = 0; g < NP; ++g) {
        const int c0 = 4 * (col + (part * NP + g) * kRT);
        if (c0 < K) {
            ld4(v[g], row + c0);
            ld4(r[g], a.range + c0);
            ld4(o[g], a.offset + c0);
        }
    }
    float xs[NP][4];
    float amax = 0.f;
#pragma unroll
    for (int g = 0; g < NP; ++g) {
        if (4 * (col + (part * NP + g) * kRT) < K) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                xs[g][i] = (float)((double)v[g][i] * (double)r[g][i]);
                amax = fmaxf(amax, fabsf(xs[g][i]));
            }
        }
    }
    amax = wmaxf(amax);
    if (lane == 0) redf[wave] = amax;
    // the zero-point sum in that kernel's order: a quarter goes on from where the one before it ended
    double z = 0.0;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        if (part == p) {
            if (p > 0) z = zs[col];
#pragma unroll
            for (int g = 0; g < NP; ++g) {
                if (4 * (col + (part * NP + g) * kRT) < K) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) z += (double)v[g][i] * o[g][i];
                }
            }
            if (p < 3) zs[col] = z;
            else {
                z = wsum(z);
                if (lane == 0) red0[wave - 3 * kRW] = z;
            }
        }
        __syncthreads();
    }
    double zp = 0.0;
    amax = redf[0];
#pragma unroll
    for (int w = 0; w < kRW; ++w) zp += red0[w];
#pragma unroll
    for (int w = 1; w < 4 * kRW; ++w) amax = fmaxf(amax, redf[w]);
    double S, invS;
    row_scale(amax, S, invS);
    double qsum = 0.0;
#pragma unroll
    for (int g = 0; g < NP; ++g) {
        const int c0 = 4 * (col + (part * NP + g) * kRT);
        if (c0 < K) qsum += emit_quad(xs[g], invS, c0, t, K >> 6, a.dig);
    }
    qsum = wsum(qsum);
    if (lane == 0) red1[wave] = qsum;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 4 * kRW; ++w) qsum += red1[w];
        a.S[t] = S; a.qs[t] = qsum; a.zp[t] = zp;
    }
}

// A handful of long rows (one token of a wide ffn): one workgroup per row would pull the whole row and its
// range / offset vectors through a single compute unit.  Two launches instead, G workgroups per row: the first
// leaves each part's max |xs| and zero-point share in `part`, the second turns them into the row's scale and
// writes the digits of its part.  The sum of the fixed-point values is added up with atomics: integers below
// 2^53, exact in any order.
constexpr int kQuantPartSeg = 3;        // groups of four values per thread: parts of up to 3072 values

struct QuantPartArgs {
    QuantArgs q;
    int G, quads_per_part;
    double *part;               // [R][G][2]: max |xs|, zero-point share
};

template <bool EMIT, typename TIn>
__global__ void __launch_bounds__(kRT) rows_quant_part_kernel(const QuantPartArgs a) {
    __shared__ double red[2 * kRW];
    __shared__ float redf[kRW];
    const int g = blockIdx.x, t = blockIdx.y, K = a.q.K, tid = threadIdx.x;
    const TIn *row = static_cast<const TIn *>(a.q.in) + (size_t)t * K;
    const int q0 = g * a.quads_per_part, q1 = min(q0 + a.quads_per_part, K >> 2);
    float xs[kQuantPartSeg][4];
    float amax = 0.f;
    double z[1] = {0.0};
#pragma unroll
    for (int s = 0; s < kQuantPartSeg; ++s) {
        const int qi = q0 + tid + s * kRT;
        if (qi < q1) {
            const int c0 = 4 * qi;
            double2 v0, v1;
            row_ld4(row + c0, v0, v1);
            const float4 r = *reinterpret_cast<const float4 *>(a.q.range + c0);
            xs[s][0] = (float)(v0.x * (double)r.x); xs[s][1] = (float)(v0.y * (double)r.y);
            xs[s][2] = (float)(v1.x * (double)r.z); xs[s][3] = (float)(v1.y * (double)r.w);
            if (!EMIT) {
                const double2 o0 = *reinterpret_cast<const double2 *>(a.q.offset + c0), o1 = *reinterpret_cast<const double2 *>(a.q.offset + c0 + 2);
                amax = fmaxf(fmaxf(amax, fmaxf(fabsf(xs[s][0]), fabsf(xs[s][1]))), fmaxf(fabsf(xs[s][2]), fabsf(xs[s][3])));
                z[0] += v0.x * o0.x; z[0] += v0.y * o0.y; z[0] += v1.x * o1.x; z[0] += v1.y * o1.y;
            }
        }
    }
    double *part = a.part + (size_t)t * a.G * 2;
    if (!EMIT) {
        amax = wmaxf(amax);
        if ((tid & 63) == 0) redf[tid >> 6] = amax;
        rsum<1>(z, red);                   // (its barriers also publish redf)
        if (tid == 0) {
            amax = redf[0];
#pragma unroll
            for (int w = 1; w < kRW; ++w) amax = fmaxf(amax, redf[w]);
            part[2 * g] = (double)amax; part[2 * g + 1] = z[0];
            if (g == 0) a.q.qs[t] = 0.0;
        }
        return;
    }
    float am = 0.f;
    double zp = 0.0;
    for (int i = 0; i < a.G; ++i) { am = fmaxf(am, (float)part[2 * i]); zp += part[2 * i + 1]; }     // fixed order
    double S, invS;
    row_scale(am, S, invS);
    const int KB = K >> 6;
    double qsum[1] = {0.0};
#pragma unroll
    for (int s = 0; s < kQuantPartSeg; ++s) {
        const int qi = q0 + tid + s * kRT;
        if (qi < q1) qsum[0] += emit_quad(xs[s], invS, 4 * qi, t, KB, a.q.dig);
    }
    rsum<1>(qsum, red);
    if (tid == 0) {
        atomicAdd(a.q.qs + t, qsum[0]);
        if (g == 0) { a.q.S[t] = S; a.q.zp[t] = zp; }
    }
}

// ---------------------------------------------------------------------------
// GEMM: tot[t, j] = sum_k q[t, k] * (code[k, j] - 128), exact in int64.
// Workgroup = 8 wavefronts = 64 tokens x 128 (or 160) columns; wavefront (wm, wn) holds
// 4 M-tiles x 4 (or 5) N-tiles of accumulators; variants for at most 32 and at most 8 rows
// follow.  With few rows the contraction is split over several workgroups; each split writes
// its own slice of integer totals and the tail kernel adds the slices (integer sums: exact in
// any order).
//
// Launch order.  Workgroups are handed to the 8 XCDs round robin, and each XCD has its own L2.  The
// grid is 1-D and workgroup i works for XCD i % 8 on that XCD's own row blocks (row block r belongs
// to XCD r % 8), walking through the column blocks with the row blocks innermost: the digit
// fragments of an XCD's rows (a few hundred KB) stay in its L2 for the whole product, and a weight
// block fetched for one row block is reused by the next.  Without this every XCD pulls every digit
// fragment through the fabric once per column block.  With fewer row blocks than XCDs (a batch of
// single tokens) the column blocks are dealt out to the XCDs instead.
// ---------------------------------------------------------------------------
constexpr int kXcds = 8;
struct GemmArgs {
    // up to kRowsMaxProducts products of one shape share a launch (the grid's split index also counts products)
    const signed char *dig[kRowsMaxProducts];   // fragments [MT][KB][1024]
    const uint8_t *w16[kRowsMaxProducts];       // blocks [NT][KB][1024]
    const double *S[kRowsMaxProducts], *qs[kRowsMaxProducts], *zp[kRowsMaxProducts];
    double *out[kRowsMaxProducts];
    long long *tot;             // [products][splits][4*MT][ldd]
    int MT, NT, KB, ldd, kb_per_split, split;     // split > 1: the contraction is split, each part writes its slice of tot
    size_t slice;                   // elements between the slices of tot
    int gx, gy, gz, per_xcd, by_rows;   // logical grid (column blocks, row blocks, splits x products) behind the 1-D launch
    // when the contraction is not split the tail of the product is applied here (see rows_finish_kernel)
    int tail, R, N;                 // tail < 0: totals only
    const float *gate;
    // NT2 > 0: the launch holds two products of different widths (same rows, same contraction, not split): product 1 has
    // NT2 tiles, N2 columns and tail2, and its workgroups follow product 0's
    int NT2, N2, tail2;
    int apart, apart2;              // few rows: round y as rows_finish_kernel does (see rounded_apart)
    // part non-null (few rows, product 0 with the relu^2 tail): what the quantiser of its result needs of every row and column
    // tile, {max |xs|, zero-point share} at [row][tile], and qs of the operand to be, cleared
    double2 *part;
    const float *next_range;
    const double *next_offset;
    double *next_qs;
};
// Columns and tail of the product a workgroup works for (kept apart from the arguments: a modified copy of those would
// live in scratch memory).
struct GemmCols { int NT, N, tail; bool apart = false; };

// Weights of the few-row kernels.  STREAM: past the caches, which keeps the digits and the next kernels' vectors there: 8
// sequences at 3B 2.25 -> 2.08 ms a step, at 14B 5.75 -> 5.30; 32 sequences (9..32-row kernel) 3.20 -> 3.15 and 6.66 -> 6.59.  Of a
// model that fits the Infinity Cache the weights are kept: 8 layers of 1024, 8 sequences 334 us, streamed 360.
template <bool STREAM>
__device__ __forceinline__ v4i ldw(const v4i *p) { return STREAM ? __builtin_nontemporal_load(p) : *p; }

constexpr int kGemmNT = 8, kGemmWideNT = 10, kGemmNarrowNT = 5;     // N-tiles per workgroup
constexpr int kWideRing = 4;                     // LDS buffers of the 64 x 160 variant

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every global load
// the wavefront has in flight, which would drain the prefetched contraction blocks at every step.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16 bytes per lane from global memory straight into LDS at lds_byte_offset + 16 * lane (the offset is uniform
// for the wavefront and travels in M0; one wait state between writing M0 and the load that reads it).
__device__ __forceinline__ void dma16(const v4i *g, unsigned lds_byte_offset) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(g), "s"(lds_byte_offset) : "memory");
}

// The same past the caches (as ldw).
__device__ __forceinline__ void dma16_stream(const v4i *g, unsigned lds_byte_offset) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" :: "v"(g), "s"(lds_byte_offset) : "memory");
}

// Accumulators of one wavefront (GM M-tiles x GN N-tiles from (mt0, nt0)) to totals or, when the contraction is not
// split, straight through the product's tail.  Lane 16g + n, register i <-> digit i of token 4*mt + g, column 16*nt + n.
//
// Nothing overlaps this part of a workgroup but the other workgroup of its compute unit, so it is kept short: the
// digit sums are joined in float64 (exact while 64 KB products of 2^30 x 2^7 stay below 2^53; a third of the
// instructions of the 64-bit integer form), the tail is chosen once and not per element, and a residual tail requests
// the next M-tile's old values before it stores this one's (a store and the load after it may not be exchanged by the
// compiler: element by element each of them waited for a round trip).  1024 tokens at width 2560, before and after: k, v, r
// 75.5 and 71.8 us, ffn key 93.1 and 89.4, att output and ffn receptance 35.1 and 30.2 (median), ffn value 94.8 and 87.7.
template <int TAIL, int GM, int GN>
__device__ __forceinline__ void gemm_tail(const GemmArgs &a, int N, bool apart, const v4i (&acc)[GM][GN], int mt0, int nt0, int mat, int lane) {
    const int g = lane >> 4, n = lane & 15;
    const double *Sv = mat == 0 ? a.S[0] : mat == 1 ? a.S[1] : a.S[2];
    const double *qsv = mat == 0 ? a.qs[0] : mat == 1 ? a.qs[1] : a.qs[2];
    const double *zpv = mat == 0 ? a.zp[0] : mat == 1 ? a.zp[1] : a.zp[2];
    double *outv = mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : a.out[2];
    constexpr bool kAdd = TAIL == ROW_ADD || TAIL == ROW_GATE_ADD;
    const bool exact53 = a.KB <= 512;
    double old[2][GN];
    float gate[2][GN];
    auto at = [&](int i, int j) { return (size_t)min(4 * (mt0 + i) + g, a.R - 1) * N + min(16 * (nt0 + j) + n, N - 1); };   // (clamped: loads stay in bounds)
    auto fetch = [&](int i) {
#pragma unroll
        for (int j = 0; j < GN; ++j) {
            if (kAdd) old[i & 1][j] = outv[at(i, j)];
            if (TAIL == ROW_GATE_ADD) gate[i & 1][j] = a.gate[at(i, j)];
        }
    };
    fetch(0);
#pragma unroll
    for (int i = 0; i < GM; ++i) {
        if (i + 1 < GM) fetch(i + 1);
        const int t = 4 * (mt0 + i) + g;
        const bool live = t < a.R;
        const int tc = live ? t : a.R - 1;
        // y = S tot + (128 S q + zp), or with zp added last, as where slices are added up (-0.0 changes nothing)
        const double S = Sv[tc], sq = 128.0 * (S * qsv[tc]), zp = zpv[tc], add = apart ? sq : sq + zp, last = apart ? zp : -0.0;
#pragma unroll
        for (int j = 0; j < GN; ++j) {
            const v4i d = acc[i][j];
            double tot;
            if (exact53) tot = fma(fma(fma((double)d.x, 256.0, (double)d.y), 256.0, (double)d.z), 256.0, (double)d.w);
            else tot = (double)(((((long long)d.x * 256 + d.y) * 256 + d.z) * 256) + d.w);
            const int col = 16 * (nt0 + j) + n;
            const double y = (S * tot + add) + last;
            const size_t o = (size_t)t * N + col;
            if (live && col < N) {
                if (TAIL == ROW_STORE) outv[o] = y;
                else if (TAIL == ROW_STORE_F32) reinterpret_cast<float *>(outv)[o] = (float)y;
                else if (TAIL == ROW_RELU2) {                                                       // block.py:97, kept as float32 (see RowTail)
                    const double r = y > 0.0 ? y : 0.0;
                    reinterpret_cast<float *>(outv)[o] = (float)(r * r);
                }
                else if (TAIL == ROW_ADD) outv[o] = old[i & 1][j] + y;                              // block.py:80
                else outv[o] = old[i & 1][j] + y * (double)sigmoid_f32(gate[i & 1][j]);             // block.py:95-100; the gate in float32 as in the single-token kernel
            }
        }
    }
}

template <int GM, int GN>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs &a, const GemmCols &cols, const v4i (&acc)[GM][GN], int mt0, int nt0, int mat,
                                              int bz, int lane) {
    switch (cols.tail) {
        case ROW_STORE: return gemm_tail<ROW_STORE, GM, GN>(a, cols.N, cols.apart, acc, mt0, nt0, mat, lane);
        case ROW_STORE_F32: return gemm_tail<ROW_STORE_F32, GM, GN>(a, cols.N, cols.apart, acc, mt0, nt0, mat, lane);
        case ROW_RELU2: return gemm_tail<ROW_RELU2, GM, GN>(a, cols.N, cols.apart, acc, mt0, nt0, mat, lane);
        case ROW_ADD: return gemm_tail<ROW_ADD, GM, GN>(a, cols.N, cols.apart, acc, mt0, nt0, mat, lane);
        case ROW_GATE_ADD: return gemm_tail<ROW_GATE_ADD, GM, GN>(a, cols.N, cols.apart, acc, mt0, nt0, mat, lane);
        default: break;
    }
    const int g = lane >> 4, n = lane & 15;
    long long *totv = a.tot + (size_t)(mat * a.split + bz) * a.slice;      // this part's slice
#pragma unroll
    for (int i = 0; i < GM; ++i) {
        if (mt0 + i >= a.MT) continue;
#pragma unroll
        for (int j = 0; j < GN; ++j) {
            if (nt0 + j >= cols.NT) continue;
            const v4i d = acc[i][j];
            totv[(size_t)(4 * (mt0 + i) + g) * a.ldd + 16 * (nt0 + j) + n] = ((((long long)d.x * 256 + d.y) * 256 + d.z) * 256) + d.w;
        }
    }
}

// One workgroup of the product: 64 tokens x 16*WN*GN columns, WM*WN wavefronts as WM x WN, each 16/WM M-tiles x GN
// N-tiles, RING LDS buffers.  <4, 4, 2, 3> is the general shape (8 wavefronts of 4 x 4 tiles, two workgroups per
// compute unit); <5, 4, 2, 4> (4 x 5 tiles, one workgroup per compute unit) is used where it turns a grid of 1.25
// workgroups per compute unit into exactly one (2560 columns: 16 column blocks instead of 20).  <5, 8, 1, 4> (64 x 80: eight wavefronts of 2 x 5
// tiles) serves grids that leave compute units idle (general_narrow).
template <int GN, int WM, int WN, int RING, bool STREAM>
__device__ __forceinline__ void gemm8_body(const GemmArgs a) {
    // Both operands of a contraction block are fetched once per workgroup into LDS and read from there by
    // the wavefronts that need each fragment (one barrier per block).
    constexpr int kGN = GN, kNT = WN * GN, kGM = 16 / WM, kNW = WN * WM;
    constexpr int kGemmFrags = 16 + kNT;                // fragments of one contraction block: 16 M-tiles of digits, kNT N-tiles of weights
    constexpr int kGemmLoads = (kGemmFrags + kNW - 1) / kNW;    // per thread and contraction block (wave w fetches fragments w, w + kNW, ...)
    constexpr int kSlots = kNW * kGemmLoads, kGemmRing = RING;
    __shared__ v4i frag[kGemmRing][kSlots][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int xcd = blockIdx.x % kXcds;
    int item = blockIdx.x / kXcds, bx, by, bz;
    if (a.by_rows) {                                    // (split, column block, row slot) of this XCD, row slot fastest
        const int rslot = item % a.per_xcd; item /= a.per_xcd;
        bx = item % a.gx; bz = item / a.gx;
        by = xcd + kXcds * rslot;
    } else {                                            // few row blocks: the XCDs share out the column blocks instead
        const int cslot = item % a.per_xcd; item /= a.per_xcd;
        by = item % a.gy; bz = item / a.gy;
        bx = xcd + kXcds * cslot;
    }
    if (by >= a.gy || bx >= a.gx || bz >= a.gz) return;
    int mat = bz / a.split;                             // which product; then which part of its contraction
    bz -= mat * a.split;
    GemmCols cols = {a.NT, a.N, a.tail, a.apart != 0};
    if (a.NT2 > 0) {                                    // two products side by side: gx counts the column blocks of both
        const int gx0 = (a.NT + kNT - 1) / kNT;
        if (bx >= gx0) { bx -= gx0; mat = 1; cols = GemmCols{a.NT2, a.N2, a.tail2, a.apart2 != 0}; }
    }
    const signed char *dig = mat == 0 ? a.dig[0] : mat == 1 ? a.dig[1] : a.dig[2];
    const uint8_t *w16 = mat == 0 ? a.w16[0] : mat == 1 ? a.w16[1] : a.w16[2];
    const int mt0 = by * 16 + wm * kGM, nt0 = bx * kNT + wn * kGN;
    const int kb0 = bz * a.kb_per_split;
    int kb1 = kb0 + a.kb_per_split;
    if (kb1 > a.KB) kb1 = a.KB;
    if (kb0 >= kb1) return;                             // (uniform for the workgroup)
    const int nk = kb1 - kb0;

    const v4i *src[kGemmLoads];
#pragma unroll
    for (int i = 0; i < kGemmLoads; ++i) {
        const int f = wave + kNW * i;                   // fragment this thread helps to fetch
        if (f < 16) {
            int mt = by * 16 + f;
            if (mt >= a.MT) mt = a.MT - 1;              // clamped: loads stay unconditional, results are dropped
            src[i] = reinterpret_cast<const v4i *>(dig + ((size_t)mt * a.KB + kb0) * 1024) + lane;
        } else {
            int nt = bx * kNT + (f - 16 < kNT ? f - 16 : 0);   // (slots past the last fragment: a copy nobody reads)
            if (nt >= cols.NT) nt = cols.NT - 1;
            src[i] = reinterpret_cast<const v4i *>(w16 + ((size_t)nt * a.KB + kb0) * 1024) + lane;
        }
    }
    v4i acc[kGM][kGN];
#pragma unroll
    for (int i = 0; i < kGM; ++i)
#pragma unroll
        for (int j = 0; j < kGN; ++j) acc[i][j] = v4i{0, 0, 0, 0};

    // Contraction blocks travel from memory straight into a ring of kGemmRing LDS buffers (direct-to-LDS
    // loads: no registers, no LDS write instructions); block K + kGemmRing - 1 is requested in step K, into the
    // buffer block K - 1 has just left.  The compiler does not see these loads, so the waits are written here:
    // before the barrier of step K a wavefront waits until only the requests of the blocks after K are still out.
    const unsigned lds0 = (unsigned)(size_t)&frag[0][0][0] + (unsigned)wave * 1024u;
#define RWKV_GEMM_DMA(SLOT, K)                                                                       \
    do {                                                                                             \
        const size_t o_ = (size_t)((K) < nk ? (K) : nk - 1) * 64; /* past the end: the last block again (unused) */ \
        _Pragma("unroll") for (int i = 0; i < kGemmLoads; ++i) {                                     \
            if (STREAM && kNW * i >= 16) dma16_stream(src[i] + o_, lds0 + (unsigned)(((SLOT) * kSlots + kNW * i) * 1024)); \
            else dma16(src[i] + o_, lds0 + (unsigned)(((SLOT) * kSlots + kNW * i) * 1024));          \
        }                                                                                            \
    } while (0)
#define RWKV_GEMM_STEP(SLOT, K)                                                                      \
    {                                                                                                \
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" :: "n"((kGemmRing - 2) * kGemmLoads) : "memory"); \
        v4i Bv_[kGN];                                                                                \
        _Pragma("unroll") for (int j = 0; j < kGN; ++j) {                                            \
            Bv_[j] = frag[SLOT][16 + wn * kGN + j][lane];                                            \
        }                                                                                            \
        v4i Av_ = frag[SLOT][wm * kGM][lane], Aw_ = frag[SLOT][wm * kGM + 1][lane];                  \
        /* the next block is requested after this step's first LDS reads are on their way, and the wavefront */ \
        /* holds the higher issue priority while it has matrix instructions to issue (measured: -3 %)        */ \
        RWKV_GEMM_DMA(((SLOT) + kGemmRing - 1) % kGemmRing, (K) + kGemmRing - 1);                    \
        __builtin_amdgcn_s_setprio(1);                                                               \
        _Pragma("unroll") for (int i = 0; i < kGM; ++i) {                                            \
            const v4i An_ = frag[SLOT][wm * kGM + (i + 2 < kGM ? i + 2 : i)][lane];   /* two groups ahead */ \
            _Pragma("unroll") for (int j = 0; j < kGN; ++j)                                          \
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(Av_, Bv_[j], acc[i][j], 0, 0, 0);  \
            Av_ = Aw_; Aw_ = An_;                                                                    \
        }                                                                                            \
        __builtin_amdgcn_s_setprio(0);                                                               \
        __builtin_amdgcn_sched_group_barrier(0x100, kGN + 3, 0);                                     \
        _Pragma("unroll") for (int i = 0; i < kGM; ++i) {                                            \
            __builtin_amdgcn_sched_group_barrier(0x008, kGN, 0);                                     \
            if (i + 3 < kGM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      \
        }                                                                                            \
    }
#pragma unroll
    for (int s = 0; s + 1 < kGemmRing; ++s) RWKV_GEMM_DMA(s, s);
    int k0 = 0;
    for (; k0 + kGemmRing <= nk; k0 += kGemmRing) {     // whole turns of the ring: the buffer of a step is a constant
#pragma unroll
        for (int s = 0; s < kGemmRing; ++s) RWKV_GEMM_STEP(s, k0 + s)
    }
#pragma unroll
    for (int s = 0; s + 1 < kGemmRing; ++s)
        if (k0 + s < nk) RWKV_GEMM_STEP(s, k0 + s)
#undef RWKV_GEMM_STEP
#undef RWKV_GEMM_DMA
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // nothing of this wavefront may still be writing LDS when it leaves
    gemm_epilogue<kGM, kGN>(a, cols, acc, mt0, nt0, mat, bz, lane);
}

template <bool STREAM>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) gemm8_kernel(const GemmArgs a) {
    gemm8_body<4, 4, 2, 3, STREAM>(a);
}
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm8_wide_kernel(const GemmArgs a) {
    gemm8_body<5, 4, 2, kWideRing, false>(a);
}
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 4))) gemm8_narrow_kernel(const GemmArgs a) {
    gemm8_body<5, 8, 1, kWideRing, false>(a);
}

// ---------------------------------------------------------------------------
// The same product for at most 32 rows (a batch of single tokens): the weights are read once and
// hardly reused, so what counts is how many weight bytes a compute unit has in flight.  Workgroup =
// 4 wavefronts side by side = 8 M-tiles x 8 N-tiles (wavefront: 8 x 2); a contraction block is 8 digit
// fragments + 8 weight fragments, fetched kSkinnyAhead blocks ahead (48 KiB of weights per workgroup).  Up to 16 rows
// have four M-tiles: a compute unit draws 12 instead of 16 KB a block (8 layers of 4096, 16 sequences 905 -> 869 us a step, of 5120, 9 1054 -> 1017).
// ---------------------------------------------------------------------------
constexpr int kSkinnyMT = 8, kSkinnyGN = 2, kSkinnyNT = 4 * kSkinnyGN;
constexpr int kSkinnyAhead = 6;

template <int MT, bool STREAM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm8_skinny_kernel(const GemmArgs a) {
    static_assert(MT == 4 || MT == 8, "wavefront w fetches the digit fragments w and, of eight, w + 4, and the weight fragments w and w + 4");
    __shared__ v4i frag[2][MT + kSkinnyNT][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xcd = blockIdx.x % kXcds;
    int item = blockIdx.x / kXcds;
    const int cslot = item % a.per_xcd; item /= a.per_xcd;      // the XCDs share out the column blocks
    int bx = xcd + kXcds * cslot;
    int bz = item;
    if (bx >= a.gx || bz >= a.gz) return;
    int mat = bz / a.split;
    bz -= mat * a.split;
    GemmCols cols = {a.NT, a.N, a.tail, a.apart != 0};
    if (a.NT2 > 0) {                                    // two products side by side: gx counts the column blocks of both
        const int gx0 = (a.NT + kSkinnyNT - 1) / kSkinnyNT;
        if (bx >= gx0) { bx -= gx0; mat = 1; cols = GemmCols{a.NT2, a.N2, a.tail2, a.apart2 != 0}; }
    }
    const signed char *dig = mat == 0 ? a.dig[0] : mat == 1 ? a.dig[1] : a.dig[2];
    const uint8_t *w16 = mat == 0 ? a.w16[0] : mat == 1 ? a.w16[1] : a.w16[2];
    const int nt0 = bx * kSkinnyNT + wave * kSkinnyGN;
    const int kb0 = bz * a.kb_per_split;
    int kb1 = kb0 + a.kb_per_split;
    if (kb1 > a.KB) kb1 = a.KB;
    if (kb0 >= kb1) return;                             // (uniform for the workgroup)
    const int nk = kb1 - kb0;

    const v4i *src[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {                       // clamped: loads stay unconditional, results are dropped
        const int mt = min(wave + 4 * i, a.MT - 1), nt = min(bx * kSkinnyNT + wave + 4 * i, cols.NT - 1);
        src[i] = reinterpret_cast<const v4i *>(dig + ((size_t)mt * a.KB + kb0) * 1024) + lane;
        src[2 + i] = reinterpret_cast<const v4i *>(w16 + ((size_t)nt * a.KB + kb0) * 1024) + lane;
    }
    v4i acc[MT][kSkinnyGN];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < kSkinnyGN; ++j) acc[i][j] = v4i{0, 0, 0, 0};

    static_assert(kSkinnyAhead == 6, "six named stages below");
    struct Fly { v4i v0, v1, v2, v3; };                 // named members, not an array: they must stay registers
    Fly fly0, fly1, fly2, fly3, fly4, fly5;
#define RWKV_SKINNY_FETCH(F, K)                                                                      \
    do {                                                                                             \
        const size_t o_ = (size_t)((K) < nk ? (K) : nk - 1) * 64; /* past the end: the last block again (unused) */ \
        F.v0 = src[0][o_]; if (MT == 8) F.v1 = src[1][o_]; F.v2 = ldw<STREAM>(src[2] + o_); F.v3 = ldw<STREAM>(src[3] + o_); \
    } while (0)
#define RWKV_SKINNY_PARK(F, B)                                                                       \
    do {                                                                                             \
        frag[B][wave][lane] = F.v0; if (MT == 8) frag[B][wave + 4][lane] = F.v1;                     \
        frag[B][MT + wave][lane] = F.v2; frag[B][MT + 4 + wave][lane] = F.v3;                        \
    } while (0)
    // (same step as gemm8_body: the next block is parked, and its registers refilled, piece by piece between
    // this block's groups of matrix instructions.  With one wavefront to a SIMD nothing else hides the first LDS reads of a step: the last
    // groups of the step before are multiplied behind its barrier.  32 sequences, before / now: 8 layers of 5120 1209 / 1179 us a step, of 4096 1010 /
    // 986, 12 of 2560 1060 / 1050, 24 of 1024 1208 / 1182; more of them change nothing, eight blocks ahead instead of six lose 1 %, eight
    // wavefronts of half the rows gain less than 1 % with 32 rows and lose as much with 16)
#define RWKV_SKINNY_MOVE(FN, I, V, B, O)                                                             \
    { frag[B][((I) < 2 ? 0 : MT - 8) + wave + 4 * (I)][lane] = FN.V; FN.V = (I) < 2 ? src[I][O] : ldw<STREAM>(src[I] + (O)); }
#define RWKV_SKINNY_GROUP(I, A, B)                                                                   \
    _Pragma("unroll") for (int j = 0; j < kSkinnyGN; ++j)                                            \
        acc[I][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, (B)[j], acc[I][j], 0, 0, 0);
#define RWKV_SKINNY_STEP(FN, K, FIRST)                                                               \
    {                                                                                                \
        const int buf_ = (K) & 1;                                                                    \
        const size_t on_ = (size_t)((K) + 1 + kSkinnyAhead < nk ? (K) + 1 + kSkinnyAhead : nk - 1) * 64; \
        lds_barrier();                                                                               \
        v4i Bv_[kSkinnyGN], Av_[MT];                                                                 \
        _Pragma("unroll") for (int j = 0; j < kSkinnyGN; ++j)                                        \
            Bv_[j] = frag[buf_][MT + wave * kSkinnyGN + j][lane];                                    \
        Av_[0] = frag[buf_][0][lane]; Av_[1] = frag[buf_][1][lane];                                  \
        __builtin_amdgcn_sched_barrier(0);                                                           \
        RWKV_SKINNY_MOVE(FN, 0, v0, buf_ ^ 1, on_)                                                   \
        if (!(FIRST)) { _Pragma("unroll") for (int d = 0; d < kLate; ++d) RWKV_SKINNY_GROUP(MT - kLate + d, Al[d], Bl) }  \
        __builtin_amdgcn_sched_barrier(0);                                                           \
        _Pragma("unroll") for (int i = 0; i < MT - kLate; ++i) {                                     \
            if (i + 2 < MT) Av_[i + 2] = frag[buf_][i + 2][lane];                                    \
            if (MT == 8 && i == 0) RWKV_SKINNY_MOVE(FN, 1, v1, buf_ ^ 1, on_)                        \
            if (i == (MT == 8 ? 2 : 0)) RWKV_SKINNY_MOVE(FN, 2, v2, buf_ ^ 1, on_)                   \
            if (i == (MT == 8 ? 4 : 1)) RWKV_SKINNY_MOVE(FN, 3, v3, buf_ ^ 1, on_)                   \
            RWKV_SKINNY_GROUP(i, Av_[i], Bv_)                                                        \
            __builtin_amdgcn_sched_barrier(0);                                                       \
        }                                                                                            \
        _Pragma("unroll") for (int d = 0; d < kLate; ++d) Al[d] = Av_[MT - kLate + d];               \
        _Pragma("unroll") for (int j = 0; j < kSkinnyGN; ++j) Bl[j] = Bv_[j];                        \
    }
    constexpr int kLate = MT == 8 ? 2 : 1;
    v4i Al[kLate], Bl[kSkinnyGN];
    RWKV_SKINNY_FETCH(fly0, 0); RWKV_SKINNY_FETCH(fly1, 1); RWKV_SKINNY_FETCH(fly2, 2);
    RWKV_SKINNY_FETCH(fly3, 3); RWKV_SKINNY_FETCH(fly4, 4); RWKV_SKINNY_FETCH(fly5, 5);
    RWKV_SKINNY_PARK(fly0, 0);
    RWKV_SKINNY_FETCH(fly0, kSkinnyAhead);
    RWKV_SKINNY_STEP(fly1, 0, true)
    int k0 = 1;
    for (; k0 + kSkinnyAhead <= nk; k0 += kSkinnyAhead) {      // whole rounds: no branch between the steps
        RWKV_SKINNY_STEP(fly2, k0, false)
        RWKV_SKINNY_STEP(fly3, k0 + 1, false)
        RWKV_SKINNY_STEP(fly4, k0 + 2, false)
        RWKV_SKINNY_STEP(fly5, k0 + 3, false)
        RWKV_SKINNY_STEP(fly0, k0 + 4, false)
        RWKV_SKINNY_STEP(fly1, k0 + 5, false)
    }
    if (k0 < nk) RWKV_SKINNY_STEP(fly2, k0, false)
    if (k0 + 1 < nk) RWKV_SKINNY_STEP(fly3, k0 + 1, false)
    if (k0 + 2 < nk) RWKV_SKINNY_STEP(fly4, k0 + 2, false)
    if (k0 + 3 < nk) RWKV_SKINNY_STEP(fly5, k0 + 3, false)
    if (k0 + 4 < nk) RWKV_SKINNY_STEP(fly0, k0 + 4, false)
#pragma unroll
    for (int d = 0; d < kLate; ++d) RWKV_SKINNY_GROUP(MT - kLate + d, Al[d], Bl)
#undef RWKV_SKINNY_GROUP
#undef RWKV_SKINNY_STEP
#undef RWKV_SKINNY_MOVE
#undef RWKV_SKINNY_PARK
#undef RWKV_SKINNY_FETCH
    gemm_epilogue<MT, kSkinnyGN>(a, cols, acc, 0, nt0, mat, bz, lane);
}

// ---------------------------------------------------------------------------
// The same product for at most 8 rows (MT <= 2 M-tiles: a single token of a shape the persistent kernel does
// not serve, a small batch), and for up to 32 where the matrix is small (vec_rows): pure weight streaming.  No LDS staging and no barrier in the loop: a workgroup has NTW
// column tiles and the whole contraction, its NW wavefronts take every NW-th block (together they read the tiles'
// blocks in order) and each keeps U blocks per tile in flight on its own, so that a slow load holds up one wavefront,
// not the workgroup.  The digit fragments (L2-resident) are read by every wavefront itself, once for its NTW tiles.
// The wavefronts' sums are added in LDS, each sum by a wavefront of its own that also writes it.
//
// Bound: the latency of a few dependent loads per wavefront, then HBM.  So the blocks are spread over as many wavefronts
// as are resident at once (vec_shape), which needs no second launch: whole contractions, or slices where the next kernel adds them up
// (vec_split); wide products take
// several tiles per wavefront, since for two M-tiles the digits are twice a tile's bytes.  8 rows at 2560 channels (us per
// launch), 4 wavefronts of one tile with 8 blocks in flight / this: k, v, r 10.1 / 6.4, att output 7.4 / 4.9, ffn key and
// receptance 12.7 + 6.4 / 8.4, ffn value 15.5 / 11.1 (7.5 in three slices: see vec_split), head 43 / 24.9.
// ---------------------------------------------------------------------------
constexpr int kVecMT = 2, kVecMTMax = 8;

// The relu^2 tail of one tile (as gemm_tail's), and the tile's share of what rows_quant_tiles_kernel needs to know of the rows.
__device__ __forceinline__ void relu2_part(const GemmArgs &a, const v4i d, int m, int nt, int lane) {
    const int g = lane >> 4, n = lane & 15, t = 4 * m + g, col = 16 * nt + n;
    const bool live = t < a.R;
    const int tc = live ? t : a.R - 1;
    const double tot = (double)(((((long long)d.x * 256 + d.y) * 256 + d.z) * 256) + d.w);
    const double sq = 128.0 * (a.S[0][tc] * a.qs[0][tc]), zp = a.zp[0][tc];
    const bool apart = a.MT > 2 && a.apart;             // (up to 8 rows whole contractions always ended here)
    const double y = (a.S[0][tc] * tot + (apart ? sq : sq + zp)) + (apart ? zp : -0.0), r = y > 0.0 ? y : 0.0;
    const float h = (float)(r * r);
    if (live) reinterpret_cast<float *>(a.out[0])[(size_t)t * a.N + col] = h;
    const double v = live ? (double)h : 0.0;
    const float amax = row16_max(fabsf((float)(v * (double)a.next_range[col])));
    const double z = row16_sum(v * a.next_offset[col]);
    if (live && n == 0) {
        a.part[(size_t)t * a.NT + nt] = make_double2((double)amax, z);
        if (nt == 0) a.next_qs[t] = 0.0;
    }
}

// ROUNDS: more blocks to a wavefront than it has in flight (U a tile).  Each slot is then asked for again as soon as its block
// has been multiplied, not when the whole round has.  (Where one round is all, that code would only be fetched: 24 layers of 1024,
// 8 sequences, 965 -> 975 us.)
template <int MT, int NTW, int NW, int U, bool STREAM, bool ROUNDS>
__global__ void __launch_bounds__(64 * NW) gemv16_kernel(const GemmArgs a) {
    __shared__ v4i red[NW][MT * NTW][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int item = blockIdx.x, mat, bz = 0, grp;
    const int groups = (a.NT + NTW - 1) / NTW;
    GemmCols cols = {a.NT, a.N, a.tail, a.apart != 0};
    if (a.NT2 > 0) {                                    // two products of different widths side by side, not split
        mat = item >= groups ? 1 : 0;
        grp = item - mat * groups;
        if (mat) cols = GemmCols{a.NT2, a.N2, a.tail2, a.apart2 != 0};
    } else {
        grp = item % groups; item /= groups;
        bz = item % a.split; mat = item / a.split;
    }
    const int nt0 = grp * NTW;
    const signed char *dig = mat == 0 ? a.dig[0] : mat == 1 ? a.dig[1] : a.dig[2];
    const uint8_t *w16 = mat == 0 ? a.w16[0] : mat == 1 ? a.w16[1] : a.w16[2];
    const int kb0 = bz * a.kb_per_split;
    int kb1 = kb0 + a.kb_per_split;
    if (kb1 > a.KB) kb1 = a.KB;
    const v4i *bsrc[NTW], *asrc[MT];
#pragma unroll
    for (int j = 0; j < NTW; ++j)                       // (clamped: loads stay in bounds, results are dropped)
        bsrc[j] = reinterpret_cast<const v4i *>(w16 + (size_t)(nt0 + j < cols.NT ? nt0 + j : cols.NT - 1) * a.KB * 1024) + lane;
#pragma unroll
    for (int m = 0; m < MT; ++m)
        asrc[m] = reinterpret_cast<const v4i *>(dig + (size_t)(m < a.MT ? m : a.MT - 1) * a.KB * 1024) + lane;
    v4i acc[MT][NTW];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NTW; ++j) acc[m][j] = v4i{0, 0, 0, 0};
    v4i B[NTW][U], A[MT][U];
    auto fetch = [&](int i, int kb) {
        const size_t o = (size_t)min(kb, a.KB - 1) * 64;                  // past the end: a block nobody multiplies
#pragma unroll
        for (int j = 0; j < NTW; ++j) B[j][i] = ldw<STREAM>(bsrc[j] + o);
#pragma unroll
        for (int m = 0; m < MT; ++m) A[m][i] = asrc[m][o];
    };
    int k = kb0 + wave;
#pragma unroll
    for (int i = 0; i < U; ++i) fetch(i, k + NW * i);
    for (; k < kb1; k += NW * U) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if (k + NW * i < kb1) {         // uniform for the wavefront
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int j = 0; j < NTW; ++j)
                        acc[m][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[m][i], B[j][i], acc[m][j], 0, 0, 0);
            }
            if (ROUNDS && k + NW * (U + i) < kb1) fetch(i, k + NW * (U + i));      // the slot is free
        }
    }
    // digit sums of at most a thousand blocks or so (plan_products splits longer contractions): inside int32
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NTW; ++j) red[wave][m * NTW + j][lane] = acc[m][j];
    __syncthreads();
    for (int i = wave; i < MT * NTW; i += NW) {
        const int m = i / NTW, nt = nt0 + i % NTW;
        if (nt >= cols.NT) continue;           // uniform for the wavefront
        v4i sum[1][1];
        sum[0][0] = red[0][i][lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) sum[0][0] += red[w][i][lane];
        if (mat == 0 && a.part) relu2_part(a, sum[0][0], m, nt, lane);
        else gemm_epilogue<1, 1>(a, cols, sum, m, nt, mat, bz, lane);
    }
}

// Quantiser of a product whose tiles left their share of every row (relu2_part): a part of 1024 values per workgroup, one launch
// instead of a pass for the rows' maxima and one for the digits (8 rows of 10240: 4.7 us against 3.9 + 4.0).  A step of 8
// sequences at 3B 2.08 -> 2.04 ms, of 5 at 24 layers of 2048 1.40 -> 1.34, of 8 at 24 layers of 1024 1.033 -> 1.019; not for rows
// up to 3072, which one workgroup each quantises as fast (12 layers of 768, 8 sequences: 451 us that way, 458 this).  9 and 16
// sequences: 12 layers of 2560 855 -> 834 and 928 -> 906, 24 of 1024 1050 -> 1015 and 1089 -> 1058.  The sum of
// the fixed-point values is added up with atomics: integers below 2^53, exact in
// any order.
__global__ void __launch_bounds__(kRT) rows_quant_tiles_kernel(const QuantArgs a, const double2 *part, int tiles) {
    __shared__ double red0[8], red1[8];
    __shared__ float redf[16];
    const int t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, c0 = 4 * (blockIdx.x * kRT + tid);
    const bool live = c0 < a.K;                            // (whole groups of four lanes: K is a multiple of 64)
    float v[4] = {0.f, 0.f, 0.f, 0.f}, rg[4] = {0.f, 0.f, 0.f, 0.f}, amax = 0.f;
    if (live) { ld4(v, static_cast<const float *>(a.in) + (size_t)t * a.K + c0); ld4(rg, a.range + c0); }
    double z[1] = {0.0};
    for (int i = tid; i < tiles; i += kRT) {
        const double2 p = part[(size_t)t * tiles + i];
        amax = fmaxf(amax, (float)p.x); z[0] += p.y;
    }
    amax = wmaxf(amax);
    if (lane == 0) redf[tid >> 6] = amax;
    bsum<1>(z, red0, kRW);                                 // (its barrier also publishes redf)
    double S, invS, qsum[1] = {0.0};
    row_scale(row16_max((lane & 15) < kRW ? redf[lane & 15] : 0.f), S, invS);
    if (live) {
        float xs[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) xs[i] = (float)((double)v[i] * (double)rg[i]);
        qsum[0] = emit_quad(xs, invS, c0, t, a.K >> 6, a.dig);
    }
    bsum<1>(qsum, red1, kRW);
    if (tid == 0) {
        atomicAdd(a.qs + t, qsum[0]);
        if (blockIdx.x == 0) { a.S[t] = S; a.zp[t] = z[0]; }
    }
}

// ---------------------------------------------------------------------------
// y[t, j] = S_t * tot + 128 * S_t * sum q_t + zp_t, then the phase's element-wise tail.
// ---------------------------------------------------------------------------
struct FinishArgs {
    int R, N, ldd, slices;
    size_t slice;
    const long long *tot;       // [products][slices][...]
    const double *S[kRowsMaxProducts], *qs[kRowsMaxProducts], *zp[kRowsMaxProducts];
    double *out[kRowsMaxProducts];      // [R, N] each
    const float *gate;          // ROW_GATE_ADD: raw receptance [R, N]
};

template <int OP>
__global__ void __launch_bounds__(256) rows_finish_kernel(const FinishArgs a) {
    const int t = blockIdx.y, mat = blockIdx.z;
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= a.N) return;
    const double *Sv = mat == 0 ? a.S[0] : mat == 1 ? a.S[1] : a.S[2];
    const double *qsv = mat == 0 ? a.qs[0] : mat == 1 ? a.qs[1] : a.qs[2];
    const double *zpv = mat == 0 ? a.zp[0] : mat == 1 ? a.zp[1] : a.zp[2];
    double *outv = mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : a.out[2];
    const double S = Sv[t];
    long long tot = 0;                                   // integer partial sums of the contraction splits: exact in any order
    const long long *tp = a.tot + (size_t)mat * a.slices * a.slice + (size_t)t * a.ldd + j;
    for (int z = 0; z < a.slices; ++z) tot += tp[(size_t)z * a.slice];
    const double y = S * (double)tot + 128.0 * (S * qsv[t]) + zpv[t];
    double *o = outv + (size_t)t * a.N + j;
    if (OP == ROW_STORE) *o = y;
    else if (OP == ROW_STORE_F32) reinterpret_cast<float *>(outv)[(size_t)t * a.N + j] = (float)y;
    else if (OP == ROW_RELU2) { const double r = y > 0.0 ? y : 0.0; reinterpret_cast<float *>(outv)[(size_t)t * a.N + j] = (float)(r * r); }   // block.py:97
    else if (OP == ROW_ADD) *o += y;                                                          // block.py:80
    else if (OP == ROW_GATE_ADD) *o += y * (double)sigmoid_f32(a.gate[(size_t)t * a.N + j]);          // block.py:95-100
}

// ---------------------------------------------------------------------------
// WKV + receptance gate           (block.py:69-78, wkv.py:23-39, operators.cu:6-37)
// Arithmetic of the single-token kernel: sums, exponentials and the gate in float32, the exponent pp in float64
// (wkv_step_f32).  A float64 exponential is some fifty dependent instructions, and with one wavefront per 64
// channels and chunk there is nothing to hide them behind: the float64 form took three times as long.
// sequence: thread = channel, serial over the T rows; batch: thread = (row, channel).
// ---------------------------------------------------------------------------
struct WkvRowsArgs {
    int C, R, sequence;
    const float *k, *v, *r;     // [R, C]  float32: what the single-token kernel rounds them to as well
    const double *w, *u;        // [C]  (w = -exp(time_decay))
    double *state;              // rows aa, bb, pp of the layer: state + 2C; batch: + row * state_stride
    int64_t state_stride;
    float *out;                 // [R, C]  wkv * sigmoid(r): a float32 product
    RowsDeferred pend[3];       // batch rows: k, v, r still in slices, as many of each (tot null: all are read from the arrays above)
};

__global__ void __launch_bounds__(64) wkv_rows_kernel(const WkvRowsArgs a) {
    const int c = blockIdx.x * 64 + threadIdx.x;
    if (c >= a.C) return;
    const int C = a.C;
    const double w = a.w[c], u = a.u[c];
    const int t0 = a.sequence ? 0 : blockIdx.y, t1 = a.sequence ? a.R : blockIdx.y + 1;
    double *st = a.state + (a.sequence ? 0 : (size_t)blockIdx.y * a.state_stride);
    float aa = (float)st[c], bb = (float)st[C + c];
    double pp = st[2 * C + c];
    for (int t = t0; t < t1; ++t) {
        const size_t i = (size_t)t * C + c;
        float kk, vv, rr;
        if (a.pend[0].tot) {                            // (uniform; rounded to float32 exactly as ROW_STORE_F32 would have stored them)
            long long tot[3];
            with_slices(a.pend[0].slices, [&](auto count) {
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    tot[j] = slices_sum1<decltype(count)::value>(a.pend[j].tot + (size_t)t * a.pend[j].ldd + c, a.pend[j].slice);
            });
            kk = (float)deferred_y(a.pend[0], t, tot[0]); vv = (float)deferred_y(a.pend[1], t, tot[1]); rr = (float)deferred_y(a.pend[2], t, tot[2]);
        } else { kk = a.k[i]; vv = a.v[i]; rr = a.r[i]; }
        const float y = wkv_step_f32(w, u, kk, vv, aa, bb, pp);
        a.out[i] = y * sigmoid_f32(rr);
    }
    st[c] = (double)aa; st[C + c] = (double)bb; st[2 * C + c] = pp;
}


// Longer sequences, in one launch and with the same roundings as token by token: sequences of fewer than kWkvChunked steps
// are one serial recurrence; longer ones are cut into chunks of kWkvChunk steps (the recurrence is linear in (aa, bb)): every
// chunk's own sums from an empty state in float32, a serial float64 pass over the chunks for the state each of them starts from
// (a chunk decays its input by e^{n w}; float64 is also what the state keeps), and the steps again from there.  These
// orders are part of the results: logits that move by rounding move the texts of a seeded sampler.
//
// A serial recurrence need not be a chain of exponentials: the exponent pp depends on k alone (an addition and a maximum
// a step), all factors follow from it side by side, and (aa, bb) are two fused multiply-adds a step.  So SL lanes share a
// chunk, S steps each: pp and then (aa, bb) are handed from lane to lane in SL - 1 rounds (every lane runs its steps in every
// round; what it was handed counts from the round in which it is right), and the rest is done by all lanes at once.
//
// Bound: vector instructions, some 200 a step.  2560 channels and 24 / 64 / 128 / 256 / 1024 steps: 5.1 / 7.5 / 6.2 / 8.6 /
// 27.2 us; a thread per channel below 64 steps and three launches from there on, with the same results, 19.6 / 19.3 / 19.1 /
// 19.8 / 31.0 us; a log-step scan over chunk sums, in another order of additions, 5.8 / 5.6 / 6.3 / 8.0 / 23.3 us.
constexpr int kWkvSeqMin = 6;       // from here on faster than a thread per channel (1.0 us a step)
constexpr int kWkvChunk = 32, kWkvChunked = 64;
// Channels from which on there is a workgroup for every compute unit: blocks of 4 chunks, two workgroups to a unit, beat blocks
// of 8 (5120 channels, 257 / 512 / 1024 steps: 18.3 / 25.2 / 47.2 against 25.6 / 29.4 / 56.2 us; 2560: 13.8 / 18.3 / 34.6 against
// 13.3 / 14.6 / 27.2; 16 chunks spill registers: 31 us).
constexpr int kWkvWide = 4096;
// Channels up to which eight of them to a workgroup, each chunk shared by eight lanes of four steps, still leave at most one workgroup
// to a compute unit: half the steps for a lane to work out, for four more rounds of handing on.  Us a prompt with 16 channels / with 8:
// 12 layers of 512, 1024 tokens 1188 / 1149, 12 of 768, 2000 2914 / 2803, 24 of 1024, 1024 3813 / 3722, 16 of 1536, 700 3283 / 3229, 24 of
// 2048, 1000 6829 / 6751; 120 tokens, 24 of 1024 1853 / 1838.  With one block of 4 chunks half as
// many channels are enough: 80 tokens, 24 layers of 2048 2289 / 2305.  At 2560 channels, 320 workgroups, 9904 / 10087 with 1024 tokens.
constexpr int kWkvNarrow = 2048;

__device__ __forceinline__ float shfl_from(float v, int lane) { return __shfl(v, lane, 64); }
__device__ __forceinline__ double shfl_from(double v, int lane) { return __shfl(v, lane, 64); }

// The S steps of one lane: k, v and what the exponents make of them.  FULL: all of them lie inside the sequence.
template <int S, bool FULL>
struct WkvSteps {
    int n;                          // live steps
    float k[S], v[S], f1[S], f2[S];
    double w;
    __device__ __forceinline__ bool on(int i) const { return FULL || i < n; }
    __device__ __forceinline__ double exponent(double p) const {        // pp after the steps
#pragma unroll
        for (int i = 0; i < S; ++i) { const double q = fmax(p + w, (double)k[i] + w); p = on(i) ? q : p; }
        return p;
    }
    __device__ __forceinline__ double factors(double p) {               // as in wkv_step_f32; pp after the steps
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const double s = p + w, r = (double)k[i] + w, d2 = s - r;
            const float f = expf(-fabsf((float)d2));
            f1[i] = d2 >= 0.0 ? 1.f : f; f2[i] = d2 >= 0.0 ? f : 1.f;
            p = on(i) ? fmax(s, r) : p;
        }
        return p;
    }
    __device__ __forceinline__ void sums(float &aa, float &bb) const {  // (aa, bb) after the steps
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const float x = fmaf(f1[i], aa, f2[i] * v[i]), y = fmaf(f1[i], bb, f2[i]);
            aa = on(i) ? x : aa; bb = on(i) ? y : bb;
        }
    }
};

// One block from step tb on: NCH chunks of SL lanes x S steps for each of CH channels.  CHUNKED: (ca, cb, cp) is the float64
// state before the block, on return after it; else the block is the whole sequence, and the state comes back in the last lane
// of every channel.
template <int CH, int SL, int S, int NCH, bool CHUNKED, bool FULL>
__device__ __forceinline__ void wkv_seq_block(const WkvRowsArgs &a, int tb, int c, double w, double u, double (*sh)[NCH][CH],
                                              double &ca, double &cb, double &cp) {
    const int C = a.C, R = a.R;
    const int ch = threadIdx.x % CH, pos = threadIdx.x / CH, slot = pos % SL, lane = threadIdx.x & 63;
    // (a wavefront is one chunk: its number is uniform)
    const int chunk = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int t0 = tb + pos * S;
    WkvSteps<S, FULL> st;
    st.w = w;
    st.n = FULL ? S : max(0, min(S, R - t0));
    float r[S];
    auto row = [&](int i) { return (size_t)(FULL ? t0 + i : min(t0 + i, R - 1)) * C + c; };     // past the end: the last row again, unused
#pragma unroll
    for (int i = 0; i < S; ++i) { st.k[i] = a.k[row(i)]; st.v[i] = a.v[row(i)]; }
#pragma unroll
    for (int i = 0; i < S; ++i) r[i] = a.r[row(i)];
    // what a lane starts from, handed on from the lane before it
    auto hand_exponent = [&](double p) {
#pragma unroll
        for (int j = 1; j < SL; ++j) { const double q = shfl_from(st.exponent(p), lane - CH); p = slot >= j ? q : p; }
        return p;
    };
    auto hand_sums = [&](float &aa, float &bb) {
#pragma unroll
        for (int j = 1; j < SL; ++j) {
            float x = aa, y = bb;
            st.sums(x, y);
            x = shfl_from(x, lane - CH); y = shfl_from(y, lane - CH);
            aa = slot >= j ? x : aa; bb = slot >= j ? y : bb;
        }
    };
    double pp = cp;
    float aa = (float)ca, bb = (float)cb;
    if (CHUNKED) {
        // the chunk's own sums
        const double lp = st.factors(hand_exponent(-1e30));
        float la = 0.f, lb = 0.f;
        hand_sums(la, lb);
        st.sums(la, lb);
        if (tb > 0) __syncthreads();                     // the block before has been read
        if (slot == SL - 1) { sh[0][chunk][ch] = lp; sh[1][chunk][ch] = (double)la; sh[2][chunk][ch] = (double)lb; }
        __syncthreads();
        // the exponents before every chunk; this chunk's factors
        double p = cp, s_own = 0.0, p_own = 0.0;
        const int live = FULL ? NCH : (R - tb + SL * S - 1) / (SL * S);
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int nj = FULL ? SL * S : min(SL * S, R - tb - j * SL * S);
            const double s = fma((double)nj, w, p), q = fmax(s, sh[0][j][ch]);
            if (j == chunk) { pp = p; s_own = s; p_own = q; }
            p = FULL || j < live ? q : p;
        }
        cp = p;
        const double g1 = (double)expf((float)(s_own - p_own)), g2 = (double)expf((float)(sh[0][chunk][ch] - p_own));
        const double ga = g2 * sh[1][chunk][ch], gb = g2 * sh[2][chunk][ch];
        __syncthreads();
        if (slot == SL - 1) { sh[0][chunk][ch] = g1; sh[1][chunk][ch] = ga; sh[2][chunk][ch] = gb; }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const double f = sh[0][j][ch], x = fma(f, ca, sh[1][j][ch]), y = fma(f, cb, sh[2][j][ch]);
            if (j == chunk) { aa = (float)ca; bb = (float)cb; }
            ca = FULL || j < live ? x : ca; cb = FULL || j < live ? y : cb;
        }
    }
    pp = hand_exponent(pp);
    st.factors(pp);
    hand_sums(aa, bb);
    const double uw = u + w;
#pragma unroll
    for (int i = 0; i < S; ++i) {
        if (st.on(i)) {                                  // wkv_step_f32, its second pair of exponentials taken from above
            const double d = pp - (uw + (double)st.k[i]);
            const float e = expf(-fabsf((float)d));
            const float e1 = d >= 0.0 ? 1.f : e, e2 = d >= 0.0 ? e : 1.f;
            const float y = fmaf(e1, aa, e2 * st.v[i]) / fmaf(e1, bb, e2);
            a.out[row(i)] = y * sigmoid_f32(r[i]);
            aa = fmaf(st.f1[i], aa, st.f2[i] * st.v[i]);
            bb = fmaf(st.f1[i], bb, st.f2[i]);
            pp = fmax(pp + w, (double)st.k[i] + w);
        }
    }
    if (!CHUNKED) { ca = (double)aa; cb = (double)bb; cp = pp; }
}

template <int CH, int SL, int S, int NCH, bool CHUNKED>
__global__ void __launch_bounds__(CH * SL * NCH) wkv_seq_kernel(const WkvRowsArgs a) {
    static_assert(CH * SL == 64, "a chunk is a wavefront");
    __shared__ double sh[CHUNKED ? 3 : 1][NCH][CH];
    const int ch = threadIdx.x % CH, C = a.C, n = gridDim.x;                   // (C is a multiple of 64)
    // Neighbouring channels, which share their cache lines, go to one XCD: workgroup i runs on XCD i % 8, whose channels are consecutive
    // (24 layers of 2560, 500 / 1024 tokens 6721 / 9963 us a prompt without, 6661 / 9904 with this).
    const int x = blockIdx.x % kXcds, c = (x * (n / kXcds) + min(x, n % kXcds) + (int)blockIdx.x / kXcds) * CH + ch;
    const double w = a.w[c], u = a.u[c];
    double ca = a.state[c], cb = a.state[C + c], cp = a.state[2 * C + c];
    constexpr int kBlock = NCH * SL * S;
    int tb = 0;
    for (; tb + kBlock <= a.R; tb += kBlock) wkv_seq_block<CH, SL, S, NCH, CHUNKED, true>(a, tb, c, w, u, sh, ca, cb, cp);
    if (tb < a.R) wkv_seq_block<CH, SL, S, NCH, CHUNKED, false>(a, tb, c, w, u, sh, ca, cb, cp);
    if ((int)threadIdx.x / CH == (CHUNKED ? 0 : SL - 1)) { a.state[c] = ca; a.state[C + c] = cb; a.state[2 * C + c] = cp; }
}

// ---------------------------------------------------------------------------
// Stand-alone matrix-vector product for 1..8 vectors on the M16 layout, four-vector dequantisation
//   y[b,k] = r_col[k] * sum_j fp32(x[b,j] r_row[j]) code[j,k] + sum_j x[b,j] m_row[j] + m_col[k] sum_j x[b,j]
// (the T == 1 branch of MM8.forward, matmul.py:51-62, with per-column factors on top).
//
// Two launches.  mv16_quant_kernel rewrites the vectors once, for every workgroup of the product, as fixed-point
// digit fragments; the contraction is cut into chunks of CB = 4 blocks (256 rows) and every (vector, chunk) has its
// own power-of-two scale, so no workgroup of the quantiser waits for another and the fixed point is as fine as
// the chunk allows.  mv16_kernel gives one 16-column tile to a workgroup whose wavefronts take the chunks in
// turn: all loads of a chunk (CB weight blocks from HBM, CB fragments per group of four vectors from L2) are
// requested before the first matrix instruction, the integer digit sums of a chunk are exact and enter a float64
// sum scaled by the chunk's scale; the wavefronts' sums are added in a fixed order.
// ---------------------------------------------------------------------------
struct Mv16Args {
    int B, n_in, n_out, KB, n_chunks;
    const float *x;             // [B, n_in]
    const float *r_row;         // [n_in]
    const double *m_row;        // [n_in]
    const float *r_col, *m_col; // [n_out] or null
    const uint8_t *w16;         // M16 blocks [ceil(n_out/16)][KB][1024]
    signed char *dig;           // fragments [ceil(B/4)][KB][1024]
    double *rec;                // [B][n_chunks][4]: scale, 128 * scale * sum q, zero-point share, sum x
    double *y;                  // [B, n_out]
};

template <int CB>
__global__ void __launch_bounds__(256) mv16_quant_kernel(const Mv16Args a) {
    // workgroup = (chunk, group of four vectors); wavefront = one vector; a lane holds CB / 4 groups of four values
    constexpr int QPT = CB / 4;
    const int c = blockIdx.x, mt = blockIdx.y;
    const int lane = threadIdx.x & 63, t = 4 * mt + (threadIdx.x >> 6);
    if (t >= a.B) return;                          // (whole wavefronts; the kernel has no barrier)
    float xs[QPT][4];
    float amax = 0.f;
    double zp = 0.0, xsum = 0.0;
    const bool vec = (a.n_in & 3) == 0 && ((reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.r_row)) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(a.m_row) & 15) == 0;
#pragma unroll
    for (int s = 0; s < QPT; ++s) {
        const int c0 = c * CB * 64 + 4 * (lane + 64 * s);
        float xv[4] = {0.f, 0.f, 0.f, 0.f}, rv[4] = {0.f, 0.f, 0.f, 0.f};
        double mv[4] = {0.0, 0.0, 0.0, 0.0};
        if (vec && c0 + 3 < a.n_in) {
            const float4 x4 = *reinterpret_cast<const float4 *>(a.x + (size_t)t * a.n_in + c0);
            const float4 r4 = *reinterpret_cast<const float4 *>(a.r_row + c0);
            const double2 m0 = *reinterpret_cast<const double2 *>(a.m_row + c0), m1 = *reinterpret_cast<const double2 *>(a.m_row + c0 + 2);
            xv[0] = x4.x; xv[1] = x4.y; xv[2] = x4.z; xv[3] = x4.w;
            rv[0] = r4.x; rv[1] = r4.y; rv[2] = r4.z; rv[3] = r4.w;
            mv[0] = m0.x; mv[1] = m0.y; mv[2] = m1.x; mv[3] = m1.y;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = c0 + i;
                if (j < a.n_in) { xv[i] = a.x[(size_t)t * a.n_in + j]; rv[i] = a.r_row[j]; mv[i] = a.m_row[j]; }
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double xd = (double)xv[i];
            xs[s][i] = (float)(xd * (double)rv[i]);                                   // matmul.py:131
            zp += xd * mv[i];
            xsum += xd;
            amax = fmaxf(amax, fabsf(xs[s][i]));
        }
    }
    amax = wmaxf(amax);
    double S, invS;
    row_scale(amax, S, invS);
    double qsum = 0.0;
#pragma unroll
    for (int s = 0; s < QPT; ++s) {
        const int c0 = c * CB * 64 + 4 * (lane + 64 * s);
        if (c0 < a.KB * 64) qsum += emit_quad(xs[s], invS, c0, t, a.KB, a.dig);      // (whole groups of 16 lanes)
    }
    qsum = wsum(qsum); zp = wsum(zp); xsum = wsum(xsum);
    if (lane == 0) {
        double *r = a.rec + ((size_t)t * a.n_chunks + c) * 4;
        r[0] = S; r[1] = 128.0 * (S * qsum); r[2] = zp; r[3] = xsum;
    }
}

template <int MT, int CB, int NTW>
__global__ void __launch_bounds__(1024) mv16_kernel(const Mv16Args a) {
    extern __shared__ double mv_red[];            // [NW][MT][NTW][64] tile sums, then [4 MT][3] row constants
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), NW = blockDim.x >> 6;
    const int g = lane >> 4, n = lane & 15, NT = (a.n_out + 15) >> 4;
    // NTW neighbouring tiles per workgroup share every digit fragment a wavefront fetches
    const v4i *bsrc[NTW];
#pragma unroll
    for (int j = 0; j < NTW; ++j)
        bsrc[j] = reinterpret_cast<const v4i *>(a.w16 + (size_t)min((int)blockIdx.x * NTW + j, NT - 1) * a.KB * 1024) + lane;
    const v4i *asrc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) asrc[m] = reinterpret_cast<const v4i *>(a.dig + (size_t)m * a.KB * 1024) + lane;
    double sum[MT][NTW];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NTW; ++j) sum[m][j] = 0.0;
    double *red = mv_red, *rc3 = mv_red + (size_t)NW * MT * NTW * 64;
    for (int c = wave; c < a.n_chunks; c += NW) {
        v4i Bf[NTW][CB], Af[MT][CB];
        const int kb0 = c * CB;
#pragma unroll
        for (int i = 0; i < CB; ++i) {
            const size_t o = (size_t)min(kb0 + i, a.KB - 1) * 64;                   // past the end: a block nobody multiplies
#pragma unroll
            for (int j = 0; j < NTW; ++j) Bf[j][i] = __builtin_nontemporal_load(bsrc[j] + o);
#pragma unroll
            for (int m = 0; m < MT; ++m) Af[m][i] = asrc[m][o];
        }
        double rS[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) rS[m] = a.rec[((size_t)min(4 * m + g, a.B - 1) * a.n_chunks + c) * 4];
        if (c == wave && wave == NW - 1) {
            // The last wavefront, while its first blocks travel: the per-vector constants.  Lane 8 t + p adds the
            // chunks p, p + 8, ... of vector t (its loads are independent of each other), then the eight partial
            // sums are added in a fixed order.
            const int t = lane >> 3, p8 = lane & 7;
            double ad = 0.0, z = 0.0, xsm = 0.0;
            const double *r = a.rec + (size_t)min(t, a.B - 1) * a.n_chunks * 4;
#pragma unroll 4
            for (int cc = p8; cc < a.n_chunks; cc += 8) { ad += r[4 * cc + 1]; z += r[4 * cc + 2]; xsm += r[4 * cc + 3]; }
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) {
                ad += __shfl_xor(ad, off, 64); z += __shfl_xor(z, off, 64); xsm += __shfl_xor(xsm, off, 64);
            }
            if (p8 == 0 && t < 4 * MT) { rc3[3 * t] = ad; rc3[3 * t + 1] = z; rc3[3 * t + 2] = xsm; }
        }
        v4i acc[MT][NTW];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < NTW; ++j) acc[m][j] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < CB; ++i) {
            if (kb0 + i < a.KB) {                                                     // uniform for the wavefront
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int j = 0; j < NTW; ++j)
                        acc[m][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(Af[m][i], Bf[j][i], acc[m][j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                // digit sums of at most 64 CB terms of magnitude <= 2^14 each; the weighted total is below 2^53: exact
                const v4i d = acc[m][j];
                const long long tot = ((((long long)d.x * 256 + d.y) * 256 + d.z) * 256) + d.w;
                sum[m][j] += rS[m] * (double)tot;
            }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NTW; ++j) red[(((size_t)wave * MT + m) * NTW + j) * 64 + lane] = sum[m][j];
    __syncthreads();
    // wavefront j adds up tile j (fixed order) and writes its 16 columns
    if (wave >= NTW) return;
#pragma unroll
    for (int j = 0; j < NTW; ++j) {
        if (j != wave) continue;
        const int nt = blockIdx.x * NTW + j, col = 16 * nt + n;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            double s = 0.0;
            for (int w = 0; w < NW; ++w) s += red[(((size_t)w * MT + m) * NTW + j) * 64 + lane];
            const int t = 4 * m + g;
            if (nt < NT && t < a.B && col < a.n_out) {
                const double rc = a.r_col ? (double)a.r_col[col] : 1.0;
                const double mc = a.m_col ? (double)a.m_col[col] : 0.0;
                a.y[(size_t)t * a.n_out + col] = rc * (s + rc3[3 * t]) + rc3[3 * t + 1] + mc * rc3[3 * t + 2];
            }
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
size_t rows_dig_bytes(int64_t R, int64_t K) { return (size_t)(ceil_div(R, 4) * (K / 64) * 1024); }
constexpr int kMaxSplit = 8;
constexpr int kGemmWideNum = 10, kGemmWideDen = 9;     // the 64 x 160 variant is taken when its cost is below 9/10 of the 64 x 128 variant's
// ... except a contraction of 200 blocks and more, which splits in two while the grid is below the device (14B shape,
// 256-token chunks: the [256 x 20480] x [20480 x 5120] product; 14,080 against 13,190 tokens/s)
constexpr int kGemmLongFillWgs = 256, kGemmLongBlocks = 200;
constexpr int kSkinnyFillWgs = 128;     // 9..32 rows (weight streaming): contractions of a grid below this many workgroups are cut in slices, in how many skinny_split says (when it was the number of workgroups to reach, a batch-32 step took 8.07 ms at 128, 8.73 at 256, 9.17 at 64 for the 14B shape; 4.06 / 4.13 / 4.11 ms for the 3B shape)
// Row blocks of 64 tokens up to which the general kernel reads the weights past the caches: more of them find each other's weight
// blocks there (prompts, kept / streamed: 77 tokens of 24 layers of 1024 2274 / 2193 us, 100 of the 3B shape 4565 / 4416, 256 of it
// 6158 / 6248, 256 of 14B 17786 / 18992)
constexpr int kStreamRowBlocks = 2;
constexpr int kSkinnyPairWgs = 64;      // ffn key and receptance of 9..32 rows in one launch from so many workgroups on
constexpr int kGemmFillWgs = 96;         // larger products: split until the grid has this many workgroups.  A split costs a second launch and a round trip of the integer totals through memory, so it only pays for grids far below the device (3B shape, tokens/s in chunks of 64 / 128 / 256 / 512 tokens: 13,180 / 23,640 / 37,610 / 52,070 at 96; 12,480 / 21,280 / 34,650 / 49,380 at 256; 12,540 / 21,470 / 31,520 / 51,160 at 64)

// Which kernel serves n products of MT row tiles x NT column tiles over KB contraction blocks, its grid and the number of contraction
// splits (plan_products; readers: who adds the slices up, see rows_readers).  The one place these are decided.  The totals' buffer is
// sized by bounds over every number of products and readers (gemm_split_bound, rows_deferred_bytes), which a host test holds against the plans.
enum { PLAN_VEC = 0, PLAN_SKINNY, PLAN_GENERAL, PLAN_WIDE, PLAN_NARROW };
struct ProductPlan { int kind, gx, gy, split; };
// Which products of 9 to 32 rows go through gemv16_kernel.  Every workgroup of it reads the digits of all rows, gemm8_skinny_kernel
// shares them between four wavefronts of eight tiles but needs slices of the contraction, and launches that add them up, to fill
// the device.  So: few tiles, short contractions.  Us a step of 9, 16 / 17, 32 sequences, all through the other kernel / by this rule:
// 12 layers of 512 658, 668 / 684, 722 against 448, 460 / 475, 497; 24 of 1024 1500, 1549 / 1590, 1750 against 1048, 1086 / 1151,
// 1300; 12 of 1536 884, 908 / 935, 1036 against 652, 690 / 744, 815; 8 of 2048 582, 600 / 615, 665 against 512, 538 / 590, 645; 12 of 2560
// 985, 1028 / 1057, 1165 against 860, 935 / 1005, 1096; 8 of 4096 905, 920 / 950, 1025 against 865, 905 / 930, 1024.  Beyond it that
// kernel wins: three M-tiles of 5120 channels 561 against 572, four 601 against 615 to 646, five of 4096 951 against 978 with its 768 tiles of k, v, r.
static bool vec_rows(int64_t MT, int64_t tiles, int64_t KB) {
    if (MT <= kVecMT) return true;
    if (MT <= 4) return tiles <= 1280 && MT * KB <= (tiles <= 256 ? 700 : 200);
    return MT <= kVecMTMax && tiles <= 512 && MT * KB <= 400;
}
// Whether a contraction of 9 to 32 rows is cut in gemm8_skinny_kernel, whether it is the kernel that runs or not (see rounded_apart).
static bool skinny_cut(int64_t NT, int64_t KB, int n) { return ceil_div(NT, kSkinnyNT) * n < kSkinnyFillWgs && KB >= 16; }
// In how many slices: as vec_split, what the busiest compute unit draws (eight tiles' weights and the digits of 16 or 32 rows), and what it
// costs to add them up: in the LayerNorm kernel as there, in the WKV kernel, whose workgroups are many, little, in a launch of its own 4 to 5 us, and
// the two that then wait for it.  (So no power of two: 40 column blocks of 5120 channels fill 240 compute units in six slices, 160 in four.)  Us a
// step of 32 sequences before (the power of two that brings 128 workgroups, up to eight) / now: 24 layers of 1024 1308 / 1220, 12 of 2560 1096 /
// 1071, 8 of 4096 1023 / 1011, 8 of 5120 1289 / 1254; of 16, with four M-tiles (gemm8_skinny_kernel), 905 / 848 of 4096 and 1106 / 1031 of 5120.
// The launch hands the XCDs whole column blocks, so it is the XCD with the most of them that must not start a second round: 41 blocks of 5248
// channels in six slices are 246 workgroups, but 36 on the first XCD.  Us a step of 17 / 32 sequences of 3 layers, powers of two / 256 compute units
// counted as one / by XCD: 3584 355, 398 / 365, 408 / 358, 401; 4224 414, 459 / 417, 465 / 402, 443; 5248 514, 579 / 545, 615 / 495, 557.
static int skinny_split(int64_t MT, int64_t NT, int64_t KB, int n, int readers) {
    if (!skinny_cut(NT, KB, n)) return 1;
    const int64_t on_one = ceil_div(ceil_div(NT, kSkinnyNT), kXcds) * n;        // column blocks of the XCD that has the most
    int best = 2;
    int64_t least = INT64_MAX;
    for (int s = 2; s <= kMaxSplit && KB >= 8 * s; ++s) {
        const bool sum = readers && s <= kRowsDeferSlices;
        const int64_t cost = ceil_div(on_one * s, 256 / kXcds) * (kSkinnyNT + (MT <= 4 ? 4 : 8)) * ceil_div(KB, s) +
                             (sum && n > 1 ? 8 * s : sum ? 32 + readers * (2 * s + 1) * NT / 16 : 420 + 30 * s * n);
        if (cost < least) { least = cost; best = s; }
    }
    return best;
}
// Rounds of workgroups on 256 compute units, in matrix instructions per step: two general workgroups (w4 in all) share a
// compute unit (2 x 32), a wide one (w5) has it alone (40).
static int64_t general_cost(int64_t w4) {
    const int64_t rem = w4 % 512;
    return (w4 / 512) * 64 + (rem == 0 ? 0 : rem <= 256 ? 32 : 64);
}
// (a narrow workgroup: 20, but it waits for its LDS reads, 0.7 to a matrix instruction)
constexpr int kGemmNarrowCost = 27;
static bool general_wide(int64_t w4, int64_t w5) { return w4 >= 256 && kGemmWideNum * ceil_div(w5, 256) * 40 < kGemmWideDen * general_cost(w4); }
static int vec_split(int64_t MT, int64_t NT, int64_t KB, int readers);
// Whole contractions on a grid of the general kernel that leaves compute units idle and the others one workgroup each: 64 x 80 columns to a workgroup,
// where those are at most one to a compute unit on every XCD (by the launch order: a grid that fits as a whole but not on each, k, v, r of 256 rows of
// 1536 channels, 20 us a launch instead of 15), and from three row blocks on (fewer read the weights past the caches).  Us a launch, 64 x 128 / 64 x 80: 400 rows,
// 2560 -> 2560 23.0 / 20.3, 10240 -> 2560 69 / 57.5; 256 rows, 5120 -> 5120 40 / 35.5.  A prompt of 12 layers of 2560, 320 / 400 / 512 tokens 2765,
// 2962, 3331 -> 2619, 2746, 3186 us; of 12 of 2048, 400 and 512 2412, 2582 -> 2241, 2451; of 8 of 5120, 160 and 256 2768, 3500 -> 2712, 3413.
static bool general_narrow(const ProductPlan &p, int64_t NT, int n) {
    const int64_t gx = ceil_div(NT, kGemmNarrowNT), on_one = p.gy >= kXcds ? ceil_div(p.gy, kXcds) * gx : ceil_div(gx, kXcds) * p.gy;
    return p.split == 1 && (int64_t)p.gx * p.gy * n <= 256 && p.gy > kStreamRowBlocks && on_one * n <= 256 / kXcds;
}
static ProductPlan plan_products(int64_t MT, int64_t NT, int64_t KB, int n, int readers = 0) {
    ProductPlan p;
    p.split = 1;
    if (vec_rows(MT, NT * n, KB)) {
        // few rows: whole contractions, as long as a digit's sum of them stays inside int32 (2^20 per block)
        p.kind = PLAN_VEC; p.gx = (int)NT; p.gy = 1;
        while (ceil_div(KB, p.split) > 1024 && p.split < kMaxSplit) p.split *= 2;
        if (readers && MT <= kVecMT && n == 1 && p.split == 1) p.split = vec_split(MT, NT, KB, readers);
        return p;
    }
    p.gy = (int)ceil_div(MT, 16);
    p.kind = MT <= kSkinnyMT ? PLAN_SKINNY : PLAN_GENERAL;      // few rows: the weight-streaming variant
    if (p.kind == PLAN_GENERAL && general_wide(ceil_div(NT, kGemmNT) * p.gy * n, ceil_div(NT, kGemmWideNT) * p.gy * n)) p.kind = PLAN_WIDE;
    p.gx = (int)ceil_div(NT, p.kind == PLAN_SKINNY ? kSkinnyNT : p.kind == PLAN_WIDE ? kGemmWideNT : kGemmNT);
    // Split the contraction until the grid has a few workgroups per compute unit.
    if (p.kind == PLAN_SKINNY) p.split = skinny_split(MT, NT, KB, n, readers);
    else
        while ((int64_t)p.gx * p.gy * n * p.split < kGemmFillWgs && KB / (p.split * 2) >= 8 && p.split < kMaxSplit) p.split *= 2;
    // a long contraction on a grid still below the device: one split more (two slices at most)
    if (p.kind != PLAN_SKINNY && p.split == 1 && (int64_t)p.gx * p.gy * n < kGemmLongFillWgs && KB >= kGemmLongBlocks) p.split = 2;
    if (p.kind == PLAN_GENERAL && general_narrow(p, NT, n)) { p.kind = PLAN_NARROW; p.gx = (int)ceil_div(NT, kGemmNarrowNT); }
    return p;
}
// Which of two roundings a product's y has: one of S (tot + 128 q) + zp, exact but for the last addition, where slices of the
// contraction are added up by a launch of their own, or S tot + (128 S q + zp) in a product's own epilogue.  Products of at
// most 32 rows that once were split run whole contractions now and keep the first: the last bit of y reaches the logits, and
// with them the texts of a seeded sampler.
static bool rounded_apart(int64_t MT, int64_t NT, int64_t KB, int n) {
    if (MT > kVecMT) return MT <= kSkinnyMT ? skinny_cut(NT, KB, n) : plan_products(MT, NT, KB, n).split > 1;
    return KB >= 16 && (NT * n < 128 || (NT * n < 512 && KB >= kGemmLongBlocks));
}
// Whether a gated update that is handed on adds y * sigmoid(r) as one fused multiply-add, as a product's own epilogue and rows_finish_kernel do.
// Always, but where slices of batch rows of gemm8_skinny_kernel and the general kernel have been handed on ever since: those round the
// product for itself.  (The former takes up to eight slices, and only products of 32 column blocks and more, or of less than 64
// contraction blocks, were handed on before six could be.)
static bool gate_fused(int kind, bool sequence, int64_t NT, int64_t KB) {
    return kind == PLAN_VEC || sequence || (kind == PLAN_SKINNY && 4 * ceil_div(NT, kSkinnyNT) < kSkinnyFillWgs && KB >= 64);
}
// Shape of the few-row kernel for a launch of so many column tiles: tiles per workgroup, wavefronts per workgroup, blocks
// in flight per wavefront and tile (at most).  All workgroups resident at once; KB: the blocks of a workgroup's part of the contraction.
//
// Bound: what the busiest compute unit draws, some 40 KB a us, beside 3 us of launch and first loads.  Per contraction block a workgroup
// of ntw tiles reads their weights (ntw KB) and the digits of all rows (MT KB).  So up to 8 rows take the ntw that leaves that unit the least,
// a larger one only where it saves 32 KB or so; four tiles only where the workgroups fill four fifths of the device.  Us a launch of 8
// rows, 1 / 2 / 4 tiles: 800 tiles of 40 blocks 10.9 / 9.3 / 8.4, 480 of 40 7.2 / 6.4 / 8.0, 288 of 24 5.3 / 4.9 / 5.9, 960 of 80
// 20.2 / 16.3 / 15.1, 320 of 80 11.1 / 9.0 / 12.2, 1280 of 64 20.6 / 17.9 / 24.2; 160 of 40 4.9 / 5.9 / 7.5.  320 of 16 4.35 / 4.21 / 5.0,
// but a step of 24 layers of 1024 962 us with one tile, 975 with two.
struct VecShape { int ntw, nw, u; };
static int64_t vec_draw(int64_t tiles, int ntw, int MT) { return ceil_div(ceil_div(tiles, ntw), 256) * (ntw + MT); }
static VecShape vec_shape(int64_t tiles, int64_t KB, int MT) {
    VecShape v;
    if (MT > kVecMT) {
        if (MT > 4) v = tiles > 256 ? VecShape{2, 8, 2} : VecShape{1, 16, 2};       // (128 KB of sums in LDS)
        else if (tiles > 1280) v = VecShape{4, 8, 3};
        else if (tiles > 320) v = tiles <= 512 ? VecShape{2, 16, 3} : VecShape{2, 8, 5};
        else if (tiles > 256) v = VecShape{1, 8, 5};
        else v = VecShape{1, 16, 5};
        if (v.u > 3) v.u = 3;                               // (registers)
        // No more in flight than a wavefront has: what is past the end is loaded all the same.  With this and the refilled slots, us a
        // step of 8 sequences before / now: 12 layers of 512 437 / 433, of 768 464 / 457, 24 of 1024 1014 / 965, 12 of 1536 625 / 597, 8
        // of 2048 479 / 457, 12 of 2560 780 / 766, 8 of 4096 820 / 776, 4 of 5120 586 / 576.
        const int64_t each = ceil_div(KB, v.nw);
        if (each < v.u) v.u = each <= 1 ? 1 : each == 2 ? 2 : each == 3 ? 3 : v.u;
        return v;
    }
    const int64_t one = vec_draw(tiles, 1, MT), two = vec_draw(tiles, 2, MT), four = vec_draw(tiles, 4, MT);
    v.ntw = 1;
    if (tiles > 320 || (one - two) * KB >= 40) v.ntw = 2;
    if (tiles > 1280) v.ntw = 4;
    else if (v.ntw == 2 && (two - four) * KB >= 32 && 32 * ceil_div(tiles, 4) >= 25 * round_up(ceil_div(tiles, 4), 256)) v.ntw = 4;
    // as many wavefronts and blocks in flight as leave the fewest loads past the end (480 tiles of 32 blocks, two to a workgroup: 16
    // wavefronts of 2 blocks 5.4 us, 8 of 5 5.8; of 40 blocks 8 of 5 6.4, 16 of 3 6.8)
    const int64_t each = ceil_div(KB, 8);
    if (each <= 3) { v.nw = 8; v.u = (int)each; }
    else if (v.ntw == 4) { v.nw = 8; v.u = tiles > 1280 ? 3 : 5; }
    else if (KB <= 32) { v.nw = 16; v.u = 2; }
    else if (KB <= 40) { v.nw = 8; v.u = 5; }
    else if (KB <= 48) { v.nw = 16; v.u = 3; }
    else if (v.ntw == 1) { v.nw = 16; v.u = 5; }
    else if (ceil_div(tiles, 2) <= 256) { v.nw = 16; v.u = 3; }
    else { v.nw = 8; v.u = 5; }
    return v;
}
// Slices of a contraction of at most 8 rows whose consumer, the LayerNorm kernel behind the two residual products of a batch step,
// adds them up.  The ffn value product has few tiles and a long contraction, so whole contractions make a few compute units draw much: cut in
// slices, with more tiles to a workgroup, all of them draw, and share the digits.  8 rows, us a launch with 1 / 2 / 3 / 4 slices: 2560 channels
// 11.1 / 9.0 / 7.5 / 8.1, 5120 27.0 / 22.8 / 18.5 / 22.2, 1024 6.3 / 4.4 / 4.1 / 3.7.  The LayerNorm workgroups, one for each row and mix, pay
// for it: 8 bytes a channel and slice, and the gate's 4, measured at 1.2 to 3.4 us.  Hence the 32 KB and the line at 7/10: 4 rows and fewer
// (2560 channels 8.7 / 7.6 / 6.8 / 7.3) and 4096 channels gain no more than that costs (step of 8 layers 767 us both ways).  Us a step of 8
// sequences, before (one tile to every workgroup of up to 320) / whole contractions / this: 24 layers of 1024 970 / 962 / 925, 12 of 1536
// 589 / 579 / 560, 8 of 2048 453 / 447 / 439, 12 of 2560 764 / 744 / 722, 4 of 5120 566 / 519 / 497; all with the same bits.
static int vec_split(int64_t MT, int64_t NT, int64_t KB, int readers) {
    auto draw = [&](int s) {
        const int64_t kb = ceil_div(KB, s);
        return vec_draw(NT * s, vec_shape(NT * s, kb, (int)MT).ntw, (int)MT) * kb;
    };
    int best = 1;
    int64_t least = draw(1) * 7 / 10;
    for (int s = 2; s <= kRowsDeferSlices; ++s) {
        const int64_t cost = draw(s) + 32 + readers * (2 * s + 1) * NT / 16;
        if (cost < least) { least = cost; best = s; }
    }
    return best;
}
// The kernel of that shape; null where there is none.  (More than one round only with the most blocks in flight.)
using VecKernel = void (*)(const GemmArgs);
static VecKernel vec_kernel(int MT, const VecShape &v, bool rounds, bool stream) {
#define RWKV_VEC(MT_, LO, HI, NTW, NW, U, ROUNDS)                                                     \
    if (MT >= LO && MT <= HI && v.ntw == NTW && v.nw == NW && v.u == U && rounds == ROUNDS)           \
        return stream ? gemv16_kernel<MT_, NTW, NW, U, true, ROUNDS> : gemv16_kernel<MT_, NTW, NW, U, false, ROUNDS>;
#define RWKV_VEC12(NTW, NW, U, ROUNDS) RWKV_VEC(1, 1, 1, NTW, NW, U, ROUNDS) RWKV_VEC(2, 2, 2, NTW, NW, U, ROUNDS)
#define RWKV_VEC34(NTW, NW, U, ROUNDS) RWKV_VEC(3, 3, 3, NTW, NW, U, ROUNDS) RWKV_VEC(4, 4, 4, NTW, NW, U, ROUNDS)
// (above 16 rows one kernel for two counts of M-tiles: the last one may be a copy)
#define RWKV_VEC68(NTW, NW, U, ROUNDS) RWKV_VEC(6, 5, 6, NTW, NW, U, ROUNDS) RWKV_VEC(8, 7, 8, NTW, NW, U, ROUNDS)
    RWKV_VEC12(4, 8, 1, false)
    RWKV_VEC12(4, 8, 2, false)
    RWKV_VEC12(4, 8, 3, false) RWKV_VEC12(4, 8, 3, true)
    RWKV_VEC12(4, 8, 5, false) RWKV_VEC12(4, 8, 5, true)
    RWKV_VEC12(2, 16, 2, false)
    RWKV_VEC12(2, 16, 3, false) RWKV_VEC12(2, 16, 3, true)
    RWKV_VEC12(2, 8, 1, false)
    RWKV_VEC12(2, 8, 2, false)
    RWKV_VEC12(2, 8, 3, false)
    RWKV_VEC12(2, 8, 5, false) RWKV_VEC12(2, 8, 5, true)
    RWKV_VEC12(1, 8, 1, false)
    RWKV_VEC12(1, 8, 2, false)
    RWKV_VEC12(1, 8, 3, false)
    RWKV_VEC12(1, 8, 5, false)
    RWKV_VEC12(1, 16, 2, false)
    RWKV_VEC12(1, 16, 3, false)
    RWKV_VEC12(1, 16, 5, false) RWKV_VEC12(1, 16, 5, true)
    RWKV_VEC34(2, 16, 1, false)
    RWKV_VEC34(2, 16, 2, false)
    RWKV_VEC34(2, 16, 3, false) RWKV_VEC34(2, 16, 3, true)
    RWKV_VEC34(2, 8, 1, false)
    RWKV_VEC34(2, 8, 2, false)
    RWKV_VEC34(2, 8, 3, false) RWKV_VEC34(2, 8, 3, true)
    RWKV_VEC34(1, 8, 1, false)
    RWKV_VEC34(1, 8, 2, false)
    RWKV_VEC34(1, 8, 3, false) RWKV_VEC34(1, 8, 3, true)
    RWKV_VEC34(1, 16, 1, false)
    RWKV_VEC34(1, 16, 2, false)
    RWKV_VEC34(1, 16, 3, false) RWKV_VEC34(1, 16, 3, true)
    RWKV_VEC68(2, 8, 1, false)
    RWKV_VEC68(2, 8, 2, false) RWKV_VEC68(2, 8, 2, true)
    RWKV_VEC68(1, 16, 1, false)
    RWKV_VEC68(1, 16, 2, false) RWKV_VEC68(1, 16, 2, true)
#undef RWKV_VEC
#undef RWKV_VEC12
#undef RWKV_VEC34
#undef RWKV_VEC68
    return nullptr;
}
// What a launch of so many M-tiles, column tiles and blocks would run; null without a kernel for it, or another kernel's.
const void *vec_kernel_of(int64_t MT, int64_t tiles, int64_t KB, int64_t kb_per_split) {
    if (!vec_rows(MT, tiles, KB)) return nullptr;
    const VecShape v = vec_shape(tiles, kb_per_split, (int)MT);
    return reinterpret_cast<const void *>(vec_kernel((int)MT, v, kb_per_split > v.nw * v.u, false));
}
static int launch_vec(hipStream_t st, const GemmArgs &g, bool stream) {
    const int64_t tiles = g.NT2 > 0 ? (int64_t)g.NT + g.NT2 : (int64_t)g.NT * g.gz;
    const VecShape v = vec_shape(tiles, g.kb_per_split, g.MT);
    const VecKernel kernel = vec_kernel(g.MT, v, g.kb_per_split > v.nw * v.u, stream);
    if (!kernel)
        return set_error(RWKV_ERR_SIZE, "gemv16_kernel: no instance for %d M-tiles, %lld column tiles, %d blocks", g.MT, (long long)tiles, g.KB);
    const dim3 grid((unsigned)(g.NT2 > 0 ? ceil_div(g.NT, v.ntw) + ceil_div(g.NT2, v.ntw) : ceil_div(g.NT, v.ntw) * g.gz)), block((unsigned)(64 * v.nw));
    hipLaunchKernelGGL(kernel, grid, block, 0, st, g);
    RWKV_CHECK_LAUNCH("gemv16_kernel");
    return RWKV_OK;
}

// Upper bound of the splits plan_products chooses for R rows, N columns and contractions of up to K, whatever the number of
// products in the launch.  A longer contraction only lifts the limit on the split, so from 33 rows on the plan for an
// unbounded one bounds every real one; 9 to 32 rows are cut in any number of slices or not at all; at most 8 rows split for the
// length's sake alone, which for no model's is needed (slices that are handed on: rows_deferred_bytes).
static int gemm_split_bound(int64_t R, int64_t N, int64_t K) {
    const int64_t MT = ceil_div(R, 4), NT = ceil_div(N, 16), any = (int64_t)1 << 40;
    if (MT > kVecMT && MT <= kSkinnyMT) return skinny_cut(NT, any, 1) ? kMaxSplit : 1;
    int s = 1;
    for (int n = 1; n <= kRowsMaxProducts; ++n) {
        const int sp = plan_products(MT, NT, MT <= kVecMT ? ceil_div(K, 64) : any, n).split;
        if (sp > s) s = sp;
    }
    return s;
}
size_t rows_tot_bytes(int64_t R, int64_t N, int64_t K) {
    return (size_t)(ceil_div(R, 4) * 4 * round_up(N, 16) * 8) * (size_t)gemm_split_bound(R, N, K);
}
size_t rows_deferred_bytes(int64_t R, int64_t N) {
    return R < kRowsDeferMax ? (size_t)(ceil_div(R, 4) * 4 * round_up(N, 16) * 8) * kRowsDeferSlices : 0;
}
// What rows_quant keeps in its scratch area for R rows of K values (0: that shape does not use it).
// (a few long rows are quantised by several workgroups each, in two launches: one workgroup per row leaves most of the
// device idle - 14B shape, batch step of 32 sequences: 7.78 against 8.10 ms)
static bool quant_uses_parts(int64_t R, int64_t K) { return R <= 64 && K >= 8192; }
// Rows that have four times the threads: up to 384 of them (300 tokens, 10 layers of 5120 4883 / 4849 us a prompt, 16 of 4096 5760 / 5701; from
// 500 on, and at 2560 channels from 300 on, it makes no difference, and alone with warm caches 400 rows are 10 % slower), and of so many
// values that a wavefront of the narrower form has more than two groups a lane (from 6144 values on: 256 tokens of 5120 channels
// 4067 us, this 4049).
constexpr int kLongQuantRows = 384, kLongQuantFrom = 2048;
size_t rows_quant_scratch_bytes(int64_t R, int64_t K) {
    if (!quant_uses_parts(R, K)) return 0;
    return (size_t)(R * ceil_div(K, 4 * kRT * kQuantPartSeg) * 2 * 8);
}
size_t rows_pass_tot_bytes(int64_t R, int64_t C, int64_t F, int64_t V, int64_t head_rows) {
    const int64_t K = std::max(F, C);
    // Each product for itself: fewer columns may be cut where more are not, so the totals of the widest do not hold those of every narrower one
    // (32 rows of 1024 channels: 16000 columns of logits are cut in two, 16384 hidden values are not).  k, v, r share a launch.
    size_t n = std::max(3 * rows_tot_bytes(R, C, K), std::max(rows_tot_bytes(R, F, C), rows_tot_bytes(head_rows, V, C)));
    n = std::max(n, rows_deferred_bytes(R, C));             // a residual update handed on in slices
    return std::max(n, rows_quant_scratch_bytes(R, K));     // the quantisers' partial records, before a product starts
}
// Batches of fewer than kRowsDeferMax rows, and the short prompts of narrow models, although a row of a sequence adds up the slices of the row
// before it as well.  Us a prompt, a launch for the sums / handed on: 12 layers of 512, 40 and 127 tokens 679, 743 / 653, 720; 24 of
// 1024, 77 and 127 1741, 1840 / 1695, 1788; 12 of 1536, 77 and 100 1074, 1135 / 1056, 1142; 12 of 2048, 64 and 77 1151, 1174 / 1136, 1186; 12 of
// 2560, 32 and 127 1067, 1502 / 1076, 1556; 8 of 4096, 32 1004 / 1036.  (That is att output, and ffn value where it is cut in six at most: the general
// kernel cuts it in eight for 33 to 127 tokens of 1024 channels, 33 to 64 of 1536 and 2048, and those slices keep their launch.)
int rows_readers(int64_t R, int64_t C, bool sequence) {
    if (R >= kRowsDeferMax) return 0;
    if (!sequence) return 1;
    return C <= 2048 && R * C <= (1 << 17) ? 2 : 0;
}
void rows_plan_describe(int64_t R, int64_t K, int64_t N, int n, int readers, int out[4]) {
    const ProductPlan p = plan_products(ceil_div(R, 4), ceil_div(N, 16), K / 64, n, readers);
    out[0] = p.kind == PLAN_NARROW ? (int)PLAN_WIDE : p.kind; out[1] = p.gx; out[2] = p.gy; out[3] = p.split;
}

int rows_embed(hipStream_t st, const int64_t *tokens, int64_t R, int V, int C, const float *emb, const double *w,
               const double *b, double *x) {
    hipLaunchKernelGGL(rows_embed_kernel, dim3((unsigned)R), dim3(kRT), 0, st, tokens, V, C, emb, w, b, x);
    RWKV_CHECK_LAUNCH("rows_embed_kernel");
    return RWKV_OK;
}

bool rows_ln_width_supported(int64_t C) { return C % 4 == 0 && C <= kLnMaxWidth; }

int rows_ln_mix_quant(hipStream_t st, int n_mix, int64_t R, int C, bool sequence, const double *x, const double *ln_w,
                      const double *ln_b, const double *mu, const double *prev0, double *shift_dst,
                      int64_t prev_stride, const float *const *range, const double *const *offset,
                      const RowsOperand *out, const RowsFew *few) {
    if (C % 64 != 0 || !rows_ln_width_supported(C))
        return set_error(RWKV_ERR_SIZE, "rows_ln_mix_quant: width %d is not a multiple of 64 up to %d", C, kLnMaxWidth);
    LnQuantArgs a;
    a.C = C; a.R = (int)R; a.sequence = sequence ? 1 : 0; a.x = x; a.ln_w = ln_w; a.ln_b = ln_b; a.mu = mu;
    a.add.tot = nullptr; a.x_out = nullptr; a.shift_out = nullptr; a.commit_src = nullptr; a.commit_dst = nullptr;
    if (few) {
        if (few->add.tot && ((few->add.op != ROW_ADD && few->add.op != ROW_GATE_ADD) || few->x_out == x))
            return set_error(RWKV_ERR_ARG, "rows_ln_mix_quant: a pending product needs a residual tail and another buffer for the new x");
        if (sequence && few->add.tot && C > 4 * kLnRowThreads)          // (the registers of wider rows do not hold the row before as well)
            return set_error(RWKV_ERR_ARG, "rows_ln_mix_quant: a pending product of a sequence needs rows of at most %d channels", 4 * kLnRowThreads);
        if (R >= kRowsDeferMax && (few->add.tot || (!sequence && (few->shift_out || few->commit_src))))
            return set_error(RWKV_ERR_ARG, "rows_ln_mix_quant: pending work needs fewer than %d rows", (int)kRowsDeferMax);
        a.add = few->add; a.x_out = few->x_out; a.commit_src = few->commit_src; a.commit_dst = few->commit_dst;
        if (sequence && few->shift_out) shift_dst = few->shift_out;      // (its last row alone)
        else a.shift_out = few->shift_out;
    }
    // (a row has a workgroup for each mix: none may write what another still reads)
    for (int k = 0; n_mix > 1 && a.add.tot && k < n_mix; ++k)
        if (out[k].S == a.add.S || out[k].qs == a.add.qs || out[k].zp == a.add.zp)
            return set_error(RWKV_ERR_ARG, "rows_ln_mix_quant: the row constants of a pending product may not be those of an output");
    if (n_mix > 0 && (sequence ? prev0 == shift_dst : R < kRowsDeferMax && !a.shift_out))
        return set_error(RWKV_ERR_ARG, "rows_ln_mix_quant: few rows and sequences need their shift rows kept apart");
    a.prev0 = prev0; a.shift_dst = shift_dst; a.prev_stride = prev_stride;
    const int n_out = n_mix > 0 ? n_mix : 1;
    for (int m = 0; m < 3; ++m) {
        const int k = m < n_out ? m : 0;
        a.range[m] = range[k]; a.offset[m] = offset[k];
        a.dig[m] = out[k].dig; a.S[m] = out[k].S; a.qs[m] = out[k].qs; a.zp[m] = out[k].zp;
    }
    // few rows: a workgroup per row and mix; many rows: one per row, 256 threads with more channels each, which keeps more
    // rows resident per compute unit
    const bool many = R >= kRowsDeferMax;
    if (!many) {
        const int64_t threads = round_up(ceil_div(C, 4), 64);
        const dim3 grid((unsigned)R, (unsigned)n_out), block((unsigned)(threads < kLnRowThreads ? threads : kLnRowThreads));
        const int nseg = (int)ceil_div(C, 4 * kLnRowThreads);           // 1 .. 3 (kLnMaxWidth)
        if (n_mix == 0) {
            if (nseg == 1) hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<false, 1>), grid, block, 0, st, a);
            else if (nseg == 2) hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<false, 2>), grid, block, 0, st, a);
            else hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<false, 3>), grid, block, 0, st, a);
        } else {
            if (nseg == 1 && threads > kLnRowThreads / 2 && R * n_out > 256) hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<true, 1, true>), grid, block, 0, st, a);
            else if (nseg == 1) hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<true, 1>), grid, block, 0, st, a);
            else if (nseg == 2) hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<true, 2>), grid, block, 0, st, a);
            else hipLaunchKernelGGL((rows_ln_mix_quant_row_kernel<true, 3>), grid, block, 0, st, a);
        }
        RWKV_CHECK_LAUNCH("rows_ln_mix_quant_row_kernel");
        return RWKV_OK;
    }
    const bool small = C <= 3 * 4 * 256;
    const dim3 grid((unsigned)R), block(256);
    // A workgroup to each mix where the rows alone are too few (us a prompt of 300, 400, 500 tokens, a workgroup to each row / mix:
    // 10 layers of 5120 4884, 6350 / 4813, 6307; 16 of 4096, 300 and 500 5760, 7572 / 5666, 7708; 24 of 2560 5339, 5765, 6308 / 5344, 5845, 6517).
    if (sequence && n_mix > 1 && R <= (small ? 256 : 384)) {
        const dim3 apart((unsigned)R, (unsigned)n_mix);
        if (small) hipLaunchKernelGGL((rows_ln_mix_quant_split_kernel<3, 256>), apart, block, 0, st, a);
        else hipLaunchKernelGGL((rows_ln_mix_quant_split_kernel<6, 256>), apart, block, 0, st, a);
        RWKV_CHECK_LAUNCH("rows_ln_mix_quant_split_kernel");
        return RWKV_OK;
    }
#define RWKV_LNQ(NM)                                                                                  \
    do {                                                                                              \
        if (small && R <= 512) hipLaunchKernelGGL((rows_ln_mix_quant_few_kernel<NM, 3, 256>), grid, block, 0, st, a);   \
        else if (small) hipLaunchKernelGGL((rows_ln_mix_quant_kernel<NM, 3, 256>), grid, block, 0, st, a);   \
        else hipLaunchKernelGGL((rows_ln_mix_quant_kernel<NM, 6, 256>), grid, block, 0, st, a);       \
    } while (0)
    switch (n_mix) {
        case 0: RWKV_LNQ(0); break;
        case 2: RWKV_LNQ(2); break;
        case 3: RWKV_LNQ(3); break;
        default: return set_error(RWKV_ERR_ARG, "rows_ln_mix_quant: unsupported mix count %d", n_mix);
    }
#undef RWKV_LNQ
    RWKV_CHECK_LAUNCH("rows_ln_mix_quant_kernel");
    return RWKV_OK;
}

int rows_quant(hipStream_t st, int64_t R, int64_t K, const void *in, bool in_f32, const float *range, const double *offset,
               const RowsOperand &out, double *scratch) {
    if (K % 64 != 0) return set_error(RWKV_ERR_SIZE, "rows_quant: contraction length %lld is not a multiple of 64",
                                      (long long)K);
    QuantArgs q;
    q.K = (int)K; q.in = in; q.range = range; q.offset = offset; q.dig = out.dig; q.S = out.S; q.qs = out.qs; q.zp = out.zp;
    const dim3 grid((unsigned)R), block(kRT);
    if (scratch && quant_uses_parts(R, K)) {
        QuantPartArgs pa;
        pa.q = q; pa.G = (int)ceil_div(K, 4 * kRT * kQuantPartSeg); pa.quads_per_part = (int)round_up(ceil_div(K / 4, pa.G), 4);    // whole groups of 16 values: four lanes share a fragment slot
        pa.part = scratch;
        const dim3 pg((unsigned)pa.G, (unsigned)R);
        if (in_f32) {
            hipLaunchKernelGGL((rows_quant_part_kernel<false, float>), pg, block, 0, st, pa);
            hipLaunchKernelGGL((rows_quant_part_kernel<true, float>), pg, block, 0, st, pa);
        } else {
            hipLaunchKernelGGL((rows_quant_part_kernel<false, double>), pg, block, 0, st, pa);
            hipLaunchKernelGGL((rows_quant_part_kernel<true, double>), pg, block, 0, st, pa);
        }
        RWKV_CHECK_LAUNCH("rows_quant_part_kernel");
        return RWKV_OK;
    }
    if (R <= kLongQuantRows && K > kLongQuantFrom && K <= 20 * 4 * kRT && in_f32) {
        if (K <= 4 * 4 * kRT) hipLaunchKernelGGL((rows_quant_long_kernel<1, float>), grid, dim3(4 * kRT), 0, st, q);
        else if (K <= 8 * 4 * kRT) hipLaunchKernelGGL((rows_quant_long_kernel<2, float>), grid, dim3(4 * kRT), 0, st, q);
        else if (K <= 12 * 4 * kRT) hipLaunchKernelGGL((rows_quant_long_kernel<3, float>), grid, dim3(4 * kRT), 0, st, q);
        else hipLaunchKernelGGL((rows_quant_long_kernel<5, float>), grid, dim3(4 * kRT), 0, st, q);
        RWKV_CHECK_LAUNCH("rows_quant_long_kernel");
        return RWKV_OK;
    }
#define RWKV_QUANT_LAUNCH(T)                                                                          \
    do {                                                                                              \
        if (K <= 3 * 4 * kRT) hipLaunchKernelGGL((rows_quant4_kernel<3, T>), grid, block, 0, st, q);          \
        else if (K <= 6 * 4 * kRT) hipLaunchKernelGGL((rows_quant4_kernel<6, T>), grid, block, 0, st, q);     \
        else if (K <= 10 * 4 * kRT) hipLaunchKernelGGL((rows_quant4_kernel<10, T>), grid, block, 0, st, q);   \
        else if (K <= 20 * 4 * kRT) hipLaunchKernelGGL((rows_quant4_kernel<20, T>), grid, block, 0, st, q);   \
        else hipLaunchKernelGGL((rows_quant_kernel<3, T>), grid, block, 0, st, q);      /* any length: a second read past 12288 */ \
    } while (0)
    if (in_f32) RWKV_QUANT_LAUNCH(float);
    else RWKV_QUANT_LAUNCH(double);
#undef RWKV_QUANT_LAUNCH
    RWKV_CHECK_LAUNCH("rows_quant_kernel");
    return RWKV_OK;
}

static int launch_skinny(hipStream_t st, const GemmArgs &g, const dim3 &grid, bool stream) {
    const bool four = g.MT <= 4;
    hipLaunchKernelGGL(four ? (stream ? gemm8_skinny_kernel<4, true> : gemm8_skinny_kernel<4, false>)
                            : (stream ? gemm8_skinny_kernel<8, true> : gemm8_skinny_kernel<8, false>), grid, dim3(256), 0, st, g);
    RWKV_CHECK_LAUNCH("gemm8_skinny_kernel");
    return RWKV_OK;
}
static int launch_general(hipStream_t st, GemmArgs &g, int kind, int gx, bool stream) {
    const bool wide = kind == PLAN_WIDE;
    g.gx = gx; g.gy = (int)ceil_div(g.MT, 16); g.by_rows = g.gy >= kXcds;
    g.per_xcd = ((g.by_rows ? g.gy : gx) + kXcds - 1) / kXcds;
    const dim3 grid((unsigned)(kXcds * g.per_xcd * (g.by_rows ? gx : g.gy) * g.gz));
    if (kind == PLAN_NARROW) hipLaunchKernelGGL(gemm8_narrow_kernel, grid, dim3(512), 0, st, g);
    else if (wide) hipLaunchKernelGGL(gemm8_wide_kernel, grid, dim3(512), 0, st, g);
    else if (stream && g.gy <= kStreamRowBlocks) hipLaunchKernelGGL(gemm8_kernel<true>, grid, dim3(512), 0, st, g);
    else hipLaunchKernelGGL(gemm8_kernel<false>, grid, dim3(512), 0, st, g);
    RWKV_CHECK_LAUNCH(kind == PLAN_NARROW ? "gemm8_narrow_kernel" : wide ? "gemm8_wide_kernel" : "gemm8_kernel");
    return RWKV_OK;
}

int rows_products(hipStream_t st, int n, const RowsProduct *p, long long *tot, int64_t R, int64_t K, int64_t N, int op,
                  const float *gate, RowsDeferred *defer, bool sequence) {
    if (K % 64 != 0) return set_error(RWKV_ERR_SIZE, "rows_products: contraction length %lld is not a multiple of 64",
                                      (long long)K);
    if (n < 1 || n > kRowsMaxProducts) return set_error(RWKV_ERR_ARG, "rows_products: %d products in one launch", n);
    if (op < ROW_STORE || op > ROW_STORE_F32) return set_error(RWKV_ERR_ARG, "rows_products: unknown tail %d", op);
    GemmArgs g;
    FinishArgs f;
    for (int m = 0; m < kRowsMaxProducts; ++m) {
        const RowsProduct &q = p[m < n ? m : 0];
        g.dig[m] = q.a.dig; g.w16[m] = q.w16; g.S[m] = q.a.S; g.qs[m] = q.a.qs; g.zp[m] = q.a.zp; g.out[m] = q.out;
        f.S[m] = q.a.S; f.qs[m] = q.a.qs; f.zp[m] = q.a.zp; f.out[m] = q.out;
    }
    g.tot = tot;
    g.MT = (int)ceil_div(R, 4); g.NT = (int)ceil_div(N, 16); g.KB = (int)(K / 64); g.ldd = g.NT * 16;
    g.R = (int)R; g.N = (int)N; g.gate = gate;
    const ProductPlan pl = plan_products(g.MT, g.NT, g.KB, n, defer && R < kRowsDeferMax ? (sequence ? 2 : 1) : 0);
    const int split = pl.split;
    g.kb_per_split = (int)ceil_div(g.KB, split);
    g.split = split;
    g.slice = (size_t)g.MT * 4 * g.ldd;
    g.gz = split * n;
    g.tail = split > 1 ? -1 : op;
    g.NT2 = g.N2 = g.tail2 = 0;
    g.apart = rounded_apart(g.MT, g.NT, g.KB, n); g.apart2 = 0;
    g.part = nullptr;
    if (pl.kind == PLAN_VEC) {
        g.gx = g.NT; g.gy = 1; g.by_rows = 0; g.per_xcd = 0;
        const int rc = launch_vec(st, g, p[0].stream);
        if (rc) return rc;
    } else if (pl.kind == PLAN_SKINNY) {
        g.gx = pl.gx; g.gy = 1; g.by_rows = 0; g.per_xcd = (pl.gx + kXcds - 1) / kXcds;
        const dim3 grid((unsigned)(kXcds * g.per_xcd * g.gz));
        const int rc = launch_skinny(st, g, grid, p[0].stream);
        if (rc) return rc;
    } else {
        const int rc = launch_general(st, g, pl.kind, pl.gx, p[0].stream);
        if (rc) return rc;
    }
    for (int m = 0; defer && m < n; ++m) defer[m].tot = nullptr;
    if (split == 1) return RWKV_OK;     // the tail was applied in the product's epilogue
    if (defer && R < kRowsDeferMax && split <= kRowsDeferSlices) {   // the consumer adds the slices up
        const bool fused = gate_fused(pl.kind, sequence, g.NT, g.KB);
        for (int m = 0; m < n; ++m)
            defer[m] = RowsDeferred{tot + (size_t)m * split * g.slice, g.slice, split, g.ldd, op, g.apart != 0, fused, p[m].a.S, p[m].a.qs, p[m].a.zp, gate};
        return RWKV_OK;
    }

    f.R = (int)R; f.N = (int)N; f.ldd = g.ldd; f.slices = split; f.slice = g.slice; f.tot = tot; f.gate = gate;
    const dim3 fg((unsigned)ceil_div(N, 256), (unsigned)R, (unsigned)n), fb(256);
    switch (op) {
        case ROW_STORE: hipLaunchKernelGGL(rows_finish_kernel<ROW_STORE>, fg, fb, 0, st, f); break;
        case ROW_RELU2: hipLaunchKernelGGL(rows_finish_kernel<ROW_RELU2>, fg, fb, 0, st, f); break;
        case ROW_ADD: hipLaunchKernelGGL(rows_finish_kernel<ROW_ADD>, fg, fb, 0, st, f); break;
        case ROW_STORE_F32: hipLaunchKernelGGL(rows_finish_kernel<ROW_STORE_F32>, fg, fb, 0, st, f); break;
        default: hipLaunchKernelGGL(rows_finish_kernel<ROW_GATE_ADD>, fg, fb, 0, st, f); break;
    }
    RWKV_CHECK_LAUNCH("rows_finish_kernel");
    return RWKV_OK;
}

// Whether ffn key (NT tiles) and receptance (NT2) of more than 32 rows share a launch of the general kernel, whole contractions:
// what it saves is a launch, about 3 us at a third of a microsecond a contraction block, and part of another where slices had to
// be added up; what it may cost is a round of workgroups more.  Us a prompt apart / together: 24 layers of
// 1024, 33 / 77 / 127 / 500 tokens 2055 / 2143 / 2368 / 2912 against 1792 / 1890 / 2019 / 2763; 12 of 2560, 64 / 77 / 200 / 500 1525 / 1572 / 2198 / 3327
// against 1383 / 1416 / 2097 / 3279; 6 of 5120, 33 / 300 1244 / 3032 against 1155 / 2921.  Together all the same where the rule says apart: 6
// of 4096, 77 1255 / 1268; 12 of 1536, 300 1671 / 1702; 12 of 2560, 1000 (the receptance alone: one round of the wide kernel) 4846 / 4971.
static bool pair_general(int64_t MT, int64_t NT, int64_t NT2, int64_t KB) {
    if (MT <= kSkinnyMT || KB > 1024) return false;
    const int64_t gy = ceil_div(MT, 16);
    int64_t saved = 290;
    auto alone = [&](int64_t nt) {                          // in ninths, as kGemmWideDen weighs the wide kernel
        const ProductPlan p = plan_products(MT, nt, KB, 1);
        if (p.split > 1) saved += 60;
        if (p.kind == PLAN_NARROW) return (int64_t)kGemmWideDen * kGemmNarrowCost;
        return p.kind == PLAN_WIDE ? kGemmWideNum * 40 * ceil_div((int64_t)p.gx * p.gy, 256) : kGemmWideDen * general_cost((int64_t)p.gx * p.gy * p.split) / p.split;
    };
    const int64_t more = kGemmWideDen * general_cost((ceil_div(NT, kGemmNT) + ceil_div(NT2, kGemmNT)) * gy) - alone(NT) - alone(NT2);
    return more * KB <= kGemmWideDen * saved;
}

// Few rows: both in one launch, whole contractions (the receptance's column blocks find room beside the key's; apart they
// were up to four launches, two of them only adding slices).  With gemv16_kernel's shapes: 8 sequences at 3B 2.96 -> 2.40 ms
// a step, 32 at 14B 7.38 -> 6.66 ms (its two launches and the receptance's sum of slices: 31.8 + 13.5 + 4.6 us, one launch 37.5).
int rows_ffn_key_receptance(hipStream_t st, bool sequence, const RowsProduct &k, const RowsProduct &r, long long *tot, int64_t R, int64_t C, int64_t F,
                            const float *range, const double *offset, const RowsOperand &out) {
    GemmArgs g;
    const RowsProduct *p[2] = {&k, &r};
    for (int m = 0; m < kRowsMaxProducts; ++m) {
        const RowsProduct &q = *p[m == 1];
        g.dig[m] = q.a.dig; g.w16[m] = q.w16; g.S[m] = q.a.S; g.qs[m] = q.a.qs; g.zp[m] = q.a.zp; g.out[m] = q.out;
    }
    g.tot = nullptr; g.slice = 0; g.gate = nullptr;
    g.MT = (int)ceil_div(R, 4); g.NT = (int)ceil_div(F, 16); g.KB = (int)(C / 64); g.ldd = g.NT * 16;
    g.kb_per_split = g.KB; g.split = 1; g.gz = 1; g.gy = 1; g.by_rows = 0;
    g.tail = ROW_RELU2; g.R = (int)R; g.N = (int)F;
    g.part = nullptr;
    g.NT2 = (int)ceil_div(C, 16); g.N2 = (int)C; g.tail2 = ROW_STORE_F32;
    g.apart = rounded_apart(g.MT, g.NT, g.KB, 1); g.apart2 = rounded_apart(g.MT, g.NT2, g.KB, 1);
    const int gx = (int)(ceil_div(g.NT, kSkinnyNT) + ceil_div(g.NT2, kSkinnyNT));
    if (C % 64 == 0 && vec_rows(g.MT, g.NT + g.NT2, g.KB) && g.KB <= 1024) {
        g.gx = g.NT; g.per_xcd = 0;
        // (not for the rows of a sequence: the tiles add up the zero-point term in another order than rows_quant does, and the
        // last bit of it reaches the logits and a seeded sampler's texts)
        if (F > 3072 && !sequence) g.part = reinterpret_cast<double2 *>(tot);       // (16 bytes per row and tile: no more than a slice of totals)
        g.next_range = range; g.next_offset = offset; g.next_qs = out.qs;
        const int rc = launch_vec(st, g, k.stream);
        if (rc) return rc;
        if (!g.part) return rows_quant(st, R, F, k.out, true, range, offset, out, (double *)tot);
        QuantArgs q;
        q.K = (int)F; q.in = k.out; q.range = range; q.offset = offset; q.dig = out.dig; q.S = out.S; q.qs = out.qs; q.zp = out.zp;
        hipLaunchKernelGGL(rows_quant_tiles_kernel, dim3((unsigned)ceil_div(F, 4 * kRT), (unsigned)R), dim3(kRT), 0, st, q, g.part, g.NT);
        RWKV_CHECK_LAUNCH("rows_quant_tiles_kernel");
        return RWKV_OK;
    } else if (C % 64 == 0 && g.MT <= kSkinnyMT && gx >= kSkinnyPairWgs) {
        g.gx = gx; g.per_xcd = (gx + kXcds - 1) / kXcds;
        const dim3 grid((unsigned)(kXcds * g.per_xcd));
        const int rc = launch_skinny(st, g, grid, k.stream);
        if (rc) return rc;
    } else if (pair_general(g.MT, g.NT, g.NT2, g.KB)) {
        const int rc = launch_general(st, g, PLAN_GENERAL, (int)(ceil_div(g.NT, kGemmNT) + ceil_div(g.NT2, kGemmNT)), k.stream);
        if (rc) return rc;
    } else {
        int rc = rows_products(st, 1, &k, tot, R, C, F, ROW_RELU2, nullptr);
        if (!rc) rc = rows_products(st, 1, &r, tot, R, C, C, ROW_STORE_F32, nullptr);
        if (rc) return rc;
    }
    return rows_quant(st, R, F, k.out, true, range, offset, out, (double *)tot);
}

int rows_wkv(hipStream_t st, int64_t R, int C, bool sequence, const float *k, const float *v, const float *r,
             const double *w, const double *u, double *state, int64_t state_stride, float *out, const RowsDeferred *kvr) {
    WkvRowsArgs a;
    a.C = C; a.R = (int)R; a.sequence = sequence ? 1 : 0; a.k = k; a.v = v; a.r = r; a.w = w; a.u = u;
    a.state = state; a.state_stride = state_stride; a.out = out;
    for (int i = 0; i < 3; ++i) {
        if (kvr) a.pend[i] = kvr[i];
        else a.pend[i].tot = nullptr;
        if (a.pend[i].tot && (sequence || a.pend[i].op != ROW_STORE_F32))
            return set_error(RWKV_ERR_ARG, "rows_wkv: a pending product needs batch rows and the float32 store tail");
        if ((a.pend[i].tot == nullptr) != (a.pend[0].tot == nullptr) || (a.pend[i].tot && a.pend[i].slices != a.pend[0].slices))
            return set_error(RWKV_ERR_ARG, "rows_wkv: k, v and r are pending together, in as many slices, or none of them is");
    }
    if (sequence && R >= kWkvSeqMin) {
        // short sequences: the smallest block that covers them leaves the fewest lanes idle
        const dim3 g8((unsigned)(C / 8)), g16((unsigned)(C / 16));
        if (R <= 32) hipLaunchKernelGGL((wkv_seq_kernel<8, 8, 4, 1, false>), g8, dim3(64), 0, st, a);
        else if (R < kWkvChunked) hipLaunchKernelGGL((wkv_seq_kernel<8, 8, 8, 1, false>), g8, dim3(64), 0, st, a);
        else if (C <= kWkvNarrow / 2 && R <= 4 * kWkvChunk) hipLaunchKernelGGL((wkv_seq_kernel<8, 8, 4, 4, true>), g8, dim3(256), 0, st, a);
        else if (C <= kWkvNarrow && R > 4 * kWkvChunk) hipLaunchKernelGGL((wkv_seq_kernel<8, 8, 4, 8, true>), g8, dim3(512), 0, st, a);
        else if (R <= 4 * kWkvChunk || C >= kWkvWide) hipLaunchKernelGGL((wkv_seq_kernel<16, 4, 8, 4, true>), g16, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((wkv_seq_kernel<16, 4, 8, 8, true>), g16, dim3(512), 0, st, a);
        RWKV_CHECK_LAUNCH("wkv_seq_kernel");
        return RWKV_OK;
    }
    hipLaunchKernelGGL(wkv_rows_kernel, dim3((unsigned)ceil_div(C, 64), sequence ? 1u : (unsigned)R), dim3(64), 0, st, a);
    RWKV_CHECK_LAUNCH("wkv_rows_kernel");
    return RWKV_OK;
}

// Plan of the stand-alone product: tiles per workgroup ntw and wavefronts per workgroup nw (chunks of kMvCB blocks).
// Every workgroup must be resident at once - a second round of workgroups would start its loads only when the
// first has drained - so the wavefronts take several chunks in turn where one chunk each would not fit.  Two
// tiles per workgroup (half the fragment traffic) only where that leaves a workgroup for every compute unit.
constexpr int kMvCB = 4;
struct Mv16Plan { int ntw, nw, n_chunks; };

static Mv16Plan mv16_plan(int64_t KB, int64_t NT, int MT) {
    const int n_chunks = (int)ceil_div(KB, kMvCB);
    const int ntw = NT >= 512 ? 2 : 1;
    const int vgprs = ntw == 2 ? (MT == 2 ? 112 : 88) : (MT == 2 ? 96 : 64);      // mv16_kernel<MT, ntw> as compiled
    const int waves_per_cu = 4 * (512 / vgprs > 8 ? 8 : 512 / vgprs);
    const int64_t grid = ceil_div(NT, ntw);
    for (int rounds = 1; rounds <= n_chunks; ++rounds) {
        const int nw = (int)ceil_div(n_chunks, rounds);
        if (nw > 16) continue;
        if (nw <= ntw || grid <= 256 * (int64_t)(waves_per_cu / nw)) return Mv16Plan{ntw, nw < ntw ? ntw : nw, n_chunks};
    }
    return Mv16Plan{ntw, ntw, n_chunks};
}

size_t rows_mv16_workspace_bytes(int64_t B, int64_t n_in) {
    if (B <= 0 || n_in <= 0) return 0;
    const int64_t KB = ceil_div(n_in, 64), MT = ceil_div(B, 4);
    return (size_t)(MT * KB * 1024) + (size_t)round_up(B * ceil_div(KB, 4) * 4 * 8, 256);
}

int rows_mv16(hipStream_t st, int64_t B, int64_t n_in, int64_t n_out, const float *x, const uint8_t *w16,
              const float *r_row, const double *m_row, const float *r_col, const float *m_col, double *y, void *ws) {
    Mv16Args a;
    a.B = (int)B; a.n_in = (int)n_in; a.n_out = (int)n_out; a.KB = (int)ceil_div(n_in, 64);
    const int MT = (int)ceil_div(B, 4);
    const int64_t NT = ceil_div(n_out, 16);
    const Mv16Plan pl = mv16_plan(a.KB, NT, MT);
    const int nw = pl.nw, ntw = pl.ntw;
    a.n_chunks = pl.n_chunks;
    a.x = x; a.r_row = r_row; a.m_row = m_row; a.r_col = r_col; a.m_col = m_col; a.w16 = w16; a.y = y;
    a.dig = static_cast<signed char *>(ws);
    a.rec = reinterpret_cast<double *>(static_cast<char *>(ws) + (size_t)MT * a.KB * 1024);
    const dim3 qg((unsigned)a.n_chunks, (unsigned)MT);
    hipLaunchKernelGGL(mv16_quant_kernel<kMvCB>, qg, dim3(256), 0, st, a);
    RWKV_CHECK_LAUNCH("mv16_quant_kernel");
    const dim3 grid((unsigned)ceil_div(NT, ntw)), block((unsigned)(64 * nw));
    const size_t lds = ((size_t)nw * MT * ntw * 64 + 4 * MT * 3) * sizeof(double);
    if (ntw == 2) {
        if (MT == 1) hipLaunchKernelGGL((mv16_kernel<1, kMvCB, 2>), grid, block, lds, st, a);
        else hipLaunchKernelGGL((mv16_kernel<2, kMvCB, 2>), grid, block, lds, st, a);
    } else {
        if (MT == 1) hipLaunchKernelGGL((mv16_kernel<1, kMvCB, 1>), grid, block, lds, st, a);
        else hipLaunchKernelGGL((mv16_kernel<2, kMvCB, 1>), grid, block, lds, st, a);
    }
    RWKV_CHECK_LAUNCH("mv16_kernel");
    return RWKV_OK;
}

}  // namespace rwkv
