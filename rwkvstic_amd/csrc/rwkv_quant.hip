// Quantiser (reference agnostic/backends/modules/matmul.py:18-40) and the
// packed weight layout: pack / unpack / canonical dequantisation.
#include "rwkv_common.h"

#include <algorithm>
#include <string>

namespace rwkv {

static thread_local char g_err[512] = "";

int set_error(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

// ---------------------------------------------------------------------------
// One workgroup owns 64 input channels of weight[n_out, n_in] and walks every
// row twice: thread (jx, ky) handles channel j0+jx, rows ky, ky+4, ... so each
// load is a coalesced 256-byte row segment.  Pass 1 finds min/max; pass 2
// forms the float64 quotient, writes the truncated codes (64x64 tiles
// transposed through LDS so the [n_in, n_out] store is coalesced too) and
// accumulates the truncated fractions for the offset.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
quantize_kernel(const float *__restrict__ W, int64_t n_out, int64_t n_in,
                uint8_t *__restrict__ codes, float *__restrict__ range,
                double *__restrict__ offset) {
    __shared__ float smin[4][64], smax[4][64];
    __shared__ double sfr[4][64];
    __shared__ uint8_t tile[64][68];
    const int jx = threadIdx.x & 63, ky = threadIdx.x >> 6;
    const int64_t j0 = (int64_t)blockIdx.x * 64;
    const int64_t j = j0 + jx;
    const bool live = j < n_in;

    float lo_f = INFINITY, hi_f = -INFINITY;
    if (live)
        for (int64_t k = ky; k < n_out; k += 4) {
            const float x = W[k * n_in + j];
            lo_f = fminf(lo_f, x);
            hi_f = fmaxf(hi_f, x);
        }
    smin[ky][jx] = lo_f;
    smax[ky][jx] = hi_f;
    __syncthreads();
    lo_f = fminf(fminf(smin[0][jx], smin[1][jx]), fminf(smin[2][jx], smin[3][jx]));
    hi_f = fmaxf(fmaxf(smax[0][jx], smax[1][jx]), fmaxf(smax[2][jx], smax[3][jx]));
    // matmul.py:31-33: min in float64; range = max(x - min) / 255 in float64
    const double lo = (double)lo_f;
    const double ran = ((double)hi_f - lo) / 255.0;

    double fr = 0.0;
    for (int64_t k0 = 0; k0 < n_out; k0 += 64) {
        for (int r = ky; r < 64; r += 4) {
            const int64_t k = k0 + r;
            uint8_t c = 0;
            if (live && k < n_out && ran > 0.0) {
                const double q = ((double)W[k * n_in + j] - lo) / ran;  // matmul.py:32-34
                const double t = trunc(q);
                c = (uint8_t)(int)t;     // .to(uint8) truncates, matmul.py:21
                fr += q - t;             // out.frac(), matmul.py:35
            }
            tile[jx][r] = c;
        }
        __syncthreads();
        for (int r = ky; r < 64; r += 4) {
            const int64_t jj = j0 + r, k = k0 + jx;
            if (jj < n_in && k < n_out) codes[jj * n_out + k] = tile[r][jx];
        }
        __syncthreads();
    }
    sfr[ky][jx] = fr;
    __syncthreads();
    if (ky == 0 && live) {
        const double fsum = (sfr[0][jx] + sfr[1][jx]) + (sfr[2][jx] + sfr[3][jx]);
        offset[j] = lo + (fsum / (double)n_out) * ran;   // matmul.py:36-37
        range[j] = (float)ran;                            // matmul.py:39
    }
}

// ---------------------------------------------------------------------------
// The same quantiser for callers with a workspace: two launches that cut the matrix both ways, and the codes leave
// in any of the three layouts straight from the encoding pass.  Codes, ranges and offsets have quantize_kernel's bits.
//
// Bound: memory (the float32 matrix twice, the second time mostly from the memory-side cache, the codes once per
// layout).  quantize_kernel walks all rows with one workgroup per 64 channels, 40 workgroups at 2560 channels, and
// the packed layouts then read its codes back byte by byte.  The seven matrices of a layer of width 2560: 5.14 ms
// that way, 0.282 ms here (0.319 with the host's calls in front of them; the 511 MB at copy rate: 0.108).  The offsets' serial sums cost more
// where there are few channels for many rows: a head of 768 x 50277 takes 252 us (268 with a launch for the scales, and 97 with the fractions
// added in parallel), the layer of width 5120 1.00 ms (1.18, and 0.88).
//
//   quant_minmax_kernel   256 channels x one of the row splits: partial minimum and maximum
//   quant_encode_kernel   128 channels x kEncRows rows at a time: codes, layouts; in workgroups of its own the offsets.  Every workgroup
//                         makes lo, range and 1 / range of its channels from the partials, while its first rows travel (a launch between
//                         the two that did only that took 27 of the 320 us of a layer of width 2560)
// ---------------------------------------------------------------------------
constexpr int kEncRows = 64;            // rows of one LDS tile: 8 blocks of the P8 layout, 4 x 2 of the M16 layout
constexpr int kChainChannels = 8;       // channels of a workgroup that adds up fractions
constexpr int64_t kChainMaxBlocks = 1 << 20;    // such workgroups (a launch has at most 2^32 threads); of more channels each takes several groups
constexpr int kMinMaxSplits = 32;       // enough workgroups at 2560 channels (320); a partial to each 8 threads of quant_offsets

struct QuantWs {
    float2 *mm;                 // [splits][n_in]
    int64_t splits, split_rows; // of the minimum / maximum pass
    int64_t parts, part_rows;   // of the encoding pass: part_rows a multiple of kEncRows
    int64_t chain_blocks, col_blocks;   // its workgroups: the offsets' first, then col_blocks x parts
    size_t bytes;
};
static QuantWs quant_carve(int64_t n_out, int64_t n_in, void *ws) {
    QuantWs q;
    q.split_rows = round_up(ceil_div(n_out, kMinMaxSplits), 4);
    q.splits = ceil_div(n_out, q.split_rows);
    // one tile per workgroup until there are two workgroups per compute unit, then up to four
    int64_t tiles = ceil_div(n_out, kEncRows) * ceil_div(n_in, 128) / 512;
    tiles = tiles < 1 ? 1 : tiles > 4 ? 4 : tiles;
    q.part_rows = kEncRows * tiles;
    q.parts = ceil_div(n_out, q.part_rows);
    q.chain_blocks = std::min(round_up(ceil_div(n_in, kChainChannels), (int64_t)32), kChainMaxBlocks);
    q.col_blocks = ceil_div(n_in, 128);
    unsigned char *p = static_cast<unsigned char *>(ws);
    size_t at = 0;
    auto take = [&](int64_t bytes) { unsigned char *r = p + at; at += (size_t)round_up(bytes, 256); return r; };
    q.mm = reinterpret_cast<float2 *>(take(q.splits * n_in * 8));
    q.bytes = at;
    return q;
}

// Four consecutive channels of a row; channels past the end read as `pad`.
template <bool VEC>
__device__ __forceinline__ float4 weight4(const float *__restrict__ row, int64_t j, int64_t n_in, float pad) {
    if (VEC) return j < n_in ? *reinterpret_cast<const float4 *>(row + j) : make_float4(pad, pad, pad, pad);
    return make_float4(j < n_in ? row[j] : pad, j + 1 < n_in ? row[j + 1] : pad, j + 2 < n_in ? row[j + 2] : pad,
                       j + 3 < n_in ? row[j + 3] : pad);
}

template <bool VEC>
__global__ void __launch_bounds__(256)
quant_minmax_kernel(const float *__restrict__ W, int64_t n_out, int64_t n_in, QuantWs q) {
    __shared__ float4 slo[4][64], shi[4][64];
    const int cq = threadIdx.x & 63, rg = threadIdx.x >> 6;
    const int64_t j = (int64_t)blockIdx.x * 256 + 4 * cq;
    const int64_t k0 = (int64_t)blockIdx.y * q.split_rows, k1 = min(k0 + q.split_rows, n_out);
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, INFINITY), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
    if (j < n_in) {
        constexpr int U = 8;                // rows in flight per thread
        for (int64_t k = k0 + rg; k < k1; k += 4 * U) {
            float4 x[U];
#pragma unroll
            for (int u = 0; u < U; ++u)     // past the end: the last row again, which changes no extremum
                x[u] = weight4<VEC>(W + min(k + 4 * u, k1 - 1) * n_in, j, n_in, 0.f);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                lo.x = fminf(lo.x, x[u].x); lo.y = fminf(lo.y, x[u].y); lo.z = fminf(lo.z, x[u].z); lo.w = fminf(lo.w, x[u].w);
                hi.x = fmaxf(hi.x, x[u].x); hi.y = fmaxf(hi.y, x[u].y); hi.z = fmaxf(hi.z, x[u].z); hi.w = fmaxf(hi.w, x[u].w);
            }
        }
    }
    slo[rg][cq] = lo; shi[rg][cq] = hi;
    __syncthreads();
    const int64_t jj = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (jj < n_in) {
        const float *l = reinterpret_cast<const float *>(slo), *h = reinterpret_cast<const float *>(shi);
        const int t = threadIdx.x;
        q.mm[(int64_t)blockIdx.y * n_in + jj] = make_float2(fminf(fminf(l[t], l[256 + t]), fminf(l[512 + t], l[768 + t])),
                                                            fmaxf(fmaxf(h[t], h[256 + t]), fmaxf(h[512 + t], h[768 + t])));
    }
}

// A channel's extrema -> lo, range, 1 / range (0 for a constant channel: its quotients are formed all the same, and 0 * inf is no value to convert).
struct QuantScale { double lo, ran, inv; };
__device__ __forceinline__ QuantScale quant_scale(float lo, float hi) {
    const double ran = ((double)hi - (double)lo) / 255.0;              // matmul.py:31-33, as quantize_kernel
    return QuantScale{(double)lo, ran, ran > 0.0 ? 1.0 / ran : 0.0};
}

// The correctly rounded quotient d / b from the correctly rounded reciprocal of b (Markstein: a quotient within one
// unit in the last place is corrected by its remainder; the first step brings d * inv there): the bits of a division
// at a third of its instructions, with the reciprocal shared by a whole column.
__device__ __forceinline__ double quotient(double d, double b, double inv) {
    double x = d * inv;
    x = fma(fma(-b, x, d), inv, x);
    return fma(fma(-b, x, d), inv, x);
}

// 16 bytes of a packed layout.  They are stored past the caches, which leaves the float32 matrix there for the encoding pass
// (the seven matrices of a layer of width 2560, offsets added in parallel: 0.315 -> 0.288 ms).
typedef uint32_t Chunk __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int slot8(int lane) { return lane ^ ((lane >> 3) & 6); }
__device__ __forceinline__ int slot16(int lane, int half) { return lane ^ (((lane >> 3) & 6) | (half << 3)); }

// Offsets of eight channels.  The fractions of a channel are added in quantize_kernel's order, four serial float64 sums over
// the rows k = 0, 1, 2, 3 (mod 4), so that both give the same bits (an offset that differs in its last bit moves every logit of
// a model by rounding, and with it seeded texts).  Bound: not those n_out / 4 dependent additions (9 us of 10240 rows) but
// the reading: of every 128-byte line a workgroup needs 32 bytes.  Alone these workgroups take 54 us of [10240 x 2560] and 30 of [2560 x 10240], the
// encoding ones 26; 16 channels to a workgroup 127 and 74 with both (83 and 75 with 8), tiles of 192 rows 84 and 75.  Three wavefronts form
// the fractions of 96 rows at a time and leave them in LDS, kChainAhead such tiles requested ahead; the fourth adds, a lane
// per sum.  These workgroups run beside those that encode (launched first: they take longest).
constexpr int kChainRows = 96, kChainAhead = 4, kChainStride = kChainRows / 4 + 2;     // (+ 2: 16-byte aligned, fewer bank conflicts)
constexpr int kChainLds = 2 * 4 * kChainChannels * kChainStride * 8;

__device__ __forceinline__ void quant_offsets(const float *__restrict__ W, int n_out, int n_in, const QuantWs &q, int group, double *lds,
                                              float *__restrict__ range, double *__restrict__ offset) {
    constexpr int kChains = 4 * kChainChannels;
    double (*fr)[kChains][kChainStride] = reinterpret_cast<double (*)[kChains][kChainStride]>(lds);
    const int tiles = (n_out + kChainRows - 1) / kChainRows;
    // a partial to a thread; the eight of a wavefront's channel meet in the wavefront, its four in LDS
    static_assert(kMinMaxSplits == 256 / kChainChannels && kChainChannels == 8, "a partial to each thread");
    float2 (*ends)[kChainChannels] = reinterpret_cast<float2 (*)[kChainChannels]>(reinterpret_cast<char *>(lds) + kChainLds);
    {
        const int64_t jm = min(group * kChainChannels + (int)(threadIdx.x & 7), n_in - 1), split = min((int64_t)threadIdx.x >> 3, q.splits - 1);
        float2 e = q.mm[split * n_in + jm];
#pragma unroll
        for (int off = 8; off < 64; off <<= 1) { e.x = fminf(e.x, __shfl_xor(e.x, off, 64)); e.y = fmaxf(e.y, __shfl_xor(e.y, off, 64)); }
        if ((threadIdx.x & 63) < kChainChannels) ends[threadIdx.x >> 6][threadIdx.x & 63] = e;
    }
    auto scale_of = [&](int c) {
        return quant_scale(fminf(fminf(ends[0][c].x, ends[1][c].x), fminf(ends[2][c].x, ends[3][c].x)),
                           fmaxf(fmaxf(ends[0][c].y, ends[1][c].y), fmaxf(ends[2][c].y, ends[3][c].y)));
    };
    if (threadIdx.x >= 64) {
        const int pt = threadIdx.x - 64, ch = pt & 7, r = pt >> 3;          // rows r, r + 24, r + 48, r + 72 of a tile
        const int j = min(group * kChainChannels + ch, n_in - 1);
        const float *col = W + j;
        float x[kChainAhead][4];
        auto fetch = [&](float (&v)[4], int t) {
            const int k = t * kChainRows;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = col[(size_t)min(k + 24 * e + r, n_out - 1) * n_in];      // past the end: the last row again, counted as zero
        };
#pragma unroll
        for (int d = 0; d < kChainAhead; ++d) fetch(x[d], d);
        __syncthreads();                                                    // the extrema are there
        const QuantScale sc = scale_of(ch);
        const double lo = sc.lo, ran = sc.ran, inv = sc.inv;
        for (int t0 = 0; t0 < tiles; t0 += kChainAhead) {
#pragma unroll
            for (int d = 0; d < kChainAhead; ++d) {
                const int t = t0 + d;
                if (t >= tiles) break;                                      // (uniform)
                // (the four side by side, then what does not count: a branch around each would leave one chain of ten float64 operations at a time)
                double f[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const double v = quotient((double)x[d][e] - lo, ran, inv);                      // matmul.py:32-34
                    f[e] = v - trunc(v);                                                            // matmul.py:35
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) f[e] = ran > 0.0 && t * kChainRows + 24 * e + r < n_out ? f[e] : 0.0;   // (adding zero changes no bit)
                fetch(x[d], t + kChainAhead);
#pragma unroll
                for (int e = 0; e < 4; ++e) fr[t & 1][4 * ch + (r & 3)][(r >> 2) + 6 * e] = f[e];
                __syncthreads();                                            // tile t is there; tile t - 1 has been added
            }
        }
        return;
    }
    const int lane = threadIdx.x, chain = lane & (kChains - 1);
    double sum = 0.0;
    __syncthreads();                                                        // (the extrema)
    for (int t = 0; t < tiles; ++t) {
        __syncthreads();
        const double2 *v = reinterpret_cast<const double2 *>(fr[t & 1][chain]);
#pragma unroll
        for (int i = 0; i < kChainRows / 8; ++i) { const double2 p = v[i]; sum += p.x; sum += p.y; }
    }
    const int first = lane & ~3;
    const double f0 = __shfl(sum, first, 64), f1 = __shfl(sum, first + 1, 64), f2 = __shfl(sum, first + 2, 64), f3 = __shfl(sum, first + 3, 64);
    const int j = group * kChainChannels + (lane >> 2);
    if (lane < kChains && (lane & 3) == 0 && j < n_in) {
        const double fsum = (f0 + f1) + (f2 + f3);
        const QuantScale sc = scale_of(lane >> 2);
        offset[j] = sc.lo + (fsum / (double)n_out) * sc.ran;                // matmul.py:36-37
        range[j] = (float)sc.ran;                                           // matmul.py:39
    }
}

template <bool VEC>
__global__ void __launch_bounds__(256)
quant_encode_kernel(const float *__restrict__ W, int64_t n_out, int64_t n_in, QuantWs q,
                    uint8_t *__restrict__ codes, uint8_t *__restrict__ packed, uint8_t *__restrict__ packed16,
                    float *__restrict__ range, double *__restrict__ offset) {
    __shared__ __align__(16) uint32_t lds[2][8][256];
    static_assert(kChainLds + 4 * kChainChannels * (int)sizeof(float2) <= (int)sizeof(lds), "the fractions and the extrema fit");
    if (blockIdx.x < q.chain_blocks) {
        // (workgroups go to the XCDs round robin: the four groups that share a 128-byte line of a row go to the same one)
        for (int64_t b = blockIdx.x; b * kChainChannels < n_in + 32 * kChainChannels; b += q.chain_blocks) {
            const int64_t xcd = b & 7, slot = b >> 3, group = (slot >> 2) * 32 + xcd * 4 + (slot & 3);
            if (group * kChainChannels < n_in) quant_offsets(W, (int)n_out, (int)n_in, q, (int)group, reinterpret_cast<double *>(lds), range, offset);
            __syncthreads();                                        // the last rows of this group have been added
        }
        return;
    }
    uint32_t (*p8)[256] = lds[0], (*m16)[256] = lds[1];
    const int64_t item = blockIdx.x - q.chain_blocks, col_block = item % q.col_blocks, part = item / q.col_blocks;
    const int cq = threadIdx.x & 31, rg = threadIdx.x >> 5;         // four channels, every eighth row
    const int64_t j0 = col_block * 128, j = j0 + 4 * cq;
    // bytes of a thread's four channels: those there are, and those that have codes
    uint32_t there = 0, coded = 0;
    const int64_t kbeg = part * q.part_rows, kend = min(kbeg + q.part_rows, n_out);
    const int64_t n_ct8 = (n_out + 7) >> 3, n_kb8 = (n_in + 127) >> 7, n_ct16 = (n_out + 15) >> 4, n_kb16 = (n_in + 63) >> 6;
    const bool words = (n_out & 3) == 0 && (reinterpret_cast<uintptr_t>(codes) & 3) == 0;
    float4 x[8];
    auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = weight4<VEC>(W + min(k0 + rg + 8 * i, n_out - 1) * n_in, j, n_in, 0.f);
    };
    double lo[4], ran[4], inv[4];
    {
        // the partials of a channel to two threads, requested ahead of the first rows
        float2 (*ends)[128] = reinterpret_cast<float2 (*)[128]>(lds);
        QuantScale *scales = reinterpret_cast<QuantScale *>(ends + 2);
        const int c = threadIdx.x & 127, half = threadIdx.x >> 7;
        const float2 *mm = q.mm + min(j0 + c, n_in - 1);
        float2 part[kMinMaxSplits / 2];
#pragma unroll
        for (int i = 0; i < kMinMaxSplits / 2; ++i) part[i] = mm[min((int64_t)(2 * i + half), q.splits - 1) * n_in];
        fetch(kbeg);
        float2 e = part[0];
#pragma unroll
        for (int i = 1; i < kMinMaxSplits / 2; ++i) e = make_float2(fminf(e.x, part[i].x), fmaxf(e.y, part[i].y));
        ends[half][c] = e;
        __syncthreads();
        if (half == 0) scales[c] = quant_scale(fminf(e.x, ends[1][c].x), fmaxf(e.y, ends[1][c].y));
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) { const QuantScale sc = scales[4 * cq + i]; lo[i] = sc.lo; ran[i] = sc.ran; inv[i] = sc.inv; }
        __syncthreads();                                            // before the codes take their place
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (j + e < n_in) {
            there |= 0x80u << (8 * e);
            if (ran[e] > 0.0) coded |= 0xffu << (8 * e);
        } else lo[e] = ran[e] = inv[e] = 0.0;                       // (past the last channel x is 0, and its code must be one that converts)
    for (int64_t k0 = kbeg; k0 < kend; k0 += kEncRows) {
        if (k0 > kbeg) {
            fetch(k0);
            __syncthreads();                                        // the tile before has been written out
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float xe[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
            const bool row = k0 + rg + 8 * i < n_out;
            // (all four, whatever counts of them: without branches their chains of float64 operations run side by side.  A layer of width
            // 2560 291 -> 283 us, with the same in quant_offsets)
            uint32_t c4 = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double v = quotient((double)xe[e] - lo[e], ran[e], inv[e]);           // matmul.py:32-34
                c4 |= (uint32_t)(uint8_t)(int)v << (8 * e);                                 // matmul.py:21
            }
            c4 &= row ? coded : 0u;
            const uint32_t live = row ? there : 0u;
            // P8: block i of the tile, lane 8 s + column, dword m, with channel 32 m + 4 s + e of the block; M16: blocks
            // (i / 2, half of the 128 channels), lane 16 g + column, dword q, code - 128 with padding 0.  In LDS the
            // columns of a group are permuted (slot8, slot16) so that the 64 stores of a wavefront hit 64 banks.
            p8[i][slot8(8 * (cq & 7) + rg) * 4 + (cq >> 3)] = c4;
            m16[(i >> 1) * 2 + (cq >> 4)][slot16(16 * ((cq & 15) >> 2) + rg + 8 * (i & 1), cq >> 4) * 4 + (cq & 3)] = c4 ^ live;
        }
        __syncthreads();
        const int b = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
            const int i = b + h;
            if (packed) {
                const int64_t ct = (k0 >> 3) + i;
                if (ct < n_ct8)
                    __builtin_nontemporal_store(*reinterpret_cast<const Chunk *>(&p8[i][slot8(lane) * 4]), reinterpret_cast<Chunk *>(packed + (ct * n_kb8 + col_block) * 1024 + lane * 16));
            }
            if (packed16) {
                const int64_t ct = (k0 >> 4) + (i >> 1), kb = col_block * 2 + (i & 1);
                if (ct < n_ct16 && kb < n_kb16)
                    __builtin_nontemporal_store(*reinterpret_cast<const Chunk *>(&m16[i][slot16(lane, i & 1) * 4]), reinterpret_cast<Chunk *>(packed16 + (ct * n_kb16 + kb) * 1024 + lane * 16));
            }
        }
        if (codes) {
            // [n_in][n_out]: channel r of the tile, 16 lanes of four rows each (gathered from the P8 tile's bytes)
            const uint8_t *tile = reinterpret_cast<const uint8_t *>(p8);
            for (int r = threadIdx.x >> 4; r < 128; r += 16) {
                const int kq = 4 * (threadIdx.x & 15);
                uint32_t v = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = kq + e;
                    v |= (uint32_t)tile[(k >> 3) * 1024 + slot8(8 * ((r & 31) >> 2) + (k & 7)) * 16 + 4 * (r >> 5) + (r & 3)] << (8 * e);
                }
                const int64_t jr = j0 + r, k = k0 + kq;
                if (jr < n_in) {
                    uint8_t *o = codes + jr * n_out + k;
                    if (words && k + 4 <= n_out) *reinterpret_cast<uint32_t *>(o) = v;
                    else
                        for (int e = 0; e < 4; ++e)
                            if (k + e < n_out) o[e] = (uint8_t)(v >> (8 * e));
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// pack / unpack: one thread per 16-byte lane chunk of a block.
// ---------------------------------------------------------------------------
template <bool PACK>
__global__ void __launch_bounds__(256)
pack_kernel(uint8_t *__restrict__ codes, int64_t stride, int64_t n_in, int64_t n_out,
            uint8_t *__restrict__ packed, int64_t n_kb, int64_t n_chunks) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_chunks) return;
    const int lane = (int)(g & 63);
    const int64_t blk = g >> 6;
    const int64_t kb = blk % n_kb, ct = blk / n_kb;
    const int s = lane >> 3, c = lane & 7;
    const int64_t col = ct * kTileCols + c;
    uint8_t *p = packed + g * 16;
    if (PACK) {
        uint32_t d[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            uint32_t v = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t row = kb * kBlockRows + 32 * m + 4 * s + e;
                const uint32_t b = (row < n_in && col < n_out) ? codes[row * stride + col] : 0u;
                v |= b << (8 * e);
            }
            d[m] = v;
        }
        *reinterpret_cast<uint4 *>(p) = make_uint4(d[0], d[1], d[2], d[3]);
    } else {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t row = kb * kBlockRows + 32 * m + 4 * s + e;
                if (row < n_in && col < n_out) codes[row * stride + col] = (uint8_t)(d[m] >> (8 * e));
            }
    }
}

__global__ void __launch_bounds__(256)
dequant_packed_kernel(const uint8_t *__restrict__ packed, const float *__restrict__ range,
                      const double *__restrict__ offset, int64_t n_in, int64_t n_out,
                      int64_t n_kb, float *__restrict__ dq) {
    // one thread per output element, consecutive threads along k
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_in * n_out) return;
    const int64_t j = g / n_out, k = g % n_out;
    const int64_t ct = k / kTileCols, kb = j / kBlockRows;
    const int c = (int)(k % kTileCols), r = (int)(j % kBlockRows);
    const int m = r / 32, s = (r % 32) / 4, e = r % 4;
    const uint8_t code = packed[(ct * n_kb + kb) * kBlockBytes + 16 * (8 * s + c) + 4 * m + e];
    dq[g] = (float)((double)code * (double)range[j] + offset[j]);
}

// ---------------------------------------------------------------------------
// "M16" layout for the int8 matrix-core decode kernel: 1 KiB blocks of 16
// output columns x 64 input rows, ordered [ceil(n_out/16)][ceil(n_in/64)].
// Lane l = 16*g + n of a wavefront owns bytes 16*l .. 16*l+15 of the block:
// rows 64*kb + 16*g + (0..15) of column 16*ct + n, stored as code - 128
// (two's complement), i.e. exactly the B operand of v_mfma_i32_16x16x64_i8.
// Padding is stored as 0 (it only ever meets zero activation digits).
// ---------------------------------------------------------------------------
template <bool PACK>
__global__ void __launch_bounds__(256)
pack_m16_kernel(uint8_t *__restrict__ codes, int64_t stride, int64_t n_in, int64_t n_out,
                uint8_t *__restrict__ packed, int64_t n_kb, int64_t n_chunks) {
    const int64_t gidx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gidx >= n_chunks) return;
    const int lane = (int)(gidx & 63);
    const int64_t blk = gidx >> 6;
    const int64_t kb = blk % n_kb, ct = blk / n_kb;
    const int g = lane >> 4, n = lane & 15;
    const int64_t col = ct * 16 + n;
    uint8_t *p = packed + gidx * 16;
    if (PACK) {
        uint32_t d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t v = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t row = kb * 64 + 16 * g + 4 * q + e;
                const uint32_t b = (row < n_in && col < n_out) ? (uint32_t)(codes[row * stride + col] ^ 0x80u) : 0u;
                v |= b << (8 * e);
            }
            d[q] = v;
        }
        *reinterpret_cast<uint4 *>(p) = make_uint4(d[0], d[1], d[2], d[3]);
    } else {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t row = kb * 64 + 16 * g + 4 * q + e;
                if (row < n_in && col < n_out) codes[row * stride + col] = (uint8_t)((d[q] >> (8 * e)) ^ 0x80u);
            }
    }
}

}  // namespace rwkv

using namespace rwkv;

extern "C" {

int rwkv_version(void) { return 100; }
const char *rwkv_last_error(void) { return rwkv::g_err; }

int rwkv_quantize_u8(rwkv_stream_t stream, const float *weight, int64_t n_out, int64_t n_in,
                     uint8_t *codes, float *range, double *offset) {
    RWKV_CHECK_ARG(weight && codes && range && offset, "rwkv_quantize_u8: null pointer");
    RWKV_CHECK_ARG(n_out > 0 && n_in > 0, "rwkv_quantize_u8: sizes must be positive");
    RWKV_CHECK_ALIGN(weight, 4);
    RWKV_CHECK_ALIGN(range, 4);
    RWKV_CHECK_ALIGN(offset, 8);
    hipLaunchKernelGGL(quantize_kernel, dim3((unsigned)ceil_div(n_in, 64)), dim3(256), 0,
                       (hipStream_t)stream, weight, n_out, n_in, codes, range, offset);
    RWKV_CHECK_LAUNCH("quantize_kernel");
    return RWKV_OK;
}

size_t rwkv_quantize_workspace_bytes(int64_t n_out, int64_t n_in) {
    if (n_out <= 0 || n_in <= 0) return 0;
    return quant_carve(n_out, n_in, nullptr).bytes;
}

int rwkv_quantize_layouts(rwkv_stream_t stream, const float *weight, int64_t n_out, int64_t n_in, uint8_t *codes,
                          uint8_t *packed, uint8_t *packed16, float *range, double *offset, void *workspace,
                          size_t workspace_bytes) {
    RWKV_CHECK_ARG(weight && range && offset && workspace, "rwkv_quantize_layouts: null pointer");
    RWKV_CHECK_ARG(codes || packed || packed16, "rwkv_quantize_layouts: no output layout");
    RWKV_CHECK_ARG(n_out > 0 && n_in > 0 && n_out < (1ll << 30) && n_in < (1ll << 30), "rwkv_quantize_layouts: bad sizes");
    RWKV_CHECK_ALIGN(weight, 4);
    RWKV_CHECK_ALIGN(range, 4);
    RWKV_CHECK_ALIGN(offset, 8);
    RWKV_CHECK_ALIGN(packed, 16);
    RWKV_CHECK_ALIGN(packed16, 16);
    RWKV_CHECK_ALIGN(workspace, 8);
    const QuantWs q = quant_carve(n_out, n_in, workspace);
    if (workspace_bytes < q.bytes)
        return set_error(RWKV_ERR_WORKSPACE, "rwkv_quantize_layouts: workspace of %zu bytes needed, %zu given", q.bytes, workspace_bytes);
    const hipStream_t st = (hipStream_t)stream;
    const bool vec = n_in % 4 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0;
    const int64_t blocks = q.chain_blocks + q.col_blocks * q.parts;
    if (blocks >= (1ll << 24))
        return set_error(RWKV_ERR_SIZE, "rwkv_quantize_layouts: %lld x %lld is more than one launch covers", (long long)n_out, (long long)n_in);
    const dim3 mg((unsigned)ceil_div(n_in, 256), (unsigned)q.splits), eg((unsigned)blocks);
    if (vec) hipLaunchKernelGGL(quant_minmax_kernel<true>, mg, dim3(256), 0, st, weight, n_out, n_in, q);
    else hipLaunchKernelGGL(quant_minmax_kernel<false>, mg, dim3(256), 0, st, weight, n_out, n_in, q);
    if (vec) hipLaunchKernelGGL(quant_encode_kernel<true>, eg, dim3(256), 0, st, weight, n_out, n_in, q, codes, packed, packed16, range, offset);
    else hipLaunchKernelGGL(quant_encode_kernel<false>, eg, dim3(256), 0, st, weight, n_out, n_in, q, codes, packed, packed16, range, offset);
    RWKV_CHECK_LAUNCH("quant_encode_kernel");
    return RWKV_OK;
}

size_t rwkv_packed_bytes(int64_t n_in, int64_t n_out) {
    if (n_in <= 0 || n_out <= 0) return 0;
    return (size_t)(ceil_div(n_out, kTileCols) * ceil_div(n_in, kBlockRows) * kBlockBytes);
}

int rwkv_pack_u8(rwkv_stream_t stream, const uint8_t *codes, int64_t codes_stride,
                 int64_t n_in, int64_t n_out, uint8_t *packed) {
    RWKV_CHECK_ARG(codes && packed, "rwkv_pack_u8: null pointer");
    RWKV_CHECK_ARG(n_in > 0 && n_out > 0 && codes_stride >= n_out, "rwkv_pack_u8: bad sizes");
    RWKV_CHECK_ALIGN(packed, 16);
    const int64_t n_kb = ceil_div(n_in, kBlockRows);
    const int64_t n_chunks = ceil_div(n_out, kTileCols) * n_kb * 64;
    hipLaunchKernelGGL(pack_kernel<true>, dim3((unsigned)ceil_div(n_chunks, 256)), dim3(256), 0,
                       (hipStream_t)stream, const_cast<uint8_t *>(codes), codes_stride, n_in, n_out,
                       packed, n_kb, n_chunks);
    RWKV_CHECK_LAUNCH("pack_kernel");
    return RWKV_OK;
}

int rwkv_unpack_u8(rwkv_stream_t stream, const uint8_t *packed, int64_t n_in, int64_t n_out,
                   uint8_t *codes, int64_t codes_stride) {
    RWKV_CHECK_ARG(codes && packed, "rwkv_unpack_u8: null pointer");
    RWKV_CHECK_ARG(n_in > 0 && n_out > 0 && codes_stride >= n_out, "rwkv_unpack_u8: bad sizes");
    RWKV_CHECK_ALIGN(packed, 16);
    const int64_t n_kb = ceil_div(n_in, kBlockRows);
    const int64_t n_chunks = ceil_div(n_out, kTileCols) * n_kb * 64;
    hipLaunchKernelGGL(pack_kernel<false>, dim3((unsigned)ceil_div(n_chunks, 256)), dim3(256), 0,
                       (hipStream_t)stream, codes, codes_stride, n_in, n_out,
                       const_cast<uint8_t *>(packed), n_kb, n_chunks);
    RWKV_CHECK_LAUNCH("unpack_kernel");
    return RWKV_OK;
}

int rwkv_dequant_packed(rwkv_stream_t stream, const uint8_t *packed, const float *range,
                        const double *offset, int64_t n_in, int64_t n_out, float *dq) {
    RWKV_CHECK_ARG(packed && range && offset && dq, "rwkv_dequant_packed: null pointer");
    RWKV_CHECK_ARG(n_in > 0 && n_out > 0, "rwkv_dequant_packed: bad sizes");
    const int64_t n = n_in * n_out;
    hipLaunchKernelGGL(dequant_packed_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, packed, range, offset, n_in, n_out,
                       ceil_div(n_in, kBlockRows), dq);
    RWKV_CHECK_LAUNCH("dequant_packed_kernel");
    return RWKV_OK;
}

size_t rwkv_packed_m16_bytes(int64_t n_in, int64_t n_out) {
    if (n_in <= 0 || n_out <= 0) return 0;
    return (size_t)(ceil_div(n_out, 16) * ceil_div(n_in, 64) * 1024);
}

int rwkv_pack_m16(rwkv_stream_t stream, const uint8_t *codes, int64_t codes_stride,
                  int64_t n_in, int64_t n_out, uint8_t *packed) {
    RWKV_CHECK_ARG(codes && packed, "rwkv_pack_m16: null pointer");
    RWKV_CHECK_ARG(n_in > 0 && n_out > 0 && codes_stride >= n_out, "rwkv_pack_m16: bad sizes");
    RWKV_CHECK_ALIGN(packed, 16);
    const int64_t n_kb = ceil_div(n_in, 64);
    const int64_t n_chunks = ceil_div(n_out, 16) * n_kb * 64;
    hipLaunchKernelGGL(pack_m16_kernel<true>, dim3((unsigned)ceil_div(n_chunks, 256)), dim3(256), 0,
                       (hipStream_t)stream, const_cast<uint8_t *>(codes), codes_stride, n_in, n_out,
                       packed, n_kb, n_chunks);
    RWKV_CHECK_LAUNCH("pack_m16_kernel");
    return RWKV_OK;
}

int rwkv_unpack_m16(rwkv_stream_t stream, const uint8_t *packed, int64_t n_in, int64_t n_out,
                    uint8_t *codes, int64_t codes_stride) {
    RWKV_CHECK_ARG(codes && packed, "rwkv_unpack_m16: null pointer");
    RWKV_CHECK_ARG(n_in > 0 && n_out > 0 && codes_stride >= n_out, "rwkv_unpack_m16: bad sizes");
    RWKV_CHECK_ALIGN(packed, 16);
    const int64_t n_kb = ceil_div(n_in, 64);
    const int64_t n_chunks = ceil_div(n_out, 16) * n_kb * 64;
    hipLaunchKernelGGL(pack_m16_kernel<false>, dim3((unsigned)ceil_div(n_chunks, 256)), dim3(256), 0,
                       (hipStream_t)stream, codes, codes_stride, n_in, n_out,
                       const_cast<uint8_t *>(packed), n_kb, n_chunks);
    RWKV_CHECK_LAUNCH("unpack_m16_kernel");
    return RWKV_OK;
}

}  // extern "C"
