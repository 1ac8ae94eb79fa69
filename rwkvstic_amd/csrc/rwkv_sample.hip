// Next-token choice on the device: the reference's `typical` sampler (agnostic/samplers/typical.py:1-17) and
// argmax, with the logit adjustment and the stop-token test of RWKVMaster.forward (rwkvMaster.py:34-54), so
// that a generation loop needs no host round trip per token.
//
// typical(logits, temp, tau):  p = softmax(float32(logits));  s = -log p;  H = sum p s (entropy);
// d = |s - H|;  in ascending order of d, the tokens before the first one whose running mass reaches tau, and
// that one, are kept (everything with d greater than its d is zeroed);  kept p^(1/temp) is sampled.
// The order itself is never needed: the cut is the smallest d* among the tokens with mass{d <= d*} >= tau.  It is found by the
// bit pattern of d (non-negative floats order like their bits): the masses by upper half of the bits tell which one holds the
// cut, one pass over all tokens checks that and lists the tokens of that half, and the lower half is settled on the list;
// where the masses do not tell, a radix search of two bits a pass.  One workgroup of 1024 threads; thread t owns the tokens
// t, t + 1024, ...  The probabilities stay in registers; of the keys the first kSKeysLds per thread live in LDS and the
// rest in registers: both arrays in registers would not fit the 128 registers a wave of a 1024-thread workgroup has.
//
// Bound: what one compute unit loads and its vector instructions (three thresholds over 50277 tokens: 3 us), so passes are
// what is saved; more workgroups would have to exchange every sum, two of three microseconds each time.  50277 tokens after a
// token step, before / now: logits in 15.4 / 5.4 us, probabilities and entropy 8 / 4, cut to 16 bits and list 23 / 10, the
// rest of the cut 3.8 / 1.9, draw 5.6 / 3.3; 54.5 / 25 us.  tau 0.9999999, where the masses do not tell: 42.5 / 43.5.
#include "rwkv_common.h"
#include "rwkv_sample.h"

#include <mutex>

namespace rwkv {

namespace {

constexpr int kST = 1024;            // threads
constexpr int kSMaxPer = 52;         // tokens per thread: vocabularies up to 53248
// Full passes settle the key's bits down to this one before the first attempt to list the undecided tokens.  It is part of
// the results: the mass below a threshold is rounded differently when it is the sum of the listed tokens on top of what
// lies below them, and a cut that moves by one token moves every draw of a seed.  (16, 18, 20, searched pass by pass: 60, 58 and 70 us at 50277
// tokens, where the list overflows at 20; 18 changed 8 of 24000 draws.)
constexpr int kSFirstBit = 16;
constexpr int kSList = 2048;         // most tokens that may share the upper half of the cut's key and still be listed
constexpr int kSBins = 2 * kSList;   // masses of keys by their upper half, from 2^-28 to 16
constexpr unsigned kSBin0 = 0x3180;
constexpr float kSMass = 2147483648.0f;      // their unit: whole numbers, as a float addition in LDS takes about as many clocks as there are lanes, times three
constexpr int kSKeysLds = 32;        // keys per thread kept in LDS ([k][thread]: conflict-free), 128 KiB

// Sum over a wavefront: the butterfly of lanes 32, 16, 8, 4, 2, 1 apart in this order (it reaches the cut, and with it the
// draws of a seed), by permlane swaps and DPP rotations in place of six dependent trips through the LDS crossbar.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false)); }
__device__ __forceinline__ float swap32(float v, bool hi) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
    return __int_as_float(hi ? r[1] : r[0]);
}
__device__ __forceinline__ float swap16(float v, bool hi) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    return __int_as_float(hi ? r[1] : r[0]);
}
__device__ __forceinline__ float wave_sum_f(float v) {
    v = swap32(v, false) + swap32(v, true);
    v = swap16(v, false) + swap16(v, true);
    v += dpp<0x128>(v);                               // row_ror:8, then row_ror:4: what lanes 8 apart have added repeats with 8
    v += dpp<0x124>(v);
    v += dpp<0x4E>(v);                                // quad_perm: lanes 2 apart, then 1
    return v + dpp<0xB1>(v);
}
__device__ __forceinline__ float wave_max_f(float v) {
    v = fmaxf(swap32(v, false), swap32(v, true));
    v = fmaxf(swap16(v, false), swap16(v, true));
    v = fmaxf(v, dpp<0x128>(v));
    v = fmaxf(v, dpp<0x124>(v));
    v = fmaxf(v, dpp<0x4E>(v));
    return fmaxf(v, dpp<0xB1>(v));
}
__device__ __forceinline__ float block_sum_f(float v, float *scr) {
    v = wave_sum_f(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scr[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kST / 64; ++w) s += scr[w];
    return s;
}
// two sums at once; scr: 2 * kST / 64 floats
__device__ __forceinline__ void block_sum2_f(float &a, float &b, float *scr) {
    a = wave_sum_f(a); b = wave_sum_f(b);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) { scr[threadIdx.x >> 6] = a; scr[kST / 64 + (threadIdx.x >> 6)] = b; }
    __syncthreads();
    a = 0.f; b = 0.f;
#pragma unroll
    for (int w = 0; w < kST / 64; ++w) { a += scr[w]; b += scr[kST / 64 + w]; }
}
__device__ __forceinline__ float block_max_f(float v, float *scr) {
    v = wave_max_f(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scr[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = -INFINITY;
#pragma unroll
    for (int w = 0; w < kST / 64; ++w) s = fmaxf(s, scr[w]);
    return s;
}

// splitmix64 of (seed, counter) -> uniform in [0, 1) with 24 bits
__device__ __forceinline__ float uniform01(unsigned long long seed, unsigned long long counter) {
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (counter + 1ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (float)(z >> 40) * (1.0f / 16777216.0f);
}

template <int PER>
__global__ void __launch_bounds__(kST)
sample_kernel(SampleArgs a) {
    constexpr int KL = PER < kSKeysLds ? PER : kSKeysLds, KR = PER - KL > 0 ? PER - KL : 1;
    extern __shared__ unsigned key_lds[];            // [KL][kST]
    __shared__ float scr[4 * (kST / 64)];
    __shared__ float wsum[kST / 64];
    __shared__ int s_tok, s_cnt;
    __shared__ unsigned s_guess;
    __shared__ unsigned char s_below[2][kST / 64];
    __shared__ __align__(16) unsigned bins[kSBins];  // the masses by bin, then the list: its keys' bits, then its probabilities
    const int stopped = a.stop_flag ? *a.stop_flag : 0;
    const int V = a.V, tid = threadIdx.x;
    float p[PER];                                    // first the float32 logits, then the probabilities
    float mx = -INFINITY;
    int token = 0;
    if (a.greedy) {
        if (stopped) return;                         // a stop token ended the sequence: the rest of the loop is skipped
        if (a.end_adj != 0.0 && tid == 0) a.logits[0] += a.end_adj;       // rwkvMaster.py:37, kept in the returned logits (read again by this thread alone)
        // first maximum (float64 comparison on the stored logits, as the greedy loop does)
        double best = -INFINITY; int bi = 0x7fffffff;
#pragma unroll 13
        for (int k = 0; k < PER; ++k) {
            const int i = tid + kST * k;
            if (i < V) { const double x = a.logits[i]; if (x > best) { best = x; bi = i; } }      // i grows with k: the first of equals stays
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const double ob = __shfl_xor(best, off, 64); const int oi = __shfl_xor(bi, off, 64);
            if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
        }
        __shared__ double sv[kST / 64]; __shared__ int si[kST / 64];
        if ((tid & 63) == 0) { sv[tid >> 6] = best; si[tid >> 6] = bi; }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < kST / 64; ++w) if (sv[w] > best || (sv[w] == best && si[w] < bi)) { best = sv[w]; bi = si[w]; }
            s_tok = bi == 0x7fffffff ? 0 : bi;
        }
        __syncthreads();
        token = s_tok;
    } else {
        if constexpr (PER > KL) {
            // Two tokens a load: a compute unit takes in 8-byte loads at 45 bytes a nanosecond and 16-byte loads at 66 or more,
            // with the next six loads under way (400 KB: 15.4 us in four batches of thirteen 8-byte loads, 9.8 us with the
            // next batch under way, 6.2 us so).  A wavefront loads exactly its own tokens, two slots k at a time, and hands
            // them round through the LDS where its keys will be; the slots whose keys stay in registers go first.
            typedef double pair8 __attribute__((ext_vector_type(2), aligned(8)));
            constexpr int LB = 6, NP = PER / 2, NR = (PER - KL) / 2, NB = (NP + LB - 1) / LB;
            static_assert(PER % 2 == 0 && KL % 2 == 0 && PER - KL <= KL, "pairs of slots");
            const int half = (tid >> 5) & 1, col = (tid & ~63) + 2 * (tid & 31);
            pair8 x[2][LB];
            auto slot = [](int s) { return s < NR ? KL + 2 * s : 2 * (s - NR); };        // the first slot of the s-th load
            auto load = [&](int b) {
#pragma unroll
                for (int j = 0; j < LB; ++j)
                    if (b * LB + j < NP)                 // (past the end: the last pair, of which no more than its second is used; V > 8192 here)
                        x[b & 1][j] = *(const pair8 *)(a.logits + min(col + kST * (slot(b * LB + j) + half), V - 2));
            };
            load(0);
            __builtin_amdgcn_sched_barrier(0);
            if (stopped) return;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b + 1 < NB) load(b + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < LB; ++j) {
                    const int s = b * LB + j;
                    if (s >= NP) continue;
                    const int i = col + kST * (slot(s) + half);
                    pair8 v = x[b & 1][j];
                    if (slot(s) == 0 && a.end_adj != 0.0 && tid == 0) { v.x += a.end_adj; a.logits[0] = v.x; }       // rwkvMaster.py:37, kept in the returned logits
                    const float x1 = i + 1 < V ? (float)v.y : -INFINITY;
                    const float x0 = i + 1 < V ? (float)v.x : i < V ? (float)v.y : -INFINITY;
                    mx = fmaxf(mx, fmaxf(x0, x1));
                    unsigned *at = key_lds + (s < NR ? 2 * s + half : slot(s) + half) * kST + col;
                    at[0] = __float_as_uint(x0);
                    at[1] = __float_as_uint(x1);
                    if (s == NR - 1) {
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
                        for (int k = KL; k < PER; ++k) p[k] = __uint_as_float(key_lds[(k - KL) * kST + tid]);
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int k = 0; k < KL; ++k) p[k] = __uint_as_float(key_lds[k * kST + tid]);
        } else {
            if (stopped) return;
            if (a.end_adj != 0.0 && tid == 0) a.logits[0] += a.end_adj;
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int i = tid + kST * k;
                p[k] = i < V ? (float)a.logits[i] : -INFINITY;
                mx = fmaxf(mx, p[k]);
            }
        }
        if (tid == 0) { s_cnt = 0; s_guess = 0; }
        *(uint4 *)(bins + 4 * tid) = make_uint4(0, 0, 0, 0);        // (barriers before its first use: those of the maximum)
        static_assert(kSBins == 4 * kST, "four bins a thread");
        mx = block_max_f(mx, scr);
        // softmax in float32 (typical.py:5); the hardware exponential (about one ulp) is enough here: only a tie at
        // the edge of the kept set could fall the other way.  p[k] holds exp(t), t = logit - max; t itself waits where its
        // search key will be (both in registers would not fit).
        unsigned kreg[KR];
#define RWKV_KEY(k) ((k) < KL ? key_lds[(k) * kST + tid] : kreg[(k) - KL < KR ? (k) - KL : 0])
#define RWKV_SET_KEY(k, v) { const unsigned v_ = (v); if ((k) < KL) key_lds[(k) * kST + tid] = v_; else kreg[(k) - KL < KR ? (k) - KL : 0] = v_; }   /* (each thread reads back only its own) */
        float z = 0.f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const float t = p[k] - mx;
            RWKV_SET_KEY(k, __float_as_uint(t))
            p[k] = __expf(t);                            // exp(-inf) = 0 past the end
            z += p[k];
        }
        z = block_sum_f(z, scr);
        const float rz = 1.0f / z, logz = logf(z);
        // surprise s = -log p = log z - t (no logarithm per token), entropy (nansum: terms with p == 0 are skipped)
        float h = 0.f, tt = 0.f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            p[k] *= rz;
            const float t = fmaxf(__uint_as_float(RWKV_KEY(k)), -1e18f);           // (p == 0 adds 0 also where t is -inf)
            h += (logz - t) * p[k];
            tt += t * t * p[k];
        }
        block_sum2_f(h, tt, scr);
        // The cut lies no further from the entropy than `far`: no more than variance / d^2 of the mass lies further than d, and the
        // tokens less likely than (1 - tau) / V have no more than 1 - tau together.  (A percent more for rounding; where that
        // should not do, the check below finds out.  Where 1 - tau is of the size of the sums' rounding there is no guess.)
        const float rest = 1.0f - a.tau;
        const float far = rest < 1e-5f ? -1.f : 1.01f * fminf(sqrtf(fmaxf(tt - (logz - h) * (logz - h), 0.f) / rest), fmaxf(logf((float)V / rest) - h, h));
        const int reach_i = min(__float_as_int(far) - (int)(kSBin0 << 16), (kSBins << 16) - 1);
        const unsigned reach = (unsigned)max(reach_i, 0);        // keys from the first bin on; (none: keys of exactly 2^-28)
        // Distance from the entropy as the search key, and the mass of each upper half of a key: it tells where the cut lies but
        // for the rounding of sums.  (What is further than the cut can be stays out: the unlikely tokens of a peaked
        // distribution share few bins, and additions to one address take a clock each.)
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const unsigned key = p[k] > 0.f ? __float_as_uint(fabsf(logz - __uint_as_float(RWKV_KEY(k)) - h)) : 0x7f800000u;      // p == 0: d = inf
            RWKV_SET_KEY(k, key)
            asm volatile("" : "+v"(p[k]));
            const unsigned off = key - (kSBin0 << 16);
            if (off <= reach) atomicAdd(&bins[off >> 16], (unsigned)__builtin_fmaf(p[k], kSMass, 0.5f));
        }
        // Radix search, most significant bits first, two bits per round: the largest prefix P with mass{key < P} < tau.
        // `below` = mass{key < prefix}.
        // A prefix with no mass at all below it is always taken: typical.py:13-14 keeps the token at position
        // #(cumulative < tau) of the sorted distances, so the token nearest the entropy stays even with tau = 0.
        unsigned prefix = 0;
        float below = 0.f;
#define RWKV_BELOW(t) ((t) < a.tau || (t) <= 0.f)
#define RWKV_FULL_ROUND(shift)                                                                                           \
        {                                                                                                                \
            float m1 = 0.f, m2 = 0.f, m3 = 0.f;                                                                          \
            const unsigned c1 = prefix | (1u << (shift)), c2 = prefix | (2u << (shift)), c3 = prefix | (3u << (shift));  \
            _Pragma("unroll") for (int k = 0; k < PER; ++k) {                                                            \
                const unsigned key = RWKV_KEY(k);                                                                        \
                m1 += key < c1 ? p[k] : 0.f;                                                                             \
                m2 += key < c2 ? p[k] : 0.f;                                                                             \
                m3 += key < c3 ? p[k] : 0.f;                                                                             \
            }                                                                                                            \
            m1 = wave_sum_f(m1); m2 = wave_sum_f(m2); m3 = wave_sum_f(m3); /* three sums with one pair of barriers */     \
            __syncthreads();                                                                                             \
            if ((tid & 63) == 0) { scr[tid >> 6] = m1; scr[kST / 64 + (tid >> 6)] = m2; scr[2 * (kST / 64) + (tid >> 6)] = m3; } \
            __syncthreads();                                                                                             \
            float t1 = 0.f, t2 = 0.f, t3 = 0.f;                                                                          \
            _Pragma("unroll") for (int w = 0; w < kST / 64; ++w) { t1 += scr[w]; t2 += scr[kST / 64 + w]; t3 += scr[2 * (kST / 64) + w]; } \
            if (RWKV_BELOW(t3)) { prefix = c3; below = t3; } else if (RWKV_BELOW(t2)) { prefix = c2; below = t2; }       \
            else if (RWKV_BELOW(t1)) { prefix = c1; below = t1; }                                                        \
        }
        // The upper half at once: the bin that the running mass crosses tau in is taken to hold the cut, and one pass that sums
        // the masses below its two ends, as a round of the search would have, says whether it does.  (The sums grow with the
        // threshold, rounding included: the largest prefix with mass{key < P} < tau does not depend on the thresholds tried.)
        // Else, where tau is nearly everything, or nearly one token or equal tokens have the mass: round by round.
        int shift = kSFirstBit - 2;
        bool listed = false, found = false;
        {
            __syncthreads();
            const uint4 sums = *(const uint4 *)(bins + 4 * tid);
            const float4 v = make_float4((float)sums.x * (1.f / kSMass), (float)sums.y * (1.f / kSMass), (float)sums.z * (1.f / kSMass), (float)sums.w * (1.f / kSMass));
            float incl = v.x + v.y + v.z + v.w;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) { const float o = __shfl_up(incl, off, 64); if ((tid & 63) >= off) incl += o; }
            const float prev = __shfl_up(incl, 1, 64);
            if ((tid & 63) == 63) scr[tid >> 6] = incl;
            __syncthreads();
            float base = 0.f;
            for (int w = 0; w < (tid >> 6); ++w) base += scr[w];
            const float from = base + ((tid & 63) ? prev : 0.f), to = base + incl;
            if (RWKV_BELOW(from) && !RWKV_BELOW(to)) {
                const float e1 = from + v.x, e2 = e1 + v.y, e3 = e2 + v.z;
                const unsigned bin = 4 * tid + (RWKV_BELOW(e3) ? 3 : RWKV_BELOW(e2) ? 2 : RWKV_BELOW(e1) ? 1 : 0);
                s_guess = (kSBin0 + bin) << 16;
            }
            __syncthreads();                           // the bins have been read: the list may take their place
            const unsigned c1 = s_guess, c2 = c1 + (1u << kSFirstBit);
            if (c1) {                                  // (uniform)
                float m1 = 0.f, m2 = 0.f;
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const unsigned key = RWKV_KEY(k);
                    m1 += key < c1 ? p[k] : 0.f;
                    m2 += key < c2 ? p[k] : 0.f;
                    asm volatile("" : "+v"(m1), "+v"(m2));        // (summed here: else the masks of 52 comparisons wait in spilled registers)
                    if (key < c2 && !(key < c1)) {
                        const int at = atomicAdd(&s_cnt, 1);
                        if (at < kSList) { bins[at] = key; bins[kSList + at] = __float_as_uint(p[k]); }
                    }
                }
                m1 = wave_sum_f(m1); m2 = wave_sum_f(m2);
                if ((tid & 63) == 0) { scr[kST / 64 + (tid >> 6)] = m1; scr[2 * (kST / 64) + (tid >> 6)] = m2; }
                __syncthreads();
                float t1 = 0.f, t2 = 0.f;
#pragma unroll
                for (int w = 0; w < kST / 64; ++w) { t1 += scr[kST / 64 + w]; t2 += scr[2 * (kST / 64) + w]; }
                found = RWKV_BELOW(t1) && !RWKV_BELOW(t2);
                if (found) { prefix = c1; below = t1; listed = s_cnt <= kSList; }
            }
        }
        if (!found) {
            constexpr unsigned c1 = 0x40000000u;       // the top two bits: 01 from 2 on, and no key has the highest one
            float m = 0.f, q = 0.f;
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                m += RWKV_KEY(k) < c1 ? p[k] : 0.f;
                q += p[k];
            }
            block_sum2_f(m, q, scr);
            if (RWKV_BELOW(q)) { prefix = 0xffffffffu; shift = -2; }      // all of it stays below tau: every token is kept
            else {
                if (RWKV_BELOW(m)) { prefix = c1; below = m; }
                for (int at = 28; at >= kSFirstBit; at -= 2) RWKV_FULL_ROUND(at)
            }
        }
        // Only the tokens that share the settled bits with the cut can still decide the rest.  As soon as they fit a list of
        // kSList entries it is searched without passes over all tokens.
        while (!listed && shift >= 0) {                // (uniform) shift = next undecided bit pair
            __syncthreads();                           // everybody has read the count before it is cleared again
            if (tid == 0) s_cnt = 0;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const unsigned key = RWKV_KEY(k);
                if (((key ^ prefix) >> (shift + 2)) == 0u) {
                    const int at = atomicAdd(&s_cnt, 1);
                    if (at < kSList) { bins[at] = key; bins[kSList + at] = __float_as_uint(p[k]); }
                }
            }
            __syncthreads();
            if (s_cnt <= kSList) { listed = true; break; }
            RWKV_FULL_ROUND(shift)
            shift -= 2;
            if (shift >= 0) { RWKV_FULL_ROUND(shift) shift -= 2; }
        }
        if (listed) {
            // four bits a round, a threshold to a wavefront
            const int n_list = s_cnt, wave = tid >> 6;
            static_assert(kST / 64 == 16, "sixteen thresholds");
            for (int at = shift - 2; at >= 0; at -= 4) {
                const unsigned c = prefix | ((unsigned)wave << at);
                float m = 0.f;
                for (int i = tid & 63; i < n_list; i += 64) m += bins[i] < c ? __uint_as_float(bins[kSList + i]) : 0.f;
                const float t = below + wave_sum_f(m);
                unsigned char *flags = s_below[(at >> 2) & 1];
                if ((tid & 63) == 0) flags[wave] = wave == 0 || RWKV_BELOW(t);
                __syncthreads();
                const unsigned long long mask = __ballot(flags[tid & 15] != 0);
                prefix |= (unsigned)(__popcll(mask & 0xffffull) - 1) << at;
            }
        }
#undef RWKV_FULL_ROUND
#undef RWKV_BELOW
        // prefix = d* as bits (mass{key < d*} < tau <= mass{key <= d*}); if the whole mass stays below tau every
        // finite key passes.  Kept tokens, temperature, total.
        const float inv_t = a.temp != 1.0f ? 1.0f / a.temp : 1.0f;
        float q = 0.f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            p[k] = RWKV_KEY(k) <= prefix ? p[k] : 0.f;
        }
        if (a.temp != 1.0f) {        // (as one block: skipped token by token it is 50 KB of code to jump through)
#pragma unroll
            for (int k = 0; k < PER; ++k)
                if (p[k] > 0.f) p[k] = __powf(p[k], inv_t);           // hardware log2 / exp2: a few ulp, immaterial for a sampling weight
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) q += p[k];
        // inverse CDF in the order (thread, k): scan of the per-thread sums, then a walk inside one thread's tokens
        float own = q;
        float incl = own;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) { const float o = __shfl_up(incl, off, 64); if ((tid & 63) >= off) incl += o; }
        __syncthreads();
        if ((tid & 63) == 63) wsum[tid >> 6] = incl;
        __syncthreads();
        float before = 0.f, total = 0.f;
#pragma unroll
        for (int w = 0; w < kST / 64; ++w) { if (w < (tid >> 6)) before += wsum[w]; total += wsum[w]; }
        const float lo = before + incl - own, hi = before + incl;
        const float target = uniform01(a.seed, a.counter) * total;
        if (tid == 0) s_tok = -1;
        __syncthreads();
        if (own > 0.f && target >= lo && target < hi) {
            // (a token that is not kept adds nothing, and is never the first one that the sum passes the target at)
            float acc = lo;
            int n = 0, last = 0;
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                acc += p[k];
                n += target >= acc ? 1 : 0;
                last = p[k] > 0.f ? k : last;
            }
            const int pick = tid + kST * (n < PER ? n : last);        // (rounding at the upper edge: the thread's last kept token)
            atomicMax(&s_tok, pick);
        }
        __syncthreads();
        if (s_tok < 0) {
            // The target fell on a boundary nobody claimed, or every kept weight underflowed under the temperature
            // (total 0): the kept token with the largest logit, the first of equals.  p[] holds the weights by now, so
            // the logits are read again; the kept set is never empty (the token nearest the entropy is always in it).
            double bp = -INFINITY; int bi = 0x7fffffff;
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int i = tid + kST * k;
                if (i < V && RWKV_KEY(k) <= prefix) { const double x = a.logits[i]; if (x > bp) { bp = x; bi = i; } }
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) {
                const double ob = __shfl_xor(bp, off, 64); const int oi = __shfl_xor(bi, off, 64);
                if (ob > bp || (ob == bp && oi < bi)) { bp = ob; bi = oi; }
            }
            __shared__ double fv[kST / 64]; __shared__ int fi[kST / 64];
            if ((tid & 63) == 0) { fv[tid >> 6] = bp; fi[tid >> 6] = bi; }
            __syncthreads();
            if (tid == 0) {
                for (int w = 1; w < kST / 64; ++w) if (fv[w] > bp || (fv[w] == bp && fi[w] < bi)) { bp = fv[w]; bi = fi[w]; }
                s_tok = bi < V ? bi : 0;
            }
            __syncthreads();
        }
#undef RWKV_KEY
#undef RWKV_SET_KEY
        token = s_tok;
    }
    if (tid == 0) {
        a.out_token[0] = token;
        if (a.n_done) a.n_done[0] += 1;
        bool stop = false;
        for (int i = 0; i < a.n_stop; ++i) stop = stop || a.stop_tokens[i] == (int64_t)token;
        if (stop && a.stop_flag) *a.stop_flag = 1;     // rwkvMaster.py:49-50: the stop token itself is still part of the output
    }
}

}  // namespace

int sample_launch(hipStream_t st, const SampleArgs &a) {
    if (a.V <= 0 || a.V > kST * kSMaxPer) return set_error(RWKV_ERR_SIZE, "sampler: vocabulary %d exceeds %d", a.V, kST * kSMaxPer);
    constexpr size_t kSmall = (size_t)8 * kST * 4, kLarge = (size_t)kSKeysLds * kST * 4;
    {   // the large variant's dynamic LDS exceeds the default limit: raised once per device
        static std::mutex mu;
        static bool configured[64] = {};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return set_error(RWKV_ERR_DEVICE, "sampler: no current device");
        std::lock_guard<std::mutex> lock(mu);
        if (!configured[dev]) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&sample_kernel<kSMaxPer>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLarge);
            if (e != hipSuccess) return set_error(RWKV_ERR_HIP, "sampler: %s", hipGetErrorString(e));
            configured[dev] = true;
        }
    }
    if (a.V <= kST * 8) hipLaunchKernelGGL(sample_kernel<8>, dim3(1), dim3(kST), kSmall, st, a);
    else hipLaunchKernelGGL(sample_kernel<kSMaxPer>, dim3(1), dim3(kST), kLarge, st, a);
    RWKV_CHECK_LAUNCH("sample_kernel");
    return RWKV_OK;
}

}  // namespace rwkv
