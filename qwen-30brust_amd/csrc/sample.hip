// Device sampler: src/sampling.rs:26-63 (greedy, top-k, temperature, top-p
// and the seeded draw) over the logits in HBM, with the padding-vocab mask of
// src/main.rs:262-266 applied on the fly.
//
//   1. k_sample_scan, the whole chip: finiteness ("invalid logits"), the first
//      id under the sort of sampling.rs:31 (descending total order, lowest
//      index on ties; temperature 0 returns it, sampling.rs:32-35) and a
//      histogram of the keys' top 11 bits;
//   2. K = top_k (every id when top_k is 0 or above the vocabulary).  Up to
//      kSampleMax: the histogram gives the digit that holds rank K - 1, so the
//      ids at or above that digit contain the K first; k_sample_gather
//      collects them and one workgroup sorts them in LDS (k_sample_small);
//   3. more ids (or more than kSampleMax of them in those digits): all of them
//      are radix-sorted in HBM (k_radix_count / k_radix_scatter, four stable
//      8-bit passes) and one workgroup folds the first K (k_sample_fold);
//   4. the probabilities in parallel, then the sequential f32 folds of
//      sampling.rs:44-62 (total, cumulative top-p cut, the draw scaled by the
//      kept mass, the walk) with the reference's rounding at every step
//      (Fold, below).
// The draw itself (rand's gen::<f32>()) comes from the host's ChaCha12
// stream and is passed in.
//
// Bound: latency.  The data is 608 KB of logits (plus 152 KB of mask); one
// workgroup walking it alone took about 20 us a pass, five passes a draw.
// A draw from 151,936 host logits, their copy to the device (22 us of kernels)
// included: top_k 20 372 -> 61 us, the whole support 2.3-3.3 ms -> 0.20-0.25 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdint>

#include "kernels.hpp"
#include "qh_device.hpp"

namespace qh {

namespace {

constexpr uint32_t kST = 1024;         // threads of the one-workgroup kernels
constexpr uint32_t kSW = kST / 64;     // their waves
constexpr uint32_t kBins = 2048;       // histogram of the keys' top 11 bits

// Unsigned key with the order of f32::total_cmp.
__device__ __forceinline__ uint32_t ukey(float v) { return (uint32_t)total_key(v) ^ 0x80000000u; }
// The float of a key (the inverse of ukey).
__device__ __forceinline__ float key_float(uint32_t u) {
    const uint32_t t = u ^ 0x80000000u;  // total_key
    return __uint_as_float(t ^ ((uint32_t)((int32_t)t >> 31) >> 1));
}
// Composite key: larger = earlier in the sampler's sort (key, then lower index).
__device__ __forceinline__ unsigned long long ckey(float v, uint32_t i) {
    return ((unsigned long long)ukey(v) << 32) | (uint32_t)~i;
}
__device__ __forceinline__ uint32_t ck_index(unsigned long long k) { return ~(uint32_t)k; }
__device__ __forceinline__ float ck_float(unsigned long long k) { return key_float((uint32_t)(k >> 32)); }

__device__ __forceinline__ float masked(const float* lg, const uint8_t* valid, uint32_t i) {
    return (valid && !valid[i]) ? -FLT_MAX : lg[i];  // f32::MIN (main.rs:262-266)
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, uint32_t lane) {
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// -------------------------------------------------------------- the scan --
// kPer consecutive rounds of loads are issued together: the pass is one or
// two memory round trips, whatever the vocabulary.
__global__ __launch_bounds__(kBlock) void k_sample_scan(SampleArgs a, int want_hist) {
    __shared__ uint32_t hist[kBins];
    __shared__ unsigned long long wbest[kWaves];
    constexpr uint32_t kPer = 8;
    const uint32_t tid = threadIdx.x, n = a.n, stride = gridDim.x * kBlock;
    if (want_hist) {
        for (uint32_t b = tid; b < kBins; b += kBlock) hist[b] = 0;
        __syncthreads();
    }
    unsigned long long best = 0;
    bool bad = false;
    for (uint32_t i0 = blockIdx.x * kBlock + tid; i0 < n; i0 += kPer * stride) {
        float v[kPer];
#pragma unroll
        for (uint32_t j = 0; j < kPer; j++) v[j] = masked(a.logits, a.valid, min(i0 + j * stride, n - 1));
#pragma unroll
        for (uint32_t j = 0; j < kPer; j++) {
            const uint32_t i = i0 + j * stride;
            if (i >= n) break;
            bad |= !finite_f(v[j]);
            const unsigned long long k = ckey(v[j], i);
            best = k > best ? k : best;
            if (want_hist) atomicAdd(&hist[(uint32_t)(k >> 53)], 1u);
        }
    }
#pragma unroll
    for (uint32_t o = 32; o > 0; o >>= 1) {
        const unsigned long long t = __shfl_xor(best, o, 64);
        best = t > best ? t : best;
    }
    if ((tid & 63) == 0) wbest[tid >> 6] = best;
    if (bad) atomicOr(&a.st->bad, 1u);
    __syncthreads();
    if (tid == 0) {
        for (uint32_t w = 1; w < kWaves; w++) best = wbest[w] > best ? wbest[w] : best;
        atomicMax(&a.st->top, best);
    }
    if (want_hist)
        for (uint32_t b = tid; b < kBins; b += kBlock)
            if (hist[b]) atomicAdd(&a.st->hist[b], hist[b]);
}

// The ids whose top digit is at or above the one that holds rank K - 1, to
// st->cand in any order, when there are at most kSampleMax of them; st->count
// = their number.  Every workgroup finds the digit itself (the histogram is 8
// KB).
__global__ __launch_bounds__(kBlock) void k_sample_gather(SampleArgs a, uint32_t K) {
    __shared__ uint32_t wsum[kWaves], digit, count;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n = a.n;
    constexpr uint32_t kB = kBins / kBlock;  // bins per thread, walked from the top
    uint32_t c[kB], s = 0;
#pragma unroll
    for (uint32_t j = 0; j < kB; j++) {
        c[j] = a.st->hist[kBins - 1 - (kB * tid + j)];
        s += c[j];
    }
    const uint32_t incl = wave_incl_scan(s, lane);
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    uint32_t run = incl - s;
    for (uint32_t w = 0; w < wv; w++) run += wsum[w];
#pragma unroll
    for (uint32_t j = 0; j < kB; j++) {
        if (run < K && run + c[j] >= K) {  // one thread, one bin: K <= n
            digit = kBins - 1 - (kB * tid + j);
            count = run + c[j];
        }
        run += c[j];
    }
    __syncthreads();
    if (blockIdx.x == 0 && tid == 0) a.st->count = count;
    if (count > kSampleMax) return;
    const uint32_t stride = gridDim.x * kBlock;
    for (uint32_t i = blockIdx.x * kBlock + tid; i < n; i += stride) {
        const unsigned long long k = ckey(masked(a.logits, a.valid, i), i);
        if ((uint32_t)(k >> 53) >= digit) {
            const uint32_t slot = atomicAdd(&a.st->ncand, 1u);
            if (slot < kSampleMax) a.st->cand[slot] = k;
        }
    }
}

// ------------------------------------------------------------- the folds --
// The sequential f32 folds s <- s + x_i (or s - x_i), each step rounded as the
// reference rounds it, computed in parallel.  While s stays in one binade
// [2^e, 2^(e+1)) it is an integer n in [2^23, 2^24) of units u = 2^(e-23), and
// a step adds RNE(x / u) with ties decided by n's parity alone.  So a step is
// a map (parity -> integer added), maps compose associatively, and a prefix
// scan over the threads' kSeg-element segments gives every segment's exact
// starting value; each thread then walks its segment in plain f32.  The first
// segment that leaves the binade has the right start, hence the right end:
// the fold restarts after it in the new binade (at most a few dozen times).
// x is non-increasing (sorted probabilities), so a step that leaves s
// unchanged ends the fold.
constexpr uint32_t kSeg = 16;
constexpr int kSat = 1 << 26;  // saturation of a map's sums: past 2^24 only "left the binade" matters
enum : uint32_t { kEvNone = 0u, kEvCross = 1u, kEvHit = 2u, kEvStall = 3u };

constexpr uint32_t kSerialCut = 640, kSerialAll = 256;  // most ids folded by one lane (pick_rank)

struct FoldLds {
    int w0[kSW], w1[kSW];
    uint32_t first;   // first thread with an event
    uint32_t kind;    // its event
    uint32_t at;      // element index of a hit
    float s;          // the fold's value after that thread
    float head[kSerialCut];  // the probabilities of a serial fold
};

// A then B.
__device__ __forceinline__ void compose(int& a0, int& a1, int b0, int b1) {
    a0 = min(a0 + ((a0 & 1) ? b1 : b0), kSat);
    a1 = min(a1 + ((a1 & 1) ? b0 : b1), kSat);  // parity of 1 + a1
}

// Folds x(i), i < K, from s in index order; hit(s_before, s_after, x) stops at
// the first element for which it holds (its index in `at`, else K).  Every
// thread of the workgroup (kST of them) calls it with the same arguments and
// gets the same results.  store(segment, value) is called with the fold's
// value before each kSeg-element segment it went through.  Returns the value
// after the last element folded.
template <bool SUB, class X, class Hit, class Store>
__device__ __forceinline__ float fold(FoldLds& F, uint32_t K, float s, X x, Hit hit, Store store, uint32_t& at,
                                      uint32_t& segs) {
#pragma clang fp contract(off)
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    at = K;
    segs = 0;
    for (uint32_t base = 0; base < K; base += kST * kSeg) {
        const uint32_t i0 = base + kSeg * tid;
        float v[kSeg];
#pragma unroll
        for (uint32_t j = 0; j < kSeg; j++) v[j] = i0 + j < K ? x(i0 + j) : 0.f;
        uint32_t done = 0;  // threads of this chunk already folded
        while (done < kST && base + kSeg * done < K) {
            const uint32_t e = (__float_as_uint(s) >> 23) & 0xffu;
            // s = n 2^(e - 150); too small for the scaling: one segment at a time
            const bool scaled = e > 30 && e < 230;
            const float inv = __uint_as_float((277u - min(max(e, 31u), 229u)) << 23);  // 2^(150 - e)
            const float u = __uint_as_float((min(max(e, 31u), 229u) - 23u) << 23);     // 2^(e - 150)
            const int n = (int)((__float_as_uint(s) & 0x7fffffu) | 0x800000u);
            int t0 = 0, t1 = 0;
            bool big = false;
            if (tid >= done) {
#pragma unroll
                for (uint32_t j = 0; j < kSeg; j++) {
                    float y = v[j] * inv, d0, d1;
                    if (SUB) {
                        big |= y > 4194304.f;
                        y = fminf(y, 4194304.f);
                        d0 = 12582912.f - (12582912.f - y);
                        d1 = 12582913.f - (12582913.f - y);
                    } else {
                        y = fminf(y, 8388608.f);
                        d0 = (8388608.f + y) - 8388608.f;
                        d1 = (8388609.f + y) - 8388609.f;
                    }
                    compose(t0, t1, (int)d0, (int)d1);
                }
            }
            // exclusive scan of the maps over the threads
            int c0 = t0, c1 = t1;
#pragma unroll
            for (uint32_t o = 1; o < 64; o <<= 1) {
                int p0 = __shfl_up(c0, o, 64), p1 = __shfl_up(c1, o, 64);
                if (lane >= o) {
                    compose(p0, p1, c0, c1);
                    c0 = p0;
                    c1 = p1;
                }
            }
            int x0 = __shfl_up(c0, 1, 64), x1 = __shfl_up(c1, 1, 64);
            if (lane == 0) x0 = x1 = 0;
            __syncthreads();  // the previous round's readers of F are done
            if (lane == 63) {
                F.w0[wv] = c0;
                F.w1[wv] = c1;
            }
            if (tid == 0) F.first = kST;
            __syncthreads();
            int a0 = 0, a1 = 0;
            for (uint32_t w = 0; w < wv; w++) compose(a0, a1, F.w0[w], F.w1[w]);
            compose(a0, a1, x0, x1);
            const int d = (n & 1) ? a1 : a0;
            // this segment in plain f32 from its start (right while no earlier
            // segment has an event)
            float q = tid <= done ? s : (float)(SUB ? n - d : n + d) * u;
            const float q0 = q;
            uint32_t ev = kEvNone, hit_at = 0;
            if (tid >= done && i0 < K) {
                const bool lost = tid > done && (!scaled || (SUB ? n - d < (1 << 23) : n + d >= (1 << 24)));
                float before = q;
#pragma unroll
                for (uint32_t j = 0; j < kSeg; j++) {
                    if (i0 + j >= K || ev == kEvHit) continue;
                    before = q;
                    const float t = SUB ? q - v[j] : q + v[j];
                    if (hit(before, t, v[j])) {
                        ev = kEvHit;
                        hit_at = i0 + j;
                    } else {
                        q = t;
                    }
                }
                if (ev == kEvNone) {
                    if (q == before && i0 + kSeg <= K) ev = kEvStall;  // the segment's last step changed nothing
                    else if (big || !scaled || (__float_as_uint(q) >> 23) != (__float_as_uint(s) >> 23)) ev = kEvCross;
                }
                if (lost) ev = kEvCross;  // an earlier segment has the event; this one's values are not used
            }
            if (ev != kEvNone) atomicMin(&F.first, tid);
            __syncthreads();
            const uint32_t first = F.first;
            if (tid >= done && tid <= first && i0 < K) store(i0 / kSeg, q0);
            const uint32_t lastt = min(first, min(kST, (K - base + kSeg - 1) / kSeg) - 1);  // last segment folded
            if (tid == lastt) {
                F.s = q;
                F.kind = first < kST ? ev : (uint32_t)kEvNone;
                F.at = hit_at;
            }
            __syncthreads();
            s = F.s;
            segs = base / kSeg + lastt + 1;
            if (F.kind == kEvHit) {
                at = F.at;
                return s;
            }
            if (F.kind == kEvStall) return s;
            done = lastt + 1;
        }
    }
    return s;
}

// sampling.rs:47-62 over the K sorted probabilities p(i): total, the top-p
// cut m, the kept mass (a prefix of the total's fold: its value before segment
// i is kept in seg[i]), the walk.  Returns the picked rank in every thread.
// A few ids are folded by one lane: up to kSerialCut where a top-p cut ends its
// second loop early, up to kSerialAll without one.  It takes 0.05-0.1 us an id,
// a fold() about 10 us and more over flat probabilities.  A draw from 2,000
// (32,000) host logits, one lane / three folds: top_p 0.95, top_k 256 52 / 64
// (71 / 84) us, 512 73 / 77 (95 / 97), 700 81 / 82 (111 / 101); top_p 1, 256
// 60 / 65 (75 / 85), with a few likely ids 59 / 57 (62 / 60), 384 72 / 59 (83 / 70).
template <class P>
__device__ __forceinline__ uint32_t pick_rank(FoldLds& F, uint32_t K, const SampleArgs& a, P p, float* seg,
                                              uint32_t& m_out) {
#pragma clang fp contract(off)
    if (K <= (a.top_p < 1.f ? kSerialCut : kSerialAll)) {
        for (uint32_t i = threadIdx.x; i < K; i += kST) F.head[i] = p(i);
        __syncthreads();
        if (threadIdx.x == 0) {
            float total = -0.0f, cumulative = 0.f, kept = -0.0f;
            for (uint32_t i = 0; i < K; i++) total += F.head[i];
            uint32_t m = K, r = 0;
            for (uint32_t i = 0; i < K; i++) {
                const float x = F.head[i];
                cumulative += x / total;
                kept += x;
                if (cumulative >= a.top_p) {
                    m = i + 1;
                    break;
                }
            }
            float draw = a.draw * kept;
            for (; r < m; r++) {
                const float x = F.head[r];
                if (draw < x) break;
                draw -= x;
            }
            F.first = m;
            F.at = r < m ? r : m - 1;  // ids.last()
        }
        __syncthreads();
        m_out = F.first;
        return F.at;
    }
    uint32_t at, segs, unused;
    const float total = fold<false>(F, K, -0.0f, p, [](float, float, float) { return false; },
                                    [&](uint32_t i, float v) { seg[i] = v; }, at, segs);
    const float top_p = a.top_p;
    fold<false>(F, K, 0.0f, [&](uint32_t i) { return p(i) / total; },
                [&](float, float after, float) { return after >= top_p; }, [](uint32_t, float) {}, at, unused);
    const uint32_t m = min(at + 1, K);  // K when the cut is never reached
    float kept = total;
    if (m < K && m / kSeg < segs) {
        kept = seg[m / kSeg];
        for (uint32_t i = m / kSeg * kSeg; i < m; i++) kept += p(i);
    }
    fold<true>(F, m, a.draw * kept, p, [](float before, float, float x) { return before < x; }, [](uint32_t, float) {},
               at, unused);
    m_out = m;
    return at < m ? at : m - 1;  // ids.last()
}

// exp((v - max) / T), sampling.rs:43-46
__device__ __forceinline__ float prob_of(float v, float mx, float T) {
#pragma clang fp contract(off)
    return expf((v - mx) / T);
}

// The K first ids among the gathered candidates: sorted in LDS, folded.
__global__ __launch_bounds__(kST) void k_sample_small(SampleArgs a, uint32_t K) {
    __shared__ unsigned long long cand[kSampleMax];
    __shared__ float p[kSampleMax], seg[kSampleMax / kSeg];
    __shared__ FoldLds F;
    const uint32_t tid = threadIdx.x, C = a.st->count;
    if (a.st->bad) {
        if (tid == 0) a.st->status = kSampleBadLogits;
        return;
    }
    if (C > kSampleMax) {
        if (tid == 0) a.st->status = kSampleSupport;
        return;
    }
    if (C <= kST) {
        // each key's rank counted directly: no barrier per step, C LDS reads
        // that every lane shares
        const unsigned long long mine = tid < C ? a.st->cand[tid] : 0ull;
        cand[tid] = mine;
        __syncthreads();
        uint32_t r = 0;
        if (tid < C)
            for (uint32_t i = 0; i < C; i++) r += cand[i] > mine;
        __syncthreads();
        if (tid < C) cand[r] = mine;  // keys are distinct
        __syncthreads();
    } else {
        uint32_t np = 2 * kST;
        while (np < C) np <<= 1;
        for (uint32_t i = tid; i < np; i += kST) cand[i] = i < C ? a.st->cand[i] : 0ull;  // 0: below every finite key
        __syncthreads();
        for (uint32_t k = 2; k <= np; k <<= 1) {
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                for (uint32_t t = tid; t < np / 2; t += kST) {
                    const uint32_t i = 2 * t - (t & (j - 1)), l = i + j;  // i has bit j clear
                    const unsigned long long x = cand[i], y = cand[l];
                    const bool down = (i & k) == 0;  // descending runs first: overall descending
                    if (down ? x < y : x > y) {
                        cand[i] = y;
                        cand[l] = x;
                    }
                }
                __syncthreads();
            }
        }
    }
    const float mx = ck_float(a.st->top), T = a.temperature;
    for (uint32_t i = tid; i < K; i += kST) p[i] = prob_of(ck_float(cand[i]), mx, T);
    __syncthreads();
    uint32_t m;
    const uint32_t r = pick_rank(F, K, a, [&](uint32_t i) { return p[i]; }, seg, m);
    if (tid == 0) {
        a.st->id = ck_index(cand[r]);
        a.st->status = 0;
        a.st->kept = m;
    }
}

// ---------------------------------------------------------- the full sort --
// LSD radix sort of the n ids by ~key (descending keys), stable, so that equal
// keys keep ascending ids: four passes over 8-bit digits of (~key << 32 | id)
// words.  A workgroup owns kRBlk consecutive words; pass 0 reads the logits.
constexpr uint32_t kRPer = 8, kRBlk = kBlock * kRPer;  // words per thread, per workgroup

__device__ __forceinline__ unsigned long long radix_word(const SampleArgs& a, const unsigned long long* in, uint32_t i) {
    return in ? in[i] : ((unsigned long long)~ukey(masked(a.logits, a.valid, i)) << 32) | i;
}

// table[workgroup][digit] = its count of the digit.
__global__ __launch_bounds__(kBlock) void k_radix_count(SampleArgs a, const unsigned long long* in, uint32_t shift,
                                                        uint32_t* table) {
    __shared__ uint32_t cnt[256];
    const uint32_t tid = threadIdx.x, b0 = blockIdx.x * kRBlk;
    cnt[tid] = 0;
    unsigned long long w[kRPer];
#pragma unroll
    for (uint32_t j = 0; j < kRPer; j++) w[j] = radix_word(a, in, min(b0 + j * kBlock + tid, a.n - 1));
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kRPer; j++)
        if (b0 + j * kBlock + tid < a.n) atomicAdd(&cnt[(uint32_t)(w[j] >> shift) & 255u], 1u);
    __syncthreads();
    table[blockIdx.x * 256 + tid] = cnt[tid];
}

// Each word to its place: the digit's base (the counts of lower digits, and of
// this digit in earlier workgroups: every workgroup sums the table itself),
// the counts of earlier waves, and its rank in the wave.  A wave's words are
// consecutive, 64 per round, so the ranks keep the order.
__global__ __launch_bounds__(kBlock) void k_radix_scatter(SampleArgs a, const unsigned long long* in, uint32_t shift,
                                                          const uint32_t* table, unsigned long long* out) {
    __shared__ uint32_t wcnt[kWaves][256], wsum[kWaves];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nwg = gridDim.x;
    const uint32_t i0 = blockIdx.x * kRBlk + wv * 64 * kRPer + lane;
    unsigned long long w[kRPer];
#pragma unroll
    for (uint32_t j = 0; j < kRPer; j++) w[j] = radix_word(a, in, min(i0 + 64 * j, a.n - 1));
    for (uint32_t k = 0; k < kWaves; k++) wcnt[k][tid] = 0;
    // thread d: digit d's total and its count in earlier workgroups
    uint32_t total = 0, before = 0;
    for (uint32_t g0 = 0; g0 < nwg; g0 += 16) {
        uint32_t c[16];
#pragma unroll
        for (uint32_t j = 0; j < 16; j++) c[j] = table[min(g0 + j, nwg - 1) * 256 + tid];
#pragma unroll
        for (uint32_t j = 0; j < 16; j++) {
            const uint32_t g = g0 + j, v = g < nwg ? c[j] : 0u;
            total += v;
            before += g < blockIdx.x ? v : 0u;
        }
    }
    const uint32_t incl = wave_incl_scan(total, lane);
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();  // wcnt is clear
    uint32_t base = incl - total + before;
    for (uint32_t k = 0; k < wv; k++) base += wsum[k];
    uint32_t rank[kRPer];
#pragma unroll
    for (uint32_t j = 0; j < kRPer; j++) {
        const bool ok = i0 + 64 * j < a.n;
        const uint32_t d = (uint32_t)(w[j] >> shift) & 255u;
        unsigned long long same = __ballot(ok);
#pragma unroll
        for (uint32_t bit = 0; bit < 8; bit++) {
            const unsigned long long set = __ballot((d >> bit) & 1);
            same &= ((d >> bit) & 1) ? set : ~set;
        }
        const unsigned long long lower = same & ((1ull << lane) - 1);
        rank[j] = wcnt[wv][d] + (uint32_t)__popcll(lower);
        // the wave's LDS operations run in order: every lane has read the count
        __builtin_amdgcn_wave_barrier();
        if (ok && lower == 0) wcnt[wv][d] += (uint32_t)__popcll(same);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t run = base;  // thread d: where each wave's words of digit d start
    for (uint32_t k = 0; k < kWaves; k++) {
        const uint32_t c = wcnt[k][tid];
        wcnt[k][tid] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kRPer; j++)
        if (i0 + 64 * j < a.n) out[wcnt[wv][(uint32_t)(w[j] >> shift) & 255u] + rank[j]] = w[j];
}

// Probabilities of the first K sorted ids.
__global__ __launch_bounds__(kBlock) void k_sample_prob(SampleArgs a, const unsigned long long* sorted, uint32_t K,
                                                        float* prob) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const float mx = ck_float(a.st->top);
    if (i < K) prob[i] = prob_of(key_float(~(uint32_t)(sorted[i] >> 32)), mx, a.temperature);
}

__global__ __launch_bounds__(kST) void k_sample_fold(SampleArgs a, const unsigned long long* sorted, const float* prob,
                                                     uint32_t K, float* seg) {
    __shared__ FoldLds F;
    if (a.st->bad) {
        if (threadIdx.x == 0) a.st->status = kSampleBadLogits;
        return;
    }
    uint32_t m;
    const uint32_t r = pick_rank(F, K, a, [&](uint32_t i) { return prob[i]; }, seg, m);
    if (threadIdx.x == 0) {
        a.st->id = (uint32_t)sorted[r];
        a.st->status = 0;
        a.st->kept = m;
    }
}

uint32_t scan_grid(uint32_t n) { return std::min<uint32_t>((n + 4 * kBlock - 1) / (4 * kBlock), 128); }
uint32_t radix_wgs(uint32_t n) { return (n + kRBlk - 1) / kRBlk; }

}  // namespace

void launch_sample_scan(const SampleArgs& a, bool want_hist, hipStream_t s) {
    k_sample_scan<<<scan_grid(a.n), kBlock, 0, s>>>(a, (int)want_hist);
}

void launch_sample_small(const SampleArgs& a, uint32_t K, hipStream_t s) {
    k_sample_gather<<<scan_grid(a.n), kBlock, 0, s>>>(a, K);
    k_sample_small<<<1, kST, 0, s>>>(a, K);
}

size_t sample_sort_bytes(uint32_t n) {
    return (size_t)n * 16 + (size_t)radix_wgs(n) * 1024 + (size_t)n * 4 + ((size_t)n / kSeg + 2) * 4;
}

void launch_sample_full(const SampleArgs& a, uint32_t K, void* work, hipStream_t s) {
    auto* w0 = static_cast<unsigned long long*>(work);
    auto* w1 = w0 + a.n;
    auto* table = reinterpret_cast<uint32_t*>(w1 + a.n);
    float* prob = reinterpret_cast<float*>(table + (size_t)radix_wgs(a.n) * 256);
    float* seg = prob + a.n;
    const uint32_t g = radix_wgs(a.n);
    const unsigned long long* in = nullptr;
    for (uint32_t pass = 0; pass < 4; pass++) {
        unsigned long long* out = pass & 1 ? w1 : w0;
        k_radix_count<<<g, kBlock, 0, s>>>(a, in, 32 + 8 * pass, table);
        k_radix_scatter<<<g, kBlock, 0, s>>>(a, in, 32 + 8 * pass, table, out);
        in = out;
    }
    k_sample_prob<<<(K + kBlock - 1) / kBlock, kBlock, 0, s>>>(a, in, K, prob);
    k_sample_fold<<<1, kST, 0, s>>>(a, in, prob, K, seg);
}

}  // namespace qh
