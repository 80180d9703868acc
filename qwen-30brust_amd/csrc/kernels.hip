// gfx950 kernels behind the engine's raw test surfaces: repack of GGUF rows
// into the device layout, bit-exact dequantisation, single matvecs
// (Backend::matvec, src/backend.rs:29-52), router top-k (src/ops.rs:45-56),
// greedy argmax (src/sampling.rs:26-35) and GQA attention
// (src/ops.rs:57-98).  The token-step kernels live in step.hip.
#include "qh_block.hpp"

namespace qh {

// ============================================================ API kernels ==

// GGUF block rows -> device row layout (one thread per source byte).
__global__ __launch_bounds__(kBlock) void k_repack(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                   uint32_t kind, uint32_t cols, size_t rows,
                                                   size_t src_rb, size_t dst_rb) {
    uint32_t blk_el, blk_bytes;
    layout(kind, blk_el, blk_bytes);
    const RowGeo g = row_geo(kind, cols);
    const size_t total = rows * src_rb;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (size_t)gridDim.x * kBlock) {
        size_t r = i / src_rb, o = i % src_rb;
        uint32_t b = (uint32_t)(o / blk_bytes), j = (uint32_t)(o % blk_bytes);
        dst[r * dst_rb + dev_offset(kind, g, b, j)] = src[i];
    }
}

// p[i] = v for i < n: clears device memory inside a stream (or a captured
// graph) without a memset node.
__global__ __launch_bounds__(kBlock) void k_fill_u32(uint32_t* __restrict__ p, size_t n, uint32_t v) {
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) p[i] = v;
}

// dst[0, n) = src[0, n), dst[n, padded) = 0 (32-bit words): copies between
// device memory and the engine's pinned host memory, 16 bytes per lane where
// both sides are aligned.  A kernel in the stream costs a launch (about 3 us of
// host time); hipMemcpyAsync on a caller's pageable memory 10-20 us a call, and
// it returns only when the copy is done.
__global__ __launch_bounds__(kBlock) void k_stage(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src,
                                                  uint32_t n, uint32_t padded) {
    const uint32_t i0 = blockIdx.x * kBlock + threadIdx.x, stride = gridDim.x * kBlock;
    const bool vec = ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0;
    const uint32_t n4 = vec ? n / 4 : 0;
    for (uint32_t i = i0; i < n4; i += stride) reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
    for (uint32_t i = 4 * n4 + i0; i < padded; i += stride) dst[i] = i < n ? src[i] : 0u;
}

// The step state before a call, and (token_at not null) the token it runs.
__global__ void k_put_state(DevState* st, uint32_t pos, uint32_t n_given, uint32_t* token_at, uint32_t token) {
    if (threadIdx.x == 0) {
        *st = DevState{pos, n_given, 0u, 0u, {0u, 0u, 0u, 0u}};
        if (token_at) *token_at = token;
    }
}

// Bit-exact dequantisation of rows [0, rows) (src/quant.rs:81-84).
__global__ __launch_bounds__(kBlock) void k_dequant(DevMat m, size_t row0, size_t rows, float* __restrict__ out) {
    const size_t total = rows * m.cols;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (size_t)gridDim.x * kBlock) {
        size_t r = i / m.cols;
        uint32_t c = (uint32_t)(i % m.cols);
        out[i] = dequant_value(m.w + (row0 + r) * m.drb, m.kind, m.geo, c);
    }
}

// Router fold of one layer: F[e][k] = sum_j (router[e][j] ffn_norm[j]) wo[j][k]
// for 8 experts e0..e0+7 per workgroup and one column k per thread, f64
// accumulation of exact f64 products, rounded once to f32.  wo is the
// dequantised attn_output ([rows][cols] f32).
__global__ __launch_bounds__(kBlock) void k_router_fold(DevMat router, const float* __restrict__ norm,
                                                        const float* __restrict__ wo, uint32_t rows, uint32_t cols,
                                                        uint32_t experts, float* __restrict__ out) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x, e0 = blockIdx.y * 8;
    if (k >= cols) return;
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (uint32_t j = 0; j < rows; j++) {
        const double w = (double)wo[(size_t)j * cols + k], g = (double)norm[j];
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            if (e0 + i < experts) {
                const float r = reinterpret_cast<const float*>(router.w + (size_t)(e0 + i) * router.drb)[j];
                acc[i] = fma((double)r * g, w, acc[i]);
            }
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < 8; i++)
        if (e0 + i < experts) out[(size_t)(e0 + i) * cols + k] = (float)acc[i];
}

// y = W x for one matrix (Backend::matvec, src/backend.rs:29-52).  x is
// staged in LDS (x_global = false) or read from a zero-padded global copy.
template <int R>
__global__ __launch_bounds__(kBlock) void k_matvec(DevMat m, const float* __restrict__ x,
                                                   float* __restrict__ y, int x_in_lds) {
    extern __shared__ float4 smem4[];
    float* xs = reinterpret_cast<float*>(smem4);
    const float* xp = x;
    if (x_in_lds) {
        stage_lds(x, m.cols, pad32(m.cols), xs);
        xp = xs;
    }
    mv_all<R>(m, m.w, xp, [&](uint32_t r, float v) { y[r] = v; });
}
template __global__ void k_matvec<1>(DevMat, const float*, float*, int);
template __global__ void k_matvec<2>(DevMat, const float*, float*, int);
template __global__ void k_matvec<4>(DevMat, const float*, float*, int);
template __global__ void k_matvec<8>(DevMat, const float*, float*, int);

__global__ __launch_bounds__(kBlock) void k_route(const float* logits, uint32_t n, uint32_t top,
                                                  uint32_t* ids, float* w, uint32_t* err) {
    extern __shared__ float4 smem4[];
    route_block(logits, n, top, ids, w, err, reinterpret_cast<float*>(smem4));
}

// Greedy argmax (src/sampling.rs:26-35) over n logits: per-block partials,
// the last block reduces them.
__global__ __launch_bounds__(kBlock) void k_argmax(const float* logits, uint32_t n, int32_t* pkey,
                                                   uint32_t* pidx, uint32_t* counter, uint32_t* out,
                                                   uint32_t* err) {
    int32_t k = INT32_MIN;
    uint32_t idx = 0xffffffffu;
    bool bad = false;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        float v = logits[i];
        bad |= !finite_f(v);
        best_merge(k, idx, total_key(v), i);
    }
    if (bad) atomicOr(err, kErrLogits);
    block_best(k, idx);
    if (threadIdx.x == 0) {
        pkey[blockIdx.x] = k;
        pidx[blockIdx.x] = idx;
    }
    if (!last_arrival(counter, gridDim.x)) return;
    k = INT32_MIN;
    idx = 0xffffffffu;
    for (uint32_t b = threadIdx.x; b < gridDim.x; b += kBlock) best_merge(k, idx, pkey[b], pidx[b]);
    block_best(k, idx);
    if (threadIdx.x == 0) *out = idx;
}

// ================================================================ attention ==
// GQA causal attention for one query vector over T cached positions
// (src/ops.rs:57-98).  Grid (kvheads, chunks); chunk c covers keys
// [c*span, min(T, (c+1)*span)), taken in tiles of tc keys with an online
// softmax (running max m, running sum l, exp-weighted V sum rescaled by
// exp(m_old - m_new) per tile), so the chunk count, and with it the partial
// buffer, stays bounded for any T.  Element j of head g at time t lives at
// K[g*sh + t*st + j].  Each block computes, for the G = heads/kvheads query
// heads of its KV head, the chunk's (m, l, o); the last block of each KV
// head merges the chunks.  Scores are (q . k) / sqrt(d), as the reference
// divides (ops.rs:87).

__device__ __forceinline__ void attention_block(const AttnArgs& a, uint32_t T) {
    extern __shared__ float4 smem4[];
    float* sm = reinterpret_cast<float*>(smem4);
    const uint32_t g = blockIdx.x, ch = blockIdx.y;
    const uint32_t span = a.span, nch = (T + span - 1) / span;
    if (nch > a.max_chunks || nch > gridDim.y) {  // never index past the partial buffer
        if (a.err && g == 0 && ch == 0 && threadIdx.x == 0) atomicOr(a.err, kErrContext);
        return;
    }
    if (ch >= nch) return;
    const uint32_t G = a.heads / a.kvheads, d = a.d, tc = a.tc;
    const uint32_t k0 = ch * span, k1 = min(T, k0 + span);
    float* qs = sm;                    // [G][d]
    float* ks = qs + G * d;            // [tc][d+1]
    float* vs = ks + tc * (d + 1);     // [tc][d]
    float* ps = vs + tc * d;           // [G][tc]
    float* ml = ps + G * tc;           // [G][2]  running max and sum
    float* al = ml + 2 * G;            // [G]     rescale factor of the current tile
    float* os = al + G;                // [G][d]  running exp-weighted V sum
    for (uint32_t i = threadIdx.x; i < G * d; i += kBlock) {
        qs[i] = a.q[(g * G) * d + i];
        os[i] = 0.f;
    }
    for (uint32_t h = threadIdx.x; h < G; h += kBlock) {
        ml[2 * h] = -INFINITY;
        ml[2 * h + 1] = 0.f;
    }
    const float root = sqrtf((float)d);
    const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (uint32_t t0 = k0; t0 < k1; t0 += tc) {
        const uint32_t n = min(k1, t0 + tc) - t0;
        __syncthreads();  // the previous tile's readers are done
        for (uint32_t i = threadIdx.x; i < n * d; i += kBlock) {
            uint32_t t = i / d, j = i % d;
            size_t off = (size_t)g * a.sh + (size_t)(t0 + t) * a.st + j;
            ks[t * (d + 1) + j] = a.k[off];
            vs[t * d + j] = a.v[off];
        }
        __syncthreads();
        for (uint32_t p = threadIdx.x; p < G * n; p += kBlock) {
            uint32_t h = p / n, t = p % n;
            const float* qh = qs + h * d;
            const float* kt = ks + t * (d + 1);
            float s = 0.f;
            for (uint32_t j = 0; j < d; j++) s = fmaf(qh[j], kt[j], s);
            ps[h * tc + t] = s / root;
        }
        __syncthreads();
        for (uint32_t h = wv; h < G; h += kWaves) {
            float mt = -INFINITY;
            for (uint32_t t = lane; t < n; t += 64) mt = fmaxf(mt, ps[h * tc + t]);
            const float mo = ml[2 * h], M = fmaxf(mo, wave_max(mt));
            float l = 0.f;
            for (uint32_t t = lane; t < n; t += 64) {
                float e = expf(ps[h * tc + t] - M);
                ps[h * tc + t] = e;
                l += e;
            }
            l = wave_sum(l);
            const float alpha = expf(mo - M);  // 0 on the first tile
            if (lane == 0) {
                ml[2 * h] = M;
                ml[2 * h + 1] = fmaf(ml[2 * h + 1], alpha, l);
                al[h] = alpha;
            }
        }
        __syncthreads();
        for (uint32_t p = threadIdx.x; p < G * d; p += kBlock) {
            uint32_t h = p / d, j = p % d;
            float o = os[p] * al[h];
            for (uint32_t t = 0; t < n; t++) o = fmaf(ps[h * tc + t], vs[t * d + j], o);
            os[p] = o;
        }
    }
    // each thread writes the os entries it owns; ml was written before the
    // last barrier
    for (uint32_t p = threadIdx.x; p < G * d; p += kBlock) {
        uint32_t h = p / d, j = p % d;
        float* dst = a.part + ((size_t)(g * G + h) * a.max_chunks + ch) * (d + 2);
        dst[2 + j] = os[p];
        if (j == 0) {
            dst[0] = ml[2 * h];
            dst[1] = ml[2 * h + 1];
        }
    }
    if (!last_arrival(&a.counter[g], nch)) return;
    for (uint32_t p = threadIdx.x; p < G * d; p += kBlock) {
        uint32_t h = p / d, j = p % d;
        const float* base = a.part + (size_t)(g * G + h) * a.max_chunks * (d + 2);
        float M = -INFINITY;
        for (uint32_t c = 0; c < nch; c++) M = fmaxf(M, base[c * (d + 2)]);
        float L = 0.f, O = 0.f;
        for (uint32_t c = 0; c < nch; c++) {
            const float* pc = base + c * (d + 2);
            float e = expf(pc[0] - M);
            L = fmaf(pc[1], e, L);
            O = fmaf(pc[2 + j], e, O);
        }
        a.out[(g * G + h) * d + j] = O / L;
    }
    if (a.done) {
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(a.done, 1ull);
    }
}

__global__ __launch_bounds__(kBlock) void k_attention_api(AttnArgs a, uint32_t T) { attention_block(a, T); }

// The same for head_dim D = 128 or 64, at most 8 query heads per KV head and
// 16-byte aligned q, k, v (k_attention_api reads single floats, any shape).
// Bound by latency: at 3,581 keys the 14.7 MB of K and V are 2.3 us of HBM
// time, spread over one workgroup per CU.  So a workgroup requests a whole
// 64-key tile of K and V (and its q) at once, with 16-byte loads, and keeps
// them in registers; eight lanes share a key's dot products with the (up to)
// eight heads and exchange partial sums in 7 lane steps; a head's softmax is
// one wave over the tile's keys; each wave adds its own 16 keys to all heads'
// outputs.  The chunks are merged by a second launch with a workgroup per head
// (k_attention_merge): merged by the last workgroup of each KV head, four
// workgroups read all the partials.  32 / 4 heads of 128, 3,581 keys:
// k_attention_api 158 us a call on one stream, these two 11 (tile 8.1, merge
// 3.8 alone), and 7-8 in turn on three streams, which overlap.
template <int D>
__global__ __launch_bounds__(kBlock) void k_attention_tile(AttnArgs a, uint32_t T) {
    constexpr int NQ = D / 32, NV = D / 64;  // float4s of a key's row per lane, dims per lane of a V row
    constexpr uint32_t kTile = 64, kPW = 16;  // keys per tile, per wave
    __shared__ float sc[8][kTile + 1];        // scores
    __shared__ __align__(16) float ps[kTile][8];  // probabilities
    __shared__ float al[8], red[kWaves][8][D];
    const uint32_t g = blockIdx.x, ch = blockIdx.y, G = a.heads / a.kvheads;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6, kl = lane >> 3, p = lane & 7;
    const uint32_t k0 = ch * a.span, k1 = min(T, k0 + a.span);
    if (k0 >= T) return;
    const float* kb = a.k + (size_t)g * a.sh;
    const float* vb = a.v + (size_t)g * a.sh;
    float4 q[8][NQ];
#pragma unroll
    for (int h = 0; h < 8; h++)
#pragma unroll
        for (int i = 0; i < NQ; i++)
            q[h][i] = gld<float4>(a.q + (size_t)(g * G + min((uint32_t)h, G - 1)) * D + 4 * (p + 8 * i));
    float acc[8][NV];
#pragma unroll
    for (int h = 0; h < 8; h++)
#pragma unroll
        for (int i = 0; i < NV; i++) acc[h][i] = 0.f;
    const float root = sqrtf((float)D);
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};  // of heads 2 wv and 2 wv + 1
    for (uint32_t t0 = k0; t0 < k1; t0 += kTile) {
        float4 kr[2][NQ];
        float vr[kPW][NV];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int i = 0; i < NQ; i++)
                kr[r][i] = gld<float4>(kb + (size_t)min(t0 + kPW * wv + 8 * r + kl, k1 - 1) * a.st + 4 * (p + 8 * i));
        // values of keys past the end are read as 0, by the bounds of a buffer
        // resource over the tile: an infinite one times its probability 0 would
        // be NaN (zeroed behind the loads instead, a call took 0.5 us longer)
        const __amdgpu_buffer_rsrc_t vt =
            buf_rsrc(vb + (size_t)t0 * a.st, ((min(k1 - t0, kTile) - 1) * (uint32_t)a.st + D) * 4);
#pragma unroll
        for (uint32_t j = 0; j < kPW; j++) {
            const int off = (int)(((kPW * wv + j) * (uint32_t)a.st + NV * lane) * 4);
            if constexpr (NV == 2) {
                const float2 t = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(vt, off, 0, 0));
                vr[j][0] = t.x;
                vr[j][1] = t.y;
            } else {
                vr[j][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vt, off, 0, 0));
            }
        }
#pragma unroll
        for (int r = 0; r < 2; r++) {
            float s[8];
#pragma unroll
            for (int h = 0; h < 8; h++) {
                s[h] = 0.f;
#pragma unroll
                for (int i = 0; i < NQ; i++) {
                    s[h] = fmaf(q[h][i].x, kr[r][i].x, s[h]);
                    s[h] = fmaf(q[h][i].y, kr[r][i].y, s[h]);
                    s[h] = fmaf(q[h][i].z, kr[r][i].z, s[h]);
                    s[h] = fmaf(q[h][i].w, kr[r][i].w, s[h]);
                }
            }
            // sums over the key's eight lanes; lane p ends with head p's
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) {
                const bool up = p & o;
#pragma unroll
                for (int h = 0; h < o; h++) {
                    const float keep = up ? s[h + o] : s[h], send = up ? s[h] : s[h + o];
                    s[h] = keep + __shfl_xor(send, o, 64);
                }
            }
            sc[p][kPW * wv + 8 * r + kl] = s[0];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t i = 0; i < 2; i++) {
            const uint32_t h = 2 * wv + i;
            const float v = t0 + lane < k1 ? sc[h][lane] / root : -INFINITY;
            const float M = fmaxf(m[i], wave_max(v)), e = expf(v - M), alpha = expf(m[i] - M);  // 0 on the first tile
            l[i] = fmaf(l[i], alpha, wave_sum(e));
            m[i] = M;
            ps[lane][h] = e;
            if (lane == 0) al[h] = alpha;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 8; h++)
#pragma unroll
            for (int i = 0; i < NV; i++) acc[h][i] *= al[h];
#pragma unroll
        for (uint32_t j = 0; j < kPW; j++) {
            const float4 pa = *reinterpret_cast<const float4*>(&ps[kPW * wv + j][0]),
                         pb = *reinterpret_cast<const float4*>(&ps[kPW * wv + j][4]);
            const float w[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
#pragma unroll
            for (int h = 0; h < 8; h++)
#pragma unroll
                for (int i = 0; i < NV; i++) acc[h][i] = fmaf(w[h], vr[j][i], acc[h][i]);
        }
        // the next tile's scores go to sc, read before the barrier above; its
        // probabilities are written after the next barrier
    }
#pragma unroll
    for (int h = 0; h < 8; h++)
#pragma unroll
        for (int i = 0; i < NV; i++) red[wv][h][NV * lane + i] = acc[h][i];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < G * D; i += kBlock) {
        const uint32_t h = i / D, j = i % D;
        a.part[((size_t)(g * G + h) * a.max_chunks + ch) * (D + 2) + 2 + j] =
            (red[0][h][j] + red[1][h][j]) + (red[2][h][j] + red[3][h][j]);
    }
#pragma unroll
    for (uint32_t i = 0; i < 2; i++) {
        const uint32_t h = 2 * wv + i;
        if (lane < 2 && h < G)
            a.part[((size_t)(g * G + h) * a.max_chunks + ch) * (D + 2) + lane] = lane ? l[i] : m[i];
    }
}

// out[h] = the merge of head h's nch <= 64 chunk partials (m, l, o).
template <int D>
__global__ __launch_bounds__(kBlock) void k_attention_merge(AttnArgs a, uint32_t nch) {
    constexpr uint32_t NG = kBlock / D;  // chunks taken in turn by NG groups of D threads
    __shared__ float w[64], red[NG][D];
    const uint32_t lane = threadIdx.x & 63, j = threadIdx.x % D, grp = threadIdx.x / D;
    const float* base = a.part + (size_t)blockIdx.x * a.max_chunks * (D + 2);
    const bool ok = lane < nch;
    const float* mine = base + (size_t)min(lane, nch - 1) * (D + 2);
    const float mc = ok ? mine[0] : -INFINITY, lc = ok ? mine[1] : 0.f;
    constexpr uint32_t kPer = 64 / NG;
    float o[kPer];
#pragma unroll
    for (uint32_t i = 0; i < kPer; i++) o[i] = base[(size_t)min(grp + NG * i, nch - 1) * (D + 2) + 2 + j];
    const float M = wave_max(mc), e = ok ? expf(mc - M) : 0.f, L = wave_sum(lc * e);
    if (threadIdx.x < 64) w[lane] = e;
    __syncthreads();
    float O = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kPer; i++)
        if (grp + NG * i < nch) O = fmaf(w[grp + NG * i], o[i], O);
    red[grp][j] = O;
    __syncthreads();
    if (threadIdx.x == 0 && a.done) atomicAdd(a.done, 1ull);  // the partials have been read
    if (grp == 0) {
        for (uint32_t k = 1; k < NG; k++) O += red[k][j];
        a.out[(size_t)blockIdx.x * D + j] = O / L;
    }
}
template __global__ void k_attention_tile<64>(AttnArgs, uint32_t);
template __global__ void k_attention_tile<128>(AttnArgs, uint32_t);
template __global__ void k_attention_merge<64>(AttnArgs, uint32_t);
template __global__ void k_attention_merge<128>(AttnArgs, uint32_t);

// k_attention_tile and k_attention_merge in one launch that uses no memory
// besides its arguments: one workgroup per query head takes the chunks four at
// a time (four waves each, k_attention_tile's work for one head), keeps their
// partials in LDS and merges them.  Every sum has the two kernels' terms in
// their order, so the bits are theirs.
// Bound by one CU's share of the bandwidth (a head's K and V, 3.7 MB at 3,581
// keys of 128) and the tiles' barriers: 70 us a graph replay at 32 / 4 heads of
// 128 and 3,581 keys, 41 at 1,024, 16 at 64 (the two kernels, whose scratch a
// replay could share with another call: 16, 15, 15; of an eager call each 10-11).
template <int D>
__global__ __launch_bounds__(kDirectBlock) void k_attention_direct(AttnArgs a, uint32_t T) {
    constexpr int NQ = D / 32, NV = D / 64;
    constexpr uint32_t kTile = 64, kPW = 16, NC = kDirectBlock / kBlock;  // chunks at a time
    __shared__ float part[64][D + 2];
    __shared__ float sc[NC][kTile], ps[NC][kTile], al[NC], red[NC][kWaves][D], w[64];
    const uint32_t h = blockIdx.x, g = h / (a.heads / a.kvheads), nch = a.max_chunks;
    const uint32_t cg = threadIdx.x / kBlock, tid = threadIdx.x % kBlock;
    const uint32_t lane = tid & 63, wv = tid >> 6, kl = lane >> 3, p = lane & 7;
    const float* kb = a.k + (size_t)g * a.sh;
    const float* vb = a.v + (size_t)g * a.sh;
    float4 q[NQ];
#pragma unroll
    for (int i = 0; i < NQ; i++) q[i] = gld<float4>(a.q + (size_t)h * D + 4 * (p + 8 * i));
    const float root = sqrtf((float)D);
    for (uint32_t c0 = 0; c0 < nch; c0 += NC) {  // every thread passes every barrier
        const uint32_t ch = c0 + cg, k0 = ch * a.span, k1 = min(T, k0 + a.span);
        const bool live = ch < nch;
        float acc[NV], m = -INFINITY, l = 0.f;
#pragma unroll
        for (int i = 0; i < NV; i++) acc[i] = 0.f;
        for (uint32_t t = 0; t < a.span; t += kTile) {
            const uint32_t t0 = k0 + t;
            const bool on = live && t0 < k1;
            float4 kr[2][NQ];
            float vr[kPW][NV];
            if (on) {
#pragma unroll
                for (int r = 0; r < 2; r++)
#pragma unroll
                    for (int i = 0; i < NQ; i++)
                        kr[r][i] =
                            gld<float4>(kb + (size_t)min(t0 + kPW * wv + 8 * r + kl, k1 - 1) * a.st + 4 * (p + 8 * i));
#pragma unroll
                for (uint32_t j = 0; j < kPW; j++) {
                    const float* row = vb + (size_t)min(t0 + kPW * wv + j, k1 - 1) * a.st;
                    if constexpr (NV == 2) {
                        const float2 x = gld<float2>(row + 2 * lane);
                        vr[j][0] = x.x;
                        vr[j][1] = x.y;
                    } else {
                        vr[j][0] = gld<float>(row + lane);
                    }
                }
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    float s = 0.f;
#pragma unroll
                    for (int i = 0; i < NQ; i++) {
                        s = fmaf(q[i].x, kr[r][i].x, s);
                        s = fmaf(q[i].y, kr[r][i].y, s);
                        s = fmaf(q[i].z, kr[r][i].z, s);
                        s = fmaf(q[i].w, kr[r][i].w, s);
                    }
#pragma unroll
                    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
                    if (p == 0) sc[cg][kPW * wv + 8 * r + kl] = s;
                }
            }
            __syncthreads();
            if (on && wv == 0) {
                const float v = t0 + lane < k1 ? sc[cg][lane] / root : -INFINITY;
                const float M = fmaxf(m, wave_max(v)), e = expf(v - M), alpha = expf(m - M);
                l = fmaf(l, alpha, wave_sum(e));
                m = M;
                ps[cg][lane] = e;
                if (lane == 0) al[cg] = alpha;
            }
            __syncthreads();
            if (on) {
                if (t0 + kPW * wv + kPW > k1) {  // as there: no value past the end
#pragma unroll
                    for (uint32_t j = 0; j < kPW; j++)
#pragma unroll
                        for (int i = 0; i < NV; i++) vr[j][i] = t0 + kPW * wv + j < k1 ? vr[j][i] : 0.f;
                }
#pragma unroll
                for (int i = 0; i < NV; i++) acc[i] *= al[cg];
#pragma unroll
                for (uint32_t j = 0; j < kPW; j++) {
                    const float e = ps[cg][kPW * wv + j];
#pragma unroll
                    for (int i = 0; i < NV; i++) acc[i] = fmaf(e, vr[j][i], acc[i]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NV; i++) red[cg][wv][NV * lane + i] = acc[i];
        __syncthreads();
        if (live) {
            if (tid < D) part[ch][2 + tid] = (red[cg][0][tid] + red[cg][1][tid]) + (red[cg][2][tid] + red[cg][3][tid]);
            if (tid < 2) part[ch][tid] = tid ? l : m;  // of wave 0
        }
    }
    __syncthreads();
    constexpr uint32_t NG = kBlock / D, kPer = 64 / NG;
    float(*rg)[D] = red[0];
    const uint32_t j = tid % D, grp = tid / D;
    const bool ok = lane < nch;
    const uint32_t mine = min(lane, nch - 1);
    const float mc = ok ? part[mine][0] : -INFINITY, lc = ok ? part[mine][1] : 0.f;
    const float M = wave_max(mc), e = ok ? expf(mc - M) : 0.f, L = wave_sum(lc * e);
    if (threadIdx.x < 64) w[lane] = e;
    __syncthreads();
    float O = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kPer; i++)
        if (grp + NG * i < nch) O = fmaf(w[grp + NG * i], part[grp + NG * i][2 + j], O);
    if (cg == 0) rg[grp][j] = O;
    __syncthreads();
    if (threadIdx.x < D) {
        for (uint32_t k = 1; k < NG; k++) O += rg[k][j];
        a.out[(size_t)h * D + j] = O / L;
    }
}
template __global__ void k_attention_direct<64>(AttnArgs, uint32_t);
template __global__ void k_attention_direct<128>(AttnArgs, uint32_t);

// The same for other shapes of up to 8 E elements a head, without LDS partials:
// eight lanes share a key, with E elements of its row each, and keep the (m, l,
// o) of their own keys, so there is no barrier before the merge at the end.
// Another order of sums than k_attention_api's.
template <int E>
__global__ __launch_bounds__(kAnyBlock) void k_attention_any(AttnArgs a, uint32_t T) {
    constexpr uint32_t kW = kAnyBlock / 64, U = E <= 16 ? 2 : 1;  // waves; keys per lane group and step
    __shared__ float red[kW][8 * E], rm[kW], rl[kW];
    const uint32_t h = blockIdx.x, g = h / (a.heads / a.kvheads), d = a.d;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6, kl = lane >> 3, p = lane & 7;
    auto load = [&](float (&x)[E], const float* row) {  // elements p + 8 i, 0 past d
#pragma unroll
        for (int i = 0; i < E; i++) {
            const float t = gld<float>(row + min(p + 8 * i, d - 1));
            x[i] = p + 8 * i < d ? t : 0.f;
        }
    };
    float q[E], o[E], m = -INFINITY, l = 0.f;
    load(q, a.q + (size_t)h * d);
#pragma unroll
    for (int i = 0; i < E; i++) o[i] = 0.f;
    const float root = sqrtf((float)d);
    for (size_t t0 = 8 * wv; t0 < T; t0 += 8 * kW * U) {  // the wave's first key of the step
        float kr[U][E], vr[U][E], s[U], M = m;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) load(kr[u], a.k + g * a.sh + min(t0 + kl + 8 * kW * u, (size_t)T - 1) * a.st);
#pragma unroll
        for (uint32_t u = 0; u < U; u++) load(vr[u], a.v + g * a.sh + min(t0 + kl + 8 * kW * u, (size_t)T - 1) * a.st);
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            float t = 0.f;
#pragma unroll
            for (int i = 0; i < E; i++) t = fmaf(q[i], kr[u][i], t);
#pragma unroll
            for (int x = 1; x < 8; x <<= 1) t += __shfl_xor(t, x, 64);
            s[u] = t0 + kl + 8 * kW * u < T ? t / root : -INFINITY;
            M = fmaxf(M, s[u]);
        }
        const float Mf = M == -INFINITY ? 0.f : M, alpha = expf(m - Mf);  // 0 while no key came
        m = M;
        l *= alpha;
#pragma unroll
        for (int i = 0; i < E; i++) o[i] *= alpha;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const float e = expf(s[u] - Mf);
            if (t0 + kl + 8 * kW * u < T) {  // not 0 times the value of a key past the end
                l += e;
#pragma unroll
                for (int i = 0; i < E; i++) o[i] = fmaf(e, vr[u][i], o[i]);
            }
        }
    }
    // the wave's eight lane groups, then the waves
    float M = m;
#pragma unroll
    for (int x = 8; x < 64; x <<= 1) M = fmaxf(M, __shfl_xor(M, x, 64));
    const float e = expf(m - (M == -INFINITY ? 0.f : M));
    l *= e;
#pragma unroll
    for (int i = 0; i < E; i++) o[i] *= e;
#pragma unroll
    for (int x = 8; x < 64; x <<= 1) {
        l += __shfl_xor(l, x, 64);
#pragma unroll
        for (int i = 0; i < E; i++) o[i] += __shfl_xor(o[i], x, 64);
    }
    if (kl == 0) {
#pragma unroll
        for (int i = 0; i < E; i++) red[wv][p + 8 * i] = o[i];
    }
    if (lane == 0) {
        rm[wv] = M;
        rl[wv] = l;
    }
    __syncthreads();
    if (threadIdx.x < d) {
        float Ma = -INFINITY, L = 0.f, O = 0.f;
        for (uint32_t x = 0; x < kW; x++) Ma = fmaxf(Ma, rm[x]);
        if (Ma == -INFINITY) Ma = 0.f;
        for (uint32_t x = 0; x < kW; x++) {
            const float f = expf(rm[x] - Ma);
            L = fmaf(rl[x], f, L);
            O = fmaf(red[x][threadIdx.x], f, O);
        }
        a.out[(size_t)h * d + threadIdx.x] = O / L;
    }
}
template __global__ void k_attention_any<8>(AttnArgs, uint32_t);
template __global__ void k_attention_any<16>(AttnArgs, uint32_t);
template __global__ void k_attention_any<32>(AttnArgs, uint32_t);

// The same for heads of more than 256 elements (the LDS budget of the entry
// points ends at 4,094): tiles of 64 keys, eight lanes a
// key for the scores, then a thread per output element and key of the tile.
__global__ __launch_bounds__(kAnyBlock) void k_attention_wide(AttnArgs a, uint32_t T) {
    constexpr uint32_t kTile = 64, kMax = 8;  // keys per tile, output elements per thread
    __shared__ float ps[kTile], al, lsum;
    const uint32_t h = blockIdx.x, g = h / (a.heads / a.kvheads), d = a.d;
    const uint32_t lane = threadIdx.x & 63, key = threadIdx.x >> 3, p = threadIdx.x & 7;
    static_assert(kAnyBlock == 8 * kTile, "eight lanes a key");
    const float* q = a.q + (size_t)h * d;
    const float root = sqrtf((float)d);
    float o[kMax], m = -INFINITY, l = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kMax; i++) o[i] = 0.f;
    for (size_t t0 = 0; t0 < T; t0 += kTile) {
        const uint32_t n = (uint32_t)min((size_t)kTile, T - t0);
        const float* kt = a.k + g * a.sh + (t0 + min(key, n - 1)) * a.st;
        float s = 0.f;
        for (uint32_t j = p; j < d; j += 8) s = fmaf(gld<float>(q + j), gld<float>(kt + j), s);
#pragma unroll
        for (int x = 1; x < 8; x <<= 1) s += __shfl_xor(s, x, 64);
        if (p == 0) ps[key] = key < n ? s / root : -INFINITY;
        __syncthreads();
        if (threadIdx.x < 64) {
            const float v = ps[lane], M = fmaxf(m, wave_max(v)), Mf = M == -INFINITY ? 0.f : M;
            const float e = expf(v - Mf), alpha = expf(m - Mf);
            l = fmaf(l, alpha, wave_sum(e));
            m = M;
            ps[lane] = e;
            if (lane == 0) {
                al = alpha;
                lsum = l;
            }
        }
        __syncthreads();
        const float* vt = a.v + g * a.sh + t0 * a.st;
#pragma unroll
        for (uint32_t i = 0; i < kMax; i++) {
            const uint32_t j = threadIdx.x + kAnyBlock * i;
            if (j >= d) break;
            float x = o[i] * al;
#pragma unroll 8
            for (uint32_t t = 0; t < n; t++) x = fmaf(ps[t], gld<float>(vt + t * a.st + j), x);
            o[i] = x;
        }
        __syncthreads();  // the next tile's scores overwrite ps
    }
#pragma unroll
    for (uint32_t i = 0; i < kMax; i++) {
        const uint32_t j = threadIdx.x + kAnyBlock * i;
        if (j < d) a.out[(size_t)h * d + j] = o[i] / lsum;
    }
}

}  // namespace qh
