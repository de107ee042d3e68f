// attn_mq.hip -- multi-query (prefill) GQA attention over an f16 KV cache for
// gfx950: the query_len > 1 form of the reference attention dispatch
// (runtime/zig/tests/tsir/real/attention_head256_f16kv/
// attention_head256_f16kv.wgsl:72-267).
//
// Semantics (that file):  query i of the call sits at absolute position
// start_pos + i; it sees logical keys p in [lo_i, hi_i) where hi_i =
// min(L, abs - kv_start + 1) when causal (0 when abs < kv_start) else L, and
// lo_i = abs - window + 1 - kv_start when a sliding window is set and abs >=
// window (clamped to [0, L]), L = seq_len or kv_len_buffer[0]; logical key p
// lives in cache row kv_start + p, that modulo the window (a ring) or through
// the page table (:51-63).  Scores are q.k * scale, softcapped as
// tanh(s / cap) * cap, softmax over the visible keys; a query without keys
// writes zeros.
//
// Kernels.  head_dim 64 / 128 / 256 runs attn_mq32_kernel (below).  head_dim 512
// (whose Q and O do not fit one wave's registers there), caches of 2 GiB and
// more and attn_mq.queries = 16 run attn_mq_kernel: one workgroup = 16
// consecutive queries x HG query heads of one KV head (one wave per head), keys
// in blocks of 32 staged in LDS and shared by the waves: K row-major for S = Q
// K^T and V transposed for O = P V, both on
// v_mfma_f32_16x16x32_f16.  Q is f32: each query row is scaled by a power of
// two (max near 2^14) and split into f16 hi + lo (~22 bits), so the scores
// carry f32 quality; P is rounded to f16 once (used for both the numerator
// and the row sum).  S and O accumulators share their row mapping (lane l
// holds rows 4 (l / 16) + r), so the online-softmax rescale needs no
// exchange; row max / sum go over the 16 lanes of a DPP row.
#include "common.h"

#include <math.h>
#include <algorithm>
#include <mutex>

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float max16(float v) {
    v = fmaxf(v, dpp<0xB1>(v));
    v = fmaxf(v, dpp<0x4E>(v));
    v = fmaxf(v, dpp<0x141>(v));
    return fmaxf(v, dpp<0x140>(v));
}
__device__ __forceinline__ float sum16(float v) {
    v += dpp<0xB1>(v);
    v += dpp<0x4E>(v);
    v += dpp<0x141>(v);
    return v + dpp<0x140>(v);
}

struct MqArgs {
    const float *q;  // [query][num_heads][D] with q_row_stride floats per query
    const _Float16 *k, *v;
    float *out;      // [query][num_heads][D] with out_row_stride floats per query
    const uint32_t *kv_len_dev;  // non-null: L = kv_len_dev[0]
    const uint32_t *page_table;
    long row_stride, head_stride;  // halves between cache rows / kv heads
    int q_row_stride, out_row_stride;
    int num_heads, num_kv_heads, heads_per_wg, query_len, seq_len, capacity;
    int start_pos, kv_start, causal, window, kv_map, ring, page_size, page_table_len;
    float scale, softcap;
    // key split (splits > 1, grid z): split z walks its share of the query
    // block's key blocks and writes the unnormalised (o, m, l) of each row to
    // ws_o [z][query][head][D] and ws_ml [z][query][head][2]; a second kernel
    // merges them
    int splits;
    float *ws_o, *ws_ml;
};

constexpr int kKeys = 32;  // keys per block

__device__ __forceinline__ long cache_row(const MqArgs &a, int p) {
    long r = (long)a.kv_start + p;
    if (a.kv_map == 1) {
        r %= a.ring;
    } else if (a.kv_map == 2) {
        long pg = r / a.page_size;
        const long in_page = r - pg * a.page_size;
        pg = pg < a.page_table_len ? pg : a.page_table_len - 1;
        r = (long)a.page_table[pg] * a.page_size + in_page;
    }
    return r < 0 ? 0 : (r >= a.capacity ? a.capacity - 1 : r);
}

// Key range [lo, hi) of the query at absolute position abs.
__device__ __forceinline__ void key_range(const MqArgs &a, int L, long abs, int &lo, int &hi) {
    hi = L;
    if (a.causal) hi = abs < a.kv_start ? 0 : (int)min((long)L, abs - a.kv_start + 1);
    lo = 0;
    if (a.window > 0 && abs >= a.window) {
        const long mk = abs - a.window + 1;
        if (mk > a.kv_start) lo = (int)min((long)L, mk - a.kv_start);
    }
}

template <int D>
struct MqLds {
    static constexpr int QROW = D + 8, KROW = D + 8, VROW = kKeys + 8, PROW = kKeys + 8;
    static size_t bytes(int hg) {
        return ((size_t)hg * 2 * 16 * QROW + (size_t)kKeys * KROW + (size_t)D * VROW + (size_t)hg * 16 * PROW) * 2 +
               (size_t)hg * 16 * 4;
    }
};

// NTH = 64 HG threads.  A key block is staged as 16-byte pieces c = tid +
// NTH i (key c % 32, dims 8 (c / 32) ..): up to eight pieces per thread are
// fetched into registers for the next block while the current one is
// computed, the rest (head_dim 512) just before it is staged.
template <int D, int NTH>
__global__ __launch_bounds__(NTH) void attn_mq_kernel(MqArgs a) {
    using Lds = MqLds<D>;
    constexpr int PIECES = kKeys * (D / 8);
    constexpr int PPT = (PIECES + NTH - 1) / NTH;
    constexpr int PF = PPT < 8 ? PPT : 8;
    constexpr int QROW = Lds::QROW, KROW = Lds::KROW, VROW = Lds::VROW, PROW = Lds::PROW;
    constexpr int NT = D / 16;  // O tiles of 16 dims
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int HG = a.heads_per_wg;
    _Float16 *qs = reinterpret_cast<_Float16 *>(lds_raw);     // [HG][2][16][QROW]
    _Float16 *ks = qs + (size_t)HG * 2 * 16 * QROW;           // [32][KROW]
    _Float16 *vt = ks + (size_t)kKeys * KROW;                 // [D][VROW]
    _Float16 *ps = vt + (size_t)D * VROW;                     // [HG][16][PROW]
    float *qinv = reinterpret_cast<float *>(ps + (size_t)HG * 16 * PROW);  // [HG][16]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g4 = lane >> 4, c16 = lane & 15;
    const int q0 = blockIdx.x * 16;
    const int kvh = blockIdx.y / (a.num_heads / a.num_kv_heads / HG);
    const int hg = blockIdx.y % (a.num_heads / a.num_kv_heads / HG);
    const int head = kvh * (a.num_heads / a.num_kv_heads) + hg * HG + wave;
    // keys beyond what the cache addressing can hold are never visited
    // (a device length is bounded so a bad value cannot make the loop run away)
    const long lmax = a.kv_map == 0 ? (long)a.capacity - min(a.kv_start, a.capacity)
                                    : (a.kv_map == 2 ? (long)a.page_table_len * a.page_size : (1L << 24));
    const int L = (int)min(lmax, (long)(a.kv_len_dev ? a.kv_len_dev[0] : (uint32_t)a.seq_len));

    // Per-row key ranges of this lane's four rows, and the union over the 16
    // queries (the same for every head of the workgroup).
    int rlo[4], rhi[4];
    int ulo = 1 << 30, uhi = 0;
    for (int i = 0; i < 16; ++i) {
        int lo, hi;
        key_range(a, L, (long)a.start_pos + q0 + i, lo, hi);
        const bool valid = q0 + i < a.query_len;
        if (valid && hi > lo) {
            ulo = min(ulo, lo);
            uhi = max(uhi, hi);
        }
        if ((i >> 2) == g4) {
            rlo[i & 3] = valid ? lo : 0;
            rhi[i & 3] = valid ? hi : 0;
        }
    }
    const float log2e = 1.4426950408889634f;
    const _Float16 *kb = a.k + (size_t)kvh * a.head_stride;
    const _Float16 *vb = a.v + (size_t)kvh * a.head_stride;
    const _Float16 *qh = qs + (size_t)(wave * 2 + 0) * 16 * QROW;
    const _Float16 *ql = qs + (size_t)(wave * 2 + 1) * 16 * QROW;
    _Float16 *pw = ps + (size_t)wave * 16 * PROW;

    // pieces [i0, i0 + n) of the block at p0: global -> registers -> LDS
    auto fetch = [&](int p0, int i0, int n, h8 *kd, h8 *vd) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const int c = tid + (i0 + i) * NTH;
            const int key = c % kKeys, d0 = (c / kKeys) * 8;
            const int p = p0 + key;
            h8 kv = h8{0, 0, 0, 0, 0, 0, 0, 0}, vv = kv;
            if (c < PIECES && p < L) {
                const long row = cache_row(a, p);
                kv = *reinterpret_cast<const h8 *>(kb + row * a.row_stride + d0);
                vv = *reinterpret_cast<const h8 *>(vb + row * a.row_stride + d0);
            }
            kd[i] = kv;
            vd[i] = vv;
        }
    };
    auto put = [&](int i0, int n, const h8 *kd, const h8 *vd) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const int c = tid + (i0 + i) * NTH;
            if (c < PIECES) {
                const int key = c % kKeys, d0 = (c / kKeys) * 8;
                *reinterpret_cast<h8 *>(ks + (size_t)key * KROW + d0) = kd[i];
                // consecutive lanes hold consecutive keys: each V^T row's
                // writes land in consecutive halves
#pragma unroll
                for (int e = 0; e < 8; ++e) vt[(size_t)(d0 + e) * VROW + key] = vd[i][e];
            }
        }
    };
    // this split's key blocks: a contiguous share of the union's blocks
    int p0 = (ulo / kKeys) * kKeys;
    if (a.splits > 1 && p0 < uhi) {
        const int nblk = (uhi - p0 + kKeys - 1) / kKeys, per = (nblk + a.splits - 1) / a.splits;
        const int b0 = (int)blockIdx.z * per;
        uhi = min(uhi, p0 + (b0 + per) * kKeys);
        p0 += b0 * kKeys;
    }
    // the first block's loads go out before Q is read and staged
    h8 kr[PF], vr[PF];
    if (p0 < uhi) fetch(p0, 0, PF, kr, vr);
    // Q: 4 lanes per query, D / 4 dims each; per-row power-of-two scale, hi/lo.
    {
        const int i = lane >> 2, part = lane & 3;
        const int qi = q0 + i;
        const bool valid = qi < a.query_len;
        const float *src = a.q + (size_t)(valid ? qi : 0) * a.q_row_stride + (size_t)head * D + part * (D / 4);
        float amax = 0.0f;
#pragma unroll 4
        for (int d = 0; d < D / 4; d += 4) {
            const float4 f = valid ? *reinterpret_cast<const float4 *>(src + d) : make_float4(0.f, 0.f, 0.f, 0.f);
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fmaxf(fabsf(f.z), fabsf(f.w))));
        }
        amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
        amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
        int sg = 0;
        if (amax > 0.0f && amax <= 3.0e38f) {
            sg = 14 - __builtin_amdgcn_frexp_expf(amax);
            sg = sg < -100 ? -100 : (sg > 100 ? 100 : sg);
        }
        const float sc = __builtin_amdgcn_ldexpf(1.0f, sg);
        _Float16 *hrow = qs + ((size_t)(wave * 2 + 0) * 16 + i) * QROW + part * (D / 4);
        _Float16 *lrow = qs + ((size_t)(wave * 2 + 1) * 16 + i) * QROW + part * (D / 4);
#pragma unroll 2
        for (int d = 0; d < D / 4; d += 8) {
            h8 hv, lv;
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const float4 f = valid ? *reinterpret_cast<const float4 *>(src + d + e) : make_float4(0.f, 0.f, 0.f, 0.f);
                const float t[4] = {f.x * sc, f.y * sc, f.z * sc, f.w * sc};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const _Float16 h = (_Float16)t[j];
                    hv[e + j] = h;
                    lv[e + j] = (_Float16)(t[j] - (float)h);
                }
            }
            *reinterpret_cast<h8 *>(hrow + d) = hv;
            *reinterpret_cast<h8 *>(lrow + d) = lv;
        }
        if (part == 0) qinv[wave * 16 + i] = __builtin_amdgcn_ldexpf(1.0f, -sg);
    }

    __syncthreads();
    float rowf[4];  // score scale of each row: scale / (the row's Q scale)
#pragma unroll
    for (int r = 0; r < 4; ++r) rowf[r] = a.scale * qinv[wave * 16 + 4 * g4 + r];

    f32x4 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m[4], l[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        m[r] = -INFINITY;
        l[r] = 0.0f;
    }
    for (; p0 < uhi; p0 += kKeys) {
        __syncthreads();  // every wave is done with the previous block
        put(0, PF, kr, vr);
        if constexpr (PPT > PF) {
            // the rest in chunks of eight pieces (eight loads in flight each)
#pragma unroll 1
            for (int i0 = PF; i0 < PPT; i0 += 8) {
                h8 k2[8], v2[8];
                fetch(p0, i0, 8, k2, v2);
                put(i0, 8, k2, v2);
            }
        }
        __syncthreads();
        if (p0 + kKeys < uhi) fetch(p0 + kKeys, 0, PF, kr, vr);  // in flight during this block

        // S = Q K^T: two 16-key tiles, Q hi and lo
        f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int c = 0; c < D / 32; ++c) {
            const h8 ah = *reinterpret_cast<const h8 *>(qh + (size_t)c16 * QROW + 32 * c + 8 * g4);
            const h8 al = *reinterpret_cast<const h8 *>(ql + (size_t)c16 * QROW + 32 * c + 8 * g4);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const h8 bk = *reinterpret_cast<const h8 *>(ks + (size_t)(16 * t + c16) * KROW + 32 * c + 8 * g4);
                s[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bk, s[t], 0, 0, 0);
                s[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bk, s[t], 0, 0, 0);
            }
        }
        // online softmax per row (lane holds rows 4 g4 + r, key p0 + 16 t + c16)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float x[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int p = p0 + 16 * t + c16;
                float v = s[t][r] * rowf[r];
                if (a.softcap > 0.0f) v = tanhf(v / a.softcap) * a.softcap;
                x[t] = (p >= rlo[r] && p < rhi[r]) ? v * log2e : -INFINITY;
            }
            const float bm = max16(fmaxf(x[0], x[1]));
            const float mn = fmaxf(m[r], bm);
            float corr = 1.0f;
            _Float16 ph[2] = {(_Float16)0.0f, (_Float16)0.0f};
            if (mn != -INFINITY) {
                corr = m[r] == -INFINITY ? 0.0f : exp2f(m[r] - mn);
#pragma unroll
                for (int t = 0; t < 2; ++t) ph[t] = (_Float16)(x[t] == -INFINITY ? 0.0f : exp2f(x[t] - mn));
                m[r] = mn;
            }
            l[r] = fmaf(l[r], corr, sum16((float)ph[0] + (float)ph[1]));
#pragma unroll
            for (int t = 0; t < NT; ++t) o[t][r] *= corr;
#pragma unroll
            for (int t = 0; t < 2; ++t) pw[(size_t)(4 * g4 + r) * PROW + 16 * t + c16] = ph[t];
        }
        __builtin_amdgcn_wave_barrier();
        // O += P V
        const h8 ap = *reinterpret_cast<const h8 *>(pw + (size_t)c16 * PROW + 8 * g4);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const h8 bv = *reinterpret_cast<const h8 *>(vt + (size_t)(16 * t + c16) * VROW + 8 * g4);
            o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ap, bv, o[t], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();  // P is rewritten by the next block
    }

#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int qi = q0 + 4 * g4 + r;
        if (qi >= a.query_len) continue;
        if (a.splits > 1) {
            const size_t pr = ((size_t)blockIdx.z * a.query_len + qi) * a.num_heads + head;
            float *dst = a.ws_o + pr * D + c16;
#pragma unroll
            for (int t = 0; t < NT; ++t) dst[16 * t] = o[t][r];
            if (c16 == 0) *reinterpret_cast<float2 *>(a.ws_ml + 2 * pr) = make_float2(m[r], l[r]);
            continue;
        }
        const float inv = l[r] > 0.0f ? 1.0f / l[r] : 0.0f;
        float *dst = a.out + (size_t)qi * a.out_row_stride + (size_t)head * D + c16;
#pragma unroll
        for (int t = 0; t < NT; ++t) dst[16 * t] = o[t][r] * inv;
    }
}

// ---------------------------------------------------------------------------
// head_dim 64 / 128 / 256: one workgroup = 32 queries of one head; its four waves
// take every fourth block of 32 keys and merge their (o, m, l) in LDS at the end,
// so no wave waits for another in between.
//   * S^T = K Q^T on v_mfma_f32_32x32x16_f16: a query per lane column (its max
//     and sum are one lane-half exchange), Q as f16 hi + lo in registers.
//   * S^T's sums are P^T's operand order of O^T = V^T P^T as they stand (the
//     keys of a step in the order the lane halves hold them), so P stays in
//     registers, as f16 hi + lo; V is read transposed (ds_read_b64_tr_b16).
//   * K and V go to LDS row by row by direct loads, one buffer of each per
//     wave: the next K block is under way during the softmax and P V, the next
//     V block during Q K.  The 16-byte chunks of a row are exchanged by key so
//     that the lanes' reads fall on different banks.
//   * The running max is raised only when a block's exceeds it by 2^8 (P at
//     most 256), so most blocks skip the rescale of O.  P in one f16 would lose
//     the largest P's exactness with that (1.5e-4 -> 1.8e-4 from float64) and
//     gain 3 us of 31; raising it every time costs what the second part costs
//     (34.6 against 34.1 us), and two parts give 2-4e-7.
// Bound, at head_dim 256, by the 128 KB of K and V that a CU's four waves read
// per round of blocks (~4500 cycles against 2800 of MFMA and softmax; loads
// issued earlier, further ahead or between the MFMAs measured no faster), and
// for a short prompt by the 4 us of launch, Q and first K before it.  us, with
// the 16-query kernel above (32-key blocks behind two barriers, V transposed
// by 2-byte stores) in brackets: 1000 tokens, 8 / 4 heads x 256 28 (80); 128
// tokens 11 (18); 1000 tokens, 16 / 4 x 128 19-20.5 (60.6); 1500 tokens, 16 / 4 x
// 64 17.5-18.9 (84); 40 queries, 8 / 4 x 256, over 8000 keys 30 (70).
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

template <int D>
struct Mq32Lds {
    static constexpr int kB = 32 * D * 2;  // bytes of a K or V block: four waves' K, their V; then the waves' O (f32 [D][32])
    static constexpr int kMl = 8 * kB, kBytes = kMl + 4 * 32 * 8;
};

// At most N vector-memory operations outstanding; LDS reads stay below it.
template <int N>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | (((N >> 4) & 3) << 14));
    __asm__ volatile("" ::: "memory");
}

// MAP: a ring or paged cache (kv_map 1 / 2).
template <int D, bool MAP>
__global__ __launch_bounds__(256, D == 256 ? 1 : 2) void attn_mq32_kernel(MqArgs a) {
    constexpr int NS = D / 16, NT = D / 32, CH = D / 8, NL = D / 16, VB = Mq32Lds<D>::kB;  // NL loads per block
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qc = lane & 31, lh = lane >> 5;
    // the last query blocks see the most keys: first
    const int head = blockIdx.x % a.num_heads, qb = (a.query_len + 31) / 32 - 1 - blockIdx.x / a.num_heads;
    const int q0 = qb * 32, kvh = head / (a.num_heads / a.num_kv_heads);
    // this wave's eight queries' rows, loaded first
    constexpr int QL = D / 4, QPL = 64 / QL, NQ = 8 / QPL;  // lanes per row, rows per load, loads
    const int dl = lane % QL;
    float4 f[NQ];
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        const int q = q0 + 8 * wave + j * QPL + lane / QL;
        f[j] = *reinterpret_cast<const float4 *>(a.q + (size_t)min(q, a.query_len - 1) * a.q_row_stride +
                                                 (size_t)head * D + 4 * dl);
    }
    const long lmax = !MAP ? (long)a.capacity - min(a.kv_start, a.capacity)
                           : (a.kv_map == 2 ? (long)a.page_table_len * a.page_size : (1L << 24));
    const int L = (int)min(lmax, (long)(a.kv_len_dev ? a.kv_len_dev[0] : (uint32_t)a.seq_len));

    // this lane's query's key range, the union over the 32 queries, and the
    // range that every one of them sees whole
    const int qi = q0 + qc;
    const bool valid = qi < a.query_len;
    int lo, hi;
    key_range(a, L, (long)a.start_pos + qi, lo, hi);
    int ulo = valid && hi > lo ? lo : 1 << 30, uhi = valid && hi > lo ? hi : 0;
    int flo = valid ? lo : 0, fhi = valid ? hi : 1 << 30;
#pragma unroll
    for (int x = 16; x > 0; x >>= 1) {
        ulo = min(ulo, __shfl_xor(ulo, x, 64));
        uhi = max(uhi, __shfl_xor(uhi, x, 64));
        flo = max(flo, __shfl_xor(flo, x, 64));
        fhi = min(fhi, __shfl_xor(fhi, x, 64));
    }
    ulo = __builtin_amdgcn_readfirstlane(ulo);
    uhi = __builtin_amdgcn_readfirstlane(uhi);
    flo = __builtin_amdgcn_readfirstlane(flo);
    fhi = __builtin_amdgcn_readfirstlane(fhi);
    // this split's blocks, of which this wave takes every fourth
    int b0 = ulo / 32, b1 = uhi > ulo ? (uhi + 31) / 32 : b0;
    if (a.splits > 1) {
        const int per = (b1 - b0 + a.splits - 1) / a.splits;
        b0 += (int)blockIdx.y * per;
        b1 = min(b1, b0 + per);
    }

    // Rows past L read as zero.  A load brings 64 / CH rows of CH chunks; place
    // c' of row `key` holds chunk c' ^ swz_k(key) of K, c' ^ swz_v(key) of V
    // (row strides are multiples of the row, so the exchange stays within it)
    const uint32_t row2 = (uint32_t)a.row_stride * 2u;
    const size_t base = (size_t)kvh * a.head_stride + (MAP ? 0 : (size_t)a.kv_start * a.row_stride);
    const int rows = MAP ? a.capacity : L;
    const int kv_bytes = rows > 0 ? (int)((uint32_t)(rows - 1) * row2 + 2u * D) : 0;
    const __amdgpu_buffer_rsrc_t krsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.k + base), (short)0, kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.v + base), (short)0, kv_bytes, 0x00020000);
    auto swz_k = [](int key) { return D == 64 ? (key >> 1) & 7 : key & 15; };  // 16 keys over all banks
    auto swz_v = [](int key) { return D == 64 ? 4 * ((key >> 1) & 1) : 4 * (key & 3); };  // 4 keys' 64 bytes
    uint32_t l_chunk = (uint32_t)(lane % CH);
    uint8_t *kmine = lds_raw + wave * VB, *vmine = kmine + 4 * VB;
    // a mapped cache: lane = key of block b, its row's offset (past L none)
    auto mapped_row = [&](int b) __attribute__((always_inline)) {
        return b * 32 + qc < L ? (uint32_t)cache_row(a, b * 32 + qc) * row2 : 0x80000000u;
    };
    auto load_block = [&](const __amdgpu_buffer_rsrc_t &rsrc, uint8_t *dst, int b, bool is_v) __attribute__((always_inline)) {
        const uint32_t mapped = MAP ? mapped_row(b) : 0;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int key0 = i * (64 / CH), key = key0 + lane / CH;
            const uint32_t row = MAP ? (uint32_t)__shfl((int)mapped, key, 64) : (uint32_t)(lane / CH) * row2;
            const uint32_t chunk = (l_chunk ^ (uint32_t)(is_v ? swz_v(key) : swz_k(key))) * 16u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(dst + i * 1024), 16,
                                                     row + chunk, MAP ? 0u : ((uint32_t)b * 32u + (uint32_t)key0) * row2, 0, 0);
        }
    };
    // K operand of step i: key qc, dims 16 i + 8 lh (chunk 2 i + lh)
    uint32_t k_off = (uint32_t)(qc * (2 * D) + ((lh ^ swz_k(qc)) * 16));
    auto read_k = [&](int i) __attribute__((always_inline)) {
        return *reinterpret_cast<const h8 *>(kmine + (k_off ^ (uint32_t)(32 * i)));
    };
    // V^T operand of tile t, step st: keys 16 st + 4 lh + 0..3 and + 8, dim 32 t
    // + lane % 32; a lane's address is that of a quad of one key's dims
    constexpr int NVA = D == 64 ? 2 : 4;
    uint32_t va[NVA];
    {
        const int key = 4 * lh + ((lane >> 2) & 3), c0 = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
        for (int t = 0; t < NVA; ++t)
            va[t] = (uint32_t)(key * D * 2 + ((c0 + 4 * t) ^ swz_v(key)) * 16 + (lane & 1) * 8);
    }
    auto read_v = [&](int t, int st) __attribute__((always_inline)) {
        const uint8_t *p = vmine + va[t % NVA] + (t / NVA) * (64 * NVA) + st * (32 * D);
        typedef __attribute__((address_space(3))) s16x4 lds_s4;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p);
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(p + 16 * D));
        return __builtin_bit_cast(h8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    int b = b0 + wave;
    if (b < b1) load_block(krsrc, kmine, b, false);
    // Q: each wave scales its rows by a power of two each (max near 2^14), splits
    // them hi / lo and passes them to all waves through the V buffers in operand
    // order: unit (2 i + h) 32 + query (the queries exchanged by 2 i + h) holds
    // the eight dims 16 i + 8 h ..
    h8 qh[NS], ql[NS];
    float rowf;
    {
        uint8_t *qbuf = lds_raw + 4 * VB;
        float *qscale = reinterpret_cast<float *>(lds_raw + Mq32Lds<D>::kMl);
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            const int q = 8 * wave + j * QPL + lane / QL;
            float amax = fmaxf(fmaxf(fabsf(f[j].x), fabsf(f[j].y)), fmaxf(fabsf(f[j].z), fabsf(f[j].w)));
            amax = max16(amax);
            if (QL > 16) amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
            if (QL > 32) amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
            int sg = 0;
            if (amax > 0.0f && amax <= 3.0e38f) {
                sg = 14 - __builtin_amdgcn_frexp_expf(amax);
                sg = sg < -100 ? -100 : (sg > 100 ? 100 : sg);
            }
            const float sc = __builtin_amdgcn_ldexpf(1.0f, sg);
            const float t[4] = {f[j].x * sc, f[j].y * sc, f[j].z * sc, f[j].w * sc};
            h4 hv, lv;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                hv[e] = (_Float16)t[e];
                lv[e] = (_Float16)(t[e] - (float)hv[e]);
            }
            const int ih = dl >> 1;  // 2 i + h
            uint8_t *dst = qbuf + (ih * 32 + (q ^ (ih & 31))) * 16 + (dl & 1) * 8;
            *reinterpret_cast<h4 *>(dst) = hv;
            *reinterpret_cast<h4 *>(dst + VB) = lv;
            if (dl == 0) qscale[q] = a.scale * __builtin_amdgcn_ldexpf(1.0f, -sg);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int ih = 2 * i + lh;
            const uint8_t *src = qbuf + (ih * 32 + (qc ^ (ih & 31))) * 16;
            qh[i] = *reinterpret_cast<const h8 *>(src);
            ql[i] = *reinterpret_cast<const h8 *>(src + VB);
        }
        rowf = qscale[qc];
        __syncthreads();
        if (b < b1) load_block(vrsrc, vmine, b, true);
    }
    const float log2e = 1.4426950408889634f;
    const f32x16 zero = {0.0f};
    f32x16 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = zero;
    float m = -INFINITY, l = 0.0f;

    for (; b < b1; b += 4) {
        const int bn = b + 4 < b1 ? b + 4 : b;  // (the last block again: never used)
        // (addresses formed in the loop: kept across it they would take the
        // registers that Q and O need)
        __asm__ volatile("" : "+v"(l_chunk), "+v"(k_off));
        f32x16 s = zero;
        wait_vm<NL>();  // K has landed; V is younger
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const h8 kf = read_k(i);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qh[i], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, ql[i], s, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // every K read has returned (its MFMAs are issued)
        load_block(krsrc, kmine, bn, false);
        __builtin_amdgcn_sched_barrier(0);
        // lane: query qc, keys p0 + 4 lh + (r % 4) + 8 (r / 4)
        const int p0 = 32 * b;
        float x[16];
        if (a.softcap > 0.0f) {
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = tanhf(s[r] * rowf / a.softcap) * a.softcap * log2e;
        } else {
            const float f = rowf * log2e;
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = s[r] * f;
        }
        if (p0 < flo || p0 + 32 > fhi) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int p = p0 + 4 * lh + (r & 3) + 8 * (r >> 2);
                x[r] = p >= lo && p < hi ? x[r] : -INFINITY;
            }
        }
        float bm = x[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) bm = fmaxf(bm, x[r]);
        bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
        if (__any(bm > m + 8.0f)) {  // (m = -inf: any finite score)
            const float mn = bm > m + 8.0f ? bm : m;
            const float corr = mn == m ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            const bool empty = m == -INFINITY;
            m = mn;
            l *= corr;
            if (!__all(empty))
#pragma unroll
                for (int r = 0; r < 16 * NT; ++r) {
                    if constexpr (D == 256) {
                        // O fills 128 accumulator registers, Q as many VGPRs: scaled in
                        // place (as plain code O changes register files in every block).
                        // The MFMAs that wrote O are a Q K phase older.
                        float e = o[r >> 4][r & 15], tmp;
                        __asm__ volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                                         : "+a"(e), "=&v"(tmp)
                                         : "v"(corr));
                        o[r >> 4][r & 15] = e;
                    } else {
                        o[r >> 4][r & 15] *= corr;
                    }
                }
        }
        const float mref = m == -INFINITY ? 0.0f : m;
        h8 pf[2], pl[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float p = __builtin_amdgcn_exp2f(x[r] - mref);
            l += p;
            pf[r >> 3][r & 7] = (_Float16)p;
            pl[r >> 3][r & 7] = (_Float16)(p - (float)pf[r >> 3][r & 7]);
        }
        wait_vm<NL>();  // V has landed; the next K is younger
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const h8 v0 = read_v(t, 0), v1 = read_v(t, 1);
            o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, pf[0], o[t], 0, 0, 0);
            o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, pf[1], o[t], 0, 0, 0);
            o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, pl[0], o[t], 0, 0, 0);
            o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, pl[1], o[t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_block(vrsrc, vmine, bn, true);
        __builtin_amdgcn_sched_barrier(0);
    }

    // merge: every wave's O as [dim / 4][query] float4 over the K and V buffers (the
    // queries exchanged by dim so that the reads along dim spread over the banks)
    l += __shfl_xor(l, 32, 64);
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (0 << 8) | (0 << 14));
    __asm__ volatile("" ::: "memory");
    __syncthreads();  // every wave is done with its blocks
    float4 *om = reinterpret_cast<float4 *>(lds_raw + wave * 2 * VB);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int quad = 8 * t + 2 * g + lh;
            om[quad * 32 + (qc ^ (quad & 31))] = make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
        }
    float2 *ml = reinterpret_cast<float2 *>(lds_raw + Mq32Lds<D>::kMl);
    if (lh == 0) ml[wave * 32 + qc] = make_float2(m, l);
    __syncthreads();
    constexpr int QUADS = D / 4, QPI = 64 / QUADS;  // queries per pass of a wave
#pragma unroll
    for (int it = 0; it < 8 / QPI; ++it) {
        const int q = wave * 8 + it * QPI + lane / QUADS, quad = lane % QUADS;
        float2 w[4];
        float M = -INFINITY;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            w[k] = ml[k * 32 + q];
            M = fmaxf(M, w[k].x);
        }
        float lt = 0.0f;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float f = w[k].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(w[k].x - M);
            const float4 ov = reinterpret_cast<const float4 *>(lds_raw + k * 2 * VB)[quad * 32 + (q ^ (quad & 31))];
            lt = fmaf(w[k].y, f, lt);
            v.x = fmaf(ov.x, f, v.x);
            v.y = fmaf(ov.y, f, v.y);
            v.z = fmaf(ov.z, f, v.z);
            v.w = fmaf(ov.w, f, v.w);
        }
        if (q0 + q >= a.query_len) continue;
        if (a.splits > 1) {
            const size_t pr = ((size_t)blockIdx.y * a.query_len + q0 + q) * a.num_heads + head;
            *reinterpret_cast<float4 *>(a.ws_o + pr * D + 4 * quad) = v;
            if (quad == 0) *reinterpret_cast<float2 *>(a.ws_ml + 2 * pr) = make_float2(M, lt);
            continue;
        }
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        float *dst = a.out + (size_t)(q0 + q) * a.out_row_stride + (size_t)head * D + 4 * quad;
        dst[0] = v.x * inv;
        dst[1] = v.y * inv;
        dst[2] = v.z * inv;
        dst[3] = v.w * inv;
    }
}

// The key splits of one (query, head) row merged: M = max m_s, L = sum l_s
// 2^(m_s - M), out = sum o_s 2^(m_s - M) / L (zero where no key was visible).
__global__ __launch_bounds__(512) void attn_mq_combine_kernel(MqArgs a, int D) {
    const int row = blockIdx.x, qi = row / a.num_heads, head = row - qi * a.num_heads, d = threadIdx.x;
    const size_t stride = (size_t)a.query_len * a.num_heads;
    float M = -INFINITY;
    for (int z = 0; z < a.splits; ++z) M = fmaxf(M, a.ws_ml[2 * (z * stride + row)]);
    float L = 0.0f, O = 0.0f;
    if (M != -INFINITY) {
        for (int z = 0; z < a.splits; ++z) {
            const float2 ml = *reinterpret_cast<const float2 *>(a.ws_ml + 2 * (z * stride + row));
            const float f = ml.x == -INFINITY ? 0.0f : exp2f(ml.x - M);
            L = fmaf(ml.y, f, L);
            O = fmaf(a.ws_o[(z * stride + row) * D + d], f, O);
        }
    }
    a.out[(size_t)qi * a.out_row_stride + (size_t)head * D + d] = L > 0.0f ? O / L : 0.0f;
}

// Key-split partials: a library-owned grow-only workspace (see the header's
// workspace rule), and the split count (0 automatic, n > 0 forced).
std::mutex g_mq_mu;
void *g_mq_ws = nullptr;
size_t g_mq_ws_bytes = 0;
int g_mq_cus = 0;
int g_mq_splits = 0;
int g_mq_queries = 0;  // 0 automatic, 16: attn_mq_kernel at any head_dim

// The workspace of `splits` key splits' (o, m, l) in a.
int split_workspace(MqArgs &a, int D) {
    const size_t rows = (size_t)a.query_len * a.num_heads;
    const size_t o_bytes = (size_t)a.splits * rows * D * 4, need = o_bytes + (size_t)a.splits * rows * 8;
    std::lock_guard<std::mutex> lk(g_mq_mu);
    if (g_mq_ws_bytes < need) {
        doe::retire_workspace(g_mq_ws);  // queued kernels and captured graphs may still use it
        g_mq_ws = nullptr;
        g_mq_ws_bytes = 0;
        DOE_HIP_CHECK(hipMalloc(&g_mq_ws, need));
        g_mq_ws_bytes = need;
    }
    a.ws_o = (float *)g_mq_ws;
    a.ws_ml = (float *)((char *)g_mq_ws + o_bytes);
    return DOE_OK;
}

int launch_combine(const MqArgs &a, int D, hipStream_t st) {
    hipLaunchKernelGGL(attn_mq_combine_kernel, dim3((unsigned)(a.query_len * a.num_heads)), dim3(D), 0, st, a, D);
    DOE_LAUNCH_CHECK("attn_mq_combine_kernel");
    return DOE_OK;
}

// The 32-query kernel: caches that a 32-bit buffer offset reaches.  A short
// prompt over a long cache splits the key blocks that its queries can see over
// the grid, up to one workgroup per CU and at least eight blocks (two per wave)
// each, at head_dim 256 two where there are 16 and more.  us, 17 queries, in
// 1 / 2 / 4 / 8 / 16 splits: 8 / 4 heads x 256 over 145 keys 13.2 / 13.3 / 13.8
// / 15.1 / 17.5, 517 keys 19.7 / 17.5 / 16.3 / 15.7 / 17.8, 2017 keys 42.6 /
// 28.8 / 21.2 / 18.8 / 18.9, with a window of 512 after 8000 keys 20.0 / 18.3 /
// 17.2 / 15.9 / 17.8; 32 / 4 heads x 128 there 11.6 / 11.9 / 11.7 / 12.0 / 15.8
// and over 1017 keys 14.9 / 13.2 / 12.1 / 12.6 / 16.2.
template <int D>
int launch_mq32(const MqArgs &a0, hipStream_t st) {
    MqArgs a = a0;
    const int64_t base = (int64_t)((a.query_len + 31) / 32) * a.num_heads;
    DOE_REQUIRE(base <= 0x7fffffff, DOE_E_UNSUPPORTED, "too many queries");
    a.splits = 1;
    if (g_mq_splits > 0) {
        a.splits = g_mq_splits;
    } else if (!a.kv_len_dev && base < g_mq_cus) {
        int64_t keys = std::min(a.seq_len, a.capacity);
        if (a.causal) keys = std::max<int64_t>(0, std::min(keys, (int64_t)a.start_pos + a.query_len - a.kv_start));
        int64_t nkb = (keys + 31) / 32;
        // (32 queries' windows: window + 31 keys, from any place in a block on)
        if (a.causal && a.window > 0) nkb = std::min(nkb, ((int64_t)a.window + 61) / 32 + 1);
        const int64_t each = D == 256 && nkb >= 16 ? 2 : 8;
        const int64_t sp = std::min({(int64_t)g_mq_cus / base, nkb / each, (int64_t)16});
        if (sp > 1) a.splits = (int)sp;
    }
    if (a.splits > 1) {
        const int rc = split_workspace(a, D);
        if (rc) return rc;
    }
    constexpr int lds = Mq32Lds<D>::kBytes;
    static const hipError_t attr_rc = [] {
        hipError_t e = hipSuccess;
        for (const void *f : {(const void *)attn_mq32_kernel<D, false>, (const void *)attn_mq32_kernel<D, true>})
            if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        return e;
    }();
    DOE_HIP_CHECK(attr_rc);
    const dim3 grid((unsigned)base, (unsigned)a.splits);
    if (a.kv_map) hipLaunchKernelGGL((attn_mq32_kernel<D, true>), grid, dim3(256), lds, st, a);
    else hipLaunchKernelGGL((attn_mq32_kernel<D, false>), grid, dim3(256), lds, st, a);
    DOE_LAUNCH_CHECK("attn_mq32_kernel");
    return a.splits > 1 ? launch_combine(a, D, st) : DOE_OK;
}

template <int D>
int launch_mq(const MqArgs &a0, hipStream_t st) {
    MqArgs a = a0;
    if (g_mq_cus == 0) {
        int dev = 0, cus = 0;
        DOE_HIP_CHECK(hipGetDevice(&dev));
        DOE_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        g_mq_cus = cus > 0 ? cus : 256;
    }
    if constexpr (D <= 256) {
        if (g_mq_queries == 0 && (int64_t)a.capacity * a.row_stride * 2 < ((int64_t)1 << 31))
            return launch_mq32<D>(a, st);
    }
    const int G = a.num_heads / a.num_kv_heads;
    int hg = D <= 128 ? 8 : (D == 256 ? 4 : 2);
    while (hg > 1 && G % hg) hg >>= 1;
    if (hg > G) hg = G;
    a.heads_per_wg = hg;
    // Key split: a short prompt gives few workgroups (a 128-token prompt of
    // 4 kv heads: 32), whose last query blocks walk every key block in turn;
    // split the key blocks over the grid until about two workgroups per CU
    // (host-known key counts only: a device length keeps one split).
    const int qblocks = (a.query_len + 15) / 16, ygrid = a.num_kv_heads * (G / hg);
    int splits = 1;
    if (g_mq_splits > 0) {
        splits = g_mq_splits;
    } else if (!a.kv_len_dev) {
        const long nkb = ((long)min(a.seq_len, a.capacity) + kKeys - 1) / kKeys;
        const long base = (long)qblocks * ygrid;
        if (nkb > 1 && base < g_mq_cus) {
            long sp = 2L * g_mq_cus / base;
            sp = sp < nkb ? sp : nkb;
            splits = (int)(sp < 16 ? sp : 16);
        }
    }
    a.splits = splits;
    if (splits > 1) {
        const int rc = split_workspace(a, D);
        if (rc) return rc;
    }
    const size_t lds = MqLds<D>::bytes(hg);
    static const hipError_t attr_rc = [] {
        hipError_t e = hipSuccess;
        for (const void *f : {(const void *)attn_mq_kernel<D, 64>, (const void *)attn_mq_kernel<D, 128>,
                              (const void *)attn_mq_kernel<D, 256>, (const void *)attn_mq_kernel<D, 512>})
            if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        return e;
    }();
    DOE_HIP_CHECK(attr_rc);
    DOE_REQUIRE(lds <= 160 * 1024, DOE_E_UNSUPPORTED, "attention needs %zu bytes of LDS", lds);
    const dim3 grid((unsigned)qblocks, (unsigned)ygrid, (unsigned)splits);
    switch (hg) {
        case 1: hipLaunchKernelGGL((attn_mq_kernel<D, 64>), grid, dim3(64), lds, st, a); break;
        case 2: hipLaunchKernelGGL((attn_mq_kernel<D, 128>), grid, dim3(128), lds, st, a); break;
        case 4: hipLaunchKernelGGL((attn_mq_kernel<D, 256>), grid, dim3(256), lds, st, a); break;
        default: hipLaunchKernelGGL((attn_mq_kernel<D, 512>), grid, dim3(512), lds, st, a); break;
    }
    DOE_LAUNCH_CHECK("attn_mq_kernel");
    return splits > 1 ? launch_combine(a, D, st) : DOE_OK;
}

int mq_impl(MqArgs a, int64_t head_dim, hipStream_t st) {
    int rc = doe::require_init();
    if (rc) return rc;
    DOE_REQUIRE(a.num_heads > 0 && a.num_kv_heads > 0 && a.num_heads % a.num_kv_heads == 0, DOE_E_INVALID,
                "num_heads %d is not a positive multiple of num_kv_heads %d", a.num_heads, a.num_kv_heads);
    DOE_REQUIRE(head_dim == 64 || head_dim == 128 || head_dim == 256 || head_dim == 512, DOE_E_UNSUPPORTED,
                "head_dim %lld unsupported (64, 128, 256, 512)", (long long)head_dim);
    DOE_REQUIRE(a.query_len >= 0 && a.capacity > 0, DOE_E_INVALID, "bad query_len / cache capacity");
    if (a.query_len == 0) return DOE_OK;
    DOE_REQUIRE(a.q && a.k && a.v && a.out, DOE_E_INVALID, "null pointer");
    DOE_REQUIRE(((uintptr_t)a.q & 15) == 0 && (a.q_row_stride & 3) == 0 && ((uintptr_t)a.k & 15) == 0 &&
                    ((uintptr_t)a.v & 15) == 0 && (a.row_stride & 7) == 0 && (a.head_stride & 7) == 0,
                DOE_E_INVALID, "q, k and v must be 16-byte aligned (row strides too)");
    DOE_REQUIRE(a.kv_len_dev || (a.seq_len >= 0 && (a.kv_map != 0 || a.kv_start != 0 || a.seq_len <= a.capacity)),
                DOE_E_INVALID, "seq_len %d outside the %d-row cache", a.seq_len, a.capacity);
    switch (head_dim) {
        case 64: return launch_mq<64>(a, st);
        case 128: return launch_mq<128>(a, st);
        case 256: return launch_mq<256>(a, st);
        default: return launch_mq<512>(a, st);
    }
}

}  // namespace

namespace doe {

int mq_set_splits(int value) {
    DOE_REQUIRE(value >= 0 && value <= 16, DOE_E_INVALID, "attn_mq.splits is 0..16");
    g_mq_splits = value;
    return DOE_OK;
}

int mq_set_queries(int value) {
    DOE_REQUIRE(value == 0 || value == 16, DOE_E_INVALID, "attn_mq.queries is 0 or 16");
    g_mq_queries = value;
    return DOE_OK;
}

// The query_len > 1 form of doe_attention_dispatch (the reference's own
// uniforms; K/V [capacity][num_kv_heads][head_dim]).
int attention_dispatch_mq(const doe_attention_uniforms *u, const float *q, const uint16_t *k, const uint16_t *v,
                          float *output, const uint32_t *kv_len_buffer, const uint32_t *page_table,
                          int64_t page_table_len, int64_t kv_capacity, doe_stream_t stream) {
    MqArgs a{};
    a.q = q;
    a.k = reinterpret_cast<const _Float16 *>(k);
    a.v = reinterpret_cast<const _Float16 *>(v);
    a.out = output;
    a.kv_len_dev = u->kv_len_source ? kv_len_buffer : nullptr;
    a.page_table = page_table;
    a.row_stride = (long)u->num_kv_heads * u->head_dim;
    a.head_stride = u->head_dim;
    a.q_row_stride = a.out_row_stride = (int)(u->num_heads * u->head_dim);
    a.num_heads = (int)u->num_heads;
    a.num_kv_heads = (int)u->num_kv_heads;
    a.query_len = (int)u->query_len;
    a.seq_len = (int)u->seq_len;
    a.capacity = (int)kv_capacity;
    a.start_pos = (int)u->start_pos;
    a.kv_start = (int)u->kv_start;
    a.causal = u->is_causal != 0;
    a.window = (int)u->sliding_window;
    if (u->kv_layout == 1 && u->sliding_window > 0) {
        a.kv_map = 1;
        a.ring = (int)u->sliding_window;
    } else if (u->kv_layout == 2) {
        a.kv_map = 2;
        a.page_size = (int)u->page_size;
        a.page_table_len = (int)page_table_len;
    }
    a.scale = u->scale;
    a.softcap = u->attn_softcap;
    return mq_impl(a, u->head_dim, (hipStream_t)stream);
}

}  // namespace doe

extern "C" int doe_attn_prefill_f16kv(const float *q, int64_t q_row_stride, const uint16_t *k_cache,
                                      const uint16_t *v_cache, float *output, int64_t out_row_stride,
                                      int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t query_len,
                                      int64_t kv_len, int64_t kv_stride, int kv_layout, int64_t start_pos,
                                      float scale, float softcap, int64_t sliding_window, doe_stream_t stream) {
    DOE_REQUIRE(kv_layout == 0 || kv_layout == 1, DOE_E_UNSUPPORTED,
                "kv_layout %d (0: [kv_head][pos][dim], 1: [pos][kv_head][dim])", kv_layout);
    DOE_REQUIRE(num_heads > 0 && num_kv_heads > 0 && head_dim > 0 && query_len >= 0 && kv_stride > 0 &&
                    kv_len >= 0 && kv_len <= kv_stride && start_pos >= 0 && sliding_window >= 0 &&
                    q_row_stride >= num_heads * head_dim && out_row_stride >= num_heads * head_dim &&
                    kv_stride < (1 << 30) && query_len < (1 << 30) && start_pos < (1 << 30),
                DOE_E_INVALID, "bad prefill attention shape");
    MqArgs a{};
    a.q = q;
    a.k = reinterpret_cast<const _Float16 *>(k_cache);
    a.v = reinterpret_cast<const _Float16 *>(v_cache);
    a.out = output;
    a.row_stride = kv_layout == 0 ? head_dim : num_kv_heads * head_dim;
    a.head_stride = kv_layout == 0 ? kv_stride * head_dim : head_dim;
    a.q_row_stride = (int)q_row_stride;
    a.out_row_stride = (int)out_row_stride;
    a.num_heads = (int)num_heads;
    a.num_kv_heads = (int)num_kv_heads;
    a.query_len = (int)query_len;
    a.seq_len = (int)kv_len;
    a.capacity = (int)kv_stride;
    a.start_pos = (int)start_pos;
    a.causal = 1;
    a.window = (int)sliding_window;
    a.scale = scale;
    a.softcap = softcap;
    return mq_impl(a, head_dim, (hipStream_t)stream);
}
