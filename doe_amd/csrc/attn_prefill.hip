// attn_prefill.hip -- causal GQA prefill attention (flash form) on gfx950 matrix cores.
//
// out[i][h][:] = softmax_j(q[i][h] . k[kvh][j] * scale) v[kvh][j], kvh = h / (Hq/Hkv),
// keys j <= start_pos + i when causal -- the reference's tiled attention
// (attention_head256_f16kv.wgsl:72-267 with is_causal, query blocks; CPU
// tiled online softmax run_csl_webgpu_emulator.mjs:646-720).  q is bf16
// [q_len][Hq][128], k/v bf16 [Hkv][kv_stride][128] (the cache layout
// [kv_head][pos][dim]), out f32 or bf16 [q_len][Hq][128].
//
// One workgroup = four or eight waves: 64 or 128 rows (32 or 64 queries of two
// heads that share K and V, of one head where the group is odd), each 32 of
// them to two waves that take one half of the keys each.  Keys are staged in LDS
// in blocks of 64, K by direct loads, V through registers as f16.
// Per wave and key block (32 keys of it):
//   * S^T = K . Q^T on v_mfma_f32_32x32x16_bf16 (bf16 inputs are exact, f32
//     accumulate).  The transposed product puts one query per lane column, so
//     the online softmax needs no cross-lane reductions except one exchange
//     between the two lane halves that hold the same query.
//   * P = exp2(S*scale*log2e - m) in f32 (one fma and one exp per score),
//     rounded to f16, and O^T += V^T . P^T on v_mfma_f32_32x32x16_f16: P's
//     registers are used in place as the B operand (the key order of the
//     product follows the MFMA's D layout; V is read transposed in the same
//     order).  The row sum l adds the same f16 P values (v_dot2_f32_f16).
//   * The running max m is raised (and O, l rescaled) only when some query's
//     block max exceeds it by more than 2^8: P stays <= 256, well inside f16,
//     and the O rescale runs on a few blocks instead of every block.
//   * The causal mask is evaluated only on the blocks that cross the
//     diagonal (or the end of the keys); blocks every query sees fully skip it.
// V in f16 is exact for |v| in [2^-14, 65504]; f16 P keeps the output near 1e-4
// rel-L2, where a bf16 P would sit at ~1e-3.  The two key halves merge their (O,
// m, l) through LDS at the end.
//
// What bounds it: at 2048 queries x 32 / 16 heads, all CUs full, the clock (1.8
// GHz under this load, 2.3 with half of the CUs at work; 2130 cycles per block
// and wave pair in both, of which the matrix cores take 1024 and the vector
// unit about 1300); otherwise the workgroup with the most key blocks.  us, with
// 128 queries of one head per workgroup, every wave reading all keys (32 KB of
// LDS per 32 MFMAs, the LDS port's own rate) and V^T from a pre-pass, in
// brackets, timed in turn: 2048 x 32 / 16 heads 48.6-49.6 (54.6-55.8; alone under
// sustained load 54-56); 2048 x 8 / 8 27-28 (44.6); 1500 after 512 x 4 / 4 24.5
// (43.0); 1100 x 32 / 16 22.9 (34.8); 65 x 4 / 4 6.0 (10.6).  Two tiles of 32 rows to a wave (half of the LDS reads, one wave per
// SIMD) took 55 and 43 on the first two; three blocks of K in flight instead of
// two, or a block's first K operands read before the barrier, changed nothing.
#include "common.h"

#include <math.h>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kD = 128, kBKV = 64;
constexpr float kLazy = 8.0f;  // the running max is raised only past m + 8 (P <= 2^8)
constexpr int kBlock = kBKV * kD * 2;  // bytes of a staged K or V block
constexpr int kKRing = 3, kVRing = 2;
constexpr int kLds = (kKRing + kVRing) * kBlock;
static_assert(8 * 64 * (128 + 8) <= kLds, "the merge's state (eight waves' 64 lanes x 32 floats, m and l) fits the rings");

struct PrefillArgs {
    const uint16_t *q, *k, *v;
    void *out;
    int hq, hkv, q_len, kv_len, kv_stride, start_pos, causal, out_bf16;
    int pair, units, cols;  // heads of a workgroup's tiles 2 c, 2 c + 1 (pair) or c; query units; c's count
    float scale_log2;  // softmax scale * log2(e)
};

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t bf16pair_to_f16pair(uint32_t w) {
    const float2v f = {__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, half2v));
}

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rsrc, void *lds, uint32_t lane_off, uint32_t off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)lds, 16, lane_off, off, 0, 0);
}

// A transposed read of LDS.  (As the access of a restrict parameter: without
// alias information the compiler holds it back until every load to LDS has landed.)
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
__device__ __forceinline__ s16x4 read_tr(lds_s16x4 *__restrict__ p) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16(p); }

// max / sum over the two lane halves that hold the same query
__device__ __forceinline__ float halves_max(float x) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

// At most N vector-memory operations outstanding, no LDS operation, and every
// wave here: what they wrote to LDS can be read.  (Not a fence: that would wait
// for the loads to LDS that are still under way.)
template <int N>
__device__ __forceinline__ void wait_barrier() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | (((N >> 4) & 3) << 14));
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

template <int W>
__global__ __launch_bounds__(64 * W, 8 / W) void attn_prefill_kernel(PrefillArgs a) {
    constexpr int kExchange = W * 64 * 128;  // the merge: the waves' 64 lanes x 32 floats
    constexpr int NP = 16 / W, kStep = kBlock / NP;  // 16-byte loads of a thread per staged block
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, lg = lane >> 5;
    const int qt = wave % (W / 2), kh = wave / (W / 2);
    // the units of the last queries see the most keys: first
    const int col = blockIdx.x % a.cols, unit = a.units - 1 - blockIdx.x / a.cols;
    const int uq = a.pair ? 8 * W : 16 * W;  // queries of a unit
    const int q0 = unit * uq, q_end = min(q0 + uq, a.q_len);
    const int head = a.pair ? 2 * col + (qt & 1) : col, kvh = head / (a.hq / a.hkv);
    const int kv_end = a.causal ? min(a.kv_len, a.start_pos + q_end) : a.kv_len;
    const int nkb = (kv_end + kBKV - 1) / kBKV;
    // this lane's query (column of S^T) and the keys [0, limit) that it sees
    const int qi = q0 + 32 * (a.pair ? qt >> 1 : qt) + lr;
    const int limit = qi < a.q_len && a.causal ? min(a.kv_len, a.start_pos + qi + 1) : kv_end;

    // Q^T operand fragments: Q[qi][h][16 s + 8 lg .. + 8]
    bf16x8 qf[8];
    {
        const uint16_t *qp = a.q + ((size_t)min(qi, a.q_len - 1) * a.hq + head) * kD + 8 * lg;
#pragma unroll
        for (int s = 0; s < 8; ++s) qf[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(qp + 16 * s));
    }

    // K and V of this KV head as buffers: per-lane offsets fixed for the whole
    // loop, the block a scalar; keys past kv_len read as zero (masked).  A row
    // of 16 chunks; place c' of row `key` holds chunk c' ^ (key & 15) of K, c' ^
    // 4 (key & 3) of V, so that the lanes' reads fall on different banks.
    const __amdgpu_buffer_rsrc_t krsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.k + (size_t)kvh * a.kv_stride * kD), (short)0, a.kv_len * (kD * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vrsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.v + (size_t)kvh * a.kv_stride * kD), (short)0, a.kv_len * (kD * 2), 0x00020000);
    // wave w stages rows 4 NP w + 4 i + lane / 16 of K, thread t row 4 W i + t / 16 of V
    uint32_t k_voff[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int key = 4 * NP * wave + 4 * i + (lane >> 4);
        k_voff[i] = (uint32_t)(key * 256 + (((lane & 15) ^ (key & 15)) * 16));
    }
    const uint32_t v_voff = (uint32_t)tid * 16u;  // + kStep i
    const uint32_t v_lds = (uint32_t)((tid >> 4) * 256 + ((tid & 15) ^ (4 * ((tid >> 4) & 3))) * 16);  // + kStep i
    auto load_k = [&](int kb, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NP; ++i)
            load_lds16(krsrc, lds + slot * kBlock + (NP * wave + i) * 1024, k_voff[i],
                       (uint32_t)min(kb, nkb - 1) * (uint32_t)kBlock);
    };
    u32x4 rv[NP];
    auto load_v = [&](int i, int kb) __attribute__((always_inline)) {
        rv[i] = __builtin_amdgcn_raw_buffer_load_b128(vrsrc, v_voff + (uint32_t)(i * kStep),
                                                      (uint32_t)min(kb, nkb - 1) * (uint32_t)kBlock, 0);
    };
    auto convert_v = [&](int i, int part) __attribute__((always_inline)) {
        rv[i][2 * part] = bf16pair_to_f16pair(rv[i][2 * part]);
        rv[i][2 * part + 1] = bf16pair_to_f16pair(rv[i][2 * part + 1]);
    };
    auto store_v = [&](int i, int slot) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4 *>(lds + (kKRing + slot) * kBlock + v_lds + i * kStep) = rv[i];
    };
    // K operand s: key 32 kh + lr, dims 16 s + 8 lg (chunk 2 s + lg)
    const uint32_t k_off = (uint32_t)((32 * kh + lr) * 256 + ((lg ^ (lr & 15)) * 16));
    auto kfrag = [&](int s, uint32_t slot_off) __attribute__((always_inline)) {
        return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(lds + ((k_off ^ (uint32_t)(32 * s)) + slot_off)));
    };
    // V^T operand of dims 32 t .., step st: keys 32 kh + 16 st + 4 lg + 0..3 and
    // + 8, dim 32 t + lr; a lane's address is that of a quad of one key's dims
    uint32_t va[4];
    {
        const int key = 4 * lg + ((lane >> 2) & 3), c0 = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            va[t] = (uint32_t)(kKRing * kBlock + (32 * kh + key) * 256 + ((c0 + 4 * t) ^ (4 * (key & 3))) * 16 + (lane & 1) * 8);
    }
    auto vfrag = [&](int t, int st, uint32_t slot_off) __attribute__((always_inline)) {
        const uint8_t *p = lds + (va[t] + slot_off) + st * 4096;
        const s16x4 v0 = read_tr((lds_s16x4 *)p), v1 = read_tr((lds_s16x4 *)(p + 2048));
        return __builtin_bit_cast(half8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    const float16v zero = {0.0f};
    float16v o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = zero;
    float m_i = -INFINITY, l_i = 0.0f, bmax = -INFINITY;
    // key blocks [0, nkb_full) hold only keys that every query of the workgroup sees
    const int nkb_full = min(nkb, (a.causal ? min(a.kv_len, a.start_pos + q0 + 1) : a.kv_len) / kBKV);
    const half2v ones = {(_Float16)1.0f, (_Float16)1.0f};
    // score r: key 32 kh + (r % 4) + 8 (r / 4) + 4 lg of the block
    auto masked = [&](float x, int r, int kb) __attribute__((always_inline)) {
        return kb * kBKV + 32 * kh + (r & 3) + 8 * (r >> 2) + 4 * lg < limit ? x : -INFINITY;
    };

    // Prologue: K(0 .. 2) and V(0), V(1) are loaded, V(0) converted, S(0) formed
    load_k(0, 0);
#pragma unroll
    for (int i = 0; i < NP; ++i) load_v(i, 0);
    load_k(1, 1);
    load_k(2, 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        convert_v(i, 0);
        convert_v(i, 1);
        store_v(i, 0);
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) load_v(i, 1);
    wait_barrier<3 * NP>();
    float16v sa, sb;
#pragma unroll
    for (int s = 0; s < 8; ++s)
        sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfrag(s, 0), qf[s], s ? sa : zero, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (nkb_full == 0) sa[r] = masked(sa[r], r, 0);
        bmax = fmaxf(bmax, sa[r]);
    }
    bmax = halves_max(bmax);
    wait_barrier<2 * NP>();  // K(1) has landed; every wave has read K(0)

    // Iteration kb: sc holds block kb's scores, sn receives block kb + 1's (mode
    // 0: none of them masked, 1: masked, 2: there is none).  At its start K(kb +
    // 1) and V(kb) are in LDS, K(kb + 2) and V(kb + 1) under way; it issues K(kb
    // + 3) and, as V(kb + 1)'s registers come free, V(kb + 2) (past the last: the
    // last again, never used).  A wave issues in order: what the vector unit does
    // is dealt out between the MFMAs, each step its own scheduling region.
    uint32_t ks_next = kBlock;  // K(kb + 1)'s place in the ring
    int ks_load = 0;            // K(kb + 3)'s
    auto iter = [&](const int kb, const int mode, float16v &sc, float16v &sn) __attribute__((always_inline)) {
        const uint32_t vs = (uint32_t)(kb & 1) * kBlock;
        bf16x8 kf[4];
        if (mode != 2) {
#pragma unroll
            for (int s = 0; s < 3; ++s) kf[s] = kfrag(s, ks_next);
            load_k(kb + 3, ks_load);
        }
        const float mb = bmax * a.scale_log2;
        if (__builtin_amdgcn_ballot_w64(mb > m_i + kLazy) != 0) {  // wave-uniform
            const float m_new = fmaxf(m_i, mb);
            const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_i - m_new);
            m_i = m_new;
            l_i *= alpha;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
        }
        const float nm = m_i == -INFINITY ? 0.0f : -m_i;
        // Score pair p (step p / 4 of P V): its exp2s are issued in one step and
        // converted and summed in the next, so that nothing waits on a
        // just-issued transcendental (the wave issues in order).
        half8 pf[2];
        float pp0 = 0.0f, pp1 = 0.0f;
        auto finish_pair = [&](int p) __attribute__((always_inline)) {
            const half2v h = __builtin_convertvector((float2v{pp0, pp1}), half2v);
            l_i = __builtin_amdgcn_fdot2(h, ones, l_i, false);
            pf[p >> 2][2 * (p & 3)] = h[0];
            pf[p >> 2][2 * (p & 3) + 1] = h[1];
        };
        auto do_pair = [&](int p) __attribute__((always_inline)) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[2 * p], a.scale_log2, nm));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[2 * p + 1], a.scale_log2, nm));
            if (p > 0) finish_pair(p - 1);
            pp0 = p0;
            pp1 = p1;
        };
        constexpr int kEarly = 5;  // pairs under Q K; the other three under P V's first step
        half8 vf[4];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (mode != 2) {
                sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[i & 3], qf[i], i ? sn : zero, 0, 0, 0);
                if (i + 3 < 8) kf[(i + 3) & 3] = kfrag(i + 3, ks_next);
            }
            if (i >= 5) vf[i - 5] = vfrag(i - 5, 0, vs);
#pragma unroll
            for (int p = i * kEarly / 8; p < (i + 1) * kEarly / 8; ++p) do_pair(p);
            if (mode != 2) __builtin_amdgcn_sched_barrier(0);
        }
        float bm[2] = {-INFINITY, -INFINITY};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {  // step i / 4, dims 32 (i % 4)
            o[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i & 3], pf[i >> 2], o[i & 3], 0, 0, 0);
            if (i + 3 < 8) vf[(i + 3) & 3] = vfrag((i + 3) & 3, (i + 3) >> 2, vs);
            if (i < 8 - kEarly) do_pair(kEarly + i);
            if (i == 8 - kEarly) finish_pair(7);
            if (mode != 2 && i >= 4) {  // V(kb + 1), and the next block's mask and max
                constexpr int kPer = 4 / NP;  // PV steps per piece
                const int c = (i - 4) / kPer;
#pragma unroll
                for (int part = 0; part < 2 / kPer; ++part) convert_v(c, kPer == 2 ? i & 1 : part);
                if ((i - 4) % kPer == kPer - 1) {
                    store_v(c, (kb + 1) & 1);
                    load_v(c, kb + 2);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * (i - 4) + e;
                    if (mode == 1) sn[r] = masked(sn[r], r, kb + 1);
                    bm[e & 1] = fmaxf(bm[e & 1], sn[r]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (mode != 2) {
            bmax = halves_max(fmaxf(bm[0], bm[1]));
            ks_next = ks_next == (kKRing - 1) * kBlock ? 0 : ks_next + kBlock;
            ks_load = ks_load == kKRing - 1 ? 0 : ks_load + 1;
            wait_barrier<2 * NP>();  // K(kb + 2) has landed, V(kb + 1) is written
        }
    };
    int kb = 0;
    for (; kb + 2 < nkb_full; kb += 2) {  // two iterations whose next blocks need no mask
        iter(kb, 0, sa, sb);
        iter(kb + 1, 0, sb, sa);
    }
    for (; kb + 2 < nkb; kb += 2) {  // (a mask on blocks that every query sees is a no-op)
        iter(kb, 1, sa, sb);
        iter(kb + 1, 1, sb, sa);
    }
    if (kb + 1 < nkb) {
        iter(kb, 1, sa, sb);
        iter(kb + 1, 2, sb, sa);
    } else {
        iter(kb, 2, sa, sb);
    }

    // Merge: the waves of the two key halves (w, w ^ (W / 2)) hold the same queries; each
    // passes its lanes' sums of the other's half of the dims on
    wait_barrier<0>();  // every wave is done with the rings, every load has landed
    const float l = halves_sum(l_i);
    float4 *xo = reinterpret_cast<float4 *>(lds);
    float2 *xm = reinterpret_cast<float2 *>(lds + kExchange);
    auto finish = [&](const int t0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float16v &ot = o[(2 - t0) + (i >> 2)];
            const int g = 4 * (i & 3);
            xo[(wave * 8 + i) * 64 + lane] = make_float4(ot[g], ot[g + 1], ot[g + 2], ot[g + 3]);
        }
        xm[wave * 64 + lane] = make_float2(m_i, l);
        wait_barrier<0>();
        const float2 p = xm[(wave ^ (W / 2)) * 64 + lane];
        const float M = fmaxf(m_i, p.x);
        const float f0 = m_i == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_i - M);
        const float f1 = p.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(p.x - M);
        const float lt = l * f0 + p.y * f1;
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        const float i0 = f0 * inv, i1 = f1 * inv;
        if (qi >= a.q_len) return;
        const size_t obase = ((size_t)qi * a.hq + head) * kD;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float16v &ot = o[t0 + (i >> 2)];
            const int g = 4 * (i & 3), d0 = 32 * (t0 + (i >> 2)) + 8 * (i & 3) + 4 * lg;
            const float4 w = xo[((wave ^ (W / 2)) * 8 + i) * 64 + lane];
            const float v0 = ot[g] * i0 + w.x * i1, v1 = ot[g + 1] * i0 + w.y * i1;
            const float v2 = ot[g + 2] * i0 + w.z * i1, v3 = ot[g + 3] * i0 + w.w * i1;
            if (a.out_bf16) {
                const u32x2 b = {(uint32_t)f32_to_bf16_rne(v0) | ((uint32_t)f32_to_bf16_rne(v1) << 16),
                                 (uint32_t)f32_to_bf16_rne(v2) | ((uint32_t)f32_to_bf16_rne(v3) << 16)};
                *reinterpret_cast<u32x2 *>(reinterpret_cast<uint16_t *>(a.out) + obase + d0) = b;
            } else {
                *reinterpret_cast<float4 *>(reinterpret_cast<float *>(a.out) + obase + d0) = make_float4(v0, v1, v2, v3);
            }
        }
    };
    if (kh == 0)
        finish(0);
    else
        finish(2);
}

int g_num_cus = 0;

template <int W>
int launch(const PrefillArgs &a, int64_t blocks, hipStream_t st) {
    static const hipError_t attr_rc = hipFuncSetAttribute((const void *)attn_prefill_kernel<W>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    DOE_HIP_CHECK(attr_rc);
    hipLaunchKernelGGL((attn_prefill_kernel<W>), dim3((unsigned)blocks), dim3(64 * W), kLds, st, a);
    DOE_LAUNCH_CHECK("attn_prefill_kernel");
    return DOE_OK;
}

}  // namespace

extern "C" {

int doe_attn_prefill(const uint16_t *q, const uint16_t *k, const uint16_t *v, void *out, int out_bf16,
                     int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t q_len,
                     int64_t kv_len, int64_t kv_stride, int64_t start_pos, float scale, int causal,
                     doe_stream_t stream) {
    int rc = doe::require_init();
    if (rc) return rc;
    DOE_REQUIRE(num_heads > 0 && num_kv_heads > 0 && q_len >= 0 && kv_len >= 0 && start_pos >= 0,
                DOE_E_INVALID, "bad prefill attention shape");
    DOE_REQUIRE(num_heads % num_kv_heads == 0, DOE_E_INVALID,
                "num_heads %lld is not a multiple of num_kv_heads %lld", (long long)num_heads,
                (long long)num_kv_heads);
    DOE_REQUIRE(head_dim == kD, DOE_E_UNSUPPORTED, "prefill attention supports head_dim 128 (got %lld)",
                (long long)head_dim);
    DOE_REQUIRE(kv_stride >= kv_len, DOE_E_INVALID, "kv_stride %lld < kv_len %lld", (long long)kv_stride,
                (long long)kv_len);
    DOE_REQUIRE(num_heads <= 4096 && q_len <= (1 << 24) && kv_stride <= (1 << 24) && kv_len <= (1 << 22) &&
                    num_kv_heads * kv_stride * kD <= ((int64_t)1 << 40),
                DOE_E_UNSUPPORTED, "prefill attention shape too large");
    if (q_len == 0) return DOE_OK;
    DOE_REQUIRE(q && out && (kv_len == 0 || (k && v)), DOE_E_INVALID, "null pointer");
    DOE_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) == 0, DOE_E_INVALID,
                "q, k, v and out must be 16-byte aligned");
    PrefillArgs a;
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.hq = (int)num_heads;
    a.hkv = (int)num_kv_heads;
    a.q_len = (int)q_len;
    a.kv_len = (int)kv_len;
    a.kv_stride = (int)kv_stride;
    a.start_pos = (int)start_pos;
    a.causal = causal ? 1 : 0;
    a.out_bf16 = out_bf16 ? 1 : 0;
    a.pair = (num_heads / num_kv_heads) % 2 == 0;
    a.cols = (int)(a.pair ? num_heads / 2 : num_heads);
    const int64_t rows = a.pair ? 2 * q_len : q_len;  // of a column
    if (g_num_cus == 0) {
        int dev = 0, cus = 0;
        DOE_HIP_CHECK(hipGetDevice(&dev));
        DOE_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        g_num_cus = cus > 0 ? cus : 256;
    }
    // Eight waves once the four-wave workgroups (two per CU) come to well over one
    // round, two and a half per CU: half of the staging, which then counts (704 of
    // them 30.3 against 32.7 us, 1024 56 against 60, back to back); up to there
    // four: more, shorter workgroups (560: 23.1 against 24.6; 512: 36.7 against
    // 39.5; 96: 24 against 33)
    const bool wide = (rows + 63) / 64 * a.cols * 2 > 5 * (int64_t)g_num_cus;
    a.units = (int)(wide ? (rows + 127) / 128 : (rows + 63) / 64);
    a.scale_log2 = scale * 1.4426950408889634f;
    hipStream_t st = (hipStream_t)stream;
    if (kv_len == 0) {
        // no keys: the empty softmax contributes nothing (zero output)
        const size_t bytes = (size_t)q_len * num_heads * kD * (out_bf16 ? 2 : 4);
        return doe::fill_bytes_async(out, 0, bytes, st);
    }
    const int64_t blocks = (int64_t)a.units * a.cols;
    DOE_REQUIRE(blocks <= 0x7fffffff, DOE_E_UNSUPPORTED, "too many blocks");
    return wide ? launch<8>(a, blocks, st) : launch<4>(a, blocks, st);
}

}  // extern "C"
