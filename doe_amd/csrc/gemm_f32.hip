// gemm_f32.hip -- f32-accurate GEMM over quantized rows for f32 activations:
// the decoder's batched prompt (C[m][n] = sum_k A[m][k] dequant(B)[n][k], B
// Q4_K_M or Q8_0 rows) on v_mfma_f32_32x32x16_f16.
//
// Numerics.  A is scaled per row by a power of two (max just under 2^14) and
// carried as f16 hi + lo (~22 bits).  B goes to the matrix cores as the
// integers it is stored as, exact in f16, so two products per step (a_hi b,
// a_lo b) carry the full accuracy; the block scales are applied to the f32
// sums afterwards:
//   * Q4_K: b = sc q - z (|b| < 2048), z the integer next to a sub-block's
//     dmin m / d.  A 256-element block's sum is d sum(b x) + sum_s r_s sum(x of
//     sub-block s), r = d z - dmin m: two more MFMAs per block, A's sub-block
//     sums (f16 hi + lo, eight of each) against r as f16 hi + lo.  b d is the
//     weight up to r, and |r| at most d: neither sum is larger than the
//     result's own terms.  (With b = sc q and the minima in the second sum the
//     two cancel wherever the activations of a row have a common sign.)
//   * Q8_0: b = q (int8); a 32-element block's sum is d sum(q x).
// Measured, rows of A with mean 0 to 30 deviations or after ReLU, minima tied to
// the scales or not, K 2304 to 13000: Q4_K 1.3-1.8e-7 from float64, Q8_0
// 1.1-1.7e-7.  (Splitting the dequantised f32 weight into f16 hi + lo instead
// takes a third product per step and ~6 VALU operations per weight instead of
// 1.1, and gives 1.9-3.7e-7; b = sc q takes 4 % less time here, and gives
// 3.2e-7, with a mean 1.4-3.0e-6.)
//
// Layout.  The pre-pass writes A in operand order: per 32 rows and 32
// elements of K four 1 KB fragments (step 0 hi, lo, step 1 hi, lo), each the
// 64 lanes' 16 bytes in lane order, so a fragment goes to LDS by one
// global_load_lds_dwordx4 and is read back by one conflict-free b128.  K is
// permuted inside a 32-element sub-block to what a nibble dword unpacks to
// with one AND per two weights: lane half h holds bytes 16 h .. 16 h + 15,
// step t the dwords 2 t and 2 t + 1 of them, each as bytes 0, 2, 1, 3.
//
// Tiling.  Four waves side by side in N, tiles of 128 x 128 or 64 x 128: every
// wave dequantises its own 32 columns once for all the tile's rows.  K runs in
// sub-blocks of 32 through a four-deep LDS ring of A (two workgroups per CU),
// loaded three stages ahead; per stage and wave of a 128-row tile 16
// MFMAs (512 cycles), 16 fragment reads and ~25 VALU operations.
// Measured (us per call, pre-pass and second pass included; the three-product
// kernel with per-workgroup dequantisation that this replaced in brackets):
// Q4_K GeGLU 1000 x 18432 x 2304 189 (391-398; matrix cores busy 56 % of the
// kernel's cycles, the clock down to 1.7 GHz under them), Q8_0 333 x 2304 x 9216
// 61-63 (83); 128-token calls are bound by the one or two waves per SIMD that a
// short prompt gives.
#include "gemm_f32.h"

#include <math.h>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));  // rows of any float address
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kGroupM = 8;
constexpr int kBufFlags = 0x00020000;  // raw buffer, 32-bit data format
constexpr int kSubUnits = 256;  // 16-byte units of a 32-row x 32-element piece of A: four fragments

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }

// ---------------------------------------------------------------------------
// Pre-pass: A f32 [M][K] -> fragments, optionally through RMSNorm first (bit
// for bit the rmsnorm op: the same per-thread sums of squares over k = t, t +
// 256, ..., the same four-wave sum, inv = 1 / sqrt(ss / K + eps), y = x * inv
// * (w or 1 + w)).  One workgroup per row; a thread holds its G granules of
// eight elements (K <= 2048 G) in registers, loaded at once, so the row costs
// one memory round trip (two with the norm's second order of the row, in
// flight together); G = 0 re-reads the row.  Four neighbouring rows share
// 64-byte lines of the fragments, so four workgroups of one XCD (id mod 8)
// take four consecutive rows.
// ---------------------------------------------------------------------------
template <int G, bool NORM, bool SUMS>
__global__ __launch_bounds__(256) void a_fragments_kernel(const float *__restrict__ a, const float *__restrict__ w,
                                                          float eps, int weight_offset, u32x4 *__restrict__ frag,
                                                          _Float16 *__restrict__ sums, int *__restrict__ sig, int M,
                                                          int K, int nsub) {
    const int m = ((((int)blockIdx.x >> 5) << 3) + (blockIdx.x & 7)) * 4 + (((int)blockIdx.x >> 3) & 3);
    if (m >= M) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const float *row = a + (size_t)m * K;
    __shared__ float sh[4];
    __shared__ float shmax[4];
    // granule g: the elements 8 g .. 8 g + 7 (zero past K)
    auto load = [&](const float *p, int g, float (&v)[8]) __attribute__((always_inline)) {
        const int k0 = 8 * g;
        if (k0 + 8 <= K) {
            const f32x4 v0 = *reinterpret_cast<const f32x4 *>(p + k0);
            const f32x4 v1 = *reinterpret_cast<const f32x4 *>(p + k0 + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = v0[e];
                v[4 + e] = v1[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = k0 + e < K ? p[k0 + e] : 0.0f;
        }
    };
    float x[G > 0 ? G : 1][8], nw[G > 0 && NORM ? G : 1][8];
#pragma unroll
    for (int i = 0; i < G; ++i) {
        load(row, t + 256 * i, x[i]);
        if (NORM) load(w, t + 256 * i, nw[NORM ? i : 0]);
    }
    float inv = 1.0f;
    if (NORM) {
        float ss = 0.0f;
        if (G > 0) {
            float xv[G > 0 ? 8 * G : 1];
#pragma unroll
            for (int j = 0; j < 8 * G; ++j) xv[j] = t + 256 * j < K ? row[t + 256 * j] : 0.0f;
#pragma unroll
            for (int j = 0; j < 8 * G; ++j)
                if (t + 256 * j < K) ss = fmaf(xv[j], xv[j], ss);
        } else {
            for (int k = t; k < K; k += 256) ss = fmaf(row[k], row[k], ss);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
        if (lane == 0) sh[wave] = ss;
        __syncthreads();
        float tot = 0.0f;
        for (int j = 0; j < 4; ++j) tot += sh[j];
        inv = 1.0f / sqrtf(tot / (float)K + eps);
    }
    auto normed = [&](float (&v)[8], const float (&wv)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = NORM ? v[e] * inv * (weight_offset ? 1.0f + wv[e] : wv[e]) : v[e];
    };
    float amax = 0.0f;
    auto grow = [&](const float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[e]));
    };
    if (G > 0) {
#pragma unroll
        for (int i = 0; i < G; ++i) {
            normed(x[i], nw[NORM ? i : 0]);
            grow(x[i]);
        }
    } else {
        for (int g = t; 8 * g < K; g += 256) {
            float v[8], wv[8];
            load(row, g, v);
            if (NORM) load(w, g, wv);
            normed(v, wv);
            grow(v);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    if (lane == 0) shmax[wave] = amax;
    __syncthreads();
    const float mx = fmaxf(fmaxf(shmax[0], shmax[1]), fmaxf(shmax[2], shmax[3]));
    int s = 0;
    if (mx > 0.0f && mx <= 3.0e38f) {
        s = 14 - __builtin_amdgcn_frexp_expf(mx);
        s = s < -120 ? -120 : (s > 120 ? 120 : s);
    }
    if (t == 0) sig[m] = s;
    const float scale = __builtin_amdgcn_ldexpf(1.0f, s);

    // granule g = sub-block g / 4, lane half (g / 2) % 2, step g % 2
    u32x4 *ftile = frag + (size_t)(m >> 5) * nsub * kSubUnits + (m & 31);
    auto store = [&](int g, const float (&x8)[8]) __attribute__((always_inline)) {
        constexpr int kOrder[8] = {0, 2, 1, 3, 4, 6, 5, 7};
        float v[8];
        half8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = x8[e] * scale;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            hi[e] = (_Float16)v[kOrder[e]];
            lo[e] = (_Float16)(v[kOrder[e]] - (float)hi[e]);
        }
        const int sub = g >> 2, h = (g >> 1) & 1, step = g & 1;
        u32x4 *dst = ftile + (size_t)sub * kSubUnits + step * 128 + 32 * h;
        dst[0] = __builtin_bit_cast(u32x4, hi);
        dst[64] = __builtin_bit_cast(u32x4, lo);
        if (SUMS) {
            // x / 64 keeps a sub-block's sum below 2^13; the minima carry the 64
            float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            sum += __shfl_xor(sum, 1, 64);
            sum += __shfl_xor(sum, 2, 64);
            sum *= 0.015625f;
            if ((g & 3) == 0) {
                const _Float16 top = (_Float16)sum;
                _Float16 *sd = sums + (((size_t)(m >> 5) * (nsub >> 3) + (sub >> 3)) * 64 + (m & 31)) * 8 + (sub & 7);
                sd[0] = top;
                sd[32 * 8] = (_Float16)(sum - (float)top);
            }
        }
    };
    if (G > 0) {
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (t + 256 * i < nsub * 4) store(t + 256 * i, x[i]);
    } else {
        for (int g = t; g < nsub * 4; g += 256) {
            float v[8], wv[8];
            load(row, g, v);
            if (NORM) load(w, g, wv);
            normed(v, wv);
            store(g, v);
        }
    }
}

struct XArgs {
    const u32x4 *frag;  // A's fragments [M / 32][nsub][4][64]
    const u32x4 *sums;  // Q4_K: the sub-block sums' fragments [M / 32][nsub / 8][64]
    const int *sig;
    const uint8_t *b;
    float *c, *part;
    const float *res;
    int M, N, nb, nsub, tiles_m, tiles_n, splits, nchunk, cps, pairs;
};

// Waits until at most N of the wave's vector-memory operations and L of its LDS
// operations are outstanding, then the workgroup's barrier.  (A release fence
// in its place waits for every load to LDS; the empty asm statements keep
// memory operations on their side.)
template <int N, int L>
__device__ __forceinline__ void wait_barrier() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (L << 8) | (((N >> 4) & 3) << 14));
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}
// One 16-byte piece per lane, voff + soff bytes into the buffer, to LDS at
// dst + 16 lane (dst the same in every lane).
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rsrc, void *dst, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)dst, 16, voff, soff, 0, 0);
}

// Eight f16 operands (sc q - z) 2^-14 from two nibble dwords: a nibble in bits
// 0..3 of a half is the subnormal q 2^-24 (scale sc 2^10), in bits 4..7 q 2^-20
// (scale sc 2^6); nz is -z 2^-14, every result is exact.
template <bool HIGH>
__device__ __forceinline__ half8 q4_operands(uint32_t w0, uint32_t w1, half2v sc, half2v nz) {
    constexpr uint32_t mask = HIGH ? 0x00f000f0u : 0x000f000fu;
    auto two = [&](uint32_t w) { return as_u32(__builtin_elementwise_fma(as_h2(w & mask), sc, nz)); };
    return __builtin_bit_cast(half8, u32x4{two(w0), two(w0 >> 8), two(w1), two(w1 >> 8)});
}
// The 6-bit scales or minima of sub-blocks 2 c and 2 c + 1, from the two dwords of all eight.
__device__ __forceinline__ half2v six_pair(const uint32_t (&v)[2], int c) {
    const half2v k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    return as_h2(__builtin_amdgcn_perm(0x64646464u, v[c >> 1], c & 1 ? 0x04030402u : 0x04010400u)) - k1024;
}
// Eight f16 operands q from two dwords of int8 (1024 + (q + 128) - 1152).
__device__ __forceinline__ half8 q8_operands(uint32_t w0, uint32_t w1) {
    const half2v bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t x0 = w0 ^ 0x80808080u, x1 = w1 ^ 0x80808080u;
    const uint32_t u[4] = {as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, x0, 0x04020400u)) - bias),
                           as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, x0, 0x04030401u)) - bias),
                           as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, x1, 0x04020400u)) - bias),
                           as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, x1, 0x04030401u)) - bias)};
    return __builtin_bit_cast(half8, u32x4{u[0], u[1], u[2], u[3]});
}

// Four waves side by side in N, each 32 TM rows x 32 columns.  LDS: A, a ring
// of four 32-element sub-blocks; B, a ring of three 64-element chunks of
// nibbles and two block headers per row, or two chunks of quants.  TM 4: 80 KB,
// two workgroups per CU; TM 2: 48 KB (there the registers allow two).
template <int FMT, int TM>
struct XTile {
    static constexpr int BM = 32 * TM, BN = 128;
    static constexpr int kA = TM * 4096, kB = (FMT == 0 ? 2 : 4) * BN * 16;
    static constexpr int kBq = 4 * kA, kBh = kBq + (FMT == 0 ? 3 : 2) * kB, kBytes = kBh + (FMT == 0 ? 2 * BN * 16 : 0);
};

// Q4_K: the loads a wave issues in stage u of a block: a fragment of A per
// tile, a chunk of B at even stages, tile u's sums in the first TM, a header at 2.
template <int TM>
constexpr int q4_loads(int u) {
    return TM + (u % 2 == 0) + (u < TM) + (u == 2);
}

// FMT 0: Q4_K rows; 1: Q8_0 rows.
template <int FMT, int TM>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(XArgs g) {
    using Tl = XTile<FMT, TM>;
    constexpr int BM = Tl::BM, BN = Tl::BN;
    // (one dynamic array: over separate static ones the compiler waits for
    // every load to LDS before any LDS read, the prefetched ones included)
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    auto As = [&](int slot) __attribute__((always_inline)) {  // [32 rows][fragment][lane]
        return reinterpret_cast<u32x4 *>(lds + slot * Tl::kA);
    };
    // Q4_K: 16 of a chunk's 32 nibble bytes [lane half][row]; Q8_0: quants [sub-block][lane half][row]
    auto Bq = [&](int slot, int i) __attribute__((always_inline)) {
        return reinterpret_cast<u32x4 *>(lds + Tl::kBq + slot * Tl::kB) + i * BN;
    };
    auto Bh = [&](int slot) __attribute__((always_inline)) {  // Q4_K block headers
        return reinterpret_cast<u32x4 *>(lds + Tl::kBh) + slot * BN;
    };

    // work order: K split, then an M-grouped raster of tiles; each XCD
    // (workgroup id mod 8) takes a contiguous range, so its resident tiles
    // share A's K range and B in its L2
    const int T = g.tiles_m * g.tiles_n, W = T * g.splits, xcd = blockIdx.x & 7;
    const int work = xcd * (W >> 3) + min(xcd, W & 7) + (int)(blockIdx.x >> 3);
    const int split = work / T, t = work - split * T;
    const int per_group = kGroupM * g.tiles_n;
    const int grp = t / per_group;
    const int first_m = grp * kGroupM;
    const int gsize = min(kGroupM, g.tiles_m - first_m);
    const int within = t - grp * per_group;
    const int m0 = (first_m + within % gsize) * BM, n0 = (within / gsize) * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, lh = lane >> 5;
    const int sig_row = g.sig[min(m0 + min(tid, BM - 1), g.M - 1)];

    // Loads to LDS are buffer loads: the lane's part of the address is fixed,
    // the piece of K a scalar.  A: wave w stages fragments w TM .. + TM - 1 of
    // the sub-block's 4 TM (rows past M read a tile that exists and are never
    // stored)
    const int mtiles = (g.M + 31) >> 5;
    const uint32_t tile_bytes = (uint32_t)g.nsub * 4096u;
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(g.frag + (size_t)(m0 >> 5) * g.nsub * kSubUnits), (short)0,
        (int)((uint32_t)min(TM, mtiles - (m0 >> 5)) * tile_bytes), kBufFlags);
    uint32_t a_off[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int p = wave * TM + i;
        a_off[i] = (uint32_t)min(p >> 2, mtiles - 1 - (m0 >> 5)) * tile_bytes + (uint32_t)(p & 3) * 1024u + 16u * lane;
    }
    auto load_a = [&](int sub, int slot, int i) __attribute__((always_inline)) {
        load_lds16(arsrc, As(slot) + (wave * TM + i) * 64, a_off[i], (uint32_t)sub * 4096u);
    };
    // Q4_K: wave w stages lane half w / 2 of rows 64 (w % 2) .. + 63, and the
    // headers of those rows (two waves write the same bytes)
    const int bhalf = wave >> 1, brow0 = (wave & 1) * 64;
    const uint32_t row_bytes = (uint32_t)g.nb * DOE_Q4K_BLOCK_BYTES;
    const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(g.b + (size_t)n0 * (FMT == 0 ? row_bytes : 0)), (short)0,
        FMT == 0 ? (int)((uint32_t)min(BN, g.N - n0) * row_bytes) : 0, kBufFlags);
    const uint32_t b_off = (uint32_t)min(brow0 + lane, g.N - 1 - n0) * row_bytes;
    auto load_b4 = [&](int kc, int slot) __attribute__((always_inline)) {
        load_lds16(brsrc, Bq(slot, bhalf) + brow0, b_off,
                   (uint32_t)(kc >> 2) * DOE_Q4K_BLOCK_BYTES + 16u + 32u * (kc & 3) + 16u * bhalf);
    };
    auto load_h4 = [&](int blk) __attribute__((always_inline)) {
        load_lds16(brsrc, Bh(blk & 1) + brow0, b_off, (uint32_t)blk * DOE_Q4K_BLOCK_BYTES);
    };
    // Q8_0: thread t holds 16 quants of row t / 2 (half t % 2) of both blocks
    // of a chunk, from the dword-aligned 20-byte window around them; buffer
    // loads over the whole matrix, its size rounded up to a dword (the last
    // quants share one with up to two bytes past the matrix); blocks past the
    // row's end read as zero
    const __amdgpu_buffer_rsrc_t b8 = __builtin_amdgcn_make_buffer_rsrc(
        (void *)g.b, (short)0, FMT == 1 ? (int)(((uint32_t)g.N * (uint32_t)g.nb * 34u + 3u) & ~3u) : 0, kBufFlags);
    const uint32_t b8row = (uint32_t)min(n0 + (tid >> 1), g.N - 1) * (uint32_t)g.nb;
    const uint32_t b8col = (uint32_t)min(n0 + wave * 32 + lr, g.N - 1) * (uint32_t)g.nb;
    struct Q8 {
        u32x4 q[2];
        uint32_t tail[2];
    };
    auto load_b8 = [&](int kc, Q8 &r) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const uint32_t blk = (uint32_t)(2 * kc + s);
            const uint32_t o = blk < (uint32_t)g.nb ? (b8row + blk) * 34u + 2u + 16u * (tid & 1) : 0x80000000u;
            r.q[s] = __builtin_amdgcn_raw_buffer_load_b128(b8, o & ~3u, 0, 0);
            r.tail[s] = __builtin_amdgcn_raw_buffer_load_b32(b8, (o & ~3u) + 16u, 0, 0);
        }
    };
    auto store_b8 = [&](int kc, int slot, const Q8 &r) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            // block offsets are 34 b + 2 + 16 h: the quants start 2 bytes into the window where b is even
            const uint32_t sel = (b8row + (uint32_t)(2 * kc + s)) & 1u ? 0x03020100u : 0x05040302u;
            const u32x4 w = r.q[s];
            Bq(slot, 2 * s + (tid & 1))[tid >> 1] =
                u32x4{__builtin_amdgcn_perm(w.y, w.x, sel), __builtin_amdgcn_perm(w.z, w.y, sel),
                      __builtin_amdgcn_perm(w.w, w.z, sel), __builtin_amdgcn_perm(r.tail[s], w.w, sel)};
        }
    };
    auto load_d8 = [&](int kc, uint32_t (&d)[2]) __attribute__((always_inline)) {  // this lane's column's scales
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const uint32_t blk = (uint32_t)(2 * kc + s);
            d[s] = __builtin_amdgcn_raw_buffer_load_b16(b8, blk < (uint32_t)g.nb ? (b8col + blk) * 34u : 0x80000000u, 0, 0);
        }
    };

    float16v acc[TM], D[TM];
    const float16v zero = {0.0f};
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i] = D[i] = zero;

    const int ncol = wave * 32 + lr;  // this lane's column within the tile
    half8 bf[2];                      // B operands of the stage's two steps
    // A's fragments (step 0 hi, lo, step 1 hi, lo) of the tiles at hand: stage
    // u's tile i in fr[(u TM + i) % 4]
    half8 fr[4][4];
    auto read_tile = [&](int u, int i) __attribute__((always_inline)) {
        const u32x4 *src = As(u & 3) + i * 256 + lane;
#pragma unroll
        for (int j = 0; j < 4; ++j) fr[(u * TM + i) & 3][j] = __builtin_bit_cast(half8, src[j * 64]);
    };
    auto mfma_tile = [&](int u, int i, const half8 (&b)[2], bool fresh) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            D[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[(u * TM + i) & 3][j], b[j >> 1],
                                                          fresh && j == 0 ? zero : D[i], 0, 0, 0);
    };

    // Pipeline.  Stage u (one sub-block of A, in slot u % 4) opens with a
    // barrier by which sub-blocks u and u + 1 have landed and u - 1 has been
    // read by every wave; during it u + 3 is loaded into u - 1's slot, the
    // fragments are read two tiles ahead (the last two of them the next
    // stage's) and the next stage's B operands are formed, so behind a
    // barrier a wave's MFMAs start at once.  A scheduling region per tile
    // holds four MFMAs and its share of all that (left to itself the compiler
    // reads each fragment right before its MFMA).  The barrier waits for all
    // but the loads issued in the stage before, whose number is fixed: past
    // the range's end the loads repeat its last piece, into slots that are
    // not read again or with the bytes they hold.  Of the LDS operations only
    // the eight reads of the next stage's fragments are left outstanding.
    const int kc0 = split * g.cps, kc1 = min(g.nchunk, kc0 + g.cps), s1 = 2 * kc1;
    if constexpr (FMT == 0) {
        const int blk0 = kc0 >> 2, blk1 = kc1 >> 2;
        load_h4(blk0);
#pragma unroll
        for (int c = 0; c < 3; ++c) load_b4(kc0 + c, c);
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
            for (int i = 0; i < TM; ++i) load_a(2 * kc0 + u, u, i);
        const uint32_t sblocks = (uint32_t)g.nsub >> 3;
        const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(g.sums + (size_t)(m0 >> 5) * sblocks * 64), (short)0,
            (int)((uint32_t)min(TM, mtiles - (m0 >> 5)) * sblocks * 1024u), kBufFlags);
        auto load_sums = [&](int i, int blk) __attribute__((always_inline)) {
            return __builtin_amdgcn_raw_buffer_load_b128(
                srsrc, 16u * lane, ((uint32_t)min(i, mtiles - 1 - (m0 >> 5)) * sblocks + (uint32_t)blk) * 1024u, 0);
        };
        half2v sc[4], nz[4];
        u32x4 raw;
        int bslot = 0;  // of the current chunk
        auto next_bslot = [&]() __attribute__((always_inline)) { return bslot == 2 ? 0 : bslot + 1; };
        // part `part` of TM of the operands of stage u of block blk (8: the next block's first)
        auto operands = [&](int blk, int u, int slot, int part) __attribute__((always_inline)) {
            if (part == 0 && (u & 7) == 0) {
                const u32x4 h = Bh((blk + (u >> 3)) & 1)[ncol];
                const uint32_t sc6[2] = {h.y & 0x3f3f3f3fu, (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u)};
                const uint32_t mn6[2] = {h.z & 0x3f3f3f3fu, ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u)};
                const half2v up = {(_Float16)1024.0f, (_Float16)64.0f};
                // z = m dmin / d to an integer in 0..1023 (the sum's ulp is 1; any
                // integer is right, a near one makes r small)
                const _Float16 t = (_Float16)(doe_half_bits_to_float(h.x >> 16) *
                                              __builtin_amdgcn_rcpf(doe_half_bits_to_float(h.x)));
                const half2v lo = {(_Float16)1024.0f, (_Float16)1024.0f}, hi = {(_Float16)2047.0f, (_Float16)2047.0f};
                const half2v s14 = {(_Float16)-0x1p-14f, (_Float16)-0x1p-14f}, k = {(_Float16)0x1p-4f, (_Float16)0x1p-4f};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    sc[c] = six_pair(sc6, c) * up;
                    half2v z = __builtin_elementwise_fma(six_pair(mn6, c), half2v{t, t}, lo);
                    z = __builtin_elementwise_max(__builtin_elementwise_min(z, hi), lo);
                    nz[c] = __builtin_elementwise_fma(z, s14, k);
                }
            }
            if (part == 0 && (u & 1) == 0) raw = Bq(slot, lh)[ncol];
            if (part < TM - 2) return;
            const half2v sv = sc[(u >> 1) & 3], zv = nz[(u >> 1) & 3];
            const int t = part - (TM - 2);  // the last two parts form step 0 and step 1
            const uint32_t w0 = t ? raw.z : raw.x, w1 = t ? raw.w : raw.y;
            bf[t] = u & 1 ? q4_operands<true>(w0, w1, half2v{sv.y, sv.y}, half2v{zv.y, zv.y})
                          : q4_operands<false>(w0, w1, half2v{sv.x, sv.x}, half2v{zv.x, zv.x});
        };
        // a block's sums are scaled as its last MFMAs end, a tile behind
        float dl = 0.0f;
        auto scale_tile = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = fmaf(D[i][r], dl, acc[i][r]);
        };
        // r of the eight sub-blocks 2^(14 - E) (E: the block's largest dmin m and
        // d z are below 2^E), formed a pair at a time in the first stages after the
        // header's; tile i's sums are loaded in stage i and added in stage 3 + i
        uint32_t rh[4], rl[4], mn6[2] = {0, 0};
        float d_up = 0.0f, dmin_up = 0.0f, dm = 0.0f;
        u32x4 sf[3];
        float16v ms = zero;
        auto remainders = [&](int blk, int c) __attribute__((always_inline)) {
            if (c == 0) {
                const u32x4 h = Bh(blk & 1)[ncol];
                mn6[0] = h.z & 0x3f3f3f3fu;
                mn6[1] = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
                const float d = doe_half_bits_to_float(h.x), dmin = doe_half_bits_to_float(h.x >> 16);
                dl = d * 16384.0f;
                const int e = __builtin_amdgcn_frexp_expf(fmaxf(fabsf(d) * 1024.0f, fabsf(dmin) * 64.0f));
                d_up = __builtin_amdgcn_ldexpf(d, 28 - e);  // (nz holds 2^-14)
                dmin_up = __builtin_amdgcn_ldexpf(dmin, 14 - e);
                dm = __builtin_amdgcn_ldexpf(1.0f, e - 8);  // (the sums hold 2^-6)
            }
            const half2v m = six_pair(mn6, c);
            half2v top, low;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float r = -fmaf((float)nz[c][j], d_up, (float)m[j] * dmin_up);
                top[j] = (_Float16)r;
                low[j] = (_Float16)(r - (float)top[j]);
            }
            rh[c] = as_u32(top);
            rl[c] = as_u32(low);
        };
        wait_barrier<2 * TM, 0>();
#pragma unroll
        for (int i = 0; i < TM; ++i) operands(blk0, 0, 0, i);
        read_tile(0, 0);
        read_tile(0, 1);
        for (int blk = blk0; blk < blk1; ++blk) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int kc = 4 * blk + (u >> 1), s = 8 * blk + u;
                __builtin_amdgcn_sched_barrier(0);
                switch (u) {
                    case 0: case 6: wait_barrier<q4_loads<TM>(7), 8>(); break;
                    case 1: wait_barrier<q4_loads<TM>(0), 8>(); break;
                    case 2: wait_barrier<q4_loads<TM>(1), 8>(); break;
                    case 3: wait_barrier<q4_loads<TM>(2), 8>(); break;
                    case 4: wait_barrier<q4_loads<TM>(3), 8>(); break;
                    default: wait_barrier<q4_loads<TM>(4), 8>(); break;
                }
                const half8 cur[2] = {bf[0], bf[1]};
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    __builtin_amdgcn_sched_barrier(0);
                    load_a(min(s + 3, s1 - 1), (u + 3) & 3, i);
                    if (i == 0 && (u & 1) == 0) load_b4(min(kc + 3, kc1 - 1), bslot);
                    if (i == 1 && u == 2) load_h4(min(blk + 1, blk1 - 1));
                    if (i == TM - 1 && u < TM) sf[u % 3] = load_sums(u, blk);
                    read_tile(u + (i + 2) / TM, (i + 2) % TM);
                    if (u == 0 && i == 0) scale_tile(TM - 1);
                    if (u == 7 && i > 0) scale_tile(i - 1);
                    mfma_tile(u, i, cur, u == 0);
                    if (u >= 1 && (u - 1) * TM + i < 4) remainders(blk, (u - 1) * TM + i);
                    if (u >= 3 && u < 3 + TM) {
                        const half8 x = __builtin_bit_cast(half8, sf[u % 3]);
                        if (i == 0) {
                            ms = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                x, __builtin_bit_cast(half8, u32x4{rh[0], rh[1], rh[2], rh[3]}), zero, 0, 0, 0);
                            ms = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                x, __builtin_bit_cast(half8, u32x4{rl[0], rl[1], rl[2], rl[3]}), ms, 0, 0, 0);
                        } else if (i == TM / 2) {
#pragma unroll
                            for (int r = 0; r < 16; ++r) acc[u - 3][r] = fmaf(ms[r], dm, acc[u - 3][r]);
                        }
                    }
                    operands(blk, u + 1, next_bslot(), i);
                }
                if (u & 1) bslot = next_bslot();
            }
        }
        scale_tile(TM - 1);
    } else {
        // quants: one chunk ahead in LDS, two more in registers
        Q8 q[2];
        uint32_t dq[2][2];
        u32x4 raw;
        load_b8(kc0, q[0]);
        load_b8(kc0 + 1, q[1]);
        load_d8(kc0, dq[0]);
        load_d8(kc0 + 1, dq[1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TM; ++i) load_a(2 * kc0, 0, i);
        store_b8(kc0, 0, q[0]);
        load_b8(kc0 + 2, q[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 1; u < 3; ++u)
#pragma unroll
            for (int i = 0; i < TM; ++i) load_a(min(2 * kc0 + u, s1 - 1), u, i);
        auto operands = [&](int slot, int sub, int part) __attribute__((always_inline)) {
            if (part == 0) raw = Bq(slot, 2 * sub + lh)[ncol];
            if (part < TM - 2) return;
            const int t = part - (TM - 2);
            bf[t] = t ? q8_operands(raw.z, raw.w) : q8_operands(raw.x, raw.y);
        };
        wait_barrier<2 * TM, 0>();
#pragma unroll
        for (int i = 0; i < TM; ++i) operands(0, 0, i);
        read_tile(0, 0);
        read_tile(0, 1);
        float dprev = 0.0f;
        auto chunk = [&](int kc, int p) __attribute__((always_inline)) {  // p = (kc - kc0) % 2
            const float d[2] = {doe_half_bits_to_float(dq[p][0]), doe_half_bits_to_float(dq[p][1])};
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const int u = 2 * p + v, s = 2 * kc + v;
                __builtin_amdgcn_sched_barrier(0);
                // the stage before: A, with v = 1 also four loads of quants and two of scales
                if (v == 0) wait_barrier<TM, 8>();
                else wait_barrier<TM + 6, 8>();
                const half8 cur[2] = {bf[0], bf[1]};
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (v == 0 && i == 0) {
                        store_b8(kc + 1, p ^ 1, q[p ^ 1]);
                        load_b8(kc + 3, q[p ^ 1]);
                        load_d8(kc + 2, dq[p]);
                    }
                    load_a(min(s + 3, s1 - 1), (u + 3) & 3, i);
                    read_tile(u + (i + 2) / TM, (i + 2) % TM);
                    // a tile's sums are scaled a tile behind
                    const int last = i ? i - 1 : TM - 1;
                    const float dd = i ? d[v] : dprev;
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[last][r] = fmaf(D[last][r], dd, acc[last][r]);
                    mfma_tile(u, i, cur, true);
                    operands(v ? p ^ 1 : p, v ^ 1, i);
                }
                dprev = d[v];
            }
        };
        for (int kc = kc0; kc < kc1; kc += 2) {
            chunk(kc, 0);
            if (kc + 1 < kc1) chunk(kc + 1, 1);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[TM - 1][r] = fmaf(D[TM - 1][r], dprev, acc[TM - 1][r]);
    }

    // the repeated loads land and every wave has read its fragments: the
    // rows' unscaling factors take their place
    wait_barrier<0, 0>();
    float *rowscale = reinterpret_cast<float *>(lds);
    if (tid < BM) rowscale[tid] = __builtin_amdgcn_ldexpf(1.0f, -sig_row);
    wait_barrier<0, 0>();

    // D lane l, r: row (r % 4) + 8 (r / 4) + 4 (l / 32), column l % 32
    const bool parts = g.splits > 1;
    float *cout = parts ? g.part + (size_t)split * g.M * g.N : g.c;
    const int n = n0 + ncol;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int mb = 32 * i + 4 * lh;
        if (!parts && g.pairs) {
            // gate and up columns sit in neighbouring lanes: an even lane takes
            // rows r of the pair, an odd one rows r + 8
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int r0 = mb + (r & 3) + 8 * (r >> 2);
                const float v0 = acc[i][r] * rowscale[r0], v1 = acc[i][r + 8] * rowscale[r0 + 16];
                const float p0 = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v0), 0xB1, 0xf, 0xf, false));
                const float p1 = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v1), 0xB1, 0xf, 0xf, false));
                const float gate = lane & 1 ? p1 : v0, up = lane & 1 ? v1 : p0;
                const int m = m0 + r0 + 16 * (lane & 1);
                if (m < g.M && n < g.N) cout[(size_t)m * (g.N >> 1) + (n >> 1)] = doe_gelu_tanh_clamped(gate) * up;
            }
            continue;
        }
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = acc[i][r] * rowscale[mb + (r & 3) + 8 * (r >> 2)];
        if (!parts && g.res) {  // every residual of the tile in flight before the first store
            float q[16];
#pragma unroll
            for (int r = 0; r < 16; ++r)
                q[r] = g.res[(size_t)min(m0 + mb + (r & 3) + 8 * (r >> 2), g.M - 1) * g.N + min(n, g.N - 1)];
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] += q[r];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + mb + (r & 3) + 8 * (r >> 2);
            if (m < g.M && n < g.N) cout[(size_t)m * g.N + n] = v[r];
        }
    }
}

template <int FMT, int TM>
int launch(XArgs &x, hipStream_t st) {
    using Tl = XTile<FMT, TM>;
    static const hipError_t attr_rc = hipFuncSetAttribute((const void *)gemm_f32_kernel<FMT, TM>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, Tl::kBytes);
    DOE_HIP_CHECK(attr_rc);
    x.tiles_m = (x.M + Tl::BM - 1) / Tl::BM;
    x.tiles_n = (x.N + Tl::BN - 1) / Tl::BN;
    const int64_t work = (int64_t)x.tiles_m * x.tiles_n * x.splits;
    DOE_REQUIRE(work <= 0x7fffffff, DOE_E_UNSUPPORTED, "too many tiles");
    hipLaunchKernelGGL((gemm_f32_kernel<FMT, TM>), dim3((unsigned)work), dim3(256), Tl::kBytes, st, x);
    DOE_LAUNCH_CHECK("gemm_f32_kernel");
    return DOE_OK;
}

constexpr int64_t kChunkK = 64;

int64_t padded_k(int64_t k, int fmt) { return fmt == 0 ? (k + 255) / 256 * 256 : (k + kChunkK - 1) / kChunkK * kChunkK; }
int64_t frag_bytes(int64_t m, int64_t k, int fmt) { return (m + 31) / 32 * 32 * padded_k(k, fmt) * 4; }
int64_t sums_bytes(int64_t m, int64_t k, int fmt) { return fmt == 0 ? (m + 31) / 32 * (padded_k(k, 0) / 256) * 1024 : 0; }

}  // namespace

namespace doe {

// 64- or 128-row tiles and the K splits (each at least 256 elements of K, at
// most 32: their partials are written and summed once more), by the least of
//   blocks of 256 K on the busiest CU x us per block + the partials' cost.
// A CU takes 3.8 us per block of a 128-row Q4_K tile with one workgroup or two
// (5.0 Q8_0), 2.2 of a 64-row one (3.2), and 0.35 of a block to fill the
// pipeline; the summing pass costs 3.5 us and its bytes at 7 TB/s (tens of MB,
// read back from the last-level cache).  Chosen over every (height, splits) of 16
// weight shapes x 19 prompt lengths; of the 31 shapes where it decides other than
// with the partials at 4 TB/s for Q4_K and 8 for Q8_0 and a fill for Q8_0 alone,
// 24 are faster (Q4_K 33 x 18432 x 2304 27.6 -> 25.2 us, 400 x 3072 x 3072 38.3 ->
// 34.9, Q8_0 80 x 1536 x 4096 24.4 -> 21.0, 110 x 2304 x 2048 22.7 -> 19.7), the
// worst 64 x 9000 x 1152 with GeGLU 17.8 -> 18.9 (200 x 18432 x 2304 Q8_0 with GeGLU
// over halves, which takes a second pass in any case, 85 -> 92).  Height and splits, us, with
// the rule / without: Q4_K 128 x 4096 x 2304 64 rows in three 21.6 / unsplit 27;
// 512 x 2304 x 9216 128 rows in three 66.5 / 64 rows 70.5; Q8_0 128 x 18432 x
// 2304 128 rows in three 47.2 / unsplit 50.6.
GemmF32Plan gemm_f32_plan(int64_t m, int64_t n, int64_t k, int fmt, int num_cus) {
    GemmF32Plan p{};
    const int64_t nblk = (padded_k(k, fmt) + 255) / 256;
    double best = 0.0;
    for (int rows = 64; rows <= 128; rows += 64) {
        const double block_us = rows == 64 ? (fmt == 0 ? 2.2 : 3.2) : (fmt == 0 ? 3.8 : 5.0);
        const int64_t tiles = ((m + rows - 1) / rows) * ((n + 127) / 128);
        for (int64_t want = 1; want <= 32 && want <= nblk && (want == 1 || tiles * want <= 3 * num_cus); ++want) {
            const int64_t per = (nblk + want - 1) / want, splits = (nblk + per - 1) / per;
            double us = (double)((tiles * splits + num_cus - 1) / num_cus) * ((double)per + 0.35) * block_us;
            if (splits > 1) us += 3.5 + (double)splits * (double)(m * n) * 8e-6 / 7.0;
            if (p.tile_rows == 0 || us < best) {
                best = us;
                p.tile_rows = rows;
                p.splits = splits;
                p.chunks_per_split = 4 * per;
            }
        }
    }
    p.a_bytes = frag_bytes(m, k, fmt) + sums_bytes(m, k, fmt) + (m * 4 + 15) / 16 * 16;
    return p;
}

int gemm_f32_launch(const GemmF32Args &g, const GemmF32Plan &plan, void *workspace, hipStream_t st) {
    const int64_t kp = padded_k(g.k, g.fmt);
    const int nsub = (int)(kp / 32);
    u32x4 *frag = (u32x4 *)workspace;
    char *sums = (char *)workspace + frag_bytes(g.m, g.k, g.fmt);
    int *sig = (int *)(sums + sums_bytes(g.m, g.k, g.fmt));
    const dim3 rows((unsigned)((g.m + 31) / 32 * 32));  // 32 ids hold 32 rows (four per XCD)
    const int64_t granules = (kp / 8 + 255) / 256;       // per thread
#define DOE_A_FRAG(G, NORM, SUMS)                                                                                   \
    hipLaunchKernelGGL((a_fragments_kernel<G, NORM, SUMS>), rows, dim3(256), 0, st, g.a, g.norm_w, g.norm_eps,      \
                       g.norm_offset, frag, (_Float16 *)sums, sig, (int)g.m, (int)g.k, nsub)
#define DOE_A_FRAG_G(G)                                            \
    do {                                                           \
        if (g.fmt == 0) {                                          \
            if (g.norm_w) DOE_A_FRAG(G, true, true);               \
            else DOE_A_FRAG(G, false, true);                       \
        } else {                                                   \
            if (g.norm_w) DOE_A_FRAG(G, true, false);              \
            else DOE_A_FRAG(G, false, false);                      \
        }                                                          \
    } while (0)
    if (granules <= 1) DOE_A_FRAG_G(1);
    else if (granules <= 2) DOE_A_FRAG_G(2);
    else if (granules <= 3) DOE_A_FRAG_G(3);
    else if (granules <= 6) DOE_A_FRAG_G(6);
    else DOE_A_FRAG_G(0);
#undef DOE_A_FRAG_G
#undef DOE_A_FRAG
    DOE_LAUNCH_CHECK("a_fragments_kernel");
    XArgs x;
    x.frag = frag;
    x.sums = (const u32x4 *)sums;
    x.sig = sig;
    x.b = (const uint8_t *)g.b;
    x.c = g.c;
    x.part = g.part;
    x.res = g.residual;
    x.pairs = g.pairs;
    x.M = (int)g.m;
    x.N = (int)g.n;
    x.nb = (int)(g.fmt ? (g.k + 31) / 32 : (g.k + 255) / 256);
    x.nsub = nsub;
    x.splits = (int)plan.splits;
    x.nchunk = (int)(kp / kChunkK);
    x.cps = (int)plan.chunks_per_split;
    if (plan.tile_rows == 64) return g.fmt == 0 ? launch<0, 2>(x, st) : launch<1, 2>(x, st);
    return g.fmt == 0 ? launch<0, 4>(x, st) : launch<1, 4>(x, st);
}

}  // namespace doe
