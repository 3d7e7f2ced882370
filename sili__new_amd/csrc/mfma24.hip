// mfma24.hip -- gathers over a dense enough scattered store on the sparse
// matrix cores (linear_disldo.hpp:68-126 and its transpose: out[b, r] =
// sum_c in[b, c] W(r, c) over the shadow store for the forward, the canonical
// one for the grad-input).
//
// A synapse's multiply-adds on the vector units cost B / 64 instructions and a
// row of B input values from L2 or LDS whatever the layer's density: at 10 %
// density and batch 128 that bound the staged gather (12 synapse-columns per
// ns).  The matrix cores multiply every cell, stored or not, and gfx950's 2:4
// form (v_smfmac_f32_32x32x32_bf16: of every 4 consecutive columns at most 2
// are stored) does so at 4.16 PFLOP/s as measured, so from about 1 % density
// on they are ahead (the rule and both sides' times stand at mfma24_wanted).
// Nothing of fp32 is given up:
//   - an FP4 code is exact in bf16 (the column scale is applied to the input
//     in fp32 beforehand, the row scale to the sum, as in the staged gather);
//   - an fp32 input is the exact sum of three bf16 pieces (8 + 8 + 8 bits), so
//     three products with fp32 accumulation stand for the one;
//   - inputs (times their column scale) are shifted by 2^60 before they are
//     split, the sums back by the row scale's product: every fp32 input down to
//     the subnormals then has its pieces in bf16's normal range, and no sum of
//     the 2^21 columns at most overflows.  Batch rows holding an input outside
//     that window (non-finite, or 2^42 and more) are seen by the split kernel
//     and computed from the store's synapses by the same kernel in the order of
//     the other gathers (code * (row scale * column scale)) * input.
// Columns of a group of 4 beyond the second go to an overflow list (1 % of the
// synapses at 10 % density), added in fp32 before the output is written.
//
// The store's derived copy (built on first use, dropped when weights or
// structure change): per 32 rows x 128 columns, 1 KiB of FP4 codes (lane l: 4
// dwords, one per 32 columns, 8 codes each) and 512 bytes of positions (lane l:
// 2 dwords, 16 bits per 32 columns), in the order the instruction's A operand
// takes them: 0.375 bytes per cell.
#include "../../include/sili_hip.h"
#include "layer.hpp"
#include "wave.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace sili {

namespace {

constexpr unsigned TPB = 256;
inline unsigned nblk(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int64_t KB = 128;       // columns per block of the copy
// The copy's blocks of a layer: a multiple of 4, so that the kernels' rings of
// registers go round without a branch (at which the compiler waits for every
// load in flight).
inline int64_t n_blocks(int64_t cols) { return ((cols + KB - 1) / KB + 3) & ~int64_t(3); }
constexpr int64_t MAX_B = 512;    // batches that the gather serves
constexpr int64_t BUILD_K = 4096;  // columns a build block holds in LDS (48 KiB)

// ---- building the copy ---------------------------------------------------------

// The operand place of column kk (0..31) of a 32-column step, as measured from
// the instruction: lanes [0, 32) hold columns 0-7 and 16-23, lanes [32, 64)
// 8-15 and 24-31, each as 4 groups of 4 columns with 2 slots.
__device__ __forceinline__ uint32_t place_half(uint32_t kk) { return (kk >> 3) & 1u; }
__device__ __forceinline__ uint32_t place_group(uint32_t kk) { return ((kk >> 4) << 1) | ((kk >> 2) & 1u); }

// How many of the row's entries before e fall into e's group of 4 columns
// (counted up to 2: the entry then goes to the overflow list).
__device__ __forceinline__ uint32_t group_rank(const int32_t *__restrict__ cols, uint32_t e, uint32_t lo) {
    const uint32_t g = (uint32_t)cols[e] >> 2;
    uint32_t rank = 0;
    if (e > lo && (uint32_t)cols[e - 1] >> 2 == g) rank = 1;
    if (e > lo + 1 && (uint32_t)cols[e - 2] >> 2 == g) rank = 2;
    return rank;
}

__global__ void k_m24_clear(uint32_t *p, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0u;
}

// ovf_n[r] = the row's overflow entries (codes other than 0): one wave per row.
__global__ __launch_bounds__(256) void k_m24_count(const uint32_t *__restrict__ elem_start,
                                                   const int32_t *__restrict__ cols, const uint8_t *__restrict__ val,
                                                   int64_t rows, uint32_t *__restrict__ ovf_n,
                                                   uint32_t *__restrict__ most) {
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const uint32_t lane = lane_id(), lo = elem_start[r], hi = elem_start[r + 1];
    uint32_t n = 0;
    for (uint32_t e0 = lo; e0 < hi; e0 += 64u) {
        const uint32_t e = e0 + lane;
        const bool over = e < hi && (val[e] >> 4) != 0 && group_rank(cols, e, lo) >= 2u;
        n += (uint32_t)__popcll(__ballot(over));
    }
    if (lane == 0u) {
        ovf_n[r] = n;
        if (n > 0u) atomicMax(most, n);
    }
}

// The overflow entries of every row in column order: (row's low 9 bits << 23 |
// column, the code's value): one wave per row.
__global__ __launch_bounds__(256) void k_m24_overflow(const uint32_t *__restrict__ elem_start,
                                                      const int32_t *__restrict__ cols,
                                                      const uint8_t *__restrict__ val, int64_t rows,
                                                      const uint32_t *__restrict__ ovf_start,
                                                      uint2 *__restrict__ ovf) {
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const uint32_t lane = lane_id(), lo = elem_start[r], hi = elem_start[r + 1];
    uint32_t at = ovf_start[r];
    if (at == ovf_start[r + 1]) return;
    for (uint32_t e0 = lo; e0 < hi; e0 += 64u) {
        const uint32_t e = e0 + lane;
        const bool over = e < hi && (val[e] >> 4) != 0 && group_rank(cols, e, lo) >= 2u;
        const uint64_t m = __ballot(over);
        if (over) {
            const uint32_t k = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            ovf[at + k] = make_uint2(((uint32_t)(r & 511) << 23) | (uint32_t)cols[e],
                                     __builtin_bit_cast(uint32_t, fp4_decode(val[e] >> 4)));
        }
        at += (uint32_t)__popcll(m);
    }
}

// One block: 32 rows (blockIdx.x) x BUILD_K columns (blockIdx.y) of the copy,
// assembled in LDS by bitwise or and written out whole.
__global__ __launch_bounds__(256) void k_m24_build(const uint32_t *__restrict__ elem_start,
                                                   const int32_t *__restrict__ cols, const uint8_t *__restrict__ val,
                                                   int64_t rows, int64_t nkb, uint4 *__restrict__ out_val,
                                                   uint2 *__restrict__ out_idx) {
    constexpr uint32_t NB = (uint32_t)(BUILD_K / KB);
    __shared__ __align__(16) uint32_t s_val[NB * 64 * 4];
    __shared__ __align__(16) uint32_t s_idx[NB * 64 * 2];
    __shared__ uint32_t s_range[64];
    const uint32_t t = threadIdx.x;
    for (uint32_t i = t; i < NB * 256; i += TPB) s_val[i] = 0u;
    for (uint32_t i = t; i < NB * 128; i += TPB) s_idx[i] = 0u;
    const int64_t r0 = (int64_t)blockIdx.x * 32, k0 = (int64_t)blockIdx.y * BUILD_K;
    if (t < 64u) {  // the 32 rows' first entry at or past k0, and past the block's end
        const int64_t r = r0 + (t & 31u);
        uint32_t lo = 0, hi = 0;
        if (r < rows) {
            lo = elem_start[r];
            hi = elem_start[r + 1];
            const int64_t key = k0 + (t >= 32u ? BUILD_K : 0);
            while (lo < hi) {
                const uint32_t mid = lo + ((hi - lo) >> 1);
                if ((int64_t)cols[mid] < key) lo = mid + 1;
                else hi = mid;
            }
        }
        s_range[t] = lo;
    }
    __syncthreads();
    for (uint32_t m = t >> 6; m < 32u; m += 4u) {
        const int64_t r = r0 + m;
        if (r >= rows) break;
        const uint32_t row_lo = elem_start[r], hi = s_range[32u + m];
        for (uint32_t e = s_range[m] + (t & 63u); e < hi; e += 64u) {
            const uint32_t code = (uint32_t)(val[e] >> 4);
            const uint32_t rank = group_rank(cols, e, row_lo);
            if (code == 0u || rank >= 2u) continue;
            const uint32_t k = (uint32_t)((int64_t)cols[e] - k0), kk = k & 31u;
            const uint32_t lane = place_half(kk) * 32u + m, slot = 2u * place_group(kk) + rank;
            const uint32_t kb = k >> 7, ks = (k >> 5) & 3u;
            atomicOr(&s_val[(kb * 64u + lane) * 4u + ks], code << (4u * slot));
            atomicOr(&s_idx[(kb * 64u + lane) * 2u + (ks >> 1)], (kk & 3u) << (2u * slot + 16u * (ks & 1u)));
        }
    }
    __syncthreads();
    const int64_t kb0 = k0 / KB;
    const uint32_t nb = (uint32_t)min<int64_t>(NB, nkb - kb0);
    const int64_t base = ((int64_t)blockIdx.x * nkb + kb0) * 64;
    for (uint32_t i = t; i < nb * 64u; i += TPB) {
        out_val[base + i] = reinterpret_cast<const uint4 *>(s_val)[i];
        out_idx[base + i] = reinterpret_cast<const uint2 *>(s_idx)[i];
    }
}

// ---- the input's pieces ----------------------------------------------------------

// v = p[0] + p[1] + p[2] exactly, each a bf16 (round to nearest: the
// remainders have at most 16 and 8 significant bits); v = x * scale.  False
// where v is outside the window: below 2^-102 the last piece would be
// subnormal, and 2^21 columns of 6 * 2^102 are what a sum holds.
__device__ __forceinline__ bool split3(float x, float scale, __bf16 (&p)[3]) {
    const float v = x * scale;
    p[0] = (__bf16)v;
    const float r1 = v - (float)p[0];
    p[1] = (__bf16)r1;
    p[2] = (__bf16)(r1 - (float)p[1]);
    const float a = __builtin_fabsf(v);
    return (a == 0.0f && (x == 0.0f || scale == 0.0f)) || (a >= 0x1p-102f && a < 0x1p102f);
}
constexpr float SHIFT = 0x1p60f;
// A sum of shifted terms, times the row scale (neither product leaves the
// range on the way unless the result does).
__device__ __forceinline__ float unshifted(float sum, float rs) {
    return __builtin_fabsf(rs) < 1.0f / SHIFT ? (sum * rs) * (1.0f / SHIFT) : sum * (rs * (1.0f / SHIFT));
}

struct SplitArgs {
    const float *in;      // batch-major input [B][ld]
    int64_t ld, cols, B;
    const float *ent;     // column scales, or NULL
    float *xT;            // the input feature-major [cols][B] (without the scales), or NULL
    __bf16 *out;
    uint32_t *flag;       // per batch row: set to epoch, this call's number, when an input has no pieces
    uint32_t epoch;
    int64_t nsteps;       // 32-column steps (a multiple of 4)
    int nt;               // column tiles of 32
};

// The B operands in the order the instruction takes them: a lane holds 16
// consecutive columns of one batch row, kept as two 1 KiB halves (8 columns of
// 64 lanes each) so that LDS reads and writes are linear.  Thread (step, tile,
// lane).
//   SMALL: operand column c = piece * B + b (tiles of 32 such columns); one
//     operand per (step, tile);
//   else:  operand column = batch row (tiles of 32, chunks of at most 4 tiles
//     per launch row); operands [chunk][step][piece][tile of the chunk].
template <bool SMALL>
__global__ __launch_bounds__(256) void k_m24_split(SplitArgs a) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    const uint32_t lane = (uint32_t)(i & 63);
    const int64_t tile = (i >> 6) % a.nt, step = (i >> 6) / a.nt;
    if (step >= a.nsteps) return;
    const int64_t k0 = step * 32 + (lane >> 5) * 16;
    const int64_t n = tile * 32 + (lane & 31u);
    const int64_t b = SMALL ? n % a.B : n;
    const int piece = SMALL ? (int)(n / a.B) : 0;
    const bool on = SMALL ? piece < 3 : b < a.B;
    bool ok = true;
    const float *src = a.in + (on ? b : 0) * a.ld;
    __bf16 h[SMALL ? 1 : 3][16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int64_t k = k0 + j;
        float x = 0.0f, scale = SHIFT;
        if (on && k < a.cols) {
            x = src[k];
            if (a.xT && piece == 0) a.xT[k * a.B + b] = x;
            if (a.ent) scale *= a.ent[k];
        }
        __bf16 p[3];
        // (up to 2^60, a column scale's products with the shift and a code are finite)
        ok = split3(x, scale, p) && __builtin_fabsf(scale) <= 0x1p120f && ok;
        if constexpr (SMALL) {
            h[0][j] = piece == 0 ? p[0] : piece == 1 ? p[1] : p[2];
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q) h[q][j] = p[q];
        }
    }
    if (!ok) a.flag[b] = a.epoch;
    // (as in k_transpose)
    if (a.xT && a.B % 4 != 0 && blockIdx.x == 0 && threadIdx.x < (uint32_t)BATCH_SLACK) a.xT[a.cols * a.B + threadIdx.x] = 0.0f;
    uint4 *o = reinterpret_cast<uint4 *>(a.out);
    struct Two {
        uint4 lo, hi;
    };
    struct H16 {
        __bf16 h[16];
    };
    const int64_t chunk = SMALL ? 0 : tile >> 2, ct = SMALL ? 0 : tile & 3, cnt = SMALL ? 1 : min<int64_t>(4, a.nt - chunk * 4);
    const int64_t base = SMALL ? (step * a.nt + tile) * 128
                               : chunk * 4 * 3 * a.nsteps * 128 + (step * 3 * cnt + ct) * 128;
#pragma unroll
    for (int q = 0; q < (SMALL ? 1 : 3); ++q) {
        H16 t;
#pragma unroll
        for (int j = 0; j < 16; ++j) t.h[j] = h[q][j];
        const Two v = __builtin_bit_cast(Two, t);
        o[base + q * cnt * 128 + lane] = v.lo;
        o[base + q * cnt * 128 + 64 + lane] = v.hi;
    }
}

// ---- the products ----------------------------------------------------------------

struct M24Args {
    const uint4 *val;           // the copy
    const uint2 *idx;
    const uint32_t *ovf_start;  // [rows + 1]
    const uint2 *ovf;
    int64_t rows, cols, nkb, ntile;
    const __bf16 *xf;           // the input's operands
    const uint32_t *flag;       // per batch row; epoch: an input of this call has no pieces
    uint32_t epoch;
    const float *inT;           // feature-major input [cols][B] and its column scales (or NULL)
    const float *ent;
    const float *rs;            // row scales, or NULL
    int64_t B;
    float *out;                 // [B][out_ld], written
    int64_t out_ld;
    // the store itself, for inputs without pieces
    const uint32_t *byte_start, *elem_start;
    const uint8_t *sidx, *sval;
    int nt;                     // operand column tiles of the whole call
};

__device__ __forceinline__ bf8 codes_to_bf16(uint32_t w) {
    const bf2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 0);
    const bf2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 1);
    const bf2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 2);
    const bf2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 3);
    return bf8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef unsigned int u2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ bf16x16 operand(const u4 (&b)[2]) {
    return __builtin_bit_cast(bf16x16, __builtin_shufflevector(b[0], b[1], 0, 1, 2, 3, 4, 5, 6, 7));
}
template <int KS>
__device__ __forceinline__ f16v smfmac(bf8 A, bf16x16 Bv, f16v C, const u2 &ix) {
    const int w = (int)ix[KS >> 1];
    return __builtin_amdgcn_smfmac_f32_32x32x32_bf16(A, Bv, C, w, 0, KS & 1);
}

// Whether batch row b0 + lane holds an input without pieces.
__device__ __forceinline__ uint32_t row_flag(const M24Args &a, int64_t b0) {
    return a.flag[min<int64_t>(b0 + lane_id(), a.B - 1)];
}
__device__ __forceinline__ uint64_t odd_rows(const M24Args &a, int64_t b0, uint32_t flag) {
    return __ballot(b0 + lane_id() < a.B && flag == a.epoch);
}
// out rows [r0, r1) of the batch rows b0 + (bits of todo), from the store's
// synapses in fp32: one wave, a lane per synapse of a 64-byte window, 4
// neighbouring batch rows a turn (one load a synapse for them; the others of
// the 4 are not written).  R rows go side by side, without a branch between
// their loads: a row alone is a chain of a window's bytes, its values and its
// inputs.  At 5120 x 204800, 10 %, a call holding one such batch row took 1.25 ms
// at batch 128 (0.52 without; the segment gather 1.4) and 0.97 at batch 8 (0.10;
// the stream kernels 0.14), one holding nothing else 20 and 1.7 ms.  (A whole
// call's loop over the batch columns instead, wherever one input was below
// 2^-110, not finite or too large: 32 and 9.3 ms.)
__device__ __forceinline__ void rows_in_fp32(const M24Args &a, int64_t r0, int64_t r1, int64_t b0, uint64_t todo) {
    constexpr int R = 4;
    const uint32_t lane = lane_id();
    for (; todo; todo >>= 4, b0 += 4) {
        if ((todo & 15ull) == 0ull) continue;
        for (int64_t r = r0; r < r1; r += R) {
            float f[R];
            float4 acc[R];
            uint32_t pos[R], end[R], ebase[R], carry[R];
            bool more = false;
#pragma unroll
            for (int q = 0; q < R; ++q) {  // past the last row: an empty one
                const int64_t row = min<int64_t>(r + q, r1 - 1);
                f[q] = a.rs ? a.rs[row] : 1.0f;
                pos[q] = a.byte_start[row];
                end[q] = r + q < r1 ? a.byte_start[row + 1] : pos[q];
                ebase[q] = a.elem_start[row];
                carry[q] = 0;
                more = more || pos[q] < end[q];
                acc[q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            while (more) {
                uint32_t byte[R];
                Chunk ch[R];
                float w[R];
                float4 x[R];
                // (a lane without a byte or a synapse loads what another one does)
#pragma unroll
                for (int q = 0; q < R; ++q) byte[q] = a.sidx[pos[q] + lane < end[q] ? pos[q] + lane : 0u];
#pragma unroll
                for (int q = 0; q < R; ++q) ch[q] = decode_window(pos[q] + lane < end[q] ? byte[q] : 0x80u, carry[q]);
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    w[q] = fp4_decode((uint32_t)(a.sval[ch[q].term ? ebase[q] + ch[q].rank : 0u] >> 4)) *
                           (a.ent ? f[q] * a.ent[ch[q].col] : f[q]);
                    x[q] = load_f4(a.inT + (uint64_t)ch[q].col * (uint32_t)a.B + b0);  // (3 floats past the last input at most)
                }
                more = false;
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    acc[q].x = ch[q].term ? __builtin_fmaf(w[q], x[q].x, acc[q].x) : acc[q].x;
                    acc[q].y = ch[q].term ? __builtin_fmaf(w[q], x[q].y, acc[q].y) : acc[q].y;
                    acc[q].z = ch[q].term ? __builtin_fmaf(w[q], x[q].z, acc[q].z) : acc[q].z;
                    acc[q].w = ch[q].term ? __builtin_fmaf(w[q], x[q].w, acc[q].w) : acc[q].w;
                    if (ch[q].T == 0ull) pos[q] = end[q];
                    else carry[q] = chunk_advance(ch[q], pos[q], ebase[q]);
                    more = more || pos[q] < end[q];
                }
            }
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const float4 sum = make_float4(wave_sum(acc[q].x), wave_sum(acc[q].y), wave_sum(acc[q].z), wave_sum(acc[q].w));
                if (lane < 4u && ((todo >> lane) & 1ull) && r + q < r1)
                    a.out[(b0 + lane) * a.out_ld + r + q] = lane < 2u ? (lane == 0u ? sum.x : sum.y) : (lane == 2u ? sum.z : sum.w);
            }
        }
    }
}

// A wave's LDS byte address of a shared array.
__device__ __forceinline__ uint32_t lds_address(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}
// NF B operands of 2 KiB each, STRIDE bytes apart, from LDS byte address at
// (the lane's 16 bytes of the first half): read and waited for in one block.
// The compiler orders a plain LDS read behind every direct global -> LDS load
// in flight, also those into other buffers, which left no load in flight while
// a step was multiplied (851 us against 424 at 5120 x 204800, batch 128).
template <int STRIDE>
__device__ __forceinline__ void read_operands(uint32_t at, u4 (&b)[1][2]) {
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:1024\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(b[0][0]), "=&v"(b[0][1])
                 : "v"(at)
                 : "memory");
}
template <int STRIDE>
__device__ __forceinline__ void read_operands(uint32_t at, u4 (&b)[2][2]) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:1024\n\t"
                 "ds_read_b128 %2, %4 offset:%5\n\tds_read_b128 %3, %4 offset:%6\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
                 : "v"(at), "n"(STRIDE), "n"(STRIDE + 1024)
                 : "memory");
}
template <int STRIDE>
__device__ __forceinline__ void read_operands(uint32_t at, u4 (&b)[3][2]) {
    asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:1024\n\t"
                 "ds_read_b128 %2, %6 offset:%7\n\tds_read_b128 %3, %6 offset:%8\n\t"
                 "ds_read_b128 %4, %6 offset:%9\n\tds_read_b128 %5, %6 offset:%10\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1]), "=&v"(b[2][0]), "=&v"(b[2][1])
                 : "v"(at), "n"(STRIDE), "n"(STRIDE + 1024), "n"(2 * STRIDE), "n"(2 * STRIDE + 1024)
                 : "memory");
}
// Ends a stage's window of issued loads: waits until at most N of this wave's
// vector memory operations are in flight, then for the block.  No load moves
// across it (a volatile block with a memory clobber, and a scheduling barrier),
// so a window's loads are issued between its two ends in some order, and N may
// count every load of the windows after the one whose loads must have landed,
// none of that window itself.
template <int N>
__device__ __forceinline__ void landed_for_block() {
    static_assert(N < 64, "the counter's range");
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// The A operands of up to mt row tiles from tile0 as buffer loads: a scalar
// offset per (tile, block) and one lane offset, where address pairs per tile
// would not fit beside the accumulators.  Tiles and blocks past the last are
// the last one again (their results are not used); the hardware's range check
// plays no part.
struct ACopy {
    __amdgpu_buffer_rsrc_t val, idx;
    uint32_t nkb, last, lane;
    __device__ __forceinline__ ACopy(const M24Args &a, int64_t tile0, int mt) {
        const int64_t t = min<int64_t>(tile0, a.ntile - 1), n = min<int64_t>(mt, a.ntile - t);
        val = buffer_rsrc(a.val + t * a.nkb * 64, (uint32_t)(n * a.nkb * 1024));
        idx = buffer_rsrc(a.idx + t * a.nkb * 64, (uint32_t)(n * a.nkb * 512));
        nkb = (uint32_t)a.nkb;
        last = (uint32_t)n - 1u;
        lane = lane_id();
    }
    template <int AUX>
    __device__ __forceinline__ void load(int i, uint32_t kb, u4 &v, u2 &ix) const {
        const uint32_t at = min((uint32_t)i, last) * nkb + min(kb, nkb - 1u);
        v = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(val, (int)(lane * 16u), (int)(at * 1024u), AUX));
        ix = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(idx, (int)(lane * 8u), (int)(at * 512u), AUX));
    }
};
constexpr int AUX_NT = 2;  // non-temporal: read once per call, not kept in the caches
// 1 KiB of the operand array (at byte offset off) to LDS address to by a direct
// load.
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, uint32_t off, uint8_t *to) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)to, 16, (int)(lane_id() * 16u),
                                             (int)off, 0, 0);
}

// A wave's accumulators of one 32-row tile and one operand column tile into
// LDS, column-major with an odd stride of ld floats, so that a batch row's rows
// leave as one run.
__device__ __forceinline__ void tile_to_lds(float *s, uint32_t ld, const f16v &acc) {
    const uint32_t lane = lane_id(), half = lane >> 5, n = lane & 31u;
#pragma unroll
    for (int q = 0; q < 16; ++q)  // row (q / 4) * 8 + half * 4 + q % 4 of column n
        s[n * ld + (q >> 2) * 8 + half * 4 + (q & 3)] = acc[q];
}

// The overflow entries of rows [r0, r1), times the batch rows from x
// (feature-major, C = 1 or 2 per lane), added to the lane's columns of the tile
// in LDS (col: row r0 of the first one), one wave, in order.  64 entries are
// loaded at a time, a lane each, and handed round as scalars, so an entry costs
// one vector load for all its columns; a row's run is summed in registers.
// (Each lane loading every entry for itself, and float adds in LDS at ~150
// clocks a wave instruction, took 840 of 1260 us at 5120 x 204800, batch 128;
// LDS updates in their place 160.)
template <int C, bool ENT>
__device__ __forceinline__ void add_overflow(const M24Args &a, float *col, uint32_t ld, const float *x, int64_t r0,
                                             int64_t r1) {
    constexpr int U = 8;
    const uint32_t lane = lane_id();
    const uint32_t o0 = a.ovf_start[r0], o1 = a.ovf_start[r1];
    if (o0 >= o1) return;
    uint32_t row = 0;  // the row whose run is being summed, within [r0, r1)
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = col[c * ld];
    for (uint32_t o = o0; o < o1; o += 64u) {
        const uint32_t n = min(64u, o1 - o);
        const uint2 e = a.ovf[min(o + lane, o1 - 1u)];
        float w = __builtin_bit_cast(float, e.y) * SHIFT;
        if constexpr (ENT) w *= a.ent[e.x & 0x7FFFFFu];
        for (uint32_t j = 0; j < n; j += U) {
            float v[U][C], we[U];
            uint32_t re[U];
#pragma unroll
            for (uint32_t i = 0; i < U; ++i) {  // past the end: the last entry, weight 0
                const int l = (int)min(j + i, n - 1u);
                const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)e.x, l);
                we[i] = j + i < n ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), l)) : 0.0f;
                re[i] = ((k >> 23) - (uint32_t)r0) & 511u;
                const float *src = x + (uint64_t)(k & 0x7FFFFFu) * (uint32_t)a.B;
                if constexpr (C == 2) {  // (at most one float past the last input: the buffer is padded)
                    const float2 t = load_f2(src);
                    v[i][0] = t.x;
                    v[i][1] = t.y;
                } else {
                    v[i][0] = src[0];
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < U; ++i) {
                if (re[i] != row) {
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        col[c * ld + row] = acc[c];
                        acc[c] = col[c * ld + re[i]];
                    }
                    row = re[i];
                }
#pragma unroll
                for (int c = 0; c < C; ++c) acc[c] = __builtin_fmaf(we[i], v[i][c], acc[c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) col[c * ld + row] = acc[c];
}

// Batches above 21: a block of 8 waves takes 32*MT*(8/WN) rows and 32*WN batch
// rows; wave (wm, wn) MT row tiles and one column tile.  The leading pieces'
// products and the two small pieces' have accumulators of their own: added into
// one, the small terms are rounded at the sum's size three times as often
// (3.8e-7 against 7e-8 off 64 bits at 512 synapses a row).  The B operands (6
// KiB per 32-column step and column tile) come to LDS by direct loads in
// stages of 24 KiB, two stages ahead in a ring of three, so that two blocks (4
// waves per SIMD) share a CU (MT = 4 with one block a CU was behind at every
// size).  Each wave reads an operand once per MT products; MT = 1 is for
// layers of few blocks.  What it waits for (5120 x 204800, 10 %, batch 128, 481
// us): no unit is busy throughout -- the matrix cores 39 % of the cycles, the
// CU's load path (operand stages and the copy) 66, LDS 22, VALU issue 17, HBM at
// 1.6 TB/s; a block's waves meet at a barrier per stage.  A operands come
// straight from the copy, a 128-column block ahead, and are issued behind the
// stage loads of their block, so that waiting for a stage does not wait for them.
template <int MT, int WN>
__global__ __launch_bounds__(512, 4) void k_m24(M24Args a) {
    constexpr int WM = 8 / WN, SPS = 4 / WN;                   // row groups; steps per stage
    constexpr uint32_t STEP = 3u * WN * 2048u, STAGE = 24576;  // bytes
    constexpr uint32_t NR = 3;                                 // stages in the ring
    constexpr int DOPS = 3, AOPS = 2 * MT;                     // a wave's loads per stage, per 128-column block
    static_assert(SPS * STEP == STAGE && STAGE == 8 * DOPS * 1024, "a stage is 3 KiB per wave");
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t lane = lane_id(), wave = uniform(threadIdx.x >> 6), wm = wave / WN, wn = wave % WN;
    const int64_t tile0 = ((int64_t)blockIdx.x * WM + wm) * MT;
    const int64_t b0 = (int64_t)blockIdx.y * 128;
    const uint32_t flag0 = row_flag(a, b0), flag1 = WN == 4 ? row_flag(a, b0 + 64) : 0u;
    const uint32_t nstages = (uint32_t)a.nkb * WN;
    const __amdgpu_buffer_rsrc_t xf = buffer_rsrc(
        reinterpret_cast<const uint8_t *>(a.xf) + (int64_t)blockIdx.y * 4 * 3 * a.nkb * 4 * 2048, nstages * STAGE);
    // stage t into its place of the ring (past the end: the last one again, to a
    // place that is not read any more, and the counts below stay the same)
    auto stage = [&](uint32_t t) {
        const uint32_t at = (t % NR) * STAGE + wave * 1024u;
#pragma unroll
        for (uint32_t i = 0; i < DOPS; ++i)
            load_to_lds(xf, min(t, nstages - 1u) * STAGE + wave * 1024u + i * 8192u, lds + at + i * 8192u);
    };
    const ACopy ac(a, tile0, MT);
    u4 rv[2][MT];
    u2 ri[2][MT];
    auto fetch = [&](auto slot, uint32_t kb) {
        constexpr int R = decltype(slot)::value;
#pragma unroll
        for (int i = 0; i < MT; ++i) ac.load<0>(i, kb, rv[R][i], ri[R][i]);
    };
    f16v hi[MT], lo[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q) hi[i][q] = lo[i][q] = 0.0f;
    fetch(std::integral_constant<int, 0>{}, 0);
    stage(0);
    stage(1);
    landed_for_block<0>();
    const uint64_t odd0 = odd_rows(a, b0, flag0), odd1 = WN == 4 ? odd_rows(a, b0 + 64, flag1) : 0ull;
    const uint32_t bs0 = lds_address(lds) + wn * 2048u + lane * 16u;
    auto block = [&](auto slot, uint32_t kb) {
        constexpr int R = decltype(slot)::value;
        auto step = [&](auto ksc) {
            constexpr int KS = decltype(ksc)::value;
            const uint32_t t = kb * WN + KS / SPS;
            if constexpr (KS % SPS == 0) stage(t + NR - 1);
            if constexpr (KS == 0) fetch(std::integral_constant<int, 1 - R>{}, kb + 1);
            u4 b[3][2];
            read_operands<WN * 2048>(bs0 + (t % NR) * STAGE + (KS % SPS) * STEP, b);
            bf8 A[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) A[i] = codes_to_bf16(rv[R][i][KS]);
#pragma unroll
            for (int i = 0; i < MT; ++i) hi[i] = smfmac<KS>(A[i], operand(b[0]), hi[i], ri[R][i]);
#pragma unroll
            for (int i = 0; i < MT; ++i) lo[i] = smfmac<KS>(A[i], operand(b[1]), lo[i], ri[R][i]);
#pragma unroll
            for (int i = 0; i < MT; ++i) lo[i] = smfmac<KS>(A[i], operand(b[2]), lo[i], ri[R][i]);
            // stage t + 1, asked for in the window before, must have landed:
            // since then stage t + 2, and the next block's A operands in a
            // block's first window
            if constexpr (KS % SPS == SPS - 1) landed_for_block<DOPS + (KS / SPS == 0 ? AOPS : 0)>();
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
    };
    for (uint32_t kb = 0; kb < (uint32_t)a.nkb; kb += 2) {
        block(std::integral_constant<int, 0>{}, kb);
        block(std::integral_constant<int, 1>{}, kb + 1);
    }
    landed_for_block<0>();  // the ring's last loads: its LDS becomes the block's output tile
    constexpr uint32_t R = WM * MT * 32, LD = R + 1, RW = R / 8;  // the block's rows; a wave's share below
    float *s = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int i = 0; i < MT; ++i) tile_to_lds(s + wn * 32 * LD + (wm * MT + i) * 32, LD, hi[i] + lo[i]);
    __syncthreads();
    const int64_t r0 = (int64_t)blockIdx.x * R;
    const uint32_t nb = (uint32_t)min<int64_t>(a.B - b0, 32 * WN);
    {
        constexpr int C = WN == 4 ? 2 : 1;
        const int64_t w0 = min<int64_t>(r0 + wave * RW, a.rows), w1 = min<int64_t>(w0 + RW, a.rows);
        // (lanes past the tile's columns repeat one; a column past the batch takes
        // any value, its place is not written out)
        const uint32_t c0 = (lane * C) % (32u * WN);
        float *col = s + c0 * LD + wave * RW;
        const float *x = a.inT + b0 + min(c0, nb - 1u);
        if (w0 < w1) {
            if (a.ent) add_overflow<C, true>(a, col, LD, x, w0, w1);
            else add_overflow<C, false>(a, col, LD, x, w0, w1);
        }
    }
    __syncthreads();
    const uint32_t nr = (uint32_t)min<int64_t>(R, a.rows - r0);
    for (uint32_t m = lane; m < nr; m += 64u) {
        const float f = a.rs ? a.rs[r0 + m] : 1.0f;
        float *out = a.out + b0 * a.out_ld + r0 + m;
#pragma unroll 4
        for (uint32_t b = wave; b < nb; b += 8u) out[b * a.out_ld] = unshifted(s[b * LD + m], f);
    }
    if (odd0 | odd1) {
        __syncthreads();  // (over what was written above)
        const int64_t w0 = min<int64_t>(r0 + wave * RW, a.rows), w1 = min<int64_t>(w0 + RW, a.rows);
        for (int h = 0; h < 2; ++h) rows_in_fp32(a, w0, w1, b0 + 64 * h, h ? odd1 : odd0);
    }
}

// Batches up to 21: the 3 pieces are operand columns of their own (3 B <= 32
// NT), so one product per row tile and 32 columns serves the whole batch, and
// the copy's bytes are what is waited for (4.3 TB/s at 5120 x 204800, batch 8, 5.5
// at 1310720 rows; the load path busy 58 % of the cycles, the matrix cores 13): 4
// waves of MT row tiles each share the B operands (a 128-column block per stage,
// in a ring of four), and read their A operands three blocks ahead.
constexpr int SMALL_B = 21;
// 32 rows of a wave, all batch rows: the pieces' sums, then the overflow
// entries of a row by the two lanes that hold it (half h: batch rows [h
// ceil(B/2), ...)).
template <int Q, bool ENT>  // Q: batch rows per lane at most, a multiple of 4
__device__ __forceinline__ void write_rows_small(const M24Args &a, const float *s, int64_t tile, uint32_t odd) {
    constexpr uint32_t LD = 33u;
    constexpr int U = 4;
    const uint32_t lane = lane_id(), half = lane >> 5, m = lane & 31u;
    const int nb = (int)a.B, b0 = half ? (nb + 1) / 2 : 0, b1 = half ? nb : (nb + 1) / 2;
    const int64_t r = tile * 32 + m;
    uint32_t o = a.ovf_start[min<int64_t>(r, a.rows)];
    const uint32_t o1 = a.ovf_start[min<int64_t>(r + 1, a.rows)];
    const float *x = a.inT + b0;
    uint2 next[U];
#pragma unroll
    for (int i = 0; i < U; ++i) next[i] = o + i < o1 ? a.ovf[o + i] : make_uint2(0u, 0u);
    wave_lds_sync();
    float y[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int b = b0 + q;
        y[q] = b < b1 ? (s[b * LD + m] + s[(b + nb) * LD + m]) + s[(b + 2 * nb) * LD + m] : 0.0f;
    }
    for (; o < o1; o += U) {  // lanes whose row is done drop out
        float4 v[U][Q / 4];
        float w[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const uint32_t k = next[i].x & 0x7FFFFFu;
            w[i] = __builtin_bit_cast(float, next[i].y) * SHIFT;
            if constexpr (ENT) w[i] *= a.ent[k];
#pragma unroll
            for (int q = 0; q < Q / 4; ++q)  // (reads up to Q floats from b0: the input's buffer is padded by 64 bytes)
                v[i][q] = load_f4(x + (uint64_t)k * (uint32_t)nb + 4 * q);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) next[i] = o + U + i < o1 ? a.ovf[o + U + i] : make_uint2(0u, 0u);
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int q = 0; q < Q / 4; ++q) {
                y[4 * q] = __builtin_fmaf(w[i], v[i][q].x, y[4 * q]);
                y[4 * q + 1] = __builtin_fmaf(w[i], v[i][q].y, y[4 * q + 1]);
                y[4 * q + 2] = __builtin_fmaf(w[i], v[i][q].z, y[4 * q + 2]);
                y[4 * q + 3] = __builtin_fmaf(w[i], v[i][q].w, y[4 * q + 3]);
            }
    }
    const float f = a.rs && r < a.rows ? a.rs[r] : 1.0f;
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (b0 + q < b1 && r < a.rows && !((odd >> (b0 + q)) & 1u)) a.out[(int64_t)(b0 + q) * a.out_ld + r] = unshifted(y[q], f);
    wave_lds_sync();
}

constexpr int RING = 4;
template <int MT, int NT>
__global__ __launch_bounds__(256, NT == 1 ? 4 : 2) void k_m24_small(M24Args a) {
    constexpr uint32_t STEP = NT * 2048u, STAGE = 4 * STEP;  // bytes
    constexpr int DOPS = STAGE / 4096, AOPS = 2 * MT, AHEAD = 3;
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t lane = lane_id(), wave = uniform(threadIdx.x >> 6);
    const int64_t tile0 = ((int64_t)blockIdx.x * 4 + wave) * MT;
    const __amdgpu_buffer_rsrc_t xf = buffer_rsrc(a.xf, (uint32_t)a.nkb * STAGE);
    auto stage = [&](uint32_t t) {
        const uint32_t at = (t & (RING - 1)) * STAGE + wave * 1024u;
#pragma unroll
        for (uint32_t i = 0; i < DOPS; ++i)
            load_to_lds(xf, min(t, (uint32_t)a.nkb - 1u) * STAGE + wave * 1024u + i * 4096u, lds + at + i * 4096u);
    };
    const ACopy ac(a, tile0, MT);
    f16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;
    u4 rv[RING][MT];
    u2 ri[RING][MT];
    auto fetch = [&](auto slot, uint32_t kb) {
        constexpr int R = decltype(slot)::value;
#pragma unroll
        for (int i = 0; i < MT; ++i) ac.load<AUX_NT>(i, kb, rv[R][i], ri[R][i]);
    };
    stage(0);
    fetch(std::integral_constant<int, 0>{}, 0);
    stage(1);
    fetch(std::integral_constant<int, 1>{}, 1);
    stage(2);
    fetch(std::integral_constant<int, 2>{}, 2);
    landed_for_block<0>();
    const uint32_t bs0 = lds_address(lds) + lane * 16u;
    auto block = [&](auto slot, uint32_t kb) {
        constexpr int R = decltype(slot)::value;
        stage(kb + 3);
        fetch(std::integral_constant<int, (R + AHEAD) % RING>{}, kb + AHEAD);
        auto step = [&](auto ksc) {
            constexpr int KS = decltype(ksc)::value;
            u4 b[NT][2];
            read_operands<2048>(bs0 + R * STAGE + KS * STEP, b);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const bf8 A = codes_to_bf16(rv[R][i][KS]);
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = smfmac<KS>(A, operand(b[j]), acc[i][j], ri[R][i]);
            }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        // stage kb + 1, asked for two windows ago, must have landed
        landed_for_block<2 * (DOPS + AOPS)>();
    };
    for (uint32_t kb = 0; kb < (uint32_t)a.nkb; kb += RING) {
        block(std::integral_constant<int, 0>{}, kb);
        block(std::integral_constant<int, 1>{}, kb + 1);
        block(std::integral_constant<int, 2>{}, kb + 2);
        block(std::integral_constant<int, 3>{}, kb + 3);
    }
    landed_for_block<0>();
    const uint32_t odd = (uint32_t)odd_rows(a, 0, row_flag(a, 0));  // (B <= SMALL_B)
    float *s = reinterpret_cast<float *>(lds) + wave * (NT * 32 * 33u);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (tile0 + i >= a.ntile) break;
#pragma unroll
        for (int j = 0; j < NT; ++j) tile_to_lds(s + j * 32 * 33u, 33u, acc[i][j]);
        if (NT == 1 && a.B <= 8) {
            if (a.ent) write_rows_small<4, true>(a, s, tile0 + i, odd);
            else write_rows_small<4, false>(a, s, tile0 + i, odd);
        } else {
            if (a.ent) write_rows_small<NT == 1 ? 8 : 12, true>(a, s, tile0 + i, odd);
            else write_rows_small<NT == 1 ? 8 : 12, false>(a, s, tile0 + i, odd);
        }
    }
    if (odd) rows_in_fp32(a, min<int64_t>(a.rows, tile0 * 32), min<int64_t>(a.rows, (tile0 + MT) * 32), 0, odd);
}

// Operand column tiles of a batch (of its pieces, up to SMALL_B).
int operand_tiles(int64_t B) {
    if (B <= SMALL_B) return (int)((3 * B + 31) / 32);
    const int nt = (int)((B + 31) / 32);
    return nt > 2 ? (nt + 3) & ~3 : nt;  // whole chunks of 4 column tiles
}

template <int MT, int WN>
void go(const M24Args &a, int64_t chunks, hipStream_t st) {
    constexpr uint32_t ring = 3u * 24576u, out = 32u * WN * ((8u / WN) * MT * 32u + 1u) * 4u, lds = ring > out ? ring : out;
    SILI_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_m24<MT, WN>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int64_t per = (8 / WN) * MT;
    launch(k_m24<MT, WN>, dim3((unsigned)((a.ntile + per - 1) / per), (unsigned)chunks), dim3(512), lds, st, a);
}
template <int MT, int NT>
void go_small(const M24Args &a, hipStream_t st) {
    constexpr uint32_t ring = RING * NT * 8192u, out = 4u * NT * 32u * 33u * 4u, lds = ring > out ? ring : out;
    SILI_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_m24_small<MT, NT>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    launch(k_m24_small<MT, NT>, dim3((unsigned)((a.ntile + 4 * MT - 1) / (4 * MT))), dim3(256), lds, st, a);
}

}  // namespace

namespace {

// Estimated times in us, fitted to measurements (MI355X) on the shapes 1024^2
// to 16384^2, 5120 x 16384, 4096 x 65536, 1024 x 100000 and 5120 x 204800 at
// densities 0.01 to 0.1 and batches 4 to 128; the dispatch below compares them
// and takes the matrix cores where they are ahead by a tenth.  Both sides as
// measured, us (other path / this one):
//   5120 x 204800, 10 %: batch 4 62 / 97, 8 128 / 99, 16 552 / 135, 32 678 / 153,
//     64 1196 / 248, 128 1339 / 464
//   16384^2, 2 %: 16 39 / 67, 32 44 / 98, 64 77 / 114, 128 167 (segments) / 163;
//     10 %: 16 167 / 77, 32 195 / 144, 64 324 / 137, 128 547 / 178
//   8192^2, 2 %: 8 40 / 31, 64 24 / 66, 128 40 / 87; 10 %: 64 82 / 77, 128 160 / 94
//   4096 x 65536, 2 %: 32 50 / 40, 64 74 / 58, 128 115 / 104; 5 %: 16 73 / 39
//   4096^2, 10 %: 16 16 / 30, 64 27 / 46, 128 49 / 54; 1024^2: always behind
struct Shape {
    int64_t ntile, nkb;
    double nnz, cells, ovf, ovf_row;
    explicit Shape(const DScatter &s) : ntile((s.rows + 31) / 32), nkb(n_blocks(s.cols)), nnz((double)s.nnz) {
        cells = (double)ntile * 32.0 * (double)nkb * 128.0;
        const double d = nnz / ((double)s.rows * (double)s.cols);
        // entries beyond two of a group of 4: those of uniform columns until
        // the copy's own counts are there
        ovf = s.m24_valid ? (double)s.m24_n_ovf : cells * d * d * d;
        ovf_row = s.m24_valid ? (double)s.m24_max_ovf : ovf / (double)s.rows;
    }
};
int column_tiles(int64_t B) { return B <= 32 ? 1 : B <= 64 ? 2 : 4; }
// row tiles per wave: one while every CU then has at most one block
int row_tiles(const Shape &h, int64_t B) {
    return (h.ntile + 8 / column_tiles(B) - 1) / (8 / column_tiles(B)) <= 256 ? 1 : 2;
}
double mfma24_us(const Shape &h, int64_t B) {
    const double bytes = 1.15 * h.cells * 0.375 / 5.2e6;
    const double overflow = std::max(4e-5 * h.ovf, 0.08 * h.ovf_row);
    if (B <= SMALL_B) return 10.0 + 0.25 * overflow + (3 * B <= 32 ? 1.0 : 1.4) * std::max(0.29 * (double)h.nkb, bytes);
    const int wn = column_tiles(B), mt = row_tiles(h, B);
    const double step = wn == 1 ? (mt == 1 ? 0.165 : 0.29) : wn == 2 ? (mt == 1 ? 0.2 : 0.32) : (mt == 1 ? 0.295 : 0.39);
    const double blocks = std::ceil((double)h.ntile / (8.0 / wn * mt));
    const double chunks = std::ceil((double)B / 128.0);
    return 10.0 + chunks * (std::max(4.0 * (double)h.nkb * step * std::max(1.0, 1.15 * blocks / 256.0), bytes) + overflow);
}
double others_us(const DScatter &s, int64_t B) {
    const double nnz = (double)s.nnz;
    if ((B == 2 || B == 4 || B == 8) && s.nbytes >= (int64_t(1) << 20) && env_int("SILI_B1_STREAM", 1) != 0) {
        const double blocks = std::ceil((double)(s.cols + 1) * (double)B * 4.0 / 150e3);
        return 6.0 + 1.5 * (double)B * blocks + 0.14e-6 * (double)B * nnz;
    }
    if (B > 64 && B <= 128 && B % 4 == 0 && staged_wanted(s, B)) return std::min(segments_us(s, B), staged_us(s));
    return segments_us(s, B);
}

}  // namespace

// The other gathers serve this layer until its structure changes.
static void release(DScatter &s) {
    s.free_m24();
    s.m24_valid = false;
    s.m24_failed = true;
}

// The copy and the workspace of batch B; false: no memory for them (the copy
// takes SILI_MFMA24_FREE_PCT percent of the free memory at most).
static bool ensure_mfma24(Layer &L, DScatter &s, int64_t B, hipStream_t st) {
    const int64_t ntile = (s.rows + 31) / 32, nkb = n_blocks(s.cols);
    const size_t ops = (size_t)(nkb * 4 * operand_tiles(B) * (B <= SMALL_B ? 1 : 3) * 1024);
    if (s.m24_valid && L.m24_flag.p && L.ws_m24.n >= ops) return true;
    try {
        L.ws_m24.ensure(ops);
        if (!L.m24_flag.p) {
            L.m24_flag.ensure(MAX_B);
            launch(k_m24_clear, dim3(1), dim3(64), 0, st, L.m24_flag.p, (uint32_t)MAX_B);
            L.m24_epoch = 0;
        }
        if (s.m24_valid) return true;
        // a copy takes a part of what is free at most, so that those of many
        // layers leave room for everything else on the device
        size_t free = 0, all = 0;
        SILI_HIP(hipMemGetInfo(&free, &all));
        const double bytes = (double)(ntile * nkb) * 64.0 * 24.0 + 9.0 * (double)s.nnz;  // with what its building takes
        if (bytes > 0.01 * env_int("SILI_MFMA24_FREE_PCT", 25) * (double)free) {
            release(s);
            return false;
        }
        ProfScope ps("mfma24_build", st);
        s.m24_val.ensure((size_t)(ntile * nkb * 64));
        s.m24_idx.ensure((size_t)(ntile * nkb * 64));
        s.m24_ovf_start.ensure((size_t)s.rows + 1);
        DevBuf<int32_t> cols;
        DevBuf<uint32_t> cnt;
        cols.ensure((size_t)s.nnz + 1);
        cnt.ensure((size_t)s.rows + 2);  // the scan's, and the most of a row
        launch(k_m24_clear, dim3(1), dim3(64), 0, st, cnt.p + s.rows + 1, 1u);
        launch_decode(s.plan(), ScaleView{nullptr, nullptr, 1}, cols.p, nullptr, nullptr, st);
        const dim3 rgrid((unsigned)((s.rows + 3) / 4));
        launch(k_m24_count, rgrid, dim3(TPB), 0, st, (const uint32_t *)s.elem_start.p, (const int32_t *)cols.p,
               (const uint8_t *)s.val.p, s.rows, cnt.p, cnt.p + s.rows + 1);
        SILI_HIP(hipStreamSynchronize(st));  // the scan runs on the layer's stream
        device_exclusive_scan_u32(L, cnt.p, s.m24_ovf_start.p, s.rows + 1);
        uint32_t total = 0, most = 0;
        ReadBack rb(L);
        rb.add(&total, s.m24_ovf_start.p + s.rows, 4);
        rb.add(&most, cnt.p + s.rows + 1, 4);
        rb.wait();
        s.m24_n_ovf = total;
        s.m24_max_ovf = most;
        s.m24_ovf.ensure((size_t)total + 1);
        if (total > 0)
            launch(k_m24_overflow, rgrid, dim3(TPB), 0, st, (const uint32_t *)s.elem_start.p, (const int32_t *)cols.p,
                   (const uint8_t *)s.val.p, s.rows, (const uint32_t *)s.m24_ovf_start.p, s.m24_ovf.p);
        launch(k_m24_build, dim3((unsigned)ntile, (unsigned)((nkb * KB + BUILD_K - 1) / BUILD_K)), dim3(TPB), 0, st,
               (const uint32_t *)s.elem_start.p, (const int32_t *)cols.p, (const uint8_t *)s.val.p, s.rows, nkb,
               s.m24_val.p, s.m24_idx.p);
        SILI_HIP(hipGetLastError());
        SILI_HIP(hipStreamSynchronize(st));  // cols and cnt are freed on return
    } catch (const Error &e) {
        if (e.code != SILI_ERR_NOMEM) throw;
        (void)hipGetLastError();
        release(s);
        return false;
    }
    s.m24_valid = true;
    return true;
}

// Whether a forward or grad-input over s takes the matrix cores.  The copy is
// built once the calls since the values last changed have spent as much more
// than they had to as its building costs (at 5120 x 204800, 10 %, 2 ms: the
// third call at batch 128, the 60th at batch 8), and twice as late each time a
// copy was dropped before it had paid for itself: a layer used a few times or
// trained between its forwards keeps the other paths.  Under stream capture
// never: a graph would go on reading the copy after the weights have changed.
// The first call of each batch takes the other kernels, which leaves a program
// that runs a batch before it captures it all that the captured call needs.
bool mfma24_wanted(Layer &L, DScatter &s, const ScaleView &sc, int64_t B, int skip, hipStream_t st) {
    if (B < 2 || B > MAX_B || s.cols > (int64_t(1) << 21)) return false;
    if (s.nnz == 0 || s.m24_failed || L.has_nonfinite || skip != SKIP_NONE || sc.rank != 1) return false;
    // SILI_MFMA24 (read per call): 0 never, 2 whenever it can and at once, 1
    // (default) by the estimates
    const int mode = env_int("SILI_MFMA24", 1);
    if (mode == 0) return false;
    const double other = others_us(s, B);
    const auto gain = [&] { return 0.9 * other - mfma24_us(Shape(s), B); };
    if (mode != 2) {
        // few rows: not a block for every CU
        if (s.repeatable || s.rows < 2048 || ((B == 2 || B == 4 || B == 8) && env_int("SILI_B1_STREAM", 1) == 2)) return false;
        const double g = gain();
        if (Shape(s).cells * 0.375 > 8e9 || g < 0) return false;
        s.m24_saved += g + 0.1 * other;
        if (!s.m24_valid) s.m24_cost = 500.0 + 1.7e-5 * (double)s.nnz;
        const bool warm = s.m24_warm.test((size_t)B);
        s.m24_warm.set((size_t)B);
        if (!warm || (!s.m24_valid && s.m24_saved < s.m24_cost * s.m24_wait)) return false;
    }
    if (capturing(st)) return false;
    const bool built = s.m24_valid;
    if (!ensure_mfma24(L, s, B, st)) return false;
    if (mode != 2 && !built && gain() < 0) {  // the overflow entries are more than estimated
        release(s);
        return false;
    }
    return true;
}

void launch_mfma24(Layer &L, DScatter &s, const ScaleView &sc, const float *in, int64_t in_ld, const float *inT,
                   float *xT, int64_t B, float *out, int64_t out_ld, hipStream_t st) {
    const int64_t ntile = (s.rows + 31) / 32, nkb = n_blocks(s.cols), nsteps = nkb * 4;
    const bool small = B <= SMALL_B;
    const int nt = operand_tiles(B);
    const int64_t chunks = small ? 1 : (nt + 3) / 4;
    const uint32_t epoch = ++L.m24_epoch;
    {
        ProfScope ps("mfma24_split", st);
        const SplitArgs a{in, in_ld, s.cols, B, sc.ent, xT, reinterpret_cast<__bf16 *>(L.ws_m24.p), L.m24_flag.p, epoch,
                          nsteps, nt};
        const dim3 grid(nblk(nsteps * nt * 64));
        if (small) launch(k_m24_split<true>, grid, dim3(TPB), 0, st, a);
        else launch(k_m24_split<false>, grid, dim3(TPB), 0, st, a);
    }
    ProfScope ps("mfma24", st);
    M24Args a{s.m24_val.p, s.m24_idx.p, s.m24_ovf_start.p, s.m24_ovf.p, s.rows, s.cols, nkb, ntile,
              reinterpret_cast<const __bf16 *>(L.ws_m24.p), L.m24_flag.p, epoch, inT, sc.ent, sc.row, B, out, out_ld,
              s.byte_start.p, s.elem_start.p, s.idx.p, s.val.p, nt};
    const int mt = row_tiles(Shape(s), B);
    if (small) {
        if (nt == 1) go_small<2, 1>(a, st);
        else go_small<2, 2>(a, st);
    } else if (nt == 1) {
        if (mt == 1) go<1, 1>(a, chunks, st);
        else go<2, 1>(a, chunks, st);
    } else if (nt == 2) {
        if (mt == 1) go<1, 2>(a, chunks, st);
        else go<2, 2>(a, chunks, st);
    } else {
        if (mt == 1) go<1, 4>(a, chunks, st);
        else go<2, 4>(a, chunks, st);
    }
    SILI_HIP(hipGetLastError());
}

}  // namespace sili
