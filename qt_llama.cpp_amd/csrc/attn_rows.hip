// attn_rows.hip -- attention of many query rows at once (the prefill of a
// chunk whose K/V rows are in the cache), exact path.
//
// Row z sits at position n_past0 + z and sees the last min(position + 1,
// limit) positions; per row and head the arithmetic is the decode form's
// (model.rs:1457-1590, kv_cache.rs:72-124, ops.rs:133-158):
//   s_t = (q . k_t, from -0.0 in dim order) * scale
//   p_t = expf(s_t - max) * (1 / (0 + e_0 + e_1 + ...))
//   out[d] = 0 + p_0 v_0[d] + p_1 v_1[d] + ...
// every product and add rounded by itself.
//
// Both contractions are therefore ordered chains of one multiply and one add
// per term, and the f32 VALU bounds them (measured on gfx950: 1.05 ns per
// wave instruction and SIMD with two or more waves there, 2.1 ns for a wave
// alone; a conversion, a v_fma_mix or a DPP operand costs 1.85).  Everything
// else is arranged so that little but those two instructions is issued:
//   - a wave runs M chain rows (row x query head) side by side, so one K or V
//     value, converted to f32 once, feeds M multiplies;
//   - the other factor (q in the scores, p in the weighted sum) is the same
//     for the whole wave: it comes through scalar loads into SGPRs, a step
//     ahead, and costs no LDS bandwidth and no vector instruction;
//   - K tiles go through LDS (lane = position); V is read straight from the
//     cache (lane = dim, coalesced), several batches ahead, with no barrier.
// At 512 rows x 8 heads of 256 dims behind 2048 positions this took the three
// launches from 593 us (two launches, a workgroup a row and kv head) to 340.
// Which of the forms below, or of decode.hip's, a call takes: plans.h.

#include <algorithm>

#include "attn_common.h"
#include "device.h"
#include "exact_sum.h"
#include "internal.h"

namespace mrml {

namespace {

typedef float f32x8u __attribute__((ext_vector_type(8), aligned(4)));
#define CONST_AS __attribute__((address_space(4)))
typedef const CONST_AS f32x8u *ConstF8;
typedef const CONST_AS float *ConstF;

__device__ __forceinline__ uint64_t uniform_addr(const void *p)
{
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a) |
           ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)) << 32);
}

// Scalar loads (and LDS reads) issued so far have arrived; loads issued after
// it stay after it, so they overlap the arithmetic that follows.
__device__ __forceinline__ void scalar_wait()
{
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
}

// ---- scores ------------------------------------------------------------------
// Workgroup (tile of 64 absolute positions that the block's rows can see, kv
// head, block of 4 * M * reps chain rows): the tile's K rows are staged in LDS
// once (row stride 16 bytes past the data: conflict-free 16-byte reads of 64
// rows), then wave w runs chain rows M at a time, lane p the chain of position
// T0 + p.  Chain row c of a kv head is row c / G, head c % G of the group.  Row
// blocks are taken in reverse order: the latest rows, with the most tiles, are
// dispatched first.
// First position of the workgroup's tile.  all: tile blockIdx.x of the launch's.
// Otherwise one of the gridDim.x tiles from the one that the block's first
// row's window (start0) starts in, each at a blockIdx.x that its number alone
// decides, so that blocks of rows find it in the same XCD's L2 and the workgroups
// past a block's last position fall to every XCD alike.  (The division is half
// a microsecond of scalar code, 3 % of a launch of a few rows.)
__device__ __forceinline__ int block_tile(int all, int start0, int t_lo)
{
    if (all) return t_lo + (int)blockIdx.x * kRowsP;
    const uint32_t n = gridDim.x, first = (uint32_t)(start0 - t_lo) / kRowsP;
    const int r = (int)blockIdx.x - (int)(first % n);
    return t_lo + ((int)first + (r < 0 ? r + (int)n : r)) * kRowsP;
}

template <int M>
__global__ __launch_bounds__(64 * kRowsW) void attn_rows_scores_kernel(
    const float *__restrict__ q, int q_stride, const uint16_t *__restrict__ k_cache, int n_past0, int nchains,
    int n_heads, int n_kv_heads, int head_dim, float scale, int capacity, int wlimit, int t_lo, int all_tiles,
    int reps, float *__restrict__ scores)
{
    extern __shared__ __align__(16) uint8_t k_s[];
    const int NT = 64 * kRowsW, HD = head_dim, KR = rows_k_stride(HD), G = n_heads / n_kv_heads;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = blockIdx.y, per = kRowsW * M * reps, c0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * per;
    const int cl = (c0 + per < nchains ? c0 + per : nchains) - 1;  // the block's last chain row
    int win0, start0;
    attn_window(nullptr, n_past0 + c0 / G, wlimit, win0, start0);
    const int T0 = block_tile(all_tiles, start0, t_lo), pos_l = n_past0 + cl / G;
    if (T0 > pos_l || start0 - T0 >= kRowsP) return;  // no row of the block has a position in this tile
    // one load a 128-byte line of the block's q rows, so that the scalar loads
    // below find them in this XCD's L2
    const int qlines = HD / 32, qrows = cl + 1 - c0;
    float touch = 0.0f;
    for (int i = tid; i < qrows * qlines; i += NT) {
        const int c = c0 + i / qlines, z = c / G;
        touch = q[(size_t)z * q_stride + (size_t)(kvh * G + c - z * G) * HD + 32 * (i % qlines)];
    }
    // K rows: thread -> 16-byte chunk tid % cpr of rows tid / cpr, + rpp, ...
    // Positions past the block's newest one reload that row; their scores are
    // not stored (with a test a load instead, each waits for the one before: 130
    // us against 124 at 500 rows of 8 x 512 dims).  The tile's rows follow the
    // first one's around the ring.
    const size_t kv_dim = (size_t)n_kv_heads * HD;
    const uint16_t *kh = k_cache + (size_t)kvh * HD;
    constexpr int kPer = 8;  // rows a thread loads before it stores any
    const int cpr = HD / 8, rpp = NT / cpr, rl = pos_l - T0 < kRowsP - 1 ? pos_l - T0 : kRowsP - 1;
    const int tr = tid / cpr, to = tid - tr * cpr, row0 = (int)cache_row_of(T0, capacity);
    if (tr < rpp) {
        for (int r0 = tr; r0 < kRowsP; r0 += kPer * rpp) {
            u32x4 tmp[kPer];
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                const int r = r0 + k * rpp;
                int row = row0 + (r < rl ? r : rl);
                row = capacity >= kRowsP ? (row >= capacity ? row - capacity : row) : row % capacity;
                tmp[k] = reinterpret_cast<const u32x4 *>(kh + row * kv_dim)[to];
            }
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                const int r = r0 + k * rpp;
                if (r < kRowsP) *reinterpret_cast<u32x4 *>(k_s + r * KR + to * 16) = tmp[k];
            }
        }
    }
    asm volatile("" ::"v"(touch));
    __syncthreads();
    const u32x4 *krow = reinterpret_cast<const u32x4 *>(k_s + lane * KR);
    const int t = T0 + lane, steps = HD / 8;
    for (int rep = 0; rep < reps; ++rep) {
        const int cw = c0 + (rep * kRowsW + wave) * M;
        if (cw >= nchains) return;
        uint64_t qa[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int c = cw + m < nchains ? cw + m : nchains - 1, z = c / G;
            qa[m] = uniform_addr(q + (size_t)z * q_stride + (size_t)(kvh * G + c - z * G) * HD);
        }
        float dot[M];
#pragma unroll
        for (int m = 0; m < M; ++m) dot[m] = -0.0f;
        f32x8u qs[2][M];
        u32x4 kw[2];
        auto fetch = [&](int s, int b) {
            kw[b] = krow[s];
#pragma unroll
            for (int m = 0; m < M; ++m) qs[b][m] = *reinterpret_cast<ConstF8>(qa[m] + (uint64_t)s * 32);
        };
        auto step = [&](int s, int b) {
            scalar_wait();
            fetch(s + 1 < steps ? s + 1 : s, b ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t w[4] = {kw[b].x, kw[b].y, kw[b].z, kw[b].w};
            // multiplies and adds in groups of 8 (the barriers): a multiply next to
            // its own add costs 1.47 ns an instruction and SIMD, groups 1.1
            float k[8];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                k[e] = f16_bits_to_f32(w[e >> 1] & 0xffffu);
                k[e + 1] = f16_bits_to_f32(w[e >> 1] >> 16);
            }
            constexpr int E = M >= 4 ? 2 : (M == 2 ? 4 : 8);  // dims a group
#pragma unroll
            for (int e0 = 0; e0 < 8; e0 += E) {
                float t[E][M];
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int m = 0; m < M; ++m) t[e][m] = qs[b][m][e0 + e] * k[e0 + e];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < E; ++e)
#pragma unroll
                    for (int m = 0; m < M; ++m) dot[m] = dot[m] + t[e][m];
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        fetch(0, 0);
        for (int s = 0; s < steps; s += 2) {  // head_dim is a multiple of 32
            step(s, 0);
            step(s + 1, 1);
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int c = cw + m, z = c / G;
            if (c < nchains) {
                int window, start;
                attn_window(nullptr, n_past0 + z, wlimit, window, start);
                if (t >= start && t < start + window)
                    scores[((size_t)z * n_heads + kvh * G + c - z * G) * capacity + (t - start)] = dot[m] * scale;
            }
        }
    }
}

// Quantised K rows (KF 1: Q8_0, 2: Q4_0): dot_head is the block-ordered fold
// s = s + (float)isum_b * (d_k * d_q) against the query's Q8_0 blocks
// (kv_cache.rs:73-95).  The same tiling: the tile's blocks are re-laid in LDS
// once (4-byte-aligned quants, f32 scales, odd row strides) and serve
// kRowsQC chain rows a pass, `reps` passes, four a wave.  One row a workgroup
// spent ten times its dots on that re-laying: 300 rows x 8 heads of 256 dims
// over a window of 512 took 143 us.
__host__ __device__ constexpr int rows_q_kstride(int kf, int nb) { return nb * (kf == 2 ? 4 : 8) + 1; }  // dwords
inline size_t rows_q_lds(int kf, int nb)
{
    return 4 * ((size_t)kRowsP * (rows_q_kstride(kf, nb) + (nb | 1)) + 3 + (size_t)kRowsQC * nb * 10);
}

template <int KF>
__global__ __launch_bounds__(64 * kRowsW) void attn_rows_scores_q_kernel(
    const float *__restrict__ q, int q_stride, const uint8_t *__restrict__ k_cache, int n_past0, int nchains,
    int n_heads, int n_kv_heads, int nb, float scale, int capacity, int wlimit, int t_lo, int all_tiles,
    int reps, float *__restrict__ scores)
{
    constexpr int M = kRowsQM, NT = 64 * kRowsW, BB = KF == 1 ? 34 : 18, QW = KF == 1 ? 8 : 4;
    extern __shared__ __align__(16) uint32_t q_lds[];
    const int HD = 32 * nb, KS = rows_q_kstride(KF, nb), DS = nb | 1, G = n_heads / n_kv_heads;
    uint32_t *kq = q_lds;                                                   // [64][KS] quants
    float *kd = reinterpret_cast<float *>(kq + kRowsP * KS);                // [64][DS] scales
    uint32_t *qq = q_lds + ((kRowsP * (KS + DS) + 3) & ~3);                 // [kRowsQC][nb][8] query quants
    float *qd = reinterpret_cast<float *>(qq + kRowsQC * nb * 8);           // [kRowsQC][nb] scales
    int *qs = reinterpret_cast<int *>(qd + kRowsQC * nb);                   // [kRowsQC][nb] quant sums
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = blockIdx.y, per = kRowsQC * reps, c0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * per;
    const int cl = (c0 + per < nchains ? c0 + per : nchains) - 1;  // the block's last chain row
    int win0, start0;
    attn_window(nullptr, n_past0 + c0 / G, wlimit, win0, start0);
    const int T0 = block_tile(all_tiles, start0, t_lo), pos_l = n_past0 + cl / G;
    if (T0 > pos_l || start0 - T0 >= kRowsP) return;  // no row of the block has a position in this tile
    {   // four threads a row, blocks tid % 4, + 4, ...
        const int r = tid >> 2, t = T0 + r <= pos_l ? T0 + r : pos_l;
        const uint8_t *krow = k_cache + (cache_row_of(t, capacity) * n_kv_heads + kvh) * ((size_t)nb * BB);
        for (int b = tid & 3; b < nb; b += 4) {
            const uint16_t *src = reinterpret_cast<const uint16_t *>(krow + b * BB);
            uint32_t h[2 * QW];
            const uint32_t d = src[0];
#pragma unroll
            for (int i = 0; i < 2 * QW; ++i) h[i] = src[1 + i];
            kd[r * DS + b] = f16_bits_to_f32(d);
#pragma unroll
            for (int i = 0; i < QW; ++i) kq[r * KS + b * QW + i] = h[2 * i] | (h[2 * i + 1] << 16);
        }
    }
    const int t = T0 + lane;
    for (int rep = 0; rep < reps; ++rep) {
        const int cp = c0 + rep * kRowsQC;
        if (cp >= nchains) return;
        __syncthreads();  // the tile is whole; the previous pass's queries are read
        // eight lanes a block (every lane takes part in the quantiser's reductions)
        for (int i0 = 0; i0 < kRowsQC * nb * 8; i0 += NT) {
            const int i = i0 + tid, l = i & 7, cb = i >> 3, ci = cb / nb, b = cb - ci * nb;
            const int c = cp + ci < nchains ? cp + ci : nchains - 1, z = c / G;
            const float *src = q + (size_t)z * q_stride + (size_t)(kvh * G + c - z * G) * HD + 32 * b + 4 * l;
            uint32_t dbits;
            int sum;
            const uint32_t v = q8_0_block8x4(make_float4(src[0], src[1], src[2], src[3]), dbits, sum);
            if (ci >= kRowsQC) continue;  // (whole waves, past the pass's queries)
            qq[i] = v;
            if (l == 0) {
                qd[cb] = f16_bits_to_f32(dbits);
                qs[cb] = sum;
            }
        }
        __syncthreads();
        float acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = 0.0f;
        for (int b = 0; b < nb; ++b) {
            uint32_t kw[8];
#pragma unroll
            for (int i = 0; i < QW; ++i) {
                const uint32_t w = kq[lane * KS + b * QW + i];
                if constexpr (KF == 1) {
                    kw[i] = w;
                } else {  // low nibbles pair with values 0..15, high ones with 16..31
                    kw[i] = w & 0x0F0F0F0Fu;
                    kw[4 + i] = (w >> 4) & 0x0F0F0F0Fu;
                }
            }
            const float d = kd[lane * DS + b];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int cb = (wave * M + m) * nb + b;
                const u32x4 q0 = *reinterpret_cast<const u32x4 *>(&qq[cb * 8]);
                const u32x4 q1 = *reinterpret_cast<const u32x4 *>(&qq[cb * 8 + 4]);
                int isum = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) isum = sdot4(kw[i], q0[i], isum);
#pragma unroll
                for (int i = 0; i < 4; ++i) isum = sdot4(kw[4 + i], q1[i], isum);
                if constexpr (KF == 2) isum -= 8 * qs[cb];  // (n - 8) . a = n . a - 8 * sum(a)
                const float term = (float)isum * (d * qd[cb]);
                acc[m] = acc[m] + term;
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int c = cp + wave * M + m, z = c / G;
            if (c < nchains) {
                int window, start;
                attn_window(nullptr, n_past0 + z, wlimit, window, start);
                if (t >= start && t < start + window)
                    scores[((size_t)z * n_heads + kvh * G + c - z * G) * capacity + (t - start)] = acc[m] * scale;
            }
        }
    }
}

// ---- softmax -----------------------------------------------------------------
// Workgroup (head, row): the row's scores become its weights, in place.  Each
// thread keeps four exps in registers for the register form of the exact
// sequential sum; windows past 4 * NT positions run in chunks of 4 * NT - 1,
// the running sum prepended to each as its first term (0 + s = s is exact, so
// the chunked sum is the one sequential loop).
template <int NT>
__global__ __launch_bounds__(NT) void attn_rows_softmax_kernel(float *__restrict__ scores, int n_past0, int n_heads,
                                                               int capacity, int wlimit, int expf_fused)
{
    __shared__ float red[NT / 64];
    __shared__ uint64_t exp_tab[32];
    __shared__ __align__(16) mrml_xsum::Shared4 xs;
    const int tid = threadIdx.x, z = (int)gridDim.y - 1 - (int)blockIdx.y;
    int window, start;
    attn_window(nullptr, n_past0 + z, wlimit, window, start);
    float *sc = scores + ((size_t)z * n_heads + blockIdx.x) * capacity;
    if (tid < 32) exp_tab[tid] = mrml_libm::kExpfT.t[tid];
    const bool fused = expf_fused != 0, one = window <= 4 * NT;
    float sv[4];
    float mx = -INFINITY;  // the max is exact in any order
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = 4 * tid + i;
        sv[i] = p < window ? sc[p] : -INFINITY;
        mx = fmaxf(mx, sv[i]);
    }
    for (int p = 4 * NT + tid; p < window; p += NT) mx = fmaxf(mx, sc[p]);
    mx = max32(mx);
    mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mx), 32)));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) mx = fmaxf(mx, red[w]);
    if (one) {
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            e[i] = 4 * tid + i < window ? mrml_libm::expf_t(sv[i] - mx, fused, exp_tab) : 0.0f;
        const float sum = mrml_xsum::block_seq_sum_nonneg4(make_float4(e[0], e[1], e[2], e[3]), window, xs);
        const float inv = sum > 0.0f ? 1.0f / sum : 1.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * tid + i < window) sc[4 * tid + i] = sum > 0.0f ? e[i] * inv : e[i];
        return;
    }
    constexpr int C = 4 * NT - 1;  // scores a chunk
    float sum = 0.0f;
    for (int c0 = 0; c0 < window; c0 += C) {
        const int n = window - c0 < C ? window - c0 : C;
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 4 * tid + i - 1;  // term 0 is the running sum
            e[i] = k < 0 ? sum : (k < n ? mrml_libm::expf_t(sc[c0 + k] - mx, fused, exp_tab) : 0.0f);
        }
        const float s = mrml_xsum::block_seq_sum_nonneg4(make_float4(e[0], e[1], e[2], e[3]), n + 1, xs);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 4 * tid + i - 1;
            if (k >= 0 && k < n) sc[c0 + k] = e[i];
        }
        sum = s;
        __syncthreads();  // the sum's LDS is reused
    }
    if (sum > 0.0f) {
        const float inv = 1.0f / sum;
        for (int c0 = 0; c0 < window; c0 += C) {  // each thread scales what it stored
            const int n = window - c0 < C ? window - c0 : C;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = 4 * tid + i - 1;
                if (k >= 0 && k < n) sc[c0 + k] = sc[c0 + k] * inv;
            }
        }
    }
}

// ---- weighted sum of values -----------------------------------------------------
// A wave owns M chain rows of a kv head and 64 * D dims (lane: D adjacent
// dims) over all their positions, with no LDS and no barrier.  Positions that
// every one of its rows sees run in batches of B without a test: V rows kNS-1
// batches ahead, weights one batch ahead.  The few at either end that only some
// rows see (rows M apart, sliding windows) are tested per row, in scalar code.
// Workgroups are dealt kv head first, so that an XCD (workgroups go to the
// eight in turn) reads few kv heads' V through its L2.
template <int VF, int D>
struct VVal {
    uint32_t q;  // D f16 values, or D quants
    uint32_t d;  // the block's f16 scale (quantised rows)
};

// VF 0: f16 rows.  VF 1 (Q8_0, 34-byte blocks) and 2 (Q4_0, 18-byte blocks):
// f16 scale, then the quants (Q4_0: dims 0..15 low nibbles, 16..31 high).
// Buffer loads: the row's offset is a scalar operand, the lane's offset one
// register for the whole kernel, so a load costs no vector address arithmetic
// (64-bit addresses took three VALU instructions a load).
template <int VF, int D>
__device__ __forceinline__ VVal<VF, D> v_load(__amdgpu_buffer_rsrc_t cache, uint32_t row, uint32_t off,
                                              uint32_t scale_off)
{
    VVal<VF, D> r;
    r.d = 0;
    if constexpr (VF == 0 && D == 2) {
        r.q = __builtin_amdgcn_raw_buffer_load_b32(cache, off, row, 0);
    } else if constexpr (VF == 0 || D == 2) {
        r.q = __builtin_amdgcn_raw_buffer_load_b16(cache, off, row, 0);
    } else {
        r.q = __builtin_amdgcn_raw_buffer_load_b8(cache, off, row, 0);
    }
    if constexpr (VF != 0) r.d = __builtin_amdgcn_raw_buffer_load_b16(cache, scale_off, row, 0);
    return r;
}

template <int VF, int D>
__device__ __forceinline__ float v_value(const VVal<VF, D> &r, int i, int shift)
{
    if constexpr (VF == 0) return f16_bits_to_f32((r.q >> (16 * i)) & 0xffffu);
    if constexpr (VF == 1) return (float)(int)(int8_t)((r.q >> (8 * i)) & 0xffu);
    return (float)((int)((r.q >> (8 * i + shift)) & 15u) - 8);
}

template <int VF, int M, int D>
__global__ __launch_bounds__(256) void attn_rows_pv_kernel(const float *__restrict__ p,
                                                           const uint8_t *__restrict__ v_cache, int n_past0,
                                                           int nchains, int n_heads, int n_kv_heads, int head_dim,
                                                           int capacity, int wlimit, int nblk, int nsl,
                                                           float *__restrict__ out)
{
    // Batches of 8 positions in two slots, so that the loop is short: its time
    // follows its length (512 rows behind 2048 positions: two slots of 8
    // positions 154 us, four 168, eight 198; the arithmetic alone is 80).  One
    // chain row a wave is bound by latency instead and takes four slots of 16.
    constexpr int B = M == 1 ? 16 : 8, NS = M == 1 ? 4 : 2;
    constexpr int kAhead = 128;  // positions
    constexpr int BB = VF == 0 ? 64 : (VF == 1 ? 34 : 18);  // cache bytes per 32 values
    const int HD = head_dim, G = n_heads / n_kv_heads;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int kvh = (int)(blockIdx.x % n_kv_heads), unit = (int)(blockIdx.x / n_kv_heads) * 4 + wave;
    const int cb = nblk - 1 - unit / nsl;  // the longest rows first
    if (cb < 0) return;
    const int d0 = (unit % nsl * 64 + lane) * D;
    const bool live = d0 < HD;
    const int dd = live ? d0 : 0;
    // the lane's dims within a cache row
    const uint32_t row_bytes = (uint32_t)(n_kv_heads * (HD / 32) * BB);
    const uint32_t blk = (uint32_t)((kvh * HD + dd) >> 5) * BB, in = (uint32_t)dd & 31;
    const uint32_t off = VF == 0 ? blk + 2 * in : (VF == 1 ? blk + 2 + in : blk + 2 + (in & 15));
    const int shift = VF == 2 && in >= 16 ? 4 : 0;

    // chain row m of the wave; formed anew where it is used (through the empty
    // asm), so that the main loop's scalar registers are its weights'
    auto chain = [&](int m, int &start, int &end, uint32_t &row) {
        int n = nchains;
        asm volatile("" : "+s"(n));
        const int c = cb * M + m < n ? cb * M + m : n - 1, z = c / G;
        int window;
        attn_window(nullptr, n_past0 + z, wlimit, window, start);
        end = n_past0 + z;
        row = (uint32_t)(z * n_heads + kvh * G + c - z * G);
    };
    int lo, hi, flo, fhi;
    uint64_t base;     // address of chain row 0's scores
    uint32_t rel[M];   // of each chain row's weight of position 0, from there (as if its window began at 0)
    {
        uint32_t row0;
        chain(0, lo, fhi, row0);
        base = uniform_addr(p + (size_t)row0 * capacity);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            uint32_t row;
            chain(m, flo, hi, row);
            rel[m] = (uint32_t)((row - row0) * (uint32_t)capacity - (uint32_t)(flo - lo)) * 4;
        }
    }
    const uint32_t cache_bytes = (uint32_t)capacity * row_bytes;  // < 2^32 (the launch checks)
    const __amdgpu_buffer_rsrc_t cache =
        __builtin_amdgcn_make_buffer_rsrc((void *)v_cache, (short)0, (int)cache_bytes, 0x00020000);

    float acc[M][D];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < D; ++i) acc[m][i] = 0.0f;

    // The lane's offsets of B consecutive cache rows: a batch then takes one
    // scalar offset, and no instruction but its loads (a wave issues one
    // instruction in about 2 ns, scalar ones too, so a row counter with its
    // wrap test a position would be a fourth of the loop).
    uint32_t voff[B], soff[VF == 0 ? 1 : B];
#pragma unroll
    for (int k = 0; k < B; ++k) {
        voff[k] = off + k * row_bytes;
        if constexpr (VF != 0) soff[k] = blk + k * row_bytes;
    }
    auto load_v = [&](VVal<VF, D> (&v)[B], uint32_t row) {
#pragma unroll
        for (int k = 0; k < B; ++k) v[k] = v_load<VF, D>(cache, row, voff[k], soff[VF == 0 ? 0 : k]);
    };
    auto add1 = [&](const VVal<VF, D> &v, int m, float w) {
        const float wd = VF == 0 ? w : f16_bits_to_f32(v.d) * w;
#pragma unroll
        for (int i = 0; i < D; ++i) acc[m][i] = acc[m][i] + wd * v_value<VF, D>(v, i, shift);
    };
    // positions t .. t+n-1 (n <= B), each row only those of its window
    auto part = [&](int t, int n) {
        VVal<VF, D> v[B];
        float w[M][B];
        int start[M], end[M];
        uint32_t row = (uint32_t)cache_row_of(t, capacity) * row_bytes;
#pragma unroll
        for (int k = 0; k < B; ++k) {  // (a cache row past the n positions too)
            v[k] = v_load<VF, D>(cache, row, voff[0], soff[0]);
            row += row_bytes;
            row = row == cache_bytes ? 0 : row;
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            uint32_t r;
            chain(m, start[m], end[m], r);
#pragma unroll
            for (int k = 0; k < B; ++k) {
                const int tk = std::min(std::max(t + k, start[m]), end[m]);
                w[m][k] = *reinterpret_cast<ConstF>(base + (uint32_t)(rel[m] + (uint32_t)(tk - lo) * 4));
            }
        }
#pragma unroll
        for (int k = 0; k < B; ++k)
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (k < n && t + k >= start[m] && t + k <= end[m]) add1(v[k], m, w[m][k]);
    };

    // the weights' lines of 32 positions, kAhead positions early: one vector
    // load brings them into this XCD's L2 (the softmax ran on another), where
    // the scalar loads then find them
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, -1, 0x00020000);
    uint32_t lane_rel = rel[0];
#pragma unroll
    for (int m = 1; m < M; ++m) lane_rel = (lane & (M - 1)) == m ? rel[m] : lane_rel;

    // nb whole batches from t on, the rows of all of them one after another in the cache
    auto batches = [&](int t, const int nb) {
        VVal<VF, D> v[NS][B];
        f32x8u w[2][M][B / 8];
        uint32_t touched;
        const uint32_t w_last = (uint32_t)(t - lo + (nb - 1) * B) * 4;
        uint32_t row = (uint32_t)cache_row_of(t, capacity) * row_bytes, wt = (uint32_t)(t - lo) * 4;
        const uint32_t row_last = row + (uint32_t)(nb - 1) * (B * row_bytes);
        // (loads past the last batch repeat it)
        auto load_w = [&](uint32_t o, int s) {
            o = o < w_last ? o : w_last;
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int j = 0; j < B / 8; ++j)
                    w[s][m][j] = *reinterpret_cast<ConstF8>(base + (uint32_t)(rel[m] + o) + 32 * j);
        };
        auto next_v = [&](VVal<VF, D> (&d)[B]) {
            load_v(d, row);
            row = row < row_last ? row + B * row_bytes : row;
        };
        auto batch = [&](int s) {  // slot s of NS, s & 1 of the weights
            scalar_wait();
            load_w(wt + 4 * B, (s & 1) ^ 1);
            if (s % (32 / B) == 0) {
                asm volatile("" ::"v"(touched));
                const uint32_t o = wt + 4 * kAhead;
                touched = __builtin_amdgcn_raw_buffer_load_b32(wbuf, lane_rel, o < w_last ? o : w_last, 0);
            }
            next_v(v[(s + NS - 1) % NS]);
            wt += 4 * B;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < B; ++k) {
                float vf[D];
#pragma unroll
                for (int i = 0; i < D; ++i) vf[i] = v_value<VF, D>(v[s][k], i, shift);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const float wk = w[s & 1][m][k / 8][k % 8];
                    const float wd = VF == 0 ? wk : f16_bits_to_f32(v[s][k].d) * wk;
#pragma unroll
                    for (int i = 0; i < D; ++i) acc[m][i] = acc[m][i] + wd * vf[i];
                }
            }
        };
        load_w(wt, 0);
        {   // lines 0..kAhead: lane m + M * j takes line j
            const uint32_t o = wt + 128 * (lane / M);
            touched = __builtin_amdgcn_raw_buffer_load_b32(wbuf, lane_rel + (o < w_last ? o : w_last), 0, 0);
        }
#pragma unroll
        for (int s = 0; s < NS - 1; ++s) next_v(v[s]);
        for (int b = 0;;) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                batch(s);
                if (++b == nb) return;
            }
        }
    };
    for (int t = lo; t <= hi;) {
        // positions from t on that every row sees, up to the ring's end
        const int left = capacity - (int)cache_row_of(t, capacity);
        const int common = t < flo ? 0 : (fhi + 1 - t < left ? fhi + 1 - t : left);
        if (common >= B) {
            batches(t, common / B);
            t += common / B * B;
        } else {
            int n = t < flo ? flo - t : (common > 0 && common == left ? common : hi + 1 - t);
            n = n < B ? n : B;
            part(t, n);
            t += n;
        }
    }

    if (live) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            int start, end;
            uint32_t row;
            chain(m, start, end, row);
            if (cb * M + m < nchains) {
                float *o = out + (size_t)row * HD + d0;
#pragma unroll
                for (int i = 0; i < D; ++i) o[i] = acc[m][i];
            }
        }
    }
}

// ---- softmax and weighted sum in one launch ---------------------------------------
// Workgroup (head, row) where every head has its own K/V head, short windows
// of f16 rows of 256 dims: thread d forms four weights (kept in LDS), then runs
// dim d's chain, 32 positions in flight, the first of them loaded ahead of the
// softmax.  Such a launch is bound by its latencies, so a second launch, or a
// softmax for each 32 dims, costs more than the kernels above save (the line
// and its figures: plans.h).
__global__ __launch_bounds__(kRowsShortHD) void attn_rows_short_kernel(const float *__restrict__ scores,
                                                                       const uint16_t *__restrict__ v_cache,
                                                                       int n_past0, int n_heads, int capacity,
                                                                       int wlimit, int expf_fused,
                                                                       float *__restrict__ out)
{
    constexpr int HD = kRowsShortHD, B = 32;
    __shared__ __align__(16) float p_s[kRowsShortMax];
    __shared__ float red[HD / 64];
    __shared__ uint64_t exp_tab[32];
    __shared__ __align__(16) mrml_xsum::Shared4 xs;
    const int h = blockIdx.x, z = (int)gridDim.y - 1 - (int)blockIdx.y, d = threadIdx.x;  // longest rows first
    int window, start;
    attn_window(nullptr, n_past0 + z, wlimit, window, start);
    const float *sc = scores + ((size_t)z * n_heads + h) * capacity;
    const size_t kv_dim = (size_t)n_heads * HD;
    const uint16_t *vb = v_cache + (size_t)h * HD + d;
    int row = (int)cache_row_of(start, capacity);  // the window's rows are consecutive modulo capacity
    // (rows past the window are cache rows too: they are loaded, not added)
    auto load = [&](uint16_t (&v)[B]) {
#pragma unroll
        for (int k = 0; k < B; ++k) {
            v[k] = vb[(size_t)row * kv_dim];
            row = row + 1 == capacity ? 0 : row + 1;
        }
    };
    uint16_t va[B], vn[B];
    load(va);  // in flight during the softmax
    if (d < 32) exp_tab[d] = mrml_libm::kExpfT.t[d];
    float sv[4], mx = -INFINITY;  // the max is exact in any order
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sv[i] = 4 * d + i < window ? sc[4 * d + i] : -INFINITY;
        mx = fmaxf(mx, sv[i]);
    }
    mx = max32(mx);
    mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mx), 32)));
    if ((d & 63) == 0) red[d >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        e[i] = 4 * d + i < window ? mrml_libm::expf_t(sv[i] - mx, expf_fused != 0, exp_tab) : 0.0f;
    const float sum = mrml_xsum::block_seq_sum_nonneg4(make_float4(e[0], e[1], e[2], e[3]), window, xs);
    const float inv = sum > 0.0f ? 1.0f / sum : 1.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (4 * d + i < window) p_s[4 * d + i] = sum > 0.0f ? e[i] * inv : e[i];
    __syncthreads();

    float acc = 0.0f;
    auto add = [&](const uint16_t (&v)[B], int t0) {
        if (t0 + B <= window) {
#pragma unroll
            for (int i = 0; i < B; i += 4) {
                const float4 p4 = *reinterpret_cast<const float4 *>(p_s + t0 + i);
                acc = acc + p4.x * f16_bits_to_f32(v[i]);
                acc = acc + p4.y * f16_bits_to_f32(v[i + 1]);
                acc = acc + p4.z * f16_bits_to_f32(v[i + 2]);
                acc = acc + p4.w * f16_bits_to_f32(v[i + 3]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < B; ++k)
                if (t0 + k < window) acc = acc + p_s[t0 + k] * f16_bits_to_f32(v[k]);
        }
    };
    for (int t0 = 0; t0 < window; t0 += 2 * B) {
        if (t0 + B < window) load(vn);  // in flight while va is added
        add(va, t0);
        if (t0 + 2 * B < window) load(va);
        if (t0 + B < window) add(vn, t0 + B);
    }
    out[((size_t)z * n_heads + h) * HD + d] = acc;
}

}  // namespace

int load_attn_rows(mrml_hip_ctx *ctx)
{
    if (ctx->rows_loaded) return MRML_HIP_OK;
    hipFuncAttributes attr;
    if (hipError_t e = hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(attn_rows_short_kernel)))
        return hip_fail(ctx, e, "attn_rows_short_kernel");
    ctx->rows_loaded = true;
    return MRML_HIP_OK;
}

int launch_attn_rows_short(mrml_hip_ctx *ctx, const float *scores, const void *v_cache, float *out, int n_past0,
                           int rows, int n_heads, int capacity, int wlimit)
{
    hipLaunchKernelGGL(attn_rows_short_kernel, dim3(n_heads, rows), dim3(kRowsShortHD), 0, ctx->stream, scores,
                       (const uint16_t *)v_cache, n_past0, n_heads, capacity, wlimit, (int)host_expf_fused(), out);
    return check_launch(ctx, "attn_rows_short_kernel");
}

int launch_attn_rows_scores(mrml_hip_ctx *ctx, const AttnRowsPlan &plan, const float *q, int q_stride,
                            const void *k_cache, int n_past0, int rows, int n_heads, int n_kv_heads, int head_dim,
                            int k_fmt, float scale, int capacity, int wlimit, float *scores)
{
    const int nchains = rows * (n_heads / n_kv_heads), t_lo = plan.t_lo, reps = plan.score_reps,
              all = plan.all_tiles;
    const dim3 grid((unsigned)plan.tiles, (unsigned)n_kv_heads, (unsigned)plan.score_blocks(nchains));
    if (k_fmt != 0) {
#define ROWS_SCQ(KF)                                                                                               \
    hipLaunchKernelGGL(attn_rows_scores_q_kernel<KF>, grid, dim3(64 * kRowsW), rows_q_lds(KF, head_dim / 32),       \
                       ctx->stream, q, q_stride, (const uint8_t *)k_cache, n_past0, nchains, n_heads, n_kv_heads,   \
                       head_dim / 32, scale, capacity, wlimit, t_lo, all, reps, scores)
        if (k_fmt == 1) ROWS_SCQ(1);
        else ROWS_SCQ(2);
#undef ROWS_SCQ
        return check_launch(ctx, "attn_rows_scores_q_kernel");
    }
    const size_t lds = (size_t)kRowsP * rows_k_stride(head_dim);
#define ROWS_SC(M)                                                                                               \
    hipLaunchKernelGGL(attn_rows_scores_kernel<M>, grid, dim3(64 * kRowsW), lds, ctx->stream, q, q_stride,          \
                       (const uint16_t *)k_cache, n_past0, nchains, n_heads, n_kv_heads, head_dim, scale, capacity, \
                       wlimit, t_lo, all, reps, scores)
    if (plan.score_m == 4) ROWS_SC(4);
    else if (plan.score_m == 2) ROWS_SC(2);
    else ROWS_SC(1);
#undef ROWS_SC
    return check_launch(ctx, "attn_rows_scores_kernel");
}

// Softmax in place over the scores, then the weighted sum of values.
int launch_attn_rows_softmax_v(mrml_hip_ctx *ctx, const AttnRowsPlan &plan, float *scores, const void *v_cache,
                               float *out, int n_past0, int rows, int n_heads, int n_kv_heads, int head_dim, int v_fmt,
                               int capacity, int wlimit)
{
    const int fe = (int)host_expf_fused(), nt = plan.softmax_threads;
    const dim3 sgrid((unsigned)n_heads, (unsigned)rows);
#define ROWS_SM(NT)                                                                                              \
    hipLaunchKernelGGL(attn_rows_softmax_kernel<NT>, sgrid, dim3(NT), 0, ctx->stream, scores, n_past0, n_heads,   \
                       capacity, wlimit, fe)
    if (nt == 64) ROWS_SM(64);
    else if (nt == 256) ROWS_SM(256);
    else if (nt == 512) ROWS_SM(512);
    else ROWS_SM(1024);
#undef ROWS_SM
    if (int rc = check_launch(ctx, "attn_rows_softmax_kernel")) return rc;

    const int nchains = rows * (n_heads / n_kv_heads);
    const uint8_t *v = reinterpret_cast<const uint8_t *>(v_cache);
#define ROWS_PV(VF, M, D)                                                                                          \
    do {                                                                                                           \
        const int nblk = (nchains + M - 1) / M, nsl = (head_dim + 64 * D - 1) / (64 * D);                          \
        const unsigned wgs = (unsigned)(((int64_t)nblk * nsl + 3) / 4) * (unsigned)n_kv_heads;                     \
        hipLaunchKernelGGL((attn_rows_pv_kernel<VF, M, D>), dim3(wgs), dim3(256), 0, ctx->stream, scores, v,       \
                           n_past0, nchains, n_heads, n_kv_heads, head_dim, capacity, wlimit, nblk, nsl, out);     \
    } while (0)
#define ROWS_PV_MD(VF)  /* (4 x 1 over Q8_0: never chosen, not built) */                                           \
    do {                                                                                                           \
        if (plan.pv_m == 4 && (VF == 1 || plan.pv_d == 2)) ROWS_PV(VF, 4, 2);                                      \
        else if (plan.pv_m == 4) ROWS_PV(VF, 4, (VF == 1 ? 2 : 1));                                                \
        else if (plan.pv_m == 2) ROWS_PV(VF, 2, 1);                                                                \
        else ROWS_PV(VF, 1, 1);                                                                                    \
    } while (0)
    if (v_fmt == 0) ROWS_PV_MD(0);
    else if (v_fmt == 1) ROWS_PV_MD(1);
    else ROWS_PV_MD(2);
#undef ROWS_PV_MD
#undef ROWS_PV
    return check_launch(ctx, "attn_rows_pv_kernel");
}

}  // namespace mrml
