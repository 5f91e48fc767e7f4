// Causal attention of single rows over a paged key/value cache, in true 32-bit arithmetic.
//
// Row t of the request in slot[t] at position pos[t] sees the
// keys at positions lo .. pos[t] of its own request, lo = max(0, pos - window + 1) with a window,
// the start of the row's chunk, pos - pos % chunk, with a mask cut into chunks, and 0 without either;
// query head h uses key/value head h / (n_heads / n_kv).  Scores are scaled by `scale` (the caller's,
// 1/sqrt(hd) by default) after the dot product (src/model/transformer.cpp:228-255, src/gpu/device_kernels.inc:377-449).  The softmax's
// denominator is a 64-bit sum over groups of keys, as the reference's (src/kernels/kernels.cpp:95-100): a 32-bit
// running sum over tens of thousands of keys loses digits that every output of the head then lacks.
// The order of every sum depends on (pos, window, chunk, hd) only, so a row's result has the same bits
// whatever else is in the batch and whichever pages hold its request.
//
// With `cap` > 0 a scaled score s becomes cap * tanh(s / cap) before the softmax.
// With `sinks` [n_heads] the softmax's denominator also holds exp(sinks[h]): a score that has no key and no value (the
// running maximum starts there and the running sum at 1).  With `gate` the head's output is multiplied by
// sigmoid(gate[t * gate_stride + h]), or, with gate_channels = vd, channel d of it by sigmoid(gate[t * gate_stride + h * vd + d]).
//
// Cache of one layer: per page the keys [kv_head][place][hd], then the values transposed
// [kv_head][vd][place] (vd channels a value head, hd a key head); table[slot][i] is the page of
// positions i*page_size .. (i+1)*page_size - 1.
//
// Two kernels.  Which one serves depends on the data types and on hd, vd, the page size, the window and the chunk alone, so one layer meets one of them:
//   tiles    32-bit throughout, hd and vd multiples of 16 up to 128, pages of a multiple of 4, rows that may see more than 16 keys: both products
//            on the 32-bit matrix instructions, four waves a workgroup, long contexts shared out over workgroups (in blocks of 64 keys, by a kernel of the same sums, where the tiles are few);
//   rows     everything else: one wave per (row, query head), keys 64 at a time.
#include "common.h"

namespace {

constexpr int MAX_HD = 640;

// --------------------------------------------------------------------------------------------- tiles
// A workgroup takes up to 16 (row, query head) pairs of one key/value head: the heads that share it, for one row (decoding) or for
// several neighbouring rows of the batch.  Keys are taken in spans of 256 positions that start at multiples of 256, a block of 64 to each
// of the four waves.  A block gives, for each pair, the largest score m, the sum l of exp(s - m) and O = sum of exp(s - m) v; the
// span's four blocks meet in LDS (largest m first, then the scaled l and O in order), and spans are merged one behind the other in
// order of position, either by the workgroup itself or, where the context is shared out (`part`), by the second kernel: the same
// operations either way.
// The scores of 16 keys come out of the matrix instruction in the very registers in which the second product wants the probabilities
// (a lane has the keys 4g .. 4g+3 of pair r), and the cache's transposed values are 16-byte pieces along the keys: nothing is laid
// out anew.  Bound by the latency of a span's loads (all of a wave's keys and values are asked for at once) until the contexts are
// long; one wave per (row, head) that walked its keys 64 at a time, every lane a key of its own, took 169 us a layer for 3 rows at 600
// positions of the Llama-3.2-1B shape and 215 for a prompt of 301.
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int BLOCK = 64, SPAN = 4 * BLOCK, PAIRS = 16, MAX_SPANS = 65535;

// A span joins what came before it (m, l, and every O with the two factors): nothing happens for a row that sees no key of the span, which its
// positions tell and not the scores (a score that is no number does not show in the largest one: the row's sums must hand it on, and so must
// a value that is none, whatever factor it meets).
struct Join { float before, span; };             // span < 0: the row sees none of it
__device__ __forceinline__ Join join(float& m, double& l, bool sees, float m_span, double l_span) {
    if (!sees) return {1.f, -1.f};
    const float top = fmaxf(m, m_span);
    // (m = -inf at the first span without sinks: 0; both -inf: sums of zeros, or ones that are no numbers)
    const Join f = top == -INFINITY ? Join{1.f, 1.f} : Join{expf(m - top), expf(m_span - top)};
    l = fma(l_span, (double)f.span, l * (double)f.before);
    m = top;
    return f;
}
__device__ __forceinline__ float joined(float o, float o_span, Join f) { return f.span < 0.f ? o : fmaf(o_span, f.span, o * f.before); }

__device__ __forceinline__ int first_key(int pos, int window, int chunk) {
    int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    return chunk > 0 ? max(lo, pos - pos % chunk) : lo;
}

// what becomes of a head's channel in the end
__device__ __forceinline__ float finished(float o, double l, const float* gate, long gate_stride, int gate_channels, int t, int h, int d) {
    float inv = 1.0f / (float)l;
    if (gate && !gate_channels) inv *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_stride + h]));
    o *= inv;
    if (gate && gate_channels) o *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_stride + (size_t)h * gate_channels + d]));
    return o;
}

// One (row, head, span) of `part`: vd sums, then l (64-bit), then m.
__host__ __device__ constexpr int part_floats(int vd) { return vd + 4; }

// n / size for n >= 0, without the division (magic = floor(2^32 (2^shift - size) / size) + 1, shift = ceil(log2(size)))
struct Divisor { int size; unsigned magic; int shift; };
__device__ __forceinline__ int quotient(int n, const Divisor& by) { return (int)((__umulhi(by.magic, (unsigned)n) + (unsigned)n) >> by.shift); }

template <int D>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void attention_exact_tiles_kernel(const float* __restrict__ q, const float* __restrict__ cache, float* __restrict__ out,
                                                                   const int* __restrict__ pos, const int* __restrict__ slot, const int* __restrict__ table,
                                                                   int table_stride, long page_stride, Divisor pages, int n_rows, int n_heads, int n_kv, int hd, int vd,
                                                                   int window, int chunk, float scale, float cap, const float* __restrict__ sinks,
                                                                   const float* __restrict__ gate, long gate_stride, int gate_channels, int n_single, int rows_a_tile,
                                                                   float* __restrict__ part, int n_spans) {
    __shared__ float o_s[4][PAIRS][D + 4];
    __shared__ float m_s[4][PAIRS], l_s[4][PAIRS], f_s[4][PAIRS];        // of the blocks; f: their factors, negative where the pair sees none of the block's keys
    __shared__ float m_all[PAIRS];
    __shared__ double l_all[PAIRS];
    __shared__ Join join_s[PAIRS];
    __shared__ int t_s[PAIRS], h_s[PAIRS], run_s[PAIRS], lo_s[PAIRS], pos_s[PAIRS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int group = n_heads / n_kv, head_tiles = (group + PAIRS - 1) / PAIRS;
    const int tile = blockIdx.x / (n_kv * head_tiles), kv = blockIdx.x / head_tiles % n_kv, ht = blockIdx.x % head_tiles;
    const int heads_here = min(PAIRS, group - ht * PAIRS);
    const int rows_here = tile < n_single ? 1 : rows_a_tile, t_first = tile < n_single ? tile : n_single + (tile - n_single) * rows_a_tile;
    const int place = r / heads_here, t = t_first + place, h = kv * group + ht * PAIRS + r % heads_here;
    const bool valid = place < rows_here && t < n_rows;
    const int my_pos = valid ? pos[t] : 0, my_slot = valid ? slot[t] : -1, my_lo = valid ? first_key(my_pos, window, chunk) : 0;
    f32x4 qv[D / 16];
#pragma unroll
    for (int c = 0; c < D / 16; ++c)
        qv[c] = valid && c * 16 < hd ? *reinterpret_cast<const f32x4*>(q + ((size_t)t * n_heads + h) * hd + c * 16 + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
    const int page_size = pages.size;
    const long v_plane = (long)n_kv * page_size * hd;   // from a page's keys to its values

    // Rows of one request at a time: a tile with rows of several requests takes as many turns, shared out over gridDim.z workgroups.  (One after the
    // other, with single rows in such tiles too, they took 237 us where a wave per (row, head) takes 39: 16 requests of one row at 100 positions and a
    // prompt of 48 rows, 16 heads of 128 with keys of their own; 37 now.)
    bool todo = valid;
    unsigned turn = 0;
    while (__ballot(todo) != 0) {
        const int run_slot = __shfl(my_slot, (int)__ffsll((unsigned long long)__ballot(todo)) - 1, 64);
        const bool in_run = todo && my_slot == run_slot;
        todo = todo && !in_run;
        if (turn++ % gridDim.z != blockIdx.z) continue;
        int lo_min = in_run ? my_lo : 2147483647, lo_max = in_run ? my_lo : 0, p_min = in_run ? my_pos : 2147483647, p_max = in_run ? my_pos : 0;
#pragma unroll
        for (int off = 1; off < PAIRS; off <<= 1) {
            lo_min = min(lo_min, __shfl_xor(lo_min, off, 64));
            lo_max = max(lo_max, __shfl_xor(lo_max, off, 64));
            p_min = min(p_min, __shfl_xor(p_min, off, 64));
            p_max = max(p_max, __shfl_xor(p_max, off, 64));
        }
        lo_min = __builtin_amdgcn_readfirstlane(lo_min);
        p_max = __builtin_amdgcn_readfirstlane(p_max);
        const int* tab = table + (size_t)run_slot * table_stride;
        if (tid < PAIRS) {
            m_all[tid] = sinks && valid ? sinks[h] : -INFINITY;
            l_all[tid] = sinks ? 1.0 : 0.0;
            t_s[tid] = t; h_s[tid] = h; run_s[tid] = in_run; lo_s[tid] = my_lo; pos_s[tid] = my_pos;
        }
        float o_all[PAIRS * D / 256];
#pragma unroll
        for (int e = 0; e < PAIRS * D / 256; ++e) o_all[e] = 0.f;

        for (int s = lo_min / SPAN + blockIdx.y; s <= p_max / SPAN; s += gridDim.y) {
            const int b0 = s * SPAN + wave * BLOCK;
            float m = -INFINITY, l = 0.f;
            if (b0 <= p_max && b0 + BLOCK > lo_min) {                     // (the same for the wave)
                // Groups of 16 keys that no row of the tile sees are loaded (from a place that one does see) and left out.  A wave alone on its SIMD
                // takes seven clocks or so an instruction, and at short contexts and windows a span is little else.
                bool live[4];
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) live[kt] = b0 + kt * 16 <= p_max && b0 + kt * 16 + 16 > lo_min;
                f32x4 kk[4][D / 16], vv[4][D / 16];
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    const int key = max(min(b0 + kt * 16 + r, p_max), lo_min);
                    const int page = quotient(key, pages);
                    const float* from = cache + (size_t)tab[page] * page_stride + ((size_t)kv * page_size + key - page * page_size) * hd + 4 * g;
#pragma unroll
                    for (int c = 0; c < D / 16; ++c) kk[kt][c] = c * 16 < hd ? *reinterpret_cast<const f32x4*>(from + c * 16) : f32x4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    const int first = b0 + kt * 16 + 4 * g, key = max(min(first, p_max), lo_min) & ~3;
                    const int page = quotient(key, pages);
                    const float* from = cache + (size_t)tab[page] * page_stride + v_plane + ((size_t)kv * vd + r) * page_size + key - page * page_size;
#pragma unroll
                    for (int c = 0; c < D / 16; ++c) vv[kt][c] = c * 16 < vd ? *reinterpret_cast<const f32x4*>(from + (size_t)c * 16 * page_size) : f32x4{0.f, 0.f, 0.f, 0.f};
                }
                f32x4 sc[4];
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    sc[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (!live[kt]) continue;
#pragma unroll
                    for (int c = 0; c < D / 16; ++c)
                        if (c * 16 < hd) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) sc[kt] = mfma(kk[kt][c][j], qv[c][j], sc[kt]);
                        }
                }
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    if (!live[kt]) continue;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = b0 + kt * 16 + 4 * g + i;
                        float x = sc[kt][i] * scale;
                        if (cap > 0.f) x = cap * tanhf(x / cap);
                        sc[kt][i] = in_run && key <= my_pos && key >= my_lo ? x : -INFINITY;
                        m = fmaxf(m, sc[kt][i]);
                    }
                }
                m = fmaxf(m, __shfl_xor(m, 16, 64));
                m = fmaxf(m, __shfl_xor(m, 32, 64));
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    if (!live[kt]) continue;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        sc[kt][i] = sc[kt][i] == -INFINITY ? 0.f : expf(sc[kt][i] - m);
                        l += sc[kt][i];
                    }
                }
                l += __shfl_xor(l, 16, 64);
                l += __shfl_xor(l, 32, 64);
                // A probability of zero must not meet a value that is no number: places nobody has written, and, where some pair of the
                // tile does not see all of the block, values a pair does not see (rare: then every row's own sum with those left out).
                bool odd = false;
                const bool all_seen = b0 >= lo_max && b0 + BLOCK - 1 <= p_min;
                if (!all_seen) {
#pragma unroll
                    for (int kt = 0; kt < 4; ++kt) {
                        if (!live[kt]) continue;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int key = b0 + kt * 16 + 4 * g + i;
#pragma unroll
                            for (int c = 0; c < D / 16; ++c) {
                                if (key > p_max || key < lo_min) vv[kt][c][i] = 0.f;
                                odd = odd || !(fabsf(vv[kt][c][i]) < INFINITY);
                            }
                        }
                    }
                }
                f32x4 o[D / 16];
#pragma unroll
                for (int c = 0; c < D / 16; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    if (!live[kt]) continue;
#pragma unroll
                    for (int c = 0; c < D / 16; ++c)
                        if (c * 16 < vd) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) o[c] = mfma(vv[kt][c][j], sc[kt][j], o[c]);
                        }
                }
                if (__ballot(odd) != 0) {
                    for (int row = 0; row < rows_here; ++row) {
                        const int row_pos = __shfl(my_pos, row * heads_here, 64), row_lo = __shfl(my_lo, row * heads_here, 64);
#pragma unroll
                        for (int c = 0; c < D / 16; ++c) {
                            f32x4 own = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                            for (int kt = 0; kt < 4; ++kt) {
                                if (!live[kt]) continue;
#pragma unroll
                                for (int j = 0; j < 4; ++j) {
                                    const int key = b0 + kt * 16 + 4 * g + j;
                                    own = mfma(key > row_pos || key < row_lo ? 0.f : vv[kt][c][j], sc[kt][j], own);
                                }
                            }
                            if (place == row) o[c] = own;
                        }
                    }
                }
#pragma unroll
                for (int c = 0; c < D / 16; ++c)
                    if (c * 16 < vd) *reinterpret_cast<f32x4*>(&o_s[wave][r][c * 16 + 4 * g]) = o[c];
            }
            if (g == 0) { m_s[wave][r] = m; l_s[wave][r] = l; }
            __syncthreads();
            if (tid < PAIRS) {
                float top = -INFINITY;
#pragma unroll
                for (int b = 0; b < 4; ++b) top = fmaxf(top, m_s[b][tid]);
                double sum = 0.0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const bool sees = in_run && s * SPAN + b * BLOCK <= my_pos && s * SPAN + (b + 1) * BLOCK > my_lo;      // (lane `tid` has pair `tid`)
                    const float f = m_s[b][tid] == -INFINITY ? 0.f : expf(m_s[b][tid] - top);
                    f_s[b][tid] = sees ? f : -1.f;
                    if (sees) sum = fma((double)l_s[b][tid], (double)f, sum);
                }
                if (part) {
                    const int at = s - lo_s[tid] / SPAN;
                    if (run_s[tid] && at >= 0 && s <= pos_s[tid] / SPAN && at < n_spans) {
                        float* p = part + (((size_t)t_s[tid] * n_heads + h_s[tid]) * n_spans + at) * part_floats(vd) + vd;
                        *reinterpret_cast<double*>(p) = sum;
                        p[2] = top;
                    }
                } else {
                    float m_now = m_all[tid];
                    double l_now = l_all[tid];
                    join_s[tid] = join(m_now, l_now, in_run && s * SPAN <= my_pos && (s + 1) * SPAN > my_lo, top, sum);
                    m_all[tid] = m_now;
                    l_all[tid] = l_now;
                }
            }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < PAIRS * D / 256; ++e) {
                const int pair = (tid + 256 * e) / D, d = (tid + 256 * e) % D;
                if (d >= vd) continue;
                float o = 0.f;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float f = f_s[b][pair];
                    if (!(f < 0.f)) o = fmaf(o_s[b][pair][d], f, o);       // (a block the pair sees nothing of may have left nothing there)
                }
                if (part) {
                    const int span = s - lo_s[pair] / SPAN;
                    if (run_s[pair] && span >= 0 && s <= pos_s[pair] / SPAN && span < n_spans)
                        part[(((size_t)t_s[pair] * n_heads + h_s[pair]) * n_spans + span) * part_floats(vd) + d] = o;
                } else {
                    o_all[e] = joined(o_all[e], o, join_s[pair]);
                }
            }
            __syncthreads();
        }
        if (!part) {
#pragma unroll
            for (int e = 0; e < PAIRS * D / 256; ++e) {
                const int pair = (tid + 256 * e) / D, d = (tid + 256 * e) % D;
                if (d < vd && run_s[pair])
                    out[((size_t)t_s[pair] * n_heads + h_s[pair]) * vd + d] = finished(o_all[e], l_all[pair], gate, gate_stride, gate_channels, t_s[pair], h_s[pair], d);
            }
        }
        __syncthreads();                                  // the next turn writes the pairs' numbers anew
    }
}

// The same numbers where the tiles are few: a workgroup per block of 64 keys, its four waves each with 16 of the keys for the scores and with every fourth 16 channels for the second product
// (the probabilities change hands in LDS).  Every sum is the one above, of the same operands in the same order.  What a block gives is left in `part` (per (row, head, block): vd
// sums, then l and m); the meeting of a span's blocks is the join kernel's too.  Bound by a wave's chain of
// instructions, which is a third of the one above, and by its loads' two round trips.  With the join, spans to a workgroup and blocks: 3 rows at 600 positions, 32/8 heads of 64, 17.5 us and 10.7;
// 1 row 15.3 and 9.6, 8 rows at 1,000 18.1 and 15.7; 24/8 heads of 128, 3 rows at 600 25.7 and 12.9, 16 at 1,000 51 and 41.
template <int D>
__global__ __launch_bounds__(256, 2) void attention_exact_blocks_kernel(const float* __restrict__ q, const float* __restrict__ cache, const int* __restrict__ pos, const int* __restrict__ slot,
                                                                       const int* __restrict__ table, int table_stride, long page_stride, Divisor pages, int n_rows, int n_heads, int n_kv,
                                                                       int hd, int vd, int window, int chunk, float scale, float cap, int n_single, int rows_a_tile, float* __restrict__ part,
                                                                       int n_blocks) {
    constexpr int OWN = D / 64;                                    // groups of 16 channels a wave has: wave, wave + 4, ...
    __shared__ float m_s[4][PAIRS];
    __shared__ f32x4 p_s[4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
    const int group = n_heads / n_kv, head_tiles = (group + PAIRS - 1) / PAIRS;
    const int tile = blockIdx.x / (n_kv * head_tiles), kv = blockIdx.x / head_tiles % n_kv, ht = blockIdx.x % head_tiles;
    const int heads_here = min(PAIRS, group - ht * PAIRS);
    const int rows_here = tile < n_single ? 1 : rows_a_tile, t_first = tile < n_single ? tile : n_single + (tile - n_single) * rows_a_tile;
    const int place = r / heads_here, t = t_first + place, h = kv * group + ht * PAIRS + r % heads_here;
    const bool valid = place < rows_here && t < n_rows;
    const int my_pos = valid ? pos[t] : 0, my_slot = valid ? slot[t] : -1, my_lo = valid ? first_key(my_pos, window, chunk) : 0;
    f32x4 qv[D / 16];
#pragma unroll
    for (int c = 0; c < D / 16; ++c)
        qv[c] = valid && c * 16 < hd ? *reinterpret_cast<const f32x4*>(q + ((size_t)t * n_heads + h) * hd + c * 16 + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
    const int page_size = pages.size;
    const long v_plane = (long)n_kv * page_size * hd;
    bool todo = valid;
    unsigned turn = 0;
    while (__ballot(todo) != 0) {                                  // (a request's rows at a time, as above)
        const int run_slot = __builtin_amdgcn_readfirstlane(__shfl(my_slot, (int)__ffsll((unsigned long long)__ballot(todo)) - 1, 64));
        const bool in_run = todo && my_slot == run_slot;
        todo = todo && !in_run;
        if (turn++ % gridDim.z != blockIdx.z) continue;
        int lo_min = in_run ? my_lo : 2147483647, lo_max = in_run ? my_lo : 0, p_min = in_run ? my_pos : 2147483647, p_max = in_run ? my_pos : 0;
#pragma unroll
        for (int off = 1; off < PAIRS; off <<= 1) {
            lo_min = min(lo_min, __shfl_xor(lo_min, off, 64));
            lo_max = max(lo_max, __shfl_xor(lo_max, off, 64));
            p_min = min(p_min, __shfl_xor(p_min, off, 64));
            p_max = max(p_max, __shfl_xor(p_max, off, 64));
        }
        lo_min = __builtin_amdgcn_readfirstlane(lo_min);
        p_max = __builtin_amdgcn_readfirstlane(p_max);
        const int* tab = table + (size_t)run_slot * table_stride;
        for (int block = lo_min / BLOCK + blockIdx.y; block <= p_max / BLOCK; block += gridDim.y) {
            const int b0 = block * BLOCK;
            bool live[4];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) live[kt] = b0 + kt * 16 <= p_max && b0 + kt * 16 + 16 > lo_min;
            f32x4 kk[D / 16], vv[4][OWN];
            {
                const int key = max(min(b0 + wave * 16 + r, p_max), lo_min), page = quotient(key, pages);
                const float* from = cache + (size_t)tab[page] * page_stride + ((size_t)kv * page_size + key - page * page_size) * hd + 4 * g;
#pragma unroll
                for (int c = 0; c < D / 16; ++c) kk[c] = c * 16 < hd ? *reinterpret_cast<const f32x4*>(from + c * 16) : f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                const int key = max(min(b0 + kt * 16 + 4 * g, p_max), lo_min) & ~3, page = quotient(key, pages);
                const float* from = cache + (size_t)tab[page] * page_stride + v_plane + ((size_t)kv * vd + r) * page_size + key - page * page_size;
#pragma unroll
                for (int e = 0; e < OWN; ++e) {
                    const int c = wave + 4 * e;
                    vv[kt][e] = c * 16 < vd ? *reinterpret_cast<const f32x4*>(from + (size_t)c * 16 * page_size) : f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
            f32x4 sc = {0.f, 0.f, 0.f, 0.f};
            float m = -INFINITY;
            const bool mine = b0 + wave * 16 <= p_max && b0 + wave * 16 + 16 > lo_min;
            if (mine) {
#pragma unroll
                for (int c = 0; c < D / 16; ++c)
                    if (c * 16 < hd) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) sc = mfma(kk[c][j], qv[c][j], sc);
                    }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = b0 + wave * 16 + 4 * g + i;
                    float x = sc[i] * scale;
                    if (cap > 0.f) x = cap * tanhf(x / cap);
                    sc[i] = in_run && key <= my_pos && key >= my_lo ? x : -INFINITY;
                    m = fmaxf(m, sc[i]);
                }
                m = fmaxf(m, __shfl_xor(m, 16, 64));
                m = fmaxf(m, __shfl_xor(m, 32, 64));
            }
            if (g == 0) m_s[wave][r] = m;
            __syncthreads();
            m = fmaxf(fmaxf(m_s[0][r], m_s[1][r]), fmaxf(m_s[2][r], m_s[3][r]));
            if (mine) {
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[i] = sc[i] == -INFINITY ? 0.f : expf(sc[i] - m);
                p_s[wave][lane] = sc;
            }
            __syncthreads();
            f32x4 p[4];
            float l = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                p[kt] = p_s[kt][lane];                             // (nobody has written what is not live)
                if (!live[kt]) continue;
#pragma unroll
                for (int i = 0; i < 4; ++i) l += p[kt][i];
            }
            l += __shfl_xor(l, 16, 64);
            l += __shfl_xor(l, 32, 64);
            __syncthreads();                                       // the next block writes them anew
            bool odd = false;                                      // (values that are no numbers: as above)
            if (!(b0 >= lo_max && b0 + BLOCK - 1 <= p_min)) {
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    if (!live[kt]) continue;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = b0 + kt * 16 + 4 * g + i;
#pragma unroll
                        for (int e = 0; e < OWN; ++e) {
                            if (key > p_max || key < lo_min) vv[kt][e][i] = 0.f;
                            odd = odd || !(fabsf(vv[kt][e][i]) < INFINITY);
                        }
                    }
                }
            }
            f32x4 o[OWN];
#pragma unroll
            for (int e = 0; e < OWN; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                if (!live[kt]) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < OWN; ++e) o[e] = mfma(vv[kt][e][j], p[kt][j], o[e]);
            }
            if (__ballot(odd) != 0) {
                for (int row = 0; row < rows_here; ++row) {
                    const int row_pos = __shfl(my_pos, row * heads_here, 64), row_lo = __shfl(my_lo, row * heads_here, 64);
#pragma unroll
                    for (int e = 0; e < OWN; ++e) {
                        f32x4 own = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int kt = 0; kt < 4; ++kt) {
                            if (!live[kt]) continue;
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                const int key = b0 + kt * 16 + 4 * g + j;
                                own = mfma(key > row_pos || key < row_lo ? 0.f : vv[kt][e][j], p[kt][j], own);
                            }
                        }
                        if (place == row) o[e] = own;
                    }
                }
            }
            const int at = block - my_lo / BLOCK;
            if (!in_run || at < 0 || block > my_pos / BLOCK || at >= n_blocks) continue;
            float* to = part + (((size_t)t * n_heads + h) * n_blocks + at) * part_floats(vd);
#pragma unroll
            for (int e = 0; e < OWN; ++e)
                if ((wave + 4 * e) * 16 < vd) *reinterpret_cast<f32x4*>(to + (wave + 4 * e) * 16 + 4 * g) = o[e];
            if (wave == 0 && g == 0) *reinterpret_cast<float2*>(to + vd) = float2{l, m};
        }
    }
}

// What those blocks left of a (row, head), joined: a span's four blocks as the kernel above joins them, then span after span.  Four spans' numbers are asked for at once.
__global__ __launch_bounds__(128) void attention_exact_join_blocks_kernel(const float* __restrict__ part, float* __restrict__ out, const int* __restrict__ pos, int n_heads, int vd,
                                                                         int window, int chunk, const float* __restrict__ sinks, const float* __restrict__ gate, long gate_stride,
                                                                         int gate_channels, int n_blocks) {
    const int t = blockIdx.x / n_heads, h = blockIdx.x % n_heads, d = threadIdx.x, p = pos[t], lo = first_key(p, window, chunk);
    const int first = lo / BLOCK, last = min(p / BLOCK, first + n_blocks - 1), channel = min(d, vd - 1);
    const float* from = part + (size_t)blockIdx.x * n_blocks * part_floats(vd);
    float m = sinks ? sinks[h] : -INFINITY, o = 0.f;
    double l = sinks ? 1.0 : 0.0;
    constexpr int AT_ONCE = 4;
    for (int s0 = first / 4; s0 <= last / 4; s0 += AT_ONCE) {
        float o_block[4 * AT_ONCE];
        float2 lm[4 * AT_ONCE];
#pragma unroll
        for (int b = 0; b < 4 * AT_ONCE; ++b) {
            const float* block = from + (size_t)(min(max(s0 * 4 + b, first), last) - first) * part_floats(vd);
            o_block[b] = block[channel];
            lm[b] = *reinterpret_cast<const float2*>(block + vd);
        }
#pragma unroll
        for (int s = 0; s < AT_ONCE; ++s) {
            if (s0 + s > last / 4) break;
            float top = -INFINITY;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int block = (s0 + s) * 4 + b;
                if (block >= first && block <= last) top = fmaxf(top, lm[4 * s + b].y);
            }
            double l_span = 0.0;
            float o_span = 0.f;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int block = (s0 + s) * 4 + b;
                if (block < first || block > last) continue;
                const float f = lm[4 * s + b].y == -INFINITY ? 0.f : expf(lm[4 * s + b].y - top);
                l_span = fma((double)lm[4 * s + b].x, (double)f, l_span);
                o_span = fmaf(o_block[4 * s + b], f, o_span);
            }
            const Join f = join(m, l, true, top, l_span);
            o = joined(o, o_span, f);
        }
    }
    if (d < vd) out[(size_t)blockIdx.x * vd + d] = finished(o, l, gate, gate_stride, gate_channels, t, h, d);
}

// The spans of a (row, head), left by several workgroups, joined in order.
__global__ __launch_bounds__(128) void attention_exact_join_kernel(const float* __restrict__ part, float* __restrict__ out, const int* __restrict__ pos, int n_heads, int vd,
                                                                  int window, int chunk, const float* __restrict__ sinks, const float* __restrict__ gate, long gate_stride,
                                                                  int gate_channels, int n_spans) {
    const int t = blockIdx.x / n_heads, h = blockIdx.x % n_heads, d = threadIdx.x, p = pos[t];
    const int count = min(p / SPAN - first_key(p, window, chunk) / SPAN + 1, n_spans);
    const float* from = part + (size_t)blockIdx.x * n_spans * part_floats(vd);
    float m = sinks ? sinks[h] : -INFINITY, o = 0.f;
    double l = sinks ? 1.0 : 0.0;
    const int channel = min(d, vd - 1);
    for (int s = 0; s < count; ++s, from += part_floats(vd)) {
        const float o_span = from[channel];
        const Join f = join(m, l, true, from[vd + 2], *reinterpret_cast<const double*>(from + vd));
        o = joined(o, o_span, f);
    }
    if (d < vd) out[(size_t)blockIdx.x * vd + d] = finished(o, l, gate, gate_stride, gate_channels, t, h, d);
}

// ---------------------------------------------------------------------------------------------- rows

template <typename TQ, typename TC, typename TO>
__global__ __launch_bounds__(64) void attention_exact_kernel(const TQ* __restrict__ q, const TC* __restrict__ cache, TO* __restrict__ out,
                                                            const int* __restrict__ pos, const int* __restrict__ slot,
                                                            const int* __restrict__ table, int table_stride, long page_stride,
                                                            int page_size, int n_heads, int n_kv, int hd, int vd, int window, int chunk, float scale, float cap,
                                                            const float* __restrict__ sinks, const float* __restrict__ gate, long gate_stride, int gate_channels) {
    __shared__ float q_s[MAX_HD];
    __shared__ float p_s[64];
    __shared__ long v_off[64];
    const int lane = threadIdx.x;
    const int t = blockIdx.x / n_heads, h = blockIdx.x % n_heads, g = h / (n_heads / n_kv);
    const int p_row = pos[t];
    const int* tab = table + (size_t)slot[t] * table_stride;
    const int lo = first_key(p_row, window, chunk);
    for (int d = lane; d < hd; d += 64) q_s[d] = load_f32(q, (size_t)t * n_heads * hd + h * hd + d);
    __syncthreads();

    const long v_plane = (long)n_kv * page_size * hd;   // from a page's keys to its values
    float m = sinks ? sinks[h] : -INFINITY;
    double l = sinks ? 1.0 : 0.0;
    float acc[MAX_HD / 64] = {};
    for (int j0 = lo; j0 <= p_row; j0 += 64) {
        const int j = j0 + lane;
        const bool valid = j <= p_row;
        float s = -INFINITY;
        long off = 0, voff = 0;
        if (valid) {
            const long page = (long)tab[j / page_size] * page_stride;
            off = page + ((long)g * page_size + j % page_size) * hd;
            voff = page + v_plane + (long)g * vd * page_size + j % page_size;
            float dot = 0.f;
            for (int d = 0; d < hd; ++d) dot = fmaf(q_s[d], load_f32(cache, off + d), dot);
            s = dot * scale;
            if (cap > 0.f) s = cap * tanhf(s / cap);
        }
        const float m_new = fmaxf(m, wave_max(s));
        const float p = valid ? expf(s - m_new) : 0.f;
        const float corr = expf(m - m_new);      // 0 at the first tile (m = -inf)
        l = l * (double)corr + (double)wave_sum(p);
        m = m_new;
        __syncthreads();                         // the previous tile's p_s and v_off have been read
        p_s[lane] = p;
        v_off[lane] = voff;
        __syncthreads();
        const int n_here = min(64, p_row - j0 + 1);
#pragma unroll
        for (int i = 0; i < MAX_HD / 64; ++i) acc[i] *= corr;
        for (int jj = 0; jj < n_here; ++jj) {
            const float pj = p_s[jj];
            const long vo = v_off[jj];
#pragma unroll
            for (int i = 0; i < MAX_HD / 64; ++i) {
                const int d = lane + 64 * i;
                if (d < vd) acc[i] = fmaf(pj, load_f32(cache, vo + (long)d * page_size), acc[i]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MAX_HD / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < vd) store_f32(out, (size_t)t * n_heads * vd + h * vd + d, finished(acc[i], l, gate, gate_stride, gate_channels, t, h, d));
    }
}

}  // namespace

GI_API int gi_attention_exact_max_head_size() { return MAX_HD; }

// Whether the kernel with tiles serves these sizes (all operands 32-bit and aligned).  Not where a window or a chunk leaves a row 16 keys at most: a block
// of 64 keys costs a tile much the same however few it sees of them.  Microseconds of rows and tiles, 16 single rows at 400 positions and more and a prompt of 300, 32/8 heads of 64:
// windows of 8 keys 6 and 13, 18 and 22; of 16 8 and 13, 28 and 23; of 32 11 and 14, 46 and 24; of 64 19 and 16, 82 and 28; of 256 74 and 22, 204 and 32.  (The
// tiles took 19 and 31 at all of the first three while they divided by the page size and worked on keys that nobody sees.)
static bool takes_tiles(int hd, int vd, int page_size, int window, int chunk) {
    if ((window > 0 && window <= 16) || (chunk > 0 && chunk <= 16)) return false;
    return hd % 16 == 0 && vd % 16 == 0 && hd <= 128 && vd <= 128 && page_size % 4 == 0;
}

// Rows of a tile: what its 16 pairs have room for.  The first `n_single` rows of a step, its requests' only ones (decoded rows), have tiles of their own.
static int rows_a_tile(int group) { return group < PAIRS ? PAIRS / group : 1; }
static long count_tiles(int n_rows, int n_single, int n_kv, int group) {
    const int a_tile = rows_a_tile(group);
    return (long)(n_single + (n_rows - n_single + a_tile - 1) / a_tile) * n_kv * ((group + PAIRS - 1) / PAIRS);
}

// How many spans of 256 keys the widest row of a step has at most, 0 where they are not shared out: `seen` positions at most are seen by a row.
// They are shared out while the tiles alone give fewer than two workgroups a compute unit, and the parts stay under 64 MB and in number
// under what a grid's second dimension holds.
GI_API int gi_attention_exact_spans(int n_rows, int n_single, int n_heads, int n_kv, int hd, int vd, int page_size, int seen) {
    if (n_rows <= 0 || n_single < 0 || n_single > n_rows || n_kv <= 0 || n_heads % n_kv != 0 || seen <= SPAN || !takes_tiles(hd, vd, page_size, 0, 0)) return 0;
    const long tiles = count_tiles(n_rows, n_single, n_kv, n_heads / n_kv);
    const long spans = ((long)seen + SPAN - 1) / SPAN + 1;
    if (tiles >= 2L * gi_compute_units() || spans > MAX_SPANS || spans * n_rows * n_heads * part_floats(vd) > (16L << 20)) return 0;
    return (int)spans;
}
// Whether the spans' blocks of 64 keys then go out one by one, by `walks`, the spans that the tiles see at most (workgroups of the kernel of spans), and how many rounds those make on the compute
// units.  3,094 steps (1 to 400 rows of their own, of a prompt and of both, 280 to 40,000 positions, 11 shapes of heads; both kernels with their joins): nowhere more than 2 % slower than spans and 30 % less
// time in the mean where blocks serve, which are 2 to 54 % slower in 160 of the others.
// Heads of more than 64 channels, one workgroup of spans or two of blocks a unit.  Microseconds, spans and blocks:
//   not where the spans' workgroups nearly fill their first round, for the blocks are then two full ones (24/8 heads of 128, 1,000 positions: a prompt of 24 rows 25.5 and 20.8, of 32 25.7 and 28.4, of 60 46.0 and
//   36.3; 3 rows of their own at 2,000 28.2 and 21.9, 2 at 4,000 32.4 and 34.4).  With up to three spans a row that tells later, and only where many rows join (500 positions: a prompt of 64 rows 26.7 and 27.3,
//   of 80 27.6 and 29.9; 16/16 heads, 100 rows at 300 26.4 and 19.3);
//   not where rows have more spans than the rounds saved are worth, for the join walks four parts a span (16/2 heads of 128, 8 rows of their own at 8,000 58.7 and 59.8, 10 of 8/1 heads at 12,000 70 and 74, 24/8 heads, 1 row
//   at 8,000 37.2 and 44.2, 3 of 8/1 heads at 40,000 105 and 144).
// Heads of up to 64 channels, two workgroups of spans a unit: up to so many blocks, fewer where contexts are long, and while the join has few parts to read (32/8 heads of 64: 12 rows at 300, 600 positions
// 15.9 and 11.6, 19.5 and 15.3, at 1,000 22.6 and 23.4; 5 at 2,000 23.3 and 24.2; 1 at 4,000 20.8 and 19.7, 16/2 heads, 1 row at 8,000 26.9 and 28.8; a prompt of 16 rows at 1,000 16.6 and 13.3, at 2,000 18.9 and 21.2).
static bool by_blocks(int n_rows, int n_single, int n_heads, int n_kv, int hd, int vd, int n_spans) {
    if (4L * n_spans * n_rows * n_heads * part_floats(vd) > (16L << 20) || 4 * n_spans > MAX_SPANS) return false;
    const long pairs = (long)n_rows * n_heads, walks = count_tiles(n_rows, n_single, n_kv, n_heads / n_kv) * (n_spans - 1), units = gi_compute_units();
    if (hd <= 64 && vd <= 64) return pairs <= 512 && n_spans <= 17 && 4 * walks <= (n_spans <= 5 ? 1152 : n_spans <= 9 ? 896 : 512);
    const bool nearly_one_round = walks <= units && (n_spans > 4 ? 4 * walks > 3 * units : 8 * walks > 7 * units && pairs >= 900);
    return !nearly_one_round && n_spans - 1 <= 22 * ((walks + units - 1) / units) + 2;
}
// Floats for the parts: what spans leave, and what the call asks for (with fewer than blocks leave it goes by spans).
GI_API long gi_attention_exact_span_floats(int n_rows, int n_heads, int vd, int n_spans) { return (long)n_rows * n_heads * n_spans * part_floats(vd); }
GI_API long gi_attention_exact_part_floats(int n_rows, int n_single, int n_heads, int n_kv, int hd, int vd, int n_spans) {
    return gi_attention_exact_span_floats(n_rows, n_heads, vd, n_spans) * (by_blocks(n_rows, n_single, n_heads, n_kv, hd, vd, n_spans) ? 4 : 1);
}

GI_API int gi_attention_exact(const void* q, int q_dtype, const void* cache, int cache_dtype, void* out, int out_dtype, const int* pos,
                              const int* slot, const int* table, int table_stride, long page_stride, int page_size, int n_rows,
                              int n_heads, int n_kv, int hd, int vd, int window, int chunk, float scale, float cap, const float* sinks, const float* gate,
                              long gate_stride, int gate_channels, int n_single, int n_requests, float* part, long part_size, int n_spans, hipStream_t stream) {
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0, "attention_exact: bad head counts (%d rows, %d heads, %d kv heads)",
               n_rows, n_heads, n_kv);
    GI_REQUIRE(hd > 0 && hd <= MAX_HD, "attention_exact: head size %d is outside 1..%d", hd, MAX_HD);
    GI_REQUIRE(vd > 0 && vd <= MAX_HD, "attention_exact: value head size %d is outside 1..%d", vd, MAX_HD);
    GI_REQUIRE(window >= 0 && chunk >= 0 && cap >= 0.f && (gate_channels == 0 || gate_channels == vd) &&
                   (gate == nullptr || gate_stride >= (long)n_heads * (gate_channels ? vd : 1)), "attention_exact: bad window, chunk or gate stride");
    GI_REQUIRE(page_size > 0 && page_stride >= (long)n_kv * page_size * (hd + vd), "attention_exact: page stride %ld too small", page_stride);
    GI_REQUIRE((long)n_rows * n_heads < 2147483647L, "attention_exact: too many (row, head) pairs");
    const unsigned grid = (unsigned)(n_rows * n_heads);
    const auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    if (q_dtype == GI_F32 && cache_dtype == GI_F32 && out_dtype == GI_F32 && takes_tiles(hd, vd, page_size, window, chunk) && page_stride % 4 == 0 && aligned(q) && aligned(cache)) {
        GI_REQUIRE(n_single >= 0 && n_single <= n_rows, "attention_exact: %d single rows of %d", n_single, n_rows);
        const int a_tile = rows_a_tile(n_heads / n_kv), turns = n_single == n_rows ? 1 : n_requests > 0 && n_requests < a_tile ? n_requests : a_tile;
        if (n_spans > 0) {
            GI_REQUIRE(part != nullptr && aligned(part) && part_size >= gi_attention_exact_span_floats(n_rows, n_heads, vd, n_spans) && n_spans <= MAX_SPANS,
                       "attention_exact: sharing the keys out needs %ld floats", gi_attention_exact_span_floats(n_rows, n_heads, vd, n_spans));
        } else {
            part = nullptr;
        }
        Divisor pages = {page_size, 0, 0};
        while ((1LL << pages.shift) < page_size) ++pages.shift;
        pages.magic = (unsigned)((((1ULL << pages.shift) - page_size) << 32) / page_size + 1);
        const dim3 tiles((unsigned)count_tiles(n_rows, n_single, n_kv, n_heads / n_kv), part ? n_spans : 1, turns);
        if (part && by_blocks(n_rows, n_single, n_heads, n_kv, hd, vd, n_spans) && part_size >= 4 * gi_attention_exact_span_floats(n_rows, n_heads, vd, n_spans)) {
            const int n_blocks = 4 * n_spans;
            const dim3 blocks(tiles.x, n_blocks, tiles.z);
#define BLOCKS(D)                                                                                                                          \
    attention_exact_blocks_kernel<D><<<blocks, 256, 0, stream>>>((const float*)q, (const float*)cache, pos, slot, table, table_stride, page_stride, pages, n_rows, n_heads, n_kv, hd, vd, window, \
                                                                 chunk, scale, cap, n_single, a_tile, part, n_blocks)
            if (hd <= 64 && vd <= 64) BLOCKS(64);
            else BLOCKS(128);
#undef BLOCKS
            GI_CHECK_LAUNCH("attention_exact (blocks)");
            attention_exact_join_blocks_kernel<<<grid, 128, 0, stream>>>(part, (float*)out, pos, n_heads, vd, window, chunk, sinks, gate, gate_stride, gate_channels, n_blocks);
            GI_CHECK_LAUNCH("attention_exact (join)");
            return 0;
        }
#define TILES(D)                                                                                                                           \
    attention_exact_tiles_kernel<D><<<tiles, 256, 0, stream>>>((const float*)q, (const float*)cache, (float*)out, pos, slot, table, table_stride, page_stride, pages, n_rows, \
                                                               n_heads, n_kv, hd, vd, window, chunk, scale, cap, sinks, gate, gate_stride, gate_channels, n_single, a_tile, part, n_spans)
        if (hd <= 64 && vd <= 64) TILES(64);
        else TILES(128);
#undef TILES
        if (part) attention_exact_join_kernel<<<grid, 128, 0, stream>>>(part, (float*)out, pos, n_heads, vd, window, chunk, sinks, gate, gate_stride, gate_channels, n_spans);
        GI_CHECK_LAUNCH("attention_exact (tiles)");
        return 0;
    }
#define GO(TQ, TC, TO)                                                                                                          \
    attention_exact_kernel<TQ, TC, TO><<<grid, 64, 0, stream>>>((const TQ*)q, (const TC*)cache, (TO*)out, pos, slot, table, table_stride, \
                                                                page_stride, page_size, n_heads, n_kv, hd, vd, window, chunk, scale, cap, sinks, gate, gate_stride, gate_channels)
    if (q_dtype == GI_F32 && cache_dtype == GI_F32 && out_dtype == GI_F32) GO(float, float, float);
    else if (q_dtype == GI_BF16 && cache_dtype == GI_BF16 && out_dtype == GI_BF16) GO(bf16_t, bf16_t, bf16_t);
    else return gi_fail("attention_exact: dtypes (%d, %d, %d) must be all float32 or all bfloat16", q_dtype, cache_dtype, out_dtype);
#undef GO
    GI_CHECK_LAUNCH("attention_exact");
    return 0;
}
