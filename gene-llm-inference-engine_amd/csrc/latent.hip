// Attention through latents: what lies between the down projections and the attention kernel.
//
// A layer of this kind projects a row down twice: to a query latent of `q_rank` numbers, and to a key/value latent of `kv_rank`
// numbers with `rot` more that are one rotated key part for all heads.  Both latents are RMS-normed with weights of their own.
// Only the normed key/value latent c and the rotated part are cached, nothing per head, because with the up projections folded
// into the query (q' = W_uk^T q per head) and into the output (o = W_uv sum_j p_j c_j) the latent is key and value at once:
//     score_j = q' . c_j + q_rot . k_rot_j          out = sum_j softmax(score)_j c_j
// A page holds its places' keys [place][kv_rank + rot] and, behind them, the latent once more with the places innermost
// [kv_rank][place]: the layout of a layer with one key/value head whose values are shorter than its keys, which every attention
// kernel reads, and both operands of the matrix instructions come out of memory as they lie.
// The rotation turns neighbouring channels, the pair (2i, 2i + 1), or the pair (i, i + rot/2), by pos * f_i.
//
//   latent_prepare   one wave per (row, which): the query latent normed into the rows the up projection reads; the key/value
//                    latent normed and the rotated part turned, both written to the row's place in its page
//   latent_queries   one wave per (row, head): a head's unrotated channels into the rows the folding product reads, its
//                    rotated channels turned and written behind the place where that product puts q'
//   latent_direct    both of these in one launch, where the queries have no latent and so stand in the same rows as the key/value latent
//   heads_product    out[t, h, :] = a[t, h, :] W_h^T for every head in one launch (the folding of W_uk into the queries and the
//                    product with W_uv behind the attention, whose results a gate per channel may multiply on the way), on the matrix cores
//   latent_attention one wave per (row, 16 heads, share of the context): all heads read the same keys, so 16 of them are the
//                    columns of one matrix instruction even for a single decoded row; for the rows of prompts a workgroup takes a
//                    few consecutive rows with all their heads and stages the keys they see once in LDS
#include "common.h"

namespace {

// A row's rot channels at src, turned, to dst: pairs of neighbours, or (half_split) the pairs (i, i + rot/2).
template <typename TC>
__device__ __forceinline__ void turn_pairs(const float* __restrict__ src, const float* __restrict__ cos_t, const float* __restrict__ sin_t, size_t t, int rot, int half_split,
                                           int lane, TC* __restrict__ dst) {
    for (int i = lane; i < rot / 2; i += 64) {
        const int a = half_split ? i : 2 * i, b = half_split ? i + rot / 2 : 2 * i + 1;
        const float u = src[a], v = src[b];
        const float c = cos_t[t * (rot / 2) + i], s = sin_t[t * (rot / 2) + i];
        store_f32(dst, a, u * c - v * s);
        store_f32(dst, b, v * c + u * s);
    }
}

// A latent's numbers, a lane those 64 apart: up to 64 LATENT_HELD of them stay in registers, all asked for at once (read twice, 5 rows
// of 768 and 256 + 32 numbers took 9.4 us, so 5.3); longer ones are read a second time.
constexpr int LATENT_HELD = 16;
template <typename TW, typename STORE>
__device__ __forceinline__ void norm_latent(const float* __restrict__ src, const TW* __restrict__ w, int n, float eps, int lane, STORE store) {
    float ss = 0.f;
    if (n <= 64 * LATENT_HELD) {
        float x[LATENT_HELD], g[LATENT_HELD];
#pragma unroll
        for (int i = 0; i < LATENT_HELD; ++i) {
            if (64 * i >= n) break;
            const int d = min(lane + 64 * i, n - 1);
            x[i] = src[d], g[i] = load_f32(w, d);
        }
#pragma unroll
        for (int i = 0; i < LATENT_HELD; ++i) {
            if (64 * i >= n) break;
            if (lane + 64 * i < n) ss = fmaf(x[i], x[i], ss);
        }
        const float r = 1.0f / sqrtf(wave_sum(ss) / (float)n + eps);
#pragma unroll
        for (int i = 0; i < LATENT_HELD; ++i) {
            if (64 * i >= n) break;
            if (lane + 64 * i < n) store(lane + 64 * i, g[i] * (r * x[i]));
        }
        return;
    }
    for (int d = lane; d < n; d += 64) ss = fmaf(src[d], src[d], ss);
    const float r = 1.0f / sqrtf(wave_sum(ss) / (float)n + eps);
    for (int d = lane; d < n; d += 64) store(d, load_f32(w, d) * (r * src[d]));
}

// The key/value latent at src normed, and the rotated part behind it turned, to the row's place of its page: one wave.
template <typename TW, typename TC>
__device__ __forceinline__ void store_latent(const float* __restrict__ src, size_t t, int kv_rank, int rot, int half_split, const TW* __restrict__ w, float eps,
                                             const float* __restrict__ cos_t, const float* __restrict__ sin_t, int p, long page, TC* __restrict__ cache, long page_stride,
                                             int page_size, int lane) {
    TC* dst = cache + page * page_stride + (size_t)(p % page_size) * (kv_rank + rot);
    TC* as_value = cache + page * page_stride + (size_t)page_size * (kv_rank + rot) + p % page_size;      // [kv_rank][place]
    turn_pairs(src + kv_rank, cos_t, sin_t, t, rot, half_split, lane, dst + kv_rank);
    norm_latent(src, w, kv_rank, eps, lane, [&](int d, float c) {
        store_f32(dst, d, c);
        store_f32(as_value, (size_t)d * page_size, c);
    });
}

// A head's query at src parted: its unrotated channels to `plain`, the turned ones to `turned`: one wave.
template <typename TA, typename TC>
__device__ __forceinline__ void part_query(const float* __restrict__ src, size_t t, int dim, int rot, int half_split, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                           int lane, TA* __restrict__ plain, TC* __restrict__ turned) {
    for (int d = lane; d < dim; d += 64) store_f32(plain, d, src[d]);
    turn_pairs(src + dim, cos_t, sin_t, t, rot, half_split, lane, turned);
}

template <typename TW, typename TA, typename TC>
__global__ __launch_bounds__(64) void latent_prepare_kernel(const float* __restrict__ proj, long ld, int q_rank, int kv_rank, int rot,
                                                           const TW* __restrict__ q_norm, const TW* __restrict__ kv_norm, float eps,
                                                           const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                           const int* __restrict__ pos, const int* __restrict__ slot, const int* __restrict__ table,
                                                           int table_stride, TA* __restrict__ cq, long ldcq, TC* __restrict__ cache, long page_stride,
                                                           int page_size, int half_split) {
    const int t = blockIdx.x, lane = threadIdx.x;
    const float* src = proj + (size_t)t * ld;
    if (blockIdx.y == 0) {
        norm_latent(src, q_norm, q_rank, eps, lane, [&](int d, float c) { store_f32(cq, (size_t)t * ldcq + d, c); });
        return;
    }
    const int p = pos[t];
    store_latent(src + q_rank, t, kv_rank, rot, half_split, kv_norm, eps, cos_t, sin_t, p, (long)table[(size_t)slot[t] * table_stride + p / page_size], cache, page_stride, page_size, lane);
}

// (Four heads' waves to a workgroup: 57,000 workgroups of a wave took 14.7 us, most of it to start them.)
template <typename TA, typename TC>
__global__ __launch_bounds__(256) void latent_queries_kernel(const float* __restrict__ q, long ldq, const float* __restrict__ cos_t,
                                                           const float* __restrict__ sin_t, TA* __restrict__ plain, long ld_plain,
                                                           TC* __restrict__ folded, long ld_folded, int n_heads, int dim, int rot, int kv_rank, int half_split) {
    const size_t t = blockIdx.x, h = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (h >= (size_t)n_heads) return;
    part_query(q + t * ldq + h * (dim + rot), t, dim, rot, half_split, cos_t, sin_t, threadIdx.x & 63, plain + t * ld_plain + h * dim, folded + t * ld_folded + h * (kv_rank + rot) + kv_rank);
}

// item 0: the row's key/value latent into its page; items 1 ..: the heads' queries.
template <typename TW, typename TA, typename TC>
__global__ __launch_bounds__(64) void latent_direct_kernel(const float* __restrict__ q, long ldq, const float* __restrict__ kv, long ldkv, const TW* __restrict__ kv_norm, float eps,
                                                          const float* __restrict__ cos_t, const float* __restrict__ sin_t, const int* __restrict__ pos, const int* __restrict__ slot,
                                                          const int* __restrict__ table, int table_stride, TA* __restrict__ plain, long ld_plain, TC* __restrict__ folded,
                                                          long ld_folded, TC* __restrict__ cache, long page_stride, int page_size, int dim, int rot, int kv_rank, int half_split) {
    const size_t t = blockIdx.x;
    if (blockIdx.y == 0) {
        const int p = pos[t];
        store_latent(kv + t * ldkv, t, kv_rank, rot, half_split, kv_norm, eps, cos_t, sin_t, p, (long)table[(size_t)slot[t] * table_stride + p / page_size], cache, page_stride, page_size,
                     (int)threadIdx.x);
        return;
    }
    const size_t h = blockIdx.y - 1;
    part_query(q + t * ldq + h * (dim + rot), t, dim, rot, half_split, cos_t, sin_t, threadIdx.x, plain + t * ld_plain + h * dim, folded + t * ld_folded + h * (kv_rank + rot) + kv_rank);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int uintx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }
constexpr float LOG2E = 1.4426950408889634f;

// out[t, h*n_out + n] = sum_k a[t, h*k_dim + k] * w[h][n][k], bfloat16 operands, 32-bit sums.  One wave per (16 RT rows, head, 16 J
// columns): the operands of the 16x16x32 matrix instruction are 16-byte pieces of a's and w's rows as they lie in memory; w's rows come in the order that
// leaves a lane 4 J neighbouring columns of its row, stored 16 bytes at a time.  With `gate` (float32 [n_rows, ldg], head h's channels from h*n_out on) every
// result is multiplied by sigmoid(gate).
// A few rows are bound by a round trip to memory (16 columns a wave, all of k asked for at once), the rows of prompts by how often w is read (64 rows a
// wave) and by the stores: 1,777 rows of 32 heads, 64 -> 256 and 256 -> 64 channels together 45.0 us with 16 rows a wave and stores of 2 bytes, so 29.4;
// 5 rows 11.8 with 64 columns a wave, so 7.5.  Where 64 rows a wave leave fewer waves than three quarters of the compute units, 16 rows a wave are
// the faster ones: 257 rows of 4 heads, 64 -> 36 channels 3.1 us (5.0 with 64 rows a wave), of 8 heads, 512 -> 128 6.5 (8.9), 500 rows 6.7 (8.9; 128 waves),
// but 700 rows 9.1 (8.9; 176 waves), 400 rows of 32 heads, 256 -> 64 6.7 (5.9; 224 waves).  And where strips of 16 columns are more than eight waves a compute
// unit, so are 64 columns a wave for a few rows: 128 heads, 128 -> 512 (4,096 waves), 8 rows 4.7 us (5.4), 16 rows 5.0 (6.3).
template <typename TO, int RT, int J>
__global__ __launch_bounds__(64) void heads_product_kernel(const bf16_t* __restrict__ a, long lda, const bf16_t* __restrict__ w, TO* __restrict__ out, long ldo,
                                                          long out_head_stride, int n_rows, int k_dim, int n_out, const float* __restrict__ gate, long ldg) {
    const int lane = threadIdx.x, r = lane & 15, q4 = lane >> 4;
    const int row0 = blockIdx.x * (16 * RT), h = blockIdx.y, col0 = blockIdx.z * (16 * J);
    const bf16_t* arow[RT];
    const bf16_t* wrow[J];
#pragma unroll
    for (int i = 0; i < RT; ++i) arow[i] = a + (size_t)min(row0 + 16 * i + r, n_rows - 1) * lda + (size_t)h * k_dim;
#pragma unroll
    for (int j = 0; j < J; ++j) wrow[j] = w + ((size_t)h * n_out + min(col0 + 4 * J * (r >> 2) + 4 * j + (r & 3), n_out - 1)) * k_dim;
    floatx4 acc[RT][J];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = floatx4{};
#pragma unroll (RT == 1 ? 8 : 2)
    for (int k0 = 0; k0 < k_dim; k0 += 32) {
        const int k = k0 + 8 * q4;
        const bool in = k < k_dim;                       // (k_dim is a multiple of 8: a piece is inside or outside as a whole)
        uint4 av[RT], wv[J];
#pragma unroll
        for (int i = 0; i < RT; ++i) av[i] = *reinterpret_cast<const uint4*>(arow[i] + (in ? k : 0));
#pragma unroll
        for (int j = 0; j < J; ++j) wv[j] = *reinterpret_cast<const uint4*>(wrow[j] + (in ? k : 0));
        if (!in) {
#pragma unroll
            for (int i = 0; i < RT; ++i) av[i] = uint4{0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < J; ++j) wv[j] = uint4{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wv[j]), as_bf16x8(av[i]), acc[i][j], 0, 0, 0);
    }
    // element v of acc[i][j]: row row0 + 16 i + r, column col0 + 4 J q4 + 4 j + v
    const int col = col0 + 4 * J * q4;
    const bool whole = col + 4 * J <= n_out && (((uintptr_t)out | (size_t)ldo * sizeof(TO) | (size_t)out_head_stride * sizeof(TO)) & (J == 1 && sizeof(TO) == 2 ? 7 : 15)) == 0;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int t = row0 + 16 * i + r;
        if (t >= n_rows) break;
        if (gate) {
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][j][v] = acc[i][j][v] / (1.0f + expf(-gate[(size_t)t * ldg + (size_t)h * n_out + min(col + 4 * j + v, n_out - 1)]));
        }
        TO* to = out + (size_t)t * ldo + (size_t)h * out_head_stride + col;
        if (whole) {
            if constexpr (sizeof(TO) == 4) {
#pragma unroll
                for (int j = 0; j < J; ++j) *reinterpret_cast<floatx4*>(to + 4 * j) = acc[i][j];
            } else if constexpr (J == 1) {
                *reinterpret_cast<uint2*>(to) = uint2{f32x2_to_bf16x2(acc[i][0][0], acc[i][0][1]), f32x2_to_bf16x2(acc[i][0][2], acc[i][0][3])};
            } else {
#pragma unroll
                for (int j = 0; j < J; j += 2)
                    *reinterpret_cast<uint4*>(to + 4 * j) = uint4{f32x2_to_bf16x2(acc[i][j][0], acc[i][j][1]), f32x2_to_bf16x2(acc[i][j][2], acc[i][j][3]),
                                                                  f32x2_to_bf16x2(acc[i][j + 1][0], acc[i][j + 1][1]), f32x2_to_bf16x2(acc[i][j + 1][2], acc[i][j + 1][3])};
            }
        } else {
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (col + 4 * j + v < n_out) store_f32(to, 4 * j + v, acc[i][j][v]);
        }
    }
}

// The queries of up to 16 rows parted (latent_queries_kernel) and folded into the latents' channels (heads_product_kernel with 16 rows and 16 columns a wave) in one launch, in the bits of
// both: folded[t, h][n] = sum_k bfloat16(q[t, h][k]) * w[h][n][k], and behind a head's kv_rank channels the turned ones, by the last wave of a head.  Either launch is little more than its
// two round trips to memory: 32 heads, 64 + 32 channels into 256 + 32, in a captured chain 1 / 5 / 16 rows 4.1 / 4.4 / 4.4 us, in one 2.2 / 2.3 / 3.0.
__global__ __launch_bounds__(64) void latent_fold_kernel(const float* __restrict__ q, long ldq, const float* __restrict__ cos_t, const float* __restrict__ sin_t, const bf16_t* __restrict__ w,
                                                        bf16_t* __restrict__ folded, long ld_folded, int n_rows, int dim, int rot, int kv_rank, int half_split) {
    const int lane = threadIdx.x, h = blockIdx.x, r = lane & 15, q4 = lane >> 4, col0 = blockIdx.y * 16;
    if (col0 >= kv_rank) {
        for (int e = lane; e < n_rows * (rot / 2); e += 64) {                           // (turn_pairs, all rows' pairs side by side)
            const int t = e / (rot / 2), i = e - t * (rot / 2), a = half_split ? i : 2 * i, b = half_split ? i + rot / 2 : 2 * i + 1;
            const float* src = q + t * ldq + (size_t)h * (dim + rot) + dim;
            const float u = src[a], v = src[b], c = cos_t[e], s = sin_t[e];
            bf16_t* dst = folded + t * ld_folded + (size_t)h * (kv_rank + rot) + kv_rank;
            store_f32(dst, a, u * c - v * s);
            store_f32(dst, b, v * c + u * s);
        }
        return;
    }
    const float* arow = q + (size_t)min(r, n_rows - 1) * ldq + (size_t)h * (dim + rot);
    const bf16_t* wrow = w + ((size_t)h * kv_rank + min(col0 + r, kv_rank - 1)) * dim;
    floatx4 acc = floatx4{};
#pragma unroll 4
    for (int k0 = 0; k0 < dim; k0 += 32) {
        const int k = k0 + 8 * q4;
        const bool in = k < dim;                         // (dim is a multiple of 8)
        const float4 a0 = *reinterpret_cast<const float4*>(arow + (in ? k : 0)), a1 = *reinterpret_cast<const float4*>(arow + (in ? k : 0) + 4);
        uint4 wv = *reinterpret_cast<const uint4*>(wrow + (in ? k : 0));
        uint4 av = {f32x2_to_bf16x2(a0.x, a0.y), f32x2_to_bf16x2(a0.z, a0.w), f32x2_to_bf16x2(a1.x, a1.y), f32x2_to_bf16x2(a1.z, a1.w)};
        if (!in) av = wv = uint4{0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wv), as_bf16x8(av), acc, 0, 0, 0);
    }
    if (r >= n_rows) return;
    bf16_t* to = folded + r * ld_folded + (size_t)h * (kv_rank + rot);
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (col0 + 4 * q4 + v < kv_rank) to[col0 + 4 * q4 + v] = f32_to_bf16(acc[v]);
}

// Attention over the latent pages on the matrix cores.  One wave: row t, heads 16 hg .. 16 hg + 15, share `sp` of the row's
// context.  Tiles of 32 positions (two blocks of 16, each inside one page): S^T = K Q^T puts a position's scores for the 16 heads
// into one lane group, so that a head's maximum and sum are a lane's own plus two exchanges; the probabilities, as they lie, are
// the second operand of O^T = V^T P^T.  KS = key channels / 32 (rounded up: pieces beyond the key are zeros), DT = value channels / 16.
// Shares of one row meet in `part` ([row][head][share]{m, l, o[vd]}, 32-bit) and `latent_merge_kernel` adds them; with one share
// the wave writes the heads' outputs itself.  `rows`: the step's rows that this launch serves (nullptr: all, in order).
// `sinks` [heads], where given: a score per head that joins the softmax's sum and has no value; the row's first share starts from it.
template <int KS, int DT, bool EARLY>
__global__ __launch_bounds__(64) void latent_attention_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, bf16_t* __restrict__ out,
                                                             float* __restrict__ part, const int* __restrict__ rows, const int* __restrict__ pos,
                                                             const int* __restrict__ slot, const int* __restrict__ table, int table_stride, long page_stride,
                                                             int page_size, int n_heads, int kd, int vd, int window, float scale2, int n_splits,
                                                             const float* __restrict__ sinks) {
    const int lane = threadIdx.x, r = lane & 15, q4 = lane >> 4;
    const int t = rows ? rows[blockIdx.x] : blockIdx.x, hg = blockIdx.y, sp = blockIdx.z;
    const int head = hg * 16 + r;
    const bool head_ok = head < n_heads;
    const int p = pos[t];
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int* tab = table + (size_t)slot[t] * table_stride;
    // this share's tiles
    const int first_tile = lo >> 5, n_tiles = (p >> 5) - first_tile + 1;
    const int per = (n_tiles + n_splits - 1) / n_splits;
    const int tile0 = first_tile + sp * per, tile1 = min(tile0 + per, first_tile + n_tiles);
    const long v_plane = (long)page_size * kd;

    bf16x8 qreg[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int c = 32 * ks + 8 * q4;
        uint4 v = *reinterpret_cast<const uint4*>(q + ((size_t)t * n_heads + (head_ok ? head : 0)) * kd + (c < kd ? c : 0));
        if (!head_ok || c >= kd) v = uint4{0, 0, 0, 0};
        qreg[ks] = as_bf16x8(v);
    }
    floatx4 o[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) o[i] = floatx4{};
    float m = -INFINITY, l = 0.f;
    if (sinks && sp == 0) m = sinks[head_ok ? head : 0] * LOG2E, l = 1.f;

    for (int tile = tile0; tile < tile1; ++tile) {
        const int kv0 = tile << 5;
        const bf16_t* page[2];
        int place[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {                    // a block that lies outside what the row sees is read from a place that it does see
            const int j0 = min(max(kv0 + 16 * b, lo & ~15), p & ~15);
            page[b] = cache + (long)tab[j0 / page_size] * page_stride;
            place[b] = j0 % page_size;
        }
        // EARLY: the values are asked for with the keys (up to keys of 288 channels: registers): behind the scores they were a second round trip to memory, most of
        // the time of a share of one tile (5 rows of 32 heads at 212 positions: 13.4 us, so 8.7).  See the launch for where they are not.
        uint4 k_early[2][EARLY ? KS : 1];
        uint2 v_early[2][EARLY ? DT : 1];
        const auto value = [&](int b, int i) {
            const int c = 16 * i + r;
            return *reinterpret_cast<const uint2*>(page[b] + v_plane + (size_t)(c < vd ? c : 0) * page_size + place[b] + 4 * q4);
        };
        const auto key = [&](int b, int ks) {
            return *reinterpret_cast<const uint4*>(page[b] + (size_t)(place[b] + r) * kd + (32 * ks + 8 * q4 < kd ? 32 * ks + 8 * q4 : 0));
        };
        if constexpr (EARLY) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) k_early[b][ks] = key(b, ks);
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < DT; ++i) v_early[b][i] = value(b, i);
            __builtin_amdgcn_sched_barrier(0);
        }
        floatx4 s[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            s[b] = floatx4{};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                uint4 k;
                if constexpr (EARLY) k = k_early[b][ks];
                else k = key(b, ks);
                if (32 * ks + 8 * q4 >= kd) k = uint4{0, 0, 0, 0};
                s[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), qreg[ks], s[b], 0, 0, 0);
            }
        }
        // element v of s[b]: position kv0 + 16*b + 4*q4 + v, head r
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = kv0 + 16 * b + 4 * q4 + v;
                s[b][v] = (j >= lo && j <= p) ? s[b][v] * scale2 : -INFINITY;
                mx = fmaxf(mx, s[b][v]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m, mx);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float corr = exp2_fast(m - m_use);
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                s[b][v] = exp2_fast(s[b][v] - m_use);
                sum += s[b][v];
            }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        l = l * corr + sum;
        m = m_new;
        const uint4 pb = {f32x2_to_bf16x2(s[0][0], s[0][1]), f32x2_to_bf16x2(s[0][2], s[0][3]), f32x2_to_bf16x2(s[1][0], s[1][1]), f32x2_to_bf16x2(s[1][2], s[1][3])};
        // a block whose positions are all masked was read from another block's place: its probabilities are zeros, which is all that matters
#pragma unroll
        for (int i = 0; i < DT; ++i) {
            uint2 v0, v1;
            if constexpr (EARLY) v0 = v_early[0][i], v1 = v_early[1][i];
            else v0 = value(0, i), v1 = value(1, i);
            if (16 * i + r >= vd) v0 = v1 = uint2{0, 0};
#pragma unroll
            for (int v = 0; v < 4; ++v) o[i][v] *= corr;
            o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(uint4{v0.x, v0.y, v1.x, v1.y}), as_bf16x8(pb), o[i], 0, 0, 0);
        }
    }
    // element v of o[i]: channel 16*i + 4*q4 + v, head r
    if (!head_ok) return;
    if (n_splits == 1) {
        const float inv = 1.0f / l;                      // (a row always sees itself: l > 0)
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int c = 16 * i + 4 * q4 + v;
                if (c < vd) out[((size_t)t * n_heads + head) * vd + c] = f32_to_bf16(o[i][v] * inv);
            }
        return;
    }
    float* mine = part + (((size_t)blockIdx.x * n_heads + head) * n_splits + sp) * (vd + 2);
    if (q4 == 0) { mine[0] = m; mine[1] = l; }
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = 16 * i + 4 * q4 + v;
            if (c < vd) mine[2 + c] = o[i][v];
        }
}

// The shares of one (row, head): out = sum_s 2^(m_s - m) o_s / sum_s 2^(m_s - m) l_s.  Lane s fetches share s's maximum and sum (all
// at once, not one behind the other); the weights wait in LDS; a lane then adds its channels over the shares, in their order, eight
// loads in flight.
__global__ __launch_bounds__(64) void latent_merge_kernel(const float* __restrict__ part, bf16_t* __restrict__ out, const int* __restrict__ rows, int n_heads,
                                                         int vd, int n_splits) {
    __shared__ float weight[64];
    const size_t rh = blockIdx.x;
    const size_t to = (size_t)(rows ? rows[blockIdx.x / n_heads] : blockIdx.x / n_heads) * n_heads + blockIdx.x % n_heads;
    const int lane = threadIdx.x;
    const float* mine = part + rh * n_splits * (vd + 2);
    const float ms = lane < n_splits ? mine[(size_t)lane * (vd + 2)] : -INFINITY;
    const float ls = lane < n_splits ? mine[(size_t)lane * (vd + 2) + 1] : 0.f;
    const float m = wave_max(ms);
    const float w = ms == -INFINITY ? 0.f : exp2_fast(ms - m);
    const float inv = 1.0f / wave_sum(w * ls);
    weight[lane] = w;
    __syncthreads();
    for (int c = lane; c < vd; c += 64) {
        float acc = 0.f;
        int s = 0;
        for (; s + 8 <= n_splits; s += 8) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = mine[(size_t)(s + e) * (vd + 2) + 2 + c];
#pragma unroll
            for (int e = 0; e < 8; ++e) acc = fmaf(weight[s + e], v[e], acc);
        }
        for (; s < n_splits; ++s) acc = fmaf(weight[s], mine[(size_t)s * (vd + 2) + 2 + c], acc);
        out[to * vd + c] = f32_to_bf16(acc * inv);
    }
}

// The rows of prompts: a workgroup takes TR consecutive rows of one request (a piece of one of the attention plan's tiles) and all
// their heads, a wave per (row, 16 heads) as above, and the tiles of 32 positions that any of its rows sees are staged once in LDS
// for all of them: the keys [32][key channels, padded so that 16 rows' 16-byte reads fall into different banks], the values
// [value channels][32 places + 8].  Every wave masks by its own row's position and window and skips the tiles it sees nothing of;
// what a workgroup fetches from the L2 is shared by TR rows x all heads instead of 16 heads.
template <int KS, int DT, bool AHEAD>
__global__ __launch_bounds__(512) void latent_attention_tiles_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, bf16_t* __restrict__ out,
                                                                    const int4* __restrict__ tiles, int pieces_per_tile, int TR, int HG,
                                                                    const int* __restrict__ table, int table_stride, long page_stride, int page_size,
                                                                    int n_heads, int kd, int vd, int window, float scale2, const float* __restrict__ sinks) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int KP = KS * 32 + 8, VP = 40;
    bf16_t* Ks = reinterpret_cast<bf16_t*>(lds);         // [32][KP]
    bf16_t* Vs = Ks + 32 * KP;                           // [DT * 16][VP]
    const int tid = threadIdx.x, NT = blockDim.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, q4 = lane >> 4;
    const int4 tile = tiles[blockIdx.x / pieces_per_tile];
    const int piece = blockIdx.x % pieces_per_tile;
    const int row0 = tile.x + piece * TR, n_tok = min(TR, tile.x + tile.y - row0);
    if (n_tok <= 0) return;                              // (the whole workgroup, before any barrier)
    const int p_first = tile.z + piece * TR, p_last = p_first + n_tok - 1;
    const int lo_all = (window > 0 && p_first - window + 1 > 0) ? p_first - window + 1 : 0;
    const int* tab = table + (size_t)tile.w * table_stride;
    const long v_plane = (long)page_size * kd;
    for (int i = tid; i < (32 * KP + DT * 16 * VP) / 2; i += NT) reinterpret_cast<uint32_t*>(lds)[i] = 0;      // channels beyond the key's and the value's stay zeros

    const int ti = min(wave / HG, n_tok - 1), hg = wave % HG;
    const bool tok_ok = wave / HG < n_tok;
    const int t = row0 + ti, p = p_first + ti;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int head = hg * 16 + r;
    const bool head_ok = tok_ok && head < n_heads;
    bf16x8 qreg[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int c = 32 * ks + 8 * q4;
        uint4 v = *reinterpret_cast<const uint4*>(q + ((size_t)t * n_heads + (head < n_heads ? head : 0)) * kd + (c < kd ? c : 0));
        if (!head_ok || c >= kd) v = uint4{0, 0, 0, 0};
        qreg[ks] = as_bf16x8(v);
    }
    floatx4 o[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) o[i] = floatx4{};
    float m = -INFINITY, l = 0.f;
    if (sinks) m = sinks[head < n_heads ? head : 0] * LOG2E, l = 1.f;
    const int k_pieces = kd >> 3;
    // A tile on its way: every position's key in 16-byte pieces, every value channel's 32 places in four.  With AHEAD the next
    // tile is asked for into registers before this one is worked on (workgroups have 320 threads or more: a thread brings at most
    // KPER + VPER pieces); without (the largest sizes, whose registers are spoken for) a tile is fetched when its turn comes.
    constexpr int KPER = (32 * KS * 4 + 319) / 320, VPER = (DT * 16 * 4 + 319) / 320;
    uintx4 k_reg[AHEAD ? KPER : 1], v_reg[AHEAD ? VPER : 1];
    auto k_source = [&](int kv0, int idx) {
        const int key = idx / k_pieces, piece8 = idx % k_pieces;
        const int j = min(max(kv0 + key, lo_all), p_last);               // (a position nobody sees is read from one that somebody does)
        return cache + (long)tab[j / page_size] * page_stride + (size_t)(j % page_size) * kd + 8 * piece8;
    };
    auto v_source = [&](int kv0, int idx) {
        const int c = idx >> 2, b = (idx >> 1) & 1, e = idx & 1;
        const int j0 = min(max(kv0 + 16 * b, lo_all & ~15), p_last & ~15);
        return cache + (long)tab[j0 / page_size] * page_stride + v_plane + (size_t)c * page_size + j0 % page_size + 8 * e;
    };
    const int tk_last = p_last >> 5;
    {
        if constexpr (AHEAD) {
#pragma unroll
            for (int e = 0; e < KPER; ++e) k_reg[e] = *reinterpret_cast<const uintx4*>(k_source((lo_all >> 5) << 5, min(tid + e * NT, 32 * k_pieces - 1)));
#pragma unroll
            for (int e = 0; e < VPER; ++e) v_reg[e] = *reinterpret_cast<const uintx4*>(v_source((lo_all >> 5) << 5, min(tid + e * NT, vd * 4 - 1)));
        }
    }
    __syncthreads();

    for (int tk = lo_all >> 5; tk <= tk_last; ++tk) {
        const int kv0 = tk << 5;
        if constexpr (AHEAD) {
#pragma unroll
            for (int e = 0; e < KPER; ++e) {
                const int idx = tid + e * NT;
                if (idx < 32 * k_pieces) *reinterpret_cast<uintx4*>(Ks + (idx / k_pieces) * KP + 8 * (idx % k_pieces)) = k_reg[e];
            }
#pragma unroll
            for (int e = 0; e < VPER; ++e) {
                const int idx = tid + e * NT;
                if (idx < vd * 4) *reinterpret_cast<uintx4*>(Vs + (idx >> 2) * VP + 16 * ((idx >> 1) & 1) + 8 * (idx & 1)) = v_reg[e];
            }
        } else {
            for (int idx = tid; idx < 32 * k_pieces; idx += NT)
                *reinterpret_cast<uint4*>(Ks + (idx / k_pieces) * KP + 8 * (idx % k_pieces)) = *reinterpret_cast<const uint4*>(k_source(kv0, idx));
            for (int idx = tid; idx < vd * 4; idx += NT)
                *reinterpret_cast<uint4*>(Vs + (idx >> 2) * VP + 16 * ((idx >> 1) & 1) + 8 * (idx & 1)) = *reinterpret_cast<const uint4*>(v_source(kv0, idx));
        }
        __syncthreads();
        if (tk < tk_last) {
        if constexpr (AHEAD) {
#pragma unroll
            for (int e = 0; e < KPER; ++e) k_reg[e] = *reinterpret_cast<const uintx4*>(k_source(kv0 + 32, min(tid + e * NT, 32 * k_pieces - 1)));
#pragma unroll
            for (int e = 0; e < VPER; ++e) v_reg[e] = *reinterpret_cast<const uintx4*>(v_source(kv0 + 32, min(tid + e * NT, vd * 4 - 1)));
        }
        }
        if (tok_ok && tk >= (lo >> 5) && tk <= (p >> 5)) {
            floatx4 s[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                s[b] = floatx4{};
                const bf16_t* krow = Ks + (16 * b + r) * KP + 8 * q4;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    s[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(*reinterpret_cast<const uint4*>(krow + 32 * ks)), qreg[ks], s[b], 0, 0, 0);
            }
            float mx = -INFINITY;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int j = kv0 + 16 * b + 4 * q4 + v;
                    s[b][v] = (j >= lo && j <= p) ? s[b][v] * scale2 : -INFINITY;
                    mx = fmaxf(mx, s[b][v]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m, mx);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
            const float corr = exp2_fast(m - m_use);
            float sum = 0.f;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    s[b][v] = exp2_fast(s[b][v] - m_use);
                    sum += s[b][v];
                }
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            l = l * corr + sum;
            m = m_new;
            const uint4 pb = {f32x2_to_bf16x2(s[0][0], s[0][1]), f32x2_to_bf16x2(s[0][2], s[0][3]), f32x2_to_bf16x2(s[1][0], s[1][1]), f32x2_to_bf16x2(s[1][2], s[1][3])};
#pragma unroll
            for (int i = 0; i < DT; ++i) {
                const bf16_t* vrow = Vs + (16 * i + r) * VP + 4 * q4;
                const uint2 v0 = *reinterpret_cast<const uint2*>(vrow), v1 = *reinterpret_cast<const uint2*>(vrow + 16);
#pragma unroll
                for (int v = 0; v < 4; ++v) o[i][v] *= corr;
                o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(uint4{v0.x, v0.y, v1.x, v1.y}), as_bf16x8(pb), o[i], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    if (!head_ok) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = 16 * i + 4 * q4 + v;
            if (c < vd) out[((size_t)t * n_heads + head) * vd + c] = f32_to_bf16(o[i][v] * inv);
        }
}

// The rows of prompts where the heads come in whole groups of 32: a wave takes one row's 32 heads (the columns of the 32x32x16 matrix instruction), a workgroup up
// to eight (row, group) pairs of consecutive rows, all on the same tiles of 32 positions.  What bounds the kernel above is LDS (a wave reads a whole tile for 16
// columns, twice the time of its products) and a tile's round trip through registers; here a tile serves 32 columns a wave and goes from memory
// into LDS directly, into the one of two places that the waves are not reading, while they multiply.  Layout of a tile in LDS: keys [32 positions][pieces
// of 16 bytes], then values [channels][4 pieces], a row's pieces in fours exchanged by (row / 4) % 4, so that 16 rows' reads of a piece fall into different
// banks.  A lane reads the key rows in the order that makes its 16 scores the positions 8 h + 0 .. 7 and 16 + 8 h + 0 .. 7 (h: which half of the
// wave): as they lie, packed, they are the second operand of O^T = V^T P^T, and its first operand is one piece.  A column's maximum follows its scores
// only when it lags by more than LATENT_SLACK (in units of log2 e; any reference gives the same O / l), which takes the rescaling of the sums off most tiles.
// A wave's pieces of a tile are asked for some ahead of their products: with each waited for in turn 1,777 rows of 32 heads, keys of 288 and values of 256 channels, a window of
// 1,024, took 87 us for now 78 (223 in the kernel above), 500 rows at 3,000 to 3,500 positions 226 and 188.  What bounds it: of the 3,900 clocks of a tile the matrix instructions take 2,180, the
// other wave of the SIMD beside it mostly doing the same; more pieces ahead have no registers (at 256 of them), and half of the waves a step behind the others was slower (85 us).
typedef float floatx16 __attribute__((ext_vector_type(16)));
constexpr float LATENT_SLACK = 8.f;
template <int KS, int VT>          // keys of up to 32 KS channels, values of up to 32 VT
__global__ __launch_bounds__(512) void latent_attention_wide_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, bf16_t* __restrict__ out,
                                                                   const int4* __restrict__ tiles, int pieces_per_tile, int TR, int HG,
                                                                   const int* __restrict__ table, int table_stride, long page_stride, int page_size,
                                                                   int n_heads, int kd, int vd, int window, float scale2, const float* __restrict__ sinks) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int AHEAD = KS > 5 ? 3 : 4;                 // pieces of a tile asked for ahead of their product (as many as there are registers for)
    constexpr int KPIECES = 4 * KS, K_BYTES = 32 * KPIECES * 16, V_BYTES = VT * 32 * 64, STAGE = K_BYTES + V_BYTES, PARTS = STAGE / 1024, MOST = (PARTS + 7) / 8;
    static_assert(K_BYTES % 1024 == 0 && V_BYTES % 1024 == 0, "a wave-wide load fills 1 KB");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, half = lane >> 5;
    const int4 tile = tiles[blockIdx.x / pieces_per_tile];
    const int piece = blockIdx.x % pieces_per_tile;
    const int row0 = tile.x + piece * TR, n_tok = min(TR, tile.x + tile.y - row0);
    if (n_tok <= 0) return;                              // (the whole workgroup, before any barrier)
    const int p_first = tile.z + piece * TR, p_last = p_first + n_tok - 1;
    const int lo_all = (window > 0 && p_first - window + 1 > 0) ? p_first - window + 1 : 0;
    const int* tab = table + (size_t)tile.w * table_stride;
    const bool works = wave < n_tok * HG;                // (every wave loads; one without a row multiplies nothing)
    const int ti = min(wave / HG, n_tok - 1), head = (wave % HG) * 32 + r;
    const int t = row0 + ti, p = p_first + ti;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;

    // This wave's loads of a tile: 1 KB each, parts wave, wave + 8, ..  Where a lane's 16 bytes lie: bytes behind its block's first key, or behind its block's
    // first place of channel 0; the highest bit says which of the tile's two blocks of 16 positions (each within one page).
    unsigned from[MOST];
#pragma unroll
    for (int i = 0; i < MOST; ++i) {
        const int part = wave + i * 8, slot = part * 64 + lane;
        if (part * 1024 < K_BYTES) {
            const int row = slot / KPIECES, c = (slot % KPIECES) ^ ((row >> 2) & 3);
            from[i] = (unsigned)((row & 15) * kd * 2 + min(c, (kd >> 3) - 1) * 16) | (row >= 16 ? 0x80000000u : 0u);       // (beyond the key: any piece that is numbers; the query has zeros there)
        } else {
            const int s = slot - K_BYTES / 16, e = (s & 3) ^ ((s >> 4) & 3);
            from[i] = (unsigned)(min(s >> 2, vd - 1) * page_size * 2 + (e & 1) * 16) | (e >= 2 ? 0x80000000u : 0u);
        }
    }
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lds;
    int tk = lo_all >> 5;
    const int tk_last = p_last >> 5;
    // Where the two blocks of the next tile to ask for lie: their pages are looked up a tile ahead, so that no load waits for the table's answer.
    int page_next = (tk << 5) / page_size, place_next = (tk << 5) % page_size, pages[2], places[2];
    auto look_up = [&](int tk) {
        int at_page[2], at_place[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            at_page[b] = page_next;
            at_place[b] = place_next;
            place_next += 16;
            if (place_next == page_size) { place_next = 0; ++page_next; }
        }
        // a block that nobody sees is read from the tile's other one
        const int b0 = (tk << 5) + 16 <= lo_all ? 1 : 0, b1 = (tk << 5) + 16 > p_last ? 0 : 1;
        places[0] = b0 ? at_place[1] : at_place[0];
        places[1] = b1 ? at_place[1] : at_place[0];
        pages[0] = tab[b0 ? at_page[1] : at_page[0]];
        pages[1] = tab[b1 ? at_page[1] : at_page[0]];
    };
    auto load_tile = [&](int place) {
        const char *keys[2], *values[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const bf16_t* page = cache + (long)pages[b] * page_stride;
            keys[b] = (const char*)(page + (long)places[b] * kd);
            values[b] = (const char*)(page + (long)page_size * kd + places[b]);
        }
#pragma unroll
        for (int i = 0; i < MOST; ++i) {
            const int part = wave + i * 8;
            if (part < PARTS) {
                unsigned where = from[i];
                asm volatile("" : "+v"(where));          // (or what follows from it is kept in registers from tile to tile)
                const bool is_key = part * 1024 < K_BYTES, second = (int)where < 0;
                const char* src = (is_key ? (second ? keys[1] : keys[0]) : (second ? values[1] : values[0])) + (where & 0x7fffffffu);
                const unsigned dst = __builtin_amdgcn_readfirstlane(lds_base + place * STAGE + part * 1024);
                // (as assembly, so that the compiler does not wait for them before every read of LDS: the wait and the barrier below order them)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "memory", "m0");
            }
        }
    };
    look_up(tk);
    load_tile(0);
    if (tk < tk_last) look_up(tk + 1);
    bf16x8 qreg[2 * KS];
#pragma unroll
    for (int s = 0; s < 2 * KS; ++s) {
        const int c = 16 * s + 8 * half;
        uint4 v = *reinterpret_cast<const uint4*>(q + ((size_t)t * n_heads + head) * kd + (c < kd ? c : 0));
        if (c >= kd) v = uint4{0, 0, 0, 0};
        qreg[s] = as_bf16x8(v);
    }
    floatx16 o[VT];
#pragma unroll
    for (int i = 0; i < VT; ++i) o[i] = floatx16{};
    float m = -INFINITY, l = 0.f;                        // (l: this lane's share of its column's sum)
    if (sinks) m = sinks[head] * LOG2E, l = half == 0 ? 1.f : 0.f;
    const int key = 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3), k_swz = (key >> 2) & 3, v_swz = (r >> 2) & 3;
    const unsigned char* k_row = lds + key * (KPIECES * 16);
    const unsigned char* v_row = lds + K_BYTES + r * 64;
    const int k_off[2] = {(half ^ k_swz) * 16, ((2 + half) ^ k_swz) * 16}, v_off[2] = {(half ^ v_swz) * 16, ((2 + half) ^ v_swz) * 16};

    auto lane_again = [] {                               // (what is rarely used is not kept in registers across the tiles, which take all there are)
        int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
        asm volatile("" : "+v"(l));
        return l;
    };
    for (int place = 0; tk <= tk_last; ++tk, place ^= 1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                               // this wave's loads of the tile have landed
        __builtin_amdgcn_s_barrier();                                                  // everyone's have, and nobody reads the other place any more
        asm volatile("" ::: "memory");
        if (tk < tk_last) load_tile(place ^ 1);
        if (tk + 1 < tk_last) look_up(tk + 2);
        const int kv0 = tk << 5;
        if (!works || kv0 + 31 < lo || kv0 > p) continue;
        const unsigned char *kr = k_row + place * STAGE, *vr = v_row + place * STAGE;
        // piece f of the tile: the keys' along the channels, then the values', all channels of the first 16 positions before the others
        auto piece_at = [&](int f) {
            const int i = f - 2 * KS;
            return as_bf16x8(*reinterpret_cast<const uint4*>(i < 0 ? kr + (f >> 1) * 64 + k_off[f & 1] : vr + (i % VT) * 2048 + v_off[i / VT]));
        };
        bf16x8 piece_of[AHEAD];
#pragma unroll
        for (int f = 0; f < AHEAD; ++f) piece_of[f] = piece_at(f);
        __builtin_amdgcn_sched_barrier(0);
        floatx16 s = floatx16{};
#pragma unroll
        for (int f = 0; f < 2 * KS; ++f) {
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(piece_of[f % AHEAD], qreg[f], s, 0, 0, 0);
            piece_of[f % AHEAD] = piece_at(f + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
        }
        // element v: position kv0 + 16 (v / 8) + 8 half + v % 8, head `head`
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] *= scale2;
        asm volatile("" : "+v"(s));                         // (one set of registers either way)
        if (kv0 < lo || kv0 + 31 > p) {
            const int first = kv0 + 8 * (lane_again() >> 5);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int j = first + 16 * (v >> 3) + (v & 7);
                s[v] = j >= lo && j <= p ? s[v] : -INFINITY;
            }
        }
        float mx = s[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const bool follow = mx > m + LATENT_SLACK;
        if (__any(follow)) {
            const float m_new = follow ? mx : m, corr = follow ? exp2_fast(m - m_new) : 1.f;
            m = m_new;
            l *= corr;
#pragma unroll
            for (int i = 0; i < VT; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[i][v] *= corr;
        }
        const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = exp2_fast(s[v] - m_use);
        l += (((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]))) + (((s[8] + s[9]) + (s[10] + s[11])) + ((s[12] + s[13]) + (s[14] + s[15])));
        const bf16x8 pb[2] = {as_bf16x8(uint4{f32x2_to_bf16x2(s[0], s[1]), f32x2_to_bf16x2(s[2], s[3]), f32x2_to_bf16x2(s[4], s[5]), f32x2_to_bf16x2(s[6], s[7])}),
                              as_bf16x8(uint4{f32x2_to_bf16x2(s[8], s[9]), f32x2_to_bf16x2(s[10], s[11]), f32x2_to_bf16x2(s[12], s[13]), f32x2_to_bf16x2(s[14], s[15])})};
#pragma unroll
        for (int f = 0; f < 2 * VT; ++f) {
            o[f % VT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(piece_of[(2 * KS + f) % AHEAD], pb[f / VT], o[f % VT], 0, 0, 0);
            if (f + AHEAD < 2 * VT) piece_of[(2 * KS + f) % AHEAD] = piece_at(2 * KS + f + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (!works) return;
    l += __shfl_xor(l, 32, 64);
    const float inv = 1.0f / l;                          // (a row always sees itself)
    const int end_lane = lane_again(), end_half = end_lane >> 5;
    bf16_t* to = out + ((size_t)t * n_heads + (wave % HG) * 32 + (end_lane & 31)) * vd;
#pragma unroll
    for (int i = 0; i < VT; ++i)
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            const int c = 32 * i + 2 * v + 4 * end_half;  // element v: channel 32 i + 8 (v / 4) + 4 half + v % 4
            if (c < vd) *reinterpret_cast<uint2*>(to + c) = uint2{f32x2_to_bf16x2(o[i][v] * inv, o[i][v + 1] * inv), f32x2_to_bf16x2(o[i][v + 2] * inv, o[i][v + 3] * inv)};
        }
}

}  // namespace

// proj: float32 [n_rows, ld] = [query latent (q_rank) | key/value latent (kv_rank) | rotated key part (rot)]; cos, sin: float32
// [n_rows, rot/2]; cq: [n_rows, ldcq] gets the normed query latent; the cache's pages hold [place][kv_rank + rot], then [kv_rank][place].
GI_API int gi_latent_prepare(const float* proj, long ld, int q_rank, int kv_rank, int rot, const void* q_norm, const void* kv_norm, int norm_dtype,
                             float eps, const float* cos_t, const float* sin_t, const int* pos, const int* slot, const int* table, int table_stride,
                             void* cq, int cq_dtype, long ldcq, void* cache, int cache_dtype, long page_stride, int page_size, int half_split, int n_rows,
                             hipStream_t stream) {
    GI_REQUIRE(n_rows > 0 && q_rank > 0 && kv_rank > 0 && rot >= 0 && rot % 2 == 0, "latent_prepare: bad sizes (rows %d, latents %d and %d, %d rotated channels)",
               n_rows, q_rank, kv_rank, rot);
    GI_REQUIRE(ld >= (long)q_rank + kv_rank + rot && ldcq >= q_rank && page_size > 0 && page_stride >= (long)page_size * (2L * kv_rank + rot),
               "latent_prepare: rows or pages too small for these latents");
    GI_REQUIRE(rot == 0 || (cos_t != nullptr && sin_t != nullptr), "latent_prepare: a rotation needs its cosines and sines");
    dim3 grid(n_rows, 2);
#define GO(TW, TA, TC)                                                                                                                        \
    latent_prepare_kernel<TW, TA, TC><<<grid, 64, 0, stream>>>(proj, ld, q_rank, kv_rank, rot, (const TW*)q_norm, (const TW*)kv_norm, eps, cos_t, sin_t, pos, \
                                                               slot, table, table_stride, (TA*)cq, ldcq, (TC*)cache, page_stride, page_size, half_split)
    if (norm_dtype == GI_F32 && cq_dtype == GI_F32 && cache_dtype == GI_F32) GO(float, float, float);
    else if (norm_dtype == GI_BF16 && cq_dtype == GI_BF16 && cache_dtype == GI_BF16) GO(bf16_t, bf16_t, bf16_t);
    else if (norm_dtype == GI_F32 && cq_dtype == GI_BF16 && cache_dtype == GI_BF16) GO(float, bf16_t, bf16_t);
    else if (norm_dtype == GI_F32 && cq_dtype == GI_F32 && cache_dtype == GI_BF16) GO(float, float, bf16_t);
    else if (norm_dtype == GI_BF16 && cq_dtype == GI_F32 && cache_dtype == GI_BF16) GO(bf16_t, float, bf16_t);
    else return gi_fail("latent_prepare: dtypes (%d, %d, %d) are not served", norm_dtype, cq_dtype, cache_dtype);
#undef GO
    GI_CHECK_LAUNCH("latent_prepare");
    return 0;
}

// q: float32 [n_rows, ldq], per head [dim unrotated | rot rotated]; plain: [n_rows, ld_plain] gets the heads' unrotated channels
// [n_heads][dim]; folded: [n_rows, ld_folded], per head [kv_rank + rot], gets the turned channels behind each head's first kv_rank.
GI_API int gi_latent_queries(const float* q, long ldq, const float* cos_t, const float* sin_t, void* plain, int plain_dtype, long ld_plain, void* folded,
                             int folded_dtype, long ld_folded, int n_rows, int n_heads, int dim, int rot, int kv_rank, int half_split, hipStream_t stream) {
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && n_heads <= 65535 && dim > 0 && rot >= 0 && rot % 2 == 0 && kv_rank > 0, "latent_queries: bad sizes (rows %d, heads %d, %d + %d channels)",
               n_rows, n_heads, dim, rot);
    GI_REQUIRE(ldq >= (long)n_heads * (dim + rot) && ld_plain >= (long)n_heads * dim && ld_folded >= (long)n_heads * (kv_rank + rot), "latent_queries: rows too short");
    GI_REQUIRE(rot == 0 || (cos_t != nullptr && sin_t != nullptr), "latent_queries: a rotation needs its cosines and sines");
    dim3 grid(n_rows, (n_heads + 3) / 4);
#define GO(TA, TC) latent_queries_kernel<TA, TC><<<grid, 256, 0, stream>>>(q, ldq, cos_t, sin_t, (TA*)plain, ld_plain, (TC*)folded, ld_folded, n_heads, dim, rot, kv_rank, half_split)
    if (plain_dtype == GI_F32 && folded_dtype == GI_F32) GO(float, float);
    else if (plain_dtype == GI_BF16 && folded_dtype == GI_BF16) GO(bf16_t, bf16_t);
    else if (plain_dtype == GI_F32 && folded_dtype == GI_BF16) GO(float, bf16_t);
    else return gi_fail("latent_queries: dtypes (%d, %d) are not served", plain_dtype, folded_dtype);
#undef GO
    GI_CHECK_LAUNCH("latent_queries");
    return 0;
}

// Whether gi_latent_fold takes queries of these sizes: as many rows as a matrix instruction has, and waves of 16 columns at most eight a compute unit (as gi_heads_product has it).
GI_API int gi_latent_fold_takes(int n_rows, int n_heads, int dim, int rot, int kv_rank) {
    return n_rows > 0 && n_rows <= 16 && n_heads > 0 && dim > 0 && dim % 8 == 0 && rot >= 0 && rot % 4 == 0 && kv_rank > 0 && (kv_rank + 15) / 16 < 65535 &&
           (long)n_heads * ((kv_rank + 15) / 16) <= 8L * gi_compute_units();
}

// gi_latent_queries into bfloat16 and gi_heads_product of what it parts with w [n_heads][kv_rank][dim], in one launch: folded [n_rows, ld_folded], per head [kv_rank | rot].
GI_API int gi_latent_fold(const float* q, long ldq, const float* cos_t, const float* sin_t, const void* w, void* folded, long ld_folded, int n_rows, int n_heads, int dim, int rot, int kv_rank,
                          int half_split, hipStream_t stream) {
    GI_REQUIRE(gi_latent_fold_takes(n_rows, n_heads, dim, rot, kv_rank), "latent_fold: sizes (rows %d, heads %d, %d + %d channels, %d of the latent) are not taken", n_rows, n_heads, dim, rot, kv_rank);
    GI_REQUIRE(ldq >= (long)n_heads * (dim + rot) && ldq % 4 == 0 && ((uintptr_t)q & 15) == 0 && ((uintptr_t)w & 15) == 0 && ld_folded >= (long)n_heads * (kv_rank + rot),
               "latent_fold: rows too short, or not at multiples of 16 bytes");
    GI_REQUIRE(rot == 0 || (cos_t != nullptr && sin_t != nullptr), "latent_fold: a rotation needs its cosines and sines");
    latent_fold_kernel<<<dim3(n_heads, (kv_rank + 15) / 16 + (rot > 0 ? 1 : 0)), 64, 0, stream>>>(q, ldq, cos_t, sin_t, (const bf16_t*)w, (bf16_t*)folded, ld_folded, n_rows, dim, rot, kv_rank, half_split);
    GI_CHECK_LAUNCH("latent_fold");
    return 0;
}

// q: float32 [n_rows, ldq], per head [dim unrotated | rot rotated]; kv: float32 [n_rows, ldkv] = [key/value latent (kv_rank) | rotated key
// part (rot)]; plain, folded and the cache as the two above fill them.
GI_API int gi_latent_direct(const float* q, long ldq, const float* kv, long ldkv, const void* kv_norm, int norm_dtype, float eps, const float* cos_t, const float* sin_t,
                            const int* pos, const int* slot, const int* table, int table_stride, void* plain, int plain_dtype, long ld_plain, void* folded, long ld_folded,
                            void* cache, int cache_dtype, long page_stride, int page_size, int half_split, int n_rows, int n_heads, int dim, int rot, int kv_rank,
                            hipStream_t stream) {
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && n_heads < 65535 && dim > 0 && rot >= 0 && rot % 2 == 0 && kv_rank > 0, "latent_direct: bad sizes (rows %d, heads %d, %d + %d channels, latent %d)",
               n_rows, n_heads, dim, rot, kv_rank);
    GI_REQUIRE(ldq >= (long)n_heads * (dim + rot) && ldkv >= (long)kv_rank + rot && ld_plain >= (long)n_heads * dim && ld_folded >= (long)n_heads * (kv_rank + rot) && page_size > 0 &&
               page_stride >= (long)page_size * (2L * kv_rank + rot), "latent_direct: rows or pages too short");
    GI_REQUIRE(rot == 0 || (cos_t != nullptr && sin_t != nullptr), "latent_direct: a rotation needs its cosines and sines");
    dim3 grid(n_rows, n_heads + 1);
#define GO(TW, TA, TC)                                                                                                                                   \
    latent_direct_kernel<TW, TA, TC><<<grid, 64, 0, stream>>>(q, ldq, kv, ldkv, (const TW*)kv_norm, eps, cos_t, sin_t, pos, slot, table, table_stride, (TA*)plain, ld_plain, \
                                                              (TC*)folded, ld_folded, (TC*)cache, page_stride, page_size, dim, rot, kv_rank, half_split)
    if (norm_dtype == GI_F32 && plain_dtype == GI_F32 && cache_dtype == GI_F32) GO(float, float, float);
    else if (norm_dtype == GI_BF16 && plain_dtype == GI_BF16 && cache_dtype == GI_BF16) GO(bf16_t, bf16_t, bf16_t);
    else if (norm_dtype == GI_F32 && plain_dtype == GI_BF16 && cache_dtype == GI_BF16) GO(float, bf16_t, bf16_t);
    else if (norm_dtype == GI_F32 && plain_dtype == GI_F32 && cache_dtype == GI_BF16) GO(float, float, bf16_t);
    else if (norm_dtype == GI_BF16 && plain_dtype == GI_F32 && cache_dtype == GI_BF16) GO(bf16_t, float, bf16_t);
    else return gi_fail("latent_direct: dtypes (%d, %d, %d) are not served", norm_dtype, plain_dtype, cache_dtype);
#undef GO
    GI_CHECK_LAUNCH("latent_direct");
    return 0;
}

// a: bfloat16 [n_rows, lda], head h's operand in columns [h*k_dim, (h+1)*k_dim); w: bfloat16 [n_heads][n_out][k_dim]; out: [n_rows, ldo],
// head h's result in columns [h*out_head_stride, h*out_head_stride + n_out).
GI_API int gi_heads_product_supports(int k_dim, int n_out) { return k_dim > 0 && n_out > 0 && k_dim % 8 == 0; }

GI_API int gi_heads_product(const void* a, long lda, const void* w, void* out, int out_dtype, long ldo, long out_head_stride, int n_rows, int n_heads, int k_dim,
                            int n_out, const float* gate, long ldg, hipStream_t stream) {
    GI_REQUIRE(gate == nullptr || ldg >= (long)n_heads * n_out, "heads_product: the gates' rows are too short");
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && n_heads <= 65535 && gi_heads_product_supports(k_dim, n_out), "heads_product: bad sizes (rows %d, heads %d, k %d, n %d; k a multiple of 8)",
               n_rows, n_heads, k_dim, n_out);
    GI_REQUIRE(lda % 8 == 0 && lda >= (long)n_heads * k_dim && ((uintptr_t)a & 15) == 0 && ((uintptr_t)w & 15) == 0 && out_head_stride >= n_out &&
               ldo >= (long)(n_heads - 1) * out_head_stride + n_out, "heads_product: operands must be 16-byte aligned with row strides that are multiples of 8, and rows long enough");
    GI_REQUIRE((n_out + 63) / 64 <= 65535, "heads_product: too many columns");
    const bool few_strips = (long)n_heads * ((n_out + 15) / 16) <= 8L * gi_compute_units();      // (of one row of 16; so the grid takes them)
    const bool few_waves = (long)((n_rows + 63) / 64) * n_heads * ((n_out + 63) / 64) < gi_compute_units() * 3 / 4;
#define GO_AS(TO, RT, J)                                                                                                                            \
    heads_product_kernel<TO, RT, J><<<dim3((n_rows + 16 * RT - 1) / (16 * RT), n_heads, (n_out + 16 * J - 1) / (16 * J)), 64, 0, stream>>>(           \
        (const bf16_t*)a, lda, (const bf16_t*)w, (TO*)out, ldo, out_head_stride, n_rows, k_dim, n_out, gate, ldg)
#define GO(TO)                                  \
    do {                                        \
        if (n_rows <= 16 && few_strips) GO_AS(TO, 1, 1);      \
        else if (n_rows <= 256 || few_waves) GO_AS(TO, 1, 4); \
        else GO_AS(TO, 4, 4);                   \
    } while (0)
    if (out_dtype == GI_F32) GO(float);
    else if (out_dtype == GI_BF16) GO(bf16_t);
    else return gi_fail("heads_product: unknown output dtype %d", out_dtype);
#undef GO
#undef GO_AS
    GI_CHECK_LAUNCH("heads_product");
    return 0;
}

// Sizes the matrix-core latent attention takes: keys of up to 576 channels in 16-byte pieces, values of up to 512 channels, pages of whole blocks of 16 places.
GI_API int gi_latent_attention_supports(int kd, int vd, int page_size) {
    return kd > 0 && kd % 8 == 0 && kd <= 576 && vd > 0 && vd <= 512 && vd <= kd && page_size > 0 && page_size % 16 == 0;
}
GI_API long gi_latent_attention_scratch_floats(int n_rows, int n_heads, int vd, int n_splits) {
    return n_splits > 1 ? (long)n_rows * n_heads * n_splits * (vd + 2) : 0;
}

// q: bfloat16 [n_rows, n_heads*kd] (folded queries); cache: bfloat16 pages [place][kd] then [vd][place]; out: bfloat16 [n_rows, n_heads*vd].
// rows: the n_rows rows of the step to serve (nullptr: rows 0 .. n_rows - 1).  share_tiles: how many tiles of 32 positions the longest share has, as far as the
// caller knows (for the choice of a kernel alone: any number gives the same results).
GI_API int gi_latent_attention_bf16(const void* q, const void* cache, void* out, float* part, long part_floats, const int* rows, const int* pos, const int* slot,
                                    const int* table, int table_stride, long page_stride, int page_size, int n_rows, int n_heads, int kd, int vd, int window,
                                    float scale, int n_splits, int share_tiles, const float* sinks, hipStream_t stream) {
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && gi_latent_attention_supports(kd, vd, page_size), "latent_attention: sizes (rows %d, heads %d, keys %d, values %d, pages of %d) are not taken",
               n_rows, n_heads, kd, vd, page_size);
    GI_REQUIRE(window >= 0 && n_splits >= 1 && n_splits <= 64 && page_stride >= (long)page_size * (kd + vd) && page_stride % 8 == 0 && ((uintptr_t)cache & 15) == 0 &&
               ((uintptr_t)q & 15) == 0, "latent_attention: bad window, shares, page stride or alignment");
    GI_REQUIRE(part_floats >= gi_latent_attention_scratch_floats(n_rows, n_heads, vd, n_splits) && (n_splits == 1 || part != nullptr), "latent_attention: scratch of %ld floats needed, %ld given",
               gi_latent_attention_scratch_floats(n_rows, n_heads, vd, n_splits), part_floats);
    GI_REQUIRE((long)n_rows * n_heads < 2147483647L && (n_heads + 15) / 16 <= 65535, "latent_attention: too many rows or heads");
    dim3 grid(n_rows, (n_heads + 15) / 16, n_splits);
    const float scale2 = scale * 1.4426950408889634f;
#define GO(KS, DT, EARLY_)                                                                                                                              \
    latent_attention_kernel<KS, DT, EARLY_><<<grid, 64, 0, stream>>>((const bf16_t*)q, (const bf16_t*)cache, (bf16_t*)out, part, rows, pos, slot, table, table_stride, \
                                                                     page_stride, page_size, n_heads, kd, vd, window, scale2, n_splits, sinks)
    // At keys of 288 channels the values' registers leave a SIMD one wave (two without): shares of one tile of positions that are more than that, or of two that
    // are at most half as many again, wait for a second round behind it.  40 rows of 32 heads at 500 positions (1,280 waves) 35.5 us, values behind the scores 31.7; 12
    // rows at 4,000 (1,536 waves of two tiles) 51.6 and 49.0; but 40 rows at 1,000 (2,000 waves of two) 39.9 and 41.8, 64 rows at 4,000 (eight tiles) 88 and 115.
    const long waves = (long)n_rows * grid.y * n_splits, places = 4L * gi_compute_units();
    const bool second_round = waves > places && (share_tiles == 1 || (share_tiles == 2 && 2 * waves <= 3 * places));
    if (kd <= 96 && vd <= 64) GO(3, 4, true);
    else if (kd <= 160 && vd <= 128) GO(5, 8, true);
    else if (kd <= 288 && vd <= 256) { if (second_round) GO(9, 16, false); else GO(9, 16, true); }
    else GO(18, 32, false);
#undef GO
    GI_CHECK_LAUNCH("latent_attention");
    if (n_splits > 1) {
        latent_merge_kernel<<<(unsigned)(n_rows * n_heads), 64, 0, stream>>>(part, (bf16_t*)out, rows, n_heads, vd, n_splits);
        GI_CHECK_LAUNCH("latent_merge");
    }
    return 0;
}

// The rows of prompts, by the attention plan's tiles ({first row, rows, first position, slot}, of up to tile_rows rows each): heads in
// groups of 16, at most 8 groups (128 heads).
GI_API int gi_latent_attention_tiles_supports(int n_heads, int kd, int vd, int page_size) {
    return gi_latent_attention_supports(kd, vd, page_size) && (n_heads + 15) / 16 <= 8;
}

template <int KS, int DT>
static int allow_latent_tiles_lds() {
    static bool allowed = false;                         // (per instantiation; more than 64 KiB of LDS must be asked for)
    if (!allowed) {
        const size_t lds_bytes = (size_t)(32 * (KS * 32 + 8) + DT * 16 * 40) * 2;
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attention_tiles_kernel<KS, DT, (KS <= 9)>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
            return gi_fail("latent_attention: %zu bytes of LDS are not granted", lds_bytes);
        allowed = true;
    }
    return 0;
}

template <int KS, int VT>
static int allow_latent_wide_lds() {
    static bool allowed = false;
    if (!allowed) {
        const int lds_bytes = 2 * (KS * 2048 + VT * 2048);
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attention_wide_kernel<KS, VT>), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
            return gi_fail("latent_attention: %d bytes of LDS are not granted", lds_bytes);
        allowed = true;
    }
    return 0;
}

// Asks for the kernels' LDS once, outside any captured pass (a part calls it when it is built).
GI_API int gi_latent_attention_tiles_prepare() {
    int rc = allow_latent_wide_lds<3, 2>();
    if (!rc) rc = allow_latent_wide_lds<5, 4>();
    if (!rc) rc = allow_latent_wide_lds<9, 8>();
    if (!rc) rc = allow_latent_tiles_lds<3, 4>();
    if (!rc) rc = allow_latent_tiles_lds<5, 8>();
    if (!rc) rc = allow_latent_tiles_lds<9, 16>();
    if (!rc) rc = allow_latent_tiles_lds<18, 32>();
    return rc;
}

template <int KS, int DT>
static int launch_latent_tiles(const void* q, const void* cache, void* out, const void* tiles, int n_tiles, int tile_rows, const int* table, int table_stride,
                               long page_stride, int page_size, int n_heads, int kd, int vd, int window, float scale2, const float* sinks, hipStream_t stream) {
    const int HG = (n_heads + 15) / 16, TR = 8 / HG > 0 ? 8 / HG : 1;
    const int pieces = (tile_rows + TR - 1) / TR;
    const size_t lds_bytes = (size_t)(32 * (KS * 32 + 8) + DT * 16 * 40) * 2;
    if (int rc = allow_latent_tiles_lds<KS, DT>()) return rc;
    latent_attention_tiles_kernel<KS, DT, (KS <= 9)><<<(unsigned)(n_tiles * pieces), 64 * TR * HG, lds_bytes, stream>>>(
        (const bf16_t*)q, (const bf16_t*)cache, (bf16_t*)out, (const int4*)tiles, pieces, TR, HG, table, table_stride, page_stride, page_size, n_heads, kd, vd, window, scale2,
        sinks);
    return 0;
}

template <int KS, int VT>
static int launch_latent_wide(const void* q, const void* cache, void* out, const void* tiles, int n_tiles, int tile_rows, const int* table, int table_stride,
                              long page_stride, int page_size, int n_heads, int kd, int vd, int window, float scale2, const float* sinks, hipStream_t stream) {
    const int HG = n_heads / 32, TR = 8 / HG, pieces = (tile_rows + TR - 1) / TR;
    if (int rc = allow_latent_wide_lds<KS, VT>()) return rc;
    latent_attention_wide_kernel<KS, VT><<<(unsigned)(n_tiles * pieces), 512, 2 * (KS * 2048 + VT * 2048), stream>>>(
        (const bf16_t*)q, (const bf16_t*)cache, (bf16_t*)out, (const int4*)tiles, pieces, TR, HG, table, table_stride, page_stride, page_size, n_heads, kd, vd, window, scale2, sinks);
    return 0;
}

GI_API int gi_latent_attention_tiles_bf16(const void* q, const void* cache, void* out, const void* tiles, int n_tiles, int tile_rows, const int* table, int table_stride,
                                          long page_stride, int page_size, int n_heads, int kd, int vd, int window, float scale, const float* sinks, hipStream_t stream) {
    GI_REQUIRE(n_tiles > 0 && tile_rows > 0 && n_heads > 0 && gi_latent_attention_tiles_supports(n_heads, kd, vd, page_size),
               "latent_attention (tiles): sizes (%d tiles of %d rows, heads %d, keys %d, values %d, pages of %d) are not taken", n_tiles, tile_rows, n_heads, kd, vd, page_size);
    GI_REQUIRE(window >= 0 && page_stride >= (long)page_size * (kd + vd) && page_stride % 8 == 0 && ((uintptr_t)cache & 15) == 0 && ((uintptr_t)q & 15) == 0 &&
               ((uintptr_t)tiles & 15) == 0, "latent_attention (tiles): bad window, page stride or alignment");
    GI_REQUIRE((long)n_tiles * tile_rows < 2147483647L, "latent_attention (tiles): too many rows");
    const float scale2 = scale * 1.4426950408889634f;
    int rc;
#define GO(KS, DT) rc = launch_latent_tiles<KS, DT>(q, cache, out, tiles, n_tiles, tile_rows, table, table_stride, page_stride, page_size, n_heads, kd, vd, window, scale2, sinks, stream)
#define WIDE(KS, VT) rc = launch_latent_wide<KS, VT>(q, cache, out, tiles, n_tiles, tile_rows, table, table_stride, page_stride, page_size, n_heads, kd, vd, window, scale2, sinks, stream)
    // whole groups of 32 heads whose sums fit in registers: 32 columns a wave (other numbers of heads would leave columns idle)
    const bool wide = n_heads % 32 == 0 && n_heads <= 256 && kd <= 288 && vd <= 256 && vd % 8 == 0 && ((uintptr_t)out & 7) == 0 && (long)vd * page_size < (1L << 29);
    if (kd <= 96 && vd <= 64) { if (wide) WIDE(3, 2); else GO(3, 4); }
    else if (kd <= 160 && vd <= 128) { if (wide) WIDE(5, 4); else GO(5, 8); }
    else if (kd <= 288 && vd <= 256) { if (wide) WIDE(9, 8); else GO(9, 16); }
    else GO(18, 32);
#undef WIDE
#undef GO
    if (rc) return rc;
    GI_CHECK_LAUNCH("latent_attention (tiles)");
    return 0;
}
