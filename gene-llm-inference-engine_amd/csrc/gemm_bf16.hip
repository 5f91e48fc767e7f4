// C[m, n] (=|+=) sum_k A[m, k] * W[n, k] with bfloat16 operands on the matrix cores, 32-bit sums.
//
// Both operands are row-major with k contiguous, so each lane's operand of a matrix instruction is
// one 16-byte load of 8 consecutive k.  Seven kernels:
//
//   pingpong  large prompt-sized products (256 x 256 tiles for most of the compute units): operands loaded
//           from global memory straight into LDS, two stages of A and three of W; the workgroup's eight waves form two
//           groups that take turns at reading LDS and at the matrix instructions.
//   tall    those in between: the same on tiles of 256 x 128 and three LDS stages.
//   piped   the other products of 128 rows or more (K a multiple of 64): tiles of 128 x 128,
//           operands loaded from global memory straight into a ring of LDS stages, several
//           blocks of k in flight; v_mfma_f32_32x32x16_bf16.
//   tiled   the other shapes above 64 rows: a BM x 128 tile of C per workgroup of 4 waves,
//           operands staged through registers into LDS in k-blocks of 64.
//   strips  up to 128 rows of A (K a multiple of 64), and more where k is shared out: 64 rows of weights and all rows of A, or a tile of up
//           to 256, a workgroup, both straight into a ring of LDS stages.  Wide outputs are finished by the workgroup that sees all of k;
//           for narrow ones k is split over workgroups and the partial sums are added in a fixed order by a second kernel.
//   skinny  the other shapes of up to 128 rows: weights stream from HBM straight into registers and are used
//           once, activations go through LDS; v_mfma_f32_16x16x32_bf16.  Wide and narrow outputs likewise.
//   slim    at most 16 rows of A (decode): a workgroup of 8 waves owns 8 to 32 weight rows, its
//           waves take interleaved steps of k and add their sums through LDS in a fixed order, so
//           one launch does the whole product and its epilogue.
//
// The "gated" epilogue serves SwiGLU: the weight is [gate; up] interleaved in groups of 16 rows
// (16 gate rows, the 16 up rows of the same outputs, and so on), and the output column c of a
// pair of groups is silu(gate_c) * up_c, stored as bfloat16: the stacked product never reaches
// memory.
//
// Requirements (checked on the host): K a multiple of 8, rows of A and W 16-byte aligned.  The
// output is float32 (stored or added onto what is there) or bfloat16 (stored).
#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

enum Epilogue : int { EPI_STORE_F32 = 0, EPI_ADD_F32 = 1, EPI_STORE_BF16 = 2, EPI_GATED_BF16 = 3, EPI_QKV_ROPE = 4, EPI_GATED_GELU_BF16 = 5, EPI_GATED_CLAMP_BF16 = 6, EPI_XIELU = 7 };
// The gated epilogues differ in the activation alone: SiLU (EPI_GATED_BF16), the tanh form of GELU, or the clamped form
// g sigmoid(1.702 g) (u + 1) with g <- min(g, limit), u <- clamp(u, -limit, limit) (EPI_GATED_CLAMP_BF16; `limit` comes with `NormIn`).
__host__ __device__ constexpr bool is_gated(int epi) { return epi == EPI_GATED_BF16 || epi == EPI_GATED_GELU_BF16 || epi == EPI_GATED_CLAMP_BF16; }

__device__ __forceinline__ float silu_gate(float g, float u) { return (g * (1.0f / (1.0f + expf(-g)))) * u; }
// The same with the hardware's exp2 and reciprocal (each within a unit or two in the last place of 32 bits): for results
// that are rounded to bfloat16's 8 bits at once.  The exact form above costs some thirty vector instructions a value,
// which in a prompt-sized product's epilogue is a tenth of the kernel.
__device__ __forceinline__ float silu_gate_fast(float g, float u) {
    return (g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f))) * u;
}

// gelu_tanh(g) = 0.5 g (1 + tanh(c (g + 0.044715 g^3))), c = sqrt(2 / pi); 0.5 (1 + tanh z) = 1 / (1 + e^(-2z)) for the quick form.
__device__ __forceinline__ float gelu_gate(float g, float u) { return (0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)))) * u; }
__device__ __forceinline__ float gelu_gate_fast(float g, float u) {
    const float z = 0.7978845608028654f * (g + 0.044715f * g * g * g);
    return (g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -2.8853900817779268f))) * u;
}
__device__ __forceinline__ float clamp_gate(float g, float u, float limit) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * (1.0f / (1.0f + expf(-1.702f * g))) * (u + 1.0f);
}
__device__ __forceinline__ float clamp_gate_fast(float g, float u, float limit) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return (g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * (-1.702f * 1.4426950408889634f)))) * (u + 1.0f);
}
template <int EPI>
__device__ __forceinline__ float gate_of(float g, float u, float limit) {
    return EPI == EPI_GATED_CLAMP_BF16 ? clamp_gate(g, u, limit) : EPI == EPI_GATED_GELU_BF16 ? gelu_gate(g, u) : silu_gate(g, u);
}
template <int EPI>
__device__ __forceinline__ float gate_fast_of(float g, float u, float limit) {
    return EPI == EPI_GATED_CLAMP_BF16 ? clamp_gate_fast(g, u, limit) : EPI == EPI_GATED_GELU_BF16 ? gelu_gate_fast(g, u) : silu_gate_fast(g, u);
}

__device__ __forceinline__ uint4 load16(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

template <int EPI>
__device__ __forceinline__ void write_out(void* C, size_t o, float v) {
    if constexpr (EPI == EPI_STORE_F32) ((float*)C)[o] = v;
    else if constexpr (EPI == EPI_ADD_F32) ((float*)C)[o] += v;
    else ((bf16_t*)C)[o] = f32_to_bf16(v);
}

// ----------------------------------------------------------------- an RMS norm between two products of a few rows
// The norm of a row x is g * x * r with r = rsqrt(mean(x^2) + eps), and r, one number a row, commutes with the product that reads
// the normed row.  A product that adds onto the rows x also writes g * x of the sums it has just made, in bfloat16, and what its
// columns give to the sum of squares of every row, one number per row and piece of the row (`NormOut`); the product that reads
// those rows multiplies its results by r, which it gets from those numbers, added in a fixed order (`NormIn`).  No kernel for
// the norm, no second pass over the rows.
struct NormOut {                 // for a product that adds onto x: all null if it does not hand the norm on
    const float* g;              // the norm's weights [N]
    bf16_t* scaled;              // out: g * x, [M, ld]
    long ld;
    float* squares;              // out: [M, parts]
};
struct NormIn {                  // for a product whose rows A are g * x without r: squares null if they are ready-made rows
    const float* squares;        // [M, parts]
    int parts;
    float eps;
    int dim;                     // r = rsqrt(sum / dim + eps)
    union {                      // (nothing of the norm's: it travels here because every kernel takes this struct)
        float limit;             // of the clamped gated epilogue
        int first;               // of the epilogue with xielu: the first column that goes through it
    };
};
// The epilogue with xielu (a feed-forward without a gate) takes no further arguments either, as longer ones made every launch of a decoded
// row slower (818 -> 831 us a step of 1B parameters with 32 bytes more): the two parameters are NormOut::g - for the kernel that takes none,
// NormIn::squares, its rows being ready-made - and the few rows' activated columns NormOut::scaled, of leading dimension NormOut::ld.

// Where an attention layer wants the sums of its q/k/v product (columns: n_heads * hd queries, n_kv * hd keys, n_kv * hd values):
// queries rotated into q_out, keys rotated and values as they are into the page table[slot][pos / page_size] at place
// pos % page_size (pairs (i, i + hd/2): a' = a cos - b sin, b' = a sin + b cos; the page's layout as the attention kernels read
// it: keys [kv_head][place][hd], then values [kv_head][hd][place]).
struct RopeStore {
    const float* cos_t;          // [M, hd/2], or null with sin_t: no rotation
    const float* sin_t;
    const int* pos;              // [M]
    const int* slot;             // [M]
    const int* table;
    int table_stride;
    bf16_t* q_out;               // [M, n_heads * hd]
    bf16_t* cache;
    long page_stride;
    int page_size, n_heads, n_kv, hd;
};


constexpr int PIPED_MAX_PARTS = 64;            // pieces of a row's sum of squares that a kernel for more than 128 rows reads

// r = rsqrt(mean square + eps) of the `rows` rows from `first` on into `scales` (LDS), by a workgroup of NT threads; rows
// beyond M get 1.  The caller puts a barrier before the use.
template <int NT>
__device__ __forceinline__ void tile_row_scales(float* scales, const NormIn& n, int first, int rows, int M) {
    for (int row = threadIdx.x; row < rows; row += NT) {
        float sum = 0.f;
        if (first + row < M)
            for (int p = 0; p < n.parts; ++p) sum += n.squares[(size_t)(first + row) * n.parts + p];
        scales[row] = first + row < M ? 1.0f / sqrtf(sum / (float)n.dim + n.eps) : 1.0f;
    }
}

// The factor of one row: rsqrt(mean square + eps) from the pieces of its sum of squares, added in their order.  The first eight
// pieces are asked for at once, by every lane (an index beyond the pieces is clamped and what it brings not added): a caller can
// ask early (`row_pieces`) and finish where the factor is needed (`row_scale_from`), with its other loads in flight in between.
struct RowPieces {
    float v[8];
};
__device__ __forceinline__ RowPieces row_pieces(const NormIn& n, int row) {
    RowPieces r;
    const float* pieces = n.squares + (size_t)row * n.parts;
#pragma unroll
    for (int u = 0; u < 8; ++u) r.v[u] = pieces[min(u, n.parts - 1)];
    return r;
}
__device__ __forceinline__ float row_scale_from(const NormIn& n, int row, const RowPieces& r) {
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (u < n.parts) sum += r.v[u];
    for (int p = 8; p < n.parts; ++p) sum += n.squares[(size_t)row * n.parts + p];
    return 1.0f / sqrtf(sum / (float)n.dim + n.eps);
}
__device__ __forceinline__ float row_scale_of(const NormIn& n, int row) { return row_scale_from(n, row, row_pieces(n, row)); }

// Where the rows of a tile of 128 go in the cache: per row the page's offset and the place in the page, and per window of
// eight rows the one in it (or -1) from which on eight rows are eight consecutive positions of one request that begin at a multiple of eight
// (rows of a prompt, wherever its first row lies in the tile).
struct TilePlaces {
    long page[128];              // page * page_stride
    int place[128];
    int run[16];
};

// One row's of it, for the row's thread (rows 64 .. and the threads of a wave go together; each row's page is two loads that depend on each other: done once per row here,
// not once per piece of a row).
struct RowPlace {
    long page;
    int place, run;
};
__device__ __forceinline__ RowPlace row_place(int row, int m0, int M, const RopeStore& rs) {
    RowPlace t;
    const int m = min(m0 + row, M - 1), p = rs.pos[m], slot = rs.slot[m];
    t.page = (long)rs.table[(size_t)slot * rs.table_stride + p / rs.page_size] * rs.page_stride;
    t.place = p % rs.page_size;
    bool begins = p % 8 == 0 && rs.page_size % 8 == 0 && row + 7 < 128 && m0 + row + 7 < M;
    if (begins) {
#pragma unroll
        for (int i = 1; i < 8; ++i) begins = begins & (rs.pos[m + i] == p + i) & (rs.slot[m + i] == slot);
    }
    const unsigned here = (unsigned)(__ballot(begins) >> (row & 56)) & 0xffu;         // (two such rows are eight apart or more)
    t.run = here ? (row & ~7) + __ffs(here) - 1 : -1;                                   // of the row's window
    return t;
}
__device__ __forceinline__ void keep_place(TilePlaces& t, int row, const RowPlace& of) {
    t.page[row] = of.page;
    t.place[row] = of.place;
    if ((row & 7) == 0) t.run[row >> 3] = of.run;
}
// Filled by the workgroup's first 128 threads; the caller puts a barrier before the use.
__device__ __forceinline__ void tile_places(TilePlaces& t, int m0, int M, const RopeStore& rs) {
    const int row = threadIdx.x;
    if (row < 128) keep_place(t, row, row_place(row, m0, M, rs));
}

// A tile of 128 x 128 sums of a q/k/v product, row-major in LDS, goes where `RopeStore` says.  Whole heads lie inside the
// tile (hd divides 128, the tile starts at a multiple of 128 columns), so the other half of every pair is in LDS too.  Queries
// and keys: a thread takes four pairs of a row at a time, whose two halves leave as 8-byte pieces of contiguous rows; the
// cosines and sines of four such items are asked for at once.  Values are stored transposed in their pages ([hd][place]),
// so they are taken column by column: runs of eight positions (`TilePlaces`) leave as 16-byte pieces, the rows that belong to none
// one by one (a step's portions begin anywhere: with runs looked for at every eighth row of the tile only, the product of a mixed step of 2,048
// rows of 5,120 x 3,072 took 125 us, 99 now).
template <int NT>
__device__ __forceinline__ void qkv_tile_rope_store(const float* tile, const TilePlaces& at, int m0, int n0, int M, int N, const RopeStore& rs) {
    const int a_dim = rs.n_heads * rs.hd, kv_dim = rs.n_kv * rs.hd, half = rs.hd / 2;
    if (n0 < a_dim + kv_dim && rs.cos_t != nullptr) {
        // An item is four pairs (i, i + hd/2) of a row: two pieces of four columns, hd/2 apart, that share their cosines and sines.
        constexpr int BATCH = 4;
        const int per_head = rs.hd / 8;                                          // items of a head; 16 items a row of the tile
        for (int e0 = threadIdx.x; e0 < 128 * 16; e0 += NT * BATCH) {
            float4 cc[BATCH], ss[BATCH];
#pragma unroll
            for (int b = 0; b < BATCH; ++b) {
                const int e = min(e0 + b * NT, 128 * 16 - 1), m = min(m0 + (e >> 4), M - 1), kq = (e & 15) % per_head;
                cc[b] = *reinterpret_cast<const float4*>(rs.cos_t + (size_t)m * half + kq * 4);
                ss[b] = *reinterpret_cast<const float4*>(rs.sin_t + (size_t)m * half + kq * 4);
            }
#pragma unroll
            for (int b = 0; b < BATCH; ++b) {
                const int e = e0 + b * NT, row = e >> 4, item = e & 15, m = m0 + row;
                const int c_lo = (item / per_head) * rs.hd + (item % per_head) * 4, col = n0 + c_lo;      // in the tile; in the product
                if (e >= 128 * 16 || m >= M || col >= a_dim + kv_dim) continue;
                const float4 a = *reinterpret_cast<const float4*>(tile + row * 128 + c_lo);
                const float4 o = *reinterpret_cast<const float4*>(tile + row * 128 + c_lo + half);
                const uint2 lo = {f32x2_to_bf16x2(a.x * cc[b].x - o.x * ss[b].x, a.y * cc[b].y - o.y * ss[b].y),
                                  f32x2_to_bf16x2(a.z * cc[b].z - o.z * ss[b].z, a.w * cc[b].w - o.w * ss[b].w)};
                const uint2 hi = {f32x2_to_bf16x2(a.x * ss[b].x + o.x * cc[b].x, a.y * ss[b].y + o.y * cc[b].y),
                                  f32x2_to_bf16x2(a.z * ss[b].z + o.z * cc[b].z, a.w * ss[b].w + o.w * cc[b].w)};
                const bool key = col >= a_dim;
                const int c = key ? col - a_dim : col;                           // the column among the queries, or the keys
                bf16_t* dst = key ? rs.cache + at.page[row] + ((size_t)(c / rs.hd) * rs.page_size + at.place[row]) * rs.hd + c % rs.hd
                                  : rs.q_out + (size_t)m * a_dim + c;
                *reinterpret_cast<uint2*>(dst) = lo;
                *reinterpret_cast<uint2*>(dst + half) = hi;
            }
        }
    } else if (n0 < a_dim + kv_dim) {                                            // no rotation: the sums as they are
        for (int e = threadIdx.x; e < 128 * 32; e += NT) {
            const int row = e >> 5, c4 = (e & 31) * 4, m = m0 + row, col = n0 + c4;
            if (m >= M || col >= a_dim + kv_dim) continue;
            const float4 v = *reinterpret_cast<const float4*>(tile + row * 128 + c4);
            const uint2 packed = {f32x2_to_bf16x2(v.x, v.y), f32x2_to_bf16x2(v.z, v.w)};
            const bool key = col >= a_dim;
            const int c = key ? col - a_dim : col;
            bf16_t* dst = key ? rs.cache + at.page[row] + ((size_t)(c / rs.hd) * rs.page_size + at.place[row]) * rs.hd + c % rs.hd
                              : rs.q_out + (size_t)m * a_dim + c;
            *reinterpret_cast<uint2*>(dst) = packed;
        }
    }
    if (n0 + 128 > a_dim + kv_dim) {
        const size_t v_plane = (size_t)rs.n_kv * rs.page_size * rs.hd;           // from a page's keys to its values
        const bool aligned = ((uintptr_t)rs.cache & 15) == 0 && rs.page_stride % 8 == 0;
        for (int e = threadIdx.x; e < 16 * 128; e += NT) {
            const int window = e >> 7, c1 = e & 127, col = n0 + c1, run = at.run[window], before = window ? at.run[window - 1] : -1;
            if (col >= N || col < a_dim + kv_dim) continue;
            const size_t c = v_plane + (size_t)(col - a_dim - kv_dim) * rs.page_size;     // (h * hd + kk) * page_size
            const bool whole = aligned && run >= 0;
            if (whole) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = tile[(run + i) * 128 + c1];
                const uint4 packed = {f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]), f32x2_to_bf16x2(v[4], v[5]), f32x2_to_bf16x2(v[6], v[7])};
                *reinterpret_cast<uint4*>(rs.cache + at.page[run] + c + at.place[run]) = packed;
            }
            // the window's rows that neither its run nor the one that reaches in from the window before covers
            const int from = max(window * 8, aligned && before >= 0 ? before + 8 : 0), to = min(whole ? run : window * 8 + 8, M - m0);
            for (int row = from; row < to; ++row) rs.cache[at.page[row] + c + at.place[row]] = f32_to_bf16(tile[row * 128 + c1]);
        }
    }
}

// ------------------------------------------------------------------------------------------ tiled
constexpr int BN = 128, BK = 64, LDS_STRIDE = BK + 8;     // +8 bf16 (16 bytes) of padding: conflict-free 16-byte reads

template <int BM, int EPI>
__global__ __launch_bounds__(256) void gemm_bf16_tiled_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C,
                                                             int M, int N, int K, long lda, long ldw, long ldc, float gate_limit) {
    constexpr int WM = BM / 2;                 // rows of a wave's tile (waves sit 2 x 2)
    constexpr int TM = WM / 32, TN = 2;        // 32x32 tiles per wave
    constexpr int A_CHUNKS = BM * BK / 8 / 256, W_CHUNKS = BN * BK / 8 / 256;   // 16-byte chunks per thread
    __shared__ __attribute__((aligned(16))) bf16_t As[BM * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) bf16_t Ws[BN * LDS_STRIDE];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * 64;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx16{};

    uint4 a_reg[A_CHUNKS], w_reg[W_CHUNKS];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int c = 0; c < A_CHUNKS; ++c) {
            const int e = tid + 256 * c, row = e / (BK / 8), kc = (e % (BK / 8)) * 8;
            const int m = m0 + row, k = k0 + kc;
            a_reg[c] = (m < M && k < K) ? load16(A + (size_t)m * lda + k) : uint4{0, 0, 0, 0};
        }
#pragma unroll
        for (int c = 0; c < W_CHUNKS; ++c) {
            const int e = tid + 256 * c, row = e / (BK / 8), kc = (e % (BK / 8)) * 8;
            const int n = n0 + row, k = k0 + kc;
            w_reg[c] = (n < N && k < K) ? load16(W + (size_t)n * ldw + k) : uint4{0, 0, 0, 0};
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int c = 0; c < A_CHUNKS; ++c) {
            const int e = tid + 256 * c, row = e / (BK / 8), kc = (e % (BK / 8)) * 8;
            *reinterpret_cast<uint4*>(&As[row * LDS_STRIDE + kc]) = a_reg[c];
        }
#pragma unroll
        for (int c = 0; c < W_CHUNKS; ++c) {
            const int e = tid + 256 * c, row = e / (BK / 8), kc = (e % (BK / 8)) * 8;
            *reinterpret_cast<uint4*>(&Ws[row * LDS_STRIDE + kc]) = w_reg[c];
        }
    };

    fetch(0);
    for (int k0 = 0; k0 < K; k0 += BK) {
        __syncthreads();                       // everyone has finished reading the previous block
        stash();
        __syncthreads();
        if (k0 + BK < K) fetch(k0 + BK);       // in flight while the products below run
        const int r = lane & 31, kq = (lane >> 5) * 8;
#pragma unroll
        for (int ks = 0; ks < BK; ks += 16) {
            bf16x8 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = as_bf16x8(*reinterpret_cast<const uint4*>(&As[(wm + i * 32 + r) * LDS_STRIDE + ks + kq]));
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = as_bf16x8(*reinterpret_cast<const uint4*>(&Ws[(wn + j * 32 + r) * LDS_STRIDE + ks + kq]));
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    // Element v of a lane's 32x32 result: row 8*(v/4) + 4*(lane/32) + v%4, column lane%32.
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3);
                const int n = n0 + wn + j * 32 + (lane & 31);
                if constexpr (is_gated(EPI)) {
                    // columns 32b .. 32b+15 are gates, 32b+16 .. 32b+31 the ups of outputs 16b .. 16b+15
                    const float up = __shfl_xor(acc[i][j][v], 16, 64);
                    if ((lane & 16) == 0 && m < M && n < N)
                        ((bf16_t*)C)[(size_t)m * ldc + (n >> 5) * 16 + (lane & 15)] = f32_to_bf16(gate_of<EPI>(acc[i][j][v], up, gate_limit));
                } else {
                    if (m < M && n < N) write_out<EPI>(C, (size_t)m * ldc + n, acc[i][j][v]);
                }
            }
}

// A tile of 128 x 128 sums, row-major in LDS, goes onto 32-bit rows, 32 threads a row with four columns each.  `old`: what the sums are
// added onto, all of a thread's rows (a row beyond M is clamped, and not written).
template <int NT>
struct TileOld { float4 v[128 / (NT / 32)]; };
template <int NT>
__device__ __forceinline__ void tile_old(TileOld<NT>& old, const float* C, long ldc, int m0, int n0, int M) {
#pragma unroll
    for (int it = 0; it < 128 / (NT / 32); ++it)
        old.v[it] = *reinterpret_cast<const float4*>(C + (size_t)min(m0 + (int)(threadIdx.x >> 5) + it * (NT / 32), M - 1) * ldc + n0 + (threadIdx.x & 31) * 4);
}
// ... where N or the rows' stride need not be whole tiles or pieces: a lane whose four columns are not whole in the rows asks for nothing.
template <int NT>
__device__ __forceinline__ void tile_old_within(TileOld<NT>& old, const float* C, long ldc, int m0, int n0, int M, int N) {
    if (n0 + (int)(threadIdx.x & 31) * 4 + 3 < N && (ldc & 3) == 0 && ((uintptr_t)C & 15) == 0) tile_old<NT>(old, C, ldc, m0, n0, M);
}
// ... with a norm handed on: the rows' new values, the same times the norm's weights in bfloat16, and the tile's piece of every row's
// sum of squares (N is a multiple of 128).
template <int NT>
__device__ __forceinline__ void tile_add_handing_norm(const float* tile, const TileOld<NT>& old, float* C, long ldc, int m0, int n0, int M, const NormOut& norm_out,
                                                      int piece, int pieces) {
    const int tid = threadIdx.x, c4 = (tid & 31) * 4;
    const float4 g = *reinterpret_cast<const float4*>(norm_out.g + n0 + c4);
#pragma unroll
    for (int it = 0; it < 128 / (NT / 32); ++it) {
        const int row = (tid >> 5) + it * (NT / 32), m = m0 + row;
        float square = 0.f;
        if (m < M) {
            const float4 t = *reinterpret_cast<const float4*>(tile + row * 128 + c4);
            float4 x = old.v[it];
            x.x += t.x; x.y += t.y; x.z += t.z; x.w += t.w;
            *reinterpret_cast<float4*>(C + (size_t)m * ldc + n0 + c4) = x;
            *reinterpret_cast<uint2*>(norm_out.scaled + (size_t)m * norm_out.ld + n0 + c4) =
                uint2{f32x2_to_bf16x2(g.x * x.x, g.y * x.y), f32x2_to_bf16x2(g.z * x.z, g.w * x.w)};
            square = x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) square += __shfl_xor(square, off, 64);
        if ((tid & 31) == 0 && m < M) norm_out.squares[(size_t)m * pieces + piece] = square;
    }
}

// Results of a prompt's product that nobody reads soon from the same L2 leave it as they come: what an L2 holds of them at a kernel's end is written back before
// the next begins.  2,048 rows of 16,384 x 2,048 gated 121 -> 116.5 us, 8,192 of 28,672 x 4,096 1,470 -> 1,433, 1,777 of 8,192 x 2,048 through xielu in its
// step 72 -> 66, 32-bit stores of 1,777 x 5,376 there 34 -> 32.  Not the rows a product adds onto, nor queries, keys and values: what reads those next got
// slower by as much (attention behind them 82.5 -> 84.3 us, the products onto 3,072 columns 90.7 -> 92.4).
typedef unsigned gi_uint4 __attribute__((ext_vector_type(4)));
typedef unsigned gi_uint2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_streaming(void* p, uint4 v) { __builtin_nontemporal_store(gi_uint4{v.x, v.y, v.z, v.w}, (gi_uint4*)p); }
__device__ __forceinline__ void store_streaming(void* p, uint2 v) { __builtin_nontemporal_store(gi_uint2{v.x, v.y}, (gi_uint2*)p); }

// ------------------------------------------------------------------------------------------ piped
// The same product for large shapes, with the operands going from global memory straight into LDS
// (global_load_lds_dwordx4: no registers in between) through a ring of blocks of 64 k, so that
// several blocks are in flight while one is multiplied.  Workgroup: 4 waves (2 x 2), a tile of
// BM x BN; a wave owns (BM/2) x (BN/2).  A stage holds BM rows of A, then BN rows of W, 128 bytes
// (a cache line) each; a wave-wide load fills 8 rows.  The 16-byte chunk c of row `row` lies at
// chunk position c ^ ((row >> 1) & 7): the loads write LDS contiguously, and the 16-byte reads
// of 16 consecutive rows (what one clock serves: 64 banks of 4 bytes) hit 16 different slots,
// without padding (a load cannot pad).  Needs K % 64 == 0; rows beyond M or N are read from the
// last valid row and their results are dropped.  With few tiles, k is split over the grid's z: each
// workgroup then writes the sums of its share to its own [M, N] slab of 32-bit partial results, and the
// reduce kernel below adds the slabs in order and applies the epilogue.
constexpr int PK = 64;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// (`tile_m`: which tile of BM rows the workgroup makes; blockIdx.x and .z say which columns and which share of k.)
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int EPI>
__device__ __forceinline__ void piped_tile(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C, int M, int N, int K, long lda,
                                           long ldw, long ldc, int k_per_split, long split_stride, const NormIn& norm_in, const RopeStore& rope,
                                           const NormOut& norm_out, const int tile_m) {
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 32, TN = WN / 32;
    constexpr int ROWS = BM + BN, STAGE_BYTES = ROWS * 128, LOADS = ROWS / 8 / (WAVES_M * WAVES_N);      // loads per wave and stage
    static_assert(ROWS % (8 * WAVES_M * WAVES_N) == 0, "the rows of a stage must divide among the waves' loads");
    static_assert(STAGES >= 2 && STAGES <= 4, "the counted waits below cover 2 to 4 stages");
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];               // STAGES * STAGE_BYTES
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WAVES_N) * WM, wn = (wave % WAVES_N) * WN;
    const int m0 = tile_m * BM, n0 = blockIdx.x * BN;

    const bf16_t* src[LOADS];                  // this lane's source of each of its wave's loads, at k = 0
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        src[i] = row < BM ? A + (size_t)min(m0 + row, M - 1) * lda + 8 * c : W + (size_t)min(n0 + row - BM, N - 1) * ldw + 8 * c;
        src[i] += (size_t)blockIdx.z * k_per_split;           // this workgroup's share of k (all of it without a split)
    }
    if (split_stride) C = (float*)C + (size_t)blockIdx.z * split_stride;       // ... and its own partial result
    // The loads are written as assembly so that the compiler does not see them: it would otherwise wait for all of
    // them before every read of LDS and at every barrier, and nothing would stay in flight.  What orders them against
    // the reads is below: the counted wait, then the barrier.
    const unsigned ring_base = (unsigned)(size_t)(lds_ptr_t)ring;
    auto issue = [&](int slot, int k0) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const unsigned dst = __builtin_amdgcn_readfirstlane(ring_base + slot * STAGE_BYTES + (wave * LOADS + i) * 1024);   // the wave's 1 KB; lane l lands at + 16 l
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src[i] + k0) : "memory", "m0");
        }
    };

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx16{};

    const int n_k = min(K - (int)blockIdx.z * k_per_split, k_per_split) / PK;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < n_k) issue(s, s * PK);
    const int r = lane & 31, swz = (r >> 1) & 7;
    const unsigned char* a_rows = ring + (wm + r) * 128;
    const unsigned char* b_rows = ring + (BM + wn + r) * 128;
    for (int it = 0; it < n_k; ++it) {
        // this wave's part of block `it` has landed when at most the loads of the blocks after it are outstanding
        const int ahead = min(n_k - 1 - it, STAGES - 2);
        if (ahead >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else if (ahead == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();          // everyone's part has landed, and everyone has finished block it-1
        asm volatile("" ::: "memory");
        if (it + STAGES - 1 < n_k) issue((it + STAGES - 1) % STAGES, (it + STAGES - 1) * PK);      // into the slot of block it-1
        const int stage_off = (it % STAGES) * STAGE_BYTES;
        // operands of the next 16 k are read while the products of these 16 run
        bf16x8 a[2][TM], b[2][TN];
        auto read_operands = [&](int ks, bf16x8* av, bf16x8* bv) {
            const int chunk = (((ks >> 3) + (lane >> 5)) ^ swz) * 16;
#pragma unroll
            for (int i = 0; i < TM; ++i) av[i] = as_bf16x8(*reinterpret_cast<const uint4*>(a_rows + stage_off + i * 32 * 128 + chunk));
#pragma unroll
            for (int j = 0; j < TN; ++j) bv[j] = as_bf16x8(*reinterpret_cast<const uint4*>(b_rows + stage_off + j * 32 * 128 + chunk));
        };
        read_operands(0, a[0], b[0]);
#pragma unroll
        for (int step = 0; step < PK / 16; ++step) {
            if (step + 1 < PK / 16) read_operands(16 * (step + 1), a[(step + 1) & 1], b[(step + 1) & 1]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[step & 1][i], b[step & 1][j], acc[i][j], 0, 0, 0);
        }
    }
    // Element v of a lane's 32x32 result: row 8*(v/4) + 4*(lane/32) + v%4, column lane%32.
    if constexpr (EPI == EPI_QKV_ROPE) {
        // The sums of a q/k/v product do not go out as they are: the tile is laid into LDS (the ring is free once everyone has
        // read the last block), scaled by a norm handed on if there is one, and leaves rotated, queries to their rows, keys and
        // values to their pages.
        static_assert(BM == 128 && BN == 128 && STAGES * STAGE_BYTES >= 128 * 128 * 4, "the tile in LDS is 128 x 128 floats");
        __shared__ float row_scale[128];
        __shared__ TilePlaces places;
        const bool scaled_rows = norm_in.squares != nullptr;
        if (scaled_rows) tile_row_scales<64 * WAVES_M * WAVES_N>(row_scale, norm_in, m0, 128, M);
        if (n0 + 128 > rope.n_heads * rope.hd) tile_places(places, m0, M, rope);       // (a tile of queries alone needs no pages)
        __syncthreads();
        float* tile = reinterpret_cast<float*>(ring);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = wm + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3);
                    tile[row * 128 + wn + j * 32 + (lane & 31)] = scaled_rows ? acc[i][j][v] * row_scale[row] : acc[i][j][v];
                }
        __syncthreads();
        qkv_tile_rope_store<64 * WAVES_M * WAVES_N>(tile, places, m0, n0, M, N, rope);
        return;
    }
    if constexpr (EPI == EPI_ADD_F32 && BM == 128 && BN == 128 && STAGES * STAGE_BYTES >= 128 * 128 * 4) {
        if (norm_out.scaled != nullptr) {
            // The sums go onto 32-bit rows whose next reader is a norm: the tile is laid into LDS (the ring is free once everyone
            // has read the last block) and leaves row by row, 32 threads a row with four columns each: the rows' new values, the
            // same times the norm's weights in bfloat16, and the tile's piece of every row's sum of squares (N is a multiple of 128).
            // What the sums are added onto is asked for first, all of a thread's rows at once (a row beyond M is clamped and not
            // written): read row by row behind the tile, it was a round trip to memory a row, eight in a row at the end of the kernel.
            constexpr int NT = 64 * WAVES_M * WAVES_N;
            TileOld<NT> old;
            tile_old<NT>(old, (const float*)C, ldc, m0, n0, M);
            __syncthreads();
            float* tile = reinterpret_cast<float*>(ring);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        tile[(wm + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3)) * 128 + wn + j * 32 + (lane & 31)] = acc[i][j][v];
            __syncthreads();
            tile_add_handing_norm<NT>(tile, old, (float*)C, ldc, m0, n0, M, norm_out, blockIdx.x, gridDim.x);
            return;
        }
    }
    float act_a = 0.f, act_b = 0.f;
    if constexpr (EPI == EPI_XIELU) { act_a = softplus_f32(norm_out.g[0]); act_b = 0.5f + softplus_f32(norm_out.g[1]); }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            [[maybe_unused]] float before[16];                                     // what sums are added onto, a result's sixteen at once (one by one 2,048 rows of 2,048 x 2,048 took 34.3 us for 30.0, 900 of 5,000 x 1,024 24.4 for 21.7)
            if constexpr (EPI == EPI_ADD_F32) {
                const int n = min(n0 + wn + j * 32 + (lane & 31), N - 1);
#pragma unroll
                for (int v = 0; v < 16; ++v) before[v] = ((const float*)C)[(size_t)min(m0 + wm + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3), M - 1) * ldc + n];
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3);
                const int n = n0 + wn + j * 32 + (lane & 31);
                if constexpr (is_gated(EPI)) {
                    const float up = __shfl_xor(acc[i][j][v], 16, 64);
                    if ((lane & 16) == 0 && m < M && n < N)
                        ((bf16_t*)C)[(size_t)m * ldc + (n >> 5) * 16 + (lane & 15)] = f32_to_bf16(gate_of<EPI>(acc[i][j][v], up, norm_in.limit));
                } else if constexpr (EPI == EPI_ADD_F32) {
                    if (m < M && n < N) ((float*)C)[(size_t)m * ldc + n] = before[v] + acc[i][j][v];
                } else if constexpr (EPI != EPI_QKV_ROPE) {
                    float sum = acc[i][j][v];
                    if constexpr (EPI == EPI_XIELU) sum = xielu(sum, act_a, act_b);
                    if (m < M && n < N) write_out<EPI>(C, (size_t)m * ldc + n, sum);
                }
            }
        }
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int EPI>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_bf16_piped_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C,
                                                             int M, int N, int K, long lda, long ldw, long ldc, int k_per_split,
                                                             long split_stride, NormIn norm_in, RopeStore rope, NormOut norm_out) {
    piped_tile<BM, BN, WAVES_M, WAVES_N, STAGES, EPI>(A, W, C, M, N, K, lda, ldw, ldc, k_per_split, split_stride, norm_in, rope, norm_out, blockIdx.y);
}

// The same tiles for many matrices at once: the rows of A lie in runs of whole tiles of 128, every run multiplied by its own
// matrix W + group * group_stride; `tile_group` [tiles] names every tile's matrix (negative: the tile is not in use).  Rows that
// fill up a run's last tile hold anything; their results are stored like the others and nobody reads them.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_bf16_grouped_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C, int M, int N,
                                                               int K, long lda, long ldw, long ldc, const int* __restrict__ tile_group, long group_stride, float gate_limit) {
    const int g = tile_group[blockIdx.y];
    if (g < 0) return;
    const NormIn no_norm_in = {nullptr, 0, 0.f, 1, gate_limit};
    const NormOut no_norm_out = {nullptr, nullptr, 0, nullptr};
    const RopeStore no_rope = {nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, nullptr, 0, 0, 0, 0, 0};
    piped_tile<128, 128, 2, 2, 2, EPI>(A, W + (size_t)g * group_stride, C, M, N, K, lda, ldw, ldc, K, 0L, no_norm_in, no_rope, no_norm_out, blockIdx.y);
}

// --------------------------------------------------------------------------------------- pingpong
// A 256 x 256 tile and LDS stages of 64 k, two of A and three of W, filled straight from global memory like the piped kernel's, with another
// order of work inside the workgroup.  Its eight waves form two groups of four, and a compute unit's four SIMDs hold
// one wave of each group.  A group alternates between a phase R in which it reads the operands of a block's 64 k from
// LDS into registers (and issues loads that refill the stages) and a phase M in which it does nothing but matrix
// instructions on them; a workgroup barrier ends every phase, and one group runs a barrier behind the other, so at any
// time one group reads while the other multiplies: on every SIMD the matrix unit always has a wave that has its
// operands at hand, instead of two waves that read together and then multiply together.
//
//   barrier number      0        1        2        3        4
//   group 0:    R(0)  |  M(0)  |  R(1)  |  M(1)  |  R(2)  | ...
//   group 1:          |  R(0)  |  M(0)  |  R(1)  |  M(1)  | ...        R(b), M(b): the phases of block b
//
// Every wave passes the same number of barriers: group 1's one ahead is matched by one more of group 0 at the end.
// Who loads which rows of which block when is said where the loads are set up, below.  Measured (cycle stamps per
// phase): M takes 1,080 clocks for its 32 matrix instructions, R 500 for its 24 reads plus what its 8 loads take to
// issue, which is what bounds the interval between two barriers; a load costs the wave that issues it
// 23 clocks when nothing else runs and 70 to 140 here, wherever in the two phases it is put.  How far ahead the loads are sent
// counts as well (all of LDS is taken for it): with two stages of W, sent for one block ahead, 8,192 rows of 28,672 x 4,096 gated took 1,558 us,
// of 4,096 x 14,336 831, of 6,144 x 4,096 368; with three 1,470, 740 and 332.  At K = 2,048, 32 blocks a tile, it is 0 to 2 %: 1,500 rows
// of 16,384 gated 104.8 and 102.6 us, 2,048 rows 118.4 and 118.0, 3,000 rows 174.8 and 174.1, 8,192 rows 460 and 451.
template <int BN, int EPI>
__global__ __launch_bounds__(512) void gemm_bf16_pingpong_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C,
                                                                int M, int N, int K, long lda, long ldw, long ldc, NormIn norm_in, RopeStore rope) {
    static_assert(BN == 256, "the sharing of the loads below is written for 256 x 256 tiles");
    constexpr int BM = 256, WAVES = 8, WM = 64, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int ROWS = BM + BN, A_BYTES = BM * 128, W_BYTES = BN * 128, LOADS = ROWS / 8 / WAVES;      // a wave-wide load fills 8 rows of 128 bytes
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];               // two blocks of A, three of W
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = wave >> 2;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;

    // Row `row` of a stage (0 .. 255: rows of A, 256 .. 511: rows of W): where this lane's 16 bytes of it lie, in bytes from the
    // tile's first row of A or of W at k = 0.  The piece c of a row lies at piece position c ^ ((row >> 1) & 7): see the piped kernel.
    // A load's address is a scalar base (the tile's first row, advanced by the block's k) plus this offset, so that issuing one
    // needs no vector instruction: those wait behind a matrix instruction that is under way.
    const bf16_t* a_tile = A + (size_t)m0 * lda;
    const bf16_t* w_tile = W + (size_t)n0 * ldw;
    auto source = [&](int row) -> unsigned {
        const int c = (lane & 7) ^ ((row >> 1) & 7);
        return row < BM ? (unsigned)(((size_t)min(row, M - 1 - m0) * lda + 8 * c) * 2) : (unsigned)(((size_t)min(row - BM, N - 1 - n0) * ldw + 8 * c) * 2);
    };
    const unsigned ring_base = (unsigned)(size_t)(lds_ptr_t)ring;
    auto load_rows = [&](unsigned from, int first_row, int block, int w_slot) {      // 8 rows from `first_row` (the same for the wave) of block `block`
        const unsigned dst = ring_base + (first_row < BM ? (block & 1) * A_BYTES + first_row * 128 : 2 * A_BYTES + w_slot * W_BYTES + (first_row - BM) * 128);
        const bf16_t* base = (first_row < BM ? a_tile : w_tile) + block * PK;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(from), "s"(base) : "memory", "m0");
    };
    // What a wave loads, 8 loads of 1 KB a block.  The memory pipeline takes such a load every 23 clocks or so, 64 of them a block:
    // three quarters of the time the block's matrix instructions take; and a wave that issues one is held for as long as the loads
    // of its workgroup that are ahead of it take, with its next instructions behind it.  So the loads are issued by the group that
    // reads, behind its reads of LDS (while it would wait for those and then for the other group's matrix instructions anyway), and
    // they are spread evenly over the block's two barrier intervals.  They are sent for as far ahead as LDS has room: A has two places, W, which
    // comes from memory where A was just written, three.  Which rows can be loaded when follows from who reads them:
    //   group 0 reads the first 128 rows of A and all of W, in the first interval of a block; group 1 the last 128 rows of A and all of W, in the second.
    //   group 0, R(b):  the last 128 rows of A of block b + 1 (group 1 read those of block b - 1 in the interval before) and half of W of block b + 2
    //   group 1, R(b):  the first 128 rows of A of block b + 2 (group 0 has just read those of block b) and the other half of W of block b + 2
    // and who has waited for them when: group 0 for its rows of A (the older of its loads) behind R(b + 1), a barrier before group 1 reads
    // them, and for its half of W behind M(b + 1); group 1 for both behind R(b + 1): in both cases a barrier before group 0's R(b + 2).
    const int turn = wave & 3;
    auto row_of = [&](int i) { return i < 4 ? (1 - group) * 128 + turn * 32 + 8 * i : BM + group * 128 + turn * 32 + 8 * (i - 4); };      // of the wave's load i
    unsigned src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) src[i] = source(row_of(i) + (lane >> 3));
    const int n_k = K / PK;
    auto load_ahead = [&](int block, int w_slot) {                                  // this wave's loads during R(block); w_slot: where W of block + 2 goes
        const int a_block = block + 1 + group;
        if (a_block < n_k) {
#pragma unroll
            for (int i = 0; i < 4; ++i) load_rows(src[i], row_of(i), a_block, 0);
        }
        if (block + 2 < n_k) {
#pragma unroll
            for (int i = 4; i < LOADS; ++i) load_rows(src[i], row_of(i), block + 2, w_slot);
        }
    };
    auto phase_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx16{};

    // to begin with: all of block 0, and of block 1 the first 128 rows of A and all of W
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_rows(source((wave * LOADS + i) * 8 + (lane >> 3)), (wave * LOADS + i) * 8, 0, 0);
    if (n_k > 1) {
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int first_row = (wave * 6 + i) * 8 + (wave * 6 + i >= 16 ? 128 : 0);
            load_rows(source(first_row + (lane >> 3)), first_row, 1, 1);
        }
    }
    // With a norm handed on (the gated product: the rows of A are g * x, and the results lack the rows' rsqrt(mean square + eps)),
    // the tile's 256 rows' factors are worked out once, a thread a row (16-byte reads of the row's pieces where they allow it: a lane
    // that asked for its rows' pieces one by one cost the kernel 18 us at 16 pieces), and wait in LDS for the epilogue (asked for behind the first block's loads; the
    // ring has no room for them before the loop is through).
    float my_row_scale = 1.0f;
    if constexpr (is_gated(EPI)) {
        if (norm_in.squares != nullptr) {
            if (tid < BM) {
                const float* pieces = norm_in.squares + (size_t)min(m0 + tid, M - 1) * norm_in.parts;
                float sum = 0.f;
                if ((norm_in.parts & 3) == 0 && ((uintptr_t)norm_in.squares & 15) == 0) {
                    for (int p = 0; p < norm_in.parts; p += 4) {
                        const float4 v = *reinterpret_cast<const float4*>(pieces + p);
                        sum += v.x; sum += v.y; sum += v.z; sum += v.w;
                    }
                } else {
                    for (int p = 0; p < norm_in.parts; ++p) sum += pieces[p];
                }
                my_row_scale = 1.0f / sqrtf(sum / (float)norm_in.dim + norm_in.eps);
            }
        }
    }
    // Likewise where the rows' keys and values go.
    [[maybe_unused]] RowPlace my_place = {0, 0, -1};
    [[maybe_unused]] bool places_wanted = false;
    if constexpr (EPI == EPI_QKV_ROPE) {
        places_wanted = n0 + BN > rope.n_heads * rope.hd;                               // (a tile of queries alone needs no pages)
        if (places_wanted && wave < 4) my_place = row_place(tid & 127, m0 + (tid & 128), M, rope);
    }
    if (n_k > 1 && !(is_gated(EPI) && norm_in.squares != nullptr) && !places_wanted) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    phase_barrier();
    if (group == 1) phase_barrier();            // group 1 runs one barrier behind group 0's phases

    const int r = lane & 31, swz = (r >> 1) & 7;
    const unsigned char* a_rows = ring + (wm + r) * 128;
    const unsigned char* b_rows = ring + 2 * A_BYTES + (wn + r) * 128;
    int w_slot = 0;
    for (int block = 0; block < n_k; ++block) {
        const int a_off = (block & 1) * A_BYTES, b_off = w_slot * W_BYTES, w_ahead = w_slot == 0 ? 2 : w_slot - 1;       // w_ahead: the place of blocks b - 1 and b + 2
        w_slot = w_slot == 2 ? 0 : w_slot + 1;
        const bool more = block + 2 < n_k;
        // ---- R: the operands of the block's 64 k into registers, and behind the reads this wave's loads
        // (two of the group's waves send their loads first and read then, two the other way round: the memory pipeline is at work
        // from the start of the interval, and nobody's reads wait behind everybody's loads)
        bf16x8 a[PK / 16][TM], b[PK / 16][TN];
        if (turn & 1) load_ahead(block, w_ahead);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int step = 0; step < PK / 16; ++step) {
            const int chunk = ((2 * step + (lane >> 5)) ^ swz) * 16;
#pragma unroll
            for (int i = 0; i < TM; ++i) a[step][i] = as_bf16x8(*reinterpret_cast<const uint4*>(a_rows + a_off + i * 32 * 128 + chunk));
#pragma unroll
            for (int j = 0; j < TN; ++j) b[step][j] = as_bf16x8(*reinterpret_cast<const uint4*>(b_rows + b_off + j * 32 * 128 + chunk));
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!(turn & 1)) load_ahead(block, w_ahead);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                          // the reads are done before anyone may refill the stage
        // (in the last block but one group 0 sends for its rows of A alone and group 1 for nothing, in the last nobody for anything)
        const bool last_rows = block + 2 == n_k;
        if (group == 0) {                                                           // the rows of A sent for a block ago have landed
            if (more) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
            else if (last_rows) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else {                                                                    // what was sent for a block ago has
            if (more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        phase_barrier();
        // ---- M: nothing but matrix instructions
#pragma unroll
        for (int step = 0; step < PK / 16; ++step)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (EPI == EPI_QKV_ROPE) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[step][i], b[step][j], acc[i][j], 0, 0, 0);
                    else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[step][j], a[step][i], acc[i][j], 0, 0, 0);
                }
        if (group == 0) {                                                           // the half of W sent for a block ago has landed
            if (more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else if (last_rows) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        phase_barrier();
    }
    if (group == 0) phase_barrier();
    if constexpr (EPI == EPI_QKV_ROPE) {
        // The sums (element v of a lane's result: row 8*(v/4) + 4*(lane/32) + v%4, column lane%32) are laid into LDS as two tiles of 128 x 128, a group's 128 rows at a
        // time, and leave rotated, queries to their rows, keys and values to their pages (some 8 us a tile beyond what stored ones take: 8,192 rows of 6,144 x 4,096 298 and 318 us).
        TilePlaces* places = reinterpret_cast<TilePlaces*>(ring + 2 * 128 * 128 * 4);
        static_assert(2 * 128 * 128 * 4 + 2 * sizeof(TilePlaces) <= 2 * A_BYTES + 3 * W_BYTES, "two tiles and their rows' places fit the ring");
        if (places_wanted && wave < 4) keep_place(places[tid >> 7], tid & 127, my_place);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (m0 + half * 128 >= M) break;
            if (group == half) {
                float* tile = reinterpret_cast<float*>(ring) + (wave & 1) * (128 * 128);
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            tile[(wm - half * 128 + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3)) * 128 + j * 32 + (lane & 31)] = acc[i][j][v];
            }
            __syncthreads();
            const float* tiles = reinterpret_cast<const float*>(ring);
            qkv_tile_rope_store<512>(tiles, places[half], m0 + half * 128, n0, M, N, rope);
            qkv_tile_rope_store<512>(tiles + 128 * 128, places[half], m0 + half * 128, n0 + 128, M, N, rope);
            __syncthreads();
        }
        return;
    }
    float* row_scale = reinterpret_cast<float*>(ring + 2 * A_BYTES + W_BYTES);      // (behind what the waves' results pass through)
    if constexpr (is_gated(EPI)) {
        if (norm_in.squares != nullptr) {
            if (tid < BM) row_scale[tid] = my_row_scale;
            __syncthreads();
        }
    }
    // The weights were the first operand: a lane's 32x32 result holds row (of A) m = lane%32 and, as element v, column
    // (row of W) n = 8*(v/4) + 4*(lane/32) + v%4, four neighbouring columns at a time.  The results leave through LDS
    // (the ring is free now: every wave has passed the barrier behind its last read), 128 bytes of 64 rows at a time
    // in a part of it that is this wave's own, so that every store instruction writes whole cache lines: eight rows of
    // 128 bytes instead of 32 pieces of 16 or 32 bytes.  Rows lie 144 bytes apart in LDS (16 consecutive rows then
    // start in 16 different groups of banks, for the 8- and 16-byte writes as for the 16-byte reads).
    constexpr int STAGE_ROW = 144;
    unsigned char* mine = ring + wave * (WM * STAGE_ROW);
    const int frow = lane >> 3, fchunk = lane & 7;                                 // the flush: lane -> (row within 8, 16-byte piece of 128)
    if constexpr (is_gated(EPI)) {
        // columns 32b .. 32b+15 are gates, 32b+16 .. 32b+31 the ups of outputs 16b .. 16b+15: element v beside element v + 8.
        // The wave's WN columns become WN/2 outputs: 2 * WN/2 bytes a row, flushed 64 outputs (128 bytes) at a time.
        static_assert(WN % 128 == 0, "the gated flush takes 64 outputs at a time");
#pragma unroll
        for (int part = 0; part < WN / 128; ++part) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const int j = 4 * part + jj;
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float rs = norm_in.squares != nullptr ? row_scale[wm + i * 32 + (lane & 31)] : 1.0f;
                        const uint2 packed = {f32x2_to_bf16x2(gate_fast_of<EPI>(acc[i][j][4 * q] * rs, acc[i][j][4 * q + 8] * rs, norm_in.limit), gate_fast_of<EPI>(acc[i][j][4 * q + 1] * rs, acc[i][j][4 * q + 9] * rs, norm_in.limit)),
                                              f32x2_to_bf16x2(gate_fast_of<EPI>(acc[i][j][4 * q + 2] * rs, acc[i][j][4 * q + 10] * rs, norm_in.limit), gate_fast_of<EPI>(acc[i][j][4 * q + 3] * rs, acc[i][j][4 * q + 11] * rs, norm_in.limit))};
                        *reinterpret_cast<uint2*>(mine + (i * 32 + (lane & 31)) * STAGE_ROW + (jj * 16 + 8 * q + 4 * (lane >> 5)) * 2) = packed;
                    }
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int it = 0; it < WM / 8; ++it) {
                const int row = it * 8 + frow, m = m0 + wm + row, c = (n0 + wn) / 2 + part * 64 + fchunk * 8;      // output column
                const uint4 v = *reinterpret_cast<const uint4*>(mine + row * STAGE_ROW + fchunk * 16);
                if (m < M && c + 7 < N / 2 && (ldc & 7) == 0) store_streaming((bf16_t*)C + (size_t)m * ldc + c, v);
                else if (m < M) {
                    const bf16_t* e = reinterpret_cast<const bf16_t*>(&v);
#pragma unroll
                    for (int x = 0; x < 8; ++x)
                        if (c + x < N / 2) ((bf16_t*)C)[(size_t)m * ldc + c + x] = e[x];
                }
            }
        }
    } else if constexpr (EPI == EPI_STORE_BF16 || EPI == EPI_XIELU) {
        if constexpr (EPI == EPI_XIELU) {
            const float act_a = softplus_f32(norm_in.squares[0]), act_b = 0.5f + softplus_f32(norm_in.squares[1]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] = xielu(acc[i][j][v], act_a, act_b);
        }
#pragma unroll
        for (int part = 0; part < TN / 2; ++part) {                                // 64 columns = 128 bytes a row at a time
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const floatx16& t = acc[i][2 * part + jj];
                        *reinterpret_cast<uint2*>(mine + (i * 32 + (lane & 31)) * STAGE_ROW + (jj * 32 + 8 * q + 4 * (lane >> 5)) * 2) =
                            uint2{f32x2_to_bf16x2(t[4 * q], t[4 * q + 1]), f32x2_to_bf16x2(t[4 * q + 2], t[4 * q + 3])};
                    }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int it = 0; it < WM / 8; ++it) {
                const int row = it * 8 + frow, m = m0 + wm + row, c = n0 + wn + part * 64 + fchunk * 8;
                const uint4 v = *reinterpret_cast<const uint4*>(mine + row * STAGE_ROW + fchunk * 16);
                if (m < M && c + 7 < N && (ldc & 7) == 0) store_streaming((bf16_t*)C + (size_t)m * ldc + c, v);
                else if (m < M) {
                    const bf16_t* e = reinterpret_cast<const bf16_t*>(&v);
#pragma unroll
                    for (int x = 0; x < 8; ++x)
                        if (c + x < N) ((bf16_t*)C)[(size_t)m * ldc + c + x] = e[x];
                }
            }
        }
    } else {
        // What the sums are added onto is asked for 32 columns ahead, all of a lane's rows at once (a row beyond M is clamped and not written): read row by row as each leaves,
        // behind the store of the one before, it was 32 round trips to memory at the end of a tile.  8,192 rows of 4,096 x 4,096 added 231.9 -> 227.3 us, 4,096 of 4,096 x 14,336 366 -> 362.
        constexpr int ROWS_OF_LANE = EPI == EPI_ADD_F32 ? WM / 8 : 1;
        [[maybe_unused]] float4 before[2][ROWS_OF_LANE];
        const bool rows_whole = (ldc & 3) == 0 && (((uintptr_t)C) & 15) == 0;
        auto ask = [&](int j, float4 (&into)[ROWS_OF_LANE]) __attribute__((always_inline)) {
            const int c = n0 + wn + j * 32 + fchunk * 4;
            if (c + 3 < N && rows_whole) {
#pragma unroll
                for (int it = 0; it < ROWS_OF_LANE; ++it) into[it] = *reinterpret_cast<const float4*>((const float*)C + (size_t)min(m0 + wm + it * 8 + frow, M - 1) * ldc + c);
            }
        };
        if constexpr (EPI == EPI_ADD_F32) ask(0, before[0]);
#pragma unroll
        for (int j = 0; j < TN; ++j) {                                             // 32 columns = 128 bytes a row at a time
            if constexpr (EPI == EPI_ADD_F32) {
                if (j + 1 < TN) ask(j + 1, before[(j + 1) & 1]);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(mine + (i * 32 + (lane & 31)) * STAGE_ROW + (8 * q + 4 * (lane >> 5)) * 4) =
                        float4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int it = 0; it < WM / 8; ++it) {
                const int row = it * 8 + frow, m = m0 + wm + row, c = n0 + wn + j * 32 + fchunk * 4;
                float4 v = *reinterpret_cast<const float4*>(mine + row * STAGE_ROW + fchunk * 16);
                if (m >= M) continue;
                float* dst = (float*)C + (size_t)m * ldc + c;
                if (c + 3 < N && rows_whole) {
                    if constexpr (EPI == EPI_ADD_F32) {
                        const float4 old = before[j & 1][it];
                        v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
                        *reinterpret_cast<float4*>(dst) = v;
                    } else {
                        store_streaming(dst, uint4{__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)});
                    }
                } else {
                    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (c + x < N) write_out<EPI>(C, (size_t)m * ldc + c + x, e[x]);
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------ tall
// The ping-pong kernel's order of work on tiles of 256 x 128 (group 0 makes the tile's first 128 rows, group 1 its last; a wave 64 x 64), for
// products that have more than one 128 x 128 tile a compute unit and no round number of 256 x 256 tiles.
// The ring has three blocks of 48 KB: in its R(b) a wave
// sends for its six loads (8 rows each) of block b + 2, whose place held block b - 1, last read by group 1 in the interval before group 0's
// R(b).  Block b + 1, sent for in R(b - 1), is read from group 0's R(b + 1) on: by the barrier before it group 0 has waited for its loads
// behind M(b) and group 1 behind R(b), each with the six of block b + 2 still in flight.
// Bound by the loads into LDS and by how far ahead they are sent: a block takes 1,720 clocks, of which its matrix instructions are 1,024; with
// two blocks in the ring and one ahead (which is all that 256 x 256 tiles leave room for) it took 2,100 to 2,600.  2,048 rows of
// 3,072 x 2,048 take 36.0 us, of 3,072 x 3,072 45, 3,072 x 8,192 104, 5,120 x 3,072 87; with two or three rounds of 128 x 128 tiles 52.5, 64,
// 137 and 115.  With several rounds a compute unit the 13 us that a tile takes to begin and to end count as much: 2,048 rows of 16,384 x 2,048
// gated take 152 us here and 120 in the ping-pong kernel, 8,192 of 28,672 x 4,096 1,660 and 1,470.  The sums of an element are
// taken in the order of the kernel with tiles of 128 x 128, whose epilogues serve, one group's 128 rows at a time.
// Which tile a workgroup makes.  Workgroups go to the eight dies in turn, each with an L2 of its own, and a die's tiles walk k together:
// what a die fetches from beyond its L2 is a strip of rows for every different row and column of tiles it holds.  So a die gets a run of
// neighbouring tiles in panels of `panel` columns, about as many bytes high as wide (2,048 x 8,192 at 3,000 and 4,096 rows: 121 -> 113 and
// 158 -> 149 us against columns dealt out in turn; nothing at short k).
struct TileOrder {
    int m_tiles, n_tiles, each, panel;         // each: tiles a die
    struct Tile { int m, n; };
    __device__ __forceinline__ Tile at(int u) const {
        const int in_panel = panel * m_tiles, p = u / in_panel, rest = u - p * in_panel, width = min(panel, n_tiles - p * panel);
        return {rest / width, p * panel + rest % width};
    }
};
// The tiles of the last, incomplete round share their k out: with at most half as many left as there are compute units, each is made by
// `shares` workgroups, every one of which sums a part of k.  The one that comes last to its end adds the others' sums to its own, in the order of k whoever it
// is, and goes on to the epilogue.  An earlier one leaves its sums in its place and ends.  A tile's two counters are drawn from when a workgroup has its sums
// and raised when these are in memory: the last waits, but only for workgroups that have drawn, whose way to the second counter holds no wait of their own
// (and not for ever: `others_came`).
// The sums go past the L2s, which belong to one die each (stores and loads of device scope): no fence, whose write-back of a whole L2 costs more than
// all of this.
struct TileShares {
    int whole, rest, shares;                   // tiles made by one workgroup; those shared out; by how many (1: none)
    float* sums;                               // [rest][shares][32,768], each in the order of the lanes' registers
    unsigned* counters;                        // [rest][2 halves][2], 0 at the start and at the end
};
__global__ void clear_counters_kernel(unsigned* counters, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) counters[i] = 0;
}
constexpr int TALL_MAX_SHARES = 4;
constexpr int DEVICE_SCOPE = 16;               // sc1 in a buffer access's cache policy
// SHARED: the launch has tiles in shares.  Launches that have none, which are most, are a kernel of their own, without the counters and the way to the shares.
template <int EPI, bool SHARED>
__global__ __launch_bounds__(512) void gemm_bf16_tall_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C, int M, int N, int K,
                                                            long lda, long ldw, long ldc, NormIn norm_in, RopeStore rope, NormOut norm_out, TileOrder order, TileShares shared, bool quick_gate) {
    int u = (blockIdx.x & 7) * order.each + (blockIdx.x >> 3), share = 0;
    bool part = false;
    if (!SHARED || (int)blockIdx.x < 8 * order.each) {
        if (u >= shared.whole) return;
    } else {                                                                            // (a die's shares are of neighbouring tiles and mostly of one part of k)
        const int id = blockIdx.x - 8 * order.each, pieces = shared.rest * shared.shares, each = (pieces + 7) / 8, piece = (id & 7) * each + (id >> 3);
        if ((id >> 3) >= each || piece >= pieces) return;
        share = piece / shared.rest;
        u = shared.whole + piece - share * shared.rest;
        part = true;
    }
    const TileOrder::Tile at_tile = order.at(u);
    constexpr int BM = 256, BN = 128, NT = 512, TM = 2, TN = 2, ROWS = BM + BN, STAGE_BYTES = ROWS * 128, LOADS = 6;
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];               // 3 * STAGE_BYTES
    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = wave >> 2, turn = wave & 3;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int m0 = at_tile.m * BM, n0 = at_tile.n * BN;
    const int all_blocks = K / PK, first_block = part ? all_blocks * share / shared.shares : 0;
    const int n_k = (part ? all_blocks * (share + 1) / shared.shares : all_blocks) - first_block;
    const bf16_t* a_tile = A + (size_t)m0 * lda + (size_t)first_block * PK;
    const bf16_t* w_tile = W + (size_t)n0 * ldw + (size_t)first_block * PK;
    auto source = [&](int row) -> unsigned {                                            // where this lane's 16 bytes of a stage's row lie, in bytes from the tile's first row of A or of W at k = 0
        const int c = (lane & 7) ^ ((row >> 1) & 7);
        return row < BM ? (unsigned)(((size_t)min(row, M - 1 - m0) * lda + 8 * c) * 2) : (unsigned)(((size_t)min(row - BM, N - 1 - n0) * ldw + 8 * c) * 2);
    };
    const unsigned ring_base = (unsigned)(size_t)(lds_ptr_t)ring;
    unsigned src[LOADS];                                                                // this wave's loads: rows (wave * 6 + i) * 8 .. + 7 of every block
#pragma unroll
    for (int i = 0; i < LOADS; ++i) src[i] = source((wave * LOADS + i) * 8 + (lane >> 3));
    auto load_block = [&](int block, int slot) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int first_row = (wave * LOADS + i) * 8;
            const unsigned dst = ring_base + slot * STAGE_BYTES + first_row * 128;
            const bf16_t* base = (first_row < BM ? a_tile : w_tile) + block * PK;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(src[i]), "s"(base) : "memory", "m0");
        }
    };
    auto phase_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx16{};
    load_block(0, 0);
    if (n_k > 1) load_block(1, 1);
    // With a norm handed on (the rows of A are g * x, and the results lack the rows' rsqrt(mean square + eps)),
    // the tile's 256 rows' factors are worked out once, a thread a row (16-byte reads of the row's pieces where they allow it: a lane
    // that asked for its rows' pieces one by one cost 18 us at 16 pieces), and wait in LDS for the epilogue (asked for behind the first
    // blocks' loads; the barriers of the loop lie between this write and the epilogue's reads).
    __shared__ float row_scale[EPI == EPI_QKV_ROPE || is_gated(EPI) ? BM : 1];
    const bool scaled_rows = (EPI == EPI_QKV_ROPE || is_gated(EPI)) && norm_in.squares != nullptr;
    if (scaled_rows && tid < BM) {
        const float* pieces = norm_in.squares + (size_t)min(m0 + tid, M - 1) * norm_in.parts;
        float sum = 0.f;
        if ((norm_in.parts & 3) == 0 && ((uintptr_t)norm_in.squares & 15) == 0) {
            for (int p = 0; p < norm_in.parts; p += 4) {
                const float4 v = *reinterpret_cast<const float4*>(pieces + p);
                sum += v.x; sum += v.y; sum += v.z; sum += v.w;
            }
        } else {
            for (int p = 0; p < norm_in.parts; ++p) sum += pieces[p];
        }
        row_scale[tid] = 1.0f / sqrtf(sum / (float)norm_in.dim + norm_in.eps);
    }
    // Likewise where the rows' keys and values go (two loads that depend on each other).
    __shared__ TilePlaces places[EPI == EPI_QKV_ROPE ? 2 : 1];
    bool asked = scaled_rows;
    if constexpr (EPI == EPI_QKV_ROPE) {
        if (n0 + BN > rope.n_heads * rope.hd) {                                          // (a tile of queries alone needs no pages)
            tile_places(places[0], m0, M, rope);
            tile_places(places[1], m0 + 128, M, rope);
            asked = true;
        }
    }
    if (n_k > 1 && !asked) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    phase_barrier();
    if (group == 1) phase_barrier();            // group 1 runs one barrier behind group 0's phases
    const int r = lane & 31, swz = (r >> 1) & 7;
    const unsigned char* a_rows = ring + (wm + r) * 128;
    const unsigned char* b_rows = ring + (BM + wn + r) * 128;
    int slot = 0;
    // Where the loop lies in memory counts: begun 8 to 24 bytes behind a multiple of 32 it takes 2 to 3 % less than at one or just before one (3,433 rows of
    // 2,048 x 8,192 stored 112.0 -> 104.9 us, added 112.3 -> 109.9; 2,048 of 3,072 x 2,048 added 34.9 -> 34.3), and what stands before it differs from end to end: the
    // kernels with shares that gate or rotate have 8 bytes more between here and there.
    if constexpr (SHARED && (is_gated(EPI) || EPI == EPI_QKV_ROPE)) asm volatile(".p2align 5");
    else asm volatile(".p2align 5\n\ts_nop 0\n\ts_nop 0");
    for (int block = 0; block < n_k; ++block) {
        const int stage_off = slot * STAGE_BYTES, ahead = slot == 0 ? 2 : slot - 1;      // ahead: the place of blocks b - 1 and b + 2
        slot = slot == 2 ? 0 : slot + 1;
        const bool more = block + 2 < n_k;
        bf16x8 a[PK / 16][TM], b[PK / 16][TN];
        if ((turn & 1) && more) load_block(block + 2, ahead);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int step = 0; step < PK / 16; ++step) {
            const int chunk = ((2 * step + (lane >> 5)) ^ swz) * 16;
#pragma unroll
            for (int i = 0; i < TM; ++i) a[step][i] = as_bf16x8(*reinterpret_cast<const uint4*>(a_rows + stage_off + i * 32 * 128 + chunk));
#pragma unroll
            for (int j = 0; j < TN; ++j) b[step][j] = as_bf16x8(*reinterpret_cast<const uint4*>(b_rows + stage_off + j * 32 * 128 + chunk));
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!(turn & 1) && more) load_block(block + 2, ahead);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                          // the reads are done before anyone may refill the stage
        // what this wave sent for a block ago has landed: group 1 sees to it here, group 0 behind its products, one barrier before group 0 reads it
        auto landed = [&]() {
            if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        };
        if (group == 1) landed();
        phase_barrier();
#pragma unroll
        for (int step = 0; step < PK / 16; ++step)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[step][i], b[step][j], acc[i][j], 0, 0, 0);
        if (group == 0) landed();
        phase_barrier();
    }
    if (group == 0) phase_barrier();
    // Element v of a lane's 32x32 result: row 8*(v/4) + 4*(lane/32) + v%4, column lane%32.  The sums leave through LDS (the ring is free:
    // every wave has passed the barrier behind its last read), a group's 128 rows at a time.
    float* tile = reinterpret_cast<float*>(ring);
    auto lay_out = [&](int half, int i, int j, const floatx16& sums) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int row = wm - half * 128 + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v & 3);
            tile[row * 128 + wn + j * 32 + (lane & 31)] = scaled_rows ? sums[v] * row_scale[half * 128 + row] : sums[v];
        }
    };
    auto leave = [&](int half, const TileOld<NT>& old) {                                 // (all of the half's rows are laid out)
        const int first = m0 + half * 128;
        __syncthreads();
        if constexpr (EPI == EPI_QKV_ROPE) {
            qkv_tile_rope_store<NT>(tile, places[half], first, n0, M, N, rope);
        } else if (EPI == EPI_ADD_F32 && norm_out.scaled != nullptr) {
            tile_add_handing_norm<NT>(tile, old, (float*)C, ldc, first, n0, M, norm_out, at_tile.n, order.n_tiles);
        } else if constexpr (is_gated(EPI)) {
            // Columns 32b .. 32b+15 are gates, 32b+16 .. 32b+31 the ups of outputs 16b .. 16b+15; a thread makes two neighbouring outputs.
            // The quick gate is the ping-pong kernel's, whose products with many tiles these may be; the others have the gate of the
            // kernel with tiles of 128 x 128, in bits (at 300 rows of 16,384 x 2,048 it costs 2.5 us of 39).
            const int o = (tid & 31) * 2, c = n0 / 2 + o;
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int row = (tid >> 5) + it * 16, m = first + row;
                if (m >= M || c >= N / 2) continue;
                const float* from = tile + row * 128 + (o >> 4) * 32 + (o & 15);
                const float2 g = *reinterpret_cast<const float2*>(from), u = *reinterpret_cast<const float2*>(from + 16);
                const uint32_t both = quick_gate ? f32x2_to_bf16x2(gate_fast_of<EPI>(g.x, u.x, norm_in.limit), gate_fast_of<EPI>(g.y, u.y, norm_in.limit))
                                                 : f32x2_to_bf16x2(gate_of<EPI>(g.x, u.x, norm_in.limit), gate_of<EPI>(g.y, u.y, norm_in.limit));
                bf16_t* to = (bf16_t*)C + (size_t)m * ldc + c;
                if ((ldc & 1) == 0 && ((uintptr_t)C & 3) == 0) {                          // (N / 2 is a multiple of 16: both exist)
                    *reinterpret_cast<uint32_t*>(to) = both;
                } else {
                    to[0] = (bf16_t)(both & 0xffffu);
                    to[1] = (bf16_t)(both >> 16);
                }
            }
        } else {
            constexpr int ELEM = EPI == EPI_STORE_BF16 || EPI == EPI_XIELU ? 2 : 4;
            float act_a = 0.f, act_b = 0.f;
            if constexpr (EPI == EPI_XIELU) { act_a = softplus_f32(norm_out.g[0]); act_b = 0.5f + softplus_f32(norm_out.g[1]); }
            const int c = n0 + (tid & 31) * 4;
            const bool whole = c + 3 < N && (ldc & 3) == 0 && ((uintptr_t)C & (4 * ELEM - 1)) == 0;
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int row = (tid >> 5) + it * 16, m = first + row;
                if (m >= M) continue;
                float4 v = *reinterpret_cast<const float4*>(tile + row * 128 + (tid & 31) * 4);
                if constexpr (EPI == EPI_XIELU) v = float4{xielu(v.x, act_a, act_b), xielu(v.y, act_a, act_b), xielu(v.z, act_a, act_b), xielu(v.w, act_a, act_b)};
                const size_t at = (size_t)m * ldc + c;
                if (whole) {
                    if constexpr (ELEM == 2) {
                        store_streaming((bf16_t*)C + at, uint2{f32x2_to_bf16x2(v.x, v.y), f32x2_to_bf16x2(v.z, v.w)});
                    } else {
                        if constexpr (EPI == EPI_ADD_F32) {
                            const float4 o = old.v[it];
                            v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
                            *reinterpret_cast<float4*>((float*)C + at) = v;
                        } else {
                            store_streaming((float*)C + at, uint4{__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)});
                        }
                    }
                } else {
                    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (c + x < N) write_out<EPI == EPI_QKV_ROPE || is_gated(EPI) ? EPI_STORE_F32 : EPI>(C, at + x, e[x]);
                }
            }
        }
        __syncthreads();
    };
    if (!part) {
        TileOld<NT> old[2];
        if constexpr (EPI == EPI_ADD_F32) {                                              // (all of a thread's rows at once: row by row as each leaves 3,000 rows of 3,072 x 3,072 took 72.3 us for 68.2)
            tile_old_within<NT>(old[0], (const float*)C, ldc, m0, n0, M, N);
            tile_old_within<NT>(old[1], (const float*)C, ldc, m0 + 128, n0, M, N);
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (m0 + half * 128 >= M) break;
            if (group == half) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) lay_out(half, i, j, acc[i][j]);
            }
            leave(half, old[half]);
        }
        return;
    }
    // A half at a time: first the one that another share would rather finish.
    __shared__ unsigned drawn[2];
    __shared__ float start[2];                                                           // 0, or no number where the others never came
    unsigned* const counters = shared.counters + (u - shared.whole) * 4;
    float* const places_of_tile = shared.sums + (size_t)(u - shared.whole) * shared.shares * (BM * BN);
    auto place = [&](int of) { return __builtin_amdgcn_make_buffer_rsrc(places_of_tile + (size_t)of * (BM * BN), 0, BM * BN * 4, 0x00027000); };
    const int at = (wave * TM * TN * 4 * 64 + lane) * 16;                                // four registers a lane and store: a wave's are 1 KB together
#pragma unroll 1
    for (int turn_of = 0; turn_of < 2; ++turn_of) {
        int half = (share & 1) ^ 1 ^ turn_of;
        asm volatile("" : "+s"(half), "+v"(tid), "+v"(lane));                            // (the compiler would keep what both turns share in registers that the sums need)
        if (m0 + half * 128 >= M) continue;                                             // (nobody has rows there)
        unsigned* const counter = counters + 2 * half;
        if (tid == 0) drawn[turn_of] = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if ((int)drawn[turn_of] + 1 < shared.shares) {
            if (group == half) {
                const auto mine = place(share);
#pragma unroll
                for (int f = 0; f < TM * TN * 4; ++f) {
                    const floatx16& from = acc[f >> 3][(f >> 2) & 1];
                    const int v = (f & 3) * 4;
                    __builtin_amdgcn_raw_buffer_store_b128(gi_uint4{__float_as_uint(from[v]), __float_as_uint(from[v + 1]), __float_as_uint(from[v + 2]), __float_as_uint(from[v + 3])},
                                                           mine, at, f * 1024, DEVICE_SCOPE);
                }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                         // this wave's sums are in memory
            }
            __syncthreads();
            if (tid == 0) __hip_atomic_fetch_add(counter + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            continue;
        }
        TileOld<NT> old;
        if constexpr (EPI == EPI_ADD_F32) tile_old_within<NT>(old, (const float*)C, ldc, m0 + half * 128, n0, M, N);
        if (tid == 0) start[turn_of] = others_came(counter + 1, shared.shares - 1) ? 0.f : __builtin_nanf("");
        __syncthreads();
        if (tid < 2) __hip_atomic_store(counter + tid, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // as the next product of the step wants them
        if (group == half) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                floatx16 total[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j) total[j] = floatx16{} + start[turn_of];
#pragma unroll 1
                for (int of = 0; of < shared.shares; ++of) {
                    if (of == share) {
#pragma unroll
                        for (int j = 0; j < TN; ++j) total[j] += acc[i][j];
                        continue;
                    }
                    const auto theirs = place(of);
                    gi_uint4 sums[TN * 4];
#pragma unroll
                    for (int f = 0; f < TN * 4; ++f) sums[f] = __builtin_amdgcn_raw_buffer_load_b128(theirs, at, (i * TN * 4 + f) * 1024, DEVICE_SCOPE);
#pragma unroll
                    for (int f = 0; f < TN * 4; ++f)
#pragma unroll
                        for (int e = 0; e < 4; ++e) total[f >> 2][(f & 3) * 4 + e] += __uint_as_float(sums[f][e]);
                }
#pragma unroll
                for (int j = 0; j < TN; ++j) lay_out(half, i, j, total[j]);
            }
        }
        leave(half, old);
    }
}

// ----------------------------------------------------------------------------------------- skinny
// Workgroup: 8 waves = 4 strips of 16 weight rows x 2 halves of each 256-wide block of k; the
// workgroup covers 64 weight rows and the k range [k_begin, k_end) of its grid row.  Weights stream
// from HBM straight into registers, two blocks ahead of their use: for the j-th product of a
// block, lane (r = lane%16, q = lane/16) holds k0 + 128*half + 32j + 8q .. +8 of weight row r, so
// the four lanes of a row read 64 contiguous bytes per load.  The activations of a block go
// through LDS (they are shared by the strips) and are fetched into registers one block ahead.
// Cycle stamps of a workgroup's blocks (64 rows, gate/up: 5,300 clocks a block) showed a wait for every load in flight where the
// block's activations are stored into LDS (the weights asked for one block earlier included: the compiler counts loads exactly
// only if none of them is skipped by a lane or a block) and the products waiting for one LDS read each (1,250 clocks for 16
// products); with every load issued by everyone, barriers that wait for LDS only and the reads one product ahead: 850 clocks for
// the products, gate/up 21.4 -> 18.8 us at 17 rows, 25.5 -> 23.1 at 64, the decode step 2 to 3 % shorter at 17 to 128 rows.
// (Up to four tiles of rows the kernel stays within 128 registers, two workgroups a compute unit.)
// The halves' sums meet in LDS.  PARTIAL: the sums of the k range go to P[split][M][N] and a
// second kernel adds the splits in order; otherwise the workgroup saw all of k and writes the
// result with its epilogue itself.
constexpr int SK = 128;                               // k per product group of a wave (4 products of 32)
constexpr int SKINNY_MAX_ROWS = 128;                  // rows of A the skinny kernel takes (8 tiles of 16)
constexpr int KB = 2 * SK, X_STRIDE = KB + 8;         // k per block of the workgroup; +8 bf16 of padding

// The kernel for at most 16 rows: a thread keeps 8 pieces while the products run (more would cost the kernel its second
// workgroup per compute unit); 64 threads share a row where there are at most 8 rows, 32 otherwise.
constexpr int SLIM_PIECES = 8;
__host__ __device__ constexpr int slim_max_parts(int M) { return SLIM_PIECES * (M <= 8 ? 64 : 32); }
// The kernels for 17 to 128 rows: the kernel that adds the partial sums onto x writes one piece per 1024 columns.
constexpr int REDUCE_COLUMNS = 1024, REDUCE_MAX_PARTS = 8;


// The same for all M rows into `scales` (LDS, at least 32 floats or M), by a workgroup of 512 threads; the caller puts a barrier
// before the use.  With many pieces (the writer was a kernel for at most 32 rows with a piece per workgroup: at most
// TILES_MAX_PARTS for 17 to 32 rows, slim_max_parts for fewer) 16 or 32 threads share a row and ask for 16 pieces each at once.
constexpr int TILES_MAX_PARTS = 256;
__device__ __forceinline__ void row_pieces_shared(const NormIn& n, int M, int sharing, float (&piece)[16]) {
    const int row = threadIdx.x / sharing, at = threadIdx.x % sharing;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int p = at + sharing * i;
        piece[i] = (row < M && p < n.parts) ? n.squares[(size_t)row * n.parts + p] : 0.f;
    }
}
__device__ __forceinline__ void row_scales_shared(float* scales, const NormIn& n, int M, int sharing, const float (&piece)[16]) {
    const int row = threadIdx.x / sharing, at = threadIdx.x % sharing;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum += piece[i];
    if (sharing == 32) sum += __shfl_xor(sum, 16, 64);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (at == 0 && row < M) scales[row] = 1.0f / sqrtf(sum / (float)n.dim + n.eps);
}
__device__ __forceinline__ void row_scales_into(float* scales, const NormIn& n, int M) {
    const int tid = threadIdx.x;
    if (n.parts <= REDUCE_MAX_PARTS) {
        if (tid < M) scales[tid] = row_scale_of(n, tid);
        return;
    }
    const int sharing = M <= 16 ? 32 : 16;                                                 // M <= 32 here
    float piece[16];
    row_pieces_shared(n, M, sharing, piece);
    row_scales_shared(scales, n, M, sharing, piece);
}

template <int MT, int EPI, bool PARTIAL>
__global__ __launch_bounds__(512, MT == 2 ? 4 : 2) void gemm_bf16_skinny_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C,
                                                              float* __restrict__ P, int M, int N, int K, long lda, long ldw, long ldc,
                                                              int k_per_split, NormIn norm_in) {
    __shared__ __attribute__((aligned(16))) bf16_t Xs[MT * 16 * X_STRIDE];
    __shared__ float other[4][MT][64][4];
    __shared__ float row_scale[MT * 16 < 32 ? 32 : MT * 16];
    const bool scaled_rows = !PARTIAL && norm_in.squares != nullptr;       // the rows of A lack their norm's rsqrt(mean square + eps)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int strip = wave & 3, half = wave >> 2;
    const int r = lane & 15, q = lane >> 4;
    const int n = blockIdx.x * 64 + strip * 16 + r;
    const int k_begin = blockIdx.y * k_per_split, k_end = min(K, k_begin + k_per_split);
    const bf16_t* wrow = W + (size_t)min(n, N - 1) * ldw + SK * half + 8 * q;

    floatx4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = floatx4{};

    // Every load of the loop is issued by every lane in every block (addresses beyond the range are clamped into it) and the
    // barriers wait for LDS only, so the compiler counts the loads in flight exactly: a block waits for its own activations and
    // weights and leaves the two blocks of weights and the block of activations behind them on their way (with a load that some
    // lanes or blocks skip it waits for all of them at the first use).  What a clamped load brings is finite and meets a zero or
    // is dropped: weights of k beyond the range are replaced by zeros where the range's last block is ragged, and results of rows
    // beyond M are never written.
    uint4 w_buf[3][4], x_reg[MT];
    const int w_last = K - 8 - (SK * half + 8 * q);           // the last 16 bytes of a weight row, from `wrow`
    auto fetch_w = [&](int k0, uint4 (&w)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = load16(wrow + min(k0 + 32 * j, w_last));
    };
    const int x_row = tid / (KB / 8), x_k = (tid % (KB / 8)) * 8;             // of this thread's first 16 bytes of a block; its others lie 16 rows further each
    auto fetch_x = [&](int k0) {
#pragma unroll
        for (int c = 0; c < MT; ++c) x_reg[c] = load16(A + (size_t)min(x_row + 16 * c, M - 1) * lda + min(k0 + x_k, K - 8));
    };
    fetch_x(k_begin);
    fetch_w(k_begin, w_buf[0]);
    fetch_w(k_begin + KB, w_buf[1]);
    if (scaled_rows) row_scales_into(row_scale, norm_in, M);                   // (the loop's barriers lie before its use)
    // One block of 256 k: `w_use` holds its weights, `w_fill` takes those of the block after the next.  The activations of the
    // products' next 32 k are read from LDS while those of these 32 are multiplied.
    auto block = [&](int kk, const uint4 (&w_use)[4], uint4 (&w_fill)[4]) __attribute__((always_inline)) {
        barrier_lds();                                // everyone has finished reading the previous block
#pragma unroll
        for (int c = 0; c < MT; ++c) {
            const int e = tid + 512 * c;
            *reinterpret_cast<uint4*>(&Xs[(e / (KB / 8)) * X_STRIDE + (e % (KB / 8)) * 8]) = x_reg[c];
        }
        barrier_lds();
        fetch_x(kk + KB);
        fetch_w(kk + 2 * KB, w_fill);
        const bool ragged = kk + KB > k_end;          // the same for the whole workgroup
        const bf16_t* x_rows = &Xs[r * X_STRIDE + SK * half + 8 * q];
        bf16x8 a[2][MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) a[0][t] = as_bf16x8(*reinterpret_cast<const uint4*>(x_rows + t * 16 * X_STRIDE));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j + 1 < 4) {
#pragma unroll
                for (int t = 0; t < MT; ++t) a[(j + 1) & 1][t] = as_bf16x8(*reinterpret_cast<const uint4*>(x_rows + t * 16 * X_STRIDE + 32 * (j + 1)));
            }
            uint4 w = w_use[j];
            if (ragged && kk + SK * half + 32 * j + 8 * q >= k_end) w = uint4{0, 0, 0, 0};
            const bf16x8 b = as_bf16x8(w);
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j & 1][t], b, acc[t], 0, 0, 0);
        }
    };
    int kk = k_begin;
    for (; kk + 2 * KB < k_end; kk += 3 * KB) {       // three blocks a trip (the last may be ragged): the buffers' roles come round
        block(kk, w_buf[0], w_buf[2]);
        block(kk + KB, w_buf[1], w_buf[0]);
        block(kk + 2 * KB, w_buf[2], w_buf[1]);
    }
    if (kk < k_end) {
        block(kk, w_buf[0], w_buf[2]);
        if (kk + KB < k_end) block(kk + KB, w_buf[1], w_buf[0]);
    }
    // the second half's sums join the first's
    if (half == 1) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) other[strip][t][lane][v] = acc[t][v];
    }
    __syncthreads();
    if (half == 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[t][v] += other[strip][t][lane][v];
    }
    // Element v of a lane's 16x16 result: row (activation row) 4*(lane/16) + v, column (weight row) lane%16.
    if constexpr (is_gated(EPI) && !PARTIAL) {
        // strips 0 and 2 hold gates, strips 1 and 3 the ups of the same outputs: the ups cross over through LDS
        __syncthreads();
        if (half == 0 && (strip & 1)) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) other[strip][t][lane][v] = acc[t][v];
        }
        __syncthreads();
        if (half == 0 && !(strip & 1) && n < N) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = t * 16 + 4 * q + v;
                    const float rs = scaled_rows ? row_scale[m] : 1.0f;
                    if (m < M) ((bf16_t*)C)[(size_t)m * ldc + blockIdx.x * 32 + (strip >> 1) * 16 + r] = f32_to_bf16(gate_of<EPI>(acc[t][v] * rs, other[strip + 1][t][lane][v] * rs, norm_in.limit));
                }
        }
    } else if (half == 0 && n < N) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = t * 16 + 4 * q + v;
                if (m >= M) continue;
                if constexpr (PARTIAL) P[((size_t)blockIdx.y * M + m) * N + n] = acc[t][v];
                else write_out<EPI>(C, (size_t)m * ldc + n, scaled_rows ? acc[t][v] * row_scale[m] : acc[t][v]);
            }
    }
}

// Where in its steps of 64 k a workgroup of the kernels for few rows begins: all at the same k would ask the same memory channels, and the same of an L2's for the rows that they
// share.  Workgroups go to the eight compute dies in turn, so those of one die take the places 3, 6, 9, ... apart, modulo a power of two (`turn` + 1).  Microseconds with one place for
// all, with the workgroup's number, and so: 16,384 x 2,048 gated at 64 rows 18.2, 17.1, 16.1, at 24 rows 17.2, 15.8, 14.5, at one row 12.6, 12.1, 12.2; 28,672 x 4,096 gated at 8 rows
// 43.0 with its number, 41.4, at 64 rows 54.1, 50.7, 49.9; 128,256 x 2,048 at 64 rows 119.7, 120.9, 115.9.
__device__ __forceinline__ int first_step(int turn) { return (int)((blockIdx.x >> 3) * 3) & turn; }
static int turn_of_steps(int steps) {
    int turn = 1;
    while (2 * turn <= steps) turn *= 2;
    return turn - 1;
}

// ------------------------------------------------------------------------------------------ strips
// All rows of A (up to 32 TM of them) against 64 rows of W and the k range of the workgroup's grid row: both operands go from memory straight into
// a ring of LDS stages of 64 k (chunks placed as in the kernels above), STAGES - 1 of them in flight.  Eight waves: two halves of 32
// columns times four quarters of every stage's k, so that a wave's one fragment of weights meets all rows and a fragment of rows is read by two waves only; the
// quarters' sums meet in LDS, (0 + 2) + (1 + 3).  A wave reads the next stage's operands while it multiplies this one's.
// Bound by the weights on their way from memory (a strip of 64 rows gives 256 workgroups 28 to 56 KB each of them in flight), and from 100 rows or so on by what
// a unit takes in of A besides: one tile for all rows reads the weights once, where 131 rows in two tiles of 128 had half of the units load them for three rows.  Microseconds
// a product, in a captured chain of products that each have weights of their own (640 MB of them a chain), with the kernel that adds up where k is shared out; before (weights
// through registers up to 128 rows, tiles of 128 x 128 above) and now:
//   rows                     17            64            128           131           192
//   16,384 x 2,048 gated     18.2, 14.7    21.8, 16.1    29.8, 21.5    28.4, 21.8    28.9, 25.8
//   28,672 x 4,096 gated     53.2, 43.0    63.3, 49.9    90.0, 65.0    (as before)
//   2,048 x 2,048 added      (other)       10.1, 9.4     14.0, 11.0    14.5, 11.1    16.7, 11.9
//   2,048 x 8,192 added      12.8, 11.8    15.1, 13.5    20.4, 17.9    23.8, 19.0    25.4, 21.6
//   3,072 x 8,192 added      17.9, 15.4    21.2, 17.7    27.2, 22.5    37.5, 23.3    39.7, 28.3
//   4,096 x 14,336 added     27.2, 26.0    33.6, 30.0    42.9, 39.5    57.0, 38.5    59.9, 46.9
//   128,256 x 2,048 stored   107.1, 101.9  134.7, 121.1  184.7, 149.2  (as before)
// The sums of a product have fewer and longer chains than before; against 64 bits they are nearer (2,048 x 8,192: 1.1e-7 for 1.4 to 1.9e-7).
constexpr int strip_ring(int tm, int stages) { return stages * (64 + 32 * tm) * 128; }
constexpr int strip_chunk(int tm, int stages) { return strip_ring(tm, stages) / 32768 < tm ? strip_ring(tm, stages) / 32768 : tm; }       // fragments whose quarters' sums fit the ring
constexpr int strip_bytes(int tm, int stages) {
    const int end = strip_chunk(tm, stages) * 32768 + (tm <= 4 ? 32 * tm * 4 : 0);
    return strip_ring(tm, stages) > end ? strip_ring(tm, stages) : end;
}
template <int TM, int STAGES, int EPI, bool PARTIAL>
__global__ __launch_bounds__(512, TM <= 2 ? 4 : 2) void gemm_bf16_strip_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C,
                                                                              float* __restrict__ P, int all_rows, int N, int K, long lda, long ldw, long ldc, int k_per_split, int tile_rows, int turn, NormIn norm_in) {
    const int m_first = PARTIAL ? blockIdx.z * tile_rows : 0, M = PARTIAL ? min(tile_rows, all_rows - m_first) : all_rows;       // of this tile
    constexpr int BM = 32 * TM, STAGE_BYTES = (64 + BM) * 128, CHUNK = strip_chunk(TM, STAGES);
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];               // strip_bytes(TM, STAGES)
    float* const row_scale = reinterpret_cast<float*>(ring + CHUNK * 32768);            // (behind the sums of the end)
    const bool scaled_rows = TM <= 4 && !PARTIAL && norm_in.squares != nullptr;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The pieces of the rows' sums of squares: asked for ahead of everything, used at the end.  Up to 32 rows they may be many (`row_scales_into`).
    constexpr int EACH = TM == 1 ? 16 : 1;
    const int sharing = M <= 16 ? 32 : 16;
    [[maybe_unused]] RowPieces pieces;
    [[maybe_unused]] float piece[EACH];
    if constexpr (TM == 1) {
        if (scaled_rows) row_pieces_shared(norm_in, M, sharing, piece);
    } else {
        if (scaled_rows && tid < M) pieces = row_pieces(norm_in, tid);
    }
    const int half = wave & 1, quarter = wave >> 1, n0 = blockIdx.x * 64;
    const int k_begin = blockIdx.y * k_per_split, n_k = (min(K, k_begin + k_per_split) - k_begin) / PK;
    // A wave loads eight rows of W and every eighth group of eight rows of A; groups beyond M are left out (what then lies in LDS makes rows that nobody writes).
    constexpr int MOST = (BM / 8 + 7) / 8;                                              // (M > BM - 32: a wave has so many groups, or one fewer)
    const bool most = wave + 8 * (MOST - 1) < (M + 7) / 8;
    const bf16_t *w_tile = W + (size_t)n0 * ldw + k_begin, *a_tile = A + (size_t)m_first * lda + k_begin;
    unsigned w_src, a_src[MOST];
    {
        const int row = wave * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        w_src = (unsigned)(((size_t)min(row, N - 1 - n0) * ldw + 8 * c) * 2);
#pragma unroll
        for (int i = 0; i < MOST; ++i) {
            const int r = row + 64 * i;
            a_src[i] = (unsigned)(((size_t)min(r, M - 1) * lda + 8 * c) * 2);           // (rows 64 apart have the same permutation of chunks)
        }
    }
    const unsigned ring_base = (unsigned)(size_t)(lds_ptr_t)ring;
    const int first_block = first_step(turn + 1 > n_k ? 0 : turn);
    auto issue = [&](int step_, int slot) {
        const int ahead = step_ + first_block, block = ahead < n_k ? ahead : ahead - n_k;
        const unsigned at = ring_base + slot * STAGE_BYTES + wave * 1024;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at), "v"(w_src), "s"(w_tile + block * PK) : "memory", "m0");
#pragma unroll
        for (int i = 0; i < MOST; ++i)
            if (i + 1 < MOST || most)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at + (64 + 64 * i) * 128), "v"(a_src[i]), "s"(a_tile + block * PK) : "memory", "m0");
    };
    // waits until at most the loads of so many stages are outstanding
#define LOADS_OF(N_)                                                                                                                    \
    do {                                                                                                                                \
        if (most) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((N_) * (1 + MOST)) : "memory");                                              \
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((N_) * MOST) : "memory");                                                         \
    } while (0)
    auto wait = [&](int stages) {
        static_assert(STAGES >= 3 && STAGES <= 8 && (STAGES - 1) * (1 + MOST) < 64, "waits for 0 to 7 stages");
        if (stages >= STAGES - 1) LOADS_OF(STAGES - 1);
        else if (stages == STAGES - 2) LOADS_OF(STAGES - 2);
        else if (stages == 1) LOADS_OF(1);
        else if (stages == 2) LOADS_OF(2);
        else if (stages == 3) LOADS_OF(3);
        else if (stages == 4) LOADS_OF(4);
        else if (stages == 5) LOADS_OF(5);
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
#undef LOADS_OF
    floatx16 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i] = floatx16{};
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < n_k) issue(s, s);
    const int r = lane & 31, chunk = ((quarter * 2 + (lane >> 5)) ^ ((r >> 1) & 7)) * 16;
    const unsigned char *w_at = ring + (half * 32 + r) * 128 + chunk, *a_at = ring + (64 + r) * 128 + chunk;
    bf16x8 w[2], a[2][TM];
    auto read = [&](int slot, int into) {
        w[into] = as_bf16x8(*reinterpret_cast<const uint4*>(w_at + slot * STAGE_BYTES));
#pragma unroll
        for (int i = 0; i < TM; ++i) a[into][i] = as_bf16x8(*reinterpret_cast<const uint4*>(a_at + slot * STAGE_BYTES + i * 32 * 128));
    };
    auto meet = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    wait(min(n_k, STAGES) - 1);
    meet();
    read(0, 0);
    int slot = 0;
    auto step = [&](int it, int now) __attribute__((always_inline)) {
        const int here = slot;
        slot = slot + 1 == STAGES ? 0 : slot + 1;
        __builtin_amdgcn_s_waitcnt(0xc07f);                                             // lgkmcnt(0), in a form that the compiler counts with: this wave has read stage `it`
        if (it + 1 < n_k) {
            if (it + STAGES <= n_k) wait(STAGES - 2);                                   // its part of stage it + 1 has landed
            else wait(n_k - 2 - it);
            meet();                                                                     // everyone's; everyone has read stage `it`
            read(slot, now ^ 1);
            if (it + STAGES < n_k) issue(it + STAGES, here);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[now][i], w[now], acc[i], 0, 0, 0);
    };
    for (int it = 0; it < n_k; it += 2) {
        step(it, 0);
        if (it + 1 < n_k) step(it + 1, 1);
    }
    // Element v of a lane's 32x32 result: row 8*(v/4) + 4*(lane/32) + v%4, column lane%32.  CHUNK fragments of rows at a time.
    float4* const sums = reinterpret_cast<float4*>(ring);                               // [quarter][half][fragment][v / 4][lane]
    auto at = [&](int of_quarter, int of_half, int f, int vg, int of_lane) { return (((of_quarter * 2 + of_half) * CHUNK + f) * 4 + vg) * 64 + of_lane; };
    auto sum_of = [&](int of_half, int f, int vg, int of_lane) {
        const float4 s0 = sums[at(0, of_half, f, vg, of_lane)], s1 = sums[at(1, of_half, f, vg, of_lane)], s2 = sums[at(2, of_half, f, vg, of_lane)], s3 = sums[at(3, of_half, f, vg, of_lane)];
        return float4{(s0.x + s2.x) + (s1.x + s3.x), (s0.y + s2.y) + (s1.y + s3.y), (s0.z + s2.z) + (s1.z + s3.z), (s0.w + s2.w) + (s1.w + s3.w)};
    };
#pragma unroll
    for (int first = 0; first < TM; first += CHUNK) {
        __syncthreads();
        if (first == 0 && scaled_rows) {
            if constexpr (TM == 1) row_scales_shared(row_scale, norm_in, M, sharing, piece);
            else if (tid < M) row_scale[tid] = row_scale_from(norm_in, tid, pieces);
        }
#pragma unroll
        for (int f = 0; f < CHUNK; ++f)
            if (first + f < TM) {
#pragma unroll
                for (int vg = 0; vg < 4; ++vg) {
                    const floatx16& from = acc[first + f < TM ? first + f : 0];
                    sums[at(quarter, half, f, vg, lane)] = float4{from[4 * vg], from[4 * vg + 1], from[4 * vg + 2], from[4 * vg + 3]};
                }
            }
        __syncthreads();
        const int here = min(CHUNK, TM - first);
        if constexpr (is_gated(EPI) && !PARTIAL) {
            // columns 0 .. 15 of a half are gates, 16 .. 31 the ups of the same outputs
            for (int e = wave; e < here * 4; e += 8) {
                const int f = e >> 2, vg = e & 3, o = lane & 31, from = (o & 15) + (lane & 32), row = (first + f) * 32 + 8 * vg + 4 * (lane >> 5);
                const float4 g = sum_of(o >> 4, f, vg, from), u = sum_of(o >> 4, f, vg, from + 16);
                const float gs[4] = {g.x, g.y, g.z, g.w}, us[4] = {u.x, u.y, u.z, u.w};
                if (n0 + (o >> 4) * 32 >= N) continue;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (row + v < M) {
                        const float rs = scaled_rows ? row_scale[row + v] : 1.0f;
                        ((bf16_t*)C)[(size_t)(row + v) * ldc + n0 / 2 + o] = f32_to_bf16(gate_of<EPI>(gs[v] * rs, us[v] * rs, norm_in.limit));
                    }
            }
        } else {
            for (int e = wave; e < here * 8; e += 8) {
                const int f = e >> 3, vg = e & 3, of_half = (e >> 2) & 1, n = n0 + of_half * 32 + (lane & 31), row = (first + f) * 32 + 8 * vg + 4 * (lane >> 5);
                const float4 s = sum_of(of_half, f, vg, lane);
                const float ss[4] = {s.x, s.y, s.z, s.w};
                if (n >= N) continue;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (row + v < M) {
                        if constexpr (PARTIAL) P[((size_t)blockIdx.y * all_rows + m_first + row + v) * N + n] = ss[v];
                        else write_out<EPI>(C, (size_t)(row + v) * ldc + n, scaled_rows ? ss[v] * row_scale[row + v] : ss[v]);
                    }
            }
        }
    }
}

// Adds the k-split partial sums [splits][M][N] in ascending split order and writes the result.  A thread takes VEC neighbouring
// columns and asks for its values of up to eight splits at once: the kernel is one round trip to memory, not one per split.
// With `norm_in` the sums are multiplied by their row's rsqrt(mean square + eps).  With `norm_out` (adding onto 32-bit rows, four
// columns a thread, rows of a multiple of 1024 columns: a workgroup then lies in one row, and no workgroup is cut short) the rows'
// new values times g go out in bfloat16 beside them, and the workgroup's share of the row's sum of squares.
template <int EPI, int VEC>
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float* __restrict__ P, void* __restrict__ C, int M, int N, int splits, long ldc,
                                                            NormIn norm_in, NormOut norm_out) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC, slab = (size_t)M * N;
    if (i >= slab) return;
    const size_t row = i / N, col = i % N, o = row * ldc + col;      // (VEC divides N: the VEC columns lie in one row)
    // Everything the result needs besides the partial sums (the row's pieces of the norm before, the old values and the gains of
    // the norm behind) is asked for ahead of them: one round trip to memory for all of it, not one after the other.
    [[maybe_unused]] RowPieces pieces;
    if (norm_in.squares != nullptr) pieces = row_pieces(norm_in, (int)row);
    [[maybe_unused]] float4 old4 = {0.f, 0.f, 0.f, 0.f}, gain4 = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC == 4 && EPI == EPI_ADD_F32) {
        old4 = *reinterpret_cast<const float4*>((const float*)C + o);
        if (norm_out.scaled != nullptr) gain4 = *reinterpret_cast<const float4*>(norm_out.g + col);
    }
    float s[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) s[v] = 0.f;
    for (int sp0 = 0; sp0 < splits; sp0 += 8) {
        float part[8][VEC];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float* src = P + (size_t)min(sp0 + u, splits - 1) * slab + i;
            if constexpr (VEC == 4) {
                const float4 x = *reinterpret_cast<const float4*>(src);
                part[u][0] = x.x; part[u][1] = x.y; part[u][2] = x.z; part[u][3] = x.w;
            } else {
                part[u][0] = *src;
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (sp0 + u < splits) {
#pragma unroll
                for (int v = 0; v < VEC; ++v) s[v] += part[u][v];
            }
    }
    if (norm_in.squares != nullptr) {
        const float rs = row_scale_from(norm_in, (int)row, pieces);
#pragma unroll
        for (int v = 0; v < VEC; ++v) s[v] *= rs;
    }
    if constexpr (VEC == 4) {                                        // (the host has checked that rows of C start at multiples of 16 bytes)
        if constexpr (EPI == EPI_STORE_BF16) {
            uint2 packed;
            packed.x = (unsigned)f32_to_bf16(s[0]) | ((unsigned)f32_to_bf16(s[1]) << 16);
            packed.y = (unsigned)f32_to_bf16(s[2]) | ((unsigned)f32_to_bf16(s[3]) << 16);
            *reinterpret_cast<uint2*>((bf16_t*)C + o) = packed;
        } else {
            float4* dst = reinterpret_cast<float4*>((float*)C + o);
            float4 x = old4;
            x.x += s[0]; x.y += s[1]; x.z += s[2]; x.w += s[3];
            *dst = x;
            if constexpr (EPI == EPI_ADD_F32) {
                if (norm_out.scaled != nullptr) {                    // (the same for every thread of the kernel)
                    __shared__ float wave_squares[4];
                    const float4 g = gain4;
                    uint2 packed;
                    packed.x = (unsigned)f32_to_bf16(g.x * x.x) | ((unsigned)f32_to_bf16(g.y * x.y) << 16);
                    packed.y = (unsigned)f32_to_bf16(g.z * x.z) | ((unsigned)f32_to_bf16(g.w * x.w) << 16);
                    *reinterpret_cast<uint2*>(norm_out.scaled + row * norm_out.ld + col) = packed;
                    float square = (x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w);
#pragma unroll
                    for (int off = 32; off > 0; off >>= 1) square += __shfl_xor(square, off, 64);
                    if ((threadIdx.x & 63) == 0) wave_squares[threadIdx.x >> 6] = square;
                    __syncthreads();
                    if (threadIdx.x == 0) {
                        const int per_row = N / REDUCE_COLUMNS;
                        norm_out.squares[row * per_row + blockIdx.x % per_row] = (wave_squares[0] + wave_squares[1]) + (wave_squares[2] + wave_squares[3]);
                    }
                }
            }
        }
    } else {
        write_out<EPI>(C, o, s[0]);
    }
}

// The same sums onto 32-bit rows, whole rows at a time (a workgroup a row of up to 4096 columns), and the norm that reads the rows next beside them:
// out = bfloat16(g * (x * rsqrt(mean(x^2) + eps))), as the norm's own kernel makes it, in bits.  131 rows of 2,048 out of eight shares: 5.0 us, as the
// kernel without the norm, whose kernel behind it took 5.1.
struct WholeNorm {
    const float* g;
    bf16_t* out;
    long ld;
    float eps;
};
constexpr int WHOLE_NORM_COLUMNS = 4096;
template <int EACH>
__global__ __launch_bounds__(256) void skinny_reduce_norm_kernel(const float* __restrict__ P, float* __restrict__ C, int M, int N, int splits, long ldc, WholeNorm norm) {
    __shared__ float red[4];
    const size_t row = blockIdx.x, slab = (size_t)M * N;
    float4 x[EACH], sum[EACH], g[EACH];
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
        const int c = 4 * (threadIdx.x + 256 * e);
        x[e] = sum[e] = g[e] = float4{0.f, 0.f, 0.f, 0.f};
        if (c < N) {
            x[e] = *reinterpret_cast<const float4*>(C + row * ldc + c);
            g[e] = *reinterpret_cast<const float4*>(norm.g + c);
        }
    }
    for (int sp0 = 0; sp0 < splits; sp0 += 4) {
        float4 part[4][EACH];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < EACH; ++e)
                part[u][e] = *reinterpret_cast<const float4*>(P + (size_t)min(sp0 + u, splits - 1) * slab + row * N + min(4 * (int)(threadIdx.x + 256 * e), N - 4));
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (sp0 + u < splits) {
#pragma unroll
                for (int e = 0; e < EACH; ++e) { sum[e].x += part[u][e].x; sum[e].y += part[u][e].y; sum[e].z += part[u][e].z; sum[e].w += part[u][e].w; }
            }
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
        const int c = 4 * (threadIdx.x + 256 * e);
        if (c < N) {
            x[e].x += sum[e].x; x[e].y += sum[e].y; x[e].z += sum[e].z; x[e].w += sum[e].w;
            *reinterpret_cast<float4*>(C + row * ldc + c) = x[e];
            ss = fmaf(x[e].x, x[e].x, ss); ss = fmaf(x[e].y, x[e].y, ss); ss = fmaf(x[e].z, x[e].z, ss); ss = fmaf(x[e].w, x[e].w, ss);
        }
    }
    ss = block_sum<256>(ss, red);
    const float scale = 1.0f / sqrtf(ss / (float)N + norm.eps);
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
        const int c = 4 * (threadIdx.x + 256 * e);
        if (c < N)
            *reinterpret_cast<uint2*>(norm.out + row * norm.ld + c) =
                uint2{f32x2_to_bf16x2(g[e].x * (scale * x[e].x), g[e].y * (scale * x[e].y)), f32x2_to_bf16x2(g[e].z * (scale * x[e].z), g[e].w * (scale * x[e].w))};
    }
}

// The same for the gated product: columns 32b .. 32b+15 of the partial sums are gates, 32b+16 .. 32b+31 the ups of
// outputs 16b .. 16b+15; the output [M, N/2] is silu(gate) * up in bfloat16.
__global__ void skinny_reduce_gated_kernel(const float* __restrict__ P, bf16_t* __restrict__ C, int M, int N, int splits, long ldc, int epi, float limit) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int half = N / 2;
    if (i >= (size_t)M * half) return;
    const size_t m = i / half;
    const int c = (int)(i % half), col = (c >> 4) * 32 + (c & 15);
    float gate = 0.f, up = 0.f;
    for (int sp = 0; sp < splits; ++sp) {
        gate += P[((size_t)sp * M + m) * N + col];
        up += P[((size_t)sp * M + m) * N + col + 16];
    }
    C[m * ldc + c] = f32_to_bf16(epi == EPI_GATED_CLAMP_BF16 ? clamp_gate(gate, up, limit) : epi == EPI_GATED_GELU_BF16 ? gelu_gate(gate, up) : silu_gate(gate, up));
}

// The same for the q/k/v product of an attention layer, N = (n_heads + 2 n_kv) * hd columns: the sums of a row are its queries,
// keys and values, and instead of writing them out for a kernel that rotates them and puts them into the cache, this one does
// that itself: queries rotated into q_out, keys rotated and values as they are into the page table[slot][pos / page_size] at
// place pos % page_size (pairs (i, i + hd/2): a' = a cos - b sin, b' = a sin + b cos; the page's layout as the attention
// kernels read it: keys [kv_head][place][hd], then values [kv_head][hd][place]).  A thread has four neighbouring columns; the
// other half of its pairs is with the thread hd/8 lanes away, in the same wave (hd a power of two from 8 to 256, and rows of a
// multiple of 256 columns, so that a wave lies in one row and holds whole heads).
__global__ __launch_bounds__(256) void skinny_reduce_rope_store_kernel(const float* __restrict__ P, int M, int N, int splits, NormIn norm_in, RopeStore rs) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4, slab = (size_t)M * N;
    if (i >= slab) return;                                   // (whole waves: 256 divides N, so the exchange below has all its lanes)
    const size_t row = i / N;
    const int col = (int)(i % N);
    const int a_dim = rs.n_heads * rs.hd, kv_dim = rs.n_kv * rs.hd, half = rs.hd / 2;
    const int which = col < a_dim ? 0 : col < a_dim + kv_dim ? 1 : 2;                        // queries, keys, values
    const int c = which == 0 ? col : which == 1 ? col - a_dim : col - a_dim - kv_dim;        // the column among them
    const int h = c / rs.hd, kk = c % rs.hd;
    // Everything is asked for at once, by every lane: position and slot first (the page number, which needs them, then waits for
    // them alone), the row's pieces of the norm, the angles (a lane with values asks too and drops them), the first eight splits.
    const int p = rs.pos[row], slot = rs.slot[row];
    [[maybe_unused]] RowPieces pieces;
    if (norm_in.squares != nullptr) pieces = row_pieces(norm_in, (int)row);
    float4 cc = {1.f, 1.f, 1.f, 1.f}, ss = {0.f, 0.f, 0.f, 0.f};
    if (rs.cos_t != nullptr) {
        cc = *reinterpret_cast<const float4*>(rs.cos_t + row * half + kk % half);
        ss = *reinterpret_cast<const float4*>(rs.sin_t + row * half + kk % half);
    }
    float4 part[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) part[u] = *reinterpret_cast<const float4*>(P + (size_t)min(u, splits - 1) * slab + i);
    const long page = rs.table[(size_t)slot * rs.table_stride + p / rs.page_size];
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (u < splits) {
            s[0] += part[u].x; s[1] += part[u].y; s[2] += part[u].z; s[3] += part[u].w;
        }
    for (int sp0 = 8; sp0 < splits; sp0 += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) part[u] = *reinterpret_cast<const float4*>(P + (size_t)min(sp0 + u, splits - 1) * slab + i);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (sp0 + u < splits) {
                s[0] += part[u].x; s[1] += part[u].y; s[2] += part[u].z; s[3] += part[u].w;
            }
    }
    if (norm_in.squares != nullptr) {
        const float scale = row_scale_from(norm_in, (int)row, pieces);
#pragma unroll
        for (int v = 0; v < 4; ++v) s[v] *= scale;
    }
    float out[4] = {s[0], s[1], s[2], s[3]};
    if (rs.cos_t != nullptr) {                               // (every lane takes part in the exchange, whatever it holds)
        float other[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) other[v] = __shfl_xor(s[v], half / 4, 64);
        if (which != 2) {
            const float cs[4] = {cc.x, cc.y, cc.z, cc.w}, sn[4] = {ss.x, ss.y, ss.z, ss.w};
#pragma unroll
            for (int v = 0; v < 4; ++v) out[v] = kk < half ? s[v] * cs[v] - other[v] * sn[v] : other[v] * sn[v] + s[v] * cs[v];
        }
    }
    uint2 packed;
    packed.x = (unsigned)f32_to_bf16(out[0]) | ((unsigned)f32_to_bf16(out[1]) << 16);
    packed.y = (unsigned)f32_to_bf16(out[2]) | ((unsigned)f32_to_bf16(out[3]) << 16);
    if (which == 0) {
        *reinterpret_cast<uint2*>(rs.q_out + row * a_dim + c) = packed;
        return;
    }
    const int place = p % rs.page_size;
    bf16_t* keys = rs.cache + page * rs.page_stride;
    bf16_t* values = keys + (size_t)rs.n_kv * rs.page_size * rs.hd;
    if (which == 1) {
        *reinterpret_cast<uint2*>(keys + ((size_t)h * rs.page_size + place) * rs.hd + kk) = packed;
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) values[((size_t)h * rs.hd + kk + v) * rs.page_size + place] = f32_to_bf16(out[v]);
    }
}

// ------------------------------------------------------------------------------------------- slim
// At most 16 rows of A.  A workgroup of 8 waves owns `rows` weight rows in GROUPS groups of 8 (the last may be partly full); k goes in steps of 64, and wave w takes the steps w, w + 8, ...,
// counted from a place of the workgroup's own.  Both operands go from global memory straight into registers (the activations are few and stay in cache):
// lane l holds row l % 8 of a group, and of a step's 64 k the 8 from 8 (l / 16) + 32 (l / 8 % 2) on, for weights and activations alike, so the eight
// lanes of a row read 128 contiguous bytes, a cache line, in one load.  To the matrix instruction that is 16 rows by 32 k on either side, rows 8 to 15 being
// the same 8 rows' next 32 k: of the 16 x 16 result the two 8 x 8 blocks on the diagonal are the two halves' sums (the other two mix the halves and are dropped).
// XT groups of 8 rows of A share the weights; GROUPS groups of weights share the activations.
// Loads run DEPTH steps ahead of the products.  The waves' sums meet in LDS and are added in the order of the waves, the lower halves before the upper.
//
// What bounds it is weights on their way from memory, and behind them the activations, of which every workgroup reads all.  67 MB of weights in a bare read take
// 12.8 us, 11.4 past the caches (each line is read once, by one load; with 16 rows' 64 bytes a load, as this kernel read them before, 14.1 and 14.8).  All workgroups
// starting at the same k would ask the same memory channels first (rows lie a multiple of 4 KB apart): 12.6 us, 11.9 from a place of their own.  Microseconds, with half lines and all
// workgroups at the same k and so, in chains of products with weights of their own (400 to 1,050 MB in all; +: made by strips):
//   rows                        1               8               16
//   16,384 x 2,048 gated        15.7, 11.7      16.2, 11.7      16.7+, 13.5
//   28,672 x 4,096 gated        45.7+, 34.6     45.3+, 39.3     46.1+, 40.7+
//   2,048 x 8,192 added         8.7, 7.4        10.7, 9.5       13.2, 13.1
//   2,048 x 2,048 added         3.9, 3.7        4.4, 4.3        5.3, 5.4
//   4,096 x 14,336 added        24.1, 19.0      25.3, 21.9      31.5, 27.7
//   6,144 x 4,096 stored        10.9, 9.4       14.8, 9.7       16.8, 11.6
//   128,256 x 2,048 stored      78.7, 74.3      96.9+, 75.2     99.7+, 89.1
//   4,096 x 768 gated           4.2, 3.5        4.7, 3.6        5.2, 4.0         (200 MB of such weights, which the caches could hold: 3.7, 3.5; 4.2, 3.6; 4.7, 3.9)
//   1,024 x 512 stored          2.4, 2.4        2.6, 2.5        2.8, 2.8         (2.2, 2.4; 2.4, 2.6; 2.6, 2.8)
// HAND: with the two halves of a norm handed from product to product (`NormIn`, `NormOut` above).
// Strides come in pieces of 16 bytes, so that all that the first loads need is in the registers that are filled with the launch.  FAR: rows so far apart that 64 bits are needed to
// reckon with them (`slim_reach`).
template <bool FAR> struct SlimPlaces { typedef int Stride; typedef unsigned At; };
template <> struct SlimPlaces<true> { typedef long Stride; typedef size_t At; };
template <int GROUPS, int EPI, bool HAND, int XT, bool FAR = false>
__global__ __launch_bounds__(512, 4) void gemm_bf16_slim_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, typename SlimPlaces<FAR>::Stride lda8,
                                                                typename SlimPlaces<FAR>::Stride ldw8, int M, int N, int K, int rows, int turn,
                                                                void* __restrict__ C, long ldc, NormIn norm_in, NormOut norm_out) {
    typedef typename SlimPlaces<FAR>::At At;
    constexpr bool GATED = is_gated(EPI);                              // the weights are 16 gates, their 16 ups, and so on
    constexpr int DEPTH = GROUPS == 1 ? 4 : GROUPS == 2 ? 4 : 2;
    static_assert(!GATED || GROUPS == 2 || GROUPS == 4, "as many groups of gates as of ups");
    const int out = GATED ? 4 * GROUPS : rows;                         // columns of the output
    float act_p = 0.f, act_q = 0.f;
    if constexpr (EPI == EPI_XIELU) { act_p = norm_out.g[0]; act_q = norm_out.g[1]; }
    __shared__ float red[8][XT][GROUPS][2][8][8];                      // [wave][rows of A][weights][half of a step][row][weight row]
    __shared__ float row_scale[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 7, k_lane = 8 * (lane >> 4) + 32 * ((lane >> 3) & 1);
    // A row beyond an operand is clamped into it and lands in results that are never written.  In a row's last, ragged step k is clamped too and the activations
    // beyond K become zeros.
    const int base = GATED ? (blockIdx.x / (4 / GROUPS)) * 32 + (blockIdx.x % (4 / GROUPS)) * 8 : blockIdx.x * rows;
    const bf16_t* w_base[GROUPS];
    // Where the lane's rows begin, in pieces of 16 bytes, or in bytes where the registers are scarce (one 32-bit distance from a scalar address; the host sees to it that it holds
    // a row's place and the one in k behind it).
    constexpr int PIECE = GROUPS == 4 ? 1 : 16;
    At w_at[GROUPS], x_at[XT];
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
        w_base[g] = W + 8 * ((size_t)(base + (GATED ? 32 / GROUPS * g : 0)) * ldw8);
        const int row = GATED ? r : min(8 * g + r, min(rows, N - base) - 1);
        w_at[g] = ((At)row * (At)ldw8 + k_lane / 8) * (16 / PIECE);
    }
#pragma unroll
    for (int t = 0; t < XT; ++t) x_at[t] = ((At)min(8 * t + r, M - 1) * (At)lda8 + k_lane / 8) * (16 / PIECE);
    const int k_last = K - 8 - k_lane;                                 // the last 16 bytes of a row, from `w_row` and `x_row`
    const int steps = (K + 63) / 64, first = first_step(turn);
    const int mine = (steps - wave + 7) / 8;                           // of this wave
    auto place = [&](int i) {                                          // k where the wave's step i begins
        const int step = wave + 8 * i + first;
        return 64 * (step < steps ? step : step - steps);
    };
    uint4 w_buf[DEPTH][GROUPS], x_buf[DEPTH][XT];
    auto fetch = [&](int i, uint4 (&w)[GROUPS], uint4 (&x)[XT]) __attribute__((always_inline)) {
        const At at = (At)((min(place(i), k_last) >> 3) * (16 / PIECE));         // (below 0 for a lane beyond a K under 64: the sums with it are not)
        auto whereof = [](const bf16_t* p, At pieces) { return (const bf16_t*)((const char*)p + (PIECE == 1 ? (size_t)pieces : (size_t)pieces * PIECE)); };
#pragma unroll
        for (int t = 0; t < XT; ++t) x[t] = load16(whereof(A, x_at[t] + at));
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) w[g] = load16_once(whereof(w_base[g], w_at[g] + at));
    };
    floatx4 acc[XT][GROUPS];
#pragma unroll
    for (int t = 0; t < XT; ++t)
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) acc[t][g] = floatx4{};
    auto products = [&](int i, const uint4 (&w)[GROUPS], uint4 (&x)[XT]) __attribute__((always_inline)) {
        const int at = place(i);
        if (at + 64 > K) {                                             // the row's end lies in this step
#pragma unroll
            for (int t = 0; t < XT; ++t)
                if (at + k_lane >= K) x[t] = uint4{0, 0, 0, 0};
        }
#pragma unroll
        for (int t = 0; t < XT; ++t)
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) acc[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x[t]), as_bf16x8(w[g]), acc[t][g], 0, 0, 0);
    };
    // The thread's element of the output: row `m`, the workgroup's column `c`.  What the epilogue adds onto (the 32-bit rows, and the next norm's gain for
    // the column) is asked for before anything else: it comes from the memory-side cache while the weights stream, not behind them as one more round trip.
    constexpr int SHARE = GATED ? 4 * GROUPS : GROUPS == 3 ? 32 : 8 * GROUPS;       // threads to a row
    const int m = tid / SHARE, c = tid % SHARE;
    const int col = blockIdx.x * out + c;
    [[maybe_unused]] float old_value = 0.f, gain = 0.f;
    if constexpr (EPI == EPI_ADD_F32) {
        old_value = ((const float*)C)[(size_t)min(m, M - 1) * ldc + min(col, N - 1)];
        if constexpr (HAND) {
            if (norm_out.scaled != nullptr) gain = norm_out.g[min(col, N - 1)];
        }
    }
    // The pieces of the rows' sums of squares, 32 or 64 threads a row: asked for ahead of the first weights (loads come back in
    // the order they were issued) and added up behind the requests for those, so that one register waits for the epilogue, not eight.
    float piece[HAND ? SLIM_PIECES : 1];
    [[maybe_unused]] float pieces_sum = 0.f;
    const int sharing = M <= 8 ? 64 : 32, piece_row = M <= 8 ? tid >> 6 : tid >> 5;
    auto ask_pieces = [&]() __attribute__((always_inline)) {
        if constexpr (HAND) {
            if (norm_in.squares != nullptr) {
                const float* row_pieces = norm_in.squares + (size_t)min(piece_row, M - 1) * norm_in.parts;
#pragma unroll
                for (int i = 0; i < SLIM_PIECES; ++i) piece[i] = row_pieces[min((tid & (sharing - 1)) + sharing * i, norm_in.parts - 1)];
            }
        }
    };
    auto add_pieces = [&]() __attribute__((always_inline)) {
        if constexpr (HAND) {
            if (norm_in.squares != nullptr) {
#pragma unroll
                for (int i = 0; i < SLIM_PIECES; ++i)
                    if (piece_row < M && (tid & (sharing - 1)) + sharing * i < norm_in.parts) pieces_sum += piece[i];
            }
        }
    };
    ask_pieces();
    if (__builtin_expect(mine >= DEPTH, 1)) {                          // (the usual way lies straight ahead for the instruction fetch)
        // Every load of a trip is issued and nothing is skipped: the compiler counts the loads in flight, and a step's products wait for that step alone.
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) fetch(d, w_buf[d], x_buf[d]);
        add_pieces();
        int i = 0;
        for (; i + 2 * DEPTH <= mine; i += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                products(i + d, w_buf[d], x_buf[d]);
                fetch(i + DEPTH + d, w_buf[d], x_buf[d]);
            }
        }
        const int rest = mine - i - DEPTH;                             // steps not asked for yet, fewer than DEPTH
        if (__builtin_expect(rest > 0, 0)) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                products(i + d, w_buf[d], x_buf[d]);
                if (d < rest) fetch(i + DEPTH + d, w_buf[d], x_buf[d]);
            }
#pragma unroll
            for (int d = 0; d < DEPTH - 1; ++d)
                if (d < rest) products(i + DEPTH + d, w_buf[d], x_buf[d]);
        } else {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) products(i + d, w_buf[d], x_buf[d]);
        }
    } else {
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d)
            if (d < mine) fetch(d, w_buf[d], x_buf[d]);
        add_pieces();
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d)
            if (d < mine) products(d, w_buf[d], x_buf[d]);
    }
    // Element v of a lane's result: row 4 (lane / 16) + v, weight row lane % 16, each modulo 8; on the diagonal where both are below 8 or both are not.
    if ((lane < 32) == ((lane & 8) == 0)) {
#pragma unroll
        for (int t = 0; t < XT; ++t)
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[wave][t][g][lane >> 5][4 * ((lane >> 4) & 1) + v][r] = acc[t][g][v];
    }
    if constexpr (HAND) {
        if (norm_in.squares != nullptr) {
            float sum = pieces_sum;
            if (sharing == 64) sum += __shfl_xor(sum, 32, 64);
#pragma unroll
            for (int off = 16; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
            if ((tid & (sharing - 1)) == 0 && piece_row < 16) row_scale[piece_row] = 1.0f / sqrtf(sum / (float)norm_in.dim + norm_in.eps);
        }
    }
    __syncthreads();
    auto sum_of = [&](int column) {
        float sum = 0.f;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int w = 0; w < 8; ++w) sum += red[w][XT == 1 ? 0 : m >> 3][column >> 3][half][m & 7][column & 7];
        return sum;
    };
    if (tid < 8 * XT * SHARE) {
        float scale = 1.0f;
        if constexpr (HAND) scale = norm_in.squares != nullptr ? row_scale[m] : 1.0f;
        float square = 0.f;
        if (m < M && c < out) {
            if constexpr (GATED) {
                float gate = sum_of(c), up = sum_of(4 * GROUPS + c);
                if constexpr (HAND) { gate *= scale; up *= scale; }
                ((bf16_t*)C)[(size_t)m * ldc + col] = f32_to_bf16(gate_of<EPI>(gate, up, norm_in.limit));
            } else if (col < N) {
                float sum = sum_of(c);
                if constexpr (HAND) sum *= scale;
                if constexpr (EPI == EPI_ADD_F32) {
                    const float x = old_value + sum;
                    ((float*)C)[(size_t)m * ldc + col] = x;
                    if constexpr (HAND) {
                        if (norm_out.scaled != nullptr) {
                            norm_out.scaled[(size_t)m * norm_out.ld + col] = f32_to_bf16(gain * x);
                            square = x * x;
                        }
                    }
                } else if constexpr (EPI == EPI_XIELU) {
                    if (col < norm_in.first) ((float*)C)[(size_t)m * ldc + col] = sum;
                    else norm_out.scaled[(size_t)m * norm_out.ld + col - norm_in.first] = f32_to_bf16(xielu(sum, softplus_f32(act_p), 0.5f + softplus_f32(act_q)));
                } else {
                    write_out<EPI>(C, (size_t)m * ldc + col, sum);
                }
            }
        }
        if constexpr (HAND && EPI == EPI_ADD_F32) {
            if (norm_out.scaled != nullptr) {                   // the threads of a row: its columns of this workgroup
#pragma unroll
                for (int off = SHARE / 2; off > 0; off >>= 1) square += __shfl_xor(square, off, 64);
                if (c == 0 && m < M) norm_out.squares[(size_t)m * gridDim.x + blockIdx.x] = square;
            }
        }
    }
}

// The same for a few more rows of A (MT tiles of 16) and outputs too narrow to fill the chip with strips of 64 weight rows: a workgroup owns 16
// weight rows and all of k, its 8 waves take interleaved 128-wide blocks of k, and each wave multiplies its weights with MT tiles
// of 16 activation rows, all straight from global memory into registers (the waves share nothing: every wave reads another part
// of k; the activations come from L2, as many bytes again for every 16 rows as the strip has weights, which pays up to 32 rows).
// One launch does the product and its epilogue; the alternative, k shared out over workgroups with partial sums in memory and a
// second kernel to add them, costs that kernel's launch and as many bytes of partial sums as the output projection has weights.
template <int MT, int EPI>
__global__ __launch_bounds__(512, 4) void gemm_bf16_slim_tiles_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ C,
                                                                  int M, int N, int K, long lda, long ldw, long ldc, NormIn norm_in, NormOut norm_out,
                                                                  int strip_rows) {
    constexpr int SLICES = 8, STEP = SLICES * SK, DEPTH = 2;
    __shared__ float red[SLICES][MT][64][4];
    __shared__ float row_scale[MT * 16 < 32 ? 32 : MT * 16];
    static_assert(MT == 2, "the epilogue's sums of squares take every thread's one result to lie in one row of 16 threads");
    const int tid = threadIdx.x, lane = tid & 63, slice = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    // strip_rows (8, 12 or 16) of the product's 16 weight rows are the workgroup's own; lanes beyond them ask for its last row again
    // (the same cache line) and their results are dropped
    const int n = blockIdx.x * strip_rows + min(r, strip_rows - 1);
    const bf16_t* wrow = W + (size_t)min(n, N - 1) * ldw + 8 * q;         // (every lane issues every load of a block, as in the kernel above)
    const bf16_t* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xrow[t] = A + (size_t)min(t * 16 + r, M - 1) * lda + 8 * q;
    const int k_last = K - 8 - 8 * q;
    floatx4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = floatx4{};
    uint4 w_buf[DEPTH][4], x_buf[DEPTH][MT][4];
    auto fetch = [&](int k0, uint4* w, uint4 (*x)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int at = min(k0 + 32 * j, k_last);
            w[j] = load16(wrow + at);
#pragma unroll
            for (int t = 0; t < MT; ++t) x[t][j] = load16(xrow[t] + at);
        }
    };
    // (what the epilogue adds onto is asked for first, as in the kernel above: every thread has one result, e = tid below)
    [[maybe_unused]] float old_value = 0.f, gain = 0.f;
    if constexpr (EPI == EPI_ADD_F32) {
        const int e_row = 16 * (tid >> 8) + ((tid >> 4) & 15), e_col = blockIdx.x * strip_rows + (tid & 15);
        old_value = ((const float*)C)[(size_t)min(e_row, M - 1) * ldc + min(e_col, N - 1)];
        if (norm_out.scaled != nullptr) gain = norm_out.g[min(e_col, N - 1)];
    }
    const int k_first = slice * SK;
    const int n_blocks = k_first < K ? (K - k_first + STEP - 1) / STEP : 0;       // of this wave
    if (n_blocks > 0) fetch(k_first, w_buf[0], x_buf[0]);
    if (norm_in.squares != nullptr) row_scales_into(row_scale, norm_in, M);      // (the barrier behind the products lies before its use)
    auto products = [&](int b, uint4* w, uint4 (*x)[4]) __attribute__((always_inline)) {
        const int kb = k_first + b * STEP;
        if (kb + SK > K) {                                    // the row's end lies in this block: weights of k beyond it become zeros
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (kb + 32 * j + 8 * q >= K) w[j] = uint4{0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x[t][j]), as_bf16x8(w[j]), acc[t], 0, 0, 0);
    };
    int b = 0;
    for (; b + 2 * DEPTH - 1 <= n_blocks; b += DEPTH) {      // trips in which nothing is skipped
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            fetch(k_first + (b + d + 1) * STEP, w_buf[(d + 1) % DEPTH], x_buf[(d + 1) % DEPTH]);
            products(b + d, w_buf[d], x_buf[d]);
        }
    }
    for (; b < n_blocks; b += DEPTH) {                        // the end of the wave's blocks
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            if (b + d + 1 < n_blocks) fetch(k_first + (b + d + 1) * STEP, w_buf[(d + 1) % DEPTH], x_buf[(d + 1) % DEPTH]);
            if (b + d < n_blocks) products(b + d, w_buf[d], x_buf[d]);
        }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[slice][t][lane][v] = acc[t][v];
    __syncthreads();
    // Element v of a lane's result for tile t: activation row 16*t + 4*q + v, weight row r of the strip.
    for (int e = tid; e < MT * 256; e += 512) {
        const int t = e >> 8, m = (e >> 4) & 15, c = e & 15;
        const int src_lane = c + 16 * (m >> 2), v = m & 3, row = 16 * t + m, col = c < strip_rows ? blockIdx.x * strip_rows + c : N;
        float sum = 0.f;
#pragma unroll
        for (int s = 0; s < SLICES; ++s) sum += red[s][t][src_lane][v];
        if (norm_in.squares != nullptr && row < M) sum *= row_scale[row];
        if constexpr (EPI == EPI_ADD_F32) {
            if (norm_out.scaled != nullptr) {                   // (every thread comes here once: MT * 256 results, 512 threads)
                float square = 0.f;
                if (row < M && col < N) {
                    const float x = old_value + sum;
                    ((float*)C)[(size_t)row * ldc + col] = x;
                    norm_out.scaled[(size_t)row * norm_out.ld + col] = f32_to_bf16(gain * x);
                    square = x * x;
                }
#pragma unroll
                for (int off = 8; off > 0; off >>= 1) square += __shfl_xor(square, off, 64);
                if (c == 0 && row < M) norm_out.squares[(size_t)row * gridDim.x + blockIdx.x] = square;
                continue;
            }
            if (row < M && col < N) ((float*)C)[(size_t)row * ldc + col] = old_value + sum;
            continue;
        }
        if (row < M && col < N) write_out<EPI>(C, (size_t)row * ldc + col, sum);
    }
}

int epilogue_of(int c_dtype, int accumulate) {
    if (c_dtype == GI_F32) return accumulate ? EPI_ADD_F32 : EPI_STORE_F32;
    if (c_dtype == GI_BF16 && !accumulate) return EPI_STORE_BF16;
    return -1;
}

}  // namespace

// Number of k-splits of the skinny kernel for a product with 17..128 rows (what scratch a product wants, strips' shares among it, gi_gemm_bf16_scratch_floats says);
// 0: the output is wide enough to fill the chip without a split, no scratch is needed.  Workgroups for three quarters of the chip or more, each with at least one block of k (measured at 33 to
// 64 rows, product and reduce kernel together: 192 to 384 workgroups on 256 compute units, with two blocks of k each, take 11 us for N = 3072, K = 2048 and
// 16 us for N = 2048, K = 8192; twice the workgroups with one block each 12.5 and 17.5 us, half of them 13 and 22 us).
GI_API int gi_gemm_bf16_skinny_splits(int N, int K) {
    const int strips = (N + 63) / 64, most_of_the_chip = gi_compute_units() * 3 / 4;
    if (strips >= most_of_the_chip) return 0;
    int splits = 1;
    while (strips * splits < most_of_the_chip && K / (splits * 2) >= KB) splits *= 2;
    return splits;
}

// Splits of k for the LDS-ring kernel (more than 64 rows): with fewer tiles of 128 x 128 than three quarters of the compute units the tiles alone
// leave compute units idle and the weights stream too slowly; every share keeps at least 256 of k.
GI_API int gi_gemm_bf16_piped_splits(int M, int N, int K) {
    if (M <= SKINNY_MAX_ROWS || K % PK != 0 || N < 128) return 1;
    const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
    const int most_of_the_chip = gi_compute_units() * 3 / 4;
    int splits = 1;
    while (tiles * splits < most_of_the_chip && K % (splits * 2 * PK) == 0 && K / (splits * 2) >= 256) splits *= 2;
    return splits;
}

// The most pieces a reader of M rows takes: what a writer of as many rows makes.
static int consumer_max_parts(int M) { return M <= 16 ? slim_max_parts(M) : M <= 32 ? TILES_MAX_PARTS : REDUCE_MAX_PARTS; }

// Whether a product of more than 128 rows is one of a long prompt or a wide output: 256 x 256 results for three quarters of the compute units or
// more.  Such a gated product finishes a norm handed on; such a product onto the residual hands none on, and such a q/k/v product takes
// none: the norm's own kernel runs there.
static bool many_tiles(int M, int N) { return (long)((M + 255) / 256) * ((N + 255) / 256) >= gi_compute_units() * 3 / 4; }

// Which kernel takes a product of more than 128 rows that does not share k out: what counts are the rounds of tiles on the compute units,
// each with what a tile takes to begin and to end.  Microseconds, fitted to measurements at K = 128 to 8,192 (2,048 rows of 3,072 x 2,048 added onto
// what is there: 51.5 with 128 x 128 tiles in two rounds, 35.0 with 256 x 128 in one; 300 rows of 16,384 x 2,048 gated 42 and 39; 3,000 rows of
// 3,072 x 2,048 88 and 66; 2,048 rows of 16,384 x 2,048 gated 152 with 256 x 128 in four rounds, 120 with 256 x 256 in two).  A tile of 128 x 128 ends
// soonest where its sums leave as they are or through LDS (stored, rotated, added with a norm handed on) and latest where they are added one by
// one: at short k several rounds of those are the faster ones (2,600 rows of 4,096 x 512 stored: 21 us in three, 25.5 with 256 x 128 in two; of
// 4,096 x 1,536 the same either way; 2,048 rows of 5,120 x 1,024 rotated 36 and 42).  Only the two larger tiles finish a
// norm handed on to a gated product; the q/k/v product takes one handed on in tiles of 128 columns alone.
enum Large { PIPED_128, TALL_256, PINGPONG_256 };

// How the tall kernel's tiles are made (`TileShares`): a last round of at most half as many tiles as there are compute units in shares of k, where
// that is the faster way.  `us`: what all of it takes.  A block of k takes longer with the whole chip at work on different parts of k (0.85 us), a tile ends
// some 5 us later for the exchange, and 2 for every share.  Alone, 2,048 rows of 2,048 x 8,192 take 76 us in two shares (95 as 128 x 128 tiles, one a unit),
// of 2,048 x 4,096 47 (58), of 2,048 x 2,048 33 (31: not taken); 3,000 rows of 3,072 x 8,192, one round and 32 tiles, 163 in four shares and 180 in two
// (203 in two rounds), of 3,072 x 3,072 83 (96); 2,048 rows of 5,120 x 3,072 76 in four (78).  Fewer than 8 blocks a share are not worth the exchange.
// Of 874 products that were shared out where these times alone spoke for it, 35 were slower than before by up to a quarter; the lines here and in `large_kernel` leave those
// out.  Beside whole tiles the times have to promise 7.5 %: 1,161 rows of 8,192 x 2,048, promised 7 %, took 69 us for 62.
// clears: no counters are given, and the launch that clears them takes 4 us (2 to 5).
constexpr double CLEAR_US = 4;
struct TallCut { int whole, rest, shares; double us; };
static TallCut tall_cut(int M, int N, int K, bool may_share, bool clears) {
    const int units = gi_compute_units(), tiles = ((M + 255) / 256) * ((N + 127) / 128), rest = tiles % units;
    const double blocks = K / PK, each = blocks * 0.715 + 13;
    TallCut cut = {tiles, 0, 1, (tiles + units - 1) / units * each};
    if (!may_share || rest == 0 || 2 * rest > units) return cut;
    const double before = tiles / units * each, whole = cut.us;
    for (int shares = 2; shares * rest <= units && shares <= TALL_MAX_SHARES && blocks >= 8 * shares; ++shares) {
        const double us = before + ((int)blocks + shares - 1) / shares * 0.85 + 16 + 2 * shares;
        if (us < 0.925 * whole && us + (clears ? CLEAR_US : 0) < 0.95 * whole && us < cut.us) cut = {tiles - rest, rest, shares, us};
    }
    return cut;
}
// Floats of scratch for it: the counters, then the sums.
static long tall_counter_floats(const TallCut& cut) { return (4L * cut.rest + 63) / 64 * 64; }
static long tall_scratch_floats(const TallCut& cut) { return cut.shares > 1 ? tall_counter_floats(cut) + (long)cut.rest * cut.shares * 256 * 128 : 0; }

// (the ping-pong kernel's rotated ends; 8 us a round leave out what is no faster.  33 products, 2,048 to 8,192 rows, in tiles of 256 x 128 or 128 x 128 and of 256 x 256: 4,096 rows of 3,072 x 2,048
// 64.6 us and 52.9, 3,072 of 5,120 x 3,072 97.8 and 83.8, 8,192 of 6,144 x 4,096 368.9 and 317.6; of the 14 that it takes none gains less than 14 %)
constexpr double ROPE_US = 8;
struct LargeChoice { Large kernel; TallCut cut; };              // cut: how the tall kernel makes its tiles, where that is the one
static LargeChoice large_kernel(int M, int N, int K, int epi, bool rope, bool hands_norm, bool scaled_rows, bool may_share, bool clears) {
    const long units = gi_compute_units(), m128 = (M + 127) / 128, m256 = (M + 255) / 256, n128 = (N + 127) / 128, n256 = (N + 255) / 256;
    const auto rounds = [&](long tiles) { return (double)((tiles + units - 1) / units); };
    const bool many = many_tiles(M, N), gated = !rope && is_gated(epi);
    // what a round of 128 x 128 tiles takes to end, and what of the last round's others need not wait for
    struct { double each, less; } ends = {10, 0};                                            // added one by one (and stores with many tiles)
    if (gated) ends = {6, 0};
    else if (rope) ends = {7.4, 5};
    else if (hands_norm || (!many && epi == EPI_STORE_BF16)) ends = {8, 4};
    else if (!many && epi == EPI_STORE_F32) ends = {9, 8.4};
    const double blocks = K / PK, small = rounds(m128 * n128);
    // (one: measured 31 us at 32 blocks, 50 to 58 at 64, 95 at 128)
    double piped = small > 1 ? small * (blocks * 0.45 + ends.each) * (small > 2 ? 1.15 : 1) - ends.less : blocks * 0.65 + 10.5;      // (several: two workgroups a unit)
    if (scaled_rows && !rope) piped = 1e30;
    const TallCut whole = tall_cut(M, N, K, false, false), cut = tall_cut(M, N, K, may_share, clears);
    const double pingpong = many && !(rope && scaled_rows) ? rounds(m256 * n256) * (blocks * 1.45 + 14 + (rope ? ROPE_US : 0)) : 1e30;
    // (gating 256 x 128 sums at a time costs the tall kernel 3 us a round more: 1,500 rows by 16,384 of 2,048, three rounds of it against one and a
    // half of the ping-pong kernel: 114 us against 103.  Shares do not take its products: with 160 to 192 tiles a block takes it 1.3 us, and 4,096 rows of
    // 3,072 x 8,192 added took 182 with it and 198 shared, 1,368 of 8,192 x 6,784 stored 149 and 160)
    if (pingpong < piped && 0.95 * pingpong <= whole.us + (gated ? 3 * rounds(m256 * n128) : 0)) return {PINGPONG_256, whole};
    if (whole.us < piped) return {TALL_256, cut};
    if (cut.shares > 1) {
        if (small > 1) return cut.us + (clears ? CLEAR_US : 0) < piped ? LargeChoice{TALL_256, cut} : LargeChoice{PIPED_128, whole};
        // Both in one round that may leave units idle, which the times above do not know: fitted to 534 products of 128 to 1,024 rows and of more by few columns, whose
        // 128 x 128 tiles take so long within 5 % and whose shares within 7.  3 us ahead they are never the slower ones (273 rows of 8,192 x 3,072 handing a norm on: 34 us
        // as 128 x 128 tiles, 42 in shares, 31 expected), and what is left out by that gains 2 %.
        const bool through_lds = rope || hands_norm, added = !rope && epi == EPI_ADD_F32;
        const double fill = (double)(m128 * n128) / units, shared_fill = (double)(cut.rest * cut.shares) / units;
        const double one_round = 4.7 + blocks * (0.41 + 0.207 * fill) + (through_lds ? 1.4 : added ? 7.4 : 0);
        const double shared = 6 + ((int)blocks + cut.shares - 1) / cut.shares * (0.45 + 0.476 * shared_fill) + 1.77 * cut.shares + (through_lds ? 2.9 : added ? 3.3 : gated ? 1.9 : 0);
        if (shared + (clears ? CLEAR_US : 0) + 3 < one_round) return {TALL_256, cut};
    }
    return {PIPED_128, whole};
}
// Kinds as for gi_gemm_bf16_large_kernel.
static LargeChoice large_kernel_of_kind(int M, int N, int K, int kind, bool counters) {
    const int epi = kind == 0 ? EPI_STORE_F32 : kind <= 2 ? EPI_ADD_F32 : kind == 6 ? EPI_XIELU : kind == 7 ? EPI_STORE_BF16 : EPI_GATED_BF16;
    return large_kernel(M, N, K, epi, kind == 5, kind == 2, kind == 4, kind != 6, !counters);
}
static bool takes_large(int M, int N, int K) { return M > SKINNY_MAX_ROWS && K % PK == 0 && N >= 128; }

// Products whose k is shared out, in strips: tiles of rows (one to some, of equal height), shares of k, and about how long it takes with the kernel that adds up.  The times are fitted
// to 4,600 products (24 numbers of rows from 17 to 1,400, 12 sizes of weights, every cut), which they meet within 6 %; the cut they choose is 0.7 % slower than the best one on average, 11 % at worst.
// What the fit misses at other sizes (few columns, long shares) find_shared_strips allows for.  128 rows of 2,048 x 2,048 take 12.2 us as one tile in four shares, 10.2 as two in three; 301 of 2,048 x 8,192 27 as two in four, 32 as three in two.
struct StripCut { int tiles, splits; double us; };
static StripCut strip_cut(int M, int N, int K) {
    const int strips = (N + 63) / 64, units = gi_compute_units(), all = K / PK;
    StripCut best = {0, 0, 0};
    double least = 0;
    for (int tiles = (M + 255) / 256; tiles <= (M + 63) / 64; ++tiles) {
        const int rows = (M + tiles - 1) / tiles, height = (rows + 31) / 32, together = height <= 3 ? 2 : 1;       // (workgroups that a unit's LDS holds)
        for (int want = 1; want <= 16 && (want == 1 || all / want >= 3); ++want) {
            const int blocks = (all + want - 1) / want, splits = (all + blocks - 1) / blocks;
            if (splits != want) continue;
            const long groups = (long)strips * tiles * splits;
            if (best.tiles && (groups > 2 * units || (groups > units && rows > 64 && (tiles > 1 || rows > 96)))) break;
            const long a_unit = (groups + units - 1) / units;
            const double one = blocks * (0.121 + 0.00116 * rows + 0.0283 * height) + 0.39, sums = 1.85e-6 * splits * M * N;
            const double busy = 5.2 + (a_unit / together * (together == 2 ? 1.38 : 1) + a_unit % together) * one + sums;
            const double memory = 5.2 + 0.27e-6 * N * K + sums + 4.5e-6 * (rows + 64) * groups * blocks;
            const double both = busy * busy * busy * busy + memory * memory * memory * memory;
            if (best.tiles == 0 || both < least) { least = both; best = {tiles, splits, 0}; }
        }
    }
    best.us = sqrt(sqrt(least));
    return best;
}
// Whether a product ends in strips, with all of k in a workgroup.  Above 128 rows the tiles of 128 or 256 x 128 are the better ones for gated products whose strips do not fit one
// round (160 rows of 28,672 x 4,096: 75 us and 82), for k above 4,096, where what a strip takes in of A tells (160 rows of 12,288 x 4,096 42.0 us and 39.2, x 6,144 60.1 and 61.3, x 14,336 112 and 128), and from 169 rows on
// for k above 2,048 where the strips leave a tenth of the units idle (184 rows of 12,288 x 3,072 33.1 and 34.4, of 16,384 x 3,072 40.5 and 37.2).
// Below 1,024 of k strips would be faster too (131 rows of 16,384 x 512 12.8 us and 10.7), but there a gated product's sums are in bits those of the larger tiles that more rows take, and stay so.
// A few rows with k of two blocks of the skinny kernel, or nearly, stay with that: it asks for all its weights at once (16 rows of 16,384 x 512 stored 5.8 us and 6.4 in strips, of
// 16,384 x 768 9.1 and 7.6; from 20 rows and beyond two rounds of strips they are level).
static bool ends_in_strips(int M, int N, int K) {
    const int strips = (N + 63) / 64, units = gi_compute_units();
    if (K % PK != 0 || (M < 20 && K > 384 && K <= 512 && strips <= 2 * units)) return false;
    return M <= SKINNY_MAX_ROWS || (M <= 192 && K >= 1024 && K <= 4096 && strips <= units && (M <= 168 || K <= 2048 || strips * 10 >= units * 9));
}
// How strips make a product whose k is shared out, which the kernels beside them cut into `splits`; no tiles where they do not: from 129 rows on where the tiles of 128 x 128 promise to
// be as fast (a fit like the one above; 350 rows of 3,072 x 8,192 43.1 us and 44.5, 600 71 and 58).  Strips have to promise more where the fit knows less of what they take in (1,900 products
// of 14 sizes of columns, 128 to 11,264, and nine of k, 512 to 28,672: with these lines none of more than 128 rows is over 5 % slower than the tiles, without them 40 are, up to 27 %):
//   many workgroups with long shares (300 rows of 6,144 x 14,336 116 us in tiles and 125 in strips), one tile of more than 192 rows (256 of 11,264 x 768 23.6 and 25.2), and
//   few columns, whose strips read more of A than of the weights (900 rows of 500 x 8,192 22.8 and 26.4, 1,400 of 320 x 28,672 66 and 81; 400 of 500 x 4,096 15.2 and 12.4).
constexpr int STRIP_MAX_ROWS = 1536;
static StripCut find_shared_strips(int M, int N, int K, int splits) {
    const StripCut none = {0, 0, 0};
    if (K % PK != 0 || M > STRIP_MAX_ROWS || splits == 0) return none;
    const int strips = (N + 63) / 64;
    if (N < 768 && M > 256 && (double)M * K * strips > 24e6) return none;
    const StripCut cut = strip_cut(M, N, K);
    if (M <= SKINNY_MAX_ROWS) return cut;
    const bool two = (long)((M + 127) / 128) * ((N + 127) / 128) * splits > gi_compute_units();
    const int groups = strips * cut.tiles * cut.splits, blocks = (K / PK + cut.splits - 1) / cut.splits;
    const double least = groups > gi_compute_units() && blocks > 64 ? 0.88 : cut.tiles * cut.splits == 1 && M > 192 ? 0.9 : 0.98;
    return cut.us < least * (6.6 + K / splits / PK * (two ? 0.951 : 0.882) + 1.55e-6 * splits * M * N) ? cut : none;
}
// Found once for the sizes that a thread asks for again and again (a step's layers have the same few): looking at up to 140 cuts takes 0.3 to 2 us of the host's time, for every product of a pass
// that is not captured.
static StripCut shared_strips(int M, int N, int K, int splits) {
    struct Found { int M, N, K, splits; StripCut cut; };
    static thread_local Found found[32] = {};
    Found& at = found[(unsigned)(M + 5 * (N / 64) + 11 * (K / 64)) % 32];
    if (at.M != M || at.N != N || at.K != K || at.splits != splits) at = {M, N, K, splits, find_shared_strips(M, N, K, splits)};
    return at.cut;
}
static bool strip_strides(long lda, long ldw) { return lda < (1L << 22) && ldw < (1L << 22); }       // (a tile's rows within 32-bit offsets)
// The most shares of k that a product may be cut into.
static int shared_out(int M, int N, int K, int splits) {
    const int strips = shared_strips(M, N, K, splits).splits;
    return strips > splits ? strips : splits;
}

// By how many workgroups each tile of the last round of a product is made that has all the scratch it asks for (1: one), with or without counters.
GI_API int gi_gemm_bf16_shares(int M, int N, int K, int kind, int counters) {
    if (!takes_large(M, N, K) || gi_gemm_bf16_piped_splits(M, N, K) > 1 || (kind == 3 && ends_in_strips(M, N, K))) return 1;
    const LargeChoice choice = large_kernel_of_kind(M, N, K, kind, counters != 0);
    return choice.kernel == TALL_256 ? choice.cut.shares : 1;
}

// Floats of scratch a product of these sizes and kind asks for (partial sums where k is shared out), 0 if none.  It does without where gi_gemm_bf16_shares says
// more than one: the kernels that share nothing out serve then.
GI_API long gi_gemm_bf16_scratch_floats(int M, int N, int K, int kind, int counters) {
    if (M <= SKINNY_MAX_ROWS) return (long)shared_out(M, N, K, gi_gemm_bf16_skinny_splits(N, K)) * M * N;
    const int splits = gi_gemm_bf16_piped_splits(M, N, K);
    if (splits > 1) return (long)shared_out(M, N, K, splits) * M * N;
    return gi_gemm_bf16_shares(M, N, K, kind, counters) > 1 ? tall_scratch_floats(large_kernel_of_kind(M, N, K, kind, counters != 0).cut) : 0;
}

// The least that such a product does with: with less than the above the kernels beside strips make it, and beside shared tiles (0: they need none).
GI_API long gi_gemm_bf16_least_scratch_floats(int M, int N, int K) {
    if (M <= SKINNY_MAX_ROWS) return (long)gi_gemm_bf16_skinny_splits(N, K) * M * N;
    const int splits = gi_gemm_bf16_piped_splits(M, N, K);
    return splits > 1 ? (long)splits * M * N : 0;
}

static const NormIn NO_NORM_IN = {nullptr, 0, 0.f, 1, 0.f};
static const NormOut NO_NORM_OUT = {nullptr, nullptr, 0, nullptr};

static int reduce_partials(const float* scratch, void* C, int epi, int M, int N, int splits, long ldc, hipStream_t stream, NormIn norm_in = NO_NORM_IN,
                           NormOut norm_out = NO_NORM_OUT, const WholeNorm* whole = nullptr) {
    if (whole != nullptr) {
#define WHOLE(EACH_) skinny_reduce_norm_kernel<EACH_><<<M, 256, 0, stream>>>(scratch, (float*)C, M, N, splits, ldc, *whole)
        if (N <= 1024) WHOLE(1); else if (N <= 2048) WHOLE(2); else if (N <= 3072) WHOLE(3); else WHOLE(4);
#undef WHOLE
    } else if (is_gated(epi)) {
        GI_REQUIRE(norm_in.squares == nullptr, "gemm_bf16: a gated product whose k is shared out cannot finish a norm handed on");
        skinny_reduce_gated_kernel<<<(unsigned)(((size_t)M * (N / 2) + 255) / 256), 256, 0, stream>>>(scratch, (bf16_t*)C, M, N, splits, ldc, epi, norm_in.limit);
    } else {
#define REDUCE(VEC_)                                                                                                                    \
    do {                                                                                                                                \
        const unsigned blocks = (unsigned)(((size_t)M * N / VEC_ + 255) / 256);                                                         \
        if (epi == EPI_STORE_F32) skinny_reduce_kernel<EPI_STORE_F32, VEC_><<<blocks, 256, 0, stream>>>(scratch, C, M, N, splits, ldc, norm_in, norm_out);  \
        else if (epi == EPI_ADD_F32) skinny_reduce_kernel<EPI_ADD_F32, VEC_><<<blocks, 256, 0, stream>>>(scratch, C, M, N, splits, ldc, norm_in, norm_out); \
        else skinny_reduce_kernel<EPI_STORE_BF16, VEC_><<<blocks, 256, 0, stream>>>(scratch, C, M, N, splits, ldc, norm_in, norm_out);                      \
    } while (0)
        const bool four = N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)scratch & 15) == 0 && ((uintptr_t)C & 15) == 0;
        GI_REQUIRE(norm_out.scaled == nullptr || (four && epi == EPI_ADD_F32 && N % REDUCE_COLUMNS == 0 && N / REDUCE_COLUMNS <= REDUCE_MAX_PARTS && norm_out.ld % 4 == 0 &&
                                                  ((uintptr_t)norm_out.scaled & 7) == 0 && ((uintptr_t)norm_out.g & 15) == 0),
                   "gemm_bf16: handing a norm on from %d rows needs rows of a multiple of %d columns, at most %d, and aligned operands", M, REDUCE_COLUMNS,
                   REDUCE_COLUMNS * REDUCE_MAX_PARTS);
        if (four) REDUCE(4); else REDUCE(1);
#undef REDUCE
    }
    GI_CHECK_LAUNCH("gemm_bf16 (reduce)");
    return 0;
}

// Up to 16 rows the slim kernel (no LDS staging, one launch) is the faster one, except where its per-workgroup reading of the activations costs more than staging them.
// Where the weight-streaming kernel is the other one (K no multiple of 64) the longer the rows and the more strips, the sooner, between 3 and 12: 16,384 x 2,056 gated takes 16.6 us
// and 17.7 at 8 rows, 17.1 and 17.8 at 12, 18.1 and 17.9 at 16; 32,000 x 1,000 stored 14.9, 15.3; 15.9, 15.6; 16.7, 15.9.
static int streamed_from_row(int strips, int K) {
    const double fitted = 12.0 * (2048.0 / K) * (256.0 / strips);
    return fitted < 3 ? 3 : fitted > 12 ? 12 : (int)(fitted + 0.5);
}
// Where K is a multiple of 64 the other one is the strips' (the weight-streaming one for some of a short k, `ends_in_strips`).  What decides is how the workgroups of either fill the compute units: strips
// of 64 columns, one a unit where they are one round or less, two of which a unit runs side by side, against workgroups of at most 32 weight rows in so many more rounds, each with its end; and the
// activations, which every workgroup of the slim kernel reads and strips share.  Microseconds, slim and strips, in chains of products with weights of their own:
//   gated                 1 row         8 rows        12 rows       16 rows         stored                1 row         8 rows        12 rows       16 rows
//   12,288 x 2,048        9.6, 11.5     10.8, 11.9    12.9, 12.0    13.6, 12.0      12,288 x 2,048        9.9, 11.5     10.9, 11.7    12.2, 11.7    13.0, 11.7
//   16,384 x 2,048        12.4, 14.2    12.3, 14.5    13.1, 14.6    13.9, 14.6      16,384 x 8,192        44.4, 50.6    43.4, 50.9    44.5, 51.2    46.6, 50.5
//   18,432 x 4,096        26.0, 35.7    29.8, 36.4    33.0, 37.0    35.0, 37.2      18,432 x 4,096        24.4, 35.6    26.3, 36.3    30.3, 36.7    32.2, 37.1
//   28,672 x 4,096        36.4, 40.8    40.4, 41.3    43.0, 41.0    45.3, 41.5      28,672 x 4,096        36.8, 40.9    37.7, 41.5    41.2, 42.8    43.9, 43.2
//   36,864 x 3,072        34.1, 45.1    39.2, 46.1    42.2, 46.3    44.9, 46.6      128,256 x 2,048       75.6, 89.8    77.2, 92.1    84.1, 94.1    90.4, 96.0
//   28,672 x 512          7.7, 7.8      8.1, 8.2      9.1, 8.3      9.5, 8.5        100,352 x 512         21.9, 22.0    23.9, 23.0    27.6, 23.2    29.0, 23.6
// Of 7,742 products (30 widths to 152,064 columns, 28 k, stored and gated, 1 to 16 rows) the choice is 0.3 % slower than the faster of the two on average, 15 with over 10 % (k of 64, 320 and 704); of 576
// gated ones that finish a norm 0.8 %.
static bool slim_beside_strips(int M, int strips, int K, bool gated) {
    const int units = gi_compute_units();
    if (K < 256 && strips > units) return false;                      // (most of a workgroup's waves have no k)
    if (K <= 640) {
        if (strips * 2 <= units * 3) return gated || K < 512 || strips * 10 > units * 9 || M <= 10;
        return K > 256 && M <= (gated || strips > 2 * units ? 8 : 4);
    }
    if (M <= 8) return true;
    if (strips * 10 <= units * 9) return K < 1536 && M <= 12;
    if (strips * 5 > units * 8 && strips * 20 <= units * 37) return M <= (gated ? 10 : K < 1536 ? 12 : 16);
    return true;
}
// xielu: the product ends through that activation, which of the kernels only slim has.
static bool takes_slim(int M, int N, int K, bool gated, bool xielu = false) {
    const int strips = (N + 63) / 64;
    if (M > 16 || gi_gemm_bf16_skinny_splits(N, K) > 0) return M <= 16;
    if (K % PK != 0 || xielu) return M < (strips >= 1024 ? 5 : streamed_from_row(strips, K));
    return slim_beside_strips(M, strips, K, gated);
}

// Weight rows per workgroup of the slim kernel.  A round of workgroups, one per compute unit, takes as long as its weights, a sixth of a row for each that is missing from a group of 8, a fifth of a row
// for each row of A (all of which every workgroup reads; half a row from nine on), two rows' time to begin and end, and what finishing a norm takes, about 0.7 us (which gated products alone go by:
// they have two heights to choose from, and many workgroups); more than 24 rows, with fewer loads in flight, take 5 % longer where k is long, and a round that is not full costs four fifths of one at least.  So an output that
// 256 workgroups of at most 32 rows cover has one round, and wider ones as few as fill it well.  23 outputs of 512 to 16,384 columns, k of 256 to 8,192, 1 to 16 rows, ten to
// thirteen heights each: the choice is 1 % slower than the fastest on average, 14 % at worst; of 16 or 32 rows for 18 gated outputs to 65,536 columns 1 %.  Microseconds by weight rows a workgroup:
//                                      8       12      16      20      24      32
//   6,144 x 4,096 at 1 row             10.05   10.53   11.21   13.65   9.87    11.47
//   6,144 x 4,096 at 8 rows            13.09   12.33   13.26   15.56   10.26   12.33
//   2,048 x 8,192 at 8 rows            9.78    11.93   13.13   15.59   16.82
//   128,256 x 2,048 at 8 rows          119.1   107.0   90.8    91.0    84.7    80.9
//   8,192 x 512 added at 8 rows        4.54            3.93    4.58    4.46           (17: 4.76)
//   28,672 x 4,096 gated, 1 and 12                     37.0, 48.7              42.1, 45.7
//   28,672 x 1,024 gated with a norm, 1 and 8          16.6, 18.7              13.7, 14.5
// Gated columns come in pairs of 16 weight rows, half of which or all a workgroup takes; what adds onto rows stays below 32, whose registers it lacks, and makes no more pieces of a row's
// sum of squares than a reader takes where that can be done (else it hands no norm on).
static int slim_strip_rows(int M, int N, int K, int epi, bool normed) {
    const int units = gi_compute_units();
    const double ends = 2 + (normed && is_gated(epi) ? 8192.0 / K : 0.0);
    auto cost = [&](int rows) {
        const int groups = (N + rows - 1) / rows, whole = groups / units, rest = groups % units;
        const double share = rest == 0 ? 0.0 : whole == 0 ? 1.0 : rest * 5 < units * 4 ? 0.8 : (double)rest / units;
        return (whole + share) * (rows + (8 - rows % 8) % 8 / 6.0 + (M <= 8 ? 0.2 : 0.5) * M + ends) * (rows > 24 && K > 2048 ? 1.05 : 1.0);
    };
    if (is_gated(epi)) return cost(16) < cost(32) ? 16 : 32;
    const int most = epi == EPI_ADD_F32 ? 24 : 32, fit = epi == EPI_ADD_F32 ? (N + slim_max_parts(M) - 1) / slim_max_parts(M) : 8;
    int best = fit <= 8 || fit > most ? 8 : fit;
    for (int rows = best + 1; rows <= most; ++rows)
        if (cost(rows) < cost(best)) best = rows;
    return best;
}
// How the slim kernel reaches rows so far apart.  It adds a row's place and the one in k behind it in 32 bits: in bytes for more than 24 weight rows a workgroup, in pieces of
// 16 bytes for fewer, so the end of the last row that a workgroup reads, from its first, has to lie within.  Beyond the former fewer weight rows a workgroup, beyond the latter
// (68 GB) the variant that reckons in 64 bits, of which there is one for each kind of end.
struct SlimReach { int rows; bool far; };
static SlimReach slim_reach(int M, int N, int K, int epi, bool normed, long lda, long ldw) {
    int rows = slim_strip_rows(M, N, K, epi, normed);
    auto pieces = [&]() {
        const long apart = is_gated(epi) ? 7 : min(rows, N) - 1, w = apart * (ldw / 8), a = (M - 1) * (lda / 8);       // (gated: every group of 8 rows has an address of its own)
        return (w > a ? w : a) + K / 8;
    };
    const int fewer = is_gated(epi) ? 16 : 24;
    if (rows > 24 && pieces() > 1L << 28) rows = fewer;
    const bool far = pieces() > 1L << 32;
    return {far && rows > fewer ? fewer : rows, far};
}

// Workgroups of the slim kernel for an output of N columns that is added onto rows: the pieces a row's sum of squares comes in.
static int slim_parts(int M, int N, int K) {
    const int rows = slim_strip_rows(M, N, K, EPI_ADD_F32, false);
    return (N + rows - 1) / rows;
}

static int launch_slim(const void* A, const void* W, void* C, int epi, int M, int N, int K, long lda, long ldw, long ldc, NormIn norm_in,
                       NormOut norm_out, hipStream_t stream) {
    const bool hand = norm_in.squares != nullptr || (norm_out.scaled != nullptr && epi != EPI_XIELU);
    const auto [rows, far] = slim_reach(M, N, K, epi, norm_in.squares != nullptr, lda, ldw);
    const dim3 grid((N + rows - 1) / rows);
    const int turn = turn_of_steps((K + 63) / 64);
    if (far) {
#define SLIM_FAR(GROUPS_, EPI_) gemm_bf16_slim_kernel<GROUPS_, EPI_, true, 2, true><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, lda / 8, ldw / 8, M, N, K, rows, turn, C, ldc, norm_in, norm_out)
        if (epi == EPI_GATED_BF16) SLIM_FAR(2, EPI_GATED_BF16); else if (epi == EPI_GATED_GELU_BF16) SLIM_FAR(2, EPI_GATED_GELU_BF16); else if (is_gated(epi)) SLIM_FAR(2, EPI_GATED_CLAMP_BF16);
        else if (epi == EPI_STORE_F32) SLIM_FAR(3, EPI_STORE_F32); else if (epi == EPI_ADD_F32) SLIM_FAR(3, EPI_ADD_F32);
        else if (epi == EPI_XIELU) SLIM_FAR(3, EPI_XIELU); else SLIM_FAR(3, EPI_STORE_BF16);
#undef SLIM_FAR
        GI_CHECK_LAUNCH("gemm_bf16 (slim, far)");
        return 0;
    }
#define SLIM_XT(GROUPS_, EPI_, XT_)                                                                                                                    \
    do {                                                                                                                                               \
        if (hand) gemm_bf16_slim_kernel<GROUPS_, EPI_, true, XT_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, (int)(lda / 8), (int)(ldw / 8), M, N, K, rows, turn, C, ldc, norm_in, norm_out); \
        else gemm_bf16_slim_kernel<GROUPS_, EPI_, false, XT_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, (int)(lda / 8), (int)(ldw / 8), M, N, K, rows, turn, C, ldc, norm_in, norm_out);     \
    } while (0)
#define SLIM(GROUPS_, EPI_) do { if (M <= 8) SLIM_XT(GROUPS_, EPI_, 1); else SLIM_XT(GROUPS_, EPI_, 2); } while (0)
#define SLIM_EPI(GROUPS_)                                                                                                                              \
    do {                                                                                                                                               \
        if (epi == EPI_STORE_F32) SLIM(GROUPS_, EPI_STORE_F32); else if (epi == EPI_ADD_F32) SLIM(GROUPS_, EPI_ADD_F32);                               \
        else if (epi == EPI_XIELU) SLIM(GROUPS_, EPI_XIELU); else SLIM(GROUPS_, EPI_STORE_BF16);                                                       \
    } while (0)
#define SLIM_GATED(GROUPS_)                                                                                                                            \
    do {                                                                                                                                               \
        if (epi == EPI_GATED_BF16) SLIM(GROUPS_, EPI_GATED_BF16); else if (epi == EPI_GATED_GELU_BF16) SLIM(GROUPS_, EPI_GATED_GELU_BF16);             \
        else SLIM(GROUPS_, EPI_GATED_CLAMP_BF16);                                                                                                      \
    } while (0)
    if (is_gated(epi)) { if (rows == 32) SLIM_GATED(4); else SLIM_GATED(2); }
    else if (rows > 24) {
        if (epi == EPI_STORE_F32) SLIM(4, EPI_STORE_F32); else if (epi == EPI_XIELU) SLIM(4, EPI_XIELU); else SLIM(4, EPI_STORE_BF16);
    }
    else if (rows > 16) SLIM_EPI(3);
    else if (rows > 8) SLIM_EPI(2);
    else SLIM_EPI(1);
#undef SLIM_GATED
#undef SLIM_EPI
#undef SLIM
#undef SLIM_XT
    GI_CHECK_LAUNCH("gemm_bf16 (slim)");
    return 0;
}

// 17 to 32 rows, a narrow output and a short k: one launch of the slim kernel with two tiles of activation rows.  Measured at
// N = 3072 and 2048, K = 2048 against the skinny kernel's partial sums and their second kernel: 9 against 13 us at 17 and 32 rows,
// 11 against 13 at 48, 13 against 13 at 64; at K = 8192 (every workgroup reads all the activations: 1 MB at 64 rows) 21 to 43 us
// against 16 to 19, so longer k and more rows stay with the skinny kernel.  Rows beyond 32 given to further workgroups of two tiles (a
// second grid dimension: 256 workgroups at 64 rows and N = 2048, each with 64 KB of weights and its own 128 KB of A) measured
// equal at 33 to 64 rows and 3 % slower in the whole step from 65 rows on: not kept.
static bool takes_slim_tiles(int M, int N, int K, int epi) {
    return !takes_slim(M, N, K, is_gated(epi)) && M <= 32 && K <= 2048 && !is_gated(epi) && gi_gemm_bf16_skinny_splits(N, K) > 0;
}

// Weight rows per workgroup of that kernel: 16, or 12 or 8 where strips of 16 fill the compute units unevenly and those fill
// them evenly (2,048 columns: 256 strips of 8, not 128 of 16; 3,072: 256 of 12, not 192 of 16: the decode step of the 1B shape at 17 to 32
// rows 1 to 1.5 % faster), never more strips than a reader takes pieces.
static int tiles_strip_rows(int N) {
    const int units = gi_compute_units();
    auto evenness = [&](int rows) {
        const int groups = (N + rows - 1) / rows;
        return (double)groups / ((groups + units - 1) / units * units);
    };
    if (evenness(16) >= 0.8) return 16;
    for (int rows : {12, 8})
        if (evenness(rows) >= 0.95 && (N + rows - 1) / rows <= TILES_MAX_PARTS) return rows;
    return 16;
}

static int launch_slim_tiles(const void* A, const void* W, void* C, int epi, int M, int N, int K, long lda, long ldw, long ldc, NormIn norm_in,
                             NormOut norm_out, hipStream_t stream) {
    const int strip_rows = tiles_strip_rows(N);
    dim3 grid((N + strip_rows - 1) / strip_rows);
#define SLIM_TILES(MT_)                                                                                                                             \
    do {                                                                                                                                            \
        if (epi == EPI_STORE_F32) gemm_bf16_slim_tiles_kernel<MT_, EPI_STORE_F32><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, norm_in, norm_out, strip_rows); \
        else if (epi == EPI_ADD_F32) gemm_bf16_slim_tiles_kernel<MT_, EPI_ADD_F32><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, norm_in, norm_out, strip_rows); \
        else gemm_bf16_slim_tiles_kernel<MT_, EPI_STORE_BF16><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, norm_in, norm_out, strip_rows); \
    } while (0)
    SLIM_TILES(2);
#undef SLIM_TILES
    GI_CHECK_LAUNCH("gemm_bf16 (slim, tiles)");
    return 0;
}

// cut.splits == 0: all of k is one workgroup's, which ends the product with `epi`; else the sums go to `scratch`.
static int launch_strips(const void* A, const void* W, void* C, int epi, int M, int N, int K, long lda, long ldw, long ldc, float* scratch, StripCut cut, NormIn norm_in, hipStream_t stream) {
    const int splits = cut.splits, k_per_split = splits == 0 ? K : (K / PK + splits - 1) / splits * PK;
    const int tile_rows = (M + cut.tiles - 1) / cut.tiles;
    dim3 grid((N + 63) / 64, splits == 0 ? 1 : splits, cut.tiles);
    // Places of their own in k (`first_step`): where k is shared out too, up to 160 rows (54 products 2 % faster in the mean, 64 rows of 2,048 x 2,048 11.2 us -> 10.0, 131 of 2,048 x 8,192 18.1 -> 17.6),
    // but not above, where 42 products were 0.5 % slower (200 rows of 4,096 x 14,336 48.1 and 50.6).
    const int turn = splits != 0 && M > 160 ? 0 : turn_of_steps(k_per_split / PK);
#define STRIP(TM_, ST_, EPI_, PARTIAL_)                                                                                                 \
    do {                                                                                                                                \
        constexpr int bytes = strip_bytes(TM_, ST_);                                                                                    \
        static bool raised = false;                                                                                                     \
        if (!raised) {                                                                                                                  \
            if (hipFuncSetAttribute((const void*)gemm_bf16_strip_kernel<TM_, ST_, EPI_, PARTIAL_>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) \
                return gi_fail("gemm_bf16: cannot reserve %d bytes of LDS", bytes);                                                     \
            raised = true;                                                                                                              \
        }                                                                                                                               \
        gemm_bf16_strip_kernel<TM_, ST_, EPI_, PARTIAL_><<<grid, 512, bytes, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, tile_rows, turn, norm_in); \
    } while (0)
#define STRIP_TM(EPI_, PARTIAL_)                                                                                                        \
    do {                                                                                                                                \
        if (tile_rows <= 32) STRIP(1, 6, EPI_, PARTIAL_); else if (tile_rows <= 64) STRIP(2, 4, EPI_, PARTIAL_); else if (tile_rows <= 96) STRIP(3, 4, EPI_, PARTIAL_); \
        else if (!one_round) STRIP(4, 3, EPI_, PARTIAL_); else STRIP(4, 6, EPI_, PARTIAL_);                                             \
    } while (0)
#define STRIP_GATED(EPI_)                                                                                                               \
    do {                                                                                                                                \
        if (M <= 128) STRIP_TM(EPI_, false); else if (M <= 160) STRIP(5, 5, EPI_, false); else STRIP(6, 4, EPI_, false);                \
    } while (0)
    // Up to 128 rows two workgroups fit a compute unit's LDS, but where there are no more workgroups than units a deeper ring serves better (128 rows of 16,384 x 2,048
    // gated 24.2 us with six stages, 25.4 with three; of 28,672 x 4,096 75.6 and 71.5).
    const bool one_round = (long)grid.x * grid.y * grid.z <= gi_compute_units();
    if (splits != 0 && tile_rows <= 128) STRIP_TM(EPI_STORE_F32, true);
    else if (splits != 0) {
        if (tile_rows <= 160) STRIP(5, 5, EPI_STORE_F32, true); else if (tile_rows <= 192) STRIP(6, 4, EPI_STORE_F32, true);
        else if (tile_rows <= 224) STRIP(7, 4, EPI_STORE_F32, true); else STRIP(8, 4, EPI_STORE_F32, true);
    }
    else if (epi == EPI_GATED_BF16) STRIP_GATED(EPI_GATED_BF16);
    else if (epi == EPI_GATED_GELU_BF16) STRIP_GATED(EPI_GATED_GELU_BF16);
    else if (epi == EPI_GATED_CLAMP_BF16) STRIP_GATED(EPI_GATED_CLAMP_BF16);
    else if (M > 128) return gi_fail("gemm_bf16 (strips): %d rows are not taken", M);
    else if (epi == EPI_STORE_F32) STRIP_TM(EPI_STORE_F32, false);
    else if (epi == EPI_ADD_F32) STRIP_TM(EPI_ADD_F32, false);
    else STRIP_TM(EPI_STORE_BF16, false);
#undef STRIP_GATED
#undef STRIP_TM
#undef STRIP
    GI_CHECK_LAUNCH("gemm_bf16 (strips)");
    return 0;
}

// Up to 128 rows the weights are the traffic and every workgroup streams its share of them once (measured on the decode step of
// the Llama-3.2-1B shape: 72 rows took 2.69 ms through the tiles of 128 rows of the kernels for more rows, against 2.11 ms at 64 rows).
static int launch_skinny(const void* A, const void* W, void* C, int epi, int M, int N, int K, long lda, long ldw, long ldc, float* scratch,
                         long scratch_floats, NormIn norm_in, NormOut norm_out, hipStream_t stream, const RopeStore* rope = nullptr, const WholeNorm* whole = nullptr) {
    const int splits = gi_gemm_bf16_skinny_splits(N, K), mt = (M + 15) / 16;
#define SKINNY_MT(EPI_, PARTIAL_)                                                                                                   \
    do {                                                                                                                            \
        if (mt == 1) gemm_bf16_skinny_kernel<1, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else if (mt == 2) gemm_bf16_skinny_kernel<2, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else if (mt == 3) gemm_bf16_skinny_kernel<3, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else if (mt == 4) gemm_bf16_skinny_kernel<4, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else if (mt == 5) gemm_bf16_skinny_kernel<5, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else if (mt == 6) gemm_bf16_skinny_kernel<6, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else if (mt == 7) gemm_bf16_skinny_kernel<7, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
        else gemm_bf16_skinny_kernel<8, EPI_, PARTIAL_><<<grid, 512, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, scratch, M, N, K, lda, ldw, ldc, k_per_split, norm_in); \
    } while (0)
    GI_REQUIRE(norm_in.squares == nullptr || norm_in.parts <= consumer_max_parts(M), "gemm_bf16: %d pieces of a sum of squares, at most %d for %d rows",
               norm_in.parts, consumer_max_parts(M), M);
    if (splits == 0) {                             // a wide output: every workgroup sees all of k and finishes its columns
        GI_REQUIRE(norm_out.scaled == nullptr && rope == nullptr, "gemm_bf16: a product this wide does not hand a norm on, or its rows to the cache");
        if (ends_in_strips(M, N, K) && strip_strides(lda, ldw)) return launch_strips(A, W, C, epi, M, N, K, lda, ldw, ldc, nullptr, StripCut{1, 0, 0}, norm_in, stream);
        const int k_per_split = K;
        dim3 grid((N + 63) / 64, 1);
        if (epi == EPI_GATED_BF16) SKINNY_MT(EPI_GATED_BF16, false); else if (epi == EPI_GATED_GELU_BF16) SKINNY_MT(EPI_GATED_GELU_BF16, false); else if (epi == EPI_GATED_CLAMP_BF16) SKINNY_MT(EPI_GATED_CLAMP_BF16, false); else if (epi == EPI_STORE_F32) SKINNY_MT(EPI_STORE_F32, false);
        else if (epi == EPI_ADD_F32) SKINNY_MT(EPI_ADD_F32, false); else SKINNY_MT(EPI_STORE_BF16, false);
        GI_CHECK_LAUNCH("gemm_bf16 (skinny)");
        return 0;
    }
    GI_REQUIRE(scratch != nullptr && scratch_floats >= (long)splits * M * N, "gemm_bf16: scratch of %ld floats needed, %ld given",
               (long)splits * M * N, scratch_floats);
    int parts = splits;
    const StripCut cut = strip_strides(lda, ldw) ? shared_strips(M, N, K, splits) : StripCut{0, 0, 0};
    if (cut.tiles && scratch_floats >= (long)cut.splits * M * N) {
        parts = cut.splits;
        if (int rc = launch_strips(A, W, nullptr, EPI_STORE_F32, M, N, K, lda, ldw, (long)N, scratch, cut, NO_NORM_IN, stream)) return rc;
    } else {
        const int k_per_split = ((K + splits - 1) / splits + KB - 1) / KB * KB;
        dim3 grid((N + 63) / 64, splits);
        SKINNY_MT(EPI_STORE_F32, true);
    }
#undef SKINNY_MT
    GI_CHECK_LAUNCH("gemm_bf16 (skinny)");
    if (rope != nullptr) {                         // the sums go where an attention layer wants its queries, keys and values
        skinny_reduce_rope_store_kernel<<<(unsigned)(((size_t)M * N / 4 + 255) / 256), 256, 0, stream>>>(scratch, M, N, parts, norm_in, *rope);
        GI_CHECK_LAUNCH("gemm_bf16 (reduce, rotate, store)");
        return 0;
    }
    return reduce_partials(scratch, C, epi, M, N, parts, ldc, stream, norm_in, norm_out, whole);
}

static TileOrder tall_order(int M, int N, int whole) {
    TileOrder o = {(M + 255) / 256, (N + 127) / 128, 0, 1};
    o.each = (whole + 7) / 8;
    const int all = (o.m_tiles * o.n_tiles + 7) / 8, run = all < gi_compute_units() / 8 ? all : gi_compute_units() / 8;       // of a die at a time
    while ((o.panel + 1) * (o.panel + 1) <= 2 * run) ++o.panel;
    if (o.panel * o.m_tiles < run) o.panel = (run + o.m_tiles - 1) / o.m_tiles;
    if (o.panel > o.n_tiles) o.panel = o.n_tiles;
    return o;
}

static const RopeStore NO_ROPE = {nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, nullptr, 0, 0, 0, 0, 0};

// The pieces per row that a product of more than 128 rows writes when it hands a norm on, 0 if it cannot: one per tile of 128 columns
// from the epilogue of the kernel with tiles of 128 x 128, one per 1024 columns where k is shared out and a second kernel adds the
// shares; none from a product with many tiles.
static int large_norm_parts(int M, int N, int K) {
    if (K % PK != 0 || N < 128 || many_tiles(M, N)) return 0;
    if (gi_gemm_bf16_piped_splits(M, N, K) > 1) return N % REDUCE_COLUMNS == 0 && N / REDUCE_COLUMNS <= REDUCE_MAX_PARTS ? N / REDUCE_COLUMNS : 0;
    return N % 128 == 0 && N / 128 <= PIPED_MAX_PARTS ? N / 128 : 0;
}

// More than 128 rows, K a multiple of 64, 128 columns or more: the kernels that load their operands straight into LDS.
// `rope` != null: the sums are those of an attention layer's q/k/v product and go where it says (`epi` is then not looked at).
static int launch_large(const void* A, const void* W, void* C, int epi, int M, int N, int K, long lda, long ldw, long ldc, float* scratch,
                        long scratch_floats, NormIn norm_in, const RopeStore* rope, hipStream_t stream, NormOut norm_out = NO_NORM_OUT, const WholeNorm* whole = nullptr,
                        unsigned* counters = nullptr) {
    const NormIn limit_in = {nullptr, 0, 0.f, 1, norm_in.limit};          // no norm to finish, the clamped gate's limit alone
#define PIPED(BM_, BN_, WM_, WN_, ST_, EPI_, OUT_, LDC_, SPLITS_, KPS_, SLAB_, NORM_, ROPE_)                                            \
    do {                                                                                                                                \
        constexpr int bytes = ST_ * (BM_ + BN_) * 128;                                                                                  \
        static bool raised = false;                                                                                                     \
        if (!raised) {                                                                                                                  \
            if (hipFuncSetAttribute((const void*)gemm_bf16_piped_kernel<BM_, BN_, WM_, WN_, ST_, EPI_>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) \
                return gi_fail("gemm_bf16: cannot reserve %d bytes of LDS", bytes);                                                     \
            raised = true;                                                                                                              \
        }                                                                                                                               \
        dim3 grid((N + BN_ - 1) / BN_, (M + BM_ - 1) / BM_, SPLITS_);                                                                   \
        gemm_bf16_piped_kernel<BM_, BN_, WM_, WN_, ST_, EPI_><<<grid, 64 * WM_ * WN_, bytes, stream>>>((const bf16_t*)A, (const bf16_t*)W, OUT_, M, N, K, lda, \
                                                                                                        ldw, LDC_, KPS_, SLAB_, NORM_, ROPE_, norm_out); \
    } while (0)
#define PIPED_EPI(BM_, BN_, WM_, WN_, ST_)                                                                                              \
    do {                                                                                                                                \
        if (rope != nullptr) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_QKV_ROPE, nullptr, 0L, 1, K, 0L, norm_in, *rope);                       \
        else if (epi == EPI_STORE_F32) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_STORE_F32, C, ldc, 1, K, 0L, NO_NORM_IN, NO_ROPE);            \
        else if (epi == EPI_ADD_F32) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_ADD_F32, C, ldc, 1, K, 0L, NO_NORM_IN, NO_ROPE);                \
        else if (epi == EPI_STORE_BF16) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_STORE_BF16, C, ldc, 1, K, 0L, NO_NORM_IN, NO_ROPE);          \
        else if (epi == EPI_XIELU) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_XIELU, C, ldc, 1, K, 0L, NO_NORM_IN, NO_ROPE);                    \
        else if (epi == EPI_GATED_BF16) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_GATED_BF16, C, ldc, 1, K, 0L, NO_NORM_IN, NO_ROPE);          \
        else if (epi == EPI_GATED_GELU_BF16) PIPED(BM_, BN_, WM_, WN_, ST_, EPI_GATED_GELU_BF16, C, ldc, 1, K, 0L, NO_NORM_IN, NO_ROPE); \
        else PIPED(BM_, BN_, WM_, WN_, ST_, EPI_GATED_CLAMP_BF16, C, ldc, 1, K, 0L, limit_in, NO_ROPE);                                 \
    } while (0)
    const int splits = gi_gemm_bf16_piped_splits(M, N, K);
    if (splits > 1) {                              // few tiles: k is shared out, the sums are finished by the reduce kernel
        GI_REQUIRE(scratch != nullptr && scratch_floats >= (long)splits * M * N, "gemm_bf16: scratch of %ld floats needed, %ld given",
                   (long)splits * M * N, scratch_floats);
        int parts = splits;
        const StripCut cut = strip_strides(lda, ldw) ? shared_strips(M, N, K, splits) : StripCut{0, 0, 0};
        if (cut.tiles && scratch_floats >= (long)cut.splits * M * N) {
            parts = cut.splits;
            if (int rc = launch_strips(A, W, nullptr, EPI_STORE_F32, M, N, K, lda, ldw, (long)N, scratch, cut, NO_NORM_IN, stream)) return rc;
        } else {
            PIPED(128, 128, 2, 2, 2, EPI_STORE_F32, scratch, (long)N, splits, K / splits, (long)M * N, NO_NORM_IN, NO_ROPE);
        }
        GI_CHECK_LAUNCH("gemm_bf16 (piped, split)");
        if (rope != nullptr) {
            skinny_reduce_rope_store_kernel<<<(unsigned)(((size_t)M * N / 4 + 255) / 256), 256, 0, stream>>>(scratch, M, N, parts, norm_in, *rope);
            GI_CHECK_LAUNCH("gemm_bf16 (reduce, rotate, store)");
            return 0;
        }
        return reduce_partials(scratch, C, epi, M, N, parts, ldc, stream, norm_in, norm_out, whole);
    }
    if (rope == nullptr && is_gated(epi) && norm_in.squares == nullptr && ends_in_strips(M, N, K) && strip_strides(lda, ldw)) return launch_strips(A, W, C, epi, M, N, K, lda, ldw, ldc, nullptr, StripCut{1, 0, 0}, limit_in, stream);
    const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);
    GI_REQUIRE(norm_out.scaled == nullptr || (!many_tiles(M, N) && large_norm_parts(M, N, K) > 0), "gemm_bf16: a product of M %d, N %d, K %d hands no norm on", M, N, K);
    GI_REQUIRE(norm_in.squares == nullptr || rope != nullptr || (is_gated(epi) && many_tiles(M, N) && norm_in.parts <= PIPED_MAX_PARTS),
               "gemm_bf16: a product of M %d, N %d, K %d takes no norm handed on in %d pieces", M, N, K, norm_in.parts);
    GI_REQUIRE(!many_tiles(M, N) || (lda < (1L << 22) && ldw < (1L << 22)), "gemm_bf16: row strides %ld, %ld are too large for the tile-relative addressing", lda, ldw);
    const bool clears = counters == nullptr;
    const long sharing = tall_scratch_floats(tall_cut(M, N, K, true, clears));
    const bool may_share = sharing > 0 && scratch != nullptr && scratch_floats >= sharing && ((uintptr_t)scratch & 15) == 0;
    LargeChoice choice = {PIPED_128, {}};
    if (lda < (1L << 22) && ldw < (1L << 22))
        choice = large_kernel(M, N, K, epi, rope != nullptr, norm_out.scaled != nullptr, norm_in.squares != nullptr, may_share, clears);
    const Large which = choice.kernel;
    if (which == PINGPONG_256) {
#define PINGPONG(EPI_)                                                                                                                  \
    do {                                                                                                                                \
        constexpr int bytes = (2 * 256 + 3 * 256) * 128;                                                                                            \
        static bool raised = false;                                                                                                     \
        if (!raised) {                                                                                                                  \
            if (hipFuncSetAttribute((const void*)gemm_bf16_pingpong_kernel<256, EPI_>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) \
                return gi_fail("gemm_bf16: cannot reserve %d bytes of LDS", bytes);                                                     \
            raised = true;                                                                                                              \
        }                                                                                                                               \
        dim3 grid((N + 255) / 256, (M + 255) / 256);                                                                                    \
        gemm_bf16_pingpong_kernel<256, EPI_><<<grid, 512, bytes, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, norm_in, rope != nullptr ? *rope : NO_ROPE); \
    } while (0)
        if (rope != nullptr) PINGPONG(EPI_QKV_ROPE);
        else if (epi == EPI_STORE_F32) PINGPONG(EPI_STORE_F32); else if (epi == EPI_ADD_F32) PINGPONG(EPI_ADD_F32);
        else if (epi == EPI_XIELU) { norm_in.squares = norm_out.g; PINGPONG(EPI_XIELU); }
        else if (epi == EPI_STORE_BF16) PINGPONG(EPI_STORE_BF16); else if (epi == EPI_GATED_BF16) PINGPONG(EPI_GATED_BF16); else if (epi == EPI_GATED_GELU_BF16) PINGPONG(EPI_GATED_GELU_BF16); else PINGPONG(EPI_GATED_CLAMP_BF16);
#undef PINGPONG
        GI_CHECK_LAUNCH("gemm_bf16 (pingpong)");
        return 0;
    }
    if (which == TALL_256) {
        const TallCut& cut = choice.cut;
        const TileOrder order = tall_order(M, N, cut.whole);
        const TileShares shared = {cut.whole, cut.rest, cut.shares, cut.shares > 1 ? scratch + tall_counter_floats(cut) : nullptr, counters != nullptr ? counters : (unsigned*)scratch};
        if (cut.shares > 1 && clears) {
            clear_counters_kernel<<<1, 256, 0, stream>>>(shared.counters, 4 * cut.rest);
            GI_CHECK_LAUNCH("gemm_bf16 (counters)");
        }
#define TALL_AS(EPI_, SHARED_)                                                                                                          \
    do {                                                                                                                                \
        constexpr int bytes = 3 * 384 * 128;                                                                                            \
        static bool raised = false;                                                                                                     \
        if (!raised) {                                                                                                                  \
            if (hipFuncSetAttribute((const void*)gemm_bf16_tall_kernel<EPI_, SHARED_>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) \
                return gi_fail("gemm_bf16: cannot reserve %d bytes of LDS", bytes);                                                     \
            raised = true;                                                                                                              \
        }                                                                                                                               \
        dim3 grid(8 * order.each + (SHARED_ ? (cut.rest * cut.shares + 7) / 8 * 8 : 0));                                                 \
        gemm_bf16_tall_kernel<EPI_, SHARED_><<<grid, 512, bytes, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, norm_in, \
                                                                           rope != nullptr ? *rope : NO_ROPE, norm_out, order, shared, many_tiles(M, N)); \
    } while (0)
#define TALL(EPI_)                              \
    do {                                        \
        if (cut.shares > 1) TALL_AS(EPI_, true); \
        else TALL_AS(EPI_, false);              \
    } while (0)
        if (rope != nullptr) TALL(EPI_QKV_ROPE); else if (epi == EPI_STORE_F32) TALL(EPI_STORE_F32); else if (epi == EPI_ADD_F32) TALL(EPI_ADD_F32);
        else if (epi == EPI_XIELU) TALL_AS(EPI_XIELU, false);      // (never shared out)
        else if (epi == EPI_STORE_BF16) TALL(EPI_STORE_BF16); else if (epi == EPI_GATED_BF16) TALL(EPI_GATED_BF16); else if (epi == EPI_GATED_GELU_BF16) TALL(EPI_GATED_GELU_BF16); else TALL(EPI_GATED_CLAMP_BF16);
#undef TALL
#undef TALL_AS
        GI_CHECK_LAUNCH("gemm_bf16 (tall)");
        return 0;
    }
    // tiles of 128 x 128: two workgroups per unit with two stages each when there are enough tiles, else one of eight waves with four stages
    if (tiles128 > gi_compute_units()) PIPED_EPI(128, 128, 2, 2, 2);
    else PIPED_EPI(128, 128, 2, 4, 4);
#undef PIPED_EPI
#undef PIPED
    GI_CHECK_LAUNCH("gemm_bf16 (piped)");
    return 0;
}

// The pieces per row that a product of these sizes writes when it hands a norm on (gi_gemm_bf16_handing with `scaled_out`);
// 0 if it cannot: a shape whose kernel does not do it.  One piece per workgroup from the kernels that finish a product of up to
// 16 or 32 rows in one launch; up to 128 rows one per 1024 columns, from the kernel that adds the partial sums of the shares of k
// onto the rows.
GI_API int gi_gemm_bf16_norm_parts(int M, int N, int K) {
    if (takes_slim(M, N, K, false)) {
        const int parts = slim_parts(M, N, K);
        return parts <= slim_max_parts(M) ? parts : 0;
    }
    if (takes_slim_tiles(M, N, K, EPI_ADD_F32)) {
        const int parts = (N + tiles_strip_rows(N) - 1) / tiles_strip_rows(N);
        return parts <= TILES_MAX_PARTS ? parts : 0;
    }
    if (M > SKINNY_MAX_ROWS) return large_norm_parts(M, N, K);
    if (M <= 16 || gi_gemm_bf16_skinny_splits(N, K) == 0) return 0;
    return N % REDUCE_COLUMNS == 0 && N / REDUCE_COLUMNS <= REDUCE_MAX_PARTS ? N / REDUCE_COLUMNS : 0;
}

// Whether a product of these sizes can read rows whose norm was handed on (gi_gemm_bf16_handing with `squares_in`) by a product
// of as many rows.
GI_API int gi_gemm_bf16_takes_norm(int M, int N, int K, int gated) {
    if (takes_slim(M, N, K, gated != 0) || takes_slim_tiles(M, N, K, gated ? EPI_GATED_BF16 : EPI_STORE_F32)) return 1;
    if (M > SKINNY_MAX_ROWS)                      // the rows of prompts: the gated product with many tiles scales in its epilogue
        return gated && K % PK == 0 && N >= 128 && many_tiles(M, N) ? 1 : 0;
    if (gi_gemm_bf16_skinny_splits(N, K) == 0) return 1;      // the weight-streaming kernel finishes its columns and scales them
    return M > 32 && !gated ? 1 : 0;                          // the kernel that adds the shares of k scales: with a few pieces only
}

// gi_gemm_bf16 for at most 128 rows, with an RMS norm handed from one product to the next instead of a kernel of its own.
// squares_in != null: the rows A are g * x of some rows x, in bfloat16, and squares_in [M, parts_in] holds the pieces of every
// row's sum of x^2; the results are multiplied by rsqrt(sum / K + eps).  scaled_out != null (needs accumulate onto 32-bit C):
// beside C += A W^T, scaled_out [M, ld_scaled] = bfloat16(g * C) and squares_out [M, gi_gemm_bf16_norm_parts(M, N, K)] = the
// pieces of the rows' sums of C^2, for the next product.  Where the two queries above say no, it fails.
GI_API int gi_gemm_bf16_handing(const void* A, const void* W, void* C, int c_dtype, int accumulate, int gated, float gate_limit, int M, int N, int K, long lda,
                                long ldw, long ldc, float* scratch, long scratch_floats, const float* squares_in, int parts_in, float eps,
                                const float* g, void* scaled_out, long ld_scaled, float* squares_out, unsigned* counters, hipStream_t stream) {
    GI_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_bf16: M %d, N %d, K %d must be positive", M, N, K);
    GI_REQUIRE(K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0, "gemm_bf16: K %d and the row strides (%ld, %ld) must be multiples of 8", K, lda, ldw);
    GI_REQUIRE(((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_bf16: operands must be 16-byte aligned");
    GI_REQUIRE(lda >= K && ldw >= K && ldc >= (gated ? N / 2 : N), "gemm_bf16: leading dimensions too small");
    int epi = epilogue_of(c_dtype, accumulate);
    if (gated) {
        GI_REQUIRE(N % 32 == 0 && c_dtype == GI_BF16 && !accumulate, "gemm_bf16: the gated product needs N %% 32 == 0 and a bfloat16 output");
        epi = gated == 3 ? EPI_GATED_CLAMP_BF16 : gated == 2 ? EPI_GATED_GELU_BF16 : EPI_GATED_BF16;
    }
    GI_REQUIRE(epi >= 0, "gemm_bf16: output dtype %d with accumulate %d is not supported", c_dtype, accumulate);
    GI_REQUIRE(squares_in == nullptr || (parts_in > 0 && gi_gemm_bf16_takes_norm(M, N, K, gated)),
               "gemm_bf16: a product of these sizes (M %d, N %d, K %d%s) cannot finish a norm handed on", M, N, K, gated ? ", gated" : "");
    GI_REQUIRE(scaled_out == nullptr || (epi == EPI_ADD_F32 && g != nullptr && squares_out != nullptr && ld_scaled >= N && gi_gemm_bf16_norm_parts(M, N, K) > 0),
               "gemm_bf16: handing a norm on needs a product that adds onto 32-bit rows, of sizes that allow it (M %d, N %d, K %d), the norm's weights and "
               "room for the sums of squares", M, N, K);
    const NormIn norm_in = {squares_in, parts_in, eps, K, gate_limit};
    const NormOut norm_out = {g, (bf16_t*)scaled_out, ld_scaled, squares_out};
    if (takes_slim(M, N, K, gated != 0)) {
        GI_REQUIRE(squares_in == nullptr || parts_in <= slim_max_parts(M), "gemm_bf16: %d pieces of a sum of squares, at most %d", parts_in, slim_max_parts(M));
        return launch_slim(A, W, C, epi, M, N, K, lda, ldw, ldc, norm_in, norm_out, stream);
    }
    if (takes_slim_tiles(M, N, K, epi)) {
        GI_REQUIRE(squares_in == nullptr || parts_in <= consumer_max_parts(M), "gemm_bf16: %d pieces of a sum of squares, at most %d", parts_in, consumer_max_parts(M));
        return launch_slim_tiles(A, W, C, epi, M, N, K, lda, ldw, ldc, norm_in, norm_out, stream);
    }
    if (M > SKINNY_MAX_ROWS) {                   // the rows of prompts: a norm is handed on (to a q/k/v product that takes it), none is taken
        GI_REQUIRE(scaled_out == nullptr || (ldc % 4 == 0 && ld_scaled % 4 == 0 && ((uintptr_t)C & 15) == 0 && ((uintptr_t)scaled_out & 7) == 0 && ((uintptr_t)g & 15) == 0),
                   "gemm_bf16: handing a norm on from %d rows needs aligned operands", M);
        return launch_large(A, W, C, epi, M, N, K, lda, ldw, ldc, scratch, scratch_floats, norm_in, nullptr, stream, norm_out, nullptr, counters);
    }
    return launch_skinny(A, W, C, epi, M, N, K, lda, ldw, ldc, scratch, scratch_floats, norm_in, norm_out, stream);
}

// Whether a product of these sizes can make the whole norm of the rows it adds onto (gi_gemm_bf16_onto_norm): where k is shared out over workgroups, the kernel
// that adds the shares up sees whole rows.
GI_API int gi_gemm_bf16_onto_norm_takes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || N % 4 != 0 || N > WHOLE_NORM_COLUMNS || K <= 0 || K % 8 != 0) return 0;
    if (M <= SKINNY_MAX_ROWS) return !takes_slim(M, N, K, false) && !takes_slim_tiles(M, N, K, EPI_ADD_F32) && gi_gemm_bf16_skinny_splits(N, K) > 0;
    return K % PK == 0 && N >= 128 && gi_gemm_bf16_piped_splits(M, N, K) > 1;
}

// C += A W^T onto 32-bit rows C [M, ldc], and normed [M, ld_normed] = bfloat16(g * (C * rsqrt(mean(C^2) + eps))), the norm that reads the rows next.
GI_API int gi_gemm_bf16_onto_norm(const void* A, const void* W, float* C, int M, int N, int K, long lda, long ldw, long ldc, float* scratch, long scratch_floats, const float* g,
                                  float eps, void* normed, long ld_normed, hipStream_t stream) {
    GI_REQUIRE(gi_gemm_bf16_onto_norm_takes(M, N, K), "gemm_bf16 (norm): sizes M %d, N %d, K %d are not taken", M, N, K);
    GI_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K && ((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0,
               "gemm_bf16 (norm): rows must be 16-byte aligned (strides %ld, %ld)", lda, ldw);
    GI_REQUIRE(C != nullptr && g != nullptr && normed != nullptr && ldc >= N && ldc % 4 == 0 && ld_normed >= N && ld_normed % 4 == 0 &&
                   (((uintptr_t)C | (uintptr_t)g | (uintptr_t)scratch) & 15) == 0 && ((uintptr_t)normed & 7) == 0,
               "gemm_bf16 (norm): outputs or weights are missing or not aligned (strides %ld, %ld)", ldc, ld_normed);
    const WholeNorm whole = {g, (bf16_t*)normed, ld_normed, eps};
    if (M <= SKINNY_MAX_ROWS) return launch_skinny(A, W, C, EPI_ADD_F32, M, N, K, lda, ldw, ldc, scratch, scratch_floats, NO_NORM_IN, NO_NORM_OUT, stream, nullptr, &whole);
    return launch_large(A, W, C, EPI_ADD_F32, M, N, K, lda, ldw, ldc, scratch, scratch_floats, NO_NORM_IN, nullptr, stream, NO_NORM_OUT, &whole);
}

// Whether gi_gemm_bf16_qkv_rope_store takes a q/k/v product of these sizes with heads of hd channels.  17 or 33 to 128 rows: the
// shapes whose k is shared out over workgroups, whose sums a second kernel adds up anyway.  More rows: the kernels with tiles of
// 128 x 128, 256 x 128 and 256 x 256, whose epilogues lay 128 rows of the tile into LDS (of 256 columns as two such tiles) and send them off rotated (whole heads must lie
// inside 128 columns), or, where they share k out, that second kernel again.
GI_API int gi_gemm_bf16_qkv_rope_store_takes(int M, int N, int K, int hd) {
    if (hd < 8 || hd > 256 || (hd & (hd - 1)) != 0) return 0;
    if (M <= SKINNY_MAX_ROWS)
        return !takes_slim(M, N, K, false) && !takes_slim_tiles(M, N, K, EPI_STORE_F32) && gi_gemm_bf16_skinny_splits(N, K) > 0 && N % 256 == 0 ? 1 : 0;
    if (K % PK != 0 || N < 128) return 0;
    return gi_gemm_bf16_piped_splits(M, N, K) > 1 ? N % 256 == 0 : hd <= 128;
}

// The most pieces of a row's sum of squares that gi_gemm_bf16_qkv_rope_store reads for a product of M rows.
GI_API int gi_gemm_bf16_qkv_rope_store_max_parts(int M, int N, int K) {
    return M <= SKINNY_MAX_ROWS || gi_gemm_bf16_piped_splits(M, N, K) > 1 ? REDUCE_MAX_PARTS : many_tiles(M, N) ? 0 : PIPED_MAX_PARTS;
}

// The q/k/v product of an attention layer, A [M, K] x W [N, K]^T with N = (n_heads + 2 n_kv) * hd, whose results do not come back:
// the queries go, rotated, to q_out [M, n_heads * hd] in bfloat16, the keys (rotated) and values into the pages of a bfloat16
// cache, as gi_rope_store would put them (cos_t, sin_t [M, hd/2] or both null; pos, slot [M]; table, cache, page_stride, page_size
// as there).  squares_in, parts_in, eps: a norm handed on, as for gi_gemm_bf16_handing (null: none).
GI_API int gi_gemm_bf16_qkv_rope_store(const void* A, const void* W, int M, int N, int K, long lda, long ldw, float* scratch, long scratch_floats,
                                       const float* squares_in, int parts_in, float eps, const float* cos_t, const float* sin_t, const int* pos,
                                       const int* slot, const int* table, int table_stride, void* q_out, void* cache, long page_stride, int page_size,
                                       int n_heads, int n_kv, int hd, unsigned* counters, hipStream_t stream) {
    GI_REQUIRE(M > 0 && N > 0 && K > 0 && n_heads > 0 && n_kv > 0 && hd > 0 && N == (n_heads + 2 * n_kv) * hd,
               "gemm_bf16 (q/k/v): M %d, N %d, K %d, %d heads, %d key/value heads of %d do not fit together", M, N, K, n_heads, n_kv, hd);
    GI_REQUIRE(K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K, "gemm_bf16: K %d and the row strides (%ld, %ld) must be multiples of 8", K, lda, ldw);
    GI_REQUIRE(((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0 && ((uintptr_t)scratch & 15) == 0, "gemm_bf16: operands must be 16-byte aligned");
    GI_REQUIRE(gi_gemm_bf16_qkv_rope_store_takes(M, N, K, hd), "gemm_bf16 (q/k/v): sizes M %d, N %d, K %d, heads of %d are not taken", M, N, K, hd);
    GI_REQUIRE((cos_t == nullptr) == (sin_t == nullptr) && ((uintptr_t)cos_t & 15) == 0 && ((uintptr_t)sin_t & 15) == 0,
               "gemm_bf16 (q/k/v): cos and sin must both be given or both be absent, 16-byte aligned");
    GI_REQUIRE(pos != nullptr && slot != nullptr && table != nullptr && q_out != nullptr && cache != nullptr && page_size > 0 &&
               page_stride >= 2L * n_kv * page_size * hd && ((uintptr_t)q_out & 7) == 0 && ((uintptr_t)cache & 7) == 0 && page_stride % 4 == 0,
               "gemm_bf16 (q/k/v): positions, slots, a table, q_out and a cache with a page stride of at least 2*n_kv*page_size*hd are needed");
    GI_REQUIRE(squares_in == nullptr || (parts_in > 0 && parts_in <= gi_gemm_bf16_qkv_rope_store_max_parts(M, N, K)),
               "gemm_bf16 (q/k/v): %d pieces of a sum of squares, at most %d", parts_in, gi_gemm_bf16_qkv_rope_store_max_parts(M, N, K));
    const RopeStore rope = {cos_t, sin_t, pos, slot, table, table_stride, (bf16_t*)q_out, (bf16_t*)cache, page_stride, page_size, n_heads, n_kv, hd};
    if (M > SKINNY_MAX_ROWS)
        return launch_large(A, W, nullptr, EPI_STORE_F32, M, N, K, lda, ldw, (long)N, scratch, scratch_floats, NormIn{squares_in, parts_in, eps, K}, &rope, stream, NO_NORM_OUT, nullptr,
                            counters);
    return launch_skinny(A, W, nullptr, EPI_STORE_F32, M, N, K, lda, ldw, (long)N, scratch, scratch_floats, NormIn{squares_in, parts_in, eps, K}, NO_NORM_OUT,
                         stream, &rope);
}

// Which kernel makes a product of more than 128 rows whose rows lie whole in memory: 0 the tiles of 128 x 128, 1 those of 256 x 128, 2 those of 256 x 256,
// 3 the first or strips with k shared out over workgroups, 4 strips; -1 for sizes that none of these takes.  kind: 0 stored, 1 added, 2 added with a norm handed on, 3 gated,
// 4 gated with a norm taken, 5 rotated into the pages, 6 through xielu, 7 stored in bfloat16.  With counters, and the scratch it asks for.
GI_API int gi_gemm_bf16_large_kernel(int M, int N, int K, int kind) {
    if (!takes_large(M, N, K) || kind < 0 || kind > 7) return -1;
    if (gi_gemm_bf16_piped_splits(M, N, K) > 1) return 3;
    if (kind == 3 && ends_in_strips(M, N, K)) return 4;
    return large_kernel_of_kind(M, N, K, kind, true).kernel;
}

// Which kernel makes a product of up to 128 rows: 0 slim, 1 slim's tiles of 17 to 32 rows, 2 strips, 3 the weight-streaming one; -1 for more rows.
GI_API int gi_gemm_bf16_small_kernel(int M, int N, int K, int gated) {
    if (M <= 0 || N <= 0 || K <= 0 || M > SKINNY_MAX_ROWS) return -1;
    if (takes_slim(M, N, K, gated != 0)) return 0;
    if (takes_slim_tiles(M, N, K, gated ? EPI_GATED_BF16 : EPI_STORE_F32)) return 1;
    const int splits = gi_gemm_bf16_skinny_splits(N, K);
    return splits == 0 ? ends_in_strips(M, N, K) ? 2 : 3 : shared_strips(M, N, K, splits).tiles ? 2 : 3;
}

// How a product of at most 16 rows that the slim kernel makes reaches rows lda and ldw elements apart (`slim_reach`): weight rows a workgroup, and 100 more where it reckons in 64 bits.
GI_API int gi_gemm_bf16_slim_reach(int M, int N, int K, int gated, int accumulate, long lda, long ldw) {
    if (M <= 0 || M > 16 || N <= 0 || K <= 0) return -1;
    const SlimReach reach = slim_reach(M, N, K, gated ? EPI_GATED_BF16 : accumulate ? EPI_ADD_F32 : EPI_STORE_F32, false, lda, ldw);
    return reach.rows + (reach.far ? 100 : 0);
}

// How strips make a product whose k is shared out: 100 times the tiles of rows and the shares of k (at most 16); 0 where they do not.
GI_API int gi_gemm_bf16_strip_cut(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || (M <= SKINNY_MAX_ROWS ? gi_gemm_bf16_small_kernel(M, N, K, 0) != 2 : !takes_large(M, N, K) || gi_gemm_bf16_piped_splits(M, N, K) == 1)) return 0;
    const StripCut cut = shared_strips(M, N, K, M <= SKINNY_MAX_ROWS ? gi_gemm_bf16_skinny_splits(N, K) : gi_gemm_bf16_piped_splits(M, N, K));
    return 100 * cut.tiles + cut.splits;
}

// The same where the tiles of 256 x 128 make such a product, of whatever kind, with counters.
GI_API int gi_gemm_bf16_tall_shares(int M, int N, int K) {
    return !takes_large(M, N, K) || gi_gemm_bf16_piped_splits(M, N, K) > 1 ? 1 : tall_cut(M, N, K, true, false).shares;
}

// So many 32-bit counters, all 0, are what a product may be given as `counters`; it leaves them 0 again.  Without (null) it makes its own with a launch.  Products
// that may run at the same time must not be given the same.
GI_API int gi_gemm_bf16_counters() { return 2 * gi_compute_units(); }

// Whether gi_gemm_bf16_xielu takes a product of these sizes: up to 16 rows where the kernel for those serves; the rows of prompts
// where all of a tile's k is one workgroup's, with all columns through the activation.
GI_API int gi_gemm_bf16_xielu_takes(int M, int N, int K, int first) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 8 != 0 || first < 0 || first >= N) return 0;
    if (takes_slim(M, N, K, false, true)) return 1;
    return M > SKINNY_MAX_ROWS && first == 0 && K % PK == 0 && N >= 128 && gi_gemm_bf16_piped_splits(M, N, K) == 1;
}

// A product whose columns from `first` on are a feed-forward's that has no gate: they leave through the activation xielu (params: its two
// numbers) as act_out [M, ld_act] in bfloat16, the columns before as 32-bit C [M, ldc] (null where first is 0).  squares_in, parts_in, eps: a
// norm handed on, as for gi_gemm_bf16_handing (null: none; up to 16 rows only).
GI_API int gi_gemm_bf16_xielu(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int first, const float* params, void* act_out,
                              long ld_act, const float* squares_in, int parts_in, float eps, hipStream_t stream) {
    GI_REQUIRE((M + 63) / 64 <= 65535, "gemm_bf16: M %d is too large", M);
    GI_REQUIRE(gi_gemm_bf16_xielu_takes(M, N, K, first), "gemm_bf16 (xielu): sizes M %d, N %d, K %d with %d columns as they are are not taken", M, N, K, first);
    GI_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K && ((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0,
               "gemm_bf16 (xielu): rows must be 16-byte aligned (strides %ld, %ld)", lda, ldw);
    GI_REQUIRE(params != nullptr && act_out != nullptr && ld_act >= N - first && (first == 0 || (C != nullptr && ldc >= first)), "gemm_bf16 (xielu): outputs or parameters are missing");
    const bool slim = takes_slim(M, N, K, false, true);
    GI_REQUIRE(squares_in == nullptr || (slim && parts_in > 0 && parts_in <= slim_max_parts(M)), "gemm_bf16 (xielu): %d pieces of a sum of squares are not taken", parts_in);
    NormIn in = {squares_in, parts_in, eps, K, 0.f};
    in.first = first;
    if (slim) return launch_slim(A, W, C, EPI_XIELU, M, N, K, lda, ldw, ldc, in, NormOut{params, (bf16_t*)act_out, ld_act, nullptr}, stream);
    return launch_large(A, W, act_out, EPI_XIELU, M, N, K, lda, ldw, ld_act, nullptr, 0, NO_NORM_IN, nullptr, stream, NormOut{params, nullptr, 0, nullptr});
}

// `gated` != 0: W is [gate; up] interleaved in groups of 16 rows (N rows in all, a multiple of 32)
// and C is bfloat16 [M, N/2] = silu(gate) * up.
GI_API int gi_gemm_bf16(const void* A, const void* W, void* C, int c_dtype, int accumulate, int gated, float gate_limit, int M, int N, int K, long lda,
                        long ldw, long ldc, float* scratch, long scratch_floats, unsigned* counters, hipStream_t stream) {
    GI_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_bf16: M %d, N %d, K %d must be positive", M, N, K);
    GI_REQUIRE(K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0, "gemm_bf16: K %d and the row strides (%ld, %ld) must be multiples of 8", K, lda, ldw);
    GI_REQUIRE(((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_bf16: operands must be 16-byte aligned");
    GI_REQUIRE(lda >= K && ldw >= K && ldc >= (gated ? N / 2 : N), "gemm_bf16: leading dimensions too small");
    int epi = epilogue_of(c_dtype, accumulate);
    if (gated) {
        GI_REQUIRE(N % 32 == 0 && c_dtype == GI_BF16 && !accumulate, "gemm_bf16: the gated product needs N %% 32 == 0 and a bfloat16 output");
        epi = gated == 3 ? EPI_GATED_CLAMP_BF16 : gated == 2 ? EPI_GATED_GELU_BF16 : EPI_GATED_BF16;
    }
    GI_REQUIRE(epi >= 0, "gemm_bf16: output dtype %d with accumulate %d is not supported", c_dtype, accumulate);

    const NormIn plain_in = {nullptr, 0, 0.f, 1, gate_limit};          // no norm to finish; the clamped gate's limit
    if (takes_slim(M, N, K, gated != 0)) return launch_slim(A, W, C, epi, M, N, K, lda, ldw, ldc, plain_in, NO_NORM_OUT, stream);

    if (takes_slim_tiles(M, N, K, epi)) return launch_slim_tiles(A, W, C, epi, M, N, K, lda, ldw, ldc, plain_in, NO_NORM_OUT, stream);
    if (M <= SKINNY_MAX_ROWS) return launch_skinny(A, W, C, epi, M, N, K, lda, ldw, ldc, scratch, scratch_floats, plain_in, NO_NORM_OUT, stream);

    GI_REQUIRE((M + 63) / 64 <= 65535, "gemm_bf16: M %d is too large", M);
    if (K % PK == 0 && N >= 128) return launch_large(A, W, C, epi, M, N, K, lda, ldw, ldc, scratch, scratch_floats, plain_in, nullptr, stream, NO_NORM_OUT, nullptr, counters);
#define TILED(BM_, EPI_) gemm_bf16_tiled_kernel<BM_, EPI_><<<grid, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, gate_limit)
    if ((long)((M + 127) / 128) * ((N + BN - 1) / BN) < 512) {   // few tiles: smaller ones fill more of the chip
        dim3 grid((N + BN - 1) / BN, (M + 63) / 64);
        if (epi == EPI_STORE_F32) TILED(64, EPI_STORE_F32); else if (epi == EPI_ADD_F32) TILED(64, EPI_ADD_F32);
        else if (epi == EPI_STORE_BF16) TILED(64, EPI_STORE_BF16); else if (epi == EPI_GATED_BF16) TILED(64, EPI_GATED_BF16); else if (epi == EPI_GATED_GELU_BF16) TILED(64, EPI_GATED_GELU_BF16); else TILED(64, EPI_GATED_CLAMP_BF16);
    } else {
        dim3 grid((N + BN - 1) / BN, (M + 127) / 128);
        if (epi == EPI_STORE_F32) TILED(128, EPI_STORE_F32); else if (epi == EPI_ADD_F32) TILED(128, EPI_ADD_F32);
        else if (epi == EPI_STORE_BF16) TILED(128, EPI_STORE_BF16); else if (epi == EPI_GATED_BF16) TILED(128, EPI_GATED_BF16); else if (epi == EPI_GATED_GELU_BF16) TILED(128, EPI_GATED_GELU_BF16); else TILED(128, EPI_GATED_CLAMP_BF16);
    }
#undef TILED
    GI_CHECK_LAUNCH("gemm_bf16 (tiled)");
    return 0;
}

// C[rows of tile t] = A[rows of tile t] * W[tile_group[t]]^T for every tile t of 128 rows of A that is in use (see the kernel).  M rows
// of A and C exist (a multiple of 128); W is [groups][N][K].  Output: float32 stored, bfloat16 stored, or the gated form.
GI_API int gi_gemm_bf16_grouped(const void* A, const void* W, void* C, int c_dtype, int gated, float gate_limit, int M, int N, int K, long lda, long ldw, long ldc,
                                const int* tile_group, long group_stride, hipStream_t stream) {
    GI_REQUIRE(M > 0 && M % 128 == 0 && N >= 128 && K > 0 && K % PK == 0 && lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K && ldc >= (gated ? N / 2 : N)
               && group_stride % 8 == 0 && M / 128 <= 65535,
               "gemm_bf16_grouped: M %d (a multiple of 128), N %d (128 or more), K %d (a multiple of %d) or the strides do not fit", M, N, K, PK);
    GI_REQUIRE(((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_bf16_grouped: operands must be 16-byte aligned");
    int epi = epilogue_of(c_dtype, 0);
    if (gated) {
        GI_REQUIRE(N % 32 == 0 && c_dtype == GI_BF16, "gemm_bf16_grouped: the gated product needs N %% 32 == 0 and a bfloat16 output");
        epi = gated == 3 ? EPI_GATED_CLAMP_BF16 : gated == 2 ? EPI_GATED_GELU_BF16 : EPI_GATED_BF16;
    }
    GI_REQUIRE(epi >= 0, "gemm_bf16_grouped: output dtype %d is not supported", c_dtype);
    constexpr int bytes = 2 * 256 * 128;
    dim3 grid((N + 127) / 128, M / 128);
#define GROUPED(EPI_)                                                                                                                               \
    do {                                                                                                                                            \
        static bool raised = false;                                                                                                                 \
        if (!raised) {                                                                                                                              \
            if (hipFuncSetAttribute((const void*)gemm_bf16_grouped_kernel<EPI_>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) \
                return gi_fail("gemm_bf16_grouped: cannot reserve %d bytes of LDS", bytes);                                                         \
            raised = true;                                                                                                                          \
        }                                                                                                                                           \
        gemm_bf16_grouped_kernel<EPI_><<<grid, 256, bytes, stream>>>((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldw, ldc, tile_group, group_stride, gate_limit); \
    } while (0)
    if (epi == EPI_STORE_F32) GROUPED(EPI_STORE_F32);
    else if (epi == EPI_STORE_BF16) GROUPED(EPI_STORE_BF16);
    else if (epi == EPI_GATED_BF16) GROUPED(EPI_GATED_BF16);
    else if (epi == EPI_GATED_GELU_BF16) GROUPED(EPI_GATED_GELU_BF16);
    else GROUPED(EPI_GATED_CLAMP_BF16);
#undef GROUPED
    GI_CHECK_LAUNCH("gemm_bf16 (grouped)");
    return 0;
}
