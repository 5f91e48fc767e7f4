// C[m, n] (=|+=) sum_k A[m, k] * W[n, k] in true 32-bit arithmetic.
//
// Both operands are row-major with k contiguous (activations [M, K], weights [N, K] as checkpoints
// store them); operands may be stored as bfloat16 and are widened exactly.  This is the 32-bit path of
// every matrix product, and the slow stand-in of the bfloat16 path for shapes the matrix-core kernels refuse.
//
// The order of a sum depends on K alone, never on M, the row's place in the batch or the kernel that serves it, so a row computed
// alone has the same bits as the same row inside a large batch (the reference keeps the same rule, src/gpu/device_kernels.inc:97-100):
//   * k is cut into 8 ranges of L = 32 * ceil(K / 256) (the last ones shorter or empty);
//   * a range's sum is one chain of 16x16x4 32-bit matrix instructions from zero, 16 of k after 16 of k, the four instructions of
//     such a block taking k0 + 4g + j (g = 0..3 inside the instruction) for j = 0, 1, 2, 3; what lies beyond K counts as zero;
//   * the ranges' sums are added as a tree, ((s0 + s1) + (s2 + s3)) + ((s4 + s5) + (s6 + s7)); what C held is added last.
// The tree is what lets a product of a few rows be shared out over the chip (a chain over all of K leaves one lane or wave per column
// walking K alone) and what one with few tiles is cut along; its error is smaller than the single chain's.
#include "common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int RANGES = 8;
__host__ __device__ constexpr int range_length(int K) { return 32 * ((K + 32 * RANGES - 1) / (32 * RANGES)); }

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// four consecutive elements, widened
__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 load4(const bf16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
}

// The sum of range q joins the tree: t[0..2] hold the finished left halves; what is finished so far comes back.
template <int N>
__device__ __forceinline__ void fold(int q, f32x4 (&acc)[N], f32x4 (&t)[3][N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (!(q & 1)) { t[0][i] = acc[i]; continue; }
        acc[i] = t[0][i] + acc[i];
        if (!(q & 2)) { t[1][i] = acc[i]; continue; }
        acc[i] = t[1][i] + acc[i];
        if (!(q & 4)) { t[2][i] = acc[i]; continue; }
        acc[i] = t[2][i] + acc[i];
    }
}

// ... where the ranges behind the first n have nothing of k in them: the tree's open branches are closed (their other halves are zeros).
template <int N>
__device__ __forceinline__ void close(int n, f32x4 (&acc)[N], const f32x4 (&t)[3][N]) {
#pragma unroll
    for (int b = 1; b < 3; ++b) {
        if (!(n >> b & 1) || (n & ((1 << b) - 1)) == 0) continue;
#pragma unroll
        for (int i = 0; i < N; ++i) acc[i] = t[b][i] + acc[i];
    }
}

template <typename TC, bool ACCUMULATE>
__device__ __forceinline__ void put(TC* C, size_t o, float v) {
    if constexpr (ACCUMULATE) store_f32(C, o, load_f32(C, o) + v);
    else store_f32(C, o, v);
}

// ------------------------------------------------------------------------------------------ many rows
// A workgroup of four waves makes a tile of BM rows x 64 columns, both operands staged through LDS 32 of k at a time (two stages,
// the next one's loads in flight in registers meanwhile).  Bound by the matrix cores (256 flop a clock and compute unit in 32-bit,
// a sixteenth of bfloat16's): a wave's tile of 32 x 32 (BM 64) needs 4 KB of LDS for 512 clocks of matrix instructions, so what
// counts is enough workgroups a compute unit to cover the loads' latency and no compute unit left idle; hence small tiles and, where the
// tiles are few, the eight ranges of k shared out over `splits` workgroups (each finishes its part of the tree and leaves it in
// `part`, a second kernel adds the parts).  The ring kernel below reaches 123 TFLOP/s of the 154 that a bare loop of these instructions
// makes (600 rows of 128,256 x 2,048; tiles of 64 x 128, 128 x 64 and 128 x 128 reach no more; 110 before a stage had almost no vector
// instructions of its own); the kernel of single fused multiply-adds
// that stood here before made 19 at 301 rows of the Llama-3.2-1B shape, where this one makes 70 to 120.
constexpr int BN = 64, BK = 32;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// LDS: rows of 32 floats; the eight 16-byte chunks of a row are permuted by the row so that 16 rows' reads of one chunk meet 16 different places
__device__ __forceinline__ int chunk_at(int row, int c) { return row * BK + ((c ^ ((row >> 1) & 7)) << 2); }

// a lane's four results of a tile of 16 x 16 are four neighbouring columns of one row
template <int TM, int TN, typename TC, bool ACCUMULATE>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[TN * TM], TC* C, float* part, int m_first, int n_first, int z, int M, int N, long ldc) {
    const bool whole_rows = part ? (N & 3) == 0 : sizeof(TC) == 4 && (ldc & 3) == 0 && ((uintptr_t)C & 15) == 0;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m_first + i * 16;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n_first + j * 16;
            const f32x4 v = acc[j * TM + i];
            if (whole_rows && n + 3 < N) {
                f32x4* to = reinterpret_cast<f32x4*>(part ? part + ((size_t)z * M + m) * N + n : (float*)C + (size_t)m * ldc + n);
                *to = ACCUMULATE && !part ? *to + v : v;
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (n + e >= N) break;
                if (part) part[((size_t)z * M + m) * N + n + e] = v[e];
                else put<TC, ACCUMULATE>(C, (size_t)m * ldc + n + e, v[e]);
            }
        }
    }
}

// VECTOR: K and the leading dimensions are multiples of 4 and the bases aligned to 4 elements
template <bool VECTOR, typename T>
__device__ __forceinline__ f32x4 fetch(const T* base, long ld, int row, int rows, int k, int K) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    const T* p = base + (size_t)min(row, rows - 1) * ld;
    if constexpr (VECTOR) {
        v = load4(p + min(k, K - 4));
        if (k >= K) v = f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
        // (asked for by every lane, wherever K ends: a load under a condition is waited for before the next)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = load_f32(p, (size_t)min(k + i, K - 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = k + i < K ? v[i] : 0.f;
    }
    return v;
}

template <int BM, bool VECTOR, typename TA, typename TW, typename TC, bool ACCUMULATE>
__global__ __launch_bounds__(256) void gemm_exact_tiled_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, float* __restrict__ part,
                                                               int M, int N, int K, long lda, long ldw, long ldc, int m_tiles, int n_tiles, int splits) {
    constexpr int WAVES_M = BM / 32, WAVES_N = 4 / WAVES_M, TN = BN / WAVES_N / 16, TM = 2;        // a wave: 32 rows x 64 / WAVES_N columns
    constexpr int LOADS_A = BM * BK / 4 / 256, LOADS_W = BN * BK / 4 / 256;
    __shared__ float lds[2][(BM + BN) * BK];
    // the tiles of one strip of weights follow each other on one die (workgroups go to the eight dies in turn), whose L2 then reads the strip once
    const int total = m_tiles * n_tiles * splits, each = (total + 7) / 8, u = (blockIdx.x & 7) * each + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= each || u >= total) return;
    const int m0 = (u % m_tiles) * BM, n0 = (u / m_tiles % n_tiles) * BN, z = u / (m_tiles * n_tiles);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    const int wm = (wave % WAVES_M) * 32, wn = (wave / WAVES_M) * (BN / WAVES_N);

    const int stages_all = (K + BK - 1) / BK, per_range = range_length(K) / BK;
    const int q0 = z * (RANGES / splits), q1 = q0 + RANGES / splits;
    const int s_end = min(q1 * per_range, stages_all);
    f32x4 next_a[LOADS_A], next_w[LOADS_W];
    auto ask = [&](int s) {
#pragma unroll
        for (int i = 0; i < LOADS_A; ++i) { const int e = tid + 256 * i; next_a[i] = fetch<VECTOR>(A, lda, m0 + (e >> 3), M, s * BK + (e & 7) * 4, K); }
#pragma unroll
        for (int i = 0; i < LOADS_W; ++i) { const int e = tid + 256 * i; next_w[i] = fetch<VECTOR>(W, ldw, n0 + (e >> 3), N, s * BK + (e & 7) * 4, K); }
    };
    auto lay = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LOADS_A; ++i) { const int e = tid + 256 * i; *reinterpret_cast<f32x4*>(&lds[buf][chunk_at(e >> 3, e & 7)]) = next_a[i]; }
#pragma unroll
        for (int i = 0; i < LOADS_W; ++i) { const int e = tid + 256 * i; *reinterpret_cast<f32x4*>(&lds[buf][BM * BK + chunk_at(e >> 3, e & 7)]) = next_w[i]; }
    };

    f32x4 acc[TN * TM], t[3][TN * TM];
    int s = q0 * per_range;
    if (s < s_end) { ask(s); lay(s & 1); }
    __syncthreads();
    const int q_end = max(q0, min(q1, (s_end + per_range - 1) / per_range));              // (short k leaves ranges empty)
#pragma unroll
    for (int i = 0; i < TN * TM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int q = q0; q < q_end; ++q) {
#pragma unroll
        for (int i = 0; i < TN * TM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int stop = min((q + 1) * per_range, s_end);
        for (; s < stop; ++s) {
            const bool more = s + 1 < s_end;
            if (more) ask(s + 1);
            const float *as = lds[s & 1], *ws = as + BM * BK;
#pragma unroll
            for (int b = 0; b < BK / 16; ++b) {
                f32x4 a[TM], w[TN];
#pragma unroll
                for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const f32x4*>(&as[chunk_at(wm + i * 16 + r, b * 4 + g)]);
#pragma unroll
                for (int j = 0; j < TN; ++j) w[j] = *reinterpret_cast<const f32x4*>(&ws[chunk_at(wn + j * 16 + r, b * 4 + g)]);
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int i = 0; i < TM; ++i) acc[j * TM + i] = mfma(w[j][kk], a[i][kk], acc[j * TM + i]);
            }
            if (more) lay((s + 1) & 1);
            __syncthreads();
        }
        fold(q - q0, acc, t);              // (the workgroup's ranges are a whole branch of the tree)
    }
    close(q_end - q0, acc, t);
    store_tile<TM, TN, TC, ACCUMULATE>(acc, C, part, m0 + wm + r, n0 + wn + 4 * g, z, M, N, ldc);
}

// The same for 32-bit operands whose rows are whole blocks of 32 k: the operands go from memory straight into LDS, a ring of three
// stages with two in flight while one is multiplied (asked for and waited for as the bfloat16 ring kernel does), so a stage costs a
// wave four loads and a barrier beside its matrix instructions.
// What bounds it is how much of a wave's time the matrix instructions do not fill, wherever a compute unit has fewer than three workgroups.  So a half of a
// stage is read from LDS while the half before it is multiplied, and the barrier that hands the next stage over lies between a stage's halves: behind it a wave
// has 16 matrix instructions whose operands are in registers, under which the next stage's loads go out and its first half is read.  With reads, barrier
// and loads at the beginning of a stage, ahead of its products, 301 rows of 16,384 x 2,048 (five tiles a unit: three together, then two) took 200 us,
// 177 now, of 2,048 x 8,192 112 and 101, 600 of 2,048 x 2,048 59 and 55; where three workgroups share a unit all the time it makes no difference (600 rows
// of 16,384 x 2,048 331 and 328, 120 to 133 TFLOP/s).  Two stages (five workgroups fit the LDS, but not the registers) or four are no faster.
template <int BM, bool ACCUMULATE>
__global__ __launch_bounds__(256) void gemm_exact_ring_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, float* __restrict__ part,
                                                             int M, int N, int K, long lda, long ldw, long ldc, int m_tiles, int n_tiles, int splits) {
    constexpr int WAVES_M = BM / 32, WAVES_N = 4 / WAVES_M, TN = BN / WAVES_N / 16, TM = 2, STAGES = 3;
    constexpr int ROWS = BM + BN, LOADS = ROWS / 32;                       // a wave's loads a stage, each 8 rows of 128 bytes
    __shared__ __attribute__((aligned(16))) float ring[STAGES * ROWS * BK];
    const int total = m_tiles * n_tiles * splits, each = (total + 7) / 8, u = (blockIdx.x & 7) * each + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= each || u >= total) return;
    const int m0 = (u % m_tiles) * BM, n0 = (u / m_tiles % n_tiles) * BN, z = u / (m_tiles * n_tiles);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int wm = (wave % WAVES_M) * 32, wn = (wave / WAVES_M) * (BN / WAVES_N);
    const int per_range = range_length(K) / BK, q0 = z * (RANGES / splits), q1 = q0 + RANGES / splits;
    const int s_begin = q0 * per_range, s_end = max(s_begin, min(q1 * per_range, K / BK));

    // Vector instructions take the matrix instructions' place, so a stage has hardly any: a load's address is a scalar base (the tile's
    // first row, advanced by the stage's k) plus an offset that stays, an LDS read's one of four registers plus a constant.
    // LDS is filled in order, so a lane chooses the chunk that belongs at its place.
    const float *a_tile = A + (size_t)m0 * lda, *w_tile = W + (size_t)n0 * ldw;
    unsigned src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        src[i] = (unsigned)((row < BM ? min(row, M - 1 - m0) * lda : min(row - BM, N - 1 - n0) * ldw) + 4 * c) * 4;
    }
    const unsigned ring_base = (unsigned)(size_t)(lds_ptr_t)ring;
    // (written as assembly so that the compiler does not wait for them; the counted wait and the barrier below order them against the reads)
    auto issue = [&](int s, int slot) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const unsigned dst = ring_base + (slot * ROWS + (wave * LOADS + i) * 8) * BK * 4;
            const float* base = ((wave * LOADS + i) * 8 < BM ? a_tile : w_tile) + s * BK;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(src[i]), "s"(base) : "memory", "m0");
        }
    };
    f32x4 acc[TN * TM], t[3][TN * TM];
#pragma unroll
    for (int i = 0; i < STAGES; ++i)
        if (s_begin + i < s_end) issue(s_begin + i, i);
    const int a_at[2] = {chunk_at(wm + r, g), chunk_at(wm + r, 4 + g)}, w_at[2] = {BM * BK + chunk_at(wn + r, g), BM * BK + chunk_at(wn + r, 4 + g)};
    f32x4 a[2][TM], w[2][TN];
    auto read_half = [&](int slot, int b) {                 // (rows 16 apart have the same permutation of chunks)
        const float* stage = ring + slot * ROWS * BK;
#pragma unroll
        for (int i = 0; i < TM; ++i) a[b][i] = *reinterpret_cast<const f32x4*>(stage + a_at[b] + i * 16 * BK);
#pragma unroll
        for (int j = 0; j < TN; ++j) w[b][j] = *reinterpret_cast<const f32x4*>(stage + w_at[b] + j * 16 * BK);
    };
    auto multiply_half = [&](int b) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) acc[j * TM + i] = mfma(w[b][j][kk], a[b][i][kk], acc[j * TM + i]);
    };
    int s = s_begin, slot = 0;
    if (s < s_end) {
        const int behind = min(s_end - s, STAGES) - 1;      // stages asked for behind the first
        if (behind == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else if (behind == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read_half(0, 0);
    }
    const int q_end = max(q0, min(q1, (s_end + per_range - 1) / per_range));              // (short k leaves ranges empty)
#pragma unroll
    for (int i = 0; i < TN * TM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int q = q0; q < q_end; ++q) {
#pragma unroll
        for (int i = 0; i < TN * TM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < TN * TM; ++i) asm volatile("" : "+v"(acc[i]));        // (four zeros, not one in four places: the compiler else moves the sums about in every stage)
        const int stop = min((q + 1) * per_range, s_end);
        for (; s < stop; ++s) {
            read_half(slot, 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply_half(0);
            __builtin_amdgcn_sched_barrier(0);
            const int here = slot;
            slot = slot + 1 == STAGES ? 0 : slot + 1;
            __builtin_amdgcn_s_waitcnt(0xc07f);                // lgkmcnt(0), in a form that the compiler counts with: this wave's reads of stage s are done
            if (s + 1 < s_end) {
                if (s + 2 < s_end) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");        // its part of stage s + 1 has landed
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();                                                  // everyone's
                asm volatile("" ::: "memory");
                read_half(slot, 0);
                if (s + STAGES < s_end) issue(s + STAGES, here);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply_half(1);
        }
        fold(q - q0, acc, t);
    }
    close(q_end - q0, acc, t);
    store_tile<TM, TN, float, ACCUMULATE>(acc, C, part, m0 + wm + r, n0 + wn + 4 * g, z, M, N, ldc);
}

// The parts of the tree that `splits` workgroups left, added up: splits is 2, 4 or 8, a part's neighbours in the tree its neighbours here.
template <typename TC, bool ACCUMULATE>
__global__ __launch_bounds__(256) void gemm_exact_add_parts_kernel(const float* __restrict__ part, TC* __restrict__ C, int M, int N, long ldc, int splits) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x, plane = (size_t)M * N;
    if (e >= plane) return;
    float v[RANGES];
#pragma unroll
    for (int z = 0; z < RANGES; ++z) v[z] = z < splits ? part[z * plane + e] : 0.f;
    for (int n = splits; n > 1; n >>= 1) {
#pragma unroll
        for (int z = 0; z < RANGES / 2; ++z)
            if (z < n / 2) v[z] = v[2 * z] + v[2 * z + 1];
    }
    put<TC, ACCUMULATE>(C, (e / N) * ldc + e % N, v[0]);
}

// ------------------------------------------------------------------------------------------- few rows
// Up to 16 rows (decoding): bound by reading the weights once.  A workgroup owns a strip of weight rows and all of k, a wave one
// range of k (strips of 16 rows, 8 waves) or two (strips of 8 rows and at most 8 rows of activations, 4 waves: the idle half of
// every matrix instruction takes the second range, weight rows 8..15 and activation rows 8..15 of the instruction standing for the
// same rows at the other range's k; twice the workgroups for the same waves, which is what narrow outputs lack).  The operands go
// from memory straight into the matrix instructions' registers: 32-bit weights a whole cache line of 8 rows a load, past the caches, four pairs of blocks of 16 k
// in flight behind the products (with 16 rows' 64 bytes a load, eight blocks asked for at once and all awaited: the figures before); bfloat16 weights AHEAD blocks at once.
// The ranges' sums meet in LDS and are added there.  At 3 rows, before and now, in chains of products with weights of their own: 16,384 x 2,048 gated 28.4, 26.6 us (5.0 TB/s), 2,048 x 8,192
// added 17.4, 15.4 (4.35; a bare read of these places 13.0), 2,048 x 2,048 added 7.4, 6.2, 3,072 x 2,048 8.8, 8.4, 128,256 x 2,048 184, 178 (5.9); what is added onto is
// asked for first (a microsecond of the added ones); one lane per column, each walking all of k alone, took 290 us, 1.15 ms and 400 us.
constexpr int FEW_ROWS = 16, AHEAD = 8;

// GATED: W is [gate; up], a strip of 16 is 8 gates and the 8 ups of the same columns, and act(gate) * up goes out in the bits of the gate's own kernel, which
// read both again (3 rows of 16,384 x 2,048: 27.4 us and 5 for the gate, 27.4 in one).  The norm of the rows was tried here too (every workgroup working the rows'
// factors out for itself while its first weights are on their way, in the bits of the norm's kernel): 1,024 workgroups that each read all rows once more took 39 us
// for 27.4 and the norm's 5, 3,072 x 2,048 13 for 8.6 and 5.  Not kept.
struct Plain { static constexpr int KIND = 0; };
struct Gate { static constexpr int KIND = 1; int act; float limit; };
// Turn: the product is an attention layer's q/k/v, a strip of 8 is four channels of a head's first half and the four they are turned with, and queries and keys
// leave turned, keys and values into the pages (rope_store_kernel's places and bits; 3 rows of 3,072 x 2,048: 8.6 us and 5 for that
// launch, 10.5 in one).
struct Turn {
    static constexpr int KIND = 2;
    const float *cos_t, *sin_t;                // [M, hd / 2], null: not turned
    const int *pos, *slot, *table;
    int table_stride;
    float *q_out, *cache;
    long page_stride;
    int page_size, n_heads, n_kv, hd;
};

__device__ __forceinline__ f32x4 load4_once(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p)); }      // of bytes that this launch reads no second time
// Lane l of either load holds row l % 8 and the 4 k from 4 (l / 16) + 16 (l / 8 % 2) on (`low`: rows 0 to 7, `high`: 8 to 15); afterwards row l % 16 and the 4 k from 4 (l / 16)
// on (`low`) and those 16 further (`high`): within 16 lanes the upper half of `low` and the lower half of `high` change places.
__device__ __forceinline__ void rows_of_halves(f32x4& low, f32x4& high) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = __float_as_int(low[i]), b = __float_as_int(high[i]);
        low[i] = __int_as_float(__builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false));         // (rotated by 8 within 16 lanes; lanes 8 to 15 take it)
        high[i] = __int_as_float(__builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false));        // (lanes 0 to 7)
    }
}

template <int STRIP, typename TA, typename TW, typename TC, bool ACCUMULATE, typename End>
__global__ __launch_bounds__(STRIP == 16 ? 512 : 256) void gemm_exact_few_rows_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C,
                                                                                      int M, int N, int K, long lda, long ldw, long ldc, End end) {
    constexpr bool GATED = End::KIND == 1, TURNED = End::KIND == 2;
    static_assert(!GATED || STRIP == 16, "a strip of gates and ups");
    static_assert(!TURNED || STRIP == 8, "a strip of pairs");
    __shared__ f32x4 sums[RANGES][STRIP == 16 ? 64 : 16];                 // per range: [group of 4 columns][row]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (GATED ? 8 : STRIP), L = range_length(K), inter = N / 2;
    const int q = STRIP == 16 ? wave : 2 * wave + (r >> 3), row = STRIP == 16 ? r : r & 7;
    const int q_last = STRIP == 16 ? wave : 2 * wave + 1, q_first = STRIP == 16 ? wave : 2 * wave;       // of the wave
    const int base = q * L + 4 * g;
    int first_row = GATED ? min(n0 + (row & 7), inter - 1) + (row >> 3) * inter : min(n0 + row, N - 1);
    f32x4 cs = f32x4{1.f, 1.f, 1.f, 1.f}, sn = f32x4{0.f, 0.f, 0.f, 0.f};
    int head = 0, channel = 0, place = 0;
    long page = 0;
    if constexpr (TURNED) {
        const int strips = end.hd / 8, half = end.hd / 2;       // of a head
        head = blockIdx.x / strips;
        channel = (blockIdx.x % strips) * 4;
        first_row = head * end.hd + channel + (row & 3) + (row >> 2) * half;
        if (threadIdx.x < 16 && (threadIdx.x & 7) < M) {        // what the end needs of row threadIdx.x % 8, on its way while the products run
            const int m = threadIdx.x & 7;
            if (end.cos_t != nullptr) {
                cs = load4(end.cos_t + (size_t)m * half + channel);
                sn = load4(end.sin_t + (size_t)m * half + channel);
            }
            if (head >= end.n_heads) {
                const int p = end.pos[m];
                page = end.table[(size_t)end.slot[m] * end.table_stride + p / end.page_size];
                place = p % end.page_size;
            }
        }
    }
    const TW* w_row = W + (size_t)first_row * ldw;
    const TA* a_row = A + (size_t)min(row, M - 1) * lda;
    // What the sums are added onto is asked for first: behind the weights it would be one more round trip.
    [[maybe_unused]] f32x4 old;
    if constexpr (ACCUMULATE) {
        const int e = threadIdx.x % (STRIP * STRIP / 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) old[i] = load_f32(C, (size_t)min(e % STRIP, M - 1) * ldc + min(n0 + 4 * (e / STRIP) + i, N - 1));
    }
    const int blocks = max(0, min(L, K - q_first * L) + 15) / 16;             // until both of the wave's ranges are through
    const int guarded = max(0, min(L, K - q_last * L)) / 16;                  // ... of them with nothing to guard
    f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
    int whole;
    if constexpr (sizeof(TW) == 4) {
        // 32-bit weights: a load brings 32 k of 8 rows, a whole cache line of each, past the caches; two of them hold two blocks of 16 rows' (or 8 rows' in both
        // ranges) operands, whose halves then change places.  DEPTH such pairs are in flight.
        constexpr int DEPTH = 4;
        const int w_k = 4 * (g + 4 * (r >> 3)), low_row = __shfl(first_row, r & 7, 64), high_row = STRIP == 16 ? __shfl(first_row, 8 + (r & 7), 64) : low_row;
        const float *w_low = W + (size_t)low_row * ldw + q_first * L + w_k, *w_high = W + (size_t)high_row * ldw + q_last * L + w_k;
        const int pairs = guarded / 2;
        whole = 2 * pairs;
        f32x4 w[DEPTH][2], a[DEPTH][2];
        auto fetch = [&](int i, int d) __attribute__((always_inline)) {
            w[d][0] = load4_once(w_low + 32 * i);
            w[d][1] = load4_once(w_high + 32 * i);
            a[d][0] = load4(a_row + base + 32 * i);
            a[d][1] = load4(a_row + base + 32 * i + 16);
        };
        auto products = [&](int d) __attribute__((always_inline)) {
            rows_of_halves(w[d][0], w[d][1]);
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) acc[0] = mfma(w[d][half][kk], a[d][half][kk], acc[0]);
        };
        if (__builtin_expect(pairs >= DEPTH, 1)) {                            // nothing is skipped in a trip: a pair's products wait for that pair alone
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) fetch(d, d);
            int i = 0;
            for (; i + 2 * DEPTH <= pairs; i += DEPTH) {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) {
                    products(d);
                    fetch(i + DEPTH + d, d);
                }
            }
            const int rest = pairs - i - DEPTH;                               // not asked for yet, fewer than DEPTH
            if (__builtin_expect(rest > 0, 0)) {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) {
                    products(d);
                    if (d < rest) fetch(i + DEPTH + d, d);
                }
#pragma unroll
                for (int d = 0; d < DEPTH - 1; ++d)
                    if (d < rest) products(d);
            } else {
#pragma unroll
                for (int d = 0; d < DEPTH; ++d) products(d);
            }
        } else {
#pragma unroll
            for (int d = 0; d < DEPTH - 1; ++d)
                if (d < pairs) fetch(d, d);
#pragma unroll
            for (int d = 0; d < DEPTH - 1; ++d)
                if (d < pairs) products(d);
        }
    } else {
        whole = guarded / AHEAD * AHEAD;                                      // in groups
        for (int b = 0; b < whole; b += AHEAD) {
            f32x4 w[AHEAD], a[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) w[i] = load4(w_row + base + (b + i) * 16);
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) a[i] = load4(a_row + base + (b + i) * 16);
            __builtin_amdgcn_sched_barrier(0);                     // all of them in flight before the first product
#pragma unroll
            for (int i = 0; i < AHEAD; ++i)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) acc[0] = mfma(w[i][kk], a[i][kk], acc[0]);
        }
    }
    for (int b = whole; b < blocks; ++b) {
        const int k = base + b * 16, at = min(k, K - 4);
        f32x4 w = load4(w_row + at), a = load4(a_row + at);
        if (k >= K) w = a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) acc[0] = mfma(w[kk], a[kk], acc[0]);
    }
    if constexpr (STRIP == 16) sums[q][g * 16 + r] = acc[0];
    else if ((g >> 1) == (r >> 3)) sums[q][(g & 1) * 8 + (r & 7)] = acc[0];     // (the instruction's other two quarters mix the ranges)
    __syncthreads();
    const int e = threadIdx.x;
    if (e >= STRIP * STRIP / 4) return;
    const int m = e % STRIP, n = n0 + 4 * (e / STRIP);
    if (!GATED && !TURNED && m >= M) return;
    f32x4 v[RANGES];
#pragma unroll
    for (int z = 0; z < RANGES; ++z) v[z] = sums[z][e];
    const f32x4 sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    if constexpr (GATED) {                                      // lanes 0 .. 31 hold gates, the lane 32 further the ups of the same columns and row
        f32x4 up;
#pragma unroll
        for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(sum[i], 32, 64);
        if (e >= 32 || m >= M) return;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < inter) store_f32(C, (size_t)m * ldc + n + i, gated_act(sum[i], up[i], end.act, end.limit));
    } else if constexpr (TURNED) {                              // threads 0 .. 7 hold the first halves' channels of their row, the thread 8 further those they are turned with
        f32x4 other;
#pragma unroll
        for (int i = 0; i < 4; ++i) other[i] = __shfl_xor(sum[i], 8, 64);
        if (m >= M) return;
        const bool second = e >= 8;
        const int at = channel + (second ? end.hd / 2 : 0);
        f32x4 turned;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a = second ? other[i] : sum[i], b = second ? sum[i] : other[i];
            turned[i] = second ? fmaf(a, sn[i], b * cs[i]) : fmaf(a, cs[i], -(b * sn[i]));      // (rounded where rope_store_kernel's a sin + b cos and a cos - b sin are)
        }
        if (head < end.n_heads) {
            *reinterpret_cast<f32x4*>(end.q_out + ((size_t)m * end.n_heads + head) * end.hd + at) = turned;
            return;
        }
        float* keys = end.cache + page * end.page_stride;
        const int kv = head - end.n_heads;
        if (kv < end.n_kv) {
            *reinterpret_cast<f32x4*>(keys + ((size_t)kv * end.page_size + place) * end.hd + at) = turned;
            return;
        }
        float* values = keys + (size_t)end.n_kv * end.page_size * end.hd + ((size_t)(kv - end.n_kv) * end.hd + at) * end.page_size + place;
#pragma unroll
        for (int i = 0; i < 4; ++i) values[(size_t)i * end.page_size] = sum[i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (n + i >= N) continue;
            if constexpr (ACCUMULATE) store_f32(C, (size_t)m * ldc + n + i, old[i] + sum[i]);
            else store_f32(C, (size_t)m * ldc + n + i, sum[i]);
        }
    }
}

// ------------------------------------------------------------------------------------------- dispatch
// Which products of up to 16 rows the kernel without tiles serves.  With 9 to 16 rows a narrow output has only its strips of 16 columns for
// workgroups, and each reads the activations for itself: 2,048 x 8,192 at 16 rows takes 32 us there and 21 with tiles and k shared out,
// 2,048 x 2,048 takes 10 against 11, 3,072 x 2,048 10 against 13.
bool few_rows(int M, int N, int K) { return M <= 8 || (M <= FEW_ROWS && (K <= 4096 || N >= 16 * gi_compute_units())); }

struct Cut { int bm, m_tiles, n_tiles, splits; };

// Tiles of 64 rows, or of 32 where those hold at least a tenth fewer rows beyond M.  The ranges of k go to 1, 2, 4 or 8 workgroups: what
// counts is the compute unit with the most of them (they share its matrix cores, and reach about half, two thirds and 0.72 of its 0.6
// TFLOP/s when there are one, two and three or more), against writing and reading the parts.  301 rows of 2,048 x 2,048 (160 tiles): 42
// us with one workgroup a tile, 35 with four.  Of 54 products of 17 to 600 rows it takes the fastest cut or one within 6 %, but for four (9 to 11 %).
Cut cut_for(int M, int N, int K) {
    const int units = gi_compute_units();
    Cut c;
    const long rows64 = (M + 63) / 64 * 64, rows32 = (M + 31) / 32 * 32;
    c.bm = rows32 * 10 <= rows64 * 9 ? 32 : 64;
    c.m_tiles = (M + c.bm - 1) / c.bm;
    c.n_tiles = (N + BN - 1) / BN;
    double best = 0;
    c.splits = 1;
    for (int z = 1; z <= RANGES; z *= 2) {
        const long a_unit = ((long)c.m_tiles * c.n_tiles * z + units - 1) / units;
        const double reached = a_unit == 1 ? 0.48 : a_unit == 2 ? 0.64 : 0.72;
        const double compute = (double)a_unit * 2.0 * c.bm * BN * ((double)K / z + 64) / 6.0e5 / reached;                               // us
        const double parts = z == 1 ? 0.0 : 4.0 + (double)z * M * N * 8 / 4.0e6;                                                         // us: a launch, 4 TB/s
        if (z == 1 || compute + parts < best) { best = compute + parts; c.splits = z; }
    }
    return c;
}

template <typename TA, typename TW, typename TC, bool ACC>
int launch(const TA* A, const TW* W, TC* C, float* part, long part_floats, int M, int N, int K, long lda, long ldw, long ldc, hipStream_t stream) {
    const auto by4 = [](const void* p, size_t elem) { return ((uintptr_t)p & (4 * elem - 1)) == 0; };
    const bool vector = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && by4(A, sizeof(TA)) && by4(W, sizeof(TW));
    if (vector && few_rows(M, N, K)) {
        // strips of 8 where strips of 16 would give fewer than two workgroups a compute unit
        if (M <= 8 && N < 32 * gi_compute_units())
            gemm_exact_few_rows_kernel<8, TA, TW, TC, ACC, Plain><<<(N + 7) / 8, 256, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, Plain{});
        else
            gemm_exact_few_rows_kernel<16, TA, TW, TC, ACC, Plain><<<(N + 15) / 16, 512, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, Plain{});
        return 0;
    }
    Cut c = cut_for(M, N, K);
    if (c.splits > 1 && (part == nullptr || part_floats < (long)c.splits * M * N)) c.splits = 1;
    const long total = (long)c.m_tiles * c.n_tiles * c.splits;
    GI_REQUIRE(total < 2147483647L - 8, "gemm_exact: M %d, N %d have too many tiles", M, N);
    const unsigned grid = (unsigned)((total + 7) / 8 * 8);
    float* to = c.splits > 1 ? part : nullptr;
    if constexpr (sizeof(TA) == 4 && sizeof(TW) == 4 && sizeof(TC) == 4) {
        if (vector && K % BK == 0 && lda < (1L << 22) && ldw < (1L << 22)) {           // (a tile's rows within 32-bit offsets)
#define RING(BM) gemm_exact_ring_kernel<BM, ACC><<<grid, 256, 0, stream>>>(A, W, C, to, M, N, K, lda, ldw, ldc, c.m_tiles, c.n_tiles, c.splits)
            if (c.bm == 64) RING(64);
            else RING(32);
#undef RING
            if (to) gemm_exact_add_parts_kernel<TC, ACC><<<(unsigned)(((size_t)M * N + 255) / 256), 256, 0, stream>>>(part, C, M, N, ldc, c.splits);
            return 0;
        }
    }
#define TILED(BM, VEC) gemm_exact_tiled_kernel<BM, VEC, TA, TW, TC, ACC><<<grid, 256, 0, stream>>>(A, W, C, to, M, N, K, lda, ldw, ldc, c.m_tiles, c.n_tiles, c.splits)
    if (c.bm == 64) { if (vector) TILED(64, true); else TILED(64, false); }
    else { if (vector) TILED(32, true); else TILED(32, false); }
#undef TILED
    if (to) gemm_exact_add_parts_kernel<TC, ACC><<<(unsigned)(((size_t)M * N + 255) / 256), 256, 0, stream>>>(part, C, M, N, ldc, c.splits);
    return 0;
}

}  // namespace

// floats of scratch the product wants for the parts of its sums (0: none; it also runs, slower, without)
GI_API long gi_gemm_exact_scratch_floats(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || few_rows(M, N, K)) return 0;
    const Cut c = cut_for(M, N, K);
    return c.splits > 1 ? (long)c.splits * M * N : 0;
}

GI_API int gi_gemm_exact(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype, int accumulate, int M, int N, int K,
                         long lda, long ldw, long ldc, float* part, long part_floats, hipStream_t stream) {
    GI_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_exact: M %d, N %d, K %d must be positive", M, N, K);
    GI_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_exact: leading dimensions (%ld, %ld, %ld) too small for K %d, N %d", lda, ldw, ldc, K, N);
    GI_REQUIRE(K <= 2147483647 - 256, "gemm_exact: K %d is too large", K);
    int rc;
#define GO(TA, TW, TC, ACC) rc = launch<TA, TW, TC, ACC>((const TA*)A, (const TW*)W, (TC*)C, part, part_floats, M, N, K, lda, ldw, ldc, stream)
#define BY_OUT(TA, TW)                                                  \
    if (c_dtype == GI_F32 && accumulate) GO(TA, TW, float, true);       \
    else if (c_dtype == GI_F32) GO(TA, TW, float, false);               \
    else if (c_dtype == GI_BF16 && !accumulate) GO(TA, TW, bf16_t, false); \
    else return gi_fail("gemm_exact: output dtype %d with accumulate %d is not supported", c_dtype, accumulate)
    if (a_dtype == GI_F32 && w_dtype == GI_F32) { BY_OUT(float, float); }
    else if (a_dtype == GI_F32 && w_dtype == GI_BF16) { BY_OUT(float, bf16_t); }
    else if (a_dtype == GI_BF16 && w_dtype == GI_BF16) { BY_OUT(bf16_t, bf16_t); }
    else if (a_dtype == GI_BF16 && w_dtype == GI_F32) { BY_OUT(bf16_t, float); }
    else return gi_fail("gemm_exact: unknown operand dtypes %d, %d", a_dtype, w_dtype);
#undef BY_OUT
#undef GO
    if (rc) return rc;
    GI_CHECK_LAUNCH("gemm_exact");
    return 0;
}

// Whether gi_gemm_exact_gated takes a product of these sizes.
GI_API int gi_gemm_exact_gated_takes(int M, int N, int K) { return M > 0 && N > 0 && N % 2 == 0 && K > 0 && K % 4 == 0 && few_rows(M, N, K); }
// And whether it is the faster way.  Its strips are 16 rows of weights; where the product alone has strips of 8 and its busiest compute unit so reads fewer
// rows, the two launches are the faster ones from k = 2,048 on: 1,024 x 4,096 10.5 us apart and 13.4 in one for 1 row, 2,048 x 3,072 11.0 and 11.9, 5,632 x 4,096
// 23.2 and 26.8 (8 rows 28.8 and 29.5); at k = 2,048 only for a strip a unit or two rows (1,024 columns 7.4 and 7.8, 6,144 for 1 row 14.8 and 15.5, for 8
// 17.9 and 16.5).
GI_API int gi_gemm_exact_gated_pays(int M, int N, int K) {
    const int units = gi_compute_units(), strips16 = (N + 15) / 16, strips8 = (N + 7) / 8;
    const bool more_rows = M <= 8 && N < 32 * units && (strips16 + units - 1) / units * 2 > (strips8 + units - 1) / units;
    return gi_gemm_exact_gated_takes(M, N, K) && !(more_rows && (K > 2048 || (K == 2048 && (N <= 4 * units || (M <= 2 && N > 16 * units)))));
}

// C [M, N / 2] = act(gate) * up of A W^T with W = [gate; up] (N rows in all), 32-bit throughout: the bits of gi_gemm_exact and gi_act_mul.  C must not be what A reads.
GI_API int gi_gemm_exact_gated(const float* A, const float* W, float* C, int act, float limit, int M, int N, int K, long lda, long ldw, long ldc, hipStream_t stream) {
    GI_REQUIRE(act >= 0 && act < GI_N_ACTIVATIONS && gi_gemm_exact_gated_takes(M, N, K), "gemm_exact (gated): sizes M %d, N %d, K %d or activation %d are not taken", M, N, K, act);
    GI_REQUIRE(lda >= K && ldw >= K && ldc >= N / 2 && lda % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0,
               "gemm_exact (gated): rows must be 16-byte aligned (strides %ld, %ld, %ld)", lda, ldw, ldc);
    gemm_exact_few_rows_kernel<16, float, float, float, false, Gate><<<(N / 2 + 7) / 8, 512, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, Gate{act, limit});
    GI_CHECK_LAUNCH("gemm_exact (gated)");
    return 0;
}

// Whether gi_gemm_exact_qkv_rope_store takes a q/k/v product of these sizes with heads of hd channels.
GI_API int gi_gemm_exact_qkv_rope_store_takes(int M, int N, int K, int hd) {
    return M > 0 && M <= 8 && N > 0 && N < 32 * gi_compute_units() && K > 0 && K % 4 == 0 && hd >= 8 && hd % 8 == 0 && N % hd == 0;
}

// The q/k/v product of an attention layer in 32-bit for a few rows, A [M, K] x W [N, K]^T with N = (n_heads + 2 n_kv) * hd, whose results do not come back: the bits
// and places of gi_gemm_exact and gi_rope_store.
GI_API int gi_gemm_exact_qkv_rope_store(const float* A, const float* W, int M, int N, int K, long lda, long ldw, const float* cos_t, const float* sin_t, const int* pos,
                                        const int* slot, const int* table, int table_stride, float* q_out, float* cache, long page_stride, int page_size, int n_heads, int n_kv,
                                        int hd, hipStream_t stream) {
    GI_REQUIRE(n_heads > 0 && n_kv > 0 && N == (n_heads + 2 * n_kv) * hd && gi_gemm_exact_qkv_rope_store_takes(M, N, K, hd),
               "gemm_exact (q/k/v): M %d, N %d, K %d with %d heads and %d key/value heads of %d are not taken", M, N, K, n_heads, n_kv, hd);
    GI_REQUIRE(lda >= K && ldw >= K && lda % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)q_out | (uintptr_t)cache | (uintptr_t)cos_t | (uintptr_t)sin_t) & 15) == 0,
               "gemm_exact (q/k/v): operands must be 16-byte aligned (strides %ld, %ld)", lda, ldw);
    GI_REQUIRE((cos_t == nullptr) == (sin_t == nullptr) && pos != nullptr && slot != nullptr && table != nullptr && q_out != nullptr && cache != nullptr && page_size > 0 &&
                   page_stride >= 2L * n_kv * page_size * hd && page_stride % 4 == 0,
               "gemm_exact (q/k/v): positions, slots, a table, q_out, both tables of the rotation or none, and a cache with a page stride of at least 2*n_kv*page_size*hd are needed");
    const Turn turn = {cos_t, sin_t, pos, slot, table, table_stride, q_out, cache, page_stride, page_size, n_heads, n_kv, hd};
    gemm_exact_few_rows_kernel<8, float, float, float, false, Turn><<<N / 8, 256, 0, stream>>>(A, W, nullptr, M, N, K, lda, ldw, 0L, turn);
    GI_CHECK_LAUNCH("gemm_exact (q/k/v)");
    return 0;
}
