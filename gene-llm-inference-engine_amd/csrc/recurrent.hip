// Recurrent mixers: a step's rows cut into the requests' runs on the device, the matrix memory with exponential gates
// (mLSTM) stepped token by token in 32-bit, and the norm and gate on its heads' outputs.
//
// The matrix memory of one head is S [dk][dv] with a normaliser n [dk] and a running maximum m of the gates' logarithms:
//     m_t = max(f_t + m_(t-1), i_t)
//     S_t = exp(f_t + m_(t-1) - m_t) S_(t-1) + exp(i_t - m_t) k_t v_t^T        n_t likewise with k_t alone
//     o_t = S_t^T q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6)
// with i_t = cap * tanh(pre_i / cap) and f_t = logsigmoid(cap * tanh(pre_f / cap)); S, n and m are zero at a sequence's start
// (m = 0, not minus infinity).  Columns of S never meet, and n is the column that S would have for a value that is always 1.
// So one wave owns a "tile" of four columns, three of S and n, for one head of one request, and walks the request's rows of this
// step in order; every tile of a head computes n and m alike and keeps its own copy (a tile that read them from a common place
// would race with the tile that writes them).  State of one request slot: [head][tile]{[dk][4], m, 3 unused}, 32-bit.
//
// Lane = (column, group of rows): a lane keeps ROWS rows (16 apart) of one column in registers; the 16 groups' shares of a
// column's S^T q (neighbouring lanes) are added by the vector unit's lane moves, and n . q, which every column's output is
// divided by, is read from the last column's lane.  A token so costs no barrier and no trip through LDS for the sums, three
// instructions per row of a lane, and the chip gets heads * dv / 3 independent waves: the recurrence is sequential in the
// tokens, so what counts is how few instructions a wave spends on one.
// Per token k and q*scale come through LDS (read as broadcasts).  The k, q and v of a block of tokens are asked for while the
// block before it is worked on and laid into LDS at its end, so that no token waits for memory.  The gates of 64 tokens are made
// at once, lane by token: m runs along them one after the other (an addition and a maximum each), and the exponentials it needs
// are then taken for all 64 at once.  Every sum's order is fixed by dk alone: a request's results have the same bits however
// its rows are cut into steps.
//
// The gated delta rule keeps a memory M [dk][dv] per head.  A token with decay d, step size s, unit key k and query q lets it decay,
// M <- d M, moves what it holds along k towards v, M <- M + k e^T with e = s (v - M^T k), and reads it, y = M^T q: the read-out
// sees the token's own write.  Columns of M never meet here either, so a wave owns four of them, lanes as above; a token costs
// two sums over the key's rows, which the kernel takes in one pass over the memory as it was before the token.  Before the rule,
// q, k and v pass a short causal convolution over the request's rows (the last taps - 1 rows before a step are part of the
// request's state) and SiLU, and q and k are made unit vectors; after it, a head's output is divided by its root mean square, as
// the matrix memory's.  The decay is one number per head, or one per head and key channel, which then scales the memory's row of that channel.
#include "common.h"

namespace {

// Rows of a step, in order, are runs of single requests; a run starts where the slot changes or the position does not follow.
// One workgroup, a row a thread (one wave that went through 1,777 rows 64 at a time took 26 us, a round trip to memory for each).
__global__ __launch_bounds__(1024) void segments_kernel(const int* __restrict__ slot, const int* __restrict__ pos, int n_rows,
                                                       int* __restrict__ seg_start, int* __restrict__ seg_len, int n_segs) {
    __shared__ int starts[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n_waves = blockDim.x >> 6;
    int count = 0;
    for (int base = 0; base < n_rows; base += blockDim.x) {
        const int t = base + threadIdx.x;
        const bool first = t < n_rows && (t == 0 || slot[t] != slot[t - 1] || pos[t] != pos[t - 1] + 1);
        const unsigned long long mask = __ballot(first);
        if (lane == 0) starts[wave] = __popcll(mask);
        __syncthreads();
        int idx = count + __popcll(mask & ((1ull << lane) - 1ull));
        for (int w = 0; w < n_waves; ++w) {
            if (w < wave) idx += starts[w];
            count += starts[w];
        }
        if (first && idx < n_segs) seg_start[idx] = t;
        __syncthreads();
    }
    __threadfence_block();
    __syncthreads();
    for (int s = threadIdx.x; s < n_segs; s += blockDim.x) seg_len[s] = s < count ? ((s + 1 < count ? seg_start[s + 1] : n_rows) - seg_start[s]) : 0;
}

// Lane `u`'s value of x, u the same for every lane.
__device__ __forceinline__ float lane_value(float x, int u) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), u)); }

// Sum over each group of RG neighbouring lanes (4, 8 or 16: within a row of 16 lanes), by the data-parallel moves of the vector
// unit: a lane and its mirror image in the group, then lanes two apart, then neighbours.  Every lane of a group ends with the
// same bits (each level adds the same two numbers on both sides).
template <int CTRL>
__device__ __forceinline__ float dpp_moved(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
template <int RG>
__device__ __forceinline__ float group_sum(float x) {
    static_assert(RG == 4 || RG == 8 || RG == 16, "groups of 4, 8 or 16 lanes");
    if constexpr (RG == 16) x += dpp_moved<0x140>(x);        // row_mirror: lane i <-> 15 - i
    if constexpr (RG >= 8) x += dpp_moved<0x141>(x);         // row_half_mirror: lane i <-> 7 - i
    x += dpp_moved<0x4E>(x);                                 // quad_perm [2, 3, 0, 1]
    x += dpp_moved<0xB1>(x);                                 // quad_perm [1, 0, 3, 2]
    return x;
}

// w . l with the numbers of l rounded to bfloat16 as a product's rows are: one output of a product behind a narrow middle, made by one
// lane, eight weights a load where the row allows it.  One ascending sum.
__device__ __forceinline__ float narrow_dot(const float* __restrict__ l, const bf16_t* __restrict__ w, int rank) {
    float a = 0.f;
    if (rank % 8 == 0 && ((uintptr_t)w & 15) == 0) {
#pragma unroll 4
        for (int r = 0; r < rank; r += 8) {
            const uint4 v = *reinterpret_cast<const uint4*>(w + r);
            const uint32_t p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a = fmaf(bf16_to_f32(f32_to_bf16(l[r + 2 * i])), __uint_as_float(p[i] << 16), a);
                a = fmaf(bf16_to_f32(f32_to_bf16(l[r + 2 * i + 1])), __uint_as_float(p[i] & 0xffff0000u), a);
            }
        }
        return a;
    }
    for (int r = 0; r < rank; ++r) a = fmaf(bf16_to_f32(f32_to_bf16(l[r])), bf16_to_f32(w[r]), a);
    return a;
}

__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

template <int ROWS>
__global__ __launch_bounds__(64) void mlstm_scan_kernel(const float* __restrict__ proj, long ld, int q_off, int k_off, int v_off, int i_off, int f_off,
                                                       const float* __restrict__ i_bias, const float* __restrict__ f_bias, float cap, float q_scale,
                                                       const int* __restrict__ seg_start, const int* __restrict__ seg_len,
                                                       const int* __restrict__ row_slot, float* __restrict__ state, long state_stride,
                                                       float* __restrict__ out, long ldo, float* __restrict__ den, int dk, int dv) {
    constexpr int C = 4, VC = 3;                 // columns a wave holds: three of S and n (as the column of a value that is always 1)
    constexpr int RG = 64 / C;                   // groups of rows: lane = column * RG + group, so that a column's groups are neighbouring lanes
    constexpr int KQ = RG * ROWS;                // rows a token's k and q cover (dk, padded with zeros)
    constexpr int TB = 1024 / KQ;                // tokens staged at a time: their k, q and v wait in LDS while the block before them is worked on
    constexpr int PER = TB * KQ / 64;            // (k, q) pairs a lane brings per block
    static_assert(TB >= 2 && TB <= 16 && 64 % TB == 0 && TB * VC <= 64, "staging blocks divide the gates' blocks of 64 tokens; a lane brings one value");
    __shared__ float2 kq_s[2][TB][KQ];
    __shared__ float v_s[2][TB][C];
    __shared__ float4 coef[64];                  // per token of the gates' block: {decay of what is held, weight of what comes, exp(-m), -}
    const int seg = blockIdx.x, h = blockIdx.y, vt = blockIdx.z, n_tiles = gridDim.z;
    const int lane = threadIdx.x, c = lane / RG, rg = lane % RG;
    const int n = seg_len[seg];
    if (n <= 0) return;
    const int t0 = seg_start[seg];
    const int col = vt * VC + c;
    const bool live = c < VC && col < dv;
    float* st = state + (size_t)row_slot[t0] * state_stride + ((size_t)h * n_tiles + vt) * ((size_t)dk * C + 4);
    float* st_m = st + (size_t)dk * C;

    float S[ROWS];
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        const int i = rr * RG + rg;                  // (a lane's rows lie RG apart: the groups' reads of LDS then fall into different banks)
        S[rr] = i < dk ? st[(size_t)i * C + c] : 0.f;
    }
    float m = st_m[0];
    const float bi = i_bias[h], bf = f_bias[h];

    // A block of TB tokens from `first` on (rows beyond the request's last are read as its last: finite, and never used).
    float2 kq_reg[PER];
    float v_reg;
    auto fetch = [&](int first) {
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int idx = lane + 64 * e, u = idx / KQ, i = idx % KQ;
            const float* row = proj + (size_t)(t0 + min(first + u, n - 1)) * ld;
            const int ic = min(i, dk - 1);
            const float kk = row[k_off + h * dk + ic], qq = row[q_off + h * dk + ic] * q_scale;
            kq_reg[e] = i < dk ? float2{kk, qq} : float2{0.f, 0.f};
        }
        const int idx = min(lane, TB * VC - 1), u = idx / VC, cc = min(vt * VC + idx % VC, dv - 1);
        v_reg = proj[(size_t)(t0 + min(first + u, n - 1)) * ld + v_off + h * dv + cc];
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int idx = lane + 64 * e;
            kq_s[buf][idx / KQ][idx % KQ] = kq_reg[e];
        }
        if (lane < TB * VC) v_s[buf][lane / VC][lane % VC] = v_reg;
    };
    if (lane < 2 * TB) v_s[lane / TB][lane % TB][VC] = 1.0f;          // the value that makes a column of S the normaliser n
    fetch(0);
    stash(0);
    int buf = 0;

    for (int b0 = 0; b0 < n; b0 += 64) {
        const int count = min(64, n - b0);
        // The gates of this block's tokens, lane u token u; then m along the block, one token after the other (two numbers a
        // token: cheap), each lane keeping the m before and after its own token; then the exponentials, all tokens at once.
        const float* g = proj + (size_t)(t0 + b0 + min(lane, count - 1)) * ld;
        const float li = cap * tanhf((g[i_off + h] + bi) / cap);
        const float lf = log_sigmoid(cap * tanhf((g[f_off + h] + bf) / cap));
        float m_before = 0.f, m_after = 0.f;
        for (int u = 0; u < count; ++u) {
            const float m_new = fmaxf(lane_value(lf, u) + m, lane_value(li, u));        // (u is the same for the whole wave)
            if (lane == u) { m_before = m; m_after = m_new; }
            m = m_new;
        }
        __syncthreads();                             // (one wave: orders this block's reads of coef before the writes)
        coef[lane] = float4{expf(lf + m_before - m_after), expf(li - m_after), expf(-m_after), 0.f};
        __syncthreads();
        for (int s0 = 0; s0 < count; s0 += TB, buf ^= 1) {
            const bool more = b0 + s0 + TB < n;
            if (more) fetch(b0 + s0 + TB);
            const int here = min(TB, count - s0);
            // One token: the memory takes it in; the lane's share of its column's S^T q comes back (of n . q in the last column).
            auto token = [&](int u, float& acc, float& floor_) {
                const float4 cf = coef[s0 + u];
                const float a = cf.x, bv = cf.y * v_s[buf][u][c];
                acc = 0.f, floor_ = cf.z;
#pragma unroll
                for (int rr = 0; rr < ROWS; ++rr) {
                    const float2 kq = kq_s[buf][u][rr * RG + rg];
                    S[rr] = fmaf(a, S[rr], kq.x * bv);
                    acc = fmaf(S[rr], kq.y, acc);
                }
            };
            // The groups' shares are added by lane moves; n . q is then in the last column's lanes, the same for the whole wave.
            // The columns' sums leave undivided; what they are to be divided by, max(|n . q|, exp(-m)) + 1e-6, one number per
            // token and head, is written by the head's first tile, and whoever reads the sums divides (the kernel behind this
            // one reads every sum once anyway; a division per token in every wave is a sixth of what a wave does here).
            auto finish = [&](int u, float acc, float floor_) {
                acc = group_sum<RG>(acc);
                const size_t t = (size_t)(t0 + b0 + s0 + u);
                if (rg == 0 && live) out[t * ldo + h * dv + col] = acc;
                if (vt == 0 && lane == VC * RG) den[t * gridDim.y + h] = fmaxf(fabsf(acc), floor_) + 1e-6f;
            };
            constexpr int UB = TB >= 4 ? 4 : TB;     // so many tokens at a time, so that their reads of LDS go out together
            int u = 0;
            for (; u + UB <= here; u += UB) {
                float acc[UB], floor_[UB];
#pragma unroll
                for (int k = 0; k < UB; ++k) token(u + k, acc[k], floor_[k]);
#pragma unroll
                for (int k = 0; k < UB; ++k) finish(u + k, acc[k], floor_[k]);
            }
            for (; u < here; ++u) {
                float acc, floor_;
                token(u, acc, floor_);
                finish(u, acc, floor_);
            }
            __syncthreads();                         // this block's reads are done before the buffer after next is written
            if (more) stash(buf ^ 1);
            __syncthreads();
        }
    }
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        const int i = rr * RG + rg;
        if (i < dk && (live || c == VC)) st[(size_t)i * C + c] = S[rr];
    }
    if (lane == 0) st_m[0] = m;
}

// y[t, h*dv + d] = w[h*dv + d] * o[t, h, d] * rsqrt(mean_d(o[t, h, :]^2) + eps) * sigmoid(g[t, h*dv + d]): one wave per (row, head).
// With `den` [rows, heads], o is what the rows hold divided by den[t, h] (the matrix memory's sums and their divisor).
// w_head_stride: dv where every head has weights of its own, 0 where all heads share one [dv]; gate_act 0: sigmoid(g), 1: SiLU, g sigmoid(g).
// With `low` (float32 rows of stride ldg, `rank` numbers each) g is made here, g[t, i] = w_up[i] . low[t], the numbers rounded to bfloat16 as a
// product's rows are: the form for a few rows, whose workgroups are NT = 256 threads (a wave otherwise).
template <typename TW, typename TO, int NT>
__global__ __launch_bounds__(NT) void head_norm_gate_kernel(const float* __restrict__ o, long ldo, const float* __restrict__ den,
                                                           const float* __restrict__ g, long ldg, const TW* __restrict__ w,
                                                           TO* __restrict__ y, long ldy, int n_heads, int dv, float eps, int w_head_stride, int gate_act,
                                                           const float* __restrict__ low, int rank, const bf16_t* __restrict__ w_up) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const float* orow = o + (size_t)t * ldo + (size_t)h * dv;
    const float by = den ? den[(size_t)t * n_heads + h] : 1.0f;
    float ss = 0.f;
    for (int d = lane; d < dv; d += NT) {
        const float v = den ? orow[d] / by : orow[d];
        ss = fmaf(v, v, ss);
    }
    if constexpr (NT == 64) {
        ss = wave_sum(ss);
    } else {
        __shared__ float red[NT / 64];
        ss = block_sum<NT>(ss, red);
    }
    const float r = 1.0f / sqrtf(ss / (float)dv + eps);
    for (int d = lane; d < dv; d += NT) {
        const float v = den ? orow[d] / by : orow[d];
        const float z = low ? narrow_dot(low + (size_t)t * ldg, w_up + ((size_t)h * dv + d) * rank, rank) : g[(size_t)t * ldg + (size_t)h * dv + d];
        const float gate = (gate_act ? z : 1.0f) / (1.0f + expf(-z));
        store_f32(y, (size_t)t * ldy + (size_t)h * dv + d, load_f32(w, (size_t)h * w_head_stride + d) * (v * r) * gate);
    }
}


// ------------------------------------------------------------------------------------- gated delta rule
constexpr int DELTA_MAX_TAPS = 16;

__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// How many of the rows before row t belong to the same request's run in this step, up to `most`.
__device__ __forceinline__ int rows_before(const int* __restrict__ slot, const int* __restrict__ pos, int t, int most) {
    int r = 0;
    while (r < most && t - r - 1 >= 0 && slot[t - r - 1] == slot[t] && pos[t - r - 1] == pos[t] - r - 1) ++r;
    return r;
}

// What the rule needs of one row, one wave per (row, item).  The convolved columns of `proj` are [conv_off, conv_off + n_conv):
// query heads [n_kv][dk], key heads [n_kv][dk], value heads [n_heads][dv], in this order; `taps` [n_conv][n_taps] float32, the
// last tap the row's own; `tail` [slots][n_taps - 1][n_conv] the request's last rows before this step (zeros at its start).
//   items 0 .. 2 n_kv - 1     a query or key head: convolution, SiLU, divided by sqrt(sum of squares + 1e-6); queries times q_scale
//   items 2 n_kv .. + n_heads a value head: convolution, SiLU
//   the last item             per head the decay exp(-exp(a_log) softplus(pre_a + dt_bias)) and the step size sigmoid(pre_b)
// qkv: float32 [rows, n_conv] in the columns' order; gates: float32 [rows, 2 n_heads], decays then step sizes.
// With decays per channel (dn = dk numbers a head, else 1) there are n_heads last items, one per head, and gates is [rows, n_heads dk +
// n_heads].  pre_a [rows, lda] holds the heads' dn numbers; or, with `low` (bfloat16 weights w_up [n_heads dn][rank] on the numbers
// low [rows, rank], which are rounded to bfloat16 as a product's rows are), pre_a is made here: the form for a few rows.
// move_tail: every row of the step is its request's only one (a decode step); the thread that has read a channel's tail then also
// moves it on by the row's own input, and no other kernel needs to (with several rows of a request in a step, rows read the tail
// that others would be writing: `delta_tail_kernel` does it behind this one).
__global__ __launch_bounds__(64) void delta_prepare_kernel(const float* __restrict__ proj, long ld, int conv_off, const float* __restrict__ pre_a, long lda, int b_off,
                                                          const float* __restrict__ taps, int n_taps, float* __restrict__ tail, long tail_stride, int move_tail,
                                                          const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                                                          const int* __restrict__ slot, const int* __restrict__ pos, float* __restrict__ qkv,
                                                          float* __restrict__ gates, int n_heads, int n_kv, int dk, int dv, float q_scale, int dn,
                                                          const float* __restrict__ low, int rank, const bf16_t* __restrict__ w_up) {
    const int t = blockIdx.x, item = blockIdx.y, lane = threadIdx.x;
    if (item >= 2 * n_kv + n_heads) {
        const int h0 = dn > 1 ? item - 2 * n_kv - n_heads : 0, h1 = dn > 1 ? h0 + 1 : n_heads;
        float* out = gates + (size_t)t * n_heads * (dn + 1);
        for (int i = h0 * dn + lane; i < h1 * dn; i += 64) {
            const float a = low ? narrow_dot(low + (size_t)t * ld, w_up + (size_t)i * rank, rank) : pre_a[(size_t)t * lda + i];
            out[i] = expf(-expf(a_log[i / dn]) * softplus_f(a + dt_bias[i]));
        }
        for (int h = h0 + lane; h < h1; h += 64) out[n_heads * dn + h] = 1.0f / (1.0f + expf(-proj[(size_t)t * ld + b_off + h]));
        return;
    }
    const int n_conv = 2 * n_kv * dk + n_heads * dv;
    const bool unit = item < 2 * n_kv;
    const int first = unit ? item * dk : 2 * n_kv * dk + (item - 2 * n_kv) * dv, width = unit ? dk : dv;
    const int before = rows_before(slot, pos, t, n_taps - 1);
    float* old = tail + (size_t)slot[t] * tail_stride;
    float ss = 0.f;
    for (int d = lane; d < width; d += 64) {
        const int c = first + d;
        float y = 0.f;
        for (int j = 0; j < n_taps; ++j) {
            const int back = n_taps - 1 - j;                      // rows before t that tap j reads
            const float x = back <= before ? proj[(size_t)(t - back) * ld + conv_off + c] : old[(size_t)(n_taps - 1 - (back - before)) * n_conv + c];
            y = fmaf(taps[(size_t)c * n_taps + j], x, y);
        }
        if (move_tail) {
            for (int i = 0; i + 2 < n_taps; ++i) old[(size_t)i * n_conv + c] = old[(size_t)(i + 1) * n_conv + c];
            if (n_taps > 1) old[(size_t)(n_taps - 2) * n_conv + c] = proj[(size_t)t * ld + conv_off + c];
        }
        y = y / (1.0f + expf(-y));
        qkv[(size_t)t * n_conv + c] = y;                          // (read back below by the lane that wrote it)
        ss = fmaf(y, y, ss);
    }
    if (!unit) return;
    const float r = (item < n_kv ? q_scale : 1.0f) / sqrtf(wave_sum(ss) + 1e-6f);
    for (int d = lane; d < width; d += 64) qkv[(size_t)t * n_conv + first + d] *= r;
}

// The same for the rows of prompts (up to four taps, a decay a head, query and key heads of up to 64 channels): a wave takes PREPARE_ROWS rows of an item, whose inputs it
// asks for at once, each once, with the taps and the rows' places in their runs, and four items' waves are a workgroup (1,777 rows of 17 items as waves of
// their own, each with its chain of places, inputs and taps: 23.2 us, so 14.7).  Every number is made as above: the same bits.
constexpr int PREPARE_ROWS = 8, PREPARE_TAPS = 4;
__global__ __launch_bounds__(256) void delta_prepare_rows_kernel(const float* __restrict__ proj, long ld, int conv_off, const float* __restrict__ pre_a, long lda, int b_off,
                                                                const float* __restrict__ taps, int n_taps, const float* __restrict__ tail, long tail_stride,
                                                                const float* __restrict__ a_log, const float* __restrict__ dt_bias, const int* __restrict__ slot,
                                                                const int* __restrict__ pos, float* __restrict__ qkv, float* __restrict__ gates, int n_rows, int n_heads, int n_kv,
                                                                int dk, int dv, float q_scale) {
    const int t0 = blockIdx.x * PREPARE_ROWS, item = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n = min(PREPARE_ROWS, n_rows - t0);
    if (item > 2 * n_kv + n_heads) return;
    if (item == 2 * n_kv + n_heads) {
        for (int i = lane; i < n * n_heads; i += 64) {
            const size_t t = t0 + i / n_heads;
            const int h = i % n_heads;
            gates[t * 2 * n_heads + h] = expf(-expf(a_log[h]) * softplus_f(pre_a[t * lda + h] + dt_bias[h]));
            gates[t * 2 * n_heads + n_heads + h] = 1.0f / (1.0f + expf(-proj[t * ld + b_off + h]));
        }
        return;
    }
    // bit l of `follows`: row t0 - 2 + l belongs to the run of the row before it
    const int mine = t0 - (PREPARE_TAPS - 2) + lane;
    const bool there = lane < PREPARE_ROWS + PREPARE_TAPS - 2 && mine > 0 && mine < n_rows;
    const int at = there ? mine : 0, at_before = there ? mine - 1 : 0;
    const bool same = slot[at_before] == slot[at] && pos[at_before] == pos[at] - 1;
    const unsigned follows = (unsigned)__ballot(there && same);
    const int n_conv = 2 * n_kv * dk + n_heads * dv;
    const bool unit = item < 2 * n_kv;
    const int first = unit ? item * dk : 2 * n_kv * dk + (item - 2 * n_kv) * dv, width = unit ? dk : dv;
    for (int d0 = 0; d0 < width; d0 += 64) {                                            // (a query or key head: once)
        const bool live = d0 + lane < width;
        const int c = first + min(d0 + lane, width - 1);
        float x[PREPARE_ROWS + PREPARE_TAPS - 1], w[PREPARE_TAPS];                      // w[b]: of the row b before
#pragma unroll
        for (int i = 0; i < PREPARE_ROWS + PREPARE_TAPS - 1; ++i) x[i] = proj[(size_t)min(max(t0 - (PREPARE_TAPS - 1) + i, 0), n_rows - 1) * ld + conv_off + c];
#pragma unroll
        for (int b = 0; b < PREPARE_TAPS; ++b) w[b] = taps[(size_t)c * n_taps + max(n_taps - 1 - b, 0)];
#pragma unroll
        for (int i = 0; i < PREPARE_ROWS; ++i) {
            if (i >= n) break;
            const unsigned run = follows >> i;                                          // bits 2, 1, 0: the row, the one before it, the one before that
            const int before = run & 4 ? (run & 2 ? (run & 1 ? 3 : 2) : 1) : 0;
            float y = 0.f;
#pragma unroll
            for (int b = PREPARE_TAPS - 1; b >= 0; --b) {
                if (b >= n_taps) continue;
                float from = x[i + PREPARE_TAPS - 1 - b];
                if (b > before) from = tail[(size_t)slot[t0 + i] * tail_stride + (size_t)(n_taps - 1 - (b - before)) * n_conv + c];      // (the request's rows before this step)
                y = fmaf(w[b], from, y);
            }
            y = y / (1.0f + expf(-y));
            float r = 1.0f;
            if (unit) r = (item < n_kv ? q_scale : 1.0f) / sqrtf(wave_sum(live ? fmaf(y, y, 0.f) : 0.f) + 1e-6f);
            if (live) qkv[(size_t)(t0 + i) * n_conv + c] = unit ? y * r : y;
        }
    }
}

// And for steps of single rows (two to four taps, heads of up to 64 and 128 channels): no row has one of its request's before it, and a channel's tail, input and taps
// are asked for at once (one after the other, with the tail's places moved on in between, 5 rows took 6.9 us, so 4.6).
__global__ __launch_bounds__(64) void delta_prepare_single_kernel(const float* __restrict__ proj, long ld, int conv_off, const float* __restrict__ pre_a, long lda, int b_off,
                                                                 const float* __restrict__ taps, int n_taps, float* __restrict__ tail, long tail_stride,
                                                                 const float* __restrict__ a_log, const float* __restrict__ dt_bias, const int* __restrict__ slot,
                                                                 float* __restrict__ qkv, float* __restrict__ gates, int n_heads, int n_kv, int dk, int dv, float q_scale) {
    const int item = blockIdx.y, lane = threadIdx.x;
    const size_t t = blockIdx.x;
    if (item == 2 * n_kv + n_heads) {
        for (int h = lane; h < n_heads; h += 64) {
            gates[t * 2 * n_heads + h] = expf(-expf(a_log[h]) * softplus_f(pre_a[t * lda + h] + dt_bias[h]));
            gates[t * 2 * n_heads + n_heads + h] = 1.0f / (1.0f + expf(-proj[t * ld + b_off + h]));
        }
        return;
    }
    const int n_conv = 2 * n_kv * dk + n_heads * dv;
    const bool unit = item < 2 * n_kv;
    const int first = unit ? item * dk : 2 * n_kv * dk + (item - 2 * n_kv) * dv, width = unit ? dk : dv;
    float* old = tail + (size_t)slot[t] * tail_stride;
    float x[2][PREPARE_TAPS], w[2][PREPARE_TAPS];                                       // x[.][0] the row's own input, x[.][b] the one b before; w likewise
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int c = first + min(lane + 64 * e, width - 1);
        x[e][0] = proj[t * ld + conv_off + c];
#pragma unroll
        for (int b = 0; b < PREPARE_TAPS; ++b) w[e][b] = taps[(size_t)c * n_taps + max(n_taps - 1 - b, 0)];
#pragma unroll
        for (int b = 1; b < PREPARE_TAPS; ++b) x[e][b] = old[(size_t)max(n_taps - 1 - b, 0) * n_conv + c];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        if (64 * e >= width) break;
        const bool live = lane + 64 * e < width;
        const int c = first + min(lane + 64 * e, width - 1);
        float y = 0.f;
#pragma unroll
        for (int b = PREPARE_TAPS - 1; b >= 0; --b)
            if (b < n_taps) y = fmaf(w[e][b], x[e][b], y);
        y = y / (1.0f + expf(-y));
        float r = 1.0f;
        if (unit) r = (item < n_kv ? q_scale : 1.0f) / sqrtf(wave_sum(live ? fmaf(y, y, 0.f) : 0.f) + 1e-6f);
        if (!live) continue;
        qkv[t * n_conv + c] = unit ? y * r : y;
#pragma unroll
        for (int b = 0; b < PREPARE_TAPS - 1; ++b)
            if (b < n_taps - 1) old[(size_t)(n_taps - 2 - b) * n_conv + c] = x[e][b];
    }
}

// After a step's rows the request's tail is its last n_taps - 1 inputs: of this step's rows, and of the old tail where the step
// brought fewer.  A thread reads all it needs of a channel before it writes; a request's channels lie over the grid's second dimension
// (one workgroup a request that went through 1,536 channels 256 at a time took 7.5 us).
__global__ __launch_bounds__(256) void delta_tail_kernel(const float* __restrict__ proj, long ld, int conv_off, int n_conv, int n_taps,
                                                        const int* __restrict__ seg_start, const int* __restrict__ seg_len,
                                                        const int* __restrict__ slot, float* __restrict__ tail, long tail_stride) {
    const int n = seg_len[blockIdx.x];
    if (n <= 0) return;
    const int t0 = seg_start[blockIdx.x], keep = n_taps - 1;
    float* mine = tail + (size_t)slot[t0] * tail_stride;
    for (int c = blockIdx.y * 256 + threadIdx.x; c < n_conv; c += 256 * gridDim.y) {
        float held[DELTA_MAX_TAPS];
#pragma unroll
        for (int s = 0; s < DELTA_MAX_TAPS; ++s) {
            if (s >= keep) break;
            const int e = n - keep + s;                           // row of the step, or (negative) place before it
            held[s] = e >= 0 ? proj[(size_t)(t0 + e) * ld + conv_off + c] : mine[(size_t)(keep + e) * n_conv + c];
        }
#pragma unroll
        for (int s = 0; s < DELTA_MAX_TAPS; ++s) {
            if (s >= keep) break;
            mine[(size_t)s * n_conv + c] = held[s];
        }
    }
}

// The rule itself: one wave per (request of the step, head, four columns of M).  lane = column * 16 + group of rows; a lane keeps
// the rows 16 apart of its column.  State of a request slot: [head][tile]{[dk][4]}.
// With M the memory before the token, M' = d M + k e^T after it and e = s (v - d M^T k), the read-out is
//     y = M'^T q = d M^T q + e (k . q):
// both sums over the old memory's rows (M^T k and M^T q) are taken in one pass and reduced side by side, the memory is
// updated behind them, and a token's chain of dependent steps is one pass and one reduction, not two of each.  Every sum over the
// key's rows is the lanes' own shares in a fixed order, then the 16 groups by lane moves: the bits do not depend on the cut.
// CHANNEL: the decay is a number per key channel, so the sums are taken over D M, whose rows the decays have scaled already:
//     e = s (v - (D M)^T k),   y = (D M)^T q + e (k . q).
// Bound by the seven clocks or so that each instruction of a wave alone on its SIMD takes, token after token (one wave a compute unit at 8
// heads of 64 x 128), so nothing stands in a token that can stand elsewhere: a block's keys and queries are asked for a block ahead, four
// channels a load, and wait in LDS; a token's numbers leave LDS while the token before is worked on; k . q, in which nothing of the memory
// is, is summed for four tokens at once before the block.  Microseconds for 1,777 tokens of 8 such heads, five requests of 200, 1,024
// tokens of 32 heads of 128 x 128 with decays per channel: 207, 38, 270; each token's reads waited for in its turn and k . q summed in it: 279, 51,
// 317; two columns a wave (rows of a lane neighbours, another order of the sums), a token's numbers loaded straight into registers: 192, 69,
// 246, but 115 for 64 single rows of 32 heads of 128 x 128 that take 57 with four columns.
// A token's numbers for a lane's rows of a column: {k, q} of every row, the rows' decays where there is one per channel, and own = {decay, step, v, k . q}.
template <int ROWS, bool CHANNEL>
struct DeltaToken {
    float2 kq[ROWS];
    float d[CHANNEL ? ROWS : 1];
    float4 own;
};

// A lane's share of k . q (the form with decays per channel rounds every product).
template <int ROWS, bool CHANNEL>
__device__ __forceinline__ float delta_key_query(const float2 (&x)[ROWS]) {
#pragma clang fp contract(off)
    float kq = 0.f;
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) kq = CHANNEL ? kq + x[rr].x * x[rr].y : fmaf(x[rr].x, x[rr].y, kq);
    return kq;
}

// One token for one lane's rows of a column: the memory moves on, the column's read-out comes back (in every lane of the column).
template <int ROWS, bool CHANNEL>
__device__ __forceinline__ float delta_token(float (&S)[ROWS], const DeltaToken<ROWS, CHANNEL>& x) {
    const float decay = x.own.x, step = x.own.y, v = x.own.z, kq = x.own.w;
    float sk = 0.f, sq = 0.f;
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        if constexpr (CHANNEL) S[rr] *= x.d[rr];
        sk = fmaf(S[rr], x.kq[rr].x, sk);
        sq = fmaf(S[rr], x.kq[rr].y, sq);
    }
    sk = group_sum<16>(sk);
    sq = group_sum<16>(sq);
    if constexpr (CHANNEL) {
        const float w = step * (v - sk);
#pragma unroll
        for (int rr = 0; rr < ROWS; ++rr) S[rr] = fmaf(x.kq[rr].x, w, S[rr]);
        return fmaf(w, kq, sq);
    } else {
        const float w = step * (v - decay * sk);               // s (v - d M^T k)
#pragma unroll
        for (int rr = 0; rr < ROWS; ++rr) S[rr] = fmaf(decay, S[rr], x.kq[rr].x * w);
        return fmaf(decay, sq, w * kq);
    }
}

// A lane keeps a block's keys and queries as they come until they are laid into LDS.
template <int N>
struct DeltaBlock {
    float k[N], q[N], d[N];
    float v, decay, step;
};

// EVERY: keys of 16 ROWS channels and every token's numbers at multiples of 16 bytes, so that they come four at a time and nothing is masked.
template <int ROWS, bool CHANNEL, bool EVERY>
__global__ __launch_bounds__(64) void delta_scan_kernel(const float* __restrict__ qkv, long ld, const float* __restrict__ gates,
                                                       const int* __restrict__ seg_start, const int* __restrict__ seg_len,
                                                       const int* __restrict__ row_slot, float* __restrict__ state, long state_stride,
                                                       float* __restrict__ out, long ldo, int n_heads, int n_kv, int dk, int dv, int below) {
    constexpr int C = 4, RG = 16, KQ = RG * ROWS;
    constexpr int TB = (1024 / KQ) < 16 ? (1024 / KQ) : 16;      // tokens staged at a time
    constexpr int PER = TB * KQ / 64, WIDE = EVERY ? 4 : 1;      // (k, q) pairs a lane brings per block, and at a time
    static_assert(TB >= 2 && TB * C <= 64, "a block of 2 to 16 tokens; a lane brings one token's numbers of one column");
    __shared__ __attribute__((aligned(16))) float2 kq_s[2][TB][KQ];
    __shared__ __attribute__((aligned(16))) float d_s[2][TB][CHANNEL ? KQ : 4];
    __shared__ float4 own_s[2][TB][C];                           // per token and column {decay, step, v, k . q}
    const int seg = blockIdx.x, h = blockIdx.y, vt = blockIdx.z, n_tiles = gridDim.z;
    const int lane = threadIdx.x, c = lane / RG, rg = lane % RG;
    const int n = seg_len[seg];
    if (n <= 0 || (below && n >= below)) return;
    const int t0 = seg_start[seg];
    const int col = vt * C + c, kvh = h / (n_heads / n_kv);
    const bool live = col < dv;
    float* st = state + (size_t)row_slot[t0] * state_stride + ((size_t)h * n_tiles + vt) * ((size_t)dk * C);
    const int q_at = kvh * dk, k_at = (n_kv + kvh) * dk, v_at = 2 * n_kv * dk + h * dv;

    float S[ROWS];
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        const int i = rr * RG + rg;
        S[rr] = EVERY || i < dk ? st[(size_t)i * C + c] : 0.f;
    }
    // A block of TB tokens from `first` on (rows beyond the request's last are read as its last: finite, and never used).
    const int dn = CHANNEL ? dk : 1;             // decays a head
    const size_t ldg = (size_t)n_heads * (dn + 1);
    // The numbers stay as they come until they are laid into LDS: a condition or a product here would make the wave wait for each.
    DeltaBlock<PER> r;
    const auto four = [](float* to, const void* from) {
        const float4 x = *reinterpret_cast<const float4*>(from);
        to[0] = x.x, to[1] = x.y, to[2] = x.z, to[3] = x.w;
    };
    // Keys of up to 256 channels: a lane brings the same channels of several tokens, from one token's row to the next a scalar step.
    constexpr bool STEPS = EVERY && KQ <= 256;
    const char* from_row = (const char*)(qkv + (size_t)(t0 + lane * 4 / KQ) * ld + q_at + lane * 4 % KQ);
    const char* from_gates = (const char*)(gates + (size_t)(t0 + lane * 4 / KQ) * ldg + (size_t)h * dk + lane * 4 % KQ);
    const size_t row_step = (size_t)ld * (4 * 256 / KQ), gates_step = ldg * (4 * 256 / KQ), to_keys = (size_t)n_kv * dk * 4;
    auto fetch = [&](int first) {
        if (STEPS && first + TB <= n) {
            const size_t row = (size_t)first * ld * 4, row_gates = (size_t)first * ldg * 4;
#pragma unroll
            for (int e = 0; e < PER; e += WIDE) {
                four(&r.q[e], from_row + (row + e / 4 * row_step));
                four(&r.k[e], from_row + (row + e / 4 * row_step + to_keys));
                if constexpr (CHANNEL) four(&r.d[e], from_gates + (row_gates + e / 4 * gates_step));
            }
        } else {
#pragma unroll
            for (int e = 0; e < PER; e += WIDE) {
                const int idx = lane * WIDE + 64 * e, u = idx / KQ, i = idx % KQ;
                const size_t t = t0 + min(first + u, n - 1);
                const float *row = qkv + t * ld, *decays = gates + t * ldg + h * dk;
                if constexpr (EVERY) {
                    four(&r.k[e], row + k_at + i);
                    four(&r.q[e], row + q_at + i);
                    if constexpr (CHANNEL) four(&r.d[e], decays + i);
                } else {
                    const int ic = min(i, dk - 1);
                    r.k[e] = row[k_at + ic], r.q[e] = row[q_at + ic];
                    if constexpr (CHANNEL) r.d[e] = decays[ic];
                }
            }
        }
        const size_t t = t0 + min(first + min(lane / C, TB - 1), n - 1);
        r.v = qkv[t * ld + v_at + min(vt * C + lane % C, dv - 1)];
        const float* g = gates + t * ldg;
        r.decay = CHANNEL ? 0.f : g[h], r.step = g[n_heads * dn + h];
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int e = 0; e < PER; e += WIDE) {
            const int idx = lane * WIDE + 64 * e, i = idx % KQ;
            const int u = idx / KQ;
            if constexpr (EVERY) {
                float4* to = reinterpret_cast<float4*>(&kq_s[buf][u][i]);
                to[0] = float4{r.k[e], r.q[e], r.k[e + 1], r.q[e + 1]};
                to[1] = float4{r.k[e + 2], r.q[e + 2], r.k[e + 3], r.q[e + 3]};
                if constexpr (CHANNEL) *reinterpret_cast<float4*>(&d_s[buf][u][i]) = float4{r.d[e], r.d[e + 1], r.d[e + 2], r.d[e + 3]};
            } else {
                const int keep = i < dk ? -1 : 0;                     // (zeros beyond the key, without a branch)
                const auto kept = [&](float x) { return __int_as_float(__float_as_int(x) & keep); };
                kq_s[buf][u][i] = float2{kept(r.k[e]), kept(r.q[e])};
                if constexpr (CHANNEL) d_s[buf][u][i] = kept(r.d[e]);
            }
        }
        if (lane < TB * C) own_s[buf][lane / C][lane % C] = float4{r.decay, r.step, r.v, 0.f};
    };
    // k . q of a block's tokens, a token per column of lanes at a time: nothing of the memory is in it, so it does not stand in the tokens' way.
    auto key_queries = [&](int buf) {
#pragma unroll
        for (int j = 0; j < TB; j += C) {
            const int u = min(j + c, TB - 1);
            float2 x[ROWS];
#pragma unroll
            for (int rr = 0; rr < ROWS; ++rr) x[rr] = kq_s[buf][u][rr * RG + rg];
            const float kq = group_sum<16>(delta_key_query<ROWS, CHANNEL>(x));
            if (rg < C) own_s[buf][u][rg].w = kq;
        }
    };
    fetch(0);
    stash(0);
    barrier_lds();
    int buf = 0;
    for (int b0 = 0; b0 < n; b0 += TB, buf ^= 1) {
        const int here = min(TB, n - b0);
        const bool more = b0 + TB < n;
        if (more) fetch(b0 + TB);
        key_queries(buf);
        barrier_lds();
        auto read = [&](int u, DeltaToken<ROWS, CHANNEL>& x) {
#pragma unroll
            for (int rr = 0; rr < ROWS; ++rr) x.kq[rr] = kq_s[buf][u][rr * RG + rg];
            if constexpr (CHANNEL) {
#pragma unroll
                for (int rr = 0; rr < ROWS; ++rr) x.d[rr] = d_s[buf][u][rr * RG + rg];
            }
            x.own = own_s[buf][u][c];
        };
        if (ROWS <= 8 && here == TB) {           // a whole block: straight code, a token's numbers leave LDS while the one before is worked on, the results one store
            float mine = 0.f;                    // (the lanes of a column hold equal results: lane u of it keeps token u's)
            DeltaToken<ROWS, CHANNEL> x[2];
            read(0, x[0]);
#pragma unroll
            for (int u = 0; u < TB; ++u) {
                if (u + 1 < TB) read(u + 1, x[(u + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
                const float y = delta_token<ROWS, CHANNEL>(S, x[u & 1]);
                mine = rg == u ? y : mine;
            }
            asm volatile("" : "+v"(mine));       // (else the read-outs' last steps move behind the branch, three instructions a token for one)
            if (rg < TB && live) out[(size_t)(t0 + b0 + rg) * ldo + h * dv + col] = mine;
        } else {
            for (int u = 0; u < here; ++u) {
                DeltaToken<ROWS, CHANNEL> x;
                read(u, x);
                const float y = delta_token<ROWS, CHANNEL>(S, x);
                if (rg == 0 && live) out[(size_t)(t0 + b0 + u) * ldo + h * dv + col] = y;
            }
        }
        if (more) stash(buf ^ 1);                // (the buffer the block before this one was read from)
        barrier_lds();
    }
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        const int i = rr * RG + rg;
        if (EVERY || i < dk) st[(size_t)i * C + c] = S[rr];
    }
}

// The same for steps in which every request brings one row: nothing is staged, a wave takes its row's numbers as they lie, and a
// workgroup is four waves (tiles).  Every sum in the scan's order: the same bits.
template <int ROWS, bool CHANNEL>
__global__ __launch_bounds__(256) void delta_single_kernel(const float* __restrict__ qkv, long ld, const float* __restrict__ gates,
                                                          const int* __restrict__ seg_start, const int* __restrict__ seg_len,
                                                          const int* __restrict__ row_slot, float* __restrict__ state, long state_stride,
                                                          float* __restrict__ out, long ldo, int n_heads, int n_kv, int dk, int dv) {
    constexpr int C = 4, RG = 16;
    const int seg = blockIdx.x, h = blockIdx.y, vt = blockIdx.z * 4 + (threadIdx.x >> 6), n_tiles = (dv + C - 1) / C;
    const int lane = threadIdx.x & 63, c = lane / RG, rg = lane % RG;
    if (vt >= n_tiles || (seg_len && seg_len[seg] <= 0)) return;
    const size_t t = seg_start ? seg_start[seg] : seg;
    const int col = vt * C + c, kvh = h / (n_heads / n_kv), dn = CHANNEL ? dk : 1;
    float* st = state + (size_t)row_slot[t] * state_stride + ((size_t)h * n_tiles + vt) * ((size_t)dk * C);
    const float* row = qkv + t * ld;
    const float* g = gates + t * n_heads * (dn + 1);
    float S[ROWS];
    DeltaToken<ROWS, CHANNEL> x;
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        const int i = rr * RG + rg, ic = min(i, dk - 1);
        const float s = st[(size_t)ic * C + c], k = row[(n_kv + kvh) * dk + ic], q = row[kvh * dk + ic], d = CHANNEL ? g[h * dk + ic] : 0.f;
        S[rr] = i < dk ? s : 0.f;
        x.kq[rr] = i < dk ? float2{k, q} : float2{0.f, 0.f};
        if constexpr (CHANNEL) x.d[rr] = i < dk ? d : 0.f;
    }
    const float v = row[2 * n_kv * dk + h * dv + min(col, dv - 1)];
    x.own = float4{CHANNEL ? 0.f : g[h], g[n_heads * dn + h], v, group_sum<16>(delta_key_query<ROWS, CHANNEL>(x.kq))};
    const float y = delta_token<ROWS, CHANNEL>(S, x);
    if (rg == 0 && col < dv) out[t * ldo + h * dv + col] = y;
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
        const int i = rr * RG + rg;
        if (i < dk) st[(size_t)i * C + c] = S[rr];
    }
}

// ------------------------------------------------------------------------------------- gated delta rule, a prompt's rows in blocks
// The same rule for requests that bring many rows (keys of 64 channels, one decay a head), by the published chunked form of the delta rule: the block's updates
// in their WY form, from a unit lower triangular system (the UT transform; Yang and others, "Parallelizing Linear Transformers with the Delta Rule over Sequence
// Length", 2024, with the decays of "Gated Delta Networks", 2024).  With d_t the decays, R_ti = d_{i+1} .. d_t and
// g_t = d_0 .. d_t inside a block of 64 rows, S_0 the memory before it, the rule's updates w_t = s_t (v_t - d_t S_{t-1}^T k_t) are the
// solution of (1 + A) W = s (V - g K S_0), A_ti = s_t R_ti (k_t . k_i) below the diagonal.  So with U = (1 + A)^-1 s V and P = (1 + A)^-1 s g K,
// which need no memory,
//     S_64 = g_63 S_0 + (N - M S_0),     M = K'^T P,  N = K'^T U   (K' the keys times R_63,i)
//     O    = Q' S_0 + B U,  Q' = g Q - B P,  B_ti = R_ti (q_t . k_i) up to the diagonal
// and only the first line goes from block to block.  Three kernels: every block's M, N, Q' and B U, all blocks at once; the blocks' memories, one
// product of 64 x 64 a block; Q' S_0 onto B U, all blocks at once.  What is kept is 32-bit, the products are on the matrix instructions of 16 x 16 x 4.  The places
// of k in a matrix instruction are chosen so that a lane's four are neighbours (lane group g takes 4 g + v in instruction v): operands leave LDS and
// memory 16 bytes at a time, and a result as it lies is an operand of the next product.
// Distance to 64 bits: products of decays, k . k, q . k and the keys' products with U and P are summed in 64 bits (the decays' products alone brought the
// memories from 1.2 to 2.5 times the scan's distance down to 0.9), the other sums in parts of 8 or 16 terms that meet in a tree, and what a block
// forgets of a memory is taken off its product with g_63, not multiplied in with it.  1,777 rows: read-outs 1.1e-7 (scan 1.3e-7), memories 0.9e-7 (1.2e-7).
// A product with a block of zeros would spread a number that is no number to rows before its own: blocks with such an input, and all behind
// them, go token by token, as does all of a memory that holds one.
// Bound by the chain of blocks in the second kernel (0.7 us a block) and by a workgroup's matrix instructions and barriers in the first, where it has a compute
// unit to itself.  1,777 rows of 8 heads of 64 x 128: 28, 25 and 10 us, the scan 203; the rule of choice is `ops.delta_chunks_pay`.
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int CHUNK = 64, CHUNK_DK = 64, CHUNK_LD = 68;               // rows of LDS 68 numbers apart: 16 rows' pieces of 16 bytes lie in different banks
constexpr int CHUNK_WAVES = 12;

// (first row, number of rows) of block `index` among the runs of at least `from` rows; rows 0: there are no so many blocks.
struct ChunkPlace { int row, rows; };
__device__ __forceinline__ ChunkPlace chunk_place(const int* __restrict__ seg_start, const int* __restrict__ seg_len, int n_segs, int from, int index) {
    const int lane = threadIdx.x & 63;
    for (int s0 = 0; s0 < n_segs; s0 += 64) {
        const bool there = s0 + lane < n_segs;
        const int n = there ? seg_len[s0 + lane] : 0, start = there ? seg_start[s0 + lane] : 0, mine = n >= from ? (n + CHUNK - 1) / CHUNK : 0;
        int sum = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int other = __shfl_up(sum, off, 64);
            if (lane >= off) sum += other;
        }
        const unsigned long long past = __ballot(sum > index);
        if (past) {
            const int l = __ffsll(past) - 1, block = index - __shfl(sum - mine, l, 64);
            return {__shfl(start, l, 64) + block * CHUNK, min(CHUNK, __shfl(n, l, 64) - block * CHUNK)};
        }
        index -= __shfl(sum, 63, 64);
    }
    return {0, 0};
}
// The blocks of the runs before `run`.
__device__ __forceinline__ int chunks_before(const int* __restrict__ seg_len, int run, int from) {
    const int lane = threadIdx.x & 63;
    int sum = 0;
    for (int s = lane; s < run; s += 64) sum += seg_len[s] >= from ? (seg_len[s] + CHUNK - 1) / CHUNK : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    return sum;
}
__device__ __forceinline__ bool no_number(float x) { return !(fabsf(x) <= 3.402823466e38f); }
__device__ __forceinline__ floatx4 four_of(const float* p) { return *reinterpret_cast<const floatx4*>(p); }
__device__ __forceinline__ void mfma_four(floatx4 a, floatx4 b, floatx4& acc) {
#pragma unroll
    for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[v], b[v], acc, 0, 0, 0);
}

// The same in 64 bits.  Result v of a lane is row 4 v + g of the instruction's there: `spread` names the row to give place c, so that it is row 4 g + v as above.
typedef double doublex4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int spread(int c) { return 4 * (c & 3) + (c >> 2); }
__device__ __forceinline__ void mfma_four(floatx4 a, floatx4 b, doublex4& acc) {
#pragma unroll
    for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[v], (double)b[v], acc, 0, 0, 0);
}
__device__ __forceinline__ floatx4 mfma_part(floatx4 a, floatx4 b) {
    floatx4 acc = floatx4{};
    mfma_four(a, b, acc);
    return acc;
}

// Numbers a block and head leave for the kernels behind: M [64][64], N^T [dv][64], Q' [64][64], S_0^T [dv][64], then g_63, whether the
// block goes token by token (0 or 1), and two unused.
__host__ __device__ constexpr long chunk_floats(int dv) { return 2L * CHUNK_DK * (CHUNK + dv) + 4; }

// One workgroup per (block, head): a wave takes columns of [V | K], 16 at a time, from the solution to everything made of it.
__global__ __launch_bounds__(64 * CHUNK_WAVES) void delta_chunk_prepare_kernel(const float* __restrict__ qkv, long ld, const float* __restrict__ gates, const int* __restrict__ seg_start,
                                                                               const int* __restrict__ seg_len, int n_segs, int from, float* __restrict__ scratch,
                                                                               float* __restrict__ out, long ldo, int n_heads, int n_kv, int dv) {
    __shared__ __attribute__((aligned(16))) float Ks[CHUNK][CHUNK_LD], Qs[CHUNK][CHUNK_LD], KT[CHUNK_DK][CHUNK_LD], As[CHUNK][CHUNK_LD], Bs[CHUNK][CHUNK_LD];
    __shared__ float step_s[CHUNK], since_s[CHUNK], last_s[CHUNK];     // s, g and R_63
    const int h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4, n_waves = blockDim.x >> 6;
    const ChunkPlace at = chunk_place(seg_start, seg_len, n_segs, from, blockIdx.x);
    if (at.rows <= 0) return;
    const int n = at.rows, kvh = h / (n_heads / n_kv), v_tiles = dv / 16;
    const size_t t0 = at.row;
    const float *q_rows = qkv + t0 * ld + kvh * CHUNK_DK, *k_rows = q_rows + n_kv * CHUNK_DK, *v_rows = qkv + t0 * ld + 2 * n_kv * CHUNK_DK + h * dv;
    float* mine = scratch + ((size_t)blockIdx.x * n_heads + h) * chunk_floats(dv);
    float *M = mine, *NT = M + CHUNK_DK * CHUNK_DK, *Qp = NT + (size_t)dv * CHUNK_DK;

    bool bad = false;
    for (int i = tid; i < CHUNK * CHUNK_DK / 4; i += blockDim.x) {                      // rows behind the run's last: zeros, and decays of 1
        const int t = i / (CHUNK_DK / 4), d = i % (CHUNK_DK / 4) * 4;
        floatx4 k = floatx4{}, q = floatx4{};
        if (t < n) k = four_of(k_rows + (size_t)t * ld + d), q = four_of(q_rows + (size_t)t * ld + d);
#pragma unroll
        for (int v = 0; v < 4; ++v) bad |= no_number(k[v]) || no_number(q[v]);
        *reinterpret_cast<floatx4*>(&Ks[t][d]) = k;
        *reinterpret_cast<floatx4*>(&Qs[t][d]) = q;
    }
    floatx4 x[4];                                                                       // x[I][v]: row 16 I + 4 g + v, column 16 tile + c
    const auto fetch_values = [&](int tile) {
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
            for (int v = 0; v < 4; ++v) x[I][v] = v_rows[(size_t)min(16 * I + 4 * g + v, n - 1) * ld + 16 * tile + c];
    };
    for (int tile = wave + n_waves; tile < v_tiles; tile += n_waves) {
        fetch_values(tile);
#pragma unroll
        for (int e = 0; e < 16; ++e) bad |= no_number(x[e / 4][e % 4]);
    }
    fetch_values(min(wave, v_tiles - 1));                                               // (the wave's first columns stay)
    if (wave == n_waves - 1) {
        const float* at_t = gates + (t0 + min(lane, n - 1)) * 2 * n_heads;
        const float d = lane < n ? at_t[h] : 1.f, s = lane < n ? at_t[n_heads + h] : 0.f;
        bad |= no_number(d) || no_number(s);
        // R's column `lane` into B's place, and g: products of up to 64 decays, in 64 bits (their error is that of everything that is kept)
        double r = 0., since = 1., mine_since = 0.;
#pragma unroll
        for (int t = 0; t < CHUNK; ++t) {
            const double dt = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d), t));
            r = t == lane ? 1. : r * dt;
            since *= dt;
            mine_since = t == lane ? since : mine_since;
            Bs[t][lane] = (float)r;
        }
        step_s[lane] = s, since_s[lane] = (float)mine_since, last_s[lane] = (float)r;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) bad |= no_number(x[e / 4][e % 4]);
    bad = __syncthreads_or(bad);
    if (tid == 0) *reinterpret_cast<float2*>(mine + 2L * CHUNK_DK * (CHUNK + dv)) = float2{since_s[CHUNK - 1], bad ? 1.f : 0.f};
    if (bad) return;
    // A and B, 16 x 16 at a time, on and below the diagonal; the keys' transpose
    for (int block = wave; block < 10; block += n_waves) {
        const int I = block < 1 ? 0 : block < 3 ? 1 : block < 6 ? 2 : 3, J = block - I * (I + 1) / 2;
        const auto sums = [&](const float (*rows)[CHUNK_LD]) {
            doublex4 sum = {};
#pragma unroll
            for (int m = 0; m < 4; ++m) mfma_four(four_of(&rows[16 * I + spread(c)][16 * m + 4 * g]), four_of(&Ks[16 * J + c][16 * m + 4 * g]), sum);
            return floatx4{(float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]};
        };
        const floatx4 k_sum = sums(Ks);
        __builtin_amdgcn_sched_barrier(0);                                              // (else both sums' parts want registers at once; likewise below)
        const floatx4 q_sum = sums(Qs);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 16 * I + 4 * g + v, i = 16 * J + c;
            const float r = Bs[t][i];
            As[t][i] = t > i ? -(step_s[t] * (r * k_sum[v])) : 0.f;
            Bs[t][i] = t >= i ? r * q_sum[v] : 0.f;
        }
    }
    for (int i = tid; i < CHUNK * CHUNK_DK; i += blockDim.x) {
        const int t = i % CHUNK, d = i / CHUNK;
        KT[d][t] = Ks[t][d] * last_s[t];
    }
    __syncthreads();
    // the inverses of the diagonal's blocks, a column a lane, in place
    if (wave < 4) {
        floatx4 row[4];                                                                 // a lane holds row c
#pragma unroll
        for (int m = 0; m < 4; ++m) row[m] = four_of(&As[16 * wave + c][16 * wave + 4 * m]);
        float y[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float sum = t == c ? 1.f : 0.f;
#pragma unroll
            for (int i = 0; i < t; ++i) sum = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(row[i / 4][i % 4]), t)), y[i], sum);
            y[t] = sum;
        }
        if (g == 0) {
#pragma unroll
            for (int t = 0; t < 16; ++t) As[16 * wave + t][16 * wave + c] = y[t];
        }
    }
    __syncthreads();
    for (int tile = wave; tile < v_tiles + CHUNK_DK / 16; tile += n_waves) {
        const bool values = tile < v_tiles;
        const int col0 = 16 * (values ? tile : tile - v_tiles);
        if (values && tile != wave) fetch_values(tile);
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
            for (int v = 0; v < 4; ++v) {                                               // (step sizes behind the run's last row are 0)
                const int t = 16 * I + 4 * g + v;
                x[I][v] = values ? step_s[t] * x[I][v] : (step_s[t] * since_s[t]) * Ks[t][col0 + c];
            }
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            floatx4 part = floatx4{};
#pragma unroll
            for (int J = 0; J < I; ++J) part += mfma_part(four_of(&As[16 * I + c][16 * J + 4 * g]), x[J]);
            x[I] = mfma_part(four_of(&As[16 * I + c][16 * I + 4 * g]), x[I] + part);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < CHUNK_DK / 16; ++r) {
            doublex4 sum = {};
            // values: [v] is key channel 16 r + 4 g + v, column col0 + c; keys: column col0 + 4 v + g, key channel 16 r + c
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const floatx4 k = four_of(&KT[16 * r + (values ? spread(c) : c)][16 * m + 4 * g]);
                if (values) mfma_four(k, x[m], sum);
                else mfma_four(x[m], k, sum);
            }
            if (values) *reinterpret_cast<floatx4*>(NT + (size_t)(col0 + c) * CHUNK_DK + 16 * r + 4 * g) = floatx4{(float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]};
            else {
#pragma unroll
                for (int v = 0; v < 4; ++v) M[(size_t)(16 * r + c) * CHUNK_DK + col0 + 4 * v + g] = (float)sum[v];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            floatx4 acc = floatx4{};                                                    // acc[v]: column col0 + 4 g + v, row 16 I + c
#pragma unroll
            for (int m = 0; m <= I; ++m) acc += mfma_part(x[m], four_of(&Bs[16 * I + c][16 * m + 4 * g]));
            const int t = 16 * I + c;
            if (!values) {
                const floatx4 q = four_of(&Qs[t][col0 + 4 * g]);
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = since_s[t] * q[v] - acc[v];
                *reinterpret_cast<floatx4*>(Qp + (size_t)t * CHUNK_DK + col0 + 4 * g) = acc;
            } else if (t < n) {
                *reinterpret_cast<floatx4*>(out + (t0 + t) * ldo + h * dv + col0 + 4 * g) = acc;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The memories from block to block: one workgroup of four waves per (run, head, 16 columns), 16 rows a wave; the blocks' M and N come
// CHUNK_AHEAD blocks ahead (they were just written by other compute dies and come from beyond the L2: two ahead 1.1 us a block).
constexpr int CHUNK_AHEAD = 6;
__global__ __launch_bounds__(256) void delta_chunk_scan_kernel(const float* __restrict__ qkv, long ld, const float* __restrict__ gates, const int* __restrict__ seg_start,
                                                               const int* __restrict__ seg_len, int from, const int* __restrict__ row_slot, float* __restrict__ state, long state_stride,
                                                               float* __restrict__ scratch, int* __restrict__ by_token, float* __restrict__ out, long ldo,
                                                               int n_heads, int n_kv, int dv) {
    __shared__ __attribute__((aligned(16))) float St[2][16][CHUNK_LD];                  // [column][key channel]
    const int run = blockIdx.x, h = blockIdx.y, tile = blockIdx.z, n_tiles = gridDim.z;
    const int n = seg_len[run];
    if (n < from) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int before = chunks_before(seg_len, run, from), n_chunks = (n + CHUNK - 1) / CHUNK;
    const size_t t0 = seg_start[run], per = chunk_floats(dv);
    float* st = state + (size_t)row_slot[t0] * state_stride + ((size_t)h * (dv / 4) + tile * 4) * (CHUNK_DK * 4);       // [four columns][key channel][4]
    const size_t step = (size_t)n_heads * per;
    float* base = scratch + ((size_t)before * n_heads + h) * per;
    const float *M = base + (size_t)(16 * wave + c) * CHUNK_DK + 4 * g;
    const size_t in_tile = (size_t)(16 * tile + c) * CHUNK_DK + 16 * wave + 4 * g;
    const float* NT = base + CHUNK_DK * CHUNK_DK + in_tile;
    float* S0 = base + CHUNK_DK * (2 * CHUNK_DK + (size_t)dv) + in_tile;
    const float* word = base + 2L * CHUNK_DK * (CHUNK + dv);
    struct Ahead { floatx4 m[4], n; float since; } ahead[CHUNK_AHEAD];
    int by_lane = 0;                                       // (a vector load: scalar ones come back in any order, so each would be waited for with the newest)
    asm volatile("" : "+v"(by_lane));
    auto fetch = [&](int b, Ahead& x) {
        const size_t off = min(b, n_chunks - 1) * step;
#pragma unroll
        for (int i = 0; i < 4; ++i) x.m[i] = four_of(M + off + 16 * i);
        x.n = four_of(NT + off);
        x.since = word[off + by_lane];
    };
#pragma unroll
    for (int b = 0; b < CHUNK_AHEAD; ++b) fetch(b, ahead[b]);
    floatx4 own;
#pragma unroll
    for (int v = 0; v < 4; ++v) own[v] = st[((size_t)(c / 4) * CHUNK_DK + 16 * wave + 4 * g + v) * 4 + c % 4];
    *reinterpret_cast<floatx4*>(&St[0][c][16 * wave + 4 * g]) = own;
    // the blocks up to the first that goes token by token (found beforehand: with a choice in it the loop would wait for every load in flight)
    int n_fast = 0;
    for (bool all = true; all && n_fast < n_chunks;) {
        const unsigned long long slow = __ballot(n_fast + lane < n_chunks && word[(size_t)min(n_fast + lane, n_chunks - 1) * step + 1] != 0.f);
        n_fast = min(n_chunks, n_fast + (slow ? __ffsll(slow) - 1 : 64));
        all = !slow;
    }
    if (__syncthreads_or(no_number(own[0]) || no_number(own[1]) || no_number(own[2]) || no_number(own[3]))) n_fast = 0;
    n_fast = __builtin_amdgcn_readfirstlane(n_fast);
    for (int b = tid; b < n_chunks; b += 256) by_token[((size_t)(before + b) * n_heads + h) * n_tiles + tile] = b >= n_fast;
    auto block = [&](int b, Ahead& x) {
        const int buf = b & 1;
        *reinterpret_cast<floatx4*>(S0 + b * step) = own;
        floatx4 part[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) part[i] = mfma_part(x.m[i], four_of(&St[buf][c][16 * i + 4 * g]));
        const floatx4 put = x.n - ((part[0] + part[1]) + (part[2] + part[3]));
#pragma unroll
        for (int v = 0; v < 4; ++v) own[v] = fmaf(x.since, own[v], put[v]);
        *reinterpret_cast<floatx4*>(&St[buf ^ 1][c][16 * wave + 4 * g]) = own;
        fetch(b + CHUNK_AHEAD, x);
        barrier_lds();
    };
    for (int b = 0;; b += CHUNK_AHEAD) {
#pragma unroll
        for (int i = 0; i < CHUNK_AHEAD; ++i) {
            if (b + i >= n_fast) goto walked;
            block(b + i, ahead[i]);
        }
    }
walked:
    if (n_fast < n_chunks) {
        const int col = tid >> 4, rg = tid & 15, kvh = h / (n_heads / n_kv);
        float S[4];
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) S[rr] = St[n_fast & 1][col][16 * rr + rg];
        for (size_t t = t0 + n_fast * CHUNK; t < t0 + n; ++t) {
            const float* row = qkv + t * ld;
            DeltaToken<4, false> x;
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) x.kq[rr] = float2{row[(n_kv + kvh) * CHUNK_DK + 16 * rr + rg], row[kvh * CHUNK_DK + 16 * rr + rg]};
            x.own = float4{gates[t * 2 * n_heads + h], gates[t * 2 * n_heads + n_heads + h], row[2 * n_kv * CHUNK_DK + h * dv + tile * 16 + col],
                           group_sum<16>(delta_key_query<4, false>(x.kq))};
            const float y = delta_token<4, false>(S, x);
            if (rg == 0) out[t * ldo + h * dv + tile * 16 + col] = y;
        }
        __syncthreads();
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) St[0][col][16 * rr + rg] = S[rr];
        __syncthreads();
        own = four_of(&St[0][c][16 * wave + 4 * g]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) st[((size_t)(c / 4) * CHUNK_DK + 16 * wave + 4 * g + v) * 4 + c % 4] = own[v];
}

// Q' S_0 onto the blocks' read-outs: one workgroup per (block, head), a wave per 16 columns.
__global__ __launch_bounds__(512) void delta_chunk_read_kernel(const int* __restrict__ seg_start, const int* __restrict__ seg_len, int n_segs, int from, const float* __restrict__ scratch,
                                                               const int* __restrict__ by_token, float* __restrict__ out, long ldo, int n_heads, int dv) {
    const int h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4, n_tiles = dv / 16, n_waves = blockDim.x >> 6;
    const float* mine = scratch + ((size_t)blockIdx.x * n_heads + h) * chunk_floats(dv);
    const float *Qp = mine + CHUNK_DK * (CHUNK_DK + (size_t)dv), *S0 = Qp + CHUNK * CHUNK_DK;
    floatx4 s[4], q[4][4];                                 // (asked for before the block's rows are known)
    const auto fetch = [&](int tile) {
#pragma unroll
        for (int m = 0; m < 4; ++m) s[m] = four_of(S0 + (size_t)(16 * tile + c) * CHUNK_DK + 16 * m + 4 * g);
    };
    fetch(wave);
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int m = 0; m < 4; ++m) q[I][m] = four_of(Qp + (size_t)(16 * I + c) * CHUNK_DK + 16 * m + 4 * g);
    const ChunkPlace at = chunk_place(seg_start, seg_len, n_segs, from, blockIdx.x);
    for (int tile = wave; tile < n_tiles && at.rows > 0; tile += n_waves) {
        if (tile != wave) fetch(tile);
        const int slow = by_token[((size_t)blockIdx.x * n_heads + h) * n_tiles + tile];
        floatx4 block[4];
        float* to[4];
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            to[I] = out + ((size_t)at.row + min(16 * I + c, at.rows - 1)) * ldo + h * dv + 16 * tile + 4 * g;
            block[I] = four_of(to[I]);
        }
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            floatx4 part[8] = {};
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int v = 0; v < 4; ++v) part[2 * m + v / 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[m][v], q[I][m][v], part[2 * m + v / 2], 0, 0, 0);
            const floatx4 sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
            if (16 * I + c < at.rows && !slow) *reinterpret_cast<floatx4*>(to[I]) = sum + block[I];
        }
    }
}

}  // namespace

GI_API int gi_segments(const int* slot, const int* pos, int n_rows, int* seg_start, int* seg_len, int n_segs, hipStream_t stream) {
    GI_REQUIRE(n_rows > 0 && n_segs > 0 && n_segs <= n_rows, "segments: %d rows in %d runs", n_rows, n_segs);
    segments_kernel<<<1, n_rows > 64 ? 1024 : 64, 0, stream>>>(slot, pos, n_rows, seg_start, seg_len, n_segs);
    GI_CHECK_LAUNCH("segments");
    return 0;
}

// Floats of one request slot's state for `n_heads` heads of dk x dv: per head and tile of three value channels, [dk][4] and m (padded to 4).
GI_API long gi_mlstm_state_floats(int n_heads, int dk, int dv) {
    return (long)n_heads * ((dv + 2) / 3) * ((long)dk * 4 + 4);
}

GI_API int gi_mlstm_max_key_dim() { return 512; }

// proj: float32 [n_rows, ld], whose columns q_off.. hold q [heads*dk], k_off.. k [heads*dk], v_off.. v [heads*dv], i_off.. and
// f_off.. the gates' pre-activations [heads]; out: float32 [n_rows, ldo] gets the heads' sums S^T q [heads*dv], den: float32
// [n_rows, heads] what each head's sums are to be divided by (o = out / den); state: [slots, state_stride].
GI_API int gi_mlstm_scan(const float* proj, long ld, int q_off, int k_off, int v_off, int i_off, int f_off, const float* i_bias, const float* f_bias,
                         float cap, float q_scale, const int* seg_start, const int* seg_len, int n_segs, const int* row_slot, float* state,
                         long state_stride, float* out, long ldo, float* den, int n_heads, int dk, int dv, hipStream_t stream) {
    GI_REQUIRE(den != nullptr, "mlstm_scan: the divisors need a place");
    GI_REQUIRE(n_segs > 0 && n_heads > 0 && dk > 0 && dk <= 512 && dv > 0, "mlstm_scan: bad sizes (runs %d, heads %d, dk %d, dv %d; dk at most 512)", n_segs, n_heads, dk, dv);
    GI_REQUIRE(cap > 0.f && state_stride >= gi_mlstm_state_floats(n_heads, dk, dv) && ldo >= (long)n_heads * dv, "mlstm_scan: bad cap, state stride or output stride");
    const int tiles = (dv + 2) / 3;
    GI_REQUIRE(n_heads <= 65535 && tiles <= 65535, "mlstm_scan: too many heads or value channels");
    dim3 grid(n_segs, n_heads, tiles);
#define GO(R) mlstm_scan_kernel<R><<<grid, 64, 0, stream>>>(proj, ld, q_off, k_off, v_off, i_off, f_off, i_bias, f_bias, cap, q_scale, seg_start, seg_len, \
                                                           row_slot, state, state_stride, out, ldo, den, dk, dv)
    if (dk <= 64) GO(4); else if (dk <= 128) GO(8); else if (dk <= 256) GO(16); else GO(32);
#undef GO
    GI_CHECK_LAUNCH("mlstm_scan");
    return 0;
}

// Floats of one request slot's state of the gated delta rule: the memories, per head and tile of four value channels [dk][4],
// then the convolutions' tail [n_taps - 1][2 n_kv dk + n_heads dv].
GI_API long gi_delta_memory_floats(int n_heads, int dk, int dv) { return (long)n_heads * ((dv + 3) / 4) * ((long)dk * 4); }
GI_API long gi_delta_state_floats(int n_heads, int n_kv, int dk, int dv, int n_taps) {
    return gi_delta_memory_floats(n_heads, dk, dv) + (long)(n_taps - 1) * (2L * n_kv * dk + (long)n_heads * dv);
}
GI_API int gi_delta_max_key_dim() { return 512; }
GI_API int gi_delta_max_taps() { return DELTA_MAX_TAPS; }

// proj: float32 [n_rows, ld]; see delta_prepare_kernel.  state: [slots, state_stride], a slot's memories then its tail.
// pre_a: float32 [n_rows, lda], the decays' pre-activations, one a head, or (channel != 0) one a head and key channel; or low: float32 rows
// of proj's stride with `rank` numbers each, and w_up bfloat16 [heads or heads*dk][rank], from which they are made here.
GI_API int gi_delta_prepare(const float* proj, long ld, int conv_off, const float* pre_a, long lda, int b_off, const float* taps, int n_taps, const float* a_log,
                            const float* dt_bias, const int* slot, const int* pos, float* state, long state_stride, float* qkv, float* gates,
                            int n_rows, int n_heads, int n_kv, int dk, int dv, float q_scale, int move_tail, int channel, const float* low, int rank, const void* w_up,
                            hipStream_t stream) {
    const int dn = channel ? dk : 1;
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0 && dk > 0 && dv > 0, "delta_prepare: bad sizes (rows %d, heads %d, kv heads %d, dk %d, dv %d)",
               n_rows, n_heads, n_kv, dk, dv);
    GI_REQUIRE(n_taps >= 1 && n_taps <= DELTA_MAX_TAPS, "delta_prepare: %d taps, 1 to %d are served", n_taps, DELTA_MAX_TAPS);
    const long n_conv = 2L * n_kv * dk + (long)n_heads * dv;
    GI_REQUIRE(conv_off >= 0 && b_off >= 0 && ld >= conv_off + n_conv && ld >= b_off + n_heads, "delta_prepare: the columns named lie outside the rows");
    GI_REQUIRE(low != nullptr ? (rank > 0 && w_up != nullptr) : (pre_a != nullptr && lda >= (long)n_heads * dn), "delta_prepare: the decays' inputs are missing or too short");
    GI_REQUIRE(state_stride >= gi_delta_state_floats(n_heads, n_kv, dk, dv, n_taps) && 2 * n_kv + 2 * n_heads <= 65535, "delta_prepare: state stride %ld too small, or too many heads", state_stride);
    dim3 grid(n_rows, 2 * n_kv + n_heads + (dn > 1 ? n_heads : 1));
    float* tail = state + gi_delta_memory_floats(n_heads, dk, dv);
    const bool common = dn == 1 && low == nullptr && n_taps <= PREPARE_TAPS && dk <= 64;
    if (common && move_tail && n_taps >= 2 && dv <= 128) {
        delta_prepare_single_kernel<<<grid, 64, 0, stream>>>(proj, ld, conv_off, pre_a, lda, b_off, taps, n_taps, tail, state_stride, a_log, dt_bias, slot, qkv, gates, n_heads, n_kv, dk,
                                                             dv, q_scale);
        GI_CHECK_LAUNCH("delta_prepare (single rows)");
        return 0;
    }
    if (common && !move_tail && n_rows >= 64) {
        delta_prepare_rows_kernel<<<dim3((n_rows + PREPARE_ROWS - 1) / PREPARE_ROWS, (2 * n_kv + n_heads + 1 + 3) / 4), 256, 0, stream>>>(
            proj, ld, conv_off, pre_a, lda, b_off, taps, n_taps, tail, state_stride, a_log, dt_bias, slot, pos, qkv, gates, n_rows, n_heads, n_kv, dk, dv, q_scale);
        GI_CHECK_LAUNCH("delta_prepare (rows)");
        return 0;
    }
    delta_prepare_kernel<<<grid, 64, 0, stream>>>(proj, ld, conv_off, pre_a, lda, b_off, taps, n_taps, tail, state_stride, move_tail,
                                                  a_log, dt_bias, slot, pos, qkv, gates, n_heads, n_kv, dk, dv, q_scale, dn, low, rank, (const bf16_t*)w_up);
    GI_CHECK_LAUNCH("delta_prepare");
    return 0;
}

GI_API int gi_delta_tail(const float* proj, long ld, int conv_off, int n_taps, const int* seg_start, const int* seg_len, int n_segs, const int* slot,
                         float* state, long state_stride, int n_heads, int n_kv, int dk, int dv, hipStream_t stream) {
    GI_REQUIRE(n_segs > 0 && n_taps >= 1 && n_taps <= DELTA_MAX_TAPS, "delta_tail: %d runs, %d taps", n_segs, n_taps);
    const long n_conv = 2L * n_kv * dk + (long)n_heads * dv;
    GI_REQUIRE(conv_off >= 0 && ld >= conv_off + n_conv && state_stride >= gi_delta_state_floats(n_heads, n_kv, dk, dv, n_taps), "delta_tail: columns outside the rows, or state stride too small");
    if (n_taps == 1) return 0;
    delta_tail_kernel<<<dim3(n_segs, n_conv < 256L * 64 ? (unsigned)((n_conv + 255) / 256) : 64), 256, 0, stream>>>(proj, ld, conv_off, (int)n_conv, n_taps, seg_start, seg_len, slot, state + gi_delta_memory_floats(n_heads, dk, dv), state_stride);
    GI_CHECK_LAUNCH("delta_tail");
    return 0;
}

// qkv: float32 [n_rows, ld], a row's unit queries [n_kv][dk], unit keys [n_kv][dk], values [n_heads][dv]; gates: float32 [n_rows, 2 n_heads],
// or [n_rows, n_heads dk + n_heads] with a decay per head and key channel (channel != 0); with `single`, seg_start and seg_len null: run i is row i;
// out: float32 [n_rows, ldo] gets the heads' read-outs [n_heads][dv].  below > 0: only the runs of fewer rows than that (not with `single`).
GI_API int gi_delta_scan(const float* qkv, long ld, const float* gates, const int* seg_start, const int* seg_len, int n_segs, const int* row_slot,
                         float* state, long state_stride, float* out, long ldo, int n_heads, int n_kv, int dk, int dv, int channel, int single, int below, hipStream_t stream) {
    GI_REQUIRE(n_segs > 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0 && dk > 0 && dk <= 512 && dv > 0, "delta_scan: bad sizes (runs %d, heads %d, kv heads %d, dk %d, dv %d; dk at most 512)",
               n_segs, n_heads, n_kv, dk, dv);
    GI_REQUIRE(ld >= 2L * n_kv * dk + (long)n_heads * dv && ldo >= (long)n_heads * dv && state_stride >= gi_delta_memory_floats(n_heads, dk, dv), "delta_scan: row or state strides too small");
    const int tiles = (dv + 3) / 4;
    GI_REQUIRE(n_heads <= 65535 && tiles <= 65535, "delta_scan: too many heads or value channels");
    GI_REQUIRE((seg_start == nullptr) == (seg_len == nullptr) && (seg_start != nullptr || single), "delta_scan: the runs of a step that is not of single rows are missing");
    dim3 grid(n_segs, n_heads, tiles);
#define ARGS qkv, ld, gates, seg_start, seg_len, row_slot, state, state_stride, out, ldo, n_heads, n_kv, dk, dv
    const bool aligned = ld % 4 == 0 && ((uintptr_t)qkv & 15) == 0 && (!channel || (((long)n_heads * (dk + 1)) % 4 == 0 && ((uintptr_t)gates & 15) == 0));
#define KIND(R, CH)                                                                                                             \
    do {                                                                                                                        \
        if (single) delta_single_kernel<R, CH><<<dim3(n_segs, n_heads, (tiles + 3) / 4), 256, 0, stream>>>(ARGS);               \
        else if (aligned && dk == 16 * R) delta_scan_kernel<R, CH, true><<<grid, 64, 0, stream>>>(ARGS, below);                        \
        else delta_scan_kernel<R, CH, false><<<grid, 64, 0, stream>>>(ARGS, below);                                                    \
    } while (0)
#define GO(R) do { if (channel) KIND(R, true); else KIND(R, false); } while (0)
    if (dk <= 32) GO(2); else if (dk <= 64) GO(4); else if (dk <= 128) GO(8); else if (dk <= 256) GO(16); else GO(32);
#undef GO
#undef KIND
#undef ARGS
    GI_CHECK_LAUNCH("delta_scan");
    return 0;
}

// The runs of at least `from` rows, in blocks of 64 (delta_chunk_prepare_kernel); n_chunks: their blocks together.  Keys of 64 channels, one decay a head,
// values of a multiple of 16 channels, rows of qkv and out at multiples of 16 bytes.  scratch: float32, gi_delta_chunk_floats(n_chunks, n_heads, dv) numbers,
// at a multiple of 16 bytes.
GI_API long gi_delta_chunk_floats(int n_chunks, int n_heads, int dv) { return (long)n_chunks * n_heads * (chunk_floats(dv) + dv / 16); }
GI_API int gi_delta_chunks(const float* qkv, long ld, const float* gates, const int* seg_start, const int* seg_len, int n_segs, int from, int n_chunks, const int* row_slot,
                           float* state, long state_stride, float* scratch, float* out, long ldo, int n_heads, int n_kv, int dv, hipStream_t stream) {
    GI_REQUIRE(n_segs > 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0 && dv > 0 && dv % 16 == 0 && from > 0 && n_chunks > 0,
               "delta_chunks: bad sizes (runs %d, heads %d, kv heads %d, dv %d, from %d rows, %d blocks)", n_segs, n_heads, n_kv, dv, from, n_chunks);
    GI_REQUIRE(ld >= 2L * n_kv * CHUNK_DK + (long)n_heads * dv && ldo >= (long)n_heads * dv && state_stride >= gi_delta_memory_floats(n_heads, CHUNK_DK, dv),
               "delta_chunks: row or state strides too small");
    GI_REQUIRE(ld % 4 == 0 && ldo % 4 == 0 && (((uintptr_t)qkv | (uintptr_t)out | (uintptr_t)scratch) & 15) == 0, "delta_chunks: rows must lie at multiples of 16 bytes");
    GI_REQUIRE(n_heads <= 65535 && dv / 16 <= 65535, "delta_chunks: too many heads or value channels");
    int* by_token = (int*)(scratch + (long)n_chunks * n_heads * chunk_floats(dv));
    const int tiles = dv / 16, waves = tiles + CHUNK_DK / 16 < CHUNK_WAVES ? tiles + CHUNK_DK / 16 : CHUNK_WAVES;
    delta_chunk_prepare_kernel<<<dim3(n_chunks, n_heads), 64 * waves, 0, stream>>>(qkv, ld, gates, seg_start, seg_len, n_segs, from, scratch, out, ldo, n_heads, n_kv, dv);
    GI_CHECK_LAUNCH("delta_chunks");
    delta_chunk_scan_kernel<<<dim3(n_segs, n_heads, tiles), 256, 0, stream>>>(qkv, ld, gates, seg_start, seg_len, from, row_slot, state, state_stride, scratch, by_token, out, ldo,
                                                                              n_heads, n_kv, dv);
    GI_CHECK_LAUNCH("delta_chunks");
    delta_chunk_read_kernel<<<dim3(n_chunks, n_heads), 64 * (tiles < 8 ? tiles : 8), 0, stream>>>(seg_start, seg_len, n_segs, from, scratch, by_token, out, ldo, n_heads, dv);
    GI_CHECK_LAUNCH("delta_chunks");
    return 0;
}

GI_API int gi_head_norm_gate(const float* o, long ldo, const float* den, const float* g, long ldg, const void* w, int w_dtype, void* y, int y_dtype, long ldy, int n_rows,
                             int n_heads, int dv, float eps, int shared_weight, int gate_act, const float* low, int rank, const void* w_up, hipStream_t stream) {
    GI_REQUIRE(low != nullptr ? (rank > 0 && w_up != nullptr && ldg >= rank) : g != nullptr, "head_norm_gate: the gates' inputs are missing");
    GI_REQUIRE(n_rows > 0 && n_heads > 0 && n_heads <= 65535 && dv > 0, "head_norm_gate: bad sizes (rows %d, heads %d, dv %d)", n_rows, n_heads, dv);
    GI_REQUIRE(gate_act == 0 || gate_act == 1, "head_norm_gate: the gate is a sigmoid (0) or SiLU (1)");
    dim3 grid(n_rows, n_heads);
    const int w_head_stride = shared_weight ? 0 : dv;
#define GO_NT(TW, TO, NT) head_norm_gate_kernel<TW, TO, NT><<<grid, NT, 0, stream>>>(o, ldo, den, g, ldg, (const TW*)w, (TO*)y, ldy, n_heads, dv, eps, w_head_stride, gate_act, low, rank, (const bf16_t*)w_up)
#define GO(TW, TO)                           \
    do {                                     \
        if (low && dv > 64) GO_NT(TW, TO, 256); \
        else GO_NT(TW, TO, 64);              \
    } while (0)
    if (w_dtype == GI_F32 && y_dtype == GI_F32) GO(float, float);
    else if (w_dtype == GI_F32 && y_dtype == GI_BF16) GO(float, bf16_t);
    else if (w_dtype == GI_BF16 && y_dtype == GI_BF16) GO(bf16_t, bf16_t);
    else if (w_dtype == GI_BF16 && y_dtype == GI_F32) GO(bf16_t, float);
    else return gi_fail("head_norm_gate: unknown dtypes %d, %d", w_dtype, y_dtype);
#undef GO
#undef GO_NT
    GI_CHECK_LAUNCH("head_norm_gate");
    return 0;
}
