// The matrix states of picolm_call_state_scan (mixers.h) without a walk token by token: a decode step in one
// kernel, and a prompt in chunks of 64 tokens whose work is products on the matrix cores in 32-bit
// (v_mfma_f32_16x16x4_f32: float operands, float sums).  Sizes: keys of 64 or 128, values in multiples of 16
// (32 in a decode step); others are walked (mixers.hip).
//
// A chunk, with p_i the product of its decays up to token i and D_ij that of those behind j up to i:
//   u_t = w_t (v_t - p_t S0^T k_t - sum_(j < t) D_tj (k_j . k_t) u_j)      (delta rule)
//   u_t = w_t v_t                                                            (outer product)
//   o_i = p_i S0^T q_i + sum_(j <= i) D_ij (q_i . k_j) u_j,    S_end = p_C S0 + sum_j D_Cj k_j u_j^T
// The delta rule's u is a triangular system, (I + T) U = diag(w) V - diag(w p) K S0 with T_tj = w_t D_tj (k_j . k_t):
// X = (I + T)^-1 comes from its blocks of 16 (each turned over column by column; the blocks below the
// diagonal, -X_II sum_K T_IK X_KJ, are products), and U = X diag(w) V - (X diag(w p) K) S0.  Every factor is a product
// of decays; nothing is divided by one.  (The chunked form of the delta rule is that of Yang, Wang, Zhang, Shen and Kim, "Parallelizing
// Linear Transformers with the Delta Rule over Sequence Length", 2024; inverting a unit lower triangle by blocks is textbook.)  Two kernels:
//   prepare  per (sequence, chunk, head), side by side: A_ij = D_ij (q_i . k_j), and for the delta rule
//            -X diag(w p) K and X diag(w) V; p and D_C.  A token's share of them is a row of scratch memory.
//   walk     per (sequence, head, 16 or 32 value columns), chunk by chunk in order: U, the outputs, and the next
//            state, which stays in LDS.
// Bound by the walk's chain, 8.7 us a chunk: three products (3 us of the matrix cores), two meetings of the waves, and the
// chunk's operands from L2 and beyond (115 KB; asked for a chunk ahead it was no faster, and where two
// workgroups share a CU slower: 204 against 160 us).  (Counted: the matrix cores 20 to 30 % busy, 42 % of the LDS cycles bank conflicts.)  Four prompts of 301 to 1,203 tokens: a layer of 16 heads of 128 x 128
// with the delta rule 253 us (the walk in chunks of its own, in mixers.hip, 1,087), of 64 heads of 128 x 64 with outer
// products 230 (1,160); a decode step of four sequences 7.9 and 6.9 us (26.6 and 22.8 with the kernel that prepares).
#include "mixers.h"

#include "api.h"
#include "common.h"
#include "gemm_mfma.h"

#define SC_LEN 64                   // tokens of a chunk
#define SC_LD (SC_LEN + 4)          // rows of 64 floats in LDS: 16 rows of a chunk column, or four adjacent rows of 16 columns, touch every bank once

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }

struct StateChunks {
    const float* in;         // rows with the raw decays and strengths (a decode step)
    const float* qkv;
    const float* aw;         // rows [2 heads]: decay and strength of every head (a prompt)
    float* scratch;          // rows [heads][per]: A_i [64] | W_i [key_dim] | U_i [value_dim] | p_i, D_Ci
    float* out;
    float* state;
    const float* skip;
    const float* A_log;
    const float* dt_bias;
    const int32_t* cu_seqlens;
    const int32_t* seq_slot;
    int64_t slot_floats;
    int in_stride, a_off, w_off, qkv_stride, q_off, k_off, v_off;
    int heads, key_heads, value_dim, chunks_per_seq, per;
    int rule, unit_qk;
    float unit_eps, q_scale;
};
// floats of scratch that a head needs of a token
static int scratch_floats(int rule, int key_dim, int value_dim) { return SC_LEN + (rule == 1 ? key_dim + value_dim : 0) + 4; }

__device__ __forceinline__ f32x4 mul4(const f32x4& a, float s) { return a * s; }
// Sums of products over 16 columns of the inner dimension at a time, each element of the chunks into sums of its own:
// chains of a quarter of the length, which round half as much (outputs of the delta rule 2.7e-7 from 64 bits
// with one chain, 1.7e-7 with four, as the walk's are) and follow each other without waiting.
struct Sums {
    f32x4 part[4];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int e = 0; e < 4; ++e) part[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __device__ __forceinline__ void add(const f32x4& a, const f32x4& b) {
#pragma unroll
        for (int e = 0; e < 4; ++e) Operand<float>::multiply(a, b, part[e], e);
    }
    // A block on the diagonal of a lower triangle, whose zeros above it meet tokens that come later: a number of theirs that is
    // not finite must not reach the rows before.  (Where there is one, the block's finite part goes through the MFMAs, and
    // the rest to the rows from its token on.)
    __device__ __forceinline__ void add_lower(const f32x4& a, const f32x4& b) {
        bool fine = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) fine = fine && __builtin_isfinite(b[e]);
        if (__all(fine)) {
            add(a, b);
            return;
        }
        f32x4 finite;
#pragma unroll
        for (int e = 0; e < 4; ++e) finite[e] = __builtin_isfinite(b[e]) ? b[e] : 0.f;
        add(a, finite);
        const int lane = threadIdx.x % 64, col = lane % 16, q = lane / 16;
        for (int jq = 0; jq < 4; ++jq)
#pragma unroll
            for (int je = 0; je < 4; ++je) {                // token 4 jq + je of the block
                const float x = __shfl(b[je], 16 * jq + col, WAVE);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float factor = __shfl(a[je], 16 * jq + 4 * q + e, WAVE);
                    if (!__builtin_isfinite(x) && 4 * q + e >= 4 * jq + je) part[0][e] += factor * x;
                }
            }
    }
    __device__ __forceinline__ f32x4 total() const { return (part[0] + part[1]) + (part[2] + part[3]); }
};

// ---- prepare ---------------------------------------------------------------------------------------------
template <int KC, int RULE>
__global__ __launch_bounds__(256) void state_chunk_prepare_kernel(StateChunks a) {
    constexpr int KD = 16 * KC, KLD = KD + 4;
    extern __shared__ __attribute__((aligned(16))) float sc_lds[];
    float* Ks = sc_lds;                      // [64][KLD]
    float* T = Ks + SC_LEN * KLD;            // [64][SC_LD]: D, then T
    float* X = T + SC_LEN * SC_LD;           // [64][SC_LD] (delta rule)
    __shared__ float as[SC_LEN], ws[SC_LEN], ps[SC_LEN], wp[SC_LEN];
    const int head = blockIdx.x % a.heads, chunk = blockIdx.x / a.heads % a.chunks_per_seq, seq = blockIdx.x / a.heads / a.chunks_per_seq;
    const int row0 = a.cu_seqlens[seq] + chunk * SC_LEN, n = min(SC_LEN, a.cu_seqlens[seq + 1] - row0);
    if (n <= 0) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64, r16 = lane % 16, q = lane / 16;
    const int kh = head / (a.heads / a.key_heads);
    const float* qp = a.qkv + (size_t)row0 * a.qkv_stride + a.q_off + (size_t)kh * KD;
    const float* kp = a.qkv + (size_t)row0 * a.qkv_stride + a.k_off + (size_t)kh * KD;
    for (int idx = tid; idx < SC_LEN * KD / 4; idx += 256) {          // (rows past the last repeat it)
        const int t = idx / (KD / 4), c = idx % (KD / 4) * 4;
        *(f32x4*)(Ks + t * KLD + c) = *(const f32x4*)(kp + (size_t)min(t, n - 1) * a.qkv_stride + c);
    }
    if (tid < SC_LEN) {
        const float* row = a.aw + (size_t)(row0 + min(tid, n - 1)) * 2 * a.heads + head;
        as[tid] = tid < n ? row[0] : 1.f;
        ws[tid] = tid < n ? row[a.heads] : 0.f;
    }
    __syncthreads();
    {
        // D_ij, a running product from j = i down (in 64 bits, so that each is rounded once); four threads share a row
        const int i = tid % SC_LEN, low = tid / SC_LEN * 16;
        if (low <= i) {
            double prod = 1.0;
            int j = i;
            for (; j > low + 15; --j) prod *= as[j];
            for (; j >= low; --j) {
                T[i * SC_LD + j] = (float)prod;
                prod *= as[j];
            }
            if (low == 0) ps[i] = (float)prod, wp[i] = (float)(-ws[i] * prod);
        }
    }
    // q_i . k_j (and k_i . k_j) of the ten pairs of blocks I >= J, three at most a wave
    f32x4 qk[3], kk[3];
    int bi[3], bj[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int idx = wave + 4 * u;
        Sums qs, ks;
        qs.clear(), ks.clear();
        qk[u] = kk[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        bi[u] = -1, bj[u] = 0;
        if (idx >= 10) continue;
        int I = 0;
        while ((I + 1) * (I + 2) / 2 <= idx) ++I;
        bi[u] = I, bj[u] = idx - I * (I + 1) / 2;
        const float* qrow = qp + (size_t)min(16 * I + r16, n - 1) * a.qkv_stride + 4 * q;
        const float* ki = Ks + (16 * I + r16) * KLD + 4 * q;
        const float* kj = Ks + (16 * bj[u] + r16) * KLD + 4 * q;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const f32x4 k = *(const f32x4*)(kj + 16 * c);
            qs.add(*(const f32x4*)(qrow + 16 * c), k);
            if (RULE == 1) ks.add(*(const f32x4*)(ki + 16 * c), k);
        }
        qk[u] = qs.total(), kk[u] = ks.total();
    }
    __syncthreads();
    float* scratch = a.scratch + (size_t)row0 * a.heads * a.per + (size_t)head * a.per;
    const size_t srow = (size_t)a.heads * a.per;
    if (tid < n) {
        scratch[tid * srow + a.per - 4] = ps[tid];
        scratch[tid * srow + a.per - 3] = T[(n - 1) * SC_LD + tid];
        scratch[tid * srow + a.per - 2] = ws[tid];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        if (bi[u] < 0) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * bi[u] + 4 * q + e, j = 16 * bj[u] + r16;
            const float d = j <= i ? T[i * SC_LD + j] : 0.f;
            if (i < n) scratch[i * srow + j] = j <= i ? d * qk[u][e] : 0.f;
            if (RULE == 1) T[i * SC_LD + j] = j < i ? ws[i] * d * kk[u][e] : 0.f;
        }
    }
    if (RULE == 0) return;
    __syncthreads();
    if (lane < 16) {
        // a block on the diagonal, a lane a column of its inverse
        float x[16];
        const float* t = T + 16 * wave * SC_LD + 16 * wave;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float s = i == lane ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < i; ++j) s -= t[i * SC_LD + j] * x[j];
            x[i] = s;
            X[(16 * wave + i) * SC_LD + 16 * wave + lane] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int d = 1; d < 4; ++d) {
        const int J = wave, I = J + d;
        if (I < 4) {
            Sums ys, xs;
            ys.clear(), xs.clear();
            for (int k = J; k < I; ++k) {
                f32x4 b;
#pragma unroll
                for (int e = 0; e < 4; ++e) b[e] = X[(16 * k + 4 * q + e) * SC_LD + 16 * J + r16];
                ys.add(*(const f32x4*)(T + (16 * I + r16) * SC_LD + 16 * k + 4 * q), b);
            }
            xs.add_lower(*(const f32x4*)(X + (16 * I + r16) * SC_LD + 16 * I + 4 * q), ys.total());   // (rows 4q + e of the one are the operand's)
            const f32x4 x = xs.total();
#pragma unroll
            for (int e = 0; e < 4; ++e) X[(16 * I + 4 * q + e) * SC_LD + 16 * J + r16] = -x[e];
        }
        __syncthreads();
    }
    // -X diag(w p) K, then X diag(w) V, a column tile at a time; row tile I takes blocks J <= I
    const float* vp = a.qkv + (size_t)row0 * a.qkv_stride + a.v_off + (size_t)head * a.value_dim;
    for (int tile = wave; tile < KC + a.value_dim / 16; tile += 4) {
        const bool keys = tile < KC;
        const int c = 16 * (keys ? tile : tile - KC) + r16;
        f32x4 b[4], o[4];
#pragma unroll
        for (int J = 0; J < 4; ++J)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * J + 4 * q + e;
                b[J][e] = keys ? Ks[t * KLD + c] * wp[t] : vp[(size_t)min(t, n - 1) * a.qkv_stride + c] * ws[t];
            }
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            Sums t;
            t.clear();
#pragma unroll
            for (int J = 0; J < I; ++J) t.add(*(const f32x4*)(X + (16 * I + r16) * SC_LD + 16 * J + 4 * q), b[J]);
            t.add_lower(*(const f32x4*)(X + (16 * I + r16) * SC_LD + 16 * I + 4 * q), b[I]);
            o[I] = t.total();
        }
        float* to = scratch + SC_LEN + (keys ? 0 : KD) + c;
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 16 * I + 4 * q + e;
                if (i < n) to[i * srow] = o[I][e];
            }
    }
}

// ---- walk ------------------------------------------------------------------------------------------------
template <int KC, int VT, int RULE>
__global__ __launch_bounds__(256) void state_chunk_walk_kernel(StateChunks a) {
    constexpr int KD = 16 * KC, KLD = KD + 4, VB = 16 * VT, KT = KC / 4;
    __shared__ __attribute__((aligned(16))) float St[VB * KLD];       // the state's columns
    __shared__ __attribute__((aligned(16))) float Ut[VB * SC_LD];     // u, and u times the decays behind it
    __shared__ __attribute__((aligned(16))) float Dt[VB * SC_LD];
    const int n_cb = a.value_dim / VB;
    const int cb = blockIdx.x % n_cb, head = blockIdx.x / n_cb % a.heads, seq = blockIdx.x / n_cb / a.heads;
    const int first_row = a.cu_seqlens[seq], end_row = a.cu_seqlens[seq + 1], vd = a.value_dim;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64, r16 = lane % 16, q = lane / 16;
    if (end_row <= first_row) return;
    const int kh = head / (a.heads / a.key_heads);
    float* st = a.state + (size_t)a.seq_slot[seq] * a.slot_floats + (size_t)head * KD * vd + cb * VB;
    for (int idx = tid; idx < KD * VB; idx += 256) St[idx % VB * KLD + idx / VB] = st[(size_t)(idx / VB) * vd + idx % VB];
    const size_t srow = (size_t)a.heads * a.per;
    const float skip = a.skip ? a.skip[head] : 0.f;
    __syncthreads();
    struct Operands {
        f32x4 qf[KC], wf[RULE == 1 ? KC : 1], af[4], kf[KT][4];       // kf: K^T, rows of the keys' entries with tokens along
        float p, pc, dc[4], u0[VT][4], vv[VT][4];                     // dc, u0, vv: of tokens 16 wave + 4 q + e
    };
    auto load = [&](int row0, Operands& x) {
        const int n = min(SC_LEN, end_row - row0);
        const int t_row = min(16 * wave + r16, n - 1);                // this lane's token as a row of the first operand
        const float* scratch = a.scratch + (size_t)row0 * srow + (size_t)head * a.per;
        const float* mine = scratch + t_row * srow;
        const float* qkv = a.qkv + (size_t)row0 * a.qkv_stride;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            x.qf[c] = *(const f32x4*)(qkv + (size_t)t_row * a.qkv_stride + a.q_off + (size_t)kh * KD + 16 * c + 4 * q);
            if (RULE == 1) x.wf[RULE == 1 ? c : 0] = *(const f32x4*)(mine + SC_LEN + 16 * c + 4 * q);
        }
        x.p = mine[a.per - 4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = min(16 * wave + 4 * q + e, n - 1);
            x.dc[e] = scratch[t * srow + a.per - 3];
            const float w = RULE == 0 ? scratch[t * srow + a.per - 2] : 0.f;
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const int col = cb * VB + 16 * v + r16;
                x.vv[v][e] = RULE == 0 || a.skip ? qkv[(size_t)t * a.qkv_stride + a.v_off + (size_t)head * vd + col] : 0.f;
                x.u0[v][e] = RULE == 0 ? w : scratch[t * srow + SC_LEN + KD + col];
            }
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) x.af[g] = g <= wave ? *(const f32x4*)(mine + 16 * g + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < KT; ++m)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    x.kf[m][g][e] = qkv[(size_t)min(16 * g + 4 * q + e, n - 1) * a.qkv_stride + a.k_off + (size_t)kh * KD + 16 * (wave + 4 * m) + r16];
        x.pc = scratch[(n - 1) * srow + a.per - 4];
    };
    for (int row0 = first_row; row0 < end_row; row0 += SC_LEN) {
        const int n = min(SC_LEN, end_row - row0);
        Operands x;
        load(row0, x);
        Sums us[VT], os[VT];
        f32x4 u[VT];
#pragma unroll
        for (int v = 0; v < VT; ++v) us[v].clear(), os[v].clear();
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const f32x4 qs = mul4(x.qf[c], x.p);
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const f32x4 s = *(const f32x4*)(St + (16 * v + r16) * KLD + 16 * c + 4 * q);
                if (RULE == 1) us[v].add(x.wf[RULE == 1 ? c : 0], s);
                os[v].add(qs, s);
            }
        }
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            f32x4 d;
            const f32x4 more = RULE == 1 ? us[v].total() : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                u[v][e] = RULE == 1 ? x.u0[v][e] + more[e] : x.u0[v][e] * x.vv[v][e];
                if (16 * wave + 4 * q + e >= n) u[v][e] = 0.f;
                d[e] = u[v][e] * x.dc[e];
            }
            *(f32x4*)(Ut + (16 * v + r16) * SC_LD + 16 * wave + 4 * q) = u[v];
            *(f32x4*)(Dt + (16 * v + r16) * SC_LD + 16 * wave + 4 * q) = d;
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < VT; ++v) {
#pragma unroll
            for (int g = 0; g < 4; ++g)
                if (g < wave) os[v].add(x.af[g], *(const f32x4*)(Ut + (16 * v + r16) * SC_LD + 16 * g + 4 * q));
                else if (g == wave) os[v].add_lower(x.af[g], *(const f32x4*)(Ut + (16 * v + r16) * SC_LD + 16 * g + 4 * q));
            // (St has been read by every wave; a wave reads and writes its own rows of it here)
#pragma unroll
            for (int m = 0; m < KT; ++m) {
                float* to = St + (16 * v + r16) * KLD + 16 * (wave + 4 * m) + 4 * q;
                Sums s;
                s.clear();
#pragma unroll
                for (int g = 0; g < 4; ++g) s.add(x.kf[m][g], *(const f32x4*)(Dt + (16 * v + r16) * SC_LD + 16 * g + 4 * q));
                *(f32x4*)to = mul4(*(const f32x4*)to, x.pc) + s.total();
            }
            const f32x4 o = os[v].total();
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * wave + 4 * q + e;
                if (t < n) a.out[(size_t)(row0 + t) * a.heads * vd + (size_t)head * vd + cb * VB + 16 * v + r16] = o[e] + skip * x.vv[v][e];
            }
        }
        __syncthreads();
    }
    for (int idx = tid; idx < KD * VB; idx += 256) st[(size_t)(idx / VB) * vd + idx % VB] = St[idx % VB * KLD + idx / VB];
}

// ---- a decode step ----------------------------------------------------------------------------------------
// One workgroup per (sequence, head, 32 value columns): a thread has four columns of KPT rows of the state, all
// on their way at once; what it adds up over the rows (the state along k and along q, and q . k and the
// two squares that make them unit vectors) meets once, and the state is written back.
template <int KPT>
__global__ __launch_bounds__(256) void state_step_kernel(StateChunks a) {
    constexpr int KD = 32 * KPT;
    __shared__ float meet[4][8][12];
    const int n_cb = a.value_dim / 32;
    const int cb = blockIdx.x % n_cb, head = blockIdx.x / n_cb % a.heads, seq = blockIdx.x / n_cb / a.heads;
    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, c4 = tid % 8, rg = tid / 8;
    const int kh = head / (a.heads / a.key_heads), col = cb * 32 + 4 * c4;
    float* st = a.state + (size_t)a.seq_slot[seq] * a.slot_floats + (size_t)head * KD * a.value_dim + col;
    f32x4 S[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) S[i] = *(const f32x4*)(st + (size_t)(rg + 32 * i) * a.value_dim);
    const float* row = a.qkv + (size_t)seq * a.qkv_stride;
    float qv[KPT], kv[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        qv[i] = row[a.q_off + kh * KD + rg + 32 * i];
        kv[i] = row[a.k_off + kh * KD + rg + 32 * i];
    }
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = row[a.v_off + (size_t)head * a.value_dim + col + j];
    const float bias = a.dt_bias ? a.dt_bias[head] : 0.f, ra = a.in[(size_t)seq * a.in_stride + a.a_off + head],
                rw = a.in[(size_t)seq * a.in_stride + a.w_off + head];
    const float decay = expf(-expf(a.A_log[head]) * softplus_f(ra + bias)), w = a.rule == 0 ? softplus_f(rw + bias) : sigmoid_f(rw);
    // sums over the rows: S^T k [4], S^T q [4], q . k, q . q, k . k
    float sum[11];
#pragma unroll
    for (int j = 0; j < 11; ++j) sum[j] = 0.f;
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            sum[j] += S[i][j] * kv[i];
            sum[4 + j] += S[i][j] * qv[i];
        }
        sum[8] += qv[i] * kv[i];
        sum[9] += qv[i] * qv[i];
        sum[10] += kv[i] * kv[i];
    }
#pragma unroll
    for (int j = 0; j < 11; ++j) {
#pragma unroll
        for (int off = 8; off < 64; off <<= 1) sum[j] += __shfl_xor(sum[j], off, WAVE);
        if (lane < 8) meet[wave][c4][j] = sum[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 11; ++j) sum[j] = meet[0][c4][j] + meet[1][c4][j] + meet[2][c4][j] + meet[3][c4][j];
    const float sq = a.q_scale * (a.unit_qk ? 1.f / sqrtf(sum[9] + a.unit_eps) : 1.f), sk = a.unit_qk ? 1.f / sqrtf(sum[10] + a.unit_eps) : 1.f;
    const float along = sq * sk * sum[8], skip = a.skip ? a.skip[head] : 0.f;
    f32x4 u;
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        u[j] = a.rule == 1 ? w * (v[j] - decay * sk * sum[j]) : w * v[j];
        o[j] = decay * sq * sum[4 + j] + along * u[j] + skip * v[j];
        u[j] *= sk;
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) S[i][j] = decay * S[i][j] + kv[i] * u[j];
        *(f32x4*)(st + (size_t)(rg + 32 * i) * a.value_dim) = S[i];
    }
    if (rg == 0) *(f32x4*)(a.out + (size_t)seq * a.heads * a.value_dim + (size_t)head * a.value_dim + col) = f32x4{o[0], o[1], o[2], o[3]};
}

// ---- host ---------------------------------------------------------------------------------------------------
static StateChunks describe(const picolm_state_scan_args* a, const picolm_step_view* v) {
    StateChunks s = {};
    s.in = (const float*)v->in;
    s.qkv = (const float*)v->extra[0];
    s.aw = (const float*)v->extra[1];
    s.scratch = (float*)v->extra[2];
    s.out = (float*)v->out;
    s.state = (float*)v->state + a->state_off;
    s.skip = a->skip;
    s.A_log = a->A_log;
    s.dt_bias = a->dt_bias;
    s.cu_seqlens = v->cu_seqlens;
    s.seq_slot = v->seq_slot;
    s.slot_floats = v->state_bytes_per_slot / 4;
    s.in_stride = a->in_stride, s.a_off = a->a_off, s.w_off = a->w_off;
    s.qkv_stride = a->qkv_stride, s.q_off = a->q_off, s.k_off = a->k_off, s.v_off = a->v_off;
    s.heads = a->n_heads, s.key_heads = a->n_key_heads, s.value_dim = a->value_dim;
    s.per = scratch_floats(a->rule, a->key_dim, a->value_dim);
    s.rule = a->rule, s.unit_qk = a->unit_qk, s.unit_eps = a->unit_eps;
    s.q_scale = a->q_scale != 0.f ? a->q_scale : 1.f;
    return s;
}

bool picolm_state_step_takes_(const picolm_state_scan_args* a, const picolm_step_view* v) {
    return v->is_decode && (a->key_dim == 64 || a->key_dim == 128) && a->value_dim % 32 == 0 && a->state_off % 4 == 0 &&
           v->state_bytes_per_slot % 16 == 0 && (((uintptr_t)v->state | (uintptr_t)v->out) & 15) == 0 &&
           (int64_t)v->n_seq * a->n_heads * (a->value_dim / 32) < (1ll << 31);
}
int picolm_state_step_(const picolm_state_scan_args* a, const picolm_step_view* v) {
    const StateChunks s = describe(a, v);
    const unsigned grid = (unsigned)(v->n_seq * a->n_heads * (a->value_dim / 32));
    if (a->key_dim == 64) state_step_kernel<2><<<grid, 256, 0, v->stream>>>(s);
    else state_step_kernel<4><<<grid, 256, 0, v->stream>>>(s);
    PICOLM_LAUNCH_CHECK("state_scan (step)");
    return 0;
}

bool picolm_state_chunks_takes_(const picolm_state_scan_args* a, const picolm_step_view* v, int most_new) {
    return (a->key_dim == 64 || a->key_dim == 128) && a->value_dim % 16 == 0 && a->qkv_stride % 4 == 0 && a->q_off % 4 == 0 && a->k_off % 4 == 0 &&
           v->extra[2] && v->extra_row_bytes[2] >= (int64_t)a->n_heads * scratch_floats(a->rule, a->key_dim, a->value_dim) * 4 &&
           (((uintptr_t)v->extra[0] | (uintptr_t)v->extra[2]) & 15) == 0 &&
           (int64_t)v->n_seq * ceil_div(most_new, SC_LEN) * a->n_heads < (1ll << 31) &&
           (int64_t)v->n_seq * a->n_heads * (a->value_dim / 16) < (1ll << 31);
}
template <int KC, int RULE>
static int launch_chunks(const StateChunks& s, int n_seq, hipStream_t stream) {
    const size_t lds = sizeof(float) * ((size_t)SC_LEN * (16 * KC + 4) + (RULE == 1 ? 2 : 1) * SC_LEN * SC_LD);
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void*)state_chunk_prepare_kernel<KC, RULE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        PICOLM_REQUIRE(e == hipSuccess, "state_scan: cannot raise the LDS limit to %zu: %s", lds, hipGetErrorString(e));
        raised = true;
    }
    state_chunk_prepare_kernel<KC, RULE><<<(unsigned)(n_seq * s.chunks_per_seq * s.heads), 256, lds, stream>>>(s);
    PICOLM_LAUNCH_CHECK("state_scan (chunks)");
    // 32 columns a workgroup where that gives every CU one
    const bool wide = s.value_dim % 32 == 0 && (int64_t)n_seq * s.heads * (s.value_dim / 32) >= n_compute_units();
    const unsigned grid = (unsigned)(n_seq * s.heads * (s.value_dim / (wide ? 32 : 16)));
    if (wide) state_chunk_walk_kernel<KC, 2, RULE><<<grid, 256, 0, stream>>>(s);
    else state_chunk_walk_kernel<KC, 1, RULE><<<grid, 256, 0, stream>>>(s);
    PICOLM_LAUNCH_CHECK("state_scan (walk)");
    return 0;
}
// (the decays and strengths, and the unit vectors, are there: state_scan's own preparation)
int picolm_state_chunks_(const picolm_state_scan_args* a, const picolm_step_view* v, int most_new) {
    StateChunks s = describe(a, v);
    s.chunks_per_seq = ceil_div(most_new, SC_LEN);
    if (a->key_dim == 64) return a->rule == 1 ? launch_chunks<4, 1>(s, v->n_seq, v->stream) : launch_chunks<4, 0>(s, v->n_seq, v->stream);
    return a->rule == 1 ? launch_chunks<8, 1>(s, v->n_seq, v->stream) : launch_chunks<8, 0>(s, v->n_seq, v->stream);
}
