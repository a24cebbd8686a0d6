// A routed feed-forward (mixers.h): every row picks a few experts by its router logits and only
// their weights are read.  Logits, picks, weights and sums are float.
//
// 32-bit weights, and widths that are no multiples of 8: the picked experts' hidden units (a workgroup
// per (row, pick, 16 hidden units)); the down products with the weighted sum over a row's picks (a
// workgroup per (row, 16 outputs)), so that a row's result is added up in one place and in a fixed
// order.  A wave takes one weight row at a time, 16 bytes a lane, against the row's input in LDS.
//
// A decode batch in bfloat16 (up to 63 rows): the picked experts' weights are read once for all of their rows,
// and a last kernel adds a row's picks up; the same sums in the same order (expert_chains_kernel).
// Some more rows of many experts: the like with sums in the order of the bfloat16 MFMAs (expert_stream_kernel).
//
// A prompt (64 rows and more of fewer experts, bfloat16) goes through tiles on the matrix cores: the (row, pick) pairs
// are sorted by expert in one workgroup, a workgroup takes 128 pairs of one expert by 64 or 128 hidden units
// (up to 256 outputs) through LDS with v_mfma_f32_32x32x16_bf16; the hidden units are rounded to bfloat16
// once, as every product's input is; a last kernel adds a row's picks up in their order.  Which
// pairs share a tile changes no pair's result.
#include "mixers.h"

#include "api.h"
#include "common.h"
#include "gemm_direct.h"

#define VIEW_REQUIRE(who, v)                                                                                      \
    PICOLM_REQUIRE((v) && (v)->struct_bytes == (int32_t)sizeof(picolm_step_view), "%s: the step view is of another version", who)

static inline int elem_bytes(int dt) { return dt == PICOLM_F32 ? 4 : 2; }

// ---- the pick --------------------------------------------------------------------------------------
// a thread a row; the picks come out in the order (logit falling, index rising)
__global__ void route_top_kernel(const float* __restrict__ logits, int in_stride, const float* __restrict__ bias, int32_t* __restrict__ out, int E,
                                 int top, int n_rows, int scoring, float scale) {
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= n_rows) return;
    const float* z = logits + (size_t)row * in_stride;
    int32_t* ids = out + (size_t)row * 2 * top;
    float* w = (float*)(ids + top);
    if (scoring == 2) {
        // s = sigmoid of every output; the picks are the largest s + bias, their weights the picked s themselves
        float last_c = INFINITY;
        int last_e = -1;
        for (int k = 0; k < top; ++k) {
            float best = -INFINITY, best_s = 0.f;
            int be = -1;
            for (int e = 0; e < E; ++e) {
                const float se = 1.f / (1.f + expf(-z[e])), ce = se + (bias ? bias[e] : 0.f);
                const bool after_last = ce < last_c || (ce == last_c && e > last_e);
                if (after_last && (be < 0 || ce > best)) best = ce, be = e, best_s = se;
            }
            if (be < 0) be = k % E, best = -INFINITY, best_s = 0.f;     // (only logits that are no numbers lead here)
            ids[k] = be;
            w[k] = best_s * scale;
            last_c = best, last_e = be;
        }
        return;
    }
    if (scoring == 1 || scoring == 3) {
        // s = softmax over every output; the picks are the largest s + bias, their weights the picked s over their sum or (3) as they are
        float zmax = -INFINITY, den = 0.f;
        for (int e = 0; e < E; ++e) zmax = fmaxf(zmax, z[e]);
        for (int e = 0; e < E; ++e) den += expf(z[e] - zmax);
        float last_c = INFINITY, sum = 0.f;
        int last_e = -1;
        for (int k = 0; k < top; ++k) {
            float best = -INFINITY, best_s = 0.f;
            int be = -1;
            for (int e = 0; e < E; ++e) {
                const float se = expf(z[e] - zmax) / den, ce = se + (bias ? bias[e] : 0.f);
                const bool after_last = ce < last_c || (ce == last_c && e > last_e);
                if (after_last && (be < 0 || ce > best)) best = ce, be = e, best_s = se;
            }
            if (be < 0) be = k % E, best = -INFINITY, best_s = 0.f;     // (only logits that are no numbers lead here)
            ids[k] = be;
            w[k] = best_s;
            sum += best_s;
            last_c = best, last_e = be;
        }
        for (int k = 0; k < top; ++k) w[k] = (scoring == 1 ? w[k] / (sum + 1e-20f) : w[k]) * scale;
        return;
    }
    float last_z = INFINITY, first_z = 0.f, sum = 0.f;
    int last_e = -1;
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY;
        int be = -1;
        for (int e = 0; e < E; ++e) {
            const float ze = z[e] + (bias ? bias[e] : 0.f);
            const bool after_last = ze < last_z || (ze == last_z && e > last_e);
            if (after_last && (be < 0 || ze > best)) best = ze, be = e;
        }
        if (be < 0) be = k % E, best = -INFINITY;     // (only logits that are no numbers lead here)
        if (k == 0) first_z = best;
        const float p = expf(best - first_z);
        ids[k] = be;
        w[k] = p;
        sum += p;
        last_z = best, last_e = be;
    }
    for (int k = 0; k < top; ++k) w[k] /= sum;
}

// The same with a wave a row and a lane an output, for up to 64 outputs: a thread that walks over its
// row's outputs for every pick waits for each of them (16 rows of eight outputs, two picks: 6.8 us against 3.4).
// Sums run over the outputs in the same order, by lane broadcasts, so that the results are the same.
__global__ __launch_bounds__(256) void route_top_wave_kernel(const float* __restrict__ logits, int in_stride, const float* __restrict__ bias,
                                                             int32_t* __restrict__ out, int E, int top, int n_rows, int scoring, float scale) {
    const int row = blockIdx.x * 4 + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (row >= n_rows) return;
    const bool mine = lane < E;
    const float z = mine ? logits[(size_t)row * in_stride + lane] : 0.f, add = mine && bias ? bias[lane] : 0.f;
    auto from_lane = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
    float s = z;                    // what a pick's weight comes from; what is compared is s + bias
    if (scoring == 2) s = 1.f / (1.f + expf(-z));
    if (scoring == 1 || scoring == 3) {
        const float zmax = wave_max(mine ? z : -INFINITY), x = expf(z - zmax);
        float den = 0.f;
        for (int e = 0; e < E; ++e) den += from_lane(x, e);
        s = x / den;
    }
    const float c = s + add;
    float last_c = INFINITY, first_c = 0.f, sum = 0.f, my_w = 0.f;
    int last_e = -1, my_id = 0;
    for (int k = 0; k < top; ++k) {
        const bool open = mine && (c < last_c || (c == last_c && lane > last_e));
        float best = wave_max(open ? c : -INFINITY);
        const unsigned long long at = __ballot(open && c == best);
        int be = __ffsll((long long)at) - 1;
        float w = be < 0 ? 0.f : from_lane(s, be);
        if (be < 0) be = k % E, best = -INFINITY;       // (only logits that are no numbers lead here)
        if (scoring == 0) {
            if (k == 0) first_c = best;
            w = expf(best - first_c);
        }
        sum += w;
        if (lane == k) my_id = be, my_w = w;
        last_c = best, last_e = be;
    }
    if (lane >= top) return;
    int32_t* ids = out + (size_t)row * 2 * top;
    ids[lane] = my_id;
    ((float*)(ids + top))[lane] = scoring == 0 ? my_w / sum : scoring == 1 ? my_w / (sum + 1e-20f) * scale : my_w * scale;
}

extern "C" int picolm_call_route_top(void* user, const picolm_step_view* v) {
    const picolm_route_top_args* a = (const picolm_route_top_args*)user;
    VIEW_REQUIRE("route_top", v);
    PICOLM_REQUIRE(a && v->in && v->out && a->experts > 0 && a->top > 0 && a->top <= a->experts, "route_top: %d picks among %d experts",
                   a ? a->top : 0, a ? a->experts : 0);
    const int in_stride = a->in_stride ? a->in_stride : a->experts;
    PICOLM_REQUIRE(in_stride >= a->experts && v->in_row_bytes >= (int64_t)in_stride * 4 && v->out_row_bytes >= 2 * a->top * 4, "route_top: rows too short");
    PICOLM_REQUIRE(a->scoring >= 0 && a->scoring <= 3, "route_top: scoring %d is not known", a->scoring);
    if (v->rows <= 0) return 0;
    if (a->experts <= WAVE)
        route_top_wave_kernel<<<ceil_div(v->rows, 4), 256, 0, v->stream>>>((const float*)v->in, in_stride, a->bias, (int32_t*)v->out, a->experts,
                                                                          a->top, v->rows, a->scoring, a->scale);
    else
        route_top_kernel<<<ceil_div(v->rows, 64), 64, 0, v->stream>>>((const float*)v->in, in_stride, a->bias, (int32_t*)v->out, a->experts, a->top,
                                                                 v->rows, a->scoring, a->scale);
    PICOLM_LAUNCH_CHECK("route_top");
    return 0;
}

// ---- the picked experts ------------------------------------------------------------------------------
// a lane's share of the dot product of a weight row with floats in LDS
template <typename TW> __device__ __forceinline__ float lane_dot(const TW* __restrict__ w, const float* __restrict__ h, int K, int lane);
template <> __device__ __forceinline__ float lane_dot<bf16_t>(const bf16_t* __restrict__ w, const float* __restrict__ h, int K, int lane) {
    float acc = 0.f;
    if (K % 8 == 0) {
        for (int i = lane * 8; i < K; i += WAVE * 8) {
            const uint4 p = *(const uint4*)(w + i);
            const uint32_t u[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc += __uint_as_float(u[j] << 16) * h[i + 2 * j];
                acc += __uint_as_float(u[j] & 0xffff0000u) * h[i + 2 * j + 1];
            }
        }
    } else {
        for (int i = lane; i < K; i += WAVE) acc += bf16_bits_to_f32(w[i]) * h[i];
    }
    return acc;
}
template <> __device__ __forceinline__ float lane_dot<float>(const float* __restrict__ w, const float* __restrict__ h, int K, int lane) {
    float acc = 0.f;
    if (K % 4 == 0) {
        for (int i = lane * 4; i < K; i += WAVE * 4) {
            const float4 p = *(const float4*)(w + i);
            acc += p.x * h[i] + p.y * h[i + 1] + p.z * h[i + 2] + p.w * h[i + 3];
        }
    } else {
        for (int i = lane; i < K; i += WAVE) acc += w[i] * h[i];
    }
    return acc;
}

#define MOE_UNITS 16     // hidden units, or outputs, a workgroup of four waves takes

// what an expert's hidden unit is, from its two products g and u (mixers.h: picolm_routed_experts_args.act)
struct ExpertAct {
    int kind;
    float limit, alpha;
    int weight_on_input;
};
__device__ __forceinline__ float expert_act(const ExpertAct& x, float g, float u) {
    if (x.kind == 1) {
        g = fminf(g, x.limit);
        u = fminf(fmaxf(u, -x.limit), x.limit);
        return g / (1.f + expf(-x.alpha * g)) * (u + 1.f);
    }
    return g / (1.f + expf(-g)) * u;
}

// act[row][pick][f] = silu(W_gate[e][f] . h) * (W_up[e][f] . h); a wave has its four units' eight rows on their way at once
template <typename TW, typename TH>
__global__ __launch_bounds__(256) void expert_hidden_kernel(const TH* __restrict__ h, const int32_t* __restrict__ picks, float* __restrict__ act,
                                                            const TW* __restrict__ gate, const TW* __restrict__ up, int E, int top, int D, int F,
                                                            ExpertAct xa) {
    extern __shared__ float moe_lds[];       // [D]
    const int pair = blockIdx.x, row = pair / top, k = pair % top;
    const int e = picks[(size_t)row * 2 * top + k];
    for (int c = threadIdx.x; c < D; c += blockDim.x) moe_lds[c] = to_f32<TH>(h[(size_t)row * D + c]);
    __syncthreads();
    if (e < 0 || e >= E) return;
    const float on_input = xa.weight_on_input ? ((const float*)(picks + (size_t)row * 2 * top + top))[k] : 1.f;
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int f0 = blockIdx.y * MOE_UNITS + wave * 4;
    float g[4], u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const size_t w_row = ((size_t)e * F + min(f0 + j, F - 1)) * D;
        g[j] = lane_dot<TW>(gate + w_row, moe_lds, D, lane);
        u[j] = lane_dot<TW>(up + w_row, moe_lds, D, lane);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float gs = wave_sum(g[j]) * on_input, us = wave_sum(u[j]) * on_input;
        if (lane == 0 && f0 + j < F) act[((size_t)row * top + k) * F + f0 + j] = expert_act(xa, gs, us);
    }
}

// out[row][d] (+)= sum_k w[row][k] (W_down[e_k][d] . act[row][k])
// a row's picks that stand for "the input itself": the sum of their weights
__device__ __forceinline__ float identity_weight(const int32_t* ids, const float* w, int top, int E, int identity) {
    float total = 0.f;
    for (int k = 0; k < top; ++k)
        if (ids[k] >= E && ids[k] < E + identity) total += w[k];
    return total;
}

template <typename TW, typename TH>
__global__ __launch_bounds__(256) void expert_down_kernel(const float* __restrict__ act, const int32_t* __restrict__ picks, float* __restrict__ out,
                                                          const TW* __restrict__ down, int E, int top, int D, int F, int adds,
                                                          const TH* __restrict__ h, int identity, int plain_sum) {
    extern __shared__ float moe_lds[];       // [top][F]
    const int row = blockIdx.x;
    for (int c = threadIdx.x; c < top * F; c += blockDim.x) moe_lds[c] = act[(size_t)row * top * F + c];
    __syncthreads();
    const int32_t* ids = picks + (size_t)row * 2 * top;
    const float* w = (const float*)(ids + top);
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int d0 = blockIdx.y * MOE_UNITS + wave * 4;
    float total[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < top; ++k) {
        const int e = ids[k];
        if (e < 0 || e >= E) continue;
        float part[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) part[j] = lane_dot<TW>(down + ((size_t)e * D + min(d0 + j, D - 1)) * F, moe_lds + (size_t)k * F, F, lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) total[j] += (plain_sum ? 1.f : w[k]) * wave_sum(part[j]);
    }
    const float same = identity > 0 ? identity_weight(ids, w, top, E, identity) : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (lane == 0 && d0 + j < D) {
            const size_t at = (size_t)row * D + d0 + j;
            out[at] = (adds ? out[at] : 0.f) + total[j] + (same != 0.f ? same * to_f32<TH>(h[at]) : 0.f);
        }
}

// ---- the same for many rows, on the matrix cores ------------------------------------------------------
#define GM_ROWS 128      // pairs of a tile
#define GM_MAX_EXPERTS 4096

// plan: [0 .. E] where each expert's pairs start in the sorted list, then the sorted pairs (pair = row * top + pick)
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int32_t* __restrict__ picks, int32_t* __restrict__ plan, int E, int top,
                                                        int n_pairs) {
    extern __shared__ int32_t plan_lds[];      // counts, then cursors [E] | starts [E + 1]
    int32_t* counts = plan_lds;
    int32_t* starts = plan_lds + E;
    for (int e = threadIdx.x; e < E; e += blockDim.x) counts[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += blockDim.x) {
        const int e = picks[(size_t)(p / top) * 2 * top + p % top];
        if (e >= 0 && e < E) atomicAdd(&counts[e], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int at = 0;
        for (int e = 0; e < E; ++e) {
            starts[e] = at;
            at += counts[e];
            counts[e] = 0;
        }
        starts[E] = at;
    }
    __syncthreads();
    for (int e = threadIdx.x; e <= E; e += blockDim.x) plan[e] = starts[e];
    for (int p = threadIdx.x; p < n_pairs; p += blockDim.x) {
        const int e = picks[(size_t)(p / top) * 2 * top + p % top];
        if (e >= 0 && e < E) plan[E + 1 + starts[e] + atomicAdd(&counts[e], 1)] = p;
    }
}

// the tile of GM_ROWS pairs that a workgroup takes: its expert, and its pairs into LDS (-1 past the expert's last)
__device__ __forceinline__ int tile_of(const int32_t* __restrict__ plan, int E, int tile, int32_t* pairs_lds) {
    int e = 0, first = 0;
    for (; e < E; ++e) {
        const int n = plan[e + 1] - plan[e], tiles = (n + GM_ROWS - 1) / GM_ROWS;
        if (tile < tiles) {
            first = plan[e] + tile * GM_ROWS;
            break;
        }
        tile -= tiles;
    }
    if (e == E) return -1;
    for (int r = threadIdx.x; r < GM_ROWS; r += blockDim.x) pairs_lds[r] = first + r < plan[e + 1] ? plan[E + 1 + first + r] : -1;
    return e;
}

// The expert's tile of GM_ROWS pairs by 64 * WN weight rows, for K in whole lines: both operands go
// from memory straight into LDS, NS stages of GD_BK columns deep, as in gemm_direct.h (whose swizzle
// and schedule this is), the pairs' rows gathered by each lane's own address.  A wave takes 64 pairs
// by 64 weight rows; with HIDDEN these are the gate and the up row of 32 hidden units, a lane's
// accumulators hold both of one unit.  Workgroups of one chiplet take the pairs' tiles of the same
// weight rows, one expert behind the other, so that weights are read from memory once.
// (Staged through registers, a step at a time and 64 units wide, waves waited for memory and for each
// other.  3,200 rows, eight experts of 2,048 x 2,048, two picked: hidden units 213 -> 157 us, 690
// TFLOP/s, outputs 154 -> 79; the whole operation at 256 rows 108 -> 87, at 2,048 229 -> 205, sixteen experts of
// 4,096 x 4,096 at 256 rows 412 -> 351, at 2,048 885 -> 643.)
//   HIDDEN: out[pair][f] = bf16(act(gate_f . a[pair / top], up_f . a[pair / top])), else out[pair][d] = w0_d . a[pair], float
#define GD_BK 64
template <bool HIDDEN, int WN, int NS>
__global__ __launch_bounds__(128 * WN) void grouped_direct_kernel(const bf16_t* __restrict__ a, const int32_t* __restrict__ plan,
                                                                  void* __restrict__ out, const bf16_t* __restrict__ w0,
                                                                  const bf16_t* __restrict__ w1, int E, int top, int K, int N,
                                                                  const int32_t* __restrict__ picks, ExpertAct xa) {
    constexpr int NW = 2 * WN, BN = 64 * WN, UNITS = HIDDEN ? BN / 2 : BN;      // waves, weight rows and outputs of a tile
    constexpr int RG = 8, W_LOADS = BN / (NW * RG), A_LOADS = GM_ROWS / (NW * RG), STAGE = (BN + GM_ROWS) * GD_BK;
    extern __shared__ __attribute__((aligned(16))) bf16_t grouped_lds[];        // [NS][BN + GM_ROWS][GD_BK]
    __shared__ int32_t pairs[GM_ROWS];
    // workgroups go to the chiplets in turn: each chiplet gets a run of tiles
    int tile, unit_block;
    {
        const int nb = gridDim.x * gridDim.y, id = blockIdx.y * gridDim.x + blockIdx.x, per = nb / 8, rem = nb % 8, xcd = id % 8;
        const int at = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + id / 8;
        tile = at % gridDim.x, unit_block = at / gridDim.x;
    }
    const int e = tile_of(plan, E, tile, pairs);
    if (e < 0) return;
    __syncthreads();
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, l32 = lane % 32, kq = lane / 32;
    const int n0 = unit_block * UNITS, wn = (wave % WN) * 64, wm = (wave / WN) * 64;
    // load j of a wave fills rows (j * NW + wave) * RG .. + RG - 1 of the weights' (then the pairs') part of a stage
    const int lrow = lane / 8, lpos = lane % 8;
    unsigned w_off[W_LOADS];
    const bf16_t *w_src[W_LOADS], *a_src[A_LOADS];
#pragma unroll
    for (int j = 0; j < W_LOADS; ++j) {
        const int first = (j * NW + wave) * RG, row = first + lrow;
        // with HIDDEN, rows 64 g .. + 31 are gate's and 64 g + 32 .. + 31 up's of the same units
        const int unit = HIDDEN ? n0 + row / 64 * 32 + row % 32 : n0 + row;
        const bf16_t* matrix = HIDDEN && (first / 32) % 2 ? w1 : w0;            // (one for a wave's eight rows)
        w_src[j] = (const bf16_t*)same_in_every_lane(matrix + ((size_t)e * N + n0) * K);
        w_off[j] = (unsigned)(((min(unit, N - 1) - n0) * K + swizzled_chunk<GD_BK>(row, lpos) * 8) * 2);
    }
#pragma unroll
    for (int j = 0; j < A_LOADS; ++j) {
        const int row = (j * NW + wave) * RG + lrow, pair = pairs[row] >= 0 ? pairs[row] : pairs[0];       // (results of a repeated pair are not stored)
        a_src[j] = a + (size_t)(HIDDEN ? pair / top : pair) * K + swizzled_chunk<GD_BK>(row, lpos) * 8;
    }
    const unsigned lds_wave = __builtin_amdgcn_readfirstlane(
        (unsigned)(size_t)(__attribute__((address_space(3))) bf16_t*)grouped_lds + wave * (RG * GD_BK * 2));
    const int n_steps = K / GD_BK;
    auto issue = [&](int stage, int step) {
        const unsigned to = lds_wave + stage * (STAGE * 2);
#pragma unroll
        for (int j = 0; j < W_LOADS; ++j)
            load_16_bytes_to_lds(w_off[j], same_in_every_lane(w_src[j] + step * GD_BK), to + j * (NW * RG * GD_BK * 2));
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) gather_16_bytes_to_lds(a_src[j] + step * GD_BK, to + (BN + j * NW * RG) * (GD_BK * 2));
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
    bf16x8 wf[2][2], af[2][2];
    auto read_frags = [&](int stage, int ks, bf16x8 (&w)[2], bf16x8 (&x)[2]) {
        const bf16_t* Ws = grouped_lds + stage * STAGE;
        const bf16_t* As = Ws + BN * GD_BK;
        const int chunk = ks * 2 + kq;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = wn + 32 * i + l32;
            w[i] = *(const bf16x8*)(Ws + row * GD_BK + swizzled_chunk<GD_BK>(row, chunk) * 8);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = wm + 32 * j + l32;
            x[j] = *(const bf16x8*)(As + row * GD_BK + swizzled_chunk<GD_BK>(row, chunk) * 8);
        }
    };
    auto multiply = [&](const bf16x8 (&w)[2], const bf16x8 (&x)[2], int i_lo, int i_hi) {
#pragma unroll
        for (int i = i_lo; i < i_hi; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[j], w[i], acc[i][j], 0, 0, 0);
    };
    // Steps past the last repeat it: every wave issues the same count of loads, and the waits count.
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) issue(s, min(s, n_steps - 1));
    wait_for_loads<(W_LOADS + A_LOADS) * (NS - 2)>();
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    issue(NS - 1, min(NS - 1, n_steps - 1));
    read_frags(0, 0, wf[0], af[0]);
    int stage = 0;
    for (int it = 0; it < n_steps; ++it) {
        const int next_stage = stage + 1 == NS ? 0 : stage + 1;
#pragma unroll
        for (int ks = 0; ks < GD_BK / 16; ++ks) {
            if (ks + 1 < GD_BK / 16) {
                read_frags(stage, ks + 1, wf[(ks + 1) & 1], af[(ks + 1) & 1]);
                multiply(wf[ks & 1], af[ks & 1], 0, 2);
                __builtin_amdgcn_sched_barrier(0);
            } else {
                multiply(wf[ks & 1], af[ks & 1], 0, 1);
                __builtin_amdgcn_sched_barrier(0);
                wait_for_loads<(W_LOADS + A_LOADS) * (NS - 2)>();       // the next stage is there
                __syncthreads();                                        // ... for every wave, and none reads this one any more
                __builtin_amdgcn_sched_barrier(0);
                issue(stage, min(it + NS, n_steps - 1));
                read_frags(next_stage, 0, wf[0], af[0]);
                multiply(wf[ks & 1], af[ks & 1], 1, 2);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        stage = next_stage;
    }
    wait_for_loads<0>();
#pragma unroll
    for (int i = 0; i < (HIDDEN ? 1 : 2); ++i) {
        const int n = n0 + (HIDDEN ? wn / 2 : wn + 32 * i) + l32;
        if (n >= N) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int pair = pairs[wm + 32 * j + 8 * (q / 4) + q % 4 + 4 * kq];
                if (pair < 0) continue;
                if constexpr (HIDDEN) {
                    const float on_input = xa.weight_on_input ? ((const float*)(picks + (size_t)(pair / top) * 2 * top + top))[pair % top] : 1.f;
                    ((bf16_t*)out)[(size_t)pair * N + n] = f32_to_bf16_bits(expert_act(xa, acc[0][j][q] * on_input, acc[1][j][q] * on_input));
                } else {
                    ((float*)out)[(size_t)pair * N + n] = acc[i][j][q];
                }
            }
    }
}

template <bool HIDDEN, int WN, int NS>
static int launch_grouped_direct(const bf16_t* a, const int32_t* plan, void* out, const bf16_t* w0, const bf16_t* w1, int E, int top, int K, int N,
                                 unsigned tiles, const int32_t* picks, const ExpertAct& xa, hipStream_t stream) {
    constexpr int UNITS = HIDDEN ? 32 * WN : 64 * WN;
    constexpr size_t lds = (size_t)NS * (64 * WN + GM_ROWS) * GD_BK * 2;
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void*)grouped_direct_kernel<HIDDEN, WN, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        PICOLM_REQUIRE(e == hipSuccess, "routed_experts: cannot raise the LDS limit to %zu: %s", lds, hipGetErrorString(e));
        raised = true;
    }
    grouped_direct_kernel<HIDDEN, WN, NS><<<dim3(tiles, ceil_div(N, UNITS)), 128 * WN, lds, stream>>>(a, plan, out, w0, w1, E, top, K, N, picks, xa);
    PICOLM_LAUNCH_CHECK("routed_experts (grouped, direct)");
    return 0;
}

// A workgroup of four waves takes GM_ROWS pairs of one expert by GM_COLS weight rows: K goes by in
// steps of GM_BK columns that all threads stage in LDS, 16 bytes a thread and load (the pairs' rows
// gathered), in rows padded by 16 bytes so that a fragment's 32 rows spread over the banks; a wave
// takes 64 pairs by 32 weight rows.
//   HIDDEN: the weight rows are GM_COLS hidden units of gate and of up, and
//           out[pair][f] = bf16(silu(gate_f . h[pair / top]) * (up_f . h[pair / top]))
//   else:   out[pair][d] = w0_d . a[pair], float
#define GM_COLS 64
#define GM_BK 64
#define GM_LD (GM_BK + 8)
template <bool HIDDEN>
__global__ __launch_bounds__(256) void grouped_tile_kernel(const bf16_t* __restrict__ a, const int32_t* __restrict__ plan, void* __restrict__ out,
                                                           const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1, int E, int top, int K,
                                                           int N, const int32_t* __restrict__ picks, ExpertAct xa) {
    constexpr int NB = HIDDEN ? 2 : 1;
    __shared__ int32_t pairs[GM_ROWS];
    __shared__ __attribute__((aligned(16))) bf16_t As[GM_ROWS * GM_LD];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[NB * GM_COLS * GM_LD];
    const int e = tile_of(plan, E, blockIdx.x, pairs);
    if (e < 0) return;
    __syncthreads();
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, l32 = lane % 32, kq = lane / 32;
    const int rh = wave / 2, uh = wave % 2, n0 = blockIdx.y * GM_COLS;
    f32x16 acc[2][NB];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
    // what this thread stages at every step: chunk `ch` of four pairs' rows and of two (or four) weight rows
    const int ch = tid % 8, r_first = tid / 8;              // rows r_first, r_first + 32, ...
    const bf16_t* a_src[GM_ROWS / 32];
#pragma unroll
    for (int c = 0; c < GM_ROWS / 32; ++c) {
        const int pair = pairs[r_first + 32 * c];
        a_src[c] = pair >= 0 ? a + (size_t)(HIDDEN ? pair / top : pair) * K + ch * 8 : nullptr;
    }
    const bf16_t* b_src[NB * GM_COLS / 32];
#pragma unroll
    for (int c = 0; c < NB * GM_COLS / 32; ++c) {
        const int r = r_first + 32 * c;                     // rows GM_COLS and up are the second matrix's
        const bf16_t* base = r < GM_COLS ? w0 : w1;
        b_src[c] = base + ((size_t)e * N + min(n0 + r % GM_COLS, N - 1)) * K + ch * 8;
    }
    for (int k0 = 0; k0 < K; k0 += GM_BK) {
        const bool inside = k0 + ch * 8 < K;                // (K is a multiple of 16, a chunk lies inside or outside)
        bf16x8 av[GM_ROWS / 32], bv[NB * GM_COLS / 32];
#pragma unroll
        for (int c = 0; c < GM_ROWS / 32; ++c) av[c] = a_src[c] && inside ? load_chunk(a_src[c] + k0) : zero_chunk();
#pragma unroll
        for (int c = 0; c < NB * GM_COLS / 32; ++c) bv[c] = inside ? load_chunk(b_src[c] + k0) : zero_chunk();
        __syncthreads();                                    // the step before has been read
#pragma unroll
        for (int c = 0; c < GM_ROWS / 32; ++c) *(bf16x8*)(As + (r_first + 32 * c) * GM_LD + ch * 8) = av[c];
#pragma unroll
        for (int c = 0; c < NB * GM_COLS / 32; ++c) *(bf16x8*)(Bs + (r_first + 32 * c) * GM_LD + ch * 8) = bv[c];
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < GM_BK / 16; ++ks) {
            const int col = ks * 16 + kq * 8;
            const bf16x8 a0 = *(const bf16x8*)(As + (rh * 64 + l32) * GM_LD + col);
            const bf16x8 a1 = *(const bf16x8*)(As + (rh * 64 + 32 + l32) * GM_LD + col);
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const bf16x8 bj = *(const bf16x8*)(Bs + (j * GM_COLS + uh * 32 + l32) * GM_LD + col);
                acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, bj, acc[0][j], 0, 0, 0);
                acc[1][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, bj, acc[1][j], 0, 0, 0);
            }
        }
    }
    const int n = n0 + uh * 32 + l32;
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int pair = pairs[rh * 64 + i * 32 + 8 * (q / 4) + q % 4 + 4 * kq];
            if (pair < 0) continue;
            if constexpr (HIDDEN) {
                const float on_input = xa.weight_on_input ? ((const float*)(picks + (size_t)(pair / top) * 2 * top + top))[pair % top] : 1.f;
                ((bf16_t*)out)[(size_t)pair * N + n] = f32_to_bf16_bits(expert_act(xa, acc[i][0][q] * on_input, acc[i][NB - 1][q] * on_input));
            } else {
                ((float*)out)[(size_t)pair * N + n] = acc[i][0][q];
            }
        }
}

// out[row] (+)= sum_k w[row][k] y[row][k], in the order of the picks; four columns a thread (D is a
// multiple of four), so that a row's picks are asked for in one trip and a step of few rows has a
// workgroup for every 1,024 columns
// (out and the inputs need not begin at 16 bytes: in a prompt's step nothing else asks for that)
#define GSUM_AT_ONCE 8
typedef __attribute__((ext_vector_type(4), aligned(4))) float floats_anywhere;
typedef __attribute__((ext_vector_type(2), aligned(2))) unsigned bf16_four_anywhere;
__global__ __launch_bounds__(256) void grouped_sum_kernel(const float* __restrict__ y, const int32_t* __restrict__ picks, float* __restrict__ out,
                                                          int E, int top, int D, int adds, const bf16_t* __restrict__ h, int identity,
                                                          int plain_sum) {
    const size_t row = blockIdx.x;
    const int d = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
    if (d >= D) return;
    const int32_t* ids = picks + row * 2 * top;
    const float* w = (const float*)(ids + top);
    floats_anywhere* o = (floats_anywhere*)(out + row * D + d);
    floats_anywhere total = {0.f, 0.f, 0.f, 0.f}, before = total, input = total;
    if (adds) before = *o;
    for (int k0 = 0; k0 < top; k0 += GSUM_AT_ONCE) {
        floats_anywhere part[GSUM_AT_ONCE];
        float wk[GSUM_AT_ONCE];
#pragma unroll
        for (int i = 0; i < GSUM_AT_ONCE; ++i) {
            const int k = min(k0 + i, top - 1), e = ids[k];
            wk[i] = k0 + i < top && e >= 0 && e < E ? (plain_sum ? 1.f : w[k]) : 0.f;
            if (k0 + i < top) part[i] = *(const floats_anywhere*)(y + (row * top + k) * D + d);       // (of a pick without an expert: not used)
        }
#pragma unroll
        for (int i = 0; i < GSUM_AT_ONCE; ++i)
            if (k0 + i < top && ids[k0 + i] >= 0 && ids[k0 + i] < E) {
                total.x += wk[i] * part[i].x;
                total.y += wk[i] * part[i].y;
                total.z += wk[i] * part[i].z;
                total.w += wk[i] * part[i].w;
            }
    }
    const float same = identity > 0 ? identity_weight(ids, w, top, E, identity) : 0.f;
    if (same != 0.f) {
        const bf16_four_anywhere hv = *(const bf16_four_anywhere*)(h + row * D + d);
        input = floats_anywhere{__uint_as_float(hv.x << 16), __uint_as_float(hv.x & 0xffff0000u), __uint_as_float(hv.y << 16),
                                __uint_as_float(hv.y & 0xffff0000u)};
    }
    // (as expert_down_kernel adds up, to the bit)
    const auto sum = [&](float b, float t, float x) { return b + t + (same != 0.f ? same * x : 0.f); };
    *o = floats_anywhere{sum(before.x, total.x, input.x), sum(before.y, total.y, input.y), sum(before.z, total.z, input.z), sum(before.w, total.w, input.w)};
}

// ---- the same for a few rows, the experts' weights read once, to the bit -----------------------------------
// A decode batch's picks meet in the experts: 16 rows that pick two of eight bring every expert four
// rows.  A workgroup of four waves takes the weight rows of one expert (HIDDEN: 16 hidden units' rows of gate
// and of up; else 32 outputs of down) for all of the expert's pairs, up to 16 at a time, so that weights
// are read once, past the caches.  Both operands go from memory straight into LDS, the weights into each wave's own part
// of it (the first 512 columns before the pairs are known), the pairs' rows half a step or a step ahead.
//
// A pair's sums are those of the kernels above, to the bit: chain l of 64 adds the products of columns 8 l .. + 7 of
// every 512, one after another, and the chains' sums meet by halves, quarters, ... of the 64.  A chain is a block of
// v_mfma_f32_4x4x1_16b_f32, which does one FMA for each of four weight rows and four pairs in 16 chains: twice the rate of
// the vector ALU.  (The bfloat16 MFMAs, sixteen times as fast as these, add several products up in an order of their own.  A
// step's pairs are few enough for the float ones, and with other sums than a workgroup per pair has, a router behind
// them that is not sure of a pick decides otherwise.)
// Which pairs share an expert changes no pair's result.
// Bound by the experts' bytes: sixteen experts of 4,096 x 4,096 at 16 rows, two picked, 238 us with the adding
// kernel where the weights of the experts picked take 201 at 6.5 TB/s (a workgroup per pair and 16 units, which
// read an expert's weights for every pair of its own: 742); eight of 2,048 x 2,048 47.5 us, floor 31 (203).  From eight pairs
// an expert on the MFMAs' time shows (48 rows: hidden units 45 us, 13 of them if nothing else ran; 16 rows: 31.6).
#define EC_LISTED 1024         // pairs of the step of which a workgroup lists its expert's at a time
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

// One step of the meeting of a wave's sums: lanes whose bit is clear take a, the others b, each with its partner's added.
template <int BIT>
__device__ __forceinline__ float meet(float a, float b) {
    if constexpr (BIT == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    } else if constexpr (BIT == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    } else {
        const bool set = threadIdx.x & BIT;
        const float mine = set ? b : a, theirs = set ? a : b;
        if constexpr (BIT == 8) return mine + other_lane<0x128>(theirs);                   // a rotation of 16 by 8
        else return mine + other_lane<0x1B>(other_lane<0x141>(theirs));                    // eight mirrored, then each four: lane ^ 7 ^ 3
    }
}
// N sums of 16 groups of four lanes: group b is left with that of v[b / (16 / N)].
template <int N, int BIT = 32>
__device__ __forceinline__ float meet_all(float (&v)[N]) {
    constexpr int HALF = N > 1 ? N / 2 : 1;
    float half[HALF];
#pragma unroll
    for (int i = 0; i < HALF; ++i) half[i] = meet<BIT>(v[i], v[N > 1 ? i + N / 2 : i]);
    if constexpr (BIT > 4) return meet_all<HALF, BIT / 2>(half);
    else return half[0];
}

// all but the newest n loads have arrived, n known when compiled
__device__ __forceinline__ void wait_until_newest(int n) {
    switch (n) {
#define EC_CASE(i) case i: wait_for_loads<i>(); break;
        EC_CASE(14) EC_CASE(10) EC_CASE(9) EC_CASE(8) EC_CASE(7) EC_CASE(6) EC_CASE(5) EC_CASE(4) EC_CASE(3) EC_CASE(2) EC_CASE(1)
#undef EC_CASE
        default: wait_for_loads<0>(); break;      // (fewer than allowed to be on their way is always right)
    }
}

// What a wave multiplies by: eight weight rows (HIDDEN: four of gate, four of up).  A step of 512 columns is eight pieces of a
// kilobyte, piece 2 g + half chains 16 g .. + 15 of four of the rows, lane 4 b + i chain 16 g + b of row i.  A piece has a
// place in LDS and the next step's is asked for when it has been read.
struct WeightRows {
    const bf16_t* half[2];
    unsigned row_at[2];    // this lane's row of either half, in bytes
    int K;
    unsigned lds;          // of the wave's places
    __device__ __forceinline__ void ask(int piece, int s) const {          // (past the row's end its last eight columns again)
        const int lane = threadIdx.x % 64;
        const unsigned at = row_at[piece % 2] + (unsigned)min(512 * s + 128 * (piece / 2) + 8 * (lane / 4), K - 8) * 2u;
        stream_16_bytes_to_lds(at, same_in_every_lane(half[piece % 2]), lds + piece * 1024);
    }
};

// Four PG pairs at a time; the weights' first pieces have been asked for.
template <bool HIDDEN, int PG>
__device__ __forceinline__ void expert_chains_body(const void* __restrict__ a, float* __restrict__ out, const WeightRows& rows, int top, int K, int N,
                                                   const int32_t* __restrict__ picks, const ExpertAct& xa, const int32_t* pairs, int n_here, int n0,
                                                   const char* places, const char* x, unsigned x_lds) {
    // The pairs' rows come in units of G chains' sixteenths (a step, or half of one), a unit ahead.  A kilobyte of them is, for
    // chains 16 g .. + 15 of four pairs, eight columns of bfloat16 or four of float; lane 4 b + j has chain 16 g + b of pair j.
    // A unit's kilobytes are in the order [g][four pairs][first, last four columns], and every wave asks for a quarter.
    constexpr int G = !HIDDEN && PG == 4 ? 2 : 4, UNITS = 4 / G, X_PIECES = (HIDDEN ? 1 : 2) * G * PG, X_MINE = X_PIECES / 4;
    constexpr int PG_MINE = PG / UNITS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, b = lane / 4, j = lane % 4;
    const int n_steps = (K + 511) / 512;
    const char* x_row[PG_MINE];
#pragma unroll
    for (int i = 0; i < PG_MINE; ++i) {
        const int pair = pairs[min(4 * (wave % UNITS * PG_MINE + i) + j, n_here - 1)];          // pairs past the last repeat it and are never stored
        x_row[i] = (const char*)a + (HIDDEN ? (size_t)(pair / top) * K * 2 : (size_t)pair * K * 4);
    }
    auto ask_x = [&](int unit) {
        const unsigned to = x_lds + ((unit & 1) * X_PIECES + wave * X_MINE) * 1024;
        const int c = min(128 * (G * unit + wave / UNITS) + 8 * b, K - 8);
#pragma unroll
        for (int i = 0; i < PG_MINE; ++i) {
            if constexpr (HIDDEN) {
                gather_16_bytes_to_lds(x_row[i] + c * 2, to + i * 1024);
            } else {
                gather_16_bytes_to_lds(x_row[i] + c * 4, to + i * 2048);
                gather_16_bytes_to_lds(x_row[i] + c * 4 + 16, to + i * 2048 + 1024);
            }
        }
    };
    f32x4 acc[2][PG][4];                // [half][pairs][g]: four rows of this lane's chain and pair
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int pg = 0; pg < PG; ++pg)
#pragma unroll
            for (int g = 0; g < 4; ++g) acc[h][pg][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 w;                            // this lane's 16 bytes of the piece that is next
    float xv[PG][8];                    // and the chain's eight columns of the pairs' rows
    auto inputs = [&](int s, int g, bool past_end) {
        const char* from = x + ((UNITS * s + g / G & 1) * X_PIECES + g % G * (X_PIECES / G)) * 1024 + lane * 16;
#pragma unroll
        for (int pg = 0; pg < PG; ++pg) {
            u32x4 lo, hi;
            if constexpr (HIDDEN) {
                const u32x4 v = *(const u32x4*)(from + pg * 1024);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xv[pg][2 * e] = __uint_as_float(v[e] << 16);
                    xv[pg][2 * e + 1] = __uint_as_float(v[e] & 0xffff0000u);
                }
            } else {
                lo = *(const u32x4*)(from + pg * 2048);
                hi = *(const u32x4*)(from + pg * 2048 + 1024);
#pragma unroll
                for (int e = 0; e < 4; ++e) xv[pg][e] = __uint_as_float(lo[e]), xv[pg][4 + e] = __uint_as_float(hi[e]);
            }
            if (past_end)
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[pg][e] = 0.f;
        }
    };
    auto multiply = [&](int piece) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float we = __uint_as_float(e % 2 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16);
#pragma unroll
            for (int pg = 0; pg < PG; ++pg)
                acc[piece % 2][pg][piece / 2] = __builtin_amdgcn_mfma_f32_4x4x1f32(we, xv[pg][e], acc[piece % 2][pg][piece / 2], 0, 0, 0);
        }
    };
    ask_x(0);
    wait_for_loads<0>();
    __syncthreads();
    w = *(const u32x4*)(places + lane * 16);
    for (int s = 0; s + 1 < n_steps; ++s) {
#pragma unroll
        for (int piece = 0; piece < 8; ++piece) {
            if (piece % (2 * G) == 0) {
                // this wave's share of the unit has come: a step's is older than the piece that has been waited for, half a step's than four pieces
                if (UNITS == 2) wait_for_loads<4>();
                if (s + piece > 0) __syncthreads();
                ask_x(UNITS * s + piece / (2 * G) + 1);          // into the part that has been read
            }
            if (piece % 2 == 0) inputs(s, piece / 2, false);
            // The next piece comes out of LDS meanwhile: behind it six newer ones are on their way, and the rows of the units
            // that began in the last seven turns.  (The first eight pieces have come whatever the count.)
            wait_until_newest(6 + X_MINE * ((piece % (2 * G) <= 6) + (UNITS == 2 && piece % 4 <= 2)));
            const u32x4 next = *(const u32x4*)(places + (piece + 1) % 8 * 1024 + lane * 16);
            asm volatile("" : "+v"(w));          // this piece has been read: its place takes the next step's
            rows.ask(piece, s + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(piece);
            __builtin_amdgcn_sched_barrier(0);
            w = next;
        }
    }
#pragma unroll
    for (int piece = 0; piece < 8; ++piece) {
        const bool past_end = 512 * (n_steps - 1) + 128 * (piece / 2) + 8 * b >= K;
        if (piece % (2 * G) == 0) {
            if (piece > 0) wait_for_loads<0>();
            else if (UNITS == 2) wait_for_loads<4>();
            if (n_steps > 1 || piece > 0) __syncthreads();
            if (UNITS == 2 && piece == 0) ask_x(2 * n_steps - 1);
        }
        if (piece % 2 == 0) inputs(n_steps - 1, piece / 2, past_end);
        wait_until_newest(6 - piece + (UNITS == 2 && piece < 4 ? X_MINE : 0));
        const u32x4 next = *(const u32x4*)(places + (piece + 1) % 8 * 1024 + lane * 16);          // (the last one's is not used)
        if (past_end) w = u32x4{0, 0, 0, 0};
        __builtin_amdgcn_sched_barrier(0);
        multiply(piece);
        __builtin_amdgcn_sched_barrier(0);
        w = next;
    }
    // the chains' sums: bits 5 and 4 of a chain's number are g's, the others the lane's
    float sum[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float v[4 * PG];
#pragma unroll
        for (int pg = 0; pg < PG; ++pg)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[4 * pg + r] = (acc[h][pg][0][r] + acc[h][pg][2][r]) + (acc[h][pg][1][r] + acc[h][pg][3][r]);
        sum[h] = meet_all(v);
    }
    constexpr int SAME = 4 / PG;        // groups of four lanes with the same sum
    const int at = b / SAME, col = 4 * (at / 4) + j, n = n0 + (HIDDEN ? 4 : 8) * wave + at % 4;
    if (b % SAME || col >= n_here) return;
    const int pair = pairs[col];
    float* to = out + (size_t)pair * N + n;
    if constexpr (HIDDEN) {
        const float on_input = xa.weight_on_input ? ((const float*)(picks + (size_t)(pair / top) * 2 * top + top))[pair % top] : 1.f;
        if (n < N) *to = expert_act(xa, sum[0] * on_input, sum[1] * on_input);
    } else {
        if (n < N) to[0] = sum[0];
        if (n + 4 < N) to[4] = sum[1];
    }
}

// by_pair: workgroups (., y) stand for the expert of pair y, if no earlier pair has picked it; else for expert y
template <bool HIDDEN>
__global__ __launch_bounds__(256, 2) void expert_chains_kernel(const void* __restrict__ a, const int32_t* __restrict__ picks, float* __restrict__ out,
                                                               const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1, int E, int top,
                                                               int n_pairs, int K, int N, ExpertAct xa, int by_pair) {
    extern __shared__ __attribute__((aligned(1024))) char chains_lds[];          // the waves' places | the pairs' rows of two steps
    __shared__ int32_t pairs[EC_LISTED];
    __shared__ int32_t n_listed;
    const int y = blockIdx.y;
    const int e = by_pair ? picks[(size_t)(y / top) * 2 * top + y % top] : y;
    if (e < 0 || e >= E) return;            // (uniform over the workgroup)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int n0 = blockIdx.x * (HIDDEN ? 16 : 32), first_row = n0 + (HIDDEN ? 4 : 8) * wave;
    const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) char*)chains_lds);
    WeightRows rows;
    rows.half[0] = w0 + ((size_t)e * N + n0) * K;
    rows.half[1] = HIDDEN ? w1 + ((size_t)e * N + n0) * K : rows.half[0];
#pragma unroll
    for (int h = 0; h < 2; ++h)             // (past the matrix its last row)
        rows.row_at[h] = (unsigned)(min(first_row + (HIDDEN ? 0 : 4 * h) + (int)threadIdx.x % 4, N - 1) - n0) * (unsigned)K * 2u;
    rows.K = K;
    rows.lds = lds + wave * 8192;
#pragma unroll
    for (int piece = 0; piece < 8; ++piece) rows.ask(piece, 0);          // before the pairs are known
    __builtin_amdgcn_sched_barrier(0);
    constexpr int AT_ONCE = 16;
    const char* places = chains_lds + wave * 8192;
    const char* x = chains_lds + 4 * 8192;
    bool asked = true, first_pairs = true;
    for (int from = 0; from < n_pairs; from += EC_LISTED) {
        if (from > 0) __syncthreads();      // the list before has been read
        if (threadIdx.x < 64) {
            int n = 0;
            const int end = min(n_pairs, from + EC_LISTED);
            for (int p0 = from; p0 < end; p0 += 256) {
                int got[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int p = p0 + 64 * i + (int)threadIdx.x;
                    got[i] = p < end ? picks[(size_t)(p / top) * 2 * top + p % top] : -1;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint64_t mask = __ballot(got[i] == e);
                    if (got[i] == e) pairs[n + __popcll(mask & ((1ull << threadIdx.x) - 1))] = p0 + 64 * i + (int)threadIdx.x;
                    n += __popcll(mask);
                }
            }
            if (threadIdx.x == 0) n_listed = n;
        }
        __syncthreads();
        const int n = n_listed;
        if (n == 0) continue;
        if (first_pairs && by_pair && pairs[0] != y) break;          // (an earlier pair's workgroups have the expert)
        first_pairs = false;
        for (int first = 0; first < n; first += AT_ONCE) {
            const int n_here = min(AT_ONCE, n - first);
            if (!asked) {
                __syncthreads();            // the pairs before have been read
#pragma unroll
                for (int piece = 0; piece < 8; ++piece) rows.ask(piece, 0);
            }
            asked = false;
            if (n_here <= 4) expert_chains_body<HIDDEN, 1>(a, out, rows, top, K, N, picks, xa, pairs + first, n_here, n0, places, x, lds + 4 * 8192);
            else if (n_here <= 8) expert_chains_body<HIDDEN, 2>(a, out, rows, top, K, N, picks, xa, pairs + first, n_here, n0, places, x, lds + 4 * 8192);
            else expert_chains_body<HIDDEN, 4>(a, out, rows, top, K, N, picks, xa, pairs + first, n_here, n0, places, x, lds + 4 * 8192);
        }
    }
    if (asked) wait_for_loads<0>();         // (nothing may be written to LDS that is another's by then)
}

template <bool HIDDEN>
static int launch_expert_chains(const void* a, const int32_t* picks, float* out, const bf16_t* w0, const bf16_t* w1, int E, int top, int rows, int K,
                                int N, const ExpertAct& xa, hipStream_t stream) {
    const int n_pairs = rows * top, by_pair = n_pairs < E;
    constexpr size_t lds = 64 * 1024;
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void*)expert_chains_kernel<HIDDEN>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        PICOLM_REQUIRE(e == hipSuccess, "routed_experts: cannot raise the LDS limit to %zu: %s", lds, hipGetErrorString(e));
        raised = true;
    }
    const dim3 grid((unsigned)ceil_div(N, HIDDEN ? 16 : 32), (unsigned)(by_pair ? n_pairs : E));
    expert_chains_kernel<HIDDEN><<<grid, 256, lds, stream>>>(a, picks, out, w0, w1, E, top, n_pairs, K, N, xa, by_pair);
    PICOLM_LAUNCH_CHECK("routed_experts (in chains)");
    return 0;
}

// ---- the same for some more rows: bfloat16 MFMAs -----------------------------------------------------------
// A workgroup of four waves takes the weight rows of one expert as above, for up to 64 of the expert's pairs at a
// time.  The waves take K in turns of 64 columns; a wave's loads go straight into LDS stages
// of its own, a kilobyte each (as in gemm_skinny_staged_kernel of gemm_mfma.hip), weights as the first operand
// of v_mfma_f32_16x16x32_bf16 and the pairs' rows as the second; the waves' sums meet in LDS in a fixed order.
// The hidden units stay float: a wave takes a float's three bfloat16 parts of eight bits each, which add
// up to it exactly, through three MFMAs, so that every product is exact and sums are float.
// Which pairs share an expert changes no pair's result.
// Bound by the experts' bytes: sixteen experts of 4,096 x 4,096 at 64 rows, two picked, 263 us with the adding
// kernel where the weights of the experts picked take 248 at 6.5 TB/s; 64 of 1,408 x 2,048, six picked, 213 us, floor 170.
#define ES_MOST_PAIRS 512      // pairs of one expert that a workgroup lists (a row picks an expert once)
// eight floats as three bfloat16 chunks: x = hi + mid + lo (a number that is not finite lies in hi alone), as in Henry, Tang and
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019
__device__ __forceinline__ void split_chunk(const f32x4& x0, const f32x4& x1, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned hp[2], mp[2], lp[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float x = i < 2 ? x0[2 * i + j] : x1[2 * i - 4 + j];
            hp[j] = __float_as_uint(x) & 0xffff0000u;
            const float rest = __builtin_isfinite(x) ? x - __uint_as_float(hp[j]) : 0.f;
            mp[j] = __float_as_uint(rest) & 0xffff0000u;
            lp[j] = __float_as_uint(rest - __uint_as_float(mp[j]));
        }
        h[i] = (hp[0] >> 16) | hp[1];
        m[i] = (mp[0] >> 16) | mp[1];
        l[i] = (lp[0] >> 16) | (lp[1] & 0xffff0000u);
    }
    hi = __builtin_bit_cast(bf16x8, h);
    mid = __builtin_bit_cast(bf16x8, m);
    lo = __builtin_bit_cast(bf16x8, l);
}
__device__ __forceinline__ void wait_for_stages(int stages, int loads) {      // all but the newest `stages` of `loads` loads each
    switch (stages * loads) {
#define ES_CASE(i) case i: wait_for_loads<i>(); break;
        ES_CASE(5) ES_CASE(6) ES_CASE(7) ES_CASE(8) ES_CASE(9) ES_CASE(10) ES_CASE(11) ES_CASE(12) ES_CASE(13) ES_CASE(14)
        ES_CASE(15) ES_CASE(16) ES_CASE(17) ES_CASE(18) ES_CASE(19) ES_CASE(20) ES_CASE(21) ES_CASE(22) ES_CASE(24) ES_CASE(25)
        ES_CASE(26) ES_CASE(27) ES_CASE(28) ES_CASE(30) ES_CASE(32) ES_CASE(33) ES_CASE(35) ES_CASE(36) ES_CASE(39) ES_CASE(40)
        ES_CASE(42)
#undef ES_CASE
        default: wait_for_loads<0>(); break;      // (fewer than allowed to be on their way is always right)
    }
}

// MT: tiles of 16 pairs at a time
template <bool HIDDEN, int MT>
__device__ __forceinline__ void expert_stream_body(const void* __restrict__ a, float* __restrict__ out, const bf16_t* __restrict__ w0,
                                                   const bf16_t* __restrict__ w1, int top, int K, int N, const int32_t* __restrict__ picks,
                                                   const ExpertAct& xa, const int32_t* pairs, int n_pairs, int n0, char* lds, int wave_bytes) {
    constexpr int A_ROWS = HIDDEN ? 8 : 4, A_LOADS = 16 * MT / A_ROWS;       // pairs' rows in a kilobyte: 64 columns of bfloat16 or of float
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, r16 = lane % 16, q = lane / 16;
    const char* my_lds = lds + wave * wave_bytes;
    const unsigned lds_wave = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) char*)lds + wave * wave_bytes);
    const int lrow = lane / 8, lslot = lane % 8;
    unsigned w_off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 8 * i + lrow, local = HIDDEN ? row % 16 : row;
        w_off[i] = (unsigned)(min(local, N - 1 - n0) * K * 2 + (lslot ^ ((row >> 1) & 7)) * 16);
    }
    for (int first = 0; first < n_pairs; first += 16 * MT) {
        const int n_here = min(16 * MT, n_pairs - first);
        const int a_loads = (n_here + A_ROWS - 1) / A_ROWS;                   // pairs past the last repeat it and are never stored
        unsigned a_off[A_LOADS];
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            const int row = A_ROWS * i + lane / (64 / A_ROWS), slot = lane % (64 / A_ROWS);
            const int pair = pairs[first + min(row, n_here - 1)];
            a_off[i] = HIDDEN ? (unsigned)(pair / top * K * 2 + (slot ^ ((row >> 1) & 7)) * 16) : (unsigned)(pair * K * 4 + (slot ^ (row & 15)) * 16);
        }
        const int stage_bytes = (4 + a_loads) * 1024, per_step = 4 + a_loads;
        int n_stages = min(wave_bytes / stage_bytes, 8);
        while (n_stages > 1 && (n_stages - 1) * per_step > 42) --n_stages;
        const int n_slices = K / 64, n_mine = wave < n_slices ? (n_slices - wave + 3) / 4 : 0;
        auto issue = [&](int k) {
            const unsigned to = lds_wave + (k % n_stages) * stage_bytes;
            const int k0 = (wave + 4 * k) * 64;
            const void* src0 = same_in_every_lane(w0 + k0);
            const void* src1 = HIDDEN ? same_in_every_lane(w1 + k0) : src0;
#pragma unroll
            for (int i = 0; i < 4; ++i) stream_16_bytes_to_lds(w_off[i], i < 2 ? src0 : src1, to + i * 1024);
            const void* asrc = same_in_every_lane((const char*)a + (size_t)k0 * (HIDDEN ? 2 : 4));
#pragma unroll
            for (int i = 0; i < A_LOADS; ++i)
                if (i < a_loads) load_16_bytes_to_lds(a_off[i], asrc, to + (4 + i) * 1024);
        };
        f32x4 acc[2][MT];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < MT; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < min(n_stages, n_mine); ++k) issue(k);
        for (int k = 0; k < n_mine; ++k) {
            wait_for_stages(min(n_stages - 1, n_mine - 1 - k), per_step);
            __builtin_amdgcn_sched_barrier(0);
            const char* st = my_lds + (k % n_stages) * stage_bytes;
            const char* as = st + 4096;
            bf16x8 wf[2][2];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = 16 * t + r16;
                    wf[t][j] = *(const bf16x8*)(st + row * 128 + (((4 * j + q) ^ ((row >> 1) & 7)) * 16));
                }
#pragma unroll
            for (int u = 0; u < MT; ++u) {
                if (u * 16 >= n_here) break;
                const int row = (16 * u + r16) % (A_ROWS * a_loads);          // (rows that were not loaded repeat loaded ones)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if constexpr (HIDDEN) {
                        const bf16x8 af = *(const bf16x8*)(as + row * 128 + (((4 * j + q) ^ ((row >> 1) & 7)) * 16));
#pragma unroll
                        for (int t = 0; t < 2; ++t) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][j], af, acc[t][u], 0, 0, 0);
                    } else {
                        const int c = 8 * j + 2 * q;
                        const f32x4 x0 = *(const f32x4*)(as + row * 256 + ((c ^ (row & 15)) * 16));
                        const f32x4 x1 = *(const f32x4*)(as + row * 256 + (((c + 1) ^ (row & 15)) * 16));
                        bf16x8 hi, mid, lo;
                        split_chunk(x0, x1, hi, mid, lo);
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][j], lo, acc[t][u], 0, 0, 0);
                            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][j], mid, acc[t][u], 0, 0, 0);
                            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][j], hi, acc[t][u], 0, 0, 0);
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (k + n_stages < n_mine) issue(k + n_stages);
        }
        // the waves' sums, each into its own stages: [tile t][tile u][r][lane]
        float* red = (float*)my_lds;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < MT; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[((t * MT + u) * 4 + r) * 64 + lane] = acc[t][u][r];
        __syncthreads();
        for (int v = threadIdx.x; v < (HIDDEN ? 16 : 32) * 16 * MT; v += 256) {
            const int n = v % (HIDDEN ? 16 : 32), col = v / (HIDDEN ? 16 : 32);      // a weight row of the tile, a pair
            if (col >= n_here || n0 + n >= N) continue;
            const int at = ((n / 16 * MT + col / 16) * 4 + n % 4) * 64 + n % 16 / 4 * 16 + col % 16;
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float* part = (const float*)(lds + w * wave_bytes);
                s0 += part[at];
                if (HIDDEN) s1 += part[at + MT * 256];
            }
            const int pair = pairs[first + col];
            if (HIDDEN) {
                const float on_input = xa.weight_on_input ? ((const float*)(picks + (size_t)(pair / top) * 2 * top + top))[pair % top] : 1.f;
                out[(size_t)pair * N + n0 + n] = expert_act(xa, s0 * on_input, s1 * on_input);
            } else {
                out[(size_t)pair * N + n0 + n] = s0;
            }
        }
        __syncthreads();                    // (before the next pairs' stages)
    }
}

// by_pair: workgroup x stands for the expert of pair x, if no earlier pair has picked it; else for expert x
template <bool HIDDEN>
__global__ __launch_bounds__(256, 2) void expert_stream_kernel(const void* __restrict__ a, const int32_t* __restrict__ picks, float* __restrict__ out,
                                                               const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1, int E, int top,
                                                               int n_pairs, int K, int N, ExpertAct xa, int by_pair, int wave_bytes) {
    extern __shared__ __attribute__((aligned(1024))) char stream_lds[];
    __shared__ int32_t pairs[ES_MOST_PAIRS];
    __shared__ int32_t n_listed;
    const int x = blockIdx.x;
    const int e = by_pair ? picks[(size_t)(x / top) * 2 * top + x % top] : x;
    if (e < 0 || e >= E) return;            // (uniform over the workgroup)
    if (threadIdx.x < 64) {
        int n = 0;
        for (int p0 = 0; p0 < n_pairs; p0 += 256) {
            int got[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int p = p0 + 64 * i + (int)threadIdx.x;
                got[i] = p < n_pairs ? picks[(size_t)(p / top) * 2 * top + p % top] : -1;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int p = p0 + 64 * i + (int)threadIdx.x;
                const bool mine = p < n_pairs && got[i] == e;
                const uint64_t mask = __ballot(mine);
                if (by_pair && __ballot(mine && p < x) != 0) n = INT32_MIN / 2;      // an earlier pair's workgroup has it
                const int at = n + __popcll(mask & ((1ull << threadIdx.x) - 1));
                if (mine && at >= 0 && at < ES_MOST_PAIRS) pairs[at] = p;
                n += __popcll(mask);
            }
        }
        if (threadIdx.x == 0) n_listed = n;
    }
    __syncthreads();
    const int n = min(n_listed, ES_MOST_PAIRS);
    if (n <= 0) return;
    const int n0 = blockIdx.y * (HIDDEN ? 16 : 32);
    const bf16_t* rows0 = w0 + ((size_t)e * N + n0) * K;
    const bf16_t* rows1 = HIDDEN ? w1 + ((size_t)e * N + n0) * K : nullptr;
    if (n <= 16) expert_stream_body<HIDDEN, 1>(a, out, rows0, rows1, top, K, N, picks, xa, pairs, n, n0, stream_lds, wave_bytes);
    else if (n <= 32 || wave_bytes < (4 + 64 / (HIDDEN ? 8 : 4)) * 1024) expert_stream_body<HIDDEN, 2>(a, out, rows0, rows1, top, K, N, picks, xa, pairs, n, n0, stream_lds, wave_bytes);
    else expert_stream_body<HIDDEN, 4>(a, out, rows0, rows1, top, K, N, picks, xa, pairs, n, n0, stream_lds, wave_bytes);
}

template <bool HIDDEN>
static int launch_expert_stream(const void* a, const int32_t* picks, float* out, const bf16_t* w0, const bf16_t* w1, int E, int top, int rows, int K,
                                int N, const ExpertAct& xa, hipStream_t stream) {
    const int n_pairs = rows * top, by_pair = n_pairs < E;
    // two workgroups a CU while an expert's pairs are few; all of the LDS for one where their rows are as wide as the weights
    const int wave_bytes = (n_pairs > 16 * E ? 38 : 18) * 1024;
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void*)expert_stream_kernel<HIDDEN>, hipFuncAttributeMaxDynamicSharedMemorySize, 4 * 38 * 1024);
        PICOLM_REQUIRE(e == hipSuccess, "routed_experts: cannot raise the LDS limit: %s", hipGetErrorString(e));
        raised = true;
    }
    const dim3 grid((unsigned)(by_pair ? n_pairs : E), (unsigned)ceil_div(N, HIDDEN ? 16 : 32));
    expert_stream_kernel<HIDDEN><<<grid, 256, 4 * wave_bytes, stream>>>(a, picks, out, w0, w1, E, top, n_pairs, K, N, xa, by_pair, wave_bytes);
    PICOLM_LAUNCH_CHECK("routed_experts (streamed)");
    return 0;
}

// The products of a prompt's pairs.  K in whole lines and 16-byte aligned: operands straight into LDS,
// 256 weight rows a tile where that fills the CUs (not counting the tiles by which experts overlap),
// else 128, twice the workgroups; other widths are staged through registers.
template <bool HIDDEN>
static int grouped_product(const bf16_t* a, const int32_t* plan, void* out, const bf16_t* w0, const bf16_t* w1, int E, int top, int K, int N,
                           int64_t n_pairs, const int32_t* picks, const ExpertAct& xa, hipStream_t stream) {
    const unsigned tiles = (unsigned)(ceil_div64(n_pairs, GM_ROWS) + E);      // no more than these are filled; the rest leave at once
    if (K % GD_BK == 0 && K <= (1 << 21) && (((uintptr_t)a | (uintptr_t)w0 | (uintptr_t)w1) & 15) == 0) {
        const int64_t filled = ceil_div64(n_pairs, GM_ROWS);
        if (filled * ceil_div(N, HIDDEN ? 128 : 256) >= n_compute_units())
            return launch_grouped_direct<HIDDEN, 4, 3>(a, plan, out, w0, w1, E, top, K, N, tiles, picks, xa, stream);
        return launch_grouped_direct<HIDDEN, 2, 2>(a, plan, out, w0, w1, E, top, K, N, tiles, picks, xa, stream);
    }
    grouped_tile_kernel<HIDDEN><<<dim3(tiles, ceil_div(N, GM_COLS)), 256, 0, stream>>>(a, plan, out, w0, w1, E, top, K, N, picks, xa);
    PICOLM_LAUNCH_CHECK("routed_experts (grouped)");
    return 0;
}

#define GM_FROM_ROWS 64      // rows of a step from which the matrix cores take the experts

// What either kind of kernels that read an expert's weights once needs: bfloat16 throughout, 16-byte aligned buffers and rows,
// and room for the pairs' outputs
static bool reads_weights_once(const picolm_routed_experts_args* a, const picolm_step_view* v, int widths_in) {
    return v->dtype == PICOLM_BF16 && a->weight_dt == PICOLM_BF16 && a->width % widths_in == 0 && a->ff % widths_in == 0 && v->extra[2] &&
           v->extra_row_bytes[2] >= (int64_t)a->top * a->width * 4 &&
           (((uintptr_t)v->in | (uintptr_t)v->out | (uintptr_t)v->extra[1] | (uintptr_t)v->extra[2] | (uintptr_t)a->gate | (uintptr_t)a->up |
             (uintptr_t)a->down) & 15) == 0;
}
// Below 64 rows every kernel gives a row the same bits, and the chains are the fastest that do: eight experts of 2,048 x
// 2,048, two picked, 16 rows 47.5 us against 203 with a workgroup per pair, 32 rows 55 and 63 rows 83.  (The bfloat16 MFMAs
// take 46 to 51 at any of these, in another order of sums.)
static bool takes_chains(const picolm_routed_experts_args* a, const picolm_step_view* v) {
    return v->rows < GM_FROM_ROWS && a->experts <= 65535 && (int64_t)v->rows * a->top <= 65535 && reads_weights_once(a, v, 8);
}
// From 64 rows on the streamed kernels, until an expert has more pairs than their tiles of 16 take in two turns; then the tiles of
// 128 pairs win: 2,048 x 2,048, 20 pairs an expert 72 against 81 us, 24 80 against 81, 48 108 against 85; sixteen
// experts of 4,096 x 4,096, 16 pairs an expert 317 against some 340 us, 24 433 against 345.
#define ES_MOST_ROWS 255
#define ES_PAIRS_AN_EXPERT 20
static bool streams_experts(const picolm_routed_experts_args* a, const picolm_step_view* v) {
    return v->rows >= GM_FROM_ROWS && v->rows <= ES_MOST_ROWS && (int64_t)v->rows * a->top <= (int64_t)ES_PAIRS_AN_EXPERT * a->experts &&
           reads_weights_once(a, v, 64) && (int64_t)v->rows * a->top * a->ff < (1ll << 29) && (int64_t)v->rows * a->width < (1ll << 30) &&
           32ll * a->width < (1ll << 30) && 32ll * a->ff < (1ll << 30);
}

extern "C" int picolm_call_routed_experts(void* user, const picolm_step_view* v) {
    const picolm_routed_experts_args* a = (const picolm_routed_experts_args*)user;
    VIEW_REQUIRE("routed_experts", v);
    PICOLM_REQUIRE(a && a->gate && a->up && a->down && v->in && v->out && v->extra[0] && v->extra[1], "routed_experts: weights or buffers are missing");
    const int E = a->experts, top = a->top, D = a->width, F = a->ff;
    PICOLM_REQUIRE(E > 0 && top > 0 && a->identity >= 0 && top <= E + a->identity && D > 0 && F > 0 && (a->weight_dt == PICOLM_F32 || a->weight_dt == PICOLM_BF16),
                   "routed_experts: %d picks among %d experts of %d to %d", top, E, D, F);
    PICOLM_REQUIRE(v->dtype == PICOLM_BF16 || a->weight_dt == PICOLM_F32, "routed_experts: the 32-bit engine takes 32-bit weights");
    PICOLM_REQUIRE(v->in_row_bytes >= D * elem_bytes(v->dtype) && v->out_row_bytes >= D * 4 && v->extra_row_bytes[0] >= 2 * top * 4 &&
                       v->extra_row_bytes[1] >= (int64_t)top * F * 4,
                   "routed_experts: rows too short for a width of %d, %d picks and %d hidden units", D, top, F);
    PICOLM_REQUIRE(a->act == 0 || (a->act == 1 && a->limit > 0.f), "routed_experts: activation %d (limit %g) is not known", a->act, (double)a->limit);
    PICOLM_REQUIRE(!a->weight_on_input || a->identity == 0, "routed_experts: weights on the experts' input and picks that give the input back do not go together");
    const ExpertAct xa = {a->act, a->limit, a->alpha, a->weight_on_input};
    const int plain_sum = a->weight_on_input ? 1 : 0;
    const size_t lds_a = sizeof(float) * (size_t)D, lds_b = sizeof(float) * (size_t)top * F;
    PICOLM_REQUIRE(lds_a <= 64 * 1024 && lds_b <= 64 * 1024, "routed_experts: a width of %d or %d picks of %d hidden units exceed 64 KiB of LDS", D,
                   top, F);
    PICOLM_REQUIRE(ceil_div(F, MOE_UNITS) <= 65535 && ceil_div(D, MOE_UNITS) <= 65535 && (int64_t)v->rows * top < (1ll << 31),
                   "routed_experts: the sizes exceed the grid");
    if (v->rows <= 0) return 0;
    const int32_t* picks = (const int32_t*)v->extra[0];
    float* act = (float*)v->extra[1];
    const bool chains = takes_chains(a, v);
    if (chains || streams_experts(a, v)) {
        float* y = (float*)v->extra[2];
        int rc = (chains ? launch_expert_chains<true> : launch_expert_stream<true>)(v->in, picks, act, (const bf16_t*)a->gate, (const bf16_t*)a->up, E, top, v->rows, D, F, xa, v->stream);
        if (rc) return rc;
        rc = (chains ? launch_expert_chains<false> : launch_expert_stream<false>)(act, picks, y, (const bf16_t*)a->down, nullptr, E, top, v->rows, F, D, xa, v->stream);
        if (rc) return rc;
        grouped_sum_kernel<<<dim3(v->rows, ceil_div(D, 1024)), 256, 0, v->stream>>>(y, picks, (float*)v->out, E, top, D, a->adds, (const bf16_t*)v->in,
                                                                                   a->identity, plain_sum);
        PICOLM_LAUNCH_CHECK("routed_experts (sum)");
        return 0;
    }
    if (v->dtype == PICOLM_BF16 && a->weight_dt == PICOLM_BF16 && v->rows >= GM_FROM_ROWS && D % 16 == 0 && F % 16 == 0 && E <= GM_MAX_EXPERTS &&
        v->extra[2] && v->extra[3]) {
        const int64_t n_pairs = (int64_t)v->rows * top;
        PICOLM_REQUIRE(v->extra_row_bytes[2] >= (int64_t)top * D * 4 && v->extra_row_bytes[3] >= (int64_t)(top + E + 1) * 4,
                       "routed_experts: scratch rows too short for the sorted pairs or their outputs");
        int32_t* plan = (int32_t*)v->extra[3];
        float* y = (float*)v->extra[2];
        moe_plan_kernel<<<1, 1024, sizeof(int32_t) * (2 * (size_t)E + 1), v->stream>>>(picks, plan, E, top, (int)n_pairs);
        PICOLM_LAUNCH_CHECK("routed_experts (plan)");
        int rc = grouped_product<true>((const bf16_t*)v->in, plan, act, (const bf16_t*)a->gate, (const bf16_t*)a->up, E, top, D, F, n_pairs, picks, xa,
                                       v->stream);
        if (rc) return rc;
        rc = grouped_product<false>((const bf16_t*)act, plan, y, (const bf16_t*)a->down, nullptr, E, top, F, D, n_pairs, picks, xa, v->stream);
        if (rc) return rc;
        grouped_sum_kernel<<<dim3(v->rows, ceil_div(D, 1024)), 256, 0, v->stream>>>(y, picks, (float*)v->out, E, top, D, a->adds, (const bf16_t*)v->in, a->identity, plain_sum);
        PICOLM_LAUNCH_CHECK("routed_experts (sum)");
        return 0;
    }
    const dim3 grid_a((unsigned)(v->rows * top), ceil_div(F, MOE_UNITS)), grid_b(v->rows, ceil_div(D, MOE_UNITS));
    if (a->weight_dt == PICOLM_F32 && v->dtype == PICOLM_F32) {
        expert_hidden_kernel<float, float><<<grid_a, 256, lds_a, v->stream>>>((const float*)v->in, picks, act, (const float*)a->gate,
                                                                              (const float*)a->up, E, top, D, F, xa);
        PICOLM_LAUNCH_CHECK("routed_experts (hidden)");
        expert_down_kernel<float, float><<<grid_b, 256, lds_b, v->stream>>>(act, picks, (float*)v->out, (const float*)a->down, E, top, D, F, a->adds,
                                                                            (const float*)v->in, a->identity, plain_sum);
    } else if (a->weight_dt == PICOLM_F32) {
        expert_hidden_kernel<float, bf16_t><<<grid_a, 256, lds_a, v->stream>>>((const bf16_t*)v->in, picks, act, (const float*)a->gate,
                                                                               (const float*)a->up, E, top, D, F, xa);
        PICOLM_LAUNCH_CHECK("routed_experts (hidden)");
        expert_down_kernel<float, bf16_t><<<grid_b, 256, lds_b, v->stream>>>(act, picks, (float*)v->out, (const float*)a->down, E, top, D, F, a->adds,
                                                                             (const bf16_t*)v->in, a->identity, plain_sum);
    } else {
        expert_hidden_kernel<bf16_t, bf16_t><<<grid_a, 256, lds_a, v->stream>>>((const bf16_t*)v->in, picks, act, (const bf16_t*)a->gate,
                                                                                (const bf16_t*)a->up, E, top, D, F, xa);
        PICOLM_LAUNCH_CHECK("routed_experts (hidden)");
        expert_down_kernel<bf16_t, bf16_t><<<grid_b, 256, lds_b, v->stream>>>(act, picks, (float*)v->out, (const bf16_t*)a->down, E, top, D, F, a->adds,
                                                                              (const bf16_t*)v->in, a->identity, plain_sum);
    }
    PICOLM_LAUNCH_CHECK("routed_experts (down)");
    return 0;
}
