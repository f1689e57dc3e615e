// Gated GQA attention for one decode token on the device, between q/k/v_proj
// and o_proj: the numerics of QwenCPUModel.attentionForward for one token
// (QwenCPUModel.swift:285-345, applyRope :348-367), which the reference's
// GPU path runs on the host (attnCoreCPU, QwenMetalModel.swift:1086-1134).
//
// Two launches, split over the cached positions:
//   attn_partial  grid (splits, KVH): the group's queries RMS-normalised
//                 (q_norm) and rotated (partial NeoX RoPE), the new key likewise
//                 (k_norm) and appended with the new value by the split holding
//                 the current position; then the split's maximum, sum and sum
//                 of p * v per query head, with an online softmax.
//   attn_combine  grid (H, blocks of 64 dims): the splits merged
//                 (exp(m_s - M) weights), divided by the total, times
//                 sigmoid(gate).
// The cache is f32 [max_positions][KVH][hd] for k and for v, the order in
// which the reference appends rows (state.kv).
#include <algorithm>
#include <cmath>

#include "internal.hpp"
#include "route.hpp"

namespace swq {
namespace {

constexpr int kAttnMaxGroup = 16;  // query heads per kv head
constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / kWave;
constexpr int kAttnHeadsPerWave = kAttnMaxGroup / kAttnWaves;
constexpr int kAttnMaxSplits = 512;
constexpr int kAttnTargetWgs = 512;
constexpr int kAttnMaxRot = 256;

struct AttnArgs {
    const float *q_proj, *k_proj, *v_proj;
    const float *q_norm_w, *k_norm_w;
    float *cache_k, *cache_v;
    float *part;     // [H][splits][hd]: the splits' value sums
    float *part_ml;  // [H][splits][2]: their maxima and sums
    float *out;   // [H * hd]
    int32_t H, KVH, hd, rot, group, splits;
    int32_t per;  // positions per split
    int32_t position;
    float theta, eps, scale;
    // the rotation of `position`: cos and sin of position * theta^(-2j/rot),
    // j < rot/2, from the host (kernel arguments)
    float rope_cos[kAttnMaxRot / 2], rope_sin[kAttnMaxRot / 2];
};

__device__ __forceinline__ float sigmoid_acc(float v) { return 1.0f / (1.0f + expf(-v)); }


// Element e of a head vector held EPL per lane (lanes >= HD / EPL hold none).
template <int HD>
struct HeadVec {
    static constexpr int EPL = HD >= kWave ? HD / kWave : 1;
    static constexpr int LANES = HD / EPL;
    float v[EPL];
};

// This lane's elements of the norm weight, and of the rotation table at them:
// element i < rot turns with its partner i +- rot / 2 by angle i % (rot / 2).
template <int HD>
struct HeadTable {
    static constexpr int EPL = HeadVec<HD>::EPL;
    float w[EPL], c[EPL], s[EPL];
    __device__ __forceinline__ void load(const float *weight, const AttnArgs &a) {
        const int lane = threadIdx.x & (kWave - 1), half = a.rot / 2;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const int i = min(lane * EPL + e, HD - 1);
            w[e] = weight[i];
            const int j = i < half ? i : (i < a.rot ? i - half : 0);
            c[e] = a.rope_cos[j];
            s[e] = a.rope_sin[j];
        }
    }
};

template <int HD>
__device__ __forceinline__ void load_head(HeadVec<HD> &x, const float *src) {
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int e = 0; e < HeadVec<HD>::EPL; ++e)
        x.v[e] = lane < HeadVec<HD>::LANES ? src[lane * HeadVec<HD>::EPL + e] : 0.f;
}

// RMS-normalise a head vector (x *= scale * w) and rotate its first `rot`
// elements (pairs j, j + rot/2), in the reference's operation order.  The
// wave's copy goes through `lds` (HD floats) so that a lane can read its
// rotation partner.
template <int HD>
__device__ __forceinline__ void norm_rope(HeadVec<HD> &x, const HeadTable<HD> &t, float eps, int rot, float *lds) {
    constexpr int EPL = HeadVec<HD>::EPL, LANES = HeadVec<HD>::LANES;
    const int lane = threadIdx.x & (kWave - 1);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) ss += x.v[e] * x.v[e];
    ss = wave_sum_all(ss);
    const float sc = 1.0f / __fsqrt_rn(ss / static_cast<float>(HD) + eps);
    if (lane < LANES) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            x.v[e] *= sc * t.w[e];
            lds[lane * EPL + e] = x.v[e];
        }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int half = rot / 2;
    if (lane < LANES) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const int i = lane * EPL + e;
            const float o = lds[i < half ? i + half : (i < rot ? i - half : i)];
            if (i < rot) x.v[e] = i < half ? x.v[e] * t.c[e] - o * t.s[e] : x.v[e] * t.c[e] + o * t.s[e];
        }
    }
}

// One workgroup of four waves per (split, kv head), a quarter of the head's
// dims on each wave, walking the split's positions TILES * 16 at a time on the
// fp32 matrix cores (v_mfma_f32_16x16x4_f32: 32-bit products and sums), K and V
// straight from global memory to the operands, never through LDS:
//   scores  A = K: lane (r = lane % 16, q = lane / 16) holds position r's dims
//           4 KW j + KW q + e (one load of KW floats per j), B = the group's
//           queries in the same dim order, in registers; the result's lane
//           (h, q) holds head h's partial scores at positions 4 q + i, i < 4;
//           the four waves' partials meet in LDS, one barrier per step;
//   softmax online, a running maximum and sum per head, on every wave alike;
//   values  A = p: the scores' registers are the operand as they are (k step i
//           takes positions 4 q + i), B = V: lane (n, q) holds dims VW n + e of
//           position 4 q + i; the result's lane (n, q) holds heads 4 q + i of
//           the wave's dims, so no sum crosses waves.
// Heads past the group are zero queries whose results nothing reads.  The next
// step's K loads are issued before this one's values, its V loads after them.
//
// Bound: at short contexts the chain of launch, first loads, norm and rotation,
// barrier, two products (~5 us), at long ones the bytes: 33,001 positions read
// 135 MB in 33 us, 4.1 TB/s.  Before, with scores and values on the VALU over K
// transposed in LDS (120 KB, one workgroup per CU): 59 us there and 13 us at
// 4,096 positions, now 8.9.  Measured beside it: 4-wave workgroups with every
// dim on each wave, 16 positions a wave, sums merged through LDS, 13.3 us at
// 4,096 and 33 us; four tiles a step (spills), 48 us at 33,001.
template <int HD>
struct AttnDims {
    static constexpr int DW = HD / kAttnWaves;           // dims per wave
    static constexpr int KW = DW >= 16 ? 4 : DW / 4;     // floats per K load
    static constexpr int J = DW / (4 * KW);              // K loads per lane and position
    static constexpr int VW = DW >= 16 ? DW / 16 : 1;    // floats per V load (lanes past the dims idle)
};

template <int W>
__device__ __forceinline__ void load_floats(float (&d)[W], const float *p) {
    if constexpr (W == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
    } else if constexpr (W == 2) {
        const float2 v = *reinterpret_cast<const float2 *>(p);
        d[0] = v.x; d[1] = v.y;
    } else {
        d[0] = *p;
    }
}

// The maximum that exponents are taken against: 0 where every score so far is -inf, so that
// such positions count nothing instead of turning the sum into NaN.
__device__ __forceinline__ float finite_max(float m) { return m == -INFINITY ? 0.f : m; }

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <int HD, int TILES>  // TILES 1: splits of at most 16 positions; 2: any
__global__ __launch_bounds__(kAttnThreads, 2) void attn_partial(const AttnArgs a) {
    using D = AttnDims<HD>;
    constexpr int DW = D::DW, KW = D::KW, J = D::J, VW = D::VW;
    constexpr int EPL = HeadVec<HD>::EPL;
    constexpr int STEP = 16 * TILES;
    __shared__ __attribute__((aligned(16))) float s_q[kAttnMaxGroup * HD];  // operand order
    __shared__ __attribute__((aligned(16))) float s_rot[kAttnMaxGroup * HD];
    __shared__ __attribute__((aligned(16))) float s_new[HD];                // the new key
    __shared__ f32x4_t s_s[2][kAttnWaves][TILES][kWave];
    const int split = blockIdx.x, g = blockIdx.y;
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid & (kWave - 1);
    const int r = lane & 15, q = lane >> 4;
    const int G = a.group;
    const int64_t row = static_cast<int64_t>(a.KVH) * HD;
    const int p0 = split * a.per, p1 = min(p0 + a.per, a.position + 1);  // this split's positions: never empty

    // this wave's queries (heads wave, wave + 4, ...) and the tables, ahead of K and V
    HeadVec<HD> qx[kAttnHeadsPerWave];
    HeadTable<HD> qt;
    qt.load(a.q_norm_w, a);
#pragma unroll
    for (int u = 0; u < kAttnHeadsPerWave; ++u)
        load_head<HD>(qx[u], a.q_proj + static_cast<int64_t>(g * G + min(u * kAttnWaves + wave, G - 1)) * 2 * HD);
    // and, on the last wave of the split that holds the new position, its key
    const bool has_new = wave == kAttnWaves - 1 && a.position < p1;
    HeadVec<HD> kx, vx;
    HeadTable<HD> kt = qt;
    if (has_new) {
        load_head<HD>(kx, a.k_proj + g * HD);
        load_head<HD>(vx, a.v_proj + g * HD);
#pragma unroll
        for (int e = 0; e < EPL; ++e) kt.w[e] = a.k_norm_w[min(lane * EPL + e, HD - 1)];
    }

    float kr[TILES][J][KW], vr[TILES][4][VW];
    const float *ck = a.cache_k + g * HD + wave * DW + KW * q;
    const float *cv = a.cache_v + g * HD + wave * DW + min(VW * r, DW - VW);
    // K and V of the step at t0; rows past the split's positions read its last one
    auto load_k = [&](int t0) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float *p = ck + min(t0 + 16 * t + r, p1 - 1) * row;
#pragma unroll
            for (int j = 0; j < J; ++j) load_floats<KW>(kr[t][j], p + 4 * KW * j);
        }
    };
    auto load_v = [&](int t0) {
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) load_floats<VW>(vr[t][i], cv + min(t0 + 16 * t + 4 * q + i, p1 - 1) * row);
    };
    load_k(p0);
    load_v(p0);

    // the new position's key and value: into the cache, the key into LDS too
    if (has_new) {
        norm_rope<HD>(kx, kt, a.eps, a.rot, s_new);
        __builtin_amdgcn_wave_barrier();
        const int64_t at = a.position * row + g * HD;
        if (lane < HeadVec<HD>::LANES) {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const int i = lane * EPL + e;
                s_new[i] = kx.v[e];
                a.cache_k[at + i] = kx.v[e];
                a.cache_v[at + i] = vx.v[e];
            }
        }
    }
    // the group's queries, into operand order: element i of head h at lane
    // (h, q), load j of its wave; zeros for the heads past the group
#pragma unroll
    for (int u = 0; u < kAttnHeadsPerWave; ++u) {
        const int hh = u * kAttnWaves + wave;
        if (hh < G) norm_rope<HD>(qx[u], qt, a.eps, a.rot, s_rot + hh * HD);
        if (lane < HeadVec<HD>::LANES) {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const int i = lane * EPL + e;
                s_q[((i / (4 * KW)) * kWave + ((i / KW) & 3) * 16 + hh) * KW + i % KW] = hh < G ? qx[u].v[e] : 0.f;
            }
        }
    }
    lds_barrier();
    float qf[J][KW];
#pragma unroll
    for (int j = 0; j < J; ++j) load_floats<KW>(qf[j], &s_q[((wave * J + j) * kWave + lane) * KW]);

    float m = -INFINITY, l = 0.f;  // of head r (m the same in its four q lanes, l this lane's share)
    f32x4_t acc[VW];
#pragma unroll
    for (int e = 0; e < VW; ++e) acc[e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int par = 0;
    for (int t0 = p0; t0 < p1; t0 += STEP, par ^= 1) {
        const int pn = a.position - t0;  // the new row within the step, if 0 <= pn < STEP
        if (pn < STEP) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                if (16 * t + r == pn) {
#pragma unroll
                    for (int j = 0; j < J; ++j) load_floats<KW>(kr[t][j], &s_new[wave * DW + 4 * KW * j + KW * q]);
                }
        }
        f32x4_t sc[TILES], sc2[TILES];  // two chains per tile
#pragma unroll
        for (int t = 0; t < TILES; ++t) sc[t] = sc2[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int e = 0; e < KW; ++e)
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    f32x4_t &c = (e & 1) ? sc2[t] : sc[t];
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[t][j][e], qf[j][e], c, 0, 0, 0);
                }
#pragma unroll
        for (int t = 0; t < TILES; ++t) s_s[par][wave][t][lane] = sc[t] + sc2[t];
        if (t0 + STEP < p1) load_k(t0 + STEP);
        lds_barrier();
        float p[TILES][4], mt = -INFINITY;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const f32x4_t x = (s_s[par][0][t][lane] + s_s[par][1][t][lane]) + (s_s[par][2][t][lane] + s_s[par][3][t][lane]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[t][i] = t0 + 16 * t + 4 * q + i < p1 ? x[i] * a.scale : -INFINITY;
                mt = fmaxf(mt, p[t][i]);
            }
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16, kWave));
        mt = fmaxf(mt, __shfl_xor(mt, 32, kWave));
        const float mn = fmaxf(m, mt);
        const float ref = finite_max(mn);
        const float alpha = expf(m - ref);  // 0 for the first step
        m = mn;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[t][i] = expf(p[t][i] - ref);
                l += p[t][i];
            }
        if (t0 + STEP > p1 - (a.position < p1)) {
            // rows past the end count nothing, whatever they hold; the new row is the projection's
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int at = 16 * t + 4 * q + i;
                    if (t0 + at >= p1) {
#pragma unroll
                        for (int e = 0; e < VW; ++e) vr[t][i][e] = 0.f;
                    } else if (at == pn) {
#pragma unroll
                        for (int e = 0; e < VW; ++e) vr[t][i][e] = a.v_proj[g * HD + wave * DW + min(VW * r, DW - VW) + e];
                    }
                }
        }
        // each tile's positions by themselves, then one sum with the earlier steps': a chain over
        // all of a split's positions would round at every one of them (error against 64 bits at
        // 33,001 positions: 8 kv heads of 128, 516 positions a split, 4.3e-7 as one chain, 1.8e-7
        // so; 2 of 256, 129 a split, 2.6e-7 and 1.8e-7; same times)
        f32x4_t add[TILES][VW];
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int e = 0; e < VW; ++e) add[t][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int e = 0; e < VW; ++e)
                    add[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[t][i], vr[t][i][e], add[t][e], 0, 0, 0);
        if constexpr (TILES == 1) {  // a split of one tile is one step
#pragma unroll
            for (int e = 0; e < VW; ++e) acc[e] = add[0][e];
        } else {
            f32x4_t f;
#pragma unroll
            for (int i = 0; i < 4; ++i) f[i] = __shfl(alpha, 4 * q + i, kWave);
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const f32x4_t both = add[0][e] + add[TILES - 1][e];
                acc[e] = t0 == p0 ? both : acc[e] * f + both;
            }
        }
        if (t0 + STEP < p1) load_v(t0 + STEP);
    }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    if (VW * r < DW) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (4 * q + i < G) {
                float *dst = a.part + (static_cast<int64_t>(g * G + 4 * q + i) * a.splits + split) * HD + wave * DW + VW * r;
#pragma unroll
                for (int e = 0; e < VW; ++e) dst[e] = acc[e][i];
            }
        }
    }
    if (tid < G) {  // wave 0, lane (h, 0)
        float *dst = a.part_ml + (static_cast<int64_t>(g * G + tid) * a.splits + split) * 2;
        dst[0] = m;
        dst[1] = l;
    }
}

// The splits merged: one workgroup of 512 threads per (query head, 64 dims).
// M = max m_s and L = sum exp(m_s - M) l_s over the threads (a split each),
// the weights exp(m_s - M) to LDS; 16 lanes read a split's 64 dims, so a wave
// takes four splits and the workgroup 32 per round, the first rounds' loads
// issued before the weights are known; the sums meet over the lanes and in
// LDS; out = sum / L * sigmoid(gate).  Bound: launch and two round trips, 3.9
// us at 256 splits (one workgroup per head took 5.2 us at 64 splits, 22 at 516).
constexpr int kCombineThreads = 512;
constexpr int kCombineWaves = kCombineThreads / kWave;
static_assert(kAttnMaxSplits <= kCombineThreads, "a thread per split");

template <int HD>
__global__ __launch_bounds__(kCombineThreads) void attn_combine(const AttnArgs a) {
    constexpr int DB = HD < 64 ? HD : 64;           // dims per workgroup
    constexpr int LPS = DB / 4;                     // lanes per split (4 dims each)
    constexpr int SPR = kCombineThreads / LPS;      // splits per round
    constexpr int U = 8;                            // rounds in flight
    __shared__ float s_w[kAttnMaxSplits];
    __shared__ float s_red[2][kCombineWaves];
    __shared__ float s_acc[kCombineWaves][DB];
    const int h = blockIdx.x, d0 = blockIdx.y * DB, tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid & (kWave - 1);
    const float *ml = a.part_ml + static_cast<int64_t>(h) * a.splits * 2;
    const float *src = a.part + static_cast<int64_t>(h) * a.splits * HD + d0 + (tid % LPS) * 4;
    const int s0 = tid / LPS;
    const bool mine = tid < a.splits;
    const float ms = mine ? ml[2 * tid] : -INFINITY;
    const float ls = mine ? ml[2 * tid + 1] : 0.f;
    const float gate = a.q_proj[static_cast<int64_t>(h) * 2 * HD + HD + d0 + tid % DB];
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
        v[u] = *reinterpret_cast<const float4 *>(src + static_cast<int64_t>(min(s0 + u * SPR, a.splits - 1)) * HD);
    float M = wave_max_all(ms);
    if (lane == 0) s_red[0][wave] = M;
    lds_barrier();
#pragma unroll
    for (int w = 0; w < kCombineWaves; ++w) M = fmaxf(M, s_red[0][w]);
    const float wt = mine ? expf(ms - finite_max(M)) : 0.f;
    if (tid < a.splits) s_w[tid] = wt;
    const float lw = wave_sum_all(wt * ls);
    if (lane == 0) s_red[1][wave] = lw;
    lds_barrier();
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int base = 0; base < a.splits; base += U * SPR) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = base + s0 + u * SPR;
            if (s < a.splits) {
                const float w = s_w[s];
                acc[0] += w * v[u].x;
                acc[1] += w * v[u].y;
                acc[2] += w * v[u].z;
                acc[3] += w * v[u].w;
            }
        }
        if (base + U * SPR < a.splits) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                v[u] = *reinterpret_cast<const float4 *>(
                    src + static_cast<int64_t>(min(base + (U + u) * SPR + s0, a.splits - 1)) * HD);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        for (int off = LPS; off < kWave; off <<= 1) acc[e] += __shfl_xor(acc[e], off, kWave);
    }
    if (lane < LPS) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s_acc[wave][lane * 4 + e] = acc[e];
    }
    lds_barrier();
    if (tid < DB) {
        float L = 0.f, t = 0.f;
#pragma unroll
        for (int w = 0; w < kCombineWaves; ++w) L += s_red[1][w];
#pragma unroll
        for (int w = 0; w < kCombineWaves; ++w) t += s_acc[w][tid];
        a.out[h * HD + d0 + tid] = (t / L) * sigmoid_acc(gate);
    }
}

inline size_t align256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

int check_layer(const swq_attention_layer *l) {
    if (!l || l->reserved != 0) return SWQ_ERR_INVALID_ARGUMENT;
    if (l->num_heads <= 0 || l->num_kv_heads <= 0 || l->num_heads % l->num_kv_heads != 0) return SWQ_ERR_BAD_SHAPE;
    if (l->num_heads / l->num_kv_heads > kAttnMaxGroup) return SWQ_ERR_LIMIT;
    const int hd = l->head_dim;
    if (hd != 16 && hd != 32 && hd != 64 && hd != 128 && hd != 256) return SWQ_ERR_LIMIT;
    if (l->rotary_dims < 0 || l->rotary_dims > hd || l->rotary_dims % 2 != 0) return SWQ_ERR_BAD_SHAPE;
    if (l->max_positions <= 0) return SWQ_ERR_INVALID_ARGUMENT;
    if (!(l->rope_theta > 0.f) || !(l->norm_eps >= 0.f)) return SWQ_ERR_INVALID_ARGUMENT;
    if (!l->q_norm_weight || !l->k_norm_weight) return SWQ_ERR_INVALID_ARGUMENT;
    return SWQ_OK;
}

size_t half_cache(const swq_attention_layer *l) {
    return align256(static_cast<size_t>(l->max_positions) * l->num_kv_heads * l->head_dim * sizeof(float));
}

// The split of n positions over workgroups: one 16-position tile a workgroup while that takes
// no more than two workgroups per CU over all kv heads (a CU's loads come in at about 32 KB per
// round trip, so a short context is fastest spread thin), else that many workgroups, each
// walking its positions two tiles a step.  Step + merge at 33,001 positions and 2 kv heads:
// 256 workgroups 42.7 us, 512 38.5, 1,024 41.0; at 4,096 13.5, 13.7, 13.6; at 1,000 the
// 64-position workgroups of four waves took 15.0, one tile each 10.2.  Past a whole step the last
// one is mostly padding, which costs up to a fifth: at 2 kv heads 4,096 / 4,097 positions 11.8 /
// 13.4 us, 8,192 / 8,193 14.5 / 17.2, 16,384 / 16,385 19.4 / 22.8, 32,768 / 33,001 32.4 / 38.3
// (64-position chunks: 18.5 / 17.9, 23.0 / 30.6, 40.4 / 46.3, 74.4 / 81.5).
struct AttnPlan {
    int per, splits, tiles;
};

int64_t split_cap(int kvh) { return std::min(kAttnMaxSplits, std::max(1, kAttnTargetWgs / kvh)); }

AttnPlan plan_splits(int64_t n, int kvh) {
    const int64_t cap = split_cap(kvh), per = std::max<int64_t>((n + cap - 1) / cap, 16);
    return {static_cast<int>(per), static_cast<int>((n + per - 1) / per), per <= 16 ? 1 : 2};
}

// Most splits of any length up to n.
int64_t most_splits(int64_t n, int kvh) { return std::min<int64_t>((n + 15) / 16, split_cap(kvh)); }

template <int HD>
void launch(const AttnArgs &a, int tiles, hipStream_t s) {
    const dim3 grid(a.splits, a.KVH), block(kAttnThreads);
    if (tiles == 1) hipLaunchKernelGGL((attn_partial<HD, 1>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((attn_partial<HD, 2>), grid, block, 0, s, a);
    hipLaunchKernelGGL(attn_combine<HD>, dim3(a.H, HD < 64 ? 1 : HD / 64), dim3(kCombineThreads), 0, s, a);
}

}  // namespace
}  // namespace swq

using namespace swq;

extern "C" size_t swq_attention_cache_bytes(const swq_attention_layer *l) {
    return check_layer(l) == SWQ_OK ? 2 * half_cache(l) : 0;
}

extern "C" size_t swq_attention_workspace_bytes(const swq_attention_layer *l) {
    if (check_layer(l) != SWQ_OK) return 0;
    const size_t splits = most_splits(l->max_positions, l->num_kv_heads);
    return static_cast<size_t>(l->num_heads) * splits * (l->head_dim + 2) * sizeof(float);
}

static int check_step(const swq_attention_layer *l, const float *q_proj, const float *k_proj, const float *v_proj,
                      const void *cache, size_t cache_bytes, int64_t position, const float *out, const void *ws,
                      size_t ws_bytes) {
    const int st = check_layer(l);
    if (st != SWQ_OK) return st;
    if (!q_proj || !k_proj || !v_proj || !cache || !out || position < 0) return SWQ_ERR_INVALID_ARGUMENT;
    if (position >= l->max_positions) return SWQ_ERR_LIMIT;
    if (cache_bytes < swq_attention_cache_bytes(l)) return SWQ_ERR_WORKSPACE;
    if (!ws || ws_bytes < swq_attention_workspace_bytes(l)) return SWQ_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(cache) % 256 != 0 || reinterpret_cast<uintptr_t>(ws) % 256 != 0)
        return SWQ_ERR_MISALIGNED;
    return SWQ_OK;
}

extern "C" int swq_attention_step(const swq_attention_layer *l, const float *q_proj, const float *k_proj,
                                  const float *v_proj, void *cache, size_t cache_bytes, int64_t position,
                                  float *out, void *ws, size_t ws_bytes, void *stream) {
    const int st = check_step(l, q_proj, k_proj, v_proj, cache, cache_bytes, position, out, ws, ws_bytes);
    if (st != SWQ_OK) return st;
    AttnArgs a{};
    a.q_proj = q_proj;
    a.k_proj = k_proj;
    a.v_proj = v_proj;
    a.q_norm_w = l->q_norm_weight;
    a.k_norm_w = l->k_norm_weight;
    a.cache_k = static_cast<float *>(cache);
    a.cache_v = reinterpret_cast<float *>(static_cast<uint8_t *>(cache) + half_cache(l));
    a.part = static_cast<float *>(ws);
    a.out = out;
    a.H = l->num_heads;
    a.KVH = l->num_kv_heads;
    a.hd = l->head_dim;
    a.rot = l->rotary_dims;
    a.group = a.H / a.KVH;
    a.position = static_cast<int32_t>(position);
    const AttnPlan plan = plan_splits(position + 1, a.KVH);
    a.per = plan.per;
    a.splits = plan.splits;
    a.part_ml = a.part + static_cast<int64_t>(a.H) * a.splits * a.hd;
    a.theta = l->rope_theta;
    a.eps = l->norm_eps;
    // the rotation table: powf / cosf / sinf of the reference's float
    // operands (applyRope, QwenCPUModel.swift:356-358), evaluated in double and
    // rounded once, as a correctly rounded float libm returns them
    for (int j = 0; j < a.rot / 2; ++j) {
        const float ex = -static_cast<float>(2 * j) / static_cast<float>(a.rot);
        const float inv_freq = static_cast<float>(std::pow(static_cast<double>(a.theta), static_cast<double>(ex)));
        const float ang = static_cast<float>(a.position) * inv_freq;
        a.rope_cos[j] = static_cast<float>(std::cos(static_cast<double>(ang)));
        a.rope_sin[j] = static_cast<float>(std::sin(static_cast<double>(ang)));
    }
    a.scale = 1.0f / std::sqrt(static_cast<float>(a.hd));
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (a.hd) {
        case 16: launch<16>(a, plan.tiles, s); break;
        case 32: launch<32>(a, plan.tiles, s); break;
        case 64: launch<64>(a, plan.tiles, s); break;
        case 128: launch<128>(a, plan.tiles, s); break;
        default: launch<256>(a, plan.tiles, s); break;
    }
    return launch_status();
}

// The block's four launches from one entry, as swq_deltanet_token.
extern "C" size_t swq_attention_scratch_floats(const swq_attention_layer *l, const swq_qlinear *projections) {
    if (check_layer(l) != SWQ_OK || !projections) return 0;
    int64_t n = 1LL * l->num_heads * l->head_dim;
    for (int i = 0; i < 3; ++i) n += pad_floats(std::max(projections[i].out_dim, 0));
    return static_cast<size_t>(n);
}

extern "C" int swq_attention_token(const swq_attention_layer *l, const swq_qlinear *projections,
                                   const swq_qlinear *o_proj, const float *x, const void *norm_weight, int norm_dtype,
                                   float norm_eps, void *cache, size_t cache_bytes, int64_t position, float *scratch,
                                   size_t scratch_floats, float *out, void *ws, size_t ws_bytes, void *stream) {
    int st = check_layer(l);
    if (st != SWQ_OK) return st;
    if (!projections || !o_proj || !scratch || !out) return SWQ_ERR_INVALID_ARGUMENT;
    const int64_t val = 1LL * l->num_heads * l->head_dim, kv = 1LL * l->num_kv_heads * l->head_dim;
    if (projections[0].out_dim < 2 * val || projections[1].out_dim < kv || projections[2].out_dim < kv ||
        o_proj->in_dim > val)
        return SWQ_ERR_BAD_SHAPE;
    if (scratch_floats < swq_attention_scratch_floats(l, projections)) return SWQ_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(scratch) % 16 != 0) return SWQ_ERR_MISALIGNED;
    float *q = scratch, *k = q + pad_floats(projections[0].out_dim), *v = k + pad_floats(projections[1].out_dim);
    float *y = v + pad_floats(projections[2].out_dim);
    float *ys[3] = {q, k, v};
    // every check before the first launch: an error leaves the cache as it was
    st = check_gemv_multi(projections, 3, ys, x, norm_weight, norm_dtype, norm_eps);
    if (st == SWQ_OK) st = check_step(l, q, k, v, cache, cache_bytes, position, y, ws, ws_bytes);
    if (st == SWQ_OK) st = check_gemv(o_proj, y, out);
    if (st != SWQ_OK) return st;
    st = swq_encode_gemv_multi(projections, 3, ys, x, norm_weight, norm_dtype, norm_eps, stream);
    if (st == SWQ_OK) st = swq_attention_step(l, q, k, v, cache, cache_bytes, position, y, ws, ws_bytes, stream);
    if (st == SWQ_OK) st = swq_encode_gemv(o_proj, 0, 0, 0, 0, y, 0, out, 0, stream);
    return st;
}
