// The attention half of a decoder block around the TR-MoE layer: grouped-query
// attention with per-head RMSNorm on q and k and rotary embeddings
// (complexity/core/attention/gqa.py:88-165, rotary.py:17-80) over a static
// key/value cache.  Heads are 64 wide, bf16.
//
//   k_qk_rope     a prompt's fused k|q|v projection rows -> q (normed, rotated)
//                 in [token, head, 64], k and v into the caches
//   k_prefill_attn  causal attention of a prompt over its keys and values in the
//                 caches (flash form: running maximum and sum)
//   k_decode_qkv  one token per sequence, up to 16 sequences: RMSNorm of the
//                 hidden row and the k|q|v projection in one launch
//   k_decode_attn that token's q and k norm and rotation, the cache write and
//                 attention over the cache split along the positions; the last
//                 workgroup of a (sequence, kv head) merges the splits
//
// These replace chains of elementwise passes (a norm is 5 launches, a rotation
// 5, the cache writes 2, the key/value repeat 2): at a prompt of 8 x 2048 they
// took 7.0 of the 17.2 ms, and a decode step of one sequence was 470 launches.
#include "trmoe_attn.h"

#include "trmoe_common.h"
#include "trmoe_internal.h"
#include "trmoe_skinny.h"

#include <algorithm>

namespace trmoe {

namespace {

constexpr int kD = 64;        // head width
constexpr int kLanes = 8;     // lanes of a head row, 8 elements each

__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = __builtin_bit_cast(float, (uint32_t)v[j] << 16);
        f[2 * j + 1] = __builtin_bit_cast(float, (uint32_t)v[j] & 0xffff0000u);
    }
}
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
    bf16x8 r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = (bf16_t)f[j];
    return __builtin_bit_cast(u32x4, r);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kQuadXor3 = 0x1B, kHalfMirror = 0x141, kRor8 = 0x128;
// Over the 8 lanes of a head row, on the vector ALU alone (the mirror reaches
// the other quad, whose lanes all hold its sum).
__device__ __forceinline__ float sum8(float s) {
    s += dpp<kQuadXor1>(s);
    s += dpp<kQuadXor2>(s);
    s += dpp<kHalfMirror>(s);
    return s;
}
// The value of the lane 4 away in its 8: i ^ 7, then ^ 3.
__device__ __forceinline__ float xor4(float v) { return dpp<kQuadXor3>(dpp<kHalfMirror>(v)); }

// x (the lane's 8 of a head row's 64 elements) -> rope(rmsnorm(x) * w) at one
// position: element d pairs with d +- 32, which the lane 4 away holds.
__device__ __forceinline__ void norm_rope(float (&x)[8], const bf16_t* w, float eps, const float* cos,
                                          const float* sin, int c) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s += x[j] * x[j];
    const float r = rsqrtf(sum8(s) * (1.0f / kD) + eps);
    float wf[8];
    unpack8(*reinterpret_cast<const u32x4*>(w + 8 * c), wf);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = x[j] * r * wf[j];
    const float sign = c < 4 ? -1.0f : 1.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float other = xor4(x[j]);
        x[j] = x[j] * cos[8 * c + j] + sign * other * sin[8 * c + j];
    }
}

// One head row (of k, q or v) per 8 lanes.  Memory-bound: each projection row
// is read once and written once, 16 bytes per lane.
__global__ __launch_bounds__(256) void k_qk_rope(RopeArgs a) {
    const int slots = a.heads + 2 * a.kvh;
    const int64_t item = ((int64_t)blockIdx.x * 256 + threadIdx.x) / kLanes;
    if (item >= a.rows * slots) return;   // whole 8-lane groups leave together
    const int c = threadIdx.x & 7;
    const int64_t row = item / slots;
    const int slot = (int)(item - row * slots);
    const int64_t b = row / a.T, t = row - b * a.T;
    int64_t pos = a.pos0 + t;
    if (a.pos != nullptr) pos += *a.pos;
    if (pos < 0 || pos >= a.L) return;    // a position past the cache is dropped
    const u32x4 in = *reinterpret_cast<const u32x4*>(a.kqv + row * a.ldkqv + slot * kD + 8 * c);
    const int vslot = a.heads + a.kvh;
    if (slot >= vslot) {
        *reinterpret_cast<u32x4*>(a.v + ((b * a.kvh + slot - vslot) * a.L + pos) * kD + 8 * c) = in;
        return;
    }
    float x[8];
    unpack8(in, x);
    const bool is_k = slot < a.kvh;
    norm_rope(x, is_k ? a.kw : a.qw, a.eps, a.cos + pos * kD, a.sin + pos * kD, c);
    bf16_t* dst = is_k ? a.k + ((b * a.kvh + slot) * a.L + pos) * kD
                       : a.q + (row * a.heads + slot - a.kvh) * kD;
    *reinterpret_cast<u32x4*>(dst + 8 * c) = pack8(x);
}

// qkv[m][n] (fp32) = rmsnorm(x_m) . W_n for up to 16 rows: 16 output columns
// per workgroup, the 8 waves split K (groups of 32), one 16x16x32 MFMA each.
// The norm weight goes onto x before the product, the row's 1/rms onto the
// sum after it.  Latency-bound (28 KB of weights per workgroup): every load of
// a wave's first 4 groups is issued before any is used.
constexpr int kQkvWaves = 8, kQkvBatch = 4;
__global__ __launch_bounds__(64 * kQkvWaves) void k_decode_qkv(DecodeAttnArgs a) {
    __shared__ float red[kQkvWaves][4][64];
    __shared__ float s_ssq[kQkvWaves][16];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int n0 = (int)blockIdx.x * 16;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < a.B * a.kvh; i += 64 * kQkvWaves) a.counters[i] = 0;
    const int groups = a.H / 32, per = (groups + kQkvWaves - 1) / kQkvWaves;
    const int g0 = wave * per, g1 = std::min(g0 + per, groups);
    const bf16_t* xr = a.x + (int64_t)(r < a.B ? r : 0) * a.ldx + 8 * q;
    const bf16_t* wr = a.w_kqv + (int64_t)(n0 + r) * a.H + 8 * q;
    const bf16_t* nr = a.norm_w + 8 * q;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float ssq = 0.f;
    for (int gb = g0; gb < g1; gb += kQkvBatch) {
        u32x4 xv[kQkvBatch], wv[kQkvBatch], nv[kQkvBatch];
#pragma unroll
        for (int j = 0; j < kQkvBatch; ++j) {
            const u32x4 zero = {0u, 0u, 0u, 0u};
            const bool in = gb + j < g1;
            wv[j] = in ? *reinterpret_cast<const u32x4*>(wr + 32 * (gb + j)) : zero;
            xv[j] = in && r < a.B ? *reinterpret_cast<const u32x4*>(xr + 32 * (gb + j)) : zero;
            nv[j] = in ? *reinterpret_cast<const u32x4*>(nr + 32 * (gb + j)) : zero;
        }
#pragma unroll
        for (int j = 0; j < kQkvBatch; ++j) {
            float xf[8], nf[8];
            unpack8(xv[j], xf);
            unpack8(nv[j], nf);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                ssq += xf[e] * xf[e];
                xf[e] *= nf[e];
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pack8(xf)),
                                                          __builtin_bit_cast(bf16x8, (u32x4)wv[j]), acc, 0, 0, 0);
        }
    }
    ssq += __shfl_xor(ssq, 16);
    ssq += __shfl_xor(ssq, 32);
    if (q == 0) s_ssq[wave][r] = ssq;
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][i][lane] = acc[i];
    __syncthreads();
    if (threadIdx.x < 256) {
        const int i = threadIdx.x >> 6, m = 4 * q + i;
        if (m < a.B) {
            float s = 0.f, ss = 0.f;
#pragma unroll
            for (int w = 0; w < kQkvWaves; ++w) {
                s += red[w][i][lane];
                ss += s_ssq[w][m];
            }
            a.qkv[(int64_t)m * a.n_qkv + n0 + r] = s * rsqrtf(ss / (float)a.H + a.norm_eps);
        }
    }
}

// Attention of one new token: workgroup (split, kv head, sequence) takes the
// cache positions [split * chunk, + chunk) below the current one; the split
// that holds the current position normalises, rotates and stores its k and v
// and adds it.  Eight lanes hold one position's 64 elements, so each K and V
// row is one 128-byte read, with a running maximum and sum per query head.
// The G heads of the group are spread over the waves (HPW each), so that a
// wave normalises and merges only its own; with few heads several waves share
// them and split the positions (PW).  A step of one sequence has little
// else to hide latency behind: the first K/V rows are requested before the
// position is known, and reductions stay on the vector ALU.  Against all heads
// in every wave and one 128-position split: 14.2 us at 213 positions before.
// 16 waves and 256 positions a workgroup, against 4 waves and 64 positions: a
// quarter of the partials to merge, which pays in long caches and costs in
// short ones.  us, 14 heads on 2, 4 waves -> 16: one
// sequence at position 213 of a cache of 256 9.2 -> 10.2, of 1024 10.3 -> 13.0, at
// 1500 of 4096 17.9 -> 13.7, at 4000 of 4096 18.5 -> 13.3; 8 at 2100 of 2176 16.6 ->
// 14.1; 16 at 4000 of 4096 24.0 -> 19.7.
constexpr int kAttnWaves = 16;
constexpr int kUnroll = 4;
constexpr int kMaxSplits = 64;
constexpr int kPart = kD + 2;   // 64 sums, the maximum, the weight
template <int G>
struct HeadSplit {
    static constexpr int HW = G >= 4 ? 4 : G;          // waves over heads
    static constexpr int PW = kAttnWaves / HW;         // waves over positions
    static constexpr int HPW = (G + HW - 1) / HW;      // heads per wave
};

template <int G>
__global__ __launch_bounds__(64 * kAttnWaves) void k_decode_attn(DecodeAttnArgs a, int chunk, int splits) {
    using HS = HeadSplit<G>;
    constexpr int HPW = HS::HPW, PW = HS::PW;
    __shared__ float s_ml[PW][G][2];
    __shared__ float s_acc[PW][G][kD];
    __shared__ float s_f[G][kMaxSplits + 1];
    const int split = (int)blockIdx.x, kvh = (int)blockIdx.y, b = (int)blockIdx.z;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int hw = wave / PW, pw = wave % PW;
    const int c = lane & 7, grp = pw * 8 + (lane >> 3);
    constexpr int kStep = 8 * PW;
    const int p0 = split * chunk;
    const int64_t head_off = ((int64_t)b * a.kvh + kvh) * a.L * kD;
    const bf16_t* kc = a.k_cache + head_off + 8 * c;
    const bf16_t* vc = a.v_cache + head_off + 8 * c;
    u32x4 kv[kUnroll], vv[kUnroll];
    auto load = [&](int p) {   // rows at or past the current position are read (inside the cache) and not used
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int64_t pp = std::min<int64_t>(p + kStep * u, a.L - 1);
            kv[u] = *reinterpret_cast<const u32x4*>(kc + pp * kD);
            vv[u] = *reinterpret_cast<const u32x4*>(vc + pp * kD);
        }
    };
    load(p0 + grp);
    int64_t pos64 = *a.pos;
    pos64 = pos64 < 0 ? 0 : (pos64 >= a.L ? a.L - 1 : pos64);
    const int pos = (int)pos64;
    const int p1 = std::min(p0 + chunk, pos);
    const bool own = pos >= p0 && pos < p0 + chunk;
    const float* row = a.qkv + (int64_t)b * a.n_qkv;
    const float* cosp = a.cos + (int64_t)pos * kD;
    const float* sinp = a.sin + (int64_t)pos * kD;

    float q[HPW][8], m[HPW], l[HPW], acc[HPW][8];
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
        const int g = std::min(hw * HPW + i, G - 1);   // the last wave may repeat a head and drop it
        const float* src = row + (a.kvh + kvh * G + g) * kD + 8 * c;
#pragma unroll
        for (int j = 0; j < 8; ++j) q[i][j] = src[j];
        norm_rope(q[i], a.qn_w, a.qk_eps, cosp, sinp, c);
        m[i] = -1e30f;
        l[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            q[i][j] *= a.scale * 1.4426950408889634f;   // exp2 below
            acc[i][j] = 0.f;
        }
    }
    auto attend = [&](const float (&kf)[8], const float (&vf)[8]) {
#pragma unroll
        for (int i = 0; i < HPW; ++i) {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) s += q[i][j] * kf[j];
            s = sum8(s);
            const float mn = fmaxf(m[i], s);
            const float f = __builtin_amdgcn_exp2f(m[i] - mn), p = __builtin_amdgcn_exp2f(s - mn);
            m[i] = mn;
            l[i] = l[i] * f + p;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = acc[i][j] * f + p * vf[j];
        }
    };
    for (int p = p0 + grp;;) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (p + kStep * u < p1) {   // uniform over the position's 8 lanes
                float kf[8], vf[8];
                unpack8(kv[u], kf);
                unpack8(vv[u], vf);
                attend(kf, vf);
            }
        }
        p += kStep * kUnroll;
        if (p >= p1) break;
        load(p);
    }
    if (own && pw == 0 && lane < kLanes) {
        float kf[8], vf[8];
        const float* ks = row + kvh * kD + 8 * c;
        const float* vs = row + (a.kvh + a.kvh * G + kvh) * kD + 8 * c;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            kf[j] = ks[j];
            vf[j] = vs[j];
        }
        norm_rope(kf, a.kn_w, a.qk_eps, cosp, sinp, c);
        const u32x4 kb = pack8(kf), vb = pack8(vf);
        if (hw == 0) {
            *reinterpret_cast<u32x4*>(a.k_cache + head_off + (int64_t)pos * kD + 8 * c) = kb;
            *reinterpret_cast<u32x4*>(a.v_cache + head_off + (int64_t)pos * kD + 8 * c) = vb;
        }
        unpack8(kb, kf);   // what later steps will read
        unpack8(vb, vf);
        attend(kf, vf);
    }
    // merge the wave's 8 positions
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
        auto merge = [&](auto other) {
            const float mo = other(m[i]), lo = other(l[i]);
            const float mn = fmaxf(m[i], mo);
            const float f = __builtin_amdgcn_exp2f(m[i] - mn), fo = __builtin_amdgcn_exp2f(mo - mn);
            m[i] = mn;
            l[i] = l[i] * f + lo * fo;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = acc[i][j] * f + other(acc[i][j]) * fo;
        };
        merge([](float v) { return dpp<kRor8>(v); });
        merge([](float v) { return __shfl_xor(v, 16); });
        merge([](float v) { return __shfl_xor(v, 32); });
        const int g = hw * HPW + i;
        if (lane < kLanes && g < G) {
#pragma unroll
            for (int j = 0; j < 8; ++j) s_acc[pw][g][8 * c + j] = acc[i][j];
            if (c == 0) {
                s_ml[pw][g][0] = m[i];
                s_ml[pw][g][1] = l[i];
            }
        }
    }
    __syncthreads();
    bf16_t* out = a.attn + (int64_t)b * (a.kvh * G * kD) + kvh * G * kD;
    float* part = a.part + ((int64_t)(b * a.kvh + kvh) * splits) * (G * kPart);
    for (int i = threadIdx.x; i < G * kD; i += 64 * kAttnWaves) {
        const int g = i / kD, d = i % kD;
        float mn = s_ml[0][g][0];
#pragma unroll
        for (int w = 1; w < PW; ++w) mn = fmaxf(mn, s_ml[w][g][0]);
        float lt = 0.f, v = 0.f;
#pragma unroll
        for (int w = 0; w < PW; ++w) {
            const float f = __builtin_amdgcn_exp2f(s_ml[w][g][0] - mn);
            lt += s_ml[w][g][1] * f;
            v += s_acc[w][g][d] * f;
        }
        if (splits == 1) {
            out[i] = (bf16_t)(v / lt);
        } else {
            float* dst = part + ((int64_t)split * G + g) * kPart;
            store_dev(dst + d, v);
            if (d == 0) {
                store_dev(dst + kD, mn);
                store_dev(dst + kD + 1, lt);
            }
        }
    }
    if (splits == 1) return;
    if (!last_arrival(a.counters + b * a.kvh + kvh, splits)) return;
    // the splits' factors, one lane per split, then the weighted sums
    for (int g = wave; g < G; g += kAttnWaves) {
        const float* src = part + ((int64_t)lane * G + g) * kPart + kD;
        const float ms = lane < splits ? load_dev(src) : -1e30f, ls = lane < splits ? load_dev(src + 1) : 0.f;
        float mx = ms;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
        const float f = __builtin_amdgcn_exp2f(ms - mx);
        float lt = ls * f;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) lt += __shfl_xor(lt, off);
        s_f[g][lane] = f / lt;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < G * kD; i += 64 * kAttnWaves) {
        const int g = i / kD, d = i % kD;
        const float* src = part + (int64_t)g * kPart + d;
        float v = 0.f;
        for (int s = 0; s < splits; s += 8) {
            float t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) t[u] = load_dev(src + (int64_t)std::min(s + u, splits - 1) * (G * kPart));
#pragma unroll
            for (int u = 0; u < 8; ++u) v += s + u < splits ? t[u] * s_f[g][s + u] : 0.f;
        }
        out[i] = (bf16_t)v;
    }
}

// Causal attention of a prompt: a workgroup takes 128 queries of one head, 32
// per wave, and walks the 64-position K/V tiles up to them on a ring of LDS
// stages.  The products are transposed, S^T = K Q^T and O^T = V^T P^T, so that a
// lane owns one query: its scores lie in its own registers (one exchange with
// the lane 32 away for the maximum), the rescaling is a per-lane factor, and
// the scores' accumulator layout is the second product's operand as it stands
// (K order: positions 16 t + 4 h + 0..3 and + 8, which the transposing V reads
// follow).  The vector ALU bounds it (32 exponentials and about as much again
// per 512 clocks of MFMA); three workgroups per CU overlap one's softmax
// with another's products.  8 x 2048 tokens, 14 heads on 2: 92 us (174 us in
// the library's flash kernel).  What it took from 132: the longest rows first
// (25 us of a last wave that was nearly empty), masks on the diagonal tiles
// alone and the rescaling only where the maximum moved (6), constant offsets in
// the LDS reads (3) and two stages instead of three (6).
constexpr int kQTile = 128, kKTile = 64, kAttnStages = 2;
constexpr int kAttnStage = 2 * kKTile * kRowBytes;
__global__ __launch_bounds__(256, 2) void k_prefill_attn(PrefillAttnArgs a) {
    __shared__ __align__(16) char lds[kAttnStages * kAttnStage];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int r = lane & 31, h = lane >> 5;
    // the heads along x, the query tiles from the longest row to the shortest
    // along y: the short ones fill the gaps that the long ones leave
    const int qt = (int)(gridDim.y - 1 - blockIdx.y);
    const int b = (int)blockIdx.x / a.heads, head = (int)blockIdx.x % a.heads;
    const int kvh = head / (a.heads / a.kvh);
    const int T = (int)a.T;
    const int q0 = qt * kQTile, qw = q0 + 32 * wave;
    const int64_t kv_off = ((int64_t)b * a.kvh + kvh) * a.L * kD;
    const auto kr = make_rsrc(a.k + kv_off, (uint32_t)(T * kRowBytes));   // rows at or past T load zero
    const auto vr = make_rsrc(a.v + kv_off, (uint32_t)(T * kRowBytes));
    int off[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = (wave * 2 + j) * 8 + (lane >> 3);
        off[j] = row * kRowBytes + 16 * ((lane & 7) ^ (row & 7));
    }
    auto issue = [&](int tile, char* st) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            dma16(kr, st + (wave * 2 + j) * 8 * kRowBytes, off[j] + tile * kKTile * kRowBytes);
            dma16(vr, st + (kKTile + (wave * 2 + j) * 8) * kRowBytes, off[j] + tile * kKTile * kRowBytes);
        }
    };
    const int query = std::min(qw + r, T - 1);   // rows past the prompt repeat the last and are not stored
    const bf16_t* qrow = a.q + (((int64_t)b * T + query) * a.heads + head) * kD;
    u32x4 qf[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) qf[g] = *reinterpret_cast<const u32x4*>(qrow + 16 * g + 8 * h);
    const int nt = std::min((q0 + kQTile + kKTile - 1) / kKTile, (T + kKTile - 1) / kKTile);
#pragma unroll
    for (int s = 0; s < kAttnStages - 1; ++s) issue(s, lds + s * kAttnStage);

    f32x16 o[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
    float m = -__builtin_inff(), l = 0.f;
    const float c = a.scale * 1.4426950408889634f;   // exp2
    // transposing V reads: 16 lanes cover 4 positions x 16 columns
    const int vrow = 4 * h + ((lane & 15) >> 2), vchunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    // 16-byte chunks are swizzled by the row's low three bits alone, which rows
    // 8 apart share: every read of a tile is one of six addresses plus a constant
    int koff[4], voff[2];
#pragma unroll
    for (int g = 0; g < 4; ++g) koff[g] = r * kRowBytes + (((2 * g + h) ^ (r & 7)) << 4);
#pragma unroll
    for (int d = 0; d < 2; ++d)
        voff[d] = (kKTile + vrow) * kRowBytes + (((4 * d + vchunk) ^ vrow) << 4) + 8 * (lane & 1);
    f32x16 zero;   // the first product's C operand, instead of clearing 32 accumulators a tile
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.f;
    int cur = 0, nxt = kAttnStages - 1;
    // one K/V tile; DIAG: positions ahead of the query are masked (only the
    // tiles that reach the wave's first query hold any)
    auto step = [&](int kt, auto diag) {
        wait_vmcnt<4 * (kAttnStages - 2)>();   // this wave's loads of tile kt have landed
        wait_lgkmcnt0();                       // and its reads of tile kt - 1 are complete
        lds_barrier();                         // ... and every other wave's
        const char* ks = lds + cur * kAttnStage;
        issue(kt + kAttnStages - 1, lds + nxt * kAttnStage);
        cur = cur + 1 == kAttnStages ? 0 : cur + 1;
        nxt = nxt + 1 == kAttnStages ? 0 : nxt + 1;
        if (kt * kKTile > qw + 31) return;   // wholly ahead of the wave's queries
        f32x16 s[2];
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const u32x4 kf = *reinterpret_cast<const u32x4*>(ks + koff[g] + 32 * n * kRowBytes);
                s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf),
                                                               __builtin_bit_cast(bf16x8, (u32x4)qf[g]),
                                                               g == 0 ? zero : s[n], 0, 0, 0);
            }
        if constexpr (decltype(diag)::value) {
            const int ahead = qw + r - kt * kKTile;
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    s[n][i] = 32 * n + acc_row(lane, i) > ahead ? -__builtin_inff() : s[n][i];
        }
        float mx = m;
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[n][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // the reference point moves only when the maximum has grown by 2^8 (the
        // conditional rescaling published with FlashAttention-4): the weights
        // stay below that in fp32, and the sums need no rescaling
        if (__builtin_amdgcn_ballot_w64((mx - m) * c > 8.0f) != 0) {
            const float alpha = __builtin_amdgcn_exp2f((m - mx) * c);
            m = mx;
            l *= alpha;
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
        }
        const float mc = m * c;
        u32x4 p[4];
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                float e[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    e[i] = __builtin_amdgcn_exp2f(s[n][8 * t + i] * c - mc);
                    l += e[i];
                }
                p[2 * n + t] = pack8(e);
            }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                u32x2 v[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) v[e] = ds_read_tr16(ks + voff[d] + (16 * t + 8 * e) * kRowBytes);
                mfma_group(KindBF16{}, u32x4{v[0][0], v[0][1], v[1][0], v[1][1]}, p[t], o[d]);
            }
    };
    // tiles wholly at or before the workgroup's first query (uniform: the
    // waves share the barriers), then the diagonal ones
    const int full = std::min(nt, (q0 + 1) / kKTile);
    int kt = 0;
    for (; kt < full; ++kt) step(kt, std::false_type{});
    for (; kt < nt; ++kt) step(kt, std::true_type{});
    wait_vmcnt<0>();   // nothing writes this LDS once the workgroup has left
    if (qw + r >= T) return;
    const float inv = 1.0f / (l + __shfl_xor(l, 32));
    bf16_t* out = a.out + ((int64_t)b * T + qw + r) * (a.heads * kD) + head * kD;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
            bf16x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = (bf16_t)(o[d][4 * i + j] * inv);
            *reinterpret_cast<bf16x4*>(out + 32 * d + 8 * i + 4 * h) = v;
        }
}

}  // namespace

int launch_prefill_attn(const PrefillAttnArgs& a, int64_t sequences, hipStream_t stream) {
    const dim3 grid((unsigned)(sequences * a.heads), (unsigned)((a.T + kQTile - 1) / kQTile));
    hipLaunchKernelGGL(k_prefill_attn, grid, dim3(256), 0, stream, a);
    return check_launch("prefill_attention");
}

int launch_qk_rope(const RopeArgs& a, hipStream_t stream) {
    const int64_t lanes = a.rows * (a.heads + 2 * a.kvh) * kLanes;
    hipLaunchKernelGGL(k_qk_rope, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, stream, a);
    return check_launch("qk_norm_rope");
}

// Positions per split: at least 256 (a workgroup's first batch of loads or
// two), more when the (sequence, kv head) pairs fill the CUs or the splits would
// pass one lane each in the merge.
static int decode_chunk(int64_t L, int pairs) {
    int64_t splits = std::max(1, 256 / std::max(1, pairs));
    splits = std::min<int64_t>({splits, (L + 255) / 256, kMaxSplits});
    return (int)(((L + splits - 1) / splits + 31) / 32 * 32);
}

int64_t decode_attn_splits(int64_t L, int pairs) {
    const int chunk = decode_chunk(L, pairs);
    return (L + chunk - 1) / chunk;
}

int launch_decode_attn(const DecodeAttnArgs& a, int group, hipStream_t stream) {
    hipLaunchKernelGGL(k_decode_qkv, dim3((unsigned)(a.n_qkv / 16)), dim3(64 * kQkvWaves), 0, stream, a);
    int st = check_launch("decode_attention (qkv)");
    if (st) return st;
    const int chunk = decode_chunk(a.L, a.B * a.kvh);
    const int splits = (int)decode_attn_splits(a.L, a.B * a.kvh);
    const dim3 grid((unsigned)splits, (unsigned)a.kvh, (unsigned)a.B);
    auto kern = group == 1   ? k_decode_attn<1>
                : group == 2 ? k_decode_attn<2>
                : group == 4 ? k_decode_attn<4>
                : group == 7 ? k_decode_attn<7>
                : group == 8 ? k_decode_attn<8>
                             : nullptr;
    if (kern == nullptr) return set_error(TRMOE_ERR_UNSUPPORTED, "decode_attention: 1, 2, 4, 7 or 8 query heads per kv head");
    hipLaunchKernelGGL(kern, grid, dim3(64 * kAttnWaves), 0, stream, a, chunk, splits);
    return check_launch("decode_attention");
}

}  // namespace trmoe
