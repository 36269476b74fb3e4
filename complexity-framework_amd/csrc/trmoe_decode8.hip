// Decode (up to 128 tokens) of layers with e4m3 weights.
//
// The layer is weight-streaming: at the scaled shape (hidden 2048, shared
// 5632, 16 experts x 256) 60 MB of codes pass once per step.  The shared
// branch and every expert run as one gate|up launch and one split-K down over
// the concatenated features [shared | expert 0 | ...]: an expert's features
// carry the token's route weight (0 where the token is not routed to it), so
// there is no partition, no gather and no un-permute.  Below 16 assignments
// the experts no token reaches are skipped instead of streamed.
//
// Weights come fragment-major: the 16 rows x 64 K values of a block are 1 KiB
// whose lane l owns row l % 16, K values 16 (l / 16) .. + 15.  A lane's 16
// bytes feed two 16x16x32 MFMAs (values 0..7 and 8..15 of its run); the
// activation fragment of the second takes the following 16-byte chunk of x,
// so both operands see the same K order.
//
// Measured at 32 tokens of the scaled shape (two layers in a graph): the
// grouped prefill kernels on 64 assignments took 116 us per layer, 48 + 20 of
// them on 256-row tiles that were a quarter full; these take 36.
#include "trmoe_common.h"
#include "trmoe_gemm.h"
#include "trmoe_internal.h"
#include "trmoe_skinny.h"

#include <algorithm>

namespace trmoe {

namespace {

constexpr int kSpan = 64;        // K values per span: 128 bytes of activations, 1 KiB of weight block
constexpr int kWeightBatch = 4;  // spans whose weight loads are in flight together

// Staged spans per batch: two workgroups share a CU's 160 KiB of LDS, so
// that one's loads cover the other's reduction.
template <int MT, int NW>
constexpr int stage_batch() {
    constexpr int per = 73728 / (NW * MT * 16 * kRowBytes);
    return per < 1 ? 1 : (per > kWeightBatch ? kWeightBatch : per);
}

// Table entries outside [0, E) go to the nearest expert, as in the partition.
__device__ __forceinline__ int clamp_expert(int64_t e, int E) { return e < 0 ? 0 : (e >= E ? E - 1 : (int)e); }

// Experts that some token reaches, one bit each, for at most 16 assignments
// (every lane of the wave returns the same mask).
__device__ __forceinline__ uint32_t live_experts(const int64_t* ids, const int64_t* table, int64_t vocab, int M,
                                                 int top_k, int E) {
    const int lane = threadIdx.x & 63;
    uint32_t m = 0;
    if (lane < M * top_k) {
        int64_t id = ids[lane / top_k];
        id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
        m = 1u << clamp_expert(table[(int64_t)(lane % top_k) * vocab + id], E);
    }
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) m |= (uint32_t)__shfl_xor((int)m, off);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
}

// acc[tm][u] += x(rows tm*16..+15) . W(16-row block u)^T over spans [s0, s1):
// weight block u's span s is at byte (ublk[u] * G + s) * 1024 of wr; x goes
// through the wave's LDS region in batches of SB spans.  The weight loads of
// kWeightBatch spans are issued before the first wait.
template <int MT, int NU, int SB>
__device__ __forceinline__ void e4m3_spans(__amdgpu_buffer_rsrc_t ar, const int (&xo)[MT * 2], int kb_a, char* region,
                                           __amdgpu_buffer_rsrc_t wr, int G, int s0, int s1, f32x4 (&acc)[MT][NU]) {
    constexpr int kRows = MT * 16;
    const int lane = threadIdx.x & 63;
    const int q = lane >> 4;
    for (int wb = s0; wb < s1; wb += kWeightBatch) {
        u32x4 wv[kWeightBatch][NU];
#pragma unroll
        for (int j = 0; j < kWeightBatch; ++j)
#pragma unroll
            for (int u = 0; u < NU; ++u)
                wv[j][u] = buffer_load16(wr, wb + j < s1 ? (u * G + wb + j) * 1024 + 16 * lane : kOutOfRange);
#pragma unroll
        for (int sb = 0; sb < kWeightBatch; sb += SB) {
            if (wb + sb >= s1) break;
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                const int sp = wb + sb + j;
                if (sp < s1) {
                    char* st = region + j * kRows * kRowBytes;
#pragma unroll
                    for (int i = 0; i < MT * 2; ++i) {
                        const int o = 128 * sp + 16 * ((lane & 7) ^ lds_swz(i * 8 + (lane >> 3)));
                        dma16(ar, st + i * 8 * kRowBytes, o < kb_a ? xo[i] + 128 * sp : kOutOfRange);
                    }
                }
            }
            wait_vmcnt<0>();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                if (wb + sb + j < s1) {
                    const char* st = region + j * kRows * kRowBytes;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        u32x4 av[MT];
#pragma unroll
                        for (int tm = 0; tm < MT; ++tm)
                            av[tm] = *reinterpret_cast<const u32x4*>(st + lds_byte(tm * 16 + (lane & 15), 2 * q + h));
#pragma unroll
                        for (int u = 0; u < NU; ++u) {
                            const u32x4 b = fp8x8_to_bf16x8(u32x2{wv[sb + j][u][2 * h], wv[sb + j][u][2 * h + 1]});
#pragma unroll
                            for (int tm = 0; tm < MT; ++tm) mfma16(KindBF16{}, av[tm], b, acc[tm][u]);
                        }
                    }
                }
            }
            // the wave's reads of the batch are done before the next copies
            wait_lgkmcnt0();
            asm volatile("" ::: "memory");
        }
    }
}

template <int MT>
__device__ __forceinline__ void row_offsets(int (&xo)[MT * 2], int rows, int ld_bytes) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < MT * 2; ++j) {
        const int row = j * 8 + (lane >> 3);
        xo[j] = row < rows ? row * ld_bytes + 16 * ((lane & 7) ^ lds_swz(row)) : kOutOfRange;
    }
}

template <int MT, int NU, int NW>
constexpr int lds_bytes() {
    return std::max(NW * stage_batch<MT, NW>() * MT * 16 * kRowBytes, NW * MT * NU * 4 * 64 * 4);
}

// gate|up: one workgroup per 16 features (16 gate and 16 up rows), the waves
// split K.  Grid order: expert features first, whose route gather is a chain
// of two loads.
template <int MT, int NW>
__global__ __launch_bounds__(64 * NW) void k_gate_up_e4m3(GateUpArgs a, int shared_blocks) {
    constexpr int NT = 64 * NW;
    extern __shared__ __align__(16) char lds[];
    __shared__ int s_route[MT * 16][kMaxTopK];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int expert_blocks = (int)gridDim.x - shared_blocks;
    const int blk = (int)blockIdx.x < expert_blocks ? (int)blockIdx.x + shared_blocks
                                                    : (int)blockIdx.x - expert_blocks;
    const int64_t f0 = (int64_t)blk * 16;
    const int64_t pg = (f0 >> 5) * 64 + (f0 & 31);
    const bool routed = f0 >= a.shared_feats;
    const int64_t expert = routed ? (f0 - a.shared_feats) / a.expert_feats : -1;
    bf16_t* h = static_cast<bf16_t*>(a.h);
    if (routed && a.M * a.top_k <= 16) {
        if (!((live_experts(a.ids, a.table, a.vocab, (int)a.M, a.top_k, a.E) >> expert) & 1)) {
            for (int i = threadIdx.x; i < (int)a.M * 16; i += NT) h[(i >> 4) * a.ldh + f0 + (i & 15)] = (bf16_t)0.f;
            return;
        }
    }
    const int kb_a = a.K * 2;
    const int G = (a.K + kSpan - 1) / kSpan;
    const auto ar = make_rsrc(a.x, (uint32_t)(a.M * a.ldx * 2));
    // blocks pg / 16 (gate) and pg / 16 + 2 (up)
    const auto wr = make_rsrc(static_cast<const char*>(a.w_frag) + (pg >> 4) * (int64_t)G * 1024, (uint32_t)(3 * G * 1024));
    if (routed && threadIdx.x >= NT - MT * 16) {
        const int64_t row = threadIdx.x - (NT - MT * 16);
        int64_t id = row < a.M ? a.ids[row] : 0;
        id = id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id);
        for (int j = 0; j < kMaxTopK; ++j)
            s_route[row][j] = (j < a.top_k && row < a.M) ? clamp_expert(a.table[(int64_t)j * a.vocab + id], a.E) : -1;
    }
    const int per_wave = (G + NW - 1) / NW;
    const int s0 = wave * per_wave, s1 = std::min(s0 + per_wave, G);
    int xo[MT * 2];
    row_offsets<MT>(xo, (int)a.M, (int)(a.ldx * 2));
    f32x4 acc[MT][2];
    zero_acc16<MT, 2>(acc);
    constexpr int SB = stage_batch<MT, NW>();
    // block u of e4m3_spans is u * G spans on: the up block is two blocks after the gate's
    e4m3_spans<MT, 2, SB>(ar, xo, kb_a, lds + wave * SB * MT * 16 * kRowBytes, wr, 2 * G, s0, s1, acc);
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
    skinny_stash<MT, 2>(red, acc);
    __syncthreads();
    const float mult = routed ? 1.0f : a.shared_mult;
    for (int qi = threadIdx.x; qi < MT * 4 * 64; qi += NT) {
        const int l = qi & 63, i = (qi >> 6) & 3, tm = qi >> 8;
        const int row = tm * 16 + 4 * (l >> 4) + i;
        if (row >= a.M) continue;
        const int fl = l & 15;
        const float g = skinny_sum<MT, 2, NW>(red, tm, 0, i, l) * a.w_scale[pg + fl];
        const float u = skinny_sum<MT, 2, NW>(red, tm, 1, i, l) * a.w_scale[pg + 32 + fl];
        float hv = silu_f(g) * u * mult;
        if (routed) {
            float tw = 0.f;
#pragma unroll
            for (int j = 0; j < kMaxTopK; ++j) tw += (s_route[row][j] == expert) ? a.rw[j] : 0.f;
            hv = tw != 0.f ? hv * tw : 0.f;   // an unrouted expert's overflow stays out
        }
        h[row * a.ldh + f0 + fl] = (bf16_t)hv;
    }
}

// Split-K down over the concatenated features: workgroup (16 NU columns, K
// split), the waves take its spans in turn.  Spans [0, seg0) are the shared
// branch's, then seg1 spans per expert; each segment's columns have their own
// scale, applied to the accumulators where a wave's run leaves the segment.
// Writes the scaled partial part[split][row][col].
template <int MT, int NU, int NW>
__global__ __launch_bounds__(64 * NW) void k_down_e4m3(Down8Args a, float* part, int ncol, int splits) {
    constexpr int NT = 64 * NW;
    extern __shared__ __align__(16) char lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    // workgroups go to the XCDs in turn: neighbours share a K range of h
    const int ct = (int)blockIdx.x / splits, split = (int)blockIdx.x % splits;
    const int n0 = ct * 16 * NU;
    const int G = a.seg0 + a.E * a.seg1;
    const int p0 = (int)((int64_t)G * split / splits), p1 = (int)((int64_t)G * (split + 1) / splits);
    const int per_wave = (p1 - p0 + NW - 1) / NW;
    int s0 = p0 + wave * per_wave;
    const int s_end = std::min(s0 + per_wave, p1);
    const auto ar = make_rsrc(a.h, (uint32_t)(a.M * a.ldh * 2));
    const auto wr = make_rsrc(static_cast<const char*>(a.w_frag) + (n0 >> 4) * (int64_t)G * 1024,
                              (uint32_t)((int64_t)NU * G * 1024));
    const bool skip = a.M * a.top_k <= 16;
    const uint32_t live = skip && p1 > a.seg0 ? live_experts(a.ids, a.table, a.vocab, (int)a.M, a.top_k, a.E) : ~0u;
    int xo[MT * 2];
    row_offsets<MT>(xo, (int)a.M, (int)(a.ldh * 2));
    f32x4 total[MT][NU];
    zero_acc16<MT, NU>(total);
    constexpr int SB = stage_batch<MT, NW>();
    while (s0 < s_end) {
        const int seg = s0 < a.seg0 ? 0 : 1 + (s0 - a.seg0) / a.seg1;
        const int seg_end = seg == 0 ? a.seg0 : a.seg0 + seg * a.seg1;
        const int s1 = std::min(seg_end, s_end);
        if (seg == 0 || ((live >> (seg - 1)) & 1)) {
            float sc[NU];
#pragma unroll
            for (int u = 0; u < NU; ++u) sc[u] = a.w_scale[(int64_t)seg * a.scale_ld + n0 + u * 16 + (lane & 15)];
            f32x4 acc[MT][NU];
            zero_acc16<MT, NU>(acc);
            e4m3_spans<MT, NU, SB>(ar, xo, G * 128, lds + wave * SB * MT * 16 * kRowBytes, wr, G, s0, s1, acc);
#pragma unroll
            for (int tm = 0; tm < MT; ++tm)
#pragma unroll
                for (int u = 0; u < NU; ++u) total[tm][u] += acc[tm][u] * sc[u];
        }
        s0 = s1;
    }
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
    skinny_stash<MT, NU>(red, total);
    __syncthreads();
    float* dst = part + (int64_t)split * a.M * a.N;
    for (int qi = threadIdx.x; qi < MT * NU * 4 * 64; qi += NT) {
        const int l = qi & 63, i = (qi >> 6) & 3, u = (qi >> 8) % NU, tm = (qi >> 8) / NU;
        const int row = tm * 16 + 4 * (l >> 4) + i;
        const int col = n0 + u * 16 + (l & 15);
        if (row >= a.M || col >= a.N) continue;
        dst[row * (int64_t)a.N + col] = skinny_sum<MT, NU, NW>(red, tm, u, i, l);
    }
}

// out = sum of the partials in split order (+ residual), 4 columns a thread
// when they are whole 16-byte vectors (V = 4).
template <int V>
__global__ __launch_bounds__(256) void k_down_e4m3_sum(Down8Args a, const float* part, int splits) {
    const int nv = a.N / V;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= a.M * nv) return;
    const int64_t row = idx / nv;
    const int c0 = (int)(idx - row * nv) * V;
    const int64_t plane = a.M * a.N;
    const float* p = part + row * a.N + c0;
    using VT = std::conditional_t<V == 4, f32x4, float>;
    VT v{};
    for (int s = 0; s < splits; ++s) v += *reinterpret_cast<const VT*>(p + s * plane);
    const bf16_t* res = static_cast<const bf16_t*>(a.residual);
    bf16_t* out = static_cast<bf16_t*>(a.out) + row * a.ldo + c0;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        float o;
        if constexpr (V == 4) o = v[j]; else o = v;
        if (res != nullptr) o += (float)res[row * a.ldr + c0 + j];
        out[j] = (bf16_t)o;
    }
}

// 16-byte chunk d of block (b, g): row 16 b + d % 16, K values 64 g + 16 (d /
// 16) .. + 15; the source's columns are whole 8-byte groups, zero past cols.
__global__ __launch_bounds__(256) void k_pack_fragments_e4m3(const uint8_t* src, int64_t rows, int64_t cols8, int64_t ld,
                                                             uint8_t* dst, int64_t groups, int64_t dst_groups,
                                                             int64_t group0) {
    const int64_t total = rows / 16 * groups * 64;
    for (int64_t d = (int64_t)blockIdx.x * 256 + threadIdx.x; d < total; d += (int64_t)gridDim.x * 256) {
        const int64_t blk = d / (groups * 64), rem = d % (groups * 64);
        const int64_t g = rem / 64;
        const int l = (int)(rem % 64);
        const uint8_t* s = src + (blk * 16 + (l & 15)) * ld;
        const int64_t k = g * 64 + 16 * (l >> 4);
        u32x2 lo = {0u, 0u}, hi = {0u, 0u};
        if (k < cols8) lo = *reinterpret_cast<const u32x2*>(s + k);
        if (k + 8 < cols8) hi = *reinterpret_cast<const u32x2*>(s + k + 8);
        *reinterpret_cast<u32x4*>(dst + ((blk * dst_groups + group0 + g) * 64 + l) * 16) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
}

template <int MT, int NW>
int gate_up_mt(const GateUpArgs& a, int64_t packed_rows, hipStream_t stream) {
    auto kern = k_gate_up_e4m3<MT, NW>;
    constexpr int kLds = lds_bytes<MT, 2, NW>();
    const int st = set_kernel_lds(reinterpret_cast<const void*>(kern), kLds);
    if (st) return st;
    hipLaunchKernelGGL(kern, dim3((unsigned)(packed_rows / 32)), dim3(64 * NW), kLds, stream, a,
                       (int)(a.shared_feats / 16));
    return check_launch("gate_up_e4m3_decode");
}

// Columns per workgroup: 32 (one activation fragment feeds two weight
// blocks); splits: about 512 workgroups, two per CU, of at least 8 spans.
constexpr int kDownNU = 2;
int down_ncol(int64_t N) { return (int)((N + 16 * kDownNU - 1) / (16 * kDownNU)); }
int down_splits(int64_t N, int spans) {
    const int ncol = down_ncol(N);
    return std::max(1, std::min((512 + ncol - 1) / ncol, spans / 8));
}

template <int MT, int NW>
int down_mt(const Down8Args& a, float* part, hipStream_t stream) {
    auto kern = k_down_e4m3<MT, kDownNU, NW>;
    constexpr int kLds = lds_bytes<MT, kDownNU, NW>();
    int st = set_kernel_lds(reinterpret_cast<const void*>(kern), kLds);
    if (st) return st;
    const int ncol = down_ncol(a.N), splits = down_splits(a.N, a.seg0 + a.E * a.seg1);
    hipLaunchKernelGGL(kern, dim3((unsigned)(ncol * splits)), dim3(64 * NW), kLds, stream, a, part, ncol, splits);
    st = check_launch("down_e4m3_decode");
    if (st) return st;
    const bool vec = a.N % 4 == 0;
    const int64_t n = a.M * (vec ? a.N / 4 : a.N);
    hipLaunchKernelGGL(vec ? k_down_e4m3_sum<4> : k_down_e4m3_sum<1>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       stream, a, (const float*)part, splits);
    return check_launch("down_e4m3_decode (sum)");
}

}  // namespace

int launch_pack_fragments_e4m3(const void* src, int64_t rows, int64_t cols, int64_t ld, void* dst, int64_t dst_groups,
                               int64_t group0, hipStream_t stream) {
    const int64_t groups = (cols + kSpan - 1) / kSpan;
    int64_t blocks = (rows / 16 * groups * 64 + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_pack_fragments_e4m3, dim3((unsigned)blocks), dim3(256), 0, stream,
                       static_cast<const uint8_t*>(src), rows, (cols + 7) / 8 * 8, ld, static_cast<uint8_t*>(dst), groups,
                       dst_groups, group0);
    return check_launch("pack_fragments_e4m3");
}

int launch_gate_up_e4m3_decode(const GateUpArgs& a, int64_t packed_rows, hipStream_t stream) {
    if (a.M <= 16) return gate_up_mt<1, 8>(a, packed_rows, stream);
    if (a.M <= 32) return gate_up_mt<2, 8>(a, packed_rows, stream);
    if (a.M <= 64) return gate_up_mt<4, 8>(a, packed_rows, stream);
    return gate_up_mt<8, 4>(a, packed_rows, stream);
}

size_t down_e4m3_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    return (size_t)(down_splits(N, (int)((K + kSpan - 1) / kSpan)) * M * N) * sizeof(float);
}

int launch_down_e4m3_decode(const Down8Args& a, float* part, hipStream_t stream) {
    if (a.M <= 16) return down_mt<1, 8>(a, part, stream);
    if (a.M <= 32) return down_mt<2, 8>(a, part, stream);
    if (a.M <= 64) return down_mt<4, 8>(a, part, stream);
    return down_mt<8, 4>(a, part, stream);
}

}  // namespace trmoe
