// D3 + Q1/Q2: permute-by-expert dispatch with fused quantisation.
// Row of (t,k) = send_offset[e] + send_token_idx[t,k]  (moe_dispatch_normal.h:381-398)
// expand_idx[row] = (rank, t, k)                       (moe_dispatch_normal.h:335-344)
//
// One wave per (token, 1024-column chunk) for bf16 and fp8 rows (one wave
// per token for int8, whose scale needs the whole row).  The wave reads its
// slice of the token's row once (16-byte loads, lane l owns columns
// [1024 j + 16 l, +16)), quantises it once in registers, and writes the same
// bytes to each of the token's K destination rows as 16-byte stores: HBM
// traffic is one read of x and one write per routed row, the minimum.
//   quant_mode 0: bf16 copy.
//   quant_mode 2: int8 per token, s = 127/(amax+1e-12), q = rint(x*s), scale = 1/s
//                 (moe_dispatch_normal.h:295-332).
//   QUANT_INT8_FUSED (internal, the fused decode op): int8 per token, optional
//                 per-expert smooth scales, s = 127/amax.
//   quant_mode 3: fp8 e4m3fn per 1x128 block: amax clamped to >= 1e-4,
//                 q = e4m3_rne_sat(x * (448/amax)), scale = amax/448.  A block
//                 is 8 adjacent lanes, so its amax is a 3-step xor shuffle.
// Entries whose expert id is outside [0,E) are skipped.
#include "cam_device.h"
#include "launchers.h"
#include "prefill_dev.h"

namespace cam {

constexpr int DISP_WAVES = 4;
constexpr int DISP_NIT = 7;  // H <= 7168 = 7 * 1024
constexpr int DISP_MAX_K = 16;

// bf16 copy and fp8 1x128 quantisation: one wave per (token, 1024-column chunk) (dispatch_wave in
// prefill_dev.h).
template <int MODE>
__global__ __launch_bounds__(DISP_WAVES * 64) void dispatch_chunk_kernel(
    const uint16_t *__restrict__ x, const int32_t *__restrict__ topk_idx, const int32_t *__restrict__ send_offset,
    RankSrc rs, int T, int H, int K, int E, int rank, int cap, int nchunk,
    uint8_t *__restrict__ expand_x, float *__restrict__ scales, int32_t *__restrict__ expand_idx,
    int32_t *__restrict__ inv_out, int kmajor, int skip_unrouted)
{
    const long item = (long)blockIdx.x * DISP_WAVES + (threadIdx.x >> 6);
    if (item >= (long)T * nchunk)
        return;
    const int t = (int)(item / nchunk), j = (int)(item % nchunk);
    dispatch_wave<MODE>(x, topk_idx, send_offset, rs, t, j, T, H, K, E, rank, cap, expand_x, scales, expand_idx,
                        inv_out, kmajor, skip_unrouted, [] {});
}

// int8 per-token quantisation needs the whole row's amax: one wave per token, the row held in registers (lane l owns
// columns [1024 j + 16 l, +16)).
// FUSED = false: the prefill recipe, s = 127/(amax+1e-12) (moe_dispatch_normal.h:295-332).
// FUSED = true: the fused op's, s = 127/amax with no epsilon; a row of zeros gets q = 0 and scale 0
// (cam_moe_distribute_dispatch.h:640-681 and the shared-expert QuantToken,
// grouped_matmul_slice_m_per_token_dequant_swiglu_quant_multistage_workspace.h).
template <bool FUSED> __device__ __forceinline__ void int8_scale(float amax, float &sc, float &scale)
{
#pragma clang fp contract(off)
    if constexpr (FUSED) {
        sc = amax > 0.0f ? 127.0f / amax : 0.0f;
        scale = amax > 0.0f ? 1.0f / sc : 0.0f;
    } else {
        sc = 127.0f / (amax + 1e-12f);
        scale = 1.0f / sc;
    }
}
__device__ __forceinline__ u32x4 int8_row16(const float *f, float sc)
{
#pragma clang fp contract(off)
    u32x4 q;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t pk = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
            pk |= (uint32_t)((int)rintf(f[4 * w + b] * sc) & 0xff) << (8 * b);
        q[w] = pk;
    }
    return q;
}
__device__ __forceinline__ void row_source(int32_t *expand_idx, int row, int rank, int t, int k)
{
    expand_idx[(size_t)row * 3 + 0] = rank;
    expand_idx[(size_t)row * 3 + 1] = t;
    expand_idx[(size_t)row * 3 + 2] = k;
}

template <bool FUSED>
__global__ __launch_bounds__(DISP_WAVES * 64) void dispatch_int8_kernel(
    const uint16_t *__restrict__ x, const int32_t *__restrict__ topk_idx, const int32_t *__restrict__ send_offset,
    RankSrc rs, int T, int H, int K, int E, int rank, int cap,
    uint8_t *__restrict__ expand_x, float *__restrict__ scales, int32_t *__restrict__ expand_idx,
    int32_t *__restrict__ inv_out)
{
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * DISP_WAVES + (threadIdx.x >> 6);
    if (t >= T)
        return;
    const int dst = dispatch_dest(topk_idx, send_offset, rs, t, T, K, E, cap, lane);
    if (inv_out && lane < K)
        inv_out[(size_t)t * K + lane] = dst;
    const u32x4 *xr = reinterpret_cast<const u32x4 *>(x + (size_t)t * H);
    u32x4 raw[DISP_NIT][2];
#pragma unroll
    for (int j = 0; j < DISP_NIT; ++j) {
        const int col = j * 1024 + lane * 16;
        if (col < H) {
            raw[j][0] = __builtin_nontemporal_load(xr + (col >> 3));
            raw[j][1] = __builtin_nontemporal_load(xr + (col >> 3) + 1);
        } else {
            raw[j][0] = u32x4{0, 0, 0, 0};
            raw[j][1] = u32x4{0, 0, 0, 0};
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < DISP_NIT; ++j) {
        float f[16];
        unpack_bf16x8(raw[j][0], f);
        unpack_bf16x8(raw[j][1], f + 8);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            amax = fmaxf(amax, fabsf(f[i]));
    }
    float sc, tok_scale;
    int8_scale<FUSED>(group_max<64>(amax), sc, tok_scale);
    u32x4 q[DISP_NIT];
#pragma unroll
    for (int j = 0; j < DISP_NIT; ++j) {
        float f[16];
        unpack_bf16x8(raw[j][0], f);
        unpack_bf16x8(raw[j][1], f + 8);
        q[j] = int8_row16(f, sc);
    }
    const int ndst = K + (rs.share != nullptr);
    for (int k = 0; k < ndst; ++k) {
        const int row = __shfl(dst, k, 64);
        if (row < 0)
            continue;
        u32x4 *out = reinterpret_cast<u32x4 *>(expand_x + (size_t)row * H);
#pragma unroll
        for (int j = 0; j < DISP_NIT; ++j) {
            const int col = j * 1024 + lane * 16;
            if (col < H)
                out[col >> 4] = q[j];
        }
        if (lane == 0) {
            scales[row] = tok_scale;
            if (expand_idx && k < K)
                row_source(expand_idx, row, rank, t, k);
        }
    }
}

// The fused op's int8 rows one block per (token, destination): decode sizes, and smooth scales smooth[e, :] (e the
// destination expert, 0 for identity rows; share_smooth for the shared expert's rows), which multiply x first, so that
// every destination's row differs.  A block's 256 threads have the row and its scales in flight at once and read them
// once, where a wave per token walks its destinations in turn, two passes over the row for each (128 tokens of 7168
// columns, about one routed row each, and a shared expert, smooth scales: 6.1 us against 20 + 8.6 us that way).
constexpr int DF_THREADS = 256, DF_NIT = 2;  // H <= 7168 <= 2 * 256 * 16
// Without smooth scales the block per destination quantises a token's row once per local pick, the wave per token once in
// all.  One pick a token: the blocks always (4000 tokens of 7168 columns: 19.4 against 27.3 us).  More: up to as many picks
// as the GPU runs at once.  All picks local, 8 a token, us of the blocks against the waves: 7168 columns 7.0 and 10.9 at
// 1024 picks, 10.4 and 10.4 at 2048, 14.1 and 10.8 at 3072; 2048 columns 8.3 and 9.2 at 3072, 9.5 and 8.1 at 4096; 1024
// columns 7.2 and 7.3 at 3072, 8.4 and 7.5 at 4096.  With half of 4 picks local, 7168 columns: 8.2 and 8.5 at 2048, 12.3
// and 9.8 at 4096.
static bool int8_by_dest(long T, int K, int H) { return K == 1 || T * K <= (H <= 2048 ? 3072 : 2048); }
static_assert(DF_NIT * DF_THREADS * 16 >= DISP_NIT * 1024, "a row fits the block");
__global__ __launch_bounds__(DF_THREADS) void dispatch_int8_dest_kernel(
    const uint16_t *__restrict__ x, const int32_t *__restrict__ topk_idx, const int32_t *__restrict__ send_offset,
    RankSrc rs, int T, int H, int K, int E, int rank, int cap, uint8_t *__restrict__ expand_x,
    float *__restrict__ scales, int32_t *__restrict__ expand_idx, int32_t *__restrict__ inv_out,
    const float *__restrict__ smooth, const float *__restrict__ share_smooth)
{
#pragma clang fp contract(off)
    __shared__ float red[DF_THREADS / 64];
    const int ndst = K + (rs.share != nullptr), t = blockIdx.x / ndst, k = blockIdx.x % ndst;
    const int dst = __shfl(dispatch_dest(topk_idx, send_offset, rs, t, T, K, E, cap, threadIdx.x & 63), k, 64);
    if (inv_out && k < K && threadIdx.x == 0)
        inv_out[(size_t)t * K + k] = dst;
    if (dst < 0)
        return;
    const float *sm = k == K ? share_smooth : smooth;
    if (sm && k < K && topk_idx)
        sm += (size_t)topk_idx[(size_t)t * K + k] * H;
    const u32x4 *xr = reinterpret_cast<const u32x4 *>(x + (size_t)t * H);
    float f[DF_NIT][16], amax = 0.0f;
#pragma unroll
    for (int j = 0; j < DF_NIT; ++j) {
        const int col = (j * DF_THREADS + threadIdx.x) * 16;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            f[j][i] = 0.0f;
        if (col < H) {
            unpack_bf16x8(xr[col >> 3], f[j]);
            unpack_bf16x8(xr[(col >> 3) + 1], f[j] + 8);
            if (sm) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    f[j][i] = f[j][i] * sm[col + i];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < DF_NIT; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            amax = fmaxf(amax, fabsf(f[j][i]));
    amax = group_max<64>(amax);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = amax;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < DF_THREADS / 64; ++v)
        amax = fmaxf(amax, red[v]);
    float sc, scale;
    int8_scale<true>(amax, sc, scale);
    u32x4 *out = reinterpret_cast<u32x4 *>(expand_x + (size_t)dst * H);
#pragma unroll
    for (int j = 0; j < DF_NIT; ++j) {
        const int col = (j * DF_THREADS + threadIdx.x) * 16;
        if (col < H)
            out[col >> 4] = int8_row16(f[j], sc);
    }
    if (threadIdx.x == 0) {
        scales[dst] = scale;
        if (expand_idx && k < K)
            row_source(expand_idx, dst, rank, t, k);
    }
}

// Decode sizes (T*K <= DEC_MAX_TK): the layout (D1, the id preparation of the fused op and the count exchange
// of one rank) folded into the dispatch launch.  Every block (16 waves) computes the whole layout of the T*K
// picks in LDS -- the same stable per-expert ranks as layout_small_kernel: lanes sharing an expert found with
// one ballot per bit of its id, waves ordered by per-wave counts -- while its waves' loads of x are in flight,
// then dispatches its (token, chunk) items from the LDS copy.  Block 0 also writes the layout's outputs
// (counts, send offsets, inclusive counts, total, int64 tokens per expert); the grid clears `zero` (the
// chained GEMMs' counters).
constexpr int DEC_WAVES = 16;
constexpr int DEC_THREADS = DEC_WAVES * 64;
constexpr int DEC_MAX_TK = LAYOUT_LDS_MAX_TK;
constexpr int DEC_MAX_E = LAYOUT_LDS_MAX_E;

template <int MODE>
__global__ __launch_bounds__(DEC_THREADS) void dispatch_decode_kernel(
    const int32_t *__restrict__ ids, const uint8_t *__restrict__ active, const uint16_t *__restrict__ x, int T,
    int H, int K, int E, int cap, int nchunk, uint8_t *__restrict__ expand_x, float *__restrict__ scales,
    int32_t *__restrict__ expand_idx, int32_t *__restrict__ inv_out, int kmajor, int32_t *__restrict__ counts,
    int32_t *__restrict__ send_offset, int32_t *__restrict__ recv_count, int32_t *__restrict__ total,
    int64_t *__restrict__ tokens_per_expert, int32_t *__restrict__ zero, int nzero, int64_t *__restrict__ groups)
{
    __shared__ LayoutLds<DEC_THREADS> s;
    for (long i = (long)blockIdx.x * DEC_THREADS + threadIdx.x; i < nzero; i += (long)gridDim.x * DEC_THREADS)
        zero[i] = 0;
    auto layout = [&]() {
        layout_lds<DEC_THREADS>(ids, active, T, K, E, s);
        if (blockIdx.x == 0)
            layout_lds_store(s, E, counts, send_offset, recv_count, total, tokens_per_expert, groups, T);
    };
    const long item = (long)blockIdx.x * DEC_WAVES + (threadIdx.x >> 6);
    if (item >= (long)T * nchunk) {  // a wave without an item still takes its part in the block's layout
        layout();
        return;
    }
    const int t = (int)(item / nchunk), j = (int)(item % nchunk);
    const RankSrc rs{s.rank, nullptr, nullptr, 0, groups ? &s.total : nullptr};
    dispatch_wave<MODE>(x, s.ids, s.off, rs, t, j, T, H, K, E, 0, cap, expand_x, scales, expand_idx, inv_out,
                        kmajor, 0, layout);
}

hipError_t launch_dispatch_decode(const int32_t *ids, const uint8_t *active, const uint16_t *x, int T, int H, int K,
                                  int E, int cap, int quant_mode, void *expand_x, float *scales, int32_t *expand_idx,
                                  int32_t *inv_out, bool kmajor_scales, int32_t *counts, int32_t *send_offset,
                                  int32_t *recv_count, int32_t *total, int64_t *tokens_per_expert, hipStream_t s,
                                  int32_t *zero, int nzero, int64_t *groups)
{
    if (!dispatch_decode_fits(T, K, E) || K > DISP_MAX_K || H > DISP_NIT * 1024 || (H & 15) || nzero < 0 ||
        (quant_mode != QUANT_NONE && quant_mode != QUANT_FP8_BLOCK) || (quant_mode == QUANT_FP8_BLOCK && (H & 127)))
        return hipErrorInvalidValue;
    const int nchunk = (H + 1023) / 1024;
    const dim3 grid((unsigned)(((long)T * nchunk + DEC_WAVES - 1) / DEC_WAVES)), block(DEC_THREADS);
    uint8_t *ex = (uint8_t *)expand_x;
    if (quant_mode == QUANT_NONE)
        hipLaunchKernelGGL(dispatch_decode_kernel<QUANT_NONE>, grid, block, 0, s, ids, active, x, T, H, K, E, cap,
                           nchunk, ex, scales, expand_idx, inv_out, kmajor_scales ? 1 : 0, counts, send_offset,
                           recv_count, total, tokens_per_expert, zero, nzero, groups);
    else
        hipLaunchKernelGGL(dispatch_decode_kernel<QUANT_FP8_BLOCK>, grid, block, 0, s, ids, active, x, T, H, K, E,
                           cap, nchunk, ex, scales, expand_idx, inv_out, kmajor_scales ? 1 : 0, counts, send_offset,
                           recv_count, total, tokens_per_expert, zero, nzero, groups);
    return hipGetLastError();
}
bool dispatch_decode_fits(int T, int K, int E) { return T >= 1 && (long)T * K <= DEC_MAX_TK && E >= 1 && E <= DEC_MAX_E; }

hipError_t launch_dispatch(const uint16_t *x, const int32_t *topk_idx, const int32_t *send_offset,
                           const int32_t *send_token_idx, int T, int H, int K, int E, int rank, int cap, int quant_mode,
                           void *expand_x, float *scales, int32_t *expand_idx, hipStream_t s, int32_t *inv_out,
                           const float *smooth, bool kmajor_scales, const int32_t *chunk_base, int tpc,
                           const int32_t *chunk_rank, bool skip_unrouted, const int32_t *share,
                           const float *share_smooth)
{
    if (topk_idx && !send_token_idx && (!chunk_base || !chunk_rank || tpc < 1))
        return hipErrorInvalidValue;
    const RankSrc rs{send_token_idx, chunk_base, chunk_rank, tpc, share};
    if (T == 0)
        return hipSuccess;
    if (H > DISP_NIT * 1024 || K > DISP_MAX_K || (H & 15))
        return hipErrorInvalidValue;
    const dim3 block(DISP_WAVES * 64);
    const int nchunk = (H + 1023) / 1024;
    const dim3 grid_chunk((unsigned)(((long)T * nchunk + DISP_WAVES - 1) / DISP_WAVES));
    uint8_t *ex = (uint8_t *)expand_x;
    switch (quant_mode) {
    case QUANT_NONE:
        hipLaunchKernelGGL(dispatch_chunk_kernel<QUANT_NONE>, grid_chunk, block, 0, s, x, topk_idx, send_offset,
                           rs, T, H, K, E, rank, cap, nchunk, ex, scales, expand_idx, inv_out, 0, skip_unrouted ? 1 : 0);
        break;
    case QUANT_INT8_TOKEN:
        hipLaunchKernelGGL(dispatch_int8_kernel<false>, dim3((T + DISP_WAVES - 1) / DISP_WAVES), block, 0, s, x,
                           topk_idx, send_offset, rs, T, H, K, E, rank, cap, ex, scales, expand_idx, inv_out);
        break;
    case QUANT_INT8_FUSED:
        if (smooth || share_smooth || int8_by_dest(T, K, H))
            hipLaunchKernelGGL(dispatch_int8_dest_kernel, dim3((unsigned)T * (K + (share != nullptr))),
                               dim3(DF_THREADS), 0, s, x, topk_idx, send_offset, rs, T, H, K, E, rank, cap, ex, scales,
                               expand_idx, inv_out, smooth, share_smooth);
        else
            hipLaunchKernelGGL(dispatch_int8_kernel<true>, dim3((T + DISP_WAVES - 1) / DISP_WAVES), block, 0, s, x,
                               topk_idx, send_offset, rs, T, H, K, E, rank, cap, ex, scales, expand_idx, inv_out);
        break;
    case QUANT_FP8_BLOCK:
        if (H & 127)
            return hipErrorInvalidValue;
        hipLaunchKernelGGL(dispatch_chunk_kernel<QUANT_FP8_BLOCK>, grid_chunk, block, 0, s, x, topk_idx,
                           send_offset, rs, T, H, K, E, rank, cap, nchunk, ex, scales, expand_idx, inv_out,
                           kmajor_scales ? 1 : 0, skip_unrouted ? 1 : 0);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace cam
