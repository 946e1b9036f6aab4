// G1-G3: grouped expert GEMMs over ragged expert segments, bf16 or fp8 e4m3
// with 128x128 weight block scales and 1x128 activation scales.
//
// Semantics (CPU restatement in oracle/cam_oracle.c):
//   rows of A are in dispatch order; expert e owns rows [off_e, off_e+cnt_e),
//   off = exclusive prefix of group_list (tokens per local expert);
//   weights are stored N-major, K contiguous: W [L, N, K] (fp8 scales
//   [L, N/128, K/128]).
//   GMM1+SwiGLU (EPI_SWIGLU_*): N = 2I, rows [0,I) of W are the gate and
//     [I,2I) the up projection (block_epilogue_per_token_dequant_swiglu.h:256-286:
//     silu on the left half); h = silu(g) * u, silu(g) = g / (1 + exp(-g)) (hardware exp and reciprocal),
//     stored as bf16, or requantised to fp8 per 1x128 block of h exactly like
//     the dispatch quantiser (post_swiglu_dynamic_quant.h:164-231 requantises
//     per token in int8).
//   GMM2 (EPI_PLAIN): out = bf16(A W^T) per expert
//     (block_epilogue_per_token_dequant.hpp:338-361).
//
// Kernel design (gfx950):
//   * Output tiles of 256, 128, 64 or 32 rows x 256 W rows (SwiGLU: the gate and up rows of one 128-column
//     block of h; the decode plain GEMM 128 W rows), picked per expert from its row count (the Tile
//     struct below); the 128/256-row tiles run 8 waves in a 2 x 4 grid, the 32/64-row tiles 4 waves.  MFMA
//     16x16: v_mfma_f32_16x16x32_bf16, v_mfma_i32_16x16x64_i8, or v_mfma_scale_f32_16x16x128_f8f6f4 with
//     unit scales for fp8.
//   * Operands stream through a ring of LDS stages by direct global->LDS DMA (global_load_lds_dwordx4, or
//     buffer_load_dwordx4 ... lds through a buffer resource for the 128/256-row tiles): no staging
//     registers, and further k-steps stay in flight while one is multiplied.  Each k-step is 128 bytes of
//     every A and W row (64 bf16 / 128 one-byte elements); the fp8 activation scales of the k-step ride the
//     same DMA (4-byte lanes, read k-major [K/128, M] so that one k-step's scales of 64 rows are one
//     contiguous 256-byte run; row-major scales are transposed first).  A wave's loads are counted with
//     s_waitcnt vmcnt and published with a bare s_barrier (no fence, so outstanding prefetches are not
//     drained).
//   * LDS rows are 128 B with the 16-byte chunks XOR-swizzled by (row >> 1) & 7:
//     each lane fetches the global chunk that belongs at its DMA slot, so
//     fragment reads spread over all banks.
//   * MFMA operands are (W fragment, A fragment), so a lane's four
//     accumulators are four consecutive output columns of one row: the
//     epilogue stores 8 contiguous bytes per lane without a transpose.
//   * fp8: one MFMA of K=128 per (i,j) per k-step covers exactly one scale
//     block, so acc += mfma(...) * (a_scale[m] * w_scale[n-block]), applied by the VALU one fragment row
//     after the MFMA that produced it.
//   * Persistent grid (one block per CU) walking tiles expert by expert in
//     groups of 8 M-tiles x all N-tiles (M fastest), remapped so that the
//     blocks of one XCD take consecutive tiles: they share A and W tiles in
//     that XCD's L2.
#include <algorithm>
#include <cstdlib>
#include <atomic>
#include <type_traits>

#include "cam_device.h"
#include "gmm.h"
#include "gmm_plan.h"
#include "launchers.h"

namespace cam {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) int i32x8;

#ifndef CAM_GMM_MIN_NK256
#define CAM_GMM_MIN_NK256 16
#endif
#ifndef CAM_GMM_UNROLL2
// the 256-row tile's k-loop unrolled by two, so that the ring slot of each step is a constant and every LDS
// address an immediate offset (measured: the M = 65536 fp8 GMM1 2.18 vs 2.13 PFLOPS, config 3's bf16 GEMMs
// 1.31 vs 1.27 PFLOPS, config 4's 278-284 vs 286 us; fewer address and scalar instructions per k-step)
#define CAM_GMM_UNROLL2 1
#endif

constexpr int GBN = 256, GKB = 128;  // tile W-rows, bytes per row per k-step
constexpr int GMAX_THREADS = 512;    // block size of the largest tile
constexpr int G_MAX_L = 512;

// Tile shapes (BM rows x BN W rows, 128-byte k-steps):
//   BM = 256: 8 waves, 2 x 4 of 128 x 64, 2-stage ring -- half the L2->LDS bytes per FLOP of the
//             128-row tile, for compute-bound prefill;
//   BM = 128: 8 waves, 2 x 4 of 64 x 64, 3-stage ring;
//   BM = 32:  4 waves, 1 x 4 of 32 x 64, 4-stage ring (decode: a handful of rows per expert, the k-loop
//             is a weight stream and the extra stage keeps more of it in flight);
//   BM = 64:  4 waves, 1 x 4 of 64 x 64, 3-stage ring (a decode batch with more rows than that on an expert:
//             its weights pass once where two 32-row tiles fetch them twice);
//   BM = 32 or 64, BN = 128: 4 waves of 32 columns, 6-stage ring (the same bytes in flight) -- the decode
//             GEMM without SwiGLU, whose tiles then divide evenly over the CUs.
template <int BM_, int BN_ = GBN> struct Tile {
    static constexpr int BM = BM_, BN = BN_;
    static constexpr int NWAVES = BM >= 128 ? 8 : 4;
    static constexpr int THREADS = 64 * NWAVES;
    static constexpr int WAVES_M = BM >= 128 ? 2 : 1;
    static constexpr int WAVES_N = NWAVES / WAVES_M;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;  // wave tile
    static constexpr int IF = WM / 16, JF = WN / 16;              // MFMA fragments per wave
    static constexpr int STAGES = BM >= 256 ? 2 : BM >= 128 ? 3 : BN < 256 ? 6 : BM >= 64 ? 3 : 4;
    static constexpr int A_BYTES = BM * GKB;
    static constexpr int B_BYTES = BN * GKB;
    static constexpr int S_ROWS = WM > 64 ? WM : 64;  // activation-scale rows a wave DMAs (64 per instruction)
    static constexpr int S_DMAS = S_ROWS / 64;
    static constexpr int S_BYTES = NWAVES * S_ROWS * 4;  // per-wave copies of its rows' activation scales
    static constexpr int STAGE_BYTES = A_BYTES + B_BYTES + S_BYTES;
    static constexpr int A_LOADS = A_BYTES / 1024 / NWAVES;  // DMA instructions per wave per stage (1 KiB each)
    static constexpr int B_LOADS = B_BYTES / 1024 / NWAVES;
};

// W rows per tile: 256, except the decode tile (BM = 32) of the plain GEMM (a SwiGLU tile holds the gate and
// up rows of one 128-column scale block of h)
#ifndef CAM_GMM_SMALL_PLAIN_BN
#define CAM_GMM_SMALL_PLAIN_BN 128
#endif
constexpr int small_bn(int bm, int epi) { return bm <= 64 && epi == 0 ? CAM_GMM_SMALL_PLAIN_BN : GBN; }

// Tile classes: 256-row tiles; 128-row tiles; in int8 128-row tiles of experts of up to 32 rows, in fp8 and bf16 32-row
// tiles of these; and in the 4-wave kernels, in the place of CLS_128M, 64-row tiles.  The two 128-row classes differ in
// how they fetch their weights (see W_CACHED and W_STREAM).
enum TileClass { CLS_256 = 0, CLS_128M = 1, CLS_128S = 2, CLS_32 = 3, CLS_64 = 4 };
constexpr int G_NCLASS = 4;
constexpr int class_bm(int cls) { return cls == CLS_256 ? 256 : cls == CLS_32 ? 32 : cls == CLS_64 ? 64 : 128; }

// Expert tables of a launch, built once at kernel start: per tile class the inclusive prefix of M-tiles per
// expert, and the inclusive prefix of rows per expert (the exclusive prefix of expert e is entry e-1, or 0 for
// e = 0; no entry for it keeps the tables within the LDS budget).  The last two classes share a word: at most one
// tile per expert in either (<= 512); in a 4-wave launch (at most 48 rows per expert on average) CLS_32 alone, at most
// M / 32 + L tiles.
struct GroupTables {
    int tile_end[G_NCLASS - 2][G_MAX_L];
    uint32_t tile_end_s[G_MAX_L];  // CLS_128S << 16 | CLS_32
    int row_end[G_MAX_L];
    template <int CLS> __device__ __forceinline__ int end(int e) const
    {
        if constexpr (CLS < CLS_128S || CLS == CLS_64)
            return tile_end[CLS == CLS_64 ? CLS_128M : CLS][e];
        else
            return CLS == CLS_128S ? (int)(tile_end_s[e] >> 16) : (int)(tile_end_s[e] & 0xffffu);
    }
};
// the experts each class takes: a row count in [lo, hi) (lo >= hi: the class is not used)
struct ClassRanges {
    int lo[G_NCLASS], hi[G_NCLASS];
};

// Readiness between the two GEMMs of a chained launch (launch_gmm_chain): the GMM1 tiles of an M-tile
// produce its h rows, the GMM2 tiles of that M-tile consume them.  Counters are indexed by M-tile over the
// classes in turn (the 256-row M-tiles, then the 128-row ones, then the 32-row ones), the same in both GEMMs
// because both split every expert into the same tile height.
enum SyncRole { SYNC_NONE = 0, SYNC_PRODUCE = 1, SYNC_CONSUME = 2 };
struct GmmSync {
    int *ready;       // per M-tile: GMM1 tiles whose h rows have been stored
    int target;       // GMM1 tiles per M-tile (I / 128); one more when a test makes every wait give up
    long long ticks;  // wait bound in constant-clock ticks
};
// nonzero once a readiness wait has given up (sticky; read and cleared by the host, sync_status_read)
__device__ int g_cam_sync_status;

// The one argument of a chained kernel.  The GEMM loops already hold every scalar register they have, so the
// chained kernels keep nothing of it resident: each use re-reads the field from the kernel-argument segment
// through a pointer the compiler cannot see through (a scalar load), and each phase loads its own GEMM's
// arguments when it starts.
struct ChainParams {
    GmmArgs g1, g2;
    GmmSync sy;
};
__device__ __forceinline__ const ChainParams *chain_params()
{
    uint64_t a = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    // (a constant-address-space origin: the loads stay scalar loads)
    return (const ChainParams *)(const __attribute__((address_space(4))) ChainParams *)a;
}

// readiness counters of a chained launch: the M-tiles (at most M/32 + L), then the tile queues of the 8-wave kernel:
// GMM2's heavy tiles (one queue per XCD), the light tiles of GMM1 and of GMM2
__host__ __device__ constexpr int chain_queue_index(int M, int L) { return M / 32 + L + 1; }
__host__ __device__ constexpr int chain_light_index(int M, int L, bool gmm2) { return chain_queue_index(M, L) + 8 + gmm2; }

// h stores of a producing GMM1 tile: agent-coherent (sc1, written through to memory), so that a GMM2 tile on
// another XCD, whose L2 has never held these lines during the launch, reads them from memory
// (global address-space pointers: the atomics then need no aperture check of a flat address)
template <typename T> __device__ __forceinline__ __attribute__((address_space(1))) T *gptr(T *p)
{
    return (__attribute__((address_space(1))) T *)p;
}
template <bool CO, typename T> __device__ __forceinline__ void st_h(T *p, T v)
{
    if constexpr (CO)
        __hip_atomic_store(gptr(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        *p = v;
}

// Diagnostic build only (-DCAM_GMM_TIMELINE): every block records, per tile, its wall-clock start and end
// (100 MHz constant clock) with the tile's class, expert and index, into 128 slots per block;
// camhipDebugGmmTimeline copies them out.  Off in every product build.
#ifdef CAM_GMM_TIMELINE
constexpr int G_TL_SLOTS = 128, G_TL_BLOCKS = 1024;
__device__ uint64_t g_cam_tl[G_TL_BLOCKS * G_TL_SLOTS][3];
#define CAM_TL_DECL                                                                                             \
    int tl_k = (BM >= 256 ? 0 : BM >= 128 ? 32 : 64) + (ROLE == SYNC_CONSUME ? 16 : 0);                         \
    uint64_t tl_t0 = wall_clock64();
#define CAM_TL_REC(e, tile)                                                                                     \
    do {                                                                                                        \
        const uint64_t tl_t1 = wall_clock64();                                                                  \
        if (threadIdx.x == 0 && blockIdx.x < G_TL_BLOCKS && tl_k < G_TL_SLOTS) {                                \
            uint64_t *r = g_cam_tl[blockIdx.x * G_TL_SLOTS + tl_k];                                              \
            r[0] = ((uint64_t)blockIdx.x << 48) | ((uint64_t)BM << 36) | ((uint64_t)EPI << 32) |                 \
                   ((uint64_t)(e) << 20) | (uint64_t)(tile);                                                    \
            r[1] = tl_t0;                                                                                       \
            r[2] = tl_t1;                                                                                       \
        }                                                                                                       \
        ++tl_k;                                                                                                 \
        tl_t0 = tl_t1;                                                                                          \
    } while (0)
#else
#define CAM_TL_DECL
#define CAM_TL_REC(e, tile)
#endif

// Block-wide exclusive scans of the M-tiles of each tile class and of the rows per expert, from one read of
// the counts.  Only experts with a row count in a class's [lo, hi) get tiles of that class (a launch may
// split the experts between tile heights); the row offsets count every expert (they locate segments in
// dispatch order).
// MASK: the classes the kernel has (the others cost the scan nothing).  ntn (FOUR_WAVES): the GEMM's N-tiles.
// Returns the M-tiles of each class.
struct ClassTiles {
    int n[G_NCLASS];
};
template <int GTHREADS, int MASK, bool FOUR_WAVES = false>
__device__ ClassTiles build_group_tables(const int64_t *__restrict__ group_list, int L, GroupTables &gt, int *scratch,
                                   const ClassRanges &cr, int ntn = 0)
{
    constexpr int NQ = G_NCLASS + 1;  // tile counts per class, then rows
    constexpr int BMS[G_NCLASS] = {class_bm(0), class_bm(FOUR_WAVES ? CLS_64 : CLS_128M),
                                   FOUR_WAVES ? 32 : class_bm(2), class_bm(3)};
    constexpr int PER = (G_MAX_L + GTHREADS - 1) / GTHREADS, NWV = GTHREADS / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    auto used = [](int k) { return k == G_NCLASS || ((MASK >> k) & 1); };
    int rows[PER];  // experts PER tid + q, read once
#pragma unroll
    for (int q = 0; q < PER; ++q)
        rows[q] = tid * PER + q < L ? (int)group_list[tid * PER + q] : 0;
    int cnt[NQ] = {};
    auto add = [&](int c, int *v) {
#pragma unroll
        for (int k = 0; k < G_NCLASS; ++k)
            if (used(k))
                v[k] += (c >= cr.lo[k] && c < cr.hi[k]) ? (c + BMS[k] - 1) / BMS[k] : 0;
        v[G_NCLASS] += c;
    };
#pragma unroll
    for (int q = 0; q < PER; ++q)
        add(rows[q], cnt);
    // exclusive scan: within each wave by lane shuffles, then over the waves' totals
    int inc[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k)
        inc[k] = cnt[k];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            if (!used(k))
                continue;
            const int u = __shfl_up(inc[k], d, 64);
            if (lane >= d)
                inc[k] += u;
        }
    }
    if (lane == 63) {
#pragma unroll
        for (int k = 0; k < NQ; ++k)
            scratch[k * NWV + wv] = inc[k];
    }
    __syncthreads();
    int run[NQ], tot[NQ];  // the thread's exclusive prefix, the block's totals
    const int w = __builtin_amdgcn_readfirstlane(wv);
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        int ex = inc[k] - cnt[k], all = 0;
        if (used(k)) {
#pragma unroll
            for (int v = 0; v < NWV; ++v) {
                const int n = scratch[k * NWV + v];
                ex += v < w ? n : 0;
                all += n;
            }
        }
        run[k] = ex;
        tot[k] = __builtin_amdgcn_readfirstlane(all);
    }
    bool rows32 = false;
    if constexpr (FOUR_WAVES)  // slot 2 counts the M-tiles with 32-row tiles throughout (small_ranges)
        rows32 = small_rows32(tot[2] * ntn, (tot[CLS_128M] + tot[CLS_32]) * ntn, tot[CLS_128M] * ntn, (int)gridDim.x);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int e = tid * PER + q;
        add(rows[q], run);
        if (e < L) {
            if constexpr (FOUR_WAVES) {
                gt.tile_end[CLS_256][e] = 0;
                gt.tile_end[CLS_128M][e] = rows32 ? 0 : run[CLS_128M];
                gt.tile_end_s[e] = (uint32_t)(rows32 ? run[2] : run[CLS_32]);
                gt.row_end[e] = run[G_NCLASS];
                continue;
            }
            gt.tile_end[CLS_256][e] = run[CLS_256];
            gt.tile_end[CLS_128M][e] = run[CLS_128M];
            gt.tile_end_s[e] = (uint32_t)run[CLS_128S] << 16 | (uint32_t)run[CLS_32];
            gt.row_end[e] = run[G_NCLASS];
        }
    }
    __syncthreads();
    if constexpr (FOUR_WAVES)
        return {0, rows32 ? 0 : tot[CLS_128M], 0, rows32 ? tot[2] : tot[CLS_32]};
    return {tot[CLS_256], tot[CLS_128M], tot[CLS_128S], tot[CLS_32]};
}

// LDS byte offset of 16-byte chunk `chunk` of row `row`.  Chunks are XOR-swizzled by (row >> 1) & 7:
// two 128-byte rows share one 256-byte bank row, so the 16 rows of a fragment read (same logical
// chunk) land on 16 distinct 16-byte bank groups.
__device__ __forceinline__ int swz(int row, int chunk) { return row * GKB + ((chunk ^ ((row >> 1) & 7)) << 4); }

// the lane's index in its wave, from mbcnt (no work-item id register)
__device__ __forceinline__ int lane_id() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// the same, recomputed where it stands (FRESH): what a tile switch derives from the lane is then not kept in registers
// through the k-loop, which in the fp8 kernels spills it, each reload waiting for every store of the epilogue
// before it.  The other kernels have the registers to keep it.
template <bool FRESH> __device__ __forceinline__ int lane_here()
{
    int l = lane_id();
    if constexpr (FRESH)
        asm volatile("" : "+v"(l));
    return l;
}

// s_waitcnt with only vmcnt constrained (expcnt and lgkmcnt at their maxima)
template <int N> __device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (7 << 4) | (0xF << 8));
}

// s_waitcnt vmcnt(N) and lgkmcnt(0): this wave's older DMAs and all of its LDS reads are done
template <int N> __device__ __forceinline__ void wait_vmcnt_lgkm0()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (7 << 4));
}

// barrier without a memory fence: prefetches in flight stay in flight
__device__ __forceinline__ void bar()
{
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ void dma16(const void *g, void *lds)
{
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}
// the same with the nontemporal cache policy: a stream read once (decode weights) is not kept in L2
__device__ __forceinline__ void dma16_nt(const void *g, void *lds)
{
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds, 16, 0, 2);
}
__device__ __forceinline__ void dma4(const void *g, void *lds)
{
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds, 4, 0, 0);
}
// agent-coherent (sc1): data another XCD may have written during the launch
__device__ __forceinline__ void dma4_sc1(const void *g, void *lds)
{
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds, 4, 0, 16);
}

// The same DMAs through a buffer resource: the base sits in four SGPRs, the lane's 32-bit byte offset in one
// VGPR and the k-step's offset in an SGPR, so a DMA needs no 64-bit address registers and no address
// arithmetic per k-step.  Offsets are 32-bit, as the flat addresses' per-lane offsets already are: the C ABI
// rejects activations or one expert's weights of 4 GiB or more, and the activation scales are a 32nd of the
// activations.  The record count is unbounded (no range check, as with flat addresses).
#ifndef CAM_GMM_BUFDMA
#define CAM_GMM_BUFDMA 1
#endif
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *base)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, -1, 0x00020000);
}
template <int BYTES, int AUX>
__device__ __forceinline__ void bdma(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, void *lds)
{
    auto *l = (__attribute__((address_space(3))) void *)lds;
    if constexpr (BYTES == 4 && AUX == 16)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, l, 4, voff, soff, 0, 16);
    else if constexpr (BYTES == 4)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, l, 4, voff, soff, 0, 0);
    else if constexpr (AUX == 2)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, l, 16, voff, soff, 0, 2);
    else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, l, 16, voff, soff, 0, 0);
}

// scalar (SMEM) load of a block-uniform element of read-only data: it counts on lgkmcnt, not on the
// vmcnt of the DMA ring, so it never makes a wait drain prefetches
__device__ __forceinline__ float sload(const float *p, int idx)
{
    return ((const __attribute__((address_space(4))) float *)p)[idx];
}

// LDS-only barrier: this wave's LDS traffic has completed, then every wave meets; DMAs in flight stay
// in flight
__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_s_waitcnt(0xF | (3 << 14) | (7 << 4));  // lgkmcnt(0), vmcnt and expcnt at their maxima
    bar();
}

// The tiles of one class: this block takes a run of rn tiles rs, rs + rstride, ..., then tiles first, first + G, ...
// (an increasing sequence: the first index past the class's tiles ends it), or tickets of a queue.
// ROLE (chained launches only): SYNC_PRODUCE tiles store h agent-coherently and count each finished tile in
// sy.ready; SYNC_CONSUME tiles start their DMAs only once sy.ready of their M-tile has reached sy.target.  Waves
// beyond the tile's own (a 32-row class run by an 8-wave block) are spectators: they issue no DMA, MFMA or store
// and only meet the block's barriers.
// A dynamic tile queue: tickets off, off + 1, ... handed out one at a time by the counter SY().ready[ctr]; ticket t
// of [base, end) is tile first + t - base of the class at hand.  tk: the block's first ticket, -1 to take one.
struct TileQueue {
    int ctr, off, base, end, first, tk;
};

// EAGER (the 4-wave chained kernel): a producer's primed tile counts its predecessor at k-step edge STAGES-2
// instead of after its k-loop (a branch inside the k-loop, which the 8-wave kernels cannot afford).
// wv: the wave's index in the block (a scalar the kernel computes once; -1: from threadIdx.x).  The body
// takes the lane from mbcnt and never reads the work-item id: a register holding it through the whole kernel
// gets spilled, and each reload before a k-loop makes the loop wait for it at every iteration.
// How a tile fetches its weights: cached, nontemporally, or either by the number of the expert's M-tiles (a k-loop for
// each: the 8-wave kernels have no registers for that).  An expert that fits one M-tile has its weights read exactly
// once; the M-tiles of an expert of several, which the tile order runs side by side on one XCD, re-read them from that
// XCD's L2 (48 experts of 36 to 281 rows, fp8, K = 4096, N = 2816: 173 us cached, 205 us nontemporal).  A stream past
// the caches pays for light tiles: the 4-wave decode tiles, and in the 8-wave kernels the experts of up to 32 rows (32-row
// tiles; in int8 128-row ones).  int8, weights that differ from call to call, the layer of 8 experts of 1 to 24 rows,
// H = 2304, I = 1792: 55.0 us, 60.3 us cached; 16 experts of 2 to 194 rows, H = 4864, I = 512: 78.3 us against 86.0 with
// every single M-tile (up to 128 rows) streamed and 91.0 with none; the skewed layer of 22 touched experts, one of 2311
// rows: 342.6 against 354.7 us with every single M-tile; 32 experts of 122 rows on average, H = 4352, I = 6784: 688
// against 718 and 705 us.
enum WPolicy { W_CACHED = 0, W_STREAM = 1, W_BY_TILE = 2 };
// 64-row tiles in fp8, which has no registers for two loops: as a stream, also where an expert has several (the decode
// step of 400 tokens, 64 experts, H = 2048, I = 1408 140 against 148 us cached; 32 experts of 44 rows, H = 4096,
// I = 1536: 144 against 148 us; the steps of 16 to 4096 tokens with a shared expert on all of them within 1%).
constexpr int policy64(int dt) { return dt == DT_FP8 ? W_STREAM : W_BY_TILE; }
constexpr int class_policy(int cls) { return cls == CLS_128S || cls == CLS_32 ? W_STREAM : W_CACHED; }

template <int DT, int EPI, int CLS, int ROLE = SYNC_NONE, bool EAGER = false, int POL = class_policy(CLS), bool HALVES = false>
__device__ __forceinline__ int gmm_body(const GmmArgs &p, const GroupTables *gtab, int first, int rs = 0, int rn = 0,
                                        int rstride = 1, int wv = -1, const TileQueue &tq = TileQueue{},
                                        int half0 = 0)
{
    constexpr int BM = class_bm(CLS);
    using TC = Tile<BM, small_bn(BM, EPI)>;
    constexpr int TBN = TC::BN;
    constexpr int NW = TC::NWAVES;
    constexpr int GBM = TC::BM, WM = TC::WM, WN = TC::WN, IF = TC::IF, JF = TC::JF;
    constexpr int GSTAGES = TC::STAGES, STAGE_BYTES = TC::STAGE_BYTES;
    constexpr int A_BYTES = TC::A_BYTES, B_BYTES = TC::B_BYTES, A_LOADS = TC::A_LOADS, B_LOADS = TC::B_LOADS;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    // the epilogue's exchange area (fp8 amax, int8 row maxima) follows this class's ring
    int *scratch = reinterpret_cast<int *>(smem + GSTAGES * STAGE_BYTES);
    // HALVES (CLS_128M): the 256-row tiles from index half0 on, each as two tiles of 128 rows.  (An instance of its own: a
    // run-time choice in the light tiles' one cost them scalar registers, the fp8 GEMMs of 16 experts of 256 rows, H = 7168,
    // I = 1024 204.6 against 201.0 us, of 8 experts of 856 to 2893 rows, H = 1024, I = 13056 811 against 796 us.)
    static_assert(!HALVES || CLS == CLS_128M);
    auto tile_end = [&](int e) { return gtab->template end<HALVES ? CLS_256 : CLS>(e); };
    auto tile_prefix = [&](int e) { return e > 0 ? tile_end(e - 1) : 0; };
    auto row_off = [&](int e) { return e > 0 ? gtab->row_end[e - 1] : 0; };

    constexpr bool FRESH = DT == DT_FP8;
    const int lane = lane_id();
    const int w = wv >= 0 ? wv : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const bool first_thread = w == 0 && lane == 0;
    const int wm = w / TC::WAVES_N, wn = w % TC::WAVES_N;
    const int l16 = lane & 15, lg = lane >> 4;
    constexpr bool PRODUCE = ROLE == SYNC_PRODUCE, CONSUME = ROLE == SYNC_CONSUME;
    const bool spect = ROLE != SYNC_NONE && NW < 8 && w >= NW;  // (8-wave tiles never have spectators)
    // M-tiles of the classes before this one (the readiness counters' index base), read when needed
    auto cls_base = [&]() {
        int b = 0;
        constexpr int SLOT = CLS == CLS_64 ? CLS_128M : CLS;
        if constexpr (SLOT > CLS_256)
            b += gtab->template end<CLS_256>(p.L - 1);
        if constexpr (SLOT > CLS_128M)
            b += gtab->template end<CLS_128M>(p.L - 1);
        if constexpr (SLOT > CLS_128S)
            b += gtab->template end<CLS_128S>(p.L - 1);
        return __builtin_amdgcn_readfirstlane(b);
    };
    constexpr bool SWIGLU = EPI != EPI_PLAIN;
    constexpr bool FP8 = DT == DT_FP8;
    constexpr bool INT8 = DT == DT_INT8;
    constexpr int LOADS = A_LOADS + B_LOADS + (FP8 ? TC::S_DMAS : 0);  // DMA instructions per wave per stage
    const int esz = DT == DT_BF16 ? 2 : 1;
    const uint32_t kbytes = (uint32_t)p.K * esz;  // bytes per row
    const int nk = (int)(kbytes / GKB);
    const int half_n = p.N / 2;                    // I for SwiGLU
    const int ntn = SWIGLU ? half_n / 128 : p.N / TBN;
    int total = __builtin_amdgcn_readfirstlane(tile_prefix(p.L)) * ntn;
    if (HALVES)
        total = 2 * (total - half0);

    const int G = gridDim.x, logical = first;
    // tiles from the queue tq, in the 8-wave chained kernel: the consumer's heavy tiles (a queue per XCD) and the
    // light tiles of both GEMMs
    constexpr bool dyn = CONSUME && BM >= 256;
    constexpr bool DYNL = ROLE != SYNC_NONE && BM < 256 && !EAGER;
    int tk = tq.tk;
    auto ticket_tile = [&](int t) { return t < tq.end ? tq.first + t - tq.base : 0x7fffffff; };
    // the block's k-th tile: the run, then the strided sequence
    auto seq = [&](int k) { return k < rn ? rs + k * rstride : logical + (k - rn) * G; };

    // DMA slot of this lane inside a 1 KiB band (8 rows x 128 B): row l/8, physical chunk l%8,
    // which holds logical chunk (l%8) ^ ((row >> 1) & 7) -- see swz()

    // ---- one tile's coordinates and the per-lane sources of this wave's DMA bands
    struct Ctx {
        int e, row0, seg1, n0;
        const uint8_t *wbase;
        const float *wsb;  // this expert's weight scales (fp8 block or int8 per-channel), or null
        uint32_t ga[A_LOADS], gb[B_LOADS], gs[TC::S_DMAS];
        int wsg, wsu;  // fp8: weight-scale row offsets (gate / up n-blocks, or the wave's column block)
        int active;    // some row of this wave lies inside the segment (an int: a bool tail makes struct copies go through scratch)
        int nt;        // the expert's only M-tile (W_BY_TILE)
    };
    auto setup = [&](int index, Ctx &c) {
        const int tile = HALVES ? half0 + (index >> 1) : index;
        const int lane = lane_here<FRESH>(), band_row = lane >> 3;
        auto chunk_off = [&](int r) { return (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) << 4); };
        int lo = 0, hi = p.L - 1;
        while (lo < hi) {  // last e with tile_prefix[e]*ntn <= tile
            const int mid = (lo + hi + 1) >> 1;
            if (tile_end(mid - 1) * ntn <= tile)
                lo = mid;
            else
                hi = mid - 1;
        }
        const int e = __builtin_amdgcn_readfirstlane(lo);
        c.e = e;
        const int mt_e = __builtin_amdgcn_readfirstlane(tile_end(e) - tile_prefix(e));
        const int local = __builtin_amdgcn_readfirstlane(tile - tile_prefix(e) * ntn);
        // within the expert: groups of up to 8 M-tiles, N-tiles in turn, the group's M-tiles
        // fastest -- a run of consecutive tiles (one XCD's share of a round) covers ~8 A row blocks
        // x a few W column blocks, so both operands are re-read from that XCD's L2
        constexpr int GM = 8;
        const int grp = local / (GM * ntn), rem = local % (GM * ntn);
        const int gm = min(GM, mt_e - grp * GM);
        const int nt = rem / gm, mt = grp * GM + rem % gm;
        const int seg0 = __builtin_amdgcn_readfirstlane(row_off(e));
        c.seg1 = min(__builtin_amdgcn_readfirstlane(gtab->row_end[e]), p.M);  // never write past row M
        c.row0 = HALVES ? seg0 + mt * 2 * GBM + (index & 1) * GBM : seg0 + mt * GBM;
        c.n0 = SWIGLU ? nt * 128 : nt * TBN;  // first h-column (SwiGLU) or W row (plain)
        // a wave whose rows all lie past the segment skips its MFMAs (it still moves its share of the
        // DMA and meets every barrier): a tile of a short segment costs little more than its weights
        c.active = !spect && c.row0 + wm * WM < c.seg1;
        c.nt = mt_e == 1;

        if (e == p.ex) {
            c.wbase = p.Wx;
            c.wsb = p.Wsx;
        } else if (p.Wl) {  // separated weights: one allocation per expert, pointers read by scalar loads (a vector
                     // load here would make the tile switch wait for every DMA in flight)
            c.wbase = reinterpret_cast<const uint8_t *>(
                ((const __attribute__((address_space(4))) uint64_t *)p.Wl)[e]);
            c.wsb = p.Wsl ? reinterpret_cast<const float *>(((const __attribute__((address_space(4))) uint64_t *)p.Wsl)[e])
                          : nullptr;
        } else {
            c.wbase = p.W + (size_t)e * p.N * kbytes;
            c.wsb = !p.Ws ? nullptr : p.Ws + (INT8 ? (size_t)e * p.N : (size_t)e * (p.N / 128) * nk);
        }
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            const int r = (i * NW + w) * 8 + band_row;  // tile row 0..GBM-1
            c.ga[i] = (uint32_t)min(c.row0 + r, c.seg1 - 1) * kbytes + chunk_off(r);
        }
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i) {
            const int r = (i * NW + w) * 8 + band_row;  // LDS W row 0..255
            int wrow;
            if (SWIGLU) {
                // LDS rows [WN c, WN c + WN) feed column wave c: WN/2 gate rows, then the
                // WN/2 up rows of the same h-columns
                const int cw = r / WN, jj = r % WN;
                const int hcol = c.n0 + (WN / 2) * cw + (jj % (WN / 2));
                wrow = jj < WN / 2 ? hcol : half_n + hcol;
            } else {
                wrow = c.n0 + r;
            }
            c.gb[i] = (uint32_t)wrow * kbytes + chunk_off(r);
        }
        // fp8: this wave's activation-scale rows (the WM rows of its row block wm, 64 per DMA), placed so that
        // the IF rows a lane multiplies (16 i + l16, i < IF) sit next to each other: LDS slot p holds row
        // (p % IF) 16 + p / IF, and a lane reads its IF scales with one or two vector reads per k-step
        // (per-row 4-byte reads interleaved with the MFMAs: the M = 65536 fp8 GEMMs ~3% slower)
#pragma unroll
        for (int d = 0; d < TC::S_DMAS; ++d) {
            const int p = d * 64 + lane;
            const int r = p < WM ? (p % IF) * 16 + p / IF : p;
            c.gs[d] = (uint32_t)min(c.row0 + wm * WM + r, c.seg1 - 1);  // k-major: + kc * M
        }
        c.wsg = ((SWIGLU ? c.n0 : c.n0 + wn * WN) / 128) * nk;
        c.wsu = SWIGLU ? ((half_n + c.n0) / 128) * nk : c.wsg;
    };
    // DMA instruction q (0 <= q < LOADS) of k-step kc of tile c into ring slot `slot`: A bands, then
    // W bands (nt: nontemporally), then (fp8) the activation scales
    auto dma_one = [&](const Ctx &c, int kc, int slot, int q, auto nt) {
        constexpr bool NTW = decltype(nt)::value;
        if (spect)
            return;
        uint8_t *st = smem + slot * STAGE_BYTES;
        if constexpr (CAM_GMM_BUFDMA && BM >= 128) {  // (the decode tile measured 0.4 us slower per step this way)
            if (q < A_LOADS) {
                bdma<16, 0>(buf_rsrc(p.A), c.ga[q], (uint32_t)kc * GKB, st + (q * NW + w) * 1024);
            } else if (q < A_LOADS + B_LOADS) {
                const int i = q - A_LOADS;
                bdma<16, NTW ? 2 : 0>(buf_rsrc(c.wbase), c.gb[i], (uint32_t)kc * GKB,
                                      st + A_BYTES + (i * NW + w) * 1024);
            } else {
                const int d = q - A_LOADS - B_LOADS;
                bdma<4, CONSUME ? 16 : 0>(buf_rsrc(p.As), c.gs[d] * 4u, (uint32_t)kc * (uint32_t)p.M * 4u,
                                          st + A_BYTES + B_BYTES + w * TC::S_ROWS * 4 + d * 256);
            }
            return;
        }
        if (q < A_LOADS) {
            dma16(p.A + c.ga[q] + (uint32_t)kc * GKB, st + (q * NW + w) * 1024);
        } else if (q < A_LOADS + B_LOADS) {
            const int i = q - A_LOADS;
            if constexpr (NTW)
                dma16_nt(c.wbase + c.gb[i] + (uint32_t)kc * GKB, st + A_BYTES + (i * NW + w) * 1024);
            else
                dma16(c.wbase + c.gb[i] + (uint32_t)kc * GKB, st + A_BYTES + (i * NW + w) * 1024);
        } else {
            const int d = q - A_LOADS - B_LOADS;
            if constexpr (CONSUME)
                dma4_sc1(p.As + c.gs[d] + (size_t)kc * p.M, st + A_BYTES + B_BYTES + w * TC::S_ROWS * 4 + d * 256);
            else
                dma4(p.As + c.gs[d] + (size_t)kc * p.M, st + A_BYTES + B_BYTES + w * TC::S_ROWS * 4 + d * 256);
        }
    };

    f32x4 acc[IF][JF];
    // fp8: the lane's IF activation scales of a stage (rows 16 i + l16), contiguous in the wave's scale slot
    auto rd_scales = [&](const uint8_t *st, float *sa) {
        const float *sp = reinterpret_cast<const float *>(st + A_BYTES + B_BYTES + w * TC::S_ROWS * 4) + l16 * IF;
        if constexpr (IF % 4 == 0) {
#pragma unroll
            for (int q = 0; q < IF / 4; ++q) {
                const f32x4 v = reinterpret_cast<const f32x4 *>(sp)[q];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    sa[4 * q + u] = v[u];
            }
        } else {
#pragma unroll
            for (int q = 0; q < IF; ++q)
                sa[q] = sp[q];
        }
    };

    // ---- epilogue: lane holds rows m = row0 + wm*WM + 16 i + l16 and, per j, four
    // consecutive columns 16 j + 4 lg + q of the wave's WN-wide column range
    auto epilogue = [&](const Ctx &c) {
        if (spect) {
            if constexpr (EPI == EPI_SWIGLU_FP8) {
                lds_sync();  // the two exchange barriers of the fp8 requantisation
                lds_sync();
            }
            return;
        }
        const int row0 = c.row0, seg1 = c.seg1, n0 = c.n0;
        const int lid = lane_here<FRESH>(), l16 = lid & 15, lg = lid >> 4;
        if constexpr (EPI == EPI_PLAIN) {
            uint16_t *out = reinterpret_cast<uint16_t *>(p.C);
            if (c.e == p.ex)
                out = reinterpret_cast<uint16_t *>(p.Cx) - (size_t)__builtin_amdgcn_readfirstlane(row_off(c.e)) * p.N;
#pragma unroll
            for (int i = 0; i < IF; ++i) {
                const int m = row0 + wm * WM + i * 16 + l16;
                if (m >= seg1)
                    continue;
                uint16_t *crow = out + (size_t)m * p.N + n0 + wn * WN + 4 * lg;
#pragma unroll
                for (int j = 0; j < JF; ++j) {
                    u32x2 v;
                    v[0] = f32x2_to_bf16x2(acc[i][j][0], acc[i][j][1]);
                    v[1] = f32x2_to_bf16x2(acc[i][j][2], acc[i][j][3]);
                    *reinterpret_cast<u32x2 *>(crow + 16 * j) = v;
                }
            }
        } else {
            // h-columns of this wave: n0 + (WN/2) wn + 16 j + 4 lg + q, j < JF/2 (gate j, up j+JF/2)
            constexpr int HF = JF / 2;
            float h[IF][HF][4];
#pragma unroll
            for (int i = 0; i < IF; ++i)
#pragma unroll
                for (int j = 0; j < HF; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float g = acc[i][j][q], u = acc[i][j + HF][q];
                        // silu(g) = g / (1 + exp(-g)) with the hardware exp and reciprocal (about 1 ulp
                        // each; measured: the decode step 1 us and the M = 65536 fp8 GMM1 4% faster than
                        // the correctly rounded division)
                        h[i][j][q] = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
                    }
            if constexpr (EPI == EPI_SWIGLU_F32AMAX) {
                // fp32 h and this wave's partial row maximum of |h| (its 32 h-columns), one slot per wave and
                // row, so the requantisation needs no zeroed buffer and no atomics
#pragma unroll
                for (int i = 0; i < IF; ++i) {
                    const int m = row0 + wm * WM + i * 16 + l16;
                    float mx = 0.0f;
#pragma unroll
                    for (int j = 0; j < HF; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            mx = fmaxf(mx, fabsf(h[i][j][q]));
                    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
                    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                    if (m < seg1) {
                        float *hrow = reinterpret_cast<float *>(p.C) + (size_t)m * half_n + n0 + (WN / 2) * wn + 4 * lg;
#pragma unroll
                        for (int j = 0; j < HF; ++j)
                            *reinterpret_cast<f32x4 *>(hrow + 16 * j) =
                                f32x4{h[i][j][0], h[i][j][1], h[i][j][2], h[i][j][3]};
                        static_assert(WN / 2 == GMM_AMAX_COLS, "one partial maximum per wave's h-columns");
                        if (lg == 0)
                            p.Cs[(size_t)m * (half_n / GMM_AMAX_COLS) + n0 / GMM_AMAX_COLS + wn] = mx;
                    }
                }
            } else if constexpr (EPI == EPI_SWIGLU_BF16) {
#pragma unroll
                for (int i = 0; i < IF; ++i) {
                    const int m = row0 + wm * WM + i * 16 + l16;
                    if (m >= seg1)
                        continue;
                    uint16_t *hrow =
                        reinterpret_cast<uint16_t *>(p.C) + (size_t)m * half_n + n0 + (WN / 2) * wn + 4 * lg;
#pragma unroll
                    for (int j = 0; j < HF; ++j) {
                        const uint64_t v = (uint64_t)f32x2_to_bf16x2(h[i][j][0], h[i][j][1]) |
                                           ((uint64_t)f32x2_to_bf16x2(h[i][j][2], h[i][j][3]) << 32);
                        st_h<PRODUCE>(reinterpret_cast<uint64_t *>(hrow + 16 * j), v);
                    }
                }
            } else {
                // fp8 1x128 requant: the tile's 128 h-columns of a row are one scale block,
                // split over the column waves; exchange partial amax through LDS
                float *red = reinterpret_cast<float *>(scratch);  // [WAVES_N][GBM]
#pragma unroll
                for (int i = 0; i < IF; ++i) {
                    float mx = 0.0f;
#pragma unroll
                    for (int j = 0; j < HF; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            mx = fmaxf(mx, fabsf(h[i][j][q]));
                    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
                    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                    if (lg == 0)
                        red[wn * GBM + wm * WM + i * 16 + l16] = mx;
                }
                lds_sync();
                // every row's block maximum first, then all the stores back to back: a register reload
                // between two rows' stores would wait for the earlier stores to complete (vmcnt counts both)
                float amx[IF];
#pragma unroll
                for (int i = 0; i < IF; ++i) {
                    const int r = wm * WM + i * 16 + l16;
                    float amax = 1e-4f;
#pragma unroll
                    for (int cc = 0; cc < TC::WAVES_N; ++cc)
                        amax = fmaxf(amax, red[cc * GBM + r]);
                    amx[i] = amax;
                }
#pragma unroll
                for (int i = 0; i < IF; ++i) {
                    const int m = row0 + wm * WM + i * 16 + l16;
                    const float inv = 448.0f / amx[i];
                    if (m < seg1) {
                        uint8_t *hrow = p.C + (size_t)m * half_n + n0 + (WN / 2) * wn + 4 * lg;
#pragma unroll
                        for (int j = 0; j < HF; ++j)
                            st_h<PRODUCE>(reinterpret_cast<uint32_t *>(hrow + 16 * j),
                                          f32x4_to_e4m3(h[i][j][0] * inv, h[i][j][1] * inv, h[i][j][2] * inv,
                                                        h[i][j][3] * inv));
                        if (wn == 0 && lg == 0)
                            st_h<PRODUCE>(p.Cs + (size_t)(n0 / 128) * p.M + m, amx[i] / 448.0f);  // k-major h scales
                    }
                }
                lds_sync();  // red is reused by the next tile
            }
        }
    };
    auto clear_acc = [&]() {
#pragma unroll
        for (int i = 0; i < IF; ++i)
#pragma unroll
            for (int j = 0; j < JF; ++j)
                acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };

    // int8: per-channel x per-token dequantisation of the exact int32 sums:
    // v = ((float)acc * w_scale[n]) * x_scale[m]  (block_epilogue_per_token_dequant*.h)
    auto dequant_int8 = [&](const Ctx &cur) {
        if constexpr (INT8) {
            const int lid = lane_here<FRESH>(), l16 = lid & 15, lg = lid >> 4;
            const float *wsr = cur.wsb;
#pragma unroll
            for (int j = 0; j < JF; ++j) {
                int c0;
                if (SWIGLU) {
                    const int jj = j % (JF / 2);
                    c0 = cur.n0 + (WN / 2) * wn + 16 * jj + 4 * lg + (j >= JF / 2 ? half_n : 0);
                } else {
                    c0 = cur.n0 + wn * WN + 16 * j + 4 * lg;
                }
                const f32x4 wv = *reinterpret_cast<const f32x4 *>(wsr + c0);
#pragma unroll
                for (int i = 0; i < IF; ++i) {
                    const float xs = p.As[min(cur.row0 + wm * WM + i * 16 + l16, p.M - 1)];
                    const i32x4 iv = __builtin_bit_cast(i32x4, acc[i][j]);
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[i][j][q] = ((float)iv[q] * wv[q]) * xs;
                }
            }
        }
    };

    // ---- readiness (chained launches).  A producer counts a tile once every wave's h stores have completed:
    // each wave's vmcnt wait that covers them, then a barrier, then one atomic add by thread 0.  A consumer
    // wave polls the counter of the tile's M-tile (lane 0, agent-coherent load) before the tile's first DMA.
    auto SY = [&]() -> GmmSync { return chain_params()->sy; };  // (chained kernels only)
    // the counter of a tile's M-tile, from its context
    auto mti_ctx = [&](const Ctx &c) {
        return __builtin_amdgcn_readfirstlane(cls_base() + tile_prefix(c.e) + (c.row0 - row_off(c.e)) / GBM);
    };
    int sig = -1;      // producer: counter of the tile whose stores are still to be counted
    int gave_up = 0;   // consumer: a wait of this wave gave up (the launch's outputs are void; no more waits)
    auto signal = [&]() {
        if constexpr (PRODUCE) {
            if (sig >= 0 && first_thread)
                __hip_atomic_fetch_add(gptr(SY().ready + sig), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sig = -1;
        }
    };
    auto poll = [&](int m) -> int {
        int v = 0;
        if (lane == 0)
            v = __hip_atomic_load(gptr(SY().ready + m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_amdgcn_readfirstlane(v);
    };
    auto wait_ready = [&](int m) {
        if constexpr (CONSUME) {
            if (spect || gave_up)
                return;
            const uint64_t t0 = wall_clock64();
            while (poll(m) < SY().target) {
                if ((long long)(wall_clock64() - t0) > SY().ticks) {
                    if (lane == 0)
                        __hip_atomic_fetch_or(gptr(&g_cam_sync_status), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    gave_up = 1;
                    return;
                }
                __builtin_amdgcn_s_sleep(2);
            }
        }
    };
    // a queue's next ticket: thread 0 takes it and publishes it to the block through the epilogue's exchange area
    // (a second barrier when the epilogue that follows writes there)
    auto take = [&]() -> int {
        int t = 0;
        if constexpr (CONSUME || DYNL) {
            if (first_thread)
                t = tq.off + __hip_atomic_fetch_add(gptr(SY().ready + tq.ctr), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return t;
    };
    auto publish = [&](int t) -> int {
        if (first_thread)
            scratch[0] = t;
        lds_sync();
        t = __builtin_amdgcn_readfirstlane(scratch[0]);
        if constexpr (EPI != EPI_PLAIN)
            lds_sync();
        return t;
    };
    // the M-tile counter of a tile index (the expert search of setup, nothing else)
    auto mti_of = [&](int tile) {
        int lo = 0, hi = p.L - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (tile_end(mid - 1) * ntn <= tile)
                lo = mid;
            else
                hi = mid - 1;
        }
        const int e = __builtin_amdgcn_readfirstlane(lo);
        const int local = tile - tile_prefix(e) * ntn;
        constexpr int GM = 8;
        const int mt_e = tile_end(e) - tile_prefix(e);
        const int grp = local / (GM * ntn), rem = local % (GM * ntn);
        const int gm = min(GM, mt_e - grp * GM);
        return __builtin_amdgcn_readfirstlane(cls_base() + tile_prefix(e) + grp * GM + rem % gm);
    };

    if constexpr (BM >= 256) {
        // 256-row tile (8 waves of 128 x 64; fp8, bf16 or int8): half the L2->LDS bytes per FLOP of the 128-row
        // tile.  Its accumulators leave no room for a second register set, so: two LDS stages, the
        // W fragments of a k-step read once after the barrier, the A fragments streamed AHEAD rows
        // in front of the MFMAs that use them (the other wave on the SIMD covers the W read), the
        // next k-step's A bands issued during the first half of this k-step's MFMAs and the W bands
        // of the k-step after it from the middle on (a second barrier frees the W slot as soon as the
        // fragments are in registers).  Tiles do not overlap: each starts with its own first DMA and
        // drains at its end.  bf16 and int8 run the same loop with two chained K-half MFMAs per fragment pair
        // and no block scaling (measured against the generic two-stage loop, which waits for the whole ring
        // at every k-step: config 3's bf16 GEMMs 1.16 -> 1.27 PFLOPS, the int8 M-sweep's GMM1 +11%).
        static_assert(GSTAGES == 2, "two-stage ring");
        // A rows read ahead of their MFMAs (1, 2 or 3 measured within 1% of each other); the chained kernel
        // reads one row ahead, whose registers its scalar spill lanes need
        constexpr int AHEAD = ROLE == SYNC_NONE ? 2 : 1;
        // a tile's first DMAs: the W bands of k-step 0, its A bands and scales, then the W bands of k-step 1
        auto prime = [&](const Ctx &c) {
#pragma unroll
            for (int q = A_LOADS; q < A_LOADS + B_LOADS; ++q)
                dma_one(c, 0, 0, q, std::false_type{});
#pragma unroll
            for (int q = 0; q < LOADS; ++q)
                if (q < A_LOADS || q >= A_LOADS + B_LOADS)
                    dma_one(c, 0, 0, q, std::false_type{});
#pragma unroll
            for (int q = A_LOADS; q < A_LOADS + B_LOADS; ++q)
                dma_one(c, min(1, nk - 1), 1, q, std::false_type{});
        };
        int kt = 0, tile;
        if (dyn) {
            tk = publish(take());
            tile = min(ticket_tile(tk), total);
        } else {
            tile = seq(0);
        }
        Ctx c;
        CAM_TL_DECL
        if (tile < total) {
            setup(tile, c);
            wait_ready(mti_ctx(c));
            prime(c);
        }
        int next_ready = 0;  // consumer: the next tile's counter, polled while this tile's ring drains
        while (tile < total) {
            if constexpr (PRODUCE) {
                // the previous tile's h stores preceded this tile's first LOADS + B_LOADS DMAs (prime): once
                // no more than those are in flight in any wave, the stores have completed
                if (sig >= 0) {
                    wait_vmcnt<LOADS + B_LOADS>();
                    bar();
                    signal();
                }
            }
            clear_acc();
            f32x4 pend[JF];
            float ps[JF];
#pragma unroll
            for (int j = 0; j < JF; ++j) {
                pend[j] = f32x4{0.f, 0.f, 0.f, 0.f};
                ps[j] = 0.0f;
            }
            // one k-step; SL = ks & 1, the ring slot (a compile-time constant under CAM_GMM_UNROLL2, so that
            // every LDS address of the step is an immediate offset)
            auto kstep = [&](auto act, int ks, auto slc) {
                {
                    constexpr int SL0 = decltype(slc)::value;
                    const int SL = SL0 >= 0 ? SL0 : (ks & 1);
                    // k-step ks has landed (only the W bands of ks+1, issued last, may still be in flight);
                    // this wave's reads of k-step ks-1 are done
                    wait_vmcnt_lgkm0<B_LOADS>();
                    bar();  // ... for every wave: the A/scale slot (ks+1)%2 is free
                    const uint8_t *st = smem + SL * STAGE_BYTES;
                    const uint8_t *la = st + (wm * WM) * GKB;
                    const uint8_t *lb = st + A_BYTES + (wn * WN) * GKB;
                    i32x8 b[JF], a[IF];
                    float sa[IF];
                    auto rd_a = [&](int i) {
                        const u32x4 v0 = *reinterpret_cast<const u32x4 *>(la + swz(i * 16 + l16, lg));
                        const u32x4 v1 = *reinterpret_cast<const u32x4 *>(la + swz(i * 16 + l16, 4 + lg));
                        a[i] = i32x8{(int)v0[0], (int)v0[1], (int)v0[2], (int)v0[3],
                                     (int)v1[0], (int)v1[1], (int)v1[2], (int)v1[3]};
                    };
                    if constexpr (FP8)
                        rd_scales(st, sa);
#pragma unroll
                    for (int j = 0; j < JF; ++j) {
                        const u32x4 v0 = *reinterpret_cast<const u32x4 *>(lb + swz(j * 16 + l16, lg));
                        const u32x4 v1 = *reinterpret_cast<const u32x4 *>(lb + swz(j * 16 + l16, 4 + lg));
                        b[j] = i32x8{(int)v0[0], (int)v0[1], (int)v0[2], (int)v0[3],
                                     (int)v1[0], (int)v1[1], (int)v1[2], (int)v1[3]};
                    }
                    float sg = 0.0f, su = 0.0f;
                    if constexpr (FP8) {
                        sg = sload(c.wsb, c.wsg + ks);
                        su = SWIGLU ? sload(c.wsb, c.wsu + ks) : sg;
                    }
                    const int kn = min(ks + 1, nk - 1);  // past the end: reload the last k-step
#pragma unroll
                    for (int i = 0; i < AHEAD; ++i)
                        rd_a(i);
#pragma unroll
                    for (int i = 0; i < IF; ++i) {
                        // bf16: the rows stay in this order.  Left to itself the compiler moved reads and waits across
                        // them, another way in each build (W rows 4096 x 14336, 8 experts of 2000 rows: 1459 us with
                        // the rows held, 1527, 1543 and 1509 us in three builds without; 28672 x 4096: 2802 against
                        // 2829 to 2856 us; 4 experts of 4608 rows, K = 5248, N = 2304: 362 against 362 to 373 us)
                        if constexpr (DT == DT_BF16)
                            __builtin_amdgcn_sched_barrier(0);
                        if (i + AHEAD < IF)
                            rd_a(i + AHEAD);
                        const float sgi = FP8 ? sa[i] * sg : 0.0f, sui = FP8 ? sa[i] * su : 0.0f;
                        const int pi = i == 0 ? IF - 1 : i - 1;  // row of the pending results
#pragma unroll
                        for (int j = 0; j < JF; ++j) {
                            if constexpr (decltype(act)::value && !FP8) {
                                // bf16 / int8: the lane's two 16-byte chunks are the k-step's two K halves
                                // (32 bf16 or 64 int8 elements each); int8 accumulates exact int32 sums
                                const i32x4 b0 = {b[j][0], b[j][1], b[j][2], b[j][3]}, b1 = {b[j][4], b[j][5], b[j][6], b[j][7]};
                                const i32x4 a0 = {a[i][0], a[i][1], a[i][2], a[i][3]}, a1 = {a[i][4], a[i][5], a[i][6], a[i][7]};
                                if constexpr (INT8) {
                                    i32x4 t = __builtin_bit_cast(i32x4, acc[i][j]);
                                    t = __builtin_amdgcn_mfma_i32_16x16x64_i8(b0, a0, t, 0, 0, 0);
                                    t = __builtin_amdgcn_mfma_i32_16x16x64_i8(b1, a1, t, 0, 0, 0);
                                    acc[i][j] = __builtin_bit_cast(f32x4, t);
                                } else {
                                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                        __builtin_bit_cast(bf16x8, b0), __builtin_bit_cast(bf16x8, a0), acc[i][j], 0, 0, 0);
                                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                        __builtin_bit_cast(bf16x8, b1), __builtin_bit_cast(bf16x8, a1), acc[i][j], 0, 0, 0);
                                }
                            } else if constexpr (decltype(act)::value) {
                                const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                                const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b[j], a[i], z, 0,
                                                                                                 0, 0, 127, 0, 127);
#pragma unroll
                                for (int q = 0; q < 4; ++q)
                                    acc[pi][j][q] += pend[j][q] * ps[j];
                                pend[j] = d;
                                ps[j] = (SWIGLU && j >= JF / 2) ? sui : sgi;
                            }
                            // the A bands and scales of k-step ks+1 over the first half of the MFMAs; at the
                            // middle, when every wave has consumed its W fragments of ks, a barrier frees W
                            // slot ks%2 and the W bands of ks+2 go into it: the W stream runs 1.5 k-steps
                            // ahead in the same LDS.  All A/scale DMAs precede them (the wait above counts
                            // on the W bands being the last B_LOADS issued).
                            const int n = i * JF + j;
                            constexpr int HALF = IF * JF / 2, AS = LOADS - B_LOADS;
                            if (n < HALF) {
#pragma unroll
                                for (int u = n * AS / HALF; u < (n + 1) * AS / HALF; ++u)
                                    dma_one(c, kn, 1 - SL, u < A_LOADS ? u : u + B_LOADS, std::false_type{});
                            }
                            if (n == HALF) {
                                bar();
#pragma unroll
                                for (int q = A_LOADS; q < A_LOADS + B_LOADS; ++q)
                                    dma_one(c, min(ks + 2, nk - 1), SL, q, std::false_type{});
                            }
                            if constexpr (FP8) {
                                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
                                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // 4 VALU
                            } else {
                                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // 2 MFMA
                            }
                            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // a DMA, where one follows
                        }
                    }
                }
            };
            auto kloop = [&](auto act) {
#if CAM_GMM_UNROLL2
                int ks = 0;
                for (; ks + 1 < nk; ks += 2) {
                    kstep(act, ks, std::integral_constant<int, 0>{});
                    kstep(act, ks + 1, std::integral_constant<int, 1>{});
                }
                if (ks < nk)
                    kstep(act, ks, std::integral_constant<int, 0>{});
#else
                for (int ks = 0; ks < nk; ++ks)
                    kstep(act, ks, std::integral_constant<int, -1>{});
#endif
            };
            if (c.active)
                kloop(std::true_type{});
            else
                kloop(std::false_type{});
            if constexpr (FP8) {
#pragma unroll
                for (int j = 0; j < JF; ++j)  // the last row's pending results
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[IF - 1][j][q] += pend[j][q] * ps[j];
            }
            int ntile = 0;
            if (dyn) {
                // the queue's answer arrives while the ring drains; then the next tile's counter, answered
                // during the epilogue
                const int t = take();
                wait_vmcnt<0>();
                tk = publish(t);
                ntile = min(ticket_tile(tk), total);
                if (ntile < total && !gave_up)
                    next_ready = poll(mti_of(ntile));
            } else {
                if constexpr (CONSUME) {
                    ntile = seq(kt + 1);
                    if (ntile < total && !gave_up && !spect)
                        next_ready = poll(mti_of(ntile));  // answered while the ring drains
                }
                wait_vmcnt<0>();  // the tail's reload has landed before the next tile reuses the ring
                bar();
            }
            dequant_int8(c);
            epilogue(c);
            if constexpr (PRODUCE)
                sig = mti_ctx(c);
            CAM_TL_REC(c.e, tile);
            // int8: the dequantisation's loads have landed before the next tile (otherwise the compiler,
            // unsure of them, waits for every DMA in flight inside the k-loop)
            if constexpr (INT8)
                wait_vmcnt<0>();
            ++kt;
            tile = dyn ? ntile : seq(kt);
            if (tile < total) {
                setup(tile, c);
                if constexpr (CONSUME) {
                    if (next_ready < SY().target)
                        wait_ready(mti_ctx(c));
                }
                prime(c);
            }
        }
        if constexpr (PRODUCE) {
            wait_vmcnt<0>();
            bar();
            signal();
        }
        return tk;
    } else {
        // ---- 128/32-row tiles: software-pipelined k-loop over a ring of STAGES slots, continued
        // across the block's tiles.  Ring slots are indexed by the block's running k-step count kb+ks,
        // and the DMA of k-step ks+STAGES is spread over the MFMAs of k-step ks (or of its second
        // half); past the end of a tile it fetches the next tile's first k-steps, so a tile starts
        // with its operands already in flight.  With fewer k-steps than stages, or no next tile, the
        // past-the-end DMAs reload the tile's last k-step (the DMA count per k-step, and so every
        // vmcnt wait, stays uniform) and the ring is drained before the next tile.
        int kt = 0, tile;
        if constexpr (DYNL) {
            // Light tiles of the 8-wave chained kernel: taken from the queue only when the block is free, so that
            // no block ends a GEMM more than one light tile after the others.  The next tile's DMAs start between
            // this one's drained ring and its epilogue.
            if (tk < 0)
                tk = publish(take());
            tile = ticket_tile(tk);
        } else {
            tile = seq(0);
        }
        if (tile >= total)
            return tk;
        Ctx cur, nxt;
        setup(tile, cur);
        CAM_TL_DECL
        int kb = 0;          // the block's k-steps before the current tile
        bool primed = false;  // the current tile's first STAGES k-steps were issued by the previous tile
        int cur_ready = 0;    // consumer: the current tile's counter as polled before the previous tile's epilogue
        const bool can_chain = nk >= GSTAGES && (!(CONSUME && EAGER) || nk >= 2 * GSTAGES - 2);
        // A consumer of the 4-wave kernel chains into its next tile only when that tile's rows are ready: wave 0
        // copies the tile's counter into LDS by DMA at k-step edge nk - 2 STAGES + 2 (into the exchange area, which
        // the plain epilogue does not use), and every wave reads it at edge nk - STAGES, just before the first
        // past-the-end DMA.  (The 8-wave kernel cannot afford that branch in its k-loop; its light tiles do not
        // chain.)
        constexpr bool EAGER_C = CONSUME && EAGER;
        const int e_copy = nk - 2 * GSTAGES + 2, e_read = nk - GSTAGES;
        while (true) {
            int ntile = DYNL ? total : seq(++kt);
            bool has_next = ntile < total;
            // (int8 chains too: its dequantisation's vector loads then wait for the next tile's first DMAs,
            // which land meanwhile -- measured 8 us faster on the int8 decode step than draining first)
            int chain = has_next && can_chain;
            if (has_next)
                setup(ntile, nxt);
            else
                nxt = cur;
            auto slot = [&](int ks) { return (kb + ks) % GSTAGES; };
            auto stage_ptr = [&](int ks) { return smem + slot(ks) * STAGE_BYTES; };
            // DMA instruction q of the current tile's k-step ksx (ksx may run past the end: the next tile's first
            // k-steps go out under the current tile's cache policy)
            auto dma_ks = [&](int ksx, int q, auto nt) {
                // a uniform branch between two direct calls: selecting the context by reference would
                // place one of them in scratch memory, and every reload from there waits for the whole
                // DMA ring (vmcnt(0))
                if (ksx >= nk && chain)
                    dma_one(nxt, ksx - nk, slot(ksx), q, nt);
                else
                    dma_one(cur, min(ksx, nk - 1), slot(ksx), q, nt);
            };
            // the DMAs that follow MFMA n of NMF in a phase: spread evenly, so that a wave stalled on
            // a DMA issue still has MFMAs in the pipe
            auto dma_after = [&](int n, int nmf, int ksx, auto nt) {
#pragma unroll
                for (int q = n * LOADS / nmf; q < (n + 1) * LOADS / nmf; ++q)
                    dma_ks(ksx, q, nt);
            };
            auto by_policy = [&](auto f) {
                if constexpr (POL != W_BY_TILE)
                    f(std::bool_constant<POL == W_STREAM>{});
                else if (cur.nt)
                    f(std::true_type{});
                else
                    f(std::false_type{});
            };
            if (!primed) {
                if constexpr (CONSUME) {
                    if (cur_ready < SY().target)
                        wait_ready(mti_ctx(cur));
                }
                auto first = [&](auto nt) {
#pragma unroll
                    for (int s0 = 0; s0 < GSTAGES; ++s0)
#pragma unroll
                        for (int q = 0; q < LOADS; ++q)
                            dma_one(cur, min(s0, nk - 1), slot(s0), q, nt);
                };
                by_policy(first);
            }
            wait_vmcnt<LOADS *(GSTAGES - 1)>();  // k-step 0 has landed
            bar();
            // producer, unprimed tile: the previous tile's stores preceded these STAGES k-steps of DMAs
            if constexpr (PRODUCE) {
                if (!primed)
                    signal();
            }
            const bool poll_next = chain;  // EAGER consumer: decided inside the k-loop
            if constexpr (EAGER_C)
                chain = 0;
            clear_acc();
            // end of a k-step: k-step ks+1 has landed for every wave and every wave has read k-step ks
            int edge = 0;
            auto step_edge = [&]() {
                wait_vmcnt_lgkm0<LOADS *(GSTAGES - 2)>();
                bar();
                if constexpr (PRODUCE && EAGER) {
                    // edge STAGES-2: only LOADS (STAGES - 2) DMAs, all issued during this k-loop, may still be in
                    // flight in any wave, so the previous tile's h stores (issued before) have completed
                    if (edge == GSTAGES - 2)
                        signal();
                }
                if constexpr (EAGER_C) {
                    if (poll_next) {
                        // the copy issued at e_copy has landed by e_read: STAGES - 2 k-steps of DMAs came after it
                        if (edge == e_copy && w == 0)
                            dma4_sc1(SY().ready + mti_ctx(nxt), scratch);
                        if (edge == e_read)
                            chain = __builtin_amdgcn_readfirstlane(scratch[0]) >= SY().target;  // (bar(): read afresh)
                    }
                }
                if constexpr (EAGER)
                    ++edge;
            };

            if constexpr (FP8) {
                // One K=128 MFMA per fragment pair and k-step, and each is one scale block, so its result
                // is scaled on the VALU.  W fragments are double-buffered (but see ONE_W); A fragments are refilled row by
                // row right after the row's MFMAs have issued (one register set plus one W set in flight).
                // The scaling lags one fragment row behind (row i-1's results are scaled while row i's MFMAs
                // issue, 4 VALU : 1 MFMA), so the MFMA pipe never waits for a result it has just produced.
                // A lane's 32 K-bytes are the 16-byte chunks lg and 4+lg of the 128-byte row (not 2lg, 2lg+1):
                // the same K permutation in both operands leaves each block's dot products unchanged, and
                // this pattern reads LDS at twice the rate (no 2-way bank conflict).
                struct WRegs {
                    i32x8 b[JF];
                    float sg, su;  // weight scales of the wave's gate / up column blocks
                };
                i32x8 a[IF];
                float sa[IF];  // activation scales of the lane's rows
                f32x4 pend[JF];
                float ps[JF];
#pragma unroll
                for (int j = 0; j < JF; ++j) {
                    pend[j] = f32x4{0.f, 0.f, 0.f, 0.f};
                    ps[j] = 0.0f;
                }
                auto rd_w = [&](WRegs &r, int ks) {
                    const uint8_t *lb = stage_ptr(ks) + A_BYTES + (wn * WN) * GKB;
#pragma unroll
                    for (int j = 0; j < JF; ++j) {
                        const u32x4 v0 = *reinterpret_cast<const u32x4 *>(lb + swz(j * 16 + l16, lg));
                        const u32x4 v1 = *reinterpret_cast<const u32x4 *>(lb + swz(j * 16 + l16, 4 + lg));
                        r.b[j] = i32x8{(int)v0[0], (int)v0[1], (int)v0[2], (int)v0[3],
                                       (int)v1[0], (int)v1[1], (int)v1[2], (int)v1[3]};
                    }
                    const int kc = min(ks, nk - 1);
                    r.sg = sload(cur.wsb, cur.wsg + kc);
                    r.su = SWIGLU ? sload(cur.wsb, cur.wsu + kc) : r.sg;
                };
                auto rd_a = [&](int i, int ks) {
                    const uint8_t *st = stage_ptr(ks);
                    const uint8_t *la = st + (wm * WM) * GKB;
                    const u32x4 v0 = *reinterpret_cast<const u32x4 *>(la + swz(i * 16 + l16, lg));
                    const u32x4 v1 = *reinterpret_cast<const u32x4 *>(la + swz(i * 16 + l16, 4 + lg));
                    a[i] = i32x8{(int)v0[0], (int)v0[1], (int)v0[2], (int)v0[3],
                                 (int)v1[0], (int)v1[1], (int)v1[2], (int)v1[3]};
                    // with the last row: every row's scale of the k-step, read together (each row's scale
                    // product for the k-step before has been formed by then)
                    if (i == IF - 1)
                        rd_scales(st, sa);
                };
                // MFMAs of the k-step held in (a, wr); A rows of k-step ks_next are read behind them and
                // the DMA of k-step ks_next-1+STAGES is spread between them
                auto mm = [&](const WRegs &wr, int ks_next, auto act, auto nt) {
                    const int ks_dma = ks_next - 1 + GSTAGES;
#pragma unroll
                    for (int i = 0; i < IF; ++i) {
                        const float sgi = sa[i] * wr.sg, sui = sa[i] * wr.su;
                        const int pi = i == 0 ? IF - 1 : i - 1;  // row of the pending results
#pragma unroll
                        for (int j = 0; j < JF; ++j) {
                            if constexpr (decltype(act)::value) {
                                const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                                const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wr.b[j], a[i], z, 0,
                                                                                                 0, 0, 127, 0, 127);
#pragma unroll
                                for (int q = 0; q < 4; ++q)
                                    acc[pi][j][q] += pend[j][q] * ps[j];
                                pend[j] = d;
                                // in SwiGLU tiles a wave's columns j < JF/2 are gate rows, the rest up rows
                                ps[j] = (SWIGLU && j >= JF / 2) ? sui : sgi;
                            }
                            dma_after(i * JF + j, IF * JF, ks_dma, nt);
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
                            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // 4 VALU
                            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // a DMA, where one follows
                        }
                        rd_a(i, ks_next);
                    }
                };
                // (64-row tile: one W set, refilled behind the MFMAs that use it.  Beside 64 accumulators the second set
                // spilled, in the chained launch 19 registers that its 32-row loop reloaded too, and a weight stream
                // does not wait for those reads: the decode steps of 400 tokens, 64 experts, H = 2048, I = 1408 151 ->
                // 140 us, of 64 tokens, 32 of 256 experts and a shared one, H = 7168, I = 2048 249 -> 221 us)
                constexpr bool ONE_W = CLS == CLS_64;
                WRegs w0, w1;
#pragma unroll
                for (int i = 0; i < IF; ++i)
                    rd_a(i, 0);
                rd_w(w0, 0);
                auto kloop = [&](auto act, auto nt) {
                    int ks = 0;
                    if constexpr (ONE_W) {
                        for (; ks < nk; ++ks) {
                            step_edge();
                            mm(w0, ks + 1, act, nt);
                            rd_w(w0, ks + 1);
                        }
                        return;
                    }
                    for (; ks + 1 < nk; ks += 2) {
                        step_edge();
                        rd_w(w1, ks + 1);
                        mm(w0, ks + 1, act, nt);
                        step_edge();
                        rd_w(w0, ks + 2);
                        mm(w1, ks + 2, act, nt);
                    }
                    if (ks < nk) {
                        step_edge();
                        mm(w0, ks + 1, act, nt);
                    }
                };
                if (!spect && (TC::WAVES_M == 1 || cur.active))  // (one row-wave: a tile always has rows for it)
                    by_policy([&](auto nt) { kloop(std::true_type{}, nt); });
                else if constexpr (TC::WAVES_M > 1)
                    by_policy([&](auto nt) { kloop(std::false_type{}, nt); });
                else if constexpr (ROLE != SYNC_NONE)
                    kloop(std::false_type{}, std::false_type{});  // spectators issue no DMA
#pragma unroll
                for (int j = 0; j < JF; ++j)  // the last row's pending results
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[IF - 1][j][q] += pend[j][q] * ps[j];
            } else {
                // bf16 / int8: two phases per k-step (the K=32 / K=64 halves of the 128-byte step), each
                // phase's fragments read into the register set the previous phase is not using
                struct Regs {
                    i32x4 a[IF];
                    i32x4 b[JF];
                };
                auto rd = [&](Regs &f, int ks, int ph) {
                    const uint8_t *st = stage_ptr(ks);
                    const uint8_t *la = st + (wm * WM) * GKB;
                    const uint8_t *lb = st + A_BYTES + (wn * WN) * GKB;
#pragma unroll
                    for (int i = 0; i < IF; ++i)
                        f.a[i] = *reinterpret_cast<const i32x4 *>(la + swz(i * 16 + l16, ph * 4 + lg));
#pragma unroll
                    for (int j = 0; j < JF; ++j)
                        f.b[j] = *reinterpret_cast<const i32x4 *>(lb + swz(j * 16 + l16, ph * 4 + lg));
                };
                // MFMAs of one phase; with ks_dma >= 0 the DMA of that k-step is spread between them
                auto mm = [&](const Regs &f, int ks_dma, auto act, auto nt) {
#pragma unroll
                    for (int i = 0; i < IF; ++i)
#pragma unroll
                        for (int j = 0; j < JF; ++j) {
                            if (ks_dma >= 0)
                                dma_after(i * JF + j, IF * JF, ks_dma, nt);
                            if constexpr (!decltype(act)::value)
                                ;
                            else if constexpr (INT8)
                                acc[i][j] = __builtin_bit_cast(
                                    f32x4, __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                               f.b[j], f.a[i], __builtin_bit_cast(i32x4, acc[i][j]), 0, 0, 0));
                            else
                                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.b[j]),
                                                                                    __builtin_bit_cast(bf16x8, f.a[i]),
                                                                                    acc[i][j], 0, 0, 0);
                        }
                };
                Regs r0, r1;
                rd(r0, 0, 0);
                auto kloop = [&](auto act, auto nt) {
                    for (int ks = 0; ks < nk; ++ks) {
                        rd(r1, ks, 1);
                        mm(r0, -1, act, nt);
                        step_edge();
                        rd(r0, ks + 1, 0);
                        mm(r1, ks + GSTAGES, act, nt);
                    }
                };
                if (!spect && (TC::WAVES_M == 1 || cur.active))  // (one row-wave: a tile always has rows for it)
                    by_policy([&](auto nt) { kloop(std::true_type{}, nt); });
                else if constexpr (TC::WAVES_M > 1)
                    by_policy([&](auto nt) { kloop(std::false_type{}, nt); });
                else if constexpr (ROLE != SYNC_NONE)
                    kloop(std::false_type{}, std::false_type{});  // spectators issue no DMA
            }

            // producer, primed tile: the previous tile's stores are counted now -- the k-loop's last edge left
            // at most LOADS (STAGES - 2) DMAs in flight in every wave, all issued after those stores
            signal();
            dequant_int8(cur);
            if constexpr (DYNL) {
                const int t = take();
                wait_vmcnt<0>();  // the tail's reloads (and the ticket) have landed
                tk = publish(t);
                ntile = ticket_tile(tk);
                has_next = ntile < total;
                if (has_next) {
                    setup(ntile, nxt);
                    cur_ready = 0;
                    if constexpr (CONSUME)
                        cur_ready = spect ? 0 : poll(mti_ctx(nxt));
                    if (can_chain && (!CONSUME || cur_ready >= SY().target)) {
                        chain = 1;
#pragma unroll
                        for (int s0 = 0; s0 < GSTAGES; ++s0)
#pragma unroll
                            for (int q = 0; q < LOADS; ++q)
                                dma_one(nxt, s0, slot(nk + s0), q, std::bool_constant<POL == W_STREAM>{});
                    }
                }
            } else if (!chain) {
                if constexpr (CONSUME) {
                    if (has_next && !gave_up && !spect)
                        cur_ready = poll(mti_ctx(nxt));  // answered while the ring drains
                }
                wait_vmcnt<0>();  // the tail's reloads have landed before the next tile reuses the ring
                bar();
            }
            epilogue(cur);
            if constexpr (PRODUCE)
                sig = mti_ctx(cur);
            CAM_TL_REC(cur.e, tile);
            kb += nk;
            if (!has_next)
                break;
            primed = chain;
            tile = ntile;
            cur = nxt;
        }
        wait_vmcnt<0>();  // every DMA has landed before the block exits
        if constexpr (PRODUCE) {
            bar();
            signal();
        }
        return tk;
    }
}

__device__ __forceinline__ int blocks_for(int n)
{
    return __builtin_amdgcn_readfirstlane(plan_blocks(n, (int)gridDim.x));
}
// the block's first tile of a round-robin sequence over ge blocks that has given out n tiles before
__device__ __forceinline__ int continue_after(int n, int rank, int ge)
{
    if (n == 0 || rank >= ge)
        return rank;
    const int r = rank - n % ge;
    return __builtin_amdgcn_readfirstlane(r < 0 ? r + ge : r);
}
__device__ __forceinline__ int place_among(int g) { return plan_place((int)blockIdx.x, g, (int)gridDim.x); }

// LDS of a launch: a class's ring of stages, then that class's epilogue exchange area; the expert tables
// sit at the end of the launch's LDS (the same place for every class of a launch).
template <int BM, int BN = GBN> constexpr size_t ring_bytes() { return Tile<BM, BN>::STAGES * Tile<BM, BN>::STAGE_BYTES; }
template <int BM, int BN = GBN> constexpr size_t exchange_bytes()
{
    return (size_t)Tile<BM, BN>::WAVES_N * BM * sizeof(float);  // [WAVES_N][BM] row maxima
}
template <int BM, int BN = GBN> constexpr size_t class_bytes() { return ring_bytes<BM, BN>() + exchange_bytes<BM, BN>(); }
constexpr size_t cmax(size_t a, size_t b) { return a > b ? a : b; }
constexpr size_t G_LDS_SMALL_BYTES = cmax(cmax(class_bytes<32, GBN>(), class_bytes<32, 128>()),
                                          cmax(class_bytes<64, GBN>(), class_bytes<64, 128>())) + sizeof(GroupTables);
constexpr size_t G_LDS_BIG_BYTES =
    cmax(cmax(class_bytes<256>(), class_bytes<128>()), cmax(class_bytes<32, GBN>(), class_bytes<32, 128>())) +
    sizeof(GroupTables);
static_assert(G_LDS_SMALL_BYTES <= 163840 && G_LDS_BIG_BYTES <= 163840, "LDS budget of a gfx950 workgroup");
// the table scan's per-wave totals (before any ring use)
static_assert(sizeof(int) * (G_NCLASS + 1) * (GMAX_THREADS / 64) <= ring_bytes<32, 128>(), "table-scan scratch");

// Decode-sized segments (4 waves): 32-row tiles, and 64-row tiles for the experts of more rows (64 bf16 experts of 37
// rows on average, H = 2048, I = 1408: the decode step 245 us against 282 us with two 32-row tiles, each streaming the
// expert's weights).  fp8 and bf16 are bounded to two waves per SIMD although the LDS allows one: with up to
// 512 registers a wave the compiler keeps operands in accumulation registers and moves 24 to 64 of them per k-step (the
// int8 GMM2 alone measured faster that way, 76 against 78 us).
// Where the 64-row tiles do not save rounds of tiles, 32-row tiles run throughout (small_rows32; with no more of them than
// blocks they all run at once: 32 fp8 experts of 15 rows, K = 5888, two N-tiles each: GMM1 and GMM2 75 us against 78 us).
constexpr int G_ROWS32 = 32;
__device__ __forceinline__ ClassRanges small_ranges()
{
    return ClassRanges{{0, G_ROWS32 + 1, 1, 1}, {0, 0x7fffffff, 0x7fffffff, G_ROWS32 + 1}};
}
template <int DT, int EPI> __global__ __launch_bounds__(256, DT == DT_INT8 ? 1 : 2) void gmm_kernel_small(GmmArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    GroupTables *gt = reinterpret_cast<GroupTables *>(smem + G_LDS_SMALL_BYTES - sizeof(GroupTables));
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ntn = EPI != EPI_PLAIN ? p.N / 2 / 128 : p.N / small_bn(32, EPI);
    const ClassTiles mt = build_group_tables<Tile<32>::THREADS, 14, true>(p.group_list, p.L, *gt,
                                                                          reinterpret_cast<int *>(smem), small_ranges(), ntn);
    const int n64 = mt.n[CLS_128M] * ntn, n32 = mt.n[CLS_32] * ntn;
    // one round-robin sequence over both classes (a tile of either streams the same weight bytes)
    const int ge = blocks_for(n64 + n32), rank = place_among(ge);
    if (n64 > 0) {
        gmm_body<DT, EPI, CLS_64, SYNC_NONE, false, policy64(DT)>(p, gt, G_NOWHERE, rank, G_NOWHERE, ge, wv);
        lds_sync();
    }
    gmm_body<DT, EPI, CLS_32>(p, gt, G_NOWHERE, continue_after(n64, rank, ge), G_NOWHERE, ge, wv);
}

// Prefill: 8 waves, 128- or 256-row tile picked per launch from the actual rows per touched
// expert (counts are on the device).  The choice is block-uniform and identical in every block.
// Experts with at least this many rows take the 256-row tile (when the launch allows it).
constexpr int G_HEAVY_ROWS = 384;
// fp8 and bf16: the experts with fewer rows than this take the 32-row tile on four of the block's waves: their tiles
// are a weight stream, and that tile's four-stage ring keeps half as many weight bytes again in flight per CU as the
// 128-row tile's three stages (the int8 layer of 22 touched experts measured 390 us with them against 378 us and keeps
// the 128-row tile).  One 32-row tile per expert: two of them fetch its weights twice (48 fp8 experts of 36 to 281 rows:
// 255 us a pass at 33 rows, 272 us at 64).
#ifndef CAM_GMM_SMALL_ROWS
#define CAM_GMM_SMALL_ROWS 33
#endif
constexpr int G_SMALL_ROWS = CAM_GMM_SMALL_ROWS;

// Between two tile classes the block meets at an LDS-only barrier (lds_sync): both prefill loops have drained
// their DMAs before the last epilogue, so only the ring's LDS reads must be complete (__syncthreads would also
// wait for the epilogue's global stores; the next class's first DMAs queue behind those stores either way).
// Prefill: 8 waves.  With the 256-row tile allowed, the experts holding at least G_HEAVY_ROWS rows run 256-row tiles
// first, then the rest 128-row tiles and (fp8, bf16) those with fewer than G_SMALL_ROWS rows 32-row tiles, in one launch,
// the longest tiles first (big_schedule).  A layer whose load is skewed (a few experts with a thousand rows, many with a
// handful) gets tall tiles where they halve the operand traffic and short ones where a tall tile would multiply padding.
// short reductions keep the 128-row tile: the 256-row tile's per-tile ring fill and drain would
// not amortise over fewer than 16 k-steps (at 16, GMM2 of DeepSeek-V3's shapes: the M = 65536 fp8 GMM2
// 1.71 vs 1.57 PFLOPS, int8 1.97 vs 1.67 POPS, config 4's fp8 GMM2 116 vs 122 us)
__host__ __device__ constexpr bool big_tall(int allow256, int K, int dt)
{
    return allow256 && (int)((uint32_t)K * (dt == DT_BF16 ? 2 : 1) / GKB) >= CAM_GMM_MIN_NK256;
}
// int8: the experts of up to 32 rows are a class of 128-row tiles of their own, for the way it fetches weights (fp8 and bf16
// give them 32-row tiles)
template <int DT> __device__ __forceinline__ ClassRanges big_ranges(bool tall)
{
    constexpr int SMALL = DT == DT_INT8 ? 1 : G_SMALL_ROWS;  // rows below: the 32-row tile class
    const int top = tall ? G_HEAVY_ROWS : 0x7fffffff, small = tall ? SMALL : 1;
    const int multi = tall && DT == DT_INT8 ? G_SMALL_ROWS : small;
    return ClassRanges{{top, multi, small, 1}, {0x7fffffff, top, multi, small}};
}

// The 8-wave schedule of one GEMM over the tile classes of the launch's tables (gmm_kernel_big, gmm_chain_big): the
// 256-row tiles first, then the light ones (128-row, then 32-row).  ROLE != SYNC_NONE (the chained kernel): the
// 32-row class keeps the block's other four waves as spectators instead of ending them, since the block has more
// work after it.
template <int DT, int EPI, int ROLE>
__device__ __forceinline__ void big_schedule(const GmmArgs &p, const GroupTables *gt, int wv)
{
    const int G = gridDim.x, bid = blockIdx.x;
    const int pos = (G & 7) ? bid : (bid & 7) * (G >> 3) + (bid >> 3);  // XCD-aware order
    constexpr bool HAS32 = DT != DT_INT8;
    // tiles of each class (uniform values read from LDS go to scalar registers at once: a VGPR holding one across
    // the classes gets spilled, and its reload after a tile's k-loop makes the next k-loop wait for it at every
    // iteration)
    const int ntn = EPI != EPI_PLAIN ? p.N / 2 / 128 : p.N / 256, ntn32 = EPI != EPI_PLAIN ? ntn : p.N / small_bn(32, EPI);
    const int n0 = __builtin_amdgcn_readfirstlane(gt->template end<CLS_256>(p.L - 1)) * ntn;
    const int n1 = __builtin_amdgcn_readfirstlane(gt->template end<CLS_128M>(p.L - 1)) * ntn;
    const int n2 = __builtin_amdgcn_readfirstlane(gt->template end<CLS_128S>(p.L - 1)) * ntn;
    const int n3 = HAS32 ? __builtin_amdgcn_readfirstlane(gt->template end<CLS_32>(p.L - 1)) * ntn32 : 0;
    // A chained GEMM's light tiles: one queue over the two classes, longest tiles first.  (Tile times differ by a
    // factor of two with the load on the memory, so no static plan ends evenly: a layer of 22 touched experts, one of
    // 2311 rows, ended its GMM1 between 66 and 303 us under round-robin, against 175 us of work per block.)
    auto light_queue = [&](TileQueue q) {
        if constexpr (ROLE != SYNC_NONE) {
            q.end = n1;
            if (n1 > 0) {
                q.tk = gmm_body<DT, EPI, CLS_128M, ROLE>(p, gt, 0, 0, 0, 1, wv, q);
                lds_sync();
            }
            q.base = q.end, q.end += n3;
            if constexpr (HAS32) {
                if (n3 > 0)
                    gmm_body<DT, EPI, CLS_32, ROLE>(p, gt, 0, 0, 0, 1, wv, q);
            }
        }
    };
    if constexpr (ROLE == SYNC_CONSUME) {
        // Chained GMM2: the blocks reach it at different times (their GMM1 work differs), so the heavy tiles go
        // out through dynamic queues, one per XCD over that XCD's consecutive share (tiles sharing its L2), to
        // whichever of its blocks is free; the light tiles follow from one queue.
        if (n0 > 0) {
            const int nq = (G & 7) ? 1 : 8, x = nq == 1 ? 0 : (bid & 7);
            const int hx = (n0 + nq - 1) / nq;
            const int len = max(0, min(hx, n0 - x * hx));
            gmm_body<DT, EPI, CLS_256, ROLE>(p, gt, 0, 0, 0, 1, wv,
                                             TileQueue{chain_queue_index(p.M, p.L) + x, 0, 0, len, x * hx, -1});
            lds_sync();
        }
        TileQueue q{chain_light_index(p.M, p.L, true), 0, 0, 0, 0, -1};
        light_queue(q);
        return;
    }
    // The heavy tiles leave some of the ge blocks at work free (with one heavy tile fewer than the others): nfree of
    // them.  rank: this block's number among the free ones (is_free) or among the others, XCD by XCD.
    int ge = G;
    if (n0 == 0)
        ge = ROLE == SYNC_PRODUCE && n1 + n2 + n3 >= G ? G : blocks_for(n1 + n2 + n3);
    int nfree = ge, rank = place_among(ge);
    bool is_free = rank < ge;
    // Without light tiles to fill it, a last round of heavy tiles that would leave half of the blocks idle runs them as
    // two 128-row tiles each, which end after 0.6 to 0.7 of a heavy tile's time (a k-step alone on its CU: fp8 0.78
    // against 1.25 us, bf16 0.70 against 1.03 us; 128 heavy tiles alone, K = 7168: fp8 71 against 95 us, int8 62 against
    // 82 us, bf16 120 against 145 us; 640, K = 4096: 177 against 193, 158 against 167, 280 against 291 us).
    const int r = n0 < G ? n0 : n0 % G;
    const bool halve = ROLE == SYNC_NONE && r > 0 && 2 * r <= G && n1 + n2 + n3 == 0;
    int hs = pos, hn = halve ? n0 / G : G_NOWHERE;  // this block's heavy tiles
    if (!halve && n0 > 0 && n0 < G && (G & 7) == 0) {
        // Fewer heavy tiles than blocks.  They are split evenly over the 8 XCDs (XCD x takes the run
        // [x hx, (x + 1) hx), consecutive tiles sharing that XCD's L2), so each XCD keeps some blocks free.
        const int xcd = bid & 7, slot = bid >> 3, S = G >> 3;
        const int hx = (n0 + 7) / 8;
        auto heavy_in = [&](int x) { return max(0, min(hx, n0 - x * hx)); };
        const int len = heavy_in(xcd);
        hs = xcd * hx + slot;
        hn = slot < len ? 1 : 0;
        int free_before = 0, busy_before = 0;
        nfree = 0;
        for (int x = 0; x < 8; ++x) {
            const int h = heavy_in(x);
            free_before += x < xcd ? S - h : 0;
            busy_before += x < xcd ? h : 0;
            nfree += S - h;
        }
        is_free = slot >= len;
        rank = is_free ? free_before + slot - len : busy_before + slot;
    } else if (!halve && n0 > 0) {
        // At least as many heavy tiles as blocks: round-robin, so the first n0 % G blocks run one more than the rest
        nfree = G - r;
        is_free = pos >= r;
        rank = is_free ? pos - r : pos;
    }
    if (n0 > 0) {
        gmm_body<DT, EPI, CLS_256, ROLE>(p, gt, G_NOWHERE, hs, __builtin_amdgcn_readfirstlane(hn), G, wv);
        lds_sync();  // every wave is done with the first class's ring
    }
    if constexpr (ROLE == SYNC_PRODUCE) {
        // the light tiles through one queue; the free blocks start at their own place in it
        TileQueue q{chain_light_index(p.M, p.L, false), nfree, 0, 0, 0, is_free ? rank : -1};
        light_queue(q);
        return;
    }
    if constexpr (ROLE == SYNC_NONE) {
        // Static plan: layer by layer, each layer one light tile for every block of the group (the free blocks, the others)
        // that then ends first, counted in 20ths of a heavy tile's time.  A light tile's time against a heavy one's: 14/20 for
        // a 128-row tile (measured 73 against 105 us in GMM1, 24 against 34 us in GMM2; int8 66 against 95 us), 11/20 and
        // 5/20 for a 32-row tile with and without SwiGLU.  Within a group the tiles go round-robin, the sequence going on
        // from class to class.
        const int nbusy = ge - nfree, ng = is_free ? nfree : nbusy;
        int busy_end = 20, free_end = 0, at = 0;
        auto light = [&](int n, int cost, int &rs, int &rn) {
            int nf = 0, nb = 0, layers = 0, last = 0;  // tiles of the free blocks, of the others; this group's layers
            while (nf + nb < n) {
                const bool f = nfree > 0 && (nbusy == 0 || free_end <= busy_end);
                const int layer = min(n - nf - nb, f ? nfree : nbusy);
                nf += f ? layer : 0;
                nb += f ? 0 : layer;
                free_end += f ? cost : 0;
                busy_end += f ? 0 : cost;
                layers += f == is_free;
                last = f == is_free ? layer : last;
            }
            // (only a group's last layer can be partial)
            const int r = rank >= ng ? G_NOWHERE : rank >= at ? rank - at : rank - at + ng;
            rs = __builtin_amdgcn_readfirstlane((is_free ? 0 : nf) + r);
            rn = __builtin_amdgcn_readfirstlane(r < last ? layers : r < ng ? max(layers - 1, 0) : 0);
            at = __builtin_amdgcn_readfirstlane(at + last >= ng ? at + last - ng : at + last);
            free_end = __builtin_amdgcn_readfirstlane(free_end);
            busy_end = __builtin_amdgcn_readfirstlane(busy_end);
        };
        int rs, rn;
        if (halve) {
            gmm_body<DT, EPI, CLS_128M, ROLE, false, W_CACHED, true>(p, gt, G_NOWHERE, place_among(blocks_for(2 * r)), 1, G, wv,
                                                                     TileQueue{}, n0 - r);
            return;
        }
        if (n1 > 0) {
            light(n1, 14, rs, rn);
            gmm_body<DT, EPI, CLS_128M, ROLE>(p, gt, G_NOWHERE, rs, rn, ng, wv);
            lds_sync();
        }
        if constexpr (DT == DT_INT8) {
            if (n2 > 0) {
                light(n2, 14, rs, rn);
                gmm_body<DT, EPI, CLS_128S, ROLE>(p, gt, G_NOWHERE, rs, rn, ng, wv);
            }
        }
        if constexpr (HAS32) {
            if (n3 > 0) {
                light(n3, EPI == EPI_PLAIN ? 5 : 11, rs, rn);
                if (wv >= Tile<32>::NWAVES)
                    return;  // the 32-row tile's four waves go on (a barrier only counts the waves still running)
                gmm_body<DT, EPI, CLS_32, ROLE>(p, gt, G_NOWHERE, rs, rn, ng, wv);
            }
        }
    }
}

template <int DT, int EPI> __global__ __launch_bounds__(512, 1) void gmm_kernel_big(GmmArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    GroupTables *gt = reinterpret_cast<GroupTables *>(smem + G_LDS_BIG_BYTES - sizeof(GroupTables));
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const bool tall = big_tall(p.allow256, p.K, DT);
    // every class's expert table, from one read of the counts
    build_group_tables<GMAX_THREADS, DT == DT_INT8 ? 7 : 11>(p.group_list, p.L, *gt, reinterpret_cast<int *>(smem),
                                     big_ranges<DT>(tall));
    big_schedule<DT, EPI, SYNC_NONE>(p, gt, wv);
}

// Chained GMM1 + SwiGLU -> GMM2 (launch_gmm_chain): one table build, every block's GMM1 tiles (producing), then
// its GMM2 tiles (consuming).  A block only ever waits for GMM1 tiles, and every block runs all of its GMM1
// tiles before its first wait, so with every block resident each wait ends; a wait that outlasts the bound
// gives up instead (and the host reads the sync status).  The grid is one block per CU, the blocks' LDS keeps
// them to one per CU.
template <int DT, int EPI1> __global__ __launch_bounds__(512, 1) void gmm_chain_big(ChainParams cp)
{
    (void)cp;  // read through chain_params()
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    GroupTables *gt = reinterpret_cast<GroupTables *>(smem + G_LDS_BIG_BYTES - sizeof(GroupTables));
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    bool tall;
    {
        const GmmArgs p1 = chain_params()->g1;
        tall = big_tall(p1.allow256, p1.K, DT);  // the host checked that GMM2 makes the same choice
        build_group_tables<GMAX_THREADS, 11>(p1.group_list, p1.L, *gt, reinterpret_cast<int *>(smem),
                                         big_ranges<DT>(tall));
        big_schedule<DT, EPI1, SYNC_PRODUCE>(p1, gt, wv);
    }
    lds_sync();  // every wave is done with GMM1's last ring
    const GmmArgs p2 = chain_params()->g2;
    big_schedule<DT, EPI_PLAIN, SYNC_CONSUME>(p2, gt, wv);
}
template <int DT, int EPI1> __global__ __launch_bounds__(256, 2) void gmm_chain_small(ChainParams cp)
{
    (void)cp;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    GroupTables *gt = reinterpret_cast<GroupTables *>(smem + G_LDS_SMALL_BYTES - sizeof(GroupTables));
    // Decode tiles are weight streams of fixed size, so the two phases are balanced statically: GMM1's tiles go
    // round-robin over every block, GMM2's as plan_chain_gmm2 says.  A run's GMM2 tiles (the first experts) depend
    // only on GMM1's first rounds.
    const int G = gridDim.x;
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int t1, ge;
    ClassTiles mt;
    {
        const GmmArgs p1 = chain_params()->g1;
        const int ntn = p1.N / 2 / 128;
        mt = build_group_tables<Tile<32>::THREADS, 14, true>(p1.group_list, p1.L, *gt, reinterpret_cast<int *>(smem),
                                                             small_ranges(), ntn);
        const int n64 = mt.n[CLS_128M] * ntn, n32 = mt.n[CLS_32] * ntn;
        t1 = n64 + n32;
        ge = t1 < G ? blocks_for(t1) : G;  // (few tiles spread over the XCDs)
        const int rank = place_among(ge);
        if (n64 > 0) {
            gmm_body<DT, EPI1, CLS_64, SYNC_PRODUCE, true, policy64(DT)>(p1, gt, G_NOWHERE, rank, G_NOWHERE, ge, wv);
            lds_sync();
        }
        gmm_body<DT, EPI1, CLS_32, SYNC_PRODUCE, true>(p1, gt, G_NOWHERE, continue_after(n64, rank, ge), G_NOWHERE, ge, wv);
    }
    lds_sync();
    const GmmArgs p2 = chain_params()->g2;
    constexpr int BN2 = small_bn(32, EPI_PLAIN);
    const int m64 = mt.n[CLS_128M] * (p2.N / BN2), m32 = mt.n[CLS_32] * (p2.N / BN2);
    // the block's tiles of both classes in turn: the run [run, run + rn), then next, next + G, ...
    const ChainGmm2 g2 = plan_chain_gmm2((int)blockIdx.x, G, t1, ge, m64 + m32, GBN * chain_params()->g1.K, BN2 * p2.K);
    const int run = __builtin_amdgcn_readfirstlane(g2.run), rn = __builtin_amdgcn_readfirstlane(g2.rn);
    const int next = __builtin_amdgcn_readfirstlane(g2.next);
    if (m64 > 0) {
        gmm_body<DT, EPI_PLAIN, CLS_64, SYNC_CONSUME, true, policy64(DT)>(p2, gt, next, run, min(rn, max(m64 - run, 0)), 1, wv);
        lds_sync();
    }
    const int skip = max(m64 - run, 0), after = m64 > next ? (m64 - next + G - 1) / G : 0;
    gmm_body<DT, EPI_PLAIN, CLS_32, SYNC_CONSUME, true>(p2, gt, __builtin_amdgcn_readfirstlane(next + after * G - m64),
                                                        max(run - m64, 0), max(rn - skip, 0), 1, wv);
}

// Per-device launch state: the CU count and whether a kernel's dynamic-LDS limit has been raised.
// Both are cached per device in atomics, so concurrent first calls and several GPUs are safe (a
// racing first call only repeats the idempotent query or attribute set).
constexpr int G_MAX_DEVICES = 64;

static int current_device()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0)
        dev = 0;
    return dev;
}

static int num_cus(int dev)
{
    static std::atomic<int> cache[G_MAX_DEVICES];
    if (dev < G_MAX_DEVICES) {
        const int c = cache[dev].load(std::memory_order_relaxed);
        if (c > 0)
            return c;
    }
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        n = 256;
    if (dev < G_MAX_DEVICES)
        cache[dev].store(n, std::memory_order_relaxed);
    return n;
}

// one flag per device and kernel instantiation (the caller passes its own static array)
template <typename K> static hipError_t set_lds(K kernel, size_t lds, int dev, std::atomic<bool> *done)
{
    if (dev < G_MAX_DEVICES && done[dev].load(std::memory_order_acquire))
        return hipSuccess;
    hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess && dev < G_MAX_DEVICES)
        done[dev].store(true, std::memory_order_release);
    return e;
}

// Tile choice.  A row capacity of at most 48 rows per expert on average (decode): the 4-wave kernel, 32- and 64-row tiles.
// Otherwise the 8-wave kernel, which picks among 256-, 128- and 32-row tiles on the device from the actual counts (a
// prefill-sized capacity may still hold short segments when most rows are routed elsewhere).  One launch, no host
// synchronisation.
template <int DT, int EPI> static hipError_t launch_one(GmmArgs a, hipStream_t s)
{
    const int dev = current_device();
    const int grid = (num_cus(dev) + 7) / 8 * 8;
    if (a.M <= 48 * a.L) {
        static std::atomic<bool> done[G_MAX_DEVICES];
        const size_t lds = G_LDS_SMALL_BYTES;
        hipError_t e = set_lds(gmm_kernel_small<DT, EPI>, lds, dev, done);
        if (e != hipSuccess)
            return e;
        hipLaunchKernelGGL((gmm_kernel_small<DT, EPI>), dim3(grid), dim3(256), lds, s, a);
        return hipGetLastError();
    }
    a.allow256 = a.M >= G_HEAVY_ROWS;  // some expert may reach the 256-row tile class
    static std::atomic<bool> done[G_MAX_DEVICES];
    const size_t lds = G_LDS_BIG_BYTES;
    hipError_t e = set_lds(gmm_kernel_big<DT, EPI>, lds, dev, done);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL((gmm_kernel_big<DT, EPI>), dim3(grid), dim3(512), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_gmm(const GmmArgs &a, int dt, int epi, hipStream_t s)
{
    if (a.L <= 0 || a.L > G_MAX_L || a.M <= 0)
        return hipErrorInvalidValue;
    if (dt == DT_BF16) {
        if (epi == EPI_PLAIN)
            return launch_one<DT_BF16, EPI_PLAIN>(a, s);
        if (epi == EPI_SWIGLU_BF16)
            return launch_one<DT_BF16, EPI_SWIGLU_BF16>(a, s);
    } else if (dt == DT_INT8) {
        if (epi == EPI_PLAIN)
            return launch_one<DT_INT8, EPI_PLAIN>(a, s);
        if (epi == EPI_SWIGLU_F32AMAX)
            return launch_one<DT_INT8, EPI_SWIGLU_F32AMAX>(a, s);
    } else if (dt == DT_FP8) {
        if (epi == EPI_PLAIN)
            return launch_one<DT_FP8, EPI_PLAIN>(a, s);
        if (epi == EPI_SWIGLU_FP8)
            return launch_one<DT_FP8, EPI_SWIGLU_FP8>(a, s);
        if (epi == EPI_SWIGLU_BF16)
            return launch_one<DT_FP8, EPI_SWIGLU_BF16>(a, s);
    }
    return hipErrorInvalidValue;
}

// ---- chained GMM1 -> GMM2
#ifndef CAM_GMM_CHAIN_BIG
#define CAM_GMM_CHAIN_BIG 1  // the prefill-sized chained kernel (8 waves, all tile classes)
#endif
int gmm_chain_counters(int M, int L) { return chain_light_index(M, L, true) + 1; }

static bool chain_small(const GmmArgs &g) { return g.M <= 48 * g.L; }

// CAMHIP_GMM_CHAIN=0 in the environment turns the chained launch off (the two-launch path runs instead; for
// measuring one against the other)
static bool chain_enabled()
{
    static const bool on = [] {
        const char *v = getenv("CAMHIP_GMM_CHAIN");
        return !(v && v[0] == '0');
    }();
    return on;
}

// h above this size is not chained: the producing tiles store it agent-coherently (written through to
// memory), which for h of hundreds of MB (Mixtral-sized prefill) costs more than the overlap gains
constexpr long long G_CHAIN_MAX_H_BYTES = 64ll << 20;

bool gmm_chain_supported(const GmmArgs &g1, const GmmArgs &g2, int dt)
{
    if (dt != DT_FP8 && dt != DT_BF16)
        return false;  // int8 requantises h per token in a launch of its own
    if (!chain_enabled() || (long long)g1.M * (g1.N / 2) * (dt == DT_BF16 ? 2 : 1) > G_CHAIN_MAX_H_BYTES)
        return false;
    if (g1.M != g2.M || g1.L != g2.L || g1.group_list != g2.group_list || g2.K * 2 != g1.N)
        return false;
    if (chain_small(g1))
        return true;
#if !CAM_GMM_CHAIN_BIG
    return false;
#endif
    const int allow = g1.M >= G_HEAVY_ROWS;
    return big_tall(allow, g1.K, dt) == big_tall(allow, g2.K, dt);  // both GEMMs split every expert alike
}

static std::atomic<long long> g_sync_ticks{0};
static std::atomic<int> g_sync_unreach{0};
void sync_debug_set(long long wait_ticks, int unreachable)
{
    g_sync_ticks.store(wait_ticks, std::memory_order_relaxed);
    g_sync_unreach.store(unreachable ? 1 : 0, std::memory_order_relaxed);
}

hipError_t sync_status_read(int *status, bool clear)
{
    int v = 0;
    hipError_t e = hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_cam_sync_status), sizeof(int), 0, hipMemcpyDeviceToHost);
    if (e != hipSuccess)
        return e;
    if (clear && v != 0) {
        const int zero = 0;
        e = hipMemcpyToSymbol(HIP_SYMBOL(g_cam_sync_status), &zero, sizeof(int), 0, hipMemcpyHostToDevice);
        if (e != hipSuccess)
            return e;
    }
    *status = v;
    return hipSuccess;
}

template <int DT, int EPI1> static hipError_t launch_chain_t(GmmArgs g1, GmmArgs g2, GmmSync sy, hipStream_t s)
{
    const int dev = current_device();
    // one block per CU at most (a block's GMM2 tiles wait for GMM1 tiles of other blocks, so every block must be
    // resident at once), in whole XCD rounds where the CU count allows
    const int cus = num_cus(dev), grid = cus >= 8 ? cus / 8 * 8 : cus;
    if (chain_small(g1)) {
        static std::atomic<bool> done[G_MAX_DEVICES];
        hipError_t e = set_lds(gmm_chain_small<DT, EPI1>, G_LDS_SMALL_BYTES, dev, done);
        if (e != hipSuccess)
            return e;
        hipLaunchKernelGGL((gmm_chain_small<DT, EPI1>), dim3(grid), dim3(256), G_LDS_SMALL_BYTES, s, ChainParams{g1, g2, sy});
        return hipGetLastError();
    }
#if CAM_GMM_CHAIN_BIG
    g1.allow256 = g2.allow256 = g1.M >= G_HEAVY_ROWS;
    static std::atomic<bool> done[G_MAX_DEVICES];
    hipError_t e = set_lds(gmm_chain_big<DT, EPI1>, G_LDS_BIG_BYTES, dev, done);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL((gmm_chain_big<DT, EPI1>), dim3(grid), dim3(512), G_LDS_BIG_BYTES, s, ChainParams{g1, g2, sy});
    return hipGetLastError();
#else
    return hipErrorNotSupported;
#endif
}

hipError_t launch_gmm_chain(const GmmArgs &g1, const GmmArgs &g2, int dt, int *ready, hipStream_t s)
{
    if (g1.L <= 0 || g1.L > G_MAX_L || g1.M <= 0 || ready == nullptr)
        return hipErrorInvalidValue;
    if (!gmm_chain_supported(g1, g2, dt))
        return hipErrorNotSupported;
    const long long t = g_sync_ticks.load(std::memory_order_relaxed);
    const GmmSync sy{ready, g1.N / 2 / 128 + g_sync_unreach.load(std::memory_order_relaxed),
                     t > 0 ? t : 200000000LL};  // 2 s of the 100 MHz constant clock
    if (dt == DT_FP8)
        return launch_chain_t<DT_FP8, EPI_SWIGLU_FP8>(g1, g2, sy, s);
    return launch_chain_t<DT_BF16, EPI_SWIGLU_BF16>(g1, g2, sy, s);
}

#ifdef CAM_GMM_TIMELINE
}  // namespace cam
// diagnostic build only: copy the per-tile records out and clear them
extern "C" __attribute__((visibility("default"))) int camhipDebugGmmTimeline(void *host_dst, size_t bytes)
{
    const size_t n = std::min(bytes, sizeof(cam::g_cam_tl));
    if (hipMemcpyFromSymbol(host_dst, HIP_SYMBOL(cam::g_cam_tl), n, 0, hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    static uint8_t zeros[sizeof(cam::g_cam_tl)];
    return hipMemcpyToSymbol(HIP_SYMBOL(cam::g_cam_tl), zeros, sizeof(zeros), 0, hipMemcpyHostToDevice) == hipSuccess
               ? (int)(n / sizeof(cam::g_cam_tl[0]))
               : -1;
}
namespace cam {
#endif

// Per-token int8 requantisation of h (post_swiglu_dynamic_quant.h:164-231): one block per row.
__global__ __launch_bounds__(256) void quant_rows_int8_kernel(const float *__restrict__ h,
                                                              const float *__restrict__ amax_in,
                                                              const int64_t *__restrict__ group_list, int L, int M,
                                                              int I, int8_t *__restrict__ q, float *__restrict__ scale)
{
    __shared__ int tot;
    __shared__ float red[256 / 64];
    if (threadIdx.x == 0)
        tot = 0;
    __syncthreads();
    int part = 0;
    for (int e = threadIdx.x; e < L; e += blockDim.x)
        part += (int)group_list[e];
    if (part)
        atomicAdd(&tot, part);
    __syncthreads();
    const int total = min(tot, M);
    const int S = I / GMM_AMAX_COLS;  // partial maxima per row
    for (int m = blockIdx.x; m < total; m += gridDim.x) {
        float pm = 0.0f;
        for (int c = threadIdx.x; c < S; c += blockDim.x)
            pm = fmaxf(pm, amax_in[(size_t)m * S + c]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            pm = fmaxf(pm, __shfl_xor(pm, o, 64));
        if ((threadIdx.x & 63) == 0)
            red[threadIdx.x >> 6] = pm;
        __syncthreads();
        const float a = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        __syncthreads();  // red is rewritten for the next row
        const float inv = a > 0.0f ? 1.0f / a : 0.0f;  // rows of zeros quantise to 0 with scale 0
        const f32x4 *hr = reinterpret_cast<const f32x4 *>(h + (size_t)m * I);
        uint32_t *qr = reinterpret_cast<uint32_t *>(q + (size_t)m * I);
        for (int c = threadIdx.x; c < I / 4; c += blockDim.x) {
            const f32x4 v = hr[c];
            uint32_t pk = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b)
                pk |= (uint32_t)((int)rintf((v[b] * 127.0f) * inv) & 0xff) << (8 * b);
            qr[c] = pk;
        }
        if (threadIdx.x == 0)
            scale[m] = a * (1.0f / 127.0f);
    }
}

hipError_t launch_quant_rows_int8(const float *h, const float *amax, const int64_t *group_list, int L, int M, int I,
                                  int8_t *q, float *scale, hipStream_t s)
{
    if (M <= 0 || L <= 0 || (I % GMM_AMAX_COLS))
        return hipErrorInvalidValue;
    const int grid = M < 4096 ? M : 4096;
    hipLaunchKernelGGL(quant_rows_int8_kernel, dim3(grid), dim3(256), 0, s, h, amax, group_list, L, M, I, q, scale);
    return hipGetLastError();
}

// fp8 activation scales row-major [M, nb] -> k-major [nb, M] through an LDS tile: 64 rows x nb per block,
// read and written in contiguous runs
// One block per 64 x 64 tile of (rows, scale blocks): every load of the tile is issued at once (16 per
// thread, consecutive blocks of a row on consecutive lanes), the tile turns in LDS, and the stores run
// along the rows.  Rows at or past sum(group_list) are neither read nor written.
__global__ __launch_bounds__(256) void scales_kmajor_kernel(const float *__restrict__ src,
                                                          const int64_t *__restrict__ group_list, int L, int M,
                                                          int nb, float *__restrict__ dst)
{
    __shared__ float tile[64][65];
    __shared__ int tot;
    const int tid = threadIdx.x;
    if (tid < 64) {
        int part = 0;
#pragma unroll
        for (int q = 0; q < G_MAX_L / 64; ++q) {
            const int e = q * 64 + tid;
            part += e < L ? (int)group_list[e] : 0;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            part += __shfl_xor(part, o, 64);
        if (tid == 0)
            tot = part;
    }
    __syncthreads();
    const int rows = min(tot, M);
    const int r0 = blockIdx.x * 64, b0 = blockIdx.y * 64;
    if (r0 >= rows)
        return;
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int idx = i * 256 + tid, r = idx >> 6, b = idx & 63;
        v[i] = (r0 + r < rows && b0 + b < nb) ? src[(size_t)(r0 + r) * nb + b0 + b] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int idx = i * 256 + tid;
        tile[idx >> 6][idx & 63] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int idx = i * 256 + tid, b = idx >> 6, r = idx & 63;
        if (r0 + r < rows && b0 + b < nb)
            dst[(size_t)(b0 + b) * M + r0 + r] = tile[r][b];
    }
}

hipError_t launch_scales_to_kmajor(const float *src, const int64_t *group_list, int L, int M, int nb, float *dst,
                                   hipStream_t s)
{
    if (M < 0 || nb <= 0 || L <= 0 || L > G_MAX_L)
        return hipErrorInvalidValue;
    if (M == 0)
        return hipSuccess;
    hipLaunchKernelGGL(scales_kmajor_kernel, dim3((M + 63) / 64, (nb + 63) / 64), dim3(256), 0, s, src, group_list, L,
                       M, nb, dst);
    return hipGetLastError();
}

}  // namespace cam
