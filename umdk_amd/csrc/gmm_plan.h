// Which block of a decode GEMM launch (4 waves, gmm.hip) runs which tiles: plain integer rules, for the kernels and for
// host programs that check them.
#pragma once

#ifdef __HIPCC__
#define CAM_PLAN_FN __host__ __device__ __forceinline__
#else
#define CAM_PLAN_FN inline
#endif

namespace cam {

// 32-row tiles throughout (n32 of them), or 64-row tiles for the experts of more than 32 rows (n64 tiles of both
// heights, tall of them 64-row ones)?  Blocks run their tiles one after another, so what counts is rounds over the G
// blocks, and a round of 64-row tiles takes 1.25 to 1.35 times as long (the plain GEMM of 16 fp8 experts of 14 to 66 rows,
// K = 1024, N = 2304: 306 tiles, 198 tall, two rounds, 20.2 us, against 486 tiles, also two rounds, 15.5 us).  So 64-row
// tiles where the rounds they save make up for theirs (8 experts of 47 rows, H = 7168, I = 2048, four rounds to three in
// GMM2: int8 91 against 94 us, bf16 152 against 156 us; 64 fp8 experts of 24 rows on average, H = 1792, I = 4608, twelve to
// ten: 281 against 287 us), and where few are tall, which then only spare the memory (32 int8 experts of a few rows and a
// shared one of 128, H = 7168, I = 2048, three rounds either way: the decode step 264 against 272 us).
CAM_PLAN_FN bool small_rows32(int n32, int n64, int tall, int G)
{
    if (n32 <= G || tall == 0)
        return true;
    return 4 * tall > n64 && 4 * ((n64 + G - 1) / G) + (tall + G - 1) / G > 4 * ((n32 + G - 1) / G);
}

// Blocks that share n equal tiles in whole rounds: with R = ceil(n / G) rounds, only the first ceil(n / R) blocks
// (rounded up to whole XCDs) take tiles, R each at most, so a last partial round does not leave a few blocks streaming
// alone and a handful of tiles spreads over the XCDs.
CAM_PLAN_FN int plan_blocks(int n, int G)
{
    if (G & 7)
        return G;
    if (n > G) {  // (each division costs a kernel's start about 0.1 us)
        const int rounds = (n + G - 1) / G;
        n = (n + rounds - 1) / rounds;
    }
    n = (n + 7) & ~7;
    return n < 8 ? 8 : n < G ? n : G;
}
// The place of block b among the first g of G blocks, XCD by XCD; far past every tile for the others.  (Blocks b, b + 8,
// b + 16, ... run on the same XCD; with consecutive places they take consecutive tiles, which share that XCD's L2.)
constexpr int G_NOWHERE = 0x3fffffff;
CAM_PLAN_FN int plan_place(int b, int g, int G) { return (G & 7) ? b : b < g ? (b & 7) * (g >> 3) + (b >> 3) : G_NOWHERE; }

// The GMM2 tiles of block b in the chained decode launch (t1 GMM1 tiles, t2 GMM2 tiles): the run [run, run + rn), then
// next, next + G, ...  GMM1's tiles went round-robin over ge blocks (all G from t1 = G on), so the blocks without a tile
// of its last round, or without any, are free: they come first.  In a last round of several a free block has about one
// GMM1 tile's time, worth R GMM2 tiles (cost1 and cost2: the bytes of weights of a tile of either), but never more than
// spreads GMM2's tiles over the free blocks.  In an only round no GMM2 tile can start before the others end, so one tile
// each, then the other blocks in turn (64 tokens of 16 experts, H = 2304, I = 1024, 192 GMM1 tiles: the step 67 us fp8 and
// 91 us bf16, against 87 and 110 us with runs of 5 on the free blocks; one token through 2 of 8 bf16 experts, H = 1024:
// 16 GMM2 tiles on 16 blocks).
struct ChainGmm2 {
    int run, rn, next;
};
CAM_PLAN_FN ChainGmm2 plan_chain_gmm2(int b, int G, int t1, int ge, int t2, int cost1, int cost2)
{
    const int pos = plan_place(b, G, G);
    const bool one_round = t1 <= G;
    const int busy = ge < G ? ge : one_round ? t1 : t1 % G;  // blocks with a GMM1 tile in the last round
    const int nfree = busy > 0 ? G - busy : 0;
    const int mine = ge < G ? (b < ge ? plan_place(b, ge, G) : b) : pos;  // the busy blocks' places, then the free ones'
    const bool is_free = nfree > 0 && mine >= busy;
    int R = 1;
    if (!one_round) {
        R = (cost1 + cost2 / 2) / cost2;
        if (R > 1 && R * nfree > t2)
            R = (t2 + nfree - 1) / (nfree > 0 ? nfree : 1);
        R = R > 1 ? R : 1;
    }
    return {is_free ? (mine - busy) * R : 0, is_free ? R : 0, R * nfree + mine};
}

}  // namespace cam
