// The tile kernels of FusedQkv / MatMul for many input rows: out[m, n] = x[m, :] . W[n, :] as output tiles that one workgroup
// computes over the whole of k_dim (no partial sums to write, read and add), both operands moving from memory straight into LDS.
//
// What bounds them, and what follows from it:
//   * a chunk of a few hundred rows has few tiles, and its time is one workgroup's chain: with 64 x 64 tiles over 2048 features
//     32 steps of 16 KiB at the 110 KB/us that a CU draws from L2 would be 5 us. A step is 45 instructions per wave here: the
//     operands of step k + 1 go from LDS to registers between the products of step k, so no product waits for LDS; places in LDS
//     are constants of the loop that is unrolled over the stages; one barrier per step. (283 rows, 3072 x 2048 weights: 9.2 us
//     against 18.9 with the 128 x 128 split-K kernel and the launch that added its parts; 500 rows, 1152 x 896: 5.3 against 14.3.)
//   * the LDS loads of a wave are accepted one KiB every 20 cycles or so, and a wave waits meanwhile: issued in one go after the
//     barrier they leave the matrix cores idle. They are spread between the products (256 x 160: 98 -> 66 us at 2048 rows,
//     5120 x 3072, where the split-K form took 74.7).
//   * large launches read less per product with larger tiles but leave CUs idle where the tiles do not fill a round of
//     workgroups: six shapes, the choice by the rounds they need (choose_tile, fa_gemm.hip). 256 x 160 (F16) fills a round where
//     256 x 128 leaves a fifth of the chip to a second one - 8.4 to 10.5 million outputs, such as 2048 rows x 5120, and again at
//     twice that - and may hold rows of two matrices (JOINED), which lie anywhere: each request has the descriptor of its matrix (one
//     over all three matrices asked them to be within 4 GiB, and weights further apart took the 128 x 128 tiles: 2048 rows, 5120 x 3072
//     75 us where they now take 60 to 62 wherever they lie). 64 x 96 does so for a quarter to a half more outputs than 64 x 64 have
//     room for. (128 x 96: no faster than 128 x 128 with a third more workgroups, 22.0 us for 700 rows of 3072 x 3072.)
//   * block-quantised weights stay as they are up to the registers, where a wave turns its operands to f16 right in front of the
//     product (f16(weight * scale), as the reference's tile loader: see fa_gemm.hip). That is 14 vector instructions per 8
//     weights, and with one wave per SIMD they add to the chain; so that no two waves convert the same weights, the waves of a
//     tile share the features of a step instead of the input rows (KG) where the tile is small (283 rows, 3072 x 2048 Q8_0:
//     13.0 -> 9.7 us), and their sums meet in the write stage. The scales of the tile's rows are all in LDS from the start:
//     a request for 4 bytes of each row would cost the memory unit as much as one for 16 (15.4 -> 13.0 us).
//     With a workgroup or less per CU and 1024 features or more each wave takes the whole 64 x 64 tile for every fourth step, from
//     stages of its own (OWN): nothing is waited for but the wave's own requests, an operand is read from LDS once per tile and not
//     once per wave that shares it, and each weight is still converted once. A step is 0.13 to 0.16 us per CU instead of 0.20 (64 to
//     256 tiles): o_proj 200 rows, 2048 features x 1024 Q8_0 8.9 -> 8.2 us, Q4_0 9.4 -> 8.1; 3072 x 4096 13.4 -> 12.4, 13.9 -> 12.4;
//     FusedQkv 300 rows, 2560 x 2048 14.9 -> 13.9, 14.8 -> 13.3. Below 1024 features what it adds - the first steps of four waves
//     arrive together, four partial tiles meet in the write stage - outweighs that (896: Q8_0 6.4 -> 6.8), above 4096 the scales
//     leave room for two stages (5120: 17.8 -> 20.0). Steps of 32 features and eight waves: 5 to 10 % slower (half lines per request).
//     With a workgroup for half of the compute units or fewer, the tiles are of 32 weight rows, each wave with a quarter of every
//     step: half the weights to convert and half the products in the chain. (Against 64 x 64: o_proj 500 rows, 896 features x 896 Q8_0
//     6.2 -> 5.6 us, Q4_0 6.3 -> 5.6; 190 rows, 2048 x 2048 9.1 -> 8.2, 8.7 -> 8.3; FusedQkv 130 rows, 2560 x 2048 12.2 -> 11.1, 12.2 ->
//     11.3. 32 input rows x 64 instead: the last 11.7 and 11.9, o_proj of 2048 features up to 6 % slower than 64 x 64 with Q4_0.)
//   * a 32 x 32 x 16 matrix instruction rounds its running sum twice, so a chain's error grows with the root of its length: over 3072
//     features 5.9 x 2^-24 of the sums' size. F16 tiles of up to 128 x 128, which took the place of parts of a few hundred features
//     added in a second launch (2.2 x 2^-24), add their accumulators to a second set every FOLD steps, between the products, for
//     0.5 to 1 % of the time: 2.1 to 2.2 x 2^-24 (1.9 over 896 features, 3.3 in one chain). The larger tiles have no registers for
//     that, and the launches that they took over had one chain as well. Block-quantised weights are rounded to f16 with their scale,
//     2^-12 of each operand, beside which a chain's error is small (1000 x 2^-24 of the sums' size with either). Their waves have
//     SETS of accumulators that a wave's products go to in turn, so that a sum is KG * SETS chains and no launch is less exact than
//     where it was before it came to these tiles (the 128 x 64 tiles' four chains for 64 x 96, the panel kernel's eight for a chunk
//     with a norm). Q8_0, one set and two, x 2^-24: 340 rows, 3072 x 3072 3.5 -> 2.4; 200 rows, 2048 x 2048 2.0 -> 1.6; FusedQkv
//     100 rows, 2112 x 1280 1.7 -> 1.4, 416 rows, 3072 x 896 1.7 -> 1.4 (on the panel kernel 1.5, 1.45). Q4_0's products are of
//     fewer bits: two sets where KG is 2 (1.1 to 1.8). It costs 1 % of the launches with Q8_0 weights in the mean over 74 of them, up to
//     0.5 us where 64 accumulators more are cleared and added up (577 rows, 1600 x 1536 9.1 -> 9.6), 0.2 % with Q4_0; adding a
//     second set up every few steps instead costs 5 to 9 %. The larger tiles took no launch from a kernel of more chains, and 128 x 64
//     and 128 x 128 tiles would be 1 to 2 % slower with two sets.
// F16 sums run over the features in order, whatever the tile: the shapes up to 128 x 128, and the register-staged kernel, agree to
// the bit.
#pragma once
#include "fa_gemm.h"
#include "fa_lds_dma.h"
#include "fa_norm.h"
#include <atomic>
#include <numeric>
#include <type_traits>

namespace fa_tile {

using namespace fa_gemm;
typedef uint32_t u2v_t __attribute__((ext_vector_type(2)));

// LDS layouts. The 64 lanes of a request fill one KiB of consecutive LDS bytes in lane order, so padding is impossible; instead a
// KiB holds a whole number of rows, and a lane fetches, within its row, the 16-byte piece that belongs into its slot:
//   input, row-major F16 weights   8 rows x 8 pieces,   slot = piece ^ (row / 2) % 8
//   canonical F16, row-major Q8_0  16 rows x 4 pieces,  slot = piece ^ (row / 4) % 4
//   canonical Q8_0                 32 rows x 2 pieces,  slot = piece ^ (row / 8) % 2
//   Q4_0                           64 rows x 1 piece or 32 x 2, in order
// so that the lanes of an operand read fall into different banks while the lanes of a request cover whole runs of memory. Rows
// past the end of a matrix (or of the input) are outside the buffer descriptor, or other rows of it: what they give is not stored.
//
// WB bits per weight; WM x WN waves over (input rows, weight rows), each of them KG times, for a share of every 64 features; a wave
// owns TM x TN tiles of 32 x 32; NS stages of 64 features.
template <int WB_, bool CANON_, int WM_, int WN_, int KG_, int TM_, int TN_, int NS_, bool JOINED_ = false, bool OWN_ = false>
struct Shape {
    static constexpr int WB = WB_, WM = WM_, WN = WN_, KG = KG_, TM = TM_, TN = TN_, NS = NS_;
    static constexpr bool CANON = CANON_, QUANT = WB_ != 16;
    // The tiles run over the rows of all matrices as one list (F16; whole groups of 32 rows per matrix): a tile may hold rows of two.
    static constexpr bool JOINED = JOINED_;
    static_assert(!JOINED || WB == 16, "F16 only");
    // Each wave has the whole tile, stages of its own and every KG-th step: no wave waits for another before the write stage.
    static constexpr bool OWN = OWN_;
    static_assert(!OWN || (QUANT && WM == 1 && WN == 1 && KG == 4), "16 bytes of a row's scales are those of a step of each wave");
    static constexpr int FOLD = WB_ == 16 && WM_ * TM_ * WN_ * TN_ <= 16 ? 4 : 0;  // steps, 0: one chain
    // Sets of accumulators that a wave's products go to in turn (block-quantised tiles of up to 64 x 96)
    static constexpr int SETS = QUANT && WM_ * TM_ * WN_ * TN_ <= 6 && (WB_ == 8 || KG_ == 2) ? 2 : 1;
    static constexpr int NW = WM * WN * KG, NT = NW * 64, KN = OWN ? 4 : 4 / KG, LOADERS = OWN ? 1 : NW;  // KN: products of 16 features per wave and stage
    static constexpr int MT = WM * TM * 32, NTR = WN * TN * 32;         // input rows and weight rows of the tile
    static constexpr int X_BYTES = MT * 128, W_BYTES = NTR * 8 * WB, STAGE = X_BYTES + W_BYTES;
    // 1 KiB requests of a stage, and per wave (where they do not divide, some are made twice)
    static constexpr int X_REQ = X_BYTES / 1024, XR = (X_REQ + LOADERS - 1) / LOADERS;
    static constexpr bool X_EVEN = X_REQ % LOADERS == 0;
    static constexpr int W_REQ = W_BYTES / 1024, WR = (W_REQ + LOADERS - 1) / LOADERS;
    static constexpr int REQ = XR + WR, ALL_STAGES = (OWN ? NW : 1) * NS * STAGE;
    // what a lane reads of a weight row at a time: the 8 features of a product, of both halves of the wave where they are 4 bytes
    typedef typename std::conditional<WB_ == 16, h8_t, u2v_t>::type raw_t;
    static constexpr int READS = KN * (TM + TN);
    // 32-row groups of every wave that the write stage turns at a time: all of them where the LDS of the stages holds them (a barrier
    // and a turn less; F16 128 x 64, o_proj 1000 rows, 2048 x 2048: 16.4 -> 15.2 us; the other tiles within 1 %), else one.
    static constexpr int T_STRIDE = NTR * 4 + 16, TJ = KG * WM * TM * 32 * T_STRIDE <= ALL_STAGES || OWN || NTR < 64 ? TM : 1;
    static constexpr int T_BYTES = WM * TJ * 32 * T_STRIDE;
    // LDS: the stages, then (block-quantised) all scales of the tile's rows, [8 blocks][row]; the write stage over both
    static constexpr uint32_t scale_bytes(uint32_t k_dim) { return QUANT ? NTR % 64 == 0 ? (k_dim + 255) / 256 * (NTR * 16) : ((k_dim + 255) / 256 * (NTR * 16) + 1023) & ~1023u : 0u; }
    static constexpr uint32_t lds_bytes(uint32_t k_dim) {
        const uint32_t s = ALL_STAGES + scale_bytes(k_dim);
        return s > (uint32_t)(KG * T_BYTES) ? s : (uint32_t)(KG * T_BYTES);
    }
    static_assert(X_BYTES % 1024 == 0 && W_BYTES % 1024 == 0, "whole requests");
    static_assert(!JOINED || (X_EVEN && W_REQ % LOADERS == 0), "a wave's requests fill one run of LDS");
    static_assert(lds_bytes(0) <= 160 * 1024 && REQ * (NS - 1) <= 63, "LDS of a compute unit; the request counter");
};

// input rows x weight rows (the first three: block-quantised; with stages of each wave's own, with more stages)
enum TileShape { TILE_64x32, TILE_64x64_OWN, TILE_64x64_DEEP, TILE_64x64, TILE_64x96, TILE_128x64, TILE_128x128, TILE_256x128, TILE_256x160 };

template <int N>
__device__ __forceinline__ void wait_requests() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Workgroup barrier behind which this wave's LDS reads have arrived. (The wait is the builtin and not assembly: the compiler has to
// know that no read is outstanding, or it waits again, behind the reads of the next step.)
__device__ __forceinline__ void meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// What the write stage does: alpha * sum + bias + beta * residual; KvPrepFused's, pairs in a piece (or no rotation) and half a head apart.
// ANY: a kernel has all three and the launch says which. A tile with stages of its own has a kernel for each: 33 KB of code, of which a
// launch runs through the loop and one part far from it, became 19 to 23 KB that it runs through in a row (Q4_0, FusedQkv + KvPrepFused of
// 400 rows x 2560 x 2048 19.1 -> 18.5 us, o_proj of 400 rows x 3072 x 3072 15.8 -> 15.4, 700 rows x 2048 x 2048 13.3 -> 13.0), and so have the
// block-quantised tiles of eight stages, whose loops have no scalar registers left (o_proj of 128 rows x 3072 x 3072 Q8_0 11.4 -> 10.8, Q4_0 11.0 -> 10.8)
// and 256 x 160 (0.5 %; the other tiles within 1 %).
enum Form { PLAIN, ADJACENT, APART, ANY };
template <class S, int MIN_WAVES, Form FORM>
__global__ void __launch_bounds__(S::NT, MIN_WAVES) tile_gemm_kernel(GemmDev a) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    typedef __attribute__((address_space(3))) void *lds_ptr;
    // A workgroup has nothing else to do before its first request, so the way there is time of the launch: the arguments it takes are
    // asked for at once, and its tile is found without a division (before: six trips to them and two divisions; FusedQkv + KvPrepFused of
    // 128 rows x 2560 x 2048 Q8_0 12.3 -> 11.8 us, o_proj of 500 rows x 896 x 896 6.4 -> 6.0, of 128 rows x 3072 x 3072 10.9 -> 10.4).
    asm volatile("" ::"s"(a.k_dim), "s"(a.m), "s"(a.m_tiles), "s"(a.n_tiles), "s"(a.panel_inv), "s"(a.tiles[0]), "s"(a.tiles[1]), "s"(a.rows[0]), "s"(a.rows[1]), "s"(a.x), "s"(a.w[0]),
                 "s"(a.w[1]), "s"(a.w[2]));
    if constexpr (S::QUANT) asm volatile("" ::"s"(a.scales[0]), "s"(a.scales[1]), "s"(a.scales[2]));
    if constexpr (FORM != PLAIN) asm volatile("" ::"s"(a.rope.on), "s"(a.rope.apply), "s"(a.rope.normal), "s"(a.rope.head_dim));
    if constexpr (FORM == PLAIN || FORM == ANY) asm volatile("" ::"s"(a.residual));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int loader = S::OWN ? 0 : wave;  // which of the requests of a step are this wave's
    const uint32_t own = S::OWN ? wave * (S::NS * S::STAGE) : 0;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr)smem + own;
    const int wn = wave % S::WN, wm = wave / S::WN % S::WM, kg = wave / (S::WN * S::WM);
    const uint32_t K = a.k_dim, n_steps = S::OWN ? (K / 64 + 3 - wave) / 4 : K / 64;  // (this wave's)

    // Tile of this workgroup. Workgroup ids go round the 8 XCDs; the ids of one XCD are given consecutive tiles (weight rows
    // outermost), so that a weight tile is fetched into one L2 only.
    const uint32_t total = a.n_tiles * a.m_tiles, per_xcd = (total + 7) >> 3;
    const uint32_t v = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    if (v >= total) return;
    uint32_t nt, mt;
    {
        const uint32_t G = a.m_tiles > 8 ? 4u : 1u;  // (of many input rows, the tiles at work together in an XCD are 8 x 4, not 16 x 2)
        const uint32_t panel = fa_quotient(v, G * a.m_tiles, a.panel_inv), rem = v - panel * G * a.m_tiles, w = min(G, a.n_tiles - panel * G);
        mt = w == 3 ? __umulhi(rem, 0x55555556u) : rem >> (w >> 1), nt = panel * G + rem - mt * w;
    }
    int tile_mat = 0;
    if (!S::JOINED && nt >= a.tiles[0]) {
        nt -= a.tiles[0], tile_mat = 1;
        if (nt >= a.tiles[1]) nt -= a.tiles[1], tile_mat = 2;
    }
    auto pick3 = [](int mat, auto x0, auto x1, auto x2) { return mat == 0 ? x0 : mat == 1 ? x1 : x2; };
    const uint32_t rows0 = a.rows[0], rows1 = a.rows[1], n0 = nt * S::NTR, m0 = mt * S::MT;
    const uint32_t N_tile = tile_mat == 0 ? rows0 : rows1;

    // Matrix and weight row of tile row t. With the NeoX rotation as the write stage, 32 tile rows are 16 rows of a head and the 16
    // that they are rotated with, half a head further on, so that a tile of any width holds both of a pair.
    const bool pairs = FORM == ANY ? a.rope.on && a.rope.apply && !a.rope.normal : FORM == APART;
    const uint32_t hd_shift = a.rope.head_dim == 128 ? 7u : 6u;
    auto paired = [&](uint32_t r) -> uint32_t {
        if (!pairs) return r;
        const uint32_t g = r >> 5, head = g >> (hd_shift - 5), within = g & ((1u << (hd_shift - 5)) - 1u);
        return (head << hd_shift) + within * 16 + (r & 15u) + ((r & 16u) ? 1u << (hd_shift - 1) : 0u);
    };
    auto matrix_of = [&](uint32_t &r) -> int {  // r: row of the list -> row of its matrix
        int mat = tile_mat;
        if (S::JOINED && r >= rows0) {
            r -= rows0, mat = 1;
            if (r >= rows1) r -= rows1, mat = 2;
        }
        return mat;
    };
    auto weight_row = [&](uint32_t t) -> uint32_t { return paired(n0 + t); };  // (not JOINED)

    // Requests of this wave. Input: KiB q = rows 8q .. + 7 of 128 bytes, slot = piece ^ (row / 2) % 8.
    int xv[S::XR], wv[S::WR];
#pragma unroll
    for (int i = 0; i < S::XR; ++i) {
        const uint32_t row = (S::X_EVEN ? loader * S::XR + i : (loader * S::XR + i) % S::X_REQ) * 8 + (lane >> 3);
        xv[i] = (int)(row * K * 2 + ((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    uint32_t w_block[S::WR];  // canonical: which of the stage's two 32-feature blocks
#pragma unroll
    for (int i = 0; i < S::WR; ++i) {
        const uint32_t q = (loader * S::WR + i) % S::W_REQ;
        w_block[i] = 0;
        if constexpr (S::CANON) {
            constexpr uint32_t PER_BLOCK = S::W_REQ > 1 ? S::W_REQ / 2 : 1;
            const uint32_t u = q % PER_BLOCK;
            w_block[i] = q / PER_BLOCK;
            if constexpr (S::WB == 16) {
                const uint32_t row = u * 16 + (lane >> 2);
                wv[i] = (int)(weight_row(row) * 64 + ((lane & 3) ^ ((row >> 2) & 3)) * 16);
            } else if constexpr (S::WB == 8) {
                const uint32_t row = u * 32 + (lane >> 1);
                wv[i] = (int)(weight_row(row) * 32 + ((lane & 1) ^ ((row >> 3) & 1)) * 16);
            } else {
                if constexpr (S::NTR % 64 == 0) {
                    wv[i] = (int)(weight_row(u * 64 + lane) * 16);
                } else {  // a block of the tile's rows is not whole KiB: the lanes of a request go over both
                    const uint32_t at = q * 64 + lane;
                    wv[i] = (int)(weight_row(at % S::NTR) * 16 + at / S::NTR * (N_tile * 16));
                    w_block[i] = 0;
                }
            }
        } else {
            if constexpr (S::WB == 16) {
                const uint32_t row = q * 8 + (lane >> 3);
                wv[i] = (int)(weight_row(row) * K * 2 + ((lane & 7) ^ ((row >> 1) & 7)) * 16);
            } else if constexpr (S::WB == 8) {
                const uint32_t row = q * 16 + (lane >> 2);
                wv[i] = (int)(weight_row(row) * K + ((lane & 3) ^ ((row >> 2) & 3)) * 16);
            } else {
                const uint32_t row = q * 32 + (lane >> 1);
                wv[i] = (int)(weight_row(row) * (K / 2) + (lane & 1) * 16);
            }
        }
    }
    const fa_lds_dma::rsrc_words x_rs = fa_lds_dma::make_rsrc_words(reinterpret_cast<const unsigned char *>(a.x) + (size_t)m0 * K * 2, (a.m - m0) * K * 2);
    const uint32_t w_block_bytes = N_tile * 4 * S::WB;  // canonical: one 32-feature block of the matrix
    uint32_t w_step[S::WR];                             // JOINED: bytes between the steps of a request's matrix
    fa_lds_dma::rsrc_words w_rs = {}, w_joined[S::WR];     // (JOINED: of each request's matrix, as a wave's requests may be of two)
    uint32_t w_bytes[S::WR];
    if constexpr (S::JOINED) {
#pragma unroll
        for (int i = 0; i < S::WR; ++i) {
            const uint32_t q = wave * S::WR + i, u = S::CANON ? q % (S::W_REQ / 2) : q;
            const uint32_t row = S::CANON ? u * 16 + (lane >> 2) : u * 8 + (lane >> 3);  // of the tile
            uint32_t r = min(n0 + (S::CANON ? u * 16 : u * 8), rows0 + 2 * rows1 - (S::CANON ? 16 : 8));  // (rows past the end: the last ones again)
            const int mat = matrix_of(r);
            const uint32_t wr = paired(r + (S::CANON ? lane >> 2 : lane >> 3)), rows = mat ? rows1 : rows0;
            w_bytes[i] = rows * K * 2, w_joined[i] = fa_lds_dma::make_rsrc_words(pick3(mat, a.w[0], a.w[1], a.w[2]), w_bytes[i]);
            if constexpr (S::CANON)
                wv[i] = (int)(w_block[i] * rows * 64 + wr * 64 + ((lane & 3) ^ ((row >> 2) & 3)) * 16), w_step[i] = rows * 128;
            else
                wv[i] = (int)(wr * K * 2 + ((lane & 7) ^ ((row >> 1) & 7)) * 16), w_step[i] = 128;
        }
    } else {
        w_rs = fa_lds_dma::make_rsrc_words(pick3(tile_mat, a.w[0], a.w[1], a.w[2]), N_tile * (K / 8 * S::WB));
    }
    // What the next step's requests start from: byte offsets that grow by the same amount per step. (Past the last step the
    // descriptors are made empty: nothing is read, zeros arrive, and the counts that the waits go by stay the same.)
    constexpr uint32_t STRIDE = S::OWN ? 4 : 1;  // steps between two of this wave's
    const uint32_t w_per_step = S::CANON ? 2 * w_block_bytes : 8 * S::WB;
    uint32_t asked = 0, x_soff = S::OWN ? wave * 128 : 0, w_soff = S::OWN ? wave * w_per_step : 0;
    fa_lds_dma::rsrc_words x_now = x_rs, w_now = w_rs;
    if (S::OWN && n_steps == 0) x_now.z = 0u, w_now.z = 0u;
    const uint32_t x_lds = lds_base + loader * S::XR * 1024, w_lds = lds_base + S::X_BYTES + loader * S::WR * 1024;  // (JOINED)
    auto request = [&](int r, uint32_t stage) __attribute__((always_inline)) {
        const uint32_t base = lds_base + stage;
        if (r < S::WR) {
            const uint32_t q = (loader * S::WR + r) % S::W_REQ;
            if constexpr (S::JOINED) {
                fa_lds_dma::buffer_to_lds_b128_ahead(w_joined[r], w_lds, stage + r * 1024, wv[r], 0);
                wv[r] += w_step[r];
            } else {
                const uint32_t soff = S::CANON ? w_soff + (w_block[r] ? w_block_bytes : 0u) : w_soff;
                fa_lds_dma::buffer_to_lds_b128_scalar<1, 0, 0>(w_now, base + S::X_BYTES + q * 1024, wv[r], __builtin_amdgcn_readfirstlane((int)soff));
            }
        } else {
            if constexpr (S::JOINED) fa_lds_dma::buffer_to_lds_b128_ahead(x_now, x_lds, stage + (r - S::WR) * 1024, xv[r - S::WR], (int)x_soff);
            else fa_lds_dma::buffer_to_lds_b128_scalar<1, 0, 0>(x_now, S::X_EVEN ? base + (loader * S::XR + r - S::WR) * 1024 : base + (loader * S::XR + r - S::WR) % S::X_REQ * 1024, xv[r - S::WR], (int)x_soff);
        }
        if (r == S::REQ - 1) {  // the step's last one
            ++asked, x_soff += STRIDE * 128, w_soff += STRIDE * w_per_step;
            const bool in = asked < n_steps;
            x_now.z = in ? x_rs.z : 0u;
            if constexpr (S::JOINED) {
#pragma unroll
                for (int i = 0; i < S::WR; ++i) w_joined[i].z = in ? w_bytes[i] : 0u;
            } else {
                w_now.z = in ? w_rs.z : 0u;
            }
        }
    };

    // Operand reads: lane l reads row l % 32 (+ 32 per tile) and the 8 features l / 32 of each 16. Places within a stage, of product
    // q of this wave (features 16 kk .. + 15 of the stage's 64):
    const uint32_t h = lane >> 5, r32 = lane & 31;
    uint32_t x_at[S::KN], w_at[S::KN];
    const uint32_t w_row = wn * S::TN * 32 + r32;  // (+ 32 per tile: the same place in the pattern)
    constexpr uint32_t W_TILE = S::WB == 16 ? (S::CANON ? 2048 : 4096) : S::WB == 8 ? (S::CANON ? 1024 : 2048) : (S::CANON ? 512 : 1024);
#pragma unroll
    for (int q = 0; q < S::KN; ++q) {
        const uint32_t kk = (S::OWN ? 0 : kg * S::KN) + q, b = kk >> 1, half = kk & 1;
        x_at[q] = wm * S::TM * 4096 + (r32 >> 3) * 1024 + (r32 & 7) * 128 + ((2 * kk + h) ^ ((r32 >> 1) & 7)) * 16;
        if constexpr (S::WB == 16) {
            w_at[q] = S::CANON ? b * (S::NTR * 64) + (w_row >> 4) * 1024 + (w_row & 15) * 64 + ((2 * half + h) ^ ((w_row >> 2) & 3)) * 16
                               : (w_row >> 3) * 1024 + (w_row & 7) * 128 + ((2 * kk + h) ^ ((r32 >> 1) & 7)) * 16;
        } else if constexpr (S::WB == 8) {
            w_at[q] = S::CANON ? b * (S::NTR * 32) + (w_row >> 5) * 1024 + (w_row & 31) * 32 + (half ^ ((w_row >> 3) & 1)) * 16 + h * 8
                               : (w_row >> 4) * 1024 + (w_row & 15) * 64 + (kk ^ ((w_row >> 2) & 3)) * 16 + h * 8;
        } else {  // (the 8 bytes of both halves of the wave: 4 bytes per lane would be two lanes to a bank)
            w_at[q] = S::CANON ? b * (S::NTR * 16) + w_row * 16 + half * 8 : (w_row >> 5) * 1024 + (w_row & 31) * 32 + kk * 8;
        }
        w_at[q] += S::X_BYTES;
    }
    // The operands of one stage as they lie in LDS (block-quantised weights become f16 in registers, in front of the product).
    struct Operands {
        typename S::raw_t w[S::TN][S::KN];
        h8_t x[S::TM][S::KN];
    };
    auto fetch = [&](Operands &o, uint32_t stage, int e) __attribute__((always_inline)) {  // read number e of the stage
        const int q = e / (S::TM + S::TN), t = e % (S::TM + S::TN);
        if (t < S::TM) o.x[t][q] = *reinterpret_cast<const h8_t *>(smem + own + x_at[q] + stage + t * 4096);
        else o.w[t - S::TM][q] = *reinterpret_cast<const typename S::raw_t *>(smem + own + w_at[q] + stage + (t - S::TM) * W_TILE);
    };
    u4v_t scales[S::TN] = {};  // of the wave's rows, 8 blocks = 4 stages
    const unsigned char *scale_at = smem + S::ALL_STAGES + w_row * 16 + (S::OWN ? wave * 4 : 0);
    auto fetch_scales = [&]() __attribute__((always_inline)) {
        if constexpr (S::QUANT) {
#pragma unroll
            for (int i = 0; i < S::TN; ++i) {
                if constexpr (S::OWN) scales[i].x = *reinterpret_cast<const uint32_t *>(scale_at + i * 512);
                else scales[i] = *reinterpret_cast<const u4v_t *>(scale_at + i * 512);
            }
            scale_at += S::NTR * 16;
        }
    };
    auto w_operand = [&](const Operands &o, int i, int q, int ks4) __attribute__((always_inline)) -> h8_t {
        if constexpr (S::WB == 16) {
            return o.w[i][q];
        } else {
            const uint32_t pair = scales[i][S::OWN ? 0 : ks4];  // (a copy: the bit cast of a vector's element takes element 0)
            const h2v_t s2 = __builtin_bit_cast(h2v_t, pair);
            _Float16 s;
            if constexpr (S::KN == 4) s = s2[q >> 1];
            else if constexpr (S::KG == 2) s = kg ? s2[1] : s2[0];
            else s = kg >= 2 ? s2[1] : s2[0];
            const h8_t sc = {s, s, s, s, s, s, s, s};
            if constexpr (S::WB == 8) return fa_quant::q8_to_f16(o.w[i][q].x, o.w[i][q].y) * sc;
            else return fa_quant::q4_to_f16(h ? o.w[i][q].y : o.w[i][q].x) * sc;
        }
    };

    f16v_t acc[S::SETS][S::TN][S::TM], sums[S::TN][S::TM];  // (FOLD: of the last steps, and of all before)
#pragma unroll
    for (int i = 0; i < S::TN; ++i)
#pragma unroll
        for (int j = 0; j < S::TM; ++j) {
            sums[i][j] = f16v_t{};
#pragma unroll
            for (int t = 0; t < S::SETS; ++t) acc[t][i][j] = f16v_t{};
        }

    // The write stage turns pieces of 8 outputs: piece i of a thread is number tid + i NT of the turn's, row after row, so that a thread
    // comes back to the same NCOL columns and what depends on them - matrix, head, bias, place of the first output - is worked out once.
    // What the pieces take from memory is asked for BATCH pieces at a time, from addresses that are valid whatever the piece. (One after
    // the other, with the columns worked out and up to three trips to memory in a row per piece, us: 2048 rows, FusedQkv + KvPrepFused
    // of 2560 x 2048 F16, paged 45.2 -> 40.1, with the norm; 5120 x 3072 83.2 -> 81.0; o_proj 3072 x 3072 39.2 -> 37.2; 1000 rows, 2048 x
    // 2048 Q8_0 16.2 -> 15.4; 500 rows, 1152 x 896 Q8_0, paged 11.5 -> 11.1, o_proj of it 6.63 -> 6.76, which has nothing to ask for.)
    constexpr bool EARLY = S::MT * S::NTR <= 64 * 96;
    constexpr int PIECES = S::NTR / 8, TURN_PIECES = S::WM * S::TJ * 32 * PIECES, PER_TURN = (TURN_PIECES + S::NT - 1) / S::NT, TURNS = S::TM / S::TJ;
    constexpr int NCOL = PIECES / std::gcd(S::NT, PIECES), BATCH = EARLY ? PER_TURN * TURNS : PER_TURN > 5 ? PER_TURN / 2 : PER_TURN, BATCHES = EARLY ? 1 : PER_TURN / BATCH;
    static_assert(TURN_PIECES % S::NT == 0 || PER_TURN == 1, "the threads share the pieces evenly, or some have none");
    static_assert(EARLY ? PER_TURN % NCOL == 0 : PER_TURN % BATCH == 0 && BATCH % NCOL == 0, "piece i of a batch has column i % NCOL");
    // Piece i of a column is STEP rows of LDS below the one before, and ROW_STEP input rows.
    constexpr int STEP = NCOL * S::NT / PIECES, ROW_STEP = S::TJ == S::TM ? STEP : STEP * S::TM;
    static_assert(S::TJ == S::TM || (S::TJ == 1 && STEP % 32 == 0) || PER_TURN <= NCOL, "the rows of a column are evenly apart");
    h8_t early[EARLY ? BATCH : 1];  // the residual
    struct Column {
        int mat;
        uint32_t gn;           // row of its matrix
        uint32_t at, mate_at;  // its first piece in LDS (mate_at: the one that it is rotated with)
        uint32_t row;          // ... and the input row of that one
        bool in;               // there is such a column
        h8_t bias, mate_bias;  // (mate_bias: of the half of a head that the piece is rotated with)
    } column[NCOL];
    // Piece i of a turn: its row in LDS, and which input row that is.
    auto lds_row = [&](int thread, int i) __attribute__((always_inline)) -> uint32_t {
        const uint32_t t = (uint32_t)(thread + i * S::NT) / PIECES;
        return TURN_PIECES % S::NT == 0 ? t : min(t, (uint32_t)(S::WM * S::TJ * 32) - 1);
    };
    auto input_row = [&](uint32_t t) __attribute__((always_inline)) -> uint32_t { return m0 + ((t >> 5) / S::TJ * S::TM + (t >> 5) % S::TJ) * 32 + (t & 31); };
    // The residual, asked for ahead of everything else where the tile leaves registers for it: at the end of the one chain that a
    // launch of a round of such tiles is, it would be a trip to memory more (3072 x 3072, 320 rows: F16 12.8 -> 12.3 us, Q8_0 12.2 ->
    // 11.7, Q4_0 12.0 -> 11.6; 896 x 896, 500 rows: 6.3 -> 6.0, 6.8 -> 6.5, 6.7 -> 6.5). The rest is asked for behind the loop: ahead of it
    // the addresses of all that are worked out while nothing has been asked for yet (Q8_0, 500 rows, 1152 x 896: 10.2 -> 10.3 us), and
    // behind the first requests the first steps wait for it (10.7).
    if constexpr (EARLY) {
        if (a.residual) {
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                const uint32_t gm = input_row(lds_row(tid, i % PER_TURN)) + i / PER_TURN * (S::TJ * 32), r = n0 + (uint32_t)(tid + i % PER_TURN * S::NT) % PIECES * 8;
                early[i] = fa_norm::load_global<h8_t>(a.residual + (gm < a.m && r < N_tile ? (size_t)gm * N_tile + r : 0));
            }
        }
    }
    // The launch's arguments, read where the write stage begins and not kept from the entry on, for tiles whose loop has no scalar
    // registers to spare. (The smaller tiles would wait for them there: 0.1 us of 6.6.) For speed only: kept in lanes of a vector register,
    // as a few of the smaller tiles' are, they are read back as they were written. Built that way the largest tiles pass the same tests,
    // and no lane of any kernel is found to be read before or after its time (tests/test_spilled_scalars.py looks at the built code).
    static_assert(std::is_trivially_copyable<GemmDev>::value, "read as raw bytes from the argument block, where it is the first member");
    auto arguments = []() __attribute__((always_inline)) -> const GemmDev & {
        auto g = __builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(g));
        return *(const GemmDev *)g;
    };
    // The write stage's code is there once for each of what it does, so that none of it runs through the others' branches.
    auto by_what = [&](const GemmDev &g, auto &&f) __attribute__((always_inline)) {
        if constexpr (FORM != ANY) f(std::integral_constant<int, FORM>{});
        else if (!g.rope.on) f(std::integral_constant<int, PLAIN>{});
        else if (!pairs) f(std::integral_constant<int, ADJACENT>{});
        else f(std::integral_constant<int, APART>{});
    };
    auto ask_columns = [&](auto what, const GemmDev &g, int thread) __attribute__((always_inline)) {
        constexpr int W = decltype(what)::value;
#pragma unroll
        for (int i = 0; i < NCOL; ++i) {
            Column &col = column[i];
            const uint32_t n8 = (uint32_t)(thread + i * S::NT) % PIECES, t = lds_row(thread, i);
            const uint32_t at = n0 + n8 * 8, end = S::JOINED ? rows0 + 2 * rows1 : N_tile;
            uint32_t r = min(at, end - 8);
            col.in = at < end && (TURN_PIECES % S::NT == 0 || thread < TURN_PIECES);
            col.mat = matrix_of(r), col.gn = W == APART ? paired(r) : r;
            col.row = input_row(t), col.at = t * S::T_STRIDE + n8 * 32, col.mate_at = t * S::T_STRIDE + (n8 ^ 2) * 32;
            if (g.bias[0]) {  // (all matrices have one, or none has)
                const __half *const bias = pick3(col.mat, g.bias[0], g.bias[1], g.bias[2]);
                col.bias = fa_norm::load_global<h8_t>(bias + col.gn);
                if constexpr (W == APART) col.mate_bias = fa_norm::load_global<h8_t>(bias + paired(r ^ 16));
            }
        }
    };
    if constexpr (S::QUANT) {  // all scales first: 16 bytes (8 blocks) of 64 rows per request
        const __half *sp = pick3(tile_mat, a.scales[0], a.scales[1], a.scales[2]);
        const fa_lds_dma::rsrc_words s_rs = fa_lds_dma::make_rsrc_words(sp, N_tile * (K / 32) * 2);
        const uint32_t requests = S::NTR % 64 == 0 ? (K + 255) / 256 * (S::NTR / 64) : S::scale_bytes(K) / 1024;
        for (uint32_t q = wave; q < requests; q += S::NW) {
            constexpr uint32_t PER = S::NTR % 64 == 0 ? S::NTR / 64 : 1;  // requests per 16 bytes of all rows, where that is whole ones
            const uint32_t at = S::NTR % 64 == 0 ? q % PER * 64 + lane : q * 64 + lane, unit = S::NTR % 64 == 0 ? 0u : at / S::NTR;
            fa_lds_dma::buffer_to_lds_b128_scalar<1, 0, 0>(s_rs, lds_base - own + S::ALL_STAGES + q * 1024, (int)(weight_row(at % S::NTR) * (K / 32) * 2 + unit * 16),
                                                    (int)(S::NTR % 64 == 0 ? q / PER * 16 : 0u));
        }
    }
#pragma unroll
    for (int s = 0; s < S::NS; ++s)
#pragma unroll
        for (int r = 0; r < S::REQ; ++r) request(r, s * S::STAGE);
    Operands o0, o1;
    wait_requests<S::REQ *(S::NS - 1)>();
    meet();
#pragma unroll
    for (int e = 0; e < S::READS; ++e) fetch(o0, 0, e);
    // A step multiplies the operands that are in registers while it fetches the next step's from LDS. At its barrier every wave has
    // the operands of step ks in registers - their stage is free for step ks + NS - and step ks + 1 has landed for everybody.
    // The requests go out between the products: the memory unit takes a KiB in about 20 cycles, and a wave that issues all of its
    // requests in one go leaves its matrix core idle for as long.
    auto step = [&](uint32_t cur, uint32_t next, int ks4, int set, bool fold, const Operands &now, Operands &then) __attribute__((always_inline)) {
        wait_requests<S::REQ *(S::NS - 2)>();
        if constexpr (S::OWN) __builtin_amdgcn_s_waitcnt(0xC07F);  // (lgkmcnt(0): the operands have left the stage that is asked for again)
        else meet();
        constexpr int NM = S::KN * S::TN * S::TM;
        if (S::OWN || ks4 == 0) fetch_scales();
        h8_t fa[S::TN];
#pragma unroll
        for (int p = 0; p < NM; ++p) {
            const int q = p / (S::TN * S::TM), i = p / S::TM % S::TN, j = p % S::TM;
#pragma unroll
            for (int e = p * S::READS / NM; e < (p + 1) * S::READS / NM; ++e) fetch(then, next, e);
            if (j == 0) fa[i] = w_operand(now, i, q, ks4);
            f16v_t &sum = acc[(set + q) % S::SETS][i][j];
            f16v_t chain = sum;
            if (fold && q == 0) sums[i][j] += chain, chain = f16v_t{};
            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], now.x[j][q], chain, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0x6);  // (vector and scalar arithmetic may move: addresses, the conversion of weights)
#pragma unroll
            for (int r = p * S::REQ / NM; r < (p + 1) * S::REQ / NM; ++r) request(r, cur);
            __builtin_amdgcn_sched_barrier(0x6);
        }
    };
    // (unrolled over the stages, so that their places are constants; operands of even and odd steps in registers of their own)
    constexpr int UNROLL = (S::QUANT && !S::OWN) || S::FOLD ? S::NS * 4 / (S::NS % 4 == 0 ? 4 : S::NS % 2 == 0 ? 2 : 1) : S::NS % 2 == 0 ? S::NS : 2 * S::NS;
    static_assert(UNROLL * S::KN % S::SETS == 0, "the sets come round with the unrolled loop");
    // Behind a multiple of 32 bytes, the unit in which instructions are fetched: of the loop's instructions, 4 and 8 bytes in a row with few
    // waits between them, fewer then lie over an end of it. (Q8_0 tiles with stages of their own, 4-byte steps from 0 to 28: 64 rows x 3072 x
    // 3072 11.05 us at 0, 11.4 to 11.6 at the others, 160 rows x 2048 x 2048 9.2 and 9.3 to 9.5, FusedQkv + KvPrepFused of 48 rows x 5120 x 3072
    // 14.65 and 15.0 to 15.1; the other tiles within 1 %.)
    asm volatile(".p2align 5");
    for (uint32_t left = n_steps;;) {
        bool done = false;
        if (S::OWN && left == 0) break;  // (a wave without a step)
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t cur = u % S::NS * S::STAGE, next = (u + 1) % S::NS * S::STAGE;
            const bool fold = S::FOLD != 0 && u % 4 == 3;
            if (u % 2 == 0) step(cur, next, u % 4, u * S::KN % S::SETS, fold, o0, o1);
            else step(cur, next, u % 4, u * S::KN % S::SETS, fold, o1, o0);
            if (--left == 0) {
                done = true;
                break;
            }
        }
        if (done) break;
    }
    wait_requests<0>();  // (the last ones delivered nothing, but they have to be over before the write stage reuses the LDS)
    if constexpr (S::FOLD != 0) {
#pragma unroll
        for (int i = 0; i < S::TN; ++i)
#pragma unroll
            for (int j = 0; j < S::TM; ++j) acc[0][i][j] = sums[i][j] + acc[0][i][j];
    }
#pragma unroll
    for (int t = 1; t < S::SETS; ++t)
#pragma unroll
        for (int i = 0; i < S::TN; ++i)
#pragma unroll
            for (int j = 0; j < S::TM; ++j) acc[0][i][j] += acc[t][i][j];

    // (The largest block-quantised tile has no register left to keep the lane's number in through the loop: with it the Q8_0 row-major
    // kernel kept operands of its loop in memory, 6 to 12 % of its time; 1442 rows, 3072 x 3072 44.5 us, 39.8 without.)
    constexpr bool FULL = S::QUANT && S::MT * S::NTR > 128 * 128;
    const int lane_w = FULL ? (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) : lane;
    const int tid_w = FULL ? wave * 64 + lane_w : tid;
    const uint32_t h_w = FULL ? (uint32_t)lane_w >> 5 : h, r32_w = FULL ? (uint32_t)lane_w & 31u : r32;

    // Write stage: accumulators -> LDS as f32 [input row][weight row], 32 input rows of every wave at a time, then
    // alpha * sum + bias + beta * residual, one rounding to f16, 16-byte stores (or the rotation and the stores of KvPrepFused).
    const GemmDev &g = EARLY ? a : arguments();
    // What the column gives to each of its pieces: where the output of input row 0 would be, and the row from which on nothing is stored.
    struct Target {
        __half *first;  // (of a paged cache: of row 0 of page 0, 64 bits, as everything in a pool: one page of all heads may be 8 GiB)
        uint32_t stride, end;
        bool paged, turn;
        const __half *cos_t, *sin_t;  // the tables at its first column
    };
    Target target[NCOL];
    // What a piece takes from memory. (Nothing is done with it where it is asked for, and there is no branch around it - a table that is
    // not wanted is read at its first row, or the input in its place -: what waits for one piece's, ahead of the next piece's request, is
    // a trip to memory per piece. With the columns of both pairings behind a branch, and copied out of it, the write stage of FusedQkv +
    // KvPrepFused, 2048 rows of 5120 x 3072, took 16 us where that of the projections alone takes 6; with the rotation's products and sums
    // from the f16 halves (rope_mix) and the rows of a column a constant apart it takes 8. With the norm, before -> now: F16 2048 rows of 5120 x
    // 3072 76.0 -> 69.1 us, 1200 rows 50.0 -> 47.8, Q4_0 2048 rows 94.2 -> 87.7, Q8_0 1000 rows 49.2 -> 46.0, 500 rows 31.1 -> 29.6, 500 rows of
    // 1152 x 896 10.8 -> 10.7; o_proj of 1500 rows x 2048 x 2048 Q8_0 19.3 -> 18.5, F16 17.3 -> 17.2.)
    struct Side {
        h8_t c, s;     // columns of the RoPE tables, half a head apart; c = the residual
        h4v_t c4, s4;  // ... of pairs in a piece
        uint32_t page;
    };
    // (the kernel's arguments as far as every piece needs them)
    const uint32_t m_all = g.m, pos0 = g.rope.position_offset, last_entry = g.rope.table_rows - 1, last_row = g.rope.capacity - 1;
    const uint32_t half_dim = g.rope.on && g.rope.apply ? g.rope.head_dim >> 1 : 0u, page_size = g.rope.block_size, page_shift = g.page_shift;
    const float alpha = g.alpha, beta = g.beta;
    const int32_t *const table = g.rope.block_table;
    const __half *const residual = g.residual;
    const bool has_bias = g.bias[0] != nullptr;
    auto find_targets = [&](auto what) __attribute__((always_inline)) {
        constexpr int W = decltype(what)::value;
#pragma unroll
        for (int i = 0; i < NCOL; ++i) {
            const Column &col = column[i];
            Target &o = target[i];
            o.first = pick3(col.mat, g.out[0], g.out[1], g.out[2]);
            o.end = col.in ? m_all : 0u, o.paged = false, o.turn = false;
            if constexpr (W == PLAIN) {
                o.stride = S::JOINED ? (col.mat ? rows1 : rows0) : N_tile;
                o.first += col.gn;
            } else {
                const uint32_t D = g.rope.head_dim, head = col.gn >> hd_shift, hd = col.gn & (D - 1), room = g.rope.capacity > pos0 ? g.rope.capacity - pos0 : 0u;
                const uint32_t first_column = W == APART ? hd & ((D >> 1) - 1) : hd >> 1;
                o.stride = D;
                o.paged = col.mat != 0 && table, o.turn = col.mat != 2 && (W == APART || half_dim != 0);
                if (col.mat != 0) o.end = min(o.end, room);  // never outside the cache
                o.first += (col.mat == 0 ? (size_t)head * m_all : o.paged ? (size_t)head * page_size : (size_t)head * g.rope.max_seq_len + pos0) * D + hd;
                o.cos_t = half_dim ? g.rope.cos_t + first_column : reinterpret_cast<const __half *>(g.x);
                o.sin_t = half_dim ? g.rope.sin_t + first_column : reinterpret_cast<const __half *>(g.x);
            }
        }
    };
    auto ask = [&](auto what, Side &w, int i, uint32_t row) __attribute__((always_inline)) {  // (of column i)
        constexpr int W = decltype(what)::value;
        const uint32_t gm = min(row, m_all - 1);
        const Target &o = target[i];
        if constexpr (W == PLAIN) {
            if (!EARLY && residual) w.c = fa_norm::load_global<h8_t>(residual + (size_t)gm * N_tile + column[i].gn);
        } else {
            const uint32_t pos = pos0 + gm;
            const size_t at = (size_t)min(pos, last_entry) * half_dim;
            if constexpr (W == APART) w.c = fa_norm::load_global<h8_t>(o.cos_t + at), w.s = fa_norm::load_global<h8_t>(o.sin_t + at);
            else w.c4 = fa_norm::load_global<h4v_t>(o.cos_t + at), w.s4 = fa_norm::load_global<h4v_t>(o.sin_t + at);
            if (table) {
                const uint32_t cache_row = min(pos, last_row);
                w.page = fa_norm::load_global<uint32_t>(table + (page_shift < 32 ? cache_row >> page_shift : cache_row / page_size));
            }
        }
    };
    auto write = [&](auto what, int i, const Side &w, uint32_t down, uint32_t row) __attribute__((always_inline)) {  // column i, `down` bytes of LDS below its first piece
        constexpr int W = decltype(what)::value;
        const Column &col = column[i];
        const Target &o = target[i];
        const uint32_t gm = row;
        auto value = [&](uint32_t place, h8_t bias) __attribute__((always_inline)) -> h8_t {
            f4v_t s0 = *reinterpret_cast<const f4v_t *>(smem + place);
            f4v_t s1 = *reinterpret_cast<const f4v_t *>(smem + place + 16);
#pragma unroll
            for (int k = 1; k < S::KG; ++k) {
                s0 += *reinterpret_cast<const f4v_t *>(smem + k * S::T_BYTES + place);
                s1 += *reinterpret_cast<const f4v_t *>(smem + k * S::T_BYTES + place + 16);
            }
            float v[8];
            {   // (every step rounded to f32, whatever follows: a product and a sum made into one with the rounding to f16 gives other bits)
#pragma clang fp contract(off)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = (e < 4 ? s0[e & 3] : s1[e & 3]) * alpha;
                if (has_bias) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += (float)bias[e];
                }
            }
            if (W == PLAIN && residual) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = fmaf(beta, (float)w.c[e], v[e]);
            }
            h8_t y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = (_Float16)v[e];
            return y;
        };
        h8_t y = value(col.at + down, col.bias);
        __half *dst = o.first + (size_t)gm * o.stride;
        if constexpr (W != PLAIN) {
            h8_t turned;
            if constexpr (W == APART) turned = rope_apart(y, value(col.mate_at + down, col.mate_bias), w.c, w.s, (col.gn & (g.rope.head_dim - 1)) < half_dim);
            else turned = rope_adjacent(y, w.c4, w.s4);
            y = o.turn ? turned : y;
            if (table) {
                const uint32_t pos = pos0 + gm, in_page = page_shift < 32 ? pos & (page_size - 1) : pos % page_size;
                __half *const there = o.first + ((size_t)w.page * g.rope.n_kv_heads * page_size + in_page) * g.rope.head_dim;
                dst = o.paged ? there : dst;
            }
        }
        if (gm < o.end) fa_norm::store_global(dst, y);
    };
    auto to_lds = [&](int j0) __attribute__((always_inline)) {
        // register r of lane l of a 32 x 32 tile is weight row 8 (r / 4) + 4 (l / 32) + r % 4 and input row l % 32
#pragma unroll
        for (int j = j0; j < j0 + S::TJ; ++j)
#pragma unroll
            for (int i = 0; i < S::TN; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f4v_t *>(smem + kg * S::T_BYTES + ((wm * S::TJ + j - j0) * 32 + r32_w) * S::T_STRIDE + (wn * S::TN * 32 + i * 32 + q * 8 + h_w * 4) * 4) =
                        f4v_t{acc[0][i][j][q * 4 + 0], acc[0][i][j][q * 4 + 1], acc[0][i][j][q * 4 + 2], acc[0][i][j][q * 4 + 3]};
    };
    by_what(g, [&](auto what) __attribute__((always_inline)) {
        ask_columns(what, g, tid_w);
        find_targets(what);
        if constexpr (EARLY) {
            Side side[BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                if (decltype(what)::value == PLAIN) side[i].c = early[i];
                ask(what, side[i], i % NCOL, column[i % NCOL].row + i % PER_TURN / NCOL * ROW_STEP + i / PER_TURN * (S::TJ * 32));
            }
#pragma unroll
            for (int turn = 0; turn < TURNS; ++turn) {
                __syncthreads();  // every wave is done with the stages / the previous rows have been read out
                to_lds(turn * S::TJ);
                __syncthreads();
#pragma unroll
                for (int i = 0; i < PER_TURN; ++i)
                    write(what, i % NCOL, side[turn * PER_TURN + i], i / NCOL * (STEP * S::T_STRIDE), column[i % NCOL].row + i / NCOL * ROW_STEP + turn * (S::TJ * 32));
            }
        } else {
            // (One copy of the code for all turns and batches, the accumulators moving up by a turn: run once it comes from memory,
            // and the instructions of 20 pieces are more than the stores take. What a batch takes from memory is asked for ahead of
            // the one before it.)
            constexpr int PER_COLUMN = BATCH / NCOL;  // pieces of a column in a batch
            Side now[BATCH], next[BATCH];
            auto ask_batch = [&](Side(&side)[BATCH], uint32_t rows) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < BATCH; ++i) ask(what, side[i], i % NCOL, column[i % NCOL].row + i / NCOL * ROW_STEP + rows);
            };
            if (BATCHES > 1) ask_batch(now, 0);
#pragma unroll 1
            for (int turn = 0; turn < TURNS; ++turn) {
                auto after = [&](int n) __attribute__((always_inline)) -> uint32_t {  // rows of the batch behind batch n (past the last: nobody takes them)
                    return n + 1 < BATCHES ? (n + 1) * (PER_COLUMN * ROW_STEP) + turn * (S::TJ * 32) : (turn + 1) * (S::TJ * 32);
                };
                if (BATCHES > 1) ask_batch(next, after(0));
                else ask_batch(now, turn * (S::TJ * 32));
                __syncthreads();
                to_lds(0);
#pragma unroll
                for (int j = 0; j + S::TJ < S::TM; ++j)
#pragma unroll
                    for (int i = 0; i < S::TN; ++i) acc[0][i][j] = acc[0][i][j + S::TJ];
                __syncthreads();
#pragma unroll 1
                for (int n = 0; n < BATCHES; ++n) {
                    const uint32_t rows = n * (PER_COLUMN * ROW_STEP) + turn * (S::TJ * 32);
                    if (n > 0) ask_batch(next, after(n));
#pragma unroll
                    for (int i = 0; i < BATCH; ++i)
                        write(what, i % NCOL, now[i], (uint32_t)(n * PER_COLUMN + i / NCOL) * (STEP * S::T_STRIDE), column[i % NCOL].row + i / NCOL * ROW_STEP + rows);
                    if (BATCHES > 1) {
#pragma unroll
                        for (int i = 0; i < BATCH; ++i) now[i] = next[i];
                    }
                }
            }
        }
    });
}

template <class S, int MIN_WAVES, Form FORM>
fa_status launch_form(fa_ctx *ctx, FaLaunchScope &scope, GemmDev &a) {
    static std::atomic<bool> lds_allowed_on[64];  // per device (contexts of several threads may get here together: the calls are idempotent)
    std::atomic<bool> &lds_allowed = lds_allowed_on[ctx->device & 63];
    if (!lds_allowed.load(std::memory_order_acquire)) {
        FA_HIP(hipFuncSetAttribute((const void *)tile_gemm_kernel<S, MIN_WAVES, FORM>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        lds_allowed.store(true, std::memory_order_release);
    }
    a.n_tiles = 0, a.m_tiles = ceil_div_u32(a.m, S::MT);
    for (int i = 0; i < 3; ++i) a.tiles[i] = ceil_div_u32(a.rows[i], S::NTR), a.n_tiles += a.tiles[i];
    if (S::JOINED) a.n_tiles = ceil_div_u32(a.rows[0] + 2 * a.rows[1], S::NTR);
    a.panel_inv = fa_inverse(a.m_tiles > 8 ? 4 * a.m_tiles : a.m_tiles);
    const uint32_t grid = ceil_div_u32(a.n_tiles * a.m_tiles, 8) * 8;
    scope.launch((tile_gemm_kernel<S, MIN_WAVES, FORM>), dim3(grid), dim3(S::NT), S::lds_bytes(a.k_dim), a);
    return FA_OK;
}

template <class S, int MIN_WAVES>
fa_status launch_shape(fa_ctx *ctx, FaLaunchScope &scope, GemmDev &a) {
    if constexpr (S::OWN || (S::QUANT && S::NS == 8) || S::JOINED) {
        if (!a.rope.on) return launch_form<S, MIN_WAVES, PLAIN>(ctx, scope, a);
        if (a.rope.apply && !a.rope.normal) return launch_form<S, MIN_WAVES, APART>(ctx, scope, a);
        return launch_form<S, MIN_WAVES, ADJACENT>(ctx, scope, a);
    } else {
        return launch_form<S, MIN_WAVES, ANY>(ctx, scope, a);
    }
}

template <int WB, bool CANON>
fa_status launch_tile(fa_ctx *ctx, FaLaunchScope &scope, TileShape shape, GemmDev &a) {
    if constexpr (WB == 16) {
        switch (shape) {
            case TILE_64x64_OWN:
            case TILE_64x32:
            case TILE_64x64_DEEP:
            case TILE_64x64: return launch_shape<Shape<WB, CANON, 2, 2, 1, 1, 1, 4>, 2>(ctx, scope, a);
            case TILE_64x96: return launch_shape<Shape<WB, CANON, 2, 3, 1, 1, 1, 4>, 2>(ctx, scope, a);
            case TILE_128x64: return launch_shape<Shape<WB, CANON, 2, 2, 1, 2, 1, 3>, 2>(ctx, scope, a);
            case TILE_128x128: return launch_shape<Shape<WB, CANON, 2, 4, 1, 2, 1, 4>, 2>(ctx, scope, a);
            case TILE_256x128: return launch_shape<Shape<WB, CANON, 4, 2, 1, 2, 2, 3>, 2>(ctx, scope, a);
            case TILE_256x160: return launch_shape<Shape<WB, CANON, 4, 1, 1, 2, 5, 3, true>, 1>(ctx, scope, a);
        }
    } else {
        switch (shape) {
            case TILE_64x64_OWN: return launch_shape<Shape<WB, CANON, 1, 1, 4, 2, 2, 3, false, true>, 1>(ctx, scope, a);
            case TILE_64x64_DEEP: return launch_shape<Shape<WB, CANON, 1, 2, 2, 2, 1, 8>, 1>(ctx, scope, a);
            case TILE_64x32: return launch_shape<Shape<WB, CANON, 1, 1, 4, 2, 1, 8>, 1>(ctx, scope, a);
            case TILE_64x64: return launch_shape<Shape<WB, CANON, 1, 2, 2, 2, 1, 4>, 2>(ctx, scope, a);
            case TILE_64x96:
                if constexpr (WB == 4) {  // (3072 x 3072, 340 rows, canonical and row-major: 16.8 -> 14.8 us, 18.4 -> 15.3; Q8_0 has room for two stages, 16.4 -> 16.9)
                    if (a.k_dim >= 1024) return launch_shape<Shape<WB, CANON, 1, 1, 4, 2, 3, 3, false, true>, 1>(ctx, scope, a);
                }
                return launch_shape<Shape<WB, CANON, 1, 3, 2, 2, 1, 4>, 2>(ctx, scope, a);
            case TILE_128x64: return launch_shape<Shape<WB, CANON, 1, 2, 4, 4, 1, 4>, 2>(ctx, scope, a);
            case TILE_128x128: return launch_shape<Shape<WB, CANON, 1, 4, 2, 4, 1, 4>, 2>(ctx, scope, a);
            case TILE_256x128: return launch_shape<Shape<WB, CANON, 2, 4, 1, 4, 1, 3>, 2>(ctx, scope, a);
            case TILE_256x160: break;
        }
    }
    return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "no such tile");
}

fa_status launch_f16(fa_ctx *ctx, FaLaunchScope &scope, TileShape shape, GemmDev &a, bool canonical);
fa_status launch_q8(fa_ctx *ctx, FaLaunchScope &scope, TileShape shape, GemmDev &a, bool canonical);
fa_status launch_q4(fa_ctx *ctx, FaLaunchScope &scope, TileShape shape, GemmDev &a, bool canonical);

}  // namespace fa_tile
