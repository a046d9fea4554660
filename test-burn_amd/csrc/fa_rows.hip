// Attention of a chunk or a prompt of moderate size: a workgroup owns 32 query rows and attends all of their keys (or one of a few
// splits of them), its waves each a stream of 32-key tiles of their own.
//
// Arithmetic contract = the prefill kernel's (crates/metallic-foundry/src/metals/flashattention/flash_prefill.metal:93-446: key j
// visible to row r iff !causal or j <= query_offset + r; f32 accumulation; running max from -1e30; out = acc / l when l is finite and
// |l| > 1e-6, else 0).
//
// What bounds such a launch is one workgroup's chain. The tiled kernel (fa_prefill.hip) has few items for a chunk - 500 rows of 14
// heads are 56 of 128 rows -, each a start, a chain of barrier-separated phases and an end that meet only within the workgroup, and,
// with its keys split over more workgroups, a state of 32 to 64 KB to store and a second launch. Here
//   * the heads of a KV group are one list of rows, position by position, cut every 32 (a chunk of 5 rows and 7 heads is two
//     blocks, not seven): 224 workgroups for those 500 rows;
//   * wave w attends key tiles w, w + NW, ...: K and V go from memory into LDS that only this wave reads, so that there is no barrier
//     between the first tile and the last, and a wave waits for its own loads alone. The next tile's K is asked for when the last
//     operand of this one's has been read, V likewise: one tile's room per wave, and the other waves of the SIMD fill the gaps
//     (at D 64 two stages per wave, which leave room for half as many waves, are 5 to 20 % slower);
//   * the waves' sums meet once, in LDS, and a thread folds its (row, 4 dims) of all of them and writes the row out.
//   * the blocks that read the same keys through one L2 begin at different ones of them, so that what the first to come asks of memory
//     is there for the others, and they do not all ask one channel of the L2 at a time (RowsTurn).
// It reads a block's keys once per 32 rows, 131 KB/us and CU along the rows (fa_lds_dma.h), which is why long keys under many rows
// stay with the tiled kernel (once per 128 rows): fa_prefill_rows_plan. us before and now (tiled or short-chunk kernel before):
//   H14 / Hkv2 / D64:   32 rows after 500 10.7 -> 4.6; 500 after 1000 14.9 -> 7.5; 2048 rows 22.7 -> 16.2; 32 after 8160 21.0 -> 9.3
//   H24 / Hkv8 / D128:  32 after 500 12.6 -> 6.9; 128 after 1000 16.8 -> 9.5; 500 rows 12.6 -> 8.3; 32 after 8160 17.6 -> 13.0 (those from the
//                       last-level cache; from memory 17.1, the short-chunk kernel 17.2)
//   H16 / Hkv2 / D128:  500 after 1000 23.8 -> 12.2; 32 after 8160 32.6 -> 12.6
// (The splits combined by the last workgroup of a block to finish, in the launch: 12.8 to 16.3 us for the last of these, against
// 12.6 with the merge launch - one compute unit reads all of the block's states there.)
#include "fa_internal.h"
#include "fa_lds_dma.h"
#include <type_traits>

namespace {

using fa_lds_dma::buffer_to_lds_b128;
using fa_lds_dma::make_rsrc_words;
using fa_lds_dma::rows16_lane_src;
using fa_lds_dma::rows16_operand;
using fa_lds_dma::rsrc_words;

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef float f16_t __attribute__((ext_vector_type(16)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

template <bool BF16>
__device__ __forceinline__ _Float16 to_elem(float v) {
    if (BF16) return __builtin_bit_cast(_Float16, (__bf16)v);
    return (_Float16)v;
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
template <bool BF16>
__device__ __forceinline__ f16_t mfma(h8_t a, h8_t b, f16_t c) {
    return BF16 ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8_t, a), __builtin_bit_cast(bf8_t, b), c, 0, 0, 0)
                : __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// (x[l], x[l ^ 32]), the lower half's value first
__device__ __forceinline__ u2_t both_halves(float x) { return __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false); }

struct RowsDev {
    const __half *q, *k, *v;
    __half *out;
    uint64_t q_stride_h, q_stride_m, k_stride_h, v_stride_h, out_stride_h, out_stride_m;
    const int32_t *block_table;
    uint32_t group_size, rcp_group /* floor(2^32 / group_size) + 1, 0 for 1: exact quotients */, q_len, kv_len, query_offset, causal, block_size, block_shift, n_kv_heads;
    uint32_t pool_bytes32;  // paged: size of each pool when below 4 GiB (whole pages then go by a 32-bit offset), else 0
    uint32_t n_blocks;      // blocks per KV head
    uint32_t inv_splits, inv_kv_heads;  // fa_inverse
    uint32_t turn;          // TURN: rounds that the workgroups of a KV head attend in turned orders, a power of two up to 32
    uint32_t pair_step;     // log2 of how many blocks apart two of a KV head on one XCD are
    uint32_t splits;        // > 1: a block's keys are divided over as many workgroups, whose states a merge launch combines
    float *part_acc, *part_ml;  // [KV head][block][split][32][D] unnormalised sums, [..][32][2] (max, sum)
    float scale_log2e;
};

constexpr int KT = 32;  // keys per tile

// POOL: 0 a contiguous cache, 1 paged, 2 paged with pools of 4 GiB or more (no 32-bit offsets)
// TURN: the workgroups that read the same keys through one L2 begin at different ones (RowsTurn)
template <int D, int NW, bool BF16, int POOL, bool TURN>
__global__ void __launch_bounds__(NW * 64, D == 64 ? 4 : 2) flash_rows_kernel(RowsDev a_by_value) {
    static_assert(std::is_trivially_copyable<RowsDev>::value, "read as raw bytes from the argument block, where it is the first member");
    const RowsDev a = *(const RowsDev *)__builtin_amdgcn_kernarg_segment_ptr();
    (void)a_by_value;
    asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.out), "s"(a.q_stride_h), "s"(a.q_stride_m), "s"(a.k_stride_h), "s"(a.v_stride_h),
                 "s"(a.out_stride_h), "s"(a.out_stride_m), "s"(a.block_table), "s"(a.group_size), "s"(a.rcp_group), "s"(a.q_len),
                 "s"(a.kv_len), "s"(a.query_offset), "s"(a.causal), "s"(a.block_size), "s"(a.block_shift), "s"(a.n_kv_heads));
    asm volatile("" ::"s"(a.pool_bytes32), "s"(a.n_blocks), "s"(a.splits), "s"(a.part_acc), "s"(a.part_ml), "s"(a.scale_log2e), "s"(a.inv_splits), "s"(a.inv_kv_heads),
                 "s"(TURN ? a.turn : 0), "s"(TURN ? a.pair_step : 0));
    constexpr bool PAGED = POOL != 0;
    constexpr int DSTEPS = D / 16, DBLKS = D / 32, ROWB = D * 2;
    constexpr int RB_BYTES = 16 * ROWB;                 // 16 rows of K in LDS (rows16 layout), or of V
    constexpr int HALF = 2 * RB_BYTES, TILE = 2 * HALF;  // K or V of a tile; both
    constexpr int COLS = ROWB / 64;                     // 64-byte columns of a row = loads per 16 rows
    constexpr int RG_BYTES = 4 * ROWB;                  // one 4-row group of a V tile
    constexpr int Q_BYTES = 2 * RB_BYTES, STAGES = NW * TILE;
    // After the tiles: the waves' sums as [wave][quad of 4 dims][row] float4, a quad's 32 rows padded by one, then (m, l)
    constexpr int QUADS = D / 4, QUAD_BYTES = 32 * 16 + 16, ACC_BYTES = QUADS * QUAD_BYTES;
    constexpr int LDS_BYTES = (STAGES + Q_BYTES > NW * (ACC_BYTES + 256)) ? STAGES + Q_BYTES : NW * (ACC_BYTES + 256);
    __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];
    typedef __attribute__((address_space(3))) void *lds_ptr;
    const uint32_t lds_addr = (uint32_t)(uintptr_t)(lds_ptr)lds;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, hi = lane >> 5;

    // ---- the workgroup's rows, heaviest (latest) blocks first. Workgroup ids equal modulo 8 share an L2: an XCD has every eighth
    // (block, KV head) pair, so that with 2, 4 or 8 KV heads it reads one of them. (Three divisions here were 0.05 us of 4.1 to 7.8.)
    const uint32_t id = blockIdx.x >> 3, j = fa_quotient(id, a.splits, a.inv_splits), split = id - j * a.splits, pair = (blockIdx.x & 7u) + 8u * j;
    const uint32_t from_last = fa_quotient(pair, a.n_kv_heads, a.inv_kv_heads), kvh = pair - from_last * a.n_kv_heads;
    if (from_last >= a.n_blocks) return;
    const uint32_t block = a.n_blocks - 1 - from_last, G = a.group_size, n_rows = G * a.q_len;
    // row r of the KV head's list (its heads' rows of one position after the other) -> query row; head = r - G * that
    auto position = [&](uint32_t r) __attribute__((always_inline)) -> uint32_t { return a.rcp_group ? __umulhi(r, a.rcp_group) : r; };
    const uint32_t row0 = block * 32, pos0 = position(row0), pos1 = position(min(row0 + 31, n_rows - 1));
    uint32_t kv_end = a.kv_len;  // keys that some row sees
    if (a.causal) kv_end = (uint32_t)min((uint64_t)a.kv_len, (uint64_t)pos1 + a.query_offset + 1);
    kv_end = (uint32_t)__builtin_amdgcn_readfirstlane((int)kv_end);  // (uniform, and so that the loads' scalar operands are)
    // tiles of this workgroup: [t_lo, n_tiles); wave w attends t_lo + w, + NW, ...
    const uint32_t all_tiles = (kv_end + KT - 1) / KT, per_split = fa_quotient(all_tiles + a.splits - 1, a.splits, a.inv_splits);
    const uint32_t t_lo = min(all_tiles, split * per_split), n_tiles = min(all_tiles, t_lo + per_split);

    // ---- requests
    rsrc_words krs, vrs;
    if (PAGED) {
        krs = make_rsrc_words(a.k, a.pool_bytes32), vrs = make_rsrc_words(a.v, a.pool_bytes32);
    } else {
        krs = make_rsrc_words(a.k + (size_t)kvh * a.k_stride_h, kv_end * (uint32_t)ROWB);
        vrs = make_rsrc_words(a.v + (size_t)kvh * a.v_stride_h, kv_end * (uint32_t)ROWB);
    }
    const uint32_t page_bytes = a.n_kv_heads * a.block_size * (uint32_t)ROWB;  // of one page, all heads
    const uint32_t bs_shift = a.block_shift;
    // Paged: where the 16-row groups of the wave's next 32 tiles lie, group l % 2 of tile l / 2 in lane l: page, offset in a pool of less
    // than 4 GiB, and the end of the rows that are wanted of the group. (Worked out for each request, from a page id that came
    // through the scalar cache, that took a tile from 0.7 to 1.0 us: 500 rows after 1000, H14 / Hkv2 / D64 10.4 -> 8.7 us,
    // 500 after 1000, H16 / Hkv2 / D128 17.2 -> 13.1.)
    int32_t page_ids = 0, page_off = 0, page_end = 0;
    auto fetch_pages = [&](uint32_t first_tile) __attribute__((always_inline)) {
        if (PAGED) {
            const uint32_t key = (first_tile + NW * ((uint32_t)lane >> 1)) * KT + 16 * ((uint32_t)lane & 1u), end = min(kv_end, n_tiles * KT);
            const uint32_t entry = bs_shift < 32 ? key >> bs_shift : key / a.block_size, rip = key - entry * a.block_size;
            page_ids = key < end ? a.block_table[entry] : 0;
            page_off = (int)((uint32_t)page_ids * page_bytes + (kvh * a.block_size + rip) * (uint32_t)ROWB);
            page_end = page_off + (int)((key < end ? min(16u, end - key) : 0u) * (uint32_t)ROWB);
        }
    };
    const int k_src = rows16_lane_src(lane, ROWB);
    const int v_src = ((lane / (16 * COLS)) * 4 + ((lane & 15) >> 2)) * ROWB + ((lane >> 4) % COLS) * 64 + (lane & 3) * 16;
    // K or V of a tile into this wave's part of the LDS. (A tile past the last is requested from an empty range: nothing is read, zeros
    // arrive, and the counts that the waits go by stay the same.)
    auto request = [&](bool is_k, uint32_t tile, uint32_t nth /* of the fetched ones */) __attribute__((always_inline)) {
        const uint32_t dst = lds_addr + (uint32_t)wave * TILE + (is_k ? 0 : HALF);
        auto rows16 = [&](int g, const rsrc_words &rs, int so) __attribute__((always_inline)) {
            if (is_k) buffer_to_lds_b128<COLS, 64, 1024>(rs, dst + g * RB_BYTES, k_src, so);
            else buffer_to_lds_b128<COLS, 1024, 1024>(rs, dst + g * RB_BYTES, v_src, so);
        };
        if constexpr (!PAGED) {
            rsrc_words rs = is_k ? krs : vrs;
            if (tile >= n_tiles) rs.z = 0;
            rs.z = (uint32_t)__builtin_amdgcn_readfirstlane((int)rs.z);
#pragma unroll
            for (int g = 0; g < 2; ++g) rows16(g, rs, __builtin_amdgcn_readfirstlane((int)((tile * KT + 16 * g) * (uint32_t)ROWB)));
        } else {
#pragma unroll
            for (int g = 0; g < 2; ++g) {  // (a descriptor that ends with the group's last wanted row)
                const int off = __builtin_amdgcn_readlane(page_off, (int)(2 * nth + g)), end = __builtin_amdgcn_readlane(page_end, (int)(2 * nth + g));
                rsrc_words rs = is_k ? krs : vrs;
                if constexpr (POOL == 1) {
                    rs.z = (uint32_t)end;
                    rows16(g, rs, off);
                } else {
                    const size_t page = (size_t)__builtin_amdgcn_readlane(page_ids, (int)(2 * nth + g));
                    const uint32_t key = tile * KT + 16 * g, rip = bs_shift < 32 ? key & (a.block_size - 1) : key % a.block_size;
                    rs = make_rsrc_words(reinterpret_cast<const unsigned char *>(is_k ? a.k : a.v) + ((page * a.n_kv_heads + kvh) * a.block_size + rip) * (size_t)ROWB, (uint32_t)(end - off));
                    rs.x = (uint32_t)__builtin_amdgcn_readfirstlane((int)rs.x), rs.y = (uint32_t)__builtin_amdgcn_readfirstlane((int)rs.y);
                    rs.z = (uint32_t)__builtin_amdgcn_readfirstlane((int)rs.z);
                    rows16(g, rs, 0);
                }
            }
        }
    };
    constexpr int REQ = 2 * COLS;  // loads of K, or of V, of a tile
    auto wait_but = [&](auto count) __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(count)::value) : "memory"); };
    auto lds_reads_done = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
    };

    const uint32_t first_tile = t_lo + (uint32_t)wave;
    uint32_t tile = first_tile, nth = 0;  // (tile nth of those that pages have been looked up for)
    fetch_pages(tile);
    // TURN: the wave's tiles are first_tile + NW r, r < rounds, in windows of a.turn rounds from `base` on, each attended from a round
    // of its own on and around (a last window that is shorter than that round is far: from its last)
    uint32_t rounds = 0, turned = 0, base = 0, len = 0, left = 0, next = 0;
    if constexpr (TURN) {
        rounds = first_tile < n_tiles ? (n_tiles - first_tile + NW - 1) / NW : 0;
        turned = ((from_last >> a.pair_step) * 5) & (a.turn - 1);  // (neighbours far apart)
        len = left = min(a.turn, rounds), nth = next = len ? min(turned, len - 1) : 0;
        tile = first_tile + NW * nth;
    }
    auto find_next = [&]() __attribute__((always_inline)) {  // (while a tile is waited for)
        if constexpr (TURN) {
            if (--left == 0) {
                base += len, len = left = min(a.turn, rounds - base);
                next = base + (len ? min(turned, len - 1) : 0);
            } else if (++next == base + len) {
                next = base;
            }
        }
    };
    auto next_tile = [&]() __attribute__((always_inline)) {
        if constexpr (!TURN) {
            tile += NW, nth = (nth + 1) & 31u;
            if (PAGED && nth == 0) fetch_pages(tile);
        } else {
            if (PAGED && left == len && (base & 31u) == 0) fetch_pages(first_tile + NW * base);
            tile = len ? first_tile + NW * next : n_tiles, nth = next & 31u;
        }
    };
    // Query rows: 2 COLS loads of 1 KiB, one per wave as far as they go, in the layout of a K tile behind the stages
    {
        const size_t q_bytes = ((size_t)(G - 1) * a.q_stride_h + (size_t)(a.q_len - 1) * a.q_stride_m + D) * 2;
        const rsrc_words qrs = make_rsrc_words(a.q + (size_t)kvh * G * a.q_stride_h, (uint32_t)q_bytes);
#pragma unroll
        for (int i = 0; i < (2 * COLS + NW - 1) / NW; ++i) {
            const uint32_t r = (uint32_t)(wave + i * NW), g = r / COLS, col = r % COLS, row = min(row0 + 16 * g + (uint32_t)(lane >> 2), n_rows - 1);
            const uint32_t pos = position(row), at = (row - pos * G) * (uint32_t)(a.q_stride_h * 2) + pos * (uint32_t)(a.q_stride_m * 2);
            if (r >= 2 * COLS) continue;
            buffer_to_lds_b128<1, 0, 0>(qrs, lds_addr + STAGES + r * 1024, (int)(at + (uint32_t)rows16_lane_src(lane, 0)), (int)(col * 64));
        }
    }
    request(true, tile, nth), request(false, tile, nth);
    wait_but(std::integral_constant<int, 2 * REQ>{});  // this wave's part of the query rows (requested first) is there
    __syncthreads();
    h8_t qreg[DSTEPS];
    {
        const unsigned char *qp = lds + STAGES + (n >> 4) * RB_BYTES;
        const int at = rows16_operand(n, hi);
#pragma unroll
        for (int s = 0; s < DSTEPS; ++s) qreg[s] = *reinterpret_cast<const h8_t *>(qp + (s & 1 ? at ^ 32 : at) + s / 2 * 1024);
    }
    f16_t oacc[DBLKS];
#pragma unroll
    for (int b = 0; b < DBLKS; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[b][i] = 0.0f;
    float m_run = -1e30f, l_run = 0.0f;  // running max in the exp2 domain; this lane's share of the row sum
    const float c = a.scale_log2e;
    const uint32_t q_abs = position(min(row0 + (uint32_t)n, n_rows - 1)) + a.query_offset;  // last visible key of this lane's row when causal
    const uint32_t min_limit = a.causal ? pos0 + a.query_offset : 0xffffffffu;              // ... of the first row
    const int k_at = (n >> 4) * RB_BYTES + rows16_operand(n, hi);
    const int v_at = hi * RG_BYTES + ((lane & 15) >> 2) * 64 + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;

    const unsigned char *k_lds = lds + wave * TILE, *v_lds = k_lds + HALF + v_at;
    while (tile < n_tiles) {
        find_next();
        wait_but(std::integral_constant<int, REQ>{});  // K is there
        f16_t s = {};
        h8_t kk[DSTEPS];
#pragma unroll
        for (int i = 0; i < DSTEPS; ++i) kk[i] = *reinterpret_cast<const h8_t *>(k_lds + (i & 1 ? k_at ^ 32 : k_at) + i / 2 * 1024);
#pragma unroll
        for (int i = 0; i < DSTEPS; ++i) s = mfma<BF16>(kk[i], qreg[i], s);
        lds_reads_done();
        const uint32_t key0 = tile * KT;
        next_tile();
        request(true, tile, nth);
        // accumulator i is key 32 tile + 8 (i / 4) + 4 hi + i % 4
        if (key0 + KT - 1 > min_limit || key0 + KT > kv_end) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const uint32_t key = key0 + (i / 4) * 8 + hi * 4 + (i % 4);
                s[i] = key < kv_end && (!a.causal || key <= q_abs) ? s[i] : -INFINITY;
            }
        }
        float part[4] = {s[0], s[1], s[2], s[3]};
#pragma unroll
        for (int i = 4; i < 16; ++i) part[i & 3] = fmaxf(part[i & 3], s[i]);
        const u2_t mx = both_halves(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])));
        const float mloc = fmaxf(__uint_as_float(mx.x), __uint_as_float(mx.y)) * c;
        // lazy rescale: only when a row maximum has grown by more than 2^8 (the final division removes the common factor)
        if (__any(mloc > m_run + 8.0f)) {
            const float m_new = fmaxf(m_run, mloc);
            const float alpha = fast_exp2(m_run - m_new);
            l_run *= alpha;
            m_run = m_new;
#pragma unroll
            for (int b = 0; b < DBLKS; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) oacc[b][i] *= alpha;
        }
        float psum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        h8_t pb[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float p = fast_exp2(fmaf(s[i], c, -m_run));
            psum[i & 3] += p;
            pb[i / 8][i % 8] = to_elem<BF16>(p);
        }
        l_run += (psum[0] + psum[1]) + (psum[2] + psum[3]);
        wait_but(std::integral_constant<int, REQ>{});  // V is there
        // k-slot j of k-step ks <-> accumulator 8 ks + j; V operand of k-step ks: the 4-row groups 4 ks + hi and 4 ks + hi + 2
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int b = 0; b < DBLKS; ++b) {
                const unsigned char *p0 = v_lds + (ks * 4) * RG_BYTES + b * 256;
                union {
                    fp16x4_t f[2];
                    h8_t h;
                } va;
                va.f[0] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((fp16x4_t __attribute__((address_space(3))) *)(p0));
                va.f[1] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((fp16x4_t __attribute__((address_space(3))) *)(p0 + 2 * RG_BYTES));
                oacc[b] = mfma<BF16>(va.h, pb[ks], oacc[b]);
            }
        lds_reads_done();
        request(false, tile, nth);
    }
    wait_but(std::integral_constant<int, 0>{});  // (what was requested past the last tile delivered nothing, but must be over)
    __syncthreads();

    // ---- the waves' states meet: (m, l) and sums in LDS, then a thread folds its (row, 4 dims) of all waves and writes them out
    {
        const u2_t lh = both_halves(l_run);
        float *ml = reinterpret_cast<float *>(lds + NW * ACC_BYTES) + wave * 64;
        ml[lane] = hi ? __uint_as_float(lh.x) + __uint_as_float(lh.y) : m_run;  // [wave]{m[32], l[32]}
        unsigned char *acc = lds + wave * ACC_BYTES + n * 16;
#pragma unroll
        for (int b = 0; b < DBLKS; ++b)
#pragma unroll
            for (int gi = 0; gi < 4; ++gi) {  // accumulators 4 gi .. + 3 of block b are dims 32 b + 8 gi + 4 hi ..
                const f4_t v = {oacc[b][gi * 4], oacc[b][gi * 4 + 1], oacc[b][gi * 4 + 2], oacc[b][gi * 4 + 3]};
                *reinterpret_cast<f4_t *>(acc + (b * 8 + gi * 2 + hi) * QUAD_BYTES) = v;
            }
    }
    __syncthreads();
    constexpr int RPP = NW * 64 / QUADS;  // rows per pass
    const int quad = tid % QUADS;
#pragma unroll
    for (int r0 = 0; r0 < 32; r0 += RPP) {
        const int r = r0 + tid / QUADS;
        const float *ml = reinterpret_cast<const float *>(lds + NW * ACC_BYTES) + r;
        float mw[NW], m = -1e30f, L = 0.0f;
        f4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NW; ++w) mw[w] = ml[w * 64], m = fmaxf(m, mw[w]);
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float e = fast_exp2(mw[w] - m);
            L += ml[w * 64 + 32] * e;
            o += *reinterpret_cast<const f4_t *>(lds + w * ACC_BYTES + quad * QUAD_BYTES + r * 16) * e;
        }
        const uint32_t row = row0 + (uint32_t)r;
        if (row >= n_rows) continue;
        if (a.splits > 1) {  // flash_prefill.metal:592-617
            const size_t prow = (((size_t)kvh * a.n_blocks + block) * a.splits + split) * 32 + (uint32_t)r;
            *reinterpret_cast<f4_t *>(a.part_acc + prow * D + quad * 4) = o;
            if (quad == 0) *reinterpret_cast<f2_t *>(a.part_ml + prow * 2) = f2_t{m, L};
        } else {
            const float inv_l = (isfinite(L) && fabsf(L) > 1e-6f) ? (1.0f / L) : 0.0f;  // flash_prefill.metal:255-261
            h4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = to_elem<BF16>(o[e] * inv_l);
            const uint32_t pos = position(row), head = kvh * G + row - pos * G;
            *reinterpret_cast<h4_t *>(a.out + (size_t)head * a.out_stride_h + (size_t)pos * a.out_stride_m + quad * 4) = h;
        }
    }
}

template <int D, int NW, bool BF16, bool TURN>
void launch_rows(FaLaunchScope &scope, const RowsDev &a, uint32_t grid, bool paged) {
    if (!paged) scope.launch(flash_rows_kernel<D, NW, BF16, 0, TURN>, dim3(grid), dim3(NW * 64), 0, a);
    else if (a.pool_bytes32) scope.launch(flash_rows_kernel<D, NW, BF16, 1, TURN>, dim3(grid), dim3(NW * 64), 0, a);
    else scope.launch(flash_rows_kernel<D, NW, BF16, 2, TURN>, dim3(grid), dim3(NW * 64), 0, a);
}
template <int D, int NW>
void launch_rows(FaLaunchScope &scope, const RowsDev &a, uint32_t grid, bool bf16, bool paged) {
    if (bf16) a.turn ? launch_rows<D, NW, true, true>(scope, a, grid, paged) : launch_rows<D, NW, true, false>(scope, a, grid, paged);
    else a.turn ? launch_rows<D, NW, false, true>(scope, a, grid, paged) : launch_rows<D, NW, false, false>(scope, a, grid, paged);
}

}  // namespace

// log2 of how many blocks apart two blocks of a KV head are that run on the same XCD (which has every eighth pair)
static uint32_t mates_apart(uint32_t n_kv_heads) {
    uint32_t step = 0;
    while (((n_kv_heads << step) & 7u) != 0) ++step;
    return step;
}

// Which launches attend their keys in turned orders, in windows of how many rounds (0: all blocks in one order).
// Blocks of a KV head that share an XCD read the same keys. In one order they ask for the same lines at the same time, so that memory is
// asked for one block's worth of tiles and its latency stands in every round; each from another round on, the first requests of all are
// the whole window, and later rounds find it in the L2. (Memory is read once either way: 33.7 MB fetched of 33.6 MB of keys, H24 / Hkv8 /
// D128, 32 rows after 8160.) A window's tiles of all streams of an XCD (its KV heads, times the splits) take
// 3.1 MB of its 4: at 4.2 MB and beyond keys are read again (H16 / Hkv2 / D128, 30 rows after 33878, 16 splits: 29.0 us in one order, 31.7
// with windows of 4 MB, 38.9 of 8). The longer start and the scalar work of a round are 0.1 to 0.3 us: turned from 4 MB of keys on where a unit
// has one workgroup, 8 where it has several, and, split, from 9 (D 64: 16). Turned / one order in the mean of 1400 launches of 2 to 8000 rows
// after 0 to 100000, keys from memory (800 with keys in the last-level cache in brackets):
//   one workgroup   4-8 MB 0.99 (0.96)    8-16 0.86 (0.99)    from 16 0.82 (0.83)
//   several         up to 8 1.00 (1.00)   8-16 0.96 (1.00)    from 16 0.97 (0.99)
//   split, D 128    up to 9 1.04 (1.02)   9-16 0.96 (1.04)    from 16 0.94 (1.00)
//          D 64     up to 8 1.06 (1.04)   8-16 1.02 (1.05)    from 16 0.94 (1.00)
// us in one order -> turned, keys from memory:
//   H24 / Hkv8 / D128:  500 after 1000 20.5 -> 17.7; 187 after 1130 14.8 -> 12.5; 32 after 8160 18.3 -> 17.0; 68 after 13543 35.0 -> 30.6
//   H32 / Hkv8 / D128:  194 after 2151 21.1 -> 16.9; H8 / Hkv8: 1928 after 1015 34.4 -> 27.8; H16 / Hkv2: 131 after 11517 34.5 -> 29.6
//   D 64:  H32 / Hkv8, 1447 after 591 31.7 -> 27.7; H14 / Hkv2, 992 after 10818 64.8 -> 59.1
struct RowsTurn {
    uint32_t longest = 0, xcd_heads_kb = 0;  // 0: in one order
    bool wide = false;
    RowsTurn(const PrefillLaunch &L, uint32_t wgs, uint32_t n_blocks, uint32_t longest_, float kv_mb, uint32_t n_cus) : longest(longest_), wide(L.head_dim == 128) {
        if (kv_mb <= (wgs <= n_cus ? 4.0f : 8.0f) || (n_blocks - 1) >> mates_apart(L.n_kv_heads) == 0) return;
        const uint32_t twos = L.n_kv_heads & (0u - L.n_kv_heads);
        xcd_heads_kb = L.n_kv_heads / (twos < 8 ? twos : 8) * (KT * L.head_dim * 4 / 1024);  // of a tile for each wave of a stream
    }
    uint32_t operator()(uint32_t waves, uint32_t splits) const {
        if (!xcd_heads_kb) return 0;
        const uint32_t rounds = ceil_div_u32(ceil_div_u32(longest, splits), waves), held = 3100 / (xcd_heads_kb * waves * splits);
        uint32_t most = rounds < held ? rounds : held;
        most = most < 32 ? most : 32;
        const uint32_t turn = most ? 1u << (31 - __builtin_clz(most)) : 0u;
        return turn >= (wide ? 2u : 4u) ? turn : 0u;
    }
};

// How the kernel would be launched, and what that takes by estimate: fitted to 2664 shapes (2 to 8000 rows after 0 to 100000, 14
// combinations of heads, each timed with every choice, with the tiled and with the short-chunk kernel, over as many layers' caches as
// put the keys in memory and not in a cache), within 5 to 7 % (rms) of the times that are near the best.
//   one launch: the time of the workgroup with the most keys, or of the compute unit with the most work: its n-th workgroup is
//   the launch's 256 n-th, later ones have fewer keys; and the tiles of all units together (their L2, their clock);
//   keys split: the longest workgroup, and the merge launch by the splits and the MB of partial states;
//   both: the MB of keys and values (of a layer; from 9 MB on the layers of a model no longer fit the last-level cache, and a unit's only
//   workgroup waits for memory in each round of its waves), and, split, what of them an XCD draws (a block's splits lie on one: with
//   few blocks the other XCDs have none).
// 8 waves, one workgroup to a CU at D 128 and two at D 64, are faster up to 256 workgroups, 4 waves (two and four) beyond.
// H24 / Hkv8 / D128, us with 8 and 4 waves: 256 rows after 2000 15.6, 15.5; 500 rows 11.2, 8.3; 500 after 1000 20.6, 17.8.
// H14 / Hkv2 / D64: 500 after 1000 7.5, 8.5; 1000 rows 7.7, 7.3; 2048 rows 17.9, 16.2.
RowsPlan fa_prefill_rows_plan(const fa_ctx *ctx, const PrefillLaunch &L) {
    RowsPlan plan;
    const uint32_t G = L.group_size;
    if (L.q_len == 0 || L.kv_len == 0 || (L.head_dim != 128 && L.head_dim != 64)) return plan;
    // 32-bit offsets of a KV head's query rows; products with the reciprocal are exact quotients
    if (((uint64_t)(G - 1) * L.q_stride_h + (uint64_t)(L.q_len - 1) * L.q_stride_m + L.head_dim) * 2 >= (1ull << 32)) return plan;
    if (G > 256 || (uint64_t)G * L.q_len >= (1ull << 24)) return plan;
    if (!L.paged && (uint64_t)L.kv_len * L.head_dim * 2 >= (1ull << 32)) return plan;  // (the tiled kernel reports it)
    const uint32_t n_cus = ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u;
    const uint32_t n_blocks = ceil_div_u32(G * L.q_len, 32), wgs = L.n_kv_heads * n_blocks;
    if ((uint64_t)L.n_kv_heads * n_blocks > 32 * n_cus) return plan;  // (many rows: never ahead of the tiled kernel)
    auto tiles = [&](uint32_t block) -> uint32_t {  // key tiles that a block attends
        const uint32_t last = (block * 32 + 31 < G * L.q_len ? block * 32 + 31 : G * L.q_len - 1) / G;
        const uint64_t end = L.causal ? (uint64_t)last + L.query_offset + 1 : L.kv_len;
        return (uint32_t)(((end < L.kv_len ? end : L.kv_len) + KT - 1) / KT);
    };
    const bool wide = L.head_dim == 128;
    const uint32_t longest = tiles(n_blocks - 1);
    float chain = 0.0f, n = 0.0f;
    for (uint32_t i = 0; i < wgs; i += n_cus) chain += (float)tiles(n_blocks - 1 - i / L.n_kv_heads), n += 1.0f;
    const float all = (float)wgs * (float)(longest + tiles(0)) / (float)(2 * n_cus);
    auto larger = [](float x, float y) { return x > y ? x : y; };
    const float r8 = (float)ceil_div_u32(longest, 8), r4 = (float)ceil_div_u32(longest, 4);
    const float head_mb = (float)longest * (float)(KT * L.head_dim) * 4e-6f, kv_mb = head_mb * (float)L.n_kv_heads;
    const bool waited = wgs <= n_cus && kv_mb > 9.0f;
    const RowsTurn turned(L, wgs, n_blocks, longest, kv_mb, n_cus);
    const uint32_t turn8 = turned(8, 1), turn4 = turned(4, 1);
    // (turned: 390 launches, 4 to 5 % rms)
    const float us8 = turn8 ? (wide ? 2.69f + larger(1.086f * r8, 3.11f * n + 0.122f * chain + 0.0135f * all) + (wgs <= n_cus ? 0.188f : 0.133f) * kv_mb
                                    : 3.48f + larger(0.583f * r8, 0.970f * n + 0.042f * chain + 0.0334f * all) + 0.359f * kv_mb)
                      : wide ? 2.65f + larger(1.24f * r8, 2.53f * n + 0.137f * chain + 0.0265f * all) + (waited ? 0.386f : 0.03f) * kv_mb
                             : 3.08f + larger(0.629f * r8, 0.857f * n + 0.0707f * chain + 0.02f * all) + (waited ? 0.206f : 0.055f) * kv_mb;
    const float us4 = turn4 ? (wide ? 4.93f + larger(0.638f * r4, 0.987f * n + 0.0872f * chain + 0.0565f * all) + (wgs <= n_cus ? 0.103f : 0.08f) * kv_mb
                                    : 3.17f + larger(0.434f * r4, 0.397f * n + 0.0519f * chain + 0.0243f * all) + 0.355f * kv_mb)
                      : wide ? 4.19f + larger(0.61f * r4, 0.487f * n + 0.122f * chain + 0.0515f * all) + (waited ? 0.536f : 0.065f) * kv_mb
                             : 3.25f + larger(0.453f * r4, 0.271f * n + 0.0556f * chain + 0.0408f * all) + (waited ? 0.232f : 0.074f) * kv_mb;
    plan.waves = us4 < us8 ? 4 : 8, plan.us = us4 < us8 ? us4 : us8, plan.turn = us4 < us8 ? turn4 : turn8, plan.splits = 1;
    // Keys split: all workgroups resident at once, one to a CU. (The merge launch reads the splits of a row 4, 8, 16 or 32 at a time.)
    float best = plan.us / 1.05f;
    const uint32_t most = n_cus / (ceil_div_u32(wgs, 8) * 8);
    const uint32_t twos = L.n_kv_heads & (0u - L.n_kv_heads), xcd_heads = L.n_kv_heads / (twos < 8 ? twos : 8), xcd_blocks = ceil_div_u32(wgs, 8);
    const float xcd_mb = head_mb * (float)(xcd_heads < xcd_blocks ? xcd_heads : xcd_blocks);
    for (uint32_t s = 2; s <= most && s * 4 <= longest && s <= 32; s = s == 16 ? 32 : s + 1) {
        const float r = (float)ceil_div_u32(ceil_div_u32(longest, s), 8), mb = (float)wgs * (float)(32 * L.head_dim) * (float)s * 4e-6f;
        const uint32_t turn = turned(8, s);
        const float us = turn ? (wide ? 6.99f + 1.183f * r + 0.0149f * (float)s + 0.3715f * mb + 0.0674f * kv_mb + 0.507f * xcd_mb
                                      : 6.28f + 0.674f * r + 0.0385f * (float)s + 0.4104f * mb + 0.0761f * kv_mb + 0.337f * xcd_mb)
                         : wide ? 5.77f + 1.464f * r + 0.0768f * (float)s + 0.549f * mb + 0.0547f * kv_mb + 0.35f * xcd_mb
                                : 5.28f + 0.644f * r + 0.0752f * (float)s + 0.4585f * mb + 0.0584f * kv_mb + 0.41f * xcd_mb;
        if (us < best) best = us, plan.us = us, plan.splits = s, plan.waves = 8, plan.turn = turn;
    }
    if (plan.splits > 1 && kv_mb <= (wide ? 9.0f : 16.0f)) plan.turn = 0;  // (see RowsTurn; which division is best the estimates above still tell)
    return plan;
}

fa_status fa_launch_prefill_rows(fa_ctx *ctx, const PrefillLaunch &L, const RowsPlan &plan) {
    const uint32_t G = L.group_size;
    RowsDev a;
    a.q = L.q, a.k = L.k, a.v = L.v, a.out = L.out;
    a.q_stride_h = L.q_stride_h, a.q_stride_m = L.q_stride_m, a.k_stride_h = L.k_stride_h, a.v_stride_h = L.v_stride_h;
    a.out_stride_h = L.out_stride_h, a.out_stride_m = L.out_stride_m;
    a.block_table = L.block_table;
    a.group_size = G, a.rcp_group = G > 1 ? (uint32_t)((1ull << 32) / G) + 1u : 0u;
    a.q_len = L.q_len, a.kv_len = L.kv_len, a.query_offset = L.query_offset, a.causal = L.causal ? 1u : 0u;
    a.block_size = L.block_size, a.n_kv_heads = L.n_kv_heads;
    a.pool_bytes32 = (L.paged && L.pool_bytes > 0 && L.pool_bytes < (1ull << 32)) ? (uint32_t)L.pool_bytes : 0u;
    a.block_shift = 32;
    if (L.paged && L.block_size && (L.block_size & (L.block_size - 1)) == 0) a.block_shift = (uint32_t)__builtin_ctz(L.block_size);
    a.n_blocks = ceil_div_u32(G * L.q_len, 32);
    a.scale_log2e = L.scale * 1.4426950408889634f;
    a.splits = plan.splits, a.inv_splits = fa_inverse(a.splits), a.inv_kv_heads = fa_inverse(a.n_kv_heads);
    a.part_acc = a.part_ml = nullptr;
    a.turn = plan.turn, a.pair_step = mates_apart(L.n_kv_heads);
    const uint32_t pairs = L.n_kv_heads * a.n_blocks, grid = ceil_div_u32(pairs, 8) * 8 * a.splits;
    if (a.splits > 1) {  // (at most one workgroup per CU: 4.2 MB)
        const size_t rows = (size_t)pairs * a.splits * 32, acc_bytes = rows * L.head_dim * sizeof(float);
        FA_TRY(fa_ensure_workspace(ctx, acc_bytes + rows * 2 * sizeof(float)));
        a.part_acc = (float *)ctx->workspace, a.part_ml = (float *)((char *)ctx->workspace + acc_bytes);
    }
    {
        FaLaunchScope scope(ctx, a.turn ? "flash_rows_kernel_turned" : "flash_rows_kernel", true);
        if (L.head_dim == 128) {
            if (plan.waves == 8) launch_rows<128, 8>(scope, a, grid, L.bf16, L.paged);
            else launch_rows<128, 4>(scope, a, grid, L.bf16, L.paged);
        } else {
            if (plan.waves == 8) launch_rows<64, 8>(scope, a, grid, L.bf16, L.paged);
            else launch_rows<64, 4>(scope, a, grid, L.bf16, L.paged);
        }
        FA_TRY(scope.finish());
    }
    if (a.splits == 1) return FA_OK;
    PrefillMerge g;
    g.out = L.out, g.out_stride_h = L.out_stride_h, g.out_stride_m = L.out_stride_m;
    g.part_acc = a.part_acc, g.part_ml = a.part_ml, g.n_lists = L.n_kv_heads, g.n_rows = G * L.q_len, g.group = G, g.rcp_group = a.rcp_group;
    g.splits = a.splits, g.tile_rows = 32, g.part_rows = 32;
    return fa_launch_prefill_merge(ctx, g, L.head_dim, L.bf16);
}
