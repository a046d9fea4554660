// Loads from a buffer straight into LDS (buffer_load ... lds) for the kernels that stage K/V tiles there.
#pragma once
#include "fa_internal.h"

namespace fa_lds_dma {

// 16 bytes per lane from a buffer straight into LDS: lane l's bytes land at lds_addr + imm + 16 l, read from
// base + voff + soff + imm; out-of-range lanes deliver zeros. Written as assembly so that the compiler does not
// serialise every later LDS read behind it (it cannot tell which LDS bytes such a load writes); completion is
// tracked by vmcnt, and the waits are placed by hand.
typedef unsigned int rsrc_words __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rsrc_words make_rsrc_words(const void *base, uint32_t bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    rsrc_words r;
    r.x = (uint32_t)b, r.y = (uint32_t)(b >> 32) & 0xffffu, r.z = bytes, r.w = 0x00020000u;
    return r;
}
// N such loads whose sources are SRC_STEP bytes apart and whose destinations are DST_STEP bytes apart. When the two
// steps are equal the instruction's immediate offset (which moves source and destination alike) does the stepping.
// buffer_to_lds_b128 is for tiles that other workgroups read again (they should stay in L2); buffer_to_lds_b128_nt
// marks rows that are read once per launch as non-temporal, so that a launch's stream does not push the kernel's
// own code out of L2 (a workgroup then starts with instruction fetches from memory). (When the steps differ, the
// source-offset update sits between the m0 write and the load that needs it.) A vector memory instruction must come five wait
// states after a vector instruction (v_readlane of a page's place, of a spilled scalar) that wrote a scalar it reads. The compiler keeps
// them for its own instructions and does not look into these, which had as few as two: the move to m0 and the s_nop 3 are five.
// buffer_to_lds_b128_scalar and _ahead, of the tile kernels, wait for m0 alone: their loops issue these loads one by one, and the three
// states more of each were 3 to 6 % of a launch of block-quantised weights (Q8_0, 64 rows x 3072 x 3072 11.4 -> 12.0 us, 160 rows x 2048 x
// 2048 9.4 -> 9.8; Q4_0, 160 rows x 3072 x 3072 11.8 -> 12.4). Their scalars come from the scalar unit, and that no vector instruction
// writes one of them, a spilled one's return included, less than five states ahead is looked for in the built code, with that of all other
// kernels, by tests/test_lds_load_waits.py.
#define FA_LDS_DMA_DEFINE(NAME, POLICY, NOPS) \
template <int N, int SRC_STEP, int DST_STEP> \
__device__ __forceinline__ void NAME(rsrc_words rs, uint32_t lds_addr, int voff, int soff) { \
    static_assert(N == 1 || N == 2 || N == 4, "1, 2 or 4 loads"); \
    if constexpr (SRC_STEP == DST_STEP) { \
        static_assert((N - 1) * SRC_STEP < 4096, "12-bit immediate"); \
        if constexpr (N == 4) \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop " NOPS "\n\t" \
                         "buffer_load_dwordx4 %1, %2, %3 offen" POLICY " lds" "\n\t" \
                         "buffer_load_dwordx4 %1, %2, %3 offen offset:%4" POLICY " lds" "\n\t" \
                         "buffer_load_dwordx4 %1, %2, %3 offen offset:%5" POLICY " lds" "\n\t" \
                         "buffer_load_dwordx4 %1, %2, %3 offen offset:%6" POLICY " lds" \
                         : \
                         : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff), "n"(SRC_STEP), "n"(2 * SRC_STEP), "n"(3 * SRC_STEP) \
                         : "memory"); \
        else if constexpr (N == 2) \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop " NOPS "\n\t" \
                         "buffer_load_dwordx4 %1, %2, %3 offen" POLICY " lds" "\n\t" \
                         "buffer_load_dwordx4 %1, %2, %3 offen offset:%4" POLICY " lds" \
                         : \
                         : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff), "n"(SRC_STEP) \
                         : "memory"); \
        else \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop " NOPS "\n\tbuffer_load_dwordx4 %1, %2, %3 offen" POLICY " lds" \
                         : \
                         : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff) \
                         : "memory"); \
    } else { \
        int so = soff; \
        if constexpr (N == 4) \
            asm volatile("s_mov_b32 m0, %1\n\ts_nop " NOPS "\n\t" \
                         "buffer_load_dwordx4 %2, %3, %0 offen" POLICY " lds" "\n\t" \
                         "s_add_i32 m0, %1, %5\n\ts_add_i32 %0, %0, %4\n\t" \
                         "buffer_load_dwordx4 %2, %3, %0 offen" POLICY " lds" "\n\t" \
                         "s_add_i32 m0, %1, %6\n\ts_add_i32 %0, %0, %4\n\t" \
                         "buffer_load_dwordx4 %2, %3, %0 offen" POLICY " lds" "\n\t" \
                         "s_add_i32 m0, %1, %7\n\ts_add_i32 %0, %0, %4\n\t" \
                         "buffer_load_dwordx4 %2, %3, %0 offen" POLICY " lds" \
                         : "+s"(so) \
                         : "s"(lds_addr), "v"(voff), "s"(rs), "n"(SRC_STEP), "n"(DST_STEP), "n"(2 * DST_STEP), "n"(3 * DST_STEP) \
                         : "memory", "scc"); \
        else if constexpr (N == 2) \
            asm volatile("s_mov_b32 m0, %1\n\ts_nop " NOPS "\n\t" \
                         "buffer_load_dwordx4 %2, %3, %0 offen" POLICY " lds" "\n\t" \
                         "s_add_i32 m0, %1, %5\n\ts_add_i32 %0, %0, %4\n\t" \
                         "buffer_load_dwordx4 %2, %3, %0 offen" POLICY " lds" \
                         : "+s"(so) \
                         : "s"(lds_addr), "v"(voff), "s"(rs), "n"(SRC_STEP), "n"(DST_STEP) \
                         : "memory", "scc"); \
        else \
            asm volatile("s_mov_b32 m0, %0\n\ts_nop " NOPS "\n\tbuffer_load_dwordx4 %1, %2, %3 offen" POLICY " lds" \
                         : \
                         : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff) \
                         : "memory"); \
    } \
}
FA_LDS_DMA_DEFINE(buffer_to_lds_b128, "", "3")
FA_LDS_DMA_DEFINE(buffer_to_lds_b128_scalar, "", "0")
// One such load to lds_addr + ahead, a number that is known when the kernel is built: for loops with more places in LDS than there
// are scalar registers to keep their addresses in.
__device__ __forceinline__ void buffer_to_lds_b128_ahead(rsrc_words rs, uint32_t lds_addr, uint32_t ahead, int voff, int soff) {
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff), "i"(ahead)
                 : "memory", "scc");
}
FA_LDS_DMA_DEFINE(buffer_to_lds_b128_nt, " nt", "3")
#undef FA_LDS_DMA_DEFINE

// Layout of 16 rows of K (or of query rows) in LDS, for the operand reads of a 32 x 32 x 16 matrix instruction (lane = row, 16
// bytes of it): a load fills 1 KiB with a 64-byte column of the 16 rows, [row][slot of 16 bytes], and the next loads with the next
// columns. Neighbouring lanes fetch neighbouring memory: the four lanes of a row have its 64 bytes between them, and a compute unit
// then draws 64 bytes a cycle through its address unit (131 KB/us with all CUs at it, 149 with one), where lanes that go down
// the rows first, 16 bytes each, get 16 (37 KB/us). Within a row the pieces are exchanged by row number, slot = piece ^ (row / 4) % 4,
// so that the 16 rows of an operand read lie in different banks.
__device__ __forceinline__ int rows16_lane_src(int lane, int row_stride) { return (lane >> 2) * row_stride + ((lane & 3) ^ (lane >> 4)) * 16; }
// Place of a lane's operand piece, of row `row` and lane half hi: k-step s is at (s / 2) KiB + this, with the odd steps' places ^ 32.
__device__ __forceinline__ int rows16_operand(int row, int hi) { return (row & 15) * 64 + ((hi ^ ((row >> 2) & 3)) * 16); }

}  // namespace fa_lds_dma
