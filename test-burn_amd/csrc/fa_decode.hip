// Host-side launch logic of the flash-decode kernels (partition sizing, scratch, kernel selection).
#include "fa_decode_impl.h"

#include <algorithm>
#include <mutex>

// Decode partials of the entry point that allocates nothing (fa_decode_step_fused_noalloc): every GPU the library runs
// on holds its own copy of this array until the process ends. In host code the name is only a handle for
// hipGetSymbolAddress: kernels are given the address that call returns, never the name.
static __device__ __align__(256) unsigned char scratch[FA_STATIC_SCRATCH_BYTES];

fa_status fa_decode_static_scratch(int device, void **ptr, size_t *bytes) {
    constexpr int MAX_DEVICES = 64;
    static std::mutex mu;
    static void *per_device[MAX_DEVICES] = {};
    if (device < 0 || device >= MAX_DEVICES)
        return fa_fail(FA_ERR_DEVICE_NOT_FOUND, "Device not found (device %d: the static scratch table holds %d)", device, MAX_DEVICES);
    std::lock_guard<std::mutex> lock(mu);
    if (!per_device[device]) {
        // the caller has made `device` current: the symbol resolves to that GPU's copy
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fa_fail(FA_ERR_OPERATION_FAILED, "hipGetSymbolAddress(scratch) failed on device %d: %s", device, hipGetErrorString(e));
        per_device[device] = p;
    }
    *ptr = per_device[device];
    *bytes = FA_STATIC_SCRATCH_BYTES;
    return FA_OK;
}

// One word per workgroup: the XCD it runs on.
__global__ void xcd_probe_kernel(uint32_t *out) {
    if (threadIdx.x == 0) out[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = __builtin_amdgcn_s_getreg((4 - 1) << 11 | 0 << 6 | 20);
}

fa_status fa_decode_probe_xcd(fa_ctx *ctx) {
    ctx->xcd_round_robin = false;
    const dim3 grid(12, 4, 2);  // the 3-D shape of a decode launch
    const uint32_t n = grid.x * grid.y * grid.z;
    if (!ctx->workspace || ctx->workspace_bytes < n * sizeof(uint32_t)) return FA_OK;
    uint32_t *d = (uint32_t *)ctx->workspace;
    FA_HIP(hipMemsetAsync(d, 0xff, n * sizeof(uint32_t), ctx->stream));
    hipLaunchKernelGGL(xcd_probe_kernel, grid, dim3(64), 0, ctx->stream, d);
    std::vector<uint32_t> h(n);
    FA_HIP(hipMemcpyAsync(h.data(), d, n * sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    FA_HIP(hipStreamSynchronize(ctx->stream));
    bool ok = true;
    // the first workgroup of a launch continues where the previous launch stopped: only the step of one XCD per id matters
    for (uint32_t i = 0; i < n; ++i) ok = ok && h[i] < 8u && h[i] == ((h[0] + i) & 7u);
    ctx->xcd_round_robin = ok;
    return FA_OK;
}

namespace {

// Heads of a group served by one workgroup: the largest divisor of the group that fits the MFMA N dimension.
int heads_per_workgroup(uint32_t group) {
    for (int o = fa_decode::MAX_GT; o > 1; --o)
        if (group % (uint32_t)o == 0) return o;
    return 1;
}

}  // namespace

fa_status fa_launch_decode(fa_ctx *ctx, const DecodeLaunch &L) {
    using namespace fa_decode;
    const uint32_t group = L.n_heads / L.n_kv_heads;
    const int gt = heads_per_workgroup(group);
    const uint32_t sub_per_kv = group / (uint32_t)gt;
    const uint32_t ny = L.n_kv_heads * sub_per_kv;
    const uint32_t bound = L.kv_len_bound < L.capacity ? L.kv_len_bound : L.capacity;
    if (bound == 0) return fa_fail(FA_ERR_INVALID_SHAPE, "flash decode: kv_len bound is 0");

    // Context partition per workgroup, in 16-key blocks. At most one workgroup per CU: what bounds a small launch
    // is the number of requests a CU can keep outstanding, so a CU that gets two partitions takes nearly twice as
    // long and every other one waits for it in the merge. Within that limit the partitions are as small as the
    // granularity allows, but not below one block per wave.
    // Workgroup size: 8 waves (one workgroup per CU) while the launch has at most one workgroup per CU; otherwise
    // 4 waves (two resident per CU), so that one workgroup's ~5 us of start and end overlap the other's stream and
    // the rounds of workgroups balance at a finer grain.
    uint32_t chunk = ctx->decode_variant.keys_per_split;
    const uint64_t groups = (uint64_t)L.batch * ny;
    const uint64_t n_cus = (uint64_t)(ctx->n_cus > 0 ? ctx->n_cus : 256);
    auto auto_chunk = [&](uint32_t nw, uint64_t slots) {
        const uint32_t s_max = groups >= slots ? 1u : (uint32_t)(slots / groups);
        // Long partitions are cut further, into a whole number of workgroups per slot, so that a batch of ragged
        // sequences (whose short members leave most of their partitions empty) still balances over the CUs - but
        // not too far: a workgroup costs about 5 us before and after its keys stream in at 31 KB per microsecond,
        // which 768 keys (393 KB) do not amortise when workgroups run one after the other on a CU
        // (C3, 8 waves: 62.9 us with <= 768 keys, 52.0 us with <= 1536).
        const uint32_t long_chunk = 4u * nw * MBX * BK;  // four rounds of a workgroup: 1536 keys at 8 waves
        // (One sequence has nothing to balance: its partitions stay whole, one per slot, and with every workgroup
        // resident the merge runs inside the launch instead of as a second one.)
        const uint32_t per_slot = L.batch == 1 ? 1u : ceil_div_u32(ceil_div_u32(bound, s_max), long_chunk);
        uint32_t c = ceil_div_u32(ceil_div_u32(bound, s_max * per_slot), (uint32_t)BK) * BK;
        if (c < nw * BK) c = nw * BK;
        return c;
    };
    uint32_t waves = ctx->decode_waves;  // 0 = by the rule above
    const uint32_t n4 = (uint32_t)gt * L.head_dim / 4;  // records (float4 columns of all heads) per partition
    const bool one = L.batch == 1 && ctx->decode_waves == 0;
    const bool one_pass = n4 <= 128, int8 = L.sage_fused || L.q_scale;  // (one_pass: two lanes of four waves' for each record)
    bool short_context = false;
    // As few keys as four waves have in one round of requests: one partition, which writes the output itself. (The longest sequence 80 / 120
    // keys, partitions of 64 or 128 -> one: H24 / Hkv8 / D128 5.87, 5.93 -> 4.94, 5.00 us; H16 / Hkv2 / D128 6.21, 6.30 -> 5.11, 5.24;
    // H14 / Hkv2 / D64 5.06, 4.99 -> 4.03, 4.09; 8 paged sequences of 16-140, H16 / Hkv2 / D128 7.54 -> 6.33. 180 keys in two rounds: 5.97 ->
    // 5.91, 7.13 -> 6.20, 5.06 -> 4.79, but H16 / Hkv4 5.76 -> 6.18.) Not where units go without (60 sequences of 90-100, Hkv4: 6.35, 6.81),
    // and a contiguous cache whose length the device has is asked for up to the bound: with more than two head groups the rows
    // past the length cost as much below 64 keys (a block of H24 / Hkv8: 17.6 -> 18.2) as the merge does above (18.7 -> 18.3).
    const bool whole = waves == 0 && !chunk && 2 * groups <= n_cus && (L.paged || !L.d_len || ny <= 2) && bound <= (int8 ? 8u : 3u * MBX) * BK;
    if (whole) {
        waves = 4, chunk = ceil_div_u32(bound, (uint32_t)BK) * BK;
    } else if (waves == 0) {
        const uint32_t c8 = chunk ? chunk : auto_chunk(8, n_cus);
        waves = groups * ceil_div_u32(bound, (c8 + BK - 1) / BK * BK) > n_cus ? 4u : 8u;
        // A context so short that even four waves get at most one block each (at most 64 keys per compute unit's
        // share): 4-wave workgroups, still one per CU - half the waves to start, fold and keep in step. Measured,
        // H24 / Hkv8 / D128: 512 keys 6.86 -> 6.61 us, 1024 6.90 -> 6.69, 2048 7.12 -> 6.90; H14 / Hkv2 / D64 at 1025: 6.40 -> 6.28.
        if (waves == 8 && !chunk) {
            const uint32_t s_max = groups >= n_cus ? 1u : (uint32_t)(n_cus / groups);
            short_context = ceil_div_u32(bound, s_max) <= 4u * BK;
            // One sequence: up to 128 keys to a unit's share (one round of a workgroup's three streaming waves) where the four waves
            // fold and merge their heads in one pass, up to 64 where they do not, and only as far as 64 partitions of 128 keys go, the
            // most that are merged in registers. us, the better of eight waves and 64 keys -> this:
            //   H24 / Hkv8 / D128: 2100 keys 6.41 -> 5.78, 3000 6.83 -> 6.24, 4000 7.07 -> 7.03; H32 / Hkv32 / D128: 600 6.36 -> 5.67
            //   H16 / Hkv4 / D128: 5000 8.64 -> 7.47, 8000 9.32 -> 8.73 (int8 9.1 -> 9.9: not for its four groups)
            //   H14 / Hkv2 / D64: 5000 6.89 -> 5.91, 8000 7.04 -> 6.48; eight and four waves beyond: 8300 7.12, 7.35, 10000 7.26, 7.46 (int8 7.4, 7.5)
            //   H16 / Hkv2 / D128, two passes: 6200 9.25 -> 8.65, 7000 9.35 -> 8.59, 8100 9.26 -> 8.49 (int8 6200
            //   10.2 -> 10.9: not there)
            if (one && one_pass && (!int8 || s_max > 64)) short_context = ceil_div_u32(bound, std::min(s_max, 64u)) <= 8u * BK;
            else if (one && !one_pass) short_context = short_context && bound <= (int8 ? 96u * 4u * BK : 64u * 8u * BK);
            // A batch: eight waves where four fold in two passes. (H16 / Hkv2 / D128: 2 sequences of 125-1000 tokens 8.85 -> 8.25 us, of
            // 500-4000 10.04 -> 9.27, 5 of 37-300 8.55 -> 7.87, 32 of 12-100 6.84 -> 6.29)
            else if (L.batch >= 2 && !one_pass) short_context = false;
            if (short_context) waves = 4;
        }
    }
    if (chunk == 0) {
        chunk = waves == 4 ? auto_chunk(4, short_context ? n_cus : 2 * n_cus) : auto_chunk(8, n_cus);
        if (one) {
            // One sequence of few head groups has units for more partitions than are worth their records. Up to 64 partitions are merged
            // in registers, more of them through LDS: they stay at 64 as long as that leaves four waves 128 keys, eight waves 320 (of int8
            // keys 512), beyond which eight waves have 256 and int8 keys that fold in one pass as many as the units; eight waves that
            // fold in two passes have 192 at least. us, by the units -> by this rule:
            //   H16 / Hkv2 / D128: 9000 keys 10.74 -> 9.18, 12000 11.11 -> 9.50, 16000 11.96 -> 10.23, 17000 11.56 -> 10.63, 20000 11.68 -> 11.39; 256
            //   keys: 25000 12.28 -> 12.16, 30000 12.89 -> 12.78 (64 partitions of 400 at 25000: 0.6 more); int8 20000 12.1 -> 10.7, 24000 12.5 ->
            //   11.5, from there to 32768 by what the units' number is rounded to: 26000 12.0 -> 12.4, 28000 12.7 -> 12.4, 30000 12.3 -> 12.7
            //   H14 / Hkv2 / D64: 9000 8.07 -> 7.13, 12000 8.12 -> 7.55, 17000 8.52 -> 7.53, 20000 8.69 -> 7.80; 256 keys: 25000 9.06 -> 8.80, 30000 9.05 ->
            //   8.99; int8 20000 8.9 -> 7.7, 32768 9.0 -> 8.9
            // Four waves stay at 32 as long as that leaves no more than two blocks to each of the three that stream, 96 keys: half a wave
            // merges a column then instead of a whole one. us, 64 keys -> this: H32 / Hkv4 / D128: 2560 8.20 -> 6.63, 3000 8.39 -> 7.03; H16 /
            // Hkv4 / D128: 2560 6.97 -> 6.26, 3000 6.93 -> 6.71; H16 / Hkv2 / D128: 2560 7.61 -> 7.03, 3000 7.95 -> 7.36 (int8 10.4 -> 8.7); H12 /
            // Hkv6 / D64: 3000 5.70 -> 5.04; H9 / Hkv3 / D64 0.98 to 1.03 times; 96 keys in 42 partitions: 4000 7.77 -> 8.14. Not for one or two
            // head groups of f16 that fold in one pass: 32 partitions put each of them on one XCD (below), which their rows come into no faster than
            // that, and more of them spread over all: H14 / Hkv2 / D64: 2560 5.47 -> 5.72, 3072 5.47 -> 5.77; H4 / Hkv1 / D64: 2560
            // 5.14 -> 5.75; H4 / Hkv2 / D128: 3072 6.10 -> 6.85. (int8 rows are half as many bytes: H14 / Hkv2 / D64 7.5 -> 6.9.)
            const uint32_t by64 = ceil_div_u32(ceil_div_u32(bound, 64u), (uint32_t)BK) * BK, by32 = ceil_div_u32(ceil_div_u32(bound, 32u), (uint32_t)BK) * BK;
            // Where the device has the length, or a second launch merges (a step that allocates nothing), the bound is mostly above it, and up to half
            // of it the units that 64 partitions leave idle are missed where a key is 512 bytes and the fold takes two passes: 192 keys from
            // 273 (257) on. us, by the units with records as they were (a partition's columns side by side), by 64 partitions, this; lengths of a
            // sixteenth, a quarter, half and all of the bound:
            //   H16 / Hkv2 / D128, bound 18432: 9.06 10.07 10.56 12.06, 9.64 10.21 10.42 10.76, 8.56 9.33 9.32 11.14
            //     20480: 9.28 10.19 10.60 12.22, 9.94 10.58 10.81 11.18, 8.84 9.53 9.69 11.65; allocating nothing 9.85 10.19 10.83 12.26, 11.17
            //     11.42 11.65 12.34, 9.71 9.99 10.70 12.15;  17408, 272 keys: 9.01 9.87 10.23 11.75, 9.31 9.90 10.12 10.51 (192 keys 11.22)
            //   H8 / Hkv1 / D128, bound 20480: 8.97 9.60 10.70 11.40, 9.60 10.16 10.31 10.60, 8.29 8.93 9.15 10.68
            // Elsewhere 64 partitions are ahead at every length, or lose less at short ones than they gain (H16 / Hkv2 / D128, bound 16384: by the
            // units as they were 9.50 10.26 10.78 12.30, 8.79 9.28 9.67 10.04; 8192, allocating nothing: 7.95 8.32 8.88 10.25, 8.29 8.53 8.75 9.48; of one head
            // group, H8 / Hkv1 / D128, 16384: 8.11 8.68 9.62 11.28, 8.44 8.89 9.07 9.50).
            const bool beyond = !int8 && !one_pass && L.head_dim > 64 && (L.d_len || L.static_scratch);
            uint32_t least = 0;
            if (waves == 4) least = !short_context ? 0u : by32 <= 6u * BK && (ny > 2 || !one_pass || int8) ? by32 : std::min(8u * BK, by64);
            else if (beyond && by64 > (L.static_scratch ? 16u : 17u) * BK && by64 <= 20u * BK) least = 12u * BK;
            else if (by64 <= (int8 ? 32u : 20u) * BK) least = std::max(one_pass ? 0u : 12u * BK, by64);
            else if (!int8 || !one_pass) least = 16u * BK;
            chunk = std::max(chunk, least);
        }
    }
    chunk = (chunk + BK - 1) / BK * BK;
    // the int8 step in one launch: the open 32-row block must lie inside one partition
    if (L.sage_fused) chunk = (chunk + FA_SAGE_BLOCK - 1) / FA_SAGE_BLOCK * FA_SAGE_BLOCK;
    uint32_t S = ceil_div_u32(bound, chunk);
    // The polled merge needs every workgroup of the launch resident at once (the merging workgroup of a head group
    // occupies its compute unit while it waits) and its partials in the context's pattern-filled buffer.
    const uint64_t slots = waves == 4 ? 2 * n_cus : n_cus;
    // a workgroup reads ceil(n4 / partitions) columns of every partition (fewer than n4 + partitions records for
    // any partition count up to S), at most POLL_IPT records per thread
    const bool polled = ctx->decode_variant.merge == 2 && !L.static_scratch && S > 1 && groups * S <= slots &&
                        (size_t)groups * S * n4 * 32 <= ctx->poll_ws_bytes && (uint64_t)n4 + S <= (uint64_t)waves * 64 * POLL_IPT;
    // A paged batch whose partitions the kernel deals out by the lengths (batch_place): one round of resident workgroups, merged
    // inside the launch, from where the rule above would give a workgroup 512 keys of 128 dims or more - below that a workgroup has
    // one round of requests whatever its keys, and looking for its place is not repaid (Hkv 2, D 128, 8 sequences of 500 to 4000
    // tokens, 256 keys: 10.3 -> 12.4 us). Eight waves while there are two slots per sequence, four (twice the slots) beyond; with
    // fewer than two the quotients leave too much idle. us per step, by the bound and by the lengths:
    //   Hkv 2, D 128: 24 sequences of 100-4000 tokens 20.6 -> 17.8, 32 of 512-16384 59.9 -> 53.3, 64 of 16-2000 23.3 -> 19.7
    //   Hkv 8, D 128: 8 of 100-2080 13.9 -> 12.1, 8 of 100-8000 40.4 -> 31.4, 24 of 100-4000 50.5 -> 41.0 (eight waves: 48.0)
    //   Hkv 2, D 64:  40 of 16-8000 29.3 -> 21.9;  Hkv 4, D 128: 50 of 500-3000 51.8 -> 39.3
    // About equal lengths have nothing to gain and lose what reading them all takes: Hkv 2, D 128: 8 of 11000-12000 21.6 -> 21.8, 24
    // of 3900-4000 22.0 -> 22.8; Hkv 8, D 128: 8 of 2000 15.5 -> 15.8, 8 of 4000 25.6 -> 25.9; Hkv 4, D 128: 8 of 3000-4000 15.0 -> 15.6.
    // Its workgroups wait for each other (the polled merge) only where those of the rule above would. Where that rule has more
    // workgroups than fit at once, and so a merge that waits for nobody, the last one of a sequence to finish merges it: 1.2 to 1.6
    // us more than polled (32 of 512-16384: 52.2 against 53.4; 8 of 100-8000, Hkv 8: 29.9 against 31.3), and right on a GPU that
    // other work has part of, as those batches were before.
    uint32_t bal_slots = 0;
    if (L.paged && L.d_len && L.batch >= 2 && L.batch <= 64 && ctx->decode_variant.keys_per_split == 0 && ctx->decode_variant.merge == 2 &&
        !L.static_scratch && bound <= (1u << 24) && auto_chunk(8, n_cus) * L.head_dim >= 512u * 128u) {
        const uint32_t per8 = (uint32_t)(n_cus / ny);
        const uint32_t w = ctx->decode_waves ? ctx->decode_waves : 2u * L.batch <= per8 ? 8u : 4u;
        const uint32_t n = w == 4u ? 2u * per8 : per8;
        if (n >= 2u * L.batch && (size_t)n * ny * n4 * 32 <= ctx->poll_ws_bytes) bal_slots = S = n, waves = w;
    }
    // a contiguous cache slab is addressed with 32-bit byte offsets (tile base included)
    if (!L.paged && ((uint64_t)L.capacity + chunk + MBX * BK) * L.head_dim * 2 >= (1ull << 32))
        return fa_fail(FA_ERR_INVALID_SHAPE, "flash decode: one KV head of the contiguous cache must stay below 4 GiB");

    DecodeDev a;
    memset(&a, 0, sizeof(a));
    a.q = (const __half *)L.q, a.k = (const __half *)L.k, a.v = L.v, a.out = L.out;
    a.q_stride_b = L.q_stride_b, a.q_stride_h = L.q_stride_h, a.k_stride_b = L.k_stride_b, a.k_stride_h = L.k_stride_h;
    a.v_stride_b = L.v_stride_b, a.v_stride_h = L.v_stride_h, a.out_stride_b = L.out_stride_b;
    a.out_stride_h = L.out_stride_h;
    a.d_len = L.d_len, a.block_table = L.block_table;
    a.kv_len = L.kv_len, a.d_len_stride = L.d_len_stride, a.kv_len_add = L.kv_len_add, a.kv_len_bound = bound;
    a.capacity = L.capacity, a.chunk = chunk, a.n_kv_heads = L.n_kv_heads, a.sub_per_kv = sub_per_kv;
    a.gt = (uint32_t)gt;
    a.bf16 = L.bf16 ? 1u : 0u;
    a.bt_stride = L.bt_stride, a.block_size = L.block_size;
    a.block_shift = (L.block_size && (L.block_size & (L.block_size - 1)) == 0) ? (uint32_t)__builtin_ctz(L.block_size) : 32u;
    a.merge_in_kernel = ctx->decode_variant.merge == 0 ? 1u : 0u;
    a.scale_log2e = L.scale * 1.4426950408889634f;
    a.q_scale = L.q_scale, a.k_scale = L.k_scale, a.ks_stride = L.ks_stride;
    a.k_in = L.k_in, a.v_in = L.v_in, a.cos_t = L.cos_t, a.sin_t = L.sin_t, a.q_rot_out = L.q_rot_out;
    a.qin_stride_b = L.qin_stride_b, a.kvin_stride_b = L.kvin_stride_b, a.qrot_stride_b = L.qrot_stride_b;
    a.rope_normal = L.rope_normal, a.apply_rope = L.apply_rope, a.table_rows = L.table_rows;
    a.status = ctx->d_status;
    a.sage_tail = L.sage_tail, a.sage_mean = L.sage_mean, a.q_q_out = L.q_q_out, a.q_scale_out = L.q_scale_out;
    uint32_t ny_grid = ny;  // the grid's y dimension (see the padded form below)
    if (bal_slots) {
        auto rcp = [](uint32_t d) { return (uint32_t)((1ull << 32) / d) + 1u; };  // (exact for the few hundred workgroups of such a launch)
        const uint32_t per_xcd = ctx->xcd_round_robin && bal_slots * ny % 8 == 0 ? bal_slots * ny / 8 : 0u;
        // Dealt evenly: within the slots that a KV head has on one XCD, where every XCD gets a sequence.
        uint32_t cell = bal_slots, per_cell = L.batch;
        if (per_xcd && bal_slots % per_xcd == 0) {
            const uint32_t cells = bal_slots / per_xcd, seqs = ceil_div_u32(L.batch, cells);
            if (cells <= L.batch && per_xcd >= 2 * seqs) cell = per_xcd, per_cell = seqs;
        }
        const uint32_t even = cell / per_cell < 64u ? cell / per_cell : 64u;
        a.bal_seqs = L.batch | even << 8 | per_cell << 16, a.bal_slots = cell | per_xcd << 16;
        a.rcp_gx = rcp(bal_slots), a.rcp_even = rcp(even), a.rcp_cell = rcp(cell);
    }
    if (polled) {
        a.merge_in_kernel = 2u;
        a.xcd_local = !bal_slots && ctx->xcd_round_robin && groups % 8 == 0 && S <= 64 ? 1u : 0u;  // (up to 64: merged in registers)
        // Fewer than 8 head groups (Qwen2.5-0.5B has 2 KV heads) and few enough partitions for an XCD to hold a group's
        // workgroups: the grid is padded to 8 head groups, group g's workgroups land on XCD g, and the workgroups of
        // the groups that do not exist leave at once. Such a launch is all latency (its partitions were sized for that
        // above), and the exchange through one XCD's L2 is most of a microsecond shorter than through device-coherent
        // accesses (6.15 -> 5.4 us per launch at 1K context). A workgroup to a compute unit: with up to two, the XCDs of the groups
        // are what the launch waits for (H14 / Hkv2 / D64, 2100 keys, 33 partitions 6.74 padded, 6.19 not, 4000 keys 7.50, 6.68; H16 / Hkv4 /
        // D128, 4000 8.86, 8.12), except with three groups and more of int8 rows (4000 keys 10.6, 10.8) or many records (H32 / Hkv4 /
        // D128, 2100 keys 9.61, 9.96), and with int8 rows and many records whatever the groups (H16 / Hkv2 / D128 int8, 3200 / 3600 / 4000
        // keys 10.04, 10.42 / 9.53, 9.82 / 9.80, 10.03; H16 / Hkv1 / D64 9.12, 9.40 / 8.59, 8.92 / 8.80, 8.92; of one and two
        // groups with few records 0.96 to 1.02 times).
        if (!a.xcd_local && ctx->xcd_round_robin && L.batch == 1 && groups < 8 && waves == 4) {  // (only the 4-wave kernels know of the padding)
            const uint64_t per_xcd = std::min<uint64_t>(64u, ((int8 ? ny > 2 || !one_pass : ny > 2 && !one_pass) ? 2u : 1u) * (n_cus / 8u));
            const size_t need_pad = (size_t)8 * S * n4 * 32;
            if (S <= per_xcd && (uint64_t)8 * S <= slots && need_pad <= ctx->poll_ws_bytes) ny_grid = 8, a.xcd_local = 1u, a.ny_real = ny;
        }
        a.poll_ticks = (unsigned long long)ctx->poll_spin_us * 100ull;
    } else if (bal_slots) {
        a.merge_in_kernel = 1u;
    }
    if (L.static_scratch) {
        // Nothing may be allocated on this path: no workspace growth, no event creation. The partitions' partial
        // states go to the static device array and a second launch merges them (no arrival counters to keep zero).
        if (ctx->profiling)
            return fa_fail(FA_ERR_OPERATION_FAILED, "the entry point that allocates nothing cannot run with per-kernel profiling enabled (events are created per launch)");
        a.merge_in_kernel = 0;
    }
    if (S > 1) {
        const size_t rows = (size_t)(bal_slots ? 1u : L.batch) * ny * S * gt;
        const size_t acc_bytes = rows * L.head_dim * sizeof(float);
        const size_t ml_bytes = rows * 2 * sizeof(float);
        if (L.static_scratch) {
            if (acc_bytes + ml_bytes > ctx->static_scratch_bytes || !ctx->static_scratch)
                return fa_fail(FA_ERR_INVALID_SHAPE,
                               "Invalid shape: this decode launch needs %zu bytes of partition partials (%u partitions x %u head rows), "
                               "the static scratch of the entry point that allocates nothing holds %zu",
                               acc_bytes + ml_bytes, S, (uint32_t)(L.batch * ny * gt), ctx->static_scratch_bytes);
            a.part_acc = (float *)ctx->static_scratch;
            a.part_ml = (float *)((char *)ctx->static_scratch + acc_bytes);
        } else if (polled) {
            a.part_acc = (float *)ctx->poll_ws;
            a.part_ml = nullptr;
        } else {
            FA_TRY(fa_ensure_workspace(ctx, acc_bytes + ml_bytes));
            FA_TRY(fa_ensure_counters(ctx, L.batch * ny));
            a.part_acc = (float *)ctx->workspace;
            a.part_ml = (float *)((char *)ctx->workspace + acc_bytes);
            a.counters = ctx->counters;
        }
    }
#ifdef FA_DECODE_TRACE
    a.trace = (ctx->clock_buf && (uint64_t)S * ny_grid * L.batch * (waves * 16 / 2) <= ctx->clock_buf_workgroups) ? ctx->clock_buf : nullptr;
#endif
    int mode = MODE_PLAIN;
    if (L.sage_fused)
        mode = MODE_SAGE_FUSED;
    else if (L.q_scale)
        mode = MODE_SAGE;
    else if (L.fused)
        mode = L.paged ? MODE_FUSED_PAGED : MODE_FUSED;
    else if (L.paged)
        mode = MODE_PAGED;
    if (!bal_slots) {  // (divisions that every wave would otherwise do before its first request)
        const uint32_t streaming = (mode == MODE_FUSED || mode == MODE_FUSED_PAGED || mode == MODE_SAGE_FUSED) ? waves - 1 : waves;
        a.nb_q = (chunk / BK) / streaming, a.nb_r = (chunk / BK) % streaming;
    }
    dim3 grid(S, ny_grid, bal_slots ? 1u : L.batch);
    if (a.xcd_local) {
        // the kernel's reciprocals (see there): every workgroup index and both divisors stay below 2^16
        // (a divisor of 1 has no such reciprocal in 32 bits)
        if ((uint64_t)S * ny_grid * L.batch >= 65536u || S >= 65536u || ny_grid >= 65536u || S < 2 || (ny_grid < 2 && !a.ny_real)) a.xcd_local = 0;
        else a.rcp_gx = (uint32_t)((1ull << 32) / S) + 1u, a.rcp_gy = (uint32_t)((1ull << 32) / ny_grid) + 1u;
    }
    if (L.head_dim == 128) return waves == 4 ? fa_decode_launch_d128_w4(ctx, a, grid, mode) : fa_decode_launch_d128(ctx, a, grid, mode);
    if (L.head_dim == 64) return waves == 4 ? fa_decode_launch_d64_w4(ctx, a, grid, mode) : fa_decode_launch_d64(ctx, a, grid, mode);
    return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "Flash Decode only supports head_dim=64 or 128, got %u", L.head_dim);
}
