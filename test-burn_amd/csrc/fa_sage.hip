// Sage-style int8 quantisers for the decode path (K mean-smoothing, per-32-token K scales, per-head Q scale).
// The reference holds only a prose design for this variant (docs/SAGE.md:51-65,117-126; docs/FLASH.md:153-170).
// Every step is elementwise f32 with IEEE division and round-half-even, so results are reproducible
// bit for bit on the host given the same mean.
#include "fa_internal.h"
#include "fa_sage_quant.h"

namespace {

typedef float sg_f4_t __attribute__((ext_vector_type(4)));
typedef unsigned int sg_u4_t __attribute__((ext_vector_type(4)));
typedef unsigned int sg_u2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float h_lo(unsigned w) { return __half2float(__ushort_as_half((unsigned short)(w & 0xffffu))); }
__device__ __forceinline__ float h_hi(unsigned w) { return __half2float(__ushort_as_half((unsigned short)(w >> 16))); }

// Column sums of K over the sequence, as a streaming reduction: the kernel only reads (and stores a few KB of partial
// sums), 16 bytes per lane and request, MEAN_UNROLL requests per lane in flight before the first is used (non-temporal:
// the rows are read once). A workgroup of 256 threads owns `rows_per_part` consecutive rows of one head; thread t reads
// dims 8 (t % CPR) .. of rows t / CPR, + RPI, ... (CPR = D / 8 chunks per row, RPI = 256 / CPR rows per pass) and keeps
// 8 f32 sums; the RPI row lanes of a column are then added through LDS in lane order. A second, small launch adds the
// parts in part order and divides (tickets that let the last workgroup of a head finish inside the first launch were
// measured: a thousand device-scope atomics on a handful of counters cost more than the second launch).
constexpr int MEAN_UNROLL = 8;
constexpr uint32_t MEAN_MAX_PARTS = 1024;

template <int D>
__global__ void __launch_bounds__(256)
sage_k_colsum_kernel(const __half *k, uint32_t capacity, uint32_t kv_len, uint32_t rows_per_part, uint32_t n_parts,
                     float *partial) {
    constexpr int CPR = D / 8, RPI = 256 / CPR;
    __shared__ float sm[256 * 8];
    const uint32_t h = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
    const uint32_t ch = tid % CPR, rl = tid / CPR;
    const uint32_t r0 = part * rows_per_part, r1 = min(kv_len, r0 + rows_per_part);
    const __half *base = k + ((size_t)h * capacity) * D + ch * 8;
    float s[8] = {};
    for (uint32_t r = r0 + rl; r < r1; r += RPI * MEAN_UNROLL) {
        sg_u4_t x[MEAN_UNROLL];
#pragma unroll
        for (int u = 0; u < MEAN_UNROLL; ++u) {
            const uint32_t row = r + u * RPI;
            x[u] = row < r1 ? __builtin_nontemporal_load(reinterpret_cast<const sg_u4_t *>(base + (size_t)row * D)) : sg_u4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int u = 0; u < MEAN_UNROLL; ++u) {
#pragma unroll
            for (int w = 0; w < 4; ++w) s[2 * w] += h_lo(x[u][w]), s[2 * w + 1] += h_hi(x[u][w]);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) sm[i * 256 + tid] = s[i];
    __syncthreads();
    if (tid < D) {
        // column d = tid: chunk d / 8, element d % 8, the RPI row lanes in order
        const uint32_t c = tid / 8, e = tid % 8;
        float t = 0.0f;
        for (uint32_t j = 0; j < (uint32_t)RPI; ++j) t += sm[e * 256 + j * CPR + c];
        partial[((size_t)h * n_parts + part) * D + tid] = t;
    }
}

// The order in which the parts of a head are added up, whoever does it: part lane l (of MEAN_LANES) takes the parts l, l +
// MEAN_LANES, ... one after the other, the lanes are added in a tree, l with l + 32, l + 16, ..., l + 1. `lane_tree` is the last part of
// it: v[i] holds lane first + i * STRIDE, for which it leaves the sum in v[0].
constexpr int MEAN_LANES = 64;

template <typename T, int N>
__device__ __forceinline__ T lane_tree(T (&v)[N]) {
#pragma unroll
    for (int half = N / 2; half >= 1; half >>= 1) {
#pragma unroll
        for (int i = 0; i < half; ++i) v[i] += v[i + half];
    }
    return v[0];
}

// The mean as a launch of its own: a workgroup of 1024 threads owns MEAN_FIN_COLS columns of one head, so that a launch has
// D / MEAN_FIN_COLS workgroups per head and every thread adds at most a few parts, all of its loads in flight at once. Thread
// (column d = tid % COLS, part lane tid / COLS); the first wave adds the lanes, 16 to a thread and the last four by lane
// exchanges. Latency-bound: with one workgroup of 256 threads per head, 32 dependent batches of loads deep, SmolLM3 at 32K
// (4 heads x 512 parts x 128 columns, 1 MB) took 8.0 us.
constexpr int MEAN_FIN_COLS = 16, MEAN_FIN_NT = MEAN_FIN_COLS * MEAN_LANES;
constexpr int MEAN_FIN_LOADS = MEAN_MAX_PARTS / MEAN_LANES;  // parts per thread at most

template <int D>
__global__ void __launch_bounds__(MEAN_FIN_NT)
sage_k_mean_finish_kernel(const float *partial, uint32_t n_parts, uint32_t kv_len, float *mean) {
    __shared__ float sm[MEAN_FIN_NT];
    const uint32_t h = blockIdx.y, tid = threadIdx.x;
    const uint32_t d = blockIdx.x * MEAN_FIN_COLS + tid % MEAN_FIN_COLS, pl = tid / MEAN_FIN_COLS;
    const float *hp = partial + (size_t)h * n_parts * D + d;
    float v[MEAN_FIN_LOADS];
#pragma unroll
    for (int u = 0; u < MEAN_FIN_LOADS; ++u) {
        const uint32_t p = pl + u * MEAN_LANES;
        v[u] = p < n_parts ? hp[(size_t)p * D] : 0.0f;
    }
    float t = 0.0f;
#pragma unroll
    for (int u = 0; u < MEAN_FIN_LOADS; ++u) t += v[u];
    sm[tid] = t;
    __syncthreads();
    if (tid >= 64) return;
    constexpr int PER = 64 / MEAN_FIN_COLS;  // lanes of the tree that are threads of the wave
    float l[MEAN_LANES / PER];
#pragma unroll
    for (int i = 0; i < MEAN_LANES / PER; ++i) l[i] = sm[tid + 64 * i];
    t = lane_tree(l);
#pragma unroll
    for (int half = 64 / 2; half >= MEAN_FIN_COLS; half >>= 1) t += __shfl_down(t, half);
    if (tid < MEAN_FIN_COLS) mean[(size_t)h * D + d] = kv_len ? t / (float)kv_len : 0.0f;
}

// The same mean inside a workgroup of NT threads that needs all of it, where no lane has more than one part: D values into `mu`.
// Thread t asks for four columns (t % CH) of the lanes g, g + G, ... (g = t / CH, G = NT / CH groups): the tree's upper levels are sums
// of its own rows, the lower ones of the G groups' sums through LDS. Ends with a barrier.
template <int D, int NT>
struct LaneSums {
    static constexpr int CH = D / 4, G = NT / CH, NL = MEAN_LANES / G;
    static_assert(NT % CH == 0 && (G & (G - 1)) == 0 && NL >= 1 && D <= NT, "groups of whole lanes");
    sg_f4_t v[NL];
    __device__ __forceinline__ void ask(const float *parts, uint32_t n_parts) {
        const uint32_t c = threadIdx.x % CH, g = threadIdx.x / CH;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint32_t l = g + i * G;
            v[i] = l < n_parts ? *reinterpret_cast<const sg_f4_t *>(parts + (size_t)l * D + c * 4) : sg_f4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    __device__ __forceinline__ void mean(uint32_t kv_len, float (&sums)[G][D], float (&mu)[D]) {
        const uint32_t c = threadIdx.x % CH, g = threadIdx.x / CH;
        const sg_f4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < NL; ++i) v[i] = zero + v[i];  // as the one part of a lane is added to its empty sum
        *reinterpret_cast<sg_f4_t *>(&sums[g][c * 4]) = lane_tree(v);
        __syncthreads();
        if (threadIdx.x < D) {
            float t[G];
#pragma unroll
            for (int i = 0; i < G; ++i) t[i] = sums[i][threadIdx.x];
            mu[threadIdx.x] = lane_tree(t) / (float)kv_len;
        }
        __syncthreads();
    }
};

// One wave per 32-row block of one head: the block is read ONCE - 16 bytes per lane and request, all of a lane's requests in
// flight together - held in registers as f32 differences from the mean, reduced to the block's scale with lane exchanges,
// quantised and stored 8 bytes per lane and row. Lane l owns dims 8 (l % CPR) .. of rows l / CPR + RPP i. (Stored past the caches
// the build is 0.5 us shorter at 32K and the first steps that read the rows are 4.5 us longer.) Bound by its arithmetic beside its
// loads and stores, which one wave's share does not overlap: with seven instructions per value (14 before, and a branch per row)
// the build of SmolLM3's 32768 rows takes 19.0 us instead of 20.9, of 2 heads of 100000 rows 26.1 instead of 29.5.
constexpr int QUANT_NT = 256;

template <int D>
struct SageBlock {
    static constexpr int CPR = D / 8, RPP = 64 / CPR, NI = 32 / RPP;  // chunks per row, rows per pass of the wave, passes
    sg_u4_t raw[NI];
    // Everything goes through descriptors that end with the block's `rows` rows (1 .. 32): rows past them read as zero and are not
    // written, without a branch per row.
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t slab(const void *p, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
    }
    __device__ __forceinline__ void ask(const __half *src, uint32_t rows) {
        const uint32_t lane = threadIdx.x & 63u;
        const __amdgpu_buffer_rsrc_t rs = slab(src, rows * D * 2);
#pragma unroll
        for (int i = 0; i < NI; ++i)
            raw[i] = __builtin_bit_cast(sg_u4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(lane * 16 + i * RPP * D * 2), 0, 2 /* nt */));
    }
    // the rows as they are, for a `dst` of any alignment that an f16 array has
    __device__ __forceinline__ void copy(uint32_t rows, __half *dst) const {
        typedef unsigned int any_u4_t __attribute__((ext_vector_type(4), aligned(2)));
        const uint32_t lane = threadIdx.x & 63u, ch = lane % CPR, rl = lane / CPR;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const uint32_t row = rl + i * RPP;
            if (row < rows) *reinterpret_cast<any_u4_t *>(dst + (size_t)row * D + ch * 8) = raw[i];
        }
    }
    // `mean`: the head's, in global memory or LDS
    __device__ __forceinline__ void quantize(uint32_t rows, const float *mean, int8_t *dst, __half *scale) const {
        const uint32_t lane = threadIdx.x & 63u, ch = lane % CPR, rl = lane / CPR;
        const sg_f4_t m0 = *reinterpret_cast<const sg_f4_t *>(mean + ch * 8);
        const sg_f4_t m1 = *reinterpret_cast<const sg_f4_t *>(mean + ch * 8 + 4);
        const float mu[8] = {m0[0], m0[1], m0[2], m0[3], m1[0], m1[1], m1[2], m1[3]};
        float x[NI][8];
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            float peak = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                x[i][2 * w] = sage_lo_minus(raw[i][w], mu[2 * w]), x[i][2 * w + 1] = sage_hi_minus(raw[i][w], mu[2 * w + 1]);
                peak = sage_max3(peak, x[i][2 * w], x[i][2 * w + 1]);
            }
            amax = fmaxf(amax, rl + i * RPP < rows ? peak : 0.0f);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
        const __half sc16 = __float2half_rn(amax / 127.0f);
        const SageDivisor dv = sage_divisor(__half2float(sc16));
        if (lane == 0) *scale = sc16;
        const __amdgpu_buffer_rsrc_t rs = slab(dst, rows * D);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            sg_u2_t o;
#pragma unroll
            for (int w = 0; w < 2; ++w)
                o[w] = sage_quant4_i8(x[i][4 * w], x[i][4 * w + 1], x[i][4 * w + 2], x[i][4 * w + 3], dv);
            __builtin_amdgcn_raw_buffer_store_b64(o, rs, (int)(lane * 8 + i * RPP * D), 0, 0);
        }
    }
};

// Rows [row_begin, row_end). `tail` (may be null): where the exact rows of a last block that is not whole go. MEAN: the head's mean is
// not there yet and is added up from the n_parts (at most MEAN_LANES) rows of column sums of `partial`, by every workgroup for
// itself; the first one of a head stores it to `mean`.
template <int D, bool MEAN>
__global__ void __launch_bounds__(QUANT_NT)
sage_quantize_k_kernel(const __half *k, float *mean, uint32_t capacity, uint32_t row_begin, uint32_t row_end, int8_t *k_q, __half *k_scale,
                       uint32_t n_scale_blocks, __half *tail, const float *partial, uint32_t n_parts) {
    const uint32_t h = blockIdx.y, blk = row_begin / FA_SAGE_BLOCK + blockIdx.x * (QUANT_NT / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const uint32_t b0 = blk * FA_SAGE_BLOCK, rows = b0 < row_end ? min(row_end - b0, FA_SAGE_BLOCK) : 0u;
    const size_t row0 = (size_t)h * capacity + b0;
    SageBlock<D> block;
    if constexpr (MEAN) {
        typedef LaneSums<D, QUANT_NT> Sums;
        __shared__ alignas(16) float sums[Sums::G][D];
        __shared__ alignas(16) float own[D];
        Sums lanes;
        lanes.ask(partial + (size_t)h * n_parts * D, n_parts);
        block.ask(k + row0 * D, rows);
        lanes.mean(row_end, sums, own);
        if (blockIdx.x == 0 && threadIdx.x < D) mean[(size_t)h * D + threadIdx.x] = own[threadIdx.x];
        if (tail && rows < FA_SAGE_BLOCK) block.copy(rows, tail + (size_t)h * FA_SAGE_BLOCK * D);
        if (rows) block.quantize(rows, own, k_q + row0 * D, k_scale + (size_t)h * n_scale_blocks + blk);
    } else {
        if (rows == 0) return;  // uniform over the wave
        block.ask(k + row0 * D, rows);
        if (tail && rows < FA_SAGE_BLOCK) block.copy(rows, tail + (size_t)h * FA_SAGE_BLOCK * D);
        block.quantize(rows, mean + (size_t)h * D, k_q + row0 * D, k_scale + (size_t)h * n_scale_blocks + blk);
    }
}

// One workgroup of head_dim threads (<= 256) per head.
__global__ void sage_quantize_q_kernel(const __half *q, uint32_t head_dim, int8_t *q_q, float *q_scale) {
    __shared__ float sm[4];
    const uint32_t h = blockIdx.x, d = threadIdx.x;
    const float x = d < head_dim ? __half2float(q[(size_t)h * head_dim + d]) : 0.0f;
    float amax = fabsf(x);
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = 0.0f;
    for (uint32_t w = 0; w < (blockDim.x + 63) / 64; ++w) amax = fmaxf(amax, sm[w]);
    const float sc = amax / 127.0f;
    if (d == 0) q_scale[h] = sc;
    if (d < head_dim) q_q[(size_t)h * head_dim + d] = (int8_t)sage_quant_byte(x, sage_divisor(sc));
}


// Argument block of the int8 decode step's append kernel.
struct SageAppendDev {
    const __half *q, *k, *v;       // raw projections of the new token: [H * D], [Hkv * D], [Hkv * D]
    const __half *cos_t, *sin_t;   // [table_rows, D / 2]
    const float *mean;             // [Hkv, D], fixed since the cache was built
    __half *tail;                  // [Hkv, 32, D]: the exact rotated rows of the open 32-row block
    int8_t *k_q;                   // [Hkv, capacity, D]
    __half *k_scale;               // [Hkv, ceil(capacity / 32)]
    __half *v_cache;               // [Hkv, capacity, D]
    int8_t *q_q;                   // [H, D]
    float *q_scale;                // [H]
    const uint32_t *d_position;    // nullable
    uint32_t *status;
    uint32_t position, bound, capacity, head_dim, n_heads, n_kv_heads, rope_normal, apply_rope, table_rows;
};

// Workgroups [0, Hkv): RoPE of the new K row (kv_prep_fused.metal:66-82 arithmetic, rounded once to f16), stored as row
// P % 32 of the head's tail; V row appended; then the open block (rows 32 (P / 32) .. P, all exact in the tail) is
// quantised anew with the fixed mean - scale = max|k - mean| / 127 as f16, values rint((k - mean) / scale) - so that
// the int8 rows and the scale are at every step what quantising those rows from scratch gives. A thread owns 8
// consecutive dims of one row of the block (one 16-byte load, one 8-byte store): short code - a kernel that runs for a
// few microseconds on cold state is bound by fetching its own instructions as much as by its loads.
// Workgroups [Hkv, Hkv + H): RoPE of one query head (rounded to f16, the value the f16 path would attend with), then
// its per-head int8 quantisation, one thread per dim.
__global__ void __launch_bounds__(256) sage_append_kernel(SageAppendDev a) {
    __shared__ float sm[4];
    const uint32_t D = a.head_dim, half = D >> 1, tid = threadIdx.x;
    const uint32_t n_raw = (a.d_position ? *a.d_position : a.position) + 1;
    const uint32_t lim = a.bound < a.capacity ? a.bound : a.capacity;
    if (n_raw > lim) {  // beyond the launch bound or the cache: nothing is appended (reported at the next synchronize)
        if (blockIdx.x == 0 && tid == 0 && a.status) a.status[FA_DEVSTAT_APPEND_DROPPED] = 1u;
        return;
    }
    const uint32_t P = n_raw - 1;
    const bool normal = a.rope_normal != 0, rope = a.apply_rope != 0;
    const uint32_t tp = P < a.table_rows ? P : a.table_rows - 1;
    auto rotate = [&](const __half *row, uint32_t d) -> __half {  // element d of the rotated row
#pragma clang fp contract(off)
        if (!rope) return row[d];
        const uint32_t pair = normal ? (d >> 1) : (d < half ? d : d - half);
        const bool first = normal ? ((d & 1u) == 0u) : (d < half);
        const uint32_t mate = normal ? (first ? d + 1 : d - 1) : (first ? d + half : d - half);
        const float c = __half2float(a.cos_t[(size_t)tp * half + pair]), sn = __half2float(a.sin_t[(size_t)tp * half + pair]);
        const float p0 = __half2float(row[d]) * c, p1 = __half2float(row[mate]) * sn;
        return __float2half_rn(first ? p0 - p1 : p0 + p1);
    };
    auto wg_max = [&](float v) -> float {
        for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
        if ((tid & 63) == 0) sm[tid >> 6] = v;
        __syncthreads();
        v = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
        __syncthreads();
        return v;
    };
    if (blockIdx.x < a.n_kv_heads) {
        const uint32_t h = blockIdx.x, r = P % FA_SAGE_BLOCK, b0 = P - r, cpr = D >> 3;  // 16-byte chunks per row
        __half *tail = a.tail + (size_t)h * FA_SAGE_BLOCK * D;
        union H8 {
            uint4 u;
            __half e[8];
        };
        H8 val[2];
        float x[2][8];
        float amax = 0.0f;
#pragma unroll
        for (int it = 0; it < 2; ++it) {  // 32 rows x (D / 8) chunks over 256 threads: two items at D = 128, one at D = 64
            const uint32_t item = tid + it * 256, j = item / cpr, ch = item % cpr;
            val[it].u = make_uint4(0, 0, 0, 0);
            if (j < r) {
                val[it].u = *reinterpret_cast<const uint4 *>(tail + (size_t)j * D + ch * 8);
            } else if (j == r) {
#pragma unroll
                for (int i = 0; i < 8; ++i) val[it].e[i] = rotate(a.k + (size_t)h * D, ch * 8 + i);
                *reinterpret_cast<uint4 *>(tail + (size_t)r * D + ch * 8) = val[it].u;
                *reinterpret_cast<uint4 *>(a.v_cache + ((size_t)h * a.capacity + P) * D + ch * 8) =
                    *reinterpret_cast<const uint4 *>(a.v + (size_t)h * D + ch * 8);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                x[it][i] = j <= r ? __half2float(val[it].e[i]) - a.mean[(size_t)h * D + ch * 8 + i] : 0.0f;
                amax = fmaxf(amax, fabsf(x[it][i]));
            }
        }
        amax = wg_max(amax);
        const __half sc16 = __float2half_rn(amax / 127.0f);
        const SageDivisor dv = sage_divisor(__half2float(sc16));
        if (tid == 0) a.k_scale[(size_t)h * ((a.capacity + FA_SAGE_BLOCK - 1) / FA_SAGE_BLOCK) + b0 / FA_SAGE_BLOCK] = sc16;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const uint32_t item = tid + it * 256, j = item / cpr, ch = item % cpr;
            if (j <= r) {
                const uint2 o = make_uint2(sage_quant4_i8(x[it][0], x[it][1], x[it][2], x[it][3], dv),
                                           sage_quant4_i8(x[it][4], x[it][5], x[it][6], x[it][7], dv));
                *reinterpret_cast<uint2 *>(a.k_q + ((size_t)h * a.capacity + b0 + j) * D + ch * 8) = o;
            }
        }
    } else {
        const uint32_t h = blockIdx.x - a.n_kv_heads, d = tid;
        const float x = d < D ? __half2float(rotate(a.q + (size_t)h * D, d)) : 0.0f;
        const float amax = wg_max(fabsf(x));
        const float sc = amax / 127.0f;
        if (d == 0) a.q_scale[h] = sc;
        if (d < D) a.q_q[(size_t)h * D + d] = (int8_t)sage_quant_byte(x, sage_divisor(sc));
    }
}

}  // namespace

fa_status fa_launch_sage_append(fa_ctx *ctx, const SageAppendLaunch &l) {
    SageAppendDev a;
    a.q = l.q, a.k = l.k, a.v = l.v, a.cos_t = l.cos_t, a.sin_t = l.sin_t, a.mean = l.mean, a.tail = l.tail;
    a.k_q = l.k_q, a.k_scale = l.k_scale, a.v_cache = l.v_cache, a.q_q = l.q_q, a.q_scale = l.q_scale;
    a.d_position = l.d_position, a.status = ctx->d_status;
    a.position = l.position, a.bound = l.bound, a.capacity = l.capacity, a.head_dim = l.head_dim;
    a.n_heads = l.n_heads, a.n_kv_heads = l.n_kv_heads, a.rope_normal = l.rope_normal, a.apply_rope = l.apply_rope;
    a.table_rows = l.table_rows;
    FaLaunchScope scope(ctx, "sage_append_kernel", true);
    scope.launch(sage_append_kernel, dim3(l.n_kv_heads + l.n_heads), dim3(256), 0, a);
    return scope.finish();
}

// The column sums of rows [0, kv_len) of every head, part by part, into the workspace.
static fa_status launch_colsum(fa_ctx *ctx, const void *k, uint32_t n_kv_heads, uint32_t capacity, uint32_t head_dim, uint32_t kv_len,
                               float *&partial, uint32_t &n_parts) {
    if (((uintptr_t)k & 15u) != 0) return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "the K tensor must be 16-byte aligned");
    // Parts: about eight workgroups per compute unit over all heads (a workgroup has all of a pass - 256 threads x
    // MEAN_UNROLL requests of 16 bytes = 32 KiB - in flight at once, and eight of them fit a compute unit), each a whole
    // number of passes, at most MEAN_MAX_PARTS per head.
    const uint32_t rows_per_pass = (256u / (head_dim / 8u)) * MEAN_UNROLL;
    const uint64_t n_cus = (uint64_t)(ctx->n_cus > 0 ? ctx->n_cus : 256);
    uint32_t want = (uint32_t)((8 * n_cus + n_kv_heads - 1) / n_kv_heads);
    if (want > MEAN_MAX_PARTS) want = MEAN_MAX_PARTS;
    if (want == 0) want = 1;
    const uint32_t rows_per_part = ceil_div_u32(ceil_div_u32(kv_len ? kv_len : 1u, want), rows_per_pass) * rows_per_pass;
    n_parts = ceil_div_u32(kv_len ? kv_len : 1u, rows_per_part);
    FA_TRY(fa_ensure_workspace(ctx, (size_t)n_kv_heads * n_parts * head_dim * sizeof(float)));
    partial = (float *)ctx->workspace;
    FaLaunchScope scope(ctx, "sage_k_colsum_kernel", true);
    auto kernel = head_dim == 128 ? sage_k_colsum_kernel<128> : sage_k_colsum_kernel<64>;
    scope.launch(kernel, dim3(n_parts, n_kv_heads), dim3(256), 0, (const __half *)k, capacity, kv_len, rows_per_part, n_parts, partial);
    return scope.finish();
}

static fa_status launch_mean_finish(fa_ctx *ctx, const float *partial, uint32_t n_parts, uint32_t n_kv_heads, uint32_t head_dim,
                                    uint32_t kv_len, float *mean) {
    FaLaunchScope scope(ctx, "sage_k_mean_finish_kernel", true);
    auto kernel = head_dim == 128 ? sage_k_mean_finish_kernel<128> : sage_k_mean_finish_kernel<64>;
    scope.launch(kernel, dim3(head_dim / MEAN_FIN_COLS, n_kv_heads), dim3(MEAN_FIN_NT), 0, partial, n_parts, kv_len, mean);
    return scope.finish();
}

// partial: null, or the n_parts rows of column sums that the mean is still to be made of
static fa_status launch_quantize_k(fa_ctx *ctx, const void *k, float *mean, uint32_t n_kv_heads, uint32_t capacity, uint32_t head_dim,
                                   uint32_t row_begin, uint32_t row_end, void *k_q, void *k_scale, void *tail, const float *partial,
                                   uint32_t n_parts) {
    const dim3 grid(ceil_div_u32(row_end - row_begin, FA_SAGE_BLOCK * (QUANT_NT / 64)), n_kv_heads);
    FaLaunchScope scope(ctx, "sage_quantize_k_kernel", true);
    auto kernel = head_dim == 128 ? (partial ? sage_quantize_k_kernel<128, true> : sage_quantize_k_kernel<128, false>)
                                  : (partial ? sage_quantize_k_kernel<64, true> : sage_quantize_k_kernel<64, false>);
    scope.launch(kernel, grid, dim3(QUANT_NT), 0, (const __half *)k, mean, capacity, row_begin, row_end, (int8_t *)k_q, (__half *)k_scale,
                 ceil_div_u32(capacity, FA_SAGE_BLOCK), (__half *)tail, partial, n_parts);
    return scope.finish();
}

static fa_status check_quantize_k(const void *k, const float *mean, const void *k_q) {
    if ((((uintptr_t)k | (uintptr_t)mean) & 15u) != 0 || ((uintptr_t)k_q & 7u) != 0)
        return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "K and the mean must be 16-byte aligned, the int8 cache 8-byte aligned");
    return FA_OK;
}

fa_status fa_launch_sage_k_mean(fa_ctx *ctx, const void *k, uint32_t n_kv_heads, uint32_t capacity, uint32_t head_dim,
                                uint32_t kv_len, float *mean_out) {
    float *partial;
    uint32_t n_parts;
    FA_TRY(launch_colsum(ctx, k, n_kv_heads, capacity, head_dim, kv_len, partial, n_parts));
    return launch_mean_finish(ctx, partial, n_parts, n_kv_heads, head_dim, kv_len, mean_out);
}

fa_status fa_launch_sage_quantize_k(fa_ctx *ctx, const void *k, const float *mean, uint32_t n_kv_heads,
                                    uint32_t capacity, uint32_t head_dim, uint32_t row_begin, uint32_t row_end,
                                    void *k_q, void *k_scale) {
    if (row_end <= row_begin) return FA_OK;
    FA_TRY(check_quantize_k(k, mean, k_q));
    return launch_quantize_k(ctx, k, const_cast<float *>(mean), n_kv_heads, capacity, head_dim, row_begin, row_end, k_q, k_scale, nullptr, nullptr, 0);
}

fa_status fa_launch_sage_build(fa_ctx *ctx, const void *k, uint32_t n_kv_heads, uint32_t capacity, uint32_t head_dim, uint32_t kv_len,
                               void *k_q, void *k_scale, float *mean, void *tail) {
    if (kv_len == 0) return fa_launch_sage_k_mean(ctx, k, n_kv_heads, capacity, head_dim, kv_len, mean);
    FA_TRY(check_quantize_k(k, mean, k_q));
    float *partial;
    uint32_t n_parts;
    FA_TRY(launch_colsum(ctx, k, n_kv_heads, capacity, head_dim, kv_len, partial, n_parts));
    // Where a lane has one part at most (up to 64 of them: their number grows with the rows, by one per 128 at D 128 and 256 at D 64, and
    // falls with the heads) every workgroup of the quantiser adds them up itself: a launch less for sums that are read once per 128 rows
    // from its XCD's L2. 4 heads of D 128, 300 rows 8.1 -> 6.3 us, 4000 9.6 -> 8.4, 8000 10.4 -> 10.1. What they all read again has to
    // stay small beside that launch, 24 MB at D 128 and 48 at D 64 (16 heads of D 128, 4000 rows, 8 MB 13.5 -> 12.2, 8000, 33 MB 19.1 ->
    // 19.5; 32 heads, 4000, 17 MB 19.2 -> 18.6, 8000, 65 MB 31.9 -> 33.4, 16000, 129 MB 58.8 -> 61.9; D 64, 16 heads, 16000, 32 MB 20.2 ->
    // 19.3, 32 heads, 65 MB 32.9 -> 33.1), or what each of them does: up to 32 parts, half of its own rows (64 heads of D 128, 8000 rows
    // 58.8 -> 59.4, 16000 109.7 -> 107.9, 32000 222.7 -> 217.2). Beyond 64 parts a launch of its own is ahead: 64 sums per head made by 64
    // workgroups of 1024 threads, which the quantiser could add up as well, took 21.6 us against 21.2 at 32768 rows of 4 heads, 36.8 against
    // 29.4 for 2 heads of 100000.
    const uint64_t again = (uint64_t)n_kv_heads * ceil_div_u32(kv_len, FA_SAGE_BLOCK * (QUANT_NT / 64)) * n_parts * head_dim * sizeof(float);
    const bool own_mean = n_parts <= MEAN_LANES / 2 || (n_parts <= MEAN_LANES && again <= (head_dim == 128 ? 24u : 48u) << 20);
    if (!own_mean) FA_TRY(launch_mean_finish(ctx, partial, n_parts, n_kv_heads, head_dim, kv_len, mean));
    return launch_quantize_k(ctx, k, mean, n_kv_heads, capacity, head_dim, 0, kv_len, k_q, k_scale, tail, own_mean ? partial : nullptr, n_parts);
}

fa_status fa_launch_sage_quantize_q(fa_ctx *ctx, const void *q, uint32_t n_heads, uint32_t head_dim, void *q_q,
                                    float *q_scale) {
    FaLaunchScope scope(ctx, "sage_quantize_q_kernel", true);
    scope.launch(sage_quantize_q_kernel, dim3(n_heads), dim3((head_dim + 63) / 64 * 64), 0,
                       (const __half *)q, head_dim, (int8_t *)q_q, q_scale);
    return scope.finish();
}
