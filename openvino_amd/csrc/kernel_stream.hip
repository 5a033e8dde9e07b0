// Weight-streaming kernel for a few rows (up to 48) of large tiled nodes.
//
//   grid = (ceil(N / 16 / 8), split along K, slices of a grouped launch), block = 512: eight waves, each with a channel
//   tile of its own whose weights go straight from memory into the MFMA weight operand, a stage (two k-blocks) at a
//   time, three stages ahead (four of 4-bit weights, which are half as large).  The activations of a stage, 16 MT rows x 256 inputs, pass through registers into
//   one of two LDS buffers that all eight waves read: one barrier per stage, which waits for LDS only.
//
// The small-batch kernel (kernel_batch.hip) brings a workgroup's whole slice of X to LDS before the first product and
// has to cut K until that slice fits (8192 inputs of 32 rows: eight parts), so a launch is a chain of round trips --
// slice, weights, partial tiles out, ticket, partial tiles back.  Here K is cut only to fill the chip (plan_stream), the
// weight stream starts with the wave and never pauses.  Bound by HBM for 8-bit nodes: u8 8192 -> 57344 at 24 rows runs
// at 5.7 TB/s (83 us; the small-batch kernel 110), 28672 -> 8192 at 5.3 (44; 71); a layer of four such nodes at 24 rows
// went from 231 to 165 us.  4-bit nodes of 10-60 MB are bound by the start and the fix-up of a launch: i4 in groups of
// 64, 4096 -> 6144 at 24 rows 12.3 -> 9.8 us.
//
// Arithmetic as in the small-batch kernel: exact halves q - zp, v_mfma_f32_16x16x32_f16 with A = activations, the f32
// partial sum of a group multiplied by its scale in f32 -- once at the end where a channel has one scale, whose k-blocks
// are summed from zero each and added two at a time.  (One chain of MFMAs over a whole part of K rounds worse: u8 28672
// -> 1024 at 24 rows 2.4e-7 from 64 bits against 0.9e-7, the small-batch kernel 1.2e-7.  It was 3 % faster at 33-48 rows,
// 1 % up to 16; a wait for the matrix cores after every k-block would cost 4 % and 1 %.)  Split parts are parked with
// device-scope stores and added by the last to arrive, always in the same order, four at a time.
#include "device_common.h"

namespace ovfcc {

namespace {

constexpr int SR_WAVES = kStreamWaves;
constexpr int SR_PITCH = 2 * kBlockK + 8;  // halves per staged row; 16 bytes of padding spread the rows over the banks

// What a workgroup multiplies: one node, or one slice of a grouped launch.
struct StreamItem {
    const uint4_t* w;
    const half_t* scale;
    const uint8_t* zp;
    const half_t* bias;
    const half_t* x;
    void* y;
    const int* row_map;  // row r of the slice is row row_map[r] of x (negative: none); null: row r
    int M;
    int64_t x_rows;      // rows of x
};

struct StreamShape {
    int N, K, kb_total, kb_per_group, ng, zp_const, kb_per_split, split_k, n_tiles, out_f32, glu;
};

// MODE: 0 one scale per channel, 1 groups of whole k-blocks, 2 / 4 groups of 64 / 32 inputs (4-bit weights)
template <int BITS, int MT, bool ZP_TABLE, int MODE>
__device__ __forceinline__ void stream_body(const StreamItem& it, const StreamShape& sh, float* __restrict__ ws,
                                            unsigned* __restrict__ counters) {
    static_assert(MODE < 2 || BITS == 4, "groups below 128 inputs: 4-bit weights only");
    constexpr int TPB = BITS == 4 ? 1 : 2;              // tiles per k-block
    constexpr int DEPTH = BITS == 4 ? 4 : 3;            // stages of weights in flight or in use
    constexpr int GPB = MODE >= 2 ? MODE : 1;           // groups per k-block
    __shared__ __attribute__((aligned(16))) half_t stage_lds[2][16 * MT * SR_PITCH];
    __shared__ unsigned ticket_s;

    const int tid = threadIdx.x;
    const int lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = blockIdx.x, ks = blockIdx.y;
    const int kb_begin = ks * sh.kb_per_split, kb_end = min(sh.kb_total, kb_begin + sh.kb_per_split);
    const int stages = (kb_end - kb_begin + 1) >> 1;
    const int tile = grp * SR_WAVES + wave;
    const bool mine = tile < sh.n_tiles;  // the last workgroup may have waves without channels

    constexpr unsigned kOob = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;
    const size_t t0 = mine ? (size_t)tile : 0;
    // (the range ends with this part of K: of a stage's second k-block past it every code reads as zero, a weight of -zp)
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint4_t*>(it.w + t0 * sh.kb_total * TPB * 64), 0, mine ? kb_end * TPB * kTileBytes : 0, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(it.scale + t0 * sh.ng * 16), 0,
                                                                        mine ? sh.ng * 32 : 0, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(ZP_TABLE ? it.zp + t0 * sh.ng * 16 : it.zp), 0, ZP_TABLE && mine ? sh.ng * 16 : 0, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<half_t*>(it.x), 0, (int)(it.x_rows * sh.K * 2), kRsrcFlags);
    // kb / kb_per_group as the high word of 2 kb ceil(2^31 / kb_per_group): exact for kb kb_per_group < 2^31 (a node has
    // fewer than 2^16 k-blocks, a group at most half of them), and without a branch -- two loads of one register on two
    // sides of a branch made every stage wait for all weights in flight
    const unsigned g_mul = (unsigned)((0x80000000ull + sh.kb_per_group - 1) / sh.kb_per_group);

    // ---- activations: chunk i of the thread is eight inputs of row 16 i + (tid >> 5) ----
    unsigned x_ofs[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        int row = 16 * i + (tid >> 5);
        bool live = row < it.M;
        if (it.row_map) {
            row = live ? it.row_map[row] : -1;
            live = row >= 0;
        }
        x_ofs[i] = live ? (unsigned)(row * sh.K + (tid & 31) * 8) * 2u : kOob;
    }
    uint4_t xr[MT];
    auto load_x = [&](int s) {
        const unsigned k = (unsigned)(kb_begin + 2 * s) * kBlockK;
        // inputs past this part of K are zeros, which is what makes half a stage right: the weights that meet them are -zp
        const unsigned oob = k + (tid & 31) * 8u >= (unsigned)kb_end * kBlockK ? kOob : 0u;
#pragma unroll
        for (int i = 0; i < MT; ++i)
            xr[i] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, (x_ofs[i] + k * 2u) | oob, 0, 0));
    };
    auto store_x = [&](int b) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            *reinterpret_cast<uint4_t*>(&stage_lds[b][(16 * i + (tid >> 5)) * SR_PITCH + (tid & 31) * 8]) = xr[i];
    };
    auto barrier = [&] {  // waits for this wave's LDS accesses; its loads stay in flight
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // ---- weights and the parameters of their groups ----
    struct Slot {
        uint4_t w[2][TPB];
        uint32_t scale[2][GPB == 4 ? 2 : 1];
        uint32_t zp[2];
    };
    auto issue = [&](int s, Slot& q) {
        const unsigned past = (unsigned)((stages - 1 - s) >> 31) & kOob;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const unsigned kb = (unsigned)(kb_begin + 2 * s + b);
            const unsigned wofs = (kb * (unsigned)(TPB * kTileBytes) + lane * 16u) | past;
#pragma unroll
            for (int t = 0; t < TPB; ++t)
                q.w[b][t] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, wofs + t * kTileBytes, 0, 2));
        }
        if constexpr (MODE != 0) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const unsigned kb = (unsigned)(kb_begin + 2 * s + b);
                const unsigned g = __umulhi(2 * kb, g_mul);
                const unsigned idx = MODE == 1 ? g * 16u + col : (kb * 16u + col) * GPB;
                if constexpr (GPB == 1)
                    q.scale[b][0] = __builtin_amdgcn_raw_buffer_load_b16(rs, (idx * 2u) | past, 0, 0);
                else if constexpr (GPB == 2)
                    q.scale[b][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, (idx * 2u) | past, 0, 0);
                else {
                    const uint2_t v = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rs, (idx * 2u) | past, 0, 0));
                    q.scale[b][0] = v.x, q.scale[b][1] = v.y;
                }
                if constexpr (ZP_TABLE) {
                    if constexpr (GPB == 1)
                        q.zp[b] = __builtin_amdgcn_raw_buffer_load_b8(rz, idx | past, 0, 0);
                    else if constexpr (GPB == 2)
                        q.zp[b] = __builtin_amdgcn_raw_buffer_load_b16(rz, idx | past, 0, 0);
                    else
                        q.zp[b] = __builtin_amdgcn_raw_buffer_load_b32(rz, idx | past, 0, 0);
                }
            }
        }
    };

    load_x(0);
    Slot slot[DEPTH];
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
        issue(u, slot[u]);
    uint32_t chan_scale = 0, chan_zp = 0;
    if constexpr (MODE == 0) {
        chan_scale = __builtin_amdgcn_raw_buffer_load_b16(rs, col * 2u, 0, 0);
        if constexpr (ZP_TABLE)
            chan_zp = __builtin_amdgcn_raw_buffer_load_b8(rz, (unsigned)col, 0, 0);
    }
    store_x(0);
    load_x(1);
    barrier();

    float4_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
        acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const float zp_uniform = (float)sh.zp_const;

    auto consume = [&](int buf, const Slot& q) {
        const half_t* xs = &stage_lds[buf][col * SR_PITCH + 8 * kq];
        // one scale per channel: both k-blocks' sums first, so that the additions wait for the matrix cores once
        float4_t sums[MODE == 0 ? 2 : 1][MT];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            auto& part = sums[MODE == 0 ? b : 0];
#pragma unroll
            for (int gi = 0; gi < GPB; ++gi) {
                float zpv = zp_uniform;
                if constexpr (ZP_TABLE)
                    zpv = (float)(MODE == 0 ? chan_zp & 0xFFu : (q.zp[b] >> (8 * gi)) & 0xFFu);
                const half2_t off = splat(1024.f + zpv), off_hi = splat(64.f + zpv);
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    part[t] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = gi * (4 / GPB); j < (gi + 1) * (4 / GPB); ++j) {
                    Frag8 f;
                    if constexpr (BITS == 4)
                        unpack4(q.w[b][0][j], off, off_hi, f);
                    else
                        unpack8(q.w[b][j >> 1][2 * (j & 1)], q.w[b][j >> 1][2 * (j & 1) + 1], off, f);
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        part[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            *reinterpret_cast<const half8_t*>(xs + 16 * t * SR_PITCH + b * kBlockK + 32 * j), f.v, part[t], 0, 0, 0);
                }
                if constexpr (MODE != 0) {
                    const float scale = (float)__builtin_bit_cast(half_t, (uint16_t)(q.scale[b][gi >> 1] >> (16 * (gi & 1))));
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[t] += scale * part[t];
                }
            }
        }
        if constexpr (MODE == 0) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] += sums[0][t] + sums[1][t];
        }
    };

    for (int s0 = 0; s0 < stages; s0 += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            const int s = s0 + u;
            if (s >= stages)
                break;
            consume(s & 1, slot[u]);
            issue(s + DEPTH, slot[u]);
            store_x((s + 1) & 1);
            load_x(s + 2);
            barrier();
        }
    }

    float sum[MT][4];
    const float end_scale = MODE == 0 ? (float)__builtin_bit_cast(half_t, (uint16_t)chan_scale) : 1.f;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            sum[t][q] = MODE == 0 ? acc[t][q] * end_scale : acc[t][q];

    if (sh.split_k > 1) {
        // partial layout: [group][part][wave][MT][64 lanes] float4
        constexpr int kAuxDeviceScope = 16;  // sc1
        constexpr unsigned kPart = SR_WAVES * MT * 1024u;
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<char*>(ws) + (size_t)grp * sh.split_k * kPart, 0, sh.split_k * (int)kPart, kRsrcFlags);
        const unsigned at = (unsigned)(wave * MT * 1024 + lane * 16);
#pragma unroll
        for (int t = 0; t < MT; ++t)
            __builtin_amdgcn_raw_buffer_store_b128(
                __builtin_bit_cast(uint4_t, float4_t{sum[t][0], sum[t][1], sum[t][2], sum[t][3]}), rp,
                (unsigned)ks * kPart + at + t * 1024u, 0, kAuxDeviceScope);
        // device-scope stores write through; once every wave's are acknowledged the ticket may be drawn
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0)
            ticket_s = __hip_atomic_fetch_add(counters + grp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (ticket_s != (unsigned)(sh.split_k - 1))
            return;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                sum[t][q] = 0.f;
        for (int z0 = 0; z0 < sh.split_k; z0 += 4) {  // four parts in flight; a part past the last reads zeros
            float4_t v[4][MT];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    v[u][t] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                               rp, (unsigned)(z0 + u) * kPart + at + t * 1024u, 0, kAuxDeviceScope));
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sum[t][q] += (v[0][t][q] + v[1][t][q]) + (v[2][t][q] + v[3][t][q]);
        }
        if (tid == 0)
            __hip_atomic_store(counters + grp, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    const float bias = it.bias && mine ? (float)it.bias[tile * 16 + col] : 0.f;
    if (sh.glu) {
        // even waves own gate tiles, the next wave the matching up tile, handed over through LDS (every wave is past
        // its last stage)
        float* hand = reinterpret_cast<float*>(&stage_lds[0][0]);  // [4][MT][4][64 lanes]
        __syncthreads();
        if (wave & 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    hand[(((wave >> 1) * MT + t) * 4 + q) * 64 + lane] = sum[t][q] + bias;
        }
        __syncthreads();
        if (!(wave & 1) && mine) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int m = 4 * kq + q + 16 * t;
                    if (m < it.M)
                        store_out(it.y, (size_t)m * (sh.N / 2) + (tile >> 1) * 16 + col,
                                  glu_value(sh.glu, sum[t][q] + bias, hand[(((wave >> 1) * MT + t) * 4 + q) * 64 + lane]), sh.out_f32);
                }
        }
        return;
    }
    if (mine) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int m = 4 * kq + q + 16 * t;
                if (m < it.M)
                    store_out(it.y, (size_t)m * sh.N + tile * 16 + col, sum[t][q] + bias, sh.out_f32);
            }
    }
}

}  // namespace

// Two workgroups share a compute unit: four waves per SIMD, 128 registers each (48 rows of nodes with a zero-point table
// would take 130).
template <int BITS, int MT, bool ZP_TABLE, int MODE>
__global__ __launch_bounds__(512, 4) void fcc_stream_kernel(StreamItem it, StreamShape sh, float* __restrict__ ws,
                                                         unsigned* __restrict__ counters) {
    stream_body<BITS, MT, ZP_TABLE, MODE>(it, sh, ws, counters);
}

// Slice blockIdx.z of the table that the routing kernel wrote: at most 16 MT rows of one expert.  Slices in use come
// first in the table; the others have no rows.  Bound by the weights that the reached experts have: 6 rows through eight
// experts of 4096 / 14336, top two, take 139 us with routing and the weighted sum, the two projections fetching their
// weights at 4.5 to 4.7 TB/s.  The grouped prefill kernel, whose slices are 64 rows high at least, multiplies and unpacks
// for rows that are not there and took 195.
template <int MT, bool ZP_TABLE, int MODE>
__global__ __launch_bounds__(512) void fcc_stream_grouped_kernel(const BatchGroupItem* __restrict__ tab, StreamShape sh,
                                                                 float* __restrict__ ws, unsigned* __restrict__ counters,
                                                                 const int* __restrict__ row_map, int64_t x_rows) {
    const BatchGroupItem t = tab[blockIdx.z];
    const int rows = __builtin_amdgcn_readfirstlane(t.M);
    if (rows <= 0)
        return;
    // the same for every lane, which the compiler cannot tell (kernel_prefill_async.hip)
    StreamItem it;
    it.w = (const uint4_t*)uniform_ptr(t.w), it.scale = (const half_t*)uniform_ptr(t.scale);
    it.zp = (const uint8_t*)uniform_ptr(t.zp), it.bias = (const half_t*)uniform_ptr(t.bias);
    it.x = (const half_t*)uniform_ptr(t.x), it.y = const_cast<void*>(uniform_ptr(t.y));
    it.row_map = row_map ? row_map + __builtin_amdgcn_readfirstlane(t.reserved) : nullptr;
    it.M = rows, it.x_rows = row_map ? x_rows : rows;
    const size_t at = (size_t)blockIdx.z * gridDim.x;
    stream_body<4, MT, ZP_TABLE, MODE>(it, sh, ws + at * sh.split_k * (SR_WAVES * MT * 256), counters + at);
}

static StreamShape stream_shape(const FcDeviceArgs& a, const LaunchPlan& p) {
    const Layout& L = a.layout;
    StreamShape sh;
    sh.N = (int)a.N, sh.K = (int)a.K, sh.kb_total = (int)L.k_blocks, sh.kb_per_group = (int)L.kblocks_per_group;
    sh.ng = (int)L.groups, sh.zp_const = L.zp_const, sh.kb_per_split = p.kblocks_per_split, sh.split_k = p.split_k;
    sh.n_tiles = (int)L.n_tiles, sh.out_f32 = a.out_f32, sh.glu = L.glu;
    return sh;
}

int launch_stream(const FcDeviceArgs& a, const LaunchPlan& p, void* stream) {
    const Layout& L = a.layout;
    if (!stream_applies(a) || (int64_t)p.grid[0] * SR_WAVES < L.n_tiles || p.grid[1] != (unsigned)p.split_k ||
        (int64_t)p.split_k * p.kblocks_per_split < L.k_blocks || (p.kblocks_per_split & 1) || p.tile_m < a.M ||
        (p.split_k > 1 && !(a.workspace && a.counters)))
        return (int)hipErrorInvalidValue;
    StreamItem it;
    it.w = (const uint4_t*)a.w, it.scale = (const half_t*)a.scale, it.zp = (const uint8_t*)a.zp, it.bias = (const half_t*)a.bias;
    it.x = (const half_t*)a.x, it.y = a.y, it.row_map = nullptr, it.M = (int)a.M, it.x_rows = a.M;
    const StreamShape sh = stream_shape(a, p);
    const int mode = L.groups == 1 ? 0 : L.groups_per_kblock;
    const dim3 grid(p.grid[0], p.grid[1], 1), block(p.block);
    hipStream_t s = static_cast<hipStream_t>(stream);
#define OVFCC_STREAM(B, T, Z, G) hipLaunchKernelGGL((fcc_stream_kernel<B, T, Z, G>), grid, block, 0, s, it, sh, a.workspace, a.counters)
#define OVFCC_STREAM_MT(B, Z, G)                                   \
    do {                                                           \
        if (p.tile_m == 16)                                        \
            OVFCC_STREAM(B, 1, Z, G);                              \
        else if (p.tile_m == 32)                                   \
            OVFCC_STREAM(B, 2, Z, G);                              \
        else                                                       \
            OVFCC_STREAM(B, 3, Z, G);                              \
    } while (0)
#define OVFCC_STREAM_ZP(B, G)                                      \
    do {                                                           \
        if (L.zp_table)                                            \
            OVFCC_STREAM_MT(B, true, G);                           \
        else                                                       \
            OVFCC_STREAM_MT(B, false, G);                          \
    } while (0)
    if (L.bits == 8) {
        if (mode == 0)
            OVFCC_STREAM_ZP(8, 0);
        else
            OVFCC_STREAM_ZP(8, 1);
    } else if (mode == 0)
        OVFCC_STREAM_ZP(4, 0);
    else if (mode == 1)
        OVFCC_STREAM_ZP(4, 1);
    else if (mode == 2)
        OVFCC_STREAM_ZP(4, 2);
    else
        OVFCC_STREAM_ZP(4, 4);
#undef OVFCC_STREAM_ZP
#undef OVFCC_STREAM_MT
#undef OVFCC_STREAM
    return (int)hipGetLastError();
}

template <bool ZP_TABLE, int MODE>
static int launch_stream_grouped_mode(const BatchGroupItem* tab, const FcDeviceArgs& a, const LaunchPlan& p, hipStream_t s) {
    const StreamShape sh = stream_shape(a, p);
    const dim3 grid(p.grid[0], p.grid[1], p.grid[2]), block(p.block);
    auto kern = p.tile_m == 16 ? fcc_stream_grouped_kernel<1, ZP_TABLE, MODE> : fcc_stream_grouped_kernel<2, ZP_TABLE, MODE>;
    hipLaunchKernelGGL(kern, grid, block, 0, s, tab, sh, a.workspace, a.counters, a.row_map, a.x_rows);
    return (int)hipGetLastError();
}

int launch_stream_grouped(const BatchGroupItem* tab, const FcDeviceArgs& a, const LaunchPlan& p, void* stream) {
    const Layout& L = a.layout;
    if (!tab || !p.stream || !L.tiled || L.bits != 4 || (int64_t)p.grid[0] * SR_WAVES < L.n_tiles ||
        p.grid[1] != (unsigned)p.split_k || (int64_t)p.split_k * p.kblocks_per_split < L.k_blocks || (p.kblocks_per_split & 1) ||
        (p.tile_m != 16 && p.tile_m != 32) || (p.split_k > 1 && !(a.workspace && a.counters)) ||
        a.K * 2 * p.tile_m >= ((int64_t)1 << 31) ||
        (a.row_map && (a.x_rows < 1 || a.x_rows * a.K * 2 >= ((int64_t)1 << 31))))
        return (int)hipErrorInvalidValue;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int mode = L.groups == 1 ? 0 : L.groups_per_kblock;
#define OVFCC_STREAM_MODE(G) \
    (L.zp_table ? launch_stream_grouped_mode<true, G>(tab, a, p, s) : launch_stream_grouped_mode<false, G>(tab, a, p, s))
    return mode == 0 ? OVFCC_STREAM_MODE(0) : mode == 1 ? OVFCC_STREAM_MODE(1) : mode == 2 ? OVFCC_STREAM_MODE(2) : OVFCC_STREAM_MODE(4);
#undef OVFCC_STREAM_MODE
}

}  // namespace ovfcc
