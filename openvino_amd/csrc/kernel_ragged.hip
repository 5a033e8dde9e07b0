// Nodes with one scale per channel whose widths fit no tile (N = 1000, K = 1160, ...: classifier heads, encoder layers).
//
// Their weights are stored in operand order with N and K padded (Layout::ragged, ovfcc_internal.h); the activations
// stay the caller's rows of K halves and are set to zero beyond K on their way into LDS.  Weights become exact halves
// q - zp in registers, v_mfma_f32_16x16x32_f16 sums in f32, and the channel's scale multiplies the f32 sum: one
// rounding, at the output.
// MFMA roles: A = weights (rows = channels), B = activations (columns = rows m of X); the result lane holds column
// m = lane & 15, channels 4 (lane >> 4) + q.
//
// Two kernels share this arithmetic:
//   fcc_ragged_rows_kernel  few rows (plan_ragged draws the line): one workgroup per 16 channels, its waves share K (wave w: k-blocks
//                           w, w + waves, ...) and stage their own activations.  Bound by latency: a wave's life is
//                           one or two dependent loads and a reduction through LDS.
//   fcc_ragged_tile_kernel  more rows: 64 rows x 64 channels per workgroup of four waves; each wave contracts one of
//                           the four 32-input steps of a k-block against all 64 x 64 outputs, so that a weight is
//                           unpacked once per 64 rows and an activation operand read from LDS meets four MFMAs
//                           (half of what LDS delivers at the matrix cores' rate; waves side by side along N would
//                           need all of it).  Three workgroups share a compute unit and hide each other's loads,
//                           which travel two k-blocks ahead through registers: rows may start anywhere.
//   fcc_ragged_tile_dma_kernel  the same tiles where rows start at dwords: the activations go to LDS without registers
//                           or LDS stores.  577 x 1160 -> 3480 (552 tiles) 18.1 -> 15.2 us, 1160 -> 4300 18.4 -> 15.7, 4300
//                           -> 1160 23.2 -> 18.9, 1500 x 1600 -> 4800 51.5 -> 46.1; a k-block of three workgroups takes 0.97 us
//                           against 0.32 of matrix-core work (by the counters their pipe is busy 20 % of the launch and
//                           waves wait 36-39 % of their cycles).  What takes the rest: a wave's k-block holds 143 vector
//                           instructions (32 to unpack; the rest offsets, selects and moves for the row's last k-block), 11
//                           branches and 11 waits around its 16 MFMAs, and 32 load instructions a workgroup at 16
//                           cycles of the address path each would be 0.64 us (counted, not measured).  A fourth stage
//                           leaves room for two workgroups only (17.8).
// What a load costs the compute unit is the number of 64-byte pieces its 64 lanes name in lane order: weights read
// where OpenVINO left them (neighbouring lanes in different rows) kept the cache's tag stage busy every cycle of the
// launch -- 577 x 4640 -> 3480 took 61.6 us that way and takes 42.1 in operand order.
// An encoder layer of hidden size 1160 (four nodes, 577 rows) takes 66 us where one wave per output took 7 850.
#include <atomic>

#include "device_common.h"

namespace ovfcc {

namespace {

constexpr int RG_BM = kRaggedTile, RG_BN = kRaggedTile, RG_PITCH = kRaggedPitch;
constexpr int RG_STAGE_HALVES = RG_BM * RG_PITCH;
constexpr int RD_STAGES = 3;

template <class T>
__device__ __forceinline__ T load_unaligned(const void* p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

// What the channels' constants look like to a lane.
struct RaggedNode {
    const uint8_t* w;
    const half_t* scale;
    const uint8_t* zp;
    const half_t* bias;
    const half_t* x;
    void* y;
    int M, N, K;
    int zp_kind;    // 0: none (zp_const), 1: u4 packed, 2: u8
    int zp_scalar;  // one element for all channels
    int zp_const;
    int out_f32;
};

// Offsets of C channels' weights against the stored codes (signed codes are stored with their sign bit flipped); the
// loads of all of them go out before the first is used.
template <int C>
__device__ __forceinline__ void zero_points(const RaggedNode& a, const int (&n)[C], half2_t (&off)[C], half2_t (&off_hi)[C]) {
    int z[C];
    const int nibble = a.zp_kind == 1 ? 1 : 0;
#pragma unroll
    for (int i = 0; i < C; ++i)
        z[i] = 0;
    if (a.zp_kind != 0) {
#pragma unroll
        for (int i = 0; i < C; ++i)
            z[i] = a.zp[(a.zp_scalar ? 0 : n[i]) >> nibble];
        if (nibble)
#pragma unroll
            for (int i = 0; i < C; ++i)
                z[i] = (z[i] >> (a.zp_scalar ? 0 : 4 * (n[i] & 1))) & 15;
    }
#pragma unroll
    for (int i = 0; i < C; ++i)
        off[i] = splat(1024.f + (float)(z[i] + a.zp_const)), off_hi[i] = splat(64.f + (float)(z[i] + a.zp_const));
}

// The eight weights of a lane and step as exact halves.
template <int BITS>
__device__ __forceinline__ void unpack_ragged(const uint32_t (&d)[BITS / 4], half2_t off, half2_t off_hi, Frag8& f) {
    if constexpr (BITS == 8)
        unpack8(d[0], d[1], off, f);
    else
        unpack4(d[0], off, off_hi, f);
}

template <int BITS>
__device__ __forceinline__ void load_weights(const uint8_t* p, uint32_t (&d)[BITS / 4]) {
    if constexpr (BITS == 8) {
        const uint2_t v = *reinterpret_cast<const uint2_t*>(p);
        d[0] = v.x, d[1] = v.y;
    } else {
        d[0] = *reinterpret_cast<const uint32_t*>(p);
    }
}

// The eight activations of a row from input k on, zero beyond K.  The load itself stays inside the row (it begins at
// K - 8 at the latest; K >= 8): tail_shift, called for the last k-block only, moves what it got into place.
__device__ __forceinline__ uint4_t load_x(const half_t* row, int k, int K) {
    return load_unaligned<uint4_t>(row + min(k, K - 8));
}
__device__ __forceinline__ uint4_t tail_shift(uint4_t v, int k, int K) {
    const int s = max(0, k - (K - 8)), d = s >> 1;  // halves, whole dwords
    uint32_t t[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        t[i] = 0;
#pragma unroll
        for (int j = i; j < 4; ++j)
            t[i] = d == j - i ? v[j] : t[i];
    }
    const bool odd = s & 1;
    return uint4_t{odd ? __builtin_amdgcn_alignbit(t[1], t[0], 16) : t[0], odd ? __builtin_amdgcn_alignbit(t[2], t[1], 16) : t[1],
                   odd ? __builtin_amdgcn_alignbit(t[3], t[2], 16) : t[2], odd ? __builtin_amdgcn_alignbit(t[4], t[3], 16) : t[3]};
}

// Four consecutive channels n .. n + 3 of output row m.
__device__ __forceinline__ void store4(const RaggedNode& a, int m, int n, const float (&v)[4]) {
    const size_t at = (size_t)m * a.N + n;
    if (n + 4 <= a.N) {
        if (a.out_f32) {
            const float4_t o{v[0], v[1], v[2], v[3]};
            __builtin_memcpy(static_cast<float*>(a.y) + at, &o, sizeof(o));
        } else {
            const half4_t o{to_half_rne(v[0]), to_half_rne(v[1]), to_half_rne(v[2]), to_half_rne(v[3])};
            __builtin_memcpy(static_cast<half_t*>(a.y) + at, &o, sizeof(o));
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (n + q < a.N)
                store_out(a.y, at + q, v[q], a.out_f32);
    }
}

// Scales and bias of channels n .. n + 3, fetched early and kept packed.
struct ChannelParams {
    half4_t scale, bias;
};
__device__ __forceinline__ ChannelParams channel_params(const RaggedNode& a, int n) {
    ChannelParams p;
    p.bias = half4_t{0, 0, 0, 0};
    if (n + 4 <= a.N) {
        p.scale = load_unaligned<half4_t>(a.scale + n);
        if (a.bias)
            p.bias = load_unaligned<half4_t>(a.bias + n);
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = min(n + q, a.N - 1);
            p.scale[q] = a.scale[c];
            if (a.bias)
                p.bias[q] = a.bias[c];
        }
    }
    return p;
}
__device__ __forceinline__ void finish4(const RaggedNode& a, int m, int n, float4_t sum, const ChannelParams& p) {
    if (m >= a.M || n >= a.N)
        return;
    const float v[4] = {sum.x * (float)p.scale[0] + (float)p.bias[0], sum.y * (float)p.scale[1] + (float)p.bias[1],
                        sum.z * (float)p.scale[2] + (float)p.bias[2], sum.w * (float)p.scale[3] + (float)p.bias[3]};
    store4(a, m, n, v);
}

// The end of a 64 x 64 tile: out[r] holds channel tile r of row tile `wave` over this part of K.
__device__ __forceinline__ void finish_tile(const RaggedNode& a, float* __restrict__ ws, unsigned* __restrict__ counters, int tile,
                                            int split, int part, int m0, int n0, float4_t (&out)[4],
                                            const ChannelParams (&params)[4], unsigned* ticket) {
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (split > 1) {
        // partial tiles are parked with device-scope stores; the last part to arrive adds them in order
        constexpr int kAuxDeviceScope = 16;
        constexpr unsigned kTileFloats = RG_BM * RG_BN;
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(ws + (size_t)tile * split * kTileFloats, 0,
                                                                            split * (int)(kTileFloats * 4), 0x00020000);
        const unsigned mine = (unsigned)(wave * 64 + lane) * 16u;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, out[i]), rp,
                                                   (unsigned)part * (kTileFloats * 4) + i * 4096u + mine, 0, kAuxDeviceScope);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            *ticket = __hip_atomic_fetch_add(counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*ticket != (unsigned)(split - 1))
            return;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            out[i] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int z = 0; z < split; ++z) {
            float4_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                        rp, (unsigned)z * (kTileFloats * 4) + i * 4096u + mine, 0, kAuxDeviceScope));
#pragma unroll
            for (int i = 0; i < 4; ++i)
                out[i] += v[i];
        }
        if (threadIdx.x == 0)
            __hip_atomic_store(counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

#pragma unroll
    for (int r = 0; r < 4; ++r)
        finish4(a, m0 + 16 * wave + col, n0 + 16 * r + 4 * kq, out[r], params[r]);
}

}  // namespace

// grid = (ceil(N / 16), ceil(M / (16 MT))), block = 64 waves, dynamic LDS = waves * ragged_wave_lds(MT).
template <int BITS, int MT>
__global__ __launch_bounds__(1024) void fcc_ragged_rows_kernel(RaggedNode a, int kb_total) {
    constexpr int WD = BITS / 4;            // dwords of a lane's eight weights
    constexpr int kStep = 64 * 4 * WD;      // bytes of one step of 32 inputs
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    half_t* stage = reinterpret_cast<half_t*>(lds + wave * ragged_wave_lds(MT));  // [16 MT][RG_PITCH], this wave's own
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
    const uint8_t* w_tile = a.w + (size_t)blockIdx.x * kb_total * 4 * kStep + lane * 4 * WD;
    // activations: load i of the lane is chunk lane & 15 (eight inputs) of row 4 i + (lane >> 4)
    const half_t* x_row[4 * MT];
#pragma unroll
    for (int i = 0; i < 4 * MT; ++i)
        x_row[i] = a.x + (size_t)min(m0 + 4 * i + kq, a.M - 1) * a.K;

    struct Block {
        uint32_t w[4][WD];
        uint4_t x[4 * MT];
    };
    auto load = [&](int kb, Block& b) {
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i)
            b.x[i] = load_x(x_row[i], kb * kBlockK + 8 * col, a.K);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            load_weights<BITS>(w_tile + (size_t)(kb * 4 + j) * kStep, b.w[j]);
    };
    Block b0, b1;
    const int last = kb_total - 1;
    // (a wave has at least one k-block; what it loads past its last one is the last one again and goes unused)
    load(min(wave, last), b0);
    load(min(wave + waves, last), b1);
    const ChannelParams params = channel_params(a, n0 + 4 * kq);
    half2_t off[1], off_hi[1];
    zero_points<1>(a, {min(n0 + col, a.N - 1)}, off, off_hi);
    float4_t acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
        acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    auto consume = [&](int kb, Block& b) {
        if (kb == last) {
#pragma unroll
            for (int i = 0; i < 4 * MT; ++i)
                b.x[i] = tail_shift(b.x[i], kb * kBlockK + 8 * col, a.K);
        }
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i)
            *reinterpret_cast<uint4_t*>(&stage[(4 * i + kq) * RG_PITCH + 8 * col]) = b.x[i];
        // (LDS keeps a wave's own accesses in order)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            Frag8 wf;
            unpack_ragged<BITS>(b.w[j], off[0], off_hi[0], wf);
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    wf.v, *reinterpret_cast<const half8_t*>(&stage[(16 * t + col) * RG_PITCH + 32 * j + 8 * kq]), acc[t], 0, 0, 0);
        }
    };
    for (int kb = wave; kb < kb_total; kb += 2 * waves) {
        consume(kb, b0);
        load(min(kb + 2 * waves, last), b0);
        if (kb + waves < kb_total)
            consume(kb + waves, b1);
        load(min(kb + 3 * waves, last), b1);
    }
    // the waves' sums meet in the first kilobytes of their own stages
#pragma unroll
    for (int t = 0; t < MT; ++t)
        reinterpret_cast<float4_t*>(stage)[t * 64 + lane] = acc[t];
    __syncthreads();
    // one wave per row tile adds them in wave order
    for (int t = wave; t < MT; t += waves) {
        float4_t sum{0.f, 0.f, 0.f, 0.f};
        for (int u = 0; u < waves; ++u)
            sum += reinterpret_cast<const float4_t*>(lds + u * ragged_wave_lds(MT))[t * 64 + lane];
        finish4(a, m0 + 16 * t + col, n0 + 4 * kq, sum, params);
    }
}

// 1-D grid: 8 ceil(tiles / 8) workgroups times split parts along K.  An XCD gets a run of tiles that is contiguous
// along N (all row tiles of a channel block before the next), so the weights cross to one XCD's L2 each.
template <int BITS>
__global__ __launch_bounds__(256) void fcc_ragged_tile_kernel(RaggedNode a, int kb_total, int tiles_m, int tiles, int split,
                                                              int kb_per_split, float* __restrict__ ws,
                                                              unsigned* __restrict__ counters) {
    __shared__ __attribute__((aligned(16))) half_t stage[2][RG_STAGE_HALVES];
    __shared__ unsigned ticket_s;
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int run = (tiles + 7) >> 3;
    const int tile = (int)(blockIdx.x & 7) * run + (int)((blockIdx.x >> 3) % run), part = (int)((blockIdx.x >> 3) / run);
    if (tile >= tiles)
        return;
    const int n0 = tile / tiles_m * RG_BN, m0 = tile % tiles_m * RG_BM;
    const int kb_lo = part * kb_per_split, kb_hi = min(kb_total, kb_lo + kb_per_split);

    // weights: this wave's step of the k-block, for each of the four channel tiles (past the last one: that one again)
    constexpr int WD = BITS / 4, kStep = 64 * 4 * WD;
    const uint8_t* w_tile[4];
    int n_of[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        n_of[r] = min(n0 + 16 * r + col, a.N - 1);
        w_tile[r] = a.w + (size_t)min(n0 / 16 + r, (a.N - 1) / 16) * kb_total * 4 * kStep + wave * kStep + lane * 4 * WD;
    }
    // activations: chunk i of the thread is eight inputs of one of the 64 rows
    const int xc = threadIdx.x & 15, xr = threadIdx.x >> 4;
    const half_t* x_row[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        x_row[i] = a.x + (size_t)min(m0 + xr + 16 * i, a.M - 1) * a.K;

    uint32_t w0[4][WD], w1[4][WD];
    uint4_t x0[4], x1[4];
    auto load_w = [&](int kb, uint32_t(&w)[4][WD]) {
        kb = min(kb, kb_hi - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            load_weights<BITS>(w_tile[r] + (size_t)kb * 4 * kStep, w[r]);
    };
    auto load_rows = [&](int kb, uint4_t(&xv)[4]) {
        kb = min(kb, kb_hi - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            xv[i] = load_x(x_row[i], kb * kBlockK + 8 * xc, a.K);
    };
    auto store_rows = [&](int kb, int s, uint4_t(&xv)[4]) {
        if (kb == kb_total - 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                xv[i] = tail_shift(xv[i], kb * kBlockK + 8 * xc, a.K);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<uint4_t*>(&stage[s][(xr + 16 * i) * RG_PITCH + 8 * xc]) = xv[i];
    };
    // a barrier that waits for this wave's LDS accesses only: the loads for the next k-blocks stay in flight
    auto barrier = [&] {
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    load_rows(kb_lo, x0);
    load_w(kb_lo, w0);
    load_rows(kb_lo + 1, x1);
    load_w(kb_lo + 1, w1);
    half2_t off[4], off_hi[4];
    zero_points<4>(a, n_of, off, off_hi);
    ChannelParams params[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        params[r] = channel_params(a, n0 + 16 * r + 4 * kq);
    float4_t acc[4][4];  // [channel tile][row tile]
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc[r][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    store_rows(kb_lo, 0, x0);
    load_rows(kb_lo + 2, x0);
    barrier();

    auto compute = [&](int s, const uint32_t(&w)[4][WD]) {
        const half_t* xs = &stage[s][col * RG_PITCH + 32 * wave + 8 * kq];
        half8_t xf[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            xf[t] = *reinterpret_cast<const half8_t*>(xs + 16 * t * RG_PITCH);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            Frag8 wf;
            unpack_ragged<BITS>(w[r], off[r], off_hi[r], wf);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf.v, xf[t], acc[r][t], 0, 0, 0);
        }
    };
    // two k-blocks per trip so that stages and weight registers are static; a k-block past the end is the last one
    // again, staged where nobody reads it
    for (int kb = kb_lo; kb < kb_hi; kb += 2) {
        compute(0, w0);
        load_w(kb + 2, w0);
        store_rows(kb + 1, 1, x1);
        load_rows(kb + 3, x1);
        barrier();
        if (kb + 1 < kb_hi)
            compute(1, w1);
        load_w(kb + 3, w1);
        store_rows(kb + 2, 0, x0);
        load_rows(kb + 4, x0);
        barrier();
    }

    // The four waves' sums over their steps meet in LDS, two channel tiles at a time: wave w finishes row tile w.
    float4_t* hand = reinterpret_cast<float4_t*>(&stage[0][0]);  // [wave][3][2][64 lanes]: 24 KiB of the 34
    float4_t out[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h)
            barrier();
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t != wave)
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    hand[((wave * 3 + (t > wave ? t - 1 : t)) * 2 + r) * 64 + lane] = acc[2 * h + r][t];
        barrier();
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            float4_t v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 4; ++u)  // in wave order
                if (u == wave) {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (t == wave)
                            v += acc[2 * h + r][t];
                } else {
                    v += hand[((u * 3 + (wave > u ? wave - 1 : wave)) * 2 + r) * 64 + lane];
                }
            out[2 * h + r] = v;
        }
    }

    finish_tile(a, ws, counters, tile, split, part, m0, n0, out, params, &ticket_s);
}

// The same tiles where rows hold an even number of halves and begin at a multiple of four bytes: the activations travel to
// LDS by direct-to-LDS loads (RD_STAGES stages of 256-byte rows, the sixteen 16-byte chunks of row r at chunk ^ (r & 15)),
// the weights to registers two k-blocks ahead.  A load's pieces start at any multiple of four bytes and stay inside their
// row or, past its end, inside the activations; what they hold of the next row is set to zero when the last k-block's
// operands are read.  Rows past M and k-blocks past the end lie beyond the descriptor's range and arrive as zeros.
template <int BITS>
__global__ __launch_bounds__(256, 3) void fcc_ragged_tile_dma_kernel(RaggedNode a, int kb_total, int tiles_m, int tiles,
                                                                     int split, int kb_per_split, float* __restrict__ ws,
                                                                     unsigned* __restrict__ counters) {
    constexpr int NT = 4, A_BYTES = RG_BM * 256, STAGES = RD_STAGES;
    constexpr int AL = 4;  // direct-to-LDS loads per wave and k-block, four rows each
    constexpr int WD = BITS / 4, kStep = 64 * 4 * WD;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ unsigned ticket_s;
    const lds_byte_ptr lds3 = (lds_byte_ptr)lds;
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int run = (tiles + 7) >> 3;  // tiles of an XCD, as in the kernel above
    // (divisions and minima run on the vector ALU; told to be the same in every lane, they leave the descriptors below
    // scalar: else each buffer load sits in a loop that looks for lanes with equal ones)
    const int part = __builtin_amdgcn_readfirstlane((int)((blockIdx.x >> 3) / run));
    const int tile = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3) - part * run;
    if (tile >= tiles)
        return;
    const int column = __builtin_amdgcn_readfirstlane(tile / tiles_m);
    const int n0 = column * RG_BN, m0 = (tile - column * tiles_m) * RG_BM;
    const int kb_lo = part * kb_per_split, kb_hi = min(kb_total, kb_lo + kb_per_split);

    constexpr unsigned kOob = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;
    // (every offset goes through the vector operand: the scalar offset of a buffer load is not range-checked)
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(a.x), 0, a.M * a.K * 2, kRsrcFlags);
    const int nt0 = n0 / 16;  // channel tiles past the last one have no range
    const int nts = __builtin_amdgcn_readfirstlane(max(0, min(4, (a.N + 15) / 16 - nt0)));
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(uniform_ptr(a.w + (size_t)nt0 * kb_total * 4 * kStep)), 0, nts * kb_total * 4 * kStep, kRsrcFlags);
    unsigned a_voff[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i) {
        const int r0 = 4 * AL * wave + 4 * i;
        a_voff[i] = (unsigned)(m0 + r0 + kq) * (unsigned)a.K * 2u + ((unsigned)(col ^ kq ^ (r0 & 15)) << 4);
    }
    const unsigned w_voff = (unsigned)(wave * kStep + lane * 4 * WD);
    // The waits below count loads, so these stay in the order of the source: arithmetic and LDS accesses may move past, loads
    // from memory may not.  (Left to itself the compiler asked for the second k-block's weights ahead of the first one's,
    // and every second k-block then waited for the loads of the next.)
    auto in_order = [] { __builtin_amdgcn_sched_barrier(0x0081); };
    auto dma_x = [&](int kb, int s) {
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            unsigned at = a_voff[i] + (unsigned)(kb * 256);
            if (kb == kb_total - 1) {  // the piece that crosses the row's end holds the row's last eight inputs instead
                const int past = kb * kBlockK + 8 * (col ^ kq ^ ((4 * AL * wave + 4 * i) & 15)) - (a.K - 8);
                at -= past > 0 && past < 8 ? 2u * past : 0u;
            }
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_ptr)(lds3 + s * A_BYTES + (AL * wave + i) * 1024), 16,
                                                     kb < kb_hi ? at : kOob, 0, 0, 0);
        }
        in_order();
    };
    uint32_t w[2][4][WD];
    auto load_w = [&](int kb, uint32_t(&d)[4][WD]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const unsigned at = kb < kb_hi ? w_voff + (unsigned)((r * kb_total + kb) * 4 * kStep) : kOob;
            if constexpr (BITS == 8) {
                const uint2_t v = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rw, at, 0, 0));
                d[r][0] = v.x, d[r][1] = v.y;
            } else {
                d[r][0] = __builtin_amdgcn_raw_buffer_load_b32(rw, at, 0, 0);
            }
        }
        in_order();
    };
    // (a bare barrier that waits for this wave's LDS accesses only)
    auto barrier = [&] {
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    int n_of[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        n_of[r] = min(n0 + 16 * r + col, a.N - 1);
    half2_t off[4], off_hi[4];
    zero_points<4>(a, n_of, off, off_hi);
    in_order();
    dma_x(kb_lo, 0);
    load_w(kb_lo, w[0]);
    dma_x(kb_lo + 1, 1);
    load_w(kb_lo + 1, w[1]);
    float4_t acc[4][NT];  // [channel tile][row tile]
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            acc[r][t] = float4_t{0.f, 0.f, 0.f, 0.f};

    typedef __attribute__((address_space(3))) const half8_t* lds_frag_ptr;
    // two k-blocks per trip so that the weight registers are static; one past the end multiplies zeros
    int s = 0;  // the k-block's stage
    for (int kb0 = kb_lo; kb0 < kb_hi; kb0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int kb = kb0 + u;
            // this k-block's activations have landed once no more is out than what was asked for after them: its
            // weights, activations and weights of the next one
            __builtin_amdgcn_s_waitcnt(wait_vmcnt_imm(AL + 8));
            barrier();  // everyone's have; everyone is done with the stage of k-block kb - 1
            dma_x(kb + STAGES - 1, s == 0 ? STAGES - 1 : s - 1);
            const lds_byte_ptr xs = lds3 + s * A_BYTES + col * 256 + (((4 * wave + kq) ^ col) << 4);
            Frag8 xf[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                xf[t].v = *(lds_frag_ptr)(xs + t * 4096);
            if (kb >= kb_total - 1) {
                // the row's last k-block: a piece past its end is the next row's, the one across it is moved into place
                const int past = kb * kBlockK + 32 * wave + 8 * kq - (a.K - 8);
                int d = past <= 0 ? 0 : min(past, 8) >> 1;  // dwords to move by; 4: nothing is left
                asm volatile("" : "+v"(d));                 // (a branch around the moves, not selects in every k-block)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        uint32_t v = d == 0 ? xf[t].u[j] : 0u;
#pragma unroll
                        for (int i = 1; i < 4; ++i)
                            if (j + i < 4)
                                v = d == i ? xf[t].u[j + i] : v;
                        xf[t].u[j] = v;
                    }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                Frag8 wf;
                unpack_ragged<BITS>(w[u][r], off[r], off_hi[r], wf);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf.v, xf[t].v, acc[r][t], 0, 0, 0);
            }
            load_w(kb + 2, w[u]);
            s = s == STAGES - 1 ? 0 : s + 1;
        }
    }
    ChannelParams params[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        params[r] = channel_params(a, n0 + 16 * r + 4 * kq);
    __builtin_amdgcn_s_waitcnt(wait_vmcnt_imm(0));  // the loads past the end still target LDS
    barrier();

    // The four waves' sums over their steps meet in LDS, two channel tiles at a time: wave w finishes row tile w.
    float4_t* hand = reinterpret_cast<float4_t*>(lds);  // [wave][3][2][64 lanes]: 24 KiB
    float4_t out[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h)
            barrier();
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t != wave)
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    hand[((wave * 3 + (t > wave ? t - 1 : t)) * 2 + r) * 64 + lane] = acc[2 * h + r][t];
        barrier();
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            float4_t v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 4; ++u)  // in wave order
                if (u == wave) {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (t == wave)
                            v += acc[2 * h + r][t];
                } else {
                    v += hand[((u * 3 + (wave > u ? wave - 1 : wave)) * 2 + r) * 64 + lane];
                }
            out[2 * h + r] = v;
        }
    }
    finish_tile(a, ws, counters, tile, split, part, m0, n0, out, params, &ticket_s);
}

// One thread per eight weights of the arranged node.
__global__ __launch_bounds__(256) void fcc_ragged_repack_kernel(const uint8_t* __restrict__ w, uint8_t* __restrict__ out, int N,
                                                                int K, int64_t units, int steps, int bits, uint32_t flip) {
    const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (u >= units)
        return;
    const int lane = (int)(u & 63);
    const int64_t s = u >> 6, nt = s / steps;
    const int n = (int)(nt * kTileRows) + (lane & 15), k = (int)(s % steps) * 32 + 8 * (lane >> 4);
    const int valid = n < N ? min(8, K - k) : 0;
    const int64_t at = (int64_t)n * K + k;
    if (bits == 8) {
        uint64_t v = 0;
        for (int e = 0; e < valid; ++e)
            v |= (uint64_t)(w[at + e] ^ flip) << (8 * e);
        reinterpret_cast<uint64_t*>(out)[u] = v;
    } else {
        uint32_t v = 0;
        for (int e = 0; e < valid; ++e) {
            const uint32_t q = ((w[(at + e) >> 1] >> (4 * ((at + e) & 1))) & 15u) ^ flip;
            v |= q << (4 * ((e >> 1) + 4 * (e & 1)));  // the tile layout's nibble order
        }
        reinterpret_cast<uint32_t*>(out)[u] = v;
    }
}

int launch_ragged_repack(const ovfcc_fc_desc& d, const Layout& L, const void* w, void* w_out, void* stream) {
    const int64_t units = (int64_t)(L.w_bytes / L.bits), groups = (units + 255) / 256;
    if (!L.ragged || groups > 0x7FFFFFFF || L.k_blocks * 4 > 0x7FFFFFFF)
        return (int)hipErrorInvalidValue;
    const uint32_t flip = d.w_type == OVFCC_I8 ? 0x80u : d.w_type == OVFCC_I4 ? 8u : 0u;
    hipLaunchKernelGGL(fcc_ragged_repack_kernel, dim3((unsigned)groups), dim3(256), 0, static_cast<hipStream_t>(stream),
                       (const uint8_t*)w, (uint8_t*)w_out, (int)d.N, (int)d.K, units, (int)(L.k_blocks * 4), L.bits, flip);
    return (int)hipGetLastError();
}

// More than 64 KiB of LDS has to be asked for, once per kernel (the attribute is idempotent: a race only repeats it).
static int ask_for_lds(const void* kern, std::atomic<bool>& done, int bytes) {
    if (done.load(std::memory_order_relaxed))
        return 0;
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess)
        done.store(true, std::memory_order_relaxed);
    return (int)e;
}

int launch_ragged(const FcDeviceArgs& a, const LaunchPlan& p, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool four = a.layout.bits == 4;
    if (!a.layout.ragged || (p.split_k > 1 && !(a.workspace && a.counters)))
        return (int)hipErrorInvalidValue;
    RaggedNode r;
    r.w = (const uint8_t*)a.w, r.scale = (const half_t*)a.scale, r.zp = (const uint8_t*)a.zp, r.bias = (const half_t*)a.bias;
    r.x = (const half_t*)a.x, r.y = a.y;
    r.M = (int)a.M, r.N = (int)a.N, r.K = (int)a.K;
    r.zp_kind = a.zp_type == OVFCC_NONE ? 0 : a.zp_type == OVFCC_U4 ? 1 : 2;
    r.zp_scalar = a.zp_scalar, r.zp_const = a.layout.zp_offset;
    r.out_f32 = a.out_f32;
    const int kb = (int)a.layout.k_blocks;
    const dim3 grid(p.grid[0], p.grid[1], 1), block(p.block);
    if (p.tile_n == 16) {
        if ((int64_t)p.grid[0] * 16 < a.N || (int64_t)p.grid[1] * p.tile_m < a.M || (int)(p.block / 64) > kb)
            return (int)hipErrorInvalidValue;
        auto kern = p.tile_m == 16 ? (four ? fcc_ragged_rows_kernel<4, 1> : fcc_ragged_rows_kernel<8, 1>)
                                   : (four ? fcc_ragged_rows_kernel<4, 2> : fcc_ragged_rows_kernel<8, 2>);
        static std::atomic<bool> asked[2][2] = {};
        if (int e = ask_for_lds(reinterpret_cast<const void*>(kern), asked[four ? 0 : 1][p.tile_m == 16 ? 0 : 1],
                                16 * ragged_wave_lds(p.tile_m / 16)))
            return e;
        hipLaunchKernelGGL(kern, grid, block, p.dynamic_lds, s, r, kb);
    } else {
        const int64_t tiles = (int64_t)p.tiles_x * p.tiles_y;
        if ((int64_t)p.tiles_x * RG_BN < a.N || (int64_t)p.tiles_y * RG_BM < a.M ||
            (int64_t)p.split_k * p.kblocks_per_split < kb || p.grid[0] != (unsigned)((tiles + 7) / 8 * 8 * p.split_k))
            return (int)hipErrorInvalidValue;
        if (p.to_lds && !ragged_rows_at_dwords(a))
            return (int)hipErrorInvalidValue;
        auto kern = p.to_lds ? (four ? fcc_ragged_tile_dma_kernel<4> : fcc_ragged_tile_dma_kernel<8>)
                             : (four ? fcc_ragged_tile_kernel<4> : fcc_ragged_tile_kernel<8>);
        hipLaunchKernelGGL(kern, grid, block, p.to_lds ? RD_STAGES * RG_BM * kBlockK * 2 : 0, s, r, kb, p.tiles_y, (int)tiles, p.split_k,
                           p.kblocks_per_split, a.workspace, a.counters);
    }
    return (int)hipGetLastError();
}

}  // namespace ovfcc
