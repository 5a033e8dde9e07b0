// Prefill kernels for 4-bit weights that run two workgroups on a compute unit: tiles of 64 to 128 rows x 256 channels,
// four waves of 256 registers each.  They run the slices of a mixture-of-experts layer and single nodes (pair_preferred in
// plan.cpp draws the line against the 8-wave and the 256 x 256 kernel).
//
// Against the 8-wave kernel (kernel_prefill_async.hip), which has a compute unit to itself: the two workgroups share no
// barrier, so one contracts while the other starts, waits or stores, and on every SIMD the vector ALU unpacks for one
// wave while the matrix cores run the other; a wave contracts all of K for its 64 channels, so nothing is handed over at the
// end; weights go from memory to the registers of the one wave that uses them and not through LDS.  Bound: the vector ALU's
// unpacking beside the matrix cores -- 258 vector instructions (4 cycles each) to 80 MFMAs (16 cycles) per wave and k-block at
// 80 rows; without the subtraction and the scaling the 256 rows below take 43 us less, without the barriers 3, without the
// activation loads 16.  Expert block of eight experts, 4096 / 14336, top two, u4 in groups of 128 with zero-points, against
// the 8-wave kernel's slices: 256 rows 282 -> 244 us, 330 rows 350 -> 275, 400 rows 363 -> 325, 1000 rows 808 -> 643; with K cut
// for two workgroups on a compute unit 295 -> 247 at 256 rows, another card.  Single nodes: pair_preferred's comment; 4096 -> 28672
// with a gated linear unit at 2048 rows 358 us, 1.34 PFLOP/s, against 430 in 256 x 256 tiles.
//
// Tiles of 128 channels (R = 2 channel tiles a wave; single nodes): a wave alone on its SIMD pays 5 cycles for every vector
// instruction beyond two per MFMA, and at R = 4 and 64 rows it has four.  The same MFMAs as 128 rows x 128 channels have half
// of the unpacking: a k-block takes 1.02 us against 1.03, of 64 rows 0.62 (4096 -> 6144 at 117 rows 20.7 -> 16.9 us, 14336 -> 4096
// 29.7 -> 25.8).  Against that, an operand read from LDS meets two MFMAs and not four, which is more than half of what LDS gives;
// long launches keep 256 channels (plan_pair).
//
// 1-D grid, block = 256: workgroup -> (tile, part of K) by tile_work (device_common.h).  A tile has the height that its rows
// need (64, 80, 96 or 128: a branch per workgroup), whatever the launch's tile height is.
//
// Per k-block of 128 inputs:
//   - weights: a wave's four channel tiles, one 128-bit load per lane each, three k-blocks ahead (two at 128 rows, where a
//     k-block takes longer and registers end); scale and zero-point of the lane (kq, col) belong to channel tile kq, one
//     load each, and are exchanged between the lanes (permlane swaps);
//   - activations: direct-to-LDS loads, two k-blocks (three halves) ahead, as half k-blocks of 128-byte rows whose eight
//     16-byte chunks sit at chunk ^ ((row >> 1) & 7), which spreads an operand read over all banks.
// One barrier per stage.  Its wait counts loads, so their order is pinned (sched_barrier after every MFMA) and read back
// from the assembly by a test.  A row past M, a k-block past the part's end: the load has no range and brings zeros.
// The loop is pipelined by hand: after every MFMA a few of the operations that unpack the next step's weights.
//
// MFMA roles: A = weights, B = activations; a lane holds column m = lane & 15, channels 4 (lane >> 4) + q.  Weights:
// (q - zp) * s rounded once to f16; with one group per channel exact integers, the scale multiplies the f32 sum.  A row's
// sum runs over K in ascending order whatever the height, so results do not depend on the tile that a row sits in.
#include <type_traits>

#include "device_common.h"

namespace ovfcc {

constexpr int pp_bn(int r) { return 64 * r; }  // channels of a tile: four waves of r channel tiles each
constexpr int PP_BN = pp_bn(4);
constexpr int pp_half_bytes(int nt) { return nt * 16 * 128; }  // 64 inputs of a tile's rows
// The order of a k-block's steps (each of its halves on its own): any is as good as another, results that sit on a tie of f16
// move with it.
constexpr int pp_dword(int step) { return step ^ 1; }
// stages of activations: three k-blocks, with 128-row tiles four halves of one
constexpr bool pp_by_halves(int nt) { return nt == 8; }
constexpr unsigned pp_lds_bytes(int nt) { return (unsigned)((pp_by_halves(nt) ? 4 : 6) * pp_half_bytes(nt)); }
// waves per SIMD; the one form whose registers do not fit twice (in slices of up to 80 rows they do) runs alone
constexpr int pp_waves(int nt, int gpb, bool zp_table) { return nt == 8 && gpb == 4 && zp_table ? 1 : 2; }
constexpr unsigned PP_LDS = pp_lds_bytes(6);  // the largest of the four heights: 72 KiB, twice on a compute unit

template <bool ZP_TABLE, bool PRESCALE, int NT, int GPB, int R>
__device__ __forceinline__ void prefill_pair_body(const uint4_t* __restrict__ wt, const half_t* __restrict__ st,
                                                   const uint8_t* __restrict__ zt, const half_t* __restrict__ x,
                                                   const half_t* __restrict__ bias, void* __restrict__ y,
                                                   float* __restrict__ ws, unsigned* __restrict__ counters, int M, int N,
                                                   int K, int kb_total, int kb_per_group, int ng, int zp_const,
                                                   int out_f32, int glu, const TileWork wk,
                                                   const int* __restrict__ row_map, int x_rows, int park_rows) {
    constexpr bool HALVES = pp_by_halves(NT);
    constexpr bool BURST = R == 4 && NT >= 6;  // no registers for a second set of parameters
    static_assert(GPB == 1 || ((GPB == 2 || GPB == 4) && PRESCALE), "several groups per k-block: scales go into the weights");
    constexpr int HB = pp_half_bytes(NT);
    constexpr int S = R * NT;                           // MFMAs of a step (32 inputs)
    constexpr int BN = pp_bn(R);
    constexpr int NOPS = 5 + 4 + (PRESCALE ? 4 : 0);    // unpack operations per weight dword
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const lds_byte_ptr lds3 = (lds_byte_ptr)lds_raw;
    typedef __attribute__((address_space(3))) const half8_t* lds_frag_ptr;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, kq = lane >> 4;
    const int n0 = wk.tile_x * BN, m0 = wk.m0, split_k = wk.split_k;
    const int kb_lo = wk.kb_lo, kb_hi = wk.kb_hi;
    constexpr unsigned kOob = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;

    const int nt0 = n0 / 16 + R * wave;
    const int nts = n0 + 16 * R * wave < N ? R : 0;  // the wave's channel tiles: none where the node ends on half a tile
    auto live = [&](int kb, int bytes) { return kb < kb_hi ? bytes : 0; };
#define PP_DESC_X(kb) \
    __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(x), 0, live(kb, (row_map ? x_rows : M) * K * 2), kRsrcFlags)
#define PP_DESC_W(kb) \
    __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4_t*>(wt + (size_t)nt0 * kb_total * 64), 0, live(kb, nts * kb_total * kTileBytes), kRsrcFlags)
#define PP_DESC_S(kb) \
    __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(st + (size_t)nt0 * ng * 16), 0, live(kb, nts * ng * 32), kRsrcFlags)
#define PP_DESC_Z(kb)                                                                                       \
    __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(ZP_TABLE ? zt + (size_t)nt0 * ng * 16 : zt), 0, \
                                      ZP_TABLE ? live(kb, nts * ng * 16) : 0, kRsrcFlags)
    // group of a k-block: kb / kb_per_group without a branch
    const int g_one = kb_per_group == 1 ? 1 : 0;
    const unsigned g_mul = kb_per_group == 1 ? 0u : (unsigned)((0x100000000ull + kb_per_group - 1) / kb_per_group);

    // ---- activations: 4 NT loads per k-block, NT per wave; load i = wave NT + q: half i / (2 NT) of the k-block, rows
    // 8 (i % (2 NT)) ..+7; lane -> row lane >> 3 of those, slot lane & 7, which holds chunk slot ^ ((row >> 1) & 7) ----
    // (with stages of half a k-block: load q of a wave covers rows 8 (4 wave + q) of the half)
    constexpr int AV = HALVES ? NT / 2 : NT;
    unsigned a_voff[8];  // AV entries in use (a bound that depends on NT does not pass the host pass)
#pragma unroll
    for (int q = 0; q < AV; ++q) {
        const int i = wave * AV + q, half = !HALVES && i >= 2 * NT ? 1 : 0, r0 = 8 * (i - half * 2 * NT);
        const int rl = r0 + (lane >> 3);
        int row = m0 + rl;
        unsigned dead = 0;
        if (row_map) {
            const int src = row < M ? row_map[row] : -1;
            dead = src < 0 ? kOob : 0u;
            row = src < 0 ? 0 : src;
        }
        a_voff[q] = ((unsigned)(row * K) * 2u + half * 128u + (unsigned)(((lane & 7) ^ ((rl >> 1) & 7)) << 4)) | dead;
    }
    auto dma_a = [&](int kb, int stage, int q) {
        const __amdgpu_buffer_rsrc_t d_ = PP_DESC_X(kb);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(d_, (lds_void_ptr)(lds3 + stage * 2 * HB + (wave * NT + q) * 1024), 16,
                                                 a_voff[q], kb * (kBlockK * 2), 0, 0);
    };

    auto dma_h = [&](int hh, int stage, int q) {  // half k-block hh (of all K) into half-stage `stage`
        const __amdgpu_buffer_rsrc_t d_ = PP_DESC_X(hh >> 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(d_, (lds_void_ptr)(lds3 + stage * HB + (wave * AV + q) * 1024), 16, a_voff[q],
                                                 hh * 128, 0, 0);
    };
    // ---- weights of one k-block ----
    struct WSlot {
        uint4_t w[R];
        uint32_t s[GPB == 4 ? 2 : 1];  // scales (and, with one group per k-block, zero-points) of tile kq, channel col
        uint32_t z;
    };
    auto load_w = [&](int kb, WSlot& s, int r) {
        const __amdgpu_buffer_rsrc_t d_ = PP_DESC_W(kb);
        s.w[r] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(d_, lane * 16u, (r * kb_total + kb) * kTileBytes, 0));
    };
    // (all as whole dwords: two channels' scales, four, two or one channels' zero-points; prepare picks the lane's)
    constexpr int ZB = GPB;  // bytes of a channel's zero-points in a k-block
    const unsigned p_voff = (unsigned)((kq & (R - 1)) * (GPB == 1 ? ng : kb_total) * 16 + col) * GPB;
    const unsigned s_shift = GPB == 1 ? 16u * (col & 1) : 0u, z_shift = 8u * ((col * ZB) & 3);
    auto load_p = [&](int kb, WSlot& s, int which) {
        const int g = GPB == 1 ? kb * g_one + (int)__umulhi((unsigned)kb, g_mul) : kb;
        if (which == 0) {
            if constexpr (PRESCALE) {
                const __amdgpu_buffer_rsrc_t d_ = PP_DESC_S(kb);
                if constexpr (GPB == 4) {
                    const uint2_t v = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(d_, p_voff * 2u, g * 128, 0));
                    s.s[0] = v.x, s.s[GPB == 4 ? 1 : 0] = v.y;
                } else {
                    s.s[0] = __builtin_amdgcn_raw_buffer_load_b32(d_, (p_voff * 2u) & ~3u, g * (32 * GPB), 0);
                }
            }
        } else if constexpr (ZP_TABLE) {
            const __amdgpu_buffer_rsrc_t d_ = PP_DESC_Z(kb);
            s.z = __builtin_amdgcn_raw_buffer_load_b32(d_, p_voff & ~3u, g * (16 * GPB), 0);
        }
    };
    constexpr int LW = R + (PRESCALE ? 1 : 0) + (ZP_TABLE ? 1 : 0);

    // ---- parameters of the slot being unpacked, one register per channel tile ----
    uint32_t ps[GPB == 4 ? 2 : 1][4], pz[4];
    half2_t off_lo[4], off_hi[4];
    auto spread = [&](uint32_t v, uint32_t (&o)[4]) {
        const uint2_t h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        const uint2_t a = __builtin_amdgcn_permlane16_swap(h.x, h.x, false, false);
        const uint2_t b = __builtin_amdgcn_permlane16_swap(h.y, h.y, false, false);
        o[0] = a.x, o[1] = a.y, o[2] = b.x, o[3] = b.y;
    };
    const half2_t off_lo_c = as_half2(__builtin_amdgcn_readfirstlane(as_u32(splat(1024.f + (float)zp_const))));
    const half2_t off_hi_c = as_half2(__builtin_amdgcn_readfirstlane(as_u32(splat(64.f + (float)zp_const))));
    // offsets of the subtractions for channel tile r, group g of the k-block
    auto offsets = [&](const uint32_t (&z)[4], int r, int g, half2_t (&lo)[4], half2_t (&hi)[4]) {
        if constexpr (ZP_TABLE) {
            const uint32_t zpv = GPB == 1 ? (PRESCALE ? z[r] >> 16 : z[r]) : (z[r] >> (8 * g)) & 0xFFu;
            lo[r] = as_half2(zpv * 0x00010001u + 0x64006400u);
            hi[r] = lo[r] - half2_t{(half_t)960.f, (half_t)960.f};
        }
    };
    // The next slot's parameters, in seven pieces that sit between MFMAs: the lanes' own values, their exchange, the offsets.
    uint32_t raw_s[GPB == 4 ? 2 : 1], raw_z, ps_n[GPB == 4 ? 2 : 1][4], pz_n[4];
    half2_t lo_n[4], hi_n[4];
    auto prepare = [&](const WSlot& s, int piece) {
        if (piece == 0) {
            if constexpr (PRESCALE)
                raw_s[0] = GPB == 1 ? (s.s[0] >> s_shift) & 0xFFFFu : s.s[0];
            if constexpr (GPB == 4)
                raw_s[GPB == 4 ? 1 : 0] = s.s[GPB == 4 ? 1 : 0];
            if constexpr (ZP_TABLE)
                raw_z = GPB == 1 ? (s.z >> z_shift) & 0xFFu : s.z >> z_shift;
            if constexpr (GPB == 1 && PRESCALE && ZP_TABLE)
                raw_s[0] |= raw_z << 16;
        } else if (piece == 1) {
            if constexpr (PRESCALE)
                spread(raw_s[0], ps_n[0]);
            if constexpr (GPB == 1 && PRESCALE && ZP_TABLE) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    pz_n[r] = ps_n[0][r];
            }
        } else if (piece == 2) {
            if constexpr (GPB == 4)
                spread(raw_s[GPB == 4 ? 1 : 0], ps_n[GPB == 4 ? 1 : 0]);
            if constexpr (ZP_TABLE && (GPB != 1 || !PRESCALE))
                spread(raw_z, pz_n);
        } else {
            offsets(pz_n, piece - 3, GPB == 4 ? pp_dword(0) : 0, lo_n, hi_n);
        }
    };
    auto commit = [&]() {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (PRESCALE)
                ps[0][r] = ps_n[0][r];
            if constexpr (GPB == 4)
                ps[GPB == 4 ? 1 : 0][r] = ps_n[GPB == 4 ? 1 : 0][r];
            if constexpr (ZP_TABLE)
                pz[r] = pz_n[r], off_lo[r] = lo_n[r], off_hi[r] = hi_n[r];
        }
    };
    const Unpack4Consts uc = unpack4_consts();
    auto unpack_op = [&](const WSlot& s, int r, int j, int op, Frag8& f) {
        const uint32_t w = j == 0 ? s.w[r].x : j == 1 ? s.w[r].y : j == 2 ? s.w[r].z : s.w[r].w;
        if (op == 0)
            f.u[3] = w >> 8;
        else if (op == 1)
            f.u[0] = (w & uc.mask_lo) | uc.magic_lo;
        else if (op == 2)
            f.u[1] = (w & uc.mask_hi) | uc.magic_hi;
        else if (op == 3)
            f.u[2] = (f.u[3] & uc.mask_lo) | uc.magic_lo;
        else if (op == 4)
            f.u[3] = (f.u[3] & uc.mask_hi) | uc.magic_hi;
        else if (op < 9) {
            const int k = op - 5;
            f.h2[k] = f.h2[k] - (ZP_TABLE ? ((k & 1) ? off_hi[r] : off_lo[r]) : ((k & 1) ? off_hi_c : off_lo_c));
        } else if constexpr (PRESCALE) {
            const half2_t sv = as_half2(ps[GPB == 4 ? j >> 1 : 0][r]);
            const half_t h = GPB == 1 ? sv[0] : GPB == 2 ? sv[j >> 1] : sv[j & 1];
            f.h2[op - 9] *= half2_t{h, h};
        }
    };

    float4_t acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            acc[r][t] = float4_t{0.f, 0.f, 0.f, 0.f};

    constexpr int XQ = NT < 6 ? 4 : NT == 6 && ZP_TABLE && !PRESCALE ? 2 : 3;  // (as many as fit)
    constexpr int NS = HALVES ? 2 : 3;  // k-blocks of weights in registers
    const int x_sw = (col >> 1) & 7;
    const lds_byte_ptr xa0 = lds3 + col * 128 + ((kq ^ x_sw) << 4);
    const lds_byte_ptr xa1 = lds3 + col * 128 + (((4 + kq) ^ x_sw) << 4);
    auto top = [&](auto behind) {
        // the activations of this stage have landed, `behind` loads that this wave issued after them may be under way
        __builtin_amdgcn_s_waitcnt(wait_vmcnt_imm(decltype(behind)::value));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // One k-block (stage: its number among the stages): step js multiplies wf[js & 1] with the row tiles while dword
    // js + 1 of slot sa (dword 0 of sb in the last step) is unpacked into the other set
    auto block = [&](int kb_, int stage, Frag8 (&wf)[2][R], WSlot& sa, WSlot& sb) {
        const int kb = __builtin_amdgcn_readfirstlane(kb_);
        auto x_at = [&](int n) {  // operand n: step n / NT, row tile n % NT
            const int js = n / NT, t = n % NT;
            return *(lds_frag_ptr)(((pp_dword(js) & 1) ? xa1 : xa0) + stage * 2 * HB + (js >> 1) * HB + t * 2048);
        };
        half8_t xq[XQ];
        auto slot = [&](int js, int i) {
            const int t = i / R, r = i % R, n = js * NT + t;
            constexpr int last = 4 * NT;
            const int limit = HALVES && js < 2 ? 2 * NT : last;
            if (r == 0 && n + XQ - 1 < limit)
                xq[(n + XQ - 1) % XQ] = x_at(n + XQ - 1);
            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[js & 1][r].v, xq[n % XQ], acc[r][t], 0, 0, 0);
            if (!BURST && js == 2 && i >= S - 7)
                prepare(sb, i - (S - 7));
            if (js == 3 && i == 0) {
                if constexpr (BURST) {
#pragma unroll
                    for (int piece = 0; piece < 7; ++piece)
                        prepare(sb, piece);
                }
                commit();
            }
            if ((GPB == 4 && js < 3 && i == 0) || (GPB == 2 && js == 1 && i == 0)) {
#pragma unroll
                for (int rr = 0; rr < R; ++rr)
                    offsets(pz, rr, GPB == 4 ? pp_dword(js + 1) : 1, off_lo, off_hi);
            }
#pragma unroll
            for (int g = i * R * NOPS / S; g < (i + 1) * R * NOPS / S; ++g) {
                if (js < 3)
                    unpack_op(sa, g / NOPS, pp_dword(js + 1), g % NOPS, wf[(js & 1) ^ 1][g / NOPS]);
                else
                    unpack_op(sb, g / NOPS, pp_dword(0), g % NOPS, wf[0][g / NOPS]);
            }
            // activations two k-blocks ahead (three halves), into the stage that the barrier freed
            if constexpr (HALVES) {
                if (!(js & 1) && i % (2 * R) == 2)
                    dma_h(2 * kb + (js >> 1) + 3, (2 * stage + (js >> 1) + 3) & 3, i / (2 * R));
            } else if (js < 3 && i % (2 * R) == 2) {
                const int q = js * ((NT + 2) / 3) + i / (2 * R);
                if (i / (2 * R) < (NT + 2) / 3 && q < NT)
                    dma_a(kb + 2, (stage + 2) % 3, q);
            }
            // weights and parameters NS k-blocks ahead, into this k-block's own registers, unpacked by then
            if (js == 3) {
                if ((i & 3) == 1 && (i >> 2) < R)
                    load_w(kb + NS, sa, i >> 2);
                if (i == 3)
                    load_p(kb + NS, sa, 0);
                if (i == 7)
                    load_p(kb + NS, sa, 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto fill = [&](int n0) {
#pragma unroll
            for (int n = 0; n < XQ - 1; ++n)
                xq[(n0 + n) % XQ] = x_at(n0 + n);
        };
        // behind a stage's own loads this wave asked for: two k-blocks of weights and parameters and one of activations;
        // with half stages for two halves of activations and one or two k-blocks of weights
        top(std::integral_constant<int, 2 * LW + (HALVES ? 2 * AV : NT)>{});
        fill(0);
#pragma unroll
        for (int i = 0; i < S; ++i)
            slot(0, i);
#pragma unroll
        for (int i = 0; i < S; ++i)
            slot(1, i);
        if constexpr (HALVES) {
            top(std::integral_constant<int, 2 * AV + LW>{});
            fill(2 * NT);
        }
#pragma unroll
        for (int i = 0; i < S; ++i)
            slot(2, i);
#pragma unroll
        for (int i = 0; i < S; ++i)
            slot(3, i);
    };

    WSlot ws0, ws1, ws2;
    auto load_all = [&](int kb, WSlot& s) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            load_w(kb, s, r);
        load_p(kb, s, 0);
        load_p(kb, s, 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto dma_all = [&](int kb, int stage) {
#pragma unroll
        for (int q = 0; q < NT; ++q)
            dma_a(kb, stage, q);
        __builtin_amdgcn_sched_barrier(0);
    };
    // (in the order of the loop, whose waits count on it)
    if constexpr (HALVES) {
        auto half_all = [&](int hh) {
#pragma unroll
            for (int q = 0; q < AV; ++q)
                dma_h(2 * kb_lo + hh, hh, q);
            __builtin_amdgcn_sched_barrier(0);
        };
        half_all(0);
        load_all(kb_lo, ws0);
        half_all(1);
        half_all(2);
        load_all(kb_lo + 1, ws1);
    } else {
        load_all(kb_lo, ws0);
        dma_all(kb_lo, 0);
        load_all(kb_lo + 1, ws1);
        dma_all(kb_lo + 1, 1);
        load_all(kb_lo + 2, ws2);
    }
    Frag8 wf[2][R];
#pragma unroll
    for (int i = 0; i < 7; ++i)
        prepare(ws0, i);
    commit();
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int op = 0; op < NOPS; ++op)
            unpack_op(ws0, r, pp_dword(0), op, wf[0][r]);
    __builtin_amdgcn_sched_barrier(0);

    // As many k-blocks per trip as there are slots, so that slots and stages are static; the rest behind the loop, at 128 rows
    // a k-block of zeros if their number is odd.  (With tests between the blocks the compiler moved loads behind them and
    // slots between registers, and waited for both; a second copy of the 128-row block spills.)
    int kb = kb_lo;
    if constexpr (HALVES) {
        for (; kb < kb_hi; kb += 2) {
            block(kb, 0, wf, ws0, ws1);
            block(kb + 1, 1, wf, ws1, ws0);
        }
    } else {
        for (; kb + 3 <= kb_hi; kb += 3) {
            block(kb, 0, wf, ws0, ws1);
            block(kb + 1, 1, wf, ws1, ws2);
            block(kb + 2, 2, wf, ws2, ws0);
        }
        if (kb < kb_hi)
            block(kb, 0, wf, ws0, ws1);
        if (kb + 1 < kb_hi)
            block(kb + 1, 1, wf, ws1, ws2);
    }
    __builtin_amdgcn_s_waitcnt(wait_vmcnt_imm(0));  // the out-of-range loads of the last trips still target LDS
    // Every way out uses every slot: otherwise the compiler may move a k-block's weight loads behind a test, into the block
    // that unpacks them, and the counted waits above would count loads that were not issued.
    auto hold = [&](const WSlot& s) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            asm volatile("" ::"v"(s.w[r]));
        if constexpr (PRESCALE)
            asm volatile("" ::"v"(s.s[0]));
        if constexpr (GPB == 4)
            asm volatile("" ::"v"(s.s[GPB == 4 ? 1 : 0]));
        if constexpr (ZP_TABLE)
            asm volatile("" ::"v"(s.z));
    };
    hold(ws0), hold(ws1);
    if constexpr (!HALVES)
        hold(ws2);
#pragma unroll
    for (int r = 0; r < R; ++r)
        asm volatile("" ::"v"(wf[0][r].v));  // (the same for the first step's operands, unpacked a k-block ahead)

    // (the lane's coordinates once more, so that nothing derived from them lives through the loop)
    unsigned lane_e = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane_e));
    const int col_e = lane_e & 15, kq_e = lane_e >> 4;

    // ---- split-K: park, draw a ticket, the last arrival adds the parts in order ----
    if (split_k > 1) {
        constexpr int kAuxDeviceScope = 16;
        constexpr unsigned kParkBytes = 4 * (R * NT) * 64 * 16;
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<char*>(ws) + (size_t)wk.park_slot * split_k * park_rows * (BN * 4), 0, split_k * (int)kParkBytes, kRsrcFlags);
        const unsigned at = (unsigned)(wave * R * NT * 64 + lane_e) * 16u;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, acc[r][t]), rp,
                                                       wk.z * kParkBytes + at + (unsigned)(r * NT + t) * 1024u, 0, kAuxDeviceScope);
        __shared__ unsigned ticket_s;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (wave == 0 && lane_e == 0)
            ticket_s = __hip_atomic_fetch_add(counters + wk.park_slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (ticket_s != (unsigned)(split_k - 1))
            return;
        if (nts == 0)
            return;  // (wave 0, which resets the counter, is never beyond the node's end)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[r][t] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int z = 0; z < split_k; ++z) {
#pragma unroll
            for (int r0 = 0; r0 < R; r0 += 2) {  // (half of a part's loads in flight at a time: all of them do not fit)
                float4_t part[2][NT];
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        part[r][t] = __builtin_bit_cast(
                            float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                          rp, (unsigned)z * kParkBytes + at + (unsigned)((r0 + r) * NT + t) * 1024u, 0, kAuxDeviceScope));
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        float4_t& sum = acc[r0 + r][t];
                        sum.x += part[r][t].x, sum.y += part[r][t].y, sum.z += part[r][t].z, sum.w += part[r][t].w;
                    }
            }
        }
        if (wave == 0 && lane_e == 0)
            __hip_atomic_store(counters + wk.park_slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---- scale, bias, gated linear unit, stores ----
    if (nts == 0)
        return;
    const int nw = n0 + 16 * R * wave;
    auto channel_params = [&](int r, float (&sc)[4], float (&bs)[4]) {
        const int n = nw + 16 * r + 4 * kq_e;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            sc[q] = 1.f, bs[q] = 0.f;
        if constexpr (!PRESCALE) {
            const half4_t s4 = *reinterpret_cast<const half4_t*>(st + n);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                sc[q] = (float)s4[q];
        }
        if (bias) {
            const half4_t b4 = *reinterpret_cast<const half4_t*>(bias + n);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                bs[q] = (float)b4[q];
        }
    };
    auto put = [&](size_t idx, const float (&o)[4]) {
        if (out_f32)
            *reinterpret_cast<float4_t*>(static_cast<float*>(y) + idx) = float4_t{o[0], o[1], o[2], o[3]};
        else
            *reinterpret_cast<half4_t*>(static_cast<half_t*>(y) + idx) =
                half4_t{to_half_rne(o[0]), to_half_rne(o[1]), to_half_rne(o[2]), to_half_rne(o[3])};
    };
    float sc[R][4], bs[R][4];
#pragma unroll
    for (int r = 0; r < R; ++r)
        channel_params(r, sc[r], bs[r]);
    if (glu) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int m = m0 + 16 * t + col_e;
#pragma unroll
            for (int j = 0; j < R / 2; ++j) {
                const float4_t g = acc[2 * j][t], u = acc[2 * j + 1][t];
                const float o[4] = {
                    glu_value(glu, g.x * sc[2 * j][0] + bs[2 * j][0], u.x * sc[2 * j + 1][0] + bs[2 * j + 1][0]),
                    glu_value(glu, g.y * sc[2 * j][1] + bs[2 * j][1], u.y * sc[2 * j + 1][1] + bs[2 * j + 1][1]),
                    glu_value(glu, g.z * sc[2 * j][2] + bs[2 * j][2], u.z * sc[2 * j + 1][2] + bs[2 * j + 1][2]),
                    glu_value(glu, g.w * sc[2 * j][3] + bs[2 * j][3], u.w * sc[2 * j + 1][3] + bs[2 * j + 1][3])};
                if (m < M)
                    put((size_t)m * (N / 2) + nw / 2 + 16 * j + 4 * kq_e, o);
            }
        }
        return;
    }
    if constexpr (R == 4) {
    if (!out_f32 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
        half_t* yh = static_cast<half_t*>(y);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            uint32_t p[4][2];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float4_t v = acc[r][t];
                const half4_t h = half4_t{to_half_rne(v.x * sc[r][0] + bs[r][0]), to_half_rne(v.y * sc[r][1] + bs[r][1]),
                                          to_half_rne(v.z * sc[r][2] + bs[r][2]), to_half_rne(v.w * sc[r][3] + bs[r][3])};
                const uint2_t u = __builtin_bit_cast(uint2_t, h);
                p[r][0] = u.x, p[r][1] = u.y;
            }
            uint32_t q[8];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const uint2_t s02 = __builtin_amdgcn_permlane32_swap(p[0][d], p[2][d], false, false);
                const uint2_t s13 = __builtin_amdgcn_permlane32_swap(p[1][d], p[3][d], false, false);
                const uint2_t lo = __builtin_amdgcn_permlane16_swap(s02.x, s13.x, false, false);
                const uint2_t hi = __builtin_amdgcn_permlane16_swap(s02.y, s13.y, false, false);
                q[d] = lo.x, q[2 + d] = lo.y, q[4 + d] = hi.x, q[6 + d] = hi.y;
            }
            const int m = m0 + 16 * t + col_e;
            if (m < M) {
                uint4_t* dst = reinterpret_cast<uint4_t*>(yh + (size_t)m * N + nw + 16 * kq_e);
                __builtin_nontemporal_store(uint4_t{q[0], q[1], q[2], q[3]}, dst);
                __builtin_nontemporal_store(uint4_t{q[4], q[5], q[6], q[7]}, dst + 1);
            }
        }
        return;
    }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int m = m0 + 16 * t + col_e;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float4_t v = acc[r][t];
            const float o[4] = {v.x * sc[r][0] + bs[r][0], v.y * sc[r][1] + bs[r][1], v.z * sc[r][2] + bs[r][2],
                                v.w * sc[r][3] + bs[r][3]};
            if (m < M)
                put((size_t)m * N + nw + 16 * r + 4 * kq_e, o);
        }
    }
}
#undef PP_DESC_X
#undef PP_DESC_W
#undef PP_DESC_S
#undef PP_DESC_Z

// Grouped launch: tile row tile_y is item tile_y of the table (of the one node that it holds, rows from tile_y tile_rows on), a node of the common shape and format with at most
// tile_rows rows of its own (the experts of a mixture-of-experts layer over their gathered rows).  Workgroups of one
// item sit together in a super-tile and share its activations in L2.
template <bool ZP_TABLE, bool PRESCALE, int NT, int GPB, int R>
__global__ __launch_bounds__(256, pp_waves(NT, GPB, R == 4 && ZP_TABLE)) void fcc_prefill_async_grouped_kernel(
    const BatchGroupTable tab, const BatchGroupItem* __restrict__ dev_tab, const RoutedHeader* __restrict__ dev_hdr,
    float* __restrict__ ws, unsigned* __restrict__ counters, int N, int K, int kb_total, int kb_per_group, int ng,
    int zp_const, int out_f32, int glu, int tiles_x, int tiles_y, int tile_rows, int full_tiles, int tail_split, int kb_per_split,
    const int* __restrict__ row_map, int x_rows, int one_node) {
    // the table travels in the kernel arguments, or -- when the rows were bucketed on the device -- lies in memory,
    // with the slice count and the cut along K that the routing kernel chose for it
    if (dev_tab) {
        const RoutedHeader h = *dev_hdr;
        if ((int)blockIdx.x >= h.grid)
            return;
        tiles_y = h.tiles_y, tail_split = h.split_k, kb_per_split = h.kb_per_split, full_tiles = h.full_tiles;
    }
    TileWork wk = tile_work(tiles_x, tiles_y, full_tiles, tail_split, kb_per_split, kb_total, tile_rows, pp_bn(R) / 2);
    BatchGroupItem it = dev_tab ? dev_tab[wk.tile_y] : tab.item[one_node ? 0 : wk.tile_y];
    if (one_node) {  // its rows wk.m0 .. + tile_rows
        it.x = static_cast<const half_t*>(it.x) + (size_t)wk.m0 * K;
        it.y = static_cast<char*>(it.y) + (size_t)wk.m0 * (glu ? N / 2 : N) * (out_f32 ? 4 : 2);
        it.M = min(tile_rows, it.M - wk.m0);
    }
    // The item and its share of the work are the same for every lane, but the compiler cannot tell: without this, every
    // buffer load of the body sits in a loop that looks for lanes with equal descriptors (six vector instructions and a
    // branch per load).
    it.w = uniform_ptr(it.w), it.scale = uniform_ptr(it.scale), it.zp = uniform_ptr(it.zp);
    it.bias = uniform_ptr(it.bias), it.x = uniform_ptr(it.x), it.y = const_cast<void*>(uniform_ptr(it.y));
    it.M = __builtin_amdgcn_readfirstlane(it.M);
    if (it.M <= 0)
        return;
    wk.m0 = 0;
    wk.tile_x = __builtin_amdgcn_readfirstlane(wk.tile_x), wk.z = __builtin_amdgcn_readfirstlane(wk.z);
    wk.split_k = __builtin_amdgcn_readfirstlane(wk.split_k), wk.park_slot = __builtin_amdgcn_readfirstlane(wk.park_slot);
    wk.kb_lo = __builtin_amdgcn_readfirstlane(wk.kb_lo), wk.kb_hi = __builtin_amdgcn_readfirstlane(wk.kb_hi);
    auto body = [&](auto rows) {
        prefill_pair_body<ZP_TABLE, PRESCALE, decltype(rows)::value, GPB, R>(
            (const uint4_t*)it.w, (const half_t*)it.scale, (const uint8_t*)it.zp, (const half_t*)it.x, (const half_t*)it.bias,
            it.y, ws, counters, it.M, N, K, kb_total, kb_per_group, ng, zp_const, out_f32, glu, wk,
            row_map ? row_map + __builtin_amdgcn_readfirstlane(it.reserved) : nullptr, x_rows, tile_rows);
    };
    if (it.M <= 64)
        body(std::integral_constant<int, 4>{});
    else if (NT == 5 || it.M <= 80)
        body(std::integral_constant<int, 5>{});
    else if (it.M <= 96)
        body(std::integral_constant<int, 6>{});
    else
        body(std::integral_constant<int, NT>{});
}

template <typename Kern>
static int allow_lds(Kern kern, bool* done) {
    if (*done)
        return 0;  // the attribute is idempotent, a race only repeats it
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)PP_LDS);
    if (e == hipSuccess)
        *done = true;
    return (int)e;
}

template <bool ZPT, bool PRE, int NT, int GPB, int R = 4>
static int launch_grouped_impl(const BatchGroupTable& tab, const BatchGroupItem* dev_tab, const RoutedHeader* dev_hdr,
                               const FcDeviceArgs& a, const LaunchPlan& p, hipStream_t s, int one_node) {
    const Layout& L = a.layout;
    auto kern = fcc_prefill_async_grouped_kernel<ZPT, PRE, NT, GPB, R>;
    static bool attr_set = false;  // per instantiation
    if (int e = allow_lds(kern, &attr_set))
        return e;
    hipLaunchKernelGGL(kern, dim3(p.grid[0], 1, 1), dim3(256), PP_LDS, s, tab, dev_tab, dev_hdr, a.workspace, a.counters,
                       (int)a.N, (int)a.K, (int)L.k_blocks, (int)L.kblocks_per_group, (int)L.groups, L.zp_const, a.out_f32,
                       L.glu, p.tiles_x, p.tiles_y, p.tile_m, p.full_tiles, p.split_k, p.kblocks_per_split, a.row_map,
                       (int)a.x_rows, one_node);
    return (int)hipGetLastError();
}

static int launch_pair(const BatchGroupTable& tab, const BatchGroupItem* dev_tab, const RoutedHeader* dev_hdr, const FcDeviceArgs& a,
                       const LaunchPlan& p, hipStream_t s, int one_node) {
    const Layout& L = a.layout;
    if (p.tile_n == PP_BN / 2) {
        if (!one_node || L.groups == 1)
            return (int)hipErrorInvalidValue;
        if (L.groups_per_kblock == 2)
            return L.zp_table ? launch_grouped_impl<true, true, 8, 2, 2>(tab, dev_tab, dev_hdr, a, p, s, 1)
                              : launch_grouped_impl<false, true, 8, 2, 2>(tab, dev_tab, dev_hdr, a, p, s, 1);
        if (L.groups_per_kblock == 4)
            return L.zp_table ? launch_grouped_impl<true, true, 8, 4, 2>(tab, dev_tab, dev_hdr, a, p, s, 1)
                              : launch_grouped_impl<false, true, 8, 4, 2>(tab, dev_tab, dev_hdr, a, p, s, 1);
        return L.zp_table ? launch_grouped_impl<true, true, 8, 1, 2>(tab, dev_tab, dev_hdr, a, p, s, 1)
                          : launch_grouped_impl<false, true, 8, 1, 2>(tab, dev_tab, dev_hdr, a, p, s, 1);
    }
    if (L.groups_per_kblock == 2)
        return L.zp_table ? launch_grouped_impl<true, true, 8, 2>(tab, dev_tab, dev_hdr, a, p, s, one_node)
                          : launch_grouped_impl<false, true, 8, 2>(tab, dev_tab, dev_hdr, a, p, s, one_node);
    if (L.groups_per_kblock == 4 && L.zp_table)
        return p.tile_m <= 80 ? launch_grouped_impl<true, true, 5, 4>(tab, dev_tab, dev_hdr, a, p, s, one_node)
                              : launch_grouped_impl<true, true, 8, 4>(tab, dev_tab, dev_hdr, a, p, s, one_node);
    if (L.groups_per_kblock == 4)
        return launch_grouped_impl<false, true, 8, 4>(tab, dev_tab, dev_hdr, a, p, s, one_node);
    if (L.groups == 1)
        return L.zp_table ? launch_grouped_impl<true, false, 8, 1>(tab, dev_tab, dev_hdr, a, p, s, one_node)
                          : launch_grouped_impl<false, false, 8, 1>(tab, dev_tab, dev_hdr, a, p, s, one_node);
    return L.zp_table ? launch_grouped_impl<true, true, 8, 1>(tab, dev_tab, dev_hdr, a, p, s, one_node)
                      : launch_grouped_impl<false, true, 8, 1>(tab, dev_tab, dev_hdr, a, p, s, one_node);
}

// The launch must be what tile_work assumes: a 1-D grid of full_tiles whole tiles plus split_k parts of each remaining
// tile, parts that cover K.
static bool pair_plan_ok(const FcDeviceArgs& a, const LaunchPlan& p) {
    const int64_t tiles = (int64_t)p.tiles_x * p.tiles_y;
    return (p.tile_n == PP_BN || p.tile_n == PP_BN / 2) && p.tiles_x == (a.N + p.tile_n - 1) / p.tile_n && a.N % (PP_BN / 2) == 0 && p.tiles_y >= 1 && p.full_tiles >= 0 &&
           p.full_tiles <= tiles && p.split_k >= 1 && (int64_t)p.kblocks_per_split * p.split_k >= a.layout.k_blocks &&
           (p.full_tiles == tiles || (p.kblocks_per_split >= 1 && (int64_t)p.kblocks_per_split * (p.split_k - 1) < a.layout.k_blocks)) &&
           p.grid[0] == (unsigned)(p.full_tiles + (tiles - p.full_tiles) * p.split_k) && p.grid[1] == 1 && p.grid[2] == 1 &&
           (p.split_k == 1 || (a.workspace && a.counters));
}

// p plans one node of n_items * tile_m rows: its tile rows are the items of the table.  dev_tab and dev_hdr
// (optional, both or none): table and header in device memory, written by the routing kernel earlier on the same
// stream -- at most n_items entries of at most tile_m rows each; how many are in use and how K is cut for them is
// the header's word, and p only sizes the launch: a 1-D grid, workspace and counters that hold
// routed_header(tiles_x, t, k_blocks, .).grid workgroups for every t <= n_items.  `tab` is then ignored and n_items
// is not limited to kMaxGroupItems.
int launch_prefill_async_grouped(const BatchGroupTable& tab, int n_items, const FcDeviceArgs& a, const LaunchPlan& p,
                                 void* stream, const BatchGroupItem* dev_tab, const RoutedHeader* dev_hdr) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Layout& L = a.layout;
    if (L.bits != 4 || a.N % PP_BN != 0 || n_items < 1 || p.tiles_y != n_items || !dev_tab != !dev_hdr ||
        (p.tile_m != 128 && p.tile_m != 96 && p.tile_m != 80 && p.tile_m != 64) ||
        (a.row_map && (!dev_tab || a.x_rows < 1 || a.x_rows * a.K * 2 >= ((int64_t)1 << 31))))
        return (int)hipErrorInvalidValue;
    if (!dev_tab) {
        if (!pair_plan_ok(a, p) || n_items > kMaxGroupItems)
            return (int)hipErrorInvalidValue;
        for (int i = 0; i < n_items; ++i)
            if (tab.item[i].M < 1 || tab.item[i].M > p.tile_m)
                return (int)hipErrorInvalidValue;
    } else {
        if (p.tiles_x != a.N / PP_BN || p.grid[1] != 1 || p.grid[2] != 1)
            return (int)hipErrorInvalidValue;
        for (int t = 1; t <= n_items; ++t) {
            const RoutedHeader h = routed_header(p.tiles_x, t, (int)L.k_blocks, p.n_cus);
            if ((unsigned)h.grid > p.grid[0] ||
                (h.split_k > 1 && (!a.workspace || !a.counters ||
                                   (size_t)routed_parked_tiles(h, p.tiles_x) * p.tile_m * PP_BN * sizeof(float) > p.workspace_bytes ||
                                   (size_t)p.tiles_x * t > p.counter_count)))
                return (int)hipErrorInvalidValue;
        }
    }
    return launch_pair(tab, dev_tab, dev_hdr, a, p, s, 0);
}

// One node of any number of rows, as plan_pair plans it: the grouped kernel over the node's own row tiles.
int launch_prefill_pair(const FcDeviceArgs& a, const LaunchPlan& p, void* stream) {
    if (a.layout.bits != 4 || a.M < 1 || a.M * a.K * 2 >= ((int64_t)1 << 31) || (int64_t)p.tiles_y * p.tile_m < a.M ||
        (p.tile_m != 128 && p.tile_m != 96 && p.tile_m != 80 && p.tile_m != 64) || !pair_plan_ok(a, p))
        return (int)hipErrorInvalidValue;
    BatchGroupTable tab = {};
    tab.item[0] = BatchGroupItem{a.w, a.scale, a.zp, a.bias, a.x, a.y, (int)a.M, 0};
    return launch_pair(tab, nullptr, nullptr, a, p, static_cast<hipStream_t>(stream), 1);
}

}  // namespace ovfcc
