// Kernel choice and launch decomposition (host only).
//
// Policy: nodes that fit no tile run the ragged kernels (one scale per channel; plan_ragged) or the plain kernel; tiled
// nodes run a decode kernel for M <= 48 and a prefill kernel for more (the roofline ridge of int4 g128 sits near
// M = 83).  plan_launch chooses among the decode kernels that keep their activations (one channel tile per workgroup,
// matrix-vector, 16-row, small-batch); of its choices the weight-streaming kernel takes what stream_preferred names.
// The caller cuts 48 < M <= 128 into decode launches: a single 128-row prefill tile per column block leaves most of
// the chip idle.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "ovfcc_internal.h"

namespace ovfcc {

// Overrides from the process environment, read once -- at the first use, which ovfcc_init forces -- and again only
// by env_reload (tests and experiments that change the environment of a running process).
//   tuning:  OVFCC_DECODE_WAVES = 4 | 8 | 16 (workgroup size), OVFCC_DECODE_RT = 1 | 2 | 4 (channel tiles per
//            workgroup or wave), OVFCC_DECODE_XLDS = 0 | 1 (activations via LDS), OVFCC_DECODE_BATCH = 0 | 1
//            (small-batch kernel instead of the streaming kernel), OVFCC_GEMV = 0 | 1, OVFCC_GEMV_C = 2 | 4 | 8,
//            OVFCC_GEMV16 = 0 | 1 (the 16-row kernel with stationary activations for 5-48 rows),
//            OVFCC_GEMV16_GRID = n (its workgroups per row tile), OVFCC_GEMV16_SPLIT = 1 | 2 | 4 | 8 (parts it cuts K in),
//            OVFCC_GEMV16_STREAM = 0 | 1 (the 16-row kernel that streams its activations, 5-16 rows),
//            OVFCC_GEMV16_STREAM_TILES = 1 | 2 | 4 (its channel tiles per workgroup),
//            OVFCC_STREAM = 0 | 1 (the weight-streaming kernel nowhere, wherever it can run; without it any of the
//            overrides above keeps the kernel that they are about),
//            OVFCC_PREFILL_{DIRECT, ASYNC, WIDE, BIG, TAIL} = 0 | 1 (BIG: 256 x 256 tiles of 4-bit and of int8-activation nodes), OVFCC_PREFILL_ROWS = 64 | 128,
//            OVFCC_PREFILL_PAIR = 0 | 1 (two workgroups per compute unit nowhere, wherever that kernel can run; without it any of
//            the overrides above keeps the kernel that they are about),
//            OVFCC_MOE_HOST_ROUTING = 1, OVFCC_MLP_FUSED = 1 (an MLP node of up to four rows as one launch instead of two),
//            OVFCC_MLP_GRID = n (its workgroups), OVFCC_MLP_SPIN_LIMIT = n (polls after which that launch's wait for its workgroups gives up; tests);
//   logging: OVFCC_VERBOSE = 1 (one line per launch on stderr), 2 (also weights and requests as they come and go).
namespace {
struct EnvEntry {
    const char* name;
    bool decode;  // chooses or shapes one of the older decode kernels
    std::atomic<int> set{0};
    std::atomic<int> value{0};
    explicit EnvEntry(const char* n, bool d = false) : name(n), decode(d) {}
};
EnvEntry g_env[] = {EnvEntry("OVFCC_DECODE_WAVES", true),   EnvEntry("OVFCC_DECODE_RT", true),
                    EnvEntry("OVFCC_DECODE_XLDS", true),    EnvEntry("OVFCC_DECODE_BATCH", true),
                    EnvEntry("OVFCC_GEMV", true),           EnvEntry("OVFCC_GEMV_C", true),
                    EnvEntry("OVFCC_GEMV16", true),         EnvEntry("OVFCC_GEMV16_GRID", true),
                    EnvEntry("OVFCC_GEMV16_SPLIT", true),   EnvEntry("OVFCC_GEMV16_STREAM", true),
                    EnvEntry("OVFCC_GEMV16_STREAM_TILES", true), EnvEntry("OVFCC_STREAM"),
                    EnvEntry("OVFCC_PREFILL_DIRECT"), EnvEntry("OVFCC_PREFILL_ASYNC"),  EnvEntry("OVFCC_PREFILL_WIDE"),
                    EnvEntry("OVFCC_PREFILL_BIG"),    EnvEntry("OVFCC_PREFILL_PAIR"),    EnvEntry("OVFCC_PREFILL_TAIL"),   EnvEntry("OVFCC_PREFILL_ROWS"),
                    EnvEntry("OVFCC_MOE_HOST_ROUTING"), EnvEntry("OVFCC_MLP_FUSED"),      EnvEntry("OVFCC_MLP_SPIN_LIMIT"),
                    EnvEntry("OVFCC_MLP_GRID"),
                    EnvEntry("OVFCC_VERBOSE")};
std::atomic<bool> g_decode_overridden{false};
std::atomic<unsigned> g_env_generation{0};
std::once_flag g_env_once;

void env_read_all() {
    bool decode = false;
    for (EnvEntry& e : g_env) {
        const char* v = std::getenv(e.name);
        e.value.store(v ? std::atoi(v) : 0, std::memory_order_relaxed);
        e.set.store(v ? 1 : 0, std::memory_order_release);
        decode |= v && e.decode;
    }
    g_decode_overridden.store(decode, std::memory_order_release);
    g_env_generation.fetch_add(1, std::memory_order_acq_rel);
}
}  // namespace

void env_reload() {
    std::call_once(g_env_once, [] {});  // a later first use must not read again on top of this
    env_read_all();
}

unsigned env_generation() {
    std::call_once(g_env_once, env_read_all);
    return g_env_generation.load(std::memory_order_acquire);
}

bool decode_overridden() {
    std::call_once(g_env_once, env_read_all);
    return g_decode_overridden.load(std::memory_order_acquire);
}

int env_int(const char* name, int fallback) {
    std::call_once(g_env_once, env_read_all);
    for (EnvEntry& e : g_env)
        if (std::strcmp(e.name, name) == 0)
            return e.set.load(std::memory_order_acquire) ? e.value.load(std::memory_order_relaxed) : fallback;
    const char* v = std::getenv(name);  // a name the table does not know
    return v ? std::atoi(v) : fallback;
}

// k-blocks per wave of the matrix-vector kernel for this node (0: the kernel does not fit it).  The waves of one
// channel tile (of a gate / up tile pair) share a workgroup of at most 16 waves and each takes 2, 4 or 8 whole
// k-blocks; of the divisions that fit, the coarsest one that still gives every SIMD of the chip about two waves,
// but no coarser than a workgroup of eight waves needs.
// OVFCC_GEMV_C overrides for experiments.
int gemv_kblocks_per_wave(const Layout& L, int n_cus) {
    const int tiles_per_wg = L.glu ? 2 : 1;
    if (L.glu && (L.n_tiles & 1))
        return 0;
    auto fits = [&](int c) { return L.k_blocks % c == 0 && (L.k_blocks / c) * tiles_per_wg <= 16; };
    const int forced = env_int("OVFCC_GEMV_C", 0);
    if ((forced == 2 || forced == 4 || forced == 8) && fits(forced))
        return forced;
    int best = 0;
    for (int c : {2, 4, 8})
        if (fits(c) && (best == 0 || L.n_tiles * (L.k_blocks / c) >= (int64_t)8 * n_cus))
            best = c;
    // Eight k-blocks per wave leave a plain node of K = 4096 with four waves per workgroup; eight waves of four
    // k-blocks stream the same bytes faster (gate / up at one row: 7.0 against 7.3 us) and give the 16-row kernel
    // two waves per SIMD (16 rows: 10.7 against 12.8 us).
    if (best == 8 && !L.glu && fits(4) && L.k_blocks / 4 <= 8)
        best = 4;
    return best;
}

// Dynamic LDS of the matrix-vector kernel: every wave stages its rows (1, 2 or 4 carried; c k-blocks of 256 bytes
// each plus a 64-byte pad per row) and leaves 16 partial sums per row.
size_t gemv_lds_bytes(int c, int m, int waves) {
    const int mr = m == 1 ? 1 : m == 2 ? 2 : 4;
    return (size_t)waves * mr * (c * 256 + 64) + (size_t)waves * mr * 16 * sizeof(float);
}

int plan_launch(const FcDeviceArgs& a, int force_kernel, int force_split, int n_cus, LaunchPlan* plan) {
    LaunchPlan p;
    const Layout& L = a.layout;
    int kernel = force_kernel;
    if (kernel == OVFCC_KERNEL_AUTO)
        kernel = !L.tiled ? OVFCC_KERNEL_PLAIN : (a.M <= kDecodeMaxRows ? OVFCC_KERNEL_DECODE : OVFCC_KERNEL_PREFILL);
    if (kernel != OVFCC_KERNEL_PLAIN && !L.tiled)
        return fail(OVFCC_EUNSUPPORTED, "this node fits no tile; only the plain family can run it");
    if (kernel == OVFCC_KERNEL_PLAIN && L.tiled)
        return fail(OVFCC_EUNSUPPORTED, "this node was repacked into tiles; the plain family runs nodes that fit no tile");
    if (kernel == OVFCC_KERNEL_DECODE && a.M > kDecodeMaxRows)
        return fail(OVFCC_EUNSUPPORTED, "the decode kernels handle at most 48 rows per launch");
    if (kernel == OVFCC_KERNEL_PREFILL && (a.N % kPrefillTileN) != 0)
        return fail(OVFCC_EUNSUPPORTED, "the prefill kernel needs N % 128 == 0");
    p.kernel = kernel;
    // Small-batch kernel: waves own channel tiles, the workgroup shares one staged slice of X.  It pays
    // for its split-K epilogue, so the streaming kernel keeps M <= 4 and, for small nodes, M <= 16.
    const bool want_batch =
        env_int("OVFCC_DECODE_BATCH", (a.M > 16 || (a.M > 4 && L.w_bytes >= ((size_t)16 << 20))) ? 1 : 0) != 0;
    auto plan_batch = [&]() -> int {
        const int kb = (int)L.k_blocks;
        const int mt = (int)((a.M + 15) / 16);
        int rt = 1;
        const int rt_env = env_int("OVFCC_DECODE_RT", 0);
        if (rt_env == 1 || rt_env == 2)
            rt = rt_env;
        int nw = 8;
        const int nw_env = env_int("OVFCC_DECODE_WAVES", 0);
        if (nw_env == 4 || nw_env == 8)
            nw = nw_env;
        const int64_t groups = (L.n_tiles + nw * rt - 1) / (nw * rt);
        auto x_bytes = [&](int per) { return (size_t)16 * mt * ((size_t)per * kBlockK + 8) * 2; };
        const size_t lds_budget = 96 * 1024;
        int split = force_split;
        if (split <= 0) {
            // split K until the grid covers the compute units (keeping at least two k-blocks per workgroup)
            split = 1;
            while (groups * split < n_cus && split < 8 && kb / (split * 2) >= 2)
                split *= 2;
        }
        if (split > kb)
            split = kb;
        while (split < kb && x_bytes((kb + split - 1) / split) > lds_budget)
            split = split * 2 < kb ? split * 2 : kb;  // the staged slice of X has to fit in LDS
        const int per = (kb + split - 1) / split;
        split = (kb + per - 1) / per;  // no empty splits
        if (x_bytes(per) > lds_budget)
            return fail(OVFCC_EUNSUPPORTED, "one k-block of the activations does not fit in LDS");
        p.batch = true;
        p.split_k = split;
        p.kblocks_per_split = per;
        p.tiles_per_group = rt;
        p.grid[0] = (unsigned)groups;
        p.grid[1] = (unsigned)split;
        p.block = 64u * nw;
        p.tile_m = 16 * mt;
        p.tile_n = 16 * rt * nw;
        p.workspace_bytes = split > 1 ? (size_t)groups * split * nw * rt * mt * 256 * sizeof(float) : 0;
        p.counter_count = split > 1 ? (size_t)groups : 0;
        p.dynamic_lds = (unsigned)x_bytes(per);
        p.name = L.bits == 4 ? "fcc_batch_w4" : "fcc_batch_w8";
        return OVFCC_OK;
    };
    // Five to 48 rows of a 4-bit node with groups of 128 inputs whose 16 rows x K of activations fit in LDS (and,
    // divided among the waves, in registers): the 16-row sibling of the matrix-vector kernel.  Every workgroup
    // keeps its row tile of the activations and walks channel tiles; the grid is as many workgroups as the chip
    // holds at once, rounded so that all of them visit the same number of tiles.
    auto plan_gemv16 = [&]() -> bool {
        if (a.M <= 4 || a.M > kDecodeMaxRows || !a.scale_cm || L.bits != 4 || L.groups_per_kblock != 1 ||
            L.kblocks_per_group != 1 || force_split > 0 || L.gemv_c == 0 || (L.glu && (L.n_tiles & 1)) ||
            env_int("OVFCC_GEMV16", 1) == 0 ||
            env_int("OVFCC_DECODE_BATCH", -1) >= 0 || L.n_tiles * L.k_blocks * kTileBytes >= ((int64_t)1 << 30))
            return false;
        const size_t lds_limit = 160 * 1024 - 64;
        const int64_t rows = (a.M + 15) / 16;
        const int64_t units = L.glu ? L.n_tiles / 2 : L.n_tiles;  // visited in one go: tiles, or pairs of gate and up tile
        // K whole where 16 rows x K fit in LDS and the waves in the register file; else cut in 2, 4 or 8 parts whose
        // partial sums a second launch adds (OVFCC_GEMV16_SPLIT picks the number of parts)
        const int split_env = env_int("OVFCC_GEMV16_SPLIT", 0);
        for (int split : {1, 2, 4, 8}) {
            if (split_env > 0 && split != split_env)
                continue;
            // (up to 16 rows, four parts and their second launch only tie with the small-batch kernel -- 14336 -> 4096:
            // 12.8 against 12.7 us; from 17 rows on they are ahead, 16.2 against 21.5 us at 32 rows -- while two
            // parts are ahead from the start: 8192 -> 8192 at 16 rows 12.5 against 14.7 us)
            if (split > 1 && (L.glu || L.gemv_c % split != 0 || (a.N & 3) || (a.M <= 16 && split > 2 && split_env <= 0)))
                continue;
            // the kernel's registers allow 8 and 16 waves per compute unit with 4 and 2 k-blocks per wave
            const int c = gemv16_kblocks_per_wave(L.gemv_c, split);
            if (c != 2 && c != 4)
                continue;
            const int waves = (int)(L.k_blocks / c / split);
            const int cu_waves = c == 4 ? 8 : 16;
            if (waves < 1 || waves > cu_waves)
                continue;
            const size_t lds2 = gemv16_lds_bytes(c, waves, 2);
            const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>((int64_t)(160 * 1024 / lds2), cu_waves / waves));
            const int64_t at_once = std::max<int64_t>(1, (int64_t)n_cus * per_cu / (rows * split));
            int64_t visits = (units + at_once - 1) / at_once;
            int64_t grid = (units + visits - 1) / visits;
            const int grid_env = env_int("OVFCC_GEMV16_GRID", 0);
            if (grid_env > 0) {
                grid = std::min<int64_t>(grid_env, units);
                visits = (units + grid - 1) / grid;
            }
            const size_t lds = gemv16_lds_bytes(c, waves, (L.glu || grid < units) ? 2 : 1);
            if (lds > lds_limit)
                continue;
            p.gemv16 = true;
            p.gemv_c = L.gemv_c;
            p.split_k = split;
            p.kblocks_per_split = (int)(L.k_blocks / split);
            p.tiles_per_group = (int)(visits * (L.glu ? 2 : 1));
            p.grid[0] = (unsigned)grid;
            p.grid[1] = (unsigned)rows;
            p.grid[2] = (unsigned)split;
            p.block = 64u * waves;
            p.tile_m = 16;
            p.tile_n = 16;
            p.dynamic_lds = (unsigned)lds;
            p.workspace_bytes = split > 1 ? (size_t)split * 16 * rows * a.N * sizeof(float) : 0;
            p.name = "fcc_gemv16_w4";
            return true;
        }
        return false;
    };
    // Five to sixteen rows where the kernel above has nothing to keep -- K too long for it (the down projection of
    // an MLP), or no more channel tiles than compute units, so that every workgroup would visit one tile and wait
    // for all of its activations first: the 16-row kernel that streams its activations k-block by k-block, one
    // workgroup per channel tile over all of K -- no split along K, no second launch (4096 -> 4096 at 16 rows:
    // 4.8 against 5.4 us; 14336 -> 4096 at 8 rows: 10.1 against 12.4 us for the small-batch kernel, at 16 rows 12.1
    // against 12.7; 4096 -> 1024, a quarter of the compute units: 3.75-4.7 against 3.9-4.8).  From 17 rows on every
    // tile's weights would be streamed twice.  OVFCC_GEMV16_STREAM = 0 switches it off, = 1 takes
    // it wherever it can run (before the kernel above, and whatever the number of channel tiles).
    const int stream_env = env_int("OVFCC_GEMV16_STREAM", -1);
    // Channel tiles per workgroup (their activations travel once for all of them): two where the node has more
    // tiles than the chip has compute units; OVFCC_GEMV16_STREAM_TILES = 1 | 2 | 4 overrides.  Measured against the
    // kernel above (8 / 16 rows): 4096 -> 8192 5.96 / 6.55 against 6.92 / 7.71 us, 4096 -> 6144 5.51 / 6.02 against
    // 6.53 / 7.22, 8192 -> 8192 9.08 / 10.29 against 11.90 / 12.45 (K in two parts and a summing launch) -- one round
    // of workgroups, taken up to 16 rows; 4096 -> 14336 (448 workgroups) 8.60 / 9.90 against 9.19 / 9.96 -- taken up
    // to 8 rows; 4096 -> 28672 (896 workgroups) 14.7 against 13.3 -- left to the kernel above.
    const int stream_tiles =
        env_int("OVFCC_GEMV16_STREAM_TILES", L.n_tiles > n_cus && L.n_tiles % 2 == 0 ? 2 : 1);
    const int64_t stream_wgs = L.n_tiles / (stream_tiles == 2 || stream_tiles == 4 ? stream_tiles : 1);
    const bool stream_first = stream_env == 1 || stream_wgs <= n_cus || (stream_wgs <= 2 * (int64_t)n_cus && a.M <= 8);
    auto plan_gemv16_stream = [&]() -> bool {
        if (a.M <= 4 || a.M > 16 || !a.scale_cm || L.bits != 4 || L.groups_per_kblock != 1 || L.kblocks_per_group != 1 ||
            force_split > 0 || L.gemv_c == 0 || L.glu || env_int("OVFCC_GEMV16", 1) == 0 ||
            stream_env == 0 || env_int("OVFCC_GEMV16_SPLIT", 0) > 0 || env_int("OVFCC_GEMV16_GRID", 0) > 0 ||
            env_int("OVFCC_DECODE_BATCH", -1) >= 0 || L.n_tiles * L.k_blocks * kTileBytes >= ((int64_t)1 << 31))
            return false;
        const int waves = (int)(L.k_blocks / L.gemv_c);
        if (L.k_blocks % L.gemv_c != 0 || waves < 1 || waves > 16 || (stream_env != 1 && L.n_tiles * 4 < n_cus))
            return false;
        int tiles = stream_tiles;
        if ((tiles != 1 && tiles != 2 && tiles != 4) || L.n_tiles % tiles != 0)
            tiles = 1;
        while (tiles > 1 && gemv16s_lds_bytes(waves, tiles) > 160 * 1024 - 64)
            tiles >>= 1;
        if (gemv16s_lds_bytes(waves, tiles) > 160 * 1024 - 64)
            return false;
        p.gemv16_stream = true;
        p.gemv_c = L.gemv_c;
        p.split_k = 1;
        p.kblocks_per_split = (int)L.k_blocks;
        p.tiles_per_group = tiles;
        p.grid[0] = (unsigned)(L.n_tiles / tiles);
        p.grid[1] = 1;
        p.grid[2] = 1;
        p.block = 64u * waves;
        p.tile_m = 16;
        p.tile_n = 16;
        p.dynamic_lds = (unsigned)gemv16s_lds_bytes(waves, tiles);
        p.workspace_bytes = 0;
        p.name = "fcc_gemv16s_w4";
        return true;
    };
    if (kernel == OVFCC_KERNEL_PLAIN) {
        if (a.M > 65535)
            return fail(OVFCC_EUNSUPPORTED, "the plain kernel handles at most 65535 rows");
        p.grid[0] = (unsigned)a.N_out;
        p.grid[1] = (unsigned)a.M;
        p.block = 64;
        p.name = "fcc_plain";
    } else if (kernel == OVFCC_KERNEL_DECODE && ((stream_first && plan_gemv16_stream()) || plan_gemv16() || plan_gemv16_stream())) {
        // planned
    } else if (kernel == OVFCC_KERNEL_DECODE && want_batch) {
        if (int rc = plan_batch())
            return rc;
    } else if (kernel == OVFCC_KERNEL_DECODE && a.M <= 4 && a.scale_cm && L.bits == 4 && L.groups_per_kblock == 1 &&
               L.kblocks_per_group == 1 && force_split <= 0 && env_int("OVFCC_GEMV", 1) != 0 && L.gemv_c != 0) {
        // One to four rows of a 4-bit node with groups of 128 inputs: the matrix-vector kernel.
        const int c = L.gemv_c;
        const int tiles_per_wg = L.glu ? 2 : 1;
        const int waves = (int)(L.k_blocks / c) * tiles_per_wg;
        p.gemv = true;
        p.gemv_c = c;
        p.split_k = 1;
        p.kblocks_per_split = (int)L.k_blocks;
        p.tiles_per_group = tiles_per_wg;
        p.grid[0] = (unsigned)(L.n_tiles / tiles_per_wg);
        p.block = 64u * waves;
        p.tile_m = 16;
        p.tile_n = 16 * tiles_per_wg;
        p.dynamic_lds = (unsigned)gemv_lds_bytes(c, (int)a.M, waves);
        p.name = "fcc_gemv_w4";
    } else if (kernel == OVFCC_KERNEL_DECODE) {
        if (a.M > 32)
            return fail(OVFCC_EUNSUPPORTED, "the streaming decode kernel handles at most 32 rows");
        const int kb = (int)L.k_blocks;
        const int mt = a.M <= 16 ? 1 : 2;
        // Activations go through LDS for M <= 4 when the k-range of one workgroup fits 40 KiB.
        bool xlds = a.M <= 4;
        const int x_env = env_int("OVFCC_DECODE_XLDS", -1);
        if (x_env == 0)
            xlds = false;
        int split = force_split;
        if (split <= 0) {
            split = 1;
            // K is split over workgroups only when the grid would otherwise leave compute units idle
            // (few channel tiles, long rows)
            const int64_t want_waves = (int64_t)16 * n_cus;
            while (split < 8 && L.n_tiles * 16 * split * 2 <= want_waves && kb / (split * 2) >= 32)
                split *= 2;
        }
        if (split > kb)
            split = kb;
        const int per = (kb + split - 1) / split;
        split = (kb + per - 1) / per;  // no empty splits
        const size_t x_bytes = (size_t)a.M * ((size_t)per * kBlockK + 8) * 2;
        if (x_bytes > 40 * 1024)  // does not fit beside the reduction buffer: read the operand from L2 instead
            xlds = false;
        // Two to four rows of a long-K, large node whose activations do not fit: the small-batch kernel's
        // shared staged slice beats per-lane reads of X from L2 (measured on K = 14336, N = 4096).
        if (!xlds && x_env != 0 && a.M > 1 && a.M <= 4 && L.w_bytes >= ((size_t)16 << 20) &&
            env_int("OVFCC_DECODE_BATCH", -1) < 0 && force_split <= 0) {
            if (int rc = plan_batch())
                return rc;
            *plan = p;
            return OVFCC_OK;
        }
        // Channel tiles per workgroup: one.  More tiles would share a staged activation copy between more
        // weights, but measured slower at M <= 4 (fewer, longer workgroups); the override stays for experiments.
        int rt = 1;
        if (xlds) {
            const int rt_max = L.bits == 4 ? 4 : 2;
            const int rt_env = env_int("OVFCC_DECODE_RT", 0);
            if ((rt_env == 1 || rt_env == 2 || rt_env == 4) && rt_env <= rt_max && L.n_tiles % rt_env == 0)
                rt = rt_env;
        }
        // A gated linear unit needs a gate tile and its up tile in one workgroup, which only the LDS-staged form
        // of this kernel offers; otherwise the small-batch kernel takes the node.
        if (L.glu && !xlds) {
            if (int rc = plan_batch())
                return rc;
            *plan = p;
            return OVFCC_OK;
        }
        if (L.glu && rt < 2)
            rt = 2;
        const int64_t groups = L.n_tiles / rt;
        // waves per workgroup: as many as the k-range feeds with four k-blocks each (the prefetch depth),
        // at most 16, and no more than about 16 waves per compute unit in total
        int nw = 16;
        while (nw > 4 && (per < 4 * nw || groups * split * nw > (int64_t)16 * n_cus || nw * rt > 32))
            nw >>= 1;
        const int nw_env = env_int("OVFCC_DECODE_WAVES", 0);
        if ((nw_env == 4 || nw_env == 8 || nw_env == 16) && nw_env * rt <= 32)
            nw = nw_env;
        p.split_k = split;
        p.kblocks_per_split = per;
        p.tiles_per_group = rt;
        p.x_in_lds = xlds;
        p.grid[0] = (unsigned)groups;
        p.grid[1] = (unsigned)split;
        p.block = 64u * nw;
        p.tile_m = 16 * mt;
        p.tile_n = 16 * rt;
        p.workspace_bytes = split > 1 ? (size_t)groups * split * rt * mt * 256 * sizeof(float) : 0;
        p.counter_count = split > 1 ? (size_t)groups : 0;
        p.dynamic_lds = (unsigned)((size_t)nw * rt * mt * 256 * sizeof(float) + (xlds ? x_bytes : 0));
        p.name = L.bits == 4 ? "fcc_decode_w4" : "fcc_decode_w8";
    } else {
        // The register-fed kernels with 256-channel tiles run whatever they can, however small the launch: they split K and
        // keep their loads in flight, where the square kernel waits for every k-block (u4 in groups of 128, 129 rows:
        // 2048 -> 2048 40.8 us there against 18.7, 14336 -> 512 268 / 27; u8 2048 -> 2048 40.7 / 27.2; i8 512 -> 1152, 200
        // rows, 13.2 / 12.2, but 384 -> 1152 11.8 / 12.2: 8-bit nodes of three k-blocks stay).  The line at 256 KiB is not
        // where the kernels cross: smaller nodes would gain too (129 rows, u4 in groups of 128: 512 -> 256 15.5 / 8.7, 1024 ->
        // 384 23.0 / 12.2; u8 512 -> 256 15.4 / 13.0) and stay only because tests check the square kernel through their calls.
        // A grouped run shares a launch only where that covers half the chip (its other slices run one by one), and
        // p.fills tells a caller that could cut the rows into decode launches.  The LDS-dequantising kernel also needs
        // K % 256 == 0.  OVFCC_PREFILL_WIDE = 0 | 1 and OVFCC_PREFILL_DIRECT = 0 | 1 override for experiments.
        const int64_t m_tiles = (a.M + kPrefillTileM - 1) / kPrefillTileM;
        const int tiles_per_kb = L.bits == 4 ? 1 : 2;
        // The register-fed kernels also run nodes that end on half a tile (its other half multiplies zeros: 1 / 46 of the
        // work at N = 5760), except grouped launches.  A node of half a tile only stays with the square kernel.
        const bool whole = (a.N % kPrefillWideN) == 0;
        const bool direct_ok = (whole || ((a.N % kPrefillTileN) == 0 && a.N > kPrefillWideN && a.tile_rows == 0 && !a.want_async)) &&
                               a.M * a.K * 2 < ((int64_t)1 << 31) &&
                               (int64_t)16 * L.k_blocks * tiles_per_kb * kTileBytes < ((int64_t)1 << 31);
        const bool wide_ok = direct_ok && whole && (a.K % 256) == 0;
        const int64_t n_wide = (a.N + kPrefillWideN - 1) / kPrefillWideN;
        // (the register-fed kernels can also split K, which multiplies their grid by up to eight)
        const bool may_split = direct_ok && env_int("OVFCC_PREFILL_DIRECT", 1) != 0;
        const bool may_async = may_split && L.bits == 4 && env_int("OVFCC_PREFILL_ASYNC", 1) != 0;
        // (and the 4-bit one has a form with 64-row tiles, which doubles the tile count of a grid that fits one round)
        int64_t reach = n_wide * m_tiles;
        if (may_split) {
            const int64_t tiles64 = n_wide * ((a.M + 63) / 64);
            if (may_async && tiles64 <= n_cus)
                reach = tiles64;
            for (int split = 1; split < 8 && reach * 2 <= n_cus && L.k_blocks / (split * 2) >= 8; split *= 2)
                reach *= 2;
        }
        p.fills = reach * 2 >= n_cus;
        bool big = p.fills || (a.want_async && may_async) || (a.tile_rows == 0 && may_split && L.w_bytes >= ((size_t)256 << 10) && (L.bits == 4 || L.k_blocks >= 4));
        const int wide_env = env_int("OVFCC_PREFILL_WIDE", -1);
        if (wide_env >= 0)
            big = wide_env != 0;
        // Groups of 32 or 64 inputs: only the all-asynchronous kernel and the square kernel carry several groups
        // per k-block.
        const bool small_groups = L.groups_per_kblock != 1;
        p.direct = big && direct_ok && env_int("OVFCC_PREFILL_DIRECT", 1) != 0 && (!small_groups || may_async);
        const bool wide = p.direct || (big && wide_ok && !small_groups);
        // 4-bit nodes take the variant whose operands all travel by direct-to-LDS loads
        p.async_dma = p.direct && L.bits == 4 && env_int("OVFCC_PREFILL_ASYNC", 1) != 0;
        p.tile_m = kPrefillTileM;
        p.tile_n = wide ? kPrefillWideN : kPrefillTileN;
        p.grid[0] = (unsigned)(wide ? n_wide : a.N / kPrefillTileN);
        p.grid[1] = (unsigned)m_tiles;
        if (p.async_dma) {
            // 64-row tiles while they still fit the compute units in one round: a 64-row tile takes two thirds of
            // the time of a 128-row tile (same weight traffic and unpack work, half the MFMAs), so it pays only
            // where 128-row tiles would leave half the chip idle.  (OVFCC_PREFILL_ROWS = 64 | 128 overrides;
            // a.tile_rows, set by the grouped run, wins over both.)
            int rows = (int64_t)p.grid[0] * ((a.M + 63) / 64) <= n_cus ? 64 : 128;
            if (const int env_rows = env_int("OVFCC_PREFILL_ROWS", 0); env_rows == 64 || env_rows == 128)
                rows = env_rows;
            if (a.tile_rows == 64 || a.tile_rows == 128)
                rows = a.tile_rows;
            // (80 and 96 rows: grouped runs only)
            if (a.tile_rows == 80 || a.tile_rows == 96)
                rows = a.tile_rows;
            if (rows != 128) {
                p.tile_m = rows == 80 || rows == 96 ? rows : 64;
                p.grid[1] = (unsigned)((a.M + p.tile_m - 1) / p.tile_m);
            }
        }
        p.kblocks_per_split = (int)L.k_blocks;
        if (p.direct) {
            // Split K while the tiles alone leave compute units idle (at least eight k-blocks per workgroup): the
            // f32 tiles are parked in the workspace and added by the last workgroup to arrive.
            // OVFCC_PREFILL_TAIL = 1 (an experiment, off by default) also splits, with more tiles than compute
            // units, the tiles of the last, partial round.  It does not pay: the chip is power-limited, a
            // half-empty round runs at a higher clock, and time is linear in tiles rather than in rounds.
            const int64_t tiles = (int64_t)p.grid[0] * p.grid[1];
            int split = force_split > 0 ? force_split : 1;
            int64_t full = 0;
            if (force_split <= 0) {
                while (split < 8 && tiles * split * 2 <= n_cus && L.k_blocks / (split * 2) >= 8)
                    split *= 2;
                const int64_t rest = tiles % n_cus;
                if (split == 1 && tiles > n_cus && rest * 2 <= n_cus && rest > 0 && L.k_blocks >= 16 &&
                    env_int("OVFCC_PREFILL_TAIL", 0) != 0) {
                    full = tiles - rest;
                    split = 2;
                    while (split < 8 && rest * split * 2 <= n_cus && L.k_blocks / (split * 2) >= 8)
                        split *= 2;
                }
            }
            if (split > L.k_blocks)
                split = (int)L.k_blocks;
            const int per = (int)((L.k_blocks + split - 1) / split);
            split = (int)((L.k_blocks + per - 1) / per);
            if (split == 1)
                full = tiles;
            p.split_k = split;
            p.kblocks_per_split = per;
            p.tiles_x = (int)p.grid[0];
            p.tiles_y = (int)p.grid[1];
            p.full_tiles = (int)full;
            p.grid[0] = (unsigned)(full + (tiles - full) * split);
            p.grid[1] = 1;
            p.workspace_bytes = split > 1 ? (size_t)(tiles - full) * split * p.tile_m * kPrefillWideN * sizeof(float) : 0;
            p.counter_count = split > 1 ? (size_t)(tiles - full) : 0;
        }
        p.block = wide ? 512 : 256;
        // 256 x 256 tiles (four waves with 512 registers each), where every unpacked weight meets twice the rows:
        // measured, such a tile costs 1.7 to 1.8 times a 128 x 256 tile.  It is whole tiles only, so it pays where
        // its rounds of tiles over the compute units, at that price, are no more than the rounds of the smaller
        // tiles: 256, 448, 512, 896, 1792 tiles yes; 128 or 300 no.  OVFCC_PREFILL_BIG = 0 | 1 overrides (1: whenever
        // the kernel can run the node).  A grouped run (a.tile_rows set) keeps its one row tile per slice.
        if (p.async_dma && p.split_k == 1 && p.tile_m == kPrefillTileM && L.groups_per_kblock == 1 && force_split <= 0 &&
            a.tile_rows == 0) {
            const int64_t big_tiles = n_wide * ((a.M + 255) / 256);
            const int64_t big_rounds = (big_tiles + n_cus - 1) / n_cus;
            const int64_t small_rounds = ((int64_t)p.tiles_x * p.tiles_y + n_cus - 1) / n_cus;
            const int big_env = env_int("OVFCC_PREFILL_BIG", -1);
            if (big_env > 0 || (big_env < 0 && big_tiles >= n_cus && big_rounds * 100 <= small_rounds * 58)) {
                p.big = true;
                p.tile_m = 256;
                p.tiles_y = (int)((a.M + 255) / 256);
                p.full_tiles = p.tiles_x * p.tiles_y;
                p.grid[0] = (unsigned)p.full_tiles;
                p.block = 256;
            }
        }
        if (p.big)
            p.name = "fcc_prefill_big_w4";
        else
        p.name = L.bits == 4 ? (p.async_dma ? "fcc_prefill_async_w4" : p.direct ? "fcc_prefill_direct_w4" : wide ? "fcc_prefill_wide_w4" : "fcc_prefill_w4")
                             : (p.direct ? "fcc_prefill_direct_w8" : wide ? "fcc_prefill_wide_w8" : "fcc_prefill_w8");
    }
    *plan = p;
    return OVFCC_OK;
}

int launch_fc(const FcDeviceArgs& a, const LaunchPlan& p, void* stream) {
    if (a.M == 0)
        return 0;
    switch (p.kernel) {
    case OVFCC_KERNEL_PLAIN:
        return launch_plain(a, p, stream);
    case OVFCC_KERNEL_DECODE:
        return p.gemv     ? launch_gemv(a, p, stream)
               : p.gemv16 ? launch_gemv16(a, p, stream)
               : p.gemv16_stream ? launch_gemv16_stream(a, p, stream)
               : p.batch  ? launch_batch(a, p, stream)
                          : launch_decode(a, p, stream);
    default:
        if (p.big)
            return launch_prefill_big(a, p, stream);
        if (p.async_dma)
            return launch_prefill_async(a, p, stream);
        if (p.direct)
            return launch_prefill_direct(a, p, stream);
        return p.tile_n == kPrefillWideN ? launch_prefill_wide(a, p, stream) : launch_prefill(a, p, stream);
    }
}

// ---- two workgroups per compute unit (kernel_prefill_pair.hip), one node --------------------------------------

// Time of a prefill launch, us: its start and end, the k-blocks that a compute unit goes through, and the sums of parts of K --
// parked, and added by the last part to arrive alone.  Fitted to calls of 4096 -> 6144 / 4096 / 28672 and 14336 -> 4096, i4 in
// groups of 64 and u4 in groups of 128, 66 to 2048 rows (off by 12 % at most): kblock_us is what a k-block of a tile that has
// a compute unit to itself takes; of tiles that share it, each takes `shared` of that.  cost: rows x 256 channels of a tile.
static double prefill_us(int64_t tiles, int64_t kb, int split, double cost, double kblock_us, double shared, int n_cus) {
    const int64_t rounds = (tiles * split + n_cus - 1) / n_cus;
    return 4.0 + (double)((kb + split - 1) / split) * kblock_us * (rounds == 1 ? 1.0 : shared * (double)rounds) +
           (split > 1 ? 1.0 + 2e-4 * (double)(tiles * split) * cost + 0.01 * split * cost : 0.0);
}

// Whether it can run a call that plan_launch gave to another of the 4-bit kernels.  (Not with one scale per channel: the others
// keep such weights exact and add the halves of two wave groups, this one sums K in one chain.)
bool pair_applies(const FcDeviceArgs& a, const LaunchPlan& p) {
    return p.kernel == OVFCC_KERNEL_PREFILL && p.async_dma && a.layout.groups > 1 && a.tile_rows == 0 && !a.want_async &&
           a.M > kDecodeMaxRows;
}

// Its best launch by prefill_us.  Tiles of 128 channels do half the unpacking per row of their k-block and take 0.6 of the time of
// tiles of 256: they win where one round of tiles covers the call, the others where the work is long (activations cross LDS half as
// often per product).  4096 -> 4096, 117 rows 18.9 / 14.4 us, 600 rows 32 / 27; 4096 -> 28672, 80 rows 33 / 27.5, but 371 rows 82 / 90.
// K is cut only to fill the chip once: beyond, parts cost more than they fill (14336 -> 4096 at 1000 rows 106 us in 256 or in 512
// workgroups of 256 channels, 4096 -> 4096 36 in 256 and 42 in 512).  That also keeps the parked sums within 32 MiB.
double plan_pair(const FcDeviceArgs& a, int n_cus, LaunchPlan* plan, double shared) {
    static const int heights[4] = {128, 96, 80, 64};
    static const double kblock_us[2][4] = {{1.66, 1.34, 1.20, 1.06}, {1.02, 0.81, 0.74, 0.62}};  // 256 channels, 128
    static const double share[2][4] = {{1.00, 1.00, 1.00, 1.00}, {1.10, 1.00, 0.98, 1.10}};
    const Layout& L = a.layout;
    LaunchPlan p = *plan;
    // four waves instead of eight apply a gated linear unit (4096 -> 28672, 220 rows 53 / 58.8 us in tiles of 256 channels); with
    // two zero-points a step the 8-wave kernel is the slower one (3200 -> 18176, 1509 rows 208 / 186)
    const double unit = L.glu ? 1.06 : 1.0, more = L.groups_per_kblock == 4 && L.zp_table ? 0.95 : 1.0;
    double best = -1.0;
    for (int h = 0; h < 8; ++h) {
        const int rows = heights[h & 3], channels = h < 4 ? kPrefillWideN : kPrefillWideN / 2;
        if (rows > 80 && channels == kPrefillWideN && L.groups_per_kblock == 4 && L.zp_table)
            continue;  // (these run alone on a compute unit)
        const int64_t nx = (a.N + channels - 1) / channels, ny = (a.M + rows - 1) / rows, tiles = nx * ny;
        const double cost = (double)rows * channels / kPrefillWideN;
        for (int want = 1; want <= 8; ++want) {
            const int64_t per = (L.k_blocks + want - 1) / want;
            const int split = (int)((L.k_blocks + per - 1) / per);
            if (split != want || (split > 1 && (per < 8 || tiles * split > n_cus)))
                continue;
            const double us = prefill_us(tiles, L.k_blocks, split, cost, (h < 4 ? unit * more : more) * kblock_us[h >> 2][h & 3], shared * share[h >> 2][h & 3], n_cus);
            if (best >= 0.0 && us >= best)
                continue;
            best = us;
            p.tile_m = rows, p.tile_n = channels, p.tiles_x = (int)nx, p.tiles_y = (int)ny;
            p.split_k = split, p.kblocks_per_split = (int)per;
            p.full_tiles = split == 1 ? (int)tiles : 0;
            p.grid[0] = (unsigned)(tiles * split), p.grid[1] = p.grid[2] = 1;
            p.workspace_bytes = split > 1 ? (size_t)tiles * split * rows * channels * sizeof(float) : 0;
            p.counter_count = split > 1 ? (size_t)tiles : 0;
        }
    }
    p.pair = true, p.big = false;
    p.block = 256;
    p.name = "fcc_prefill_async_w4";
    *plan = p;
    return best;
}

// Whether it is the faster one.
bool pair_preferred(const FcDeviceArgs& a, const LaunchPlan& p, int n_cus) {
    for (const char* name : {"OVFCC_PREFILL_DIRECT", "OVFCC_PREFILL_ASYNC", "OVFCC_PREFILL_WIDE", "OVFCC_PREFILL_BIG",
                             "OVFCC_PREFILL_TAIL", "OVFCC_PREFILL_ROWS"})
        if (env_int(name, -1) >= 0)
            return false;
    if (!pair_applies(a, p))
        return false;
    LaunchPlan pair = p;
    const int64_t tiles = (int64_t)p.tiles_x * p.tiles_y, kb = a.layout.k_blocks;
    // 256 x 256 tiles: 2.95 us a k-block and round, 3.4 with a gated linear unit; launches of that size run into the power limit,
    // where the two workgroups gain less.  4096 -> 28672 with the unit, 2048 rows 430 / 358 us, 5003 rows 991 / 888; without it
    // 4096 -> 14336, 5003 rows 465 / 434, but 8192 rows 682 / 688; 14336 -> 4096, 8192 rows 667 / 689.
    if (p.big)
        return plan_pair(a, n_cus, &pair, 0.90) < prefill_us(tiles, kb, 1, 256.0, a.layout.glu ? 3.4 : 2.95, 1.0, n_cus);
    // The 8-wave kernel, which has a compute unit to itself: ahead where its tiles fit one round (7936 -> 7936 in groups of 32, 970
    // rows 117 / 133 us; 4096 -> 4096, 914 rows 39 / 43), behind where they do not or a lower or finer cut fits better
    // (4096 -> 28672, 371 rows 109 / 80; 14336 -> 4096, 600 rows 106 / 73; 4096 -> 6144, 3000 rows 174 / 127).
    return plan_pair(a, n_cus, &pair) < prefill_us(tiles, kb, p.split_k, p.tile_m, p.tile_m == 64 ? 1.05 : 1.52, 1.0, n_cus);
}

// Slice height of a grouped prefill launch over items of these row counts: every item is cut into equal slices of
// at most that many rows and every slice is one tile.  Measured on a mixture-of-experts layer, a tile of 64 / 80 /
// 96 rows costs 0.78 / 0.84 / 0.89 of a 128-row tile (the unpack work and the data movement of a tile do not
// depend on its height), so the height that needs the fewest tiles wins unless a lower one needs no more.
// mid_ok: tiles of 80 and 96 rows exist (one group per k-block).  OVFCC_PREFILL_ROWS = 64 | 80 | 96 | 128 overrides.
int rows_cap_for(const int64_t* rows, int n, bool mid_ok) {
    static const int caps[4] = {64, 80, 96, 128}, cost[4] = {780, 836, 890, 1000};
    if (const int forced = env_int("OVFCC_PREFILL_ROWS", 0))
        return forced == 64 ? 64 : ((forced == 80 || forced == 96) && mid_ok) ? forced : kPrefillGroupRows;
    int best = kPrefillGroupRows;
    int64_t best_cost = -1;
    for (int c = 0; c < 4; ++c) {
        if (!mid_ok && (caps[c] == 80 || caps[c] == 96))
            continue;
        int64_t total = 0;
        for (int i = 0; i < n; ++i)
            total += (rows[i] + caps[c] - 1) / caps[c] * cost[c];
        if (best_cost < 0 || total < best_cost)
            best_cost = total, best = caps[c];
    }
    return best;
}

// ---- 8-bit nodes over int8 activations (kernel_prefill_i8.hip) ----------------------------------------------

void plan_prefill_i8(const FcDeviceArgs& a, int n_cus, LaunchPlan* plan) {
    LaunchPlan p;
    p.kernel = OVFCC_KERNEL_PREFILL;
    const int64_t kb = a.layout.k_blocks;
    const int64_t tiles128 = a.N / 256 * ((a.M + 127) / 128), tiles = a.N / 256 * ((a.M + 255) / 256);
    const int64_t rounds128 = (tiles128 + n_cus - 1) / n_cus, rounds = (tiles + n_cus - 1) / n_cus;
    // A round of 256 x 256 tiles over the compute units takes 1.3 times a round of 128 x 256 tiles: 16 us + 1.07 per k-block
    // against 15 + 0.81 (u8 8192 -> 57344, 1024 rows, 7 rounds or 4, 487 us / 381; 5120 -> 10240, 1076 rows, 2 / 1, 109 / 67;
    // 4096 -> 12288, 2000 rows, 3 / 2, 132 / 111).  Where 128-row tiles fit in one round they stay (4096 -> 16384, 500 rows,
    // 48.5 / 56.7) unless K is so long that half of it costs less than the 38 us that parking and adding sums takes: K in two
    // parts, 28672 -> 8192 at 1024 rows 223 / 206, 20864 -> 7936 at 835 rows 199 / 155, but 8192 -> 8192 76 / 81.
    // OVFCC_PREFILL_BIG = 0 | 1 overrides.
    const bool halves = tiles * 2 <= n_cus && kb >= 144;
    const int big_env = env_int("OVFCC_PREFILL_BIG", -1);
    if (big_env > 0 || (big_env < 0 && (rounds * 100 <= rounds128 * 75 || (rounds128 == 1 && halves)))) {
        p.big = true;
        p.tiles_x = (int)(a.N / 256), p.tiles_y = (int)((a.M + 255) / 256);
        const int64_t per = halves ? (kb + 1) / 2 : kb;
        p.split_k = halves ? 2 : 1, p.kblocks_per_split = (int)per;
        p.grid[0] = (unsigned)(tiles * p.split_k);
        p.block = 256;
        p.tile_m = 256, p.tile_n = 256;
        p.workspace_bytes = halves ? (size_t)(tiles * 2) * 256 * 256 * sizeof(int) : 0;
        p.counter_count = halves ? (size_t)tiles : 0;
    } else {
        p.tile_m = 128, p.tile_n = 256, p.block = 512;
        p.grid[0] = (unsigned)(a.N / 256), p.grid[1] = (unsigned)((a.M + 127) / 128);
    }
    *plan = p;
}

// ---- weight-streaming kernel (kernel_stream.hip) ----------------------------------------------------------

bool stream_applies(const FcDeviceArgs& a) {
    const Layout& L = a.layout;
    return L.tiled && a.M > 0 && a.M <= kDecodeMaxRows && a.M * a.K * 2 < ((int64_t)1 << 31) &&
           L.k_blocks * L.tiles_per_kblock * kTileBytes < ((int64_t)1 << 31) && L.groups * 32 < ((int64_t)1 << 31);
}

// Which calls it takes from the kernel that plan_launch chose (figures: that kernel against this one, us).
bool stream_preferred(const FcDeviceArgs& a, const LaunchPlan& p, int n_cus) {
    const Layout& L = a.layout;
    // (nodes under 256 KiB stay where they are: their launches cost the same wherever they run)
    if (p.kernel != OVFCC_KERNEL_DECODE || !stream_applies(a) || L.w_bytes < ((size_t)256 << 10))
        return false;
    // All of the small-batch kernel's: u8 8192 -> 57344 at 24 rows 110 / 83, 28672 -> 8192 71 / 44; i4 in groups of 64,
    // 4096 -> 28672 at 24 rows 28.1 / 20.4, at 48 39.1 / 26.4; i8 1024 -> 1024 at 32 rows 8.9 / 5.8.  (Over 60 drawn nodes
    // the worst are 4-bit ones of groups of 128 with a zero-point table, up to 8 rows: 11648 -> 3584 11.6 / 11.9, 7296 ->
    // 6896 12.4 / 12.7.)
    if (p.batch)
        return true;
    // The 16-row kernel with stationary activations where it streams many weights once per row tile, or cuts K of a
    // large node in two and adds the parts in a second launch: 4096 -> 28672 at 40 rows 32.6 / 26.4, 6144 -> 9216 at 24
    // rows 15.3 / 13.7, at 48 rows 22.4 / 17.1.  It stays for 4096 -> 28672 at 32 rows (19.5 / 20.6), for smaller nodes
    // (4096 -> 6144 at 48 rows 11.7 / 12.1; two parts of 8 to 17 MB at 40 rows: 7680 -> 2368 12.4 / 14.5, 7168 -> 3824 12.9 /
    // 14.5, 5632 -> 6304 14.7 / 15.5, with a few the other way: 4608 -> 6864 15.0 / 13.3) and with K in four parts.
    if (p.gemv16)
        return a.M > 16 && ((p.split_k == 2 && L.w_bytes >= ((size_t)20 << 20)) || (p.split_k == 1 && a.M > 32 && L.w_bytes >= ((size_t)32 << 20)));
    if (p.gemv || p.gemv16_stream)
        return false;
    // The streaming kernel of one channel tile per workgroup: 8-bit nodes whose K is too long for its LDS (u8 28672 ->
    // 8192 at 1 row 42.8 / 38.5, 15104 -> 4416 18.3 / 15.8), and from five rows on nodes of 10 MB and more (larger ones
    // than 16 MB are the small-batch kernel's).  There its time grows with the rows and with K, which one workgroup
    // contracts, while this kernel's is what its many parts and their sum take, 8 to 10 us: 3552 channels of 8 bits, K =
    // 4096, 6.5 / 8.5 at 5 rows, 8.4 / 8.6 at 16; 5376 -> 2256 7.4 / 8.6 at 5 rows, 8.3 / 8.6 at 10; 7936 -> 2032 9.7 / 10.2
    // at 8; 9728 -> 1584 12.6 / 9.8 at 16; i4 in groups of 128, 7808 -> 3472 8.3 / 9.5 at 5; in groups of 32, 7424 -> 2944 9.3
    // / 9.8 at 6, even at 9.  Where its workgroups need a second round and its groups cost it most (several to a k-block,
    // or 4-bit ones with a zero-point table), all move: i4 in groups of 64, 4096 -> 6144 at 8 rows 10.6 / 8.2.
    if (L.bits == 8 && !p.x_in_lds && L.w_bytes >= ((size_t)64 << 20))
        return true;
    const bool slow_rounds = L.n_tiles > n_cus && (L.groups_per_kblock != 1 || (L.bits == 4 && L.zp_table && L.groups > 1));
    return a.M > 4 && L.w_bytes >= ((size_t)10 << 20) && (slow_rounds || a.K * (a.M + 10) >= 145000);
}

constexpr int64_t kStreamMaxParts = 16;

// Parts along K (max_parts at most) for a launch of `groups` workgroups per part, and the stages of a part.
static void stream_parts(const Layout& L, int64_t groups, int64_t max_parts, int n_cus, int64_t* split_out, int64_t* per_out) {
    const int64_t stages = (L.k_blocks + 1) / 2;
    // Parts along K: as many as make the launch shortest, counted in stages -- rounds of workgroups over the compute
    // units times a part's stages and two more for its start and end.  (Two workgroups fit a compute unit, but a second
    // round costs a round all the same: 8192 -> 10240 u8 at 16 rows, 80 groups, takes 17.8 us in 3 parts, 22.5 in 4.)
    const int64_t stage_bytes = 2 * L.tiles_per_kblock * kTileBytes;
    int64_t split = 1, per = stages, best = -1;
    for (int64_t s = 1; s <= max_parts && s <= stages; ++s) {
        int64_t n = (stages + s - 1) / s;
        // a part that begins a multiple of 32 KiB into its tile makes all streams of the launch meet in the same
        // memory channels (8192 -> 8192 u8 at 16 rows: parts of 8 stages 20.5 us, of 10 15.4)
        if (s > 1 && n * stage_bytes % (32 * 1024) == 0)
            n += 2;
        const int64_t parts = (stages + n - 1) / n;
        const int64_t cost = (groups * parts + n_cus - 1) / n_cus * (n + 2);
        if (best < 0 || cost < best)
            best = cost, split = parts, per = n;
    }
    *split_out = split, *per_out = per;
}

void plan_stream(const FcDeviceArgs& a, int n_cus, LaunchPlan* plan) {
    const Layout& L = a.layout;
    LaunchPlan p;
    p.kernel = OVFCC_KERNEL_DECODE;
    p.stream = true;
    p.name = L.bits == 4 ? "fcc_stream_w4" : "fcc_stream_w8";
    const int64_t groups = (L.n_tiles + kStreamWaves - 1) / kStreamWaves;
    const int mt = (int)((a.M + 15) / 16);
    // (no more parts than the fixed scratch array holds, so that the entry point that allocates nothing runs this launch
    // too: u8 122880 -> 32896 at one row would take 16, and 33.7 MB of the array's 33.5)
    const int64_t held = (int64_t)(kStaticWorkspaceBytes / ((size_t)groups * kStreamWaves * mt * 1024));
    const int64_t max_parts =
        groups * (int64_t)sizeof(unsigned) <= (int64_t)kStaticCounterBytes ? std::min(kStreamMaxParts, held) : 1;
    int64_t split, per;
    stream_parts(L, groups, std::max<int64_t>(1, max_parts), n_cus, &split, &per);
    p.split_k = (int)split, p.kblocks_per_split = (int)(2 * per);
    p.grid[0] = (unsigned)groups, p.grid[1] = (unsigned)split;
    p.block = 64 * kStreamWaves;
    p.tile_m = 16 * mt, p.tile_n = 16 * kStreamWaves;
    p.workspace_bytes = split > 1 ? (size_t)groups * split * kStreamWaves * mt * 1024 : 0;
    p.counter_count = split > 1 ? (size_t)groups : 0;
    *plan = p;
}

bool plan_stream_routed(const FcDeviceArgs& a, int64_t pairs, int n_experts, int n_cus, LaunchPlan* plan, int* cap) {
    const Layout& L = a.layout;
    // The counts stay on the device: slices of the average bucket plus twice its square root (what random routing stays
    // under), up to 32 rows.  Expert block of eight experts, hidden size 4096, MLP width 14336, top two, against the
    // grouped prefill kernel: 1 row 79 / 57 us, 40 rows (slices of 32) 237 / 198, 80 rows 248 / 213;
    // with slices of 48 rows it loses (100 rows 244 / 277).  Sixteen experts of 2048 x 2048, top four: 1 row 46 / 27,
    // 80 rows 60 / 49.  (Nodes under 1 MiB were not measured and keep the prefill kernel.)
    const double avg = (double)pairs / n_experts;
    const int64_t likely = (int64_t)std::ceil(avg + 2.0 * std::sqrt(avg));
    const int mt = (int)((likely + 15) / 16);
    if (!L.tiled || L.bits != 4 || mt > 2 || L.w_bytes < ((size_t)1 << 20) || L.groups * 32 >= ((int64_t)1 << 31) ||
        L.k_blocks * kTileBytes >= ((int64_t)1 << 31) || a.K * 2 * 16 * mt >= ((int64_t)1 << 31))
        return false;
    const int64_t slices = std::min(pairs, (pairs + 16 * mt - 1) / (16 * mt) + n_experts);
    if (slices > 65535)
        return false;
    LaunchPlan p;
    p.kernel = OVFCC_KERNEL_DECODE;
    p.stream = true;
    p.name = "fcc_stream_grouped_w4";
    p.n_cus = n_cus;
    const int64_t groups = (L.n_tiles + kStreamWaves - 1) / kStreamWaves;
    const double reached = n_experts * (1.0 - std::pow(1.0 - 1.0 / n_experts, (double)pairs));
    int64_t split, per;
    stream_parts(L, groups * std::max<int64_t>(1, std::llround(reached)), kStreamMaxParts, n_cus, &split, &per);
    p.split_k = (int)split, p.kblocks_per_split = (int)(2 * per);
    p.grid[0] = (unsigned)groups, p.grid[1] = (unsigned)split, p.grid[2] = (unsigned)slices;
    p.block = 64 * kStreamWaves;
    p.tiles_x = (int)groups, p.tiles_y = (int)slices;
    p.tile_m = 16 * mt, p.tile_n = 16 * kStreamWaves;
    p.workspace_bytes = split > 1 ? (size_t)(slices * groups * split) * kStreamWaves * mt * 1024 : 0;
    p.counter_count = split > 1 ? (size_t)(slices * groups) : 0;
    *plan = p;
    *cap = 16 * mt;
    return true;
}

// ---- nodes with one scale per channel that fit no tile (kernel_ragged.hip) ---------------------------------

// What fcc_ragged_tile_dma_kernel assumes of its operands: rows that begin at a multiple of four bytes and hold a load's
// eight inputs, offsets into activations and into a channel tile's weights that fit the range check of a buffer load.
bool ragged_rows_at_dwords(const FcDeviceArgs& a) {
    return a.K % 2 == 0 && a.K >= 8 && (reinterpret_cast<uintptr_t>(a.x) & 3) == 0 && a.M * a.K * 2 < ((int64_t)1 << 31) &&
           a.layout.k_blocks * 8 * kTileBytes < ((int64_t)1 << 31);
}

void plan_ragged(const FcDeviceArgs& a, int n_cus, LaunchPlan* plan) {
    LaunchPlan p;
    p.kernel = OVFCC_KERNEL_PLAIN;
    const bool four = a.layout.bits == 4;
    const int64_t kb = a.layout.k_blocks;
    // The rows kernel up to 16 rows, and up to the row count at which its workgroups (32 rows each) still fit the chip
    // in one round: N = 1000, K = 1160 at 128 rows (252 workgroups) 6.0 us against 8.8 for the tile kernel, at 192 rows
    // (378) 10.3 against 8.8; N = 2000 at 64 rows 5.8 against 8.7, at 96 rows 10.1 against 8.9; N = 4300 at 32 rows (269)
    // 10.0 against 8.9.
    // Row tiles of 16 as long as they fit in one round: each wave has half of the rows to stage.
    const int mt = a.M <= 16 || (a.N + 15) / 16 * ((a.M + 15) / 16) <= n_cus ? 1 : 2;
    if (a.M <= 16 || (a.N + 15) / 16 * ((a.M + 31) / 32) <= n_cus) {
        const int64_t waves = kb < 16 ? kb : 16;
        p.grid[0] = (unsigned)((a.N + 15) / 16), p.grid[1] = (unsigned)((a.M + 16 * mt - 1) / (16 * mt));
        p.block = (unsigned)(64 * waves);
        p.tile_m = 16 * mt, p.tile_n = 16;
        p.name = four ? "fcc_ragged_rows_w4" : "fcc_ragged_rows_w8";
        p.dynamic_lds = (unsigned)(waves * ragged_wave_lds(mt));
    } else {
        p.tiles_x = (int)((a.N + kRaggedTile - 1) / kRaggedTile), p.tiles_y = (int)((a.M + kRaggedTile - 1) / kRaggedTile);
        // three workgroups fit a compute unit: K is split until the launch has about that many, four k-blocks at least
        // to each (1160 -> 1160 at 577 rows, 190 tiles, two parts)
        const int64_t tiles = (int64_t)p.tiles_x * p.tiles_y;
        int64_t split = 1;
        while (split < 8 && tiles * split * 2 <= 3 * (int64_t)n_cus && kb / (split * 2) >= 4)
            split *= 2;
        const int64_t per = (kb + split - 1) / split;
        split = (kb + per - 1) / per;
        p.split_k = (int)split, p.kblocks_per_split = (int)per;
        p.grid[0] = (unsigned)((tiles + 7) / 8 * 8 * split);
        p.block = 256;
        p.tile_m = kRaggedTile, p.tile_n = kRaggedTile;
        // Activations straight to LDS where rows start at dwords (and offsets fit 32 bits) and some compute units get three
        // workgroups.  Up to two, where a workgroup's own latency counts, the kernel that holds its scales and bias from the
        // start is ahead (577 x 1160 -> 1160, 384 workgroups, 11.2 us against 11.8; 256 x 1160 -> 3480, 448, 11.6 / 12.2).
        p.to_lds = ragged_rows_at_dwords(a) && tiles * split > 2 * (int64_t)n_cus;
        p.name = four ? "fcc_ragged_tile_w4" : "fcc_ragged_tile_w8";
        p.workspace_bytes = split > 1 ? (size_t)tiles * split * kRaggedTile * kRaggedTile * sizeof(float) : 0;
        p.counter_count = split > 1 ? (size_t)tiles : 0;
    }
    *plan = p;
}

}  // namespace ovfcc
