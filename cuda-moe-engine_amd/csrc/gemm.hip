// Host side of the grouped GEMMs: which kernel of gemm_ring.h a launch takes, and its grid.
#include <atomic>

#include "gemm_ring.h"

namespace moe {

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
// Upper bound on the persistent GEMM's workgroups (0: one per CU), process-wide.
static std::atomic<int> g_gemm_workgroup_limit{0};

void set_gemm_workgroup_limit(int workgroups) {
    g_gemm_workgroup_limit.store(workgroups, std::memory_order_relaxed);
}

// Compute units of the current device, cached per device id.
static int device_cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cached[dev] == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        cached[dev] = cus;
    }
    return cached[dev];
}

// f(integral_constant<bool, GATHER>, integral_constant<bool, TAIL>) for these
// parameters (gathered rows come with K a multiple of 64, the ABI's check).
template <bool SWIGLU, typename F>
static void with_source(const GemmParams& p, F&& f) {
    if constexpr (SWIGLU) {
        if (p.a_rows != nullptr) return f(std::true_type{}, std::false_type{});
    }
    if (p.k % kStageK == 0)
        f(std::false_type{}, std::false_type{});
    else
        f(std::false_type{}, std::true_type{});
}

template <bool SWIGLU>
static int launch_gemm_t(GemmParams p, int64_t rows, hipStream_t stream) {
    constexpr int64_t kRows = 256, kCols = SWIGLU ? 128 : 256;  // the wide tiles' output
    if (p.a_rows != nullptr && p.k % kStageK != 0)
        return fail(MOE_ERR_UNSUPPORTED, "gathered A rows need K a multiple of 64");
    p.n_tiles = static_cast<int>((p.n_out + kCols - 1) / kCols);
    // Upper bound on row tiles: sum_e ceil(span_e/256) <= ceil(R/256) + E.
    const int64_t m_bound = (rows + kRows - 1) / kRows + p.experts;
    const int64_t blocks = m_bound * p.n_tiles;
    if (blocks == 0) return MOE_OK;
    // Narrow tiles for weight streaming: at most 128 rows in all, or at most 128
    // per expert on average when the wide tiles (rows spread evenly over the
    // experts) would not give every CU one. Measured at C1 (E=8, ~32 rows each):
    // gate/up 9.4 -> 7.2 us, down 11.6 -> 7.4 us; at C3 T=256 the gate/up GEMM's
    // 256 wide tiles streamed faster than narrow ones (22.9 vs 24.9 us).
    const int64_t per_expert = (rows + p.experts - 1) / p.experts;
    const int64_t wide_tiles = static_cast<int64_t>(p.experts) * ((per_expert + kRows - 1) / kRows) * p.n_tiles;
    const bool narrow = rows <= 128 || (rows <= 128 * static_cast<int64_t>(p.experts) &&
                                        wide_tiles < device_cu_count());
    if (narrow) {
        const int max_rows = rows <= 64 ? 64 : 128;
        // The narrowest tiles; the kernel may take wider ones (fewer).
        const int cols = max_rows == 64 ? narrow_cols<SWIGLU, 64>() : narrow_cols<SWIGLU, 128>();
        p.n_tiles = static_cast<int>((p.n_out + cols - 1) / cols);
        // Upper bound on row tiles: sum_e ceil(span_e/max_rows) <= ceil(R/max_rows) + E.
        const int64_t tiles = ((rows + max_rows - 1) / max_rows + p.experts) * p.n_tiles;
        if (tiles > INT32_MAX) return fail(MOE_ERR_CAPACITY, "grouped GEMM grid too large");
        // As many workgroups as fit the CUs' LDS, at most one per tile.
        const uint32_t lds = rows <= 64 ? decode_lds_bytes<SWIGLU, 64>() : decode_lds_bytes<SWIGLU, 128>();
        int64_t grid = static_cast<int64_t>(device_cu_count()) * (kRingBytes / lds);
        if (tiles < grid) grid = tiles;
        with_source<SWIGLU>(p, [&](auto gather_c, auto tail_c) {
            launch_ring<SWIGLU, decltype(gather_c)::value, decltype(tail_c)::value>(
                p, max_rows == 64 ? RingKernel::kStream64 : RingKernel::kStream128, static_cast<unsigned>(grid), stream);
        });
        return check_launch("grouped_gemm_decode_kernel");
    }
    // One workgroup per CU (the ring fills a CU's LDS), each walking the
    // virtual workgroups of the device-side plan, whose XCD ranges need a
    // multiple of 8 workgroups. Row offsets fit 32 bits (checked by the ABI).
    if (blocks > INT32_MAX) return fail(MOE_ERR_CAPACITY, "grouped GEMM grid too large");
    int64_t grid = device_cu_count();
    const int limit = g_gemm_workgroup_limit.load(std::memory_order_relaxed);
    if (limit > 0 && limit < grid) grid = limit;
    // Gate/up tiles split into pieces only where the estimated tiles (rows spread
    // evenly) leave a last round at most half full in the first four, or where so
    // few rows per expert leave it open how many experts hold any. The instance
    // that splits is 390 KB of code instead of 220, and a launch that fetches it
    // cold takes 2-3 us longer: forwards at H=1024, I=2048, 16 experts, 8192 rows
    // 153 -> 156 us with it, at H=2048, I=1408, 64 experts, 288 rows 219.7 ->
    // 221.4; against 603 -> 550 (with the down GEMM's widths) at H=4096, I=14336, 8
    // experts, 666 rows, whose 896 tiles fill three and a half rounds. (`rows` is the
    // buffer's padded capacity: E=64, top-6 counts as few rows up to 47 tokens at
    // alignment 8 and never from 16 on, where one token takes 17.4 us against 15.3.)
    bool pieces = !SWIGLU;
    if constexpr (SWIGLU) {
        const int64_t cus = device_cu_count(), last = wide_tiles % cus;
        pieces = per_expert < 12 || (last > 0 && 2 * last <= cus && wide_tiles < 4 * cus);
    }
    // At most one workgroup per unit of work: tiles, or the halves and quarters
    // the plan may split them into.
    const int64_t units = pieces ? 4 * blocks : blocks;
    if (units < grid) grid = units;
    grid = grid / kNumXcd * kNumXcd;
    if (grid < kNumXcd) grid = kNumXcd;
    with_source<SWIGLU>(p, [&](auto gather_c, auto tail_c) {
        constexpr bool G = decltype(gather_c)::value, T = decltype(tail_c)::value;
        if constexpr (SWIGLU) {
            if (pieces) return launch_pieces<G, T>(p, static_cast<unsigned>(grid), stream);
        }
        launch_ring<SWIGLU, G, T>(p, RingKernel::kPersistent, static_cast<unsigned>(grid), stream);
    });
    return check_launch("grouped_gemm_persistent_kernel");
}

int launch_grouped_gemm(const uint16_t* a, const uint16_t* b, int64_t ldb, uint16_t* c, const int32_t* offsets,
                        int64_t rows, int64_t n, int64_t k, int experts, hipStream_t stream) {
    GemmParams p{};
    p.rows = rows;
    p.a = a;
    p.b = b;
    p.c = c;
    p.offsets = offsets;
    p.k = k;
    p.ldb = ldb;
    p.nb = n;
    p.n_out = n;
    p.ldc = n;
    p.experts = experts;
    return launch_gemm_t<false>(p, rows, stream);
}

int launch_gateup_swiglu(const uint16_t* a, const uint16_t* gate_up, int64_t ldb, uint16_t* act,
                         const int32_t* offsets, int64_t rows, int64_t hidden,
                         int64_t intermediate, int experts, hipStream_t stream) {
    GemmParams p{};
    p.rows = rows;
    p.a = a;
    p.b = gate_up;
    p.c = act;
    p.offsets = offsets;
    p.k = hidden;
    p.ldb = ldb;
    p.nb = 2 * intermediate;
    p.n_out = intermediate;
    p.ldc = intermediate;
    p.experts = experts;
    return launch_gemm_t<true>(p, rows, stream);
}

// launch_gateup_swiglu with A row r read from row a_rows[r] of x (zero when
// negative): the dispatch's row table instead of its packed copy. Needs the
// ring kernels (hidden a multiple of 64; the ABI checks it).
int launch_gateup_swiglu_gathered(const uint16_t* x, const int32_t* a_rows, int64_t x_rows, const uint16_t* gate_up,
                                  int64_t ldb, uint16_t* act, const int32_t* offsets, int64_t rows, int64_t hidden,
                                  int64_t intermediate, int experts, hipStream_t stream) {
    GemmParams p{};
    p.rows = rows;
    p.a = x;
    p.a_rows = a_rows;
    p.a_src_rows = x_rows;
    p.b = gate_up;
    p.c = act;
    p.offsets = offsets;
    p.k = hidden;
    p.ldb = ldb;
    p.nb = 2 * intermediate;
    p.n_out = intermediate;
    p.ldc = intermediate;
    p.experts = experts;
    return launch_gemm_t<true>(p, rows, stream);
}

}  // namespace moe
