// MFMA GEMM for a short K (up to 256 bytes: 128 of a 16-bit type) and a C far larger than the operands: the scores of an
// attention head (32 x (2048x2048x128)), outer-product-like layers.
//
// Such a problem is a stream of C into memory with a little arithmetic in front of it.  A kernel of one tile per workgroup
// spends most of a tile's time where nothing is written -- on its start, on the trip of its operands, on its MFMAs -- and writes
// in a burst at the end.  Here a workgroup keeps its rows of A, the whole K of them, in registers as MFMA fragments and walks along
// a run of column tiles, and two of them share a CU (80 KB of LDS each), so that one multiplies while the other writes back; the next
// tile of B is fetched behind the write-back.
//
// Tiles of 64 x 256: what bounds the kernel is the rate at which memory takes C, and that follows the shape of the pieces (a kernel
// that only stores 256 MB in rows 4 KB apart: 46 us in tiles of 32 rows x 512 bytes and flatter, 50 in 64 x 512, 56 in 128 x 256; the
// copy engine's order, row after row, 40).  32 x (2048x2048x128) fp16 x 0.125, 268 MB of C, us: 256 x 256 tiles of the four-wave kernel 85 to 87,
// this loop on 128 x 128 tiles 72, on 64 x 256 56 (4.8 TB/s); K = 64 67 / 50.  Without MFMAs or without fills it is as slow to 10 %.  The slab is worth its
// LDS traffic: stores straight from the registers, 16 rows x 64 bytes, take 71.
//
// Same role as the reference's tensorized plan with its A fragments cached (MMA_FRAGMENT cache,
// /root/reference/accera/transforms/src/exec/ExecutionPlanToAffineLoweringPass.cpp:2705-2726).
// Staging, swizzles and fragment reads are those of gemm_mfma.h / gemm_mfma16.h (16x16 instruction shapes, operands swapped: a
// lane holds one row and four neighbouring columns of a block).
#pragma once
#include "gemm_mfma16.h"

namespace acc950 {

// STEPS: k-steps of 64 bytes (1 to 4).  OS: bytes of an element of C.  CONSTANT: floats, a SET constant other than 0.
template <int IN_, bool A_KC_, bool B_KC_, int STEPS_, int OS_, bool CONSTANT_>
struct ShortKConfig {
    static constexpr bool CONSTANT = CONSTANT_;
    static constexpr int IN = IN_, STEPS = STEPS_, OS = OS_, BM = 64, BN = 256, NT = 256;
    static constexpr bool A_KC = A_KC_, B_KC = B_KC_;
    static constexpr int KB = STEPS_ % 2 == 0 ? 128 : 64; // bytes of K of one staged sub-tile
    static constexpr int SUBS = STEPS_ * 64 / KB;
    static constexpr int PANEL_BYTES = BN * STEPS_ * 64; // a tile of B (and A's rows, once)
    static constexpr int SLAB_BYTES = 4096;              // per wave: 16 rows of 64 columns
    static constexpr int LDS_BYTES = PANEL_BYTES + 4 * SLAB_BYTES;
    static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups to a CU");
};

template <typename Cfg>
__global__ void __launch_bounds__(256, 2) gemm_short_k_kernel(ACC950_HEAD_PARAMS, int run_tiles, GemmArgs p)
{
    constexpr int IN = Cfg::IN, STEPS = Cfg::STEPS, OS = Cfg::OS, BM = Cfg::BM, BN = Cfg::BN, NT = Cfg::NT, KB = Cfg::KB, SUBS = Cfg::SUBS;
    constexpr bool A_KC = Cfg::A_KC, B_KC = Cfg::B_KC;
    constexpr int ES = InTraits<IN>::ES, BK = KB / ES, VEC = 16 / ES;
    constexpr int TM = BM / 16, TN = BN / 4 / 16; // 64 x 64 per wave, the four side by side
    constexpr int VPL = 16 / OS; // elements of C per store and lane
    // (LDS layout and fragment reads only: with as many threads a fill instruction covers a whole period of the swizzle, which the tile's own
    // fills rely on and the ones below do not)
    using TA = OperandTile<IN, BM, A_KC, 512, KB, true>;
    using TB = OperandTile<IN, BN, B_KC, 512, KB, true>;
    using acc_t = typename In16Traits<IN>::acc_t;
    using scalar_t = typename In16Traits<IN>::scalar_t;

    extern __shared__ __attribute__((aligned(1024))) char smem[];
    ACC950_TAKE_HEAD_TILES(p, BM, BN);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wc0 = wave * (TN * 16);

    // Workgroup -> (problem of the batch, row of tiles, run of column tiles).  Ids equal modulo 8 share an XCD: each XCD takes a
    // consecutive range of (problem, run, row of tiles), rows fastest, so that what runs on it together reads the same tiles of B.
    const int runs = (p.tiles_n + run_tiles - 1) / run_tiles;
    int id = blockIdx.x;
    {
        const int total = (int)gridDim.x, per = total / 8, rest = total % 8, x = id % 8, y = id / 8;
        id = x * per + (x < rest ? x : rest) + y;
    }
    const int per_problem = p.tiles_m * runs;
    const int z = id / per_problem, in_problem = id % per_problem;
    const int tile_m = in_problem % p.tiles_m, m0 = tile_m * BM;
    const int t0 = (in_problem / p.tiles_m) * run_tiles;
    const int len = p.tiles_n - t0 < run_tiles ? p.tiles_n - t0 : run_tiles;
    if (z) {
        p.A = (const char*)p.A + (int64_t)z * p.a_bs * ES;
        p.B = (const char*)p.B + (int64_t)z * p.b_bs * ES;
        p.C = (char*)p.C + (int64_t)z * p.c_bs * OS;
    }
    const int64_t lda = A_KC ? p.a_rs : p.a_cs, ldb = B_KC ? p.b_cs : p.b_rs;
    const unsigned smem_addr = (unsigned)(size_t)(ACC950_LDS char*)smem;
    const unsigned wave_lds = __builtin_amdgcn_readfirstlane((unsigned)(wave * 1024));
    // Workgroups one above the other start at different tiles of their run: with rows of C a multiple of 4 KB apart they would all
    // write to the same part of the memory channels at a time.
    int at = tile_m % len;

    // All K of a tile of an operand into LDS at `to`.  Rows (chunks of a row, where the tile's rows run along M / N) past the end
    // are fetched from the last one: what comes of them is never stored.
    auto fill = [&](auto tile_tag, const char* base, int r0, int rmax, int64_t ld, unsigned to) __attribute__((always_inline)) {
        using T = decltype(tile_tag);
        constexpr bool KC = std::is_same<T, TA>::value ? A_KC : B_KC;
        static_assert(T::CHUNKS % NT == 0 && NT % T::CPR == 0);
        const int left = rmax - r0;
        int id_f = tid; // (an opaque copy: the lanes' offsets are worked out for every tile, not kept in registers beside the sums)
        asm volatile("" : "+v"(id_f));
#pragma unroll
        for (int u = 0; u < SUBS; ++u)
#pragma unroll
            for (int f = 0; f < T::CHUNKS / NT; ++f) {
                const int row = f * (NT / T::CPR) + id_f / T::CPR, c = T::swizzle(row, id_f % T::CPR);
                unsigned off;
                if constexpr (KC) off = (unsigned)((row < left ? row : left - 1) * (int)ld * ES) + c * 16;
                else off = (unsigned)(row * (int)ld * ES) + (c * VEC < left ? c * VEC : left - VEC) * ES;
                const char* tile = base + (KC ? ((int64_t)r0 * ld + u * BK) * ES : ((int64_t)u * BK * ld + r0) * ES);
                T::direct_issue_uniform(to + u * T::TILE_BYTES + wave_lds + f * NT * 16, off, tile);
            }
    };
    auto barrier = []() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // ---- A's rows go through B's buffer into registers
    fill(TA{}, (const char*)p.A, m0, p.M, lda, smem_addr);
    wait_vmcnt<0>();
    barrier();
    i32x4 af[STEPS][TM];
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
            af[s][i] = TA::read_frag16(smem + (s * 64 / KB) * TA::TILE_BYTES, i * 16, s % (KB / 64), lane);
    barrier();
    fill(TB{}, (const char*)p.B, (t0 + at) * BN, p.N, ldb, smem_addr);

    const unsigned row_bytes = (unsigned)p.c_rs * OS;
    // Descriptor of the workgroup's rows of C: an offset past it is dropped.
    const int rows = p.M - m0 < BM ? p.M - m0 : BM;
    const auto c_rsrc = __builtin_amdgcn_make_buffer_rsrc((char*)p.C + (int64_t)m0 * p.c_rs * OS, 0, (int)((unsigned)(rows - 1) * row_bytes + (unsigned)p.N * OS), 0x00020000);
    const bool whole_lines = !c_part_lines(p.C, p.c_rs, OS);
    constexpr unsigned kOutside = 0x80000000u; // (C's rows of a tile span less than 2 GiB)
    // The SET constant: integers start from it; floats add it once to the whole sum, as the other kernels do (a constant far above the products would
    // round every step of the sum at its own size: 100, K = 96, fp32 result, 3.8e-8 from float64 where one addition is 2.2e-8).  In kernels of their own:
    // a test for it beside those for the ops cost a ReLU without one up to 7 % (us, with / without: fp16 32 x (2048x2048x128) 62.6 / 58.6, 18 x (752x2624x96) 19.4 / 18.0, bf16
    // 20 x (272x4096x128) 14.0 / 13.5; 0.5 % over 42 problems).
    const scalar_t set_value = (scalar_t)p.prologue_arg, start = IN == IN_I8 ? set_value : scalar_t(0);
    const scalar_t epi_arg = (scalar_t)p.epilogue_arg;

    for (int n = 0; n < len; ++n) {
        const int t = t0 + at;
        at = at + 1 < len ? at + 1 : 0;
        // This tile's fills are older than the stores of the tile before, which may still be on their way (memory operations complete
        // in the order issued, and every lane issues every store, outside or not).
        if (n > 0) wait_vmcnt<TM * TN * 4 / VPL>();
        else wait_vmcnt<0>();
        barrier();

        acc_t acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{start, start, start, start};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            i32x4 bf[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[j] = TB::read_frag16(smem + (s * 64 / KB) * TB::TILE_BYTES, wc0 + j * 16, s % (KB / 64), lane);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) mfma16<IN>(bf[j], af[s][i], acc[i][j]);
        }

        barrier(); // every wave has its fragments
        if (n + 1 < len) fill(TB{}, (const char*)p.B, (t0 + at) * BN, p.N, ldb, smem_addr);
        auto each = [&](auto&& fn) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = fn(acc[i][j][e]);
        };
        if constexpr (Cfg::CONSTANT) each([&](scalar_t v) { return v + set_value; });
        if (p.epilogue == EPI_RELU) each([](scalar_t v) { return v > scalar_t(0) ? v : scalar_t(0); });
        else if (p.epilogue == EPI_SCALE) each([&](scalar_t v) { return wrap_mul(v, epi_arg); });

        // ---- write-back: 16 rows of the wave's columns at a time through its slab, out of which they come as 16-byte pieces of whole rows
        int lane_w = lane, wave_w = wave;
        asm volatile("" : "+v"(lane_w), "+v"(wave_w)); // (as in fill: offsets are not kept across the loop)
        const int li = lane_w & 15, kg = lane_w >> 4, n0 = t * BN + wave_w * (TN * 16);
        char* slab = smem + Cfg::PANEL_BYTES + wave_w * Cfg::SLAB_BYTES;
        auto store_as = [&](auto aux_tag, auto&& pack) __attribute__((always_inline)) {
            constexpr int AUX = decltype(aux_tag)::value;
            constexpr int CPR = TN * 16 * OS / 16; // pieces of a row: 16, 8, 4
            // (spread over the banks by the row: a row of 256 bytes, two of 128 or four of 64 are all banks)
            auto place = [](int row, int c) { return row * (CPR * 16) + (c ^ (CPR == 16 ? row : CPR == 8 ? (row >> 1) & 7 : (row >> 2) & 3)) * 16; };
#pragma unroll
            for (int i = 0; i < TM; ++i) {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const auto w = pack(acc[i][j]);
                    const int byte = j * 16 * OS + kg * 4 * OS; // of the row
                    *(std::remove_const_t<decltype(w)>*)(slab + place(li, byte / 16) + byte % 16) = w;
                }
#pragma unroll
                for (int q = 0; q < 16 * CPR / 64; ++q) {
                    const int piece = q * 64 + lane_w, r = piece / CPR, c = piece % CPR, col = n0 + c * VPL;
                    const i32x4 v = *(const i32x4*)(slab + place(r, c));
                    const unsigned off = (unsigned)(i * 16 + r) * row_bytes + (unsigned)col * OS;
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), c_rsrc, col < p.N ? off : kOutside, 0, AUX);
                }
            }
        };
        // (nt: 32 x (2048x2048x128) 56 us, 68 without; but where rows of C end inside a line, two workgroups write parts of it and the L2 has to
        // put them together: 16 x (2048x2056x128) 78 us with nt, 51 without)
        auto store = [&](auto&& pack) __attribute__((always_inline)) {
            if (whole_lines) store_as(std::integral_constant<int, 2>{}, pack);
            else store_as(std::integral_constant<int, 0>{}, pack);
        };
        auto pack_f16 = [](const acc_t& v) {
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            return __builtin_bit_cast(i32x2, h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]});
        };
        auto pack_bf16 = [](const acc_t& v) {
            typedef __bf16 b4 __attribute__((ext_vector_type(4)));
            return __builtin_bit_cast(i32x2, b4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]});
        };
        auto pack_i16 = [](const acc_t& v) {
            return i32x2{(int)(((unsigned)v[0] & 0xffffu) | ((unsigned)v[1] << 16)), (int)(((unsigned)v[2] & 0xffffu) | ((unsigned)v[3] << 16))};
        };
        auto pack_i8 = [](const acc_t& v) {
            return (int)(((unsigned)v[0] & 0xffu) | (((unsigned)v[1] & 0xffu) << 8) | (((unsigned)v[2] & 0xffu) << 16) | ((unsigned)v[3] << 24));
        };
        if constexpr (OS == 4) store([](const acc_t& v) { return __builtin_bit_cast(i32x4, v); });
        else if constexpr (IN == IN_I8 && OS == 2) store(pack_i16);
        else if constexpr (IN == IN_I8) store(pack_i8);
        else if (p.out_type == T_F16) store(pack_f16);
        else store(pack_bf16);
    }
}

// Column tiles a workgroup walks: the fewest tile times of the rounds of workgroups (two to a CU) there are, a workgroup's start
// counted as one and a fifth.
inline int short_k_run(int64_t tiles_m, int64_t tiles_n, int64_t batch)
{
    int best = 1;
    double best_cost = 0;
    for (int run = 1; run <= tiles_n; ++run) {
        const int64_t wgs = batch * tiles_m * ((tiles_n + run - 1) / run);
        const double cost = (double)((wgs + 2 * kComputeUnits - 1) / (2 * kComputeUnits)) * (run + 1.2);
        if (run == 1 || cost < best_cost) { best = run; best_cost = cost; }
        if (wgs <= 2 * kComputeUnits && run > 1 && cost > 2 * best_cost) break;
    }
    return best;
}

template <int IN, bool A_KC, bool B_KC, int STEPS, int OS, bool CONSTANT = false>
hipError_t launch_short_k_steps(const GemmArgs& args, int run, unsigned grid, hipStream_t stream)
{
    if constexpr (IN != IN_I8 && !CONSTANT)
        if (args.prologue_arg != 0.f) return launch_short_k_steps<IN, A_KC, B_KC, STEPS, OS, true>(args, run, grid, stream);
    using Cfg = ShortKConfig<IN, A_KC, B_KC, STEPS, OS, CONSTANT>;
    auto kern = gemm_short_k_kernel<Cfg>;
    static LdsLimitOnce lds_limit; // per instantiation
    if (hipError_t e = lds_limit.ensure((const void*)kern, Cfg::LDS_BYTES); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(Cfg::NT), Cfg::LDS_BYTES, stream, ACC950_HEAD_OF(args), run, args);
    return hipGetLastError();
}

template <int IN, bool A_KC, bool B_KC>
hipError_t launch_short_k_layout(const GemmArgs& a, hipStream_t stream, LaunchGeom* geom, bool dry_run)
{
    constexpr int ES = InTraits<IN>::ES;
    const int steps = a.K * ES / 64;
    if (a.K * ES % 64 || steps < 1 || steps > 4 || a.prologue != PRO_SET || (a.epilogue != EPI_NONE && a.epilogue != EPI_RELU && a.epilogue != EPI_SCALE)) return hipErrorInvalidValue;
    GemmArgs args = a;
    args.tiles_m = (a.M + 63) / 64;
    args.tiles_n = (a.N + 255) / 256;
    const int64_t batch = a.batch > 1 ? a.batch : 1;
    const int run = short_k_run(args.tiles_m, args.tiles_n, batch);
    const int64_t grid = batch * args.tiles_m * ((args.tiles_n + run - 1) / run);
    if (grid > 0x7fffffffll) return hipErrorInvalidValue;
    if (geom) {
        geom->grid[0] = (unsigned)grid;
        geom->grid[1] = geom->grid[2] = 1;
        geom->block[0] = 256;
        geom->block[1] = geom->block[2] = 1;
        geom->dyn_lds = 256 * steps * 64 + 4 * 4096;
    }
    if (dry_run) return hipSuccess;
    const auto with_os = [&](auto steps_tag) {
        constexpr int S = decltype(steps_tag)::value;
        if (a.out_type == T_F32 || a.out_type == T_I32) return launch_short_k_steps<IN, A_KC, B_KC, S, 4>(args, run, (unsigned)grid, stream);
        if constexpr (IN == IN_I8)
            if (a.out_type == T_I8) return launch_short_k_steps<IN, A_KC, B_KC, S, 1>(args, run, (unsigned)grid, stream);
        return launch_short_k_steps<IN, A_KC, B_KC, S, 2>(args, run, (unsigned)grid, stream);
    };
    switch (steps) {
    case 1: return with_os(std::integral_constant<int, 1>{});
    case 2: return with_os(std::integral_constant<int, 2>{});
    case 3: return with_os(std::integral_constant<int, 3>{});
    default: return with_os(std::integral_constant<int, 4>{});
    }
}

} // namespace acc950
