// Second step of a K split of the MFMA kernels: C = epilogue(prologue(C) + slice 0 + slice 1 + ...).
//
// The first step is the GEMM kernel itself, launched as a batch of `splits` partial products over consecutive ranges of
// K (blockIdx.z picks the range) that writes 32-bit sums into a workspace, slice after slice, each an M x N row-major
// matrix.  This kernel adds the slices of every element in slice order -- a fixed order, so the result does not depend
// on which workgroup finished first -- and then does what the GEMM kernel's write-back does for an unsplit problem: the
// prologue op on the old C, the epilogue op (the fused ReLU comes after the whole sum), the narrowing store.
//
// The reference has no counterpart (its `k_split` is the K depth of the block tile); shapes of its sweep lists with a
// small output and a long K (/root/reference/tools/benchmarkers/gemm_bert_assorted.csv: 768 x 320 x 30522,
// gemm_resnet_inception.csv: 288 x 64 x 21609) are the ones that leave most compute units idle without it.
#include "common.h"
#include "variants.h"

namespace acc950 {

struct SplitReduceArgs {
    const void* ws;       // [splits][M][N] float or int
    int splits, M, N;
    void* C;
    int64_t c_rs, c_cs;
    int out_type, is_int;
    int prologue, epilogue;
    float prologue_arg, epilogue_arg;
};

// One thread per four consecutive columns of a row.  Every slice's piece is one 16-byte load at whatever dword it starts (the
// hardware takes it); past the end of a row it brings the start of the next, past the last row up to three elements behind the
// slices, which the workspace has room for; those are added up and not stored.
// (Pieces that are not 16 bytes aligned were up to four loads behind a test each, slice after slice: 16x382x7997 bf16 in 31 slices, C read, 31 -> 12.5 us; 456x115x6256 22 -> 13; 128x153x1088 12.7 -> 9.)
// (ws, C, splits, M, N, c_rs, c_cs come as arguments of their own as well: the first 14 dwords of a kernel's arguments are
// preloaded into scalar registers at dispatch, and the loads of the slices need nothing else)
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const void* head_ws, void* head_C, int head_splits, int head_M, int head_N,
                                                            int64_t head_c_rs, int64_t head_c_cs, SplitReduceArgs p)
{
    p.ws = head_ws; p.C = head_C; p.splits = head_splits; p.M = head_M; p.N = head_N; p.c_rs = head_c_rs; p.c_cs = head_c_cs;
    const int groups_n = (p.N + 3) / 4;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (int64_t)p.M * groups_n) return;
    const int row = (int)(id / groups_n), col0 = (int)(id % groups_n) * 4;
    const int64_t slice = (int64_t)p.M * p.N;
    const int cols = p.N - col0 < 4 ? p.N - col0 : 4;
    // Old C, where it is read: asked for before the slices (the columns past the last are the last once more).
    const bool reads_c = p.prologue != PRO_SET;
    int64_t idx[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) idx[e] = (int64_t)row * p.c_rs + (int64_t)(e < cols ? col0 + e : p.N - 1) * p.c_cs;
    // The loads of eight slices are issued together (one trip through memory per batch instead of one per slice); the adds
    // stay in slice order.
    auto add_slices = [&](auto zero, auto&& add) {
        using T = decltype(zero);
        typedef T T4 __attribute__((ext_vector_type(4)));
        typedef T4 __attribute__((aligned(4))) T4_dword;
        T4 sum = {zero, zero, zero, zero};
        const T* w = (const T*)p.ws + (int64_t)row * p.N + col0;
        for (int s0 = 0; s0 < p.splits; s0 += 8) {
            T4 x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < p.splits) x[u] = *(const T4_dword*)(w + (int64_t)(s0 + u) * slice);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < p.splits)
                    for (int e = 0; e < 4; ++e) sum[e] = add(sum[e], x[u][e]);
        }
        return sum;
    };
    // Four finished outputs that lie side by side, aligned, leave as one store.
    const int os = p.out_type == T_I8 ? 1 : (p.out_type == T_F32 || p.out_type == T_I32) ? 4 : 2;
    const bool vec_out = cols == 4 && p.c_cs == 1 && (((size_t)p.C + (size_t)idx[0] * os) & (size_t)(4 * os - 1)) == 0;
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    if (p.is_int) {
        int old[4] = {0, 0, 0, 0};
        if (reads_c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) old[e] = load_out_int(p.C, p.out_type, idx[e]);
        }
        const auto sum = add_slices(0, [](int a, int b) { return wrap_add(a, b); });
        int r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = apply_epilogue<int>(apply_prologue<int>(sum[e], p.prologue, p.prologue_arg, [&]() { return old[e]; }), p.epilogue, p.epilogue_arg);
        if (vec_out) {
            if (p.out_type == T_I32) *(i32x4*)((int*)p.C + idx[0]) = i32x4{r[0], r[1], r[2], r[3]};
            else if (p.out_type == T_I16)
                *(u32x2*)((int16_t*)p.C + idx[0]) = u32x2{((unsigned)r[0] & 0xffffu) | ((unsigned)r[1] << 16), ((unsigned)r[2] & 0xffffu) | ((unsigned)r[3] << 16)};
            else
                *(unsigned*)((int8_t*)p.C + idx[0]) = ((unsigned)r[0] & 0xffu) | (((unsigned)r[1] & 0xffu) << 8) | (((unsigned)r[2] & 0xffu) << 16) | ((unsigned)r[3] << 24);
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < cols) store_out_int(p.C, p.out_type, idx[e], r[e]);
    } else {
        float old[4] = {0.f, 0.f, 0.f, 0.f};
        if (reads_c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) old[e] = load_out(p.C, p.out_type, idx[e]);
        }
        const auto sum = add_slices(0.f, [](float a, float b) { return a + b; });
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = apply_epilogue<float>(apply_prologue<float>(sum[e], p.prologue, p.prologue_arg, [&]() { return old[e]; }), p.epilogue, p.epilogue_arg);
        if (vec_out) {
            if (p.out_type == T_F32) *(f32x4*)((float*)p.C + idx[0]) = f32x4{r[0], r[1], r[2], r[3]};
            else if (p.out_type == T_F16)
                *(u32x2*)((uint16_t*)p.C + idx[0]) = u32x2{(unsigned)float_to_f16_bits(r[0]) | ((unsigned)float_to_f16_bits(r[1]) << 16),
                                                           (unsigned)float_to_f16_bits(r[2]) | ((unsigned)float_to_f16_bits(r[3]) << 16)};
            else
                *(u32x2*)((uint16_t*)p.C + idx[0]) = u32x2{(unsigned)float_to_bf16_bits(r[0]) | ((unsigned)float_to_bf16_bits(r[1]) << 16),
                                                           (unsigned)float_to_bf16_bits(r[2]) | ((unsigned)float_to_bf16_bits(r[3]) << 16)};
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < cols) store_out(p.C, p.out_type, idx[e], r[e]);
    }
}

// g: the caller's problem (its C, strides, output type and ops); ws: the slices the first step wrote
hipError_t launch_splitk_reduce(const GemmArgs& g, const void* ws, int splits, hipStream_t stream)
{
    SplitReduceArgs a{};
    a.ws = ws; a.splits = splits; a.M = g.M; a.N = g.N;
    a.C = g.C; a.c_rs = g.c_rs; a.c_cs = g.c_cs;
    a.out_type = g.out_type; a.is_int = g.in_type == T_I8;
    a.prologue = g.prologue; a.epilogue = g.epilogue; a.prologue_arg = g.prologue_arg; a.epilogue_arg = g.epilogue_arg;
    const int64_t threads = (int64_t)g.M * ((g.N + 3) / 4);
    const int64_t blocks = (threads + 255) / 256;
    if (blocks <= 0 || blocks > 0x7fffffffll) return hipErrorInvalidValue;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a.ws, a.C, a.splits, a.M, a.N, a.c_rs, a.c_cs, a);
    return hipGetLastError();
}

} // namespace acc950
