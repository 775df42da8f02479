// gemm_h16.hip -- group-scaled W4A4 GEMM for prefill-sized M on fp16 MFMA
// (csrc/gemm_s4.cu:85-379 is the reference contract).
//
//   y[m][n] = sum_g sum_{k in g} (qx[m][k] * sx[m][g]) * (qw[n][k] * sw[n][g])
//
// The int8 kernels fold every 32x32 block of exact group dots into fp32 with
// two VALU operations per output and group, which bounds them at a quarter of
// the int8 MFMA rate.  Here the scales go into the operands instead: a code
// (3 bits of magnitude) times a bf16 scale (8-bit significand) is exact in
// fp16 (11-bit significand) once the scale sits in fp16's exponent range, and
// the product of two such operands is exact in fp32 (22 bits).  So
// v_mfma_f32_32x32x16_f16 accumulates exact terms in fp32 over the whole K and
// nothing runs per output in the main loop.
//
// Range: every activation row m gets a power of two 2^ea[m], chosen from the
// row's largest scale so that it lands in [2^12, 2^13) (code * scale <= 7 *
// 2^13 < 65504); likewise 2^eb[n] per weight column.  The epilogue multiplies
// by 2^-(ea[m] + eb[n]) with v_ldexp_f32 (exact).  Every scale down to
// 2^-29 of its row's largest converts exactly (its lowest significand bit
// stays at or above fp16's 2^-24); smaller ones keep fewer bits (an absolute
// error below 2^-37 of the row's largest scale per scale operand).  A row or column with a non-finite scale
// gives NaN, as the reference's dequantized product does (code 0 * inf).
//
// Workgroup: 8 wavefronts in 2 x 4, a 256 x 256 output tile, each wavefront
// 128 x 64 (8 accumulator blocks), one workgroup per CU.  A stage is one
// group (K = 32): thread t converts row t of the activation tile (t < 256)
// or column t - 256 of the weight tile (16 code bytes each) to fp16 in a
// double-buffered LDS tile laid out fragment-major, [K16 slice][32-row block]
// [k-half][row][8 halves], so that a wavefront's operand read of one 32-row
// block is 1 KiB contiguous (lane l at 16*l) and the conversion writes of
// 64 consecutive rows are contiguous too.  Global loads run in batches of four
// groups (64 bytes of every row, four stages ahead), four lanes per row so an
// instruction reads 16 rows of 64 contiguous bytes, then a 4 x 4 in-quad
// transpose gives every lane its own row; addresses are clamped, so the loop
// has no conditional loads.
#include "gemm_h16_device.h"
#include "gemm_h16.h"
#include "setup.h"

namespace wush {
namespace {

#ifndef WUSH_H16_XCD
#define WUSH_H16_XCD 1                           // XCD-aware tile order in the 8-wavefront kernel
#endif

// 8 wavefronts per workgroup (2 per SIMD): the MFMA tiles are 128 x 64 per
// wavefront (2 x 4 wavefronts, 128 fp32 accumulators), and wavefronts 0-3
// convert the activation rows, 4-7 the weight columns.  A second wavefront
// per SIMD lets the conversion VALU of one run beside the MFMAs of the other
// (with 4 wavefronts of 128 x 128, L70 M=4096 took 4.51 ms against 3.75).
template <bool VEC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_h16w8_kernel(const uint8_t* __restrict__ xq, const uint16_t* __restrict__ xs,
                       const uint8_t* __restrict__ wq, const uint16_t* __restrict__ ws,
                       uint16_t* __restrict__ y, float* __restrict__ partial, int M, int N, int K,
                       int groups_per_split) {
    extern __shared__ __align__(16) uint8_t smem[];
    int* sh_e = reinterpret_cast<int*>(smem + 2 * kH16Buf);   // [0, 256) rows, [256, 512) columns

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
#if WUSH_H16_XCD
    // Workgroup i runs on XCD i % 8.  When the column tiles split evenly
    // over the 8 XCDs, XCD x takes column tiles x, x + 8, ... and walks all
    // row tiles of one before the next, so the workgroups in flight on an XCD
    // share a few weight tiles in its L2.
    int tm = blockIdx.y, tn = blockIdx.x;
    if ((gridDim.x & 7) == 0) {
        const uint64_t id = (uint64_t)blockIdx.y * gridDim.x + blockIdx.x;
        const uint64_t slot = id >> 3;
        tm = (int)(slot % gridDim.y);
        tn = (int)((slot / gridDim.y) * 8 + (id & 7));
    }
    const int m0 = tm * kH16Tile;
    const int n0 = tn * kH16Tile;
#else
    const int m0 = blockIdx.y * kH16Tile;
    const int n0 = blockIdx.x * kH16Tile;
#endif
    const int GR = K >> 5;                       // groups of a row
    const int K2 = K >> 1;
    // K slice of this workgroup (blockIdx.z): groups [gb, gb + G), G % 8 == 0
    const int gb = blockIdx.z * groups_per_split;
    const int G = min(GR - gb, groups_per_split);

    // conversion role (wavefront-uniform): operand, its row r in the tile
    const bool wside = wave >= 4;
    const int r = tid & 255;
    const uint8_t* codes = wside ? wq : xq;
    const int lim = (wside ? N : M) - 1;
    const int base = wside ? n0 : m0;
    const uint16_t* ps = (wside ? ws : xs) + (size_t)min(base + r, lim) * GR + gb;

    uint32_t mx, mx2;
    h16_row_max<VEC>(ps, ps, G, mx, mx2);
    const int e = h16_shift(mx);
    sh_e[tid] = e;

    const int p4 = lane & 3;
    const int wrow = base + (wave & 3) * 64 + (lane & ~3);
    const uint8_t* qc[kH16Batch];
#pragma unroll
    for (int i = 0; i < kH16Batch; ++i) qc[i] = codes + (size_t)min(wrow + i, lim) * K2 + gb * 16 + p4 * 16;

    struct Batch {
        uint4 c[kH16Batch];
        uint32_t s[kH16Batch];
    };
    auto load_batch = [&](int b, Batch& rr) {
        const int g0 = min(b * kH16Batch, G - kH16Batch) * 16;
#pragma unroll
        for (int i = 0; i < kH16Batch; ++i) rr.c[i] = *reinterpret_cast<const uint4*>(qc[i] + g0);
        if constexpr (VEC) {
            const uint2 v = *reinterpret_cast<const uint2*>(ps + min(b * kH16Batch, G - kH16Batch));
            rr.s[0] = v.x; rr.s[1] = v.y;
        } else {
#pragma unroll
            for (int i = 0; i < kH16Batch; ++i) rr.s[i] = ps[min(b * kH16Batch + i, G - 1)];
        }
    };
    const bool odd1 = (lane & 1) != 0;
    const bool odd2 = (lane & 2) != 0;
    auto transpose = [&](uint4 (&x)[kH16Batch]) {
        uint4 z[kH16Batch];
#pragma unroll
        for (int i = 0; i < kH16Batch; ++i) {
            const bool own = ((i & 1) != 0) == odd1;
            const uint4 o = x[i ^ 1];
            z[i].x = h16_xchg<0xB1>(x[i].x, o.x, !own);
            z[i].y = h16_xchg<0xB1>(x[i].y, o.y, !own);
            z[i].z = h16_xchg<0xB1>(x[i].z, o.z, !own);
            z[i].w = h16_xchg<0xB1>(x[i].w, o.w, !own);
        }
#pragma unroll
        for (int i = 0; i < kH16Batch; ++i) {
            const bool own = ((i & 2) != 0) == odd2;
            const uint4 o = z[i ^ 2];
            x[i].x = h16_xchg<0x4E>(z[i].x, o.x, !own);
            x[i].y = h16_xchg<0x4E>(z[i].y, o.y, !own);
            x[i].z = h16_xchg<0x4E>(z[i].z, o.z, !own);
            x[i].w = h16_xchg<0x4E>(z[i].w, o.w, !own);
        }
    };

    Batch R0, R1;
    load_batch(0, R0);
    load_batch(1, R1);

    const int wofs = (wside ? kH16Op : 0) + (r >> 5) * 1024;
    auto convert = [&](int buf, Batch& rr, int i) {
        if (i == 0) transpose(rr.c);
        uint8_t* dst = smem + buf * kH16Buf + wofs;
        const h2 sc = h16_scale(h16_batch_scale<VEC>(rr.s, i), e);
        const uint32_t w4[4] = {rr.c[i].x, rr.c[i].y, rr.c[i].z, rr.c[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            frag_write(dst + (j >> 1) * kH16Slice, (r & 31) + 32 * (j & 1), h16_codes(w4[j], sc));
    };

    v16f acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (v16f){0.0f};

    const int rba = (wave >> 2) * 4;             // this wavefront's first 32-row block
    const int rbb = (wave & 3) * 2;              // ... and first 32-column block
    auto compute = [&](int buf) {
        const uint8_t* b0 = smem + buf * kH16Buf;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            h8 af[4], bf[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) af[i] = frag_read(b0 + kk * kH16Slice + (rba + i) * 1024, lane);
#pragma unroll
            for (int j = 0; j < 2; ++j) bf[j] = frag_read(b0 + kH16Op + kk * kH16Slice + (rbb + j) * 1024, lane);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    };

    convert(0, R0, 0);
    __syncthreads();

    for (int s0 = 0; s0 < G; s0 += 2 * kH16Batch) {
#pragma unroll
        for (int j = 0; j < 2 * kH16Batch; ++j) {
            compute(j & 1);
            if (j < kH16Batch - 1) convert((j + 1) & 1, R0, j + 1);
            else if (j == kH16Batch - 1) convert(0, R1, 0);
            else if (j < 2 * kH16Batch - 1) convert((j + 1) & 1, R1, j + 1 - kH16Batch);
            else convert(0, R0, 0);
            if (j == kH16Batch - 1) load_batch(s0 / kH16Batch + 2, R0);
            if (j == 2 * kH16Batch - 1) load_batch(s0 / kH16Batch + 3, R1);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    const int half = lane >> 5;
    const int l32 = lane & 31;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int cl = (rbb + j) * 32 + l32;
        const int col = n0 + cl;
        const int e_col = sh_e[256 + cl];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int rl = (rba + i) * 32 + 8 * (q >> 2) + 4 * half + (q & 3);
                const int row = m0 + rl;
                const int e_row = sh_e[rl];
                float v = __builtin_ldexpf(acc[i][j][q], -(e_row + e_col));
                if (e_row == kH16NonFinite || e_col == kH16NonFinite) v = __builtin_nanf("");
                if (row < M && col < N) {
                    if (partial != nullptr)
                        partial[((size_t)blockIdx.z * M + row) * N + col] = v;
                    else
                        y[(size_t)row * N + col] = f32_to_f16_bits(v);
                }
            }
        }
    }
}

}  // namespace

size_t gemm_h16_smem_bytes() { return 2 * kH16Buf + 2 * kH16Tile * sizeof(int); }

int gemm_h16_init_device() {
    // the workgroup's LDS is above the default 64 KiB limit of dynamic LDS
    const int smem = (int)gemm_h16_smem_bytes();
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_h16w8_kernel<true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_h16w8_kernel<false>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    return (int)e;
}

int launch_gemm_h16(const uint8_t* xq, const uint16_t* xs, const uint8_t* wq, const uint16_t* ws,
                    uint16_t* y, float* partial, int M, int N, int K, int splits, int groups_per_split,
                    hipStream_t stream) {
    const int G = K >> 5;
    // every K slice holds a positive multiple of 8 groups
    if (M <= 0 || N <= 0 || K <= 0 || K % 256 != 0 || splits < 1 || groups_per_split <= 0 ||
        groups_per_split % 8 != 0 || (long long)splits * groups_per_split < G ||
        (long long)(splits - 1) * groups_per_split >= G || (splits > 1 && partial == nullptr))
        return (int)hipErrorInvalidValue;
    int dev = 0;
    const int st = device_setup(&dev);
    if (st != 0) return st;
    const bool vec = G % 8 == 0 && ((reinterpret_cast<uintptr_t>(xs) | reinterpret_cast<uintptr_t>(ws)) & 15u) == 0;
    dim3 grid((unsigned)((N + kH16Tile - 1) / kH16Tile), (unsigned)((M + kH16Tile - 1) / kH16Tile), (unsigned)splits);
    const size_t smem = gemm_h16_smem_bytes();
    if (vec)
        gemm_h16w8_kernel<true><<<grid, 512, smem, stream>>>(xq, xs, wq, ws, y, partial, M, N, K, groups_per_split);
    else
        gemm_h16w8_kernel<false><<<grid, 512, smem, stream>>>(xq, xs, wq, ws, y, partial, M, N, K, groups_per_split);
    return (int)hipGetLastError();
}

}  // namespace wush
