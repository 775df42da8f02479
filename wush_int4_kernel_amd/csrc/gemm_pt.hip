// gemm_pt.hip -- per-tensor W4A4 GEMM for prefill-sized products on int8 MFMA
// (csrc/gemm_cutlass_int4.cu:132-188 is the reference contract):
// y = alpha * (xq @ wq^T), an exact int32 dot over all of K.
//
// Workgroup: 4 wavefronts in 2 x 2, each owning 16 RB x 16 CB outputs (256 x
// 256, 256 x 128 or 128 x 128 per workgroup), one wavefront per SIMD.  K
// advances 256 codes (a row's 128-byte line) per super-stage; the packed codes
// are DMA'd into LDS as whole lines, 8 rows per instruction, NB super-stages
// deep.  A lane of quarter q takes the 32 bytes [32 q, 32 q + 32) of its row's
// line, 16 per half super-stage, so each 16-byte LDS read feeds two K = 64
// MFMA steps (any order of K serves a dot product, the same on both sides).
//
// The codes are unpacked to 16 * code int8 in registers (6 VALU per operand),
// 1.5 VALU per v_mfma_i32_16x16x64_i8, placed by hand behind the MFMAs: a
// wavefront alternating up to two VALU with each 16-cycle MFMA keeps the MFMA
// rate (506 cycles for 32 MFMAs and 64 VALU against 503 for the MFMAs alone;
// in blocks, 724).
//
// Measured against the 128 x 128 tiles of gemm_s4.hip (8-byte fragments
// unpacked behind LDS stores, no order over the XCDs): 512 x 24576 x 4096 62.2 ->
// 46.6 us (2.2 POP/s; three quarters of one round of 256 x 256), 2048 x 4096 x
// 4096 41.9 -> 30.7, 4096^3 75.6 -> 52.0, 4096 x 57344 x 8192 1918 -> 1151 (3.3
// POP/s), 203 x 8192 x 8192 45.0 -> 28.4, 256 x 4096 x 4096 24.8 -> 16.2.
// Bound by the MFMAs (1024 of about 1240 cycles per K = 64 step of a lone 256 x
// 256 tile) and, on the full chip, by its power.
#include "gemm_h16_device.h"
#include "gemm_pt.h"

namespace wush {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

// c += a * b (int32, exact), accumulator in place; waits as mfma16_inplace
__device__ __forceinline__ void mfma_i8_inplace(v4i& c, const v4i& a, const v4i& b) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

template <int RB, int CB, int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_pt_kernel(const uint8_t* __restrict__ xq, const uint8_t* __restrict__ wq, uint16_t* __restrict__ y, int M,
                    int N, int K, float alpha, const float* __restrict__ alpha_dev) {
    constexpr int TR = 32 * RB, TC = 32 * CB;
    constexpr int DA = TR / 32, DB = TC / 32;    // DMAs per wavefront and super-stage (8 rows each)
    constexpr int ND = DA + DB;
    constexpr int kA = TR * 128, kBuf = kA + TC * 128;
    constexpr int kStage = 4 * (16 * RB) * (32 * CB);    // fp16 outputs staged, 32 CB bytes a row
    constexpr int kSmem = NB * kBuf > kStage ? NB * kBuf : kStage;
    __shared__ __align__(16) uint8_t smem[kSmem];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int l16 = lane & 15, kq = lane >> 4;
    const int wr = wave >> 1, wc = wave & 1;
    const int K2 = K >> 1, NS = K >> 8;
    int tm, tn;
    h16_tile((int)blockIdx.x, (M + TR - 1) / TR, (N + TC - 1) / TC, tm, tn);
    const int m0 = tm * TR, n0 = tn * TC;
    const uint32_t lds0 = lds_addr(smem);

    // DMA k of a super-stage: 8 rows; lane l fetches piece (l % 8) ^ f(r) of
    // row r = 8 k' + l / 8, f(r) = (r / 2) % 8, so that 16 consecutive rows'
    // reads of one piece hit distinct banks.  Rows past M or N read the last.
    uint32_t voff[ND];
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        const int r = 8 * (k < DA ? wave * DA + k : wave * DB + k - DA) + (lane >> 3);
        const int lim = (k < DA ? M - m0 : N - n0) - 1;
        voff[k] = (uint32_t)min(r, lim) * (uint32_t)K2 + 16u * ((lane & 7) ^ ((r >> 1) & 7));
    }
    const uint8_t* abase = xq + (size_t)m0 * K2;
    const uint8_t* bbase = wq + (size_t)n0 * K2;
    auto issue = [&](int st, int buf, int k) {   // past the end: the last super-stage
        const size_t o = (size_t)min(st, NS - 1) * 128;
        const uint32_t dst = lds0 + buf * kBuf;
        if (k < DA) dma16_uniform(abase + o, voff[k], dst + (wave * DA + k) * 1024);
        else dma16_uniform(bbase + o, voff[k], dst + kA + (wave * DB + k - DA) * 1024);
    };

    v4i acc[RB][CB];
    u32v4 ra[2][RB], rb[2][CB];                  // packed codes [half][block]
    v4i ua[2], ub[2][CB];                        // unpacked operands: two row blocks, two steps' columns
    const int fsw = (l16 >> 1) & 7;
    const uint8_t* arow = smem + (wr * RB * 16 + l16) * 128;
    const uint8_t* brow = smem + kA + (wc * CB * 16 + l16) * 128;
    // read q (columns first) of half h of the super-stage in buffer buf
    auto read_raw = [&](int h, int buf, int q) {
        const int o = buf * kBuf + 16 * ((2 * kq + h) ^ fsw);
        if (q < CB) rb[h][q] = *reinterpret_cast<const u32v4*>(brow + o + q * 2048);
        else ra[h][q - CB] = *reinterpret_cast<const u32v4*>(arow + o + (q - CB) * 2048);
    };
    // VALU t (of 6) of unpacking dwords 2s, 2s + 1 of r
    auto unpack = [&](v4i& u, const u32v4& r, int s, int t) {
        const uint32_t w = r[2 * s + t / 3];
        const int e = 2 * (t / 3);
        if (t % 3 == 0) u[e] = (int)(w << 4);
        else if (t % 3 == 1) u[e] = (int)((uint32_t)u[e] & 0xF0F0F0F0u);
        else u[e + 1] = (int)(w & 0xF0F0F0F0u);
    };

#pragma unroll
    for (int s = 0; s < NB; ++s)
#pragma unroll
        for (int k = 0; k < ND; ++k) issue(s, s, k);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = (v4i){0, 0, 0, 0};
    WUSH_WAIT_VMCNT((NB - 1) * ND);
    WUSH_LDS_BARRIER();
#pragma unroll
    for (int q = 0; q < RB + CB; ++q) read_raw(0, 0, q);
#pragma unroll
    for (int t = 0; t < 6; ++t) {
#pragma unroll
        for (int j = 0; j < CB; ++j) unpack(ub[0][j], rb[0][j], 0, t);
        unpack(ua[0], ra[0][0], 0, t);
    }
    asm volatile("s_nop 7");                     // the zeroed accumulators before the first MFMA
    __builtin_amdgcn_sched_barrier(0);

    int buf = 0;                                 // LDS buffer of super-stage st
    for (int st = 0; st < NS; ++st) {
        const int nbuf = buf + 1 == NB ? 0 : buf + 1;
        static_for<2>([&](auto hc) {
            constexpr int h = hc.value;
            static_for<2>([&](auto sc) {
                constexpr int s = sc.value;
                // operands prepared: the next step's, in half h (s = 0) or the next one
                constexpr int hn = s == 0 ? h : h ^ 1, sn = s ^ 1;
                static_for<RB * CB>([&](auto mc) {
                    constexpr int m = mc.value, i = m / CB, j = m % CB;
                    mfma_i8_inplace(acc[i][j], ub[s][j], ua[i & 1]);
                    // row block i + 1 (or 0 of the next step) in the group's
                    // first MFMAs, a column block of the next step behind it
                    constexpr int t0 = j * 6 / (CB - 1), t1 = (j + 1) * 6 / (CB - 1);
                    static_for<(t1 < 6 ? t1 : 6) - (t0 < 6 ? t0 : 6)>([&](auto tc) {
                        constexpr int t = t0 + tc.value;
                        if constexpr (i + 1 < RB) unpack(ua[(i + 1) & 1], ra[h][i + 1], s, t);
                        else unpack(ua[0], ra[hn][0], sn, t);
                    });
                    constexpr int c0 = m * 6 * CB / (RB * CB), c1 = (m + 1) * 6 * CB / (RB * CB);
                    static_for<c1 - c0>([&](auto cc) {
                        constexpr int c = c0 + cc.value;
                        unpack(ub[s ^ 1][c / 6], rb[hn][c / 6], sn, c % 6);
                    });
                    // the next half's packed codes, over the first step (the
                    // second step's unpacking already takes column block 0)
                    if constexpr (s == 0) {
                        constexpr int q0 = m * (RB + CB) / (RB * CB - RB), q1 = (m + 1) * (RB + CB) / (RB * CB - RB);
                        static_for<(q1 < RB + CB ? q1 : RB + CB) - (q0 < RB + CB ? q0 : RB + CB)>([&](auto qc) {
                            read_raw(h ^ 1, h == 0 ? buf : nbuf, q0 + qc.value);
                        });
                    }
                    // second half: every read of this buffer is done
                    if constexpr (h == 1) {
                        constexpr int p = s * RB * CB + m, d0 = p * ND / (2 * RB * CB), d1 = (p + 1) * ND / (2 * RB * CB);
                        if constexpr (d1 > d0) issue(st + NB, buf, d0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            if constexpr (h == 0) {
                // super-stage st + 1 has landed in all wavefronts' view, and
                // all have read this one's second half
                WUSH_WAIT_VMCNT((NB - 2) * ND);
                WUSH_LDS_BARRIER();
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        buf = nbuf;
    }
    WUSH_WAIT_VMCNT(0);
    asm volatile("s_nop 15\n\ts_nop 15");        // the last MFMAs' results
    __syncthreads();

    // outputs through LDS: rows of 32 CB bytes, chunk c of row r at c ^ (r % chunks)
    const float out_scale = (alpha_dev ? *alpha_dev : alpha) * (1.0f / 256.0f);   // operands carry 16 * 16
    constexpr int kRow = 32 * CB, kChunks = kRow / 16;
    uint8_t* stg = smem + wave * (16 * RB * kRow);
    uint8_t* wst = stg + l16 * kRow + (kq & 1) * 8;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        uint8_t* w = wst + ((2 * j + (kq >> 1)) ^ (l16 & (kChunks - 1))) * 16;
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            v4f v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (float)acc[i][j][r] * out_scale;
            *reinterpret_cast<h4*>(w + i * 16 * kRow) = __builtin_convertvector(v, h4);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    const bool vec = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0;
    const int mw = m0 + wr * RB * 16, nw = n0 + wc * CB * 16;
    if (!vec) {
        if ((N & 1) == 0 && (reinterpret_cast<uintptr_t>(y) & 3u) == 0)
            store_staged<kRow, uint32_t>(stg, 16 * RB, y, mw, M, nw, N, lane);
        else
            store_staged<kRow, uint16_t>(stg, 16 * RB, y, mw, M, nw, N, lane);
        return;
    }
    constexpr int kRows = 64 / kChunks;          // rows per store instruction
    const int r0 = lane / kChunks, c = lane % kChunks;
#pragma unroll 8
    for (int k = 0; k < 16 * RB / kRows; ++k) {
        const int r = k * kRows + r0;
        const uint4 v = *reinterpret_cast<const uint4*>(stg + r * kRow + ((c ^ (r & (kChunks - 1))) * 16));
        if (mw + r < M && nw + c * 8 < N) *reinterpret_cast<uint4*>(y + (size_t)(mw + r) * N + nw + c * 8) = v;
    }
}

}  // namespace

int launch_gemm_pt(const uint8_t* xq, const uint8_t* wq, uint16_t* y, int M, int N, int K, float alpha,
                   const float* alpha_dev, int tile_rows, int tile_cols, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K < 256 || K % 256 != 0) return (int)hipErrorInvalidValue;
    const long long tiles = (long long)((M + tile_rows - 1) / tile_rows) * ((N + tile_cols - 1) / tile_cols);
    if (tiles > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)tiles);
    if (tile_rows == 256 && tile_cols == 256)
        gemm_pt_kernel<8, 8, 2><<<grid, 256, 0, stream>>>(xq, wq, y, M, N, K, alpha, alpha_dev);
    else if (tile_rows == 256 && tile_cols == 128)
        gemm_pt_kernel<8, 4, 3><<<grid, 256, 0, stream>>>(xq, wq, y, M, N, K, alpha, alpha_dev);
    else if (tile_rows == 128 && tile_cols == 128)
        gemm_pt_kernel<4, 4, 4><<<grid, 256, 0, stream>>>(xq, wq, y, M, N, K, alpha, alpha_dev);
    else
        return (int)hipErrorInvalidValue;
    return (int)hipGetLastError();
}

}  // namespace wush
