// gemm_h16q.hip -- the fp16-MFMA prefill GEMM with activations converted once
// into a workspace and weights converted in registers, one wavefront per SIMD
// (csrc/gemm_s4.cu:85-379 is the reference contract; operands and numerics as
// in gemm_h16.hip).
//
// Workgroup: 4 wavefronts side by side over 256 weight columns, wavefront w
// owning all of the tile's rows (256, 128 or 64) and columns 64w .. 64w + 63.
// Because no other wavefront needs its columns, a wavefront converts its
// weight codes straight into MFMA operand registers: no LDS traffic for
// converted weights.  The activations, converted once by h16_prep_kernel in
// the matching layout, are DMA'd into a 4-slot LDS ring and read by all four.
//
// What bounds it on MI355X: power (the clock is 2.0 GHz at 4096 cubed with the
// MFMA pipes 62% busy, 1.6-1.7 at L70 M=4096 with 76%).  There an MFMA-only
// loop of the same tile runs at 1.5-1.6 PFLOP/s with the clock near 1.5 GHz,
// so the MFMA form matters: v_mfma_f32_16x16x32_f16 moves a third less
// accumulator data per flop than 32x32x16 and the same loop ran 7-10% faster
// (4096 x 16384 x 8192, operands in LDS: 907 -> 806 us).  The accumulators
// are written in place by an asm MFMA: left to the compiler, tiles that do
// not fill the AGPRs rotate them (each MFMA writing the next one's input),
// which ran 40% slower.
//
// With one wavefront per SIMD there is no second wavefront to run the memory
// work beside the MFMAs, so each stage (one group of K per lane quarter, 32
// in all) interleaves by hand: after each MFMA of stage t at most one LDS read
// of stage t+1's activations, one or two VALU of the conversion of stage
// t+1's weights, or one DMA of stage t+4 (DMAs issued four in a row held the
// MFMAs up: 926 -> 870 us in the loop above when spread).  One barrier per stage.
//
// Stage layout: a weight column's 16 code bytes of group 4b + q sit in lane
// quarter q, and stage 4b + s takes dword s of all four: a lane reads 16
// contiguous bytes once per four stages and converts one scale for them.
//
// Weight codes come in double batches of 8 groups, each column's whole
// 128-byte line per 8 lanes (a load touching 32 lines costs the vector memory
// path about as much as one reading them whole), one DMA per stage.  Every
// global load of the loop is an LDS DMA issued by asm that the compiler does
// not see; the kernel counts them itself.  Every stage issues NA activation
// DMAs and one code DMA, and stage 4 of each 8 the scale DMAs (one, or four for
// a K that is not a multiple of 256); at a stage's end all but those of the
// last two stages have landed, so what a stage issues is read three stages
// later at the earliest.
//
// Outputs: fp16 through LDS (the ring and code buffers are free after the
// last stage) as 8-byte writes -- the weights are the MFMA's row operand, so
// a lane holds 4 consecutive columns of one row -- and 16-byte row chunks to
// memory.  The shifts come from LDS and non-finite rows from NaN operands, so
// an output costs four VALU (accumulator read, add, ldexp, half a conversion);
// with per-output tests and 2-byte writes a 256 x 256 tile spent 15-20 us
// outside its K loop, now about 10.
//
// Rows and columns whose scales span more than the operands hold (h16_loses_bits)
// are found by the conversion kernel, and a tile ends by computing their
// outputs from the codes and bf16 scales: inputs without them pay one test per
// row and column.
//
// Measured (layer with the fused transform, same box, against the 32x32x16
// form with burst DMAs): K=8192 N=57344 M=4096 3179 -> 2679 us (1.45 PFLOP/s;
// a library fp16 GEMM of the shape 2560-2850), M=256 238 -> 197, M=128 146 ->
// 126; K=N=8192 M=4096 511 -> 431, M=512 116 -> 94; K=4096 N=24576 M=1024
// 232 -> 185.
#include "gemm_h16_device.h"
#include "gemm_h16.h"
#include "setup.h"

namespace wush {
namespace {

constexpr int kH16qStage = kH16Tile * 64;        // workspace bytes of one stage of a 256-row tile
// Row/column shift marking codes whose scale loses bits as a shifted fp16
// operand: it is more than 2^29 below the row's largest over the K slice (the
// largest lies in [2^12, 2^13), fp16's lowest bit is 2^-24, a bf16 has 8).
constexpr int kH16Wide = 1 << 21;

__device__ __forceinline__ bool h16_loses_bits(uint32_t bits, uint32_t mx) {
    return (int)(mx >> 7) - max((int)(bits >> 7), 1) > 29;
}

// Outputs of R rows (or columns) `u` against each lane's column (or row) `l`,
// all indexes into (rows, GR) groups of codes and scales: exact int32 dots of
// groups [g0, g1) summed in fp64; NaN where a scale is not finite, whatever the
// codes.  For the outputs of wide rows and columns only.  Alone (R = 1) bound by
// the latency of the lane side's loads, 64 rows of one 16-byte group each, so
// AHEAD groups go out at a time; by their number where many are wide, so they
// meet R rows of the other side, whose address is the same in every lane.
// 2048 x 4096 x 4096, product: 72 us without a wide row, 95 with one, 249 with
// a tenth of them, 1.5 ms with all (one row and 8 groups at a time: 117, 868,
// 8.1 ms; the per-tile kernel, which loses the bits, 97).
template <int R, int AHEAD>
__device__ __forceinline__ void h16_exact_outputs(const uint8_t* __restrict__ uq, const uint16_t* __restrict__ us,
                                                  const uint8_t* __restrict__ lq, const uint16_t* __restrict__ ls,
                                                  const int (&u)[R], int l, int GR, int g0, int g1, float (&out)[R]) {
    const uint4* lc = reinterpret_cast<const uint4*>(lq) + (size_t)l * GR;
    const uint16_t* lsc = ls + (size_t)l * GR;
    double acc[R];
    uint32_t top[R], ltop = 0;                   // largest scale bits, sign cleared
#pragma unroll
    for (int k = 0; k < R; ++k) {
        acc[k] = 0.0;
        top[k] = 0;
    }
    auto take = [&](auto nc, int g) {            // groups g .. g + n - 1
        constexpr int n = nc.value;
        uint4 b[n];
        uint32_t sl[n];
#pragma unroll
        for (int i = 0; i < n; ++i) {
            b[i] = lc[g + i];
            sl[i] = lsc[g + i];
        }
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint4* uc = reinterpret_cast<const uint4*>(uq) + (size_t)u[k] * GR + g;
            const uint16_t* usc = us + (size_t)u[k] * GR + g;
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const uint4 a = uc[i];
                const uint32_t w = usc[i];
                int d = __builtin_amdgcn_sdot8((int)a.x, (int)b[i].x, 0, false);
                d = __builtin_amdgcn_sdot8((int)a.y, (int)b[i].y, d, false);
                d = __builtin_amdgcn_sdot8((int)a.z, (int)b[i].z, d, false);
                d = __builtin_amdgcn_sdot8((int)a.w, (int)b[i].w, d, false);
                top[k] = max(top[k], w & 0x7fffu);
                acc[k] += (double)d * ((double)__uint_as_float(w << 16) * (double)__uint_as_float(sl[i] << 16));
            }
        }
#pragma unroll
        for (int i = 0; i < n; ++i) ltop = max(ltop, sl[i] & 0x7fffu);
    };
    int g = g0;
#pragma unroll 1
    for (; g + AHEAD <= g1; g += AHEAD) take(std::integral_constant<int, AHEAD>{}, g);
#pragma unroll 1
    for (; g + 8 <= g1; g += 8) take(std::integral_constant<int, 8>{}, g);
#pragma unroll 1
    for (; g < g1; g += 2) take(std::integral_constant<int, 2>{}, g);    // K % 64 == 0: whole pairs
#pragma unroll
    for (int k = 0; k < R; ++k) out[k] = max(top[k], ltop) >= 0x7f80u ? __builtin_nanf("") : (float)acc[k];
}

// RB: 16-row blocks per wavefront, 16 (256-row tiles), 8 or 4 (128- and 64-row
// tiles: fewer accumulators, the same weight conversion per stage).  PAD: K is
// a multiple of 64 but not of 256: the last double batch reads the row's last
// groups again in place of those past the end, whose activations and weight
// scales are zero, and scales come 4 bytes at a time (rows of them are only
// 4-byte aligned).
template <int RB, bool PAD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_h16q_kernel(const uint8_t* __restrict__ a16, const int* __restrict__ ea, const int* __restrict__ eb,
                      const uint8_t* __restrict__ wq, const uint16_t* __restrict__ ws, uint16_t* __restrict__ y,
                      float* __restrict__ partial, int M, int N, int K, int groups_per_split,
                      const uint8_t* __restrict__ xq, const uint16_t* __restrict__ xs) {
    constexpr int TR = 16 * RB, TC = kH16Tile;
    constexpr int NA = TR / 64;                  // activation DMAs per wavefront and stage
    constexpr int NM = 4 * RB;                   // MFMAs per stage
    constexpr int kSlot = TR * 64;               // LDS: activation ring of 4 slots,
    constexpr int kCodes = 4 * kSlot;            // two double batches of codes per wavefront
    constexpr int kScales = kCodes + 2 * 4 * 8192;   // [64 columns][128 B, pieces swizzled], their
    constexpr int kShifts = kScales + 2 * 4 * 1024;  // scales [64 columns][8 groups], row and column shifts
    __shared__ __align__(16) uint8_t smem[kShifts + 2048];
    static_assert(4 * TR * 128 <= kScales, "outputs staged over the ring and code buffers");

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int l16 = lane & 15, kq = lane >> 4;   // row or column of an operand, lane quarter
    const int GR = K >> 5, GP = PAD ? (GR + 7) & ~7 : GR;   // groups of a row, and whole double batches of them
    const int K2 = K >> 1;
    const int NR = (M + TR - 1) / TR, NC = (N + TC - 1) / TC;
    // shifts and converted activations are laid out over 256-row padding
    const int mpad = (M + kH16Tile - 1) / kH16Tile * kH16Tile, npad = NC * kH16Tile;
    const int slice = blockIdx.x / (NR * NC);
    int tm, tn;
    h16_tile((int)blockIdx.x - slice * (NR * NC), NR, NC, tm, tn);
    const int m0 = tm * TR;
    const int n0 = tn * TC;
    const int gb = slice * groups_per_split;
    const int G = min(GP - gb, groups_per_split);
    const uint32_t lds0 = lds_addr(smem);

    // activation DMA of this wavefront: KiB NA w .. NA w + NA - 1 of a stage
    const uint8_t* asrc = a16 + ((size_t)(m0 >> 8) * GP + gb) * kH16qStage + (m0 & 255) * 64 + wave * (NA * 1024);
    const uint32_t avoff = lane * 16;
    auto issue_a = [&](int st, int slot, int d) {    // past the slice: the last stage
        dma16_uniform(asrc + (size_t)min(st, G - 1) * kH16qStage + d * 1024, avoff,
                      lds0 + slot * kSlot + wave * (NA * 1024) + d * 1024);
    };
    // Code DMA k of a double batch: columns 8k .. 8k+7 of the wavefront's 64.
    // Lane l fetches piece (l % 8) ^ f(c) of column c = 8k + l / 8, so that
    // piece p of column c sits at 128 c + 16 (p ^ f(c)) with f(c) = (c / 2) %
    // 8: 16 consecutive readers (columns c .. c+15, one piece) hit distinct
    // banks.  Columns past N read column N - 1.
    const int col0 = n0 + wave * 64;
    auto issue_c = [&](int d, int buf, int k) {
        const int o = min(d * 8, G - 8);
        const int c = 8 * k + (lane >> 3);
        const int p = (lane & 7) ^ ((c >> 1) & 7);
        const int col = min(col0 + c, N - 1);
        const int g = PAD ? min(gb + o + p, GR - 1) : gb + o + p;
        dma16(wq + (size_t)col * K2 + (size_t)g * 16,
              lds0 + kCodes + (buf * 4 + wave) * 8192 + k * 1024);
    };
    // scales of a double batch: [column][8 groups], PAD: [group pair][column][2]
    constexpr int kScaleDmas = PAD ? 4 : 1;
    const uint16_t* ssrc = ws + (size_t)min(col0 + lane, N - 1) * GR;
    auto issue_s = [&](int d, int buf) {
        const int g = gb + min(d * 8, G - 8);
        const uint32_t dst = lds0 + kScales + (buf * 4 + wave) * 1024;
        if constexpr (PAD) {
#pragma unroll
            for (int k = 0; k < 4; ++k) dma4(ssrc + min(g + 2 * k, GR - 2), dst + k * 256);
        } else {
            dma16(ssrc + g, dst);
        }
    };

    v4f acc[RB][4];
    h8 fa[2][RB];                                // [register set][row block]
    uint32_t fb[2][4][4];                        // [register set][column block][dword]
    const uint8_t* abase = smem + lane * 16;
    auto read_a = [&](int P, int slot, int i) {
        fa[P][i] = *reinterpret_cast<const h8*>(abase + slot * kSlot + i * 1024);
    };
    // A weight batch (four stages) in registers: per column block the lane's
    // 16 code bytes (group 4b + kq) and their fp16 scale
    struct Batch {
        u32v4 c[4];
        h2 s[4];
    };
    Batch R[2];
    uint32_t sraw[4];
    int ecol[4];
    const int fsw = (l16 >> 1) & 7;              // f(c) of the lane's columns
    auto read_batch = [&](int b, Batch& r) {
        const uint8_t* cb = smem + kCodes + (((b >> 1) & 1) * 4 + wave) * 8192 + l16 * 128 +
                            16 * ((4 * (b & 1) + kq) ^ fsw);
        const int gq = 4 * (b & 1) + kq;         // the lane's group of the double batch
        const uint8_t* sb = smem + kScales + (((b >> 1) & 1) * 4 + wave) * 1024 +
                            (PAD ? (gq >> 1) * 256 + l16 * 4 + 2 * (gq & 1) : l16 * 16 + 2 * gq);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r.c[j] = *reinterpret_cast<const u32v4*>(cb + j * 2048);
            sraw[j] = *reinterpret_cast<const uint16_t*>(sb + j * (PAD ? 64 : 256));
        }
        if constexpr (PAD) {
            if (gb + 4 * b + kq >= GR) {
#pragma unroll
                for (int j = 0; j < 4; ++j) sraw[j] = 0;
            }
        }
    };
    auto make_scale = [&](Batch& r, int j) { r.s[j] = h16_scale(__uint_as_float(sraw[j] << 16), ecol[j]); };
    // Step k (of 52) of h16_codes for stage s of batch r: column block k / 13
    // into register set P, one VALU instruction a step.
    uint32_t w8 = 0;
    h2 pr[4];
    auto convert_step = [&](int P, const Batch& r, int s, int k) {
        const int jb = k / 13, q = k % 13;
        const uint32_t w = r.c[jb][s];
        const h2 b0 = {(_Float16)1032.0f, (_Float16)1032.0f};
        const h2 b1 = {(_Float16)72.0f, (_Float16)72.0f};
        if (q == 0) w8 = w >> 8;
        else if (q == 1) pr[0] = __builtin_bit_cast(h2, h16_nib(w, 0x000F000Fu, 0x64086408u));
        else if (q == 2) pr[1] = __builtin_bit_cast(h2, h16_nib(w, 0x00F000F0u, 0x54805480u));
        else if (q == 3) pr[2] = __builtin_bit_cast(h2, h16_nib(w8, 0x000F000Fu, 0x64086408u));
        else if (q == 4) pr[3] = __builtin_bit_cast(h2, h16_nib(w8, 0x00F000F0u, 0x54805480u));
        else if (q < 9) pr[q - 5] = pr[q - 5] - ((q & 1) ? b0 : b1);
        else fb[P][jb][q - 9] = __builtin_bit_cast(uint32_t, (h2)(pr[q - 9] * r.s[jb]));
    };

    // Prologue: shifts, double batch 0, then "stages" -4 .. -1 of the loop's
    // DMA pattern (activation stages 0-3, half of double batch 1).
    if (64 * wave < TR)
        dma4(ea + (size_t)slice * mpad + m0 + wave * 64 + lane, lds0 + kShifts + wave * 256);
    dma4(eb + (size_t)slice * npad + n0 + wave * 64 + lane, lds0 + kShifts + 1024 + wave * 256);
#pragma unroll
    for (int k = 0; k < 8; ++k) issue_c(0, 0, k);
    issue_s(0, 0);
    issue_s(1, 1);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int d = 0; d < NA; ++d) issue_a(s, s, d);
        issue_c(1, 1, s);
    }
    constexpr int kInFlight = 2 * (NA + 1);      // DMAs of two stages
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    WUSH_WAIT_VMCNT(kInFlight);
    WUSH_LDS_BARRIER();
    const int* sh_e = reinterpret_cast<const int*>(smem + kShifts);   // minus the shift; [256..] columns
#pragma unroll
    for (int j = 0; j < 4; ++j) ecol[j] = -sh_e[256 + wave * 64 + j * 16 + l16];
    read_batch(0, R[0]);
#pragma unroll
    for (int j = 0; j < 4; ++j) make_scale(R[0], j);
    static_for<52>([&](auto k) { convert_step(0, R[0], 0, k.value); });
#pragma unroll
    for (int i = 0; i < RB; ++i) read_a(0, 0, i);
    asm volatile("s_nop 7");                     // the zeroed accumulators before the first MFMA
    __builtin_amdgcn_sched_barrier(0);

    for (int s0 = 0; s0 < G; s0 += 8) {
        // fully unrolled: register sets, slots and batches are picked by j
        static_for<8>([&](auto jc) {
            constexpr int j = jc.value, P = j & 1;
            const int t = s0 + j;
            Batch& Rc = R[((j + 1) >> 2) & 1];   // batch of stage t + 1
            Batch& Rn = R[((j + 2) >> 2) & 1];   // batch read at j = 2 and 6
            static_for<NM>([&](auto mc) {
                constexpr int m = mc.value, i = m >> 2, jb = m & 3;
                mfma16_inplace(acc[i][jb],
                               __builtin_bit_cast(h8, (u32v4){fb[P][jb][0], fb[P][jb][1], fb[P][jb][2], fb[P][jb][3]}),
                               fa[P][i]);
                // stage t + 4 into the slot of stage t, whose fragments were
                // all read (and waited for) before the last barrier
                if constexpr (m % (NM / 4) == 1 && m / (NM / 4) < NA) issue_a(t + 4, j & 3, m / (NM / 4));
                // double batch d's buffer is free once its second batch is in
                // registers (j = 2): the codes of d + 2 from j = 4 on
                if constexpr (m == NM * 7 / 8) {
                    if constexpr (j < 4) issue_c(s0 / 8 + 1, (s0 / 8 + 1) & 1, j + 4);
                    else issue_c(s0 / 8 + 2, (s0 / 8) & 1, j - 4);
                }
                if constexpr (j == 4 && m == NM / 2 + 2) issue_s(s0 / 8 + 2, (s0 / 8) & 1);
                if constexpr ((j & 3) == 2) {
                    if constexpr (m == 0) read_batch(s0 / 4 + (j >> 2) + 1, Rn);
                    if constexpr (m >= NM / 2 && (m - NM / 2) % (NM / 8) == 0) make_scale(Rn, (m - NM / 2) / (NM / 8));
                }
                // the activation reads end NM / 8 MFMAs before the stage, so
                // that the barrier's LDS wait finds them done (past the last
                // stage they read a stale slot, unused)
                constexpr int kReadMs = NM - NM / 8;
                static_for<RB>([&](auto r) {
                    if constexpr (r.value * kReadMs / RB == m) read_a(P ^ 1, (j + 1) & 3, r.value);
                });
                constexpr int k0 = (m * 52 + NM - 1) / NM, k1 = ((m + 1) * 52 + NM - 1) / NM;
                static_for<k1 - k0>([&](auto k) { convert_step(P ^ 1, Rc, (j + 1) & 3, k0 + k.value); });
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (j == 4 || j == 5) WUSH_WAIT_VMCNT(kInFlight + kScaleDmas);   // the scales of j = 4
            else WUSH_WAIT_VMCNT(kInFlight);
            WUSH_LDS_BARRIER();
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    // The stages past the slice DMA'd copies of its last stage into the ring
    WUSH_WAIT_VMCNT(0);
    asm volatile("s_nop 15\n\ts_nop 15");        // the last MFMAs' results
    __syncthreads();                             // the ring is free

    // the lane number again: kept over the loop, what derives from it would
    // spill a register of the 256-row tile
    const int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int lr = ln & 15, lq = ln >> 4;
    const int wn0 = n0 + wave * 64;
    int er[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) er[i] = sh_e[i * 16 + lr];
    const int4* ec4 = reinterpret_cast<const int4*>(sh_e + 256 + wave * 64 + 4 * lq);
    // accumulator [i][j][q]: row 16 i + lr, column 16 j + 4 lq + q
    auto out4 = [&](int i, int j, const int4& ec) {
        v4f v;
        v[0] = __builtin_ldexpf(acc[i][j][0], er[i] + ec.x);
        v[1] = __builtin_ldexpf(acc[i][j][1], er[i] + ec.y);
        v[2] = __builtin_ldexpf(acc[i][j][2], er[i] + ec.z);
        v[3] = __builtin_ldexpf(acc[i][j][3], er[i] + ec.w);
        return v;
    };
    if (partial != nullptr) {
        // fp32 partials of a K slice, 64 contiguous bytes per row and instruction
        const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(partial) & 15u) == 0;
        float* prow = partial + ((size_t)slice * M + m0 + lr) * N + wn0 + 4 * lq;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int4 ec = ec4[j * 4];
            const int n = wn0 + j * 16 + 4 * lq;
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const v4f v = out4(i, j, ec);
                if (m0 + i * 16 + lr < M) {
                    float* dst = prow + (size_t)(i * 16) * N + j * 16;
                    if (vec) {
                        if (n < N) *reinterpret_cast<v4f*>(dst) = v;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < N) dst[e] = v[e];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        // fp16: each wavefront's TR x 64 outputs through LDS, 128 bytes a row,
        // 16-byte chunk c of row r at chunk c ^ (r % 8)
        uint8_t* stg = smem + wave * (TR * 128);
        uint8_t* wst = stg + lr * 128 + (lq & 1) * 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int4 ec = ec4[j * 4];
            uint8_t* w = wst + ((j * 2 + (lq >> 1)) ^ (lr & 7)) * 16;
#pragma unroll
            for (int i = 0; i < RB; ++i)
                *reinterpret_cast<h4*>(w + i * 16 * 128) = __builtin_convertvector(out4(i, j, ec), h4);
            __builtin_amdgcn_sched_barrier(0);       // one column block at a time
        }
        const bool vec = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0;
        if (vec) {
            const int r0 = ln >> 3, cc = ln & 7;
            const int n = wn0 + cc * 8;
            const uint8_t* rst = stg + r0 * 128 + (cc ^ r0) * 16;    // row 8 k + r0: (8 k + r0) % 8 == r0
            uint16_t* yrow = y + (size_t)(m0 + r0) * N + n;
#pragma unroll
            for (int k = 0; k < TR / 8; ++k) {
                const uint4 v = *reinterpret_cast<const uint4*>(rst + k * 1024);
                if (m0 + 8 * k + r0 < M && n < N) *reinterpret_cast<uint4*>(yrow + (size_t)(8 * k) * N) = v;
            }
        } else if ((N & 1) == 0 && (reinterpret_cast<uintptr_t>(y) & 3u) == 0) {
            store_staged<128, uint32_t>(stg, TR, y, m0, M, wn0, N, ln);
        } else {
            store_staged<128, uint16_t>(stg, TR, y, m0, M, wn0, N, ln);
        }
    }
    // Over what was stored: outputs of wide rows and columns, then NaN for the
    // columns with a non-finite scale.
    auto put = [&](int m, int n, float v) {
        if (m >= M || n >= N) return;
        if (partial != nullptr) partial[((size_t)slice * M + m) * N + n] = v;
        else reinterpret_cast<_Float16*>(y)[(size_t)m * N + n] = (_Float16)v;
    };
    const int ecl = sh_e[256 + wave * 64 + ln];     // one column per lane
    uint64_t bad = __ballot(ecl == kH16NonFinite);
    const uint64_t wide_cols = __ballot(ecl == kH16Wide);
    const int g1 = min(GR, gb + groups_per_split);
    for (int it = 0; it < 2 * (TR / 64); ++it) {
        // wide rows of 64 against the lanes' columns, then (cols) wide columns
        // against the lanes' 64 rows
        const bool cols = it >= TR / 64;
        const int r = (cols ? it - TR / 64 : it) * 64;
        uint64_t wide = cols ? wide_cols : __ballot(sh_e[r + ln] == kH16Wide);
        if (wide == 0) continue;
        WUSH_WAIT_VMCNT(0);
        const int l = cols ? m0 + r + ln : wn0 + ln, lim = cols ? M : N;
        while (wide != 0) {
            const int base = cols ? wn0 : m0 + r;
            auto run = [&](auto rc, auto ahead) {
                constexpr int R = rc.value;
                int u[R];
                float v[R];
#pragma unroll
                for (int k = 0; k < R; ++k) {    // the last one again where fewer are left
                    u[k] = base + __builtin_ctzll(wide);
                    if (k == R - 1 || (wide & (wide - 1)) != 0) wide &= wide - 1;
                }
                h16_exact_outputs<R, ahead.value>(cols ? wq : xq, cols ? ws : xs, cols ? xq : wq, cols ? xs : ws, u,
                                                  min(l, lim - 1), GR, gb, g1, v);
#pragma unroll
                for (int k = 0; k < R; ++k)
                    if (l < lim) put(cols ? l : u[k], cols ? u[k] : l, v[k]);
            };
            if ((wide & (wide - 1)) == 0) run(std::integral_constant<int, 1>{}, std::integral_constant<int, 32>{});
            else run(std::integral_constant<int, 4>{}, std::integral_constant<int, 8>{});
        }
    }
    if (bad != 0) WUSH_WAIT_VMCNT(0);
    for (; bad != 0; bad &= bad - 1)
        for (int m = m0 + ln; m < min(M, m0 + TR); m += 64)
            put(m, wn0 + __builtin_ctzll(bad), __builtin_nanf(""));
}

// ------------------------------------------------ pre-converted activations
// a16 layout: [256-row tile][stage][16-row block][64 lanes][16 B]; stage
// 4b + s, lane (row % 16) + 16 q holds the 8 fp16 operands of dword s of group
// 4b + q.  ea[slice][row] and eb[slice][column] hold MINUS the power-of-two
// shift over the K slice, kH16NonFinite for a column with a non-finite scale
// (its outputs are set to NaN; a row with one gets NaN operands), or kH16Wide
// for a row or column with nonzero codes under a scale that would lose bits
// (its outputs are computed apart).  Rows past M are zero (shift 0 for them
// and for columns past N).
//
// Workgroups [0, na) convert 32 rows by `chunk` groups of one slice each
// (scanning the rows' scales of the slice first, 8 threads a row); the rest
// take 32 weight columns' shifts of one slice.  A wavefront load reads 8 whole
// 128-byte lines of codes and its stores write whole 128-byte lines.
// HBM-bound: 4096 x 8192 in 17.4 us (4.9 TB/s over 84 MB), against 28.5 us
// with each thread loading 16 bytes of its own row and one 32-row block per
// workgroup (most of a wave of workgroups idle at small M).
// PAD: G % 8 != 0, so rows of scales are 4-byte aligned (G is even).
//
// Bits (sign cleared) of the largest scale, and of the smallest nonzero one
// less 1 (0xffff: all are zero).
struct ScaleRange {
    uint32_t mx, mn;
};

template <bool PAD>
__device__ __forceinline__ ScaleRange slice_scale_range(const uint16_t* p, int n, int part) {
    u16x2 m2 = {0, 0}, n2 = {0xffff, 0xffff};
    auto take = [&](uint32_t w) {
        const u16x2 v = abs_bits2(w);
        m2 = __builtin_elementwise_max(m2, v);
        n2 = __builtin_elementwise_min(n2, (u16x2)(v - (u16x2){1, 1}));
    };
    if constexpr (PAD) {
        const uint32_t* p1 = reinterpret_cast<const uint32_t*>(p);
#pragma unroll 4
        for (int i = part; i < (n >> 1); i += 8) take(p1[i]);
    } else {
        const uint4* p4 = reinterpret_cast<const uint4*>(p);
#pragma unroll 4
        for (int i = part; i < (n >> 3); i += 8) {
            const uint4 v = p4[i];
            take(v.x);
            take(v.y);
            take(v.z);
            take(v.w);
        }
    }
    return {max((uint32_t)m2.x, (uint32_t)m2.y), min((uint32_t)n2.x, (uint32_t)n2.y)};
}

constexpr int kPrepChunk = 32;                   // groups per converting workgroup

template <bool PAD>
__global__ __launch_bounds__(256) void h16_prep_kernel(const uint8_t* __restrict__ xq,
                                                       const uint16_t* __restrict__ xs,
                                                       uint8_t* __restrict__ a16, int* __restrict__ ea,
                                                       const uint8_t* __restrict__ wq,
                                                       const uint16_t* __restrict__ ws, int* __restrict__ eb,
                                                       int M, int N, int G, int groups_per_split, int mblocks,
                                                       int nblocks, int chunks, int na) {
    const int tid = threadIdx.x;
    const int r = tid >> 3, part = tid & 7;
    const bool wside = (int)blockIdx.x >= na;
    const int id = wside ? blockIdx.x - na : blockIdx.x;
    const int blk = id % (wside ? nblocks : mblocks);
    const int rest = id / (wside ? nblocks : mblocks);
    const int chunk = wside ? 0 : rest % chunks;
    const int slice = wside ? rest : rest / chunks;
    const int sg0 = slice * groups_per_split, sg1 = min(G, sg0 + groups_per_split);
    const int row = blk * 32 + r;
    const bool ok = row < (wside ? N : M);
    const uint16_t* s = (wside ? ws : xs) + (size_t)row * G;
    const uint8_t* q = (wside ? wq : xq) + (size_t)row * G * 16;
    ScaleRange sr = {0x3f80u, 0xffffu};
    if (ok) sr = slice_scale_range<PAD>(s + sg0, sg1 - sg0, part);
#pragma unroll
    for (int x = 1; x <= 4; x *= 2) {
        sr.mx = max(sr.mx, (uint32_t)__shfl_xor((int)sr.mx, x));
        sr.mn = min(sr.mn, (uint32_t)__shfl_xor((int)sr.mn, x));
    }
    const int e = h16_shift(sr.mx);
    if (wside || chunk == 0) {
        int code = !ok ? 0 : e == kH16NonFinite ? (wside ? kH16NonFinite : 0) : -e;
        if (e != kH16NonFinite && sr.mn != 0xffffu && h16_loses_bits(sr.mn + 1, sr.mx)) {
            // a scale too small for the row's shift: wide unless its codes are 0
            int wide = 0;
            for (int g = sg0 + part; g < sg1; g += 8) {
                const uint32_t bits = s[g] & 0x7fffu;
                if (bits == 0 || !h16_loses_bits(bits, sr.mx)) continue;
                const uint4 w = *reinterpret_cast<const uint4*>(q + (size_t)g * 16);
                if ((w.x | w.y | w.z | w.w) != 0) wide = 1;
            }
#pragma unroll
            for (int x = 1; x <= 4; x *= 2) wide |= __shfl_xor(wide, x);
            if (wide) code = kH16Wide;
        }
        if (part == 0) {
            if (wside) eb[(size_t)slice * (nblocks * 32) + row] = code;
            else ea[(size_t)slice * (mblocks * 32) + row] = code;
        }
    }
    if (wside) return;
    const int GP = PAD ? (G + 7) & ~7 : G;
    uint8_t* dst = a16 + (size_t)(blk >> 3) * GP * kH16qStage + (blk & 7) * 2048 + (r >> 4) * 1024 + (r & 15) * 16;
    const int g1 = min(min(GP, sg0 + groups_per_split), sg0 + (chunk + 1) * kPrepChunk);
#pragma unroll 4
    for (int g = sg0 + chunk * kPrepChunk + part; g < g1; g += 8) {
        uint4 w = {0, 0, 0, 0};
        float f = 0.0f;
        if (ok && (!PAD || g < G)) {
            w = *reinterpret_cast<const uint4*>(q + (size_t)g * 16);
            f = __uint_as_float((uint32_t)s[g] << 16);
        }
        if (e == kH16NonFinite) f = __builtin_nanf("");
        const h2 sc = h16_scale(f, e);
        uint8_t* d = dst + (size_t)(g & ~3) * kH16qStage + (g & 3) * 256;
        *reinterpret_cast<uint4*>(d) = h16_codes(w.x, sc);
        *reinterpret_cast<uint4*>(d + kH16qStage) = h16_codes(w.y, sc);
        *reinterpret_cast<uint4*>(d + 2 * kH16qStage) = h16_codes(w.z, sc);
        *reinterpret_cast<uint4*>(d + 3 * kH16qStage) = h16_codes(w.w, sc);
    }
}

}  // namespace

size_t gemm_h16a_workspace_bytes(int64_t M, int64_t N, int64_t K, int splits) {
    const int64_t mpad = (M + kH16Tile - 1) / kH16Tile * kH16Tile;
    const int64_t npad = (N + kH16Tile - 1) / kH16Tile * kH16Tile;
    return (size_t)mpad * (size_t)((K + 255) / 256 * 256) * 2 + (size_t)splits * (size_t)(mpad + npad) * sizeof(int);
}

int launch_gemm_h16a(const uint8_t* xq, const uint16_t* xs, const uint8_t* wq, const uint16_t* ws,
                     uint16_t* y, float* partial, int M, int N, int K, int splits, int groups_per_split,
                     void* a_ws, int tile_rows, hipStream_t stream) {
    const int G = K >> 5;
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || splits < 1 || groups_per_split <= 0 ||
        groups_per_split % 8 != 0 || (long long)splits * groups_per_split < G ||
        (tile_rows != 64 && tile_rows != 128 && tile_rows != 256) ||
        (long long)(splits - 1) * groups_per_split >= G || (splits > 1 && partial == nullptr) || a_ws == nullptr ||
        ((reinterpret_cast<uintptr_t>(xs) | reinterpret_cast<uintptr_t>(ws) | reinterpret_cast<uintptr_t>(a_ws)) &
         15u) != 0)
        return (int)hipErrorInvalidValue;
    const int mpad = (M + kH16Tile - 1) / kH16Tile * kH16Tile;
    const int npad = (N + kH16Tile - 1) / kH16Tile * kH16Tile;
    uint8_t* a16 = static_cast<uint8_t*>(a_ws);
    const bool pad = G % 8 != 0;
    int* ea = reinterpret_cast<int*>(a16 + (size_t)mpad * ((K + 255) / 256 * 256) * 2);
    int* eb = ea + (size_t)splits * mpad;
    const int mblocks = mpad / 32, nblocks = npad / 32;
    const int chunks = (groups_per_split + kPrepChunk - 1) / kPrepChunk;
    const long long na = (long long)mblocks * splits * chunks, nprep = na + (long long)nblocks * splits;
    const long long tiles = (long long)((N + kH16Tile - 1) / kH16Tile) * ((M + tile_rows - 1) / tile_rows) * splits;
    if (nprep > 0x7fffffffLL || tiles > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const auto prep = pad ? h16_prep_kernel<true> : h16_prep_kernel<false>;
    prep<<<dim3((unsigned)nprep), 256, 0, stream>>>(xq, xs, a16, ea, wq, ws, eb, M, N, G, groups_per_split, mblocks, nblocks,
                                                    chunks, (int)na);
    const int e = (int)hipGetLastError();
    if (e != 0) return e;
    const auto kernel = tile_rows == 64    ? (pad ? gemm_h16q_kernel<4, true> : gemm_h16q_kernel<4, false>)
                        : tile_rows == 128 ? (pad ? gemm_h16q_kernel<8, true> : gemm_h16q_kernel<8, false>)
                                           : (pad ? gemm_h16q_kernel<16, true> : gemm_h16q_kernel<16, false>);
    kernel<<<dim3((unsigned)tiles), 256, 0, stream>>>(a16, ea, eb, wq, ws, y, partial, M, N, K, groups_per_split, xq,
                                                    xs);
    return (int)hipGetLastError();
}

}  // namespace wush
