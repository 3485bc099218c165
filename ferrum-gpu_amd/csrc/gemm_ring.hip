// The precise MFMA dequant-GEMM for products of some tens to some thousands of rows on resident Q8_0 /
// Q4_0 weights: y[M, N] = x[M, K] W^T (FH_PATH_TILED; the streaming kernel of gemm.hip takes the largest).
// Numerics and x order of the precise path (gemm.hip): x = hi + lo in f16, exact f16 integer quants, per
// 32 x 32 tile and block four v_mfma_f32_32x32x16_f16, then acc += d P.
//
// What bounds such a product is not the matrix cores but the latency of a K step: with a few hundred
// workgroups on the chip a stage of 32 k is 0.25 us of MFMAs per wavefront pair, a load from L2 or HBM
// takes 0.5 to 1 us, and one stage of lookahead through registers therefore ran at a quarter of the matrix
// cores' rate (512 x 2048 x 2560, Q4_0: 1.8 us a stage). So every operand goes from memory straight into
// LDS (buffer loads with an LDS destination, no registers) through a ring of NS stages (a stage's loads go out while
// the stage NS before it is computed).
//
// A workgroup is eight wavefronts on one CU: a 32 MTW x 128 tile, the blocks of K dealt to four pairs of
// wavefronts (each pair its own ring), whose sums meet in LDS in order at the end. So a few hundred tiles
// fill the chip without partial products in memory (the K splits of 128 x 128 tiles before wrote and
// read up to 64 MB for a 4 MB output). Where even then half the CUs would idle, K is split over two
// workgroups, which add into y (zeroed by the x split; two addends onto +0 give the same bits in either
// order) or leave two parts for the consumer. Where its sums would be longer chains than the tiled kernels' K splits
// make, a workgroup does K in phases or keeps totals (ring_plan).
//
// A wavefront owns 64 columns: their packed quants and scales are its own part of the ring and are unpacked
// in its registers, and the x rows (128 bytes per row and block) are shared by the pair. One barrier a
// stage: behind it the stage's x has landed for everybody (each wavefront first waits for its own
// loads, counted: loads complete in order) and the slot read in the stage before may be filled again.
//
// The f16 product (FH_PATH_TILED_F16) runs here too, with x in one part (64 bytes per row and block, two MFMAs
// per tile and block: 0.8 us a stage) and a row scale at the end.
//
// Measured (us, x split included, the 128 x 128 kernel and its reduction before / now, Q4_0): 512 rows 2048 x
// 2560 34.5 / 32.7 (in two phases, by ring_plan's rounding), 2048 x 2048 33.9 / 22.7, 2048 x 11264 98.8 / 67.2, 5632 x
// 2048 52.5 / 40.0; 200 rows 896 x 1152 22.5 / 12.3; 128 rows 2048 x 2560 28.8 / 14.7. GGUF rows (gemm_ext_kernel, one
// stage ahead through registers, before / now): FP8 2048 x 11264 300 rows 77 / 50, 1024 rows 181 / 144, 64 rows 30 /
// 23; MXFP4 69 / 47, 152 / 131, 31 / 21; F16 69 / 47, 167 / 133, 28 / 18.5; 5632 x 2048 300 rows 50 / 39, 46 / 34,
// 46 / 38. A stage takes 0.99 us, 1,085 TFLOP/s of matrix-core work on 256 CUs (a plain bf16 product reaches 1,210 on
// the card); what is left is a workgroup's own 6 us and the last round.
//
// LDS: x row r of a slot keeps its 16-byte chunk c at c ^ ((r >> 1) & 7) (gemm.hip: the sixteen rows that
// one cycle of a fragment read serves fall on sixteen different bank groups). Q8_0 quants are stored as
// [half block][column][16 bytes], Q4_0 as [column][16 bytes].
#include <algorithm>
#include <cmath>

#include "device_common.hpp"
#include "gemm_parts.hpp"
#include "internal.hpp"

namespace fh {
namespace {

// The other formats' weights are GGUF rows (a block's scale and quants together, at 34- or 17-byte steps from any
// byte; ds is null). A wavefront's part of a stage holds of each of its 64 columns the bytes from the block's
// start, rounded down to a dword, on:
//   FP8    [column][32 bytes], then [column][4]   F16 (a block is 64 codes' bytes, no scale) [column][64 bytes],
//   MXFP4  [column][32 bytes]                     16-byte chunk c of a column at c ^ (column / 4) % 4
// loaded 2 (F16: 4) lanes per column, since a load takes a cycle per cache line that it touches (a lane per column
// would take 64 a load, 192 cycles of a stage's 2400 for each of eight wavefronts). In registers a lane shifts its
// dwords to the byte with v_perm and the hardware converts the codes to f16, exactly.
// KG groups of wavefronts share K (4 pairs and a 128-column tile, or 2 fours and a 256-column tile).
template <int KIND, int MTW, int KG, int XP = 2>
struct Ring {
    static constexpr int WPG = 8 / KG, BN = 64 * WPG;  // wavefronts of a group
    static constexpr uint32_t QB = KIND == FH_F16 ? 64 : KIND == FH_Q4_0 ? 16 : 32;
    static constexpr uint32_t XB = 64 * XP;         // bytes of an x row and block
    static constexpr uint32_t X = 32 * MTW * XB;   // bytes of a group's stage: x,
    static constexpr uint32_t WQ = 64 * QB;        // a wavefront's quants
    static constexpr uint32_t D = KIND == FH_F16 || KIND == FH_MXFP4 ? 0 : 256;
    static constexpr uint32_t W = WQ + D;          // and its scale (FP8: last) dwords
    static constexpr uint32_t GROUP = X + WPG * W, STAGE = KG * GROUP;
    static constexpr int XL = X / 1024 / WPG;                        // x load instructions of a wavefront (1 KB each)
    static constexpr int LOADS = XL + WQ / 1024 + D / 256;  // load instructions per wavefront and stage
    static constexpr int NS = 163840 / STAGE < 6 ? 163840 / STAGE : 6;
    static constexpr uint32_t SUMS = 8 * MTW * 8192;  // the wavefronts' sums (after the loop)
    static constexpr uint32_t LDS = NS * STAGE > SUMS ? NS * STAGE : SUMS;
    static_assert(XL >= 1 && NS >= 3 && (NS - 1) * LOADS < 64 && LDS <= 163840, "ring size");
};

constexpr uint32_t kFlush = 8;

// Blocks st0 .. st1 - 1 of the tile at (m0, n0). ADD: its sums are added into y (two K splits onto zeros); else stored
// or (again) added to what this workgroup's last phase stored.
// XP: x parts, 2 (the precise product) or 1 (the f16 product: rows of x scaled to f16, output rows times rs).
template <int KIND, int MTW, int KG, bool ADD, bool PHASED, int XP>
__device__ __forceinline__ void ring_phase(uint8_t *arena, const _Float16 *__restrict__ xs, const uint8_t *__restrict__ qs,
                                           const uint16_t *__restrict__ ds, float *__restrict__ y, uint32_t M, uint32_t nb,
                                           uint32_t N, uint32_t m0, uint32_t n0, uint32_t st0, uint32_t st1, bool again,
                                           uint32_t wave, const float *__restrict__ rs) {
    using R = Ring<KIND, MTW, KG, XP>;
    constexpr int NS = R::NS;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t *)arena, nb8 = (nb + 7) / 8;
    uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));  // (a phase makes its own offsets: none is kept in registers through the stages)
    const uint32_t fr = lane % 32, hf = lane / 32;
    const uint32_t wn = wave % R::WPG, kg = wave / R::WPG;

    // Loads of block b into ring slot `slot`. Rows past M and columns past the padded weight rows fall past
    // their resource's end by their offsets alone and read 0; a block past the phase reads 0 through empty
    // resources (the count of loads in flight stays the same).
    constexpr uint32_t XR = 1024 / R::XB, XC = R::XB / 16;  // rows of an x instruction, 16-byte chunks of a row
    const uint32_t xrow = XR * R::XL * wn + lane / XC;      // instruction i: rows XR i further
    const uint32_t g0 = n0 / 32 + 2 * wn;            // the wavefront's first group of 32 columns
    const uint32_t xoff = (m0 + xrow) * nb * R::XB, ncol = n0 + 64 * wn + lane;
    const uint32_t woff = KIND == FH_Q8_0 ? g0 * nb * 1024 + (lane % 32) * 32 + (lane / 32) * 16
                                          : (g0 + lane / 32) * nb * 512 + (lane % 32) * 16;
    const uint32_t doff = (ncol >> 5) * nb8 * 512 + (ncol & 31) * 16;
    // GGUF rows: the byte offset of what the lane loads (row, chunk), 64 / GL columns an instruction, and of its FP8
    // last dword; columns past N read the last one (their outputs are dropped)
    constexpr int GI = kGguf<KIND> ? R::WQ / 1024 : 1, GL = KIND == FH_F16 ? 4 : 2;  // instructions, lanes a column
    constexpr uint32_t GB = kGgufBlock<KIND>;
    uint32_t grow[GI] = {}, grow4 = 0, gsh = 0;
    if constexpr (kGguf<KIND>) {
        const uint32_t chunk = KIND == FH_F16 ? lane % 4 ^ lane / 16 : lane % 2;  // (lane / 16 = column / 4 % 4)
#pragma unroll
        for (int i = 0; i < GI; i++)
            grow[i] = min(n0 + 64 * wn + 64 / GL * i + lane / GL, N - 1) * nb * GB + 16 * chunk;
        grow4 = min(ncol, N - 1) * nb * GB + 32;
        // the byte of block b's start in its first dword: (bits 16 j .. of gsh) + b GB, modulo 4
        gsh = (min(n0 + 64 * wn + fr, N - 1) * nb * GB & 3) | (min(n0 + 64 * wn + 32 + fr, N - 1) * nb * GB & 3) << 16;
    }
    auto xswap = [](uint32_t r) { return XP == 2 ? (r >> 1) & 7 : (r >> 2) & 3; };
    auto dma = [&](uint32_t b, uint32_t slot, int part) {  // part 0: weights and scales; 1: x
        const bool live = b < st1;
        const uint32_t x0 = lds0 + slot * R::STAGE + kg * R::GROUP, w0 = x0 + R::X + wn * R::W;
        if (part == 0 && kGguf<KIND>) {
            const i32x4 rq = sgpr_rsrc(qs, live ? N * nb * GB + 64 : 0u);  // (the allocation has 256 bytes past it)
#pragma unroll
            for (int i = 0; i < GI; i++)
                asm_load_lds16(rq, w0 + 1024 * i, (grow[i] + b * GB) & ~3u);
            if constexpr (kFp8<KIND>) asm_load_lds4(rq, w0 + R::WQ, (grow4 + b * GB) & ~3u);
            return;
        }
        if (part == 0) {
            const i32x4 rq = sgpr_rsrc(qs, live ? (N + 31) / 32 * 32 * nb * R::QB : 0u);
            const i32x4 rd = sgpr_rsrc(ds, live ? (N + 31) / 32 * 512 * nb8 : 0u);
            if constexpr (KIND == FH_Q8_0) {
                asm_load_lds16(rq, w0, woff + b * 1024);
                asm_load_lds16(rq, w0 + 1024, woff + (nb + b) * 1024);
            } else {
                asm_load_lds16(rq, w0, woff + b * 512);
            }
            asm_load_lds4(rd, w0 + R::WQ, doff + (b / 8) * 512 + (b % 8) / 2 * 4);
            return;
        }
        const i32x4 rx = sgpr_rsrc(xs, live ? M * nb * R::XB : 0u);
#pragma unroll
        for (int i = 0; i < R::XL; i++)
            asm_load_lds16(rx, x0 + 1024 * (R::XL * wn + i),
                           xoff + XR * i * nb * R::XB + b * R::XB + ((lane % XC) ^ xswap(xrow + XR * i)) * 16);
    };

    // The sums; those of 32-row tiles go into a total every kFlush blocks, an even number, (64-row tiles leave no registers for it).
    constexpr bool TOTALS = MTW == 1 && XP == 2;
    f32x16 acc[MTW][2], total[TOTALS ? MTW : 1][2];
#pragma unroll
    for (int i = 0; i < MTW; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = total[TOTALS ? i : 0][j][r] = 0.0f;

    // One stage's operands in registers: x fragments (hi and lo, k16 steps 0 and 1), the packed quants of the
    // lane's share of the two column tiles, their scale dwords (blocks b & ~1 and b | 1).
    struct Frag {
        f16x8 h[MTW][2], l[MTW][XP == 2 ? 2 : 1];
        u32x2 q[2][KIND == FH_Q8_0 ? 2 : 1];
        u32x4 g[2][2];  // GGUF rows: the lane's dwords
        uint32_t e[2], d[2];
    };
    auto read_w = [&](Frag &f, uint32_t slot) {
        const uint8_t *sw = arena + slot * R::STAGE + kg * R::GROUP + R::X + wn * R::W;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t c = j * 32 + fr;
            if constexpr (kFp8<KIND>) {  // dwords 4 half .. + 4: codes 16 half .. + 15
                f.g[j][0] = *(const u32x4 *)(sw + c * 32 + 16 * hf);
                f.e[j] = *(const uint32_t *)(sw + (hf ? R::WQ + c * 4 : c * 32 + 16));
                f.d[j] = *(const uint32_t *)(sw + c * 32);
                continue;
            }
            if constexpr (KIND == FH_MXFP4) {  // dwords 2 half .. + 2: bytes 8 half .. + 7 of the nibbles
                const u32x2 v = *(const u32x2 *)(sw + c * 32 + 8 * hf);
                f.g[j][0] = u32x4{v[0], v[1], *(const uint32_t *)(sw + c * 32 + 8 * hf + 8), 0u};
                f.d[j] = *(const uint32_t *)(sw + c * 32);
                continue;
            }
            if constexpr (KIND == FH_F16) {
#pragma unroll
                for (int s = 0; s < 2; s++) f.g[j][s] = *(const u32x4 *)(sw + c * 64 + ((2 * hf + s) ^ (fr / 4 % 4)) * 16);
                continue;
            }
            if constexpr (KIND == FH_Q8_0) {
#pragma unroll
                for (int s = 0; s < 2; s++) f.q[j][s] = *(const u32x2 *)(sw + j * 1024 + s * 512 + fr * 16 + 8 * hf);
            } else {  // dword 2 s + half: positions 16 s + 8 half ..
#pragma unroll
                for (int s = 0; s < 2; s++) f.q[j][0][s] = *(const uint32_t *)(sw + (j * 32 + fr) * 16 + 8 * s + 4 * hf);
            }
            f.d[j] = *(const uint32_t *)(sw + R::WQ + (j * 32 + fr) * 4);
        }
    };
    auto read_x = [&](Frag &f, uint32_t slot, int i) {
        const uint32_t r = i * 32 + fr;
        const uint8_t *row = arena + slot * R::STAGE + kg * R::GROUP + r * R::XB;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint32_t c = kGguf<KIND> ? 2 * hf + s : hf + 2 * s;  // (GGUF rows: a lane's codes are consecutive)
            f.h[i][s] = *(const f16x8 *)(row + (c ^ xswap(r)) * 16);
            if constexpr (XP == 2) f.l[i][s] = *(const f16x8 *)(row + ((4 + c) ^ xswap(r)) * 16);
        }
    };
    // Column tile j of block blk: exact f16 values; returns the block's scale. A block that holds an infinity or
    // NaN has a NaN scale (an E4M3 NaN makes its outputs NaN by itself): the split x would otherwise meet an
    // infinity with lo = 0 or of the other sign.
    auto unpack = [&](const Frag &f, int j, uint32_t blk, f16x8 (&b)[2]) {
        if constexpr (kFp8<KIND>) {
            const uint32_t sh = ((gsh >> (16 * j)) + blk * GB) & 2, sel = sh ? 0x07060504u : 0x05040302u;
            const u32x4 &w = f.g[j][0];
            uint32_t bad = 0;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                u32x4 o;
#pragma unroll
                for (int i = 0; i < 2; i++) {  // codes 8 s + 4 i .. + 3
                    const int at = 2 * s + i;
                    const uint32_t v = __builtin_amdgcn_perm(at == 3 ? f.e[j] : w[(at + 1) % 4], w[at], sel);
                    if constexpr (KIND == FH_FP8_E5M2) {  // the top byte of an f16
                        o[2 * i] = __builtin_amdgcn_perm(v, 0u, 0x050c040cu);
                        o[2 * i + 1] = __builtin_amdgcn_perm(v, 0u, 0x070c060cu);
                        bad |= ((v & 0x7c7c7c7cu) + 0x04040404u) & 0x80808080u;
                    } else {
                        o[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, false));
                        o[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, true));
                    }
                }
                b[s] = __builtin_bit_cast(f16x8, o);
            }
            const float d = half_to_float((sh ? f.d[j] >> 16 : f.d[j]) & 0xffffu);
            if constexpr (KIND == FH_FP8_E4M3) return d;
            const auto r = __builtin_amdgcn_permlane32_swap(bad, bad, false, false);  // (both halves of the block)
            return r[0] | r[1] ? __uint_as_float(0x7fc00000u) : d;
        } else if constexpr (KIND == FH_MXFP4) {  // (values times two, 0 .. 12; x order: byte i's two elements side by side)
            const uint32_t sh = ((gsh >> (16 * j)) + blk * GB) & 3, sel = 0x04030201u + 0x01010101u * sh;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const uint32_t v = __builtin_amdgcn_perm(f.g[j][0][s + 1], f.g[j][0][s], sel);
                b[s] = __builtin_bit_cast(
                    f16x8, u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 0)),
                                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 1)),
                                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 2)),
                                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 3))});
            }
            return e8m0_half_scale((f.d[j] >> (8 * sh)) & 0xffu);
        } else if constexpr (KIND == FH_F16) {
            uint32_t bad = 0;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                b[s] = __builtin_bit_cast(f16x8, f.g[j][s]);
#pragma unroll
                for (int c = 0; c < 4; c++) bad |= (f.g[j][s][c] & 0x7c007c00u) + 0x04000400u;
            }
            const auto r = __builtin_amdgcn_permlane32_swap(bad, bad, false, false);
            return (r[0] | r[1]) & 0x80008000u ? __uint_as_float(0x7fc00000u) : 1.0f;
        } else if constexpr (KIND == FH_Q8_0) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const u32x2 q = f.q[j][s] ^ 0x80808080u;
                b[s] = __builtin_bit_cast(
                    f16x8, u32x4{f16x2_add(__builtin_amdgcn_perm(0x64646464u, q[0], 0x04020400u), (_Float16)-1152.0f),
                                 f16x2_add(__builtin_amdgcn_perm(0x64646464u, q[0], 0x04030401u), (_Float16)-1152.0f),
                                 f16x2_add(__builtin_amdgcn_perm(0x64646464u, q[1], 0x04020400u), (_Float16)-1152.0f),
                                 f16x2_add(__builtin_amdgcn_perm(0x64646464u, q[1], 0x04030401u), (_Float16)-1152.0f)});
            }
        } else {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const uint32_t q = f.q[j][0][s];
                b[s] = __builtin_bit_cast(
                    f16x8, u32x4{f16x2_add((q & 0x000f000fu) | 0x64006400u, (_Float16)-1032.0f),
                                 f16x2_add(((q >> 8) & 0x000f000fu) | 0x64006400u, (_Float16)-1032.0f),
                                 f16x2_add(((q >> 4) & 0x000f000fu) | 0x64006400u, (_Float16)-1032.0f),
                                 f16x2_add(((q >> 12) & 0x000f000fu) | 0x64006400u, (_Float16)-1032.0f)});
            }
        }
        if constexpr (!kGguf<KIND>) return half_to_float(blk & 1 ? f.d[j] >> 16 : f.d[j] & 0xffffu);
    };
    // Block b (fragments f): tile v's MFMAs (a dependent chain), each followed by a share of tile v - 1's scale
    // FMAs, or, in the first tile, of the second column tile's unpacking. The stage's other work, the
    // next stage's LDS reads (from `after`) and the loads into `slot`, is issued among the MFMAs: in front of
    // them it held up both wavefronts of a SIMD while the matrix cores idled (1.08 us a stage; the MFMAs
    // alone 0.64).
    auto compute = [&](const Frag &f, Frag &nxt, uint32_t b, uint32_t slot, uint32_t after) {
        constexpr int V = 2 * MTW;
        f16x8 bq[2][2];
        float dq[2];
        dq[0] = unpack(f, 0, b, bq[0]);
        f32x16 pr[2];
#pragma unroll
        for (int v = 0; v <= V; v++) {
            const int j = v / MTW, i = v % MTW, vp = v - 1, jp = vp / MTW, ip = vp % MTW;
            f32x16 q = {};
            if (v == 0) {
                dq[1] = unpack(f, 1, b, bq[1]);
                read_w(nxt, after);
            }
            if (v == 1) read_x(nxt, after, 0);
            if (v == 2 && MTW == 2) read_x(nxt, after, MTW - 1);
            if (v == V - 1) dma(b + KG * NS, slot, 0);
            if (v == V) dma(b + KG * NS, slot, 1);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (v < V && s < 2 * XP)
                    q = __builtin_amdgcn_mfma_f32_32x32x16_f16(s < 2 ? f.h[i][s] : f.l[i][s - 2], bq[j][s % 2], q, 0, 0, 0);
                if (v > 0) {
#pragma unroll
                    for (int r = 4 * s; r < 4 * s + 4; r++) acc[ip][jp][r] = fmaf(dq[jp], pr[vp % 2][r], acc[ip][jp][r]);
                }
            }
            if (v < V) pr[v % 2] = q;
            if (v > 0) asm volatile("" : "+v"(acc[ip][jp]));  // the FMAs stay here
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (v < V && s < 2 * XP) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (v == 0)
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                else if (v < V)
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (v == 0)
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                else
                    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Stage p (four blocks, one a pair): its fragments were read during stage p - 1; behind the barrier stage
    // p + 1's loads have landed and are read while stage p's MFMAs run, and stage p + NS's go out into the
    // slot that stage p was read from.
    uint32_t slot = 0;
#pragma unroll
    for (int p = 0; p < NS; p++) {
        dma(st0 + KG * p + kg, p, 0);
        dma(st0 + KG * p + kg, p, 1);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * R::LOADS) : "memory");
    __syncthreads();
    Frag fa, fb;
    read_w(fa, 0);
#pragma unroll
    for (int i = 0; i < MTW; i++) read_x(fa, 0, i);
    auto stage = [&](const Frag &cur, Frag &nxt, uint32_t b) {
        const uint32_t after = slot + 1 == NS ? 0 : slot + 1;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * R::LOADS) : "memory");
        __syncthreads();
        compute(cur, nxt, b, slot, after);
        slot = after;
    };
    // (b0: the blocks of a total's next chain; without totals all of them)
    for (uint32_t b0 = st0, b1; b0 < st1; b0 = b1) {
        b1 = TOTALS ? min(st1, b0 + KG * kFlush) : st1;
        for (uint32_t b = b0 + kg; b < b1 + kg; b += 2 * KG) {  // (b - kg: uniform over the workgroup)
            stage(fa, fb, b);
            if (b - kg + KG >= b1) break;
            stage(fb, fa, b + KG);
        }
        if constexpr (TOTALS)
#pragma unroll
            for (int i = 0; i < MTW; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        total[i][j][r] += acc[i][j][r];
                        acc[i][j][r] = 0.0f;
                    }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the last loads, past the phase, write zeros into LDS)
    __syncthreads();
    // the groups' sums in order. D layout of a 32 x 32 tile: register r of lane l is row 8 (r / 4) +
    // 4 (l / 32) + r % 4, column l % 32
    float *sums = (float *)arena;  // [group][64 columns][tile i, j][register][lane]
    constexpr uint32_t PART = R::WPG * MTW * 2 * 16 * 64;
#pragma unroll
    for (int i = 0; i < MTW; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                sums[kg * PART + (((wn * MTW + i) * 2 + j) * 16 + r) * 64 + lane] =
                    TOTALS ? total[TOTALS ? i : 0][j][r] : acc[i][j][r];
    // output c of this thread: element (64 columns, i, j, register) c * 8 + wave of lane `lane`
    constexpr int OUT = 4 * MTW * R::WPG;
    auto place = [&](int c, uint32_t &row, uint32_t &col) {
        const uint32_t e = c * 8 + wave, r = e % 16, j = e / 16 % 2, i = e / 32 % MTW, h = e / (32 * MTW);
        row = m0 + i * 32 + 8 * (r / 4) + 4 * hf + r % 4;
        col = n0 + 64 * h + j * 32 + fr;
    };
    float last[OUT];  // what this thread stored in the phase before (all loads in flight together)
#pragma unroll
    for (int c = 0; c < OUT; c++) last[c] = 0.0f;
    if (PHASED && again) {
#pragma unroll
        for (int c = 0; c < OUT; c++) {
            uint32_t row, col;
            place(c, row, col);
            last[c] = y[(size_t)min(row, M - 1) * N + min(col, N - 1)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < OUT; c++) {
        const uint32_t e = c * 8 + wave;
        float v = sums[e * 64 + lane];
#pragma unroll
        for (int p = 1; p < KG; p++) v += sums[p * PART + e * 64 + lane];
        uint32_t row, col;
        place(c, row, col);
        if (row < M && col < N) {
            if constexpr (XP == 1) v *= rs[row];
            if (ADD)
                unsafeAtomicAdd(y + (size_t)row * N + col, v);
            else
                y[(size_t)row * N + col] = PHASED && again ? last[c] + v : v;
        }
    }
}

// A tile, split blockIdx.y of K (its sums at y + blockIdx.y M N, or ADD), in phases of `phase` blocks.
template <int KIND, int MTW, int KG, bool ADD, bool PHASED, int XP = 2>
__global__ __launch_bounds__(512, 2) void gemm_ring_kernel(const _Float16 *__restrict__ xs, const uint8_t *__restrict__ qs,
                                                           const uint16_t *__restrict__ ds, float *__restrict__ y,
                                                           uint32_t M, uint32_t K, uint32_t N, uint32_t mt, uint32_t nt,
                                                           uint32_t split_stages, uint32_t phase,
                                                           const float *__restrict__ rs) {
    using R = Ring<KIND, MTW, KG, XP>;
    __shared__ __attribute__((aligned(1024))) uint8_t arena[R::LDS];
    // XCD x (workgroups x, x + 8, ...) owns the x-th equal run of the tiles, column by column: its
    // workgroups share weight columns (read once from HBM) and x rows in its L2
    const uint32_t tiles = mt * nt, per_xcd = (tiles + 7) / 8, t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || t >= tiles) return;  // whole workgroup: no barrier is left waiting
    const uint32_t m0 = t % mt * 32 * MTW, n0 = t / mt * R::BN, nb = K / 32;
    const uint32_t st0 = blockIdx.y * split_stages, st1 = min(nb, st0 + split_stages);
    if (!ADD) y += (size_t)blockIdx.y * M * N;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    for (uint32_t p0 = st0;;) {
        const uint32_t p1 = PHASED ? min(st1, p0 + phase) : st1;
        ring_phase<KIND, MTW, KG, ADD, PHASED, XP>(arena, xs, qs, ds, y, M, nb, N, m0, n0, p0, p1, p0 != st0, wave, rs);
        if (!PHASED || (p0 = p1) >= st1) return;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores are out of the next phase's load counts,
        __syncthreads();                                  // and its loads may overwrite the sums
    }
}

}  // namespace

// The row tile, group count, K splits and phases of a product, and its time in us: rounds of a workgroup per CU, each
// its stages (64 rows: 0.99 us, measured 0.9 to 1.1; 32 rows: 0.5 us with few workgroups and 0.85 with one on
// every CU, for twice the weight loads and unpacking per row) and a workgroup's own cost (first loads and epilogue,
// 7 and 4 us). Two splits only where one leaves half of the CUs idle, at the cost of zeroing y and of two additions
// per output. GGUF rows cost a stage more by the factor f. (512 rows: 2048 x 2560 26 us with 128-column tiles, 42 with
// 256-column ones; 896 x 9728 at 300 rows 29 and 26. 32-row tiles where 64-row ones are few: Q8_0 5632 x 2048
// 128 rows 29 with 64-row tiles, 23 with 32-row ones; 2048 x 11264 128 rows 25 and 29.)
//
// Rounding. The variance of an output's relative error is 0.064 v + 0.58 in units of (1e-7)^2 (F16 0.80; fitted to 20
// products of 896 to 11008 inputs), v being the roundings of f32 sums in units of the last one: chains of l of nb
// equal addends give l / 2, n partial sums one after the other (n + 1) / 2 - 1 / n. The plan keeps v no larger than
// the K splits of the tiled kernels (gemm_sum_parts) make it: by more groups or splits, by 32-row tiles, whose chains
// are kFlush blocks, or with K in 2 to 4 phases of a workgroup, each added to the one before in y (6.5 us a turn: the
// sums' way through LDS, their stores and the first loads of a phase). Relative error (1e-7) and us of Q8_0, fastest
// plan / this one / 128 x 128 tiles: 3600 rows 3808 x 736 1.59 / 1.13 / 1.16 and 77 / 102 / 116; 300 rows 2048 x 11264
// 1.28 / 1.04 / 1.08 and 42 / 53 / 79; 975 rows 1344 x 3052 1.14 / 1.02 / 1.02 and 32 / 40 / 56; 512 rows 2048 x 2560
// 1.11 / 1.02 / 1.07 and 25 / 30 / 34; 975 rows 6912 x 1344 1.56 / 1.29 / 1.46 and 65 / 71 / 81.
struct RingPlan {
    uint32_t mtw, kg, splits, phases;
    float us;
};
static float added_in_turn(uint32_t n) { return (float)(n + 1) / 2 - 1 / (float)n; }
static float sum_roundings(size_t nb, uint32_t mtw, uint32_t kg, uint32_t outer) {
    kg = (uint32_t)std::min<size_t>(kg, nb);
    const float chain = (float)nb / (float)(kg * outer), flush = (float)kFlush;
    const float one = mtw == 1 && chain > flush ? (flush + chain / flush) / 2 : chain / 2;
    return one + added_in_turn(kg) + added_in_turn(outer);
}
static RingPlan ring_plan(int kind, size_t rows, size_t k, size_t n, bool close = true, int xp = 2) {
    const size_t nb = k / 32;
    rows = (rows + 31) / 32 * 32;  // (one plan for the rows of a 32-row tile)
    const float f = kind == FH_MXFP4 ? 1.15f : kind == FH_FP8_E4M3 || kind == FH_FP8_E5M2 ? 1.25f : xp == 1 ? 0.8f : 1.0f;
    const uint32_t parts = close ? gemm_sum_parts(kind, rows, k, n) : 1;
    const float most = close ? 1.02f * ((float)nb / (float)(2 * parts) + added_in_turn(parts)) + 0.17f : INFINITY;  // (+ 1%)
    RingPlan best{1, 4, 1, 1, INFINITY};
    for (uint32_t mtw : {2u, 1u})
        for (uint32_t kg : {4u, 2u})
            for (uint32_t sp : {1u, 2u}) {
                if (xp == 1 && mtw == 1 && kg == 2) continue;
                if (mtw == 2 && (rows <= 32 || (kind == FH_F16 && kg == 4))) continue;  // (that stage does not fit LDS three times)
                const uint64_t tiles = (rows + 32 * mtw - 1) / (32 * mtw) * ((n + 512 / kg - 1) / (512 / kg));
                if (sp == 2 && (tiles > 128 || nb < 4 * kg)) continue;
                uint32_t ph = 1;
                while (ph < 4 && sp == 1 && mtw == 2 && sum_roundings(nb, mtw, kg, ph) > most) ph++;
                if (sum_roundings(nb, mtw, kg, sp * ph) > most) continue;
                const float fk = kind == FH_F16 ? (mtw == 2 ? 1.15f : 0.97f) : f;
                const float stages = (float)((nb + sp * kg - 1) / (sp * kg)), turn = 6.5f * (float)(ph - 1);
                const float c32 = fk * (0.45f + 0.4f * std::min((float)(tiles * sp) / 256, 1.0f)), c64 = fk * 0.99f;
                const float us = (float)((tiles * sp + 255) / 256) * ((mtw == 2 ? c64 * stages + 7 : c32 * stages + 4) + turn) +
                                 (sp == 2 ? 1.5f + 3e-6f * (float)rows * (float)n : 0);
                if (us < best.us) best = RingPlan{mtw, kg, sp, ph, us};
            }
    // (two or three blocks: every plan has a rounding more than one chain, 1 to 2.6% of the error)
    return best.us < INFINITY ? best : ring_plan(kind, rows, k, n, false, xp);
}
uint32_t ring_splits(int kind, size_t rows, size_t k, size_t n, bool close) { return ring_plan(kind, rows, k, n, close).splits; }
float ring_us(int kind, size_t rows, size_t k, size_t n, bool close) { return ring_plan(kind, rows, k, n, close).us; }

bool ring_one_round(size_t rows, size_t k, size_t n, bool close) {
    const RingPlan p = ring_plan(FH_Q8_0, rows, k, n, close);
    return (rows + 32 * p.mtw - 1) / (32 * p.mtw) * ((n + 512 / p.kg - 1) / (512 / p.kg)) * p.splits <= 256;
}

bool ring_supported(size_t rows, size_t k, size_t n) {
    // every byte offset a workgroup forms (rows and columns up to the last tile's end) fits in 32 bits
    const size_t lim = (size_t)1 << 31;
    return (rows + 63) * k * 4 < lim && (n + 255) * (k / 32 + 8) * 32 < lim && (rows + 63) / 32 * ((n + 127) / 128) < (1u << 26);
}
bool ring_gguf_supported(int kind, size_t rows, size_t k, size_t n) {
    return kind != FH_Q2_K && ring_supported(rows, k, n) && n * (k / 32) * 64 + 128 < ((size_t)1 << 31);
}

template <int KIND, int MTW, int KG, int XP = 2>
static hipError_t run_ring(hipStream_t s, const _Float16 *xs, const uint8_t *qs, const uint16_t *ds, float *out, uint32_t M,
                           uint32_t K, uint32_t N, uint32_t sp, bool add, uint32_t phases, const float *rs = nullptr) {
    constexpr uint32_t BN = Ring<KIND, MTW, KG, XP>::BN;
    const uint32_t mt = (M + 32 * MTW - 1) / (32 * MTW), nt = (N + BN - 1) / BN, nb = K / 32;
    const dim3 grid((mt * nt + 7) / 8 * 8, sp);
    const uint32_t per = ((nb + sp - 1) / sp + KG - 1) / KG * KG, phase = ((per + phases - 1) / phases + KG - 1) / KG * KG;
    if (add)
        gemm_ring_kernel<KIND, MTW, KG, true, false, XP><<<grid, 512, 0, s>>>(xs, qs, ds, out, M, K, N, mt, nt, per, phase, rs);
    else if (MTW == 2 && XP == 2 && phases > 1)
        gemm_ring_kernel<KIND, MTW, KG, false, MTW == 2 && XP == 2, XP>
            <<<grid, 512, 0, s>>>(xs, qs, ds, out, M, K, N, mt, nt, per, phase, rs);
    else
        gemm_ring_kernel<KIND, MTW, KG, false, false, XP><<<grid, 512, 0, s>>>(xs, qs, ds, out, M, K, N, mt, nt, per, phase, rs);
    return hipGetLastError();
}

template <int KIND>
static hipError_t run_ring_kind(hipStream_t s, const _Float16 *xs, const uint8_t *qs, const uint16_t *ds, float *out,
                                uint32_t M, uint32_t K, uint32_t N, uint32_t sp, bool add, bool close) {
    const RingPlan p = ring_plan(KIND, M, K, N, close);
    if (p.mtw == 1)
        return p.kg == 4 ? run_ring<KIND, 1, 4>(s, xs, qs, ds, out, M, K, N, sp, add, p.phases)
                         : run_ring<KIND, 1, 2>(s, xs, qs, ds, out, M, K, N, sp, add, p.phases);
    if constexpr (KIND != FH_F16)
        if (p.kg == 4) return run_ring<KIND, 2, 4>(s, xs, qs, ds, out, M, K, N, sp, add, p.phases);
    return run_ring<KIND, 2, 2>(s, xs, qs, ds, out, M, K, N, sp, add, p.phases);
}

template <int KIND>
static hipError_t run_ring_f16(hipStream_t s, const _Float16 *xs, const float *rs, const uint8_t *qs, const uint16_t *ds,
                               float *out, uint32_t M, uint32_t K, uint32_t N) {
    const RingPlan p = ring_plan(KIND, M, K, N, false, 1);
    const bool add = p.splits > 1;
    if (p.mtw == 1) return run_ring<KIND, 1, 4, 1>(s, xs, qs, ds, out, M, K, N, p.splits, add, 1, rs);
    if (p.kg == 4) return run_ring<KIND, 2, 4, 1>(s, xs, qs, ds, out, M, K, N, p.splits, add, 1, rs);
    return run_ring<KIND, 2, 2, 1>(s, xs, qs, ds, out, M, K, N, p.splits, add, 1, rs);
}
float ring_f16_us(size_t rows, size_t k, size_t n) { return ring_plan(FH_Q8_0, rows, k, n, false, 1).us; }
uint32_t ring_f16_splits(size_t rows, size_t k, size_t n) { return ring_plan(FH_Q8_0, rows, k, n, false, 1).splits; }
hipError_t launch_gemm_ring_f16(hipStream_t s, int kind, const _Float16 *xs, const float *rs, const uint8_t *qs,
                                const uint16_t *ds, float *out, uint32_t M, uint32_t K, uint32_t N) {
    return kind == FH_Q8_0 ? run_ring_f16<FH_Q8_0>(s, xs, rs, qs, ds, out, M, K, N)
                           : run_ring_f16<FH_Q4_0>(s, xs, rs, qs, ds, out, M, K, N);
}

hipError_t launch_gemm_ring(hipStream_t s, int kind, const _Float16 *xs, const uint8_t *qs, const uint16_t *ds, float *out,
                            uint32_t M, uint32_t K, uint32_t N, uint32_t splits, bool add, bool close) {
    switch (kind) {
    case FH_Q8_0: return run_ring_kind<FH_Q8_0>(s, xs, qs, ds, out, M, K, N, splits, add, close);
    case FH_Q4_0: return run_ring_kind<FH_Q4_0>(s, xs, qs, ds, out, M, K, N, splits, add, close);
    case FH_F16: return run_ring_kind<FH_F16>(s, xs, qs, nullptr, out, M, K, N, splits, add, close);
    case FH_FP8_E4M3: return run_ring_kind<FH_FP8_E4M3>(s, xs, qs, nullptr, out, M, K, N, splits, add, close);
    case FH_FP8_E5M2: return run_ring_kind<FH_FP8_E5M2>(s, xs, qs, nullptr, out, M, K, N, splits, add, close);
    case FH_MXFP4: return run_ring_kind<FH_MXFP4>(s, xs, qs, nullptr, out, M, K, N, splits, add, close);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace fh
