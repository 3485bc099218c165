// The precise MFMA dequant-GEMM for products of some tens to some thousands of rows on resident Q8_0 /
// Q4_0 weights: y[M, N] = x[M, K] W^T (FH_PATH_TILED; the streaming kernel of gemm.hip takes the largest).
// Numerics and x order of the precise path (gemm.hip): x = hi + lo in f16, exact f16 integer quants, per
// 32 x 32 tile and block four v_mfma_f32_32x32x16_f16, then acc += d P.
//
// What bounds such a product is not the matrix cores but the latency of a K step: with a few hundred
// workgroups on the chip a stage of 32 k is 0.25 us of MFMAs per wavefront pair, a load from L2 or HBM
// takes 0.5 to 1 us, and one stage of lookahead through registers therefore ran at a quarter of the matrix
// cores' rate (512 x 2048 x 2560, Q4_0: 1.8 us a stage). So every operand goes from memory straight into
// LDS (buffer loads with an LDS destination, no registers) through a ring of NS stages, NS - 1 stages ahead.
//
// A workgroup is eight wavefronts on one CU: a 32 MTW x 128 tile, the blocks of K dealt to four pairs of
// wavefronts (each pair its own ring), whose sums meet in LDS in order at the end. So a few hundred tiles
// fill the chip without partial products in memory (the K splits of 128 x 128 tiles before wrote and
// read up to 64 MB for a 4 MB output). Where even then half the CUs would idle, K is split over two
// workgroups, which add into y (zeroed by the x split; two addends onto +0 give the same bits in either
// order) or leave two parts for the consumer.
//
// A wavefront owns 64 columns: their packed quants and scales are its own part of the ring and are unpacked
// in its registers, and the x rows (128 bytes per row and block) are shared by the pair. One barrier a
// stage: behind it the stage's x has landed for everybody (each wavefront first waits for its own
// loads, counted: loads complete in order) and the slot read in the stage before may be filled again.
//
// Measured (us, x split included, the 128 x 128 kernel and its reduction before / now, Q4_0): 512 rows 2048 x
// 2560 35.8 / 28.1, 2048 x 2048 34.5 / 26.2, 2048 x 11264 99.8 / 71.0, 5632 x 2048 54.4 / 41.9, 896 x 1152
// 28.0 / 15.3; 96 rows 2048 x 2560 27.2 / 16.2. A stage takes 0.99 us, 1,085 TFLOP/s of matrix-core work on
// 256 CUs (a plain bf16 product reaches 1,210 on the card); what is left is a workgroup's own 6 us and the
// last round.
//
// LDS: x row r of a slot keeps its 16-byte chunk c at c ^ ((r >> 1) & 7) (gemm.hip: the sixteen rows that
// one cycle of a fragment read serves fall on sixteen different bank groups). Q8_0 quants are stored as
// [half block][column][16 bytes], Q4_0 as [column][16 bytes].
#include <cmath>

#include "device_common.hpp"
#include "gemm_parts.hpp"
#include "internal.hpp"

namespace fh {
namespace {

// KG groups of wavefronts share K (4 pairs and a 128-column tile, or 2 fours and a 256-column tile).
template <int KIND, int MTW, int KG>
struct Ring {
    static constexpr int WPG = 8 / KG, BN = 64 * WPG;  // wavefronts of a group
    static constexpr uint32_t QB = KIND == FH_Q8_0 ? 32 : 16;
    static constexpr uint32_t X = 32 * MTW * 128;  // bytes of a group's stage: x,
    static constexpr uint32_t WQ = 64 * QB;        // a wavefront's quants
    static constexpr uint32_t W = WQ + 256;        // and its scale dwords
    static constexpr uint32_t GROUP = X + WPG * W, STAGE = KG * GROUP;
    static constexpr int XL = 4 * MTW / WPG;                         // x load instructions of a wavefront (1 KB each)
    static constexpr int LOADS = XL + (KIND == FH_Q8_0 ? 2 : 1) + 1;  // load instructions per wavefront and stage
    static constexpr int NS = 163840 / STAGE < 6 ? 163840 / STAGE : 6;
    static constexpr uint32_t SUMS = 8 * MTW * 8192;  // the wavefronts' sums (after the loop)
    static constexpr uint32_t LDS = NS * STAGE > SUMS ? NS * STAGE : SUMS;
    static_assert(NS >= 3 && (NS - 1) * LOADS < 64 && LDS <= 163840, "ring size");
};

// ADD: the workgroup's sums are added into y (two K splits onto zeros); else stored, split blockIdx.y at
// y + blockIdx.y M N.
template <int KIND, int MTW, int KG, bool ADD>
__global__ __launch_bounds__(512, 2) void gemm_ring_kernel(const _Float16 *__restrict__ xs, const uint8_t *__restrict__ qs,
                                                           const uint16_t *__restrict__ ds, float *__restrict__ y,
                                                           uint32_t M, uint32_t K, uint32_t N, uint32_t mt, uint32_t nt,
                                                           uint32_t split_stages) {
    using R = Ring<KIND, MTW, KG>;
    constexpr int BM = 32 * MTW, NS = R::NS;
    __shared__ __attribute__((aligned(1024))) uint8_t arena[R::LDS];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t *)arena;

    // XCD x (workgroups x, x + 8, ...) owns the x-th equal run of the tiles, column by column: its
    // workgroups share weight columns (read once from HBM) and x rows in its L2
    const uint32_t tiles = mt * nt, per_xcd = (tiles + 7) / 8, t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || t >= tiles) return;  // whole workgroup: no barrier is left waiting
    const uint32_t m0 = t % mt * BM, n0 = t / mt * R::BN;
    const uint32_t nb = K / 32, nb8 = (nb + 7) / 8;
    const uint32_t st0 = blockIdx.y * split_stages, st1 = min(nb, st0 + split_stages);
    if (!ADD) y += (size_t)blockIdx.y * M * N;

    const uint32_t tid = threadIdx.x, lane = tid % 64, fr = lane % 32, hf = lane / 32;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64), wn = wave % R::WPG, kg = wave / R::WPG;

    // Loads of block b into ring slot `slot`. Rows past M and columns past the padded weight rows fall past
    // their resource's end by their offsets alone and read 0; a block past the split reads 0 through empty
    // resources (the count of loads in flight stays the same).
    const uint32_t xrow = 8 * R::XL * wn + lane / 8;  // instruction i: rows 8 i further
    const uint32_t g0 = n0 / 32 + 2 * wn;            // the wavefront's first group of 32 columns
    const uint32_t xoff = (m0 + xrow) * nb * 128, ncol = n0 + 64 * wn + lane;
    const uint32_t woff = KIND == FH_Q8_0 ? g0 * nb * 1024 + (lane % 32) * 32 + (lane / 32) * 16
                                          : (g0 + lane / 32) * nb * 512 + (lane % 32) * 16;
    const uint32_t doff = (ncol >> 5) * nb8 * 512 + (ncol & 31) * 16;
    auto dma = [&](uint32_t b, uint32_t slot, int part) {  // part 0: weights and scales; 1: x
        const bool live = b < st1;
        const uint32_t x0 = lds0 + slot * R::STAGE + kg * R::GROUP, w0 = x0 + R::X + wn * R::W;
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
        const i32x4 rx = sgpr_rsrc(xs, live ? M * nb * 128 : 0u);
#pragma unroll
        for (int i = 0; i < R::XL; i++) {
            const uint32_t r = xrow + 8 * i;
            asm_load_lds16(rx, x0 + 8 * (R::XL * wn + i) * 128,
                           xoff + 8 * i * nb * 128 + b * 128 + ((lane % 8) ^ ((r >> 1) & 7)) * 16);
        }
    };

    f32x16 acc[MTW][2];
#pragma unroll
    for (int i = 0; i < MTW; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // One stage's operands in registers: x fragments (hi and lo, k16 steps 0 and 1), the packed quants of the
    // lane's share of the two column tiles, their scale dwords (blocks b & ~1 and b | 1).
    struct Frag {
        f16x8 h[MTW][2], l[MTW][2];
        u32x2 q[2][KIND == FH_Q8_0 ? 2 : 1];
        uint32_t d[2];
    };
    auto read_w = [&](Frag &f, uint32_t slot) {
        const uint8_t *sw = arena + slot * R::STAGE + kg * R::GROUP + R::X + wn * R::W;
#pragma unroll
        for (int j = 0; j < 2; j++) {
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
        const uint8_t *row = arena + slot * R::STAGE + kg * R::GROUP + r * 128;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            f.h[i][s] = *(const f16x8 *)(row + (((hf + 2 * s) ^ ((r >> 1) & 7)) * 16));
            f.l[i][s] = *(const f16x8 *)(row + (((4 + hf + 2 * s) ^ ((r >> 1) & 7)) * 16));
        }
    };
    auto unpack = [&](const Frag &f, int j, f16x8 (&b)[2]) {  // exact f16 integers
        if constexpr (KIND == FH_Q8_0) {
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
        unpack(f, 0, bq[0]);
#pragma unroll
        for (int j = 0; j < 2; j++) dq[j] = half_to_float(b & 1 ? f.d[j] >> 16 : f.d[j] & 0xffffu);
        f32x16 pr[2];
#pragma unroll
        for (int v = 0; v <= V; v++) {
            const int j = v / MTW, i = v % MTW, vp = v - 1, jp = vp / MTW, ip = vp % MTW;
            f32x16 q = {};
            if (v == 0) {
                unpack(f, 1, bq[1]);
                read_w(nxt, after);
            }
            if (v == 1) read_x(nxt, after, 0);
            if (v == 2 && MTW == 2) read_x(nxt, after, MTW - 1);
            if (v == V - 1) dma(b + KG * NS, slot, 0);
            if (v == V) dma(b + KG * NS, slot, 1);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (v < V)
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
                if (v < V) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
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
    for (uint32_t b = st0 + kg; b < st1 + kg; b += 2 * KG) {  // (b - kg: uniform over the workgroup)
        stage(fa, fb, b);
        if (b - kg + KG >= st1) break;
        stage(fb, fa, b + KG);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the last loads, past the split, write zeros into LDS)
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
            for (int r = 0; r < 16; r++) sums[kg * PART + (((wn * MTW + i) * 2 + j) * 16 + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4 * MTW * R::WPG; c++) {
        const uint32_t e = c * 8 + wave;  // (64 columns, i, j, register)
        const uint32_t r = e % 16, j = e / 16 % 2, i = e / 32 % MTW, h = e / (32 * MTW);
        float v = sums[e * 64 + lane];
#pragma unroll
        for (int p = 1; p < KG; p++) v += sums[p * PART + e * 64 + lane];
        const uint32_t row = m0 + i * 32 + 8 * (r / 4) + 4 * hf + r % 4, col = n0 + 64 * h + j * 32 + fr;
        if (row < M && col < N) {
            if (ADD)
                unsafeAtomicAdd(y + (size_t)row * N + col, v);
            else
                y[(size_t)row * N + col] = v;
        }
    }
}

}  // namespace

// The group count and K splits of a product, and its time in us: rounds of a workgroup per CU, each its stages
// (0.99 us; measured 0.9 to 1.1) and a workgroup's own cost (first loads and epilogue, 6 us). Two splits only
// where one leaves half of the CUs idle. (512 rows: 2048 x 2560 26 us with 128-column tiles, 42 with
// 256-column ones; 896 x 9728 at 300 rows 29 and 26.)
struct RingPlan {
    uint32_t kg, splits;
    float us;
};
static RingPlan ring_plan(size_t rows, size_t k, size_t n) {
    const size_t bm = rows <= 32 ? 32 : 64, mt = (rows + bm - 1) / bm, nb = k / 32;
    RingPlan best{4, 1, INFINITY};
    for (uint32_t kg : {4u, 2u})
        for (uint32_t sp : {1u, 2u}) {
            const uint64_t tiles = mt * ((n + 512 / kg - 1) / (512 / kg));
            if (sp == 2 && (tiles > 128 || nb < 4 * kg)) continue;
            const float us = (float)((tiles * sp + 255) / 256 * ((nb + sp * kg - 1) / (sp * kg) + 6) + (sp == 2 ? 2 : 0));
            if (us < best.us) best = RingPlan{kg, sp, us};
        }
    return best;
}
uint32_t ring_splits(size_t rows, size_t k, size_t n) { return ring_plan(rows, k, n).splits; }
float ring_us(size_t rows, size_t k, size_t n) { return ring_plan(rows, k, n).us; }

bool ring_supported(size_t rows, size_t k, size_t n) {
    // every byte offset a workgroup forms (rows and columns up to the last tile's end) fits in 32 bits
    const size_t lim = (size_t)1 << 31;
    return (rows + 63) * k * 4 < lim && (n + 255) * (k / 32 + 8) * 32 < lim && (rows + 63) / 32 * ((n + 127) / 128) < (1u << 26);
}

template <int KIND, int MTW, int KG>
static hipError_t run_ring(hipStream_t s, const _Float16 *xs, const uint8_t *qs, const uint16_t *ds, float *out, uint32_t M,
                           uint32_t K, uint32_t N, uint32_t sp, bool add) {
    constexpr uint32_t BN = Ring<KIND, MTW, KG>::BN;
    const uint32_t mt = (M + 32 * MTW - 1) / (32 * MTW), nt = (N + BN - 1) / BN, nb = K / 32;
    const dim3 grid((mt * nt + 7) / 8 * 8, sp);
    const uint32_t per = ((nb + sp - 1) / sp + KG - 1) / KG * KG;
    if (add)
        gemm_ring_kernel<KIND, MTW, KG, true><<<grid, 512, 0, s>>>(xs, qs, ds, out, M, K, N, mt, nt, per);
    else
        gemm_ring_kernel<KIND, MTW, KG, false><<<grid, 512, 0, s>>>(xs, qs, ds, out, M, K, N, mt, nt, per);
    return hipGetLastError();
}

template <int KIND>
static hipError_t run_ring_kind(hipStream_t s, const _Float16 *xs, const uint8_t *qs, const uint16_t *ds, float *out,
                                uint32_t M, uint32_t K, uint32_t N, uint32_t sp, bool add) {
    const uint32_t kg = ring_plan(M, K, N).kg;
    if (M <= 32)
        return kg == 4 ? run_ring<KIND, 1, 4>(s, xs, qs, ds, out, M, K, N, sp, add)
                       : run_ring<KIND, 1, 2>(s, xs, qs, ds, out, M, K, N, sp, add);
    return kg == 4 ? run_ring<KIND, 2, 4>(s, xs, qs, ds, out, M, K, N, sp, add)
                   : run_ring<KIND, 2, 2>(s, xs, qs, ds, out, M, K, N, sp, add);
}

hipError_t launch_gemm_ring(hipStream_t s, fh_kind kind, const _Float16 *xs, const uint8_t *qs, const uint16_t *ds,
                            float *out, uint32_t M, uint32_t K, uint32_t N, uint32_t splits, bool add) {
    return kind == FH_Q8_0 ? run_ring_kind<FH_Q8_0>(s, xs, qs, ds, out, M, K, N, splits, add)
                           : run_ring_kind<FH_Q4_0>(s, xs, qs, ds, out, M, K, N, splits, add);
}

}  // namespace fh
