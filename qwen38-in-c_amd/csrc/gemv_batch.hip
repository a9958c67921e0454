// gemv_batch.hip -- batched decode, more than eight tokens below the prefill
// GEMM: every weight byte is read once for up to 32 tokens, with the row-split
// decode GEMV's arithmetic (gemv_rows.hip) and, output for output, its bits.
//
// Replaces the token loop of qwen35-c/src/q35_mm.c:158-172 (q35_mm_fp8_batch)
// for 9..63 tokens of weights gemv_rows_shape() selects, and for any longer
// batch of a weight the prefill GEMM refuses.
//
// The row-split GEMV serves up to eight tokens a launch, so 24 tokens read
// the weights three times and 61 eight times, and every 32-row workgroup
// splits the activations of its K range again.  Here
//  - split_act_kernel splits the activations once, exactly, into three bf16
//    parts and writes them in MFMA A-operand order;
//  - a workgroup owns one K range (the NR = 4 or 8 ranges the row-split
//    GEMV's wavefronts have) of a 128-row group, four wavefronts with one
//    32-row sub-tile each, for a tile of T = 16 or 32 tokens.  It streams the
//    weights HBM -> registers and the split activations, shared by the four
//    wavefronts, into an LDS ring, both four stages ahead;
//  - tokens beyond one tile are further workgroups of the same launch, placed
//    so that those of one row group share an XCD's L2 (plain weight loads
//    then: 61 tokens of 5120 -> 14336 32.8 us against 38.9 non-temporal);
//  - the range sums (fp32) go to memory and batch_combine_kernel adds them in
//    range order, or, of an MLP's gate and up, batch_swiglu_kernel adds them
//    and writes silu(gate) * up already split for the down product.
//
// What bounds it: at 24 tokens (T = 32) gate and up of 5120 -> 2 x 17408
// (178 MB) take 50 us, 3.5 TB/s; HBM alone would take 30.  The CU's pipes are
// all busy half the time or more and overlap in part: per K block a SIMD's
// wavefront has 24 MFMAs (768 cycles), ~450 cycles of conversions and
// scaling, 24 LDS reads, and the CU copies 24 KiB of activations beside its
// 16 KiB of weights.  Ranges one after another in one workgroup instead (272
// workgroups for the same launch, no range sums) took 65.8 us: two chains on
// some CUs, one on the others.  Down (17408 -> 5120, 160 workgroups, 26 us)
// is bound by each wavefront's chain of 34 K blocks.
//
// Whole calls against the row-split GEMV in groups of eight, us: 5120 ->
// 16480 at 24 tokens 66.3 -> 36.6, at 63 tokens 176.9 -> 50.9; 17408 -> 5120
// 77.5 -> 38.0 and 207.8 -> 55.4.  (The runtime's batch_pays says from which
// sizes on it is taken.)
//
// Bits.  The decode GEMV sums each of its K ranges block by block (one fmaf
// with the block's scale per block and part), adds the three parts, then the
// ranges in order.  Every step is kept: MFMA A rows only select tokens and
// parts, so which rows they sit in does not change a sum.  (Wide values shift
// a K block for the eight tokens of their launch there, their eight here.)
#include <algorithm>
#include <type_traits>

#include "q35mm_device.h"
#include "q35mm_internal.h"

namespace q35mm {

namespace {

typedef __attribute__((address_space(3))) uint8_t lds_u8;

// A stage is 12 KiB of split activations: half a K block at 32 tokens, a
// whole one at 16.
constexpr uint32_t kRing = 4;        // stages of activations in LDS, of weights in registers
constexpr uint32_t kPieces = 3;      // 1 KiB activation copies per wavefront and stage
// Scale factors of a range, at most 4 per K block (32 tokens), 2 at 16
constexpr uint32_t kTabFloats = 4 * ((kGemvRsMaxKb + 3) / 4);

// Per K block: 8 MFMA steps (chunk j < 4, half q < 2), each an MFMA's A
// operand after another as its lanes read them (lane * 16: consecutive, or
// the two halves of a wavefront meet in the same LDS banks):
//   T = 32: one operand per part, rows = tokens
//   T = 16: parts 0 and 1 (rows 16 part + token), then part 2 (16 rows)
// part_off gives the place of (h = lane / 32, part, token) in a step.
template <uint32_t T>
struct BatchGeo {
    static constexpr uint32_t kStep = 3 * T * 2 * 16;
    static constexpr uint32_t kBlk = 8 * kStep;       // one K block
    static constexpr uint32_t kStages = T / 16;       // per K block
    static constexpr uint32_t kStage = kBlk / kStages;
    static constexpr uint32_t kChunks = 4 / kStages;  // 32-column chunks (1 KiB weight loads) per stage
    // MFMAs per step: 32 A rows hold one part of 32 tokens, or parts 0 and 1
    // of 16 tokens and, in a second MFMA, part 2
    static constexpr uint32_t kOps = T == 32 ? 3 : 2;
    static constexpr uint32_t kRegs = T / 2;          // token rows per lane and part
    static constexpr uint32_t kGroups = T / kGemvMaxM;   // of eight tokens, each shifted by itself
    static_assert(kStage == 4 * kPieces * kChunkBytes, "four wavefronts copy a stage");
    static __device__ __forceinline__ uint32_t part_off(uint32_t h, uint32_t part, uint32_t t) {
        if constexpr (T == 32) return part * 1024 + h * 512 + t * 16;
        return part < 2 ? h * 512 + part * 256 + t * 16 : 1024 + h * 256 + t * 16;
    }
};

// One wavefront copies 1 KiB to LDS: lane l's 16 bytes at base + soff + voff
// go to lds + 16 l.  A buffer load, not global_load_lds: the compiler takes
// the latter for a FLAT access that may complete out of order, and then
// waits for every load in flight before it uses a weight.
__device__ __forceinline__ void copy_1k(const uint8_t *base, uint32_t bytes, lds_u8 *l, uint32_t voff, uint32_t soff) {
    constexpr uint32_t kRaw32 = 0x00020000;   // resource word 3: raw 32-bit data, no swizzle
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, bytes, kRaw32), l, 16, voff, soff, 0, 0);
}

// s_waitcnt immediate: vmcnt <= n and lgkmcnt == 0 (gfx9 encoding, as in
// gemm_fp8.hip).
constexpr uint32_t wait_vm_lgkm0(uint32_t n) { return (n & 15u) | ((n >> 4) << 14) | (7u << 4); }

}  // namespace

// Eight columns of a token, split (shifted first if the block is wide), to
// the three parts' places in unit u of the K block at blk (columns 8u..8u+7).
template <uint32_t T>
__device__ __forceinline__ void store_split(uint8_t *blk, uint32_t u, uint32_t t, const float (&v)[8], bool wide) {
    using Geo = BatchGeo<T>;
    const uint32_t j = u >> 2, h = (u >> 1) & 1, q = u & 1;   // columns 32 j + 16 h + 8 q
    uint32_t p0[4], p1[4], p2[4];
#pragma unroll
    for (uint32_t e = 0; e < 4; e++) {
        if (__builtin_expect(wide, 0)) {
            split3_bf16x2(v[2 * e] * kActShift, v[2 * e + 1] * kActShift, p0[e], p1[e], p2[e]);
            split3_fix_inf(p0[e], p1[e], p2[e]);
        } else {
            split3_bf16x2(v[2 * e], v[2 * e + 1], p0[e], p1[e], p2[e]);
        }
    }
    uint8_t *const d = blk + (j * 2 + q) * Geo::kStep;
    *reinterpret_cast<u32x4_t *>(d + Geo::part_off(h, 0, t)) = u32x4_t{p0[0], p0[1], p0[2], p0[3]};
    *reinterpret_cast<u32x4_t *>(d + Geo::part_off(h, 1, t)) = u32x4_t{p1[0], p1[1], p1[2], p1[3]};
    *reinterpret_cast<u32x4_t *>(d + Geo::part_off(h, 2, t)) = u32x4_t{p2[0], p2[1], p2[2], p2[3]};
}

// Bit g: one of the workgroup's threads with tokens 8g..8g+7 of the tile (tt:
// a thread's token) holds a wide value.  The row-split GEMV shifts a K block
// for the eight tokens of a launch, so each eight here have a factor of
// their own: values below 2^-62 of the tile's other tokens keep their bits.
template <uint32_t T>
__device__ __forceinline__ uint32_t wide_groups(bool wide, uint32_t tt) {
    __shared__ uint32_t found[T / 4];   // per wavefront
    uint32_t bits = 0;
#pragma unroll
    for (uint32_t g = 0; g < BatchGeo<T>::kGroups; g++)
        bits |= __builtin_amdgcn_ballot_w64(wide && tt / kGemvMaxM == g) != 0 ? 1u << g : 0u;
    if ((threadIdx.x & 63) == 0) found[threadIdx.x >> 6] = bits;
    __syncthreads();
    bits = 0;
#pragma unroll
    for (uint32_t w = 0; w < T / 4; w++) bits |= found[w];
    return bits;
}

// The scale factors of a tile's K block, its groups of eight tokens in order.
template <uint32_t T>
__device__ __forceinline__ void store_factors(float *__restrict__ xf, uint32_t groups) {
    constexpr uint32_t kG = BatchGeo<T>::kGroups;
    if (threadIdx.x < kG) xf[(size_t)blockIdx.x * kG + threadIdx.x] = groups >> threadIdx.x & 1 ? kActUnshift : 1.0f;
}

// X fp32 [m][ldx] -> split A operands (BatchGeo's layout per token tile and
// K block) and one scale factor per tile, K block and eight tokens: 1, or
// kActUnshift if they hold a wide value and were staged times kActShift.  Tokens past
// m and columns past k are zeros.  One workgroup per tile and K block; a
// thread splits eight columns of a token.
template <uint32_t T, bool VEC>
__global__ __launch_bounds__(16 * T) void split_act_kernel(const float *__restrict__ x, uint32_t ldx, uint32_t m,
                                                           uint32_t k, uint32_t kb_total, uint8_t *__restrict__ xs,
                                                           float *__restrict__ xf) {
    const uint32_t kb = blockIdx.x % kb_total, tile = blockIdx.x / kb_total;
    const uint32_t tt = threadIdx.x % T, u = threadIdx.x / T, t = tile * T + tt, c = kb * kBlock + u * 8;
    const float *row = x + (size_t)min(t, m - 1) * ldx;
    float v[8];
    if constexpr (VEC) {   // rows 16-byte aligned, k % 8 == 0
        const float4 a = *reinterpret_cast<const float4 *>(row + min(c, k - 8));
        const float4 b = *reinterpret_cast<const float4 *>(row + min(c, k - 8) + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 8; e++) v[e] = row[min(c + e, k - 1)];
    }
#pragma unroll
    for (uint32_t e = 0; e < 8; e++)
        if (t >= m || c + e >= k) v[e] = 0.0f;
    const uint32_t groups = wide_groups<T>(max_abs(v) >= kActWide, tt);
    store_factors<T>(xf, groups);
    store_split<T>(xs + (size_t)blockIdx.x * BatchGeo<T>::kBlk, u, tt, v, groups >> tt / kGemvMaxM & 1);
}

// silu(gate) * up of the range sums of two weights (segments 0 and 1), split
// as split_act_kernel splits a stored product: the next weight's activations
// without its fp32 rows in between.  One workgroup per token tile and K block
// of the next weight, one thread per token and eight columns, columns fastest
// (the range sums, 8 x 4 bytes an output, outweigh the 6 written).
template <uint32_t T>
__global__ __launch_bounds__(16 * T) void batch_swiglu_kernel(BatchParams p, uint32_t kb_total, uint8_t *__restrict__ xs,
                                                              float *__restrict__ xf) {
    using Geo = BatchGeo<T>;
    constexpr uint32_t NR = kPairWaves;
    const uint32_t kb = blockIdx.x % kb_total, tile = blockIdx.x / kb_total;
    const uint32_t u = threadIdx.x & 15, tt = threadIdx.x >> 4, t = tile * T + tt, c = kb * kBlock + u * 8;
    const uint32_t rows = p.seg[0].rows;
    const size_t ld = (size_t)p.seg[0].nb * kBlock;
    float v[8] = {};
    if (t < p.m) {
        // every range's sums are loaded before the first is used: one memory
        // round trip, not one per range
        float4 w[2][NR][2];
#pragma unroll
        for (uint32_t z = 0; z < 2; z++) {
            const float *src = p.ws + p.seg[z].ws_off + (size_t)t * ld + c;   // rows padded to whole K blocks
#pragma unroll
            for (uint32_t r = 0; r < NR; r++)
#pragma unroll
                for (uint32_t i = 0; i < 2; i++)
                    w[z][r][i] = *reinterpret_cast<const float4 *>(src + (size_t)r * p.m * ld + 4 * i);
        }
        float sum[2][8];
#pragma unroll
        for (uint32_t z = 0; z < 2; z++)
#pragma unroll
            for (uint32_t r = 0; r < NR; r++)
#pragma unroll
                for (uint32_t i = 0; i < 2; i++) {
                    const float4 f = w[z][r][i];
                    const float q[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                    for (uint32_t e = 0; e < 4; e++) sum[z][4 * i + e] = r == 0 ? q[e] : sum[z][4 * i + e] + q[e];
                }
#pragma unroll
        for (uint32_t e = 0; e < 8; e++) v[e] = c + e < rows ? swiglu1(sum[0][e], sum[1][e]) : 0.0f;
    }
    const uint32_t groups = wide_groups<T>(max_abs(v) >= kActWide, tt);
    store_factors<T>(xf, groups);
    store_split<T>(xs + (size_t)blockIdx.x * Geo::kBlk, u, tt, v, groups >> tt / kGemvMaxM & 1);
}

// One K range of a 128-row group for T tokens: its sums to p.ws.
template <uint32_t T, bool STREAM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
void gemv_batch_kernel(BatchParams p) {
    using Geo = BatchGeo<T>;
    extern __shared__ __align__(16) uint8_t lds[];
    // block scales (times the shifted blocks' factor), after the ring.  One
    // LDS object: with two, the compiler drains every copy in flight (vmcnt
    // 0) before each operand read.
    float *const tab = reinterpret_cast<float *>(lds + kRing * Geo::kStage);

    // Workgroup b -> (item, token tile): the tiles of one item are 8
    // workgroups apart, i.e. on one XCD (workgroups go round-robin over 8).
    const uint32_t per = 8 * p.tiles;
    const uint32_t tile = (blockIdx.x % per) / 8, item = blockIdx.x / per * 8 + blockIdx.x % 8;
    if (item >= p.groups * p.nr) return;
    const uint32_t grp = item % p.groups, range = item / p.groups;

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // 32-row sub-tile
    uint32_t si = 0;
#pragma unroll
    for (uint32_t i = 1; i < 4; i++)
        if (i < p.nseg && grp >= p.seg[i].cta_begin) si = i;
    const GemvSeg &sg = p.seg[si];
    const uint32_t KB = p.kb, NR = p.nr;
    const uint32_t rg = grp - sg.cta_begin;   // 128-row group of the segment
    const uint32_t k0 = range * KB / NR, n = (range + 1) * KB / NR - k0;

    // ---- block scales, loaded before the stream so that waiting for them
    // waits for nothing else ----
    // (thread i: K block i / kG, tokens 8 (i % kG) on)
    constexpr uint32_t kG = Geo::kGroups;
    const uint32_t kbl = k0 + min(threadIdx.x / kG, n - 1);
    const float sc = sg.scale[(size_t)rg * KB + kbl] * p.xf[((size_t)tile * KB + kbl) * kG + threadIdx.x % kG];

    // ---- weight and activation streams: stage s is issued, activations
    // first, at the end of stage s - 4 and waited for at the end of stage
    // s - 1.  Loads are unconditional (in a whole turn stages past the end
    // read the last one again), so that wait is static: everything but the
    // two newest ----
    const uint32_t ns = n * Geo::kStages;
    const uint8_t *const codes = sg.codes + ((size_t)rg * KB + k0) * kBlockBytes + wv * kSubBytes + lane * 16;
    const uint8_t *const xsrc = p.xs + ((size_t)tile * KB + k0) * Geo::kBlk;
    const uint32_t xbytes = n * Geo::kBlk;
    const uint32_t xoff = wv * (kPieces * kChunkBytes);
    lds_u8 *const ring = (lds_u8 *)lds + xoff;
    u32x4_t wbuf[kRing][Geo::kChunks];
    auto issue = [&](uint32_t slot, uint32_t s) {
        const uint32_t st = min(s, ns - 1);
#pragma unroll
        for (uint32_t i = 0; i < kPieces; i++)
            copy_1k(xsrc, xbytes, ring + slot * Geo::kStage + i * kChunkBytes, lane * 16,
                    st * Geo::kStage + xoff + i * kChunkBytes);
        const uint8_t *src = codes + (size_t)(st / Geo::kStages) * kBlockBytes +
                             (st % Geo::kStages) * (Geo::kChunks * kChunkBytes);
#pragma unroll
        for (uint32_t j = 0; j < Geo::kChunks; j++)
            if constexpr (STREAM)
                wbuf[slot][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(src + j * kChunkBytes));
            else
                wbuf[slot][j] = *reinterpret_cast<const u32x4_t *>(src + j * kChunkBytes);
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t d = 0; d < kRing; d++) {
        issue(d, d);
        // stage by stage, as the waits count them (left to the compiler, two
        // weight loads of stage 0 went last, and every turn drained the ring)
        __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(kTabFloats <= 256, "one thread per factor");
    if (threadIdx.x < n * kG) tab[threadIdx.x] = sc;

    const uint32_t hh = lane >> 5, mrow = lane & 31;
    const uint32_t a0 = lane * 16, a1 = 1024 + (T == 32 ? lane * 16 : hh * 256 + (mrow & 15) * 16);

    // Software pipeline of one wavefront.  The MFMAs of step i (its operands
    // and its bf16 weights in registers) run with, beside each of them, the
    // LDS read of one operand and two of the conversions of step i + 1 and
    // the scaling of two or three sums of the previous K block (part is
    // double): left in one piece after the block's last MFMA, the scaling
    // and the first reads of a stage cost a lone wavefront half its time.
    constexpr uint32_t kSteps = 2 * Geo::kChunks;              // per stage
    constexpr uint32_t kSlots = 8 * Geo::kOps;                 // MFMAs per K block
    constexpr uint32_t kSums = T == 32 ? 48 : 24;              // acc[e / 16][e % 16], e < kSums
    f32x16_t acc[Geo::kOps] = {}, part[2][Geo::kOps] = {};
    const f32x16_t zero = {};
    u32x4_t aop[2][Geo::kOps], bop[2];
    typedef float scale_t __attribute__((ext_vector_type(kG)));   // of a K block, per eight tokens
    scale_t sc_prev = 0.0f, sc_cur = 0.0f;
    // sum x is of rows 8 (x / 4) + 0..7 of an operand, which are tokens 8 ((x / 4) % kG) + 0..7
    auto group = [](uint32_t x) { return x / 4 % kG; };
    auto read_a = [&](uint32_t slot, uint32_t i, uint32_t o) {
        aop[i & 1][o] = *reinterpret_cast<const u32x4_t *>(lds + slot * Geo::kStage + i * Geo::kStep +
                                                           (o == 0 ? a0 : a1 + (o - 1) * 1024));
    };
    auto cvt_b = [&](uint32_t slot, uint32_t i, uint32_t w) {   // dword w (0, 1) of step i's weights: two conversions
        const uint32_t c = wbuf[slot][i / 2][2 * (i % 2) + w];
        bop[i & 1][2 * w] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c, 1.0f, false));
        bop[i & 1][2 * w + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(c, 1.0f, true));
    };
    constexpr uint32_t kStageLoads = kPieces + Geo::kChunks;
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((kRing - 1) * kStageLoads));
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (uint32_t o = 0; o < Geo::kOps; o++) read_a(0, 0, o);
    cvt_b(0, 0, 0);
    cvt_b(0, 0, 1);
    // Stage s of the range, in ring slot d = s % kRing; tail >= 0: step tail
    // of the last, part turn, which issues nothing.
    auto step = [&](auto dc, uint32_t s, auto tc) {
        constexpr uint32_t d = decltype(dc)::value, dn = (d + 1) % kRing;
        constexpr int tail = decltype(tc)::value;
        constexpr uint32_t blk = d / Geo::kStages % 2;   // the K block's half of part
        if constexpr (d % Geo::kStages == 0) {
            sc_prev = sc_cur;
            sc_cur = reinterpret_cast<const scale_t *>(tab)[s / Geo::kStages];
        }
#pragma unroll
        for (uint32_t i = 0; i < kSteps; i++) {
            if (i == kSteps - 1) {
                // this wavefront has read all of stage s, whose slot the
                // copies take, and stage s+1 has landed; then all have.
                // (Without an issue each step leaves one stage fewer in
                // flight: loads nobody uses would not be there to count.)
                __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((kRing - 2 - (tail < 0 ? 0 : tail)) * kStageLoads));
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (tail < 0) issue(d, s + kRing);
            }
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t ns_slot = i == kSteps - 1 ? dn : d, ni = (i + 1) % kSteps;
#pragma unroll
            for (uint32_t o = 0; o < Geo::kOps; o++) {
                part[blk][o] = mfma32x32x16(__builtin_bit_cast(bf16x8_t, aop[i & 1][o]),
                                            __builtin_bit_cast(bf16x8_t, bop[i & 1]),
                                            d % Geo::kStages == 0 && i == 0 ? zero : part[blk][o]);
                read_a(ns_slot, ni, o);
                if (o < 2) cvt_b(ns_slot, ni, o);
                const uint32_t k = ((d % Geo::kStages) * kSteps + i) * Geo::kOps + o;
#pragma unroll
                for (uint32_t x = k * kSums / kSlots; x < (k + 1) * kSums / kSlots; x++)
                    acc[x / 16][x % 16] = __builtin_fmaf(sc_prev[group(x)], part[blk ^ 1][x / 16][x % 16], acc[x / 16][x % 16]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Whole turns of the ring without an exit inside, then the rest: a way
    // out of the middle of a turn would, to the compiler's count of loads in
    // flight, also lead back to its start, and each turn would wait for the
    // newest weights.
    using std::integral_constant;
    const integral_constant<uint32_t, 0> d0;
    const integral_constant<uint32_t, 1> d1;
    const integral_constant<uint32_t, 2> d2;
    const integral_constant<uint32_t, 3> d3;
    const integral_constant<int, -1> turn;
    uint32_t s = 0;
    for (; s + kRing <= ns; s += kRing) {
        step(d0, s, turn);
        step(d1, s + 1, turn);
        step(d2, s + 2, turn);
        step(d3, s + 3, turn);
    }
    static_assert(kRing == 4, "steps of a turn");
    if (s < ns) step(d0, s, integral_constant<int, 0>{});
    if (s + 1 < ns) step(d1, s + 1, integral_constant<int, 1>{});
    if constexpr (Geo::kStages == 1)
        if (s + 2 < ns) step(d2, s + 2, integral_constant<int, 2>{});
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));   // no copy outlives the loop
#pragma unroll
    for (uint32_t x = 0; x < kSums; x++) {   // the last K block's sums
        const float v = n & 1 ? part[0][x / 16][x % 16] : part[1][x / 16][x % 16];
        acc[x / 16][x % 16] = __builtin_fmaf(sc_cur[group(x)], v, acc[x / 16][x % 16]);
    }

    // per token row: (part 0 + part 1) + part 2
    const size_t ld = (size_t)sg.nb * kBlock;
    float *dst = p.ws + sg.ws_off + (size_t)range * p.m * ld + rg * kBlock + wv * kSubRows + mrow;
#pragma unroll
    for (uint32_t r = 0; r < Geo::kRegs; r++) {
        const uint32_t t = tile * T + 8 * (r >> 2) + 4 * hh + (r & 3);
        const float v = T == 32 ? (acc[0][r] + acc[1][r]) + acc[Geo::kOps - 1][r]
                                : (acc[0][r] + acc[0][(r + 8) & 15]) + acc[1][r];
        if (t < p.m) dst[(size_t)t * ld] = v;
    }
}

// y = (resid +) the range sums of one segment, added in range order.
template <uint32_t NR>
__global__ __launch_bounds__(256) void batch_combine_kernel(BatchParams p) {
    const GemvSeg &sg = p.seg[blockIdx.z];
    const uint32_t row = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (row >= sg.rows) return;
    const size_t ld = (size_t)sg.nb * kBlock, o = (size_t)t * sg.ldy + row;
    const float *src = p.ws + sg.ws_off + (size_t)t * ld + row;
    float v[NR];
#pragma unroll
    for (uint32_t r = 0; r < NR; r++) v[r] = src[(size_t)r * p.m * ld];
    const float x = sg.resid ? sg.resid[o] : 0.0f;
    float sum = v[0];
#pragma unroll
    for (uint32_t r = 1; r < NR; r++) sum += v[r];
    sg.y[o] = sg.resid ? x + sum : sum;
}

uint32_t batch_tile(uint32_t m) { return m <= 16 ? 16 : 32; }

size_t batch_act_bytes(uint32_t m, uint32_t kb) {
    return (size_t)((m + 31) / 32) * kb * BatchGeo<32>::kBlk;
}

size_t batch_xf_floats(uint32_t m, uint32_t kb) { return (size_t)((m + 31) / 32) * kb * BatchGeo<32>::kGroups; }

size_t batch_ws_floats(uint32_t m, uint32_t nb, uint32_t nr) { return (size_t)nr * m * nb * kBlock; }

hipError_t launch_split_act(const float *x, uint32_t ldx, uint32_t m, uint32_t k, uint32_t kb, bool vec, uint32_t T,
                            uint8_t *xs, float *xf, hipStream_t stream) {
    if (m == 0 || k == 0 || kb != (k + kBlock - 1) / kBlock || (vec && k % 8 != 0) || (T != 16 && T != 32))
        return hipErrorInvalidValue;
    const dim3 grid((m + T - 1) / T * kb), block(16 * T);
    if (T == 16)
        hipLaunchKernelGGL((vec ? split_act_kernel<16, true> : split_act_kernel<16, false>), grid, block, 0, stream, x,
                           ldx, m, k, kb, xs, xf);
    else
        hipLaunchKernelGGL((vec ? split_act_kernel<32, true> : split_act_kernel<32, false>), grid, block, 0, stream, x,
                           ldx, m, k, kb, xs, xf);
    return hipGetLastError();
}

hipError_t launch_gemv_batch(const BatchParams &pin, bool combine, hipStream_t stream) {
    BatchParams p = pin;
    const uint32_t T = p.tile;
    if (p.m == 0 || p.nseg == 0 || p.nseg > 4 || (p.nr != 4 && p.nr != 8) ||
        !gemv_rows_shape(p.kb, p.nr) || (T != 16 && T != 32) || (T == 16 && p.m > T))
        return hipErrorInvalidValue;
    p.tiles = (p.m + T - 1) / T;
    p.groups = 0;
    uint32_t max_rows = 0;
    for (uint32_t s = 0; s < p.nseg; s++) {
        p.seg[s].cta_begin = p.groups;
        p.groups += p.seg[s].nb;
        max_rows = std::max(max_rows, p.seg[s].rows);
    }
    const dim3 grid((p.groups * p.nr + 7) / 8 * 8 * p.tiles);
    const uint32_t lds = kRing * BatchGeo<16>::kStage + kTabFloats * sizeof(float);
    static_assert(BatchGeo<16>::kStage == BatchGeo<32>::kStage, "one ring size");
    using Kernel = void (*)(BatchParams);
    const Kernel kernel = T == 16 ? gemv_batch_kernel<16, true>
                                  : p.tiles == 1 ? gemv_batch_kernel<32, true> : gemv_batch_kernel<32, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !combine) return e;
    hipLaunchKernelGGL((p.nr == 4 ? batch_combine_kernel<4> : batch_combine_kernel<8>),
                       dim3((max_rows + 255) / 256, p.m, p.nseg), dim3(256), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_batch_swiglu(const BatchParams &p, uint32_t kb, uint8_t *xs, float *xf, hipStream_t stream) {
    const GemvSeg &g = p.seg[0], &u = p.seg[1];
    if (p.m == 0 || p.nseg != 2 || g.rows != u.rows || g.nb != u.nb || kb != g.nb || (p.tile != 16 && p.tile != 32) ||
        p.nr != kPairWaves)
        return hipErrorInvalidValue;
    const uint32_t T = p.tile;
    const dim3 grid((p.m + T - 1) / T * kb);
    hipLaunchKernelGGL((T == 16 ? batch_swiglu_kernel<16> : batch_swiglu_kernel<32>), grid, dim3(16 * T), 0, stream, p, kb, xs, xf);
    return hipGetLastError();
}

}  // namespace q35mm
