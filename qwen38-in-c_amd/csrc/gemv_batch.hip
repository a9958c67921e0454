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
//  - a workgroup owns a 128-row group of one weight (four wavefronts, one
//    32-row sub-tile each) for a tile of T = 16 or 32 tokens.  It streams the
//    weights HBM -> registers two K blocks ahead and copies each K block's
//    split activations (12 or 24 KiB, shared by the four wavefronts) into a
//    three-deep LDS ring with global_load_lds.  Matrix work per weight byte
//    is what bounds it then: 24 MFMAs per 4 KiB sub-tile at T = 32 are 768
//    cycles of a SIMD's matrix core, which for a layer's 383 MB is 29 us at
//    32 tokens against 76 us of HBM traffic at 5 TB/s;
//  - tokens beyond one tile are further workgroups of the same launch, placed
//    so that the workgroups of one row group share an XCD's L2.
//
// Bits.  The decode GEMV sums each of its NR (4 or 8) K ranges block by block
// (one fmaf with the block's scale per block and part), adds the three parts,
// then the ranges in order.  Every step is kept: MFMA A rows only select
// tokens and parts, so which rows they sit in does not change a sum.
// Ranges either run one after another in one workgroup (SEQ) or as NR
// workgroups whose sums batch_combine_kernel adds in range order; the bits
// are the same.
#include <algorithm>
#include <type_traits>

#include "q35mm_device.h"
#include "q35mm_internal.h"

namespace q35mm {

namespace {

typedef __attribute__((address_space(3))) uint8_t lds_u8;

constexpr uint32_t kRing = 3;        // K blocks of activations in LDS, of weights in registers
constexpr uint32_t kWLoads = 4;      // 1 KiB weight loads per wavefront and K block

// Per K block: 8 MFMA steps (chunk j < 4, half q < 2) of 3 T rows x 2 x 16
// bytes: step (j, q), h = lane / 32, part, token at
// ((((j*2 + q) * 2 + h) * 3 + part) * T + token) * 16.
template <uint32_t T>
struct BatchGeo {
    static constexpr uint32_t kHalf = 48 * T;         // one h of a step
    static constexpr uint32_t kStep = 2 * kHalf;
    static constexpr uint32_t kStage = 8 * kStep;     // 12 or 24 KiB
    static constexpr uint32_t kPieces = kStage / kChunkBytes / 4;   // 1 KiB copies per wavefront
    // MFMAs per step: 32 A rows hold one part of 32 tokens, or parts 0 and 1
    // of 16 tokens and, in a second MFMA, part 2
    static constexpr uint32_t kOps = T == 32 ? 3 : 2;
    static constexpr uint32_t kRegs = T / 2;          // token rows per lane and part
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

// X fp32 [m][ldx] -> split A operands (BatchGeo's layout per token tile and
// K block) and one scale factor per tile and K block: 1, or kActUnshift for a
// block that holds a wide value and was staged times kActShift.  Tokens past
// m and columns past k are zeros.  One workgroup per tile and K block; a
// thread splits eight columns of a token.
template <uint32_t T, bool VEC>
__global__ __launch_bounds__(256) void split_act_kernel(const float *__restrict__ x, uint32_t ldx, uint32_t m,
                                                        uint32_t k, uint32_t kb_total, uint8_t *__restrict__ xs,
                                                        float *__restrict__ xf) {
    using Geo = BatchGeo<T>;
    constexpr uint32_t N = T * 16 / 256;
    const uint32_t kb = blockIdx.x % kb_total, tile = blockIdx.x / kb_total;
    float v[N][8];
#pragma unroll
    for (uint32_t i = 0; i < N; i++) {
        const uint32_t idx = threadIdx.x + 256 * i, t = tile * T + idx % T, c = kb * kBlock + (idx / T) * 8;
        const float *row = x + (size_t)min(t, m - 1) * ldx;
        if constexpr (VEC) {   // rows 16-byte aligned, k % 8 == 0
            const float4 a = *reinterpret_cast<const float4 *>(row + min(c, k - 8));
            const float4 b = *reinterpret_cast<const float4 *>(row + min(c, k - 8) + 4);
            v[i][0] = a.x; v[i][1] = a.y; v[i][2] = a.z; v[i][3] = a.w;
            v[i][4] = b.x; v[i][5] = b.y; v[i][6] = b.z; v[i][7] = b.w;
        } else {
#pragma unroll
            for (uint32_t e = 0; e < 8; e++) v[i][e] = row[min(c + e, k - 1)];
        }
#pragma unroll
        for (uint32_t e = 0; e < 8; e++)
            if (t >= m || c + e >= k) v[i][e] = 0.0f;
    }
    bool w = false;
#pragma unroll
    for (uint32_t i = 0; i < N; i++) w |= max_abs(v[i]) >= kActWide;
    const bool wide = __syncthreads_or(w) != 0;
    if (threadIdx.x == 0) xf[blockIdx.x] = wide ? kActUnshift : 1.0f;
    uint8_t *const base = xs + (size_t)blockIdx.x * Geo::kStage;
#pragma unroll
    for (uint32_t i = 0; i < N; i++) {
        const uint32_t idx = threadIdx.x + 256 * i, t = idx % T, u = idx / T;
        const uint32_t j = u >> 2, h = (u >> 1) & 1, q = u & 1;   // columns 32 j + 16 h + 8 q
        uint32_t p0[4], p1[4], p2[4];
#pragma unroll
        for (uint32_t e = 0; e < 4; e++) {
            if (__builtin_expect(wide, 0)) {
                split3_bf16x2(v[i][2 * e] * kActShift, v[i][2 * e + 1] * kActShift, p0[e], p1[e], p2[e]);
                split3_fix_inf(p0[e], p1[e], p2[e]);
            } else {
                split3_bf16x2(v[i][2 * e], v[i][2 * e + 1], p0[e], p1[e], p2[e]);
            }
        }
        u32x4_t *dst = reinterpret_cast<u32x4_t *>(base + (j * 2 + q) * Geo::kStep + h * Geo::kHalf + t * 16);
        dst[0] = u32x4_t{p0[0], p0[1], p0[2], p0[3]};
        dst[T] = u32x4_t{p1[0], p1[1], p1[2], p1[3]};
        dst[2 * T] = u32x4_t{p2[0], p2[1], p2[2], p2[3]};
    }
}

// T tokens per workgroup; SEQ: all K ranges in the workgroup, else one of
// them, its sums to p.ws; PAIR (SEQ only): 64 rows of gate (segment 0) and
// the same rows of up (segment 1), writing silu(gate) * up.
template <uint32_t T, bool SEQ, bool PAIR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(T == 16 ? 4 : 2, 8)))
void gemv_batch_kernel(BatchParams p) {
    static_assert(SEQ || !PAIR, "paired rows need whole sums");
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
    if (item >= p.items) return;
    const uint32_t grp = SEQ ? item : item % p.groups, range = SEQ ? 0 : item / p.groups;

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t si = 0;
    if constexpr (PAIR) {
        si = wv >> 1;
    } else {
#pragma unroll
        for (uint32_t i = 1; i < 4; i++)
            if (i < p.nseg && grp >= p.seg[i].cta_begin) si = i;
    }
    const GemvSeg &sg = p.seg[si];
    const uint32_t KB = p.kb, NR = p.nr;
    // this wavefront's 32-row sub-tile of the segment and its 128-row group
    const uint32_t sub = PAIR ? grp * 2 + (wv & 1) : (grp - sg.cta_begin) * 4 + wv;
    const uint32_t rg = sub >> 2;
    const uint32_t k0 = SEQ ? 0 : range * KB / NR, k1 = SEQ ? KB : (range + 1) * KB / NR, n = k1 - k0;

    // ---- block scales, loaded before the stream so that waiting for them
    // waits for nothing else ----
    constexpr uint32_t kTabs = PAIR ? 2 : 1;
    float sc[kTabs];
#pragma unroll
    for (uint32_t z = 0; z < kTabs; z++) {
        const GemvSeg &ss = PAIR ? p.seg[z] : sg;
        const uint32_t kb = k0 + min(threadIdx.x, n - 1);
        sc[z] = ss.scale[(size_t)rg * KB + kb] * p.xf[(size_t)tile * KB + kb];
    }

    // ---- weight and activation streams: K block s of the range is waited
    // for at step s and issued at step s - 2, activations first.  Loads are
    // unconditional (blocks past the end read the last one again), so the
    // wait before each step is static: everything but the next block's ----
    const uint8_t *const codes = sg.codes + ((size_t)rg * KB + k0) * kBlockBytes + (sub & 3) * kSubBytes + lane * 16;
    const uint8_t *const xsrc = p.xs + ((size_t)tile * KB + k0) * Geo::kStage;
    const uint32_t xbytes = n * Geo::kStage;
    const uint32_t xoff = wv * (Geo::kPieces * kChunkBytes);
    lds_u8 *const ring = (lds_u8 *)lds + wv * (Geo::kPieces * kChunkBytes);
    u32x4_t wbuf[kRing][kWLoads];
    auto issue = [&](uint32_t slot, uint32_t s) {
        const uint32_t kb = min(s, n - 1);
#pragma unroll
        for (uint32_t i = 0; i < Geo::kPieces; i++)
            copy_1k(xsrc, xbytes, ring + slot * Geo::kStage + i * kChunkBytes, lane * 16,
                    kb * Geo::kStage + xoff + i * kChunkBytes);
        const uint8_t *src = codes + (size_t)kb * kBlockBytes;
#pragma unroll
        for (uint32_t j = 0; j < kWLoads; j++)
            wbuf[slot][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(src + j * kChunkBytes));
    };
    __builtin_amdgcn_sched_barrier(0);
    issue(0, 0);
    issue(1, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t z = 0; z < kTabs; z++)
        if (threadIdx.x < n) tab[z * kGemvRsMaxKb + threadIdx.x] = sc[z];

    // This lane's A row: a part of a token (T = 32: token = row; T = 16: row
    // / 16 = part 0 or 1, the second MFMA's rows all part 2)
    const uint32_t hh = lane >> 5, mrow = lane & 31;
    const uint32_t a0 = hh * Geo::kHalf + mrow * 16;
    const uint32_t a1 = T == 32 ? a0 + 512 : hh * Geo::kHalf + 512 + (mrow & 15) * 16;
    const float *const mytab = tab + (PAIR ? si * kGemvRsMaxKb : 0);

    f32x16_t acc[Geo::kOps] = {};
    const f32x16_t zero = {};
    float tot[Geo::kRegs];
    // The sum of a finished range, per token row: (part 0 + part 1) + part 2
    auto range_sum = [&](uint32_t r) {
        if constexpr (T == 32)
            return (acc[0][r] + acc[1][r]) + acc[Geo::kOps - 1][r];
        else
            return (acc[0][r] + acc[0][r + 8]) + acc[1][r];
    };
    uint32_t rdone = 0, rend = KB / NR;   // SEQ: ranges finished, end of the current one

    auto step = [&](auto dc, uint32_t s) {   // K block s of the range, in ring slot d = s % kRing
        constexpr uint32_t d = decltype(dc)::value;
        // block s has landed and this wavefront has read all of block
        // s-1 (whose slot the copies below take); then the same for all
        __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(Geo::kPieces + kWLoads));
        __builtin_amdgcn_s_barrier();
        issue((d + 2) % kRing, s + 2);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t *const la = lds + d * Geo::kStage;
        f32x16_t part[Geo::kOps];
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
#pragma unroll
            for (uint32_t q = 0; q < 2; q++) {
                const bf16x8_t bop = e4m3x8_to_bf16x8_cvt(wbuf[d][j][2 * q], wbuf[d][j][2 * q + 1], 1.0f);
#pragma unroll
                for (uint32_t o = 0; o < Geo::kOps; o++) {
                    const uint32_t off = (j * 2 + q) * Geo::kStep + (o == 0 ? a0 : a1 + (o - 1) * 512);
                    const bf16x8_t aop =
                        __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t *>(la + off));
                    part[o] = mfma32x32x16(aop, bop, j == 0 && q == 0 ? zero : part[o]);
                }
            }
        const float scale = mytab[s];
#pragma unroll
        for (uint32_t o = 0; o < Geo::kOps; o++)
#pragma unroll
            for (uint32_t r = 0; r < (T == 16 && o == 1 ? 8u : 16u); r++)
                acc[o][r] = __builtin_fmaf(scale, part[o][r], acc[o][r]);
        if constexpr (SEQ) {
            if (s + 1 == rend) {
#pragma unroll
                for (uint32_t r = 0; r < Geo::kRegs; r++) {
                    const float v = range_sum(r);
                    tot[r] = rdone ? tot[r] + v : v;
                }
#pragma unroll
                for (uint32_t o = 0; o < Geo::kOps; o++) acc[o] = zero;
                rdone++;
                rend = (rdone + 1) * KB / NR;
            }
        }
    };
    // Whole turns of the ring without an exit inside, then the rest: a way
    // out of the middle of a turn would, to the compiler's count of loads in
    // flight, also lead back to its start, and each turn would wait for the
    // newest weights.
    using std::integral_constant;
    uint32_t b = 0;
    for (; b + kRing <= n; b += kRing) {
        step(integral_constant<uint32_t, 0>{}, b);
        step(integral_constant<uint32_t, 1>{}, b + 1);
        step(integral_constant<uint32_t, 2>{}, b + 2);
    }
    static_assert(kRing == 3, "steps of a turn");
    if (b < n) step(integral_constant<uint32_t, 0>{}, b);
    if (b + 1 < n) step(integral_constant<uint32_t, 1>{}, b + 1);
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));   // no copy outlives the loop

    const uint32_t col = sub * kSubRows + mrow;      // weight row
    auto token = [&](uint32_t r) { return tile * T + 8 * (r >> 2) + 4 * hh + (r & 3); };
    if constexpr (!SEQ) {
        float *dst = p.ws + sg.ws_off + (size_t)range * p.m * (sg.nb * kBlock) + col;
#pragma unroll
        for (uint32_t r = 0; r < Geo::kRegs; r++)
            if (token(r) < p.m) dst[(size_t)token(r) * (sg.nb * kBlock)] = range_sum(r);
    } else if constexpr (!PAIR) {
#pragma unroll
        for (uint32_t r = 0; r < Geo::kRegs; r++)
            if (token(r) < p.m && col < sg.rows) {
                const size_t o = (size_t)token(r) * sg.ldy + col;
                sg.y[o] = sg.resid ? sg.resid[o] + tot[r] : tot[r];
            }
    } else {
        // gate wavefront w and up wavefront w + 2 hold the same outputs:
        // each hands half of its token rows to the other through LDS and
        // forms silu(gate) * up of the other half
        constexpr uint32_t H = Geo::kRegs / 2;
        float *const xch = reinterpret_cast<float *>(lds);
        const bool up = wv >= 2;
        __builtin_amdgcn_s_barrier();   // every wavefront is done with the ring
#pragma unroll
        for (uint32_t r = 0; r < H; r++) xch[(wv * H + r) * 64 + lane] = up ? tot[r] : tot[r + H];
        __syncthreads();
#pragma unroll
        for (uint32_t r = 0; r < H; r++) {
            const float other = xch[((wv ^ 2) * H + r) * 64 + lane];
            const float mine = up ? tot[r + H] : tot[r];
            const uint32_t t = token(up ? r + H : r);
            if (t < p.m && col < sg.rows)
                p.seg[0].y[(size_t)t * sg.ldy + col] = swiglu1(up ? other : mine, up ? mine : other);
        }
    }
}

// y = (resid +) the range sums of one segment, added in range order.
__global__ __launch_bounds__(256) void batch_combine_kernel(BatchParams p) {
    const GemvSeg &sg = p.seg[blockIdx.z];
    const uint32_t row = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (row >= sg.rows) return;
    const size_t ld = (size_t)sg.nb * kBlock;
    const float *src = p.ws + sg.ws_off + (size_t)t * ld + row;
    float sum = src[0];
    for (uint32_t r = 1; r < p.nr; r++) sum += src[(size_t)r * p.m * ld];
    const size_t o = (size_t)t * sg.ldy + row;
    sg.y[o] = sg.resid ? sg.resid[o] + sum : sum;
}

uint32_t batch_tile(uint32_t m) { return m <= 16 ? 16 : 32; }

size_t batch_act_bytes(uint32_t m, uint32_t kb) {
    const uint32_t T = batch_tile(m);
    const size_t blocks = (size_t)((m + T - 1) / T) * kb;
    return blocks * (768 * T) + ((blocks * sizeof(float) + 255) & ~(size_t)255);
}

hipError_t launch_split_act(const float *x, uint32_t ldx, uint32_t m, uint32_t k, uint32_t kb, bool vec, uint8_t *xs,
                            float *xf, hipStream_t stream) {
    if (m == 0 || k == 0 || kb != (k + kBlock - 1) / kBlock || (vec && k % 8 != 0)) return hipErrorInvalidValue;
    const uint32_t T = batch_tile(m);
    const dim3 grid((m + T - 1) / T * kb), block(256);
    if (T == 16)
        hipLaunchKernelGGL((vec ? split_act_kernel<16, true> : split_act_kernel<16, false>), grid, block, 0, stream, x,
                           ldx, m, k, kb, xs, xf);
    else
        hipLaunchKernelGGL((vec ? split_act_kernel<32, true> : split_act_kernel<32, false>), grid, block, 0, stream, x,
                           ldx, m, k, kb, xs, xf);
    return hipGetLastError();
}

hipError_t launch_gemv_batch(const BatchParams &pin, bool seq, bool pair, hipStream_t stream) {
    BatchParams p = pin;
    if (p.m == 0 || p.nseg == 0 || p.nseg > 4 || !gemv_rows_shape(p.kb, p.nr) || (pair && (!seq || p.nseg != 2)))
        return hipErrorInvalidValue;
    const uint32_t T = batch_tile(p.m);
    p.tiles = (p.m + T - 1) / T;
    uint32_t groups = 0, max_rows = 0;
    for (uint32_t s = 0; s < p.nseg; s++) {
        p.seg[s].cta_begin = groups;
        groups += p.seg[s].nb;
        max_rows = std::max(max_rows, p.seg[s].rows);
    }
    if (pair) {
        if (p.seg[0].rows != p.seg[1].rows || p.seg[0].nb != p.seg[1].nb) return hipErrorInvalidValue;
        groups = (p.seg[0].rows + 63) / 64;
    }
    p.groups = groups;
    p.items = seq ? groups : groups * p.nr;
    using Kernel = void (*)(BatchParams);
    static const Kernel kernels[6] = {gemv_batch_kernel<16, false, false>, gemv_batch_kernel<16, true, false>,
                                      gemv_batch_kernel<16, true, true>,   gemv_batch_kernel<32, false, false>,
                                      gemv_batch_kernel<32, true, false>,  gemv_batch_kernel<32, true, true>};
    static bool attr_set = false;
    if (!attr_set) {
        for (Kernel k : kernels) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
            if (e != hipSuccess) return e;
        }
        attr_set = true;
    }
    const uint32_t lds = kRing * 8 * 96 * T + (pair ? 2 : 1) * kGemvRsMaxKb * sizeof(float);
    hipLaunchKernelGGL(kernels[(T == 32 ? 3 : 0) + (pair ? 2 : seq ? 1 : 0)], dim3((p.items + 7) / 8 * 8 * p.tiles),
                       dim3(256), lds, stream, p);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && !seq) {
        hipLaunchKernelGGL(batch_combine_kernel, dim3((max_rows + 255) / 256, p.m, p.nseg), dim3(256), 0, stream, p);
        e = hipGetLastError();
    }
    return e;
}

}  // namespace q35mm
