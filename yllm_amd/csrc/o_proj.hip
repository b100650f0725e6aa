// o_proj.hip -- the step after attention: x[b] += W_o . att[b]
// (engine.c:969-973: matmul(att_out, x2, SLOT_O) then the residual add;
// matmul_f16 / matmul_f32, matvec.c:98-122).
//
// W_o is [hidden][qdim] (f16 or f32), att [B][qdim] f32 (or f16 when the
// attention kernel wrote f16; f16 att takes f16 weights), x [B][hidden] f32.
//  * Few tokens (decode, B <= kGemvRows; with f16 weights fewer than
//    rows_from): oproj_gemv_kernel reads W_o once from HBM and applies it to
//    all B rows; activations stay f32 and every product and sum is f32 (the
//    reference's arithmetic, summed in another order).  A wave owns kRows
//    output rows; its lanes take 8 consecutive inputs each (16-byte weight
//    loads at f16), eight iterations of loads in flight (all of a 4096-wide
//    row), then a shuffle reduction and the residual add.
//  * Then up to kRowsMax tokens with f16 weights (the engine's 64-token prefill calls):
//    oproj_rows_kernel streams W_o through MFMA, a workgroup per 16 output
//    rows and its waves splitting the contraction.
//  * More tokens: oproj_gemm_kernel, an f16 MFMA GEMM with f32 accumulation
//    and the residual add in its epilogue.
// In both MFMA kernels f32 att enters as f16 hi + lo parts (hi = f16(att),
// lo = f16(att - hi)), split in registers as the fragments are read, and both
// products accumulate in the same registers, which keeps about 22 bits of
// each activation; attention outputs are convex combinations of f16 V rows
// (times a gate <= 1), so |att| <= 65504 and hi never overflows.  f32 weights
// are split the same way and hi.Whi + lo.Whi + hi.Wlo accumulate.
#include "common.hpp"
#include "internal.hpp"

namespace yhip {
namespace {

constexpr uint32_t kRows = 2;  // output rows per wave of the GEMV
// Up to this many tokens (f16 weights) the rows kernel, above it the GEMM: at
// 64 tokens 3584 x 3584 takes 19 us against 32 (f32 att) and 16 against 29
// (f16), at 96 tokens (two passes over the weights) 38 against 31 and 28
// against 25.
constexpr uint32_t kRowsMax = 64;

template <int W_F16, int A_F16, int NB>
__global__ __launch_bounds__(256) void oproj_gemv_kernel(OProjArgs a)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t o0 = (blockIdx.x * 4u + (threadIdx.x >> 6)) * kRows;
    if (o0 >= a.hidden) return;  // wave-uniform
    float acc[kRows][NB];
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[r][b] = 0.0f;

#pragma unroll 8
    for (uint32_t i0 = lane * 8u; i0 < a.qdim; i0 += 512u) {
        // the weights are read once per call: non-temporal loads (one token,
        // 4096 x 4096 f16: 9.3 -> 8.8 us)
        float w[kRows][8];
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            const uint32_t o = min(o0 + r, a.hidden - 1);  // a missing last row repeats a real one, unused
            if (W_F16) {
                const f16x8 v = __builtin_nontemporal_load(reinterpret_cast<const f16x8*>(reinterpret_cast<const _Float16*>(a.w) +
                                                                (size_t)o * a.qdim + i0));
#pragma unroll
                for (int e = 0; e < 8; ++e) w[r][e] = (float)v[e];
            } else {
                const float* p = reinterpret_cast<const float*>(a.w) + (size_t)o * a.qdim + i0;
                const f32x4 v0 = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
                const f32x4 v1 = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p + 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    w[r][e] = v0[e];
                    w[r][4 + e] = v1[e];
                }
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if ((uint32_t)b >= a.B) break;  // uniform
            float xv[8];
            if (A_F16) {
                const f16x8 v = *reinterpret_cast<const f16x8*>(reinterpret_cast<const _Float16*>(a.att) +
                                                                (size_t)b * a.att_stride + i0);
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[e] = (float)v[e];
            } else {
                const float* p = reinterpret_cast<const float*>(a.att) + (size_t)b * a.att_stride + i0;
                const f32x4 x0 = *reinterpret_cast<const f32x4*>(p);
                const f32x4 x1 = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xv[e] = x0[e];
                    xv[4 + e] = x1[e];
                }
            }
#pragma unroll
            for (uint32_t r = 0; r < kRows; ++r) {
                float s = acc[r][b];
#pragma unroll
                for (int e = 0; e < 8; ++e) s += xv[e] * w[r][e];
                acc[r][b] = s;
            }
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b)
            acc[r][b] = xor_sum<64>(acc[r][b]);
    if (lane == 0) {
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            if (o0 + r >= a.hidden) break;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if ((uint32_t)b >= a.B) break;
                a.x[(size_t)b * a.x_stride + o0 + r] += acc[r][b];
            }
        }
    }
}

constexpr int kBK = 32;  // K per step of the MFMA kernels

// 16-byte chunk swizzle (XOR into the chunk index) of an LDS row of 32 k.
// Rows of 4 chunks (f16, 64 bytes): 8 consecutive rows hit 8 distinct bank
// groups (32 banks, b128 reads in groups of 8 lanes), and 16 consecutive rows
// 16 (64 banks, groups of 16 lanes).  Rows of 8 chunks (f32, 128 bytes): 8
// consecutive rows hit 8 distinct chunk columns, 16 rows each half of a
// 256-byte window 8.  Both depend on bits 0..3 of the row only.
template <bool F32>
__device__ inline int row_swz(int r)
{
    return F32 ? (r & 7) ^ ((r >> 3) & 1) : ((r >> 1) ^ (r >> 2)) & 3;
}

// s_waitcnt vmcnt(n), no wait on the other counters
template <int N>
__device__ inline void wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

__device__ inline f32x16 mfma32(const f16x8& a, const f16x8& b, const f32x16& c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// one 16-byte HBM -> LDS load per lane (lane i writes at lds + 16 i)
__device__ inline void lds_load16(__amdgpu_buffer_rsrc_t r, char* lds, uint32_t voff, uint32_t soff)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, (int)voff, (int)soff,
                                             0, 0);
}

__device__ inline __amdgpu_buffer_rsrc_t rsrc_of(const char* p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), 0, (int)bytes, 0x00020000);
}

constexpr uint32_t kOutside = 0xfffffff0u;  // a buffer offset past every operand: reads zeros

// 8 consecutive k of an operand row as an MFMA fragment: f16 as it is, f32 as
// hi = f16(v) and lo = f16(v - hi)
template <bool F32>
struct Raw {
    f16x8 h;
};
template <>
struct Raw<true> {
    f32x4 v[2];
};
template <bool F32>
__device__ inline void split_raw(const Raw<F32>& raw, f16x8& hi, f16x8& lo)
{
    if constexpr (F32) {
        // v - hi is exact, as the multiply-add -1 hi + v too, which takes hi as
        // f16 and can round to f16 in one instruction; the factor is opaque or
        // the compiler would turn it back into widen, subtract, convert (4
        // instead of 2 instructions per element: the rows kernel at 64 tokens
        // 3584 x 3584 took 20.6 us with that, 18.7 without)
        float m1 = -1.0f;
        asm("" : "+s"(m1));
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            const f32x2 v = {raw.v[j / 4][j % 4], raw.v[j / 4][j % 4 + 1]};
            const f16x2 h = __builtin_convertvector(v, f16x2);
            hi[j] = h[0];
            hi[j + 1] = h[1];
            lo[j] = (_Float16)__builtin_fmaf((float)h[0], m1, v[0]);
            lo[j + 1] = (_Float16)__builtin_fmaf((float)h[1], m1, v[1]);
        }
    } else {
        hi = raw.h;
    }
}

// ---- few tokens: x[t][o] += sum_k att[t][k] W[o][k] for at most 16 NT tokens ----
//
// Bound by streaming W_o once (3584 x 3584: 25.7 MB, ~5 us) and by the token
// rows, which every workgroup reads whole from L2 (64 f32 tokens: 0.9 MB per
// workgroup at 64 bytes per cycle and CU).  A workgroup owns 16 output rows,
// so hidden / 16 workgroups cover the chip (224 of 256 CUs at 3584), and its 8
// waves split the contraction: each takes a run of 32-k steps, loads the W
// fragments of 16 steps into registers at once (all of a 4096-wide row: one
// HBM round trip) and walks its steps with the token rows coming through its
// own LDS ring (direct-to-LDS loads, kDep steps deep, no barrier: a wave
// reads only what it loaded).  Read straight into registers, a token
// fragment's load instruction would touch 16 rows, a quarter of the lines'
// rate; through LDS it covers whole 128-byte rows.  The waves' sums meet in LDS in
// wave order, so the result does not depend on timing.  3584 x 3584, us for 64
// / 32 / 16 f32 tokens: 18.7 / 14.4 / 12.0; the 64 x 64 GEMM tiles before it
// (56 workgroups, 224 steps each, and a launch to split att) took 79.
//
// X32 (f32 tokens, up to kGemvRows of them): the products stay f32, on the
// f32 MFMA (k-slot g of MFMA e is k 8 g + e), with the one-pass kernel's range
// and error; 8 x 16 cycles more per step than the f16 parts, under the loads.
template <int NT, bool AF32, bool X32 = false>
__global__ __launch_bounds__(512, 1) void oproj_rows_kernel(OProjArgs a)
{
    static_assert(!X32 || (AF32 && NT == 1), "a few f32 tokens");
    constexpr int EB = AF32 ? 4 : 2, CPR = kBK * EB / 16;  // bytes per element, chunks per row of 32 k
    constexpr int SB = NT * 16 * kBK * EB;                 // bytes of a stage: 16 NT rows
    constexpr int NLD = SB / 1024;                         // loads per lane and step
    constexpr int kDep = 8 * 2 * SB > 65536 ? 2 : 4;       // ring depth: at most 128 KB over the 8 waves
    constexpr int RW = 16;                                 // steps per round
    __shared__ __attribute__((aligned(16))) char ring[8][kDep][SB];
    static_assert(sizeof(ring) >= 8 * NT * 1024, "the reduction reuses the ring");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const uint32_t o0 = blockIdx.x * 16u, nt = a.B;

    // this thread's part of the output: token 16 (tid / 64) + 4 g + i, row o0 + r16
    const uint32_t ot = 16u * wave + 4u * g, oo = o0 + r16;
    float xv[4];
    if (wave < NT) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            xv[i] = a.x[(size_t)min(ot + i, nt - 1) * a.x_stride + min(oo, a.hidden - 1)];
    }

    const uint32_t K = a.qdim, ksteps = (K + kBK - 1) / kBK, per = (ksteps + 7) / 8;
    const uint32_t s0 = wave * per, n = s0 < ksteps ? min(per, ksteps - s0) : 0;
    // operands of this workgroup: 16 W rows, the tokens' rows
    const char* wp = reinterpret_cast<const char*>(a.w) + (size_t)o0 * K * 2;
    const char* tp = reinterpret_cast<const char*>(a.att);
    const uint32_t wbytes = min(16u, a.hidden - o0) * K * 2u;
    const uint32_t tbytes = ((nt - 1) * a.att_stride + K) * EB;
    const uint32_t woff = (r16 * K + 8u * g) * 2u;
    // load u of a step covers rows 64 u / CPR ..; at 8 rows per load the even and odd loads differ in bit 3 of the
    // row, hence in the swizzled chunk: tk is that chunk's first k
    uint32_t tk[2], toff[NLD];
#pragma unroll
    for (int p = 0; p < 2; ++p) tk[p] = ((lane % CPR) ^ row_swz<AF32>((64 * p + lane) / CPR & 15)) * (16u / EB);
#pragma unroll
    for (int u = 0; u < NLD; ++u) toff[u] = ((64u * u + lane) / CPR * a.att_stride + tk[u & 1]) * EB;

    f32x4 acc[NT];
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // 16 tokens and fewer: more accumulators, for shorter sums (the one-pass kernel's error, and no longer chain)
    constexpr int NX = X32 ? 8 : NT == 1 ? 2 : 1;
    f32x4 accx[NX];
#pragma unroll
    for (int e = 0; e < NX; ++e) accx[e] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (uint32_t r0 = 0; r0 < n; r0 += RW) {
        // step i of the round covers k0 .. k0 + 31; past this wave's steps and past K every load reads zeros
        auto k0_of = [&](int i) { return (s0 + r0 + i) * kBK; };
        auto issue = [&](int i) {
            const bool in = r0 + i < n;
            const __amdgpu_buffer_rsrc_t rt = rsrc_of(tp, in ? tbytes : 0u);
            const uint32_t k0 = in ? k0_of(i) : 0u;
#pragma unroll
            for (int u = 0; u < NLD; ++u) {
                lds_load16(rt, ring[wave][i % kDep] + u * 1024, k0 + tk[u & 1] < K ? toff[u] : kOutside, k0 * EB);
            }
        };
        f16x8 w[RW];
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            const bool in = r0 + i < n;
            const uint32_t k0 = in ? k0_of(i) : 0u;
            const uint32_t off = k0 + 8u * g < K ? woff : kOutside;
            // read once per call: non-temporal
            w[i] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc_of(wp, in ? wbytes : 0u), (int)off,
                                                                                   (int)(k0 * 2u), 2));
        }
#pragma unroll
        for (int i = 0; i < kDep; ++i) issue(i);
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            if (i % 4 == 0 && r0 + i >= n) break;  // uniform over the wave
            constexpr int last = RW - 1;
            // this step's rows have landed; later steps' loads may stay in flight
            switch (last - i < kDep - 1 ? last - i : kDep - 1) {
            case 0: wait_vm<0>(); break;
            case 1: wait_vm<NLD>(); break;
            case 2: wait_vm<2 * NLD>(); break;
            default: wait_vm<3 * NLD < 64 ? 3 * NLD : 63>(); break;
            }
            asm volatile("" ::: "memory");
            Raw<AF32> raw[NT];
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                const char* row = ring[wave][i % kDep] + (16 * b + r16) * (kBK * EB);
                if constexpr (AF32) {
                    raw[b].v[0] = *reinterpret_cast<const f32x4*>(row + ((2 * g) ^ row_swz<AF32>(r16)) * 16);
                    raw[b].v[1] = *reinterpret_cast<const f32x4*>(row + ((2 * g + 1) ^ row_swz<AF32>(r16)) * 16);
                } else {
                    raw[b].h = *reinterpret_cast<const f16x8*>(row + (g ^ row_swz<AF32>(r16)) * 16);
                }
            }
            if (i + kDep < RW) {
                __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads are done, the stage may be overwritten
                asm volatile("" ::: "memory");
                issue(i + kDep);
            }
            if constexpr (X32) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    accx[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(raw[0].v[e / 4][e % 4], (float)w[i][e], accx[e], 0, 0, 0);
            } else {
#pragma unroll
                for (int b = 0; b < NT; ++b) {
                    f16x8 hi, lo;
                    split_raw<AF32>(raw[b], hi, lo);
                    f32x4& c = NT == 1 ? accx[i & 1] : acc[b];
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, w[i], c, 0, 0, 0);
                    if (AF32) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, w[i], c, 0, 0, 0);
                }
            }
        }
        wait_vm<0>();  // nothing in flight into the ring before it is used again
    }
    if constexpr (X32) acc[0] = ((accx[0] + accx[1]) + (accx[2] + accx[3])) + ((accx[4] + accx[5]) + (accx[6] + accx[7]));
    else if constexpr (NT == 1) acc[0] = accx[0] + accx[1];
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(&ring[0][0][0]);  // [wave][block][lane]
#pragma unroll
    for (int b = 0; b < NT; ++b) red[(wave * NT + b) * 64 + lane] = acc[b];
    __syncthreads();
    if (wave >= NT) return;
    f32x4 sum = red[wave * 64 + lane];
#pragma unroll
    for (int w = 1; w < 8; ++w) sum += red[(w * NT + wave) * 64 + lane];
    if (oo < a.hidden) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (ot + i < nt) a.x[(size_t)(ot + i) * a.x_stride + oo] = xv[i] + sum[i];
    }
}

// ---- the GEMM: x[t][o] += sum_k T[t][k] * W[o][k] ----
//
// T (tokens, the MFMA A operand) and W (W_o rows, the B operand) are f16 or
// f32 rows with K innermost.  A workgroup (4 waves, WT x WO) owns BT tokens x
// BO outputs; a wave owns (TM x 32) x (TN x 32) of them in TM x TN
// v_mfma_f32_32x32x16_f16 accumulators.
//
// The bound is the matrix pipe, and next to it the LDS: a 32 x 32 x 16 MFMA
// takes 32 cycles, in which the four SIMDs can take 4 KB of operands from a
// 128-byte-per-cycle LDS, tile writes included.  A wave of 128 x 128 (f16, one
// wave per SIMD) reads 8 fragments for 16 MFMAs and its workgroup writes 32 KB
// per 128 MFMAs: 0.75 KB per MFMA, where 64 x 128 waves took 1.13 KB, over
// the limit.  With f32 tokens the hi and lo products share the W fragment: 64
// x 128 waves read 4 + 4 (f32 fragments are two reads) for 16 MFMAs.
//
// K advances 32 at a time through four LDS stages; both tiles go from HBM
// straight into LDS (16 bytes per lane) in XOR-swizzled rows.  With one wave
// per SIMD nothing else covers a wave's waits, so the loop is pipelined across
// the barrier: a step's first half issues its MFMAs while the second half's
// fragments are read; then the barrier, which says that the stage is read
// and the next one (loaded three steps ago) has landed; then the second
// half's MFMAs issue while the next step's first fragments are read and the
// loads four steps ahead go into the stage just read.  The four stages are
// separate variables and the loop is unrolled by four, so the compiler sees
// loads in flight never alias the reads.  f16 8192 x 4096 x 4096, operands from
// HBM, 350 -> 291 us (945 TFLOP/s; 1250 in the loop alone; repeated on one set of
// operands, whose 235 MB the last-level cache holds, 328 -> 265); f32 att 2048 x
// 3584 x 3584, repeated, 186 with its split pass -> 103.
struct GemmArgs {
    const char* t;  // token rows
    const char* w;  // W_o rows, ld K
    float* x;
    uint32_t t_ld, x_stride, N, M, K;
};

constexpr int kStages = 4;

// issue order of a half step: each of NRD fragment reads is followed by its
// share of the NLD tile loads and of the NMF MFMAs
template <int NRD, int NLD, int NMF, int I>
__device__ inline void spread()
{
    if constexpr (I < NRD) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        constexpr int nl = NLD * (I + 1) / NRD - NLD * I / NRD, nm = NMF * (I + 1) / NRD - NMF * I / NRD;
        if constexpr (nl > 0) __builtin_amdgcn_sched_group_barrier(0x020, nl, 0);
        if constexpr (nm > 0) __builtin_amdgcn_sched_group_barrier(0x008, nm, 0);
        spread<NRD, NLD, NMF, I + 1>();
    }
}

template <int TM, int TN, int WT, int WO, bool AF32, bool WF32, int WPC>
__global__ __launch_bounds__(256, WPC) void oproj_gemm_kernel(GemmArgs a)
{
    static_assert(WT * WO == 4, "four waves");
    constexpr int BT = WT * TM * 32, BO = WO * TN * 32;   // workgroup tile
    constexpr int EA = AF32 ? 4 : 2, EW = WF32 ? 4 : 2;
    constexpr int RBA = kBK * EA, RBW = kBK * EW;          // row bytes
    constexpr int CA = RBA / 16, CW = RBW / 16;            // chunks per row
    constexpr int NLA = BT * CA / 256, NLW = BO * CW / 256;  // loads per thread and step
    constexpr int NLD = NLA + NLW;
    constexpr int SB = BT * RBA + BO * RBW;                // stage bytes
    static_assert(BT * CA % 256 == 0 && BO * CW % 256 == 0, "whole load instructions per operand");
    __shared__ __attribute__((aligned(16))) char S0[SB], S1[SB], S2[SB], S3[SB];
    auto stage = [&](int s) -> char* { return s == 0 ? S0 : s == 1 ? S1 : s == 2 ? S2 : S3; };

    // the wave index in a scalar register: the LDS destination of a
    // direct-to-LDS load (M0) must be uniform
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r32 = lane & 31, hh = lane >> 5;
    const int wt = wave / WO, wo = wave % WO;
    // Tile order: the hardware deals consecutive workgroups to the 8 XCDs in
    // turn; workgroup x takes position (x % 8) * (grid / 8) + x / 8 of the
    // order below, so each XCD works through a contiguous run of it, and the
    // order walks groups of 4 token tiles across the output tiles, so the
    // workgroups an XCD runs at once share a few token and weight tiles in
    // its L2 (grid is a multiple of 8).
    const uint32_t n_ot = (a.M + BO - 1) / BO, n_tt = (a.N + BT - 1) / BT;
    const uint32_t per_xcd = gridDim.x / 8u;
    const uint32_t pid = (blockIdx.x % 8u) * per_xcd + blockIdx.x / 8u;
    const uint32_t grp = pid / (4u * n_ot), in_g = pid % (4u * n_ot);
    const uint32_t g_rows = min(4u, n_tt - grp * 4u);
    if (pid >= n_ot * n_tt) return;
    const uint32_t t0 = (grp * 4u + in_g % g_rows) * BT, o0 = (in_g / g_rows) * BO;
    const uint32_t nt = min((uint32_t)BT, a.N - t0), no = min((uint32_t)BO, a.M - o0);
    const uint32_t K = a.K, nsteps = (K + kBK - 1) / kBK;

    // Offsets of this thread's chunks from the tile's first row at k 0; a row
    // past the tile's last lies past the resource's end and reads zeros.
    // Load i covers 256 / CA rows, a multiple of 16: the swizzle is the same
    // for every i.
    const int ca = (tid % CA) ^ row_swz<AF32>(tid / CA), cw = (tid % CW) ^ row_swz<WF32>(tid / CW);
    uint32_t ta[NLA], tw[NLW];
#pragma unroll
    for (int i = 0; i < NLA; ++i) ta[i] = (256 / CA * i + tid / CA) * (a.t_ld * EA) + ca * 16u;
#pragma unroll
    for (int i = 0; i < NLW; ++i) tw[i] = (256 / CW * i + tid / CW) * (K * EW) + cw * 16u;
    const char* tp = a.t + (size_t)t0 * a.t_ld * EA;
    const char* wp = a.w + (size_t)o0 * K * EW;
    const uint32_t tbytes = ((nt - 1) * a.t_ld + K) * EA, wbytes = no * K * EW;
    const uint32_t ka = ca * 16u / EA, kw = cw * 16u / EW;  // k of the chunks within a step
    // load i of step st into stage s; a step past the last and the chunks past
    // K of a partial last step read zeros
    struct Step {
        __amdgpu_buffer_rsrc_t rt, rw;
        uint32_t k0, ma, mw;
    };
    auto step_of = [&](uint32_t st) {
        const bool in = st < nsteps;  // workgroup-uniform
        const uint32_t k0 = in ? st * kBK : 0u;
        return Step{rsrc_of(tp, in ? tbytes : 0u), rsrc_of(wp, in ? wbytes : 0u), k0, k0 + ka < K ? 0u : kOutside,
                    k0 + kw < K ? 0u : kOutside};
    };
    auto issue = [&](const Step& p, int s, int i) {
        if (i < NLA)
            lds_load16(p.rt, stage(s) + (256 * i + 64 * wave) * 16, ta[i < NLA ? i : 0] | p.ma, p.k0 * EA);
        else
            lds_load16(p.rw, stage(s) + BT * RBA + (256 * (i - NLA) + 64 * wave) * 16, tw[i < NLA ? 0 : i - NLA] | p.mw,
                       p.k0 * EW);
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[m][n][i] = 0.0f;

    // fragments of half kk of a stage: row r32 of each 32-row block, k 16 kk + 8 hh ..
    struct Frags {
        Raw<AF32> t[TM];
        Raw<WF32> w[TN];
    };
    // (each address is one offset from its stage: through a chain of them the
    // compiler loses track of the variable and waits for every load in flight)
    const int swa = row_swz<AF32>(r32 & 15), sww = row_swz<WF32>(r32 & 15);
    const int ra = (wt * TM * 32 + r32) * RBA, rw = BT * RBA + (wo * TN * 32 + r32) * RBW;
    auto read_row = [&](auto& f, int s, int off, int kk, int swz) {
        if constexpr (sizeof(f) == 32) {
            f.v[0] = *reinterpret_cast<const f32x4*>(stage(s) + (off + (((4 * kk + 2 * hh) ^ swz) << 4)));
            f.v[1] = *reinterpret_cast<const f32x4*>(stage(s) + (off + (((4 * kk + 2 * hh + 1) ^ swz) << 4)));
        } else {
            f.h = *reinterpret_cast<const f16x8*>(stage(s) + (off + (((2 * kk + hh) ^ swz) << 4)));
        }
    };
    auto read = [&](Frags& f, int s, int kk) {
#pragma unroll
        for (int n = 0; n < TN; ++n) read_row(f.w[n], s, rw + n * 32 * RBW, kk, sww);
#pragma unroll
        for (int m = 0; m < TM; ++m) read_row(f.t[m], s, ra + m * 32 * RBA, kk, swa);
    };
    auto mma = [&](const Frags& f) {
        f16x8 wh[TN], wl[WF32 ? TN : 1];
#pragma unroll
        for (int n = 0; n < TN; ++n) split_raw<WF32>(f.w[n], wh[n], wl[WF32 ? n : 0]);
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            f16x8 hi, lo;
            split_raw<AF32>(f.t[m], hi, lo);
#pragma unroll
            for (int n = 0; n < TN; ++n) acc[m][n] = mfma32(hi, wh[n], acc[m][n]);
            if constexpr (AF32) {
#pragma unroll
                for (int n = 0; n < TN; ++n) acc[m][n] = mfma32(lo, wh[n], acc[m][n]);
            }
            if constexpr (WF32) {
#pragma unroll
                for (int n = 0; n < TN; ++n) acc[m][n] = mfma32(hi, wl[n], acc[m][n]);
            }
        }
    };
    constexpr int NMF = TM * TN * (1 + AF32 + WF32);              // MFMAs per half step
    constexpr int NRD = TM * (AF32 ? 2 : 1) + TN * (WF32 ? 2 : 1);  // fragment reads per half step

    // the residual of a whole tile: accumulator (m, n, i) is token 32 m + 8 (i /
    // 4) + i % 4 + 4 hh of the wave's, output 32 n + r32: a scalar row and a lane
    // offset
    const bool whole = nt == (uint32_t)BT && no == (uint32_t)BO;  // workgroup-uniform
    float* const xw = a.x + (size_t)(t0 + wt * TM * 32) * a.x_stride + o0 + wo * TN * 32;
    const uint32_t xlane = 4u * hh * a.x_stride + r32;
    auto x_row = [&](int m, int i) { return xw + (size_t)(32 * m + 8 * (i / 4) + i % 4) * a.x_stride; };
    float xv[2][16][TN];
    auto load_x = [&](int m) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
            for (int n = 0; n < TN; ++n) xv[m & 1][i][n] = x_row(m, i)[xlane + 32 * n];
    };
    constexpr bool kEarlyX = TM < 4;  // (256 x 256 tiles have no registers left for it and spilled: 271 -> 362 us)
    if (kEarlyX && whole) load_x(0);

    Frags f0, f1;
#pragma unroll
    for (int s = 0; s < kStages; ++s) {
        const Step p = step_of(s);
#pragma unroll
        for (int i = 0; i < NLD; ++i) issue(p, s, i);
    }
    wait_vm<(kStages - 1) * NLD>();
    lds_barrier();
    read(f0, 0, 0);
    for (uint32_t st = 0; st < nsteps; st += kStages) {
#pragma unroll
        for (int s = 0; s < kStages; ++s) {  // step st + s; past the last its operands are zeros
            read(f1, s, 1);
            mma(f0);
            spread<NRD, 0, NMF, 0>();
            __builtin_amdgcn_sched_barrier(0);
            wait_vm<(kStages - 2) * NLD>();  // step st + s + 1 has landed
            lds_barrier();                   // for every wave, and every wave has read stage s
            const Step p = step_of(st + s + kStages);
            read(f0, (s + 1) % kStages, 0);
#pragma unroll
            for (int i = 0; i < NLD; ++i) issue(p, s, i);
            mma(f1);
            spread<NRD, NLD, NMF, 0>();
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    wait_vm<0>();  // the loads past the end land before the workgroup ends

    // x[t][o] += acc.  Whole tiles: the loads of one row of blocks ahead of
    // the adds and stores of the one before, the first row's from before the K
    // loop where they fit (as float atomics the epilogue took three times as
    // long: 8192 x 4096 x 4096, f16, repeated, 312 -> 265 us).  Partial tiles, where
    // each access has its own bounds test: float atomics, which nothing waits for
    // (one add per element, so the result is the load, add and store's).
    if (whole) {
        if (!kEarlyX) load_x(0);
#pragma unroll
        for (int m = 0; m < TM; ++m) {
            if (m + 1 < TM) load_x(m + 1);
#pragma unroll
            for (int i = 0; i < 16; ++i)
#pragma unroll
                for (int n = 0; n < TN; ++n) x_row(m, i)[xlane + 32 * n] = xv[m & 1][i][n] + acc[m][n][i];
        }
        return;
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t t = wt * TM * 32 + 4 * hh + 32 * m + 8 * (i / 4) + i % 4, o = wo * TN * 32 + r32;
            float* row = a.x + (size_t)(t0 + t) * a.x_stride + o0;
#pragma unroll
            for (int n = 0; n < TN; ++n)
                if (t < nt && o + 32u * n < no) unsafeAtomicAdd(row + o + 32 * n, acc[m][n][i]);
        }
}

template <int TM, int TN, int WT, int WO, bool AF32, bool WF32, int WPC>
hipError_t launch_gemm_tiles(const GemmArgs& a, hipStream_t st)
{
    constexpr uint32_t BT = WT * TM * 32, BO = WO * TN * 32;
    const uint32_t tiles = ((a.N + BT - 1) / BT) * ((a.M + BO - 1) / BO);
    hipLaunchKernelGGL((oproj_gemm_kernel<TM, TN, WT, WO, AF32, WF32, WPC>), dim3((tiles + 7) / 8 * 8), dim3(256), 0,
                       st, a);
    return hipGetLastError();
}

// Tile choice: the largest tile of which there are enough for three quarters
// of the CUs.  A larger tile moves fewer LDS and L2 bytes per MFMA, but one
// workgroup per CU cannot fill a chip of which it leaves a quarter idle.
// us with each tile, largest first, operands from HBM.  f16 att, 4096 x 4096,
// 256 x 256 / 128 x 256 / 128 x 128 / 64 x 128 / 64 x 64: 8192 tokens 294 / 341 /
// 375 / 492 / 608, 2048 122 / 95 / 98 / 139 / 175, 1024 117 / 81 / 57 / 75 / 92, 512
// 111 / 76 / 50 / 43 / 50, 256 101 / 69 / 48 / 43 / 31.  f32 att, 3584 x 3584, 128 x
// 256 / 64 x 128 / 64 x 64: 2048 111 / 143 / 171, 1024 89 / 71 / 94, 512 81 / 44 /
// 53, 256 74 / 38 / 30.  f32 weights, 3584 x 3584, 128 x 128 / 64 x 64: 2048 181 /
// 233, 1024 93 / 128, 512 78 / 67, 256 73 / 41.  It does not see a part-filled last
// round: 640 tokens 4096 x 4096 f16 run 60 us as 320 tiles of 64 x 128, 52 as 160 of
// 128 x 128.
hipError_t launch_gemm(const GemmArgs& a, bool af32, bool wf32, hipStream_t st)
{
    const uint64_t enough = (uint64_t)n_cus() * 3 / 4;
    auto fits = [&](uint32_t bt, uint32_t bo) {
        return (uint64_t)((a.N + bt - 1) / bt) * ((a.M + bo - 1) / bo) >= enough;
    };
    if (wf32) {
        if (fits(128, 128)) return launch_gemm_tiles<2, 2, 2, 2, true, true, 1>(a, st);
        return launch_gemm_tiles<1, 1, 2, 2, true, true, 2>(a, st);
    }
    if (af32) {
        if (fits(128, 256)) return launch_gemm_tiles<2, 4, 2, 2, true, false, 1>(a, st);
        if (fits(64, 128)) return launch_gemm_tiles<1, 2, 2, 2, true, false, 2>(a, st);
        return launch_gemm_tiles<1, 1, 2, 2, true, false, 2>(a, st);
    }
    if (fits(256, 256)) return launch_gemm_tiles<4, 4, 2, 2, false, false, 1>(a, st);
    if (fits(128, 256)) return launch_gemm_tiles<2, 4, 2, 2, false, false, 1>(a, st);
    if (fits(128, 128)) return launch_gemm_tiles<2, 2, 2, 2, false, false, 2>(a, st);
    if (fits(64, 128)) return launch_gemm_tiles<1, 2, 2, 2, false, false, 2>(a, st);
    return launch_gemm_tiles<1, 1, 2, 2, false, false, 2>(a, st);
}

template <int W_F16, int A_F16>
hipError_t launch_gemv(const OProjArgs& a, hipStream_t st)
{
    const uint32_t waves = (a.hidden + kRows - 1) / kRows;
    const dim3 grid((waves + 3) / 4);
    if (a.B <= 1)
        hipLaunchKernelGGL((oproj_gemv_kernel<W_F16, A_F16, 1>), grid, dim3(256), 0, st, a);
    else if (a.B <= 2)
        hipLaunchKernelGGL((oproj_gemv_kernel<W_F16, A_F16, 2>), grid, dim3(256), 0, st, a);
    else if (a.B <= 4)
        hipLaunchKernelGGL((oproj_gemv_kernel<W_F16, A_F16, 4>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((oproj_gemv_kernel<W_F16, A_F16, 8>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

template <bool AF32>
hipError_t launch_rows(const OProjArgs& a, hipStream_t st)
{
    const uint32_t gx = (a.hidden + 15) / 16;
    if (a.B <= 16)
        hipLaunchKernelGGL((oproj_rows_kernel<1, AF32>), dim3(gx), dim3(512), 0, st, a);
    else if (a.B <= 32)
        hipLaunchKernelGGL((oproj_rows_kernel<2, AF32>), dim3(gx), dim3(512), 0, st, a);
    else
        hipLaunchKernelGGL((oproj_rows_kernel<4, AF32>), dim3(gx), dim3(512), 0, st, a);
    return hipGetLastError();
}

// The fewest tokens that take the rows kernel instead of the one-pass kernel
// (f16 weights; kGemvRows at most).  It reads each token row once per 16 output
// rows, the other once per two, but starts slower (a ring and a reduction in
// LDS), and as one workgroup per CU, so that a part-filled last round costs a
// whole one.  us one-pass / rows, weights from HBM (in the caches the one-pass
// kernel is up to 10 % better at these edges): f16 3 tokens 4096 x 4096 13.7 /
// 9.6, 2048 x 4096 10.4 / 8.7, 1024 x 2048 6.5 / 6.2 (in the caches 5.4 / 6.3),
// 896 x 896 4.8 / 4.8 (4.4 / 5.0), 8192 x 8192 29.7 / 30.9; 4 tokens 896 x 896
// 5.5 / 5.0, 8192 x 8192 36.0 / 31.3; 320 or 384 workgroups: 5120 x 5120 4
// tokens 22.7 / 23.2, 6 26.1 / 23.1.  f32 5 tokens 4096 x 4096 16.1 / 13.2,
// 11008 x 4096 36.2 / 28.8, 1536 x 1536 7.1 / 7.7, 5120 x 5120 21.1 / 28.0; 6
// tokens 896 x 896 6.6 / 5.8, 5120 x 5120 24.3 / 28.4, 7 29.0 / 28.7.
uint32_t rows_from(uint32_t hidden, uint32_t qdim, bool att_f16)
{
    const uint32_t wgs = (hidden + 15) / 16, cus = (uint32_t)n_cus(), rounds = (wgs + cus - 1) / cus;
    const bool one = rounds == 1, full = (uint64_t)wgs * 20 >= (uint64_t)rounds * cus * 17;
    if (att_f16) return one && qdim >= 3072 ? 3u : one || full ? 4u : 6u;
    return full ? 5u : one ? 6u : 7u;
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// f32 rows of 4 cols4 elements, `stride` elements apart, to a contiguous matrix
__global__ __launch_bounds__(256) void oproj_copy_kernel(f32x4* dst, const float* src, uint32_t stride, uint32_t cols4,
                                                         uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    dst[i] = *reinterpret_cast<const f32x4*>(src + i / cols4 * stride + i % cols4 * 4u);
}

hipError_t copy_rows(void* dst, const void* src, uint32_t stride, uint32_t rows, uint32_t cols, hipStream_t st)
{
    const uint64_t n = (uint64_t)rows * (cols / 4);
    hipLaunchKernelGGL(oproj_copy_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<f32x4*>(dst), reinterpret_cast<const float*>(src), stride, cols / 4, n);
    return hipGetLastError();
}

}  // namespace

// whether some byte lies both in a row of a and in a row of b
bool rows_overlap(const Rows& a, const Rows& b)
{
    const uint64_t pa = (uint64_t)(uintptr_t)a.p, pb = (uint64_t)(uintptr_t)b.p;
    if (pa + (a.n - 1) * a.step + a.bytes <= pb || pb + (b.n - 1) * b.step + b.bytes <= pa) return false;
    if (a.step != b.step) return true;  // (or taken to)
    // column ranges of one matrix: where b's rows start within a's step
    const uint64_t d = pb >= pa ? (pb - pa) % a.step : (a.step - (pa - pb) % a.step) % a.step;
    return d < a.bytes || d + b.bytes > a.step;
}

size_t oproj_workspace(uint32_t B, uint32_t qdim, uint32_t w_f16, uint32_t att_f16, uint32_t hidden)
{
    if (B <= kGemvRows || att_f16) return 0;
    // Room for a copy of each f32 operand, which a call whose operands overlap x needs (launch_oproj).
    return 2 * align256((size_t)B * qdim * 2) + (w_f16 ? 0 : 2 * align256((size_t)hidden * qdim * 2));
}

const char* launch_oproj(const OProjArgs& in, void* ws, hipStream_t st)
{
    OProjArgs a = in;
    // the MFMA kernels address a tile's rows with 32-bit byte offsets
    auto reach = [&] { return 256ull * 4 * (a.att_stride > a.qdim ? a.att_stride : a.qdim) < 0xf0000000ull; };
    bool near = reach();
    // The MFMA kernels read an operand in many workgroups while others already update x.  An f32 operand that
    // overlaps x (x += W x) is read from a copy; so are rows too far apart, which would take the one-pass kernel.
    if (a.B > kGemvRows && !a.att_f16 && ws) {
        const Rows x = {a.x, a.x_stride * 4ull, a.hidden * 4ull, a.B}, row = {a.att, a.att_stride * 4ull, a.qdim * 4ull, a.B},
                   w = {a.w, a.qdim * 4ull, a.qdim * 4ull, a.hidden};
        hipError_t e = hipSuccess;
        if (!a.w_f16 && rows_overlap(x, w)) {
            char* dst = reinterpret_cast<char*>(ws) + 2 * align256((size_t)a.B * a.qdim * 2);
            e = copy_rows(dst, a.w, a.qdim, a.hidden, a.qdim, st);
            a.w = dst;
        }
        if (e == hipSuccess && (!near || rows_overlap(x, row))) {
            e = copy_rows(ws, a.att, a.att_stride, a.B, a.qdim, st);
            a.att = ws;
            a.att_stride = a.qdim;
            near = reach();
        }
        if (e != hipSuccess) return hipGetErrorString(e);
    }
    if (a.B <= kGemvRows) {
        hipError_t e;
        if (a.w_f16 && a.B >= rows_from(a.hidden, a.qdim, a.att_f16) && near) {
            const dim3 grid((a.hidden + 15) / 16);
            if (a.att_f16) hipLaunchKernelGGL((oproj_rows_kernel<1, false>), grid, dim3(512), 0, st, a);
            else hipLaunchKernelGGL((oproj_rows_kernel<1, true, true>), grid, dim3(512), 0, st, a);
            e = hipGetLastError();
            return e == hipSuccess ? nullptr : hipGetErrorString(e);
        }
        if (a.w_f16)
            e = a.att_f16 ? launch_gemv<1, 1>(a, st) : launch_gemv<1, 0>(a, st);
        else
            e = a.att_f16 ? launch_gemv<0, 1>(a, st) : launch_gemv<0, 0>(a, st);
        return e == hipSuccess ? nullptr : hipGetErrorString(e);
    }
    // rows too long for the MFMA kernels go through the one-pass kernel, eight tokens at a time
    if (!near) {
        for (uint32_t b0 = 0; b0 < a.B; b0 += kGemvRows) {
            OProjArgs p = a;
            p.B = a.B - b0 < kGemvRows ? a.B - b0 : kGemvRows;
            p.x = a.x + (size_t)b0 * a.x_stride;
            p.att = reinterpret_cast<const char*>(a.att) + (size_t)b0 * a.att_stride * (a.att_f16 ? 2 : 4);
            if (const char* msg = launch_oproj(p, nullptr, st)) return msg;
        }
        return nullptr;
    }
    hipError_t e;
    if (a.w_f16 && a.B <= kRowsMax) {
        e = a.att_f16 ? launch_rows<false>(a, st) : launch_rows<true>(a, st);
    } else {
        GemmArgs g = {};
        g.t = reinterpret_cast<const char*>(a.att);
        g.w = reinterpret_cast<const char*>(a.w);
        g.x = a.x;
        g.t_ld = a.att_stride;
        g.x_stride = a.x_stride;
        g.N = a.B;
        g.M = a.hidden;
        g.K = a.qdim;
        e = launch_gemm(g, !a.att_f16, !a.w_f16, st);
    }
    return e == hipSuccess ? nullptr : hipGetErrorString(e);
}

}  // namespace yhip
