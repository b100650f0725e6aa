// rope.hip -- rotary position embedding of q and k fused with the K and V
// stores into the head-major HBM cache: the step before attention
// (engine.c:1054-1072 llama / qwen, engine.c:910-934 qwen35).
//
// Kinds (matvec.c:890-939), per head of head_dim d, position pos, pair j:
//   PAIRS  (rope_inplace, llama):        (v[2j], v[2j+1]),        j < d/2
//   HALF   (rope_inplace_qwen, qwen):    (v[j], v[j+d/2]),        j < d/2
//   MROPE  (rope_inplace_mrope, qwen35): (v[j], v[j+n_rot/2]),    j < n_rot/2,
//          dims n_rot..d-1 unchanged
// with freq = powf(theta, -2j/dn) (dn = d, or n_rot for MROPE),
// ang = freq * pos, (a, b) -> (a cos - b sin, a sin + b cos), in float like
// the reference.  The frequencies come in the launch arguments, computed by
// the host C library's powf as in the reference: a 1-ulp frequency error
// would grow to about pos * 6e-8 rad at position pos (8e-3 rad at 131071).
// The angle is then bit for bit the reference's; the device cosf / sinf
// differ from the host library by an ulp or two.
//
// One launch, two kinds of workgroup:
//  * rotation blocks: a wave per token (for few tokens, a few waves per
//    token, each with a range of its heads).  Its lanes own the token's
//    pairs (two heads per pass at d = 64, two pairs per lane at d = 256);
//    each lane computes its angles' sine and cosine once and applies them to
//    the pair in every head of its range, loading four passes ahead of
//    their stores.  Loads and stores are 8 / 4 bytes per lane where the
//    pair is two adjacent elements.  q goes to
//    q_out (f32 / f16 / bf16); k is rounded with the reference f32->f16
//    rounding (platform.c:340-379) into the token's K row of each kv head.
//    Up to kScatterRows tokens the same waves also write the token's V
//    elements into the tiles.
//  * V tile blocks (more than kScatterRows tokens): 64 positions x 64 channels
//    through LDS, read along source rows and written along tile rows, rounded
//    the same way.
#include "common.hpp"
#include "internal.hpp"

#include <math.h>

namespace yhip {
namespace {

// Up to this many tokens the rotation waves write V too, one pass each, with
// no tile blocks (a memory round trip through LDS and a barrier): 28 / 4 heads
// of 128, us with / without tile blocks: 17 tokens 5.4 / 3.3, 64 tokens 5.5 /
// 3.8, 128 tokens 5.5 / 4.7, 256 tokens 5.7 / 5.4 (32 / 8 heads 6.2 / 6.8).
constexpr uint32_t kScatterRows = 128;

__device__ inline uint16_t bf16_bits(float x)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__device__ inline uint16_t half_bits(float x, uint32_t dt)
{
    return dt == kF16 ? __builtin_bit_cast(uint16_t, (_Float16)x) : bf16_bits(x);
}

// two elements e0, e1 of q_out row `o`
__device__ inline void store_q_pair(void* out, size_t o, uint32_t e0, uint32_t e1, uint32_t dt, float x0, float x1)
{
    if (dt == kF32) {
        float* p = reinterpret_cast<float*>(out) + o;
        if (e1 == e0 + 1) {
            *reinterpret_cast<float2*>(p + e0) = make_float2(x0, x1);
        } else {
            p[e0] = x0;
            p[e1] = x1;
        }
    } else {
        uint16_t* p = reinterpret_cast<uint16_t*>(out) + o;
        const uint16_t h0 = half_bits(x0, dt), h1 = half_bits(x1, dt);
        if (e1 == e0 + 1) {
            *reinterpret_cast<uint32_t*>(p + e0) = (uint32_t)h0 | ((uint32_t)h1 << 16);
        } else {
            p[e0] = h0;
            p[e1] = h1;
        }
    }
}

// V tile block vb: 64 destination positions, aligned to 64 so that 8 positions
// never straddle a tile, times 64 channels (of one kv head: D is a multiple of
// 64).  Each thread's eight 8-byte loads go out together, from clamped, valid
// rows: one row per trip of a loop with the load under its bounds test was a
// memory round trip per trip, which launches of up to 700 tokens waited for
// (28 / 4 heads of 128, 300 tokens: 9.4 us, now 5.8).  The tile is stored
// transposed in LDS; 8 positions of one channel leave as one 16-byte store
// where all of them are stored rows and the cache allows it.
template <int D>
__device__ void v_tile_block(const RopeArgs& a, uint32_t vb)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    constexpr uint32_t TP = 66;  // halfs per channel: even, so words stay aligned; 33 words spread the banks
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * TP];
    const uint32_t ntx = a.n_kv * D / 64u;
    const uint32_t j0 = (vb % ntx) * 64u, p0 = (a.pos_start & ~63u) + (vb / ntx) * 64u;
    const uint32_t end = a.pos_start + a.B;
    const uint32_t c2 = (threadIdx.x & 31u) * 2u, r0 = threadIdx.x >> 5;  // channels c2, c2 + 1; rows r0, r0 + 8, ...
    f32x2 x[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) {
        const uint32_t pos = min(max(p0 + r0 + 8u * u, a.pos_start), end - 1u);
        x[u] = __builtin_nontemporal_load(
            reinterpret_cast<const f32x2*>(a.v + (size_t)(pos - a.pos_start) * a.v_stride + j0 + c2));
    }
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) {
        tile[c2 * TP + r0 + 8u * u] = f32_to_f16_ref(x[u][0]);
        tile[(c2 + 1) * TP + r0 + 8u * u] = f32_to_f16_ref(x[u][1]);
    }
    __syncthreads();
    const uint32_t h = j0 / D, d0 = j0 - h * D;
    const bool wide = ((uintptr_t)a.vc & 15u) == 0;
#pragma unroll
    for (uint32_t it = 0; it < 2; ++it) {
        const uint32_t g = threadIdx.x + 256u * it, dl = g >> 3, q0 = (g & 7u) * 8u, pos0 = p0 + q0;
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = *reinterpret_cast<const uint32_t*>(&tile[dl * TP + q0 + 2 * e]);
        uint16_t* dst = a.vc + v_index(h, pos0, d0 + dl, D, a.kv_stride);
        if (wide && pos0 >= a.pos_start && pos0 + 8u <= end) {
            *reinterpret_cast<u32x4*>(dst) = w;
        } else {
#pragma unroll
            for (uint32_t e = 0; e < 8; ++e)
                if (pos0 + e >= a.pos_start && pos0 + e < end) dst[e] = (uint16_t)(w[e / 2] >> (16 * (e & 1u)));
        }
    }
}

template <uint32_t KIND, int D>
__global__ __launch_bounds__(256) void rope_kv_kernel(RopeArgs a)
{
    // products and differences rounded separately, as the reference
#pragma clang fp contract(off)
    // the two roles alternate over the first 2 * min(rotation, tile) workgroups,
    // so the V tiles stream alongside the rotation instead of after it
    uint32_t blk = blockIdx.x;
    {
        const uint32_t m = min(a.rope_blocks, a.v_blocks);
        bool tile_role;
        if (blk < 2 * m) {
            tile_role = blk & 1u;
            blk >>= 1;
        } else {
            tile_role = a.v_blocks > a.rope_blocks;
            blk -= m;
        }
        if (tile_role) {  // workgroup-uniform
            v_tile_block<D>(a, blk);
            return;
        }
    }
    constexpr uint32_t P = D / 2;                  // pairs per head
    constexpr uint32_t HPI = P >= 64 ? 1 : 64 / P;  // heads per pass
    constexpr uint32_t PPL = P >= 64 ? P / 64 : 1;  // pairs per lane
    constexpr uint32_t U = 4;                      // passes whose loads are issued together
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = blk * 4u + (threadIdx.x >> 6);
    const uint32_t b = w / a.groups, g = w % a.groups;
    if (b >= a.B) return;  // wave-uniform; no barrier follows in this role
    const uint32_t pos = a.pos_start + b;
    const uint32_t sub = HPI > 1 ? lane / P : 0;

    uint32_t e0[PPL], e1[PPL];
    float c[PPL], s[PPL];
    bool rot[PPL];
#pragma unroll
    for (uint32_t r = 0; r < PPL; ++r) {
        const uint32_t p = HPI > 1 ? lane % P : lane + 64u * r;
        const uint32_t nr2 = a.n_rot / 2;
        if (KIND == kRopeHalf) {
            e0[r] = p;
            e1[r] = p + P;
            rot[r] = true;
        } else if (KIND == kRopeMrope && p < nr2) {
            e0[r] = p;
            e1[r] = p + nr2;
            rot[r] = true;
        } else {  // PAIRS, and the unrotated dims of MROPE / NONE
            e0[r] = 2 * p;
            e1[r] = 2 * p + 1;
            rot[r] = KIND == kRopePairs;
        }
        c[r] = 1.0f;
        s[r] = 0.0f;
        if (rot[r]) sincosf(a.freq[p] * (float)pos, &s[r], &c[r]);
    }

    // this wave's heads: [h_lo, h_hi) of q heads then kv heads (kv heads only without q_out)
    const uint32_t heads = a.n_heads + a.n_kv;
    const uint32_t h_first = a.q_out ? 0u : a.n_heads;
    const uint32_t h_lo = h_first + g * a.heads_per_wave;
    const uint32_t h_hi = min(heads, h_lo + a.heads_per_wave);
    for (uint32_t h0 = h_lo; h0 < h_hi; h0 += HPI * U) {
        // loads of U passes first, then their stores (q_out may be q: every
        // lane reads its own elements before it writes them)
        float x0[U][PPL], x1[U][PPL];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t h = h0 + u * HPI + sub;
            if (h >= h_hi) break;
            const bool is_q = h < a.n_heads;
            const float* src = is_q ? a.q + (size_t)b * a.q_stride + (size_t)h * D
                                    : a.k + (size_t)b * a.k_stride + (size_t)(h - a.n_heads) * D;
#pragma unroll
            for (uint32_t r = 0; r < PPL; ++r) {
                if (e1[r] == e0[r] + 1) {
                    typedef float f32x2_ __attribute__((ext_vector_type(2)));
                    const f32x2_ v = __builtin_nontemporal_load(reinterpret_cast<const f32x2_*>(src + e0[r]));
                    x0[u][r] = v[0];
                    x1[u][r] = v[1];
                } else {
                    x0[u][r] = __builtin_nontemporal_load(src + e0[r]);
                    x1[u][r] = __builtin_nontemporal_load(src + e1[r]);
                }
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t h = h0 + u * HPI + sub;
            if (h >= h_hi) break;
            const bool is_q = h < a.n_heads;
#pragma unroll
            for (uint32_t r = 0; r < PPL; ++r) {
                float y0 = x0[u][r], y1 = x1[u][r];
                if (rot[r]) {
                    y0 = x0[u][r] * c[r] - x1[u][r] * s[r];
                    y1 = x0[u][r] * s[r] + x1[u][r] * c[r];
                }
                if (is_q) {
                    store_q_pair(a.q_out, (size_t)b * a.q_out_stride + (size_t)h * D, e0[r], e1[r], a.q_out_dtype,
                                 y0, y1);
                } else {
                    uint16_t* row = a.kc + k_index(h - a.n_heads, pos, 0, D, a.kv_stride);
                    const uint16_t k0 = f32_to_f16_ref(y0), k1 = f32_to_f16_ref(y1);
                    if (e1[r] == e0[r] + 1) {
                        *reinterpret_cast<uint32_t*>(row + e0[r]) = (uint32_t)k0 | ((uint32_t)k1 << 16);
                    } else {
                        row[e0[r]] = k0;
                        row[e1[r]] = k1;
                    }
                }
            }
        }
    }
    if (a.B <= kScatterRows) {
        // few tokens: the token's waves write its V elements (2-byte scatters into the tiles)
        const uint32_t kv_dim = a.n_kv * D;
        for (uint32_t j = g * 64u + lane; j < kv_dim; j += 64u * a.groups) {
            const uint32_t h = j / D, d = j - h * D;
            a.vc[v_index(h, pos, d, D, a.kv_stride)] = f32_to_f16_ref(a.v[(size_t)b * a.v_stride + j]);
        }
    }
}

template <uint32_t KIND>
hipError_t launch_kind(const RopeArgs& a, dim3 grid, hipStream_t st)
{
    switch (a.D) {
    case 64: hipLaunchKernelGGL((rope_kv_kernel<KIND, 64>), grid, dim3(256), 0, st, a); break;
    case 128: hipLaunchKernelGGL((rope_kv_kernel<KIND, 128>), grid, dim3(256), 0, st, a); break;
    case 256: hipLaunchKernelGGL((rope_kv_kernel<KIND, 256>), grid, dim3(256), 0, st, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_rope_kv(RopeArgs a, hipStream_t st)
{
    // Passes (of hpi heads) per wave.  A wave reuses its token's sines and
    // cosines over all its passes and issues four passes' loads together, so
    // it takes a multiple of four; few waves with many passes leave too few
    // bytes in flight and drain unevenly.  So about 8192 waves, four to twelve
    // passes each (four at d 256, where a pass is two pairs per lane).  us at
    // 32 / 8 heads of 128 with 1 / 4 / 8 / 12 / 20 / 40 passes: 64 tokens 5.0 /
    // 5.0 / 5.5 / 6.0 / 7.8 / 11.7, 700 tokens 15.4 / 9.7 / 10.1 / 10.3 / 12.5 /
    // 18.6, 8191 tokens 129 / 67.5 / 58.5 / 58.9 / 60.4 / 68.8 (all heads in one
    // wave: before); 16 / 2 heads of 256 at 8191 (18 passes) 77 / 60.4 / 63.3 /
    // 68.3 / 82.  Up to kScatterRows tokens, which write V too, one pass.
    const uint32_t hpi = a.D >= 128 ? 1u : 64u / (a.D / 2);
    const uint32_t active = a.q_out ? a.n_heads + a.n_kv : a.n_kv;
    const uint32_t passes = (active + hpi - 1) / hpi;
    const uint32_t cap = a.D > 128 ? 4u : 12u;
    const uint64_t share = ((uint64_t)a.B * passes + 32767u) / 32768u * 4u;
    const uint32_t per0 = a.B <= kScatterRows ? 1u : share < cap ? (uint32_t)share : cap;
    const uint32_t groups = (passes + per0 - 1) / per0;
    const uint32_t per = (passes + groups - 1) / groups;  // passes per wave, evenly
    a.heads_per_wave = per * hpi;
    a.groups = (passes + per - 1) / per;
    a.rope_blocks = (uint32_t)(((uint64_t)a.B * a.groups + 3u) / 4u);
    a.v_blocks = a.B > kScatterRows ? a.n_kv * a.D / 64u * (((a.pos_start & 63u) + a.B + 63u) / 64u) : 0u;
    const dim3 grid(a.rope_blocks + a.v_blocks);
    switch (a.kind) {
    case kRopeNone: return launch_kind<kRopeNone>(a, grid, st);
    case kRopePairs: return launch_kind<kRopePairs>(a, grid, st);
    case kRopeHalf: return launch_kind<kRopeHalf>(a, grid, st);
    case kRopeMrope: return launch_kind<kRopeMrope>(a, grid, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace yhip
