// MultiHeadAttention core on already projected q / k / v (gfx950).
//
// Prefill shape (many query rows): one fused pass for head depths 32 / 64 / 128 (scores, softmax
// and P V on fp32 MFMA with the probabilities kept in registers); any other depth runs as
// scores = scale * Q K^T (one batched NT GEMM over (sequence, head)), row softmax in the
// reference's log-sum form with an optional causal prefix limit, then P V as a second batched
// NT GEMM against V^T.
// Decode shape (one query row per sequence): a dedicated HBM-bound kernel that streams
// the token-major key / value cache once.
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdlib>

#include "bf16_split.hpp"
#include "common.hpp"

namespace fdx {
fdx_status transpose_launch(const float* in, int batch, int rows, int cols, int64_t ld_in, int64_t in_batch, float* out);

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One workgroup per (sequence, head).  Phase 1: each thread owns keys j = tid, tid+256, ...
// and dots the query (LDS) with the key row (16-byte loads).  Phase 2: block max / sum,
// probabilities back to LDS.  Phase 3: lanes run along the value depth so each cached row
// is read as one contiguous run; 256/dv key partitions are combined through LDS.
__global__ __launch_bounds__(256) void mha_decode_kernel(const float* __restrict__ q, const float* __restrict__ kc,
    const float* __restrict__ vc, float* __restrict__ out, int heads, int dk, int dv, int len, int max_len, float scale)
{
    extern __shared__ float smem[]; // [dk] query, [len] scores, [256] reduction scratch
    float* sq = smem;
    float* sp = smem + dk;
    float* red = sp + len;
    const int b = blockIdx.x / heads, h = blockIdx.x % heads, tid = threadIdx.x;
    const int64_t krow = (int64_t)heads * dk, vrow = (int64_t)heads * dv;
    for (int d = tid; d < dk; d += 256)
        sq[d] = q[(int64_t)b * krow + h * dk + d];
    __syncthreads();
    float m = -FLT_MAX;
    for (int j = tid; j < len; j += 256) {
        const float* kr = kc + ((int64_t)b * max_len + j) * krow + h * dk;
        float s = 0.f;
        if ((dk & 3) == 0) {
            for (int d = 0; d < dk; d += 4) {
                const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + d);
                s += sq[d] * kv[0] + sq[d + 1] * kv[1] + sq[d + 2] * kv[2] + sq[d + 3] * kv[3];
            }
        } else {
            for (int d = 0; d < dk; ++d)
                s += sq[d] * kr[d];
        }
        s *= scale;
        sp[j] = s;
        m = fmaxf(m, s);
    }
    // block max
    for (int o = 32; o > 0; o >>= 1)
        m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((tid & 63) == 0)
        red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sum = 0.f;
    for (int j = tid; j < len; j += 256)
        sum += expf(sp[j] - m);
    for (int o = 32; o > 0; o >>= 1)
        sum += __shfl_xor(sum, o, 64);
    __syncthreads();
    if ((tid & 63) == 0)
        red[tid >> 6] = sum;
    __syncthreads();
    const float ls = logf(red[0] + red[1] + red[2] + red[3]);
    for (int j = tid; j < len; j += 256) {
        const float p = expf(sp[j] - m - ls);
        sp[j] = isinf(p) ? 0.f : p;
    }
    __syncthreads();
    // P V
    const int parts = dv <= 256 ? 256 / dv : 1;
    for (int d0 = 0; d0 < dv; d0 += 256) {
        const int d = d0 + (parts > 1 ? tid % dv : tid), part = parts > 1 ? tid / dv : 0;
        float acc = 0.f;
        if (d < dv && part < parts)
            for (int j = part; j < len; j += parts)
                acc += sp[j] * vc[((int64_t)b * max_len + j) * vrow + h * dv + d];
        if (parts > 1) {
            __syncthreads();
            red[tid] = acc;
            __syncthreads();
            if (tid < dv) {
                float r = red[tid];
                for (int pidx = 1; pidx < parts; ++pidx)
                    r += red[pidx * dv + tid];
                out[(int64_t)b * vrow + h * dv + tid] = r;
            }
        } else if (d < dv) {
            out[(int64_t)b * vrow + h * dv + d] = acc;
        }
    }
}

// ---- fused prefill attention: scores, softmax and P V in one pass, nothing but the output written --------------------
//
// Depth 128; depths 32 and 64 take flash_split_kernel below (its operands of depth 128 would not fit two waves per SIMD).
// One workgroup = 128 query rows of one (sequence, head), one wave = 32 of them; keys / values pass through LDS in
// tiles of 64.  The products are taken transposed on the 32x32x2 fp32 MFMA: S^T = K Q^T puts a query on a lane
// (column) and keys on the accumulator registers, so the running maximum, the running sum and the rescaling of the
// flash-attention recurrence are per-lane scalars, and the probabilities P^T are already laid out as the B operand of
// O^T = V^T P^T -- they never leave the registers.  The contraction index of either product may be visited in any
// order as long as both operands agree, which is what lets the accumulator layout (keys 8j + 4*half + i in register
// 4j + i) feed the second product directly.
//
// Softmax as the reference takes it (include/fdeep/tensor.hpp:1165-1192) is exp(x - max - log(sum exp(x - max)));
// here the running maximum replaces max and the division by the running sum comes last, which agrees to rounding.
struct FlashParams {
    const float* q; int64_t ldq, q_batch;
    const float* k; int64_t ldk, k_batch;
    const float* v; int64_t ldv, v_batch;
    float* out; int64_t ldo, o_batch;
    int t, s, heads, causal;
    float scale;
};

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int DK, int DV>
__global__ __launch_bounds__(256) void flash_prefill_kernel(FlashParams p)
{
    constexpr int KS = DK + 4;  // LDS row strides: 16-byte fragment reads along a key row stay conflict-free
    constexpr int VS = DV + 8;  // lanes read along the depth; rows 4 apart (the two lane halves) fall on disjoint banks
    constexpr int KL = DK / 16, VL = DV / 16; // 16-byte loads per thread for a 64-row tile
    __shared__ __attribute__((aligned(16))) float ks[64 * KS];
    __shared__ __attribute__((aligned(16))) float vs[64 * VS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, half = lane >> 5;
    const int b = blockIdx.y / p.heads, h = blockIdx.y % p.heads;
    const int q_first = blockIdx.x * 128;
    const int query = q_first + wave * 32 + c;
    const bool q_ok = query < p.t;
    const int shift = p.s - p.t; // causal: query i sees keys 0 .. i + shift

    // this lane's half of its query row: depth 8u + 4*half .. + 3, the same split the key fragments use
    f32x4 qreg[DK / 8];
    {
        const float* qrow = p.q + (int64_t)b * p.q_batch + (int64_t)(q_ok ? query : 0) * p.ldq + h * DK + 4 * half;
#pragma unroll
        for (int u = 0; u < DK / 8; ++u)
            qreg[u] = q_ok ? *reinterpret_cast<const f32x4*>(qrow + 8 * u) : f32x4 { 0.f, 0.f, 0.f, 0.f };
    }

    // keys this workgroup needs: all of them, or up to the last one its last query may see
    int s_end = p.s;
    if (p.causal) {
        const int q_last = (q_first + 128 < p.t ? q_first + 128 : p.t) - 1;
        s_end = q_last + shift + 1 < p.s ? q_last + shift + 1 : p.s;
    }
    const int tiles = (s_end + 63) / 64;
    const int wave_q_last = q_first + wave * 32 + 31;

    const float* kbase = p.k + (int64_t)b * p.k_batch + h * DK;
    const float* vbase = p.v + (int64_t)b * p.v_batch + h * DV;
    f32x4 kst[KL], vst[VL];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const int idx = tid + 256 * i, row = idx / (DK / 4), c4 = idx % (DK / 4);
            kst[i] = j0 + row < p.s ? *reinterpret_cast<const f32x4*>(kbase + (int64_t)(j0 + row) * p.ldk + 4 * c4)
                                     : f32x4 { 0.f, 0.f, 0.f, 0.f };
        }
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            const int idx = tid + 256 * i, row = idx / (DV / 4), c4 = idx % (DV / 4);
            vst[i] = j0 + row < p.s ? *reinterpret_cast<const f32x4*>(vbase + (int64_t)(j0 + row) * p.ldv + 4 * c4)
                                     : f32x4 { 0.f, 0.f, 0.f, 0.f };
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const int idx = tid + 256 * i, row = idx / (DK / 4), c4 = idx % (DK / 4);
            *reinterpret_cast<f32x4*>(&ks[row * KS + 4 * c4]) = kst[i];
        }
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            const int idx = tid + 256 * i, row = idx / (DV / 4), c4 = idx % (DV / 4);
            *reinterpret_cast<f32x4*>(&vs[row * VS + 4 * c4]) = vst[i];
        }
    };

    f32x16 oacc[DV / 32];
#pragma unroll
    for (int d = 0; d < DV / 32; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            oacc[d][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    if (tiles > 0)
        fetch(0);
    for (int tile = 0; tile < tiles; ++tile) {
        const int j0 = tile * 64;
        __syncthreads(); // every wave is done with the previous tile
        stage();
        __syncthreads();
        if (tile + 1 < tiles)
            fetch(j0 + 64); // in flight while this tile is worked on
        if (p.causal && j0 > wave_q_last + shift)
            continue; // nothing in this tile is visible to any of this wave's queries (wave-uniform)

        // S^T tile: 64 keys x 32 queries
        f32x16 sacc[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int e = 0; e < 16; ++e)
                sacc[kb][e] = 0.f;
#pragma unroll
            for (int u = 0; u < DK / 8; ++u) {
                const f32x4 kf = *reinterpret_cast<const f32x4*>(&ks[(kb * 32 + c) * KS + 8 * u + 4 * half]);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    sacc[kb] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qreg[u][e], sacc[kb], 0, 0, 0);
            }
        }
        // scale, mask, running maximum
        const int key_limit = p.causal ? (query + shift < p.s - 1 ? query + shift : p.s - 1) : p.s - 1;
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int key = j0 + kb * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
                const float sv = key <= key_limit ? sacc[kb][e] * p.scale : -INFINITY;
                sacc[kb][e] = sv;
                mx = fmaxf(mx, sv);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx);
        // a query that has seen no key yet (rows past the end of the sequence) keeps zeros instead of NaNs
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float corr = expf(m_run - m_use);
        float rs = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float pv = __expf(sacc[kb][e] - m_use);
                sacc[kb][e] = pv;
                rs += pv;
            }
        rs += __shfl_xor(rs, 32, 64);
        l_run = l_run * corr + rs;
        m_run = m_new;
#pragma unroll
        for (int d = 0; d < DV / 32; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                oacc[d][e] *= corr;
        // O^T += V^T P^T
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float* vrow = &vs[(kb * 32 + 8 * (e >> 2) + 4 * half + (e & 3)) * VS + c];
#pragma unroll
                for (int d = 0; d < DV / 32; ++d)
                    oacc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * d], sacc[kb][e], oacc[d], 0, 0, 0);
            }
    }

    if (q_ok) {
        const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
        float* orow = p.out + (int64_t)b * p.o_batch + (int64_t)query * p.ldo + h * DV + 4 * half;
#pragma unroll
        for (int d = 0; d < DV / 32; ++d)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 o = { oacc[d][4 * g] * inv, oacc[d][4 * g + 1] * inv, oacc[d][4 * g + 2] * inv, oacc[d][4 * g + 3] * inv };
                *reinterpret_cast<f32x4*>(orow + 32 * d + 8 * g) = o;
            }
    }
}

// The queries first + {bits of `odd`} of one (sequence, head) in plain fp32, over the keys that each may see, by one whole wave: four
// at a time, so that keys and values are read once for four.  A lane has a key's score, then a depth of the output.  A sum of
// probabilities that is NaN makes all of a query's outputs NaN: the walk ends where the four are.
template <int D>
__device__ __forceinline__ void flash_plain_queries(const FlashParams& p, int b, int h, int first, uint32_t odd)
{
    constexpr int G = 4, W = 64 / D; // queries at a time; keys per step of the output sums
    const int lane = threadIdx.x & 63, depth = lane % D, sub = lane / D;
    const float* kbase = p.k + (int64_t)b * p.k_batch + h * D;
    const float* vbase = p.v + (int64_t)b * p.v_batch + h * D + depth;
#pragma clang loop unroll(disable)
    while (odd) {
        const float* q[G];
        int query[G], limit[G], n = 0;
        float m[G], l[G], o[G], pr[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (odd) {
                query[g] = __builtin_amdgcn_readfirstlane(first + __builtin_ctz(odd));
                odd &= odd - 1;
                n = g + 1;
            } else {
                query[g] = query[g - 1 < 0 ? 0 : g - 1];
            }
            limit[g] = p.causal && query[g] + p.s - p.t < p.s - 1 ? query[g] + p.s - p.t : p.s - 1;
            q[g] = p.q + (int64_t)b * p.q_batch + (int64_t)query[g] * p.ldq + h * D;
            m[g] = -INFINITY;
            l[g] = o[g] = 0.f;
        }
        const int last = limit[G - 1]; // the largest: queries ascend
#pragma clang loop unroll(disable)
        for (int j0 = 0; j0 <= last; j0 += 64) {
            const int key = j0 + lane;
            const float* kp = kbase + (int64_t)(key < p.s ? key : p.s - 1) * p.ldk;
            float sc[G] = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll 4
            for (int d = 0; d < D; d += 4) {
                const f32x4 kv = *reinterpret_cast<const f32x4*>(kp + d);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const f32x4 qv = *reinterpret_cast<const f32x4*>(q[g] + d);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        sc[g] = fmaf(kv[e], qv[e], sc[g]);
                }
            }
            bool all_nan = true;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                sc[g] = key <= limit[g] ? sc[g] * p.scale : -INFINITY;
                float mx = sc[g];
                for (int w = 32; w > 0; w >>= 1)
                    mx = fmaxf(mx, __shfl_xor(mx, w, 64));
                const float m_new = fmaxf(m[g], mx), m_use = m_new == -INFINITY ? 0.f : m_new, corr = __expf(m[g] - m_use);
                pr[g] = __expf(sc[g] - m_use);
                float rs = pr[g];
                for (int w = 32; w > 0; w >>= 1)
                    rs += __shfl_xor(rs, w, 64);
                l[g] = l[g] * corr + rs;
                o[g] *= corr;
                m[g] = m_new;
                all_nan = all_nan && l[g] != l[g];
            }
            if (all_nan) {
#pragma unroll
                for (int g = 0; g < G; ++g)
                    o[g] = l[g];
                break;
            }
#pragma clang loop unroll(disable)
            for (int jj = 0; jj < 64 && j0 + jj <= last; jj += 4 * W) {
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int at = j0 + jj + u * W + sub;
                    v[u] = at <= last ? vbase[(int64_t)at * p.ldv] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int at = jj + u * W + sub;
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const float pj = __shfl(pr[g], at, 64);
                        o[g] = j0 + at <= limit[g] ? fmaf(pj, v[u], o[g]) : o[g];
                    }
                }
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (W == 2)
                o[g] += __shfl_xor(o[g], 32, 64);
            if (g < n && sub == 0)
                p.out[(int64_t)b * p.o_batch + (int64_t)query[g] * p.ldo + h * D + depth] = l[g] == 0.f ? 0.f : o[g] / l[g];
        }
    }
}

// The same recurrence with both products on the bf16 matrix instructions, every fp32 operand (queries, keys, values,
// probabilities) as the exact sum of three bf16 values and six of the nine partial products taken (see igemm_fast.hpp): the
// fp32 MFMA is what bounds the kernel above (its products alone are 8192 of a 64-key tile's cycles at depth 64; here 3072,
// beside about 2600 of vector instructions).  32 sequences of 256 tokens, 8 heads of 64: 54.5 -> 37.9 us a
// launch; error against 64-bit results (2-norm, unit operands) 3.3e-7 -> 1.4e-7.
//  * Keys and values are split on their way into LDS, once for the workgroup's 128 queries.  LDS holds blocks of eight
//    contraction indices: keys [plane][depth block][key][16 bytes], values [plane][key block][depth][16 bytes].
//  * Depth block 4 g + l holds depths 32 g + 4 l .. + 3 and 32 g + 16 + 4 l .. + 3, the two 16-byte chunks that lane l of four
//    fetches of a key row; a key block holds the eight keys whose probabilities one lane half has in eight consecutive
//    accumulator registers: 16 s + 4 half + {0 .. 3, 8 .. 11}.
//  * Scores and a tile's share of the output start from zero, small products first, and meet the running output in one
//    multiply-add (its rescaling), so sums are rounded at their own size a few times per tile.
//  * The scale of the scores is taken to base two, so a probability is one subtraction and one hardware exponential.  It also takes
//    back the factor of the split operands; the output keeps it until the end.
//  * A query whose result is not finite (infinite or NaN operands do not survive the split) is taken again in plain fp32: 32
//    sequences of 256 tokens, 8 heads of 64, finite 35 us, all NaN 87, one NaN key in each sequence 93 (7200 by one lane per query).
template <int D>
__global__ __launch_bounds__(256, 2) void flash_split_kernel(FlashParams p)
{
    constexpr int KB = D / 8;                // depth blocks
    constexpr int KBLK = 64 * 16 + 32, VBLK = D * 16 + 32; // bytes of a block: 64 keys / D depths, offset against each other
    constexpr int STEPS = D / 16;            // MFMA steps over the depth
    constexpr int KL = D / 32;               // pairs of 16-byte key loads per thread
    constexpr int VD = D / 32;               // depths per thread when values are staged
    static_assert(D == 32 || D == 64, "depths whose operands fit two waves per SIMD");
    __shared__ __attribute__((aligned(16))) unsigned char ks[3 * KB * KBLK];
    __shared__ __attribute__((aligned(16))) unsigned char vs[3 * 8 * VBLK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, half = lane >> 5;
    const int b = blockIdx.y / p.heads, h = blockIdx.y % p.heads;
    const int q_first = blockIdx.x * 128;
    const int query = q_first + wave * 32 + c;
    const bool q_ok = query < p.t;
    const int shift = p.s - p.t; // causal: query i sees keys 0 .. i + shift
    const float* qrow = p.q + (int64_t)b * p.q_batch + (int64_t)(q_ok ? query : 0) * p.ldq + h * D;

    u32x4 qf[STEPS][3];
#pragma unroll
    for (int u = 0; u < STEPS; ++u) { // depth block 2 u + half
        const int blk = 2 * u + half, d0 = 32 * (blk >> 2) + 4 * (blk & 3);
        f32x4 lo = { 0.f, 0.f, 0.f, 0.f }, hi = lo;
        if (q_ok) {
            lo = *reinterpret_cast<const f32x4*>(qrow + d0);
            hi = *reinterpret_cast<const f32x4*>(qrow + d0 + 16);
        }
        const float x[8] = { lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3] };
        split3x8(x, qf[u]);
    }

    int s_end = p.s;
    if (p.causal) {
        const int q_last = (q_first + 128 < p.t ? q_first + 128 : p.t) - 1;
        s_end = q_last + shift + 1 < p.s ? q_last + shift + 1 : p.s;
    }
    const int tiles = (s_end + 63) / 64;
    const int wave_q_first = q_first + wave * 32, wave_q_last = wave_q_first + 31;

    const float* kbase = p.k + (int64_t)b * p.k_batch + h * D;
    const float* vbase = p.v + (int64_t)b * p.v_batch + h * D;
    // keys: lane l of four has chunks l and 4 + l of each 32-float run of its key; values: VD depths of one block's eight keys
    const int krow = tid >> 2, kl = tid & 3;
    const int vblk = tid >> 5, vd = (tid & 31) * VD;
    f32x4 kst[KL][2];
    float vst[8][VD];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int g = 0; g < KL; ++g)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                kst[g][e] = j0 + krow < p.s ? *reinterpret_cast<const f32x4*>(kbase + (int64_t)(j0 + krow) * p.ldk + 32 * g + 16 * e + 4 * kl)
                                            : f32x4 { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int key = j0 + 16 * (vblk >> 1) + 4 * (vblk & 1) + 8 * (j >> 2) + (j & 3);
#pragma unroll
            for (int d = 0; d < VD; ++d)
                vst[j][d] = key < p.s ? vbase[(int64_t)key * p.ldv + vd + d] : 0.f;
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int g = 0; g < KL; ++g) {
            const float x[8] = { kst[g][0][0], kst[g][0][1], kst[g][0][2], kst[g][0][3], kst[g][1][0], kst[g][1][1], kst[g][1][2], kst[g][1][3] };
            u32x4 planes[3];
            split3x8(x, planes);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<u32x4*>(&ks[(q * KB + 4 * g + kl) * KBLK + krow * 16]) = planes[q];
        }
#pragma unroll
        for (int d = 0; d < VD; ++d) {
            const float x[8] = { vst[0][d], vst[1][d], vst[2][d], vst[3][d], vst[4][d], vst[5][d], vst[6][d], vst[7][d] };
            u32x4 planes[3];
            split3x8(x, planes);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<u32x4*>(&vs[(q * 8 + vblk) * VBLK + (vd + d) * 16]) = planes[q];
        }
    };
    auto mfma = [](const u32x4& a, const u32x4& bb, const f32x16& acc) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bb), acc, 0, 0, 0);
    };
    constexpr f32x16 kZero = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };

    f32x16 oacc[D / 32];
#pragma unroll
    for (int d = 0; d < D / 32; ++d)
        oacc[d] = kZero;
    const float scale2 = p.scale * 1.44269504088896340736f * kSplitDown;
    const int key_limit = p.causal ? (query + shift < p.s - 1 ? query + shift : p.s - 1) : p.s - 1;
    float m_run = -INFINITY, l_run = 0.f; // maximum in units of log2

    if (tiles > 0)
        fetch(0);
    for (int tile = 0; tile < tiles; ++tile) {
        const int j0 = tile * 64;
        __syncthreads(); // every wave is done with the previous tile
        stage();
        __syncthreads();
        if (tile + 1 < tiles)
            fetch(j0 + 64); // in flight while this tile is worked on
        if (p.causal && j0 > wave_q_last + shift)
            continue; // nothing in this tile is visible to any of this wave's queries (wave-uniform)

        // S^T tile: 64 keys x 32 queries
        f32x16 sacc[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            f32x16 lo = kZero, hi = kZero;
#pragma unroll
            for (int u = 0; u < STEPS; ++u) {
                u32x4 kf[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    kf[q] = *reinterpret_cast<const u32x4*>(&ks[(q * KB + 2 * u + half) * KBLK + (kb * 32 + c) * 16]);
                hi = mfma(kf[0], qf[u][0], hi);
                lo = mfma(kf[2], qf[u][0], lo);
                lo = mfma(kf[1], qf[u][1], lo);
                lo = mfma(kf[0], qf[u][2], lo);
                lo = mfma(kf[1], qf[u][0], lo);
                lo = mfma(kf[0], qf[u][1], lo);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e)
                sacc[kb][e] = (hi[e] + lo[e]) * scale2;
        }
        // mask where a query of this wave does not see the whole tile, running maximum
        if (j0 + 64 > p.s || (p.causal && j0 + 63 > wave_q_first + shift)) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (j0 + kb * 32 + 8 * (e >> 2) + 4 * half + (e & 3) > key_limit)
                        sacc[kb][e] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                mx = fmaxf(mx, sacc[kb][e]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx);
        // a query that has seen no key yet (rows past the end of the sequence) keeps zeros instead of NaNs
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float corr = __builtin_amdgcn_exp2f(m_run - m_use);
        float rs = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                sacc[kb][e] = __builtin_amdgcn_exp2f(sacc[kb][e] - m_use);
                rs += sacc[kb][e];
            }
        rs += __shfl_xor(rs, 32, 64);
        l_run = l_run * corr + rs;
        m_run = m_new;
        // O^T = O^T corr + V^T P^T
        f32x16 hi[D / 32], lo[D / 32];
#pragma unroll
        for (int d = 0; d < D / 32; ++d)
            hi[d] = lo[d] = kZero;
#pragma unroll
        for (int u = 0; u < 4; ++u) { // keys of block 2 u + half: registers 8 (u % 2) .. + 7 of half tile u / 2
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[j] = sacc[u >> 1][8 * (u & 1) + j];
            u32x4 pf[3];
            split3x8(x, pf);
#pragma unroll
            for (int d = 0; d < D / 32; ++d) {
                u32x4 vf[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    vf[q] = *reinterpret_cast<const u32x4*>(&vs[(q * 8 + 2 * u + half) * VBLK + (d * 32 + c) * 16]);
                hi[d] = mfma(vf[0], pf[0], hi[d]);
                lo[d] = mfma(vf[2], pf[0], lo[d]);
                lo[d] = mfma(vf[1], pf[1], lo[d]);
                lo[d] = mfma(vf[0], pf[2], lo[d]);
                lo[d] = mfma(vf[1], pf[0], lo[d]);
                lo[d] = mfma(vf[0], pf[1], lo[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < D / 32; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                oacc[d][e] = oacc[d][e] * corr + (hi[d][e] + lo[d][e]);
    }

    float size = l_run;
#pragma unroll
    for (int d = 0; d < D / 32; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            size += fabsf(oacc[d][e]);
    // the wave's queries whose result is not finite: the two lanes of a query hold half of its depths each
    const uint64_t odd_lanes = __ballot(q_ok && !(size < INFINITY));
    const uint32_t odd = (uint32_t)odd_lanes | (uint32_t)(odd_lanes >> 32);
    if (__builtin_expect(odd != 0, 0))
        flash_plain_queries<D>(p, b, h, wave_q_first, odd);
    if (q_ok && !((odd >> c) & 1)) {
        const float inv = l_run > 0.f ? kSplitDown / l_run : 0.f;
        float* orow = p.out + (int64_t)b * p.o_batch + (int64_t)query * p.ldo + h * D + 4 * half;
#pragma unroll
        for (int d = 0; d < D / 32; ++d)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 o = { oacc[d][4 * g] * inv, oacc[d][4 * g + 1] * inv, oacc[d][4 * g + 2] * inv, oacc[d][4 * g + 3] * inv };
                *reinterpret_cast<f32x4*>(orow + 32 * d + 8 * g) = o;
            }
    }
}

// The same products for launches with few queries in flight: one workgroup = 32 query rows of one (sequence, head), its
// four waves take every fourth block of 32 keys, each with a running maximum, sum and output of its own, and meet once at
// the end.  What bounds a short launch of the kernel above is one wave's serial walk over the keys (a block of 32 keys
// costs it D MFMAs of 64 cycles, 1.7 us at depth 64) and CUs without a workgroup: one sequence of 77 / 256 / 512 tokens
// with 8 heads of 64 takes 13.0 / 23.2 / 42.6 us there and 6.3 / 9.8 / 16.2 here (launches back to back).
// A wave stages its key / value block through a strip of LDS of its own, so the loop has no barrier; the next block's
// loads are in flight while a block is worked on.
template <int D>
__global__ __launch_bounds__(256) void flash_keysplit_kernel(FlashParams p)
{
    constexpr int KS = D + 4, VS = D + 8;  // as above
    constexpr int LD = D / 8;              // 16-byte loads per lane for a block of 32 rows
    constexpr int RPL = 256 / D;           // rows per load
    constexpr int STRIP = 32 * (KS + VS), OS = D + 4;
    __shared__ __attribute__((aligned(16))) float smem[4 * STRIP];
    __shared__ float part_m[4][32], part_l[4][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, half = lane >> 5;
    const int b = blockIdx.y / p.heads, h = blockIdx.y % p.heads;
    const int q_first = blockIdx.x * 32, query = q_first + c;
    const bool q_ok = query < p.t;
    const int shift = p.s - p.t; // causal: query i sees keys 0 .. i + shift
    float* ks = smem + wave * STRIP;
    float* vs = ks + 32 * KS;

    int s_end = p.s;
    if (p.causal) {
        const int q_last = (q_first + 32 < p.t ? q_first + 32 : p.t) - 1;
        s_end = q_last + shift + 1 < p.s ? q_last + shift + 1 : p.s;
    }
    const int blocks = (s_end + 31) / 32;

    const float* kbase = p.k + (int64_t)b * p.k_batch + h * D;
    const float* vbase = p.v + (int64_t)b * p.v_batch + h * D;
    const int lrow = lane / (D / 4), lcol = 4 * (lane % (D / 4));
    f32x4 kst[LD], vst[LD];
    auto fetch = [&](int blk) {
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            const int row = blk * 32 + i * RPL + lrow;
            kst[i] = vst[i] = f32x4 { 0.f, 0.f, 0.f, 0.f };
            if (row < p.s) {
                kst[i] = *reinterpret_cast<const f32x4*>(kbase + (int64_t)row * p.ldk + lcol);
                vst[i] = *reinterpret_cast<const f32x4*>(vbase + (int64_t)row * p.ldv + lcol);
            }
        }
    };
    if (wave < blocks)
        fetch(wave);

    // this lane's half of its query row: depth 8u + 4*half .. + 3, the same split the key fragments use
    f32x4 qreg[D / 8];
    {
        const float* qrow = p.q + (int64_t)b * p.q_batch + (int64_t)(q_ok ? query : 0) * p.ldq + h * D + 4 * half;
#pragma unroll
        for (int u = 0; u < D / 8; ++u)
            qreg[u] = q_ok ? *reinterpret_cast<const f32x4*>(qrow + 8 * u) : f32x4 { 0.f, 0.f, 0.f, 0.f };
    }

    f32x16 oacc[D / 32];
#pragma unroll
    for (int d = 0; d < D / 32; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            oacc[d][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    const int key_limit = p.causal ? (query + shift < p.s - 1 ? query + shift : p.s - 1) : p.s - 1;

    for (int blk = wave; blk < blocks; blk += 4) { // uniform over the wave
        // a wave's LDS accesses complete in order, so the strip needs no second buffer
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            *reinterpret_cast<f32x4*>(&ks[(i * RPL + lrow) * KS + lcol]) = kst[i];
            *reinterpret_cast<f32x4*>(&vs[(i * RPL + lrow) * VS + lcol]) = vst[i];
        }
        if (blk + 4 < blocks)
            fetch(blk + 4);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // S^T block: 32 keys x 32 queries
        f32x16 sacc;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            sacc[e] = 0.f;
#pragma unroll
        for (int u = 0; u < D / 8; ++u) {
            const f32x4 kf = *reinterpret_cast<const f32x4*>(&ks[c * KS + 8 * u + 4 * half]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qreg[u][e], sacc, 0, 0, 0);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int key = blk * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
            sacc[e] = key <= key_limit ? sacc[e] * p.scale : -INFINITY;
            mx = fmaxf(mx, sacc[e]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new; // no visible key yet
        const float corr = expf(m_run - m_use);
        float rs = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            sacc[e] = __expf(sacc[e] - m_use);
            rs += sacc[e];
        }
        rs += __shfl_xor(rs, 32, 64);
        l_run = l_run * corr + rs;
        m_run = m_new;
#pragma unroll
        for (int d = 0; d < D / 32; ++d)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                oacc[d][e] *= corr;
        // O^T += V^T P^T
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float* vrow = &vs[(8 * (e >> 2) + 4 * half + (e & 3)) * VS + c];
#pragma unroll
            for (int d = 0; d < D / 32; ++d)
                oacc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * d], sacc[e], oacc[d], 0, 0, 0);
        }
    }

    // the waves' shares meet: [query][depth] in the wave's own strip
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int d = 0; d < D / 32; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(&ks[c * OS + 32 * d + 8 * g + 4 * half])
                = f32x4 { oacc[d][4 * g], oacc[d][4 * g + 1], oacc[d][4 * g + 2], oacc[d][4 * g + 3] };
    if (half == 0) {
        part_m[wave][c] = m_run;
        part_l[wave][c] = l_run;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
        const int idx = tid + 256 * i, row = idx / (D / 4), col = 4 * (idx % (D / 4));
        if (q_first + row >= p.t)
            continue;
        float m = fmaxf(fmaxf(part_m[0][row], part_m[1][row]), fmaxf(part_m[2][row], part_m[3][row]));
        m = m == -INFINITY ? 0.f : m;
        float l = 0.f;
        f32x4 o = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float f = expf(part_m[w][row] - m);
            l += f * part_l[w][row];
            o += f * *reinterpret_cast<const f32x4*>(&smem[w * STRIP + row * OS + col]);
        }
        *reinterpret_cast<f32x4*>(p.out + (int64_t)b * p.o_batch + (int64_t)(q_first + row) * p.ldo + h * D + col)
            = o * (l > 0.f ? 1.0f / l : 0.f);
    }
}

// Which of the two, from 292 timed problems (4 to 16 heads of 32, 64 and 128, 1 to 64 sequences of 16 to 512 tokens, causal
// and not).  Up to 32 queries the kernel above has work for one of its four waves: 1.2 to 1.8 times faster here, at depth
// 128 (one workgroup per CU by LDS) as long as every CU takes one.  Beyond, a workgroup here reads keys and values for 32
// queries instead of 128, which shows as soon as CUs take turns: with one workgroup per CU 1.2 to 2.7 times faster; up to
// 448 with more than one 64-key tile 1.1 to 1.7 times (two keys' blocks only, 384 workgroups: 9.6 against 8.2 us); from 512
// on 0.6 to 1.3 times.  Against the split form at depths 32 and 64 (110 problems) the line lies in the same place: 1.0 to 1.9 times
// faster below it, 0.97 to 1.05 above.
static bool keysplit_better(const FlashParams& p, int batch, int d)
{
    const int64_t groups = (int64_t)((p.t + 31) / 32) * batch * p.heads;
    return groups <= 256 || (p.t <= 32 && d < 128) || (groups <= 448 && p.s > 64);
}

template <int DK, int DV>
static void flash_launch(const FlashParams& p, int batch)
{
    if (DK == DV && keysplit_better(p, batch, DK)) {
        hipLaunchKernelGGL(flash_keysplit_kernel<DK>, dim3((unsigned)((p.t + 31) / 32), (unsigned)(batch * p.heads)), dim3(256), 0, stream(), p);
        return;
    }
    const dim3 grid((unsigned)((p.t + 127) / 128), (unsigned)(batch * p.heads));
    if constexpr (DK == DV && DK <= 64)
        hipLaunchKernelGGL(flash_split_kernel<DK>, grid, dim3(256), 0, stream(), p);
    else
        hipLaunchKernelGGL((flash_prefill_kernel<DK, DV>), grid, dim3(256), 0, stream(), p);
}

static bool flash_enabled()
{
    static const bool on = [] {
        const char* e = std::getenv("FDX_FLASH");
        return !(e && e[0] == '0');
    }();
    return on;
}

// true when the fused kernel took the call
static bool flash_prefill(const FlashParams& p, int batch, int dk, int dv)
{
    if (!flash_enabled())
        return false;
    auto aligned = [](const void* ptr, int64_t ld, int64_t bs) {
        return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0 && (ld & 3) == 0 && (bs & 3) == 0;
    };
    if (!aligned(p.q, p.ldq, p.q_batch) || !aligned(p.k, p.ldk, p.k_batch) || !aligned(p.v, p.ldv, p.v_batch)
        || !aligned(p.out, p.ldo, p.o_batch))
        return false;
    profile_begin();
    if (dk == 64 && dv == 64)
        flash_launch<64, 64>(p, batch);
    else if (dk == 32 && dv == 32)
        flash_launch<32, 32>(p, batch);
    else if (dk == 128 && dv == 128)
        flash_launch<128, 128>(p, batch);
    else
        return false;
    const double pairs = p.causal ? (double)p.t * (p.s - p.t) + 0.5 * (double)p.t * (p.t + 1) : (double)p.t * p.s;
    profile_end("mha_flash_f32", 2.0 * batch * p.heads * pairs * (dk + dv),
        4.0 * batch * p.heads * ((double)p.t * (dk + dv) + (double)p.s * (dk + dv)));
    return true;
}

} // namespace fdx

using namespace fdx;

extern "C" size_t fdx_mha_scratch_bytes(int batch, int heads, int t, int s, int dv)
{
    return sizeof(float) * ((size_t)batch * heads * t * s + (size_t)batch * heads * dv * s) + 256;
}

namespace fdx {
// q/k/v/out rows may be strided (ld*) and sequences apart by *_batch elements, so the key/value
// operands can live in a token-major cache and q/k/v can be column blocks of one fused projection.
fdx_status mha_prefill_strided(const float* q, int64_t ldq, int64_t q_batch, const float* k, int64_t ldk, int64_t k_batch,
    const float* v, int64_t ldv, int64_t v_batch, int batch, int t, int s, int heads, int dk, int dv, int causal,
    float* out, int64_t ldo, int64_t o_batch, void* scratch_dev)
{
    FDX_REQUIRE(q && k && v && out && scratch_dev, "mha_prefill: null pointer");
    FDX_REQUIRE(batch > 0 && t > 0 && s > 0 && heads > 0 && dk > 0 && dv > 0, "mha_prefill: bad shape");
    FDX_REQUIRE(!causal || s >= t, "mha_prefill: causal attention needs at least as many keys as queries");
    FDX_REQUIRE((int64_t)batch * heads <= 65535, "mha_prefill: batch * heads too large");
    // 1 / sqrt(key_dim) applied to the scores after the product (multi_head_attention_layer.hpp:91-93)
    const float scale = (float)(1.0 / std::sqrt((double)dk));
    {
        FlashParams fp { q, ldq, q_batch, k, ldk, k_batch, v, ldv, v_batch, out, ldo, o_batch, t, s, heads, causal, scale };
        if (flash_prefill(fp, batch, dk, dv)) {
            FDX_LAUNCH_CHECK();
            return FDX_OK;
        }
    }
    float* scores = static_cast<float*>(scratch_dev);
    float* vt = scores + (((size_t)batch * heads * t * s + 3) & ~(size_t)3);
    const int64_t v_row = (int64_t)heads * dv;
    fdx_gemm_batch bt {};
    bt.batch = batch * heads;
    bt.inner = heads;
    bt.a_outer = q_batch; bt.a_inner = dk;
    bt.b_outer = k_batch; bt.b_inner = dk;
    bt.c_outer = (int64_t)heads * t * s; bt.c_inner = (int64_t)t * s;
    fdx_status st = fdx_gemm_bias_act_f32(q, ldq, k, ldk, t, s, dk, scale, nullptr, 0, nullptr, nullptr, scores, s, &bt);
    if (st != FDX_OK)
        return st;
    st = fdx_softmax_f32(scores, (int64_t)batch * heads * t, s, causal ? t : 0, causal ? s - t : 0, scores);
    if (st != FDX_OK)
        return st;
    st = transpose_launch(v, batch, s, (int)v_row, ldv, v_batch, vt); // [b][s][H*dv] -> [b][H*dv][s]
    if (st != FDX_OK)
        return st;
    bt.a_outer = (int64_t)heads * t * s; bt.a_inner = (int64_t)t * s;
    bt.b_outer = v_row * s; bt.b_inner = (int64_t)dv * s;
    bt.c_outer = o_batch; bt.c_inner = dv;
    return fdx_gemm_bias_act_f32(scores, s, vt, s, t, dv, s, 1.0f, nullptr, 0, nullptr, nullptr, out, ldo, &bt);
}
}

extern "C" fdx_status fdx_mha_prefill_f32(const float* q, const float* k, const float* v, int batch, int t, int s,
    int heads, int dk, int dv, int causal, float* out, void* scratch_dev)
{
    const int64_t qk = (int64_t)heads * dk, vr = (int64_t)heads * dv;
    return fdx::mha_prefill_strided(q, qk, t * qk, k, qk, s * qk, v, vr, s * vr, batch, t, s, heads, dk, dv, causal, out, vr,
        t * vr, scratch_dev);
}

extern "C" fdx_status fdx_mha_decode_f32(const float* q, const float* k_cache, const float* v_cache, int batch, int heads,
    int dk, int dv, int len, int max_len, float* out)
{
    FDX_REQUIRE(q && k_cache && v_cache && out, "mha_decode: null pointer");
    FDX_REQUIRE(batch > 0 && heads > 0 && dk > 0 && dv > 0 && len > 0 && len <= max_len, "mha_decode: bad shape");
    const size_t smem = sizeof(float) * ((size_t)dk + len + 256);
    FDX_REQUIRE(smem <= 64 * 1024, "mha_decode: context length %d exceeds the single-pass kernel's LDS budget", len);
    const float scale = (float)(1.0 / std::sqrt((double)dk));
    profile_begin();
    hipLaunchKernelGGL(mha_decode_kernel, dim3(batch * heads), dim3(256), smem, stream(), q, k_cache, v_cache, out, heads, dk,
        dv, len, max_len, scale);
    profile_end("mha_decode_f32", 4.0 * batch * heads * (double)len * dk,
        4.0 * ((double)batch * len * heads * (dk + dv) + (double)batch * heads * (dk + dv)));
    FDX_LAUNCH_CHECK();
    return FDX_OK;
}
