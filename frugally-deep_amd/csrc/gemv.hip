// Dense layers on one to six activation rows (gfx950): the decode step of a few sequences.
//
// The tile kernels of decode_kernels.hip pad such rows to sixteen, turn them into matrix operands and add eight waves' tiles in LDS:
// barriers and chains of dependent instructions between the weights' arrival and the store, in a launch whose bytes need one to
// two microseconds.  Here a wave owns C output columns from end to end.  Weights lie row by row, so its loads are whole kilobytes
// of one column each; the row lies across its lanes, which multiply, add up and meet in the data-parallel primitives of the
// vector unit.  LayerNormalization's statistics come from the same registers while the weights are on their way (two passes, mean
// taken off before the product).  Up to K = 1024 nothing passes between waves; longer rows are cut between the four waves of a
// workgroup, which meet once in LDS.
#include <cmath>

#include "common.hpp"
#include "global_ptr.hpp"
#include "skinny.hpp"

namespace fdx {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// what the store needs (the arguments in front of it are in scalar registers when a wave starts)
struct GemvTail {
    const int* len_dev;
    float* ptr[3];
    int64_t ld[3], len_stride[3];
    int col[3], n_seg;
    Act act;
    float eps;
};

// A lane's output of a wave that owns M rows x C columns from n0 on: where it goes, and what is added in front of the activation.
struct GemvOutput {
    bool ok;
    float add;
    float* dst;
};
template <int M, int C>
__device__ __forceinline__ GemvOutput gemv_output(const float* bias, const float* residual, int m, int n, int ldr, const GemvTail& tail, int n0, int lane)
{
    const int r = lane / C, c = n0 + lane - r * C;
    GemvOutput o { lane < M * C && r < m && c < n, 0.f, nullptr };
    if (o.ok) {
        if (bias)
            o.add = as_global(bias)[c];
        if (residual)
            o.add += as_global(residual)[(int64_t)r * ldr + c];
        const int s = (tail.n_seg > 1 && c >= tail.col[1] ? 1 : 0) + (tail.n_seg > 2 && c >= tail.col[2] ? 1 : 0);
        o.dst = (s == 0 ? tail.ptr[0] : s == 1 ? tail.ptr[1] : tail.ptr[2]) + (int64_t)r * (s == 0 ? tail.ld[0] : s == 1 ? tail.ld[1] : tail.ld[2]) + c
            - (s == 0 ? tail.col[0] : s == 1 ? tail.col[1] : tail.col[2]);
        const int64_t stride = s == 0 ? tail.len_stride[0] : s == 1 ? tail.len_stride[1] : tail.len_stride[2];
        if (stride)
            o.dst += (int64_t)(*as_global(tail.len_dev)) * stride;
    }
    return o;
}

// the wave's sums over K, row r and column c in lane r * C + c
template <int M, int KQ, int C, typename Row>
__device__ __forceinline__ float gemv_sums(const f32x4 (&wa)[C][KQ], int lane, Row row)
{
    f32x4 s[M][C];
#pragma unroll
    for (int r = 0; r < M; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c)
            s[r][c] = f32x4 { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
    for (int q = 0; q < KQ; ++q)
#pragma unroll
        for (int r = 0; r < M; ++r) {
            const f32x4 x = row(r, q);
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s[r][c][e] += x[e] * wa[c][q][e];
        }
    float v = 0.f;
#pragma unroll
    for (int r = 0; r < M; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const float total = wave_all<false>((s[r][c][0] + s[r][c][1]) + (s[r][c][2] + s[r][c][3]));
            v = lane == r * C + c ? total : v;
        }
    return v;
}

// K up to 256 KQ: eight waves of a column each over the whole of K.  The first M waves bring a row each, centred and with its
// 1 / deviation where it is normalised, into LDS while all waves' weights are on their way: read by every wave for itself
// the rows took the path from L2 longer than the weights did.
constexpr int kGemvWaves = 8;
template <int M, int KQ, bool LN>
__global__ __launch_bounds__(64 * kGemvWaves) void gemv_kernel(const float* x, const float* w, const float* bias, const float* residual, int m, int n,
    int k, int ldx, int ldr, GemvTail tail)
{
    __shared__ f32x4 rows[M][KQ * 64];
    __shared__ float row_rstd[M];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = (int)blockIdx.x * kGemvWaves + wave;
    const f32x4 zero = { 0.f, 0.f, 0.f, 0.f };
    f32x4 xa[KQ], wa[1][KQ];
#pragma unroll
    for (int q = 0; q < KQ; ++q) {
        xa[q] = zero;
        if (wave < M && wave < m && (q * 64 + lane) * 4 < k)
            xa[q] = *reinterpret_cast<gptr<const f32x4>>(as_global(x) + (int64_t)wave * ldx + (q * 64 + lane) * 4);
    }
#pragma unroll
    for (int q = 0; q < KQ; ++q) {
        wa[0][q] = zero;
        if (n0 < n && (q * 64 + lane) * 4 < k) // every weight is used once per launch
            wa[0][q] = __builtin_nontemporal_load(reinterpret_cast<gptr<const f32x4>>(as_global(w) + (int64_t)n0 * k + (q * 64 + lane) * 4));
    }
    const GemvOutput o = gemv_output<M, 1>(bias, residual, m, n, ldr, tail, n0, lane);
    if (wave < M) {
        if (LN) {
            float s = 0.f;
#pragma unroll
            for (int q = 0; q < KQ; ++q)
                s += (xa[q][0] + xa[q][1]) + (xa[q][2] + xa[q][3]);
            const float mean = wave_all<false>(s) / (float)k;
            float dev = 0.f;
#pragma unroll
            for (int q = 0; q < KQ; ++q) {
                const float off = (q * 64 + lane) * 4 < k ? mean : 0.f; // places beyond the row hold zeros and stay zero
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xa[q][e] -= off;
                    dev += xa[q][e] * xa[q][e];
                }
            }
            const float rstd = 1.0f / sqrtf(wave_all<false>(dev) / (float)k + tail.eps);
            if (lane == 0)
                row_rstd[wave] = rstd;
        }
#pragma unroll
        for (int q = 0; q < KQ; ++q)
            rows[wave][q * 64 + lane] = xa[q];
    }
    __syncthreads();
    float v = gemv_sums<M, KQ, 1>(wa, lane, [&](int r, int q) { return rows[r][q * 64 + lane]; });
    if (o.ok) {
        if (LN)
            v *= row_rstd[lane];
        *as_global(o.dst) = apply_act(v + o.add, tail.act);
    }
}

// Longer rows: the four waves of a workgroup take a quarter of K each, of the same C columns.
template <int M, int KQ, int C>
__global__ __launch_bounds__(256) void gemv_split_kernel(const float* x, const float* w, const float* bias, const float* residual, int m, int n, int k,
    int ldx, int ldr, GemvTail tail)
{
    __shared__ float part[4][M * C];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = (int)blockIdx.x * C, k0 = wave * KQ * 256 + lane * 4;
    const f32x4 zero = { 0.f, 0.f, 0.f, 0.f };
    f32x4 xa[M][KQ], wa[C][KQ];
#pragma unroll
    for (int r = 0; r < M; ++r)
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            xa[r][q] = zero;
            if (r < m && k0 + q * 256 < k)
                xa[r][q] = *reinterpret_cast<gptr<const f32x4>>(as_global(x) + (int64_t)r * ldx + k0 + q * 256);
        }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            wa[c][q] = zero;
            if (n0 + c < n && k0 + q * 256 < k)
                wa[c][q] = __builtin_nontemporal_load(reinterpret_cast<gptr<const f32x4>>(as_global(w) + (int64_t)(n0 + c) * k + k0 + q * 256));
        }
    GemvOutput o { false, 0.f, nullptr };
    if (wave == 0)
        o = gemv_output<M, C>(bias, residual, m, n, ldr, tail, n0, lane);
    float v = gemv_sums<M, KQ, C>(wa, lane, [&](int r, int q) { return xa[r][q]; });
    if (lane < M * C)
        part[wave][lane] = v;
    __syncthreads();
    if (o.ok) {
        v = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
        *as_global(o.dst) = apply_act(v + o.add, tail.act);
    }
}

constexpr int kGemvRows = 6, kGemvK = 4096; // most rows and longest K

// (a grid has fewer than 2^32 threads: 256 a column at most)
bool gemv_covers(int m, int n, int k, int64_t ldx, int64_t ldw, int64_t ldr, bool ln)
{
    return m > 0 && m <= kGemvRows && n > 0 && n < (1 << 24) && k > 0 && k % 4 == 0 && k <= (ln ? 1024 : kGemvK) && ldw == k && ldx < (1LL << 31)
        && ldr < (1LL << 31);
}

// Not where the wide-output kernel strides over thousands of columns, nor with the embedding prologue.  A step of 12 layers of 768, us, tile
// kernels / here: 1 row 322 / 248, 2 331 / 270, 3 337 / 297, 4 345 / 301, 6 350 / 327, 7 351 / 350, 8 353 / 359.  Of 6 layers, 1 and 6 rows: width 64
// 138 / 101 and 140 / 119, 128 140 / 103 and 144 / 122, 256 150 / 109 and 155 / 133, 512 160 / 119 and 166 / 145, 1024 208 / 162 and 219 /
// 217.  Single launches on weights row by row, K 16 to 4096 x N 64 to 12288 x 1 to 6 rows: 0.39 to 0.96 of the tile kernels' time in 575 of
// 576 (32 x 12288 with six rows 1.01); also where few lanes hold any of K: 16 x 64, one row 2.3 / 4.3, six 2.8 / 3.8, 64 x 4096, six 3.5 / 4.5.
bool gemv_by_rule(const SkinnyParams& p)
{
    return p.M <= kGemvRows && !p.emb_x && !p.emb_res && !p.amax_parts && gemv_covers(p.M, p.N, p.K, p.ldx, p.ldw, p.ldr, p.ln != 0) && skinny_wide_grid(p) == 0;
}

template <int M, int KQ>
static void gemv_start(const SkinnyParams& p, const GemvTail& tail)
{
    const dim3 grid((unsigned)((p.N + kGemvWaves - 1) / kGemvWaves)), block(64 * kGemvWaves);
    if (p.K > 1024) {
        // A column a workgroup; three from three rows on, which then share the reading of the rows (a step of 12 layers of 768 with 1 / 2 / 3
        // columns, us: one row 248 / 252 / 252, four rows 302 / 303 / 299, six 332 / 332 / 327).
        constexpr int C = M > 2 ? 3 : 1;
        hipLaunchKernelGGL((gemv_split_kernel<M, KQ, C>), dim3((unsigned)((p.N + C - 1) / C)), dim3(256), 0, stream(), p.X, p.W, p.bias, p.residual, p.M,
            p.N, p.K, (int)p.ldx, (int)p.ldr, tail);
    } else if (p.ln) // (whole rows: a column a wave; with two everywhere that step took 274, 330 and 357 us)
        hipLaunchKernelGGL((gemv_kernel<M, KQ, true>), grid, block, 0, stream(), p.X, p.W, p.bias, p.residual, p.M, p.N, p.K, (int)p.ldx, (int)p.ldr, tail);
    else
        hipLaunchKernelGGL((gemv_kernel<M, KQ, false>), grid, block, 0, stream(), p.X, p.W, p.bias, p.residual, p.M, p.N, p.K, (int)p.ldx, (int)p.ldr, tail);
}

template <int M>
static void gemv_k(const SkinnyParams& p, const GemvTail& tail)
{
    const int per = p.K > 1024 ? (p.K + 3) / 4 : p.K; // of K a wave
    if (per <= 256)
        gemv_start<M, 1>(p, tail);
    else if (per <= 512)
        gemv_start<M, 2>(p, tail);
    else if (per <= 768)
        gemv_start<M, 3>(p, tail);
    else
        gemv_start<M, 4>(p, tail);
}

// Launches the rows' kernel for parameters that gemv_covers accepts.
void gemv_launch(const SkinnyParams& p)
{
    GemvTail t;
    t.len_dev = p.len_dev;
    t.n_seg = p.n_seg;
    t.act = p.act;
    t.eps = p.ln_eps;
    for (int i = 0; i < 3; ++i) {
        const SkinnySegment& s = p.seg[i < p.n_seg ? i : 0];
        t.ptr[i] = s.ptr;
        t.ld[i] = s.ld;
        t.len_stride[i] = s.len_stride;
        t.col[i] = s.col_begin;
    }
    switch (p.M) {
    case 1: gemv_k<1>(p, t); break;
    case 2: gemv_k<2>(p, t); break;
    case 3: case 4: gemv_k<4>(p, t); break;
    default: gemv_k<6>(p, t); break;
    }
}

} // namespace fdx

extern "C" int fdx_debug_dense_rows_form(int m, int n, int k, int layernorm)
{
    fdx::SkinnyParams p {};
    p.M = m; p.N = n; p.K = k; p.ldx = p.ldw = k; p.ldr = n; p.ln = layernorm;
    return fdx::gemv_by_rule(p) ? 1 : 0;
}
