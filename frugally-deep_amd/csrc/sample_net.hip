// A small network as one launch (gfx950): every workgroup takes one sample through all layers, tensors, weights and offset
// tables in LDS.
//
// A network on 32 x 32 images of a few convolutions is a chain of launches of 1.5 to 8 us that each do a fraction of a
// microsecond of work on a few CUs.  Samples do not meet in any layer, so a workgroup can keep one to itself: what is left is one
// launch, the image's way in and the sample's arithmetic on one CU (fp32 MFMA, 256 multiply-adds a cycle).
//
//  * 16 waves, four per SIMD: a convolution is dealt out as 16-pixel x 16 or 32-channel tiles, each wave walks K on its own in short chains; with four
//    waves a SIMD's matrix pipe stays busy through the two dependent LDS reads in front of a product (offset, then pixel).
//  * the filter is the MFMA's row operand and the pixels its columns, so that a lane ends up with four neighbouring channels of
//    a pixel: 16-byte stores.
//  * an offset table takes the place of the walk over taps and channels: offset of every K element (of every four where the
//    channels are a multiple of four) from tap (0, 0).  Tensors whose readers pad lie inside a frame of zeros, so no tap is tested.
//  * a pixel's stride is an odd number of 16-byte pieces: 16 pixels side by side lie in different banks.
#include "sample_net.hpp"

#include <cfloat>

#include "igemm_params.hpp"

namespace fdx {

// x / d for x and d below 2^16, with ceil(2^32 / d) from the host (exact there: x times the ceiling's excess stays below 2^32)
__device__ __forceinline__ int quotient(int x, uint32_t by) { return by ? (int)__umulhi((uint32_t)x, by) : x; }

// positions in LDS: 24-bit products, a quarter of the 32-bit ones' time
__device__ __forceinline__ int product(int a, int b) { return (int)__umul24((unsigned)a, (unsigned)b); }
__device__ __forceinline__ int position(int y, int x, int row, int pix) { return product(y, row) + product(x, pix); }

// ReLU of N values.  Without slope and threshold one instruction a value, and one that finds what is not finite (0 * value is zero
// otherwise): that takes the general form, six a value.  With the 24-bit positions the small CNN's first convolution took 600 of 11300 cycles less.
template <int N>
__device__ __forceinline__ void sample_relu(const SampleStep& s, float* r)
{
    if (s.act_slope == 0.f && s.act_threshold == 0.f && s.act_max >= 0.f) {
        float odd = 0.f;
#pragma unroll
        for (int z = 0; z < N; ++z)
            odd = fmaf(r[z], 0.f, odd);
        if (!__any(odd != 0.f)) {
#pragma unroll
            for (int z = 0; z < N; ++z)
                r[z] = __builtin_amdgcn_fmed3f(r[z], 0.f, s.act_max);
            return;
        }
    }
#pragma unroll
    for (int z = 0; z < N; ++z) {
        const float low = r[z] >= s.act_threshold ? r[z] : s.act_slope * (r[z] - s.act_threshold);
        r[z] = r[z] >= s.act_max ? s.act_max : low;
    }
}

__device__ __forceinline__ void sample_frame(const SampleStep& s, float* lds, int t)
{
    // the frame of zeros around a tensor: its cells are nobody else's
    const int cells = s.frame_h * s.frame_w;
    for (int i = t; i < cells; i += kSampleThreads) {
        const int y = quotient(i, s.by_frame_w), x = i - product(y, s.frame_w);
        if ((unsigned)(y - s.frame_top) < (unsigned)s.out_h && (unsigned)(x - s.frame_left) < (unsigned)s.out_w)
            continue;
        float* p = lds + s.frame_base + position(y, x, s.out_row, s.out_pix);
        int c = 0;
        if (s.out_pix % 4 == 0)
            for (; c + 4 <= s.out_c; c += 4)
                *reinterpret_cast<f32x4*>(p + c) = f32x4 { 0.f, 0.f, 0.f, 0.f };
        for (; c < s.out_c; ++c)
            p[c] = 0.f;
    }
}

// items of MT x 16 pixels by NT x 16 channels, dealt out to the waves
template <bool VEC, int MT, int NT>
__device__ __forceinline__ void sample_conv(const SampleStep& s, float* lds, float* out, int t)
{
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), fr = lane & 15, fg = lane >> 4;
    const int pixels = s.out_h * s.out_w, m_items = (pixels + 16 * MT - 1) / (16 * MT), groups = s.n_tiles / NT;
    const int step_y = s.sy * s.in_row, step_x = s.sx * s.in_pix;
    const int* tab = reinterpret_cast<const int*>(lds) + s.tab + fg * s.tab_stride;
    int g = 0, mt = wave;
    for (; mt >= m_items && g < groups; ++g)
        mt -= m_items;
    while (g < groups) {
        const float* w = lds + s.weights + (g * NT * s.chunks * 64 + lane) * 4;
        f32x4 acc[MT][NT];
#pragma unroll
        for (int j = 0; j < NT; ++j)
            acc[0][j] = *reinterpret_cast<const f32x4*>(lds + s.bias + (g * NT + j) * 16 + fg * 4);
        int oy[MT], ox[MT];
        const float* a[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int m = (mt * MT + i) * 16 + fr, mm = m < pixels ? m : 0;
            oy[i] = quotient(mm, s.by_out_w);
            ox[i] = mm - product(oy[i], s.out_w);
            a[i] = lds + s.in_base + position(oy[i], ox[i], step_y, step_x);
        }
#pragma unroll
        for (int i = 1; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = acc[0][j];
        auto filter = [&](f32x4 (&wv)[NT], int kc) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
                wv[j] = *reinterpret_cast<const f32x4*>(w + (j * s.chunks + kc) * 256);
        };
        // One chain over all of K rounds the whole sum at every step: 2-norm error against 64 bits of 3x3 filters on 16 / 32 / 64 channels 2.1 /
        // 2.9 / 3.9 e-7, 1.2 / 1.3 / 1.6 as launches.  So a chunk's products start from zero, and chunks add up by fours before they join the
        // rest: 0.9 / 1.0 / 1.0 e-7, small CNN 17.35 -> 17.55 us a call.  (The chains of up to two tiles at once; of four they spill, two by two as well.)
        auto multiply = [&](const f32x4 (&av)[MT], const f32x4 (&wv)[NT], f32x4 (&sum)[MT][NT], bool first) {
            constexpr int SIDE = MT * NT <= 2 ? MT * NT : 1; // tiles side by side
#pragma unroll
            for (int z = 0; z < MT * NT; z += SIDE) {
                f32x4 part[SIDE];
#pragma unroll
                for (int q = 0; q < SIDE; ++q)
                    part[q] = f32x4 { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int q = 0; q < SIDE; ++q)
                        part[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[(z + q) % NT][e], av[(z + q) / NT][e], part[q], 0, 0, 0);
#pragma unroll
                for (int q = 0; q < SIDE; ++q)
                    sum[(z + q) / NT][(z + q) % NT] = first ? part[q] : sum[(z + q) / NT][(z + q) % NT] + part[q];
            }
        };
        auto join = [&](const f32x4 (&sum)[MT][NT]) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] += sum[i][j];
        };
        f32x4 av[MT], wv[NT], four[MT][NT];
        if (VEC) { // a lane's offsets of four chunks lie side by side
            int kc = 0;
            for (; kc + 4 <= s.whole; kc += 4) {
                const i32x4 off = *reinterpret_cast<const i32x4*>(tab + kc);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
#pragma unroll
                    for (int i = 0; i < MT; ++i)
                        av[i] = *reinterpret_cast<const f32x4*>(a[i] + off[u]);
                    filter(wv, kc + u);
                    multiply(av, wv, four, u == 0);
                }
                join(four);
            }
            if (kc < s.chunks) {
                const i32x4 off = *reinterpret_cast<const i32x4*>(tab + kc); // (the table's rows are whole fours of chunks)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (kc + u >= s.chunks)
                        break;
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        av[i] = *reinterpret_cast<const f32x4*>(a[i] + max(off[u], 0));
                        if (off[u] < 0) // beyond K: the filter is zero there, and what it meets must be finite
                            av[i] = f32x4 { 0.f, 0.f, 0.f, 0.f };
                    }
                    filter(wv, kc + u);
                    multiply(av, wv, four, u == 0);
                }
                join(four);
            }
        } else {
            for (int kc = 0; kc < s.whole; ++kc) {
                const i32x4 off = *reinterpret_cast<const i32x4*>(tab + kc * 4);
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    av[i] = f32x4 { a[i][off[0]], a[i][off[1]], a[i][off[2]], a[i][off[3]] };
                filter(wv, kc);
                multiply(av, wv, acc, false);
            }
            if (s.whole < s.chunks) {
                const i32x4 off = *reinterpret_cast<const i32x4*>(tab + s.whole * 4);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = a[i][max(off[e], 0)];
                        av[i][e] = off[e] < 0 ? 0.f : v;
                    }
                filter(wv, s.whole);
                multiply(av, wv, acc, false);
            }
        }
        float r[MT * NT * 4];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int n = (g * NT + j) * 16 + fg * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    r[(i * NT + j) * 4 + e] = acc[i][j][e];
                if (s.res_base >= 0)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < s.out_c)
                            r[(i * NT + j) * 4 + e] += lds[s.res_base + position(oy[i], ox[i], s.res_row, s.res_pix) + n + e];
            }
        if (s.act_kind == FDX_ACT_RELU) // (GELU is a step of its own)
            sample_relu<MT * NT * 4>(s, r);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int m = (mt * MT + i) * 16 + fr;
            if (m >= pixels)
                continue;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int n = (g * NT + j) * 16 + fg * 4;
                const float* v = r + (i * NT + j) * 4;
                if (n >= s.out_c)
                    continue;
                if (s.out_base >= 0 && s.out_pix % 4 == 0 && s.out_c % 4 == 0)
                    *reinterpret_cast<f32x4*>(lds + s.out_base + position(oy[i], ox[i], s.out_row, s.out_pix) + n) = f32x4 { v[0], v[1], v[2], v[3] };
                else {
                    float* o = s.out_base < 0 ? out + m * s.out_c : lds + s.out_base + position(oy[i], ox[i], s.out_row, s.out_pix);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < s.out_c)
                            o[n + e] = v[e];
                }
            }
        }
        for (mt += kSampleThreads / 64; mt >= m_items && g < groups; ++g)
            mt -= m_items;
    }
}

__device__ __forceinline__ float* sample_out(const SampleStep& s, float* lds, float* out, int y, int x)
{
    return s.out_base < 0 ? out + (y * s.out_w + x) * s.out_c : lds + s.out_base + position(y, x, s.out_row, s.out_pix);
}

// windows in the order of pool2d_kernel: cells outside the image count for neither the maximum nor the average
template <int VEC, bool MAX>
__device__ __forceinline__ void sample_pool(const SampleStep& s, float* lds, float* out, int t)
{
    const int cv = s.out_c / VEC, total = s.out_h * s.out_w * cv;
    for (int i = t; i < total; i += kSampleThreads) {
        const int pix = quotient(i, s.by_out_c), c = (i - product(pix, cv)) * VEC, oy = quotient(pix, s.by_out_w), ox = pix - product(oy, s.out_w);
        const int y = oy * s.sy - s.pad_top, x = ox * s.sx - s.pad_left;
        const int y0 = max(y, 0), y1 = min(y + s.kh, s.in_h), x0 = max(x, 0), x1 = min(x + s.kw, s.in_w);
        const float* p = lds + s.in_base + position(y0, x0, s.in_row, s.in_pix) + c;
        float val[VEC];
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            val[v] = MAX ? -FLT_MAX : 0.f;
        if (VEC == 4 && s.whole) { // 2 x 2 inside the image
            const f32x4 z[4] = { *reinterpret_cast<const f32x4*>(p), *reinterpret_cast<const f32x4*>(p + s.in_pix),
                *reinterpret_cast<const f32x4*>(p + s.in_row), *reinterpret_cast<const f32x4*>(p + s.in_row + s.in_pix) };
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    val[v] = either<MAX>(val[v], z[u][v]);
        } else
            for (int fy = y0; fy < y1; ++fy, p += s.in_row) {
                const float* q = p;
                for (int fx = x0; fx < x1; fx += 2, q += 2 * s.in_pix) { // two columns on their way at once
                    const float* q1 = fx + 1 < x1 ? q + s.in_pix : q;
                    float z[2][VEC];
                    if constexpr (VEC == 4) {
                        const f32x4 z0 = *reinterpret_cast<const f32x4*>(q), z1 = *reinterpret_cast<const f32x4*>(q1);
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            z[0][v] = z0[v];
                            z[1][v] = z1[v];
                        }
                    } else {
                        z[0][0] = q[0];
                        z[1][0] = q1[0];
                    }
#pragma unroll
                    for (int v = 0; v < VEC; ++v) {
                        val[v] = either<MAX>(val[v], z[0][v]);
                        val[v] = fx + 1 < x1 ? either<MAX>(val[v], z[1][v]) : val[v];
                    }
                }
            }
        const float count = (float)((y1 - y0) * (x1 - x0));
        float* o = sample_out(s, lds, out, oy, ox) + c;
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            val[v] = MAX ? val[v] : val[v] / count;
        if constexpr (VEC == 4)
            *reinterpret_cast<f32x4*>(o) = f32x4 { val[0], val[1], val[2], val[3] };
        else
            o[0] = val[0];
    }
}

// A matrix times one pixel: eight neighbouring lanes a row, weights as rows of a multiple of four.  On the matrix instructions
// fifteen of sixteen columns would be padding and K a serial chain: 32 -> 10 took 2400 cycles there.
__device__ __forceinline__ void sample_row(const SampleStep& s, float* lds, float* out, int t)
{
    const int k_all = s.in_c, stride = (k_all + 3) & ~3, l = t & 7;
    const float* x = lds + s.in_base;
    for (int n = t >> 3; n < s.out_c; n += kSampleThreads / 8) {
        const float* w = lds + s.weights + n * stride;
        float sum[2] = { 0.f, 0.f };
        if (s.vec) {
            for (int k = l * 4; k < k_all; k += 64) {
                const bool more = k + 32 < k_all;
                const f32x4 w0 = *reinterpret_cast<const f32x4*>(w + k), x0 = *reinterpret_cast<const f32x4*>(x + k);
                const f32x4 w1 = *reinterpret_cast<const f32x4*>(w + (more ? k + 32 : k)), x1 = *reinterpret_cast<const f32x4*>(x + (more ? k + 32 : k));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sum[0] = fmaf(w0[e], x0[e], sum[0]);
                    sum[1] = more ? fmaf(w1[e], x1[e], sum[1]) : sum[1];
                }
            }
        } else
            for (int k = l; k < k_all; k += 8)
                sum[0] = fmaf(w[k], x[k], sum[0]);
        float r = half_row_all<false>(sum[0] + sum[1]);
        if (l == 0) {
            r += lds[s.bias + n];
            if (s.res_base >= 0)
                r += lds[s.res_base + n];
            if (s.act_kind == FDX_ACT_RELU)
                sample_relu<1>(s, &r);
            (s.out_base < 0 ? out : lds + s.out_base)[n] = r;
        }
    }
}

// Lanes take the positions of a channel (vec: eight neighbouring lanes those of four channels), slots of them meet in LDS.
template <bool MAX>
__device__ __forceinline__ void sample_global_pool(const SampleStep& s, float* lds, float* out, int t)
{
    const int positions = s.in_h * s.in_w, c = s.in_c, most = s.vec ? kSampleThreads / 2 : kSampleThreads;
    float* scratch = lds + s.scratch;
    for (int c0 = 0; c0 < c; c0 += most) {
        // a power of two of lanes a slot, so that nothing is divided
        const int width = c - c0 < most ? c - c0 : most, log2w = width > 1 ? 32 - __builtin_clz((unsigned)width - 1) : 0;
        const int slots = most >> log2w;
        const float* p = lds + s.in_base + c0;
        if (s.vec) {
            const int octet = t >> 3, l = t & 7, ch = (octet << 2) & ((1 << log2w) - 1), slot = octet >> (log2w - 2);
            f32x4 val, v[2];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                val[e] = MAX ? -FLT_MAX : 0.f;
            if (ch < width) {
                for (int i = slot * 8 + l; i < positions; i += 16 * slots) {
                    const bool more = i + 8 * slots < positions;
                    v[0] = *reinterpret_cast<const f32x4*>(p + product(i, s.in_pix) + ch);
                    v[1] = *reinterpret_cast<const f32x4*>(p + product(more ? i + 8 * slots : i, s.in_pix) + ch);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        val[e] = either<MAX>(val[e], v[0][e]);
                        val[e] = more ? either<MAX>(val[e], v[1][e]) : val[e];
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    val[e] = half_row_all<MAX>(val[e]);
                if (l == 0)
                    *reinterpret_cast<f32x4*>(scratch + (slot << log2w) + ch) = val;
            }
        } else {
            const int slot = t >> log2w, ch = t & ((1 << log2w) - 1);
            float val = MAX ? -FLT_MAX : 0.f;
            if (ch < width)
                for (int i = slot; i < positions; i += 4 * slots) {
                    float v[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) { // a place beyond the end reads its first one again
                        const int at = i + u * slots < positions ? i + u * slots : i, y = quotient(at, s.by_in_w), x = at - product(y, s.in_w);
                        v[u] = p[position(y, x, s.in_row, s.in_pix) + ch];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        val = i + u * slots < positions ? either<MAX>(val, v[u]) : val;
                }
            scratch[t] = val;
        }
        __syncthreads();
        for (int i = t >> 3; i < width; i += kSampleThreads / 8) { // eight neighbouring lanes a channel
            float val = MAX ? -FLT_MAX : 0.f;
            for (int q = t & 7; q < slots; q += 16) {
                const bool more = q + 8 < slots;
                const float v0 = scratch[(q << log2w) + i], v1 = scratch[((more ? q + 8 : q) << log2w) + i];
                val = either<MAX>(val, v0);
                val = more ? either<MAX>(val, v1) : val;
            }
            val = half_row_all<MAX>(val);
            if ((t & 7) == 0)
                (s.out_base < 0 ? out : lds + s.out_base)[c0 + i] = MAX ? val : val / (float)positions;
        }
        if (c0 + most < c)
            __syncthreads();
    }
}

// a wave per pixel, in the reference's form exp(x - m - log sum) with infinite results as zero
__device__ __forceinline__ void sample_softmax(const SampleStep& s, float* lds, float* out, int t)
{
    const int lane = t & 63;
    for (int p = __builtin_amdgcn_readfirstlane(t >> 6); p < s.in_h * s.in_w; p += kSampleThreads / 64) {
        const int y = quotient(p, s.by_in_w), x = p - product(y, s.in_w);
        const float* v = lds + s.in_base + position(y, x, s.in_row, s.in_pix);
        float* o = sample_out(s, lds, out, y, x);
        float m = -FLT_MAX, sum = 0.f;
        for (int i = lane; i < s.in_c; i += 64)
            m = fmaxf(m, v[i]);
        m = wave_all<true>(m);
        for (int i = lane; i < s.in_c; i += 64)
            sum += expf(v[i] - m);
        const float ls = logf(wave_all<false>(sum));
        for (int i = lane; i < s.in_c; i += 64) {
            const float r = expf(v[i] - m - ls);
            o[i] = isinf(r) ? 0.f : r;
        }
    }
}

__device__ __forceinline__ void sample_activation(const SampleStep& s, float* lds, float* out, int t)
{
    const Act act { s.act_kind, s.act_max, s.act_slope, s.act_threshold };
    const int total = s.in_h * s.in_w * s.in_c;
    for (int i = t; i < total; i += kSampleThreads) {
        const int pix = quotient(i, s.by_out_c), c = i - product(pix, s.in_c), y = quotient(pix, s.by_in_w), x = pix - product(y, s.in_w);
        sample_out(s, lds, out, y, x)[c] = apply_act_full(lds[s.in_base + position(y, x, s.in_row, s.in_pix) + c], act);
    }
}

// What bounds it, on the small CNN of 32 x 32 x 3 (two 3x3 convolutions of 16 and 32 channels, pooling, classifier), cycles of a CU per
// sample: way in 5800, first convolution 10200 (matrix pipes 4100, the rest its scattered 4-byte reads and the epilogue), pooling 1900,
// second convolution 14000 (9200), global pooling 2600, Dense 1300, softmax 1700.  16.6 us a call for one sample and 17.5 up to 256, where
// seven launches take 24 and 59; 8192 samples 485 us, 906 as launches.  Image and input on their way together, Dense off the matrix
// instructions, 2 x 2 windows and pooled channels by fours took 1.2 us off it.  Nothing may go to scratch memory: 20 bytes a lane of it
// cost 7 us a launch.
__global__ __launch_bounds__(kSampleThreads) void sample_net_kernel(const float* __restrict__ in, float* __restrict__ out,
    const f32x4* __restrict__ image, int image_quads, const SampleStep* __restrict__ program, int steps, int in_volume, int out_volume, int batch)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int t = threadIdx.x;
    const bool quads = in_volume % 4 == 0; // (the input is 16-byte aligned)
    auto piece = [&](int b, int u) {
        const float* p = in + (int64_t)b * in_volume;
        const int i = (t + u * kSampleThreads) * 4;
        f32x4 v = { 0.f, 0.f, 0.f, 0.f };
        if (quads) {
            if (i < in_volume)
                v = *reinterpret_cast<const f32x4*>(p + i);
        } else
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (i + e < in_volume)
                    v[e] = p[i + e];
        return v;
    };
    auto place_piece = [&](const SampleStep& s, int u, const f32x4& v) {
        const int i = (t + u * kSampleThreads) * 4;
        if (i >= in_volume)
            return;
        const int pix = quotient(i, s.by_out_c);
        int y = quotient(pix, s.by_out_w), x = pix - product(y, s.out_w), c = i - product(pix, s.out_c);
        if (s.vec) {
            *reinterpret_cast<f32x4*>(lds + s.out_base + position(y, x, s.out_row, s.out_pix) + c) = v;
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (i + e < in_volume)
                lds[s.out_base + position(y, x, s.out_row, s.out_pix) + c] = v[e];
            if (++c == s.out_c) {
                c = 0;
                if (++x == s.out_w) {
                    x = 0;
                    ++y;
                }
            }
        }
    };
    // half a sample's registers on their way: the next one's trip runs under the current one's steps (all of it: spills)
    f32x4 pre[2];
    auto fetch = [&](int b) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
            pre[u] = piece(b, u);
    };
    auto place = [&](const SampleStep& s, int b) {
        if (in_volume > 8 * kSampleThreads) {
            const f32x4 v2 = piece(b, 2), v3 = piece(b, 3);
            place_piece(s, 2, v2);
            place_piece(s, 3, v3);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
            place_piece(s, u, pre[u]);
    };
    fetch(blockIdx.x);
    {
        // the first steps' lines into the scalar cache, all on their way at once
        int lines = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int* q = reinterpret_cast<const int*>(program + (i < steps ? i : 0));
            lines |= q[0] | q[16] | q[32];
        }
        asm volatile("" ::"s"(lines));
    }
    f32x4 first[2]; // the image's first pieces, on their way while the input's frame is cleared
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = t + u * kSampleThreads;
        first[u] = image[i < image_quads ? i : 0];
    }
    {
        const SampleStep s = program[0]; // Load
        if (s.frame_h > 0)
            sample_frame(s, lds, t);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (t + u * kSampleThreads < image_quads)
                reinterpret_cast<f32x4*>(lds)[t + u * kSampleThreads] = first[u];
        for (int i = t + 2 * kSampleThreads; i < image_quads; i += 4 * kSampleThreads) {
            f32x4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u] = image[i + u * kSampleThreads < image_quads ? i + u * kSampleThreads : i];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (i + u * kSampleThreads < image_quads)
                    reinterpret_cast<f32x4*>(lds)[i + u * kSampleThreads] = v[u];
        }
        place(s, blockIdx.x);
    }
    for (int b = blockIdx.x;;) {
        const int next = b + (int)gridDim.x;
        if (next < batch)
            fetch(next);
        __syncthreads();
        float* result = out + (int64_t)b * out_volume;
        for (int step = 1; step < steps; ++step) {
            const SampleStep s = program[step];
            // all of it at once: left alone, every branch below waits for its own fields
            asm volatile("" ::"s"(s.kind), "s"(s.out_base), "s"(s.frame_h), "s"(s.in_base), "s"(s.kh), "s"(s.tab), "s"(s.weights), "s"(s.res_base),
                "s"(s.scratch), "s"(s.act_threshold));
            if (s.frame_h > 0)
                sample_frame(s, lds, t);
            switch (s.kind) {
            case SampleStep::Conv:
                switch (s.form) {
                case 0: sample_conv<false, 1, 1>(s, lds, result, t); break;
                case 1: sample_conv<false, 4, 1>(s, lds, result, t); break;
                case 2: sample_conv<true, 1, 1>(s, lds, result, t); break;
                case 3: sample_conv<true, 4, 1>(s, lds, result, t); break;
                case 4: sample_conv<true, 1, 2>(s, lds, result, t); break;
                default: sample_conv<true, 2, 2>(s, lds, result, t); break;
                }
                break;
            case SampleStep::Pool:
                if (s.vec && s.mode == 0)
                    sample_pool<4, true>(s, lds, result, t);
                else if (s.vec)
                    sample_pool<4, false>(s, lds, result, t);
                else if (s.mode == 0)
                    sample_pool<1, true>(s, lds, result, t);
                else
                    sample_pool<1, false>(s, lds, result, t);
                break;
            case SampleStep::Row: sample_row(s, lds, result, t); break;
            case SampleStep::GlobalPool:
                if (s.mode == 0)
                    sample_global_pool<true>(s, lds, result, t);
                else
                    sample_global_pool<false>(s, lds, result, t);
                break;
            case SampleStep::Softmax: sample_softmax(s, lds, result, t); break;
            default: sample_activation(s, lds, result, t); break;
            }
            if (step + 1 < steps)
                __syncthreads();
        }
        if (next >= batch)
            return;
        b = next;
        __syncthreads(); // the input's place may be that of a tensor read last
        const SampleStep s = program[0];
        if (s.frame_h > 0)
            sample_frame(s, lds, t);
        place(s, b);
    }
}

SampleProgram::~SampleProgram()
{
    if (image)
        (void)hipFree(image);
}

int sample_net_cus()
{
    static const int cus = [] {
        int dev = 0, n = 256;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        return n;
    }();
    return cus;
}

fdx_status sample_net_launch(const SampleProgram& p, const float* in, int batch, float* out)
{
    FDX_REQUIRE(in && out && batch > 0 && p.image && p.in_volume <= kSampleInput && p.lds_floats <= kSampleLdsFloats
            && (reinterpret_cast<uintptr_t>(in) & 15) == 0, "sample net: bad arguments");
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(sample_net_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
        kSampleLdsFloats * 4);
    FDX_HIP(attr);
    const int cus = sample_net_cus();
    profile_begin();
    hipLaunchKernelGGL(sample_net_kernel, dim3((unsigned)(batch < cus ? batch : cus)), dim3(kSampleThreads), (size_t)p.lds_floats * 4, stream(),
        in, out, reinterpret_cast<const f32x4*>(p.image), p.image_floats / 4, p.program, p.steps, p.in_volume, p.out_volume, batch);
    profile_end("sample_net_f32", p.flops * batch, 4.0 * (p.image_floats + (double)batch * (p.in_volume + p.out_volume)));
    FDX_LAUNCH_CHECK();
    return FDX_OK;
}

} // namespace fdx
