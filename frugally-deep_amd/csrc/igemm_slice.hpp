// Problems with few output tiles (included inside namespace fdx by igemm.hip after igemm_fast.hpp): a network at batch 1,
// short sequences, the last stages of a small batch.
//
// There the tiled kernel leaves most of the chip idle: a 64 x 64 tile of a 14 x 14 map walks K = 2304 slab by slab, each
// slab a round trip to memory, an LDS pass and a barrier (one image, weights out of memory, per launch: 14 x 14 3x3
// 256 -> 256 19.6 us, 1x1 1024 -> 256 13.6, 7 x 7 3x3 512 -> 512 26.8; here 8.0, 4.6, 10.4, of which 3.5 are the launch
// itself; ResNet50 at batch 1 761 -> 330 us).  What bounds it is the path from L2 into a CU.  Here the eight (or four) waves
// of a workgroup share one small output tile and cut its K range between them, every wave on its own:
//
//  * a wave loads its units (UK consecutive k of all tile rows) as runs of 64 or 128 bytes per row, DEPTH units in flight from
//    the first instruction on, and turns them into MFMA operands through a strip of LDS of its own: no barrier in the loop.
//    (Loaded straight in operand order, 16x16x4 MFMA's neighbouring lanes lie in different rows, which the address unit
//    takes one lane at a time: 77 cycles per 16-byte load and CU measured, whatever the rows' pitch.)
//  * the waves' partial tiles meet once in LDS and are added in wave order (the sum does not depend on timing), the
//    epilogue runs on the sum.  Bias and residual are requested in front of the K walk.
//  * tiles are numbered so that an XCD owns neighbours that share the larger operand's rows: it passes through one L2.

// f with n, at most MOST, as a compile-time constant
template <int MOST, typename F>
__device__ __forceinline__ void by_count(int n, F&& f)
{
    if constexpr (MOST > 0) {
        if (n == MOST)
            f(std::integral_constant<int, MOST>());
        else
            by_count<MOST - 1>(n, f);
    } else
        f(std::integral_constant<int, 0>());
}

template <int TM, int TN, int NW, int UK, bool CONV, bool DUAL, bool SEG = false>
__global__ __launch_bounds__(64 * NW) void igemm_slice_kernel(GemmParams p)
{
    constexpr int BM = 16 * TM, BN = 16 * TN;
    constexpr int CPR = UK / 4, RPI = 64 / CPR;         // 16-byte chunks per row and unit; rows per load instruction
    constexpr int AL = BM / RPI, BL = BN / RPI;         // load instructions per unit
    constexpr int DEPTH = AL + BL <= 2 ? 8 : AL + BL <= 4 ? 4 : AL + BL <= 8 ? 2 : 1; // units in flight: up to 64 registers
    constexpr int US = UK + 4, RS = BN + 4;             // LDS rows: a staged unit, a partial tile
    constexpr int STRIP = (BM + BN) * US > BM * RS ? (BM + BN) * US : BM * RS;
    constexpr uint32_t OOB = 0x80000000u;
    static_assert(!DUAL || !CONV, "two sources: GEMM form only");
    static_assert(!SEG || (!CONV && !DUAL), "segmented outputs: GEMM form only");
    __shared__ __attribute__((aligned(16))) float smem[NW * STRIP];

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const int lrow = lane / CPR, lchunk = lane % CPR;
    float* strip = smem + wave * STRIP;
    const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
    int id = blockIdx.x;
    {
        const int total = tiles_m * tiles_n, xcd = id & 7, per = total >> 3, rem = total & 7;
        id = xcd * per + (xcd < rem ? xcd : rem) + (id >> 3);
    }
    int mt, nt;
    if (p.M >= p.N) {
        mt = id / tiles_n;
        nt = id - mt * tiles_n;
    } else {
        nt = id / tiles_m;
        mt = id - nt * tiles_m;
    }
    const int m0 = mt * BM, n0 = nt * BN;

    uint32_t a_voff[AL], a2_voff[DUAL ? AL : 1], b_voff[BL];
    int a_y[CONV ? AL : 1], a_x[CONV ? AL : 1]; // where tap (0, 0) of a row lies in the image
#pragma unroll
    for (int i = 0; i < AL; ++i) {
        const int m = m0 + i * RPI + lrow;
        a_voff[i] = OOB;
        a_y[CONV ? i : 0] = a_x[CONV ? i : 0] = -(1 << 30);
        if (DUAL)
            a2_voff[i] = OOB;
        if (m < p.M) {
            if (CONV) {
                const int img = m / (p.OH * p.OW), rm = m - img * (p.OH * p.OW);
                const int oy = rm / p.OW, ox = rm - oy * p.OW;
                a_y[CONV ? i : 0] = oy * p.sy - p.pad_top;
                a_x[CONV ? i : 0] = ox * p.sx - p.pad_left;
                a_voff[i] = (uint32_t)(((img * p.H + oy * p.sy) * p.W + ox * p.sx) * p.pix_stride) * 4u + lchunk * 16;
            } else {
                a_voff[i] = (uint32_t)((int64_t)m * p.lda) * 4u + lchunk * 16;
                if (DUAL) {
                    const int img = m / (p.OH * p.OW), rm = m - img * (p.OH * p.OW);
                    const int oy = rm / p.OW, ox = rm - oy * p.OW;
                    a2_voff[DUAL ? i : 0] = (uint32_t)(((img * p.H2 + oy * p.s2y) * p.W2 + ox * p.s2x) * p.C2) * 4u + lchunk * 16;
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < BL; ++j) {
        const int n = n0 + j * RPI + lrow;
        b_voff[j] = n < p.N ? (uint32_t)((int64_t)n * p.ldb) * 4u + lchunk * 16 : OOB;
    }

    // this wave's units of UK k
    const int units = p.K / UK;
    const int u_lo = (int)((int64_t)units * wave / NW), u_n = (int)((int64_t)units * (wave + 1) / NW) - u_lo;
    int soff_b = u_lo * (UK * 4), soff_a = soff_b, fx = 0, fy = 0, c0 = 0;
    if (CONV) {
        const int k = u_lo * UK;
        const int tap = k / p.Cin;
        c0 = k - tap * p.Cin;
        fy = tap / p.kw;
        fx = tap - fy * p.kw;
        soff_a = ((fy * p.dy * p.W + fx * p.dx) * p.pix_stride + c0) * 4;
    }
    f32x4 ra[DEPTH][AL], rb[DEPTH][BL];
    uint32_t a_eff[CONV ? AL : 1]; // a_voff under the current filter tap: out of range where the tap lies outside the image
    // (compared at each tap: a mask of all taps, made in front of the first load, held that up; 3 x 3 launches of ResNet50 on one image 10.2 and 9.6 us with it, 8.4 and 7.2 without)
    auto enter_tap = [&]() {
        if (CONV) {
#pragma unroll
            for (int i = 0; i < AL; ++i) {
                const bool inside = (unsigned)(a_y[CONV ? i : 0] + fy * p.dy) < (unsigned)p.H && (unsigned)(a_x[CONV ? i : 0] + fx * p.dx) < (unsigned)p.W;
                a_eff[CONV ? i : 0] = inside ? a_voff[i] : OOB;
            }
        }
    };
    enter_tap();
    auto issue = [&](int d) {
        const __amdgpu_buffer_rsrc_t srd_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.B), 0, (int)p.b_records, 0x00020000);
        if (DUAL && soff_b >= p.K1 * 4) {
            const __amdgpu_buffer_rsrc_t srd_a2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A2), 0, (int)p.a2_records, 0x00020000);
#pragma unroll
            for (int i = 0; i < AL; ++i)
                ra[d][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_a2, (int)a2_voff[DUAL ? i : 0], soff_b - p.K1 * 4, 0));
        } else {
            const __amdgpu_buffer_rsrc_t srd_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A), 0, (int)p.a_records, 0x00020000);
#pragma unroll
            for (int i = 0; i < AL; ++i)
                ra[d][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_a, (int)(CONV ? a_eff[CONV ? i : 0] : a_voff[i]), soff_a, 0));
        }
#pragma unroll
        for (int j = 0; j < BL; ++j)
            rb[d][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_b, (int)b_voff[j], soff_b, 0));
        soff_b += UK * 4;
        if (CONV) {
            c0 += UK;
            if (c0 == p.Cin) {
                c0 = 0;
                if (++fx == p.kw) {
                    fx = 0;
                    ++fy;
                }
                enter_tap();
            }
            soff_a = ((fy * p.dy * p.W + fx * p.dx) * p.pix_stride + c0) * 4;
        } else {
            soff_a += UK * 4;
        }
    };
    // what the epilogue reads, requested behind the first operands
    constexpr int QUADS = BM * BN / 4, QPT = (QUADS + 64 * NW - 1) / (64 * NW);
    f32x4 bias4[QPT], res4[QPT];
    auto request_epilogue = [&]() {
#pragma unroll
        for (int q = 0; q < QPT; ++q) {
            const int quad = t + q * 64 * NW, row = quad / (BN / 4), col = (quad % (BN / 4)) * 4;
            const bool ok = quad < QUADS && m0 + row < p.M && n0 + col < p.N; // N is a multiple of 4 on this path
            bias4[q] = res4[q] = f32x4 { 0.f, 0.f, 0.f, 0.f };
            if (ok && p.bias)
                bias4[q] = *reinterpret_cast<const f32x4*>(p.bias + n0 + col);
            if (ok && p.residual)
                res4[q] = *reinterpret_cast<const f32x4*>(p.residual + (int64_t)(m0 + row) * p.ldc + n0 + col);
        }
    };
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            acc[i][j] = f32x4 { 0.f, 0.f, 0.f, 0.f };
    auto take = [&](int d, auto more) {
        // a wave's LDS accesses complete in order, so the strip needs no second buffer
#pragma unroll
        for (int i = 0; i < AL; ++i)
            *reinterpret_cast<f32x4*>(&strip[(i * RPI + lrow) * US + lchunk * 4]) = ra[d][i];
#pragma unroll
        for (int j = 0; j < BL; ++j)
            *reinterpret_cast<f32x4*>(&strip[(BM + j * RPI + lrow) * US + lchunk * 4]) = rb[d][j];
        if (more())
            issue(d);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        f32x4 af[TM][UK / 16], bf[TN][UK / 16];
#pragma unroll
        for (int h = 0; h < UK / 16; ++h) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
                af[i][h] = *reinterpret_cast<const f32x4*>(&strip[(i * 16 + fr) * US + h * 16 + fg * 4]);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                bf[j][h] = *reinterpret_cast<const f32x4*>(&strip[(BM + j * 16 + fr) * US + h * 16 + fg * 4]);
        }
#pragma unroll
        for (int h = 0; h < UK / 16; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i][h][e], bf[j][h][e], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // No load is issued for a unit beyond the range (through a descriptor of extent zero it brings nothing, but takes the address
    // unit's time: 1 x 1 1024 -> 256 on 14 x 14, four units a wave and four more without content, 4.8 us against 4.6; 384 -> 64 on 7 of 11 x 11 4.25 / 3.82), and none
    // behind a branch inside the walk, where the compiler would have to assume the fewest loads in flight at every wait: what is left
    // over past whole rounds of DEPTH has code of its own for every count.
    using yes = std::integral_constant<bool, true>;
    using no = std::integral_constant<bool, false>;
    auto rest = [&](auto count) { // DEPTH units in flight, count() more to come
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            if (d < count())
                take(d, yes());
            else
                take(d, no());
#pragma unroll
        for (int d = 0; d < count(); ++d)
            take(d, no());
    };
    auto few = [&](auto count) { // fewer than DEPTH in all
#pragma unroll
        for (int d = 0; d < count(); ++d)
            issue(d);
        request_epilogue();
#pragma unroll
        for (int d = 0; d < count(); ++d)
            take(d, no());
    };
    if constexpr (DEPTH == 1 && !CONV) {
        // one unit in flight, which every wait waits for: the branch costs nothing, and one short loop is faster than code for every count (us
        // a launch, 231 rows, 256 -> 1024 6.2 -> 5.7, 512 -> 2048 8.4 -> 8.2; a convolution's walk from tap to tap gets slower by it, 64 -> 64 on
        // 56 x 56 11.9 -> 12.6)
        if (u_n > 0)
            issue(0);
        request_epilogue();
        for (int u = 1; u <= u_n; ++u)
            take(0, [&] { return u < u_n; });
    } else if (u_n >= DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            issue(d);
        request_epilogue();
        int left = u_n - DEPTH;
        for (; left >= DEPTH; left -= DEPTH)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d)
                take(d, yes());
        by_count<DEPTH - 1>(left, rest);
    } else
        by_count<DEPTH - 1>(u_n, few);

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                strip[(i * 16 + 4 * fg + e) * RS + j * 16 + fr] = acc[i][j][e];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QPT; ++q) {
        const int quad = t + q * 64 * NW, row = quad / (BN / 4), col = (quad % (BN / 4)) * 4;
        if (quad >= QUADS || m0 + row >= p.M || n0 + col >= p.N)
            continue;
        f32x4 s = *reinterpret_cast<const f32x4*>(&smem[row * RS + col]);
#pragma unroll
        for (int w = 1; w < NW; ++w)
            s += *reinterpret_cast<const f32x4*>(&smem[w * STRIP + row * RS + col]);
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = s[e] * p.alpha + bias4[q][e] + res4[q][e];
        apply_act_block(r, p.act);
        if (SEG) {
            const int sg = seg_of(p, n0);
            *reinterpret_cast<f32x4*>(reinterpret_cast<char*>(p.seg_ptr[sg]) + seg_offset(p, sg, m0 + row, n0 + col)) = f32x4 { r[0], r[1], r[2], r[3] };
        } else
            *reinterpret_cast<f32x4*>(p.C + (int64_t)(m0 + row) * p.ldc + n0 + col) = f32x4 { r[0], r[1], r[2], r[3] };
    }
}

// (rows / 16, columns / 16, waves) of the forms, by configuration number - kSliceCfg
constexpr int kSliceCfg = 40, kSliceForms = 5;
struct SliceForm {
    int tm, tn, nw;
};
constexpr SliceForm kSliceForm[kSliceForms] = { { 1, 1, 8 }, { 1, 2, 8 }, { 2, 2, 8 }, { 2, 2, 4 }, { 4, 2, 8 } };

// The form for a problem, or -1 where the tiled kernel (its cost by tile_pick) is the better one.  The forms were timed on 1000
// problems (M 1-16384, N 16-3072, K 16-4608, up to 6 GFLOP, GEMM and convolution, weights out of memory, launches back to
// back) and follow, in microseconds, with w = tiles per CU rounded up, to 13-21 % rms
//     t0 + w (c1 + c2 (rows + columns of the tile) K / 10^4):
// a workgroup costs what it pulls through its CU's path from L2, about 36 cycles per KB.  With one round of tiles (the first row of a form)
// K counts up to whole units of all waves: where it is one unit of 32, waves have nothing to do, and the form of four is the fastest (337 x
// 1144 x 32: 8 / 4 waves 5.0 / 3.8 us); there the choice among the forms takes 0.6 % longer than the best of them, past a round
// 2.5 %.  Up to 32 columns the other side is the
// general kernel's narrow tile, which wins from about 600 row blocks of 64 on (N = 32, K = 144-192: 20000 rows 8.2-9.7 against
// 6.3-7.2 us here, 50000 rows 11.0-14.5 against 11.1-14.0, convolutions 13.9 against 17.1); between 32 and 64 columns the tiled
// kernel's half empty 64-column tile beats it (97733 x 40 x 288 31.5 against 40.9 us, 24000 x 36 x 512 17.4 / 21.7).
// A convolution has constants of its own, and two rounds of tiles a row of theirs: the workgroups of both run side by side.  With one
// round a workgroup takes longer where more CUs pull at once:
//     t0 + (rows + columns of the tile) K / 10^4 (c2 + c1 tiles / CUs).
// Fitted to 1000 timed convolutions (3x3, 3x3 and 1x1 of stride 2, 5x5; M 20-30000, K 16-8000, weights from the memory-side cache), 5 to 7 %
// rms.  Over 1000 others the choice of form and kernel takes 0.4 % longer than the best (0.8 % with constants that were
// 13 to 24 % too high in one round, 0.7 % without the last term), and with Winograd beside them, 478 problems, 0.3 %.
static int64_t slice_tiles(int M, int N, int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); }
static float slice_rounds(int64_t tiles) { return (float)((tiles + 255) / 256); }
static float slice_cost(int form, bool conv, int M, int N, int K)
{
    static const float kGemm[2][kSliceForms][3] = { // t0, c1, c2; one round of tiles, more
        { { 2.46f, 0.64f, 0.39f }, { 2.73f, 0.25f, 0.47f }, { 2.01f, 0.77f, 0.65f }, { 2.89f, 0.19f, 0.68f }, { 1.62f, 1.19f, 0.80f } },
        { { 2.18f, 1.29f, 0.42f }, { 2.13f, 1.07f, 0.50f }, { 2.24f, 1.47f, 0.64f }, { 2.52f, 0.71f, 0.76f }, { 1.52f, 2.43f, 0.83f } }
    };
    static const float kConv[3][kSliceForms][3] = { // one round, two, more
        { { 3.53f, 0.07f, 0.45f }, { 3.34f, 0.08f, 0.52f }, { 3.49f, 0.08f, 0.69f }, { 3.78f, 0.06f, 0.78f }, { 4.54f, 0.06f, 0.86f } },
        { { 4.95f, 0.f, 0.50f }, { 4.35f, 0.f, 0.50f }, { 6.84f, 0.f, 0.70f }, { 4.83f, 0.f, 0.69f }, { 11.35f, 0.f, 0.86f } },
        { { 2.27f, 1.37f, 0.51f }, { 2.93f, 1.08f, 0.48f }, { 1.95f, 2.36f, 0.74f }, { 3.09f, 0.97f, 0.68f }, { 1.71f, 4.60f, 0.91f } }
    };
    const int bm = 16 * kSliceForm[form].tm, bn = 16 * kSliceForm[form].tn, unit = 32 * kSliceForm[form].nw;
    const int64_t tiles = slice_tiles(M, N, bm, bn);
    const float rounds = slice_rounds(tiles);
    const float pulled = 1e-4f * (float)(bm + bn) * (float)(rounds > 1.f ? K : (K + unit - 1) / unit * unit);
    const float* c = conv ? kConv[rounds > 2.f ? 2 : rounds > 1.f ? 1 : 0][form] : kGemm[rounds > 1.f][form];
    if (conv && rounds <= 1.f)
        return c[0] + pulled * (c[2] + c[1] * (float)tiles / 256.f);
    return c[0] + rounds * (c[1] + c[2] * pulled);
}
// whether a launch of this form stays below the 2^32 threads a grid can have
static bool slice_fits(int form, int M, int N)
{
    const SliceForm& f = kSliceForm[form];
    return slice_tiles(M, N, 16 * f.tm, 16 * f.tn) * 64 * f.nw < (1LL << 32);
}
static int slice_pick(bool conv, int M, int N, int K, float tiled_cost)
{
    const int64_t t64 = slice_tiles(M, N, 64, 64);
    const bool narrow = N <= 32;
    if (narrow && t64 > 512)
        return -1;
    int best = -1;
    // Below a round of tiles the tiled kernel takes longer than its cost says, which was fitted to 0.2 GFLOP and more: on 600 small problems by
    // 1.4 us up to K = 128 (4204 x 64 x 64 5.7 against 3.6 us here), on 1700 convolutions by 2.2 us up to a cost of 9, 1.2 at 16, 0.4 at 25.  Kernel
    // choices then take 1.7 % (convolutions 0.4 %) longer than the best; GEMMs 5.2 % with 0.95 of the cost.  Past a round operands
    // re-read cost the neighbours, too.
    const float fade = 15.f / std::max(15.f, tiled_cost);
    float best_cost = narrow ? 1e30f : t64 > 256 ? 0.95f * tiled_cost : tiled_cost + (conv ? 2.2f : 1.5f) * fade * fade;
    for (int i = 0; i < kSliceForms; ++i) {
        const float cost = slice_cost(i, conv, M, N, K);
        if (cost < best_cost && slice_fits(i, M, N)) {
            best_cost = cost;
            best = kSliceCfg + i;
        }
    }
    return best;
}

template <int I, int UK>
static void slice_launch_form(const GemmParams& q, bool conv, hipStream_t s)
{
    constexpr SliceForm f = kSliceForm[I];
    const dim3 grid((unsigned)(((q.M + 16 * f.tm - 1) / (16 * f.tm)) * ((q.N + 16 * f.tn - 1) / (16 * f.tn)))), block(64u * f.nw);
    if (conv)
        hipLaunchKernelGGL((igemm_slice_kernel<f.tm, f.tn, f.nw, UK, true, false>), grid, block, 0, s, q);
    else if (q.A2)
        hipLaunchKernelGGL((igemm_slice_kernel<f.tm, f.tn, f.nw, UK, false, true>), grid, block, 0, s, q);
    else
        hipLaunchKernelGGL((igemm_slice_kernel<f.tm, f.tn, f.nw, UK, false, false>), grid, block, 0, s, q);
}

// the form for outputs in segments, K a multiple of 32
template <int I>
static void slice_launch_seg(const GemmParams& q, hipStream_t s)
{
    constexpr SliceForm f = kSliceForm[I];
    const dim3 grid((unsigned)(((q.M + 16 * f.tm - 1) / (16 * f.tm)) * ((q.N + 16 * f.tn - 1) / (16 * f.tn)))), block(64u * f.nw);
    hipLaunchKernelGGL((igemm_slice_kernel<f.tm, f.tn, f.nw, 32, false, false, true>), grid, block, 0, s, q);
}

static void slice_launch(int cfg, const GemmParams& q, bool conv, hipStream_t s)
{
    // the longer unit where a unit stays inside a filter tap / one of two sources
    const bool wide = (conv ? q.Cin : q.A2 ? (q.K | q.K1) : q.K) % 32 == 0;
    switch (cfg - kSliceCfg) {
#define FDX_SLICE(I_)                                \
    case I_:                                         \
        if (wide)                                    \
            slice_launch_form<I_, 32>(q, conv, s);   \
        else                                         \
            slice_launch_form<I_, 16>(q, conv, s);   \
        break;
        FDX_SLICE(0)
        FDX_SLICE(1)
        FDX_SLICE(2)
        FDX_SLICE(3)
        FDX_SLICE(4)
#undef FDX_SLICE
    }
}
