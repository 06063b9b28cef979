// Fast path of the implicit-GEMM Conv2D / GEMM (included inside namespace fdx by igemm.hip).
//
// For the shapes that dominate real networks (Cin, or K for a plain GEMM, a multiple of 16; N a multiple of 4).  fp32
// operands, fp32 accumulators and fp32 accuracy, on the bf16 matrix cores:
//
//  * The fp32 MFMA (157 TFLOP/s) is what bounds this work; the bf16 one has 16 times its rate.  An fp32 value is exactly
//    the sum of three bf16 values (8 + 8 + 8 bits, each the rounding of what the ones before leave), so a product of two
//    is nine bf16 products, of which the three smallest (a1 b2, a2 b1, a2 b2 with planes counted from 0) are left out: six
//    MFMAs for sixteen steps of K instead of eight fp32 ones of twice the length.  They are at most 2^-24 of the product
//    (2^-24.02 for two operands of 0x1.00fe8p0), 2^-27.5 on average, with either sign: a sum that is one product is off by up to
//    1.5 roundings of fp32 where the fp32 MFMA is off by one, longer ones are closer than there.
//    The MFMA adds exact products in fp32, to nearest.  The leading product has accumulators of its own, so a result is
//    rounded at its own size once per 16 steps of K where the fp32 MFMA does so eight times: against 64-bit sums the
//    relative error (2-norm, normal operands, K = 64 / 512 / 4608) is 0.5 / 1.3 / 4.2 e-7, with the fp32 MFMA 1.4 / 4.1 / 12 e-7.
//    8192 x 2048 x 512: 147 -> 88.5 us, 194 TFLOP/s; with nothing but its MFMAs the kernel runs at 302 and the clock falls to
//    1.9 GHz: the power limit, not the issue rate, is the next bound.
//  * Both operands are split by the threads that stage them, on the way from registers to LDS (6.5 vector instructions a
//    value, hidden behind the MFMAs): operands stay fp32 in memory, nothing is prepared or kept.  Splitting the filter once
//    at load instead was measured slower (half as many vector instructions, but 6 bytes a value through L2 instead of 4).
//  * A row of a slab (32 floats) is fetched by four lanes, two 16-byte chunks each (k = 4q.. and 16 + 4q.. for lane q); the
//    eight values are one MFMA operand (16 bytes) in each plane.  The matrix product does not care which k sit together as
//    long as both operands agree.  LDS holds blocks of one lane number: block q of a plane = 16 bytes per tile row, so that
//    a wave's operand reads are two runs of 512 bytes, and blocks are offset by 32 bytes against each other, so that a
//    wave's writes meet each bank once.
//  * The largest four-wave tile keeps one slab in LDS (two workgroups on a CU then: one's staging beside the other's
//    products); its operands go to registers in front of a barrier.  The others keep two.
//  * Registers: 256 a lane bound the larger tiles.  The 256-row tile keeps 4 to 8 values in scratch memory, its halo form 21, none
//    of them touched in the K loop but one; the four-wave 128 x 128 tile keeps 32 to 60, of which its plain form reads 35 back per
//    slab and its column-segment form 32.  The cost rule was fitted to them as they are.
//  * Operands are fetched with raw buffer loads: each lane keeps ONE 32-bit byte offset per
//    tile row for the whole K loop, the walk along K is a scalar offset shared by the
//    workgroup (filter tap and channel are uniform within a slab), and a padded or
//    out-of-range tap is an offset beyond the buffer's extent, which the hardware answers
//    with zeros -- no branches, no per-slab address arithmetic.  A's base is shifted down by
//    the top-left padding so offsets stay non-negative.
//  * Workgroups are persistent: each walks a strided list of output tiles.  Before it writes a finished tile it
//    already has the first slab of its next tile in flight, and the tile's stores drain while
//    the next tile computes: output traffic and first-load latency overlap with MFMA work
//    instead of adding to it (with one tile per workgroup all workgroups of a round reach
//    their epilogue together and the matrix cores idle while HBM drains).
//  * The epilogue goes through LDS so that bias, residual and output move as 16-byte
//    accesses along the channel axis.
//  * SPLIT: a layer with too few output tiles for the chip (late stages of a CNN at small
//    batch) cuts every tile's K range into `splits` units.  A unit leaves its accumulators in a
//    workspace and takes a ticket on the tile; the last unit to arrive adds all partial tiles
//    in split order (so the sum does not depend on arrival order) and runs the epilogue.
//    Nothing waits on another workgroup.  Partials are written and read with agent-scope
//    accesses, which pass the per-XCD L2s, instead of a fence that writes a whole L2 back.
//  * SPLIT with splits == 0 ("stream-K"): the slabs of all tiles form one line that is cut into
//    as many equal pieces as there are workgroups, so every workgroup does the same amount of
//    MFMA work whatever the tile count.  A workgroup's piece covers the end of one tile, some
//    whole tiles and the beginning of another; the (at most two) partial tiles go through the
//    same workspace / ticket / ordered-sum path, with the number of contributors of a tile
//    and their workspace slots computed from the cut points.
// LDS slabs per workgroup and waves per SIMD (the register budget) of a tile.
constexpr int split_tile_buffers(int bm, int bn, int waves_m, int waves_n)
{
    return waves_m * waves_n == 4 && bm * bn >= 128 * 128 ? 1 : 2;
}
constexpr int kHaloSpan = 128; // HALO: pixels of a slab of A beyond the tile's rows
constexpr int split_tile_waves(int bm, int bn, int waves_m, int waves_n)
{
    return waves_m * waves_n == 8 || bm * bn > 64 * 64 ? 2 : 3;
}

// The elements of a 32 x 32 block (its accumulators, rows from m0, columns from n0, of problem z) that are not finite, again as
// plain fp32 sums on the fp32 MFMA: what infinite or NaN operands, or ones beyond the largest split value, give.  Lane (row or
// column fr, half fh) takes four consecutive k of eight at a time straight from memory.  A running sum that is NaN stays so: the
// walk ends where all of the elements that it is for are.  One whole wave comes here.  (One lane per element and one k at a time
// took 15 ms for 8192 x 2048 x 512 of NaN, 137 us this way; the product of finite operands 87.)
template <bool CONV, bool DUAL>
__device__ __forceinline__ void plain_block(const GemmParams& p, int z, int m0, int n0, f32x16& acc)
{
    const int lane = threadIdx.x & 63, fh = lane >> 5, m = m0 + (lane & 31), n = n0 + (lane & 31);
    const bool m_ok = m < p.M, n_ok = n < p.N;
    const float* A = p.A + (z / p.inner) * p.a_outer + (z % p.inner) * p.a_inner;
    const float* B = p.B + (z / p.inner) * p.b_outer + (z % p.inner) * p.b_inner + (int64_t)n * p.ldb;
    const float* A2 = p.A2;
    int iy0 = 0, ix0 = 0;
    if (CONV || DUAL) {
        const int img = m / (p.OH * p.OW), rm = m - img * (p.OH * p.OW), oy = rm / p.OW, ox = rm - oy * p.OW;
        if (CONV) {
            A += ((int64_t)(img * p.H + oy * p.sy) * p.W + ox * p.sx) * p.pix_stride; // A starts (pad_top, pad_left) early
            iy0 = oy * p.sy - p.pad_top;
            ix0 = ox * p.sx - p.pad_left;
        } else {
            A2 += ((int64_t)(img * p.H2 + oy * p.s2y) * p.W2 + ox * p.s2x) * p.C2;
        }
    }
    if (!CONV)
        A += (int64_t)m * p.lda;
    f32x16 sum = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };
    int fy = 0, fx = 0, c = 0;
    const int k_end = p.a_valid_k > 0 ? p.a_valid_k : p.K; // a multiple of 4
#pragma clang loop unroll(disable)
    for (int k = 0; k < k_end; k += 16) { // sixteen k lie within one filter tap, and in one source
        bool a_ok = m_ok;
        const float* a_at = A + k;
        if (CONV) {
            const int iy = iy0 + fy * p.dy, ix = ix0 + fx * p.dx;
            a_ok = m_ok && iy >= 0 && iy < p.H && ix >= 0 && ix < p.W;
            a_at = A + ((int64_t)fy * p.dy * p.W + fx * p.dx) * p.pix_stride + c;
            c += 16;
            if (c == p.Cin) {
                c = 0;
                if (++fx == p.kw) {
                    fx = 0;
                    ++fy;
                }
            }
        } else if (DUAL && k >= p.K1) {
            a_at = A2 + (k - p.K1);
        }
        f32x4 a[2], b[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int at = 8 * u + 4 * fh;
            const bool in_k = k + at < k_end;
            a[u] = b[u] = f32x4 { 0.f, 0.f, 0.f, 0.f };
            if (a_ok && in_k)
                a[u] = *reinterpret_cast<const f32x4*>(a_at + at);
            if (n_ok && in_k)
                b[u] = *reinterpret_cast<const f32x4*>(B + k + at);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sum = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][e], b[u][e], sum, 0, 0, 0);
        if ((k & 48) == 48) {
            bool open = false;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                open = open || (!(fabsf(acc[e]) < INFINITY) && sum[e] == sum[e]);
            if (!__any(open))
                break;
        }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e)
        acc[e] = fabsf(acc[e]) < INFINITY ? acc[e] : sum[e];
}

// Where row m, column n of a tile whose first column is n0 lies with SEG, in bytes from the start of its segment; segments
// begin at multiples of the tile width, so a tile's segment is uniform.
__device__ __forceinline__ uint32_t seg_offset(const GemmParams& p, int sg, int m, int n)
{
    const int seq = m / p.seg_rows, row = m - seq * p.seg_rows;
    return (uint32_t)(seq * p.seg_stride[sg] + row * p.seg_ld[sg] + n - (sg ? p.seg_col[sg - 1] : 0)) * 4u;
}
__device__ __forceinline__ int seg_of(const GemmParams& p, int n0) { return (n0 >= p.seg_col[0]) + (n0 >= p.seg_col[1]); }

// Bit y * kw + x: filter tap (y, x) lies inside the image, for a row whose tap (0, 0) lies at (iy, ix).  Columns and rows apart and without
// branches: tap by tap, with lanes taking branches of their own, nine taps of eight rows held up every tile's first load (ResNet50 of 64
// images 0.5 % longer).
template <typename Mask>
__device__ __forceinline__ Mask taps_inside(const GemmParams& p, int iy, int ix)
{
    Mask row = 0, all = 0;
    for (int x = 0; x < p.kw; ++x, ix += p.dx)
        row |= (Mask)((unsigned)ix < (unsigned)p.W) << x;
    for (int y = 0, at = 0; y < p.kh; ++y, iy += p.dy, at += p.kw)
        all |= (unsigned)iy < (unsigned)p.H ? row << at : (Mask)0;
    return all;
}

//  * DUAL (GEMM form, whole tiles only): the rows of A come from two tensors -- the first K1 columns from A with row
//    stride lda, the other K - K1 from A2, whose row for output pixel (image, y, x) is pixel (y * s2y, x * s2x) of an
//    [H2][W2][C2] map.  That is the sum of two pointwise convolutions as one GEMM over the concatenated channels
//    (a residual block whose shortcut is a 1x1 convolution: the shortcut's output is never written or read back).
//  * LNF (GEMM form, whole tiles only, K = the whole row): the rows of A are layer-normalised over K on the way,
//        C = act(LN(A) . B^T + bias)  with  LN(a) = (a - mean) / sqrt(var + eps)   (gamma folded into B, beta into bias
//    by the caller; include/fdeep/layers/layer_normalization_layer.hpp:37-63).  A tile's K loop reads its rows from end
//    to end anyway, so the row statistics are gathered from the operand registers on their way to LDS (sums of the
//    differences to the row's first value a thread sees, which keeps them small whatever the row's mean), merged over
//    the lanes that share a row after the loop, and applied in the epilogue as
//        rstd * (acc - mean * rowsum(B)) + bias:
//    no pass over A of its own, and the normalised tensor never exists.
//  * SEG (GEMM form): the columns of C go to up to three tensors, the rows of each in sequences that lie
//    apart: the stacked query / key / value projection of prompts, keys and values straight into their cache rows (2048 rows,
//    768 -> 3 x 768: 54 us in the stream-K form; three launches of 768 columns each leave 96 tiles of 128 x 128 on 256 CUs).
//  * HALO (convolution whose map keeps its size, stride 1): K is walked channel slab by channel slab and tap by tap inside a
//    slab, and a slab of A is the run of input pixels that all taps of the tile's rows touch (rows of a tile are neighbours in
//    raster order, so is what they read: BM + (kh - 1) dy W + (kw - 1) dx pixels).  It is fetched and split once for all taps
//    instead of once per tap -- nine times less of that work, and of the traffic from L2, for a 3x3 filter -- and a tap's
//    operands are read from LDS at its distance; a lane whose row has no such pixel (the convolution's padding) reads a
//    pixel of zeros kept behind the run.  64 images: 28 x 28 x 128 -> 128 84 -> 77 us, 14 x 14 x 256 -> 256 87 -> 77,
//    56 x 56 x 64 -> 64 113 -> 85; 16 images 32 -> 29, 35 (few-tiles ranges) -> 36, 34 -> 26.
template <int BM, int BN, int WAVES_M, int WAVES_N, bool CONV, bool SPLIT = false, bool STREAMK = false, bool DUAL = false,
    bool LNF = false, bool SEG = false, bool HALO = false>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, split_tile_waves(BM, BN, WAVES_M, WAVES_N))
void igemm_fast_kernel(GemmParams p)
{
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    static_assert(NT == 256 || NT == 512, "four or eight waves");
    static_assert(!DUAL || (!CONV && !SPLIT), "the two-source form is a whole-tile GEMM");
    static_assert(!LNF || (!CONV && !SPLIT && !DUAL), "the normalising form is a whole-tile GEMM");
    static_assert(!SEG || (!CONV && !DUAL && !LNF), "the form with segmented outputs is a GEMM");
    constexpr int BKT = 32;
    constexpr bool DB = split_tile_buffers(BM, BN, WAVES_M, WAVES_N) == 2;
    constexpr int RPP = NT / 4; // tile rows filled per loader pass: four lanes per row, two 16-byte chunks each
    static_assert(!HALO || (CONV && !STREAMK && DB), "the halo form is a convolution with whole tiles or K ranges");
    constexpr int ROWS_A = HALO ? BM + kHaloSpan : BM; // pixels of A in LDS
    constexpr int A_UNITS = ROWS_A / RPP, B_UNITS = BN / RPP;
    static_assert(ROWS_A % RPP == 0 && BN % RPP == 0, "tile rows must be a multiple of the loader pass");
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
    constexpr int TM = WTM / 32, TN = WTN / 32;
    constexpr int OSTRIDE = WTN + 4; // epilogue scratch row
    // LDS of one slab: per operand three planes of four blocks (one per lane of a row), a block = 16 bytes per tile row
    // (HALO: one slab of A, whose last 16 bytes of a block are the pixel of zeros, and two of B)
    constexpr int A_BLK = ROWS_A * 16 + 32, B_BLK = BN * 16 + 32, A_BYTES = 12 * A_BLK;
    constexpr int A_STEP = HALO ? 0 : A_BYTES + 12 * B_BLK, B_STEP = HALO ? 12 * B_BLK : A_STEP; // from buffer 0 to buffer 1
    constexpr int SMEM_BYTES = A_BYTES + 12 * B_BLK + (DB ? B_STEP : 0);
    static_assert(SMEM_BYTES >= WAVES_M * WAVES_N * 32 * OSTRIDE * 4, "epilogue scratch must fit in the operand buffers");
    constexpr uint32_t OOB = 0x80000000u; // beyond any extent this path accepts: the load returns zeros

    __shared__ __attribute__((aligned(16))) unsigned char smem_raw[SMEM_BYTES];
    float* const smem = reinterpret_cast<float*>(smem_raw);
    __shared__ int last_flag;
    __shared__ float ln_stats[LNF ? 2 * BM : 2]; // (mean, 1 / sqrt(var + eps)) per tile row

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int kq = t & 3, r0 = t >> 2;
    const int fr = lane & 31, fh = lane >> 5;

    const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
    const int per_problem = tiles_m * tiles_n;
    const int S = SPLIT ? p.splits : 1;
    const int all_tiles = per_problem * p.batch;
    // Units of work: the first n_dp tiles are computed whole; every later tile is cut into S K ranges ("split
    // units").  XCD x (workgroups with blockIdx % 8 == x) owns a contiguous range of the whole tiles and one of the
    // split units, so tiles that share an A row block also share that XCD's L2 and both kinds of work are spread
    // evenly; its workgroups stride through the two ranges one after the other.
    const int n_dp = SPLIT ? p.split_dp_tiles : all_tiles, n_su = SPLIT ? (all_tiles - n_dp) * S : 0;
    const int xcd = blockIdx.x & 7, wg_in_xcd = blockIdx.x >> 3;
    const int wgs_in_xcd = ((int)gridDim.x - xcd + 7) >> 3;
    const int alo = xcd * (n_dp >> 3) + (xcd < (n_dp & 7) ? xcd : (n_dp & 7)), na = (n_dp >> 3) + (xcd < (n_dp & 7) ? 1 : 0);
    const int blo = xcd * (n_su >> 3) + (xcd < (n_su & 7) ? xcd : (n_su & 7)), nb = (n_su >> 3) + (xcd < (n_su & 7) ? 1 : 0);
    const int hi = na + nb; // local unit indices [0, hi)
    const int KT = (p.K + BKT - 1) / BKT; // the second half of the last slab may lie behind the end of K: zeros

    // stream-K: workgroup g (numbered XCD by XCD, so an XCD owns a contiguous stretch of tiles) takes the slabs
    // [g * W / G, (g + 1) * W / G) of the W = tiles * KT slabs; its units are the tiles that stretch touches
    // (a template argument: carried as a run-time flag, the extra index arithmetic cost the plain split variant a
    // tenth of its speed)
    static_assert(!STREAMK || SPLIT, "stream-K is a form of the split variant");
    constexpr bool sk = STREAMK;
    const int G = (int)gridDim.x;
    const int g_lin = xcd * (G >> 3) + (xcd < (G & 7) ? xcd : (G & 7)) + wg_in_xcd;
    const int64_t W = (int64_t)all_tiles * KT;
    const int64_t sk_lo = sk ? g_lin * W / G : 0, sk_hi = sk ? (g_lin + 1) * W / G : 0;
    const int sk_first = sk ? (int)(sk_lo / KT) : 0;
    const int sk_units = (sk && sk_hi > sk_lo) ? (int)((sk_hi - 1) / KT) - sk_first + 1 : 0;

    // ---- per-tile loader state
    uint32_t a_voff[A_UNITS], b_voff[B_UNITS];
    uint32_t a2_voff[DUAL ? A_UNITS : 1];
    uint64_t a_mask[HALO ? 1 : A_UNITS];
    uint32_t row_mask[TM]; // HALO: taps of this lane's operand rows that lie inside the image
    const int taps = HALO ? p.kh * p.kw : 1;
    int slab_c = 0;        // HALO: first channel of the next slab of A
    int read_tap = 0, read_fx = 0, read_shift = 0; // HALO: the tap whose operands are read next and its distance in pixels
    __amdgpu_buffer_rsrc_t srd_a, srd_b;
    const __amdgpu_buffer_rsrc_t srd_a2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(DUAL ? p.A2 : p.A), 0,
        DUAL ? (int)p.a2_records : 0, 0x00020000);
    // the walk along K goes by half slabs of 16 floats; in a convolution one half slab lies within one filter tap
    int tap, fx, fy, c0, soff_a, soff_b;
    f32x4 ra[A_UNITS][2], rb[B_UNITS][2];
    int kt_n = KT; // slabs of the current unit

    int cur_su = -1;  // workspace slot of the current work item's partial tile, -1 for a whole tile
    int cur_tile = 0; // its output tile
    auto setup = [&](int local, int& m0, int& n0, int64_t& c_off) {
        int tile = alo + local, kt_lo = 0;
        cur_su = -1;
        kt_n = KT;
        if (sk) {
            tile = sk_first + local;
            const int64_t t0 = (int64_t)tile * KT;
            kt_lo = sk_lo > t0 ? (int)(sk_lo - t0) : 0;
            const int kt_hi = sk_hi - t0 < KT ? (int)(sk_hi - t0) : KT;
            kt_n = kt_hi - kt_lo;
            // a workgroup leaves at most two partial tiles: one that began before its stretch (slot 2g) and one that
            // ends after it (slot 2g + 1)
            if (kt_n < KT)
                cur_su = 2 * g_lin + (sk_lo > t0 ? 0 : 1);
        } else if (SPLIT && local >= na) {
            cur_su = blo + (local - na);
            tile = n_dp + cur_su / S;
            const int split = cur_su - (cur_su / S) * S;
            kt_lo = (int)((int64_t)split * KT / S);
            kt_n = (int)((int64_t)(split + 1) * KT / S) - kt_lo;
        }
        cur_tile = tile;
        const int z = tile / per_problem, id = tile - z * per_problem;
        if (p.strip_w > 0) {
            const int per_strip = tiles_m * p.strip_w, last = (tiles_n - 1) / p.strip_w;
            int strip = id / per_strip;
            strip = strip < last ? strip : last; // the last strip may be narrower
            const int rem = id - strip * per_strip, left = tiles_n - strip * p.strip_w;
            const int w_eff = p.strip_w < left ? p.strip_w : left;
            const int mt = rem / w_eff;
            m0 = mt * BM;
            n0 = (strip * p.strip_w + (rem - mt * w_eff)) * BN;
        } else {
            m0 = (id / tiles_n) * BM;
            n0 = (id % tiles_n) * BN;
        }
        const float* A = p.A + (z / p.inner) * p.a_outer + (z % p.inner) * p.a_inner;
        const float* B = p.B + (z / p.inner) * p.b_outer + (z % p.inner) * p.b_inner;
        c_off = (z / p.inner) * p.c_outer + (z % p.inner) * p.c_inner;
        const int halo_lo = HALO ? p.pad_top * p.W + p.pad_left : 0;
        if (HALO) // A starts halo_lo pixels early
            srd_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A) + (int64_t)halo_lo * p.Cin, 0, (int)((uint32_t)p.M * p.Cin * 4u), 0x00020000);
        else
            srd_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, (int)p.a_records, 0x00020000);
        srd_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), 0, (int)p.b_records, 0x00020000);
        if (HALO) {
            const int span = (p.kh - 1) * p.dy * p.W + (p.kw - 1) * p.dx;
#pragma unroll
            for (int i = 0; i < A_UNITS; ++i) {
                const int slot = r0 + i * RPP, px = m0 - halo_lo + slot;
                a_voff[i] = slot < BM + span && px >= 0 && px < p.M ? (uint32_t)px * p.Cin * 4u + kq * 16 : OOB;
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int m = m0 + wm * WTM + i * 32 + fr;
                const int rm = m % (p.OH * p.OW), oy = rm / p.OW, ox = rm - oy * p.OW;
                row_mask[i] = m < p.M ? taps_inside<uint32_t>(p, oy - p.pad_top, ox - p.pad_left) : 0u;
            }
        } else
#pragma unroll
        for (int i = 0; i < A_UNITS; ++i) {
            const int m = m0 + r0 + i * RPP;
            a_voff[i] = OOB;
            a_mask[HALO ? 0 : i] = 0;
            if (m < p.M) {
                if (CONV) {
                    const int img = m / (p.OH * p.OW), rm = m - img * (p.OH * p.OW);
                    const int oy = rm / p.OW, ox = rm - oy * p.OW;
                    // byte offset from the shifted base (shift = (pad_top*W + pad_left)*Cin elements)
                    a_voff[i] = (uint32_t)(((img * p.H + oy * p.sy) * p.W + ox * p.sx) * p.pix_stride) * 4u + kq * 16;
                    a_mask[HALO ? 0 : i] = taps_inside<uint64_t>(p, oy * p.sy - p.pad_top, ox * p.sx - p.pad_left);
                } else {
                    a_voff[i] = (uint32_t)((int64_t)m * p.lda) * 4u + kq * 16;
                    a_mask[HALO ? 0 : i] = ~0ull;
                }
            }
            if (DUAL) {
                a2_voff[i] = OOB;
                if (m < p.M) {
                    const int img = m / (p.OH * p.OW), rm = m - img * (p.OH * p.OW);
                    const int oy = rm / p.OW, ox = rm - oy * p.OW;
                    a2_voff[i] = (uint32_t)(((img * p.H2 + oy * p.s2y) * p.W2 + ox * p.s2x) * p.C2) * 4u + kq * 16;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < B_UNITS; ++i) {
            const int n = n0 + r0 + i * RPP;
            b_voff[i] = n < p.N ? (uint32_t)((int64_t)n * p.ldb) * 4u + kq * 16 : OOB;
        }
        tap = fx = fy = c0 = 0;
        soff_a = soff_b = 0;
        if (HALO) {
            const int cs = kt_lo / taps;
            tap = read_tap = kt_lo - cs * taps;
            slab_c = c0 = cs * BKT;
            soff_b = (tap * p.Cin + c0) * 4;
            const int y = tap / p.kw;
            read_fx = tap - y * p.kw;
            read_shift = y * p.dy * p.W + read_fx * p.dx;
        } else if (SPLIT && kt_lo > 0) {
            const int k_start = kt_lo * BKT;
            soff_b = k_start * 4;
            if (CONV) {
                tap = k_start / p.Cin;
                c0 = k_start - tap * p.Cin;
                fy = tap / p.kw;
                fx = tap - fy * p.kw;
                soff_a = ((fy * p.dy * p.W + fx * p.dx) * p.pix_stride + c0) * 4;
            } else {
                soff_a = k_start * 4;
            }
        }
    };
    const int k_bytes = p.K * 4;
    // Requests half h of the next slab; dead: no such slab, the offsets are out of range and nothing is fetched.
    auto load_half = [&](int h, bool live) {
        const bool in_k = live && soff_b < k_bytes;
        const uint32_t off = in_k ? 0u : OOB;
        if (DUAL && soff_b >= p.K1 * 4) { // the half slab lies in the second tensor's columns (uniform over the workgroup)
#pragma unroll
            for (int i = 0; i < A_UNITS; ++i)
                ra[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_a2, (int)(a2_voff[DUAL ? i : 0] | off), soff_b - p.K1 * 4, 0));
        } else {
#pragma unroll
            for (int i = 0; i < A_UNITS; ++i) {
                const uint32_t vo = CONV ? (in_k && ((a_mask[HALO ? 0 : i] >> tap) & 1) ? a_voff[i] : OOB) : (a_voff[i] | off);
                ra[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_a, (int)vo, soff_a, 0));
            }
        }
#pragma unroll
        for (int i = 0; i < B_UNITS; ++i)
            rb[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_b, (int)(b_voff[i] | off), soff_b, 0));
        soff_b += 64;
        if (CONV) {
            c0 += 16;
            if (c0 == p.Cin) {
                c0 = 0;
                ++tap;
                if (++fx == p.kw) {
                    fx = 0;
                    ++fy;
                }
            }
            soff_a = ((fy * p.dy * p.W + fx * p.dx) * p.pix_stride + c0) * 4;
        } else {
            soff_a += 64;
        }
    };
    // HALO: B of the next (channel slab, tap), A of the next channel slab
    auto load_halo_b = [&](bool live) {
        const uint32_t off = live ? 0u : OOB;
#pragma unroll
        for (int i = 0; i < B_UNITS; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                rb[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_b, (int)(b_voff[i] | off), soff_b + 64 * h, 0));
        soff_b += p.Cin * 4;
        if (++tap == taps) {
            tap = 0;
            c0 += BKT;
            soff_b = c0 * 4;
        }
    };
    auto load_halo_a = [&]() { // behind the last slab nothing is fetched
        const uint32_t off = slab_c < p.Cin ? 0u : OOB;
#pragma unroll
        for (int i = 0; i < A_UNITS; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                ra[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(srd_a, (int)(a_voff[i] | off), slab_c * 4 + 64 * h, 0));
        slab_c += BKT;
    };
    auto load_tiles = [&](bool live) {
        if (HALO) {
            load_halo_b(live);
            return;
        }
        load_half(0, live);
        load_half(1, live);
    };
    float ln_shift[LNF ? A_UNITS : 1], ln_s[LNF ? A_UNITS : 1], ln_q[LNF ? A_UNITS : 1];
    // The slab's staging in steps of two floats: a thread's unit of eight (chunks kq and 4 + kq of a row, 16 bytes of each plane)
    // is written behind its last pair.  Units of A come before those of B.
    constexpr int A_PAIRS = 4 * A_UNITS, PAIRS = A_PAIRS + 4 * B_UNITS;
    uint32_t planes[3][4];
    auto stage_pair = [&](int i, int buf) {
        const int unit = i / 4, e = i % 4, b_unit = unit < A_UNITS ? 0 : unit - A_UNITS, a_unit = unit < A_UNITS ? unit : 0;
        const f32x4(&r)[2] = unit < A_UNITS ? ra[a_unit] : rb[b_unit];
        split3(r[e >> 1][2 * (e & 1)] * kSplitUp, r[e >> 1][2 * (e & 1) + 1] * kSplitUp, planes[0][e], planes[1][e], planes[2][e]);
        if (e == 3) {
            unsigned char* dst = unit < A_UNITS ? smem_raw + buf * A_STEP + kq * A_BLK + (r0 + a_unit * RPP) * 16
                                                : smem_raw + buf * B_STEP + A_BYTES + kq * B_BLK + (r0 + b_unit * RPP) * 16;
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<u32x4*>(dst + q * (unit < A_UNITS ? 4 * A_BLK : 4 * B_BLK)) = u32x4 { planes[q][0], planes[q][1], planes[q][2], planes[q][3] };
        }
    };
    // LNF: the statistics of the slab that is staged next
    auto gather_rows = [&](bool first) {
#pragma unroll
        for (int i = 0; i < (LNF ? A_UNITS : 0); ++i) {
            if (first) {
                ln_shift[LNF ? i : 0] = ra[i][0][0];
                ln_s[LNF ? i : 0] = 0.f;
                ln_q[LNF ? i : 0] = 0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float dlt = ra[i][e >> 2][e & 3] - ln_shift[LNF ? i : 0];
                ln_s[LNF ? i : 0] += dlt;
                ln_q[LNF ? i : 0] += dlt * dlt;
            }
        }
    };
    auto store_a = [&](int buf) {
#pragma unroll
        for (int i = 0; i < A_PAIRS; ++i)
            stage_pair(i, buf);
        if (HALO && t < 12)
            *reinterpret_cast<u32x4*>(smem_raw + t * A_BLK + ROWS_A * 16) = u32x4 { 0u, 0u, 0u, 0u };
    };
    auto store_b = [&](int buf) {
#pragma unroll
        for (int i = A_PAIRS; i < PAIRS; ++i)
            stage_pair(i, buf);
    };

    int tile = sk ? 0 : wg_in_xcd; // local unit index
    const int unit_step = sk ? 1 : wgs_in_xcd, unit_end = sk ? sk_units : hi;
    if (tile >= unit_end)
        return; // uniform per workgroup
    int m0, n0;
    int64_t c_off;
    setup(tile, m0, n0, c_off);
    if (HALO)
        load_halo_a();
    load_tiles(true);

    for (;;) {
        // the leading products of a tile in one set of accumulators, the five small ones in a second: a result is rounded
        // against its own size once per 16 steps of K instead of once per product
        f32x16 acc[TM][TN], acc_lo[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    acc[i][j][e] = acc_lo[i][j][e] = 0.f;

        const int kt_end = kt_n;
        gather_rows(true);
        store_a(0);
        store_b(0);
        load_tiles(1 < kt_end);
        if (HALO)
            load_halo_a();
        __syncthreads();
        bf16x8 af[2][TM][3], bf[2][TN][3];
        auto read_frags = [&](int s, int buf) {
            const unsigned char* as = smem_raw + buf * A_STEP + (2 * s + fh) * A_BLK + (HALO ? 0 : (wm * WTM + fr) * 16);
            const unsigned char* bs = smem_raw + buf * B_STEP + A_BYTES + (2 * s + fh) * B_BLK + (wn * WTN + fr) * 16;
            int row[TM]; // where operand row i lies
#pragma unroll
            for (int i = 0; i < TM; ++i)
                row[i] = !HALO ? i * 512 : (row_mask[i] >> read_tap) & 1 ? (wm * WTM + i * 32 + fr + read_shift) * 16 : ROWS_A * 16;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    af[s][i][q] = *reinterpret_cast<const bf16x8*>(as + q * 4 * A_BLK + row[i]);
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    bf[s][j][q] = *reinterpret_cast<const bf16x8*>(bs + q * 4 * B_BLK + j * 512);
            }
        };
        // Both halves of a slab are read from LDS in front of the first one's products: behind the staging writes of operand A
        // the second half's reads would wait for them, with the matrix pipe drained (128 x 128 tiles 7 % faster this way,
        // 128 x 64 2 %; the 256-row tile has no registers for it, 3 % slower).
        constexpr bool READ_AHEAD = BM <= 128;
        // The halo form in eight waves of 128 rows: the barrier lies between the halves, and the next slab's first half is read
        // under the second half's products (7 % faster; 128 x 64 tiles, two workgroups on a CU, gain nothing, the tiles that
        // stage A for every slab lose 6 %).
        constexpr bool CARRIED = HALO && READ_AHEAD && NT == 512;
        auto product = [&](int s, int x, int y, f32x16(&d)[TM][TN]) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    d[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[s][i][x], bf[s][j][y], d[i][j], 0, 0, 0);
        };
        // The six products of half a slab; pairs [from, to) of the next slab's staging are spread over those from number `first` on:
        // a wave issues a product's MFMAs and splits floats while they run (the empty asm pins a pair to its place: without it
        // the compiler moves the splitting together).  The slab's first products stand alone, its loads arrive meanwhile.
        auto multiply = [&](int s, int from = 0, int to = 0, int buf = 0, int first = 0) {
            // the 256-row tile keeps A's plane from one product to the next (2.6 % faster: fewer operand changes, and power is
            // what bounds it); where the next half's operands are at hand the other order is 2 % faster
            constexpr int X[6] = { 0, 0, READ_AHEAD ? 1 : 0, 1, READ_AHEAD ? 0 : 1, 2 };
            constexpr int Y[6] = { 0, 1, READ_AHEAD ? 0 : 2, READ_AHEAD ? 1 : 0, READ_AHEAD ? 2 : 1, 0 };
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                product(s, X[q], Y[q], q == 0 ? acc : acc_lo);
                if (to == from || q < first)
                    continue;
                const int lo = from + (to - from) * (q - first) / (6 - first), hi = from + (to - from) * (q + 1 - first) / (6 - first);
#pragma unroll
                for (int i = lo; i < hi; ++i) {
                    stage_pair(i, buf);
                    asm volatile("" : "+v"(planes[0][i % 4]), "+v"(planes[1][i % 4]), "+v"(planes[2][i % 4]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // all slabs but the last: the next slab goes to LDS beside this one's products, and the one after that is requested into
        // the registers this frees.  Staging spread over the products, against all MFMAs in front of all the splitting as the
        // compiler orders them, in the tiles that keep two slabs and read ahead: 8192 x 1536 x 512 in 128 x 128 tiles 81 -> 77 us,
        // 8192 x 512 x 2048 97 -> 91, 2048 x 768 x 3072 120 -> 101, 128 x 64 tiles 2 to 9 %, 64 x 64 2 %; the 256-row tile and the
        // halo form gain nothing or lose 2 to 8 %.
        for (int kt = 0; kt + 1 < kt_end; ++kt) {
            const int buf = DB ? kt & 1 : 0;
            if (HALO) {
                if (!CARRIED || kt == 0)
                    read_frags(0, buf);
                if (READ_AHEAD)
                    read_frags(1, buf);
                multiply(0);
                if (!READ_AHEAD)
                    read_frags(1, buf);
                store_b(buf ^ 1);
                if (!CARRIED)
                    multiply(1);
                load_tiles(kt + 2 < kt_end);
                read_shift += p.dx;
                if (++read_fx == p.kw) {
                    read_fx = 0;
                    read_shift += p.dy * p.W - p.kw * p.dx;
                }
                if (++read_tap == taps) { // the next slab of channels
                    read_tap = read_fx = read_shift = 0;
                    __syncthreads();
                    store_a(0);
                    load_halo_a();
                }
                __syncthreads();
                if (CARRIED) {
                    read_frags(0, buf ^ 1);
                    multiply(1);
                }
                continue;
            }
            if (DB) {
                read_frags(0, buf);
                if (READ_AHEAD)
                    read_frags(1, buf);
                gather_rows(false);
                if (READ_AHEAD) {
                    multiply(0, 0, PAIRS / 3, buf ^ 1, 3);
                    multiply(1, PAIRS / 3, PAIRS, buf ^ 1);
                } else {
                    multiply(0);
                    store_a(buf ^ 1);
                    read_frags(1, buf);
                    multiply(1);
                    store_b(buf ^ 1);
                }
            } else {
                read_frags(0, 0);
                read_frags(1, 0);
                __syncthreads();
                gather_rows(false);
                multiply(0);
                store_a(0);
                multiply(1);
                store_b(0);
            }
            load_tiles(kt + 2 < kt_end);
            __syncthreads();
        }
        {
            const int buf = DB ? (kt_end - 1) & 1 : 0;
            if (!CARRIED || kt_end == 1)
                read_frags(0, buf);
            if (READ_AHEAD)
                read_frags(1, buf);
            multiply(0);
            if (!READ_AHEAD)
                read_frags(1, buf);
            multiply(1);
            if (LNF) {
                // Every slab has passed through gather_rows by now, so every thread has seen 8 * KT values of each of its
                // rows.  The four lanes that share a row (a quad) merge their means and sums of
                // squared deviations pairwise, equal counts on both sides at each step, on the VALU's lane swaps.  Done here,
                // behind the last slab's MFMAs and in front of the barrier below, it costs no barrier of its own.
#pragma unroll
                for (int i = 0; i < A_UNITS; ++i) {
                    float cnt = 8.0f * (float)KT;
                    float mean = ln_shift[LNF ? i : 0] + ln_s[LNF ? i : 0] / cnt;
                    float m2 = ln_q[LNF ? i : 0] - ln_s[LNF ? i : 0] * ln_s[LNF ? i : 0] / cnt;
                    auto merge = [&](float om, float o2) {
                        const float dlt = om - mean;
                        mean = 0.5f * (mean + om);
                        m2 = m2 + o2 + dlt * dlt * (0.5f * cnt);
                        cnt *= 2.0f;
                    };
                    merge(dpp_move<0xB1>(mean), dpp_move<0xB1>(m2));   // quad_perm [1, 0, 3, 2]
                    merge(dpp_move<0x4E>(mean), dpp_move<0x4E>(m2));   // quad_perm [2, 3, 0, 1]
                    if (kq == 0) {
                        ln_stats[2 * (r0 + i * RPP)] = mean;
                        ln_stats[2 * (r0 + i * RPP) + 1] = 1.0f / sqrtf(fmaxf(m2, 0.f) / cnt + p.ln_eps);
                    }
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    acc[i][j][e] += acc_lo[i][j][e];

        // this tile's coordinates for the epilogue; the loader state moves on to the next tile
        const int em0 = m0, en0 = n0;
        float* __restrict__ C = p.C + c_off;
        const float* __restrict__ R = p.residual ? p.residual + c_off : nullptr;
        const int su_done = cur_su, tile_done = cur_tile;
        // What the epilogue reads from memory -- the bias and the residual rows of the first 32-row band -- is requested
        // before the next tile's operands: loads complete in the order of their issue, so behind those operands their
        // first use would wait for the whole prefetch.
        constexpr int LPR = WTN / 4;  // lanes per scratch row
        constexpr int RPS = 64 / LPR; // rows per store pass
        const int srow = lane / LPR, scol = (lane % LPR) * 4;
        const int n = en0 + wn * WTN + scol;
        const bool n_ok = n < p.N; // N is a multiple of 4 on this path
        f32x4 bias4 = { 0.f, 0.f, 0.f, 0.f };
        f32x4 rr[32 / RPS];
        auto request_residual = [&](int i) {
#pragma unroll
            for (int ps = 0; ps < 32 / RPS; ++ps) {
                const int m = em0 + wm * WTM + i * 32 + ps * RPS + srow;
                rr[ps] = f32x4 { 0.f, 0.f, 0.f, 0.f };
                if (R && m < p.M && n_ok)
                    rr[ps] = *reinterpret_cast<const f32x4*>(R + (int64_t)m * p.ldc + n);
            }
        };
        f32x4 wsum4 = { 0.f, 0.f, 0.f, 0.f };
        auto request_epilogue = [&]() {
            if (p.bias && n_ok)
                bias4 = *reinterpret_cast<const f32x4*>(p.bias + n);
            if (LNF && n_ok)
                wsum4 = *reinterpret_cast<const f32x4*>(p.ln_wsum + n);
            request_residual(0);
        };
        // (the split variants hold partial tiles in registers across the exchange below; there the requests wait
        // until the exchange is over)
        if (!SPLIT)
            request_epilogue();
        tile += unit_step;
        const bool more = tile < unit_end;
        if (more) {
            setup(tile, m0, n0, c_off);
            if (HALO)
                load_halo_a();
            load_tiles(true); // in flight while this tile is written out
        }

        if (SPLIT && su_done >= 0) {
            constexpr int TILE_F = BM * BN;
            // contributors of this output tile, its ticket, and where contributor number sp left its partial
            int parts = S, out_tile = sk ? tile_done : su_done / S, g_a = 0;
            const int64_t t0 = (int64_t)tile_done * KT;
            if (sk) {
                g_a = (int)(((t0 + 1) * G + W - 1) / W) - 1; // the workgroup whose stretch holds the tile's first slab
                parts = (int)(((t0 + KT) * G + W - 1) / W) - g_a; // ... up to the one that holds its last slab
            }
            auto slot_of = [&](int sp) -> int64_t {
                if (!sk)
                    return (int64_t)out_tile * S + sp;
                const int gg = g_a + sp;
                return 2 * (int64_t)gg + (gg * W / G > t0 ? 0 : 1);
            };
            float* mine = p.split_ws + (int64_t)su_done * TILE_F + t;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        __hip_atomic_store(mine + ((i * TN + j) * 16 + e) * NT, acc[i][j][e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // every lane's partials have left the CU before the ticket is taken
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (t == 0) {
                const int ticket = __hip_atomic_fetch_add(p.split_tickets + out_tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const int last = ticket == parts - 1;
                if (last)
                    __hip_atomic_store(p.split_tickets + out_tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // next launch
                last_flag = last;
            }
            __syncthreads();
            const bool is_last = last_flag != 0;
            __syncthreads(); // last_flag is rewritten by the next unit
            if (!is_last) {
                if (!more)
                    break;
                continue;
            }
            // Partials are summed in split order.  The own one comes from the workspace like the others where a second
            // copy of the accumulators would not fit beside them (64 x 64 outputs a wave: of the cut forms the 256-row tile
            // of the halo form; re-reading it costs a tile of loads); the others keep it in registers.
            constexpr bool REREAD_OWN = TM * TN >= 4;
            f32x16 own[REREAD_OWN ? 1 : TM][REREAD_OWN ? 1 : TN];
            int my_part = -1;
            if (!REREAD_OWN) {
                my_part = sk ? g_lin - g_a : su_done - out_tile * S;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        own[REREAD_OWN ? 0 : i][REREAD_OWN ? 0 : j] = acc[i][j];
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        acc[i][j][e] = 0.f;
            for (int sp = 0; sp < parts; ++sp) {
                const float* part = p.split_ws + slot_of(sp) * TILE_F + t;
                const bool self = sp == my_part;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            acc[i][j][e] += self ? own[REREAD_OWN ? 0 : i][REREAD_OWN ? 0 : j][e]
                                                 : __hip_atomic_load(part + ((i * TN + j) * 16 + e) * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        // one 32x32 block's loads at a time: hoisting all of them would need a register per load
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }

        // the factor of the split operands (partial tiles keep it: a result among the subnormal numbers is rounded once)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    acc[i][j][e] *= kSplitDown;

        // ---- epilogue: accumulators -> per-wave LDS scratch [32][WTN] -> 16-byte row accesses
        float* scratch = smem + wave * 32 * OSTRIDE;
        if (SPLIT)
            request_epilogue();
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            // the residual rows of a later 32-row band are requested before the accumulators go through LDS, so their
            // latency is covered by the transposition instead of stalling every store
            if (i > 0)
                request_residual(i);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    scratch[(8 * (e >> 2) + 4 * fh + (e & 3)) * OSTRIDE + j * 32 + fr] = acc[i][j][e];
            // the scratch band is private to this wave and a wave's LDS accesses complete in order: no workgroup barrier
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // Inf and NaN do not survive the split (Inf - Inf in the remainders), and a value from 2^112 on makes an infinite bf16:
            // such elements are summed again in plain fp32.  (A band of huge finite values may come here too and finds nothing to
            // do.)  Behind the transposition, where the band's accumulators are free.
            float size = 0.f;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    size += fabsf(acc[i][j][e]);
            if (__builtin_expect(__any(!(size < INFINITY)), 0)) {
#pragma clang loop unroll(disable)
                for (int j = 0; j < TN; ++j) {
                    float* const block = scratch + 4 * fh * OSTRIDE + j * 32 + fr;
                    f32x16 v;
                    float block_size = 0.f;
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        v[e] = block[(8 * (e >> 2) + (e & 3)) * OSTRIDE];
                        block_size += fabsf(v[e]);
                    }
                    if (!__any(!(block_size < INFINITY)))
                        continue;
                    plain_block<CONV, DUAL>(p, tile_done / per_problem, em0 + wm * WTM + i * 32, en0 + wn * WTN + j * 32, v);
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        block[(8 * (e >> 2) + (e & 3)) * OSTRIDE] = v[e];
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            // all rows of the band are finished in registers before the first of them is stored: the wait for the
            // residual loads would otherwise also wait, pass after pass, for the store of the pass before
            f32x4 done[32 / RPS];
#pragma unroll
            for (int ps = 0; ps < 32 / RPS; ++ps) {
                const int row = ps * RPS + srow;
                const f32x4 v = *reinterpret_cast<const f32x4*>(&scratch[row * OSTRIDE + scol]);
                float r[4];
                if (LNF) {
                    const int trow = wm * WTM + i * 32 + row;
                    const float mu = ln_stats[2 * trow], rs = ln_stats[2 * trow + 1];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        r[e] = rs * (v[e] - mu * wsum4[e]) + bias4[e] + rr[ps][e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        r[e] = v[e] * p.alpha + bias4[e] + rr[ps][e];
                }
                apply_act_block(r, p.act);
                done[ps] = f32x4 { r[0], r[1], r[2], r[3] };
            }
#pragma unroll
            for (int ps = 0; ps < 32 / RPS; ++ps) {
                const int m = em0 + wm * WTM + i * 32 + ps * RPS + srow;
                if (SEG) {
                    if (m < p.M && n_ok) {
                        const int sg = seg_of(p, en0);
                        const __amdgpu_buffer_rsrc_t srd_c = __builtin_amdgcn_make_buffer_rsrc(p.seg_ptr[sg], 0, -1, 0x00020000);
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, done[ps]), srd_c, (int)seg_offset(p, sg, m, n), 0, 16);
                    }
                } else if (m < p.M && n_ok) {
                    // written through to memory (agent scope) rather than left dirty in this XCD's L2: the next layer's
                    // workgroups run on all XCDs, and what a kernel leaves dirty is written back at its end with nothing
                    // else running (ResNet50 +0.4 %; the non-temporal hint instead: -0.8 %).  A buffer store because that
                    // is the store the compiler lets carry the scope bit: the descriptor starts at the band's first row
                    // (uniform), the lane's offset covers at most 32 rows (ldc < 2^24 on this path).
                    const __amdgpu_buffer_rsrc_t srd_c = __builtin_amdgcn_make_buffer_rsrc(
                        C + (int64_t)(em0 + __builtin_amdgcn_readfirstlane(wm) * WTM + i * 32) * p.ldc, 0, -1, 0x00020000);
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, done[ps]), srd_c,
                        (int)((uint32_t)((ps * RPS + srow) * p.ldc + n) * 4u), 0, 16);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (!more)
            break;
        __syncthreads(); // every wave is done with its scratch before the next tile's operands overwrite it
    }
}
