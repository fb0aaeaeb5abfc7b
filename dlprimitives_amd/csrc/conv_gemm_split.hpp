// fp32 convolutions on the bf16 matrix instruction, without loss of precision.  Included by conv_gemm.hip.
//
// A float is the exact sum of three bf16 numbers (3 x 8 significant bits, each piece rounded to nearest, so that the next one takes what
// is left over): a = a0 + a1 + a2 with |a1| <= 2^-8 |a0| and |a2| <= 2^-16 |a0|.  A product a * b is then the sum of nine products of
// bf16 numbers, each exact in fp32; the three smallest (a1 b2, a2 b1, a2 b2: at most 2^-23 of a * b together, without bias, 2^-25 in the
// root mean square) are left out, six remain.  v_mfma_f32_32x32x16_bf16 is sixteen times as fast per product as the fp32 instruction,
// so six of them leave it 2.7 times ahead -- and it adds several k of a product to the accumulator at once, where the fp32 instruction
// rounds after every k; with the five small products in an accumulator of their own the error against 64 bits is smaller than the fp32
// instruction's (2-norm, K = 64 / 576 / 1152: 4.8e-8 / 1.1e-7 / 1.6e-7 against 1.0e-7 / 3.1e-7 / 4.0e-7).
//
// What does not split is computed on the fp32 instruction: an operand that is infinite, not a number, or so close to the largest float
// that its first piece rounds to infinity leaves an infinity or a NaN in the sums, and a tile whose sums are not all finite is
// computed again, whole, from the same operands as they were (the three pieces of a packed weight add up to it).  So is a tile whose sums
// are so small that bits lost from operands below 2^-110 could count (dlp_internal.hpp), and one with a weight below 2^-110 or above
// 2^16: the packing kernel writes such a weight as a NaN and its 32 bits; weights read in place are looked at as they pass, and so is the input then.
//
//  * K tile = one filter tap x 16 channels = one matrix step; the input is gathered as in conv_gemm_f32_kernel (one masked pixel per
//    lane, a channel per load), split in registers by the thread that loaded it, and stored as three 16-byte pieces of eight channels;
//    the weights are split once, by the packing kernel, into the image of the LDS tile ([piece][half of the channels][row][8]);
//    1x1 convolutions whose weights are not packed ahead read and split the weight tensor in place.
//  * LDS holds [piece][half][row][8 k]: an operand is one 16-byte read per lane, 32 lanes read 512 consecutive bytes.
//  * A wavefront owns 64x64 of the output (64x32 with tiles of 64x128): at six matrix instructions per operand pair of 32x32x16 (192
//    clocks) a 32x32 tile would want 128 bytes per clock and CU from LDS, all there is; 64x64 wants half of that.
//
// Reaches 200 to 215 TFLOP/s of products on long launches (1x1 1024->1024 at 28x28, batch 128: 1662 us on the fp32 instruction, 1038 here; 3x3
// 256->256 at 14x14, batch 512: 825, 563): 1.2e15 bf16 operations a second on operands of random bits, what the library's bf16 product
// reaches on the same card.  At batch 64 (128->128 at 28x28: 151 to 168 TFLOP/s) the matrix units are busy 43 % of the time: a
// launch is little more than one round of workgroups, a SIMD has 1.4 wavefronts on average (2.3 in tiles of 64x128), and a wavefront spends half
// its life ready but not issued, a fifth at barriers and waits, 7 % of it on LDS (11 % in tiles of 64x128; no bank conflicts).
// Loads two K tiles further ahead, or a second set of registers for them, made no difference.

// eight consecutive k of a row -> the 16-byte pieces of its three parts
__device__ __forceinline__ void split8(const float *v, u32x4 (&o)[3])
{
#pragma unroll
    for (int q = 0; q < 4; q++) {
        uint32_t r[3];
        split_pair(v[2 * q], v[2 * q + 1], r);
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
            o[pl][q] = r[pl];
    }
}

// ... for weights: one that is too small to be split, or too large, is left as kWholeWeight (a NaN, which no other weight becomes) and its
// upper and lower 16 bits
constexpr uint32_t kWholeWeight = 0x7FFFu;
__device__ __forceinline__ void split8_weights(const float *v, u32x4 (&o)[3])
{
    split8(v, o);
    uint32_t smallest = kSplitNoSum, largest = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        smallest = split_smallest(smallest, v[e]);
        largest = max(largest, __builtin_bit_cast(uint32_t, v[e]) & 0x7FFFFFFFu);
    }
    if (smallest >= kSplitSmall && largest <= __builtin_bit_cast(uint32_t, kSplitLarge))
        return;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int sh = (e & 1) * 16;
        const uint32_t bits = __builtin_bit_cast(uint32_t, v[e]);
        if (split_smallest(kSplitNoSum, v[e]) >= kSplitSmall && (bits & 0x7FFFFFFFu) <= __builtin_bit_cast(uint32_t, kSplitLarge))
            continue;
        const uint32_t piece[3] = {kWholeWeight, bits >> 16, bits & 0xFFFFu};
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
            o[pl][e / 2] = (o[pl][e / 2] & ~(0xFFFFu << sh)) | (piece[pl] << sh);
    }
}

// PHASED: the workgroups of one of several convolutions of one launch (conv_phases_f32_kernel): `a` is that convolution, its workgroups are
// numbered from zero, its counters and images begin at a.sk_cnt and image_base.
template <int BM, int BN, int WM, int WN, bool ADIR, bool RAGGED, bool PHASED>
__device__ __forceinline__ void conv_split_tile(const GemmArgs &a, const int bid, const uint32_t image_base)
{
    static_assert(WM * WN == 4 && (BN == 128 || BN == 64) && (BM == 64 || BM == 128), "tile shape");
    constexpr int CH = BN / 16; // channels of its pixel that a thread loads
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int TM = WTM / 32, TN = WTN / 32;
    constexpr int A_BYTES = BM * 96, B_BYTES = BN * 96, BUF = A_BYTES + B_BYTES;
    constexpr int A_PIECES = BM * 6;
    constexpr int A_LD = ADIR ? 2 : (A_PIECES + kThreads - 1) / kThreads;

    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * BUF];
    __shared__ float bias_early[BM];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int h = lane >> 5;
    const int wm = wave / WN, wn = wave % WN;

    // tile and K slice of this workgroup: as in conv_gemm_f32_kernel
    int t, slice, splitk = a.splitk, kt_per_slice = a.kt_per_slice;
    uint32_t image0;
    {
        const int tiles = a.mtiles * a.ntiles * a.groups, tiles_main = tiles - a.tail_tiles;
        if (PHASED || bid < a.main_wgs) {
            const int nb = a.main_wgs;
            const int q = nb >> 3, r = nb & 7;
            const int xcd = bid & 7, slot = bid >> 3;
            t = (xcd < r) ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
            slice = (int)fast_div((uint32_t)t, a.tm_magic, a.tm_shift);
            t -= slice * tiles_main;
            image0 = image_base + (uint32_t)(t * splitk);
        } else {
            t = bid - a.main_wgs;
            slice = (int)fast_div((uint32_t)t, a.tt_magic, a.tt_shift);
            t -= slice * a.tail_tiles;
            image0 = (uint32_t)((splitk > 1 ? tiles_main * splitk : 0) + t * a.tail_splitk);
            t += tiles_main;
            splitk = a.tail_splitk;
            kt_per_slice = a.tail_kt;
        }
    }
    const int tm = (int)fast_div((uint32_t)t, a.mt_magic, a.mt_shift);
    const int mt = t - tm * a.mtiles;
    const int g = (int)fast_div((uint32_t)tm, a.ntl_magic, a.ntl_shift);
    const int nt = tm - g * a.ntiles;
    const int m0 = mt * BM, n0 = nt * BN;
    const int kt_begin = slice * kt_per_slice;
    const int kt_end = min(kt_begin + kt_per_slice, a.nkt);
    if (tid < BM)
        bias_early[tid] = (a.bias && m0 + tid < a.M) ? a.bias[g * a.M + m0 + tid] : 0.0f;

    const __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc((void *)((const char *)a.x - a.x_shift), 0, a.x_bytes + a.x_shift, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, a.wp_bytes, 0x00020000);
    ConstInt *ktab = (ConstInt *)a.ktab;

    // ---- the input: one output pixel per thread, its window origin and the mask of its taps inside the image ----
    const int p = tid % BN;
    const int part = __builtin_amdgcn_readfirstlane(tid / BN); // of a K tile's channels, CH of them
    uint32_t vbase, my = 0;
    {
        const int n = n0 + p;
        const int b = (int)fast_div((uint32_t)n, a.ohw_magic, a.ohw_shift);
        const int pix = n - b * a.OHW;
        const int oy = (int)fast_div((uint32_t)pix, a.ow_magic, a.ow_shift);
        const int ox = pix - oy * a.OW;
        const int iy = PHASED ? oy + a.off_h : oy * a.sh, ix = PHASED ? ox + a.off_w : ox * a.sw;
        vbase = (uint32_t)((((b * a.Cin + g * a.Cin_g) * a.H + iy) * a.W + ix) * 4);
        if (n < a.N) {
            uint32_t rx = 0;
            for (int kx = 0; kx < a.KW; kx++) {
                const int xx = ix - a.pw + kx * a.dw;
                rx |= (xx >= 0 && xx < a.W ? 1u : 0u) << kx;
            }
            for (int ky = 0; ky < a.KH; ky++) {
                const int yy = iy - a.ph + ky * a.dh;
                if (yy >= 0 && yy < a.H)
                    my |= rx << (ky * a.KW);
            }
        }
    }
    // ---- the weights: 16-byte pieces of the packed tile in order, or (ADIR) eight channels of a row of the weight tensor ----
    const uint32_t a_tile_bytes = ADIR ? (uint32_t)(BK * 4) : (uint32_t)(a.pack_bm * 96);
    const uint32_t a_row_base = ADIR ? 0u : (uint32_t)((g * a.pack_mtiles + m0 / a.pack_bm) * a.nkt) * a_tile_bytes;
    const int arow = tid % BM, ahalf = tid / BM;
    const int pack_row = m0 % a.pack_bm; // of the packed tile, first row of this one
    uint32_t a_voff[A_LD];
#pragma unroll
    for (int j = 0; j < A_LD; j++) {
        if (ADIR)
            a_voff[j] = (ahalf < 2 && m0 + arow < a.M) ? (uint32_t)(((g * a.M + m0 + arow) * a.K + 8 * ahalf + 4 * j) * 4) : kOutOfRange;
        else
            a_voff[j] = tid + j * kThreads < A_PIECES
                            ? (uint32_t)(((tid + j * kThreads) / BM * a.pack_bm + pack_row + (tid + j * kThreads) % BM) * 16)
                            : kOutOfRange;
    }

    float rb[CH];
    u32x4 ra[A_LD];
    float largest = 0.0f; // ADIR: of this thread's operands
    auto load_b = [&](int kt) {
        ConstInt *e = ktab + min(kt, a.nkt + 1) * 4; // (tiles past the end of K are never multiplied)
        const uint32_t xoff = (uint32_t)e[0], tap = (uint32_t)e[1];
        const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)my, tap, 1u);
        const uint32_t v = opaque((vbase & m) | (kOutOfRange & ~m));
#pragma unroll
        for (int i = 0; i < CH; i++)
            rb[i] = buf_load<float>(xr, v, xoff + (uint32_t)(part * CH + i) * a.hw4);
    };
    auto load_a = [&](int kt) {
        const uint32_t soff = a_row_base + (uint32_t)min(kt, a.nkt - 1) * a_tile_bytes;
#pragma unroll
        for (int j = 0; j < A_LD; j++)
            ra[j] = __builtin_amdgcn_raw_buffer_load_b128(wr, a_voff[j], soff, 0);
    };
    auto store_tile = [&](auto buf_c) {
        unsigned char *const buf = smem + decltype(buf_c)::value * BUF;
        u32x4 o[3];
        if (ADIR) {
            const f32x4 lo = __builtin_bit_cast(f32x4, ra[0]), hi = __builtin_bit_cast(f32x4, ra[1]);
            const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if (BM == 128 || tid < 2 * BM) {
#pragma unroll
                for (int e = 0; e < 8; e += 2)
                    largest = split_largest(largest, v[e], v[e + 1]);
                split8(v, o);
#pragma unroll
                for (int pl = 0; pl < 3; pl++)
                    *(u32x4 *)(buf + ((pl * 2 + ahalf) * BM + arow) * 16) = o[pl];
            }
        } else {
#pragma unroll
            for (int j = 0; j < A_LD; j++)
                if (A_PIECES % kThreads == 0 || tid + j * kThreads < A_PIECES)
                    *(u32x4 *)(buf + (tid + j * kThreads) * 16) = ra[j];
        }
        if (ADIR)
#pragma unroll
            for (int i = 0; i < CH; i += 2)
                largest = split_largest(largest, rb[i], rb[i + 1]);
        if constexpr (CH == 8) {
            split8(rb, o);
#pragma unroll
            for (int pl = 0; pl < 3; pl++)
                *(u32x4 *)(buf + A_BYTES + ((pl * 2 + part) * BN + p) * 16) = o[pl];
        } else {
            uint32_t lo[3], hi[3];
            split_pair(rb[0], rb[1], lo);
            split_pair(rb[2], rb[3], hi);
#pragma unroll
            for (int pl = 0; pl < 3; pl++)
                *(u32x2 *)(buf + A_BYTES + ((pl * 2 + part / 2) * BN + p) * 16 + part % 2 * 8) = (u32x2){lo[pl], hi[pl]};
        }
    };
    // the five small products are summed on their own: in one accumulator with the large one, every step would round the sum six
    // times as often, at its full size
    f32x16 acc[TM][TN], small[TM][TN];
    auto clear = [&](f32x16 (&v)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    v[i][j][r] = 0.0f;
    };
    clear(acc);
    clear(small);

    bf16x8 fa[3][TM], fb[3][TN]; // operands of the K tile at hand, by piece
    auto read_piece = [&](auto buf_c, int pl) {
        const unsigned char *const buf = smem + decltype(buf_c)::value * BUF;
#pragma unroll
        for (int i = 0; i < TM; i++)
            fa[pl][i] = *(const bf16x8 *)(buf + ((pl * 2 + h) * BM + wm * WTM + i * 32 + l32) * 16);
#pragma unroll
        for (int j = 0; j < TN; j++)
            fb[pl][j] = *(const bf16x8 *)(buf + A_BYTES + ((pl * 2 + h) * BN + wn * WTN + j * 32 + l32) * 16);
    };
    auto multiply = [&](f32x16 (&c)[TM][TN], int pa, int pb) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[pa][i], fb[pb][j], c[i][j], 0, 0, 0);
    };
    // One K tile, its operands in registers.  One barrier, in the middle: before it the next tile is split and goes from its registers to
    // LDS[P ^ 1] (and the one after is requested); behind it the next tile's operands replace this one's, piece by piece, as soon as the
    // last product that wants a piece has been issued, so that a wavefront alone on its SIMD does not wait for LDS either.
    auto k_step = [&](auto par, int kt) {
        using Other = std::integral_constant<int, decltype(par)::value ^ 1>;
        multiply(small, 1, 1);
        multiply(small, 1, 0);
        store_tile(Other{});
        load_b(kt + 2);
        load_a(kt + 2);
        __syncthreads();
        multiply(small, 0, 1);
        __builtin_amdgcn_sched_barrier(0); // keep this order: the scheduler would sink the operand reads to their uses
        read_piece(Other{}, 1);
        multiply(small, 2, 0);
        multiply(small, 0, 2);
        __builtin_amdgcn_sched_barrier(0);
        read_piece(Other{}, 2);
        multiply(acc, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        read_piece(Other{}, 0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    load_b(kt_begin);
    load_a(kt_begin);
    store_tile(I0{});
    load_b(kt_begin + 1);
    load_a(kt_begin + 1);
    __syncthreads();
    read_piece(I0{}, 1);
    read_piece(I0{}, 2);
    read_piece(I0{}, 0);
    int kt = kt_begin;
    for (; kt + 1 < kt_end; kt += 2) {
        k_step(I0{}, kt);
        k_step(I1{}, kt + 1);
    }
    if (kt < kt_end)
        k_step(I0{}, kt);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
            acc[i][j] += small[i][j];

    // sums that are not finite or too small, operands too large: the tile again on the fp32 instruction
    float finite = 0.0f; // 0 * infinity and 0 * NaN are NaN, which is not equal to zero
    bool small_sum = false;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                v[r] = acc[i][j][r];
                finite = fmaf(v[r], 0.0f, finite);
            }
            small_sum |= split_small_sum(v);
        }
    if (__syncthreads_or(finite != 0.0f || small_sum || largest > kSplitLarge)) {
        clear(acc);
        float *const Af = reinterpret_cast<float *>(smem), *const Bf = Af + BK * BM; // [k][row], [k][pixel]
        for (kt = kt_begin; kt < kt_end; kt++) {
            load_b(kt);
            if (tid < 2 * BM) {
                const uint32_t soff = a_row_base + (uint32_t)kt * a_tile_bytes;
                float v[8];
                if (ADIR) {
                    load_a(kt);
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        v[e] = __builtin_bit_cast(f32x4, ra[e / 4])[e % 4];
                } else {
                    u32x4 o[3];
#pragma unroll
                    for (int pl = 0; pl < 3; pl++)
                        o[pl] = __builtin_amdgcn_raw_buffer_load_b128(wr, (uint32_t)(((pl * 2 + ahalf) * a.pack_bm + pack_row + arow) * 16), soff, 0);
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        uint32_t piece[3]; // in the upper half
#pragma unroll
                        for (int pl = 0; pl < 3; pl++)
                            piece[pl] = (e & 1) ? o[pl][e / 2] & 0xFFFF0000u : o[pl][e / 2] << 16;
                        v[e] = __builtin_bit_cast(float, piece[0]) + __builtin_bit_cast(float, piece[1]) + __builtin_bit_cast(float, piece[2]);
                        if (piece[0] == kWholeWeight << 16)
                            v[e] = __builtin_bit_cast(float, piece[1] | (piece[2] >> 16));
                    }
                }
#pragma unroll
                for (int e = 0; e < 8; e++)
                    Af[(ahalf * 8 + e) * BM + arow] = v[e];
            }
#pragma unroll
            for (int i = 0; i < CH; i++)
                Bf[(part * CH + i) * BN + p] = rb[i];
            __syncthreads();
#pragma unroll
            for (int kk = 0; kk < BK / 2; kk++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(Af[(2 * kk + h) * BM + wm * WTM + i * 32 + l32],
                                                                         Bf[(2 * kk + h) * BN + wn * WTN + j * 32 + l32], acc[i][j], 0, 0, 0);
            __syncthreads();
        }
    }
    gemm_tile_output<float, BM, BN, WM, WN, ACT_CLAMP, RAGGED, PHASED>(a, acc, reinterpret_cast<float *>(smem), m0, n0, g, slice, splitk, image0, wm, wn,
                                                                       h, l32, tid, bias_early);
}

template <int BM, int BN, int WM, int WN, bool ADIR, bool RAGGED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void conv_split_f32_kernel(GemmArgs a)
{
    conv_split_tile<BM, BN, WM, WN, ADIR, RAGGED, false>(a, blockIdx.x, 0);
}

// All stride phases of a backward-data pass or transposed convolution in one launch: stride-1 convolutions of one input with filters,
// extents and paddings of their own, every one storing its share of the pixels of y, with bias, activation and old value.  One launch a phase
// into planes that another kernel interleaved left the chip half empty four times over (BM x BN tiles of one phase: 100 to 230 workgroups)
// and took the output through memory twice more.
struct SplitPhase {
    const int32_t *ktab;
    uint32_t wp_offset; // bytes into the packed weights
    int nkt, N, ntiles, KH, KW, ph, pw, dh, dw, off_h, off_w, OW, OHW, out_off;
    uint32_t x_shift, ohw_magic, ohw_shift, ow_magic, ow_shift, ntl_magic, ntl_shift, tm_magic, tm_shift;
    int block0, blocks;    // workgroups
    int splitk, kt_per_slice, counter0;
    uint32_t image0;
};
constexpr int kMaxMergedPhases = 9;
struct PhasesArgs {
    GemmArgs a; // what the phases have in common
    int n;
    SplitPhase ph[kMaxMergedPhases];
};
template <int BM, int BN, int WM, int WN, bool RAGGED>
__device__ __forceinline__ void conv_phases_tile(const PhasesArgs &args)
{
    int i = 0;
    while (i + 1 < args.n && (int)blockIdx.x >= args.ph[i + 1].block0)
        i++;
    const SplitPhase &p = args.ph[i];
    GemmArgs a = args.a;
    a.ktab = p.ktab;
    a.wp = (const float *)((const char *)a.wp + p.wp_offset);
    a.wp_bytes -= p.wp_offset;
    a.nkt = p.nkt;
    a.N = p.N;
    a.ntiles = p.ntiles;
    a.KH = p.KH; a.KW = p.KW; a.ph = p.ph; a.pw = p.pw; a.dh = p.dh; a.dw = p.dw;
    a.off_h = p.off_h; a.off_w = p.off_w; a.OW = p.OW; a.OHW = p.OHW; a.out_off = p.out_off;
    a.x_shift = p.x_shift;
    a.ohw_magic = p.ohw_magic; a.ohw_shift = p.ohw_shift; a.ow_magic = p.ow_magic; a.ow_shift = p.ow_shift;
    a.ntl_magic = p.ntl_magic; a.ntl_shift = p.ntl_shift; a.tm_magic = p.tm_magic; a.tm_shift = p.tm_shift;
    a.splitk = p.splitk;
    a.kt_per_slice = p.kt_per_slice;
    a.tail_tiles = 0;
    a.main_wgs = p.blocks;
    a.sk_cnt = p.splitk > 1 ? a.sk_cnt + p.counter0 : nullptr;
    conv_split_tile<BM, BN, WM, WN, false, RAGGED, true>(a, (int)blockIdx.x - p.block0, p.image0);
}
// tiles as conv_split_f32_kernel has them for one convolution, and smaller ones for launches below its sizes
template <int BM, int BN, int WM, int WN, bool ADIR, bool RAGGED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void conv_split_f32_kernel(PhasesArgs args)
{
    conv_phases_tile<BM, BN, WM, WN, RAGGED>(args);
}
template <int BM, int BN, int WM, int WN, bool RAGGED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void conv_phases_f32_kernel(PhasesArgs args)
{
    conv_phases_tile<BM, BN, WM, WN, RAGGED>(args);
}

// Weights -> [group][m tile][K tile][piece][half][row][8 channels of one tap], zero padded.  One workgroup moves 16 filters x 16 channels
// through LDS (read in runs of whole filter rows, 16 bytes per lane where the tensor is aligned); a thread then splits eight channels
// of a filter at a time.  floats: the same weights once more, as tiles of f_bm rows for the kernels on the fp32 instruction.
__global__ __launch_bounds__(256) void pack_weights_split_kernel(GemmPlan p, int ncb, int khw, int aligned, const float *__restrict__ w,
                                                                 u32x4 *__restrict__ out, float *__restrict__ floats, int f_bm, int f_mtiles)
{
    extern __shared__ __align__(16) unsigned char split_smem[];
    float *lds = reinterpret_cast<float *>(split_smem);
    const int run = BK * khw, ld = run + 1;
    const int mchunks = p.BM / 16;
    int bid = (int)blockIdx.x;
    const int mc = bid % mchunks;
    bid /= mchunks;
    const int cb = bid % ncb;
    bid /= ncb;
    const int mt = bid % p.mtiles;
    const int g = bid / p.mtiles;
    const int m_base = mt * p.BM + mc * 16;
    const float *src = w + (size_t)g * p.M * p.K + (size_t)cb * run;
    const int wv = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    if (aligned) {
        for (int j = lane * 4; j < run; j += 256) {
            f32x4 v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int m = m_base + wv + 4 * q;
                v[q] = (f32x4)0.0f;
                if (m < p.M)
                    v[q] = *reinterpret_cast<const f32x4 *>(src + (size_t)m * p.K + j);
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    lds[(wv + 4 * q) * ld + j + e] = v[q][e];
        }
    } else {
        for (int j = lane; j < run; j += 64)
            for (int q = 0; q < 4; q++) {
                const int m = m_base + wv + 4 * q;
                lds[(wv + 4 * q) * ld + j] = m < p.M ? src[(size_t)m * p.K + j] : 0.0f;
            }
    }
    __syncthreads();
    u32x4 *const tile0 = out + ((size_t)(g * p.mtiles + mt) * p.nkt + (size_t)cb * khw) * (6 * p.BM) + mc * 16;
    for (int idx = (int)threadIdx.x; idx < 32 * khw; idx += 256) {
        const int r = idx % 16, half = (idx / 16) % 2, tap = idx / 32;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++)
            v[e] = lds[r * ld + (half * 8 + e) * khw + tap];
        u32x4 o[3];
        split8_weights(v, o);
        u32x4 *const dst = tile0 + (size_t)tap * (6 * p.BM) + half * p.BM + r;
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
            dst[(size_t)pl * 2 * p.BM] = o[pl];
    }
    if (floats != nullptr && m_base / f_bm < f_mtiles) { // rows 16 at a time: f_bm is a multiple
        float *const ftile0 = floats + ((size_t)(g * f_mtiles + m_base / f_bm) * p.nkt + (size_t)cb * khw) * (BK * f_bm) + m_base % f_bm;
        for (int idx = (int)threadIdx.x; idx < 16 * BK * khw; idx += 256) {
            const int r = idx % 16, k = (idx / 16) % BK, tap = idx / (16 * BK);
            ftile0[(size_t)tap * (BK * f_bm) + k * f_bm + r] = lds[r * ld + k * khw + tap];
        }
    }
}

// Filters of a backward-data pass, packed straight from w[group][k][c][KH][KW]: a phase's convolution maps dy (channels k) to dx (rows c)
// with the taps (rh0 + (nh - 1 - jh) * rhstep, rw0 + (nw - 1 - jw) * rwstep).  One launch for all phases, about 5 us, in the place of one
// transposing and one packing launch per phase at 4 to 5 us each whatever their size.  A thread has one k (float tiles) or eight
// consecutive k (split tiles) of one row; rows are contiguous in the packed tile, so the stores coalesce and the caches serve the loads.
struct PhasePack {
    void *out;
    int nh, nw, rh0, rhstep, rw0, rwstep;
    int BM, nkt, mtiles, split;
    uint32_t units, block0; // threads with something to do, first workgroup
};
struct PhasePackArgs {
    int n, cout_g, cin_g, KH, KW;
    int *zero; // tile counters of the launch that follows
    int nzero;
    PhasePack ph[kMaxPhases];
};
__global__ __launch_bounds__(256) void phase_pack_kernel(const float *__restrict__ w, PhasePackArgs a)
{
    for (int z = blockIdx.x * 256 + threadIdx.x; z < a.nzero; z += gridDim.x * 256)
        a.zero[z] = 0;
    int i = 0;
    while (i + 1 < a.n && blockIdx.x >= a.ph[i + 1].block0)
        i++;
    const PhasePack &p = a.ph[i];
    const uint32_t unit = (blockIdx.x - p.block0) * 256u + threadIdx.x;
    if (unit >= p.units)
        return;
    const uint32_t per_row = p.split ? 2 : BK;
    uint32_t q = unit / (uint32_t)p.BM;
    const int row = (int)(unit - q * (uint32_t)p.BM);
    const int k = (int)(q % per_row);
    q /= per_row;
    const uint32_t tile = q; // (group, m tile, K tile)
    const int kt = (int)(q % (uint32_t)p.nkt);
    q /= (uint32_t)p.nkt;
    const int mt = (int)(q % (uint32_t)p.mtiles), g = (int)(q / (uint32_t)p.mtiles);
    const int taps = p.nh * p.nw, cb = kt / taps, tap = kt - cb * taps;
    const int jh = tap / p.nw, jw = tap - jh * p.nw;
    const int rh = p.rh0 + (p.nh - 1 - jh) * p.rhstep, rw = p.rw0 + (p.nw - 1 - jw) * p.rwstep;
    const int c = mt * p.BM + row;
    const bool ok = c < a.cin_g;
    const size_t step = (size_t)a.cin_g * a.KH * a.KW; // from one k to the next
    const float *src = w + (size_t)(g * a.cout_g + cb * BK) * step + ((size_t)c * a.KH + rh) * a.KW + rw;
    if (!p.split) {
        ((float *)p.out)[unit] = ok ? src[k * step] : 0.0f;
        return;
    }
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++)
        v[e] = ok ? src[(k * 8 + e) * step] : 0.0f;
    u32x4 o[3];
    split8_weights(v, o);
    u32x4 *const dst = (u32x4 *)p.out + (size_t)tile * (6 * p.BM) + k * p.BM + row;
#pragma unroll
    for (int pl = 0; pl < 3; pl++)
        dst[(size_t)pl * 2 * p.BM] = o[pl];
}
