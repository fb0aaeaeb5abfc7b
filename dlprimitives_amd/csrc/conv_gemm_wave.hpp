// Convolutions too small for the tiles of the other kernels: one 32x32 output tile per workgroup, its reduction dealt to the wavefronts.
// Included by conv_gemm.hip.
//
// A network run on one image is a chain of dependent launches, each of which is over before a chip of 256 CUs is full: what counts is
// the time from the first load to the last store, not throughput.  Tiles of 128x128 give a 14x14 layer 4 to 16 workgroups whose K
// loop (72 K tiles of 32 for 3x3 256->256) runs serially, behind a barrier a K tile, and K slices need a second launch to be added up.  Here:
//  * Tiles of 32x32, or 16x16: 49 to 800 workgroups for the layers of a ResNet on one image.
//  * The K tiles are dealt to KW wavefronts of the workgroup; each has four (eight) K tiles on their way, four lanes to the 64 bytes a K
//    tile has of a pixel or filter.  (Loaded in operand order, a lane to a pixel, a load takes a cycle a lane instead of a quarter: 55 GB/s a CU
//    instead of 150 and 13.5 us instead of 9.8 for 32 tiles of 144 K tiles.)  They go through a part of LDS of the wavefront's own to
//    the registers of the matrix instruction: no barrier in the loop, a wavefront waits for its own loads only.
//  * The partial sums meet in LDS, once; every thread adds up some outputs and stores them.  Old values and bias are requested before the loop.
// What it gives up is reuse: an operand byte read from the caches serves 32 outputs, not 128, so that a launch of many tiles is bound by what
// the CUs read from the caches (bf16_wave; 64x64 tiles of four wavefronts on the same lines were no faster).
// ResNet-50 on one image: 618 us on the tiles of 128x128 and the LDS-patch kernel, 295 on these (of launches captured in a graph).

template <int TILE, int KW, bool YCL>
__global__ __launch_bounds__(KW * 64) void conv_wave_bf16_kernel(GemmArgs a)
{
    static_assert(TILE == 32 || TILE == 16, "shapes of the matrix instruction");
    constexpr int R = TILE * TILE / 64;      // accumulators of a lane
    constexpr int V = R >= KW ? R / KW : 1;  // outputs per thread
    constexpr int S = TILE / 16;             // matrix instructions per K tile
    constexpr int DEPTH = 8 / S;             // K tiles on their way
    typedef float acc_t __attribute__((ext_vector_type(R)));
    __shared__ __attribute__((aligned(16))) unsigned char smem[KW * TILE * 128]; // operands: [wavefront][input, weights][row][64 bytes]
    float(*const red)[R][64] = reinterpret_cast<float(*)[R][64]>(smem);          // sums: [wavefront][register][lane]
    static_assert(KW * R * 64 * sizeof(float) <= sizeof(smem), "the sums fit the operands' place");

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int l = lane % TILE;
    const int h = lane / TILE; // eight k of an instruction's 8 * 64 / TILE

    int t; // pixel tiles fastest; an XCD gets a run of tiles, so that its L2 holds few rows of weights
    {
        const int nb = gridDim.x, bid = blockIdx.x;
        const int q = nb >> 3, r = nb & 7;
        const int xcd = bid & 7, slot = bid >> 3;
        t = (xcd < r) ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
    }
    const int tm = (int)fast_div((uint32_t)t, a.ntl_magic, a.ntl_shift);
    const int n0 = (t - tm * a.ntiles) * TILE;
    const int g = (int)fast_div((uint32_t)tm, a.mt_magic, a.mt_shift);
    const int m0 = (tm - g * a.mtiles) * TILE;

    const __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc((void *)((const char *)a.x - a.x_shift), 0, a.x_bytes + a.x_shift, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, a.wp_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);

    // ---- what this lane loads of a K tile: 16 bytes of S pixels and S weight rows, four lanes the 64 bytes of one ----
    uint32_t xbase[S], xmask[S], a_voff[S], slot[S];
    uint32_t a_tile_bytes = (uint32_t)(a.pack_bm * BK2 * 2);
    uint32_t a_base = (uint32_t)((g * a.pack_mtiles + m0 / a.pack_bm) * a.nkt) * a_tile_bytes;
    if (a.wdirect) { // the weight tensor itself
        a_tile_bytes = BK2 * 2;
        a_base = 0;
    }
#pragma unroll
    for (int s = 0; s < S; s++) {
        const int row = lane / 4 + 16 * s, piece = lane % 4;
        slot[s] = (uint32_t)(row * 64 + (piece ^ ((row >> 1) & 3)) * 16);
        if (a.wdirect)
            a_voff[s] = m0 + row < a.M ? (uint32_t)((g * a.M + m0 + row) * a.K * 2 + piece * 16) : kOutOfRange;
        else
            a_voff[s] = (uint32_t)((m0 % a.pack_bm + row) * (BK2 * 2) + piece * 16);
        const int n = n0 + row;
        const int b = (int)fast_div((uint32_t)n, a.ohw_magic, a.ohw_shift);
        const int pix = n - b * a.OHW;
        const int oy = (int)fast_div((uint32_t)pix, a.ow_magic, a.ow_shift);
        const int ox = pix - oy * a.OW;
        xbase[s] = kOutOfRange;
        xmask[s] = 0;
        if (n < a.N) {
            xbase[s] = (uint32_t)((((b * a.H + oy * a.sh) * a.W + ox * a.sw) * a.Cin + g * a.Cin_g) * 2 + piece * 16);
            uint32_t rx = 0;
            for (int kx = 0; kx < a.KW; kx++) {
                const int xx = ox * a.sw - a.pw + kx * a.dw;
                rx |= (xx >= 0 && xx < a.W ? 1u : 0u) << kx;
            }
            for (int ky = 0; ky < a.KH; ky++) {
                const int yy = oy * a.sh - a.ph + ky * a.dh;
                if (yy >= 0 && yy < a.H)
                    xmask[s] |= rx << (ky * a.KW);
            }
        }
    }

    // ---- this wavefront's K tiles: one tap x 32 channels each, the channels of a tap one behind the other (whole lines of a pixel) ----
    const int taps = a.KH * a.KW, ncb = a.nkt / taps;
    const int kt_begin = wave * a.nkt / KW, kt_end = (wave + 1) * a.nkt / KW;
    int lt = kt_begin, cb, tap, kx; // next tile to be loaded, its channels, its tap and the tap's column
    uint32_t tap_byte;              // ... and byte offset
    {
        tap = (int)fast_div((uint32_t)lt, a.ncb_magic, a.ncb_shift);
        cb = lt - tap * ncb;
        const int ky = a.KW == 1 ? tap : tap / a.KW;
        kx = tap - ky * a.KW;
        tap_byte = (uint32_t)((ky * a.dh * a.W + kx * a.dw) * a.Cin * 2);
    }
    u32x4 xv[DEPTH][S], wv[DEPTH][S];
    auto load = [&](auto slot_c) {
        constexpr int Q = decltype(slot_c)::value;
        if (lt >= kt_end)
            return;
        const uint32_t xoff = tap_byte + (uint32_t)cb * (BK2 * 2), woff = a_base + (uint32_t)(cb * taps + tap) * a_tile_bytes;
#pragma unroll
        for (int s = 0; s < S; s++) {
            const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)xmask[s], (uint32_t)tap, 1u);
            xv[Q][s] = __builtin_amdgcn_raw_buffer_load_b128(xr, opaque((xbase[s] & m) | (kOutOfRange & ~m)), xoff, 0);
            wv[Q][s] = __builtin_amdgcn_raw_buffer_load_b128(wr, a_voff[s], woff, 0);
        }
        lt++;
        if (++cb == ncb) {
            cb = 0;
            tap++;
            tap_byte += (uint32_t)(a.dw * a.Cin * 2);
            if (++kx == a.KW) {
                kx = 0;
                tap_byte += (uint32_t)((a.dh * a.W - a.KW * a.dw) * a.Cin * 2);
            }
        }
    };
    static_for_n<DEPTH>(load);

    // ---- this thread's outputs: the tile's accumulator r is row 8 * (r / 4) + 4 * h + r % 4, column l ----
    const bool mine = wave * V < R;
    uint32_t yoff[V];
    float bias[V];
    uint32_t old[V];
    const bool pre = a.pre != 0 && a.factor != 0.0f;
#pragma unroll
    for (int v = 0; v < V; v++) {
        const int r = wave * V + v, row = 8 * (r >> 2) + 4 * h + (r & 3);
        const int m = m0 + (YCL ? l : row), n = n0 + (YCL ? row : l);
        yoff[v] = kOutOfRange;
        bias[v] = 0.0f;
        old[v] = 0;
        if (mine && m < a.M && n < a.N) {
            if (YCL)
                yoff[v] = (uint32_t)(n * a.Cout + g * a.M + m) * 2u;
            else {
                const int b = (int)fast_div((uint32_t)n, a.ohw_magic, a.ohw_shift);
                yoff[v] = (uint32_t)((b * a.Cout + g * a.M + m) * a.OHW + n - b * a.OHW) * 2u;
            }
            if (a.bias)
                bias[v] = a.bias[g * a.M + m];
        }
        if (a.factor != 0.0f)
            old[v] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(yr, yoff[v], 0, 0);
    }

    unsigned char *const mine_s = smem + wave * (TILE * 128);
    uint32_t read[S]; // of this lane's row, the eight k it gives to matrix instruction s
#pragma unroll
    for (int s = 0; s < S; s++)
        read[s] = (uint32_t)(l * 64 + ((s * (4 / S) + h) ^ ((l >> 1) & 3)) * 16);
    acc_t acc;
#pragma unroll
    for (int r = 0; r < R; r++)
        acc[r] = 0.0f;
    for (int kt = kt_begin; kt < kt_end; kt += DEPTH)
        static_for_n<DEPTH>([&](auto slot_c) {
            constexpr int Q = decltype(slot_c)::value;
            if (kt + Q < kt_end) {
                // LDS works a wavefront's instructions off in order, and nobody else touches its part: no barrier, no second buffer
#pragma unroll
                for (int s = 0; s < S; s++) {
                    *(u32x4 *)(mine_s + slot[s]) = xv[Q][s];
                    *(u32x4 *)(mine_s + TILE * 64 + slot[s]) = wv[Q][s];
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                bf16x8 xf[S], wf[S];
#pragma unroll
                for (int s = 0; s < S; s++) {
                    xf[s] = *(const bf16x8 *)(mine_s + read[s]);
                    wf[s] = *(const bf16x8 *)(mine_s + TILE * 64 + read[s]);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int s = 0; s < S; s++) {
                    const bf16x8 x = xf[s], w = wf[s];
                    const bf16x8 rows = YCL ? x : w, cols = YCL ? w : x;
                    if constexpr (TILE == 32)
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rows, cols, acc, 0, 0, 0);
                    else
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rows, cols, acc, 0, 0, 0);
                }
                load(slot_c);
            }
        });

    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++)
        red[wave][r][lane] = acc[r];
    __syncthreads();
    if (!mine)
        return;
#pragma unroll
    for (int v = 0; v < V; v++) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < KW; w++)
            sum += red[w][wave * V + v][lane];
        sum += bias[v];
        const float o = __builtin_bit_cast(float, old[v] << 16);
        if (pre)
            sum = fmaf(o, a.factor, sum);
        if (a.act != DLP_ACT_IDENTITY) // identity must keep NaNs: no min/max
            sum = clamp_med3(sum, a.clamp_lo, a.clamp_hi);
        if (!pre && a.factor != 0.0f)
            sum = fmaf(o, a.factor, sum);
        __builtin_amdgcn_raw_buffer_store_b16((short)to_bf16(sum).bits, yr, yoff[v], 0, 0);
    }
}

// The same for float tensors, [image][channel][pixel], on the weight tensor as it lies: nothing is packed.  k = (channel, tap) as in a row of
// the weight tensor; a K tile is KT consecutive k.
//  * Weights: the KT * 4 bytes a K tile has of a row are loaded by consecutive lanes and go through a part of LDS of the wavefront's own; a
//    lane then reads the eight k that it gives to the matrix instruction.
//  * Input: a load a k, consecutive lanes on consecutive pixels, straight into the register of that k.  Where k lies and which tap of the window it
//    is comes from a table in LDS, made when the workgroup starts (POINT: 1x1, no table).
//  * Both are split into three bf16 parts as in conv_split_f32_kernel, by every lane for the eight k it has of its row and of its pixel: six
//    products in two accumulators.  A tile that such products cannot hold (operands above 2^16, sums not finite or too small) is computed again,
//    whole, on the fp32 instruction.
// A K tile of a 32x32 tile takes a CU some 140 clocks of vector instructions (two splits), 100 of loads, 48 of matrix instructions.
template <int TILE, int KW, bool POINT>
__global__ __launch_bounds__(KW * 64) void conv_wave_f32_kernel(GemmArgs a)
{
    static_assert(TILE == 32 || TILE == 16, "shapes of the matrix instruction");
    constexpr int R = TILE * TILE / 64;     // accumulators of a lane
    constexpr int V = R >= KW ? R / KW : 1; // outputs per thread
    constexpr int KT = TILE == 32 ? 16 : 32;
    constexpr int PIECES = KT / 4; // of 16 bytes, of a row
    constexpr int DEPTH = 2;       // K tiles on their way
    typedef float acc_t __attribute__((ext_vector_type(R)));
    // weights [wavefront][row][KT], later the sums [wavefront][register][lane] | table {byte offset, tap} [K, rounded up]
    constexpr int OPERANDS = KW * TILE * KT * 4, SUMS = KW * R * 256;
    extern __shared__ __attribute__((aligned(16))) unsigned char wave_smem[];
    float(*const red)[R][64] = reinterpret_cast<float(*)[R][64]>(wave_smem);
    u32x2 *const tab = reinterpret_cast<u32x2 *>(wave_smem + (OPERANDS > SUMS ? OPERANDS : SUMS));

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int l = lane % TILE;
    const int h = lane / TILE; // eight k of the K tile

    int t; // as in conv_wave_bf16_kernel
    {
        const int nb = gridDim.x, bid = blockIdx.x;
        const int q = nb >> 3, r = nb & 7;
        const int xcd = bid & 7, slot = bid >> 3;
        t = (xcd < r) ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
    }
    const int tm = (int)fast_div((uint32_t)t, a.ntl_magic, a.ntl_shift);
    const int n0 = (t - tm * a.ntiles) * TILE;
    const int g = (int)fast_div((uint32_t)tm, a.mt_magic, a.mt_shift);
    const int m0 = (tm - g * a.mtiles) * TILE;

    const __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc((void *)((const char *)a.x - a.x_shift), 0, a.x_bytes + a.x_shift, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, a.wp_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);

    const int nkt = (a.K + KT - 1) / KT, taps = a.KH * a.KW;
    if constexpr (!POINT) {
        for (int k = threadIdx.x; k < nkt * KT; k += KW * 64) {
            const int c = (int)fast_div((uint32_t)k, a.ncb_magic, a.ncb_shift), tap = k - c * taps;
            const int ky = (int)fast_div((uint32_t)tap, a.nt_magic, a.nt_shift), kx = tap - ky * a.KW;
            u32x2 e = {(uint32_t)(((c * a.H + ky * a.dh) * a.W + kx * a.dw) * 4), (uint32_t)tap};
            if (k >= a.K)
                e = (u32x2){0, 31}; // a tap that no window has
            tab[k] = e;
        }
        __syncthreads();
    }

    // ---- this lane's pixel ----
    uint32_t xbase = POINT ? kOutOfRange : 0u, xmask = 0;
    {
        const int n = n0 + l;
        const int b = (int)fast_div((uint32_t)n, a.ohw_magic, a.ohw_shift);
        const int pix = n - b * a.OHW;
        const int oy = (int)fast_div((uint32_t)pix, a.ow_magic, a.ow_shift);
        const int ox = pix - oy * a.OW;
        if (n < a.N) {
            xbase = (uint32_t)((((b * a.Cin + g * a.Cin_g) * a.H + oy * a.sh) * a.W + ox * a.sw) * 4);
            uint32_t rx = 0;
            for (int kx = 0; kx < a.KW; kx++) {
                const int xx = ox * a.sw - a.pw + kx * a.dw;
                rx |= (xx >= 0 && xx < a.W ? 1u : 0u) << kx;
            }
            for (int ky = 0; ky < a.KH; ky++) {
                const int yy = oy * a.sh - a.ph + ky * a.dh;
                if (yy >= 0 && yy < a.H)
                    xmask |= rx << (ky * a.KW);
            }
            if (POINT) {
                xbase = (xmask & 1u) ? xbase + (uint32_t)(8 * h) * a.hw4 : kOutOfRange;
            }
        }
    }
    // ---- what this lane loads of the weights: 16 bytes of two rows, and where they go ----
    uint32_t wvoff[2], slot[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int row = (lane + 64 * s) / PIECES, piece = (lane + 64 * s) % PIECES;
        wvoff[s] = m0 + row < a.M ? (uint32_t)(((g * a.M + m0 + row) * a.K + piece * 4) * 4) : kOutOfRange;
        slot[s] = (uint32_t)((row * PIECES + (piece ^ (TILE == 32 ? (row >> 1) & 3 : row & 7))) * 16);
    }
    unsigned char *const mine_s = wave_smem + wave * (TILE * KT * 4);
    uint32_t read[2];
#pragma unroll
    for (int s = 0; s < 2; s++)
        read[s] = (uint32_t)((l * PIECES + ((2 * h + s) ^ (TILE == 32 ? (l >> 1) & 3 : l & 7))) * 16);

    const int kt_begin = wave * nkt / KW, kt_end = (wave + 1) * nkt / KW;
    float xv[DEPTH][8];
    u32x4 wv[DEPTH][2];
    auto load = [&](auto slot_c, int kt) {
        constexpr int Q = decltype(slot_c)::value;
        if (kt >= kt_end)
            return;
        if ((kt + 1) * KT <= a.K) {
#pragma unroll
            for (int s = 0; s < 2; s++)
                wv[Q][s] = __builtin_amdgcn_raw_buffer_load_b128(wr, wvoff[s], (uint32_t)(kt * KT * 4), 0);
        } else { // what follows the row's end is the next row, or nothing
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int k = kt * KT + (lane + 64 * s) % PIECES * 4 + e;
                    wv[Q][s][e] = __builtin_amdgcn_raw_buffer_load_b32(wr, opaque(k < a.K ? wvoff[s] : kOutOfRange), (uint32_t)((kt * KT + e) * 4), 0);
                }
        }
        if constexpr (POINT) {
            const int left = a.K - kt * KT - 8 * h; // of this lane's k inside the reduction
#pragma unroll
            for (int e = 0; e < 8; e++)
                xv[Q][e] = buf_load<float>(xr, opaque(e < left ? xbase : kOutOfRange), (uint32_t)(kt * KT + e) * a.hw4);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const u32x2 te = tab[kt * KT + 8 * h + e];
                const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)xmask, te[1], 1u);
                xv[Q][e] = buf_load<float>(xr, opaque(((xbase + te[0]) & m) | (kOutOfRange & ~m)), 0);
            }
        }
    };
    static_for_n<DEPTH>([&](auto slot_c) { load(slot_c, kt_begin + decltype(slot_c)::value); });

    // ---- this thread's outputs: the tile's accumulator r is row 8 * (r / 4) + 4 * h + r % 4 (a filter), column l (a pixel) ----
    const bool mine = wave * V < R;
    uint32_t yoff[V];
    float bias[V], old[V];
    const bool pre = a.pre != 0 && a.factor != 0.0f;
#pragma unroll
    for (int v = 0; v < V; v++) {
        const int r = wave * V + v, m = m0 + 8 * (r >> 2) + 4 * h + (r & 3), n = n0 + l;
        yoff[v] = kOutOfRange;
        bias[v] = old[v] = 0.0f;
        if (mine && m < a.M && n < a.N) {
            const int b = (int)fast_div((uint32_t)n, a.ohw_magic, a.ohw_shift);
            yoff[v] = (uint32_t)((b * a.Cout + g * a.M + m) * a.OHW + n - b * a.OHW) * 4u;
            if (a.bias)
                bias[v] = a.bias[g * a.M + m];
        }
        if (a.factor != 0.0f)
            old[v] = buf_load<float>(yr, yoff[v], 0);
    }

    acc_t acc, small;
#pragma unroll
    for (int r = 0; r < R; r++)
        acc[r] = small[r] = 0.0f;
    float largest = 0.0f;
    auto multiply = [&](acc_t &c, const u32x4 &w, const u32x4 &x) {
        const bf16x8 wf = __builtin_bit_cast(bf16x8, w), xf = __builtin_bit_cast(bf16x8, x);
        if constexpr (TILE == 32)
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, xf, c, 0, 0, 0);
        else
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf, c, 0, 0, 0);
    };
    // IN_FLOATS: the products on the fp32 instruction, whose k a lane gives one at a time
    auto reduce = [&](auto in_floats_c) {
        constexpr bool IN_FLOATS = decltype(in_floats_c)::value;
        for (int kt = kt_begin; kt < kt_end; kt += DEPTH)
            static_for_n<DEPTH>([&](auto slot_c) {
                constexpr int Q = decltype(slot_c)::value;
                if (kt + Q < kt_end) {
                    // LDS works a wavefront's instructions off in order, and nobody else touches its part: no barrier, no second buffer
#pragma unroll
                    for (int s = 0; s < 2; s++)
                        *(u32x4 *)(mine_s + slot[s]) = wv[Q][s];
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    float w[8], x[8];
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        const f32x4 p = *(const f32x4 *)(mine_s + read[s]);
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            w[4 * s + e] = p[e];
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        x[e] = xv[Q][e];
                    load(slot_c, kt + Q + DEPTH);
                    if constexpr (IN_FLOATS) {
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            if constexpr (TILE == 32)
                                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(w[e], x[e], acc, 0, 0, 0);
                            else
                                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[e], acc, 0, 0, 0);
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            largest = split_largest(largest, w[e], w[e + 1]);
                            largest = split_largest(largest, x[e], x[e + 1]);
                        }
                        u32x4 wp[3], xp[3];
                        split8(w, wp);
                        split8(x, xp);
                        multiply(acc, wp[0], xp[0]);
                        multiply(small, wp[1], xp[1]);
                        multiply(small, wp[1], xp[0]);
                        multiply(small, wp[0], xp[1]);
                        multiply(small, wp[2], xp[0]);
                        multiply(small, wp[0], xp[2]);
                    }
                }
            });
    };
    reduce(std::false_type{});

    // sums that are not finite or too small, operands too large: the whole tile again on the fp32 instruction
    float sums[R], finite = 0.0f; // 0 * infinity and 0 * NaN are NaN, which is not equal to zero
#pragma unroll
    for (int r = 0; r < R; r++) {
        sums[r] = acc[r] + small[r];
        finite = fmaf(sums[r], 0.0f, finite);
    }
    if (__syncthreads_or(finite != 0.0f || split_small_sum(sums) || largest > kSplitLarge)) {
#pragma unroll
        for (int r = 0; r < R; r++)
            acc[r] = 0.0f;
        static_for_n<DEPTH>([&](auto slot_c) { load(slot_c, kt_begin + decltype(slot_c)::value); });
        reduce(std::true_type{});
#pragma unroll
        for (int r = 0; r < R; r++)
            sums[r] = acc[r];
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; r++)
        red[wave][r][lane] = sums[r];
    __syncthreads();
    if (!mine)
        return;
#pragma unroll
    for (int v = 0; v < V; v++) {
        const int r = wave * V + v;
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < KW; w++)
            sum += red[w][r][lane];
        sum += bias[v];
        if (pre)
            sum = fmaf(old[v], a.factor, sum);
        if (a.act == DLP_ACT_TANH || a.act == DLP_ACT_SIGMOID)
            sum = apply_act(sum, a.act);
        else if (a.act != DLP_ACT_IDENTITY) // identity must keep NaNs: no min/max
            sum = clamp_med3(sum, a.clamp_lo, a.clamp_hi);
        if (!pre && a.factor != 0.0f)
            sum = fmaf(old[v], a.factor, sum);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sum), yr, yoff[v], 0, 0);
    }
}
