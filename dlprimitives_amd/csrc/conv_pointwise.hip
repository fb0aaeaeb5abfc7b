// Pointwise (1x1, stride 1, no padding, one group) convolutions with at most 32 output channels over many pixels, fp32:
//   Y_b[M x HW] = act(W[M x K] * X_b[K x HW] + bias),  M = Cout <= 32, K = Cin a multiple of 16, H * W a multiple of 4,
//   at least 1024 tiles of 128 pixels (MobileNet's 144 -> 24 at 56 x 56 from batch 42 on).
//
// Replaces, for these shapes, the generic path of conv_gemm.hip (reference: the 1x1 fast path of sgemm.cl,
// src/kernels/sgemm.cl:78-93, under Conv2DForwardGEMM, src/core/conv.cpp:45-111).  Such a layer reads six times more than it
// writes and sits on the bandwidth leg of the roofline: what counts is that X is read once, in wide pieces, with many loads in flight.
//  * NCHW keeps the pixels of a channel contiguous, which is the operand layout of v_mfma_f32_32x32x2_f32: lane
//    (column n, half h) holds B[k = h][n].  A wavefront therefore loads X straight from memory into operand registers:
//    one 16-byte buffer load per pair of channels (lanes 0-31 channel 2p, lanes 32-63 channel 2p + 1) feeds four matrix
//    instructions, the MFMA block j taking pixel 4 n + j; eight pairs (8 KB) are in flight per wavefront.  No LDS traffic, no barrier
//    and no vector-ALU instruction for the big operand; the output leaves in 16-byte stores.
//  * The filter is small: it goes through LDS in chunks of 64 channels, transposed to [k][m] on the way in (an operand fetch is
//    then a conflict-free ds_read_b32), double buffered, one barrier per chunk; operands are read eight pairs at a time.
//  * The kernel is written for any split of a workgroup's four wavefronts into MS slices of the output channels times 4 / MS pixel
//    tiles, MTW blocks of 32 rows per wavefront and 1 or 4 pixels per lane.  Measured alone on cold tensors at batch 64, only the
//    shape above beats the LDS-tiled kernel (144->24 at 56x56: 30.7 against 33.7 us; 144->32 at 28x28 with one pixel per lane 14.0
//    against 12.4; 192->64 at 14x14 11.8 against 9.3; 64->64 at 56x56 with two blocks per wavefront 42.8 against 34.2): the small layers
//    are bound by the fixed 2 us each of prologue (first filter chunk) and epilogue, not by how X arrives.  Only that variant is built.
// The sum over k runs in channel order, two channels per matrix instruction, accumulated in fp32.
#include "dlp_internal.hpp"
// the output runs are whole cache lines that this launch does not read again: non-temporal stores (144->24 at 56x56, batch 64: 31.5 -> 28.9 us)
#ifndef PW_STORE_AUX
#define PW_STORE_AUX 2
#endif

#include <algorithm>
#include <type_traits>

namespace dlp {

typedef float pw_f32x16 __attribute__((ext_vector_type(16)));
typedef float pw_f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kPwThreads = 256;
constexpr int kPwChunk = 64;  // channels of a filter chunk in LDS
#ifndef DLP_PW_DEPTH1
#define DLP_PW_DEPTH1 32
#endif
#ifndef DLP_PW_DEPTH4
#define DLP_PW_DEPTH4 8
#endif
constexpr uint32_t kPwOutOfRange = 0x80000000u;

struct PwArgs {
    const float *x, *w, *bias;
    float *y;
    int M, K, HW, N;      // output channels, input channels, pixels per image, pixels in all (batch * HW)
    int mpad;             // rows of the LDS filter chunk: M rounded up to 32 * MS * MTW
    uint32_t x_bytes, y_bytes, w_bytes;
    uint32_t hw_magic, hw_shift;
    float factor;
    int pre;              // y = act(conv + bias + factor * y) (Epilogue::accumulate_first)
    int clamp;            // 0: identity
    float clamp_lo, clamp_hi;
};

template <int PX>
struct PwB {
    float v[PX];
};

template <int PX>
__device__ __forceinline__ PwB<PX> pw_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff)
{
    PwB<PX> b;
    if constexpr (PX == 4) {
        const pw_f32x4 t = __builtin_bit_cast(pw_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
        b.v[0] = t[0], b.v[1] = t[1], b.v[2] = t[2], b.v[3] = t[3];
    } else
        b.v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    return b;
}

// PX: pixels per lane (1, 4); MTW: 32-row blocks per wavefront; MS: slices of the output channels among the wavefronts
template <int PX, int MTW, int MS>
__global__ __launch_bounds__(kPwThreads) void conv_pointwise_f32_kernel(PwArgs a)
{
    static_assert(MS == 1 || MS == 2 || MS == 4, "wavefront split");
    constexpr int MPAD = 32 * MTW * MS;             // rows of the filter chunk
    constexpr int PT = 4 / MS;                       // pixel tiles per workgroup
    constexpr int TILE = 32 * PX;                    // pixels per pixel tile
    constexpr int A_F4 = MPAD * kPwChunk / 4;        // 16-byte pieces of a filter chunk
    constexpr int A_LD = (A_F4 + kPwThreads - 1) / kPwThreads;
    constexpr int kPwDepth = PX == 1 ? DLP_PW_DEPTH1 : DLP_PW_DEPTH4; // channel pairs in flight per wavefront
    __shared__ float As[2][kPwChunk][MPAD];
    __shared__ float bias_s[MPAD];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int ms = wave % MS, pt = wave / MS;
    const int n0 = ((int)blockIdx.x * PT + pt) * TILE + l32 * PX; // this lane's first pixel

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, 0, a.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)a.w, 0, a.w_bytes, 0x00020000);

    // ---- X: byte offset of (image, channel h, pixel) for this lane; a pair of channels further is 2 * HW * 4 bytes on ----
    const int b_img = (int)fast_div((uint32_t)n0, a.hw_magic, a.hw_shift);
    const int pix = n0 - b_img * a.HW;
    const uint32_t xvoff = n0 < a.N ? (uint32_t)(((b_img * a.K + h) * a.HW + pix) * 4) : kPwOutOfRange;
    const uint32_t pair_bytes = (uint32_t)(2 * a.HW * 4);
    const int npairs = a.K / 2;

    // ---- filter chunk loader: thread (m = t % MPAD, c4 = t / MPAD) takes W[m][c0 + 4 c4 .. + 3] and scatters the four values down
    //      a column of the [k][m] chunk (consecutive lanes, consecutive m: no bank conflicts) ----
    pw_f32x4 ra[A_LD];
    auto load_chunk = [&](int c0) {
#pragma unroll
        for (int q = 0; q < A_LD; q++) {
            const int t = tid + q * kPwThreads;
            const int m = t % MPAD, c = c0 + 4 * (t / MPAD);
            const bool ok = (A_F4 % kPwThreads == 0 || t < A_F4) && m < a.M && c < a.K;
            ra[q] = __builtin_bit_cast(pw_f32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, ok ? (uint32_t)((m * a.K + c) * 4) : kPwOutOfRange, 0, 0));
        }
    };
    auto store_chunk = [&](int buf) {
#pragma unroll
        for (int q = 0; q < A_LD; q++) {
            const int t = tid + q * kPwThreads;
            if (A_F4 % kPwThreads == 0 || t < A_F4) {
                const int m = t % MPAD, k4 = 4 * (t / MPAD);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    As[buf][k4 + e][m] = ra[q][e];
            }
        }
    };

    pw_f32x16 acc[MTW][PX];
#pragma unroll
    for (int i = 0; i < MTW; i++)
#pragma unroll
        for (int j = 0; j < PX; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                acc[i][j][r] = 0.0f;

    // ---- prologue: the first channel pairs of X and the first filter chunk ----
    PwB<PX> fb[kPwDepth];
#pragma unroll
    for (int d = 0; d < kPwDepth; d++)
        fb[d] = pw_load<PX>(xr, xvoff, (uint32_t)min(d, npairs - 1) * pair_bytes);
    load_chunk(0);
    if (tid < MPAD) // the bias waits in LDS for the epilogue: a global load per output row there would cost its latency sixteen times
        bias_s[tid] = (a.bias && tid < a.M) ? a.bias[tid] : 0.0f;
    store_chunk(0);
    __syncthreads();

    const int nchunks = (a.K + kPwChunk - 1) / kPwChunk;
    for (int ch = 0; ch < nchunks; ch++) {
        const int buf = ch & 1;
        const int c0 = ch * kPwChunk;
        const int pairs = min(kPwChunk, a.K - c0) / 2; // a multiple of 8: K is a multiple of 16
        if (ch + 1 < nchunks)
            load_chunk(c0 + kPwChunk);
        // The filter operands are read from LDS eight pairs at a time: a ds_read right in front of its matrix instruction exposes the LDS
        // latency in every step (measured: 170 to 210 instead of 64 clocks per step), eight in flight expose it once per eight steps.
        constexpr int G = 8;
        float fa[G][MTW];
        for (int p0 = 0; p0 < pairs; p0 += kPwDepth) {
#pragma unroll
            for (int d = 0; d < kPwDepth; d++) {
                const int p = p0 + d;           // pair inside the chunk: channels c0 + 2 p, c0 + 2 p + 1
                if (d % G == 0) {
                    if (p >= pairs)             // uniform: only the last chunk of a K that is no multiple of 2 * kPwDepth stops early (pairs % 8 == 0)
                        break;
#pragma unroll
                    for (int e = 0; e < G; e++)
#pragma unroll
                        for (int i = 0; i < MTW; i++)
                            fa[e][i] = As[buf][2 * (p + e) + h][(ms * MTW + i) * 32 + l32];
                }
                const int gp = c0 / 2 + p;      // pair of the tensor
                const PwB<PX> cur = fb[d];
                // the pair kPwDepth further on takes this register (pairs past the end re-read the last one and are never multiplied)
                fb[d] = pw_load<PX>(xr, xvoff, (uint32_t)min(gp + kPwDepth, npairs - 1) * pair_bytes);
#pragma unroll
                for (int i = 0; i < MTW; i++)
#pragma unroll
                    for (int j = 0; j < PX; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[d % G][i], cur.v[j], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0); // keep every load where it is: right behind the use of its register, kPwDepth pairs ahead of its own
            }
        }
        if (ch + 1 < nchunks) {
            store_chunk(buf ^ 1); // nobody reads that buffer: its chunk was finished before the previous barrier
            __syncthreads();
        }
    }

    // ---- epilogue: accumulator register r of block (i, j) is row 32 * (ms * MTW + i) + 8 * (r / 4) + 4 * h + r % 4, pixel n0 + j ----
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);
    const bool use_old = a.factor != 0.0f;
    const bool pre = a.pre != 0 && use_old;
    const uint32_t yvoff = n0 < a.N ? (uint32_t)((b_img * a.M * a.HW + pix) * 4) : kPwOutOfRange;
#pragma unroll
    for (int i = 0; i < MTW; i++) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = (ms * MTW + i) * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (m >= a.M)
                continue;
            const float bias = bias_s[m];
            const uint32_t voff = yvoff == kPwOutOfRange ? kPwOutOfRange : yvoff + (uint32_t)(m * a.HW * 4);
            PwB<PX> old;
            if (use_old)
                old = pw_load<PX>(yr, voff, 0);
            float v[PX];
#pragma unroll
            for (int j = 0; j < PX; j++) {
                v[j] = acc[i][j][r] + bias;
                if (pre)
                    v[j] = fmaf(old.v[j], a.factor, v[j]);
                const float c = clamp_med3(v[j], a.clamp_lo, a.clamp_hi);
                v[j] = a.clamp ? c : v[j]; // identity keeps NaNs: no clamp
                if (use_old && !pre)
                    v[j] = fmaf(old.v[j], a.factor, v[j]);
            }
            if constexpr (PX == 4)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) uint32_t, (pw_f32x4){v[0], v[1], v[2], v[3]}), yr,
                                                       voff, 0, PW_STORE_AUX);
            else
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v[0]), yr, voff, 0, 0);
        }
    }
}

// ---- the other way round: few input channels, many filters (the expansion of an inverted residual block, 24 -> 144 at 56x56), fp32 ----
// Such a layer writes six times what it reads.  In 32x128 tiles of the gathering kernel every workgroup gathered its 24 channels pixel by pixel for
// 16 KB of output, five workgroups the same ones.  Here a wavefront keeps four pixels per lane of all K channels in registers (16-byte loads, one
// pair of channels each, as above) and walks RB blocks of 32 filters over them; a filter block's weights lie in LDS as [k][m].  Stores are 16
// bytes a lane, 512 consecutive bytes a row, and stay in the caches for the next layer to read.  24 -> 144 at 56x56, batch 64 (135 MB): 56 -> 37 us.
// (The offset of a store is all in its vector register: with a scalar one besides, the compiler lets the next instruction overwrite the
// first of the four data registers of a 16-byte store, and lanes 12 to 15 of every 16 stored what came after.)
template <int KP>
__global__ __launch_bounds__(kPwThreads) void conv_expand_f32_kernel(PwArgs a, int rb)
{
    constexpr int PX = 4;
    extern __shared__ __attribute__((aligned(16))) float ex_lds[]; // [2 * KP][32 * rb] weights, [32 * rb] bias
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int n0 = ((int)blockIdx.x * 4 + wave) * (32 * PX) + l32 * PX; // this lane's first pixel
    const int rows = 32 * rb, m0 = (int)blockIdx.y * rows;
    float *const bias_s = ex_lds + 2 * KP * rows;

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, 0, a.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);
    const int b_img = (int)fast_div((uint32_t)n0, a.hw_magic, a.hw_shift);
    const int pix = n0 - b_img * a.HW; // PX divides the plane: the lane's pixels stay in one image
    const uint32_t xvoff = n0 < a.N ? (uint32_t)(((b_img * a.K + h) * a.HW + pix) * 4) : kPwOutOfRange;
    const uint32_t pair_bytes = (uint32_t)(2 * a.HW * 4);
    float x[KP][PX];
#pragma unroll
    for (int p = 0; p < KP; p++) {
        const uint32_t v = 2 * p + h < a.K ? xvoff : kPwOutOfRange;
        const pw_f32x4 t = __builtin_bit_cast(pw_f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, v, (uint32_t)p * pair_bytes, 0));
#pragma unroll
        for (int j = 0; j < PX; j++)
            x[p][j] = t[j];
    }
    for (int i = tid; i < rows * 2 * KP; i += kPwThreads) { // a filter's channels by consecutive lanes
        const int m = i / (2 * KP), k = i % (2 * KP);
        ex_lds[k * rows + m] = m0 + m < a.M && k < a.K ? a.w[(m0 + m) * a.K + k] : 0.0f;
    }
    for (int i = tid; i < rows; i += kPwThreads)
        bias_s[i] = a.bias && m0 + i < a.M ? a.bias[m0 + i] : 0.0f;
    __syncthreads();

    const uint32_t yvoff = n0 < a.N ? (uint32_t)(((b_img * a.M + m0 + 4 * h) * a.HW + pix) * 4) : kPwOutOfRange;
    const int pairs = (a.K + 1) / 2;
    for (int i = 0; i < rb; i++) {
        if (m0 + 32 * i >= a.M)
            break;
        pw_f32x16 acc[PX];
#pragma unroll
        for (int j = 0; j < PX; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                acc[j][r] = 0.0f;
        const float *const wl = ex_lds + h * rows + 32 * i + l32;
#pragma unroll
        for (int p0 = 0; p0 < KP; p0 += 4) {
            if (p0 >= pairs)
                break;
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                f[e] = wl[2 * (p0 + e) * rows];
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int j = 0; j < PX; j++)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[e], x[p0 + e][j], acc[j], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = 32 * i + 8 * (r >> 2) + (r & 3); // + 4 * h
            const float bias = bias_s[row + 4 * h];
            const uint32_t voff = yvoff != kPwOutOfRange && m0 + row + 4 * h < a.M ? yvoff + (uint32_t)(row * a.HW * 4) : kPwOutOfRange;
            float v[PX];
#pragma unroll
            for (int j = 0; j < PX; j++) {
                v[j] = acc[j][r] + bias;
                const float c = clamp_med3(v[j], a.clamp_lo, a.clamp_hi);
                v[j] = a.clamp ? c : v[j]; // identity keeps NaNs: no clamp
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) uint32_t, (pw_f32x4){v[0], v[1], v[2], v[3]}), yr, voff,
                                                   0, 0);
        }
    }
}

struct PwShape {
    int px, mtw, ms;
};

// How the wavefronts are cut for a layer: enough wavefront tasks for the chip (about one per SIMD), wide loads when there are
// pixels to spare.
PwShape pw_shape(const ConvGeom &g)
{
    const long long N = (long long)g.B * g.H * g.W;
    const int mblocks = (g.Cout + 31) / 32;
    PwShape s;
    s.px = ((g.H * g.W) % 4 == 0 && N / 128 >= 1024) ? 4 : 1;
    if (mblocks == 1) {
        s.ms = 1;
        s.mtw = 1;
    } else if (N / (32 * s.px) * 1 >= 1536) { // many pixel tiles: every wavefront takes all rows of its own
        s.ms = 1;
        s.mtw = mblocks;
    } else { // few pixel tiles: the wavefronts share one and split the rows
        s.ms = mblocks <= 2 ? 2 : 4;
        s.mtw = 1;
    }
    return s;
}

} // namespace

bool conv_pointwise_supported(const ConvGeom &g, int activation)
{
    if (g.dtype != DLP_FLOAT || g.KH != 1 || g.KW != 1 || g.sh != 1 || g.sw != 1 || g.ph != 0 || g.pw != 0 || g.groups != 1)
        return false;
    if (activation == DLP_ACT_TANH || activation == DLP_ACT_SIGMOID)
        return false;
    if (g.Cin % 16 != 0 || g.Cout > 128)
        return false;
    const PwShape s = pw_shape(g);
    return s.px == 4 && s.mtw == 1 && s.ms == 1;
}

int conv_pointwise_launch(const ConvGeom &g, const void *x, const void *w, void *y, const Epilogue &ep, hipStream_t stream)
{
    DLP_REQUIRE(conv_pointwise_supported(g, ep.activation), "geometry is not served by the pointwise kernel");
    DLP_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) == 0, "pointwise kernel: tensors must be 16-byte aligned");
    if (g.B == 0)
        return DLP_OK;
    const size_t HW = (size_t)g.H * g.W;
    const size_t x_bytes = (size_t)g.B * g.Cin * HW * 4, y_bytes = (size_t)g.B * g.Cout * HW * 4;
    if (x_bytes >= kPwOutOfRange || y_bytes >= kPwOutOfRange)
        return fail(DLP_ERR_NOT_IMPLEMENTED, "tensors of 2 GiB or more are not supported by the 32-bit buffer addressing");
    const PwShape s = pw_shape(g);
    PwArgs a;
    a.x = (const float *)x;
    a.w = (const float *)w;
    a.bias = ep.bias;
    a.y = (float *)y;
    a.M = g.Cout;
    a.K = g.Cin;
    a.HW = (int)HW;
    a.N = (int)(g.B * HW);
    a.mpad = 32 * s.mtw * s.ms;
    a.x_bytes = (uint32_t)x_bytes;
    a.y_bytes = (uint32_t)y_bytes;
    a.w_bytes = (uint32_t)((size_t)g.Cout * g.Cin * 4);
    make_magic((uint32_t)HW, a.hw_magic, a.hw_shift);
    a.factor = ep.factor;
    a.pre = ep.accumulate_first;
    a.clamp = ep.activation != DLP_ACT_IDENTITY;
    a.clamp_lo = 0.0f;
    a.clamp_hi = ep.activation == DLP_ACT_RELU6 ? 6.0f : __builtin_huge_valf();
    const int per_wg = 32 * s.px * (4 / s.ms); // pixels per workgroup
    const dim3 grid((unsigned)((a.N + per_wg - 1) / per_wg)), block(kPwThreads);
    TimingScope ts("conv_gemm", stream);
#define DLP_PW_CASE(PX, MTW, MS)                                                                                         \
    if (s.px == PX && s.mtw == MTW && s.ms == MS) {                                                                      \
        DLP_LAUNCH_TIMED(ts, (conv_pointwise_f32_kernel<PX, MTW, MS>), grid, block, 0, stream, a);                       \
        DLP_HIP_TRY(hipGetLastError());                                                                                  \
        return DLP_OK;                                                                                                   \
    }
    DLP_PW_CASE(4, 1, 1)
#undef DLP_PW_CASE
    return fail(DLP_ERR_RUNTIME, "pointwise kernel: no instantiation for this shape");
}

bool conv_expand_geometry(const ConvGeom &g)
{
    return g.dtype == DLP_FLOAT && g.KH == 1 && g.KW == 1 && g.sh == 1 && g.sw == 1 && g.ph == 0 && g.pw == 0 && g.groups == 1 && g.Cin <= 24 && g.Cout > 32 &&
           (g.H * g.W) % 4 == 0;
}

bool conv_expand_serves(const ConvGeom &g, const Epilogue &ep, const void *x, const void *y)
{
    if (!conv_expand_geometry(g) || g.B <= 0 || ep.activation == DLP_ACT_TANH || ep.activation == DLP_ACT_SIGMOID || ep.factor != 0.0f)
        return false;
    if ((((uintptr_t)x | (uintptr_t)y) & 15) != 0)
        return false;
    const size_t N = (size_t)g.B * g.H * g.W;
    // From some size of the output on; below, a wavefront that walks many filter blocks takes longer than the other kernels' many workgroups, and how much
    // longer goes with how their tiles suit the filters.  us, others / this, filters packed:
    //  * 40 MB: filters off multiples of 8, which the others store element by element (8 -> 142 at 38x38, batch 80, 66 MB 32 / 18; 24 -> 162 at 54x54,
    //    batch 51, 96 MB 54 / 36); up to 8 channels into up to 128 filters (8 -> 48 at 42x42, batch 128, 43 MB 16 / 15; 8 -> 128 at 86x86, 33, 125 MB
    //    29 / 26; but 8 -> 256 at 42x42, 75, 135 MB 31 / 34); filters that leave a last tile of 64 at least half empty (17 -> 144 at 38x38, 79, 66 MB 28 / 24, 24 -> 144 at
    //    106x106, 15, 97 MB 39 / 35, 24 -> 144 at 56x56, batch 64, 116 MB 56 / 37);
    //  * 190 MB: the rest (24 -> 128 at 68x68, 28, 66 MB 22 / 28, 16 -> 64 at 112x112, 42, 135 MB 31 / 37, 20 -> 128 at 68x68, 61, 144 MB 42 / 43; 24 -> 64 at
    //    106x106, 69, 198 MB 77 / 59, 20 -> 256 at 60x60, 60, 221 MB 59 / 52).
    // More than 24 channels were tried with two pixels a lane only: 40 -> 240 at 56x56, batch 24 38 / 41, 64 -> 256 at batch 64 89 / 118.  (24 channels take 100
    // registers with four pixels, 32 would take some 16 more.)
    const int rest = g.Cout % 64;
    const size_t from = g.Cout % 8 != 0 || (g.Cin <= 8 && g.Cout <= 128) || (rest != 0 && rest <= 32) ? 40000000 : 190000000;
    return N * g.Cin * 4 < kPwOutOfRange && N * g.Cout * 4 < kPwOutOfRange && N * g.Cout * 4 >= from;
}

int conv_expand_launch(const ConvGeom &g, const void *x, const void *w, void *y, const Epilogue &ep, hipStream_t stream)
{
    PwArgs a = PwArgs();
    a.x = (const float *)x;
    a.w = (const float *)w;
    a.bias = ep.bias;
    a.y = (float *)y;
    a.M = g.Cout;
    a.K = g.Cin;
    a.HW = g.H * g.W;
    a.N = g.B * a.HW;
    a.x_bytes = (uint32_t)((size_t)a.N * a.K * 4);
    a.y_bytes = (uint32_t)((size_t)a.N * a.M * 4);
    make_magic((uint32_t)a.HW, a.hw_magic, a.hw_shift);
    a.clamp = ep.activation != DLP_ACT_IDENTITY;
    a.clamp_lo = 0.0f;
    a.clamp_hi = ep.activation == DLP_ACT_RELU6 ? 6.0f : __builtin_huge_valf();
    const int kp = a.K <= 16 ? 8 : 12, blocks = (a.M + 31) / 32;
    // filter blocks per wavefront: one to six, as many as leave nearly two workgroups per compute unit (24 -> 144 above: 1, 2, 3, 4, 5 blocks 48, 43, 40, 37, 36 us, the
    // same tensors again 45, 39, 36, 33, 35; 24 -> 96 at batch 48: 1, 2, 3 blocks 25, 23, 24)
    const long long gx = (a.N + 511) / 512, two = 2 * dlp_cu_count();
    const int rb = (int)std::max<long long>(1, std::min<long long>(std::min(blocks, 6), (gx * blocks + two - 1) / two));
    const dim3 grid((unsigned)gx, (unsigned)((blocks + rb - 1) / rb));
    const size_t lds = (size_t)(2 * kp + 1) * 32 * rb * sizeof(float);
    void (*kernel)(PwArgs, int) = conv_expand_f32_kernel<12>;
    if (kp == 8)
        kernel = conv_expand_f32_kernel<8>;
    TimingScope ts("conv_gemm", stream);
    DLP_LAUNCH_TIMED(ts, kernel, grid, dim3(kPwThreads), lds, stream, a, rb);
    DLP_HIP_TRY(hipGetLastError());
    return DLP_OK;
}

} // namespace dlp
