// ONNX ConvInteger (ConvIntegerKernels.Encode, ConvIntegerKernels.cs:97-253): the kernels of its own besides the int8
// product.
//
// Pack (ConvIntegerPack.hlsl): the windows of every image and group unfold into a byte matrix of K = CinG * KH * KW
// rows and OH * OW columns (Chellapilla, Puri and Simard, 2006), row (c * KH + kh) * KW + kw, column oh * OW + ow
// holding x[n, g * CinG + c, oh * SH - PH + kh * DH, ow * SW - PW + kw * DW], or x's zero point where that position lies
// in the padding (so a padded tap adds nothing once the product subtracts the zero point). Rows are padded to a multiple
// of 16 bytes (ldb) so that the MFMA product can feed them to LDS with 16-byte DMA; the padding columns hold the zero
// point too and the product never reads them. One thread writes 16 bytes of one row.
//
// Padded depth: when K is at least 64 and not a multiple of 64, the launcher pads it to one (kp) so that the products
// take the LDS-DMA kernel. Rows k .. kp - 1 of every column matrix hold x's zero point, so each padded tap adds
// (w - wz) (xz - xz) = 0, and the same launch copies the weights into rows of kp bytes, zero past k; the 16-byte
// chunks of both go through one grid-stride loop (the column chunks first).
//
// Depthwise (one input channel a group): no matrix at all. The usual windows over enough outputs go by tiles through LDS
// (k_conv_depthwise_tile); any other convolution has a thread per output element, which sums its KH * KW taps,
// (x - xz) * (w - wz[m]) in 32-bit wrap-around, skipping taps in the padding (they are the real value zero).
#include "og_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace og {

namespace {

constexpr int kConvThreads = 256;

__device__ __forceinline__ int32_t byte_val(uint8_t b, bool is_signed) { return is_signed ? (int32_t)(int8_t)b : (int32_t)b; }

template <bool ALIGNED16>
__global__ __launch_bounds__(kConvThreads) void k_conv_pack(ConvPackArgs a)
{
    const int64_t chunks_per_row = a.ldb / 16;
    const int64_t rows = (int64_t)a.images * a.groups * a.kp;
    const int64_t total = rows * chunks_per_row, wchunks = a.kp / 16, wtotal = (int64_t)a.wrows * wchunks;
    const int32_t taps = a.kh * a.kw;
    const uint32_t pad = a.xz ? (uint32_t)*a.xz : 0u;
    const int32_t ncols = a.oh * a.ow;
    for (int64_t t = (int64_t)blockIdx.x * kConvThreads + threadIdx.x; t < total + wtotal;
         t += (int64_t)gridDim.x * kConvThreads) {
        if (t >= total) {
            // Weight chunk: row m, bytes 16 c .. + 15 of the padded copy.
            const int64_t tw = t - total, m = tw / wchunks;
            const int32_t c0 = 16 * (int32_t)(tw - m * wchunks);
            uint32_t word[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                uint32_t wv = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int32_t kk = c0 + 4 * q + e;
                    wv |= (kk < a.k ? (uint32_t)a.wt[m * a.k + kk] : 0u) << (8 * e);
                }
                word[q] = wv;
            }
            *reinterpret_cast<uint4 *>(a.wp + m * a.kp + c0) = make_uint4(word[0], word[1], word[2], word[3]);
            continue;
        }
        const int64_t r = t / chunks_per_row;
        const int32_t c16 = (int32_t)(t - r * chunks_per_row);
        const int64_t ig = r / a.kp;
        const int32_t k = (int32_t)(r - ig * a.kp);
        uint8_t *dst = a.cols + r * a.ldb + 16 * (int64_t)c16;
        if (k >= a.k) {   // a padding row
            const uint32_t pw4 = pad * 0x01010101u;
            if constexpr (ALIGNED16) {
                *reinterpret_cast<uint4 *>(dst) = make_uint4(pw4, pw4, pw4, pw4);
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) reinterpret_cast<uint32_t *>(dst)[q] = pw4;
            }
            continue;
        }
        const int64_t img = ig / a.groups;
        const int32_t g = (int32_t)(ig - img * a.groups);
        const int32_t c = k / taps, kk = k - c * taps, kh = kk / a.kw, kw = kk - kh * a.kw;
        const uint8_t *plane = a.x + (img * a.cin + (int64_t)g * a.cin_g + c) * (int64_t)a.h * a.w;
        // Column n = 16 * c16 + e; its (oh, ow) advance one column at a time.
        int32_t n = 16 * c16, row_o = n / a.ow, col_o = n - row_o * a.ow;
        uint32_t word[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            uint32_t wv = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                uint32_t v = pad;
                if (n < ncols) {
                    const int64_t ih = (int64_t)row_o * a.sh + (int64_t)kh * a.dh - a.ph;
                    const int64_t iw = (int64_t)col_o * a.sw + (int64_t)kw * a.dw - a.pw;
                    if (ih >= 0 && ih < a.h && iw >= 0 && iw < a.w) v = plane[ih * a.w + iw];
                }
                wv |= v << (8 * e);
                n++;
                if (++col_o == a.ow) {
                    col_o = 0;
                    row_o++;
                }
            }
            word[q] = wv;
        }
        if constexpr (ALIGNED16) {
            *reinterpret_cast<uint4 *>(dst) = make_uint4(word[0], word[1], word[2], word[3]);
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) reinterpret_cast<uint32_t *>(dst)[q] = word[q];
        }
    }
}

// K3: the window is 3 x 3 (known at compile time), so the nine taps' loads are all issued before the first is used
// (a tap in the padding loads the plane's first byte and adds nothing); otherwise a loop over the window.
template <bool XS, bool WS, bool K3>
__global__ __launch_bounds__(kConvThreads) void k_conv_depthwise(ConvDepthwiseArgs a)
{
    const int64_t plane = (int64_t)a.oh * a.ow;
    const int64_t total = (int64_t)a.batch * a.cout * plane;
    const int32_t cout_g = a.cout / a.cin;   // output channels of one input channel
    const int32_t xz = a.xz ? byte_val(*a.xz, XS) : 0;
    for (int64_t t = (int64_t)blockIdx.x * kConvThreads + threadIdx.x; t < total; t += (int64_t)gridDim.x * kConvThreads) {
        const int64_t nm = t / plane;
        const int32_t p = (int32_t)(t - nm * plane);
        const int64_t n = nm / a.cout;
        const int32_t m = (int32_t)(nm - n * a.cout);
        const int32_t i = p / a.ow, j = p - (p / a.ow) * a.ow;
        const uint8_t *xp = a.x + (n * a.cin + m / cout_g) * (int64_t)a.h * a.w;
        const uint8_t *wp = a.wt + (int64_t)m * a.kh * a.kw;
        const int32_t wz = a.wz ? byte_val(a.wz[a.wz_per_channel ? m : 0], WS) : 0;
        uint32_t acc = 0;
        if constexpr (K3) {
            int64_t off[9];
            bool in[9];
#pragma unroll
            for (int q = 0; q < 9; q++) {
                const int64_t ih = (int64_t)i * a.sh + (int64_t)(q / 3) * a.dh - a.ph;
                const int64_t iw = (int64_t)j * a.sw + (int64_t)(q % 3) * a.dw - a.pw;
                in[q] = ih >= 0 && ih < a.h && iw >= 0 && iw < a.w;
                off[q] = in[q] ? ih * a.w + iw : 0;
            }
            uint8_t xv[9], wv[9];
#pragma unroll
            for (int q = 0; q < 9; q++) {
                xv[q] = xp[off[q]];
                wv[q] = wp[q];
            }
#pragma unroll
            for (int q = 0; q < 9; q++)
                if (in[q]) acc += (uint32_t)(byte_val(xv[q], XS) - xz) * (uint32_t)(byte_val(wv[q], WS) - wz);
            a.y[t] = (int32_t)acc;
            continue;
        }
        for (int32_t kh = 0; kh < a.kh; kh++) {
            const int64_t ih = (int64_t)i * a.sh + (int64_t)kh * a.dh - a.ph;
            if (ih < 0 || ih >= a.h) continue;
            for (int32_t kw = 0; kw < a.kw; kw++) {
                const int64_t iw = (int64_t)j * a.sw + (int64_t)kw * a.dw - a.pw;
                if (iw < 0 || iw >= a.w) continue;
                const int32_t xv = byte_val(xp[ih * a.w + iw], XS) - xz;
                const int32_t wv = byte_val(wp[kh * a.kw + kw], WS) - wz;
                acc += (uint32_t)xv * (uint32_t)wv;
            }
        }
        a.y[t] = (int32_t)acc;
    }
}

// The windows most depthwise layers have (KH x KW of 3 x 3, 5 x 5, 1 x 3 or 1 x 5, both strides S = 1 or 2, undilated), a
// tile of output positions a workgroup. A thread per output position (k_conv_depthwise) is bound by its byte loads, two a
// tap; here the workgroup stages the input its tile reaches once into LDS, the padding written out as x's zero point, and a
// thread forms four neighbouring outputs in each of R rows: of every input row it reads the two or three words that hold
// its windows, shifts out four bytes for each output, and multiplies them with a row of taps by one four-way dot product
// (a fifth tap takes a second one). Both operands are flipped to signed bytes first (x ^ 0x80 = x - 128), which their zero
// points follow, and then
//   sum (x - xz)(w - wz) = sum x w - wz sum x - xz sum w + KH KW xz wz,
// whole numbers that wrap in 32 bits like the sum itself. The sum of x is formed only where wz is not zero.
// A tile is `c` planes (whole ones, or a part of one) of `trg` groups of R rows of `tcq` quads of columns.
// Bound by memory at the large end: 8 x 512 channels of 112 x 112, 5 x 5, 770 -> 92 us (205 MB of results and 51 MB of input
// are 50 us at the rate of a large copy), 3 x 3 299 -> 66, with strides of 2 90 -> 36; 2 x 64 of 223 x 223, 5 x 5 by 2, 34.0 -> 8.7;
// one dimension, 8 x 512 of 2999, 5 taps, 69.6 -> 26.9. Small ones are bound by the launch and by staging (depthwise_by_output).
struct DepthwiseTile {
    int32_t tcq, trg, c, coltiles, rowtiles, rows_in, stride, planes, cout_g;   // stride: words of a staged row
    uint32_t magic_stride, magic_rows;                                          // as ConvView's
};

template <int KH, int KW, int S, int R>
__global__ __launch_bounds__(kConvThreads) void k_conv_depthwise_tile(ConvDepthwiseArgs a, DepthwiseTile t)
{
    constexpr int ROWS = (R - 1) * S + KH, WORDS = S == 1 ? 2 : 3;
    extern __shared__ uint32_t tile[];
    typedef int32_t i4u __attribute__((ext_vector_type(4), aligned(4)));
    const uint32_t ct = blockIdx.x % (uint32_t)t.coltiles, rest = blockIdx.x / (uint32_t)t.coltiles;
    const uint32_t rt = rest % (uint32_t)t.rowtiles;
    const int32_t plane0 = (int32_t)(rest / (uint32_t)t.rowtiles) * t.c;
    const int32_t i0 = (int32_t)rt * t.trg * R, j0 = (int32_t)ct * t.tcq * 4;
    const int32_t ih0 = i0 * S - a.ph, iw0 = j0 * S - a.pw;
    const uint32_t flip_x = a.x_signed ? 0u : 0x80808080u, flip_w = a.w_signed ? 0u : 0x80808080u;
    const uint32_t xz_raw = a.xz ? *a.xz : 0u;
    // The taps, requested before the input: wv[kh] the first four of a row (three: the fourth zero), w5[kh] the fifth. Threads
    // without an output take a plane that is there.
    const uint32_t quads = (uint32_t)t.tcq, cq = threadIdx.x % quads, g = threadIdx.x / quads;
    const uint32_t rg = g % (uint32_t)t.trg, c = g / (uint32_t)t.trg;
    const int32_t plane = plane0 + (int32_t)c, i = i0 + (int32_t)rg * R, j = j0 + 4 * (int32_t)cq;
    const int32_t m = min(plane, t.planes - 1) % a.cout;
    const uint8_t *const wp = a.wt + (int64_t)m * (KH * KW);
    const uint32_t wz_raw = a.wz ? a.wz[a.wz_per_channel ? m : 0] : 0u;
    uint8_t wb[KH * KW];
#pragma unroll
    for (int q = 0; q < KH * KW; q++) wb[q] = wp[q];

    // Every load is made, from a row and a word that are there, so that four are in flight; what lies in the padding is
    // shifted or swapped out afterwards. Rows shorter than a word go byte by byte.
    const uint32_t staged = (uint32_t)(t.c * t.rows_in * t.stride), pad = xz_raw * 0x01010101u;
    const auto place = [&](uint32_t at, int32_t &iw, bool &in) {
        const uint32_t row = __umulhi(at, t.magic_stride), q = at - row * (uint32_t)t.stride;
        const uint32_t cc = t.rows_in == 1 ? row : __umulhi(row, t.magic_rows);
        const int32_t ih = ih0 + (int32_t)(row - cc * (uint32_t)t.rows_in), from = plane0 + (int32_t)cc;
        iw = iw0 + 4 * (int32_t)q;
        in = at < staged && from < t.planes && ih >= 0 && ih < a.h;
        // Output plane n cout + m reads input plane n cin + m / cout_g.
        return a.x + (in ? ((int64_t)(from / t.cout_g) * a.h + ih) * (int64_t)a.w : 0);
    };
    if (a.w >= 4) {
        for (uint32_t first = threadIdx.x; first < staged; first += 4 * blockDim.x) {
            uint32_t word[4];
            int32_t shift[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                int32_t iw;
                bool in;
                const uint8_t *const src = place(first + u * blockDim.x, iw, in);
                const int32_t from = min(max(iw, 0), a.w - 4);
                shift[u] = in ? iw - from : 4;
                __builtin_memcpy(&word[u], src + from, 4);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t v = shift[u] >= 0 ? __builtin_amdgcn_alignbyte(pad, word[u], shift[u])
                                                 : __builtin_amdgcn_alignbyte(word[u], pad, 4 + shift[u]);
                if (first + u * blockDim.x < staged) tile[first + u * blockDim.x] = (shift[u] > -4 && shift[u] < 4 ? v : pad) ^ flip_x;
            }
        }
    } else {
        for (uint32_t at = threadIdx.x; at < staged; at += blockDim.x) {
            int32_t iw;
            bool in;
            const uint8_t *const src = place(at, iw, in);
            uint32_t word = pad;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (in && iw + e >= 0 && iw + e < a.w) word = (word & ~(0xFFu << (8 * e))) | ((uint32_t)src[iw + e] << (8 * e));
            tile[at] = word ^ flip_x;
        }
    }
    __syncthreads();
    if (c >= (uint32_t)t.c || plane >= t.planes || i >= a.oh || j >= a.ow) return;

    const int32_t wz = byte_val((uint8_t)wz_raw, a.w_signed) - (a.w_signed ? 0 : 128);
    const int32_t xz = byte_val((uint8_t)xz_raw, a.x_signed) - (a.x_signed ? 0 : 128);
    constexpr uint32_t ONES = KW == 3 ? 0x010101u : 0x01010101u, TAPS = KW == 3 ? 0xFFFFFFu : 0xFFFFFFFFu;
    uint32_t wv[KH], w5[KH];
    int32_t sum_w = 0;
#pragma unroll
    for (int kh = 0; kh < KH; kh++) {
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < (KW < 4 ? KW : 4); e++) v |= (uint32_t)wb[kh * KW + e] << (8 * e);
        wv[kh] = (v ^ flip_w) & TAPS;
        w5[kh] = KW == 5 ? ((uint32_t)wb[kh * KW + KW - 1] ^ flip_w) & 0xFFu : 0u;
        sum_w = __builtin_amdgcn_sdot4((int)wv[kh], (int)ONES, sum_w, false);
        if constexpr (KW == 5) sum_w += (int32_t)(int8_t)w5[kh];
    }
    const uint32_t offset = (uint32_t)(KH * KW) * (uint32_t)xz * (uint32_t)wz - (uint32_t)xz * (uint32_t)sum_w;
    const uint32_t *const src = tile + ((int32_t)c * t.rows_in + (int32_t)rg * (R * S)) * t.stride + (int32_t)cq * S;
    int32_t acc[R][4] = {}, sum_x[R][4] = {};
    const auto rows = [&](auto with_sum) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            uint32_t d[WORDS];
#pragma unroll
            for (int q = 0; q < WORDS; q++) d[q] = src[r * t.stride + q];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                // Output e's window starts at byte S e; its fifth byte is byte S e + 4.
                const int lo = S * e / 4, sh = S * e % 4;
                const uint32_t x4 = sh == 0 ? d[lo] : __builtin_amdgcn_alignbyte(d[lo + 1], d[lo], sh);
                int32_t part = 0;
                if constexpr (with_sum.value) {
                    part = __builtin_amdgcn_sdot4((int)x4, (int)ONES, 0, false);
                    if constexpr (KW == 5) part = __builtin_amdgcn_sdot4((int)d[lo + 1], 1 << (8 * sh), part, false);
                }
#pragma unroll
                for (int o = 0; o < R; o++) {
                    const int kh = r - o * S;
                    if (kh < 0 || kh >= KH) continue;
                    acc[o][e] = __builtin_amdgcn_sdot4((int)x4, (int)wv[kh], acc[o][e], false);
                    if constexpr (KW == 5) acc[o][e] = __builtin_amdgcn_sdot4((int)d[lo + 1], (int)(w5[kh] << (8 * sh)), acc[o][e], false);
                    if constexpr (with_sum.value) sum_x[o][e] += part;
                }
            }
        }
    };
    if (wz != 0) rows(std::true_type{});
    else rows(std::false_type{});
    int32_t *const y = a.y + ((int64_t)plane * a.oh + i) * (int64_t)a.ow + j;
#pragma unroll
    for (int o = 0; o < R; o++) {
        if (i + o >= a.oh) break;
        i4u v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = (int32_t)((uint32_t)acc[o][e] + offset - (uint32_t)wz * (uint32_t)sum_x[o][e]);
        int32_t *const dst = y + (int64_t)o * a.ow;
        if (j + 4 <= a.ow) {
            *reinterpret_cast<i4u *>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (j + e < a.ow) dst[e] = v[e];
        }
    }
}

template <int KH, int KW, int S, int R>
hipError_t launch_depthwise_tile(const ConvDepthwiseArgs &a, hipStream_t s)
{
    const auto ceil_div = [](int64_t x, int64_t d) { return (x + d - 1) / d; };
    DepthwiseTile t{};
    t.planes = a.batch * a.cout;   // at most the results' number, below 2^31
    t.cout_g = a.cout / a.cin;
    const int64_t quads = ceil_div(a.ow, 4), groups = ceil_div(a.oh, R);
    t.coltiles = (int32_t)ceil_div(quads, kConvThreads);
    t.tcq = (int32_t)ceil_div(quads, t.coltiles);
    t.rowtiles = (int32_t)ceil_div(groups, std::min<int64_t>(groups, kConvThreads / t.tcq));
    // A chip of 256 CUs first: smaller tiles while there are fewer of them than that, then more planes in a tile.
    while ((int64_t)t.coltiles * t.rowtiles * t.planes < 256 && t.rowtiles < groups) t.rowtiles = (int32_t)std::min<int64_t>(groups, 2 * t.rowtiles);
    t.trg = (int32_t)ceil_div(groups, t.rowtiles);
    t.rowtiles = (int32_t)ceil_div(groups, t.trg);
    t.c = 1;
    if (t.coltiles == 1 && t.rowtiles == 1)
        t.c = (int32_t)std::max<int64_t>(1, std::min<int64_t>(kConvThreads / (t.tcq * t.trg), t.planes / 256));
    t.rows_in = (t.trg * R - 1) * S + KH;
    t.stride = t.tcq * S + 1;
    t.magic_stride = (uint32_t)((1ull << 32) / (uint64_t)t.stride + 1);
    t.magic_rows = t.rows_in == 1 ? 0u : (uint32_t)((1ull << 32) / (uint64_t)t.rows_in + 1);
    const int64_t grid = (int64_t)t.coltiles * t.rowtiles * ceil_div(t.planes, t.c);
    // A thread per quad and group, and more to stage the input where that takes more than one round of four loads.
    const int32_t words = t.c * t.rows_in * t.stride;
    const uint32_t threads = (uint32_t)std::min(kConvThreads, (std::max(t.c * t.trg * t.tcq, words / 4) + 63) / 64 * 64);
    const uint32_t lds = (uint32_t)words * 4;
    hipLaunchKernelGGL((k_conv_depthwise_tile<KH, KW, S, R>), dim3((uint32_t)grid), dim3(threads), lds, s, a, t);
    return hipGetLastError();
}

// Whether a thread per output is the faster, by what both kernels measured over 64 to 16384 planes of 1 to 12544 outputs (us,
// thread per output against tile):
//  - 3 x 3, staging costs more than 18 byte loads until there are some 180000 outputs: 1024 x 10 x 10 3.6, 4.0; 1024 x 14 x 14 4.4, 4.1;
//    4096 x 14 x 14 8.4, 5.6; on planes of under 16 outputs at any number: 16384 x 3 x 3 4.0, 5.2. With strides of 2, which stage four
//    times the outputs, the planes must be larger: 4096 x 10 x 10 5.9, 6.5; 16384 x 10 x 10 13.3, 12.4; 1024 x 20 x 20 5.8, 5.3;
//  - 5 x 5, 50 byte loads, the tile wins on all but the smallest planes: 1024 x 3 x 3 5.5, 4.1; 4096 x 2 x 2 3.9, 5.1;
//  - one dimension: 256 x 300 3.3, 3.2; 1024 x 300 4.4, 3.8; 64 x 300 2.9, 3.2.
bool depthwise_by_output(const ConvDepthwiseArgs &a, int64_t results)
{
    const int64_t plane = (int64_t)a.oh * a.ow;
    if (a.kh == 1) return results < (a.sw == 1 ? 75000 : 150000);
    if (a.kh == 3) return a.sw == 1 ? results < 180000 || plane < 16 : results < (plane < 400 ? 800000 : 180000) || plane < 100;
    return plane < 9 && !(a.sw == 2 && plane >= 4 && results <= 4096 * plane);
}

// Whether k_conv_depthwise_tile covers the window; the extents and the results' number keep its 32-bit positions and grid.
bool depthwise_tile_ok(const ConvDepthwiseArgs &a, int64_t results)
{
    constexpr int32_t limit = 1 << 28;
    return !depthwise_by_output(a, results) && results < (1 << 30) && a.dh == 1 && a.dw == 1 && (a.kw == 3 || a.kw == 5) && (a.kh == a.kw || a.kh == 1) && (a.sw == 1 || a.sw == 2) &&
           (a.sh == a.sw || (a.kh == 1 && a.oh == 1)) && a.h < limit && a.w < limit && a.oh < limit && a.ow < limit &&
           a.ph < limit && a.pw < limit;
}

int64_t conv_grid(int64_t threads)
{
    return std::max<int64_t>(1, std::min<int64_t>((threads + kConvThreads - 1) / kConvThreads, int64_t(1) << 20));
}

}  // namespace

hipError_t launch_conv_pack(const ConvPackArgs &a, hipStream_t s, const char **kernel)
{
    *kernel = "conv-pack16";
    const int64_t total = (int64_t)a.images * a.groups * a.kp * (a.ldb / 16) + (int64_t)a.wrows * (a.kp / 16);
    if (total == 0) return hipSuccess;
    const dim3 grid((uint32_t)conv_grid(total)), block(kConvThreads);
    if (((uintptr_t)a.cols & 15) == 0) hipLaunchKernelGGL(k_conv_pack<true>, grid, block, 0, s, a);
    else hipLaunchKernelGGL(k_conv_pack<false>, grid, block, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_conv_depthwise(const ConvDepthwiseArgs &a, hipStream_t s, const char **kernel)
{
    *kernel = "conv-depthwise-i8";
    const int64_t total = (int64_t)a.batch * a.cout * a.oh * a.ow;
    if (total == 0) return hipSuccess;
    if (depthwise_tile_ok(a, total)) {
        *kernel = "conv-depthwise-tile-i8";
        const bool one = a.sw == 1;
        if (a.kh == 3) return one ? launch_depthwise_tile<3, 3, 1, 4>(a, s) : launch_depthwise_tile<3, 3, 2, 4>(a, s);
        if (a.kh == 5) return one ? launch_depthwise_tile<5, 5, 1, 4>(a, s) : launch_depthwise_tile<5, 5, 2, 4>(a, s);
        if (a.kw == 3) return one ? launch_depthwise_tile<1, 3, 1, 1>(a, s) : launch_depthwise_tile<1, 3, 2, 1>(a, s);
        return one ? launch_depthwise_tile<1, 5, 1, 1>(a, s) : launch_depthwise_tile<1, 5, 2, 1>(a, s);
    }
    const dim3 grid((uint32_t)conv_grid(total)), block(kConvThreads);
#define OG_DW(XS, WS)                                                                                     \
    do {                                                                                                 \
        if (a.kh == 3 && a.kw == 3) hipLaunchKernelGGL((k_conv_depthwise<XS, WS, true>), grid, block, 0, s, a);  \
        else hipLaunchKernelGGL((k_conv_depthwise<XS, WS, false>), grid, block, 0, s, a);                       \
    } while (0)
    if (a.x_signed) {
        if (a.w_signed) OG_DW(true, true);
        else OG_DW(true, false);
    } else {
        if (a.w_signed) OG_DW(false, true);
        else OG_DW(false, false);
    }
#undef OG_DW
    return hipGetLastError();
}

}  // namespace og
