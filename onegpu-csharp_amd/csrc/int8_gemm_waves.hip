// The int8 product for small results and for operands of any alignment: every wave of a workgroup computes the whole
// output tile over its own share of K, straight from global memory, and the waves' sums meet in LDS once at the end.
//
//  - A tile is 16 FM x 16 FN (v_mfma_i32_16x16x64_i8); the workgroup's WAVES waves take its 64-deep steps in turn (step
//    s belongs to wave s % WAVES), so the loop has no barrier and no wave waits for another's loads. Each wave keeps D
//    steps of both operands in flight in its registers (D (FM + FN) KB a wave; the LDS-DMA ring of the 128 tile holds
//    80 KB a workgroup), which is what a small grid needs: it is bound by the latency of its first bytes and by how
//    much it has in flight, not by the matrix cores.
//  - A, and B stored N x K: a fragment (lane l: row l % 16, k 16 (l / 16) .. + 15) is one 16-byte load of that row, 64
//    contiguous bytes a row across the wave. The loads take any byte address. In the last, partial step a row's final
//    16 bytes are read instead and moved down to their place with zeros behind (K >= 16), so nothing past the row
//    is read.
//  - B stored K x N: the step's 64 rows of 16 FN bytes go through a patch of LDS of the wave's own and come back
//    transposed (ds_read_b64_tr_b8). The last tile of a row of tiles starts at column N - 16 FN (N >= 16 FN) and
//    leaves the columns that the tile before it has to that one, so no load needs a column mask. Rows past K read
//    as zero (the buffer's range).
//  - Byte sums for the zero points: v_dot4 of each fragment with ones (in the last step, with the ones of the k that
//    exist); sum (s - z')(t - w') = sum s t - w' sum s - z' sum t + K z' w'   (mod 2^32).
//  - ksplit > 1: blockIdx also picks a slice of K; each slice's sums (its zero points applied) go to a dense int32
//    buffer of [batch * ksplit + slice][M][N] which the summing pass of the split 128 tile adds up.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "og_internal.hpp"

namespace og {

namespace {

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef int32_t v2i __attribute__((ext_vector_type(2)));

// Position of 16-byte chunk c of staged row k of B (rows of 16 FN bytes). LDS serves 256 bytes a cycle: the 16 rows of
// one chunk that half a transpose read touches (k % 16 < 8 or >= 8 of rows k and k + 16) must fall on 16 different
// 16-byte slots of 256 bytes; rows 256 / (16 FN) apart share their slots, so the bits of k above that, and bit 4,
// move the chunk.
template <int FN>
__device__ __forceinline__ int wv_pos(int k, int c)
{
    if constexpr (FN == 8) return c ^ (((k >> 1) & 3) | (((k >> 4) & 1) << 2));
    else if constexpr (FN == 4) return c ^ (((k >> 2) & 1) | (((k >> 4) & 1) << 1));
    else if constexpr (FN == 2) return c ^ ((k >> 4) & 1);
    else return c;
}

// The 16 bytes of v moved down by sh bytes, zeros behind them.
__device__ __forceinline__ v4i wv_shift(v4i v, int32_t sh)
{
    uint64_t lo = (uint32_t)v.x | ((uint64_t)(uint32_t)v.y << 32), hi = (uint32_t)v.z | ((uint64_t)(uint32_t)v.w << 32);
    const int32_t b = 8 * (sh & 7);
    const uint64_t carry = b ? hi << (64 - b) : 0ull;
    lo = (lo >> b) | carry;
    hi >>= b;
    if (sh >= 8) {
        lo = hi;
        hi = 0;
    }
    if (sh >= 16) lo = 0;
    return (v4i){(int32_t)lo, (int32_t)(lo >> 32), (int32_t)hi, (int32_t)(hi >> 32)};
}

// ... moved up by sh bytes, zeros before them.
__device__ __forceinline__ v4i wv_shift_up(v4i v, int32_t sh)
{
    uint64_t lo = (uint32_t)v.x | ((uint64_t)(uint32_t)v.y << 32), hi = (uint32_t)v.z | ((uint64_t)(uint32_t)v.w << 32);
    const int32_t b = 8 * (sh & 7);
    const uint64_t carry = b ? lo >> (64 - b) : 0ull;
    hi = (hi << b) | carry;
    lo <<= b;
    if (sh >= 8) {
        hi = lo;
        lo = 0;
    }
    if (sh >= 16) hi = 0;
    return (v4i){(int32_t)lo, (int32_t)(lo >> 32), (int32_t)hi, (int32_t)(hi >> 32)};
}

__device__ __forceinline__ int32_t wv_dot16(v4i v, v4i ones, int32_t acc)
{
    acc = dot4((uint32_t)v.x, (uint32_t)ones.x, acc);
    acc = dot4((uint32_t)v.y, (uint32_t)ones.y, acc);
    acc = dot4((uint32_t)v.z, (uint32_t)ones.z, acc);
    return dot4((uint32_t)v.w, (uint32_t)ones.w, acc);
}

// Ints of LDS a wave uses: its patch of B (B stored K x N) and later its sums, [16 FM][16 FN + 4] (the pad puts the four
// row groups of an accumulator register on different banks), A's row sums and B's column sums.
template <int FM, int FN, bool TRANS_B>
constexpr int wv_region()
{
    const int part = 16 * FM * (16 * FN + 4) + 16 * FM + 16 * FN;
    const int patch = TRANS_B ? 0 : 64 * 16 * FN / 4;
    return part > patch ? part : patch;
}

// The instances whose XCDs may share the tiles out as a grid (waves_xcd_rows).
template <int FM, int FN, bool TRANS_B, bool CONV>
constexpr bool waves_xcd_grid = FM == 4 && FN == 4 && !TRANS_B && !CONV;

}  // namespace

// CONV: B is the column matrix of a convolution that is never written down (ConvView); row k holds channel k / taps at
// tap k % taps. With unit strides and rows of the output as long as the input's, 16 columns of a row are 16 consecutive
// bytes of that channel's plane, and which of them lie in the padding depends on the tap and the columns alone: a mask
// for each tap and 16-byte piece of the tile, made once. A piece that reaches past the image is read from its first or last
// 16 bytes and moved into place.
template <int FM, int FN, bool TRANS_B, int WAVES, int D, bool SUM_A, bool MIS, bool CONV>
__device__ __forceinline__ void waves_tile(const GemmArgs &g, const ConvView &cv, int32_t tiles_n, int32_t tiles_m,
                                           int32_t ksplit, int32_t slice_steps, int32_t xcd_m)
{
    static_assert(!CONV || (!TRANS_B && !MIS), "a column matrix is K x N");
    constexpr int BM = 16 * FM, BN = 16 * FN, THREADS = 64 * WAVES, LDT = BN + 4, REGION = wv_region<FM, FN, TRANS_B>();
    constexpr int ROWS_AT = BM * LDT, COLS_AT = ROWS_AT + BM;   // a region's row and column sums
    __shared__ __attribute__((aligned(1024))) int32_t smem[WAVES * REGION + 4 * BN + BM];
    __shared__ float red[2 * WAVES];
    __shared__ uint16_t pad_mask[CONV ? kConvMaxTaps * FN : 1];   // bit e: column 16 j + e of tap t reads the image
    int32_t *const ColW = smem + WAVES * REGION, *const ColIB = ColW + BN, *const RowZ = ColIB + BN;
    float *const ColSc = reinterpret_cast<float *>(RowZ + BM), *const ColFb = ColSc + BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g4 = lane >> 4;
    // The hardware deals workgroup ids round-robin to the 8 XCDs: each XCD takes one run of tiles (row tiles of a column
    // of tiles next to each other), so that what neighbours share, down to the halves of a cache line, is in its L2; or
    // (xcd_m > 0) one block of tiles of an xcd_m x 8 / xcd_m grid of them (waves_xcd_rows).
    const int32_t tiles = tiles_n * tiles_m, blocks = tiles * g.batch, per_xcd = (blocks + 7) >> 3;
    int32_t bid = (int32_t)(blockIdx.x & 7u) * per_xcd + (int32_t)(blockIdx.x >> 3);
    if (waves_xcd_grid<FM, FN, TRANS_B, CONV> && xcd_m > 0) {
        const int32_t x = (int32_t)(blockIdx.x & 7u), i = (int32_t)(blockIdx.x >> 3), rows = (tiles_m + xcd_m - 1) / xcd_m;
        const int32_t xn = x / xcd_m, cols = (tiles_n * xcd_m + 7) >> 3, in = i / rows;
        const int32_t xtm = (x - xn * xcd_m) * rows + (i - in * rows), xtn = xn * cols + in;
        bid = in < cols && xtm < tiles_m && xtn < tiles_n ? xtn * tiles_m + xtm : blocks;
    }
    if (bid >= blocks) return;   // whole workgroup
    const int32_t slot = bid;
    const int32_t bsplit = bid / tiles;
    bid -= bsplit * tiles;
    const int32_t batch = bsplit / ksplit, kc = bsplit - batch * ksplit;
    const int32_t tn = bid / tiles_m, tm = bid - tn * tiles_m;
    const int32_t M = g.M, N = g.N, K = g.K, lda = g.lda, ldb = g.ldb;
    const int32_t m0 = tm * BM;
    // The first column the tile reads, and the first it stores (B stored K x N: the last tile moves back to N - BN).
    const int32_t n_own = tn * BN, n0 = TRANS_B ? n_own : min(n_own, N - BN);
    const int32_t s_end = (K + 63) >> 6, s0 = kc * slice_steps, s1 = min(s_end, s0 + slice_steps);
    const bool a_signed = g.flags & OG_GEMM_A_INT8, b_signed = g.flags & OG_GEMM_B_INT8;
    const int32_t flip_a = a_signed ? 0 : (int32_t)0x80808080, flip_b = b_signed ? 0 : (int32_t)0x80808080;

    // The tile's operand ranges (MIS: from and to a whole dword; what a dword holds past the operand is never used, and
    // lies inside the operand's buffer, GEMM_WHOLE_DWORDS).
    const uint8_t *const a_at = g.A + batch * g.strideA + (int64_t)m0 * lda;
    const uint8_t *const b_at = g.B + batch * g.strideB + (CONV ? (int64_t)0 : TRANS_B ? (int64_t)n0 * ldb : (int64_t)n0);
    const uint32_t a_skip = MIS ? (uint32_t)(uintptr_t)a_at & 3u : 0u, b_skip = MIS ? (uint32_t)(uintptr_t)b_at & 3u : 0u;
    const uint8_t *const a_base = a_at - a_skip, *const b_base = b_at - b_skip;
    int32_t a_bytes = (min(BM, M - m0) - 1) * lda + K;
    int32_t b_bytes = CONV ? cv.bytes : TRANS_B ? (min(BN, N - n0) - 1) * ldb + K : (K - 1) * ldb + BN;
    if constexpr (MIS) {
        a_bytes = (a_bytes + (int32_t)a_skip + 3) & ~3;
        b_bytes = (b_bytes + (int32_t)b_skip + 3) & ~3;
    }

    // Byte offsets of this lane's loads at step 0; rows past the operand repeat its last row (their sums are not
    // stored). `back`: how far the lane's 16 bytes move back in the last, partial step to end at K.
    uint32_t off_a[FM], off_b[FN];
#pragma unroll
    for (int i = 0; i < FM; i++) off_a[i] = a_skip + (uint32_t)(min(16 * i + i16, M - 1 - m0) * lda + 16 * g4);
#pragma unroll
    for (int j = 0; j < FN; j++) {
        if constexpr (TRANS_B) off_b[j] = b_skip + (uint32_t)(min(16 * j + i16, N - 1 - n0) * ldb + 16 * g4);
        else off_b[j] = b_skip + (uint32_t)(((64 / FN) * j + lane / FN) * ldb + 16 * (lane % FN));
    }
    const int32_t tail_step = (K & 63) ? s_end - 1 : -1;
    const int32_t back = max(0, 64 * (s_end - 1) + 16 * g4 + 16 - K);
    auto step_a = [&](int32_t s) { return (uint32_t)(64 * s) - (uint32_t)(s == tail_step ? back : 0); };
    auto step_b = [&](int32_t s) { return TRANS_B ? step_a(s) : (uint32_t)(64 * s) * (uint32_t)ldb; };

    // 16 bytes at any address: as they are, or (MIS) the four whole dwords from the one that holds the first byte, and
    // the fifth where they do not start on a dword; put together when they are used.
    struct Piece {
        v4i v;
        int32_t x;
    };
    auto fetch = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
        Piece p;
        if constexpr (MIS) {
            p.v = __builtin_amdgcn_raw_buffer_load_b128(r, off & ~3u, 0, 0);
            p.x = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (off & 3u) ? (off & ~3u) + 16u : 0x80000000u, 0, 0);
        } else {
            p.v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
            p.x = 0;
        }
        return p;
    };
    auto whole = [](const Piece &p, uint32_t off) {
        if constexpr (!MIS) return p.v;
        return (v4i){(int32_t)__builtin_amdgcn_alignbyte((uint32_t)p.v.y, (uint32_t)p.v.x, off),
                     (int32_t)__builtin_amdgcn_alignbyte((uint32_t)p.v.z, (uint32_t)p.v.y, off),
                     (int32_t)__builtin_amdgcn_alignbyte((uint32_t)p.v.w, (uint32_t)p.v.z, off),
                     (int32_t)__builtin_amdgcn_alignbyte((uint32_t)p.x, (uint32_t)p.v.w, off)};
    };

    // CONV: the piece of row k, columns n0 + 16 (lane % FN) ..: its tap in the low half of x, how far its bytes are from
    // their place (16 and more: none is wanted) in the high half.
    auto fetch_conv = [&](__amdgpu_buffer_rsrc_t r, uint32_t k) {
        const uint32_t c = __umulhi(k, cv.magic_taps), t = k - c * (uint32_t)cv.taps;
        const uint32_t th = __umulhi(t, cv.magic_kw), tw = t - th * (uint32_t)cv.kw;
        const int32_t start = (int32_t)(c * (uint32_t)cv.plane) + n0 + 16 * (lane % FN) +
                              ((int32_t)th * cv.dh - cv.ph) * cv.w + (int32_t)tw * cv.dw - cv.pw;
        const int32_t at = min(max(start, 0), cv.bytes - 16);
        Piece p;
        p.v = __builtin_amdgcn_raw_buffer_load_b128(r, (uint32_t)at, 0, 0);
        p.x = (int32_t)t | (min(max(start - at, -16), 16) << 16);
        return p;
    };
    const uint32_t xz4 = CONV && g.ZB ? *g.ZB * 0x01010101u : 0u;   // what a tap in the padding reads
    auto whole_conv = [&](const Piece &p) {
        v4i v = p.v;
        const int32_t sh = p.x >> 16;
        if (__any(sh != 0)) v = sh >= 0 ? wv_shift(v, sh) : wv_shift_up(v, -sh);
        const uint32_t m = pad_mask[(p.x & 0xFFFF) * FN + lane % FN];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t keep = ((((m >> (4 * q)) & 15u) * 0x00204081u) & 0x01010101u) * 0xFFu;
            v[q] = (int32_t)(((uint32_t)v[q] & keep) | (xz4 & ~keep));
        }
        return v;
    };

    Piece fa[D][FM], fb[D][FN];
    auto load = [&](int d, int32_t s) {
        // A step past this slice's last loads nothing (an empty range).
        const bool in = s < s1;
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)a_base, (short)0, in ? a_bytes : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)b_base, (short)0, in ? b_bytes : 0, 0x00020000);
        const uint32_t ka = step_a(s), kb = step_b(s);
#pragma unroll
        for (int i = 0; i < FM; i++) fa[d][i] = fetch(ra, off_a[i] + ka);
#pragma unroll
        for (int j = 0; j < FN; j++) {
            if constexpr (CONV) fb[d][j] = fetch_conv(rb, (uint32_t)(64 * s + (64 / FN) * j + lane / FN));
            else fb[d][j] = fetch(rb, off_b[j] + kb);
        }
    };

#pragma unroll
    for (int d = 0; d < D; d++) load(d, s0 + wave + WAVES * d);

    // The epilogue's operands, requested behind the first loads and kept as stored, so that nothing waits for them (or
    // for the loads before them) here: thread t < BN column n0 + t's, thread t < BM row m0 + t's zero point.
    const uint32_t epi = g.epi;
    uint32_t zb_raw = 0, za_raw = 0, ib = 0;
    float sc = 0.0f, act = 0.0f, fbias = 0.0f;
    {
        const int32_t n = min(n0 + min(tid, BN - 1), N - 1), m = min(m0 + min(tid, BM - 1), M - 1);
        if (g.ZB) zb_raw = g.ZB[(g.flags & OG_GEMM_ZB_PER_COL) ? n : 0];
        if (g.ZA) za_raw = g.ZA[(g.flags & OG_GEMM_ZA_PER_ROW) ? m : 0];
        if (epi & OG_EPI_INT_BIAS) ib = (uint32_t)g.bias[n];
        if (epi & (OG_EPI_FLOAT | EPI_REQUANT)) sc = g.scale[(epi & OG_EPI_SCALE_PER_COL) ? n : 0];
        if (epi & EPI_SCALE_PRODUCT) act = *g.act_scale;
        if (epi & OG_EPI_FLOAT_BIAS) fbias = g.fbias[n];
    }

    if constexpr (CONV) {
        for (int e = tid; e < cv.taps * FN; e += THREADS) {
            const int32_t t = e / FN, th = t / cv.kw, tw = t - th * cv.kw;
            int32_t n = n0 + 16 * (e - t * FN), oh = n / cv.w, ow = n - oh * cv.w;
            uint32_t m = 0;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int32_t ih = oh + th * cv.dh - cv.ph, iw = ow + tw * cv.dw - cv.pw;
                m |= (ih >= 0 && ih < cv.h && iw >= 0 && iw < cv.w ? 1u : 0u) << i;
                if (++ow == cv.w) {
                    ow = 0;
                    oh++;
                }
            }
            pad_mask[e] = (uint16_t)m;
        }
        __syncthreads();
    }

    v4i acc[FM][FN];
    int32_t rs[FM], cs[FN];
#pragma unroll
    for (int i = 0; i < FM; i++) {
        rs[i] = 0;
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = (v4i){0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < FN; j++) cs[j] = 0;
    int32_t *const region = smem + wave * REGION;

    auto use = [&](int d, int32_t s) {
        v4i a[FM], b[FN], ones = (v4i){0x01010101, 0x01010101, 0x01010101, 0x01010101};
        const uint32_t ka = step_a(s), kb = step_b(s);
        if constexpr (TRANS_B) {
#pragma unroll
            for (int j = 0; j < FN; j++) b[j] = whole(fb[d][j], off_b[j] + kb) ^ flip_b;
        } else {
            uint8_t *const patch = reinterpret_cast<uint8_t *>(region);
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int k = (64 / FN) * j + lane / FN;
                *reinterpret_cast<v4i *>(patch + k * BN + 16 * wv_pos<FN>(k, lane % FN)) =
                    CONV ? whole_conv(fb[d][j]) : whole(fb[d][j], off_b[j] + kb);
            }
            // A wave's LDS accesses are performed in order, so its reads see its writes; only the compiler is held back.
            asm volatile("" ::: "memory");
#pragma unroll
            for (int j = 0; j < FN; j++) {
                v2i t[2];
#pragma unroll
                for (int hh = 0; hh < 2; hh++) {
                    const int k = 16 * g4 + 8 * hh + (i16 >> 1);
                    t[hh] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                        (__attribute__((address_space(3))) v2i *)(patch + k * BN + 16 * wv_pos<FN>(k, j) + 8 * (i16 & 1)));
                }
                b[j] = (v4i){t[0].x, t[0].y, t[1].x, t[1].y} ^ flip_b;
            }
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int i = 0; i < FM; i++) a[i] = whole(fa[d][i], off_a[i] + ka) ^ flip_a;
        if (s == tail_step) {
#pragma unroll
            for (int i = 0; i < FM; i++) a[i] = wv_shift(a[i], back);
            if constexpr (TRANS_B) {
#pragma unroll
                for (int j = 0; j < FN; j++) b[j] = wv_shift(b[j], back);
            }
            ones = wv_shift(ones, back);
        }
        if constexpr (SUM_A) {
#pragma unroll
            for (int i = 0; i < FM; i++) rs[i] = wv_dot16(a[i], ones, rs[i]);
        }
#pragma unroll
        for (int j = 0; j < FN; j++) cs[j] = wv_dot16(b[j], ones, cs[j]);
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i], b[j], acc[i][j], 0, 0, 0);
    };

    for (int32_t s = s0 + wave; s < s1; s += WAVES * D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (s + WAVES * d < s1) use(d, s + WAVES * d);
            load(d, s + WAVES * (d + D));
        }
    }

    // Every wave's sums into its region (MFMA 16 x 16 layout: lane l holds rows 4 (l / 16) + r of column l % 16), the byte
    // sums of the four k groups (lanes l, l + 16, l + 32, l + 48) added first.
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) region[(16 * i + 4 * g4 + r) * LDT + 16 * j + i16] = acc[i][j][r];
    if constexpr (SUM_A) {
#pragma unroll
        for (int i = 0; i < FM; i++) {
            int32_t v = rs[i] + __shfl_xor(rs[i], 16);
            v += __shfl_xor(v, 32);
            if (g4 == 0) region[ROWS_AT + 16 * i + i16] = v;
        }
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
        int32_t v = cs[j] + __shfl_xor(cs[j], 16);
        v += __shfl_xor(v, 32);
        if (g4 == 0) region[COLS_AT + 16 * j + i16] = v;
    }
    if (tid < BN) {
        ColW[tid] = b_signed ? sext8(zb_raw) : (int32_t)zb_raw - 128;
        ColIB[tid] = (int32_t)ib;
        ColSc[tid] = (epi & EPI_SCALE_PRODUCT) ? __fmul_rn(act, sc) : sc;
        ColFb[tid] = fbias;
    }
    if (tid < BM) RowZ[tid] = a_signed ? sext8(za_raw) : (int32_t)za_raw - 128;
    __syncthreads();

    // Store, V columns a thread (4 where the rows of C are whole 16-byte pieces, 4 bytes of a requantized row), the
    // waves' sums added up:  C = sum - w' s_m - z' (t_n - k w')  (+ int bias, and the epilogue).
    const uint32_t k_len = (uint32_t)(min(64 * s1, K) - 64 * s0);
    float rmn = __int_as_float(0x7F800000), rmx = __int_as_float(0xFF800000);
    const int64_t c_at = bsplit * g.strideC;
    // MODE 0: int32 (+ bias); 1: float32; 2: requantized bytes.
    auto store = [&](auto v_tag, auto mode_tag) __attribute__((always_inline)) {
        constexpr int V = decltype(v_tag)::value, MODE = decltype(mode_tag)::value, CG = BN / V, EROWS = THREADS / CG;
        static_assert(THREADS % CG == 0, "a thread's columns are the same in every row it stores");
        const int c = V * (tid % CG), r0 = tid / CG;
        const int32_t n = n0 + c;
        if (n >= N || n < n_own) return;   // V = 4: N and n_own are multiples of 4
        uint32_t wz[V], ct[V];
#pragma unroll
        for (int e = 0; e < V; e++) {
            wz[e] = (uint32_t)ColW[c + e];
            ct[e] = 0u - k_len * wz[e];
#pragma unroll
            for (int w = 0; w < WAVES; w++) ct[e] += (uint32_t)smem[w * REGION + COLS_AT + c + e];
        }
#pragma unroll 2
        for (int row = r0; row < BM; row += EROWS) {
            const int32_t m = m0 + row;
            if (m >= M) break;
            uint32_t v[V], ss = 0;
#pragma unroll
            for (int e = 0; e < V; e++) v[e] = (uint32_t)ColIB[c + e];
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                const int32_t *const p = smem + w * REGION + row * LDT + c;
                if constexpr (V == 4) {
                    const v4i t = *reinterpret_cast<const v4i *>(p);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] += (uint32_t)t[e];
                } else {
                    v[0] += (uint32_t)p[0];
                }
                if constexpr (SUM_A) ss += (uint32_t)smem[w * REGION + ROWS_AT + row];
            }
            const uint32_t zz = (uint32_t)RowZ[row];
            const int64_t at = c_at + (int64_t)m * N + n;
            uint32_t word = 0;
            float f[V];
#pragma unroll
            for (int e = 0; e < V; e++) {
                if constexpr (SUM_A) v[e] -= wz[e] * ss;
                v[e] -= zz * ct[e];
                if constexpr (MODE == 1) {
                    f[e] = __fmul_rn((float)(int32_t)v[e], ColSc[c + e]);
                    if (epi & OG_EPI_FLOAT_BIAS) f[e] = __fadd_rn(f[e], ColFb[c + e]);
                    rmn = fminf(rmn, f[e]);
                    rmx = fmaxf(rmx, f[e]);
                } else if constexpr (MODE == 2) {
                    word |= requantize_byte(v[e], ColSc[c + e], g.zp_y, (epi & EPI_REQUANT_U8) != 0) << (8 * e);
                }
            }
            if constexpr (MODE == 2) {
                if constexpr (V == 4) *reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(g.C) + at) = word;
                else static_cast<uint8_t *>(g.C)[at] = (uint8_t)word;
            } else if constexpr (MODE == 1) {
                float *const o = static_cast<float *>(g.C) + at;
                if constexpr (V == 4)
                    *reinterpret_cast<v4i *>(o) = (v4i){__float_as_int(f[0]), __float_as_int(f[1]), __float_as_int(f[2]), __float_as_int(f[3])};
                else *o = f[0];
            } else {
                int32_t *const o = static_cast<int32_t *>(g.C) + at;
                if constexpr (V == 4) *reinterpret_cast<v4i *>(o) = (v4i){(int32_t)v[0], (int32_t)v[1], (int32_t)v[2], (int32_t)v[3]};
                else *o = (int32_t)v[0];
            }
        }
    };
    const int esize = (epi & EPI_REQUANT) ? 1 : 4;
    const bool vec = N % 4 == 0 && (((uintptr_t)g.C + (uint64_t)c_at * esize) & (4 * esize - 1)) == 0;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    if (epi & EPI_REQUANT) {
        if (vec) store(I4{}, I2{});
        else store(I1{}, I2{});
    } else if (epi & OG_EPI_FLOAT) {
        if (vec) store(I4{}, I1{});
        else store(I1{}, I1{});
    } else {
        if (vec) store(I4{}, I0{});
        else store(I1{}, I0{});
    }
    if (g.ranges) store_workgroup_range<THREADS>(rmn, rmx, red, g.ranges, (uint32_t)slot);
}

template <int FM, int FN, bool TRANS_B, int WAVES, int D, bool SUM_A, bool MIS>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_waves(GemmArgs g, int32_t tiles_n, int32_t tiles_m, int32_t ksplit,
                                                           int32_t slice_steps, int32_t xcd_m)
{
    waves_tile<FM, FN, TRANS_B, WAVES, D, SUM_A, MIS, false>(g, ConvView{}, tiles_n, tiles_m, ksplit, slice_steps, xcd_m);
}

template <int FM, int FN, int WAVES, int D, bool SUM_A>
__global__ __launch_bounds__(64 * WAVES) void k_conv_waves(GemmArgs g, ConvView cv, int32_t tiles_n, int32_t tiles_m,
                                                           int32_t ksplit, int32_t slice_steps, int32_t xcd_m)
{
    waves_tile<FM, FN, false, WAVES, D, SUM_A, false, true>(g, cv, tiles_n, tiles_m, ksplit, slice_steps, xcd_m);
}

namespace {

// Whether some row of A or of B (stored N x K) does not start on a dword.
bool waves_off_dword(const GemmArgs &g)
{
    return ((g.lda | g.ldb | g.strideA | g.strideB | (int64_t)(uintptr_t)g.A | (int64_t)(uintptr_t)g.B) & 3) != 0;
}

// The rows of the XCDs' grid of tile blocks, xm x 8 / xm, each XCD one block of the result: its L2 is then filled with that
// block's rows of A and columns of B, where a run of tiles down the columns takes most of A into every one. 0: runs, where
// no grid reads less by a tenth, a block would be more tiles than an XCD's 32 CUs take at once, or batches and slices
// of K share the XCDs out already. For the 64 x 64 tile with B stored K x N: 1024 x 768 x 1536 9.4 -> 8.7 us, x 3072 13.5 -> 12.7,
// 1024 x 1024 x 4096 16.3 -> 15.7, 777 x 768 x 2048 10.6 -> 10.2. With B stored N x K, bound by its loads of 64 bytes a row,
// it gives nothing (1024 x 768 x 3072 15.2 -> 15.3), and the smaller tiles pay for the mapping (200 x 256 x 2048 6.1 -> 6.2).
int32_t waves_xcd_rows(int64_t tm, int64_t tn, int64_t batch, int bm, int bn)
{
    const int64_t blocks = tm * tn * batch, per = (blocks + 7) / 8;
    if (batch != 1 || blocks > 256 || blocks < 16) return 0;
    const int64_t run = std::min(tm, per) * bm + (per + tm - 1) / tm * bn;
    int32_t best = 0;
    int64_t least = run * 9 / 10;
    for (int32_t xm = 1; xm <= 8; xm *= 2) {
        const int64_t rows = (tm + xm - 1) / xm, cols = (tn * xm + 7) / 8;
        if (rows * cols <= 32 && rows * bm + cols * bn < least) {
            least = rows * bm + cols * bn;
            best = xm;
        }
    }
    return best;
}

// The instances: the tile in 16 x 16 blocks, the waves, and the steps each wave keeps in flight.
enum Shape { S16x16W4, S16x32W4, S16x64W4, S16x64W1, S16x128W4, S32x32W2, S32x32W4, S32x64W4, S32x64W1, S64x64W4, S64x64W2 };

template <int FM, int FN, int WAVES, int D>
void launch_waves_as(const GemmArgs &g, int32_t ksplit, int32_t slice_steps, const ConvView *cv, hipStream_t s)
{
    const int32_t tn = (g.N + 16 * FN - 1) / (16 * FN), tm = (g.M + 16 * FM - 1) / (16 * FM);
    const bool grid_ok = waves_xcd_grid<FM, FN, false, false> && !(g.flags & OG_GEMM_TRANSPOSE_B) && !cv;
    const int32_t xm = grid_ok ? waves_xcd_rows(tm, tn, g.batch, 16 * FM, 16 * FN) : 0;
    const int64_t per_xcd = xm ? (int64_t)((tm + xm - 1) / xm) * ((tn * xm + 7) / 8) : ((int64_t)tn * tm * g.batch + 7) / 8;
    const dim3 grid(8u * (uint32_t)per_xcd), block(64 * WAVES);
    // A's byte sums are needed only when B's shifted zero point can be non-zero; B's are always formed.
    const bool sum_a = (g.flags & OG_GEMM_ZB) || !(g.flags & OG_GEMM_B_INT8);
    if (cv) {
        if (sum_a) hipLaunchKernelGGL((k_conv_waves<FM, FN, WAVES, D, true>), grid, block, 0, s, g, *cv, tn, tm, ksplit, slice_steps, xm);
        else hipLaunchKernelGGL((k_conv_waves<FM, FN, WAVES, D, false>), grid, block, 0, s, g, *cv, tn, tm, ksplit, slice_steps, xm);
        return;
    }
#define OG_W(T, SA, MIS) hipLaunchKernelGGL((k_gemm_waves<FM, FN, T, WAVES, D, SA, MIS>), grid, block, 0, s, g, tn, tm, ksplit, slice_steps, xm)
    if (g.flags & OG_GEMM_TRANSPOSE_B) {
        if (waves_off_dword(g)) {
            if (sum_a) OG_W(true, true, true);
            else OG_W(true, false, true);
        } else {
            if (sum_a) OG_W(true, true, false);
            else OG_W(true, false, false);
        }
    } else {
        if (sum_a) OG_W(false, true, false);
        else OG_W(false, false, false);
    }
#undef OG_W
}

}  // namespace

// Conditions of the kernel: rows of at least one 16-byte piece, every offset of a tile's buffer under 2^31, and fewer than
// 2^32 threads in the grid, which is what a launch takes (a batch of millions of narrow products passes that on four waves
// a tile). The form for N x K operands off a dword reads whole dwords, which must lie inside the operands' buffers.
bool waves_ok(const GemmArgs &g)
{
    const bool trans_b = g.flags & OG_GEMM_TRANSPOSE_B;
    const int64_t lim = 0x7FFFFFFFll - 512;
    if (trans_b && waves_off_dword(g) && !(g.flags & GEMM_WHOLE_DWORDS)) return false;
    if (g.M < 1 || g.N < 1 || g.K < 16 || (!trans_b && g.N < 16)) return false;
    if ((int64_t)63 * g.lda + g.K > lim) return false;
    if (trans_b ? (int64_t)127 * g.ldb + g.K > lim : (int64_t)(g.K + 63) * g.ldb > lim) return false;
    if ((int64_t)((g.M + 15) / 16) * ((g.N + 15) / 16) * g.batch > (lim >> 5)) return false;
    return (waves_count(g, waves_plan(g)) + 64) * 64 < (1ll << 32);
}

// Whether the 128 tile's split form is the faster for a walk of `steps` on t tiles: it cuts K finer than this kernel does.
//  - Not sliced here, 80 steps and more (150 x 3456 x 5504 15.9 us there against 18.4, 32 x 8192 x 5120 14.5 against 16.7; 300 x 2048 x
//    4672 15.4 against 18.4); from 60 with B stored N x K and CUs to spare (150 x 3456 x 4096 16.1 against 18.8, 46 x 4261 x 4608 14.2
//    against 16.2, x 3584 equal; on 256 workgroups 64 x 4096 x 4672 14.4 against 9.3), from 70 where a fifth of the 64 x 64 tiles' rows is
//    padding (96 x 8192 x 4608 18.9 against 22.1, x 4096 22.7 against 20.4). 5 to 16 rows of B stored N x K: 200 (16 x 1024 x 14336 13 against 16 to 17.5, x 8192 12 against 11).
//  - B stored K x N, where the 128 tile splits: a step reads pieces of 64 rows, which HBM answers late. The line is where the mean of B
//    from HBM and from the Infinity Cache is equal: on two waves 44 steps up to 32 rows (17 x 4096 x 3072 from HBM 11 against 15 us,
//    from the cache 11 against 10; x 4096 13, 19 and 11, 12), 56 up to 64 (64 x 3072 x 4096 15, 20 and 14, 13), past that 60 on few
//    tiles (96 x 1024 x 4096 13, 19 and 12, 10); 72 on larger tiles (64 x 5120 x 4608 19, 22 and 16, 16; 128 x 5120 x 4608 22, 26).
//  - Sliced here: the slices are at most 8 to 16, there up to 64, which tells from 160 steps on wide results and from 200 on narrower
//    ones (64 x 4096 x 11008 17 to 21.6 against 19 to 23.4; 96 x 2048 x 14336 N x K 17 against 21; but 64 x 512 x 11008 N x K 15 against 10).
bool waves_walk_too_deep(const GemmArgs &g, int shape, int64_t t, int64_t steps, int64_t slices)
{
    const bool nk = g.flags & OG_GEMM_TRANSPOSE_B;
    const int64_t cols = (int64_t)g.N * g.batch;
    if (g.M <= 16) return nk && g.M > 4 && slices == 1 && steps >= 200;
    if (slices > 1) return (!nk || g.M > 32) && (steps >= 200 ? cols >= 1536 : steps >= 160 && cols >= 3072);
    if (steps >= 80) return true;
    if (nk) return t <= 192 ? steps >= 60 : steps >= 70 && shape == S64x64W4 && (g.M + 63) / 64 * 256 > g.M * 5;
    const int64_t most = shape == S32x32W2 ? (g.M <= 32 ? 44 : g.M <= 64 ? 56 : t <= 100 ? 60 : 80)
                         : shape == S64x64W4 || (shape == S32x64W4 && g.M <= 64) ? 72 : 80;
    return steps >= most && direct_split(g) > 1;
}

// The tile, waves and slices of K, from what sweeps of both layouts measured (MI355X, three sets of operands in turn):
//  - The smallest tile whose workgroups still go round the chip's 256 CUs once is the fastest: its workgroups read
//    the least each. 128 x 384 x 384: 32 x 32 (48 workgroups) 4.2 us, 32 x 64 5.2, 64 x 64 6.2; 512 x 768 x 3072: 32 x 64
//    (192) 10.7 us, 64 x 64 (96) 14.9; 1 x 8192 x 1024: 16 x 32 (256) 5.0 us, 16 x 64 5.2, 16 x 16 (512) 5.8.
//    A depth of 80 steps and more takes a larger tile for that, in slices that fill the round: 128 x 1024 x 8192 32 x 64 in
//    four 12.3 us, 32 x 32 whole 22.6; 2 x 96 x 900 x 9856 64 x 64 in four 16.8, 32 x 32 whole 49.
//  - Against the 128 tile fed by LDS DMA, one whole round of 64 x 64 also needs 16 steps to win (1024 x 1024 x 4096
//    21.4 -> 17.3 us, 256 x 4096 x 1024 8.8 -> 8.4, 1024 x 768 x 768 equal; 512 x 1536 x 384 6.5 -> 6.8). A deep K goes to its split
//    form (waves_walk_too_deep).
//  - With more than one round (one_round false), the largest tile on one or two waves, so that several workgroups
//    share a CU: 2000 x 2001 x 2003: 64 x 64 on two waves 54 us, on four 60; 333 x 64 x 333 x 96: 32 x 64 on one wave 12.4 us, 64 x 64
//    on two 13.5; 1 x 51865 x 768: 16 x 64 on one wave 10.3 us, on four 12.9.
//  - Slices of K cost a second launch (3.5 to 4 us): only where the waves' walk is longer than that: few tiles and at
//    least 56 steps (512 x 49 x 4608: 8.5 us in 8 slices, over 10 whole), or few rows of a deep B stored K x N, whose
//    narrow tiles read pieces of lines (1 x 1537 x 8192: 16 x 64 in 8 slices 9.2 us, 16 x 16 whole over 10).
WavesPlan waves_plan(const GemmArgs &g)
{
    WavesPlan p{};
    const bool trans_b = g.flags & OG_GEMM_TRANSPOSE_B;
    const int64_t steps = (g.K + 63) / 64;
    auto tiles = [&](int bm, int bn) { return (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * g.batch; };
    auto fits = [&](int bn) { return trans_b || g.N >= bn; };   // K x N: the last tile moves back inside the row
    constexpr int64_t kRound = 256;
    int64_t t = 0, slices = 1;
    p.one_round = true;
    if (g.M <= 16) {
        const bool deep = !trans_b && fits(64) && steps >= (g.N % 16 ? 64 : 96) && tiles(16, 64) <= kRound;
        if (!deep && (t = tiles(16, 16)) <= kRound) p.shape = S16x16W4;
        else if (!deep && fits(32) && (t = tiles(16, 32)) <= kRound) p.shape = S16x32W4;
        else if (fits(64) && (t = tiles(16, 64)) <= kRound) p.shape = S16x64W4;
        else if (!trans_b && fits(128) && (t = tiles(16, 128)) <= kRound) p.shape = S16x128W4;
        else {
            p.one_round = false;
            p.shape = fits(64) ? S16x64W1 : fits(32) ? S16x32W4 : S16x16W4;
        }
        if (deep) slices = std::min(kRound / t, steps / 8);
    } else if (!fits(32)) {
        p.shape = S16x16W4;
        p.one_round = (t = tiles(16, 16)) <= kRound;
    } else {
        const bool deep = steps >= 80 && tiles(32, 32) > 64 && fits(64);
        if (deep && (t = tiles(32, 64)) <= 64) p.shape = S32x64W4;
        else if (deep && g.M > 32 && (t = tiles(64, 64)) <= 64) p.shape = S64x64W4;
        else if ((t = tiles(32, 32)) <= kRound) p.shape = steps >= 24 && t <= 64 ? S32x32W4 : S32x32W2;
        else if (fits(64) && (t = tiles(32, 64)) <= kRound) p.shape = S32x64W4;
        else if (fits(64) && g.M > 32 && (t = tiles(64, 64)) <= kRound) p.shape = S64x64W4;
        else {
            p.one_round = false;
            // 32 rows where 64 would be padded by more, or K too short for two waves to share.
            const bool rows32 = g.M <= 32 || steps <= 2 ||
                                (steps <= 8 && (int64_t)(g.M + 31) / 32 * 32 * 108 <= (int64_t)(g.M + 63) / 64 * 64 * 100);
            p.shape = !fits(64) ? S32x32W2 : rows32 ? S32x64W1 : S64x64W2;
        }
        if (p.one_round && t <= 64 && steps >= 56) slices = std::min(kRound / t, steps / 8);
    }
    // The slices' int32 sums stay within what every context's workspace and the fixed scratch hold from the start.
    slices = std::min<int64_t>(slices, kWavesMaxPartials / std::max<int64_t>((int64_t)g.M * g.N * g.batch * 4, 1));
    slices = std::max<int64_t>(slices, 1);
    p.beats_direct = p.one_round && !(slices == 1 && p.shape == S64x64W4 && steps < 16) && !waves_walk_too_deep(g, p.shape, t, steps, slices);
    p.slice_steps = (int32_t)((steps + slices - 1) / slices);
    p.slices = (int32_t)((steps + p.slice_steps - 1) / p.slice_steps);
    return p;
}

// Few rows, B stored K x N. The few-rows kernels request all of B at once, which is what HBM answers fastest, and then hand
// their parts over, which costs more the more rows there are; here a wave walks its steps one memory latency after the
// other, with a few in flight. So the line is a depth that grows with the rows and with the columns (more waves to hide
// a latency, up to one round of the CUs), and rows of B that are multiples of 1 KiB, which keep to few of the memory
// channels, draw it in. It lies where the two are equal in the mean of B from HBM and B from the Infinity Cache (us, few-rows
// kernel against this one):
//   1 x 4096 x 1280     from HBM 7.2, 6.7    from the cache 6.9, 6.4      16 x 4096 x 4096    11.5, 13.8    10.9, 10.4
//   1 x 4096 x 3584              8.8, 12.1             7.9, 9.2           16 x 11008 x 4096   16.7, 15.0    16.1, 11.0
//   5 x 8192 x 4096              13, 16                 12, 11.5          16 x 3072 x 5120    12, 16        -
// Past one round the walk is one wave's alone: 40960 columns of 3072, one row, 27 against 39 us; of 1024, 16 against 16, from the
// cache 15 against 12. A depth of at most 512 is one part, with nothing to hand over: 1 x 28672 x 512 8.0 against 8.5. Under 16 slabs
// of columns the other choice is the two-launch form: 1 x 1024 x 1024 7.7 against 5.3, 8 x 1024 x 4096 8.1 against 11.6.
bool waves_few_rows(const GemmArgs &g)
{
    const int64_t cols = (int64_t)g.N * g.batch, slabs = (int64_t)((g.N + 127) / 128) * g.batch;
    if (slabs < 16) return g.K <= 3072;
    if (g.M <= 4 && g.K >= 4096) return false;
    if (!waves_plan(g).one_round) return g.M > 8 ? g.K <= 1536 : g.K <= 1024 && cols * g.K <= 70'000'000;
    if (g.M <= 8 && g.K > 256 && g.K <= 512 && cols > 16384) return false;
    return g.K <= 5120 && g.K <= 1536 + 128 * g.M + std::min<int64_t>(cols, 32768) / 32 + (g.ldb % 1024 ? 384 : 0);
}

// Past one round of the CUs, an aligned product whose K is no multiple of 64 (or whose rows of B are whole dwords only) has
// the register-staged tiles (k_gemm_tiled) as the other choice: they start late, read far less a 64-deep step and win where K
// is deep. Both as fitted to what they measured (us; k in 1024s, kn and nk the two layouts of B):
//  - waves: 4 and, a round of 1024 tiles of 64 x 64, 13.5 k (14.4 k nk); a partly filled second round costs 26 k; tall results
//    15% more, for each XCD reads all of A; and B itself at 2 to 3.4 TB/s, by how many rows of tiles read it.
//  - 256 tiles: 56 + 23 k a round of 256. 128 tiles: 21.5 + 12.5 k (11.9 k nk) a full round of 512, 18.5 + 9.6 k (7.3 k nk) where the
//    last round gives a CU at most one.
// 4096 x 4096 x 4080 kn 149 (256 tiles) against 234 us, x 400 66 against 36; 2048 x 4096 x 3088 56 (128) against 80, x 1040 33 against 30;
// 2000 x 1504 x 4112 56 against 42; 128 x 50304 x 4112 nk 91 against 133.
bool staged_tile_faster(const GemmArgs &g)
{
    const bool nk = g.flags & OG_GEMM_TRANSPOSE_B;
    const double k = g.K / 1024.0;
    auto tiles = [&](int64_t t) { return (double)(((g.M + t - 1) / t) * ((g.N + t - 1) / t) * g.batch); };
    const double n64 = tiles(64), n128 = tiles(128);
    double slope = n64 <= 1024 ? 13.5 * std::max(0.65, n64 / 1024) : std::max(26.0, 0.0142 * n64);
    slope *= (nk ? 1.07 : 1.0) * (g.M >= 4 * (int64_t)g.N ? 1.15 : 1.0);
    const double waves = 4 + k * std::max(slope, (double)g.N * g.batch / (g.M <= 16 ? 3300 : g.M <= 32 ? 2800 : g.M <= 64 ? 2440 : 2000));
    double staged = 0;
    if (tiled_uses_large(g.M, g.N, g.batch)) {
        staged = std::ceil(tiles(256) / 256) * (56 + 23 * k);
    } else {
        const double full = std::floor(n128 / 512), rest = n128 - 512 * full;
        const double two = 21.5 + (nk ? 11.9 : 12.5) * k, one = (18.5 + (nk ? 7.3 : 9.6) * k) * (full > 0 ? 0.85 : 1.0);
        staged = full * two + (rest > 256 ? two : rest > 0 ? one : 0);
    }
    return staged < waves;
}

constexpr int kShapeWaves[] = {4, 4, 4, 1, 4, 2, 4, 4, 1, 4, 2};

int64_t waves_count(const GemmArgs &g, const WavesPlan &p) { return (int64_t)waves_range_groups(g, p) * kShapeWaves[p.shape]; }

double waves_walk(const WavesPlan &p) { return (double)p.slice_steps / kShapeWaves[p.shape]; }

uint32_t waves_range_groups(const GemmArgs &g, const WavesPlan &p)
{
    static const int bm[] = {16, 16, 16, 16, 16, 32, 32, 32, 32, 64, 64}, bn[] = {16, 32, 64, 64, 128, 32, 32, 64, 64, 64, 64};
    const int64_t n = (int64_t)((g.M + bm[p.shape] - 1) / bm[p.shape]) * ((g.N + bn[p.shape] - 1) / bn[p.shape]) * g.batch;
    return (uint32_t)std::min<int64_t>(n, int64_t(1) << 30);
}

// The tile's rows, columns and waves; "-splitk" where K is cut into slices.
const char *waves_name(const WavesPlan &p, bool conv)
{
#define OG_N(tile) {{"mfma-i8-waves" tile, "mfma-i8-waves" tile "-splitk"}, {"conv-waves" tile, "conv-waves" tile "-splitk"}}
    static const char *const names[][2][2] = {OG_N("16x16x4"), OG_N("16x32x4"), OG_N("16x64x4"), OG_N("16x64x1"), OG_N("16x128x4"),
                                              OG_N("32x32x2"), OG_N("32x32x4"), OG_N("32x64x4"), OG_N("32x64x1"),
                                              OG_N("64x64x4"), OG_N("64x64x2")};
#undef OG_N
    return names[p.shape][conv][p.slices > 1];
}

hipError_t launch_gemm_waves(const GemmArgs &g, const WavesPlan &p, const Workspace &ws, hipStream_t s,
                             const char **kernel, const ConvView *cv)
{
    *kernel = waves_name(p, cv != nullptr);
    GemmArgs a = g;
    if (p.slices > 1) {
        a.C = ws.partials;
        a.strideC = (int64_t)g.M * g.N;
        a.batch = g.batch * p.slices;
        a.epi = 0;
        a.ranges = nullptr;   // the summing pass records the ranges
    }
    switch (p.shape) {
    case S16x16W4: launch_waves_as<1, 1, 4, 6>(a, p.slices, p.slice_steps, cv, s); break;
    case S16x32W4: launch_waves_as<1, 2, 4, 5>(a, p.slices, p.slice_steps, cv, s); break;
    case S16x64W4: launch_waves_as<1, 4, 4, 4>(a, p.slices, p.slice_steps, cv, s); break;
    case S16x64W1: launch_waves_as<1, 4, 1, 4>(a, p.slices, p.slice_steps, cv, s); break;
    case S16x128W4: launch_waves_as<1, 8, 4, 3>(a, p.slices, p.slice_steps, cv, s); break;
    case S32x32W2: launch_waves_as<2, 2, 2, 5>(a, p.slices, p.slice_steps, cv, s); break;
    case S32x32W4: launch_waves_as<2, 2, 4, 5>(a, p.slices, p.slice_steps, cv, s); break;
    case S32x64W4: launch_waves_as<2, 4, 4, 4>(a, p.slices, p.slice_steps, cv, s); break;
    case S32x64W1: launch_waves_as<2, 4, 1, 4>(a, p.slices, p.slice_steps, cv, s); break;
    case S64x64W4: launch_waves_as<4, 4, 4, 3>(a, p.slices, p.slice_steps, cv, s); break;
    default: launch_waves_as<4, 4, 2, 3>(a, p.slices, p.slice_steps, cv, s); break;
    }
    return hipGetLastError();
}

}  // namespace og
