// Normalised cross-correlation block matcher for gfx950.
//
// Reference: BlockMatcherNCC (CluTec.Cuda.MultiView/BlockMatcherNCC.cu): EvalMsd :338-373
// (base mean / std-dev), EvalSim :180-336 (ncc = (E[IJ] - muI muJ) / (sdI sdJ), zero when
// the norm is small, clamped at 0 before quantisation), strict '>' winner-take-all over d
// (:298).  The reference forms E[x^2] - mu^2 in float, which cancels catastrophically;
// here every box sum is an exact integer:
//     cov = N*SIJ - SI*SJ,  var = N*SS - S^2,  score = cov / sqrt(varI * varJ)
// and only the last step is FP32: score = float(cov) * rI * rJ with rI = 1/sqrt(varI)
// rounded once from FP64.  A window whose standard deviation is below one grey level
// (var < N^2) scores 0.  The winner key is ((floor(max(score,0) * 2^23)) << 8 | 255-d):
// the best score, lowest d on ties, the same key layout as the SAD / census matcher so
// the right-view merge and the check are shared.
//
// The sum of products is a contraction: for one image row, SIJ of every left pixel x of a block
// of 32 against every right pixel x' of another is one 32 x 32 integer matrix product over the
// window's N pixels.  Pixels enter as signed bytes I - 128, J - 128: the covariance does not
// change (SI and SJ shift with them), and every product and sum stays exact in int32.  See
// ncc_mm_kernel for the layout, and ncc_sums_kernel for short ranges.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "window_mm.hpp"

namespace stereo {
namespace ncc {

using namespace winmm;

constexpr int XT = 128;       // left pixels of a workgroup's tile: 32 per wave
constexpr int RBMAX = 4;      // image rows of a tile
constexpr int RCOLS = XT + 256;  // right pixels x0 - 256 .. x0 + 127 that the tile's candidates reach
constexpr int MAXROWS = RBMAX + 11;

// Per-pixel window statistics: .x = centre times the window sum of I - 128 (int; centre -1 for
// the left image, 1 for the right one, so that a product of the two is -SI SJ), .y = float bits of the
// reciprocal standard-deviation factor scale / sqrt(N SS - S^2) (0 when the
// variance is below N^2, and 0 outside the matchable area).  A workgroup does a
// 64 x 32 block: the input rows it needs go to LDS, the horizontal sums of v and v^2
// over the window's columns -- byte sums and byte dot products of whole dwords -- go to LDS, and
// each lane slides the vertical sums down 8 rows of one column.  Both images of a pair go
// through one launch (blockIdx.z).  What bounds it: the 33 MB that a 1920x1080 pair writes;
// with a loop over the window's bytes and FP64 square root and division per pixel it took 28.5 us.
// Now 16.8 us.
constexpr int ST_W = 64, ST_H = 32;

// float(scale / sqrt(var)) as FP64 square root and division give it.  A reciprocal square root of
// FP32 accuracy and one cubic step in FP64 are within 2^-50 of that value; where the result lies
// within 2^-44 of the middle of two floats, the long way decides.
__device__ __forceinline__ float inv_deviation(uint32_t var, float scale)
{
    const double v = (double)var, y = (double)__builtin_amdgcn_rsqf((float)var);
    const double e = __builtin_fma(-v * y, y, 1.0);
    const double r = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y) * (double)scale;
    // the 29 bits of r below a float's last: half way is 1 << 28
    const uint32_t low = (uint32_t)__double_as_longlong(r) & 0x1FFFFFFFu;
    if (low - ((1u << 28) - 256u) <= 512u) return (float)((double)scale / sqrt(v));
    return (float)r;
}

template <int A>
__global__ __launch_bounds__(256) void ncc_stats_kernel(View img0, int2* out0, float scale0, View img1, int2* out1,
                                                        float scale1, int pitch_px)
{
    const View img = blockIdx.z ? img1 : img0;
    const int sign = blockIdx.z ? 1 : -1;
    int2* const out = blockIdx.z ? out1 : out0;
    const float scale = blockIdx.z ? scale1 : scale0;
    constexpr int ROWS = ST_H + 2 * A, P = 2 * A + 1, N = P * P;
    constexpr int PD = (ST_W + 2 * A + 3) / 4 + 1, ND = (P + 3) / 4;  // dwords of a row, of a window row
    constexpr uint32_t TAIL = P % 4 == 1 ? 0xFFu : 0xFFFFFFu;
    static_assert(N <= 181, "32-bit variances");
    __shared__ uint32_t pix[ROWS * PD];
    __shared__ uint2 hs[ROWS][ST_W];
    const int x0 = blockIdx.x * ST_W, y0 = blockIdx.y * ST_H;
    {
        const int c = threadIdx.x & 31, x = x0 - A + 4 * c;
        const bool whole = x >= 0 && x + 4 <= img.w;
        int xs[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) xs[j] = clampi(x + j, 0, img.w - 1);
        if (c < PD) {
#pragma unroll
            for (int i = 0; i < (ROWS + 7) / 8; ++i) {
                const int r = (threadIdx.x >> 5) + 8 * i;
                const uint8_t* row = row_ptr<const uint8_t>(img, clampi(y0 - A + r, 0, img.h - 1));
                uint32_t w = 0;
                if (whole) __builtin_memcpy(&w, row + x, 4);
                else w = row[xs[0]] | (uint32_t)row[xs[1]] << 8 | (uint32_t)row[xs[2]] << 16 | (uint32_t)row[xs[3]] << 24;
                if (r < ROWS) pix[r * PD + c] = w;
            }
        }
    }
    __syncthreads();
    const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
#pragma unroll 4
    for (int r = rg; r < ROWS; r += 4) {
        const uint32_t* q = pix + r * PD + (c >> 2);
        uint32_t w[ND + 1];
#pragma unroll
        for (int k = 0; k <= ND; ++k) w[k] = q[k];
        uint32_t a = 0, b = 0;
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            uint32_t d = __builtin_amdgcn_alignbyte(w[k + 1], w[k], c & 3);
            if (k == ND - 1) d &= TAIL;
            a = __builtin_amdgcn_sad_u8(d, 0u, a);
            b = __builtin_amdgcn_udot4(d, d, b, false);
        }
        hs[r][c] = make_uint2(a, b);
    }
    __syncthreads();
    const int x = x0 + c;
    uint32_t sv = 0, ssv = 0;
#pragma unroll
    for (int j = 0; j < 2 * A; ++j) {
        sv += hs[rg * 8 + j][c].x;
        ssv += hs[rg * 8 + j][c].y;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = rg * 8 + i;  // output row y0 + r uses LDS rows r .. r + 2 A
        const uint2 in = hs[r + 2 * A][c], old = hs[r][c];
        sv += in.x;
        ssv += in.y;
        const int y = y0 + r;
        if (x < img.w && y < img.h) {
            int2 o = make_int2(0, 0);
            if (x >= A && x < img.w - A && y >= A && y < img.h - A) {
                const uint32_t var = (uint32_t)N * ssv - sv * sv;
                o.x = sign * ((int)sv - 128 * N);
                o.y = __float_as_int(var >= (uint32_t)(N * N) ? inv_deviation(var, scale) : 0.0f);
            }
            out[(size_t)y * pitch_px + x] = o;
        }
        sv -= old.x;
        ssv -= old.y;
    }
}

__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }

// max over the 32 lanes of each half-wave of 16 values: lane (bits 4 .. 1 = r) receives value r.
// A level folds two values into one register, half of the lanes each.
__device__ __forceinline__ uint32_t fold_max(uint32_t (&v)[16], int lane)
{
    uint32_t a[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const auto sw = __builtin_amdgcn_permlane16_swap(v[r], v[r + 8], false, false);
        a[r] = umax(sw[0], sw[1]);
    }
    uint32_t b[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t t0 = umax(a[r], dpp_mov<0x128>(a[r])), t1 = umax(a[r + 4], dpp_mov<0x128>(a[r + 4]));  // row_ror:8
        b[r] = (lane & 8) ? t1 : t0;
    }
    uint32_t c[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint32_t t0 = umax(b[r], dpp_mov<0x141>(b[r])), t1 = umax(b[r + 2], dpp_mov<0x141>(b[r + 2]));  // row_half_mirror
        c[r] = (lane & 4) ? t1 : t0;
    }
    const uint32_t t0 = umax(c[0], dpp_mov<0x4E>(c[0])), t1 = umax(c[1], dpp_mov<0x4E>(c[1]));  // quad_perm [2,3,0,1]
    const uint32_t d = (lane & 2) ? t1 : t0;
    return umax(d, dpp_mov<0xB1>(d));  // quad_perm [1,0,3,2]
}

// Keys of one 32 x 32 block, in the tile's own form: score << 8 | (287 - (xb - x'b) - c_r), the
// disparity without the lane's part, which is constant for a lane (its row r is left pixel
// xb + c_r + 4 half, its column right pixel x'b + n).  The largest of a register row and of a
// lane are then the winners, and the lane's part is taken off once at the end (lane_sub); 0: no
// candidate.  MASK: only the candidates whose bit c_r is set in ok.
template <int P, bool MASK>
__device__ __forceinline__ void block_keys(const v16i& acc, uint32_t (&t)[16], const int (&nsi)[16], const float (&rfi)[16],
                                           int sj, float rj, uint32_t top, uint32_t ok)
{
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int c = 8 * (r >> 2) + (r & 3);
        int prod;  // -SI SJ, both below 2^14 in size
        asm("v_mul_i32_i24 %0, %1, %2" : "=v"(prod) : "v"(nsi[r]), "v"(sj));
        const int cov = __mul24(P * P, acc[r]) + prod;
        const float sc = (float)cov * rfi[r] * rj;
        // v_cvt_u32_f32 truncates and clamps negative values to 0: floor(max(score, 0) * 2^23)
        uint32_t q;
        asm("v_cvt_u32_f32 %0, %1" : "=v"(q) : "v"(sc));
        // kept whole in a scalar register: one v_lshl_add_u32
        uint32_t add = top - (uint32_t)c;
        asm("" : "+s"(add));
        t[r] = (q << 8) + add;
        if (MASK) t[r] &= (uint32_t)__builtin_amdgcn_sbfe((int)ok, c, 1);  // all ones or 0
    }
}

__device__ __forceinline__ uint32_t row_max(const uint32_t (&t)[16])
{
    uint32_t m = umax(t[0], t[1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) m = umax(umax(m, t[r]), t[r + 1]);
    return m;
}

// Bits c (0 .. 27) of the candidates with disparity d + c in [ds, de), bin by bin (8 disparities
// a bit of `bins`) for the band search.
template <bool BAND>
__device__ __forceinline__ uint32_t disparity_bits(int d, int ds, int de, uint32_t bins)
{
    const int lo = clampi(ds - d, 0, 32), hi = clampi(de - d, 0, 32);
    uint32_t m = (uint32_t)(((1ull << hi) - 1ull) & ~((1ull << lo) - 1ull));
    if (BAND) {
        const int b = d >> 3;  // the bin of c = 0 (-4 at the least), its bit at bit 0 of g
        const uint32_t g = b >= 0 ? bins >> min(b, 31) : bins << min(-b, 31);
        uint64_t e = 0;
#pragma unroll
        for (int j = 0; j < 5; ++j) e |= (uint64_t)(((g >> j) & 1u) * 0xFFu) << (8 * j);
        m &= (uint32_t)(e >> (d & 7));
    }
    return m;
}

// A workgroup takes XT left pixels of `rb` image rows and the disparities of one segment; wave w the
// 32 left pixels from x0 + 32 w.  The tile's pixels of both images are staged in LDS; then each
// wave works alone: per image row, the left operand once, and for each block of 32 right pixels
// its operand from LDS, STEPS matrix instructions and the 16 keys a lane holds of the block.  The
// left winners stay in registers over the blocks and are folded across the lanes at the end of the
// row; the right winners meet in LDS, and in the right key plane at the end of the tile.
//
// What bounds it: the VALU operations of the key, 8 per candidate (covariance 2, to float and
// two factors 3, quantise and pack 2, the two maxima 0.5 each), where products and
// running sums on the VALU took 18.9; the matrix cores are busy a fifth of the time.  1920x1080,
// 256 disparities, 11 x 11: 411 -> 214 us (the frame 429 -> 225).  Tiles of 4 rows: with 8 the 2025
// workgroups end in a part-filled round (the frame 6 us longer).
template <int P, bool BAND>
__global__ __launch_bounds__(256, 3) void ncc_mm_kernel(NccParams p)
{
    using S = Shape<P>;
    constexpr int A = P / 2;
    // a window's last byte is 10 columns on
    constexpr int RDW = RCOLS / 4 + 3, LDW = XT / 4 + 3;
    constexpr int RCS = ((MAXROWS * RDW + 23) & ~31) + 8;
    static_assert(RCS > MAXROWS * RDW && RCS % 32 == 8, "whole copies, in different banks");
    __shared__ uint32_t rimg[4 * RCS];
    __shared__ uint32_t limg[MAXROWS * LDW];
    __shared__ uint32_t rkey[RBMAX * RCOLS];
    const int nty = (p.H + p.rb - 1) / p.rb;
    // segments of a tile together, then tiles along the row.  The band search keeps the
    // hardware's round-robin over the XCDs: its work sits in a few image regions, and a
    // contiguous range per XCD would load some XCDs far more than others
    const int w = BAND ? (int)blockIdx.x : xcd_remap(blockIdx.x, gridDim.x);
    const int seg = w % p.nseg, rest = w / p.nseg;
    const int tx = rest % p.ntx, ty = rest / p.ntx;
    if (ty >= nty) return;
    const int x0 = tx * XT, y0 = ty * p.rb;
    const int W = p.W, H = p.H;
    const int ds = seg * p.seg_len, de = min(p.D, ds + p.seg_len);

    // the right columns that the tile's disparities reach
    int dlo = ds, dhi = de;
    if (BAND) {
        uint32_t any = 0;
        for (int bx = 0; bx < XT / BM_TILE_W; ++bx)
            for (int by = y0 / BM_TILE_H; by <= min(y0 + p.rb - 1, H - 1) / BM_TILE_H; ++by)
                if (tx * (XT / BM_TILE_W) + bx < p.bins_ntx) any |= p.bins[by * p.bins_ntx + tx * (XT / BM_TILE_W) + bx];
        const int b0 = ds >> 3, b1 = (de - 1) >> 3;
        any &= (uint32_t)((2ull << b1) - (1ull << b0));
        dlo = any ? 8 * __builtin_ctz(any) : de;
        dhi = any ? 8 * (32 - __builtin_clz(any)) : de;
    }
    const int k0 = dlo >> 5, k1 = dhi > dlo ? (dhi + 30) >> 5 : -1;
    if (k1 >= k0) {
        stage_image<6, LDW, 1, 0>(limg, p.L, x0 - A, y0 - A, p.rb + S::ROWS - 1, 0, LDW);
        stage_image<7, RDW, 4, RCS>(rimg, p.R, x0 - 256 - A, y0 - A, p.rb + S::ROWS - 1, 8 * (8 - k1), 8 * (12 - k0) + 3);
    }
    for (int i = threadIdx.x; i < p.rb * RCOLS; i += 256) rkey[i] = 0u;
    __syncthreads();

    const int lane = threadIdx.x & 63, n = lane & 31, half = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xb = x0 + 32 * wv;
    const uint32_t lane_sub = 32u - (uint32_t)n + 4u * half;
    // left pixels of the block that may match, as bits of c_r for this half
    const int xlo = max(0, p.bx - xb), xhi = min(32, W - p.bx - xb);
    const uint32_t xbits = xhi <= xlo ? 0u : (xhi - xlo >= 32 ? ~0u : ((1u << (xhi - xlo)) - 1u) << xlo);
    const uint32_t xmask = xbits >> (4 * half);
    const uint32_t* const lsrc = limg + half * S::HR * LDW + 8 * wv + (n >> 2);
    const uint32_t* const rsrc = rimg + (n & 3) * RCS + half * S::HR * RDW + 8 * (wv + 8) + (n >> 2);

    for (int i = 0; i < p.rb && xbits; ++i) {
        const int y = y0 + i;
        if (y < p.by || y >= H - p.by) continue;
        uint32_t bins = ~0u;
        if (BAND) bins = p.bins[(y / BM_TILE_H) * p.bins_ntx + xb / BM_TILE_W];
        // what block k holds: 0 nothing to search, 1 candidates to mask, 2 only candidates
        auto holds = [&](int k) {
            const int lo = 32 * k - 31, hi = 32 * k + 31;  // disparities of the block
            if (xb - 32 * k + 31 < p.bx) return 0;
            bool part = lo < ds || hi >= de || xb - 32 * k < p.bx || xbits != ~0u;
            if (BAND) {
                const int b0 = max(lo, ds) >> 3, b1 = min(hi, de - 1) >> 3;
                const uint32_t need = (uint32_t)((2ull << b1) - (1ull << b0));
                if ((bins & need) == 0u) return 0;
                part = part || (bins & need) != need;
            }
            return part ? 1 : 2;
        };
        uint32_t key = 0;
        int k = k0;
        while (k <= k1 && !holds(k)) ++k;
        if (k <= k1) {
            uint32_t lacc[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) lacc[r] = 0u;
            v4i av[S::STEPS];
            load_operand_shifted<P, LDW>(av, lsrc + i * LDW, n & 3);
            mask_row<P>(av, S::HR - 1, half ? 0u : ~0u);  // row P
            // left statistics of rows c_r + 4 half: groups of four pixels (the array has room past W)
            int nsi[16];
            float rfi[16];
            const int2* const ls = p.lstats + (size_t)y * p.stats_pitch + xb + 4 * half;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int2 st = ls[8 * (r >> 2) + (r & 3)];
                nsi[r] = st.x;
                rfi[r] = __int_as_float(st.y);
            }
            const int2* const rs = p.rstats + (size_t)y * p.stats_pitch;
            auto products = [&](int kk) {
                v4i bv[S::STEPS];
                load_operand<P, RDW>(bv, rsrc + i * RDW - 8 * kk);
                v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < S::STEPS; ++s) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[s], bv[s], acc, 0, 0, 0);
                return acc;
            };
            auto right = [&](int kk, uint32_t m) {
                atomicMax(&rkey[i * RCOLS + 256 + 32 * (wv - kk) + n], __builtin_elementwise_sub_sat(m, lane_sub));
            };
            auto mask = [&](int kk) {
                const uint32_t bits = disparity_bits<BAND>(32 * kk + 4 * half - n, ds, de, bins);
                return xb - 32 * kk + n >= p.bx ? xmask & bits : 0u;
            };
            // two blocks at once: their left keys take one maximum of three a row
            auto pair = [&](int kk, auto m0) {
                constexpr bool M0 = decltype(m0)::value;
                const int xr = xb - 32 * kk + n;
                const int2 s0 = rs[xr], s1 = rs[xr - 32];
                const v16i a0 = products(kk), a1 = products(kk + 1);
                uint32_t t0[16], t1[16];
                block_keys<P, M0>(a0, t0, nsi, rfi, s0.x, __int_as_float(s0.y), 287u - 32u * (uint32_t)kk, M0 ? mask(kk) : 0u);
                right(kk, row_max(t0));
                block_keys<P, false>(a1, t1, nsi, rfi, s1.x, __int_as_float(s1.y), 255u - 32u * (uint32_t)kk, 0u);
                right(kk + 1, row_max(t1));
#pragma unroll
                for (int r = 0; r < 16; ++r) lacc[r] = umax(umax(lacc[r], t0[r]), t1[r]);
            };
            // most often the first block holds candidates to mask (d < 0) and the next ones none
            if (k < k1 && holds(k + 1) == 2) {
                pair(k, std::true_type{});
                k += 2;
            }
            while (k <= k1) {
                while (k < k1 && holds(k) == 2 && holds(k + 1) == 2) {
                    pair(k, std::false_type{});
                    k += 2;
                }
                if (k <= k1 && holds(k)) {
                    const int2 st = rs[max(xb - 32 * k + n, 0)];
                    const v16i acc = products(k);
                    uint32_t t[16];
                    block_keys<P, true>(acc, t, nsi, rfi, st.x, __int_as_float(st.y), 287u - 32u * (uint32_t)k, mask(k));
                    right(k, row_max(t));
#pragma unroll
                    for (int r = 0; r < 16; ++r) lacc[r] = umax(lacc[r], t[r]);
                }
                ++k;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) lacc[r] = __builtin_elementwise_sub_sat(lacc[r], lane_sub);
            key = fold_max(lacc, lane);
        }
        // the row's winners: lane (r, 0) of each half writes left pixel xb + c_r + 4 half
        const int r = n >> 1, x = xb + 8 * (r >> 2) + (r & 3) + 4 * half;
        if ((lane & 1) == 0 && x < W) p.lkey[(size_t)seg * W * H + (size_t)y * W + x] = key;
    }
    __syncthreads();
    for (int r = 0; r < p.rb && y0 + r < H; ++r)
        for (int c = threadIdx.x; c < RCOLS; c += 256) {
            const uint32_t v = rkey[r * RCOLS + c];
            const int x = x0 - 256 + c;
            if (v && x >= 0 && x < W) atomicMax(&p.rkey[(size_t)(y0 + r) * W + x], v);
        }
}

// ------------------------------------------------------------------------------------
// Short ranges: running sums on the VALU
// ------------------------------------------------------------------------------------
// A block of the matrix kernel holds 32 x 32 candidates whatever the range, so a range of 8 costs
// it as much as one of 32, with the staging and the operands of each row on top.  Running sums
// cost what the range has, 18.9 VALU operations per candidate.  What bounds them: VALU issue (67 %
// busy at D = 256) and the barriers behind it.  1920x1080, 11x11, D = 8: frame 54.6 us, 120 with the
// matrix kernel.  Where the line lies, with both sides measured: ncc_short_range.
//
// One disparity per step: workgroup = 4 waves, tile = 64 columns x 52 rows.  Row phase: lane = (H row
// 0..63, run of 19 columns), products I*J(x-d) and their horizontal sums over 2*AX+1 columns
// (halo from the neighbouring runs by DPP) into LDS (one buffer, two barriers per disparity).
// Column phase: lane = column, wave = 13 rows: vertical running sums give SIJ, the right window's
// (SJ, rJ) come from an LDS tile of the right statistics that is refreshed every 16
// disparities, the left window's are registers.  Left winner in a register, right winner carried
// along the wave by a DPP shift (see bm.hip) and folded into the right key plane.  The images
// are the padded copies (BM_PAD_LEFT), so that the loads need no clamping.
constexpr int TW = 64;
constexpr int RG = 13;
constexpr int TH = 4 * RG;  // 52
constexpr int HROWS = 64;
constexpr int RUN = 19;
constexpr int COLS = 4 * RUN;  // 76 cost columns: tile columns [-6, 70)
constexpr int HSTRIDE = 76;
constexpr int DCH = 8;         // disparities per group (one band-search bin)
constexpr int SDC = 16;        // disparities per right-statistics tile
constexpr int EMIT = 32;       // right-view values parked per wave between flushes
constexpr int SCOLS = TW + SDC - 1;
static_assert(TW == BM_TILE_W, "one column of band-search tiles");

template <int AX, int AY, bool EDGE, bool BAND>
__device__ __forceinline__ void sums_tile(const NccParams& p, uint32_t* hb, int16_t* ssum, float* srinv,
                                         uint32_t (*ebuf)[RG][EMIT], int tx, int ty, int seg)
{
    static_assert(TH + 2 * AY <= HROWS, "tile too tall for the window");
    static_assert(AX <= 6 && 2 * AX + 64 <= COLS, "window wider than the run layout");
    const int tid = threadIdx.x;
    const int x0 = tx * TW, y0 = ty * TH;
    const int W = p.W, H = p.H;
    const int ds = seg * p.seg_len;
    const int de = min(p.D, ds + p.seg_len);
    constexpr int N = (2 * AX + 1) * (2 * AY + 1);

    // row phase identity
    const int run = tid & 3;
    const int hr = tid >> 2;
    const int gyr = clampi(y0 - AY + hr, 0, H - 1);
    const int xs = x0 - 6 + RUN * run;
    const uint8_t* const rowL = row_ptr<const uint8_t>(p.L, gyr) + xs;
    const uint8_t* const rowR = row_ptr<const uint8_t>(p.R, gyr) + xs;
    uint32_t il[RUN];
#pragma unroll
    for (int i = 0; i < RUN; ++i) il[i] = rowL[i];

    // column phase identity
    const int lane = tid & 63;
    const int gw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x = x0 + lane;
    const int rows_here = H - (y0 + gw * RG);
    uint32_t* const rp = p.rkey + (size_t)(y0 + gw * RG) * W;
    uint32_t* const eb = &ebuf[gw][0][0];  // [RG][EMIT]
    const bool lane_ok = x >= p.bx && x < W - p.bx;
    const int dlim = x - p.bx;
    int nsi[RG];     // -SI of the left window
    float rfi[RG];   // 2^23 / sqrt(varI), or 0
    uint32_t lacc[RG], racc[RG];
#pragma unroll
    for (int i = 0; i < RG; ++i) {
        const int y = min(y0 + gw * RG + i, H - 1);
        const int2 st = p.lstats[(size_t)y * p.stats_pitch + min(x, W - 1)];
        nsi[i] = st.x - 128 * N;
        rfi[i] = __int_as_float(st.y);
        lacc[i] = 0;
        racc[i] = 0;
    }
    // band search: the tile's rows lie in at most two 64 x BM_TILE_H bin tiles; rows before
    // ysplit take m0, the others m1 (uniform per wave and row); a group of disparities
    // whose bins neither mask holds is skipped
    uint32_t m0 = ~0u, m1 = ~0u;
    int ysplit = 1 << 30;
    if (BAND) {
        const int tb0 = y0 / BM_TILE_H, tb1 = min(y0 + TH - 1, H - 1) / BM_TILE_H;
        m0 = p.bins[tb0 * p.bins_ntx + tx];
        m1 = p.bins[tb1 * p.bins_ntx + tx];
        ysplit = (tb0 + 1) * BM_TILE_H;
        const int b0 = ds >> 3, b1 = (de - 1) >> 3;
        if (((m0 | m1) & (uint32_t)((2ull << b1) - (1ull << b0))) == 0u) {
            // nothing to search in this segment: every left key is the empty key
            if (x < W) {
                uint32_t* lk = p.lkey + (size_t)seg * W * H + (size_t)(y0 + gw * RG) * W + x;
                for (int i = 0; i < min(RG, rows_here); ++i) lk[(size_t)i * W] = 0u;
            }
            return;
        }
    }

    // right pixels of the run for the current disparity d, byte i of rw = R(xs + i - d)
    // (little-endian over RWW words), and the one that enters next, R(xs - d - 1): one load
    // per disparity instead of RUN (every offset down to xs - de - 1 lies in the matcher's
    // left padding)
    constexpr int RWW = (RUN + 3) / 4;
    // after disparity d: at the end of a block of EMIT disparities (or of the segment) the
    // right-view values parked in the wave's LDS rows go to the right key plane
    auto flush = [&](int d) {
        if ((d & (EMIT - 1)) == EMIT - 1 || d == de - 1) {
            const int base = d & ~(EMIT - 1);
            const int xr = x0 + 63 - (base + lane);
            if (lane <= (d & (EMIT - 1)) && base + lane >= ds && xr >= 0 && xr < W) {
#pragma unroll
                for (int i = 0; i < RG; ++i) {
                    const uint32_t v = eb[i * EMIT + lane];
                    if (i < rows_here && v) atomicMax(&rp[(size_t)i * W + xr], v);
                }
            }
        }
    };
    uint32_t rw[RWW], rnext = 0;
    int wd = -1;  // the disparity rw holds
    int sdc = -SDC;  // the first disparity of the right-statistics tile in LDS (none yet)
    for (int dc = ds; dc < de; dc += DCH) {
        const int dce = min(de, dc + DCH);
        // the band search: rows of this wave that search the group (bit r: row r), wave-uniform
        uint32_t keep = (1u << RG) - 1u;
        if (BAND) {
            const uint32_t bit = 1u << (dc >> 3);  // the group's bin (dc is a multiple of 8)
            const uint32_t lo_rows = (1u << clampi(ysplit - (y0 + gw * RG), 0, RG)) - 1u;
            keep = ((m0 & bit) ? lo_rows : 0u) | ((m1 & bit) ? (((1u << RG) - 1u) & ~lo_rows) : 0u);
            if (((m0 | m1) & bit) == 0u) {
                // no pixel of the tile searches these 8 disparities: the right-view chain
                // moves on by 8 lanes with no new candidates.  The values that leave the
                // wave at lane 63 during those 8 steps sit in lanes 62 .. 55 now.
                if (lane >= 63 - DCH && lane < 63) {
                    const int slot = (dc + 62 - lane) & (EMIT - 1);
#pragma unroll
                    for (int i = 0; i < RG; ++i) eb[i * EMIT + slot] = racc[i];
                }
#pragma unroll
                for (int i = 0; i < RG; ++i) {
                    const uint32_t v = __shfl_up(racc[i], DCH);
                    racc[i] = lane >= DCH ? v : 0u;
                }
                flush(dce - 1);
                continue;
            }
        }
        // right statistics for disparities sdc .. sdc+SDC-1 (right columns x0-sdc-(SDC-1) ..
        // x0+63-sdc), rows of the tile, loaded when the group leaves the tile in LDS: the
        // thread's loads (the last index repeated past the end) are all issued before the
        // barrier, the LDS stores after it
        if (dc - sdc >= SDC) {
            sdc = dc;
            constexpr int SN = TH * SCOLS, SIT = (SN + 255) / 256, SB = SIT;
            static_assert(SIT % SB == 0, "whole batches");
            // an opaque copy of the thread index: the addresses are recomputed here rather
            // than hoisted out of the disparity loop into live registers
            int t0 = tid;
            asm volatile("" : "+v"(t0));
            auto sload = [&](int j) {
                const int k = min(t0 + 256 * j, SN - 1);
                const int r = k / SCOLS, c = k - r * SCOLS;
                const int y = min(y0 + r, H - 1);
                const int xc = clampi(x0 - sdc - (SDC - 1) + c, 0, W - 1);
                return p.rstats[(size_t)y * p.stats_pitch + xc];
            };
#pragma unroll
            for (int j0 = 0; j0 < SIT; j0 += SB) {
                int2 v[SB];
#pragma unroll
                for (int j = 0; j < SB; ++j) v[j] = sload(j0 + j);
                if (j0 == 0) __syncthreads();
#pragma unroll
                for (int j = 0; j < SB; ++j) {
                    const int k = tid + 256 * (j0 + j);
                    if (k < SN) {
                        ssum[k] = (int16_t)(v[j].x + 128 * N);
                        srinv[k] = __int_as_float(v[j].y);
                    }
                }
            }
        }
        if (wd != dc) {
            uint32_t b[RUN];
#pragma unroll
            for (int i = 0; i < RUN; ++i) b[i] = rowR[i - dc];
            rnext = rowR[-dc - 1];
#pragma unroll
            for (int k = 0; k < RWW; ++k) {
                uint32_t w = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * k + j < RUN) w |= b[4 * k + j] << (8 * j);
                rw[k] = w;
            }
        }
        for (int d = dc; d < dce; ++d) {
            // ---- row phase: products and horizontal sums for disparity d
            uint32_t e[RUN + 2 * AX];
#pragma unroll
            for (int i = 0; i < RUN; ++i) e[AX + i] = il[i] * ((rw[i >> 2] >> (8 * (i & 3))) & 0xffu);
#pragma unroll
            for (int k = RWW - 1; k > 0; --k) rw[k] = __builtin_amdgcn_alignbyte(rw[k], rw[k - 1], 3);
            rw[0] = (rw[0] << 8) | rnext;
            rnext = rowR[-d - 2];
            wd = d + 1;
            __syncthreads();  // the previous column phase has read the H buffer
#pragma unroll
            for (int i = 0; i < AX; ++i) {
                e[i] = dpp_mov<DPP_ROW_SHR1>(e[AX + RUN - AX + i]);
                e[AX + RUN + i] = dpp_mov<DPP_ROW_SHL1>(e[AX + i]);
            }
            uint32_t h = 0;
#pragma unroll
            for (int i = 0; i <= 2 * AX; ++i) h += e[i];
            uint32_t* hrow = hb + hr * HSTRIDE + RUN * run;
#pragma unroll
            for (int i = 0; i < RUN; ++i) {
                if (i > 0) h = slide(h, e[i - 1], e[i + 2 * AX]);
                hrow[i] = h;
            }
            __syncthreads();

            // ---- column phase
            uint32_t hv[RG + 2 * AY];
            const uint32_t* hcol = hb + gw * RG * HSTRIDE + lane + 6;
#pragma unroll
            for (int i = 0; i < RG + 2 * AY; ++i) hv[i] = hcol[i * HSTRIDE];
            uint32_t sij = 0;
#pragma unroll
            for (int i = 0; i <= 2 * AY; ++i) sij += hv[i];
            const int soff = (gw * RG) * SCOLS + lane + (SDC - 1) - (d - sdc);
            const int16_t* srow_s = ssum + soff;
            const float* srow_r = srinv + soff;
            const uint32_t dd = 255u - (uint32_t)d;
            bool ok = true;
            if (EDGE) ok = lane_ok && d <= dlim;
            uint32_t key[RG];
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                if (i > 0) sij = slide(sij, hv[i - 1], hv[i + 2 * AY]);
                const int sj = srow_s[i * SCOLS];
                const int cov = __mul24(nsi[i], sj) + (int)__umul24((uint32_t)N, sij);
                const float sc = (float)cov * rfi[i] * srow_r[i * SCOLS];
                // v_cvt_u32_f32 truncates and clamps negative values to 0: the key's
                // floor(max(score, 0) * 2^23) in one instruction
                uint32_t q;
                asm("v_cvt_u32_f32 %0, %1" : "=v"(q) : "v"(sc));
                uint32_t k = (q << 8) | dd;
                if (EDGE) k = ok ? k : 0u;
                if (BAND) k = ((keep >> i) & 1u) ? k : 0u;
                key[i] = k;
                lacc[i] = lacc[i] > k ? lacc[i] : k;
            }
            static_assert(RG == 13, "right-view chain written for 13 rows");
            max_shift_in13(racc, key);
            if (lane == 63) {
#pragma unroll
                for (int i = 0; i < RG; ++i) eb[i * EMIT + (d & (EMIT - 1))] = racc[i];
            }
            flush(d);
        }
    }
    {
        // what is still in flight belongs to right pixels x0 + lane - (de - 1)
        const int xr = x0 + lane - (de - 1);
        if (xr >= 0 && xr < W) {
#pragma unroll
            for (int i = 0; i < RG; ++i)
                if (i < rows_here && racc[i]) atomicMax(&rp[(size_t)i * W + xr], racc[i]);
        }
    }
    if (x < W) {
        uint32_t* lk = p.lkey + (size_t)seg * W * H + (size_t)(y0 + gw * RG) * W + x;
#pragma unroll
        for (int i = 0; i < RG; ++i)
            if (i < rows_here) lk[(size_t)i * W] = lacc[i];
    }
}

// BAND: the band search's instantiation, a kernel of its own so that the full-range
// kernel keeps its register count (and three workgroups per CU)
template <int AX, int AY, bool BAND>
__global__ __launch_bounds__(256, 3) void ncc_sums_kernel(NccParams p)
{
    __shared__ uint32_t hbuf[HROWS * HSTRIDE];
    // right statistics of the tile: window sums (at most 121 x 255, an int16) and 1/sigma
    __shared__ int16_t ssum[TH * SCOLS];
    __shared__ float srinv[TH * SCOLS];
    __shared__ uint32_t ebuf[4][RG][EMIT];
    // one-dimensional grid of ntx * nty * nseg workgroups, renumbered per XCD
    const int nty = (p.H + TH - 1) / TH;
    // the band search keeps the hardware's round-robin over the XCDs: its work sits in a
    // few segments and image regions, and a contiguous range per XCD would load some
    // XCDs far more than others
    const int w = BAND ? (int)blockIdx.x : xcd_remap(blockIdx.x, gridDim.x);
    const int tx = w % p.ntx, rest = w / p.ntx;
    const int ty = rest % nty, seg = rest / nty;
    const int x0 = tx * TW;
    const int de = min(p.D, (seg + 1) * p.seg_len);
    const bool edge = (x0 < p.bx + de - 1) || (x0 + TW > p.W - p.bx);
    if (edge)
        sums_tile<AX, AY, true, BAND>(p, hbuf, ssum, srinv, ebuf, tx, ty, seg);
    else
        sums_tile<AX, AY, false, BAND>(p, hbuf, ssum, srinv, ebuf, tx, ty, seg);
}

// Winning score of every left pixel: the same FP32 arithmetic as the matcher, on a
// window sum computed directly for the winning disparity.
__global__ __launch_bounds__(256) void ncc_score_kernel(NccScoreParams f)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= f.W || y >= f.H) return;
    float out = __int_as_float(0x7fc00000);  // NaN: no match
    uint32_t lk = 0;
    if (x >= f.bx && x < f.W - f.bx && y >= f.by && y < f.H - f.by)
        for (int s = 0; s < f.nseg; ++s) {
            const uint32_t v = f.lkey[(size_t)s * f.W * f.H + (size_t)y * f.W + x];
            lk = v > lk ? v : lk;
        }
    const int d = key_disp(lk);
    if (d >= 0) {
        int sij = 0;
        for (int j = -f.ay; j <= f.ay; ++j) {
            const uint8_t* rl = row_ptr<const uint8_t>(f.L, y + j);
            const uint8_t* rr = row_ptr<const uint8_t>(f.R, y + j);
            for (int i = -f.ax; i <= f.ax; ++i) sij += ((int)rl[x + i] - 128) * ((int)rr[x + i - d] - 128);
        }
        const int2 a = f.lstats[(size_t)y * f.stats_pitch + x];
        const int2 b = f.rstats[(size_t)y * f.stats_pitch + x - d];
        const int n = (2 * f.ax + 1) * (2 * f.ay + 1);
        // the products of I - 128 and J - 128 under the centred sums: the same covariance
        const int cov = n * sij + a.x * b.x;
        // lstats carry the 2^23 key scale; undo it exactly (power of two)
        out = (float)cov * (__int_as_float(a.y) * (1.0f / 8388608.0f)) * __int_as_float(b.y);
    }
    row_ptr<float>(f.score, y)[x] = out;
}

}  // namespace ncc

bool ncc_supported(int ww, int wh, int D)
{
    if (D < 8 || D > 256 || (D % 8) != 0) return false;
    return (ww == 11 && wh == 11) || (ww == 9 && wh == 9) || (ww == 5 && wh == 5) || (ww == 7 && wh == 7);
}

// Which kernel a frame takes: the running sums where the range is short and the frame large enough
// that their two barriers a disparity are hidden (rb = 0).  The matrix kernel costs the same for all
// ranges up to 32, and more with the window; the running sums hardly see the window.  Whole frames in
// us, matrix kernel / running sums:
//    5x5    D =    8         16         24         32         48         64
//    640x480   29.6/29.8  29.8/37.9  29.9/46.8  29.6/42.0  32.3/46.2  31.5/48.7
//   1280x720   57.6/41.4  57.8/50.9  57.9/61.9  57.2/59.6  66.4/75.9  62.7/83.3
//   1920x1080  96.2/53.4  96.3/64.8  96.1/79.3  96.0/90.7   114/131    105/132
//   2560x1440   158/82     158/100    157/121    156/137    190/209    173/211
//   11x11
//    640x480   34.7/29.9  35.1/37.7  35.1/46.4  34.6/41.9  38.3/47.4  37.0/49.4
//   1280x720   68.7/41.9  69.6/51.8  69.7/62.9  68.8/60.4  79.1/75.2  75.6/83.7
//   1920x1080   120/55     120/67     120/82     120/92     142/134    132/135
//   2560x1440   198/82     198/101    198/124    197/138    235/212    218/214
// With an initial map the running sums skip what is masked more finely: at 1920 x 1080, a quarter of
// the size, 11x11, D = 64 150/112, 5x5 119/110; at 1280 x 720 85/67 and 70/65; at 640 x 480 42/51.
static bool ncc_short_range(int W, int H, int D, int ww, bool band)
{
    const double px = (double)W * H;
    const bool wide = ww >= 9;
    if (band) return D <= (wide ? 64 : 48) && px >= 880e3;
    return D <= (wide ? 48 : 32) && px * (wide ? 2 : 1) >= 55e3 * D;
}

void ncc_grid(int W, int H, int D, int ww, bool band, int* ntx, int* rb, int* nseg, int* seg_len)
{
    if (ncc_short_range(W, H, D, ww, band)) {
        *rb = 0;
        *ntx = (W + ncc::TW - 1) / ncc::TW;
        const int tiles = *ntx * ((H + ncc::TH - 1) / ncc::TH);
        int n = (1200 + tiles - 1) / tiles;
        if (n > D / 16) n = D / 16;
        if (n > BM_MAX_SEG) n = BM_MAX_SEG;
        if (n < 1) n = 1;
        const int len = ((D + n - 1) / n + 15) & ~15;
        *seg_len = len;
        *nseg = (D + len - 1) / len;
        return;
    }
    // Tiles of 4 rows where they give every CU four workgroups (three are resident); 2 rows stage
    // more pixels for the same work, so a smaller frame first takes those, and only then splits
    // the disparities, which costs a left key plane per segment.
    *ntx = (W + ncc::XT - 1) / ncc::XT;
    int r = ncc::RBMAX, n = 1, len = (D + 31) & ~31;
    while (r > 2 && *ntx * ((H + r - 1) / r) < 1024) r /= 2;
    while (n < BM_MAX_SEG && len > 64 && *ntx * ((H + r - 1) / r) * n < 512) {
        n *= 2;
        len = ((D + n - 1) / n + 31) & ~31;
    }
    *rb = r;
    *seg_len = len;
    *nseg = (D + len - 1) / len;
}

hipError_t launch_ncc_stats_pair(const View& img0, int2* out0, float scale0, const View& img1, int2* out1, float scale1,
                                 int pitch_px, int ww, hipStream_t s)
{
    if (img0.w != img1.w || img0.h != img1.h) return hipErrorInvalidValue;
    dim3 grid((img0.w + ncc::ST_W - 1) / ncc::ST_W, (img0.h + ncc::ST_H - 1) / ncc::ST_H, 2);
#define NCC_STATS(A)                                                                                                        \
    hipLaunchKernelGGL(ncc::ncc_stats_kernel<A>, grid, dim3(256), 0, s, img0, out0, scale0, img1, out1, scale1, pitch_px); \
    break
    switch (ww) {
    case 11: NCC_STATS(5);
    case 9: NCC_STATS(4);
    case 7: NCC_STATS(3);
    case 5: NCC_STATS(2);
    default: return hipErrorInvalidValue;
    }
#undef NCC_STATS
    return hipGetLastError();
}

template <int P>
static void launch_ncc_p(const NccParams& p, hipStream_t s)
{
    if (p.rb == 0) {
        const dim3 grid(p.ntx * ((p.H + ncc::TH - 1) / ncc::TH) * p.nseg);
        if (p.bins) hipLaunchKernelGGL((ncc::ncc_sums_kernel<P / 2, P / 2, true>), grid, dim3(256), 0, s, p);
        else hipLaunchKernelGGL((ncc::ncc_sums_kernel<P / 2, P / 2, false>), grid, dim3(256), 0, s, p);
    } else {
        const dim3 grid(p.ntx * ((p.H + p.rb - 1) / p.rb) * p.nseg);
        if (p.bins) hipLaunchKernelGGL((ncc::ncc_mm_kernel<P, true>), grid, dim3(256), 0, s, p);
        else hipLaunchKernelGGL((ncc::ncc_mm_kernel<P, false>), grid, dim3(256), 0, s, p);
    }
}

hipError_t launch_ncc(int ww, const NccParams& p, hipStream_t s)
{
    // segments of whole blocks: 32 disparities, or 16 for the running sums
    if (p.rb < 0 || p.rb > ncc::RBMAX || p.nseg < 1 || p.seg_len % (p.rb ? 32 : 16) || p.D > 256 || !p.rkey)
        return hipErrorInvalidValue;
    switch (ww) {
    case 11: launch_ncc_p<11>(p, s); break;
    case 9: launch_ncc_p<9>(p, s); break;
    case 7: launch_ncc_p<7>(p, s); break;
    default: launch_ncc_p<5>(p, s);
    }
    return hipGetLastError();
}

hipError_t launch_ncc_score(const NccScoreParams& f, hipStream_t s)
{
    dim3 grid((f.W + 63) / 64, (f.H + 3) / 4);
    hipLaunchKernelGGL(ncc::ncc_score_kernel, grid, dim3(256), 0, s, f);
    return hipGetLastError();
}

}  // namespace stereo
