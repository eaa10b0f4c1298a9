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
// ncc_mm_kernel for the layout.
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
// 256 disparities, 11 x 11: 411 -> 212 us.  Tiles of 4 rows: with 8 the 2025 workgroups end in a
// part-filled round (218 us).
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

void ncc_grid(int W, int H, int D, int* ntx, int* rb, int* nseg, int* seg_len)
{
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

hipError_t launch_ncc(int ww, const NccParams& p, hipStream_t s)
{
    if (p.rb < 1 || p.rb > ncc::RBMAX || p.nseg < 1 || p.seg_len % 32 || p.D > 256 || !p.rkey) return hipErrorInvalidValue;
    dim3 grid(p.ntx * ((p.H + p.rb - 1) / p.rb) * p.nseg);
#define NCC_LAUNCH(P)                                                                          \
    if (p.bins)                                                                                   \
        hipLaunchKernelGGL((ncc::ncc_mm_kernel<P, true>), grid, dim3(256), 0, s, p);               \
    else                                                                                          \
        hipLaunchKernelGGL((ncc::ncc_mm_kernel<P, false>), grid, dim3(256), 0, s, p);              \
    break
    switch (ww) {
    case 11: NCC_LAUNCH(11);
    case 9: NCC_LAUNCH(9);
    case 7: NCC_LAUNCH(7);
    default: NCC_LAUNCH(5);
    }
#undef NCC_LAUNCH
    return hipGetLastError();
}

hipError_t launch_ncc_score(const NccScoreParams& f, hipStream_t s)
{
    dim3 grid((f.W + 63) / 64, (f.H + 3) / 4);
    hipLaunchKernelGGL(ncc::ncc_score_kernel, grid, dim3(256), 0, s, f);
    return hipGetLastError();
}

}  // namespace stereo
