// Sums of products of two pixel windows on the matrix cores, shared by the two NCC matchers.
//
// For an image row, the sum of L R over the P x P windows of 32 left pixels against those of 32 right
// pixels is one 32 x 32 product over the window's pixels, v_mfma_i32_32x32x32_i8 over
// Shape<P>::STEPS steps.  Pixels enter as signed bytes I - 128.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace stereo {
namespace winmm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Stages I - 128 of `rows` rows from y0 and dword columns [c0, c1) from x0 (clamped to the image;
// whole dwords are loaded, at any alignment, where none is cut) in rows of DW dwords.  1 << LOG
// threads take a row.  COPIES == 4: copy c, CS dwords on, holds the rows shifted by c bytes, so that
// the bytes from any column on start at a dword of copy (column & 3); with CS 8 mod 32 the 32
// lanes of a block (8 dwords of each copy) read 32 different banks.
template <int LOG, int DW, int COPIES, int CS>
__device__ __forceinline__ void stage_image(uint32_t* dst, const View& img, int x0, int y0, int rows, int c0, int c1)
{
    const int c = c0 + (threadIdx.x & ((1 << LOG) - 1)), x = x0 + 4 * c;
    const bool mine = c < c1;
    if (mine) {
        // a column is cut at the image's edge, or whole in all rows
        const bool whole = x >= 0 && x + 4 <= img.w;
        int xs[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) xs[j] = clampi(x + j, 0, img.w - 1);
#pragma unroll 5
        for (int r = threadIdx.x >> LOG; r < rows; r += 256 >> LOG) {
            const uint8_t* row = row_ptr<const uint8_t>(img, clampi(y0 + r, 0, img.h - 1));
            uint32_t w = 0;
            if (whole) __builtin_memcpy(&w, row + x, 4);
            else w = row[xs[0]] | (uint32_t)row[xs[1]] << 8 | (uint32_t)row[xs[2]] << 16 | (uint32_t)row[xs[3]] << 24;
            dst[r * DW + c] = w ^ 0x80808080u;
        }
    }
    if (COPIES == 1) return;
    __syncthreads();
    if (mine) {
        for (int r = threadIdx.x >> LOG; r < rows; r += 256 >> LOG) {
            // (the last column takes a neighbour that no window reaches)
            const uint32_t* q = dst + r * DW + c;
            const uint32_t lo = q[0], hi = q[1];
#pragma unroll
            for (int k = 1; k < COPIES; ++k) dst[k * CS + r * DW + c] = __builtin_amdgcn_alignbyte(hi, lo, k);
        }
    }
}

// How a P x P window lies in the K of v_mfma_i32_32x32x32_i8.  A window row is DWR dwords (the bytes
// past its P are zero in one of the two operands, so the other may hold anything there).  An
// operand reads ROWS = P + 1 image rows, so that either the first P or the last P of them are the
// window; HR rows are the operand of lanes 0 .. 31, the rest that of lanes 32 .. 63, each a run of
// dwords cut into steps of four.
template <int P>
struct Shape {
    static constexpr int DWR = (P + 3) / 4;
    static constexpr int HR = (P + 1) / 2;
    static constexpr int STEPS = (HR * DWR + 3) / 4;
    static constexpr int ROWS = 2 * HR;
    static constexpr uint32_t TAIL = P % 4 == 1 ? 0xFFu : 0xFFFFFFu;  // window bytes of a row's last dword
    static_assert(P % 2 == 1 && (DWR == 2 || DWR == 3), "odd windows of two or three dwords a row");
    // dword k of a lane's run: the first two dwords of each of its rows, then the third ones (a pair
    // is one read that lands as it lies in the operand); past the end it repeats the last one
    static constexpr bool past(int k) { return k >= DWR * HR; }
    static constexpr int row(int k) { return k < 2 * HR ? k / 2 : past(k) ? HR - 1 : k - 2 * HR; }
    static constexpr int dword(int k) { return k < 2 * HR ? k % 2 : DWR - 1; }
};

// One lane's operand from the four copies.  src: the dword of the copy that holds the lane's first
// column, in its half's first row, rows DW dwords apart.
template <int P, int DW>
__device__ __forceinline__ void load_operand(v4i (&v)[Shape<P>::STEPS], const uint32_t* src)
{
    using S = Shape<P>;
#pragma unroll
    for (int k = 0; k < 4 * S::STEPS; ++k) {
        if (k >= 2 * S::HR) {
            v[k / 4][k % 4] = (int)src[S::row(k) * DW + S::dword(k)];
        } else if (k % 2 == 0) {
            uint64_t two;
            __builtin_memcpy(&two, src + S::row(k) * DW, 8);
            v[k / 4][k % 4] = (int)(uint32_t)two;
            v[k / 4][k % 4 + 1] = (int)(uint32_t)(two >> 32);
        }
    }
}

// The same from a single copy, shifted here by the column's low bits, with zeros in the bytes past a
// row's P and past the run's end.
template <int P, int DW>
__device__ __forceinline__ void load_operand_shifted(v4i (&v)[Shape<P>::STEPS], const uint32_t* src, uint32_t shift)
{
    using S = Shape<P>;
#pragma unroll
    for (int k = 0; k < 4 * S::STEPS; ++k) {
        const uint32_t* q = src + S::row(k) * DW + S::dword(k);
        uint32_t d = __builtin_amdgcn_alignbyte(q[1], q[0], shift);
        if (S::dword(k) == S::DWR - 1) d &= S::TAIL;
        v[k / 4][k % 4] = S::past(k) ? 0 : (int)d;
    }
}

// Row r of the run kept where `keep` is all ones, zero where it is 0.
template <int P>
__device__ __forceinline__ void mask_row(v4i (&v)[Shape<P>::STEPS], int r, uint32_t keep)
{
#pragma unroll
    for (int k = 0; k < 4 * Shape<P>::STEPS; ++k)
        if (Shape<P>::row(k) == r && !Shape<P>::past(k)) v[k / 4][k % 4] &= (int)keep;
}

}  // namespace winmm
}  // namespace stereo
