// What goes in front of the wide right multiply's kernels (k_rmm_mfma.hip, k_rmm_digits.hip): B in k_rmm_mfma's layout, the constants' row, the counter.
#pragma once
#include "cla_device.hpp"

namespace cla {

// B slab in LDS: row k at k * MF_BK, inside it the 16 values of lane column j (accumulators jg = 0..15)
// at j * MF_BJ: the 16 distinct 16-byte pieces of a wave's read fall on 16 distinct
// bank quads (row stride 16 banks, j stride 36 banks)
constexpr int MF_BJ = 18;
constexpr int MF_BK = 4 * MF_BJ;

constexpr int MF_BL_THREADS = 256;
constexpr int MF_BL_ROWS = MF_BL_THREADS / 128; // rows of B per block

struct MfPrep {
	const double* B;
	const int32_t* rowCol;      // decoded column per row of the list, -1: padding
	double* Bl;
	const double* constV;       // nullptr: no constants
	double* constRow;           // constV x B
	unsigned long long* nnz;    // cleared (nullptr: a pass behind the first)
	int q, n0, nRowCol, nCols;
	int blocks() const { return (nRowCol + MF_BL_ROWS - 1) / MF_BL_ROWS + (constV != nullptr || nnz != nullptr ? 1 : 0); }
};

// B in the slab layout: row r of the list (decoded column rowCol[r], -1 = padding) at r * MF_BK,
// output column n0 + 8 (jg / 2) + 2 j + jg % 2 at j * MF_BJ + jg. The block behind the last row makes the constants' row of the pass, rounded
// and skipped like the tables' (k_preagg), and clears the counter. Bound: one launch; before, k_preagg made tables in front that nobody read and k_mfma_blayout was a
// launch of its own beside k_rmm_digits_b: 2,914 x 10 by 31 14.3 -> 12.1 us, 500 x 100 by 64 38 -> 25, 150,000 x 100 by 64 69 -> 55, two-byte codes 50,000 x 50 of 4000 tuples by 16 71 -> 63.
__device__ __forceinline__ void mf_prep(const MfPrep& P, int block) {
	const int t = threadIdx.x & 127, r = block * MF_BL_ROWS + (threadIdx.x >> 7);
	if(block * MF_BL_ROWS < P.nRowCol) {
		if(t >= MF_BK || r >= P.nRowCol) return;
		const int j = t / MF_BJ, jg = t - j * MF_BJ, col = P.n0 + 8 * (jg >> 1) + 2 * j + (jg & 1), gc = P.rowCol[r];
		P.Bl[(size_t) r * MF_BK + t] = (jg < 16 && gc >= 0 && col < P.q) ? P.B[(size_t) gc * P.q + col] : 0.0;
		return;
	}
	if(P.nnz != nullptr) nnz_clear(P.nnz);
	const int col = P.n0 + (int) threadIdx.x;
	if(P.constV == nullptr || threadIdx.x >= 64 || col >= P.q) return;
	double acc = 0.0;
#pragma unroll 8
	for(int c = 0; c < P.nCols; c++) {
		const double a = P.constV[c], x = __dadd_rn(acc, __dmul_rn(a, P.B[(size_t) c * P.q + col]));
		acc = a != 0.0 ? x : acc;
	}
	P.constRow[col] = acc;
}

} // namespace cla
