// Blocks of a few "varying" columns (one value per row behind a plain stream) next to run-length columns: the plan that the
// kernels without tiles share (k_gram_direct.hip, k_lmm_direct.hip).
#pragma once
#include "cla_runs.hpp"

namespace cla {

// A varying column as the Gram kernel reads it.
struct GdrCol {            // 32 bytes
	const uint8_t* src;    // its codes; a dense column: codes 0, n, 2 n .. 7 n of eight rows in the wave's copy of its group, n columns wide
	int32_t bpr;           // bytes per row of src (1 or 2); 0: a dense column
	int32_t base8;         // bytes from the LDS base: the column's values by tuple; a dense column: its place in a row, in bytes
	int32_t dense0;        // -1: behind codes; else the dense columns in front of its group's
	int32_t width;         // a dense column: of its group
	int32_t col;           // column of the matrix
	int32_t pad;
};
struct GdrDense {          // a group of dense columns, fetched as it lies
	const uint8_t* src;
	int32_t bpr;           // bytes per row
	int32_t before;        // columns of the groups in front
};
struct GdrArgs {
	const GdrCol* cols;
	const double* vals;    // values of the code columns by tuple, constants added: the head of LDS as it is
	const RunCol* runs;
	const GdrDense* dense;
	int nV, nR, nDense;        // varying columns, run-length columns, dense groups
	int valDoubles;        // even
	int64_t nRows;
	double* out;
	int nCols;
	double* acc;               // the call's only kernel: the blocks add here and the last one writes out (gram_tail)
	unsigned* done;            // its ticket counter (nullptr: the blocks add into out, the caller fills and finishes)
	unsigned long long* nnz;
};

// A varying column as the left multiply reads it: straight from its stream.
struct LdCol {
	const uint8_t* src;    // its code (or value) of row 0
	int32_t stride;        // bytes per row; 0: a filler
	int32_t base8;         // bytes from the LDS base: values by tuple
	uint32_t mask;         // of a code; 0: a filler, which looks a zero up
	int32_t col;           // column of the matrix, -1: a filler
};

struct LdCols { LdCol c[12]; };

struct GdrPlan {
	int rc = 1;            // 0 usable, 1 the block does not qualify
	void* dImg = nullptr;
	int64_t bytes = 0;
	size_t lds = 0;        // of k_tsmm_direct, which these belong to as well: quads of varying columns, pieces of dense values per lane, waves per block
	int quads = 0, densePieces = 0, waves = 0;
	bool gram = false;     // whether that kernel holds them
	GdrArgs A;
	int spread = -1;       // 1: a varying column next to run-length columns spans too many magnitudes (GDR_SPREAD); -1: not looked at yet
	bool codeSpread = false; // the same of the columns behind codes, from their dictionaries
	LdCols ld;             // ldNC code columns (fillers behind the real ones), ldND dense ones; ldNC == 0: no such form
	int ldNC = 0, ldND = 0;
	int64_t runEnds = 0;   // of the run-length groups that are followed by run (inside the matrix)
};

// A block's copy of the values into LDS: 16-byte pieces, several requested together (one dictionary after the other, each a
// round trip to memory, took 15 us of a call).
template <int THREADS>
__device__ __forceinline__ void gdr_copy_vals(double* smem, const double* __restrict__ vals, int valDoubles) {
	const f64x2* src = (const f64x2*) vals;
	const int n = valDoubles / 2;
	for(int i0 = threadIdx.x; i0 < n; i0 += 8 * THREADS) {
		f64x2 d[8];
#pragma unroll
		for(int j = 0; j < 8; j++) d[j] = src[min(i0 + j * THREADS, n - 1)];
#pragma unroll
		for(int j = 0; j < 8; j++)
			if(i0 + j * THREADS < n) ((f64x2*) smem)[i0 + j * THREADS] = d[j];
	}
}

// The value of lane ^ 1, ^ 2 or ^ 4 on the vector unit.
template <int CTRL>
__device__ __forceinline__ double gdr_dpp(double v) {
	int p[2];
	__builtin_memcpy(p, &v, 8);
	p[0] = __builtin_amdgcn_update_dpp(0, p[0], CTRL, 0xf, 0xf, false);
	p[1] = __builtin_amdgcn_update_dpp(0, p[1], CTRL, 0xf, 0xf, false);
	double r;
	__builtin_memcpy(&r, p, 8);
	return r;
}
__device__ __forceinline__ double gdr_xchg1(double v) { return gdr_dpp<0xB1>(v); }
__device__ __forceinline__ double gdr_xchg2(double v) { return gdr_dpp<0x4E>(v); }
__device__ __forceinline__ double gdr_xchg4(double v) { // banks 0 and 2 from the bank above, 1 and 3 from the bank below
	int p[2];
	__builtin_memcpy(p, &v, 8);
#pragma unroll
	for(int h = 0; h < 2; h++) {
		int r = __builtin_amdgcn_update_dpp(0, p[h], 0x104, 0xf, 0x5, false); // row_shl:4
		p[h] = __builtin_amdgcn_update_dpp(r, p[h], 0x114, 0xf, 0xA, false);   // row_shr:4
	}
	double r;
	__builtin_memcpy(&r, p, 8);
	return r;
}

// The block's plan, built on first use; P.rc says whether it qualifies. Negative: an error.
int gdr_plan(cla_block* b, const GdrPlan*& P);

} // namespace cla
