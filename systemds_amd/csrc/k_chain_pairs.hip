// The multiply chain t(X) %*% (w * (X %*% v)) on blocks whose groups are all column pairs with two-byte codes, in one pass over the codes.
//
// A thread takes a row at a time: it looks up all of the row's tuples, 16 bytes each (from LDS where the dictionaries fit, else from global memory),
// sums their products with v, which are uniform, applies the row's weight and adds the result times the tuples to its sums of all columns.
// Tuples and sums of up to 25 pairs are 200 registers; the next row's codes come while a row is worked on. At the end a wave folds its lanes' sums (every exchange
// halves the values a lane holds), and the blocks hand theirs over (chain_hand_over): the call is this one launch.
// Bound: on short blocks the start and the hand-over, two round trips to memory each; with the dictionaries in LDS then LDS (a look-up of 16 bytes takes
// a wave 23 cycles) beside HBM, out of LDS the vector memory path, a cycle per lane and line. Three launches before (k_preagg, k_rmm_q1_short or its form
// for few rows, k_lmm_q1_short), which look every tuple up twice: 186,893 x 8 of 2665 tuples 22.4 -> 9.7 us, 162,880 x 16 of 2857 23.7 -> 13.6, 50,000 x 50 of 4096 23.7 -> 18.2,
// 400,000 x 40 of 300 37.5 -> 22.7, 8,000,000 x 6 of 2000 66 -> 34, 6,956,825 x 36 of 500 161 -> 104; of more than 8192 tuples (generic kernels) 2,500,000 x 18
// of 40,000 245 -> 85.
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include <algorithm>

namespace cla {

constexpr int CP_THREADS = 512, CP_WAVES = CP_THREADS / WAVE, CP_GROUPS = 25;

struct CpGroups { // columns and first tuple of a group; behind the last one column -1 and tuple 0
	int32_t c0[CP_GROUPS], c1[CP_GROUPS], at[CP_GROUPS];
};

__device__ __forceinline__ double cp_uniform(double x) {
	const long long b = __double_as_longlong(x);
	const uint32_t lo = (uint32_t) __builtin_amdgcn_readfirstlane((int) b), hi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (b >> 32));
	return __longlong_as_double((long long) ((uint64_t) hi << 32 | lo));
}

// Groups of the instantiation that a block of nG takes
static constexpr int cp_groups(int nG) { return nG <= 4 ? 4 : nG <= 8 ? 8 : nG <= 12 ? 12 : nG <= 16 ? 16 : nG <= 20 ? 20 : 25; }

template <int NG, bool LDS, bool OP>
__global__ __launch_bounds__(CP_THREADS, NG <= 8 ? 4 : 2) void k_chain_pairs(const uint8_t* __restrict__ arena, size_t arenaStride, int nG, const CpGroups P,
	const f64x2* __restrict__ dict, int nTuples, const double* __restrict__ v, const double* __restrict__ w, int minus, int64_t nRows,
	double* __restrict__ part, double* __restrict__ out, int nCols, unsigned* __restrict__ done, unsigned long long* __restrict__ nnz, double* __restrict__ hostOut,
	unsigned long long* __restrict__ hostCount) {
	extern __shared__ __attribute__((aligned(16))) double smem[]; // the dictionaries; at the end the sums
	constexpr int N2 = 2 * NG, FOLD = N2 <= 8 ? 8 : N2 <= 16 ? 16 : N2 <= 32 ? 32 : 64;
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	uint32_t code[NG];
	double wv = 0.0;
	auto load = [&](int64_t row) {
		const int64_t r = min(row, nRows - 1);
#pragma unroll
		for(int g = 0; g < NG; g++) code[g] = *(const uint16_t*) (arena + (size_t) min(g, nG - 1) * arenaStride + 2 * r);
		if(OP) wv = w[r];
	};
	const int64_t step = (int64_t) gridDim.x * CP_THREADS;
	int64_t row = (int64_t) blockIdx.x * CP_THREADS + tid;
	load(row);
	double vv[N2];
	bool bad = false;
#pragma unroll
	for(int g = 0; g < NG; g++) {
		const double a = v[max(P.c0[g], 0)], b = v[max(P.c1[g], 0)];
		vv[2 * g] = cp_uniform(g < nG ? a : 0.0);
		vv[2 * g + 1] = cp_uniform(g < nG ? b : 0.0);
		bad |= !isfinite(vv[2 * g]) || !isfinite(vv[2 * g + 1]);
	}
	if(LDS) {
		for(int i0 = tid; i0 < nTuples; i0 += 8 * CP_THREADS) {
			f64x2 d[8];
#pragma unroll
			for(int j = 0; j < 8; j++) d[j] = dict[min(i0 + j * CP_THREADS, nTuples - 1)];
#pragma unroll
			for(int j = 0; j < 8; j++)
				if(i0 + j * CP_THREADS < nTuples) ((f64x2*) smem)[i0 + j * CP_THREADS] = d[j];
		}
		__syncthreads();
	}
	f64x2 acc[NG];
#pragma unroll
	for(int g = 0; g < NG; g++) acc[g] = f64x2{0.0, 0.0};
	const char* const from = LDS ? (const char*) smem : (const char*) dict;
	for(int64_t r0 = (int64_t) blockIdx.x * CP_THREADS; r0 < nRows; r0 += step, row += step) {
		f64x2 x[NG];
#pragma unroll
		for(int g = 0; g < NG; g++) x[g] = *(const f64x2*) (from + (((uint32_t) P.at[g] + (g < nG ? code[g] : 0u)) << 4));
		const double wr = wv;
		__builtin_amdgcn_sched_barrier(0);
		load(row + step); // (behind the last row: that one's again)
		__builtin_amdgcn_sched_barrier(0);
		double s0 = 0.0, s1 = 0.0;
		if(!bad) {
#pragma unroll
			for(int g = 0; g < NG; g++) {
				s0 = __builtin_fma(x[g].x, vv[2 * g], s0);
				s1 = __builtin_fma(x[g].y, vv[2 * g + 1], s1);
			}
		}
		else { // a zero dictionary cell stays out of X %*% v whatever v holds (Dictionary.preaggValuesFromDense)
#pragma unroll
			for(int g = 0; g < NG; g++) {
				s0 = x[g].x == 0.0 ? s0 : __builtin_fma(x[g].x, vv[2 * g], s0);
				s1 = x[g].y == 0.0 ? s1 : __builtin_fma(x[g].y, vv[2 * g + 1], s1);
			}
		}
		double s = s0 + s1;
		if(OP) s = row_op(s, wr, minus);
		s = row < nRows ? s : 0.0;
#pragma unroll
		for(int g = 0; g < NG; g++) {
			acc[g].x = __builtin_fma(x[g].x, s, acc[g].x);
			acc[g].y = __builtin_fma(x[g].y, s, acc[g].y);
		}
	}
	// lane l of a wave: the sum of column l % FOLD
	double t[FOLD];
#pragma unroll
	for(int i = 0; i < FOLD; i++) t[i] = i < N2 ? (i & 1 ? acc[i / 2 < NG ? i / 2 : 0].y : acc[i / 2 < NG ? i / 2 : 0].x) : 0.0;
#pragma unroll
	for(int h = FOLD / 2; h >= 1; h /= 2) {
		const bool upper = (lane & h) != 0;
#pragma unroll
		for(int i = 0; i < h; i++) t[i] = (upper ? t[i + h] : t[i]) + __shfl_xor(upper ? t[i] : t[i + h], h);
	}
#pragma unroll
	for(int h = FOLD; h < 64; h *= 2) t[0] += __shfl_xor(t[0], h);
	__syncthreads(); // (the dictionaries have been read)
	double* const sums = smem + CP_WAVES * FOLD;
	if(lane < FOLD) smem[wave * FOLD + lane] = t[0];
	__syncthreads();
	if(tid < 2 * nG) {
		double s = 0.0;
		for(int i = 0; i < CP_WAVES; i++) s += smem[i * FOLD + tid];
		sums[tid] = s;
	}
	__syncthreads();
	chain_hand_over<CP_THREADS>(sums, 2 * nG, part, smem, [&](int i) { return i & 1 ? P.c1[i / 2] : P.c0[i / 2]; }, out, nCols, done, nnz, hostOut, hostCount);
}

struct CpLaunch {
	int ng = 0;       // groups of the instantiation
	bool inLds = false;
	unsigned grid = 0;
	size_t lds = 0;
};

// 1: the block is not of this kernel's shape
static int cp_shape(cla_block* b, CpLaunch& L) {
	const int nG = (int) b->groups.size();
	if(!b->opt.chainFused || b->dArena == nullptr || b->arenaWidth != 2 || nG == 0 || nG > CP_GROUPS || b->hasConst || b->dictNonFinite || b->nRows == 0 ||
		b->nRows >= (int64_t) 1 << 31 || (b->opt.rmmDisable & 3) || (b->opt.lmmDisable & 1))
		return 1;
	std::vector<char> seen((size_t) b->nCols, 0);
	for(const HostGroup& H : b->groups) {
		if(H.d.nColG != 2 || H.d.nVals < 1) return 1;
		for(int c : H.cols) {
			if(seen[c]) return 1;
			seen[c] = 1;
		}
	}
	L.ng = cp_groups(nG);
	const size_t room = (size_t) g_ldsPerBlock - 512, dict = (size_t) b->totalVals * 16, sums = (size_t) (CP_WAVES * 64 + 64) * 8;
	L.inLds = dict <= room;
	L.lds = std::max(L.inLds ? dict : 0, sums);
	const int64_t blocks = (b->nRows + CP_THREADS - 1) / CP_THREADS;
	L.grid = (unsigned) std::min<int64_t>(blocks, (int64_t) g_numCU * (L.ng <= 8 && L.lds <= (size_t) 78 * 1024 ? 2 : 1));
	// Dictionaries out of LDS: up to 12,500,000 look-ups, or always where the products have no tables in LDS either (us, two products / here, 4096 tuples: 50 columns
	// 300,000 rows 42 / 32, 600,000 52 / 46, 1,000,000 58 / 63; 18 columns 1,000,000 37 / 31, 1,500,000 42 / 42, 2,500,000 51 / 61; 10 columns 2,500,000 43 / 39; 9000 tuples
	// 50 columns 600,000 82 / 54, 2,500,000 199 / 162).
	if(!L.inLds && b->maxVals <= 8192 && b->nRows * nG > 12500000) return 1;
	return 0;
}

// The workspace of the chains to come, where the block's run in this kernel.
int prepare_chain_pairs(cla_block* b) {
	CpLaunch L;
	return cp_shape(b, L) ? 0 : ensure_chain(b, (size_t) L.grid * 2 * b->groups.size());
}

// Returns 1 when the block is not eligible (the chain then runs as two products), 0 when the chain has been queued.
int launch_chain_pairs(cla_block* b, const double* dV, const double* dW, int ctype, double* dOut, unsigned long long* dNnz, ChainHost& host) {
	CpLaunch L;
	if(cp_shape(b, L)) return 1;
	const int nG = (int) b->groups.size();
	int rc = ensure_chain(b, (size_t) L.grid * 2 * nG);
	if(rc) return rc;
	CpGroups P;
	for(int g = 0; g < CP_GROUPS; g++) {
		P.c0[g] = g < nG ? b->groups[g].cols[0] : -1;
		P.c1[g] = g < nG ? b->groups[g].cols[1] : -1;
		P.at[g] = g < nG ? b->groups[g].d.tblOff : 0;
	}
	clear_stats(b);
	Prof pf(b, "k_chain_pairs", L.grid, CP_THREADS, (long) L.lds, (double) b->nRows * (2 * nG + (ctype ? 8 : 0)) + (double) b->totalVals * 16);
	auto go = [&](auto kern) {
		CLA_HIP(allow_full_lds((const void*) kern));
		hipLaunchKernelGGL(kern, dim3(L.grid), dim3(CP_THREADS), L.lds, b->stream, b->dArena, b->arenaStride, nG, P, (const f64x2*) b->dAllDict, b->totalVals, dV, dW,
			ctype == 2 ? 1 : 0, b->nRows, b->dChain, dOut, b->nCols, b->lmm_ticket(), dNnz, host.out, host.count);
		return 0;
	};
#define CP_CASE(N)                                                                                                                \
	case N:                                                                                                                       \
		if(L.inLds) rc = ctype ? go(k_chain_pairs<N, true, true>) : go(k_chain_pairs<N, true, false>);                            \
		else rc = ctype ? go(k_chain_pairs<N, false, true>) : go(k_chain_pairs<N, false, false>);                                 \
		break;
	switch(L.ng) { CP_CASE(4) CP_CASE(8) CP_CASE(12) CP_CASE(16) CP_CASE(20) CP_CASE(25) }
#undef CP_CASE
	if(rc) return rc;
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
