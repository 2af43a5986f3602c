// The multiply chain t(X) %*% (w * (X %*% v)) on blocks whose groups are all single-column DDC with byte codes, in one pass over
// the codes: a row's sum and that sum times the row's values need the same lookups.
//
// A wave takes 64 rows and all column blocks of 16 groups. Lane (k, c), k = lane / 16, c = lane % 16, reads 16 codes of group c of
// a column block (rows 16 k .. 16 k + 15 of the 64) with one 16-byte load and looks them up in the dictionaries in LDS
// ([code][16 groups]: the 16 lanes of a quarter read 16 different banks whatever their codes), 4 rows of each quarter per step,
// all columns:
//   X %*% v        the lane's part of 4 row sums (multiply-adds with its own values of v), then a fold over the 16 lanes of the
//                  quarter (two exchanges that halve the sums a lane holds, two that add all of it): lane c ends up with the sum of
//                  row c % 4, and the lanes whose own rows the step's are apply their weights;
//   t(X) %*% tmp   the sums go back over the quarter lane by lane (row_newbcast) and meet the looked-up values, which are still in
//                  registers; the lane's sums of its columns stay in registers over all rows of the block.
// A unit's 64 rows are a chain of additions of their own, as in k_lmm_u8_dot.
//
// The blocks hand their sums over in a workspace, a row each, and the last one to arrive adds them up in block order, writes the
// output and counts its non-zeros: the call is this one launch, without a fill in front of it.
//
// Bound: vector issue (about 410 instructions of 4 cycles per 64 rows at 4 column blocks; the fold over the lanes costs the same
// whatever the number of columns): 81 % of the CUs' busy cycles on 8,000,001 x 54, LDS 50 (half of it bank conflicts), the vector memory address
// unit 40, next to HBM (8,000,001 x 100: 3.7 TB/s). On small blocks the start, the copy of the dictionaries and the hand-over: vector issue 34 % on
// 250,007 x 54, nothing else above. Why not rows per thread as in k_rmm_q1_u8: the second product would add a value per thread, group
// and pass through LDS, and sums over 100 columns do not fit a thread's registers. Measured (before: k_rmm_q1_u8, k_lmm_u8_dot or
// k_lmm_u8_vec and a fill): 1,000 x 5 5.8 us (16.5), 250,007 x 54 13.8 (36), 1,000,003 x 80 29 (62), 8,000,001 x 48 108 (202), 8,000,001 x
// 100 216 (334), 8,000,001 x 10 49 (82); nowhere slower, so every block that fits takes it.
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include <algorithm>

namespace cla {

using std::integral_constant;
constexpr int CH_THREADS = 512;
constexpr int CH_WAVES = CH_THREADS / WAVE;

// x of lane T of the lane's row of 16
template <int T>
__device__ __forceinline__ double ch_bcast(double x) {
	return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(x), 0x150 + T, 0xf, 0xf, true)); // row_newbcast:T, both halves at once
}
// x of another lane of the row of 16 (every lane has one)
template <int CTRL>
__device__ __forceinline__ double ch_dpp(double x) {
	int p[2];
	__builtin_memcpy(p, &x, 8);
	p[0] = __builtin_amdgcn_mov_dpp(p[0], CTRL, 0xf, 0xf, true);
	p[1] = __builtin_amdgcn_mov_dpp(p[1], CTRL, 0xf, 0xf, true);
	double r;
	__builtin_memcpy(&r, p, 8);
	return r;
}

template <int NCB, bool OP>
__global__ __launch_bounds__(CH_THREADS, NCB <= 3 ? 4 : 2) void k_chain_u8(const uint8_t* __restrict__ arena, size_t arenaStride, int nGroups,
	const double* __restrict__ dictT, int nVals, const int32_t* __restrict__ col0, const double* __restrict__ v, const double* __restrict__ w,
	int minus, int64_t nRows, double* __restrict__ part, double* __restrict__ out, int nCols, unsigned* __restrict__ done,
	unsigned long long* __restrict__ nnz, double* __restrict__ hostOut, unsigned long long* __restrict__ hostCount) {
	extern __shared__ __attribute__((aligned(16))) double smem[]; // the dictionaries; at the end the sums
	__shared__ int lastS;
	__shared__ int cntS[CH_WAVES];
	constexpr int NC = NCB * 16;
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int c = lane & 15, k = lane >> 4;
	const int64_t nUnits = nRows / WAVE; // whole ones
	const int64_t u0 = nUnits * blockIdx.x / gridDim.x, u1 = nUnits * (blockIdx.x + 1) / gridDim.x;

	const uint8_t* codeBase[NCB]; // this lane's stream of every column block
	double vv[NCB];               // v of its columns; 0 where the last column block has none
	bool bad = false;
#pragma unroll
	for(int cb = 0; cb < NCB; cb++) {
		const int g = cb * 16 + c;
		codeBase[cb] = arena + (size_t) min(g, nGroups - 1) * arenaStride + 16 * k;
	}
	const double* const wBase = OP ? w + lane : nullptr;
	u32x4 codes[NCB], next[NCB];
	double wv = 0.0, wn = 0.0;
	auto load = [&](u32x4 (&dst)[NCB], double& dw, int64_t u) {
#pragma unroll
		for(int cb = 0; cb < NCB; cb++) dst[cb] = *(const u32x4*) (codeBase[cb] + u * WAVE);
		if(OP) dw = wBase[u * WAVE];
	};
	int64_t u = u0 + wave;
	if(u < u1) load(codes, wv, u);
#pragma unroll
	for(int cb = 0; cb < NCB; cb++) {
		const int g = cb * 16 + c;
		const double x = v[col0[min(g, nGroups - 1)]];
		vv[cb] = g < nGroups ? x : 0.0;
		bad |= !isfinite(vv[cb]);
	}
	{
		const f64x2* src = (const f64x2*) dictT;
		const int n = NCB * nVals * 8;
		for(int i0 = tid; i0 < n; i0 += 8 * CH_THREADS) {
			f64x2 d[8];
#pragma unroll
			for(int j = 0; j < 8; j++) d[j] = src[min(i0 + j * CH_THREADS, n - 1)];
#pragma unroll
			for(int j = 0; j < 8; j++)
				if(i0 + j * CH_THREADS < n) ((f64x2*) smem)[i0 + j * CH_THREADS] = d[j];
		}
	}
	// a zero dictionary cell stays out of X %*% v whatever v holds (Dictionary.preaggValuesFromDense)
	const bool careful = __syncthreads_or(bad) != 0;

	const char* const tb = (const char*) smem + c * 8;
	const int cbBytes = nVals * 128;
	const bool b0 = (lane & 1) != 0, b1 = (lane & 2) != 0;
	double acc[NCB], tot[NCB]; // of a unit's rows, of the units in front of it
#pragma unroll
	for(int cb = 0; cb < NCB; cb++) acc[cb] = tot[cb] = 0.0;
	double d[2][NCB][4]; // rows 4 q .. 4 q + 3 of every quarter, those of the step behind requested before a step is worked on
	auto look = [&](auto qTag, const u32x4 (&cv)[NCB]) __attribute__((always_inline)) {
		constexpr int q = decltype(qTag)::value;
#pragma unroll
		for(int cb = 0; cb < NCB; cb++) {
			const char* t0 = tb + cb * cbBytes;
#pragma unroll
			for(int t = 0; t < 4; t++) d[q & 1][cb][t] = *(const double*) (t0 + (((cv[cb][q] >> (8 * t)) & 0xffu) << 7));
		}
	};
	// live: false for a lane whose row (16 k + c of the unit) is behind the last one
	auto work = [&](auto qTag, auto cTag, bool live) __attribute__((always_inline)) {
		constexpr int q = decltype(qTag)::value;
		const double (&dq)[NCB][4] = d[q & 1];
		double p[4];
#pragma unroll
		for(int t = 0; t < 4; t++) {
			p[t] = decltype(cTag)::value && dq[0][t] == 0.0 ? 0.0 : dq[0][t] * vv[0];
#pragma unroll
			for(int cb = 1; cb < NCB; cb++) {
				const double x = __builtin_fma(dq[cb][t], vv[cb], p[t]);
				p[t] = decltype(cTag)::value && dq[cb][t] == 0.0 ? p[t] : x;
			}
		}
		double x2[2]; // (quad_perm: lane ^ 1, lane ^ 2)
#pragma unroll
		for(int j = 0; j < 2; j++) x2[j] = (b0 ? p[2 * j + 1] : p[2 * j]) + ch_dpp<0xB1>(b0 ? p[2 * j] : p[2 * j + 1]);
		double s = (b1 ? x2[1] : x2[0]) + ch_dpp<0x4E>(b1 ? x2[0] : x2[1]); // (of row c % 4 of the step, over the lane's four)
		s += ch_dpp<0x124>(s); // row_ror:4
		s += ch_dpp<0x128>(s); // row_ror:8
		if(OP) s = row_op(s, wv, minus); // (lanes 4 q .. 4 q + 3 hold their own rows' sums, the others' are not used)
		s = live ? s : 0.0;
		auto add = [&](auto tTag) __attribute__((always_inline)) {
			constexpr int t = decltype(tTag)::value;
			const double st = ch_bcast<4 * q + t>(s);
#pragma unroll
			for(int cb = 0; cb < NCB; cb++) acc[cb] = __builtin_fma(dq[cb][t], st, acc[cb]);
		};
		add(integral_constant<int, 0>()); add(integral_constant<int, 1>()); add(integral_constant<int, 2>()); add(integral_constant<int, 3>());
	};
	auto next_unit = [&]() __attribute__((always_inline)) {
#pragma unroll
		for(int cb = 0; cb < NCB; cb++) {
			tot[cb] += acc[cb];
			acc[cb] = 0.0;
		}
	};
	// (two copies of the loop: one with the test in it takes 50 registers more per column block)
	auto rows = [&](auto cTag) __attribute__((always_inline)) {
		if(u < u1) look(integral_constant<int, 0>(), codes);
		for(; u < u1; u += CH_WAVES) {
			load(next, wn, u + CH_WAVES < u1 ? u + CH_WAVES : u); // (the last turn requests its own rows again)
			auto step = [&](auto qTag) __attribute__((always_inline)) {
				constexpr int q = decltype(qTag)::value;
				if constexpr(q < 3) look(integral_constant<int, q + 1>(), codes);
				else look(integral_constant<int, 0>(), next);
				__builtin_amdgcn_sched_barrier(0);
				work(qTag, cTag, true);
				__builtin_amdgcn_sched_barrier(0);
			};
			step(integral_constant<int, 0>()); step(integral_constant<int, 1>()); step(integral_constant<int, 2>()); step(integral_constant<int, 3>());
#pragma unroll
			for(int cb = 0; cb < NCB; cb++) codes[cb] = next[cb];
			wv = wn;
			next_unit();
		}
		// the rows behind the whole units (outside the loop: a load under a condition makes the compiler wait for all loads in flight).
		// A stream's stride is a multiple of 256 bytes and what lies behind its last row is code 0, so only the rows' sums are cut.
		if(blockIdx.x == gridDim.x - 1 && wave == CH_WAVES - 1 && nUnits * WAVE < nRows) {
			const bool live = lane < (int) (nRows - nUnits * WAVE);
#pragma unroll
			for(int cb = 0; cb < NCB; cb++) codes[cb] = *(const u32x4*) (codeBase[cb] + nUnits * WAVE);
			if(OP) wv = live ? wBase[nUnits * WAVE] : 0.0;
			auto step = [&](auto qTag) __attribute__((always_inline)) {
				look(qTag, codes);
				__builtin_amdgcn_sched_barrier(0);
				work(qTag, cTag, live);
				__builtin_amdgcn_sched_barrier(0);
			};
			step(integral_constant<int, 0>()); step(integral_constant<int, 1>()); step(integral_constant<int, 2>()); step(integral_constant<int, 3>());
			next_unit();
		}
	};
	if(careful) rows(std::true_type());
	else rows(std::false_type());

	// the block's sums: 4 quarters x 8 waves per column
	__syncthreads();
#pragma unroll
	for(int cb = 0; cb < NCB; cb++) smem[(wave * 4 + k) * NC + cb * 16 + c] = tot[cb];
	__syncthreads();
	if(tid < NC) {
		double s = 0.0;
#pragma unroll
		for(int i = 0; i < CH_WAVES * 4; i++) s += smem[i * NC + tid];
		// (exchanged, not stored: performed at device scope, past the caches that the chip's parts do not share, see lmm_tail)
		(void) __hip_atomic_exchange((unsigned long long*) part + (size_t) blockIdx.x * NC + tid, (unsigned long long) __double_as_longlong(s), __ATOMIC_RELAXED,
			__HIP_MEMORY_SCOPE_AGENT);
	}
	asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
	__syncthreads();
	if(tid == 0) lastS = last_block(done, gridDim.x);
	__syncthreads();
	if(!lastS) return;
	// the last block: the others' sums in block order, a share of the blocks per group of NC threads
	constexpr int NP = CH_THREADS / NC;
	const int col = tid % NC, share = tid / NC;
	double s = 0.0;
	if(share < NP) {
		for(int b0i = share; b0i < (int) gridDim.x; b0i += 8 * NP) {
			unsigned long long r[8];
#pragma unroll
			for(int j = 0; j < 8; j++) {
				const int bj = b0i + j * NP;
				r[j] = bj < (int) gridDim.x
					? __hip_atomic_load((const unsigned long long*) part + (size_t) bj * NC + col, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
			}
#pragma unroll
			for(int j = 0; j < 8; j++) s += __longlong_as_double((long long) r[j]);
		}
		smem[share * NC + col] = s;
	}
	if(nCols > nGroups) // columns that no group covers
		for(int i = tid; i < nCols; i += CH_THREADS) {
			out[i] = 0.0;
			if(hostOut != nullptr) hostOut[i] = 0.0;
		}
	nnz_clear(nnz);
	__syncthreads();
	int nz = 0;
	if(tid < nGroups) {
		s = smem[tid];
#pragma unroll
		for(int i = 1; i < NP; i++) s += smem[i * NC + tid];
		out[col0[tid]] = s;
		if(hostOut != nullptr) hostOut[col0[tid]] = s;
		nz = s != 0.0; // (a NaN counts, a negative zero does not)
	}
	nz = wave_sum_i32(nz);
	if(lane == 0) cntS[wave] = nz;
	__syncthreads();
	if(tid == 0) {
		int n = 0;
		for(int i = 0; i < CH_WAVES; i++) n += cntS[i];
		*nnz = (unsigned long long) n;
		if(hostCount != nullptr) *hostCount = (unsigned long long) n;
	}
	clear_tickets(done);
}

// What a launch on a block takes.
struct ChainLaunch {
	decltype(&k_chain_u8<1, false>) kern = nullptr; // nullptr: the block is not eligible
	unsigned grid = 0;
	size_t lds = 0, wsDoubles = 0;
};

static int chain_shape(cla_block* b, bool op, ChainLaunch& L) {
	const int nG = (int) b->groups.size();
	// what X %*% v and t(y) %*% X of the block would run on the byte-code kernels, with nothing to add behind them; a column per group
	if(b->dDictPad == nullptr || !b->u8ColsDistinct || b->hasConst || b->dictNonFinite || b->nRows == 0 || (b->opt.rmmDisable & 3) || (b->opt.lmmDisable & 1) ||
		!b->opt.chainFused)
		return 0;
	const int nCb = (nG + 15) / 16;
	L.lds = std::max((size_t) nCb * b->maxVals * 128, (size_t) CH_WAVES * 4 * nCb * 16 * 8);
	if(L.lds > (size_t) g_ldsPerBlock) return 0; // (before the kernel is asked: the first question of a process loads its code, 1.1 ms)
	decltype(&k_chain_u8<1, false>) kern = nullptr;
#define CH_CASE(N) case N: kern = op ? k_chain_u8<N, true> : k_chain_u8<N, false>; break;
	switch(nCb) { CH_CASE(1) CH_CASE(2) CH_CASE(3) CH_CASE(4) CH_CASE(5) CH_CASE(6) CH_CASE(7) default: return 0; }
#undef CH_CASE
	size_t room = 0;
	CLA_HIP(max_dynamic_lds((const void*) kern, room));
	if(L.lds > room) return 0;
	const int64_t nUnits = std::max<int64_t>(b->nRows / WAVE, 1);
	const int perCU = nCb <= 3 && L.lds <= (size_t) 78 * 1024 ? 2 : 1;
	L.grid = (unsigned) std::min<int64_t>((nUnits + CH_WAVES - 1) / CH_WAVES, (int64_t) g_numCU * perCU);
	L.wsDoubles = (size_t) L.grid * nCb * 16;
	L.kern = kern;
	return 0;
}

// The workspace of the chains to come, where the block's run in this kernel.
int prepare_chain_u8(cla_block* b) {
	for(bool op : {false, true}) {
		ChainLaunch L;
		int rc = chain_shape(b, op, L);
		if(rc == 0 && L.kern != nullptr) rc = ensure_chain(b, L.wsDoubles);
		if(rc) return rc;
	}
	return 0;
}

// Returns 1 when the block is not eligible (the chain then runs as two products), 0 when the chain has been queued.
int launch_chain_u8(cla_block* b, const double* dV, const double* dW, int ctype, double* dOut, unsigned long long* dNnz, ChainHost& host) {
	const int nG = (int) b->groups.size();
	const int64_t nRows = b->nRows;
	ChainLaunch L;
	int rc = chain_shape(b, ctype != 0, L);
	if(rc || L.kern == nullptr) return rc ? rc : 1;
	// (not the tables of the products: those of a captured one may not move)
	if((rc = ensure_chain(b, L.wsDoubles))) return rc;
	const int32_t* dCol0 = (const int32_t*) (b->dDictPad + (size_t) nG * 256);
	clear_stats(b);
	const double algo = (double) nRows * nG + (dW != nullptr ? (double) nRows * 8 : 0.0);
	Prof pf(b, "k_chain_u8", L.grid, CH_THREADS, (long) L.lds, algo);
	hipLaunchKernelGGL(L.kern, dim3(L.grid), dim3(CH_THREADS), L.lds, b->stream, b->dArena, b->arenaStride, nG, b->dDictPad + b->dictTOff, b->maxVals, dCol0,
		dV, dW, ctype == 2 ? 1 : 0, nRows, b->dChain, dOut, b->nCols, b->lmm_ticket(), dNnz, host.out, host.count);
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
