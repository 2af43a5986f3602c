// Products with one vector on blocks whose groups are all DDC with two-byte codes.
//
//   k_rmm_q1_short   X %*% v: the tables dict x v of two groups at a time in LDS
//   k_rmm_q1_short_rows  the same on few rows, straight from global memory
//   k_lmm_q1_short   t(y) %*% X: the dictionaries of a few groups in LDS, every looked-up tuple times y into registers
//
// A lookup straight in global memory costs the vector memory path a cycle per lane and line (62.9 M lookups: 76 us for 8
// bytes, 99 us for tuples of 16 bytes, one group at a time; 170 us with several groups per instruction); the whole kernels with
// lookups in LDS take 40 and 39 us on as many. So a block holds what its lookups need in LDS: the right multiply owns rows and walks the groups (its
// sums stay in registers), the left multiply owns groups and walks the rows (its sums are one cell per column).
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include <algorithm>

namespace cla {

constexpr int SV_THREADS = 1024;
constexpr int SV_WAVES = SV_THREADS / WAVE;
constexpr int SV_BUF = 8192; // table entries of a buffer: 8 per thread on their way from global memory, two buffers of 64 KiB
constexpr int SV_NU = 4;     // most units of 256 rows per wave (128 registers per thread: 8 for the sums of a unit, 4 for its codes)

typedef double f64x2_sv __attribute__((ext_vector_type(2), aligned(8)));

// X %*% v: a block owns a share of the rows, lane l of a wave 4 consecutive rows of each of its NU units of 256. For every
// pair of groups (GS = 1: every group) the tables come through registers into the LDS buffer that the pair before does not
// use, while that pair is looked up. Groups are added in list order, as the reference does.
// Bound: the vector memory path (its address unit is busy 71 % of the time at 2,500,009 x 50: 8 bytes of codes per lane and group,
// and all tables once per 16,384 rows at most), LDS 39 %, vector issue 31 %; about 1 us per group below that.
// 2,500,009 x 50 (25 groups of 4096 tuples) 191 -> 44 us (a thread per row and group before), of 1000 tuples 101 -> 43
// (slabs of eight tables, reloaded by every block of 4096 rows); 8,000,000 x 50 703 -> 123.
template <int NU>
__global__ __launch_bounds__(SV_THREADS) void k_rmm_q1_short(const uint8_t* __restrict__ arena, size_t arenaStride, int nGroups, int gs,
	const int32_t* __restrict__ tblOff, const double* __restrict__ T, int constIdx, double* __restrict__ out, int64_t nRows,
	unsigned long long* __restrict__ nnz, const RowOp op) {
	extern __shared__ double tbl[]; // two buffers
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int64_t n4 = (nRows + 3) / 4;
	const int64_t s0 = n4 * blockIdx.x / gridDim.x, s1 = n4 * (blockIdx.x + 1) / gridDim.x;
	const int64_t w0 = s0 + (s1 - s0) * wave / SV_WAVES, w1 = s0 + (s1 - s0) * (wave + 1) / SV_WAVES;
	int64_t at[NU]; // quarter rows of this lane (behind the wave's last one: that one again, not stored)
#pragma unroll
	for(int j = 0; j < NU; j++) at[j] = min(min(w0 + j * 64 + lane, max(w1 - 1, w0)), n4 - 1);
	double acc[NU][4];
#pragma unroll
	for(int j = 0; j < NU; j++)
#pragma unroll
		for(int i = 0; i < 4; i++) acc[j][i] = 0.0;

	const int nSlabs = (nGroups + gs - 1) / gs;
	u32x2 codes[2][2][NU];
	double stage[8];
	auto load_tables = [&](int s) {
		const int e0 = tblOff[s * gs], n = tblOff[min(s * gs + gs, nGroups)] - e0;
#pragma unroll
		for(int i = 0; i < 8; i++) stage[i] = T[e0 + min(tid + i * SV_THREADS, max(n - 1, 0))];
	};
	auto load_codes = [&](u32x2 (&c)[2][NU], int s) {
#pragma unroll
		for(int g = 0; g < 2; g++) {
			const uint8_t* base = arena + (size_t) min(s * gs + min(g, gs - 1), nGroups - 1) * arenaStride;
#pragma unroll
			for(int j = 0; j < NU; j++) c[g][j] = *(const u32x2*) (base + at[j] * 8);
		}
	};
	auto write_tables = [&](int buf) {
#pragma unroll
		for(int i = 0; i < 8; i++) tbl[buf * SV_BUF + tid + i * SV_THREADS] = stage[i];
	};
	auto add = [&](const u32x2 (&c)[NU], const double* t) {
#pragma unroll
		for(int j = 0; j < NU; j++) {
			acc[j][0] += t[c[j].x & 0xffffu]; acc[j][1] += t[c[j].x >> 16];
			acc[j][2] += t[c[j].y & 0xffffu]; acc[j][3] += t[c[j].y >> 16];
		}
	};
	load_tables(0);
	load_codes(codes[0], 0);
	write_tables(0);
	lds_barrier();
	auto step = [&](int s, auto parity) {
		constexpr int P = decltype(parity)::value;
		const int next = min(s + 1, nSlabs - 1); // (the last slab requests itself again)
		load_tables(next);
		load_codes(codes[P ^ 1], next);
		const int g0 = s * gs;
		add(codes[P][0], tbl + P * SV_BUF);
		if(gs == 2 && g0 + 1 < nGroups) add(codes[P][1], tbl + P * SV_BUF + (tblOff[g0 + 1] - tblOff[g0]));
		write_tables(P ^ 1);
		lds_barrier();
	};
	for(int s = 0; s < nSlabs; s += 2) {
		step(s, std::integral_constant<int, 0>());
		if(s + 1 < nSlabs) step(s + 1, std::integral_constant<int, 1>());
	}

	const double cadd = constIdx >= 0 ? T[constIdx] : 0.0;
	int cnt = 0;
#pragma unroll
	for(int j = 0; j < NU; j++) {
		if(w0 + j * 64 + lane >= w1) continue;
		const int64_t row = (w0 + j * 64 + lane) * 4;
		if(constIdx >= 0) {
#pragma unroll
			for(int i = 0; i < 4; i++) acc[j][i] += cadd;
		}
		if(op.w != nullptr) {
#pragma unroll
			for(int i = 0; i < 4; i++) acc[j][i] = row_op(acc[j][i], op.w[min(row + i, nRows - 1)], op.minus);
		}
		if(row + 4 <= nRows) {
#pragma unroll
			for(int i = 0; i < 4; i += 2) {
				cnt += (acc[j][i] != 0.0) + (acc[j][i + 1] != 0.0);
				f64x2_sv d;
				d.x = acc[j][i]; d.y = acc[j][i + 1];
				*(f64x2_sv*) (out + row + i) = d;
			}
		}
		else {
#pragma unroll
			for(int i = 0; i < 4; i++)
				if(row + i < nRows) { cnt += acc[j][i] != 0.0; out[row + i] = acc[j][i]; }
		}
	}
	count_add(nnz, cnt);
}

// The same on few rows: a thread per row looks its groups up straight in global memory, SV_NB at a time.
// Bound: latency (codes, then values, per batch), then the vector memory path, a cycle per lane and line.
// (8, 10, 13, 16, 25 at a time: 25 groups of 4096 tuples, 20,003 rows 13.0, 12.4, 12.1, 12.6, 11.9 us, 300,000 rows 37.0, 36.4, 36.0,
// 37.1, 36.1; 30 groups of 700 24.7, 26.0, 27.7, 27.1, 31.2; places behind the last group look the last one up again.)
constexpr int SV_NB = 13;
__global__ __launch_bounds__(256) void k_rmm_q1_short_rows(const uint8_t* __restrict__ arena, size_t arenaStride, int nGroups,
	const int32_t* __restrict__ tblOff, const double* __restrict__ T, int constIdx, double* __restrict__ out, int64_t nRows,
	unsigned long long* __restrict__ nnz, const RowOp op) {
	const int64_t row = (int64_t) blockIdx.x * 256 + threadIdx.x;
	const uint8_t* at = arena + 2 * min(row, nRows - 1);
	double acc = 0.0;
	for(int g0 = 0; g0 < nGroups; g0 += SV_NB) {
		uint32_t code[SV_NB];
		double v[SV_NB];
#pragma unroll
		for(int j = 0; j < SV_NB; j++) code[j] = *(const uint16_t*) (at + (size_t) min(g0 + j, nGroups - 1) * arenaStride);
#pragma unroll
		for(int j = 0; j < SV_NB; j++) v[j] = T[tblOff[min(g0 + j, nGroups - 1)] + (int) code[j]];
#pragma unroll
		for(int j = 0; j < SV_NB; j++)
			if(g0 + j < nGroups) acc += v[j];
	}
	if(constIdx >= 0) acc += T[constIdx];
	if(op.w != nullptr) acc = row_op(acc, op.w[min(row, nRows - 1)], op.minus);
	if(row < nRows) out[row] = acc;
	count_add(nnz, row < nRows && acc != 0.0);
}

// Returns 1 when the block is not eligible. `tables`: dict x v of all groups and, at constIdx, the constants' term.
int launch_rmm_q1_short(cla_block* b, const double* tables, int constIdx, double* dOut, unsigned long long* dNnz, RowOp* op) {
	const int nG = (int) b->groups.size();
	if(b->dArena == nullptr || b->arenaWidth != 2 || nG == 0 || b->nRows == 0 || b->maxVals > SV_BUF) return 1;
	const RowOp rowOp = op != nullptr ? *op : RowOp();
	// Few rows straight from global memory: 20,000 x 50 11 against 27 us, 200,000 x 50 18 against 28. Its lookups slow down as the tables
	// grow: up to 1000 tuples the two meet between 300 and 400 thousand rows (30 groups of 700 23 / 30 at 200,003, 35 / 31 at 399,001),
	// from there on at 300,000 (30 of 1100 31.7 / 31.4, of 4000 42 / 33; 90 of 4000 399,001 rows 147 / 78). Tables that come one at a time
	// (more than 4096 tuples) cost the form with the tables in LDS twice the time, and k_rmm_rows has its range between the two from a few groups on, up to
	// 450,000 rows: 90 of 8000 tuples 350,003 rows 157 straight / 129 there / 146 in LDS, 30 of 4500 399,001 rows 57 / 44 / 55, 499,001
	// 65 / 54 / 55 (90 of 4500 172 / 154 / 143; 2 of 4500 399,001 rows 14 / 10 / 11).
	if(b->nRows > 300000 && b->nRows <= 450000 && 2 * b->maxVals > SV_BUF && nG >= 8) return 1;
	if(b->nRows <= (b->maxVals <= 1000 ? 400000 : 300000)) {
		const unsigned grid = (unsigned) ((b->nRows + 255) / 256);
		Prof pf(b, "k_rmm_q1_short_rows", grid, 256, 0, (double) b->nRows * (2 * nG + 8) + (double) b->totalVals * 8);
		hipLaunchKernelGGL(k_rmm_q1_short_rows, dim3(grid), dim3(256), 0, b->stream, b->dArena, b->arenaStride, nG, b->dTblOff, tables,
			constIdx, dOut, b->nRows, dNnz, rowOp);
		CLA_HIP(hipGetLastError());
		if(op != nullptr) op->done = true;
		return 0;
	}
	const int gs = 2 * b->maxVals <= SV_BUF ? 2 : 1;
	const int64_t n4 = (b->nRows + 3) / 4, perBlock = (int64_t) SV_WAVES * WAVE * SV_NU;
	const int64_t turns = (n4 + perBlock * g_numCU - 1) / (perBlock * g_numCU); // even shares: a whole number of blocks per CU
	// (fewer rows than a wave's 64 lanes per block and CU: fewer blocks, each of which brings all tables in)
	const unsigned grid = (unsigned) std::min<int64_t>(turns * g_numCU, (n4 + SV_THREADS / 4 - 1) / (SV_THREADS / 4));
	const int64_t perWave = ((n4 + grid - 1) / grid + SV_WAVES - 1) / SV_WAVES;
	const int nu = (int) ((perWave + WAVE - 1) / WAVE);
	const size_t lds = (size_t) 2 * SV_BUF * 8;
	Prof pf(b, "k_rmm_q1_short", grid, SV_THREADS, (long) lds, (double) b->nRows * (2 * nG + 8) + (double) b->totalVals * 8);
#define SV_LAUNCH(NU)                                                                                                        \
	do {                                                                                                                     \
		CLA_HIP(allow_full_lds((const void*) k_rmm_q1_short<NU>));                                                           \
		hipLaunchKernelGGL(k_rmm_q1_short<NU>, dim3(grid), dim3(SV_THREADS), lds, b->stream, b->dArena, b->arenaStride, nG, gs, \
			b->dTblOff, tables, constIdx, dOut, b->nRows, dNnz, rowOp);                                                               \
	} while(0)
	if(nu <= 1) SV_LAUNCH(1);
	else if(nu == 2) SV_LAUNCH(2);
	else if(nu == 3) SV_LAUNCH(3);
	else SV_LAUNCH(4);
#undef SV_LAUNCH
	CLA_HIP(hipGetLastError());
	if(op != nullptr) op->done = true;
	return 0;
}

// t(y) %*% X: a block owns a slab of at most GS groups and a share of the rows. A wave takes 512 rows at a time, lane l the
// rows 2 l and 2 l + 1 of each 128 (whole lines of y and of the codes per instruction), the next 512 on their way meanwhile.
// Bound: LDS lookups of 8 NC bytes (busy 71 % of the time, more than half of it bank conflicts; vector memory path 54 %, vector
// issue 34 %); y comes once per slab from L2 or the memory-side cache. 2,500,009 x 50, 4096 tuples, 278 -> 42 us
// (rows decoded into tiles for the matrix cores before, with a wait for the host's look at y), 20,000 x 50 62 -> 11.
template <int NC, int GS>
__global__ __launch_bounds__(SV_THREADS) void k_lmm_q1_short(const DGroup* __restrict__ groups, const uint8_t* __restrict__ arena,
	size_t arenaStride, int nGroups, const int32_t* __restrict__ tblOff, const double* __restrict__ dict, const double* __restrict__ y,
	int64_t nRows, int nSlabs, double* __restrict__ out, int nCols, unsigned* __restrict__ done, unsigned long long* __restrict__ nnz) {
	extern __shared__ __attribute__((aligned(16))) double smem[];
	typedef double val __attribute__((ext_vector_type(NC)));
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	// the slabs of a share of the rows are blocks of one XCD that start together (blocks go to the XCDs in turn): y from its L2
	const int slab = blockIdx.x / 8 % nSlabs, share = blockIdx.x / 8 / nSlabs * 8 + blockIdx.x % 8, nShares = gridDim.x / nSlabs;
	const int g0 = (int) ((int64_t) nGroups * slab / nSlabs), nG = (int) ((int64_t) nGroups * (slab + 1) / nSlabs) - g0;
	const int64_t nUnits = nRows / 512; // whole ones
	const int64_t u0 = nUnits * share / nShares, u1 = nUnits * (share + 1) / nShares;

	const uint8_t* base[GS];
	uint32_t tab[GS]; // byte offset of the group's tuples in LDS
	const int e0 = tblOff[g0];
#pragma unroll
	for(int g = 0; g < GS; g++) {
		const int gg = g0 + min(g, nG - 1); // (a slab of fewer groups: its last one again, not used)
		base[g] = arena + (size_t) gg * arenaStride;
		tab[g] = (uint32_t) (tblOff[gg] - e0) * (uint32_t) (NC * 8);
	}
	val acc[GS];
#pragma unroll
	for(int g = 0; g < GS; g++) acc[g] = val(0.0);
	uint32_t codes[2][GS][4];
	f64x2_sv yv[2][4];
	auto load = [&](int64_t u, auto set) {
		constexpr int Q = decltype(set)::value;
		const int64_t r = u * 512 + 2 * lane;
#pragma unroll
		for(int j = 0; j < 4; j++) {
			yv[Q][j] = *(const f64x2_sv*) (y + r + 128 * j);
#pragma unroll
			for(int g = 0; g < GS; g++) codes[Q][g][j] = *(const uint32_t*) (base[g] + 2 * (r + 128 * j));
		}
	};
	auto work = [&](auto set) {
		constexpr int Q = decltype(set)::value;
#pragma unroll
		for(int g = 0; g < GS; g++)
#pragma unroll
			for(int j = 0; j < 4; j++) {
				const uint32_t c = codes[Q][g][j];
				const val a = *(const val*) ((const char*) smem + tab[g] + (c & 0xffffu) * (NC * 8));
				const val b2 = *(const val*) ((const char*) smem + tab[g] + (c >> 16) * (NC * 8));
#pragma unroll
				for(int h = 0; h < NC; h++) {
					acc[g][h] = __builtin_fma(yv[Q][j].x, a[h], acc[g][h]);
					acc[g][h] = __builtin_fma(yv[Q][j].y, b2[h], acc[g][h]);
				}
			}
	};
	using std::integral_constant;
	int64_t u = u0 + wave;
	if(u < u1) load(u, integral_constant<int, 0>());
	{
		const val* src = (const val*) (dict + (size_t) e0 * NC);
		const int n = tblOff[g0 + nG] - e0;
		for(int i0 = tid; i0 < n; i0 += 8 * SV_THREADS) {
			val d[8];
#pragma unroll
			for(int j = 0; j < 8; j++) d[j] = src[min(i0 + j * SV_THREADS, n - 1)];
#pragma unroll
			for(int j = 0; j < 8; j++)
				if(i0 + j * SV_THREADS < n) ((val*) smem)[i0 + j * SV_THREADS] = d[j];
		}
	}
	__syncthreads();
	for(; u < u1; u += 2 * SV_WAVES) {
		load(u + SV_WAVES < u1 ? u + SV_WAVES : u, integral_constant<int, 1>());
		work(integral_constant<int, 0>());
		if(u + SV_WAVES >= u1) break;
		load(u + 2 * SV_WAVES < u1 ? u + 2 * SV_WAVES : u, integral_constant<int, 0>());
		work(integral_constant<int, 1>());
	}
	if(share == nShares - 1 && wave == SV_WAVES - 1 && nUnits * 512 < nRows) { // the rows behind the whole units
		const int64_t last = (nRows - 1) & ~(int64_t) 1;
#pragma unroll
		for(int j = 0; j < 4; j++) {
			const int64_t r = nUnits * 512 + 128 * j + 2 * lane;
			yv[0][j].x = r < nRows ? y[r] : 0.0;
			yv[0][j].y = r + 1 < nRows ? y[r + 1] : 0.0;
#pragma unroll
			for(int g = 0; g < GS; g++) codes[0][g][j] = *(const uint32_t*) (base[g] + 2 * min(r, last)); // (codes behind the last row are valid ones)
		}
		work(integral_constant<int, 0>());
	}
	__syncthreads();
#pragma unroll
	for(int g = 0; g < GS; g++)
#pragma unroll
		for(int h = 0; h < NC; h++) {
			const double s = wave_sum_f64(acc[g][h]);
			if(lane == 0) smem[(g * NC + h) * SV_WAVES + wave] = s;
		}
	__syncthreads();
	if(tid < nG * NC) {
		double s = 0.0;
		for(int w = 0; w < SV_WAVES; w++) s += smem[tid * SV_WAVES + w];
		if(s != 0.0) unsafeAtomicAdd(&out[groups[g0 + tid / NC].cols[tid % NC]], s);
	}
	// (a slab's blocks alone add to its cells: on one line / on eight, in us, 500,000 rows: two slabs 14.2 / 14.7, three 16.9 / 15.2, seven 19.6 / 18.8)
	lmm_tail(done, gridDim.x, out, nCols, nnz, nSlabs > 2 ? TICKET_FEW : TICKET_QUEUED);
}

// Groups per slab of k_lmm_q1_short; 0: the block is not of its shape. One row of Y; all groups with one or with two columns.
// (Non-finite dictionary values: the reference sums y per tuple first, see launch_lmm_joint.)
int lmm_q1_short_groups(const cla_block* b) {
	if(b->dArena == nullptr || b->arenaWidth != 2 || b->dictNonFinite || b->groups.empty() || (b->opt.lmmDisable & 1)) return 0;
	const int nc = b->groups[0].d.nColG;
	if(nc != 1 && nc != 2) return 0;
	for(const HostGroup& g : b->groups)
		if(g.d.nColG != nc || g.d.nVals < 1) return 0;
	const int room = (g_ldsPerBlock - 512) / (b->maxVals * nc * 8); // (the tail's static LDS)
	return std::min(room, 4);
}

// Returns 1 when the block is not eligible, 0 when the groups' contributions have been added to dOut.
int launch_lmm_q1_short(cla_block* b, const double* dY, double* dOut) {
	const int most = lmm_q1_short_groups(b);
	if(most < 1) return 1;
	const int nG = (int) b->groups.size(), nc = b->groups[0].d.nColG;
	const int nSlabs = (nG + most - 1) / most, gs = (nG + nSlabs - 1) / nSlabs;
	const size_t lds = std::max((size_t) gs * b->maxVals * nc * 8, (size_t) gs * nc * SV_WAVES * 8);
	const int64_t nUnits = (b->nRows + 511) / 512;
	const int64_t perXcd = std::max<int64_t>(1, std::min<int64_t>(g_numCU / 8 / nSlabs, (nUnits + 63) / 64));
	const unsigned grid = (unsigned) (perXcd * 8 * nSlabs);
	Prof pf(b, "k_lmm_q1_short", grid, SV_THREADS, (long) lds, (double) b->nRows * (2 * nG + 8) + (double) b->totalVals * nc * 8);
	const bool tail = b->lmmTailWanted;
#define SV_LAUNCH(NC, GS)                                                                                                        \
	do {                                                                                                                         \
		CLA_HIP(allow_full_lds((const void*) k_lmm_q1_short<NC, GS>));                                                           \
		hipLaunchKernelGGL((k_lmm_q1_short<NC, GS>), dim3(grid), dim3(SV_THREADS), lds, b->stream, b->dGroups, b->dArena,        \
			b->arenaStride, nG, b->dTblOff, b->dAllDict, dY, b->nRows, nSlabs, dOut, b->nCols, tail ? b->lmm_ticket() : nullptr, \
			b->dCounters);                                                                                                       \
	} while(0)
#define SV_LAUNCH_N(GS) do { if(nc == 1) SV_LAUNCH(1, GS); else SV_LAUNCH(2, GS); } while(0)
	if(gs == 1) SV_LAUNCH_N(1);
	else if(gs == 2) SV_LAUNCH_N(2);
	else if(gs == 3) SV_LAUNCH_N(3);
	else SV_LAUNCH_N(4);
#undef SV_LAUNCH_N
#undef SV_LAUNCH
	b->lmmTailDone = tail;
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
