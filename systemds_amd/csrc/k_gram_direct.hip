// t(X) %*% X of blocks that are a few "varying" columns next to run-length columns, without tiles in LDS
// (the reference decompresses such blocks and multiplies the rows, CLALibTSMM.java:73-77; the run-length
// side replaces the per-row loop of ColGroupRLE.java:104-141 by work per run).
//
// Varying columns (NV <= 12): one value per row behind a plain stream - DDC codes of one or two bytes, the
// one-code-per-row copy of an SDCZeros group (0xff = the row has no entry), a column of an uncompressed
// group. Run-length columns (nR <= 8): columns of RLE groups, followed by run cursors (cla_runs.hpp).
//
// Lane = column and eight rows: of the wave's 64 lanes l, k = l / 16 and c = l % 16, lane (k, c) decodes column slot c at rows
// 8 k .. 8 k + 7 of a unit of 32 rows, straight from the column's stream (16 bytes of codes per lane, a unit ahead by two) and the values
// by tuple in LDS. The looked-up values are both operands of v_mfma_f64_4x4x4, four products of 4 x 4 columns over 4 rows:
//   V x V   x times itself and x times x rotated by four lanes: all pairs of three groups of four columns (quads) in two
//           instructions per 4 rows, in two registers per lane (one or two quads fill the
//           slots with 4 or 2 sets of rows). The sums of 78 products per row on the vector unit, lane = row, took 156 registers: one
//           wave per SIMD, and every wait of it a wait of the SIMD;
//   R x V   a run-length column is never looked up per row. The rows between two run ends (of any column) are a stretch on
//           which all of them are constant: a lane keeps the sum of its column's values over the stretch, and where the
//           stretch ends that sum times each run-length column's value joins the lane's own cell of the pair;
//   R x R   likewise with the number of rows of the stretch, a lane per pair.
// No value of a run-length column is ever looked up per row, and no one-code-per-row copy of it is read.
//
// Dense columns go through a wave's LDS (16 bytes per lane and unit, as they lie), from where they are "looked up" by row.
//
// Bound: matrix and vector issue, which do not overlap on a SIMD (per 32 rows of 9 - 12 columns 16 matrix instructions of 17 - 19 cycles and 54
// vector instructions, 140 more where a run ends; four waves per SIMD: vector 50 %, matrix 37 % of the CUs' busy cycles), next to HBM. Measured
// (lane = row on the vector unit before, one wave per SIMD): 50,000,000 rows, 8 run-length, 8 two-byte, 2 offset-list, 2 dense columns 802 ->
// 478 us (3.5 TB/s), 5,000,000 113 -> 58, 1,000,000 56 -> 23; 40,000,000 of 2 / 2 / 1 / 1 176 -> 103, 300,000 of 4 / 3 / 1 / 1 45 -> 13.
#include "../../include/cla_hip.h"
#include "cla_gdr.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

namespace cla {

constexpr int GDR_VMAX = 12;                 // varying columns
constexpr int GDR_NP = 16 + RC_MAX;          // block tile: index < 16 varying column, 16 + a run-length column a
constexpr int GDR_WDOUBLES = 64 + 32;        // per wave: window values, window ends
constexpr int GDR_STAGE = 2048;              // per wave: bytes of a unit's dense values
constexpr int GDR_REBASE = 32;               // most units that a chain of additions runs over

constexpr int gdr_sets(int nq) { return nq == 1 ? 4 : nq == 2 ? 2 : 1; } // sets of 32 rows in a unit

__device__ __forceinline__ uint32_t gdr_lds(const void* p) { return (uint32_t) (size_t) (const __attribute__((address_space(3))) uint8_t*) p; }
// base + 8 times half HI of a pair of codes, in one instruction
template <int HI>
__device__ __forceinline__ uint32_t gdr_at8(uint32_t pair, uint32_t base) {
	uint32_t r;
	if constexpr(HI) asm("v_mad_u32_u16 %0, %1, 8, %2 op_sel:[1,0,0,0]" : "=v"(r) : "v"(pair), "v"(base));
	else asm("v_mad_u32_u16 %0, %1, 8, %2" : "=v"(r) : "v"(pair), "v"(base));
	return r;
}

// x of the lane four places on, in the lane's row of 16
__device__ __forceinline__ double gdr_next_quad(double x) {
	int p[2];
	__builtin_memcpy(p, &x, 8);
	p[0] = __builtin_amdgcn_mov_dpp(p[0], 0x12C, 0xf, 0xf, true); // row_ror:12
	p[1] = __builtin_amdgcn_mov_dpp(p[1], 0x12C, 0xf, 0xf, true);
	double r;
	__builtin_memcpy(&r, p, 8);
	return r;
}

// NQ quads of varying columns, ND pieces of 16 bytes of dense values per lane and unit, WAVES per block
template <int NQ, int ND, bool HASR, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void k_tsmm_direct(const GdrArgs A) {
	extern __shared__ __align__(16) double smem[];
	constexpr int THREADS = WAVES * 64, SETS = gdr_sets(NQ), UR = 32 * SETS;
	constexpr int NM = NQ == 1 ? 1 : 2; // matrix instructions per 4 rows
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int k = lane >> 4, c = lane & 15, b = c >> 2;
	double* const gramS = smem + A.valDoubles;
	double* const wbase = gramS + GDR_NP * GDR_NP + wave * GDR_WDOUBLES;
	double* const winVal = wbase;
	int32_t* const winEnd = (int32_t*) (wbase + 64);
	char* const stage = (char*) (gramS + GDR_NP * GDR_NP + WAVES * GDR_WDOUBLES) + wave * GDR_STAGE;

	const int32_t nRows = (int32_t) A.nRows;
	const int nUnits = (nRows + UR - 1) / UR, nW = gridDim.x * WAVES, gw = blockIdx.x * WAVES + wave;
	const int u0 = (int) ((int64_t) nUnits * gw / nW), u1 = (int) ((int64_t) nUnits * (gw + 1) / nW), uF = min(u1, nRows / UR);
	const int nR = HASR ? A.nR : 0;

	// the lane's column: quad by slot, set of rows where quads are fewer than slots
	auto quad_of = [](int bb) { return NQ == 1 ? 0 : NQ == 2 ? bb & 1 : bb == 3 ? 0 : bb; };
	const int rowIn = 8 * (k + 4 * (NQ == 1 ? b : NQ == 2 ? b >> 1 : 0));
	const GdrCol C = A.cols[min(4 * quad_of(b) + (c & 3), A.nV - 1)];
	const bool pad = C.col < 0 || 4 * quad_of(b) + (c & 3) >= A.nV;
	const int bpr = C.bpr;
	// A lane of one-byte codes loads the 16 bytes that hold its eight; its codes become two-byte ones like the others'.
	const bool odd = (k & 1) != 0;
	const uint32_t sel0 = pad ? 0x0c0c0c0cu : bpr == 1 ? 0x0c010c00u : 0x07060504u, sel1 = pad ? 0x0c0c0c0cu : bpr == 1 ? 0x0c030c02u : 0x07060504u;
	// LDS address of the value of code 0 (the last of the values is a zero)
	uint32_t base = gdr_lds(smem) + (uint32_t) (pad ? A.valDoubles * 8 - 8 : C.base8);
	if(!pad && C.dense0 >= 0) base = gdr_lds(stage) + (uint32_t) (C.dense0 * 8 * UR + rowIn * C.width * 8 + C.base8);
	const uint8_t* const src = (const uint8_t*) as_global(C.src);
	auto codes_at = [&](int32_t row) { return src + ((size_t) (uint32_t) row * (uint32_t) bpr & ~(size_t) 15); };
	// The lane's pieces of the dense columns. (A lane without one fetches what nobody reads: no branch around a load, which would
	// wait for the load.)
	const uint8_t* dptr[ND > 0 ? ND : 1];
	int32_t dstep[ND > 0 ? ND : 1]; // bytes from unit to unit
	auto dense_at = [&](int i, int u, int32_t& step) { // piece i of unit u; the last unit: no piece that starts behind the end of its rows
		const uint8_t* p = (const uint8_t*) A.vals;
		step = 0;
		for(int g = 0; g < A.nDense; g++) {
			const GdrDense G = A.dense[g];
			const int at = (lane + 64 * i) * 16 - G.before * 8 * UR;
			if(at < 0 || at >= G.bpr * UR) continue;
			step = G.bpr * UR;
			const size_t from = (size_t) u * (uint32_t) step + (uint32_t) at;
			if(from < (size_t) nRows * (uint32_t) G.bpr) p = G.src + from;
		}
		return (const uint8_t*) as_global(p);
	};
#pragma unroll
	for(int i = 0; i < ND; i++) dptr[i] = dense_at(i, min(u0, max(uF - 1, 0)), dstep[i]);

	u32x4 W[2];
	f64x2 dv[2][ND > 0 ? ND : 1];
	const uint8_t* cptr = codes_at(u0 * UR + rowIn);
	const int32_t cstep = bpr * UR;
	auto request = [&](auto pTag, bool more) __attribute__((always_inline)) { // the unit at the pointers, which move on if there is another
		constexpr int P = decltype(pTag)::value;
		W[P] = *(const u32x4*) cptr;
		cptr += more ? cstep : 0;
#pragma unroll
		for(int i = 0; i < ND; i++) {
			dv[P][i] = *(const f64x2*) dptr[i];
			dptr[i] += more ? dstep[i] : 0;
		}
	};
	using std::integral_constant;
	if(u0 < uF) {
		request(integral_constant<int, 0>(), u0 + 1 < uF);
		request(integral_constant<int, 1>(), u0 + 2 < uF);
	}
	gdr_copy_vals<THREADS>(smem, A.vals, A.valDoubles);
	for(int i = tid; i < GDR_NP * GDR_NP; i += THREADS) gramS[i] = 0.0;
	RunCursors rc;
	if(u0 < u1) rc.start(A.runs, nR, winEnd, winVal, u0 * UR, lane);
	__syncthreads();

	if(u0 < u1) {
		double acc[NM], tot[NM]; // of the units since the last rebase, of those in front of it
#pragma unroll
		for(int m = 0; m < NM; m++) acc[m] = tot[m] = 0.0;
		double U = 0.0, H[HASR ? RC_MAX : 1], rr = 0.0; // the lane's sum over the stretch; its cells of the pairs with run-length columns; pair (lane / 8, lane % 8) of those
#pragma unroll
		for(int a = 0; a < (HASR ? RC_MAX : 1); a++) H[a] = 0.0;
		int32_t eNext = HASR ? rc.next_end() : RC_NEVER, from = u0 * UR; // the stretch's first row

		auto stretch = [&](int32_t upTo) __attribute__((always_inline)) { // rows from .. upTo - 1
#pragma unroll
			for(int a = 0; a < RC_MAX; a++) H[HASR ? a : 0] = __builtin_fma(rc.value(a), U, H[HASR ? a : 0]); // (unused cursors hold the value 0)
			const double va = __shfl(rc.val, RC_LANE0 + (lane >> 3), WAVE), vb = __shfl(rc.val, RC_LANE0 + (lane & 7), WAVE);
			rr = __builtin_fma((double) (upTo - from) * va, vb, rr);
			U = 0.0;
			from = upTo;
		};
		// unit u, whose codes and dense values are in the registers of its parity; tail: rows behind the end of the matrix count as zeros
		auto unit = [&](auto pTag, int u, auto tailTag, auto then) __attribute__((always_inline)) {
			constexpr int P = decltype(pTag)::value;
			constexpr bool TAIL = decltype(tailTag)::value;
			const int32_t row0 = u * UR + rowIn;
			const u32x4 w = W[P];
			const uint32_t e0 = odd ? w.z : w.x, e1 = odd ? w.w : w.y;
			uint32_t cd[4] = {__builtin_amdgcn_perm(w.x, e0, sel0), __builtin_amdgcn_perm(w.y, e0, sel1), __builtin_amdgcn_perm(w.z, e1, sel0),
				__builtin_amdgcn_perm(w.w, e1, sel1)};
#pragma unroll
			for(int i = 0; i < ND; i++) *(f64x2*) (stage + (lane + 64 * i) * 16) = dv[P][i];
			if(ND > 0) wave_lds_sync();
			double x[8];
#pragma unroll
			for(int t = 0; t < 8; t++) {
				if(TAIL && C.dense0 < 0) cd[t >> 1] = row0 + t < nRows ? cd[t >> 1] : cd[t >> 1] & (t & 1 ? 0x0000ffffu : 0xffff0000u); // (behind the last row: never an index)
				x[t] = *(const __attribute__((address_space(3))) double*) (size_t) (t & 1 ? gdr_at8<1>(cd[t >> 1], base) : gdr_at8<0>(cd[t >> 1], base));
				if(TAIL) x[t] = row0 + t < nRows ? x[t] : 0.0;
			}
			if(ND > 0) wave_lds_sync(); // (the next unit's dense values come behind these reads)
			then();
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for(int t = 0; t < 8; t++) {
				acc[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[t], x[t], acc[0], 0, 0, 0);
				if(NQ > 1) acc[NQ > 1 ? 1 : 0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[t], gdr_next_quad(x[t]), acc[NQ > 1 ? 1 : 0], 0, 0, 0);
			}
			if(HASR) {
				const int32_t uEnd = TAIL ? nRows : (u + 1) * UR;
				if(__builtin_expect(eNext >= uEnd, 1)) U += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
				else {
					int32_t lo = 0; // rows of the lane in front of the last run end
					while(eNext < uEnd) { // (uniform)
						const int32_t hi = eNext - row0;
#pragma unroll
						for(int t = 0; t < 8; t++) U += t >= lo && t < hi ? x[t] : 0.0;
						stretch(eNext);
						lo = hi;
						rc.advance(eNext, lane);
						eNext = rc.next_end();
					}
#pragma unroll
					for(int t = 0; t < 8; t++) U += t >= lo ? x[t] : 0.0;
				}
			}
		};
		auto rebase = [&](int32_t upTo) __attribute__((always_inline)) {
			if(HASR) stretch(upTo);
#pragma unroll
			for(int m = 0; m < NM; m++) { tot[m] += acc[m]; acc[m] = 0.0; }
		};
		for(int uB = u0; uB < uF; uB += GDR_REBASE) {
			const int uE = min(uB + GDR_REBASE, uF);
			for(int u = uB; u < uE; u += 2) {
				unit(integral_constant<int, 0>(), u, std::false_type(), [&]() __attribute__((always_inline)) { request(integral_constant<int, 0>(), u + 3 < uF); });
				if(u + 1 < uE) unit(integral_constant<int, 1>(), u + 1, std::false_type(), [&]() __attribute__((always_inline)) { request(integral_constant<int, 1>(), u + 4 < uF); });
			}
			rebase(uE * UR);
		}
		if(uF < u1) { // the last, partly filled unit of the matrix
			W[0] = *(const u32x4*) codes_at(min(uF * UR + rowIn, (nRows - 1) & ~7));
#pragma unroll
			for(int i = 0; i < ND; i++) {
				int32_t step;
				dv[0][i] = *(const f64x2*) dense_at(i, uF, step);
			}
			unit(integral_constant<int, 0>(), uF, std::true_type(), [] {});
			rebase(nRows);
		}

		// the wave's sums into the block's tile: lane (k, c) holds row k of quad qa, column c % 4 of quad qb of its slot's products
#pragma unroll
		for(int m = 0; m < NM; m++) {
			const int qa = quad_of(b), qb = quad_of((b + m) & 3), i = 4 * qa + k, j = 4 * qb + (c & 3);
			const bool mine = m == 0 ? (NQ == 3 ? b < 3 : true) && k <= (c & 3) : NQ == 2 ? (b & 1) == 0 : b < 3;
			if(mine && tot[m] != 0.0) unsafeAtomicAdd(&gramS[min(i, j) * GDR_NP + max(i, j)], tot[m]);
		}
		if(HASR) {
			if(NQ != 3 || b < 3)
#pragma unroll
				for(int a = 0; a < RC_MAX; a++)
					if(a < nR && H[a] != 0.0) unsafeAtomicAdd(&gramS[(4 * quad_of(b) + (c & 3)) * GDR_NP + 16 + a], H[a]);
			const int a = lane >> 3, b2 = lane & 7;
			if(a <= b2 && b2 < nR && rr != 0.0) unsafeAtomicAdd(&gramS[(16 + a) * GDR_NP + 16 + b2], rr);
		}
	}
	__syncthreads();
	double* const into = A.done != nullptr ? A.acc + gram_way(A.nCols) : A.out;
	for(int idx = tid; idx < GDR_NP * GDR_NP; idx += THREADS) {
		const double s = gramS[idx];
		if(s == 0.0) continue;
		const int i = idx / GDR_NP, j = idx - i * GDR_NP;
		const int ci = i < 16 ? (i < A.nV ? A.cols[i].col : -1) : (i - 16 < nR ? A.runs[i - 16].col : -1);
		const int cj = j < 16 ? (j < A.nV ? A.cols[j].col : -1) : (j - 16 < nR ? A.runs[j - 16].col : -1);
		if(ci < 0 || cj < 0) continue;
		unsafeAtomicAdd(&into[(size_t) min(ci, cj) * A.nCols + max(ci, cj)], s);
	}
	if(A.done != nullptr) gram_tail(A.done, gridDim.x, A.acc, A.out, A.nCols, A.nnz, (unsigned*) gramS);
}

// Blocks whose varying columns span many magnitudes next to run-length columns take the tile kernel: a column stays here while its
// largest value is within 2^GDR_SPREAD of all but a sixteenth of its nonzero ones. (Normal values span 2^7 by this measure,
// log-normal ones of sigma 2 and 50 M rows 2^20, counts up to a million 2^20.) The line stems from sums by parts, where a row enters
// sums that a run-length column with the value 0 there has to cancel again. Sums by stretch hold no such rows, so this kernel does
// not need it; the route of such blocks has been left as it was.
constexpr int GDR_SPREAD = 20;
constexpr int GDR_BINS = 2048; // exponents of a double; the last one: infinities and NaN

// The exponents of |x| counted, column c of a dense group: bins[c][exponent].
__global__ __launch_bounds__(256) void k_exponents(const double* __restrict__ dense, int nColG, int64_t nRows, unsigned long long* __restrict__ bins) {
	__shared__ unsigned h[GDR_BINS];
	for(int k = threadIdx.x; k < GDR_BINS; k += 256) h[k] = 0;
	__syncthreads();
	for(int64_t r = (int64_t) blockIdx.x * 256 + threadIdx.x; r < nRows; r += (int64_t) gridDim.x * 256)
		atomicAdd(&h[__double2hiint(dense[r * nColG + blockIdx.y]) >> 20 & (GDR_BINS - 1)], 1u);
	__syncthreads();
	for(int k = threadIdx.x; k < GDR_BINS; k += 256)
		if(h[k]) atomicAdd(&bins[(size_t) blockIdx.y * GDR_BINS + k], (unsigned long long) h[k]);
}

static bool gdr_spread(const unsigned long long* bins) {
	if(bins[GDR_BINS - 1] != 0) return true;
	unsigned long long n = 0, below = 0;
	int top = 0, low = 1;
	for(int k = 1; k < GDR_BINS; k++) // (zeros and what is smaller than any normal number: bin 0)
		if(bins[k]) { n += bins[k]; top = k; }
	while(low < top && (below += bins[low]) * 16 < n) low++;
	return top - low > GDR_SPREAD;
}

// P.spread, from the dense columns and P.codeSpread.
static int gdr_look(cla_block* b, GdrPlan& P) {
	int spread = P.codeSpread ? 1 : 0;
	for(const HostGroup& H : b->groups) {
		if(spread || P.A.nR == 0) break;
		if(H.d.type != G_UNC) continue;
		std::vector<unsigned long long> bins((size_t) H.d.nColG * GDR_BINS, 0);
		const int rc = ensure_scratch(b, bins.size() * sizeof(bins[0]));
		if(rc) return rc;
		unsigned long long* d = (unsigned long long*) b->dScratch;
		CLA_HIP(hipMemsetAsync(d, 0, bins.size() * sizeof(bins[0]), b->stream));
		hipLaunchKernelGGL(k_exponents, dim3((unsigned) std::min<int64_t>((b->nRows + 2047) / 2048, 2 * g_numCU), (unsigned) H.d.nColG), dim3(256), 0, b->stream,
			H.d.dense, H.d.nColG, b->nRows, d);
		CLA_HIP(hipGetLastError());
		CLA_HIP(hipMemcpyAsync(bins.data(), d, bins.size() * sizeof(bins[0]), hipMemcpyDeviceToHost, b->stream));
		CLA_HIP(hipStreamSynchronize(b->stream));
		for(int c = 0; c < H.d.nColG; c++) spread |= gdr_spread(&bins[(size_t) c * GDR_BINS]);
	}
	P.spread = spread; // (only now: a call that fails on the way looks again)
	return 0;
}

// Which columns of the block are streams, which are followed by run cursors; 1 when the block is not of this shape.
static int gdr_build_plan(cla_block* b, GdrPlan& P) {
	P.rc = 1;
	const int nG = (int) b->groups.size();
	if(b->nRows <= 0 || b->nRows >= ((int64_t) 1 << 31) - 256 || b->nCols > 64) return 0;
	std::vector<GdrCol> byClass[3];  // columns by class: two-byte codes, one-byte codes, dense
	std::vector<GdrDense> dense;
	int nD = 0;
	std::vector<double> vals; // by tuple: the column's constant plus the dictionary's value
	std::vector<RunCol> runs;
	std::vector<char> seen((size_t) b->nCols, 0);
	int covered = 0;
	for(int g = 0; g < nG; g++) {
		const DGroup& G = b->groups[g].d;
		const auto& hc = b->groups[g].cols;
		for(int c : hc) {
			if(seen[c]) return 0; // overlapping groups
			seen[c] = 1;
		}
		if(G.type == G_UNC) {
			if(((uintptr_t) G.dense & 15) != 0 || G.nColG > 8) return 0;
			for(int h = 0; h < G.nColG; h++) {
				if(b->constV[hc[h]] != 0.0) return 0; // (a dense column next to a constant: the tile kernel adds it)
				byClass[2].push_back(GdrCol{(const uint8_t*) G.dense, 0, h * 8, nD, G.nColG, hc[h], 0});
			}
			dense.push_back(GdrDense{(const uint8_t*) G.dense, G.nColG * 8, nD});
			nD += G.nColG;
			covered += G.nColG;
			continue;
		}
		if(G.type != G_DDC && G.type != G_RLE && !(G.type == G_SDCZ && G.nOffsets > 0)) continue; // no row data
		const bool haveStream = g < (int) b->expCodes.size() && b->expCodes[g] != nullptr;
		if(G.type == G_RLE && !haveStream) {
			for(int h = 0; h < G.nColG; h++) runs.push_back(RunCol{G.runStart, G.runCode, G.dict, b->constV[hc[h]], G.nRuns, G.nColG, h, hc[h]});
			covered += G.nColG;
			P.runEnds += std::max(G.nRuns - 1, 0);
			continue;
		}
		const uint8_t* src;
		int cls, fill;
		if(G.type == G_DDC) {
			if(G.codeWidth > 2) return 0;
			src = (const uint8_t*) G.codes;
			cls = G.codeWidth == 2 ? 0 : 1;
			fill = G.nVals;
		}
		else {
			if(!haveStream) return 0;
			src = b->expCodes[g];
			cls = 1;
			fill = 256; // code 0xff: no value on the row
		}
		if(((uintptr_t) src & 15) != 0) return 0;
		for(int h = 0; h < G.nColG; h++) {
			byClass[cls].push_back(GdrCol{src, cls == 0 ? 2 : 1, (int32_t) (8 * vals.size()), -1, 0, hc[h], 0});
			for(int t = 0; t < fill; t++) vals.push_back(b->constV[hc[h]] + (t < G.nVals ? b->groups[g].dict[(size_t) t * G.nColG + h] : 0.0));
			std::vector<unsigned long long> bins(GDR_BINS, 0);
			for(size_t t = vals.size() - fill; t < vals.size() - fill + G.nVals + (fill > G.nVals); t++) bins[std::isfinite(vals[t]) ? std::max(0, std::ilogb(vals[t]) + 1023) : GDR_BINS - 1]++;
			P.codeSpread |= gdr_spread(bins.data());
		}
		covered += G.nColG;
	}
	// (columns that no group holds row data for are constants: the tile kernel and the pair kernels serve them)
	if(covered != b->nCols) return 0;
	// An infinite or NaN run-length value meets a stretch's sum here, each row's own value in the tile kernel (infinity times 0 where the sum
	// is 0 and the values are not): such blocks take that kernel, which forms every row's cells.
	bool nonFinite = b->dictNonFinite;
	for(const RunCol& R : runs) nonFinite |= !std::isfinite(R.add);
	if(nonFinite && !runs.empty()) return 0;
	std::vector<GdrCol> all;
	for(const auto& cols : byClass) all.insert(all.end(), cols.begin(), cols.end());
	const int nCode = (int) (byClass[0].size() + byClass[1].size()), nR = (int) runs.size();
	const size_t zeroAt = vals.size();
	vals.resize((vals.size() + 3) & ~(size_t) 1, 0.0); // two zeros and an even number: what fillers and the lanes without a column look up
	const int nV = (int) all.size();
	if(nCode < 1 || nV > GDR_VMAX || nR > RC_MAX) return 0;
	const size_t valD = vals.size();
	P.quads = (nV + 3) / 4;
	P.densePieces = (nD * 32 * gdr_sets(P.quads) / 2 + 63) / 64;
	auto lds_of = [&](int waves) { return (valD + GDR_NP * GDR_NP + (size_t) waves * GDR_WDOUBLES) * 8 + (nD ? (size_t) waves * GDR_STAGE : 0); };
	const size_t room = (size_t) std::min(g_ldsPerBlock, 160 * 1024) - 1024;
	P.waves = lds_of(16) <= room ? 16 : 8;
	P.lds = lds_of(P.waves);
	if(P.lds > room) return 0;
	// (more dense columns than a wave stages: the Gram matrix on the tile kernel. The left multiply stages none)
	P.gram = P.densePieces <= GDR_STAGE / 1024;
	const size_t colBytes = all.size() * sizeof(GdrCol), dictBytes = valD * sizeof(double), runBytes = runs.size() * sizeof(RunCol);
	const size_t denseBytes = dense.size() * sizeof(GdrDense);
	// the same columns as the left multiply wants them: straight from their streams, filled up to a shape it exists for
	std::vector<LdCol> ld;
	{
		P.ldND = nD == 0 ? 0 : nD <= 2 ? 2 : 4;
		P.ldNC = nCode <= 4 ? 4 : nCode <= 8 ? 8 : nCode <= 10 && P.ldND == 2 ? 10 : 12;
		if(nD <= 4 && P.ldNC + P.ldND <= GDR_VMAX) {
			for(int k = 0; k < 3; k++) {
				for(const GdrCol& C : byClass[k]) // (dense: base8 is the column's place in the row)
					ld.push_back(LdCol{C.src + (k == 2 ? C.base8 : 0), k == 2 ? C.width * 8 : C.bpr, k == 2 ? 0 : C.base8, k == 0 ? 0xffffu : 0xffu, C.col});
				if(k == 1)
					while((int) ld.size() < P.ldNC) ld.push_back(LdCol{ld[0].src, ld[0].stride, (int32_t) (8 * zeroAt), 0u, -1});
			}
			while((int) ld.size() < P.ldNC + P.ldND) ld.push_back(LdCol{nullptr, 0, 0, 0u, -1}); // (src: a zero, below)
		}
	}
	if(ld.empty()) P.ldNC = 0;
	// the values, codes 0, n, 2 n .. 7 n of dense columns by the width n of their group, run-length columns, dense groups, columns, a zero
	uint16_t rowCodes[9][8];
	for(int n = 0; n < 9; n++)
		for(int t = 0; t < 8; t++) rowCodes[n][t] = (uint16_t) (n * t);
	const size_t codesAt = (dictBytes + 15) & ~(size_t) 15, runsAt = codesAt + sizeof(rowCodes), denseAt = runsAt + runBytes, colsAt = denseAt + denseBytes;
	std::vector<uint8_t> img(colsAt + colBytes + 24, 0); // (structs with pointers: 8-byte aligned)
	uint8_t* d = nullptr;
	CLA_HIP(hipMalloc((void**) &d, img.size() + 64));
	P.dImg = d;
	P.bytes = (int64_t) img.size() + 64;
	for(GdrCol& C : all)
		if(C.dense0 >= 0) C.src = d + codesAt + (size_t) C.width * sizeof(rowCodes[0]);
	std::memcpy(img.data(), vals.data(), dictBytes);
	std::memcpy(img.data() + codesAt, rowCodes, sizeof(rowCodes));
	if(runBytes) std::memcpy(img.data() + runsAt, runs.data(), runBytes);
	if(denseBytes) std::memcpy(img.data() + denseAt, dense.data(), denseBytes);
	std::memcpy(img.data() + colsAt, all.data(), colBytes);
	for(size_t i = 0; i < ld.size(); i++) {
		P.ld.c[i] = ld[i];
		if(ld[i].src == nullptr) P.ld.c[i].src = d + colsAt + colBytes; // a zero
	}
	CLA_HIP(hipMemcpy(d, img.data(), img.size(), hipMemcpyHostToDevice));
	P.A.vals = (const double*) d;
	P.A.runs = (const RunCol*) (d + runsAt);
	P.A.dense = (const GdrDense*) (d + denseAt);
	P.A.cols = (const GdrCol*) (d + colsAt);
	P.A.nV = nV; P.A.nR = nR; P.A.nDense = (int) dense.size();
	P.A.valDoubles = (int) valD;
	P.A.nRows = b->nRows;
	P.A.nCols = b->nCols;
	P.rc = 0;
	return 0;
}

void gdr_plan_drop(cla_block* b) {
	if(b->gdrPlan == nullptr) return;
	if(b->gdrPlan->dImg) { (void) hipFree(b->gdrPlan->dImg); b->derivedBytes -= b->gdrPlan->bytes; }
	delete b->gdrPlan;
	b->gdrPlan = nullptr;
}

int gdr_plan(cla_block* b, const GdrPlan*& P) {
	if(b->gdrPlan == nullptr) {
		int rc = ensure_expanded(b);
		if(rc) return rc;
		std::unique_ptr<GdrPlan> plan(new GdrPlan()); // (the block's only when it is complete)
		rc = gdr_build_plan(b, *plan);
		if(rc < 0) {
			if(plan->dImg) (void) hipFree(plan->dImg);
			return rc;
		}
		if(plan->dImg) b->derivedBytes += plan->bytes;
		b->gdrPlan = plan.release();
	}
	P = b->gdrPlan;
	return 0;
}

// dOut (nCols x nCols, zeroed) += upper triangle of t(D) %*% D of the decoded rows, constants included. Returns 1
// when the block is not of this kernel's shape (the caller takes the tile kernel on the matrix cores).
int launch_tsmm_direct(cla_block* b, double* dOut, unsigned long long* dNnz) {
	if(!b->opt.tsmmDirect || b->crossSplit > 0 || b->crossBlocks > 0) return 1;
	const GdrPlan* P = nullptr;
	if(const int rc = gdr_plan(b, P)) return rc;
	if(P->rc || !P->gram) return 1;
	if(P->spread < 0)
		if(const int rc = gdr_look(b, *b->gdrPlan)) return rc;
	if(P->spread && P->A.nR > 0) return 1;
	const int nUnits = (int) ((b->nRows + 32 * gdr_sets(P->quads) - 1) / (32 * gdr_sets(P->quads)));
	// A wave takes the run ends of its rows one after the other, 0.4 us each: a unit per wave where there are many (100,003 rows of 9 columns, 8
	// run-length of mean run 100: 19 us, two units 27; of 5000 12 and 12, 300,007 rows 12.9 and 12.1), else two.
	const int share = P->waves * (P->runEnds * 400 > b->nRows ? 1 : 2);
	const unsigned grid = (unsigned) std::max(1, std::min((nUnits + share - 1) / share, g_numCU));
	// The tile kernel hardly notices run ends, but takes 35 ns more per 1000 rows. Both meet at 9 run ends per wave on 20,011 rows, 10 on
	// 100,003, 22 on 300,007, 43 on 1,000,003 and 195 on 5,000,011 (one column behind codes, 8, 4 and 2 run-length ones; in us here / there:
	// 20,011 rows, 8 of mean run 100 17.5 / 19.2, of 48 25 / 19; 300,007, 8 of 48 29 / 34, of 24 43 / 32; 5,000,011, 4 of 48 99 / 162, of 12 290 / 160).
	if(P->runEnds / ((int64_t) grid * P->waves) > 8 + b->nRows / 27000) {
		const int rc = tsmm_decode_fits(b);
		if(rc <= 0) return rc < 0 ? rc : 1;
	}
	GdrArgs A = P->A;
	A.out = dOut;
	A.acc = nullptr; A.done = nullptr; A.nnz = nullptr;
	if(dNnz != nullptr) {
		const int rc = ensure_gram_acc(b);
		if(rc) return rc;
		A.acc = b->dGramAcc; A.done = b->gram_ticket(); A.nnz = dNnz;
	}
	Prof pf(b, "k_tsmm_direct", grid, P->waves * 64, (long) P->lds, (double) b->device_bytes_cached);
	bool launched = false;
#define GDR_CASE(NQV, NDV, HASRV, WV)                                                                                             \
	if(!launched && P->quads == NQV && P->densePieces == NDV && HASRV == (A.nR > 0) && P->waves == WV) {                          \
		CLA_HIP(allow_full_lds((const void*) k_tsmm_direct<NQV, NDV, HASRV, WV>));                                                \
		hipLaunchKernelGGL((k_tsmm_direct<NQV, NDV, HASRV, WV>), dim3(grid), dim3(WV * 64), P->lds, b->stream, A);                \
		launched = true;                                                                                                          \
	}
#define GDR_CASES(NQV, HASRV, WV) GDR_CASE(NQV, 0, HASRV, WV) GDR_CASE(NQV, 1, HASRV, WV) GDR_CASE(NQV, 2, HASRV, WV)
#define GDR_QUADS(HASRV, WV) GDR_CASES(1, HASRV, WV) GDR_CASES(2, HASRV, WV) GDR_CASES(3, HASRV, WV)
	GDR_QUADS(true, 16) GDR_QUADS(false, 16) GDR_QUADS(true, 8) GDR_QUADS(false, 8)
#undef GDR_QUADS
#undef GDR_CASES
#undef GDR_CASE
	if(!launched) return 1;
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
