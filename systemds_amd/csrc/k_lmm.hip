// Left multiply Y %*% X on a compressed block (gfx950).
//
//   k_lmm_preagg_rows   per-code aggregation of Y over DDC / RLE groups (row parallel),
//                       block-private fp64 bins in LDS, flushed with global atomics
//   k_lmm_preagg_sdc    the same for SDCZeros groups, parallel over offset-list chunks
//   k_lmm_unc           uncompressed groups: Y %*% U on the matrix cores
//   k_lmm_rowsum        rowSums(Y) for the constant correction
//   k_lmm_post          preAgg x dictionary into the output columns
//   k_lmm_finish        + rowSum (x) constV, non-zero count
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include "cla_runs.hpp"
#include <algorithm>
#include <cstring>

namespace cla {

constexpr int LMM_RPT = 16;        // rows per thread
constexpr int LMM_THREADS = 256;
constexpr int LMM_BIN_BYTES = 32 * 1024;

// Slab = consecutive groups [g0, g1) whose bins fit LDS; binOff[g - g0] = offset of
// the group's bins inside the LDS slab. One block covers `rowsPerBlock` rows.
__global__ __launch_bounds__(LMM_THREADS) void k_lmm_preagg_rows(const DGroup* __restrict__ groups, int g0, int g1,
	const double* __restrict__ Y, int64_t nRows, int64_t rowsPerBlock, double* __restrict__ pre, int totalVals,
	int direct) {
	// direct != 0: the group's bins do not fit LDS, aggregate straight into `pre` in HBM
	extern __shared__ double ldsBins[];
	const int i = blockIdx.y; // row of Y
	const int base = groups[g0].tblOff;
	const int nBins = groups[g1 - 1].tblOff + groups[g1 - 1].nVals - base;
	double* bins = direct ? pre + (size_t) i * totalVals + base : ldsBins;
	if(!direct) {
		for(int k = threadIdx.x; k < nBins; k += LMM_THREADS) bins[k] = 0.0;
		__syncthreads();
	}
	const double* y = Y + (size_t) i * nRows;
	const int64_t rb = (int64_t) blockIdx.x * rowsPerBlock;
	const int64_t re = min(rb + rowsPerBlock, nRows);
	for(int64_t r0 = rb + (int64_t) threadIdx.x * LMM_RPT; r0 < re; r0 += (int64_t) LMM_THREADS * LMM_RPT) {
		const int n = (int) min((int64_t) LMM_RPT, re - r0);
		double yv[LMM_RPT];
#pragma unroll
		for(int t = 0; t < LMM_RPT; t++) yv[t] = t < n ? y[r0 + t] : 0.0;
		for(int g = g0; g < g1; g++) {
			const DGroup G = dgroup(groups + (g));
			double* bg = bins + (G.tblOff - base);
			if(G.type == G_DDC) {
				if(n == LMM_RPT && G.codeWidth == 1) {
					const uint4 c = *(const uint4*) ((const uint8_t*) G.codes + r0);
					const uint32_t w[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
					for(int t = 0; t < LMM_RPT; t++) unsafeAtomicAdd(&bg[(w[t >> 2] >> (8 * (t & 3))) & 0xff], yv[t]);
				}
				else {
					for(int t = 0; t < n; t++) unsafeAtomicAdd(&bg[load_code(G.codes, G.codeWidth, r0 + t)], yv[t]);
				}
			}
			else if(G.type == G_RLE) {
				// walk the merged run table, adding each run's partial sum once
				int j = rle_find(G.runStart, G.nRuns, (int32_t) r0);
				int t = 0;
				while(t < n) {
					const int64_t runEnd = G.runStart[j + 1];
					const int code = G.runCode[j];
					double s = 0.0;
					while(t < n && r0 + t < runEnd) s += yv[t++];
					if(code >= 0) unsafeAtomicAdd(&bg[code], s);
					j++;
				}
			}
		}
	}
	if(direct) return;
	__syncthreads();
	double* dst = pre + (size_t) i * totalVals + base;
	for(int k = threadIdx.x; k < nBins; k += LMM_THREADS) {
		const double v = bins[k];
		if(v != 0.0) unsafeAtomicAdd(&dst[k], v);
	}
}

// SDCZeros: one block walks `chunksPerBlock` chunks of SDC_CK offset entries of one
// group; bins[code] += Y[i, row].
template <int W>
__global__ __launch_bounds__(256) void k_lmm_preagg_sdc(const DGroup* __restrict__ groups, int g, const double* __restrict__ Y,
	int64_t nRows, int chunksPerBlock, double* __restrict__ pre, int totalVals, int direct) {
	extern __shared__ double ldsBins[];
	const DGroup G = dgroup(groups + (g));
	const int i = blockIdx.y;
	const double* y = Y + (size_t) i * nRows;
	double* bins = direct ? pre + (size_t) i * totalVals + G.tblOff : ldsBins;
	if(!direct) {
		for(int k = threadIdx.x; k < G.nVals; k += 256) bins[k] = 0.0;
		__syncthreads();
	}
	if(blockIdx.x == 0 && threadIdx.x == 0 && G.nOffsets > 0)
		unsafeAtomicAdd(&bins[load_code(G.codes, G.codeWidth, 0)], y[G.first]);
	const int wave = threadIdx.x >> 6;
	const int c0 = blockIdx.x * chunksPerBlock;
	const int c1 = min(c0 + chunksPerBlock, G.nCkpt);
	for(int c = c0; c < c1; c++) {
		const OffState st = G.ckpt[c];
		int32_t row = st.row, emit = st.emit;
		int32_t rows[4], didx[4];
		unsigned mask;
		const int64_t base = (int64_t) c * SDC_CK;
		for(int w = 0; w < wave; w++) sdc_decode256<W>(G.deltas, G.nDeltas, base + w * 256, row, emit, rows, didx, mask);
		sdc_decode256<W>(G.deltas, G.nDeltas, base + wave * 256, row, emit, rows, didx, mask);
#pragma unroll
		for(int k = 0; k < 4; k++)
			if(mask & (1u << k)) unsafeAtomicAdd(&bins[load_code(G.codes, G.codeWidth, didx[k])], y[rows[k]]);
	}
	if(direct) return;
	__syncthreads();
	double* dst = pre + (size_t) i * totalVals + G.tblOff;
	for(int k = threadIdx.x; k < G.nVals; k += 256) {
		const double v = bins[k];
		if(v != 0.0) unsafeAtomicAdd(&dst[k], v);
	}
}

// uncompressed group: out[i, cols[j]] += sum_r Y[i,r] * U[r,j] on v_mfma_f64_16x16x4_f64. Block = (range of rows,
// 16 rows of Y, LU_NBJ blocks of 16 columns of the group); wave w takes rows 4 w .. 4 w + 3 of every 16; lane
// (k4, i16) holds Y[16 ib + i16, row k4] and U[row k4, 16 jb + i16]. The group is read once per 16 rows of Y, in
// pieces of 128 bytes per row (the scalar form it replaces read it once per row of Y and column: 1.6 ms per row of Y
// on 1M rows x 90 columns).
constexpr int LU_NBJ = 4;
typedef double lu_f64x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_lmm_unc(const DGroup* __restrict__ groups, int g, const double* __restrict__ Y, int p,
	int64_t nRows, int64_t rowsPerBlock, double* __restrict__ out, int nCols) {
	__shared__ double red[LU_NBJ * 256];
	const DGroup G = dgroup(groups + (g));
	const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
	const int i16 = lane & 15, k4 = lane >> 4;
	const int nC = G.nColG, nb = (nC + 15) / 16;
	const int ib = blockIdx.y, jb0 = blockIdx.z * LU_NBJ;
	const int nj = min(LU_NBJ, nb - jb0);
	const int yi = ib * 16 + i16;
	const bool yIn = yi < p;
	const double* y = as_global(Y) + (size_t) (yIn ? yi : 0) * nRows;
	const int64_t r0 = (int64_t) blockIdx.x * rowsPerBlock, r1 = min(nRows, r0 + rowsPerBlock);
	lu_f64x4 acc[LU_NBJ];
#pragma unroll
	for(int j = 0; j < LU_NBJ; j++) acc[j] = lu_f64x4{0.0, 0.0, 0.0, 0.0};
	for(int64_t r = r0 + wave * 4; r < r1; r += 16) {
		const int64_t row = r + k4;
		const bool in = row < r1;
		const double a = in && yIn ? y[row] : 0.0;
		const double* drow = G.dense + (size_t) (in ? row : r0) * nC;
#pragma unroll
		for(int j = 0; j < LU_NBJ; j++) {
			if(j >= nj) break;
			const int cbj = (jb0 + j) * 16 + i16;
			const double bv = in && cbj < nC ? drow[cbj] : 0.0;
			acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bv, acc[j], 0, 0, 0);
		}
	}
	for(int i = tid; i < LU_NBJ * 256; i += 256) red[i] = 0.0;
	__syncthreads();
#pragma unroll
	for(int j = 0; j < LU_NBJ; j++)
#pragma unroll
		for(int v = 0; v < 4; v++)
			if(j < nj) unsafeAtomicAdd(&red[j * 256 + (4 * v + k4) * 16 + i16], acc[j][v]);
	__syncthreads();
	for(int i = tid; i < nj * 256; i += 256) {
		const int j = i >> 8, rr = (i >> 4) & 15, cc = i & 15;
		const int gr = ib * 16 + rr, gc = (jb0 + j) * 16 + cc;
		if(gr < p && gc < nC && red[i] != 0.0) unsafeAtomicAdd(&out[(size_t) gr * nCols + G.cols[gc]], red[i]);
	}
}

__global__ __launch_bounds__(256) void k_lmm_rowsum(const double* __restrict__ Y, int64_t nRows, int64_t rowsPerBlock,
	double* __restrict__ rs) {
	__shared__ double red[4];
	const int i = blockIdx.y;
	const double* y = Y + (size_t) i * nRows;
	const int64_t rb = (int64_t) blockIdx.x * rowsPerBlock, re = min(rb + rowsPerBlock, nRows);
	double s = 0.0;
	for(int64_t r = rb + threadIdx.x; r < re; r += 256) s += y[r];
	s = wave_sum_f64(s);
	if((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
	__syncthreads();
	if(threadIdx.x == 0) unsafeAtomicAdd(&rs[i], red[0] + red[1] + red[2] + red[3]);
}

// K9: out[i, cols_g[j]] += sum_k pre[i, tblOff_g + k] * dict_g[k, j]; block = (group, i)
__global__ __launch_bounds__(256) void k_lmm_post(const DGroup* __restrict__ groups, const double* __restrict__ pre,
	int totalVals, double* __restrict__ out, int nCols) {
	__shared__ double red[4];
	const DGroup G = dgroup(groups + (blockIdx.x));
	if(G.type == G_UNC) return;
	const int i = blockIdx.y;
	const double* p = pre + (size_t) i * totalVals + G.tblOff;
	for(int j = 0; j < G.nColG; j++) {
		double s = 0.0;
		for(int k = threadIdx.x; k < G.nVals; k += 256) s += p[k] * G.dict[(size_t) k * G.nColG + j];
		s = wave_sum_f64(s);
		if((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
		__syncthreads();
		if(threadIdx.x == 0) unsafeAtomicAdd(&out[(size_t) i * nCols + G.cols[j]], red[0] + red[1] + red[2] + red[3]);
		__syncthreads();
	}
}

// out[i, c] += rowSum[i] * constV[c] (skipped for rowSum == 0, as the reference does); nnz
__global__ __launch_bounds__(256) void k_lmm_finish(double* __restrict__ out, int p, int nCols, const double* __restrict__ rs,
	const double* __restrict__ constV, unsigned long long* __restrict__ nnz) {
	const int64_t idx = (int64_t) blockIdx.x * 256 + threadIdx.x;
	int cnt = 0;
	if(idx < (int64_t) p * nCols) {
		const int i = (int) (idx / nCols), c = (int) (idx - (int64_t) i * nCols);
		double v = out[idx];
		if(rs != nullptr) {
			const double vl = rs[i];
			if(vl != 0.0) v += vl * constV[c];
			out[idx] = v;
		}
		cnt = v != 0.0;
	}
	count_add(nnz, cnt);
}

// Behind a Y %*% X on decoded rows: takes the result out of its stage and counts the non-zeros. The kernels on decoded rows give
// a row that a group does not cover the value 0.0, which an infinite Y turns into NaN; in the reference such a row does not enter the
// group's sums. They report a non-finite Y in *bad, and then the blocks of this kernel form anew, from a group's own rows only, the
// columns whose group leaves rows out or that a constant is added to, row sums times constants apart, as the bin kernels do
// (ColGroupRLE.java:759-796, AOffset.java:288-430); the others have the same sums either way. The flag stays on the
// device: the host looking at it cost 15 - 20 us per call (wait, copy, and the launches behind it), a mixed block of 5,000,011 x 20 by 6 rows
// 114 us per call against 91 us (with an infinity in Y 611, on the bin kernels 1502).
constexpr int LT_THREADS = 512;
constexpr int LT_P = 8;            // rows of Y per look at a group's codes
constexpr int LT_COLS = 64;        // most columns of a block
struct LmmTake {
	const DGroup* groups;
	int nGroups;
	const double* Y;
	int p;
	int64_t nRows;
	double* stage;                 // p x nCols, what the kernel in front has summed; left at zero, like the next three
	double* anew;                  // p x nCols and p row sums, zero
	unsigned long long* bad;
	unsigned long long* count;     // zero
	const double* constV;          // nullptr: no constants
	unsigned long long redo;       // columns that a non-finite Y takes anew
	double* out;
	int nCols;
	unsigned* done;
	unsigned long long* nnz;
};

__global__ __launch_bounds__(LT_THREADS) void k_take_block(const LmmTake A) {
	__shared__ int lastS;
	__shared__ int cntS[LT_THREADS / WAVE];
	__shared__ double sumS[LT_P * (LT_COLS + 1)]; // the block's sums of some rows of Y: by column, then the row sum
	__shared__ int32_t runS[LT_THREADS / WAVE][2 * WAVE + 1]; // per wave: starts of 64 runs and the end of the last, their codes
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = A.p * A.nCols;
	double* const rs = A.anew + n;
	const bool anew = *A.bad != 0 && (A.redo != 0 || A.constV != nullptr);
	const int nTake = min((int) gridDim.x, (n + LT_THREADS * 4 - 1) / (LT_THREADS * 4)); // blocks that take the result out of its stage
	if(!anew && (int) blockIdx.x >= nTake) return;
	if(anew) {
		auto product = [&](auto pTag) { // a few rows of Y per look at a group's codes; a share of the rows and those rows of Y per turn of a block
			constexpr int LP = decltype(pTag)::value;
			const int nY = (A.p + LP - 1) / LP, nParts = max(1, (int) gridDim.x / nY);
			for(int turn = blockIdx.x; turn < nParts * nY; turn += gridDim.x) {
				const int part = turn / nY, i0 = (turn - part * nY) * LP;
				const int64_t r0 = A.nRows * part / nParts, r1 = A.nRows * (part + 1) / nParts;
				const double* y[LP];
#pragma unroll
				for(int i = 0; i < LP; i++) y[i] = A.Y + (size_t) min(i0 + i, A.p - 1) * A.nRows;
				const int np = min(LP, A.p - i0);
				for(int i = tid; i < LP * (LT_COLS + 1); i += LT_THREADS) sumS[i] = 0.0;
				__syncthreads();
				// (4096 waves' adds to a cell in memory, 11.4 ns each, were most of the time: in LDS first)
				auto give_all = [&](const double (&s)[LP], int col) {
#pragma unroll
					for(int i = 0; i < LP; i++)
						if(i < np) {
							const double w = wave_sum_f64(s[i]);
							if(lane == 0) unsafeAtomicAdd(&sumS[i * (LT_COLS + 1) + col], w);
						}
				};
				for(int g = 0; g < A.nGroups; g++) {
					const DGroup G = dgroup(A.groups + g);
					for(int h = 0; h < G.nColG; h++) {
						if((A.redo >> G.cols[h] & 1) == 0) continue;
						double s[LP] = {};
						if(G.type == G_DDC || G.type == G_UNC) {
#pragma unroll 2
							for(int64_t r = r0 + tid; r < r1; r += LT_THREADS) {
								const double x = G.type == G_DDC ? G.dict[(size_t) load_code(G.codes, G.codeWidth, r) * G.nColG + h] : G.dense[(size_t) r * G.nColG + h];
#pragma unroll
								for(int i = 0; i < LP; i++) s[i] += y[i][r] * x;
							}
						}
						else if(G.type == G_RLE && G.nRuns > 0) {
							// Consecutive rows per wave, 64 at a time. The run table comes 64 runs at a time through LDS, where every lane finds its
							// row's: followed in memory lane by lane it takes a gather or more per row.
							int32_t* const start = runS[wave];
							int32_t* const code = start + WAVE + 1;
							const int64_t w0 = r0 + (r1 - r0) * wave / (LT_THREADS / WAVE), w1 = r0 + (r1 - r0) * (wave + 1) / (LT_THREADS / WAVE);
							int base = 0;
							auto window = [&](int64_t row) { // the runs from the one of `row` on
								base = __builtin_amdgcn_readfirstlane(rle_find(G.runStart, G.nRuns, (int32_t) row));
								wave_lds_sync();
								start[lane] = G.runStart[min(base + lane, G.nRuns)];
								code[lane] = G.runCode[min(base + lane, G.nRuns - 1)];
								if(lane == 0) start[WAVE] = G.runStart[min(base + WAVE, G.nRuns)]; // (the last run ends at the last row)
								wave_lds_sync();
							};
							if(w0 < w1) window(w0);
							for(int64_t row0 = w0; row0 < w1; row0 += WAVE) {
								if(start[WAVE] < min(row0 + WAVE, w1)) window(row0); // (a run has a row at least: 64 runs hold 64 rows)
								const int64_t r = min(row0 + lane, w1 - 1);
								int k = 0;
#pragma unroll
								for(int half = WAVE / 2; half > 0; half >>= 1) k += start[k + half] <= r ? half : 0;
								const int c = code[k];
								if(row0 + lane >= w1 || c < 0) continue;
								const double x = G.dict[(size_t) c * G.nColG + h];
#pragma unroll
								for(int i = 0; i < LP; i++) s[i] += y[i][r] * x;
							}
						}
						else if(G.type == G_SDCZ && G.nOffsets > 0) {
							auto take = [&](int64_t row, int idx) {
								const double x = G.dict[(size_t) load_code(G.codes, G.codeWidth, idx) * G.nColG + h];
#pragma unroll
								for(int i = 0; i < LP; i++) s[i] += y[i][row] * x;
							};
							constexpr int CW = SDC_CK / 256, CB = LT_THREADS / WAVE / CW; // waves per chunk, 256 entries each; chunks per block
							static_assert(CB >= 1, "a wave per 256 entries of a chunk");
							if(part == 0 && tid == 0) take(G.first, 0);
							if(wave < CW * CB) for(int c = part * CB + wave / CW; c < G.nCkpt; c += nParts * CB) {
								const OffState st = G.ckpt[c];
								int32_t row = st.row, emit = st.emit, rows[4], didx[4];
								unsigned mask;
								const int64_t base = (int64_t) c * SDC_CK;
								for(int w = 0; w <= wave % CW; w++) {
									if(G.deltaWidth == 1) sdc_decode256<1>(G.deltas, G.nDeltas, base + w * 256, row, emit, rows, didx, mask);
									else sdc_decode256<2>(G.deltas, G.nDeltas, base + w * 256, row, emit, rows, didx, mask);
								}
#pragma unroll
								for(int k = 0; k < 4; k++)
									if(mask & (1u << k)) take(rows[k], didx[k]);
							}
						}
						give_all(s, G.cols[h]);
					}
				}
				if(A.constV != nullptr) {
					double s[LP] = {};
					for(int64_t r = r0 + tid; r < r1; r += LT_THREADS)
#pragma unroll
						for(int i = 0; i < LP; i++) s[i] += y[i][r];
					give_all(s, LT_COLS);
				}
				__syncthreads();
				for(int idx = tid; idx < np * (LT_COLS + 1); idx += LT_THREADS) {
					const int i = idx / (LT_COLS + 1), c = idx % (LT_COLS + 1);
					if(sumS[idx] != 0.0) unsafeAtomicAdd(c < LT_COLS ? A.anew + (size_t) (i0 + i) * A.nCols + c : rs + i0 + i, sumS[idx]); // (a NaN is unequal to zero)
				}
				__syncthreads();
			}
		};
		if(A.p <= 2) product(std::integral_constant<int, 2>());
		else product(std::integral_constant<int, LT_P>());
		asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (see lmm_tail)
		__syncthreads();
		if(tid == 0) lastS = last_block(A.done, gridDim.x);
		__syncthreads();
		if(!lastS) return;
	}
	auto summed = [&](const double* at) {
		return __longlong_as_double((long long) __hip_atomic_load((const unsigned long long*) at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
	};
	int cnt = 0;
	const int step = LT_THREADS * (anew ? 1 : nTake);
	for(int idx = tid + (anew ? 0 : (int) blockIdx.x * LT_THREADS); idx < n; idx += step) {
		double v;
		if(anew) {
			v = A.redo >> (idx % A.nCols) & 1 ? summed(A.anew + idx) : A.stage[idx];
			if(A.constV != nullptr) { // (skipped for a row sum of zero, as in k_lmm_finish)
				const double vl = summed(rs + idx / A.nCols);
				if(vl != 0.0) v += vl * A.constV[idx % A.nCols];
			}
		}
		else v = A.stage[idx];
		A.stage[idx] = 0.0; // (nobody else reads it)
		A.out[idx] = v;
		cnt += v != 0.0;
	}
	cnt = wave_sum_i32(cnt);
	if(lane == 0) cntS[wave] = cnt;
	__syncthreads();
	if(tid == 0) {
		unsigned long long s = 0;
		for(int w = 0; w < LT_THREADS / WAVE; w++) s += (unsigned) cntS[w];
		lastS = 1;
		if(!anew && nTake > 1) {
			atomicAdd(A.count, s);
			asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
			lastS = last_block(A.done, nTake);
			s = __hip_atomic_load(A.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		if(lastS) // (the way that the counter's reader adds up first; the others are cleared below)
			A.nnz[0] = s;
	}
	__syncthreads();
	if(!lastS) return;
	if(tid > 0 && tid < NNZ_WAYS) A.nnz[tid * NNZ_STEP] = 0;
	clear_tickets(A.done);
	if(anew) // (all blocks have taken a ticket: nobody reads these any more)
		for(int i = tid; i < n + A.p; i += LT_THREADS) A.anew[i] = 0.0;
	if(tid == 0) *A.bad = *A.count = 0; // (a report that no column or constant of this block heeds, too: the word is a sum of a call of more rows)
}

// (a kernel, not hipMemsetAsync: a memset node of a captured graph has given wrong results on its replays)
__global__ __launch_bounds__(256) void k_zero(double* __restrict__ p, size_t n) {
	for(size_t i = (size_t) blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t) gridDim.x * 256) p[i] = 0.0;
}

int launch_zero(cla_block* b, double* p, size_t n) {
	hipLaunchKernelGGL(k_zero, dim3((unsigned) std::min<size_t>((n + 255) / 256, 1024)), dim3(256), 0, b->stream, p, n);
	CLA_HIP(hipGetLastError());
	return 0;
}

int launch_lmm_take(cla_block* b, const double* dY, int p, double* ws, double* dOut, unsigned long long* dNnz) {
	const size_t n = (size_t) p * b->nCols;
	LmmTake A;
	A.groups = b->dGroups; A.nGroups = (int) b->groups.size();
	A.Y = dY; A.p = p; A.nRows = b->nRows; A.nCols = b->nCols;
	A.stage = ws; A.anew = ws + n; A.bad = (unsigned long long*) (ws + 2 * n + p); A.count = (unsigned long long*) (ws + 2 * n + p + 1);
	A.constV = b->hasConst ? b->dConstV : nullptr;
	A.redo = ~0ull; // (at most LT_COLS columns)
	for(const HostGroup& H : b->groups)
		if(H.d.type == G_DDC || H.d.type == G_UNC)
			for(int c : H.cols)
				if(b->constV[c] == 0.0) A.redo &= ~(1ull << c);
	if(b->nCols < LT_COLS) A.redo &= (1ull << b->nCols) - 1;
	A.out = dOut; A.done = b->lmm_ticket(); A.nnz = dNnz;
	const unsigned grid = (unsigned) std::max<int64_t>(1, std::min<int64_t>((b->nRows + 1023) / 1024 * ((p + LT_P - 1) / LT_P), b->nRows < 2000000 ? g_numCU : 2 * g_numCU));
	Prof pf(b, "k_take_block", grid, LT_THREADS, 0, 0);
	hipLaunchKernelGGL(k_take_block, dim3(grid), dim3(LT_THREADS), 0, b->stream, A);
	CLA_HIP(hipGetLastError());
	return 0;
}

// dOut != nullptr (whole-block calls): groups whose products can be summed directly write into dOut
// and leave their part of dPre zero.
static int run_preagg(cla_block* b, const double* dY, int p, double* dPre, int onlyGroup, double* dOut) {
	const int nG = (int) b->groups.size();
	const int64_t nRows = b->nRows;
	hipStream_t st = b->stream;
	// all groups DDC with byte codes in one arena: one persistent kernel for the whole block
	if(onlyGroup < 0) {
		const int r = launch_lmm_u8(b, dY, p, dPre);
		if(r == 0) b->preUsed = true;
		if(r <= 0) return r;
	}
	// row-parallel groups (DDC, RLE) in LDS-sized slabs
	int64_t rowsPerBlock = 64 * 1024;
	while(rowsPerBlock > 4096 && (nRows + rowsPerBlock - 1) / rowsPerBlock * p < (int64_t) g_numCU * 2) rowsPerBlock /= 2;
	const unsigned gridRows = (unsigned) std::max<int64_t>((nRows + rowsPerBlock - 1) / rowsPerBlock, 1);
	int g = 0;
	while(g < nG) {
		const DGroup& G = b->groups[g].d;
		const bool rowPar = (G.type == G_DDC || G.type == G_RLE) && (onlyGroup < 0 || onlyGroup == g);
		if(!rowPar) { g++; continue; }
		const int direct = (size_t) G.nVals * 8 > (size_t) 60 * 1024;
		int g1 = g;
		size_t bytes = 0;
		const size_t budget = (size_t) G.nVals * 8 > LMM_BIN_BYTES ? (size_t) G.nVals * 8 : LMM_BIN_BYTES;
		while(g1 < nG) {
			const DGroup& H = b->groups[g1].d;
			if(!((H.type == G_DDC || H.type == G_RLE) && (onlyGroup < 0 || onlyGroup == g1))) break;
			if(bytes + (size_t) H.nVals * 8 > budget) break;
			bytes += (size_t) H.nVals * 8;
			g1++;
			if(direct) break;
		}
		if(nRows > 0) {
			b->preUsed = true;
			const size_t lds = direct ? 0 : bytes;
			Prof pf(b, "k_lmm_preagg_rows", (long) gridRows * p, LMM_THREADS, (long) lds, 0);
			CLA_HIP(allow_full_lds((const void*) k_lmm_preagg_rows));
			hipLaunchKernelGGL(k_lmm_preagg_rows, dim3(gridRows, p), dim3(LMM_THREADS), lds, st, b->dGroups, g, g1, dY,
				nRows, rowsPerBlock, dPre, b->totalVals, direct);
		}
		g = g1;
	}
	// SDCZeros groups: all lists walked tile by tile with the Y tile in LDS; the
	// per-group chunk kernel below only serves dictionaries too large for LDS bins
	{
		const int r = nRows > 0 ? launch_lmm_sdc_tiles(b, dY, p, dPre, onlyGroup, dOut) : 0;
		if(r < 0) return r;
		if(r == 0) { CLA_HIP(hipGetLastError()); return 0; }
	}
	for(g = 0; g < nG; g++) {
		const DGroup& G = b->groups[g].d;
		if(G.type != G_SDCZ || G.nOffsets == 0 || (onlyGroup >= 0 && onlyGroup != g)) continue;
		const int direct = (size_t) G.nVals * 8 > (size_t) 60 * 1024;
		int cpb = 1;
		while(cpb < 16 && (G.nCkpt + cpb - 1) / cpb * p > g_numCU * 8) cpb *= 2;
		const unsigned grid = (unsigned) std::max((G.nCkpt + cpb - 1) / cpb, 1);
		const size_t bytes = direct ? 0 : (size_t) G.nVals * 8;
		const double algo = (double) G.nDeltas * G.deltaWidth + (double) G.nOffsets * (G.codeWidth + 8.0);
		b->preUsed = true;
		Prof pf(b, "k_lmm_preagg_sdc", (long) grid * p, 256, (long) bytes, algo);
		if(G.deltaWidth == 1) {
			CLA_HIP(allow_full_lds((const void*) k_lmm_preagg_sdc<1>));
			hipLaunchKernelGGL(k_lmm_preagg_sdc<1>, dim3(grid, p), dim3(256), bytes, st, b->dGroups, g, dY, nRows, cpb, dPre,
				b->totalVals, direct);
		}
		else {
			CLA_HIP(allow_full_lds((const void*) k_lmm_preagg_sdc<2>));
			hipLaunchKernelGGL(k_lmm_preagg_sdc<2>, dim3(grid, p), dim3(256), bytes, st, b->dGroups, g, dY, nRows, cpb, dPre,
				b->totalVals, direct);
		}
	}
	CLA_HIP(hipGetLastError());
	return 0;
}

int launch_preagg(cla_block* b, int group, const double* dY, int p, double* dPre) {
	clear_stats(b);
	const DGroup& G = b->groups[group].d;
	if(G.type == G_UNC) { set_error("preagg: group %d is uncompressed", group); return -CLA_ERR_UNSUPPORTED; }
	// aggregate into a full-width scratch (p x totalVals) and slice the group's bins out
	int rc = ensure_tables(b, (size_t) p * b->totalVals);
	if(rc) return rc;
	CLA_HIP(hipMemsetAsync(b->dTables, 0, sizeof(double) * (size_t) p * b->totalVals, b->stream));
	if((rc = run_preagg(b, dY, p, b->dTables, group, nullptr))) return rc;
	CLA_HIP(hipMemcpy2DAsync(dPre, sizeof(double) * (size_t) G.nVals, b->dTables + G.tblOff,
		sizeof(double) * (size_t) b->totalVals, sizeof(double) * (size_t) G.nVals, (size_t) p, hipMemcpyDeviceToDevice,
		b->stream));
	return 0;
}

int launch_lmm(cla_block* b, const double* dY, int p, double* dOut, unsigned long long* dNnz) {
	const int nG = (int) b->groups.size();
	const int64_t nRows = b->nRows;
	hipStream_t st = b->stream;
	clear_stats(b);
	// mixed blocks of few columns: one pass on the decoded Gram kernel
	{
		const int j = launch_lmm_joint(b, dY, p, dOut, dNnz);
		if(j <= 0) return j;
	}
	int rc = ensure_tables(b, (size_t) p * b->totalVals + (size_t) p + 8);
	if(rc) return rc;
	double* dPre = b->dTables;
	double* dRs = b->dTables + (size_t) p * b->totalVals;
	CLA_HIP(hipMemsetAsync(dOut, 0, sizeof(double) * (size_t) p * b->nCols, st));
	// Blocks that one kernel serves whole (byte-code DDC groups of one column; SDCZeros lists only) and that have no
	// constants to add: that kernel also counts the result's non-zeros, and nothing else runs.
	b->preUsed = false;
	b->lmmTailWanted = !b->hasConst && dNnz == b->dCounters && (int64_t) p * b->nCols < ((int64_t) 1 << 30);
	b->lmmTailDone = false;
	// One row of Y: up to 1.5 M rows the matrix-core form (250,007 x 100 19 against 32 us, 1,000,003 x 54 29 against 32), beyond
	// the vector form, which streams the codes in whole lines (2,000,003 x 54 38 against 44, 8,000,001 x 100 172 against 242).
	int dot = 1;
	if(p == 1 && nRows > 1500000) dot = launch_lmm_u8_vec(b, dY, dOut);
	if(dot == 1 && nRows > 0) dot = launch_lmm_u8_dot(b, dY, p, dOut);
	if(dot == 1 && nRows > 0 && p == 1) dot = launch_lmm_q1_short(b, dY, dOut);
	if(dot < 0) return dot;
	if(dot != 0 && nRows > 0 && b->lmmTailWanted && b->opt.sdcLanes && !b->dictNonFinite && b->hasSdc && !b->hasUnc && !b->hasRle) {
		bool onlyLists = true;
		for(int g = 0; g < nG && onlyLists; g++) onlyLists = b->groups[g].d.type == G_SDCZ && b->groups[g].d.nOffsets > 0;
		if(onlyLists) {
			if((rc = sdc_plan_all(b))) return rc;
			const int r = launch_lmm_sdc_lanes(b, dY, p, dOut);
			if(r < 0) return r;
		}
	}
	b->lmmTailWanted = false;
	if(b->lmmTailDone) {
		CLA_HIP(hipGetLastError());
		return 0;
	}
	CLA_HIP(hipMemsetAsync(dPre, 0, sizeof(double) * ((size_t) p * b->totalVals + (size_t) p), st));
	CLA_HIP(hipMemsetAsync(dNnz, 0, NNZ_BYTES, st));
	if(dot != 0 && (rc = run_preagg(b, dY, p, dPre, -1, dOut))) return rc;

	int64_t rowsPerBlock = 256 * 1024;
	while(rowsPerBlock > 8192 && (nRows + rowsPerBlock - 1) / rowsPerBlock * p < (int64_t) g_numCU * 2) rowsPerBlock /= 2;
	const unsigned gridRows = (unsigned) std::max<int64_t>((nRows + rowsPerBlock - 1) / rowsPerBlock, 1);
	for(int g = 0; g < nG; g++) {
		const DGroup& G = b->groups[g].d;
		if(G.type != G_UNC || nRows == 0 || G.nColG == 0) continue;
		const int nbY = (p + 15) / 16, nbC = ((G.nColG + 15) / 16 + LU_NBJ - 1) / LU_NBJ;
		int64_t rpb = 16384;
		while(rpb > 1024 && (nRows + rpb - 1) / rpb * nbY * nbC < (int64_t) g_numCU * 8) rpb /= 2;
		const dim3 grid((unsigned) ((nRows + rpb - 1) / rpb), (unsigned) nbY, (unsigned) nbC);
		Prof pf(b, "k_lmm_unc", (long) grid.x * grid.y * grid.z, 256, 0, (double) nRows * G.nColG * 8);
		hipLaunchKernelGGL(k_lmm_unc, grid, dim3(256), 0, st, b->dGroups, g, dY, p, nRows, rpb, dOut, b->nCols);
	}
	if(b->hasConst && nRows > 0) {
		Prof pf(b, "k_lmm_rowsum", (long) gridRows * p, 256, 0, 0);
		hipLaunchKernelGGL(k_lmm_rowsum, dim3(gridRows, p), dim3(256), 0, st, dY, nRows, rowsPerBlock, dRs);
	}
	if(nG > 0 && dot != 0 && b->preUsed) {
		Prof pf(b, "k_lmm_post", (long) nG * p, 256, 0, 0);
		hipLaunchKernelGGL(k_lmm_post, dim3(nG, p), dim3(256), 0, st, b->dGroups, dPre, b->totalVals, dOut, b->nCols);
	}
	{
		const int64_t n = (int64_t) p * b->nCols;
		Prof pf(b, "k_lmm_finish", (long) ((n + 255) / 256), 256, 0, 0);
		hipLaunchKernelGGL(k_lmm_finish, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, dOut, p, b->nCols,
			b->hasConst ? dRs : nullptr, b->dConstV, dNnz);
	}
	CLA_HIP(hipGetLastError());
	return 0;
}

// CLALibMMChain.mmChain: tmp = X %*% v ; tmp *= w (XtwXv) or tmp -= w (XtXvy) ; out = t(tmp) %*% X.
__global__ __launch_bounds__(256) void k_mul_inplace(double* __restrict__ x, const double* __restrict__ w, int64_t n) {
	const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
	if(i < n) x[i] *= w[i];
}

__global__ __launch_bounds__(256) void k_sub_inplace(double* __restrict__ x, const double* __restrict__ y, int64_t n) {
	const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
	if(i < n) x[i] -= y[i];
}

// Small vectors of a host-pointer call on their way through pinned host memory: the device reads the operand and writes the result and the count
// itself, so that the host waits once and no copy engine is started (two copies from and one to pageable memory and two waits of the
// host took 32 of the 48 us of a chain of 250,007 x 54).
__global__ __launch_bounds__(512) void k_fetch(double* __restrict__ dst, const double* __restrict__ host, int n) {
	if((int) threadIdx.x < n) dst[threadIdx.x] = host[threadIdx.x];
}

__global__ __launch_bounds__(512) void k_deliver(double* __restrict__ host, const double* __restrict__ src, int n, unsigned long long* __restrict__ hostCount,
	const unsigned long long* __restrict__ nnz) {
	if((int) threadIdx.x < n) host[threadIdx.x] = src[threadIdx.x];
	if(threadIdx.x < NNZ_WAYS) {
		static_assert(NNZ_WAYS == WAVE, "a way per lane");
		long long s = (long long) nnz[threadIdx.x * NNZ_STEP];
		for(int o = WAVE / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
		if(threadIdx.x == 0) *hostCount = (unsigned long long) s;
	}
}

static_assert(HOST_VEC_MAX <= 512, "an element per thread");

// v (host, n <= HOST_VEC_MAX) into dst; the pinned buffer is the call's until it has waited for the stream
int launch_fetch(cla_block* b, double* dst, const double* v, int n) {
	double* const host = (double*) b->hCounters + 1;
	memcpy(host, v, (size_t) n * sizeof(double));
	hipLaunchKernelGGL(k_fetch, dim3(1), dim3(512), 0, b->stream, dst, host, n);
	CLA_HIP(hipGetLastError());
	return 0;
}

// Where a chain's only kernel writes for deliver(): a launch less (250,007 x 54 34.6 -> 33.2 us, 3,085 x 23 26.8 -> 24.4).
ChainHost chain_host(cla_block* b) {
	ChainHost h;
	h.out = (double*) b->hCounters + 1 + HOST_VEC_MAX;
	h.count = b->hCounters;
	return h;
}

// src (n <= HOST_VEC_MAX) into out (host); waits for the stream and returns the count in dNnz. there: both are on their way to chain_host(b) already.
int64_t deliver(cla_block* b, double* out, const double* src, int n, const unsigned long long* dNnz, bool there) {
	double* const host = (double*) b->hCounters + 1 + HOST_VEC_MAX;
	if(!there) hipLaunchKernelGGL(k_deliver, dim3(1), dim3(512), 0, b->stream, host, src, n, b->hCounters, dNnz);
	CLA_HIP(hipGetLastError());
	CLA_HIP(hipStreamSynchronize(b->stream));
	memcpy(out, host, (size_t) n * sizeof(double));
	return (int64_t) b->hCounters[0];
}

int launch_mmchain(cla_block* b, const double* dV, const double* dW, int ctype, double* dOut, unsigned long long* dNnz, ChainHost* host) {
	const int64_t nRows = b->nRows;
	{
		ChainHost none;
		ChainHost& to = host != nullptr ? *host : none;
		int r = launch_chain_u8(b, dV, dW, ctype, dOut, dNnz, to);
		if(r == 1) r = launch_chain_sdc(b, dV, dW, ctype, dOut, dNnz, to);
		if(r == 1) r = launch_chain_pairs(b, dV, dW, ctype, dOut, dNnz, to);
		to.done = r == 0;
		if(r <= 0) return r;
	}
	// the intermediate vector has a workspace of its own: the multiplies below may resize the shared scratch
	int rc = ensure_chain(b, (size_t) std::max<int64_t>(nRows, 1));
	if(rc) return rc;
	double* tmp = b->dChain;
	// (the weights are read where X %*% v writes its rows: a pass of its own over 10 M rows takes 40 us)
	RowOp op;
	if(ctype != 0) { op.w = dW; op.minus = ctype == 2; }
	if((rc = launch_rmm(b, dV, 1, tmp, dNnz, 0, nullptr, 0, &op))) return rc;
	b->nnzSlot = 0; // the left multiply below counts the result's non-zeros into dNnz
	std::vector<KernelStat> first;
	first.swap(b->lastStats);
	if(ctype == 1 && !op.done && nRows > 0)
		hipLaunchKernelGGL(k_mul_inplace, dim3((unsigned) ((nRows + 255) / 256)), dim3(256), 0, b->stream, tmp, dW, nRows);
	if(ctype == 2 && !op.done && nRows > 0)
		hipLaunchKernelGGL(k_sub_inplace, dim3((unsigned) ((nRows + 255) / 256)), dim3(256), 0, b->stream, tmp, dW, nRows);
	rc = launch_lmm(b, tmp, 1, dOut, dNnz);
	b->lastStats.insert(b->lastStats.begin(), first.begin(), first.end());
	return rc;
}

} // namespace cla
