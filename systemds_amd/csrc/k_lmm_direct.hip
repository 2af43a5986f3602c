// Y %*% X of blocks that are a few "varying" columns next to run-length columns (the shape of k_tsmm_direct, whose plan this
// kernel shares), on the vector unit.
//
// Lane = two consecutive rows, read straight from their streams: a wave takes 128 rows at a time. A varying column is looked up
// in LDS once for all P rows of Y: acc[i][c] += y_i x_c, lane-private sums reduced over the lanes once at the end. A
// run-length column is never looked up per row: the rows between two run ends (of any column) are a stretch on which all of
// them are constant, and a stretch adds its sums of y times the columns' values. The lanes fold their P sums eight to one first,
// so that a stretch adds one value per lane to each column's cell in LDS.
// (Not by summation by parts, which adds only where a column's own run ends, its value's step times the sum of y so far: rows on
// which the column is zero enter such sums and must cancel again. A y of 1e14 on one of them left an error of 4e-7 of the sum of |y||x|.)
//
// Why not the tile kernel on the matrix cores (k_lmm_decode, which it precedes): Y %*% X has as few multiply-adds as P times
// the columns per row and is bound by its streams; the tiles went through LDS twice, the matrix instruction pads both P and the
// columns to 16, and the waves walked the stages in step.
//
// More rows of Y than 6 (8 where at most 8 columns vary) take passes (the sums of 12 columns by 6 rows are 144 registers; two
// waves per SIMD; what spills from two rows per lane there cost 60 of 154 us, so such shapes take one).
// Bound: HBM (Y once, the streams once per pass; vector memory path 67 % busy, vector issue 40 %), 14 us of start and end. 5,000,011 x
// 20 (8 run-length, 8 two-byte, 2 offset-list, 2 dense columns) by 6 rows of Y 88 us (414 MB: 4.7 TB/s). Calls, with the fill in
// front and k_take_block behind (k_lmm_decode with a host's look at Y; this kernel with one): by 6 301, 114 -> 91 us, by 13 241 -> 215; 1,000,000
// rows by 6 58 -> 32, 100,000 by 2 40 -> 15.
#include "../../include/cla_hip.h"
#include "cla_gdr.hpp"
#include <algorithm>

namespace cla {

constexpr int LD_THREADS = 512;
constexpr int LD_WAVES = LD_THREADS / WAVE;
constexpr int LD_PMAX = 8;
constexpr int LD_REBASE = 128;              // most steps that a stretch's sums run over (a power of two)
constexpr int LD_WDOUBLES = 64 + 32 + RC_MAX * 64; // per wave: window values, window ends, the run-length columns' cells

typedef double f64x2_ld __attribute__((ext_vector_type(2), aligned(8))); // (a row of Y starts at any multiple of 8 bytes)

// Rows per lane and step: two (half as many load instructions) where their values fit the registers next to the sums.
constexpr int ld_rows(int nv, int p) { return nv * p > 54 ? 1 : 2; }

// NC code columns, ND dense ones, P rows of Y, R rows per lane and step
template <int NC, int ND, int P, int R>
__global__ __launch_bounds__(LD_THREADS, 2) void k_lmm_direct(const GdrArgs A, const LdCols L, const double* __restrict__ Y,
	double* __restrict__ out, unsigned long long* __restrict__ badY) {
	extern __shared__ __align__(16) double smem[];
	constexpr int NV = NC + ND;
	constexpr int LD_CH = WAVE * R;             // rows per wave and step
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const char* const ldsBytes = (const char*) smem;
	double* const sums = smem + A.valDoubles;                       // P x (NV + RC_MAX)
	double* const wbase = sums + P * (NV + RC_MAX) + wave * LD_WDOUBLES;
	double* const winVal = wbase;
	int32_t* const winEnd = (int32_t*) (wbase + 64);
	double* const cells = wbase + 96 + lane;                        // column a: cells[64 a]

	gdr_copy_vals<LD_THREADS>(smem, A.vals, A.valDoubles);
	for(int i = tid; i < P * (NV + RC_MAX); i += LD_THREADS) sums[i] = 0.0;
#pragma unroll
	for(int a = 0; a < RC_MAX; a++) cells[64 * a] = 0.0;
	__syncthreads();

	const int32_t nRows = (int32_t) A.nRows;
	const int nChunks = (nRows + LD_CH - 1) / LD_CH;
	const int nW = gridDim.x * LD_WAVES, gw = blockIdx.x * LD_WAVES + wave;
	const int ch0 = (int) ((int64_t) nChunks * gw / nW), ch1 = (int) ((int64_t) nChunks * (gw + 1) / nW);
	const int nR = A.nR;
	if(ch0 < ch1) {
		double acc[NV][P], S[P];
#pragma unroll
		for(int i = 0; i < P; i++) {
			S[i] = 0.0;
#pragma unroll
			for(int c = 0; c < NV; c++) acc[c][i] = 0.0;
		}
		RunCursors rc;
		rc.start(A.runs, nR, winEnd, winVal, ch0 * LD_CH, lane);
		int32_t eNext = rc.next_end();
		bool bad = false;

		const bool fb0 = (lane & 1) != 0, fb1 = (lane & 2) != 0, fb2 = (lane & 4) != 0;
		// lane k of every group of eight: the group's sum of el(k), k < P
		auto fold = [&](auto el) __attribute__((always_inline)) {
			double w[4], u[2];
#pragma unroll
			for(int j = 0; j < 4; j++) {
				const double lo = 2 * j < P ? el(2 * j < P ? 2 * j : 0) : 0.0, hi = 2 * j + 1 < P ? el(2 * j + 1 < P ? 2 * j + 1 : 0) : 0.0;
				w[j] = (fb0 ? hi : lo) + gdr_xchg1(fb0 ? lo : hi);
			}
#pragma unroll
			for(int i = 0; i < 2; i++) u[i] = (fb1 ? w[2 * i + 1] : w[2 * i]) + gdr_xchg2(fb1 ? w[2 * i] : w[2 * i + 1]);
			return (fb2 ? u[1] : u[0]) + gdr_xchg4(fb2 ? u[0] : u[1]);
		};
		// A stretch of rows on which every run-length column is constant ends (el(i): the lane's sums of y over it): each column
		// takes its value times the stretch's sums. (Unused cursors hold the value 0.)
		auto stretch = [&](auto el) __attribute__((always_inline)) {
			const double f = fold(el);
			bad |= !(__builtin_fabs(f) <= 1.7976931348623157e308); // (a value of y that is not finite stays in its sum)
			auto take = [&](auto a0Tag) __attribute__((always_inline)) { // four columns, their cells requested together
				constexpr int a0 = decltype(a0Tag)::value;
				double h[4];
#pragma unroll
				for(int a = 0; a < 4; a++) h[a] = cells[64 * (a0 + a)];
#pragma unroll
				for(int a = 0; a < 4; a++) cells[64 * (a0 + a)] = __builtin_fma(f, rc.value(a0 + a), h[a]);
			};
			if(nR > 0) take(std::integral_constant<int, 0>());
			if(nR > 4) take(std::integral_constant<int, 4>());
		};
		auto restart = [&]() __attribute__((always_inline)) {
			stretch([&](int i) __attribute__((always_inline)) { return S[i]; });
#pragma unroll
			for(int i = 0; i < P; i++) S[i] = 0.0;
		};

		// the word that holds the lane's codes, for streams of two bytes and of one, and the place in it
		const uint32_t off2 = (uint32_t) (lane * R * 2) & ~3u, off1 = (uint32_t) (lane * R) & ~3u;
		const uint32_t sh2 = (uint32_t) (lane * R * 2 & 3) * 8u, sh1 = (uint32_t) (lane * R & 3) * 8u;
		// one step: rows s0 .. s0 + LD_CH - 1; tail: rows behind the end of the matrix count as zeros
		auto chunk = [&](int ch, auto tailTag) __attribute__((always_inline)) {
			constexpr bool TAIL = decltype(tailTag)::value;
			const int32_t s0 = ch * LD_CH, row = s0 + R * lane;
			uint32_t raw[NC];
			double xd[R][ND > 0 ? ND : 1], y[R][P];
			auto in = [&](int h) { return TAIL ? min(row + h, nRows - 1) : row + h; };
			// everything the step reads is requested first (scalar bases, 32-bit offsets)
#pragma unroll
			for(int c = 0; c < NC; c++) {
				const LdCol& C = L.c[c];
				if(TAIL) raw[c] = *(const uint32_t*) (C.src + ((size_t) (uint32_t) in(0) * (uint32_t) C.stride & ~(size_t) 3)); // (a stream ends in whole words)
				else raw[c] = *(const uint32_t*) (C.src + (size_t) (uint32_t) s0 * (uint32_t) C.stride + (C.stride == 2 ? off2 : off1));
			}
#pragma unroll
			for(int i = 0; i < P; i++) {
				const double* yi = Y + (size_t) i * nRows;
				if(!TAIL && R == 2) {
					const f64x2_ld d = *(const f64x2_ld*) (yi + s0 + 2 * lane);
					y[0][i] = d.x; y[R - 1][i] = d.y;
				}
				else {
#pragma unroll
					for(int h = 0; h < R; h++) y[h][i] = yi[in(h)];
				}
			}
#pragma unroll
			for(int c = 0; c < ND; c++) {
				const LdCol& C = L.c[NC + c];
				const uint8_t* p = C.src + (size_t) (uint32_t) s0 * (uint32_t) C.stride;
#pragma unroll
				for(int h = 0; h < R; h++) xd[h][c] = *(const double*) (p + (uint32_t) (in(h) - s0) * (uint32_t) C.stride);
			}
			__builtin_amdgcn_sched_barrier(0);
			if(TAIL) {
#pragma unroll
				for(int i = 0; i < P; i++)
#pragma unroll
					for(int h = 0; h < R; h++) y[h][i] = row + h < nRows ? y[h][i] : 0.0;
				// (the value beside such a zero as well: the last row, which stands in for the rows behind it, may hold an infinity)
#pragma unroll
				for(int c = 0; c < ND; c++)
#pragma unroll
					for(int h = 0; h < R; h++) xd[h][c] = row + h < nRows ? xd[h][c] : 0.0;
			}
#pragma unroll
			for(int h = 0; h < R; h++) { // (one row after the other: both rows' values do not fit the registers next to the sums)
				double x[NC];
#pragma unroll
				for(int c = 0; c < NC; c++) {
					const LdCol& C = L.c[c];
					uint32_t w = raw[c];
					if(TAIL) w >>= ((uint32_t) in(0) * (uint32_t) C.stride & 3u) * 8u;
					else w >>= C.stride == 2 ? sh2 : sh1;
					if(h) w >>= 8 * C.stride;
					uint32_t code = w & C.mask;
					if(TAIL) code = row + h < nRows ? code : 0u; // (behind the last row: never an index)
					x[c] = *(const double*) (ldsBytes + C.base8 + (code << 3));
					if(TAIL) x[c] = row + h < nRows ? x[c] : 0.0; // (a column's constant may be infinite)
				}
#pragma unroll
				for(int c = 0; c < NC; c++)
#pragma unroll
					for(int i = 0; i < P; i++) acc[c][i] = __builtin_fma(y[h][i], x[c], acc[c][i]);
#pragma unroll
				for(int c = 0; c < ND; c++)
#pragma unroll
					for(int i = 0; i < P; i++) acc[NC + c][i] = __builtin_fma(y[h][i], xd[h][c], acc[NC + c][i]);
				// (the empty asm keeps the multiply-adds here: moved behind the run ends below they would keep all values alive)
#pragma unroll
				for(int c = 0; c < NV; c++)
#pragma unroll
					for(int i = 0; i < P; i++) asm volatile("" : "+v"(acc[c][i]));
				__builtin_amdgcn_sched_barrier(0);
			}
			while(eNext < s0 + LD_CH) { // (uniform) runs that end inside the step: the rows in front of the end leave the sums
				const bool m0 = row < eNext, m1 = row + 1 < eNext;
				stretch([&](int i) __attribute__((always_inline)) { return S[i] + (R == 1 ? (m0 ? y[0][i] : 0.0) : (m0 ? y[0][i] : 0.0) + (m1 ? y[R - 1][i] : 0.0)); });
#pragma unroll
				for(int i = 0; i < P; i++) {
					S[i] = 0.0;
					y[0][i] = m0 ? 0.0 : y[0][i];
					if(R > 1) y[R - 1][i] = m1 ? 0.0 : y[R - 1][i];
				}
				rc.advance(eNext, lane);
				eNext = rc.next_end();
			}
#pragma unroll
			for(int i = 0; i < P; i++) S[i] += R == 1 ? y[0][i] : y[0][i] + y[R - 1][i];
		};
		const int chFull = min(ch1, nRows / LD_CH);
		for(int chB = ch0; chB < chFull; chB += LD_REBASE) {
			const int chE = min(chB + LD_REBASE, chFull);
			for(int ch = chB; ch < chE; ch++) chunk(ch, std::false_type());
			restart();
		}
		if(chFull < ch1) {
			chunk(chFull, std::true_type());
			restart();
		}
		if(__ballot(bad) != 0 && lane == 0) atomicOr(badY, 1ull);

		// the wave's sums into the block's
#pragma unroll
		for(int c = 0; c < NV; c++) { // lane k of every group of eight: its group's share of row k of Y
			const double f = fold([&](int i) __attribute__((always_inline)) { return acc[c][i]; });
			if((lane & 7) < P) unsafeAtomicAdd(&sums[(lane & 7) * (NV + RC_MAX) + c], f);
		}
		for(int a = 0; a < nR; a++)
			if((lane & 7) < P) unsafeAtomicAdd(&sums[(lane & 7) * (NV + RC_MAX) + NV + a], cells[64 * a]);
	}
	__syncthreads();
	for(int idx = tid; idx < P * (NV + RC_MAX); idx += LD_THREADS) {
		const int i = idx / (NV + RC_MAX), c = idx - i * (NV + RC_MAX);
		const int col = c < NV ? L.c[c].col : c - NV < nR ? A.runs[c - NV].col : -1;
		if(col >= 0 && sums[idx] != 0.0) unsafeAtomicAdd(&out[(size_t) i * A.nCols + col], sums[idx]);
	}
}

// dOut (p x nCols, zeroed) += Y %*% D of the decoded rows, constants included; *dBad is set when Y holds a value that is not
// finite (dOut is then not used, see k_take_block). Returns 1 when the block is not of this kernel's shape.
int launch_lmm_direct(cla_block* b, const double* dY, int p, double* dOut, unsigned long long* dBad) {
	if(!b->opt.tsmmDirect || b->crossSplit > 0 || b->crossBlocks > 0) return 1;
	const GdrPlan* P = nullptr;
	if(const int rc = gdr_plan(b, P)) return rc;
	const int nc = P->ldNC, nd = P->ldND;
	if(P->rc || nc == 0) return 1;
	const int most = nc + nd > 8 ? 6 : LD_PMAX; // rows of Y per pass
	const int passes = (p + most - 1) / most;
	// A pass costs 14 us before its first row; the tile kernel takes 16 rows of Y in one (500,000 x 11 by 11 rows 40 against 47 us,
	// 100,003 x 20 by 6 29 against 20; 5,000,011 x 20 by 16 332 against 247).
	if(passes > 1 && b->nRows <= (int64_t) 500000 * (passes - 1)) return 1;
	// A run end takes 0.24 - 0.32 ns of a pass (by 1 and 6 rows of Y, all waves together), the tile kernel hardly notices it. One to six rows
	// and a pass is where they met when that kernel tested the code width on every row; it has become faster since and they meet at
	// one to ten by 6 rows of Y, one to eight by 1 (in us here / there: 3,000,017 rows by 6, 8 run-length columns of mean run 48 228 / 145,
	// 66 178 / 148, 100 130 / 150; 4 of 24 200 / 135, of 48 122 / 137; 2 of 12 211 / 133, of 24 122 / 131; by 1, 8 of 66 132 / 134; 300,007 rows
	// by 6, 4 of 24 42 / 37, of 48 30 / 38). The line has been left.
	if(P->runEnds * passes * 6 > b->nRows) return 1;
	const size_t lds = ((size_t) P->A.valDoubles + LD_PMAX * (nc + nd + RC_MAX) + (size_t) LD_WAVES * LD_WDOUBLES) * 8;
	if(lds > (size_t) std::min(g_ldsPerBlock, 160 * 1024)) return 1;
	for(int k = 0, p0 = 0; k < passes; k++) {
		const int ph = p / passes + (k < p % passes ? 1 : 0);
		const double* y = dY + (size_t) p0 * b->nRows;
		double* out = dOut + (size_t) p0 * b->nCols;
		const int rows = WAVE * ld_rows(nc + nd, ph);
		const int nChunks = (int) ((b->nRows + rows - 1) / rows);
		const unsigned grid = (unsigned) std::max(1, std::min((nChunks + LD_WAVES - 1) / LD_WAVES, g_numCU));
		Prof pf(b, "k_lmm_direct", grid, LD_THREADS, (long) lds, (double) b->device_bytes_cached + (double) b->nRows * ph * 8);
		bool launched = false;
#define LD_CASE_P(NCV, NDV, PV)                                                                                                \
	if(!launched && nc == NCV && nd == NDV && ph == PV) {                                                                      \
		const auto kern = k_lmm_direct<NCV, NDV, PV, ld_rows(NCV + NDV, PV)>;                                                  \
		CLA_HIP(allow_full_lds((const void*) kern));                                                                           \
		hipLaunchKernelGGL(kern, dim3(grid), dim3(LD_THREADS), lds, b->stream, P->A, P->ld, y, out, dBad);                     \
		launched = true;                                                                                                       \
	}
#define LD_CASE(NCV, NDV) \
	LD_CASE_P(NCV, NDV, 1) LD_CASE_P(NCV, NDV, 2) LD_CASE_P(NCV, NDV, 3) LD_CASE_P(NCV, NDV, 4) LD_CASE_P(NCV, NDV, 5) LD_CASE_P(NCV, NDV, 6)
#define LD_CASE_8(NCV, NDV) LD_CASE(NCV, NDV) LD_CASE_P(NCV, NDV, 7) LD_CASE_P(NCV, NDV, 8)
		LD_CASE_8(4, 0) LD_CASE_8(4, 2) LD_CASE_8(4, 4) LD_CASE_8(8, 0) LD_CASE(8, 2) LD_CASE(8, 4) LD_CASE(10, 2) LD_CASE(12, 0)
#undef LD_CASE_8
#undef LD_CASE
#undef LD_CASE_P
		if(!launched) return 1;
		CLA_HIP(hipGetLastError());
		p0 += ph;
	}
	return 0;
}

} // namespace cla
