// t(X) %*% X of a block whose groups are all DDC with one code width (one or two bytes), 13 to 128 columns, as the Gram
// matrix of the decoded rows: every row is decoded once, into a tile of doubles in LDS that all waves multiply from.
//
// A workgroup of 8 waves (one per CU or two, gt_blocks_per_cu) takes a contiguous share of the rows in tiles of R = 32 m rows, two tile buffers in
// LDS. Decoding is dealt by (16 columns, 32 rows): lane (k, c), k = lane / 16, c = lane % 16, holds 8 consecutive codes of
// column c, looks them up (in LDS where the column block's dictionaries fit beside the tiles, [code][16 columns], else
// straight in global memory) and writes the values to its rows of the tile. Multiplying: lane (k, c) reads X[row 4 s + k, 16 b + c],
// which is both operands of v_mfma_f64_16x16x4 for column block b, so a step of 4 rows costs one LDS read per column block
// for all its tiles. Up to 5 column blocks a wave keeps all tiles on or above the diagonal and the waves share the
// tile's rows; from 6 on two waves share a set of rows and the tiles (the sums of 14 of 28 tiles take 112 registers).
// A last column block of at most 8 columns goes through v_mfma_f64_4x4x4 (4 columns x 16, 17 cycles instead of 70).
//
// Two-byte codes of column pairs (co-coded groups): a wave's 64 lanes look up one group at 64 rows (below 64 rows per tile two
// groups), a whole tuple of 16 bytes per lane, and write it to the lane's row of the tile. Dealt like the others the gathers
// of 8 bytes bound the kernel: 10,000,000 x 50, 4096 tuples (Zipf), 1001 us; so 934, with the gathers spread between the
// matrix instructions 692 (matrix pipe 496, gathers 400), with the codes of two tiles per load 654.
//
// The stages of three tiles overlap: while a tile is multiplied, the values of the next one but one are looked up and the
// codes behind those are on their way (pairs: a lane reads the codes of two rows at a time, one for each of two tiles). One barrier per tile that waits for LDS only: loads stay in flight over it.
//
// Bound: the fp64 matrix pipe (70 cycles per tile and 4 rows): busy 72 % of the time at 2,000,003 x 100 byte codes (vector issue 12 %,
// LDS 19 %, vector memory path 38 %), 73 % at 10,000,000 x 50 column pairs, where the gathers keep the vector memory path busy 55 % (64 with a code load per tile).
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include "cla_runs.hpp"
#include <algorithm>
#include <cstring>
#include <memory>

namespace cla {

constexpr int GT_THREADS = 512;
typedef double f64x4_gt __attribute__((ext_vector_type(4)));

// a decoded column
struct GtCol {
	int32_t dictOff;  // bytes from the dictionary base to its first value
	int32_t stride;   // bytes from one code's value to the next one's (0: a column that only carries a constant)
	int32_t group;    // code stream
	int32_t col;      // column of the block (-1: padding)
};

struct GtArgs {
	const uint8_t* arena;
	size_t arenaStride;
	const GtCol* cols;       // NCB * 16
	const double* dict;
	const double* img;       // column blocks [0, nLds): imgV x 16 values each
	int64_t nRows;
	int nTiles, nLds, imgV, nCols, nGroups;
	double* acc;             // where the blocks add (upper triangle)
	double* out;
	unsigned* done;          // nullptr: no tail (acc is the caller's output)
	unsigned long long* nnz;
	int skipOwn;             // cells inside a group and of columns without one come from the code counts (k_tsmm_self)
};

// How the codes are dealt: one-byte codes, two-byte codes, two-byte codes of column pairs (every group two columns)
constexpr int GT_BYTE = 1, GT_SHORT = 2, GT_PAIR = 3;
// 32 m rows per tile (m * ncb <= 8 where a wave decodes one part; pairs: whole waves of rows as far as LDS goes)
__host__ __device__ constexpr int gt_m(int ncb, int kind) { return ncb == 1 ? 8 : ncb == 2 ? (kind == GT_PAIR ? 4 : 3) : ncb <= 4 ? 2 : 1; }
// Tiles that a block takes together. Pairs: a lane's codes of two tiles are those of two neighbouring rows, one load of four bytes, requested
// two tiles before the first is looked up. A load per tile, one tile ahead, left HBM's latency in the open where tiles are short, and
// kept the vector memory path busy: 10,000,000 x 50 678 -> 654 us, 4,000,000 x 20 112 -> 101 (four rows and tiles: 654, 103).
__host__ __device__ constexpr int gt_group(int kind) { return kind == GT_PAIR ? 2 : 1; }
// doubles per row: rows 128 bytes apart in the banks; pairs, written by row with 16 bytes per lane: 144 bytes apart
__host__ __device__ constexpr int gt_stride(int ncb, int kind) { return kind == GT_PAIR ? ncb * 16 + (ncb & 1 ? 2 : 18) : ncb * 16 + (ncb & 1 ? 0 : 16); }

// NF full column blocks, then one of NN groups of 4 columns (NN = 0: none)
template <int NF, int NN, int KIND>
__global__ __launch_bounds__(GT_THREADS, 2) void k_gram_tiles(GtArgs A) {
	constexpr int NCB = NF + (NN ? 1 : 0), T = NF * (NF + 1) / 2;
	constexpr int W = KIND == GT_BYTE ? 1 : 2;
	constexpr int M = gt_m(NCB, KIND), R = 32 * M, S = gt_stride(NCB, KIND);
	constexpr bool SPLIT = NF > 5;              // two waves share the tiles of a set of rows
	constexpr int NK = SPLIT ? 2 * M : M;       // steps of 4 rows per wave and tile
	constexpr int BUF = R * S;
	// what a wave keeps of the T tiles and of the NCB products of a narrow group: SPLIT deals tiles [0, T0) and even
	// column blocks to waves 0 - 3, the others to waves 4 - 7
	constexpr int T0 = SPLIT ? T / 2 : T, TW = SPLIT ? T - T0 : T, NB = SPLIT ? (NCB + 1) / 2 : NCB;
	extern __shared__ __attribute__((aligned(16))) double smem[]; // two tile buffers, the dictionaries
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int c = lane & 15, k = lane >> 4;
	constexpr int G = gt_group(KIND);
	const int nShares = (A.nTiles + G - 1) / G;
	const int t0 = (int) ((int64_t) nShares * blockIdx.x / gridDim.x) * G, t1 = (int) ((int64_t) nShares * (blockIdx.x + 1) / gridDim.x) * G;

	// this wave's part of the decoding: column block, 32 rows of the tile
	const int myCb = wave % NCB, sub = wave / NCB;
	const int mode = wave >= NCB * M || t0 >= t1 ? 0 : myCb < A.nLds ? 1 : 2; // nothing, dictionary in LDS, in global memory
	const GtCol C = A.cols[myCb * 16 + c];
	const uint8_t* stream = A.arena + (size_t) C.group * A.arenaStride;
	const char* ldsDict = (const char*) (smem + 2 * BUF) + (size_t) myCb * A.imgV * 128 + c * 8;
	const char* gDict = (const char*) A.dict;
	const int64_t rowLast = (A.nRows - 1) & ~(int64_t) 7;
	double* const put = smem + (sub * 32 + 8 * k) * S + myCb * 16 + c;

	f64x4_gt acc[TW];
	double nacc[NN ? NN : 1][NB];
#pragma unroll
	for(int t = 0; t < TW; t++) acc[t] = f64x4_gt{0.0, 0.0, 0.0, 0.0};
#pragma unroll
	for(int i = 0; i < (NN ? NN : 1); i++)
#pragma unroll
		for(int b = 0; b < NB; b++) nacc[i][b] = 0.0;

	// pairs: a wave decodes units of 64 lanes, one tuple each: UR rows of 64 / UR neighbouring groups
	constexpr bool PAIR = KIND == GT_PAIR;
	constexpr int UR = R < 64 ? R : 64, UG = 64 / UR, RB = R / UR;  // rows and groups of a unit, units that share a group
	constexpr int NU = PAIR ? (NCB * 8 / UG * RB + 7) / 8 : 1;       // most units of a wave
	const int uRow = lane & (UR - 1);
	const int nUnits = ((A.nGroups + UG - 1) / UG * RB - wave + 7) / 8; // this wave's

	auto loop = [&](auto modeTag, auto halfTag) {
		constexpr int MODE = decltype(modeTag)::value, HALF = decltype(halfTag)::value;
		constexpr int U = PAIR ? NU - MODE : 0; // units of the wave (no branch around a load: it would wait for the load)
		auto unit_row = [&](int i) { return (wave + 8 * i) % RB * UR; };
		uint32_t pcode[U > 0 ? U : 1], pnext[U > 0 ? U : 1]; // codes of the two tiles looked up next, of the two behind them
		f64x2 pv[2][U > 0 ? U : 1];
		const uint8_t* pstream[U > 0 ? U : 1];
		const char* pdict[U > 0 ? U : 1];
		double* pput[U > 0 ? U : 1];
		if constexpr(PAIR) {
#pragma unroll
			for(int i = 0; i < U; i++) {
				const int g = min((wave + 8 * i) / RB * UG + (UG > 1 ? lane / UR : 0), A.nGroups - 1); // (an odd last group: twice)
				pstream[i] = A.arena + (size_t) g * A.arenaStride;
				pdict[i] = gDict + A.cols[2 * g].dictOff;
				pput[i] = smem + (unit_row(i) + uRow) * S + 2 * g;
			}
		}
		CodeVec<W, 8> codes[2];
		double v[2][8];
		auto load_codes = [&](int tile, auto parity) { // (codes and values of a tile sit in the sets of its parity)
			constexpr int Q = decltype(parity)::value;
			if(MODE == 0) return;
			const int64_t row = min((int64_t) min(tile, t1 - 1) * R + sub * 32 + 8 * k, rowLast);
			if constexpr(W == 1) codes[Q].raw.v = *(const u32x2*) (stream + row);
			else codes[Q].raw.v = *(const u32x4*) (stream + 2 * row);
		};
		auto load_pairs = [&](uint32_t (&dst)[U > 0 ? U : 1], int tile) { // of an even tile and the next one
#pragma unroll
			for(int i = 0; i < U; i++) {
				const int64_t row = min((int64_t) min(tile, t1 - 2) * R + 2 * (unit_row(i) + uRow), (A.nRows - 1) & ~(int64_t) 1);
				dst[i] = *(const uint32_t*) (pstream[i] + 2 * row);
			}
		};
		constexpr int NL = PAIR ? U : MODE == 0 ? 0 : 8; // lookups per lane and tile
		auto look_one = [&](int i, auto parity) {
			constexpr int Q = decltype(parity)::value;
			if constexpr(PAIR) pv[Q][i] = *(const f64x2*) (pdict[i] + (((pcode[i] >> (16 * Q)) & 0xffffu) << 4));
			else {
				const uint32_t code = (uint32_t) codes[Q].get(i);
				if(MODE == 1) v[Q][i] = *(const double*) (ldsDict + (code << 7));
				else v[Q][i] = *(const double*) (gDict + (uint32_t) (__umul24(code, (uint32_t) C.stride) + (uint32_t) C.dictOff));
			}
		};
		auto look = [&](auto parity) {
#pragma unroll
			for(int i = 0; i < NL; i++) look_one(i, parity);
		};
		auto write = [&](const double (&d)[8], int tile, int buf) {
			if constexpr(PAIR) { // (tile t goes from value set to buffer of the same parity)
#pragma unroll
				for(int i = 0; i < U; i++) {
					const bool in = (int64_t) (tile & ~1) * R + 2 * (unit_row(i) + uRow) + (tile & 1) < A.nRows; // zeros behind the last row of the matrix
					f64x2 x = buf == 0 ? pv[0][i] : pv[1][i];
					x.x = in ? x.x : 0.0; x.y = in ? x.y : 0.0;
					*(f64x2*) (pput[i] + buf * BUF) = x;
				}
				return;
			}
			if(MODE == 0) return;
			double* p = put + buf * BUF;
			if((int64_t) (tile + 1) * R <= A.nRows) {
#pragma unroll
				for(int t = 0; t < 8; t++) p[t * S] = d[t];
			}
			else { // zeros behind the last row of the matrix
				const int64_t row = (int64_t) tile * R + sub * 32 + 8 * k;
#pragma unroll
				for(int t = 0; t < 8; t++) p[t * S] = row + t < A.nRows ? d[t] : 0.0;
			}
		};
		// Multiplies the tile in a buffer. Two-byte codes: the lookups of the next tile but one are spread between the matrix
		// instructions, so that the two pipes work side by side (all in front of them, the gathers hold up every wave first:
		// 10,000,000 x 50 as pairs 934 instead of 692 us; byte codes, half of whose lookups go to LDS: 441 instead of 465 us).
		constexpr bool SPREAD = KIND != GT_BYTE;
		auto multiply = [&](int buf, auto parity) {
			constexpr int NM = NK * ((HALF == 0 ? T0 : T - T0) + NN * (SPLIT ? (NCB + 1 - HALF) / 2 : NCB)); // matrix instructions
			int at = 0, done = 0;
			auto between = [&]() {
				at++;
				if(SPREAD && done < NL && done * NM < at * NL) {
					__builtin_amdgcn_sched_barrier(0);
					look_one(done++, parity);
					__builtin_amdgcn_sched_barrier(0);
				}
			};
			const double* x0 = smem + buf * BUF + ((SPLIT ? wave & 3 : wave) * 4 + k) * S;
			double x[2][NCB], a[2][NN ? NN : 1];
			auto read = [&](int j) {
				const double* p = x0 + j * (SPLIT ? 16 : 32) * S;
#pragma unroll
				for(int b = 0; b < NCB; b++) x[j & 1][b] = p[16 * b + c];
#pragma unroll
				for(int i = 0; i < NN; i++) a[j & 1][i] = p[16 * NF + 4 * i + (lane & 3)];
			};
			read(0);
#pragma unroll
			for(int j = 0; j < NK; j++) {
				if(j + 1 < NK) read(j + 1);
				int t = 0;
#pragma unroll
				for(int p = 0; p < NF; p++)
#pragma unroll
					for(int q = p; q < NF; q++, t++)
						if((t < T0) == (HALF == 0)) {
							acc[t - HALF * T0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[j & 1][p], x[j & 1][q], acc[t - HALF * T0], 0, 0, 0);
							between();
						}
#pragma unroll
				for(int i = 0; i < NN; i++)
#pragma unroll
					for(int b = 0; b < NCB; b++)
						if(!SPLIT || (b & 1) == HALF) {
							nacc[i][SPLIT ? b / 2 : b] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[j & 1][i], x[j & 1][b], nacc[i][SPLIT ? b / 2 : b], 0, 0, 0);
							between();
						}
			}
#pragma unroll
			for(int i = 0; i < NL; i++)
				if(SPREAD && i >= done) look_one(i, parity); // (more lookups than matrix instructions)
		};
		using std::integral_constant;
		if constexpr(PAIR) { load_pairs(pcode, t0); load_pairs(pnext, t0 + 2); }
		else load_codes(t0, integral_constant<int, 0>());
		{
			// the dictionaries of the first column blocks, 8 pieces of 16 bytes per thread requested together
			const f64x2* src = (const f64x2*) A.img;
			f64x2* dst = (f64x2*) (smem + 2 * BUF);
			const int n = A.nLds * A.imgV * 8;
			for(int i0 = tid; i0 < n; i0 += 8 * GT_THREADS) {
				f64x2 d[8];
#pragma unroll
				for(int j = 0; j < 8; j++) d[j] = src[min(i0 + j * GT_THREADS, n - 1)];
#pragma unroll
				for(int j = 0; j < 8; j++)
					if(i0 + j * GT_THREADS < n) dst[i0 + j * GT_THREADS] = d[j];
			}
		}
		lds_barrier();
		if constexpr(!PAIR) load_codes(t0 + 1, integral_constant<int, 1>());
		look(integral_constant<int, 0>());
		if constexpr(!PAIR) load_codes(t0 + 2, integral_constant<int, 0>());
		look(integral_constant<int, 1>());
		write(v[0], t0, 0);
		lds_barrier();
		auto step = [&](int tile, auto parity) {
			constexpr int P = decltype(parity)::value;
			if constexpr(PAIR && P == 0) {
#pragma unroll
				for(int i = 0; i < U; i++) pcode[i] = pnext[i];
				load_pairs(pnext, tile + 4);
			}
			if(!SPREAD) look(parity);      // of tile + 2
			if constexpr(!PAIR) load_codes(tile + 3, integral_constant<int, P ^ 1>());
			multiply(P, parity);
			write(v[P ^ 1], min(tile + 1, t1 - 1), P ^ 1); // (behind the last tile: values nobody reads)
			lds_barrier();
		};
		for(int tile = t0; tile < t1; tile += 2) {
			step(tile, integral_constant<int, 0>());
			if(PAIR || tile + 1 < t1) step(tile + 1, integral_constant<int, 1>());
		}
	};
	if(t0 < t1) {
		using std::integral_constant;
		if constexpr(PAIR) {
			auto units = [&](auto halfTag) {
				if(nUnits >= NU) loop(integral_constant<int, 0>(), halfTag);
				else if(nUnits == NU - 1) loop(integral_constant<int, 1>(), halfTag);
				else loop(integral_constant<int, 2>(), halfTag);
			};
			if(SPLIT && wave >= 4) units(integral_constant<int, 1>());
			else units(integral_constant<int, 0>());
		}
		else if(SPLIT && wave >= 4) {
			if(mode == 0) loop(integral_constant<int, 0>(), integral_constant<int, 1>());
			else if(mode == 1) loop(integral_constant<int, 1>(), integral_constant<int, 1>());
			else loop(integral_constant<int, 2>(), integral_constant<int, 1>());
		}
		else {
			if(mode == 0) loop(integral_constant<int, 0>(), integral_constant<int, 0>());
			else if(mode == 1) loop(integral_constant<int, 1>(), integral_constant<int, 0>());
			else loop(integral_constant<int, 2>(), integral_constant<int, 0>());
		}
	}

	// the waves' sums of a tile, one set of rows after the other
	double* sum = smem;
	const int half = SPLIT ? wave >> 2 : 0, set = SPLIT ? wave & 3 : wave;
	for(int s = 0; s < (SPLIT ? 4 : 8); s++) {
		if(set == s) {
#pragma unroll
			for(int l = 0; l < TW; l++) {
				const int t = l + half * T0;
				if(half == 0 && l >= T0) continue;
#pragma unroll
				for(int i = 0; i < 4; i++) {
					double* p = &sum[t * 256 + i * 64 + lane];
					*p = s == 0 ? acc[l][i] : *p + acc[l][i];
				}
			}
#pragma unroll
			for(int i = 0; i < NN; i++)
#pragma unroll
				for(int l = 0; l < NB; l++) {
					const int b = SPLIT ? 2 * l + half : l;
					if(b >= NCB) continue;
					double* p = &sum[T * 256 + (i * NCB + b) * 64 + lane];
					*p = s == 0 ? nacc[i][l] : *p + nacc[i][l];
				}
		}
		__syncthreads();
	}
	double* const into = A.acc + (A.done != nullptr ? gram_way(A.nCols) : 0);
	auto add = [&](int ia, int ib, double d) {
		const GtCol Ca = A.cols[ia], Cb = A.cols[ib];
		if(A.skipOwn && (Ca.group == Cb.group || Ca.stride == 0 || Cb.stride == 0)) return;
		const int ca = Ca.col, cb = Cb.col;
		if(ca >= 0 && cb >= 0 && d != 0.0) unsafeAtomicAdd(&into[(size_t) min(ca, cb) * A.nCols + max(ca, cb)], d);
	};
	for(int i = tid; i < T * 256; i += GT_THREADS) {
		int t = i >> 8, p = 0;
		while(t >= NF - p) { t -= NF - p; p++; }
		const int q = p + t, r = ((i >> 6) & 3) * 4 + ((i & 63) >> 4), cc = i & 15;
		if(p != q || r <= cc) add(16 * p + r, 16 * q + cc, sum[i]);
	}
	for(int i = tid; i < NN * NCB * 64; i += GT_THREADS) {
		const int g = i / (NCB * 64), b = i / 64 % NCB, r = 4 * g + ((i & 63) >> 4), cc = i & 15;
		if(b < NF || r <= cc) add(16 * NF + r, 16 * b + cc, sum[T * 256 + i]);
	}
	if(A.done != nullptr) {
		__syncthreads();
		gram_tail(A.done, gridDim.x, A.acc, A.out, A.nCols, A.nnz, (unsigned*) smem);
	}
}

// ---- plan (kept with the block, dropped with the decode plans)

struct GtPlan {
	int rc = 0;       // 1: not of this kernel's shape
	GtArgs A;
	void* dImg = nullptr;
	int64_t bytes = 0;
	int nf = 0, nn = 0, kind = 0;
	size_t lds = 0;
	int perCU = 1;    // blocks per CU, one after the other where LDS holds one
	const int32_t* constCols = nullptr; // columns without a group whose constant is not zero
	int nConst = 0;
};

// Blocks per CU. A wave adds up its part of the block's rows in one chain, whose error grows with its length (like terms drift). Where
// k_tsmm_decode ran twice as many waves' sums side by side, two blocks share a CU's rows: diagonal cells of 4,000,000 rows of 7 values,
// rms relative error 20 columns 1.2e-14 -> 7.4e-15 (k_tsmm_decode 7.1e-15), 38 1.3e-14 -> 7.6e-15 (7.6e-15), 100 2.3e-14 -> 1.2e-14
// (1.0e-14); column pairs of 300 tuples, 20 columns 4.1e-15 -> 2.0e-15 (2.1e-15). A second block costs 8 - 23 us where it starts behind the first
// (2,000,003 rows of 256 values: 20 columns 73 -> 81 us, 100 columns 438 -> 461; 10,000,000 x 20 of 7 values, side by side: 280 -> 239).
static int gt_blocks_per_cu(int nf, int nn, int kind, int nTiles, int nCols) {
	// (below 1e-15 with one block; pairs below 13 columns ran in shorter chains before: diagonal cells of 1,000,003 x 10 4.0e-16, 1.0e-15 with one block, 3.8e-16 with two)
	if(nTiles < (nCols < 13 ? 2 : 16) * g_numCU) return 1;
	if(nf > 5) return 2;
	const int ncb = nf + (nn ? 1 : 0);
	return kind == GT_PAIR ? (nf == 1 && nn < 2) || ncb == 3 ? 2 : 1 : ncb <= 3 ? 2 : 1;
}

static int gt_build_plan(cla_block* b, GtPlan& P) {
	P.rc = 1;
	const int n = b->nCols;
	if(b->dArena == nullptr || b->arenaWidth > 2 || n < 4 || n > 128 || b->nRows == 0 || b->crossSplit > 0 || b->crossBlocks > 0) return 0;
	std::vector<int> groupOf((size_t) n, -1);
	for(size_t g = 0; g < b->groups.size(); g++)
		for(int col : b->groups[g].cols) {
			if(groupOf[col] >= 0) return 0; // overlapping groups
			groupOf[col] = (int) g;
		}
	// columns in the groups' order, then those that only carry a constant
	const int last = n - n / 16 * 16;
	P.nn = n < 16 ? 0 : last >= 1 && last <= 4 ? 1 : last >= 5 && last <= 8 ? 2 : 0;
	P.nf = n < 16 ? 1 : n / 16 + (last > 8 ? 1 : 0);
	bool pairs = b->arenaWidth == 2 && n == 2 * (int) b->groups.size();
	for(const HostGroup& H : b->groups) pairs &= H.d.nColG == 2;
	if(n < 13 && !pairs) return 0;
	// Column pairs whose dictionaries LDS cannot hold: a unit's lanes all look up one group, 16 bytes at a time. The lanes
	// share the lines of the frequent tuples, and each lookup gives two columns: 62.9 M tuples of 24 dictionaries of 4096
	// (Zipf) take 99 us of gathers like this, 170 us as 8 bytes per column with 8 groups per instruction.
	P.kind = b->arenaWidth == 1 ? GT_BYTE : pairs ? GT_PAIR : GT_SHORT;
	const int ncb = P.nf + (P.nn ? 1 : 0);
	bool consts = false; // the dictionaries are copied with the constants added
	for(int col = 0; col < n; col++) consts |= b->constV[col] != 0.0 || groupOf[col] < 0;
	std::vector<GtCol> cols;
	std::vector<double> dict;
	std::vector<const double*> src; // host values of a column (nullptr: only a constant)
	size_t total = 0;
	for(size_t g = 0; g < b->groups.size(); g++) {
		const HostGroup& H = b->groups[g];
		const int nc = H.d.nColG;
		for(int h = 0; h < nc; h++) {
			cols.push_back(GtCol{(int32_t) ((total + h) * 8), nc * 8, (int32_t) g, H.cols[h]});
			src.push_back(H.dict.data() + h);
		}
		if(consts)
			for(size_t i = 0; i < H.dict.size(); i++) dict.push_back(H.dict[i] + b->constV[H.cols[i % nc]]);
		total += H.dict.size();
	}
	for(int col = 0; col < n; col++)
		if(groupOf[col] < 0) {
			cols.push_back(GtCol{(int32_t) (total * 8), 0, 0, col});
			src.push_back(nullptr);
			dict.push_back(b->constV[col]);
			total++;
		}
	if(total * 8 >= ((size_t) 1 << 31) || (int) cols.size() != n) return 0;
	const int real = n;
	while((int) cols.size() < ncb * 16) { GtCol p = cols[real - 1]; p.col = -1; cols.push_back(p); src.push_back(src[real - 1]); }
	// column blocks whose dictionaries fit LDS beside the tiles
	const size_t tileBytes = (size_t) 2 * 32 * gt_m(ncb, P.kind) * gt_stride(ncb, P.kind) * 8;
	const size_t sumBytes = ((size_t) P.nf * (P.nf + 1) / 2 * 256 + (size_t) P.nn * ncb * 64) * 8;
	const size_t room = (size_t) g_ldsPerBlock - tileBytes;
	const int imgV = std::max(b->maxVals, 1);
	const int nLds = P.kind == GT_PAIR ? 0 : (int) std::min<size_t>(ncb, room / ((size_t) imgV * 128));
	P.lds = std::max(tileBytes + (size_t) nLds * imgV * 128, sumBytes);
	if(P.lds > (size_t) g_ldsPerBlock) return 0;
	std::vector<double> img((size_t) nLds * imgV * 16, 0.0);
	for(int s = 0; s < nLds * 16; s++) {
		const GtCol& C = cols[s];
		const double add = b->constV[cols[std::min(s, real - 1)].col];
		const int nV = src[s] ? b->groups[C.group].d.nVals : imgV;
		for(int kk = 0; kk < nV; kk++)
			img[((size_t) (s / 16) * imgV + kk) * 16 + s % 16] = (src[s] ? src[s][(size_t) kk * (C.stride / 8)] : 0.0) + add;
	}
	const size_t colBytes = cols.size() * sizeof(GtCol), imgBytes = img.size() * 8, dictBytes = consts ? dict.size() * 8 : 0;
	std::vector<int32_t> constCols;
	for(int col = 0; col < n; col++)
		if(groupOf[col] < 0 && b->constV[col] != 0.0) constCols.push_back(col);
	const size_t constBytes = constCols.size() * sizeof(int32_t);
	std::vector<uint8_t> all(colBytes + imgBytes + dictBytes + constBytes + 16, 0);
	std::memcpy(all.data(), cols.data(), colBytes);
	if(imgBytes) std::memcpy(all.data() + colBytes, img.data(), imgBytes);
	if(dictBytes) std::memcpy(all.data() + colBytes + imgBytes, dict.data(), dictBytes);
	if(constBytes) std::memcpy(all.data() + colBytes + imgBytes + dictBytes, constCols.data(), constBytes);
	uint8_t* d = nullptr;
	CLA_HIP(hipMalloc((void**) &d, all.size()));
	P.dImg = d;
	P.bytes = (int64_t) all.size();
	CLA_HIP(hipMemcpy(d, all.data(), all.size(), hipMemcpyHostToDevice));
	GtArgs& A = P.A;
	A.arena = b->dArena; A.arenaStride = b->arenaStride;
	A.cols = (const GtCol*) d;
	A.img = (const double*) (d + colBytes);
	A.dict = consts ? (const double*) (d + colBytes + imgBytes) : b->dAllDict;
	P.constCols = (const int32_t*) (d + colBytes + imgBytes + dictBytes);
	P.nConst = (int) constCols.size();
	A.nRows = b->nRows;
	A.nTiles = (int) ((b->nRows + 32 * gt_m(ncb, P.kind) - 1) / (32 * gt_m(ncb, P.kind)));
	P.perCU = gt_blocks_per_cu(P.nf, P.nn, P.kind, A.nTiles, n);
	A.nLds = nLds; A.imgV = imgV; A.nCols = n; A.nGroups = (int) b->groups.size();
	P.rc = 0;
	return 0;
}

void gt_plan_drop(cla_block* b) {
	if(b->gtPlan == nullptr) return;
	if(b->gtPlan->dImg) { (void) hipFree(b->gtPlan->dImg); b->derivedBytes -= b->gtPlan->bytes; }
	delete b->gtPlan;
	b->gtPlan = nullptr;
}

template <int NF, int NN>
static int gt_launch(cla_block* b, const GtPlan& P, const GtArgs& A, unsigned grid) {
	const auto kern = P.kind == GT_BYTE ? k_gram_tiles<NF, NN, GT_BYTE> : P.kind == GT_SHORT ? k_gram_tiles<NF, NN, GT_SHORT> : k_gram_tiles<NF, NN, GT_PAIR>;
	CLA_HIP(allow_full_lds((const void*) kern));
	hipLaunchKernelGGL(kern, dim3(grid), dim3(GT_THREADS), P.lds, b->stream, A);
	CLA_HIP(hipGetLastError());
	return 0;
}

static int gt_launch_shape(cla_block* b, const GtPlan& P, const GtArgs& A, unsigned grid) {
	Prof pf(b, "k_gram_tiles", grid, GT_THREADS, (long) P.lds, (double) b->device_bytes_cached);
#define GT_CASE(NF) \
	case NF: return P.nn == 0 ? gt_launch<NF, 0>(b, P, A, grid) : P.nn == 1 ? gt_launch<NF, 1>(b, P, A, grid) : gt_launch<NF, 2>(b, P, A, grid);
	switch(P.nf) {
		case 1: return P.nn == 0 ? gt_launch<1, 0>(b, P, A, grid) : P.nn == 1 ? gt_launch<1, 1>(b, P, A, grid) : gt_launch<1, 2>(b, P, A, grid);
		GT_CASE(2) GT_CASE(3) GT_CASE(4) GT_CASE(5) GT_CASE(6) GT_CASE(7)
		case 8: return gt_launch<8, 0>(b, P, A, grid);
	}
#undef GT_CASE
	return 1;
}

// Where k_tsmm_decode stays the better kernel: two-byte codes of blocks that are not all column pairs, up to 48 columns, whose dictionaries
// do not fit beside the tiles of one column block or exceed an XCD's L2 by far. 1: there; 2: there if it holds all dictionaries in LDS.
// Both in us: 16 columns of 890 values, which its smaller tiles leave room for, 150,003 rows 21.7 / 22.6 here, 250,007 24 / 27, 1,000,003
// 40 / 63, 4,000,003 106 / 203 (100,003: 20.4 / 13.6 at 700 values); dictionaries in global memory, up to its second turn of tiles, 16 of
// 20,000 values, 50,003 rows 18.9 / 19.3, 100,003 21.4 / 23.0, 200,003 27.7 / 30.9, 400,003 48 / 43; past the L2, 16 of 60,000 values
// 70,001 rows 32 / 38, 1,000,003 139 / 149, 20 of 60,000 206 / 216 (100,003: 41 / 41), 32 of 30,000 200,003 rows 70 / 76, 300,007
// 129 / 102, 1,000,003 269 / 293, 48 of 60,000 200,003 rows 161 / 171, 300,007 277 / 266, 1,000,003 683 / 732; 64 columns of 60,000 1148 / 1002. Pairs of 60,000 tuples stay within 4 %.
int gram_tiles_behind_decode(const cla_block* b) {
	const int n = b->nCols;
	if(b->dArena == nullptr || b->arenaWidth != 2 || n < 13 || n > 48) return 0;
	bool pairs = n == 2 * (int) b->groups.size();
	size_t bytes = 0;
	for(const HostGroup& H : b->groups) { pairs &= H.d.nColG == 2; bytes += H.dict.size() * 8; }
	if(pairs) return 0;
	const int64_t rows = b->nRows;
	if(bytes > ((size_t) 4 << 20) && rows > 150000 && rows <= 250000) return 1;
	if(bytes > ((size_t) 6 << 20)) return rows > (n <= 16 ? 60000 : n <= 32 && bytes > ((size_t) 9 << 20) ? 90000 : 500000);
	if(n > 16 || (size_t) b->maxVals * 128 + (size_t) 64 * gt_m(1, GT_SHORT) * gt_stride(1, GT_SHORT) * 8 <= (size_t) g_ldsPerBlock) return 0;
	if(bytes <= 120 * 1024) return rows > 150000 ? 2 : 0;
	return bytes <= ((size_t) 4 << 20) && rows > 60000 && rows <= 250000;
}

// Like launch_tsmm_decode: dNnz != nullptr: the call's only kernel, which writes dOut whole; else dOut (zeroed) gets the upper
// triangle. ownByCounts: cells inside a group are exact code counts times dictionary products, as on the way by pairs of groups (one
// more kernel in front). Returns 1 when the block is not of this kernel's shape.
int launch_gram_tiles(cla_block* b, double* dOut, unsigned long long* dNnz, bool ownByCounts) {
	if(b->gtPlan == nullptr) {
		std::unique_ptr<GtPlan> plan(new GtPlan()); // (the block's only when it is complete: half a plan would refuse the block for good)
		const int rc = gt_build_plan(b, *plan);
		if(rc < 0) {
			if(plan->dImg) (void) hipFree(plan->dImg);
			return rc;
		}
		if(plan->dImg) b->derivedBytes += plan->bytes;
		b->gtPlan = plan.release();
	}
	const GtPlan& P = *b->gtPlan;
	if(P.rc) return P.rc;
	GtArgs A = P.A;
	A.acc = dOut; A.out = dOut; A.done = nullptr; A.nnz = nullptr;
	if(dNnz != nullptr) {
		const int rc = ensure_gram_acc(b);
		if(rc) return rc;
		A.acc = b->dGramAcc; A.done = b->gram_ticket(); A.nnz = dNnz;
	}
	A.skipOwn = ownByCounts;
	const unsigned grid = (unsigned) std::min((A.nTiles + gt_group(P.kind) - 1) / gt_group(P.kind), g_numCU * P.perCU);
	auto fp64 = [&](double* out) { // the upper triangle into a zeroed matrix, as the call would have it
		GtArgs F = A;
		F.out = out; F.skipOwn = 0;
		if(F.done == nullptr) F.acc = out;
		return gt_launch_shape(b, P, F, grid);
	};
	int rc = P.kind == GT_BYTE ? gram_digits_plan(b, ownByCounts, fp64) : 1;
	if(rc < 0) return rc;
	const bool digits = rc == 0;
	// (where k_gram_tiles does not follow, an exception on the way included, nothing clears what the counts' kernel has added)
	struct Clear {
		cla_block* b;
		bool on;
		~Clear() { if(on) (void) hipMemsetAsync(b->dGramAcc, 0, (size_t) (1 + GRAM_WAYS) * b->nCols * b->nCols * sizeof(double), b->stream); }
	} clear{b, ownByCounts && dNnz != nullptr};
	// (into an accumulator that gram_tail reads: see gram_ways)
	double* const own = A.acc + (A.done != nullptr && !digits && grid > 4 * GRAM_WAYS ? (size_t) b->nCols * b->nCols : 0);
	if(ownByCounts && (rc = launch_tsmm_self(b, own, nullptr, b->hasConst ? b->dConstV : nullptr, P.constCols, P.nConst))) return rc;
	rc = digits ? launch_gram_digits(b, A.acc, A.out, A.nnz, A.skipOwn, dNnz != nullptr) : gt_launch_shape(b, P, A, grid);
	if(rc == 0) clear.on = false;
	return rc;
}

} // namespace cla
