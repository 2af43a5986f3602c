// Left multiply Y %*% X by several rows of Y on blocks whose groups are all single-column DDC with byte codes: one pass
// over the codes for up to 16 rows of Y, on the fp64 matrix cores.
//
// A wave takes 64 rows of X and up to 4 column blocks of 16 groups. Lane (k, c), k = lane / 16, c = lane % 16, reads 16
// codes of group c of a column block (rows 16 k .. 16 k + 15 of the 64) with one 16-byte load and looks them up in the
// column block's dictionaries in LDS, one row of each quarter per step: the looked-up values are the B operand (4 rows x 16
// columns) of the matrix instruction as they come, and the A operand is Y at the same rows. The sums stay in registers over
// all rows of the block: one LDS add per wave and cell at the end, where k_lmm_u8_vec adds once per thread and group.
// A unit's 64 rows are a chain of additions of their own (one chain over a wave's share drifts where the terms are alike: a row
// of like values times columns of 7 values, 4,000,000 rows, 1.7e-14 relative error instead of 5e-16; 0.8 % of the time).
// Up to 12 rows of Y go through v_mfma_f64_4x4x4 (four 4 x 4 x 4 products, 4 rows of Y each: 17 - 19 cycles per 4 rows of Y),
// more through v_mfma_f64_16x16x4 (70 cycles for 16).
//
// LDS holds a column block as [code][16 groups]: the 16 lanes of a quarter read 16 different banks whatever their codes.
//
// Y goes through LDS: as the matrix operand wants it, neighbouring lanes hold different rows of Y, and the vector memory
// path serves such a load one lane a cycle (it was busy 70 - 80 % of the kernel and 2,000,003 x 100 by 8 rows took 118 us).
//
// Bound: matrix and vector issue (they do not overlap on a SIMD; 55 and 35 % of the time by 8 rows of Y, LDS 40 %): per 64 rows and column block 16 lookups of two vector
// instructions and 16 x ceil(p / 4) matrix instructions of 17 cycles; under that HBM (codes once, Y once per slab of 4
// column blocks). Measured (before: a pass of k_lmm_u8_vec per row of Y): 2,000,003 x 100 by 8 rows of Y 346 -> 105 us
// (3.1 TB/s), 8,000,001 x 100 by 16 2199 -> 742 us, 70,014 x 54 by 4 92 -> 15.5 us.
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include <algorithm>

namespace cla {

constexpr int LM_THREADS = 512;
constexpr int LM_NCB = 4; // column blocks per slab (LDS: 32 KiB each at 256 values)
constexpr int LM_YS = 34; // doubles per row of Y in LDS: 32 and 2 more, so that rows lie 16 bytes apart in the banks

typedef double f64x4_lm __attribute__((ext_vector_type(4)));
typedef double f64x2_a8 __attribute__((ext_vector_type(2), aligned(8))); // (a row of Y starts at any multiple of 8 bytes)

// The rows of a block: NCB column blocks from cb0 on, units [u0, u1) of 64 rows, and where `tail` is set the last rows of the
// matrix behind the whole units. Leaves the sums in LDS: [column block][rows 4 i + k of Y][16 columns].
template <int NI, int NCB>
__device__ __forceinline__ void lmm_mfma_rows(double* smem, double* yLds, const uint8_t* __restrict__ arena, size_t arenaStride, int nGroups,
	const double* __restrict__ dictT, int nVals, const double* __restrict__ Y, int pHere, int64_t nRows, int cb0, int64_t u0, int64_t u1,
	bool tail) {
	constexpr int NY = NI == 4 ? 1 : NI; // values of Y per lane and step
	constexpr int NW = LM_THREADS / WAVE;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int c = lane & 15, k = lane >> 4;
	const uint8_t* codeBase[NCB]; // this lane's stream of every column block
#pragma unroll
	for(int cb = 0; cb < NCB; cb++) codeBase[cb] = arena + (size_t) min((cb0 + cb) * 16 + c, nGroups - 1) * arenaStride + 16 * k;
	// Y of half a unit (rows 8 h .. 8 h + 7 of each quarter): lane (i4, quarter, piece) requests 16 bytes of row 4 i + i4 of Y,
	// four lanes a 64-byte run, a unit ahead; through LDS of the wave's own into the operand's order
	double* const yw = yLds + wave * (NI * 4 * LM_YS);
	const double* yBase[NI];
#pragma unroll
	for(int i = 0; i < NI; i++) yBase[i] = Y + (size_t) min(4 * i + k, pHere - 1) * nRows + 16 * (c >> 2) + 2 * (c & 3);
	double* const ywPut = yw + k * LM_YS + 8 * (c >> 2) + 2 * (c & 3);
	const double* const ywGet = yw + (NI == 4 ? c : lane & 3) * LM_YS + 8 * k;

	u32x4 codes[2][NCB];
	f64x2_a8 raw[2][NI];
	auto load_codes = [&](u32x4 (&dst)[NCB], int64_t u) {
#pragma unroll
		for(int cb = 0; cb < NCB; cb++) dst[cb] = *(const u32x4*) (codeBase[cb] + u * WAVE);
	};
	auto load_y = [&](int64_t u, int h) {
#pragma unroll
		for(int i = 0; i < NI; i++) raw[h][i] = *(const f64x2_a8*) (yBase[i] + u * WAVE + 8 * h);
	};
	// the same for the rows behind the whole units: zeros behind the last row of the matrix
	auto load_y_tail = [&](int64_t u, int h) {
		const int64_t r = u * WAVE + 8 * h, row = r + 16 * (c >> 2) + 2 * (c & 3);
#pragma unroll
		for(int i = 0; i < NI; i++) {
			double v0 = 0.0, v1 = 0.0;
			if(row < nRows) v0 = yBase[i][r];
			if(row + 1 < nRows) v1 = yBase[i][r + 1];
			raw[h][i].x = v0;
			raw[h][i].y = v1;
		}
	};
	auto put_y = [&](int h) {
#pragma unroll
		for(int i = 0; i < NI; i++) {
			f64x2 d;
			d.x = raw[h][i].x; d.y = raw[h][i].y;
			*(f64x2*) (ywPut + 4 * i * LM_YS) = d;
		}
		// (the wave's accesses to its LDS are performed in order; the compiler must keep them so)
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	};

	double acc[NCB][NI], tot[NCB][NI]; // of a unit's rows, of the units in front of it; [.][0 .. 3]: the four values of the 16 x 16 form
#pragma unroll
	for(int cb = 0; cb < NCB; cb++)
#pragma unroll
		for(int i = 0; i < NI; i++) acc[cb][i] = tot[cb][i] = 0.0;
	auto next_unit = [&]() {
#pragma unroll
		for(int cb = 0; cb < NCB; cb++)
#pragma unroll
			for(int i = 0; i < NI; i++) {
				tot[cb][i] += acc[cb][i];
				acc[cb][i] = 0.0;
			}
	};

	const char* tb = (const char*) smem + c * 8;
	const int cbBytes = nVals * 128;
	// the lookups of a column block are requested before the matrix instructions of the one in front of it
	auto work = [&](const u32x4 (&cv)[NCB], auto half) {
		constexpr int h = decltype(half)::value;
		f64x2 yv[NY][4];
#pragma unroll
		for(int i = 0; i < NY; i++)
#pragma unroll
			for(int t = 0; t < 4; t++) yv[i][t] = *(const f64x2*) (ywGet + 4 * i * LM_YS + 2 * t);
		double v[2][8];
		auto look = [&](int cb) {
			const char* t0 = tb + cb * cbBytes;
			const uint32_t w[2] = {h ? cv[cb].z : cv[cb].x, h ? cv[cb].w : cv[cb].y};
#pragma unroll
			for(int t = 0; t < 8; t++) v[cb & 1][t] = *(const double*) (t0 + (((w[t >> 2] >> (8 * (t & 3))) & 0xffu) << 7));
		};
		look(0);
#pragma unroll
		for(int cb = 0; cb < NCB; cb++) {
			if(cb + 1 < NCB) look(cb + 1);
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for(int t = 0; t < 8; t++) {
				if constexpr(NI == 4) {
					f64x4_lm a = {acc[cb][0], acc[cb][1], acc[cb][2], acc[cb][3]};
					a = __builtin_amdgcn_mfma_f64_16x16x4f64(yv[0][t >> 1][t & 1], v[cb & 1][t], a, 0, 0, 0);
					acc[cb][0] = a[0]; acc[cb][1] = a[1]; acc[cb][2] = a[2]; acc[cb][3] = a[3];
				}
				else {
#pragma unroll
					for(int i = 0; i < NI; i++)
						acc[cb][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(yv[i][t >> 1][t & 1], v[cb & 1][t], acc[cb][i], 0, 0, 0);
				}
			}
			__builtin_amdgcn_sched_barrier(0);
		}
	};

	int64_t u = u0 + wave;
	if(u < u1) { load_codes(codes[0], u); load_y(u, 0); load_y(u, 1); }
	{
		// the slab's dictionaries, 8 pieces of 16 bytes per thread requested together
		const f64x2* src = (const f64x2*) (dictT + (size_t) cb0 * nVals * 16);
		const int n = NCB * nVals * 8;
		for(int i0 = tid; i0 < n; i0 += 8 * LM_THREADS) {
			f64x2 d[8];
#pragma unroll
			for(int j = 0; j < 8; j++) d[j] = src[min(i0 + j * LM_THREADS, n - 1)];
#pragma unroll
			for(int j = 0; j < 8; j++)
				if(i0 + j * LM_THREADS < n) ((f64x2*) smem)[i0 + j * LM_THREADS] = d[j];
		}
	}
	__syncthreads();
	using std::integral_constant;
	for(; u < u1; u += NW) {
		const int64_t un = u + NW < u1 ? u + NW : u; // (the last turn requests its own rows again)
		put_y(0);
		load_codes(codes[1], un);
		load_y(un, 0);
		work(codes[0], integral_constant<int, 0>());
		put_y(1);
		load_y(un, 1);
		work(codes[0], integral_constant<int, 1>());
#pragma unroll
		for(int cb = 0; cb < NCB; cb++) codes[0][cb] = codes[1][cb];
		next_unit();
	}
	// (outside the loop: a load under a condition makes the compiler wait for all loads in flight)
	if(tail && wave == NW - 1) {
		const int64_t ut = nRows / WAVE;
		load_codes(codes[0], ut);
		load_y_tail(ut, 0);
		load_y_tail(ut, 1);
		put_y(0);
		work(codes[0], integral_constant<int, 0>());
		put_y(1);
		work(codes[0], integral_constant<int, 1>());
		next_unit();
	}

	__syncthreads();
	for(int i = tid; i < NCB * NI * 64; i += LM_THREADS) smem[i] = 0.0;
	__syncthreads();
#pragma unroll
	for(int cb = 0; cb < NCB; cb++)
#pragma unroll
		for(int i = 0; i < NI; i++) unsafeAtomicAdd(&smem[(cb * NI + i) * 64 + lane], tot[cb][i]);
	__syncthreads();
}

template <int NI>
__global__ __launch_bounds__(LM_THREADS, 2) void k_lmm_u8_dot(const uint8_t* __restrict__ arena, size_t arenaStride, int nGroups,
	const double* __restrict__ dictT, int nVals, const int32_t* __restrict__ col0, const double* __restrict__ Y, int p, int64_t nRows,
	int nSlabs, double* __restrict__ out, int nCols, unsigned* __restrict__ done, unsigned long long* __restrict__ nnz) {
	// (16-byte accesses to LDS want their alignment: 64 instead of 8 cycles each behind the 72 bytes of the tail)
	extern __shared__ __attribute__((aligned(16))) double smem[]; // column blocks of the slab, nVals x 16 each; the sums at the end
	const int p0 = blockIdx.y * 16;      // rows of Y of this pass: p0 .. p0 + 15
	const int pHere = min(16, p - p0);
	// The slabs of a share of the rows are blocks of one XCD (blocks go to the XCDs in turn) that start together: Y comes
	// from HBM once, the other slabs find it in the XCD's L2.
	const int nCb = (nGroups + 15) / 16;
	const int slab = blockIdx.x / 8 % nSlabs, share = blockIdx.x / 8 / nSlabs * 8 + blockIdx.x % 8, nShares = gridDim.x / nSlabs;
	const int cb0 = nCb * slab / nSlabs, myCb = nCb * (slab + 1) / nSlabs - cb0;
	const int64_t nUnits = nRows / WAVE; // whole ones
	const int64_t u0 = nUnits * share / nShares, u1 = nUnits * (share + 1) / nShares;
	const bool tail = share == nShares - 1 && nUnits * WAVE < nRows;
	const double* y = Y + (size_t) p0 * nRows;
	double* yLds = smem + (size_t) ((nCb + nSlabs - 1) / nSlabs) * nVals * 16;
	if(myCb == 4) lmm_mfma_rows<NI, 4>(smem, yLds, arena, arenaStride, nGroups, dictT, nVals, y, pHere, nRows, cb0, u0, u1, tail);
	else if(myCb == 3) lmm_mfma_rows<NI, 3>(smem, yLds, arena, arenaStride, nGroups, dictT, nVals, y, pHere, nRows, cb0, u0, u1, tail);
	else if(myCb == 2) lmm_mfma_rows<NI, 2>(smem, yLds, arena, arenaStride, nGroups, dictT, nVals, y, pHere, nRows, cb0, u0, u1, tail);
	else lmm_mfma_rows<NI, 1>(smem, yLds, arena, arenaStride, nGroups, dictT, nVals, y, pHere, nRows, cb0, u0, u1, tail);

	// lane (k, c) held rows 4 i + k of Y, column c of every column block
	for(int i = threadIdx.x; i < myCb * NI * 64; i += LM_THREADS) {
		const int cb = i / (NI * 64), row = (i / 64 % NI) * 4 + ((i & 63) >> 4), g = (cb0 + cb) * 16 + (i & 15);
		if(row < pHere && g < nGroups && smem[i] != 0.0) unsafeAtomicAdd(&out[(size_t) (p0 + row) * nCols + col0[g]], smem[i]);
	}
	lmm_tail(done, gridDim.x * gridDim.y, out, p * nCols, nnz);
}

// Returns 1 when the block is not eligible, 0 when the groups' contributions have been added to dOut.
int launch_lmm_u8_dot(cla_block* b, const double* dY, int p, double* dOut) {
	const int nG = (int) b->groups.size();
	if(b->dDictPad == nullptr || b->dictNonFinite || (b->opt.lmmDisable & 1)) return 1; // (non-finite dictionary values: the reference sums Y per tuple first, see launch_lmm_joint)
	const int nCb = (nG + 15) / 16, nPass = (p + 15) / 16;
	const int nV = b->maxVals;
	const int ni = p > 12 ? 4 : (p + 3) / 4; // (also the last rows of a larger p: the passes share one launch)
	const size_t yBytes = (size_t) (LM_THREADS / WAVE) * ni * 4 * LM_YS * 8, cbBytes = (size_t) nV * 128;
	const size_t room = (size_t) g_ldsPerBlock - 256; // (the tail's static LDS)
	const int most = (int) std::min<size_t>(LM_NCB, (room - yBytes) / cbBytes);
	const int nSlabs = (nCb + most - 1) / most;
	const size_t lds = std::max((nCb + nSlabs - 1) / nSlabs * cbBytes + yBytes, (size_t) LM_NCB * 4 * 64 * 8);
	const int64_t nUnits = (b->nRows + WAVE - 1) / WAVE;
	// a block per CU, fewer where a wave would not get a unit of 64 rows; whole turns of 8 shares (one per XCD)
	const int64_t perXcd = std::max<int64_t>(1, std::min<int64_t>(g_numCU / 8 / nSlabs, (nUnits + 63) / 64));
	const unsigned grid = (unsigned) (perXcd * 8 * nSlabs);
	const int32_t* dCol0 = (const int32_t*) (b->dDictPad + (size_t) nG * 256);
	const double algo = (double) nPass * b->nRows * nG + (double) p * b->nRows * 8;
	Prof pf(b, "k_lmm_u8_dot", (long) grid * nPass, LM_THREADS, (long) lds, algo);
	const bool tail = b->lmmTailWanted; // (this kernel serves every group of the block)
#define LM_LAUNCH(NI)                                                                                                             \
	do {                                                                                                                          \
		CLA_HIP(allow_full_lds((const void*) k_lmm_u8_dot<NI>));                                                                  \
		hipLaunchKernelGGL(k_lmm_u8_dot<NI>, dim3(grid, nPass), dim3(LM_THREADS), lds, b->stream, b->dArena, b->arenaStride, nG,   \
			b->dDictPad + b->dictTOff, nV, dCol0, dY, p, b->nRows, nSlabs, dOut, b->nCols, tail ? b->lmm_ticket() : nullptr, b->dCounters); \
	} while(0)
	if(ni == 4) LM_LAUNCH(4);
	else if(ni == 3) LM_LAUNCH(3);
	else if(ni == 2) LM_LAUNCH(2);
	else LM_LAUNCH(1);
#undef LM_LAUNCH
	b->lmmTailDone = tail;
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
