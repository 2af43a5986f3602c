// X %*% v on byte-code blocks (single-column groups) of few rows: all tables in LDS at once, few rows per thread.
//
// k_rmm_q1_u8 gives a thread 16 rows, which a block of 8 waves needs 8192 rows to fill: 100,000 rows kept 49 of 256 CUs busy, two
// waves each, and every block staged its tables slab by slab behind barriers. Here a thread takes RPT = 1, 2 or 4 rows, so that
// the rows spread over all CUs, requests the codes of 16 groups at a time two batches ahead, and a block makes all its tables once
// (dict[code] * v[col], as in k_rmm_q1_u8), their stride the block's largest dictionary. Groups are visited in list order and a
// product rounds before it is added: bit for bit the same sums.
//
// Bound: the launch and three round trips to memory (columns, v, dictionaries), then the copy of the tables: 1,000 rows of 5 columns
// take 6.3 us, of 54 columns of 200 values 10.5; on 100,000 x 20 vector issue is busy 30 % of the CUs' busy cycles, the vector memory address unit 34. Measured (k_rmm_q1_u8 before): 100,000 x 20 9.6 -> 7.1 us, 250,007 x 54 18.7 -> 12.5,
// 100,000 x 100 27.6 -> 14.5, 600,000 x 100 34.5 -> 25.
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include <algorithm>

namespace cla {

constexpr int UF_NB = 16;   // groups per batch of codes
constexpr int uf_tpt(int threads) { return threads == 1024 ? 20 : 38; } // table entries per thread at most

// RPT consecutive codes of a group
template <int RPT>
struct UfCodes { typedef uint8_t type; };
template <>
struct UfCodes<2> { typedef uint16_t type; };
template <>
struct UfCodes<4> { typedef uint32_t type; };

template <int THREADS, int RPT>
__global__ __launch_bounds__(THREADS) void k_rmm_q1_u8_few(const uint8_t* __restrict__ arena, size_t arenaStride, int nGroups,
	const double* __restrict__ dictPad, int stride, uint32_t magic, const double* __restrict__ constTerm, double* __restrict__ out, int64_t nRows,
	unsigned long long* __restrict__ nnz, const int32_t* __restrict__ col0, const double* __restrict__ v, unsigned long long* __restrict__ nnzNext,
	const RowOp op) {
	extern __shared__ __attribute__((aligned(16))) double tbl[]; // nGroups tables of `stride` entries, a table of zeros, v by group
	typedef typename UfCodes<RPT>::type Codes;
	constexpr int TPT = uf_tpt(THREADS), NS = RPT == 4 ? UF_NB / 2 : UF_NB; // groups whose lookups are in flight together
	const int tid = threadIdx.x;
	const int64_t row0 = ((int64_t) blockIdx.x * THREADS + tid) * RPT;
	const bool any = row0 < nRows;
	const int nTbl = nGroups * stride; // entries
	double* const vS = tbl + nTbl + stride;
	// (a stream's stride is a multiple of 256 bytes, and what lies behind its last row is code 0)
	const uint8_t* const mine = arena + (any ? row0 : 0);
	uint32_t ping[UF_NB], pong[UF_NB];
	auto request = [&](uint32_t (&c)[UF_NB], int g0) {
#pragma unroll
		for(int j = 0; j < UF_NB; j++) c[j] = *(const Codes*) (mine + (size_t) min(g0 + j, nGroups - 1) * arenaStride);
	};
	request(ping, 0);
	// entry f of the tables: group f / stride (by its reciprocal), code f % stride
	auto group_of = [&](int f) { return (int) __umulhi((uint32_t) f, magic); };
	double stage[TPT];
	auto fetch = [&](int k0) {
#pragma unroll
		for(int k = 0; k < TPT / 2; k++) {
			const int f = min(tid + (k0 + k) * THREADS, nTbl - 1), g = group_of(f);
			stage[k0 + k] = dictPad[(size_t) g * 256 + (f - g * stride)];
		}
	};
	const bool second = TPT / 2 * THREADS < nTbl; // (uniform)
	fetch(0);
	if(second) fetch(TPT / 2);
	int bad = 0;
	for(int g = tid; g < nGroups; g += THREADS) {
		const double x = v[col0[g]];
		vS[g] = x;
		bad |= !isfinite(x);
	}
	for(int i = tid; i < stride; i += THREADS) tbl[nTbl + i] = 0.0;
	if(blockIdx.x == 0) nnz_clear(nnzNext);
	// a zero dictionary cell stays zero whatever v holds (Dictionary.preaggValuesFromDense)
	const bool careful = __syncthreads_or(bad) != 0;
	auto put = [&](int k0) {
#pragma unroll
		for(int k = k0; k < k0 + TPT / 2; k++) {
			const int f = tid + k * THREADS;
			if(f < nTbl) {
				const double vv = vS[group_of(f)];
				tbl[f] = careful && stage[k] == 0.0 ? 0.0 : stage[k] * vv;
			}
		}
	};
	put(0);
	if(second) put(TPT / 2);
	request(pong, UF_NB);
	__syncthreads();

	double acc[RPT];
#pragma unroll
	for(int i = 0; i < RPT; i++) acc[i] = 0.0;
	const int strideB = stride * 8;
	auto consume = [&](const uint32_t (&c)[UF_NB], int g0) {
#pragma unroll
		for(int h = 0; h < UF_NB; h += NS) {
			double t[NS][RPT];
#pragma unroll
			for(int j = 0; j < NS; j++) {
				const char* tb = (const char*) tbl + min(g0 + h + j, nGroups) * strideB; // (behind the last group: zeros)
#pragma unroll
				for(int i = 0; i < RPT; i++) t[j][i] = *(const double*) (tb + (((c[h + j] >> (8 * i)) & 0xffu) << 3));
			}
#pragma unroll
			for(int j = 0; j < NS; j++)
#pragma unroll
				for(int i = 0; i < RPT; i++) acc[i] += t[j][i];
		}
	};
	for(int g0 = 0; g0 < nGroups; g0 += 2 * UF_NB) {
		consume(ping, g0);
		request(ping, g0 + 2 * UF_NB);
		if(g0 + UF_NB < nGroups) consume(pong, g0 + UF_NB);
		request(pong, g0 + 3 * UF_NB);
	}

	const double cadd = constTerm != nullptr ? *constTerm : 0.0;
	int cnt = 0;
	if(any) {
		double r[RPT];
#pragma unroll
		for(int i = 0; i < RPT; i++) {
			r[i] = acc[i] + cadd;
			if(op.w != nullptr) r[i] = row_op(r[i], op.w[min(row0 + i, nRows - 1)], op.minus);
			cnt += row0 + i < nRows && r[i] != 0.0;
		}
		if(RPT > 1 && row0 + RPT <= nRows && ((size_t) out & 15) == 0) {
#pragma unroll
			for(int i = 0; i < RPT; i += 2) {
				f64x2 d;
				d.x = r[i]; d.y = r[RPT > 1 ? i + 1 : 0];
				*(f64x2*) (out + row0 + i) = d;
			}
		}
		else {
#pragma unroll
			for(int i = 0; i < RPT; i++)
				if(row0 + i < nRows) out[row0 + i] = r[i];
		}
	}
	count_add(nnz, cnt);
}

// Returns 1 when the block has too many rows or tables for it, 0 when the product has been queued.
int launch_rmm_q1_u8_few(cla_block* b, const double* dB, const double* constTerm, double* dOut, unsigned long long* dNnz, unsigned long long* nnzNext,
	const RowOp& op) {
	const int nG = (int) b->groups.size();
	const int64_t nRows = b->nRows;
	const int stride = std::max((b->maxVals + 1) & ~1, 2);
	const size_t lds = ((size_t) (nG + 1) * stride + nG) * 8;
	const int threads = nRows <= (int64_t) g_numCU * 2048 ? 512 : 1024;
	const int rpt = threads == 1024 ? 4 : nRows <= (int64_t) g_numCU * 512 ? 1 : nRows <= (int64_t) g_numCU * 1024 ? 2 : 4;
	const auto kern = threads == 1024 ? k_rmm_q1_u8_few<1024, 4> : rpt == 1 ? k_rmm_q1_u8_few<512, 1> : rpt == 2 ? k_rmm_q1_u8_few<512, 2> : k_rmm_q1_u8_few<512, 4>;
	// (1,000,003 rows, in us here and on k_rmm_q1_u8: 5 columns 10.4 / 10.3, 20 12.1 / 13.0, 54 21 / 24, 100 28 / 35; 1,500,000, two turns of blocks, 54
	// columns 37 / 27. Blocks of 512 threads, two per CU: 600,000 x 20 11.6 against 11.0, 600,000 x 30 13.6 against 12.3)
	if(nRows > (int64_t) g_numCU * (nG <= 8 ? 3072 : 4096) || (size_t) nG * stride > (size_t) uf_tpt(threads) * threads || lds > (size_t) g_ldsPerBlock) return 1;
	size_t room = 0;
	CLA_HIP(max_dynamic_lds((const void*) kern, room));
	if(lds > room) return 1;
	const unsigned grid = (unsigned) ((nRows + (int64_t) threads * rpt - 1) / ((int64_t) threads * rpt));
	const uint32_t magic = (uint32_t) ((((uint64_t) 1 << 32) + stride - 1) / stride); // (f / stride = f * magic >> 32 for f < 2^32 / stride)
	const int32_t* dCol0 = (const int32_t*) (b->dDictPad + (size_t) nG * 256);
	Prof pf(b, "k_rmm_q1_u8_few", grid, threads, (long) lds, (double) nRows * nG + (double) nRows * 8 + (double) b->totalVals * 8);
	hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, b->stream, b->dArena, b->arenaStride, nG, b->dDictPad, stride, magic, constTerm, dOut, nRows,
		dNnz, dCol0, dB, nnzNext, op);
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
