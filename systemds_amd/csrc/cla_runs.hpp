// Run cursors: how a wave that walks consecutive rows follows the run-length columns of a block without
// looking any row up. A run-length column (one column of a ColGroupRLE, CG/ColGroupRLE.java:104-141) is
// constant over a run, and a run is long against the 64 rows a wave handles per step, so the wave keeps per
// column the current value and the row where its run ends and only acts where a run ends inside its step.
// Lane RC_LANE0 + a of the wave is the cursor of run-length column a; a window of the next RC_WIN runs of
// every column sits in LDS and is refilled (run ends, codes, dictionary values: three dependent loads) only
// when a cursor leaves it.
#pragma once
#include "cla_device.hpp"
#include <vector>

namespace cla {

constexpr int RC_MAX = 8;     // run-length columns a wave follows
constexpr int RC_WIN = 8;     // runs per column in the wave's window (RC_MAX * RC_WIN = 64 lanes refill it)
constexpr int RC_LANE0 = 16;  // first cursor lane
constexpr int32_t RC_NEVER = 0x7fffffff;

struct RunCol {
	const int32_t* runStart;  // nRuns + 1 run starts of the merged run table (last = nRows)
	const int32_t* runCode;   // tuple per run, -1 = rows that no run covers
	const double* dict;       // nVals x nC
	double add;               // added to every value of the column (its constant where the caller wants decoded cells)
	int32_t nRuns, nC, h;     // h: the column's place in a tuple
	int32_t col;              // column of the matrix
};

// Merged run table of a block's run-length columns (k_runs.hip).
struct Mrt {
	void* base = nullptr;
	int32_t* start = nullptr;     // nSeg + 1
	int32_t* codes = nullptr;     // nSeg x nR
	int32_t* sliceRec = nullptr;  // 8 per slice: segment of the first row, run starts inside the slice, the first six of them
	double* sums = nullptr;       // nSeg x 16: workspace of the product at hand
	int nSeg = 0, nR = 0, sliceRows = 0;
	int64_t nSlices = 0, bytes = 0;
};

// Same-wave LDS traffic is ordered by the hardware; this keeps the compiler from moving accesses across.
__device__ __forceinline__ void wave_lds_sync() {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct RunCursors {
	int32_t j;     // cursor lanes: run the column is in
	int32_t jw;    // cursor lanes: run in slot 0 of the column's window
	int32_t end;   // cursor lanes: first row behind the run; RC_NEVER on all other lanes and behind the last run
	double val;    // cursor lanes: the column's value on the run
	const RunCol* cols;
	int nR;
	int32_t* winEnd;   // RC_MAX * RC_WIN, wave-private LDS
	double* winVal;

	// Window slot (a, k) = run jw_a + k of column a, loaded by lane 8 a + k.
	__device__ __forceinline__ void refill(int lane) {
		const int a = lane >> 3, k = lane & 7;
		const int jb = __shfl(j, RC_LANE0 + a, WAVE);
		int32_t e = RC_NEVER;
		double v = 0.0;
		if(a < nR) {
			const RunCol* C = as_global(cols + a);
			const int jj = jb + k;
			if(jj < C->nRuns) {
				e = as_global(C->runStart)[jj + 1];
				const int code = as_global(C->runCode)[jj];
				v = C->add + (code < 0 ? 0.0 : as_global(C->dict)[(size_t) code * C->nC + C->h]);
			}
		}
		wave_lds_sync();
		winEnd[lane] = e;
		winVal[lane] = v;
		wave_lds_sync();
		jw = j;
	}

	__device__ __forceinline__ void read_window(int lane) {
		const int a = lane - RC_LANE0;
		if(a >= 0 && a < nR) {
			end = winEnd[a * RC_WIN + (j - jw)];
			val = winVal[a * RC_WIN + (j - jw)];
		}
	}

	// Cursors at row r0 (every column's run that holds r0).
	__device__ __forceinline__ void start(const RunCol* c, int n, int32_t* we, double* wv, int32_t r0, int lane) {
		cols = c; nR = n; winEnd = we; winVal = wv;
		j = 0; jw = 0; end = RC_NEVER; val = 0.0;
		if(nR > 0) {
			// lanes 8 a .. 8 a + 7 look for column a's run together, eight places at a time (one lane per column, halving, is
			// three times as many round trips to memory)
			const int a = lane >> 3, k = lane & 7;
			int lo = 0, hi = 0; // the last run that starts at or before r0 is in [lo, hi]
			const int32_t* starts = nullptr;
			if(a < nR) {
				const RunCol* C = as_global(cols + a);
				starts = as_global(C->runStart);
				hi = C->nRuns - 1;
			}
			while(__ballot(lo < hi) != 0) {
				const int n = hi - lo;                                              // runs behind lo
				const int at = lo + 1 + (int) ((int64_t) n * k / 8);                  // k = 0: lo + 1; at <= hi where n > 0
				const bool below = n > 0 && starts[min(at, hi)] <= r0;
				const int found = __builtin_popcount((unsigned) (__ballot(below) >> (8 * a)) & 0xffu); // places at or before r0: the first ones
				const int l2 = found == 0 ? lo : lo + 1 + (int) ((int64_t) n * (found - 1) / 8);
				const int h2 = found == 8 ? hi : lo + (int) ((int64_t) n * found / 8);
				if(n > 0) { lo = l2; hi = h2; }
			}
			j = __shfl(lo, 8 * (lane - RC_LANE0) & 63, WAVE);
			if(lane < RC_LANE0 || lane >= RC_LANE0 + nR) j = 0;
			refill(lane);
			read_window(lane);
		}
	}

	// First row at which some column's run ends (RC_NEVER: none does any more).
	__device__ __forceinline__ int32_t next_end() const {
		int32_t v = end;
		v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false)); // row_shr:1
		v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false)); // row_shr:2
		v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false)); // row_shr:4
		return __builtin_amdgcn_readlane(v, RC_LANE0 + RC_MAX - 1);
	}

	// Every column whose run ends at row e moves to its next run.
	__device__ __forceinline__ void advance(int32_t e, int lane) {
		const bool mine = end == e; // (never true outside the cursor lanes: e < RC_NEVER)
		if(mine) j++;
		if(__ballot(mine && j - jw >= RC_WIN) != 0) refill(lane);
		if(mine) read_window(lane);
	}

	// Value of column a (uniform).
	__device__ __forceinline__ double value(int a) const {
		int p[2];
		__builtin_memcpy(p, &val, 8);
		p[0] = __builtin_amdgcn_readlane(p[0], RC_LANE0 + a);
		p[1] = __builtin_amdgcn_readlane(p[1], RC_LANE0 + a);
		double r;
		__builtin_memcpy(&r, p, 8);
		return r;
	}
};

// Where a block of a one-kernel t(X) %*% X adds: its XCD's accumulator, where there are few blocks the one of all.
__device__ __forceinline__ bool gram_ways() { return gridDim.x > 4 * GRAM_WAYS; }
__device__ __forceinline__ size_t gram_way(int nCols) { return (size_t) (gram_ways() ? 1 + blockIdx.x % GRAM_WAYS : 0) * nCols * nCols; }

// Tail of a t(X) %*% X whose kernel is the only one of the call. The blocks have added their tiles' upper triangles
// into acc (1 + GRAM_WAYS of nCols x nCols, all zero when the kernel starts); every block comes here behind its last add. The last one
// of an XCD to arrive may add that XCD's accumulator to the first; the last of all copies the sum
// to out, mirrored, counts out's non-zeros into *nnz and leaves everything at zero for the next
// launch: what a fill of out in front of the kernel and a kernel of its own behind it would do. `lds`: 17 words of the
// block's LDS that nobody else uses any more (no static LDS here: k_gram_tiles fills LDS to the device's limit).
__device__ __forceinline__ void gram_tail(unsigned* done, unsigned nBlocks, double* acc, double* out, int nCols, unsigned long long* nnz,
	unsigned* lds) {
	int& lastS = (int&) lds[0];
	int* const gramPartS = (int*) lds + 1;
	// rows r and nCols - 1 - r of the upper triangle together are nCols + 1 cells
	const int w = nCols + 1, n = (nCols + 1) / 2 * w;
	const float perW = 1.0f / (float) w;
	auto cell_of = [&](int idx, int& i, int& j) {
		const int r = (int) (((float) idx + 0.5f) * perW), k = idx - r * w; // (exact: idx < 2^14, and idx + 0.5 is at least 1 / 2 w from a multiple of w)
		const bool first = k < nCols - r;
		i = first ? r : nCols - 1 - r;
		j = first ? r + k : i + k - (nCols - r);
		return idx < n && (first || i != r); // (the middle row is on its own)
	};
	// the cells of an accumulator, or of M added up, left at zero; NB cells per thread requested together: each is a round trip past the caches
	auto take = [&](double* from, auto waysTag, auto cellsTag, auto f) __attribute__((always_inline)) {
		constexpr int M = decltype(waysTag)::value, NB = decltype(cellsTag)::value;
		const size_t way = (size_t) nCols * nCols;
		for(int idx0 = threadIdx.x; idx0 < n; idx0 += NB * blockDim.x) {
			unsigned long long bits[NB][M];
			int i, j;
#pragma unroll
			for(int k = 0; k < NB; k++) {
				const size_t at = cell_of(idx0 + k * (int) blockDim.x, i, j) ? (size_t) i * nCols + j : 0;
#pragma unroll
				for(int m = 0; m < M; m++) bits[k][m] = __hip_atomic_load((const unsigned long long*) from + m * way + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
#pragma unroll
			for(int k = 0; k < NB; k++) {
				if(!cell_of(idx0 + k * (int) blockDim.x, i, j)) continue;
				double v = 0.0;
#pragma unroll
				for(int m = 0; m < M; m++) {
					__hip_atomic_store((unsigned long long*) from + m * way + (size_t) i * nCols + j, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					v += __longlong_as_double((long long) bits[k][m]);
				}
				f(i, j, v);
			}
		}
	};
	// true for the block that `ticket` names, once this block's adds have been acknowledged (the adds, the tickets and the reads are
	// all performed at device scope, past the caches that the chip's parts do not share)
	auto last = [&](auto ticket) __attribute__((always_inline)) {
		asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
		__syncthreads();
		if(threadIdx.x == 0) lastS = ticket();
		__syncthreads();
		return lastS != 0;
	};
	// a cell or two per thread: the last block reads all accumulators; more: the last block of each XCD adds its accumulator to the first
	// one before (20 columns 24 against 26 us, 100 columns of 10,000 rows 40 against 43)
	const bool ways = gram_ways(), few = n <= 2 * (int) blockDim.x, apart = ways && !few;
	if(!last([&]() { return apart ? last_of_way(done, nBlocks) : last_block(done, nBlocks); })) return;
	int cnt = 0;
	auto give = [&](int i, int j, double v) __attribute__((always_inline)) {
		out[(size_t) i * nCols + j] = v;
		out[(size_t) j * nCols + i] = v;
		cnt += v != 0.0 ? (i == j ? 1 : 2) : 0;
	};
	using std::integral_constant;
	if(apart) {
		take(acc + gram_way(nCols), integral_constant<int, 1>(), integral_constant<int, 8>(), [&](int i, int j, double v) {
			if(v != 0.0) unsafeAtomicAdd(&acc[(size_t) i * nCols + j], v); // (a NaN is unequal to zero)
		});
		if(!last([&]() { return last_of_ways(done, nBlocks); })) return;
	}
	if(!few) take(acc, integral_constant<int, 1>(), integral_constant<int, 8>(), give);
	else if(ways) take(acc + (size_t) nCols * nCols, integral_constant<int, GRAM_WAYS>(), integral_constant<int, 1>(), give);
	else take(acc, integral_constant<int, 1>(), integral_constant<int, 1>(), give); // (code that no block has run yet comes from memory, too)
	cnt = wave_sum_i32(cnt);
	if((threadIdx.x & (WAVE - 1)) == 0) gramPartS[threadIdx.x >> 6] = cnt;
	nnz_clear(nnz);
	__syncthreads();
	if(threadIdx.x == 0) {
		int s = 0;
		for(unsigned w = 0; w < (blockDim.x + WAVE - 1) / WAVE; w++) s += gramPartS[w];
		*nnz = (unsigned long long) s;
	}
	clear_tickets(done);
}

int mrt_build(cla_block* b, const std::vector<RunCol>& runs, int sliceRows, Mrt& T);
void mrt_free(Mrt& T);
int launch_run_sums(cla_block* b, const std::vector<RunCol>& runs, const Mrt& T, const double* dB, int ld, int q, const double* dConstRow);

} // namespace cla
