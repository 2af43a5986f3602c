// Right multiply X %*% B on byte-code blocks of 64 - 100 columns: rows decoded into 8-bit digits, products on the integer matrix cores.
//
// Every column of X (its dictionary) and every column of B is scaled by a power of two to |x| < 1 and rounded to a whole number of seven signed
// base-256 digits, x = sum of d_i 2^(-7 - 8 i), i = 0 .. 6; row k of B takes the scale of column k of X with it. An output is the sum over the weights w = i + j <= 6
// of exact 32-bit sums of digit products (28 of the 49), joined in fp64. What is lost are the products of weight 7 (6 a column, of either sign) and the rounding of
// the values: rms 1.1e-16 sqrt(K / 100) of the largest possible term. Against 80-bit products, relative to the sum of the terms' magnitudes and normally distributed
// (rms; fp64 kernel / here): 64 columns 5.2e-17 / 3.7e-17 - 4.7e-17, 80 5.3e-17 / 3.5e-17 - 4.6e-17, 100 5.2e-17 / 3.0e-17 - 4.2e-17; of few distinct values less.
// From fewer than 64 columns the fp64 kernel loses less (32: 5.2e-17 / 5.1e-17 - 6.5e-17, 16: 5.1e-17 / 6.3e-17): they do not come here.
//
// That error is absolute, an output's terms need not reach their columns' largest values. Columns of B whose outputs do not reach enough of it on average are fp64's
// (k_rmm_digits_b, which says how much is enough). An eighth byte holds a value's magnitude in 1 / 128 of the largest (rounded down), and one more product sums
// those of an output's terms. 32 rows that have an output far below the column's average are marked and left to the fp64 kernel, which follows
// and otherwise finds nothing to do; so are all rows if B holds an infinity or a NaN, and a workgroup's further rows if most of its first ones are.
//
// v_mfma_i32_32x32x32_i8, lane l: A row l % 32, columns 16 (l / 32) .. + 15; B column l % 32, rows alike; D column l % 32, place r row 8 (r / 4) + 4 (l / 32) + r % 4.
// A workgroup of 8 waves, one per CU, takes 256 rows at a time, a wave 32 of them. B's digits stay in LDS; the tables (2 KB a column) come 32 columns at a time:
// a lane looks up 16 columns of its row, 8 bytes each, and turns four columns' bytes into a word of each digit (v_perm), which is the A operand. When all columns are decoded (100 registers)
// the products run, 32 columns of B at a time, three or four weights at a time (a digit of B is read once for them), while the next tables and codes are on their way.
// Up to 4 columns beside a whole number of 32 take one step for all their digits: place 8 column + i of A holds digit i as it comes from the
// table, B's operand of weight w holds digit w - i there: 7 products instead of 28.
//
// Bound: a tile of 256 x 100 rows and 64 columns of B takes 27,000 cycles, 14,000 of them the matrix cores' (380 products per SIMD); decoding (5,600) is LDS reads with barriers
// between, the outputs (128 KB) wait for their turn with the tables behind the products; the clock is 2.0 GHz under this load. 10,000,000 x 100 of 256 values times 64 columns 2.57 ms in fp64, 2.28 - 2.32 here;
// 400,000 rows 171 / 114 us, 150,000 92 / 56, 500 56 / 26; 400,000 x 64 120 / 98 (both in their present form). Taken back: outputs kept until the next tile's products (64 registers more: 3.6 ms), the
// next tables ordered between the products (3.0), products of a step between the look-ups of the next (2.28: LDS and matrix cores still take turns), two columns a
// lane for 16-byte stores (2.29).
#include "../../include/cla_hip.h"
#include "k_rmm_prep.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <type_traits>

namespace cla {

constexpr int RD_THREADS = 512, RD_WAVES = 8, RD_ROWS = 256;
constexpr int RD_COLS = 100;                      // most columns of X
constexpr int RD_TABLE = 2048;                    // bytes of a column's table in LDS and in the image
constexpr int RD_CODES = 2 * 1024 + 128;          // a wave's codes: two steps' 32 columns x 32 rows, 4 x 32 behind them
typedef int i32x4_rd __attribute__((ext_vector_type(4)));
typedef int i32x16_rd __attribute__((ext_vector_type(16)));
typedef double f64x2_rd __attribute__((ext_vector_type(2), aligned(8)));

struct RdArgs {
	const uint8_t* arena;
	size_t arenaStride;
	const int32_t* streams;   // code stream per place
	const uint8_t* tabs;      // tables, RD_TABLE bytes per place
	const uint8_t* bImg;      // B's operands: per 32 columns S * 8 + 8 T pieces of 1 KB
	const double* scale;      // per column of the pass: 2^(exponent - 22)
	const int32_t* least;     // ... sum of magnitudes from which its outputs stand
	const int32_t* bad;       // per 32 columns: B not finite or out of range, or a column that digits do not suit
	const float* over;        // ... above zero over the pass: its columns together
	const double* constRow;
	double* out;
	uint8_t* marks;           // per 32 rows: 1: left to the fp64 kernel
	unsigned long long* nnz;
	int64_t nRows;
	int q, n0, nTiles;        // columns of B, first of the pass
};

// four columns' 4 bytes each -> the four bytes' columns
__device__ __forceinline__ void rd_transpose(uint32_t a, uint32_t b, uint32_t c, uint32_t d, int (&o)[4]) {
	const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u), ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
	const uint32_t cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u), cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
	o[0] = (int) __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
	o[1] = (int) __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
	o[2] = (int) __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
	o[3] = (int) __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
}

// The value, which the compiler takes for a new one: addresses made from it are computed where they are needed, not kept (and spilled) over the loop
__device__ __forceinline__ uint32_t rd_anew(uint32_t x) {
	asm volatile("" : "+v"(x));
	return x;
}

// S steps of 32 columns, T: one of up to 4 behind them, C: 32 columns of B once or twice
template <int S, int T, int C>
__global__ __launch_bounds__(RD_THREADS, 2) void k_rmm_mfma_i8(RdArgs A) {
	extern __shared__ __attribute__((aligned(16))) uint8_t rd_smem[]; // tables of a step, of the last 4 columns, B's operands, codes
	constexpr int PIECES = S * 8 + 8 * T;
	constexpr int oLast = 32 * RD_TABLE, oB = oLast + 4 * T * RD_TABLE, oCodes = oB + C * PIECES * 1024, oCol = oCodes + RD_WAVES * RD_CODES, oStream = oCol + C * 32 * 24;
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	uint8_t* const myCodes = rd_smem + oCodes + wave * RD_CODES;
	// (the lane anew: what is derived from it is computed in each part of a tile, the registers are full between them)
	auto lane_now = [&]() { return (int) rd_anew((uint32_t) lane); };
	const int tile0 = blockIdx.x;
	auto mark = [&](int tile, int m) {
		const int64_t at = (int64_t) tile * RD_WAVES + wave;
		if(lane_now() == 0 && at * 32 < A.nRows) A.marks[at] = (uint8_t) m;
	};
	bool give = A.bad[0] != 0 || (C > 1 && A.bad[C - 1] != 0) || A.over[0] + (C > 1 ? A.over[C - 1] : 0.0f) > 0.0f;
	if(give || tile0 >= A.nTiles) { // (uniform)
		for(int tile = tile0; tile < A.nTiles; tile += gridDim.x) mark(tile, 1);
		return;
	}

	// global -> LDS without registers, 1 KB per wave instruction
	auto copy_by = [&](const uint8_t* src, int to, int bytes, int wave, int waves) {
#pragma unroll 1
		for(int off = wave * 1024; off < bytes; off += waves * 1024)
			__builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) (src + off + (uint32_t) lane_now() * 16u),
				(__attribute__((address_space(3))) void*) (rd_smem + to + off), 16, 0, 0);
	};
	auto copy = [&](const uint8_t* src, int to, int bytes) { copy_by(src, to, bytes, wave, RD_WAVES); };
	// this lane's 16 codes of a step: column 16 h + r / 2, rows 16 (r % 2) of the wave's 32; of the last 4 columns: lanes below 8. Those of the first
	// two steps and of the last columns go straight into LDS a tile ahead (there are no registers for them), the others are requested when the tile begins.
	u32x4 codes[S > 2 ? S - 2 : 1];
	int32_t* const streamS = (int32_t*) (rd_smem + oStream); // [step][lane]
	for(int i = tid; i < (S + T) * 64; i += RD_THREADS) {
		const int s = i >> 6, l = i & 63;
		streamS[i] = A.streams[s < S ? s * 32 + 16 * (l >> 5) + ((l & 31) >> 1) : S * 32 + (l & 7) / 2];
	}
	auto codes_at = [&](int tile, int s, int l) {
		return A.arena + (int64_t) tile * RD_ROWS + wave * 32 + 16 * (l & 1) + (size_t) (uint32_t) streamS[s * 64 + l] * A.arenaStride;
	};
	auto code_to_lds = [&](int tile, int s, int l, int to) {
		__builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) codes_at(tile, s, l), (__attribute__((address_space(3))) void*) (myCodes + to), 16, 0, 0);
	};
	auto load_codes = [&](int tile) {
		const int l = lane_now();
#pragma unroll
		for(int s = 0; s < 2; s++) code_to_lds(tile, s, l, s * 1024);
		if(T && l < 8) code_to_lds(tile, S, l, 2048);
	};
	struct Col { double scale, add; int least, pad; };
	Col* const cols = (Col*) (rd_smem + oCol);
	if(tid < 32 * C) cols[tid] = Col{A.scale[tid], A.constRow != nullptr ? A.constRow[min(A.n0 + tid, A.q - 1)] : 0.0, A.least[tid], 0};

	copy(A.bImg, oB, C * PIECES * 1024);
	if(T) copy(A.tabs + S * 32 * RD_TABLE, oLast, 4 * RD_TABLE);
	copy(A.tabs, 0, 32 * RD_TABLE);
	__syncthreads();
	load_codes(tile0);
	// what this wave has requested has landed, behind the barrier what all waves have
	auto tables_landed = [&]() {
		__builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0)
		lds_barrier();
	};
	// Tables of a step from the second on, on their way into registers (and the codes of that step that have no place in LDS)
	constexpr int PARTS = 32 * RD_TABLE / 16 / RD_THREADS;
	u32x4 stage[PARTS];
	auto request = [&](int tile, int s) {
		const int l = lane_now();
		const uint32_t at16 = (uint32_t) (wave * 64 + l) * 16u;
		if(s == 1) {
#pragma unroll
			for(int i = 2; i < S; i++) codes[i - 2] = *(const u32x4*) codes_at(tile, i, l);
		}
#pragma unroll
		for(int i = 0; i < PARTS; i++) stage[i] = *(const u32x4*) (A.tabs + s * 32 * RD_TABLE + i * RD_THREADS * 16 + at16);
	};
	int cnt = 0;
	// The 32 columns of block c: stores without a branch, so that the compiler knows how many are on their way (what is out of the rows or the columns is dropped by
	// the descriptor's bound). All of one wave instruction are 256-byte pieces of two rows.
	auto put = [&](int tile, int c, const double (&t)[16], bool marked) {
		const int l = lane_now(), r = l & 31, h = l >> 5;
		const int col = A.n0 + 32 * c + r;
		const Col of = cols[32 * c + r];
		const int64_t first = (int64_t) tile * RD_ROWS + wave * 32;
		const int rows = marked ? 0 : (int) max((int64_t) 0, min((int64_t) 32, A.nRows - first));
		const auto to = __builtin_amdgcn_make_buffer_rsrc((void*) (A.out + first * A.q), 0, rows * A.q * 8, 0x00027000);
		const int mine = col < A.q ? (4 * h * A.q + col) * 8 : 0x7fffffff - 256 * A.q;
		double v[16];
#pragma unroll
		for(int i = 0; i < 16; i++) {
			const int row = 8 * (i >> 2) + (i & 3);
			v[i] = __builtin_fma(t[i], of.scale, of.add); // (the scale is a power of two: one rounding)
			__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v[i]), to, mine + row * A.q * 8, 0, 2);
		}
		const uint64_t in = __ballot(col < A.q);
		if(rows == 32) {
#pragma unroll
			for(int i = 0; i < 16; i++) cnt += __builtin_popcountll(__ballot(v[i] != 0.0) & in);
		}
		else
#pragma unroll
			for(int i = 0; i < 16; i++) cnt += __builtin_popcountll(__ballot(4 * h + 8 * (i >> 2) + (i & 3) < rows && v[i] != 0.0) & in);
	};
	tables_landed();
	request(tile0, 1);
#pragma unroll
	for(int i = 0; i < PARTS; i++) asm volatile("" : "+v"(stage[i])); // (nothing on its way where the loop begins: else the wait in it would be for the stores, too)
#pragma unroll
	for(int i = 2; i < S; i++) asm volatile("" : "+v"(codes[i - 2]));
	for(int tile = tile0; tile < A.nTiles; tile += gridDim.x) {
		if(give) {
			mark(tile, 1);
			continue;
		}
		const int next = tile + (int) gridDim.x;
		// ---- decode
		// The first step's tables and the codes have come straight into LDS during the products before; the others' come through registers, requested before
		// the last outputs were stored (loads and stores come back in order) and while the step before is looked up.
		if(wave < RD_WAVES / 2) __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0)
		lds_barrier();
		i32x4_rd a[S][8], last;
		uint32_t code[16];
		auto read_codes = [&](int s) {
			const int l = lane_now(), r = l & 31, h = l >> 5;
			if(s >= 2) *(u32x4*) (myCodes + (s & 1) * 1024 + l * 16) = codes[s - 2];
			const uint8_t* at = myCodes + (s & 1) * 1024 + h * 512 + r;
#pragma unroll
			for(int i = 0; i < 16; i++) code[i] = at[i * 32];
		};
		read_codes(0);
#pragma unroll
		for(int s = 0; s < S; s++) {
			const int l = lane_now(), r = l & 31, h = l >> 5;
			const uint32_t at16 = (uint32_t) (wave * 64 + l) * 16u;
			u32x2 v[16];
#pragma unroll
			for(int i = 0; i < 16; i++) v[i] = *(const u32x2*) (rd_smem + h * 16 * RD_TABLE + i * RD_TABLE + (code[i] << 3));
			if(s + 1 < S) read_codes(s + 1);
			__builtin_amdgcn_sched_barrier(0); // (all on their way before the first is needed)
#pragma unroll
			for(int g = 0; g < 4; g++) {
				int o[4];
				rd_transpose(v[4 * g].x, v[4 * g + 1].x, v[4 * g + 2].x, v[4 * g + 3].x, o);
#pragma unroll
				for(int d = 0; d < 4; d++) a[s][d][g] = o[d];
				rd_transpose(v[4 * g].y, v[4 * g + 1].y, v[4 * g + 2].y, v[4 * g + 3].y, o);
#pragma unroll
				for(int d = 0; d < 4; d++) a[s][4 + d][g] = o[d];
			}
			if(T && s == 0) {
				const uint8_t* al = myCodes + 2048 + h * 64 + r;
#pragma unroll
				for(int i = 0; i < 2; i++) {
					const uint32_t code = al[i * 32];
					const u32x2 v = *(const u32x2*) (rd_smem + oLast + (2 * h + i) * RD_TABLE + (code << 3));
					last[2 * i] = (int) v.x;
					last[2 * i + 1] = (int) v.y;
				}
			}
			lds_barrier(); // all waves have looked up: the next step's tables may come
			if(s + 1 < S) {
#pragma unroll
				for(int i = 0; i < PARTS; i++) *(u32x4*) (rd_smem + i * RD_THREADS * 16 + at16) = stage[i];
				if(s + 2 < S) request(tile, s + 2);
				lds_barrier();
			}
		}
		if(next < A.nTiles) {
			if(C == 1) load_codes(next);
		}

		// ---- multiply
		const int l = lane_now();
		const int rows = (int) max((int64_t) 0, min((int64_t) 32, A.nRows - ((int64_t) tile * RD_ROWS + wave * 32)));
		auto b_at = [&](int c, int piece) { return *(const i32x4_rd*) (rd_smem + oB + (c * PIECES + piece) * 1024 + l * 16); };
		i32x16_rd m[C];
#pragma unroll
		for(int c = 0; c < C; c++)
#pragma unroll
			for(int i = 0; i < 16; i++) m[c][i] = 0;
		auto magnitudes = [&](int s0, int s1) {
			i32x4_rd bm[S + T][C];
#pragma unroll
			for(int s = s0; s < s1; s++)
#pragma unroll
				for(int c = 0; c < C; c++) bm[s][c] = b_at(c, s * 8 + 7);
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for(int s = s0; s < s1; s++)
#pragma unroll
				for(int c = 0; c < C; c++) m[c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(s < S ? a[s < S ? s : 0][7] : last, bm[s][c], m[c], 0, 0, 0);
			bool low = false;
#pragma unroll
			for(int c = 0; c < C; c++) {
				const int least = cols[32 * c + (l & 31)].least;
				if(rows < 32) {
					const int left = rows - 4 * (l >> 5);
#pragma unroll
					for(int i = 0; i < 16; i++) low |= 8 * (i >> 2) + (i & 3) < left && m[c][i] < least;
				}
				else {
					int lowest = m[c][0];
#pragma unroll
					for(int i = 1; i < 16; i++) lowest = min(lowest, m[c][i]);
					low |= lowest < least;
				}
			}
			return __ballot(low) != 0;
		};
		bool marked = magnitudes(0, 2); // (64 columns' sums are nearly always enough)
		if(marked && S + T > 2) marked = magnitudes(2, S + T);
		__builtin_amdgcn_sched_barrier(0);
		mark(tile, marked);
#pragma unroll
		for(int c = 0; c < C; c++) {
			double t[16];
#pragma unroll
			for(int half = 1; half >= 0; half--) { // weights 4 - 6, 0 - 3
				constexpr int J1 = 7, J0 = 4; // digits of B in them
				const int W = half ? 3 : 4;
				const int J = half ? J1 : J0, N = S * J + W * T;
				i32x16_rd acc[4];
#pragma unroll
				for(int w = 0; w < 4; w++)
#pragma unroll
					for(int i = 0; i < 16; i++) acc[w][i] = 0;
				auto piece = [&](int n) { return n < S * J ? n / J * 8 + n % J : S * 8 + 4 * half + n - S * J; };
				i32x4_rd b[2];
				b[0] = b_at(c, piece(0));
#pragma unroll
				for(int n = 0; n < N; n++) {
					if(n + 1 < N) b[(n + 1) & 1] = b_at(c, piece(n + 1));
					if(n < S * J) {
#pragma unroll
						for(int w = 0; w < W; w++) {
							const int i = 4 * half + w - n % J;
							if(i >= 0 && i <= 6) acc[w] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[n / J][i], b[n & 1], acc[w], 0, 0, 0);
						}
					}
					else acc[n - S * J] = __builtin_amdgcn_mfma_i32_32x32x32_i8(last, b[n & 1], acc[n - S * J], 0, 0, 0);
					__builtin_amdgcn_sched_barrier(0);
				}
				// two weights' sums in one 32-bit number: a weight w's is at most (w + 1) 2^14 a column, and 256 times that of weight 4 below 2^31 - 2^25
				static_assert(5 * (S * 32 + 4 * T) <= 500, "");
				if(half == 1) {
#pragma unroll
					for(int i = 0; i < 16; i++) t[i] = (double) acc[2][i];
				}
#pragma unroll
				for(int w = half ? 0 : 2; w >= 0; w -= 2) {
					const double down = half ? 1.0 / 256.0 : 1.0 / 65536.0;
#pragma unroll
					for(int i = 0; i < 16; i++) {
						t[i] = __builtin_fma(t[i], down, (double) (acc[w][i] * 256 + acc[w + 1][i]));
						if(w == 0) asm volatile("" : "+v"(t[i])); // (here, not where it is stored: the sums it is made from take twice its registers)
					}
				}
				__builtin_amdgcn_sched_barrier(0);
			}
			if(c == C - 1) { // (before its stores: a wait for what comes behind them would be one for them)
				__builtin_amdgcn_s_waitcnt(C == 1 ? 0x0f70 : 0x4f70); // the codes have landed: vmcnt(0), or 16, the stores of the first block's columns
				request(min(next, A.nTiles - 1), 1);
				__builtin_amdgcn_sched_barrier(0);
			}
			if(C > 1 && c == 0 && next < A.nTiles) load_codes(next);
			put(tile, c, t, marked);
			__builtin_amdgcn_sched_barrier(0);
		}
		// (by the waves that go first where two share a SIMD: they are done with the tile long before the others)
		if(wave < RD_WAVES / 2 && next < A.nTiles) copy_by(A.tabs, 0, 32 * RD_TABLE, wave, RD_WAVES / 2);
		// most of the first rows are marked: the others will be, too
		if(tile == tile0) give = __syncthreads_count(marked && lane == 0) > RD_WAVES / 2;
	}
	__builtin_amdgcn_s_waitcnt(0x0f70); // (rows given up: tables for them may be on their way into LDS)
	count_add(A.nnz, lane == 0 ? cnt : 0);
}

// ---- B's operands

static_assert(MF_BL_THREADS == 256, "blocks of k_rmm_digits_b");
constexpr int RB_THREADS = MF_BL_THREADS, RB_PIECES = 32; // (3 steps of 8, and 8)
constexpr double RD_LOST = 1.2e-16, RD_FP64 = 4.5e-17;    // (1.1e-16 for the products of weight 7, the rest for the values' rounding)
// Block c: 32 columns of B of the pass into their operands, scales and least sums. What the digits leave out of an output is RD_LOST sqrt(K / 100) (rms) of the largest possible
// term, whatever the values, and how far an output's terms come on average is known from X's mean magnitudes: a column's mean error is the quotient. The pass goes
// to fp64 if the rms of that over its columns exceeds RD_FP64, the least that fp64 leaves of values that are not short, or one column's 2^-53; rows are left to
// fp64 where an output's terms come to a fifth of the column's mean only. (Rms error over the sum of the terms' magnitudes, fp64 / digits, expected: normal values 64 columns
// 5.3e-17 / 3.9e-17, 3.6e-17, 100 5.1e-17 / 3.2e-17, 3.0e-17, uniform 4.5e-17 / 1.6e-17, 1.5e-17; in fp64 then: B of Student's t, 3 degrees 5.8e-17 / 6.9e-17,
// X of it 6.0e-17 / 1.6e-16, X lognormal 6.6e-17 / 1.5e-16, X normal with one value at 8 5.5e-17 / 1.1e-16.)
// leastSum > 0: rows whose outputs' terms come to that are enough, whatever the columns'.
// The blocks behind those make what the fp64 kernel reads (mf_prep).
__global__ __launch_bounds__(RB_THREADS) void k_rmm_digits_b(const MfPrep P, int blocks, int K, int S, int T, const int32_t* __restrict__ rowCol,
	const double* __restrict__ up, const double* __restrict__ mean, uint8_t* __restrict__ bImg, double* __restrict__ scale, int32_t* __restrict__ least, int32_t* __restrict__ bad,
	float* __restrict__ over, int leastSum) {
	if((int) blockIdx.x >= blocks) {
		mf_prep(P, (int) blockIdx.x - blocks);
		return;
	}
	const double* __restrict__ const B = P.B;
	const int q = P.q, n0 = P.n0;
	__shared__ __attribute__((aligned(16))) uint8_t img[RB_PIECES * 1024];
	__shared__ double most[RB_THREADS / 32][32];
	__shared__ int badS;
	const int c = blockIdx.x, tid = threadIdx.x, r = tid & 31, slice = tid >> 5, col = n0 + 32 * c + r;
	const int pieces = S * 8 + 8 * T;
	// all of a thread's values requested at once, in two round trips (walked twice, one after the other, they took 14.5 us of a call, 7.0 now). up[k]: 2^(exponent
	// of X's column k)
	constexpr int VALS = (RD_COLS + RB_THREADS / 32 - 1) / (RB_THREADS / 32);
	double v[VALS], xm[VALS];
	{
		int32_t at[VALS];
#pragma unroll
		for(int i = 0; i < VALS; i++) at[i] = rowCol[min(slice + i * (RB_THREADS / 32), K - 1)];
#pragma unroll
		for(int i = 0; i < VALS; i++) xm[i] = mean[min(slice + i * (RB_THREADS / 32), K - 1)];
#pragma unroll
		for(int i = 0; i < VALS; i++) v[i] = B[(size_t) at[i] * q + min(col, q - 1)] * up[min(slice + i * (RB_THREADS / 32), K - 1)];
	}
	if(tid == 0) badS = 0;
	for(int i = tid; i < pieces * 256; i += RB_THREADS) ((uint32_t*) img)[i] = 0;
	double m = 0.0;
	bool odd = false;
#pragma unroll
	for(int i = 0; i < VALS; i++) {
		if(col >= q || slice + i * (RB_THREADS / 32) >= K) v[i] = 0.0;
		odd |= !(fabs(v[i]) <= 1e300); // (a NaN, an infinity or close to it)
		m = fabs(v[i]) > m ? fabs(v[i]) : m;
	}
	most[slice][r] = m;
	__syncthreads();
	for(int i = 0; i < RB_THREADS / 32; i++) m = most[i][r] > m ? most[i][r] : m;
	int e = 0;
	if(m > 0.0) {
		const double f = frexp(m, &e);
		if(f >= 0.99) e++;
	}
	odd |= m > 0.0 && e < -900;
	double terms = 0.0;
#pragma unroll
	for(int i = 0; i < VALS; i++) terms += xm[i] * fabs(ldexp(v[i], -e)); // (zeros from K on)
	__syncthreads();
	most[slice][r] = terms;
	__syncthreads();
	if(slice == 0) {
		for(int i = 1; i < RB_THREADS / 32; i++) terms += most[i][r];
		const double lost = RD_LOST * sqrt(K * 0.01) / terms; // (a column of zeros: nothing)
		const bool any = m > 0.0 && leastSum == 0;
		odd |= any && !(lost <= 0x1p-53);
		scale[32 * c + r] = ldexp(1.0, e - 22);
		least[32 * c + r] = any ? (int) fmin(16384.0 / 5 * terms, 1e9) : m > 0.0 ? leastSum : 0;
		float o = any ? (float) (lost * lost / (RD_FP64 * RD_FP64)) - 1.0f : 0.0f;
#pragma unroll
		for(int d = 1; d < 32; d *= 2) o += __shfl_xor(o, d);
		if(r == 0) over[c] = o;
	}
	if(odd) badS = 1;
	if(col < q)
#pragma unroll
		for(int j = 0; j < VALS; j++) {
			const int k = slice + j * (RB_THREADS / 32);
			if(k >= K) break;
			const double x = ldexp(v[j], -e);
			int64_t X = odd ? 0 : (int64_t) rint(x * (double) ((int64_t) 1 << 55));
			const int mag = odd ? 0 : min(127, (int) (fabs(x) * 128.0));
			int d[7];
#pragma unroll
			for(int i = 6; i > 0; i--) {
				d[i] = (int) (int8_t) (uint8_t) (X & 255);
				X = (X - d[i]) >> 8;
			}
			d[0] = (int) X;
			const int kk = k & 31;
			if(k < S * 32) {
				uint8_t* const at = img + (k >> 5) * 8192 + ((kk >> 4) * 32 + r) * 16 + (kk & 15);
#pragma unroll
				for(int i = 0; i < 7; i++) at[i * 1024] = (uint8_t) d[i];
				at[7 * 1024] = (uint8_t) mag;
			}
			else { // place 8 kk + i of weight w: digit w - i
				uint8_t* const at = img + S * 8192 + ((kk >> 1) * 32 + r) * 16 + (kk & 1) * 8;
#pragma unroll
				for(int w = 0; w < 7; w++)
#pragma unroll
					for(int i = 0; i <= w; i++) at[w * 1024 + i] = (uint8_t) d[w - i];
				at[7 * 1024 + 7] = (uint8_t) mag;
			}
		}
	__syncthreads();
	u32x4* const to = (u32x4*) (bImg + (size_t) c * pieces * 1024);
	for(int i = tid; i < pieces * 64; i += RB_THREADS) to[i] = ((const u32x4*) img)[i];
	if(tid == 0) bad[c] = badS;
}

constexpr int RM_THREADS = 256, RM_ONE = 1 << 20;
// sums[place] += the sum over the rows of column `place`'s magnitudes, in 1 / RM_ONE of its scale (mags, 256 codes a place). (Once per block: 10,000,000 x 100 0.30 ms.)
__global__ __launch_bounds__(RM_THREADS) void k_rmm_digits_means(const uint8_t* __restrict__ arena, size_t arenaStride, const int32_t* __restrict__ streams,
	const uint32_t* __restrict__ mags, int64_t nRows, unsigned long long* __restrict__ sums) {
	__shared__ uint32_t tab[256];
	const int place = blockIdx.y, tid = threadIdx.x;
	tab[tid] = mags[place * 256 + tid];
	__syncthreads();
	const uint8_t* const stream = arena + (size_t) (uint32_t) streams[place] * arenaStride;
	unsigned long long sum = 0;
	for(int64_t row = ((int64_t) blockIdx.x * RM_THREADS + tid) * 16; row < nRows; row += (int64_t) gridDim.x * RM_THREADS * 16) {
		const u32x4 codes = *(const u32x4*) (stream + row);
		uint32_t s = 0;
#pragma unroll
		for(int i = 0; i < 16; i++) s += row + i < nRows ? tab[(codes[i >> 2] >> (8 * (i & 3))) & 0xffu] : 0u;
		sum += s;
	}
#pragma unroll
	for(int d = 1; d < WAVE; d *= 2) sum += __shfl_xor(sum, d, WAVE);
	if((tid & (WAVE - 1)) == 0) atomicAdd(&sums[place], sum);
}

constexpr int RL_THREADS = 512, RL_TILES = RL_THREADS * 4 / 512; // 4 rows a thread; 512 rows are a tile of the fp64 kernel
// low += the tiles of 512 rows with a row whose magnitudes (mags, 256 codes a place, in any unit) sum to less than `least`. (Once per block: 10,000,000 x 100 0.19 ms.)
__global__ __launch_bounds__(RL_THREADS) void k_rmm_digits_low(const uint8_t* __restrict__ arena, size_t arenaStride, const int32_t* __restrict__ streams,
	const uint16_t* __restrict__ mags, int K, int64_t nRows, uint32_t least, int* __restrict__ low) {
	extern __shared__ __attribute__((aligned(16))) uint16_t rl_smem[];
	__shared__ int lowS[RL_TILES];
	const int tid = threadIdx.x;
	for(int i = tid; i < K * 256; i += RL_THREADS) rl_smem[i] = mags[i];
	int n = 0;
	for(int64_t row0 = (int64_t) blockIdx.x * RL_THREADS * 4; row0 < nRows; row0 += (int64_t) gridDim.x * RL_THREADS * 4) {
		if(tid < RL_TILES) lowS[tid] = 0;
		__syncthreads();
		const int64_t row = row0 + tid * 4;
		uint32_t s[4] = {0, 0, 0, 0};
		if(row < nRows) { // (the streams are padded to more than 4 rows)
#pragma unroll 8
			for(int k = 0; k < K; k++) {
				const uint32_t codes = *(const uint32_t*) (arena + (size_t) (uint32_t) streams[k] * arenaStride + row);
#pragma unroll
				for(int i = 0; i < 4; i++) s[i] += rl_smem[k * 256 + ((codes >> (8 * i)) & 0xffu)];
			}
#pragma unroll
			for(int i = 0; i < 4; i++)
				if(row + i < nRows && s[i] < least) lowS[tid / 128] = 1;
		}
		__syncthreads();
		if(tid == 0)
			for(int t = 0; t < RL_TILES; t++) n += lowS[t];
		__syncthreads();
	}
	if(tid == 0 && n > 0) atomicAdd(low, n);
}

struct RdPlan {
	int rc = 0; // 1: not of this kernel's shape
	RdArgs A;
	void* dImg = nullptr;
	int64_t bytes = 0;
	const int32_t* rowCol = nullptr;
	const double *up = nullptr, *mean = nullptr;
	uint8_t* bImg = nullptr;
	double* scale = nullptr;
	int32_t *least = nullptr, *bad = nullptr;
	float* over = nullptr;
	int K = 0, S = 0, T = 0;
	bool suits = true; // a B of even magnitudes could come to what fp64 leaves, and would leave it few rows
	~RdPlan() { if(dImg) (void) hipFree(dImg); }
};

void rd_plan_drop(cla_block* b) {
	if(b->rdPlan == nullptr) return;
	b->derivedBytes -= b->rdPlan->bytes;
	delete b->rdPlan;
	b->rdPlan = nullptr;
}

// 1: no room on the device for the plan
static int rd_build_plan(cla_block* b, RdPlan& P) {
	P.rc = 1;
	if(b->dArena == nullptr || b->arenaWidth != 1 || b->dictNonFinite || b->nRows == 0) return 0;
	int K = 0;
	for(const HostGroup& H : b->groups) K += H.d.nColG;
	const int rest = K % 32, T = rest >= 1 && rest <= 4 ? 1 : 0, S = T ? K / 32 : (K + 31) / 32;
	if(K < 64 || K > RD_COLS) return 0;
	P.K = K; P.S = S; P.T = T;
	const int places = S * 32 + 4 * T;
	std::vector<int32_t> streams((size_t) places, 0), rowCol((size_t) places, 0);
	std::vector<double> up((size_t) places, 1.0), mean((size_t) places, 0.0); // (mean: of a column's magnitudes, in parts of its scale)
	std::vector<uint32_t> mags((size_t) places * 256, 0);
	std::vector<uint8_t> tabs((size_t) places * RD_TABLE, 0);
	int place = 0;
	for(size_t g = 0; g < b->groups.size(); g++) {
		const HostGroup& H = b->groups[g];
		const int nc = H.d.nColG, nV = H.d.nVals;
		for(int j = 0; j < nc; j++, place++) {
			double most = 0.0;
			for(int i = 0; i < nV; i++) most = std::max(most, std::fabs(H.dict[(size_t) i * nc + j]));
			int e = 0;
			if(most > 0.0 && std::frexp(most, &e) >= 0.99) e++;
			if(e < -300 || e > 300) return 0;
			streams[place] = (int32_t) g;
			rowCol[place] = H.cols[j];
			up[place] = std::ldexp(1.0, e);
			const double down = std::ldexp(1.0, -e);
			for(int i = 0; i < nV; i++) {
				const double x = H.dict[(size_t) i * nc + j] * down;
				int64_t X = (int64_t) std::nearbyint(x * (double) ((int64_t) 1 << 55));
				uint8_t* d = tabs.data() + (size_t) place * RD_TABLE + (size_t) i * 8;
				for(int t = 6; t > 0; t--) {
					const int v = (int) (int8_t) (uint8_t) (X & 255);
					d[t] = (uint8_t) v;
					X = (X - v) >> 8;
				}
				d[0] = (uint8_t) X;
				d[7] = (uint8_t) std::min(127, (int) (std::fabs(x) * 128.0));
				mags[(size_t) place * 256 + i] = (uint32_t) (std::fabs(x) * RM_ONE);
			}
		}
	}
	auto up256 = [](size_t n) { return (n + 255) & ~(size_t) 255; };
	const size_t oRow = up256((size_t) places * 4), oUp = oRow + up256((size_t) places * 4), oMean = oUp + up256((size_t) places * 8);
	const size_t oTabs = oMean + up256((size_t) places * 8), oB = oTabs + tabs.size();
	const size_t oScale = oB + (size_t) 2 * RB_PIECES * 1024, oLeast = oScale + 512, oBad = oLeast + 256, oMarks = oBad + 256;
	const size_t total = oMarks + up256((size_t) (b->nRows + 511) / 512 * 16);
	std::vector<uint8_t> all(oB, 0);
	std::memcpy(all.data(), streams.data(), streams.size() * 4);
	std::memcpy(all.data() + oRow, rowCol.data(), rowCol.size() * 4);
	std::memcpy(all.data() + oUp, up.data(), up.size() * 8);
	std::memcpy(all.data() + oTabs, tabs.data(), tabs.size());
	uint8_t* d = nullptr;
	if(no_room((void**) &d, total)) return 1;
	P.dImg = d;
	P.bytes = (int64_t) total;
	CLA_HIP(hipMemcpy(d, all.data(), all.size(), hipMemcpyHostToDevice));
	CLA_HIP(hipMemset(d + oMarks, 0, total - oMarks)); // (behind the last row)
	{
		struct Tmp { void* p = nullptr; ~Tmp() { if(p) (void) hipFree(p); } } tmp;
		const size_t sumBytes = up256((size_t) places * 8);
		if(no_room(&tmp.p, sumBytes + mags.size() * 4)) return 1;
		CLA_HIP(hipMemsetAsync(tmp.p, 0, sumBytes, b->stream));
		CLA_HIP(hipMemcpyAsync((char*) tmp.p + sumBytes, mags.data(), mags.size() * 4, hipMemcpyHostToDevice, b->stream));
		const unsigned gx = (unsigned) std::min<int64_t>((b->nRows + RM_THREADS * 16 - 1) / (RM_THREADS * 16), (8 * g_numCU + K - 1) / K);
		hipLaunchKernelGGL(k_rmm_digits_means, dim3(gx, (unsigned) K), dim3(RM_THREADS), 0, b->stream, b->dArena, b->arenaStride, (const int32_t*) d,
			(const uint32_t*) ((char*) tmp.p + sumBytes), b->nRows, (unsigned long long*) tmp.p);
		CLA_HIP(hipGetLastError());
		std::vector<unsigned long long> sums((size_t) K);
		CLA_HIP(hipMemcpyAsync(sums.data(), tmp.p, (size_t) K * 8, hipMemcpyDeviceToHost, b->stream));
		CLA_HIP(hipStreamSynchronize(b->stream));
		double all = 0.0;
		for(int k = 0; k < K; k++) all += mean[k] = (double) sums[k] / RM_ONE / (double) b->nRows;
		P.suits = 0.5 * all >= RD_LOST / RD_FP64 * std::sqrt(K / 100.0);
		// Rows whose magnitudes are below a quarter of the mean would be marked whatever B, and 512 rows with one of them go through both kernels (us, fp64 / here: 2,000,000 x 100 by
		// 64 with no such tile 570 / 437 - 462, 10 % 570 / 547 - 616, 22 % 570 / 665 - 747, all 570 / 933; 60,000 rows, whose one round of tiles is all or nothing, none 56 / 28, one and more 56 / 60 - 79).
		if(P.suits) {
			double largest = 0.0, sum = 0.0;
			for(int k = 0; k < K; k++) {
				largest = std::max(largest, up[k]);
				sum += mean[k] * up[k];
			}
			std::vector<uint16_t> share((size_t) K * 256);
			for(size_t i = 0; i < share.size(); i++) share[i] = (uint16_t) (mags[i] * (65535.0 / RM_ONE) * (up[i / 256] / largest));
			int low = 0;
			CLA_HIP(hipMemcpyAsync((char*) tmp.p + sumBytes, share.data(), share.size() * 2, hipMemcpyHostToDevice, b->stream));
			CLA_HIP(hipMemsetAsync(tmp.p, 0, sizeof(int), b->stream));
			const int64_t tiles = (b->nRows + 511) / 512;
			const unsigned blocks = (unsigned) std::min<int64_t>((tiles + RL_TILES - 1) / RL_TILES, 3 * g_numCU);
			hipLaunchKernelGGL(k_rmm_digits_low, dim3(blocks), dim3(RL_THREADS), (size_t) K * 512, b->stream, b->dArena, b->arenaStride, (const int32_t*) d,
				(const uint16_t*) ((char*) tmp.p + sumBytes), K, b->nRows, (uint32_t) (sum / largest * 65535.0 / 4), (int*) tmp.p);
			CLA_HIP(hipGetLastError());
			CLA_HIP(hipMemcpyAsync(&low, tmp.p, sizeof(int), hipMemcpyDeviceToHost, b->stream));
			CLA_HIP(hipStreamSynchronize(b->stream));
			P.suits = low == 0 || (tiles > 2 * g_numCU && low * 20 <= tiles);
		}
		CLA_HIP(hipMemcpy(d + oMean, mean.data(), mean.size() * 8, hipMemcpyHostToDevice));
	}
	P.rowCol = (const int32_t*) (d + oRow); P.up = (const double*) (d + oUp); P.mean = (const double*) (d + oMean);
	P.bImg = d + oB; P.scale = (double*) (d + oScale); P.least = (int32_t*) (d + oLeast); P.bad = (int32_t*) (d + oBad); P.over = (float*) (d + oBad + 128);
	RdArgs& A = P.A;
	A.arena = b->dArena; A.arenaStride = b->arenaStride;
	A.streams = (const int32_t*) d; A.tabs = d + oTabs; A.bImg = P.bImg;
	A.scale = P.scale; A.least = P.least; A.bad = P.bad; A.over = P.over; A.marks = d + oMarks;
	A.nRows = b->nRows; A.nTiles = (int) ((b->nRows + RD_ROWS - 1) / RD_ROWS);
	P.rc = 0;
	return 0;
}

// Where this pays, p columns of B in the pass (us, fp64 / here, 256 values): up to 200,000 rows always, 500 x 64 of 8 columns of B 25 / 17, 500 x 100 of 64 56 / 26, 150,000 x 64
// of 8 34 / 30, x 72 of 8 36 / 36, of 64 67 / 55, x 100 of 64 92 / 56. Past that, 16 columns of B at most (half of the products are for nothing) 250,000 x 64 of 8 34 / 36, x 100 of
// 16 52 / 49, 400,000 x 80 71 / 72, 1,000,000 x 80 119 / 146, 3,000,000 x 100 368 / 436; 33 - 48 columns (the fp64 kernel is at its best) 250,000 x 80 of 40 66 / 67, 400,000
// 121 / 106, 1,000,000 x 80 of 48 220 / 230, x 100 250 / 231, 3,000,000 x 100 631 / 669; 17 - 32 and 49 - 64 at any number of rows, 3,000,000 x 64 of 32 350 / 317, x 80
// 428 / 407, of 64 665 / 645, x 100 805 / 697. 69 - 79 columns (the last step a fifth or a half full), of 32 and of 64 columns of B, 250,000 x 72 45 / 48 and 66 / 70, x 78 54 / 48 and
// 76 / 71, 400,000 x 72 84 / 74 and 129 / 109, 1,000,000 147 / 151 and 233 / 228, 3,000,000 378 / 399 and 599 / 634: left to fp64, with what some 400,000 rows of them would give.
static bool rd_pays(const cla_block* b, int K, int p) {
	if(p < 8) return false;
	if(b->nRows <= 200000) return true;
	if((K > 68 && K < 80) || p <= 16) return false;
	return p <= 32 || p > 48 || b->nRows <= 1000000;
}

// 0: columns n0 .. of B go this way (the block's plan is made), 1: they do not, negative: an error.
int rmm_digits_plan(cla_block* b, int q, int n0) {
	if(b->opt.rmmDigits == 0 || q > 1 << 20) return 1; // (byte offsets of 256 rows of the output in 31 bits)
	int K = 0;
	for(const HostGroup& H : b->groups) K += H.d.nColG;
	if(b->opt.rmmDigits == 1 && !rd_pays(b, K, std::min(64, q - n0))) return 1;
	if(b->rdPlan == nullptr) {
		// (a block prepared for other widths, which the rule may leave to fp64: a capture refuses the plan's allocation)
		hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
		CLA_HIP(hipStreamIsCapturing(b->stream, &capturing));
		if(capturing != hipStreamCaptureStatusNone) return 1;
		std::unique_ptr<RdPlan> plan(new RdPlan()); // (the block's only when it is complete)
		const int rc = rd_build_plan(b, *plan);
		if(rc) return rc;
		b->derivedBytes += plan->bytes;
		b->rdPlan = plan.release();
	}
	return b->rdPlan->rc || (b->opt.rmmDigits == 1 && !b->rdPlan->suits);
}

template <int S, int T, int C>
static int rd_launch(cla_block* b, const RdArgs& A) {
	constexpr int lds = 32 * RD_TABLE + 4 * T * RD_TABLE + C * (S * 8 + 8 * T) * 1024 + RD_WAVES * RD_CODES + C * 32 * 24 + (S + T) * 256;
	const unsigned grid = (unsigned) std::min(A.nTiles, g_numCU);
	Prof pf(b, "k_rmm_mfma_i8", grid, RD_THREADS, lds, (double) b->device_bytes_cached + (double) b->nRows * std::min(32 * C, A.q - A.n0) * 8);
	CLA_HIP(allow_full_lds((const void*) k_rmm_mfma_i8<S, T, C>));
	hipLaunchKernelGGL((k_rmm_mfma_i8<S, T, C>), dim3(grid), dim3(RD_THREADS), lds, b->stream, A);
	CLA_HIP(hipGetLastError());
	return 0;
}

// Up to 64 columns of B from n0 on; the rows that are left (*marks: per 32 rows) are the caller's.
int launch_rmm_digits(cla_block* b, const MfPrep& prep, double* dOut, unsigned long long* dNnz, const uint8_t** marks) {
	const int q = prep.q, n0 = prep.n0;
	const RdPlan& P = *b->rdPlan;
	const int cols = std::min(64, q - n0), c32 = (cols + 31) / 32;
	// asked for by option: 2^-2 sqrt(K / 100) of the largest possible term, in squares of 1 / 128
	const int leastSum = b->opt.rmmDigits == 2 ? (int) (16384.0 / 4 * std::sqrt(P.K / 100.0)) : 0;
	{
		const int blocks = c32 + prep.blocks();
		Prof pf(b, "k_rmm_digits_b", blocks, RB_THREADS, 0, 0);
		hipLaunchKernelGGL(k_rmm_digits_b, dim3((unsigned) blocks), dim3(RB_THREADS), 0, b->stream, prep, c32, P.K, P.S, P.T, P.rowCol, P.up, P.mean, P.bImg, P.scale,
			P.least, P.bad, P.over, leastSum);
	}
	RdArgs A = P.A;
	A.constRow = prep.constRow; A.out = dOut; A.nnz = dNnz; A.q = q; A.n0 = n0;
	*marks = A.marks;
#define RD_CASE(SV, TV) case SV * 2 + TV: return c32 == 1 ? rd_launch<SV, TV, 1>(b, A) : rd_launch<SV, TV, 2>(b, A);
	switch(P.S * 2 + P.T) { RD_CASE(2, 0) RD_CASE(2, 1) RD_CASE(3, 0) RD_CASE(3, 1) }
#undef RD_CASE
	return 1;
}

} // namespace cla
