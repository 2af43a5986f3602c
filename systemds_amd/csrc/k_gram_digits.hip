// t(X) %*% X of a block whose groups are all DDC with byte codes, 17 to 112 columns, on the 8-bit integer matrix cores.
//
// A column's values (dictionary + constant) are scaled by a power of two to |x| < 1 and rounded to X = x 2^55, a whole number of seven signed
// base-256 digits. A row's lookup brings all seven (8 bytes, like the fp64 value), the products of digits i + j <= 6 are
// summed as 32-bit integers, exactly, one sum per weight i + j, and at the end or every 18,688 rows the seven sums are joined in fp64. So
// a cell's error is that of the rounded values (2^-56 of the column's largest) and of the products left out (six of up to 2^-56 of both columns'
// largest), not that of chains of fp64 additions. It is absolute, in parts of the columns' largest values; gd_build_plan and gd_compare say which blocks
// that suits. Rms over cells of the error divided by the sum of the terms' magnitudes, against exact counts times products in long double, 256 normal
// values, Zipf(1.1) codes (k_gram_tiles): 2,000,003 x 100 3.5e-17 (1.2e-15); more beside gd_compare. The same sums in every call: no atomic adds.
//
// A workgroup of 8 waves, one per CU, takes a contiguous share of the rows in tiles of 64 rows per set of waves. Decoding is dealt by (16 columns, 64
// rows): lane (k, c) looks up 16 consecutive codes of column c (in LDS where the column block's tables fit beside the tile, else in global
// memory), turns the 16 x 7 bytes into seven 16-byte vectors (v_perm) and, once all waves are done with the tile before, writes
// them where lane (k, c) of a reader finds them: both operands of v_mfma_i32_16x16x64_i8 are such vectors. Pairs of column blocks are
// dealt to the waves so that a wave's pairs share few blocks (its reads) and the four SIMDs have the same work (gd_role).
//
// Why integers: 28 products of 16 cycles per 64 rows and pair of column blocks stand against 16 fp64 steps of 64 (v_mfma_f64_16x16x4), and,
// unlike those, leave the SIMD's vector unit to the other wave. 2,000,003 x 100 441 -> 289 us (of 40 values, all tables in LDS, 235 without the join), 200,003 x 100
// 97 -> 52, 2,000,003 x 64 209 -> 119, x 40 121 -> 90, x 20 65 -> 53.
// Bound: the integer matrix pipe (2,400 cycles per 64 rows of 100 columns at 8.5 ns per 16: the clock drops under it; two buffers for the tile, or the lookups
// elsewhere in it, change nothing) and, where tables are in global memory, the vector memory path: a lookup of 64 lanes takes it 57 cycles.
#include "../../include/cla_hip.h"
#include "cla_device.hpp"
#include "cla_runs.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <memory>

namespace cla {

constexpr int GD_THREADS = 512, GD_DIGITS = 7;
constexpr int GD_BITS = 55;             // X = x 2^GD_BITS, |x| < 127.5 / 128: the first digit fits
constexpr int GD_CHUNK = 18688;         // rows between two joins: a weight's sum grows by at most 7 2^14 a row
constexpr int GD_MAG = 128;             // magnitudes of the rules below in 1 / GD_MAG
typedef int i32x4_gd __attribute__((ext_vector_type(4)));

// a decoded column
struct GdCol {
	uint32_t tab;     // bytes from the tables' start to its first entry (8 bytes per code: digits, magnitude)
	int32_t stream;   // code stream
	int32_t group;    // -1: only a constant
	int32_t col;      // column of the block (-1: padding)
	double scale;     // 2^(e - 7): value = X 2^(e - 55)
};

struct GdArgs {
	const uint8_t* arena;
	size_t arenaStride;
	const GdCol* cols;   // 16 per full column block, 4 of the narrow one
	const uint8_t* tabs;
	int64_t nRows;
	int nTiles, nLds, ldsTab; // column blocks [0, nLds) have their tables in LDS, as the narrow one has: the first ldsTab bytes
	double* parts;       // per workgroup gd_slots() x 256 sums
	double* setParts;    // several sets of waves, shares of more than GD_CHUNK rows: the same per set
	unsigned long long* nnz;
};

// ---- who multiplies what
//
// The column blocks are NF blocks of 16 columns, in the kernels with NARROW = 1 followed by one of at most 4 whose digits share two operands: row 4 i + column
// of the first holds digit i = 0 .. 3 of a column, of the second digit 4 + i. Against a block's digit j they take one product or, for j <= 2, two: 10 instead of 28.

// A pair of column blocks p < q, all 28 products of it or a half (weights 0, 5, 6 or 1 - 4, 14 products each); a block with itself
// (digits i <= j: 16 products, the cell takes those with i < j from both sides of the diagonal); the narrow block with block p; with itself.
enum : int { GD_FULL, GD_HALF_A, GD_HALF_B, GD_OWN, GD_NARROW, GD_NARROW_OWN };
struct GdUnit { int8_t p, q, kind; };
struct GdRole { int8_t decodes, n; GdUnit u[6]; }; // column block whose codes the wave looks up (-1: none, NF: the narrow one), what it multiplies
constexpr int gd_sums(int kind) { return kind == GD_FULL ? 7 : kind == GD_HALF_A ? 3 : kind == GD_HALF_B ? 4 : kind == GD_NARROW_OWN ? 2 : 10; }
constexpr int gd_products(int kind) { return kind == GD_FULL ? 28 : kind == GD_OWN ? 16 : kind == GD_NARROW ? 10 : kind == GD_NARROW_OWN ? 2 : 14; }

// Sets of waves, each with 64 rows of a tile, and the roles of a set's waves. Waves w and w + 4 run on one SIMD; the roles give all four about as many
// products. A role reads at most three blocks (7 blocks' pairs are seven triangles, 6 blocks' four triangles and three pairs) and of the one it has looked up
// itself nothing, whose products with itself come first where it has them: there all waves read LDS. Blocks 3 and up, whose tables may not fit LDS, are looked
// up by waves whose sums leave them registers for that on their way.
constexpr int gd_sets(int nf) { return nf == 2 ? 4 : nf <= 4 ? 2 : 1; }
constexpr int gd_roles(int nf) { return 8 / gd_sets(nf); }
constexpr GdRole gd_role(int nf, int narrow, int role) {
	constexpr int F = GD_FULL, A = GD_HALF_A, B = GD_HALF_B, O = GD_OWN, N = GD_NARROW, NO = GD_NARROW_OWN;
	constexpr GdRole r2[2] = {{0, 2, {{0, 0, O}, {0, 1, A}}}, {1, 2, {{1, 1, O}, {0, 1, B}}}};
	constexpr GdRole r3[4] = {{0, 2, {{0, 0, O}, {0, 1, A}}}, {1, 2, {{1, 1, O}, {0, 1, B}}}, {-1, 2, {{0, 2, F}, {1, 2, A}}}, {2, 2, {{2, 2, O}, {1, 2, B}}}};
	constexpr GdRole n3[4] = {{0, 3, {{0, 0, O}, {0, 0, N}, {0, 1, A}}}, {1, 3, {{1, 1, O}, {1, 1, N}, {0, 1, B}}}, {3, 3, {{0, 2, F}, {0, 0, NO}, {1, 2, A}}},
		{2, 3, {{2, 2, O}, {2, 2, N}, {1, 2, B}}}};
	constexpr GdRole r4[4] = {{0, 3, {{0, 0, O}, {0, 1, F}, {0, 2, A}}}, {1, 3, {{1, 1, O}, {1, 2, F}, {1, 3, A}}}, {2, 3, {{2, 2, O}, {2, 3, F}, {0, 2, B}}},
		{3, 3, {{3, 3, O}, {0, 3, F}, {1, 3, B}}}};
	constexpr GdRole r5[8] = {{0, 3, {{0, 0, O}, {0, 1, F}, {0, 2, F}}}, {1, 3, {{1, 1, O}, {1, 3, F}, {1, 4, F}}}, {2, 3, {{2, 2, O}, {2, 3, F}, {2, 4, F}}},
		{-1, 2, {{0, 3, F}, {0, 4, F}}}, {-1, 1, {{1, 2, F}}}, {4, 1, {{4, 4, O}}}, {3, 1, {{3, 3, O}}}, {-1, 1, {{3, 4, F}}}};
	constexpr GdRole n5[8] = {r5[0], r5[1], r5[2], {-1, 3, {{0, 3, F}, {0, 0, N}, {0, 4, F}}}, {5, 2, {{0, 0, NO}, {1, 2, F}}}, {4, 3, {{4, 4, O}, {4, 4, N}, {1, 1, N}}},
		{3, 3, {{3, 3, O}, {3, 3, N}, {2, 2, N}}}, r5[7]};
	constexpr GdRole r6[8] = {{0, 4, {{0, 0, O}, {0, 1, F}, {0, 2, F}, {1, 2, F}}}, {1, 4, {{1, 1, O}, {1, 3, F}, {1, 5, F}, {3, 5, F}}},
		{4, 3, {{0, 4, F}, {4, 5, F}, {0, 5, F}}}, {2, 4, {{2, 2, O}, {2, 3, F}, {2, 4, F}, {3, 4, F}}}, {3, 1, {{0, 3, F}}}, {5, 1, {{2, 5, F}}},
		{-1, 2, {{4, 4, O}, {1, 4, F}}}, {-1, 2, {{3, 3, O}, {5, 5, O}}}};
	constexpr GdRole n6[8] = {r6[0], r6[1], r6[2], r6[3], {3, 2, {{3, 3, O}, {0, 3, F}}}, {5, 2, {{5, 5, O}, {2, 5, F}}},
		{6, 4, {{4, 4, O}, {4, 4, N}, {1, 4, F}, {1, 1, N}}}, {-1, 5, {{0, 0, NO}, {0, 0, N}, {2, 2, N}, {3, 3, N}, {5, 5, N}}}};
	constexpr GdRole r7[8] = {{3, 3, {{0, 3, F}, {3, 4, F}, {0, 4, F}}}, {5, 3, {{0, 5, F}, {5, 6, F}, {0, 6, F}}}, {4, 3, {{2, 4, F}, {4, 5, F}, {2, 5, F}}},
		{0, 4, {{0, 0, O}, {0, 1, F}, {0, 2, F}, {1, 2, F}}}, {1, 4, {{1, 1, O}, {1, 3, F}, {1, 5, F}, {3, 5, F}}}, {2, 4, {{2, 2, O}, {2, 3, F}, {2, 6, F}, {3, 6, F}}},
		{-1, 4, {{4, 4, O}, {1, 4, F}, {4, 6, F}, {1, 6, F}}}, {6, 3, {{6, 6, O}, {3, 3, O}, {5, 5, O}}}};
	return nf == 2 ? r2[role & 1] : nf == 3 ? (narrow ? n3 : r3)[role & 3] : nf == 4 ? r4[role & 3] : nf == 5 ? (narrow ? n5 : r5)[role] :
		nf == 6 ? (narrow ? n6 : r6)[role] : r7[role];
}
constexpr int gd_role_sums(const GdRole& R, int units) {
	int s = 0;
	for(int i = 0; i < units; i++) s += gd_sums(R.u[i].kind);
	return s;
}
constexpr int gd_role_products(const GdRole& R) {
	int s = 0;
	for(int i = 0; i < R.n; i++) s += gd_products(R.u[i].kind);
	return s;
}
// A unit's place among the sums of a set of waves: units are counted role by role
constexpr int gd_slot0(int nf, int narrow, int role) {
	int s = 0;
	for(int r = 0; r < role; r++) s += gd_role(nf, narrow, r).n;
	return s;
}
constexpr int gd_slots(int nf, int narrow) { return gd_slot0(nf, narrow, gd_roles(nf)); }
// the blocks a role reads, in the order of their first use; of the narrow block only whether
struct GdBlocks { int n; int b[8]; bool narrow; };
constexpr GdBlocks gd_blocks(const GdRole& R) {
	GdBlocks B{0, {0, 0, 0, 0, 0, 0, 0, 0}, false};
	for(int i = 0; i < R.n; i++) {
		B.narrow |= R.u[i].kind >= GD_NARROW;
		for(int e = 0; e < 2 && R.u[i].kind != GD_NARROW_OWN; e++) {
			const int b = e == 0 ? R.u[i].p : R.u[i].q;
			bool seen = false;
			for(int k = 0; k < B.n; k++) seen |= B.b[k] == b;
			if(!seen) B.b[B.n++] = b;
		}
	}
	return B;
}
constexpr int gd_place(const GdBlocks& B, int b) {
	for(int k = 0; k < B.n; k++)
		if(B.b[k] == b) return k;
	return 0;
}
constexpr int GD_SURE = 3; // column blocks whose tables fit LDS whatever their size (49 KB of digits, 32 KB of tables each)

// four rows' 4 bytes each -> the four bytes' rows
__device__ __forceinline__ void gd_transpose(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t (&o)[4]) {
	const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u), ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
	const uint32_t cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u), cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
	o[0] = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
	o[1] = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
	o[2] = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
	o[3] = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
}

// MODE of a wave's decoding: 0 none, 1 tables in LDS, 2 in global memory, 3 the narrow block (tables in LDS)
template <int NF, int NARROW, int ROLE, int MODE>
__device__ __forceinline__ void gd_loop(const GdArgs& A, uint8_t* smem, int t0, int t1) {
	constexpr int KT = gd_sets(NF), R = 64 * KT, CHUNK = GD_CHUNK / R;
	constexpr GdRole ROLES = gd_role(NF, NARROW, ROLE);
	constexpr GdBlocks BLOCKS = gd_blocks(ROLES);
	constexpr int NSUM = gd_role_sums(ROLES, ROLES.n), NX = BLOCKS.n > 0 ? BLOCKS.n : 1, CB = ROLES.decodes < 0 ? 0 : ROLES.decodes;
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int c = lane & 15, k = lane >> 4;
	const int set = wave / (8 / KT); // 64 rows of the tile
	const GdCol C = A.cols[CB * 16 + (MODE == 3 ? c & 3 : c)];
	const uint8_t* stream = A.arena + (size_t) C.stream * A.arenaStride + set * 64 + 16 * k;
	constexpr int TILE = (NF * GD_DIGITS + 2 * NARROW) * KT * 1024;
	const uint32_t ldsTab = (uint32_t) TILE + C.tab;
	i32x4_gd* const put = (i32x4_gd*) (smem + (CB * GD_DIGITS * KT + set) * 1024 + lane * 16); // (narrow: lane (k, column), digit d four places on)
	const i32x4_gd* const get = (const i32x4_gd*) (smem + set * 1024 + lane * 16);

	i32x4_gd acc[NSUM];
#pragma unroll
	for(int i = 0; i < NSUM; i++) acc[i] = i32x4_gd{0, 0, 0, 0};

	u32x4 codes, codesNext;
	u32x2 raw[16];
	i32x4_gd digits[GD_DIGITS];
	auto load_codes = [&](int tile) {
		if constexpr(MODE != 0) codesNext = *(const u32x4*) (stream + (int64_t) min(tile, t1 - 1) * R);
	};
	auto look_one = [&](int t) {
		const uint32_t code = (codes[t >> 2] >> (8 * (t & 3))) & 0xffu;
		if constexpr(MODE == 2) raw[t] = *(const u32x2*) (A.tabs + (uint32_t) (C.tab + (code << 3)));
		else raw[t] = *(const u32x2*) (smem + ldsTab + (code << 3));
	};
	auto look = [&]() {
		if constexpr(MODE != 0) {
#pragma unroll
			for(int t = 0; t < 16; t++) look_one(t);
		}
	};
	auto turn = [&](int tile) { // rows' digits -> digits' rows
		if constexpr(MODE != 0) {
			if((int64_t) (tile + 1) * R > A.nRows) { // zeros behind the last row of the matrix
				const int64_t row = (int64_t) tile * R + set * 64 + 16 * k;
#pragma unroll
				for(int t = 0; t < 16; t++) raw[t] = row + t < A.nRows ? raw[t] : u32x2{0, 0};
			}
#pragma unroll
			for(int g = 0; g < 4; g++) {
				uint32_t o[4];
				gd_transpose(raw[4 * g].x, raw[4 * g + 1].x, raw[4 * g + 2].x, raw[4 * g + 3].x, o);
#pragma unroll
				for(int d = 0; d < 4; d++) digits[d][g] = (int) o[d];
				gd_transpose(raw[4 * g].y, raw[4 * g + 1].y, raw[4 * g + 2].y, raw[4 * g + 3].y, o);
#pragma unroll
				for(int d = 4; d < GD_DIGITS; d++) digits[d][g] = (int) o[d - 4];
			}
		}
	};
	auto write = [&]() {
		if constexpr(MODE == 3) {
			if(c < 4) {
#pragma unroll
				for(int d = 0; d < GD_DIGITS; d++) put[(d >> 2) * KT * 64 + (d & 3) * 4] = digits[d];
			}
		}
		else if constexpr(MODE != 0) {
#pragma unroll
			for(int d = 0; d < GD_DIGITS; d++) put[d * KT * 64] = digits[d];
		}
	};
	// Multiplies a tile; on the way the next tile's digits, in front of the last unit. Tables in LDS: its lookups a unit before. In global memory: spread between the
	// products from the last unit of the tile before on, as the vector memory path needs most of a tile's time for them and holds up a wave that brings all at once.
	constexpr int NM = gd_role_products(ROLES), LAST = gd_products(ROLES.u[ROLES.n - 1].kind);
	constexpr auto wanted = [](int products) { return products * 18 / NM < 16 ? products * 18 / NM : 16; }; // behind so many since they began
	auto multiply = [&](int tile) {
		i32x4_gd x[NX][GD_DIGITS], nx[2];
		int at = 0, done = wanted(LAST), have = 0;
		auto need = [&](int slot) { // (slots come in order)
			if(slot < have || slot >= BLOCKS.n) return;
			have++;
#pragma unroll
			for(int d = 0; d < GD_DIGITS; d++) x[slot][d] = (MODE == 1 || MODE == 2) && BLOCKS.b[slot] == CB ? digits[d] : get[(BLOCKS.b[slot] * GD_DIGITS + d) * KT * 64];
		};
		auto product = [&](int s, i32x4_gd a, i32x4_gd b) {
			acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, acc[s], 0, 0, 0);
			at++;
			const int since = at > NM - LAST ? at - (NM - LAST) : at + LAST;
			if(MODE == 2 && done < wanted(since)) {
				__builtin_amdgcn_sched_barrier(0);
				look_one(done++);
				__builtin_amdgcn_sched_barrier(0);
			}
		};
		need(0);
		need(1);
		if constexpr(BLOCKS.narrow) {
			nx[0] = get[NF * GD_DIGITS * KT * 64];
			nx[1] = get[(NF * GD_DIGITS + 1) * KT * 64];
		}
#pragma unroll
		for(int i = 0; i < ROLES.n; i++) {
			const int sp = gd_place(BLOCKS, ROLES.u[i].p), sq = gd_place(BLOCKS, ROLES.u[i].q), kind = ROLES.u[i].kind, a0 = gd_role_sums(ROLES, i);
			if(kind != GD_NARROW_OWN) {
				need(min(sp, sq));
				need(max(sp, sq));
				if(MODE == 2) need(max(sp, sq) + 1);
			}
			if((MODE == 1 || MODE == 3) && i == (ROLES.n > 1 ? ROLES.n - 2 : 0)) look();
			if(MODE != 0 && i == ROLES.n - 1) {
				if(MODE == 2) {
#pragma unroll
					for(; done < 16; done++) look_one(done);
					done = 0;
				}
				turn(min(tile + 1, t1 - 1));
				codes = codesNext;
				load_codes(tile + 3);
			}
			if(kind == GD_NARROW_OWN) {
				product(a0, nx[0], nx[0]);
				product(a0 + 1, nx[0], nx[1]);
				continue;
			}
			if(kind == GD_NARROW) {
#pragma unroll
				for(int d = 0; d < GD_DIGITS; d++) {
					product(a0 + d, nx[0], x[sp][d]);
					if(d < 3) product(a0 + GD_DIGITS + d, nx[1], x[sp][d]);
				}
				continue;
			}
#pragma unroll
			for(int da = 0; da < GD_DIGITS; da++)
#pragma unroll
				for(int db = 0; da + db < GD_DIGITS; db++) {
					const int w = da + db;
					int s = -1;
					if(kind == GD_FULL) s = w;
					else if(kind == GD_HALF_A) s = w == 0 ? 0 : w >= 5 ? w - 4 : -1;
					else if(kind == GD_HALF_B) s = w >= 1 && w <= 4 ? w - 1 : -1;
					else s = da == db ? 6 + da : da < db ? w - 1 : -1;
					if(s >= 0) product(a0 + s, x[sp][da], x[sq][db]);
				}
		}
	};
	// The weights' sums joined. Into this workgroup's part of the workspace; where several sets of waves have sums of the same cells, on the way
	// into a part of the set's own, the last time into LDS, which nobody reads any more, where k_gram_tiles_i8 adds the sets up.
	constexpr int SLOTS = gd_slots(NF, NARROW), SLOT0 = gd_slot0(NF, NARROW, ROLE);
	double* const part = KT == 1 ? A.parts + ((size_t) blockIdx.x * SLOTS + SLOT0) * 256 : A.setParts + ((size_t) (blockIdx.x * KT + set) * SLOTS + SLOT0) * 256;
	double* const ldsPart = (double*) smem + (set * SLOTS + SLOT0) * 256;
	auto join = [&](bool more, bool last) {
		constexpr double S = 1.0 / 256.0, S4 = S * S * S * S;
#pragma unroll
		for(int u = 0; u < ROLES.n; u++) {
			const int kind = ROLES.u[u].kind, a0 = gd_role_sums(ROLES, u);
			double* const to = part + u * 256;
			auto give = [&](int at, double v) {
				if(more) v += to[at];
				if(KT > 1 && last) ldsPart[u * 256 + at] = v;
				else to[at] = v;
			};
			double m[4][2];
#pragma unroll
			for(int i = 0; i < 4; i++) {
				const int r = 4 * k + i;
				auto at = [&](int s) { return (double) acc[a0 + s][i]; };
				if(kind == GD_FULL) give(r * 16 + c, (((((at(6) * S + at(5)) * S + at(4)) * S + at(3)) * S + at(2)) * S + at(1)) * S + at(0));
				else if(kind == GD_HALF_A) give(r * 16 + c, (at(2) * S + at(1)) * (S4 * S) + at(0));
				else if(kind == GD_HALF_B) give(r * 16 + c, (((at(3) * S + at(2)) * S + at(1)) * S + at(0)) * S);
				else if(kind == GD_OWN) {
					const double off = (((((at(5) * S + at(4)) * S + at(3)) * S + at(2)) * S + at(1)) * S + at(0)) * S;
					const double own = ((at(9) * (S * S) + at(8)) * (S * S) + at(7)) * (S * S) + at(6);
					give(r * 16 + c, (r == c ? 2.0 * off : off) + (r <= c ? own : 0.0));
				}
				else { // lane (k, c), place i: digit k (second operand 4 + k) of narrow column i
					const double wk = k == 0 ? 1.0 : k == 1 ? S : k == 2 ? S * S : S * S * S;
					if(kind == GD_NARROW) {
						m[i][0] = (((((at(6) * S + at(5)) * S + at(4)) * S + at(3)) * S + at(2)) * S + at(1)) * S + at(0);
						m[i][0] = (((at(9) * S + at(8)) * S + at(7)) * S4 + m[i][0]) * wk;
						m[i][0] += __shfl_xor(m[i][0], 16, WAVE);
						m[i][0] += __shfl_xor(m[i][0], 32, WAVE);
						if(k == 0) give(i * 16 + c, m[i][0]);
					}
					else { // ... times digit c / 4 (4 + c / 4) of narrow column c % 4
						const double wc = c < 4 ? 1.0 : c < 8 ? S : c < 12 ? S * S : S * S * S;
#pragma unroll
						for(int h = 0; h < 2; h++) {
							m[i][h] = at(h) * (h ? wk * wc * S4 : wk * wc);
#pragma unroll
							for(int d = 4; d < WAVE; d *= 2) m[i][h] += __shfl_xor(m[i][h], d, WAVE);
							if(lane < 4) give(h * 16 + i * 4 + lane, m[i][h]);
						}
					}
				}
				__builtin_amdgcn_sched_barrier(0); // (a few at a time: the sums fill the registers)
			}
		}
#pragma unroll
		for(int i = 0; i < NSUM; i++) acc[i] = i32x4_gd{0, 0, 0, 0};
	};

	load_codes(t0);
	{
		// the tables, 8 pieces of 16 bytes per thread requested together
		const u32x4* src = (const u32x4*) A.tabs;
		u32x4* dst = (u32x4*) (smem + TILE);
		const int n = A.ldsTab / 16;
		for(int i0 = tid; i0 < n; i0 += 8 * GD_THREADS) {
			u32x4 d[8];
#pragma unroll
			for(int j = 0; j < 8; j++) d[j] = src[min(i0 + j * GD_THREADS, n - 1)];
#pragma unroll
			for(int j = 0; j < 8; j++)
				if(i0 + j * GD_THREADS < n) dst[i0 + j * GD_THREADS] = d[j];
		}
		// (the narrow block's second operand has digits 4 - 6 only)
		if(NARROW && tid < KT * 64) ((i32x4_gd*) (smem + (NF * GD_DIGITS + 1) * KT * 1024))[tid] = i32x4_gd{0, 0, 0, 0};
	}
	lds_barrier();
	codes = codesNext;
	load_codes(t0 + 1);
	look();
	turn(t0);
	write();
	codes = codesNext;
	load_codes(t0 + 2);
	if constexpr(MODE == 2) {
#pragma unroll
		for(int t = 0; t < wanted(LAST); t++) look_one(t);
	}
	lds_barrier();
	for(int first = t0; first < t1; first += CHUNK) {
		const int behind = min(first + CHUNK, t1);
		for(int tile = first; tile < behind; tile++) {
			multiply(tile);
			lds_barrier();
			write();
			lds_barrier();
		}
		join(first > t0, behind == t1);
	}
}

template <int NF, int NARROW>
__global__ __launch_bounds__(GD_THREADS, 2) void k_gram_tiles_i8(GdArgs A) {
	extern __shared__ __attribute__((aligned(16))) uint8_t gd_smem[]; // the tile's digits, the tables
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int t0 = (int) ((int64_t) A.nTiles * blockIdx.x / gridDim.x), t1 = (int) ((int64_t) A.nTiles * (blockIdx.x + 1) / gridDim.x);
	if(A.nnz != nullptr && blockIdx.x == 0) nnz_clear(A.nnz); // (k_gram_join counts)
	// (three column blocks: the second set's waves take the roles the other way round, so that the SIMDs share the longer ones)
	const int role = NF == 3 ? (wave + (wave >> 2) * 2) & 3 : wave % gd_roles(NF);
	auto run = [&](auto roleTag) {
		constexpr int ROLE = decltype(roleTag)::value, D = gd_role(NF, NARROW, ROLE).decodes;
		if constexpr(D < 0) gd_loop<NF, NARROW, ROLE, 0>(A, gd_smem, t0, t1);
		else if constexpr(D == NF) gd_loop<NF, NARROW, ROLE, 3>(A, gd_smem, t0, t1);
		else if constexpr(D < GD_SURE) gd_loop<NF, NARROW, ROLE, 1>(A, gd_smem, t0, t1);
		else if(D < A.nLds) gd_loop<NF, NARROW, ROLE, 1>(A, gd_smem, t0, t1);
		else gd_loop<NF, NARROW, ROLE, 2>(A, gd_smem, t0, t1);
	};
	using std::integral_constant;
	if(role == 0) run(integral_constant<int, 0>());
	else if(role == 1) run(integral_constant<int, 1>());
	if constexpr(gd_roles(NF) >= 4) {
		if(role == 2) run(integral_constant<int, 2>());
		else if(role == 3) run(integral_constant<int, 3>());
	}
	if constexpr(gd_roles(NF) == 8) {
		if(role == 4) run(integral_constant<int, 4>());
		else if(role == 5) run(integral_constant<int, 5>());
		else if(role == 6) run(integral_constant<int, 6>());
		else if(role == 7) run(integral_constant<int, 7>());
	}
	constexpr int KT = gd_sets(NF), SUMS = gd_slots(NF, NARROW) * 256;
	if constexpr(KT > 1) {
		__syncthreads();
		const double* from = (const double*) gd_smem;
		for(int i = threadIdx.x; i < SUMS; i += GD_THREADS) {
			double v = from[i];
#pragma unroll
			for(int t = 1; t < KT; t++) v += from[t * SUMS + i];
			A.parts[(size_t) blockIdx.x * SUMS + i] = v;
		}
	}
}

// ---- the workgroups' sums

// 256 cells of the result: two column blocks (p < q: one unit or the two halves of one), one with itself (p = q < NF), the narrow one with block p, with itself
struct GdTile { int16_t p, q, a, b; }; // a, b: units' slots (b = -1: one unit)

constexpr int GJ_THREADS = 1024, GJ_CELLS = 16, GJ_SLICES = GJ_THREADS / GJ_CELLS;
// The parts of all workgroups added up: into out, both triangles, non-zeros counted. A block takes 16 cells of a tile, every 64th of
// the parts per group of 16 threads. Bound: round trips past the XCDs' caches, of which a CU has only so many on their way, so the cells go to
// many blocks. (As atomic adds of every workgroup into an accumulator per XCD, whose last workgroups joined those, the sums of 10,007 x 100 took 14 us longer.)
__global__ __launch_bounds__(GJ_THREADS) void k_gram_join(const GdTile* __restrict__ tiles, const GdCol* __restrict__ cols, int nf, const double* __restrict__ parts,
	int nParts, int slots, double* acc, int skipOwn, int clearAcc, double* out, int nCols, unsigned long long* __restrict__ nnz) {
	constexpr int WAVES = GJ_THREADS / WAVE, PER = 256 / GJ_CELLS;
	__shared__ double sums[WAVES][GJ_CELLS], lows[WAVES][GJ_CELLS];
	const GdTile T = tiles[blockIdx.x / PER];
	const int tid = threadIdx.x, cell = tid % GJ_CELLS, e = blockIdx.x % PER * GJ_CELLS + cell, slice = tid / GJ_CELLS;
	int i = T.p * 16 + (e >> 4), j = T.q * 16 + (e & 15); // columns in the kernel's order, i <= j
	int o0 = T.a * 256 + e, o1 = -1, o2 = -1;
	bool real = true;
	if(T.q < nf) {
		if(T.p == T.q) {
			real = i <= j;
			if(i < j) o1 = T.a * 256 + (e & 15) * 16 + (e >> 4);
		}
		else if(T.b >= 0) o1 = T.b * 256 + e;
	}
	else if(T.p < nf) { // place narrow column * 16 + column of block p
		real = e < 64;
		j = nf * 16 + (e >> 4);
		i = T.p * 16 + (e & 15);
	}
	else {
		const int a = (e >> 2) & 3, b = e & 3;
		real = e < 16 && a <= b;
		i = nf * 16 + a; j = nf * 16 + b;
		o1 = T.a * 256 + 16 + a * 4 + b; o2 = T.a * 256 + 16 + b * 4 + a;
	}
	// (with what each addition rounds off kept beside the sum: the parts are sums of many rows each, and there are up to 1024 of them)
	double s = 0.0, low = 0.0;
	auto add = [&](double v) {
		const double t = s + v, w = t - s;
		low += (s - (t - w)) + (v - w);
		s = t;
	};
	if(real) {
		const size_t step = (size_t) slots * 256;
		const double* p = parts + slice * step;
#pragma unroll 4
		for(int n = slice; n < nParts; n += GJ_SLICES, p += GJ_SLICES * step) {
			const double v0 = p[o0], v1 = o1 >= 0 ? p[o1] : 0.0, v2 = o2 >= 0 ? p[o2] : 0.0;
			add(v0);
			add(v1);
			add(v2);
		}
	}
#pragma unroll
	for(int d = GJ_CELLS; d < WAVE; d *= 2) {
		const double so = __shfl_xor(s, d, WAVE), lo = __shfl_xor(low, d, WAVE);
		low += lo;
		add(so);
	}
	if((tid & (WAVE - 1)) < GJ_CELLS) {
		sums[tid / WAVE][cell] = s;
		lows[tid / WAVE][cell] = low;
	}
	__syncthreads();
	int cnt = 0;
	if(tid < GJ_CELLS && real) {
#pragma unroll
		for(int n = 1; n < WAVES; n++) {
			low += lows[n][cell];
			add(sums[n][cell]);
		}
		s += low;
		const GdCol a = cols[i], b = cols[j];
		if(a.col >= 0 && b.col >= 0) {
			const size_t up = (size_t) min(a.col, b.col) * nCols + max(a.col, b.col), down = (size_t) max(a.col, b.col) * nCols + min(a.col, b.col);
			s = s * a.scale * b.scale;
			if(skipOwn && (a.group == b.group || a.group < 0 || b.group < 0)) { // from the code counts
				s = acc[up];
				if(clearAcc) acc[up] = 0.0;
			}
			out[up] = s;
			out[down] = s;
			cnt = s != 0.0 ? (i == j ? 1 : 2) : 0;
		}
	}
	if(nnz != nullptr) count_add(nnz, cnt);
}

// ---- which blocks

// For pairs of column blocks p <= q: left += the sums over the rows of the digit products of weight 7, the largest that the kernel above leaves out (the rounding of the
// values is among them, as an eighth digit), mags += those of the products of the magnitudes (of the first digits, 1 / GD_MAG of the largest value). 16 NCB cells a
// row of either. A workgroup takes a pair of column blocks, a wave 64 rows at a time. (Once per block: 2,000,003 x 100 1.3 ms, and where gd_compare needs it a call of either kernel.)
constexpr int GC_UNITS = 240; // 64 rows each, between two flushes: a sum grows by at most 8 2^14 a row
constexpr int GC_TAB = 16 * 256 * 8, GC_LDS = 2 * GC_TAB;
__global__ __launch_bounds__(GD_THREADS, 2) void k_gram_left(const uint8_t* __restrict__ arena, size_t arenaStride, const GdCol* __restrict__ cols, int places, int ncb,
	const uint8_t* __restrict__ digitTabs, int64_t nRows, unsigned long long* __restrict__ left, unsigned long long* __restrict__ mags) {
	extern __shared__ __attribute__((aligned(16))) uint8_t gd_smem[]; // digits of block p, of q
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, k = lane >> 4;
	int p = 0, q = blockIdx.y;
	while(q >= ncb - p) { q -= ncb - p; p++; }
	q += p;
	for(int i = tid; i < 2 * GC_TAB / 16; i += GD_THREADS) {
		const int side = i / (GC_TAB / 16);
		((u32x4*) gd_smem)[i] = ((const u32x4*) (digitTabs + (size_t) (side ? q : p) * GC_TAB))[i % (GC_TAB / 16)];
	}
	__syncthreads();
	i32x4_gd l{0, 0, 0, 0}, m{0, 0, 0, 0};
	auto flush = [&]() {
#pragma unroll
		for(int i = 0; i < 4; i++) {
			const size_t at = (size_t) (16 * p + 4 * k + i) * (16 * ncb) + 16 * q + c;
			atomicAdd(&left[at], (unsigned long long) (int64_t) l[i]);
			atomicAdd(&mags[at], (unsigned long long) (int64_t) m[i]);
		}
		l = m = i32x4_gd{0, 0, 0, 0};
	};
	const int64_t nUnits = (nRows + 63) / 64;
	int since = 0;
	for(int64_t u = (int64_t) blockIdx.x * 8 + wave; u < nUnits; u += (int64_t) gridDim.x * 8) {
		const int64_t row = u * 64 + 16 * k;
		i32x4_gd x[2][8], xm[2];
#pragma unroll
		for(int side = 0; side < 2; side++) {
			const u32x4 codes = *(const u32x4*) (arena + (size_t) cols[min((side ? q : p) * 16 + c, places - 1)].stream * arenaStride + row); // (behind them: zeros, whatever the code)
			const uint8_t* const digits = gd_smem + side * GC_TAB + c * 2048;
#pragma unroll
			for(int g = 0; g < 4; g++) {
				u32x2 raw[4];
#pragma unroll
				for(int t = 0; t < 4; t++) raw[t] = *(const u32x2*) (digits + (((codes[g] >> (8 * t)) & 0xffu) << 3));
				if((u + 1) * 64 > nRows) {
#pragma unroll
					for(int t = 0; t < 4; t++) raw[t] = row + 4 * g + t < nRows ? raw[t] : u32x2{0, 0};
				}
				uint32_t o[4];
				gd_transpose(raw[0].x, raw[1].x, raw[2].x, raw[3].x, o);
#pragma unroll
				for(int d = 0; d < 4; d++) x[side][d][g] = (int) o[d];
				const uint32_t sign = (o[0] >> 7) & 0x01010101u;
				xm[side][g] = (int) ((o[0] ^ (sign * 255u)) + sign); // the first digit's magnitude, byte by byte (at most 127)
				gd_transpose(raw[0].y, raw[1].y, raw[2].y, raw[3].y, o);
#pragma unroll
				for(int d = 0; d < 4; d++) x[side][4 + d][g] = (int) o[d];
			}
		}
#pragma unroll
		for(int i = 0; i < 8; i++) l = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[0][i], x[1][7 - i], l, 0, 0, 0);
		m = __builtin_amdgcn_mfma_i32_16x16x64_i8(xm[0], xm[1], m, 0, 0, 0);
		if(++since == GC_UNITS) {
			flush();
			since = 0;
		}
	}
	if(since > 0) flush();
}

struct GdPlan {
	int rc = 0;       // 1: not of this kernel's shape, or its errors would not suit the block
	GdArgs A;
	void* dImg = nullptr;
	int64_t bytes = 0;
	int nf = 0, narrow = 0;
	const GdTile* tiles = nullptr;
	int nCellTiles = 0, grid = 0;
	size_t lds = 0;
	// Until the results have been compared: per column its place's group and column, per cell i <= j what is left out and the terms' magnitudes (NaN: exact or zero)
	std::vector<GdCol> cols;
	std::vector<double> left, mags;
	bool compared = false;
	bool suits[2] = {false, false}; // all cells / those across groups: no further from the exact sums than the fp64 kernel's
	~GdPlan() { if(dImg) (void) hipFree(dImg); }
};

void gd_plan_drop(cla_block* b) {
	if(b->gdPlan == nullptr) return;
	b->derivedBytes -= b->gdPlan->bytes;
	delete b->gdPlan;
	b->gdPlan = nullptr;
}

// The digits of x 2^GD_BITS rounded to a whole number, and of what that lost; true if nothing was rounded
static bool gd_digits(double x, int8_t (&d)[GD_DIGITS + 1]) {
	const double scaled = x * (double) ((int64_t) 1 << GD_BITS), whole = std::nearbyint(scaled);
	int64_t X = (int64_t) whole;
	for(int i = GD_DIGITS - 1; i > 0; i--) {
		d[i] = (int8_t) (uint8_t) (X & 255);
		X = (X - d[i]) >> 8;
	}
	d[0] = (int8_t) X;
	d[GD_DIGITS] = (int8_t) std::min(127.0, std::nearbyint((scaled - whole) * 256.0));
	return whole == scaled;
}

// 1: no room on the device for the plan
static int gd_build_plan(cla_block* b, GdPlan& P) {
	P.rc = 1;
	const int n = b->nCols;
	if(b->dArena == nullptr || b->arenaWidth != 1 || n < 17 || n > 112 || b->nRows == 0 || b->dictNonFinite || b->crossSplit > 0 || b->crossBlocks > 0) return 0;
	if(b->nRows > (int64_t) 131072 * 8 * 64) return 0; // (longer ones have not been measured)
	std::vector<int> groupOf((size_t) n, -1);
	for(size_t g = 0; g < b->groups.size(); g++)
		for(int col : b->groups[g].cols) {
			if(groupOf[col] >= 0) return 0; // overlapping groups
			groupOf[col] = (int) g;
		}
	// a last block of at most 4 columns is a narrow one where a wave is free to decode it
	const int ncb = (n + 15) / 16, narrow = n % 16 >= 1 && n % 16 <= 4 && (n / 16 == 3 || n / 16 >= 5) ? 1 : 0, nf = narrow ? n / 16 : ncb;
	P.nf = nf; P.narrow = narrow;
	const int places = narrow ? nf * 16 + 4 : nf * 16;
	std::vector<GdCol> cols((size_t) places);
	std::vector<uint8_t> tabs;
	std::vector<uint8_t> digitTabs((size_t) ncb * GC_TAB, 0);
	std::vector<char> exact((size_t) n), zero((size_t) n); // few digits and nothing rounded; only zeros
	struct Src { int col, group, h; };
	std::vector<Src> src; // columns in the groups' order, then those that only carry a constant
	for(size_t g = 0; g < b->groups.size(); g++)
		for(int h = 0; h < b->groups[g].d.nColG; h++) src.push_back(Src{b->groups[g].cols[h], (int) g, h});
	for(int col = 0; col < n; col++)
		if(groupOf[col] < 0) src.push_back(Src{col, -1, 0});
	if((int) src.size() != n) return 0;
	auto add_column = [&](int place) {
		const Src from = src[place];
		const HostGroup* H = from.group >= 0 ? &b->groups[from.group] : nullptr;
		const int nc = H ? H->d.nColG : 1, nV = H ? H->d.nVals : 1, entries = H ? nV : 256; // (without a group: any code of stream 0 will do)
		std::vector<double> val((size_t) nV);
		double most = 0.0;
		for(int i = 0; i < nV; i++) {
			val[i] = (H ? H->dict[(size_t) i * nc + from.h] : 0.0) + b->constV[from.col];
			most = std::isfinite(val[i]) ? std::max(most, std::fabs(val[i])) : INFINITY;
		}
		int e = 0;
		if(most > 0.0 && std::isfinite(most) && std::frexp(most, &e) >= 0.99) e++;
		if(!std::isfinite(most) || e < -300 || e > 300) return false; // (sums of products stay far from the ends of fp64's range)
		const double down = std::ldexp(1.0, -e);
		GdCol& C = cols[place];
		C.tab = (uint32_t) tabs.size(); C.stream = std::max(from.group, 0); C.group = from.group; C.col = from.col; C.scale = std::ldexp(1.0, e - 7);
		tabs.resize(tabs.size() + (size_t) entries * 8, 0);
		bool ex = true;
		for(int i = 0; i < entries; i++) {
			const double x = val[std::min(i, nV - 1)] * down; // (exact: what is lost of values 2^-700 of the largest is below every digit)
			int8_t d[GD_DIGITS + 1];
			ex &= gd_digits(x, d) && d[4] == 0 && d[5] == 0 && d[6] == 0;
			std::memcpy(tabs.data() + C.tab + (size_t) i * 8, d, GD_DIGITS);
			std::memcpy(digitTabs.data() + ((size_t) place * 256 + i) * 8, d, GD_DIGITS + 1);
		}
		exact[place] = ex; zero[place] = most == 0.0;
		return true;
	};
	// tables: the narrow block's, then block by block
	uint32_t padTab = 0;
	if(n < places) { // padding: zeros
		padTab = (uint32_t) tabs.size();
		tabs.resize(tabs.size() + 256 * 8, 0);
	}
	for(int place = n; place < places; place++) {
		GdCol& pad = cols[place];
		pad.tab = padTab; pad.stream = 0; pad.group = -1; pad.col = -1; pad.scale = 0.0;
	}
	for(int place = nf * 16; place < n; place++)
		if(!add_column(place)) return 0;
	std::vector<size_t> end; // of the tables up to each block
	for(int p = 0; p < nf; p++) {
		for(int place = p * 16; place < std::min(n, p * 16 + 16); place++)
			if(!add_column(place)) return 0;
		end.push_back((tabs.size() + 15) & ~(size_t) 15);
	}
	tabs.resize((tabs.size() + 15) & ~(size_t) 15, 0);
	// column blocks whose tables fit LDS beside the tile
	const size_t tileBytes = (size_t) (nf * GD_DIGITS + 2 * narrow) * gd_sets(nf) * 1024;
	int nLds = 0;
	while(nLds < nf && tileBytes + end[nLds] <= (size_t) g_ldsPerBlock) nLds++;
	if(nLds < std::min(nf, GD_SURE)) return 0;
	const size_t ldsTab = end[nLds - 1];
	P.lds = std::max(tileBytes + ldsTab, gd_sets(nf) > 1 ? (size_t) gd_sets(nf) * gd_slots(nf, narrow) * 256 * 8 : 0); // (the sets' sums, at the end)

	std::vector<GdTile> tiles;
	for(int p = 0; p < nf + narrow; p++)
		for(int q = p; q < nf + narrow; q++) tiles.push_back(GdTile{(int16_t) p, (int16_t) q, -1, -1});
	for(int r = 0, slot = 0; r < gd_roles(nf); r++) {
		const GdRole R = gd_role(nf, narrow, r);
		for(int u = 0; u < R.n; u++, slot++)
			for(GdTile& t : tiles) {
				const int kind = R.u[u].kind;
				if(t.p != (kind == GD_NARROW_OWN ? nf : R.u[u].p) || t.q != (kind >= GD_NARROW ? nf : R.u[u].q)) continue;
				(t.a < 0 ? t.a : t.b) = (int16_t) slot;
			}
	}

	const int rows = 64 * gd_sets(nf);
	GdArgs& A = P.A;
	A.nTiles = (int) ((b->nRows + rows - 1) / rows);
	P.grid = std::min(A.nTiles, g_numCU);
	P.nCellTiles = (int) tiles.size();
	const size_t colBytes = cols.size() * sizeof(GdCol), nMag = (size_t) ncb * 16 * ncb * 16;
	const size_t oTiles = (colBytes + 255) & ~(size_t) 255, oTabs = (oTiles + tiles.size() * sizeof(GdTile) + 255) & ~(size_t) 255;
	const size_t oParts = (oTabs + tabs.size() + 255) & ~(size_t) 255, partBytes = (size_t) P.grid * gd_slots(nf, narrow) * 256 * 8;
	const bool chunks = gd_sets(nf) > 1 && (A.nTiles + P.grid - 1) / P.grid > GD_CHUNK / rows; // sums of a set on their way
	std::vector<uint8_t> all(oTabs + tabs.size(), 0);
	std::memcpy(all.data(), cols.data(), colBytes);
	std::memcpy(all.data() + oTiles, tiles.data(), tiles.size() * sizeof(GdTile));
	std::memcpy(all.data() + oTabs, tabs.data(), tabs.size());
	uint8_t* d = nullptr;
	if(no_room((void**) &d, oParts + partBytes * (chunks ? 1 + gd_sets(nf) : 1))) return 1;
	P.dImg = d;
	P.bytes = (int64_t) (oParts + partBytes * (chunks ? 1 + gd_sets(nf) : 1));
	CLA_HIP(hipMemcpy(d, all.data(), all.size(), hipMemcpyHostToDevice));
	A.arena = b->dArena; A.arenaStride = b->arenaStride;
	A.cols = (const GdCol*) d; A.tabs = d + oTabs;
	A.parts = (double*) (d + oParts); A.setParts = chunks ? (double*) (d + oParts + partBytes) : nullptr;
	P.tiles = (const GdTile*) (d + oTiles);
	A.nRows = b->nRows;
	A.nLds = nLds; A.ldsTab = (int) ldsTab;

	// The errors are parts of the columns' largest values, a cell's terms need not be: every cell whose columns are not both free of
	// rounding has to reach, on average over the rows, 2^-10 of the product of their largest values, whoever asks.
	// (Six products left out of up to 2^14 2^-70 and two roundings of up to 2^-56: 2^-53.0 a row, all of one sign where a tuple has nearly all rows: up to 2^-43 of the
	// terms' sum. Unasked a block comes here only if gd_compare finds less than in fp64.)
	struct Tmp { void* p = nullptr; ~Tmp() { if(p) (void) hipFree(p); } } tmp;
	const size_t sumBytes = nMag * sizeof(unsigned long long);
	if(no_room(&tmp.p, 2 * sumBytes + digitTabs.size())) return 1;
	unsigned long long* const dLeft = (unsigned long long*) tmp.p;
	uint8_t* const dDigits = (uint8_t*) tmp.p + 2 * sumBytes;
	CLA_HIP(hipMemsetAsync(dLeft, 0, 2 * sumBytes, b->stream));
	CLA_HIP(hipMemcpyAsync(dDigits, digitTabs.data(), digitTabs.size(), hipMemcpyHostToDevice, b->stream));
	const int pairs = ncb * (ncb + 1) / 2;
	const unsigned gx = (unsigned) std::min<int64_t>((b->nRows + 511) / 512, (2 * g_numCU + pairs - 1) / pairs);
	CLA_HIP(allow_full_lds((const void*) k_gram_left));
	hipLaunchKernelGGL(k_gram_left, dim3(gx, (unsigned) pairs), dim3(GD_THREADS), GC_LDS, b->stream, A.arena, A.arenaStride, A.cols, places, ncb, dDigits, A.nRows,
		dLeft, dLeft + nMag);
	CLA_HIP(hipGetLastError());
	std::vector<unsigned long long> sums(2 * nMag);
	CLA_HIP(hipMemcpyAsync(sums.data(), dLeft, 2 * sumBytes, hipMemcpyDeviceToHost, b->stream));
	CLA_HIP(hipStreamSynchronize(b->stream));
	P.cols = std::move(cols);
	P.left.assign((size_t) n * n, NAN);
	P.mags.assign((size_t) n * n, NAN);
	const double least = (double) b->nRows * GD_MAG * GD_MAG / 1024.0;
	for(int i = 0; i < n; i++)
		for(int j = i; j < n; j++) {
			if(zero[i] || zero[j] || (exact[i] && exact[j])) continue;
			const size_t at = (size_t) i * ncb * 16 + j;
			if((double) sums[nMag + at] < least) return 0;
			const double largest = P.cols[i].scale * P.cols[j].scale * (GD_MAG * GD_MAG); // product of the columns' scales
			P.left[(size_t) i * n + j] = (double) (int64_t) sums[at] * std::ldexp(largest, -70);
			P.mags[(size_t) i * n + j] = (double) sums[nMag + at] * largest / (GD_MAG * GD_MAG);
		}
	P.rc = 0;
	return 0;
}

template <int NF, int NARROW>
static int gd_launch(cla_block* b, const GdPlan& P, const GdArgs& A) {
	const auto kern = k_gram_tiles_i8<NF, NARROW>;
	CLA_HIP(allow_full_lds((const void*) kern));
	hipLaunchKernelGGL(kern, dim3((unsigned) P.grid), dim3(GD_THREADS), P.lds, b->stream, A);
	CLA_HIP(hipGetLastError());
	return 0;
}

// Where this pays: a call is two launches, the second of which reads a part per CU, and the fp64 kernel has its second block per CU from 262,144 rows on
// and, side by side, where dictionaries are small. Both in us (fp64 / here): more than 56 columns always, 64 columns 100 rows 15.6 / 11.6, 40,000
// 25.7 / 21.7, 112 columns of 256 values 100 rows 28.8 / 16.0; 49 columns 8,000 rows 16.4 / 13.7, 40,000 20.1 / 21.5, 100,000 24.9 / 23.9; 40 columns
// 2,000 12.0 / 11.5, 40,000 15.6 / 19.2, 200,000 24.4 / 25.6, 300,000 of 128 values 36.8 / 28.8, of 4 28.4 / 27.0; 33 of 4 values 500,000 33.2 / 34.5;
// 17 of 64 values 500,000 26.8 / 25.4, of 32 1,000,000 30.9 / 35.2, 2,500,000 61.4 / 62.3, 4,000,000 92 / 88; 24 of 8 values 1,000,000 36.3 / 35.0.
static bool gd_pays(const cla_block* b) {
	const int n = b->nCols, v = b->maxVals;
	const int64_t rows = b->nRows;
	if(n > 56) return true;
	if(n > 48) return rows <= 10000 || rows >= 100000;
	if(n > 32) return (n >= 40 && rows <= 10000) || rows >= (n < 40 && v <= 64 ? 1000000 : 262144);
	return rows >= (v > 48 ? 500000 : n >= 24 ? 1000000 : 3000000);
}

// Is the block's result on digits no further from the exact sums than the fp64 kernel's, which `fp64` writes to a zeroed matrix (its upper triangle at least)? Both
// are formed once and compared: what the digits leave out of a cell is known (k_gram_left), so the exact sums are, but for what is left out at weight 8. Neither the rms over the cells of the
// error divided by the sum of the terms' magnitudes nor the largest of them may exceed fp64's. (That depends on how the codes are distributed, more than on the values:
// where few tuples have most rows, the same rounding is added again and again, in fp64 in the long chains of many rows, on digits at any number. Rms fp64 / digits, diagonal
// and other cells, Zipf(1.1) codes of 256 normal values, 100 columns: 2,000 rows 8.0e-17 / 7.9e-17 and 8.8e-18 / 2.0e-17, which stay in fp64 as up to some 20,000 rows do, 50,000 1.7e-16 / 1.1e-16 and
// 1.0e-17 / 2.4e-17, 200,003 3.5e-16 / 8.9e-17 and 1.6e-17 / 2.3e-17, 2,000,003 2.4e-15 / 1.0e-16 and 7.5e-17 / 3.0e-17; uniform codes 10,007 rows 1.0e-16 / 5.2e-17 and
// 4.3e-18 / 3.4e-18. One value at 5 among them stays in fp64 at 200,003 rows, three decades of values, or a tuple with 99 % of the rows far below the largest, at any number measured.)
static int gd_compare(cla_block* b, GdPlan& P, const std::function<int(double*)>& fp64) {
	const int n = b->nCols;
	auto relative = [&](size_t at) { return P.left[at] / P.mags[at]; };
	double sum = 0.0, most = 0.0;
	int cells = 0;
	for(size_t at = 0; at < P.left.size(); at++)
		if(!std::isnan(P.left[at])) {
			sum += relative(at) * relative(at);
			most = std::max(most, std::fabs(relative(at)));
			cells++;
		}
	if(sum <= 1e-34 * cells && most <= 0x1p-55) P.suits[0] = P.suits[1] = true; // (fp64 1.5e-17 and more on any block that is not exact)
	else {
		struct Tmp { void* p = nullptr; ~Tmp() { if(p) (void) hipFree(p); } } tmp;
		const size_t nn = (size_t) n * n;
		if(no_room(&tmp.p, 2 * nn * sizeof(double))) return 1;
		double* const d = (double*) tmp.p;
		int rc = launch_zero(b, d, nn);
		if(rc || (rc = fp64(d)) || (rc = launch_gram_digits(b, nullptr, d + nn, nullptr, 0, 0))) return rc;
		std::vector<double> out(2 * nn);
		CLA_HIP(hipMemcpyAsync(out.data(), d, 2 * nn * sizeof(double), hipMemcpyDeviceToHost, b->stream));
		CLA_HIP(hipStreamSynchronize(b->stream));
		struct { double ours = 0.0, theirs = 0.0, oursMost = 0.0, theirsMost = 0.0; } of[2]; // all cells, those across groups
		for(int i = 0; i < n; i++)
			for(int j = i; j < n; j++) {
				const size_t at = (size_t) i * n + j;
				if(std::isnan(P.left[at])) continue;
				const GdCol &a = P.cols[i], &c = P.cols[j];
				const size_t cell = (size_t) std::min(a.col, c.col) * n + std::max(a.col, c.col);
				const double e = relative(at), f = (out[cell] - out[nn + cell] - P.left[at]) / P.mags[at];
				const double r = 0.58 * 0x1p-54 * out[cell] / P.mags[at]; // both results are rounded, and f has the rounding of either
				for(int s = 0; s < (a.group != c.group && a.group >= 0 && c.group >= 0 ? 2 : 1); s++) {
					of[s].ours += e * e + 2.0 * r * r;
					of[s].theirs += f * f;
					of[s].oursMost = std::max(of[s].oursMost, std::fabs(e));
					of[s].theirsMost = std::max(of[s].theirsMost, std::fabs(f));
				}
			}
		for(int s = 0; s < 2; s++) P.suits[s] = of[s].ours <= of[s].theirs && of[s].oursMost <= of[s].theirsMost;
	}
	P.compared = true;
	P.cols = {}; P.left = {}; P.mags = {};
	return 0;
}

// 0: the block goes this way (its plan is made), 1: it does not, negative: an error. across: only cells across groups are wanted of it. fp64: see gd_compare.
int gram_digits_plan(cla_block* b, bool across, const std::function<int(double*)>& fp64) {
	if(b->opt.tsmmDigits == 0 || (b->opt.tsmmDigits == 1 && !gd_pays(b))) return 1;
	if(b->gdPlan == nullptr) {
		// (a capture refuses the plan's allocations and its wait: the fp64 kernel)
		hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
		CLA_HIP(hipStreamIsCapturing(b->stream, &capturing));
		if(capturing != hipStreamCaptureStatusNone) return 1;
		std::unique_ptr<GdPlan> plan(new GdPlan()); // (the block's only when it is complete)
		const int rc = gd_build_plan(b, *plan);
		if(rc) return rc;
		if(plan->dImg && plan->rc) { (void) hipFree(plan->dImg); plan->dImg = nullptr; plan->bytes = 0; }
		b->derivedBytes += plan->bytes;
		b->gdPlan = plan.release();
	}
	GdPlan& P = *b->gdPlan;
	if(P.rc || b->opt.tsmmDigits == 2) return P.rc;
	if(!P.compared) {
		hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
		CLA_HIP(hipStreamIsCapturing(b->stream, &capturing));
		if(capturing != hipStreamCaptureStatusNone) return 1;
		// (its launches are not the call's)
		const size_t stats = b->lastStats.size();
		const NoProfile quiet(b);
		const int rc = gd_compare(b, P, fp64);
		b->lastStats.resize(stats);
		if(rc) return rc;
	}
	return P.suits[across] ? 0 : 1;
}

// dOut = t(X) %*% X, both triangles; dNnz (may be null): its non-zeros. skipOwn: cells inside a group and of columns without one
// are taken from acc, which is left at zero there if clearAcc.
int launch_gram_digits(cla_block* b, double* acc, double* dOut, unsigned long long* dNnz, int skipOwn, int clearAcc) {
	const GdPlan& P = *b->gdPlan;
	GdArgs A = P.A;
	A.nnz = dNnz;
	Prof pf(b, "k_gram_tiles", P.grid, GD_THREADS, (long) P.lds, (double) b->device_bytes_cached); // (its integer form, and what joins the sums)
	int rc = 1;
	switch(P.nf * 2 + P.narrow) {
		case 4: rc = gd_launch<2, 0>(b, P, A); break;
		case 6: rc = gd_launch<3, 0>(b, P, A); break;
		case 7: rc = gd_launch<3, 1>(b, P, A); break;
		case 8: rc = gd_launch<4, 0>(b, P, A); break;
		case 10: rc = gd_launch<5, 0>(b, P, A); break;
		case 11: rc = gd_launch<5, 1>(b, P, A); break;
		case 12: rc = gd_launch<6, 0>(b, P, A); break;
		case 13: rc = gd_launch<6, 1>(b, P, A); break;
		case 14: rc = gd_launch<7, 0>(b, P, A); break;
	}
	if(rc) return rc;
	hipLaunchKernelGGL(k_gram_join, dim3((unsigned) P.nCellTiles * (256 / GJ_CELLS)), dim3(GJ_THREADS), 0, b->stream, P.tiles, A.cols, P.nf, A.parts, P.grid,
		gd_slots(P.nf, P.narrow), acc, skipOwn, clearAcc, dOut, b->nCols, dNnz);
	CLA_HIP(hipGetLastError());
	return 0;
}

} // namespace cla
