/*
 * Test driver of libclahip.so's behaviour when host memory runs out inside a call: its own operator new fails the k-th
 * allocation that the library makes during cla_mmchain, k = 0, 1, ... until the call gets through. Each failure has to
 * come back as an error code, and the block has to answer the next plain X %*% v as if nothing had happened (the weights
 * of the failed chain must not show in it). The same for cla_tsmm of a block of two wide groups, whose kernels add into an
 * accumulator that the block keeps: the next t(X) %*% X must hold nothing of the failed one.
 *
 * Its own hipLaunchKernel fails the k-th launch of a Y %*% X on decoded rows, whose workspace is left at zero by a call: neither a
 * replay of a call captured before nor the next call may hold anything of the failed one.
 *
 * Its own hipMalloc fails the k-th device allocation of a first X %*% B and t(X) %*% X of a byte-code block: the plans of the forms on digits
 * are none that a call fails for.
 *
 * Host memory running out inside a first t(X) %*% X of a byte-code block, or inside cla_block_prepare, leaves the profiling mode as it was set.
 *
 * Prints "ALLOC-DRIVER OK" at the end; exit code 0 only then.
 */
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <new>
#include <vector>
#include "cla_hip.h"

static thread_local long allocLeft = -1; // allocations of the library until one fails; -1: none does
static thread_local bool allocFailed = false;

// Allocations of other libraries (the HIP runtime's among them) always succeed: the caller's code must lie in libclahip.so.
static bool from_library(void* ret) {
	Dl_info info;
	return dladdr(ret, &info) && info.dli_fname && strstr(info.dli_fname, "libclahip");
}

__attribute__((noinline)) void* operator new(size_t n) {
	if(allocLeft >= 0 && from_library(__builtin_return_address(0)) && allocLeft-- == 0) {
		allocFailed = true;
		throw std::bad_alloc();
	}
	if(void* p = malloc(n ? n : 1)) return p;
	throw std::bad_alloc();
}
__attribute__((noinline)) void operator delete(void* p) noexcept { free(p); }
__attribute__((noinline)) void operator delete(void* p, size_t) noexcept { free(p); }

static thread_local long launchLeft = -1; // launches of the library until one fails; -1: none does
static thread_local int launchError = 0;
static thread_local bool launchFailed = false;
static thread_local long roomLeft = -1; // device allocations of the library until one fails; -1: none does
static thread_local bool roomFailed = false;
struct Dim3 { uint32_t x, y, z; };

extern "C" int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t lds, void* stream) {
	static const auto next = (int (*)(const void*, Dim3, Dim3, void**, size_t, void*)) dlsym(RTLD_NEXT, "hipLaunchKernel");
	if(launchLeft >= 0 && launchLeft-- == 0) {
		launchFailed = true;
		return launchError = 2;
	}
	return next(f, grid, block, args, lds, stream);
}
extern "C" int hipMalloc(void** p, size_t bytes) {
	static const auto next = (int (*)(void**, size_t)) dlsym(RTLD_NEXT, "hipMalloc");
	if(roomLeft >= 0 && roomLeft-- == 0) {
		roomFailed = true;
		return 2;
	}
	return next(p, bytes);
}
extern "C" int hipGetLastError() {
	static const auto next = (int (*)()) dlsym(RTLD_NEXT, "hipGetLastError");
	const int injected = launchError;
	launchError = 0;
	return injected ? injected : next();
}

// The rest of the HIP runtime that libclahip.so has loaded
template <typename... A> static int hip(const char* name, A... a) {
	const auto f = (int (*)(A...)) dlsym(RTLD_DEFAULT, name);
	const int rc = f ? f(a...) : -1;
	if(rc) printf("%s: error %d\n", name, rc);
	return rc;
}

static const int64_t N = 1031;
enum { COLS = 3 };

// kind 0: byte codes, 1: two-byte codes, 2: offset lists of every third row
static cla_handle make_block(int kind, std::vector<double>& X) {
	cla_handle h = cla_block_create(N, COLS);
	X.assign((size_t) N * COLS, 0.0);
	for(int32_t c = 0; h && c < COLS; c++) {
		double dict[7];
		for(int k = 0; k < 7; k++) dict[k] = 0.5 + k + 10 * c;
		int rc;
		if(kind == 2) {
			std::vector<uint8_t> codes, deltas;
			for(int64_t r = c; r < N; r += 3) {
				codes.push_back((uint8_t) (r % 7));
				if(r > c) deltas.push_back(3);
				X[(size_t) r * COLS + c] = dict[r % 7];
			}
			rc = cla_block_add_sdc(h, &c, 1, dict, 7, nullptr, codes.data(), 1, deltas.data(), 1, (int32_t) deltas.size(), c,
				(int32_t) (c + 3 * (int64_t) (codes.size() - 1)), (int32_t) codes.size());
		}
		else {
			std::vector<uint8_t> bytes;
			std::vector<uint16_t> words;
			for(int64_t r = 0; r < N; r++) {
				const int k = (int) ((r * 5 + c) % 7);
				bytes.push_back((uint8_t) k);
				words.push_back((uint16_t) k);
				X[(size_t) r * COLS + c] = dict[k];
			}
			rc = cla_block_add_ddc(h, &c, 1, dict, 7, kind == 0 ? (const void*) bytes.data() : (const void*) words.data(), kind + 1);
		}
		if(rc < 0) { fprintf(stderr, "add: %s\n", cla_last_error()); return nullptr; }
	}
	if(!h || cla_block_finalize(h) < 0) { fprintf(stderr, "block: %s\n", cla_last_error()); return nullptr; }
	return h;
}

// t(X) %*% X of two groups of 8 columns with each allocation of the library failing in turn.
static int gram_failures(int& thrown) {
	enum { W = 8, M = 2 * W };
	int fails = 0;
	for(long k = 0;; k++) {
		cla_handle h = cla_block_create(N, M);
		std::vector<double> X((size_t) N * M), dict(7 * W), out(M * M);
		for(int g = 0; h && g < 2; g++) {
			std::vector<uint8_t> codes((size_t) N);
			int32_t cols[W];
			for(int c = 0; c < W; c++) cols[c] = g * W + c;
			for(int i = 0; i < 7 * W; i++) dict[(size_t) i] = 1 + i % 13 + g;
			for(int64_t r = 0; r < N; r++) {
				codes[(size_t) r] = (uint8_t) ((r * (3 + g)) % 7);
				for(int c = 0; c < W; c++) X[(size_t) r * M + g * W + c] = dict[(size_t) codes[(size_t) r] * W + c];
			}
			if(cla_block_add_ddc(h, cols, W, dict.data(), 7, codes.data(), 1) < 0) return 1;
		}
		if(!h || cla_block_finalize(h) < 0) { printf("gram block: %s\n", cla_last_error()); return 1; }
		allocFailed = false;
		allocLeft = k;
		const int64_t rc = cla_tsmm(h, out.data());
		allocLeft = -1;
		if(allocFailed) thrown++;
		if(allocFailed && rc >= 0) { printf("gram: allocation %ld failed without an error\n", k); fails++; }
		if(!allocFailed && rc < 0) { printf("gram: %s\n", cla_last_error()); fails++; }
		if(cla_tsmm(h, out.data()) < 0) { printf("gram: %s\n", cla_last_error()); fails++; }
		char stats[2048] = "";
		(void) cla_stats(h, stats, sizeof(stats));
		if(!strstr(stats, "k_gram_tiles")) { printf("gram, allocation %ld: the next call took another kernel: %s\n", k, stats); fails++; }
		int bad = 0;
		for(int i = 0; i < M; i++)
			for(int j = 0; j < M; j++) { // (whole numbers: exact)
				double s = 0;
				for(int64_t r = 0; r < N; r++) s += X[(size_t) r * M + i] * X[(size_t) r * M + j];
				bad += out[(size_t) i * M + j] != s;
			}
		if(bad) { printf("gram, allocation %ld: %d cells of the next t(X) %%*%% X are wrong\n", k, bad); fails++; }
		cla_block_free(h);
		if(!allocFailed) return fails;
	}
}

// Y %*% X on decoded rows with each launch of the library failing in turn, a replay of a captured call and a plain call behind each.
static int left_failures(int& thrown) {
	enum { M = 4, P = 2 };
	std::vector<double> X((size_t) N * M), Y((size_t) P * N), want(P * M, 0.0), got(P * M);
	std::vector<double> dict(2 * 300), dense((size_t) N * 2);
	std::vector<uint16_t> codes((size_t) N);
	for(int i = 0; i < 300; i++) { dict[2 * i] = i % 7; dict[2 * i + 1] = 3 - i % 5; }
	for(int64_t r = 0; r < N; r++) {
		codes[(size_t) r] = (uint16_t) (r * 7 % 300);
		for(int c = 0; c < 2; c++) {
			X[(size_t) r * M + c] = dict[2 * codes[(size_t) r] + c];
			X[(size_t) r * M + 2 + c] = dense[(size_t) r * 2 + c] = (double) ((r + c) % 9);
		}
		for(int i = 0; i < P; i++) Y[(size_t) i * N + r] = (double) ((r + 3 * i) % 11) - 4;
		for(int i = 0; i < P; i++)
			for(int c = 0; c < M; c++) want[(size_t) i * M + c] += Y[(size_t) i * N + r] * X[(size_t) r * M + c];
	}
	const int32_t c01[2] = {0, 1}, c23[2] = {2, 3};
	cla_handle h = cla_block_create(N, M);
	void *dY = nullptr, *dOut = nullptr, *stream = nullptr, *graph = nullptr, *exec = nullptr;
	const size_t outBytes = sizeof(double) * P * M;
	if(!h || cla_block_add_ddc(h, c01, 2, dict.data(), 300, codes.data(), 2) < 0 || cla_block_add_uncompressed(h, c23, 2, dense.data()) < 0 || cla_block_finalize(h) < 0 ||
		hip("hipMalloc", &dY, Y.size() * 8) || hip("hipMalloc", &dOut, outBytes) || hip("hipMemcpy", dY, (const void*) Y.data(), Y.size() * 8, 1) || hip("hipStreamCreate", &stream) ||
		cla_block_set_stream(h, stream) < 0 || cla_block_prepare(h, CLA_PRODUCT_LMM, 0, P) < 0 || hip("hipStreamBeginCapture", stream, 0) ||
		cla_lmm_dev_async(h, (const double*) dY, P, (double*) dOut) < 0 || hip("hipStreamEndCapture", stream, &graph) ||
		hip("hipGraphInstantiate", &exec, graph, (void*) nullptr, (char*) nullptr, (size_t) 0)) {
		printf("left: %s\n", cla_last_error());
		return 1;
	}
	char stats[2048] = "";
	(void) cla_stats(h, stats, sizeof(stats));
	if(!strstr(stats, "k_take_block")) { printf("left: another kernel: %s\n", stats); return 1; }
	int fails = 0;
	auto right = [&](const char* what, long k) { // (whole numbers: exact)
		if(hip("hipStreamSynchronize", stream) || hip("hipMemcpy", (void*) got.data(), (const void*) dOut, outBytes, 2) || got != want) {
			printf("left, launch %ld: %s is wrong\n", k, what);
			fails++;
		}
	};
	for(long k = 0;; k++) {
		launchFailed = false;
		launchLeft = k;
		const int64_t rc = cla_lmm_dev(h, (const double*) dY, P, (double*) dOut);
		launchLeft = -1;
		if(launchFailed == (rc >= 0)) { printf("left, launch %ld: %s\n", k, rc < 0 ? cla_last_error() : "no error"); fails++; }
		if(launchFailed) thrown++;
		for(int i = 0; i < 2; i++) {
			if(hip("hipGraphLaunch", exec, stream)) return fails + 1;
			right("a replay", k);
		}
		if(cla_lmm_dev(h, (const double*) dY, P, (double*) dOut) < 0) { printf("left: %s\n", cla_last_error()); fails++; }
		right("the next call", k);
		if(!launchFailed) break;
	}
	cla_block_free(h);
	if(hip("hipGraphExecDestroy", exec) || hip("hipGraphDestroy", graph) || hip("hipStreamDestroy", stream) || hip("hipFree", dY) || hip("hipFree", dOut)) fails++;
	return fails;
}

// X %*% B and t(X) %*% X of 64 byte-code columns with each device allocation of the first call failing in turn: with digits as many calls fail as
// without, and the results and the next call are right.
static int room_failures(int& thrown) {
	enum { M = 64, Q = 16, V = 5 };
	std::vector<uint8_t> codes((size_t) N * M);
	std::vector<double> dict(V), B((size_t) M * Q), X((size_t) N * M), want[2], got;
	for(int i = 0; i < V; i++) dict[(size_t) i] = i - 2 + (i == 2 ? 3 : 0);
	for(int64_t r = 0; r < N; r++)
		for(int c = 0; c < M; c++) X[(size_t) r * M + c] = dict[codes[(size_t) c * N + r] = (uint8_t) ((r * (c + 3) + c) % V)];
	for(int i = 0; i < M * Q; i++) B[(size_t) i] = i % 7 - 3;
	want[0].assign((size_t) N * Q, 0.0);
	want[1].assign(M * M, 0.0);
	for(int64_t r = 0; r < N; r++)
		for(int c = 0; c < M; c++) {
			for(int j = 0; j < Q; j++) want[0][(size_t) r * Q + j] += X[(size_t) r * M + c] * B[(size_t) c * Q + j];
			for(int j = 0; j < M; j++) want[1][(size_t) c * M + j] += X[(size_t) r * M + c] * X[(size_t) r * M + j];
		}
	int fails = 0;
	for(int gram = 0; gram < 2; gram++) {
		int failed[2] = {0, 0};
		for(int digits = 0; digits < 2; digits++)
			for(long k = 0;; k++) {
				cla_handle h = cla_block_create(N, M);
				bool ok = h != nullptr;
				for(int32_t c = 0; c < M && ok; c++) ok = cla_block_add_ddc(h, &c, 1, dict.data(), V, codes.data() + (size_t) c * N, 1) >= 0;
				if(!ok || cla_block_finalize(h) < 0 || cla_block_set_option(h, gram ? "tsmm_digits" : "rmm_digits", 2 * digits) < 0) { printf("room: %s\n", cla_last_error()); return fails + 1; }
				got.assign(want[gram].size(), -1.0);
				auto call = [&]() { return gram ? cla_tsmm(h, got.data()) : cla_rmm(h, B.data(), Q, got.data()); };
				roomFailed = false;
				roomLeft = k;
				const int64_t rc = call();
				roomLeft = -1;
				if(roomFailed) thrown++;
				failed[digits] += rc < 0;
				if(rc >= 0 && got != want[gram]) { printf("room, allocation %ld, gram %d, digits %d: the result is wrong\n", k, gram, digits); fails++; }
				got.assign(want[gram].size(), -1.0);
				if(call() < 0 || got != want[gram]) { printf("room, allocation %ld, gram %d, digits %d: the next call is wrong\n", k, gram, digits); fails++; }
				char stats[2048] = "";
				(void) cla_stats(h, stats, sizeof(stats));
				if(!gram && rc >= 0 && digits != (strstr(stats, "k_rmm_mfma_i8") != nullptr)) { printf("room, allocation %ld: the next call took another kernel: %s\n", k, stats); fails++; }
				cla_block_free(h);
				if(!roomFailed) break;
			}
		if(failed[0] != failed[1]) { printf("room, gram %d: %d failed calls without digits, %d with\n", gram, failed[0], failed[1]); fails++; }
	}
	return fails;
}

// t(X) %*% X of 64 byte-code columns, called or prepared, with each allocation of the library failing in turn while profiling is on: the next call's
// kernels have their times. (Values that digits round: both kernels run and their results are compared; those launches are not the call's.)
static int profile_failures(int& thrown) {
	enum { M = 64, V = 5 };
	std::vector<uint8_t> codes((size_t) N);
	std::vector<double> dict(V), out(M * M);
	for(int i = 0; i < V; i++) dict[(size_t) i] = 1.0 / (3 + i);
	int fails = 0;
	for(int prepare = 0; prepare < 2; prepare++)
		for(long k = 0;; k++) {
			cla_handle h = cla_block_create(N, M);
			bool ok = h != nullptr;
			for(int32_t c = 0; c < M && ok; c++) {
				for(int64_t r = 0; r < N; r++) codes[(size_t) r] = (uint8_t) ((r * (c + 3) + c) % V);
				ok = cla_block_add_ddc(h, &c, 1, dict.data(), V, codes.data(), 1) >= 0;
			}
			if(!ok || cla_block_finalize(h) < 0 || cla_block_profile(h, 1) < 0) { printf("profile: %s\n", cla_last_error()); return fails + 1; }
			allocFailed = false;
			allocLeft = k;
			const int64_t rc = prepare ? cla_block_prepare(h, CLA_PRODUCT_TSMM, 0, 0) : cla_tsmm(h, out.data());
			allocLeft = -1;
			if(allocFailed) thrown++;
			if(allocFailed == (rc >= 0)) { printf("profile, allocation %ld: %s\n", k, rc < 0 ? cla_last_error() : "no error"); fails++; }
			char stats[2048] = "";
			if(cla_tsmm(h, out.data()) < 0 || cla_stats(h, stats, sizeof(stats)) < 0) { printf("profile: %s\n", cla_last_error()); fails++; }
			if(!strstr(stats, "k_gram_tiles") || strstr(stats, "\"ms\":-")) { printf("profile, allocation %ld, prepare %d: the next call's times: %s\n", k, prepare, stats); fails++; }
			cla_block_free(h);
			if(!allocFailed) break;
		}
	return fails;
}

int main() {
	if(cla_init(0) < 0) { fprintf(stderr, "cla_init: %s\n", cla_last_error()); return 2; }
	int fails = 0, thrown = 0;
	for(int kind = 0; kind < 3; kind++)
		for(int ctype = 1; ctype <= 2; ctype++)
			for(long k = 0;; k++) {
				std::vector<double> X, w((size_t) N), out((size_t) N);
				cla_handle h = make_block(kind, X);
				if(!h) return 2;
				if(kind == 2 && cla_block_prepare(h, CLA_PRODUCT_RMM | CLA_PRODUCT_LMM, 1, 1) < 0) return 2; // (the lists' copies are no part of this)
				const double v[COLS] = {1.0, 0.25, -2.0};
				for(int64_t r = 0; r < N; r++) w[(size_t) r] = 3.0 + (double) (r % 5);
				double chain[COLS];
				allocFailed = false;
				allocLeft = k;
				const int64_t rc = cla_mmchain(h, v, w.data(), ctype, chain);
				allocLeft = -1;
				if(allocFailed) thrown++;
				if(allocFailed && rc >= 0) { printf("kind %d, allocation %ld failed without an error\n", kind, k); fails++; }
				if(!allocFailed && rc < 0) { printf("kind %d: %s\n", kind, cla_last_error()); fails++; }
				if(cla_rmm(h, v, 1, out.data()) < 0) { printf("kind %d: rmm: %s\n", kind, cla_last_error()); fails++; }
				int64_t bad = 0;
				for(int64_t r = 0; r < N; r++) { // (small multiples of 1/8: exact)
					double s = 0;
					for(int c = 0; c < COLS; c++) s += X[(size_t) r * COLS + c] * v[c];
					bad += out[(size_t) r] != s;
				}
				if(bad) { printf("kind %d, type %d, allocation %ld: %lld rows of the next X %%*%% v are wrong\n", kind, ctype, k, (long long) bad); fails++; }
				cla_block_free(h);
				if(!allocFailed) break;
			}
	int gramThrown = 0;
	fails += gram_failures(gramThrown);
	int leftThrown = 0;
	fails += left_failures(leftThrown);
	int roomThrown = 0;
	fails += room_failures(roomThrown);
	int profileThrown = 0;
	fails += profile_failures(profileThrown);
	printf("%d + %d + %d failed allocations, %d failed launches, %d failed device allocations\n", thrown, gramThrown, profileThrown, leftThrown, roomThrown);
	if(fails || thrown < 4 || gramThrown < 2 || leftThrown < 2 || roomThrown < 8 || profileThrown < 8) { printf("FAIL\n"); return 1; }
	printf("ALLOC-DRIVER OK\n");
	return 0;
}
