// FP64 GEMM NT and SYRK (lower) on the CDNA matrix cores (gfx950).
//
// C = beta*C + alpha*A*B^T with A (m x k), B (n x k), C (m x n), column-major.
// Two kernels on v_mfma_f64_16x16x4f64:
//
// k_dgemm_lds  workgroup tiles of 64x64 or 32x32, operands staged in LDS: a
//              single tile product (a tile task alone, or a few of them in
//              flight), any size, alignment and leading dimension.
// k_dgemm_nt   128x128 workgroup tiles (64x64 waves), operands from L2
//              straight into registers: large products, and many tile
//              products in flight, where two workgroups share a compute unit.

#include <atomic>

#include "sa_common.h"
#include "starpu_amd_kernels.h"

namespace {

// k_dgemm_nt: each wave owns a (16*WB) x (16*WB) block of C as WB x WB MFMA
// tiles; a workgroup has WVM x WVN waves.  Rows inside a wave are
// interleaved (MFMA tile b, MFMA row r -> C row WB*r + b) so each lane's A
// and B fragments for one k are WB contiguous doubles (16-byte loads) and
// its C values come in WB-row runs.  Operands stream from L2 straight into
// registers through a two-stage register pipeline; stages past k load
// clamped addresses and are zeroed with selects, so the loop body has no
// branches and the accumulators stay in AGPRs.
template <bool EDGE, int WB>
__device__ __forceinline__ void loadw(double (&v)[WB], const double *__restrict__ X, long ld,
                                      int row, int nrows, int k, int K)
{
	const bool kin = k < K;
	const long kc = kin ? k : K - 1;
	if (!EDGE) {
		const double *p = X + row + kc * ld;
#pragma unroll
		for (int h = 0; h < WB / 2; h++) {
			const sa_d2 t = *reinterpret_cast<const sa_d2 *>(p + 2 * h);
			v[2 * h] = kin ? t.x : 0.0;
			v[2 * h + 1] = kin ? t.y : 0.0;
		}
	} else {
#pragma unroll
		for (int b = 0; b < WB; b++) {
			const int rr = row + b;
			const bool in = kin && rr < nrows;
			const double val = X[(in ? rr : nrows - 1) + kc * ld];
			v[b] = in ? val : 0.0;
		}
	}
}

template <int WB, int WVM, int WVN, int KU, bool EDGE, bool LOWER, bool BETA0, int OCC = 1>
__global__ __launch_bounds__(64 * WVM * WVN, OCC)
void k_dgemm_nt(int M, int N, int K, double alpha, const double *__restrict__ A, long lda,
                const double *__restrict__ B, long ldb, double beta, double *__restrict__ C,
                long ldc, int tiles_m, int ktri)
{
	constexpr int WT = 16 * WB;
	constexpr int KS = 4 * KU;
	static_assert(!LOWER || WVM == WVN, "SYRK needs square workgroup tiles");
	int tm, tn;
	if (LOWER) {
		const int t = blockIdx.x;
		int i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
		while ((i + 1) * (i + 2) / 2 <= t) i++;
		while (i * (i + 1) / 2 > t) i--;
		tm = i;
		tn = t - i * (i + 1) / 2;
	} else {
		// Workgroups are dealt to the 8 XCDs round robin (XCD = id % 8), and
		// each XCD has its own L2.  Give each XCD a contiguous run of
		// logical ids and walk the tiles in groups of G tile rows (G a power
		// of two dividing tiles_m, G*G <= workgroups per XCD), so one XCD
		// covers a near-square block of C tiles: for a 1024x1024 product in
		// 64x64 workgroups a 4x8 block (4 A and 8 B operand panels instead
		// of 2 and 16), in 128x128 workgroups a 2x4 block (instead of 1x8).
		int t = blockIdx.x;
		const int T = gridDim.x;
		if ((T & 7) == 0)
			t = (t & 7) * (T >> 3) + (t >> 3);
		const int tiles_n = T / tiles_m;
		int G = 1;
		while (2 * G <= tiles_m && tiles_m % (2 * G) == 0 && 4 * G * G <= (T >> 3))
			G *= 2;
		tm = (t / (G * tiles_n)) * G + t % G;
		tn = (t / G) % tiles_n;
	}
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	const int row0 = tm * WT * WVM + (wave % WVM) * WT;
	const int col0 = tn * WT * WVN + (wave / WVM) * WT;
	if (LOWER && row0 + WT <= col0)
		return;         // wave block strictly above the diagonal
	if (EDGE && (row0 >= M || col0 >= N))
		return;
	// ktri: B (N x K) is lower triangular with zeros stored above its
	// diagonal, so the wave's columns col0 .. col0+WT-1 take only
	// k < col0 + WT (the terms left out are exact zeros; no barrier ties the
	// waves, so each stops at its own bound)
	if (ktri && col0 + WT < K)
		K = col0 + WT;
	const int r = lane & 15;
	const int g = lane >> 4;
	const int arow = row0 + WB * r;
	const int bcol = col0 + WB * r;

	sa_d4 acc[WB][WB];
	double fa0[KU][WB], fb0[KU][WB], fa1[KU][WB], fb1[KU][WB];

	auto load_stage = [&](double (&fa)[KU][WB], double (&fb)[KU][WB], int kb) {
#pragma unroll
		for (int s = 0; s < KU; s++) {
			const int k = kb + 4 * s + g;
			loadw<EDGE, WB>(fa[s], A, lda, arow, M, k, K);
			loadw<EDGE, WB>(fb[s], B, ldb, bcol, N, k, K);
		}
	};
	auto compute_stage = [&](const double (&fa)[KU][WB], const double (&fb)[KU][WB]) {
#pragma unroll
		for (int s = 0; s < KU; s++)
#pragma unroll
			for (int i = 0; i < WB; i++)
#pragma unroll
				for (int j = 0; j < WB; j++)
					acc[i][j] = sa_mfma(fa[s][i], fb[s][j], acc[i][j]);
	};

	// The first two stages are peeled and the first MFMA takes a zero
	// accumulator, so the accumulators are born in AGPRs and stay there.
	load_stage(fa0, fb0, 0);
	load_stage(fa1, fb1, KS);
#pragma unroll
	for (int s = 0; s < KU; s++)
#pragma unroll
		for (int i = 0; i < WB; i++)
#pragma unroll
			for (int j = 0; j < WB; j++)
				acc[i][j] = sa_mfma(fa0[s][i], fb0[s][j], s == 0 ? sa_d4{0.0, 0.0, 0.0, 0.0} : acc[i][j]);
	load_stage(fa0, fb0, 2 * KS);
	compute_stage(fa1, fb1);
	for (int kb = 2 * KS; kb < K; kb += 2 * KS) {
		load_stage(fa1, fb1, kb + KS);
		compute_stage(fa0, fb0);
		load_stage(fa0, fb0, kb + 2 * KS);
		compute_stage(fa1, fb1);
	}

	// acc[i][j][q] is C(row0 + WB*(4q+g) + i, col0 + WB*r + j).
#pragma unroll
	for (int j = 0; j < WB; j++) {
		const int col = col0 + WB * r + j;
		if (EDGE && col >= N)
			continue;
#pragma unroll
		for (int q = 0; q < 4; q++) {
			const int row = row0 + WB * (4 * q + g);
			double *p = C + row + (long)col * ldc;
			const bool fast = !EDGE && !(LOWER && row < col);
			if (fast) {
#pragma unroll
				for (int h = 0; h < WB / 2; h++) {
					sa_d2 v = BETA0 ? sa_d2{0.0, 0.0} : *reinterpret_cast<sa_d2 *>(p + 2 * h) * beta;
					v.x += alpha * acc[2 * h][j][q];
					v.y += alpha * acc[2 * h + 1][j][q];
					*reinterpret_cast<sa_d2 *>(p + 2 * h) = v;
				}
			} else {
#pragma unroll
				for (int i = 0; i < WB; i++) {
					const int rr = row + i;
					if ((EDGE && rr >= M) || (LOWER && rr < col))
						continue;
					const double c0 = BETA0 ? 0.0 : beta * p[i];
					p[i] = c0 + alpha * acc[i][j][q];
				}
			}
		}
	}
}

// The LDS-staged form: workgroup tiles of 32 WB x 32 WB (2 x 2 waves, each a
// (16 WB) x (16 WB) block).  The operand panels go through registers into
// LDS KC columns at a time: a thread loads single elements (64 or 32
// consecutive rows per column, so a wave's load is whole lines whatever the
// alignment), PF chunks ahead of their use, and each operand element is read
// from the cache once per workgroup instead of once per wave.  Rows past the
// matrix are read from its last row and not stored, columns k >= K are zero.
// Two LDS buffers, one barrier a chunk.  C is loaded at the start, ahead of
// everything that needs it.  The MFMA computes the transposed block, so that
// a lane's values of C are in consecutive lanes' rows: acc[j][i][q] =
// C(16 i + r, 16 j + 4q + g) of the wave's block.  The terms are added in the
// order of k, as in k_dgemm_nt.
//
// Bound: the MFMAs, and before that a wave's in-order issue.  There is
// mostly one wave per SIMD, whose LDS and memory instructions cost their
// issue and wait unless MFMAs stand between them: with the same loads,
// stores and MFMAs in three groups per chunk a 512^3 product took 31 us,
// interleaved one by one 22 (64x64 tiles; 20 with the MFMAs alone).  Alone /
// four in flight (us each): 256^3 6.1 / 4.5 with 32x32 tiles; 500^3 with
// an odd leading dimension 9.8 / 7.4; 512^3 9.4 / 6.9; 960^3 39.9 / 33.8 and
// 1024^3 42.7 / 36.8 with 64x64 tiles (58 TFLOP/s).  The same products took
// 15.0 / 8.0, 40.0 / 24.6, 25.8 / 16.3, 48.9 / 40.5 and 50.7 / 42.7 with
// 64x64 workgroups on k_dgemm_nt's register pipeline, where every wave loads
// its own operands.
template <int WB, int KC, int PF, bool LOWER, bool BETA0>
__global__ __launch_bounds__(256)
void k_dgemm_lds(int M, int N, int K, double alpha, const double *__restrict__ A, long lda,
                 const double *__restrict__ B, long ldb, double beta, double *__restrict__ C, long ldc,
                 int tiles_m, int ktri)
{
	constexpr int BT = 32 * WB, WT = 16 * WB;
	constexpr int KSTEP = 256 / BT;           // columns one load of all threads covers
	constexpr int NL = KC / KSTEP;            // loads per thread, operand and chunk
	constexpr int LDT = BT + 16;              // LDS row: the four columns of an MFMA step in different banks
	static_assert(PF % 2 == 0, "a chunk's LDS buffer follows from its register stage");
	__shared__ double As[2][KC * LDT], Bs[2][KC * LDT];
	int tm, tn;
	if (LOWER) {
		const int t = blockIdx.x;
		int i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
		while ((i + 1) * (i + 2) / 2 <= t) i++;
		while (i * (i + 1) / 2 > t) i--;
		tm = i;
		tn = t - i * (i + 1) / 2;
	} else {
		// tile order as k_dgemm_nt: near-square groups per XCD
		int t = blockIdx.x;
		const int T = gridDim.x;
		if ((T & 7) == 0)
			t = (t & 7) * (T >> 3) + (t >> 3);
		const int tiles_n = T / tiles_m;
		int G = 1;
		while (2 * G <= tiles_m && tiles_m % (2 * G) == 0 && 4 * G * G <= (T >> 3))
			G *= 2;
		tm = (t / (G * tiles_n)) * G + t % G;
		tn = (t / G) % tiles_n;
	}
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
	const int wr = (wave & 1) * WT, wc = (wave >> 1) * WT;
	const int row0 = tm * BT + wr, col0 = tn * BT + wc;
	// ktri: as k_dgemm_nt, here for the workgroup's columns together
	if (ktri && tn * BT + BT < K)
		K = tn * BT + BT;
	const bool active = row0 < M && col0 < N && !(LOWER && row0 + WT <= col0);

	double cv[WB][WB][4];
	if (!BETA0 && active) {
#pragma unroll
		for (int j = 0; j < WB; j++)
#pragma unroll
			for (int q = 0; q < 4; q++)
#pragma unroll
				for (int i = 0; i < WB; i++) {
					const int row = row0 + 16 * i + r, col = col0 + 16 * j + 4 * q + g;
						const int cc = col < N ? col : N - 1;
					const int rc = row < M ? row : M - 1;
					cv[j][i][q] = C[(LOWER && rc < cc ? cc : rc) + (long)cc * ldc];
				}
	}

	// a thread's element of a chunk's load i: uniform base + its own offset
	const int lr = tid % BT, lk = tid / BT;
	const long oa = (tm * BT + lr < M ? lr : M - 1 - tm * BT) + lk * lda;
	const long ob = (tn * BT + lr < N ? lr : N - 1 - tn * BT) + lk * ldb;
	const double *A0 = A + tm * BT, *B0 = B + tn * BT;
	const int nfull = K / KC, nch = (K + KC - 1) / KC;
	double ra[PF][NL], rb[PF][NL];
	// chunk c, or the last full one in place of those past it (never used)
	auto load = [&](int c, double (&xa)[NL], double (&xb)[NL]) {
		const long k = (long)(c < nfull ? c : nfull - 1) * KC;
#pragma unroll
		for (int i = 0; i < NL; i++) {
			xa[i] = (A0 + (k + KSTEP * i) * lda)[oa];
			xb[i] = (B0 + (k + KSTEP * i) * ldb)[ob];
		}
	};
	auto store = [&](int buf, const double (&xa)[NL], const double (&xb)[NL]) {
#pragma unroll
		for (int i = 0; i < NL; i++) {
			As[buf][(KSTEP * i + lk) * LDT + lr] = xa[i];
			Bs[buf][(KSTEP * i + lk) * LDT + lr] = xb[i];
		}
	};
	sa_d4 acc[WB][WB];
#pragma unroll
	for (int j = 0; j < WB; j++)
#pragma unroll
		for (int i = 0; i < WB; i++)
			acc[j][i] = sa_d4{0.0, 0.0, 0.0, 0.0};
	double fa[2][KC / 4][WB], fb[2][KC / 4][WB];
	auto fetch = [&](int buf, double (&xa)[KC / 4][WB], double (&xb)[KC / 4][WB]) {
#pragma unroll
		for (int s = 0; s < KC / 4; s++)
#pragma unroll
			for (int i = 0; i < WB; i++) {
				xa[s][i] = As[buf][(4 * s + g) * LDT + wr + 16 * i + r];
				xb[s][i] = Bs[buf][(4 * s + g) * LDT + wc + 16 * i + r];
			}
	};
	auto compute = [&](const double (&xa)[KC / 4][WB], const double (&xb)[KC / 4][WB]) {
#pragma unroll
		for (int s = 0; s < KC / 4; s++)
#pragma unroll
			for (int j = 0; j < WB; j++)
#pragma unroll
				for (int i = 0; i < WB; i++)
					acc[j][i] = sa_mfma(xb[s][j], xa[s][i], acc[j][i]);
	};
	// One chunk: the MFMAs on its fragments, and between them, one by one,
	// the LDS reads of the next chunk's, the LDS stores of the chunk after
	// that and the loads of the chunk PF further on.  A wave issues in order
	// and there is mostly one per SIMD, so memory instructions in a row
	// would leave the matrix core idle.  No branch: what goes past the last
	// full chunk repeats it and is not used.
	auto step = [&](int c, int u) {
		fetch((u + 1) & 1, fa[(u + 1) & 1], fb[(u + 1) & 1]);
		store(u & 1, ra[(u + 2) % PF], rb[(u + 2) % PF]);
		load(c + 2 + PF, ra[(u + 2) % PF], rb[(u + 2) % PF]);
		compute(fa[u & 1], fb[u & 1]);
		constexpr int NM = (KC / 4) * WB * WB;                     // MFMAs
		constexpr int NR = (KC / 4) * WB, NS = 2 * NL;             // LDS reads (pairs), stores, loads
#pragma unroll
		for (int q = 0; q < NM; q++) {
			__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
			// first half of the MFMAs: the reads; second half: stores, loads
			const int h = NM / 2;
			if (q < h) {
				__builtin_amdgcn_sched_group_barrier(0x100, (NR + h - 1) / h, 0);
			} else {
				__builtin_amdgcn_sched_group_barrier(0x200, (NS + h - 1) / h, 0);
				__builtin_amdgcn_sched_group_barrier(0x020, (NS + h - 1) / h, 0);
			}
		}
		__builtin_amdgcn_sched_barrier(0);
		__syncthreads();
		__builtin_amdgcn_sched_barrier(0);
	};
	if (nfull > 0) {
#pragma unroll
		for (int u = 0; u < PF; u++)
			load(u, ra[u], rb[u]);
		store(0, ra[0], rb[0]);
		load(PF, ra[0], rb[0]);
		store(1, ra[1], rb[1]);
		load(PF + 1, ra[1], rb[1]);
		__syncthreads();
		fetch(0, fa[0], fb[0]);
		__syncthreads();
		int c0 = 0;
		for (; c0 + PF <= nfull; c0 += PF) {
#pragma unroll
			for (int u = 0; u < PF; u++)
				step(c0 + u, u);
		}
#pragma unroll
		for (int u = 0; u < PF - 1; u++)
			if (c0 + u < nfull)
				step(c0 + u, u);
	}
	if (nfull < nch) {
		// the last K % KC columns, zero past K
#pragma unroll
		for (int i = 0; i < NL; i++) {
			const int k = nfull * KC + KSTEP * i + lk;
			const long back = k < K ? 0 : k - (K - 1);
			const double xa = (A0 + (long)(nfull * KC + KSTEP * i) * lda)[oa - back * lda];
			const double xb = (B0 + (long)(nfull * KC + KSTEP * i) * ldb)[ob - back * ldb];
			As[0][(KSTEP * i + lk) * LDT + lr] = k < K ? xa : 0.0;
			Bs[0][(KSTEP * i + lk) * LDT + lr] = k < K ? xb : 0.0;
		}
		__syncthreads();
		fetch(0, fa[0], fb[0]);
		compute(fa[0], fb[0]);
	}
	if (!active)
		return;
#pragma unroll
	for (int j = 0; j < WB; j++)
#pragma unroll
		for (int q = 0; q < 4; q++)
#pragma unroll
			for (int i = 0; i < WB; i++) {
				const int row = row0 + 16 * i + r, col = col0 + 16 * j + 4 * q + g;
				if (row < M && col < N && (!LOWER || row >= col))
					C[row + (long)col * ldc] = (BETA0 ? 0.0 : beta * cv[j][i][q]) + alpha * acc[j][i][q];
			}
}

// X <- a*X over an m x n region (lower: only i >= j).
__global__ void k_scale(int m, int n, double *X, long ld, double a, int lower)
{
	const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (idx >= (long)m * n)
		return;
	const int i = (int)(idx % m), j = (int)(idx / m);
	if (lower && i < j)
		return;
	double *p = X + i + (long)j * ld;
	*p = (a == 0.0) ? 0.0 : a * *p;
}

template <int WB, int WV, int KU, bool LOWER, int OCC = 1>
int gemm_shape(hipStream_t s, int m, int n, int k, double alpha, const double *A, int lda,
               const double *B, int ldb, double beta, double *C, int ldc, int ktri = 0)
{
	constexpr int BT = 16 * WB * WV;
	const int tiles_m = (m + BT - 1) / BT;
	const int tiles_n = (n + BT - 1) / BT;
	const unsigned grid = LOWER ? (unsigned)(tiles_m * (tiles_m + 1) / 2) : (unsigned)(tiles_m * tiles_n);
	const bool vec = sa_aligned16(A) && sa_aligned16(B) && sa_aligned16(C) && (lda % 2 == 0) &&
	                 (ldb % 2 == 0) && (ldc % 2 == 0);
	const bool edge = !vec || (m % BT) || (n % BT);
	const bool b0 = (beta == 0.0);
	const dim3 blk(64 * WV * WV);
#define SA_GEMM_LAUNCH(E, Z)                                                                      \
	hipLaunchKernelGGL((k_dgemm_nt<WB, WV, WV, KU, E, LOWER, Z, OCC>), dim3(grid), blk, 0, s, m, n, k,  \
	                   alpha, A, (long)lda, B, (long)ldb, beta, C, (long)ldc, tiles_m, ktri)
	if (edge) {
		if (b0) SA_GEMM_LAUNCH(true, true); else SA_GEMM_LAUNCH(true, false);
	} else {
		if (b0) SA_GEMM_LAUNCH(false, true); else SA_GEMM_LAUNCH(false, false);
	}
#undef SA_GEMM_LAUNCH
	return sa_launch_status();
}

template <int WB, int KC, int PF, bool LOWER>
int gemm_lds(hipStream_t s, int m, int n, int k, double alpha, const double *A, int lda, const double *B, int ldb,
             double beta, double *C, int ldc, int ktri)
{
	constexpr int BT = 32 * WB;
	const int tiles_m = (m + BT - 1) / BT, tiles_n = (n + BT - 1) / BT;
	const unsigned grid = LOWER ? (unsigned)(tiles_m * (tiles_m + 1) / 2) : (unsigned)(tiles_m * tiles_n);
	if (beta == 0.0)
		hipLaunchKernelGGL((k_dgemm_lds<WB, KC, PF, LOWER, true>), dim3(grid), dim3(256), 0, s, m, n, k, alpha, A,
		                   (long)lda, B, (long)ldb, beta, C, (long)ldc, tiles_m, ktri);
	else
		hipLaunchKernelGGL((k_dgemm_lds<WB, KC, PF, LOWER, false>), dim3(grid), dim3(256), 0, s, m, n, k, alpha, A,
		                   (long)lda, B, (long)ldb, beta, C, (long)ldc, tiles_m, ktri);
	return sa_launch_status();
}

// Launches the caller keeps in flight on one device (sa_set_launch_concurrency).
std::atomic<int> g_concurrency{1};

// Forced workgroup tile (64 or 128), or 0 for the choice by launch
// concurrency.  Read from SA_GEMM_SHAPE on first use; sa_set_gemm_shape
// changes it at run time.
std::atomic<int> g_shape_override{-1};

int tile_shape_override()
{
	int v = g_shape_override.load(std::memory_order_relaxed);
	if (v < 0) {
		const char *e = getenv("SA_GEMM_SHAPE");
		const int w = e ? atoi(e) : 0;
		g_shape_override.compare_exchange_strong(v, (w == 64 || w == 128) ? w : 0);
		v = g_shape_override.load(std::memory_order_relaxed);
	}
	return v;
}

// Workgroup tile edge (64 or 128) that a product of this shape runs with.
// 128x128 workgroups (half the operand traffic per flop) while the
// launches in flight together give every compute unit about 1.5 of them;
// otherwise the LDS-staged kernel with smaller ones.  With 12 streams of
// 1024^3 products in flight over 16 hardware queues, 128x128 workgroups run
// the N=32768 tile-1024 factorisation at 57 TFLOP/s; with the four queues of
// a default process, where a 128x128 launch is 64 workgroups, the 64x64
// workgroups do better (36.8 us a product against 87).
int pick_shape(bool lower, int m, int n)
{
	const int forced = tile_shape_override();
	if (forced == 64 || forced == 128)
		return forced;
	const long big_tiles = lower ? (long)((m + 127) / 128) * ((m + 127) / 128 + 1) / 2
	                             : (long)((m + 127) / 128) * ((n + 127) / 128);
	return big_tiles * g_concurrency.load(std::memory_order_relaxed) >= 384 ? 128 : 64;
}

} // namespace

int sa_scale_launch(hipStream_t s, int m, int n, double *X, int ld, double a, bool lower)
{
	const long cnt = (long)m * n;
	if (cnt == 0)
		return 0;
	hipLaunchKernelGGL(k_scale, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, s, m, n, X,
	                   (long)ld, a, lower ? 1 : 0);
	return sa_launch_status();
}

namespace {

int gemm_launch(hipStream_t s, bool lower, int m, int n, int k, double alpha, const double *A, int lda,
                const double *B, int ldb, double beta, double *C, int ldc, int ktri)
{
	if (m == 0 || n == 0)
		return 0;
	if (k == 0)
		return beta == 1.0 ? 0 : sa_scale_launch(s, m, n, C, ldc, beta, lower);
	const int shape = pick_shape(lower, m, n);
	// 128x128: two k-steps per pipeline stage, so that two workgroups fit on
	// a CU (216 VGPRs); with four k-steps per stage (316 registers, one
	// workgroup per CU) the tile-1024 factorisation ran at 51.2 against 54.0
	// TFLOP/s and an 8192^3 product at 63 against 66 TFLOP/s; one k-step per
	// stage at three workgroups per CU (164 VGPRs) ran it at 47.2.
	if (shape == 128)
		return lower ? gemm_shape<4, 2, 2, true, 2>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ktri)
		             : gemm_shape<4, 2, 2, false, 2>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ktri);
	// 32x32 workgroups where 64x64 ones would not reach most of the 256
	// compute units: 4 times as many, a quarter of the MFMAs each.  Alone /
	// four in flight (us), 32x32 against 64x64: 256^3 6.1 / 4.5 and 13.3 / 7.5;
	// 512^3 (64 of the latter) 9.4 / 6.9 and 22.6 / 12.0; the lower 1024^3 (136)
	// 33.8 / 26.1 and 41.2 / 28.1; 960^3 (225) 42.5 / 37.8 and 39.9 / 33.8.
	const long t64m = (m + 63) / 64, t64n = (n + 63) / 64;
	if ((lower ? t64m * (t64m + 1) / 2 : t64m * t64n) < 192)
		return lower ? gemm_lds<1, 16, 4, true>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ktri)
		             : gemm_lds<1, 16, 4, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ktri);
	return lower ? gemm_lds<2, 16, 2, true>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ktri)
	             : gemm_lds<2, 16, 2, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, ktri);
}

} // namespace

int sa_gemm_launch(hipStream_t s, bool lower, int m, int n, int k, double alpha, const double *A,
                   int lda, const double *B, int ldb, double beta, double *C, int ldc)
{
	return gemm_launch(s, lower, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, 0);
}

extern "C" int sa_set_launch_concurrency(int n)
{
	return g_concurrency.exchange(n > 0 ? n : 1);
}

extern "C" int sa_set_gemm_shape(int edge)
{
	if (edge != 0 && edge != 64 && edge != 128)
		return -EINVAL;
	tile_shape_override();   // settle the environment's value first
	return g_shape_override.exchange(edge);
}

extern "C" int sa_gemm_tile_shape(int lower, int m, int n)
{
	if (m <= 0 || n <= 0)
		return -EINVAL;
	return pick_shape(lower != 0, m, lower ? m : n);
}

extern "C" int sa_dgemm_nt(hipStream_t s, int m, int n, int k, double alpha, const double *A,
                           int lda, const double *B, int ldb, double beta, double *C, int ldc)
{
	if (m < 0 || n < 0 || k < 0 || ldc < (m > 1 ? m : 1) ||
	    (k > 0 && (lda < (m > 1 ? m : 1) || ldb < (n > 1 ? n : 1))))
		return -EINVAL;
	return sa_gemm_launch(s, false, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

extern "C" int sa_dgemm_nt_ltri(hipStream_t s, int m, int n, double alpha, const double *A, int lda,
                                const double *L, int ldl, double beta, double *C, int ldc)
{
	if (m < 0 || n < 0 || ldc < (m > 1 ? m : 1) || (n > 0 && (lda < (m > 1 ? m : 1) || ldl < (n > 1 ? n : 1))))
		return -EINVAL;
	return gemm_launch(s, false, m, n, n, alpha, A, lda, L, ldl, beta, C, ldc, 1);
}

extern "C" int sa_dsyrk_ln(hipStream_t s, int n, int k, double alpha, const double *A, int lda,
                           double beta, double *C, int ldc)
{
	if (n < 0 || k < 0 || ldc < (n > 1 ? n : 1) || (k > 0 && lda < (n > 1 ? n : 1)))
		return -EINVAL;
	return sa_gemm_launch(s, true, n, n, k, alpha, A, lda, A, lda, beta, C, ldc);
}
