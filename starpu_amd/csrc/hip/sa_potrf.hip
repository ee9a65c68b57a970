// Cholesky factorisation of one diagonal tile (n <= 2048), with the inverse
// of its factor, in a single persistent kernel (gfx950).
//
// Inside a task graph the diagonal-tile POTRF heads the critical path, and
// while it runs the other HIP streams keep every compute unit busy with
// tile GEMMs.  A POTRF built from one kernel launch per 64-column step (a
// 64x64 factor-and-invert, a panel apply, a trailing update: three
// dependent launches per step, 48 for a 1024 tile) then waits for the
// command processor and for free workgroup slots at every launch.  Here the
// whole tile is one launch: its workgroups wait for each other through
// counters in device memory instead.
//
// Work is split into items on 64x64 blocks (block b covers rows and columns
// 64b .. 64b+w_b-1 of the tile), left-looking: an item owns one block, sums
// its products over all the columns to its left in registers and touches
// the block in memory once.  The factorisation:
//   chain(j)  by workgroup 0, which keeps the blocks of its step in LDS:
//             D(j) factors and inverts the diagonal block, L(j+1,j) =
//             A(j+1,j) inv(L(j,j))^T, and the last update of the next
//             diagonal block, A(j+1,j+1) -= L(j+1,j) L(j+1,j)^T, stays in LDS
//   S(j)      A(j+1,j) -= sum_{t<j} L(j+1,t) L(j,t)^T            (MFMA)
//   G(j)      A(j+1,j+1) -= sum_{t<j} L(j+1,t) L(j+1,t)^T        (MFMA)
//   P(i,j)    L(i,j) = (A(i,j) - sum_{t<j} L(i,t) L(j,t)^T) inv(L(j,j))^T
//             for i > j + 1                                      (MFMA)
// S and G prepare what the chain takes at step j; the product with t = j - 1
// of S(j) is the only work that lies between two steps of the chain, and it
// runs beside D(j).  When the inverse is asked for, W = L^-T (upper) block by
// block, W(j,j) = inv(L(j,j))^T,
// W(j,i) = -(sum_{t=j}^{i-1} W(j,t) L(i,t)^T) inv(L(i,i))^T:
//   WD(t)     W(t,t), from the inverse D(t) formed
//   WX(j,i)   W(j,i), the sum in registers, one store
// with Linv = L^-1 = W^T written beside W by WD and WX when asked for.
// These are the inverse's flops (n^3/3) on the same matrix cores, overlapped
// with the factorisation's critical chain instead of following it.
//
// Ordering and progress.  Every item depends only on items that come earlier
// in one fixed global order: step by step, chain(j), S(j), G(j), P(i,j) from
// i = j + 2 on, then the inverse items of block column j - 1, WD(j-1) and
// WX(t, j-1) for t < j-1 (one step late, so that the factor items the chain
// waits for come first).  Within a step chain(j) follows S(j) and G(j), which
// need no more of step j than nothing: their inputs are of steps before it.
// Workgroup 0 runs the chain; the other workgroups take the remaining items
// in that order from a ticket counter.  Each workgroup processes its items in
// increasing order, so the lowest unfinished item always has all its inputs
// ready and a running workgroup holds it: the grid always drains.  The blocks
// of a row of L (and of W) become final from left to right, each after the
// one before it, so one counter per row tells how many are: an item reads
// two counters and then runs through every product that is ready without
// another look.  The products of a block are added in the order of t, so the
// result does not depend on timing.  Inverting an already factored tile
// (sa_dtrtri_tile) runs the same inverse items after D items that only
// invert, so a solve on a resident factor multiplies by the same bits.
//
// Bound: the chain, 17.6 us a step alone on the chip (8.5 the block, 3.3 the
// stores, the look at what is prepared and its loads, 1.3 the panel product,
// 0.9 its publication, 2.4 the diagonal update, taken apart; about 1 the waits
// for the two write-backs), from about 31 bulk
// workgroups on up to n = 1024, and the bulk beyond: a 1024 tile with both
// inverses takes 338 us with 31 workgroups and 302 with 63, a 2048 tile 1537
// with 31 and 968 with 63.  One item per block and update step (right-looking),
// each block read and written at every step and the chain's blocks handed
// on through memory, took 43 us a step and 1357, 1056 and 907 us for a 1024
// tile with 31, 63 and 127.
//
// Every wait is bounded: a counter that does not reach its value within
// seconds (which cannot happen unless the order above is broken) raises
// an abort flag, after which no wait waits any more: every workgroup runs
// through its items on whatever memory holds (in bounds all the same), the
// grid drains and the factorisation reports info = -1, so a fault of the
// ordering shows as an error, not as a hung device.  The chain writes info
// while the last inverse items may still run; a wait of theirs that gives up
// after that writes -1 itself (give_up).  Inverting a factored tile has no
// info to report in.
//
// Visibility across workgroups (possibly on different XCDs, each with its own
// L2) uses agent-scope release fences before a counter is raised and an
// agent-scope acquire after a wait.
#include <cstdlib>
#include <mutex>

#include "sa_block64.h"
#include "starpu_amd_kernels.h"

namespace {
using namespace sa64;

constexpr int PF_MAXN = 2048;

// Workgroups that take the bulk items (besides the chain's): more finish a
// tile sooner alone, fewer leave more compute units to the kernels running
// beside it.  SA_POTRF_WORKGROUPS overrides (1..255).
int max_bulk()
{
	static int v = -1;
	if (v < 0) {
		const char *e = getenv("SA_POTRF_WORKGROUPS");
		const int x = e ? atoi(e) : 0;
		v = (x >= 1 && x <= 255) ? x : 31;
	}
	return v;
}

// The counters, 64 bytes apart (two to a 128-byte cache line): rows of L, then
// "A(i,i) / A(i+1,i) prepared" and "D(i) done" flags, rows of W, the ticket
// and the abort flag.
constexpr int FLAG_STRIDE = 16;       // unsigned per line
constexpr int flag_words(int nb) { return (5 * nb + 2) * FLAG_STRIDE; }

struct PfArgs {
	int n, nb, nbulk;
	int factor;         // 1: factor A in place; 0: A holds the factor already
	int inv;            // form W = L^-T (and Linv = L^-1 when Linv is given)
	int delay;          // steps the inverse items trail the factor items by
	sa_gd *A;
	long lda;
	sa_gd *W;
	long ldw;
	sa_gd *Linv;
	long ldi;
	sa_gd *Dinv;      // nb blocks of 64x64 (ld 64)
	sa_gu *flags;
	unsigned stop;      // bits of the abort word that end a wait: ABORT_GAVE_UP
	int *info;
	__device__ sa_gu *rowl(int i) const { return flags + FLAG_STRIDE * i; }          // L(i,t) final for t < value
	__device__ sa_gu *diag(int i) const { return flags + FLAG_STRIDE * (nb + i); }   // A(i,i) but for t = i - 1
	__device__ sa_gu *sub(int i) const { return flags + FLAG_STRIDE * (2 * nb + i); } // A(i+1,i), all t < i
	__device__ sa_gu *dfin(int i) const { return flags + FLAG_STRIDE * (3 * nb + i); }
	__device__ sa_gu *roww(int j) const { return flags + FLAG_STRIDE * (4 * nb + j); } // W(j,t) final for t < value
	__device__ sa_gu *ticket() const { return flags + FLAG_STRIDE * (5 * nb); }
	__device__ sa_gu *abortf() const { return flags + FLAG_STRIDE * (5 * nb + 1); }
};

__device__ __forceinline__ int bw(const PfArgs &p, int b) { return (p.n - 64 * b) < 64 ? (p.n - 64 * b) : 64; }

__device__ __forceinline__ unsigned flag_read(const sa_gu *f)
{
	return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A wait gives up after SPIN_LIMIT polls.  Each poll is two or three
// device-coherent loads of about a microsecond and a short sleep, so 2^22
// polls are several seconds: far beyond any wait of a correct schedule (an
// item takes tens of microseconds).
constexpr unsigned SPIN_LIMIT = 1u << 22;

// The abort word: a wait gave up; the chain has written info (and what it
// wrote is in memory).  Each side sets its bit and looks at the other's in one
// atomic step, so one of them sees both and the -1 is the last store to info.
constexpr unsigned ABORT_GAVE_UP = 1, ABORT_REPORTED = 2;

__device__ __forceinline__ unsigned abort_or(const PfArgs &p, unsigned bit)
{
	return __hip_atomic_fetch_or(p.abortf(), bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void give_up(const PfArgs &p)
{
	if ((threadIdx.x & 63) == 0 && (abort_or(p, ABORT_GAVE_UP) & ABORT_REPORTED) && p.info)
		*p.info = -1;
}

// One wave waits until both counters have reached v (or the run is
// abandoned) and then sees the data published before they were raised.
// Returns the smaller counter, at least v.
__device__ __forceinline__ int await(const PfArgs &p, const sa_gu *f1, const sa_gu *f2, int v)
{
	unsigned it = 0;
	int m;
	for (;;) {
		const int a = (int)flag_read(f1), b = (int)flag_read(f2);
		m = __builtin_amdgcn_readfirstlane(a < b ? a : b);
		if (m >= v)
			break;
		if (((unsigned)__builtin_amdgcn_readfirstlane((int)flag_read(p.abortf())) & p.stop) || ++it > SPIN_LIMIT) {
			give_up(p);
			m = v;
			break;
		}
		__builtin_amdgcn_s_sleep(1);
	}
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
	return m;
}

// Every thread's stores become visible at agent scope, then the counter is
// raised.  Each wave waits for its own stores to complete before the
// barrier; thread 0's agent-scope release then covers them all, so the L2
// write-back runs once per item rather than once per wave.  The wait for that
// write-back is written out: the compiler takes the wait before the barrier
// for proof that nothing is outstanding and drops the one of a release
// fence or store that follows it, and the counter then reaches another XCD
// before the data has left this one's L2.
__device__ __forceinline__ void publish(sa_gu *f, unsigned v)
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
	__builtin_amdgcn_s_waitcnt(0);
	__syncthreads();
	if (threadIdx.x == 0) {
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
		__builtin_amdgcn_s_waitcnt(0);
		__hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
}

// acc += Pr Pc^T over the columns 64 t0 .. 64 t1 - 1 of two block rows, for
// the wave's 32x32 quadrant (rows i0 = 32 (wave & 1).., columns j0 = 32
// (wave >> 1)..).  Pr and Pc are the lanes' addresses of column 0 in the two
// block rows: rows r and r + 16 of the quadrant's half, columns k = 4s + g.
// The MFMA computes the transposed product so a lane's results are
// consecutive rows: acc[bj][bi][q] = (Pr Pc^T)(i0 + 16 bi + r,
// j0 + 16 bj + 4q + g).  Blocks t of the two rows are ready for t below both
// counters.  Operands come in stages of 32 columns, one stage ahead of the
// MFMAs; while a block's first half is multiplied the counters are read
// again, so that a run goes on without a pause when more has become ready.
struct Operand {
	const sa_gd *p[2];      // the lane's two rows, column g
	long ld;
};

__device__ __forceinline__ Operand operand(const sa_gd *X, long ld, int row0, int last)
{
	const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	Operand o;
#pragma unroll
	for (int b = 0; b < 2; b++) {
		const int row = row0 + 16 * b + r;
		o.p[b] = X + (row < last ? row : last) + g * ld;
	}
	o.ld = ld;
	return o;
}

__device__ __forceinline__ void load_half(const Operand &o, int k, double (&x)[2][8])
{
#pragma unroll
	for (int s = 0; s < 8; s++)
#pragma unroll
		for (int b = 0; b < 2; b++)
			x[b][s] = o.p[b][(long)(k + 4 * s) * o.ld];
}

__device__ __forceinline__ void mul_half(const double (&xr)[2][8], const double (&xc)[2][8], sa_d4 (&acc)[2][2])
{
#pragma unroll
	for (int s = 0; s < 8; s++)
#pragma unroll
		for (int bj = 0; bj < 2; bj++)
#pragma unroll
			for (int bi = 0; bi < 2; bi++)
				acc[bj][bi] = sa_mfma(xc[bj][s], xr[bi][s], acc[bj][bi]);
}

__device__ __forceinline__ void accumulate(const PfArgs &p, const Operand &Pr, const Operand &Pc,
                                           const sa_gu *fr, const sa_gu *fc, int t0, int t1,
                                           sa_d4 (&acc)[2][2])
{
	double r0[2][8], c0[2][8], r1[2][8], c1[2][8];
#pragma unroll
	for (int a = 0; a < 2; a++)
#pragma unroll
		for (int b = 0; b < 2; b++)
			acc[a][b] = sa_d4{0.0, 0.0, 0.0, 0.0};
	int ready = t0;
	bool staged = false;            // the first half of block t is in r0, c0
	for (int t = t0; t < t1; t++) {
		if (!staged) {
			if (ready <= t)
				ready = await(p, fr, fc, t + 1);
			load_half(Pr, 64 * t, r0);
			load_half(Pc, 64 * t, c0);
		}
		load_half(Pr, 64 * t + 32, r1);
		load_half(Pc, 64 * t + 32, c1);
		unsigned fa = 0, fb = 0;
		const bool look = ready <= t + 1 && t + 1 < t1;
		if (look) {
			fa = flag_read(fr);
			fb = flag_read(fc);
		}
		mul_half(r0, c0, acc);
		if (look) {
			const int m = __builtin_amdgcn_readfirstlane((int)(fa < fb ? fa : fb));
			if (m > ready) {
				__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
				ready = m;
			}
		}
		staged = t + 1 < t1 && ready > t + 1;
		if (staged) {
			load_half(Pr, 64 * t + 64, r0);
			load_half(Pc, 64 * t + 64, c0);
		}
		mul_half(r1, c1, acc);
	}
}

// X = T inv^T for the wave's 16 rows 16 wave ..: T (64x64) in LDS, inv a
// lower 64x64 block with leading dimension ldd (its zeros above the diagonal
// are not multiplied).  x[cb][q] = X(16 wave + r, 16 cb + 4q + g).
__device__ __forceinline__ void apply_inv(const double *T, const sa_gd *Dj, long ldd, sa_d4 (&x)[4])
{
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	double dv[40];
#pragma unroll
	for (int cb = 0, q = 0; cb < 4; cb++)
#pragma unroll
		for (int s = 0; s < 4 * (cb + 1); s++, q++)
			dv[q] = Dj[(16 * cb + r) + (4 * s + g) * ldd];
#pragma unroll
	for (int cb = 0; cb < 4; cb++)
		x[cb] = sa_d4{0.0, 0.0, 0.0, 0.0};
	// k outermost: the four column blocks are independent accumulators
#pragma unroll
	for (int s = 0; s < 16; s++) {
		const double t = T[(16 * wave + r) + (4 * s + g) * LD];
#pragma unroll
		for (int cb = 0; cb < 4; cb++)
			if (s < 4 * (cb + 1))
				x[cb] = sa_mfma(dv[2 * cb * (cb + 1) + s], t, x[cb]);
	}
}

// ---- factorisation items ---------------------------------------------------

// S(j) (l = j) and G(j) (l = j + 1): A(j+1,l) -= sum_{t<j} L(j+1,t) L(l,t)^T.
__device__ __noinline__ void item_prepare(const PfArgs &p, int j, int l)
{
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	const int i0 = 32 * (wave & 1), j0 = 32 * (wave >> 1);
	const int i = j + 1, wr = bw(p, i), wc = bw(p, l);
	sa_gd *C = p.A + 64 * i + 64L * l * p.lda;
	double cv[2][4][2];
#pragma unroll
	for (int bj = 0; bj < 2; bj++)
#pragma unroll
		for (int q = 0; q < 4; q++)
#pragma unroll
			for (int bi = 0; bi < 2; bi++) {
				const int ic = i0 + 16 * bi + r, jc = j0 + 16 * bj + 4 * q + g;
				cv[bj][q][bi] = C[(ic < wr ? ic : 0) + (long)(jc < wc ? jc : 0) * p.lda];
			}
	sa_d4 acc[2][2];
	accumulate(p, operand(p.A, p.lda, 64 * i + i0, p.n - 1), operand(p.A, p.lda, 64 * l + j0, p.n - 1), p.rowl(i),
	           p.rowl(l), 0, j, acc);
#pragma unroll
	for (int bj = 0; bj < 2; bj++)
#pragma unroll
		for (int q = 0; q < 4; q++)
#pragma unroll
			for (int bi = 0; bi < 2; bi++) {
				const int ic = i0 + 16 * bi + r, jc = j0 + 16 * bj + 4 * q + g;
				if (ic < wr && jc < wc && (l != i || ic >= jc))
					C[ic + (long)jc * p.lda] = cv[bj][q][bi] - acc[bj][bi][q];
			}
	publish(l == i ? p.diag(i) : p.sub(j), 1u);
}

// T = C - sum in LDS, for P and (C = 0) WX; columns from wc on are zero.
__device__ __forceinline__ void stage_block(const double (&cv)[2][4][2], const sa_d4 (&acc)[2][2], int wc, double *T)
{
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	const int i0 = 32 * (wave & 1), j0 = 32 * (wave >> 1);
#pragma unroll
	for (int bj = 0; bj < 2; bj++)
#pragma unroll
		for (int q = 0; q < 4; q++)
#pragma unroll
			for (int bi = 0; bi < 2; bi++) {
				const int ic = i0 + 16 * bi + r, jc = j0 + 16 * bj + 4 * q + g;
				T[ic + jc * LD] = jc < wc ? cv[bj][q][bi] - acc[bj][bi][q] : 0.0;
			}
	__syncthreads();
}

__device__ __noinline__ void item_P(const PfArgs &p, int i, int j, double *T)
{
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	const int i0 = 32 * (wave & 1), j0 = 32 * (wave >> 1);
	const int wr = bw(p, i);            // block column j < i is full
	sa_gd *C = p.A + 64 * i + 64L * j * p.lda;
	double cv[2][4][2];
#pragma unroll
	for (int bj = 0; bj < 2; bj++)
#pragma unroll
		for (int q = 0; q < 4; q++)
#pragma unroll
			for (int bi = 0; bi < 2; bi++) {
				const int ic = i0 + 16 * bi + r, jc = j0 + 16 * bj + 4 * q + g;
				cv[bj][q][bi] = C[(ic < wr ? ic : 0) + (long)jc * p.lda];
			}
	sa_d4 acc[2][2];
	accumulate(p, operand(p.A, p.lda, 64 * i + i0, p.n - 1), operand(p.A, p.lda, 64 * j + j0, p.n - 1), p.rowl(i),
	           p.rowl(j), 0, j, acc);
	stage_block(cv, acc, 64, T);
	await(p, p.dfin(j), p.dfin(j), 1);
	sa_d4 x[4];
	apply_inv(T, p.Dinv + 4096L * j, 64, x);
	const int row = 16 * wave + r;
	if (row < wr)
#pragma unroll
		for (int cb = 0; cb < 4; cb++)
#pragma unroll
			for (int q = 0; q < 4; q++)
				C[row + (long)(16 * cb + 4 * q + g) * p.lda] = x[cb][q];
	publish(p.rowl(i), (unsigned)j + 1);
}

// The inverse of diagonal block j of a tile that is factored already.
__device__ __noinline__ void item_D(const PfArgs &p, int j, double *S, double *Li)
{
	block_potrf_inv64<false>(bw(p, j), (double *)(p.A + 64 * j + 64L * j * p.lda), p.lda, (double *)(p.Dinv + 4096L * j), S,
	                         Li);
	publish(p.dfin(j), 1u);
}

// ---- inverse items ---------------------------------------------------------

// W(t,t) = inv(L(t,t))^T (upper; zero below the diagonal) and Linv(t,t) =
// inv(L(t,t)) (lower; zero above), from the block inverse D(t) formed.
__device__ __noinline__ void item_WD(const PfArgs &p, int t)
{
	await(p, p.dfin(t), p.dfin(t), 1);
	const int w = bw(p, t);
	const sa_gd *D = p.Dinv + 4096L * t;
	sa_gd *Wb = p.W + 64 * t + 64L * t * p.ldw;
	double u[16], v[16];
#pragma unroll
	for (int q = 0; q < 16; q++) {
		const int i = b64_i(q), j = b64_j(q);
		u[q] = D[j + 64 * i];
		v[q] = D[i + 64 * j];
	}
#pragma unroll
	for (int q = 0; q < 16; q++) {
		const int i = b64_i(q), j = b64_j(q);
		if (i < w && j < w) {
			Wb[i + (long)j * p.ldw] = i <= j ? u[q] : 0.0;
			if (p.Linv)
				p.Linv[(64 * t + i) + (64L * t + j) * p.ldi] = i >= j ? v[q] : 0.0;
		}
	}
	publish(p.roww(t), (unsigned)t + 1);
}

// W(j,i) for j < i: the sum of W(j,t) L(i,t)^T over t = j..i-1 in registers,
// then W(j,i) = -sum inv(L(i,i))^T, with Linv(i,j) = W(j,i)^T; the mirrored
// blocks W(i,j) and Linv(j,i) are zero.
__device__ __noinline__ void item_WX(const PfArgs &p, int j, int i, double *T, double *X)
{
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	const int i0 = 32 * (wave & 1), j0 = 32 * (wave >> 1);
	const int wc = bw(p, i);            // block row j < i is full
	sa_d4 acc[2][2];
	accumulate(p, operand(p.W, p.ldw, 64 * j + i0, p.n - 1), operand(p.A, p.lda, 64 * i + j0, p.n - 1), p.roww(j),
	           p.rowl(i), j, i, acc);
	const double zero[2][4][2] = {};
	stage_block(zero, acc, wc, T);
	await(p, p.dfin(i), p.dfin(i), 1);
	sa_d4 x[4];
	apply_inv(T, p.Dinv + 4096L * i, 64, x);
	const int row = 16 * wave + r;
	sa_gd *Wb = p.W + 64 * j + 64L * i * p.ldw;
#pragma unroll
	for (int cb = 0; cb < 4; cb++)
#pragma unroll
		for (int q = 0; q < 4; q++) {
			const int c = 16 * cb + 4 * q + g;
			if (c < wc)
				Wb[row + (long)c * p.ldw] = x[cb][q];
			if (p.Linv)
				X[c + row * LD] = x[cb][q];
		}
	publish(p.roww(j), (unsigned)i + 1);
	for (int q = 0; q < 16; q++) {
		const int a = b64_i(q), c = b64_j(q);
		if (a < wc)
			p.W[(64 * i + a) + (64L * j + c) * p.ldw] = 0.0;
		if (p.Linv) {
			if (a < wc)
				p.Linv[(64 * i + a) + (64L * j + c) * p.ldi] = X[a + c * LD];
			if (c < wc)
				p.Linv[(64 * j + a) + (64L * i + c) * p.ldi] = 0.0;
		}
	}
}

// ---- the critical chain ----------------------------------------------------

// Step j: S (LDS) holds A(j,j) with all its updates.  The block is factored
// and inverted in LDS and its inverse published; L(j+1,j) is formed from the
// prepared A(j+1,j) and the inverse in LDS, published, and kept in LDS for
// the last update of A(j+1,j+1), which becomes the next S.
__device__ __forceinline__ void run_chain(const PfArgs &p, double *S, double *Li)
{
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	int first_bad = 0;
	if (p.nb > 0)
		block_load64<double>(bw(p, 0), (double *)p.A, p.lda, S, Li);
	for (int j = 0; j < p.nb; j++) {
		const int wj = bw(p, j);
		const int bad = block_core64<double, true>(S, Li);
		if (threadIdx.x == 0 && bad && bad <= wj && first_bad == 0)
			first_bad = 64 * j + bad;
		store_inv64<double>(Li, (double *)(p.Dinv + 4096L * j));
		store_lower64<double>(wj, S, (double *)(p.A + 64 * j + 64L * j * p.lda), p.lda);
		if (j + 1 == p.nb) {
			if (threadIdx.x == 0)
				*p.info = first_bad;     // in memory once D(j) is published
			publish(p.dfin(j), 1u);
			break;
		}
		const int wn = bw(p, j + 1);
		sa_gd *P = p.A + 64 * (j + 1) + 64L * j * p.lda, *C = p.A + 64 * (j + 1) + 64L * (j + 1) * p.lda;
		// the wave's 16 rows of A(j+1,j), and its blocks of the lower half of
		// A(j+1,j+1): 16x16 blocks 4u + wave of the ten, row by row
		const int row = 16 * wave + r, rowc = row < wn ? row : wn - 1;
		double t[16], cv[3][4];
		auto load_next = [&] {
#pragma unroll
			for (int s = 0; s < 16; s++)
				t[s] = P[rowc + (long)(4 * s + g) * p.lda];
#pragma unroll
			for (int u = 0; u < 3; u++) {
				const int b = 4 * u + wave, I = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, K = b - I * (I + 1) / 2;
#pragma unroll
				for (int q = 0; q < 4; q++) {
					const int ic = 16 * I + r, jc = 16 * K + 4 * q + g;
					cv[u][q] = (b < 10 && ic < wn && jc < wn) ? C[ic + (long)jc * p.lda] : 0.0;
				}
			}
		};
		// they are mostly there by now: one look while the inverse is on its
		// way to memory, and the loads in flight while it is published
		const unsigned ra = flag_read(p.sub(j)), rb = flag_read(p.diag(j + 1));
		const bool there = __builtin_amdgcn_readfirstlane((int)(ra & rb)) != 0;
		if (there) {
			__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
			load_next();
		}
		publish(p.dfin(j), 1u);
		if (!there) {
			await(p, p.sub(j), p.diag(j + 1), 1);
			load_next();
		}
		sa_d4 x[4];
#pragma unroll
		for (int cb = 0; cb < 4; cb++)
			x[cb] = sa_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
		for (int s = 0; s < 16; s++)
#pragma unroll
			for (int cb = 0; cb < 4; cb++)
				if (s < 4 * (cb + 1))
					x[cb] = sa_mfma(Li[(16 * cb + r) + (4 * s + g) * LD], t[s], x[cb]);
		__syncthreads();                 // L(j,j) has left S
#pragma unroll
		for (int cb = 0; cb < 4; cb++)
#pragma unroll
			for (int q = 0; q < 4; q++) {
				const int c = 16 * cb + 4 * q + g;
				S[row + c * LD] = x[cb][q];
				if (row < wn)
					P[row + (long)c * p.lda] = x[cb][q];
			}
		__syncthreads();                 // S is whole
		sa_d4 acc[3];
#pragma unroll
		for (int u = 0; u < 3; u++) {
			const int b = 4 * u + wave, I = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, K = b - I * (I + 1) / 2;
			acc[u] = sa_d4{0.0, 0.0, 0.0, 0.0};
			if (b < 10)
#pragma unroll
				for (int s = 0; s < 16; s++)
					acc[u] = sa_mfma(S[16 * K + r + (4 * s + g) * LD], S[16 * I + r + (4 * s + g) * LD], acc[u]);
		}
		publish(p.rowl(j + 1), (unsigned)j + 1);     // with a barrier: L(j+1,j) has left S
#pragma unroll
		for (int u = 0; u < 3; u++) {
			const int b = 4 * u + wave, I = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, K = b - I * (I + 1) / 2;
			if (b < 10)
#pragma unroll
				for (int q = 0; q < 4; q++) {
					const int ic = 16 * I + r, jc = 16 * K + 4 * q + g;
					S[ic + jc * LD] = (ic < wn && jc < wn) ? cv[u][q] - acc[u][q] : ic == jc ? 1.0 : 0.0;
				}
		}
		__syncthreads();
	}
	if (threadIdx.x == 0) {
		if (p.nb == 0)
			*p.info = 0;
		else if (abort_or(p, ABORT_REPORTED) & ABORT_GAVE_UP)
			*p.info = -1;
	}
}

// ---- the bulk order --------------------------------------------------------
// Step s: S(s) and G(s) (1 <= s < nb - 1), P(a, s) for a = s+2..nb-1
// (factorisation, s < nb), then for t = s - delay: WD(t), WX(a, t) for a < t
// (inverse).  Without the factorisation, step 0 starts with D(a), a < nb.
// Host and device walk it with the same code (the host counts the items).

enum { PH_D = 0, PH_S, PH_G, PH_P, PH_WD, PH_WX, PH_END };

struct PfOrder {
	int nb, factor, inv, delay;
};

struct Cursor {
	int s, ph, a;
};

// First a of a phase of step s, and the one after its last (none if not above).
__host__ __device__ inline int phase_first(const PfOrder &, int s, int ph) { return ph == PH_P ? s + 2 : 0; }

__host__ __device__ inline int phase_last(const PfOrder &o, int s, int ph)
{
	const int t = s - o.delay;
	switch (ph) {
	case PH_D:
		return !o.factor && s == 0 ? o.nb : 0;
	case PH_S:
	case PH_G:
		return o.factor && s >= 1 && s + 1 < o.nb ? 1 : 0;
	case PH_P:
		return o.factor ? o.nb : 0;
	case PH_WD:
		return o.inv && t >= 0 && t < o.nb ? 1 : 0;
	default:
		return o.inv && t < o.nb ? t : 0;
	}
}

// Moves c to the first item at or after its position; false past the end.
__host__ __device__ inline bool cursor_norm(Cursor &c, const PfOrder &o)
{
	const int last = o.nb - 1 + (o.factor && o.inv ? o.delay : 0);
	while (c.s <= last) {
		if (c.a < phase_last(o, c.s, c.ph))
			return true;
		if (++c.ph >= PH_END) {
			c.s++;
			c.ph = 0;
		}
		c.a = phase_first(o, c.s, c.ph);
	}
	return false;
}

__host__ __device__ inline Cursor cursor_first(const PfOrder &o, bool *valid)
{
	Cursor c = {0, 0, 0};
	*valid = cursor_norm(c, o);
	return c;
}

// The bulk workgroups take items in the bulk order from a shared ticket
// counter: whichever workgroup is free takes the next item, so an item is
// never queued behind another workgroup's unrelated work.  Tickets only grow
// and every item waits only for items earlier in the order, so the earliest
// unfinished item is always held by a running workgroup with its inputs
// ready; an item not yet handed out blocks nobody.
__device__ __forceinline__ void run_bulk(const PfArgs &p, double *S, double *Li, int *s_ticket)
{
	const PfOrder o = {p.nb, p.factor, p.inv, p.delay};
	bool valid;
	Cursor c = cursor_first(o, &valid);
	int pos = 0;
	for (;;) {
		__syncthreads();                  // the last item's reads of LDS are done
		if (threadIdx.x == 0)
			*s_ticket = (int)__hip_atomic_fetch_add(p.ticket(), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		__syncthreads();
		const int t = *s_ticket;
		while (valid && pos < t) {
			c.a++;
			valid = cursor_norm(c, o);
			pos++;
		}
		if (!valid)
			break;                        // past the last item: this workgroup is done
		switch (c.ph) {
		case PH_D:
			item_D(p, c.a, S, Li);
			break;
		case PH_S:
			item_prepare(p, c.s, c.s);
			break;
		case PH_G:
			item_prepare(p, c.s, c.s + 1);
			break;
		case PH_P:
			item_P(p, c.a, c.s, S);
			break;
		case PH_WD:
			item_WD(p, c.s - p.delay);
			break;
		default:
			item_WX(p, c.a, c.s - p.delay, S, Li);
			break;
		}
	}
}

__global__ __launch_bounds__(256)
void k_potrf_tile(PfArgs p)
{
	__shared__ double S[64 * LD];
	__shared__ double Li[64 * LD];
	__shared__ int s_ticket;
	if (p.factor && blockIdx.x == 0)
		run_chain(p, S, Li);
	else
		run_bulk(p, S, Li, &s_ticket);
}

// Counters of a launch.  When the tile is factored already, every row of L
// is final.  Nothing has to be prepared for A(1,0) and A(1,1).  A kernel, not
// a memset, so that a captured graph replays it correctly.
__global__ void k_init_counters(unsigned *flags, int nb, int factor)
{
	for (int idx = threadIdx.x; idx < flag_words(nb); idx += blockDim.x) {
		const int b = idx / FLAG_STRIDE;
		unsigned v = 0u;
		if (idx % FLAG_STRIDE == 0 && nb > 1) {     // one block: nothing waits
			if (b < nb)
				v = factor ? 0u : (unsigned)nb;     // rows of L
			else if (b == nb + 1 || b == 2 * nb)
				v = 1u;                             // diag(1), sub(0)
		}
		flags[idx] = v;
	}
}

constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Workspace of a tile: the 64x64 block inverses and the counters.
constexpr size_t tile_bytes(int n)
{
	return align256((size_t)(n > 0 ? (n + 63) / 64 : 1) * 4096 * sizeof(double)) +
	       align256((size_t)flag_words(n > 0 ? (n + 63) / 64 : 1) * sizeof(unsigned));
}

long count_items(const PfOrder &o)
{
	bool valid;
	Cursor c = cursor_first(o, &valid);
	long k = 0;
	while (valid) {
		k++;
		c.a++;
		valid = cursor_norm(c, o);
	}
	return k;
}

// factor: A is factored in place (info receives the pivot report); else A
// holds the factor.  W (and Linv, optional) receive the inverse when W is
// given.  bulk: workgroups for the bulk items (<= 0: max_bulk()).
int launch_tile(hipStream_t s, int n, double *A, int lda, int *dev_info, void *work, double *W, int ldw,
                double *Linv, int ldi, int factor, int bulk = 0, unsigned stop = ABORT_GAVE_UP)
{
	const int nb = n > 0 ? (n + 63) / 64 : 0;
	char *ws = (char *)work;
	PfArgs p;
	p.n = n;
	p.nb = nb;
	p.factor = factor;
	p.inv = W != nullptr;
	p.delay = factor ? 1 : 0;
	p.A = (sa_gd *)A;
	p.lda = lda;
	p.W = (sa_gd *)W;
	p.ldw = ldw;
	p.Linv = (sa_gd *)Linv;
	p.ldi = ldi;
	p.Dinv = (sa_gd *)ws;
	p.flags = (sa_gu *)(ws + align256((size_t)(nb ? nb : 1) * 4096 * sizeof(double)));
	p.stop = stop;
	p.info = dev_info;
	if (nb == 0) {
		if (!factor)
			return 0;
		// n = 0: reports info = 0
		p.nbulk = 0;
		hipLaunchKernelGGL(k_init_counters, dim3(1), dim3(64), 0, s, (unsigned *)p.flags, 1, 1);
		int e = sa_launch_status();
		if (e)
			return e;
		hipLaunchKernelGGL(k_potrf_tile, dim3(1), dim3(256), 0, s, p);
		return sa_launch_status();
	}
	const long items = count_items(PfOrder{nb, factor, p.inv, p.delay});
	const int want = bulk > 0 ? (bulk < 255 ? bulk : 255) : max_bulk();
	p.nbulk = (int)(items < want ? items : want);
	hipLaunchKernelGGL(k_init_counters, dim3(1), dim3(256), 0, s, (unsigned *)p.flags, nb, factor);
	int e = sa_launch_status();
	if (e)
		return e;
	const int grid = (factor ? 1 : 0) + p.nbulk;
	if (grid == 0)
		return 0;
	hipLaunchKernelGGL(k_potrf_tile, dim3((unsigned)grid), dim3(256), 0, s, p);
	return sa_launch_status();
}

} // namespace

// Workspace: the block inverses and the counters, or for tiles past the
// single-launch limit the substitution inverse's.
extern "C" size_t sa_dpotrf_tile_worksize(int n)
{
	if (n <= PF_MAXN)
		return tile_bytes(n);
	return sa_dtrtri_lt_worksize(n);
}

extern "C" int sa_dpotrf_tile_maxn(void) { return PF_MAXN; }

static int potrf_tile(hipStream_t s, int n, double *A, int lda, double *Linv, int ldl, double *W, int ldw,
                      int *dev_info, void *work, size_t work_bytes, int workgroups, unsigned stop)
{
	if (n < 0 || n > PF_MAXN || lda < (n > 1 ? n : 1) || !dev_info || !work ||
	    work_bytes < sa_dpotrf_tile_worksize(n) || (Linv && !W) ||
	    (W && ldw < (n > 1 ? n : 1)) || (Linv && ldl < (n > 1 ? n : 1)))
		return -EINVAL;
	return launch_tile(s, n, A, lda, dev_info, work, W, ldw, Linv, ldl, 1, workgroups, stop);
}

extern "C" int sa_dpotrf_tile_wg(hipStream_t s, int n, double *A, int lda, double *Linv, int ldl, double *W,
                                 int ldw, int *dev_info, void *work, size_t work_bytes, int workgroups)
{
	return potrf_tile(s, n, A, lda, Linv, ldl, W, ldw, dev_info, work, work_bytes, workgroups, ABORT_GAVE_UP);
}

extern "C" int sa_dpotrf_tile_cut(hipStream_t s, int n, double *A, int lda, double *Linv, int ldl, double *W,
                                  int ldw, int *dev_info, void *work, size_t work_bytes, int workgroups)
{
	return potrf_tile(s, n, A, lda, Linv, ldl, W, ldw, dev_info, work, work_bytes, workgroups,
	                  ABORT_GAVE_UP | ABORT_REPORTED);
}

extern "C" int sa_dpotrf_tile(hipStream_t s, int n, double *A, int lda, double *Linv, int ldl, double *W, int ldw,
                              int *dev_info, void *work, size_t work_bytes)
{
	return sa_dpotrf_tile_wg(s, n, A, lda, Linv, ldl, W, ldw, dev_info, work, work_bytes, 0);
}

extern "C" int sa_dtrtri_tile(hipStream_t s, int n, const double *L, int ldl, double *Linv, int ldx, double *W,
                              int ldw, void *work, size_t work_bytes)
{
	if (n < 0 || ldl < (n > 1 ? n : 1) || !Linv || !W || ldx < (n > 1 ? n : 1) || ldw < (n > 1 ? n : 1) ||
	    !work || work_bytes < sa_dpotrf_tile_worksize(n > 0 ? n : 1))
		return -EINVAL;
	if (n == 0)
		return 0;
	if (n <= PF_MAXN)
		return launch_tile(s, n, const_cast<double *>(L), ldl, nullptr, work, W, ldw, Linv, ldx, 0);
	int e = sa_dtrtri_lt(s, n, L, ldl, W, ldw, work, work_bytes);
	return e ? e : sa_dtranspose(s, n, n, W, ldw, Linv, ldx);
}

// ---------------------------------------------------------------------------
// Allocation-free tile factorisation (sa_dpotrf_tile_noalloc).  Its
// workspace -- the 64x64 block inverses and the counters of the largest
// tile accepted -- is this file-scope device array: each GPU the library
// runs on holds one copy until the process ends.  Host code never passes
// `scratch` itself to a kernel (on the host the name is only a stand-in);
// it uses the device address hipGetSymbolAddress returns, looked up once per
// device.  Overlapping calls on one GPU share the array and race; the
// counters are cleared by a kernel (k_init_counters) before every
// factorisation, so a call does not depend on what the previous one left
// there.

constexpr int NOALLOC_MAXN = PF_MAXN;
constexpr size_t NOALLOC_BYTES = tile_bytes(NOALLOC_MAXN);
constexpr int NOALLOC_MAXDEV = 64;

static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

static std::mutex g_scratch_mu;
static void *g_scratch_dev[NOALLOC_MAXDEV];

// Device address of `scratch` on the current device (looked up on the first
// call per device), or null.
static void *scratch_address(int *err)
{
	int dev = -1;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess || dev < 0 || dev >= NOALLOC_MAXDEV) {
		*err = e != hipSuccess ? (int)e : -ENODEV;
		return nullptr;
	}
	std::lock_guard<std::mutex> lock(g_scratch_mu);
	if (!g_scratch_dev[dev]) {
		void *p = nullptr;
		e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
		if (e != hipSuccess || !p) {
			*err = e != hipSuccess ? (int)e : -ENODEV;
			return nullptr;
		}
		g_scratch_dev[dev] = p;
	}
	return g_scratch_dev[dev];
}

extern "C" int sa_dpotrf_tile_noalloc_maxn(void) { return NOALLOC_MAXN; }

extern "C" int sa_dpotrf_tile_noalloc(hipStream_t s, int n, double *A, int lda, double *Linv, int ldl, double *W,
                                      int ldw, int *dev_info)
{
	if (n > NOALLOC_MAXN || sa_dpotrf_tile_worksize(n) > NOALLOC_BYTES)
		return -EOVERFLOW;
	int err = 0;
	void *ws = scratch_address(&err);
	if (!ws)
		return err;
	return sa_dpotrf_tile(s, n, A, lda, Linv, ldl, W, ldw, dev_info, ws, NOALLOC_BYTES);
}
