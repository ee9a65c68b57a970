// Device building blocks on 64x64 diagonal blocks of a lower Cholesky
// factor (gfx950): 16x16 register Cholesky and inverse, 16x16x16 MFMA
// block products on LDS operands, the factor-and-invert of one 64x64 block
// by a 256-thread workgroup, and the application of a block inverse to a
// panel.  Shared by the tile kernels (sa_chol.hip, sa_potrf.hip) and the
// batched persistent kernels (sa_batched.hip).
//
// Everything is a template on the element type T (double or float).  The
// FP32 and FP64 16x16x4 MFMAs read their operands alike (lane l supplies
// A(l%16, k) and B(k, l%16) for k = l/16 of the step) but return the 16x16
// result in different orders: register q of lane l holds row 4q + l/16
// (FP64) or row 4(l/16) + q (FP32) of column l%16 -- drow<T> below.  The
// double-named entry points at the end keep the FP64 interface of the
// callers.
#ifndef SA_BLOCK64_H
#define SA_BLOCK64_H

#include "sa_common.h"

namespace sa64 {

constexpr int LD = 65;      // LDS leading dimension of a 64x64 block (bank spread)

template <typename T> struct V4;
template <> struct V4<double> { typedef sa_d4 type; };
template <> struct V4<float> { typedef sa_f4 type; };

// v_mfma_f32_16x16x4f32: the lane layout of sa_mfma's FP64 form.
using ::sa_mfma;
__device__ __forceinline__ sa_f4 sa_mfma(float a, float b, sa_f4 c)
{
	return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Row of the 16x16 MFMA result held in register q of the lanes of group g
// (g = lane / 16; the column is lane % 16).
template <typename T> __device__ __forceinline__ constexpr int drow(int q, int g);
template <> __device__ __forceinline__ constexpr int drow<double>(int q, int g) { return 4 * q + g; }
template <> __device__ __forceinline__ constexpr int drow<float>(int q, int g) { return 4 * g + q; }

template <typename T>
__device__ __forceinline__ typename V4<T>::type zero4()
{
	return typename V4<T>::type{T(0), T(0), T(0), T(0)};
}

// v of lane K of each 16-lane row, broadcast to the whole row with the DPP
// row_newbcast mode (a VALU move: no SGPR round trip as with v_readlane).
template <int K>
__device__ __forceinline__ double rb(double v)
{
	const long long bits = __double_as_longlong(v);
	const int lo = __builtin_amdgcn_update_dpp(0, (int)(bits & 0xffffffffll), 0x150 + K, 0xf, 0xf, false);
	const int hi = __builtin_amdgcn_update_dpp(0, (int)(bits >> 32), 0x150 + K, 0xf, 0xf, false);
	return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int K>
__device__ __forceinline__ float rb(float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xf, 0xf, false));
}

// v of lane `lane` (< 16) broadcast to the whole wave through SGPRs.
__device__ __forceinline__ double bcast_rl(double v, int lane)
{
	const long long bits = __double_as_longlong(v);
	const int lo = __builtin_amdgcn_readlane((int)(bits & 0xffffffffll), lane);
	const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), lane);
	return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ float bcast_rl(float v, int lane)
{
	return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// k is a compile-time constant wherever this is called from fully unrolled
// loops, so the switch folds to one broadcast.
template <typename T>
__device__ __forceinline__ T bcast(T v, int k)
{
	switch (k) {
	case 0: return rb<0>(v);
	case 1: return rb<1>(v);
	case 2: return rb<2>(v);
	case 3: return rb<3>(v);
	case 4: return rb<4>(v);
	case 5: return rb<5>(v);
	case 6: return rb<6>(v);
	case 7: return rb<7>(v);
	case 8: return rb<8>(v);
	case 9: return rb<9>(v);
	case 10: return rb<10>(v);
	case 11: return rb<11>(v);
	case 12: return rb<12>(v);
	case 13: return rb<13>(v);
	case 14: return rb<14>(v);
	default: return rb<15>(v);
	}
}

// 16x16 block products on LDS operands (block origins, leading dimension LD).
// The result is in MFMA output layout: register q of lane l holds element
// (drow<T>(q, l/16), l%16).
template <typename T>
__device__ __forceinline__ typename V4<T>::type mm16_nt(const T *A, const T *B, typename V4<T>::type acc, T sign)
{
	const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
#pragma unroll
	for (int s = 0; s < 4; s++)
		acc = sa_mfma(sign * A[r + (4 * s + g) * LD], B[r + (4 * s + g) * LD], acc);
	return acc;
}

template <typename T>
__device__ __forceinline__ typename V4<T>::type mm16_nn(const T *A, const T *B, typename V4<T>::type acc)
{
	const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
#pragma unroll
	for (int s = 0; s < 4; s++)
		acc = sa_mfma(A[r + (4 * s + g) * LD], B[(4 * s + g) + r * LD], acc);
	return acc;
}

// acc += A * T with T a 16x16 block already in MFMA output layout: register
// s of lane l holds T(k, l%16) with k = drow<T>(s, l/16), so k-step s takes
// Tb[s] as its B operand and A(l%16, k) as its A operand (the 16 k values
// are covered once over the four steps, in a permuted order for FP32).
template <typename T>
__device__ __forceinline__ typename V4<T>::type mm16_nreg(const T *A, typename V4<T>::type Tb,
                                                          typename V4<T>::type acc)
{
	const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
#pragma unroll
	for (int s = 0; s < 4; s++)
		acc = sa_mfma(A[r + drow<T>(s, g) * LD], Tb[s], acc);
	return acc;
}

template <typename T>
__device__ __forceinline__ void st16(T *P, typename V4<T>::type acc, T sign)
{
	const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
#pragma unroll
	for (int q = 0; q < 4; q++)
		P[drow<T>(q, g) + r * LD] = sign * acc[q];
}

template <typename T>
__device__ __forceinline__ typename V4<T>::type ld16(const T *P)
{
	const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
	typename V4<T>::type acc;
#pragma unroll
	for (int q = 0; q < 4; q++)
		acc[q] = P[drow<T>(q, g) + r * LD];
	return acc;
}

// The hardware estimate r of 1/sqrt(d) (about 24 bits in either type) and
// e = 1 - d r^2, from which both of a column's scalings come to full
// precision: 1/sqrt(d), for double by a third-order step
// r + r e (1/2 + 3/8 e), whose error is of order e^3, for float by a Newton
// step; and x / d = x r^2 / (1 - e), for double x r^2 (1 + e + e^2), for
// float x r^2 (1 + e).  x r is formed first: |x| <= sqrt(d a) for a the
// diagonal entry of x's row, so it stays in range, and x r^2 as long as
// sqrt(a / d) does, which only a subnormal d can break.  1/d does not: it
// overflows for an FP64 pivot below 2^-1024, and from 2^126 on an FP32 one's
// is a subnormal that the reciprocal instruction flushes, which would leave
// the elimination out.
__device__ __forceinline__ double rsqrt_est(double d) { return __builtin_amdgcn_rsq(d); }
__device__ __forceinline__ float rsqrt_est(float d) { return __builtin_amdgcn_rsqf(d); }

__device__ __forceinline__ double rsqrt_err(double d, double r) { return fma(-d * r, r, 1.0); }
__device__ __forceinline__ float rsqrt_err(float d, float r) { return fmaf(-d * r, r, 1.0f); }

__device__ __forceinline__ double rsqrt_nr(double r, double e) { return fma(r * e, fma(0.375, e, 0.5), r); }
__device__ __forceinline__ float rsqrt_nr(float r, float e) { return fmaf(r, 0.5f * e, r); }

__device__ __forceinline__ double quot_nr(double x, double r, double e)
{
	const double x0 = x * r * r;
	return fma(x0, fma(e, e, e), x0);
}

__device__ __forceinline__ float quot_nr(float x, float r, float e)
{
	const float x0 = x * r * r;
	return fmaf(x0, e, x0);
}

// Lane t < 16 holds row t of a 16x16 lower block in x[0..15] (columns
// above the diagonal are ignored), lanes 16..63 up to 48 rows of the panel
// below it.  In-place Cholesky of the block, the panel rows solved against
// it on the way (the other lanes run the same instructions anyway); returns
// the 1-based index of the first non-positive pivot, or 0.  The chain from
// one pivot d to the next is kept short: the columns to the right take
// x_j -= (x_k / d) x_jk with the unscaled multipliers x_jk, which are
// broadcast while the quotient is formed; the column itself is scaled by
// d^{-1/2} off that chain and handed to done(k, column).  The broadcasts are
// v_readlane: the row-broadcast DPP form reaches only the lanes of one
// 16-lane row.
template <typename T, typename F>
__device__ __forceinline__ int potrf16_regs(T (&x)[16], F done)
{
	unsigned long long bad = 0;
#pragma unroll
	for (int k = 0; k < 16; k++) {
		const T d = bcast_rl(x[k], k);
		const T r = rsqrt_est(d);
		__builtin_amdgcn_sched_barrier(0);
		// all multipliers of the column in scalar registers, behind the
		// estimate's latency and before the first is used: a readlane's
		// result may not be read at once
		T m[16];
#pragma unroll
		for (int j = k + 1; j < 16; j++)
			m[j] = bcast_rl(x[k], j);
		const T e = rsqrt_err(d, r), z = quot_nr(x[k], r, e);
		bad |= __ballot(!(x[k] > T(0))) & (1ull << k);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int j = k + 1; j < 16; j++)
			x[j] -= z * m[j];
		x[k] *= rsqrt_nr(r, e);
		done(k, x[k]);
	}
	return __ffsll((long long)bad);
}

// LDS written by other lanes of the same wave is read next: keep the order.
__device__ __forceinline__ void wave_lds_order()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inverse of the factored 16x16 lower diagonal block J of S into the same
// block of Li (zeros above its diagonal), by one wave.  The two 8x8 diagonal
// halves first, lane c (mod 16) taking column c of the one it falls in: one
// division per lane, all lanes at once, then the columns of L from left to
// right, y_q = s_q / L(q,q), s_i -= L(i,q) y_q for i > q (L from LDS, each
// half's element a broadcast).  Then the block below by two 16x16x16 MFMA
// products with everything but the needed quarter zero: -C^{-1} (B A^{-1}).
// Half the chain and a quarter of the multiply-adds of sixteen columns in
// one.  The block may just have been factored or loaded: the inverse has the
// same bits.
template <typename T>
__device__ __forceinline__ void inv16(const T *S, int J, T *Li)
{
	typedef typename V4<T>::type V;
	const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, c = r & 7, h = r & 8;
	const T *B = S + 16 * J + 16 * J * LD;
	const T *H = B + h + h * LD;
	T *I = Li + 16 * J + 16 * J * LD;
	const T rd = T(1) / H[c + c * LD];
	T y[8];
#pragma unroll
	for (int i = 0; i < 8; i++)
		y[i] = (c == i) ? T(1) : T(0);
#pragma unroll
	for (int q = 0; q < 8; q++) {
		const T lo = bcast(rd, q), hi = bcast(rd, q + 8);
		y[q] *= h ? hi : lo;
#pragma unroll
		for (int i = q + 1; i < 8; i++)
			y[i] -= H[i + q * LD] * y[q];
	}
	// column r of the block: its half's rows, zero in the other half's
	if (lane < 16)
#pragma unroll
		for (int i = 0; i < 8; i++) {
			I[i + r * LD] = h ? T(0) : y[i];
			I[8 + i + r * LD] = h ? y[i] : T(0);
		}
	wave_lds_order();
	V t = zero4<T>();
#pragma unroll
	for (int s = 0; s < 4; s++) {
		const int k = 4 * s + g;
		const T b = B[r + k * LD];
		t = sa_mfma(r >= 8 && k < 8 ? b : T(0), I[k + r * LD], t);
	}
	const V x = mm16_nreg(I, t, zero4<T>());
#pragma unroll
	for (int q = 0; q < 4; q++)
		if (drow<T>(q, g) >= 8 && r < 8)
			I[drow<T>(q, g) + r * LD] = -x[q];
}

// sum_{K=J}^{I-1} L_IK Li_KJ, the product that block (I, J) of the inverse
// takes before its scaling by -Li_II, in MFMA output layout.
template <typename T>
__device__ __forceinline__ typename V4<T>::type inv_sum(const T *S, const T *Li, int I, int J)
{
	typename V4<T>::type t = zero4<T>();
	for (int K = J; K < I; K++)
		t = mm16_nn(&S[16 * I + 16 * K * LD], &Li[16 * K + 16 * J * LD], t);
	return t;
}

template <typename T>
__device__ __forceinline__ void inv_scale(T *Li, int I, int J, typename V4<T>::type t)
{
	st16(&Li[16 * I + 16 * J * LD], mm16_nreg(&Li[16 * I + 16 * I * LD], t, zero4<T>()), T(-1));
}

// The w x w lower block D into S, identity past w, zeros above the diagonal;
// Li zeroed.  All 16 loads of a thread are in flight before the first LDS
// store (the block sits in L2; one round trip instead of sixteen).
template <typename T>
__device__ __forceinline__ void block_load64(int w, const T *__restrict__ D, long ldd, T *__restrict__ S,
                                             T *__restrict__ Li)
{
	const int tid = threadIdx.x;
	T v[16];
#pragma unroll
	for (int q = 0; q < 16; q++) {
		const int i = (tid + 256 * q) & 63, j = (tid + 256 * q) >> 6;
		const bool in = i < w && j < w && i >= j;
		const T x = D[(in ? i : 0) + (long)(in ? j : 0) * ldd];
		v[q] = in ? x : ((i == j && (i >= w || j >= w)) ? T(1) : T(0));
	}
#pragma unroll
	for (int q = 0; q < 16; q++) {
		const int i = (tid + 256 * q) & 63, j = (tid + 256 * q) >> 6;
		S[i + j * LD] = v[q];
		Li[i + j * LD] = T(0);
	}
	__syncthreads();
}

// FACTOR: Cholesky of the lower block in S, in place, and its inverse into
// the lower part of Li.  !FACTOR: S holds the factor already; only the
// inverse is formed, with the same bits.  One 256-thread workgroup; S and Li
// are two LDS blocks of 64 * LD elements, Li's blocks of 16 above the
// diagonal zero on entry (they are not written); S above its diagonal is
// neither used nor kept.  Returns, in every thread of wave 0, the 1-based
// column of the first non-positive pivot within the block (or 0); other
// threads return 0.  Ends with a workgroup barrier.
// Bound: the 64 dependent columns.  Wave 0 runs them as four panels of 16
// columns over all the rows below (potrf16_regs), and everything else
// overlaps the next panel: the trailing blocks, the 16x16 inverses and the
// columns of the inverse, one per wave.  Only the update of the next 16
// columns stands between two panels.
template <typename T, bool FACTOR>
__device__ __forceinline__ int block_core64(T *__restrict__ S, T *__restrict__ Li)
{
	typedef typename V4<T>::type V;
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	int bad = 0;
	if (FACTOR) {
		// wave q = 1..3 keeps the sum of the next block of its inverse column
		V t = zero4<T>();
		const int Jc = wave - 1;
		// unrolled: the conditions on J below fold, at the price of four
		// copies of the panel code
#pragma unroll
		for (int J = 0; J < 4; J++) {
			if (wave == 0) {
				// lanes past the block take the padding row 64 of each column, so
				// that no branch breaks up the column loop
				const int row = 16 * J + lane < 64 ? 16 * J + lane : 64;
				T *P = S + row + 16 * J * LD;
				T x[16];
#pragma unroll
				for (int c = 0; c < 16; c++)
					x[c] = P[c * LD];
				// the diagonal block's upper half, which nothing reads, receives
				// what the elimination leaves there
				const int b = potrf16_regs(x, [&](int c, T v) { P[c * LD] = v; });
				if (b && !bad)
					bad = 16 * J + b;
			} else if (J > 0) {
				// trailing blocks right of column block J, by column block J - 1
				int p = 0;
				for (int K = J + 1; K < 4; K++)
					for (int I = K; I < 4; I++, p++)
						if (p % 3 == wave - 1) {
							V acc = ld16(&S[16 * I + 16 * K * LD]);
							acc = mm16_nt(&S[16 * I + 16 * (J - 1) * LD], &S[16 * K + 16 * (J - 1) * LD], acc, T(-1));
							st16(&S[16 * I + 16 * K * LD], acc, T(1));
						}
				// inverse: row J - 2 of the column is scaled now that Li(J-2,J-2)
				// is there, then the sum for row J - 1; Li(J-1,J-1)
				if (wave == 3)
					inv16(S, J - 1, Li);
				if (Jc < J - 2)
					inv_scale(Li, J - 2, Jc, t);
				if (Jc < J - 1) {
					wave_lds_order();
					t = inv_sum(S, Li, J - 1, Jc);
				}
			}
			__syncthreads();
			// column block J + 1 by the panel just factored
			if (wave < 3 - J) {
				const int I = J + 1 + wave;
				V acc = ld16(&S[16 * I + 16 * (J + 1) * LD]);
				acc = mm16_nt(&S[16 * I + 16 * J * LD], &S[16 * (J + 1) + 16 * J * LD], acc, T(-1));
				st16(&S[16 * I + 16 * (J + 1) * LD], acc, T(1));
			}
			if (J < 3)
				__syncthreads();
		}
		if (wave == 0) {
			inv16(S, 3, Li);
		} else {
			if (Jc < 2)
				inv_scale(Li, 2, Jc, t);
			wave_lds_order();
			t = inv_sum(S, Li, 3, Jc);
		}
		__syncthreads();
		if (wave > 0)
			inv_scale(Li, 3, Jc, t);
	} else {
		inv16(S, wave, Li);
		__syncthreads();
		if (wave > 0)
			for (int I = wave; I < 4; I++) {
				inv_scale(Li, I, wave - 1, inv_sum(S, Li, I, wave - 1));
				wave_lds_order();
			}
	}
	__syncthreads();
	return bad;
}

// Element (i, j) and its index in an LDS block for item q of 16 of a thread.
__device__ __forceinline__ int b64_i(int q) { return (threadIdx.x + 256 * q) & 63; }
__device__ __forceinline__ int b64_j(int q) { return (threadIdx.x + 256 * q) >> 6; }

// Lower part of S into D (w x w), LDS reads of a thread ahead of its stores.
template <typename T>
__device__ __forceinline__ void store_lower64(int w, const T *__restrict__ S, T *__restrict__ D, long ldd)
{
	T o[16];
#pragma unroll
	for (int q = 0; q < 16; q++)
		o[q] = S[b64_i(q) + b64_j(q) * LD];
#pragma unroll
	for (int q = 0; q < 16; q++) {
		const int i = b64_i(q), j = b64_j(q);
		if (i < w && j < w && i >= j)
			D[i + (long)j * ldd] = o[q];
	}
}

// Li into Dinv (64 x 64, ld 64).
template <typename T>
__device__ __forceinline__ void store_inv64(const T *__restrict__ Li, T *__restrict__ Dinv)
{
	T o[16];
#pragma unroll
	for (int q = 0; q < 16; q++)
		o[q] = Li[b64_i(q) + b64_j(q) * LD];
#pragma unroll
	for (int q = 0; q < 16; q++)
		Dinv[threadIdx.x + 256 * q] = o[q];
}

// FACTOR: Cholesky of the w x w (w <= 64) lower block D (ld ldd, in place)
// and its inverse into Dinv (64 x 64, ld 64, identity past w).
// !FACTOR: D is already factored; only the inverse is formed.
// One 256-thread workgroup; S, Li and the result as block_core64.  Ends with
// a workgroup barrier, so the caller may reuse S and Li.
template <typename T, bool FACTOR>
__device__ __forceinline__ int block_potrf_inv64_t(int w, T *__restrict__ D, long ldd, T *__restrict__ Dinv, T *__restrict__ S,
                                   T *__restrict__ Li)
{
	block_load64<T>(w, D, ldd, S, Li);
	const int bad = block_core64<T, FACTOR>(S, Li);
	if (FACTOR)
		store_lower64<T>(w, S, D, ldd);
	store_inv64<T>(Li, Dinv);
	__syncthreads();
	return bad;
}

// P (m x w, w <= 64) <- P * Dinv^T for the 16 rows row0 .. row0+15 of P,
// one wave (Dinv 64x64, ld 64, identity past w).  The wave reads its rows
// completely before writing them, so the update is in place.  With PT the
// result is also written transposed there (PT(c, r) = P(r, c), ld ldpt).
template <typename T>
__device__ __forceinline__ void rows_apply_inv_t(int row0, int m, int w, const T *__restrict__ Dinv,
                                                 T *__restrict__ P, long ldp, T *__restrict__ PT = nullptr,
                                                 long ldpt = 0)
{
	typedef typename V4<T>::type V;
	const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	if (row0 >= m)
		return;
	const int row = row0 + r;
	const int rc = row < m ? row : m - 1;
	// operand loads in two batches (the panel rows with the first half of
	// Dinv, then the second half) rather than one round trip per MFMA
	T a[16], dv[2][16];
#pragma unroll
	for (int s = 0; s < 16; s++) {
		const int k = 4 * s + g;
		const T v = P[rc + (long)(k < w ? k : w - 1) * ldp];
		a[s] = k < w ? v : T(0);
	}
	V acc[4];
#pragma unroll
	for (int h = 0; h < 2; h++) {
#pragma unroll
		for (int c = 0; c < 2; c++)
#pragma unroll
			for (int s = 0; s < 16; s++)
				dv[c][s] = Dinv[(16 * (2 * h + c) + r) + (4 * s + g) * 64];
#pragma unroll
		for (int c = 0; c < 2; c++) {
			acc[2 * h + c] = zero4<T>();
#pragma unroll
			for (int s = 0; s < 16; s++)
				acc[2 * h + c] = sa_mfma(a[s], dv[c][s], acc[2 * h + c]);
		}
	}
	// acc[cb][q] = X(row0 + drow(q, g), 16cb + r)
#pragma unroll
	for (int cb = 0; cb < 4; cb++)
#pragma unroll
		for (int q = 0; q < 4; q++) {
			const int rr = row0 + drow<T>(q, g), cc = 16 * cb + r;
			if (rr < m && cc < w) {
				P[rr + (long)cc * ldp] = acc[cb][q];
				if (PT)
					PT[cc + (long)rr * ldpt] = acc[cb][q];
			}
		}
}

// FP64 entry points of the callers.
template <bool FACTOR>
__device__ __forceinline__ int block_potrf_inv64(int w, double *__restrict__ D, long ldd,
                                                 double *__restrict__ Dinv, double *__restrict__ S,
                                                 double *__restrict__ Li)
{
	return block_potrf_inv64_t<double, FACTOR>(w, D, ldd, Dinv, S, Li);
}

__device__ __forceinline__ void rows_apply_inv(int row0, int m, int w, const double *__restrict__ Dinv,
                                               double *__restrict__ P, long ldp)
{
	rows_apply_inv_t<double>(row0, m, w, Dinv, P, ldp);
}

} // namespace sa64

#endif
