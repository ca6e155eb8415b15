// qbf_device.hpp -- device building blocks for batched 2-D FFT pipelines on gfx950.
//
// A P x P complex grid (row index l, column index k, element (l, k)) is owned by
// one workgroup of T threads.  G = T / P threads share one "line" (a row or a
// column); each thread holds E = P / G elements of its line in registers.
// Four register layouts are used:
//   R_i  line = row l,    thread p holds k = p + G*s                     (s < E)  interleaved
//   R_b  line = row l,    thread p holds k = blk_lane(p) + blk_reg(u)    (u < E)  blocked
//   C_i  line = column k, thread p holds l = p + G*s
//   C_b  line = column k, thread p holds l = blk_lane(p) + blk_reg(u)
// (see LineMap)
// A forward line FFT maps an interleaved layout to the blocked one (in-register
// DFT of length E, twiddle, DFT of length G across the lanes of the line);
// the backward line FFT maps blocked to interleaved.  Rows and columns are
// exchanged through LDS (R_i -> C_b and C_b -> R_i only).  Grids that live in
// global memory between kernels are stored in "native" order: element u of
// thread t at offset u*T + t, so every load and store of a wave is coalesced.
//
// FFT sign convention: forward = exp(-2 pi i jk/n), backward = exp(+2 pi i jk/n),
// both unnormalised (FFTW_FORWARD / FFTW_BACKWARD, as used by the reference
// src/integrals.c:48-51).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace qbf {

template <typename R> struct cplx_sel;
template <> struct cplx_sel<float> { using type = float2; };
template <> struct cplx_sel<double> { using type = double2; };
template <typename R> using cx = typename cplx_sel<R>::type;

template <typename R>
__host__ __device__ __forceinline__ cx<R> mk(R a, R b)
{
	cx<R> r;
	r.x = a;
	r.y = b;
	return r;
}
template <typename R> __device__ __forceinline__ cx<R> cadd(cx<R> a, cx<R> b) { return mk<R>(a.x + b.x, a.y + b.y); }
template <typename R> __device__ __forceinline__ cx<R> csub(cx<R> a, cx<R> b) { return mk<R>(a.x - b.x, a.y - b.y); }
template <typename R> __device__ __forceinline__ cx<R> cmul(cx<R> a, cx<R> b)
{
	return mk<R>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * conj(b)
template <typename R> __device__ __forceinline__ cx<R> cmulc(cx<R> a, cx<R> b)
{
	return mk<R>(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
template <typename R> __device__ __forceinline__ cx<R> cscale(cx<R> a, R s) { return mk<R>(a.x * s, a.y * s); }
template <typename R> __device__ __forceinline__ cx<R> czero() { return mk<R>(R(0), R(0)); }

// cos / sin (2 pi j / 64), j < 64, correctly rounded double literals.
struct Tw64 {
	static constexpr double c[64] = {
		1.0, 0.9951847266721969, 0.9807852804032304, 0.9569403357322088,
		0.9238795325112867, 0.881921264348355, 0.8314696123025452, 0.773010453362737,
		0.7071067811865476, 0.6343932841636455, 0.5555702330196023, 0.4713967368259978,
		0.38268343236508984, 0.29028467725446233, 0.19509032201612833, 0.09801714032956077,
		6.123233995736766e-17, -0.09801714032956065, -0.1950903220161282, -0.29028467725446216,
		-0.3826834323650897, -0.4713967368259977, -0.555570233019602, -0.6343932841636454,
		-0.7071067811865475, -0.773010453362737, -0.8314696123025453, -0.8819212643483549,
		-0.9238795325112867, -0.9569403357322088, -0.9807852804032304, -0.9951847266721968,
		-1.0, -0.9951847266721969, -0.9807852804032304, -0.9569403357322089,
		-0.9238795325112868, -0.881921264348355, -0.8314696123025455, -0.7730104533627371,
		-0.7071067811865477, -0.6343932841636459, -0.5555702330196022, -0.47139673682599786,
		-0.38268343236509034, -0.29028467725446244, -0.19509032201612866, -0.09801714032956045,
		-1.8369701987210297e-16, 0.09801714032956009, 0.1950903220161283, 0.29028467725446205,
		0.38268343236509, 0.4713967368259976, 0.5555702330196018, 0.6343932841636456,
		0.7071067811865474, 0.7730104533627367, 0.8314696123025452, 0.8819212643483548,
		0.9238795325112865, 0.9569403357322088, 0.9807852804032303, 0.9951847266721969};
	static constexpr double sn[64] = {
		0.0, 0.0980171403295606, 0.19509032201612825, 0.29028467725446233,
		0.3826834323650898, 0.47139673682599764, 0.5555702330196022, 0.6343932841636455,
		0.7071067811865475, 0.773010453362737, 0.8314696123025452, 0.8819212643483549,
		0.9238795325112867, 0.9569403357322089, 0.9807852804032304, 0.9951847266721968,
		1.0, 0.9951847266721969, 0.9807852804032304, 0.9569403357322089,
		0.9238795325112867, 0.881921264348355, 0.8314696123025455, 0.7730104533627371,
		0.7071067811865476, 0.6343932841636455, 0.5555702330196022, 0.47139673682599786,
		0.3826834323650899, 0.2902846772544624, 0.1950903220161286, 0.09801714032956083,
		1.2246467991473532e-16, -0.09801714032956059, -0.19509032201612836, -0.2902846772544621,
		-0.38268343236508967, -0.47139673682599764, -0.555570233019602, -0.6343932841636453,
		-0.7071067811865475, -0.7730104533627367, -0.8314696123025452, -0.8819212643483549,
		-0.9238795325112865, -0.9569403357322088, -0.9807852804032303, -0.9951847266721969,
		-1.0, -0.9951847266721969, -0.9807852804032304, -0.9569403357322089,
		-0.9238795325112866, -0.881921264348355, -0.8314696123025455, -0.7730104533627369,
		-0.7071067811865477, -0.6343932841636459, -0.5555702330196022, -0.4713967368259979,
		-0.3826834323650904, -0.2902846772544625, -0.19509032201612872, -0.0980171403295605};
	static constexpr double s(int j) { return sn[j]; }
};

template <int E>
__host__ __device__ constexpr int brev(int i)
{
	int r = 0;
	for (int b = 1, rb = E >> 1; b < E; b <<= 1, rb >>= 1)
		if (i & b) r |= rb;
	return r;
}

template <int X>
__host__ __device__ constexpr int ilog2c()
{
	int l = 0;
	while ((1 << l) < X) l++;
	return l;
}

// c * exp(SIGN * 2 pi i j / m) for compile-time (after unrolling) j, m <= 64.
template <typename R, int SIGN>
__device__ __forceinline__ cx<R> twmul(cx<R> c, int j, int m)
{
	if (j == 0) return c;
	if (4 * j == m) return SIGN < 0 ? mk<R>(c.y, -c.x) : mk<R>(-c.y, c.x);
	if (4 * j == 3 * m) return SIGN < 0 ? mk<R>(-c.y, c.x) : mk<R>(c.y, -c.x);
	if (2 * j == m) return mk<R>(-c.x, -c.y);
	const R cr = (R)Tw64::c[j * (64 / m)];
	const R si = (R)(SIGN * Tw64::s(j * (64 / m)));
	return mk<R>(c.x * cr - c.y * si, c.x * si + c.y * cr);
}

// Radix-2 butterfly with a constant twiddle: a +- b exp(SIGN 2 pi i j / m), j < m / 2 (constants after
// unrolling).  FACTORED: a twiddle c (1 + i r), or i s (1 - i r) where |sin| > |cos|, takes two FMAs for the
// factor in brackets, two additions for an eighth of a turn, and four FMAs for the sums with c or s, 6
// operations instead of 8; |r| <= 1, so nothing is magnified.  For the VALU-bound FP32 grids of N <= 64 (step
// of 512 cells at N = 64: 187.6 ms, 192.9 without; the same error).  With it the error of FP64 Strang steps at N = 32
// was 3.2e-16 instead of 3.0e-16, and FP32 steps at N = 128 took 47.4 instead of 45.6 ms.
template <typename R, int SIGN, bool FACTORED>
__device__ __forceinline__ void bfly(cx<R>& a, cx<R>& b, int j, int m)
{
	if (j == 0 || 4 * j == m || !FACTORED) {
		const cx<R> t = twmul<R, SIGN>(b, j, m);
		b = csub<R>(a, t);
		a = cadd<R>(a, t);
		return;
	}
	const double wc = Tw64::c[j * (64 / m)], ws = SIGN * Tw64::s(j * (64 / m));
	const bool eighth = 8 * j == m || 8 * j == 3 * m;
	const bool big = eighth || (wc < 0 ? -wc : wc) > (ws < 0 ? -ws : ws);
	R q, tx, ty;
	if (big) {                                 // w = c (1 + i r)
		q = (R)wc;
		if (eighth) {
			const bool neg = (wc < 0) != (ws < 0);
			tx = neg ? b.x + b.y : b.x - b.y;
			ty = neg ? b.y - b.x : b.y + b.x;
		} else {
			const R r = (R)(ws / wc);
			tx = fma(-r, b.y, b.x);
			ty = fma(r, b.x, b.y);
		}
	} else {                                   // w = s (r + i)
		q = (R)ws;
		const R r = (R)(wc / ws);
		tx = fma(r, b.x, -b.y);
		ty = fma(r, b.y, b.x);
	}
	b = mk<R>(fma(-q, tx, a.x), fma(-q, ty, a.y));
	a = mk<R>(fma(q, tx, a.x), fma(q, ty, a.y));
}

// In-register DFT of length E (power of two <= 64), natural order in and out.
template <typename R, int E, int SIGN, bool FACTORED = false>
__device__ __forceinline__ void dft(cx<R>* v)
{
	if constexpr (E > 1) {
		cx<R> w[E];
#pragma unroll
		for (int i = 0; i < E; i++) w[i] = v[brev<E>(i)];
#pragma unroll
		for (int m = 2; m <= E; m <<= 1) {
#pragma unroll
			for (int b = 0; b < E; b += m) {
#pragma unroll
				for (int j = 0; j < m / 2; j++) bfly<R, SIGN, FACTORED>(w[b + j], w[b + j + m / 2], j, m);
			}
		}
#pragma unroll
		for (int i = 0; i < E; i++) v[i] = w[i];
	}
}

// The 16 lanes of a line at N = 128: bit h of p flips with a DPP permutation of them.  The xor masks 1 and
// 2 (quad permutes), 7 (half-row mirror) and 15 (row mirror) span the 16 lanes, so lane l has p = dpp_p(l)
// and its partner p ^ h is one DPP operand away for every h (with p = l, lane distances 4 and 8 went
// through the LDS unit).  FP32 Strang step of 32 cells 49.5 -> 45.6 ms.
__host__ __device__ __forceinline__ constexpr int dpp_p(int l) { return l ^ (l & 4 ? 3 : 0) ^ (l & 8 ? 4 : 0); }

template <int H>
__device__ __forceinline__ int partner_i32(int x)
{
	if constexpr (H == 1) return __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);        // quad_perm [1,0,3,2]
	else if constexpr (H == 2) return __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
	else if constexpr (H == 4) return __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false);  // row_half_mirror
	else return __builtin_amdgcn_mov_dpp(x, 0x140, 0xF, 0xF, false);                        // row_mirror
}
template <int H>
__device__ __forceinline__ double partner(double x)
{
	return __hiloint2double(partner_i32<H>(__double2hiint(x)), partner_i32<H>(__double2loint(x)));
}

// x += s * (x of the partner) for 8 floats, one v_fmac with a DPP operand each (the compiler leaves a
// move and an FMA).  A DPP operand is read two wait states after it was written at the earliest: the
// s_nop, since the compiler does not look into the block.  FIXED: a fixed point of the instruction order
// (N = 128: 45.4 ms instead of 47.7 for a step of 32 cells; k_i3fold_pair at N = 64 spills with it, 658 ms
// instead of 196 for a step of 512 cells).
#define QBF_FMAC8(ASM, DPP) \
	ASM("s_nop 1\n\t" \
		"v_fmac_f32_dpp %0, %0, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %1, %1, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %2, %2, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %3, %3, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %4, %4, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %5, %5, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %6, %6, %8 " DPP " row_mask:0xf bank_mask:0xf\n\t" \
		"v_fmac_f32_dpp %7, %7, %8 " DPP " row_mask:0xf bank_mask:0xf" \
		: "+v"(v[0].x), "+v"(v[0].y), "+v"(v[1].x), "+v"(v[1].y), "+v"(v[2].x), "+v"(v[2].y), "+v"(v[3].x), "+v"(v[3].y) \
		: "v"(s))
template <int H, bool FIXED>
__device__ __forceinline__ void fmac_partner4(float2* v, float s)
{
#define QBF_FMAC8_DPP(DPP) do { if constexpr (FIXED) QBF_FMAC8(asm volatile, DPP); else QBF_FMAC8(asm, DPP); } while (0)
	if constexpr (H == 1) QBF_FMAC8_DPP("quad_perm:[1,0,3,2]");
	else if constexpr (H == 2) QBF_FMAC8_DPP("quad_perm:[2,3,0,1]");
	else if constexpr (H == 4) QBF_FMAC8_DPP("row_half_mirror");
	else QBF_FMAC8_DPP("row_mirror");
#undef QBF_FMAC8_DPP
}
#undef QBF_FMAC8

// v += s * (v of lane p ^ H)
template <typename R, int E, int H, bool FIXED = false>
__device__ __forceinline__ void add_partner(cx<R>* v, R s)
{
	static_assert(H == 1 || H == 2 || H == 4 || H == 8, "one bit of p");
	if constexpr (sizeof(R) == 4) {
#pragma unroll
		for (int u = 0; u < E; u += 4) fmac_partner4<H, FIXED>(v + u, s);
	} else {
#pragma unroll
		for (int u = 0; u < E; u++) v[u] = mk<R>(fma(partner<H>(v[u].x), s, v[u].x), fma(partner<H>(v[u].y), s, v[u].y));
	}
}

// x and y of the lanes with bit B (16 or 32) of the lane index: y of the lower lanes <-> x of the upper
// ones.  Afterwards x holds the lower lane's values (its x in the lower, its y in the upper lane), y the
// upper lane's: one instruction transposes the lane bit with the register index.
template <int B>
__device__ __forceinline__ void lane_swap(int& x, int& y)
{
	static_assert(B == 16 || B == 32, "row and half-wave swaps");
	if constexpr (B == 16) {
		const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
		x = r[0];
		y = r[1];
	} else {
		const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
		x = r[0];
		y = r[1];
	}
}
template <int B>
__device__ __forceinline__ void lane_swap(float& x, float& y)
{
	int a = __float_as_int(x), b = __float_as_int(y);
	lane_swap<B>(a, b);
	x = __int_as_float(a);
	y = __int_as_float(b);
}
template <int B>
__device__ __forceinline__ void lane_swap(double& x, double& y)
{
	int al = __double2loint(x), ah = __double2hiint(x), bl = __double2loint(y), bh = __double2hiint(y);
	lane_swap<B>(al, bl);
	lane_swap<B>(ah, bh);
	x = __hiloint2double(ah, al);
	y = __hiloint2double(bh, bl);
}

// Where the G = 4 or 8 lanes of a line sit in a wave, and the blocked order of their elements.  Bits 5
// and 4 of the lane index are the two high bits of p, for G = 8 bit 0 is the low one; the other bits are
// the line.  The transform over p then begins (ends) with the permlane swaps that exchange bits 5 and 4
// with the two high bits of the register index: the four values of a DFT-4 over them are in one lane, with
// no selects and no lane-dependent factors, and only the last radix-2 stage of G = 8 needs a partner.  A
// swap moves two registers in the time of two moves (8.4 cycles against 4.3 of a DPP move or an FMA).
//   With p in the low lane bits, a move, an FMA and (lane distance 4) an LDS swizzle per value and stage, a
// line of 128 took 516 VALU and 32 LDS operations in FP32, now about 410 (swaps counted twice) and none,
// and the lines of a phase of LDS accesses are consecutive.  FP32 Strang step, N = 64, 512 cells:
// 204 -> 188 ms; FP64, N = 64, 16 cells: 42.5 -> 41.4; FP64, N = 16, simulation steps of 24 cells: 2.40 ->
// 2.26; FP64, N = 32, 128 cells the same (bound by L2: a quarter fewer VALU operations gained nothing).  A
// v_fmac with a DPP operand per float and stage in FP32, as at N = 128: 193.8 ms.
template <int G, int E>
struct LineMap {
	static_assert(G == 4 || G == 8, "4 or 8 lanes a line");
	static_assert(E % 4 == 0, "two bits of the register index change places with lane bits");
	static constexpr int P = G * E;
	// line and p of thread t
	static __host__ __device__ __forceinline__ constexpr int line(int t)
	{
		return G == 8 ? (t >> 6) * 8 + ((t >> 1) & 7) : (t >> 6) * 16 + (t & 15);
	}
	static __host__ __device__ __forceinline__ constexpr int lane(int t)
	{
		return G == 8 ? 2 * ((t >> 4) & 3) + (t & 1) : (t >> 4) & 3;
	}
	// index of blocked element u of lane p: blk_lane(p) + blk_reg(u)
	static __device__ __forceinline__ constexpr int blk_lane(int p)
	{
		return G == 8 ? (E / 4) * (p >> 1) + (P / 2) * (p & 1) : (E / 4) * p;
	}
	static __device__ __forceinline__ constexpr int blk_reg(int u) { return E * (u / (E / 4)) + u % (E / 4); }
};

// Geometry of one P x P grid per workgroup of T threads.
template <int P_, int T_>
struct Geo : LineMap<T_ / P_, P_ * P_ / T_> {
	static constexpr int P = P_;
	static constexpr int T = T_;
	static constexpr int G = T_ / P_;       // threads per line
	static constexpr int E = P_ / G;        // elements per thread
	static constexpr int PITCH = P_ + G / 4; // LDS row pitch (elements), see Xpose
	static constexpr int SKEW = G == 8 ? 8 : 0;
	static_assert(G * P_ == T_, "T must be a multiple of P");
	static_assert(G * E == P_, "G must divide P");
	static_assert(T_ % 64 == 0, "whole waves");
};

// Logical block index that keeps consecutive logical blocks on one XCD.  The dispatcher hands
// block b to XCD b % 8, so XCD x runs the logical blocks [x n/8, (x+1) n/8): workgroups that read
// the same grids (the outputs of one cell) share that XCD's L2.  A permutation of [0, n) for any
// n divisible by 8 (identity otherwise), so correctness never depends on the dispatch order.
__device__ __forceinline__ int xcd_block()
{
	const int n = gridDim.x, b = blockIdx.x;
	return (n & 7) ? b : (b & 7) * (n >> 3) + (b >> 3);
}

// An SGPR zero the compiler cannot see through: adding it to an LDS index keeps table loads
// next to their use instead of hoisting them (and their registers) out of the term loops.
__device__ __forceinline__ int opaque_zero()
{
	int z = 0;
	asm volatile("" : "+s"(z));
	return z;
}

// p + off with an opaque SGPR term, so the address (and the load) is formed next to its
// use; p keeps its address space (a global pointer stays a global load).
template <typename X>
__device__ __forceinline__ X* uni(X* p, long long off)
{
	typedef __attribute__((address_space(1))) X gX;
	unsigned long long a = (unsigned long long)(p + off);
	asm volatile("" : "+s"(a));
	return (X*)(gX*)a;
}

// A VGPR copy of a lane index that the compiler cannot trace: addresses formed from it are not
// hoisted out of the enclosing loop into (spilled) registers.
__device__ __forceinline__ int opaque_lane(int x)
{
	asm volatile("" : "+v"(x));
	return x;
}

// Materialise a value in VGPRs here: keeps a load unconditional (not sunk into a branch
// of the lanes that use it).
template <typename R>
__device__ __forceinline__ cx<R> pin(cx<R> w)
{
	asm volatile("" : "+v"(w.x), "+v"(w.y));
	return w;
}

// Twiddle tables of a P-point line FFT over T threads (G = T / P lanes per line): w^j (P entries),
// the per-lane table (P entries) and the cross-lane stage twiddles (G entries).
template <int P, int T>
struct TwTab {
	static constexpr int SIZE = 2 * P + T / P;
};

// The per-lane twiddle table w^(p u) is interleaved by lane, [u][p], so that the G distinct addresses
// of one read fall into distinct banks: entry u of lane p at G u + p.  (FP64, [p][u]: a fifth of the
// I3 kernel's LDS cycles were conflicts.)

// Exchange bits 5 and 4 of the lane index with the two high bits of the register index of v.
template <typename R, int E>
__device__ __forceinline__ void lane_transpose(cx<R>* v)
{
	constexpr int Q = E / 4;
#pragma unroll
	for (int u = 0; u < 2 * Q; u++) {
		lane_swap<32>(v[u].x, v[u + 2 * Q].x);
		lane_swap<32>(v[u].y, v[u + 2 * Q].y);
	}
#pragma unroll
	for (int u = 0; u < Q; u++)
#pragma unroll
		for (int h = 0; h < 4; h += 2) {
			lane_swap<16>(v[h * Q + u].x, v[(h + 1) * Q + u].x);
			lane_swap<16>(v[h * Q + u].y, v[(h + 1) * Q + u].y);
		}
}

// DFT-4 over the two high bits of the register index, in place
template <typename R, int E, int SIGN>
__device__ __forceinline__ void dft4_high(cx<R>* v)
{
	constexpr int Q = E / 4;
#pragma unroll
	for (int u = 0; u < Q; u++) {
		cx<R> w[4] = {v[u], v[Q + u], v[2 * Q + u], v[3 * Q + u]};
		dft<R, 4, SIGN>(w);
#pragma unroll
		for (int q = 0; q < 4; q++) v[q * Q + u] = w[q];
	}
}

// v times exp(SIGN 2 pi i f / 8) in the upper lanes of a pair, f the two high bits of the register index
template <typename R, int E, int SIGN>
__device__ __forceinline__ void pair_twiddle(cx<R>* v, bool up)
{
	constexpr int Q = E / 4;
	constexpr R H = (R)Tw64::c[8];
	const R c1 = up ? H : R(1), s1 = up ? SIGN * H : R(0), c3 = up ? -H : R(1);
#pragma unroll
	for (int u = 0; u < Q; u++) {
		const cx<R> a = v[Q + u], b = v[2 * Q + u], c = v[3 * Q + u];
		v[Q + u] = mk<R>(a.x * c1 - a.y * s1, a.x * s1 + a.y * c1);
		v[2 * Q + u] = SIGN < 0 ? mk<R>(up ? b.y : b.x, up ? -b.x : b.y) : mk<R>(up ? -b.y : b.x, up ? b.x : b.y);
		v[3 * Q + u] = mk<R>(c.x * c3 - c.y * s1, c.x * s1 + c.y * c3);
	}
}

// A radix-2 stage across lanes is v + s (v of the partner) with s = +-1: a + b in the lower lane p, b - a
// of its own b in the upper lane p ^ h, the negative of the butterfly's a - b.  Where the upper lane's
// values come in negated, s = -1 in the lower and +1 in the upper lane give a + b and a - b.  The signs
// are in the lane-dependent factors that precede or follow the stages.

// Forward FFT of one line: interleaved layout in, blocked layout out.
// twP[j] = (cos, sin)(2 pi j / P), j < P; the per-lane table (cos, sin)(2 pi p u / P) follows it
// (in LDS).  n = p + G s, p = (G / 4) g + b: a DFT-E over s, twiddles w^(p u), a DFT-4 over g (frequency
// f), for G = 8 twiddles w8^(f b) and the sum over b (frequency c): k = u + E f + 4 E c with the high bits
// of u in the lane.  G = 8: the upper lanes b = 1 are negated by the per-lane twiddles (load_twiddles_g)
// and here for u = 0.
template <typename R, class GE>
__device__ __forceinline__ void line_fwd(cx<R>* v, int p, const cx<R>* twP)
{
	constexpr int P = GE::P, G = GE::G, E = GE::E;
	dft<R, E, -1, sizeof(R) == 4>(v);
	const cx<R>* tl = twP + P + p + opaque_zero();
#pragma unroll
	for (int u = 1; u < E; u++) v[u] = cmulc<R>(v[u], tl[G * u]);
	const bool up = p & 1;
	const R sgn = up ? R(-1) : R(1);
	if constexpr (G == 8) v[0] = cscale<R>(v[0], sgn);
	lane_transpose<R, E>(v);
	dft4_high<R, E, -1>(v);
	if constexpr (G == 8) {
		pair_twiddle<R, E, -1>(v, up);
		add_partner<R, E, 1>(v, -sgn);
	}
}

// Backward FFT of one line: blocked layout in, interleaved layout out; the same stages in the opposite
// order (the stage over c leaves the upper lanes negated).
template <typename R, class GE>
__device__ __forceinline__ void line_bwd(cx<R>* v, int p, const cx<R>* twP)
{
	constexpr int P = GE::P, G = GE::G, E = GE::E;
	const bool up = p & 1;
	const R sgn = up ? R(-1) : R(1);
	if constexpr (G == 8) {
		add_partner<R, E, 1>(v, sgn);
		pair_twiddle<R, E, +1>(v, up);
	}
	dft4_high<R, E, +1>(v);
	lane_transpose<R, E>(v);
	const cx<R>* tl = twP + P + p + opaque_zero();
	if constexpr (G == 8) v[0] = cscale<R>(v[0], sgn);
#pragma unroll
	for (int u = 1; u < E; u++) v[u] = cmul<R>(v[u], tl[G * u]);
	dft<R, E, +1, sizeof(R) == 4>(v);
}

// (-1)^(bits 0 and 1 of p)
template <typename R>
__device__ __forceinline__ R low_parity(int p) { return (p ^ (p >> 1)) & 1 ? R(-1) : R(1); }

// The factor of a stage H >= 4: the twiddle exp(SIGN 2 pi i (p mod H) / 2H) in the upper lanes, negated there,
// and the sign s
template <typename R, int P, int H, int SIGN>
__device__ __forceinline__ cx<R> stage_factor(int p, const cx<R>* twP, R s)
{
	const cx<R> w = pin<R>(twP[2 * P + H + (p & (H - 1)) + opaque_zero()]);
	return p & H ? mk<R>(-s * w.x, SIGN * -s * w.y) : mk<R>(s, R(0));
}

// Lines of P = 16 E elements over 16 consecutive lanes (dpp_p), the blocked element u of lane p being
// k = E brev(p) + u: radix-2 stages over the bits of p
template <typename R, int P, int E>
__device__ __forceinline__ void line16_fwd(cx<R>* v, int p, const cx<R>* twP)
{
	dft<R, E, -1>(v);
	const cx<R>* tl = twP + P + p + opaque_zero();
#pragma unroll
	for (int u = 1; u < E; u++) v[u] = cmulc<R>(v[u], tl[16 * u]);
	// before the last two stages the lanes carry the sign low_parity
	add_partner<R, E, 8, true>(v, p & 8 ? R(-1) : R(1));
	const cx<R> w8 = stage_factor<R, P, 8, -1>(p, twP, R(1));
#pragma unroll
	for (int u = 0; u < E; u++) v[u] = cmul<R>(v[u], w8);
	add_partner<R, E, 4, true>(v, p & 4 ? R(-1) : R(1));
	const cx<R> w4 = stage_factor<R, P, 4, -1>(p, twP, low_parity<R>(p));
#pragma unroll
	for (int u = 0; u < E; u++) v[u] = cmul<R>(v[u], w4);
	add_partner<R, E, 2, true>(v, p & 2 ? R(1) : R(-1));
	// twiddle 1 or -i: a swap and a sign (two selects)
	const bool q = (p & 3) == 3;
#pragma unroll
	for (int u = 0; u < E; u++) v[u] = mk<R>(q ? v[u].y : v[u].x, q ? -v[u].x : v[u].y);
	add_partner<R, E, 1, true>(v, p & 1 ? R(1) : R(-1));
}

template <typename R, int P, int E>
__device__ __forceinline__ void line16_bwd(cx<R>* v, int p, const cx<R>* twP)
{
	// after the first two stages the lanes carry the sign low_parity
	add_partner<R, E, 1, true>(v, p & 1 ? R(-1) : R(1));
	const bool q = (p & 3) == 3;
#pragma unroll
	for (int u = 0; u < E; u++) v[u] = mk<R>(q ? -v[u].y : v[u].x, q ? v[u].x : v[u].y);
	add_partner<R, E, 2, true>(v, p & 2 ? R(-1) : R(1));
	const cx<R> w4 = stage_factor<R, P, 4, +1>(p, twP, low_parity<R>(p));
#pragma unroll
	for (int u = 0; u < E; u++) v[u] = cmul<R>(v[u], w4);
	add_partner<R, E, 4, true>(v, p & 4 ? R(1) : R(-1));
	const cx<R> w8 = stage_factor<R, P, 8, +1>(p, twP, R(1));
#pragma unroll
	for (int u = 0; u < E; u++) v[u] = cmul<R>(v[u], w8);
	add_partner<R, E, 8, true>(v, p & 8 ? R(1) : R(-1));
	const cx<R>* tl = twP + P + p + opaque_zero();
#pragma unroll
	for (int u = 1; u < E; u++) v[u] = cmul<R>(v[u], tl[16 * u]);
	dft<R, E, +1>(v);
}

// LDS exchanges.  The grid is stored row-major.  An 8-byte LDS access of a wave is served 128 bytes
// per phase: 16 consecutive lanes of one element each, conflict-free when their addresses are
// distinct modulo 16 elements (measured with SQ_LDS_BANK_CONFLICT of k_i3acc; 16-byte elements: 8 lanes).
//   G = 4: the lanes of a phase have one p and consecutive lines, in the accesses of columns (C_b)
// consecutive elements, in those of rows (R_i) the pitch apart, P + 1.  G = 8: eight consecutive lines with
// the two lanes of a pair, one element (rows) or P / 2 rows (columns) apart: pitch P + 2, and the rows from
// P / 2 on are skewed by 8.
//
// SPLIT: a grid that does not fit in the 160 KiB of LDS whole (FP64 128 x 128: 256 KiB) goes through
// it in two halves, real parts then imaginary parts: each half is the same grid of 8-byte elements,
// and a thread's real parts are free to take the transposed ones while its imaginary parts wait, so no
// staging registers are needed (two barriers more per exchange).  Against an exchange through a
// per-workgroup slot in global memory (35 GB of HBM traffic per 16,384 K applications): FP64 Strang
// step at N = 64, 16 cells, J = 32, M = 16, 110.8 -> 62.5 ms.
template <typename R, class GE, bool SPLIT = false>
struct Xpose {
	using El = typename std::conditional<SPLIT, R, cx<R>>::type;
	static constexpr int SIZE = GE::P * GE::PITCH + GE::SKEW;
	El* g0;
	__device__ __forceinline__ El* gp() const { return g0 + opaque_zero(); }
	__device__ __forceinline__ int a(int row, int col) const { return row * GE::PITCH + col + (row / (GE::P / 2)) * GE::SKEW; }
	// blocked element u of a column, c0 = col_base(line, p) (all of a lane's rows have its element 0's skew)
	__device__ __forceinline__ int blk(int c0, int u) const { return c0 + GE::blk_reg(u) * GE::PITCH; }
	__device__ __forceinline__ int col_base(int line, int p) const { return a(GE::blk_lane(p), line); }
	static __device__ __forceinline__ void out(El& e, cx<R> v, int c)
	{
		if constexpr (SPLIT) e = c ? v.y : v.x;
		else e = v;
	}
	static __device__ __forceinline__ void in(cx<R>& v, El e, int c)
	{
		if constexpr (SPLIT) (c ? v.y : v.x) = e;
		else v = e;
	}
	// put(g, c), get(g, c): this thread's writes and reads of half c (c = 0 only without SPLIT); the
	// first barrier waits for the reads of the previous exchange
	template <class Put, class Get>
	__device__ __forceinline__ void pass(Put put, Get get) const
	{
#pragma unroll
		for (int c = 0; c < (SPLIT ? 2 : 1); c++) {
			__syncthreads();
			put(gp(), c);
			__syncthreads();
			get((const El*)gp(), c);
		}
	}
	// one thread's share of a line in the four layouts, NZ: without the padding zeros (the elements s
	// with E/4 <= s < 3E/4, see padded_nonzero; read as zeros)
	__device__ __forceinline__ void put_Ri(El* g, const cx<R>* v, int line, int p, int c) const
	{
#pragma unroll
		for (int s = 0; s < GE::E; s++) out(g[a(line, p + GE::G * s)], v[s], c);
	}
	__device__ __forceinline__ void put_Cb(El* g, const cx<R>* v, int line, int p, int c) const
	{
		const int c0 = col_base(line, p);
#pragma unroll
		for (int u = 0; u < GE::E; u++) out(g[blk(c0, u)], v[u], c);
	}
	__device__ __forceinline__ void get_Cb(const El* g, cx<R>* v, int line, int p, int c) const
	{
		const int c0 = col_base(line, p);
#pragma unroll
		for (int u = 0; u < GE::E; u++) in(v[u], g[blk(c0, u)], c);
	}
	__device__ __forceinline__ void get_Ri(const El* g, cx<R>* v, int line, int p, int c) const
	{
#pragma unroll
		for (int s = 0; s < GE::E; s++) in(v[s], g[a(line, p + GE::G * s)], c);
	}
	// R_i -> C_b and C_b -> R_i of the whole grid
	__device__ __forceinline__ void RiCb(cx<R>* v, int line, int p) const
	{
		pass([&](El* g, int c) { put_Ri(g, v, line, p, c); }, [&](const El* g, int c) { get_Cb(g, v, line, p, c); });
	}
	__device__ __forceinline__ void CbRi(cx<R>* v, int line, int p) const
	{
		pass([&](El* g, int c) { put_Cb(g, v, line, p, c); }, [&](const El* g, int c) { get_Ri(g, v, line, p, c); });
	}
};

// Fill the LDS twiddle tables from a global table of (cos, sin)(2 pi j / 256) in double:
// twP[j] = w^j for j < P, the per-lane table w^(p*u) at twP[P + G u + p] (G = 8:
// negated for odd p, see line_fwd), and the
// twiddles of the cross-lane stages at twP[2P + h + m] = w^(m P / 2h), m < h < G, kept apart so
// that the lanes of one stage read consecutive entries; w = exp(2 pi i / P).
// (load_twiddles_g: G lanes per line, filled by the NT threads of the workgroup)
template <typename R, int P, int G, int NT>
__device__ __forceinline__ void load_twiddles_g(cx<R>* twP, const double2* tw256)
{
	for (int j = threadIdx.x; j < 2 * P + G; j += NT) {
		int k;
		if (j < P) {
			k = j;
		} else if (j < 2 * P) {
			k = ((j - P) % G) * ((j - P) / G);
		} else {
			const int i = j - 2 * P;
			int h = 1;
			while (2 * h <= i) h *= 2;
			k = i == 0 ? 0 : (i - h) * (P / (2 * h));
		}
		const double2 w = tw256[k * (256 / P)];
		const double sg = G == 8 && j >= P && j < 2 * P && (j & 1) ? -1.0 : 1.0;
		twP[j] = mk<R>((R)(sg * w.x), (R)(sg * w.y));
	}
}
template <typename R, int P, int T>
__device__ __forceinline__ void load_twiddles(cx<R>* twP, const double2* tw256)
{
	static_assert(TwTab<P, T>::SIZE == 2 * P + T / P, "table layout");
	load_twiddles_g<R, P, T / P, T>(twP, tw256);
}

// Native (coalesced) storage of a register-resident grid.
template <typename R, class GE>
__device__ __forceinline__ void store_native(cx<R>* dst, const cx<R>* v)
{
#pragma unroll
	for (int u = 0; u < GE::E; u++) uni(dst, (long long)u * GE::T)[threadIdx.x] = v[u];
}
template <typename R, class GE>
__device__ __forceinline__ void load_native(cx<R>* v, const cx<R>* src)
{
#pragma unroll
	for (int u = 0; u < GE::E; u++) v[u] = uni(src, (long long)u * GE::T)[threadIdx.x];
}

// One array in global memory through a buffer descriptor: element t + u * T (u a compile-time
// constant after unrolling) is a load with the lane's byte offset in a VGPR and u * T in a scalar
// offset, so that many loads in flight need no 64-bit scalar address each (with uni() the kernels
// that read five grids per term spilled about 60 SGPRs).  The base is opaque: loads through different
// BufRefs of one array are not merged, and none is hoisted out of a loop that constructs it (kept in
// registers from one use to the next, they spilled the accumulators).  n: elements of the array;
// accesses beyond it read zero and are not written.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
template <typename X>
struct BufRef {
	X* base;
	__amdgpu_buffer_rsrc_t rs;
	__device__ __forceinline__ BufRef(const X* p, int n)
		: base((X*)p), rs(__builtin_amdgcn_make_buffer_rsrc((void*)uni(p, 0), 0, n * (int)sizeof(X), 0x00020000)) {}
	// element voff + soff: voff per lane, soff uniform
	__device__ __forceinline__ X get(int voff, int soff) const
	{
		const int vb = voff * (int)sizeof(X), sb = soff * (int)sizeof(X);
		if constexpr (sizeof(X) == 4) return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b32(rs, vb, sb, 0));
		else if constexpr (sizeof(X) == 8) return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b64(rs, vb, sb, 0));
		else return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b128(rs, vb, sb, 0));
	}
	// 16-byte values go through a global store: a buffer_store_dwordx4 with a scalar offset reads its
	// last data lanes late, and the compiler lets the next instruction overwrite the data registers
	// (measured: lanes 12-15 of each 16 then stored the new values)
	__device__ __forceinline__ void put(int voff, int soff, X x) const
	{
		const int vb = voff * (int)sizeof(X), sb = soff * (int)sizeof(X);
		if constexpr (sizeof(X) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), rs, vb, sb, 0);
		else if constexpr (sizeof(X) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), rs, vb, sb, 0);
		else uni(base, soff)[voff] = x;
	}
};

// fn(u, ld(u)) for u < E, the loads ld issued in batches of B with the next batch in flight while one
// is used.  (Left to itself the compiler issued one load at a time in the kernels that are close to
// their register limit, each waited for before the next: FP32 step at N = 64 244 ms against 206.)
template <int E, int B, class Ld, class Fn>
__device__ __forceinline__ void batched(Ld ld, Fn fn)
{
	static_assert(E % B == 0, "whole batches");
	decltype(ld(0)) x[E];
#pragma unroll
	for (int k = 0; k < B; k++) x[k] = ld(k);
#pragma unroll
	for (int b = 0; b < E; b += B) {
		if (b + B < E)
#pragma unroll
			for (int k = 0; k < B; k++) x[b + B + k] = ld(b + B + k);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int k = 0; k < B; k++) fn(b + k, x[b + k]);
		__builtin_amdgcn_sched_barrier(0);
	}
}
template <typename X, typename Y> struct Two { X a; Y b; };

} // namespace qbf
