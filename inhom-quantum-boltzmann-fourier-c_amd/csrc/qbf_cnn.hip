// qbf_cnn.hip -- periodic 3x3 CNN surrogate of the collision operator: forward, backward and
// Adam kernels for gfx950 (no counterpart in the reference).
//
// Network: six 3x3 convolutions on the S x S velocity grid (S = N), periodic padding, GELU
// after the first five: 4 -> 64 -> 64 -> 64 -> 64 -> 64 -> 4 channels.  Activations are
// stored NHWC in bf16 (channels padded: 4 -> 32 at the input, 4 -> 32 at the output), weights
// as bf16 copies of fp32 master weights, and every convolution accumulates in fp32.
//
// The image side S is 64 or 128 (velocity grids N = 64, 128; a template parameter of the
// kernels).  Forward and backward-data convolutions are implicit GEMMs on the matrix cores
// (v_mfma_f32_16x16x32_bf16): each wave owns a 64-pixel segment of an image row times all output
// channels; K = 9 taps x input channels.
// MFMA operand layout (16 x 16 x 32): lane l holds A[l%16][8*(l/16) .. +7],
// B[8*(l/16) .. +7][l%16], and the result D[4*(l/16) + r][l%16], r < 4.
// The weight gradient (a reduction over all pixels) runs there too, over pixels.
// Options (qbf_cnn_configure): a dilation d_l per layer (tap offsets (ky-1, kx-1) * d_l), and
// per-cell normalisation: a_b = max |x[b][0]| (trace channel); the network sees x / a_b and the
// constant channel iscale * a_b, its output is scaled by oscale * a_b^2, and the training loss
// is taken on the normalised output.
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <string>
#include <type_traits>
#include <vector>

#include "../../include/qbf.h"

namespace qbfcnn {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __bf16 bf16;

constexpr int SEGP = 64;        // pixels of an image row segment (one wave of the convolutions)
constexpr int NL = 6;           // layers
constexpr int CH = 64;          // hidden channels
constexpr int CIO = 32;         // padded input / output channel count
constexpr int CREAL = 4;        // real input / output channels (Pauli components)
// channels stored of the network input (CREAL, the amplitude, zeros).  The conversion of 512 images of 64 x 64
// writes 34 MB instead of 134 (69 us with all 32 channels)
constexpr int CIN0 = 8;

__host__ __device__ constexpr int cin_of(int l) { return l == 0 ? CIO : CH; }
__host__ __device__ constexpr int cout_of(int l) { return l == NL - 1 ? CIO : CH; }

// tanh-form GELU, z * 0.5 (1 + tanh u) with u = sqrt(2/pi) (z + 0.044715 z^3), evaluated through
// 0.5 (1 + tanh u) = 1 / (1 + exp(-2u)) with the hardware base-2 exponential and reciprocal (about
// 1e-7 relative error, far below the bf16 rounding of the activations; exp overflow gives 0, the
// z -> -inf limit)
__device__ __forceinline__ float half_one_plus_tanh(float u)
{
	const float e = __builtin_amdgcn_exp2f(-2.8853900817779268f * u);   // exp(-2u) = 2^(-2 log2(e) u)
	return __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu(float z)
{
	const float c = 0.7978845608028654f;   // sqrt(2/pi)
	const float u = c * (z + 0.044715f * z * z * z);
	return z * half_one_plus_tanh(u);
}
// derivative: s + z s (1 - s) 2 u', s = 0.5 (1 + tanh u), u' = sqrt(2/pi) (1 + 3 * 0.044715 z^2)
__device__ __forceinline__ float gelu_grad(float z)
{
	const float c = 0.7978845608028654f;
	const float u = c * (z + 0.044715f * z * z * z);
	const float sg = half_one_plus_tanh(u);
	return sg + 2.0f * z * sg * (1.0f - sg) * c * (1.0f + 3.0f * 0.044715f * z * z);
}

// a[b] = max |x[b][0][.]|  (one workgroup of 256 per cell)
template <int S>
__global__ __launch_bounds__(256) void k_cell_amp(const float* __restrict__ x, float* __restrict__ amp)
{
	__shared__ float sh[4];
	const float* xb = x + (size_t)blockIdx.x * CREAL * S * S;
	float m = 0.f;
	for (int p = threadIdx.x; p < S * S; p += 256) m = fmaxf(m, fabsf(xb[p]));
	for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
	if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
	__syncthreads();
	if (threadIdx.x == 0) amp[blockIdx.x] = fmaxf(fmaxf(sh[0], sh[1]), fmaxf(sh[2], sh[3]));
}

// planar fp32 [B][4][S][S] -> NHWC bf16 [B][S][S][CIN0]: channels 0..3 = scale * x (or
// scale * x / a[b] with amp), channel 4 = scale * a[b] with amp, the rest zero (channels CIN0 ... CIO - 1
// of the first layer are zero too and not stored)
template <int S>
__global__ void k_to_nhwc(const float* __restrict__ x, bf16* __restrict__ out, int B, float scale,
	const float* __restrict__ amp)
{
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	const long long n = (long long)B * S * S;
	if (i >= n) return;
	const int b = (int)(i / (S * S)), p = (int)(i % (S * S));
	const float f = amp ? scale / fmaxf(amp[b], 1e-30f) : scale;
	bf16x8 v;
	for (int c = 0; c < CIN0; c++) v[c] = (bf16)0.0f;
	for (int c = 0; c < CREAL; c++) v[c] = (bf16)(x[((size_t)b * CREAL + c) * (S * S) + p] * f);
	if (amp) v[CREAL] = (bf16)(scale * amp[b]);
	*(bf16x8*)(out + i * CIN0) = v;
}

// Implicit-GEMM 3x3 periodic convolution on the matrix cores.
//   out[b][y][x][n] = sum_t sum_k in[b][y + DIR*d*(ky-1)][x + DIR*d*(kx-1)][k] * Wt[t][n][k]
// DIR = +1: forward (Wt = W[t][cout][cin]); DIR = -1: backward data (Wt = W^T[t][cin][cout]).
// MODE 0: out = bias + value, store GELU(out) (bf16 NHWC) and, with Z, out itself (fp32)
// MODE 1: out = bias + value, store fp32 planar [B][4][S][S] (first 4 channels), times
//         oscale (and a[b]^2 when amp is given)
// MODE 2: backward data: g = value * gelu'(zprev) -> bf16 NHWC (gradient of the previous z)
// A workgroup of CROWS waves works through a range of blocks of CROWS consecutive rows of one
// 64-pixel segment, a row each: the layer's weights are staged once in LDS, and with ROWS also, per
// block, the CROWS + 2 input rows that the taps read (each input row is read once from global memory
// instead of nine times), the next block's loaded into registers while this one is multiplied.  ROWS 1:
// dilation 1, rows of 66 pixels.  ROWS 2: other dilations at S = 64, whole rows; the block's rows are then
// dil apart (k -> dil k mod S runs through a class of S / gcd(dil, S) rows).  ROWS 0: the input fragments
// are loaded from global memory.
// The products are W in^T (rows: 16 output channels, columns: 16 pixels) and row i of channel tile t is
// channel 32 (t / 2) + 8 (i / 4) + 4 (t % 2) + i % 4, so that two tiles leave a lane with 8 consecutive
// channels of a pixel, which it writes at once, and the four lanes of a pixel 64 contiguous bytes.
// LDS: 16-byte channel chunk c of weight row n at chunk n CPP + (c ^ g(n)), of pixel px at chunk
// px CPP + (c ^ ((px / PPB) % CPP)) (CPP chunks per row or pixel, PPB pixels per 256 bytes): the 16 lanes
// of a fragment read (16 channels, 16 consecutive pixels) fall into 16 different 16-byte slots of a
// 256-byte bank line.
// What bounds it (512 images of 64 x 64, 64 -> 64 channels, ROWS 1): 191 us, of which the MFMAs alone 70
// (busy 42 %), the GELU about 60, reading and writing 536 MB at the rate of a copy 103; they overlap only in
// part.  It took 310 us with 2-byte stores (products in W^T, a channel per lane), weights staged again for every
// block and the rows staged with nothing else in flight; dilated layers, from global memory, 330.  The output
// bits are the same: taps and channels are summed in the same order.
constexpr int CROWS = 8;
constexpr int NCU = 256;           // CUs: with ROWS one workgroup runs on each (LDS), without two
template <int S, int KC, int NC, int DIR, int MODE, int ROWS, bool Z>
__global__ __launch_bounds__(64 * CROWS, ROWS ? 2 : 4) void k_conv_mfma(const bf16* __restrict__ in,
	const bf16* __restrict__ Wt, const float* __restrict__ bias, float* __restrict__ zout, bf16* __restrict__ aout,
	float* __restrict__ yout, const float* __restrict__ zprev, float oscale, int dil, const float* __restrict__ amp, int nblk)
{
	constexpr int NT = MODE == 1 ? 1 : NC / 16;   // 16-wide output-channel tiles (MODE 1: the real channels' one)
	constexpr int NR = 16 * NT;       // weight rows per tap
	constexpr int MT = SEGP / 16;     // 16-pixel tiles of a segment
	constexpr int SEG = S / SEGP;     // segments per image row
	constexpr int CPP = KC / 8;       // 16-byte channel chunks per weight row
	constexpr int KIN = DIR == 1 && KC == CIO ? CIN0 : KC;   // channels stored of the input
	constexpr int CPI = KIN / 8;      // 16-byte channel chunks per pixel
	constexpr int PPB = 16 / CPI;     // pixels per 256 bytes
	constexpr int PX = ROWS == 1 ? SEGP + 2 : SEGP;   // staged pixels of a row
	constexpr int NST = (CROWS + 2) * PX * CPI, NIT_ST = ROWS ? (NST + 64 * CROWS - 1) / (64 * CROWS) : 1;
	static_assert(MODE != 1 || CREAL == 4, "4 channels of a lane");
	static_assert(ROWS != 2 || S == SEGP, "whole rows");
	static_assert(KIN == KC || (CPI == 1 && KC == 32), "the stored channels are the first lanes' chunk");
	__shared__ __attribute__((aligned(16))) bf16x8 wl[9 * NR * CPP];
	__shared__ __attribute__((aligned(16))) bf16x8 xl[ROWS ? NST : 1];
	const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const int i16 = lane & 15, kq = lane >> 4;
	// weight row n, chunk c; pixel q of the staged rows, chunk c
	auto row_of = [](int t, int i) { return NT == 1 ? i : 32 * (t / 2) + 8 * (i / 4) + 4 * (t % 2) + i % 4; };
	auto wslot = [](int n, int c) {
		const int i4 = NT == 1 ? n / 4 : n / 8 % 4;        // i / 4
		return n * CPP + (c ^ ((CPP == 8 ? 2 * i4 + n / 2 % 2 : i4) % CPP));
	};
	auto xslot = [](int q, int c) { return q * CPI + (c ^ ((q / PPB) % CPI)); };
	const int lo = (int)((long long)nblk * blockIdx.x / gridDim.x), hi = (int)((long long)nblk * (blockIdx.x + 1) / gridDim.x);
	// block -> image, first pixel, row r = -1 ... CROWS
	auto b_of = [](int blk) { return blk / (SEG * (S / CROWS)); };
	auto x0_of = [](int blk) { return (blk / (S / CROWS)) % SEG * SEGP; };
	const int ncl = ROWS == 2 ? S / (dil & -dil) : S;      // rows of a class
	auto y_of = [&](int blk, int r) {
		const int k = blk % (S / CROWS) * CROWS;
		return ROWS == 2 ? (k / ncl + dil * (k % ncl + r + S)) & (S - 1) : (k + r) & (S - 1);
	};
	bf16x8 st[NIT_ST];
	auto load_rows = [&](int blk) {
		const int x0 = x0_of(blk);
		const bf16* src = in + (size_t)b_of(blk) * S * S * KIN;
#pragma unroll
		for (int k = 0; k < NIT_ST; k++) {
			const int q = threadIdx.x + k * 64 * CROWS;
			const int px = q / CPI, c = q % CPI;
			const int ys = y_of(blk, px / PX - 1), xs = ROWS == 1 ? (x0 - 1 + px % PX) & (S - 1) : px % PX;
			if (q < NST) st[k] = *(const bf16x8*)(src + (ys * S + xs) * KIN + c * 8);
		}
	};
	auto store_rows = [&]() {
#pragma unroll
		for (int k = 0; k < NIT_ST; k++) {
			const int q = threadIdx.x + k * 64 * CROWS;
			if (q < NST) xl[xslot(q / CPI, q % CPI)] = st[k];
		}
	};
	float bs[4 * NT];
	// the first block's rows, the weights and the bias are loaded together
	if constexpr (ROWS)
		if (lo < hi) load_rows(lo);
	constexpr int NWL = 9 * NR * CPP, NIT_W = (NWL + 64 * CROWS - 1) / (64 * CROWS);
	bf16x8 ws[NIT_W];
#pragma unroll
	for (int k = 0; k < NIT_W; k++) {
		const int v = threadIdx.x + k * 64 * CROWS;
		if (v < NWL) ws[k] = *(const bf16x8*)(Wt + ((size_t)(v / (NR * CPP)) * NC + v / CPP % NR) * KC + v % CPP * 8);
	}
	if constexpr (MODE != 2) {
#pragma unroll
		for (int k = 0; k < 4 * NT; k++) bs[k] = bias[row_of(k / 4, 4 * kq) + k % 4];
#pragma unroll
		for (int k = 0; k < 4 * NT; k++) asm volatile("" : "+v"(bs[k]));   // loaded before the loop over the blocks
	}
#pragma unroll
	for (int k = 0; k < NIT_W; k++) {
		const int v = threadIdx.x + k * 64 * CROWS;
		if (v < NWL) wl[v / (NR * CPP) * NR * CPP + wslot(v / CPP % NR, v % CPP)] = ws[k];
	}
	if constexpr (ROWS) store_rows();
	__syncthreads();
	// the results of a block: lane holds channels row_of(t, 4 kq) + r of pixel m 16 + i16
	f32x4 acc[MT][NT];
	auto finish = [&](int blk) {
		const int b = b_of(blk), x0 = x0_of(blk), y = y_of(blk, w);
		if constexpr (MODE == 1) {
			float osc = oscale;
			if (amp) osc *= amp[b] * amp[b];
			if (kq == 0)
#pragma unroll
				for (int m = 0; m < MT; m++)
#pragma unroll
					for (int r = 0; r < CREAL; r++)
						yout[((size_t)b * CREAL + r) * (S * S) + (size_t)y * S + x0 + m * 16 + i16] = osc * (acc[m][0][r] + bs[r]);
		} else {
#pragma unroll
			for (int m = 0; m < MT; m++) {
				const size_t o = (((size_t)b * S + y) * S + x0 + m * 16 + i16) * NC + kq * 8;
				bf16x8 v[NT / 2];
#pragma unroll
				for (int t = 0; t < NT; t++) {
					f32x4 zp = acc[m][t];
					if constexpr (MODE == 0) {
#pragma unroll
						for (int r = 0; r < 4; r++) zp[r] += bs[4 * t + r];
						if constexpr (Z) *(f32x4*)(zout + o + 32 * (t / 2) + 4 * (t % 2)) = zp;
#pragma unroll
						for (int r = 0; r < 4; r++) v[t / 2][t % 2 * 4 + r] = (bf16)gelu(zp[r]);
					} else {
						const f32x4 z = *(const f32x4*)(zprev + o + 32 * (t / 2) + 4 * (t % 2));
#pragma unroll
						for (int r = 0; r < 4; r++) v[t / 2][t % 2 * 4 + r] = (bf16)(zp[r] * gelu_grad(z[r]));
					}
				}
#pragma unroll
				for (int k = 0; k < NT / 2; k++) *(bf16x8*)(aout + o + 32 * k) = v[k];
			}
		}
	};
	// With ROWS the workgroup's waves keep step at the barriers; half of them write a block's results
	// only after the barriers, so that on each SIMD one wave's epilogue runs beside the other's MFMAs
	// (six layers, 512 images: 934 us without, 907 with it and the MFMAs' priority)
	const bool late = ROWS && __builtin_amdgcn_readfirstlane(w) >= CROWS / 2;
	for (int blk = lo; blk < hi; blk++) {
		const int b = b_of(blk), x0 = x0_of(blk), y = y_of(blk, w);
		if constexpr (ROWS)
			if (blk + 1 < hi) load_rows(blk + 1);
		if (late && blk > lo) finish(blk - 1);
#pragma unroll
		for (int m = 0; m < MT; m++)
#pragma unroll
			for (int t = 0; t < NT; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
		// K loop over the 9 taps x KC/32 channel blocks, the fragments of the next iteration
		// loaded while the MFMAs of this one run (two iterations per loop body: the fragments ping-pong
		// between two register sets)
		constexpr int KB = KC / 32, NIT = 9 * KB;
		bf16x8 zero;
#pragma unroll
		for (int q = 0; q < 8; q++) zero[q] = (bf16)0.0f;
		auto load_a = [&](int it, bf16x8* a) {
			const int tap = it / KB, kb = it % KB;
			if constexpr (ROWS) {
				// staged row 0 is row -1 of the block, staged pixel 0 is x0 - 1 (ROWS 1) or 0 (ROWS 2)
				const int row = (w + 1 + DIR * (tap / 3 - 1)) * PX, sh = DIR * (tap % 3 - 1);
				const int c = CPI == 1 ? 0 : kb * 4 + kq;
				const int p0 = row + 1 + sh + i16, q0 = i16 + dil * sh + 2 * S;
#pragma unroll
				for (int m = 0; m < MT; m++)
					a[m] = xl[ROWS == 1 ? xslot(p0 + m * 16, c) : xslot(row + ((q0 + m * 16) & (S - 1)), c)];
			} else {
				const int ys = (y + DIR * dil * (tap / 3 - 1) + 2 * S) & (S - 1);
				const int sh = DIR * dil * (tap % 3 - 1) + 2 * S;
				const bf16* rowp = in + ((size_t)b * S + ys) * S * KIN + (CPI == 1 ? 0 : kb * 32 + kq * 8);
#pragma unroll
				for (int m = 0; m < MT; m++)
					a[m] = *(const bf16x8*)(rowp + (size_t)((x0 + m * 16 + i16 + sh) & (S - 1)) * KIN);
			}
			if (CPI == 1 && kq)
#pragma unroll
				for (int m = 0; m < MT; m++) a[m] = zero;
		};
		auto load_w = [&](int it, bf16x8* wf) {
			const int tap = it / KB, kb = it % KB;
#pragma unroll
			for (int t = 0; t < NT; t++)
				wf[t] = wl[tap * NR * CPP + wslot(row_of(t, i16), kb * 4 + kq)];
		};
		bf16x8 a[MT], wf[NT];
		load_a(0, a);
		if constexpr (ROWS) load_w(0, wf);
		__builtin_amdgcn_s_setprio(1);   // the MFMAs before the other waves' epilogues
#pragma unroll(ROWS ? 2 : 1)
		for (int it = 0; it < NIT; it++) {
			bf16x8 an[MT], wn[NT];
			if constexpr (!ROWS) load_w(it, wf);
			load_a(it + 1 < NIT ? it + 1 : it, an);
			if constexpr (ROWS) {
				load_w(it + 1 < NIT ? it + 1 : it, wn);
				__builtin_amdgcn_sched_barrier(0);   // or the loads sink to their use
			}
#pragma unroll
			for (int m = 0; m < MT; m++)
#pragma unroll
				for (int t = 0; t < NT; t++) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t], a[m], acc[m][t], 0, 0, 0);
#pragma unroll
			for (int m = 0; m < MT; m++) a[m] = an[m];
#pragma unroll
			for (int t = 0; t < NT; t++)
				if constexpr (ROWS) wf[t] = wn[t];
		}
		__builtin_amdgcn_s_setprio(0);
		if (!late) finish(blk);
		if constexpr (ROWS)
			if (blk + 1 < hi) {
				__syncthreads();
				store_rows();
				__syncthreads();
			}
	}
	if (late && lo < hi) finish(hi - 1);
}

// Weight and bias gradients on the matrix cores, per workgroup:
//   part[blk][(t * CO + co) * CI + ci] = sum_p dz[p][co] * x[p + dil off_t][ci],
//   part[blk][9 CO CI + co] = sum_p dz[p][co]   (p over the workgroup's pixels)
// summed over the workgroups in a fixed order by k_wgrad_reduce (no atomics: the gradients are the
// same bit for bit from run to run).  The contraction runs over pixels: v_mfma_f32_16x16x32_bf16 with
// A = dz^T (16 channels co x 32 pixels) and B = x (32 pixels x 16 channels ci), products of bf16 values
// summed in fp32, as the sums over pixels on the VALU were.
// One workgroup of 8 waves per (image, 64-pixel segment, block of rows): a wave keeps the 9 taps (5
// and 4 where the layer has fewer tiles) of 32 x 16 channels in its accumulators.  The rows are staged
// in LDS by channel, pixels contiguous, so that a fragment is one 16-byte read: x three times, shifted
// by the three kx (fragments of a shifted row would not be aligned), in a ring of four rows (dil = 1:
// each row is staged once, while the previous one is multiplied), dz in two.  Channel ch, 8-pixel block
// k at word 36 ch + 4 (k ^ (ch / 8 % 8)): conflict-free for the fragment reads (pitch 36) and for the
// staging writes (8 lanes load the 64 channels of one pixel, and write 8 channel groups).
// Bound by the fragment reads and the staging (LDS) together with the matrix cores.  B = 32, N = 64,
// 64 x 64 channels: 21.8 us (443 TFLOP/s), 682 us with the sums on the VALU from fp32 rows in LDS.
constexpr int WPW = 36;              // LDS words per channel: 64 pixels of bf16 and 4 words of padding
__device__ __forceinline__ int wg_word(int ch, int k) { return ch * WPW + ((k ^ (ch / 8 % 8)) * 4); }
template <int S, int CI, int CO>
__global__ __launch_bounds__(512) void k_conv_wgrad(const bf16* __restrict__ x, const bf16* __restrict__ dz,
	float* __restrict__ part, int rows, int dil)
{
	constexpr int SEG = S / SEGP;
	constexpr int CIS = CI == CIO ? CIN0 : CI;   // channels stored of x
	constexpr int WCO = CO / 32, WCI = CI / 16, TG = 8 / (WCO * WCI);   // waves over co, ci and taps
	constexpr int NT = TG == 1 ? 9 : 5;                                 // taps per wave
	static_assert(WCO * WCI * TG == 8 && TG <= 2, "8 waves");
	constexpr int XW = CI * WPW, ZW = CO * WPW;
	constexpr int XI = 3 * (CI / 8) * 32, ZI = (CO / 8) * 32;           // staging items: 2 pixels x 8 channels
	static_assert(XI + ZI <= 1024, "two items per thread");
	__shared__ __attribute__((aligned(16))) unsigned xs[4][3][XW];
	__shared__ __attribute__((aligned(16))) unsigned zs[2][ZW];
	const int seg = blockIdx.x % SEG;
	const int b = blockIdx.x / SEG / (S / rows);
	const int y0 = (blockIdx.x / SEG % (S / rows)) * rows;
	const int x0 = seg * SEGP;
	const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, i16 = lane & 15, kq = lane >> 4;
	const int wco = w % WCO, wci = w / WCO % WCI, tg = w / (WCO * WCI);
	struct Item { uint4 a, b; };
	// items of x row yx (three shifts) and dz row yz (row indices modulo S)
	auto load = [&](int yx, int yz, Item* it) {
#pragma unroll
		for (int k = 0; k < 2; k++) {
			const int id = threadIdx.x + 512 * k;
			if (id >= XI + ZI) continue;
			const bool isz = id >= XI;
			const int e = isz ? id - XI : id % (XI / 3);
			const int sh = isz ? 0 : dil * (id / (XI / 3) - 1);
			const int nc = isz ? CO / 8 : CI / 8;
			const int c = e % nc, pr = e / nc;
			const bf16* src = isz ? dz + ((size_t)b * S + (yz & (S - 1))) * S * CO + c * 8
				: x + ((size_t)b * S + (yx & (S - 1))) * S * CIS + c * 8;
			const int st = isz ? CO : CIS;
			if (!isz && 8 * c >= CIS) {
				it[k].a = it[k].b = uint4{0, 0, 0, 0};
				continue;
			}
			it[k].a = *(const uint4*)(src + (size_t)((x0 + 2 * pr + sh) & (S - 1)) * st);
			it[k].b = *(const uint4*)(src + (size_t)((x0 + 2 * pr + 1 + sh) & (S - 1)) * st);
		}
	};
	auto store = [&](int xslot, int zslot, const Item* it) {
#pragma unroll
		for (int k = 0; k < 2; k++) {
			const int id = threadIdx.x + 512 * k;
			if (id >= XI + ZI) continue;
			const bool isz = id >= XI;
			const int e = isz ? id - XI : id % (XI / 3);
			const int nc = isz ? CO / 8 : CI / 8;
			const int c = e % nc, pr = e / nc;
			unsigned* d = (isz ? zs[zslot] : xs[xslot][id / (XI / 3)]) + wg_word(8 * c, pr / 4) + pr % 4;
			const unsigned* ua = (const unsigned*)&it[k].a;
			const unsigned* ub = (const unsigned*)&it[k].b;
#pragma unroll
			for (int q = 0; q < 4; q++) {
				d[(2 * q) * WPW] = (ua[q] & 0xffffu) | (ub[q] << 16);
				d[(2 * q + 1) * WPW] = (ua[q] >> 16) | (ub[q] & 0xffff0000u);
			}
		}
	};
	f32x4 acc[NT][2];
#pragma unroll
	for (int t = 0; t < NT; t++)
#pragma unroll
		for (int m = 0; m < 2; m++) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
	float bsum[2] = {0.f, 0.f};
	// one row of dz (zslot) against the x rows in slots (s0 + ky) & 3
	auto row = [&](int s0, int zslot) {
		bf16x8 a[2][2];
#pragma unroll
		for (int m = 0; m < 2; m++)
#pragma unroll
			for (int ks = 0; ks < 2; ks++) {
				a[m][ks] = *(const bf16x8*)&zs[zslot][wg_word(32 * wco + 16 * m + i16, 4 * ks + kq)];
				if (wci == 0 && tg == 0)
#pragma unroll
					for (int q = 0; q < 8; q++) bsum[m] += (float)a[m][ks][q];
			}
#pragma unroll
		for (int t = 0; t < NT; t++) {
			const int tap = tg * NT + t;
			if (tap < 9) {
				const unsigned* xr = xs[(s0 + tap / 3) & 3][tap % 3];
#pragma unroll
				for (int ks = 0; ks < 2; ks++) {
					const bf16x8 f = *(const bf16x8*)&xr[wg_word(16 * wci + i16, 4 * ks + kq)];
#pragma unroll
					for (int m = 0; m < 2; m++) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m][ks], f, acc[t][m], 0, 0, 0);
				}
			}
		}
	};
	Item it[2];
	if (dil == 1) {
		// x row y0 + r sits in slot (r + 1) & 3
		for (int r = -1; r <= 1; r++) {
			load(y0 + r + S, y0, it);
			store(r + 1, 0, it);
		}
		__syncthreads();
		for (int i = 0; i < rows; i++) {
			const bool more = i + 1 < rows;
			if (more) load(y0 + i + 2, y0 + i + 1, it);
			row(i, i & 1);
			// slot (i + 3) & 3 and the other dz row were last read before the previous barrier
			if (more) store((i + 3) & 3, (i + 1) & 1, it);
			__syncthreads();
		}
	} else {
		for (int i = 0; i < rows; i++) {
			const int y = y0 + i;
			__syncthreads();
			for (int r = -1; r <= 1; r++) {
				load(y + dil * r + 2 * S, y, it);
				store(r + 1, 0, it);
			}
			__syncthreads();
			row(0, 0);
		}
	}
	float* pb = part + (size_t)blockIdx.x * (9 * CO * CI + CO);
#pragma unroll
	for (int t = 0; t < NT; t++) {
		const int tap = tg * NT + t;
		if (tap < 9)
#pragma unroll
			for (int m = 0; m < 2; m++)
#pragma unroll
				for (int r = 0; r < 4; r++)
					pb[((size_t)tap * CO + 32 * wco + 16 * m + 4 * kq + r) * CI + 16 * wci + i16] = acc[t][m][r];
	}
	if (wci == 0 && tg == 0)
#pragma unroll
		for (int m = 0; m < 2; m++) {
			float v = bsum[m];
			v += __shfl_xor(v, 16);
			v += __shfl_xor(v, 32);
			if (kq == 0) pb[9 * CO * CI + 32 * wco + 16 * m + i16] = v;
		}
}

// dW[i] = sum_blk part[blk][i] (i < nw), db[i - nw] likewise (nw <= i < nw + nb): 8 threads share an
// element, thread c adds the blocks c, c + 8, ..., and the 8 sums are added in order (a read of part: 256
// workgroups of 64 x 64 channels, 38 MB, in 11 us; one thread per element took 32)
__global__ __launch_bounds__(256) void k_wgrad_reduce(const float* __restrict__ part, int nblk, int nw, int nb,
	float* __restrict__ dW, float* __restrict__ db)
{
	__shared__ float sh[8][32];
	const int c = threadIdx.x / 32, e = threadIdx.x % 32;
	const int i = blockIdx.x * 32 + e;
	const int stride = nw + nb;
	float s = 0.f;
	if (i < stride)
		for (int b = c; b < nblk; b += 8) s += part[(size_t)b * stride + i];
	sh[c][e] = s;
	__syncthreads();
	if (c || i >= stride) return;
	for (int k = 1; k < 8; k++) s += sh[k][e];
	if (i < nw) dW[i] = s;
	else db[i - nw] = s;
}

// loss = mean over elements of d^2 (per-workgroup partials into lpart, summed by k_loss_reduce),
// gradient with respect to the network output -> bf16 NHWC (CIO channels).  d = pred - target, or
// (pred - target) / (oscale a[b]^2) with amp.
template <int S>
__global__ __launch_bounds__(256) void k_loss_grad(const float* __restrict__ pred, const float* __restrict__ target,
	bf16* __restrict__ g, float* __restrict__ lpart, int B, float inv_n, float oscale, const float* __restrict__ amp)
{
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	const long long n = (long long)B * S * S;
	float part = 0.f;
	if (i < n) {
		const int b = (int)(i / (S * S)), p = (int)(i % (S * S));
		const float sc = amp ? oscale * amp[b] * amp[b] : 1.0f;
		bf16* o = g + i * CIO;
		for (int c = 0; c < CIO; c++) {
			float gv = 0.f;
			if (c < CREAL) {
				const size_t e = ((size_t)b * CREAL + c) * (S * S) + p;
				const float d = amp ? (pred[e] - target[e]) / sc : pred[e] - target[e];
				part += d * d;
				gv = amp ? 2.0f * d * inv_n : 2.0f * d * inv_n * oscale;   // d loss / d (network output)
			}
			o[c] = (bf16)gv;
		}
	}
	for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
	__shared__ float wsum[4];
	if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = part;
	__syncthreads();
	if (threadIdx.x == 0) lpart[blockIdx.x] = ((wsum[0] + wsum[1]) + (wsum[2] + wsum[3])) * inv_n;
}

// loss = sum of the per-block partials, in order (one workgroup of 256)
__global__ __launch_bounds__(256) void k_loss_reduce(const float* __restrict__ lpart, int n, float* __restrict__ loss)
{
	__shared__ float sh[256];
	float s = 0.f;
	for (int i = threadIdx.x; i < n; i += 256) s += lpart[i];
	sh[threadIdx.x] = s;
	__syncthreads();
	for (int w = 128; w > 0; w >>= 1) {
		if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
		__syncthreads();
	}
	if (threadIdx.x == 0) *loss = sh[0];
}

// Adam on fp32 master weights, then bf16 copies W[t][co][ci] and W^T[t][ci][co].
__global__ void k_adam(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v, const float* __restrict__ g,
	bf16* __restrict__ wb, bf16* __restrict__ wbt, int co_n, int ci_n, int co_real, int ci_real, int n,
	float lr, float b1, float b2, float eps, float bc1, float bc2, int is_bias)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	int co, ci, t;
	if (is_bias) { co = i; ci = 0; t = 0; }
	else { t = i / (co_n * ci_n); co = (i / ci_n) % co_n; ci = i % ci_n; }
	const bool live = co < co_real && (is_bias || ci < ci_real);
	float wv = w[i];
	if (live) {
		const float gi = g[i];
		const float mi = b1 * m[i] + (1 - b1) * gi;
		const float vi = b2 * v[i] + (1 - b2) * gi * gi;
		m[i] = mi;
		v[i] = vi;
		wv -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
	} else {
		wv = 0.f;
	}
	w[i] = wv;
	if (!is_bias) {
		wb[i] = (bf16)wv;
		wbt[((size_t)t * ci_n + ci) * co_n + co] = (bf16)wv;
	}
}

// bf16 copies of fp32 weights (after an upload)
__global__ void k_wcopy(const float* __restrict__ w, bf16* __restrict__ wb, bf16* __restrict__ wbt, int co_n, int ci_n, int n)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	const int t = i / (co_n * ci_n), co = (i / ci_n) % co_n, ci = i % ci_n;
	wb[i] = (bf16)w[i];
	wbt[((size_t)t * ci_n + ci) * co_n + co] = (bf16)w[i];
}

// surrogate midpoint step, elementwise over the [ncell][4][S][S] state; products and sums are
// rounded separately (no fused multiply-add), so the step equals its composition from single
// network evaluations bit for bit
__global__ void k_to_f32(const double* __restrict__ W, float* __restrict__ x, long long n)
{
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) x[i] = (float)W[i];
}
// C = Cv (+ D): the network's operator, plus the offset field D when one is set
__device__ __forceinline__ double op_value(const float* __restrict__ Cv, const float* __restrict__ D, long long i)
{
#pragma clang fp contract(off)
	return D ? (double)Cv[i] + (double)D[i] : (double)Cv[i];
}
// x = (float)(W + a C)
__global__ void k_half_f32(const double* __restrict__ W, const float* __restrict__ Cv, const float* __restrict__ D,
	double a, float* __restrict__ x, long long n)
{
#pragma clang fp contract(off)
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) x[i] = (float)(W[i] + a * op_value(Cv, D, i));
}
// out = W + a C
__global__ void k_update_f64(const double* __restrict__ W, const float* __restrict__ Cv, const float* __restrict__ D,
	double a, double* __restrict__ out, long long n)
{
#pragma clang fp contract(off)
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) out[i] = W[i] + a * op_value(Cv, D, i);
}

// gather cells idx[j] of W [*][CELL] into out [nsel][CELL] (CELL = 4 S S values)
template <typename V>
__global__ void k_gather_cells(const V* __restrict__ W, const int* __restrict__ idx, V* __restrict__ out, int nsel,
	int CELL)
{
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= (long long)nsel * CELL) return;
	const int j = (int)(i / CELL), e = (int)(i % CELL);
	out[i] = W[(size_t)idx[j] * CELL + e];
}

// res[0] = sum |a (+ D) - b|, res[1] = sum |b|, res[2] = sum |w|  (a and D fp32, b and w fp64), in two
// launches with a fixed summation order (the same sums bit for bit from run to run): RES_WG workgroups
// of 256 write partial sums part[wg][3] over a grid-stride range, then one workgroup adds them in order.
constexpr int RES_WG = 128;
__global__ __launch_bounds__(256) void k_l1_partial(const float* __restrict__ a, const float* __restrict__ D,
	const double* __restrict__ b, const double* __restrict__ w, long long n, double* __restrict__ part)
{
	__shared__ double sh[3][4];
	double d = 0, m = 0, s = 0;
	for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
		d += fabs(op_value(a, D, i) - b[i]);
		m += fabs(b[i]);
		s += fabs(w[i]);
	}
	for (int o = 32; o > 0; o >>= 1) {
		d += __shfl_xor(d, o);
		m += __shfl_xor(m, o);
		s += __shfl_xor(s, o);
	}
	if ((threadIdx.x & 63) == 0) {
		sh[0][threadIdx.x >> 6] = d;
		sh[1][threadIdx.x >> 6] = m;
		sh[2][threadIdx.x >> 6] = s;
	}
	__syncthreads();
	if (threadIdx.x < 3) {
		const int k = threadIdx.x;
		part[blockIdx.x * 3 + k] = ((sh[k][0] + sh[k][1]) + sh[k][2]) + sh[k][3];
	}
}

__global__ __launch_bounds__(64) void k_l1_final(const double* __restrict__ part, int nwg, double* __restrict__ res)
{
	if (threadIdx.x < 3) {
		double t = 0;
		for (int g = 0; g < nwg; g++) t += part[g * 3 + threadIdx.x];
		res[threadIdx.x] = t;
	}
}

} // namespace qbfcnn

using namespace qbfcnn;

static thread_local std::string g_cnn_err;
static int cnn_err(int c, const char* fmt, ...)
{
	char buf[512];
	va_list ap;
	va_start(ap, fmt);
	vsnprintf(buf, sizeof(buf), fmt, ap);
	va_end(ap);
	g_cnn_err = buf;
	return c;
}
#define HCHK(x)                                                              \
	do {                                                                     \
		hipError_t e_ = (x);                                                 \
		if (e_ != hipSuccess) return cnn_err(-2, "%s", hipGetErrorString(e_));  \
	} while (0)

struct qbf_cnn {
	int S = 64;                      // image side (the velocity grid N: 64 or 128)
	int maxB = 0;
	// training (qbf_cnn_gradients) works on batches of at most min(maxB, TRAIN_MAX) images: the
	// pre-activations and gradients are held for those only (inference batches may be larger)
	static constexpr int TRAIN_MAX = 256;
	int maxTrain = 0;
	hipStream_t own = nullptr;       // created by qbf_cnn_create, destroyed by qbf_cnn_destroy
	hipStream_t stream = nullptr;    // where work is launched (own, or the caller's)
	// per layer: fp32 master weights / grads / Adam moments, bf16 copies
	float *w[NL] = {}, *gw[NL] = {}, *mw[NL] = {}, *vw[NL] = {};
	float *bias[NL] = {}, *gb[NL] = {}, *mb[NL] = {}, *vb[NL] = {};
	bf16 *wb[NL] = {}, *wbt[NL] = {};
	// activations: x[l] = input of layer l (bf16 NHWC), z[l] = pre-activation (fp32 NHWC), l < NL-1
	bf16* x[NL] = {};
	float* z[NL] = {};
	bf16* g[NL] = {};     // gradient of z[l] (bf16 NHWC), g[NL-1] = gradient of the output
	float* loss = nullptr;
	// deterministic reductions: per-workgroup partials of the weight gradients of one layer and of the loss
	// image rows per workgroup of k_conv_wgrad: 16, fewer where that leaves less than one workgroup per
	// CU (a workgroup's first row is staged with two more, and every workgroup writes its partial sums,
	// so few rows cost more per row).  A training step at B = 32, N = 64: 781 us with 8 rows (256
	// workgroups), 801 with 16, 888 with 4
	int wg_rows(int B) const
	{
		int rows = 16;
		while (rows > 4 && B * (S / rows) * (S / SEGP) < 256) rows /= 2;
		return rows;
	}
	float* gpart = nullptr;
	float* lpart = nullptr;
	int dil[NL] = {1, 1, 1, 1, 1, 1};
	int norm = 0;                         // per-cell normalisation
	float* amp = nullptr;                 // per-cell amplitude [maxB]
	float *sx = nullptr, *sc = nullptr;   // surrogate step: network input / output, fp32 [maxB][4][S][S]
	double* sw = nullptr;                 // surrogate inhom step: state after the first half transport
	double* sw2 = nullptr;                // ... and after the collision step
	static constexpr int RMAX = 64;       // residual check: at most RMAX sampled cells
	int* sidx = nullptr;                  // sampled cell indices (device)
	double *swf = nullptr, *swc = nullptr; // Fourier state / exact collision of the sample (complex)
	// offset field D (fp32 [ncell][4][S][S], the caller's): the surrogate operator is net + D
	const float* off = nullptr;
	int offCells = 0;                     // the cell count D was given for
	float* soff = nullptr;                // D on the residual sample
	double* sres = nullptr;               // three sums of the residual, then their per-workgroup partials
	int step = 0;
	std::vector<void*> allocs;
	float* alloc_f(size_t n)
	{
		void* p = nullptr;
		if (hipMalloc(&p, n * sizeof(float)) != hipSuccess) return nullptr;
		allocs.push_back(p);
		if (hipMemset(p, 0, n * sizeof(float)) != hipSuccess) return nullptr;
		return (float*)p;
	}
	bf16* alloc_b(size_t n)
	{
		void* p = nullptr;
		if (hipMalloc(&p, n * sizeof(bf16)) != hipSuccess) return nullptr;
		allocs.push_back(p);
		if (hipMemset(p, 0, n * sizeof(bf16)) != hipSuccess) return nullptr;
		return (bf16*)p;
	}
	~qbf_cnn()
	{
		for (void* p : allocs) hipFree(p);
	}
};

static size_t wsize(int l) { return (size_t)9 * cout_of(l) * cin_of(l); }

extern "C" {

const char* qbf_cnn_last_error(void) { return g_cnn_err.c_str(); }

int qbf_cnn_create(int N, int maxBatch, qbf_cnn** out)
{
	if (!out || (N != 64 && N != 128) || maxBatch < 1)
		return cnn_err(-1, "qbf_cnn_create: N must be 64 or 128 and maxBatch >= 1");
	qbf_cnn* c = new qbf_cnn();
	const int S = N;
	c->S = N;
	c->maxB = maxBatch;
	c->maxTrain = maxBatch < qbf_cnn::TRAIN_MAX ? maxBatch : qbf_cnn::TRAIN_MAX;
	const size_t px = (size_t)maxBatch * S * S, pxt = (size_t)c->maxTrain * S * S;
	for (int l = 0; l < NL; l++) {
		const size_t nw = wsize(l), nb = cout_of(l);
		c->w[l] = c->alloc_f(nw); c->gw[l] = c->alloc_f(nw); c->mw[l] = c->alloc_f(nw); c->vw[l] = c->alloc_f(nw);
		c->bias[l] = c->alloc_f(nb); c->gb[l] = c->alloc_f(nb); c->mb[l] = c->alloc_f(nb); c->vb[l] = c->alloc_f(nb);
		c->wb[l] = c->alloc_b(nw); c->wbt[l] = c->alloc_b(nw);
		c->x[l] = c->alloc_b(px * (l ? CH : CIN0));
		c->g[l] = c->alloc_b(pxt * cout_of(l));
		if (l < NL - 1) c->z[l] = c->alloc_f(pxt * cout_of(l));
		if (!c->w[l] || !c->gw[l] || !c->mw[l] || !c->vw[l] || !c->bias[l] || !c->gb[l] || !c->mb[l] || !c->vb[l] ||
			!c->wb[l] || !c->wbt[l] || !c->x[l] || !c->g[l] || (l < NL - 1 && !c->z[l])) {
			delete c;
			return cnn_err(-3, "qbf_cnn_create: out of device memory");
		}
	}
	c->loss = c->alloc_f(1);
	size_t nwg = 0;
	for (int B = 1; B <= c->maxTrain; B++) {
		const size_t n = (size_t)B * (S / c->wg_rows(B)) * (S / SEGP);
		nwg = n > nwg ? n : nwg;
	}
	c->gpart = c->alloc_f(nwg * (9 * CH * CH + CH));
	c->lpart = c->alloc_f(pxt / 256 + 1);
	c->amp = c->alloc_f(maxBatch);
	c->sx = c->alloc_f(px * CREAL);
	c->sc = c->alloc_f(px * CREAL);
	c->soff = c->alloc_f((size_t)qbf_cnn::RMAX * CREAL * S * S);
	{
		void *p1 = nullptr, *p2 = nullptr;
		if (hipMalloc(&p1, px * CREAL * sizeof(double)) == hipSuccess) c->allocs.push_back(p1);
		else p1 = nullptr;
		if (hipMalloc(&p2, px * CREAL * sizeof(double)) == hipSuccess) c->allocs.push_back(p2);
		else p2 = nullptr;
		c->sw = (double*)p1;
		c->sw2 = (double*)p2;
	}
	{
		void *p1 = nullptr, *p2 = nullptr, *p3 = nullptr, *p4 = nullptr;
		const size_t cplx = (size_t)qbf_cnn::RMAX * CREAL * S * S * 2 * sizeof(double);
		if (hipMalloc(&p1, qbf_cnn::RMAX * sizeof(int)) == hipSuccess) c->allocs.push_back(p1); else p1 = nullptr;
		if (hipMalloc(&p2, cplx) == hipSuccess) c->allocs.push_back(p2); else p2 = nullptr;
		if (hipMalloc(&p3, cplx) == hipSuccess) c->allocs.push_back(p3); else p3 = nullptr;
		// the three sums, then RES_WG partial sums of each
		if (hipMalloc(&p4, 3 * (1 + RES_WG) * sizeof(double)) == hipSuccess) c->allocs.push_back(p4); else p4 = nullptr;
		c->sidx = (int*)p1;
		c->swf = (double*)p2;
		c->swc = (double*)p3;
		c->sres = (double*)p4;
	}
	if (!c->loss || !c->gpart || !c->lpart || !c->amp || !c->sx || !c->sc || !c->soff || !c->sw || !c->sw2 || !c->sidx || !c->swf || !c->swc || !c->sres) {
		delete c;
		return cnn_err(-3, "qbf_cnn_create: out of device memory");
	}
	if (hipStreamCreate(&c->own) != hipSuccess) {
		delete c;
		return cnn_err(-2, "hipStreamCreate failed");
	}
	c->stream = c->own;
	*out = c;
	return 0;
}

void qbf_cnn_destroy(qbf_cnn* c)
{
	if (!c) return;
	hipStreamSynchronize(c->stream);
	hipStreamDestroy(c->own);
	delete c;
}

int qbf_cnn_set_stream(qbf_cnn* c, void* s)
{
	if (!c) return cnn_err(-1, "bad argument");
	c->stream = s ? (hipStream_t)s : c->own;
	return 0;
}

// dilation per layer (1 <= d <= 16; NULL keeps the current ones) and per-cell normalisation (0/1)
int qbf_cnn_configure(qbf_cnn* c, const int* dil, int norm)
{
	if (!c || (norm != 0 && norm != 1)) return cnn_err(-1, "qbf_cnn_configure: bad argument");
	if (dil)
		for (int l = 0; l < NL; l++)
			if (dil[l] < 1 || dil[l] > 16) return cnn_err(-1, "qbf_cnn_configure: dilation must be in [1, 16]");
	if (dil)
		for (int l = 0; l < NL; l++) c->dil[l] = dil[l];
	c->norm = norm;
	return 0;
}

// parameter layout of the host buffer: for each layer, weights [9][cout_pad][cin_pad] then bias [cout_pad]
size_t qbf_cnn_param_count(void)
{
	size_t n = 0;
	for (int l = 0; l < NL; l++) n += wsize(l) + cout_of(l);
	return n;
}

int qbf_cnn_set_params(qbf_cnn* c, const float* host)
{
	if (!c || !host) return cnn_err(-1, "bad argument");
	size_t o = 0;
	for (int l = 0; l < NL; l++) {
		HCHK(hipMemcpy(c->w[l], host + o, wsize(l) * sizeof(float), hipMemcpyHostToDevice));
		o += wsize(l);
		HCHK(hipMemcpy(c->bias[l], host + o, cout_of(l) * sizeof(float), hipMemcpyHostToDevice));
		o += cout_of(l);
		const int n = (int)wsize(l);
		hipLaunchKernelGGL(k_wcopy, dim3((n + 255) / 256), dim3(256), 0, c->stream, c->w[l], c->wb[l], c->wbt[l],
			cout_of(l), cin_of(l), n);
		HCHK(hipGetLastError());
		HCHK(hipMemsetAsync(c->mw[l], 0, wsize(l) * sizeof(float), c->stream));
		HCHK(hipMemsetAsync(c->vw[l], 0, wsize(l) * sizeof(float), c->stream));
		HCHK(hipMemsetAsync(c->mb[l], 0, cout_of(l) * sizeof(float), c->stream));
		HCHK(hipMemsetAsync(c->vb[l], 0, cout_of(l) * sizeof(float), c->stream));
	}
	c->step = 0;
	HCHK(hipStreamSynchronize(c->stream));
	return 0;
}

int qbf_cnn_get_params(qbf_cnn* c, float* host, int grads)
{
	if (!c || !host) return cnn_err(-1, "bad argument");
	HCHK(hipStreamSynchronize(c->stream));
	size_t o = 0;
	for (int l = 0; l < NL; l++) {
		HCHK(hipMemcpy(host + o, grads ? c->gw[l] : c->w[l], wsize(l) * sizeof(float), hipMemcpyDeviceToHost));
		o += wsize(l);
		HCHK(hipMemcpy(host + o, grads ? c->gb[l] : c->bias[l], cout_of(l) * sizeof(float), hipMemcpyDeviceToHost));
		o += cout_of(l);
	}
	return 0;
}

} // extern "C"

// one layer's convolution: staged rows where the rows that a block's taps reach fit into LDS beside the weights
// (six layers of dilation 2, 512 images of 64 x 64: 1.02 ms, 2.25 ms from global memory), that is for dilation 1 and,
// at 64 x 64, for the dilations whose classes hold a whole block
template <int S, int KC, int NC, int DIR, int MODE, bool Z = false>
static void conv(qbf_cnn* c, int B, const bf16* in, const bf16* W, const float* bias, float* zout, bf16* aout, float* yout,
	const float* zprev, float oscale, int dil, const float* amp)
{
	const int nblk = B * (S / SEGP) * (S / CROWS);
	auto launch = [&](auto k, int nwg) {
		hipLaunchKernelGGL(k, dim3((unsigned)(nblk < nwg ? nblk : nwg)), dim3(64 * CROWS), 0, c->stream, in, W, bias, zout, aout,
			yout, zprev, oscale, dil, amp, nblk);
	};
	if (dil == 1) launch(k_conv_mfma<S, KC, NC, DIR, MODE, 1, Z>, NCU);
	else if (S == SEGP && S / (dil & -dil) >= CROWS) launch(k_conv_mfma<S, KC, NC, DIR, MODE, S == SEGP ? 2 : 0, Z>, NCU);
	else launch(k_conv_mfma<S, KC, NC, DIR, MODE, 0, Z>, 2 * NCU);
}

template <int S>
static int run_forward_t(qbf_cnn* c, const float* dIn, int B, float iscale, float* dOut, float oscale, bool train)
{
	const long long npx = (long long)B * S * S;
	const float* amp = c->norm ? c->amp : nullptr;
	if (c->norm) hipLaunchKernelGGL(k_cell_amp<S>, dim3(B), dim3(256), 0, c->stream, dIn, c->amp);
	hipLaunchKernelGGL(k_to_nhwc<S>, dim3((unsigned)((npx + 255) / 256)), dim3(256), 0, c->stream, dIn, c->x[0], B,
		iscale, amp);
	// hidden layers: with the pre-activations where a backward pass follows
	auto hidden = [&](auto first, int l) {
		constexpr int K = decltype(first)::value ? CIO : CH;
		if (train)
			conv<S, K, CH, 1, 0, true>(c, B, c->x[l], c->wb[l], c->bias[l], c->z[l], c->x[l + 1], nullptr, nullptr, 1.0f, c->dil[l],
				nullptr);
		else
			conv<S, K, CH, 1, 0>(c, B, c->x[l], c->wb[l], c->bias[l], nullptr, c->x[l + 1], nullptr, nullptr, 1.0f, c->dil[l],
				nullptr);
	};
	hidden(std::true_type{}, 0);
	for (int l = 1; l < NL - 1; l++) hidden(std::false_type{}, l);
	conv<S, CH, CIO, 1, 1>(c, B, c->x[NL - 1], c->wb[NL - 1], c->bias[NL - 1], nullptr, nullptr, dOut, nullptr, oscale,
		c->dil[NL - 1], amp);
	HCHK(hipGetLastError());
	return 0;
}

extern "C" {

static int run_forward(qbf_cnn* c, const float* dIn, int B, float iscale, float* dOut, float oscale, bool train)
{
	return c->S == 128 ? run_forward_t<128>(c, dIn, B, iscale, dOut, oscale, train)
	                   : run_forward_t<64>(c, dIn, B, iscale, dOut, oscale, train);
}

// out = oscale * net(iscale * in), planar fp32 [B][4][N][N] device arrays
int qbf_cnn_forward(qbf_cnn* c, const float* dIn, int B, float iscale, float* dOut, float oscale)
{
	if (!c || !dIn || !dOut || B < 1 || B > c->maxB) return cnn_err(-1, "qbf_cnn_forward: bad argument");
	return run_forward(c, dIn, B, iscale, dOut, oscale, false);
}

// gradients of loss = mean (out - target)^2 into the gradient buffers (no update); loss -> *hostLoss
} // extern "C"

template <int S>
static int gradients_t(qbf_cnn* c, const float* dIn, const float* dTarget, int B, float iscale, float oscale,
	float* dOut, float* hostLoss)
{
	int r = run_forward_t<S>(c, dIn, B, iscale, dOut, oscale, true);
	if (r) return r;
	const long long npx = (long long)B * S * S;
	const float inv_n = 1.0f / (float)(npx * CREAL);
	const int nlb = (int)((npx + 255) / 256);
	hipLaunchKernelGGL(k_loss_grad<S>, dim3((unsigned)nlb), dim3(256), 0, c->stream, dOut, dTarget, c->g[NL - 1],
		c->lpart, B, inv_n, oscale, c->norm ? c->amp : nullptr);
	hipLaunchKernelGGL(k_loss_reduce, dim3(1), dim3(256), 0, c->stream, c->lpart, nlb, c->loss);
	const int rows = c->wg_rows(B);
	const int nwb = B * (S / rows) * (S / SEGP);
	const dim3 wgrid(nwb);
	auto reduce = [&](int l) {
		const int nw = (int)wsize(l), nb = cout_of(l);
		hipLaunchKernelGGL(k_wgrad_reduce, dim3((unsigned)((nw + nb + 31) / 32)), dim3(256), 0, c->stream, c->gpart,
			nwb, nw, nb, c->gw[l], c->gb[l]);
	};
	// last layer: weight gradient, then data gradient into the last hidden pre-activation
	hipLaunchKernelGGL((k_conv_wgrad<S, CH, CIO>), wgrid, dim3(512), 0, c->stream, c->x[NL - 1], c->g[NL - 1], c->gpart, rows,
		c->dil[NL - 1]);
	reduce(NL - 1);
	conv<S, CIO, CH, -1, 2>(c, B, c->g[NL - 1], c->wbt[NL - 1], nullptr, nullptr, c->g[NL - 2], nullptr, c->z[NL - 2], 1.0f,
		c->dil[NL - 1], nullptr);
	for (int l = NL - 2; l >= 1; l--) {
		hipLaunchKernelGGL((k_conv_wgrad<S, CH, CH>), wgrid, dim3(512), 0, c->stream, c->x[l], c->g[l], c->gpart, rows,
			c->dil[l]);
		reduce(l);
		conv<S, CH, CH, -1, 2>(c, B, c->g[l], c->wbt[l], nullptr, nullptr, c->g[l - 1], nullptr, c->z[l - 1], 1.0f, c->dil[l],
			nullptr);
	}
	hipLaunchKernelGGL((k_conv_wgrad<S, CIO, CH>), wgrid, dim3(512), 0, c->stream, c->x[0], c->g[0], c->gpart, rows, c->dil[0]);
	reduce(0);
	HCHK(hipGetLastError());
	if (hostLoss) {
		HCHK(hipMemcpyAsync(hostLoss, c->loss, sizeof(float), hipMemcpyDeviceToHost, c->stream));
		HCHK(hipStreamSynchronize(c->stream));
	}
	return 0;
}

extern "C" {

int qbf_cnn_gradients(qbf_cnn* c, const float* dIn, const float* dTarget, int B, float iscale, float oscale,
	float* dOut, float* hostLoss)
{
	if (!c || !dIn || !dTarget || !dOut || B < 1 || B > c->maxTrain)
		return cnn_err(-1, "qbf_cnn_gradients: bad argument (1 <= B <= min(maxBatch, 256))");
	return c->S == 128 ? gradients_t<128>(c, dIn, dTarget, B, iscale, oscale, dOut, hostLoss)
	                   : gradients_t<64>(c, dIn, dTarget, B, iscale, oscale, dOut, hostLoss);
}

// one Adam step with the gradients of qbf_cnn_gradients
int qbf_cnn_adam(qbf_cnn* c, float lr, float b1, float b2, float eps)
{
	if (!c) return cnn_err(-1, "null cnn");
	c->step++;
	const float bc1 = 1.0f - powf(b1, (float)c->step), bc2 = 1.0f - powf(b2, (float)c->step);
	for (int l = 0; l < NL; l++) {
		const int co = cout_of(l), ci = cin_of(l);
		const int co_r = l == NL - 1 ? CREAL : CH, ci_r = l == 0 ? (c->norm ? CREAL + 1 : CREAL) : CH;
		const int n = (int)wsize(l);
		hipLaunchKernelGGL(k_adam, dim3((n + 255) / 256), dim3(256), 0, c->stream, c->w[l], c->mw[l], c->vw[l], c->gw[l],
			c->wb[l], c->wbt[l], co, ci, co_r, ci_r, n, lr, b1, b2, eps, bc1, bc2, 0);
		hipLaunchKernelGGL(k_adam, dim3((co + 255) / 256), dim3(256), 0, c->stream, c->bias[l], c->mb[l], c->vb[l],
			c->gb[l], nullptr, nullptr, co, 1, co_r, 1, co, lr, b1, b2, eps, bc1, bc2, 1);
	}
	HCHK(hipGetLastError());
	return 0;
}

// Midpoint collision step with the network in place of the collision operator, on physical
// states [ncell][4][N][N] (double, device):
//   C(W) ~ oscale * net(iscale * W),  W_half = W + dt/2 C(W),  out = W + dt C(W_half),
// then the FP64 moment correction of out - W (mask as qbf_moment_correct; 0 = none).
// Runs on the engine's stream; ncell may exceed maxBatch (processed in chunks).
int qbf_surrogate_collision_step(qbf_cnn* c, qbf_engine* e, const double* dW, int ncell, double dt, float iscale,
	float oscale, double L, int mask, double* dOut)
{
	if (!c || !e || !dW || !dOut || ncell < 1) return cnn_err(-1, "qbf_surrogate_collision_step: bad argument");
	if (qbf_engine_N(e) != c->S) return cnn_err(-1, "qbf_surrogate_collision_step: engine and network grids differ");
	if (c->off && ncell != c->offCells)
		return cnn_err(-1, "qbf_surrogate_collision_step: %d cells, but the offset field holds %d", ncell, c->offCells);
	const int S = c->S;
	if (dW == dOut) return cnn_err(-1, "qbf_surrogate_collision_step: in-place update not supported");
	hipStream_t saved = c->stream;
	c->stream = (hipStream_t)qbf_get_stream(e);
	int r = 0;
	for (int c0 = 0; c0 < ncell && !r; c0 += c->maxB) {
		const int nb = ncell - c0 < c->maxB ? ncell - c0 : c->maxB;
		const long long n = (long long)nb * CREAL * S * S;
		const size_t off = (size_t)c0 * CREAL * S * S;
		const dim3 g((unsigned)((n + 255) / 256)), b(256);
		hipLaunchKernelGGL(k_to_f32, g, b, 0, c->stream, dW + off, c->sx, n);
		r = run_forward(c, c->sx, nb, iscale, c->sc, oscale, false);
		if (r) break;
		const float* D = c->off ? c->off + off : nullptr;
		hipLaunchKernelGGL(k_half_f32, g, b, 0, c->stream, dW + off, c->sc, D, 0.5 * dt, c->sx, n);
		r = run_forward(c, c->sx, nb, iscale, c->sc, oscale, false);
		if (r) break;
		hipLaunchKernelGGL(k_update_f64, g, b, 0, c->stream, dW + off, c->sc, D, dt, dOut + off, n);
		if (hipGetLastError() != hipSuccess) r = cnn_err(-2, "surrogate step launch failed");
	}
	if (!r && mask && qbf_moment_correct(e, dW, dOut, ncell, L, mask))
		r = cnn_err(-2, "%s", qbf_last_error());
	c->stream = saved;
	return r;
}

// Residual of the surrogate on sampled cells of physical states W: the exact collision
// operator C = Cc + Cd of the engine (any precision) against C_net = oscale * net(iscale * W),
// summed over the nsample cells hostIdx[0..nsample-1]:
//   sums[0] = sum |C_net - C|,  sums[1] = sum |C|,  sums[2] = sum |W|.
// sums[0] / sums[1] is the relative error of the operator; dt * sums[0] / sums[2] the relative
// error one surrogate step adds to the state.  Synchronous (the sums are read back to the host).
int qbf_surrogate_residual(qbf_cnn* c, qbf_engine* e, const double* dW, int ncell, const int* hostIdx, int nsample,
	float iscale, float oscale, double* sums)
{
	if (!c || !e || !dW || !hostIdx || !sums || nsample < 1 || nsample > qbf_cnn::RMAX || nsample > c->maxB)
		return cnn_err(-1, "qbf_surrogate_residual: bad argument (1 <= nsample <= 64 and <= maxBatch)");
	if (qbf_engine_N(e) != c->S) return cnn_err(-1, "qbf_surrogate_residual: engine and network grids differ");
	if (c->off && ncell != c->offCells)
		return cnn_err(-1, "qbf_surrogate_residual: %d cells, but the offset field holds %d", ncell, c->offCells);
	const int S = c->S;
	for (int j = 0; j < nsample; j++)
		if (hostIdx[j] < 0 || hostIdx[j] >= ncell) return cnn_err(-1, "qbf_surrogate_residual: cell index out of range");
	hipStream_t saved = c->stream;
	c->stream = (hipStream_t)qbf_get_stream(e);
	int r = 0;
	const long long n = (long long)nsample * CREAL * S * S;
	double h[3] = {0, 0, 0};
	if (hipMemcpyAsync(c->sidx, hostIdx, nsample * sizeof(int), hipMemcpyHostToDevice, c->stream) != hipSuccess)
		r = cnn_err(-2, "index upload failed");
	if (!r) {
		hipLaunchKernelGGL(k_gather_cells<double>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, dW, c->sidx,
			c->sw, nsample, CREAL * S * S);
		if (c->off)
			hipLaunchKernelGGL(k_gather_cells<float>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, c->off,
				c->sidx, c->soff, nsample, CREAL * S * S);
		if (qbf_phys_to_fourier(e, c->sw, CREAL * nsample, c->swf) ||
			qbf_collision(e, c->swf, nsample, QBF_C, c->swc, nullptr, nullptr, nullptr, 1.0) ||
			qbf_fourier_to_phys(e, c->swc, CREAL * nsample, c->sw2))
			r = cnn_err(-2, "%s", qbf_last_error());
	}
	if (!r) {
		hipLaunchKernelGGL(k_to_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, c->sw, c->sx, n);
		r = run_forward(c, c->sx, nsample, iscale, c->sc, oscale, false);
	}
	if (!r) {
		hipLaunchKernelGGL(k_l1_partial, dim3(RES_WG), dim3(256), 0, c->stream, c->sc, c->off ? c->soff : nullptr,
			c->sw2, c->sw, n, c->sres + 3);
		hipLaunchKernelGGL(k_l1_final, dim3(1), dim3(64), 0, c->stream, c->sres + 3, RES_WG, c->sres);
		if (hipMemcpyAsync(h, c->sres, sizeof(h), hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
			hipStreamSynchronize(c->stream) != hipSuccess)
			r = cnn_err(-2, "residual read-back failed");
	}
	c->stream = saved;
	if (!r)
		for (int k = 0; k < 3; k++) sums[k] = h[k];
	return r;
}

// Offset field of the surrogate operator: C(W) ~ oscale * net(iscale * W) + D (D fp32, planar
// [ncell][4][N][N] device array, the same cells as the states passed to the surrogate calls; the
// pointer is kept until the next call; NULL: no offset).  The stepping and residual calls reject
// another cell count while D is set.
int qbf_surrogate_set_offset(qbf_cnn* c, const float* dD, int ncell)
{
	if (!c) return cnn_err(-1, "qbf_surrogate_set_offset: null network");
	if (dD && ncell < 1) return cnn_err(-1, "qbf_surrogate_set_offset: ncell must be >= 1");
	c->off = dD;
	c->offCells = dD ? ncell : 0;
	return 0;
}

// Strang step of the periodic inhomogeneous problem with the surrogate collision step:
// half transport (FP64, exact), surrogate midpoint collision step + moment correction, half
// transport.  ncell <= maxBatch (the intermediate states live in the network's buffers).
int qbf_surrogate_inhom_step_periodic(qbf_cnn* c, qbf_engine* e, const double* dW, int ncell, double L, double h,
	double dt, float iscale, float oscale, int mask, double* dOut)
{
	if (!c || !e || !dW || !dOut || ncell < 1 || ncell > c->maxB)
		return cnn_err(-1, "qbf_surrogate_inhom_step_periodic: bad argument (ncell must be in [1, maxBatch])");
	if (qbf_transport_periodic(e, dW, ncell, L, h, 0.5 * dt, c->sw)) return cnn_err(-2, "%s", qbf_last_error());
	int r = qbf_surrogate_collision_step(c, e, c->sw, ncell, dt, iscale, oscale, L, mask, c->sw2);
	if (r) return r;
	if (qbf_transport_periodic(e, c->sw2, ncell, L, h, 0.5 * dt, dOut)) return cnn_err(-2, "%s", qbf_last_error());
	return 0;
}

namespace {
struct SurrogateStepCall {
	qbf_cnn* c;
	qbf_engine* e;
	const double* W;
	int ncell;
	double L, h, dt;
	float iscale, oscale;
	int mask;
	double* out;
};
int surrogate_step_call(void* p)
{
	auto* a = (SurrogateStepCall*)p;
	return qbf_surrogate_inhom_step_periodic(a->c, a->e, a->W, a->ncell, a->L, a->h, a->dt, a->iscale, a->oscale,
		a->mask, a->out);
}
} // namespace

int qbf_graph_capture_surrogate_inhom_step_periodic(qbf_cnn* c, qbf_engine* e, const double* dW, int ncell, double L,
	double h, double dt, float iscale, float oscale, int mask, double* dOut, qbf_graph** g)
{
	if (!c || !e || !dW || !dOut || !g) return cnn_err(-1, "qbf_graph_capture_surrogate_inhom_step_periodic: null argument");
	SurrogateStepCall a{c, e, dW, ncell, L, h, dt, iscale, oscale, mask, dOut};
	if (qbf_graph_capture_calls(e, surrogate_step_call, &a, g)) return cnn_err(-2, "%s", qbf_last_error());
	return 0;
}

} // extern "C"
