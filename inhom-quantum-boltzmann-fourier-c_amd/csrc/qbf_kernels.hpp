// qbf_kernels.hpp -- argument blocks shared by the HIP kernels and the host engine.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qbf {

// Pruned 2-D FFT of zero-padded, optionally pre-multiplied N x N Fourier grids:
//   out[o] = FFT2( pad( pre_q .* src ) )        (R_b native order, P = 2N)
// o = (cell * nq + qq) * nslot + slot, src grid = src[cell * nsrc + srcOfSlot[slot]],
// pre = pre[q0 + qq] (none / real N*N / complex N*N).
struct PadFFTArgs {
	void* xs;             // per-workgroup scratch grids (N = 128)
	const double2* src;
	int nsrc;
	const void* pre;
	int preKind;          // 0 none, 1 real double, 2 complex double2
	int q0, nq;
	int nslot;
	int srcOfSlot[4];
	int ngrid;            // ncell * nq * nslot grids, two per workgroup
	void* out;
	const int* live;      // launches with q0 at or beyond *live do nothing (null: none)
	const double2* tw256;
};

// I1-type accumulation (I1 for Cc, I1 with FourierI4 tables for I4):
//   out[cell][inst] = FFT2( sum_g psi1_g .* IFFT2( (fa*Fhat + fb) .* FFT2(pad(phi_g .* src)) ) )
struct I1Args {
	void* xs;             // per-workgroup scratch grids (N = 128)
	const double2* src;   // [ncell][nsrc][N*N]
	int nsrc;
	const void* Fhat;     // [ncell][nFh][P*P] R_b native
	int nFh;
	double fa, fb;
	const double* phi;    // [nterm][N*N]
	const void* psi1n;    // [nterm][P*P] C_i native
	int nterm;
	int ninst;
	int instSrc[8];
	int instFh[8];
	int nchunk;           // terms split into nchunk ranges (partial sums, added by k_combine)
	void* out;            // [ncell][ninst][nchunk][P*P] R_b native
	const double2* tw256;
};

// I2 accumulation: out[cell][inst] = sum_q FFT2(pad(psi1_q .* f)) .* FFT2(pad(psi2_q .* g))
struct I2Args {
	void* xs;             // per-workgroup scratch grids (N = 128)
	const double2* src;
	int nsrc;
	const double* psi1;   // [nterm][N*N]
	const double* psi2;   // [nterm][N*N]
	const double2* psic;  // [nterm][N*N] psi1 + i psi2 (paired path)
	int nterm;
	int ninst;
	int instF[8];
	int instG[8];
	int nchunk;           // terms split into nchunk ranges (partial sums, added by k_combine)
	void* out;            // [ncell][ninst][nchunk][P*P] R_b native
	const double2* tw256;
};

// I3 accumulation over a range of quadrature terms (the dominant kernel):
//   acc[cell][out][chunk] (+)= sum_{qq in chunk} sum_inst w * F[f] .* K_q[ Shat[g] .* F[h] ],
//   K_q[X] = FFT2( psi2_q .* IFFT2(X) ).
struct I3Args {
	void* xs;             // per-workgroup scratch grids (N = 128)
	const void* Shat;     // [ncell][nS][P*P] R_b native
	int nS;
	const void* F;        // [ncell][nq][nF][P*P] R_b native
	int nF, nq, q0;
	const void* psi2n;    // [nqTotal][P*P] C_i native
	int nout;
	int ninst[4];
	int instF[4][4], instS[4][4], instH[4][4];
	double instW[4][4];
	int nchunk;
	int accumulate;
	void* acc;            // [ncell][nout][nchunk][P*P] R_b native
	const double2* tw256;
};

// I3 part of CdInt over mirrored quadrature terms (k_i3fold, k_i3fold_big): the layouts of F, S and
// psi2n are I3Args'; the results are partial sums acc [cell][no][na] and D [cell][no][nd] (no = 4 outputs, or 2
// packed pairs; na and nd follow from the kernel's split, see there).
struct I3FoldArgs {
	void* xs;             // per-workgroup scratch grids (N = 128)
	const void* Shat;     // [ncell][no][P*P] R_b native
	const void* F;        // [ncell][nq][no][P*P] R_b native
	int nq, q0;
	const int* terms;     // [0]: terms with an index below it stand for a mirrored pair, [1]: terms to take in all
	                      // (read on the device: a captured launch follows a table that is replaced)
	const void* psi2n;    // [nqTotal][P*P] C_i native
	const void* phase;    // [nmir][2][N+1] conj(E) along l and along k, frequencies 0 .. N/2, -N/2 .. -1, 64 bits
	int nchunk;
	int accumulate;
	void* acc;            // [ncell][no][na][P*P] R_b native
	void* D;              // [ncell][no][nd] mirror sums (MirrorBox), nblk blocks of terms per workgroup
	int nblk;
	int resumeD;          // the terms of this launch continue block 0 (nblk = 1) of the launch before
	const double2* tw256;
};

// One product term of the physical-domain combination:
//   coef * (X ? ax*X + bx : 1) .* (Y ? sum_{n<nsum} Y[n*ysum] : 1)
struct CTerm {
	const void* X;
	long long xcell;
	const void* Y;
	long long ycell;
	long long ysum;
	int nsum;
	double coef, ax, bx;
};

// Combine terms per output component, IFFT2, extract the N x N block, then
//   out = base + cf * (outScale * value + CB(Wcb, Bext)).
struct CombineArgs {
	void* xs;             // per-workgroup scratch grids (N = 128)
	const CTerm* terms;   // [nout][maxTerms]
	int maxTerms;
	int nterm[4];
	int nout;
	int outComp[4];       // component index written for each output
	double outScale;
	double2* out;         // [ncell][4][N*N]
	const double2* base;  // [ncell][4][N*N] or null
	const double2* Wcb;   // [ncell][4][N*N] or null (no magnetic rotation)
	const double* Bext;   // [ncell][3] (used when Wcb != null)
	double cf;
	// frequency-space sums of the mirrored I3 terms (k_sum_mirror), added to the extracted value with the
	// factor Dcoef[o]; null: none.  Dpair 0: [cell][4], the component's grid; 1: [cell][2], packed
	// pairs of Hermitian spectra.  Dstep: elements between the grids of a cell, Dcell: between cells.
	const double2* D;
	int Dpair;
	long long Dcell, Dstep;
	double Dcoef[4];
	const double2* tw256;
};

// Physical-domain sum of a collision evaluation (k_assemble), all grids in R_b native order.  pairAB:
// A [ncell][2][nchA] = (A_2 + i A_3, A_1), B [ncell][2][nchB] = (B_0 + i B_1, B_2 + i B_3) packed real
// grids; otherwise A [ncell][3][nchA], B [ncell][4][nchB].  pairAcc: acc [ncell][2][nchAcc] packed.
struct AssembleArgs {
	const void* What;     // [ncell][4]
	const void* A;        // null: no Cc
	const void* B;        // null: no Cd
	const void* S;        // [ncell][4][nchS]
	const void* acc;      // [ncell][4 or 2][nchAcc]
	int nchA, nchB, nchS, nchAcc;
	int pairAB, pairAcc;
	double c4, c2;
	void* V;              // [ncell][4]
	long long n, PP;      // n = ncell * PP
};

} // namespace qbf
