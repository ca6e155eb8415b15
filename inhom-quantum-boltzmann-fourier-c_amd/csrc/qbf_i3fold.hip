// qbf_i3fold.hip -- the I3 part of CdInt over mirrored quadrature terms (N = 16, 32, 64).
//
// CdInt sums, over the quadrature terms q and the components i, j (src/collision.c:110-121,
// src/integrals.c:343-378),
//   out_j = sum_q sum_i eta_i F_i,q .* K_q[S_i .* F_j,q],   F_c,q = FFT2(pad(psi1_q W_c)), S_c = FFT2(pad W_c).
// psi1_q is a translation phase, E_q(k) = exp(i y_q k), and the Gauss-Legendre nodes come in pairs
// +-rho with equal weights: every term has a mirror q' with psi1_q' = conj(psi1_q), psi2_q' = psi2_q.
// With A_ij(k) = sum_{l+m=k} W_i(l) W_j(m) E_q(m) (the spectrum of S_i .* F_j,q) the mirror's is
//   A'_ij(k) = sum W_i(l) W_j(m) conj(E_q(m)) = conj(E_q(k)) A_ji(k),
// so the mirror's outputs need no K of their own:
//   out'_j(r) = conj(E_q(r)) IFFT2( sum_i eta_i S_i .* K_q[S_j .* F_i,q] )(r)
// (k runs over [-N, N-2] and r over the N x N box: neither the sums l + m = k nor k + n = r wrap on
// the 2N grid).  One pass over the 16 products K_q[S_i .* F_j,q] therefore serves both terms, with
// one IFFT2 per mirror output more and the N x N box of the sum over q kept in frequency space (D).
//
// What bounds it: in FP32 at N = 64 the line FFTs of the K applications on the VALU (72% busy with packed pairs,
// 80% with complex grids) and a barrier phase per exchange; in FP64 the operands' traffic (N = 32: 78,000 L2
// requests per us, 27% of them misses, 3.2 TB/s of HBM, VALU 47%; N = 64: 1.45 MB of HBM a product, 5.8 TB/s, VALU
// 36%).  A term pair costs 16 applications and 16 pruned IFFT2 of three quarters of a transform (packed pairs: 8
// and 4) instead of 32 (16) applications.  Strang steps term by term -> in pairs, with k_assemble and the batched
// loads that came with them: FP32 N = 64, 512 cells 327.9 -> 204.2 ms; FP64 N = 32, 128 cells 59.9 -> 44.4 ms; FP64
// N = 64, 16 cells 62.5 -> 43.1 ms; FP32 N = 128, 32 cells 76.6 -> 49.5 ms.
#pragma once
#include "qbf_kernels.hip"

namespace qbf {

// sign of component i in the I3 sums, diag(1, -1, -1, -1)
template <typename R> __device__ __forceinline__ R eta_sgn(int i) { return i == 0 ? R(1) : R(-1); }

// conj(E(r)) = ph[idx(l)] ph[N + 1 + idx(k)] (I3FoldArgs::phase of one term, staged in LDS)
template <int N> __device__ __forceinline__ constexpr int phase_idx(int x) { return x <= N / 2 ? x : x - N + 1; }

// d + v e, formed in 64 bits: the phases are held and applied as psi1 is in k_padfft.  (FP32 N = 64, 512 cells: 187.4
// ms per step, with phases and products in FP32 187.6; 193.1 with the phases of the box from a table in memory.)
template <typename R>
__device__ __forceinline__ cx<R> add_phased(cx<R> d, cx<R> v, double2 e)
{
	const double x = v.x, y = v.y;
	return mk<R>((R)((double)d.x + x * e.x - y * e.y), (R)((double)d.y + x * e.y + y * e.x));
}

// IFFT2 of v (R_b), multiplied by conj(E(r)) and added to D on the box of the N x N grid.
template <typename R, int N, class GE, bool EDGE, class XP>
__device__ __forceinline__ void mirror_add(cx<R>* v, const XP& X, const cx<R>* tw, int line, int p, const double2* ph, cx<R>* Dp)
{
	constexpr int G = GE::G, E = GE::E, P = GE::P;
	using El = typename XP::El;
	using MB = MirrorBox<N, G, E, EDGE>;
	line = opaque_lane(line);
	p = opaque_lane(p);
	line_bwd<R, GE>(v, p, tw);
	// whole waves skip the column pass (a branch that the compiler can see is uniform): they go on to the
	// next product's row pass meanwhile
	constexpr int LW = 64 / G;                  // lines per wave
	const int l0 = __builtin_amdgcn_readfirstlane(line);
	const bool box = l0 < N / 2 + (EDGE ? 1 : 0) || l0 + LW > P - N / 2;
	X.pass(
		[&](El* g, int c) {
#pragma unroll
			for (int s = 0; s < E; s++)
				if (padded_nonzero<E>(s) || (EDGE && s == E / 4)) XP::out(g[X.a(line, p + G * s)], v[s], c);
		},
		[&](const El* g, int c) { if (box) X.get_Cb(g, v, line, p, c); });
	if (!box) return;
	line_bwd<R, GE>(v, p, tw);
	__builtin_amdgcn_sched_barrier(0);
	const bool keep = unpad<N>(line) >= 0 || (EDGE && line == N / 2);
	const BufRef<cx<R>> Dr(Dp, MB::SIZE);
	const int d0 = keep ? MB::lane(line, p) : 0;
	const double2 pk = ph[N + 1 + (keep ? phase_idx<N>(line) : 0)];
	constexpr int NB = E / 2 + EDGE;            // elements in the box, EDGE: the last one in lane 0 only
	constexpr int BL = 4;                       // loads in flight together
#pragma unroll
	for (int b = 0; b < NB; b += BL) {
		cx<R> d[BL];
#pragma unroll
		for (int k = b; k < b + BL && k < NB; k++) {
			const int s = k < E / 4 ? k : (k < E / 2 ? k + E / 2 : E / 4);
			d[k - b] = Dr.get(d0, MB::elem(s) * (MB::DL * G));      // (lanes > 0, k = E / 2: not used)
		}
#pragma unroll
		for (int k = b; k < b + BL && k < NB; k++) {
			if (E == 8 && (k - b) % 2 == 0) __builtin_amdgcn_sched_barrier(0);
			const int s = k < E / 4 ? k : (k < E / 2 ? k + E / 2 : E / 4);
			const cx<R> x = add_phased<R>(d[k - b], v[s], cmul<double>(ph[phase_idx<N>(k == E / 2 ? N / 2 : p + G * s)], pk));
			if (keep && (k < E / 2 || p == 0)) Dr.put(d0, MB::elem(s) * (MB::DL * G), x);
		}
		__builtin_amdgcn_sched_barrier(0);
	}
}

// K_q application on v (R_b), ps: psi2 (C_i native)
template <typename R, class GE, class XP>
__device__ __forceinline__ void k_apply(cx<R>* v, const R* ps, const XP& X, const cx<R>* tw, int line, int p)
{
	ifft2_reg<R, GE>(v, X, tw, line, p);
	// keep the table and operand loads next to their use (hoisted above the line FFTs they would
	// keep E extra values live)
	__builtin_amdgcn_sched_barrier(0);
	const BufRef<R> psi(ps, GE::P * GE::P);
#pragma unroll
	for (int s = 0; s < GE::E; s++) {
		const R m = psi.get(threadIdx.x, s * GE::T);
		v[s].x *= m;
		v[s].y *= m;
	}
	fft2_reg<R, GE>(v, X, tw, line, p);
	__builtin_amdgcn_sched_barrier(0);
}

// The mirror sums of FP32 grids are kept per block of DBLOCK terms (added in FP64 afterwards,
// k_sum_mirror): their low frequencies are sums over the whole grid, and 256 terms added in FP32 there
// tripled the error of a step.  Error of a step with its conservation correction, N = 64, 512 and 300 cells (term
// by term 2.20e-10, 1.91e-10): blocks of 32: 2.11e-10, 1.94e-10; 16: 2.08e-10, 1.85e-10; 8: 2.07e-10, 1.81e-10.  The
// step of 512 cells takes 189.2, 189.8 and 190.5 ms (complex grids, 256 cells: 203.6, 203.9 and 211.4).
template <typename R> constexpr int DBLOCK = sizeof(R) == 4 ? 16 : 1 << 30;

// Workgroup -> (cell, group, term range) of the fold kernels; nmir: see I3FoldArgs::terms.  none: the launch
// is beyond the table's terms
struct FoldRange {
	int chunk, grp, cell, qa, qb, nmir;
	bool none;
	__device__ __forceinline__ FoldRange(const I3FoldArgs& a, int ngrp)
	{
		nmir = __builtin_amdgcn_readfirstlane(a.terms[0]);
		const int left = __builtin_amdgcn_readfirstlane(a.terms[1]) - a.q0;
		const int nq = left < a.nq ? left : a.nq;
		none = nq <= 0;
		const int lb = xcd_block();
		chunk = lb % a.nchunk;
		grp = (lb / a.nchunk) % ngrp;
		cell = lb / (a.nchunk * ngrp);
		qa = (int)(((long long)chunk * nq) / a.nchunk);
		qb = (int)(((long long)(chunk + 1) * nq) / a.nchunk);
	}
};

// Accumulator grid of a workgroup (R_b native), in registers.  MEM (FP64, N = 64): the grid and the
// accumulator together would take all registers of a CU (215 registers a lane spilled), so there it
// stays in global memory, read and written once per product by the thread that owns the element.
template <typename R, class GE, bool MEM>
struct FoldAcc {
	static constexpr int E = GE::E, T = GE::T;
	cx<R>* mem;
	cx<R> a[MEM ? 1 : E];
	__device__ __forceinline__ FoldAcc(cx<R>* m, bool resume) : mem(m)
	{
		if constexpr (!MEM) {
			if (resume) load_native<R, GE>(a, mem);
			else
#pragma unroll
				for (int u = 0; u < E; u++) a[u] = czero<R>();
		} else if (!resume) {
#pragma unroll
			for (int u = 0; u < E; u++) uni(mem, (long long)u * T)[threadIdx.x] = czero<R>();
		}
	}
	// element u += term(u, ld(u)), ld: the loads of the term
	template <int B, class Ld, class F>
	__device__ __forceinline__ void add(Ld ld, F term)
	{
		if constexpr (MEM) {
			const BufRef<cx<R>> m(mem, E * T);
			using L = decltype(ld(0));
			batched<E, B>([&](int u) { return Two<L, cx<R>>{ld(u), m.get(threadIdx.x, u * T)}; },
				[&](int u, const Two<L, cx<R>>& x) { m.put(threadIdx.x, u * T, cadd<R>(x.b, term(u, x.a))); });
		} else {
			// pinned: the sum is formed here (sunk below the mirror's branch, its operands would be spilled)
			using L = decltype(ld(0));
			batched<E, B>(ld, [&](int u, const L& x) { a[u] = pin<R>(cadd<R>(a[u], term(u, x))); });
		}
	}
	__device__ __forceinline__ void store() const
	{
		if constexpr (!MEM) store_native<R, GE>(mem, a);
	}
};

// Registers: at N <= 32 as many waves as the LDS exchange leaves room for (FP64 32: two workgroups
// of 4 waves a CU, up to 256 registers; the others 128)
template <typename R, int N> constexpr int FOLD_WPE = sizeof(R) == 8 && N == 32 ? 2 : 4;
// Elements of a load batch (two batches are in flight, see batched)
template <typename R, int N> constexpr int FOLD_B = sizeof(R) == 8 && N == 64 ? 2 : 4;

// Complex grids.  One workgroup per (cell, output j, term range): for every i
//   acc_j += eta_i F_i Y_ij  and  D_i += mirror(eta_j S_j Y_ij).
// acc [cell][4][nchunk], D [cell][4][4 nchunk nblk] (partial sums over j, the term ranges and blocks).  (All j in one
// workgroup need one mirror transform per i instead of four, but the four accumulators leave one
// wave per SIMD: strang step at N = 32, FP64, 128 cells 89 ms against 47 ms.)
template <typename R, int N, int T, bool SP>
__global__ __launch_bounds__(T, (FOLD_WPE<R, N>)) void k_i3fold(I3FoldArgs a)
{
	using GE = Geo<2 * N, T>;
	constexpr int P = GE::P, E = GE::E, G = GE::G, B = FOLD_B<R, N>;
	using XP = Xpose<R, GE, SP>;
	using MB = MirrorBox<N, G, E, false>;
	__shared__ typename XP::El lds[XP::SIZE];
	__shared__ cx<R> tw[TwTab<P, T>::SIZE];
	__shared__ double2 ph[2 * (N + 1)];         // the mirror's phases of the current term
	const FoldRange w(a, 4);
	if (w.none) return;
	load_twiddles<R, P, T>(tw, a.tw256);
	const int j = w.grp;
	const int t = threadIdx.x;
	const int line = GE::line(t), p = GE::lane(t);
	const size_t dstep = (size_t)4 * a.nchunk * a.nblk * MB::SIZE;
	cx<R>* Dp = (cx<R>*)a.D + 4 * w.cell * dstep + (long long)((j * a.nchunk + w.chunk) * a.nblk + a.resumeD - 1) * MB::SIZE;
	int nb = 0;                                 // blocks begun
	auto phase_of = [](const I3FoldArgs& a, int qq) { return (const double2*)a.phase + (size_t)(a.q0 + qq) * (2 * (N + 1)); };
	auto next_block = [&]() {
		Dp += MB::SIZE;
		nb++;
		for (int i = 0; i < 4; i++)
			for (int e = t; e < MB::SIZE; e += T) Dp[i * dstep + e] = czero<R>();
	};
	XP X{lds};
	FoldAcc<R, GE, SP> acc((cx<R>*)a.acc + (((size_t)w.cell * 4 + j) * a.nchunk + w.chunk) * (P * P), a.accumulate);
	cx<R> v[E];
	const cx<R>* Sh = (const cx<R>*)a.Shat + (size_t)w.cell * 4 * (P * P);
	const R ej = eta_sgn<R>(j);
	__syncthreads();
	for (int qq = w.qa; qq < w.qb; qq++) {
		const cx<R>* Fq = (const cx<R>*)a.F + ((size_t)w.cell * a.nq + qq) * 4 * (P * P);
		const R* ps = (const R*)a.psi2n + (size_t)(a.q0 + qq) * (P * P);
		const bool mir = a.q0 + qq < w.nmir;
		if ((qq - w.qa) % DBLOCK<R> == 0 && (qq > w.qa || !a.resumeD)) {
			// (the term's barriers are before the mirror's reads)
			next_block();
		}
#pragma unroll 1
		for (int i = 0; i < 4; i++) {
			{
				const BufRef<cx<R>> s(Sh + (size_t)i * (P * P), P * P), h(Fq + (size_t)j * (P * P), P * P);
				batched<E, B>([&](int u) { return Two<cx<R>, cx<R>>{s.get(t, u * T), h.get(t, u * T)}; },
					[&](int u, const Two<cx<R>, cx<R>>& x) { v[u] = cmul<R>(x.a, x.b); });
			}
			k_apply<R, GE>(v, ps, X, tw, line, p);
			// (this product's barriers are behind the previous term's reads of ph, the mirror's before this one's)
			double2 phv = make_double2(0, 0);
			if (i == 0 && mir && t < 2 * (N + 1)) phv = phase_of(a, qq)[t];
			{
				const R ei = eta_sgn<R>(i);
				const BufRef<cx<R>> f(Fq + (size_t)i * (P * P), P * P);
				acc.template add<B>([&](int u) { return f.get(t, u * T); },
					[&](int u, cx<R> x) { return cscale<R>(cmul<R>(x, v[u]), ei); });
			}
			if (i == 0 && t < 2 * (N + 1)) ph[t] = phv;
			if (mir) {
				const BufRef<cx<R>> s(Sh + (size_t)j * (P * P), P * P);
				batched<E, B>([&](int u) { return s.get(t, u * T); },
					[&](int u, cx<R> x) { v[u] = cscale<R>(cmul<R>(x, v[u]), ej); });
				mirror_add<R, N, GE, false>(v, X, tw, line, p, ph, Dp + i * dstep);
			}
		}
	}
	while (nb < a.nblk - a.resumeD) next_block();
	acc.store();
}

// Real grids packed in pairs (S, F: packed W_0 + i W_1, W_2 + i W_3).  One workgroup per (cell, packed
// output pair J, packed instance pair p, term range).  The product of component i of S with the packed
// pair J of F carries the outputs 2J, 2J+1:
//   acc_J += eta_i F_i Y (real times complex),  b_i = eta_2J S_2J Re Y + eta_2J+1 S_2J+1 Im Y,
// for i = 2p, 2p+1, then D_p += mirror(b_2p + i b_2p+1).
// acc [cell][2][2 nchunk], D [cell][2][2 nchunk nblk] (partial sums over p, over J, the term ranges and
// blocks).
// Four workgroups share a cell's S and F grids, as many cells as an XCD's L2 holds (with both p in one
// workgroup: 457 KB of HBM traffic per product instead of 115 when the split was chosen, FP32, N = 64; 179 now).
template <typename R, int N, int T, bool SP>
__global__ __launch_bounds__(T, (FOLD_WPE<R, N>)) void k_i3fold_pair(I3FoldArgs a)
{
	using GE = Geo<2 * N, T>;
	constexpr int P = GE::P, E = GE::E, G = GE::G, B = FOLD_B<R, N>;
	using XP = Xpose<R, GE, SP>;
	using MB = MirrorBox<N, G, E, true>;
	__shared__ typename XP::El lds[XP::SIZE];
	__shared__ cx<R> tw[TwTab<P, T>::SIZE];
	__shared__ double2 ph[2 * (N + 1)];         // the mirror's phases of the current term
	const FoldRange w(a, 4);
	if (w.none) return;
	load_twiddles<R, P, T>(tw, a.tw256);
	const int J = w.grp >> 1, pr = w.grp & 1;
	const int t = threadIdx.x;
	const int line = GE::line(t), p = GE::lane(t);
	cx<R>* Dp = (cx<R>*)a.D + ((((size_t)w.cell * 2 + pr) * 2 + J) * a.nchunk + w.chunk) * a.nblk * MB::SIZE +
		(long long)(a.resumeD - 1) * MB::SIZE;
	int nb = 0;                                 // blocks begun
	auto phase_of = [](const I3FoldArgs& a, int qq) { return (const double2*)a.phase + (size_t)(a.q0 + qq) * (2 * (N + 1)); };
	auto next_block = [&]() {
		Dp += MB::SIZE;
		nb++;
		for (int e = t; e < MB::SIZE; e += T) Dp[e] = czero<R>();
	};
	XP X{lds};
	FoldAcc<R, GE, SP> acc((cx<R>*)a.acc + (((size_t)w.cell * 2 + J) * 2 * a.nchunk + pr * a.nchunk + w.chunk) * (P * P),
		a.accumulate);
	cx<R> v[E];
	const cx<R>* Sh = (const cx<R>*)a.Shat + (size_t)w.cell * 2 * (P * P);
	const R ei = pr ? R(-1) : R(1);              // eta_2p (eta_2p+1 = -1)
	const R ea = J ? R(-1) : R(1);               // eta_2J (eta_2J+1 = -1)
	__syncthreads();
	for (int qq = w.qa; qq < w.qb; qq++) {
		const cx<R>* Fq = (const cx<R>*)a.F + ((size_t)w.cell * a.nq + qq) * 2 * (P * P);
		const R* ps = (const R*)a.psi2n + (size_t)(a.q0 + qq) * (P * P);
		const cx<R>* Sp = Sh + (size_t)pr * (P * P);
		const cx<R>* SJ = Sh + (size_t)J * (P * P);
		const cx<R>* Fp = Fq + (size_t)pr * (P * P);
		const cx<R>* FJ = Fq + (size_t)J * (P * P);
		const bool mir = a.q0 + qq < w.nmir;
		if ((qq - w.qa) % DBLOCK<R> == 0 && (qq > w.qa || !a.resumeD)) {
			// (the term's barriers are before the mirror's reads)
			next_block();
		}
		R bx[E];
		// v = component c of the instance pair times F_J
		auto product = [&](int c) {
			const BufRef<R> s((const R*)Sp, 2 * P * P);
			const BufRef<cx<R>> h(FJ, P * P);
			batched<E, B>([&](int u) { return Two<cx<R>, R>{h.get(t, u * T), s.get(2 * t, 2 * u * T + c)}; },
				[&](int u, const Two<cx<R>, R>& x) { v[u] = cscale<R>(x.a, x.b); });
		};
		auto accumulate = [&](int c, R eta) {
			const BufRef<R> f((const R*)Fp, 2 * P * P);
			acc.template add<B>([&](int u) { return f.get(2 * t, 2 * u * T + c); },
				[&](int u, R x) { return cscale<R>(v[u], eta * x); });
		};
		product(0);
		k_apply<R, GE>(v, ps, X, tw, line, p);
		// (the barriers of this product are behind the previous term's reads of ph, those of the next before this one's)
		double2 phv = make_double2(0, 0);
		if (mir && t < 2 * (N + 1)) phv = phase_of(a, qq)[t];
		accumulate(0, ei);
		if (t < 2 * (N + 1)) ph[t] = phv;
		{
			const BufRef<cx<R>> s(SJ, P * P);
			batched<E, B>([&](int u) { return s.get(t, u * T); },
				[&](int u, cx<R> y) {
					bx[u] = (ea * y.x) * v[u].x - y.y * v[u].y;
					asm volatile("" : "+v"(bx[u]));
				});
		}
		product(1);
		k_apply<R, GE>(v, ps, X, tw, line, p);
		accumulate(1, R(-1));
		if (mir) {
			const BufRef<cx<R>> s(SJ, P * P);
			batched<E, B>([&](int u) { return s.get(t, u * T); },
				[&](int u, cx<R> y) { v[u] = mk<R>(bx[u], (ea * y.x) * v[u].x - y.y * v[u].y); });
			mirror_add<R, N, GE, true>(v, X, tw, line, p, ph, Dp);
		}
		__builtin_amdgcn_sched_barrier(0);
	}
	while (nb < a.nblk - a.resumeD) next_block();
	acc.store();
}

} // namespace qbf
