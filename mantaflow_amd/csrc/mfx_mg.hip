// Multigrid preconditioner for the pressure CG.
//
// Structure after the reference's GridMg (multigrid.cpp, Dick et al. 2015):
// vertex-centred levels of size (n+2)/2 until every axis is <= 5 or a level
// has <= 1000 vertices (:220-262), full-weighting restriction and
// (tri)linear interpolation with weights 1/2^(#odd coordinates) (:904-959),
// Galerkin coarse operators A_l = R A_{l-1} I stored as a symmetric 27-point
// (9-point in 2D) stencil (:580-666), trivial rows scaled by 1e-6 (:350-415),
// one multi-colour Gauss-Seidel pre- and post-sweep with reversed colour
// order on the way up so that the V-cycle is symmetric (:668-737).
//
// Differences, chosen for the GPU:
//  * coarse vertices are selected by a parallel rule: a coarse vertex is
//    active if any active fine vertex lies in its restriction stencil, and it
//    is dropped again when its Galerkin diagonal vanishes.  The reference's
//    sequential bucket-heap selection (:520-578) keeps the interpolation full
//    rank; here rank-deficient directions are harmless because
//  * the coarsest level is solved exactly by a dense generalised inverse in
//    FP64 (blocked symmetric sweep of the active operator with zero pivots
//    dropped, on the GPU once per hierarchy, applied as a GEMV) instead of a
//    sequential FP64 Jacobi-PCG (:796-902).  This also makes the V-cycle well
//    defined for pure-Neumann problems without pinning a pressure value.
//  * level 0 is matrix-free: its stencil comes from the per-cell matrix code.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "mfx_batch.h"
#include "mfx_mg.h"
#include "mfx_prof.h"

namespace mfx {

__device__ __host__ inline int oddc(int i, int j, int k) { return (i & 1) + (j & 1) + (k & 1); }
// 1/2^(#odd coordinates): exact powers of two (same values as the division)
__device__ inline float wgt(int i, int j, int k) {
	const int o = oddc(i, j, k);
	return o == 0 ? 1.0f : (o == 1 ? 0.5f : (o == 2 ? 0.25f : 0.125f));
}

static inline LvDev lvdev(const MgLevel& l) {
	return LvDev{l.nx, l.ny, l.nz, l.sy, l.sz, l.n, fastdiv_make((unsigned)l.nx), fastdiv_make((unsigned)l.ny)};
}

__device__ inline bool l0_active(uint8_t c) { return (c & 7) != 0; }
__device__ inline float l0_diag(uint8_t c) { return (c & 128) ? (float)(c & 7) * 1e-6f : (float)(c & 7); }
__device__ inline float l0_scale(uint8_t c) { return (c & 128) ? 1e-6f : 1.0f; }

// ---------------------------------------------------------------------------
// hierarchy construction
// ---------------------------------------------------------------------------
// Coarse vertices, a parallel restatement of genCoarseGrid
// (multigrid.cpp:520-578).  There, a fine vertex with one undecided parent
// left activates it, and a fine vertex popped with several free parents
// activates the first and removes the others, so each fine vertex adds at
// most one parent beyond the "standard" ones.  Here, in two passes:
//  1. standard: V is active iff its injection point, fine vertex 2V, is active;
//  2. every active fine vertex activates its first (loop-order) parent that
//     is not standard.
// Parents of walls and obstacles (fine 2V inactive) are thereby active where
// a fine vertex needs them, but a fine vertex never turns on several weak,
// nearly dependent parents - those make the Galerkin operator ill-conditioned.
__device__ inline bool fine_active(const uint8_t* code, const uint8_t* ftype, long long u) {
	return code ? l0_active(code[u]) : (ftype[u] != 0);
}
__global__ void k_mg_activate(LvDev c, LvDev f, int is3d, const uint8_t* __restrict__ code,
                              const uint8_t* __restrict__ ftype, uint8_t* __restrict__ ctype) {
	for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < c.n;
	     v += (long long)gridDim.x * blockDim.x) {
		const int i = (int)(v % c.nx), j = (int)((v / c.nx) % c.ny), k = (int)(v / c.sz);
		const int ux = 2 * i, uy = 2 * j, uz = is3d ? 2 * k : 0;
		bool act = false;
		if (ux < f.nx && uy < f.ny && uz < f.nz) act = fine_active(code, ftype, ux + f.sy * uy + f.sz * uz);
		ctype[v] = act ? 1 : 0;
	}
}
__global__ void k_mg_cover(LvDev c, LvDev f, int is3d, const uint8_t* __restrict__ code,
                           const uint8_t* __restrict__ ftype, uint8_t* __restrict__ ctype) {
	for (long long u = blockIdx.x * (long long)blockDim.x + threadIdx.x; u < f.n;
	     u += (long long)gridDim.x * blockDim.x) {
		if (!fine_active(code, ftype, u)) continue;
		const int ux = (int)(u % f.nx), uy = (int)((u / f.nx) % f.ny), uz = (int)(u / f.sz);
		long long pick = -1;
		for (int iz = uz / 2; iz <= (uz + 1) / 2 && pick < 0; iz++)
			for (int iy = uy / 2; iy <= (uy + 1) / 2 && pick < 0; iy++)
				for (int ix = ux / 2; ix <= (ux + 1) / 2; ix++) {
					if (ix >= c.nx || iy >= c.ny || iz >= c.nz) continue;
					const long long pi = ix + c.sy * iy + c.sz * iz;
					// pass-1 marks (1) decide "standard"; pass-2 marks (3) written by
					// other fine vertices are not standard either, so the choice
					// does not depend on the order of the writes
					if (ctype[pi] != 1) {
						pick = pi;
						break;
					}
				}
		if (pick >= 0) ctype[pick] = 3;
	}
}
__global__ void k_mg_cover_done(LvDev c, uint8_t* __restrict__ ctype) {
	for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < c.n;
	     v += (long long)gridDim.x * blockDim.x)
		if (ctype[v] == 3) ctype[v] = 1;
}

// the fine operator: level 0 from the code (7-point), coarse levels from the
// symmetric storage
struct FineOp {
	const uint8_t* code;  // level 0 if non-null
	const float* A;       // coarse storage otherwise
	const uint8_t* type;
	LvDev f;
};

// Interpolation along one axis seen from a fine vertex at offset dd (-1, 0,
// 1) of coarse vertex V's injection point: the three couplings (lower, own,
// upper) of the fine row onto the coarse offsets -1, 0, 1 of V.  A fine
// vertex of even coordinate has one parent (weight 1), of odd coordinate two
// (weight 1/2 each).
struct AxisW {
	double l0, c0, l1, c1, u1, c2, u2;
	__device__ explicit AxisW(int dd)
	    : l0(dd < 0 ? 1.0 : (dd == 0 ? 0.5 : 0.0)),
	      c0(dd < 0 ? 0.5 : 0.0),
	      l1(dd < 0 ? 0.0 : (dd == 0 ? 0.5 : 1.0)),
	      c1(dd == 0 ? 1.0 : 0.5),
	      u1(dd < 0 ? 1.0 : (dd == 0 ? 0.5 : 0.0)),
	      c2(dd > 0 ? 0.5 : 0.0),
	      u2(dd < 0 ? 0.0 : (dd == 0 ? 0.5 : 1.0)) {}
	__device__ void fold(double& l, double& c, double& u) const {
		const double a = l0 * l + c0 * c, b = l1 * l + c1 * c + u1 * u, e = c2 * c + u2 * u;
		l = a;
		c = b;
		u = e;
	}
};

// Galerkin operator A_l = R A_{l-1} I (upper half of the stencil), plus a
// diagonal scale proxy used to drop vertices whose diagonal cancels.  A group
// of 32 (2D: 16) lanes builds one coarse vertex: lane q < 27 (9) takes the
// q-th fine vertex of its restriction support, loads that row, folds it onto
// the 27 (9) coarse offsets axis by axis (three 3x3 products instead of up to
// 8 parents for each of 27 couplings), and the group adds the lanes' rows in
// lane order through LDS.  Bound by the loads of the fine rows (each row is
// read by the up to 8 vertices it contributes to, from L2).  A thread that
// built a whole vertex by itself ran its up to 27 x 27 x 8 terms one after
// another: 95x70x83, all levels, 4610 -> 59 us.  The weights are powers of
// two and the level-0 couplings small integers, so the double sums are exact
// on the first levels whatever their order.
template <bool IS3D, bool CODE>
__global__ void __launch_bounds__(256) k_mg_galerkin(FineOp F, LvDev c, const uint8_t* __restrict__ ctype,
                                                     float* __restrict__ Ac, float* __restrict__ proxyOut) {
	constexpr int NL = IS3D ? 27 : 9, GL = IS3D ? 32 : 16, NG = 256 / GL, S = IS3D ? 14 : 5, C = S - 1;
	__shared__ double sh[S + 1][NG][NL];
	const int g = threadIdx.x / GL, q = threadIdx.x % GL;
	const LvDev& f = F.f;
	const long long v = (long long)blockIdx.x * NG + g;
	const bool inv = v < c.n;
	const unsigned vu = inv ? (unsigned)v : 0u, row = fastdiv(vu, c.fdx), vk = fastdiv(row, c.fdy);
	const int vi = (int)(vu - row * (unsigned)c.nx), vj = (int)(row - vk * (unsigned)c.ny);
	const bool act = inv && ctype[vu] != 0;
	if (q < NL) {
		const int dx = q % 3 - 1, dy = (q / 3) % 3 - 1, dz = IS3D ? q / 9 - 1 : 0;
		const int ux = 2 * vi + dx, uy = 2 * vj + dy, uz = IS3D ? 2 * (int)vk + dz : 0;
		const bool in = act && ux >= 0 && uy >= 0 && uz >= 0 && ux < f.nx && uy < f.ny && uz < f.nz;
		const long long u = in ? ux + f.sy * uy + f.sz * uz : 0;
		const bool ua = in && fine_active(F.code, F.type, u);
		const double rw = (dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0) * (dz ? 0.5 : 1.0);
		// couplings of the fine row, 0 towards inactive or outside vertices
		double a[NL];
#pragma unroll
		for (int s = 0; s < NL; s++) a[s] = 0.0;
		if (ua) {
#pragma unroll
			for (int s = 0; s < NL; s++) {
				const int ex = s % 3 - 1, ey = (s / 3) % 3 - 1, ez = IS3D ? s / 9 - 1 : 0;
				if (CODE && (ex != 0) + (ey != 0) + (ez != 0) > 1) continue;
				const int wx = ux + ex, wy = uy + ey, wz = uz + ez;
				const bool win = wx >= 0 && wy >= 0 && wz >= 0 && wx < f.nx && wy < f.ny && wz < f.nz;
				const long long w = win ? u + ex + f.sy * ey + f.sz * ez : u;
				float val;
				bool wa;
				if (CODE) {
					const uint8_t cu = F.code[u], cw = F.code[w];
					wa = l0_active(cw);
					const int bit = ex ? 8 : (ey ? 16 : 32);
					if (s == C) val = l0_diag(cu);
					else val = (((s > C) ? cu : cw) & bit) ? -1.f : 0.f;
				} else {
					wa = F.type[w] != 0;
					val = s >= C ? F.A[(long long)(s - C) * f.n + u] : F.A[(long long)(C - s) * f.n + w];
				}
				a[s] = win && wa ? (double)val : 0.0;
			}
		}
		const double proxy = rw * fabs(a[C]) * rw;
		const AxisW wx(dx), wy(dy), wz(dz);
#pragma unroll
		for (int s = 0; s < NL; s += 3) wx.fold(a[s], a[s + 1], a[s + 2]);
#pragma unroll
		for (int s = 0; s < NL; s += 9)
#pragma unroll
			for (int e = 0; e < 3; e++) wy.fold(a[s + e], a[s + 3 + e], a[s + 6 + e]);
		if constexpr (IS3D) {
#pragma unroll
			for (int e = 0; e < 9; e++) wz.fold(a[e], a[9 + e], a[18 + e]);
		}
#pragma unroll
		for (int s = 0; s < S; s++) sh[s][g][q] = rw * a[C + s];
		sh[S][g][q] = proxy;
	}
	__syncthreads();
	for (int t = threadIdx.x; t < (S + 1) * NG; t += 256) {
		const int o = t / NG, h = t % NG;
		const long long vv = (long long)blockIdx.x * NG + h;
		if (vv >= c.n) continue;
		double sum = 0.0;
		for (int e = 0; e < NL; e++) sum += sh[o][h][e];
		bool ok = ctype[vv] != 0;
		if (o == S) {
			proxyOut[vv] = ok ? (float)sum : 0.f;
			continue;
		}
		const unsigned r2 = fastdiv((unsigned)vv, c.fdx), k2 = fastdiv(r2, c.fdy);
		const int s = C + o, nx = (int)((unsigned)vv - r2 * (unsigned)c.nx) + s % 3 - 1;
		const int ny = (int)(r2 - k2 * (unsigned)c.ny) + (s / 3) % 3 - 1, nz = (int)k2 + (IS3D ? s / 9 - 1 : 0);
		ok = ok && nx >= 0 && ny >= 0 && nz >= 0 && nx < c.nx && ny < c.ny && nz < c.nz &&
		     ctype[nx + c.sy * ny + c.sz * nz] != 0;
		Ac[(long long)o * c.n + vv] = ok ? (float)sum : 0.f;
	}
}

__global__ void k_mg_drop(LvDev c, uint8_t* __restrict__ ctype, const float* __restrict__ Ac,
                          const float* __restrict__ proxy) {
	for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < c.n;
	     v += (long long)gridDim.x * blockDim.x) {
		if (ctype[v] && !(Ac[v] > 1e-6f * proxy[v])) ctype[v] = 0;
	}
}

// Full 27-point (9-point in 2D) stencil of vertex v from the symmetric
// upper-half storage, entry C = S-1 being the diagonal.  Returns false when
// a neighbour lies outside the level or is inactive.
__device__ inline bool mg_full_stencil(const LvDev& c, int is3d, int S, const float* __restrict__ A,
                                       const uint8_t* __restrict__ type, long long v, float* out) {
	const int C = S - 1;
	const int i = (int)(v % c.nx), j = (int)((v / c.nx) % c.ny), k = (int)(v / c.sz);
	bool ok = true;
	int s = 0;
	for (int dz = is3d ? -1 : 0; dz <= (is3d ? 1 : 0); dz++)
		for (int dy = -1; dy <= 1; dy++)
			for (int dx = -1; dx <= 1; dx++, s++) {
				const int ni = i + dx, nj = j + dy, nk = k + dz;
				if (ni < 0 || nj < 0 || nk < 0 || ni >= c.nx || nj >= c.ny || nk >= c.nz) {
					ok = false;
					out[s] = 0.f;
					continue;
				}
				const long long nn = ni + c.sy * nj + c.sz * nk;
				if (!type[nn]) ok = false;
				out[s] = s >= C ? A[(long long)(s - C) * c.n + v] : A[(long long)(C - s) * c.n + nn];
			}
	return ok;
}

// Pick the most frequent full stencil among a lattice of up to 64 sample
// vertices whose neighbours are all active (the first of equally frequent
// ones).  One block per level: a thread per stencil entry of a sample loads
// it, then a thread per pair of samples compares them.
struct CanonSlot {
	Canon cn;
	int has;
};
__global__ void __launch_bounds__(1024) k_mg_pick(LvDev c, int is3d, const float* __restrict__ A,
                                                  const uint8_t* __restrict__ type, CanonSlot* __restrict__ out) {
	__shared__ unsigned st[64][27];
	__shared__ int bad[64], cnt[64];
	const int t = threadIdx.x, per = is3d ? 4 : 8, ns = is3d ? 27 : 9, C = is3d ? 13 : 4;
	if (t < 64) bad[t] = cnt[t] = 0;
	__syncthreads();
	for (int e = t; e < 64 * 27; e += 1024) {
		const int o = e / 27, s = e % 27;
		const int a = is3d ? o / (per * per) : o / per, b = is3d ? (o / per) % per : o % per, q = is3d ? o % per : 0;
		const int i = (int)((c.nx - 2) * (a + 0.5) / per) + 1, j = (int)((c.ny - 2) * (b + 0.5) / per) + 1;
		const int k = is3d ? (int)((c.nz - 2) * (q + 0.5) / per) + 1 : 0;
		unsigned val = 0;
		bool ok = i >= 1 && j >= 1 && i < c.nx - 1 && j < c.ny - 1 && (!is3d || (k >= 1 && k < c.nz - 1));
		if (ok && s < ns) {
			// (an inner vertex: every neighbour is inside)
			const long long v = i + c.sy * j + c.sz * k;
			const long long w = v + s % 3 - 1 + c.sy * ((s / 3) % 3 - 1) + (is3d ? c.sz * (s / 9 - 1) : 0);
			ok = type[w] != 0;
			val = __float_as_uint(s >= C ? A[(long long)(s - C) * c.n + v] : A[(long long)(C - s) * c.n + w]);
		}
		st[o][s] = val;
		if (!ok) bad[o] = 1;
	}
	__syncthreads();
	for (int e = t; e < 64 * 64; e += 1024) {
		const int o = e >> 6, p = e & 63;
		bool same = !bad[o] && !bad[p];
		for (int s = 0; s < ns && same; s++) same = st[o][s] == st[p][s];
		if (same) atomicAdd(&cnt[o], 1);
	}
	__syncthreads();
	if (t >= 64) return;
	// the largest count, of equal ones the lowest sample
	int key = cnt[t] * 64 + (63 - t);
	for (int o = 32; o > 0; o >>= 1) key = max(key, __shfl_xor(key, o, 64));
	const int best = 63 - (key & 63), has = key >= 64 ? 1 : 0;
	if (t == 0) out->has = has;
	if (t < 27) out->cn.a[t] = has ? __uint_as_float(st[best][t]) : 0.f;
}

// type 2 = active, all neighbours active, stencil bitwise equal to the
// picked one.  Only nonzero type values are ever written, so concurrent
// readers testing type != 0 are unaffected.
__global__ void k_mg_classify(LvDev c, int is3d, int S, const float* __restrict__ A, uint8_t* __restrict__ type,
                              const CanonSlot* __restrict__ pick) {
	if (!pick->has) return;
	const int ns = is3d ? 27 : 9;
	for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < c.n;
	     v += (long long)gridDim.x * blockDim.x) {
		if (!type[v]) continue;
		float st[27];
		if (!mg_full_stencil(c, is3d, S, A, type, v, st)) continue;
		bool same = true;
		for (int s = 0; s < ns; s++) same = same && (__float_as_uint(st[s]) == __float_as_uint(pick->cn.a[s]));
		if (same) type[v] = 2;
	}
}

// ---------------------------------------------------------------------------
// dense generalised inverse of the coarsest operator (FP64, on the device)
// ---------------------------------------------------------------------------
__global__ void k_fill_d(double* p, long long n) {
	for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
		p[i] = 0.0;
}
__global__ void k_fill_f(float* p, long long n) {
	for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
		p[i] = 0.f;
}
// M[a][b] = A(idx[a], idx[b]) (M cleared before), one thread per row and
// stencil entry; code: the level-0 operator of a single-level hierarchy
__global__ void __launch_bounds__(256) k_dense_assemble(LvDev c, int is3d, int S, int m, const int* __restrict__ idx,
                                                        const int* __restrict__ pos, const float* __restrict__ A,
                                                        const uint8_t* __restrict__ code, double* __restrict__ M,
                                                        double* __restrict__ diag) {
	const int t = blockIdx.x * 256 + threadIdx.x, a = t / 27, s = t % 27, C = S - 1;
	if (a >= m || (!is3d && s >= 9)) return;
	const int dx = s % 3 - 1, dy = (s / 3) % 3 - 1, dz = is3d ? s / 9 - 1 : 0;
	const long long v = idx[a];
	const int i = (int)(v % c.nx) + dx, j = (int)((v / c.nx) % c.ny) + dy, k = (int)(v / c.sz) + dz;
	if (i < 0 || j < 0 || k < 0 || i >= c.nx || j >= c.ny || k >= c.nz) return;
	const long long w = i + c.sy * j + c.sz * k;
	if (pos[w] < 0) return;
	float val;
	if (code) {
		const int nzc = (dx != 0) + (dy != 0) + (dz != 0);
		if (nzc > 1) return;
		const int bit = dx ? 8 : (dy ? 16 : 32);
		val = s == C ? l0_diag(code[v]) : (((s > C ? code[v] : code[w]) & bit) ? -1.f : 0.f);
	} else {
		val = s >= C ? A[(long long)(s - C) * c.n + v] : A[(long long)(C - s) * c.n + w];
	}
	M[(long long)a * m + pos[w]] = (double)val;
	if (s == C) diag[a] = (double)val;
}

// The inverse by sweeping blocks of kSweep pivots (the symmetric Gauss-Jordan
// step, Goodnight 1979, in blocks): with D the swept pivot block (-its
// inverse), P the matrix columns of the block and W = -P D,
//   M_ij -= W_i P_j^T,  M_iK = W_i,  M_Kj = W_j^T,  M_KK = D;
// after all pivots M is minus the inverse.  Pivots that are dropped (pinned,
// or not positive beyond round-off) are not swept: their rows and columns
// become 0.  Two launches per block: the panel (every workgroup sweeps the
// pivot block for itself, then forms its rows of W) and the update.
// On the host the same inverse (unblocked Cholesky) took about 3 ms at 294
// and 75 ms at 729 unknowns; here 0.2 and 0.6 ms (a panel 19 us, an update
// 6.5 us; blocks of 16 pivots: 8.4 and 4.9 us, twice as many).
constexpr int kSweep = 32, kDTile = 32;
__device__ inline double lane_d(double v, int lane) {
	const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
	const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
	const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
	return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__global__ void __launch_bounds__(256) k_sweep_panel(int m, int k0, const double* __restrict__ M,
                                                     const double* __restrict__ diag,
                                                     const int* __restrict__ pinned, double* __restrict__ D,
                                                     double* __restrict__ W, double* __restrict__ Pc) {
	__shared__ double d[kSweep][kSweep + 1];
	__shared__ double p[kDTile][kSweep + 1];
	__shared__ int drop[kSweep];
	const int t = threadIdx.x, nk = min(kSweep, m - k0), i0 = (int)blockIdx.x * kDTile;
	if (t < 64) {
		// the first wavefront sweeps the pivot block: lane r holds row r, the
		// pivot row comes by readlane (in LDS with two barriers per step a panel took
		// 24 us instead of 19)
		const int r = t & (kSweep - 1);
		double a[kSweep];
#pragma unroll
		for (int q = 0; q < kSweep; q++) a[q] = r < nk && q < nk ? M[(long long)(k0 + r) * m + k0 + q] : 0.0;
		const double og = r < nk ? diag[k0 + r] : 0.0;
		const int pn = r < nk ? pinned[k0 + r] : 1;
		unsigned dropped = 0;
#pragma unroll
		for (int k = 0; k < kSweep; k++) {
			const double piv = lane_d(a[k], k), orig = lane_d(og, k);
			if (__builtin_amdgcn_readlane(pn, k) || !(piv > 1e-10 * (orig > 0 ? orig : 1.0))) {
				dropped |= 1u << k;
				continue;
			}
			const double rp = 1.0 / piv;
			const bool own = r == k;
			const double cf = own ? -rp : a[k] * rp;
#pragma unroll
			for (int q = 0; q < kSweep; q++) {
				if (q == k) continue;
				a[q] = fma(-cf, lane_d(a[q], k), own ? 0.0 : a[q]);
			}
			a[k] = cf;
		}
		if (t < kSweep) {
			drop[t] = (dropped >> t) & 1;
#pragma unroll
			for (int q = 0; q < kSweep; q++) d[t][q] = ((dropped >> t) | (dropped >> q)) & 1 ? 0.0 : a[q];
		}
	} else {
		for (int e = t - 64; e < kDTile * kSweep; e += 192) {
			const int r = e / kSweep, q = e % kSweep;
			p[r][q] = i0 + r < m && q < nk ? M[(long long)(i0 + r) * m + k0 + q] : 0.0;
		}
	}
	__syncthreads();
	if (blockIdx.x == 0)
		for (int e = t; e < kSweep * kSweep; e += 256) D[e] = d[e / kSweep][e % kSweep];
	for (int e = t; e < kDTile * kSweep; e += 256) {
		const int r = e / kSweep, q = e % kSweep;
		if (i0 + r >= m) continue;
		double w = 0.0;
#pragma unroll
		for (int l = 0; l < kSweep; l++) w -= p[r][l] * d[l][q];
		W[(long long)(i0 + r) * kSweep + q] = w;
		Pc[(long long)(i0 + r) * kSweep + q] = drop[q] ? 0.0 : p[r][q];
	}
}
// last: the matrix is minus the result then
__global__ void __launch_bounds__(256) k_sweep_update(int m, int k0, double* __restrict__ M,
                                                      const double* __restrict__ D, const double* __restrict__ W,
                                                      const double* __restrict__ Pc, int last) {
	__shared__ double w[kDTile][kSweep + 1];
	__shared__ double p[kDTile][kSweep + 1];
	const int t = threadIdx.x, i0 = (int)blockIdx.y * kDTile, j0 = (int)blockIdx.x * kDTile;
	for (int e = t; e < kDTile * kSweep; e += 256) {
		const int r = e / kSweep, q = e % kSweep;
		w[r][q] = i0 + r < m ? W[(long long)(i0 + r) * kSweep + q] : 0.0;
		p[r][q] = j0 + r < m ? Pc[(long long)(j0 + r) * kSweep + q] : 0.0;
	}
	__syncthreads();
	// rows ty + 16 u, columns tx + 16 q of the tile
	constexpr int NU = kDTile / 16;
	const int tx = t & 15, ty = t >> 4;
	double acc[NU][NU] = {};
#pragma unroll 4
	for (int l = 0; l < kSweep; l++) {
		double a[NU], b[NU];
#pragma unroll
		for (int u = 0; u < NU; u++) {
			a[u] = w[ty + 16 * u][l];
			b[u] = p[tx + 16 * u][l];
		}
#pragma unroll
		for (int u = 0; u < NU; u++)
#pragma unroll
			for (int q = 0; q < NU; q++) acc[u][q] += a[u] * b[q];
	}
#pragma unroll
	for (int u = 0; u < NU; u++)
#pragma unroll
		for (int q = 0; q < NU; q++) {
			const int i = i0 + ty + 16 * u, j = j0 + tx + 16 * q;
			if (i >= m || j >= m) continue;
			const bool ik = i >= k0 && i < k0 + kSweep, jk = j >= k0 && j < k0 + kSweep;
			double v;
			if (ik && jk) v = D[(i - k0) * kSweep + j - k0];
			else if (jk) v = w[ty + 16 * u][j - k0];
			else if (ik) v = W[(long long)j * kSweep + i - k0];
			else v = M[(long long)i * m + j] - acc[u][q];
			M[(long long)i * m + j] = last ? -v : v;
		}
}

// ---------------------------------------------------------------------------
// V-cycle kernels
// ---------------------------------------------------------------------------
// Coarse-level pointwise kernels run on runs of 256 consecutive vertices (a
// thread per vertex; 32-bit indices: coarse levels hold fewer than 2^31
// vertices).
long long lc_tiles(const LvDev& c) { return (c.n + 255) / 256; }
struct VtxPos {
	int i, j, k, v;
	bool in;
};
__device__ inline VtxPos lc_vertex(const LvDev& c, long long blk) {
	VtxPos p;
	p.v = (int)blk * 256 + (int)threadIdx.x;
	p.in = p.v < c.n;
	const unsigned v = p.in ? (unsigned)p.v : 0u, row = fastdiv(v, c.fdx), k = fastdiv(row, c.fdy);
	p.i = (int)(v - row * (unsigned)c.nx);
	p.j = (int)(row - k * (unsigned)c.ny);
	p.k = (int)k;
	return p;
}

// Coarse-level stencil coefficients are FP32, or BF16 (upper 16 bits of the
// FP32 value, round-to-nearest-even) in the mixed-precision mode; the
// arithmetic is FP32 either way.
__device__ inline float ldA(const float* __restrict__ A, long long i) { return A[i]; }
__device__ inline float ldA(const uint16_t* __restrict__ A, long long i) {
	return __uint_as_float((unsigned)A[i] << 16);
}
__host__ __device__ inline uint16_t to_bf16(float f) {
	unsigned u;
	memcpy(&u, &f, 4);
	u += 0x7FFFu + ((u >> 16) & 1u);
	return (uint16_t)(u >> 16);
}
__host__ __device__ inline float from_bf16(uint16_t h) {
	const unsigned u = (unsigned)h << 16;
	float f;
	memcpy(&f, &u, 4);
	return f;
}
__global__ void k_to_bf16(const float* __restrict__ in, uint16_t* __restrict__ out, long long n) {
	for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
		out[i] = to_bf16(in[i]);
}

// Three consecutive floats at a 4-byte aligned address, read by one load.
struct __attribute__((packed, aligned(4))) FTriple {
	float a, b, c;
};

// b_c[V] = sum_{U in [2V-1,2V+1]} w(U) r_f[U]   (r_f is 0 on inactive vertices).
// Fixed 3x3x3 (3x3) trip counts with predicates: the loops unroll and all
// fine loads are in flight together; skipped terms are exact zeros.  The
// three fine values of a row (x = 2i-1, 2i, 2i+1) come from one 12-byte load
// at x0 = clamp(2i-1, 0, nx_f-3); only the first and last coarse vertex of a
// row have 2i-1 != x0 and pick their values at a shifted slot.  Fine levels
// narrower than 3 vertices in x take one load per value.
template <bool IS3D>
__device__ __forceinline__ float restrict_value(const LvDev& f, const float* __restrict__ rf,
                                                const uint8_t* __restrict__ ctype, int v, int i, int j, int k) {
	float sum = 0.f;
	if (f.nx >= 3) {
		constexpr int NZ = IS3D ? 3 : 1;
		const int x0 = min(max(2 * i - 1, 0), f.nx - 3);
		const int d = 2 * i - 1 - x0;  // -1 (i = 0), 0, 1 or 2 (last vertex of a row)
		long long ay[3], az[3];
		bool kx[3], ky[3], kz[3];
#pragma unroll
		for (int e = 0; e < 3; e++) {
			const int ux = 2 * i + e - 1, uy = 2 * j + e - 1, uz = 2 * k + (IS3D ? e - 1 : 0);
			kx[e] = ux >= 0 && ux < f.nx;
			ky[e] = uy >= 0 && uy < f.ny;
			kz[e] = uz >= 0 && uz < f.nz;
			ay[e] = ky[e] ? f.sy * uy : 0;
			az[e] = kz[e] ? f.sz * uz : 0;
		}
		const uint8_t ct = ctype[v];
		FTriple row[NZ * 3];
#pragma unroll
		for (int r = 0; r < NZ * 3; r++) row[r] = *reinterpret_cast<const FTriple*>(rf + x0 + ay[r % 3] + az[IS3D ? r / 3 : 1]);
#pragma unroll
		for (int e = 0; e < NZ * 9; e++) {
			const int ex = e % 3, ey = (e / 3) % 3, ez = IS3D ? e / 9 : 1;
			const FTriple& t = row[ey + 3 * (IS3D ? ez : 0)];
			// slot of x = 2i - 1 + ex in the triple: d + ex (0..2 whenever kx[ex])
			const int s = d + ex;
			const float val = s <= 0 ? t.a : (s == 1 ? t.b : t.c);
			const int ux = 2 * i + ex - 1, uy = 2 * j + ey - 1, uz = 2 * k + (IS3D ? ez - 1 : 0);
			if (kx[ex] && ky[ey] && kz[ez]) sum += wgt(ux, uy, uz) * val;
		}
		return ct ? sum : 0.f;
	}
	if (ctype[v]) {
		// branch-free: per-axis offsets of the fine coordinates 2V-1..2V+1
		// (0 where outside the level, so every address is valid), every load
		// issued before the sum; terms outside the level add exactly +0
		constexpr int NZ = IS3D ? 3 : 1;
		long long ax[3], ay[3], az[3];
		bool kx[3], ky[3], kz[3];
#pragma unroll
		for (int d = 0; d < 3; d++) {
			const int ux = 2 * i + d - 1, uy = 2 * j + d - 1, uz = 2 * k + (IS3D ? d - 1 : 0);
			kx[d] = ux >= 0 && ux < f.nx;
			ky[d] = uy >= 0 && uy < f.ny;
			kz[d] = uz >= 0 && uz < f.nz;
			ax[d] = kx[d] ? ux : 0;
			ay[d] = ky[d] ? f.sy * uy : 0;
			az[d] = kz[d] ? f.sz * uz : 0;
		}
		float rv[NZ * 9];
		bool ok[NZ * 9];
#pragma unroll
		for (int e = 0; e < NZ * 9; e++) {
			const int ex = e % 3, ey = (e / 3) % 3, ez = IS3D ? e / 9 : 1;
			ok[e] = kx[ex] && ky[ey] && kz[ez];
			rv[e] = rf[ax[ex] + ay[ey] + az[ez]];
		}
#pragma unroll
		for (int e = 0; e < NZ * 9; e++) {
			const int dx = e % 3 - 1, dy = (e / 3) % 3 - 1, dz = IS3D ? e / 9 - 1 : 0;
			const int ux = 2 * i + dx, uy = 2 * j + dy, uz = 2 * k + dz;
			if (ok[e]) sum += wgt(ux, uy, uz) * rv[e];
		}
	}
	return sum;
}
template <bool IS3D>
__device__ __forceinline__ void body_restrict(const RestrictP& P, long long blk, long long) {
	if (P.st->done) return;
	const VtxPos p = lc_vertex(P.c, blk);
	if (!p.in) return;
	P.bc[p.v] = restrict_value<IS3D>(P.f, P.rf, P.ctype, p.v, p.i, p.j, p.k);
}

// r = b - A x on a coarse level (0 on inactive vertices)
template <bool IS3D, typename AT>
__device__ __forceinline__ void body_resid(const ResidP& P, long long blk, long long) {
	const CgState* __restrict__ st = P.st;
	const LvDev& c = P.c;
	const AT* __restrict__ A = (const AT*)P.A;
	const uint8_t* __restrict__ type = P.type;
	const float* __restrict__ b = P.b;
	const float* __restrict__ x = P.x;
	float* __restrict__ r = P.r;
	const Canon& cn = P.cn;
	constexpr int C = IS3D ? 13 : 4;
	if (st->done) return;
	const VtxPos p = lc_vertex(c, blk);
	if (!p.in) return;
	const int i = p.i, j = p.j, k = p.k, v = p.v;
	const int sy = (int)c.sy, sz = (int)c.sz;
	const uint8_t tv = type[v];
	if (!tv) {
		r[v] = 0.f;
		return;
	}
	float sum = b[v];
	if (tv == 2) {
		// canonical stencil, every neighbour inside and active: one fused
		// multiply-add chain per z layer; the three x-neighbours of a row
		// (v-1, v, v+1 shifted by the row offset) come from one 12-byte load
		const float* __restrict__ xv = x + v - 1;
		FTriple xr[IS3D ? 9 : 3];
#pragma unroll
		for (int r = 0; r < (IS3D ? 9 : 3); r++)
			xr[r] = *reinterpret_cast<const FTriple*>(xv + sy * (r % 3 - 1) + sz * (IS3D ? r / 3 - 1 : 0));
		float acc[IS3D ? 3 : 1];
#pragma unroll
		for (int lz = 0; lz < (IS3D ? 3 : 1); lz++) {
			float sacc = 0.f;
#pragma unroll
			for (int dy = -1; dy <= 1; dy++) {
				const FTriple& t = xr[(dy + 1) + 3 * lz];
				sacc = fmaf(cn.a[3 * (dy + 1) + 9 * lz], t.a, sacc);
				sacc = fmaf(cn.a[1 + 3 * (dy + 1) + 9 * lz], t.b, sacc);
				sacc = fmaf(cn.a[2 + 3 * (dy + 1) + 9 * lz], t.c, sacc);
			}
			acc[lz] = sacc;
		}
		r[v] = sum - (IS3D ? (acc[0] + acc[1]) + acc[IS3D ? 2 : 0] : acc[0]);
		return;
	}
	// general stencil, branch-free: neighbours outside the level or inactive
	// contribute an exact +0 (every load is issued before the sum)
	constexpr int NS = IS3D ? 27 : 9;
	float av[NS], xv[NS];
	bool ok[NS];
#pragma unroll
	for (int s = 0; s < NS; s++) {
		const int dx = s % 3 - 1, dy = (s / 3) % 3 - 1, dz = IS3D ? s / 9 - 1 : 0;
		const int ni = i + dx, nj = j + dy, nk = k + dz;
		const bool in = ni >= 0 && nj >= 0 && nk >= 0 && ni < c.nx && nj < c.ny && nk < c.nz;
		const int nn = in ? ni + sy * nj + sz * nk : v;
		const uint8_t tn = type[nn];  // unconditional: nn is always a valid vertex
		ok[s] = in & (tn != 0);
		av[s] = s >= C ? ldA(A, (long long)(s - C) * c.n + v) : ldA(A, (long long)(C - s) * c.n + nn);
		xv[s] = x[nn];
	}
#pragma unroll
	for (int s = 0; s < NS; s++)
		if (ok[s]) sum -= av[s] * xv[s];
	r[v] = sum;
}

// ---------------------------------------------------------------------------
// LDS-brick kernels.  A workgroup owns a brick of cells/vertices and stages
// the brick plus a halo in LDS, so that a whole smoothing sweep (all
// colours) is one launch.
// ---------------------------------------------------------------------------
template <int BX, int BY, int BZ>
struct Brick {
	static constexpr int H = 2;
	static constexpr int RX = BX + 2 * H, RY = BY + 2 * H, RZ = BZ > 1 ? BZ + 2 * H : 1;
	static constexpr int RN = RX * RY * RZ;
	static constexpr int HZ = BZ > 1 ? H : 0;
};

__device__ inline void brick_origin(long long blk, int nx, int ny, int BX, int BY, int BZ, int& ox, int& oy,
                                    int& oz) {
	const unsigned nbx = (unsigned)(nx + BX - 1) / BX, nby = (unsigned)(ny + BY - 1) / BY;
	const unsigned b = (unsigned)blk, rest = b / nbx, kz = rest / nby;
	ox = (int)(b - rest * nbx) * BX;
	oy = (int)(rest - kz * nby) * BY;
	oz = (int)kz * BZ;
}

// sum of x over the fluid neighbours coupled to cell q (coefficient -1 each),
// for a cell in the LDS region with code cs and region strides 1/RX/RXY
template <bool IS3D>
__device__ inline float l0_nb_sum(const uint8_t* cs, const float* xs, int q, int RX, int RXY) {
	const uint8_t cc = cs[q];
	float sum = 0.f;
	if (cs[q - 1] & 8) sum += xs[q - 1];
	if (cc & 8) sum += xs[q + 1];
	if (cs[q - RX] & 16) sum += xs[q - RX];
	if (cc & 16) sum += xs[q + RX];
	if (IS3D) {
		if (cs[q - RXY] & 32) sum += xs[q - RXY];
		if (cc & 32) sum += xs[q + RXY];
	}
	return sum;
}

// Level-0 down leg: x = 0, red sweep, black sweep (exact red-black
// Gauss-Seidel: the black halo ring is recomputed from a 2-cell halo of red
// values), then the residual r0 = b - A x of the owned cells.
// Reads b (4 B) and the matrix code (1 B), writes x and r0: 13 B/cell.
template <int BX, int BY, int BZ, bool IS3D>
__device__ __forceinline__ void body_l0_down_brick(const L0DownP& P, long long blk, long long) {
	const Dims& d = P.d;
	const CgState* __restrict__ st = P.st;
	const uint8_t* __restrict__ code = P.code;
	const float* __restrict__ rin = P.rin;
	float* __restrict__ z = P.xout;
	float* __restrict__ r0 = P.r0;
	using B = Brick<BX, BY, BZ>;
	__shared__ float xs[B::RN];
	__shared__ float bs[B::RN];
	__shared__ uint8_t cs[B::RN];
	if (st->done) return;
	int ox, oy, oz;
	brick_origin(blk, d.nx, d.ny, BX, BY, BZ, ox, oy, oz);
	ox -= B::H;
	oy -= B::H;
	oz -= B::HZ;
	constexpr int RXY = B::RX * B::RY;
	for (int q = threadIdx.x; q < B::RN; q += blockDim.x) {
		const int gx = ox + q % B::RX, gy = oy + (q / B::RX) % B::RY, gz = oz + q / RXY;
		uint8_t cc = 0;
		float b = 0.f;
		if (gx >= 0 && gy >= 0 && gz >= 0 && gx < d.nx && gy < d.ny && gz < d.nz) {
			const long long g = d.idx(gx, gy, gz);
			cc = code[g];
			b = rin[g] * l0_scale(cc);
		}
		cs[q] = cc;
		bs[q] = b;
		xs[q] = (l0_active(cc) && ((gx + gy + gz) & 1) == 0) ? b / l0_diag(cc) : 0.f;
	}
	__syncthreads();
	// black cells of the region without its outermost ring
	constexpr int IX = B::RX - 2, IY = B::RY - 2, IZ = IS3D ? B::RZ - 2 : 1;
	for (int t = threadIdx.x; t < IX * IY * IZ; t += blockDim.x) {
		const int lx = 1 + t % IX, ly = 1 + (t / IX) % IY, lz = (IS3D ? 1 : 0) + t / (IX * IY);
		const int q = lx + B::RX * ly + RXY * lz;
		const int gx = ox + lx, gy = oy + ly, gz = oz + lz;
		const uint8_t cc = cs[q];
		if (((gx + gy + gz) & 1) == 1 && l0_active(cc))
			xs[q] = (bs[q] + l0_nb_sum<IS3D>(cs, xs, q, B::RX, RXY)) / l0_diag(cc);
	}
	__syncthreads();
	for (int t = threadIdx.x; t < BX * BY * BZ; t += blockDim.x) {
		const int lx = B::H + t % BX, ly = B::H + (t / BX) % BY, lz = B::HZ + t / (BX * BY);
		const int gx = ox + lx, gy = oy + ly, gz = oz + lz;
		if (gx >= d.nx || gy >= d.ny || gz >= d.nz) continue;
		const int q = lx + B::RX * ly + RXY * lz;
		const long long g = d.idx(gx, gy, gz);
		const uint8_t cc = cs[q];
		const float x = xs[q];
		z[g] = x;
		r0[g] = l0_active(cc) ? (bs[q] + l0_nb_sum<IS3D>(cs, xs, q, B::RX, RXY)) - l0_diag(cc) * x : 0.f;
	}
}

// Level-0 up leg: x = xpre + I x_1 (prolongation on load), black sweep, red
// sweep (reversed colour order), write z, and the partial sums of fl(z*r) for
// the CG scalar sigma = dot(z, r).  Reads xpre, b, code (9 B), writes z (4 B).
// Input and output are different arrays: the halo of one brick is owned by
// its neighbours, which write their result concurrently.
template <int BX, int BY, int BZ, bool IS3D>
__device__ __forceinline__ void body_l0_up_brick(const L0UpP& P, long long blk, long long slot) {
	const Dims& d = P.d;
	const CgState* __restrict__ st = P.st;
	const uint8_t* __restrict__ code = P.code;
	const float* __restrict__ rin = P.rin;
	const float* __restrict__ xpre = P.xpre;
	float* __restrict__ z = P.z;
	const LvDev& c1 = P.c1;
	const float* __restrict__ xc = P.xc;
	double* __restrict__ part = P.part;
	using B = Brick<BX, BY, BZ>;
	// coarse values covering the region's parents (inactive coarse vertices
	// always hold 0, so no type lookups are needed)
	constexpr int CRX = B::RX / 2 + 2, CRY = B::RY / 2 + 2, CRZ = IS3D ? B::RZ / 2 + 2 : 1;
	__shared__ float xs[B::RN];
	__shared__ float bs[B::RN];
	__shared__ uint8_t cs[B::RN];
	__shared__ float xcs[CRX * CRY * CRZ];
	__shared__ double sh[16];
	if (st->done) return;
	int ox, oy, oz;
	brick_origin(blk, d.nx, d.ny, BX, BY, BZ, ox, oy, oz);
	ox -= B::H;
	oy -= B::H;
	oz -= B::HZ;
	const int cx0 = ox >> 1, cy0 = oy >> 1, cz0 = oz >> 1;  // floor division
	for (int q = threadIdx.x; q < CRX * CRY * CRZ; q += blockDim.x) {
		const int px = cx0 + q % CRX, py = cy0 + (q / CRX) % CRY, pz = cz0 + q / (CRX * CRY);
		float v = 0.f;
		if (px >= 0 && py >= 0 && pz >= 0 && px < c1.nx && py < c1.ny && pz < c1.nz) v = xc[px + c1.sy * py + c1.sz * pz];
		xcs[q] = v;
	}
	__syncthreads();
	constexpr int RXY = B::RX * B::RY;
	for (int q = threadIdx.x; q < B::RN; q += blockDim.x) {
		const int gx = ox + q % B::RX, gy = oy + (q / B::RX) % B::RY, gz = oz + q / RXY;
		uint8_t cc = 0;
		float b = 0.f, x = 0.f;
		if (gx >= 0 && gy >= 0 && gz >= 0 && gx < d.nx && gy < d.ny && gz < d.nz) {
			const long long g = d.idx(gx, gy, gz);
			cc = code[g];
			b = rin[g] * l0_scale(cc);
			x = xpre[g];
			if (l0_active(cc)) {
				float sum = 0.f;
				for (int pz = gz >> 1; pz <= (gz + 1) >> 1; pz++)
					for (int py = gy >> 1; py <= (gy + 1) >> 1; py++)
						for (int px = gx >> 1; px <= (gx + 1) >> 1; px++)
							sum += xcs[(px - cx0) + CRX * (py - cy0) + CRX * CRY * (pz - cz0)];
				x += wgt(gx, gy, gz) * sum;
			}
		}
		cs[q] = cc;
		bs[q] = b;
		xs[q] = x;
	}
	__syncthreads();
	constexpr int IX = B::RX - 2, IY = B::RY - 2, IZ = IS3D ? B::RZ - 2 : 1;
	for (int t = threadIdx.x; t < IX * IY * IZ; t += blockDim.x) {
		const int lx = 1 + t % IX, ly = 1 + (t / IX) % IY, lz = (IS3D ? 1 : 0) + t / (IX * IY);
		const int q = lx + B::RX * ly + RXY * lz;
		const int gx = ox + lx, gy = oy + ly, gz = oz + lz;
		const uint8_t cc = cs[q];
		if (((gx + gy + gz) & 1) == 1 && l0_active(cc))
			xs[q] = (bs[q] + l0_nb_sum<IS3D>(cs, xs, q, B::RX, RXY)) / l0_diag(cc);
	}
	__syncthreads();
	double acc = 0.0;
	for (int t = threadIdx.x; t < BX * BY * BZ; t += blockDim.x) {
		const int lx = B::H + t % BX, ly = B::H + (t / BX) % BY, lz = B::HZ + t / (BX * BY);
		const int gx = ox + lx, gy = oy + ly, gz = oz + lz;
		if (gx >= d.nx || gy >= d.ny || gz >= d.nz) continue;
		const int q = lx + B::RX * ly + RXY * lz;
		const long long g = d.idx(gx, gy, gz);
		const uint8_t cc = cs[q];
		float x = xs[q];
		if (((gx + gy + gz) & 1) == 0 && l0_active(cc)) x = (bs[q] + l0_nb_sum<IS3D>(cs, xs, q, B::RX, RXY)) / l0_diag(cc);
		z[g] = x;
		acc += (double)(x * rin[g]);
	}
	const double s = block_sum(acc, sh);
	if (threadIdx.x == 0) part[3 * slot] = s;
}

// ---------------------------------------------------------------------------
// z-marching level-0 kernels (3D).  A workgroup owns a 64 x TY column tile
// and a chunk of planes [k0, k1).  It walks the planes once, staging each
// plane of the tile plus a 2-cell ring in a 6-slot LDS ring buffer, and runs
// the three dependent stages of red-black Gauss-Seidel as a pipeline whose
// stages are two planes apart:
//   A(p)   load plane p (code, rhs, x), first colour pointwise
//   B(p-2) second colour on plane p-2 (tile + 1-cell ring): needs the first
//          colour of planes p-3 .. p-1
//   C(p-4) final output on the tile's cells of plane p-4: needs both colours
//          of planes p-5 .. p-3
// Each stage reads only what the previous iterations finished, and the three
// touch different ring slots, so one barrier per plane suffices.  Every input
// element is read from HBM once plus 4 halo planes per chunk.  Arithmetic
// and operation order equal the brick kernels above.
// ---------------------------------------------------------------------------
constexpr int ZRING = 6;  // LDS ring slots: planes p-5 .. p
template <int TY>
struct ZTile {
	static constexpr int TX = 64, H = 2, RX = TX + 2 * H, RY = TY + 2 * H, RP = RX * RY, NS = ZRING, NT = TX * TY;
};

__device__ inline void zm_origin(long long blk, const Dims& d, int TY, int kchunk, int& ox, int& oy, int& k0,
                                 int& k1) {
	const unsigned ntx = (unsigned)(d.nx + 63) / 64, nty = (unsigned)(d.ny + TY - 1) / TY;
	const unsigned b = (unsigned)blk, rest = b / ntx, kz = rest / nty;
	ox = (int)(b - rest * ntx) * 64;
	oy = (int)(rest - kz * nty) * TY;
	k0 = (int)kz * kchunk;
	k1 = min(d.nz, k0 + kchunk);
}

// x if bit B of c is set, else +0.0: the bit pattern AND the bit's sign
// extension (v_bfe_i32 + v_and_b32 instead of a compare and a select; the
// extract is written as an instruction because the compiler turns a
// sign-extended bit of a byte back into a compare and a select)
template <int B>
__device__ inline float zm_keep(uint8_t c, float x) {
	int m;
	asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"((int)c), "i"(B));
	return __int_as_float(__float_as_int(x) & m);
}
// l0_nb_sum with the plane below (cM, xM) and above (xU) in separate slots;
// cc = cP[q].  Every neighbour is read and added, masked to +0.0 where its
// coupling flag is clear.  The running sum starts at +0.0 and a round-to-
// nearest sum is -0.0 only when both addends are, so it never is; adding
// +0.0 to it is therefore exact and this equals the conditional adds of
// l0_nb_sum, in the same order, without a branch per neighbour.
__device__ inline float zm_nb_sum(uint8_t cc, const uint8_t* cP, const float* xP, const uint8_t* cM, const float* xM,
                                  const float* xU, int q, int RX) {
	const uint8_t cw = cP[q - 1], cs = cP[q - RX], cm = cM[q];
	const float w = xP[q - 1], e = xP[q + 1], so = xP[q - RX], no = xP[q + RX], dn = xM[q], up = xU[q];
	float sum = 0.f;
	sum += zm_keep<3>(cw, w);
	sum += zm_keep<3>(cc, e);
	sum += zm_keep<4>(cs, so);
	sum += zm_keep<4>(cc, no);
	sum += zm_keep<5>(cm, dn);
	sum += zm_keep<5>(cc, up);
	return sum;
}

// (diag, 1/diag, scale) of the level-0 row codes in LDS, index (c & 7) + 8
// for the 1e-6-scaled trivial rows (bit 7); filled by threads 0..15 before
// the kernel's first barrier (scale = l0_scale, diag = l0_diag)
__device__ inline int l0_tab_index(uint8_t c) { return (c & 7) | ((c >> 4) & 8); }
__device__ inline void l0_tab_fill(float4* t) {
	if (threadIdx.x < 16) {
		const int a = threadIdx.x & 7;
		const bool tr = (threadIdx.x & 8) != 0;
		const float dg = tr ? (float)a * 1e-6f : (float)a;
		t[threadIdx.x] = make_float4(dg, a ? 1.0f / dg : 0.f, tr ? 1e-6f : 1.0f, 0.f);
	}
}
__device__ inline float4 l0_row(uint8_t c, const float4* t) { return t[l0_tab_index(c)]; }
// v / diag as q0 = v (1/d) plus one residual correction (Markstein):
// checked exhaustively over all binary32 v, it equals the IEEE quotient for
// every finite v when d = 1..5 and for every normal quotient when d = 6; on
// the 1e-6-scaled trivial rows it can differ from it in the last bit
__device__ inline float l0_div_r(float v, const float4& e) {
	const float q0 = v * e.y;
	return fmaf(fmaf(-q0, e.x, v), e.y, q0);
}


// The (at most two) region cells of one thread: q = tid and tid + NT.
template <typename T>
struct ZmCells {
	static_assert(T::RP <= 2 * T::NT, "two region cells per thread");
	unsigned g[2];   // in-plane offset i + nx*j (nx*ny < 2^31 is checked on the host)
	bool ok[2];      // inside the region and the grid
	bool par[2];     // (i + j) & 1
	__device__ ZmCells(const Dims& d, int rx0, int ry0) {
#pragma unroll
		for (int u = 0; u < 2; u++) {
			const int q = threadIdx.x + u * T::NT;
			const int gx = rx0 + q % T::RX, gy = ry0 + q / T::RX;
			ok[u] = q < T::RP && gx >= 0 && gy >= 0 && gx < d.nx && gy < d.ny;
			g[u] = ok[u] ? (unsigned)gx + (unsigned)d.nx * (unsigned)gy : 0u;
			par[u] = ((gx + gy) & 1) != 0;
		}
	}
};

// x / diag of a level-0 row (A0 = 1..6, or A0 * 1e-6 on trivial rows)
__device__ inline float l0_div(float v, uint8_t c) { return v / l0_diag(c); }

// Per-thread positions of the z-marching kernels that do not change from
// plane to plane (the plane loop only rotates ring slots).
template <typename T>
struct ZmPos {
	// load stage: at most two region cells per thread (q = tid, tid + NT)
	int qa[2];
	// second-colour stage: region without its outer ring (at most two cells)
	int qb[2];
	bool parb[2];
	bool inb[2];
	// output stage: the thread's tile cell
	int qc;
	unsigned gc;
	bool parc;
	bool inc;
	__device__ ZmPos(const Dims& d, int ox, int oy) {
		const int rx0 = ox - T::H, ry0 = oy - T::H;
		constexpr int IX = T::RX - 2, IN = IX * (T::RY - 2);
		static_assert(IN <= 2 * T::NT, "two second-colour cells per thread");
#pragma unroll
		for (int u = 0; u < 2; u++) {
			qa[u] = threadIdx.x + u * T::NT;
			const int t = threadIdx.x + u * T::NT;
			const int lx = 1 + t % IX, ly = 1 + t / IX;
			inb[u] = t < IN;
			qb[u] = lx + T::RX * ly;
			parb[u] = ((rx0 + lx + ry0 + ly) & 1) != 0;
		}
		const int lx = T::H + (threadIdx.x & 63), ly = T::H + (threadIdx.x >> 6);
		const int gx = rx0 + lx, gy = ry0 + ly;
		qc = lx + T::RX * ly;
		inc = gx < d.nx && gy < d.ny;
		gc = inc ? (unsigned)gx + (unsigned)d.nx * (unsigned)gy : 0u;
		parc = ((gx + gy) & 1) != 0;
	}
};

// Colour-packed positions of the z-marching stages.  Tile origins are even,
// so the colour of a cell is the parity of its tile-local x + y plus the
// plane.  Stage B updates the black cells of the region without its outer
// ring: IX/2 per row, one per thread for threads < BN (the other wavefronts
// skip the stage).
template <typename T>
struct ZmPack {
	static constexpr int IX = T::RX - 2, IY = T::RY - 2, BN = (IX / 2) * IY;
	static_assert(IX % 2 == 0 && BN <= T::NT, "colour packing");
	int bly, bm;  // stage B: region row (1-based) and index within the row
	__device__ ZmPack() {
		const int t = threadIdx.x;
		bly = 1 + t / (IX / 2);
		bm = t % (IX / 2);
	}
	// LDS index of the thread's stage-B black cell at plane parity par:
	// black means region-local x + y + plane odd
	__device__ int qb(int par) const { return 2 * bm + 1 + ((bly + par) & 1) + T::RX * bly; }
};

__device__ inline int ring_next(int s) { return s == ZRING - 1 ? 0 : s + 1; }
__device__ inline int ring_back(int s, int k) { return (s + ZRING - k) % ZRING; }

// Down leg (same sweeps as body_l0_down_brick): red from x = 0, black, residual.
// The stages are branch-free where lanes would diverge: plane loads read a
// clamped plane and are zeroed where used, colour and activity select
// between the new and the old value, and the division goes through the
// (diag, 1/diag) table.
template <int TY>
__device__ __forceinline__ void body_l0_down_zm(const L0DownP& P, long long blk, long long) {
	const Dims& d = P.d;
	const int kchunk = P.kchunk;
	const CgState* __restrict__ st = P.st;
	const uint8_t* __restrict__ code = P.code;
	const float* __restrict__ rin = P.rin;
	float* __restrict__ xout = P.xout;
	float* __restrict__ r0 = P.r0;
	using T = ZTile<TY>;
	// one LDS block in a fixed order: codes first (byte offsets from the
	// cell index), then the float rings contiguous, so every ring access is
	// an immediate offset (< 64 KiB) from one of two per-cell bases
	struct Lds {
		uint8_t cs[T::NS][T::RP];
		float xs[T::NS][T::RP];
		float bs[T::NS][T::RP];
		float4 dt[16];
	};
	static_assert((T::NS * T::RP) % 16 == 0 && 2 * sizeof(float) * T::NS * T::RP < 65536, "ring layout");
	__shared__ Lds lds;
	auto& cs = lds.cs;
	auto& xs = lds.xs;
	auto& bs = lds.bs;
	float4* dt = lds.dt;
	if (st->done) return;
	l0_tab_fill(dt);
	int ox, oy, k0, k1;
	zm_origin(blk, d, TY, kchunk, ox, oy, k0, k1);
	const int rx0 = ox - T::H, ry0 = oy - T::H;
	ZmCells<T> cells(d, rx0, ry0);
	const ZmPos<T> pos(d, ox, oy);
	const ZmPack<T> pk;
	// plane p's inputs are fetched into registers one plane ahead, so the
	// loads are in flight during the barriers and the sweeps of plane p-1;
	// a plane outside k0-2..k1+1 or the grid reads a clamped plane and pv
	// marks whether the values count
	const int pLo = max(k0 - 2, 0), pHi = min(k1 + 1, d.nz - 1);
	uint8_t pc[2];
	float pr[2];
	bool pv = false;
	auto fetch = [&](int p) {
		const long long pl = d.sz * min(max(p, pLo), pHi);
#pragma unroll
		for (int u = 0; u < 2; u++) {
			pc[u] = code[cells.g[u] + pl];
			pr[u] = rin[cells.g[u] + pl];
		}
		pv = p >= 0 && p < d.nz;
	};
	fetch(k0 - 2);
	__syncthreads();
	// One plane step; J = ring slot of plane p = (p - k0 + 2) mod ZRING, a
	// compile-time constant (the loop is unrolled by ZRING), so every slot
	// offset is an immediate of the LDS instructions.  k0 is even, so the
	// parity of p is that of J.
	auto step = [&](auto jc, int p) {
		constexpr int J = decltype(jc)::value;
		constexpr int sA = J, sB0 = (J + 4) % ZRING, sBm = (J + 3) % ZRING, sBu = (J + 5) % ZRING;
		constexpr int sC0 = (J + 2) % ZRING, sCm = (J + 1) % ZRING, sCu = (J + 3) % ZRING;
		constexpr int par = J & 1;
		// plane p into slot sA; the last two steps only finish earlier planes
		// (8 planes at 128^3: 16.7 us with the stage run in them, 16.4 without)
		if (p <= k1 + 1) {
			const bool pvp = pv;
#pragma unroll
			for (int u = 0; u < 2; u++) {
				const int q = pos.qa[u];
				if (q >= T::RP) continue;
				const bool ok = cells.ok[u] && pvp;
				const uint8_t cc = ok ? pc[u] : (uint8_t)0;
				const float4 e = l0_row(cc, dt);
				const float b = ok ? pr[u] * e.z : 0.f;
				cs[sA][q] = cc;
				bs[sA][q] = b;
				const float x = l0_div_r(b, e);
				xs[sA][q] = (l0_active(cc) && cells.par[u] == (par != 0)) ? x : 0.f;
			}
		}
		fetch(p + 1);
		const int pb = p - 2;
		if (pb >= k0 - 1 && pb <= k1 && pb >= 0 && pb < d.nz && threadIdx.x < ZmPack<T>::BN) {
			const int q = pk.qb(par);
			const uint8_t cc = cs[sB0][q];
			const float xo = xs[sB0][q];
			const float v =
			    l0_div_r(bs[sB0][q] + zm_nb_sum(cc, cs[sB0], xs[sB0], cs[sBm], xs[sBm], xs[sBu], q, T::RX), l0_row(cc, dt));
			xs[sB0][q] = l0_active(cc) ? v : xo;
		}
		const int pz = p - 4;
		if (pz >= k0 && pz < k1) {
			const int q = pos.qc;
			const uint8_t cc = cs[sC0][q];
			const float x = xs[sC0][q];
			const float rr = (bs[sC0][q] + zm_nb_sum(cc, cs[sC0], xs[sC0], cs[sCm], xs[sCm], xs[sCu], q, T::RX)) -
			                 l0_row(cc, dt).x * x;
			if (pos.inc) {
				const long long g = pos.gc + d.sz * pz;
				xout[g] = x;
				r0[g] = l0_active(cc) ? rr : 0.f;
			}
		}
		__syncthreads();
	};
	static_assert(ZRING == 6, "the plane loop is unrolled by the ring size");
	for (int p = k0 - 2; p <= k1 + 3; p += ZRING) {
		step(std::integral_constant<int, 0>{}, p);
		if (p + 1 <= k1 + 3) step(std::integral_constant<int, 1>{}, p + 1);
		if (p + 2 <= k1 + 3) step(std::integral_constant<int, 2>{}, p + 2);
		if (p + 3 <= k1 + 3) step(std::integral_constant<int, 3>{}, p + 3);
		if (p + 4 <= k1 + 3) step(std::integral_constant<int, 4>{}, p + 4);
		if (p + 5 <= k1 + 3) step(std::integral_constant<int, 5>{}, p + 5);
	}
}

// Up leg (same sweeps as body_l0_up_brick): x = xpre + I x_1, black, red,
// write z and the partial sums of fl(z*r).  Coarse planes are staged in a
// 2-slot ring: fine plane p needs coarse planes p>>1 and (p+1)>>1.  The x/y
// parents of the thread's region cells are fixed for the whole column, only
// the z parents change with the plane.  Branch-free in
// the same way as the down leg; the prolongation reads all four x/y parents
// of a coarse plane and adds each with a select.
template <int TY>
__device__ __forceinline__ void body_l0_up_zm(const L0UpP& P, long long blk, long long slot) {
	const Dims& d = P.d;
	const int kchunk = P.kchunk;
	const CgState* __restrict__ st = P.st;
	const uint8_t* __restrict__ code = P.code;
	const float* __restrict__ rin = P.rin;
	const float* __restrict__ xpre = P.xpre;
	float* __restrict__ z = P.z;
	const LvDev& c1 = P.c1;
	const float* __restrict__ xc = P.xc;
	double* __restrict__ part = P.part;
	using T = ZTile<TY>;
	constexpr int CRX = T::RX / 2 + 2, CRY = T::RY / 2 + 2, CRP = CRX * CRY;
	// LDS in a fixed order as in the down leg
	struct Lds {
		uint8_t cs[T::NS][T::RP];
		float xs[T::NS][T::RP];
		float rs[T::NS][T::RP];
		float xcs[2][CRP];
		double tab[kZmMaxGroups][TY];
		float4 dt[16];
	};
	static_assert((T::NS * T::RP) % 16 == 0 && 2 * sizeof(float) * T::NS * T::RP < 65536, "ring layout");
	__shared__ Lds lds;
	auto& cs = lds.cs;
	auto& xs = lds.xs;
	auto& rs = lds.rs;
	auto& xcs = lds.xcs;
	auto& tab = lds.tab;
	float4* dt = lds.dt;
	if (st->done) return;
	l0_tab_fill(dt);
	int ox, oy, k0, k1;
	zm_origin(blk, d, TY, kchunk, ox, oy, k0, k1);
	const int rx0 = ox - T::H, ry0 = oy - T::H;
	const int cx0 = rx0 >> 1, cy0 = ry0 >> 1;  // floor division
	static_assert(CRP <= T::NT, "one coarse value per thread");
	// this thread's vertex of the coarse-plane region; coarse planes outside
	// the level read a clamped plane and are zeroed where stored
	const int cq = threadIdx.x;
	const int cpx = cx0 + cq % CRX, cpy = cy0 + cq / CRX;
	const bool cok = cq < CRP && cpx >= 0 && cpy >= 0 && cpx < c1.nx && cpy < c1.ny;
	const unsigned cg = cok ? (unsigned)cpx + (unsigned)c1.sy * (unsigned)cpy : 0u;  // coarse n < 2^31
	auto cfetch = [&](int Pz) -> float { return xc[cg + (unsigned)c1.sz * (unsigned)min(max(Pz, 0), c1.nz - 1)]; };
	auto cvalid = [&](int Pz) -> bool { return cok && Pz >= 0 && Pz < c1.nz; };
	ZmCells<T> cells(d, rx0, ry0);
	const ZmPos<T> pos(d, ox, oy);
	const ZmPack<T> pk;
	// prolongation offsets (coarse-plane region) and x/y parities per region cell
	int po[2];
	bool pxo[2], pyo[2];
#pragma unroll
	for (int u = 0; u < 2; u++) {
		const int q = pos.qa[u];
		const int gx = rx0 + q % T::RX, gy = ry0 + q / T::RX;
		pxo[u] = gx & 1;
		pyo[u] = gy & 1;
		po[u] = ((gx >> 1) - cx0) + CRX * ((gy >> 1) - cy0);
	}
	const int pLo = max(k0 - 2, 0), pHi = min(k1 + 1, d.nz - 1);
	uint8_t pc[2];
	float pr[2], px[2];
	bool pv = false;
	auto fetch = [&](int p) {
		const long long pl = d.sz * min(max(p, pLo), pHi);
#pragma unroll
		for (int u = 0; u < 2; u++) {
			pc[u] = code[cells.g[u] + pl];
			pr[u] = rin[cells.g[u] + pl];
			px[u] = xpre[cells.g[u] + pl];
		}
		pv = p >= 0 && p < d.nz;
	};
	// coarse plane (k0-2)/2 goes to LDS now; later planes are fetched into a
	// register two fine planes before they are needed (k0 is even)
	if (cq < CRP) xcs[((k0 - 2) >> 1) & 1][cq] = cvalid((k0 - 2) >> 1) ? cfetch((k0 - 2) >> 1) : 0.f;
	float creg = cfetch(k0 >> 1);
	bool cregv = cvalid(k0 >> 1);
	fetch(k0 - 2);
	__syncthreads();
	double acc = 0.0;
	// One plane step, J = ring slot of plane p (compile-time, as in the down
	// leg; the parity of p is that of J)
	auto step = [&](auto jc, int p) {
		constexpr int J = decltype(jc)::value;
		constexpr int sA = J, sB0 = (J + 4) % ZRING, sBm = (J + 3) % ZRING, sBu = (J + 5) % ZRING;
		constexpr int sC0 = (J + 2) % ZRING, sCm = (J + 1) % ZRING, sCu = (J + 3) % ZRING;
		constexpr int par = J & 1;
		constexpr bool zo = (J & 1) != 0;
		// plane p into slot sA; the last two steps only finish earlier planes
		// (128^3: 18.7 us with the stage run in them, 17.4 without; 192x160x129
		// 28.2 / 26.0, 256^3 79.6 / 76.0)
		if (p <= k1 + 1) {
			const float* c0 = xcs[(p >> 1) & 1];
			const float* c1p = xcs[((p >> 1) + 1) & 1];
			const bool pvp = pv;
#pragma unroll
			for (int u = 0; u < 2; u++) {
				const int q = pos.qa[u];
				if (q >= T::RP) continue;
				const bool ok = cells.ok[u] && pvp;
				const uint8_t cc = ok ? pc[u] : (uint8_t)0;
				const float rr = ok ? pr[u] : 0.f;
				float x = ok ? px[u] : 0.f;
				// parents in the reference's loop order: z, then y, then x
				const int o = po[u];
				const bool bx = pxo[u], by = pyo[u], bxy = pxo[u] && pyo[u];
				float sum = c0[o];
				const float a01 = c0[o + 1], a10 = c0[o + CRX], a11 = c0[o + CRX + 1];
				sum = bx ? sum + a01 : sum;
				sum = by ? sum + a10 : sum;
				sum = bxy ? sum + a11 : sum;
				if (zo) {
					const float b00 = c1p[o], b01 = c1p[o + 1], b10 = c1p[o + CRX], b11 = c1p[o + CRX + 1];
					sum += b00;
					sum = bx ? sum + b01 : sum;
					sum = by ? sum + b10 : sum;
					sum = bxy ? sum + b11 : sum;
				}
				// x/y weight 1/2 per odd coordinate (exact powers of two)
				const float pw = (bx ? 0.5f : 1.0f) * (by ? 0.5f : 1.0f);
				const float xn = x + (zo ? 0.5f * pw : pw) * sum;
				x = l0_active(cc) ? xn : x;
				cs[sA][q] = cc;
				rs[sA][q] = rr;
				xs[sA][q] = x;
			}
			if (!zo) {
				// coarse plane p/2+1 is first needed by plane p+1
				if (cq < CRP) xcs[((p >> 1) + 1) & 1][cq] = cregv ? creg : 0.f;
				creg = cfetch((p >> 1) + 2);
				cregv = cvalid((p >> 1) + 2);
			}
			fetch(p + 1);
		}
		const int pb = p - 2;
		// packed positions from the plane's run-time parity (equal to par;
		// recomputed per plane instead of holding both parities' positions
		// in registers across the loop)
		const int rpar = p & 1;
		if (pb >= k0 - 1 && pb <= k1 && pb >= 0 && pb < d.nz && threadIdx.x < ZmPack<T>::BN) {
			const int q = pk.qb(rpar);
			const uint8_t cc = cs[sB0][q];
			const float xo = xs[sB0][q];
			const float4 e = l0_row(cc, dt);
			const float v =
			    l0_div_r(rs[sB0][q] * e.z + zm_nb_sum(cc, cs[sB0], xs[sB0], cs[sBm], xs[sBm], xs[sBu], q, T::RX), e);
			xs[sB0][q] = l0_active(cc) ? v : xo;
		}
		const int pz = p - 4;
		if (pz >= k0 && pz < k1) {
			const int q = pos.qc;
			const uint8_t cc = cs[sC0][q];
			const float xo = xs[sC0][q];
			const float rq = rs[sC0][q];
			const float4 e = l0_row(cc, dt);
			const float v =
			    l0_div_r(rq * e.z + zm_nb_sum(cc, cs[sC0], xs[sC0], cs[sCm], xs[sCm], xs[sCu], q, T::RX), e);
			const float x = (pos.parc == (par != 0) && l0_active(cc)) ? v : xo;
			if (pos.inc) z[pos.gc + d.sz * pz] = x;
			const double prod = (double)(x * rq);
			acc = pos.inc ? acc + prod : acc;
			if ((pz + 1) % kDotGroup == 0 || pz + 1 == k1) zm_dot_flush<TY>(acc, tab, pz, k0);
		}
		__syncthreads();
	};
	for (int p = k0 - 2; p <= k1 + 3; p += ZRING) {
		step(std::integral_constant<int, 0>{}, p);
		if (p + 1 <= k1 + 3) step(std::integral_constant<int, 1>{}, p + 1);
		if (p + 2 <= k1 + 3) step(std::integral_constant<int, 2>{}, p + 2);
		if (p + 3 <= k1 + 3) step(std::integral_constant<int, 3>{}, p + 3);
		if (p + 4 <= k1 + 3) step(std::integral_constant<int, 4>{}, p + 4);
		if (p + 5 <= k1 + 3) step(std::integral_constant<int, 5>{}, p + 5);
	}
	(void)slot;
	zm_dot_store<TY>(tab, d, zm_column(blk, d, TY), k0, k1, part);
}

// coarse-level brick: 32x4x4 vertices in 3D, 64x8 in 2D, 512 threads (rows
// of 32/64 vertices keep the region loads in whole cache lines)
constexpr int kLcBX3 = 32, kLcBY3 = 4, kLcBZ3 = 4, kLcBX2 = 64, kLcBY2 = 8;
constexpr int kSmoothNT = 512;

// Coarse-level block Gauss-Seidel: one sweep over all 8 (4 in 2D) colours of
// the 27-point (9-point) Galerkin stencil inside an LDS brick; halo values
// are the pre-sweep ones (block-hybrid smoother).  Two modes (POST):
//   pre-smoothing:  x starts at 0, forward colour order;
//   post-smoothing: x = xin + I x_{l+1} (prolongation from the next coarser
//                   level on load; inactive coarse vertices hold 0 there, so
//                   no coarse type lookups are needed), reversed colour order,
// which keeps the V-cycle symmetric.  The result goes to xout, never to xin:
// neighbouring bricks read xin as their halo.
// Threads are assigned by colour: the 64 vertices of colour c are the lanes
// of wavefront c (in 2D, 128 vertices on wavefronts 2c and 2c+1), so each
// phase runs whole wavefronts.  Every thread loads its vertex's stencil once,
// before the sweep (canonical vertices take the uniform stencil), and the
// coarse parents of the brick are staged in LDS.  The stencil sum runs as
// three fused multiply-add chains, one per z layer.  Vertex indices are
// 32-bit (coarse levels hold fewer than 2^31 vertices).
template <bool IS3D, typename AT, bool POST, bool RESTRICT>
__device__ __forceinline__ void smooth_tile(const SmoothP& P, const RestrictP* R, long long blk) {
	const CgState* __restrict__ st = P.st;
	const LvDev& c = P.c;
	const AT* __restrict__ A = (const AT*)P.A;
	const uint8_t* __restrict__ type = P.type;
	const float* __restrict__ b = P.b;
	const float* __restrict__ xin = P.xin;
	float* __restrict__ xout = P.xout;
	const LvDev& cp = P.cp;
	const float* __restrict__ xcp = P.xcp;
	const Canon& cn = P.cn;
	constexpr int BX = IS3D ? kLcBX3 : kLcBX2, BY = IS3D ? kLcBY3 : kLcBY2, BZ = IS3D ? kLcBZ3 : 1;
	constexpr int RX = BX + 2, RY = BY + 2, RZ = IS3D ? BZ + 2 : 1, RN = RX * RY * RZ, RXY = RX * RY;
	constexpr int C = IS3D ? 13 : 4, NCOL = IS3D ? 8 : 4, NS = IS3D ? 27 : 9;
	// one colour's sub-lattice of the brick and the wavefronts that hold it
	constexpr int HX = BX / 2, HY = BY / 2, NWPC = kSmoothNT / 64 / NCOL;
	static_assert(BX * BY * BZ == kSmoothNT && HX * HY * (IS3D ? BZ / 2 : 1) == 64 * NWPC, "brick/thread mismatch");
	// coarse parents of the region: coarse coordinates o/2 - 1 .. (o + B)/2
	constexpr int CRX = BX / 2 + 2, CRY = BY / 2 + 2, CRZ = IS3D ? BZ / 2 + 2 : 1, CRXY = CRX * CRY;
	constexpr int CRN = CRXY * CRZ;
	__shared__ float xs[RN];
	__shared__ float xc[POST ? CRN : 1];
	if (st->done) return;
	int ox, oy, oz;
	brick_origin(blk, c.nx, c.ny, BX, BY, BZ, ox, oy, oz);
	const int t = threadIdx.x;
	const int hz = IS3D ? 1 : 0;
	const int sy = (int)c.sy, sz = (int)c.sz;
	// this thread's vertex
	const int col = (t >> 6) / NWPC, sidx = ((t >> 6) % NWPC) * 64 + (t & 63);
	const int tx = 2 * (sidx % HX) + (col & 1), ty = 2 * ((sidx / HX) % HY) + ((col >> 1) & 1);
	const int tz = IS3D ? 2 * (sidx / (HX * HY)) + (col >> 2) : 0;
	const int gx = ox + tx, gy = oy + ty, gz = oz + tz;
	const bool valid = gx < c.nx && gy < c.ny && gz < c.nz;
	const int v = valid ? gx + sy * gy + sz * gz : 0;
	const uint8_t tl = type[v];
	// RESTRICT: the right-hand side is restricted here instead of by a launch
	// of its own, and stored for the residual and the way up
	float bv;
	if (RESTRICT) {
		bv = restrict_value<IS3D>(R->f, R->rf, type, v, valid ? gx : 0, valid ? gy : 0, valid ? gz : 0);
		if (valid) R->bc[v] = bv;
	} else bv = b[v];
	// post-smoothing: the region's old iterate and types, asked for before
	// anything waits
	constexpr int NIT = (RN + kSmoothNT - 1) / kSmoothNT;
	float xr[NIT];
	uint8_t tr[NIT];
	if (POST) {
#pragma unroll
		for (int it = 0; it < NIT; it++) {
			const int q = t + kSmoothNT * it;
			const int hx = ox - 1 + q % RX, hy = oy - 1 + (q / RX) % RY, hzz = oz - hz + q / RXY;
			const bool inb = q < RN && hx >= 0 && hy >= 0 && hzz >= 0 && hx < c.nx && hy < c.ny && hzz < c.nz;
			const int g = inb ? hx + sy * hy + sz * hzz : 0;
			xr[it] = xin[g];
			tr[it] = type[g];
		}
	}
	const uint8_t tv = valid ? tl : (uint8_t)0;
	float a[NS];
	float diag = 1.f;
	if (tv == 2) {
		diag = cn.a[C];
#pragma unroll
		for (int s = 0; s < NS; s++) a[s] = s == C ? 0.f : cn.a[s];
	} else if (tv) {
		// all coefficients in flight at once: the upper ones are the vertex's
		// own (0 towards neighbours outside the level), a lower one is its
		// neighbour's; outside the level any valid address is read and 0 taken.
		// With a branch and a wait per coefficient a small level's sweep was
		// bound by them (17^3: 7.2 us before smoothing, 7.7 after; now 6.0 and
		// 6.4; 65^3 after smoothing 13.6 -> 11.3, 129^3 41 -> 38.5).  What is
		// left of a small level's 6 us: 1.8 in the colour phases, 1 in the
		// loads' latency, 3 in the launch itself.
		const bool in[3][3] = {{gx > 0, true, gx < c.nx - 1}, {gy > 0, true, gy < c.ny - 1}, {gz > 0, true, gz < c.nz - 1}};
#pragma unroll
		for (int s = 0; s < NS; s++) {
			const int dx = s % 3 - 1, dy = (s / 3) % 3 - 1, dz = IS3D ? s / 9 - 1 : 0;
			const bool ok = s >= C || (in[0][dx + 1] && in[1][dy + 1] && (!IS3D || in[2][dz + 1]));
			const int nn = s >= C || !ok ? v : v + dx + sy * dy + sz * dz;
			a[s] = ldA(A + (long long)(s >= C ? s - C : C - s) * c.n, nn);
		}
#pragma unroll
		for (int s = 0; s < C; s++) {
			const int dx = s % 3 - 1, dy = (s / 3) % 3 - 1, dz = IS3D ? s / 9 - 1 : 0;
			if (!(in[0][dx + 1] && in[1][dy + 1] && (!IS3D || in[2][dz + 1]))) a[s] = 0.f;
		}
		diag = a[C];
	}
	if (POST) {
		const int psy = (int)cp.sy, psz = (int)cp.sz;
		const int cox = (ox >> 1) - 1, coy = (oy >> 1) - 1, coz = IS3D ? (oz >> 1) - 1 : 0;
		for (int q = t; q < CRN; q += kSmoothNT) {
			const int cx = q % CRX, cy = (q / CRX) % CRY, cz = q / CRXY;
			const int px = min(max(cox + cx, 0), cp.nx - 1), py = min(max(coy + cy, 0), cp.ny - 1);
			const int pz = IS3D ? min(max(coz + cz, 0), cp.nz - 1) : 0;
			xc[q] = xcp[px + psy * py + psz * pz];
		}
		__syncthreads();
	}
#pragma unroll
	for (int it = 0; it < NIT; it++) {
		const int q = t + kSmoothNT * it;
		if (q >= RN) break;
		const int rx = q % RX, ry = (q / RX) % RY, rz = q / RXY;
		const int hx = ox - 1 + rx, hy = oy - 1 + ry, hzz = oz - hz + rz;
		const bool inb = hx >= 0 && hy >= 0 && hzz >= 0 && hx < c.nx && hy < c.ny && hzz < c.nz;
		float x = 0.f;
		if (POST) {
			x = xr[it];
			const uint8_t tp = tr[it];
			// parents [s/2, (s+1)/2] per axis; with o even, s = o - 1 + r has
			// parity (r + 1) & 1 and its first parent in LDS slot (r + 1) >> 1
			const int odx = (rx + 1) & 1, ody = (ry + 1) & 1, odz = IS3D ? (rz + 1) & 1 : 0;
			const int base = ((rx + 1) >> 1) + CRX * ((ry + 1) >> 1) + (IS3D ? CRXY * ((rz + 1) >> 1) : 0);
			const int ex = odx, ey = CRX * ody, ez = CRXY * odz;
			float pv[IS3D ? 8 : 4];
			pv[0] = xc[base];
			pv[1] = xc[base + ex];
			pv[2] = xc[base + ey];
			pv[3] = xc[base + ex + ey];
			if constexpr (IS3D) {
				pv[4] = xc[base + ez];
				pv[5] = xc[base + ex + ez];
				pv[6] = xc[base + ey + ez];
				pv[7] = xc[base + ex + ey + ez];
			}
			float sum = 0.f;
#pragma unroll
			for (int e = 0; e < (IS3D ? 8 : 4); e++) {
				const bool use = ((e & 1) == 0 || odx) && (((e >> 1) & 1) == 0 || ody) && ((e >> 2) == 0 || odz);
				if (use) sum += pv[e];
			}
			if (tp) x += wgt(hx, hy, hzz) * sum;
			if (!inb) x = 0.f;
		}
		xs[q] = x;
	}
	__syncthreads();
	const int me = (tx + 1) + RX * (ty + 1) + RXY * (tz + hz);
	for (int ph = 0; ph < NCOL; ph++) {
		if (tv && col == (POST ? NCOL - 1 - ph : ph)) {
			float acc[IS3D ? 3 : 1];
#pragma unroll
			for (int lz = 0; lz < (IS3D ? 3 : 1); lz++) {
				float sacc = 0.f;
#pragma unroll
				for (int dy = -1; dy <= 1; dy++)
#pragma unroll
					for (int dx = -1; dx <= 1; dx++) {
						const int s = (dx + 1) + 3 * (dy + 1) + 9 * lz;
						if (s != C) sacc = fmaf(a[s], xs[me + dx + RX * dy + RXY * (lz - hz)], sacc);
					}
				acc[lz] = sacc;
			}
			const float tot = IS3D ? (acc[0] + acc[1]) + acc[IS3D ? 2 : 0] : acc[0];
			xs[me] = (bv - tot) / diag;
		}
		__syncthreads();
	}
	if (valid) xout[v] = xs[me];
}
template <bool IS3D, typename AT, bool POST>
__device__ __forceinline__ void body_smooth(const SmoothP& P, long long blk, long long) {
	smooth_tile<IS3D, AT, POST, false>(P, nullptr, blk);
}
struct RestrictSmoothP {
	RestrictP r;
	SmoothP s;
};
template <bool IS3D, typename AT>
__device__ __forceinline__ void body_restrict_smooth(const RestrictSmoothP& P, long long blk, long long) {
	smooth_tile<IS3D, AT, false, true>(P.s, &P.r, blk);
}

__device__ __forceinline__ void body_fill(const FillP& P, long long blk, long long) {
	if (P.st->done) return;
	const long long v = blk * 256 + threadIdx.x;
	if (v < P.n) P.x[v] = 0.f;
}

// coarsest level: x[cidx[i]] = sum_j G[i][j] * b[cidx[j]] (FP64), one wave per row;
// for a single-level hierarchy the rhs is the trivially scaled level-0 input
__device__ __forceinline__ void body_coarsest(const CoarsestP& P, long long blk, long long) {
	const CgState* __restrict__ st = P.st;
	const int nc = P.nc;
	const int* __restrict__ cidx = P.cidx;
	const double* __restrict__ G = P.G;
	const float* __restrict__ b = P.b;
	const uint8_t* __restrict__ code = P.code;
	float* __restrict__ x = P.x;
	// latency, not work: the state, the right-hand side's indices and the row
	// of the inverse are asked for together, kN of each per lane at a time
	// (past the end an index in range, and the value is not added): 729
	// unknowns 8.6 -> 3.6 us
	constexpr int kN = 12;
	const int done = st->done;
	const int lane = threadIdx.x & 63;
	const int row = (int)blk * 4 + (threadIdx.x >> 6);
	if (row >= nc) return;
	const int ov = cidx[row];
	double acc = 0.0;
	for (int j0 = 0; j0 < nc; j0 += 64 * kN) {
		int v[kN];
		double g[kN], bv[kN];
#pragma unroll
		for (int e = 0; e < kN; e++) v[e] = cidx[min(j0 + 64 * e + lane, nc - 1)];
#pragma unroll
		for (int e = 0; e < kN; e++) g[e] = G[(long long)row * nc + min(j0 + 64 * e + lane, nc - 1)];
#pragma unroll
		for (int e = 0; e < kN; e++) bv[e] = code ? (double)(b[v[e]] * l0_scale(code[v[e]])) : (double)b[v[e]];
#pragma unroll
		for (int e = 0; e < kN; e++)
			if (j0 + 64 * e + lane < nc) acc += g[e] * bv[e];
	}
	acc = wave_sum(acc);
	if (lane == 0 && !done) x[ov] = (float)acc;
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
MgHierarchy::~MgHierarchy() {
	if (arena) (void)hipFree(arena);
	if (hbuf) (void)hipHostFree(hbuf);
}

static unsigned nblk(long long n) {
	long long b = (n + 255) / 256;
	if (b < 1) b = 1;
	if (b > 65535) b = 65535;
	return (unsigned)b;
}

// Levels and their memory: one device block and one pinned block, laid out
// once.  A hierarchy rebuilt for another matrix of the same grid (PcMGDynamic
// in every solve, PcMIC when the flags changed) works in the same memory:
// allocating its 30 to 40 arrays and freeing them again took about 1 ms a
// solve.
void MgHierarchy::layout(Scene* s) {
	const Dims& d = s->d;
	is3d = d.is3d != 0;
	// the z-marching level-0 kernels keep in-plane offsets in 32 bits
	MFX_CHECK((long long)d.nx * d.ny < (1ll << 31), "multigrid: a grid plane has too many cells");
	S = is3d ? 14 : 5;
	L.clear();
	// level sizes (multigrid.cpp:242-262)
	MgLevel l0;
	l0.nx = d.nx;
	l0.ny = d.ny;
	l0.nz = d.nz;
	l0.n = d.n;
	l0.sy = d.nx;
	l0.sz = (long long)d.nx * d.ny;
	L.push_back(l0);
	long long n = d.n;
	for (int l = 1; l <= 100; l++) {
		const MgLevel& p = L.back();
		if (p.nx <= 5 && p.ny <= 5 && p.nz <= 5) break;
		if (n <= 1000) break;
		MgLevel c;
		c.nx = (p.nx + 2) / 2;
		c.ny = (p.ny + 2) / 2;
		c.nz = (p.nz + 2) / 2;
		c.n = (long long)c.nx * c.ny * c.nz;
		// the coarse-level kernels address vertices with 32-bit indices
		MFX_CHECK(c.n < (1ll << 31), "multigrid: coarse level has too many vertices");
		c.sy = c.nx;
		c.sz = (long long)c.nx * c.ny;
		n = c.n;
		L.push_back(c);
	}
	const int nl = (int)L.size();
	const size_t ncMax = (size_t)L[nl - 1].n;
	// two passes over the same list: sizes, then addresses
	for (int pass = 0; pass < 2; pass++) {
		size_t off = 0;
		auto take = [&](auto*& p, size_t count) {
			using T = std::remove_reference_t<decltype(*p)>;
			off = (off + 255) & ~(size_t)255;
			if (pass) p = (T*)((uint8_t*)arena + off);
			off += sizeof(T) * count;
		};
		// vectors that start at 0 (inactive vertices keep it): one run
		float* z0 = nullptr;
		take(z0, 0);
		const size_t zoff = off;
		for (int l = 1; l < nl; l++) {
			take(L[l].x, (size_t)L[l].n);
			take(L[l].xp, (size_t)L[l].n);
		}
		if (pass) {
			zero = (float*)((uint8_t*)arena + zoff);
			nzero = (long long)((off - zoff) / sizeof(float));
		}
		// what the host reads: the picked stencils, the coarsest operator
		CanonSlot* cs = nullptr;
		take(cs, (size_t)nl);
		picks = cs;
		if (nl > 1) {
			take(L[nl - 1].A, ncMax * (size_t)S);
			take(L[nl - 1].type, ncMax);
		}
		if (pass) readBytes = (size_t)((uint8_t*)arena + off - (uint8_t*)picks);
		take(L[0].r, (size_t)d.n);
		take(L[0].x, (size_t)d.n);
		for (int l = 1; l < nl; l++) {
			MgLevel& c = L[l];
			if (l < nl - 1) {
				take(c.A, (size_t)(c.n * S));
				take(c.type, (size_t)c.n);
				if (prec == 1) take(c.Ah, (size_t)(c.n * S));
			}
			take(c.b, (size_t)c.n);
			take(c.r, (size_t)c.n);
		}
		take(G, ncMax * ncMax);
		take(sweepD, (size_t)kSweep * kSweep);
		take(sweepW, ncMax * kSweep);
		take(sweepP, ncMax * kSweep);
		take(cdiag, ncMax);
		// what the host writes
		take(cidx, ncMax);
		take(cpos, ncMax);
		take(cpin, ncMax);
		if (!pass) {
			arenaBytes = off;
			MFX_HIP(hipMalloc(&arena, arenaBytes));
		}
	}
	hostBytes = std::max(readBytes, ncMax) + 256 + ((uint8_t*)(cpin + ncMax) - (uint8_t*)cidx);
	MFX_HIP(hipHostMalloc(&hbuf, hostBytes, hipHostMallocDefault));
}

void MgHierarchy::build(Scene* s, const uint8_t* code, int precision) {
	ready = false;
	if (!arena || !hbuf || prec != precision) {
		if (arena) MFX_HIP(hipFree(arena));
		if (hbuf) MFX_HIP(hipHostFree(hbuf));
		arena = hbuf = nullptr;
		prec = precision;
		layout(s);
	}
	hipStream_t q = s->stream;
	const int nl = (int)L.size();
	if (nzero) hipLaunchKernelGGL(k_fill_f, dim3(nblk(nzero)), dim3(256), 0, q, zero, nzero);
	for (int l = 1; l < nl; l++) {
		MgLevel& c = L[l];
		const MgLevel& f = L[l - 1];
		const uint8_t* fc = l == 1 ? code : nullptr;
		hipLaunchKernelGGL(k_mg_activate, dim3(nblk(c.n)), dim3(256), 0, q, lvdev(c), lvdev(f), (int)is3d, fc, f.type,
		                   c.type);
		hipLaunchKernelGGL(k_mg_cover, dim3(nblk(f.n)), dim3(256), 0, q, lvdev(c), lvdev(f), (int)is3d, fc, f.type,
		                   c.type);
		hipLaunchKernelGGL(k_mg_cover_done, dim3(nblk(c.n)), dim3(256), 0, q, lvdev(c), c.type);
		const FineOp F{fc, f.A, f.type, lvdev(f)};
		const dim3 gb((unsigned)((c.n + (is3d ? 7 : 15)) / (is3d ? 8 : 16)));
		auto* kern = is3d ? (fc ? k_mg_galerkin<true, true> : k_mg_galerkin<true, false>)
		                  : (fc ? k_mg_galerkin<false, true> : k_mg_galerkin<false, false>);
		hipLaunchKernelGGL(kern, gb, dim3(256), 0, q, F, lvdev(c), (const uint8_t*)c.type, c.A, c.r);
		hipLaunchKernelGGL(k_mg_drop, dim3(nblk(c.n)), dim3(256), 0, q, lvdev(c), c.type, (const float*)c.A,
		                   (const float*)c.r);
		// the coarsest level is solved through G; the others get a canonical stencil
		if (l == nl - 1) break;
		hipLaunchKernelGGL(k_mg_pick, dim3(1), dim3(1024), 0, q, lvdev(c), (int)is3d, (const float*)c.A,
		                   (const uint8_t*)c.type, picks + l);
		hipLaunchKernelGGL(k_mg_classify, dim3(nblk(c.n)), dim3(256), 0, q, lvdev(c), (int)is3d, S, (const float*)c.A,
		                   c.type, (const CanonSlot*)(picks + l));
	}
	build_coarsest(s, code);
	const CanonSlot* hp = (const CanonSlot*)hbuf;
	for (int l = 1; l + 1 < nl; l++) {
		MgLevel& c = L[l];
		c.hasCanon = hp[l].has != 0;
		c.canon = hp[l].cn;
		if (prec == 1) {
			// mixed precision: smoother and residual read BF16 coefficients; the
			// canonical stencil is rounded the same way so that every coupling
			// has one value seen from both of its vertices (symmetric V-cycle)
			hipLaunchKernelGGL(k_to_bf16, dim3(nblk(c.n * S)), dim3(256), 0, q, (const float*)c.A, c.Ah, c.n * S);
			for (int e = 0; e < 27; e++) c.canon.a[e] = from_bf16(to_bf16(c.canon.a[e]));
		}
	}
	ready = true;
}

// Dense generalised inverse of the coarsest operator (FP64).  The host reads
// the operator once (with the picked stencils, the only wait of a build),
// numbers its active vertices and finds the singular blocks; the matrix is
// assembled and inverted on the device.
void MgHierarchy::build_coarsest(Scene* s, const uint8_t* code0) {
	hipStream_t q = s->stream;
	const int lc = (int)L.size() - 1;
	const MgLevel& c = L[lc];
	uint8_t* hb = (uint8_t*)hbuf;
	if (lc == 0) MFX_HIP(hipMemcpyAsync(hb, code0, (size_t)c.n, hipMemcpyDeviceToHost, q));
	else MFX_HIP(hipMemcpyAsync(hb, picks, readBytes, hipMemcpyDeviceToHost, q));
	sync(s);
	const uint8_t* hcode = hb;
	const float* A = lc ? (const float*)(hb + ((uint8_t*)c.A - (uint8_t*)picks)) : nullptr;
	const uint8_t* type = lc ? hb + (c.type - (uint8_t*)picks) : nullptr;
	// host copies of cidx, cpos, cpin, laid out as on the device
	uint8_t* hw = hb + ((std::max(readBytes, (size_t)c.n) + 255) & ~(size_t)255);
	int* idx = (int*)hw;
	int* pos = (int*)(hw + ((uint8_t*)cpos - (uint8_t*)cidx));
	int* pin = (int*)(hw + ((uint8_t*)cpin - (uint8_t*)cidx));
	int m = 0;
	for (long long v = 0; v < c.n; v++) {
		const bool act = lc ? type[v] != 0 : (hcode[v] & 7) != 0;
		pos[v] = act ? m : -1;
		if (act) idx[m++] = (int)v;
	}
	nc = m;
	const int C = S - 1;
	// f(b, value) for the stored couplings of row a (b: the column)
	auto row = [&](int a, auto&& f) {
		const long long v = idx[a];
		const int i = (int)(v % c.nx), j = (int)((v / c.nx) % c.ny), k = (int)(v / c.sz);
		for (int dz = is3d ? -1 : 0; dz <= (is3d ? 1 : 0); dz++)
			for (int dy = -1; dy <= 1; dy++)
				for (int dx = -1; dx <= 1; dx++) {
					const int ni = i + dx, nj = j + dy, nk = k + dz;
					if (ni < 0 || nj < 0 || nk < 0 || ni >= c.nx || nj >= c.ny || nk >= c.nz) continue;
					const long long w = ni + c.sy * nj + c.sz * nk;
					if (pos[w] < 0) continue;
					const int si = is3d ? (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1) : (dx + 1) + 3 * (dy + 1);
					double val;
					if (lc == 0) {
						if ((dx != 0) + (dy != 0) + (dz != 0) > 1) continue;
						const uint8_t cv = hcode[v], cw = hcode[w];
						const int bit = dx ? 8 : (dy ? 16 : 32);
						if (si == C) val = (cv & 128) ? (double)((float)(cv & 7) * 1e-6f) : (double)(cv & 7);
						else val = ((si > C ? cv : cw) & bit) ? -1.0 : 0.0;
					} else {
						val = si >= C ? A[(size_t)(si - C) * c.n + v] : A[(size_t)(C - si) * c.n + w];
					}
					f(pos[w], val);
				}
	};
	// Pure-Neumann blocks (fluid pockets enclosed by obstacles, or a closed
	// domain) are singular; with float coefficients their last pivot is
	// round-off rather than zero and would put ~1e7-sized entries into G.
	// Pin one vertex of every connected component whose rows all sum to ~0.
	std::fill(pin, pin + m, 0);
	{
		std::vector<char> seen((size_t)m, 0);
		std::vector<int> stack, members;
		for (int a0 = 0; a0 < m; a0++) {
			if (seen[(size_t)a0]) continue;
			members.clear();
			seen[(size_t)a0] = 1;
			stack.push_back(a0);
			double maxSum = 0.0, maxDiag = 0.0;
			int last = a0;
			while (!stack.empty()) {
				const int a = stack.back();
				stack.pop_back();
				members.push_back(a);
				last = std::max(last, a);
				double rs = 0.0;
				row(a, [&](int b, double val) {
					rs += val;
					if (b == a) maxDiag = std::max(maxDiag, val);
					if (b != a && !seen[(size_t)b] && val != 0.0) {
						seen[(size_t)b] = 1;
						stack.push_back(b);
					}
				});
				maxSum = std::max(maxSum, std::fabs(rs));
			}
			if (members.size() > 1 && maxSum <= 1e-5 * maxDiag) pin[last] = 1;
		}
	}
	MFX_HIP(hipMemcpyAsync(cidx, hw, (size_t)((uint8_t*)(cpin + c.n) - (uint8_t*)cidx), hipMemcpyHostToDevice, q));
	if (!m) return;
	hipLaunchKernelGGL(k_fill_d, dim3(nblk((long long)m * m)), dim3(256), 0, q, G, (long long)m * m);
	hipLaunchKernelGGL(k_dense_assemble, dim3((unsigned)((27 * m + 255) / 256)), dim3(256), 0, q, lvdev(c), (int)is3d, S,
	                   m, (const int*)cidx, (const int*)cpos, (const float*)c.A, lc == 0 ? code0 : (const uint8_t*)nullptr,
	                   G, cdiag);
	const unsigned nt = (unsigned)((m + kDTile - 1) / kDTile);
	for (int k0 = 0; k0 < m; k0 += kSweep) {
		hipLaunchKernelGGL(k_sweep_panel, dim3(nt), dim3(256), 0, q, m, k0, (const double*)G, (const double*)cdiag,
		                   (const int*)cpin, sweepD, sweepW, sweepP);
		hipLaunchKernelGGL(k_sweep_update, dim3(nt, nt), dim3(256), 0, q, m, k0, G, (const double*)sweepD,
		                   (const double*)sweepW, (const double*)sweepP, k0 + kSweep >= m ? 1 : 0);
	}
}

// ---------------------------------------------------------------------------
// launches (single problem and work lists)
// ---------------------------------------------------------------------------
constexpr int kZmTY = kZmTYHost;
long long l0_tiles(const Dims& d, int* kchunk, bool tuned, int force) {
	// 3D: z-marching 64 x kZmTY column tiles over chunks of a multiple of
	// kDotGroup planes (even, as the restriction pairs planes), halved while
	// fewer than about 8192 wavefronts (one per SIMD slot of the chip) cover
	// the grid; 2D: bricks of 64x16 cells
	const int BY = d.is3d ? kZmTY : 16;
	const long long cols = (long long)((d.nx + 63) / 64) * ((d.ny + BY - 1) / BY);
	if (!d.is3d) {
		*kchunk = 2;
		return cols;
	}
	int kc = zm_chunk(d.nz);
	while (kc > 16 && cols * ((d.nz + kc - 1) / kc) < 8192 / kZmTY) kc = zm_chunk(kc / 2);
	if (tuned && zm_tuned(d).l0 > 0) kc = zm_tuned(d).l0;
	if (force > 0) kc = force;
	*kchunk = kc;
	return cols * ((d.nz + kc - 1) / kc);
}
long long lcblk_tiles(const LvDev& c, bool is3d) {
	const long long bx = is3d ? kLcBX3 : kLcBX2, by = is3d ? kLcBY3 : kLcBY2, bz = is3d ? kLcBZ3 : 1;
	return ((c.nx + bx - 1) / bx) * ((c.ny + by - 1) / by) * ((c.nz + bz - 1) / bz);
}
void run_l0_down_one(hipStream_t s, bool is3d, unsigned nb, const L0DownP& p) {
	if (is3d) launch_one<L0DownP, body_l0_down_zm<kZmTY>, 64 * kZmTY, 8>(s, nb, p);
	else launch_one<L0DownP, body_l0_down_brick<64, 16, 1, false>, 1024>(s, nb, p);
}
void run_l0_down_many(hipStream_t s, bool is3d, unsigned nb, WorkList items, const L0DownP* p) {
	if (is3d) launch_many<L0DownP, body_l0_down_zm<kZmTY>, 64 * kZmTY, 8>(s, nb, items, p);
	else launch_many<L0DownP, body_l0_down_brick<64, 16, 1, false>, 1024>(s, nb, items, p);
}
void run_l0_up_many(hipStream_t s, bool is3d, unsigned nb, WorkList items, const L0UpP* p) {
	if (is3d) launch_many<L0UpP, body_l0_up_zm<kZmTY>, 64 * kZmTY, 8>(s, nb, items, p);
	else launch_many<L0UpP, body_l0_up_brick<64, 16, 1, false>, 1024>(s, nb, items, p);
}
void run_restrict_many(hipStream_t s, bool is3d, unsigned nb, WorkList items, const RestrictP* p) {
	if (is3d) launch_many<RestrictP, body_restrict<true>, 256>(s, nb, items, p);
	else launch_many<RestrictP, body_restrict<false>, 256>(s, nb, items, p);
}
template <bool POST>
static void run_smooth_mode(hipStream_t s, bool is3d, bool bf16, unsigned nb, WorkList items,
                            const SmoothP* p) {
	if (is3d && bf16) launch_many<SmoothP, body_smooth<true, uint16_t, POST>, kSmoothNT>(s, nb, items, p);
	else if (is3d) launch_many<SmoothP, body_smooth<true, float, POST>, kSmoothNT>(s, nb, items, p);
	else if (bf16) launch_many<SmoothP, body_smooth<false, uint16_t, POST>, kSmoothNT>(s, nb, items, p);
	else launch_many<SmoothP, body_smooth<false, float, POST>, kSmoothNT>(s, nb, items, p);
}
void run_smooth_many(hipStream_t s, bool is3d, bool bf16, bool post, unsigned nb, WorkList items,
                     const SmoothP* p) {
	if (post) run_smooth_mode<true>(s, is3d, bf16, nb, items, p);
	else run_smooth_mode<false>(s, is3d, bf16, nb, items, p);
}
void run_resid_many(hipStream_t s, bool is3d, bool bf16, unsigned nb, WorkList items, const ResidP* p) {
	if (is3d && bf16) launch_many<ResidP, body_resid<true, uint16_t>, 256>(s, nb, items, p);
	else if (is3d) launch_many<ResidP, body_resid<true, float>, 256>(s, nb, items, p);
	else if (bf16) launch_many<ResidP, body_resid<false, uint16_t>, 256>(s, nb, items, p);
	else launch_many<ResidP, body_resid<false, float>, 256>(s, nb, items, p);
}
void run_coarsest_many(hipStream_t s, unsigned nb, WorkList items, const CoarsestP* p) {
	launch_many<CoarsestP, body_coarsest, 256>(s, nb, items, p);
}
void run_fill_many(hipStream_t s, unsigned nb, WorkList items, const FillP* p) {
	launch_many<FillP, body_fill, 256>(s, nb, items, p);
}

// Parameters of every V-cycle step of this hierarchy (shared by the single
// launch sequence below and by batched work lists).
MgHierarchy::Steps MgHierarchy::steps(const Dims& d, const uint8_t* code, const float* r, float* z, const CgState* st,
                                      double* part, bool tuned, int forceChunk) const {
	Steps S_;
	const int nl = (int)L.size();
	S_.nl = nl;
	S_.l0Tiles = l0_tiles(d, &S_.kchunk, tuned, forceChunk);
	S_.nPart = is3d ? zm_dot_parts(d, kZmTY) : S_.l0Tiles;
	const void* noA = nullptr;
	if (nl == 1) {
		S_.fill = FillP{st, z, d.n};
		S_.coarsest = CoarsestP{st, nc, cidx, G, r, code, z};
		return S_;
	}
	S_.down = L0DownP{d, S_.kchunk, st, code, r, L[0].x, L[0].r};
	for (int l = 1; l < nl; l++) {
		const MgLevel& c = L[l];
		const MgLevel& f = L[l - 1];
		Steps::Level q;
		q.restrict_ = RestrictP{st, lvdev(c), lvdev(f), c.type, f.r, c.b};
		q.tiles = lc_tiles(lvdev(c));
		q.blkTiles = lcblk_tiles(lvdev(c), is3d);
		if (l < nl - 1) {
			const void* A = c.Ah ? (const void*)c.Ah : (const void*)c.A;
			q.pre = SmoothP{st, lvdev(c), A, c.type, c.b, nullptr, c.x, 1, 0, lvdev(c), nullptr, c.canon};
			q.resid = ResidP{st, lvdev(c), A, c.type, c.b, c.x, c.r, c.canon};
			const MgLevel& cc = L[l + 1];
			q.post = SmoothP{st, lvdev(c), A, c.type, c.b, c.x, c.xp, 0, 1, lvdev(cc), l + 1 == nl - 1 ? cc.x : cc.xp,
			                 c.canon};
		}
		S_.lv.push_back(q);
	}
	(void)noA;
	S_.coarsest = CoarsestP{st, nc, cidx, G, L[nl - 1].b, nullptr, L[nl - 1].x};
	const MgLevel& c1 = L[1];
	S_.up = L0UpP{d, S_.kchunk, st, code, r, L[0].x, z, lvdev(c1), nl == 2 ? c1.x : c1.xp, part};
	return S_;
}

// Levels of at most this many smoother bricks restrict inside the smoother
// (single solves).  There a restriction is a launch of 3 us and its gap; on
// larger levels the smoother's colour order of vertices costs the rows' loads
// more than the launch.  Two launches / fused: 17^3 and 33^3 9.3 / 6.5 us,
// 65^3 (867 bricks) 12.5 / 10.1, 129^3 (5445) 48.3 / 49.9.
constexpr long long kFuseBricks = 1024;
int MgHierarchy::vcycle(Scene* s, const uint8_t* code, const float* r, float* z, const CgState* st) {
	const Dims& d = s->d;
	const Steps S_ = steps(d, code, r, z, st, s->dpart, true);
	hipStream_t q = s->stream;
	const bool bf = prec == 1;
	if (S_.nl == 1) {
		launch_one<FillP, body_fill, 256>(q, (d.n + 255) / 256, S_.fill);
		launch_one<CoarsestP, body_coarsest, 256>(q, coarsest_tiles(nc), S_.coarsest);
		return 0;
	}
	{
		KtScope kt("mg_l0_down", q);
		if (is3d) launch_one<L0DownP, body_l0_down_zm<kZmTY>, 64 * kZmTY, 8>(q, S_.l0Tiles, S_.down);
		else launch_one<L0DownP, body_l0_down_brick<64, 16, 1, false>, 1024>(q, S_.l0Tiles, S_.down);
	}
	const int nlv = (int)S_.lv.size();
	for (int i = 0; i < nlv; i++) {
		const Steps::Level& v = S_.lv[i];
		const bool last = i == nlv - 1, fused = !last && v.blkTiles <= kFuseBricks;
		if (!fused) {
			if (is3d) launch_one<RestrictP, body_restrict<true>, 256>(q, v.tiles, v.restrict_);
			else launch_one<RestrictP, body_restrict<false>, 256>(q, v.tiles, v.restrict_);
		}
		if (last) break;
		auto down = [&](auto d3, auto at) {
			constexpr bool D = decltype(d3)::value;
			using AT = decltype(at);
			if (fused)
				launch_one<RestrictSmoothP, body_restrict_smooth<D, AT>, kSmoothNT>(q, v.blkTiles,
				                                                                    RestrictSmoothP{v.restrict_, v.pre});
			else launch_one<SmoothP, body_smooth<D, AT, false>, kSmoothNT>(q, v.blkTiles, v.pre);
			launch_one<ResidP, body_resid<D, AT>, 256>(q, v.tiles, v.resid);
		};
		if (is3d && bf) down(std::true_type{}, uint16_t{});
		else if (is3d) down(std::true_type{}, float{});
		else if (bf) down(std::false_type{}, uint16_t{});
		else down(std::false_type{}, float{});
	}
	launch_one<CoarsestP, body_coarsest, 256>(q, coarsest_tiles(nc), S_.coarsest);
	for (int i = nlv - 2; i >= 0; i--) {
		const Steps::Level& v = S_.lv[i];
		if (is3d && bf) launch_one<SmoothP, body_smooth<true, uint16_t, true>, kSmoothNT>(q, v.blkTiles, v.post);
		else if (is3d) launch_one<SmoothP, body_smooth<true, float, true>, kSmoothNT>(q, v.blkTiles, v.post);
		else if (bf) launch_one<SmoothP, body_smooth<false, uint16_t, true>, kSmoothNT>(q, v.blkTiles, v.post);
		else launch_one<SmoothP, body_smooth<false, float, true>, kSmoothNT>(q, v.blkTiles, v.post);
	}
	{
		KtScope kt("mg_l0_up", q);
		if (is3d) launch_one<L0UpP, body_l0_up_zm<kZmTY>, 64 * kZmTY, 8>(q, S_.l0Tiles, S_.up);
		else launch_one<L0UpP, body_l0_up_brick<64, 16, 1, false>, 1024>(q, S_.l0Tiles, S_.up);
	}
	return (int)S_.nPart;
}

}  // namespace mfx
