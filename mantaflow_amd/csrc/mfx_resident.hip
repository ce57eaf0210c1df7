// Unpreconditioned CG of a whole small grid as one kernel.
//
// GridCg's iteration (conjugategrad.cpp:238-299) without a preconditioner is
// a 5- or 7-point product, two vector updates and two reductions over a few
// thousand to a few hundred thousand cells.  As four launches an iteration
// costs about 15 us whatever the grid size: every launch pays its start, the
// load of its operands from L2 and its drain, and the arithmetic in between
// is well under a microsecond.  Here the cells stay in registers for the
// whole solve: a thread owns V cells and keeps their x, r, p and matrix
// coefficients, the search direction of a workgroup's run of cells (plus one
// row, in 3D one plane, on each side) is in LDS, and only the two dot
// products and the residuals along the run's ends leave the workgroup.  An
// iteration is bound by the latency of its reductions: 64^2 (one workgroup)
// 15.6 -> 2.05 us, 353x241 (42 workgroups) 15.3 -> 4.6 us, 24^3 (7) 4.8 us.
//
// Workgroups meet through memory twice per iteration without a grid barrier:
// every word exchanged carries the number of the iteration it belongs to in
// its upper half, so one store publishes it and the reader polls the word
// itself until the number matches; no fence, no flag, no L2 write-back (the
// stores and loads are agent-scope atomics, which bypass the XCDs' L2s).  A
// slot is written again only after every reader has shown, by publishing its
// own part of the next reduction, that it has read the old value, so one
// slot per workgroup and reduction is enough.
//
// The workgroups of a solve have to be on the GPU together.  At most kResMaxWG
// are launched, and the solves in flight on a device are kept to as many as
// leave every workgroup of theirs a compute unit of its own: a workgroup that
// has not started finds a unit without one of them, whose other work ends by
// itself (cg_resident_run).  Other processes on the device are not counted, so
// every wait is bounded by the clock as well: a workgroup that waits longer
// than `limit` ticks gives up, marks the solve as aborted and leaves; the
// host then runs the solve again on the general kernels, and the next ones of
// that solver too (ResWords::rest).
#include <algorithm>
#include <limits>
#include <mutex>
#include <type_traits>
#include <vector>

#include "mfx_batch.h"
#include "mfx_internal.h"
#include "mfx_resident.h"

namespace mfx {

namespace {

constexpr int kMaxNW = 16;  // wavefronts of the largest workgroup
// exchanged words of one reduction: A = dot(q, p); B = dot(r, r), sum r^2
// (two words per double) and max |r|
constexpr int kWordsA = 2, kWordsB = 5;
constexpr long long kMaxLds = 60 * 1024;  // search direction of a run
constexpr int kSlot = 8;  // words per workgroup and reduction (one 64-byte line)

__device__ inline unsigned long long xload(const unsigned long long* p) {
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xstore(unsigned long long* p, unsigned tag, unsigned v) {
	__hip_atomic_store(p, ((unsigned long long)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum of the 16 doubles sh[0..15] in a fixed order, in every lane
__device__ inline double sum16(const double* sh) {
	double v = sh[threadIdx.x & 15];
	v += dpp_move_d<0x111, 0xf>(v);
	v += dpp_move_d<0x112, 0xf>(v);
	v += dpp_move_d<0x114, 0xf>(v);
	v += dpp_move_d<0x118, 0xf>(v);
	const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
	const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, 15);
	const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), 15);
	return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// maximum over the wavefront, valid in lane 63 (the moves of wave_sum_to_last;
// a lane that a move does not write keeps its own value)
template <int CTRL, int ROWS>
__device__ inline float dpp_max(float v) {
	const int u = __float_as_int(v);
	return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(u, u, CTRL, ROWS, 0xf, false)));
}
__device__ inline float wave_max_to_last(float v) {
	v = dpp_max<0x111, 0xf>(v);
	v = dpp_max<0x112, 0xf>(v);
	v = dpp_max<0x114, 0xf>(v);
	v = dpp_max<0x118, 0xf>(v);
	v = dpp_max<0x142, 0xa>(v);
	v = dpp_max<0x143, 0xc>(v);
	return v;
}
__device__ inline double word_pair(unsigned long long lo, unsigned long long hi) {
	return __builtin_bit_cast(double, ((hi & 0xffffffffull) << 32) | (lo & 0xffffffffull));
}

struct ResShared {
	double a[kMaxNW], b[kMaxNW], c[kMaxNW];  // the wavefronts' partials of dot(q,p); dot(r,r); sum r^2
	float m[kMaxNW];
	double tot[3];
	float totm;
	int abort;  // some thread of this workgroup gave up waiting
	int dead;   // abort as of the last reduction (the same in every thread)
};

// Words [0, NW) of every workgroup's slot with the tag: lane l reads
// workgroup l's (wavefront 0 only; at most 64 workgroups).  The wait is timed
// from its first poll in vain; a workgroup that has given up does not wait.
template <int NW>
__device__ inline void gather(const unsigned long long* slots, int nwg, unsigned tag, long long limit, int* abort,
                              unsigned long long* w) {
	const int l = threadIdx.x;
	long long since = 0;
	for (;;) {
		bool ok = true;
		if (l < nwg) {
#pragma unroll
			for (int q = 0; q < NW; q++) w[q] = xload(slots + (size_t)l * kSlot + q);
#pragma unroll
			for (int q = 0; q < NW; q++) ok = ok && (unsigned)(w[q] >> 32) == tag;
		}
		if (__all(ok)) return;
		const long long now = wall_clock64();
		if (since == 0) since = now;
		if (*abort || now - since >= limit) {
			*abort = 1;
			return;
		}
	}
}

}  // namespace

// Workgroup wg of nwg, of NT threads of V cells; MULTI: several workgroups
template <int NT, int V, bool MULTI>
__device__ __forceinline__ void body_cg_resident(const ResP& P, int wg, int nwg) {
	extern __shared__ float ps[];  // p of cells c0-H .. c0+C+H-1
	__shared__ ResShared S;
	constexpr int C = NT * V;
	const Dims& d = P.d;
	const int t = threadIdx.x, lane = t & 63, w = t >> 6;
	const int H = P.H;
	const long long n = d.n, c0 = (long long)wg * C;
	const int cnt = (int)min((long long)C, n - c0);
	const int sx = 1, sy = d.nx, sz = (int)d.sz;
	CgState* st = P.st;
	const int maxIter = st->maxIter, useL2 = st->useL2;
	const double relTol = st->relTol;
	const float acc = st->acc;
	const bool needRR = relTol > 0 || useL2;
	unsigned long long* slA = P.xs;
	unsigned long long* slB = P.xs + (size_t)kResMaxWG * kSlot;
	bool gaveUp = false;
	if (t == 0) S.abort = 0;
	if (NT < 64 * kMaxNW && t < kMaxNW) {
		// (the sums run over kMaxNW wavefronts)
		S.a[t] = S.b[t] = S.c[t] = 0.0;
		S.m[t] = -1.f;
	}
	if (NT < 64 * kMaxNW) __syncthreads();

	// the cells: r = b, x = 0, and the row's coefficients as bits (0-2 A0,
	// 3/4/5 and 8/9/10 coupled to the upper / lower x, y, z neighbour, 6 fluid)
	float x[V], r[V], p[V];
	int pk[V];
	double zr = 0, rr = 0;
#pragma unroll
	for (int v = 0; v < V; v++) {
		const int l = t + NT * v;
		const bool in = l < cnt;
		const long long c = c0 + (in ? l : 0);
		const long long xm = c - sx >= 0 ? c - sx : c, ym = c - sy >= 0 ? c - sy : c, zm = c - sz >= 0 ? c - sz : c;
		const int cc = P.code[c], cx = P.code[xm], cy = P.code[ym], cz = P.code[zm];
		const float b = P.b[c];
		r[v] = in ? b : 0.f;
		x[v] = 0.f;
		p[v] = 0.f;
		int k = cc & 127;
		if (xm != c && (cx & 8)) k |= 1 << 8;
		if (ym != c && (cy & 16)) k |= 1 << 9;
		if (d.is3d && zm != c && (cz & 32)) k |= 1 << 10;
		pk[v] = in ? k : 0;
		zr += (double)(r[v] * r[v]);
		rr += (double)r[v] * (double)r[v];
	}
	// diagonals of the row kinds: A0, or fl(fl(A0 scale) + 1)
	__shared__ float dg[8];
	if (t < 8) dg[t] = P.scaled ? (float)((double)((float)t * P.scale) + 1.0) : (float)t;
	const float off = P.scaled ? -P.scale : -1.f;

	// one reduction of (zr, rr, m) over the grid, in every thread
	float m = -1.f;
	auto reduce_b = [&](unsigned tag, double& oz, double& orr, float& om) {
		const double a = wave_sum_to_last(zr);
		const double b = needRR || tag == P.epoch ? wave_sum_to_last(rr) : 0.0;
		const float mm = wave_max_to_last(m);
		if (lane == 63) {
			S.b[w] = a;
			S.c[w] = b;
			S.m[w] = mm;
		}
		__syncthreads();
		if (!MULTI) {
			oz = sum16(S.b);
			orr = sum16(S.c);
			float q = S.m[lane & 15];
			q = dpp_max<0x111, 0xf>(q);
			q = dpp_max<0x112, 0xf>(q);
			q = dpp_max<0x114, 0xf>(q);
			q = dpp_max<0x118, 0xf>(q);
			om = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q), 15));
			return;
		}
		if (w == 0) {
			const double z0 = sum16(S.b), r0 = sum16(S.c);
			float q = S.m[lane & 15];
			q = dpp_max<0x111, 0xf>(q);
			q = dpp_max<0x112, 0xf>(q);
			q = dpp_max<0x114, 0xf>(q);
			q = dpp_max<0x118, 0xf>(q);
			const unsigned m0 = (unsigned)__builtin_amdgcn_readlane(__float_as_int(q), 15);
			const unsigned long long zu = __builtin_bit_cast(unsigned long long, z0);
			const unsigned long long ru = __builtin_bit_cast(unsigned long long, r0);
			const unsigned word = lane == 0   ? (unsigned)zu
			                      : lane == 1 ? (unsigned)(zu >> 32)
			                      : lane == 2 ? (unsigned)ru
			                      : lane == 3 ? (unsigned)(ru >> 32)
			                                  : m0;
			if (lane < kWordsB) xstore(slB + (size_t)wg * kSlot + lane, tag, word);
			unsigned long long g[kWordsB];
			gather<kWordsB>(slB, nwg, tag, P.limit, &S.abort, g);
			const bool mine = lane < nwg;
			const double sz_ = wave_sum_to_last(mine ? word_pair(g[0], g[1]) : 0.0);
			const double sr_ = wave_sum_to_last(mine ? word_pair(g[2], g[3]) : 0.0);
			const float sm_ = wave_max_to_last(mine ? __int_as_float((int)(unsigned)g[4]) : -1.f);
			if (lane == 63) {
				S.tot[1] = sz_;
				S.tot[2] = sr_;
				S.totm = sm_;
				S.dead = S.abort;
			}
		}
		__syncthreads();
		oz = S.tot[1];
		orr = S.tot[2];
		om = S.totm;
	};

	// doInit (conjugategrad.cpp:210-235)
	unsigned tag = P.epoch;
	double sumZ, sumR;
	float maxR;
	reduce_b(tag, sumZ, sumR, maxR);
	float sigma = (float)sumZ, alpha = 0.f, beta = 0.f, resNorm = 1e20f;
	const double bnorm2 = sumR;
	bool first = true, done = maxIter <= 0, converged = false, diverged = false;
	int iter = 0;
	double lastRR = 0;
	bool dead = MULTI && S.dead != 0;
	while (!done && !dead) {
		// p = r, or r + beta p; the neighbouring runs' ends from their owners
		if (MULTI) {
			for (int h = t; h < 2 * H; h += NT) {
				const long long g = h < H ? c0 - H + h : c0 + C + (h - H);
				const int q = h < H ? h : C + h;
				float pv = 0.f;
				if (g >= 0 && g < n) {
					float hr;
					if (first) {
						hr = P.b[g];
					} else {
						unsigned long long u;
						long long since = 0;
						while ((unsigned)((u = xload(P.xr + g)) >> 32) != tag && !gaveUp) {
							const long long now = wall_clock64();
							if (since == 0) since = now;
							if (now - since >= P.limit) {
								S.abort = 1;
								gaveUp = true;
							}
						}
						hr = __int_as_float((int)(unsigned)u);
					}
					pv = first ? hr : hr + beta * ps[q];
				}
				ps[q] = pv;
			}
		} else if (first) {
			for (int h = t; h < 2 * H; h += NT) ps[h < H ? h : C + h] = 0.f;
		}
#pragma unroll
		for (int v = 0; v < V; v++) {
			p[v] = first ? r[v] : r[v] + beta * p[v];
			ps[H + t + NT * v] = p[v];
		}
		tag++;
		__syncthreads();
		// q = A p in ApplyMatrix's term order (conjugategrad.h:118-151);
		// neighbours outside the grid are cells of value 0
		float q[V];
		double dq = 0;
#pragma unroll
		for (int v = 0; v < V; v++) {
			const int k = pk[v];
			const float* s = ps + H + t + NT * v;
			const float s0 = p[v];
			float a = s0 * dg[k & 7] + s[-sx] * ((k & 256) ? off : 0.f) + s[sx] * ((k & 8) ? off : 0.f) +
			          s[-sy] * ((k & 512) ? off : 0.f) + s[sy] * ((k & 16) ? off : 0.f);
			if (d.is3d) a = a + s[-sz] * ((k & 1024) ? off : 0.f) + s[sz] * ((k & 32) ? off : 0.f);
			q[v] = (k & 64) ? a : s0;
			dq += (double)(q[v] * s0);
		}
		dq = wave_sum_to_last(dq);
		if (lane == 63) S.a[w] = dq;
		__syncthreads();
		double sumA;
		if (MULTI) {
			if (w == 0) {
				const unsigned long long u = __builtin_bit_cast(unsigned long long, sum16(S.a));
				if (lane < kWordsA)
					xstore(slA + (size_t)wg * kSlot + lane, tag, lane ? (unsigned)(u >> 32) : (unsigned)u);
				unsigned long long g[kWordsA];
				gather<kWordsA>(slA, nwg, tag, P.limit, &S.abort, g);
				const double s = wave_sum_to_last(lane < nwg ? word_pair(g[0], g[1]) : 0.0);
				if (lane == 63) S.tot[0] = s;
			}
			__syncthreads();
			sumA = S.tot[0];
		} else {
			sumA = sum16(S.a);
		}
		const float dp = (float)sumA;
		alpha = fabsf(dp) > 0.f ? sigma / dp : 0.f;
		first = false;
		const float malpha = -alpha;
		zr = 0;
		rr = 0;
		m = -1.f;
#pragma unroll
		for (int v = 0; v < V; v++) {
			const int l = t + NT * v;
			x[v] = x[v] + alpha * p[v];
			r[v] = r[v] + malpha * q[v];
			if (MULTI && l < cnt && (l < H || l >= C - H)) xstore(P.xr + c0 + l, tag, (unsigned)__float_as_int(r[v]));
			const float e = r[v], ae = fabsf(e);
			if (l < cnt && ae > m) m = ae;
			zr += (double)(e * e);
		}
		if (needRR) {
#pragma unroll
			for (int v = 0; v < V; v++) rr += (double)r[v] * (double)r[v];
		}
		reduce_b(tag, sumZ, sumR, maxR);
		dead = MULTI && S.dead != 0;
		// the scalar rules of body_finalize (FIN_RES without preconditioner)
		iter++;
		lastRR = sumR;
		bool conv;
		if (relTol > 0) {
			resNorm = (float)sqrt(sumR / (bnorm2 > 0 ? bnorm2 : 1.0));
			conv = sqrt(sumR) <= relTol * sqrt(bnorm2);
		} else {
			if (useL2) resNorm = (float)sumR;
			else resNorm = maxR < 0.f ? 3.402823466e+38f : maxR;  // (no finite or infinite value: all NaN)
			conv = resNorm < acc;
		}
		if (wg == 0 && t == 0 && iter - 1 < 64) st->hist[iter - 1] = resNorm;
		if (conv) {
			sigma = resNorm;
			converged = done = true;
		} else {
			const float sigmaNew = (float)sumZ;
			beta = sigmaNew / sigma;
			sigma = sigmaNew;
			if (!(resNorm < 1e35f)) diverged = done = true;
			else if (iter >= maxIter) done = true;
		}
	}
#pragma unroll
	for (int v = 0; v < V; v++) {
		const int l = t + NT * v;
		if (l < cnt) P.x[c0 + l] = x[v];
	}
	if (dead) {
		// (any workgroup may be the one that gave up)
		if (t == 0) {
			st->pad = 1;
			st->converged = 0;
			st->done = 1;
		}
		return;
	}
	if (wg == 0 && t == 0) {
		st->sigma = sigma;
		st->alpha = alpha;
		st->beta = beta;
		st->bnorm2 = bnorm2;
		st->rr = lastRR;
		st->resNorm = resNorm;
		st->iter = iter;
		st->first = first ? 1 : 0;
		st->converged = converged ? 1 : 0;
		st->diverged = diverged ? 1 : 0;
		st->done = 1;
	}
}
template <int NT, int V, bool MULTI>
__global__ void __launch_bounds__(NT) k_cg_resident(ResP p) {
	body_cg_resident<NT, V, MULTI>(p, (int)blockIdx.x, (int)gridDim.x);
}
// the workgroups of several solves, from workgroup `base` of the list
template <int NT, int V, bool MULTI>
__global__ void __launch_bounds__(NT) k_cg_resident_many(WorkList wl, const ResP* __restrict__ params, int base) {
	const int b = base + (int)blockIdx.x, i = worklist_prob(wl, (unsigned)b), b0 = wl.start[i];
	const ResP p = params[i];
	body_cg_resident<NT, V, MULTI>(p, b - b0, wl.start[i + 1] - b0);
}

static __global__ void k_words_clear(unsigned long long* p, long long n) {
	for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
		p[i] = 0;
}

struct ResKind {
	int nt, v;  // threads, cells per thread
	bool multi;
};
constexpr ResKind kResKind[kResKinds] = {{512, 4, false}, {512, 8, false}, {1024, 8, false},
                                         {1024, 2, true}, {1024, 4, true}, {1024, 8, true}};
// f(kind as a constant)
template <typename F>
static void with_kind(int kind, F&& f) {
	switch (kind) {
	case 0: f(std::integral_constant<int, 0>{}); break;
	case 1: f(std::integral_constant<int, 1>{}); break;
	case 2: f(std::integral_constant<int, 2>{}); break;
	case 3: f(std::integral_constant<int, 3>{}); break;
	case 4: f(std::integral_constant<int, 4>{}); break;
	default: f(std::integral_constant<int, 5>{}); break;
	}
}

ResPlan cg_resident_plan(const Dims& d) {
	ResPlan r;
	const long long H = d.is3d ? d.sz : (long long)d.nx;
	auto fits = [&](long long c) { return (c + 2 * H) * (long long)sizeof(float) <= kMaxLds; };
	// One workgroup up to 8192 cells, where a second one costs more in waits
	// than it saves in arithmetic (64^2: 2.1 us an iteration, 3.9 with two;
	// 90^2: 3.0 against 4.0), of as few threads as hold the grid at up to 8
	// cells each.  Beyond, runs of as few cells as the workgroup limit allows:
	// an iteration then is the two exchanges (4.2 us at 128^2, 4.6 at 353x241
	// with 2048 cells a workgroup, 4.9 with 4096, 6.1 with 8192).  Where a plane
	// or a row is half a run and more, the words of the runs' ends add to it, and
	// it still takes less than the general kernels' four launches, a whole solve
	// per iteration: 48^3 7.4 us against 15.4, 64^3 9.8 / 15.4, 75x75x46 11.5 /
	// 15.3, 60x59x146 12.4 / 16.2, 3500x140 10.8 / 16.3.
	for (int kind = 0; kind < kResKinds; kind++) {
		const ResKind& k = kResKind[kind];
		const long long c = (long long)k.nt * k.v;
		if (!fits(c) || d.n > c * (k.multi ? kResMaxWG : 1)) continue;
		r.kind = kind;
		r.wg = (int)((d.n + c - 1) / c);
		break;
	}
	if (!r.wg) return r;
	r.H = (int)H;
	r.words = r.wg > 1 ? (size_t)d.n : 0;
	return r;
}

unsigned cg_resident_tags(ResWords& w, hipStream_t s, const ResPlan& pl, int maxIter) {
	if (pl.wg < 2) return 1;
	const unsigned need = (unsigned)std::max(maxIter, 0) + 2u;
	// stale words carry tags already used (or anything, in new memory)
	if (w.next == 0 || w.next > std::numeric_limits<unsigned>::max() - need) {
		hipLaunchKernelGGL(k_words_clear, dim3(flat_blocks((long long)w.count)), dim3(256), 0, s, w.words,
		                   (long long)w.count);
		w.next = 1;
	}
	const unsigned e = w.next;
	w.next += need;
	return e;
}

static size_t lds_bytes(const ResPlan& pl) {
	const ResKind& k = kResKind[pl.kind];
	return ((size_t)k.nt * k.v + 2 * (size_t)pl.H) * sizeof(float);
}

// Solves of several workgroups in flight on one device: a lane holds one at a
// time, or a batch all of them.  A solve takes the lane its stream used last,
// else the one unused for longest, and its stream waits (on the device) for
// the solve that was queued in it before; which lane it gets changes no
// result.
struct ResLane {
	hipEvent_t ev = nullptr;  // end of the lane's last solve
	hipStream_t last = nullptr;
	unsigned long long used = 0;
};
struct ResDevice {
	int cus = -1;  // compute units (-1: not looked up)
	std::vector<ResLane> lane;
	unsigned long long clock = 0;
};
static std::mutex g_res_mu;
static ResDevice g_res_dev[64];
static int g_res_cus = 0;
void cg_resident_cus(int override) {
	std::lock_guard<std::mutex> lk(g_res_mu);
	g_res_cus = override;
}
// compute units of the device (g_res_mu held; 0: not known)
static int units(int device) {
	if (device < 0 || device >= 64) return 0;
	ResDevice& D = g_res_dev[device];
	if (D.cus < 0) {
		// (one workgroup fits a unit: at most 1024 threads by its launch bounds,
		// at most 64 KiB of LDS.  The runtime's occupancy query is not asked: it
		// answers 0 once a second runtime is loaded in the process, as torch's is)
		static_assert(kMaxLds + sizeof(ResShared) + 64 <= 64 * 1024, "LDS of a workgroup");
		int cus = 0;
		MFX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
		D.cus = cus;
	}
	return g_res_cus > 0 ? std::min(g_res_cus, D.cus) : D.cus;
}
bool cg_resident_fits(int device, const ResPlan& pl) {
	if (pl.wg < 2) return pl.wg == 1;
	std::lock_guard<std::mutex> lk(g_res_mu);
	return pl.wg <= units(device);
}
// the device's lanes (g_res_mu held)
static std::vector<ResLane*> lanes(int device) {
	ResDevice& D = g_res_dev[device];
	const size_t n = (size_t)std::max(1, units(device) / kResMaxWG);
	while (D.lane.size() < n) {
		ResLane l;
		MFX_HIP(hipEventCreateWithFlags(&l.ev, hipEventDisableTiming));
		D.lane.push_back(l);
	}
	std::vector<ResLane*> r;
	for (size_t i = 0; i < n; i++) r.push_back(&D.lane[i]);
	return r;
}
static void enter_lane(ResLane* l, hipStream_t s) {
	if (l->last && l->last != s) MFX_HIP(hipStreamWaitEvent(s, l->ev, 0));
}
static void leave_lane(int device, ResLane* l, hipStream_t s) {
	l->last = s;
	l->used = ++g_res_dev[device].clock;
	MFX_HIP(hipEventRecord(l->ev, s));
}
void cg_resident_forget(int device, hipStream_t s) {
	if (device < 0 || device >= 64) return;
	std::lock_guard<std::mutex> lk(g_res_mu);
	for (ResLane& l : g_res_dev[device].lane)
		if (l.last == s) l.last = nullptr;
}

void cg_resident_run(int device, hipStream_t s, const ResPlan& pl, const ResP& p) {
	auto launch = [&]() {
		with_kind(pl.kind, [&](auto k) {
			constexpr ResKind K = kResKind[decltype(k)::value];
			hipLaunchKernelGGL((k_cg_resident<K.nt, K.v, K.multi>), dim3((unsigned)pl.wg), dim3(K.nt), lds_bytes(pl), s, p);
		});
	};
	if (!kResKind[pl.kind].multi) {
		launch();
		return;
	}
	std::lock_guard<std::mutex> lk(g_res_mu);
	ResLane* l = nullptr;
	for (ResLane* c : lanes(device)) {
		if (c->last == s) {
			l = c;
			break;
		}
		if (!l || c->used < l->used) l = c;
	}
	enter_lane(l, s);
	launch();
	leave_lane(device, l, s);
}

// Solves of one workgroup are one launch whatever their number.  Of the
// others as many share a launch as there are units for their workgroups, with
// no other solve in flight (all lanes held).
int cg_resident_run_many(int device, hipStream_t s, int kind, const std::vector<ResPlan>& pl, WorkList items,
                         const ResP* params) {
	size_t lds = 0;
	for (const ResPlan& q : pl)
		if (q.wg) lds = std::max(lds, lds_bytes(q));
	auto launch = [&](int base, int wgs) {
		with_kind(kind, [&](auto k) {
			constexpr ResKind K = kResKind[decltype(k)::value];
			hipLaunchKernelGGL((k_cg_resident_many<K.nt, K.v, K.multi>), dim3((unsigned)wgs), dim3(K.nt), lds, s, items,
			                   params, base);
		});
	};
	int base = 0, wgs = 0, launches = 0;
	if (!kResKind[kind].multi) {
		for (const ResPlan& q : pl) wgs += q.wg;
		if (wgs) launch(0, wgs);
		return wgs ? 1 : 0;
	}
	std::lock_guard<std::mutex> lk(g_res_mu);
	const int most = units(device);
	const std::vector<ResLane*> all = lanes(device);
	for (ResLane* l : all) enter_lane(l, s);
	auto flush = [&]() {
		if (!wgs) return;
		launch(base, wgs);
		launches++;
		base += wgs;
		wgs = 0;
	};
	for (const ResPlan& q : pl) {
		if (wgs + q.wg > most) flush();
		wgs += q.wg;
	}
	flush();
	for (ResLane* l : all) leave_lane(device, l, s);
	return launches;
}

}  // namespace mfx
