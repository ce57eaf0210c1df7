// One-kernel unpreconditioned CG for small grids (mfx_resident.hip).
#pragma once

#include "mfx_internal.h"
#include "mfx_mg.h"

namespace mfx {

constexpr int kResMaxWG = 64;                             // workgroups of one solve
constexpr size_t kResSlotWords = 2 * (size_t)kResMaxWG * 8;  // exchange words of the reductions

// how a grid is split (V == 0: too large for the one-kernel solve, which takes
// grids of up to 2^19 cells whose rows, in 3D planes, fit beside a run in LDS)
struct ResPlan {
	int V = 0;         // cells per thread
	int NT = 0;        // threads per workgroup
	int wg = 0;        // workgroups
	int H = 0;         // cells a row reaches beyond a run: a row in 2D, a plane in 3D
	size_t words = 0;  // exchange words besides the reductions' (one per cell; 0 for one workgroup)
};
ResPlan cg_resident_plan(const Dims& d);

struct ResP {
	Dims d;
	int H;
	CgState* st;          // acc, maxIter, useL2, relTol set; the rest is written
	const uint8_t* code;
	const float* b;
	float* x;             // the solution (starts at 0 whatever it holds)
	int scaled;           // scaled Laplace matrix, as MatvecP
	float scale;
	unsigned long long* xs;  // reductions' words
	unsigned long long* xr;  // the runs' ends, by cell
	unsigned epoch;          // first tag
	long long limit;         // longest wait (wall clock ticks, 100 MHz)
};
// Queues the solve on a stream of `device` (the current one).  Returns false,
// with nothing queued, where its workgroups do not fit the device together.
bool cg_resident_run(int device, hipStream_t s, const ResPlan& pl, ResP p);
// the stream has drained and goes
void cg_resident_forget(int device, hipStream_t s);
// compute units of the device as the launches count them (testing: override > 0
// replaces the device's own number, 0 restores it)
void cg_resident_cus(int override);

// First tag of a solve of at most maxIter iterations on these exchange words
// (solves that share them run one after another).
unsigned cg_resident_tags(ResWords& w, hipStream_t s, const ResPlan& pl, int maxIter);

}  // namespace mfx
