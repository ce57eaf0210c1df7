// One-kernel unpreconditioned CG for small grids (mfx_resident.hip).
#pragma once

#include <vector>

#include "mfx_batch.h"
#include "mfx_internal.h"
#include "mfx_mg.h"

namespace mfx {

constexpr int kResMaxWG = 64;                             // workgroups of one solve
constexpr size_t kResSlotWords = 2 * (size_t)kResMaxWG * 8;  // exchange words of the reductions

// how a grid is split (wg == 0: too large for the one-kernel solve, which takes
// grids of up to 2^19 cells whose rows, in 3D planes, fit beside a run in LDS)
constexpr int kResKinds = 6;
struct ResPlan {
	int kind = 0;      // threads and cells per thread, one workgroup or several
	int wg = 0;        // workgroups
	int H = 0;         // cells a row reaches beyond a run: a row in 2D, a plane in 3D
	size_t words = 0;  // exchange words besides the reductions' (one per cell; 0 for one workgroup)
};
ResPlan cg_resident_plan(const Dims& d);
// there is a plan and the device (the current one) holds its workgroups together
bool cg_resident_fits(int device, const ResPlan& pl);

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
// queues a solve that fits on a stream of the device
void cg_resident_run(int device, hipStream_t s, const ResPlan& pl, const ResP& p);
// Queues solves of one kind that fit, each with its own exchange words: items
// and params on the device, pl the problems' plans (wg 0: not of this kind).
// Returns the number of launches.
int cg_resident_run_many(int device, hipStream_t s, int kind, const std::vector<ResPlan>& pl, WorkList items,
                         const ResP* params);
// the stream has drained and goes
void cg_resident_forget(int device, hipStream_t s);
// compute units of the device as the launches count them (testing: override > 0
// replaces the device's own number, 0 restores it)
void cg_resident_cus(int override);

// First tag of a solve of at most maxIter iterations on these exchange words
// (solves that share them run one after another).
unsigned cg_resident_tags(ResWords& w, hipStream_t s, const ResPlan& pl, int maxIter);

}  // namespace mfx
