// batch.hpp -- device work lists shared by the batched solver and the server.
#pragma once

#include <string>
#include <vector>

#include "tiles.hpp"

namespace mmspx {

// One member grid: its two state buffers, geometry and folded parameters.
// The source buffer of a launch is buf[(parity + phase) & 1], so members that
// joined at different global steps can share one launch.
struct BMember {
	void* buf[2];
	Geom g;
	ModelParams p;
	int phase;
};

// One unit of work: member m, tile origin (y0, z0) of the last axes, planes [xb, xe).
struct BItem {
	int m, y0, z0, xb, xe;
};

// Strip width and depth of the 2-D kernels, planes per item of the 3-D
// Cahn-Hilliard kernel, and the persistent grid size in workgroups per CU.
struct BatchTile {
	int tz, chunk, chunk3, bpc;
	int cells;   // > 0: 2-D Allen-Cahn by runs of `cells` consecutive nodes, one workgroup each
	int tb = 0;  // > 0: periodic 2-D Allen-Cahn by temporal blocks, up to `tb` steps per pass
	// > 0 (8 or 4): 2-D Allen-Cahn and Cahn-Hilliard by the multi-step wave strips
	// of `lv` levels, `chunk` rows per wave; `edges`: some member is not periodic
	int lv = 0;
	bool edges = false;
	// > 0: 3-D Cahn-Hilliard by the four-level march on y3 x z3 tiles, chunk3 planes
	int y3 = 0, z3 = 0;
};

bool batch_model_ok(int model, const Geom& g, std::string* why);
void member_items(int m, const Geom& g, int model, const BatchTile& t, std::vector<BItem>& out2,
                  std::vector<BItem>& out3);
// Steps one pass over the items of the 2-D (dim 2) or 3-D (dim 3) members takes
// at most.
int batch_steps_per_pass(int model, const BatchTile& t, int dim);
// One pass over the `n` items of the dim-dimensional members: nsteps steps, at
// most batch_steps_per_pass.
int launch_batch_pass(int model, int prec, int fields, const BatchTile& t, const BMember* mem, const BItem* items, int n,
                      int dim, int parity, int cus, hipStream_t st, int64_t* launches, int nsteps);
// The multi-step kernels for these members, where they take all of them: lv,
// edges and chunk for the 2-D ones, y3, z3 and chunk3 for the 3-D ones.
void batch_multi_step_choice(int model, int prec, const Geom* const* g, int count, BatchTile* t);
// kernels_batch_steps.hip
int launch_batch_steps2d(int model, int prec, const BatchTile& t, const BMember* mem, const BItem* items, int n,
                         int parity, hipStream_t st, int nsteps);
int launch_batch_march4(int model, int prec, const BatchTile& t, const BMember* mem, const BItem* items, int n,
                        int parity, hipStream_t st, int nsteps);
int device_cus();
// Reorders a spatially ordered work list so that the persistent launch (item
// p runs on workgroup p mod gridDim, and workgroup ids are dealt round-robin
// over the 8 XCDs) gives each XCD one contiguous run of it: neighbouring
// tiles then share their halo reads in one L2. The multi-step kernels run one
// item per wave or workgroup and deal the runs themselves: their lists keep
// their order.
std::vector<BItem> xcd_order(const std::vector<BItem>& in);

}  // namespace mmspx
