// Internal pieces shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <string>
#include <vector>

#include "tg_program.h"

namespace tg {

extern thread_local std::string g_last_error;
int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);
int ensure_device();

// Grow-only device allocation.
struct DevBuf
{
	void* ptr = nullptr;
	size_t bytes = 0;
	int ensure(size_t need);
	void release();
	template <typename T> T* as() const { return static_cast<T*>(ptr); }
};

}  // namespace tg

struct tg_program
{
	uint64_t uid = 0;    // unique per uploaded program (caches of derived device data key on it)
	tg::DecodedProgram decoded;
	float kept = 0.0f;   // kept_share
	tg::PrunePlan plan;  // its treelets
	tg::PrunePlan split_plan;  // those of a program split over a workgroup
	tg::DevBuf device;   // Instr records
	tg::DevBuf entries;  // whole program as pruning entries, then each plan's items and treelets
	const tg::TreeletItem* items() const
	{
		return reinterpret_cast<const tg::TreeletItem*>(entries.as<const tg::HostEntry>() + decoded.entries.size());
	}
	const tg::Treelet* treelets() const { return reinterpret_cast<const tg::Treelet*>(items() + plan.items.size()); }
	const tg::TreeletItem* split_items() const { return reinterpret_cast<const tg::TreeletItem*>(treelets() + plan.treelets.size()); }
	const tg::Treelet* split_treelets() const { return reinterpret_cast<const tg::Treelet*>(split_items() + split_plan.items.size()); }
};

namespace tg {
int upload_program(const DecodedProgram& d, tg_program** out);

// Progress of a cell pruning between prune_cells_start and prune_cells_finish.
struct PruneState
{
	bool pending = false;        // a pass was issued; its counters are not read yet
	bool treelets = false;       // grid-wide treelet passes (else one wave walks the program per cell group)
	bool words = false;          // one word per entry (PruneArgs::words)
	uint64_t ncells = 0, waves = 0, capacity = 0;
	uint32_t cells_per_wave = 0;
	float decide_radius = 0.0f;
};

// Level-1 pruned programs of a cell grid (BlockDesc per cell + entry pool).
struct CellPrograms
{
	DevBuf pool, desc, counters, scratch;
	DevBuf values, lens;      // treelet passes: treelet root values per cell, program lengths
	uint64_t ncells = 0;
	uint64_t entries = 0;     // pool entries in use
	uint32_t max_stack = 0;   // over all cells
	uint32_t max_binary = 0;  // most binary entries of a packed cell program
	uint32_t max_len = 0;     // most entries of a packed cell program
	uint64_t whole_cells = 0; // cells left with the whole program (pool overflow)
	bool valid = false;       // false: the program is not prunable here
	bool reran = false;       // the last pruning emitted again after a pool overflow (desc changed)
	int emission = 0;         // after treelet passes: 0 automatic, 1 sequential walk, 2 a wave per cell
	PruneState state;
	unsigned long long* host = nullptr;  // pinned copy of the pass counters
	void release()
	{
		if (host) (void)hipHostFree(host);
		host = nullptr;
		pool.release();
		desc.release();
		counters.release();
		scratch.release();
		values.release();
		lens.release();
	}
};

// With `words` the cells' programs are one word per entry; the result is only
// valid where the treelet passes apply.
int prune_cells(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3], float radius,
	const uint32_t counts[3], bool fast, CellPrograms& out);

struct GradArgs;
struct SplitProgram;
// `p` split over a workgroup; false where it is not (one treelet, too many
// stages, LDS).
bool split_program(const tg_program* p, SplitProgram& out);
// Called when a query's points have to be on the device, if they are not yet.
using PointsReady = std::function<int()>;
// Whether that many gradients are gathered by cell.
bool gathers_gradients(const tg_program* p, uint64_t count);
// The gradients of `a` (prog, slots: p's) on `stream`.
int launch_gradients(const tg_program* p, const GradArgs& a, uint32_t flags, hipStream_t stream, const PointsReady& ready);

// Whether `p` can be pruned over ncells cells by the treelet passes.
bool treelet_prunable(const tg_program* p, uint64_t ncells);

// Device memory of `p` pruned to a word an entry over ncells cells, about.
uint64_t tile_program_bytes(const tg_program* p, uint64_t ncells);

// A cell grid to prune a program over.
struct CellGrid
{
	float origin[3], cell[3], radius;
	uint32_t counts[3];
	bool words = false;
	uint32_t room = 0;  // entries a cell in the pool's first guess (0: a quarter of the program, for words at most 64)
};

// Job tables of prune_cells_many (kept between calls: the upload reads `host`).
struct PruneLaunches
{
	DevBuf dev;
	std::vector<uint8_t> host;
};

// prune_cells_start for n programs on one stream: every program's treelet
// passes of one stage in one launch, then every emission in one launch.  Each is then finished with
// prune_cells_finish on the same stream.
int prune_cells_many(hipStream_t stream, const tg_program* const* progs, const CellGrid* grids, uint32_t n, bool fast,
	CellPrograms* const* outs, PruneLaunches& work);
// The same in two halves: start issues the passes on `stream` without waiting;
// finish waits for the stream, reruns the emission if the pool overflowed and
// fills the counts (same arguments).  Between them the caller may issue other
// work (other trees' pruning on other streams).
int prune_cells_start(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3],
	float radius, const uint32_t counts[3], bool fast, CellPrograms& out, bool words = false);
int prune_cells_finish(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3],
	const uint32_t counts[3], bool fast, CellPrograms& out);
}

namespace tg {

// Buffers of one host query (tg_eval_points, tg_gradient_points, tg_raymarch),
// kept between calls.  A call leases a workspace of its device for its whole
// length, so calls of several threads never share one; the pool keeps at most
// kPoolSpaces idle ones per device, and none larger than kPoolBytes, and gives them
// back where device memory runs out (DevBuf::ensure).
struct Workspace
{
	int device = 0;
	hipEvent_t busy = nullptr;  // the work still reading it, of a call that returned before its end
	bool in_flight = false;
	DevBuf in, out, queue, ctl;
	CellPrograms levels[2];
	PruneLaunches launches;
	std::vector<std::vector<uint8_t>> retired;  // job tables of work that may still read them
	void* pinned = nullptr;   // host staging, also addressed by kernels
	size_t pinned_bytes = 0;
	size_t bytes() const;
	void release();
};

// Frees the current device's idle workspaces; false if there were none.
bool free_idle_workspaces();

class WorkspaceLease
{
public:
	WorkspaceLease() = default;
	~WorkspaceLease();
	WorkspaceLease(const WorkspaceLease&) = delete;
	WorkspaceLease& operator=(const WorkspaceLease&) = delete;
	// A workspace of the current device, for work on `stream`: an idle one whose
	// last work is over, a new one, or one that `stream` is made to wait for.
	int take(hipStream_t stream = nullptr);
	// The work on `stream` so far goes on reading the workspace after the lease.
	int leave_to(hipStream_t stream);
	// Work on the default stream uses the workspace: unless waited() says that it is
	// over, the end of the lease waits for it (a call that fails half way).
	void queued() { queued_ = true; }
	void waited() { queued_ = false; }
	int pinned(size_t bytes);         // its staging, at least this large
	// `count` points for a kernel to read at `xyz` and `width` floats each for it
	// to write at `out`: the pinned staging itself for few points, else device
	// buffers (stage copies the points there, on the default stream).  `gathered`:
	// always device buffers, as the kernels read the points twice and write in any
	// order (100k gradients of 256 primitives 446 us in the staging, 337 so); upload copies the points.
	int stage(const float* host_xyz, uint64_t count, uint32_t width, bool gathered, const float** xyz, float** out);
	int upload(const float* host_xyz, uint64_t count);
	// Waits for the default stream's kernel and copies the staged results out.
	int collect(float* host_out, uint64_t count, uint32_t width);
	Workspace* operator->() const { return ws_; }

private:
	Workspace* ws_ = nullptr;
	bool queued_ = false;
	bool direct_ = false;             // staged in pinned memory
	bool copied_ = false;             // through it, to device buffers and back
};

}  // namespace tg

struct tg_mesher;
struct tg_surrogate;
#include "tg_mlp.h"

namespace tg {
// Device vertices of the mesher's last export (3 floats each).
const float* mesher_vertices(const tg_mesher* m);
mlp::Net surrogate_net(const tg_surrogate* s);
// Cull threshold for bricks of half-diagonal r (< 0: not calibrated); the
// certified threshold may be lower (skipped bricks are checked exactly).
float surrogate_threshold(const tg_surrogate* s, float r, bool certified = false);
}
