// Host driver of the level-1 cell pruning shared by grid export and tracing.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/tangerine_gpu.h"
#include "tg_capi_internal.h"
#include "tg_kernels.h"

#define TG_CHECK_HIP(expr, what)                         \
	do                                                   \
	{                                                    \
		hipError_t _e = (expr);                          \
		if (_e != hipSuccess) return hip_fail(_e, what); \
	} while (0)

namespace tg {

namespace {

// More stages than this (a chain of thousands of operators), or values beyond
// this: the in-kernel decision pass, one wave walking the program per group.
constexpr uint32_t kMaxStages = 32;
constexpr uint64_t kMaxValueBytes = 2ull << 30;

}  // namespace

// Grids of at most this many cells (twice as many for programs of 1024
// entries or more) emit a wave per cell (PruneArgs::columns).
constexpr uint64_t kColumnCells = 8192;

namespace {

// Zeroed before a program's passes, read after them.
struct PruneBuffers
{
	unsigned long long* counters;  // 8 words
	uint32_t* lens;                // null: no treelet passes
	uint64_t nlens;
	unsigned long long* host;      // pinned: the first five counters
};

constexpr uint32_t kResetBlocks = 8;  // workgroups to a program

// Kernels, not memsets and copies: a batch's programs take one launch each way
// (24 programs: 48 memsets and 24 copies, 0.3 ms as the host issues them).
__global__ void __launch_bounds__(256) k_prune_reset(const PruneBuffers* __restrict__ jobs, PruneBuffers one)
{
	const PruneBuffers b = jobs ? jobs[blockIdx.x / kResetBlocks] : one;
	const uint32_t part = blockIdx.x % kResetBlocks;
	if (part == 0 && threadIdx.x < 8) b.counters[threadIdx.x] = 0;
	if (!b.lens) return;
	for (uint64_t k = part * 256 + threadIdx.x; k < b.nlens; k += kResetBlocks * 256) b.lens[k] = 0;
}

__global__ void __launch_bounds__(64) k_prune_counts(const PruneBuffers* __restrict__ jobs, PruneBuffers one)
{
	const PruneBuffers b = jobs ? jobs[blockIdx.x] : one;
	if (threadIdx.x < 5) b.host[threadIdx.x] = b.counters[threadIdx.x];
}

PruneBuffers prune_buffers(const CellPrograms& out)
{
	const PruneState& ps = out.state;
	return PruneBuffers{ out.counters.as<unsigned long long>(), ps.treelets ? out.lens.as<uint32_t>() : nullptr,
		ps.waves * 64, out.host };
}

// Bytes of a pool entry.
size_t entry_bytes(const PruneState& ps) { return ps.words ? sizeof(uint32_t) : sizeof(Entry); }

// Emission arguments of a prepared pruning (pool capacity: state.capacity).
PruneArgs prune_args(const tg_program* p, const float origin[3], const float cell[3], const uint32_t counts[3],
	const CellPrograms& out)
{
	const DecodedProgram& d = p->decoded;
	const PruneState& ps = out.state;
	PruneArgs pa{};
	pa.prog = static_cast<const Instr*>(p->device.ptr);
	pa.entries = p->entries.as<const Entry>();
	pa.n_entries = uint32_t(d.entries.size());
	pa.n_binary = d.binary_entries;
	pa.ox = origin[0]; pa.oy = origin[1]; pa.oz = origin[2];
	pa.cx = cell[0]; pa.cy = cell[1]; pa.cz = cell[2];
	pa.radius = ps.decide_radius;
	pa.nx = counts[0]; pa.ny = counts[1]; pa.nz = counts[2];
	pa.slots = std::max<uint32_t>(1, d.max_stack - 1);
	pa.whole_flops = uint32_t(d.flops);
	pa.pool = out.pool.as<Entry>();
	pa.capacity = ps.capacity;
	pa.desc = out.desc.as<BlockDesc>();
	pa.counters = out.counters.as<unsigned long long>();
	pa.scratch = out.scratch.as<uint64_t>();
	pa.cells_per_wave = ps.cells_per_wave;
	// masks, liveness and lengths stay in scratch for the rerun after a pool overflow
	pa.masks_ready = ps.treelets ? 1 : 0;
	pa.counts = out.lens.as<const uint32_t>();
	// the walk: four waves per cell group while that leaves under ~4 waves per
	// SIMD (562 groups of 4095 entries: 395 us, one wave each 504; 1728 groups
	// of 511 entries: 188 us, one wave each 85)
	pa.splits = (ps.treelets && ps.waves * 4 <= 4096) ? 4u : 1u;
	// A wave per cell (a lane per entry) scans the whole program for every
	// cell: it wins on grids of few cells, whose programs are long (the walk's
	// time is the longest walk), and loses on many cells with short programs
	// (4913 cells of 4095 entries 0.10 ms against the walk's 0.69, 35,937 cells
	// of the same 0.39 against 0.41, 266,240 of 511 0.57 against 0.21).
	const bool few = ps.ncells <= kColumnCells || (ps.ncells <= 2 * kColumnCells && d.entries.size() >= 1024);
	pa.columns = (ps.treelets && (ps.words || out.emission == 2 || (out.emission == 0 && few))) ? 1 : 0;
	pa.words = ps.words ? 1 : 0;
	// One pool reservation (a device-wide atomic) for each workgroup's cells:
	// large workgroups, and several cells to a wave once the waves fill the GPU
	// anyway (30k tiles of a 31-entry program: 537 us with 4 cells to a
	// workgroup).  Whole entries: each wave has a position table in LDS (12
	// bytes per 64 entries of the program).
	pa.emit_waves = pa.words || d.entries.size() <= 8192 ? kEmitWaves : 4u;
	pa.emit_cells = ps.ncells >= 4 * 8192 ? 4u : ps.ncells >= 8192 ? 2u : 1u;
	return pa;
}

// Treelet pass arguments (without the stage) of a prepared pruning.
TreeletArgs treelet_args(const tg_program* p, const PruneArgs& pa, const CellPrograms& out)
{
	const PruneState& ps = out.state;
	TreeletArgs ta{};
	ta.prog = pa.prog;
	ta.items = p->items();
	ta.treelets = p->treelets();
	ta.ngroups = uint32_t(ps.waves);
	ta.cells_per_wave = ps.cells_per_wave;
	ta.ox = pa.ox; ta.oy = pa.oy; ta.oz = pa.oz;
	ta.cx = pa.cx; ta.cy = pa.cy; ta.cz = pa.cz;
	ta.radius = ps.decide_radius;
	ta.nx = pa.nx; ta.ny = pa.ny; ta.nz = pa.nz;
	ta.values = out.values.as<float>();
	ta.scratch = pa.scratch;
	ta.n_binary = pa.n_binary;
	ta.n_entries = pa.n_entries;
	ta.slots = pa.slots;
	ta.counts = out.lens.as<uint32_t>();
	return ta;
}

// Launches of the treelet passes: the stages upward, the last of them (the
// root's) in both directions, then the others downward.
size_t treelet_steps(const tg_program* p) { return 2 * size_t(p->plan.stages()) - 1; }

void treelet_step(TreeletArgs& ta, const PrunePlan& plan, size_t step)
{
	const size_t stages = plan.stages();
	const size_t k = step < stages ? step : 2 * stages - 2 - step;
	ta.first = plan.stage_first[k];
	ta.count = plan.stage_first[k + 1] - ta.first;
	ta.up = step < stages ? 1 : 0;
	ta.down = step + 1 >= stages ? 1 : 0;
}

// One emission pass (and, on the first, the treelet passes)
// with the pool capacity out.state.capacity; the five counters are written to
// out.host (pinned) on `stream`.
int prune_pass(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3],
	const uint32_t counts[3], bool fast, CellPrograms& out, bool first)
{
	PruneState& ps = out.state;
	int rc = out.pool.ensure(ps.capacity * entry_bytes(ps));
	if (rc) return rc;
	PruneBuffers buf = prune_buffers(out);
	if (!first) buf.lens = nullptr;
	hipLaunchKernelGGL(k_prune_reset, dim3(buf.lens ? kResetBlocks : 1u), dim3(256), 0, stream, nullptr, buf);
	hipError_t e = hipGetLastError();
	if (e != hipSuccess) return hip_fail(e, "prune reset");
	const PruneArgs pa = prune_args(p, origin, cell, counts, out);
	if (first && ps.treelets)
	{
		TreeletArgs ta = treelet_args(p, pa, out);
		for (size_t step = 0; step < treelet_steps(p); ++step)
		{
			treelet_step(ta, p->plan, step);
			e = fast ? fast::launch_prune_treelets(ta, stream) : exact::launch_prune_treelets(ta, stream);
			if (e != hipSuccess) return hip_fail(e, "treelet pruning launch");
		}
	}
	e = fast ? fast::launch_prune_cells(pa, stream) : exact::launch_prune_cells(pa, stream);
	if (e != hipSuccess) return hip_fail(e, "cell pruning launch");
	hipLaunchKernelGGL(k_prune_counts, dim3(1), dim3(64), 0, stream, nullptr, buf);
	e = hipGetLastError();
	if (e != hipSuccess) return hip_fail(e, "cell pruning counters");
	return TG_OK;
}

}  // namespace

namespace {

// Everything of prune_cells_start before the passes: sizes and buffers.  *ready is false when the program is not
// pruned here.
int prune_prepare(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3],
	float radius, const uint32_t counts[3], CellPrograms& out, bool words, uint32_t room, bool* ready)
{
	const DecodedProgram& d = p->decoded;
	*ready = false;
	out.valid = false;
	out.state.pending = false;
	if (!d.prunable() || d.entries.empty() || d.entries.size() >= 65535) return TG_OK;

	const uint64_t ncells = uint64_t(counts[0]) * counts[1] * counts[2];
	if (ncells == 0 || ncells >= (1ull << 31)) return TG_OK;
	if (!out.host)
	{
		hipError_t e = hipHostMalloc(&out.host, 64, hipHostMallocDefault);
		if (e != hipSuccess)
		{
			out.host = nullptr;
			return hip_fail(e, "pinned pruning counters");
		}
	}
	PruneState& ps = out.state;
	ps.words = words;
	ps.ncells = ncells;
	// decision radius: the cell radius with the Lipschitz tolerance and the
	// rounding slack for points of the cells' box
	float pmax = 0.0f;
	for (int i = 0; i < 3; ++i)
	{
		const float a = std::fabs(origin[i]), b = std::fabs(origin[i] + float(counts[i]) * cell[i]);
		pmax += std::max(a, b) * std::max(a, b);
	}
	ps.decide_radius = radius * (1.0f + 1.0e-5f) + rounding_slack(d, std::sqrt(pmax));
	// Fewer cells per wave only when there are very few cells (every wave
	// gathers the whole program, so smaller groups cost L2 traffic).
	uint32_t cpw = 64;
	while (!words && cpw > 16 && (ncells + cpw - 1) / cpw < 256) cpw >>= 1;
	ps.cells_per_wave = cpw;
	ps.waves = (ncells + cpw - 1) / cpw;
	int rc = out.desc.ensure(ncells * sizeof(BlockDesc));
	if (!rc) rc = out.counters.ensure(64);
	if (!rc) rc = out.scratch.ensure(ps.waves * prune_scratch_words(d.binary_entries, uint32_t(d.entries.size())) * 8);
	if (rc) return rc;
	// Grid-wide treelet passes when the stages are few and the treelets' values
	// fit: they replace the per-wave walk over the whole program.
	ps.treelets = treelet_prunable(p, ncells);
	if (words && !ps.treelets) return TG_OK;
	if (ps.treelets)
	{
		rc = out.values.ensure(std::max<uint64_t>(uint64_t(p->plan.slots) * ps.waves * 64 * 4, 256));
		if (!rc) rc = out.lens.ensure(ps.waves * 64 * 4);
		if (rc) return rc;
	}
	// First guess: a quarter of the whole program per cell, at most 1 GiB; grown
	// to the exact total and rerun if any cell did not fit (prune_cells_finish).
	// (tile programs are short: at most 64 entries each at first)
	size_t per_cell = std::max<size_t>(d.entries.size() / 4, 16);
	if (words) per_cell = std::min<size_t>(per_cell, 64);
	if (room) per_cell = room;
	ps.capacity = std::max<uint64_t>(out.pool.bytes / entry_bytes(ps),
		std::min<uint64_t>(ncells * per_cell, (1ull << 30) / entry_bytes(ps)));
	*ready = true;
	return TG_OK;
}

}  // namespace

bool treelet_prunable(const tg_program* p, uint64_t ncells)
{
	const DecodedProgram& d = p->decoded;
	if (!d.prunable() || d.entries.empty() || d.entries.size() >= 65535 || ncells == 0 || ncells >= (1ull << 31)) return false;
	// (16 cells to a group at the least)
	return p->plan.stages() <= kMaxStages && uint64_t(p->plan.slots) * ((ncells + 15) / 16) * 256 <= kMaxValueBytes;
}

uint64_t tile_program_bytes(const tg_program* p, uint64_t ncells)
{
	const DecodedProgram& d = p->decoded;
	const uint64_t waves = (ncells + 63) / 64, entries = d.entries.size();
	const uint64_t scratch = waves * prune_scratch_words(d.binary_entries, uint32_t(entries)) * 8;
	const uint64_t values = uint64_t(p->plan.slots) * waves * 256;
	// the pool: its first guess, or what the tiles keep if that is more
	const uint64_t kept = std::max(std::min<uint64_t>(std::max<uint64_t>(entries / 4, 16), 64), uint64_t(double(p->kept) * double(entries)));
	return scratch + values + waves * 256 + ncells * (sizeof(BlockDesc) + 4 * kept);
}

int prune_cells_start(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3],
	float radius, const uint32_t counts[3], bool fast, CellPrograms& out, bool words)
{
	bool ready = false;
	int rc = prune_prepare(stream, p, origin, cell, radius, counts, out, words, 0, &ready);
	if (rc || !ready) return rc;
	rc = prune_pass(stream, p, origin, cell, counts, fast, out, true);
	if (rc) return rc;
	out.state.pending = true;
	return TG_OK;
}

int prune_cells_many(hipStream_t stream, const tg_program* const* progs, const CellGrid* grids, uint32_t n, bool fast,
	CellPrograms* const* outs, PruneLaunches& work)
{
	std::vector<uint8_t> ready(n, 0);
	std::vector<PruneArgs> pas(n);
	std::vector<PruneBuffers> buffers;
	size_t steps = 0;
	for (uint32_t i = 0; i < n; ++i)
	{
		bool r = false;
		int rc = prune_prepare(stream, progs[i], grids[i].origin, grids[i].cell, grids[i].radius, grids[i].counts,
			*outs[i], grids[i].words, grids[i].room, &r);
		if (rc) return rc;
		if (!r && grids[i].words) return fail(TG_ERR_LIMIT, "tile programs need the treelet passes");
		if (!r) continue;
		CellPrograms& out = *outs[i];
		ready[i] = 1;
		rc = out.pool.ensure(out.state.capacity * entry_bytes(out.state));
		if (rc) return rc;
		buffers.push_back(prune_buffers(out));
		if (out.state.treelets) steps = std::max(steps, treelet_steps(progs[i]));
		pas[i] = prune_args(progs[i], grids[i].origin, grids[i].cell, grids[i].counts, out);
	}
	// host blob: the buffers to reset; per step, its treelet jobs then their wave
	// bases; then the emission jobs and their block bases
	std::vector<uint8_t>& blob = work.host;
	blob.clear();
	auto put = [&](const void* src, size_t bytes) {
		const size_t at = blob.size();
		blob.resize(at + ((bytes + 15) & ~size_t(15)));
		std::memcpy(blob.data() + at, src, bytes);
		return at;
	};
	const size_t buf_at = put(buffers.data(), buffers.size() * sizeof(PruneBuffers));
	struct Launch
	{
		size_t jobs, bases;
		uint32_t njobs, units;
	};
	struct StageLaunch
	{
		Launch l;
		uint32_t slots;  // most spill slots of a job that runs upward
	};
	std::vector<StageLaunch> stage_launches;
	for (size_t step = 0; step < steps; ++step)
	{
		std::vector<TreeletArgs> jobs;
		std::vector<uint32_t> base;
		uint32_t waves = 0, slots = 0;
		for (uint32_t i = 0; i < n; ++i)
		{
			const CellPrograms& out = *outs[i];
			if (!ready[i] || !out.state.treelets || step >= treelet_steps(progs[i])) continue;
			TreeletArgs ta = treelet_args(progs[i], pas[i], out);
			treelet_step(ta, progs[i]->plan, step);
			base.push_back(waves);
			waves += fast ? fast::treelet_waves(ta) : exact::treelet_waves(ta);
			if (ta.up) slots = std::max(slots, ta.slots);
			jobs.push_back(ta);
		}
		if (jobs.empty()) continue;
		const size_t j = put(jobs.data(), jobs.size() * sizeof(TreeletArgs));
		const size_t b = put(base.data(), base.size() * 4);
		stage_launches.push_back(StageLaunch{ Launch{ j, b, uint32_t(jobs.size()), waves }, slots });
	}
	// emission jobs: the sequential walk's (a wave per group part) and the
	// column emission's (a wave per cell), one launch each; `cells`: the
	// latter's workgroups
	std::vector<PruneArgs> ejobs, cjobs;
	std::vector<uint32_t> ebase, cbase;
	uint32_t blocks = 0, max_slots = 1, cells = 0, max_waves = 1;
	size_t max_lds = 0;
	for (uint32_t i = 0; i < n; ++i)
	{
		if (!ready[i]) continue;
		const PruneArgs& pa = pas[i];
		const uint32_t ncells = pa.nx * pa.ny * pa.nz;
		if (pa.masks_ready && pa.columns)
		{
			cbase.push_back(cells);
			cells += prune_column_blocks(pa);
			max_waves = std::max(max_waves, pa.emit_waves);
			// (of one job: a long program takes few waves, and its table is not every job's)
			max_lds = std::max(max_lds, column_lds_bytes(pa));
			cjobs.push_back(pa);
			continue;
		}
		const uint32_t splits = pa.masks_ready ? pa.splits : 1u;
		ebase.push_back(blocks);
		blocks += (ncells + pa.cells_per_wave - 1) / pa.cells_per_wave * splits;
		max_slots = std::max(max_slots, pa.slots);
		ejobs.push_back(pa);
	}
	size_t ej = 0, eb = 0, cj = 0, cb = 0;
	if (!ejobs.empty())
	{
		ej = put(ejobs.data(), ejobs.size() * sizeof(PruneArgs));
		eb = put(ebase.data(), ebase.size() * 4);
	}
	if (!cjobs.empty())
	{
		cj = put(cjobs.data(), cjobs.size() * sizeof(PruneArgs));
		cb = put(cbase.data(), cbase.size() * 4);
	}
	if (!blob.empty())
	{
		int rc = work.dev.ensure(blob.size());
		if (rc) return rc;
		TG_CHECK_HIP(hipMemcpyAsync(work.dev.ptr, blob.data(), blob.size(), hipMemcpyHostToDevice, stream),
			"pruning job upload");
	}
	const uint8_t* dev = work.dev.as<const uint8_t>();
	const PruneBuffers* dev_buffers = reinterpret_cast<const PruneBuffers*>(dev + buf_at);
	const uint32_t nbuf = uint32_t(buffers.size());
	if (nbuf == 0) return TG_OK;
	hipLaunchKernelGGL(k_prune_reset, dim3(nbuf * kResetBlocks), dim3(256), 0, stream, dev_buffers, PruneBuffers{});
	TG_CHECK_HIP(hipGetLastError(), "prune reset");
	for (const StageLaunch& sl : stage_launches)
	{
		const Launch& l = sl.l;
		const TreeletArgs* jobs = reinterpret_cast<const TreeletArgs*>(dev + l.jobs);
		const uint32_t* base = reinterpret_cast<const uint32_t*>(dev + l.bases);
		const hipError_t e =
			fast ? fast::launch_prune_treelets_multi(jobs, base, l.njobs, l.units, sl.slots, stream)
			     : exact::launch_prune_treelets_multi(jobs, base, l.njobs, l.units, sl.slots, stream);
		if (e != hipSuccess) return hip_fail(e, "treelet pruning launch");
	}
	if (!ejobs.empty())
	{
		const PruneArgs* jobs = reinterpret_cast<const PruneArgs*>(dev + ej);
		const uint32_t* base = reinterpret_cast<const uint32_t*>(dev + eb);
		const hipError_t e =
			fast ? fast::launch_prune_cells_multi(jobs, base, uint32_t(ejobs.size()), blocks, max_slots, stream)
			     : exact::launch_prune_cells_multi(jobs, base, uint32_t(ejobs.size()), blocks, max_slots, stream);
		if (e != hipSuccess) return hip_fail(e, "cell pruning launch");
	}
	if (!cjobs.empty())
	{
		const PruneArgs* jobs = reinterpret_cast<const PruneArgs*>(dev + cj);
		const uint32_t* base = reinterpret_cast<const uint32_t*>(dev + cb);
		const hipError_t e =
			fast ? fast::launch_prune_columns_multi(jobs, base, uint32_t(cjobs.size()), cells, max_waves, max_lds, stream)
			     : exact::launch_prune_columns_multi(jobs, base, uint32_t(cjobs.size()), cells, max_waves, max_lds, stream);
		if (e != hipSuccess) return hip_fail(e, "cell pruning launch");
	}
	hipLaunchKernelGGL(k_prune_counts, dim3(nbuf), dim3(64), 0, stream, dev_buffers, PruneBuffers{});
	TG_CHECK_HIP(hipGetLastError(), "cell pruning counters");
	for (uint32_t i = 0; i < n; ++i)
		if (ready[i]) outs[i]->state.pending = true;
	return TG_OK;
}

int prune_cells_finish(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3],
	const uint32_t counts[3], bool fast, CellPrograms& out)
{
	PruneState& ps = out.state;
	if (!ps.pending) return TG_OK;
	ps.pending = false;
	out.reran = false;
	hipError_t e = hipStreamSynchronize(stream);
	if (e != hipSuccess) return hip_fail(e, "cell pruning");
	const unsigned long long* c = out.host;
	if (c[0] > ps.capacity && c[0] * entry_bytes(ps) <= (size_t(8) << 30))
	{
		// some cells did not fit: rerun the emission with the exact total
		out.reran = true;
		ps.capacity = c[0];
		int rc = prune_pass(stream, p, origin, cell, counts, fast, out, false);
		if (rc) return rc;
		e = hipStreamSynchronize(stream);
		if (e != hipSuccess) return hip_fail(e, "cell pruning");
	}
	out.max_stack = uint32_t(c[1]);
	out.max_binary = uint32_t(c[2]);
	out.max_len = uint32_t(c[3]);
	out.whole_cells = c[4];
	out.entries = c[0];
	out.ncells = ps.ncells;
	out.valid = true;
	return TG_OK;
}

int prune_cells(hipStream_t stream, const tg_program* p, const float origin[3], const float cell[3], float radius,
	const uint32_t counts[3], bool fast, CellPrograms& out)
{
	int rc = prune_cells_start(stream, p, origin, cell, radius, counts, fast, out, false);
	if (rc) return rc;
	return prune_cells_finish(stream, p, origin, cell, counts, fast, out);
}

}  // namespace tg
