// Reference ProgramBuffer words -> device instruction records.
#pragma once

#include <cstdint>
#include <string>
#include <vector>

#include "tg_types.h"

namespace tg {

// Entry view of a program (see Entry in tg_kernels.h): rec | kind << 22 | op << 24, l, r, ord.
struct HostEntry
{
	uint32_t rec, l, r, ord;
};

struct DecodedProgram
{
	std::vector<Instr> instrs;   // ends with OP_STOP
	std::vector<HostEntry> entries;  // every record but Stop, in order
	uint32_t binary_entries = 0;
	uint32_t max_stack = 0;      // interpreter stack high-water mark
	uint32_t brushes = 0;
	uint32_t set_ops = 0;
	bool lipschitz = true;       // false if any ellipsoid (not a distance bound)
	// Most blend / flate / field-scale operators on one root-to-brush path:
	// each rounds its value once, and the pruning decisions' value-proportional
	// margin (1e-5 (|a| + |b|), about 167 roundings of 2^-24) covers at most
	// kMaxRoundingDepth of them.
	uint32_t rounding_depth = 0;
	bool prunable() const;       // lipschitz, rounding_depth <= kMaxRoundingDepth
	double flops = 0.0;          // algorithmic FP32 work per evaluation (cost table)
	// Largest world-space size of a brush: its field scale times (|its frame
	// translation| + the sum of its parameter magnitudes); bounds the operand
	// magnitudes a brush's arithmetic sees besides the point itself.
	float leaf_extent = 0.0f;
	// A box holding every brush's surface (each brush as a ball around its
	// frame's origin, radius = field scale x the sum of its parameter
	// magnitudes), widened by the largest blend threshold and flate radius;
	// scene_finite is false with a plane.  Only a placement hint (the tracer's
	// cell domain), never a bound the evaluation relies on.
	float scene_lo[3] = { 0, 0, 0 }, scene_hi[3] = { 0, 0, 0 };
	bool scene_finite = false;
};

// A program cut into treelets for the grid-wide pruning passes: subtrees of at
// most kTreeletItems items, each run by one wave per group of cells.  An item
// is an entry of the treelet, or stands for a smaller treelet's root (a cut).
// Treelets are ordered by stage; a treelet's cuts belong to earlier stages.
constexpr uint32_t kTreeletItems = 32;
// Of a program split over a workgroup, treelets above others: where a cut subtree
// occurs only this many.  The widest stage is the first; those above it leave waves
// idle, so they are cut finer: a stage of 7 items costs less than one wave running
// 31.  (One point / 50k rays, us, one scene each, before a treelet's items were read in
// one load, 32 items everywhere / 8 above: 256 primitives 32 /
// 30, 4117 / 3707; 120, 36 / 28, 2859 / 2184; 300, 52 / 33, 5757 / 3777; 2000, 122 /
// 115, 25460 / 24118; 4 and 16 within 2% of 8.)
constexpr uint32_t kSplitUpperItems = 8;
constexpr uint32_t kItemLoad = 33u << 24;  // op of a cut item: the root's value is loaded

struct TreeletItem
{
	uint32_t rec;     // the entry's word, or kItemLoad
	uint32_t index;   // binary entry: its ordinal; cut: the value slot of its treelet
	uint32_t entry;   // source entry (cut: its treelet's root entry)
	uint32_t parent;  // position of the parent's item in the treelet (root: itself) | 1 << 8 for a right operand
};

struct Treelet
{
	uint32_t first, count;  // its items, in postfix order
	uint32_t slot;          // value slot of its root (~0: the program's root)
	uint32_t depth;         // items on the longest path to its root
};

struct PrunePlan
{
	std::vector<TreeletItem> items;
	std::vector<Treelet> treelets;      // by stage
	std::vector<uint32_t> stage_first;  // first treelet of every stage, then their number
	uint32_t slots = 0;                 // value slots
	uint32_t stages() const { return stage_first.empty() ? 0u : uint32_t(stage_first.size()) - 1; }
};

// upper_items: the most in a treelet with a cut.
PrunePlan prune_plan(const DecodedProgram& d, uint32_t upper_items = kTreeletItems);

// Share of the entries that a cell's program keeps, over cells of a 24th of the scene's
// longest edge: an estimate, by the pruning's rules at a few cells with rough brushes
// (random trees of 16 to 2048 primitives 0.03 to 0.09; the same with every operator a
// blend of 0.5 units 0.15 to 0.3, of 1 unit 0.35 to 0.45, of 2 units 0.65 to 0.8, of 4
// units 0.94 to 1).  1 for programs that are never pruned, 0 (unknown) where the scene
// has no box.  It chooses routes; no value depends on it.
float kept_share(const DecodedProgram& d);

// Validates stack discipline and opcodes the way SDFInterpreter::Eval would
// (tangerine/sdf_evaluator.cpp:1397-1600) and re-encodes the program.
// Returns false with a message on malformed input.
bool decode_words(const uint32_t* words, size_t count, DecodedProgram& out, std::string& error);

// Absolute rounding slack of the pruning decisions and the brick certificate
// for points p with |p| <= pmax (see the definition in tg_program.cpp).
float rounding_slack(const DecodedProgram& d, float pmax);

// Algorithmic cost of one evaluation of a record (adds, muls, min/max and
// selects count 1, an FMA 2, sqrt and divide 1 each).  Fixed table.
double instr_flops(const Instr& in);

}  // namespace tg
