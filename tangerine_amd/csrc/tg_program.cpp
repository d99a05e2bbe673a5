#include "tg_program.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace tg {

namespace {

float as_float(uint32_t u)
{
	float f;
	std::memcpy(&f, &u, 4);
	return f;
}

uint32_t as_word(float f)
{
	uint32_t u;
	std::memcpy(&u, &f, 4);
	return u;
}

int brush_param_count(uint32_t op)
{
	switch (op)
	{
	case OP_SPHERE: return 1;
	case OP_TORUS: case OP_CYLINDER: case OP_CONE: return 2;
	case OP_ELLIPSOID: case OP_BOX: case OP_CONINDER: case OP_PLANE: return 3;
	default: return -1;
	}
}

bool is_brush(uint32_t op) { return op >= OP_SPHERE && op <= OP_PLANE; }
bool is_binary(uint32_t op) { return op >= OP_UNION && op <= OP_BLEND_DIFF; }
bool is_blend(uint32_t op) { return op >= OP_BLEND_UNION && op <= OP_BLEND_DIFF; }

// Largest singular value of the 3x3 part of a record's point transform
// (power iteration on M^T M, double precision).
double spectral_norm3(const float* rows)
{
	double a[3][3] = {};
	for (int i = 0; i < 3; ++i)
		for (int j = 0; j < 3; ++j)
			for (int k = 0; k < 3; ++k) a[i][j] += double(rows[k * 4 + i]) * double(rows[k * 4 + j]);
	double v[3] = { 1.0, 0.7548776662, 0.5698402910 };
	double lambda = 0.0;
	for (int it = 0; it < 64; ++it)
	{
		double w[3] = { 0, 0, 0 };
		for (int i = 0; i < 3; ++i)
			for (int j = 0; j < 3; ++j) w[i] += a[i][j] * v[j];
		const double n = std::sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
		if (n == 0.0) return 0.0;
		for (int i = 0; i < 3; ++i) v[i] = w[i] / n;
		lambda = n;
	}
	return std::sqrt(lambda);
}

// Reorders the records (Stop last) so that every set operator evaluates the
// operand that needs the deeper stack first (Sethi-Ullman order), flagging the
// operators whose right operand now runs first (kSwapOperands).  The stack
// then holds at most the tree's Strahler number of values: a chain of any
// length needs 2, and 17 needs a balanced tree of 65,536 brushes.  Values do
// not change: a brush record carries its own point transform, so a subtree
// evaluates to the same bits wherever it runs, and a flagged operator still
// combines (left, right).  Returns the stack high-water mark.
uint32_t reorder_operands(std::vector<Instr>& in)
{
	const size_t n = in.size() - 1;
	std::vector<uint32_t> need(n), first(n), second(n);
	std::vector<uint8_t> swap(n, 0);
	for (size_t i = 0; i < n; ++i)
	{
		const uint32_t op = instr_op(in[i]);
		if (is_brush(op))
			need[i] = 1;
		else if (is_binary(op))
		{
			// roots: the left operand ends right before the right one starts
			const uint32_t a = in[i].w[2] - 1, b = uint32_t(i) - 1;
			swap[i] = need[b] > need[a];
			first[i] = swap[i] ? b : a;
			second[i] = swap[i] ? a : b;
			need[i] = std::max(std::max(need[a], need[b]), std::min(need[a], need[b]) + 1);
		}
		else
		{
			first[i] = uint32_t(i) - 1;  // flate / field scale
			need[i] = need[i - 1];
		}
	}
	// post-order walk from the root (the last record before Stop)
	std::vector<Instr> out;
	out.reserve(in.size());
	std::vector<uint32_t> start(n);  // new index of each subtree's first record
	struct Frame
	{
		uint32_t node, state;
	};
	std::vector<Frame> todo;
	todo.push_back(Frame{ uint32_t(n - 1), 0 });
	while (!todo.empty())
	{
		const uint32_t i = todo.back().node, state = todo.back().state;
		const uint32_t op = instr_op(in[i]);
		if (state == 0) start[i] = uint32_t(out.size());
		const uint32_t arity = is_brush(op) ? 0u : is_binary(op) ? 2u : 1u;
		if (state < arity)
		{
			todo.back().state = state + 1;
			todo.push_back(Frame{ state == 0 ? first[i] : second[i], 0 });
			continue;
		}
		Instr r = in[i];
		if (arity == 2)
		{
			r.w[0] = (r.w[0] & ~kSwapOperands) | (swap[i] ? kSwapOperands : 0u);
			r.w[1] = start[first[i]];
			r.w[2] = start[second[i]];
		}
		out.push_back(r);
		todo.pop_back();
	}
	out.push_back(in[n]);
	in.swap(out);
	return need[n - 1];
}

}  // namespace

constexpr uint32_t kMaxRoundingDepth = 128;

bool DecodedProgram::prunable() const { return lipschitz && rounding_depth <= kMaxRoundingDepth; }

double instr_flops(const Instr& in)
{
	const uint32_t op = instr_op(in);
	double xf = 0.0;
	if (is_brush(op))
	{
		const uint32_t k = instr_kind(in);
		xf = (k == XF_MATRIX) ? 18.0 : (k == XF_OFFSET) ? 3.0 : 0.0;
	}
	switch (op)
	{
	case OP_SPHERE: return xf + 7.0;
	case OP_ELLIPSOID: return xf + 25.0;
	case OP_BOX: return xf + 16.0;
	case OP_TORUS: return xf + 10.0;
	case OP_CYLINDER: return xf + 15.0;
	case OP_PLANE: return xf + 5.0;
	case OP_CONE: return xf + 43.0;
	case OP_CONINDER: return xf + 38.0;
	case OP_UNION: case OP_INTER: case OP_DIFF: return 1.0;
	case OP_BLEND_UNION: case OP_BLEND_INTER: case OP_BLEND_DIFF: return 8.0;
	case OP_FLATE: case OP_SCALE_FIELD: case OP_NEGATE: return 1.0;
	default: return 0.0;
	}
}

// Pruning drops an operand of a set operator when, at a cell centre c, the
// computed operand values a, b satisfy (for union) b - a >= 2 (r' + 1e-5
// (|a| + |b|)), r' = r (1 + 1e-5) + slack, r the cell radius.  Both fields
// are 1-Lipschitz (the decoder checks the transform norm to 1e-5), so their
// exact values move by at most r (1 + 1e-5) inside the cell; the computed
// values differ from the exact ones by the rounding error E(p) of the
// interpreter, which holds at c and at every sample p.  Dropping is exact when
// 2 slack >= E_a(c) + E_a(p) + E_b(c) + E_b(p).  Per brush, the float
// arithmetic (a 3x4 transform in four roundings per component, then at most
// a few dozen operations of the primitive, the divides and square roots
// included) errs by at most K u (|p| + leaf extent) in world units, u =
// 2^-24, with K = 64 taken generously; set operators propagate the larger
// operand error (each is 1-Lipschitz in either operand; min, max and negation
// round nothing, a blend adds u |value|), and flate / field scale add
// u |value|, which the value-proportional 1e-5 term covers for up to 160 such
// roundings on a path (programs with more than 128 are not pruned).  Hence slack = 2 K u (pmax + extent),
// with pmax bounding |p| over the domain; it never goes below 2e-4.  The
// oracle's float64 interpreter measures the per-brush constant on random and
// adversarial trees (tests/test_oracle.py).
float rounding_slack(const DecodedProgram& d, float pmax)
{
	const double u = std::ldexp(1.0, -24), K = 64.0;
	const double s = 2.0 * K * u * (double(std::fabs(pmax)) + double(d.leaf_extent));
	return float(std::max(s, 2.0e-4));
}

PrunePlan prune_plan(const DecodedProgram& d, uint32_t upper_items)
{
	PrunePlan plan;
	const uint32_t n = uint32_t(d.entries.size());
	if (n == 0) return plan;
	auto op_of = [&](uint32_t e) { return (d.entries[e].rec >> 24) & 0x3fu; };
	auto operands = [&](uint32_t e, uint32_t (&c)[2]) -> uint32_t {
		const uint32_t op = op_of(e);
		if (op - OP_SPHERE <= OP_PLANE - OP_SPHERE) return 0;
		c[0] = d.entries[e].l;
		if (op == OP_FLATE || op == OP_SCALE_FIELD) return 1;
		c[1] = d.entries[e].r;
		return 2;
	};
	// Bottom up: an entry whose items (its own, its operands' uncut ones, one
	// for each cut operand) would exceed a treelet cuts the larger operand, then
	// the other.
	std::vector<uint32_t> size(n, 1), stage(n, 0);
	std::vector<uint8_t> cut(n, 0), upper(n, 0);  // upper: its treelet so far has a cut operand
	for (uint32_t e = 0; e < n; ++e)
	{
		uint32_t c[2] = { 0, 0 };
		const uint32_t k = operands(e, c);
		uint32_t total = 1;
		for (uint32_t i = 0; i < k; ++i) total += size[c[i]];
		for (uint32_t i = 0; i < k; ++i) upper[e] |= upper[c[i]] | cut[c[i]];
		for (uint32_t i = 0; i < k && total > (upper[e] ? upper_items : kTreeletItems); ++i)
		{
			uint32_t which = 0;
			if (k == 2 && (cut[c[0]] || (!cut[c[1]] && size[c[1]] > size[c[0]]))) which = 1;
			const uint32_t x = c[which];
			total -= size[x] - 1;
			cut[x] = 1;
			size[x] = 1;
			upper[e] = 1;
		}
		size[e] = total;
		for (uint32_t i = 0; i < k; ++i) stage[e] = std::max(stage[e], stage[c[i]] + (cut[c[i]] ? 1u : 0u));
	}
	cut[n - 1] = 1;
	uint32_t stages = 0;
	for (uint32_t e = 0; e < n; ++e)
		if (cut[e]) stages = std::max(stages, stage[e] + 1);
	// treelet roots by stage; their value slots in that order
	std::vector<uint32_t> slot(n, 0xffffffffu), roots;
	for (uint32_t s = 0; s < stages; ++s)
	{
		plan.stage_first.push_back(uint32_t(roots.size()));
		for (uint32_t e = 0; e < n; ++e)
			if (cut[e] && stage[e] == s) roots.push_back(e);
	}
	plan.stage_first.push_back(uint32_t(roots.size()));
	for (uint32_t e : roots)
		if (e + 1 != n) slot[e] = plan.slots++;
	for (uint32_t root : roots)
	{
		// the root's items top down, then reversed into postfix order by entry
		struct Node
		{
			uint32_t entry, parent, side, depth;  // parent: index into `nodes`
		};
		std::vector<Node> nodes{ { root, 0, 0, 1 } };
		Treelet t{ uint32_t(plan.items.size()), 0, slot[root], 0 };
		for (size_t i = 0; i < nodes.size(); ++i)
		{
			const Node x = nodes[i];
			t.depth = std::max(t.depth, x.depth);
			if (i > 0 && cut[x.entry]) continue;
			uint32_t c[2] = { 0, 0 };
			const uint32_t k = operands(x.entry, c);
			for (uint32_t j = 0; j < k; ++j) nodes.push_back({ c[j], uint32_t(i), j, x.depth + 1 });
		}
		t.count = uint32_t(nodes.size());
		// postfix order is the order of the source entries
		std::vector<uint32_t> order(t.count), at(t.count);
		for (uint32_t i = 0; i < t.count; ++i) order[i] = i;
		std::sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return nodes[a].entry < nodes[b].entry; });
		for (uint32_t i = 0; i < t.count; ++i) at[order[i]] = i;
		for (uint32_t i = 0; i < t.count; ++i)
		{
			const Node& x = nodes[order[i]];
			const bool load = order[i] != 0 && cut[x.entry];
			plan.items.push_back({ load ? kItemLoad : d.entries[x.entry].rec, load ? slot[x.entry] : d.entries[x.entry].ord,
			                       x.entry, at[x.parent] | (x.side << 8) });
		}
		plan.treelets.push_back(t);
	}
	return plan;
}

namespace {

constexpr int kSharePoints = 8;

// Distances of points from a brush, roughly: as a ball of its mean size (a torus: as
// a shell) in its own frame.
void rough_distances(const Instr& in, const float (&p)[3][kSharePoints], float (&d)[kSharePoints])
{
	const float* m = reinterpret_cast<const float*>(in.w) + 1;
	const uint32_t kind = instr_kind(in), op = instr_op(in);
	const float a = m[12], b = m[13], c = m[14];
	float q[3][kSharePoints];
	for (int r = 0; r < 3; ++r)
		for (int s = 0; s < kSharePoints; ++s)
			q[r][s] = kind == XF_MATRIX ? m[4 * r] * p[0][s] + m[4 * r + 1] * p[1][s] + m[4 * r + 2] * p[2][s] + m[4 * r + 3]
			                            : p[r][s] + (kind == XF_OFFSET ? m[4 * r + 3] : 0.0f);
	float shell = 0.0f, radius;
	switch (op)
	{
	case OP_SPHERE: radius = a; break;
	case OP_TORUS: shell = a; radius = b; break;
	case OP_CYLINDER: case OP_CONE: radius = 0.5f * (a + b); break;
	default: radius = (a + b + c) * (1.0f / 3.0f); break;
	}
	for (int s = 0; s < kSharePoints; ++s)
	{
		const float l = std::sqrt(q[0][s] * q[0][s] + q[1][s] * q[1][s] + q[2][s] * q[2][s]);
		d[s] = op == OP_PLANE ? a * q[0][s] + b * q[1][s] + c * q[2][s]
		       : op == OP_TORUS ? std::fabs(l - shell) - radius
		                        : l - radius;
	}
}

}  // namespace

float kept_share(const DecodedProgram& d)
{
	const uint32_t n = uint32_t(d.entries.size());
	if (!d.prunable() || n == 0 || n >= 65535) return 1.0f;
	if (!d.scene_finite) return 0.0f;
	float edge = 0.0f;
	for (int i = 0; i < 3; ++i) edge = std::max(edge, d.scene_hi[i] - d.scene_lo[i]);
	const float two = edge / 24.0f * 1.7320508f;  // twice a cell's radius
	// (an additive sequence of the plastic number's powers: evenly spread)
	const double step[3] = { 0.8191725134, 0.6710436067, 0.5497004779 };
	float p[3][kSharePoints];
	for (int i = 0; i < 3; ++i)
		for (int s = 0; s < kSharePoints; ++s)
		{
			const double t = 0.5 + double(s + 1) * step[i];
			p[i][s] = d.scene_lo[i] + float(t - std::floor(t)) * (d.scene_hi[i] - d.scene_lo[i]);
		}
	// bottom up the values and each operator's points that keep the left and the
	// right operand, then top down the points where an entry is left
	struct Value
	{
		float v[kSharePoints];
	};
	std::vector<Value> value(n);
	std::vector<uint8_t> left(n, 0xff), right(n, 0xff), live(n);
	const uint32_t mask = 0x3fffffu;  // an entry's record
	for (uint32_t e = 0; e < n; ++e)
	{
		const HostEntry& x = d.entries[e];
		const Instr& in = d.instrs[x.rec & mask];
		const uint32_t op = instr_op(in);
		float(&v)[kSharePoints] = value[e].v;
		if (is_brush(op))
		{
			rough_distances(in, p, v);
			continue;
		}
		const float(&vl)[kSharePoints] = value[x.l].v;
		if (!is_binary(op))
		{
			const float by = as_float(in.w[1]);
			for (int s = 0; s < kSharePoints; ++s) v[s] = op == OP_FLATE ? vl[s] - by : vl[s] * by;
			continue;
		}
		// every operator as a maximum: union -max(-l, -r), intersection max(l, r),
		// difference max(l, -r)
		const uint32_t base = is_blend(op) ? op - (OP_BLEND_UNION - OP_UNION) : op;
		const float sl = base == OP_UNION ? -1.0f : 1.0f, sr = base == OP_INTER ? 1.0f : -1.0f;
		const float t = two + (is_blend(op) ? std::max(as_float(in.w[3]), 0.0f) : 0.0f);
		const float(&vr)[kSharePoints] = value[x.r].v;
		uint32_t kl = 0, kr = 0;
		for (int s = 0; s < kSharePoints; ++s)
		{
			const float l = sl * vl[s], r = sr * vr[s];
			kl |= uint32_t(!(r - l >= t)) << s;
			kr |= uint32_t(!(l - r >= t)) << s;
			v[s] = sl * std::max(l, r);
		}
		left[e] = uint8_t(kl);
		right[e] = uint8_t(kr);
	}
	live[n - 1] = 0xff;
	uint64_t kept = 0;
	for (uint32_t e = n; e-- > 0;)
	{
		const HostEntry& x = d.entries[e];
		const uint32_t op = instr_op(d.instrs[x.rec & mask]);
		if (!is_brush(op)) live[x.l] = live[e] & left[e];
		if (is_binary(op)) live[x.r] = live[e] & right[e];
		kept += uint32_t(__builtin_popcount(live[e] & left[e] & right[e]));
	}
	return float(double(kept) / (double(kSharePoints) * double(n)));
}

bool decode_words(const uint32_t* w, size_t n, DecodedProgram& out, std::string& err)
{
	out = DecodedProgram();
	// Pending point transform: the last Offset/Matrix before a brush applies to it
	// (the interpreter overwrites Point from EvalPoint and resets it after each brush).
	uint32_t pending_kind = XF_NONE;
	float pending[12] = { 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0 };
	std::vector<uint32_t> starts;  // subtree start record per stack entry
	double last_brush_norm = 1.0;  // transform norm of the brush just emitted
	double last_brush_extent = 0.0;  // its extent in its own frame (scaled by a following ScaleField)
	double last_centre[3] = { 0, 0, 0 };  // world position of its frame's origin
	double last_radius = 0.0;        // its parameter magnitudes in its own frame
	double widen = 0.0;              // largest blend threshold / flate radius
	bool any_plane = false, any_brush = false;
	double box_lo[3] = { 1e300, 1e300, 1e300 }, box_hi[3] = { -1e300, -1e300, -1e300 };
	auto close_brush = [&](double scale) {
		const double r = last_radius * scale;
		for (int k = 0; k < 3; ++k)
		{
			box_lo[k] = std::min(box_lo[k], last_centre[k] - r);
			box_hi[k] = std::max(box_hi[k], last_centre[k] + r);
		}
		any_brush = true;
	};
	bool brush_open = false;  // a brush whose field scale may still follow
	size_t pc = 0;
	bool stopped = false;
	while (pc < n)
	{
		const uint32_t op = w[pc++];
		if (op != OP_SCALE_FIELD)
		{
			if (last_brush_norm > 1.0 + 1e-5) out.lipschitz = false;
			last_brush_norm = 1.0;
			if (brush_open) close_brush(1.0);
			brush_open = false;
		}
		if (op == OP_STOP)
		{
			if (pc != n)
			{
				err = "Stop is not the last word of the program";
				return false;
			}
			if (starts.size() != 1)
			{
				err = "program leaves " + std::to_string(starts.size()) + " values on the stack (expected 1)";
				return false;
			}
			Instr s{};
			s.w[0] = OP_STOP;
			out.instrs.push_back(s);
			stopped = true;
			break;
		}
		if (is_brush(op))
		{
			const int np = brush_param_count(op);
			if (pc + np > n)
			{
				err = "truncated brush parameters";
				return false;
			}
			Instr b{};
			b.w[0] = op | (pending_kind << 8);
			for (int i = 0; i < 12; ++i) b.w[1 + i] = as_word(pending[i]);
			for (int i = 0; i < np; ++i) b.w[13 + i] = w[pc + i];
			pc += np;
			starts.push_back(uint32_t(out.instrs.size()));
			out.instrs.push_back(b);
			out.brushes++;
			// Pruning relies on every brush being a 1-Lipschitz field: exact
			// distance functions seen through a rigid (rotation + uniform scale,
			// undone by ScaleField) transform.
			if (op == OP_ELLIPSOID) out.lipschitz = false;
			if (op == OP_PLANE)
			{
				const double nx = as_float(b.w[13]), ny = as_float(b.w[14]), nz = as_float(b.w[15]);
				if (std::sqrt(nx * nx + ny * ny + nz * nz) > 1.0 + 1e-5) out.lipschitz = false;
			}
			// checked at the next record, which may be the ScaleField undoing a scale
			last_brush_norm = (pending_kind == XF_MATRIX) ? spectral_norm3(pending) : 1.0;
			{
				double mag = std::sqrt(double(pending[3]) * pending[3] + double(pending[7]) * pending[7] +
				                       double(pending[11]) * pending[11]);
				for (int i = 0; i < np; ++i) mag += std::fabs(double(as_float(w[pc - np + i])));
				if (op == OP_CONE) mag += std::fabs(double(as_float(w[pc - np])) * as_float(w[pc - np + 1]));
				last_brush_extent = mag;
				out.leaf_extent = std::max(out.leaf_extent, float(mag));
				// frame origin in world space: q = A p + b vanishes at p = -A^-1 b
				double radius = 0.0;
				for (int i = 0; i < np; ++i) radius += std::fabs(double(as_float(w[pc - np + i])));
				if (op == OP_CONE) radius += std::fabs(double(as_float(w[pc - np])) * as_float(w[pc - np + 1]));
				last_radius = radius;
				if (op == OP_PLANE) any_plane = true;
				const double b[3] = { pending[3], pending[7], pending[11] };
				if (pending_kind == XF_MATRIX)
				{
					const double A[3][3] = { { pending[0], pending[1], pending[2] }, { pending[4], pending[5], pending[6] },
					                         { pending[8], pending[9], pending[10] } };
					const double det = A[0][0] * (A[1][1] * A[2][2] - A[1][2] * A[2][1]) -
					                   A[0][1] * (A[1][0] * A[2][2] - A[1][2] * A[2][0]) +
					                   A[0][2] * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
					if (std::fabs(det) > 1e-30)
					{
						// Cramer's rule for A c = -b
						for (int k = 0; k < 3; ++k)
						{
							double M[3][3];
							for (int r = 0; r < 3; ++r)
								for (int c = 0; c < 3; ++c) M[r][c] = (c == k) ? -b[r] : A[r][c];
							last_centre[k] = (M[0][0] * (M[1][1] * M[2][2] - M[1][2] * M[2][1]) -
							                  M[0][1] * (M[1][0] * M[2][2] - M[1][2] * M[2][0]) +
							                  M[0][2] * (M[1][0] * M[2][1] - M[1][1] * M[2][0])) / det;
						}
					}
					else
						any_plane = true;  // degenerate frame: no finite placement
				}
				else
					for (int k = 0; k < 3; ++k) last_centre[k] = -b[k];
				brush_open = true;
			}
			out.max_stack = std::max<uint32_t>(out.max_stack, uint32_t(starts.size()));
			pending_kind = XF_NONE;
			const float ident[12] = { 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0 };
			std::memcpy(pending, ident, sizeof(pending));
			continue;
		}
		if (is_binary(op))
		{
			if (starts.size() < 2)
			{
				err = "set operator with fewer than two operands on the stack";
				return false;
			}
			Instr s{};
			s.w[0] = op;
			s.w[2] = starts.back();
			starts.pop_back();
			s.w[1] = starts.back();
			if (is_blend(op))
			{
				if (pc >= n)
				{
					err = "truncated blend threshold";
					return false;
				}
				const float t = as_float(w[pc++]);
				widen = std::max(widen, std::fabs(double(t)));
				s.w[3] = as_word(t);
				s.w[4] = as_word(0.25f / t);
				// exact build: RN(0.25 / t) and 4 t in double, low word first
				const double yq = 0.25 / double(t), t4 = 4.0 * double(t);
				uint64_t b[2];
				std::memcpy(&b[0], &yq, 8);
				std::memcpy(&b[1], &t4, 8);
				s.w[5] = uint32_t(b[0]);
				s.w[6] = uint32_t(b[0] >> 32);
				s.w[7] = uint32_t(b[1]);
				s.w[8] = uint32_t(b[1] >> 32);
			}
			out.instrs.push_back(s);
			out.set_ops++;
			continue;
		}
		if (op == OP_FLATE || op == OP_SCALE_FIELD)
		{
			if (starts.empty())
			{
				err = "unary field operator on an empty stack";
				return false;
			}
			if (pc >= n)
			{
				err = "truncated operand";
				return false;
			}
			Instr u{};
			u.w[0] = op;
			u.w[1] = w[pc++];
			if (op == OP_SCALE_FIELD)
			{
				// field scale s after a transform of norm n: Lipschitz n * |s|
				const double ls = last_brush_norm * std::fabs(double(as_float(u.w[1])));
				if (ls > 1.0 + 1e-5) out.lipschitz = false;
				out.leaf_extent = std::max(out.leaf_extent,
				                           float(last_brush_extent * std::fabs(double(as_float(u.w[1])))));
				if (brush_open) close_brush(std::fabs(double(as_float(u.w[1]))));
				brush_open = false;
				last_brush_norm = 1.0;
			}
			else
				widen = std::max(widen, 2.0 * std::fabs(double(as_float(u.w[1]))));
			out.instrs.push_back(u);
			continue;
		}
		if (op == OP_OFFSET)
		{
			if (pc + 3 > n)
			{
				err = "truncated offset";
				return false;
			}
			const float ident[12] = { 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0 };
			std::memcpy(pending, ident, sizeof(pending));
			pending[3] = as_float(w[pc]);
			pending[7] = as_float(w[pc + 1]);
			pending[11] = as_float(w[pc + 2]);
			pending_kind = XF_OFFSET;
			pc += 3;
			continue;
		}
		if (op == OP_MATRIX)
		{
			if (pc + 16 > n)
			{
				err = "truncated matrix";
				return false;
			}
			// words are column-major c*4 + r; records hold rows (r*4 + c), rows 0..2.
			for (int r = 0; r < 3; ++r)
				for (int c = 0; c < 4; ++c) pending[r * 4 + c] = as_float(w[pc + c * 4 + r]);
			pending_kind = XF_MATRIX;
			pc += 16;
			continue;
		}
		err = "unknown opcode " + std::to_string(op) + " at word " + std::to_string(pc - 1);
		return false;
	}
	if (!stopped)
	{
		err = "program terminated without a Stop word";
		return false;
	}
	out.scene_finite = any_brush && !any_plane;
	if (out.scene_finite)
		for (int k = 0; k < 3; ++k)
		{
			out.scene_lo[k] = float(box_lo[k] - widen);
			out.scene_hi[k] = float(box_hi[k] + widen);
		}
	if (out.max_stack > uint32_t(kMaxStack)) out.max_stack = reorder_operands(out.instrs);
	if (out.max_stack > uint32_t(kMaxStack))
	{
		err = "program needs " + std::to_string(out.max_stack) + " stack slots in any operand order; the device "
		      "interpreter holds " + std::to_string(kMaxStack);
		return false;
	}
	// Record cost in bits 16..23 of word 0 (device-side work accounting), and
	// the entry view with operand roots for per-cell pruning.
	uint32_t ord = 0;
	std::vector<uint32_t> rdepth(out.instrs.size(), 0);
	for (size_t i = 0; i < out.instrs.size(); ++i)
	{
		Instr& in = out.instrs[i];
		const double c = instr_flops(in);
		out.flops += c;
		in.w[0] = (in.w[0] & (0xffffu | kSwapOperands)) | (uint32_t(c) << 16);
		const uint32_t op = instr_op(in);
		if (op == OP_STOP) break;
		HostEntry e{ uint32_t(i) | (instr_kind(in) << 22) | (op << 24) | (in.w[0] & kSwapOperands), 0, 0, 0 };
		if (is_binary(op))
		{
			// the operand evaluated first ends right before the second one starts
			const uint32_t below = in.w[2] - 1, top = uint32_t(i) - 1;
			const bool swapped = (in.w[0] & kSwapOperands) != 0;
			e.l = swapped ? top : below;
			e.r = swapped ? below : top;
			e.ord = ord++;
			rdepth[i] = std::max(rdepth[e.l], rdepth[e.r]) + (is_blend(op) ? 1u : 0u);
		}
		else if (op == OP_FLATE || op == OP_SCALE_FIELD)
		{
			e.l = uint32_t(i) - 1;
			rdepth[i] = rdepth[e.l] + 1;
		}
		out.rounding_depth = std::max(out.rounding_depth, rdepth[i]);
		out.entries.push_back(e);
	}
	out.binary_entries = ord;
	if (out.instrs.size() >= (1u << 22))
	{
		err = "program exceeds 2^22 records";
		return false;
	}
	return true;
}

}  // namespace tg
