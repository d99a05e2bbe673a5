#include <atomic>
// C ABI of the MI355X CSG distance path (declared in include/tangerine_gpu.h).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/tangerine_gpu.h"
#include "tg_capi_internal.h"
#include "tg_kernels.h"
#include "tg_mesh.h"
#include "tg_program.h"
#include "tg_tree.h"

using namespace tg;

// ---------------------------------------------------------------------------
// errors

namespace tg {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg)
{
	g_last_error = msg;
	return code;
}

int hip_fail(hipError_t e, const char* what)
{
	return fail(TG_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

int DevBuf::ensure(size_t need)
{
	if (need <= bytes) return TG_OK;
	if (ptr) hipFree(ptr);
	ptr = nullptr;
	bytes = 0;
	size_t grow = std::max(need, size_t(256));
	hipError_t e = hipMalloc(&ptr, grow);
	if (e != hipSuccess && free_idle_workspaces())
	{
		hipGetLastError();
		e = hipMalloc(&ptr, grow);
	}
	if (e != hipSuccess)
	{
		ptr = nullptr;
		hipGetLastError();
		return fail(TG_ERR_NOMEM, "hipMalloc of " + std::to_string(grow) + " bytes failed: " + hipGetErrorString(e));
	}
	bytes = grow;
	return TG_OK;
}

void DevBuf::release()
{
	if (ptr) hipFree(ptr);
	ptr = nullptr;
	bytes = 0;
}

int ensure_device()
{
	static int ready = -1;
	if (ready == 1) return TG_OK;
	int n = 0;
	hipError_t e = hipGetDeviceCount(&n);
	if (e != hipSuccess || n == 0)
	{
		hipGetLastError();
		return fail(TG_ERR_DEVICE, "no HIP device available");
	}
	ready = 1;
	return TG_OK;
}

namespace {

constexpr size_t kPoolSpaces = 4;
constexpr size_t kPoolBytes = size_t(256) << 20;

std::mutex g_pool_mutex;
std::vector<Workspace*>& pool()
{
	// never destroyed: the device runtime may be gone before static destructors
	static std::vector<Workspace*>* idle = new std::vector<Workspace*>;
	return *idle;
}

}  // namespace

size_t Workspace::bytes() const
{
	size_t n = in.bytes + out.bytes + queue.bytes + ctl.bytes + launches.dev.bytes + pinned_bytes;
	for (const CellPrograms& l : levels)
		n += l.pool.bytes + l.desc.bytes + l.counters.bytes + l.scratch.bytes + l.values.bytes + l.lens.bytes;
	return n;
}

void Workspace::release()
{
	if (in_flight) (void)hipEventSynchronize(busy);
	for (DevBuf* b : { &in, &out, &queue, &ctl }) b->release();
	for (CellPrograms& l : levels) l.release();
	launches.dev.release();
	if (pinned) (void)hipHostFree(pinned);
	pinned = nullptr;
	pinned_bytes = 0;
	if (busy) (void)hipEventDestroy(busy);
	busy = nullptr;
	in_flight = false;
}

bool free_idle_workspaces()
{
	int dev = 0;
	if (hipGetDevice(&dev) != hipSuccess) return false;
	std::vector<Workspace*> out;
	{
		std::lock_guard<std::mutex> lock(g_pool_mutex);
		std::vector<Workspace*>& idle = pool();
		const auto mine = std::stable_partition(idle.begin(), idle.end(), [dev](const Workspace* w) { return w->device != dev; });
		out.assign(mine, idle.end());
		idle.erase(mine, idle.end());
	}
	for (Workspace* w : out)
	{
		w->release();
		delete w;
	}
	return !out.empty();
}

int WorkspaceLease::take(hipStream_t stream)
{
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
	{
		std::lock_guard<std::mutex> lock(g_pool_mutex);
		std::vector<Workspace*>& idle = pool();
		size_t mine = 0, pick = idle.size();
		for (size_t i = 0; i < idle.size(); ++i)
		{
			Workspace* w = idle[i];
			if (w->device != dev) continue;
			++mine;
			if (w->in_flight && hipEventQuery(w->busy) == hipSuccess) w->in_flight = false;
			if (pick == idle.size() || (idle[pick]->in_flight && !w->in_flight)) pick = i;
		}
		(void)hipGetLastError();  // (an event not reached yet is no error)
		if (pick < idle.size() && (!idle[pick]->in_flight || mine >= kPoolSpaces))
		{
			ws_ = idle[pick];
			idle.erase(idle.begin() + std::ptrdiff_t(pick));
		}
	}
	if (ws_)
	{
		if (!ws_->in_flight)
		{
			ws_->retired.clear();
			return TG_OK;
		}
		ws_->retired.push_back(std::move(ws_->launches.host));
		ws_->launches.host = {};
		e = hipStreamWaitEvent(stream, ws_->busy, 0);
		return e == hipSuccess ? TG_OK : hip_fail(e, "workspace wait");
	}
	ws_ = new Workspace;
	ws_->device = dev;
	return TG_OK;
}

int WorkspaceLease::leave_to(hipStream_t stream)
{
	hipError_t e = hipSuccess;
	if (!ws_->busy) e = hipEventCreateWithFlags(&ws_->busy, hipEventDisableTiming);
	if (e == hipSuccess) e = hipEventRecord(ws_->busy, stream);
	if (e == hipSuccess)
	{
		ws_->in_flight = true;
		return TG_OK;
	}
	// no event: nothing may use the workspace before the stream is done
	(void)hipStreamSynchronize(stream);
	ws_->in_flight = false;
	return hip_fail(e, "workspace event");
}

int WorkspaceLease::pinned(size_t bytes)
{
	if (bytes <= ws_->pinned_bytes) return TG_OK;
	if (ws_->pinned) (void)hipHostFree(ws_->pinned);
	ws_->pinned = nullptr;
	ws_->pinned_bytes = 0;
	const size_t room = std::max(bytes, size_t(4096));
	const hipError_t e = hipHostMalloc(&ws_->pinned, room, hipHostMallocDefault);
	if (e != hipSuccess)
	{
		ws_->pinned = nullptr;
		hipGetLastError();
		return fail(TG_ERR_NOMEM, std::string("pinned staging: ") + hipGetErrorString(e));
	}
	ws_->pinned_bytes = room;
	return TG_OK;
}

namespace {

// Queries whose points and results are within this are read and written by the
// kernel in pinned memory, which is faster than a copy each way at every size
// measured (3 primitives, whole call, device buffers / pinned: 1 point 28 / 18 us,
// 4000 52 / 19, 40000 58 / 36, 400000 258 / 238; 100000 gradients of 256 primitives
// 373 / 335).  The bound is for the pinned memory an idle workspace keeps.
constexpr size_t kDirectBytes = size_t(16) << 20;

// Copies n words between device memory and the staging, both 16-byte aligned, on
// the stream itself: a copy engine's transfer between kernels costs two waits for
// another queue (100k gradients of 256 primitives 371 us with them).  Bound by the
// host link.
__global__ void __launch_bounds__(256) k_copy_words(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, uint32_t n)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, quads = n / 4;
	if (i < quads)
		reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
	else if (const uint32_t k = 4 * quads + (i - quads); k < n)
		dst[k] = src[k];
}

__global__ void __launch_bounds__(256) k_zero_words(uint32_t* dst, uint32_t n)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) dst[i] = 0;
}

// (n: at most kDirectBytes of words)
hipError_t copy_words(const void* src, void* dst, uint64_t n)
{
	hipLaunchKernelGGL(k_copy_words, dim3(unsigned((n / 4 + 4 + 255) / 256)), dim3(256), 0, nullptr,
		static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst), uint32_t(n));
	return hipGetLastError();
}

}  // namespace

int WorkspaceLease::stage(const float* host_xyz, uint64_t count, uint32_t width, bool gathered, const float** xyz, float** out)
{
	queued();
	const uint64_t bytes = count * (12 + 4 * width) + 16;
	size_t room = 65536;
	while (room < bytes && room < kDirectBytes) room *= 2;
	const bool held = bytes <= kDirectBytes && pinned(room) == TG_OK;
	direct_ = held && !gathered;
	copied_ = held && gathered;
	if (direct_)
	{
		std::memcpy(ws_->pinned, host_xyz, count * 12);
		*xyz = static_cast<const float*>(ws_->pinned);
		*out = static_cast<float*>(ws_->pinned) + 3 * count;
		return TG_OK;
	}
	int rc = ws_->in.ensure(count * 12);
	if (!rc) rc = ws_->out.ensure(count * 4 * width);
	if (rc) return rc;
	*xyz = ws_->in.as<const float>();
	*out = ws_->out.as<float>();
	return gathered ? TG_OK : upload(host_xyz, count);
}

int WorkspaceLease::upload(const float* host_xyz, uint64_t count)
{
	hipError_t e;
	if (copied_)
	{
		std::memcpy(ws_->pinned, host_xyz, count * 12);
		e = copy_words(ws_->pinned, ws_->in.ptr, 3 * count);
	}
	else
		e = hipMemcpy(ws_->in.ptr, host_xyz, count * 12, hipMemcpyHostToDevice);
	return e == hipSuccess ? TG_OK : hip_fail(e, "points upload");
}

int WorkspaceLease::collect(float* host_out, uint64_t count, uint32_t width)
{
	hipError_t e;
	if (direct_ || copied_)
	{
		float* results = static_cast<float*>(ws_->pinned) + (copied_ ? (3 * count + 3) / 4 * 4 : 3 * count);
		e = copied_ ? copy_words(ws_->out.ptr, results, count * width) : hipSuccess;
		if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
		if (e == hipSuccess) std::memcpy(host_out, results, count * 4 * width);
	}
	else
		e = hipMemcpy(host_out, ws_->out.ptr, count * 4 * width, hipMemcpyDeviceToHost);
	if (e == hipSuccess) waited();
	return e == hipSuccess ? TG_OK : hip_fail(e, "results download");
}

WorkspaceLease::~WorkspaceLease()
{
	if (!ws_) return;
	if (queued_) (void)hipStreamSynchronize(nullptr);
	if (ws_->bytes() <= kPoolBytes)
	{
		std::lock_guard<std::mutex> lock(g_pool_mutex);
		std::vector<Workspace*>& idle = pool();
		size_t mine = 0;
		for (const Workspace* w : idle) mine += w->device == ws_->device ? 1 : 0;
		if (mine < kPoolSpaces)
		{
			idle.push_back(ws_);
			return;
		}
	}
	ws_->release();
	delete ws_;
}

}  // namespace tg

struct tg_node
{
	NodeRef ref;
};

#define TG_CHECK_HIP(expr, what)                 \
	do                                           \
	{                                            \
		hipError_t _e = (expr);                  \
		if (_e != hipSuccess) return hip_fail(_e, what); \
	} while (0)

extern "C" const char* tg_last_error(void) { return g_last_error.c_str(); }

extern "C" int tg_device_init(int device)
{
	int rc = ensure_device();
	if (rc) return rc;
	TG_CHECK_HIP(hipSetDevice(device), "hipSetDevice");
	return TG_OK;
}

extern "C" int tg_device_synchronize(void)
{
	TG_CHECK_HIP(hipDeviceSynchronize(), "hipDeviceSynchronize");
	return TG_OK;
}

// Plain streaming copy, 16 bytes per lane per iteration.
__global__ void __launch_bounds__(256) k_copy_probe(const uint4* __restrict__ src, uint4* __restrict__ dst, uint64_t n)
{
	const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
	for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

extern "C" int tg_device_copy_probe(uint64_t bytes, int repeat, double* ms_per_copy)
{
	int rc = ensure_device();
	if (rc) return rc;
	if (bytes < 16 || repeat < 1) return fail(TG_ERR_INVALID, "tg_device_copy_probe: bytes >= 16, repeat >= 1");
	const uint64_t n = bytes / 16;
	DevBuf a, b;
	rc = a.ensure(n * 16);
	if (!rc) rc = b.ensure(n * 16);
	if (rc)
	{
		a.release();
		return rc;
	}
	hipEvent_t e0, e1;
	hipEventCreate(&e0);
	hipEventCreate(&e1);
	hipMemset(a.ptr, 1, n * 16);
	const unsigned blocks = unsigned(std::min<uint64_t>((n + 255) / 256, 256u * 8u * 8u));
	hipEventRecord(e0, nullptr);
	for (int r = 0; r < repeat; ++r)
		hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, nullptr, a.as<const uint4>(), b.as<uint4>(), n);
	hipEventRecord(e1, nullptr);
	hipError_t e = hipEventSynchronize(e1);
	float ms = 0;
	hipEventElapsedTime(&ms, e0, e1);
	hipEventDestroy(e0);
	hipEventDestroy(e1);
	a.release();
	b.release();
	if (e != hipSuccess) return hip_fail(e, "copy probe");
	if (ms_per_copy) *ms_per_copy = double(ms) / repeat;
	return TG_OK;
}

// ---------------------------------------------------------------------------
// builders

static tg_node* wrap(NodeRef r) { return r ? new tg_node{ std::move(r) } : nullptr; }

static bool finite_all(std::initializer_list<float> v)
{
	for (float f : v)
		if (!std::isfinite(f)) return false;
	return true;
}

static tg_node* bad_arg(const char* what)
{
	g_last_error = what;
	return nullptr;
}

extern "C" tg_node* tg_sphere(float r)
{
	if (!finite_all({ r })) return bad_arg("tg_sphere: non-finite radius");
	return wrap(make_sphere(r));
}
extern "C" tg_node* tg_ellipsoid(float x, float y, float z)
{
	if (!finite_all({ x, y, z })) return bad_arg("tg_ellipsoid: non-finite radius");
	return wrap(make_ellipsoid(x, y, z));
}
extern "C" tg_node* tg_box(float x, float y, float z)
{
	if (!finite_all({ x, y, z })) return bad_arg("tg_box: non-finite extent");
	return wrap(make_box(x, y, z));
}
extern "C" tg_node* tg_torus(float major, float minor)
{
	if (!finite_all({ major, minor })) return bad_arg("tg_torus: non-finite radius");
	return wrap(make_torus(major, minor));
}
extern "C" tg_node* tg_cylinder(float r, float h)
{
	if (!finite_all({ r, h })) return bad_arg("tg_cylinder: non-finite size");
	return wrap(make_cylinder(r, h));
}
extern "C" tg_node* tg_plane(float x, float y, float z)
{
	if (!finite_all({ x, y, z }) || (x == 0.0f && y == 0.0f && z == 0.0f)) return bad_arg("tg_plane: degenerate normal");
	return wrap(make_plane(x, y, z));
}
extern "C" tg_node* tg_cone(float r, float h)
{
	if (!finite_all({ r, h }) || h == 0.0f) return bad_arg("tg_cone: degenerate size");
	return wrap(make_cone(r, h));
}
extern "C" tg_node* tg_coninder(float lo, float hi, float h)
{
	if (!finite_all({ lo, hi, h })) return bad_arg("tg_coninder: non-finite size");
	return wrap(make_coninder(lo, hi, h));
}

static tg_node* set_op(uint32_t op, float t, const tg_node* l, const tg_node* r)
{
	if (!l || !r) return bad_arg("set operator: null operand");
	if (!std::isfinite(t)) return bad_arg("set operator: non-finite threshold");
	return wrap(make_set(op, l->ref, r->ref, t));
}

extern "C" tg_node* tg_union(const tg_node* l, const tg_node* r) { return set_op(OP_UNION, 0.0f, l, r); }
extern "C" tg_node* tg_inter(const tg_node* l, const tg_node* r) { return set_op(OP_INTER, 0.0f, l, r); }
extern "C" tg_node* tg_diff(const tg_node* l, const tg_node* r) { return set_op(OP_DIFF, 0.0f, l, r); }
extern "C" tg_node* tg_blend_union(float t, const tg_node* l, const tg_node* r) { return set_op(OP_BLEND_UNION, t, l, r); }
extern "C" tg_node* tg_blend_inter(float t, const tg_node* l, const tg_node* r) { return set_op(OP_BLEND_INTER, t, l, r); }
extern "C" tg_node* tg_blend_diff(float t, const tg_node* l, const tg_node* r) { return set_op(OP_BLEND_DIFF, t, l, r); }

extern "C" tg_node* tg_flate(const tg_node* n, float radius)
{
	if (!n) return bad_arg("tg_flate: null node");
	return wrap(make_flate(n->ref, radius));
}

extern "C" tg_node* tg_move(const tg_node* n, float x, float y, float z)
{
	if (!n) return bad_arg("tg_move: null node");
	NodeRef c = copy_tree(n->ref);
	move_tree(c.get(), { x, y, z });
	return wrap(c);
}

extern "C" tg_node* tg_rotate(const tg_node* n, float qx, float qy, float qz, float qw)
{
	if (!n) return bad_arg("tg_rotate: null node");
	NodeRef c = copy_tree(n->ref);
	rotate_tree(c.get(), { qw, qx, qy, qz });
	return wrap(c);
}

static tg_node* rotate_axis(const tg_node* n, int axis, float degrees)
{
	if (!n) return bad_arg("tg_rotate_*: null node");
	NodeRef c = copy_tree(n->ref);
	rotate_tree(c.get(), axis_rotation(axis, degrees));
	return wrap(c);
}

extern "C" tg_node* tg_rotate_x(const tg_node* n, float d) { return rotate_axis(n, 0, d); }
extern "C" tg_node* tg_rotate_y(const tg_node* n, float d) { return rotate_axis(n, 1, d); }
extern "C" tg_node* tg_rotate_z(const tg_node* n, float d) { return rotate_axis(n, 2, d); }

extern "C" tg_node* tg_scale(const tg_node* n, float s)
{
	if (!n) return bad_arg("tg_scale: null node");
	NodeRef c = copy_tree(n->ref);
	scale_tree(c.get(), s);
	return wrap(c);
}

extern "C" void tg_node_release(tg_node* n) { delete n; }

extern "C" int tg_node_bounds(const tg_node* n, float* mm)
{
	if (!n || !mm) return fail(TG_ERR_INVALID, "tg_node_bounds: null argument");
	Box3 b = tree_bounds(n->ref.get());
	mm[0] = b.lo.x; mm[1] = b.lo.y; mm[2] = b.lo.z;
	mm[3] = b.hi.x; mm[4] = b.hi.y; mm[5] = b.hi.z;
	return TG_OK;
}

extern "C" int tg_node_has_finite_bounds(const tg_node* n) { return n ? int(tree_has_finite_bounds(n->ref.get())) : 0; }
extern "C" int tg_node_leaf_count(const tg_node* n) { return n ? int(n->ref->leaves) : 0; }
extern "C" int tg_node_stack_size(const tg_node* n) { return n ? int(n->ref->stack_size) : 0; }

extern "C" int tg_node_compile(const tg_node* n, uint32_t* words, uint64_t cap, uint64_t* count)
{
	if (!n || !count) return fail(TG_ERR_INVALID, "tg_node_compile: null argument");
	std::vector<uint32_t> w;
	compile_tree(n->ref.get(), w);
	*count = w.size();
	if (words)
	{
		const uint64_t k = std::min<uint64_t>(cap, w.size());
		std::memcpy(words, w.data(), k * 4);
	}
	return TG_OK;
}

// ---------------------------------------------------------------------------
// programs

int tg::upload_program(const DecodedProgram& d, tg_program** out)
{
	int rc = ensure_device();
	if (rc) return rc;
	static std::atomic<uint64_t> next_uid{ 1 };
	auto p = std::make_unique<tg_program>();
	p->uid = next_uid++;
	p->decoded = d;
	p->kept = kept_share(d);
	p->plan = prune_plan(d);
	p->split_plan = prune_plan(d, kSplitUpperItems);
	static_assert(sizeof(HostEntry) == 16 && sizeof(TreeletItem) == 16 && sizeof(Treelet) == 16, "one array of 16-byte words");
	std::vector<HostEntry> blob(d.entries);
	for (const PrunePlan* plan : { &p->plan, &p->split_plan })
	{
		const size_t items = blob.size(), treelets = items + plan->items.size();
		blob.resize(std::max<size_t>(treelets + plan->treelets.size(), 1));
		if (!plan->items.empty()) std::memcpy(&blob[items], plan->items.data(), plan->items.size() * sizeof(TreeletItem));
		if (!plan->treelets.empty()) std::memcpy(&blob[treelets], plan->treelets.data(), plan->treelets.size() * sizeof(Treelet));
	}
	rc = p->device.ensure(d.instrs.size() * sizeof(Instr));
	if (!rc) rc = p->entries.ensure(blob.size() * sizeof(HostEntry));
	if (rc)
	{
		p->device.release();
		return rc;
	}
	TG_CHECK_HIP(hipMemcpy(p->device.ptr, d.instrs.data(), d.instrs.size() * sizeof(Instr), hipMemcpyHostToDevice),
		"program upload");
	TG_CHECK_HIP(hipMemcpy(p->entries.ptr, blob.data(), blob.size() * sizeof(HostEntry), hipMemcpyHostToDevice),
		"program entries upload");
	*out = p.release();
	return TG_OK;
}

extern "C" int tg_program_from_words(const uint32_t* words, uint64_t count, tg_program** out)
{
	if (!words || !out || count == 0) return fail(TG_ERR_INVALID, "tg_program_from_words: null or empty argument");
	DecodedProgram d;
	std::string err;
	if (!decode_words(words, count, d, err))
	{
		return fail(err.find("stack slots") != std::string::npos ? TG_ERR_LIMIT : TG_ERR_PROGRAM,
			"tg_program_from_words: " + err);
	}
	return upload_program(d, out);
}

extern "C" int tg_program_from_node(const tg_node* n, tg_program** out)
{
	if (!n || !out) return fail(TG_ERR_INVALID, "tg_program_from_node: null argument");
	std::vector<uint32_t> w;
	compile_tree(n->ref.get(), w);
	return tg_program_from_words(w.data(), w.size(), out);
}

static void fill_info(const DecodedProgram& d, tg_program_info* out)
{
	out->instructions = d.instrs.size();
	out->max_stack = d.max_stack;
	out->brushes = d.brushes;
	out->set_ops = d.set_ops;
	out->lipschitz = d.lipschitz ? 1u : 0u;
	out->flops_per_eval = d.flops;
	out->leaf_extent = d.leaf_extent;
	out->reserved = 0.0f;
}

extern "C" int tg_program_info_get(const tg_program* p, tg_program_info* out)
{
	if (!p || !out) return fail(TG_ERR_INVALID, "tg_program_info_get: null argument");
	fill_info(p->decoded, out);
	return TG_OK;
}

extern "C" int tg_words_inspect(const uint32_t* words, uint64_t count, tg_program_info* out)
{
	if (!words || !out || count == 0) return fail(TG_ERR_INVALID, "tg_words_inspect: null or empty argument");
	DecodedProgram d;
	std::string err;
	if (!decode_words(words, count, d, err))
		return fail(err.find("stack slots") != std::string::npos ? TG_ERR_LIMIT : TG_ERR_PROGRAM, "tg_words_inspect: " + err);
	fill_info(d, out);
	return TG_OK;
}

extern "C" void tg_program_destroy(tg_program* p)
{
	if (!p) return;
	p->device.release();
	p->entries.release();
	delete p;
}

// ---------------------------------------------------------------------------
// point queries

bool tg::split_program(const tg_program* p, SplitProgram& out)
{
	const DecodedProgram& d = p->decoded;
	out = SplitProgram{};
	out.slots = std::max<uint32_t>(1, d.max_stack - 1);
	auto fits = [&](const PrunePlan& plan) {
		return plan.stages() >= 2 && plan.stages() <= kSplitStages &&
		       split_lds_bytes(plan.slots, out.slots, kSplitWaves) <= kSplitMaxLds;
	};
	const bool narrow = fits(p->split_plan);
	const PrunePlan& plan = narrow ? p->split_plan : p->plan;
	if (!narrow && !fits(plan)) return false;
	out.prog = static_cast<const Instr*>(p->device.ptr);
	out.items = narrow ? p->split_items() : p->items();
	out.treelets = narrow ? p->split_treelets() : p->treelets();
	out.records = uint32_t(d.entries.size());
	out.stages = plan.stages();
	for (uint32_t s = 0; s <= out.stages; ++s) out.stage_first[s] = plan.stage_first[s];
	out.value_slots = plan.slots;
	return true;
}

namespace {

// Field evaluations up to which a workgroup shares 64 of them (SplitProgram):
// while they leave the GPU idle, an evaluation's latency is the call's.  (Whole
// program in one wave / split, us: 256 primitives 16384 evaluations 149 / 20, 131072
// 150 / 89, 262144 158 / 163; 2048 primitives 131072 1170 / 552; 64 primitives 131072
// 39 / 24; 24 primitives 16384 16 / 15, 131072 16 / 18.)
uint64_t split_evaluations(const tg_program* p) { return p->decoded.entries.size() >= 96 ? 131072 : 32768; }

// Whether gathering n points by cell and pruning the program for the cells costs
// less than the entries they save.  Whole program: 0.15 us an entry and 0.74 an
// entry and million points; gathered: 100 us and 0.16 an entry for the passes, 60
// us and 1.3 an entry that the cells keep a million points, 0.65 an entry kept at any
// count.  (Whole / gathered, us, random trees (0.05 of the entries kept): 256
// primitives 262144 points 184 / 195, 1M 483 / 241, 2M 802 / 297, 6M 2047 / 599; 2048
// primitives 524288 2002 / 862, 2M 5679 / 1373; 64 primitives 2M 222 / 250.  256
// primitives, 0.32 kept: 600k 362 / 412, 2M 835 / 719; 0.44: 2M 845 / 945; 1: 600k 363 /
// 617, 2M 816 / 1267.  1024 primitives, 0.22 kept: 300k 784 / 999, 600k 1382 / 1222, 2M
// 3147 / 2368; 0.38: 2M 3128 / 3273.)
bool sort_points(const tg_program* p, uint64_t n)
{
	const double m = 1e-6 * double(n), e = double(p->decoded.entries.size()), kept = p->kept;
	return n > split_evaluations(p) && m * ((0.74 - 1.3 * kept) * e - 60.0) > 100.0 + (0.01 + 0.65 * kept) * e;
}

// The same for gradients, four evaluations a point (whole call, as k_gradient /
// gathered, us: 256 primitives 50000 points 223 / 266, 100k 353 / 337, 200k 587 / 472,
// 1M 2684 / 1743; 64 primitives 200k 325 / 403, 1M 1636 / 1600; 512 primitives 20000
// 338 / 292, 100k 593 / 412; 2000 primitives 20000 1211 / 904, 100k 1847 / 1077.  256
// primitives, 0.32 of the entries kept: 200k 604 / 696, 400k 1057 / 1078, 1M 2792 / 2461;
// 0.44: 1M 2823 / 2938; 1: 100k 359 / 576, 1M 2849 / 3584.  1024 primitives, 0.22 kept:
// 100k 1057 / 1179, 200k 1747 / 1599; 0.38: 400k 3001 / 3250, 1M 7047 / 6773).
bool sort_gradients(const tg_program* p, uint64_t n)
{
	const double m = 1e-6 * double(n), e = double(p->decoded.entries.size()), kept = p->kept;
	return n > split_evaluations(p) / 8 &&
	       m * ((2.5 - 4.7 * kept) * e - 160.0) > 130.0 + (0.9 * kept - 0.11) * e;
}

constexpr uint32_t kSortCells = 24, kSortOuterCells = 8;  // per axis (fine cells, 2M points of 256 / 2048 primitives: 16 440 / 2473 us, 20 371 / 1833, 24 335 / 1467)
constexpr uint64_t kSortPoints = 4u << 20;  // points sorted at a time (their buffers: 144 MiB)

// The launches of sorted_points, with the workspace's buffers.
int sorted_launches(const tg_program* p, SortedPointsArgs& sa, const GradArgs* grad, float edge, float reach, bool fast,
	hipStream_t s, Workspace& ws, const PointsReady& ready, bool* sorted)
{
	const DecodedProgram& d = p->decoded;
	const uint64_t entries = d.entries.size(), count = sa.p.count;
	const float* xyz = sa.p.xyz;
	float* out = sa.p.out;
	sa.bins = sa.groups = 1;
	sa.chunk_shift = !grad ? 6 : grad->tetra ? 4 : 5;
	CellGrid grids[2];
	for (int L = 0; L < 2; ++L)
	{
		const uint32_t n = sa.n[L];
		const float size = L ? 4.0f * edge : edge, cell = size / float(n);
		const uint64_t nc = uint64_t(n) * n * n;
		for (int i = 0; i < 3; ++i) sa.lo[L][i] = 0.5f * (d.scene_lo[i] + d.scene_hi[i]) - 0.5f * size;
		sa.inv[L] = 1.0f / cell;
		sa.bins += uint32_t(nc);
		sa.groups += point_groups(n);
		// Nobody waits for the pruning, so the pool has to hold the programs at
		// once: a cell whose program finds no room runs the whole one.
		CellPrograms& lv = ws.levels[L];
		uint64_t room = nc * std::min<uint64_t>(std::max<uint64_t>(entries / 8, 64), 512);
		if (lv.host && lv.state.pending && !ws.in_flight)
			room = std::max<uint64_t>(room, std::min<uint64_t>(lv.host[0], 16u << 20));
		int rc = lv.pool.ensure(room * 4);
		if (rc) return rc;
		CellGrid& g = grids[L];
		for (int i = 0; i < 3; ++i)
		{
			g.origin[i] = sa.lo[L][i];
			g.cell[i] = cell;
			g.counts[i] = n;
		}
		// (points on a face of the cube's cells, the cells' centres: rounding)
		g.radius = 0.5f * cell * 1.7320508f * (1.0f + 1.0e-3f) + 1.0e-6f * (reach + 4.0f * edge);
		if (grad) g.radius += 1.7320508f * (1.0f + 1.0e-3f) * std::fabs(grad->h);
		g.words = true;
	}
	const uint64_t batch = std::min<uint64_t>(count, kSortPoints);
	int rc = ws.ctl.ensure((3 * size_t(sa.bins + 1) + (kGroupStride + 1) * size_t(sa.groups + 1)) * 4);
	if (!rc) rc = ws.out.ensure(batch * 4);
	if (!rc) rc = ws.queue.ensure(batch * 32);
	if (rc) return rc;
	const tg_program* progs[2] = { p, p };
	CellPrograms* outs[2] = { &ws.levels[0], &ws.levels[1] };
	rc = prune_cells_many(s, progs, grids, 2, fast, outs, ws.launches);
	if (rc) return rc;
	for (int L = 0; L < 2; ++L)
	{
		sa.words[L] = outs[L]->pool.as<const uint32_t>();
		sa.desc[L] = outs[L]->desc.as<const BlockDesc>();
	}
	if (ready) rc = ready();
	if (rc) return rc;
	sa.counts[0] = ws.ctl.as<uint32_t>();
	sa.counts[1] = sa.counts[0] + kGroupStride * sa.groups;
	sa.first[0] = sa.counts[1] + sa.bins;
	sa.first[1] = sa.first[0] + sa.groups + 1;
	sa.chunk = sa.first[1] + sa.bins + 1;
	sa.rank = ws.out.as<uint32_t>();
	sa.sorted[0] = ws.queue.as<float4>();
	sa.sorted[1] = sa.sorted[0] + batch;
	for (uint64_t at = 0; at < count; at += batch)
	{
		sa.p.xyz = xyz + 3 * at;
		sa.p.out = grad ? nullptr : out + at;
		sa.p.count = std::min<uint64_t>(batch, count - at);
		// (a kernel of our own: hipMemsetAsync launches two for this size, 8 us against 4)
		const uint32_t words = kGroupStride * sa.groups + sa.bins;
		hipLaunchKernelGGL(k_zero_words, dim3((words + 255) / 256), dim3(256), 0, s, sa.counts[0], words);
		TG_CHECK_HIP(hipGetLastError(), "bin reset");
		GradArgs ga{};
		if (grad)
		{
			ga = *grad;
			ga.out = grad->out + 3 * at;
		}
		const GradArgs* g = grad ? &ga : nullptr;
		const hipError_t e = fast ? fast::launch_points_sorted(sa, g, s) : exact::launch_points_sorted(sa, g, s);
		if (e != hipSuccess) return hip_fail(e, "sorted points launch");
	}
	*sorted = true;
	return TG_OK;
}

// Whether `count` points (with `gradients`, the gradients there) go through cell programs.
bool gathers(const tg_program* p, uint64_t count, bool gradients)
{
	const uint64_t ncells = uint64_t(kSortCells) * kSortCells * kSortCells;
	return (gradients ? sort_gradients(p, count) : sort_points(p, count)) && p->decoded.scene_finite &&
	       ncells * p->decoded.entries.size() <= (150ull << 20) && treelet_prunable(p, ncells);
}

// Evaluates `a` (with `grad`, the gradients there) through cell programs where
// that pays, asynchronously on `s`.  Not while `s` is captured: the call allocates.
// `ready` (if any) is called when the points are wanted, behind the pruning.
int sorted_points(const tg_program* p, const PointArgs& a, const GradArgs* grad, bool fast, hipStream_t s,
	const PointsReady& ready, bool* sorted)
{
	const DecodedProgram& d = p->decoded;
	if (!gathers(p, a.count, grad != nullptr)) return TG_OK;
	if (s)
	{
		hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
		if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
		{
			(void)hipGetLastError();
			return TG_OK;
		}
	}
	SortedPointsArgs sa{};
	sa.p = a;
	sa.n[0] = kSortCells;
	sa.n[1] = kSortOuterCells;
	float edge = 0.0f, reach = 0.0f;
	for (int i = 0; i < 3; ++i)
	{
		edge = std::max(edge, d.scene_hi[i] - d.scene_lo[i]);
		reach = std::max(reach, std::max(std::fabs(d.scene_lo[i]), std::fabs(d.scene_hi[i])));
	}
	edge = edge * 1.01f + 1e-3f;
	if (!(edge < 1e6f) || !(reach < 1e6f)) return TG_OK;
	// taps that reach beyond a cell of half the size prune little
	if (grad && !(std::fabs(grad->h) < 0.25f * edge / float(kSortCells))) return TG_OK;
	// allocations here are no part of a capture that another thread may have begun
	hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
	TG_CHECK_HIP(hipThreadExchangeStreamCaptureMode(&mode), "capture mode");
	struct Restore { hipStreamCaptureMode& m; ~Restore() { (void)hipThreadExchangeStreamCaptureMode(&m); } } restore{ mode };
	WorkspaceLease ws;
	int rc = ws.take(s);
	if (rc) return rc;
	rc = sorted_launches(p, sa, grad, edge, reach, fast, s, *ws.operator->(), ready, sorted);
	if (rc == TG_ERR_NOMEM)
	{
		// no room for the cells' programs (nothing is launched before the last
		// allocation): the whole program needs none
		ws->release();
		return TG_OK;
	}
	const int left = ws.leave_to(s);
	return rc ? rc : left;
}

}  // namespace

bool tg::gathers_gradients(const tg_program* p, uint64_t count) { return gathers(p, count, true); }

int tg::launch_gradients(const tg_program* p, const GradArgs& a, uint32_t flags, hipStream_t stream, const PointsReady& ready)
{
	const bool fast = (flags & TG_FLAG_FAST) != 0;
	PointArgs pa{};
	pa.prog = a.prog;
	pa.xyz = a.xyz;
	pa.count = a.count;
	pa.slots = a.slots;
	bool sorted = false;
	int rc = sorted_points(p, pa, &a, fast, stream, ready, &sorted);
	if (!rc && !sorted && ready) rc = ready();
	if (rc || sorted) return rc;
	SplitProgram sp;
	hipError_t e;
	// (four taps to a point and k_gradient a lane to a tap: half the evaluations;
	// 256 primitives 16384 points 210 / 105 us, 65536 276 / 275, 512 primitives 437 / 579)
	if (a.count <= split_evaluations(p) / 8 && split_program(p, sp))
		e = fast ? fast::launch_gradient_split(a, sp, stream) : exact::launch_gradient_split(a, sp, stream);
	else
		e = fast ? fast::launch_gradient(a, stream) : exact::launch_gradient(a, stream);
	return e == hipSuccess ? TG_OK : hip_fail(e, "gradient launch");
}

static int launch_eval_points(const tg_program* p, const float* xyz, uint64_t n, float* out, uint32_t flags, hipStream_t s,
	const PointsReady& ready)
{
	PointArgs a{};
	a.prog = static_cast<const Instr*>(p->device.ptr);
	a.xyz = xyz;
	a.out = out;
	a.count = n;
	a.slots = std::max<uint32_t>(1, p->decoded.max_stack - 1);
	const bool fast = (flags & TG_FLAG_FAST) != 0;
	bool sorted = false;
	int rc = sorted_points(p, a, nullptr, fast, s, ready, &sorted);
	if (!rc && !sorted && ready) rc = ready();
	if (rc || sorted) return rc;
	SplitProgram sp;
	hipError_t e;
	if (n <= split_evaluations(p) && split_program(p, sp))
		e = fast ? fast::launch_points_split(a, sp, s) : exact::launch_points_split(a, sp, s);
	else
		e = fast ? fast::launch_points(a, s) : exact::launch_points(a, s);
	if (e != hipSuccess) return hip_fail(e, "eval points launch");
	return TG_OK;
}

extern "C" int tg_eval_points_device(const tg_program* p, const float* xyz, uint64_t n, float* out, uint32_t flags,
	void* stream)
{
	if (!p || (n && (!xyz || !out))) return fail(TG_ERR_INVALID, "tg_eval_points_device: null argument");
	if (n == 0) return TG_OK;
	return launch_eval_points(p, xyz, n, out, flags, static_cast<hipStream_t>(stream), {});
}

extern "C" int tg_check_sqrt(uint32_t scramble, uint64_t* mismatches)
{
	if (!mismatches) return fail(TG_ERR_INVALID, "tg_check_sqrt: null argument");
	DevBuf d;
	int rc = d.ensure(8);
	if (rc) return rc;
	struct Guard { DevBuf& a; ~Guard() { a.release(); } } g{ d };
	TG_CHECK_HIP(hipMemset(d.ptr, 0, 8), "reset");
	TG_CHECK_HIP(exact::launch_sqrt_check(scramble, d.as<unsigned long long>(), nullptr), "sqrt check");
	unsigned long long n = 0;
	TG_CHECK_HIP(hipMemcpy(&n, d.ptr, 8, hipMemcpyDeviceToHost), "sqrt check");
	*mismatches = n;
	return TG_OK;
}

extern "C" int tg_check_quotient(const float* divisors, uint32_t n, uint64_t* mismatches, uint64_t* checked)
{
	if (!mismatches || !checked || (n && !divisors)) return fail(TG_ERR_INVALID, "tg_check_quotient: null argument");
	DevBuf d;
	int rc = d.ensure(16);
	if (rc) return rc;
	struct Guard { DevBuf& a; ~Guard() { a.release(); } } g{ d };
	TG_CHECK_HIP(hipMemset(d.ptr, 0, 16), "reset");
	for (uint32_t i = 0; i < n; ++i)
		TG_CHECK_HIP(exact::launch_quotient_check(divisors[i], d.as<unsigned long long>(), nullptr), "quotient check");
	unsigned long long c[2] = { 0, 0 };
	TG_CHECK_HIP(hipMemcpy(c, d.ptr, 16, hipMemcpyDeviceToHost), "quotient check");
	*mismatches = c[0];
	*checked = c[1];
	return TG_OK;
}

extern "C" int tg_eval_points(const tg_program* p, const float* xyz, uint64_t n, float* out, uint32_t flags)
{
	if (!p || (n && (!xyz || !out))) return fail(TG_ERR_INVALID, "tg_eval_points: null argument");
	if (n == 0) return TG_OK;
	WorkspaceLease ws;
	const float* in = nullptr;
	float* res = nullptr;
	int rc = ws.take();
	const bool gathered = gathers(p, n, false);
	if (!rc) rc = ws.stage(xyz, n, 1, gathered, &in, &res);
	if (!rc)
		rc = launch_eval_points(p, in, n, res, flags, nullptr,
			gathered ? PointsReady([&] { return ws.upload(xyz, n); }) : PointsReady());
	if (!rc) rc = ws.collect(out, n, 1);
	return rc;
}
