// Fourier-feature MLP surrogate: forward (prediction, brick flagging) and
// training (forward + backward + Adam) kernels for gfx950.
//
// Matrix products use v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32
// accumulation).  Operands live in LDS with the reduction index contiguous:
// an A operand is a row-major [M][K] array, a B operand is an [N][K] array
// (each output column's K values contiguous), so that every lane fetches its
// eight K values with one 16-byte read.  For a 16x16 output tile the lane
// layout is
//   A[i][k]: lane = i + 16 * (k / 8), element k % 8
//   B[k][j]: lane = j + 16 * (k / 8), element k % 8
//   D[i][j]: lane = j + 16 * (i / 4), element i % 4
// A wave processes 32 points at a time; hidden activations are written to LDS
// point-major ([point][unit], the next layer's B operand) and, in training, also
// unit-major ([unit][point], operands of the weight-gradient products whose
// reduction runs over points).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "tg_mlp.h"

namespace tg {
namespace mlp {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t to_bf16(float f)
{
	// round to nearest even (finite inputs)
	uint32_t u = __float_as_uint(f);
	u += 0x7fffu + ((u >> 16) & 1u);
	return uint16_t(u >> 16);
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }

__device__ __forceinline__ float silu_grad(float z)
{
	const float s = 1.0f / (1.0f + __expf(-z));
	return s * (1.0f + z * (1.0f - s));
}

// acc += A[16m.., k-block kb] * B[k-block kb, 16n..]
__device__ __forceinline__ f32x4 mma(const uint16_t* A, int lda, int m, const uint16_t* B, int ldb, int n, int kb,
	f32x4 acc, int lane)
{
	const int r = lane & 15, q = lane >> 4;
	const uint4 av = *reinterpret_cast<const uint4*>(A + (16 * m + r) * lda + 32 * kb + 8 * q);
	const uint4 bv = *reinterpret_cast<const uint4*>(B + (16 * n + r) * ldb + 32 * kb + 8 * q);
	return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bv), acc,
		0, 0, 0);
}

// Shared weights of one workgroup (BF16 operands, FP32 vectors).
struct Weights
{
	uint16_t w1[kHidden * kIn];       // [out][in]
	uint16_t w2[kHidden * kHidden];   // [out][in]
	float b1[kHidden], b2[kHidden], w3[kHidden];
	float b3;
	float fourier[kFreq * 3];
};

__device__ void load_weights(Weights& w, const Net& net, int tid, int nthreads)
{
	const float* p = net.params;
	for (int i = tid; i < kHidden * kIn; i += nthreads) w.w1[i] = to_bf16(p[kW1 + i]);
	for (int i = tid; i < kHidden * kHidden; i += nthreads) w.w2[i] = to_bf16(p[kW2 + i]);
	for (int i = tid; i < kHidden; i += nthreads)
	{
		w.b1[i] = p[kB1 + i];
		w.b2[i] = p[kB2 + i];
		w.w3[i] = p[kW3 + i];
	}
	for (int i = tid; i < kFreq * 3; i += nthreads) w.fourier[i] = net.fourier[i];
	if (tid == 0) w.b3 = p[kB3];
}

// Fourier features of point `pt` (lanes 0..31: sin, lanes 32..63: cos of the
// same 48 phases), x' = (p - lo) * inv_half - 1, phase in revolutions.
__device__ __forceinline__ void features(const Net& net, const Weights& w, uint16_t* fpm, float px,
	float py, float pz, int lane)
{
	const int pt = lane & 31;
	const bool cosine = lane >= 32;
	const float x = (px - net.lo[0]) * net.inv_half - 1.0f;
	const float y = (py - net.lo[1]) * net.inv_half - 1.0f;
	const float z = (pz - net.lo[2]) * net.inv_half - 1.0f;
	for (int f = 0; f < kFreq; ++f)
	{
		const float ph = (w.fourier[3 * f] * x + w.fourier[3 * f + 1] * y) + w.fourier[3 * f + 2] * z;
		const float v = cosine ? __builtin_amdgcn_cosf(ph) : __builtin_amdgcn_sinf(ph);
		const int k = (cosine ? kFreq : 0) + f;
		fpm[pt * kIn + k] = to_bf16(v);
	}
}

// Forward pass of 32 points: y of the lane's two points (16n + (lane & 15), n = 0, 1).
__device__ __forceinline__ void forward(const Weights& w, const uint16_t* fpm, uint16_t* a1pm, float y[2], int lane)
{
	const int r = lane & 15, q = lane >> 4;
	__builtin_amdgcn_s_waitcnt(0);
	__builtin_amdgcn_wave_barrier();
#pragma unroll
	for (int m = 0; m < 4; ++m)
#pragma unroll
		for (int n = 0; n < 2; ++n)
		{
			f32x4 acc = { 0, 0, 0, 0 };
#pragma unroll
			for (int kb = 0; kb < kIn / 32; ++kb) acc = mma(w.w1, kIn, m, fpm, kIn, n, kb, acc, lane);
			const int pt = 16 * n + r;
			const int u0 = 16 * m + 4 * q;
			uint16_t h[4];
#pragma unroll
			for (int i = 0; i < 4; ++i) h[i] = to_bf16(silu(acc[i] + w.b1[u0 + i]));
			uint2 packed = make_uint2(uint32_t(h[0]) | (uint32_t(h[1]) << 16), uint32_t(h[2]) | (uint32_t(h[3]) << 16));
			*reinterpret_cast<uint2*>(a1pm + pt * kHidden + u0) = packed;
		}
	__builtin_amdgcn_s_waitcnt(0);
	__builtin_amdgcn_wave_barrier();
	float part[2] = { 0.0f, 0.0f };
#pragma unroll
	for (int m = 0; m < 4; ++m)
#pragma unroll
		for (int n = 0; n < 2; ++n)
		{
			f32x4 acc = { 0, 0, 0, 0 };
#pragma unroll
			for (int kb = 0; kb < kHidden / 32; ++kb) acc = mma(w.w2, kHidden, m, a1pm, kHidden, n, kb, acc, lane);
#pragma unroll
			for (int i = 0; i < 4; ++i)
			{
				const int u = 16 * m + 4 * q + i;
				part[n] += w.w3[u] * silu(acc[i] + w.b2[u]);
			}
		}
#pragma unroll
	for (int n = 0; n < 2; ++n)
	{
		float v = part[n];
		v += __shfl_xor(v, 16);
		v += __shfl_xor(v, 32);
		y[n] = v + w.b3;
	}
}

// ---- prediction / brick flags --------------------------------------------------

struct ActsFwd
{
	uint16_t fpm[kGroup * kIn];
	uint16_t a1pm[kGroup * kHidden];
};

struct PredictShared
{
	Weights w;
	ActsFwd a[4];
};

__global__ void __launch_bounds__(256) k_predict(PredictArgs p)
{
	extern __shared__ __align__(16) unsigned char raw[];
	PredictShared& sh = *reinterpret_cast<PredictShared*>(raw);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	load_weights(sh.w, p.net, threadIdx.x, blockDim.x);
	__syncthreads();
	ActsFwd& a = sh.a[wave];
	const uint64_t groups = (p.count + kGroup - 1) / kGroup;
	const uint64_t stride = uint64_t(gridDim.x) * (blockDim.x >> 6);
	for (uint64_t g = uint64_t(blockIdx.x) * (blockDim.x >> 6) + wave; g < groups; g += stride)
	{
		const uint64_t i = g * kGroup + (lane & 31);
		const uint64_t j = i < p.count ? i : p.count - 1;
		float px, py, pz;
		if (p.xyz)
		{
			px = p.xyz[3 * j]; py = p.xyz[3 * j + 1]; pz = p.xyz[3 * j + 2];
		}
		else
		{
			// centre of cube brick j: cells [8b, 8b + 8) -> sample span [8b, 8b + 8]
			const uint32_t bx = uint32_t(j % p.cbx), by = uint32_t((j / p.cbx) % p.cby), bz = uint32_t(j / (uint64_t(p.cbx) * p.cby));
			px = p.gx + (float(bx * 8) + 4.0f) * p.dx;
			py = p.gy + (float(by * 8) + 4.0f) * p.dy;
			pz = p.gz + (float(bz * 8) + 4.0f) * p.dz;
		}
		__builtin_amdgcn_wave_barrier();
		features(p.net, sh.w, a.fpm, px, py, pz, lane);
		float out[2];
		forward(sh.w, a.fpm, a.a1pm, out, lane);
		if (lane < 32)
		{
			const int n = lane >> 4;  // lanes 0..15 hold points 0..15 (n=0), 16..31 hold 16..31 (n=1)
			const uint64_t k = g * kGroup + uint64_t(lane);
			const float y = n ? out[1] : out[0];
			if (k < p.count)
			{
				if (p.out) p.out[k] = y;
				if (p.flags)
				{
					// brick centre of this lane's point (lanes 0..31 own points 0..31)
					const float ux = fabsf((px - p.net.lo[0]) * p.net.inv_half - 1.0f);
					const float uy = fabsf((py - p.net.lo[1]) * p.net.inv_half - 1.0f);
					const float uz = fabsf((pz - p.net.lo[2]) * p.net.inv_half - 1.0f);
					const float reach = p.radius * p.net.inv_half;
					const bool outside = fmaxf(ux, fmaxf(uy, uz)) + reach > 1.0f;
					// keep unless the prediction certifies distance (NaN keeps)
					p.flags[k] = (outside || !(fabsf(y) > p.threshold)) ? 1 : 0;
				}
			}
		}
	}
}

// ---- training ----------------------------------------------------------------------

// Eight waves to two groups of 32 points: wave (m, h) owns the 16 units of
// tile m for the points of group h, forward and backward, and the weight
// gradients' tiles (m, n) with n in its half h, of both groups.  A 16384-point
// batch (512 groups) is a workgroup on each of the 256 CUs.
//
// What bounds it is the chain features -> layer 1 -> layer 2 -> loss -> layer 2
// -> layer 1 of one group (0.3 GFLOP, under a microsecond of the matrix cores), so
// the chain is cut short: a wave's weights go from memory straight into the
// registers that its matrix products read, the gradients of the two groups are
// added in registers and stored without an accumulator in LDS, and rows are
// padded so that 16 rows' reads fall on different banks.  (As one wave per
// group, weights and gradient sums in LDS: 79 us a batch; so: 20 us.)
constexpr int kTrainWaves = 8;
constexpr int kRowF = kIn + 8;       // padded rows (bf16)
constexpr int kRowH = kHidden + 8;
constexpr int kRowP = kGroup + 8;
constexpr int kRowS = kHidden + 4;   // (float)

struct TrainActs
{
	uint16_t fpm[kGroup * kRowF];     // features [pt][feature]
	uint16_t fum[kIn * kRowP];        // [feature][pt]
	uint16_t a1pm[kGroup * kRowH];    // hidden 1 [pt][unit]
	uint16_t a1um[kHidden * kRowP];   // [unit][pt]
	uint16_t dz2pm[kGroup * kRowH];
	uint16_t dz2um[kHidden * kRowP];
	uint16_t dz1um[kHidden * kRowP];
	float s2[kGroup * kRowS];         // silu(z2) [pt][unit]
	float gw3[kHidden], gb2[kHidden], gb1[kHidden];
	float gb3, loss;
};

struct TrainShared
{
	TrainActs a[2];
};

// Sum over the 16 lanes that share q (i.e. over the lane's points), result in
// every lane.
__device__ __forceinline__ float sum16(float v)
{
	v += __shfl_xor(v, 1);
	v += __shfl_xor(v, 2);
	v += __shfl_xor(v, 4);
	v += __shfl_xor(v, 8);
	return v;
}

// Eight floats rounded to a matrix operand.
__device__ __forceinline__ bf16x8 operand(const float* v)
{
	uint32_t w[4];
#pragma unroll
	for (int i = 0; i < 4; ++i) w[i] = uint32_t(to_bf16(v[2 * i])) | (uint32_t(to_bf16(v[2 * i + 1])) << 16);
	return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

// Row 16t + r of an LDS operand, k-block kb.
__device__ __forceinline__ bf16x8 row_operand(const uint16_t* M, int ld, int t, int kb, int lane)
{
	const int r = lane & 15, q = lane >> 4;
	return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(M + (16 * t + r) * ld + 32 * kb + 8 * q));
}

__global__ void __launch_bounds__(64 * kTrainWaves) k_train_grad(TrainArgs t)
{
	extern __shared__ __align__(16) unsigned char raw[];
	TrainShared& sh = *reinterpret_cast<TrainShared*>(raw);
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
	const int m = wave & 3, h = wave >> 2;
	const int r = lane & 15, q = lane >> 4;
	const int u0 = 16 * m + 4 * q;  // the lane's four units of tile m
	const bool two = t.groups_per_block == 2;
	const bool live = h == 0 || two;
	const float* P = t.net.params;
	TrainActs& a = sh.a[h];
	// this wave's rows of W1 and W2, its columns of W2 (rows of the transpose)
	bf16x8 w1[kIn / 32], w2[kHidden / 32], w2t[kHidden / 32];
	float b1[4], b2[4], w3[kHidden / 4];
#pragma unroll
	for (int kb = 0; kb < kIn / 32; ++kb)
	{
		float v[8];
#pragma unroll
		for (int j = 0; j < 8; ++j) v[j] = P[kW1 + (16 * m + r) * kIn + 32 * kb + 8 * q + j];
		w1[kb] = operand(v);
	}
#pragma unroll
	for (int kb = 0; kb < kHidden / 32; ++kb)
	{
		float v[8], vt[8];
#pragma unroll
		for (int j = 0; j < 8; ++j)
		{
			v[j] = P[kW2 + (16 * m + r) * kHidden + 32 * kb + 8 * q + j];
			vt[j] = P[kW2 + (32 * kb + 8 * q + j) * kHidden + 16 * m + r];
		}
		w2[kb] = operand(v);
		w2t[kb] = operand(vt);
	}
#pragma unroll
	for (int i = 0; i < 4; ++i)
	{
		b1[i] = P[kB1 + u0 + i];
		b2[i] = P[kB2 + u0 + i];
#pragma unroll
		for (int mm = 0; mm < 4; ++mm) w3[4 * mm + i] = P[kW3 + 16 * mm + 4 * q + i];
	}
	const float b3 = P[kB3];
	const uint64_t s0 = t.batch_offset + (uint64_t(blockIdx.x) * t.groups_per_block + uint64_t(live ? h : 0)) * kGroup;
	const float scale = 2.0f / float(t.batch);
	float target[2];
#pragma unroll
	for (int n = 0; n < 2; ++n) target[n] = t.samples[s0 + 16 * n + r].w;
	const float4 sample = t.samples[s0 + (lane & 31)];
	if (live)
	{
		// 12 of the 96 features of a point to each lane (lanes 0..31 sines, 32..63 cosines)
		const int pt = lane & 31, c = lane >> 5;
		const float x = (sample.x - t.net.lo[0]) * t.net.inv_half - 1.0f;
		const float y = (sample.y - t.net.lo[1]) * t.net.inv_half - 1.0f;
		const float z = (sample.z - t.net.lo[2]) * t.net.inv_half - 1.0f;
		const float* fr = t.net.fourier + 3 * (kFreq / 4) * m;
		const int k0 = kFreq * c + (kFreq / 4) * m;
		uint16_t b[kFreq / 4];
#pragma unroll
		for (int f = 0; f < kFreq / 4; ++f)
		{
			const float ph = (fr[3 * f] * x + fr[3 * f + 1] * y) + fr[3 * f + 2] * z;
			b[f] = to_bf16(c ? __builtin_amdgcn_cosf(ph) : __builtin_amdgcn_sinf(ph));
			a.fum[(k0 + f) * kRowP + pt] = b[f];
		}
#pragma unroll
		for (int f = 0; f < kFreq / 4; f += 4)
			*reinterpret_cast<uint2*>(a.fpm + pt * kRowF + k0 + f) = make_uint2(
				uint32_t(b[f]) | (uint32_t(b[f + 1]) << 16), uint32_t(b[f + 2]) | (uint32_t(b[f + 3]) << 16));
	}
	__syncthreads();
	float z1[2][4], z2[2][4];
	if (live)
#pragma unroll
		for (int n = 0; n < 2; ++n)
		{
			f32x4 acc = { 0, 0, 0, 0 };
#pragma unroll
			for (int kb = 0; kb < kIn / 32; ++kb)
				acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[kb], row_operand(a.fpm, kRowF, n, kb, lane), acc, 0, 0, 0);
			uint16_t v[4];
#pragma unroll
			for (int i = 0; i < 4; ++i)
			{
				z1[n][i] = acc[i] + b1[i];
				v[i] = to_bf16(silu(z1[n][i]));
				a.a1um[(u0 + i) * kRowP + 16 * n + r] = v[i];
			}
			*reinterpret_cast<uint2*>(a.a1pm + (16 * n + r) * kRowH + u0) =
				make_uint2(uint32_t(v[0]) | (uint32_t(v[1]) << 16), uint32_t(v[2]) | (uint32_t(v[3]) << 16));
		}
	__syncthreads();
	float s2[2][4];
	if (live)
#pragma unroll
		for (int n = 0; n < 2; ++n)
		{
			f32x4 acc = { 0, 0, 0, 0 };
#pragma unroll
			for (int kb = 0; kb < kHidden / 32; ++kb)
				acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w2[kb], row_operand(a.a1pm, kRowH, n, kb, lane), acc, 0, 0, 0);
#pragma unroll
			for (int i = 0; i < 4; ++i)
			{
				z2[n][i] = acc[i] + b2[i];
				s2[n][i] = silu(z2[n][i]);
			}
			*reinterpret_cast<float4*>(a.s2 + (16 * n + r) * kRowS + u0) =
				make_float4(s2[n][0], s2[n][1], s2[n][2], s2[n][3]);
		}
	__syncthreads();
	if (live)
	{
		// output of the lane's two points (every wave of the group), dL/dy of the
		// mean squared error
		float dy[2];
		float sq = 0.0f;
#pragma unroll
		for (int n = 0; n < 2; ++n)
		{
			float v = 0.0f;
#pragma unroll
			for (int mm = 0; mm < 4; ++mm)
			{
				const float4 s = *reinterpret_cast<const float4*>(a.s2 + (16 * n + r) * kRowS + 16 * mm + 4 * q);
				v += w3[4 * mm] * s.x;
				v += w3[4 * mm + 1] * s.y;
				v += w3[4 * mm + 2] * s.z;
				v += w3[4 * mm + 3] * s.w;
			}
			v += __shfl_xor(v, 16);
			v += __shfl_xor(v, 32);
			const float e = (v + b3) - fminf(fmaxf(target[n], -t.net.clamp), t.net.clamp);
			dy[n] = scale * e;
			sq += e * e;
		}
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			float gw3 = 0.0f, gb2 = 0.0f;
#pragma unroll
			for (int n = 0; n < 2; ++n)
			{
				gw3 += dy[n] * s2[n][i];
				const float d = dy[n] * P[kW3 + u0 + i] * silu_grad(z2[n][i]);
				gb2 += d;
				const uint16_t b = to_bf16(d);
				a.dz2um[(u0 + i) * kRowP + 16 * n + r] = b;
				a.dz2pm[(16 * n + r) * kRowH + u0 + i] = b;
			}
			gw3 = sum16(gw3);
			gb2 = sum16(gb2);
			if (r == 0)
			{
				a.gw3[u0 + i] = gw3;
				a.gb2[u0 + i] = gb2;
			}
		}
		const float gb3 = sum16(dy[0] + dy[1]);
		sq = sum16(sq);
		if (m == 0 && lane == 0)
		{
			a.gb3 = gb3;
			a.loss = sq;
		}
	}
	__syncthreads();
	float* out = t.partial + size_t(blockIdx.x) * kParams;
	if (live)
	{
		// da1[u][pt] = sum_o W2[o][u] dz2[o][pt]; dz1 = da1 * silu'(z1)
		float gb1[4] = { 0, 0, 0, 0 };
#pragma unroll
		for (int n = 0; n < 2; ++n)
		{
			f32x4 acc = { 0, 0, 0, 0 };
#pragma unroll
			for (int kb = 0; kb < kHidden / 32; ++kb)
				acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w2t[kb], row_operand(a.dz2pm, kRowH, n, kb, lane), acc, 0, 0, 0);
#pragma unroll
			for (int i = 0; i < 4; ++i)
			{
				const float d = acc[i] * silu_grad(z1[n][i]);
				gb1[i] += d;
				a.dz1um[(u0 + i) * kRowP + 16 * n + r] = to_bf16(d);
			}
		}
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			const float v = sum16(gb1[i]);
			if (r == 0) a.gb1[u0 + i] = v;
		}
	}
	// dW2[o][i] = sum_pt dz2[o][pt] a1[i][pt], both groups
	{
		const bf16x8 d0 = row_operand(sh.a[0].dz2um, kRowP, m, 0, lane);
		const bf16x8 d1 = row_operand(sh.a[1].dz2um, kRowP, m, 0, lane);
#pragma unroll
		for (int j = 0; j < 2; ++j)
		{
			const int n = 2 * h + j;
			const f32x4 zero = { 0, 0, 0, 0 };
			f32x4 g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d0, row_operand(sh.a[0].a1um, kRowP, n, 0, lane), zero, 0, 0, 0);
			if (two) g += __builtin_amdgcn_mfma_f32_16x16x32_bf16(d1, row_operand(sh.a[1].a1um, kRowP, n, 0, lane), zero, 0, 0, 0);
#pragma unroll
			for (int i = 0; i < 4; ++i) out[kW2 + (u0 + i) * kHidden + 16 * n + r] = g[i];
		}
	}
	__syncthreads();
	// dW1[o][k] = sum_pt dz1[o][pt] f[k][pt], both groups
	{
		const bf16x8 d0 = row_operand(sh.a[0].dz1um, kRowP, m, 0, lane);
		const bf16x8 d1 = row_operand(sh.a[1].dz1um, kRowP, m, 0, lane);
#pragma unroll
		for (int j = 0; j < kIn / 32; ++j)
		{
			const int n = (kIn / 32) * h + j;
			const f32x4 zero = { 0, 0, 0, 0 };
			f32x4 g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d0, row_operand(sh.a[0].fum, kRowP, n, 0, lane), zero, 0, 0, 0);
			if (two) g += __builtin_amdgcn_mfma_f32_16x16x32_bf16(d1, row_operand(sh.a[1].fum, kRowP, n, 0, lane), zero, 0, 0, 0);
#pragma unroll
			for (int i = 0; i < 4; ++i) out[kW1 + (u0 + i) * kIn + 16 * n + r] = g[i];
		}
	}
	const TrainActs& g0 = sh.a[0];
	const TrainActs& g1 = sh.a[1];
	if (wave == 0)
	{
		out[kW3 + lane] = two ? g0.gw3[lane] + g1.gw3[lane] : g0.gw3[lane];
		out[kB2 + lane] = two ? g0.gb2[lane] + g1.gb2[lane] : g0.gb2[lane];
		out[kB1 + lane] = two ? g0.gb1[lane] + g1.gb1[lane] : g0.gb1[lane];
		if (lane == 0)
		{
			out[kB3] = two ? g0.gb3 + g1.gb3 : g0.gb3;
			if (t.loss_partial) t.loss_partial[blockIdx.x] = two ? g0.loss + g1.loss : g0.loss;
		}
	}
}

// A workgroup per 64 parameters (lane = parameter): wave w sums every 16th block
// partial from its own, all loads in flight at once, and the 16 sums are added in
// a fixed order (deterministic), then Adam with bias correction and cosine
// learning-rate decay to 5%.  Workgroup 0 also sums the loss partials.
// (256 partials, 10.7 MB: as 4 waves of 64 loads each 21 us, so 5 us.)
constexpr int kAdamWaves = 16;
constexpr uint32_t kAdamLoads = 16;

__global__ void __launch_bounds__(64 * kAdamWaves) k_adam(AdamArgs a)
{
	__shared__ float part[kAdamWaves][64];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const uint32_t i = blockIdx.x * 64 + uint32_t(lane);
	const bool in = i < uint32_t(kParams);
	const uint64_t step = *a.epoch * a.batches + a.batch_index + 1;
	float acc = 0.0f;
	if (in)
		for (uint32_t first = uint32_t(wave); first < a.blocks; first += kAdamWaves * kAdamLoads)
		{
			float v[kAdamLoads];
#pragma unroll
			for (uint32_t k = 0; k < kAdamLoads; ++k)
			{
				const uint32_t b = first + kAdamWaves * k;
				v[k] = b < a.blocks ? a.partial[size_t(b) * kParams + i] : 0.0f;
			}
#pragma unroll
			for (uint32_t k = 0; k < kAdamLoads; ++k) acc += v[k];
		}
	part[wave][lane] = acc;
	__syncthreads();
	if (wave == 0 && in)
	{
		// chain c holds the partials = c mod 16; sums of chains c, c + 4, c + 8, c + 12, in order of c
		float p[4];
#pragma unroll
		for (int c = 0; c < 4; ++c) p[c] = (part[c][lane] + part[c + 4][lane]) + (part[c + 8][lane] + part[c + 12][lane]);
		const float g = ((p[0] + p[1]) + p[2]) + p[3];
		const float m = a.beta1 * a.m[i] + (1.0f - a.beta1) * g;
		const float v = a.beta2 * a.v[i] + (1.0f - a.beta2) * g * g;
		a.m[i] = m;
		a.v[i] = v;
		const float c1 = 1.0f - powf(a.beta1, float(step));
		const float c2 = 1.0f - powf(a.beta2, float(step));
		const float frac = a.decay_steps ? fminf(1.0f, float(step) / float(a.decay_steps)) : 0.0f;
		const float lr = a.lr * (0.05f + 0.95f * 0.5f * (1.0f + cospif(frac)));
		a.params[i] -= lr * (m / c1) / (sqrtf(v / c2) + a.eps);
	}
	if (blockIdx.x == 0 && wave == 1 && a.loss_log && step - 1 < a.log_capacity)
	{
		float l = 0.0f;
		for (uint32_t b = uint32_t(lane); b < a.blocks; b += 64) l += a.loss_partial[b];
#pragma unroll
		for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
		if (lane == 0) a.loss_log[step - 1] = l / float(a.batch);
	}
}

__global__ void __launch_bounds__(256) k_gather_samples(const float* xyz, const float* target, const uint32_t* order,
	float4* samples, uint64_t n)
{
	const uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (k >= n) return;
	const uint64_t i = order ? order[k] : k;
	samples[k] = make_float4(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], target[i]);
}

__global__ void k_epoch_advance(uint64_t* epoch) { *epoch += 1; }

}  // namespace

hipError_t prepare()
{
	hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_predict),
		hipFuncAttributeMaxDynamicSharedMemorySize, int(sizeof(PredictShared)));
	if (e == hipSuccess)
		e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_train_grad), hipFuncAttributeMaxDynamicSharedMemorySize,
			int(sizeof(TrainShared)));
	return e;
}

hipError_t launch_predict(const PredictArgs& p, hipStream_t s)
{
	if (p.count == 0) return hipSuccess;
	const uint64_t groups = (p.count + kGroup - 1) / kGroup;
	const unsigned blocks = unsigned(std::min<uint64_t>((groups + 3) / 4, 4096));
	hipLaunchKernelGGL(k_predict, dim3(blocks), dim3(256), sizeof(PredictShared), s, p);
	return hipGetLastError();
}

hipError_t launch_train_grad(const TrainArgs& t, uint32_t blocks, hipStream_t s)
{
	hipLaunchKernelGGL(k_train_grad, dim3(blocks), dim3(64 * kTrainWaves), sizeof(TrainShared), s, t);
	return hipGetLastError();
}

hipError_t launch_adam(const AdamArgs& a, hipStream_t s)
{
	hipLaunchKernelGGL(k_adam, dim3((kParams + 63) / 64), dim3(64 * kAdamWaves), 0, s, a);
	return hipGetLastError();
}

hipError_t launch_gather_samples(const float* xyz, const float* target, const uint32_t* order, float4* samples,
	uint64_t n, hipStream_t s)
{
	if (n == 0) return hipSuccess;
	hipLaunchKernelGGL(k_gather_samples, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, xyz, target, order, samples, n);
	return hipGetLastError();
}

hipError_t launch_epoch_advance(uint64_t* epoch, hipStream_t s)
{
	hipLaunchKernelGGL(k_epoch_advance, dim3(1), dim3(1), 0, s, epoch);
	return hipGetLastError();
}

}  // namespace mlp
}  // namespace tg
