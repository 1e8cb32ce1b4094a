// MFMA operand helpers shared by the forward sweeps (gfx950 only): f16 / bf16
// packing and the surplus operands (the MFMA A side) of one node chunk.
#pragma once

#include <type_traits>

#include "hddm_lb.h"
#include "device_common.h"

namespace hddm_lb {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef float f16_t __attribute__((ext_vector_type(16)));


__device__ __forceinline__ uint32_t pack_h2(float a, float b)
{
	h2_t v;
	v[0] = (_Float16)a;
	v[1] = (_Float16)b;
	return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ uint32_t pack_b2(float a, float b)
{
	b2_t v;
	v[0] = (__bf16)a;
	v[1] = (__bf16)b;
	return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float lo_half_f16(uint32_t u) { return (float)__builtin_bit_cast(h2_t, u)[0]; }
__device__ __forceinline__ float hi_half_f16(uint32_t u) { return (float)__builtin_bit_cast(h2_t, u)[1]; }
__device__ __forceinline__ float lo_half_bf16(uint32_t u) { return __builtin_bit_cast(float, u << 16); }
__device__ __forceinline__ float hi_half_bf16(uint32_t u) { return __builtin_bit_cast(float, u & 0xffff0000u); }

template <typename V>
__device__ __forceinline__ V as_vec8(uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
	u4_t u = { a, b, c, d };
	return __builtin_bit_cast(V, u);
}

// S^T operands (the MFMA A side) of one chunk (16 nodes; 32 for F32, two
// consecutive 16-node surplus chunks), loaded ahead of use.
template <int PREC, int DT>
struct SOperands
{
	typedef typename std::conditional<PREC == HDDM_LB_F16X2, h8_t,
		typename std::conditional<PREC == HDDM_LB_BF16X3, b8_t, float>::type>::type V;
	static constexpr int kTerms = PREC == HDDM_LB_F16X2 ? 2 : (PREC == HDDM_LB_BF16X3 ? 3 : 16);
	V A[DT][kTerms];

	__device__ __forceinline__ void load(const StateDesc* sd, int chunk, int DP, int dt0, int ndt, int lane)
	{
		const int row = lane & 31;
		const int khalf = lane >> 5;
#pragma unroll
		for (int dt = 0; dt < DT; dt++)
			if (dt < ndt)
			{
				const int dr = (dt0 + dt) * 32 + row;
				if constexpr (PREC == HDDM_LB_F16X2)
				{
					const uint16_t* sc = ldc(&sd->s16) + (size_t)chunk * 2 * DP * kChunk;
					A[dt][0] = *(const h8_t*)(sc + ((size_t)dr) * kChunk + khalf * 8);
					A[dt][1] = *(const h8_t*)(sc + ((size_t)DP + dr) * kChunk + khalf * 8);
				}
				else if constexpr (PREC == HDDM_LB_BF16X3)
				{
					const uint16_t* sc = ldc(&sd->sbf) + (size_t)chunk * 3 * DP * kChunk;
#pragma unroll
					for (int term = 0; term < 3; term++)
						A[dt][term] = *(const b8_t*)(sc + ((size_t)term * DP + dr) * kChunk + khalf * 8);
				}
				else
				{
					// K-step q (nodes 2q, 2q+1 of the 32) is step q % 8 of
					// surplus chunk 2 chunk + q / 8; past the last chunk: 0
					const int nch = ldc(&sd->nchunks);
#pragma unroll
					for (int h = 0; h < 2; h++)
					{
						const int sc = 2 * chunk + h;
						const float* ap = ldc(&sd->s32) + (size_t)(sc < nch ? sc : 0) * DP * kChunk
							+ ((size_t)dr * 2 + khalf) * 8;
#pragma unroll
						for (int q = 0; q < 8; q++) A[dt][8 * h + q] = sc < nch ? ap[q] : 0.0f;
					}
				}
			}
	}
};

// Basis values are scaled by this power of two before the f16 hi/lo split, so
// that the low halves of basis values down to 2^-12 stay normal f16 numbers.
constexpr float kBScale = 4096.0f;

// Split-precision MFMA contraction of one 16-node chunk (F16X2, BF16X3):
// acc[t][dt] (points 32t.., dofs 32(dt0+dt)..) += S^T[dofs x 16 nodes] *
// B^T[16 nodes x 32 points]. The F32 path contracts in the sweep kernels.
template <int PREC, int DT, typename BT>
__device__ __forceinline__ void contract_chunk(const SOperands<PREC, DT>& so, int ndt,
	const BT (&b)[kChunk], f16_t (&acc)[2][DT])
{
	if constexpr (PREC == HDDM_LB_F16X2)
	{
		// B is scaled by 2^12 before the split so that the low halves of
		// basis values down to 2^-12 stay normal f16 numbers
		uint32_t hi[8], lo[8];
#pragma unroll
		for (int m = 0; m < 8; m++)
		{
			// split in FP32 (one rounding from FP64; the f16 pair keeps 22 bits)
			const float f0 = (float)b[2 * m] * kBScale, f1 = (float)b[2 * m + 1] * kBScale;
			hi[m] = pack_h2(f0, f1);
			lo[m] = pack_h2(f0 - lo_half_f16(hi[m]), f1 - hi_half_f16(hi[m]));
		}
		// Lanes 0-31 own points 0-31, lanes 32-63 points 32-63; each holds
		// nodes 0-15 of its point. The B operand of points 0-31 needs nodes
		// 0-7 in lanes 0-31 and nodes 8-15 in lanes 32-63: one half-swap.
#pragma unroll
		for (int m = 0; m < 4; m++)
		{
			auto rh = __builtin_amdgcn_permlane32_swap(hi[m], hi[m + 4], false, false);
			hi[m] = rh[0]; hi[m + 4] = rh[1];
			auto rl = __builtin_amdgcn_permlane32_swap(lo[m], lo[m + 4], false, false);
			lo[m] = rl[0]; lo[m + 4] = rl[1];
		}
		const h8_t Bh0 = as_vec8<h8_t>(hi[0], hi[1], hi[2], hi[3]);
		const h8_t Bh1 = as_vec8<h8_t>(hi[4], hi[5], hi[6], hi[7]);
		const h8_t Bl0 = as_vec8<h8_t>(lo[0], lo[1], lo[2], lo[3]);
		const h8_t Bl1 = as_vec8<h8_t>(lo[4], lo[5], lo[6], lo[7]);
#pragma unroll
		for (int dt = 0; dt < DT; dt++)
			if (dt < ndt)
			{
				const h8_t Ah = so.A[dt][0], Al = so.A[dt][1];
				acc[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Al, Bh0, acc[0][dt], 0, 0, 0);
				acc[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah, Bl0, acc[0][dt], 0, 0, 0);
				acc[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah, Bh0, acc[0][dt], 0, 0, 0);
				acc[1][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Al, Bh1, acc[1][dt], 0, 0, 0);
				acc[1][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah, Bl1, acc[1][dt], 0, 0, 0);
				acc[1][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah, Bh1, acc[1][dt], 0, 0, 0);
			}
	}
	else if constexpr (PREC == HDDM_LB_BF16X3)
	{
		uint32_t t1[8], t2[8], t3[8];
#pragma unroll
		for (int m = 0; m < 8; m++)
		{
			// split in FP32: three bf16 terms carry the 24 bits of the FP32 value
			const float f0 = (float)b[2 * m], f1 = (float)b[2 * m + 1];
			t1[m] = pack_b2(f0, f1);
			const float r0 = f0 - lo_half_bf16(t1[m]), r1 = f1 - hi_half_bf16(t1[m]);
			t2[m] = pack_b2(r0, r1);
			t3[m] = pack_b2(r0 - lo_half_bf16(t2[m]), r1 - hi_half_bf16(t2[m]));
		}
#pragma unroll
		for (int m = 0; m < 4; m++)
		{
			auto r1 = __builtin_amdgcn_permlane32_swap(t1[m], t1[m + 4], false, false);
			t1[m] = r1[0]; t1[m + 4] = r1[1];
			auto r2 = __builtin_amdgcn_permlane32_swap(t2[m], t2[m + 4], false, false);
			t2[m] = r2[0]; t2[m + 4] = r2[1];
			auto r3 = __builtin_amdgcn_permlane32_swap(t3[m], t3[m + 4], false, false);
			t3[m] = r3[0]; t3[m + 4] = r3[1];
		}
		b8_t B[2][3];
		B[0][0] = as_vec8<b8_t>(t1[0], t1[1], t1[2], t1[3]);
		B[1][0] = as_vec8<b8_t>(t1[4], t1[5], t1[6], t1[7]);
		B[0][1] = as_vec8<b8_t>(t2[0], t2[1], t2[2], t2[3]);
		B[1][1] = as_vec8<b8_t>(t2[4], t2[5], t2[6], t2[7]);
		B[0][2] = as_vec8<b8_t>(t3[0], t3[1], t3[2], t3[3]);
		B[1][2] = as_vec8<b8_t>(t3[4], t3[5], t3[6], t3[7]);
#pragma unroll
		for (int dt = 0; dt < DT; dt++)
			if (dt < ndt)
			{
#pragma unroll
				for (int t = 0; t < 2; t++)
				{
					// smallest products first
					acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(so.A[dt][2], B[t][0], acc[t][dt], 0, 0, 0);
					acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(so.A[dt][1], B[t][1], acc[t][dt], 0, 0, 0);
					acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(so.A[dt][0], B[t][2], acc[t][dt], 0, 0, 0);
					acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(so.A[dt][1], B[t][0], acc[t][dt], 0, 0, 0);
					acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(so.A[dt][0], B[t][1], acc[t][dt], 0, 0, 0);
					acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(so.A[dt][0], B[t][0], acc[t][dt], 0, 0, 0);
				}
			}
	}
}

} // namespace hddm_lb
