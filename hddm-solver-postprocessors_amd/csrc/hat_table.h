// What the kernels over hat tables share: a block's hats in LDS, the windows'
// alive ops, the prefix products.
#pragma once

#include "sweep_common.h"
#include "layout.h"

#include <type_traits>

namespace hddm_lb {

// The prefix products of the current trie path: P[t] is the product of its
// first t factors (t up to 7). The statements below pin them to 16 vector
// registers from BASE on, which GPR indexing needs; it writes m0, where the
// compiler keeps nothing.
typedef double dv8_t __attribute__((ext_vector_type(8)));
template <int BASE> struct Path;

// P[t + 1] = P[t] * |F|, T = 2 t: one multiply whose source and destination are
// both indexed (the index is the low 8 bits of T); F may carry a sign
#define HDDM_MULP(P0, P1, T, F) \
	"s_set_gpr_idx_on " T ", gpr_idx(SRC0,DST)\n" \
	"v_mul_f64 " P1 ", " P0 ", |" F "|\n"
#define HDDM_OUT64(P1, B) "s_set_gpr_idx_mode gpr_idx(SRC0)\n" "v_mov_b64 " B ", " P1 "\n"
#define HDDM_OUT32(P1, B) "s_set_gpr_idx_mode gpr_idx(SRC0)\n" "v_cvt_f32_f64 " B ", " P1 "\n"
// four nodes in trie order, the products returned in b (the wait states: the
// instructions that take them, row swaps and MFMAs, do not see them written
// by a VALU instruction)
#define HDDM_MULP4(P0, P1, ALL, OUT) \
	asm(HDDM_MULP(P0, P1, "%[t0]", "%[f0]") OUT(P1, "%[b0]") HDDM_MULP(P0, P1, "%[t1]", "%[f1]") OUT(P1, "%[b1]") \
		HDDM_MULP(P0, P1, "%[t2]", "%[f2]") OUT(P1, "%[b2]") HDDM_MULP(P0, P1, "%[t3]", "%[f3]") OUT(P1, "%[b3]") \
		"s_set_gpr_idx_off\n" "s_nop 1\n" \
		: [b0] "=&v"(b[0]), [b1] "=&v"(b[1]), [b2] "=&v"(b[2]), [b3] "=&v"(b[3]), "+{" ALL "}"(P) \
		: [t0] "s"(r[0]), [t1] "s"(r[1]), [t2] "s"(r[2]), [t3] "s"(r[3]), \
		  [f0] "v"(f[0]), [f1] "v"(f[1]), [f2] "v"(f[2]), [f3] "v"(f[3]) : "m0")
#define HDDM_PATH(BASE, P0, P1, ALL) \
	template <> struct Path<BASE> \
	{ \
		__device__ __forceinline__ static void mulp(dv8_t& P, uint32_t t2, double f) \
		{ \
			asm(HDDM_MULP(P0, P1, "%[t]", "%[f]") "s_set_gpr_idx_off\n" : "+{" ALL "}"(P) : [t] "s"(t2), [f] "v"(f) : "m0"); \
		} \
		template <typename B> __device__ __forceinline__ static void mulp4(dv8_t& P, const uint32_t* r, const double* f, B* b) \
		{ \
			if constexpr (sizeof(B) == 8) HDDM_MULP4(P0, P1, ALL, HDDM_OUT64); \
			else HDDM_MULP4(P0, P1, ALL, HDDM_OUT32); \
		} \
	}
HDDM_PATH(152, "v[152:153]", "v[154:155]", "v[152:167]");
HDDM_PATH(224, "v[224:225]", "v[226:227]", "v[224:239]");
#undef HDDM_PATH
#undef HDDM_MULP
#undef HDDM_MULP4
#undef HDDM_OUT64
#undef HDDM_OUT32

__device__ __forceinline__ void row_swap32(double& a, double& b)
{
	auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
	auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
	a = __hiloint2double((int)hi[0], (int)lo[0]);
	b = __hiloint2double((int)hi[1], (int)lo[1]);
}

__device__ __forceinline__ void row_swap16(double& a, double& b)
{
	auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
	auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
	a = __hiloint2double((int)hi[0], (int)lo[0]);
	b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// Exchanges the register index and the row of 16 lanes: register i of row r
// becomes register r of row i.
__device__ __forceinline__ void transpose_rows(double& b0, double& b1, double& b2, double& b3)
{
	row_swap32(b0, b2);
	row_swap32(b1, b3);
	row_swap16(b0, b1);
	row_swap16(b2, b3);
}

// The alive ops (ANDed masks of their hats in M not empty) of windows first,
// first + step, ..., nb of them: window i's 64 bits in lane i of (mlo, mhi),
// 0 in the lanes from nb on.
__device__ __forceinline__ void select_windows(const StateDesc* sd, const uint64_t* M, int first, int step, int nb, int lane,
	uint32_t& mlo, uint32_t& mhi)
{
	mlo = 0;
	mhi = 0;
	auto select = [&](auto words) {
		constexpr int W = decltype(words)::value;   // pairs of hat ids per op
		constexpr int kSel = W == 1 ? 8 : 4;        // windows in flight
		const uint32_t* hid = (const uint32_t*)ldc(&sd->thid) + ((size_t)first * kWin + lane) * W;
#pragma unroll 1
		for (int i = 0; i < nb; i += kSel)
		{
			uint32_t id[kSel][W];
#pragma unroll
			for (int j = 0; j < kSel; j++)
			{
				const uint32_t* src = hid + (size_t)(min(i + j, nb - 1) * step) * (kWin * W);
#pragma unroll
				for (int w = 0; w < W; w++) id[j][w] = src[w];
			}
#pragma unroll
			for (int j = 0; j < kSel; j++)
			{
				uint64_t m = ~(uint64_t)0;
#pragma unroll
				for (int w = 0; w < W; w++)
					m &= *(const uint64_t*)((const char*)M + (id[j][w] & 0xffffu))
						& *(const uint64_t*)((const char*)M + (id[j][w] >> 16));
				const uint64_t al = __builtin_amdgcn_ballot_w64(m != 0);
				if (lane == i + j && i + j < nb)
				{
					mlo = (uint32_t)al;
					mhi = (uint32_t)(al >> 32);
				}
			}
		}
	};
	switch (ldc(&sd->hstride))
	{
	case 2: select(std::integral_constant<int, 1>()); break;
	case 4: select(std::integral_constant<int, 2>()); break;
	case 6: select(std::integral_constant<int, 3>()); break;
	default: select(std::integral_constant<int, 4>()); break;
	}
}

} // namespace hddm_lb
