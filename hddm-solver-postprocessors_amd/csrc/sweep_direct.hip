// Direct sweep of the LinearBasis forward (gfx950).
//
// One workgroup takes one 64-point block against one range of the state's
// nodes (trie order); each of its waves contracts one 32-dof tile (waves that
// a narrow state leaves over take ranges of their own). Per item:
//   1. the block's coordinates go to LDS, one row of 64 per dimension;
//   2. every distinct hat of the state (a few hundred) is evaluated once at
//      the block's points; the 64-bit mask of the points inside its support
//      goes to LDS;
//   3. one node per lane, the masks of a node's hats are ANDed: the node is
//      alive if a point is left. 64 nodes cost a few loads and a ballot,
//      where a walk that tests prefix products visits them one by one;
//   4. the alive nodes' basis values are formed, one point per lane, in trie
//      order: P[t + 1] = P[t] * phi, the prefix products in registers under
//      GPR indexing (a node's parents are nodes before it, alive when it
//      is). Each value is an MFMA operand as it stands.
// Nothing in 4. decides which node comes next, so records and surplus rows
// of the next eight nodes load while eight are computed, and the eight hats
// are independent of each other.
//
// Contraction, one wave, 64 points x 32 dofs:
//   F32   v_mfma_f32_32x32x1_2b_f32: one node per step, the two blocks of
//         which are the two halves of the 64 points, so lane p holds the B
//         operand of point p as the basis was formed; folded into FP64 after
//         every 32 nodes of the layout;
//   FP64  v_mfma_f64_16x16x4f64: four nodes per step, brought from one point
//         per lane to its layout by two rounds of row swaps; a 16-point
//         column tile where all four nodes are zero is skipped;
//   F16X2, BF16X3  as the walking sweep, 16 nodes per step.
// Groups of nodes and folds are fixed by the layout, and what is skipped is
// exactly zero, so a point's result does not depend on the points it shares
// a block with.
//
// Measured against the walking sweeps (ms, before -> here): D=59 / 281,077
// nodes / 128 dofs / 16,384 points F32 32.3 -> 19.7, FP64 82.1 -> 27.8; D=24 /
// 12,011 nodes / 128 dofs / 30,011 points F16X2 6.0 -> 1.6, BF16X3 7.3 -> 1.8.
// At D=59 some 70 % of the nodes meet a point of any block, so nearly every
// node costs its hat, its product and its MFMAs: the vector unit's issue.
#include "sweep_common.h"
#include "kernels.h"
#include "contract.h"

#include <type_traits>

namespace hddm_lb {

namespace {

typedef double dv4_t __attribute__((ext_vector_type(4)));
typedef float fv32_t __attribute__((ext_vector_type(32)));
typedef uint32_t uv16_t __attribute__((ext_vector_type(16)));

// The prefix products of the current trie path: P[t] is the product of its
// first t factors (t up to 15). The statements below pin them to v[64:95],
// which GPR indexing needs; it writes m0, where the compiler keeps nothing.
typedef double dv16_t __attribute__((ext_vector_type(16)));

// P[t + 1] = P[t] * F, T = 2 t (its low 8 bits): one multiply whose source
// and destination are both indexed.
#define HDDM_MULP(T, F) \
	"s_set_gpr_idx_on " T ", gpr_idx(SRC0,DST)\n" \
	"v_mul_f64 v[66:67], v[64:65], " F "\n"
#define HDDM_OUT64(B) "s_set_gpr_idx_mode gpr_idx(SRC0)\n" "v_mov_b64 " B ", v[66:67]\n"
#define HDDM_OUT32(B) "s_set_gpr_idx_mode gpr_idx(SRC0)\n" "v_cvt_f32_f64 " B ", v[66:67]\n"

__device__ __forceinline__ double mulp(dv16_t& P, uint32_t t2, double phi)
{
	double b;
	asm(HDDM_MULP("%[t]", "%[f]") HDDM_OUT64("%[b]") "s_set_gpr_idx_off\n"
		: [b] "=&v"(b), "+{v[64:95]}"(P) : [t] "s"(t2), [f] "v"(phi) : "m0");
	return b;
}

// Four nodes in trie order, the products returned in b, as floats or doubles
// (the wait states: the instructions that take them, row swaps and MFMAs, do
// not see them written by a VALU instruction). A node that is not alive may
// find another path's product at its depth: its hat is zero, and its children
// are not alive either.
#define HDDM_MULP4(OUT) \
	asm(HDDM_MULP("%[t0]", "%[f0]") OUT("%[b0]") HDDM_MULP("%[t1]", "%[f1]") OUT("%[b1]") \
		HDDM_MULP("%[t2]", "%[f2]") OUT("%[b2]") HDDM_MULP("%[t3]", "%[f3]") OUT("%[b3]") \
		"s_set_gpr_idx_off\n" "s_nop 1\n" \
		: [b0] "=&v"(b0), [b1] "=&v"(b1), [b2] "=&v"(b2), [b3] "=&v"(b3), "+{v[64:95]}"(P) \
		: [t0] "s"(r0 & kRecDepth2), [t1] "s"(r1 & kRecDepth2), [t2] "s"(r2 & kRecDepth2), [t3] "s"(r3 & kRecDepth2), \
		  [f0] "v"(f0), [f1] "v"(f1), [f2] "v"(f2), [f3] "v"(f3) : "m0")

template <typename B>
__device__ __forceinline__ void mulp4(dv16_t& P, uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3,
	double f0, double f1, double f2, double f3, B& b0, B& b1, B& b2, B& b3)
{
	if constexpr (sizeof(B) == 8) HDDM_MULP4(HDDM_OUT64);
	else HDDM_MULP4(HDDM_OUT32);
}
#undef HDDM_MULP
#undef HDDM_MULP4
#undef HDDM_OUT64
#undef HDDM_OUT32

// max(0, 1 - |x i - j|)
__device__ __forceinline__ double hat(double x, double i, double nj)
{
	return fmax(1.0 - fabs(fma(x, i, nj)), 0.0);
}

// A node that is not alive gets this for the high word of -j (-1e300): its
// hat, and so its basis, is zero at every point.
constexpr uint32_t kFarHigh = 0xfe37e43cu;

// The surplus operands of a unit of kU nodes and its contraction.
template <int PREC> struct Contract;

template <>
struct Contract<HDDM_LB_F32>
{
	static constexpr int kU = 8;
	typedef float B;                // basis values as the contraction takes them
	struct S { float v[8]; };
	fv32_t acc;
	double acc64[32];
	int chunk;                      // 32-node chunk acc sums
	const float* base;
	int off[8];

	__device__ __forceinline__ void init(const StateDesc* sd, int DP, int tile, int lane, int n0)
	{
#pragma unroll
		for (int r = 0; r < 32; r++) acc64[r] = 0.0;
		zero();
		chunk = n0 >> 5;
		base = ldc(&sd->s32r) + 32 * tile;
#pragma unroll
		for (int k = 0; k < 8; k++) off[k] = k * DP + (lane & 31);
	}

	// one MFMA of zeros instead of 32 moves
	__device__ __forceinline__ void zero()
	{
		fv32_t z;
#pragma unroll
		for (int r = 0; r < 32; r++) z[r] = 0.0f;
		acc = __builtin_amdgcn_mfma_f32_32x32x1f32(0.0f, 0.0f, z, 0, 0, 0);
	}

	__device__ __forceinline__ void load(S& s, int n0, int DP)
	{
		const float* row = base + (size_t)n0 * DP;
#pragma unroll
		for (int k = 0; k < 8; k++) s.v[k] = row[off[k]];
	}

	__device__ __forceinline__ void fold()
	{
#pragma unroll
		for (int r = 0; r < 32; r++) acc64[r] += (double)acc[r];
	}

	__device__ __forceinline__ void begin(int n0)
	{
		if ((n0 >> 5) != chunk)
		{
			fold();
			zero();
			chunk = n0 >> 5;
		}
	}

	__device__ __forceinline__ void contract(const S& s, const float (&b)[8])
	{
#pragma unroll
		for (int k = 0; k < 8; k++) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(s.v[k], b[k], acc, 0, 0, 0);
	}

	__device__ __forceinline__ void finish(const StateDesc*, int, int) { fold(); }

	// D of v_mfma_f32_32x32x1_2b: block t in registers 16 t .., register r
	// of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4 (the dof) and column
	// l % 32 (the point).
	template <typename F>
	__device__ __forceinline__ void store(F out, int lane)
	{
#pragma unroll
		for (int t = 0; t < 2; t++)
		{
			double v[16];
#pragma unroll
			for (int r = 0; r < 16; r++) v[r] = acc64[16 * t + r];
			out(32 * t + (lane & 31), lane, v);
		}
	}
	static constexpr bool kRows32 = true;
};

template <>
struct Contract<HDDM_LB_FP64>
{
	static constexpr int kU = 8;
	typedef double B;
	struct S { double v[2][2]; };   // [quad][16-dof half]: S[node 4 q + lane / 16][dof 16 h + lane % 16]
	dv4_t acc[2][4];                // [16-dof half][16-point tile]

	const double* base;
	int off;

	__device__ __forceinline__ void init(const StateDesc* sd, int DP, int tile, int lane, int)
	{
#pragma unroll
		for (int h = 0; h < 2; h++)
#pragma unroll
			for (int p = 0; p < 4; p++) acc[h][p] = dv4_t{ 0.0, 0.0, 0.0, 0.0 };
		base = ldc(&sd->s64) + 32 * tile;
		off = (lane >> 4) * DP + (lane & 15);
	}

	__device__ __forceinline__ void load(S& s, int n0, int DP)
	{
		const double* row = base + (size_t)n0 * DP;
#pragma unroll
		for (int q = 0; q < 2; q++, row += 4 * (size_t)DP)
#pragma unroll
			for (int h = 0; h < 2; h++) s.v[q][h] = row[off + 16 * h];
	}

	__device__ __forceinline__ void begin(int) {}
	__device__ __forceinline__ static void swap32(double& a, double& b)
	{
		auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
		auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
		a = __hiloint2double((int)hi[0], (int)lo[0]);
		b = __hiloint2double((int)hi[1], (int)lo[1]);
	}

	__device__ __forceinline__ static void swap16(double& a, double& b)
	{
		auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
		auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
		a = __hiloint2double((int)hi[0], (int)lo[0]);
		b = __hiloint2double((int)hi[1], (int)lo[1]);
	}

	__device__ __forceinline__ void contract(const S& s, const double (&bv)[8])
	{
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			double b0 = bv[4 * q], b1 = bv[4 * q + 1], b2 = bv[4 * q + 2], b3 = bv[4 * q + 3];
			const uint64_t nz = __builtin_amdgcn_ballot_w64((b0 != 0.0) | (b1 != 0.0) | (b2 != 0.0) | (b3 != 0.0));
			if (nz)
			{
				// rows of 16 lanes: from [node][row = point tile] to [point tile][row = node]
				swap32(b0, b2);
				swap32(b1, b3);
				swap16(b0, b1);
				swap16(b2, b3);
				const double b[4] = { b0, b1, b2, b3 };
#pragma unroll
				for (int p = 0; p < 4; p++)
					if ((nz >> (16 * p)) & 0xffffull)
					{
						acc[0][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.v[q][0], b[p], acc[0][p], 0, 0, 0);
						acc[1][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.v[q][1], b[p], acc[1][p], 0, 0, 0);
					}
			}
		}
	}

	__device__ __forceinline__ void finish(const StateDesc*, int, int) {}
	static constexpr bool kRows32 = false;
};

// F16X2 and BF16X3: the operand split and products of the walking sweep.
template <int PREC>
struct ContractSplit
{
	static constexpr int kU = 16;
	static constexpr int kTerms = PREC == HDDM_LB_F16X2 ? 2 : 3;
	typedef float B;
	typedef SOperands<PREC, 1> S;
	double acc64[2][16];
	const uint16_t* base;           // rows of 16 nodes: [chunk][term][dof][16]
	int off;

	__device__ __forceinline__ void init(const StateDesc* sd, int, int tile, int lane, int)
	{
#pragma unroll
		for (int t = 0; t < 2; t++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc64[t][r] = 0.0;
		base = (PREC == HDDM_LB_F16X2 ? ldc(&sd->s16) : ldc(&sd->sbf)) + 32 * tile * kChunk;
		off = (lane & 31) * kChunk + (lane >> 5) * 8;
	}

	__device__ __forceinline__ void load(S& s, int n0, int DP)
	{
		const uint16_t* sc = base + (size_t)(n0 >> 4) * kTerms * DP * kChunk;
#pragma unroll
		for (int t = 0; t < kTerms; t++, sc += (size_t)DP * kChunk) s.A[0][t] = *(const typename S::V*)(sc + off);
	}

	__device__ __forceinline__ void begin(int) {}

	__device__ __forceinline__ void contract(const S& s, const float (&b)[16])
	{
		f16_t acc[2][1];
#pragma unroll
		for (int t = 0; t < 2; t++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc[t][0][r] = 0.0f;
		contract_chunk<PREC, 1>(s, 1, b, acc);
#pragma unroll
		for (int t = 0; t < 2; t++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc64[t][r] += (double)acc[t][0][r];
	}

	__device__ __forceinline__ void finish(const StateDesc* sd, int tile, int lane)
	{
		if constexpr (PREC == HDDM_LB_F16X2)
		{
			const double* iscale = ldc(&sd->iscale) + 32 * tile + 4 * (lane >> 5);
#pragma unroll
			for (int r = 0; r < 16; r++)
			{
				const double f = iscale[8 * (r >> 2) + (r & 3)] * (1.0 / kBScale);
				acc64[0][r] *= f;
				acc64[1][r] *= f;
			}
		}
	}

	template <typename F>
	__device__ __forceinline__ void store(F out, int lane)
	{
#pragma unroll
		for (int t = 0; t < 2; t++) out(32 * t + (lane & 31), lane, acc64[t]);
	}
	static constexpr bool kRows32 = true;
};
template <> struct Contract<HDDM_LB_F16X2> : ContractSplit<HDDM_LB_F16X2> {};
template <> struct Contract<HDDM_LB_BF16X3> : ContractSplit<HDDM_LB_BF16X3> {};

} // namespace

template <int PREC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) sweep_direct_kernel(SweepArgs a, int hats_max)
{
	extern __shared__ __attribute__((aligned(16))) double lds[];
	typedef Contract<PREC> C;
	constexpr int U = C::kU;
	constexpr uint64_t UM = ((uint64_t)1 << U) - 1;
	const int lane = threadIdx.x & 63;
	const int wave = uniform((int)(threadIdx.x >> 6));
	const int nt = uniform((int)(blockDim.x >> 6));
	char* const xl = (char*)lds + lane * 8;                 // the lane's column of the coordinate rows
	uint64_t* const M = (uint64_t*)(lds + (size_t)a.dim * kWave);
	int64_t* const slot = (int64_t*)(M + hats_max);
	const int64_t nitems = ldc(&a.hdr->nitems);

	for (;;)
	{
		__syncthreads();
		if (threadIdx.x == 0) *slot = (int64_t)atomicAdd(&a.hdr->counter, 1ull);
		__syncthreads();
		const int64_t item = (int64_t)uniform64((uint64_t)*slot);
		if (item >= nitems) break;
		// items lie state by state in cost order, each state's segment-major
		int s = 0;
		int64_t local = 0, nblk = 1;
		for (int i = 0; i < a.nstates; i++)
		{
			const int si = ldc(&a.cost_order[i]);
			const int64_t ib = ldc(&a.plans[si].item_base);
			const int64_t nb = ldc(&a.plans[si].nblk);
			const int parts = direct_parts(ldc(&a.states[si].dofs_pad) >> 5, nt);
			const int64_t ng = (ldc(&a.plans[si].nseg) + parts - 1) / parts;
			if (item < ib + nb * ng) { s = si; local = item - ib; nblk = nb; break; }
		}
		const StateDesc* sd = a.states + s;
		const StatePlan* pl = a.plans + s;
		const int64_t group = local / nblk, blk = local - group * nblk;
		const int dofs = ldc(&sd->dofs), DP = ldc(&sd->dofs_pad);
		const int nno = ldc(&sd->nno);
		const int nseg = (int)ldc(&pl->nseg);
		const int tiles = DP >> 5;
		if (a.dt_base >= tiles) continue;
		const int64_t start = ldc(&pl->start) + blk * kWave, count = ldc(&pl->count);
		const int64_t rem = count - blk * kWave;
		const int np = rem < kWave ? (int)rem : kWave;
		const uint32_t orig = a.perm[start + (lane < np ? lane : np - 1)];
		const double* xrow = a.x + (int64_t)orig * a.ldx;
		for (int d = wave; d < a.dim; d += nt) *(double*)(xl + d * (kWave * 8)) = xrow[d];
		__syncthreads();
		// the points inside each hat's support
		{
			const int hats = ldc(&sd->hats);
			const u4_t* ht = (const u4_t*)ldc(&sd->hat);
			const uint64_t valid = np < kWave ? ((uint64_t)1 << np) - 1 : ~(uint64_t)0;
			if (threadIdx.x == 0) { M[kHatAll] = valid; M[kHatNone] = 0; }
			// four hats at a time (the last group repeats its first hat)
			for (int h = kHatFirst + wave; h < hats; h += 4 * nt)
			{
				uint64_t in[4];
				int at[4];
#pragma unroll
				for (int j = 0; j < 4; j++)
				{
					at[j] = h + j * nt < hats ? h + j * nt : h;
					const u4_t e = ldc(ht + at[j]);
					const double u = (*(const double*)(xl + e[0]) + f64_from_high(e[2])) * f64_from_high(e[1]);
					in[j] = __builtin_amdgcn_ballot_w64(fmax(1.0 - fabs(u), 0.0) > 0.0) & valid;
				}
				if (lane == 0)
				{
#pragma unroll
					for (int j = 0; j < 4; j++) M[at[j]] = in[j];
				}
			}
		}
		__syncthreads();

		const int tl = tiles < nt ? tiles : nt;
		const int part = wave / tl, tile = a.dt_base + wave - part * tl;
		const int seg = (int)group * direct_parts(tiles, nt) + part;
		if (part >= direct_parts(tiles, nt) || seg >= nseg || tile >= tiles) continue;
		const int nwin = (nno + kWin - 1) / kWin;
		const int w0 = (int)((int64_t)nwin * seg / nseg), w1 = (int)((int64_t)nwin * (seg + 1) / nseg);

		const uv16_t* const recs = (const uv16_t*)ldc(&sd->rec);
		const u4_t* const ftab = (const u4_t*)ldc(&sd->ftab);
		const int fs = (int)ldc(&sd->fstride);
		dv16_t P;
#pragma unroll
		for (int i = 0; i < 16; i++) P[i] = 1.0;
		// the products of node n's path up to factor t - 1
		auto path = [&](int n, int t) -> double {
			double p = 1.0;
#pragma unroll 1
			for (int f = 0; f < t; f++)
			{
				const u4_t e = ldc(ftab + (size_t)n * fs + f);
				const double u = (*(const double*)(xl + e[0] * 256u) + f64_from_high(e[2])) * f64_from_high(e[1]);
				p = mulp(P, 2u * (uint32_t)f, fmax(1.0 - fabs(u), 0.0));
			}
			return p;
		};
		if (w0 > 0)
		{
			const uint32_t r0 = ldc((const uint32_t*)recs + (size_t)w0 * kWin * 2);
			if (!(r0 & kRecRoot)) (void)path(w0 * kWin, (int)((r0 & kRecDepth2) >> 1));
		}
		C c;
		c.init(sd, DP, tile, lane, w0 * kWin);
		uint32_t st_nodes = 0, st_chunks = 0, st_mfma = 0;

		for (int wb = w0; wb < w1; wb += kWave)
		{
			// selection: the alive nodes of window wb + i as lane i of (mlo, mhi)
			const int nb = min(kWave, w1 - wb);
			uint32_t mlo = 0, mhi = 0;
			auto select = [&](auto words) {
				constexpr int W = decltype(words)::value;   // pairs of hat ids per node
				constexpr int kSel = 16 / W < 8 ? 16 / W : 8;   // windows in flight
				const uint32_t* hid = (const uint32_t*)ldc(&sd->hid) + ((size_t)wb * kWin + lane) * W;
#pragma unroll 1
				for (int i = 0; i < nb; i += kSel)
				{
					uint32_t id[kSel][W];
#pragma unroll
					for (int j = 0; j < kSel; j++)
					{
						const uint32_t* src = hid + (size_t)min(i + j, nb - 1) * kWin * W;
#pragma unroll
						for (int w = 0; w < W; w++) id[j][w] = src[w];
					}
#pragma unroll
					for (int j = 0; j < kSel; j++)
					{
						uint64_t m = ~(uint64_t)0;
#pragma unroll
						for (int w = 0; w < W; w++)
							m &= *(const uint64_t*)((const char*)M + (id[j][w] & 0xffffu)) & *(const uint64_t*)((const char*)M + (id[j][w] >> 16));
						const uint64_t al = __builtin_amdgcn_ballot_w64(m != 0);
						// lanes nb .. are never read as windows
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
			case 8: select(std::integral_constant<int, 4>()); break;
			default: select(std::integral_constant<int, 8>()); break;
			}

			// Units of U nodes with a node alive; while one is computed the next
			// one's surplus rows and records load. Records come through the
			// scalar cache, out of order with LDS reads, so they are requested
			// only after the unit's coordinates have been read: a wait for
			// those would wait for the records too.
			struct Unit { int n0; uint32_t mask; uv16_t rec[U / 8]; };
			uint64_t wm = __builtin_amdgcn_ballot_w64((mlo | mhi) != 0u), m64 = 0;
			int cw = 0;
			auto next = [&](Unit& u) -> bool {
				if (!m64)
				{
					if (!wm) return false;
					cw = __builtin_ctzll(wm);
					wm &= wm - 1;
					m64 = ((uint64_t)__builtin_amdgcn_readlane(mhi, cw) << 32) | (uint32_t)__builtin_amdgcn_readlane(mlo, cw);
				}
				const int o = __builtin_ctzll(m64) & ~(U - 1);
				u.mask = (uint32_t)((m64 >> o) & UM);
				m64 &= ~(UM << o);
				u.n0 = (wb + cw) * kWin + o;
#pragma unroll
				for (int r = 0; r < U / 8; r++) u.rec[r] = ldc(recs + (size_t)(u.n0 >> 3) + r);
				return true;
			};
			Unit u;
			typename C::S su;
			bool more = next(u);
			if (more) c.load(su, u.n0, DP);
#pragma unroll 1
			while (more)
			{
				double x[U];
#pragma unroll
				for (int k = 0; k < U; k++) x[k] = *(const double*)(xl + (u.rec[k / 8][2 * (k % 8)] & kRecRow));
				__builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
				__builtin_amdgcn_sched_barrier(0);
				Unit v = u;
				typename C::S sv;
				more = next(v);
				c.load(sv, v.n0, DP);
				__builtin_amdgcn_sched_barrier(0);
				c.begin(u.n0);
				typename C::B b[U];
				// all hats before the products: independent chains
#pragma unroll
				for (int k = 0; k < U; k++)
				{
					const uint32_t r0 = u.rec[k / 8][2 * (k % 8)], r1 = u.rec[k / 8][2 * (k % 8) + 1];
					x[k] = hat(x[k], f64_from_high(r0 & kRecIhi), f64_from_high((u.mask >> k) & 1u ? r1 : kFarHigh));
				}
				uint32_t special = 0;
#pragma unroll
				for (int r = 0; r < U / 8; r++) special |= u.rec[r][0];
				if (special & kRecSpecial)
				{
					// rare: the root, or a node with a prefix that is no node;
					// the whole path of every node
#pragma unroll
					for (int k = 0; k < U; k++) b[k] = (typename C::B)0;
#pragma unroll 1
					for (uint32_t m = u.mask; m; m &= m - 1)
					{
						const int k = __builtin_ctz(m);
						const uint32_t r0 = ldc((const uint32_t*)recs + 2 * (size_t)(u.n0 + k));
						const double p = path(u.n0 + k, r0 & kRecRoot ? 0 : (int)((r0 & kRecDepth2) >> 1) + 1);
#pragma unroll
						for (int j = 0; j < U; j++) b[j] = k == j ? (typename C::B)p : b[j];
					}
				}
				else
				{
#pragma unroll
					for (int k = 0; k < U; k += 4)
					{
						const uv16_t& r = u.rec[k / 8];
						const int j = 2 * (k % 8);
						mulp4(P, r[j], r[j + 2], r[j + 4], r[j + 6], x[k], x[k + 1], x[k + 2], x[k + 3],
							b[k], b[k + 1], b[k + 2], b[k + 3]);
					}
				}
				c.contract(su, b);
				u = v;
				su = sv;
			}
			if (a.stats)
			{
				// counted in a pass of its own (statistics mode only)
				uint32_t alive = (uint32_t)__popc(mlo) + (uint32_t)__popc(mhi);
				uint32_t ch = PREC == HDDM_LB_F32 ? (mlo != 0u) + (mhi != 0u) : 0u;
				if constexpr (PREC != HDDM_LB_F32)
					for (int o = 0; o < 32; o += U) ch += (((mlo >> o) & (uint32_t)UM) != 0u) + (((mhi >> o) & (uint32_t)UM) != 0u);
				for (int off = 32; off; off >>= 1)
				{
					alive += __shfl_xor(alive, off, 64);
					ch += __shfl_xor(ch, off, 64);
				}
				st_nodes += alive;
				st_chunks += ch;
				st_mfma += PREC == HDDM_LB_F32 ? alive : (PREC == HDDM_LB_F16X2 ? 6u * ch : (PREC == HDDM_LB_BF16X3 ? 12u * ch : 0u));
			}
		}

		c.finish(sd, tile, lane);
		const bool split = nseg > 1;
		double* const part_s = a.partial + ldc(&pl->partial_base) + ((int64_t)seg * count + blk * kWave) * DP;
		if constexpr (C::kRows32)
			c.store([&](int qp, int ln, const double (&v)[16]) {
				const uint32_t oq = (uint32_t)__shfl((int)orig, qp, 64);
				if (qp < np)
				{
					double* out = split ? part_s + (int64_t)qp * DP : a.y + (int64_t)oq * a.ldy;
#pragma unroll
					for (int r = 0; r < 16; r++)
					{
						const int dof = 32 * tile + 8 * (r >> 2) + 4 * (ln >> 5) + (r & 3);
						if (dof < dofs) out[dof] = v[r];
					}
				}
			}, lane);
		else
		{
			// D[i][j] in lane j + 16 (i % 4), element i / 4: i the dof, j the point
#pragma unroll
			for (int p = 0; p < 4; p++)
			{
				const int qp = 16 * p + (lane & 15);
				const uint32_t oq = (uint32_t)__shfl((int)orig, qp, 64);
				if (qp < np)
				{
					double* out = split ? part_s + (int64_t)qp * DP : a.y + (int64_t)oq * a.ldy;
#pragma unroll
					for (int h = 0; h < 2; h++)
#pragma unroll
						for (int e = 0; e < 4; e++)
						{
							const int dof = 32 * tile + 16 * h + 4 * e + (lane >> 4);
							if (dof < dofs) out[dof] = c.acc[h][p][e];
						}
				}
			}
		}
		if (a.stats && lane == 0)
		{
			if (tile == a.dt_base)
			{
				atomicAdd(&a.stats[0], (unsigned long long)st_nodes);
				atomicAdd(&a.stats[2], (unsigned long long)st_chunks);
				atomicAdd(&a.stats[3], 1ull);
			}
			atomicAdd(&a.stats[4], (unsigned long long)st_mfma);
		}
	}
}

size_t sweep_direct_lds_bytes(int dim, int hats_max)
{
	return (size_t)dim * kWave * 8 + (size_t)hats_max * 8 + 16;
}

const void* sweep_direct_kernel_ptr(int prec)
{
	switch (prec)
	{
	case HDDM_LB_FP64: return (const void*)&sweep_direct_kernel<HDDM_LB_FP64>;
	case HDDM_LB_F16X2: return (const void*)&sweep_direct_kernel<HDDM_LB_F16X2>;
	case HDDM_LB_BF16X3: return (const void*)&sweep_direct_kernel<HDDM_LB_BF16X3>;
	case HDDM_LB_F32: return (const void*)&sweep_direct_kernel<HDDM_LB_F32>;
	}
	return nullptr;
}

hipError_t launch_sweep_direct(const void* kern, int grid, int waves, size_t lds, const SweepArgs& args, int hats_max, hipStream_t st)
{
	void* params[] = { (void*)&args, (void*)&hats_max };
	return hipLaunchKernel(kern, dim3(grid), dim3(waves * kWave), params, lds, st);
}

} // namespace hddm_lb
