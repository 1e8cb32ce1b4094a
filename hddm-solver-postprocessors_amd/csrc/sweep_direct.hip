// Direct sweep of the LinearBasis forward (gfx950), F32 and FP64, for states
// whose hats do not fit the LDS as a table of values.
//
// One workgroup of eight waves takes one 64-point block against one range of
// the state's nodes (trie order) and up to four 32-dof tiles. Per item:
//   1. the block's coordinates go to LDS, one row of 64 per dimension;
//   2. every distinct hat of the state (a few hundred) is evaluated once at
//      the block's points; the 64-bit mask of the points inside its support
//      goes to LDS;
//   3. the waves take windows of 64 nodes in turn. One node per lane, the
//      masks of a node's hats are ANDed: the node is alive if a point is
//      left. 64 nodes cost a few loads and a ballot, where a walk that tests
//      prefix products visits them one by one;
//   4. in rounds, every wave forms the basis of a part of its window (32
//      nodes in F32, 16 in FP64: 8 KB) into LDS, one point per lane, in trie
//      order: P[t + 1] = P[t] * phi, the prefix products in registers under
//      GPR indexing (a node's parents are nodes before it, alive when it is);
//   5. every wave contracts one dof tile against the basis of its share of
//      the waves. F32 and FP64 MFMAs run on the vector unit itself, so the
//      basis, some 75 issue cycles a node against the MFMA's 64 (F32) or 128
//      (FP64), is formed once for all tiles and not once per tile;
//   6. the sums of waves of one tile are added through LDS, in order.
//
// Contraction, one wave, 64 points x 32 dofs:
//   F32   v_mfma_f32_32x32x1_2b_f32: one alive node per step, the two blocks
//         of which are the two halves of the 64 points, so lane p holds the B
//         operand of point p as the basis was formed; folded into FP64 after
//         every 32 nodes of the layout;
//   FP64  v_mfma_f64_16x16x4f64: four nodes per step, read from LDS in its
//         operand layout; a 16-point column tile where all four nodes are
//         zero is skipped.
// Groups of nodes, folds and which wave adds which are fixed by the layout,
// and what is skipped is exactly zero, so a point's result does not depend on
// the points it shares a block with (its last bits do on how many workgroups
// share a block's nodes, see split_groups).
//
// Measured (ms; walking sweeps -> every wave forming the basis of its own tile
// -> here): D=59 / 281,077 nodes / 128 dofs / 16,384 points F32 32.5 -> 19.7 ->
// 15.5, FP64 82.3 -> 27.8 -> 21.7. At D=59 85 % of the nodes meet a point of
// any block; their MFMAs are 6.4 ms of the F32 time, forming the basis 3.1, the
// folds 1.0; 40 % of the wave cycles wait (barriers of the rounds, LDS, surplus
// rows; with three or four units' rows on their way 15.8 and more).
#include "sweep_common.h"
#include "kernels.h"

#include <type_traits>

namespace hddm_lb {

namespace {

constexpr int kDW = kDirectWaves;
constexpr int kBasisBytes = 8192;               // per wave
constexpr int kAhead = 2;                       // units whose surplus rows are on their way

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

// A node that is not alive gets this for the high word of -j, an infinity: its
// hat, and so its basis, is zero at every point (a large number is met by a
// coordinate as large).
constexpr uint32_t kFarHigh = 0xfff00000u;

// The contraction of a unit of eight nodes.
template <int PREC> struct Contract;

template <>
struct Contract<HDDM_LB_F32>
{
	typedef float B;                // basis values as the contraction takes them
	static constexpr int kSub = 32; // nodes per wave and round
	static constexpr int kAcc = 32;
	struct S { float v[8]; };
	fv32_t acc;
	double sum[32];
	int chunk;                      // 32-node chunk acc sums
	const float* base;
	int off[8];

	__device__ __forceinline__ void init(const StateDesc* sd, int DP, int tile, int lane)
	{
#pragma unroll
		for (int r = 0; r < 32; r++) sum[r] = 0.0;
		zero();
		chunk = -1;
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
		for (int r = 0; r < 32; r++) sum[r] += (double)acc[r];
	}

	__device__ __forceinline__ void begin(int n0)
	{
		if ((n0 >> 5) != chunk)
		{
			if (chunk >= 0) { fold(); zero(); }
			chunk = n0 >> 5;
		}
	}

	// the unit's basis: rows of 64 points (dead nodes are left out)
	template <bool>
	__device__ __forceinline__ void contract(const S& s, const B* basis, uint32_t mask, int lane)
	{
		float b[8];
#pragma unroll
		for (int k = 0; k < 8; k++) b[k] = basis[k * kWave + lane];
#pragma unroll
		for (int k = 0; k < 8; k++)
			if ((mask >> k) & 1u) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(s.v[k], b[k], acc, 0, 0, 0);
	}

	__device__ __forceinline__ void finish() { fold(); }
	__device__ __forceinline__ double get(int r) const { return sum[r]; }

	// D of v_mfma_f32_32x32x1_2b: block t in registers 16 t .., register r
	// of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4 (the dof) and column
	// l % 32 (the point)
	__device__ __forceinline__ static int point(int i, int lane) { return 32 * (i >> 4) + (lane & 31); }
	__device__ __forceinline__ static int dof(int i, int lane) { return 8 * ((i & 15) >> 2) + 4 * (lane >> 5) + (i & 3); }
};

template <>
struct Contract<HDDM_LB_FP64>
{
	typedef double B;
	static constexpr int kSub = 16;
	static constexpr int kAcc = 32;
	struct S { double v[2][2]; };   // [quad][16-dof half]: S[node 4 q + lane / 16][dof 16 h + lane % 16]
	dv4_t acc[2][4];                // [16-dof half][16-point tile]
	const double* base;
	int off;

	__device__ __forceinline__ void init(const StateDesc* sd, int DP, int tile, int lane)
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

	template <bool ODD>
	__device__ __forceinline__ void contract(const S& s, const B* basis, uint32_t mask, int lane)
	{
		const double* row = basis + (lane >> 4) * kWave + (lane & 15);
#pragma unroll
		for (int q = 0; q < 2; q++)
			if (const uint32_t qm = (mask >> (4 * q)) & 15u)
			{
				// dead nodes of the four: their basis is 0, and so is what stands
				// for their surplus (the selects cost 4 % at D=59: 17.7 and 18.4 ms
				// of a 12,345 point forward)
				double s0 = s.v[q][0], s1 = s.v[q][1];
				if (ODD && qm != 15u)
				{
					const bool live = (qm >> (lane >> 4)) & 1u;
					s0 = live ? s0 : 0.0;
					s1 = live ? s1 : 0.0;
				}
				double b[4];
#pragma unroll
				for (int p = 0; p < 4; p++) b[p] = row[4 * q * kWave + 16 * p];
#pragma unroll
				for (int p = 0; p < 4; p++)
					if (__builtin_amdgcn_ballot_w64(b[p] != 0.0))
					{
						acc[0][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(s0, b[p], acc[0][p], 0, 0, 0);
						acc[1][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(s1, b[p], acc[1][p], 0, 0, 0);
					}
			}
	}

	__device__ __forceinline__ void finish() {}
	__device__ __forceinline__ double get(int r) const { return acc[r >> 4][(r >> 2) & 3][r & 3]; }

	// D[i][j] in lane j + 16 (i % 4), element i / 4: i the dof, j the point
	__device__ __forceinline__ static int point(int i, int lane) { return 16 * ((i >> 2) & 3) + (lane & 15); }
	__device__ __forceinline__ static int dof(int i, int lane) { return 16 * (i >> 4) + 4 * (i & 3) + (lane >> 4); }
};

} // namespace

// ODD: dead nodes' surpluses may be no numbers (FP64)
template <int PREC, bool ODD>
__global__ void __launch_bounds__(64 * kDW) __attribute__((amdgpu_waves_per_eu(2))) sweep_direct_kernel(SweepArgs a, int hats_max)
{
	extern __shared__ __attribute__((aligned(16))) double lds[];
	typedef Contract<PREC> C;
	typedef typename C::B B;
	constexpr int U = 8, kUnits = C::kSub / U;              // units per wave and round
	constexpr uint32_t kSubMask = C::kSub == 32 ? ~0u : (1u << C::kSub) - 1u;
	const int lane = threadIdx.x & 63;
	const int wave = uniform((int)(threadIdx.x >> 6));
	B* const basis = (B*)lds;                               // [wave][node of the round][point]
	double* const X = lds + kDW * kBasisBytes / 8;
	char* const xl = (char*)X + lane * 8;                   // the lane's column of the coordinate rows
	uint64_t* const M = (uint64_t*)(X + (size_t)a.dim * kWave);
	int64_t* const slot = (int64_t*)(M + hats_max);
	uint8_t* const alive = (uint8_t*)(slot + 1);            // [wave][unit]: a round's alive nodes
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
			if (item < ib + nb * ldc(&a.plans[si].nseg)) { s = si; local = item - ib; nblk = nb; break; }
		}
		const StateDesc* sd = a.states + s;
		const StatePlan* pl = a.plans + s;
		const int64_t seg = local / nblk, blk = local - seg * nblk;
		const int dofs = ldc(&sd->dofs), DP = ldc(&sd->dofs_pad);
		const int nno = ldc(&sd->nno);
		const int tiles = DP >> 5;
		if (a.dt_base >= tiles) continue;
		const int64_t start = ldc(&pl->start) + blk * kWave, count = ldc(&pl->count);
		const int64_t rem = count - blk * kWave;
		const int np = rem < kWave ? (int)rem : kWave;
		const uint32_t orig = a.perm[start + (lane < np ? lane : np - 1)];
		const double* xrow = a.x + (int64_t)orig * a.ldx;
		for (int d = wave; d < a.dim; d += kDW) *(double*)(xl + d * (kWave * 8)) = xrow[d];
		__syncthreads();
		// the points inside each hat's support
		{
			const int hats = ldc(&sd->hats);
			const u4_t* ht = (const u4_t*)ldc(&sd->hat);
			const uint64_t valid = np < kWave ? ((uint64_t)1 << np) - 1 : ~(uint64_t)0;
			if (threadIdx.x == 0) { M[kHatAll] = valid; M[kHatNone] = 0; }
			// four hats at a time (the last group repeats its first hat)
			for (int h = kHatFirst + wave; h < hats; h += 4 * kDW)
			{
				uint64_t in[4];
				int at[4];
#pragma unroll
				for (int j = 0; j < 4; j++)
				{
					at[j] = h + j * kDW < hats ? h + j * kDW : h;
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

		// the wave's tile, and the waves whose basis it contracts
		const int tw = min(tiles - a.dt_base, 4);
		const int parts = kDW / tw;
		const int part = wave / tw, tile = a.dt_base + wave - part * tw;
		const bool on = part < parts;
		const int f0 = kDW * part / parts, f1 = kDW * (part + 1) / parts;
		const int nwin = (nno + kWin - 1) / kWin;
		const int nseg = (int)ldc(&pl->nseg);
		const int s0 = (int)((int64_t)nwin * seg / nseg), s1 = (int)((int64_t)nwin * (seg + 1) / nseg);
		const int turns = (s1 - s0 + kDW - 1) / kDW;        // windows s0 + wave + kDW i

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
		C c;
		c.init(sd, DP, tile, lane);

		for (int tb = 0; tb < turns; tb += kWave)
		{
			// selection: the alive nodes of the wave's window of turn tb + i as
			// lane i of (mlo, mhi)
			const int first = s0 + wave + tb * kDW;
			const int nb = min(kWave, (s1 - first + kDW - 1) / kDW);   // <= 0: no window
			uint32_t mlo = 0, mhi = 0;
			auto select = [&](auto words) {
				constexpr int W = decltype(words)::value;   // pairs of hat ids per node
				constexpr int kSel = 16 / W < 8 ? 16 / W : 8;   // windows in flight
				const uint32_t* hid = (const uint32_t*)ldc(&sd->hid) + ((size_t)first * kWin + lane) * W;
#pragma unroll 1
				for (int i = 0; i < nb; i += kSel)
				{
					uint32_t id[kSel][W];
#pragma unroll
					for (int j = 0; j < kSel; j++)
					{
						const uint32_t* src = hid + (size_t)(min(i + j, nb - 1) * kDW) * (kWin * W);
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
			if (a.stats)
			{
				// statistics mode: alive nodes, their chunks (F32) or units
				// (FP64), F32 MFMAs
				uint32_t nodes = (uint32_t)__popc(mlo) + (uint32_t)__popc(mhi), ch = 0;
				for (int o = 0; o < 32; o += C::kSub == 32 ? 32 : U)
				{
					const uint32_t um = C::kSub == 32 ? ~0u : 0xffu << o;
					ch += ((mlo & um) != 0u) + ((mhi & um) != 0u);
				}
				for (int off = 32; off; off >>= 1)
				{
					nodes += __shfl_xor(nodes, off, 64);
					ch += __shfl_xor(ch, off, 64);
				}
				if (lane == 0)
				{
					atomicAdd(&a.stats[0], (unsigned long long)nodes);
					atomicAdd(&a.stats[2], (unsigned long long)ch);
					if (PREC == HDDM_LB_F32) atomicAdd(&a.stats[4], (unsigned long long)nodes * tw);
				}
			}

			const int rounds = min(kWave, turns - tb) * (kWin / C::kSub);
			bool ahead = false;                             // the products above the window are there
#pragma unroll 1
			for (int r = 0; r < rounds; r++)
			{
				const int i = r / (kWin / C::kSub), sub = r % (kWin / C::kSub);
				const uint64_t m64 = ((uint64_t)__builtin_amdgcn_readlane(mhi, i) << 32) | (uint32_t)__builtin_amdgcn_readlane(mlo, i);
				const uint32_t mask = (uint32_t)(m64 >> (sub * C::kSub)) & kSubMask;
				const int wn = (first + i * kDW) * kWin, n0 = wn + sub * C::kSub;
				if (sub == 0) ahead = false;
				if (tw > 1) __syncthreads();                // the round before has been contracted
				else wave_lds_order();
				if (lane < kUnits) alive[wave * kUnits + lane] = (uint8_t)(mask >> (8 * lane));
				if (mask)
				{
					if (!ahead)
					{
						const uint32_t r0 = ldc((const uint32_t*)recs + (size_t)wn * 2);
						if (!(r0 & kRecRoot)) (void)path(wn, (int)((r0 & kRecDepth2) >> 1));
						ahead = true;
					}
					// Units with a node alive; while one is computed the next one's
					// records load. Those come through the scalar cache, out of
					// order with LDS reads, so they are requested only after the
					// unit's coordinates have been read: a wait for those would
					// wait for the records too.
					uint32_t left = mask;
					int o = __builtin_ctz(left) & ~(U - 1);
					uv16_t rec = ldc(recs + (size_t)((n0 + o) >> 3));
#pragma unroll 1
					for (;;)
					{
						const uint32_t um = (left >> o) & 0xffu;
						left &= ~(0xffu << o);
						double x[U];
#pragma unroll
						for (int k = 0; k < U; k++) x[k] = *(const double*)(xl + (rec[2 * k] & kRecRow));
						__builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
						__builtin_amdgcn_sched_barrier(0);
						const int no = left ? __builtin_ctz(left) & ~(U - 1) : o;
						const uv16_t nrec = ldc(recs + (size_t)((n0 + no) >> 3));
						__builtin_amdgcn_sched_barrier(0);
						B* const out = basis + (size_t)(wave * C::kSub + o) * kWave + lane;
						B b[U];
						if (rec[0] & kRecSpecial)
						{
							// rare: the root, or a node with a prefix that is no node;
							// the whole path of every node
#pragma unroll
							for (int k = 0; k < U; k++) b[k] = (B)0;
#pragma unroll 1
							for (uint32_t m = um; m; m &= m - 1)
							{
								const int k = __builtin_ctz(m);
								const uint32_t r0 = ldc((const uint32_t*)recs + 2 * (size_t)(n0 + o + k));
								const double p = path(n0 + o + k, r0 & kRecRoot ? 0 : (int)((r0 & kRecDepth2) >> 1) + 1);
#pragma unroll
								for (int j = 0; j < U; j++) b[j] = k == j ? (B)p : b[j];
							}
						}
						else
						{
							// all hats before the products: independent chains
#pragma unroll
							for (int k = 0; k < U; k++)
								x[k] = hat(x[k], f64_from_high(rec[2 * k] & kRecIhi), f64_from_high((um >> k) & 1u ? rec[2 * k + 1] : kFarHigh));
#pragma unroll
							for (int k = 0; k < U; k += 4)
								mulp4(P, rec[2 * k], rec[2 * k + 2], rec[2 * k + 4], rec[2 * k + 6], x[k], x[k + 1], x[k + 2], x[k + 3],
									b[k], b[k + 1], b[k + 2], b[k + 3]);
						}
#pragma unroll
						for (int k = 0; k < U; k++) out[k * kWave] = b[k];
						if (!left) break;
						o = no;
						rec = nrec;
					}
				}
				if (tw > 1) __syncthreads();                // the round's basis is there
				else wave_lds_order();
				if (!on) continue;
				// The units of this wave's share, in node order; while one is
				// contracted the surplus rows of the next ones load.
				const uint32_t av = lane < (f1 - f0) * kUnits ? alive[f0 * kUnits + lane] : 0u;
				uint64_t units = __builtin_amdgcn_ballot_w64(av != 0u);
				if (!units) continue;
				const int wfirst = s0 + f0 + (tb + i) * kDW;
				auto node = [&](int u) { return (wfirst + u / kUnits) * kWin + sub * C::kSub + (u % kUnits) * U; };
				// (past the last unit its rows load again: with no branch around
				// the loads, a wait can leave the later ones on their way)
				typename C::S sb[kAhead];
				int j[kAhead], at = 0;
				uint32_t um[kAhead];
				auto next = [&](int k) {
					at = units ? __builtin_ctzll(units) : at;
					um[k] = units ? __builtin_amdgcn_readlane(av, at) : 0u;
					units &= units - 1;
					j[k] = at;
					c.load(sb[k], node(at), DP);
				};
#pragma unroll
				for (int k = 0; k < kAhead; k++) next(k);
#pragma unroll 1
				do
				{
#pragma unroll
					for (int k = 0; k < kAhead; k++)
					{
						c.begin(node(j[k]));
						c.template contract<ODD>(sb[k], basis + (size_t)(f0 * kUnits + j[k]) * U * kWave, um[k], lane);
						__builtin_amdgcn_sched_barrier(0);
						next(k);
						__builtin_amdgcn_sched_barrier(0);
					}
				} while (um[0]);
			}
		}
		c.finish();

		// the parts' sums, in order, through LDS (the basis is done with)
		double* const buf = lds + (size_t)(tile - a.dt_base) * C::kAcc * kWave + lane;
		for (int p = 0; p + 1 < parts; p++)
		{
			__syncthreads();
			if (part == p)
			{
#pragma unroll
				for (int r = 0; r < C::kAcc; r++) buf[r * kWave] = p ? buf[r * kWave] + c.get(r) : c.get(r);
			}
		}
		if (a.stats && threadIdx.x == 0) atomicAdd(&a.stats[3], 1ull);
		__syncthreads();
		if (part == parts - 1)
		{
			const bool split = nseg > 1;
			double* const part_s = a.partial + ldc(&pl->partial_base) + (seg * count + blk * kWave) * DP;
#pragma unroll
			for (int i0 = 0; i0 < C::kAcc; i0 += 4)
			{
				const int qp = C::point(i0, lane);
				const uint32_t oq = (uint32_t)__shfl((int)orig, qp, 64);
				double* out = split ? part_s + (int64_t)qp * DP : a.y + (int64_t)oq * a.ldy;
#pragma unroll
				for (int i = i0; i < i0 + 4; i++)
				{
					const double v = parts > 1 ? buf[i * kWave] + c.get(i) : c.get(i);
					const int dof = 32 * tile + C::dof(i, lane);
					if (qp < np && dof < dofs) out[dof] = v;
				}
			}
		}
	}
}

size_t sweep_direct_lds_bytes(int dim, int hats_max)
{
	return (size_t)kDW * kBasisBytes + (size_t)dim * kWave * 8 + (size_t)hats_max * 8 + 8 + 4 * kDW;
}

const void* sweep_direct_kernel_ptr(int prec, bool odd)
{
	if (prec == HDDM_LB_FP64)
		return odd ? (const void*)&sweep_direct_kernel<HDDM_LB_FP64, true> : (const void*)&sweep_direct_kernel<HDDM_LB_FP64, false>;
	if (prec == HDDM_LB_F32) return (const void*)&sweep_direct_kernel<HDDM_LB_F32, false>;
	return nullptr;
}

hipError_t launch_sweep_direct(const void* kern, int grid, int waves, size_t lds, const SweepArgs& args, int hats_max, hipStream_t st)
{
	void* params[] = { (void*)&args, (void*)&hats_max };
	return hipLaunchKernel(kern, dim3(grid), dim3(waves * kWave), params, lds, st);
}

} // namespace hddm_lb
