// Hat-table sweep of the LinearBasis forward (gfx950).
//
// One workgroup of kTW waves takes one 64-point block against one range of
// the state's nodes (trie order). Per item:
//   1. the block's coordinates go to LDS;
//   2. every distinct hat of the state is evaluated once at the block's
//      points: its values (one row of 64 doubles) and the 64-bit mask of the
//      points inside its support stay in LDS. A sparse grid has few: 182 for
//      60,010 nodes at D=16, 186 for 100,005 at D=20;
//   3. the waves share the range out (one 32-dof tile and one contiguous part
//      of the nodes each). One node per lane, the masks of a node's hats are
//      ANDed: the node is alive if a point is left. 64 nodes cost a few
//      loads and a ballot, where a walk that tests prefix products visits
//      them one by one;
//   4. the alive nodes of a 64-node window move together (one LDS permute)
//      and are formed eight at a time, one point per lane, in trie order:
//      P[t + 1] = P[t] * hat, the prefix products in registers under GPR
//      indexing (a node's parents are nodes before it, alive when it is);
//   5. the parts' sums are added through LDS, in order.
// F32 and FP64 MFMAs run on the vector unit itself: while one runs, no vector
// instruction issues on its SIMD (measured: v_mfma_f32_32x32x1_2b 64 cycles
// and FP64 arithmetic beside it take the sum of their times). So the aim of
// 3. and 4. is few instructions per node and no MFMA for a node that no point
// of the block meets; three waves per SIMD hide the latencies.
//
// Contraction, one wave, 64 points x 32 dofs:
//   F32   v_mfma_f32_32x32x1_2b_f32: one node per step, its two blocks are
//         the two halves of the 64 points, so lane p holds the B operand of
//         point p as the basis was formed; folded into FP64 after every 32
//         nodes of the layout;
//   FP64  v_mfma_f64_16x16x4f64: four alive nodes per step (the products of a
//         step are accumulated one after the other, so how nodes are grouped
//         does not change a bit), brought from one point per lane to its
//         layout by two rounds of row swaps; a 16-point column tile where all
//         four are zero is skipped.
// Skipped terms are exactly zero and folds are fixed by the layout, so a
// point's result does not depend on the points it shares a block with (its last
// bits do on how many workgroups share a block's nodes, see split_groups).
//
// Measured against the walking sweeps (ms, before -> here): D=16 / 60,010
// nodes / 32 dofs / 2^20 points F32 15.7 -> 14.4 and 100,003 points F32 2.58
// -> 2.03, FP64 4.58 -> 2.99; D=20 / 100,005 nodes / 65,536 points F32 4.39 ->
// 2.83, FP64 8.36 -> 4.20; D=24 / 12,011 nodes / 128 dofs / 30,011 points F32
// 6.48 -> 1.03, FP64 12.6 -> 1.57; D=8 / 4,096 points F32 0.28 -> 0.056. The
// MFMAs of the alive nodes are about half of the F32 time at D=16; the rest is
// the issue of the basis products and of their surplus rows' copies.
#include "sweep_common.h"
#include "kernels.h"
#include "hat_table.h"

namespace hddm_lb {

namespace {

typedef double dv4_t __attribute__((ext_vector_type(4)));
typedef float fv32_t __attribute__((ext_vector_type(32)));

template <int PREC> struct TableContract;

template <>
struct TableContract<HDDM_LB_F32>
{
	typedef float B;
	typedef double Acc;
	static constexpr bool kHalves = true;   // batches do not cross 32 nodes: folds
	static constexpr int kAcc = 32;
	// Surplus rows of a batch on their way: one 16-byte load per lane takes
	// eight rows (lane l: slot l / 8, dofs 4 (l % 8) ..), which go through a
	// 1 KB LDS buffer of the wave to the MFMA's one dof per lane.
	static constexpr int kStage = 1024;
	typedef float f4v_t __attribute__((ext_vector_type(4)));
	struct Rows { f4v_t v; };
	struct S { float v[8]; };
	fv32_t acc;
	double sum[32];
	int chunk;                      // 32-node chunk acc sums
	const float* base;
	uint32_t DP;

	__device__ __forceinline__ void init(const StateDesc* sd, int dp, int tile)
	{
#pragma unroll
		for (int r = 0; r < 32; r++) sum[r] = 0.0;
		zero();
		chunk = -1;
		base = ldc(&sd->s32r) + 32 * tile;
		DP = (uint32_t)dp;
	}

	// one MFMA of zeros instead of 32 moves
	__device__ __forceinline__ void zero()
	{
		fv32_t z;
#pragma unroll
		for (int r = 0; r < 32; r++) z[r] = 0.0f;
		acc = __builtin_amdgcn_mfma_f32_32x32x1f32(0.0f, 0.0f, z, 0, 0, 0);
	}

	// rv: the window's compacted records, slot j in lane j; j0: the batch's first
	// n0: the node of the window's first op; zero: nodes from there to the row of zeros
	__device__ __forceinline__ void load(Rows& w, int n0, int zero, uint32_t rv, int j0, int lane)
	{
		const uint32_t r = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (j0 + (lane >> 3)), (int)rv);
		const uint32_t n = r & kTabPrefix ? (uint32_t)zero : r >> kTabNodeShift;
		w.v = *(const f4v_t*)(base + (size_t)n0 * DP + ((size_t)n * DP + 4u * (lane & 7)));
	}

	__device__ __forceinline__ void stage(S& s, const Rows& w, char* buf, int lane)
	{
		wave_lds_order();
		*(f4v_t*)(buf + 16 * lane) = w.v;
		wave_lds_order();
#pragma unroll
		for (int k = 0; k < 8; k++) s.v[k] = *(const float*)(buf + 128 * k + 4 * (lane & 31));
	}

	__device__ __forceinline__ void fold()
	{
#pragma unroll
		for (int r = 0; r < 32; r++) sum[r] += (double)acc[r];
	}

	__device__ __forceinline__ void begin(int c)
	{
		if (c != chunk)
		{
			if (chunk >= 0) { fold(); zero(); }
			chunk = c;
		}
	}

	__device__ __forceinline__ void contract(const S& s, const float (&b)[8], int count)
	{
#pragma unroll
		for (int k = 0; k < 8; k++)
			if (k == 0 || count > k) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(s.v[k], b[k], acc, 0, 0, 0);
	}

	__device__ __forceinline__ void finish() { fold(); }
	__device__ __forceinline__ double get(int r) const { return sum[r]; }
	__device__ __forceinline__ void set(int r, double v) { sum[r] = v; }

	// register 16 t + r of lane l: point 32 t + l % 32, dof 8 (r / 4) + 4 (l / 32) + r % 4
	__device__ __forceinline__ static int point(int i, int lane) { return 32 * (i >> 4) + (lane & 31); }
	__device__ __forceinline__ static int dof(int i, int lane) { return 8 * ((i & 15) >> 2) + 4 * (lane >> 5) + (i & 3); }
};

template <>
struct TableContract<HDDM_LB_FP64>
{
	typedef double B;
	static constexpr bool kHalves = false;
	static constexpr int kAcc = 32;
	// Surplus rows on their way: two 16-byte loads per lane take four rows
	// each (lane l: slot 4 q + l / 16, 16-byte piece l % 16, the two 128-byte
	// halves of odd slots exchanged so that the reads below meet no bank twice)
	static constexpr int kStage = 2048;
	typedef double d2v_t __attribute__((ext_vector_type(2)));
	struct Rows { d2v_t v[2]; };
	struct S { double v[2][2]; };   // [quad][16-dof half]: S[slot 4 q + lane / 16][dof 16 h + lane % 16]
	dv4_t acc[2][4];                // [16-dof half][16-point tile]
	const double* base;
	uint32_t DP;

	__device__ __forceinline__ void init(const StateDesc* sd, int dp, int tile)
	{
#pragma unroll
		for (int h = 0; h < 2; h++)
#pragma unroll
			for (int p = 0; p < 4; p++) acc[h][p] = dv4_t{ 0.0, 0.0, 0.0, 0.0 };
		base = ldc(&sd->s64) + 32 * tile;
		DP = (uint32_t)dp;
	}

	__device__ __forceinline__ void load(Rows& w, int n0, int zero, uint32_t rv, int j0, int lane)
	{
		const int k = lane >> 4;
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const uint32_t r = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (j0 + 4 * q + k), (int)rv);
			const uint32_t n = r & kTabPrefix ? (uint32_t)zero : r >> kTabNodeShift;
			w.v[q] = *(const d2v_t*)(base + (size_t)n0 * DP + ((size_t)n * DP + 2u * ((lane & 15) ^ (8 * (k & 1)))));
		}
	}

	__device__ __forceinline__ void stage(S& s, const Rows& w, char* buf, int lane)
	{
		wave_lds_order();
		*(d2v_t*)(buf + 16 * lane) = w.v[0];
		*(d2v_t*)(buf + 1024 + 16 * lane) = w.v[1];
		wave_lds_order();
		const int k = lane >> 4;
#pragma unroll
		for (int q = 0; q < 2; q++)
#pragma unroll
			for (int h = 0; h < 2; h++)
				s.v[q][h] = *(const double*)(buf + 1024 * q + 256 * k + 128 * (h ^ (k & 1)) + 8 * (lane & 15));
	}

	__device__ __forceinline__ void begin(int) {}

	// empty slots hold zeros
	__device__ __forceinline__ void contract(const S& s, const double (&bv)[8], int)
	{
#pragma unroll
		for (int q = 0; q < 2; q++) quad(s, q, bv + 4 * q);
	}

	__device__ __forceinline__ void quad(const S& s, int q, const double* bv)
	{
		double b0 = bv[0], b1 = bv[1], b2 = bv[2], b3 = bv[3];
		const uint64_t nz = __builtin_amdgcn_ballot_w64((b0 != 0.0) | (b1 != 0.0) | (b2 != 0.0) | (b3 != 0.0));
		// rows of 16 lanes: from [node][row = point tile] to [point tile][row = node]
		transpose_rows(b0, b1, b2, b3);
		const double b[4] = { b0, b1, b2, b3 };
#pragma unroll
		for (int p = 0; p < 4; p++)
			if ((nz >> (16 * p)) & 0xffffull)
			{
				acc[0][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.v[q][0], b[p], acc[0][p], 0, 0, 0);
				acc[1][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.v[q][1], b[p], acc[1][p], 0, 0, 0);
			}
	}

	__device__ __forceinline__ void finish() {}
	__device__ __forceinline__ double get(int r) const { return acc[r >> 4][(r >> 2) & 3][r & 3]; }
	__device__ __forceinline__ void set(int r, double v) { acc[r >> 4][(r >> 2) & 3][r & 3] = v; }

	// D[i][j] in lane j + 16 (i % 4), element i / 4: i the dof, j the point
	__device__ __forceinline__ static int point(int i, int lane) { return 16 * ((i >> 2) & 3) + (lane & 15); }
	__device__ __forceinline__ static int dof(int i, int lane) { return 16 * (i >> 4) + 4 * (i & 3) + (lane >> 4); }
};

} // namespace

// NW waves per workgroup, one workgroup per CU; BASE: registers for the compiler.
template <int PREC, int NW, int BASE>
__device__ __forceinline__ void sweep_table(const SweepArgs& a, int hats_max)
{
	extern __shared__ __attribute__((aligned(16))) double lds[];
	typedef TableContract<PREC> C;
	const int lane = threadIdx.x & 63;
	const int wave = uniform((int)(threadIdx.x >> 6));
	char* const tl = (char*)lds + lane * 8;                     // the lane's column of the hat rows
	const uint32_t lane8 = (uint32_t)lane * 8u;
	uint32_t rowmask = kTabRow;                                 // in a vector register: one v_and_or per address
	asm volatile("" : "+v"(rowmask));
	double* const X = lds + (size_t)hats_max * kWave;           // coordinate rows
	uint64_t* const M = (uint64_t*)(X + (size_t)a.dim * kWave);
	int64_t* const slot = (int64_t*)(M + ((hats_max + 1) & ~1));
	char* const stage = (char*)(slot + 2) + (size_t)wave * C::kStage;

	for (;;)
	{
		__syncthreads();
		if (threadIdx.x == 0) *slot = (int64_t)atomicAdd(&a.hdr->counter, 1ull);
		__syncthreads();
		const int64_t item = (int64_t)uniform64((uint64_t)*slot);
		if (item >= ldc(&a.hdr->nitems)) break;
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
		const int tiles = ldc(&sd->dofs_pad) >> 5;
		if (a.dt_base >= tiles) continue;
		const int64_t rem = ldc(&pl->count) - blk * kWave;
		const int np = rem < kWave ? (int)rem : kWave;
		{
			const uint32_t orig = a.perm[ldc(&pl->start) + blk * kWave + (lane < np ? lane : np - 1)];
			const double* xrow = a.x + (int64_t)orig * a.ldx;
			for (int d = wave; d < a.dim; d += NW) X[d * kWave + lane] = xrow[d];
		}
		__syncthreads();
		// the hats at the block's points, and the points inside their supports
		{
			const int hats = ldc(&sd->hats);
			const u4_t* ht = (const u4_t*)ldc(&sd->hat);
			const uint64_t valid = np < kWave ? ((uint64_t)1 << np) - 1 : ~(uint64_t)0;
			if (wave == 0)
			{
				lds[kHatNone * kWave + lane] = 0.0;
				lds[kHatAll * kWave + lane] = 1.0;
				if (lane == 0) { M[kHatNone] = 0; M[kHatAll] = valid; }
			}
#pragma unroll 1
			for (int h = kHatFirst + wave; h < hats; h += NW)
			{
				const u4_t e = ldc(ht + h);
				const double u = (*(const double*)((const char*)X + lane * 8 + e[0]) + f64_from_high(e[2])) * f64_from_high(e[1]);
				const double v = fmax(1.0 - fabs(u), 0.0);
				lds[h * kWave + lane] = v;
				const uint64_t in = __builtin_amdgcn_ballot_w64(v > 0.0) & valid;
				if (lane == 0) M[h] = in;
			}
		}
		__syncthreads();

		// wave: a tile of the pass and a part of the segment's windows
		const int tw = min(tiles - a.dt_base, 4);
		const int parts = NW / tw;
		const int part = wave / tw, tile = a.dt_base + wave - part * tw;
		const bool on = part < parts;
		C c;
		c.init(sd, ldc(&sd->dofs_pad), tile);
		if (on)
		{
			const int nwin = (ldc(&sd->nops) + kWin - 1) / kWin;
			const int nseg = (int)ldc(&pl->nseg);
			const int s0 = (int)((int64_t)nwin * seg / nseg), s1 = (int)((int64_t)nwin * (seg + 1) / nseg);
			// the wave's windows: s0 + part, s0 + part + parts, ... (neighbouring
			// windows are alive for the same points, so this is even)
			const int mine = s1 - s0 > part ? (s1 - s0 - part + parts - 1) / parts : 0;
			const uint32_t* const recs = ldc(&sd->trec);
			const int32_t* const wnode = ldc(&sd->tnode);
			const int nno = ldc(&sd->nno);
			const int hs = ldc(&sd->hstride);
			dv8_t P;
#pragma unroll
			for (int i = 0; i < 8; i++) P[i] = 1.0;
			// the products of op q's path up to factor t - 1, from its hats
			auto path = [&](int q, int t) {
#pragma unroll 1
				for (int f = 0; f < t; f++)
				{
					const uint32_t w = ldc((const uint32_t*)ldc(&sd->thid) + ((size_t)q * hs + f) / 2);
					Path<BASE>::mulp(P, 2u * (uint32_t)f, *(const double*)(tl + ((f & 1 ? w >> 16 : w & 0xffffu) * kWave)));
				}
			};
			for (int wb = 0; wb < mine; wb += kWave)
			{
				// selection: the alive ops of the wave's window wb + i as lane i
				// of (mlo, mhi)
				const int nb = min(kWave, mine - wb);
				const int first = s0 + part + wb * parts;
				uint32_t mlo, mhi;
				select_windows(sd, M, first, parts, nb, lane, mlo, mhi);

				if (a.stats && tile == a.dt_base)
				{
					// statistics mode: alive ops, 32-op halves of windows with one
					// (F32: folds; FP64: batches of eight), F32 MFMAs
					uint32_t ops = (uint32_t)__popc(mlo) + (uint32_t)__popc(mhi);
					uint32_t ch = C::kHalves ? (uint32_t)(mlo != 0u) + (uint32_t)(mhi != 0u) : (ops + 7u) / 8u;
					for (int off = 32; off; off >>= 1)
					{
						ops += __shfl_xor(ops, off, 64);
						ch += __shfl_xor(ch, off, 64);
					}
					if (lane == 0)
					{
						atomicAdd(&a.stats[0], (unsigned long long)ops);
						atomicAdd(&a.stats[2], (unsigned long long)ch);
						if (C::kHalves) atomicAdd(&a.stats[4], (unsigned long long)ops * tw);
					}
				}

				// Batches of eight slots of a window's compacted records. While
				// one batch is contracted the next one's surplus rows and hats
				// are on their way, and the records of the window after.
				uint64_t wm = __builtin_amdgcn_ballot_w64((mlo | mhi) != 0u);
				if (!wm) continue;
				int cw = __builtin_ctzll(wm);     // the window whose records are on their way
				uint32_t rnext = recs[(size_t)(first + cw * parts) * kWin + lane];
				uint32_t rv = 0;                  // compacted records, slot j in lane j
				int slots = 0, half1 = 0, j0 = 0;
				int q0 = 0, n0 = 0, depth = 0;    // the window's first op, its node and depth
				uint32_t r[8];                    // the batch's records
				int count = 0, chunk = 0, t = 0;
				double f[8];
				typename C::Rows rows;
				// the next batch: its records, its surplus rows and hats requested
				auto next = [&]() -> bool {
					if (j0 >= slots)
					{
						if (!wm) return false;
						const uint32_t lo = __builtin_amdgcn_readlane(mlo, cw), hi = __builtin_amdgcn_readlane(mhi, cw);
						const int c0 = __builtin_popcount(lo), c1 = __builtin_popcount(hi);
						half1 = C::kHalves ? (c0 + 7) & ~7 : c0;
						slots = half1 + c1;
						// an alive lane sends its record to its slot, the others
						// nothing (0) to one that is empty; slots that get none
						// read 0
						const bool alive = (((lane < 32 ? lo : hi) >> (lane & 31)) & 1u) != 0u;
						const int pos = alive
							? (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u)) + (lane >= 32 ? half1 - c0 : 0)
							: (half1 > c0 ? c0 : slots);
						rv = (uint32_t)__builtin_amdgcn_ds_permute(4 * pos, alive ? (int)rnext : 0) ^ kTabEmpty;
						q0 = (first + cw * parts) * kWin;
						n0 = ldc(wnode + first + cw * parts);
						depth = (int)((__builtin_amdgcn_readlane(rnext, 0) ^ kTabEmpty) & kTabDepth2) / 2;
						wm &= wm - 1;
						if (wm)
						{
							cw = __builtin_ctzll(wm);
							rnext = recs[(size_t)(first + cw * parts) * kWin + lane];
						}
						j0 = 0;
					}
					c.load(rows, n0, nno - n0, rv, j0, lane);
#pragma unroll
					for (int k = 0; k < 8; k++) r[k] = __builtin_amdgcn_readlane(rv, j0 + k);
#pragma unroll
					for (int k = 0; k < 8; k++) f[k] = *(const double*)((const char*)lds + ((r[k] & rowmask) | lane8));
					count = min(8, slots - j0);
					chunk = q0 / 32 + (j0 >= half1 ? 1 : 0);
					t = j0 ? 0 : depth;
					j0 += 8;
					return true;
				};
				bool more = next();
#pragma unroll 1
				while (more)
				{
					typename C::S sb;
					c.stage(sb, rows, stage, lane);
					// The parents of the window's ops that lie before the window
					// are the proper prefixes of its first op: its first batch
					// multiplies them up ahead.
					if (t > 0) path(chunk / 2 * kWin, t);
					typename C::B v[8];
					Path<BASE>::mulp4(P, r, f, v);
					Path<BASE>::mulp4(P, r + 4, f + 4, v + 4);
					// request the next batch before this one's MFMAs
					const int cnt = count, chk = chunk;
					__builtin_amdgcn_sched_barrier(0);
					more = next();
					__builtin_amdgcn_sched_barrier(0);
					c.begin(chk);
					c.contract(sb, v, cnt);
				}
			}
			c.finish();
		}

		// the parts' sums, in order, through LDS (the hat rows are done with)
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
			const int64_t count = ldc(&pl->count);
			const int dofs = ldc(&sd->dofs), DP = ldc(&sd->dofs_pad);
			const uint32_t orig = a.perm[ldc(&pl->start) + blk * kWave + (lane < np ? lane : np - 1)];
			const bool split = ldc(&pl->nseg) > 1;
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

// F32: three waves per SIMD in 168 registers each. FP64, whose time is its
// MFMAs, two.
__global__ void __launch_bounds__(64 * kTableWavesF32) __attribute__((amdgpu_waves_per_eu(3)))
	sweep_table_f32_kernel(SweepArgs a, int hats_max)
{
	sweep_table<HDDM_LB_F32, kTableWavesF32, 152>(a, hats_max);
}

__global__ void __launch_bounds__(64 * kTableWavesFP64) __attribute__((amdgpu_waves_per_eu(2)))
	sweep_table_fp64_kernel(SweepArgs a, int hats_max)
{
	sweep_table<HDDM_LB_FP64, kTableWavesFP64, 224>(a, hats_max);
}

// Rows of hats and coordinates, masks, the item slot, the staging buffers; the part sums of up to
// four tiles lie over the rows.
size_t sweep_table_lds_bytes(int dim, int hats_max, int tiles)
{
	constexpr size_t f32 = (size_t)kTableWavesF32 * TableContract<HDDM_LB_F32>::kStage;
	constexpr size_t fp64 = (size_t)kTableWavesFP64 * TableContract<HDDM_LB_FP64>::kStage;
	const size_t rows = (size_t)(hats_max + dim) * kWave * 8 + (size_t)((hats_max + 1) & ~1) * 8 + 16 + (f32 > fp64 ? f32 : fp64);
	const size_t sums = (size_t)(tiles < 4 ? tiles : 4) * 32 * kWave * 8;
	return rows > sums + 16 ? rows : sums + 16;
}

int sweep_table_waves(int prec) { return prec == HDDM_LB_F32 ? kTableWavesF32 : kTableWavesFP64; }

const void* sweep_table_kernel_ptr(int prec)
{
	if (prec == HDDM_LB_FP64) return (const void*)&sweep_table_fp64_kernel;
	if (prec == HDDM_LB_F32) return (const void*)&sweep_table_f32_kernel;
	return nullptr;
}

} // namespace hddm_lb
