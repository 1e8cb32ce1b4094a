// Adjoint of the LinearBasis forward over hat tables (gfx950), FP64, for
// states of one 32-dof tile and D <= 32. Two kernels:
//   dS_k   = sum_p B_k(x_p) g_p
//   dx_p,d = sum_k w_pk dB_k/dx_d,  w_pk = g_p . S_k
// One workgroup of eight waves takes one 64-point block against one range of
// the state's ops, as the hat-table sweep of the forward: every distinct hat
// is evaluated once at the block's points (values and masks in LDS), a
// window's alive ops are found by ANDing masks, one op per lane, moved
// together, and their basis values formed one point per lane in trie order.
// Then 16 alive nodes at a time, on v_mfma_f64_16x16x4f64:
//   dS  D[node][dof] += B[node][4 points] g[4 points][dof], 16 steps. The
//       basis goes through LDS from a point to a node per lane (rows of 528
//       bytes: eight rows meet no bank twice), in two halves of eight nodes
//       to leave room for the hats. Added to dS with atomics, four runs of
//       16 dofs per instruction.
//   dx  D[node][point] += S[node][4 dofs] g[4 dofs][point], 8 steps per 16
//       points, brought back to one point per lane by row swaps; r = w B.
//       An edge e of the trie adds R_e phi'/phi to dx[dim(e)], R_e the sum
//       of r over the nodes below it, so every node reaches each of its
//       factors once. The 16 are taken from the last back: R[t] sums what
//       the finished edges at depth t hand to the edge above, and there is
//       one step per node with no branch in it (leaving edges one by one in
//       trie order, the path decides what comes next: 465 cycles a node
//       instead of about 150). P, R and dx are in registers under GPR
//       indexing. Edges above the first of the 16 get the 16's part of
//       their sums after it.
// An FP64 MFMA runs on the vector unit, so a node costs the 128 cycles of its
// 32 products and what its basis and edges issue beside them.
//
// Measured against the per-tile kernels (ms, before -> here, 32 dofs): D=20 /
// 100,005 nodes / 65,536 points (37.7 million alive nodes of blocks) dx 16.6 ->
// 7.0, dS 14.4 -> 7.3 (4.9 without its atomics); D=16 / 60,010 nodes / 100,003
// points dx 8.7 -> 4.9, dS 9.9 -> 4.9; D=8 / 3,937 nodes / 16 dofs / 20,000
// points both 1.64 -> 0.30.
#include "sweep_common.h"
#include "hat_table.h"
#include "kernels.h"

namespace hddm_lb {

namespace {

typedef double dv4_t __attribute__((ext_vector_type(4)));
typedef double dv16_t __attribute__((ext_vector_type(16)));
typedef double d2v_t __attribute__((ext_vector_type(2)));

constexpr int kAW = 8;                          // waves
constexpr int kGRow = 33;                       // doubles per point row of g (33: no bank conflicts)
constexpr int kStageRow = 66;                   // doubles per node row of a wave's basis stage
constexpr int kStageBytes = 8 * kStageRow * 8;
constexpr int kPosShift = 26;                   // records of slots: the op's place in its window
constexpr uint32_t kInfoHigh = 0xfff00000u;     // info of an op's hat: high word of i, twice its dim

// dx: P is in v[224:239] (Path<224>), dx in v[160:223], R in v[144:159].
// The edge at depth t (T2 = 2 t) whose nodes after its own are done: its sum
// is r plus R[t + 1], which is cleared for the next edge; the sum goes to
// dx[dim] times q, and to R[t] for the edge above (entry 0: none, not read).
template <int XB>
__device__ __forceinline__ void edge_done(dv16_t& dx0, dv16_t& dx1, dv8_t& R, uint32_t info, uint32_t t2, double r, double q)
{
	double e;
#define HDDM_EDGE \
	"s_set_gpr_idx_on %[t], gpr_idx(SRC0)\n" "v_add_f64 %[e], v[146:147], %[r]\n" \
	"s_set_gpr_idx_mode gpr_idx(DST)\n" "v_mul_f64 v[146:147], 0, 0\n" \
	"s_set_gpr_idx_mode gpr_idx(SRC0,DST)\n" "v_add_f64 v[144:145], v[144:145], %[e]\n" \
	"s_set_gpr_idx_on %[i], gpr_idx(SRC2,DST)\n" "v_fma_f64 v[160:161], %[e], %[q], v[160:161]\n" "s_set_gpr_idx_off\n"
	if constexpr (XB == 1)
		asm(HDDM_EDGE : [e] "=&v"(e), "+{v[160:191]}"(dx0), "+{v[144:159]}"(R)
			: [i] "s"(info), [t] "s"(t2), [r] "v"(r), [q] "v"(q) : "m0");
	else
		asm(HDDM_EDGE : [e] "=&v"(e), "+{v[160:191]}"(dx0), "+{v[192:223]}"(dx1), "+{v[144:159]}"(R)
			: [i] "s"(info), [t] "s"(t2), [r] "v"(r), [q] "v"(q) : "m0");
#undef HDDM_EDGE
}

// phi'/phi = -i / (phi with the sign of u), from the hardware reciprocal
// refined by two Newton steps; 0 outside the support and at the peak.
__device__ __forceinline__ double hat_slope(double f, uint32_t info)
{
	const bool in = f != 0.0 && f != 1.0;
	const double ph = in ? f : 1.0;
	double rc = __builtin_amdgcn_rcp(ph);
	rc = fma(rc, fma(-ph, rc, 1.0), rc);
	rc = fma(rc, fma(-ph, rc, 1.0), rc);
	return in ? rc * -f64_from_high(info & kInfoHigh) : 0.0;
}

} // namespace

constexpr int kModeDx = 0, kModeDs = 1;

// XB: banks of 16 dims (dx)
template <int MODE, int XB>
__device__ __forceinline__ void adjoint_table(const AdjointArgs& a, int hats_max)
{
	extern __shared__ __attribute__((aligned(16))) double lds[];
	constexpr bool DS = MODE == kModeDs;
	const int lane = threadIdx.x & 63;
	const int wave = uniform((int)(threadIdx.x >> 6));
	const int col = lane & 15, row = lane >> 4;
	const uint32_t lane8 = (uint32_t)lane * 8u;
	uint32_t rowmask = kTabRow;
	asm volatile("" : "+v"(rowmask));
	double* const G = lds + (size_t)hats_max * kWave;               // [64][kGRow]
	uint64_t* const M = (uint64_t*)(G + kWave * kGRow);
	uint32_t* const info = (uint32_t*)(M + ((hats_max + 1) & ~1));               // [hats], dx
	int64_t* const slot = (int64_t*)(info + ((hats_max + 3) & ~3));
	// the coordinate rows are read before the basis stages over them are written
	double* const X = (double*)(slot + 2);
	double* const stage = X + (size_t)wave * (kStageBytes / 8);

	for (;;)
	{
		__syncthreads();
		if (threadIdx.x == 0) { slot[0] = (int64_t)atomicAdd(&a.hdr->counter, 1ull); slot[1] = 0; }
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
		const int dofs = ldc(&sd->dofs);
		const int64_t rem = ldc(&pl->count) - blk * kWave;
		const int np = rem < kWave ? (int)rem : kWave;
		const uint32_t orig = a.perm[ldc(&pl->start) + blk * kWave + (lane < np ? lane : np - 1)];
		{
			const double* xrow = a.x + (int64_t)orig * a.ldx;
			for (int d = wave; d < a.dim; d += kAW) X[d * kWave + lane] = xrow[d];
			// upstream gradient, 0 past the block and past the dofs: half a
			// row per 16 lanes
			bool odd = false;
			for (int p = 4 * wave + row; p < kWave; p += 4 * kAW)
			{
				const uint32_t op = (uint32_t)__shfl((int)orig, p, 64);
				const double* grow = a.g + (int64_t)op * a.ldg;
#pragma unroll
				for (int h = 0; h < 2; h++)
				{
					const int c = 16 * h + col;
					const double v = p < np && c < dofs ? grow[c] : 0.0;
					odd |= !(fabs(v) < __builtin_huge_val());
					G[p * kGRow + c] = v;
				}
			}
			if (!DS && odd) slot[1] = 1;
		}
		__syncthreads();
		// The hats at the block's points, and the points inside their
		// supports. For dx a value carries the sign of u = x i - j, and 1.0
		// is the peak alone (u is 0 of either sign: -0.0 at x = -0.0 and
		// j = 0): u > 0 that rounds to 1 is the value below it.
		{
			const int hats = ldc(&sd->hats);
			const u4_t* ht = (const u4_t*)ldc(&sd->hat);
			const uint64_t valid = np < kWave ? ((uint64_t)1 << np) - 1 : ~(uint64_t)0;
			if (wave == 0)
			{
				lds[kHatNone * kWave + lane] = 0.0;
				lds[kHatAll * kWave + lane] = 1.0;
				if (lane == 0) { M[kHatNone] = 0; M[kHatAll] = valid; info[kHatNone] = 0; info[kHatAll] = 0; }
			}
#pragma unroll 1
			for (int h = kHatFirst + wave; h < hats; h += kAW)
			{
				const u4_t e = ldc(ht + h);
				const double u = (*(const double*)((const char*)X + lane * 8 + e[0]) + f64_from_high(e[2])) * f64_from_high(e[1]);
				const double v = fmax(1.0 - fabs(u), 0.0);
				const uint64_t in = __builtin_amdgcn_ballot_w64(v > 0.0) & valid;
				lds[h * kWave + lane] = DS ? v : u < 0.0 ? -v : v == 1.0 && u > 0.0 ? 1.0 - 0x1p-53 : v;
				if (lane == 0)
				{
					M[h] = in;
					if (!DS) info[h] = (e[1] & kInfoHigh) | (2u * (e[0] >> 9));
				}
			}
		}
		__syncthreads();

		const bool wild = !DS && uniform((int)slot[1]) != 0;          // a gradient of the block is infinite or no number
		const int nwin = (ldc(&sd->nops) + kWin - 1) / kWin;
		const int nseg = (int)ldc(&pl->nseg);
		const int s0 = (int)((int64_t)nwin * seg / nseg), s1 = (int)((int64_t)nwin * (seg + 1) / nseg);
		const int mine = s1 - s0 > wave ? (s1 - s0 - wave + kAW - 1) / kAW : 0;
		const uint32_t* const recs = ldc(&sd->trec);
		const int32_t* const wnode = ldc(&sd->tnode);
		const int nno = ldc(&sd->nno), DP = ldc(&sd->dofs_pad);
		const int hs = ldc(&sd->hstride);
		// the dS of the copy of the XCD that the workgroup runs on
		double* ds = a.ds + (DS ? ldc(&sd->ds_offset) : 0);
		if (DS && a.ds_xcd > 0)
		{
			uint32_t xcc;
			asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
			ds += (int64_t)(xcc & 7u) * a.ds_xcd;
		}
		dv8_t P;
#pragma unroll
		for (int i = 0; i < 8; i++) P[i] = 1.0;
		dv8_t R;
		dv16_t dx0, dx1;
		if constexpr (!DS)
		{
#pragma unroll
			for (int i = 0; i < 8; i++) R[i] = 0.0;
#pragma unroll
			for (int i = 0; i < 16; i++) { dx0[i] = 0.0; dx1[i] = 0.0; }
		}

		for (int wb = 0; wb < mine; wb += kWave)
		{
			const int nb = min(kWave, mine - wb);
			const int first = s0 + wave + wb * kAW;
			uint32_t mlo, mhi;
			select_windows(sd, M, first, kAW, nb, lane, mlo, mhi);
			uint64_t wm = __builtin_amdgcn_ballot_w64((mlo | mhi) != 0u);
			if (!wm) continue;
			int cw = __builtin_ctzll(wm);     // the window whose records are on their way
			uint32_t rnext = recs[(size_t)(first + cw * kAW) * kWin + lane];
#pragma unroll 1
			for (;;)
			{
				// the window's alive ops moved together: slot j in lane j, empty
				// slots after them
				const int w = first + cw * kAW;
				const uint32_t lo = __builtin_amdgcn_readlane(mlo, cw), hi = __builtin_amdgcn_readlane(mhi, cw);
				const int slots = __builtin_popcount(lo) + __builtin_popcount(hi);
				const bool alive = (((lane < 32 ? lo : hi) >> (lane & 31)) & 1u) != 0u;
				const int pos = alive ? (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u)) : slots;
				const uint32_t rv = (uint32_t)__builtin_amdgcn_ds_permute(4 * pos, alive ? (int)(rnext | (uint32_t)lane << kPosShift) : 0) ^ kTabEmpty;
				const int n0 = ldc(wnode + w);
				wm &= wm - 1;
				const bool more = wm != 0;
				if (more)
				{
					cw = __builtin_ctzll(wm);
					rnext = recs[(size_t)(first + cw * kAW) * kWin + lane];
				}
				uint32_t iv = 0;   // infos by slot
				if constexpr (!DS) iv = info[(rv & kTabRow) >> 9];
				// The hats above slot j, by depth in the lanes, as offsets of
				// their rows; depth lanes count.
				auto above = [&](int j, int& depth) -> uint32_t {
					const uint32_t r = __builtin_amdgcn_readlane(rv, j);
					depth = (int)(r & kTabDepth2) / 2;
					const uint16_t* ids = ldc(&sd->thid) + ((size_t)w * kWin + (r >> kPosShift)) * hs;
					return (uint32_t)ids[lane < depth ? lane : 0] * kWave;
				};
				{
					// the products above the first slot: its parents, and all
					// parents of the others that lie before it
					int depth;
					const uint32_t up = above(0, depth);
#pragma unroll 1
					for (int f = 0; f < depth; f++)
						Path<224>::mulp(P, 2u * (uint32_t)f, *(const double*)((const char*)lds + __builtin_amdgcn_readlane(up, f) + lane8));
				}

#pragma unroll 1
				for (int j0 = 0; j0 < slots; j0 += 16)
				{
					if constexpr (DS)
					{
						// this lane's node of the D rows and its place in dS
						int64_t at[4];
#pragma unroll
						for (int e = 0; e < 4; e++)
						{
							const int i = j0 + 4 * e + row;
							const uint32_t r = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * i, (int)rv);
							const bool live = i < slots && !(r & kTabPrefix);
							at[e] = live ? (int64_t)ldc(&sd->order)[n0 + (int)((r >> kTabNodeShift) & 63u)] * dofs : -1;
						}
						double A[16];   // B[node col][point 16 row + s]
#pragma unroll
						for (int h = 0; h < 2; h++)
						{
							// no second eight: rows 8 .. repeat the first, not added
							if (h && slots - j0 <= 8) continue;
							uint32_t r[8];
							double f[8], b[8];
#pragma unroll
							for (int k = 0; k < 8; k++) r[k] = __builtin_amdgcn_readlane(rv, j0 + 8 * h + k);
#pragma unroll
							for (int k = 0; k < 8; k++) f[k] = *(const double*)((const char*)lds + ((r[k] & rowmask) | lane8));
							Path<224>::mulp4(P, r, f, b);
							Path<224>::mulp4(P, r + 4, f + 4, b + 4);
#pragma unroll
							for (int k = 0; k < 8; k++) stage[k * kStageRow + lane] = b[k];
							wave_lds_order();
							if (h == 0 || col >= 8)
							{
#pragma unroll
								for (int m = 0; m < 8; m++)
								{
									const d2v_t v = *(const d2v_t*)(stage + (col & 7) * kStageRow + 16 * row + 2 * m);
									A[2 * m] = v[0];
									A[2 * m + 1] = v[1];
								}
							}
							wave_lds_order();
						}
						dv4_t acc[2] = { { 0.0, 0.0, 0.0, 0.0 }, { 0.0, 0.0, 0.0, 0.0 } };
#pragma unroll
						for (int t = 0; t < 16; t++)
#pragma unroll
							for (int h = 0; h < 2; h++)
								acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[t], G[(16 * row + t) * kGRow + 16 * h + col], acc[h], 0, 0, 0);
#pragma unroll
						for (int e = 0; e < 4; e++)
							if (at[e] >= 0)
							{
#pragma unroll
								for (int h = 0; h < 2; h++)
									if (16 * h + col < dofs) unsafeAtomicAdd(ds + at[e] + 16 * h + col, acc[h][e]);
							}
					}
					else
					{
						int depth;
						const uint32_t up = above(j0, depth);
						// surplus rows: lane: slot col, dofs 8 row ..
						double S[8];
						{
							const uint32_t r = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (j0 + col), (int)rv);
							const int n = r & kTabPrefix ? nno : n0 + (int)((r >> kTabNodeShift) & 63u);
							const d2v_t* src = (const d2v_t*)(ldc(&sd->s64) + (size_t)n * DP + 8 * row);
#pragma unroll
							for (int m = 0; m < 4; m++)
							{
								const d2v_t v = src[m];
								S[2 * m] = v[0];
								S[2 * m + 1] = v[1];
							}
						}
						// w, points 16 t + col, slots 4 e + row
						dv4_t acc[4];
#pragma unroll
						for (int t = 0; t < 4; t++) acc[t] = dv4_t{ 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
						for (int q = 0; q < 8; q++)
#pragma unroll
							for (int t = 0; t < 4; t++)
								acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[q], G[(16 * t + col) * kGRow + 8 * row + q], acc[t], 0, 0, 0);
						double v[16];
#pragma unroll
						for (int e = 0; e < 4; e++)
						{
							double b0 = acc[0][e], b1 = acc[1][e], b2 = acc[2][e], b3 = acc[3][e];
							transpose_rows(b0, b1, b2, b3);
							v[4 * e] = b0;
							v[4 * e + 1] = b1;
							v[4 * e + 2] = b2;
							v[4 * e + 3] = b3;
						}
						// The second eight only where there are some: half of the
						// windows' last batches have none.
						uint32_t r[16];
						double f[16];
						auto form = [&](int h) {
#pragma unroll
							for (int k = 8 * h; k < 8 * h + 8; k++) r[k] = __builtin_amdgcn_readlane(rv, j0 + k);
#pragma unroll
							for (int k = 8 * h; k < 8 * h + 8; k++) f[k] = *(const double*)((const char*)lds + ((r[k] & rowmask) | lane8));
#pragma unroll
							for (int k = 8 * h; k < 8 * h + 8; k += 4)
							{
								double b[4];
								Path<224>::mulp4(P, r + k, f + k, b);
#pragma unroll
								for (int m = 0; m < 4; m++) v[k + m] *= b[m];
							}
							// Empty slots add nothing, nor do prefixes that are no nodes
							// where a gradient is infinite: times their zeros it is no
							// number.
							if (slots - j0 < 8 * h + 8 || wild)
							{
#pragma unroll
								for (int k = 8 * h; k < 8 * h + 8; k++) v[k] = r[k] & kTabPrefix ? 0.0 : v[k];
							}
						};
						// The edges, from the last slot back: an edge's nodes come
						// before it. The edges above the first slot get this batch's
						// part of their sums.
						auto edges = [&](int h) {
#pragma unroll
							for (int k = 8 * h + 7; k >= 8 * h; k--)
							{
								const uint32_t inf = __builtin_amdgcn_readlane(iv, j0 + k);
								edge_done<XB>(dx0, dx1, R, inf, r[k], v[k], hat_slope(f[k], inf));
							}
						};
						form(0);
						if (slots - j0 > 8)
						{
							form(1);
							edges(1);
						}
						edges(0);
						const uint32_t upinf = info[up / (8u * kWave)];
#pragma unroll 1
						for (int t = depth - 1; t >= 0; t--)
						{
							const uint32_t inf = __builtin_amdgcn_readlane(upinf, t);
							const double h = *(const double*)((const char*)lds + __builtin_amdgcn_readlane(up, t) + lane8);
							edge_done<XB>(dx0, dx1, R, inf, 2u * (uint32_t)t, 0.0, hat_slope(h, inf));
						}
					}
				}
				if (!more) break;
			}
		}

		if constexpr (!DS)
		{
			// the waves' sums, in order, through LDS (the hat rows are done with)
			double* const buf = lds + lane;
			for (int p = 0; p < kAW; p++)
			{
				__syncthreads();
				if (wave == p)
				{
#pragma unroll
					for (int d = 0; d < 16 * XB; d++)
						if (d < a.dim)
						{
							const double v = d < 16 ? dx0[d & 15] : dx1[d & 15];
							buf[d * kWave] = p ? buf[d * kWave] + v : v;
						}
				}
			}
			__syncthreads();
			if (lane < np)
			{
				double* out = nseg > 1 ? a.dxpart + ldc(&pl->dx_base) + (seg * ldc(&pl->count) + blk * kWave + lane) * a.dim
					: a.dx + (int64_t)orig * a.lddx;
				for (int d = wave; d < a.dim; d += kAW) out[d] = buf[d * kWave];
			}
		}
	}
}

template <int MODE, int XB>
__global__ void __launch_bounds__(64 * kAW) __attribute__((amdgpu_waves_per_eu(2))) adjoint_table_kernel(AdjointArgs a, int hats_max)
{
	adjoint_table<MODE, XB>(a, hats_max);
}

int adjoint_table_waves() { return kAW; }

const void* adjoint_table_kernel_ptr(bool dsurplus, int dim)
{
	if (dim > 32) return nullptr;
	if (dsurplus) return (const void*)&adjoint_table_kernel<kModeDs, 1>;
	return dim > 16 ? (const void*)&adjoint_table_kernel<kModeDx, 2> : (const void*)&adjoint_table_kernel<kModeDx, 1>;
}

// Hat rows, g, masks and infos, the item slot, then coordinates or basis
// stages; the dx sums (at most 32 rows) lie over the rows and g.
size_t adjoint_table_lds_bytes(bool dsurplus, int dim, int hats_max)
{
	const size_t coords = (size_t)dim * kWave * 8, stages = dsurplus ? (size_t)kAW * kStageBytes : 0;
	return (size_t)hats_max * kWave * 8 + (size_t)kWave * kGRow * 8 + (size_t)((hats_max + 1) & ~1) * 8
		+ (size_t)((hats_max + 3) & ~3) * 4 + 16
		+ (coords > stages ? coords : stages);
}

hipError_t launch_adjoint_table(const void* kern, int grid, size_t lds, const AdjointArgs& args, int hats_max, hipStream_t st)
{
	void* params[] = { (void*)&args, (void*)&hats_max };
	return hipLaunchKernel(kern, dim3(grid), dim3(kAW * kWave), params, lds, st);
}

} // namespace hddm_lb
