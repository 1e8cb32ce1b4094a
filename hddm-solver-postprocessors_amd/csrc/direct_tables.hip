// Tables of the direct sweep (sweep_direct.hip), built on the device from a
// state's op stream and factor table: one 8-byte record per node, the state's
// distinct hats (dim, i, j), and the hat ids of every node's factors.
#include <hip/hip_runtime.h>

#include "context.h"
#include "errors.h"
#include "kernels.h"
#include "layout_build.h"

#include <cstddef>

namespace hddm_lb {

namespace {

constexpr int kHashSlots = 8192;    // four times the most hats
constexpr int kHashProbes = 512;

// Needed while the tables are built.
struct HatTable
{
	unsigned long long key[kHashSlots];   // 0: free
	uint32_t id[kHashSlots];
};

// In the place of the records of the hats that are none (ids below kHatFirst).
struct HatCount
{
	int total;                            // hat ids
	int overflow;                         // a key found no slot, or there are more than kMaxHats
	int wide;                             // a dof column's largest value is out of F32's range
	int found;                            // keys inserted
	int odd;                              // a surplus is infinite or no number
};
static_assert(sizeof(HatCount) <= kHatFirst * 16, "fits");

// i is a power of two: its exponent, the dim and the centre name the hat.
__device__ __forceinline__ unsigned long long hat_key(const uint32_t* e)
{
	return (1ull << 63) | ((unsigned long long)(e[0] >> 1) << 44) | ((unsigned long long)(e[1] >> 20) << 32) | e[2];
}

__device__ __forceinline__ uint32_t hat_slot(unsigned long long key)
{
	key ^= key >> 29;
	key *= 0x9e3779b97f4a7c15ull;
	return (uint32_t)(key >> 40) & (kHashSlots - 1);
}

// The empty hash, the records of padding nodes (phi = max(0, 1 - |0 x - 2|) = 0)
// and of the nodes. One thread per hash slot or op.
__global__ void rec_kernel(HatTable* __restrict__ t, HatCount* __restrict__ cnt, int nno, int npad, int nops, const Op* __restrict__ ops,
	uint32_t* __restrict__ rec)
{
	const int q = blockIdx.x * blockDim.x + threadIdx.x;
	if (q < kHashSlots) t->key[q] = 0ull;
	if (q == 0) *cnt = HatCount{ 0, 0, 0, 0, 0 };
	if (q < npad - nno) { rec[2 * (nno + q)] = 0u; rec[2 * (nno + q) + 1] = 0xc0000000u; }
	if (q >= nops) return;
	const Op op = ops[q];
	if (!(op.ctrl & kOpLast)) return;
	const int n = (int)(op.ctrl >> kOpNodeShift);
	rec[2 * n] = (op.ihi & kRecIhi) | (op_dim(op.dim) << 9) | (2u * (op.ctrl & 15u)) | (op.ihi ? 0u : kRecRoot);
	rec[2 * n + 1] = op.njhi;
}

// An op that ends no node is a prefix that is no node: the nodes below it
// (a contiguous run, one wave per op) recompute their prefixes.
__global__ void __launch_bounds__(256) prefix_kernel(int nno, int nops, const Op* __restrict__ ops, uint32_t* __restrict__ rec)
{
	const int q = (int)((blockIdx.x * 256u + threadIdx.x) >> 6);
	if (q >= nops) return;
	const Op op = ops[q];
	if (op.ctrl & kOpLast) return;
	const int e = q + (int)(op.dim >> kOpSkipShift);
	const int n1 = e < nops ? (int)(ops[e].ctrl >> kOpNodeShift) : nno;
	for (int n = (int)(op.ctrl >> kOpNodeShift) + (int)(threadIdx.x & 63); n < n1; n += kWave)
		atomicOr(&rec[2 * n], kRecPrefix);
}

__global__ void special_kernel(int nno, int npad, uint32_t* __restrict__ rec)
{
	const int o = blockIdx.x * blockDim.x + threadIdx.x;
	if (8 * o >= npad) return;
	uint32_t any = 0;
	for (int k = 0; k < 8; k++) any |= rec[2 * (8 * o + k)];
	if (any & (kRecPrefix | kRecRoot)) rec[2 * (8 * o)] |= kRecSpecial;
}

// A state with too many hats gets no tables: the count stops the search early.
__global__ void hat_insert_kernel(int64_t nent, const uint32_t* __restrict__ ftab, HatTable* t, HatCount* cnt)
{
	const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= nent || __hip_atomic_load(&cnt->overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
	const uint32_t* e = ftab + 4 * k;
	if (!e[3]) return;
	const unsigned long long key = hat_key(e);
	uint32_t s = hat_slot(key);
	for (int p = 0; p < kHashProbes; p++, s = (s + 1) & (kHashSlots - 1))
	{
		unsigned long long old = __hip_atomic_load(&t->key[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		if (old == key) return;
		if (old == 0ull)
		{
			old = atomicCAS(&t->key[s], 0ull, key);
			if (old == 0ull && atomicAdd(&cnt->found, 1) >= kMaxHats - kHatFirst) cnt->overflow = 1;
			if (old == 0ull || old == key) return;
		}
	}
	cnt->overflow = 1;
}

// One workgroup of 1024 threads: ids in slot order, the hats' records, and
// whether the columns' largest values (2^14 to 2^15 iscale) lie in 2^-100 .. 2^100.
__global__ void __launch_bounds__(1024) hat_number_kernel(HatTable* t, HatCount* cnt, uint32_t* __restrict__ hat, int DP, const double* __restrict__ iscale)
{
	__shared__ int wsum[16];
	constexpr int kPer = kHashSlots / 1024;
	const int tid = threadIdx.x, lane = tid & 63;
	for (int c = tid; c < DP; c += 1024)
		if (iscale[c] < 0x1p-114 || iscale[c] > 0x1p+85) cnt->wide = 1;
	int mine = 0;
	for (int k = 0; k < kPer; k++) mine += t->key[tid * kPer + k] != 0ull;
	int x = mine;
	for (int off = 1; off < 64; off <<= 1)
	{
		const int y = __shfl_up(x, off, 64);
		if (lane >= off) x += y;
	}
	if (lane == 63) wsum[tid >> 6] = x;
	__syncthreads();
	int base = 0, total = 0;
	for (int w = 0; w < 16; w++)
	{
		if (w < (tid >> 6)) base += wsum[w];
		total += wsum[w];
	}
	int id = kHatFirst + base + x - mine;
	for (int k = 0; k < kPer; k++)
	{
		const int s = tid * kPer + k;
		const unsigned long long key = t->key[s];
		if (!key) continue;
		t->id[s] = (uint32_t)id;
		if (id < kMaxHats)
		{
			uint32_t* h = hat + 4 * id;
			h[0] = ((uint32_t)(key >> 44) & 63u) * 512u;
			h[1] = ((uint32_t)(key >> 32) & 0xfffu) << 20;
			h[2] = (uint32_t)key;
			h[3] = 0u;
		}
		id++;
	}
	if (tid == 0) cnt->total = kHatFirst + total;
}

__global__ void hat_lookup_kernel(int nno, int npad, int fstride, int hstride, const uint32_t* __restrict__ ftab, const HatTable* __restrict__ t,
	const HatCount* __restrict__ cnt, uint16_t* __restrict__ hid)
{
	const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= (int64_t)npad * hstride || cnt->overflow) return;
	const int64_t n = k / hstride;
	uint32_t id = n < nno ? kHatAll : kHatNone;
	if (id == kHatAll)
	{
		const uint32_t* e = ftab + 4 * (n * fstride + (k - n * hstride));
		if (e[3])
		{
			const unsigned long long key = hat_key(e);
			uint32_t s = hat_slot(key);
			for (int p = 0; p < kHashProbes && t->key[s] != key; p++) s = (s + 1) & (kHashSlots - 1);
			id = t->id[s];
		}
	}
	hid[k] = (uint16_t)(8 * id);
}

// The hat-table sweep's records, per op, from the hat ids of its node.
__global__ void table_rec_kernel(int nops, int npad, int hstride, const Op* __restrict__ ops, const uint16_t* __restrict__ hid,
	uint32_t* __restrict__ trec, uint16_t* __restrict__ thid, int32_t* __restrict__ tnode)
{
	const int q = blockIdx.x * blockDim.x + threadIdx.x;
	if (q >= npad) return;
	uint32_t v = kTabEmpty;
	int t = -1;
	const uint16_t* ids = hid;
	if (q < nops)
	{
		const Op op = ops[q];
		const uint32_t n = op.ctrl >> kOpNodeShift, n0 = ops[q & ~(kWin - 1)].ctrl >> kOpNodeShift;
		ids = hid + (size_t)n * hstride;
		t = op.ihi ? (int)(op.ctrl & 15u) : -1;   // the root's op has no factor
		const uint32_t id8 = t < 0 ? 8u * kHatAll : ids[t];
		v = ((id8 * 64u) & kTabRow) | (t < 0 ? 0u : 2u * (uint32_t)t) | (op.ctrl & kOpLast ? 0u : kTabPrefix)
			| ((n - n0) << kTabNodeShift);
		if (!(q & (kWin - 1))) tnode[q / kWin] = (int32_t)n;
	}
	trec[q] = v ^ kTabEmpty;
	for (int f = 0; f < hstride; f++)
		thid[(size_t)q * hstride + f] = q >= nops ? (uint16_t)(8 * kHatNone) : f <= t ? ids[f] : (uint16_t)(8 * kHatAll);
}

__global__ void odd_kernel(int64_t n, const double* __restrict__ s, HatCount* cnt)
{
	bool odd = false;
	for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
		odd |= !(fabs(s[k]) < __builtin_huge_val());
	if (odd) cnt->odd = 1;
}

int grid_for(int64_t n) { return (int)((n + 255) / 256); }

} // namespace

#define HIP_TRY(expr) do { hipError_t e_ = (expr); if (e_ != hipSuccess) return hip_fail(e_, #expr, __FILE__, __LINE__); } while (0)

// States with an index_i that is no power of two, or with more than kMaxHats
// hats, get no tables (hats = 0).
int build_direct_tables(StateDesc& d, bool centre_exact, const DeviceAlloc& alloc, const DeviceDrop& drop)
{
	d.hats = 0;
	if (!centre_exact) return HDDM_LB_SUCCESS;
	const int npad = (d.nno + kWin - 1) / kWin * kWin;
	const int fs = (int)d.fstride;
	const int hs = d.max_depth > 8 ? 16 : (d.max_depth + 1) / 2 * 2;   // at most fstride
	const int qpad = (d.nops + kWin - 1) / kWin * kWin;
	// One allocation, small next to the layout (each costs an upload of a few
	// thousand nodes some 5 %: measured with six more, 0.66 -> 0.86 ms). The
	// hat-table sweep's records of a small state take the hash's place.
	auto place = [](const size_t* bytes, int n, size_t* off) {
		off[0] = 0;
		for (int k = 0; k < n; k++) off[k + 1] = off[k] + (bytes[k] + 255) / 256 * 256;
	};
	const size_t bytes[] = { (size_t)npad * 8, (size_t)npad * hs * sizeof(uint16_t), (size_t)kMaxHats * 16, sizeof(HatTable) };
	const size_t tbytes[] = { (size_t)qpad * sizeof(uint32_t), (size_t)qpad * hs * sizeof(uint16_t), (size_t)(qpad / kWin) * sizeof(int32_t) };
	size_t off[5], toff[4];
	place(bytes, 4, off);
	place(tbytes, 3, toff);
	int rc = HDDM_LB_SUCCESS;
	char* const base = (char*)alloc(off[4], rc);
	if (rc) return rc;
	uint32_t* rec = (uint32_t*)(base + off[0]);
	uint16_t* hid = (uint16_t*)(base + off[1]);
	uint32_t* hat = (uint32_t*)(base + off[2]);
	HatCount* cnt = (HatCount*)hat;
	HatTable* t = (HatTable*)(base + off[3]);
	const hipStream_t st = nullptr;
	const int64_t nent = (int64_t)d.nno * fs;
	hipLaunchKernelGGL(rec_kernel, dim3(grid_for(d.nops > kHashSlots ? d.nops : kHashSlots)), dim3(256), 0, st, t, cnt, d.nno, npad,
		d.nops, d.ops, rec);
	const int64_t nsur = (int64_t)d.nno * d.dofs_pad;
	hipLaunchKernelGGL(odd_kernel, dim3(nsur < 2048 * 256 ? grid_for(nsur) : 2048), dim3(256), 0, st, nsur, d.s64, cnt);
	hipLaunchKernelGGL(hat_insert_kernel, dim3(grid_for(nent)), dim3(256), 0, st, nent, d.ftab, t, cnt);
	hipLaunchKernelGGL(prefix_kernel, dim3(grid_for((int64_t)d.nops * kWave)), dim3(256), 0, st, d.nno, d.nops, d.ops, rec);
	hipLaunchKernelGGL(special_kernel, dim3(grid_for(npad / 8)), dim3(256), 0, st, d.nno, npad, rec);
	hipLaunchKernelGGL(hat_number_kernel, dim3(1), dim3(1024), 0, st, t, cnt, hat, d.dofs_pad, d.iscale);
	hipLaunchKernelGGL(hat_lookup_kernel, dim3(grid_for((int64_t)npad * hs)), dim3(256), 0, st, d.nno, npad, fs, hs, d.ftab,
		(const HatTable*)t, (const HatCount*)cnt, hid);
	HIP_TRY(hipGetLastError());
	HatCount found = { 0, 0, 0, 0, 0 };
	HIP_TRY(hipMemcpy(&found, cnt, sizeof(found), hipMemcpyDeviceToHost));
	if (found.overflow || found.total > kMaxHats) { drop(base); return HDDM_LB_SUCCESS; }
	if (found.total <= kMaxTableHats && d.max_depth <= kTabMaxFactors)
	{
		char* const tb = toff[3] <= sizeof(HatTable) ? (char*)t : (char*)alloc(toff[3], rc);
		if (rc) return rc;
		d.trec = (uint32_t*)(tb + toff[0]);
		d.thid = (uint16_t*)(tb + toff[1]);
		d.tnode = (int32_t*)(tb + toff[2]);
		hipLaunchKernelGGL(table_rec_kernel, dim3(grid_for(qpad)), dim3(256), 0, st, d.nops, qpad, hs, d.ops, (const uint16_t*)hid,
			(uint32_t*)d.trec, (uint16_t*)d.thid, (int32_t*)d.tnode);
		HIP_TRY(hipGetLastError());
	}
	d.rec = rec;
	d.hid = hid;
	d.hat = hat;
	d.hstride = hs;
	d.f32_range = !found.wide;
	d.odd = found.odd;
	d.hats = found.total;
	return HDDM_LB_SUCCESS;
}

} // namespace hddm_lb
