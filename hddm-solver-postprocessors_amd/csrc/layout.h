// Device-side data layout of one uploaded state and of one forward call.
// Shared by the host library (capi.cpp, state.cpp) and the HIP kernels.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace hddm_lb {

// Points handled by one wave: one point per lane.
constexpr int kWave = 64;
// Nodes per MFMA chunk (the K extent of v_mfma_f32_32x32x16_*).
constexpr int kChunk = 16;
// Bytes of x staged per dim for one wave: 64 lanes x FP64.
constexpr int kXRowBytes = kWave * 8;
// Bits of the spatial sort key below the state id.
constexpr int kMortonBits = 40;

// One factor evaluation of the prefix-trie walk ("op"), 16 bytes, read by
// one scalar load. The ops of all nodes are stored in trie order; node n
// contributes one op per factor it does not share with node n-1.
//   dim    twice the dimension of x the factor reads (bits 0-7; the index of
//          its first 32-bit register in a bank of FP64 coordinates)
//          | (skip[op] - op) << 8
//   ctrl   depth t (bits 0-3) | last factor of its node (bit 4)
//          | relation to the previous op in the stream (bits 5-6)
//          | the op has children (bit 7) | node index << 8
//   ihi    high word of the FP64 value of i (the low word is 0)
//   njhi   high word of the FP64 value of -j (the low word is 0)
// The walk computes P[t+1] = P[t] * max(0, 1 - |x_dim * i - j|). When P[t+1]
// is zero on every lane, the run of nodes sharing the node's first t+1
// factors is skipped: skip[op] is the first op after that run.
// Relation (precomputed so the walk needs no depth compares): 0 the op is
// the first child of the previous op (its P[t] is the previous product),
// 1 a sibling (same P[t] as the previous op), 2 otherwise (P[t] is read from
// the path stack). After a skip of more than one op the target's stream
// predecessor is deeper, so its relation is 2 and the stack holds P[t].
// Children: P[t+1] is needed later only when the next op descends from this
// one, so only such ops store it on the stack.
// The device copies of ops and skip carry kOpPad sentinels after the stream.
struct Op
{
	uint32_t dim, ctrl, ihi, njhi;
};
constexpr uint32_t kOpLast = 16u;
constexpr int kOpRelShift = 5;
constexpr uint32_t kOpKids = 128u;
constexpr int kOpNodeShift = 8;
constexpr uint32_t kOpDimMask = 0xffu;
constexpr int kOpSkipShift = 8;
constexpr int kOpPad = 4;

// Dimension of x read by an op with dim word w (constexpr: host and device).
constexpr uint32_t op_dim(uint32_t w) { return (w & kOpDimMask) >> 1; }

struct StateDesc
{
	int dim, nno, dofs, dofs_pad;   // dofs_pad: dofs rounded up to 32
	int nops, nchunks;
	int nseg, max_depth;            // node segments (work-item split), max factors per node
	const Op* ops;                  // [nops + kOpPad]
	const uint32_t* skip;           // [nops + kOpPad]
	const int32_t* seg_op;          // [nseg + 1] first op of each segment
	const double* s64;              // [nno * dofs_pad] FP64 rows, trie order
	const uint16_t* s16;            // [nchunks][2][dofs_pad][16] f16 hi, lo (scaled)
	const uint16_t* sbf;            // [nchunks][3][dofs_pad][16] bf16 terms
	const float* s32;               // [nchunks][dofs_pad][2][8] f32
	const float* s32r;              // [nno * dofs_pad] f32 rows, trie order
	// Factors of every node (trie order), fstride slots of 16 bytes each:
	// {twice the dim, high word of i, high word of -j / i (the centre
	// negated), 1}, then {0, 0, 0, 0} padding (phi == 1 at u = 0, no
	// derivative). u = (x - j / i) i equals the op's fma(x, i, -j) bit for
	// bit: i is a power of two.
	const uint32_t* ftab;           // [nno rounded up to 32][fstride][4]
	int64_t fstride;
	const double* iscale;           // [dofs_pad] 2^-sigma_c undoing the f16 scaling
	const int32_t* order;           // trie position -> uploaded node index
	const uint64_t* lomask;         // [nno] dims whose support lies in [0, 1/2]
	const uint64_t* himask;         // [nno] dims whose support lies in [1/2, 1]
	int64_t ds_offset;              // first element of the state's rows in an adjoint dsurplus
	// Tables of the direct sweep (direct_tables.hip); hats == 0: the state has
	// none and runs on the walking sweeps.
	int hats, hstride;              // entries of hat; 16-bit ids per node in hid (2, 4, 6, 8 or 16)
	int odd;                        // a surplus is infinite or no number
	int f32_range;                  // largest value of every dof column 0 or within 2^-100 .. 2^100
	const uint32_t* rec;            // [nodes rounded up to 64][2], see kRec*
	const uint16_t* hid;            // [nodes rounded up to 64][hstride] 8 x the hat of each factor
	// of the hat-table sweep, per op, rounded up to windows of 64
	const uint32_t* trec;           // records, see kTab*
	const uint16_t* thid;           // [hstride] 8 x the hats of the op's path
	const int32_t* tnode;           // [windows] node of the window's first op
	const uint32_t* hat;            // [hats][4] {LDS byte offset of the coordinate row, i, -j / i, 0} (high words)
};

// Node record of the direct sweep: word 1 is the high word of -j of the node's
// last factor, word 0 packs the rest. i is a power of two, so the high word
// of its FP64 value has only the top 12 bits.
constexpr uint32_t kRecDepth2 = 0x1fu;    // twice the depth t of the last factor (P[t] is its parent product)
constexpr uint32_t kRecPrefix = 0x20u;    // a prefix of the node is no node itself: recompute them all
constexpr uint32_t kRecRoot = 0x40u;      // no factor: the basis is 1
constexpr uint32_t kRecSpecial = 0x80u;   // first node of eight: one of them has one of the two bits above
constexpr uint32_t kRecRow = 0x7e00u;     // LDS byte offset of the coordinate row (512 dim)
constexpr uint32_t kRecIhi = 0xfff00000u;
// The first two hat ids are no hats: no point (padding nodes) and every point
// (padding factors).
constexpr int kHatNone = 0;
constexpr int kHatAll = 1;
constexpr int kHatFirst = 2;
// Most hats of a state: 16 KB of masks in LDS.
constexpr int kMaxHats = 2048;
// Record of an op in the hat-table sweep: the row of its hat in LDS (512 bytes
// a row), twice its depth, its node's place after the window's first. The
// empty record is the row of zeros at the deepest depth, where no product is
// a parent's, and ends no node: it takes the surplus row of zeros, where a
// node's may be infinite or no number. Stored xor the empty record (0 is empty).
constexpr uint32_t kTabRow = 0x3fe00u;
constexpr uint32_t kTabDepth2 = 0xffu;    // alone in the low byte: GPR indexing reads that
constexpr uint32_t kTabPrefix = 0x40000u; // the op ends no node: it has no surplus
constexpr int kTabNodeShift = 20;
constexpr int kMaxTableHats = 512;
constexpr int kTabMaxFactors = 7;
constexpr uint32_t kTabEmpty = 2u * (kTabMaxFactors - 1) | kTabPrefix;
// Waves of the hat-table sweep's workgroup (one workgroup per CU).
constexpr int kTableWavesF32 = 12;
constexpr int kTableWavesFP64 = 8;
// Waves of the direct sweep's workgroup.
constexpr int kDirectWaves = 8;
// Nodes per selection window of the direct sweep: one node per lane.
constexpr int kWin = 64;

// Allocated rows of s64 and s32r: at least one past the last node.
constexpr size_t surplus_rows(int nno) { return ((size_t)nno / kWin + 1) * kWin; }
// Segments of one state in the direct and hat-table sweeps with g workgroups
// per block and nw waves each: at least a window per wave.
constexpr int sweep_nseg(int nops, int nw, int g)
{
	const int win = (nops + kWin - 1) / kWin;
	const int most = win < 2 * nw ? 1 : win / nw;
	return g < most ? g : most;
}
// Per-state plan of one forward call, written on the device by the plan kernel.
struct StatePlan
{
	int64_t start;         // first sorted position of the state's points
	int64_t count;         // number of points of the state
	int nblk;              // 64-point blocks
	int nseg;              // node segments of the state in this call
	int64_t item_base;     // first work item (items ordered by state cost)
	int64_t partial_base;  // element offset in the partial buffer (split states)
	int64_t dx_base;       // element offset in the adjoint's dx partial buffer (split states)
};
static_assert(sizeof(StatePlan) == 48, "counts towards the scratch of the allocation-free forward");

struct PlanHeader
{
	int64_t nitems;
	unsigned long long counter;   // work-queue head, reset by the plan kernel
	int64_t partial_elems;
	int64_t pad;
};

} // namespace hddm_lb
