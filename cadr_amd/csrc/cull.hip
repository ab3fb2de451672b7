// Frustum cull, LOD selection and per-StateSet stream compaction.
//
// The reference has no cull: processDrawables.comp emits every drawable and
// StateSet::recordToCommandBuffer draws StateSet k's full range
// [base_k, base_k + n_k) of the indirect buffer (src/CadR/StateSet.cpp:198-268).
// This pass keeps that range layout and writes, per view, the visible
// drawables of StateSet k compacted to the front of its range plus a draw
// count per StateSet (the operands of vkCmdDrawIndexedIndirectCount).
//
// Work is split into tiles of at most blockSize*itemsPerThread drawables that
// never cross a StateSet boundary; tiles are taken by atomic tickets in array
// order (dealt over several counters where small tiles need it, askTicket),
// so a tile waits on tiles that already run or come next, and what waits too
// long is finished at the end of the launch (finishLeft).  Within a
// tile, wave w owns a contiguous run of 64*itemsPerThread drawables (item j of
// lane l is drawable w*64*itemsPerThread + j*64 + l): loads are coalesced and
// the visibility of 64 drawables is one wave64 ballot.  Offsets come from a
// single-pass decoupled look-back: status words carry {epoch, state
// (aggregate / inclusive prefix), value}; the first tile of a StateSet
// publishes its inclusive prefix at once, and tiles are issued round-robin
// over StateSets, so the walks stay short.  Status words are tagged with a
// launch epoch and never cleared.
//
// Five kernels:
//   cullViewKernel - one view: one workgroup per tile, a 64-lane parallel
//     look-back in wave 0; each wave lists its visible drawables in LDS and
//     stores their commands with full lanes.  It resets its tickets and
//     advances the epoch itself (the last workgroup to finish), so a view
//     costs one launch.
//   cullViewLoopKernel - the same view pass as a persistent loop over tiles,
//     the next tile's loads in flight during the current tile's look-back
//     and stores; used when a view has more tiles than resident workgroups,
//     at the shapes where it is the faster one (viewLoopOf).
//   cullFusedKernel - the same for one view, with the tile's spheres computed
//     from the last transform level instead of read (cadrPropagateCullView).
//   cullKernel - many views and many scenes (jobs) in one persistent launch:
//     a tile is read from HBM once into registers and tested against all
//     views of its job, 64 views at a time; lane v of wave 0 walks the chain
//     of view v; each visible drawable's lane stores its command directly at
//     its compacted slot.  A conservative bounding sphere of a wave's items,
//     classified per view with lanes as views, lets whole (wave, view) pairs
//     skip the per-drawable test when the items are wholly outside or inside
//     the frustum.
//   cullFewKernel - jobs of few views, or small launches: work items of one
//     tile and up to four views, visible items listed per view; with one view
//     also the persistent kernel of the small tiles (viewLoopOf).
#include "internal.h"
#include "launch.h"
#include "fp32.h"
#include "matrix_io.h"

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <string>
#include <type_traits>
#include <type_traits>
#include <vector>

namespace cadr {

constexpr uint32_t kViewGroup = 64;   // views whose look-backs share one wave
constexpr uint32_t kMaxShards = 16;   // ctl words, each on its own 128-byte line
constexpr uint32_t kCtlShard = 0;     // + 64 g: tickets of shard g; + 64 g + 32: workgroups of shard g that left
constexpr uint32_t kCtlDone = kCtlShard + 64 * kMaxShards;  // shards whose workgroups all left
constexpr uint32_t kCtlEpoch = kCtlDone + 32;
constexpr uint32_t kCtlError = kCtlDone + 64;  // epoch of a launch whose look-back gave up, else 0
constexpr uint32_t kCtlWords = kCtlDone + 96;
constexpr uint32_t kLdsMeshes = 64;   // mesh tables up to this size are staged in LDS
constexpr uint64_t kDefaultWaitLimitUs = 1000000;  // 1 s: some ten thousand times a tile's run time

constexpr uint32_t kStateAggregate = 1;
constexpr uint32_t kStatePrefix = 2;
constexpr uint32_t kValueMask = 0x3fffffffu;

// The leaf transform level of a fused propagation + one-view cull launch
// (cadrPropagateCullView): node i of the level is drawable i of the job.
struct LeafParams {
	uint64_t local;        // float mat4[numDrawables]
	uint64_t parentIndex;  // uint32[numDrawables]; unused for a root level
	uint64_t parentWorld;  // float mat4[parentCount], 0 for a root level
	uint64_t world;        // float mat4[numDrawables], written
	uint64_t spheres;      // float4[numDrawables], written if not 0
	uint32_t parentCount;
};

struct CullParams {
	const cadrCullJob* jobs;
	const uint32_t* firstWork;   // [numJobs+1] prefix of the jobs' work items, more than kInlineJobs jobs only
	const uint64_t* statusBase;  // [numJobs] prefix of numViews*numTiles, likewise
	uint64_t* status;
	uint32_t* ctl;
	uint32_t shardShift;  // log2 of the ticket shards; beside ctl, so that the first ticket waits for one load
	uint32_t numJobs;
	uint32_t totalWork;
	uint32_t splitTiles;  // batched: a job's last tiles handed out per view group
	uint32_t groupShift;  // batched: log2 of the views of such a group
	uint32_t flags;
	uint64_t waitLimit;                 // steady-counter ticks a look-back may wait
	LeafParams leaf;                    // one-view fused kernel
	const cadrTransformLevel* leaves;   // fused batched kernel: leaf level of each job
};

// Addresses read from descriptors would be generic (FLAT) pointers, and a
// FLAT access counts on both the vector-memory and the LDS counters: every
// LDS wait would then also wait for outstanding output stores.  All device
// memory is therefore accessed through global (addrspace 1) pointers, and
// read-only descriptors (jobs, tiles, views, offsets) through constant
// (addrspace 4) pointers, which become scalar loads when the address is
// uniform.
template <class T>
using gptr = const __attribute__((address_space(1))) T*;
template <class T>
using gmut = __attribute__((address_space(1))) T*;
template <class T>
using cptr = const __attribute__((address_space(4))) T*;
template <class T>
__device__ __forceinline__ gptr<T> globalPtr(uint64_t a)
{
	return reinterpret_cast<gptr<T>>(a);
}
template <class T>
__device__ __forceinline__ gmut<T> globalMut(uint64_t a)
{
	return reinterpret_cast<gmut<T>>(a);
}
template <class T>
__device__ __forceinline__ cptr<T> constPtr(uint64_t a)
{
	return reinterpret_cast<cptr<T>>(a);
}
template <class T>
__device__ __forceinline__ uint64_t addr(const T* p)
{
	return reinterpret_cast<uint64_t>(p);
}

struct TileDesc {
	uint32_t start, count, segBase, k, chain;
	bool first, last;
};

// Loads item j = base + 64*j of a tile for every j, all issued before any is
// used: indices are clamped into the tile (a partial tile re-reads its last
// drawable), so no load sits behind a per-lane branch; an empty tile loads
// nothing.  Callers mask items at or beyond T.count.
template <int ITEMS>
__device__ __forceinline__ void loadTileItems(gptr<float4> spheres, gptr<uint32_t> meshIndex, const TileDesc& T,
                                              uint32_t base, float4 (&sp)[ITEMS], uint32_t (&mi)[ITEMS])
{
	if (T.count == 0) {
#pragma unroll
		for (int j = 0; j < ITEMS; j++) {
			sp[j] = make_float4(0.f, 0.f, 0.f, 0.f);
			mi[j] = 0;
		}
		return;
	}
	const uint32_t last = T.count - 1;
#pragma unroll
	for (int j = 0; j < ITEMS; j++) {
		const uint32_t e = min(base + uint32_t(j) * 64u, last);
		const gptr<float4> p = spheres + (T.start + e);
		sp[j] = make_float4(p->x, p->y, p->z, p->w);
		mi[j] = meshIndex[T.start + e];
	}
}

// Job descriptor j, field by field through a constant pointer (scalar loads).
static_assert(offsetof(cadrCullJob, numDrawables) == 56 && sizeof(cadrCullJob) == 80, "cadrCullJob layout");
__device__ __forceinline__ cadrCullJob loadJob(const cadrCullJob* jobs, uint32_t j)
{
	const uint64_t a = addr(jobs) + uint64_t(j) * sizeof(cadrCullJob);
	const cptr<uint64_t> q = constPtr<uint64_t>(a);
	const cptr<uint32_t> w = constPtr<uint32_t>(a + 56);
	cadrCullJob J;
	J.spheres = q[0]; J.meshIndex = q[1]; J.meshes = q[2]; J.tiles = q[3];
	J.views = q[4]; J.commands = q[5]; J.counts = q[6];
	J.numDrawables = w[0]; J.numTiles = w[1]; J.numStateSets = w[2];
	J.numViews = w[3]; J.commandStride = w[4]; J.numMeshes = w[5];
	return J;
}

// Leaf level of job j for the fused batched kernel (cadrTransformLevel in
// device memory, scalar loads); the parent count applies to a non-root level
// only, as in the one-view fused entry point.
static_assert(offsetof(cadrTransformLevel, numMeshes) == 64 && offsetof(cadrTransformLevel, parentCount) == 68 &&
                  sizeof(cadrTransformLevel) == 72,
              "cadrTransformLevel layout");
__device__ __forceinline__ LeafParams loadLeaf(const cadrTransformLevel* leaves, uint32_t j)
{
	const uint64_t a = addr(leaves) + uint64_t(j) * sizeof(cadrTransformLevel);
	const cptr<uint64_t> q = constPtr<uint64_t>(a);
	LeafParams L;
	L.local = q[0];
	L.parentIndex = q[1];
	L.parentWorld = q[2];
	L.world = q[3];
	L.spheres = q[7];
	L.parentCount = L.parentWorld ? constPtr<uint32_t>(a + 68)[0] : 0u;
	return L;
}

__device__ __forceinline__ TileDesc loadTile(const cadrCullJob& J, uint32_t t, uint32_t tileSize)
{
	const cptr<uint32_t> p = constPtr<uint32_t>(J.tiles) + 8 * uint64_t(t);
	const uint32_t flags = p[3];
	TileDesc d;
	d.start = p[0];
	d.count = p[1];
	d.segBase = p[2];
	d.k = flags & CADR_TILE_STATESET_MASK;
	d.first = (flags & CADR_TILE_FIRST) != 0u;
	d.last = (flags & CADR_TILE_LAST) != 0u;
	d.chain = p[4];
	if (d.chain >= J.numTiles) d.chain = t;  // malformed list: keep status accesses in range
	if (d.start >= J.numDrawables) d.count = 0;
	else if (d.count > J.numDrawables - d.start) d.count = J.numDrawables - d.start;
	if (d.count > tileSize) d.count = tileSize;
	return d;
}

// Per-view constants: scalar loads when the view index is uniform, vector
// loads when each lane takes its own view.
struct ViewC {
	float4 r0, r1, r2;
	float nearZ, farZ, sx0, sx1, sy0, sy1, lodScale, th0, th1, th2;
};

__device__ __forceinline__ ViewC loadView(uint64_t views, uint32_t v)
{
	// cadrView: viewRow[3][4], nearZ, farZ, sideX[2], sideY[2], lodScale, lodThreshold[3]
	const cptr<float> p = constPtr<float>(views + uint64_t(v) * sizeof(cadrView));
	ViewC c;
	c.r0 = make_float4(p[0], p[1], p[2], p[3]);
	c.r1 = make_float4(p[4], p[5], p[6], p[7]);
	c.r2 = make_float4(p[8], p[9], p[10], p[11]);
	c.nearZ = p[12]; c.farZ = p[13]; c.sx0 = p[14]; c.sx1 = p[15];
	c.sy0 = p[16]; c.sy1 = p[17]; c.lodScale = p[18]; c.th0 = p[19];
	c.th1 = p[20]; c.th2 = p[21];
	return c;
}

// glm mat4*vec4 order with w = 1: (m0*x + m1*y) + (m2*z + m3).
__device__ __forceinline__ float viewCoord(float4 r, float4 s)
{
	return (r.x * s.x + r.y * s.y) + (r.z * s.z + r.w);
}

// Sphere against the frustum, exactly the expression documented in cadr_hip.h.
__device__ __forceinline__ bool sphereVisible(float4 s, const ViewC& v)
{
	const float vx = viewCoord(v.r0, s);
	const float vy = viewCoord(v.r1, s);
	const float vz = viewCoord(v.r2, s);
	const bool nearOk = (vz + s.w >= v.nearZ);
	const bool farOk = (vz - s.w <= v.farZ);
	const bool xOk = (fabsf(vx) * v.sx0 - vz * v.sx1 <= s.w);
	const bool yOk = (fabsf(vy) * v.sy0 - vz * v.sy1 <= s.w);
	return nearOk & farOk & xOk & yOk;
}

// Highest LOD index of a mesh with lodCount LODs (lodCount clamped to 1..4).
__device__ __forceinline__ uint32_t maxLodOf(uint32_t lodCount)
{
	return (lodCount >= 1u ? (lodCount <= 4u ? lodCount : 4u) : 1u) - 1u;
}

__device__ __forceinline__ uint32_t lodAtDepth(float r, float vz, const ViewC& v, uint32_t maxLod)
{
	const float p = r * v.lodScale;
	const uint32_t lod = uint32_t(p < v.th0 * vz) + uint32_t(p < v.th1 * vz) + uint32_t(p < v.th2 * vz);
	return lod < maxLod ? lod : maxLod;
}

// Class of a wave's items in a view: 0 = test each drawable, 1 = all outside,
// 2 = all inside.
//
// ts is a sphere containing every drawable sphere of the wave's part of a
// tile (|c_i - C| + r_i <= R).  Each quantity the drawable test compares, v.z and
// g(c) = |v.x|*sideX[0] - v.z*sideX[1] (the larger of two linear plane
// functions), is Lipschitz in the sphere centre with constant L_P = the
// largest gradient norm among its linear pieces: |row2| for v.z, and
// |sideX[0]*row0 -+ sideX[1]*row2| for g (likewise for y), taken at least 1.
// A drawable's quantity then differs from the sphere centre's by at most
// L*|c_i - C| <= L*(R - r_i), so the items are wholly outside a plane when the
// centre is outside by more than L*R, and wholly inside when inside by more
// than L*R.  The norms are rounded up by a relative 2^-12; the margin m,
// about 2^-14 of the magnitudes involved, is some thousand times the FP32
// rounding of the per-drawable expressions, so the float test of every
// drawable agrees with the class.
// Bounds only: the hardware square root (within 1 ulp) is covered by the
// relative slack the callers add.
__device__ __forceinline__ float norm3(float x, float y, float z)
{
	return __builtin_amdgcn_sqrtf((x * x + y * y) + z * z);
}

__device__ __forceinline__ uint32_t classifyItems(float4 ts, const ViewC& v)
{
	const float vx = viewCoord(v.r0, ts);
	const float vy = viewCoord(v.r1, ts);
	const float vz = viewCoord(v.r2, ts);
	const float4 a = v.r0, b = v.r1, c = v.r2;
	float L = fmaxf(1.0f, norm3(c.x, c.y, c.z));
	L = fmaxf(L, norm3(v.sx0 * a.x - v.sx1 * c.x, v.sx0 * a.y - v.sx1 * c.y, v.sx0 * a.z - v.sx1 * c.z));
	L = fmaxf(L, norm3(v.sx0 * a.x + v.sx1 * c.x, v.sx0 * a.y + v.sx1 * c.y, v.sx0 * a.z + v.sx1 * c.z));
	L = fmaxf(L, norm3(v.sy0 * b.x - v.sy1 * c.x, v.sy0 * b.y - v.sy1 * c.y, v.sy0 * b.z - v.sy1 * c.z));
	L = fmaxf(L, norm3(v.sy0 * b.x + v.sy1 * c.x, v.sy0 * b.y + v.sy1 * c.y, v.sy0 * b.z + v.sy1 * c.z));
	L *= 1.0f + 1.0f / 4096.0f;
	const float R = ts.w * L * (1.0f + 1.0f / 4096.0f);
	const float mag = fabsf(ts.x) + fabsf(ts.y) + fabsf(ts.z) + ts.w + fabsf(v.r0.w) + fabsf(v.r1.w) +
	                  fabsf(v.r2.w) + fabsf(v.nearZ) + fabsf(v.farZ) + 1.0f;
	const float m = mag * L * (1.0f / 16384.0f);
	const float gx = fabsf(vx) * v.sx0 - vz * v.sx1;
	const float gy = fabsf(vy) * v.sy0 - vz * v.sy1;
	const bool out = (vz + R < v.nearZ - m) || (vz - R > v.farZ + m) || (gx > R + m) || (gy > R + m);
	if (out) return 1u;
	const bool in = (vz - R > v.nearZ + m) && (vz + R < v.farZ - m) && (gx + R < -m) && (gy + R < -m);
	return in ? 2u : 0u;
}

// Fused-multiply-add estimate of the drawable test: the smallest of the four
// inside margins (near, far, x sides, y sides; visible when all are >= 0),
// each computed with FMAs instead of the separately rounded glm expression.
// Its difference from the same margins taken on the glm-order values, plus the
// rounding that decides the glm-order comparisons, is below
// prefilterMargin(): when |planeMin| exceeds that bound its sign gives
// exactly the result of sphereVisible, else the caller evaluates
// sphereVisible.  Inputs: finite centres, radius finite >= 0 or -inf (then
// the centre is 0 and the result -inf, never visible); w0..w2 are the view's
// translation column (r0.w, r1.w, r2.w), passed separately so that a caller
// can keep them in vector registers (an FMA takes one scalar operand).
__device__ __forceinline__ float planeMin(float4 s, const ViewC& v, float w0, float w1, float w2)
{
	const float vx = __builtin_fmaf(v.r0.x, s.x, __builtin_fmaf(v.r0.y, s.y, __builtin_fmaf(v.r0.z, s.z, w0)));
	const float vy = __builtin_fmaf(v.r1.x, s.x, __builtin_fmaf(v.r1.y, s.y, __builtin_fmaf(v.r1.z, s.z, w1)));
	const float vz = __builtin_fmaf(v.r2.x, s.x, __builtin_fmaf(v.r2.y, s.y, __builtin_fmaf(v.r2.z, s.z, w2)));
	const float pn = (vz + s.w) - v.nearZ;
	const float pf = (v.farZ - vz) + s.w;
	const float px = __builtin_fmaf(-fabsf(vx), v.sx0, __builtin_fmaf(vz, v.sx1, s.w));
	const float py = __builtin_fmaf(-fabsf(vy), v.sy0, __builtin_fmaf(vz, v.sy1, s.w));
	return fminf(fminf(pn, pf), fminf(px, py));
}

// Bound for planeMin over spheres with |centre component| <= mc and radius
// <= w.  With u = 2^-24 and S_r = (|r.x|+|r.y|+|r.z|)*mc + |r.w| for view row
// r: each view coordinate differs between the FMA and the glm order by at
// most 6u*S_r; the FMA margins add at most 2u of their operands, and the glm
// comparisons are decided up to 2u of theirs, so every margin is within
// u*(10*(|side0|*S + |side1|*S_z) + 3*w + |near| + |far|) of a decisive one.
// The bound taken is 32u times the larger quantity
// ((1 + sum |side|) * (S_x+S_y+S_z) + w + |near| + |far|), plus 2^-100
// against underflow; it is NaN or infinite when a view constant is, and the
// caller uses the estimate only when the bound is at most 2^100 (no operand
// then comes near overflow).
__device__ __forceinline__ float prefilterMargin(const ViewC& v, float mc, float w)
{
	const float sx = (fabsf(v.r0.x) + fabsf(v.r0.y) + fabsf(v.r0.z)) * mc + fabsf(v.r0.w);
	const float sy = (fabsf(v.r1.x) + fabsf(v.r1.y) + fabsf(v.r1.z)) * mc + fabsf(v.r1.w);
	const float sz = (fabsf(v.r2.x) + fabsf(v.r2.y) + fabsf(v.r2.z)) * mc + fabsf(v.r2.w);
	const float sides = 1.0f + fabsf(v.sx0) + fabsf(v.sx1) + fabsf(v.sy0) + fabsf(v.sy1);
	return (sides * (sx + sy + sz) + w + fabsf(v.nearZ) + fabsf(v.farZ)) * 0x1p-19f + 0x1p-100f;
}

__device__ __forceinline__ uint32_t laneId() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ __forceinline__ uint32_t maskRank(uint64_t m)
{
	return __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
}

__device__ __forceinline__ uint32_t uniform(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ void waveSync()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint64_t packStatus(uint32_t epoch, uint32_t state, uint32_t value)
{
	return (uint64_t(epoch) << 32) | (uint64_t(state) << 30) | uint64_t(value & kValueMask);
}

__device__ __forceinline__ void publish(uint64_t* p, uint64_t v)
{
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint64_t readStatus(const uint64_t* p)
{
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ bool statusReady(uint64_t s, uint32_t epoch)
{
	return uint32_t(s >> 32) == epoch && (uint32_t(s) >> 30) != 0u;
}

// Look-back waits are bounded.  In a well-formed tile list every
// predecessor holds an earlier ticket and is running or done, so a wait ends
// within one tile's run time, or is left to the end of the launch (kStuck
// below).  A caller-built list that names a predecessor
// no tile publishes (a non-FIRST tile whose chainIndex - 1 is missing) would
// wait forever; instead, a wait that lasts waitLimit ticks of the steady
// counter records the launch's epoch in the error word and gives up, and
// every later wait of the same launch gives up at its first unready poll.
// The launch then ends with unspecified outputs and the workspace reports
// CADR_ERROR_TIMEOUT (cadrCullWorkspaceCheck).  Epochs are never 0, so an
// error word of 0 means no wait gave up.
struct WaitBound {
	uint32_t* ctl;
	uint64_t limit;
	uint32_t epoch;
};

// Work tickets.  An atomic add on one address takes 11-12 ns on this GPU
// whichever workgroup issues it (measured: 1024 workgroups one each, 13.5 us;
// spread over 64 lines 2.9 us), so with one ticket counter a launch of small
// tiles was bound by it (15,300 tiles of 1024 drawables in 24 jobs: 221 us
// with one counter, 155 with 8; 1,206 such tiles of one view: 40 and 14 us).
// The work items are therefore dealt to up to kMaxShards counters
// in runs of 8 (item t belongs to shard (t / 8) mod S), and workgroup b takes
// tickets of shard (b / 8) mod S only.  Launches of one workgroup per item
// have exactly as many workgroups as items in every shard.
//
// Tickets order a shard's items, so the smallest unfinished item of a launch
// is always held by a running workgroup, whose predecessors are done, or is
// the next ticket of its shard.  Workgroups are dispatched round-robin over
// the XCDs, and (b / 8) spreads a shard over all of them, so each shard has
// running workgroups as soon as 8 S of the launch's workgroups run.
//
// Where fewer do (a stream held to some compute units, other streams' kernels
// on the rest), the ones that run would wait for tiles of shards that none of
// them serves.  A wait that lasts kStuckTicks therefore leaves its item: the
// item's total is published, so no other item waits for it, the workgroup
// ends and makes room or, a persistent one, goes on with tickets of whichever
// shard is furthest behind, and the last workgroup of the launch finishes what
// was left (finishLeft), when every total is published.  So a launch
// progresses with any number of workgroups running.
constexpr uint32_t kStuck = ~0u;         // for an exclusive prefix (30 bits)
constexpr uint64_t kStuckTicks = 100000; // 1 ms: some hundred times the usual wait, and as long as most other launches
constexpr uint64_t kStuckShare = 4;      // at most this part of the wait limit
constexpr uint32_t kAgainShare = 16;     // the part of that which a workgroup waits once it was stuck
constexpr uint32_t kLeftFlag = 1u << 31; // in a count of workgroups that left: one of them left an item

struct Shard {
	uint32_t shift;  // log2 of the launch's shards
	uint32_t g;      // this workgroup's shard
};

// Tiles of this many drawables never take more than one shard (shardShiftFor):
// their kernels hold no shard registers.
constexpr bool oneShard(uint32_t tile) { return tile * 20ull >= 150000u; }

template <uint32_t TILE>
__device__ __forceinline__ Shard homeShard(const CullParams& P)
{
	if constexpr (oneShard(TILE)) return Shard{0u, 0u};
	return Shard{P.shardShift, (blockIdx.x >> 3) & ((1u << P.shardShift) - 1u)};
}

// Work item of ticket r of a shard.
__device__ __forceinline__ uint32_t itemOfTicket(Shard s, uint32_t r)
{
	return ((((r >> 3) << s.shift) + s.g) << 3) + (r & 7u);
}

// The add's result is not waited for here (the address is kept from being
// known uniform, or the compiler turns the add into a wave reduction that
// waits for it), so other loads can be in flight beside it; itemOfTicket of
// the result is.
__device__ __forceinline__ uint32_t askTicket(const CullParams& P, Shard s)
{
	uint64_t a = addr(P.ctl + kCtlShard + 64u * s.g);
	asm volatile("" : "+v"(a));
	return __hip_atomic_fetch_add(globalMut<uint32_t>(a), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Resets the tickets and retires the launch's epoch, so the next launch on the
// workspace never sees this launch's status words as its own.
__device__ __forceinline__ void endLaunch(const CullParams& P, Shard s, uint32_t epoch)
{
	const uint32_t S = 1u << s.shift;
	if (S > 1u) atomicExch(&P.ctl[kCtlDone], 0u);
	for (uint32_t g = 0; g < S; g++) {
		atomicExch(&P.ctl[kCtlShard + 64u * g], 0u);
		atomicExch(&P.ctl[kCtlShard + 64u * g + 32u], 0u);
	}
	const uint32_t e = epoch + 1u;
	atomicExch(&P.ctl[kCtlEpoch], e == 0u ? 1u : e);
}

// Called by one wave of each workgroup when it has taken its last ticket and
// published its last status word.  The workgroups of a shard count among
// themselves, then the shards.  The launch's last workgroup ends it; if items
// were left on the way, it returns true instead, and the wave goes on to
// finishLaunch when its own commands are stored.
__device__ __forceinline__ bool signOff(const CullParams& P, Shard s, uint32_t epoch, uint32_t lane)
{
	bool left = false;
	if (lane == 0) {
		const uint32_t S = 1u << s.shift, runs = gridDim.x >> (s.shift + 3u), rest = gridDim.x & (8u * S - 1u);
		const uint32_t mine = 8u * runs + (rest > s.g * 8u ? min(rest - s.g * 8u, 8u) : 0u);
		uint32_t d = atomicAdd(&P.ctl[kCtlShard + 64u * s.g + 32u], 1u);
		bool last = (d & ~kLeftFlag) == mine - 1u;
		if (last && S > 1u) {
			const uint32_t shards = min(S, (gridDim.x + 7u) / 8u);
			if ((d & kLeftFlag) != 0u) (void)atomicOr(&P.ctl[kCtlDone], kLeftFlag);
			d = atomicAdd(&P.ctl[kCtlDone], 1u);
			last = (d & ~kLeftFlag) == shards - 1u;
		}
		left = last && (d & kLeftFlag) != 0u;
		if (last && !left) endLaunch(P, s, epoch);
	}
	return __ballot(left) != 0ull;
}

// Where a workgroup's tickets come from (kept by its wave 0).
struct Tickets {
	Shard s;
	bool roam;  // it was stuck: from the shard furthest behind

	__device__ __forceinline__ explicit Tickets(Shard home) : s(home), roam(false) {}

	// The next work item, at or past P.totalWork if there is none, to *item
	// (called by wave 0).  A roaming workgroup may be the last one that serves
	// its own shard, or any other, so it ends only when every shard is empty: a
	// shard whose last ticket another took between its look and its own ticket
	// is one less to look at.
	__device__ __forceinline__ void next(const CullParams& P, uint32_t lane, uint32_t* item)
	{
		if (!roam) {
			if (lane == 0) *item = itemOfTicket(s, askTicket(P, s));
			return;
		}
		for (;;) {
			uint64_t first = ~0ull;  // the smallest (item of a shard's next ticket, shard)
			if (lane < (1u << s.shift)) {
				const uint32_t r = __hip_atomic_load(&P.ctl[kCtlShard + 64u * lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				first = (uint64_t(itemOfTicket(Shard{s.shift, lane}, r)) << 32) | lane;
			}
#pragma unroll
			for (int off = 8; off >= 1; off >>= 1) {
				const uint64_t o = __shfl_xor(first, off);
				first = o < first ? o : first;
			}
			s.g = uniform(uint32_t(first));
			uint32_t t = uniform(uint32_t(first >> 32));
			if (t < P.totalWork) {
				t = 0;
				if (lane == 0) t = itemOfTicket(s, askTicket(P, s));
				t = uniform(t);
				if (t >= P.totalWork) continue;
			}
			if (lane == 0) *item = t;
			return;
		}
	}
};

// Called by a wave whose item is left (its total is published): marks the
// launch before the workgroup can sign off.
__device__ __forceinline__ void leaveItem(const CullParams& P, Shard home, uint32_t lane)
{
	if (lane == 0) (void)atomicOr(&P.ctl[kCtlShard + 64u * home.g + 32u], kLeftFlag);
	__threadfence();
}

// Whether and when a wait leaves its item.  Only launches of several shards
// need it, and only they may: an in-place fused launch, whose items cannot be
// computed again, takes one.  The time comes from the wait limit at hand:
// another kernel argument, loaded where a look-back begins, cost fused batches
// up to 1% (and loaded at the poll, from outside the caches, several us a poll).
struct NeverStuck {
	static constexpr bool kCan = false;
	bool again = false;
	uint32_t shift = 0;
};
struct MayBeStuck {
	static constexpr bool kCan = true;
	bool again;      // the workgroup was stuck before
	uint32_t shift;  // Shard::shift
};
template <int TILE>
using StuckFor = std::conditional_t<oneShard(TILE), NeverStuck, MayBeStuck>;

constexpr uint32_t kPollAgain = 0, kGiveUp = 1, kWaitLater = 2;

// Called after an unready poll; start is 0 until the first such poll.
template <class Stuck>
__device__ __forceinline__ uint32_t waitStep(const WaitBound& B, uint64_t& start, Stuck stuck)
{
	if (__hip_atomic_load(&B.ctl[kCtlError], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == B.epoch) return kGiveUp;
	const uint64_t now = uint64_t(wall_clock64());
	if (start == 0) {
		start = now == 0 ? 1 : now;
		return kPollAgain;
	}
	if constexpr (Stuck::kCan) {
		const uint64_t most = min(B.limit / kStuckShare, kStuckTicks);
		if (stuck.shift != 0u && now - start > (stuck.again ? most / kAgainShare : most)) return kWaitLater;
	}
	if (now - start <= B.limit) return kPollAgain;
	__hip_atomic_store(&B.ctl[kCtlError], B.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	return kGiveUp;
}

// Exclusive prefix of chain position c, one chain per lane: walk back over the
// predecessors adding aggregates until an inclusive prefix is found; position
// 0 ends the walk in any case, and a wait bounded as above ends it early
// (kStuck if it is left for later).
template <class Stuck>
__device__ __forceinline__ uint32_t lookBackSerial(const uint64_t* chain, uint32_t c, const WaitBound& B, Stuck stuck)
{
	uint32_t excl = 0;
	uint32_t p = c;
	uint64_t start = 0;
	while (p > 0) {
		--p;
		uint64_t s;
		for (;;) {
			s = readStatus(chain + p);
			if (statusReady(s, B.epoch)) break;
			if (const uint32_t step = waitStep(B, start, stuck)) return step == kWaitLater ? kStuck : excl;
			__builtin_amdgcn_s_sleep(1);
		}
		excl += uint32_t(s) & kValueMask;
		if ((uint32_t(s) >> 30) == kStatePrefix) break;
	}
	return excl;
}

// Exclusive prefix of chain position c with the whole wave: lane l reads
// position p-1-l, the walk stops at the nearest inclusive prefix, and 64
// predecessors cost one round trip.  Returns the same value in every lane
// (the give-up decision is made from wave-uniform values).
template <class Stuck>
__device__ __forceinline__ uint32_t lookBackWave(const uint64_t* chain, uint32_t c, const WaitBound& B, uint32_t lane,
                                                 Stuck stuck)
{
	uint32_t excl = 0;
	int64_t p = c;
	uint64_t start = 0;
	while (p > 0) {
		const int64_t idx = p - 1 - int64_t(lane);
		const uint64_t s = idx >= 0 ? readStatus(chain + idx) : packStatus(B.epoch, kStatePrefix, 0);
		const bool ready = statusReady(s, B.epoch);
		const uint64_t pmask = __ballot(ready && (uint32_t(s) >> 30) == kStatePrefix);
		const uint64_t nmask = __ballot(!ready);
		const uint32_t f = pmask ? uint32_t(__builtin_ctzll(pmask)) : 64u;
		const uint64_t need = f >= 63u ? ~0ull : ((2ull << f) - 1ull);
		if (nmask & need) {
			if (const uint32_t step = uniform(waitStep(B, start, stuck))) return step == kWaitLater ? kStuck : excl;
			__builtin_amdgcn_s_sleep(1);
			continue;
		}
		uint32_t v = lane <= f ? (uint32_t(s) & kValueMask) : 0u;
#pragma unroll
		for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
		excl += v;
		if (f < 64u) break;
		p -= 64;
	}
	return excl;
}

// lookBackWave for 64 / W chains at once: each run of W lanes walks its own
// chain with a window of W predecessors.  c is the lane's chain's position
// (0: nothing before it); returns the lane's chain's prefix.
template <uint32_t W, class Stuck>
__device__ __forceinline__ uint32_t lookBackGroups(const uint64_t* chain, uint32_t c, const WaitBound& B, uint32_t lane,
                                                   Stuck stuck)
{
	static_assert(W >= 2 && W <= 32 && (W & (W - 1)) == 0, "lanes a chain");
	constexpr uint32_t kAll = W == 32 ? ~0u : (1u << (W & 31u)) - 1u;
	const uint32_t l = lane & (W - 1u), shift = lane & ~(W - 1u);
	uint32_t excl = 0;
	int64_t p = c;
	uint64_t start = 0;
	while (__ballot(p > 0) != 0ull) {
		const int64_t idx = p - 1 - int64_t(l);
		const uint64_t s = idx >= 0 ? readStatus(chain + idx) : packStatus(B.epoch, kStatePrefix, 0);
		const bool ready = statusReady(s, B.epoch);
		const uint32_t pmask = uint32_t(__ballot(ready && (uint32_t(s) >> 30) == kStatePrefix) >> shift) & kAll;
		const uint32_t nmask = uint32_t(__ballot(!ready) >> shift) & kAll;
		const uint32_t f = pmask ? uint32_t(__builtin_ctz(pmask)) : W;
		const uint32_t need = f + 1u >= W ? kAll : ((2u << f) - 1u);
		const bool wait = p > 0 && (nmask & need) != 0u;
		uint32_t v = l <= f ? (uint32_t(s) & kValueMask) : 0u;
#pragma unroll
		for (uint32_t off = W / 2; off >= 1; off >>= 1) v += __shfl_xor(v, int(off));
		if (!wait && p > 0) {
			excl += v;
			p = f < W ? 0 : p - int64_t(W);
		}
		if (__ballot(wait) != 0ull) {
			const uint32_t step = uniform(waitStep(B, start, stuck));
			if (step == kGiveUp) return excl;
			if (step == kWaitLater && wait) {  // the other chains go on
				excl = kStuck;
				p = 0;
			}
			__builtin_amdgcn_s_sleep(1);
		}
	}
	return excl;
}

// The mesh table of a job: an LDS copy when it is small, else device memory.
// The LDS copy is field-major (dword f of mesh m at f*kLdsMeshes + m): with
// 64-byte records every mesh's copy of a field would sit in the same two LDS
// banks, and 64 lanes reading random meshes would serialise.
// cadrMesh dwords: 0-2 centre, 3 radius, 4 lodCount, 5 vertexOffset,
// 8-11 indexCount[4], 12-15 firstIndex[4]; the LDS copy holds the highest
// LOD index (maxLodOf(lodCount)) in place of dword 4.
struct MeshTable {
	const uint32_t* lds;
	gptr<cadrMesh> mem;
	bool inLds;
	__device__ __forceinline__ uint32_t field(uint32_t f, uint32_t m) const { return lds[f * kLdsMeshes + m]; }
};

// Command fields of mesh m at the LOD the view selects for a sphere of radius
// r at view depth vz.  LDS is a compile-time choice: a run-time branch
// between the two sources would make the compiler wait for every
// outstanding vector-memory operation (output stores included) where the
// branches join.
template <bool LDS>
__device__ __forceinline__ void meshCommand(const MeshTable& M, uint32_t m, float r, float vz, const ViewC& V,
                                            uint32_t& count, uint32_t& first, uint32_t& vofs)
{
	if constexpr (LDS) {
		const uint32_t lod = lodAtDepth(r, vz, V, M.field(4, m));
		count = M.field(8 + lod, m);
		first = M.field(12 + lod, m);
		vofs = M.field(5, m);
	} else {
		const gptr<cadrMesh> mesh = M.mem + m;
		const uint32_t lod = lodAtDepth(r, vz, V, maxLodOf(mesh->lodCount));
		count = mesh->indexCount[lod];
		first = mesh->firstIndex[lod];
		vofs = uint32_t(mesh->vertexOffset);
	}
}

// Local bounding sphere {centre, radius} of mesh m (m < numMeshes).
template <bool LDS>
__device__ __forceinline__ float4 meshSphere(const MeshTable& M, uint32_t m)
{
	if constexpr (LDS) {
		return make_float4(__uint_as_float(M.field(0, m)), __uint_as_float(M.field(1, m)),
		                   __uint_as_float(M.field(2, m)), __uint_as_float(M.field(3, m)));
	} else {
		return loadF4(reinterpret_cast<gptr<float4>>(M.mem + m));
	}
}

// Mesh table of a job staged in LDS, field-major (see MeshTable), when it is
// small: loads first, LDS stores when the caller has nothing else to start.
template <int BLOCK>
struct MeshStaging {
	static constexpr int N = (16 * kLdsMeshes + BLOCK - 1) / BLOCK;
	uint32_t x[N];
	uint32_t words;  // 0: not staged

	__device__ __forceinline__ bool load(const cadrCullJob& J, uint32_t tid)
	{
		words = J.numMeshes <= kLdsMeshes ? J.numMeshes * 16u : 0u;
		if (words != 0u) {
			const gptr<uint32_t> src = globalPtr<uint32_t>(J.meshes);
#pragma unroll
			for (int k = 0; k < N; k++) x[k] = src[min(tid + uint32_t(k) * BLOCK, words - 1u)];
		}
		return J.numMeshes <= kLdsMeshes;
	}
	__device__ __forceinline__ void store(uint32_t* sMeshes, uint32_t tid) const
	{
#pragma unroll
		for (int k = 0; k < N; k++) {
			const uint32_t i = tid + uint32_t(k) * BLOCK;
			if (i < words) sMeshes[(i % 16u) * kLdsMeshes + i / 16u] = i % 16u == 4u ? maxLodOf(x[k]) : x[k];
		}
	}
};

// The fused form of loadTileItems: the wave's items are computed from the
// leaf level instead of read, exactly as cadrPropagateTransforms computes
// them (world = parentWorld[parentIndex[i]] * local[i], a parent index at or
// past parentCount or a root level giving world = local; the world sphere of
// mesh meshIndex[i], or the empty sphere for an index outside the table).
// World matrices (and spheres, if requested) are stored on the way.  Item j
// of the lane is tile offset base + 64*j + lane; the wave's 64 local
// matrices of item j are one contiguous 4-KiB block, loaded lane-contiguous
// (each instruction one KiB) and redistributed through LDS.  Parent and mesh
// indices of all items are loaded first (clamped into the tile, like
// loadTileItems); with PREFETCH the local block and parent matrix of item
// j+1 are issued before item j is computed, so each item's loads overlap the
// previous item's work.  The batched kernel prefetches only with 8 items per
// thread (both sides measured, at kKernels): with 4 it runs 4 waves per SIMD
// and has no registers for it.
struct ItemLoads {
	float4 raw[4];  // this lane's 4 float4 of the wave's 4-KiB local block
	float4 P[4];    // this lane's parent world matrix, or with COOP its 4 float4 of the
	                // wave's parent block (issueParentLoads), staged through LDS before use
};

// Every load unconditional (indices clamped), so all are in flight at once;
// lanes past the tile end load the tile's last node again and nothing of
// theirs is stored.
template <bool COOP>
__device__ __forceinline__ void issueItemLoads(const LeafParams& Lf, uint64_t first, uint64_t end, uint32_t p,
                                               uint32_t lane, ItemLoads& d)
{
	const gptr<float4> local = globalPtr<float4>(Lf.local);
#pragma unroll
	for (int k = 0; k < 4; k++) {
		const uint32_t q = uint32_t(k) * 64u + lane;  // float4 index inside the block
		const uint64_t m = min(first + q / 4u, end - 1u);
		d.raw[k] = loadF4Stream(local + (4 * m + (q & 3u)));
	}
	if constexpr (COOP) {
		if (Lf.parentCount > 0) issueParentLoads(globalPtr<float4>(Lf.parentWorld), Lf.parentCount, p, lane, d.P);
	} else {
		const uint32_t pc = p < Lf.parentCount ? p : 0u;
		if (Lf.parentCount > 0) {
			const gptr<float4> parentWorld = globalPtr<float4>(Lf.parentWorld);
#pragma unroll
			for (int c = 0; c < 4; c++) d.P[c] = loadF4(parentWorld + (4 * uint64_t(pc) + c));
		}
	}
}

// store: write the world matrices (and spheres); a tile that several work
// items of one launch share is written by one of them.
// sphere(j, s) receives the lane's world sphere of item j, in order of j.
template <int ITEMS, bool LDS, bool PREFETCH = true, bool COOP = false, class Sink>
__device__ __forceinline__ void propagateTileItems(const LeafParams& Lf, const cadrCullJob& J, const TileDesc& T,
                                                   uint32_t base, uint32_t lane, float4* stage,
                                                   const MeshTable& meshes, Sink sphere, uint32_t (&mi)[ITEMS],
                                                   bool store = true)
{
	const float4 empty = make_float4(0.f, 0.f, 0.f, -__builtin_inff());
	if (T.count == 0) {
#pragma unroll
		for (int j = 0; j < ITEMS; j++) {
			sphere(j, empty);
			mi[j] = 0;
		}
		return;
	}
	const bool root = Lf.parentWorld == 0;
	const gptr<uint32_t> parentIndex = globalPtr<uint32_t>(Lf.parentIndex);
	const gptr<uint32_t> meshIndex = globalPtr<uint32_t>(J.meshIndex);
	const uint32_t last = T.count - 1;
	uint32_t pi[ITEMS];
#pragma unroll
	for (int j = 0; j < ITEMS; j++) {
		const uint32_t node = T.start + min(base + uint32_t(j) * 64u + lane, last);
		pi[j] = root ? ~0u : parentIndex[node];
		mi[j] = meshIndex[node];
	}
	const uint64_t end = uint64_t(T.start) + T.count;
	const gmut<float4> world = globalMut<float4>(Lf.world);
	// items whose 64 nodes all lie past the tile end come last and are empty
	const uint32_t items = base >= T.count ? 0u : min(uint32_t(ITEMS), (T.count - base + 63u) / 64u);
	ItemLoads next;
	if (PREFETCH && items > 0) issueItemLoads<COOP>(Lf, uint64_t(T.start) + base, end, pi[0], lane, next);
#pragma unroll
	for (int j = 0; j < ITEMS; j++) {
		if (uint32_t(j) >= items) {
			sphere(j, empty);
			continue;
		}
		const uint64_t first = uint64_t(T.start) + base + uint32_t(j) * 64u;
		const uint64_t i = first + lane;
		const bool live = i < end;
		ItemLoads cur;
		if constexpr (PREFETCH) {
			cur = next;
			if (uint32_t(j) + 1u < items)
				issueItemLoads<COOP>(Lf, first + 64u, end, pi[j + 1 < ITEMS ? j + 1 : j], lane, next);
		} else {
			issueItemLoads<COOP>(Lf, first, end, pi[j], lane, cur);
		}
		// redistribute the local block: lane l takes matrix l
#pragma unroll
		for (int k = 0; k < 4; k++) stage[stageSlot(uint32_t(k) * 64u + lane)] = cur.raw[k];
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
		float4 L[4], W[4], P[4];
#pragma unroll
		for (int c = 0; c < 4; c++) L[c] = stage[stageSlot(4 * lane + c)];
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
		// the parent block the same way: lane l gets its own parent
		if constexpr (COOP) {
			if (Lf.parentCount > 0) stageMatrices(stage, lane, cur.P, P);
		} else {
#pragma unroll
			for (int c = 0; c < 4; c++) P[c] = cur.P[c];
		}
		if (live && pi[j] < Lf.parentCount) {
			mat4Mul(P, L, W);
		} else {
#pragma unroll
			for (int c = 0; c < 4; c++) W[c] = L[c];
		}
		if (store) storeMatrices(world, first, end, stage, lane, W);
		float4 s = empty;
		if (live && mi[j] < J.numMeshes) s = sphereTransform(W, meshSphere<LDS>(meshes, mi[j]));
		if (store && Lf.spheres && live) storeF4(globalMut<float4>(Lf.spheres) + i, s);
		sphere(j, s);
		// without the prefetch, keep the scheduler from hoisting later items'
		// loads above this one (every item's 32 registers of loads at once)
		if constexpr (!PREFETCH) __builtin_amdgcn_sched_barrier(0);
	}
}

// ------------------------------------------------------- the end of a launch

// Makes an address one that the compiler takes for a lane's own, not known
// before `after` is.
__device__ __forceinline__ uint64_t perLane(uint64_t address, float after = 0.f)
{
	asm volatile("" : "+v"(address) : "v"(after));
	return address;
}

// One tile in one view from its status word on, by one wave and without the
// mesh table's LDS copy: what a workgroup left because its look-back was stuck.
// job, tile, view, leaf: addresses.  This code almost never runs, and scalar
// registers for its descriptors would cost the kernels a wave per SIMD: it
// reads them through perLane, the view row by row.
template <int TILE, bool FUSED>
__device__ __forceinline__ void finishTile(const CullParams& P, uint64_t job, uint64_t tile, uint64_t view, uint32_t v,
                                           const LeafParams& Lf, uint64_t* chain, uint32_t pos, uint32_t epoch,
                                           uint32_t lane)
{
	const uint32_t excl = lookBackWave(chain, pos, WaitBound{P.ctl, P.waitLimit, epoch}, lane, NeverStuck{});
	tile = perLane(tile);
	// loadTile's clamps
	const uint32_t start = globalPtr<uint32_t>(tile)[0], drawables = globalPtr<uint32_t>(perLane(job))[14];
	const uint32_t count =
	    uniform(start >= drawables ? 0u : min(min(globalPtr<uint32_t>(tile)[1], drawables - start), uint32_t(TILE)));
	uint32_t at = globalPtr<uint32_t>(tile)[2] + excl, total = 0;
#pragma unroll 1
	for (uint32_t e = 0; e < count; e += 64u) {
		uint64_t J = perLane(job);
		const uint32_t i = start + min(e + lane, count - 1u);
		const uint32_t m = globalPtr<uint32_t>(globalPtr<uint64_t>(J)[1])[i];
		const bool live = e + lane < count && m < globalPtr<uint32_t>(J)[19];
		float4 s = make_float4(0.f, 0.f, 0.f, -__builtin_inff());
		if constexpr (FUSED) {
			float4 L[4], W[4];
#pragma unroll
			for (int c = 0; c < 4; c++) W[c] = L[c] = loadF4(globalPtr<float4>(Lf.local) + (4 * uint64_t(i) + c));
			const uint32_t p = Lf.parentCount > 0 ? globalPtr<uint32_t>(Lf.parentIndex)[i] : ~0u;
			if (p < Lf.parentCount) {
				float4 A[4];
#pragma unroll
				for (int c = 0; c < 4; c++) A[c] = loadF4(globalPtr<float4>(Lf.parentWorld) + (4 * uint64_t(p) + c));
				mat4Mul(A, L, W);
			}
			if (live) s = sphereTransform(W, loadF4(globalPtr<float4>(globalPtr<uint64_t>(J)[2]) + 4 * uint64_t(m)));
		} else {
			s = loadF4(globalPtr<float4>(globalPtr<uint64_t>(J)[0]) + i);
		}
		// the test of sphereVisible
		const gptr<float> r2 = globalPtr<float>(perLane(view, s.w));
		const float vz = viewCoord(make_float4(r2[8], r2[9], r2[10], r2[11]), s);
		bool vis = live & (vz + s.w >= r2[12]) & (vz - s.w <= r2[13]);
		const gptr<float> r0 = globalPtr<float>(perLane(view, vz));
		const float vx = viewCoord(make_float4(r0[0], r0[1], r0[2], r0[3]), s);
		vis &= fabsf(vx) * r0[14] - vz * r0[15] <= s.w;
		const gptr<float> r1 = globalPtr<float>(perLane(view, vx));
		const float vy = viewCoord(make_float4(r1[4], r1[5], r1[6], r1[7]), s);
		vis &= fabsf(vy) * r1[16] - vz * r1[17] <= s.w;
		const uint64_t mask = __ballot(vis);
		const uint32_t slot = at + maskRank(mask);
		J = perLane(job, vy);
		if (vis && slot < globalPtr<uint32_t>(J)[18]) {
			ViewC V{};
			const gptr<float> lod = globalPtr<float>(perLane(view, vy)) + 18;
			V.lodScale = lod[0];
			V.th0 = lod[1];
			V.th1 = lod[2];
			V.th2 = lod[3];
			uint32_t n, first, vofs;
			meshCommand<false>(MeshTable{nullptr, globalPtr<cadrMesh>(globalPtr<uint64_t>(J)[2]), false}, m, s.w, vz, V, n,
			                   first, vofs);
			const gmut<uint32_t> o = globalMut<uint32_t>(globalPtr<uint64_t>(J)[5]) +
			                         (uint64_t(v) * globalPtr<uint32_t>(J)[18] + slot) * 5ull;
			o[0] = n;
			o[1] = 1u;
			o[2] = first;
			o[3] = vofs;
			o[4] = i;
		}
		at += uint32_t(__builtin_popcountll(mask));
		total += uint32_t(__builtin_popcountll(mask));
	}
	if (lane == 0) {
		publish(chain + pos, packStatus(epoch, kStatePrefix, excl + total));
		const uint64_t J = perLane(job);
		const uint32_t flags = globalPtr<uint32_t>(tile)[3], k = flags & CADR_TILE_STATESET_MASK, K = globalPtr<uint32_t>(J)[16];
		if ((flags & CADR_TILE_LAST) != 0u && k < K)
			globalMut<uint32_t>(globalPtr<uint64_t>(J)[6])[uint64_t(v) * K + k] = excl + total;
	}
}

// The items that the launch's workgroups left: every tile and view whose
// status word holds a total and no inclusive prefix.  Called by one wave of
// the last workgroup.  (A word whose prefix is still on its way here is
// finished again, with the same outputs.)
template <int TILE, bool FUSED>
__device__ __forceinline__ void finishLeft(const CullParams& P, uint32_t epoch, uint32_t lane)
{
	uint64_t* chain = P.status;
#pragma unroll 1
	for (uint32_t j = 0; j < P.numJobs; j++) {
		const uint64_t job = addr(P.jobs) + uint64_t(j) * sizeof(cadrCullJob);
		const uint32_t numTiles = uniform(globalPtr<uint32_t>(perLane(job))[15]);
		const uint32_t numViews = uniform(globalPtr<uint32_t>(perLane(job))[17]);
		LeafParams Lf{};
		if constexpr (FUSED) Lf = P.leaves ? loadLeaf(P.leaves, j) : P.leaf;
#pragma unroll 1
		for (uint32_t v = 0; v < numViews; v++, chain += numTiles) {
#pragma unroll 1
			for (uint32_t e = 0; e < numTiles; e += 64u) {
				const uint64_t tiles = globalPtr<uint64_t>(perLane(job))[3];
				uint64_t s = 0;
				uint32_t c = 0;
				if (e + lane < numTiles) {
					c = globalPtr<uint32_t>(tiles)[8 * uint64_t(e + lane) + 4];
					if (c >= numTiles) c = e + lane;  // as loadTile
					s = readStatus(chain + c);
				}
				uint64_t left = __ballot(uint32_t(s >> 32) == epoch && (uint32_t(s) >> 30) == kStateAggregate);
#pragma unroll 1
				for (; left != 0ull; left &= left - 1ull) {
					const uint32_t l = uniform(uint32_t(__builtin_ctzll(left)));
					finishTile<TILE, FUSED>(P, job, tiles + sizeof(cadrCullTile) * uint64_t(e + l),
					                        globalPtr<uint64_t>(perLane(job))[4] + uint64_t(v) * sizeof(cadrView), v, Lf, chain,
					                        uint32_t(__builtin_amdgcn_readlane(c, l)), epoch, lane);
				}
			}
		}
	}
}

// After signOff, by the wave for which it returned true.  The kernel's
// arguments (one CullParams) are loaded anew, so that none is held for this.
template <int TILE, bool FUSED>
__device__ __forceinline__ void finishLaunch(Shard s, uint32_t epoch, uint32_t lane)
{
	uint64_t a = reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr());
	asm volatile("" : "+s"(a));
	const cptr<CullParams> K = constPtr<CullParams>(a);
	CullParams P{};
	P.jobs = K->jobs;
	P.status = K->status;
	P.ctl = K->ctl;
	P.numJobs = K->numJobs;
	P.waitLimit = K->waitLimit;
	if constexpr (FUSED) {
		P.leaves = K->leaves;
		P.leaf = LeafParams{K->leaf.local, K->leaf.parentIndex, K->leaf.parentWorld, K->leaf.world, K->leaf.spheres,
		                    K->leaf.parentCount};
	}
	finishLeft<TILE, FUSED>(P, epoch, lane);
	if (lane == 0) endLaunch(P, s, epoch);
}

// ---------------------------------------------------------------- one view

// A wave's visible items as a compact list in its own LDS, in drawable order:
// item index in the wave's run (11 bits), the LOD its projected radius
// selects before the mesh's own limit (2 bits) and the mesh (19 bits; the
// meshes of a larger table are read again).  The command stores then run with full lanes: in
// drawable order a wave stored its items one by one, each with the few lanes
// that are visible, and the CU's address path, which takes a store
// instruction's 64 lanes whether they are active or not, bound the views that
// see a part of everything (10M drawables, 25% visible in every item: 49 MB
// of commands cost 57 of 85 us).
constexpr uint32_t kRunLodShift = 11, kRunMeshShift = 13;
constexpr uint32_t kRunMeshes = 1u << (32 - kRunMeshShift);

// LOD index by projected radius alone (lodAtDepth before the mesh's limit).
__device__ __forceinline__ uint32_t lodByRadius(float r, float vz, const ViewC& v)
{
	const float p = r * v.lodScale;
	return uint32_t(p < v.th0 * vz) + uint32_t(p < v.th1 * vz) + uint32_t(p < v.th2 * vz);
}

// Tests the wave's items (first item `base` of the tile) and lists the
// visible ones; returns their number (the same in every lane).
template <int ITEMS>
__device__ __forceinline__ uint32_t listVisible(const float4 (&sp)[ITEMS], const uint32_t (&mi)[ITEMS],
                                                const TileDesc& T, uint32_t numMeshes, const ViewC& V, uint32_t base,
                                                uint32_t lane, uint32_t* run)
{
	static_assert(64 * ITEMS <= (1 << kRunLodShift), "item index bits");
	waveSync();  // the list may lie where the wave's matrices were staged
	uint32_t n = 0;
#pragma unroll
	for (int j = 0; j < ITEMS; j++) {
		const bool vis = base + j * 64 + lane < T.count && mi[j] < numMeshes && sphereVisible(sp[j], V);
		const uint64_t mask = __ballot(vis);
		if (vis) {
			const uint32_t lod = lodByRadius(sp[j].w, viewCoord(V.r2, sp[j]), V);
			run[n + maskRank(mask)] = (j * 64 + lane) | (lod << kRunLodShift) | (mi[j] << kRunMeshShift);
		}
		n = uniform(n + uint32_t(__builtin_popcountll(mask)));
	}
	return n;
}

// Stores the commands of a wave's n listed items from output slot pos on, 64
// consecutive commands per pair of stores.  first: drawable index of the
// wave's item 0.
template <bool LDS>
__device__ __forceinline__ void storeListed(const uint32_t* run, uint32_t n, uint32_t pos, uint32_t first,
                                            const MeshTable& M, uint32_t numMeshes, gptr<uint32_t> meshIndex,
                                            gmut<uint32_t> out, uint32_t stride, uint32_t lane)
{
	waveSync();  // the list is written by other lanes
	for (uint32_t c = 0; c < n; c += 64u) {
		const uint32_t i = c + lane;
		if (i >= n || pos + i >= stride) continue;
		const uint32_t e = run[i];
		const uint32_t drawable = first + (e & ((1u << kRunLodShift) - 1u)), raw = (e >> kRunLodShift) & 3u;
		uint32_t count, firstIndex, vofs;
		if constexpr (LDS) {
			const uint32_t m = e >> kRunMeshShift;
			const uint32_t lod = min(raw, M.field(4, m));
			count = M.field(8 + lod, m);
			firstIndex = M.field(12 + lod, m);
			vofs = M.field(5, m);
		} else {
			// the whole record at once, so that one round trip serves the LOD limit and its fields
			const uint32_t m = numMeshes <= kRunMeshes ? e >> kRunMeshShift : meshIndex[drawable];
			const gptr<uint4> q = reinterpret_cast<gptr<uint4>>(M.mem + m);
			const uint4 head = make_uint4(q[1].x, q[1].y, q[1].z, q[1].w);  // lodCount, vertexOffset
			const uint4 c4 = make_uint4(q[2].x, q[2].y, q[2].z, q[2].w), f4 = make_uint4(q[3].x, q[3].y, q[3].z, q[3].w);
			const uint32_t lod = min(raw, maxLodOf(head.x));
			count = lod == 0u ? c4.x : lod == 1u ? c4.y : lod == 2u ? c4.z : c4.w;
			firstIndex = lod == 0u ? f4.x : lod == 1u ? f4.y : lod == 2u ? f4.z : f4.w;
			vofs = head.y;
		}
		const gmut<uint32_t> o = out + uint64_t(pos + i) * 5ull;
		o[0] = count;
		o[1] = 1u;
		o[2] = firstIndex;
		o[3] = vofs;
		o[4] = drawable;
	}
	waveSync();  // read before the next tile's list replaces it
}

// Look-back of a tile by wave 0, from the waves' counts; the exclusive prefix
// goes to *sExclP and a StateSet's last tile writes its count.
template <int WAVES, int TILE>
__device__ __forceinline__ void tileOffset(const CullParams& P, const cadrCullJob& J, const TileDesc& T, uint32_t epoch,
                                           Shard home, Tickets& tickets, const uint32_t* sCnt, uint32_t* sExclP,
                                           uint32_t lane)
{
	uint32_t total = 0;
#pragma unroll
	for (int q = 0; q < WAVES; q++) total += sCnt[q];
	uint64_t* chain = P.status;
	uint32_t excl = 0;
	if (T.first) {
		if (lane == 0) publish(chain + T.chain, packStatus(epoch, kStatePrefix, total));
	} else {
		if (lane == 0) publish(chain + T.chain, packStatus(epoch, kStateAggregate, total));
		excl = lookBackWave(chain, T.chain, WaitBound{P.ctl, P.waitLimit, epoch}, lane, StuckFor<TILE>{tickets.roam, home.shift});
		if (excl == kStuck) {
			leaveItem(P, home, lane);
			tickets.roam = true;
			*sExclP = kStuck;
			return;
		}
		if (lane == 0) publish(chain + T.chain, packStatus(epoch, kStatePrefix, excl + total));
	}
	if (lane == 0) {
		*sExclP = excl;
		if (T.last && T.k < J.numStateSets) globalMut<uint32_t>(J.counts)[T.k] = excl + total;
	}
}

// Returns signOff's result in the wave that called it, else false.
template <int BLOCK, int ITEMS, bool LDS, bool FUSED>
__device__ __forceinline__ bool cullViewTile(const CullParams& P, const cadrCullJob& J, uint32_t t, uint32_t epoch,
                                             Shard shard, const MeshTable& meshes, uint32_t* sCnt, uint32_t* sExclP,
                                             float4* sMat, uint32_t* run, uint32_t lane, uint32_t wave)
{
	constexpr int WAVES = BLOCK / 64, WAVE_ITEMS = 64 * ITEMS;
	const TileDesc T = loadTile(J, t, BLOCK * ITEMS);
	const ViewC V = loadView(J.views, 0);
	const gptr<float4> spheres = globalPtr<float4>(J.spheres);
	const gptr<uint32_t> meshIndex = globalPtr<uint32_t>(J.meshIndex);

	// all loads first (indices clamped into the tile, so none is conditional),
	// then the tests: a wave keeps ITEMS 16-byte loads in flight at once; the
	// fused form computes the spheres from the leaf level instead
	float4 sp[ITEMS];
	uint32_t mi[ITEMS];
	if constexpr (FUSED)
		propagateTileItems<ITEMS, LDS>(P.leaf, J, T, wave * WAVE_ITEMS, lane, sMat, meshes,
		                               [&](int j, float4 q) __attribute__((always_inline)) { sp[j] = q; }, mi);
	else
		loadTileItems<ITEMS>(spheres, meshIndex, T, wave * WAVE_ITEMS + lane, sp, mi);
	const uint32_t n = listVisible<ITEMS>(sp, mi, T, J.numMeshes, V, wave * WAVE_ITEMS, lane, run);
	if (lane == 0) sCnt[wave] = n;
	__syncthreads();
	Tickets tickets(shard);
	if (wave == 0) tileOffset<WAVES, BLOCK * ITEMS>(P, J, T, epoch, shard, tickets, sCnt, sExclP, lane);
	__syncthreads();
	// the workgroup is done with the launch's tickets and status words: the
	// last wave signs off while the others store, so that no wave waits for
	// its stores behind the atomics
	bool left = false;
	if (wave == WAVES - 1) left = signOff(P, shard, epoch, lane);

	uint32_t pos = T.segBase + *sExclP;
	for (uint32_t q = 0; q < wave; q++) pos += sCnt[q];
	storeListed<LDS>(run, *sExclP == kStuck ? 0u : n, uniform(pos), T.start + wave * WAVE_ITEMS, meshes, J.numMeshes,
	                 meshIndex, globalMut<uint32_t>(J.commands), J.commandStride, lane);
	return left;
}

template <int BLOCK, int ITEMS, bool FUSED>
__device__ __forceinline__ void cullViewBody(const CullParams& P)
{
	constexpr int WAVES = BLOCK / 64;
	// a wave's 4-KiB matrix staging, done with before its list is written
	__shared__ float4 sMat[WAVES][FUSED ? 256 : 16 * ITEMS];
	__shared__ uint32_t sTicket;
	__shared__ uint32_t sCnt[WAVES];
	__shared__ uint32_t sExcl;
	__shared__ uint32_t sMeshes[16 * kLdsMeshes];

	const uint32_t tid = threadIdx.x, lane = laneId(), wave = tid / 64;
	const Shard shard = homeShard<BLOCK * ITEMS>(P);
	// ticket, epoch and mesh table in flight together
	uint32_t ticket = 0;
	if (tid == 0) ticket = askTicket(P, shard);
	const uint32_t epoch = __hip_atomic_load(&P.ctl[kCtlEpoch], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	const cadrCullJob J = loadJob(P.jobs, 0);
	MeshStaging<BLOCK> staging;
	const bool ldsMeshes = staging.load(J, tid);
	if (tid == 0) sTicket = itemOfTicket(shard, ticket);
	staging.store(sMeshes, tid);
	__syncthreads();
	const uint32_t t = uniform(sTicket);
	const MeshTable meshes{sMeshes, globalPtr<cadrMesh>(J.meshes), ldsMeshes};
	bool left = false;
	if (t >= P.totalWork) {
		if (wave == 0) left = signOff(P, shard, epoch, lane);
	} else {
		float4* mat = sMat[wave];
		uint32_t* run = reinterpret_cast<uint32_t*>(mat);
		if (ldsMeshes)
			left = cullViewTile<BLOCK, ITEMS, true, FUSED>(P, J, t, epoch, shard, meshes, sCnt, &sExcl, mat, run, lane, wave);
		else
			left = cullViewTile<BLOCK, ITEMS, false, FUSED>(P, J, t, epoch, shard, meshes, sCnt, &sExcl, mat, run, lane, wave);
	}
	if constexpr (!oneShard(BLOCK * ITEMS))
		if (left) finishLaunch<BLOCK * ITEMS, FUSED>(shard, epoch, lane);
}

template <int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void cullViewKernel(CullParams P)
{
	cullViewBody<BLOCK, ITEMS, false>(P);
}

// The one-view cull as a persistent loop: each workgroup stages the mesh
// table once and then takes tiles by ticket until none is left.  The next
// tile's ticket and its loads are issued right after the current tile's
// items are listed, into the same registers, so they are in flight during
// the current tile's look-back and stores.  Counts and the exclusive prefix
// alternate between two LDS buffers, so two barriers per tile suffice.
// Results are those of cullViewTile: the same tests, the same compaction
// order.  Launched with one workgroup per resident slot when a view has more
// tiles than that; a view of fewer tiles takes one tile per workgroup
// (cullViewKernel), which saves the loop's extra ticket and barrier.
template <int BLOCK, int ITEMS, bool LDS>
__device__ __forceinline__ bool cullViewTiles(const CullParams& P, const cadrCullJob& J, uint32_t t, uint32_t epoch,
                                              Shard shard, const MeshTable& meshes, uint32_t* sTicket,
                                              uint32_t (*sCnt)[BLOCK / 64], uint32_t* sExcl, uint32_t* run,
                                              uint32_t tid, uint32_t lane, uint32_t wave)
{
	constexpr int WAVES = BLOCK / 64, WAVE_ITEMS = 64 * ITEMS;
	const ViewC V = loadView(J.views, 0);
	const gptr<float4> spheres = globalPtr<float4>(J.spheres);
	const gptr<uint32_t> meshIndex = globalPtr<uint32_t>(J.meshIndex);
	const gmut<uint32_t> out = globalMut<uint32_t>(J.commands);
	TileDesc T = loadTile(J, t, BLOCK * ITEMS);
	float4 sp[ITEMS];
	uint32_t mi[ITEMS];
	loadTileItems<ITEMS>(spheres, meshIndex, T, wave * WAVE_ITEMS + lane, sp, mi);
	Tickets tickets(shard);
	for (uint32_t b = 0;; b ^= 1u) {
		const uint32_t n = listVisible<ITEMS>(sp, mi, T, J.numMeshes, V, wave * WAVE_ITEMS, lane, run);
		if (lane == 0) sCnt[b][wave] = n;
		if (wave == 0) tickets.next(P, lane, sTicket);
		__syncthreads();

		// the next tile's loads, in flight through this tile's look-back and stores
		const uint32_t tn = uniform(*sTicket);
		const bool more = tn < P.totalWork;
		const TileDesc Tc = T;
		if (more) {
			T = loadTile(J, tn, BLOCK * ITEMS);
			loadTileItems<ITEMS>(spheres, meshIndex, T, wave * WAVE_ITEMS + lane, sp, mi);
		}
		if (wave == 0) tileOffset<WAVES, BLOCK * ITEMS>(P, J, Tc, epoch, shard, tickets, sCnt[b], &sExcl[b], lane);
		__syncthreads();

		bool left = false;
		if (!more && wave == WAVES - 1) left = signOff(P, shard, epoch, lane);  // as in cullViewTile

		uint32_t pos = Tc.segBase + sExcl[b];
		for (uint32_t q = 0; q < wave; q++) pos += sCnt[b][q];
		storeListed<LDS>(run, sExcl[b] == kStuck ? 0u : n, uniform(pos), Tc.start + wave * WAVE_ITEMS, meshes, J.numMeshes,
		                 meshIndex, out, J.commandStride, lane);
		if (!more) return left;
	}
}

template <int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void cullViewLoopKernel(CullParams P)
{
	constexpr int WAVES = BLOCK / 64;
	__shared__ uint32_t sTicket;
	__shared__ uint32_t sRun[WAVES][64 * ITEMS];
	__shared__ uint32_t sCnt[2][WAVES];
	__shared__ uint32_t sExcl[2];
	__shared__ uint32_t sMeshes[16 * kLdsMeshes];

	const uint32_t tid = threadIdx.x, lane = laneId(), wave = tid / 64;
	const Shard shard = homeShard<BLOCK * ITEMS>(P);
	// ticket, epoch and mesh table in flight together
	uint32_t ticket = 0;
	if (tid == 0) ticket = askTicket(P, shard);
	const uint32_t epoch = __hip_atomic_load(&P.ctl[kCtlEpoch], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	const cadrCullJob J = loadJob(P.jobs, 0);
	MeshStaging<BLOCK> staging;
	const bool ldsMeshes = staging.load(J, tid);
	if (tid == 0) sTicket = itemOfTicket(shard, ticket);
	staging.store(sMeshes, tid);
	__syncthreads();
	const uint32_t t = uniform(sTicket);
	__syncthreads();  // every wave has read the first ticket before the loop rewrites it
	const MeshTable meshes{sMeshes, globalPtr<cadrMesh>(J.meshes), ldsMeshes};
	bool left = false;
	if (t >= P.totalWork) {
		if (wave == 0) left = signOff(P, shard, epoch, lane);
	} else if (ldsMeshes) {
		left = cullViewTiles<BLOCK, ITEMS, true>(P, J, t, epoch, shard, meshes, &sTicket, sCnt, sExcl, sRun[wave], tid, lane,
		                                        wave);
	} else {
		left = cullViewTiles<BLOCK, ITEMS, false>(P, J, t, epoch, shard, meshes, &sTicket, sCnt, sExcl, sRun[wave], tid, lane,
		                                         wave);
	}
	if constexpr (!oneShard(BLOCK * ITEMS))
		if (left) finishLaunch<BLOCK * ITEMS, false>(shard, epoch, lane);
}

// The fused kernel is latency-bound (a chain of dependent loads per item), so
// occupancy pays: WPE waves per SIMD is requested from the register allocator
// (4 for the small item counts, where it costs no spills).  Larger workgroups
// give each wave fewer items, so the chain per tile is shorter.
template <int BLOCK, int ITEMS, int WPE>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE))) void cullFusedKernel(CullParams P)
{
	cullViewBody<BLOCK, ITEMS, true>(P);
}

// ------------------------------------------------------- many views, jobs

// Work items of a job in a batched launch: its tiles, plus one more per
// extra view group for each of its last splitTiles tiles (workItem's rule).
// A job without views has nothing to test and owns no status words: no items,
// except in a fused launch (leaves), which writes its leaf level.
// The host checks that a launch's total fits 32 bits.
__host__ __device__ __forceinline__ uint64_t jobWorkItems(uint32_t numTiles, uint32_t numViews, uint32_t splitTiles,
                                                          uint32_t groupShift, bool leaves)
{
	if (numViews == 0 && !leaves) return 0;
	const uint64_t groups = (uint64_t(numViews) + (1u << groupShift) - 1) >> groupShift;
	const uint64_t split = groups > 1 ? (numTiles < splitTiles ? numTiles : splitTiles) : 0u;
	return numTiles + split * (groups - 1);
}

// Item u of a job: a whole tile for every view, or, among the job's last
// split tiles, one tile for one group of views (tile-major, so a tile's
// look-back predecessors still hold earlier tickets).
// Every field is made explicitly uniform: view constants loaded by an index
// that the compiler cannot prove uniform go to vector registers (measured:
// 216 against 159 registers, 2.5M drawables x 256 views 600 against 397 us).
struct WorkItem {
	uint32_t tile, viewBegin, viewEnd;
};

__device__ __forceinline__ WorkItem workItem(const CullParams& P, const cadrCullJob& J, uint32_t u)
{
	const uint32_t g = 1u << P.groupShift;
	const uint32_t groups = (J.numViews >> P.groupShift) + ((J.numViews & (g - 1u)) != 0u ? 1u : 0u);
	const uint32_t split = groups > 1 ? min(J.numTiles, P.splitTiles) : 0u;
	const uint32_t whole = J.numTiles - split;
	uint32_t t = u, begin = 0, end = J.numViews;
	if (u >= whole) {
		const uint32_t q = u - whole;
		t = whole + q / groups;
		begin = (q % groups) << P.groupShift;
		end = begin + min(J.numViews - begin, g);
	}
	return WorkItem{uniform(t), uniform(begin), uniform(end)};
}

// Where each job's work items and status words begin.  Up to kInlineJobs jobs
// every workgroup works the offsets out for itself at its start, one wave
// with lanes as jobs, from the same descriptors: about 1 us of a workgroup's
// time, where a kernel of its own before the batched one cost 4-5 us of every
// launch.  More jobs take that kernel (cullSetupKernel).
constexpr uint32_t kInlineJobs = 256;

struct JobOffsets {
	uint32_t firstWork[kInlineJobs];
	uint64_t statusBase[kInlineJobs];
};

// Fills O (wave 0; a barrier must follow before it is read).
__device__ __forceinline__ void findJobOffsets(const CullParams& P, JobOffsets& O, uint32_t lane)
{
	uint32_t runW = 0;
	uint64_t runS = 0;
	for (uint32_t base = 0; base < P.numJobs; base += 64u) {
		const uint32_t j = base + lane;
		uint32_t w = 0;
		uint64_t st = 0;
		if (j < P.numJobs) {
			const gptr<uint32_t> q = globalPtr<uint32_t>(addr(P.jobs) + uint64_t(j) * sizeof(cadrCullJob) + 56);
			const uint32_t tiles = q[1], views = q[3];
			w = uint32_t(jobWorkItems(tiles, views, P.splitTiles, P.groupShift, P.leaves != nullptr));
			st = uint64_t(views) * tiles;
		}
		uint32_t wi = w;
		uint64_t si = st;
#pragma unroll
		for (int off = 1; off < 64; off <<= 1) {
			const uint32_t a = __shfl_up(wi, off);
			const uint64_t b = __shfl_up(si, off);
			if (lane >= uint32_t(off)) {
				wi += a;
				si += b;
			}
		}
		if (j < P.numJobs) {
			O.firstWork[j] = runW + wi - w;
			O.statusBase[j] = runS + si - st;
		}
		runW += __shfl(wi, 63);
		runS += __shfl(si, 63);
	}
}

// The job of work item w, the last one whose items begin at or before it:
// with lanes as jobs where the offsets are inline, else by bisection upward
// from `job` (a workgroup's tickets only grow).
__device__ __forceinline__ uint32_t jobOfWork(const CullParams& P, const JobOffsets& O, uint32_t w, uint32_t job,
                                              uint32_t lane)
{
	if (P.numJobs == 1) return 0;
	if (P.numJobs <= kInlineJobs) {
		uint32_t n = 0;
		for (uint32_t base = 0; base < P.numJobs; base += 64u) {
			const uint32_t j = base + lane;
			n += uint32_t(__builtin_popcountll(__ballot(j < P.numJobs && O.firstWork[j] <= w)));
		}
		return uniform(n - 1u);
	}
	uint32_t lo = job, hi = P.numJobs - 1;
	while (lo < hi) {
		const uint32_t mid = (lo + hi + 1) / 2;
		if (constPtr<uint32_t>(addr(P.firstWork))[mid] <= w) lo = mid; else hi = mid - 1;
	}
	return uniform(lo);
}

__device__ __forceinline__ uint32_t firstWorkOf(const CullParams& P, const JobOffsets& O, uint32_t job)
{
	if (P.numJobs == 1) return 0;
	if (P.numJobs <= kInlineJobs) return uniform(O.firstWork[job]);
	return constPtr<uint32_t>(addr(P.firstWork))[job];
}

__device__ __forceinline__ uint64_t statusBaseOf(const CullParams& P, const JobOffsets& O, uint32_t job)
{
	if (P.numJobs == 1) return 0;
	if (P.numJobs <= kInlineJobs) {
		const uint64_t v = O.statusBase[job];
		return uint64_t(uniform(uint32_t(v))) | (uint64_t(uniform(uint32_t(v >> 32))) << 32);
	}
	return constPtr<uint64_t>(addr(P.statusBase))[job];
}

// Jobs of few views: the batched kernel without what only many views pay
// for.  No bounding sphere, no visibility bits kept per view: the workgroup
// lists the visible items of a work item's views (up to CH), wave 0 looks
// their chains back at once, and the commands are stored from the lists.  It
// holds less than half the batched kernel's registers, so more workgroups are
// resident to overlap their chains of round trips.  Persistent, like the
// batched kernel; the mesh table is staged where the launch has one job.
//
// With DEFER (one or two views) the look-back runs one item behind: a
// workgroup publishes an item's totals as soon as they are known, starts the
// next item's loads and only then looks back and stores the item before.  No
// published total ever waits for a look-back, so look-backs find their
// predecessors published and the loads are in flight all the time; without
// it, a next ticket held that early keeps its followers waiting (24 served
// scenes, 256 x 4: 118 us against 96.6, and 99.4 with the ticket taken last;
// 256 x 2: 179 / 121 / 139).  Four views take the ticket last: two lists of
// four views would halve the workgroups a CU holds.
template <int BLOCK, int ITEMS, int CH, bool DEFER>
struct FewShared {
	static constexpr int WAVES = BLOCK / 64;
	uint32_t run[DEFER ? 2 : 1][WAVES][CH][64 * ITEMS];
	uint32_t meshes[16 * kLdsMeshes];
	JobOffsets offsets;
	uint32_t cnt[2][CH][WAVES];
	uint32_t excl[2][CH];
	uint32_t ticket[2];
};

// A work item as its workgroup holds it: the job, the tile, the views and
// where their chains begin.
struct FewItem {
	cadrCullJob J;
	TileDesc T;
	uint32_t viewBegin, viewEnd;
	uint64_t* chain0;
};

template <bool JOBS>
__device__ __forceinline__ FewItem fewItem(const CullParams& P, const JobOffsets& offsets, const cadrCullJob& only,
                                           uint32_t t, uint32_t tile, uint32_t& job, uint32_t lane)
{
	FewItem f;
	if constexpr (JOBS) {
		job = jobOfWork(P, offsets, t, job, lane);
		f.J = loadJob(P.jobs, job);
		t -= firstWorkOf(P, offsets, job);
		f.chain0 = P.status + statusBaseOf(P, offsets, job);
	} else {
		f.J = only;
		f.chain0 = P.status;
	}
	const WorkItem item = workItem(P, f.J, t);
	f.T = loadTile(f.J, item.tile, tile);
	f.viewBegin = item.viewBegin;
	f.viewEnd = item.viewEnd;
	return f;
}

// The lane's view of an item in wave 0's look-back: 64 / CH lanes a view.
template <int CH>
struct FewChain {
	uint64_t* chain;
	uint32_t view;
	bool on, lead;
	__device__ __forceinline__ FewChain(const FewItem& f, uint32_t lane)
	{
		constexpr uint32_t W = 64 / CH;
		view = f.viewBegin + lane / W;
		on = view < f.viewEnd;
		lead = on && lane % W == 0u;
		chain = f.chain0 + uint64_t(on ? view : f.viewBegin) * f.J.numTiles + f.T.chain;
	}
};

// Wave 0: publishes an item's totals (per lane: its view's).
template <int CH>
__device__ __forceinline__ void fewPublish(const FewItem& f, uint32_t total, uint32_t epoch, uint32_t lane)
{
	const FewChain<CH> c(f, lane);
	if (c.lead) publish(c.chain, packStatus(epoch, f.T.first ? kStatePrefix : kStateAggregate, total));
}

// Wave 0: an item's exclusive prefixes, published as inclusive ones, to excl[].
template <int CH>
__device__ __forceinline__ void fewLookBack(const CullParams& P, const FewItem& f, uint32_t total, uint32_t epoch,
                                            Shard home, Tickets& tickets, uint32_t* excl, uint32_t lane)
{
	const FewChain<CH> c(f, lane);
	uint32_t e = 0;
	if (!f.T.first) {
		const WaitBound B{P.ctl, P.waitLimit, epoch};
		const MayBeStuck stuck{tickets.roam, home.shift};
		if constexpr (CH == 1)
			e = lookBackWave(c.chain - f.T.chain, c.on ? f.T.chain : 0u, B, lane, stuck);
		else
			e = lookBackGroups<64 / CH>(c.chain - f.T.chain, c.on ? f.T.chain : 0u, B, lane, stuck);
		if (__ballot(c.on && e == kStuck) != 0ull) {
			leaveItem(P, home, lane);
			tickets.roam = true;
		}
		if (c.lead && e != kStuck) publish(c.chain, packStatus(epoch, kStatePrefix, e + total));
	}
	if (c.lead) {
		excl[lane / (64 / CH)] = e;
		if (e != kStuck && f.T.last && f.T.k < f.J.numStateSets)
			globalMut<uint32_t>(f.J.counts)[uint64_t(c.view) * f.J.numStateSets + f.T.k] = e + total;
	}
}

// Every wave: its commands of an item, n[c] of them per view from slot off[c]
// of the tile's run on.
template <int CH, bool LDS, int N>
__device__ __forceinline__ void fewStore(const FewItem& f, const MeshTable& staged, const uint32_t (*run)[N],
                                         const uint32_t (&n)[CH], const uint32_t (&off)[CH], const uint32_t* excl,
                                         uint32_t wave, uint32_t lane)
{
	const MeshTable meshes{staged.lds, globalPtr<cadrMesh>(f.J.meshes), LDS};
#pragma unroll
	for (int c = 0; c < CH; c++) {
		if (n[c] == 0 || excl[c] == kStuck) continue;
		const uint32_t pos = uniform(f.T.segBase + excl[c] + off[c]);
		storeListed<LDS>(run[c], n[c], pos, f.T.start + wave * N, meshes, f.J.numMeshes, globalPtr<uint32_t>(f.J.meshIndex),
		                 globalMut<uint32_t>(f.J.commands) + uint64_t(f.viewBegin + c) * f.J.commandStride * 5ull,
		                 f.J.commandStride, lane);
	}
}

// Returns signOff's result in the wave that called it, else false.
template <int BLOCK, int ITEMS, int CH, bool DEFER, bool JOBS, bool LDS>
__device__ __forceinline__ bool cullFewItems(const CullParams& P, FewShared<BLOCK, ITEMS, CH, DEFER>& sh,
                                             const cadrCullJob& only, uint32_t t, Shard shard, uint32_t epoch, uint32_t tid,
                                             uint32_t lane, uint32_t wave)
{
	constexpr int WAVES = BLOCK / 64, WAVE_ITEMS = 64 * ITEMS;
	const MeshTable staged{sh.meshes, nullptr, LDS};
	uint32_t job = 0;
	FewItem cur = fewItem<JOBS>(P, sh.offsets, only, t, BLOCK * ITEMS, job, lane), prev = cur;
	float4 sp[ITEMS];
	uint32_t mi[ITEMS], nPrev[CH], offPrev[CH], totalPrev = 0;
	loadTileItems<ITEMS>(globalPtr<float4>(cur.J.spheres), globalPtr<uint32_t>(cur.J.meshIndex), cur.T,
	                     wave * WAVE_ITEMS + lane, sp, mi);
	bool pending = false;
	Tickets tickets(shard);
	for (uint32_t b = 0;; b ^= 1u) {
		asm volatile("" : "+v"(lane));  // nothing derived from it stays in registers across tiles
		uint32_t n[CH], off[CH];
#pragma unroll
		for (int c = 0; c < CH; c++) {
			n[c] = 0;
			if (cur.viewBegin + c < cur.viewEnd)
				n[c] = listVisible<ITEMS>(sp, mi, cur.T, cur.J.numMeshes, loadView(cur.J.views, cur.viewBegin + c),
				                          wave * WAVE_ITEMS, lane, sh.run[DEFER ? b : 0][wave][c]);
			if (lane == 0) sh.cnt[b][c][wave] = n[c];
		}
		if (DEFER && wave == 0) tickets.next(P, lane, &sh.ticket[b]);
		__syncthreads();
		FewItem next;
		bool more = false;
		auto takeNext = [&](FewItem& f) __attribute__((always_inline)) {
			const uint32_t tn = uniform(sh.ticket[b]);
			more = tn < P.totalWork;
			if (more) {
				f = fewItem<JOBS>(P, sh.offsets, only, tn, BLOCK * ITEMS, job, lane);
				loadTileItems<ITEMS>(globalPtr<float4>(f.J.spheres), globalPtr<uint32_t>(f.J.meshIndex), f.T,
				                     wave * WAVE_ITEMS + lane, sp, mi);
			}
		};
		// the next item's loads, in flight through the look-back and the stores
		if constexpr (DEFER) takeNext(next);
#pragma unroll
		for (int c = 0; c < CH; c++) {
			off[c] = 0;
			for (uint32_t q = 0; q < wave; q++) off[c] += sh.cnt[b][c][q];
			off[c] = uniform(off[c]);
		}
		uint32_t total = 0;
		if (wave == 0) {
			for (int q = 0; q < WAVES; q++) total += sh.cnt[b][lane / (64 / CH)][q];
			fewPublish<CH>(cur, total, epoch, lane);
			if constexpr (DEFER) {
				if (pending) fewLookBack<CH>(P, prev, totalPrev, epoch, shard, tickets, sh.excl[b], lane);
			} else {
				fewLookBack<CH>(P, cur, total, epoch, shard, tickets, sh.excl[b], lane);
			}
		}
		__syncthreads();
		if constexpr (DEFER) {
			if (pending) fewStore<CH, LDS, WAVE_ITEMS>(prev, staged, sh.run[b ^ 1u][wave], nPrev, offPrev, sh.excl[b], wave, lane);
			if (!more) {
				if (wave == 0) fewLookBack<CH>(P, cur, total, epoch, shard, tickets, sh.excl[b ^ 1u], lane);
				__syncthreads();
				bool left = false;
				if (wave == WAVES - 1) left = signOff(P, shard, epoch, lane);
				fewStore<CH, LDS, WAVE_ITEMS>(cur, staged, sh.run[b][wave], n, off, sh.excl[b ^ 1u], wave, lane);
				return left;
			}
			prev = cur;
			totalPrev = total;
			pending = true;
#pragma unroll
			for (int c = 0; c < CH; c++) {
				nPrev[c] = n[c];
				offPrev[c] = off[c];
			}
			cur = next;
		} else {
			fewStore<CH, LDS, WAVE_ITEMS>(cur, staged, sh.run[0][wave], n, off, sh.excl[b], wave, lane);
			if (wave == 0) tickets.next(P, lane, &sh.ticket[b]);
			__syncthreads();
			takeNext(cur);
			if (!more) break;
		}
	}
	return wave == 0 && signOff(P, shard, epoch, lane);
}

// (256 x 8 with one view takes one register more than the 6 waves its LDS allows)
template <int BLOCK, int ITEMS, int CH, bool DEFER, bool JOBS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(ITEMS == 8 && CH == 1 ? 6 : 1))) void cullFewKernel(CullParams P)
{
	__shared__ FewShared<BLOCK, ITEMS, CH, DEFER> sh;
	const uint32_t tid = threadIdx.x, lane = laneId(), wave = uniform(tid / 64);
	const Shard shard = homeShard<BLOCK * ITEMS>(P);
	uint32_t ticket = 0;
	if (tid == 0) ticket = askTicket(P, shard);
	const uint32_t epoch = __hip_atomic_load(&P.ctl[kCtlEpoch], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	bool ldsMeshes = false;
	cadrCullJob only{};
	if constexpr (JOBS) {
		if (wave == 0 && P.numJobs <= kInlineJobs) findJobOffsets(P, sh.offsets, lane);
	} else {
		only = loadJob(P.jobs, 0);
		MeshStaging<BLOCK> staging;
		ldsMeshes = staging.load(only, tid);
		staging.store(sh.meshes, tid);
	}
	if (tid == 0) sh.ticket[1] = itemOfTicket(shard, ticket);
	__syncthreads();
	const uint32_t t = uniform(sh.ticket[1]);
	bool left = false;
	if (t >= P.totalWork) {
		if (wave == 0) left = signOff(P, shard, epoch, lane);
	} else if (!JOBS && ldsMeshes) {
		left = cullFewItems<BLOCK, ITEMS, CH, DEFER, JOBS, true>(P, sh, only, t, shard, epoch, tid, lane, wave);
	} else {
		left = cullFewItems<BLOCK, ITEMS, CH, DEFER, JOBS, false>(P, sh, only, t, shard, epoch, tid, lane, wave);
	}
	if (left) finishLaunch<BLOCK * ITEMS, false>(shard, epoch, lane);
}

template <int BLOCK, int ITEMS>
struct CullShared {
	static constexpr int WAVES = BLOCK / 64;
	static constexpr int TILE = BLOCK * ITEMS;

	uint32_t cnt[kViewGroup][WAVES];
	uint32_t base[kViewGroup][WAVES];  // a wave's first output slot in its view's StateSet segment

	uint32_t meshes[16 * kLdsMeshes];
	uint32_t ticket[2];
	JobOffsets offsets;
};

// COOP (fused form only): parent matrices read whole, 16 per instruction
// (issueParentLoads), for leaves whose parents are scattered; it holds more
// registers, so it is chosen per shape, like WPE, the waves per SIMD asked of
// the register allocator (see the kernel table; unfused, 256 x 8 and 256 x 4
// take a register or two more than 3 and 4 waves leave them: 2.5M drawables x
// 256 views 488 us with 2 waves at 256 x 8, 407 with 3).
template <int BLOCK, int ITEMS, bool FUSED, bool COOP = false,
          int WPE = BLOCK != 256 ? 1 : ITEMS == 8 ? 3 : ITEMS == 4 ? 4 : 1>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE))) void cullKernel(CullParams P)
{
	using S = CullShared<BLOCK, ITEMS>;
	constexpr int WAVES = S::WAVES;
	constexpr int WAVE_ITEMS = 64 * ITEMS;
	__shared__ S sh;
	// the fused form keeps its spheres here instead of in registers, which
	// computing them needs: with the spheres in registers it held 237 (256 x 8)
	// and ran 2 waves per SIMD, its view loop at half the VALU's rate (64 uneven
	// scenes 977 us, now 867 with 3 waves; 512 x 4 1238 and 881 with 4)
	__shared__ float4 sSpheres[FUSED ? WAVES : 1][FUSED ? WAVE_ITEMS : 1];

	const uint32_t tid = threadIdx.x;
	uint32_t lane = laneId();
	const uint32_t wave = uniform(tid / 64);
	const uint32_t epoch = __hip_atomic_load(&P.ctl[kCtlEpoch], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	const Shard shard = homeShard<S::TILE>(P);
	uint32_t job = 0, stagedJob = ~0u;
	// the first ticket's barrier stands between this and the first use
	if (wave == 0 && P.numJobs > 1 && P.numJobs <= kInlineJobs) findJobOffsets(P, sh.offsets, lane);

	// Two tickets in turn: the barriers of an item's body are inside its view
	// groups, so without them a wave could still have to read one ticket when
	// thread 0 writes the next; it has read it by that one's barrier.
	// (Wave 0's b also holds Tickets::roam.)
	constexpr uint32_t kRoam = 2;
	for (uint32_t b = 0;; b ^= 1u) {
		if (wave == 0) {
			Tickets tickets(shard);
			tickets.roam = (b & kRoam) != 0u;
			tickets.next(P, lane, &sh.ticket[b & 1u]);
		}
		__syncthreads();
		const uint32_t w = uniform(sh.ticket[b & 1u]);
		if (w >= P.totalWork) break;
		// a lane index of its own for each tile: the compiler otherwise keeps
		// dozens of addresses derived from it in registers across tiles
		if constexpr (FUSED) asm volatile("" : "+v"(lane));

		job = jobOfWork(P, sh.offsets, w, job, lane);
		const cadrCullJob J = loadJob(P.jobs, job);
		const WorkItem item = workItem(P, J, w - firstWorkOf(P, sh.offsets, job));
		const uint32_t gBegin = item.viewBegin, gEnd = item.viewEnd;
		const bool storeLeaf = gBegin == 0;
		const TileDesc T = loadTile(J, item.tile, S::TILE);
		// the job's mesh table is staged once per run of tickets of one job
		// (every wave left the previous tile's last barrier, so no wave still
		// reads the old table)
		bool ldsMeshes = J.numMeshes <= kLdsMeshes;
		if (job != stagedJob) {
			MeshStaging<BLOCK> staging;
			ldsMeshes = staging.load(J, tid);
			staging.store(sh.meshes, tid);
			stagedJob = job;
		}

		const MeshTable meshes{sh.meshes, globalPtr<cadrMesh>(J.meshes), ldsMeshes};

		// load the tile into registers (wave-contiguous runs) and bound it for
		// the tile sphere; the fused form computes the spheres from the job's
		// leaf level instead, writing its world matrices on the way
		float4 sp[FUSED ? 1 : ITEMS];
		uint32_t mi[ITEMS];
		float4* own = sSpheres[FUSED ? wave : 0];
		if constexpr (FUSED) {
			__syncthreads();  // the sphere transforms read the LDS mesh table
			const LeafParams Lf = loadLeaf(P.leaves, job);
			constexpr bool PREFETCH = ITEMS >= 8;
			// the matrices are staged in the last 4 KiB of the wave's spheres;
			// spheres that belong there wait in registers until the last item
			static_assert(ITEMS >= 4, "4 KiB of spheres a wave");
			constexpr int EARLY = ITEMS - 4;
			float4* stage = own + 64 * EARLY;
			float4 late[4];
			auto sink = [&](int j, float4 q) __attribute__((always_inline)) {
				if (j < EARLY)
					own[j * 64 + lane] = q;
				else
					late[j - EARLY] = q;
			};
			if (ldsMeshes)
				propagateTileItems<ITEMS, true, PREFETCH, COOP>(Lf, J, T, wave * WAVE_ITEMS, lane, stage, meshes, sink,
				                                                mi, storeLeaf);
			else
				propagateTileItems<ITEMS, false, PREFETCH, COOP>(Lf, J, T, wave * WAVE_ITEMS, lane, stage, meshes, sink,
				                                                 mi, storeLeaf);
			waveSync();  // the staging is read before its place is taken
#pragma unroll
			for (int k = 0; k < 4; k++) stage[k * 64 + lane] = late[k];
			waveSync();
			asm volatile("" : "+v"(lane));
		} else {
			loadTileItems<ITEMS>(globalPtr<float4>(J.spheres), globalPtr<uint32_t>(J.meshIndex), T,
			                     wave * WAVE_ITEMS + lane, sp, mi);
		}
		auto sphereAt = [&](int j) __attribute__((always_inline)) {
			if constexpr (FUSED) return own[j * 64 + lane]; else return sp[j];
		};
		bool irregular = false;
		float mn[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
		float mx[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
#pragma unroll
		for (int j = 0; j < ITEMS; j++) {
			const uint32_t e = wave * WAVE_ITEMS + j * 64 + lane;
			float4 s = sphereAt(j);
			uint32_t m = mi[j];
			if (e >= T.count) {
				s = make_float4(0.f, 0.f, 0.f, -__builtin_inff());
				m = 0;
			} else if (m >= J.numMeshes) {
				s = make_float4(0.f, 0.f, 0.f, -__builtin_inff());  // invalid mesh: never visible
				m = 0;
			}
			if constexpr (FUSED) own[j * 64 + lane] = s; else sp[j] = s;
			mi[j] = m;

			// a sphere other than a finite one with r >= 0 or the empty sphere
			// (r = -inf, never visible) disables the wave's sphere
			if (e < T.count && s.w != -__builtin_inff() &&
			    !(__builtin_isfinite(s.x) && __builtin_isfinite(s.y) && __builtin_isfinite(s.z) &&
			      __builtin_isfinite(s.w) && s.w >= 0.f))
				irregular = true;
			if (s.w >= 0.f) {
				mn[0] = fminf(mn[0], s.x - s.w); mx[0] = fmaxf(mx[0], s.x + s.w);
				mn[1] = fminf(mn[1], s.y - s.w); mx[1] = fmaxf(mx[1], s.y + s.w);
				mn[2] = fminf(mn[2], s.z - s.w); mx[2] = fmaxf(mx[2], s.z + s.w);
			}
		}
		// a sphere around the wave's items: centre the middle of their bounding
		// box, radius the largest |c_i - C| + r_i (a second reduction), which for
		// scattered drawables is up to sqrt(3) times tighter than the box's half
		// diagonal.  Each wave bounds its own items: it needs no block barrier,
		// and its sphere is smaller than the tile's (2.5M drawables x 256 views,
		// 256 x 8: 421 -> 413 us; 64 uneven scenes fused, 256 x 4: 866 -> 837).
		bool usable = false;
		float4 bound = make_float4(0.f, 0.f, 0.f, -1.f);
		float maxCoord = 0.f;  // bound on |centre component|
		if ((P.flags & CADR_CULL_NO_TILE_SPHERES) == 0u) {
#pragma unroll
			for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
				for (int a = 0; a < 3; a++) {
					mn[a] = fminf(mn[a], __shfl_xor(mn[a], off));
					mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], off));
				}
			}
			const bool anyBad = __ballot(irregular) != 0ull;
			const float cx = (mn[0] + mx[0]) * 0.5f, cy = (mn[1] + mx[1]) * 0.5f, cz = (mn[2] + mx[2]) * 0.5f;
			float R = 0.f;
#pragma unroll
			for (int j = 0; j < ITEMS; j++) {
				const float4 q = sphereAt(j);
				if (q.w >= 0.f) R = fmaxf(R, norm3(q.x - cx, q.y - cy, q.z - cz) + q.w);
			}
#pragma unroll
			for (int off = 32; off >= 1; off >>= 1) R = fmaxf(R, __shfl_xor(R, off));
			R *= 1.0f + 1.0f / 4096.0f;
			usable = !anyBad && __builtin_isfinite(R) && __builtin_isfinite(cx) && __builtin_isfinite(cy) &&
			         __builtin_isfinite(cz);
			// inflate against rounding of the centre and radius above
			const float slack = (fabsf(cx) + fabsf(cy) + fabsf(cz) + R) * (1.0f / 65536.0f);
			bound = make_float4(cx, cy, cz, R + slack);
			maxCoord = fmaxf(fmaxf(fmaxf(fabsf(mn[0]), fabsf(mx[0])), fmaxf(fabsf(mn[1]), fabsf(mx[1]))),
			                 fmaxf(fabsf(mn[2]), fabsf(mx[2])));
		}
		const bool emptyWave = wave * WAVE_ITEMS >= T.count;  // none of the wave's items lies in the tile

		const uint64_t views = J.views;
		uint64_t* chain0 = P.status + statusBaseOf(P, sh.offsets, job);

		for (uint32_t g0 = gBegin; g0 < gEnd; g0 += kViewGroup) {
			const uint32_t vg = uniform(min(kViewGroup, gEnd - g0));

			// classes of the wave's items in the group's views, lane v holding
			// view g0+v, and the views that see some of them; the others
			// contribute nothing and are skipped (and the bound of the FMA
			// estimate for the view; NaN: not used)
			uint32_t cls = 0;
			float margin = __builtin_nanf("");
			if (emptyWave) {
				cls = 1;
			} else if (usable && lane < vg) {
				const ViewC Vl = loadView(views, g0 + lane);
				cls = classifyItems(bound, Vl);
				margin = prefilterMargin(Vl, maxCoord, bound.w);
			}
			const uint64_t active = __ballot(lane < vg && cls != 1u);
			if (lane < vg) sh.cnt[lane][wave] = 0;

			// 1. visibility bits and per-wave counts.  Lanes past the tile and
			// invalid meshes hold the empty sphere, which no test passes.  Each
			// lane keeps its own bits: bit v%32 of vlo[j] (views 0-31 of the
			// group) or vhi[j] (views 32-63) is item j's visibility in view v.
			uint32_t vlo[ITEMS], vhi[ITEMS];
#pragma unroll
			for (int j = 0; j < ITEMS; j++) vlo[j] = vhi[j] = 0u;
			for (uint64_t am = active; am != 0ull; am &= am - 1ull) {
				const uint32_t v = uint32_t(__builtin_ctzll(am));
				if constexpr (FUSED) asm volatile("" ::: "memory");  // the spheres are read again for each view
				const uint32_t c = uniform(__builtin_amdgcn_readlane(cls, v));
				const float mg = __uint_as_float(uniform(__builtin_amdgcn_readlane(__float_as_uint(margin), v)));
				const ViewC V = loadView(views, g0 + v);
				bool vis[ITEMS];
				if (c == 2u) {
#pragma unroll
					for (int j = 0; j < ITEMS; j++) vis[j] = sphereAt(j).w >= 0.f;
				} else if (mg <= 0x1p100f) {
					// the translation column in vector registers once per view
					float w0 = V.r0.w, w1 = V.r1.w, w2 = V.r2.w;
					asm volatile("" : "+v"(w0), "+v"(w1), "+v"(w2));
#pragma unroll
					for (int j = 0; j < ITEMS; j++) {
						const float4 q = sphereAt(j);
						const float p = planeMin(q, V, w0, w1, w2);
						vis[j] = p > 0.f;
						const bool unsure = !(fabsf(p) > mg);
						if (__ballot(unsure) != 0ull) vis[j] = unsure ? sphereVisible(q, V) : vis[j];
					}
				} else {
#pragma unroll
					for (int j = 0; j < ITEMS; j++) vis[j] = sphereVisible(sphereAt(j), V);
				}
				uint32_t n = 0;
				const uint32_t bit = 1u << (v & 31u);
				if (v < 32u) {
#pragma unroll
					for (int j = 0; j < ITEMS; j++) vlo[j] |= vis[j] ? bit : 0u;
				} else {
#pragma unroll
					for (int j = 0; j < ITEMS; j++) vhi[j] |= vis[j] ? bit : 0u;
				}
#pragma unroll
				for (int j = 0; j < ITEMS; j++) n += uint32_t(__builtin_popcountll(__ballot(vis[j])));
				if (lane == 0) sh.cnt[v][wave] = n;
			}
			__syncthreads();

			// 2. look-back, one view per lane of wave 0
			bool stuck = false;
			if (wave == 0 && lane < vg) {
				uint32_t total = 0;
#pragma unroll
				for (int q = 0; q < WAVES; q++) total += sh.cnt[lane][q];
				uint64_t* chain = chain0 + uint64_t(g0 + lane) * J.numTiles;
				uint32_t excl = 0;
				if (T.first) {
					publish(chain + T.chain, packStatus(epoch, kStatePrefix, total));
				} else {
					publish(chain + T.chain, packStatus(epoch, kStateAggregate, total));
					excl = lookBackSerial(chain, T.chain, WaitBound{P.ctl, P.waitLimit, epoch}, MayBeStuck{(b & kRoam) != 0u, shard.shift});
					if (excl != kStuck) publish(chain + T.chain, packStatus(epoch, kStatePrefix, excl + total));
				}
				uint32_t slot = T.segBase + excl;
#pragma unroll
				for (int q = 0; q < WAVES; q++) {
					sh.base[lane][q] = slot;
					slot += sh.cnt[lane][q];
				}
				if (excl == kStuck) {
					stuck = true;
#pragma unroll
					for (int q = 0; q < WAVES; q++) sh.cnt[lane][q] = 0;
				} else if (T.last && T.k < J.numStateSets) {
					globalMut<uint32_t>(J.counts)[uint64_t(g0 + lane) * J.numStateSets + T.k] = excl + total;
				}
			}
			if (__ballot(stuck) != 0ull) {
				leaveItem(P, shard, lane);
				b |= kRoam;
			}
			__syncthreads();

			// 3. compacted writes: each visible drawable's lane stores its command
			// at the wave's output slot plus its rank among the item's visible
			// lanes; consecutive visible lanes write consecutive commands, so a
			// store instruction covers one contiguous run and the L2 merges the
			// runs of an item into whole lines.  Views 0-31 and 32-63 of the
			// group take their bits from vlo and vhi.
			auto writeHalf = [&](auto lds, uint64_t am, uint32_t v0,
			                     const uint32_t (&bits)[ITEMS]) __attribute__((always_inline)) {
				for (; am != 0ull; am &= am - 1ull) {
					const uint32_t v = v0 + uint32_t(__builtin_ctzll(am));
					if constexpr (FUSED) asm volatile("" ::: "memory");
					const uint32_t run = uniform(sh.cnt[v][wave]);
					if (run == 0) continue;
					const ViewC V = loadView(views, g0 + v);
					const gmut<uint32_t> out = globalMut<uint32_t>(J.commands) + uint64_t(g0 + v) * J.commandStride * 5ull;
					const uint32_t base = uniform(sh.base[v][wave]);
					// slot bounds per lane only when the wave's run can reach the stride
					auto items = [&](auto checked) __attribute__((always_inline)) {
						uint32_t pos = base;
#pragma unroll
						for (int j = 0; j < ITEMS; j++) {
							const bool vis = (bits[j] >> (v & 31u)) & 1u;
							const uint64_t m = __ballot(vis);
							const uint32_t n = uint32_t(__builtin_popcountll(m));
							if (n == 0) continue;
							if (vis) {
								const float4 q = sphereAt(j);
								uint32_t count, first, vofs;
								meshCommand<decltype(lds)::value>(meshes, mi[j], q.w, viewCoord(V.r2, q), V, count,
								                                  first, vofs);
								const uint32_t r = maskRank(m);
								if (!decltype(checked)::value || pos + r < J.commandStride) {
									const gmut<uint32_t> o = out + uint64_t(pos) * 5ull + uint64_t(r * 5u);
									o[0] = count;
									o[1] = 1u;
									o[2] = first;
									o[3] = vofs;
									o[4] = T.start + wave * WAVE_ITEMS + j * 64 + lane;
								}
							}
							pos = uniform(pos + n);
						}
					};
					if (base + run <= J.commandStride)
						items(std::false_type{});
					else
						items(std::true_type{});
				}
			};
			auto writeViews = [&](auto lds) __attribute__((always_inline)) {
				writeHalf(lds, active & 0xffffffffull, 0u, vlo);
				writeHalf(lds, active >> 32, 32u, vhi);
			};
			if (meshes.inLds)
				writeViews(std::true_type{});
			else
				writeViews(std::false_type{});
			__syncthreads();
		}
	}

	if (wave == 0 && signOff(P, shard, epoch, lane)) finishLaunch<S::TILE, FUSED>(shard, epoch, lane);
}

// Job offsets of a batched launch of more than kInlineJobs jobs (prefix sums
// over jobs); one block, before the cull kernel on the same stream.
__global__ __launch_bounds__(256) void cullSetupKernel(const cadrCullJob* __restrict__ jobs, uint32_t numJobs,
                                                       uint32_t splitTiles, uint32_t groupShift, bool leaves,
                                                       uint32_t* __restrict__ firstWork,
                                                       uint64_t* __restrict__ statusBase)
{
	__shared__ uint32_t sT[256];
	__shared__ uint64_t sS[256];
	const uint32_t tid = threadIdx.x;
	uint32_t runT = 0;
	uint64_t runS = 0;
	for (uint32_t base = 0; base < numJobs; base += 256) {
		const uint32_t j = base + tid;
		uint32_t nt = 0;
		uint64_t ns = 0;
		if (j < numJobs) {
			nt = uint32_t(jobWorkItems(jobs[j].numTiles, jobs[j].numViews, splitTiles, groupShift, leaves));
			ns = uint64_t(jobs[j].numViews) * jobs[j].numTiles;
		}
		sT[tid] = nt;
		sS[tid] = ns;
		__syncthreads();
		for (uint32_t off = 1; off < 256; off <<= 1) {
			const uint32_t a = tid >= off ? sT[tid - off] : 0u;
			const uint64_t b = tid >= off ? sS[tid - off] : 0ull;
			__syncthreads();
			sT[tid] += a;
			sS[tid] += b;
			__syncthreads();
		}
		if (j < numJobs) {
			firstWork[j] = runT + sT[tid] - nt;
			statusBase[j] = runS + sS[tid] - ns;
		}
		runT += sT[255];
		runS += sS[255];
		__syncthreads();
	}
	if (tid == 0) firstWork[numJobs] = runT;
}

// Ticket shards (log2) for a launch of `workgroups` workgroups over `work`
// items that move about `bytes` bytes in all.  One counter hands out an item
// every 12 ns; an item of 75 KB takes as long at 6.3 TB/s, so as many shards
// are taken as make the tickets twice as fast as the bytes (8 for one-view
// tiles of 1024 drawables, 1 for 8192 or for many views).  More than that
// loses: the look-back waits a little longer where a chain's neighbours come
// from different counters (10M drawables in 1024 x 8 tiles, 8 shards: 64.4
// against 60.4 us with one).  Below 256 workgroups one counter costs less
// than the second level of signOff.
inline uint32_t shardShiftFor(uint32_t tile, uint64_t workgroups, uint64_t work, uint64_t bytes)
{
	if (oneShard(tile) || workgroups < 256 || work >= (1ull << 31)) return 0;
	const uint64_t item = bytes / work + 1;
	uint32_t shift = 0;
	while ((2u << shift) <= kMaxShards && workgroups >= (uint64_t(64) << shift) && (item << shift) < 150000u) shift++;
	return shift;
}

// Bytes a job moves, about: its drawables read once (and, where its leaf
// level is computed, 128 more for the matrices) and 3 per drawable and view
// written (20 for about one in seven).
inline uint64_t jobBytes(const cadrCullJob& J, bool leaf)
{
	return uint64_t(J.numDrawables) * (20u + (leaf ? 116u : 0u) + 3ull * J.numViews);
}

}  // namespace cadr

struct cadrCullWorkspace {
	uint64_t* status = nullptr;
	uint64_t statusWords = 0;
	uint32_t* ctl = nullptr;
	uint32_t* firstWork = nullptr;
	uint64_t* statusBase = nullptr;
	uint32_t maxJobs = 0;
	int device = 0;
	uint64_t waitLimit = 0;      // steady-counter ticks a look-back wait may last
	uint64_t ticksPerUs = 100;   // steady-counter rate
};

using namespace cadr;

namespace {

using KernelFn = void (*)(CullParams);

struct KernelEntry {
	uint32_t block, items;
	KernelFn batch;       // many views / jobs
	KernelFn view;        // one view, or nullptr
	KernelFn fused;       // leaf propagation + one view, or nullptr
	KernelFn fusedBatch;  // leaf propagation + many views / jobs, or nullptr
	KernelFn viewLoop;    // one view, persistent (cullViewLoopKernel), or nullptr where it is not faster
	KernelFn few[2][3];   // few views per job, 1, 2 or 4 at a time (cullFewKernel): one job, many; or nullptr
};

// viewLoop where it measured faster than one tile per workgroup (10M
// drawables, 64 StateSets, one view, 18% visible): 1024 x 2 / 4 / 8 74.0 / 62.5
// / 58.8 against 94.6 / 67.0 / 59.6 us; not at 256 x 4 / 8 / 16 (67.5 / 65.0 /
// 63.3 against 63.9 / 61.5 / 63.0), where several workgroups of a CU overlap
// each other's phases (viewLoopOf has another kernel for the smaller tiles).
// fusedBatch: parents read whole (COOP) and the items prefetched at 256 x 8,
// held to 3 waves per SIMD (4 registers spilled); neither at 256 x 4 and 512 x
// 4, held to 4.  64 uneven scenes, 1-32 views: 256 x 8 867 us (no prefetch 881,
// neither 879, registers unbounded 1002), 256 x 4 855 (COOP 923, 3 waves 910),
// 512 x 4 881 (3 waves with COOP 1255).
#define FEW(B, I)                                                                                              \
	{                                                                                                       \
		{cullFewKernel<B, I, 1, true, false>, cullFewKernel<B, I, 2, true, false>,                        \
		 cullFewKernel<B, I, 4, false, false>},                                                           \
		{cullFewKernel<B, I, 1, true, true>, cullFewKernel<B, I, 2, true, true>,                          \
		 cullFewKernel<B, I, 4, false, true>},                                                            \
	}
const KernelEntry kKernels[] = {
    {256, 2, cullKernel<256, 2, false>, cullViewKernel<256, 2>, cullFusedKernel<256, 2, 4>, nullptr, nullptr, FEW(256, 2)},
    {256, 4, cullKernel<256, 4, false>, cullViewKernel<256, 4>, cullFusedKernel<256, 4, 4>, cullKernel<256, 4, true, false, 4>, nullptr, FEW(256, 4)},
    {256, 8, cullKernel<256, 8, false>, cullViewKernel<256, 8>, cullFusedKernel<256, 8, 1>, cullKernel<256, 8, true, true, 3>, nullptr, FEW(256, 8)},
    {256, 16, cullKernel<256, 16, false>, cullViewKernel<256, 16>, cullFusedKernel<256, 16, 1>, nullptr, nullptr},
    {512, 2, cullKernel<512, 2, false>, cullViewKernel<512, 2>, cullFusedKernel<512, 2, 1>, nullptr, nullptr},
    {512, 4, cullKernel<512, 4, false>, cullViewKernel<512, 4>, cullFusedKernel<512, 4, 1>, cullKernel<512, 4, true, false, 4>, nullptr, FEW(512, 4)},
    {512, 8, nullptr, cullViewKernel<512, 8>, nullptr, nullptr, nullptr},
    {512, 16, nullptr, cullViewKernel<512, 16>, nullptr, nullptr, nullptr},
    {1024, 1, nullptr, cullViewKernel<1024, 1>, cullFusedKernel<1024, 1, 1>, nullptr, cullViewLoopKernel<1024, 1>},
    {1024, 2, nullptr, cullViewKernel<1024, 2>, cullFusedKernel<1024, 2, 1>, nullptr, cullViewLoopKernel<1024, 2>},
    {1024, 4, nullptr, cullViewKernel<1024, 4>, nullptr, nullptr, cullViewLoopKernel<1024, 4>},
    {1024, 8, nullptr, cullViewKernel<1024, 8>, nullptr, nullptr, cullViewLoopKernel<1024, 8>},
    {1024, 16, nullptr, cullViewKernel<1024, 16>, nullptr, nullptr, nullptr},
    {128, 8, cullKernel<128, 8, false>, nullptr, nullptr, nullptr, nullptr},
    {128, 16, cullKernel<128, 16, false>, nullptr, nullptr, nullptr, nullptr},
};

uint32_t computeUnits()
{
	const int cu = computeUnitCount();
	return cu > 0 ? uint32_t(cu) : 256u;
}

// Workgroups of kernel fn (block threads) resident on the current device at
// once: compute units x workgroups per CU by the occupancy calculator,
// cached per (device, kernel).  0 if the query fails.
int residentWorkgroups(KernelFn fn, uint32_t block)
{
	static std::mutex m;
	static std::vector<std::pair<std::pair<int, KernelFn>, int>> cache;
	int dev = 0;
	if (hipGetDevice(&dev) != hipSuccess) return 0;
	std::lock_guard<std::mutex> lock(m);
	for (const auto& e : cache)
		if (e.first.first == dev && e.first.second == fn) return e.second;
	int perCU = 0;
	if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, reinterpret_cast<const void*>(fn), int(block), 0) !=
	        hipSuccess ||
	    perCU <= 0)
		return 0;
	const int n = computeUnitCount() * perCU;
	if (n > 0) cache.push_back({{dev, fn}, n});
	return n;
}

const KernelEntry* findKernel(const cadrCullConfig* c)
{
	if (!c) return nullptr;
	for (const KernelEntry& k : kKernels)
		if (k.block == c->blockSize && k.items == c->itemsPerThread) return &k;
	return nullptr;
}

// The shape that runs a one-view launch of numTiles tiles given in shape ke:
// where the tiles do not fill the compute units once, the one of the same
// tile size with the most threads, so that each wave's chain of round trips is
// shorter (100k drawables, 256 x 4 against 1024 x 1: 7.4 / 6.8 us; a tree frame
// of 41k leaves 19.0 / 17.7 us, of 400k leaves, 391 tiles, 29.6 / 31.0 us).
// The fused kernel is kept at 512 threads: 41k leaves 20.4 / 20.6 us.
const KernelEntry* shapeFor(const KernelEntry* ke, uint32_t numTiles, uint32_t cu, KernelFn KernelEntry::*path)
{
	if (numTiles > cu) return ke;
	const KernelEntry* best = ke;
	for (const KernelEntry& k : kKernels)
		if (k.block * k.items == ke->block * ke->items && k.block > best->block && k.*path) best = &k;
	return best;
}

// The same for a batched launch: 512 x 4 for 256 x 8, the one pair of shapes
// that has every batched kernel (150k drawables, 4 / 20 views: 14.4 / 21.0 us at
// 256 x 8, 11.4 / 18.4 at 512 x 4; 400k, 196 tiles, 16.1 / 29.4 and 13.1 / 28.4;
// 12 small trees, leaves fused, 49.5 and 39.8).  With fused leaves up to 8 tiles
// a compute unit, where 256 x 8's longer chain per wave is not yet covered by
// other workgroups: 640 tiles, 1-10 views, 73.9 and 61.9 us (256 x 8 with its
// spheres in registers 64.8), 1,408 tiles, 1-32 views, 129.4 and 117.7, 1,930,
// 1-10 views, 141.7 and 131.2, but at 2,048, one view, 106.6 and 108.1, 9,920, 1-2
// views, 462.7 and 475.5.  Past 4 tiles a compute unit only if they are a quarter
// full, or the rounds of its fewer workgroups count for more: 512 tiles of 352
// drawables, 1-3 views, 33.4 and 27.4, but 1,280 of 274, one view, 46.9 and 49.6.
const KernelEntry* batchShapeFor(const KernelEntry* ke, uint64_t tiles, uint64_t drawables, uint32_t cu,
                                 KernelFn KernelEntry::*path)
{
	const uint64_t full = uint64_t(ke->block) * ke->items;
	if (path == &KernelEntry::fusedBatch ? tiles >= 8ull * cu || (tiles > 4ull * cu && 4 * drawables < full * tiles)
	                                     : tiles > cu)
		return ke;
	const KernelEntry* wide = shapeFor(ke, uint32_t(std::min<uint64_t>(tiles, cu)), cu, path);
	return ke->few[0][0] && wide->few[0][0] ? wide : ke;
}

}  // namespace

bool cadr::cullHasKernel(const cadrCullConfig* c, CullPath path)
{
	const KernelEntry* k = findKernel(c);
	if (!k) return false;
	switch (path) {
	case CullPath::View: return k->view != nullptr;
	case CullPath::Batch: return k->batch != nullptr;
	case CullPath::Fused: return k->fused != nullptr;
	case CullPath::FusedBatch: return k->fusedBatch != nullptr;
	}
	return false;
}

namespace {

int checkJob(const cadrCullJob& J)
{
	CADR_REQUIRE(J.numTiles == 0 || J.tiles, "cull: job without tiles");
	CADR_REQUIRE(J.numTiles == 0 || (J.spheres && J.meshIndex && J.meshes && J.views && J.commands && J.counts),
	             "cull: job with a null array");
	CADR_REQUIRE(J.spheres % 16 == 0 && J.meshes % 16 == 0 && J.views % 16 == 0 && J.tiles % 16 == 0 &&
	                 J.meshIndex % 4 == 0 && J.commands % 4 == 0 && J.counts % 4 == 0,
	             "cull: misaligned job array (spheres, meshes, views, tiles need 16 bytes)");
	CADR_REQUIRE(J.commandStride >= J.numDrawables, "cull: commandStride < numDrawables");
	return CADR_SUCCESS;
}

}  // namespace

CADR_API uint32_t cadrCullTileSize(const cadrCullConfig* config)
{
	const KernelEntry* k = findKernel(config);
	return k ? k->block * k->items : 0u;
}

CADR_API uint32_t cadrCullConfigPaths(const cadrCullConfig* config)
{
	const KernelEntry* k = findKernel(config);
	if (!k) return 0u;
	return (k->view || k->batch ? CADR_CULL_PATH_VIEW : 0u) | (k->batch ? CADR_CULL_PATH_BATCH : 0u) |
	       (k->fused ? CADR_CULL_PATH_FUSED_VIEW : 0u) | (k->fusedBatch ? CADR_CULL_PATH_FUSED_BATCH : 0u);
}

CADR_API int cadrBuildCullTiles(const uint32_t* stateSetCounts, uint32_t numStateSets, uint32_t tileSize,
                                cadrCullTile* tiles, uint32_t capacity, uint32_t* numTiles)
{
	CADR_REQUIRE(numTiles, "cadrBuildCullTiles: numTiles is NULL");
	CADR_REQUIRE(tileSize > 0, "cadrBuildCullTiles: tileSize is 0");
	CADR_REQUIRE(numStateSets == 0 || stateSetCounts, "cadrBuildCullTiles: stateSetCounts is NULL");
	CADR_REQUIRE(numStateSets <= CADR_TILE_STATESET_MASK, "cadrBuildCullTiles: too many StateSets");
	std::vector<uint64_t> base(numStateSets + 1, 0), firstTile(numStateSets + 1, 0);
	uint64_t maxTiles = 0;
	for (uint32_t k = 0; k < numStateSets; k++) {
		const uint64_t c = stateSetCounts[k];
		// look-back status words carry 30-bit counts
		if (c > CADR_TILE_STATESET_MASK)
			return setError(CADR_ERROR_INVALID_VALUE, "cadrBuildCullTiles: a StateSet holds more than 2^30-1 drawables");
		const uint64_t nt = c == 0 ? 1 : (c + tileSize - 1) / tileSize;
		base[k + 1] = base[k] + c;
		firstTile[k + 1] = firstTile[k] + nt;
		maxTiles = std::max(maxTiles, nt);
	}
	if (base[numStateSets] > 0xffffffffull)
		return setError(CADR_ERROR_INVALID_VALUE, "cadrBuildCullTiles: more than 2^32 drawables");
	const uint64_t n = firstTile[numStateSets];
	if (n > 0xffffffffull) return setError(CADR_ERROR_INVALID_VALUE, "cadrBuildCullTiles: too many tiles");
	*numTiles = uint32_t(n);
	if (!tiles) return ok();
	if (n > capacity) return setError(CADR_ERROR_INVALID_VALUE, "cadrBuildCullTiles: capacity too small");
	// round-robin over StateSets: the q-th tile of every StateSet, then the (q+1)-th
	uint64_t out = 0;
	for (uint64_t q = 0; q < maxTiles; q++) {
		for (uint32_t k = 0; k < numStateSets; k++) {
			const uint64_t c = stateSetCounts[k];
			const uint64_t nt = firstTile[k + 1] - firstTile[k];
			if (q >= nt) continue;
			const uint64_t cnt = c == 0 ? 0 : std::min<uint64_t>(tileSize, c - q * tileSize);
			uint32_t flags = k;
			if (q == 0) flags |= CADR_TILE_FIRST;
			if (q + 1 == nt) flags |= CADR_TILE_LAST;
			cadrCullTile& t = tiles[out++];
			t.start = uint32_t(base[k] + q * tileSize);
			t.count = uint32_t(cnt);
			t.stateSetBase = uint32_t(base[k]);
			t.stateSetAndFlags = flags;
			t.chainIndex = uint32_t(firstTile[k] + q);
			t.reserved[0] = t.reserved[1] = t.reserved[2] = 0;
		}
	}
	return ok();
}

CADR_API int cadrCullWorkspaceCreate(uint64_t statusWords, uint32_t maxJobs, cadrCullWorkspace** workspace)
{
	CADR_REQUIRE(workspace, "cadrCullWorkspaceCreate: workspace is NULL");
	CADR_REQUIRE(maxJobs > 0, "cadrCullWorkspaceCreate: maxJobs is 0");
	*workspace = nullptr;
	auto* w = new cadrCullWorkspace;
	CADR_CHECK_HIP(hipGetDevice(&w->device), "hipGetDevice");
	w->statusWords = statusWords > 0 ? statusWords : 1;
	w->maxJobs = maxJobs;
	hipError_t e = hipMalloc(&w->status, w->statusWords * sizeof(uint64_t));
	if (e == hipSuccess) e = hipMalloc(&w->ctl, kCtlWords * sizeof(uint32_t));
	if (e == hipSuccess) e = hipMalloc(&w->firstWork, (uint64_t(maxJobs) + 1) * sizeof(uint32_t));
	if (e == hipSuccess) e = hipMalloc(&w->statusBase, uint64_t(maxJobs) * sizeof(uint64_t));
	// epoch 0 is never a valid epoch, so zeroed status words read as "not ready"
	if (e == hipSuccess) e = hipMemset(w->status, 0, w->statusWords * sizeof(uint64_t));
	if (e == hipSuccess) e = hipMemset(w->ctl, 0, kCtlWords * sizeof(uint32_t));
	// launches start at epoch 1: 0 marks a status word never written and an
	// error word with nothing to report
	const uint32_t firstEpoch = 1;
	if (e == hipSuccess) e = hipMemcpy(w->ctl + kCtlEpoch, &firstEpoch, sizeof(firstEpoch), hipMemcpyHostToDevice);
	int khz = 0;
	if (e == hipSuccess) e = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, w->device);
	w->ticksPerUs = khz >= 1000 ? uint64_t(khz) / 1000u : 1u;
	w->waitLimit = kDefaultWaitLimitUs * w->ticksPerUs;
	if (e == hipSuccess) e = hipDeviceSynchronize();
	if (e != hipSuccess) {
		(void)hipGetLastError();
		(void)hipFree(w->status); (void)hipFree(w->ctl); (void)hipFree(w->firstWork); (void)hipFree(w->statusBase);
		delete w;
		return setError(CADR_ERROR_OUT_OF_RESOURCES, "cadrCullWorkspaceCreate: device allocation failed");
	}
	*workspace = w;
	return ok();
}

CADR_API int cadrCullWorkspaceSetWaitLimit(cadrCullWorkspace* w, uint32_t microseconds)
{
	CADR_REQUIRE(w, "cadrCullWorkspaceSetWaitLimit: workspace is NULL");
	CADR_REQUIRE(microseconds > 0, "cadrCullWorkspaceSetWaitLimit: the limit must be positive");
	w->waitLimit = uint64_t(microseconds) * w->ticksPerUs;
	return ok();
}

CADR_API int cadrCullWorkspaceCheck(cadrCullWorkspace* w)
{
	CADR_REQUIRE(w, "cadrCullWorkspaceCheck: workspace is NULL");
	int dev = 0;
	CADR_CHECK_HIP(hipGetDevice(&dev), "hipGetDevice");
	CADR_REQUIRE(dev == w->device, "cadrCullWorkspaceCheck: workspace belongs to another device");
	CADR_CHECK_HIP(hipDeviceSynchronize(), "cadrCullWorkspaceCheck: hipDeviceSynchronize");
	uint32_t err = 0;
	CADR_CHECK_HIP(hipMemcpy(&err, w->ctl + kCtlError, sizeof(err), hipMemcpyDeviceToHost),
	               "cadrCullWorkspaceCheck: read");
	if (err == 0) return ok();
	const uint32_t zero = 0;
	CADR_CHECK_HIP(hipMemcpy(w->ctl + kCtlError, &zero, sizeof(zero), hipMemcpyHostToDevice),
	               "cadrCullWorkspaceCheck: clear");
	return setError(CADR_ERROR_TIMEOUT,
	                "cull: a look-back wait gave up (the tile list names a predecessor that no tile publishes); "
	                "the outputs of launch epoch " + std::to_string(err) + " are unspecified");
}

CADR_API int cadrCullWorkspaceDestroy(cadrCullWorkspace* w)
{
	if (!w) return ok();
	hipError_t e = hipDeviceSynchronize();
	(void)hipFree(w->status); (void)hipFree(w->ctl); (void)hipFree(w->firstWork); (void)hipFree(w->statusBase);
	delete w;
	CADR_CHECK_HIP(e, "cadrCullWorkspaceDestroy: hipDeviceSynchronize");
	return ok();
}

namespace {

// Leaf level of a fused launch against its job: node i is drawable i.
int checkLeaf(const cadrTransformLevel& L, const cadrCullJob& J, const std::string& fn)
{
	CADR_REQUIRE(L.count == J.numDrawables, fn + ": the leaf level must hold the job's drawables");
	CADR_REQUIRE(L.count == 0 || (L.localMatrices && L.worldMatrices), fn + ": null matrix array");
	CADR_REQUIRE((L.localMatrices % 16) == 0 && (L.worldMatrices % 16) == 0 && (L.parentWorld % 16) == 0 &&
	                 (L.spheres % 16) == 0,
	             fn + ": matrix and sphere arrays must be 16-byte aligned");
	CADR_REQUIRE(L.parentWorld == 0 || (L.parentIndex && L.parentIndex % 4 == 0),
	             fn + ": parentIndex is NULL or misaligned for a non-root level");
	return CADR_SUCCESS;
}

// The persistent kernel of one view, or nullptr where one tile per workgroup
// is faster: cullFewKernel at 256 x 2 and 256 / 512 x 4 (10M drawables, 64
// StateSets 62.7 / 57.0 / 55.6 against 73.8 / 58.2 / 57.6 us, one StateSet 256
// x 4 68.7 against 91.1), not at 256 x 8 (60.4 against 57.3).
KernelFn viewLoopOf(const KernelEntry& ke)
{
	return ke.viewLoop ? ke.viewLoop : ke.items <= 4 ? ke.few[0][0] : nullptr;
}

// The few-view kernel for a launch, or nullptr where the many-view kernel
// (cullKernel) is the faster one.  That one reads a tile once for 64 views and
// skips the views that see none of it or all of it, but keeps its workgroups
// long on a tile; the few-view kernel tests every drawable, four views at a
// time, in many more work items.  Measured at 256 x 8, trees of clustered
// drawables, few against many: 12 views 4M drawables 93 / 107 us, 2M 53 / 59;
// 37 views 100k 19 / 39, 333k 33 / 45, 1M 68 / 62; 64 views 333k 43 / 64, 1M
// 105 / 86; 128 views 100k 33 / 64, 333k 75 / 75; 512 x 4: 16 views 865k 33 /
// 36, 27 views 1.2M 70 / 62.  So few wins up to about 16 views a drawable, and
// for more views where the tiles do not fill the chip twice and the launch has
// no more than about 2^25 tests.  A launch whose jobs differ goes by its average,
// unless jobs that are the many-view kernel's by themselves have more than 6
// tests per drawable of the others, which that kernel is slower on: 10M
// drawables x 1 view + 1M x 128 (a tree's) 332 / 187 us, 4M x 1 + 2M x 32 121 /
// 93, 8M x 1 + 1M x 64 157 / 129, but 16M x 1 in 8 scenes + 1M x 64 223 / 237,
// 10M x 1 + 100k x 256 111 / 117.  (Scattered drawables, which no bounding
// sphere helps: 310 / 377, 224 / 304 and 107 / 231 in the first and the last two.)
KernelFn fewKernelFor(const KernelEntry& ke, const cadrCullJob* jobs, uint32_t numJobs, uint32_t flags, uint32_t cu)
{
	constexpr uint64_t kFewViews = 16, kFewTests = 1ull << 25;
	uint64_t drawables = 0, tests = 0, tiles = 0;
	uint32_t mostViews = 0;
	uint64_t manyTests = 0, others = 0;  // tests of jobs of many views and tests, drawables of the other jobs
	for (uint32_t j = 0; j < numJobs; j++) {
		if (jobs[j].numViews == 0) continue;  // no work items
		// (a tile of few or no drawables costs what some 256 tests do)
		const uint64_t n = std::max<uint64_t>(jobs[j].numDrawables, 256ull * jobs[j].numTiles);
		drawables += n;
		tests += n * jobs[j].numViews;
		tiles += jobs[j].numTiles;
		mostViews = std::max(mostViews, jobs[j].numViews);
		if (jobs[j].numViews > kFewViews && n * jobs[j].numViews > kFewTests)
			manyTests += n * jobs[j].numViews;
		else
			others += n;
	}
	const bool split = (flags & CADR_CULL_WHOLE_TILES) == 0;
	const bool small = tiles <= 2 * cu && tests <= kFewTests;
	if (split ? manyTests > 6 * others || (tests > kFewViews * drawables && !small) : mostViews > 4) return nullptr;
	return ke.few[numJobs > 1][mostViews <= 1 ? 0 : mostViews == 2 ? 1 : 2];
}

// Whether a leaf level's world matrices are written over its local ones.
bool inPlace(const cadrTransformLevel& L)
{
	return L.localMatrices < L.worldMatrices + 64 * L.count && L.worldMatrices < L.localMatrices + 64 * L.count;
}

// One persistent launch of a batched kernel over numJobs jobs; leaves: the
// fused form's leaf levels (device memory, with their host copy), else null.
int launchBatch(KernelFn KernelEntry::*path, const KernelEntry& asked, const cadrCullConfig* config, uint64_t deviceJobs,
                const cadrCullJob* hostJobs, uint32_t numJobs, cadrCullWorkspace* ws, cadrStream stream,
                const cadrTransformLevel* leaves, const cadrTransformLevel* hostLeaves, const std::string& name)
{
	CADR_REQUIRE(ws, name + ": workspace is NULL");
	if (numJobs == 0) CADR_RETURN_NO_LAUNCH(stream);
	CADR_REQUIRE(deviceJobs && hostJobs, name + ": null job array");
	CADR_REQUIRE(deviceJobs % 16 == 0, name + ": deviceJobs must be 16-byte aligned");
	CADR_REQUIRE(numJobs <= ws->maxJobs, name + ": more jobs than the workspace was created for");
	// the persistent grid; unless CADR_CULL_WHOLE_TILES, a job's last grid
	// tiles are handed out per view group
	const uint32_t cu = computeUnits();
	uint64_t tiles = 0, drawables = 0;
	for (uint32_t j = 0; j < numJobs; j++) {
		tiles += hostJobs[j].numTiles;
		drawables += hostJobs[j].numDrawables;
	}
	const KernelEntry& ke = *batchShapeFor(&asked, tiles, drawables, cu, path);
	KernelFn fn = ke.*path;
	uint32_t perCU = config->workgroupsPerCU;
	if (perCU == 0) perCU = ke.block >= 512 ? 2 : 4;
	uint64_t grid = uint64_t(cu) * perCU;
	auto workItems = [&](uint32_t splitTiles, uint32_t groupShift) {
		uint64_t n = 0;
		for (uint32_t j = 0; j < numJobs; j++)
			n += jobWorkItems(hostJobs[j].numTiles, hostJobs[j].numViews, splitTiles, groupShift, leaves != nullptr);
		return n;
	};
	constexpr uint64_t kMaxWork = 0xffffffffull;  // tickets are 32 bits
	// every tile cut by four views: only what still has its tickets
	const bool cut = workItems(0xffffffffu, 2) < kMaxWork;
	const KernelFn few = leaves || !cut ? nullptr : fewKernelFor(ke, hostJobs, numJobs, config->flags, cu);
	uint32_t splitTiles = uint32_t(std::min<uint64_t>(grid, 1u << 20)), groupShift = 6;
	if (few) {
		fn = few;
		splitTiles = 0xffffffffu;
		groupShift = 2;
		if (config->workgroupsPerCU == 0)
			if (const int resident = residentWorkgroups(few, ke.block)) grid = uint64_t(resident);
	}
	else if (leaves && cut && tiles <= cu / 2) {
		// a fused launch of few tiles: four views a work item, each item
		// computing the tile's leaves again (12 trees, 74 tiles, 1-16 views: 40.8
		// -> 32.2 us; 171 tiles 39.8 -> 41.9, so not there)
		splitTiles = 0xffffffffu;
		groupShift = 2;
	}
	if (config->flags & CADR_CULL_WHOLE_TILES) splitTiles = 0;
	// every item of a tile cut by views reads the tile's local matrices, so one
	// whose world matrices take their place is left whole; nor can its items be
	// left to the end of the launch, which one ticket counter never needs
	const bool inPlaceLeaves = leaves && std::any_of(hostLeaves, hostLeaves + numJobs, inPlace);
	if (inPlaceLeaves) splitTiles = 0;
	const uint64_t totalWork = workItems(splitTiles, groupShift);
	uint64_t statusNeed = 0, bytes = 0;
	for (uint32_t j = 0; j < numJobs; j++) {
		const int rc = checkJob(hostJobs[j]);
		if (rc != CADR_SUCCESS) return rc;
		statusNeed += uint64_t(hostJobs[j].numViews) * hostJobs[j].numTiles;
		bytes += jobBytes(hostJobs[j], leaves != nullptr);
	}
	CADR_REQUIRE(totalWork < kMaxWork, name + ": too many tiles in one launch");
	CADR_REQUIRE(statusNeed <= ws->statusWords, name + ": workspace has too few status words");
	int dev = 0;
	CADR_CHECK_HIP(hipGetDevice(&dev), "hipGetDevice");
	CADR_REQUIRE(dev == ws->device, name + ": workspace belongs to another device");

	hipStream_t s = hipStream_t(stream);
	const auto* jobs = reinterpret_cast<const cadrCullJob*>(deviceJobs);
	if (totalWork == 0) CADR_RETURN_NO_LAUNCH(s);
	if (numJobs > kInlineJobs) {
		hipLaunchKernelGGL(cullSetupKernel, dim3(1), dim3(256), 0, s, jobs, numJobs, splitTiles,
		                   groupShift, leaves != nullptr, ws->firstWork, ws->statusBase);
		CADR_CHECK_HIP(hipGetLastError(), "cullSetupKernel launch");
	}
	if (grid > totalWork) grid = totalWork;
	CullParams p{};
	p.jobs = jobs;
	p.firstWork = ws->firstWork;
	p.statusBase = ws->statusBase;
	p.status = ws->status;
	p.ctl = ws->ctl;
	p.numJobs = numJobs;
	p.totalWork = uint32_t(totalWork);
	p.splitTiles = splitTiles;
	p.groupShift = groupShift;
	p.shardShift = inPlaceLeaves ? 0u : shardShiftFor(ke.block * ke.items, grid, totalWork, bytes);
	p.flags = config->flags;
	p.waitLimit = ws->waitLimit;
	p.leaves = leaves;
	launchKernel(fn, dim3(uint32_t(grid)), dim3(ke.block), s, p);
	CADR_CHECK_HIP(hipGetLastError(), "cullKernel launch");
	return ok();
}

}  // namespace

CADR_API int cadrCullBatch(const cadrCullConfig* config, uint64_t deviceJobs, const cadrCullJob* hostJobs,
                           uint32_t numJobs, cadrCullWorkspace* ws, cadrStream stream)
{
	const KernelEntry* ke = findKernel(config);
	CADR_REQUIRE(ke && ke->batch, "cadrCullBatch: unsupported blockSize/itemsPerThread");
	return launchBatch(&KernelEntry::batch, *ke, config, deviceJobs, hostJobs, numJobs, ws, stream, nullptr, nullptr,
	                   "cadrCullBatch");
}

CADR_API int cadrPropagateCullBatch(uint64_t deviceLeaves, const cadrTransformLevel* hostLeaves,
                                    const cadrCullConfig* config, uint64_t deviceJobs, const cadrCullJob* hostJobs,
                                    uint32_t numJobs, cadrCullWorkspace* ws, cadrStream stream)
{
	const KernelEntry* ke = findKernel(config);
	CADR_REQUIRE(ke && ke->fusedBatch,
	             "cadrPropagateCullBatch: unsupported blockSize/itemsPerThread (256 x 4/8, 512 x 4)");
	if (numJobs == 0) CADR_RETURN_NO_LAUNCH(stream);
	CADR_REQUIRE(deviceLeaves && hostLeaves && hostJobs, "cadrPropagateCullBatch: null leaf or job array");
	CADR_REQUIRE(deviceLeaves % 8 == 0, "cadrPropagateCullBatch: deviceLeaves must be 8-byte aligned");
	for (uint32_t j = 0; j < numJobs; j++) {
		const int rc = checkLeaf(hostLeaves[j], hostJobs[j], "cadrPropagateCullBatch");
		if (rc != CADR_SUCCESS) return rc;
	}
	return launchBatch(&KernelEntry::fusedBatch, *ke, config, deviceJobs, hostJobs, numJobs, ws, stream,
	                   reinterpret_cast<const cadrTransformLevel*>(deviceLeaves), hostLeaves, "cadrPropagateCullBatch");
}

CADR_API int cadrCullView(const cadrCullConfig* config, uint64_t deviceJob, const cadrCullJob* hostJob,
                          cadrCullWorkspace* ws, cadrStream stream)
{
	CADR_REQUIRE(hostJob && hostJob->numViews == 1, "cadrCullView: the job must hold exactly one view");
	const KernelEntry* ke = findKernel(config);
	CADR_REQUIRE(ke, "cadrCullView: unsupported blockSize/itemsPerThread");
	if (!ke->view) return cadrCullBatch(config, deviceJob, hostJob, 1, ws, stream);
	CADR_REQUIRE(ws, "cadrCullView: workspace is NULL");
	CADR_REQUIRE(deviceJob && deviceJob % 16 == 0, "cadrCullView: deviceJob must be a 16-byte aligned address");
	const int rc = checkJob(*hostJob);
	if (rc != CADR_SUCCESS) return rc;
	CADR_REQUIRE(hostJob->numTiles <= ws->statusWords, "cadrCullView: workspace has too few status words");
	int dev = 0;
	CADR_CHECK_HIP(hipGetDevice(&dev), "hipGetDevice");
	CADR_REQUIRE(dev == ws->device, "cadrCullView: workspace belongs to another device");
	if (hostJob->numTiles == 0) CADR_RETURN_NO_LAUNCH(stream);
	CullParams p{};
	p.jobs = reinterpret_cast<const cadrCullJob*>(deviceJob);
	p.status = ws->status;
	p.ctl = ws->ctl;
	p.numJobs = 1;
	p.totalWork = hostJob->numTiles;
	p.flags = config->flags;
	p.waitLimit = ws->waitLimit;
	// more tiles than workgroups fit on the GPU at once: the persistent kernel
	// (grid = resident workgroups); else one tile per workgroup, which saves
	// the loop's extra ticket and barrier on a launch-bound view
	const uint32_t cu = computeUnits();
	const KernelFn viewLoop = hostJob->numTiles > cu ? viewLoopOf(*ke) : nullptr;  // a CU holds one workgroup at least
	const int resident = viewLoop ? residentWorkgroups(viewLoop, ke->block) : 0;
	const bool loop = resident > 0 && hostJob->numTiles > uint32_t(resident);
	const uint32_t grid = loop ? uint32_t(resident) : hostJob->numTiles;
	p.shardShift = shardShiftFor(ke->block * ke->items, grid, hostJob->numTiles, jobBytes(*hostJob, false));
	if (!loop) ke = shapeFor(ke, hostJob->numTiles, cu, &KernelEntry::view);
	p.groupShift = 2;
	launchKernel(loop ? viewLoop : ke->view, dim3(grid), dim3(ke->block), hipStream_t(stream), p);
	CADR_CHECK_HIP(hipGetLastError(), "cullViewKernel launch");
	return ok();
}

CADR_API int cadrPropagateCullView(const cadrTransformLevel* leaf, const cadrCullConfig* config, uint64_t deviceJob,
                                   const cadrCullJob* hostJob, cadrCullWorkspace* ws, cadrStream stream)
{
	CADR_REQUIRE(leaf && hostJob, "cadrPropagateCullView: null argument");
	CADR_REQUIRE(hostJob->numViews == 1, "cadrPropagateCullView: the job must hold exactly one view");
	const KernelEntry* ke = findKernel(config);
	CADR_REQUIRE(ke && ke->fused,
	             "cadrPropagateCullView: unsupported blockSize/itemsPerThread (256 x 2/4/8/16, 512 x 2/4, 1024 x 1/2)");
	CADR_REQUIRE(ws, "cadrPropagateCullView: workspace is NULL");
	CADR_REQUIRE(deviceJob && deviceJob % 16 == 0, "cadrPropagateCullView: deviceJob must be a 16-byte aligned address");
	int rc = checkLeaf(*leaf, *hostJob, "cadrPropagateCullView");
	if (rc != CADR_SUCCESS) return rc;
	rc = checkJob(*hostJob);
	if (rc != CADR_SUCCESS) return rc;
	CADR_REQUIRE(hostJob->numTiles <= ws->statusWords, "cadrPropagateCullView: workspace has too few status words");
	int dev = 0;
	CADR_CHECK_HIP(hipGetDevice(&dev), "hipGetDevice");
	CADR_REQUIRE(dev == ws->device, "cadrPropagateCullView: workspace belongs to another device");
	if (hostJob->numTiles == 0) CADR_RETURN_NO_LAUNCH(stream);
	CullParams p{};
	p.jobs = reinterpret_cast<const cadrCullJob*>(deviceJob);
	p.status = ws->status;
	p.ctl = ws->ctl;
	p.numJobs = 1;
	p.totalWork = hostJob->numTiles;
	p.flags = config->flags;
	p.waitLimit = ws->waitLimit;
	p.leaf = LeafParams{leaf->localMatrices, leaf->parentIndex, leaf->parentWorld, leaf->worldMatrices, leaf->spheres,
	                    leaf->parentWorld ? leaf->parentCount : 0u};
	if (!inPlace(*leaf))  // as in launchBatch
		p.shardShift = shardShiftFor(ke->block * ke->items, hostJob->numTiles, hostJob->numTiles, jobBytes(*hostJob, true));
	if (ke->block < 512) ke = shapeFor(ke, hostJob->numTiles, computeUnits(), &KernelEntry::fused);
	launchKernel(ke->fused, dim3(hostJob->numTiles), dim3(ke->block), hipStream_t(stream), p);
	CADR_CHECK_HIP(hipGetLastError(), "fused cullViewKernel launch");
	return ok();
}

// ------------------------------------------------ allocation-free variant
//
// cadrCullBatchNoAlloc: cadrCullBatch for callers that cannot allocate device
// memory.  Its workspace (look-back status words, control words, per-job
// offsets) is one file-scope device array, `scratch`, of fixed size; each
// device holds its own copy until the process ends.  Host code never passes
// the array's name to a kernel: the name is a host-side stand-in, and the
// device address is taken once per device with hipGetSymbolAddress.
namespace {

constexpr uint64_t kScratchStatusWords = 1ull << 21;  // 16 MiB: sum of numViews x numTiles per launch
constexpr uint32_t kScratchMaxJobs = 4096;
// layout in 64-bit words: status | ctl (kCtlWords uint32) | firstWork (jobs+1 uint32) | statusBase (jobs uint64)
constexpr uint64_t kScratchCtl = kScratchStatusWords;
constexpr uint64_t kScratchFirstWork = kScratchCtl + kCtlWords / 2;
constexpr uint64_t kScratchStatusBase = kScratchFirstWork + (uint64_t(kScratchMaxJobs) + 2) / 2;
constexpr uint64_t kScratchWords = kScratchStatusBase + kScratchMaxJobs;
static_assert(kCtlWords % 2 == 0, "ctl words fill whole 64-bit words");

}  // namespace

static __device__ __align__(256) uint64_t scratch[kScratchWords];

namespace {

struct ScratchDevice {
	uint64_t* ptr = nullptr;   // device address of `scratch` on this device
	uint64_t ticksPerUs = 100;
};

std::mutex g_scratchMutex;
std::vector<ScratchDevice> g_scratchDevices;

// Device address of this device's scratch, set up on the first call on the
// device: the address from hipGetSymbolAddress, status and control words
// cleared by a fill kernel (not hipMemsetAsync, so a caller may capture
// later calls) and the epoch set to 1, complete before the call returns.
int scratchFor(int dev, hipStream_t stream, ScratchDevice& out)
{
	std::lock_guard<std::mutex> lock(g_scratchMutex);
	if (int(g_scratchDevices.size()) <= dev) g_scratchDevices.resize(size_t(dev) + 1);
	ScratchDevice& d = g_scratchDevices[size_t(dev)];
	if (!d.ptr) {
		void* p = nullptr;
		CADR_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "cadrCullBatchNoAlloc: hipGetSymbolAddress(scratch)");
		auto* base = static_cast<uint64_t*>(p);
		const uint64_t a = reinterpret_cast<uint64_t>(base);
		int rc = cadrFillU32(a, 0u, kScratchStatusBase * sizeof(uint64_t), stream);
		if (rc == CADR_SUCCESS) rc = cadrFillU32(a + kScratchCtl * 8 + kCtlEpoch * 4, 1u, 4, stream);
		if (rc != CADR_SUCCESS) return rc;
		CADR_CHECK_HIP(hipStreamSynchronize(stream), "cadrCullBatchNoAlloc: clearing scratch");
		int khz = 0;
		CADR_CHECK_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev), "hipDeviceGetAttribute");
		d.ticksPerUs = khz >= 1000 ? uint64_t(khz) / 1000u : 1u;
		d.ptr = base;
	}
	out = d;
	return ok();
}

}  // namespace

CADR_API int cadrCullBatchNoAlloc(const cadrCullConfig* config, uint64_t deviceJobs, const cadrCullJob* hostJobs,
                                  uint32_t numJobs, cadrStream stream)
{
	const KernelEntry* ke = findKernel(config);
	CADR_REQUIRE(ke && ke->batch, "cadrCullBatchNoAlloc: unsupported blockSize/itemsPerThread");
	if (numJobs == 0) CADR_RETURN_NO_LAUNCH(stream);
	CADR_REQUIRE(hostJobs, "cadrCullBatchNoAlloc: hostJobs is NULL");
	if (numJobs > kScratchMaxJobs)
		return setError(CADR_ERROR_INVALID_VALUE, "cadrCullBatchNoAlloc: " + std::to_string(numJobs) +
		                                              " jobs, more than the " + std::to_string(kScratchMaxJobs) +
		                                              " its fixed scratch holds");
	uint64_t statusNeed = 0;
	for (uint32_t j = 0; j < numJobs; j++) statusNeed += uint64_t(hostJobs[j].numViews) * hostJobs[j].numTiles;
	if (statusNeed > kScratchStatusWords)
		return setError(CADR_ERROR_INVALID_VALUE,
		                "cadrCullBatchNoAlloc: the jobs need " + std::to_string(statusNeed) +
		                    " status words (numViews x numTiles summed over jobs), more than the " +
		                    std::to_string(kScratchStatusWords) + " of its fixed scratch");
	int dev = 0;
	CADR_CHECK_HIP(hipGetDevice(&dev), "hipGetDevice");
	ScratchDevice sd;
	const int rc = scratchFor(dev, hipStream_t(stream), sd);
	if (rc != CADR_SUCCESS) return rc;
	cadrCullWorkspace w;  // a view of the scratch array, nothing allocated
	w.status = sd.ptr;
	w.statusWords = kScratchStatusWords;
	w.ctl = reinterpret_cast<uint32_t*>(sd.ptr + kScratchCtl);
	w.firstWork = reinterpret_cast<uint32_t*>(sd.ptr + kScratchFirstWork);
	w.statusBase = sd.ptr + kScratchStatusBase;
	w.maxJobs = kScratchMaxJobs;
	w.device = dev;
	w.ticksPerUs = sd.ticksPerUs;
	w.waitLimit = kDefaultWaitLimitUs * sd.ticksPerUs;
	return launchBatch(&KernelEntry::batch, *ke, config, deviceJobs, hostJobs, numJobs, &w, stream, nullptr, nullptr,
	                   "cadrCullBatchNoAlloc");
}
