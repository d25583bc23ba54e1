// cs3d_kernels.hip - CDNA4 (gfx950) kernels of the CellSim3D hot path.
//
// Cell kernels run one cell per 192-lane workgroup (3 x wave64; lanes 180..191
// are the padding slots) and grid-stride over cell slots, so a fixed launch
// covers a dynamic cell count.  Every kernel reproduces the floating-point
// operation order of the reference kernel it replaces (cited per function), so
// results match the reference arithmetic; the library is compiled with
// -ffp-contract=off and correctly rounded fp32 division and square root.
//
// Contact pairs.  The reference scans, per node, the cells listed in its
// voxel (2.9-wide grid), keeps those whose bbox lies within attraction_range of
// the node, and tests all 180 nodes of each kept cell (propagate.cu:375-442,
// 603-655).  Here each node keeps a sorted list of candidate partners: the nodes
// of other cells within attraction_range + pair_skin, found through periodic
// search bins of that edge (find_candidates).  The list is rebuilt only on steps where some
// node has moved pair_skin/2 since the last search, so it always contains every
// node now within attraction_range; after divisions only the lists near the divided
// cells are rebuilt (the partial search of search_cell).  Every step then applies the
// reference's own tests to the candidates in (cell, node) order -- the order of the
// reference's loops: the distance test, voxel-list membership and the bbox test
// (pair_terms).  Voxel-list membership is evaluated arithmetically: makeNNlist
// puts cell b into voxel v exactly when v lies in the voxel range of b's bbox
// widened by attraction_range (propagatebound.cu:224-259), so the same range test
// on the same bbox and grid answers "b in list(v)".  One bit per candidate keeps
// which pairs were accepted, for the second friction pass.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <limits>
#include <type_traits>
#include <utility>
#include <vector>

#include "cs3d_acos.h"
#include "cs3d_div.h"
#include "cs3d_dev.h"

namespace cs3d {

// The system owning a cell slot.  A launch over one system's own slot range needs
// no table read: every slot of the range belongs to it.
__device__ __forceinline__ int sys_of(const Pool& p, const Range& r, int slot) {
    return r.one_sys ? r.sys_lo : p.slot_sys[slot];
}

// The entry of a cell kernel is a chain of memory round trips that nothing else
// overlaps in a small tissue: kernel arguments, then the cell's node data beside the
// system's metadata (one scalar round trip), then what depends on them.  Read field by
// field, with a branch on each, it was 7 trips in k_con_dis, 6 in k_dis_post and 5 in
// k_integrate.  With it in three, and the division kernel's arguments and metadata read
// in one batch each, a step took 24.4 instead of 25.6 us at 8 cells, 29.6 instead of
// 30.9 at 403 and 40.5 instead of 42.3 at 2000.
// kEnded: phases of this step that have ended (SysMeta::raised of them stops it).
template <int kEnded = 0, class MP> __device__ __forceinline__ bool sys_live(MP m) {
    // every field read at once, no short-circuit branches: one memory round trip
    const int32_t active = m->active;
    const int64_t horizon = m->horizon, step = m->step;
    uint32_t stop = m->status;
#pragma unroll
    for (int k = 0; k < kEnded; ++k) stop |= m->raised[k];
    return (active != 0) & ((horizon < 0) | (step < horizon)) & !(stop & CS3D_SYS_FATAL_MASK);
}

// Whether cell slot `slot` of the system is stepped; c: its local index.  In a fused
// step no word that it reads changes during the launch, so the waves of a workgroup,
// which read apart from each other, decide alike, and so do all cells of the system.
template <int kEnded, class MP> __device__ __forceinline__ bool cell_live(MP m, int slot, int& c) {
    const int32_t base = m->base, n = m->n;
    c = slot - base;
    return sys_live<kEnded>(m) & (c < n);
}

// Status bits found by a kernel: in phase kPhase of a fused step beside the status (the
// division phase merges them at the end of the step), by an entry point into it.
template <bool kStep, int kPhase> __device__ __forceinline__ uint32_t* status_word(SysMeta* m) {
    return kStep ? &m->raised[kPhase] : &m->status;
}
__device__ __forceinline__ void flag(uint32_t* word, uint32_t bits) {
    if (bits) atomicOr(word, bits);
}

// Loads and stores at a uniform base pointer plus a 32-bit element index: the
// address is an SGPR pair plus one VGPR byte offset (the saddr form of the global
// memory instructions), so per-lane addressing costs one 32-bit register that all
// arrays of a cell share instead of a 64-bit pointer per array.  The byte offset
// must stay below 4 GiB: a cell's node offset (< 768 B), a list entry (< 31 KB),
// or a node key of a system (a context holds at most 2^30 / 192 cells, so every
// key * 4 < 2^32).
template <class T> __device__ __forceinline__ T ldu(const T* base, uint32_t i) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(T));
}
// ldu of a word whose load is issued here: as a relaxed atomic (a plain load
// instruction at this scope) it is not moved behind a branch that follows.
template <class T> __device__ __forceinline__ T load_now(const T* q) {
    static_assert(sizeof(T) == 4, "one word");
    return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
template <class T> __device__ __forceinline__ T ldu_now(const T* base, uint32_t i) {
    return load_now(reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * 4u));
}
template <class T> __device__ __forceinline__ void stu(T* base, uint32_t i, T v) {
    *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + i * (uint32_t)sizeof(T)) = v;
}

// Correctly rounded float square root: the hardware estimate and one correction
// step (the neighbours one ulp either side of the estimate, chosen by the signs of
// the exact fma residuals x - s' s).  Inputs below 2^-96, where the residuals
// would lose bits, are scaled by 2^32 and the result by 2^-16 (exact).  This is
// the library's sequence without its fix-ups for 0 and infinity, which the
// correction step already returns unchanged (as it does NaN; a negative input
// gives NaN).  Equal to sqrtf bit for bit over all 2^32 inputs (cs3d_check_sqrt).
__device__ __forceinline__ float sqrt_cr(float x) {
    const bool tiny = x < 0x1p-96f;
    const float xs = tiny ? x * 0x1p32f : x;
    const float s = __builtin_amdgcn_sqrtf(xs);
    const float sm = __int_as_float(__float_as_int(s) - 1), sp = __int_as_float(__float_as_int(s) + 1);
    const float rm = fmaf(-sm, s, xs), rp = fmaf(-sp, s, xs);
    float t = rm <= 0.f ? sm : s;
    t = rp > 0.f ? sp : t;
    return tiny ? t * 0x1p-16f : t;
}

// sqrt_cr without its scaling of inputs below 2^-96: the same steps on the same
// values for every other input.  A smaller input gives a result below 2^-40 (or
// the exact 0), so quot_ok of the result is false; the callers then take sqrt_cr.
__device__ __forceinline__ float sqrt_normal(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float sm = __int_as_float(__float_as_int(s) - 1), sp = __int_as_float(__float_as_int(s) + 1);
    const float rm = fmaf(-sm, s, x), rp = fmaf(-sp, s, x);
    const float t = rm <= 0.f ? sm : s;
    return rp > 0.f ? sp : t;
}

// RN(1/b) for quot_ok(b): the hardware reciprocal estimate and one Newton step
// with an fma residual.  Equal to 1.0f / b for every float b with quot_ok(b)
// (cs3d_check_div).
__device__ __forceinline__ float rcp_rn(float b) {
    const float y0 = __builtin_amdgcn_rcpf(b);
    const float e = fmaf(-b, y0, 1.0f);
    return fmaf(e, y0, y0);
}

// Marks the division path of a quotient as a branch: the empty volatile asm
// keeps the compiler from evaluating both paths and selecting (which it does for
// a short division otherwise).
__device__ __forceinline__ void slow_path() { asm volatile(""); }

// CS3D_SELDOM (cs3d_theta.h) marks branches hardly ever taken.  What one guards is
// done for every lane of the wave that takes it: the general forms give the same
// bits where the short ones are in range.

// 1.0f / b: from rcp_rn where quot_ok(b), by division otherwise (the same bits)
__device__ __forceinline__ float inv_rn(float b) {
    float y = rcp_rn(b);
    if (CS3D_SELDOM(!quot_ok(b))) y = 1.0f / b;
    return y;
}

// 1.0f / sqrt_cr(x2)
__device__ __forceinline__ float inv_sqrt_rn(float x2) {
    const float r = sqrt_normal(x2);
    float y = rcp_rn(r);
    if (CS3D_SELDOM(!quot_ok(r))) y = 1.0f / sqrt_cr(x2);
    return y;
}

// One bond's spring term stiffness*(R-R0)/R0*d/R for d = dx, dy, dz
// (propagate.cu:311-313).  spring_rcp takes the quotients from the reciprocals of
// R and R0 (iR0 = RN(1/R0), NaN where R0 is outside quot_ok's range) and returns
// whether every operand was in range (quot_ok, quot_num_ok); where it was, the
// terms equal spring_div's, the reference's divisions, bit for bit.  The callers
// sum a node's three bonds with spring_rcp and, where some operand was out of
// range, sum them again with spring_div (one branch per node).
__device__ __forceinline__ bool spring_rcp(float stiffness, float R, float R0, float iR0, float dx, float dy, float dz,
                                           float& tx, float& ty, float& tz) {
    const float a = stiffness * (R - R0);
    const float c = quot_rn(a, R0, iR0);
    const float yR = rcp_rn(R);
    const float nx = c * dx, ny = c * dy, nz = c * dz;
    tx = quot_rn(nx, R, yR);
    ty = quot_rn(ny, R, yR);
    tz = quot_rn(nz, R, yR);
    bool ok = quot_ok(R);  // every compare evaluated, no short-circuit branches
    ok &= quot_num_ok(a);
    ok &= quot_num_ok(nx);
    ok &= quot_num_ok(ny);
    ok &= quot_num_ok(nz);
    return ok;
}
__device__ __forceinline__ void spring_div(float stiffness, float R, float R0, float dx, float dy, float dz, float& tx,
                                           float& ty, float& tz) {
    tx = stiffness * (R - R0) / R0 * dx / R;
    ty = stiffness * (R - R0) / R0 * dy / R;
    tz = stiffness * (R - R0) / R0 * dz / R;
}

// rGrowth of the population model, GPUbounce.cu:1077-1088
template <class PP> __device__ __forceinline__ float rgrowth(PP P, int n) {
    if (__builtin_expect(P->do_pop_model == 1, 0)) {
        float r = (float)((double)P->growth_rate * (1 - (n * 1.0 / (double)P->max_pop)));
        if (r < 0) r = 0;
        return r;
    }
    return P->growth_rate;
}

// voxel coordinate of one axis, propagate.cu:360-370
__device__ __forceinline__ int vox1(float x, float mn, float DL, int div) {
    int s = (int)((x - mn) / DL);
    if (s < 0) s = 0;
    if (s >= div) s = div - 1;
    return s;
}

// Read-only views of a system's parameters and metadata in the constant address
// space: a kernel reads them with scalar loads into scalar registers (the values
// are the same for every lane of a workgroup).  Only for data no kernel writes
// while the reader runs; the scalar cache is only read through.
typedef __attribute__((address_space(4))) const cs3d_params* CParams;
typedef __attribute__((address_space(4))) const SysMeta* CMeta;
__device__ __forceinline__ CParams cparams(const cs3d_params* q) { return (CParams)q; }
__device__ __forceinline__ CMeta cmeta(const SysMeta* q) { return (CMeta)q; }
typedef __attribute__((address_space(4))) const ThetaCoeffs* CTheta;
template <class T> __device__ __forceinline__ T cld(const T* q) {
    return *(__attribute__((address_space(4))) const T*)q;
}

// The kernel's Pool argument (the first kernel parameter) read again where it is
// used: scalar loads from the kernel-argument segment behind an empty asm
// statement, so that the compiler neither hoists them nor keeps the pointers live
// (in scalar registers, or spilled to vector lanes) across the contact loop.
typedef __attribute__((address_space(4))) const Pool* CPool;
__device__ __forceinline__ CPool pool_late() {
    CPool q = (CPool)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(q));
    return q;
}

// The kernel's Pool argument as a cell kernel's loop body sees it: read again in every
// iteration (most workgroups have one).  With the argument itself the compiler computes
// every address that does not change between iterations ahead of the loop, and spills
// most of them there: k_con_dis took 8.9 instead of 8.2 us at 8 cells, 144 instead of
// 137 at 20,000.  (The shorter kernels, which do not spill, are slower with it.)
#define CS3D_LOOP_POOL(name) const auto& name = *pool_late()

// The cell slot and system of loop iteration `it` of a cell kernel: an entry of a
// list made by k_live (a multi-system step), read with one scalar load, or the
// it-th slot of the range.  Wave-uniform: the per-cell base pointers derived from
// the slot stay in scalar registers instead of becoming per-lane 64-bit induction
// variables.
template <int kLive>
__device__ __forceinline__ int2 cell_at(const Range& r, const int2* list, int it) {
    if (kLive) return int2{cld(&list[it].x), cld(&list[it].y)};
    return int2{__builtin_amdgcn_readfirstlane(r.slot_lo + it), r.sys_lo};
}

// The lane's node index as a value the compiler cannot see through (an empty asm
// statement per loop iteration): otherwise it combines "array + lane" into one
// loop-invariant 64-bit pointer per array and lane, which costs two VGPRs per
// array for the whole kernel.  With it, every access is the cell's uniform base
// plus this one 32-bit offset.
__device__ __forceinline__ uint32_t lane_index() {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// v in a vector register: an address made from it is read by a vector load.
__device__ __forceinline__ uint32_t vector_value(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A value read from LDS that the compiler may not replace by a register copy of
// what was stored there: reading a node's own position again where it is needed
// ends the live range of the register that held it.
__device__ __forceinline__ float lds_reread(const float* a, int i) {
    float v = a[i];
    asm volatile("" : "+v"(v));
    return v;
}

// XCD-aware first cell of a workgroup.  The dispatcher hands workgroup v to XCD
// v mod 8; this maps the 8 XCDs to 8 contiguous runs of workgroup indices, so the
// cells one XCD works on are neighbours in index and, for tissues placed in
// order, in space: their partner gathers hit the XCD's own L2.  A bijection on
// [0, gridDim.x): on [0, live) if fewer cells than workgroups are known to be live, and
// the identity beyond, or the last XCDs would have the workgroups without cells (2000
// cells in a larger room, a grid of 2508: 18 us of k_con_dis became 25).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int live = 0x7fffffff) {
    const int G = min((int)gridDim.x, max(live, 1)), v = blockIdx.x;
    if (v >= G) return v;
    const int q = G / kXcds, rem = G % kXcds;
    const int k = v % kXcds, j = v / kXcds;
    return k * q + min(k, rem) + j;
}

// The first iteration of a cell kernel's loop over nit cells.  The grid over a range of
// slots has at most one workgroup per slot, so its loop need not be entered by a test.
template <int kLive> __device__ __forceinline__ int first_cell(int nit, const Range& r) {
    const int it = xcd_block(r.live_hint);
    if (!kLive) __builtin_assume(it < nit);
    return it;
}

// Search bins are periodic: bin coordinate floor((x - origin) / h) modulo the bin
// count of the axis.  Regions farther apart than the bin grid alias into the same
// bins, which only adds entries the distance test rejects, so the bin edge never
// has to grow with the system's extent (outlying cells cannot coarsen the bins of
// a dense tissue).
__device__ __forceinline__ int bin1(float x, float mn, float h, int div) {
    float q = floorf((x - mn) / h);
    q = q == q ? fminf(fmaxf(q, -1.0e9f), 1.0e9f) : 0.0f;  // NaN positions go to bin 0 (flagged elsewhere)
    int s = (int)q % div;
    return s < 0 ? s + div : s;
}
__device__ __forceinline__ int wrap1(int s, int div) { return s < 0 ? s + div : (s >= div ? s - div : s); }

template <class MP> __device__ __forceinline__ int bin_of(MP M, float x, float y, float z) {
    const int bx = bin1(x, M->bmin[0], M->bh, M->bdims[0]);
    const int by = bin1(y, M->bmin[1], M->bh, M->bdims[1]);
    const int bz = bin1(z, M->bmin[2], M->bh, M->bdims[2]);
    return (bz * M->bdims[1] + by) * M->bdims[0] + bx;
}

// order-preserving int encoding of floats for atomic min/max
__device__ __forceinline__ int f2o(float f) {
    int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7FFFFFFF;
}
__device__ __forceinline__ float o2f(int i) { return __int_as_float(i >= 0 ? i : i ^ 0x7FFFFFFF); }

// 0.5 * (double)s / (double)m of the velocity kicks (propagate.cu:698-705,
// 721-723) for a float s.  On systems whose constants passed the host's
// exhaustive check (kick_consts): s times the double-double 1 / (2 m), one
// multiply and one fma with the division's exact result; a zero keeps its sign.
__device__ __forceinline__ double kick_a(float s, float m, CMeta M) {
    const double x = (double)s;
    if (M->kick_fast) {
        const double q = fma(x, M->kick_ah, x * M->kick_al);
        return s == 0.0f ? x : q;
    }
    return 0.5 * x / (double)m;
}
// 0.5 * (double)dt * (double)f / (double)m of VelocityUpdateB (propagate.cu:732-734)
__device__ __forceinline__ double kick_b(float f, float dt, float m, CMeta M) {
    const double x = (double)f;
    if (M->kick_fast) {
        const double q = fma(x, M->kick_bh, x * M->kick_bl);
        return f == 0.0f ? x : q;
    }
    return 0.5 * (double)dt * x / (double)m;
}

// Integrate's velocity half-kick of one component (propagate.cu:698-705): the
// sum in float, the rest in double (0.5 is a double literal), rounded to float.
// fr is the random force drawn in the previous step (0 without add_rands).
__device__ __forceinline__ float half_kick(float v, float fc, float fd, float fr, float dt, float rdt, float m,
                                           CMeta M) {
    return (float)((double)v + kick_a(dt * fc + dt * fd + rdt * fr, m, M));
}

// ---- random force (CalculateRanForce, propagate.cu:667-676) --------------------
// The reference draws curand_normal from per-node cuRAND states (closed library,
// not reproduced).  Here: Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel
// random numbers: as easy as 1, 2, 3", SC'11) with counter {cell * 192 + node,
// step (low, high), attempt} and key {noise_seed, 0x43533344}, turned into
// standard normals by the Marsaglia polar method.  Every operation is integer or
// correctly rounded float (the logarithm is a fixed polynomial), so the host and
// the device produce the same bits.
__device__ __forceinline__ void philox4x32_10(uint32_t* c, uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t hi0 = __umulhi(0xD2511F53u, c[0]), lo0 = 0xD2511F53u * c[0];
        const uint32_t hi1 = __umulhi(0xCD9E8D57u, c[2]), lo1 = 0xCD9E8D57u * c[2];
        const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// natural logarithm of s in (0, 1): s = m 2^e with m in [sqrt(1/2), sqrt(2)),
// ln m = 2 atanh((m - 1) / (m + 1)) by its series to z^9, e ln 2 in two parts
__device__ __forceinline__ float ln01(float s) {
    const uint32_t b = __float_as_uint(s);
    int e = (int)((b >> 23) & 0xffu) - 126;
    float m = __uint_as_float((b & 0x7fffffu) | 0x3f000000u);
    if (m < 0.70710678f) {
        m = m + m;
        e -= 1;
    }
    const float z = (m - 1.0f) / (m + 1.0f);
    const float z2 = z * z;
    float q = 0.11111111f;
    q = q * z2 + 0.14285715f;
    q = q * z2 + 0.2f;
    q = q * z2 + 0.33333334f;
    q = q * z2 + 1.0f;
    const float fe = (float)e;
    return fe * 0.693145751953125f + (2.0f * z * q + fe * 1.4286068e-06f);
}

// three standard normals of node `node` of a tissue at step `step`
__device__ __forceinline__ void noise3(uint32_t seed, uint32_t node, int64_t step, float* z) {
    int got = 0;
    z[0] = z[1] = z[2] = 0.f;
    for (uint32_t attempt = 0; got < 3 && attempt < 32; ++attempt) {
        uint32_t c[4] = {node, (uint32_t)step, (uint32_t)((uint64_t)step >> 32), attempt};
        philox4x32_10(c, seed, 0x43533344u);
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
            const float v1 = 2.0f * (((float)(c[2 * pr] >> 9) + 0.5f) * 1.1920929e-07f) - 1.0f;
            const float v2 = 2.0f * (((float)(c[2 * pr + 1] >> 9) + 0.5f) * 1.1920929e-07f) - 1.0f;
            const float s = v1 * v1 + v2 * v2;
            if (got < 3 && s > 0.0f && s < 1.0f) {
                const float f = sqrt_cr(-2.0f * ln01(s) / s);
                z[got++] = v1 * f;
                if (got < 3) z[got++] = v2 * f;
            }
        }
    }
}

// makeNNlist's voxel range of a cell (propagatebound.cu:224-245): the voxels of
// its bbox widened by attraction_range, clamped to the grid.
struct VoxRange {
    int sx, ex, sy, ey, sz, ez;
};
template <class MP, class PP> __device__ __forceinline__ VoxRange vox_range(const float* b, MP M, PP P) {
    const float DL = P->grid_dl, at = P->attraction_range;
    const float mx = M->gmin[0], my = M->gmin[1], mz = M->gmin[2];
    VoxRange v;
    v.sx = (int)((b[0] - at - mx) / DL); if (v.sx < 0) v.sx = 0;
    v.ex = (int)((b[1] + at - mx) / DL); if (v.ex >= M->dims[0]) v.ex = M->dims[0] - 1;
    v.sy = (int)((b[2] - at - my) / DL); if (v.sy < 0) v.sy = 0;
    v.ey = (int)((b[3] + at - my) / DL); if (v.ey >= M->dims[1]) v.ey = M->dims[1] - 1;
    v.sz = (int)((b[4] - at - mz) / DL); if (v.sz < 0) v.sz = 0;
    v.ez = (int)((b[5] + at - mz) / DL); if (v.ez >= M->dims[2]) v.ez = M->dims[2] - 1;
    return v;
}

// voxel range of a cell's bbox into VRANGE (lanes 0..5 of the caller store)
__device__ __forceinline__ void store_vrange(int32_t* vrange, int64_t slot, const VoxRange& v, int lane) {
    if (lane < 6) {
        const int w[6] = {v.sx, v.ex, v.sy, v.ey, v.sz, v.ez};
        vrange[slot * 6 + lane] = w[lane];
    }
}

// Grid geometry from the global extent e = {minx, maxx, miny, maxy, minz, maxz}:
// host Xdiv/Ydiv/Zdiv (GPUbounce.cu:1331-1334) with the voxel origin at the
// extent's minimum, and the search bins (edge a little above attraction_range +
// pair_skin so that every pair within that range lies in adjacent bins, two bins
// of margin, coarser when the extent outgrows the bin budget).  Returns the
// number of voxel counters to clear.  Called by one thread.
struct GridConsts {  // what set_grid_geometry needs of the parameters and metadata
    float DL, ar, skin;
    int32_t vbudget, bbudget;
};
template <class MP, class PP> __device__ __forceinline__ GridConsts grid_consts(MP M, PP P) {
    return GridConsts{P->grid_dl, P->attraction_range, P->pair_skin, M->vbudget, M->bbudget};
}
__device__ __forceinline__ int64_t set_grid_geometry(SysMeta* M, const GridConsts& k, const float* e) {
    if (!(e[1] >= e[0] && e[3] >= e[2] && e[5] >= e[4])) {
        // no cells (the extent kept its sentinels): a one-voxel grid, nothing to flag
        for (int a = 0; a < 3; ++a) {
            M->gmin[a] = 0.0f; M->dims[a] = 1;
            M->bmin[a] = 0.0f; M->bdims[a] = 3;
        }
        return 1;
    }
    const float DL = k.DL;
    const int xd = (int)((e[1] - e[0]) / DL + 1.0f);
    const int yd = (int)((e[3] - e[2]) / DL + 1.0f);
    const int zd = (int)((e[5] - e[4]) / DL + 1.0f);
    const int64_t nv = (int64_t)xd * yd * zd;
    const bool ok = xd > 0 && yd > 0 && zd > 0 && nv <= k.vbudget;
    M->gmin[0] = e[0]; M->gmin[1] = e[2]; M->gmin[2] = e[4];
    M->dims[0] = ok ? xd : 1; M->dims[1] = ok ? yd : 1; M->dims[2] = ok ? zd : 1;
    if (!ok) atomicOr(&M->status, (uint32_t)CS3D_SYS_GRID_TOO_LARGE);
    // search bins of edge attraction_range + pair_skin covering the extent, or
    // fewer along the longest axes when the budget is short (periodic bins)
    float h = (k.ar + k.skin) * 1.001f;
    if (!(h > 0.f)) h = 1.0f;
    const float sz[3] = {e[1] - e[0], e[3] - e[2], e[5] - e[4]};
    int bd[3];
    for (int a = 0; a < 3; ++a) {
        const float q = sz[a] / h;
        bd[a] = (q >= 0.f && q < 1.0e6f) ? (int)q + 5 : 1000000;
    }
    for (int it = 0; it < 200; ++it) {
        if ((int64_t)bd[0] * bd[1] * bd[2] <= k.bbudget) break;
        const int a = bd[0] >= bd[1] && bd[0] >= bd[2] ? 0 : (bd[1] >= bd[2] ? 1 : 2);
        bd[a] = max(3, (int)(bd[a] * 0.9f));
    }
    for (int a = 0; a < 3; ++a) {
        M->bmin[a] = e[2 * a] - 2.0f * h;
        M->bdims[a] = bd[a];
    }
    M->bh = h;
    return ok ? nv : (int64_t)k.vbudget;
}

// {minx, maxx, miny, maxy, minz, maxz} of the node positions of one cell
// (workgroup of 192 lanes, nodes on lanes < 180) into out[6] and, through the
// shared part[3][6], to every lane's return in box[6].  Called by all lanes.
__device__ __forceinline__ void box_of_cell(float x, float y, float z, bool node, float (*part)[6], float* out,
                                            float* box = nullptr) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    float v[6] = {node ? x : INFINITY, node ? x : -INFINITY, node ? y : INFINITY,
                  node ? y : -INFINITY, node ? z : INFINITY, node ? z : -INFINITY};
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int a = 0; a < 6; a += 2) {
            v[a] = fminf(v[a], __shfl_xor(v[a], o));
            v[a + 1] = fmaxf(v[a + 1], __shfl_xor(v[a + 1], o));
        }
    }
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 6; ++a) part[wv][a] = v[a];
    __syncthreads();
    float b[6];
#pragma unroll
    for (int a = 0; a < 6; a += 2) {
        b[a] = fminf(fminf(part[0][a], part[1][a]), part[2][a]);
        b[a + 1] = fmaxf(fmaxf(part[0][a + 1], part[1][a + 1]), part[2][a + 1]);
    }
    __syncthreads();  // part is reused
    if (out && tid < 6) {
        float val = b[0];
#pragma unroll
        for (int a = 1; a < 6; ++a)
            if (tid == a) val = b[a];
        out[tid] = val;
    }
    if (box)
#pragma unroll
        for (int a = 0; a < 6; ++a) box[a] = b[a];
}

// ------------------------------------------------------------------------------
// Integrate + ForwardTime (propagate.cu:681-712, 738-763), PressureUpdate
// (PressureKernels.cu:4-41) and insertion of the new positions into the
// search bins.
// ------------------------------------------------------------------------------
// 6 waves per SIMD (at most 80 VGPRs): 8 workgroups per CU, one round for 2048 cells
// kLive: walk Pool::LIVE (a multi-system step) instead of the range's slots; kStep: the
// flags are those of the fused step (kStepFlags)
constexpr int32_t kStepFlags = I_KICK | I_PRESSURE | I_BINS | I_IFSEARCH | I_GRIDCOUNT;
template <int kLive, bool kStep>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_integrate(Pool p, Range r,
                                                                                              int32_t run_flags,
                                                                                              int64_t step_override) {
    const int32_t flags = kStep ? kStepFlags : run_flags;
    __shared__ float ibox[3][6];
    const int tid = threadIdx.x;
    const bool node = tid < kNodes;
    // a multi-system step walks the compact list of live slots (k_live)
    const int nit = kLive ? cld(p.n_live) : r.slot_hi - r.slot_lo;
    for (int it = first_cell<kLive>(nit, r); it < nit; it += gridDim.x) {
        const int2 at = cell_at<kLive>(r, p.LIVE, it);
        const int slot = at.x, s = at.y;
        // the cell's node data are loaded before the system checks (every slot of the
        // range is allocated), so their latency overlaps the metadata reads
        // (plain 64-bit node indices here: measured faster for this short kernel than
        // the uniform-base form of the other cell kernels)
        const int64_t gi = (int64_t)slot * kSlots + tid;
        float x = load_now(p.X + gi), y = load_now(p.Y + gi), z = load_now(p.Z + gi);
        const bool kick = flags & I_KICK;
        float vx = 0.f, vy = 0.f, vz = 0.f, fcx = 0.f, fcy = 0.f, fcz = 0.f, fdx = 0.f, fdy = 0.f, fdz = 0.f;
        if (kick) {
            vx = load_now(p.VX + gi); vy = load_now(p.VY + gi); vz = load_now(p.VZ + gi);
            fcx = load_now(p.FCX + gi); fcy = load_now(p.FCY + gi); fcz = load_now(p.FCZ + gi);
            fdx = load_now(p.FDX + gi); fdy = load_now(p.FDY + gi); fdz = load_now(p.FDZ + gi);
        }
        // metadata and parameters through scalar loads: this kernel writes no field it
        // reads (only status bits, by atomics)
        SysMeta* M = p.meta + s;
        asm volatile("" : "+s"(M));  // read in the loop: ahead of it the node loads would wait
        const CMeta MC = cmeta(M);
        const CParams P = cparams(p.prm + s);
        // the cell's new box, which a grid rebuild needs, with the same round trip
        const float* bn = p.BBOXN + (int64_t)slot * 6;
        const float b[6] = {cld(bn), cld(bn + 1), cld(bn + 2), cld(bn + 3), cld(bn + 4), cld(bn + 5)};
        const int32_t rebuild = MC->rebuild;
        asm volatile("" ::"s"(b[0]), "s"(b[1]), "s"(b[2]), "s"(b[3]), "s"(b[4]), "s"(b[5]), "s"(rebuild));
        int c;
        if (!cell_live<R_INTEGRATE>(MC, slot, c)) {
            if (kLive) continue;
            break;  // one system: neither is any cell after it
        }
        uint32_t* word = status_word<kStep, R_INTEGRATE>(M);
        const CPool q = pool_late();  // pointers read again where used (see pool_late)
        bool over = false;  // a voxel count beyond its capacity: looked at after the kick, which need not wait for it
        if ((flags & I_GRIDCOUNT) && rebuild && !(MC->status & CS3D_SYS_GRID_TOO_LARGE)) {
            // the grid was rebuilt at the end of the last step: this cell's new bbox
            // becomes the one the contact rule uses, and its voxels are counted
            // (makeNNlist's atomicAdd, propagatebound.cu:246-250) to catch overflow
            float mine = b[0];
#pragma unroll
            for (int a = 1; a < 6; ++a) mine = tid == a ? b[a] : mine;
            if (tid < 6) q->BBOX[(int64_t)slot * 6 + tid] = mine;
            const VoxRange v = vox_range(b, MC, P);
            store_vrange(q->VRANGE, slot, v, tid);
            const int nx = v.ex - v.sx + 1, ny = v.ey - v.sy + 1, nz = v.ez - v.sz + 1;
            const int total = (nx > 0 && ny > 0 && nz > 0) ? nx * ny * nz : 0;
            int32_t* counts = q->vox + MC->vbase;
            const int xd = MC->dims[0], yd = MC->dims[1], cap = MC->vcap;
            for (int t = tid; t < total; t += blockDim.x) {
                const int j3 = v.sz + t % nz, j2 = v.sy + (t / nz) % ny, j1 = v.sx + t / (nz * ny);
                if (atomicAdd(&counts[j3 * xd * yd + j2 * xd + j1], 1) >= cap) over = true;
            }
        }
        if (node && kick) {
            const float dt = P->dt, m = P->mass;
            const float rdt = sqrt_cr(dt);
            const bool rnd = P->add_rands != 0;  // the previous step's random force (d_fRanList)
            vx = half_kick(vx, fcx, fdx, rnd ? q->FRX[gi] : 0.f, dt, rdt, m, MC);
            vy = half_kick(vy, fcy, fdy, rnd ? q->FRY[gi] : 0.f, dt, rdt, m, MC);
            vz = half_kick(vz, fcz, fdz, rnd ? q->FRZ[gi] : 0.f, dt, rdt, m, MC);
            x = x + vx * dt;
            y = y + vy * dt;
            z = z + vz * dt;
            q->VAX[gi] = vx; q->VAY[gi] = vy; q->VAZ[gi] = vz;
            if (flags & I_WRITEV) { q->VX[gi] = vx; q->VY[gi] = vy; q->VZ[gi] = vz; }
            q->X[gi] = x; q->Y[gi] = y; q->Z[gi] = z;
        }
        if (node && (flags & I_CLEAR)) q->bins[MC->bbase + bin_of(MC, x, y, z)] = 0;
        if ((flags & I_BINS) && (!(flags & I_IFSEARCH) || MC->need_search)) {
            // insertion into the search bins, one atomic per node (the order of a bin's
            // entries does not matter: every candidate list is sorted).  Grouping the
            // lanes of a wave that share a bin behind one atomic was slower: the loop
            // over a wave's distinct bins cost more than the atomics it saved (the colony
            // at 20,000 cells: 0.215 against 0.188 ms for this kernel).  A partial search
            // (after divisions) works on search positions: the nodes of cells that did
            // not divide are binned at their last search position
            float qx = x, qy = y, qz = z;
            if ((flags & I_IFSEARCH) && MC->need_search == 2 && node && !q->RESET[slot]) {
                qx = q->XBX[gi]; qy = q->XBY[gi]; qz = q->XBZ[gi];
            }
            const int b = node ? bin_of(MC, qx, qy, qz) : -1;
            int32_t* counts = q->bins + MC->bbase;
            if (node) {
                const int k = atomicAdd(&counts[b], 1);
                if (k < kBCap) {
                    float4* ent = reinterpret_cast<float4*>(q->bins + MC->ebase);
                    ent[(int64_t)b * kBCap + k] = make_float4(qx, qy, qz, __int_as_float(c * kSlots + tid));
                } else {
                    flag(word, CS3D_SYS_BIN_OVERFLOW);
                }
            }
        }
        if (tid == 0 && (flags & I_PRESSURE)) {
            const int64_t stepno = step_override >= 0 ? step_override : MC->step + 1;
            const float inc = rgrowth(P, MC->n) * q->GS[slot];
            const float mx = P->max_pressure;
            float pr = q->P[slot];
            if (P->use_different_stiffnesses) {
                if (stepno < P->phase_count) {
                    if (pr < mx) pr += inc;
                } else if (q->E[slot] == P->stiffness1) {
                    if (pr < mx) pr += inc;
                } else if (pr != 0.f) {
                    pr = 0.f;
                }
            } else if (pr < mx) {
                pr += inc;
            }
            q->P[slot] = pr;
        }
        if (__any(over) && (tid & 63) == __ffsll((unsigned long long)__ballot(over)) - 1)
            atomicOr(word, (uint32_t)CS3D_SYS_VOXEL_OVERFLOW);
        if (kick && (flags & I_IFSEARCH) && MC->need_search == 2 && q->RESET[slot]) {
            // a cell that divided or left the skin in the last step publishes the box of
            // its new positions: the partial search re-searches the cells within reach
            box_of_cell(x, y, z, node, ibox, q->SBOX + (int64_t)slot * 6);
        }
    }
}

// ------------------------------------------------------------------------------
// Contact candidates of one node (called per lane by a cell workgroup): every
// node j of another cell within attraction_range + pair_skin, found by scanning
// the 27 search bins around the node.  Keys b*192 + j (local cell ids) are left
// ascending in lst[0 .. n)[tid]; returns n.
// ------------------------------------------------------------------------------
template <class MP, class PP>
__device__ int find_candidates(CPool p, MP M, PP P, int c, float X, float Y, float Z, int32_t (*lst)[kSlots],
                               int tid, uint32_t& st) {
    int nc = 0;
    const float rc = P->attraction_range + P->pair_skin;
    const float rc2 = rc * rc;
    const int bx = bin1(X, M->bmin[0], M->bh, M->bdims[0]);
    const int by = bin1(Y, M->bmin[1], M->bh, M->bdims[1]);
    const int bz = bin1(Z, M->bmin[2], M->bh, M->bdims[2]);
    const int bdx = M->bdims[0], bdy = M->bdims[1], bdz = M->bdims[2];
    const int32_t* counts = p->bins + M->bbase;
    const float4* ents = reinterpret_cast<const float4*>(p->bins + M->ebase);
    auto consider = [&](const float4 en) {
        const int key = __float_as_int(en.w);
        if ((unsigned)(key - c * kSlots) < (unsigned)kSlots) return;  // a node of this cell
        const float dX = X - en.x, dY = Y - en.y, dZ = Z - en.z;
        if (dX * dX + dY * dY + dZ * dZ > rc2) return;
        if (nc < kPMax) lst[nc][tid] = key;
        ++nc;
    };
    // 9 rows of 3 x-adjacent bins; the first 4 entries of each bin of a row are
    // loaded together (independent loads), longer bins finish in a tail loop; the
    // next row's counts load while a row is scanned
    constexpr int kHead = 4;
    int bin_n[3], cnt_n[3];
    {
        const int y3 = wrap1(by - 1, bdy), z3 = wrap1(bz - 1, bdz);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            bin_n[q] = (z3 * bdy + y3) * bdx + wrap1(bx + q - 1, bdx);
            cnt_n[q] = counts[bin_n[q]];
        }
    }
    for (int row = 0; row < 9; ++row) {
        int bi[3], cn[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            bi[q] = bin_n[q];
            cn[q] = min(cnt_n[q], kBCap);
        }
        if (row < 8) {
            const int y3 = wrap1(by + (row + 1) % 3 - 1, bdy), z3 = wrap1(bz + (row + 1) / 3 - 1, bdz);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                bin_n[q] = (z3 * bdy + y3) * bdx + wrap1(bx + q - 1, bdx);
                cnt_n[q] = counts[bin_n[q]];
            }
        }
        float4 head[3][kHead];  // loads of empty slots are masked off
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int e = 0; e < kHead; ++e)
                head[q][e] = e < cn[q] ? ents[(int64_t)bi[q] * kBCap + e] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
            for (int e = 0; e < kHead; ++e)
                if (e < cn[q]) consider(head[q][e]);
            for (int e = kHead; e < cn[q]; ++e) consider(ents[(int64_t)bi[q] * kBCap + e]);
        }
    }
    if (nc > kPMax) {
        st |= CS3D_SYS_CAND_OVERFLOW;
        nc = kPMax;
    }
    for (int i = 1; i < nc; ++i) {  // insertion sort of a short list
        const int key = lst[i][tid];
        int j = i - 1;
        while (j >= 0 && lst[j][tid] > key) {
            lst[j + 1][tid] = lst[j][tid];
            --j;
        }
        lst[j + 1][tid] = key;
    }
    return nc;
}

// The reference's candidate rule for node (X, Y, Z) in voxel (vx, vy, vz) and
// cell b: b is in the node's voxel list -- makeNNlist puts b into exactly the
// voxels of its bbox widened by attraction_range (propagatebound.cu:224-259),
// whose range is kept per cell in VRANGE -- and the node lies within
// attraction_range of b's bbox (propagate.cu:382-392).
struct RuleCtx {
    float ar2, DL, gx, gy, gz;
    int xd, yd, zd;
};

struct CellBox {  // voxel range and box of a cell
    int2 r01, r23, r45;
    float2 c01, c23, c45;
};
// sVR, sBB: voxel ranges and boxes from the system's first cell (uniform); b: the
// cell's local index
__device__ __forceinline__ CellBox load_cell_box(const int32_t* __restrict__ sVR, const float* __restrict__ sBB,
                                                 uint32_t b) {
    const int2* vr = reinterpret_cast<const int2*>(sVR);
    const float2* bb = reinterpret_cast<const float2*>(sBB);
    return CellBox{ldu(vr, 3 * b), ldu(vr, 3 * b + 1), ldu(vr, 3 * b + 2),
                   ldu(bb, 3 * b), ldu(bb, 3 * b + 1), ldu(bb, 3 * b + 2)};
}
__device__ __forceinline__ bool rule_ok(const CellBox& k, int vx, int vy, int vz, float X, float Y, float Z, float ar2) {
    const bool inlist = (k.r01.x <= vx) & (vx <= k.r01.y) & (k.r23.x <= vy) & (vy <= k.r23.y) & (k.r45.x <= vz) &
                        (vz <= k.r45.y);
    const float b0 = k.c01.x, b1 = k.c01.y, b2 = k.c23.x, b3 = k.c23.y, b4 = k.c45.x, b5 = k.c45.y;
    float qx = (float)(X - b1 > 0.0f) * (X - b1);
    qx += (float)(b0 - X > 0.0f) * (b0 - X);
    float qy = (float)(Y - b3 > 0.0f) * (Y - b3);
    qy += (float)(b2 - Y > 0.0f) * (b2 - Y);
    float qz = (float)(Z - b5 > 0.0f) * (Z - b5);
    qz += (float)(b4 - Z > 0.0f) * (b4 - Z);
    return inlist && !(qx * qx + qy * qy + qz * qz > ar2);
}

template <class MP, class PP>
__device__ __forceinline__ RuleCtx rule_ctx(MP M, PP P) {
    RuleCtx R;
    const float ar = P->attraction_range;
    R.ar2 = ar * ar;
    R.DL = P->grid_dl;
    R.gx = M->gmin[0]; R.gy = M->gmin[1]; R.gz = M->gmin[2];
    R.xd = M->dims[0]; R.yd = M->dims[1]; R.zd = M->dims[2];
    return R;
}

// The angle force's quotients idk/ra2 and idk/rb2 from the reciprocals ya2, yb2
// of ra2, rb2 (cs3d_div.h) where the operands are in range (quot_ok, quot_num_ok),
// by division otherwise: the same bits either way.  (-1/sqrt(inner) is -inv_rn.)
__device__ __forceinline__ void angle_quotients(float idk, float ra2, float ya2, float rb2, float yb2, float& ca,
                                                float& cb) {
    ca = quot_rn(idk, ra2, ya2);
    cb = quot_rn(idk, rb2, yb2);
    bool ok = quot_num_ok(idk);
    ok &= quot_ok(ra2);
    ok &= quot_ok(rb2);
    if (CS3D_SELDOM(!ok)) {
        ca = idk / ra2;
        cb = idk / rb2;
    }
}

// cs3d_acos as a call: for paths that hardly ever run, where inlining it would take
// registers for its constants from the common path.
__attribute__((noinline)) __device__ double acos_call(double x) { return cs3d_acos(x); }

// Shared GetAngleForce pair (propagate.cu:26-60): Fa = F(a-v, b-v), Fb = F(b-v, a-v).
// dot, |.|^2, c1 and theta are symmetric in the two arguments, so both come from
// one evaluation with bit-identical values.
template <bool kRare = false>
__device__ __forceinline__ uint32_t angle_pair(float ax, float ay, float az, float bx, float by, float bz,
                                               float th0, float k, float* out) {
    const float idk = ax * bx + ay * by + az * bz;
    const float ra2 = ax * ax + ay * ay + az * az;
    const float rb2 = bx * bx + by * by + bz * bz;
    const float inner = (float)((double)(ra2 * rb2 - idk * idk) + 1e-3);
    const float c1 = -inv_rn(sqrt_cr(inner));
    const float den = sqrt_cr(ra2) * sqrt_cr(rb2);
    const double x = (double)idk / ((double)den + 1e-3);
    const float theta = (float)(kRare ? acos_call(x) : cs3d_acos(x));
    const float s = ((-k) * c1) * (theta - th0);
    float ca, cb;
    angle_quotients(idk, ra2, rcp_rn(ra2), rb2, rcp_rn(rb2), ca, cb);
    out[0] = s * (bx - ca * ax); out[1] = s * (by - ca * ay); out[2] = s * (bz - ca * az);
    out[3] = s * (ax - cb * bx); out[4] = s * (ay - cb * by); out[5] = s * (az - cb * bz);
    bool ok = isfinite(out[0]) && isfinite(out[1]) && isfinite(out[2]) && isfinite(out[3]) && isfinite(out[4]) &&
              isfinite(out[5]);
    return ok ? 0u : (uint32_t)CS3D_SYS_ANGLE_NONFINITE;
}

// angle_pair for bonds with squared lengths ra2, rb2 in [2^-20, 2^20] (checked by the
// caller), their roots la, lb (which the node's springs use too) and
// the reciprocals ya2, yb2 = rcp_rn of them: the angle from cs3d_theta, the square
// root without scaling and the quotients from reciprocals.  Returns whether every
// operand was in the range of those steps (cs3d_theta's, c1's root in quot_ok's
// range, |idk| at least 2^-40, |s| at most 2^70); then every bit equals
// angle_pair's, and no component overflows: |b| <= 2^10 and |idk / ra2| <= 2^40
// bound them below 2^121.
__device__ __forceinline__ bool angle_pair_fast(float ax, float ay, float az, float ra2, float ya2, float la, float bx,
                                                float by, float bz, float rb2, float yb2, float lb, float th0, float k,
                                                CTheta c, float* out) {
    const float idk = ax * bx + ay * by + az * bz;
    const float inner = (float)((double)(ra2 * rb2 - idk * idk) + 1e-3);
    const float root = sqrt_normal(inner);
    const float c1 = -rcp_rn(root);
    const float den = la * lb;
    float theta;
    bool ok = cs3d_theta(idk, den, c, &theta);
    const float s = ((-k) * c1) * (theta - th0);
    const float ca = quot_rn(idk, ra2, ya2), cb = quot_rn(idk, rb2, yb2);
    out[0] = s * (bx - ca * ax); out[1] = s * (by - ca * ay); out[2] = s * (bz - ca * az);
    out[3] = s * (ax - cb * bx); out[4] = s * (ay - cb * by); out[5] = s * (az - cb * bz);
    ok &= quot_ok(root);
    ok &= fabsf(idk) >= 0x1p-40f;
    ok &= fabsf(s) <= 0x1p70f;
    return ok;
}

// The three angles of node tid, (n0,n1), (n1,n2), (n0,n2) (propagate.cu:26-60), to
// out[18] from its bond vectors, squared lengths b2 and lengths bl: by
// angle_pair_fast, and in a wave where an operand is out of its range again by
// angle_pair (a loop that is not unrolled, on vectors read again from the positions in
// LDS: it adds nothing to the registers live in the common path).
__device__ __forceinline__ uint32_t node_angles(const float* bx, const float* by, const float* bz, const float* b2,
                                                const float* bl, const MeshRec& mt, float k, const MeshDev* mesh,
                                                const float* sx, const float* sy, const float* sz, int tid,
                                                float* out) {
    const float y2[3] = {rcp_rn(b2[0]), rcp_rn(b2[1]), rcp_rn(b2[2])};
    // a NaN length leaves idk NaN in two of the angles, which their checks catch
    bool in = fminf(fminf(b2[0], b2[1]), b2[2]) >= 0x1p-20f;
    in &= fmaxf(fmaxf(b2[0], b2[1]), b2[2]) <= 0x1p20f;
    uint32_t bad = in ? 0u : 7u;
    CTheta c = (CTheta)&mesh->theta;
    asm volatile("" : "+s"(c));  // read here, not kept across cells
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int a = q == 1 ? 1 : 0, b = q == 0 ? 1 : 2;
        const bool ok = angle_pair_fast(bx[a], by[a], bz[a], b2[a], y2[a], bl[a], bx[b], by[b], bz[b], b2[b], y2[b],
                                        bl[b], mt.f[q], k, c, out + 6 * q);
        bad |= ok ? 0u : 1u << q;
    }
    uint32_t st = 0;
    if (bad) {
        slow_path();
        const float X = lds_reread(sx, tid), Y = lds_reread(sy, tid), Z = lds_reread(sz, tid);
        const float* th0 = reinterpret_cast<const float*>(mesh->th) + 4 * tid;
#pragma unroll 1
        for (int q = 0; q < 3; ++q) {
            if (!(bad >> q & 1u)) continue;
            const int a = mesh_nn(mt.w, q == 1 ? 1 : 0), b = mesh_nn(mt.w, q == 0 ? 1 : 2);
            st |= angle_pair<true>(sx[a] - X, sy[a] - Y, sz[a] - Z, sx[b] - X, sy[b] - Y, sz[b] - Z,
                                   th0[q], k, out + 6 * q);
        }
    }
    return st;
}

// friction normal of node tid (propagate.cu:558-572), positions in LDS
__device__ __forceinline__ void node_normal(const float* sx, const float* sy, const float* sz, float sg, int N1, int N2,
                                            int N3, float& nx, float& ny, float& nz) {
    const float Ax = sx[N2] - sx[N1], Ay = sy[N2] - sy[N1], Az = sz[N2] - sz[N1];
    const float Bx = sx[N3] - sx[N1], By = sy[N3] - sy[N1], Bz = sz[N3] - sz[N1];
    const float cx = Ay * Bz - Az * By, cy = Az * Bx - Ax * Bz, cz = Ax * By - Ay * Bx;
    const float inv = inv_sqrt_rn(cx * cx + cy * cy + cz * cz);
    nx = sg * (inv * cx);
    ny = sg * (inv * cy);
    nz = sg * (inv * cz);
}

struct PairConsts {
    float ar, ar2, rr, ka, kr, gext;
};

// Partner keys are local cell * 192 + node: the index of the node in a system's
// arrays, read through the system's first slot (a uniform pointer).

// The contact pass works on pairs, not on nodes: the candidates of a cell's nodes
// lie one after another in the cell's list (node order, each node's keys ascending,
// so reference order), and lane t of the workgroup takes entry c0 + t of the list,
// kSlots entries per round.  A node has 1 to 2 candidates on average but some node
// of every wave has 5 to 7, so a loop over each node's own candidates ran 5 to 7
// rounds with most lanes idle.  The lane applies the reference's tests to its pair
// and leaves the force terms in LDS; each node then adds the terms of its accepted
// pairs in list order, so every sum has the reference's order.
// NCAND holds a node's candidate count in its low kCandBits bits and the index of
// its first entry above them.  Which entries are accepted is kept as one bit per
// entry (pair_mask) for the second friction pass; the partner lists that callers
// read (CS3D_F_PAIRS) are made from it when they are read (k_pairs_list).
struct PairLds {
    float t[9][kSlots];    // attraction, repulsion and friction terms of the round's pairs
    uint64_t ok[4];        // accepted pairs of the round, one bit each (the fourth word stays 0)
};

// the n bits (1 to 63) from bit j of the words at m (one word past them is read)
__device__ __forceinline__ uint64_t bit_range(const uint64_t* m, int j, int n) {
    const int w = j >> 6, sh = j & 63;
    uint64_t bits = m[w] >> sh;
    if (sh) bits |= m[w + 1] << (64 - sh);
    return bits & ((1ull << n) - 1);
}

// owner[j] = node whose entry c0 + j is, for this lane's entries in the round of kRound entries
template <int kRound = kSlots>
__device__ __forceinline__ void fill_owners(uint8_t* owner, int tid, int first, int nc, int c0) {
    const int lo = max(first, c0), hi = min(first + nc, c0 + kRound);
    for (int j = lo; j < hi; ++j) owner[j - c0] = (uint8_t)tid;
}

// What a pair needs of its partner, all of it known from the key: loaded together
// (one memory round trip), before the lane needs any of it.
struct PairIn {
    float x, y, z, wx, wy, wz;  // position and velocity
    CellBox box;                // voxel range and box of its cell
};
// sX .. sVZ, sVR, sBB: node arrays, voxel ranges and boxes from the system's first
// slot (uniform)
struct SysArrays {
    const float *X, *Y, *Z, *VX, *VY, *VZ;
    const int32_t* VR;
    const float* BB;
};
template <bool DIS> __device__ __forceinline__ PairIn load_pair(int key, const SysArrays& a) {
    const uint32_t g = (uint32_t)key;
    PairIn in;
    in.x = ldu(a.X, g); in.y = ldu(a.Y, g); in.z = ldu(a.Z, g);
    if (DIS) { in.wx = ldu(a.VX, g); in.wy = ldu(a.VY, g); in.wz = ldu(a.VZ, g); }
    in.box = load_cell_box(a.VR, a.BB, g / kSlots);
    return in;
}

// The reference's tests and force terms for one pair (node at X with velocity
// vi and normal n, partner in): distance (ConForce skips
// R^2 >= ar^2, DisForce R^2 > ar^2, propagate.cu:421,641), the candidate rule of
// the partner's cell, the contact terms of propagate.cu:411-440 and the friction
// term of 633-653.  A term that does not apply stays 0: the sums start at +0 and
// never become -0, so adding it changes nothing.  Returns whether the pair is
// accepted.
template <bool CON, bool DIS>
__device__ __forceinline__ bool pair_terms(const PairIn& in, float X, float Y, float Z, float vix, float viy, float viz,
                                           float nx, float ny, float nz, const RuleCtx& R, const PairConsts& k,
                                           float* t) {
    const float dX = X - in.x, dY = Y - in.y, dZ = Z - in.z;
    const float R2 = dX * dX + dY * dY + dZ * dZ;
    if (R2 > k.ar2) return false;
    // the node's voxel (propagate.cu:360-372)
    const int vx = vox1(X, R.gx, R.DL, R.xd), vy = vox1(Y, R.gy, R.DL, R.yd), vz = vox1(Z, R.gz, R.DL, R.zd);
    if (!rule_ok(in.box, vx, vy, vz, X, Y, Z, R.ar2)) return false;
    if (CON && R2 < k.ar2) {
        const float Rl = sqrt_cr(R2);
        if (Rl < k.ar) {
            t[0] = k.ka * (k.ar - Rl) / Rl * dX;
            t[1] = k.ka * (k.ar - Rl) / Rl * dY;
            t[2] = k.ka * (k.ar - Rl) / Rl * dZ;
        }
        if (Rl <= k.rr) {
            t[3] = k.kr * (k.rr - Rl) / Rl * dX;
            t[4] = k.kr * (k.rr - Rl) / Rl * dY;
            t[5] = k.kr * (k.rr - Rl) / Rl * dZ;
        }
    }
    if (DIS) {
        const float ux = vix - in.wx, uy = viy - in.wy, uz = viz - in.wz;
        const float d = ux * nx + uy * ny + uz * nz;
        t[6] = k.gext * (ux - d * nx);
        t[7] = k.gext * (uy - d * ny);
        t[8] = k.gext * (uz - d * nz);
    }
    return true;
}

// All pairs of a cell (every lane of the workgroup calls it).  cand, mask: the
// cell's candidate list (flat) and its accepted entries, uniform; in: the lane's
// pair of the first round (where tid < total); first, nc: this lane's entries;
// total: entries of the cell;
// owner: filled for the first round and visible; sx .. snz: the
// cell's own positions, velocities and normals in LDS.  u is written only after a
// barrier that ends its previous use.
template <bool CON, bool DIS>
__device__ __forceinline__ void pair_pass(const int32_t* cand, uint64_t* mask, PairIn in, int tid, int first,
                                         int nc, int total, PairLds& u, uint8_t* owner, const RuleCtx& R,
                                         const PairConsts& k, const float* sx, const float* sy, const float* sz,
                                         const float* svx, const float* svy, const float* svz, const float* snx,
                                         const float* sny, const float* snz, const SysArrays& arr, float& cfx,
                                         float& cfy, float& cfz, float& fdx, float& fdy, float& fdz) {
    for (int c0 = 0; c0 < total; c0 += kSlots) {
        float t[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        bool ok = false;
        if (c0 + tid < total) {
            const int o = owner[tid];
            ok = pair_terms<CON, DIS>(in, sx[o], sy[o], sz[o], DIS ? svx[o] : 0.f, DIS ? svy[o] : 0.f,
                                      DIS ? svz[o] : 0.f, DIS ? snx[o] : 0.f, DIS ? sny[o] : 0.f, DIS ? snz[o] : 0.f, R,
                                      k, t);
        }
        __syncthreads();  // the previous use of u, and this round's owners, are done
        const uint64_t m = __ballot(ok);
        if ((tid & 63) == 0) {
            u.ok[tid >> 6] = m;
            mask[(c0 + tid) >> 6] = m;
        }
        if (tid == 0) u.ok[3] = 0;
        if (ok) {
            if (CON) {
#pragma unroll
                for (int a = 0; a < 6; ++a) u.t[a][tid] = t[a];
            }
            if (DIS) {
#pragma unroll
                for (int a = 6; a < 9; ++a) u.t[a][tid] = t[a];
            }
        }
        if (c0 + kSlots < total) {  // the next round's pair
            fill_owners(owner, tid, first, nc, c0 + kSlots);
            if (c0 + kSlots + tid < total) in = load_pair<DIS>(ldu(cand, (uint32_t)(c0 + kSlots + tid)), arr);
        }
        __syncthreads();
        const int lo = max(first, c0), hi = min(first + nc, c0 + kSlots);
        if (lo < hi) {  // this node's accepted pairs of the round, in list order
            uint64_t bits = bit_range(u.ok, lo - c0, hi - lo);
            while (bits) {
                const int j = lo - c0 + __ffsll((unsigned long long)bits) - 1;
                bits &= bits - 1;
                if (CON) {
                    cfx += u.t[0][j]; cfy += u.t[1][j]; cfz += u.t[2][j];
                    cfx += u.t[3][j]; cfy += u.t[4][j]; cfz += u.t[5][j];
                }
                if (DIS) { fdx = fdx - u.t[6][j]; fdy = fdy - u.t[7][j]; fdz = fdz - u.t[8][j]; }
            }
        }
    }
}

// A search replaces the candidates that the accept bits of the latest contact pass belong
// to.  Until the next pass is done the old list, counts and bits stay in the cell's room
// of the partner lists (kHeldAt 1; on a step k_dis_post ends it), so that a step that ends
// at its search leaves the partners that a caller reads as they were.  key0, ncf, total:
// the list's entry of this lane, the lane's NCAND word and the list's length.  Every lane
// of the workgroup calls it; the candidates may be written after the next barrier.
__device__ __forceinline__ void hold_partners(CPool p, int slot, int tid, int key0, int ncf, int total) {
    int32_t* cand = p->CAND + (size_t)slot * (kPMax * kSlots);
    int32_t* held = p->PAIRS + (size_t)slot * (kPMax * kSlots);
    if (tid < kMaskWords) pair_mask(p->PAIRS, slot)[tid] = pair_mask(p->CAND, slot)[tid];
    held[tid] = key0;
#pragma unroll 1
    for (int e = kSlots + tid; e < total; e += kSlots) held[e] = cand[e];
    p->NPAIR[(size_t)slot * kSlots + tid] = ncf;
    if (tid == 0) cand[kHeldAt] = 1;
}
__device__ __forceinline__ void release_partners(CPool p, int slot) {
    p->CAND[(size_t)slot * (kPMax * kSlots) + kHeldAt] = 0;
}

// ------------------------------------------------------------------------------
// Contact-candidate search (one cell per workgroup): on systems whose nodes
// moved pair_skin/2 since the last search (or always, outside the fused step),
// rebuild each node's sorted candidate list and remember the positions.
// ------------------------------------------------------------------------------
struct SearchLds {
    int32_t lst[kPMax][kSlots];
    float part[3][6];
    int32_t wsum[3];
};

// The search of one cell (every lane of the workgroup calls it) at its positions X,
// Y, Z (word: where an overflow is noted).  Returns whether the cell searched; then first, nc are this lane's entries
// of the new list and total their number.  u is written only after a barrier that
// ends its previous use, and is free when it returns.  hold: hold_partners with key0,
// ncf and oldn is still to be done (where the cell searches).
template <class MP, class PP>
__device__ __forceinline__ bool search_cell(CPool p, uint32_t* word, MP MC, PP P, int slot, int c, int tid, bool always,
                                            float X, float Y, float Z, bool hold, int key0, int ncf, int oldn,
                                            SearchLds& u, int& first, int& nc, int& total) {
    const bool node = tid < kNodes;
    const size_t cb = (size_t)slot * kSlots;  // the cell's first node (uniform)
    const uint32_t ln = lane_index();
    bool reset = true;
    if (!always && MC->need_search == 2) {
        // Partial search, in search positions.  The cells listed in RSL (RESET: a
        // node of the cell would leave the skin, or the cell divided) take their
        // current positions as search positions; every other node is within
        // pair_skin/2 of its search position.  Invariant: every list holds every
        // node of another cell within attraction_range + pair_skin in search
        // positions; with the pair_skin/2 bound it holds every node that is, or
        // comes, within attraction_range before the next search.  The nodes were
        // binned at their search positions (k_integrate), and SBOX holds the box of
        // every cell's search positions (the listed cells' new boxes from
        // k_integrate).  A cell whose box is farther than that radius from every
        // listed cell's box keeps its list: the invariant holds for it with the new
        // search positions.  The listed cells and the cells near them search again
        // around their search positions, so their lists are as long as after a full
        // search.
        const bool own = p->RESET[slot] != 0;
        if (!own) {
            const float* ob = p->SBOX + (int64_t)slot * 6;
            const float b[6] = {ob[0], ob[1], ob[2], ob[3], ob[4], ob[5]};
            const int nr = MC->n_part;
            const float mg = P->attraction_range + P->pair_skin;
            bool hit = false;
            if (tid < nr) {
                const int q = p->RSL[MC->base + tid];
                const float* o = p->SBOX + (int64_t)(MC->base + q) * 6;
                hit = b[0] - mg <= o[1] && o[0] <= b[1] + mg && b[2] - mg <= o[3] && o[2] <= b[3] + mg &&
                      b[4] - mg <= o[5] && o[4] <= b[5] + mg;
            }
            if (!__syncthreads_or(hit)) return false;
            X = ldu(p->XBX + cb, ln); Y = ldu(p->XBY + cb, ln); Z = ldu(p->XBZ + cb, ln);
        }
        reset = own;
    } else {
        // full search: the current positions become the search positions; their box
        // is kept for later partial searches
        box_of_cell(X, Y, Z, node, u.part, p->SBOX + (int64_t)slot * 6);
    }
    if (hold) hold_partners(p, slot, tid, key0, ncf, oldn);
    uint32_t st = 0;
    nc = node ? find_candidates(p, MC, P, c, X, Y, Z, u.lst, tid, st) : 0;
    // the cell's candidates one after another in node order: an exclusive scan of
    // the counts (shuffles within a wave, then the wave totals)
    first = nc;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(first, o);
        if ((tid & 63) >= o) first += t;
    }
    if ((tid & 63) == 63) u.wsum[tid >> 6] = first;
    __syncthreads();
    first -= nc;
    const int w0 = u.wsum[0], w1 = u.wsum[1];
    total = w0 + w1 + u.wsum[2];
    if (tid >= 64) first += w0;
    if (tid >= 128) first += w1;
    int32_t* cstore = p->CAND + (size_t)slot * kPMax * kSlots;
    for (int i = 0; i < nc; ++i) stu(cstore, (uint32_t)(first + i), u.lst[i][tid]);
    stu(p->NCAND + cb, ln, (first << kCandBits) | nc);  // the padding lanes hold the cell's total
    if (node && reset) { stu(p->XBX + cb, ln, X); stu(p->XBY + cb, ln, Y); stu(p->XBZ + cb, ln, Z); }
    if (st) flag(word, st);
    __syncthreads();
    return true;
}

// kLive: walk Pool::SRCH (a multi-system step: the cells of the systems that search)
// instead of the range's slots
template <int kLive>
__global__ __launch_bounds__(192) void k_search(Pool p, Range r, int32_t always) {
    __shared__ SearchLds u;
    if (r.one_sys && !always) {  // one system: its flag decides for every workgroup
        const CMeta M0 = cmeta(p.meta + r.sys_lo);
        if (!M0->need_search || !sys_live<R_SEARCH>(M0)) return;
    }
    // a multi-system step walks the cells of the systems that search (k_live)
    const int nit = kLive ? cld(p.n_live + 1) : r.slot_hi - r.slot_lo;
    for (int it = first_cell<kLive>(nit, r); it < nit; it += gridDim.x) {
        const int2 at = cell_at<kLive>(r, p.SRCH, it);
        const int slot = at.x, s = at.y;
        // metadata and parameters through scalar loads: this kernel writes none of
        // the fields it reads (only status bits, by atomics)
        SysMeta* M = p.meta + s;
        const CMeta MC = cmeta(M);
        int c;
        if (!cell_live<R_SEARCH>(MC, slot, c) || !(always || MC->need_search)) {
            if (kLive) continue;
            break;
        }
        const size_t cb = (size_t)slot * kSlots;
        const uint32_t ln = lane_index();
        const float X = ldu(p.X + cb, ln), Y = ldu(p.Y + cb, ln), Z = ldu(p.Z + cb, ln);
        const bool hold = always != kSearchAgain;
        const int key0 = ldu(p.CAND + cb * kPMax, ln), ncf = ldu(p.NCAND + cb, ln);
        const int oldn = cld(p.NCAND + cb + kNodes) >> kCandBits;
        int first, nc, total;
        uint32_t* word = always ? status_word<false, R_SEARCH>(M) : status_word<true, R_SEARCH>(M);
        search_cell(pool_late(), word, MC, cparams(p.prm + s), slot, c, threadIdx.x, always, X, Y, Z, hold, key0, ncf, oldn,
                    u, first, nc, total);
    }
}

// A step whose candidate search overflows ends there: no velocity, force or random
// force of it is kept.  Where the search runs at the head of k_con_dis the cells of the
// system cannot know of each other's overflow, so on a step that searches each keeps
// what the contact pass writes over (keep_cell), and the division phase puts it back
// (take_back_cell) in a system that overflowed.
struct Kept {
    float v[9];
};
__device__ __forceinline__ Kept load_kept(CPool p, bool rands, int slot, uint32_t ln) {
    const size_t cb = (size_t)slot * kSlots;
    Kept k;
    k.v[0] = ldu(p->VX + cb, ln); k.v[1] = ldu(p->VY + cb, ln); k.v[2] = ldu(p->VZ + cb, ln);
    k.v[3] = ldu(p->FCX + cb, ln); k.v[4] = ldu(p->FCY + cb, ln); k.v[5] = ldu(p->FCZ + cb, ln);
    k.v[6] = k.v[7] = k.v[8] = 0.f;
    if (rands) { k.v[6] = ldu(p->FRX + cb, ln); k.v[7] = ldu(p->FRY + cb, ln); k.v[8] = ldu(p->FRZ + cb, ln); }
    return k;
}
__device__ __forceinline__ void keep_cell(CPool p, const Kept& k, int slot, uint32_t ln) {
    float* q = p->KEEP + (size_t)slot * (9 * kSlots);
#pragma unroll
    for (int a = 0; a < 9; ++a) stu(q, a * kSlots + ln, k.v[a]);
}
__device__ __forceinline__ void take_back_cell(CPool p, bool rands, int slot, uint32_t ln) {
    const size_t cb = (size_t)slot * kSlots;
    const float* q = p->KEEP + 9 * cb;
    float* const to[9] = {p->VX, p->VY, p->VZ, p->FCX, p->FCY, p->FCZ, p->FRX, p->FRY, p->FRZ};
    for (int a = 0; a < (rands ? 9 : 6); ++a) stu(to[a] + cb, ln, ldu(q, a * kSlots + ln));
}

// Both before a search at the head of k_con_dis; a call, since inlined it takes registers
// from the step's common path (8 cells 23.0 against 23.15 us a step, 403 28.2 against 28.5).
__attribute__((noinline)) __device__ void hold_and_keep(CPool p, bool rands, int slot, uint32_t ln, int key0, int ncf,
                                                        int total) {
    const Kept kept = load_kept(p, rands, slot, ln);
    hold_partners(p, slot, (int)ln, key0, ncf, total);
    keep_cell(p, kept, slot, ln);
}
// ------------------------------------------------------------------------------
// Conservative force (CalculateConForce, propagate.cu:183-520) fused with the
// first dissipative force (CalculateDisForce with the post-Integrate
// velocities, propagate.cu:523-665) and VelocityUpdateA/B (propagate.cu:714-736),
// over the stored contact candidates.  Modes: M_STEP (FC, V, accepted
// partners), M_CON / M_INIT (FC, accepted partners), M_PAIRS (accepted partners only).
// ------------------------------------------------------------------------------
// 6 waves per SIMD (80 VGPRs, 20,064 B of LDS): 2048 workgroups fit on the chip at
// once, so 2000 cells run in one round instead of 1.5 (at 4 waves the kernel took
// 29.5 instead of 28.0 us, and k_dis_post, which reads its outputs next, 12.8 instead
// of 11.5).  No spills at that budget: the node's position is read again from LDS
// after the angles, the mesh tables are read at a uniform base plus the opaque lane
// offset where they are used, LDS indices are the opaque lane as well, and what the
// angles hardly ever need (angle_pair, the general acos) is a loop and a call.
// What bounds it: vector-ALU issue and the latency of each cell's chain of loads and
// barriers.  Pairs on lanes instead of a loop over each node's candidates, and the
// angles' short arithmetic, took it from 1577 to 1127 vector instructions per wave
// at 2000 cells (2017 to 1088 at 20,000): 22.9 to 21.0 us and 248 to 224 us a launch.
// With friction on accept bits, grids of one workgroup per cell and the entry chain
// cut (sys_live, CS3D_LOOP_POOL) it takes 18 and 137 us.
// kLive: walk Pool::LIVE (a multi-system step) instead of the range's slots; kStep:
// mode is M_STEP (the fused step has code of its own: as a run-time value the mode
// took scalar registers, spilled, throughout the kernel); kSearch: with the step's
// search (search_in_con)
union ForceLds {
    float angF[kNodes * 18];
    PairLds pr;
};
struct ConLds {
    float x[9][kSlots];  // positions, velocities and friction normals
    uint8_t owner[kSlots];
    ForceLds u;
};
union SharedLds {
    ConLds c;
    SearchLds s;
};
struct NoLds {};
template <int kLive, bool kStep, bool kSearch>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(kSearch ? 4 : 6, 8))) void k_con_dis(Pool pk, Range r,
                                                                                                        int32_t mode) {
    // the search and the contact pass share LDS; without the search, arrays of their own
    // (as parts of one object the compiler orders their accesses: 0.2 us at 2000 cells)
    constexpr int kOwn = kSearch ? 1 : kSlots;
    __shared__ float x0[kOwn], x1[kOwn], x2[kOwn], x3[kOwn], x4[kOwn], x5[kOwn], x6[kOwn], x7[kOwn], x8[kOwn];
    __shared__ uint8_t own_owner[kOwn];
    __shared__ std::conditional_t<kSearch, NoLds, ForceLds> own_u;
    __shared__ std::conditional_t<kSearch, SharedLds, NoLds> mem;
    float *sx = x0, *sy = x1, *sz = x2, *svx = x3, *svy = x4, *svz = x5, *snx = x6, *sny = x7, *snz = x8;
    uint8_t* owner = own_owner;
    if constexpr (kSearch) {
        sx = mem.c.x[0]; sy = mem.c.x[1]; sz = mem.c.x[2];
        svx = mem.c.x[3]; svy = mem.c.x[4]; svz = mem.c.x[5];
        snx = mem.c.x[6]; sny = mem.c.x[7]; snz = mem.c.x[8];
        owner = mem.c.owner;
    }
    ForceLds& u = [&]() -> ForceLds& {
        if constexpr (kSearch) return mem.c.u;
        else return own_u;
    }();
    const int tid = threadIdx.x;
    const bool node = tid < kNodes;
    constexpr bool fused = kStep;
    const bool forces = kStep || mode != M_PAIRS;
    // a multi-system step walks the compact list of live slots (k_live)
    int nit = kLive ? cld(pk.n_live) : r.slot_hi - r.slot_lo;
    int done = -1;  // kSearch: the iteration whose cell has searched
    for (int it = first_cell<kLive>(nit, r); it < nit; it += gridDim.x) {
        CS3D_LOOP_POOL(p);
        const MeshDev* mesh = p.mesh;
        const float *rX = p.X, *rY = p.Y, *rZ = p.Z, *rVX = p.VAX, *rVY = p.VAY, *rVZ = p.VAZ, *rBB = p.BBOX;
        asm volatile("" ::"s"(rX), "s"(rY), "s"(rZ), "s"(rVX), "s"(rVY), "s"(rVZ), "s"(mesh), "s"(p.NCAND), "s"(p.CAND),
                     "s"(p.meta), "s"(p.prm));  // (in one batch)
        const int2 at = cell_at<kLive>(r, p.LIVE, it);
        const int slot = at.x, s = at.y;
        // node data first (every slot of the range is allocated): their latency
        // overlaps the metadata reads
        const size_t cb = (size_t)slot * kSlots;  // the cell's first node (uniform)
        const uint32_t ln = lane_index();
        const int lt = (int)ln;  // for LDS indices as well: nothing per lane is kept across cells
        const float X = ldu_now(rX + cb, ln), Y = ldu_now(rY + cb, ln), Z = ldu_now(rZ + cb, ln);
        float vX = 0.f, vY = 0.f, vZ = 0.f;
        if (fused) { vX = ldu_now(rVX + cb, ln); vY = ldu_now(rVY + cb, ln); vZ = ldu_now(rVZ + cb, ln); }
        const int32_t* cand = p.CAND + (size_t)slot * kPMax * kSlots;  // the cell's candidate list (uniform)
        const int ncf = ldu_now(p.NCAND + cb, ln);
        const int key0 = ldu_now(cand, ln);  // the first round's keys (in the list's room also where it is shorter)
        // entries of the list, from a padding lane (by a vector load where this kernel
        // may have just written it: the scalar cache does not see that)
        int total = kSearch ? ldu_now(p.NCAND + cb, vector_value(kNodes)) : cld(p.NCAND + cb + kNodes) >> kCandBits;
        const MeshRec mt = ldu(mesh->th, ln);
        const float sg = fused ? ldu(mesh->gs, ln).sign : 0.f;
        const MeshRec r0 = ldu(mesh->r0, ln), ir0 = ldu(mesh->ir0, ln);
        SysMeta* M = p.meta + s;
        // parameters and the fields of the metadata that this kernel does not write
        // (but for status bits, by atomics), through scalar loads
        const CMeta MC = cmeta(M);
        const int32_t need = kSearch ? MC->need_search : 0;
        int c;
        const bool live = cell_live<kStep ? R_CON : 0>(MC, slot, c);
        if (kSearch) asm volatile("" ::"s"(need), "s"(c), "s"((int)live));  // (with the same round trip)
        if (!live) {
            if (!kLive) nit = 0;  // one system: neither is any cell after it
            continue;
        }
        uint32_t* word = status_word<kStep, R_CON>(M);
        const int sbase = slot - c;
        const CParams P = cparams(p.prm + s);
        if constexpr (kSearch) {
            // the search of this step (search_in_con); the iteration then starts again
            // with the new list, so that none of its registers live through the search
            if (__builtin_expect(need && done != it, 0)) {
                int f, n, t;
                hold_and_keep(pool_late(), P->add_rands != 0, slot, ln, key0, ncf,
                              __builtin_amdgcn_readfirstlane(total) >> kCandBits);
                __syncthreads();
                search_cell(pool_late(), word, MC, P, slot, c, lt, false, X, Y, Z, false, 0, 0, 0, mem.s, f, n, t);
                done = it;
                it -= gridDim.x;
                continue;
            }
        }
        sx[lt] = X; sy[lt] = Y; sz[lt] = Z;
        if (fused) { svx[lt] = vX; svy[lt] = vY; svz[lt] = vZ; }
        if (fused && tid == 0) {  // this cell's search of this step is done; k_dis_post lists anew
            p.RESET[slot] = 0;
            if (c == 0) M->n_reset = 0;
        }
        if (!kStep && tid == 0) release_partners(pool_late(), slot);
        __syncthreads();
        uint32_t st = 0;
        const bool angles = forces && P->constrain_angles;
        float FX = 0.f, FY = 0.f, FZ = 0.f;
        if (forces) {
            if (node && (isnan(X) || isnan(Y) || isnan(Z))) st |= CS3D_SYS_NAN;  // propagate.cu:241-248
            if (fused && node) {
                float nx, ny, nz;
                node_normal(sx, sy, sz, sg, mesh_nn(mt.w, 0), mesh_nn(mt.w, 1), mesh_nn(mt.w, 2), nx, ny, nz);
                snx[lt] = nx; sny[lt] = ny; snz[lt] = nz;
            }
            if (node) {
                // the node's three bonds: vectors, squared lengths and lengths, used by the
                // node's own three angles (propagate.cu:26-60) and by the springs
                // (propagate.cu:298-314), which compute the same quantities from the same
                // vectors.  The angles write to LDS only and are summed after the pressure, as
                // in the reference.
                float bx[3], by[3], bz[3], b2[3], bl[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int N1 = mesh_nn(mt.w, i);
                    bx[i] = sx[N1] - X; by[i] = sy[N1] - Y; bz[i] = sz[N1] - Z;
                    b2[i] = bx[i] * bx[i] + by[i] * by[i] + bz[i] * bz[i];
                    bl[i] = sqrt_normal(b2[i]);
                }
                // ---- springs, propagate.cu:298-314
                const float stiffness = cld(p.E + slot);
                bool ok = true;
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    float tx, ty, tz;
                    ok &= spring_rcp(stiffness, bl[i], r0.f[i], ir0.f[i], bx[i], by[i], bz[i], tx, ty, tz);
                    FX += tx;
                    FY += ty;
                    FZ += tz;
                }
                if (CS3D_SELDOM(!ok)) {  // an operand out of range: the three springs by division
                    FX = 0.f; FY = 0.f; FZ = 0.f;
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        float tx, ty, tz;
                        spring_div(stiffness, sqrt_cr(b2[i]), r0.f[i], bx[i], by[i], bz[i], tx, ty, tz);
                        FX += tx;
                        FY += ty;
                        FZ += tz;
                    }
                }
                if (angles) {  // each angle once (propagate.cu:26-60): (n0,n1), (n1,n2), (n0,n2)
                    st |= node_angles(bx, by, bz, b2, bl, mt, P->angle_k, mesh, sx, sy, sz, lt, u.angF + lt * 18);
                }
            }
        }
        if constexpr (kSearch) total = __builtin_amdgcn_readfirstlane(total) >> kCandBits;
        const int nc = ncf & ((1 << kCandBits) - 1), first = ncf >> kCandBits;
        float fdx = 0.f, fdy = 0.f, fdz = 0.f;
        fill_owners(owner, lt, first, nc, 0);
        if (fused && node) {
            const float vix = svx[lt], viy = svy[lt], viz = svz[lt];
            const float gint = P->internal_damping;
            const uint32_t nnw = ldu(mesh->th, lane_index()).w;
            const int nn3[3] = {mesh_nn(nnw, 0), mesh_nn(nnw, 1), mesh_nn(nnw, 2)};
#pragma unroll
            for (int i = 0; i < 3; ++i) {  // bond damping, propagate.cu:547-554
                const int N = nn3[i];
                fdx = fdx - gint * (vix - svx[N]);
                fdy = fdy - gint * (viy - svy[N]);
                fdz = fdz - gint * (viz - svz[N]);
            }
        }
        // the lane's first pair and the gather table load while the barrier and the
        // gather of the angle forces pass
        const size_t sb = (size_t)sbase * kSlots;  // the system's first node
        const SysArrays arr{rX + sb, rY + sb, rZ + sb, rVX + sb, rVY + sb, rVZ + sb, p.VRANGE + (size_t)sbase * 6,
                            rBB + (size_t)sbase * 6};
        // (lanes past the list load their own node)
        const PairIn in = load_pair<fused>(lt < total ? key0 : c * kSlots + lt, arr);
        uint32_t gt[3] = {0u, 0u, 0u};
        if (angles) {
            const uint32_t lg = lane_index();
            gt[0] = ldu(mesh->r0, lg).w; gt[1] = ldu(mesh->ir0, lg).w; gt[2] = ldu(mesh->gs, lg).w;
        }
        __syncthreads();  // the angle forces, normals and owners of every node are in LDS
        if (forces) {
            if (node) {
                const float X = lds_reread(sx, lt), Y = lds_reread(sy, lt), Z = lds_reread(sz, lt);
                // ---- pressure, propagate.cu:318-330 (centre of mass from the last CenterOfMass)
                const float rx = X - cld(p.CMX + slot), ry = Y - cld(p.CMY + slot), rz = Z - cld(p.CMZ + slot);
                const float inv = inv_sqrt_rn(rx * rx + ry * ry + rz * rz);
                const float g = 3.0f * cld(p.P + slot);
                FX += g * (inv * rx);
                FY += g * (inv * ry);
                FZ += g * (inv * rz);
            }
            // ---- angle forces gathered in the summation order of CalculateAngleForce (propagate.cu:81-181)
            if (angles && node) {
                const float* a = u.angF + lt * 18;
                float ax = 0.f, ay = 0.f, az = 0.f;
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    ax = ax - (a[q * 6 + 0] + a[q * 6 + 3]);
                    ay = ay - (a[q * 6 + 1] + a[q * 6 + 4]);
                    az = az - (a[q * 6 + 2] + a[q * 6 + 5]);
                }
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    const float* f = u.angF + ((gt[q >> 1] >> (16 * (q & 1))) & 0xffffu);
                    ax = ax + f[0];
                    ay = ay + f[1];
                    az = az + f[2];
                }
                FX += ax; FY += ay; FZ += az;
            }
        }
        float cfx = 0.f, cfy = 0.f, cfz = 0.f;
        if (total > 0) {
            const RuleCtx R = rule_ctx(MC, P);
            PairConsts k;
            k.ar = P->attraction_range;
            k.ar2 = k.ar * k.ar;
            k.rr = P->repulsion_range;
            k.ka = -P->attraction_strength * P->youngs_mod;
            k.kr = +P->repulsion_strength * P->youngs_mod;
            k.gext = P->viscotic_damping;
            uint64_t* mask = pair_mask(p.CAND, slot);
            if (fused)
                pair_pass<true, true>(cand, mask, in, lt, first, nc, total, u.pr, owner, R, k, sx, sy, sz, svx,
                                           svy, svz, snx, sny, snz, arr, cfx, cfy, cfz, fdx, fdy, fdz);
            else if (forces)
                pair_pass<true, false>(cand, mask, in, lt, first, nc, total, u.pr, owner, R, k, sx, sy, sz, svx,
                                            svy, svz, snx, sny, snz, arr, cfx, cfy, cfz, fdx, fdy, fdz);
            else
                pair_pass<false, false>(cand, mask, in, lt, first, nc, total, u.pr, owner, R, k, sx, sy, sz,
                                             svx, svy, svz, snx, sny, snz, arr, cfx, cfy, cfz, fdx, fdy, fdz);
        }
        if (node) {
            const float X = lds_reread(sx, lt), Y = lds_reread(sy, lt), Z = lds_reread(sz, lt);
            if (fused) {
                const float vix = svx[lt], viy = svy[lt], viz = svz[lt];
                fdx = fdx - P->gamma_visc * vix;  // drag, propagate.cu:658
                fdy = fdy - P->gamma_visc * viy;
                fdz = fdz - P->gamma_visc * viz;
            }
            if (forces) {
                FX += cfx; FY += cfy; FZ += cfz;
                if (P->use_rigid_box) {  // propagate.cu:473-510 (lower wall at 0)
                    const float E = P->youngs_mod, thr = P->thresh_dist;
                    float g1 = X, g2 = P->box_max[0] - X;
                    if (g1 < thr) FX += -100.0f * E * (g1 - thr);
                    if (g2 < thr) FX += 100.0f * E * (g2 - thr);
                    g1 = Y; g2 = P->box_max[1] - Y;
                    if (g1 < thr) FY += -100.0f * E * (g1 - thr);
                    if (g2 < thr) FY += 100.0f * E * (g2 - thr);
                    g1 = Z; g2 = P->box_max[2] - Z;
                    if (g1 < thr) FZ += -100.0f * E * (g1 - thr);
                    if (g2 < thr) FZ += 100.0f * E * (g2 - thr);
                }
            }
            if (fused) {
                const float dt = P->dt, m = P->mass;
                const float rdt = sqrt_cr(dt);
                float frx = 0.f, fry = 0.f, frz = 0.f;
                if (P->add_rands) {  // CalculateRanForce for this step (propagate.cu:667-676)
                    float zr[3];
                    noise3(P->noise_seed, (uint32_t)(c * kSlots + lt), MC->step + 1, zr);
                    const float sc = P->rand_scale_factor;
                    frx = sc * zr[0]; fry = sc * zr[1]; frz = sc * zr[2];
                    const CPool q = pool_late();
                    stu(q->FRX + cb, ln, frx); stu(q->FRY + cb, ln, fry); stu(q->FRZ + cb, ln, frz);
                }
                const float vix = svx[lt], viy = svy[lt], viz = svz[lt];
                // VelocityUpdateA (propagate.cu:721-723) then VelocityUpdateB (:732-734)
                float vx = (float)((double)vix + kick_a(dt * FX + rdt * frx, m, MC));
                float vy = (float)((double)viy + kick_a(dt * FY + rdt * fry, m, MC));
                float vz = (float)((double)viz + kick_a(dt * FZ + rdt * frz, m, MC));
                vx = (float)((double)vx + kick_b(fdx, dt, m, MC));
                vy = (float)((double)vy + kick_b(fdy, dt, m, MC));
                vz = (float)((double)vz + kick_b(fdz, dt, m, MC));
                const CPool q = pool_late();
                stu(q->VX + cb, ln, vx); stu(q->VY + cb, ln, vy); stu(q->VZ + cb, ln, vz);
            }
        }
        if (node && forces) {
            const CPool q = pool_late();
            stu(q->FCX + cb, ln, FX); stu(q->FCY + cb, ln, FY); stu(q->FCZ + cb, ln, FZ);
        }
        if (st) flag(word, st);
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------
// Bonded part of CalculateConForce alone (springs, pressure, and angles when
// constrainAngles): propagate.cu:253-337, the same arithmetic and summation
// order as k_con_dis, in a lean streaming kernel for the standalone bonded
// entry point.  Without angles it moves x in and F_con out (24 B per node): the
// per-lane mesh data stay in registers across the cells a workgroup walks, and
// the next cell's positions are loaded while the current one is computed.
// ------------------------------------------------------------------------------
template <bool ANGLES>
__global__ __launch_bounds__(192) void k_bonded(Pool p, Range r) {
    __shared__ float sx[kSlots], sy[kSlots], sz[kSlots];
    __shared__ float angF[ANGLES ? kNodes * 18 : 1];
    const int tid = threadIdx.x;
    const bool node = tid < kNodes;
    const MeshDev* mesh = p.mesh;
    int nb[3] = {0, 0, 0};
    float r0[3] = {1.f, 1.f, 1.f}, ir0[3] = {1.f, 1.f, 1.f}, th[3] = {0.f, 0.f, 0.f};
    if (node) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            nb[i] = mesh_nn(mesh->th[tid].w, i);
            r0[i] = mesh->r0[tid].f[i];
            ir0[i] = mesh->ir0[tid].f[i];
            if (ANGLES) th[i] = mesh->th[tid].f[i];
        }
    }
    int slot = r.slot_lo + blockIdx.x;
    float X = 0.f, Y = 0.f, Z = 0.f;
    if (slot < r.slot_hi) {
        const int64_t gi = (int64_t)slot * kSlots + tid;
        X = p.X[gi]; Y = p.Y[gi]; Z = p.Z[gi];
    }
    for (; slot < r.slot_hi; slot += gridDim.x) {
        // prefetch the next cell of this workgroup (in bounds: slot < slot_hi <= capacity)
        const int nslot = slot + gridDim.x;
        float Xn = 0.f, Yn = 0.f, Zn = 0.f;
        if (nslot < r.slot_hi) {
            const int64_t gn = (int64_t)nslot * kSlots + tid;
            Xn = p.X[gn]; Yn = p.Y[gn]; Zn = p.Z[gn];
        }
        const int s = sys_of(p, r, slot);
        bool use = s >= 0;
        SysMeta* M = use ? p.meta + s : nullptr;
        const cs3d_params* P = use ? p.prm + s : nullptr;
        use = use && sys_live(M) && slot - M->base < M->n && (P->constrain_angles != 0) == ANGLES;
        if (use) {
            const int64_t gi = (int64_t)slot * kSlots + tid;
            sx[tid] = X; sy[tid] = Y; sz[tid] = Z;
            __syncthreads();
            uint32_t st = 0;
            if (ANGLES) {
                if (node) {
                    const float k = P->angle_k;
#pragma unroll 1
                    for (int q = 0; q < 3; ++q) {
                        const int a = q == 1 ? nb[1] : nb[0];
                        const int b = q == 0 ? nb[1] : nb[2];
                        const float t0 = q == 0 ? th[0] : (q == 1 ? th[1] : th[2]);
                        st |= angle_pair(sx[a] - X, sy[a] - Y, sz[a] - Z, sx[b] - X, sy[b] - Y, sz[b] - Z, t0, k,
                                         angF + (tid * 3 + q) * 6);
                    }
                }
                __syncthreads();
            }
            if (node) {
                if (isnan(X) || isnan(Y) || isnan(Z)) st |= CS3D_SYS_NAN;
                float FX = 0.f, FY = 0.f, FZ = 0.f;
                const float stiffness = p.E[slot];
                float dX[3], dY[3], dZ[3], R[3];
                bool ok = true;
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int N1 = nb[i];
                    dX[i] = sx[N1] - X; dY[i] = sy[N1] - Y; dZ[i] = sz[N1] - Z;
                    R[i] = sqrt_cr(dX[i] * dX[i] + dY[i] * dY[i] + dZ[i] * dZ[i]);
                    float tx, ty, tz;
                    ok &= spring_rcp(stiffness, R[i], r0[i], ir0[i], dX[i], dY[i], dZ[i], tx, ty, tz);
                    FX += tx;
                    FY += ty;
                    FZ += tz;
                }
                if (CS3D_SELDOM(!ok)) {  // an operand out of range: the three springs by division
                    FX = 0.f; FY = 0.f; FZ = 0.f;
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        float tx, ty, tz;
                        spring_div(stiffness, R[i], r0[i], dX[i], dY[i], dZ[i], tx, ty, tz);
                        FX += tx;
                        FY += ty;
                        FZ += tz;
                    }
                }
                const float rx = X - p.CMX[slot], ry = Y - p.CMY[slot], rz = Z - p.CMZ[slot];
                const float inv = inv_sqrt_rn(rx * rx + ry * ry + rz * rz);
                const float g = 3.0f * p.P[slot];
                FX += g * (inv * rx);
                FY += g * (inv * ry);
                FZ += g * (inv * rz);
                if (ANGLES) {
                    const float* a = angF + tid * 18;
                    float ax = 0.f, ay = 0.f, az = 0.f;
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        ax = ax - (a[q * 6 + 0] + a[q * 6 + 3]);
                        ay = ay - (a[q * 6 + 1] + a[q * 6 + 4]);
                        az = az - (a[q * 6 + 2] + a[q * 6 + 5]);
                    }
                    const uint32_t gt[3] = {mesh->r0[tid].w, mesh->ir0[tid].w, mesh->gs[tid].w};
#pragma unroll
                    for (int q = 0; q < 6; ++q) {
                        const float* f = angF + ((gt[q >> 1] >> (16 * (q & 1))) & 0xffffu);
                        ax = ax + f[0];
                        ay = ay + f[1];
                        az = az + f[2];
                    }
                    FX += ax; FY += ay; FZ += az;
                }
                p.FCX[gi] = FX; p.FCY[gi] = FY; p.FCZ[gi] = FZ;
            }
            if (st) flag(&M->status, st);
            __syncthreads();
        }
        X = Xn; Y = Yn; Z = Zn;
    }
}

// ------------------------------------------------------------------------------
// Reductions over a wave without LDS.  lane_down<o> gives a lane the value of the
// lane o above it, for the lanes that a tree reduction to lane 0 still uses at that
// level (lanes below o): the halves and rows of a wave are swapped by
// v_permlane32_swap / v_permlane16_swap, within a row of 16 the DPP row shift reads
// upwards.  The pairs are those of the shuffle tree (i, i + o), o = 32 .. 1.
// ------------------------------------------------------------------------------
template <int o> __device__ __forceinline__ float lane_down(float v) {
    const uint32_t x = __float_as_uint(v);
    if constexpr (o == 32) return __uint_as_float(__builtin_amdgcn_permlane32_swap(x, x, false, false)[1]);
    else if constexpr (o == 16) return __uint_as_float(__builtin_amdgcn_permlane16_swap(x, x, false, false)[1]);
    else return __int_as_float(__builtin_amdgcn_update_dpp(0, (int)x, 0x100 | o, 0xf, 0xf, true));
}
struct OpAdd { static __device__ __forceinline__ float f(float a, float b) { return a + b; } };
struct OpMin { static __device__ __forceinline__ float f(float a, float b) { return fminf(a, b); } };
struct OpMax { static __device__ __forceinline__ float f(float a, float b) { return fmaxf(a, b); } };
template <class Op> __device__ __forceinline__ float wave_tree(float v) {  // the result is lane 0's
    v = Op::f(v, lane_down<32>(v));
    v = Op::f(v, lane_down<16>(v));
    v = Op::f(v, lane_down<8>(v));
    v = Op::f(v, lane_down<4>(v));
    v = Op::f(v, lane_down<2>(v));
    return Op::f(v, lane_down<1>(v));
}
// the value of the even lane of each lane pair
__device__ __forceinline__ float even_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xa0, 0xf, 0xf, true));  // quad_perm 0 0 2 2
}

// ------------------------------------------------------------------------------
// Dissipative force (CalculateDisForce, propagate.cu:523-665) with the
// end-of-step velocities, then CenterOfMass (centermass.cu:8-50) and, on growth
// steps, volumes (volume.cu:5-163).  Modes: M_STEP, M_DIS_V, M_DIS_VA, M_COM,
// M_VOLUMES.
// ------------------------------------------------------------------------------
// What bounds it: at a few hundred cells the latency of one cell's chain (loads,
// barriers, dependent arithmetic), at 20,000 cells memory traffic.  Friction works
// on pairs as in k_con_dis, two entries of the cell's candidate list per lane and
// round (384 cover most cells in one round), gated by the accept bits that
// k_con_dis left; the centre of mass is one wave's work straight from the positions
// in LDS, beside the other waves' normals; the box and the trees use cross-lane
// moves instead of LDS; each face is shared by two lanes, which split its edges.
// kLive: walk Pool::LIVE (a multi-system step) instead of the range's slots; kStep:
// mode is M_STEP
template <int kLive, bool kStep>
__global__ __launch_bounds__(192) void k_dis_post(Pool p, Range r, int32_t mode, int64_t step_override,
                                                  int32_t clear_bins, const float* __restrict__ rX,
                                                  const float* __restrict__ rY, const float* __restrict__ rZ,
                                                  const float* __restrict__ rVX, const float* __restrict__ rVY,
                                                  const float* __restrict__ rVZ) {
    constexpr int kRound = 2 * kSlots;
    __shared__ float sx[kSlots], sy[kSlots], sz[kSlots];
    __shared__ float svx[kSlots], svy[kSlots], svz[kSlots];
    __shared__ float snx[kSlots], sny[kSlots], snz[kSlots];  // friction normals
    __shared__ float term[3][kRound];                        // friction terms of the round's pairs
    __shared__ uint64_t okm[kRound / 64 + 1];                // their accept bits (the last word stays 0)
    __shared__ uint8_t owner[kRound];
    __shared__ float red[2][128];
    __shared__ float cm[3];
    __shared__ float bpart[3][6];
    __shared__ int32_t moved;
    const int tid = threadIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool node = tid < kNodes;
    const MeshDev* mesh = p.mesh;
    const bool do_dis = kStep || mode == M_DIS_V || mode == M_DIS_VA;
    constexpr bool fused = kStep;
    // a multi-system step walks the compact list of live slots (k_live)
    const int nit = kLive ? cld(p.n_live) : r.slot_hi - r.slot_lo;
    for (int it = first_cell<kLive>(nit, r); it < nit; it += gridDim.x) {
        const int2 at = cell_at<kLive>(r, p.LIVE, it);
        const int slot = at.x, s = at.y;
        // node data first (every slot of the range is allocated): their latency
        // overlaps the metadata reads
        const size_t cb = (size_t)slot * kSlots;  // the cell's first node (uniform)
        const uint32_t ln = lane_index();
        const int lt = (int)ln;
        const float X = ldu_now(rX + cb, ln), Y = ldu_now(rY + cb, ln), Z = ldu_now(rZ + cb, ln);
        float vX = 0.f, vY = 0.f, vZ = 0.f;
        const int32_t* cand = p.CAND + (size_t)slot * kPMax * kSlots;
        const uint64_t* mask = pair_mask(p.CAND, slot);
        int ncf = 0, total = 0, key[2] = {0, 0};
        uint64_t m[2] = {0, 0};  // this wave's words of the first round
        if (do_dis) {
            vX = ldu_now(rVX + cb, ln); vY = ldu_now(rVY + cb, ln); vZ = ldu_now(rVZ + cb, ln);
            ncf = ldu_now(p.NCAND + cb, ln);
            key[0] = ldu_now(cand, ln); key[1] = ldu_now(cand, ln + kSlots);
            total = cld(p.NCAND + cb + kNodes) >> kCandBits;
            m[0] = cld(mask + wv); m[1] = cld(mask + 3 + wv);
        }
        float fcX = 0.f, fcY = 0.f, fcZ = 0.f, xbX = 0.f, xbY = 0.f, xbZ = 0.f;
        if (fused) {  // (padding lanes load their padding)
            fcX = ldu_now(p.FCX + cb, ln); fcY = ldu_now(p.FCY + cb, ln); fcZ = ldu_now(p.FCZ + cb, ln);
            xbX = ldu_now(p.XBX + cb, ln); xbY = ldu_now(p.XBY + cb, ln); xbZ = ldu_now(p.XBZ + cb, ln);
        }
        const uint32_t nnw = do_dis ? ldu(mesh->th, ln).w : 0u;
        const float sg = do_dis ? ldu(mesh->gs, ln).sign : 0.f;
        // metadata and parameters through scalar loads: the fields read here are not
        // written by this kernel (search_next and n_reset, which it updates by atomics,
        // are read by atomic loads)
        SysMeta* M = p.meta + s;
        const CMeta MC = cmeta(M);
        const CParams P = cparams(p.prm + s);
        int c;
        if (!cell_live<kStep ? R_POST : 0>(MC, slot, c)) {
            if (kLive) continue;
            break;  // one system: neither is any cell after it
        }
        const int nc = ncf & ((1 << kCandBits) - 1), first = ncf >> kCandBits;
        if (tid == 0) { moved = 0; okm[kRound / 64] = 0; }
        sx[lt] = X; sy[lt] = Y; sz[lt] = Z;
        if (do_dis) {
            svx[lt] = vX; svy[lt] = vY; svz[lt] = vZ;
            fill_owners<kRound>(owner, lt, first, nc, 0);
        }
        __syncthreads();
        uint32_t st = 0;
        const size_t sb = (size_t)MC->base * kSlots;  // the system's first node
        float fx = 0.f, fy = 0.f, fz = 0.f;
        float wx[2], wy[2], wz[2];  // partner velocities of the lane's accepted pairs
        bool acc[2];
        auto load_partners = [&](int c0) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool in = c0 + h * kSlots + lt < total;
                acc[h] = in && (m[h] >> (lt & 63) & 1);
                const uint32_t g = acc[h] ? (uint32_t)key[h] : (uint32_t)(c * kSlots + lt);
                wx[h] = ldu(rVX + sb, g); wy[h] = ldu(rVY + sb, g); wz[h] = ldu(rVZ + sb, g);
                if ((lt & 63) == 0) okm[3 * h + (lt >> 6)] = c0 + h * kSlots < total ? m[h] : 0;
            }
        };
        if (do_dis) load_partners(0);
        if (do_dis && node) {
            const float vix = svx[lt], viy = svy[lt], viz = svz[lt];
            const float gint = P->internal_damping;
            const int nn3[3] = {mesh_nn(nnw, 0), mesh_nn(nnw, 1), mesh_nn(nnw, 2)};
#pragma unroll
            for (int i = 0; i < 3; ++i) {  // bond damping, propagate.cu:547-554
                const int N = nn3[i];
                fx = fx - gint * (vix - svx[N]);
                fy = fy - gint * (viy - svy[N]);
                fz = fz - gint * (viz - svz[N]);
            }
            float nx, ny, nz;
            node_normal(sx, sy, sz, sg, nn3[0], nn3[1], nn3[2], nx, ny, nz);
            snx[lt] = nx; sny[lt] = ny; snz[lt] = nz;
        }
        const bool do_com = kStep || mode == M_COM;
        if (do_com && wv == 2) {
            // 256-slot tree of centermass.cu:32-41: slots t and t+128 (180 and above hold 0),
            // t and t+64, then 32..1 across the wave
            const int t = lt & 63;
            const bool hi = t + 128 < kNodes;
            const float a = (sx[t] + (hi ? sx[t + 128] : 0.0f)) + (sx[t + 64] + 0.0f);
            const float b = (sy[t] + (hi ? sy[t + 128] : 0.0f)) + (sy[t + 64] + 0.0f);
            const float d = (sz[t] + (hi ? sz[t + 128] : 0.0f)) + (sz[t + 64] + 0.0f);
            const float ra = wave_tree<OpAdd>(a), rb = wave_tree<OpAdd>(b), rd = wave_tree<OpAdd>(d);
            if (t == 0) {
                cm[0] = ra / 180.0f; cm[1] = rb / 180.0f; cm[2] = rd / 180.0f;
                const CPool q = pool_late();
                q->CMX[slot] = cm[0]; q->CMY[slot] = cm[1]; q->CMZ[slot] = cm[2];
            }
        } else if (!do_com && tid == 0) {
            const CPool q = pool_late();
            cm[0] = q->CMX[slot]; cm[1] = q->CMY[slot]; cm[2] = q->CMZ[slot];
        }
        if (fused) {  // this wave's part of the cell's bbox at the end of the step (bounding_boxes, propagatebound.cu:10-141)
            const float b0 = wave_tree<OpMin>(node ? X : INFINITY), b1 = wave_tree<OpMax>(node ? X : -INFINITY);
            const float b2 = wave_tree<OpMin>(node ? Y : INFINITY), b3 = wave_tree<OpMax>(node ? Y : -INFINITY);
            const float b4 = wave_tree<OpMin>(node ? Z : INFINITY), b5 = wave_tree<OpMax>(node ? Z : -INFINITY);
            if ((lt & 63) == 0) {
                float* b = bpart[wv];
                b[0] = b0; b[1] = b1; b[2] = b2; b[3] = b3; b[4] = b4; b[5] = b5;
            }
        }
        __syncthreads();  // normals, owners, accept bits, centre and box parts are in LDS
        if (fused && lt < 6) {
            float b = bpart[0][lt];
            b = (lt & 1) ? fmaxf(b, bpart[1][lt]) : fminf(b, bpart[1][lt]);
            b = (lt & 1) ? fmaxf(b, bpart[2][lt]) : fminf(b, bpart[2][lt]);
            stu(pool_late()->BBOXN + (size_t)slot * 6, ln, b);
        }
        if (do_dis) {
            // ---- friction, propagate.cu:633-653: the pairs' terms, then each node's sum
            const float gext = P->viscotic_damping;
            for (int c0 = 0; c0 < total; c0 += kRound) {
                if (c0 > 0) {
                    __syncthreads();  // the sums of the round before are done
                    fill_owners<kRound>(owner, lt, first, nc, c0);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int e = c0 + h * kSlots;
                        key[h] = e + lt < total ? ldu(cand, (uint32_t)(e + lt)) : 0;
                        m[h] = e < total ? cld(mask + e / 64 + wv) : 0;
                    }
                    load_partners(c0);
                    __syncthreads();
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (acc[h]) {
                        const int j = h * kSlots + lt, o = owner[j];
                        const float nx = snx[o], ny = sny[o], nz = snz[o];
                        const float vx = svx[o] - wx[h], vy = svy[o] - wy[h], vz = svz[o] - wz[h];
                        const float d = vx * nx + vy * ny + vz * nz;
                        term[0][j] = gext * (vx - d * nx);
                        term[1][j] = gext * (vy - d * ny);
                        term[2][j] = gext * (vz - d * nz);
                    }
                }
                __syncthreads();
                const int lo = max(first, c0), hi = min(first + nc, c0 + kRound);
                if (lo < hi) {
                    uint64_t bits = bit_range(okm, lo - c0, hi - lo);
                    while (bits) {
                        const int j = lo - c0 + __ffsll((unsigned long long)bits) - 1;
                        bits &= bits - 1;
                        fx = fx - term[0][j]; fy = fy - term[1][j]; fz = fz - term[2][j];
                    }
                }
            }
        }
        bool far = false;
        if (do_dis && node) {
            const float vix = svx[lt], viy = svy[lt], viz = svz[lt];
            fx = fx - P->gamma_visc * vix;  // drag, propagate.cu:658
            fy = fy - P->gamma_visc * viy;
            fz = fz - P->gamma_visc * viz;
            const CPool q = pool_late();  // pointers read again where used (see pool_late)
            stu(q->FDX + cb, ln, fx); stu(q->FDY + cb, ln, fy); stu(q->FDZ + cb, ln, fz);
            if (fused) {
                // the next step's Integrate moves this node to X + v' dt with v' from the
                // values now in V, F_con and F_dis (bit-identical to k_integrate): search
                // again next step when that is pair_skin/2 or more from the last search
                const float dt = P->dt, m_ = P->mass, rdt = sqrt_cr(dt);
                const bool rnd = P->add_rands != 0;
                const float x = lds_reread(sx, lt), y = lds_reread(sy, lt), z = lds_reread(sz, lt);
                const float qx = x + half_kick(vix, fcX, fx, rnd ? ldu(q->FRX + cb, ln) : 0.f, dt, rdt, m_, MC) * dt - xbX;
                const float qy = y + half_kick(viy, fcY, fy, rnd ? ldu(q->FRY + cb, ln) : 0.f, dt, rdt, m_, MC) * dt - xbY;
                const float qz = z + half_kick(viz, fcZ, fz, rnd ? ldu(q->FRZ + cb, ln) : 0.f, dt, rdt, m_, MC) * dt - xbZ;
                const float h = 0.5f * P->pair_skin;
                far = !(qx * qx + qy * qy + qz * qz <= h * h);
            }
        }
        // a node of this cell leaves the skin next step: the cell is listed for the next
        // (partial) search, up to the list size (by the first wave that finds one; one
        // atomic per such cell); the flag atomic is skipped once it is visibly set
        if (fused && __any(far)) {
            const uint64_t fm = __ballot(far);
            if ((lt & 63) == __ffsll((unsigned long long)fm) - 1 && atomicExch(&moved, 1) == 0) {
                pool_late()->RESET[slot] = 1;
                if (__hip_atomic_load(&M->search_next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
                    atomicOr(&M->search_next, 1);
                if (__hip_atomic_load(&M->n_reset, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <= kMaxPartial) {
                    const int k = atomicAdd(&M->n_reset, 1);
                    if (k < kMaxPartial) pool_late()->RSL[MC->base + k] = c;
                }
            }
        }
        if (clear_bins && (!kStep || MC->need_search)) {
            // the search of this step is done: this cell's share of the system's
            // search-bin counters (those of the current bin grid, which every
            // insertion since the last clear used) is cleared in one coalesced run
            const int64_t nb = min((int64_t)MC->bbudget, (int64_t)MC->bdims[0] * MC->bdims[1] * MC->bdims[2]);
            const int64_t per = (nb + MC->n - 1) / MC->n;
            const int64_t lo = (int64_t)c * per, hi = min(nb, lo + per);
            int32_t* counts = pool_late()->bins + MC->bbase;
            for (int64_t b = lo + tid; b < hi; b += blockDim.x) counts[b] = 0;
            if (kStep && tid == 0) release_partners(pool_late(), slot);
        }
        const int64_t stepno = step_override >= 0 ? step_override : MC->step + 1;
        const bool do_vol = mode == M_VOLUMES || (kStep && stepno <= P->div_time_steps && rgrowth(P, MC->n) > 0.0f);
        if (do_vol) {
            const bool sph = P->check_sphericity != 0;
            // volume.cu:22-26: local coordinates about the (fresh) centre of mass
            const float cx = cm[0], cy = cm[1], cz = cm[2];
            // volume.cu:37-119, lanes 2f and 2f + 1 on face f: its edges 0..2 and 3..5, the
            // sums running through both in edge order
            const int f = lt >> 1, h = lt & 1;
            float vol[3] = {0.f, 0.f, 0.f}, sq[3] = {0.f, 0.f, 0.f};
            if (f < CS3D_FACES) {
                const uint64_t fw = ldu(mesh->face, (uint32_t)f);
                float avX = 0.0f, avY = 0.0f, avZ = 0.0f;
#pragma unroll
                for (int i = 0; i < 6; ++i) {
                    const int n = (int)((fw >> (8 * i)) & 0xffu);
                    if (i < 5 || f >= 12) { avX += sx[n] - cx; avY += sy[n] - cy; avZ += sz[n] - cz; }
                }
                const float fac = f < 12 ? 0.2f : 0.166666667f;
                avX *= fac; avY *= fac; avZ *= fac;
                const uint32_t ew = (uint32_t)(fw >> (24 * h));  // entries 3 h .. 3 h + 3
                float ax, ay, az, bx, by, bz;
                {
                    const int n = (int)(ew & 0xffu);
                    bx = sx[n] - cx; by = sy[n] - cy; bz = sz[n] - cz;
                }
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    ax = bx; ay = by; az = bz;
                    const int n = (int)((ew >> (8 * (i + 1))) & 0xffu);
                    bx = sx[n] - cx; by = sy[n] - cy; bz = sz[n] - cz;
                    const float n1 = (by * avZ - avY * bz) * ax;
                    const float n2 = (bz * avX - avZ * bx) * ay;
                    const float n3 = (bx * avY - avX * by) * az;
                    vol[i] = fabsf(n1 + n2 + n3);
                    if (sph) {
                        const float x1 = ax - avX, y1 = ay - avY, z1 = az - avZ;
                        const float x2 = bx - avX, y2 = by - avY, z2 = bz - avZ;
                        const float xx = y1 * z2 - z1 * y2, yy = z1 * x2 - x1 * z2, zz = x1 * y2 - y1 * x2;
                        sq[i] = sqrt_cr(xx * xx + yy * yy + zz * zz);
                    }
                }
            }
            auto sum3 = [](float v, const float* e) { return ((v + e[0]) + e[1]) + e[2]; };
            auto area3 = [](float a, const float* e) {
#pragma unroll
                for (int i = 0; i < 3; ++i) a = (float)((double)a + 0.5 * (double)e[i]);
                return a;
            };
            const float totvol = sum3(even_lane(sum3(0.f, vol)), vol);  // the odd lane's is the face's
            const float faceArea = area3(even_lane(area3(0.f, sq)), sq);
            // canonical 128-slot tree over the faces (faces >= 92 contribute 0)
            if (h == 1 && f < CS3D_FACES) { red[0][f] = totvol; red[1][f] = faceArea; }
            if (lt < 128 - CS3D_FACES) { red[0][CS3D_FACES + lt] = 0.0f; red[1][CS3D_FACES + lt] = 0.0f; }
            __syncthreads();
            if (wv == 0) {
                const float a = wave_tree<OpAdd>(red[0][lt] + red[0][lt + 64]);
                const float b = wave_tree<OpAdd>(red[1][lt] + red[1][lt + 64]);
                if (lt == 0) {  // volume.cu:129-161
                    const float volume = (float)((double)a / 6.0);
                    pool_late()->VOL[slot] = volume;
                    if (!isfinite(volume)) st |= CS3D_SYS_VOLUME_NONFINITE;
                    int8_t fl = volume > P->division_vol ? 1 : 0;
                    if (sph) {
                        pool_late()->AREA[slot] = b;
                        const float cbr = cbrtf(volume);
                        const float psi = (float)(4.835975862049408 * (double)cbr * (double)cbr / (double)b);
                        if ((double)fabsf(1.0f - psi) > 0.05) fl = 0;
                    }
                    if (P->use_different_stiffnesses && P->recalc_r0 && pool_late()->E[slot] != P->stiffness1) fl = 0;
                    pool_late()->FLAG[slot] = fl;
                }
            }
        }
        if (st) flag(status_word<kStep, R_POST>(M), st);
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------
// Device RANMAR (marsaglia.h:115-144) and plane normals (RandomVector.h:8-78).
// The generator values are multiples of 2^-24 and every operation is exact in
// float, so the device stream equals the host one.
// ------------------------------------------------------------------------------
__device__ float ranmar1(cs3d_ranmar_state* st) {
    float uni = st->u[st->i97] - st->u[st->j97];
    if (uni < 0.0f) uni += 1.0f;
    st->u[st->i97] = uni;
    st->i97--;
    if (st->i97 == 0) st->i97 = 97;
    st->j97--;
    if (st->j97 == 0) st->j97 = 97;
    st->c -= st->cd;
    if (st->c < 0.0f) st->c += st->cm;
    uni -= st->c;
    if (uni < 0.0f) uni += 1.0f;
    return uni;
}

__device__ void random_vector(cs3d_ranmar_state* st, float* n) {
    float x1, x2, s;
    do {
        x1 = ranmar1(st);
        x2 = ranmar1(st);
        x1 = 2.0f * x1 - 1.0f;
        x2 = 2.0f * x2 - 1.0f;
        s = x1 * x1 + x2 * x2;
    } while (s >= 1.0f);
    n[0] = 2.0f * x1 * sqrt_cr(1.0f - x1 * x1 - x2 * x2);
    n[1] = 2.0f * x2 * sqrt_cr(1.0f - x1 * x1 - x2 * x2);
    n[2] = 1.0f - 2.0f * (x1 * x1 + x2 * x2);
}

__device__ void random_vector_basis(cs3d_ranmar_state* st, float* n, const float* basis) {
    const float r = ranmar1(st);
    const float Nv = (float)cos(2 * 3.14159 * (double)r);
    const float Nw = (float)sin(2 * 3.14159 * (double)r);
    float v[3], w[3];
    if (basis[1] != 0) {
        v[0] = 0; v[1] = basis[2]; v[2] = -1 * basis[1];
        w[0] = basis[1]; w[1] = -1 * basis[0]; w[2] = 0;
    } else {
        v[0] = 0; v[1] = 1; v[2] = 0;
        w[0] = basis[2]; w[1] = 0; w[2] = -1 * basis[0];
    }
    float f = (w[0] * v[0] + w[1] * v[1] + w[2] * w[2]) / (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    w[0] = w[0] - f * v[0]; w[1] = w[1] - f * v[1]; w[2] = w[2] - f * v[2];
    f = sqrt_cr(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    v[0] = v[0] / f; v[1] = v[1] / f; v[2] = v[2] / f;
    f = sqrt_cr(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    w[0] = w[0] / f; w[1] = w[1] / f; w[2] = w[2] / f;
    n[0] = Nv * v[0] + Nw * w[0];
    n[1] = Nv * v[1] + Nw * w[1];
    n[2] = Nv * v[2] + Nw * w[2];
}

// ------------------------------------------------------------------------------
// Division phase of one system per workgroup (256 lanes): count_and_get_div
// (GPUbounce.cu:2489-2500) as an ascending compaction of the flags, one RANMAR
// normal per event in event order, cell_division (postscriptinit.cu:185-256)
// with the daughter at index n, PressureReset (PressureKernels.cu:45-65) and
// the daughter stiffness rule (GPUbounce.cu:1254-1260).  In M_STEP it also ends
// the step: step counter, and whether the grid is rebuilt this step.
// ------------------------------------------------------------------------------
// min (even a) / max (odd a) of 12 values over a 256-lane workgroup; the result
// lands in out[0..12) (LDS), visible after the trailing barrier
__device__ __forceinline__ void block_minmax12(float* v, float (*part)[12], float* out) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int a = 0; a < 12; a += 2) {
            v[a] = fminf(v[a], __shfl_xor(v[a], o));
            v[a + 1] = fmaxf(v[a + 1], __shfl_xor(v[a + 1], o));
        }
    }
    if ((tid & 63) == 0)
#pragma unroll
        for (int a = 0; a < 12; ++a) part[tid >> 6][a] = v[a];
    __syncthreads();
    if (tid < 12) {
        float b = part[0][tid];
        const int nw = (int)(blockDim.x >> 6);
        for (int w = 1; w < nw; ++w) b = (tid & 1) ? fmaxf(b, part[w][tid]) : fminf(b, part[w][tid]);
        out[tid] = b;
    }
    __syncthreads();
}

// Division phase of system s by one 256-lane workgroup (every lane calls it; the
// early returns depend on the system only, so the workgroup stays together).  Part of its
// kernel: pool_late reads the kernel's own arguments, which a called function has not.
__device__ __forceinline__ void divide_system(const Pool& p, int s, int32_t mode) {
    __shared__ int32_t wsum[4];
    __shared__ int32_t nev, ncur, stop;
    __shared__ float nrm[3];
    __shared__ int32_t bad;
    __shared__ float redc[3][128];
    __shared__ float mpart[4][12];
    __shared__ float mres[12];
    __shared__ int64_t nclear;
    const int tid = threadIdx.x;
    SysMeta* M = p.meta + s;
    const bool step_mode = mode == M_STEP;
    // the metadata and parameters that a step without divisions needs, read up front
    // in one batch of scalar loads (this kernel writes these fields only after
    // reading them): one memory round trip instead of one per branch
    const CMeta MC = cmeta(M);
    const CParams PC = cparams(p.prm + s);
    const int32_t m_active = MC->active, n0 = MC->n, base = MC->base, cap = MC->cap;
    const int64_t m_step = MC->step, m_horizon = MC->horizon, m_cell_steps = MC->cell_steps;
    uint32_t raised[R_PHASES];
#pragma unroll
    for (int k = 0; k < R_PHASES; ++k) raised[k] = MC->raised[k];
    uint32_t m_status = MC->status;
    const int32_t m_nreset = MC->n_reset, m_search_next = MC->search_next;
    const int64_t div_time = PC->div_time_steps;
    const int32_t m_gint = PC->grid_interval, m_ccom = PC->correct_com;
    const GridConsts m_grid = grid_consts(MC, PC);
    const int64_t m_vbase = MC->vbase;
    // (read here, not behind the branches that use them)
    asm volatile("" ::"s"(m_active), "s"(n0), "s"(base), "s"(cap), "s"(m_step), "s"(m_horizon), "s"(m_status),
                 "s"(m_nreset), "s"(m_search_next), "s"(m_cell_steps));
    asm volatile("" ::"s"(div_time), "s"(m_gint), "s"(m_ccom), "s"(PC->do_pop_model), "s"(PC->growth_rate),
                 "s"(m_grid.DL), "s"(m_grid.ar), "s"(m_grid.skin), "s"(m_grid.vbudget), "s"(m_grid.bbudget), "s"(m_vbase));
    const float m_rgrowth = rgrowth(PC, n0);
    // what the phases of this step found becomes status (a candidate overflow in the
    // contact pass ended the step there: nothing else that was found in it counts)
    uint32_t found = 0;
#pragma unroll
    for (int k = 0; k < R_PHASES; ++k) found |= raised[k];
    if (__builtin_expect(found != 0, 0)) {
        const bool over = raised[R_CON] & CS3D_SYS_CAND_OVERFLOW;
        if (over) {
            found = CS3D_SYS_CAND_OVERFLOW;
            for (int c = 0; c < n0; ++c)
                if (tid < kSlots) take_back_cell(pool_late(), PC->add_rands != 0, base + c, (uint32_t)tid);
        } else if (raised[R_CON]) {  // the contact pass is done, but no k_dis_post followed
            for (int c = tid; c < n0; c += blockDim.x) release_partners(pool_late(), base + c);
        }
        m_status |= found;
        __syncthreads();  // every wave has read them
        if (tid == 0) {
            M->status = m_status;
            for (int k = 0; k < R_PHASES; ++k) M->raised[k] = 0;
        }
    }
    const bool live = m_active && (m_horizon < 0 || m_step < m_horizon) && !(m_status & CS3D_SYS_FATAL_MASK);
    // a stopped system keeps a pending grid adoption: its bboxes are adopted when it
    // resumes or when a caller reads the grid
    if (!m_active || (step_mode && !live)) {
        if (tid == 0 && step_mode) M->shift_pending = 0;
        return;
    }
    const cs3d_params* P = p.prm + s;
    const int64_t stepno = m_step + 1;
    bool growth = true;
    if (step_mode) growth = stepno <= div_time && m_rgrowth > 0.0f;
    if (tid == 0) { nev = 0; ncur = n0; stop = 0; bad = 0; }
    // whether any cell divides: most steps of a growing tissue have no event, and need
    // none of the list's scans and barriers.  The boxes that a rebuild without events
    // needs are loaded beside the flags.
    constexpr int kUnroll = 8;  // boxes per thread and pass of the extent
    float bb[kUnroll][6];
    const int gint = m_gint > 0 ? m_gint : 1;
    const bool due = step_mode && stepno % gint == 0;
    auto load_boxes = [&](int c0, int n) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const float2* b = reinterpret_cast<const float2*>(p.BBOXN + (int64_t)(base + min(c0 + u * 256 + tid, n - 1)) * 6);
            const float2 b0 = b[0], b1 = b[1], b2 = b[2];
            bb[u][0] = b0.x; bb[u][1] = b0.y; bb[u][2] = b1.x; bb[u][3] = b1.y; bb[u][4] = b2.x; bb[u][5] = b2.y;
        }
    };
    if (due && n0 > 0) load_boxes(0, n0);
    bool any = false;
    if (growth) {
        // 16 flags per load between the 16-byte boundaries, the rest one by one
        const int8_t* F = p.FLAG + base;
        const int head = min(n0, (int)(-(uint32_t)base & 15u)), vecs = (n0 - head) >> 4, tail = head + 16 * vecs;
        const uint4* v = reinterpret_cast<const uint4*>(F + head);
        auto one = [](uint32_t w) {  // whether a byte of w is 1 (the zero-byte test on w ^ 0x01010101)
            const uint32_t x = w ^ 0x01010101u;
            return ((x - 0x01010101u) & ~x & 0x80808080u) != 0;
        };
        constexpr int kVec = 4;  // loads in flight per thread (past the end: the last again)
        for (int i = tid; i < vecs; i += kVec * 256) {
            uint4 w[kVec];
#pragma unroll
            for (int u = 0; u < kVec; ++u) w[u] = v[min(i + u * 256, vecs - 1)];
#pragma unroll
            for (int u = 0; u < kVec; ++u) any |= one(w[u].x) | one(w[u].y) | one(w[u].z) | one(w[u].w);
        }
        if (tid < head) any |= F[tid] == 1;
        if (tail + tid < n0) any |= F[tail + tid] == 1;
    }
    any = __syncthreads_or(any);
    if (__builtin_expect(any, 0)) {
        const CPool late = pool_late();  // its dozen pointers are read here only
        // ascending event list in EVL[base .. base + nev), 4096 cells per pass: each
        // thread loads the flags of 16 consecutive cells at once and counts them, a scan
        // of the counts (shuffles within a wave, then the four wave totals) gives the
        // thread's first event, and it lists its events in cell order
        constexpr int kRun = 16;
        int listed = 0;  // events listed by the passes before (the same in every thread)
        for (int c0 = 0; c0 < n0; c0 += kRun * 256) {
            const int cr = c0 + kRun * tid;
            int8_t f[kRun];
#pragma unroll
            for (int j = 0; j < kRun; ++j) f[j] = cr + j < n0 ? late->FLAG[base + cr + j] : (int8_t)0;
            int cnt = 0;
#pragma unroll
            for (int j = 0; j < kRun; ++j) cnt += f[j] == 1 ? 1 : 0;
            const int lane = tid & 63, wave = tid >> 6;
            int inc = cnt;  // inclusive scan within the wave
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int t = __shfl_up(inc, o);
                if (lane >= o) inc += t;
            }
            if (lane == 63) wsum[wave] = inc;
            __syncthreads();
            int e = listed + inc - cnt;
            for (int w = 0; w < wave; ++w) e += wsum[w];
            if (cnt) {
#pragma unroll
                for (int j = 0; j < kRun; ++j)
                    if (f[j] == 1) {
                        late->EVL[base + e++] = cr + j;
                        late->FLAG[base + cr + j] = 0;
                    }
            }
            listed += wsum[0] + wsum[1] + wsum[2] + wsum[3];
            __syncthreads();  // wsum is rewritten by the next pass
        }
        if (tid == 0) nev = listed;
        __syncthreads();
        const int ne = nev;
        const float half = (float)(0.5 * (double)P->repulsion_range);
        for (int e = 0; e < ne; ++e) {
            if (tid == 0) {
                if (P->use_div_plane_basis) random_vector_basis(&M->rng, nrm, P->div_plane_basis);
                else random_vector(&M->rng, nrm);
                const float nn = sqrt_cr(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
                if ((double)fabsf(nn - 1) > 1e-3) bad |= CS3D_SYS_BAD_NORMAL;
                if (ncur >= cap) { bad |= CS3D_SYS_CAPACITY; stop = 1; }
            }
            __syncthreads();
            if (stop) break;
            const int rank = late->EVL[base + e];
            const int d = ncur;
            const int64_t pi = (int64_t)(base + rank) * kSlots + tid;
            const int64_t di = (int64_t)(base + d) * kSlots + tid;
            const float cmx = late->CMX[base + rank], cmy = late->CMY[base + rank], cmz = late->CMZ[base + rank];
            // bboxes of parent and daughter after the split (min/max pairs: parent x, y,
            // z, then daughter x, y, z)
            float bx[12];
#pragma unroll
            for (int a = 0; a < 12; a += 2) { bx[a] = INFINITY; bx[a + 1] = -INFINITY; }
            if (tid < kNodes) {
                const float x0 = late->X[pi], y0 = late->Y[pi], z0 = late->Z[pi];
#pragma unroll
                for (int side = 0; side < 2; ++side) {  // CalcAndUpdateDaughtPos, postscriptinit.cu:148-182
                    const float Nx = side ? -1 * nrm[0] : nrm[0];
                    const float Ny = side ? -1 * nrm[1] : nrm[1];
                    const float Nz = side ? -1 * nrm[2] : nrm[2];
                    float x = x0 - cmx - half * Nx, y = y0 - cmy - half * Ny, z = z0 - cmz - half * Nz;
                    const float pd = x * Nx + y * Ny + z * Nz;
                    if (pd < 0.0f || pd == 0) { x = x - pd * Nx; y = y - pd * Ny; z = z - pd * Nz; }
                    x = x + (cmx + half * Nx); y = y + (cmy + half * Ny); z = z + (cmz + half * Nz);
                    const int64_t o = side ? di : pi;
                    late->X[o] = x; late->Y[o] = y; late->Z[o] = z;
                    bx[6 * side + 0] = x; bx[6 * side + 1] = x;
                    bx[6 * side + 2] = y; bx[6 * side + 3] = y;
                    bx[6 * side + 4] = z; bx[6 * side + 5] = z;
                }
                late->VX[di] = late->VX[pi]; late->VY[di] = late->VY[pi]; late->VZ[di] = late->VZ[pi];
            } else if (tid < kSlots) {
                late->X[di] = 0.f; late->Y[di] = 0.f; late->Z[di] = 0.f;
                late->VX[di] = 0.f; late->VY[di] = 0.f; late->VZ[di] = 0.f;
            }
            if (tid < kSlots) {  // a new cell's forces start at zero (never-written slots in the reference)
                late->FCX[di] = 0.f; late->FCY[di] = 0.f; late->FCZ[di] = 0.f;
                late->FDX[di] = 0.f; late->FDY[di] = 0.f; late->FDZ[di] = 0.f;
            }
            if (step_mode) {
                block_minmax12(bx, mpart, mres);
                if (tid < 12) late->BBOXN[(int64_t)(base + (tid < 6 ? rank : d)) * 6 + tid % 6] = mres[tid];
            }
            if (tid == 0) {
                const int gd = base + d, gp = base + rank;
                late->E[gd] = P->daught_same_stiffness ? late->E[gp] : P->stiffness1;
                late->GS[gd] = late->GS[gp];
                late->CMX[gd] = 0.f; late->CMY[gd] = 0.f; late->CMZ[gd] = 0.f;
                late->P[gp] = P->min_pressure;
                late->P[gd] = P->min_pressure;
                ncur = d + 1;
            }
            __syncthreads();
        }
        if (P->daughter_com_fix) {  // opt-in: centre of mass of parent and daughter from their new nodes
            const int done = ncur - n0;
            for (int e = 0; e < done; ++e) {
                for (int q = 0; q < 2; ++q) {
                    const int cell = q ? n0 + e : late->EVL[base + e];
                    const int64_t o = (int64_t)(base + cell) * kSlots;
                    if (tid < 128) {  // same 256-slot tree as CenterOfMass
                        const bool hi = tid + 128 < kNodes;
                        redc[0][tid] = late->X[o + tid] + (hi ? late->X[o + tid + 128] : 0.0f);
                        redc[1][tid] = late->Y[o + tid] + (hi ? late->Y[o + tid + 128] : 0.0f);
                        redc[2][tid] = late->Z[o + tid] + (hi ? late->Z[o + tid + 128] : 0.0f);
                    }
                    __syncthreads();
                    if (tid < 64) {
                        float a = redc[0][tid] + redc[0][tid + 64];
                        float b = redc[1][tid] + redc[1][tid + 64];
                        float d = redc[2][tid] + redc[2][tid + 64];
#pragma unroll
                        for (int k = 32; k > 0; k >>= 1) {
                            a = a + __shfl_down(a, k);
                            b = b + __shfl_down(b, k);
                            d = d + __shfl_down(d, k);
                        }
                        if (tid == 0) {
                            late->CMX[base + cell] = a / 180.0f;
                            late->CMY[base + cell] = b / 180.0f;
                            late->CMZ[base + cell] = d / 180.0f;
                        }
                    }
                    __syncthreads();
                }
            }
        }
        __syncthreads();
        if (tid == 0) late->seen[s] = ncur;
    }
    const int events = ncur - n0;
    const bool rebuild = step_mode && (events > 0 || due);
    if (rebuild) {
        // grid rebuild from the end-of-step bboxes: minmaxpre/minmaxpost
        // (propagatebound.cu:145-204, 266-323, sentinels +-1e8) and the grid
        // geometry; the per-cell part (bbox adoption, voxel counts) is done by the
        // next step's Integrate
        float e[6];
#pragma unroll
        for (int a = 0; a < 6; a += 2) { e[a] = 1.0E8f; e[a + 1] = -1.0E8f; }
        // the boxes of 8 cells per thread are loaded before any is reduced (min and max
        // are exact in any order)
        for (int c0 = 0; c0 < ncur; c0 += kUnroll * 256) {
            if (__builtin_expect(c0 > 0 || events > 0 || !due, 0)) load_boxes(c0, ncur);
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {  // (past the end: the last cell's box again)
#pragma unroll
                for (int a = 0; a < 6; a += 2) {
                    e[a] = fminf(e[a], bb[u][a]);
                    e[a + 1] = fmaxf(e[a + 1], bb[u][a + 1]);
                }
            }
        }
#pragma unroll
        for (int a = 0; a < 6; a += 2) {
            const float lo = wave_tree<OpMin>(e[a]), hi = wave_tree<OpMax>(e[a + 1]);
            if ((tid & 63) == 0) { mpart[tid >> 6][a] = lo; mpart[tid >> 6][a + 1] = hi; }
        }
        __syncthreads();
        if (tid == 0) {
            float x[6];
#pragma unroll
            for (int a = 0; a < 6; a += 2) {
                x[a] = fminf(fminf(mpart[0][a], mpart[1][a]), fminf(mpart[2][a], mpart[3][a]));
                x[a + 1] = fmaxf(fmaxf(mpart[0][a + 1], mpart[1][a + 1]), fmaxf(mpart[2][a + 1], mpart[3][a + 1]));
            }
            nclear = set_grid_geometry(M, m_grid, x);
        }
        __syncthreads();
        int32_t* counts = pool_late()->vox + m_vbase;
        for (int64_t v = tid; v < nclear; v += blockDim.x) counts[v] = 0;
    }
    const bool shift = step_mode && m_ccom;
    if (__builtin_expect(shift, 0)) {
        // calc_sys_CM (GPUbounce.cu:2504-2520): float sums of the cell centres in
        // cell order (daughters of this step still hold 0), divided by the count;
        // the nodes are shifted by k_com_shift (CorrectCoMMotion, propagate.cu:766-776)
        const CPool q = pool_late();
        float acc = 0.f;  // lanes 0..2: one component each
        for (int c0 = 0; c0 < ncur; c0 += 128) {
            if (tid < 128 && c0 + tid < ncur) {
                redc[0][tid] = q->CMX[base + c0 + tid];
                redc[1][tid] = q->CMY[base + c0 + tid];
                redc[2][tid] = q->CMZ[base + c0 + tid];
            }
            __syncthreads();
            if (tid < 3) {
                // (the reads of 16 centres ahead of their sequential sum)
                const int m = min(128, ncur - c0);
                int k = 0;
                for (; k + 16 <= m; k += 16) {
                    float v[16];
#pragma unroll
                    for (int j = 0; j < 16; ++j) v[j] = redc[tid][k + j];
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc = acc + v[j];
                }
                for (; k < m; ++k) acc = acc + redc[tid][k];
            }
            __syncthreads();
        }
        if (tid < 3) M->sys_cm[tid] = acc / (float)ncur;
    }
    if (tid == 0) {
        M->shift_pending = shift ? 1 : 0;
        if (bad) atomicOr(&M->status, (uint32_t)bad);
        M->n_events = events;
        M->n = ncur;
        if (step_mode) {
            M->rebuild = rebuild ? 1 : 0;
            M->step = stepno;
            M->cell_steps = m_cell_steps + n0;  // the n0 cells that were stepped
            // After divisions, the divided cells and the cells listed by k_dis_post (a
            // node leaves the skin next step) are searched again next step, with the
            // cells near them (partial search).  Without divisions a node leaving the
            // skin means a full search: it resets every search position, so the next one
            // comes many steps later, where partial searches of the cells that cross the
            // skin one after another would search on almost every step.  A full search
            // also when the list is too long, or when CorrectCoMMotion shifts the nodes
            // (their search positions are not shifted).
            // RSL holds one entry per cell slot of the system (M->cap entries at
            // RSL[base]): a list that would not fit there means a full search
            int nr = m_nreset;
            const int lim = min(kMaxPartial, cap);
            bool full = (events == 0 && m_search_next) || nr > lim || nr + 2 * events > lim ||
                        (shift && (events > 0 || m_search_next));
            if (!full && events > 0) {
                const CPool q = pool_late();
                for (int e = 0; e < events; ++e) {
                    const int pc = q->EVL[base + e], dc = n0 + e;
                    q->RSL[base + nr++] = pc;
                    q->RSL[base + nr++] = dc;
                    q->RESET[base + pc] = 1;
                    q->RESET[base + dc] = 1;
                }
            }
            M->need_search = full ? 1 : (nr > 0 ? 2 : 0);
            M->n_part = full ? 0 : nr;
            M->search_next = 0;
        } else if (events > 0) {
            M->need_search = 1;
        }
    }
    __syncthreads();  // the shared state is reused by the workgroup's next system
}

// One workgroup per system, striding over the systems of the range in use.
__global__ __launch_bounds__(256) void k_sys_divide(Pool p, Range r, int32_t mode) {
    const int hi = r.one_sys ? r.sys_hi : min(r.sys_hi, *p.nsys);
    for (int s = r.sys_lo + blockIdx.x; s < hi; s += gridDim.x) divide_system(p, s, mode);
}

// Lists of the cells of a multi-system step, made at its start: LIVE, the live cells
// (c < n) of the systems that step, and SRCH, those of them whose system searches
// this step; n_live holds both counts.  The step's cell kernels walk them instead of
// every slot of each system's room; each entry is {slot, system}.  Every workgroup
// scans the counts of all systems in use, 1024 at a time, then finds the system of
// each of its entries by bisection of the offsets in LDS, so the lists' 20,000
// entries are written side by side (one system after another per workgroup took
// 36.9 us for 256 systems; the search over all live cells 38 us where none
// searched).
constexpr int kLiveThreads = 1024;

__global__ __launch_bounds__(kLiveThreads) void k_live(Pool p, Range r) {
    __shared__ int2 wsum[kLiveThreads / 64];
    __shared__ int32_t offl[kLiveThreads + 1], offs[kLiveThreads + 1], base[kLiveThreads];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int lo = r.sys_lo, hi = min(r.sys_hi, *p.nsys);
    int2 carry{0, 0};
    for (int c0 = lo; c0 < hi; c0 += kLiveThreads) {
        const int s = c0 + tid;
        int2 n{0, 0};
        if (s < hi) {
            const SysMeta* M = p.meta + s;
            const int live = sys_live(M) ? M->n : 0;
            n = int2{live, M->need_search ? live : 0};
            base[tid] = M->base;
        }
        // inclusive scan within the wave, then over the wave totals
        int2 v = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int tx = __shfl_up(v.x, o), ty = __shfl_up(v.y, o);
            if (lane >= o) { v.x += tx; v.y += ty; }
        }
        if (lane == 63) wsum[wv] = v;
        __syncthreads();
        int2 before = carry;
        for (int w = 0; w < kLiveThreads / 64; ++w) {
            const int2 t = wsum[w];
            if (w < wv) { before.x += t.x; before.y += t.y; }
            carry.x += t.x;
            carry.y += t.y;
        }
        offl[tid] = before.x + v.x - n.x;  // the system's first entry
        offs[tid] = before.y + v.y - n.y;
        if (tid == 0) { offl[kLiveThreads] = carry.x; offs[kLiveThreads] = carry.y; }
        __syncthreads();
        auto write = [&](const int32_t* off, int2* list) {
            const int end = off[kLiveThreads];
            for (int e = off[0] + blockIdx.x * kLiveThreads + tid; e < end; e += gridDim.x * kLiveThreads) {
                int k = 0;  // the last system whose first entry is at or before e
#pragma unroll
                for (int step = kLiveThreads / 2; step > 0; step >>= 1)
                    if (off[k + step] <= e) k += step;
                list[e] = int2{base[k] + e - off[k], c0 + k};
            }
        };
        write(offl, p.LIVE);
        write(offs, p.SRCH);
        __syncthreads();
    }
    if (blockIdx.x == 0 && tid < 2) p.n_live[tid] = tid == 0 ? carry.x : carry.y;
}

// n zero words from q, by the lanes t0, t0 + nt, ..: 16 bytes per store between the
// 16-byte boundaries
__device__ __forceinline__ void zero_words(void* q, int64_t n, int64_t t0, int64_t nt) {
    uint32_t* w = static_cast<uint32_t*>(q);
    const int64_t head = min(n, (int64_t)((16 - (reinterpret_cast<uintptr_t>(q) & 15)) & 15) / 4), vecs = (n - head) / 4;
    for (int64_t i = t0; i < vecs; i += nt) reinterpret_cast<uint4*>(w + head)[i] = make_uint4(0, 0, 0, 0);
    for (int64_t i = t0; i < head; i += nt) w[i] = 0;
    for (int64_t i = head + 4 * vecs + t0; i < n; i += nt) w[i] = 0;
}

// A system enters its room: cleared node, cell, voxel and bin-count arrays, the
// cells' start values, the slots' owner, parameters and metadata, in one launch
// (33 memsets and copies took 0.15 ms of a 0.3 ms cs3d_system_add).
__global__ __launch_bounds__(256) void k_room_init(Pool p, RoomInit a) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, nt = (int64_t)gridDim.x * blockDim.x;
    const SysMeta& m = a.meta;
    const int64_t base = m.base, cap = m.cap, nb = base * kSlots, nn = cap * kSlots;
    void* node[] = {p.X + nb,   p.Y + nb,   p.Z + nb,   p.VX + nb,  p.VY + nb,    p.VZ + nb,   p.VAX + nb,
                    p.VAY + nb, p.VAZ + nb, p.FCX + nb, p.FCY + nb, p.FCZ + nb,   p.FDX + nb,  p.FDY + nb,
                    p.FDZ + nb, p.FRX + nb, p.FRY + nb, p.FRZ + nb, p.NPAIR + nb, p.NCAND + nb};
    for (void* q : node) zero_words(q, nn, t0, nt);
    zero_words(p.BBOX + base * 6, cap * 6, t0, nt);
    zero_words(p.BBOXN + base * 6, cap * 6, t0, nt);
    zero_words(p.vox + m.vbase, (int64_t)m.vbudget * (1 + m.vcap), t0, nt);
    zero_words(p.bins + m.bbase, m.bbudget, t0, nt);
    for (int64_t i = base + t0; i < base + cap; i += nt) {
        p.CMX[i] = 0.f; p.CMY[i] = 0.f; p.CMZ[i] = 0.f;
        p.VOL[i] = 0.f; p.AREA[i] = 0.f;
        p.FLAG[i] = 0;
        p.P[i] = a.prm.min_pressure;
        p.E[i] = a.prm.stiffness1;
        p.GS[i] = 1.0f;
        p.slot_sys[i] = a.sys;
    }
    if (t0 == 0) {
        p.meta[a.sys] = m;
        p.prm[a.sys] = a.prm;
        *p.nsys = a.nsys;
    }
}

// A system leaves its room: no owner, no metadata.
__global__ __launch_bounds__(256) void k_room_free(Pool p, int32_t base, int32_t cap, int32_t sys, int32_t nsys) {
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    for (int i = t0; i < cap; i += nt) p.slot_sys[base + i] = -1;
    if (blockIdx.x == 0) zero_words(p.meta + sys, sizeof(SysMeta) / 4, threadIdx.x, blockDim.x);
    if (t0 == 0) *p.nsys = nsys;
}

// CorrectCoMMotion (propagate.cu:766-776) for the systems whose division phase
// just computed the system centre: every node of every cell minus sys_cm.  The
// reference's kernel also shifts the 12 padding slots of each cell; they are no
// mesh nodes and stay 0 here.  The bboxes and cell centres of the step are left
// as they are, as in the reference (they were computed before the shift).
__global__ __launch_bounds__(192) void k_com_shift(Pool p, Range r) {
    const int tid = threadIdx.x;
    if (tid >= kNodes) return;
    for (int slot = r.slot_lo + xcd_block(); slot < r.slot_hi; slot += gridDim.x) {
        const int s = sys_of(p, r, slot);
        if (s < 0) continue;
        const SysMeta* M = p.meta + s;
        if (!M->shift_pending || slot - M->base >= M->n) {
            if (r.one_sys) break;
            continue;
        }
        const int64_t gi = (int64_t)slot * kSlots + tid;
        p.X[gi] = p.X[gi] - M->sys_cm[0];
        p.Y[gi] = p.Y[gi] - M->sys_cm[1];
        p.Z[gi] = p.Z[gi] - M->sys_cm[2];
    }
}

// ------------------------------------------------------------------------------
// Grid rebuild: bounding_boxes (propagatebound.cu:10-141), minmaxpre/minmaxpost
// (:145-204, 266-323) as order-free min/max (one atomic per workgroup and
// system), host Xdiv/Ydiv/Zdiv (GPUbounce.cu:1331-1334) and the search-bin
// geometry on the device, makeNNlist (:209-263) with atomic slots and a
// per-voxel sort into ascending order.
// ------------------------------------------------------------------------------
constexpr int kBoxCells = 8;  // cells per workgroup of k_cellbox

__global__ __launch_bounds__(192) void k_cellbox(Pool p, Range r) {
    __shared__ float part[3][6];
    __shared__ int32_t acc[6];
    __shared__ int32_t accsys;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6;
    if (tid == 0) accsys = -1;
    __syncthreads();
    const int first = r.slot_lo + blockIdx.x * kBoxCells;
    for (int q = 0; q < kBoxCells; ++q) {
        const int slot = first + q;
        if (slot >= r.slot_hi) break;
        const int s = sys_of(p, r, slot);
        const SysMeta* M = s >= 0 ? p.meta + s : nullptr;
        const bool use = M && M->rebuild && (slot - M->base) < M->n;
        if (!use) continue;
        const int64_t gi = (int64_t)slot * kSlots + tid;
        const bool node = tid < kNodes;
        float v[6];
        const float x = p.X[gi], y = p.Y[gi], z = p.Z[gi];
        v[0] = node ? x : INFINITY; v[1] = node ? x : -INFINITY;
        v[2] = node ? y : INFINITY; v[3] = node ? y : -INFINITY;
        v[4] = node ? z : INFINITY; v[5] = node ? z : -INFINITY;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
            for (int a = 0; a < 6; a += 2) {
                v[a] = fminf(v[a], __shfl_xor(v[a], o));
                v[a + 1] = fmaxf(v[a + 1], __shfl_xor(v[a + 1], o));
            }
        }
        if (lane == 0)
            for (int a = 0; a < 6; ++a) part[wv][a] = v[a];
        __syncthreads();
        if (tid < 6) {
            float b = part[0][tid];
            b = (tid & 1) ? fmaxf(b, part[1][tid]) : fminf(b, part[1][tid]);
            b = (tid & 1) ? fmaxf(b, part[2][tid]) : fminf(b, part[2][tid]);
            p.BBOX[(int64_t)slot * 6 + tid] = b;
            if (accsys != s) {  // flush the previous system's partial extent
                if (accsys >= 0) {
                    SysMeta* A = p.meta + accsys;
                    if (tid & 1) atomicMax(&A->ext[tid], acc[tid]);
                    else atomicMin(&A->ext[tid], acc[tid]);
                }
                acc[tid] = f2o(b);
            } else {
                acc[tid] = (tid & 1) ? max(acc[tid], f2o(b)) : min(acc[tid], f2o(b));
            }
        }
        __syncthreads();
        if (tid == 0) accsys = s;
        __syncthreads();
    }
    if (tid < 6 && accsys >= 0) {
        SysMeta* A = p.meta + accsys;
        if (tid & 1) atomicMax(&A->ext[tid], acc[tid]);
        else atomicMin(&A->ext[tid], acc[tid]);
    }
}

// blockIdx.y = system, blockIdx.x strides over its voxels (clearing counts)
__global__ __launch_bounds__(256) void k_grid_dims(Pool p, Range r) {
    const int s = r.sys_lo + blockIdx.y;
    if (s >= r.sys_hi) return;
    SysMeta* M = p.meta + s;
    if (!M->rebuild) return;
    const cs3d_params* P = p.prm + s;
    float e[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) e[a] = o2f(M->ext[a]);
    const float DL = P->grid_dl;
    const int xd = (int)((e[1] - e[0]) / DL + 1.0f);
    const int yd = (int)((e[3] - e[2]) / DL + 1.0f);
    const int zd = (int)((e[5] - e[4]) / DL + 1.0f);
    const int64_t nv = (int64_t)xd * yd * zd;
    const bool ok = xd > 0 && yd > 0 && zd > 0 && nv <= M->vbudget;
    const int64_t nclear = ok ? nv : (int64_t)M->vbudget;
    int32_t* counts = p.vox + M->vbase;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nclear; v += (int64_t)gridDim.x * blockDim.x)
        counts[v] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) (void)set_grid_geometry(M, grid_consts(M, P), e);
}

// force = 1: fill the lists of the current grid whatever the rebuild flag says
__global__ void k_insert(Pool p, Range r, int32_t force) {
    for (int slot = r.slot_lo + blockIdx.x * blockDim.x + threadIdx.x; slot < r.slot_hi;
         slot += gridDim.x * blockDim.x) {
        const int s = sys_of(p, r, slot);
        if (s < 0) continue;
        SysMeta* M = p.meta + s;
        if (!force && !M->rebuild) continue;
        const int c = slot - M->base;
        if (c == 0) {  // extent accumulators back to the sentinels of minmaxpre (+-1e8)
#pragma unroll
            for (int a = 0; a < 3; ++a) { M->ext[2 * a] = f2o(1.0E8f); M->ext[2 * a + 1] = f2o(-1.0E8f); }
        }
        if (c >= M->n || (M->status & CS3D_SYS_GRID_TOO_LARGE)) continue;
        const cs3d_params* P = p.prm + s;
        const VoxRange vr = vox_range(p.BBOX + (int64_t)slot * 6, M, P);
        {
            const int w[6] = {vr.sx, vr.ex, vr.sy, vr.ey, vr.sz, vr.ez};
            for (int a = 0; a < 6; ++a) p.VRANGE[(int64_t)slot * 6 + a] = w[a];
        }
        const int xd = M->dims[0], yd = M->dims[1];
        int32_t* counts = p.vox + M->vbase;
        int32_t* lists = p.vox + M->lbase;
        const int cap = M->vcap;
        bool over = false;
        for (int j1 = vr.sx; j1 <= vr.ex; ++j1)
            for (int j2 = vr.sy; j2 <= vr.ey; ++j2)
                for (int j3 = vr.sz; j3 <= vr.ez; ++j3) {
                    const int v = j3 * xd * yd + j2 * xd + j1;
                    const int k = atomicAdd(&counts[v], 1);
                    if (k < cap) lists[(int64_t)v * cap + k] = c;
                    else over = true;
                }
        if (over) atomicOr(&M->status, (uint32_t)CS3D_SYS_VOXEL_OVERFLOW);
    }
}

__global__ __launch_bounds__(256) void k_sort(Pool p, Range r, int32_t force) {
    const int s = r.sys_lo + blockIdx.y;
    if (s >= r.sys_hi) return;
    SysMeta* M = p.meta + s;
    if (!force && !M->rebuild) return;
    if (M->status & CS3D_SYS_GRID_TOO_LARGE) return;
    const int64_t nv = (int64_t)M->dims[0] * M->dims[1] * M->dims[2];
    const int cap = M->vcap;
    const int32_t* counts = p.vox + M->vbase;
    int32_t* lists = p.vox + M->lbase;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (int64_t)gridDim.x * blockDim.x) {
        const int n = min(counts[v], cap);
        int32_t* L = lists + v * cap;
        for (int i = 1; i < n; ++i) {  // insertion sort of one short list
            const int key = L[i];
            int j = i - 1;
            while (j >= 0 && L[j] > key) { L[j + 1] = L[j]; --j; }
            L[j + 1] = key;
        }
    }
}

// Completes a grid whose per-cell part is pending (the fused step leaves it to
// the next step's Integrate): the new bboxes become current.  Then the voxel
// counters of the current grid are cleared so that k_insert can fill the lists.
__global__ __launch_bounds__(192) void k_grid_adopt(Pool p, Range r) {
    for (int slot = r.slot_lo + xcd_block(); slot < r.slot_hi; slot += gridDim.x) {
        const int s = sys_of(p, r, slot);
        if (s < 0) continue;
        const SysMeta* M = p.meta + s;
        if (!M->rebuild || slot - M->base >= M->n) continue;
        if (threadIdx.x < 6) p.BBOX[(int64_t)slot * 6 + threadIdx.x] = p.BBOXN[(int64_t)slot * 6 + threadIdx.x];
        if (!(M->status & CS3D_SYS_GRID_TOO_LARGE))
            store_vrange(p.VRANGE, slot, vox_range(p.BBOXN + (int64_t)slot * 6, M, p.prm + s), threadIdx.x);
    }
}

// The partner lists that callers read (CS3D_F_PAIRS, CS3D_F_PAIRCOUNT): each live
// node's accepted candidates, ascending, k-major per cell, from the candidates and their
// accept bits, or from what a search holds of them (hold_partners) in the lists' own room.
__global__ __launch_bounds__(192) void k_pairs_list(Pool p, Range r) {
    __shared__ int32_t list[kMaskAt];
    __shared__ uint64_t bits[kMaskWords];
    const int tid = threadIdx.x;
    for (int slot = r.slot_lo + blockIdx.x; slot < r.slot_hi; slot += gridDim.x) {
        const int s = sys_of(p, r, slot);
        if (s < 0) continue;
        const SysMeta* M = p.meta + s;
        if (slot - M->base >= M->n) continue;
        const size_t cb = (size_t)slot * kSlots;
        int32_t* cand = p.CAND + cb * kPMax;
        const int held = cand[kHeldAt];
        __syncthreads();  // every lane has read it (and the cell before is done)
        if (held == 2) continue;  // the lists were made of it
        const int32_t* counts = held ? p.NPAIR : p.NCAND;
        const int32_t* from = held ? p.PAIRS + cb * kPMax : cand;
        const int ncf = counts[cb + tid], total = counts[cb + kNodes] >> kCandBits;
        for (int e = tid; e < total; e += kSlots) list[e] = from[e];
        if (tid < kMaskWords) bits[tid] = pair_mask(held ? p.PAIRS : p.CAND, slot)[tid];
        __syncthreads();
        if (tid < kNodes) {
            const int nc = ncf & ((1 << kCandBits) - 1), first = ncf >> kCandBits;
            int np = 0;
            for (int j = first; j < first + nc; ++j)
                if (bits[j >> 6] >> (j & 63) & 1) p.PAIRS[cb * kPMax + np++ * kSlots + tid] = list[j];
            p.NPAIR[cb + tid] = np;
        } else {
            p.NPAIR[cb + tid] = 0;
        }
        if (tid == 0 && held) cand[kHeldAt] = 2;
    }
}

// voxel ranges of the current bboxes (after a caller sets BBOX or the grid)
__global__ void k_vrange(Pool p, Range r) {
    for (int slot = r.slot_lo + blockIdx.x * blockDim.x + threadIdx.x; slot < r.slot_hi;
         slot += gridDim.x * blockDim.x) {
        const int s = sys_of(p, r, slot);
        if (s < 0) continue;
        const SysMeta* M = p.meta + s;
        if (slot - M->base >= M->n || (M->status & CS3D_SYS_GRID_TOO_LARGE)) continue;
        const VoxRange v = vox_range(p.BBOX + (int64_t)slot * 6, M, p.prm + s);
        const int w[6] = {v.sx, v.ex, v.sy, v.ey, v.sz, v.ez};
        for (int a = 0; a < 6; ++a) p.VRANGE[(int64_t)slot * 6 + a] = w[a];
    }
}

__global__ __launch_bounds__(256) void k_vox_clear(Pool p, Range r) {
    const int s = r.sys_lo + blockIdx.y;
    if (s >= r.sys_hi) return;
    const SysMeta* M = p.meta + s;
    if (M->status & CS3D_SYS_GRID_TOO_LARGE) return;
    const int64_t nv = (int64_t)M->dims[0] * M->dims[1] * M->dims[2];
    int32_t* counts = p.vox + M->vbase;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (int64_t)gridDim.x * blockDim.x)
        counts[v] = 0;
}

// VelocityUpdateA then VelocityUpdateB (propagate.cu:714-736) on V (per-kernel entry point)
// which: 1 = VelocityUpdateA, 2 = VelocityUpdateB, 3 = A then B
__global__ __launch_bounds__(192) void k_velocity_ab(Pool p, Range r, int32_t which) {
    const int tid = threadIdx.x;
    for (int slot = r.slot_lo + xcd_block(); slot < r.slot_hi; slot += gridDim.x) {
        const int s = sys_of(p, r, slot);
        if (s < 0) continue;
        SysMeta* M = p.meta + s;
        if (slot - M->base >= M->n || tid >= kNodes) continue;
        const cs3d_params* P = p.prm + s;
        const int64_t gi = (int64_t)slot * kSlots + tid;
        const float dt = P->dt, m = P->mass, rdt = sqrt_cr(dt);
        float v[3] = {p.VX[gi], p.VY[gi], p.VZ[gi]};
        const float fc[3] = {p.FCX[gi], p.FCY[gi], p.FCZ[gi]};
        const float fd[3] = {p.FDX[gi], p.FDY[gi], p.FDZ[gi]};
        const bool rnd = P->add_rands != 0;  // the stored random force (d_fRanList)
        const float fr[3] = {rnd ? p.FRX[gi] : 0.f, rnd ? p.FRY[gi] : 0.f, rnd ? p.FRZ[gi] : 0.f};
        if (which & 1) {  // VelocityUpdateA (propagate.cu:714-725)
#pragma unroll
            for (int a = 0; a < 3; ++a)
                v[a] = (float)((double)v[a] + kick_a(dt * fc[a] + rdt * fr[a], m, cmeta(M)));
        }
        if (which & 2) {  // VelocityUpdateB (propagate.cu:727-736)
#pragma unroll
            for (int a = 0; a < 3; ++a) v[a] = (float)((double)v[a] + kick_b(fd[a], dt, m, cmeta(M)));
        }
        p.VX[gi] = v[0]; p.VY[gi] = v[1]; p.VZ[gi] = v[2];
    }
}

// minmaxpre + minmaxpost (propagatebound.cu:145-204, 266-323) over the cell boxes
// in BBOX of system r.sys_lo: {minx, maxx, miny, maxy, minz, maxz} from the
// sentinels +-1e8 with fminf / fmaxf, into out[6].  One workgroup.
__global__ __launch_bounds__(256) void k_extent(Pool p, Range r, float* __restrict__ out) {
    __shared__ float red[6][256];
    const int tid = threadIdx.x;
    const SysMeta* M = p.meta + r.sys_lo;
    float e[6] = {1.0E8f, -1.0E8f, 1.0E8f, -1.0E8f, 1.0E8f, -1.0E8f};
    for (int c = tid; c < M->n; c += blockDim.x) {
        const float* b = p.BBOX + (int64_t)(M->base + c) * 6;
#pragma unroll
        for (int a = 0; a < 6; a += 2) {
            e[a] = fminf(e[a], b[a]);
            e[a + 1] = fmaxf(e[a + 1], b[a + 1]);
        }
    }
#pragma unroll
    for (int a = 0; a < 6; ++a) red[a][tid] = e[a];
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if (tid < h) {
#pragma unroll
            for (int a = 0; a < 6; a += 2) {
                red[a][tid] = fminf(red[a][tid], red[a][tid + h]);
                red[a + 1][tid] = fmaxf(red[a + 1][tid], red[a + 1][tid + h]);
            }
        }
        __syncthreads();
    }
    if (tid < 6) out[tid] = red[tid][0];
}

// PressureReset (PressureKernels.cu:45-65): pressure of the listed cells (local
// indices of system r.sys_lo, checked on the host) set to value
__global__ __launch_bounds__(256) void k_pressure_reset(Pool p, Range r, const int32_t* __restrict__ cells,
                                                        int32_t count, float value) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p.P[p.meta[r.sys_lo].base + cells[i]] = value;
}

// plain streaming copy used to calibrate HBM byte counters
// Arithmetic self-checks of the kernels' own functions (for tests): sqrt_cr against
// sqrtf over all 2^32 inputs (count of differing results, NaNs equal), and
// cs3d_acos of n arguments.
__global__ __launch_bounds__(256) void k_check_sqrt(unsigned long long* bad) {
    unsigned long long nb = 0;
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < (1ull << 32);
         u += (uint64_t)gridDim.x * blockDim.x) {
        const float x = __uint_as_float((uint32_t)u);
        const float a = sqrt_cr(x), b = sqrtf(x);
        nb += !(__float_as_uint(a) == __float_as_uint(b) || (isnan(a) && isnan(b)));
    }
    if (nb) atomicAdd(bad, nb);
}
// Each check also counts what shows that it ran and can see a difference: the
// reciprocal check the floats it compared, the quotient checks the pairs where
// the uncorrected product RN(a * y) differs from a / b (about a quarter).
// rcp_rn against 1.0f / b for every float b with quot_ok(b): out[0] differing,
// out[1] compared
__global__ __launch_bounds__(256) void k_check_rcp(unsigned long long* out) {
    unsigned long long nb = 0, nc = 0;
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < (1ull << 32);
         u += (uint64_t)gridDim.x * blockDim.x) {
        const float b = __uint_as_float((uint32_t)u);
        if (quot_ok(b)) {
            nb += __float_as_uint(rcp_rn(b)) != __float_as_uint(1.0f / b);
            ++nc;
        }
    }
    if (nb) atomicAdd(out, nb);
    atomicAdd(out + 1, nc);
}
// quot_rn(a, b, rcp_rn(b)) against a / b: b in [1, 2), one significand per thread
// (the grid is exactly 2^23 threads), a in [1, 2) with the a_count significands
// from a_first (a_first + a_count <= 2^23, checked by the caller), and a = +-0
// with the first chunk; out[0] differing, out[1] the control
__global__ __launch_bounds__(256) void k_check_quot(unsigned long long* out, uint32_t a_first, uint32_t a_count) {
    const uint32_t bs = blockIdx.x * blockDim.x + threadIdx.x;
    const float b = __uint_as_float(0x3f800000u | bs);
    const float y = rcp_rn(b);
    uint32_t nb = 0, nc = 0;
    if (a_first == 0) {  // a = +0 and -0 keep their sign
        const float zp = __uint_as_float(0u), zm = __uint_as_float(0x80000000u);
        nb += __float_as_uint(quot_rn(zp, b, y)) != __float_as_uint(zp / b);
        nb += __float_as_uint(quot_rn(zm, b, y)) != __float_as_uint(zm / b);
    }
    for (uint32_t i = 0; i < a_count; ++i) {
        const float a = __uint_as_float(0x3f800000u | (a_first + i));
        const uint32_t t = __float_as_uint(a / b);
        nb += __float_as_uint(quot_rn(a, b, y)) != t;
        nc += __float_as_uint(a * y) != t;
    }
    if (nb) atomicAdd(out, (unsigned long long)nb);
    atomicAdd(out + 1, (unsigned long long)nc);
}
// the same on n pseudo-random pairs over the whole range quot_ok admits: a of
// either sign, both with exponents in [-40, 39] and random significands
__global__ __launch_bounds__(256) void k_check_quot_scaled(unsigned long long* out, uint64_t seed, uint64_t n) {
    unsigned long long nb = 0, nc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t h = (i + seed) * 0x9E3779B97F4A7C15ull;
        h ^= h >> 31; h *= 0xBF58476D1CE4E5B9ull; h ^= h >> 29; h *= 0x94D049BB133111EBull; h ^= h >> 32;
        const uint32_t ea = (uint32_t)(h % 80), eb = (uint32_t)((h >> 8) % 80);
        const float a = __uint_as_float((uint32_t)((h >> 63) << 31) | ((87u + ea) << 23) | (uint32_t)((h >> 16) & 0x7fffff));
        const float b = __uint_as_float(((87u + eb) << 23) | (uint32_t)((h >> 39) & 0x7fffff));
        const float y = rcp_rn(b);
        const uint32_t t = __float_as_uint(a / b);
        nb += __float_as_uint(quot_rn(a, b, y)) != t;
        nc += __float_as_uint(a * y) != t;
    }
    if (nb) atomicAdd(out, nb);
    atomicAdd(out + 1, nc);
}
__global__ __launch_bounds__(256) void k_acos(const double* __restrict__ x, double* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = cs3d_acos(x[i]);
}

__global__ __launch_bounds__(256) void k_copy_calibrate(const float4* __restrict__ src, float4* __restrict__ dst,
                                                        int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Copies the pieces of a list into dst (pinned host memory): 16 bytes per lane where
// the source allows, the host link's width is reached with 64 workgroups.
__global__ __launch_bounds__(256) void k_gather(GatherList g, uint32_t* __restrict__ dst) {
    const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    for (int k = 0; k < g.n; ++k) {
        const uint32_t* s = g.src[k];
        uint32_t* d = dst + g.dst[k];
        const uint32_t n = g.words[k], n4 = (reinterpret_cast<uintptr_t>(s) & 15) ? 0 : n / 4;
        for (uint32_t i = t0; i < n4; i += nt) reinterpret_cast<uint4*>(d)[i] = reinterpret_cast<const uint4*>(s)[i];
        for (uint32_t i = 4 * n4 + t0; i < n; i += nt) d[i] = s[i];
    }
}

// sets the grid-rebuild and candidate-search flags of systems (-1 = unchanged)
__global__ void k_set_flags(Pool p, Range r, int32_t rebuild, int32_t search) {
    const int s = r.sys_lo + blockIdx.x * blockDim.x + threadIdx.x;
    if (s < r.sys_hi && p.meta[s].active) {
        if (rebuild >= 0) p.meta[s].rebuild = rebuild;
        if (search >= 0) {
            p.meta[s].need_search = search;
            p.meta[s].n_reset = 0;
        }
    }
}

// ------------------------------------------------------------------------------
// launchers (called by cs3d_api.hip)
// ------------------------------------------------------------------------------
// Kernel timing for cs3d_step_timed: while kernel_timer is set, every launch
// carries its own start/stop events (hipExtLaunchKernelGGL), so a phase's time is
// the sum of its kernels' durations, without the launch gaps.
thread_local std::vector<std::pair<hipEvent_t, hipEvent_t>>* kernel_timer = nullptr;

template <class F, class... A>
static void launch(F kernel, dim3 grid, dim3 block, hipStream_t st, A... args) {
    if (kernel_timer) {
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
            hipExtLaunchKernelGGL(kernel, grid, block, 0, st, e0, e1, 0, args...);
            kernel_timer->push_back({e0, e1});
            return;
        }
        if (e0) (void)hipEventDestroy(e0);
    }
    hipLaunchKernelGGL(kernel, grid, block, 0, st, args...);
}

// Grid of a step's cell kernel: a workgroup for each live cell that the host knows of
// and a quarter more (cells that divide before it looks again; beyond the grid the
// workgroups stride, up to the system's last live cell), at most 256 CUs x wg_per_cu if
// the caller set that.  One cell per workgroup lets the dispatcher even out the load: at
// 20,000 cells k_con_dis takes 138 us, with 2048 workgroups 160, with 4096 161, with 6144
// 174, with 16,384 209 (k_dis_post 90; 100, 105, 113, 135).  A workgroup without a cell
// still costs its dispatch, 2 to 3 ns, so rooms far larger than their tissue are not
// launched whole.
constexpr int kMinGrid = 256;  // one workgroup per CU: a small tissue's growth needs no wider grid
static int grid_cover(const Range& r) {
    const int64_t slots = r.slot_hi - r.slot_lo, n = (int64_t)r.live_hint + r.live_hint / 4 + 8;
    return (int)std::min(slots, std::max<int64_t>(n, kMinGrid));
}
static int grid_step(const Range& r, int per_cu) {
    const int n = grid_cover(r);
    const int64_t cap = per_cu > 0 ? 256 * (int64_t)per_cu : n;
    return (int)(n < 1 ? 1 : (n < cap ? n : cap));
}
// Live cells up to which a step launches no wider grid than now: without bound where
// the room or the caller's cap already ends it.
int32_t cells_covered(const Pool& p, const Range& r) {
    const int n = grid_cover(r);
    const bool widest = n >= r.slot_hi - r.slot_lo || (p.wg_per_cu > 0 && n >= 256 * (int64_t)p.wg_per_cu);
    return widest ? std::numeric_limits<int32_t>::max() : n;
}
// Grid of the other cell kernels: one workgroup per slot up to 4096, then they stride.
static int grid_cells(const Range& r, int per_cu) {
    const int n = r.slot_hi - r.slot_lo;
    const int cap = 256 * (per_cu > 0 ? per_cu : 16);
    return n < 1 ? 1 : (n < cap ? n : cap);
}
// k_search in a multi-system step: few cells search, and which is not known here; the
// 1280 workgroups that fit the chip (31 KB of LDS each) take 45 us of a step of 256
// tissues, 4096 take 90, 20,480 110
constexpr int kSearchLive = 1280;

constexpr int kSysBlocks = 256;  // workgroups of the division phase over several systems
constexpr int kLiveBlocks = 32;  // workgroups of k_live: 32,768 entries side by side

void launch_live(const Pool& p, const Range& r, hipStream_t st) {
    launch(k_live, dim3(kLiveBlocks), dim3(kLiveThreads), st, p, r);
}
void launch_room_init(const Pool& p, const RoomInit& a, hipStream_t st) {
    // a workgroup per cell slot up to four per CU (the nodes of a slot are 15 KB)
    const int b = a.meta.cap < 64 ? 64 : (a.meta.cap < 1024 ? a.meta.cap : 1024);
    launch(k_room_init, dim3(b), dim3(256), st, p, a);
}
void launch_room_free(const Pool& p, int base, int cap, int sys, int nsys, hipStream_t st) {
    const int b = (cap + 255) / 256;
    launch(k_room_free, dim3(b < 1 ? 1 : (b < 64 ? b : 64)), dim3(256), st, p, base, cap, sys, nsys);
}

void launch_integrate(const Pool& p, const Range& r, int flags, int64_t step_override, hipStream_t st) {
    const dim3 grid(grid_step(r, p.wg_per_cu)), block(192);
    if (flags != kStepFlags) launch(k_integrate<0, false>, grid, block, st, p, r, flags, step_override);  // one system
    else if (r.live) launch(k_integrate<1, true>, grid, block, st, p, r, flags, step_override);
    else launch(k_integrate<0, true>, grid, block, st, p, r, flags, step_override);
}
// Whether a step's search runs at the head of k_con_dis (a cell's search needs the bins
// of k_integrate and nothing of another cell's search) instead of in a launch of its
// own, which on the many steps that search nothing costs as much as a small kernel.
// The search's LDS leaves room for 5 workgroups per CU instead of 8, so only where the
// grid fits the chip at that: a step of 1 cell 18.4 instead of 19.5 us, of 8 cells 22.9
// instead of 23.7, of 403 28.2 instead of 28.7, of 1000 33.1 instead of 34.0; with 2000
// cells k_con_dis would take two rounds instead of one.
static bool search_in_con(const Pool& p, const Range& r) { return grid_step(r, p.wg_per_cu) <= kSearchLive; }

void launch_search(const Pool& p, const Range& r, int always, hipStream_t st) {
    if (!always && search_in_con(p, r)) return;
    const int g = grid_step(r, p.wg_per_cu);
    if (r.live)
        launch(k_search<1>, dim3(g < kSearchLive ? g : kSearchLive), dim3(192), st, p, r, always);
    else
        launch(k_search<0>, dim3(g), dim3(192), st, p, r, always);
}
void launch_con(const Pool& p, const Range& r, int mode, hipStream_t st) {
    const dim3 grid(grid_step(r, p.wg_per_cu)), block(192);
    const bool search = search_in_con(p, r);
    auto go = [&](auto kernel) { launch(kernel, grid, block, st, p, r, mode); };
    if (mode != M_STEP) go(k_con_dis<0, false, false>);  // one system
    else if (r.live) search ? go(k_con_dis<1, true, true>) : go(k_con_dis<1, true, false>);
    else search ? go(k_con_dis<0, true, true>) : go(k_con_dis<0, true, false>);
}
// angles: 0 = systems without bending, 1 = with, -1 = both launches
void launch_bonded(const Pool& p, const Range& r, int angles, hipStream_t st) {
    if (angles <= 0) launch(k_bonded<false>, dim3(grid_cells(r, p.wg_per_cu)), dim3(192), st, p, r);
    if (angles != 0) launch(k_bonded<true>, dim3(grid_cells(r, p.wg_per_cu)), dim3(192), st, p, r);
}
void launch_dis(const Pool& p, const Range& r, int mode, int64_t step_override, int clear_bins, bool use_va,
                hipStream_t st) {
    const float* vx = use_va ? p.VAX : p.VX;
    const float* vy = use_va ? p.VAY : p.VY;
    const float* vz = use_va ? p.VAZ : p.VZ;
    const dim3 grid(grid_step(r, p.wg_per_cu)), block(192);
    if (mode != M_STEP)  // one system
        launch(k_dis_post<0, false>, grid, block, st, p, r, mode, step_override, clear_bins, p.X, p.Y, p.Z, vx, vy, vz);
    else if (r.live)
        launch(k_dis_post<1, true>, grid, block, st, p, r, mode, step_override, clear_bins, p.X, p.Y, p.Z, vx, vy, vz);
    else
        launch(k_dis_post<0, true>, grid, block, st, p, r, mode, step_override, clear_bins, p.X, p.Y, p.Z, vx, vy, vz);
}
void launch_divide(const Pool& p, const Range& r, int mode, hipStream_t st) {
    const int ns = r.sys_hi - r.sys_lo;
    launch(k_sys_divide, dim3(ns < 1 ? 1 : (ns < kSysBlocks ? ns : kSysBlocks)), dim3(256), st, p, r, mode);
}
void launch_com_shift(const Pool& p, const Range& r, hipStream_t st) {
    launch(k_com_shift, dim3(r.one_sys ? grid_step(r, p.wg_per_cu) : grid_cells(r, p.wg_per_cu)), dim3(kSlots), st, p, r);
}
void launch_grid(const Pool& p, const Range& r, int vox_blocks, hipStream_t st) {
    const int n = r.slot_hi - r.slot_lo;
    const int cb = (n + 255) / 256;
    const int bb = (n + kBoxCells - 1) / kBoxCells;
    const int ns = r.sys_hi - r.sys_lo;
    launch(k_cellbox, dim3(bb > 0 ? bb : 1), dim3(192), st, p, r);
    launch(k_grid_dims, dim3(vox_blocks, ns > 0 ? ns : 1), dim3(256), st, p, r);
    launch(k_insert, dim3(cb > 0 ? cb : 1), dim3(256), st, p, r, 0);
    launch(k_sort, dim3(vox_blocks, ns > 0 ? ns : 1), dim3(256), st, p, r, 0);
}
void launch_vrange(const Pool& p, const Range& r, hipStream_t st) {
    const int n = r.slot_hi - r.slot_lo;
    launch(k_vrange, dim3(n > 0 ? (n + 255) / 256 : 1), dim3(256), st, p, r);
}
// voxel lists of the current grid (the fused step keeps only the counts)
void launch_vox_lists(const Pool& p, const Range& r, int vox_blocks, hipStream_t st) {
    const int n = r.slot_hi - r.slot_lo;
    const int cb = (n + 255) / 256;
    const int ns = r.sys_hi - r.sys_lo;
    launch(k_grid_adopt, dim3(grid_cells(r, p.wg_per_cu)), dim3(192), st, p, r);
    launch(k_vox_clear, dim3(vox_blocks, ns > 0 ? ns : 1), dim3(256), st, p, r);
    launch(k_insert, dim3(cb > 0 ? cb : 1), dim3(256), st, p, r, 1);
    launch(k_sort, dim3(vox_blocks, ns > 0 ? ns : 1), dim3(256), st, p, r, 1);
}
void launch_pairs_list(const Pool& p, const Range& r, hipStream_t st) {
    launch(k_pairs_list, dim3(grid_cells(r, p.wg_per_cu)), dim3(192), st, p, r);
}
void launch_gather(const GatherList& g, void* dst, hipStream_t st) {
    uint64_t words = 0;
    for (int k = 0; k < g.n; ++k) words += g.words[k];
    const uint64_t b = (words + 1023) / 1024;  // one 16-byte store per thread up to 512 workgroups
    launch(k_gather, dim3(b < 1 ? 1 : (b < 512 ? (uint32_t)b : 512)), dim3(256), st, g, (uint32_t*)dst);
}
void launch_velocity_ab(const Pool& p, const Range& r, int which, hipStream_t st) {
    launch(k_velocity_ab, dim3(grid_cells(r, p.wg_per_cu)), dim3(192), st, p, r, which);
}
void launch_cellbox(const Pool& p, const Range& r, hipStream_t st) {
    const int n = r.slot_hi - r.slot_lo;
    const int bb = (n + kBoxCells - 1) / kBoxCells;
    launch(k_cellbox, dim3(bb > 0 ? bb : 1), dim3(192), st, p, r);
}
void launch_extent(const Pool& p, const Range& r, float* out, hipStream_t st) {
    launch(k_extent, dim3(1), dim3(256), st, p, r, out);
}
void launch_pressure_reset(const Pool& p, const Range& r, const int32_t* cells, int count, float value,
                           hipStream_t st) {
    launch(k_pressure_reset, dim3((count + 255) / 256), dim3(256), st, p, r, cells, count, value);
}
void launch_set_flags(const Pool& p, const Range& r, int rebuild, int search, hipStream_t st) {
    const int ns = r.sys_hi - r.sys_lo;
    launch(k_set_flags, dim3((ns + 255) / 256 > 0 ? (ns + 255) / 256 : 1), dim3(256), st, p, r, rebuild,
                       search);
}
void launch_copy_calibrate(const void* src, void* dst, int64_t n4, hipStream_t st) {
    launch(k_copy_calibrate, dim3(2048), dim3(256), st, (const float4*)src, (float4*)dst, n4);
}
void launch_check_sqrt(unsigned long long* bad, hipStream_t st) {
    launch(k_check_sqrt, dim3(16384), dim3(256), st, bad);
}
void launch_check_div(unsigned long long* bad, uint32_t a_count, uint64_t scaled_pairs, hipStream_t st) {
    launch(k_check_rcp, dim3(16384), dim3(256), st, bad);
    constexpr uint32_t kChunkA = 1024;  // about 5 ms per launch
    for (uint32_t a0 = 0; a0 < a_count; a0 += kChunkA)
        launch(k_check_quot, dim3((1u << 23) / 256), dim3(256), st, bad + 2, a0,
               a_count - a0 < kChunkA ? a_count - a0 : kChunkA);
    if (scaled_pairs > 0) launch(k_check_quot_scaled, dim3(16384), dim3(256), st, bad + 4, (uint64_t)12345, scaled_pairs);
}
void launch_acos(const double* x, double* y, int64_t n, hipStream_t st) {
    launch(k_acos, dim3(n < 1 ? 1 : (n + 255) / 256 < 16384 ? (n + 255) / 256 : 16384), dim3(256), st, x, y, n);
}

}  // namespace cs3d
