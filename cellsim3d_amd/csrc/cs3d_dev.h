// cs3d_dev.h - data layout shared by the HIP kernels and the host side of libcs3d.
//
// HBM layout (one context = one pool on one GPU):
//   node arrays  float[cap_cells * 192]  x, y, z, v, v_after_integrate, F_con, F_dis, F_ran
//                (SoA, 192-slot stride per cell as the reference's d_X, GPUbounce.cu:365-373)
//   cell arrays  float[cap_cells]        CM x/y/z, pressure, stiffness, volume, area, growth scale
//                float[cap_cells * 6]    bbox used by the contact candidate test (rebuilt with the grid)
//                float[cap_cells * 6]    bbox of the positions at the end of the latest step
//                int32[cap_cells * 6]    voxel range of the contact-rule bbox (kept with it)
//   pair lists   int32[cap_cells * kPMax * 192]  contact partners of each node, (cell, node)
//                ascending, k-major per cell, and int32[cap_cells * 192] their count: made
//                from the candidates and their accept bits when a caller reads them (until the
//                contact pass after a search is done, the room holds what that search replaced)
//                int32[cap_cells * kPMax * 192]  contact candidates (within attraction_range + skin
//                at the last search): per cell one flat list, node after node, + per node the
//                count (low kCandBits bits) and the index of its first entry (above them); behind the
//                list one accept bit per entry
//                float[cap_cells * 192] x3  node positions at the last search
//   voxel pool   int32                   per system: counts[budget] then lists[budget * capacity]
//                                        (the reference's 2.9-wide cell grid)
//   bin pool     int32                   per system: counts[bbudget] then entries[bbudget * kBCap]
//                                        float4 (x, y, z, cell*192 + node) (node bins of edge >=
//                                        attraction_range for the pair search)
//   slot table   int32[cap_cells]        system owning each cell slot (-1 = free)
// A system (tissue) owns a contiguous range of cell slots [base, base + cap), a voxel
// region and a bin region; its live cells are base .. base + n - 1 (local 0 .. n - 1).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cs3d.h"
#include "cs3d_read.h"
#include "cs3d_theta.h"

namespace cs3d {

constexpr int kSlots = CS3D_SLOTS;   // 192
constexpr int kNodes = CS3D_NODES;   // 180
constexpr int kFacePad = 128;        // rows of the face table (CS3D_FACES, the rest zero)
constexpr int kPMax = 40;            // contact candidates / partners stored per node
constexpr int kCandBits = 8;         // low bits of an NCAND word that hold the count
static_assert(kPMax < (1 << kCandBits), "a node's candidate count fits its bits");
// The candidate room of a cell (kPMax * kSlots words) holds its flat list (at most
// kPMax * kNodes words) and, behind it, one bit per entry: accepted by the contact
// tests of the latest contact pass (entry j is bit j % 64 of word j / 64).
constexpr int kMaskAt = kPMax * kNodes;
constexpr int kMaskWords = (kMaskAt + kSlots - 1) / kSlots * (kSlots / 64);
// Behind the bits, one word.  0: list and bits belong together.  1: the list has been
// searched anew; the one that the latest contact pass used is held, with its bits at the
// same places, in the cell's room of PAIRS, its counts in NPAIR.  2: the partner lists
// have been made of that.
constexpr int kHeldAt = kMaskAt + 2 * kMaskWords;
static_assert(kMaskAt % 2 == 0 && kHeldAt < kPMax * kSlots, "the mask and the word fit behind the list");
constexpr int kSearchAgain = 2;  // k_search: a search for its own sake, whose list no contact pass uses
constexpr int kBCap = CS3D_BIN_CAP;  // nodes per search bin
constexpr int kMaxSys = 4096;        // systems per context
constexpr int kMaxPartial = 192;     // listed cells beyond which the next search is a full one (at most the
                                     // 192 lanes of a search workgroup, which test one listed cell each)
static_assert(kMaxPartial <= kSlots, "the partial search tests one listed cell per lane");

// Per-system state kept on the device.
struct SysMeta {
    int32_t n;          // live cells
    int32_t cap;        // cell slots owned
    int32_t base;       // first cell slot
    int32_t active;     // 1 = stepped by cs3d_step
    int64_t step;       // completed steps
    int64_t horizon;    // stop after this many steps (-1 = none)
    uint32_t status;    // CS3D_SYS_* bits (sticky); a fused step changes it in its division phase only
    uint32_t raised[4];  // status bits found by each phase of the current fused step (R_*): a phase stops for
                        // what the phases before it found, so that it runs for all cells of a system or none;
                        // merged into status, and zero again, by the division phase
    int32_t rebuild;    // fused step: 1 = the grid was rebuilt at the end of the last step and its
                        // per-cell part (bbox adoption, voxel counts) is still to be done by the
                        // next step; explicit grid kernels: 1 = rebuild now
    int64_t vbase;      // offset of counts[] in the voxel pool
    int64_t lbase;      // offset of lists[] in the voxel pool
    int32_t vbudget;    // voxels available
    int32_t vcap;       // entries per voxel list
    float gmin[3];      // voxel grid origin (minx, miny, minz)
    int32_t dims[3];    // Xdiv, Ydiv, Zdiv
    int32_t ext[6];     // extent accumulators (order-preserving int encoding)
    int32_t n_events;   // divisions in the last division phase
    int32_t bbudget;    // search bins available
    int64_t bbase;      // offset of bin counts in the bin pool
    int64_t ebase;      // offset of bin entries in the bin pool
    float bmin[3];      // bin grid origin
    float bh;           // bin edge
    int32_t bdims[3];   // bins per axis
    int32_t need_search;  // search contact candidates this step: 0 no, 1 every cell, 2 only the
                          // cells near the cells listed in RSL (partial search)
    int32_t search_next;  // set during a step when the next step's drift takes a node pair_skin/2 away
    int32_t n_reset;      // cells that this step has listed in RSL so far (a node leaves the skin);
                          // counts past kMaxPartial mean a full search
    int32_t n_part;       // cells in RSL for the partial search of need_search 2 (at most kMaxPartial)
    float sys_cm[3];      // system centre subtracted at the end of the latest step (correct_com)
    int32_t shift_pending;  // 1 = the step that just ended computed sys_cm and its nodes are still to be
                            // shifted (set by the division phase, consumed by the shift kernel)
    int64_t cell_steps;   // sum over the completed steps of the cells stepped (node-updates / 180)
    // the velocity kicks' double divisions by the particle mass as products with
    // double-double constants, verified for every float significand (kick_consts):
    // kick_a* = 1 / (2 m) for 0.5 * s / m, kick_b* = dt / (2 m) for 0.5 * dt * f / m
    double kick_ah, kick_al, kick_bh, kick_bl;
    int32_t kick_fast;    // 1: the constants above reproduce the divisions exactly
    cs3d_ranmar_state rng;
};

// The phases of a fused step that find status bits (SysMeta::raised), in their order;
// as a count: the phases that have ended when that one runs.
enum { R_INTEGRATE = 0, R_SEARCH = 1, R_CON = 2, R_POST = 3, R_PHASES = 4 };
static_assert(R_PHASES == sizeof(SysMeta::raised) / sizeof(uint32_t), "a word per phase");

// Fills the kick constants of a system with particle mass m and time step dt and
// checks them exhaustively (on the host; results are cached per (m, dt)).
void kick_consts(float m, float dt, SysMeta& M);

// Mesh tables of a node in three 16-byte records and one of 8 bytes, so that a lane
// gets its whole topology and rest state from four loads that depend on nothing but
// the kernel arguments and are issued with the cell's own node data.
struct alignas(16) MeshRec {
    float f[3];
    uint32_t w;
};
struct MeshDev {
    MeshRec th[kSlots];   // rest angles; w: the three neighbours, 8 bits each
    MeshRec r0[kSlots];   // rest lengths; w: angle gather offsets 0, 1 (16 bits each)
    MeshRec ir0[kSlots];  // RN(1/R0) where quot_ok(R0), NaN elsewhere; w: gather offsets 2, 3
    struct alignas(8) {
        uint32_t w;       // gather offsets 4, 5
        float sign;       // orientation of the friction normal (C180NN)
    } gs[kSlots];
    // The angle gather table: for a node, six offsets (in floats) into the per-cell
    // angle-force array, in the summation order of CalculateAngleForce
    // (propagate.cu:124-178).
    // face[f]: the 7 entries of a C180_pentahexa row, 8 bits each
    uint64_t face[kFacePad];
    ThetaCoeffs theta;  // kTheta
};
__host__ __device__ inline int mesh_nn(uint32_t w, int k) { return (int)((w >> (8 * k)) & 0xffu); }

__host__ __device__ inline uint64_t* pair_mask(int32_t* cand, int64_t slot) {
    return reinterpret_cast<uint64_t*>(cand + slot * (kPMax * kSlots) + kMaskAt);
}

struct Pool {
    float *X, *Y, *Z;
    float *VX, *VY, *VZ;     // velocity at end of step
    float *VAX, *VAY, *VAZ;  // velocity after Integrate (read by the first DisForce)
    float *FCX, *FCY, *FCZ;
    float *FDX, *FDY, *FDZ;
    float *FRX, *FRY, *FRZ;  // random force drawn in the latest step (d_fRanList)
    float *CMX, *CMY, *CMZ;
    float *P, *E, *VOL, *AREA, *GS;
    int8_t* FLAG;
    float* BBOX;
    float* BBOXN;
    int32_t* VRANGE;  // makeNNlist's voxel range of BBOX (sx, ex, sy, ey, sz, ez) per cell
    int32_t* PAIRS;
    int32_t* NPAIR;
    int32_t* CAND;
    int32_t* NCAND;
    float *XBX, *XBY, *XBZ;
    float* SBOX;     // float[cap_cells * 6]: box of each cell's search positions (written by full
                     // searches, and by k_integrate for RESET cells before a partial search)
    int8_t* RESET;   // int8[cap_cells]: 1 = the cell takes its current positions as search positions at
                     // the next partial search (a node left the skin, or the cell divided)
    float* KEEP;     // float[cap_cells * 9 * 192]: V, F_con and F_ran before the contact pass of a step that
                     // searches at its head (put back if the search overflows)
    int32_t* RSL;    // int32[cap_cells]: per system, the local indices of its RESET cells (n_reset)
    int2* LIVE;      // {slot, system}[cap_cells]: live cells of the stepped systems (k_live)
    int2* SRCH;      // {slot, system}[cap_cells]: those of them whose system searches in this step
    int32_t* n_live; // int32[2]: entries of LIVE and SRCH
    int32_t* seen;   // int32[kMaxSys], pinned host memory: live cells of each system, written by the
                     // division phase of a step with divisions; the host sizes grids by it
    int32_t* EVL;
    int32_t* slot_sys;
    int32_t* nsys;   // int32[1]: system ids in use are below this (kernels over all systems read it, so a
                     // captured all-systems step stays valid when systems are added or removed)
    SysMeta* meta;
    cs3d_params* prm;
    int32_t* vox;
    int32_t* bins;
    const MeshDev* mesh;
    int32_t wg_per_cu;  // host side: the caller's cap of the grid of the cell kernels, workgroups per CU (0: none)
};

// What a launch works on: cell slots [slot_lo, slot_hi) and systems [sys_lo, sys_hi).
struct Range {
    int32_t slot_lo, slot_hi;
    int32_t sys_lo, sys_hi;
    int32_t one_sys;  // 1: the range is exactly the slot range of system sys_lo
    int32_t live;     // 1: the cell kernels walk Pool::LIVE (built by k_live) instead of the slots
    int32_t live_hint;  // host side: live cells as far as the host knows (sizes grids, nothing else)
};

// A system entering its room (k_room_init): its metadata (room, voxel and bin
// regions, geometry), parameters, id, and the count of system ids in use.
struct RoomInit {
    SysMeta meta;
    cs3d_params prm;
    int32_t sys, nsys;
};

// kernel modes
enum : int32_t {
    M_STEP = 0,        // fused step path (state flags decided on the device)
    M_CON = 1,         // CalculateConForce only -> FC
    M_DIS_V = 3,       // CalculateDisForce with V -> FD
    M_DIS_VA = 4,      // CalculateDisForce with VA -> FD
    M_COM = 5,         // CenterOfMass only
    M_VOLUMES = 6,     // volumes only (explicit step)
    M_INIT = 7,        // start-up: forces from the injected state
    M_PAIRS = 8,       // contact-partner lists only (for a following CalculateDisForce)
};

// k_integrate flags
enum : int32_t {
    I_KICK = 1,       // Integrate + ForwardTime
    I_PRESSURE = 2,   // PressureUpdate
    I_BINS = 4,       // insert the nodes into the search bins
    I_CLEAR = 8,      // clear the search-bin counters of the nodes
    I_IFSEARCH = 32,  // I_BINS only on systems that search this step
    I_GRIDCOUNT = 64, // systems whose grid was rebuilt at the end of the last step: adopt the new
                      // bboxes and count the voxel occupancy (overflow check)
    I_WRITEV = 128,   // with I_KICK: also store the new velocity in V (standalone Integrate)
};

}  // namespace cs3d
