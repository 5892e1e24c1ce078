// Stepping kernels of the nonlocal LBM on CDNA4 (gfx950).
//
// State layout in HBM: the deviations g_alpha = f_alpha - w_alpha of a node's
// Q distributions lie in one row (AoS), rows ordered [bulk | layer |
// boundary].  D3Q27 rows are padded to 32 floats (one 128-byte line).  D2Q9
// rows hold the eight moving distributions (32 bytes, four to a line, two
// 16-byte pieces); the N rest values, which streaming never moves, follow the
// rows (row_at).  The divergence stencil of fluid
// node i is a slab of k records {neighbour index, W_x, W_y(, W_z)}.
//
// Kernels that gather neighbours map one node to LPN consecutive lanes with
// lane = alpha ("lane over alpha"): the Q lanes of a node read one
// contiguous row of each neighbour, so every gather is one cache line, and
// the stencil sum over s runs sequentially inside the lane (no cross-lane
// reduction).  Kernels doing per-node algebra (macroscopic values, the FP64
// collision, the PML recurrences) map one node to one thread.
//
// One time step is twelve launches:
//   p1      macroscopic values, FP64 collision                (all nodes)
//   pl      PML local terms + partial layer sums              (nodes whose Q is used)
//   pm      layer means of the two PML auxiliary values       (2Q columns)
//   pf      PML auxiliary field rows                          (layer rows)
//   p2      PML divergence of the auxiliary fields            (nodes with layer neighbours)
//   p3      boundary interpolation of the post-PML state      (boundary;
//           the sources are read before their collision increment, which
//           p1 keeps aside for them, as the reference interpolates before
//           colliding)
//   p4      selective filter + bounce-back                    (all nodes)
//   s1..s4  the four RK4 stages of the streaming equation     (fluid nodes)
//   p5      boundary interpolation of the new state           (boundary)
#pragma once

#include "collision.hpp"
#include "naga_common.hpp"

namespace naga_amd {

// Offset of distribution a of node i in a row buffer of N nodes, and the
// distance between the a-values of consecutive nodes.
template <int Q>
NAGA_HD constexpr int64_t row_at(int64_t i, int a, int64_t N) {
    return Q == 27 ? i * Lattice<27>::RS + a : a == 0 ? 8 * N + i : 8 * i + a - 1;
}
template <int Q>
NAGA_HD constexpr int64_t row_pitch(int a) {
    return Q == 27 ? Lattice<27>::RS : a == 0 ? 1 : 8;
}

struct StepGeom {
    int64_t N;        // all nodes
    int64_t nbulk;    // [0, nbulk) bulk
    int64_t nlayer;   // [nbulk, nfluid) absorbing layer
    int64_t nfluid;   // nbulk + nlayer; [nfluid, N) boundary
    int k;            // divergence stencil width of the records (step_width)
    int kb;           // boundary interpolation stencil width
    int pml64;        // fused D3Q27 collision: PML local terms in FP64, for the stencil
                      // widths whose own kernels formed them so (all but 16, 32 and
                      // 48: none loses precision by sharing the pass).  Against the
                      // FP64 oracle, cubes with 0.3 wide layers after 60 to 100 steps
                      // differ by 1.0 to 3.1e-7 in FP32, 1.0 to 3.1e-7 in FP64 (at most
                      // 1.6 times less); FP32 steps are 1 us (1.5 %) shorter there
    int pml_ref;      // layer field reads Q at (j - nbulk) as the reference
    float dt;         // lattice time step
    float rho0;       // nominal density
    float vel_scale;  // c / c_s
    float filter;     // selective filter strength (0.75)
};

struct StepBuffers {
    float* g;        // [N][RS] current deviation state
    float* A;        // [N][RS] stage ping
    float* B;        // [N][RS] stage pong
    float* acc;      // [N][RS] RK4 stage-3 output (the fourth stage buffer)
    float4* ru;      // [N] unitless (rho - 1, u) from p1
    float* Gf;       // [N][RS] PML auxiliary field (zero outside the layer)
    const int32_t* rq_list;  // nodes whose PML Q values are maintained
    int64_t n_rq;
    float* E;        // [N][4] (rho - 1, u) of the previous step's PML local
                     // terms, from which the previous equilibrium deviation
                     // (PML Q1 - w) is recomputed
    float* Qp;       // [N][RS] previous Q1 value (PML Q2 source)
    float* Q2v;      // [N][RS] current Q2 value
    const float* slab;    // [nfluid][k][1+D] stencil records
    const float* fslab;   // [nfluid][k][2] filter records {idx, weight}
    const float* bslab;   // [nbnd][kb][2] boundary interpolation records
    const float* sigma;   // [nlayer] absorption
    const float* normals; // [nbnd][D] inward normals
    float* coll;     // [N][RS] collision increment of boundary-source nodes
    const uint8_t* bsrc;  // [nfluid] 1 if the node feeds the boundary interpolator
    const int32_t* pml_list;  // fluid nodes with a layer neighbour
    int64_t n_pml;
    const int32_t* ptiles;    // with tile unions: the tiles holding a pml_list node
    int64_t n_ptiles;
    float* rho;      // [N] density (reference semantics, FP32)
    float* u;        // [D][N] velocity
    double* partial; // [2Q][nparts] layer column sums (one column entry per part:
                     // a PML-local block, or a fused collision block)
    float* means;    // layer means: Q1 at [a], Q2 at [means_stride(Q) + a]
    int nparts;
    int part_lo;     // parts [part_lo, nparts) hold the layer sums
    const float* src;  // [N] density source of this step (physical units), or null
    // Tile unions (D3Q27 four-per-lane kernels): the fluid nodes form tiles
    // of 64 or 32; ulist[uoff[t] .. uoff[t+1]) are the distinct stencil neighbours
    // of tile t, and the index field of slab / fslab records holds the
    // neighbour's position in that list; slab and fslab rows are then
    // packed (packed_div_units, packed_filter_units).  Unions of at most
    // ucap rows are staged in LDS by the gather kernels.  A tile over the
    // cap with usplit[t] > 0 holds two half-tile unions (lengths usplit[t]
    // and the rest, each at most ucap): its block serves the first half,
    // and one more block per split tile, after the regular ones (tile
    // entries -1 - s in ptiles), serves the second half of split_tiles[s].
    const uint32_t* ulist;
    const int64_t* uoff;
    const int32_t* usplit;
    const int32_t* split_tiles;
    int64_t n_split;
    int ucap;
    int ucap_f;      // LDS union rows of the filter pass (at most ucap: its smaller
                     // records leave room for more blocks per CU)
    // Per-node stencil widths with tile unions: tile t's nodes keep
    // tile_ng[t] groups of 8 records (ragged rows of ragged_div_units /
    // ragged_filter_units(tile_ng[t]) units), its divergence and PML records
    // from unit rec_off[t] of slab / p2slab, its filter records from unit
    // frec_off[t] of fslab.  Null: every tile keeps k records per node.
    const int32_t* tile_ng;
    const int64_t* rec_off;
    const int64_t* frec_off;
    int self_first;  // every fluid node's first stencil entry is the node itself
                     // (its own row is then in its tile's union, record 0);
                     // NAGA_OWN_LDS=0 clears it
    // The same for the PML divergence, whose unions hold the layer
    // neighbours and one row outside the layer (Gf is zero there): its
    // packed records, lists, offsets and split tiles.
    const float* p2slab;
    const uint32_t* p2ulist;
    const int64_t* p2uoff;
    const int32_t* p2usplit;
    const int32_t* p2split_tiles;
    int64_t p2n_split;
    // Boundary interpolation tiles (32 boundary nodes): the distinct source
    // nodes of each tile, bulist[buoff[t] .. buoff[t+1]), and bslab index
    // fields holding positions in that list (null: no boundary unions).
    // Tiles of at most bunion_cap(kb) sources are staged in LDS.
    const uint32_t* bulist;
    const int64_t* buoff;
};

// Batched launches: one launch of a pass covers the scenes of a batch; the
// blocks [bstart[s], bstart[s+1]) of the launch belong to scene s, which
// reads its geometry, buffers and collision parameters from scenes[s].
struct SceneDesc {
    StepGeom G;
    StepBuffers S;
    CollisionParams cp;
};
struct BatchArgs {
    const SceneDesc* scenes;  // null for a single-scene launch
    const int32_t* bstart;    // nscenes + 1 block offsets of this pass
    int nscenes;
};

// Density sources: per step, field[nodes[i]] = sum over entries e in
// [off[i], off[i+1]) of prof[e] * amp[ids[e]] (sources in a fixed order).
constexpr int kMaxSources = 16;
struct SourceAmps {
    float a[kMaxSources];
};
void launch_source_field(const int32_t* nodes, const int32_t* off, const int32_t* ids,
                         const float* prof, int64_t n, const SourceAmps& amps, float* field,
                         hipStream_t stream);

// Launch the kernels of one step on `stream`.  If `events` is not null,
// events[t] is recorded before kernel t and events[kStepKernels] after the
// last (kernels with no work still get their pair of marks).
constexpr int kStepKernels = 12;
// Parts of the layer sums: blocks of the PML-local pass, or, when the
// collision pass carries the PML local terms, its 64-node blocks up to the
// last layer node; parts below pml_part_lo hold no layer node.
int64_t pml_parts(int Q, int k, int64_t N, int64_t nfluid, int64_t n_rq);
int64_t pml_part_lo(int Q, int k, int64_t N, int64_t nbulk);
template <int Q>
void launch_step(const StepGeom& geo, const StepBuffers& buf,
                 const CollisionParams& cp, hipStream_t stream,
                 hipEvent_t* events = nullptr);

// One step of every scene of a batch: kStepKernels batched launches.  The
// host-side table describes the same scenes as the device table (block
// counts and kernel choices are derived from it); bstart holds
// kStepKernels consecutive arrays of nscenes + 1 block offsets (device).
struct BatchPlan {
    int Q = 9;
    int nscenes = 0;
    const SceneDesc* dev_scenes = nullptr;
    const int32_t* dev_bstart = nullptr;
    int64_t blocks[kStepKernels] = {};  // total blocks per pass
    int k_template = 0;                 // K template of the gather kernels (0: dynamic)
    bool unions = false;                // D3Q27 four-per-lane kernels
    int ucap = 0;                       // max LDS union rows over the scenes
    int ucap_f = 0;                     // the same for the filter pass
    int gather_batch = 0;               // neighbours gathered per unrolled step (0: default)
    bool tiles = false;                 // tile unions built for every scene
    int kmax = 0;                       // largest stencil width over the scenes
    int kb = 0;                         // largest boundary stencil width
    bool ragged = false;                // per-tile record widths in every scene
    bool pml64 = false;                 // StepGeom::pml64 of every scene
    bool pair = false;                  // D2Q9: two lanes per node (else one per distribution)
};
// Block counts of each pass for one scene (the same counts launch_step
// uses).  pair: D2Q9 kernels, 1 for two lanes per node, 0 for one lane per
// distribution, -1 for the default (q9_pair).
void step_block_counts(int Q, const StepGeom& G, const StepBuffers& S, int64_t* blocks,
                       int pair = -1);
template <int Q>
void launch_step_batch(const BatchPlan& plan, hipStream_t stream);

// Whether the step runs the D3Q27 four-per-lane kernels, which may use
// the tile unions (StepBuffers::ulist/uoff/ucap) and slabs holding union
// positions: D3Q27, 12 <= k <= 48, fewer than 2^25 nodes.
constexpr int kUnionKMin = 12, kUnionKMax = 48;
bool step_uses_unions(int Q, int k, int64_t N);
// Stencil width of the step's records, which every caller that builds them
// gives them and puts in StepGeom::k: k, or for the four-per-lane kernels
// the next multiple of 8 (at least 16), the added records naming the first
// one's node again with zero weights.  A padded record costs less than the
// one-distribution-per-lane kernels do on all of them (h = 0.02 cube, k = 24:
// 254 us per step against 205 at k = 32); below k = 12 the padding would be a
// third of the records.
int step_width(int Q, int k, int64_t N);
constexpr int union_width(int k) { return k <= 16 ? 16 : (k + 7) / 8 * 8; }
// The width that the kernels are instantiated for, or 0.
constexpr int step_k_template(int k) { return k >= 16 && k <= 48 && k % 8 == 0 ? k : 0; }
constexpr bool union_widths_instantiated() {
    for (int k = kUnionKMin; k <= kUnionKMax; ++k)
        if (union_width(k) < k || step_k_template(union_width(k)) != union_width(k)) return false;
    return true;
}
static_assert(union_widths_instantiated(), "a stencil width pads to one without kernels");
// Whether the D2Q9 stencil passes run two lanes per node by default
// (NAGA_Q9_THREE=0: one lane per distribution), and whether they can (fewer
// than 2^26 nodes: 32-bit buffer offsets of 32-byte rows).
bool q9_pair(int Q, int64_t N);
bool q9_pair_fits(int64_t N);
// Nodes per union tile (= per block of the union kernels) for stencil width
// k: 64 for k <= 32 (5.4 union rows per node against 7.0 with 32-node
// tiles, two blocks per CU; 1.40 against 1.44 ms per step on the 1M-node
// D3Q27 scene), else 32; NAGA_TILE=32 selects 32-node tiles for every k.
int union_tile_nodes(int k);
// Default LDS union rows per block: 400 for 64-node tiles (two blocks per
// CU), 296 for 32-node tiles and k <= 32 (three blocks per CU), 440 for
// k = 48 (two blocks per CU, the records taking 22 KB).  A tile with a
// larger union reads its rows from HBM through the union list.
int union_cap_default(int k);
// Stride of the two rows of layer means (D3Q27: 32, so each row's
// quarters load as 16-byte vectors; padding entries stay zero).
constexpr int means_stride(int Q) { return Q == 27 ? 32 : Q; }
// LDS rows per boundary-interpolation tile: 32-node tiles of a cube's faces
// have 183 sources on average, at most 253, with kb = 32, and about 255 with
// kb = 48 (half of them over 256).
NAGA_HD constexpr int bunion_cap(int kb) { return kb <= 32 ? 256 : 320; }
constexpr int kBTileNodes = 32;   // boundary nodes per boundary-interpolation tile
constexpr int kUnionRowsMax = 512;  // LDS union rows per block, upper bound

// Per-kernel entry points (used by the profiler and the standalone C-ABI).
template <int Q>
void launch_rk4_stage(int stage, const StepGeom& geo, const StepBuffers& buf,
                      hipStream_t stream);

// Density probes (density_observer.cuh:62-113): out[p] = rho0 +
// sum_s w[p][s] (rho(idx[p][s]) - rho0), with rho the held FP32 density
// (held != null) or computed fresh from the deviation rows g of N nodes.
void launch_probe(int Q, int64_t n, int k, const uint32_t* idx, const float* w,
                  const float* held, const float* g, int64_t N, double rho0, double* out,
                  hipStream_t stream);

// A Gaussian density pulse at rest as deviation rows: g_alpha = w_alpha amp
// exp(-|x - center|^2 / (2 width^2)) in FP64, rounded once; pts [N][D].
template <int Q>
void launch_pulse(int64_t N, const float* pts, const double* center, double amp, double width,
                  float* g, hipStream_t stream);

// Two D2Q9 row buffers (row_at) to or from plain rows [N][9], the form of saved
// states: pack copies the row buffers to plain rows, else the reverse.
void launch_plain_rows_q9(int64_t N, const float* src0, const float* src1, float* dst0, float* dst1,
                          bool pack, hipStream_t stream);

// Fresh macroscopic values from the current state: rho (FP32, reference
// units), drho = rho - rho0 in FP64 without cancellation, u (FP32).
template <int Q>
void launch_macroscopic(const StepGeom& geo, const float* g, float* rho,
                        double* drho, float* u, hipStream_t stream);

}  // namespace naga_amd
