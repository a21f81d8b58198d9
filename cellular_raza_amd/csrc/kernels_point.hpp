// kernels_point.hpp -- gfx950 kernels of the per-step mechanics path for point agents.
//
// Step (run_sim.rs:380-403) as launched by the runtime:
//   k_force_tiled      pair loop over the 3^D voxel stencil (update_mechanics.rs:153-238);
//                      further workgroups scan the next order's voxel counts (scan_moves)
//   k_gather_integrate_point  the full mechanics update (solvers.rs:23-347 + apply_boundary,
//                      cartesian_cuboid_n.rs:594-631) written into the agent's slot in the
//                      next order, in which the agents that stay in a voxel keep their
//                      order and the movers are appended by previous slot
//                      (sort_cells_in_voxels, update_mechanics.rs:418-513); the force
//                      records, and the voxel each agent moves to in the step after
//                      (note_move)
//   Brownian agents, whose next position needs the force, get that voxel from
//   k_key_point (cartesian_cuboid_n.rs:469-491) and the scan from k_scan_moves, between the two.
//
// Set-up sorts (initial placement, insertion, removal, the rods' cycle) are a counting
// sort of their own: ranks (k_initial_key, k_rank_ahead), k_scan_local/tiles, k_scatter,
// k_fixup and k_gather_point; systems whose voxels fit one scan tile run k_sort_small, the
// scans and the scatter in one workgroup.
//
// Agents live in SoA arrays sorted by voxel; a voxel's agents are the slots
// [start[v], start[v+1]).
#pragma once

#include "device_math.hpp"

namespace crm {

constexpr int kBlock = 256;
// rank flag of an agent binned ahead that changes voxel (see k_rank_ahead)
constexpr uint32_t kMoved = 0x80000000u;

struct StateBuf {
    double* pos;  // [K][N]
    double* vel;  // [K][N]
    double* hdx;  // [2][K][N] Adams-Bashforth ring, position increments
    double* hdv;  // [2][K][N] velocity increments
    int32_t* species;
    uint32_t* id;   // agent index
    uint32_t* vox;  // global voxel of the slot's agent
    // rods only (null for points): RodMechanics::spring_length per rod, the step
    // of the rod's first history push (0, or the step after its division), and
    // the cycle state of the rods example
    double* spring;   // [N]
    uint32_t* birth;  // [N]
    double* growth;   // [N]
    uint64_t* ident;  // [3][N] CellIdentifier (kind, a, b)
    uint64_t* parent; // [3][N]
};

struct Arrays {
    const InstParams* ip;
    const BlockWork* work;
    Control* ctrl;
    uint32_t* start;  // [Vt + 1]
    uint32_t* start_local;  // [Vt] offset of each voxel inside its scan tile (k_scan_local, scan_moves)
    uint32_t* tile_off;     // [n_tiles + 1] sum of each scan tile (k_scan_local, scan_moves), or its offset (k_scan_tiles)
    // set-up sorts
    uint32_t* count;  // [Vt] arrivals per next voxel (atomic ranks)
    uint32_t* stay;   // [Vt] agents that stay in their voxel (zero unless ranked by k_rank_ahead)
    uint32_t* rank;   // [N] arrival rank inside the next voxel
    uint32_t* perm;   // [N] sorted slot -> previous slot
    // the step's moves (note_move), and those of the following step that the gather notes
    uint32_t* key;    // [N] next voxel
    uint32_t* key_next;
    uint32_t* head;   // [Vt] the voxel's arrivals as a list: slot + 1 of the last noted one, 0 without any
    uint32_t* head_next;
    uint32_t* link;   // [N] (arrivals) slot + 1 of the one noted before it
    uint32_t* link_next;
    int32_t* delta;   // [Vt] arrivals less departures of the voxel
    uint32_t n_scan;      // scan tiles of the step, at most kStepScanTiles
    uint32_t scan_shift;  // of kScanTile << scan_shift voxels
    double* force;    // [K][N]
    float* forcef;    // [K][N] in the same memory: point forces of the mixed path, stored in float
    double4* rec64;   // [N] (x, y, z, species) absolute, FP64 path
    int4* recq;       // [N] (qx, qy, qz, species | outside << 31) fixed point in the voxel, mixed path
    uint32_t* sense;  // [N] (rods: [N][nv]) neighbour counts by slot; null when sensing is off
    double sense_t;   // a pair is sensed when its squared distance is below this
    uint64_t N;
    uint32_t Vt;
};

// Squared norm summed in axis order with every product and sum rounded on its
// own (no fused multiply-add), as nalgebra's norm_squared computes it.
template <int D>
__device__ __forceinline__ double sum_squares_unfused(const double* z) {
#pragma clang fp contract(off)
    double d2 = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) d2 = d2 + z[k] * z[k];
    return d2;
}

__device__ __forceinline__ void raise_error(Control* c, uint32_t kind, uint64_t step, uint64_t agent) {
    atomicOr(&c->error_flags, 1u << kind);
    unsigned long long k = ((unsigned long long)step << 32) | (unsigned long long)(agent & 0xffffffffu);
    atomicMin((unsigned long long*)&c->error_key, k);
}

// An earlier step than t raised an error.  The kernels of the steps after a
// failing one do nothing, so the state stays at the end of the failing step, where
// run_simulation! returns the error (run_sim.rs:380-403).
__device__ __forceinline__ bool halted(const Control* c, uint64_t t) {
    return c->error_flags != 0 && (c->error_key >> 32) < t;
}

template <typename T>
__device__ __forceinline__ const PotParams<T>& pot_of(const InstParams& P);
template <>
__device__ __forceinline__ const PotParams<double>& pot_of<double>(const InstParams& P) { return P.pd; }
template <>
__device__ __forceinline__ const PotParams<float>& pot_of<float>(const InstParams& P) { return P.pf; }

// ---------------------------------------------------------------------------
// Force kernel.  One lane per agent; candidates are the agents of the clipped
// 3^D stencil (get_neighbor_voxel_indices, cartesian_cuboid_n.rs:641-662) plus
// the own voxel.  Weights, for the reference (one subdomain) mode:
//   same voxel:     1/2 f(i<-j by i) + 1/2 f(i<-j by j)   (update_mechanics.rs:186-203)
//   adjacent voxel: 1/2 f(i<-j by i)                        (update_mechanics.rs:90-106, 205-220)
// The physical mode gives adjacent pairs the same-voxel weight.  With a
// symmetric interaction both evaluations are equal and one is computed.
//
// Work unit: a tile of voxels -- plane a0, rows [b0, b1), columns [c0, c1) of
// one instance.  Its stencil region (planes a0-1..a0+1, rows b0-1..b1, columns
// c0-1..c1, clipped to the grid) is staged in LDS, one contiguous segment of
// sorted agents per (plane, row).
//
// Mixed precision: the force records hold 30-bit fixed-point positions relative
// to the agent's voxel origin (q = floor((p - origin) * 2^30 / dx)).  For the
// pair loop they are re-expressed relative to the tile region's origin with
// `bits` bits per voxel, bits = 31 - ceil(log2(region extent in voxels)), so that
// every coordinate and every difference is an exact int32: the displacement of
// two agents is one integer subtraction and one rounding to float.  A pair whose
// float distance lies in a narrow band around the cutoff radius (the forces jump
// there), a pair closer than 2e6 fixed-point steps (where the step would show in
// the direction), or an agent flagged as outside its voxel's fixed-point range,
// is re-evaluated from the FP64 positions, with the reference's cutoff decision.
// ---------------------------------------------------------------------------

// blockIdx -> work block, so that each XCD (blocks are dealt round-robin over 8)
// walks one contiguous slab of agents and its L2 holds that slab's records.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb) {
    const uint32_t per = nb / 8u, rem = nb % 8u;
    const uint32_t x = b % 8u, k = b / 8u;
    return x < rem ? x * (per + 1u) + k : rem * (per + 1u) + (x - rem) * per + k;
}

constexpr int kQBits = 30;
constexpr int kQOne = 1 << kQBits;
// Record word w (mixed): species in bits 0-3, the voxel's column along the last
// axis in bits 4-30, the outside-its-voxel flag in bit 31.
constexpr uint32_t kSpeciesMask = 0xfu;
constexpr int kColShift = 4;
constexpr uint32_t kColMask = 0x7ffffffu;
constexpr uint32_t kFlagBit = 0x80000000u;

template <bool MIXED>
struct RecOf {
    using type = double4;
};
template <>
struct RecOf<true> {
    using type = int4;
};

__device__ __forceinline__ const double4* rec_array(const Arrays& A, std::false_type) { return A.rec64; }
__device__ __forceinline__ const int4* rec_array(const Arrays& A, std::true_type) { return A.recq; }

// A tile's stencil region: rows b0 - 1 .. b1 (RW of them, empty where outside the
// grid), columns [cl, ch) (NC of them) and, in 3-D, planes a0 - 1 .. a0 + 1 (NP = 3;
// NP = 1 in 2-D).
struct Region {
    uint32_t a0, b0;  // tile plane and first row
    uint32_t cl, ch;  // staged columns
    uint32_t RW, NC;  // staged rows (tile rows + 2), staged columns (ch - cl)
    int bits, shift;  // tile fixed point: bits per voxel, 30 - bits
};

// Voxel-relative record -> region-relative fixed point.  oa, ob: the record's
// plane and row offsets from the region origin (a0 - 1, b0 - 1).
template <int D>
__device__ __forceinline__ int4 to_region(const int4 r, int oa, int ob, const Region& G) {
    const int oc = (int)(((uint32_t)r.w >> kColShift) & kColMask) - (int)G.cl;
    const uint32_t w = (uint32_t)r.w & (kSpeciesMask | kFlagBit);
    if constexpr (D == 3)
        return make_int4((oa << G.bits) + (r.x >> G.shift), (ob << G.bits) + (r.y >> G.shift),
                         (oc << G.bits) + (r.z >> G.shift), (int)w);
    else
        return make_int4((ob << G.bits) + (r.x >> G.shift), (oc << G.bits) + (r.y >> G.shift), 0, (int)w);
}

struct Span {
    uint32_t b, e;
};

// Candidate order of an agent at (a, b, c): stencil rows b' ascending, then
// columns c' ascending, then planes a' ascending, then slot -- i.e. the 3^D voxels
// with the row outermost.  Both sources below produce this order.
//
// LDS source: the region is staged voxel by voxel in that same (row, column,
// plane) order, so the candidates of one stencil row (3 columns x all planes)
// are one contiguous LDS range and an agent's stream is three ranges.
struct Walk3 {
    uint32_t j, je;          // current range [., je)
    uint32_t j1, e1, j2, e2; // the ranges after it
    uint32_t left;           // how many of those remain
    // Moves past exhausted ranges, carrying the overshoot; false at the end.
    __device__ __forceinline__ bool settle() {
        while (j >= je) {
            if (left == 0) return false;
            const uint32_t over = j - je;
            j = j1 + over;
            je = e1;
            j1 = j2;
            e1 = e2;
            left--;
        }
        return true;
    }
};

// Staged records in LDS, addressed by the byte offset kBytes * index: int4 (mixed), or
// one array of doubles per axis (FP64; the species are bytes beside them).  The
// capacities keep the occupancy the registers allow: 5 workgroups of at most 32000 bytes
// per CU (mixed; LDS is given out in 1280-byte granules, and 32512 bytes cost the fifth),
// 4 of at most 40960 (FP64).  The FP64 records were double4 (896 of them) and the mixed
// ones 1024: LDS bounded the tiles, whose own agents filled 64 % of the lanes on the
// 4M-agent lattice (now 84 %).
template <int D, bool MIXED>
struct LdsRecords;
template <int D>
struct LdsRecords<D, true> {
    static constexpr int kCap = 1232;
    static constexpr uint32_t kBytes = sizeof(int4);
    static constexpr uint32_t kTotal = kCap * kBytes;
    static __device__ __forceinline__ int4 at(const char* lds, uint32_t off) {
        return *reinterpret_cast<const int4*>(lds + off);
    }
    static __device__ __forceinline__ void put(char* lds, uint32_t j, const int4 r) {
        *reinterpret_cast<int4*>(lds + j * kBytes) = r;
    }
};
template <int D>
struct LdsRecords<D, false> {
    static constexpr int kCap = D == 3 ? 1152 : 1600;  // multiples of 64 (ds_read2st64 pairs two axes)
    static constexpr uint32_t kBytes = sizeof(double);
    static constexpr uint32_t kTotal = kCap * kBytes * D;
    static __device__ __forceinline__ double4 at(const char* lds, uint32_t off) {
        const double* x = reinterpret_cast<const double*>(lds + off);
        return make_double4(x[0], x[kCap], D == 3 ? x[(D - 1) * kCap] : 0.0, 0.0);
    }
    static __device__ __forceinline__ void put(char* lds, uint32_t j, const double4 r) {
        double* x = reinterpret_cast<double*>(lds) + j;
        x[0] = r.x;
        x[kCap] = r.y;
        if constexpr (D == 3) x[2 * kCap] = r.z;
    }
};

template <int D, bool MIXED>
struct LdsSource {
    using Rec = typename RecOf<MIXED>::type;
    using W = Walk3;
    const char* lds;      // staged records, converted (LdsRecords)
    const uint8_t* lsp;   // FP64: species of each staged record
    const uint16_t* vst;  // LDS index of the first agent of staged voxel v; vst[n_vox] = total
    Region G;
    uint32_t np, n_vox;
    const uint32_t* start;
    uint32_t voff, n1, n2;
    const uint16_t* sub;  // chili subdomain of each staged record's voxel (when the instance has several)
    __device__ __forceinline__ uint32_t sub_of(uint32_t j, const W&, const InstParams&) const { return sub[j]; }
    // staged voxel index of (row rb, column c, plane pa)
    __device__ __forceinline__ uint32_t vox(uint32_t rb, uint32_t c, uint32_t pa) const {
        return (rb * G.NC + (c - G.cl)) * np + pa;
    }
    using Recs = LdsRecords<D, MIXED>;
    __device__ __forceinline__ Rec record(uint32_t j, const W&) const { return Recs::at(lds, j * Recs::kBytes); }
    __device__ __forceinline__ int species(uint32_t j, const Rec& r) const {
        if constexpr (MIXED) return (int)((uint32_t)r.w & kSpeciesMask);
        else return (int)lsp[j];
    }
    // global slot of LDS index j (only on the rare FP64 re-evaluation path)
    __device__ __forceinline__ uint32_t slot(uint32_t j, const W&) const {
        uint32_t lo = 0, hi = n_vox;  // largest v with vst[v] <= j
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if ((uint32_t)vst[mid] <= j) lo = mid;
            else hi = mid;
        }
        const uint32_t pa = lo % np, t = lo / np, c = G.cl + t % G.NC, rb = t / G.NC;
        const uint32_t a = G.a0 + pa - (np == 3 ? 1u : 0u), b = G.b0 - 1 + rb;
        return start[voff + (a * n1 + b) * n2 + c] + (j - (uint32_t)vst[lo]);
    }
};

// Global source (tiles whose region does not fit in LDS): the stream walks the
// stencil voxel by voxel in the same order.
struct WalkVox {
    uint32_t j, je;
    uint32_t rb, cc, pa;     // current voxel: row b_lo + rb, column c_lo + cc, plane a_lo + pa
    uint32_t nb, ncol, na;   // stencil extent (clipped)
    uint32_t a_lo, b_lo, c_lo;
    const uint32_t* start;
    uint32_t voff, n1, n2;
    __device__ __forceinline__ uint32_t gvox() const {
        return voff + ((a_lo + pa) * n1 + (b_lo + rb)) * n2 + c_lo + cc;
    }
    __device__ __forceinline__ bool settle() {
        while (j >= je) {
            const uint32_t over = j - je;
            if (++pa == na) {
                pa = 0;
                if (++cc == ncol) {
                    cc = 0;
                    if (++rb == nb) return false;
                }
            }
            const uint32_t g = gvox();
            j = start[g] + over;
            je = start[g + 1];
        }
        return true;
    }
};

template <int D, bool MIXED>
struct GlobalSource {
    using Rec = typename RecOf<MIXED>::type;
    using W = WalkVox;
    const Rec* rec;
    Region G;
    __device__ __forceinline__ Rec record(uint32_t j, const W& w) const {
        if constexpr (MIXED)
            return to_region<D>(rec[j], (int)(w.a_lo + w.pa + 1 - G.a0), (int)(w.b_lo + w.rb + 1 - G.b0), G);
        else
            return rec[j];
    }
    __device__ __forceinline__ int species(uint32_t, const Rec& r) const {
        if constexpr (MIXED) return (int)((uint32_t)r.w & kSpeciesMask);
        else return (int)r.w;
    }
    __device__ __forceinline__ uint32_t slot(uint32_t j, const W&) const { return j; }
    __device__ __forceinline__ uint32_t sub_of(uint32_t, const W& w, const InstParams& P) const {
        return subdomain_of(P, w.gvox() - w.voff);
    }
};

// Strength row of the species matrix in four scalars (a register array indexed
// by a run-time species would be placed in scratch memory).
template <typename T>
struct Row4 {
    T v0, v1, v2, v3;
    // bit tests rather than a compare chain on k, which the compiler turns back into
    // an indexed (scratch) table
    __device__ __forceinline__ T pick(int k) const {
        const bool b0 = (k & 1) != 0, b1 = (k & 2) != 0;
        const T lo = b0 ? v1 : v0, hi = b0 ? v3 : v2;
        return b1 ? hi : lo;
    }
};

// Force on the agent in slot s: `me` is its record in the source's coordinates,
// `self` its index in the source's index space, `ov` its own voxel's range there
// (same-voxel pairs) and `w0` the start of its candidate stream.
//
// Two passes per chunk of 64 stream positions: a cheap squared-distance test
// marks the candidates that can be inside the cutoff in a 64-bit mask, then the
// chunk is replayed and only the marked pairs are evaluated, in stream order.
// Every unmarked pair is beyond the cutoff, where each potential's force is
// exactly zero, so the sums are those of the full loop without its zero terms.
// The wave pays max-over-lanes of the marked count for the expensive pass
// instead of max-over-lanes of the candidate count.
//
// Lanes per agent (LDS source): 2^lg consecutive lanes of a wave share one agent;
// lane `sub` of the group walks every 2^lg-th candidate of the stream from the sub-th
// (a cluster of close agents is spread over the lanes; with one contiguous part per
// lane 2400 crowded 3-D agents that had drawn together took 164 us with 8 lanes and
// 92 with one), and the group adds its partial sums with wavefront shuffles (a butterfly, so every
// lane of the group holds the same total) before lane 0 writes the force.
template <int D, int POT, bool MIXED, bool SENSE, typename Src>
__device__ __forceinline__ void agent_force(const Arrays& A, const StateBuf& S, const InstParams& P, uint64_t s,
                                            uint32_t self, const typename RecOf<MIXED>::type me, Span ov,
                                            typename Src::W cur, uint32_t physical, uint32_t symmetric,
                                            const Src& src, const float* unit, uint32_t sub = 0, uint32_t lg = 0) {
    using T = typename std::conditional<MIXED, float, double>::type;
    using Rec = typename RecOf<MIXED>::type;
    using W = typename Src::W;
    const uint64_t N = A.N;
    const PotParams<T>& PP = pot_of<T>(P);
    const T rc = cut_radius<POT, T>(PP);
    const float rc2 = (float)(rc * rc);
    const float band = 2e-6f * rc2;

    const int sp_i = src.species(self, me);
    bool flag_i = false;
    if constexpr (MIXED) flag_i = me.w < 0;
    // candidate test thresholds: mixed marks d2 <= rc2 + band (the band pairs are
    // re-decided in FP64) and every pair with a flagged agent; FP64 marks
    // d2 <= rc^2 (1 + 1e-12), beyond which the rounded sqrt(d2) exceeds rc.
    // Mixed pass 1 measures in units of the first axis' fixed-point step (the
    // other axes scaled by their step ratio) and keeps half a band more margin.
    float r1 = 1.0f, r2 = 1.0f, thr_f = 0.0f, close2 = 0.0f;
    if constexpr (MIXED) {
        const float u0 = unit[0];
        r1 = unit[1] / u0;
        r2 = unit[D - 1] / u0;
        thr_f = (rc2 + 1.5f * band) / (u0 * u0);
        if (!(thr_f >= 0.0f) || flag_i) thr_f = __builtin_inff();
        // pairs closer than 2e6 fixed-point steps (where the quantised direction
        // would be off by more than 1e-6) take their displacement from FP64
        const float umax = fmaxf(fmaxf(unit[0], unit[1]), unit[D - 1]);
        close2 = (2e6f * umax) * (2e6f * umax);
    }
    const double rcd = (double)cut_radius<POT, double>(P.pd);
    double thr_d = rcd * rcd * (1.0 + 1e-12);
    if (!(thr_d >= 0.0)) thr_d = __builtin_inf();

    // Neighbour sensing (NeighborSensing::accumulate_information, concepts
    // interaction.rs:64-79, called per stencil pair at update_mechanics.rs:105,
    // 199-202) counts the candidates with squared distance below sense_t, the
    // smallest double whose square root reaches the radius, so that the test is
    // the reference's norm < radius.  Pass 1 then marks up to the larger of the
    // two radii, and pass 2 replays pass 1's force test for each marked pair.
    // Mixed precision counts from the fixed-point distance outside a band that
    // bounds its error (quantisation of both ends plus float rounding) and
    // decides the band's pairs from the FP64 positions.
    constexpr bool sense = SENSE;
    uint32_t n_sense = 0;
    float mark_f = thr_f, rs2 = 0.0f, band_s = 0.0f;
    double mark_d = thr_d;
    if constexpr (SENSE) {
        if constexpr (MIXED) {
            const float umax = fmaxf(fmaxf(unit[0], unit[1]), unit[D - 1]);
            const float q = 2.0f * (float)D * umax;
            rs2 = (float)A.sense_t;
            band_s = 2e-6f * rs2 + 4.0f * sqrtf(rs2) * q + q * q;
            float t = (rs2 + 2.0f * band_s) / (unit[0] * unit[0]);
            if (!(t >= 0.0f) || flag_i) t = __builtin_inff();
            mark_f = fmaxf(thr_f, t);
        } else {
            mark_d = fmax(thr_d, A.sense_t * (1.0 + 1e-12));
        }
    }
    const bool wider = MIXED ? mark_f > thr_f : mark_d > thr_d;
    // chili with several subdomains: pairs across a subdomain border get both halves
    // (update_mechanics.rs:285-382)
    const bool subs = P.sub_on != 0;
    const uint32_t my_sub = subs ? subdomain_of(P, S.vox[s] - P.voxel_offset) : 0u;

    // species-matrix row (own species) and column (own species as ext): Morse
    // strengths, or the Langevin sorting interaction's attractions
    Row4<T> srow, scol;
    {
        T r4[CRM_MAX_SPECIES], c4[CRM_MAX_SPECIES];
#pragma unroll
        for (int k = 0; k < CRM_MAX_SPECIES; k++) {
            if constexpr (POT == CRM_POTENTIAL_MORSE_SPECIES) {
                r4[k] = PP.strength * PP.species_matrix[sp_i * CRM_MAX_SPECIES + k];
                c4[k] = PP.strength * PP.species_matrix[k * CRM_MAX_SPECIES + sp_i];
            } else if constexpr (POT == CRM_POTENTIAL_CELL_SORTING_LANGEVIN) {  // attraction
                r4[k] = PP.species_matrix[sp_i * CRM_MAX_SPECIES + k];
                c4[k] = PP.species_matrix[k * CRM_MAX_SPECIES + sp_i];
            } else {
                r4[k] = c4[k] = PP.strength;
            }
        }
        srow = Row4<T>{r4[0], r4[1], r4[2], r4[3]};
        scol = Row4<T>{c4[0], c4[1], c4[2], c4[3]};
    }
    // per-agent sums: double in FP64 mode; float in mixed mode, whose forces are
    // stored as float (a compensated Kahan sum changed the stored forces by
    // nothing measurable -- 1M-agent 3-D sorting error 4.29e-7 either way, 4M-agent
    // Mie lattice 1.91e-6 against 1.93e-6 -- and cost 5 % of the kernel; a double
    // accumulator was slower)
    double accd[D];
    float ks[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        accd[k] = 0.0;
        ks[k] = 0.0f;
    }
    auto kadd = [&](int k, float x) { ks[k] = ks[k] + x; };
    bool calc_err = false;

    // Pair displacement own - candidate; returns the squared distance.
    auto displacement = [&](const Rec& rj, T* z) -> T {
        T d2 = T(0);
        if constexpr (MIXED) {
            z[0] = (float)(me.x - rj.x) * unit[0];
            z[1] = (float)(me.y - rj.y) * unit[1];
            if constexpr (D == 3) z[2] = (float)(me.z - rj.z) * unit[2];
        } else {
            z[0] = me.x - rj.x;
            z[1] = me.y - rj.y;
            if constexpr (D == 3) z[2] = me.z - rj.z;
        }
#pragma unroll
        for (int k = 0; k < D; k++) d2 = d2 + z[k] * z[k];
        return d2;
    };

    // Pass 1's squared distance: mixed in units of the first axis' fixed-point
    // step, FP64 with fused products.
    auto mark_dist = [&](const Rec& rj) -> T {
        if constexpr (MIXED) {
            const float c0 = (float)(me.x - rj.x);
            const float c1 = (float)(me.y - rj.y) * r1;
            float d2 = fmaf(c1, c1, c0 * c0);
            if constexpr (D == 3) {
                const float c2 = (float)(me.z - rj.z) * r2;
                d2 = fmaf(c2, c2, d2);
            }
            return d2;
        } else {
            const double z0 = me.x - rj.x, z1 = me.y - rj.y;
            double d2 = fma(z1, z1, z0 * z0);
            if constexpr (D == 3) {
                const double z2 = me.z - rj.z;
                d2 = fma(z2, z2, d2);
            }
            return d2;
        }
    };

    // The pair with the candidate at walk position w, weighted as in the reference.
    auto evaluate = [&](const W& w) {
        const uint32_t j = w.j;
        const Rec rj = src.record(j, w);
        T z[D];
        const T d2 = displacement(rj, z);
        if constexpr (SENSE) {
            bool in;
            if constexpr (MIXED) {
                if (flag_i || rj.w < 0 || fabsf(d2 - rs2) <= band_s) {
                    const uint32_t gj = src.slot(j, w);
                    double zd[D];
#pragma unroll
                    for (int k = 0; k < D; k++) zd[k] = S.pos[k * N + s] - S.pos[k * N + gj];
                    in = sum_squares_unfused<D>(zd) < A.sense_t;
                } else {
                    in = d2 < rs2;
                }
            } else {
                in = sum_squares_unfused<D>(z) < A.sense_t;
            }
            n_sense += in ? 1u : 0u;
            // the force only for the pairs pass 1 marks without sensing (all of
            // them unless the sensing radius widened the marks)
            if constexpr (POT == CRM_POTENTIAL_NONE) return;
            if (wider) {
                bool fmark;
                if constexpr (MIXED) fmark = mark_dist(rj) <= thr_f || rj.w < 0;
                else fmark = mark_dist(rj) <= thr_d;
                if (!fmark) return;
            }
        }
        const bool full = physical || (j >= ov.b && j < ov.e) || (subs && src.sub_of(j, w, P) != my_sub);
        const int sp_j = src.species(j, rj);
        int cut = -1;
        if constexpr (MIXED) {
            const bool refine = flag_i || rj.w < 0 || d2 < close2 || fabsf(d2 - rc2) <= band;
            if (refine) {
                const uint32_t gj = src.slot(j, w);
                double zd[D], dd = 0.0;
#pragma unroll
                for (int k = 0; k < D; k++) {
                    zd[k] = S.pos[k * N + s] - S.pos[k * N + gj];
                    dd = dd + zd[k] * zd[k];
                    z[k] = (float)zd[k];
                }
                cut = cut_decision<POT>(P.pd, sqrt(dd));
            }
        }
        T f[D];
        const bool same_sp = sp_i == sp_j;
        calc_err |= point_force<POT, T, D>(z, same_sp, srow.pick(sp_j), PP, cut, f);
        T wgt = T(0.5);
        if (full) {
            // (only interactions of species pairs can differ by the order of the pair)
            constexpr bool by_species =
                POT == CRM_POTENTIAL_MORSE_SPECIES || POT == CRM_POTENTIAL_CELL_SORTING_LANGEVIN;
            if (!by_species || symmetric) {
                wgt = T(1);
            } else {
                T zj[D], g[D];
#pragma unroll
                for (int k = 0; k < D; k++) zj[k] = -z[k];
                calc_err |= point_force<POT, T, D>(zj, same_sp, scol.pick(sp_j), PP, cut, g);
#pragma unroll
                for (int k = 0; k < D; k++) {
                    if constexpr (MIXED) kadd(k, -g[k] * 0.5f);
                    else accd[k] = accd[k] + (-g[k]) * 0.5;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < D; k++) {
            if constexpr (MIXED) kadd(k, f[k] * wgt);
            else accd[k] = accd[k] + f[k] * wgt;
        }
    };

    if constexpr (std::is_same<W, Walk3>::value) {
        // LDS source: the stream is three ranges of LDS indices, [j0, e0), [j1, e1),
        // [j2, e2), read as one index space p in [0, L): p < B1 is range 0, p < B2
        // range 1, the rest range 2 (empty ranges fold away), so the walk needs no
        // per-candidate range bookkeeping.  The own record sits in range 1 at p_self
        // and is unmarked once per chunk.  Pass 1 marks, pass 2 evaluates the marked
        // positions in stream order -- the same pairs, order and arithmetic as the
        // generic walk below.
        const bool active = POT != CRM_POTENTIAL_NONE || sense;
        const uint32_t B1 = cur.je - cur.j, B2 = B1 + (cur.e1 - cur.j1);
        const uint32_t L = active ? B2 + (cur.e2 - cur.j2) : 0u;
        const uint32_t o1 = cur.j1 - cur.je, o2 = cur.j2 - cur.e1;  // modular offsets
        // this lane's share of the stream, the positions p = sub + (r << lg), walked by r
        // (the same for every lane of a wave, so the loop counters stay scalar)
        const uint32_t last = (1u << lg) - 1u;
        auto upto = [&](uint32_t e) -> uint32_t { return e > sub ? (e - sub + last) >> lg : 0u; };
        const uint32_t Lr = upto(L);
        const uint32_t R1 = upto(B1), R2 = upto(B2);  // first r of the later ranges
        const uint32_t p_self = B1 + (self - cur.j1);
        const uint32_t r_self = (p_self & last) == sub ? p_self >> lg : 0xffffffffu;
        // LDS byte offset of stream offset r (the range offsets scaled once, not per
        // candidate), its record and its LDS index
        using Recs = typename Src::Recs;
        constexpr uint32_t RB = Recs::kBytes;
        const uint32_t jb0 = (cur.j + sub) * RB, off1b = o1 * RB, off2b = o2 * RB, RS = RB << lg;
        auto atb = [&](uint32_t r) -> uint32_t { return jb0 + r * RS + (r >= R1 ? off1b : 0u) + (r >= R2 ? off2b : 0u); };
        auto rec_at = [&](uint32_t r) -> Rec { return Recs::at(src.lds, atb(r)); };
        auto at = [&](uint32_t r) -> uint32_t { return atb(r) / RB; };
        // unit grids (equal fixed-point steps on every axis) need no axis scaling in
        // pass 1 (r1 = r2 = 1 exactly, so the marks are the same)
        const bool cubic = !MIXED || (r1 == 1.0f && r2 == 1.0f);
        auto marked = [&](auto cub, uint32_t p) -> uint32_t {
            const Rec rj = rec_at(p);
            bool mark;
            if constexpr (MIXED) {
                float d2;
                if constexpr (decltype(cub)::value) {
                    const float c0 = (float)(me.x - rj.x), c1 = (float)(me.y - rj.y);
                    d2 = fmaf(c1, c1, c0 * c0);
                    if constexpr (D == 3) {
                        const float c2 = (float)(me.z - rj.z);
                        d2 = fmaf(c2, c2, d2);
                    }
                } else {
                    d2 = mark_dist(rj);
                }
                mark = d2 <= mark_f || rj.w < 0;
            } else {
                mark = mark_dist(rj) <= mark_d;
            }
            return mark ? 1u : 0u;
        };
        auto pass1 = [&](auto cub, uint32_t p0, uint32_t qn, uint32_t& mlo, uint32_t& mhi) {
            const uint32_t q1 = min(qn, 32u);
            for (uint32_t q = 0; q < q1; q++) mlo |= marked(cub, p0 + q) << q;
            for (uint32_t q = 32; q < qn; q++) mhi |= marked(cub, p0 + q) << (q - 32u);
        };
        for (uint32_t p0 = 0; p0 < Lr; p0 += 64u) {
            const uint32_t qn = min(64u, Lr - p0);
            uint32_t mlo = 0, mhi = 0;
            if (cubic) pass1(std::true_type{}, p0, qn, mlo, mhi);
            else pass1(std::false_type{}, p0, qn, mlo, mhi);
            const uint32_t ds = r_self - p0;  // the self pair is never evaluated
            if (ds < 32u) mlo &= ~(1u << ds);
            else if (ds < 64u) mhi &= ~(1u << (ds - 32u));
            W w = cur;
            while (mlo | mhi) {
                uint32_t q;
                if (mlo) {
                    q = (uint32_t)__builtin_ctz(mlo);
                    mlo &= mlo - 1;
                } else {
                    q = 32u + (uint32_t)__builtin_ctz(mhi);
                    mhi &= mhi - 1;
                }
                w.j = at(p0 + q);
                evaluate(w);
            }
        }
    } else {
    bool live = POT != CRM_POTENTIAL_NONE || sense;
    if (live) live = cur.settle();
    while (live) {
        const W c0 = cur;
        // pass 1: mark the candidates that can be inside the cutoff (bit p of
        // mlo / mhi for stream position p of the chunk)
        uint32_t mlo = 0, mhi = 0;
        for (uint32_t p = 0; p < 64u; p++) {
            const uint32_t j = cur.j;
            const Rec rj = src.record(j, cur);
            bool mark;
            if constexpr (MIXED) mark = mark_dist(rj) <= mark_f || rj.w < 0;
            else mark = mark_dist(rj) <= mark_d;
            mark = mark && j != self;
            const uint32_t bit = 1u << (p & 31u);
            if (p < 32u) mlo = mark ? (mlo | bit) : mlo;
            else mhi = mark ? (mhi | bit) : mhi;
            ++cur.j;
            live = cur.settle();
            if (!live) break;
        }
        // pass 2: replay the chunk and evaluate the marked pairs in stream order
        W w = c0;
        uint32_t pos = 0;
        while (mlo | mhi) {
            uint32_t p;
            if (mlo) {
                p = (uint32_t)__builtin_ctz(mlo);
                mlo &= mlo - 1;
            } else {
                p = 32u + (uint32_t)__builtin_ctz(mhi);
                mhi &= mhi - 1;
            }
            w.j += p - pos;
            pos = p;
            w.settle();
            evaluate(w);
        }
    }
    }
    double fsum[D];
#pragma unroll
    for (int k = 0; k < D; k++) fsum[k] = MIXED ? (double)ks[k] : accd[k];
    if (lg) {  // the group's partial sums, by xor butterfly (same order on every lane)
        uint32_t err = calc_err ? 1u : 0u;
        for (uint32_t o = 1; o < (1u << lg); o <<= 1) {
#pragma unroll
            for (int k = 0; k < D; k++) fsum[k] = fsum[k] + __shfl_xor(fsum[k], (int)o, 64);
            err |= (uint32_t)__shfl_xor((int)err, (int)o, 64);
            if constexpr (SENSE) n_sense += (uint32_t)__shfl_xor((int)n_sense, (int)o, 64);
        }
        calc_err = err != 0;
        if (sub) return;
    }
    if (calc_err) raise_error(A.ctrl, CRM_CALC_ERROR, A.ctrl->step, S.id[s]);
    // the domain force follows the pair forces (calculate_custom_domain_force after
    // the subdomain's pairs, run_sim.rs:277-279, update_mechanics.rs:244-274)
    const bool spring = P.dforce == CRM_DOMAIN_FORCE_SPRING;
#pragma unroll
    for (int k = 0; k < D; k++) {
        double f = fsum[k];
        if (spring) f = f + (-P.dk[k]) * (S.pos[(uint64_t)k * N + s] - P.dc[k]);
        if constexpr (MIXED) A.forcef[(uint64_t)k * N + s] = (float)f;  // the pair sums are float already
        else A.force[(uint64_t)k * N + s] = f;
    }
    if constexpr (SENSE) A.sense[s] = n_sense;
}

// A force tile: plane a0, rows [b0, b1), columns [c0, c1) of one instance.
constexpr int kTileRowsMax = 29;
constexpr int kLdsVoxelStarts = 768;    // 1.5 KiB of voxel-start indices (staged voxels + 1)
constexpr int kOwnVoxMax = 256;         // own voxels per tile
constexpr int kSortBins = 64;           // candidate-count classes for the lane order
constexpr double kWideVoxels = 1.25;    // voxel edges per cutoff above which streams are cut to the cutoff's reach

struct ForceTile {
    uint32_t inst, a0, b0, b1, c0, c1;
};

// An own agent of a force tile, looked up once: its record's LDS index, its
// voxel's LDS range, the three LDS ranges of its candidate stream, its slot.
struct OwnEntry {
    uint16_t self, ovb, ove;
    uint16_t r[6];
    uint16_t pad;
    uint32_t slot;
};

// Inclusive prefix sum over the 64 lanes of a wave (all lanes active).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(v, o, 64);
        if (lane >= (uint32_t)o) v += y;
    }
    return v;
}

// Exclusive prefix sum over the workgroup; total = the sum of all x.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t x, uint32_t& total) {
    __shared__ uint32_t wave_tot[kBlock / 64];
    const int wave = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(x);
    if ((threadIdx.x & 63) == 63) wave_tot[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int q = 0; q < kBlock / 64; q++) {
        const uint32_t wt = wave_tot[q];
        if (q < wave) before += wt;
        all += wt;
    }
    __syncthreads();
    total = all;
    return before + inc - x;
}

// ---------------------------------------------------------------------------
// The next order of a step.  Which voxel every agent moves to is known before the step's
// forces (bin_ahead) or right after them (k_key_point, k_key_rod); note_move keeps, per
// voxel, arrivals less departures and the list of arrivals.  The new voxel starts are
// then a scan of (agents now + delta), and an agent's new slot follows from its old one:
// a stayer's is its new voxel start plus the stayers before it in the voxel, counted with
// wave ballots; an arrival's is counted back from the voxel's end by the arrivals' slots.
//
// The scan needs nothing of the forces, so it is work of further workgroups of the force
// kernel, and the gather writes straight to the new slots: a step is two launches.  As a
// counting sort (ranks in the force kernel, scan, scatter, gather by the sorted order) it was four,
// each with at least 4.5 us in a chain: 50 steps of 30,000 sorting agents
// 1.71 -> 1.33 ms, 100 of 300,000 in FP64 8.10 -> 7.36, 25 of 1600 crowded cells 1.14 ->
// 0.93, 50 of 12,347 rods 5.50 -> 5.27.  The gather itself got slower, since its stores, not
// its loads, are now the unaligned side (1M agents 57 -> 65 us, 4M 201 -> 227); other
// workgroup orders and plain stores changed nothing.  Those systems move about one agent in a
// hundred per step.  Where most agents change voxel in every step, the lists and the scattered
// stores still cost less than the ranks did in voxels of several agents (free agents, a voxel
// per step: 1M in voxels of 5 344 -> 301 us a step, of 13 685 -> 359, 300,000 in voxels of
// 30 458 -> 265, 20,000 in voxels of 500 309 -> 154) and up to 6 % more with one agent per
// voxel (1M: 247 -> 264; at 0.3 of a voxel per step 172 -> 176).
// ---------------------------------------------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTileLog2 = 11;
constexpr int kScanTile = kBlock * kScanItems;
static_assert(kScanTile == 1 << kScanTileLog2, "voxels of a scan tile");
// Scan tiles of a step at most (two per thread of a gather workgroup, which scans their
// sums); larger grids get tiles of 2^scan_shift times kScanTile voxels.
constexpr uint32_t kStepScanTiles = 512;

// The agent in slot s of voxel v moves to voxel k.
__device__ __forceinline__ void note_move(int32_t* delta, uint32_t* head, uint32_t* link, uint32_t s, uint32_t v,
                                          uint32_t k) {
    if (k == v) return;
    atomicAdd(&delta[v], -1);
    atomicAdd(&delta[k], 1);
    link[s] = atomicExch(&head[k], s + 1u);
}

// Offsets of the tile's voxels inside it (start_local) and its sum (tile_off) in the
// next order; clears delta for the next step's moves, and the lists that they go to.
__device__ __forceinline__ void scan_moves(const Arrays& A, uint32_t tile) {
    static_assert(kScanItems == 8, "two 16-byte accesses per group");
    const uint32_t Vt = A.Vt;
    uint32_t carry = 0;
    for (uint32_t c = 0; c < (1u << A.scan_shift); c++) {
        const uint64_t base = (((uint64_t)tile << A.scan_shift) + c) * kScanTile + (uint64_t)threadIdx.x * kScanItems;
        uint32_t vals[kScanItems], sum = 0;
        const bool whole = base + kScanItems <= Vt;
        if (whole) {  // (start, delta, head and start_local are 256-byte aligned)
            const uint4* b4 = reinterpret_cast<const uint4*>(A.start + base);
            int4* d4 = reinterpret_cast<int4*>(A.delta + base);
            uint4* h4 = reinterpret_cast<uint4*>(A.head_next + base);
            const uint4 b0 = b4[0], b1 = b4[1];
            const uint32_t e = A.start[base + kScanItems];
            const int4 d0 = d4[0], d1 = d4[1];
            vals[0] = b0.y - b0.x + (uint32_t)d0.x;
            vals[1] = b0.z - b0.y + (uint32_t)d0.y;
            vals[2] = b0.w - b0.z + (uint32_t)d0.z;
            vals[3] = b1.x - b0.w + (uint32_t)d0.w;
            vals[4] = b1.y - b1.x + (uint32_t)d1.x;
            vals[5] = b1.z - b1.y + (uint32_t)d1.y;
            vals[6] = b1.w - b1.z + (uint32_t)d1.z;
            vals[7] = e - b1.w + (uint32_t)d1.w;
            d4[0] = d4[1] = make_int4(0, 0, 0, 0);
            h4[0] = h4[1] = make_uint4(0u, 0u, 0u, 0u);
        } else {
#pragma unroll
            for (int i = 0; i < kScanItems; i++) {
                const uint64_t q = base + i;
                vals[i] = q < Vt ? A.start[q + 1] - A.start[q] + (uint32_t)A.delta[q] : 0u;
                if (q < Vt) {
                    A.delta[q] = 0;
                    A.head_next[q] = 0u;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kScanItems; i++) sum += vals[i];
        uint32_t total;
        uint32_t run = carry + block_exclusive_scan(sum, total);
        carry += total;
        uint32_t out[kScanItems];
#pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            out[i] = run;
            run += vals[i];
        }
        if (whole) {
            uint4* o4 = reinterpret_cast<uint4*>(A.start_local + base);
            o4[0] = make_uint4(out[0], out[1], out[2], out[3]);
            o4[1] = make_uint4(out[4], out[5], out[6], out[7]);
        } else {
#pragma unroll
            for (int i = 0; i < kScanItems; i++)
                if (base + i < Vt) A.start_local[base + i] = out[i];
        }
    }
    if (threadIdx.x == 0) {
        A.tile_off[tile] = carry;
        if (tile == 0) A.ctrl->gather_step = A.ctrl->step;
    }
}

// In place of the scan after an error: the gather finds the step that is not to run (with
// the failing step's number in gather_step it would run again).
__device__ __forceinline__ void skip_scan(const Arrays& A) {
    if (blockIdx.x == 0 && threadIdx.x == 0) A.ctrl->gather_step = A.ctrl->step;
}

__global__ __launch_bounds__(kBlock) void k_scan_moves(Arrays A) {
    if (halted(A.ctrl, A.ctrl->step)) skip_scan(A);
    else scan_moves(A, blockIdx.x);
}

// An agent's old voxel v, its next voxel k, and the stayers of v in the slots before its own.
struct Move {
    uint32_t v, k, r;
};

// The moves of slots first + threadIdx.x for threadIdx.x < count; called by whole
// workgroups.  Slots are sorted by voxel, so a voxel's slots in a wave are one run of
// lanes; the part of the first lane's voxel before the wave is looked up by all lanes.
__device__ __forceinline__ Move move_of(const Arrays& A, const uint32_t* __restrict__ vox, uint32_t first,
                                        uint32_t count) {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x & ~63u, w0 = first + w;
    const bool live = threadIdx.x < count;
    Move m{0xffffffffu, 0xffffffffu, 0u};
    if (live) {
        m.v = vox[first + threadIdx.x];
        m.k = A.key[first + threadIdx.x];
    }
    uint32_t base = w0;
    bool ok = w < count && base > lane;
    uint32_t vb = ok ? vox[base - 1u - lane] : 0u, kb = ok ? A.key[base - 1u - lane] : 0u;
    const uint32_t v0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)m.v);
    ok = ok && vb == v0;
    uint32_t before = (uint32_t)__popcll(__ballot(ok && kb == v0));
    while (__ballot(ok) == ~0ull) {  // more than 64 of them
        base -= 64u;
        ok = base > lane;
        vb = ok ? vox[base - 1u - lane] : 0u;
        kb = ok ? A.key[base - 1u - lane] : 0u;
        ok = ok && vb == v0;
        before += (uint32_t)__popcll(__ballot(ok && kb == v0));
    }
    const uint32_t vp = __shfl_up(m.v, 1, 64);
    const uint64_t runs = __ballot(lane == 0u || m.v != vp), stay = __ballot(live && m.k == m.v);
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t h = 63u - (uint32_t)__clzll((long long)(runs & (below | (1ull << lane))));  // the run's first lane
    m.r = (uint32_t)__popcll(stay & below & ~((1ull << h) - 1ull)) + (h == 0u ? before : 0u);
    return m;
}

// Offsets of the scan tiles, from their sums, in s_off[kStepScanTiles].
__device__ __forceinline__ void step_tile_offsets(const Arrays& A, uint32_t* s_off) {
    if (A.n_scan == 1u) {
        if (threadIdx.x == 0) s_off[0] = 0u;
    } else {
        const uint32_t q = 2u * threadIdx.x;
        const uint32_t x = q < A.n_scan ? A.tile_off[q] : 0u, y = q + 1u < A.n_scan ? A.tile_off[q + 1u] : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive_scan(x + y, total);
        s_off[q] = ex;
        s_off[q + 1u] = ex + x;
    }
    __syncthreads();
}

// Voxel v's start in the next order (sl = start_local[v]).
__device__ __forceinline__ uint32_t next_start(const Arrays& A, const uint32_t* s_off, uint32_t v, uint32_t sl) {
    return sl + s_off[v >> (kScanTileLog2 + A.scan_shift)];
}

// Slot in the next order of the agent in slot g with move m (sl = start_local[m.k]).
__device__ __forceinline__ uint32_t next_slot(const Arrays& A, const uint32_t* s_off, uint32_t g, const Move& m,
                                              uint32_t sl) {
    if (m.k == m.v) return next_start(A, s_off, m.k, sl) + m.r;
    uint32_t n = 0, before = 0;
    for (uint32_t j = A.head[m.k]; j != 0u; j = A.link[j - 1u]) {
        n++;
        before += j - 1u < g ? 1u : 0u;
    }
    const uint32_t e = m.k + 1u < A.Vt ? next_start(A, s_off, m.k + 1u, A.start_local[m.k + 1u]) : (uint32_t)A.N;
    return e - n + before;
}

// The workgroup's share of the new voxel starts (sl = start_local of its thread's first).
__device__ __forceinline__ void write_starts(const Arrays& A, const uint32_t* s_off, uint32_t sl) {
    const uint64_t v0 = (uint64_t)blockIdx.x * kBlock + threadIdx.x, step = (uint64_t)gridDim.x * kBlock;
    if (v0 < A.Vt) A.start[v0] = next_start(A, s_off, (uint32_t)v0, sl);
    for (uint64_t v = v0 + step; v < A.Vt; v += step) A.start[v] = next_start(A, s_off, (uint32_t)v, A.start_local[v]);
    if (blockIdx.x == 0 && threadIdx.x == 0) A.start[A.Vt] = (uint32_t)A.N;
}
__device__ __forceinline__ uint32_t first_start_local(const Arrays& A) {
    const uint64_t v = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    return v < A.Vt ? A.start_local[v] : 0u;
}

// The gather's last duty towards the order: the new starts and the completed step (the
// gather itself reads gather_step).
__device__ __forceinline__ void finish_order(const Arrays& A, const uint32_t* s_off, uint32_t sl, uint64_t t) {
    write_starts(A, s_off, sl);
    if (blockIdx.x == 0 && threadIdx.x == 0) A.ctrl->step = t + 1;
}

// The new starts on their own, ahead of the gather that writes them again: in contexts
// that time the kernel classes, whose scan is a launch of its own as well.
__global__ __launch_bounds__(kBlock) void k_next_starts(Arrays A) {
    __shared__ uint32_t s_off[kStepScanTiles];
    if (halted(A.ctrl, A.ctrl->gather_step)) return;
    step_tile_offsets(A, s_off);
    write_starts(A, s_off, first_start_local(A));
}

// a / d for a < 2^14, 0 < d <= 64, with d's float reciprocal: (a + 1/2) / d keeps a
// fractional part >= 1/128 that the two float roundings cannot carry across.
__device__ __forceinline__ uint32_t small_div(uint32_t a, float inv_d) {
    return (uint32_t)(((float)a + 0.5f) * inv_d);
}

// Workgroup per tile: stage the region voxel by voxel (converted records, voxel
// starts) in LDS, then one lane per own agent sums its forces from LDS.  A tile
// whose region does not fit (local crowding) reads global memory instead; the
// candidate order and the arithmetic are the same.
// MULTI: the tiling policy gives each agent 2^lanes_log2 lanes, or the voxels are wide
// (a separate instantiation, so that the common one-lane kernel carries none of the
// group and reach logic).
template <int D, int POT, bool MIXED, bool SENSE, bool MULTI>
__global__ __launch_bounds__(kBlock, MIXED ? 5 : 4) void k_force_tiled(Arrays A, StateBuf S,
                                                                     const ForceTile* __restrict__ tiles,
                                                                     uint32_t physical, uint32_t symmetric,
                                                                     uint32_t no_lds, uint32_t n_scan,
                                                                     uint32_t lanes_log2) {
    const uint32_t lg = MULTI ? lanes_log2 : 0u;
    using Rec = typename RecOf<MIXED>::type;
    using Recs = LdsRecords<D, MIXED>;
    constexpr int CAP = Recs::kCap;
    constexpr uint32_t NP = D == 3 ? 3u : 1u;         // staged planes
    // the first n_scan workgroups scan the voxel counts (behind the others: 1M sorting agents
    // 77.8 -> 79.8 us; by the first tiles' workgroups themselves: 4M-agent lattice 495 -> 519)
    if (blockIdx.x < n_scan) {
        if (halted(A.ctrl, A.ctrl->step)) skip_scan(A);
        else scan_moves(A, blockIdx.x);
        return;
    }
    const ForceTile T = tiles[xcd_block(blockIdx.x - n_scan, gridDim.x - n_scan)];  // loaded beside the control block
    if (halted(A.ctrl, A.ctrl->step)) return;
    constexpr uint32_t PA_OWN = D == 3 ? 1u : 0u;     // the tile's own plane among them
    __shared__ __align__(16) char lds[Recs::kTotal];
    __shared__ uint8_t lsp[MIXED ? 1 : CAP];         // FP64: species of each staged record
    __shared__ uint16_t vst[kLdsVoxelStarts];        // LDS index of each staged voxel's first agent
    __shared__ uint16_t own_pre[kOwnVoxMax + 1];     // own agents before own voxel u
    __shared__ uint32_t own_gs[kOwnVoxMax];          // global slot of own voxel u's first agent
    __shared__ uint8_t ord[kBlock];                  // own agents in lane order
    __shared__ uint32_t bins[kSortBins];
    __shared__ OwnEntry own_tab[kBlock];             // own agent lookups (sorted case)
    __shared__ uint16_t lsub[CAP];                   // chili subdomain of each staged record (sub_on only)
    const Rec* __restrict__ rec = rec_array(A, std::integral_constant<bool, MIXED>());
    const InstParams& P = A.ip[T.inst];
    const uint32_t n0 = P.n[0], n1 = P.n[1], n2 = P.n[2], voff = P.voxel_offset;
    Region G;
    G.a0 = T.a0;
    G.b0 = T.b0;
    G.RW = T.b1 - T.b0 + 2;
    G.cl = T.c0 == 0 ? 0u : T.c0 - 1u;
    G.ch = min(T.c1 + 1u, n2);
    G.NC = G.ch - G.cl;
    {
        const uint32_t ext = max(max(NP, G.RW), G.NC);
        const int lg = ext <= 1 ? 0 : 32 - __clz(ext - 1);  // ceil(log2(ext))
        G.bits = min(30, 31 - lg);
        G.shift = 30 - G.bits;
    }
    float unit[3];
#pragma unroll
    for (int k = 0; k < D; k++) unit[k] = MIXED ? ldexpf(P.qunit[k + 3 - D], G.shift) : 0.0f;
    const uint32_t R = T.b1 - T.b0, W = T.c1 - T.c0;
    const uint32_t n_vox = G.RW * G.NC * NP;
    const uint32_t n_ownv = R * W;
    const bool fits = !no_lds && n_vox < (uint32_t)kLdsVoxelStarts && n_ownv <= (uint32_t)kOwnVoxMax;

    if (fits) {
        // staged voxel v = (rb * NC + c - cl) * NP + pa; thread t holds v = 3t .. 3t + 2
        // (in 3-D the three planes of one (row, column)).  Their (plane, row, column)
        // come from one decomposition of 3t, then step by one voxel each.
        uint32_t cnt[3], gs[3], sum = 0;
        int pa_q[3], rb_q[3];
        uint32_t c_q[3];
        {
            const uint32_t v0 = 3 * threadIdx.x;
            uint32_t pa, rb, c;
            if constexpr (NP == 3) {
                pa = 0;
                rb = small_div(threadIdx.x, 1.0f / (float)G.NC);
                c = G.cl + (threadIdx.x - rb * G.NC);
            } else {
                pa = 0;
                rb = small_div(v0, 1.0f / (float)G.NC);
                c = G.cl + (v0 - rb * G.NC);
            }
#pragma unroll
            for (int q = 0; q < 3; q++) {
                pa_q[q] = (int)pa;
                rb_q[q] = (int)rb;
                c_q[q] = c;
                cnt[q] = 0;
                gs[q] = 0;
                const int a = (int)T.a0 + (int)pa - (int)PA_OWN, b = (int)T.b0 - 1 + (int)rb;
                if (v0 + q < n_vox && a >= 0 && a < (int)n0 && b >= 0 && b < (int)n1) {
                    const uint32_t g = voff + ((uint32_t)a * n1 + (uint32_t)b) * n2 + c;
                    gs[q] = A.start[g];
                    cnt[q] = A.start[g + 1] - gs[q];
                }
                sum += cnt[q];
                // next voxel in the staged order
                if constexpr (NP == 3) {
                    pa++;
                } else {
                    const bool wrap = c + 1 == G.ch;
                    c = wrap ? G.cl : c + 1;
                    rb = wrap ? rb + 1 : rb;
                }
            }
        }
        // the first kPreRecs records of each voxel are loaded before the scan, so
        // that their latency overlaps its barriers (mixed: 4 int4 records, 1M-agent
        // 3-D sorting force kernel 86.7 -> 84.6 us against 2; FP64 keeps 2 double4,
        // more would spill)
        constexpr uint32_t kPreRecs = MIXED ? 4 : 2;
        Rec pre[3][kPreRecs];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (uint32_t k = 0; k < kPreRecs; k++)
                if (k < cnt[q]) pre[q][k] = rec[gs[q] + k];
        uint32_t total;
        uint32_t run = block_exclusive_scan(sum, total);
        const bool use_lds = total <= (uint32_t)CAP;  // uniform
        if (use_lds) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const uint32_t v = 3 * threadIdx.x + q;
                if (v < n_vox) {
                    vst[v] = (uint16_t)run;
                    const uint32_t pa = (uint32_t)pa_q[q], rb = (uint32_t)rb_q[q], c = c_q[q];
                    for (uint32_t k = 0; k < cnt[q]; k++) {
                        const Rec r = k < kPreRecs ? pre[q][k] : rec[gs[q] + k];
                        if constexpr (MIXED) {
                            Recs::put(lds, run + k, to_region<D>(r, (int)pa, (int)rb, G));
                        } else {
                            Recs::put(lds, run + k, r);
                            lsp[run + k] = (uint8_t)(int)r.w;
                        }
                    }
                    if (P.sub_on && cnt[q]) {
                        const int a = (int)T.a0 + (int)pa - (int)PA_OWN, b = (int)T.b0 - 1 + (int)rb;
                        const uint16_t o = (uint16_t)subdomain_of(P, ((uint32_t)a * n1 + (uint32_t)b) * n2 + c);
                        for (uint32_t k = 0; k < cnt[q]; k++) lsub[run + k] = o;
                    }
                    // own voxel u = r * W + (c - c0): its count and first global slot
                    if (pa == PA_OWN && rb >= 1 && rb <= R && c >= T.c0 && c < T.c1) {
                        const uint32_t u = (rb - 1) * W + (c - T.c0);
                        own_pre[u + 1] = (uint16_t)cnt[q];
                        own_gs[u] = gs[q];
                    }
                    run += cnt[q];
                }
            }
            if (threadIdx.x == 0) {
                vst[n_vox] = (uint16_t)total;
                own_pre[0] = 0;
            }
            __syncthreads();
            {  // own_pre: exclusive prefix of the own voxel counts (n_ownv <= 256)
                const uint32_t u = threadIdx.x;
                const uint32_t x = u < n_ownv ? (uint32_t)own_pre[u + 1] : 0u;
                uint32_t tot;
                const uint32_t ex = block_exclusive_scan(x, tot);
                if (u < n_ownv) own_pre[u + 1] = (uint16_t)(ex + x);
            }
            __syncthreads();
            const uint32_t n_own = own_pre[n_ownv];
            LdsSource<D, MIXED> src{lds, lsp, vst, G, NP, n_vox, A.start, voff, n1, n2, lsub};
            const float inv_w = 1.0f / (float)W;
            // Squared distances of an own agent to the borders of its voxel: to the rows
            // before and after it and to the columns.  What lies behind a border
            // farther than the cutoff (lim2 has 1e-5 to spare for the float arithmetic)
            // is left out of the stream: no candidate there is ever marked, so the
            // sums are the same.  With voxels of twice the cutoff that is more than half
            // of the candidates (1600 crowded 3-D agents: 28 -> 21 us); with voxels as
            // wide as the cutoff it is the corner pillars, 9.5 %, but a wave's longest
            // streams stay, and the code alone costs the one-lane kernels their last
            // registers (4M-agent lattice 501 -> 512 us): it is part of the MULTI kernels,
            // which serve every context with voxels wider than 1.25 cutoffs, and idle
            // below that.  Agents may be outside their voxel only after a position
            // without one (out_of_grid) or a failed step: then nothing is left out.
            struct Reach {
                float up2 = 0.0f, down2 = 0.0f, lo2 = 0.0f, hi2 = 0.0f;
            };
            const double rcut = cut_radius<POT, double>(P.pd);
            const bool trim = MULTI && !SENSE && fmin(P.dx[1], P.dx[2]) > kWideVoxels * rcut &&
                              A.ctrl->out_of_grid == 0 && A.ctrl->error_flags == 0;
            const float lim2 = (float)(rcut * rcut * (1.0 + 1e-5));
            auto reach_of = [&](const Rec& me, uint32_t r, uint32_t c) {  // own row r, column c
                float lo[2], hi[2];                                       // row, column
                if constexpr (MIXED) {
                    const int one = 1 << G.bits;
                    const int q[2] = {(D == 3 ? me.y : me.x) - ((int)(r + 1) << G.bits),
                                      (D == 3 ? me.z : me.y) - ((int)(c - G.cl) << G.bits)};
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        lo[k] = (float)q[k] * unit[D - 2 + k];
                        hi[k] = (float)(one - q[k]) * unit[D - 2 + k];
                    }
                } else {
                    const double x[2] = {D == 3 ? me.y : me.x, D == 3 ? me.z : me.y};
                    const uint32_t i[2] = {T.b0 + r, c};
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const double f = x[k] - (P.min[1 + k] + (double)i[k] * P.dx[1 + k]);
                        lo[k] = fmaxf((float)f, 0.0f);  // (a border's rounding may put it outside)
                        hi[k] = fmaxf((float)(P.dx[1 + k] - f), 0.0f);
                    }
                }
                return Reach{lo[0] * lo[0], hi[0] * hi[0], lo[1] * lo[1], hi[1] * hi[1]};
            };
            // own agent t: own voxel u (largest u with own_pre[u] <= t), LDS index,
            // global slot, and the three ranges of its stream
            auto own_agent = [&](uint32_t t, uint32_t& self, Span& ov, Walk3& w) -> uint32_t {
                uint32_t lo = 0, hi = n_ownv;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if ((uint32_t)own_pre[mid] <= t) lo = mid;
                    else hi = mid;
                }
                const uint32_t k = t - (uint32_t)own_pre[lo];
                const uint32_t r = small_div(lo, inv_w), c = T.c0 + (lo - r * W);
                const uint32_t vo = src.vox(r + 1, c, PA_OWN);
                self = (uint32_t)vst[vo] + k;
                ov = Span{vst[vo], vst[vo + 1]};
                // stencil rows r, r + 1, r + 2 of the region (b - 1, b, b + 1; rows
                // outside the grid are staged empty), each from its first to its last
                // column that the cutoff reaches
                Reach h;
                if (MULTI && trim) h = reach_of(Recs::at(lds, self * Recs::kBytes), r, c);
                auto range = [&](uint32_t q, float row2, uint32_t& j, uint32_t& je) {
                    const uint32_t cl = c - (c > 0u && !(row2 + h.lo2 > lim2) ? 1u : 0u);
                    const uint32_t ch = c + 1u + (c + 1u < n2 && !(row2 + h.hi2 > lim2) ? 1u : 0u);
                    j = vst[src.vox(r + q, cl, 0)];
                    je = vst[src.vox(r + q, row2 > lim2 ? cl : ch, 0)];
                };
                range(0, h.up2, w.j, w.je);
                range(1, 0.0f, w.j1, w.e1);
                range(2, h.down2, w.j2, w.e2);
                w.left = 2;
                return own_gs[lo] + k;
            };
            // Lanes take the own agents in descending order of candidate count, so
            // that a wave's lanes walk streams of similar length (a wave runs as
            // long as its longest stream).  Which lane computes an agent does not
            // change the agent's sums.
            // The sorted case looks each own agent up once and keeps the result in
            // LDS: self, own voxel range, the three stream ranges and the slot.
            const uint32_t gmask = (1u << lg) - 1u;  // lane within the agent's group
            const bool sorted = (n_own << lg) <= (uint32_t)kBlock;
            if (sorted) {
                if (threadIdx.x < kSortBins) bins[threadIdx.x] = 0;
                __syncthreads();
                uint32_t key = 0, kr = 0;
                if (threadIdx.x < n_own) {
                    uint32_t self;
                    Span ov;
                    Walk3 w;
                    const uint32_t s = own_agent(threadIdx.x, self, ov, w);
                    const uint32_t L = (w.je - w.j) + (w.e1 - w.j1) + (w.e2 - w.j2);
                    key = (uint32_t)(kSortBins - 1) - min(L >> 1, (uint32_t)(kSortBins - 1));
                    kr = atomicAdd(&bins[key], 1u);
                    OwnEntry& e = own_tab[threadIdx.x];
                    e.self = (uint16_t)self;
                    e.ovb = (uint16_t)ov.b;
                    e.ove = (uint16_t)ov.e;
                    e.r[0] = (uint16_t)w.j;
                    e.r[1] = (uint16_t)w.je;
                    e.r[2] = (uint16_t)w.j1;
                    e.r[3] = (uint16_t)w.e1;
                    e.r[4] = (uint16_t)w.j2;
                    e.r[5] = (uint16_t)w.e2;
                    e.slot = s;
                }
                __syncthreads();
                if (threadIdx.x < kSortBins) {  // exclusive scan of the class sizes (wave 0)
                    const uint32_t v = bins[threadIdx.x];
                    bins[threadIdx.x] = wave_incl_scan(v) - v;
                }
                __syncthreads();
                if (threadIdx.x < n_own) ord[bins[key] + kr] = (uint8_t)threadIdx.x;
                __syncthreads();
                if (threadIdx.x < (n_own << lg)) {
                    const OwnEntry e = own_tab[ord[threadIdx.x >> lg]];
                    Walk3 w;
                    w.j = e.r[0];
                    w.je = e.r[1];
                    w.j1 = e.r[2];
                    w.e1 = e.r[3];
                    w.j2 = e.r[4];
                    w.e2 = e.r[5];
                    w.left = 2;
                    agent_force<D, POT, MIXED, SENSE>(A, S, P, e.slot, e.self, src.record(e.self, w),
                                                      Span{e.ovb, e.ove}, w,
                                                      physical, symmetric, src, unit, MULTI ? threadIdx.x & gmask : 0u,
                                                      lg);
                }
                return;
            }
            for (uint32_t t = threadIdx.x; t < (n_own << lg); t += kBlock) {
                uint32_t self;
                Span ov;
                Walk3 w;
                const uint32_t s = own_agent(t >> lg, self, ov, w);
                agent_force<D, POT, MIXED, SENSE>(A, S, P, s, self, src.record(self, w), ov, w, physical, symmetric, src, unit,
                                                  MULTI ? t & gmask : 0u, lg);
            }
            return;
        }
    }
    // global path: own agents row by row, candidates voxel by voxel
    GlobalSource<D, MIXED> src{rec, G};
    for (uint32_t r = 0; r < R; r++) {
        const uint32_t b = T.b0 + r, base = voff + (T.a0 * n1 + b) * n2;
        const uint32_t sb = A.start[base + T.c0], se = A.start[base + T.c1];
        for (uint32_t s = sb + threadIdx.x; s < se; s += kBlock) {
            const uint32_t c = S.vox[s] - base;
            WalkVox w;
            w.start = A.start;
            w.voff = voff;
            w.n1 = n1;
            w.n2 = n2;
            w.a_lo = T.a0 == 0 || NP == 1 ? T.a0 : T.a0 - 1;
            w.b_lo = b == 0 ? 0 : b - 1;
            w.c_lo = c == 0 ? 0 : c - 1;
            w.na = (NP == 1 ? T.a0 + 1 : min(T.a0 + 2, n0)) - w.a_lo;
            w.nb = min(b + 2, n1) - w.b_lo;
            w.ncol = min(c + 2, n2) - w.c_lo;
            w.rb = w.cc = w.pa = 0;
            const uint32_t g0 = w.gvox();
            w.j = A.start[g0];
            w.je = A.start[g0 + 1];
            const Span ov{A.start[base + c], A.start[base + c + 1]};
            WalkVox wm = w;  // the own record: its voxel (a0, b, c) in region coordinates
            wm.pa = T.a0 - w.a_lo;
            wm.rb = b - w.b_lo;
            agent_force<D, POT, MIXED, SENSE>(A, S, P, s, s, src.record(s, wm), ov, w, physical, symmetric, src, unit);
        }
    }
}

// ---------------------------------------------------------------------------
// Integrator + boundary + next voxel.
// Ring semantics (chili/aux_storage.rs:41-130 with capacity = solver order):
// every step pushes (dx, dv) first, then reads the iterator (solvers.rs:178-186).
// t steps done before this one -> write slot t % cap; afterwards the ring holds
// min(t + 1, cap) entries, the oldest at slot (t + 1) % cap once full.
// ---------------------------------------------------------------------------
struct StepArgs {
    const double* noise;  // CRM_NOISE_BUFFER: this step's normals by agent index, else null
    uint64_t seed;
    double dt;
    double sqrt_dt;
    uint32_t noise_mode;
    uint32_t cap;           // solver order = ring capacity
    uint32_t newest_first;  // ring iteration order
    uint32_t pad;
};

template <int MECH, int D>
__device__ __forceinline__ void point_increment(const InstParams& P, const double* x, const double* v,
                                                const double* f, const double* z, bool have_noise, double dt,
                                                double sqrt_dt, double* dx, double* dv, double* dxr,
                                                double* dvr) {
#pragma unroll
    for (int k = 0; k < D; k++) dxr[k] = dvr[k] = 0.0;
    if constexpr (MECH == CRM_MECHANICS_NEWTON_DAMPED) {  // mechanics.rs:166-173
#pragma unroll
        for (int k = 0; k < D; k++) {
            dx[k] = v[k];
            dv[k] = f[k] / P.mass - P.damping * v[k];
        }
    } else if constexpr (MECH == CRM_MECHANICS_LANGEVIN) {  // mechanics.rs:434-463
#pragma unroll
        for (int k = 0; k < D; k++) {
            dx[k] = v[k];
            double dv1 = P.inv_mass * f[k];
            double dv2 = (-P.damping) * v[k];
            dv[k] = dv1 + dv2;
        }
        if (have_noise) {
#pragma unroll
            for (int k = 0; k < D; k++) dvr[k] = P.langevin_coeff * ((0.0 + sqrt_dt * z[k]) / dt);
        }
    } else {  // Brownian, mechanics.rs:336-357
#pragma unroll
        for (int k = 0; k < D; k++) {
            dx[k] = P.brownian_q * f[k];
            dv[k] = 0.0;
        }
        if (have_noise) {
#pragma unroll
            for (int k = 0; k < D; k++) dxr[k] = P.brownian_coeff * ((0.0 + sqrt_dt * z[k]) / dt);
        }
    }
}

// Ring bookkeeping for a step that starts after t completed steps.
struct Ring {
    uint32_t cap, wslot, n_read;
    uint32_t it[2];  // slots yielded by the iterator after the push
};

__device__ __forceinline__ Ring ring_at(uint64_t t, uint32_t cap, uint32_t newest_first) {
    Ring r;
    r.cap = cap;
    r.wslot = cap ? (uint32_t)(t % cap) : 0u;
    const uint32_t size = (uint32_t)min<uint64_t>(t + 1, cap);
    const uint32_t oldest = size < cap ? 0u : (uint32_t)((t + 1) % (cap ? cap : 1u));
    r.n_read = (cap == 2 && size == 2) ? 2u : 1u;
#pragma unroll
    for (int i = 0; i < 2; i++)
        r.it[i] = cap == 0 ? 0u
                           : (newest_first ? (oldest + size - 1 - i + 2 * cap) % cap : (oldest + i) % cap);
    return r;
}

// The ring of a point agent whose first push is at step b (0, or the step after
// it was inserted by a division, whose AuxStorage starts empty): the entries are
// the pushes of steps max(b, t + 1 - cap) .. t (ring_at(t) when b == 0).  The
// capacity is 0, 1 or 2, so the slot arithmetic is a parity.
__device__ __forceinline__ Ring ring_agent(uint64_t t, uint64_t b, uint32_t cap, uint32_t newest_first) {
    Ring r;
    r.cap = cap;
    r.wslot = cap == 2 ? (uint32_t)(t & 1u) : 0u;
    const uint32_t size = (uint32_t)min<uint64_t>(t - b + 1, cap);
    const uint32_t oldest = cap == 2 ? (uint32_t)((t + 1 - size) & 1u) : 0u;
    r.n_read = (cap == 2 && size == 2) ? 2u : 1u;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t q = newest_first ? oldest + size + 1u - (uint32_t)i : oldest + (uint32_t)i;
        r.it[i] = cap == 2 ? (q & 1u) : 0u;
    }
    return r;
}

// Standard normals of this agent and step (buffer or Philox).
template <int D>
__device__ __forceinline__ bool point_noise(const StepArgs& sa, uint32_t id, uint64_t t, double* z) {
    if (sa.noise_mode == CRM_NOISE_BUFFER && sa.noise) {
#pragma unroll
        for (int k = 0; k < D; k++) z[k] = sa.noise[(uint64_t)id * D + k];
        return true;
    }
    if (sa.noise_mode == CRM_NOISE_PHILOX) {
        double g[4];
        gaussian_pair(sa.seed, id, t, 0, g[0], g[1]);
        if (D > 2) gaussian_pair(sa.seed, id, t, 1, g[2], g[3]);
#pragma unroll
        for (int k = 0; k < D; k++) z[k] = g[k];
        return true;
    }
#pragma unroll
    for (int k = 0; k < D; k++) z[k] = 0.0;
    return false;
}

// One chili mechanics update of a point agent (solvers.rs:23-55,156-347 via
// local_mechanics_update, update_mechanics.rs:530-559) followed by
// apply_boundary (cartesian_cuboid_n.rs:594-631).  hist(i, dv) reads the value
// of the ring slot it[i] (never the slot written this step).  With
// WITH_VEL == false only the position is produced (the velocity, increments
// and, for NewtonDamped / Langevin, the noise do not influence it).
template <int D, int MECH, bool WITH_VEL, typename Hist>
__device__ __forceinline__ bool point_step(const InstParams& P, const StepArgs& sa, const Ring& rg, uint64_t t,
                                           uint32_t id, const double* x, const double* v, const double* f,
                                           Hist hist, double* nx, double* nv, double* dx, double* dv) {
    double z[D];
    const bool need_noise = WITH_VEL || MECH == CRM_MECHANICS_BROWNIAN;
    bool have_noise = false;
    if (need_noise) have_noise = point_noise<D>(sa, id, t, z);
    else {
#pragma unroll
        for (int k = 0; k < D; k++) z[k] = 0.0;
    }
    double dxr[D], dvr[D];
    point_increment<MECH, D>(P, x, v, f, z, have_noise, sa.dt, sa.sqrt_dt, dx, dv, dxr, dvr);
    if (rg.cap == 0) {  // euler, solvers.rs:302-310
#pragma unroll
        for (int k = 0; k < D; k++) {
            nx[k] = (dx[k] * sa.dt + x[k]) * 1.0 + dxr[k] * sa.dt;
            if (WITH_VEL) nv[k] = (dv[k] * sa.dt + v[k]) * 1.0 + dvr[k] * sa.dt;
        }
    } else if (rg.n_read == 2) {  // adams_bashforth_3, solvers.rs:312-329
        const double f0 = 23.0 / 12.0, f1 = (-16.0) / 12.0, f2 = 5.0 / 12.0;
#pragma unroll
        for (int k = 0; k < D; k++) {
            const double h0 = rg.it[0] == rg.wslot ? dx[k] : hist(0, k, false);
            const double h1 = rg.it[1] == rg.wslot ? dx[k] : hist(1, k, false);
            const double a = (dx[k] * f0 + (h0 * f1 + h1 * f2)) * sa.dt + x[k];
            nx[k] = a * 1.0 + dxr[k] * sa.dt;
            if (WITH_VEL) {
                const double g0 = rg.it[0] == rg.wslot ? dv[k] : hist(0, k, true);
                const double g1 = rg.it[1] == rg.wslot ? dv[k] : hist(1, k, true);
                const double b = (dv[k] * f0 + (g0 * f1 + g1 * f2)) * sa.dt + v[k];
                nv[k] = b * 1.0 + dvr[k] * sa.dt;
            }
        }
    } else {  // adams_bashforth_2, solvers.rs:331-347
        const double g0c = 3.0 / 2.0, g1c = (-1.0) / 2.0;
#pragma unroll
        for (int k = 0; k < D; k++) {
            const double h0 = rg.it[0] == rg.wslot ? dx[k] : hist(0, k, false);
            nx[k] = ((dx[k] * g0c + h0 * g1c) * sa.dt + x[k]) * 1.0 + dxr[k] * sa.dt;
            if (WITH_VEL) {
                const double q0 = rg.it[0] == rg.wslot ? dv[k] : hist(0, k, true);
                nv[k] = ((dv[k] * g0c + q0 * g1c) * sa.dt + v[k]) * 1.0 + dvr[k] * sa.dt;
            }
        }
    }
    if (WITH_VEL && MECH == CRM_MECHANICS_BROWNIAN) {
#pragma unroll
        for (int k = 0; k < D; k++) nv[k] = v[k];  // Brownian::set_velocity is a no-op
    }
    bool out = false;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const int ax = k + 3 - D;
        if (nx[k] < P.min[ax]) {
            nx[k] = 2.0 * P.min[ax] - nx[k];
            if (WITH_VEL) nv[k] = fabs(nv[k]);
        }
        if (nx[k] > P.max[ax]) {
            nx[k] = 2.0 * P.max[ax] - nx[k];
            if (WITH_VEL) nv[k] = -fabs(nv[k]);
        }
        out |= (nx[k] < P.min[ax]) || (nx[k] > P.max[ax]);
    }
    return out;
}

// Next voxel of every agent (get_index_of, cartesian_cuboid_n.rs:469-491) from
// the position it will have after this step.  A
// position whose index has no voxel keeps the old one (update_mechanics.rs:430-453).
template <int D, int MECH>
__global__ __launch_bounds__(kBlock) void k_key_point(Arrays A, StateBuf S, StepArgs sa) {
    if (halted(A.ctrl, A.ctrl->step)) return;
    const BlockWork w = A.work[blockIdx.x];
    if (threadIdx.x >= w.count) return;
    const uint64_t s = w.first + threadIdx.x;
    const InstParams& P = A.ip[w.inst];
    const uint64_t N = A.N;
    const uint64_t t = A.ctrl->step;
    const uint32_t id = S.id[s];
    const Ring rg = ring_agent(t, S.birth ? S.birth[s] : 0u, sa.cap, sa.newest_first);
    double x[D], v[D], f[D], nx[D], nv[D], dx[D], dv[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        x[k] = S.pos[k * N + s];
        v[k] = MECH == CRM_MECHANICS_BROWNIAN ? 0.0 : S.vel[k * N + s];
        f[k] = MECH != CRM_MECHANICS_BROWNIAN ? 0.0 : A.forcef ? (double)A.forcef[k * N + s] : A.force[k * N + s];
    }
    auto hist = [&](int i, int k, bool) { return S.hdx[((uint64_t)rg.it[i] * D + k) * N + s]; };
    const bool out = point_step<D, MECH, false>(P, sa, rg, t, id, x, v, f, hist, nx, nv, dx, dv);
    if (out) raise_error(A.ctrl, CRM_BOUNDARY_ERROR, t, id);
    uint32_t idx[3] = {0, 0, 0};
    bool ok = true;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const int ax = k + 3 - D;
        ok = ok && axis_index_fast(nx[k], P.min[ax], P.dx[ax], P.inv_dx[ax], P.n[ax], idx[ax]);
    }
    uint32_t key;
    if (ok) {
        key = P.voxel_offset + (idx[0] * P.n[1] + idx[1]) * P.n[2] + idx[2];
    } else {
        key = S.vox[s];
        atomicAdd((unsigned long long*)&A.ctrl->out_of_grid, 1ull);
    }
    A.key[s] = key;
    note_move(A.delta, A.head, A.link, (uint32_t)s, S.vox[s], key);
}

// Initial binning (Domain::decompose, concepts-derive/src/domain.rs:357-380 with
// get_voxel_index_of_raw, cartesian_cuboid_n.rs:320-337): min < p strictly and
// the voxel must exist; agents keep input order inside a voxel.
template <int D>
__global__ __launch_bounds__(kBlock) void k_initial_key(Arrays A, StateBuf S, uint32_t n_vertices) {
    const BlockWork w = A.work[blockIdx.x];
    if (threadIdx.x >= w.count) return;
    const uint64_t s = w.first + threadIdx.x;
    const InstParams& P = A.ip[w.inst];
    const uint64_t N = A.N;
    double p[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        if (n_vertices == 1) {
            p[k] = S.pos[k * N + s];
        } else {  // rod centroid: row_sum / nrows (bacterial_rods.rs:368-372)
            double acc = 0.0;
            for (uint32_t q = 0; q < n_vertices; q++) acc = acc + S.pos[((uint64_t)q * D + k) * N + s];
            p[k] = acc / (double)n_vertices;
        }
    }
    uint32_t idx[3] = {0, 0, 0};
    bool strict = true, ok = true;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const int ax = k + 3 - D;
        strict = strict && (P.min[ax] < p[k]);
        double xx = (p[k] - P.min[ax]) / P.dx[ax];
        bool conv = (xx > -1.0) && (xx < 4294967296.0);
        double tt = conv ? trunc(xx) : 0.0;
        uint32_t i = tt <= 0.0 ? 0u : (uint32_t)tt;
        ok = ok && conv && i < P.n[ax];
        idx[ax] = conv ? min(i, P.n[ax] - 1) : 0u;
    }
    if (!strict) raise_error(A.ctrl, CRM_BOUNDARY_ERROR, 0, S.id[s]);
    else if (!ok) raise_error(A.ctrl, CRM_INDEX_ERROR, 0, S.id[s]);
    const uint32_t key = P.voxel_offset + (idx[0] * P.n[1] + idx[1]) * P.n[2] + idx[2];
    A.key[s] = key;
    A.rank[s] = atomicAdd(&A.count[key], 1u);
}

// ---------------------------------------------------------------------------
// Counting sort by voxel (set-up sorts).
// ---------------------------------------------------------------------------
// Each thread scans kScanItems consecutive voxels of count + stay into their
// offsets inside the scan tile (start_local) and clears count for the next sort's
// ranks; whole groups move as two 16-byte loads per array and two 16-byte stores
// (count, stay and start_local are 256-byte aligned and a group starts at a
// multiple of 8 voxels).  bsum[tile] = the tile's sum.
__global__ __launch_bounds__(kBlock) void k_scan_local(uint32_t* __restrict__ count,
                                                        const uint32_t* __restrict__ stay,
                                                        uint32_t* __restrict__ start_local, uint32_t* __restrict__ bsum,
                                                        uint32_t Vt, Control* ctrl) {
    const bool skip = halted(ctrl, ctrl->step);
    // for the sort's later kernels (no block of this one reads it)
    if (blockIdx.x == 0 && threadIdx.x == 0) ctrl->skip = skip ? 1u : 0u;
    if (skip) return;
    static_assert(kScanItems == 8, "two uint4 per group");
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    const bool whole = base + kScanItems <= Vt;
    uint32_t vals[kScanItems];
    if (whole) {
        uint4* c4 = reinterpret_cast<uint4*>(count + base);
        const uint4* s4 = reinterpret_cast<const uint4*>(stay + base);
        const uint4 c0 = c4[0], c1 = c4[1], s0 = s4[0], s1 = s4[1];
        vals[0] = c0.x + s0.x;
        vals[1] = c0.y + s0.y;
        vals[2] = c0.z + s0.z;
        vals[3] = c0.w + s0.w;
        vals[4] = c1.x + s1.x;
        vals[5] = c1.y + s1.y;
        vals[6] = c1.z + s1.z;
        vals[7] = c1.w + s1.w;
        c4[0] = make_uint4(0u, 0u, 0u, 0u);
        c4[1] = make_uint4(0u, 0u, 0u, 0u);
    } else {
#pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            const uint64_t q = base + i;
            vals[i] = q < Vt ? count[q] + stay[q] : 0u;
            if (q < Vt) count[q] = 0u;
        }
    }
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) sum += vals[i];
    uint32_t total;
    uint32_t run = block_exclusive_scan(sum, total);
    uint32_t out[kScanItems];
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        out[i] = run;
        run += vals[i];
    }
    if (whole) {
        uint4* o4 = reinterpret_cast<uint4*>(start_local + base);
        o4[0] = make_uint4(out[0], out[1], out[2], out[3]);
        o4[1] = make_uint4(out[4], out[5], out[6], out[7]);
    } else {
#pragma unroll
        for (int i = 0; i < kScanItems; i++)
            if (base + i < Vt) start_local[base + i] = out[i];
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

// Single block: exclusive scan of the tile sums in place (the tile offsets), for
// grids of more than kScatterTiles scan tiles.
__global__ __launch_bounds__(kBlock) void k_scan_tiles(uint32_t* __restrict__ bsum, uint32_t n_tiles,
                                                        const Control* ctrl) {
    if (ctrl->skip) return;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < n_tiles; base += kBlock) {
        uint32_t q = base + threadIdx.x;
        uint32_t x = q < n_tiles ? bsum[q] : 0u;
        uint32_t total;
        uint32_t ex = block_exclusive_scan(x, total);
        if (q < n_tiles) bsum[q] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) bsum[n_tiles] = carry;
}

// Thread g writes the final start of voxel g (tile-local offset + tile offset) and
// places agent g in the slot list of its next voxel: a stayer at its rank, an
// arrival (kMoved) after the voxel's stayers in atomic order.  Launched over
// max(N, Vt) threads.  Thread 0 writes start[Vt].
// SCAN: every workgroup scans the tile sums itself (two per thread): one more dependent
// load and two barriers in place of k_scan_tiles, a 4.5 us launch in a chain of small
// kernels.  The scatter stays at 4.7 us for 30,000 and 4.9 for 300,000 agents and goes
// from 6.0 to 7.5 for 1M in 432 tiles; with 1728 tiles per workgroup it lost more than
// the launch, hence the line at two per thread.
constexpr uint32_t kScatterTiles = 512;
template <bool SCAN>
__global__ __launch_bounds__(kBlock) void k_scatter(Arrays A, uint32_t n_tiles) {
    if (A.ctrl->skip) return;
    __shared__ uint32_t s_off[SCAN ? kScatterTiles : 1];
    uint32_t total = 0;
    const uint32_t* off = A.tile_off;
    if constexpr (SCAN) {
        const uint32_t q = 2u * threadIdx.x;
        const uint32_t x = q < n_tiles ? A.tile_off[q] : 0u, y = q + 1u < n_tiles ? A.tile_off[q + 1u] : 0u;
        const uint32_t ex = block_exclusive_scan(x + y, total);
        s_off[q] = ex;
        s_off[q + 1u] = ex + x;
        __syncthreads();
        off = s_off;
    }
    const uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g == 0) A.start[A.Vt] = SCAN ? total : A.tile_off[n_tiles];
    if (g < A.Vt) A.start[g] = A.start_local[g] + off[g / kScanTile];
    if (g >= A.N) return;
    const uint32_t k = A.key[g], r = A.rank[g];
    const uint32_t pos = (r & kMoved) ? A.stay[k] + (r & ~kMoved) : r;
    A.perm[A.start_local[k] + off[k / kScanTile] + pos] = (uint32_t)g;
}

// Small systems (every voxel in one scan tile, at most kSmallSortAgents agents):
// k_scan_local, k_scan_tiles and k_scatter in one workgroup, with barriers in place
// of the launches between them; the voxel starts stay in LDS for the scatter.  The
// same skip flag, count reset, starts, start[Vt] and slot lists.
constexpr uint32_t kSmallSortAgents = 16384;
__global__ __launch_bounds__(kBlock) void k_sort_small(Arrays A) {
    static_assert(kScanItems == 8, "eight voxels per thread");
    __shared__ uint32_t s_start[kScanTile];
    const bool skip = halted(A.ctrl, A.ctrl->step);
    __syncthreads();  // every thread has read the control block before thread 0 writes it
    if (threadIdx.x == 0) A.ctrl->skip = skip ? 1u : 0u;
    if (skip) return;
    const uint32_t Vt = A.Vt, base = threadIdx.x * kScanItems;
    uint32_t vals[kScanItems], sum = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        const uint32_t q = base + i;
        vals[i] = q < Vt ? A.count[q] + A.stay[q] : 0u;
        if (q < Vt) A.count[q] = 0u;
        sum += vals[i];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan(sum, total);
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        const uint32_t q = base + i;
        if (q < Vt) {
            s_start[q] = run;
            A.start[q] = run;
        }
        run += vals[i];
    }
    if (threadIdx.x == 0) A.start[Vt] = total;
    __syncthreads();
    for (uint32_t g = threadIdx.x; g < (uint32_t)A.N; g += kBlock) {
        const uint32_t k = A.key[g], r = A.rank[g];
        const uint32_t pos = (r & kMoved) ? A.stay[k] + (r & ~kMoved) : r;
        A.perm[s_start[k] + pos] = g;
    }
}

// Orders each voxel's arrivals by previous slot (atomic arrival order is not
// deterministic).  The resulting list is the reference's: the cells that stay keep
// their order and the movers are appended in order of old voxel, then old position
// (sort_cells_in_voxels_step_1/2, update_mechanics.rs:418-513).  Set-up sorts rank
// every agent atomically with stay = 0 and get the whole voxel in order of previous
// slot.
__global__ __launch_bounds__(kBlock) void k_fixup(Arrays A) {
    if (A.ctrl->skip) return;
    const uint64_t v = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (v >= A.Vt) return;
    // the stayers hold [b, b + stay) in their old order; the arrivals follow, put in
    // order of previous slot, i.e. of (old voxel, old position)
    const uint32_t m = A.start[v] + A.stay[v], e = A.start[v + 1];
    for (uint32_t i = m + 1; i < e; i++) {
        uint32_t x = A.perm[i];
        uint32_t j = i;
        while (j > m) {
            uint32_t y = A.perm[j - 1];
            if (y <= x) break;
            A.perm[j] = y;
            j--;
        }
        A.perm[j] = x;
    }
}

// Force record of slot s: absolute double coordinates (FP64), or 30-bit fixed
// point relative to the voxel origin (mixed; the sign bit of w flags an agent
// outside its voxel's fixed-point range, which sends its pairs to the FP64 path).
template <int D, bool MIXED>
__device__ __forceinline__ void write_record(const Arrays& A, const InstParams& P, uint64_t s, uint32_t key,
                                             const double* p, int32_t sp) {
    if constexpr (MIXED) {
        const uint32_t lv = key - P.voxel_offset;
        uint32_t idx[3];
        const uint32_t row = udiv_by_inv(lv, P.n[2], P.inv_n2);  // lv / n2
        idx[2] = lv - row * P.n[2];
        idx[0] = udiv_by_inv(lv, P.n[2] * P.n[1], P.inv_n12);
        idx[1] = row - idx[0] * P.n[1];
        int q[3] = {0, 0, 0};
        uint32_t outside = 0;
#pragma unroll
        for (int k = 0; k < D; k++) {
            const int ax = k + 3 - D;
            const double origin = P.min[ax] + (double)idx[ax] * P.dx[ax];
            const double tq = floor((p[k] - origin) * P.qinv[ax]);
            const bool ok = tq >= 0.0 && tq < (double)kQOne;  // false for NaN
            q[k] = ok ? (int)tq : (tq < 0.0 ? 0 : kQOne - 1);
            outside |= ok ? 0u : 1u;
        }
        const uint32_t w = ((uint32_t)sp & kSpeciesMask) | ((idx[2] & kColMask) << kColShift) | (outside << 31);
        A.recq[s] = make_int4(q[0], q[1], D == 3 ? q[2] : 0, (int)w);
    } else {
        A.rec64[s] = make_double4(p[0], p[1], D == 3 ? p[D - 1] : 0.0, (double)sp);
    }
}

// Next voxel of the agent in slot s for the step that starts after t1 steps,
// from its state at that point: position x, velocity v and the ring slots r0 /
// r1 of position increments.  For NewtonDamped and Langevin the position update
// depends on neither the force nor the noise, so the re-binning of step t1 is
// known once step t1 - 1 has been integrated (k_key_point computes the same
// position).  A position whose index has no voxel keeps `vox`.
template <int D, int MECH>
__device__ __forceinline__ void bin_ahead(const Arrays& A, const InstParams& P, const StepArgs& sa, uint64_t t1,
                                          uint32_t id, uint64_t s, const double* x, const double* v,
                                          const double* r0, const double* r1, uint32_t vox, uint64_t birth) {
    const Ring rg = ring_agent(t1, birth, sa.cap, sa.newest_first);
    double f[D], nx[D], nv[D], dx[D], dv[D];
#pragma unroll
    for (int k = 0; k < D; k++) f[k] = 0.0;
    auto hist = [&](int i, int k, bool) { return rg.it[i] ? r1[k] : r0[k]; };
    point_step<D, MECH, false>(P, sa, rg, t1, id, x, v, f, hist, nx, nv, dx, dv);
    uint32_t idx[3] = {0, 0, 0};
    bool ok = true;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const int ax = k + 3 - D;
        ok = ok && axis_index_fast(nx[k], P.min[ax], P.dx[ax], P.inv_dx[ax], P.n[ax], idx[ax]);
    }
    uint32_t key = vox;
    if (ok) key = P.voxel_offset + (idx[0] * P.n[1] + idx[1]) * P.n[2] + idx[2];
    else atomicAdd((unsigned long long*)&A.ctrl->out_of_grid, 1ull);
    A.key_next[s] = key;
    note_move(A.delta, A.head_next, A.link_next, (uint32_t)s, vox, key);
}

// Ranks of a set-up sort whose agents are in voxel order already (insertion, the rods'
// cycle), with an atomic only for agents that change voxel.  Thread per voxel v of the
// current order: the agents of v that stay get consecutive ranks in slot order and
// their number goes to stay[v]; the others take an atomic rank among the arrivals of
// their next voxel (count), flagged with kMoved, which the scatter places after that
// voxel's stayers; k_fixup puts the arrivals in order.
__global__ __launch_bounds__(kBlock) void k_rank_ahead(Arrays A) {
    if (halted(A.ctrl, A.ctrl->step)) return;
    const uint64_t v = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (v >= A.Vt) return;
    const uint32_t b = A.start[v], e = A.start[v + 1];
    uint32_t n = 0;
    for (uint32_t s = b; s < e; s++) {
        const uint32_t k = A.key[s];
        if (k == v) A.rank[s] = n++;
        else A.rank[s] = kMoved | atomicAdd(&A.count[k], 1u);
    }
    A.stay[v] = n;
}

// Permutes the state into sorted order and writes the force records, without
// integrating (initial placement).  The ring holds min(step, cap) increments.
// With AHEAD the next step's voxels are binned as well.
template <int D, bool MIXED, bool AHEAD, int MECH>
__global__ __launch_bounds__(kBlock) void k_gather_point(Arrays A, StateBuf src, StateBuf dst, StepArgs sa) {
    if (A.ctrl->skip) return;
    const BlockWork w = A.work[blockIdx.x];
    if (threadIdx.x >= w.count) return;
    const uint64_t s = w.first + threadIdx.x;
    const InstParams& P = A.ip[w.inst];
    const uint64_t N = A.N;
    const uint32_t o = A.perm[s];
    const uint64_t t = A.ctrl->step;
    const uint64_t birth = src.birth ? src.birth[o] : 0u;
    // every slot when agents hold rings of different fill (inserted daughters)
    const uint32_t n_hist = src.birth ? sa.cap : (uint32_t)min<uint64_t>(t, sa.cap);
    double p[D], v[D], r0[D], r1[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        p[k] = src.pos[k * N + o];
        v[k] = src.vel[k * N + o];
        dst.pos[k * N + s] = p[k];
        dst.vel[k * N + s] = v[k];
        r0[k] = r1[k] = 0.0;
    }
    for (uint32_t h = 0; h < n_hist; h++) {
#pragma unroll
        for (int k = 0; k < D; k++) {
            const double hx = src.hdx[((uint64_t)h * D + k) * N + o];
            dst.hdx[((uint64_t)h * D + k) * N + s] = hx;
            dst.hdv[((uint64_t)h * D + k) * N + s] = src.hdv[((uint64_t)h * D + k) * N + o];
            if (h == 0) r0[k] = hx;
            else r1[k] = hx;
        }
    }
    const int32_t sp = src.species[o];
    const uint32_t id = src.id[o];
    dst.species[s] = sp;
    dst.id[s] = id;
    const uint32_t key = A.key[o];
    dst.vox[s] = key;
    write_record<D, MIXED>(A, P, s, key, p, sp);
    if (dst.birth) dst.birth[s] = (uint32_t)birth;
    if constexpr (AHEAD) bin_ahead<D, MECH>(A, P, sa, t, id, s, p, v, r0, r1, key, birth);
}

// Gather + integrate: the thread of slot o computes its agent's update (the same
// point_step as in k_key_point, so the same position) and writes the new state to the
// agent's slot s in the next order, together with the force record for the next step.
// It runs at the memory's rate: the state is read in slot order, so the loads wait for
// no other load, and the slots written are those read, shifted by the few arrivals.
template <int D, bool MIXED, int MECH>
__global__ __launch_bounds__(kBlock) void k_gather_integrate_point(Arrays A, StateBuf src, StateBuf dst,
                                                                     StepArgs sa) {
    __shared__ uint32_t s_off[kStepScanTiles];
    const uint64_t t = A.ctrl->gather_step;
    const BlockWork w = A.work[blockIdx.x];
    if (halted(A.ctrl, t)) return;
    const InstParams& P = A.ip[w.inst];
    const uint64_t N = A.N;
    const Move m = move_of(A, src.vox, (uint32_t)w.first, w.count);
    const uint32_t key = m.k;
    const bool in_block = threadIdx.x < w.count;
    const uint32_t o = (uint32_t)w.first + min(threadIdx.x, w.count - 1u);
    const uint32_t sl = in_block ? A.start_local[key] : 0u, sl0 = first_start_local(A);
    const uint32_t id = src.id[o];
    const uint64_t birth = src.birth ? src.birth[o] : 0u;
    const Ring rg = ring_agent(t, birth, sa.cap, sa.newest_first);
    double x[D], v[D], f[D], nx[D], nv[D], dx[D], dv[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        x[k] = __builtin_nontemporal_load(&src.pos[k * N + o]);
        v[k] = __builtin_nontemporal_load(&src.vel[k * N + o]);
        if constexpr (MIXED) f[k] = (double)__builtin_nontemporal_load(&A.forcef[k * N + o]);
        else f[k] = __builtin_nontemporal_load(&A.force[k * N + o]);
    }
    // the ring before this step (min(t - birth, cap) entries: with cap <= 2 the
    // slot not overwritten now, once filled), in registers, except the slot this
    // step overwrites: point_step reads the new increment in its place
    const uint32_t n_old = (uint32_t)min<uint64_t>(t - birth, rg.cap);
    double hx[2][D], hv[2][D];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const bool live = (uint32_t)h < rg.cap && (uint32_t)h != rg.wslot && n_old > 0;
#pragma unroll
        for (int k = 0; k < D; k++) {
            const uint64_t e = ((uint64_t)h * D + k) * N + o;
            hx[h][k] = live ? __builtin_nontemporal_load(&src.hdx[e]) : 0.0;
            hv[h][k] = live ? __builtin_nontemporal_load(&src.hdv[e]) : 0.0;
        }
    }
    step_tile_offsets(A, s_off);
    if (in_block) {
        const uint64_t s = next_slot(A, s_off, o, m, sl);
        auto hist = [&](int i, int k, bool is_dv) {
            const bool second = rg.it[i] != 0u;
            return is_dv ? (second ? hv[1][k] : hv[0][k]) : (second ? hx[1][k] : hx[0][k]);
        };
        const bool out = point_step<D, MECH, true>(P, sa, rg, t, id, x, v, f, hist, nx, nv, dx, dv);
        if (out) raise_error(A.ctrl, CRM_BOUNDARY_ERROR, t, id);
#pragma unroll
        for (int k = 0; k < D; k++) {
            __builtin_nontemporal_store(nx[k], &dst.pos[k * N + s]);
            __builtin_nontemporal_store(nv[k], &dst.vel[k * N + s]);
        }
        // ring: the slot written this step gets (dx, dv).  The other slot's entry, which
        // the next step overwrites before it reads the ring, is carried over by the last
        // step of a call only (48 of 332 bytes per 3-D agent; a call that ends early at
        // an error gets it from k_carry_ring)
        if (rg.cap > 0) {
            const bool both = n_old > 0 && t >= A.ctrl->last_step;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const bool keep = (uint32_t)h < rg.cap && ((uint32_t)h == rg.wslot || both);
#pragma unroll
                for (int k = 0; k < D; k++) {
                    if (h == (int)rg.wslot) {
                        hx[h][k] = dx[k];
                        hv[h][k] = dv[k];
                    }
                    if (keep) {
                        const uint64_t e = ((uint64_t)h * D + k) * N + s;
                        __builtin_nontemporal_store(hx[h][k], &dst.hdx[e]);
                        __builtin_nontemporal_store(hv[h][k], &dst.hdv[e]);
                    }
                }
            }
        }
        const int32_t sp = src.species[o];
        dst.species[s] = sp;
        dst.id[s] = id;
        dst.vox[s] = key;
        write_record<D, MIXED>(A, P, s, key, nx, sp);
        if (dst.birth) dst.birth[s] = (uint32_t)birth;
        if constexpr (MECH != CRM_MECHANICS_BROWNIAN)
            bin_ahead<D, MECH>(A, P, sa, t + 1, id, s, nx, nv, hx[0], hx[1], key, birth);
    }
    finish_order(A, s_off, sl0, t);
}

// Agents that were put in a voxel their position is not in (inserted ones).
__global__ void k_note_out_of_grid(Control* c, uint64_t n) { c->out_of_grid += n; }

// Index of the last step of the call that is about to run.
__global__ void k_set_last_step(Control* c, uint64_t t) { c->last_step = t; }

// After a call that ended at an error before its last step t: the older ring entry of
// every agent, from the failing step's source buffer (the moves and the scan still hold
// that step's) to its destination.  K components per agent.
__global__ __launch_bounds__(kBlock) void k_carry_ring(Arrays A, StateBuf src, StateBuf dst, uint64_t t, uint32_t K) {
    __shared__ uint32_t s_off[kStepScanTiles];
    const uint32_t first = blockIdx.x * kBlock, count = (uint32_t)min<uint64_t>(kBlock, A.N - first);
    const Move m = move_of(A, src.vox, first, count);
    step_tile_offsets(A, s_off);
    if (threadIdx.x >= count) return;
    const uint32_t o = first + threadIdx.x;
    const uint64_t s = next_slot(A, s_off, o, m, A.start_local[m.k]);
    if (t <= (src.birth ? src.birth[o] : 0u)) return;  // no older entry
    const uint64_t h = 1u - (t & 1u);
    for (uint32_t k = 0; k < K; k++) {
        dst.hdx[(h * K + k) * A.N + s] = src.hdx[(h * K + k) * A.N + o];
        dst.hdv[(h * K + k) * A.N + s] = src.hdv[(h * K + k) * A.N + o];
    }
}

}  // namespace crm
