// libpd_hip: bond-based peridynamics time stepping for MI355X (gfx950).
//
// One fused kernel per time step (k_step): for every node i, every live bond
// (i, j) is tested for breaking and its force gathered into i; then the force
// boundary condition is added and the integrator update (Euler,
// Euler-Cromer or Velocity-Verlet) writes u (and ud, udd) of node i.  The
// positions r = r0 + u that neighbours gather are ping-ponged between two
// record arrays, so every bond of a step sees the positions at the start of
// the step (the break-before-force order of peripy/integrators.py:339-349 and
// the single bond_force pass of cl/peridynamics.cl both read u_n only).
//
// Tiles.  The nodes are cut into tiles of up to `tile_nodes` nodes by
// recursive bisection of their initial coordinates, such that a tile's halo
// -- the tile's nodes and all their neighbours -- fits in LDS (1280 entries,
// 80 KiB, so two workgroups share a CU and one stages its halo while the
// other computes).  Within a tile the nodes are ordered by descending bond
// count, so a wavefront's nodes run loops of nearly equal length.  One
// workgroup runs one tile: it first copies the halo's records into LDS with
// coalesced loads (each record once), then every bond gathers its neighbour
// from LDS.
// A direct global gather would fetch each 64-byte record with four 16-byte
// loads from 64 different records per instruction, and the vector L1 then
// handles one 64-byte sector per clock: that, not HBM, was the bound.
// Tiles are mapped to workgroups so that each XCD (blockIdx % 8) runs a
// contiguous range of tiles, whose halos overlap in that XCD's L2.
//
// Data layout in HBM (N nodes, S bond slots).  Every per-node array is kept
// in tile order: internal node p is node tnode[p] of the caller's numbering,
// a tile's nodes are a contiguous range of p, and a halo is a few contiguous
// runs, so per-node loads and stores coalesce.  Inputs are permuted into
// this order on upload and outputs back on download.
//   rec[2][N]  NodeRec, 64 bytes: (r0x, r0y, r0z, w | rx, ry, rz, v) with
//              r = r0 + u (compact layout) or r = u (slot layout, whose
//              stretch is formed from u), the bond loop's weights w (4kV for the scalar
//              model, 2V for a stiffness field c, V for n-linear models) and
//              v (2cV for a field, else 0); ping-pong, with r0, w and v
//              static in both.
//   tiles[T]   TileInfo: node range [node_off, node_off + nodes) of p, halo
//              range in halo[], first chunk of the tile's bond slots, chunk
//              rows.
//   tnode[N]   caller's node id of internal node p; halo: internal ids per
//              tile, in the order of their LDS entries (HaloSpread).
//   bond slots, in chunks of 4: chunk (c, l) of a tile with n nodes is
//              chunk_off + c*n + l and holds four bonds of its l-th node,
//              rows sorted ascending by j; a wavefront reads its nodes' c-th
//              chunks contiguously.  A tile has as many chunk rows as its
//              longest row needs (at least one); the step kernel's look-ahead
//              loads run past the last of them, into the next tile's rows or
//              the LOC_SLACK slots that loc, state and corr have at their end
//              (the adjoint kernel's stay at the last row).
//     loc   u16  16 * (1 + halo-local index of j), the LDS offset of the
//                record's first piece; 0: broken or empty (hot loop; entry 0
//                of a staged halo is a far node of weight 0)
//     gidx  i32  j, with bit 31 DEAD and bit 30 NEW (broken in this step,
//                compact layout) -- read only on breaks and exports
//     pos   u16  reference column of the slot (exports)
//     corr  f64, state u16 (16 * (bond type * nregimes + regime), of a broken
//                bond regime 0): optional
//   chunk0[N], stride[N]: node p's chunk 0 and its tile's node count, from
//              which slot_of gives the slot of its k-th bond
//   u, ud, udd, force, body_force (N,3) f64 in the reference's layout
//   flags[N]   bit d: displacement BC on DOF d; bit 3+d: force BC on DOF d
//   meta[N]    a node's row length and its flags in one word (k_step)
//   bcv, fbcv, dens (N,3) f64, read only for flagged DOFs / dynamic
//              integrators
//   rslot (N,K) u16 + n_neigh: the reference-layout list of the compact
//              (Cython) layout, in the caller's numbering, as the slot index
//              of each row position, maintained by in-kernel compaction;
//              nlist_ref (N,K) i32 holds the caller's rows, rebuilt from
//              rslot at export.
//
// Stretch arithmetic.  Compact layout (the Cython path): exactly
// spatial.pyx's (dr = r_j - r_i with r = r0 + u, l = sqrt((dr0^2 + dr1^2) +
// dr2^2), s = (l - l0)/l0), built without floating-point contraction, so l
// and l0 are bitwise those of the Cython code.  Slot layout (the OpenCL
// integrators): cl/peridynamics.cl:65-75's (xi = r0_j - r0_i, xi_eta =
// (u_j - u_i) + xi), the squared lengths contracted as
// fma(z, z, fma(x, x, y*y)) and the updates contracted, as the OpenCL
// compiler that wrote the reference's Euler-Cromer and Velocity-Verlet
// fixtures evaluated them.  The square roots use the correctly rounded
// rsq-Goldschmidt sequence that the compiler emits for sqrt(double), without
// its range scaling (taken only for q outside [2^-767, inf), where the
// library sqrt is called).  Its by-product h ~ 0.5/sqrt(q) (relative error
// ~5e-15) replaces the two divisions; a stretch within a relative 1e-10 of any
// threshold it is compared with is recomputed with the library's square roots
// and the IEEE division, so every break and regime decision equals the one
// made with the correctly rounded s.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <string>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../include/pd_hip.h"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg)
{
    g_err = msg;
    return code;
}

#define HIPCHK(call)                                                        \
    do {                                                                    \
        hipError_t e_ = (call);                                             \
        if (e_ != hipSuccess)                                               \
            return fail(PD_E_HIP, std::string(#call) + ": " +               \
                                      hipGetErrorString(e_));               \
    } while (0)

}  // namespace

// Error reporting for the library's other translation units.
int pd_fail(int code, const char *msg) { return fail(code, msg); }

namespace pdk {

constexpr uint32_t DEAD = 0x80000000u;
constexpr uint32_t NEWB = 0x40000000u;
constexpr uint32_t KEYM = 0x3FFFFFFFu;
constexpr unsigned short LOC_DEAD = 0;  // loc of a broken or empty slot
constexpr int MAX_NODES = 1 << 26;
constexpr double GUARD = 1e-10;
constexpr int MAX_TAB = 256;  // nbond_types * nregimes
constexpr int MAX_LPN = 8;
constexpr int XCDS = 8;
// Halo capacity of a tile: entries of 4 x 16 bytes, stored piece-major (piece
// q of entry e at byte q*16*cap + 16*e), so that one address register and
// immediate offsets reach all four pieces and random entries spread over all
// LDS banks.  4*16*cap bytes (plus the n-linear tables) stay within 80 KiB,
// which lets two workgroups share a CU's 160 KiB.
constexpr int LDS_CAP_PMB = 1280;
constexpr int LDS_CAP_NLIN = 1152;
constexpr unsigned LDS_BYTES = 81920;
// The narrow form of a halo (scalar stiffness, which has no use for a
// record's last double): piece 3 holds 8 bytes per entry, at half of the
// others' offset, and 960 entries take 53,760 bytes, the most (in the LDS's
// allocation steps of 1,280) that lets three workgroups share a CU.
constexpr int LDS_CAP_NARROW = 960;
constexpr unsigned LDS_BYTES_NARROW = 56u * LDS_CAP_NARROW;
// Slots that loc, state and corr are longer than the tiles need: the step
// kernel requests chunk rows up to two rounds ahead, at most 3 rounds of
// tile_nodes * lanes_per_node <= 1024 chunks past a tile's last.
constexpr size_t LOC_SLACK = 3 * 1024 * 4;

// damage models of the step kernel
constexpr int DM_PMB = 0;    // scalar stiffness
constexpr int DM_NLIN = 1;   // n-linear / composite tables
constexpr int DM_FIELD = 2;  // PMB with k_ij = (c_i + c_j)/2

struct alignas(64) NodeRec {
    double4 a;  // r0x, r0y, r0z, V
    double4 b;  // rx, ry, rz, c
};

struct TileInfo {
    int node_off, nodes, halo_off, halo;
    long long chunk_off;
    int nch, pad;
};

constexpr int STORE_U = 1, STORE_F = 2;

struct StepArgs {
    int K, ntiles, tiles_per_xcd;
    int integrator, layout, has_corr;
    unsigned absmask;  // 0x7fffffff: break on |s|; 0xffffffff: on s
    int nregimes, ntab;
    double dt, damping, s0h;
    double lim;  // bound of bond_fast's stretch test (n-linear: its sign)
    const NodeRec *rec_old;
    NodeRec *rec_new;
    const TileInfo *tiles;
    const int *tnode, *halo;
    const double *u;  // u_n (compact layout; the slot layout's is in rec_old)
    double *u_out;    // u_{n+1}: u itself, or the next slot of a replay
    // what this step stores of that which the next one does not read (a run
    // stores those of its last step): STORE_U u of the slot layout, whose
    // next step reads the record; STORE_F force, body_force and
    // Euler-Cromer's udd
    int store;
    double *ud, *udd, *force, *body_force;
    const double *bcv, *fbcv, *dens;
    const double *dens1;  // per-node density when all three DOFs share it
    const int *meta;      // row length | flags << 16
    unsigned short *loc;
    int *gidx;
    const double *corr;
    unsigned short *state;
    const double *k_tab, *s_tab, *pc_tab;
    unsigned short *rslot;  // compact layout: row position -> slot
    int *n_neigh;
    const double *cnode;  // node stiffness c (DM_FIELD)
    int *brk;  // if set: the step at which each slot's bond broke
    int step;  // index of this step (for brk)
    // exact-order step: lower-slot counts, upper-list lengths and the fold
    // lists (slot index << 16 | halo loc), the scalar stiffness, and the
    // stretches strictly between which a bond takes the fast evaluation
    const int *nlow;
    int *nup;
    unsigned *ford;
    double kx, xlo, xhi;
};

// Slot of a row's k-th bond.  Sixteen bonds take four chunks; chunk q of the
// four holds bonds 2q, 2q+1 and 8+2q, 8+2q+1 of them, so that four lanes that
// take the four chunks run the first eight bonds before the second, and a
// row that ends in the first eight leaves the second half of its last round
// empty for all of them.
__host__ __device__ __forceinline__ size_t slot_of(long long chunk0,
                                                   int stride, int k)
{
    const int chunk = ((k >> 4) << 2) + ((k >> 1) & 3);
    return (size_t)(chunk0 + (long long)chunk * stride) * 4 +
           (((k >> 2) & 2) | (k & 1));
}

// Index of position pos of a node's fold list (exact-order step): round
// pos/8, in which lane pos%4 takes positions pos%4 and 4 + pos%4 with one
// 8-byte load; chunk0 and stride as in slot_of (a tile's lists take the place
// of its slots, two rows of pairs for a row of chunks).
__host__ __device__ __forceinline__ size_t fold_of(long long tile_chunk0,
                                                   int stride, int l, int pos)
{
    const int row = ((pos >> 3) << 2) + (pos & 3);
    return 2 * (size_t)(2 * tile_chunk0 + (long long)row * stride + l) +
           ((pos >> 2) & 1);
}

// Chunk rows of a row of cnt bonds.
__host__ __device__ __forceinline__ int chunks_of(int cnt)
{
    const int half = ((cnt & 15) + 1) >> 1;
    return ((cnt >> 4) << 2) + (half < 4 ? half : 4);
}

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------

// A 16-byte piece as the compiler's own vector (an array of HIP's double2
// that is only copied through stays in scratch).
typedef double v2d __attribute__((ext_vector_type(2)));

// f(0), f(1), ..., f(N - 1) with constant arguments.
template <int N, typename F>
__device__ __forceinline__ void static_for(F f)
{
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// sqrt(q) rounded to nearest for q in [2^-767, inf): the rsq seed, one
// Goldschmidt step for (g ~ sqrt q, h ~ 0.5/sqrt q) and two residual
// corrections of g -- the sequence LLVM emits for llvm.sqrt.f64 on gfx9,
// minus the input scaling and the zero/infinity selects it needs outside
// that range.
// Both corrections are needed: before its rounding the first leaves up to
// 3/2 d^2 = 4.4e-29 (the seed's e is at most 6e-8, the step's d = 3/2 e^2), so
// that a root within 4e-13 ulp of the middle between two doubles may take the
// wrong one (8 of 4,023 squares built to lie 7e-15 to 5e-13 ulp off it did,
// and none with the second).  The second costs the step 4 of a bond's 51 issue
// slots: 233 -> 247 us on the 1,038,230-node beam, 38.4 -> 40.2 on 141,143
// nodes, 72.6 -> 74.1 with n-linear tables on 263,407.
__device__ __forceinline__ void sqrt_core(double q, double &g, double &h)
{
    const double y = __builtin_amdgcn_rsq(q);
    g = q * y;
    h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    double d = __builtin_fma(-g, g, q);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, q);
    g = __builtin_fma(d, h, g);
}

__device__ __forceinline__ bool core_range(double q)
{
    return (q >= 0x1p-767) & (q < __builtin_inf());
}

// |x| (mask 0x7fffffff) or x (mask 0xffffffff): clears the sign bit or not
__device__ __forceinline__ double sign_mask(double x, unsigned mask)
{
    return __hiloint2double((int)((unsigned)__double2hiint(x) & mask),
                            __double2loint(x));
}

__device__ __forceinline__ uint32_t ld_slot(const int *p)
{
    return (uint32_t)__hip_atomic_load(p, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
}

// --- compaction of the compact (Cython) layout's rows -----------------------
//
// rslot (N, K) u16, rows in the caller's numbering: position p < n_neigh[m]
// of node m's reference-layout row holds the index of the slot (of m's
// internal node) whose bond it lists, so the row's entries are those slots'
// keys.  Positions from n_neigh[m] up to the row's count at set-up keep the
// values that swap-with-last left there, as the reference's rows do; the
// caller's row is rebuilt from rslot and gidx at export (k_export_rows).
//
// What peridynamics.pyx:124-156 (break_bonds) does to row i in one pass:
// first every node k < i whose bond to i broke removes itself from i's row by
// swap-with-last, in ascending k (the outer loop order of break_bonds), then
// i's own sweep replaces each broken j > i by the last entry without
// advancing.  All of it depends only on row i and on which of node i's bonds
// broke this step (its NEW slots).  Slots are sorted by key, so the lower
// neighbours are slots [0, nlow) and the upper ones [nhi, cnt).

__device__ __forceinline__ int slot_key(const int *gidx, long long c0,
                                        int stride, int k)
{
    return (int)(ld_slot(&gidx[slot_of(c0, stride, k)]) & KEYM);
}

// One node's row rs[0, n) in LDS, fl[k] = 1 for its slots that broke this
// step; i is the node's caller id (slot keys are caller ids).  Applies
// break_bonds' removals and returns the new count; nhi is set to the first
// slot whose key exceeds i.
__device__ __forceinline__ int compact_rows_seq(const int *gidx, long long c0,
                                             int stride, int cnt, int nlow,
                                             uint32_t i, unsigned short *rs,
                                             const unsigned char *fl, int n,
                                             int &nhi_out)
{
    int nhi = nlow;
    while (nhi < cnt && slot_key(gidx, c0, stride, nhi) == (int)i)
        ++nhi;
    nhi_out = nhi;
    for (int k = 0; k < nlow; ++k) {
        if (!fl[k])
            continue;
        // slots [kl, kh] repeat k's key; the reference removes the first
        // position holding that key
        const int j = slot_key(gidx, c0, stride, k);
        int kl = k, kh = k;
        while (kl > 0 && slot_key(gidx, c0, stride, kl - 1) == j)
            --kl;
        while (kh + 1 < nlow && slot_key(gidx, c0, stride, kh + 1) == j)
            ++kh;
        int p = 0;
        while (p < n && (rs[p] < kl || rs[p] > kh))
            ++p;
        if (p == n)
            continue;
        if (rs[p] != k) {
            // a repeat: the position that held slot k keeps the key, with
            // the slot that stays live
            int p2 = p + 1;
            while (p2 < n && rs[p2] != k)
                ++p2;
            if (p2 < n)
                rs[p2] = rs[p];
        }
        rs[p] = rs[n - 1];
        --n;
    }
    int rem = 0;
    for (int k = nhi; k < cnt; ++k)
        rem += fl[k];
    int p = 0;
    while (rem > 0 && p < n) {
        const int k = rs[p];
        if (k >= nhi && fl[k]) {
            rs[p] = rs[n - 1];
            --n;
            --rem;
        } else {
            ++p;
        }
    }
    return n;
}

// LDS one node's row takes in compact_tile (u16 positions, u8 break flags);
// the scratch also holds 64 bytes of counts.
__host__ __device__ constexpr unsigned compact_row_bytes(int K)
{
    return (3u * (unsigned)K + 15u) & ~15u;
}

// Every thread of the block calls this after its bond loop, with nbroken the
// node's count of bonds broken in this step (the same in all its lanes).  The
// rows of the nodes that lost bonds are staged in `scratch` (`bytes` of LDS
// the block no longer reads once every thread is here), compacted by one
// lane each, and written back; with EXACT, the upper part of the node's fold
// list (ford, nup) is rebuilt in the new row order.  NEW flags are cleared.  Nodes take
// scratch regions in groups when they do not all fit.  The first 64 bytes
// hold each wave's count of such nodes, from which every node's region
// follows without atomics.
template <int LPN, bool EXACT>
__device__ void compact_tile(const StepArgs &a, const TileInfo &ti,
                             char *scratch, unsigned bytes, bool valid,
                             int l, int sub, uint32_t i, int cnt, int nbroken)
{
    const bool mine = valid && nbroken > 0;
    __syncthreads();  // every bond loop is done: the scratch is free
    const unsigned long long bm = __ballot(mine && sub == 0);
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    int *ctr = reinterpret_cast<int *>(scratch);
    if (lane == 0)
        ctr[w] = __popcll(bm);
    __syncthreads();
    int total = 0, rank = 0;
    for (int v = 0; v < (int)(blockDim.x >> 6); ++v) {
        const int c = ctr[v];
        total += c;
        rank += v < w ? c : 0;
    }
    if (total == 0)
        return;  // the same in every thread
    rank += __popcll(bm & ((1ull << lane) - 1ull));
    rank = __shfl(rank, 0, LPN);  // the node's first lane holds its rank
    const int K = a.K;
    const unsigned nb = compact_row_bytes(K);
    const int G = (int)((bytes - 64u) / nb);
    if (G < 1)
        return;  // rows too wide: rejected by the host before any launch
    const long long c0 = ti.chunk_off + l;
    const uint32_t m = mine ? (uint32_t)a.tnode[i] : 0u;
    unsigned short *R = a.rslot + (size_t)m * K;
    for (int g0 = 0; g0 < total; g0 += G) {
        const bool act = mine && rank >= g0 && rank < g0 + G;
        unsigned short *rs = reinterpret_cast<unsigned short *>(
            scratch + 64u + (unsigned)(act ? rank - g0 : 0) * nb);
        unsigned char *fl = reinterpret_cast<unsigned char *>(rs + K);
        int n = 0;
        if (act) {
            n = a.n_neigh[m];
            for (int p = sub; p < n; p += LPN)
                rs[p] = R[p];
            for (int k = sub; k < cnt; k += LPN) {
                int *q = &a.gidx[slot_of(c0, ti.nodes, k)];
                const uint32_t e = ld_slot(q);
                fl[k] = (e & NEWB) ? 1 : 0;
                if (e & NEWB)
                    *q = (int)(e & ~NEWB);
            }
        }
        __syncthreads();
        if (act && sub == 0) {
            int nhi = 0;
            // keys are caller ids: the node's own is m
            const int n1 = compact_rows_seq(a.gidx, c0, ti.nodes, cnt,
                                            a.nlow[i], m, rs, fl, n, nhi);
            a.n_neigh[m] = n1;
            if (EXACT) {
                int pos = a.nlow[i];
                const int end = pos + a.nup[i];
                for (int p = 0; p < n1; ++p) {
                    const int k = rs[p];
                    if (k >= nhi)
                        a.ford[fold_of(ti.chunk_off, ti.nodes, l, pos++)] =
                            ((unsigned)k << 16) |
                            a.loc[slot_of(c0, ti.nodes, k)];
                }
                a.nup[i] = pos - a.nlow[i];
                for (; pos < end; ++pos)
                    a.ford[fold_of(ti.chunk_off, ti.nodes, l, pos)] =
                        LOC_DEAD;
            }
        }
        __syncthreads();
        if (act)
            for (int p = sub; p < n; p += LPN)
                R[p] = rs[p];
        __syncthreads();  // the next group reuses the scratch
    }
}

// ---------------------------------------------------------------------------
// the step kernel
// ---------------------------------------------------------------------------

template <int DM, bool NARROW = false>
constexpr unsigned piece_bytes()
{
    return 16u * (NARROW ? LDS_CAP_NARROW
                         : (DM == DM_NLIN ? LDS_CAP_NLIN : LDS_CAP_PMB));
}

// Where the halo begins in LDS: after the n-linear tables (two of MAX_TAB
// 16-byte entries), so that every read of the bond loop has an immediate
// offset below 2^16.
template <int DM>
constexpr unsigned halo_base()
{
    return DM == DM_NLIN ? 2u * 16u * MAX_TAB : 0u;
}

// Squared length of (x, y, z): spatial.pyx's ((x*x + y*y) + z*z), uncontracted
// (CLA false), or cl/peridynamics.cl:72-73's as contracted,
// fma(z, z, fma(x, x, y*y)) (CLA true).
template <bool CLA>
__device__ __forceinline__ double sq3(double x, double y, double z)
{
    if (CLA)
        return __builtin_fma(z, z, __builtin_fma(x, x, y * y));
    return (x * x + y * y) + z * z;
}

// Staging of a tile's halo records into LDS, piece-major: piece q of the
// record of entry x at D + q*PB + 16*(x + 1).  Thread t copies piece t%4 of
// entries t/4, t/4 + blockDim/4, ...; the node indices are requested as early
// as possible (they head the longest chain of dependent loads), the records
// SP pieces per thread in flight at once (a block of 512 threads needs one
// pass).  Pieces past the last entry store that entry again: a condition
// would move each load next to its store.
template <bool NARROW = false>
struct HaloLoads {
    // passes of all threads over the entries: SP at once (all of a narrow
    // halo's in a block of 512); a halo that needs at most FEW (a plate's)
    // stages no more
    static constexpr int SP = NARROW ? 8 : 10, FEW = 3;
    unsigned hi[SP];

    // byte offsets into H: four times the entry
    static __device__ __forceinline__ unsigned step()
    {
        return blockDim.x & ~3u;
    }

    __device__ __forceinline__ void request(const int *H, unsigned halo)
    {
        const char *h = reinterpret_cast<const char *>(H);
        const unsigned last = 4u * (halo - 1u);
        unsigned x = threadIdx.x & ~3u;
        static_for<SP>([&](auto k) {
            hi[k] = *reinterpret_cast<const unsigned *>(h + min(x, last));
            x += step();
        });
    }

    // this thread's piece of an entry, 4 e bytes of H in, into LDS
    static __device__ __forceinline__ void put(char *D, unsigned x, v2d v)
    {
        if (NARROW && (threadIdx.x & 3u) == 3u)
            *reinterpret_cast<double *>(D + 2u * x) = v.x;
        else
            *reinterpret_cast<v2d *>(D + 4u * x) = v;
    }

    // passes [0, N), their indices in hi
    template <int N>
    __device__ __forceinline__ void pass(const char *R, unsigned last,
                                         char *D) const
    {
        v2d v[N];
        static_for<N>([&](auto k) {
            v[k] = *reinterpret_cast<const v2d *>(
                R + (hi[k] * 64u + (threadIdx.x & 3u) * 16u));
        });
        unsigned x = threadIdx.x & ~3u;
        static_for<N>([&](auto k) {
            put(D, min(x, last), v[k]);
            x += step();
        });
    }

    // SHORT: with the short form for few passes (401 x 233 plate 14.4 -> 13.1
    // us a step; the n-linear kernel leaves it out, whose bars it costs 3 %)
    template <bool SHORT>
    __device__ __forceinline__ void stage(const NodeRec *rec, const int *H,
                                          unsigned halo, char *D, unsigned PB)
    {
        const char *h = reinterpret_cast<const char *>(H);
        const unsigned last = 4u * (halo - 1u);
        const unsigned piece = threadIdx.x & 3u;
        const char *R = reinterpret_cast<const char *>(rec);
        D += piece * PB + (NARROW && piece == 3u ? 8u : 16u);
        if (SHORT && last < FEW * step()) {
            pass<FEW>(R, last, D);
            return;
        }
        pass<SP>(R, last, D);
        const unsigned e0 = threadIdx.x & ~3u;
        for (unsigned x = e0 + SP * step(); x - e0 <= last;) {
            v2d v[4];  // the loop's trips are the same in every thread
            unsigned y = x;
            static_for<4>([&](auto k) {
                const unsigned g =
                    *reinterpret_cast<const unsigned *>(h + min(y, last));
                v[k] = *reinterpret_cast<const v2d *>(
                    R + (g * 64u + piece * 16u));
                y += step();
            });
            static_for<4>([&](auto k) {
                put(D, min(x, last), v[k]);
                x += step();
            });
        }
    }
};

// Entry 0 of a staged halo, what dead and empty slots read: a far node of
// weight 0 (CLA: records hold u, which is 0).  Threads 0-3.
template <bool CLA, bool NARROW = false>
__device__ __forceinline__ void far_entry(char *D, unsigned PB)
{
    constexpr double FAR = 0x1p300;
    const unsigned t = threadIdx.x;
    const bool r = t < 2 || !CLA;
    const double2 v = make_double2(r ? FAR : 0.0, r && !(t & 1) ? FAR : 0.0);
    if (NARROW && t == 3)
        *reinterpret_cast<double *>(D + t * PB) = v.x;
    else
        *reinterpret_cast<double2 *>(D + t * PB) = v;
}

// v of the lane whose number differs in bit OFF (1, 2 or 4).  Inside a quad
// the exchange is a DPP move of each half: no LDS access to wait for.
template <int OFF>
__device__ __forceinline__ int lane_xor(int v)
{
    if constexpr (OFF == 1)
        return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);
    else if constexpr (OFF == 2)
        return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);
    else
        return __shfl_xor(v, OFF, 2 * OFF);
}

template <int OFF>
__device__ __forceinline__ double lane_xor(double v)
{
    return __hiloint2double(lane_xor<OFF>(__double2hiint(v)),
                            lane_xor<OFF>(__double2loint(v)));
}

// Sum over a node's LPN lanes, the same in each: v + (v of lane ^ LPN/2),
// then ^ LPN/4, ...
template <int LPN, typename T>
__device__ __forceinline__ T node_sum(T v)
{
    if constexpr (LPN >= 8)
        v += lane_xor<4>(v);
    if constexpr (LPN >= 4)
        v += lane_xor<2>(v);
    if constexpr (LPN >= 2)
        v += lane_xor<1>(v);
    return v;
}

// A bond as the force needs it: the bond vector, s/2, 0.5/l and the weight;
// and the lengths that s/2 came from (for k_bond_check).
struct Bond {
    double dx, dy, dz, sh, hl, w, l, l0;
};

// The model's halved thresholds with a margin of GUARD: a stretch strictly
// inside (lo, hi) is away from every threshold and from lengths outside
// sqrt_core's range, so the bond neither breaks nor changes its regime.
// Anything else, NaN included, goes through bond_exact.
//
// Why the lengths need no test of their own: coordinates are zero or in
// [2^-290, 2^300] (else the host sets hi so that every bond takes the exact
// path), so q0 is 0 (its core value is NaN) or at least 2^-686 and below
// 2^603.  s/2 > -1/4 then means l > l0/2, so q is at least 2^-690, and a q
// that is infinite, NaN or 0 gives a NaN; a q in between but below the
// core's range gives an l of at most 2^-383, whose s/2 is -1/2.

// Compile-time switches of the step kernel, so that the common runs spend no
// instruction on what they do not use: CORR, the per-slot stiffness
// corrections multiply the force (bond_force2/4); TENS, a PMB bond breaks on
// !(s < s0) (cl/peridynamics.cl:78) instead of !(|s| < s0)
// (peridynamics.pyx:133); CLA, the OpenCL stretch (records hold u; the bond
// vector is (u_j - u_i) + xi) instead of the Cython one (records hold
// r0 + u; the bond vector is r_j - r_i).

// The fast evaluation of the bond to halo entry `ev` (byte offset of its
// piece 0); for DM_NLIN st is the byte offset of the bond's (type, regime) in
// the LDS tables.  Returns whether the result stands.
//
// A dead or empty slot (ev 0) needs no test here: entry 0 is a node at
// (2^300, 2^300, 2^300) of weight 0, so that l == l0 and the force is zero.
// lim: a.lim, or -1 where no bond of the node's may stand.
template <int DM, bool TENS, bool CLA, bool NARROW>
__device__ __forceinline__ bool bond_fast(const char *ldsb,
                                          const double4 &r0i,
                                          const double4 &ri, double ci,
                                          double lim, unsigned ev, unsigned st,
                                          Bond &o, double &kb, double &pb)
{
    constexpr unsigned PB = piece_bytes<DM, NARROW>();
    const char *pe = ldsb + halo_base<DM>() + ev;
    const double2 p0 = *reinterpret_cast<const double2 *>(pe);
    const double2 p1 = *reinterpret_cast<const double2 *>(pe + PB);
    const double2 p2 = *reinterpret_cast<const double2 *>(pe + 2 * PB);
    // c_j is read only by the node-field model
    double2 p3;
    if (DM == DM_FIELD) {
        p3 = *reinterpret_cast<const double2 *>(pe + 3 * PB);
    } else {
        p3.x = *reinterpret_cast<const double *>(
            NARROW ? ldsb + 3 * PB + (ev >> 1) : pe + 3 * PB);
        p3.y = 0.0;
    }
    const double ex = p0.x - r0i.x;
    const double ey = p0.y - r0i.y;
    const double ez = p1.x - r0i.z;
    if (CLA) {
        // cl/peridynamics.cl:65-71: xi_eta = (u_j - u_i) + xi
        o.dx = (p2.x - ri.x) + ex;
        o.dy = (p2.y - ri.y) + ey;
        o.dz = (p3.x - ri.z) + ez;
    } else {
        // spatial.pyx:20-31 with r = r0 + u: dr = r_j - r_i
        o.dx = p2.x - ri.x;
        o.dy = p2.y - ri.y;
        o.dz = p3.x - ri.z;
    }
    const double qq = sq3<CLA>(o.dx, o.dy, o.dz);
    const double q0 = sq3<CLA>(ex, ey, ez);
    double h0;
    sqrt_core(qq, o.l, o.hl);
    sqrt_core(q0, o.l0, h0);
    o.sh = (o.l - o.l0) * h0;  // s/2, from h0 ~ 0.5/l0
    // k = (c_i + c_j)/2 for a field: s k/l V_j = (s/2)(0.5/l) w with
    // w = 2(c_i+c_j)V_j = c_i (2 V_j) + (2 c_j V_j), the staged pair
    o.w = DM == DM_FIELD ? __builtin_fma(ci, p1.y, p3.y) : p1.y;
    if constexpr (DM == DM_NLIN) {
        const double2 c = *reinterpret_cast<const double2 *>(ldsb + st);
        const double2 k = *reinterpret_cast<const double2 *>(
            ldsb + 16 * MAX_TAB + st);
        kb = k.x;
        pb = k.y;
        return (o.sh < c.y) & (o.sh > c.x);
    } else if constexpr (TENS) {
        return (o.sh < lim) & (o.sh > -0.25);
    } else {
        return fabs(o.sh) < lim;
    }
}

// The stretch of the bond to halo entry `ev` with IEEE square roots and
// division (spatial.pyx:87-97, cl/peridynamics.cl:72-74), in place of
// bond_fast's.
template <int DM, bool CLA, bool NARROW>
__device__ __forceinline__ void stretch_exact(const char *ldsb,
                                              const double4 &r0i, unsigned ev,
                                              Bond &o)
{
    constexpr unsigned PB = piece_bytes<DM, NARROW>();
    const char *pe = ldsb + halo_base<DM>() + ev;
    const double2 p0 = *reinterpret_cast<const double2 *>(pe);
    const double2 p1 = *reinterpret_cast<const double2 *>(pe + PB);
    const double qq = sq3<CLA>(o.dx, o.dy, o.dz);
    const double ex = p0.x - r0i.x;
    const double ey = p0.y - r0i.y;
    const double ez = p1.x - r0i.z;
    const double q0 = sq3<CLA>(ex, ey, ez);
    o.l = sqrt(qq);
    o.l0 = sqrt(q0);
    if (!(core_range(qq) & core_range(q0)))
        o.hl = 0.5 / o.l;
    o.sh = ((o.l - o.l0) / o.l0) * 0.5;
}

// Whether a bond of that s/2 stays, by the scalar criterion.
template <bool TENS>
__device__ __forceinline__ bool stays(double sh, double s0h)
{
    return (TENS ? sh : fabs(sh)) < s0h;
}

// The bond at slot `slot` by stretch_exact: decides whether it breaks or
// changes its regime, writes that, and leaves in `o` (and kb, pb for
// DM_NLIN) what the force needs, zero for a broken or empty slot, whose
// correction `cr` becomes zero too (it may be infinite or NaN).
template <int DM, bool TENS, bool CLA, bool NARROW>
__device__ __forceinline__ void bond_exact(const StepArgs &a,
                                           const char *ldsb,
                                           const double4 &r0i, unsigned ev,
                                           unsigned st, size_t slot, Bond &o,
                                           double &kb, double &pb, double &cr,
                                           int &nbroken)
{
    bool live = ev != LOC_DEAD;
    if (live) {
        stretch_exact<DM, CLA, NARROW>(ldsb, r0i, ev, o);
        if constexpr (DM != DM_NLIN) {
            live = stays<TENS>(o.sh, a.s0h);
        } else {
            // cl/peridynamics.cl:326-378 (bond_force3/4), thresholds halved
            const int t = (int)(st >> 4) / a.nregimes;
            const int reg = (int)(st >> 4) - t * a.nregimes;
            const int base = t * a.nregimes;
            int nreg = reg;
            if (o.sh < a.s_tab[base + reg] * 0.5) {
                if (reg > 0 && o.sh < a.s_tab[base + reg - 1] * 0.5)
                    nreg = reg - 1;
            } else {
                nreg = reg + 1;
            }
            live = nreg < a.nregimes;
            // a dead slot's s of 0 lies between the thresholds of regime 0
            // (a later one's lower threshold would send it here in every
            // step: a body without a live bond 11 % a step)
            if (nreg != reg)
                a.state[slot] =
                    (unsigned short)((base + (live ? nreg : 0)) << 4);
            if (live) {
                kb = 4.0 * a.k_tab[base + nreg];
                pb = 2.0 * a.pc_tab[base + nreg];
            }
        }
        if (!live) {
            a.loc[slot] = LOC_DEAD;
            if (a.brk)
                a.brk[slot] = a.step;
            a.gidx[slot] |=
                (int)(DEAD | (a.layout == PD_LAYOUT_COMPACT ? NEWB : 0u));
            ++nbroken;
        }
    }
    if (!live) {
        // a displacement that is not finite must not reach the sum either
        o.dx = o.dy = o.dz = o.sh = o.hl = o.w = 0.0;
        kb = pb = cr = 0.0;
    }
}

// A chunk's bond data: the halo entries and, for DM_NLIN, the bond states,
// with CORR the corrections.
template <bool CORR>
struct Chunk {
    uint2 loc, st;
    double2 ca, cb;
};

template <>
struct Chunk<false> {
    uint2 loc, st;
};

// Two bonds of node i, at slots s0 and s0 + 1: `lw` their halo entries, `sw`
// their states, `cr` their corrections.  The two are straight-line code whose
// chains interleave; only a bond near a threshold (or broken by this step)
// leaves it.
template <int DM, bool CORR, bool TENS, bool CLA, bool NARROW>
__device__ __forceinline__ void bond_pair(const StepArgs &a, const char *ldsb,
                                          const double4 &r0i,
                                          const double4 &ri, double ci,
                                          double lim, unsigned lw,
                                          unsigned sw, double2 cr,
                                          size_t s0, double &fx, double &fy,
                                          double &fz, int &nbroken)
{
    Bond o[2];
    double kb[2], pb[2], c[2] = {cr.x, cr.y};
    const unsigned ev[2] = {lw & 0xffffu, lw >> 16};
    const unsigned st[2] = {sw & 0xffffu, sw >> 16};
    const bool ok0 = bond_fast<DM, TENS, CLA, NARROW>(
        ldsb, r0i, ri, ci, lim, ev[0], st[0], o[0], kb[0], pb[0]);
    const bool ok1 = bond_fast<DM, TENS, CLA, NARROW>(
        ldsb, r0i, ri, ci, lim, ev[1], st[1], o[1], kb[1], pb[1]);
    if (__builtin_expect(!(ok0 & ok1), 0)) {
        if (!ok0)
            bond_exact<DM, TENS, CLA, NARROW>(a, ldsb, r0i, ev[0], st[0], s0,
                                              o[0], kb[0], pb[0], c[0],
                                              nbroken);
        if (!ok1)
            bond_exact<DM, TENS, CLA, NARROW>(a, ldsb, r0i, ev[1], st[1],
                                              s0 + 1, o[1], kb[1], pb[1],
                                              c[1], nbroken);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        // s k/l V_j = (s/2)(0.5/l)(4 k V_j); n-linear (s k + plus_cs)/l V_j
        // = ((s/2)(4 k) + 2 plus_cs)(0.5/l) V_j, the tables scaled
        double g = DM == DM_NLIN ? __builtin_fma(o[q].sh, kb[q], pb[q])
                                 : o[q].sh;
        g = g * o[q].hl * o[q].w;
        if (CORR)
            g *= c[q];
        fx = __builtin_fma(g, o[q].dx, fx);
        fy = __builtin_fma(g, o[q].dy, fy);
        fz = __builtin_fma(g, o[q].dz, fz);
    }
}

// What bounds it on large meshes: the VALU (9.4e7 wave instructions per launch
// on the 1,038,230-node beam, mostly FP64 at 4 cycles and more, where there were
// 1.16e8: 81 % of the cycles at 4 each, 72 % in the wide form; the clock gives
// way under that load) and the LDS (about 60 %).  So the bond loop has one
// compare per bond for everything that is rare, dead slots cost no test, LDS
// offsets come ready from loc, chunk loads step one 32-bit offset, and a row
// runs half rounds: 305 -> 270 us a step there, 113 -> 77 on the 263k-node
// composite bar (its state now is the LDS offset of the bond's table entry),
// 57 -> 48 on a 141k-node bar with corrections (requested with the chunk).
// Tiles by bisection and a leaner prologue gave 257 us on the beam, 74.5 and
// 46.4 on the other two; what a run's inner steps store for nobody (force, the
// slot layout's u, Euler-Cromer's udd) left out, 250, 72 and 45.5; tiles even
// over the CUs 42.3 on the last; the narrow form takes 4 % off the beam
// (narrow_fits).
//
// DM: DM_PMB, DM_NLIN or DM_FIELD.  One workgroup per tile, LPN lanes per
// node taking its 4-bond chunks round-robin and reducing with cross-lane
// moves.  LDS (static): for DM_NLIN the damage-model tables, then the
// halo, pieces of piece_bytes<DM, NARROW>() each.
// CLA: the slot layout's OpenCL arithmetic (records hold u, updates
// contracted); otherwise the Cython path's (records hold r0 + u).
// NARROW: the narrow halo form, blocks of at most 512, and registers for six
// wavefronts per SIMD, that is three workgroups of 128 nodes per CU instead of
// two; used where a CU gets more than two tiles (narrow_fits).  The
// node's state is then read after the bonds: the registers that would hold it
// are what six wavefronts lack, and there are others to run meanwhile.
template <int DM, int LPN, bool CORR, bool TENS, bool CLA, bool NARROW>
__global__ __launch_bounds__(NARROW ? 512 : 1024, NARROW ? 6 : 1) void k_step(
    StepArgs a, double dmag, double fmag)
{
    static_assert(!NARROW || (DM == DM_PMB && CLA && !CORR),
                  "no use of c_j, and no rows to compact in LDS");
    __shared__ double2
        lds[(NARROW ? LDS_BYTES_NARROW : LDS_BYTES) / sizeof(double2)];
    const int b = blockIdx.x;
    const int tile = (b % XCDS) * a.tiles_per_xcd + b / XCDS;
    if (tile >= a.ntiles)
        return;
    const TileInfo ti = a.tiles[tile];
    char *ldsb = reinterpret_cast<char *>(lds);

    const int l = threadIdx.x / LPN;
    const int sub = threadIdx.x % LPN;
    const bool valid = l < ti.nodes;

    // the halo's node indices first: the records they name are the longest
    // chain of this kernel
    constexpr unsigned PB = piece_bytes<DM, NARROW>();
    HaloLoads<NARROW> hl;
    hl.request(a.halo + ti.halo_off, (unsigned)ti.halo);

    // node state and the first chunks of halo entries are requested before
    // the halo is staged, so their latency overlaps the staging.  Chunk rows
    // past the node's last are never used (their loads stay inside loc's
    // allocation, which is LOC_SLACK slots longer than the tiles need); past
    // the wavefront's last round the loads repeat it, as a condition around
    // them would make the loop wait for them at once.
    const char *L = reinterpret_cast<const char *>(a.loc + 4 * ti.chunk_off);
    const char *S = reinterpret_cast<const char *>(a.state + 4 * ti.chunk_off);
    const char *C = reinterpret_cast<const char *>(a.corr + 4 * ti.chunk_off);
    const unsigned cstep = 8u * LPN * (unsigned)ti.nodes;
    unsigned coff = 8u * ((valid ? (unsigned)l : 0u) +
                          (unsigned)sub * (unsigned)ti.nodes);
    auto chunk_at = [&](unsigned off) {
        Chunk<CORR> ch;
        ch.loc = *reinterpret_cast<const uint2 *>(L + off);
        if constexpr (DM == DM_NLIN)
            ch.st = *reinterpret_cast<const uint2 *>(S + off);
        else
            ch.st = make_uint2(0u, 0u);
        if constexpr (CORR) {
            const double2 *c =
                reinterpret_cast<const double2 *>(C + 4ull * off);
            ch.ca = c[0];
            ch.cb = c[1];
        }
        return ch;
    };
    Chunk<CORR> qa = chunk_at(coff), qb = chunk_at(coff + cstep);
    int cnt = 0, fl = 0;
    const uint32_t i = (uint32_t)(ti.node_off + (valid ? l : 0));
    double4 r0i = make_double4(0.0, 0.0, 0.0, 0.0), ri = r0i;
    if (valid) {
        const NodeRec *pi = a.rec_old + i;
        r0i = pi->a;
        ri = pi->b;
        const int meta = a.meta[i];
        cnt = meta & 0xffff;
        fl = meta >> 16;
    }
    const double ci = DM == DM_FIELD && valid ? a.cnode[i] : 0.0;
    // where c_i is not finite, 0 c_i of a dead slot is not 0: all of the
    // node's bonds take bond_exact, which leaves dead ones out
    const double lim =
        DM == DM_FIELD && !(fabs(ci) < __builtin_inf()) ? -1.0 : a.lim;
    // with 4 or more lanes per node, lane d < 3 updates component d: its
    // inputs are requested now too (the prescribed values, needed only on
    // flagged DOFs, are read at the update)
    constexpr bool PRE = LPN >= 4 && !NARROW;
    double pu = 0.0, pud = 0.0, pudd = 0.0, pdens = 1.0;
    if (PRE && valid && sub < 3) {
        const size_t k = 3 * (size_t)i + sub;
        if (!CLA)
            pu = a.u[k];
        if (a.integrator != PD_EULER) {
            pud = a.ud[k];
            pdens = a.dens1 ? a.dens1[i] : a.dens[k];
            if (a.integrator == PD_VELOCITY_VERLET)
                pudd = a.udd[k];
        }
    }

    hl.template stage<DM != DM_NLIN>(a.rec_old, a.halo + ti.halo_off,
                            (unsigned)ti.halo, ldsb + halo_base<DM>(), PB);
    if (threadIdx.x < 4)
        far_entry<CLA, NARROW>(ldsb + halo_base<DM>(), PB);
    // n-linear tables, one 16-byte read each: (lower, upper) halved
    // thresholds of regime r of type t with their margin, and (4 stiffness,
    // 2 plus_cs)
    if (DM == DM_NLIN) {
        double2 *tsp = reinterpret_cast<double2 *>(ldsb);
        double2 *tkp = tsp + MAX_TAB;
        for (int t = threadIdx.x; t < a.ntab; t += blockDim.x) {
            const double up = a.s_tab[t] * 0.5;
            double lo = -0.25;
            if (t % a.nregimes != 0) {
                const double c = a.s_tab[t - 1] * 0.5;
                lo = fmax(lo, c + GUARD * fabs(c));
            }
            tsp[t] = make_double2(
                lo, a.lim > 0.0 ? up - GUARD * fabs(up) : -__DBL_MAX__);
            tkp[t] = make_double2(4.0 * a.k_tab[t], 2.0 * a.pc_tab[t]);
        }
    }
    __syncthreads();

    double fx = 0.0, fy = 0.0, fz = 0.0;
    int nbroken = 0;
    // nodes are sorted by descending bond count, so the wavefront's first
    // node has its longest row: every lane runs that row's rounds (surplus
    // slots are empty).  Round k's chunks hold 2-bond groups 8 apart
    // (slot_of), so a row's last round of at most 8 bonds runs half of it.
    const int cmax = __builtin_amdgcn_readfirstlane(cnt);
    const unsigned cend = 8u * (unsigned)ti.nodes * (unsigned)ti.nch;
    auto round = [&](const Chunk<CORR> &ch, int k, unsigned off) {
        if (off >= cend)
            return;  // past the tile's rows (LPN does not divide them)
        const size_t s0 =
            4 * ((size_t)ti.chunk_off + (off >> 3));
        double2 ca = make_double2(1.0, 1.0), cb = ca;
        if constexpr (CORR) {
            ca = ch.ca;
            cb = ch.cb;
        }
        bond_pair<DM, CORR, TENS, CLA, NARROW>(
            a, ldsb, r0i, ri, ci, lim, ch.loc.x, ch.st.x, ca, s0, fx, fy, fz,
            nbroken);
        if (16 * (LPN * k / 4) + 8 < cmax)
            bond_pair<DM, CORR, TENS, CLA, NARROW>(
                a, ldsb, r0i, ri, ci, lim, ch.loc.y, ch.st.y, cb, s0 + 2, fx,
                fy, fz, nbroken);
    };
    const int rounds = (chunks_of(cmax) + LPN - 1) / LPN;
    if (valid) {
        for (int k = 0; k < rounds; k += 2) {
            round(qa, k, coff);
            coff += cstep;
            qa = chunk_at(coff + (k + 2 < rounds ? cstep : 0u));
            if (k + 1 >= rounds)
                break;
            round(qb, k + 1, coff);
            coff += cstep;
            qb = chunk_at(coff + (k + 3 < rounds ? cstep : 0u));
        }
    }

    fx = node_sum<LPN>(fx);
    fy = node_sum<LPN>(fy);
    fz = node_sum<LPN>(fz);
    nbroken = node_sum<LPN>(nbroken);
    // the compact layout (the Cython path, launched with !CLA only): once
    // the halo is no longer read, its LDS holds the rows being compacted
    if constexpr (!CLA) {
        if (a.layout == PD_LAYOUT_COMPACT)
            compact_tile<LPN, false>(a, ti, ldsb, LDS_BYTES, valid, l, sub,
                                     i, cnt, nbroken);
    }
    if (!valid)
        return;

    // the node's lanes share its three components (after the xor reduction
    // every lane holds the sums), so the per-node loads and stores coalesce
    const size_t b3 = 3 * (size_t)i;
    for (int d = sub; d < 3; d += LPN) {
        const size_t k = b3 + d;
        const double bf = d == 0 ? fx : (d == 1 ? fy : fz);
        // force boundary condition after the bond sum
        // (peridynamics.pyx:93-97, cl/peridynamics.cl:117-129)
        // body_force differs from force only on a force-BC DOF, so only
        // those store it; reads take force elsewhere
        const bool fbc = (fl >> (3 + d)) & 1;
        double F = bf;
        if (fbc)
            F = CLA ? __builtin_fma(fmag, a.fbcv[k], bf)
                    : bf + fmag * a.fbcv[k];
        if (a.store & STORE_F) {
            if (fbc)
                a.body_force[k] = bf;
            a.force[k] = F;
        }
        const bool fixed = (fl >> d) & 1;
        // the slot layout's records hold u
        double u = CLA ? (d == 0 ? ri.x : (d == 1 ? ri.y : ri.z))
                       : (PRE ? pu : a.u[k]);
        if (a.integrator == PD_EULER) {
            // peridynamics.pyx:179-185; cl/euler.cl:21-23 (contracted)
            const double un = CLA ? __builtin_fma(a.dt, F, u) : u + a.dt * F;
            u = fixed ? dmag * a.bcv[k] : un;
        } else if (a.integrator == PD_EULER_CROMER) {
            // cl/euler_cromer.cl:29-34 (contracted)
            double ud = PRE ? pud : a.ud[k];
            const double dens =
                PRE ? pdens : (a.dens1 ? a.dens1[i] : a.dens[k]);
            const double udd = __builtin_fma(-a.damping, ud, F) / dens;
            ud = __builtin_fma(udd, a.dt, ud);
            if (a.store & STORE_F)
                a.udd[k] = udd;
            a.ud[k] = ud;
            u = fixed ? dmag * a.bcv[k] : __builtin_fma(a.dt, ud, u);
        } else {
            // cl/velocity_verlet.cl:29-35 (contracted)
            const double hdt = a.dt / 2;
            const double ud1 = __builtin_fma(hdt, PRE ? pudd : a.udd[k],
                                             PRE ? pud : a.ud[k]);
            const double dens =
                PRE ? pdens : (a.dens1 ? a.dens1[i] : a.dens[k]);
            const double udd1 = __builtin_fma(-a.damping, ud1, F) / dens;
            const double ud = __builtin_fma(hdt, udd1, ud1);
            a.ud[k] = ud;
            a.udd[k] = udd1;
            u = fixed ? dmag * a.bcv[k]
                      : __builtin_fma(a.dt, __builtin_fma(hdt, udd1, ud), u);
        }
        if (!CLA || (a.store & STORE_U))
            a.u_out[k] = u;
        // the bond loop's position for the next step: r0 + u (compact) or
        // u (slot); the record's c (w) is static
        const double r0d = d == 0 ? r0i.x : (d == 1 ? r0i.y : r0i.z);
        reinterpret_cast<double *>(&a.rec_new[i].b)[d] = CLA ? u : r0d + u;
    }
}

// Whether a coordinate is in the range that bond_fast relies on.
__host__ __device__ __forceinline__ bool core_coord(double x)
{
    x = fabs(x);
    return x == 0.0 || (x >= 0x1p-290 && x <= 0x1p300);
}

// bond_fast's limit for a halved critical stretch (scalar criterion).
__host__ __device__ __forceinline__ double fast_limit(double s0h)
{
    const double m = s0h * (1.0 - GUARD);
    return 0.25 < m ? 0.25 : m;
}

// The stretch and break decision of the scalar step in plain order, one bond
// per thread, for checking: the step's own bond_fast, and stretch_exact and
// stays behind it, on a record that the thread puts into LDS.  Out come l and
// l0 (bitwise those of spatial.pyx, or of cl/peridynamics.cl:65-75 as
// contracted with CLA), the working s (2*sh), the exact s = (l - l0)/l0 and
// the decision.  With CLA, ri and rj are the displacements u_i, u_j (the
// OpenCL kernels form the bond from u); otherwise positions r0 + u.
constexpr int CHECK_BLOCK = 256;

template <bool TENS, bool CLA>
__global__ __launch_bounds__(CHECK_BLOCK) void k_bond_check(
    int n, const double *ri, const double *rj, const double *r0i,
    const double *r0j, double s0, double *l_out, double *l0_out,
    double *s_out, double *s_exact, int *broken)
{
    constexpr unsigned PB = piece_bytes<DM_PMB>();
    static_assert(CHECK_BLOCK < LDS_CAP_PMB, "an entry per thread");
    __shared__ double2 lds[LDS_BYTES / sizeof(double2)];
    const int t = blockIdx.x * CHECK_BLOCK + threadIdx.x;
    if (t >= n)
        return;
    const size_t b = 3 * (size_t)t;
    const unsigned ev = 16u * (threadIdx.x + 1u);
    char *ldsb = reinterpret_cast<char *>(lds);
    const double e[8] = {r0j[b], r0j[b + 1], r0j[b + 2], 1.0,
                         rj[b],  rj[b + 1],  rj[b + 2],  0.0};
    bool core = true;
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<double2 *>(ldsb + q * PB + ev) =
            make_double2(e[2 * q], e[2 * q + 1]);
    for (int d = 0; d < 3; ++d)
        core &= core_coord(r0i[b + d]) && core_coord(r0j[b + d]);
    const double4 own0 = make_double4(r0i[b], r0i[b + 1], r0i[b + 2], 1.0);
    const double4 own = make_double4(ri[b], ri[b + 1], ri[b + 2], 0.0);
    const double s0h = s0 * 0.5;
    Bond o;
    double kb, pb;
    bool live = true;
    if (!bond_fast<DM_PMB, TENS, CLA, false>(ldsb, own0, own, 0.0,
                                             core ? fast_limit(s0h) : -1.0, ev,
                                             0u, o, kb, pb)) {
        stretch_exact<DM_PMB, CLA, false>(ldsb, own0, ev, o);
        live = stays<TENS>(o.sh, s0h);
    }
    l_out[t] = o.l;
    l0_out[t] = o.l0;
    s_out[t] = o.sh + o.sh;
    s_exact[t] = (o.l - o.l0) / o.l0;
    broken[t] = !live;
}

// Records of both ping-pong buffers from r0, V, u and c: a = (r0, wscale V),
// b = (r0 + u, v) -- (u, v) with ucla, the slot layout's OpenCL stretch --
// with v = 2 c V for a field c, else 0.  The weights are the factors the
// bond loop multiplies by: wscale = 4k for the scalar model, 2 for the field
// model, 1 for the n-linear model (more where its tables are scaled).
__global__ void k_records(int n, double wscale, int ucla, const double *r0,
                          const double *vol, const double *u, const double *c,
                          NodeRec *rec0, NodeRec *rec1)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const size_t b = 3 * (size_t)i;
    NodeRec r;
    r.a = make_double4(r0[b], r0[b + 1], r0[b + 2], vol[i] * wscale);
    const double v = c ? 2.0 * c[i] * vol[i] : 0.0;
    r.b = ucla ? make_double4(u[b], u[b + 1], u[b + 2], v)
               : make_double4(r0[b] + u[b], r0[b + 1] + u[b + 1],
                              r0[b + 2] + u[b + 2], v);
    rec0[i] = r;
    rec1[i] = r;
}

// Lanes per node of the kernels that walk every row once.  Over the chunks of
// the rows (live counts, recordings) four: a wavefront then reads 128
// contiguous bytes of loc in each of four chunk rows, and each lane's loads
// are independent.  Over the caller's rows (lists) sixteen: 64 contiguous
// bytes of a row at a time.
constexpr int CHUNK_LANES = 4;
constexpr int ROW_LANES = 16;

// Live slots of a node, counted by its LANES lanes (every lane gets the sum):
// loc is 0 in a broken or empty slot.
template <int LANES>
__device__ __forceinline__ int live_slots(const unsigned short *loc,
                                          long long chunk0, int stride,
                                          int cnt, int sub)
{
    const uint2 *L = reinterpret_cast<const uint2 *>(loc) + chunk0;
    const int nch = chunks_of(cnt);
    int live = 0;
#pragma unroll 4
    for (int c = sub; c < nch; c += LANES) {
        const uint2 v = L[(long long)c * stride];
        live += ((v.x & 0xffffu) != 0) + ((v.x >> 16) != 0) +
                ((v.y & 0xffffu) != 0) + ((v.y >> 16) != 0);
    }
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1)
        live += __shfl_xor(live, off, LANES);
    return live;
}

// Live-slot count per node, the damage (family - n)/family
// (peridynamics.pyx:29), and, for the slot layout, the reference-layout
// neighbour list: -1 everywhere but at the live slots' columns.  LANES
// lanes handle internal node p and write row tnode[p] of the outputs.
// rows == 0 counts the live bonds without rebuilding the slot-layout rows;
// with u_out, u goes along into the caller's node order (one launch for the
// read-out of u and damage that every write interval makes).
// Without rows it reads 2 B per slot (loc): 3.8 us on a 2560-node bar and 83
// on 1,038,230 nodes, where one lane per node walking gidx took 23 and 243.
template <int LANES>
__global__ void __launch_bounds__(256)
    k_export(int n, int K, int layout, int rows, const int *tnode,
             const int *cnt, const long long *chunk0, const int *stride,
             const unsigned short *loc, const int *gidx,
             const unsigned short *pos, const int *family,
             const int *n_neigh_c, int *nlist_out, int *n_neigh_out,
             double *damage, const double *u, double *u_out)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int p = t / LANES, sub = t % LANES;
    const bool valid = p < n;
    const int i = valid ? tnode[p] : 0;
    if (u_out && valid)
        for (int d = sub; d < 3; d += LANES)
            u_out[3 * (size_t)i + d] = u[3 * (size_t)p + d];
    int live = 0;
    if (layout == PD_LAYOUT_SLOT) {
        const int c = valid ? cnt[p] : 0;
        const long long c0 = valid ? chunk0[p] : 0;
        const int st = valid ? stride[p] : 0;
        live = live_slots<LANES>(loc, c0, st, c, sub);
        if (rows) {
            int *row = nlist_out + (size_t)i * K;
            if (valid)
                for (int q = sub; q < K; q += LANES)
                    row[q] = -1;
            __syncthreads();  // the row is cleared before its bonds are set
            for (int k = sub; k < c; k += LANES) {
                const size_t s = slot_of(c0, st, k);
                const int e = gidx[s];
                if (e >= 0)
                    row[pos[s]] = e;
            }
        }
    } else if (valid) {
        live = n_neigh_c[i];
    }
    if (!valid || sub != 0)
        return;
    n_neigh_out[i] = live;
    const double f = (double)family[i];
    damage[i] = (f - (double)live) / f;
}

// The compact layout's reference-layout rows in the caller's numbering: the
// positions below the row's count at set-up list their slots' keys (live
// ones first, then what swap-with-last left behind); the others keep the
// caller's values (uploaded into nlist_ref at set-up).
__global__ void __launch_bounds__(256)
    k_export_rows(int n, int K, const int *tnode, const int *cnt,
                  const long long *chunk0, const int *stride,
                  const int *gidx, const unsigned short *rslot,
                  int *nlist_ref)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int p = t / ROW_LANES, sub = t % ROW_LANES;
    if (p >= n)
        return;
    const size_t row = (size_t)tnode[p] * K;
    const int c = cnt[p];
    for (int q = sub; q < c; q += ROW_LANES)
        nlist_ref[row + q] =
            (int)((uint32_t)gidx[slot_of(chunk0[p], stride[p],
                                         rslot[row + q])] & KEYM);
}

// Monitored sums of a write (model.py:1320-1360).  Pass 1: block b sums a
// fixed strided share of the DOFs -- u, ud, udd, force*V, body_force*V --
// and of the nodes' damage, then reduces its 256 lanes by a fixed tree, so
// the result does not depend on scheduling.
constexpr int MON_BLOCKS = 512;
constexpr int MON_SUMS = 6;

__global__ void __launch_bounds__(256)
    k_monitor_part(int n, const double *u, const double *ud,
                   const double *udd, const double *force,
                   const double *body, const int *flags, const double *vol,
                   const double *damage, double *part)
{
    __shared__ double sh[MON_SUMS][256];
    const int t = threadIdx.x;
    const size_t first = (size_t)blockIdx.x * 256 + t;
    const size_t step = (size_t)MON_BLOCKS * 256;
    double a[MON_SUMS] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (size_t q = first; q < 3 * (size_t)n; q += step) {
        const size_t p = q / 3;
        const double v = vol[p];
        const bool fbc = (flags[p] >> (3 + (int)(q - 3 * p))) & 1;
        a[0] += u[q];
        a[1] += ud[q];
        a[2] += udd[q];
        a[3] += force[q] * v;
        a[4] += (fbc ? body[q] : force[q]) * v;
    }
    for (size_t i = first; i < (size_t)n; i += step)
        a[5] += damage[i];
    for (int k = 0; k < MON_SUMS; ++k)
        sh[k][t] = a[k];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w)
            for (int k = 0; k < MON_SUMS; ++k)
                sh[k][t] += sh[k][t + w];
        __syncthreads();
    }
    if (t < MON_SUMS)
        part[(size_t)blockIdx.x * MON_SUMS + t] = sh[t][0];
}

// Pass 2 (one block): the block sums in block order, and each tip group's
// sums accumulated entry by entry from 0.0 in the order the entries were
// given -- the reference's loop over the group's (node, dof) list
// (model.py:1320-1336), so these are its values bitwise.
__global__ void __launch_bounds__(256)
    k_monitor_final(const double *part, int ngroups, const int *tip_off,
                    const int *tip_q, const double *u, const double *ud,
                    const double *udd, const double *force,
                    const double *body, const int *flags, const double *vol,
                    double *out)
{
    const int t = threadIdx.x;
    if (t < MON_SUMS) {
        double acc = 0.0;
        for (int b = 0; b < MON_BLOCKS; ++b)
            acc += part[b * MON_SUMS + t];
        out[t] = acc;
    }
    for (int g = t; g < ngroups; g += blockDim.x) {
        double a[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        for (int e = tip_off[g]; e < tip_off[g + 1]; ++e) {
            const int q = tip_q[e];
            const int p = q / 3;
            const double v = vol[p];
            const bool fbc = (flags[p] >> (3 + q - 3 * p)) & 1;
            a[0] += u[q];
            a[1] += ud[q];
            a[2] += udd[q];
            a[3] += force[q] * v;
            a[4] += (fbc ? body[q] : force[q]) * v;
        }
        for (int k = 0; k < 5; ++k)
            out[MON_SUMS + 5 * g + k] = a[k];
    }
}

__global__ void k_export_regimes(int n, int K, const int *tnode,
                                 const int *cnt, const long long *chunk0,
                                 const int *stride,
                                 const unsigned short *pos,
                                 const unsigned short *state,
                                 const int *gidx, int nregimes, int *out)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n)
        return;
    const size_t row = (size_t)tnode[p] * K;
    const int c = cnt[p];
    for (int k = 0; k < c; ++k) {
        const size_t s = slot_of(chunk0[p], stride[p], k);
        // a broken bond has walked past its last regime
        out[row + pos[s]] =
            gidx[s] < 0 ? nregimes : (state[s] >> 4) % nregimes;
    }
}

__global__ void __launch_bounds__(256)
    k_live(int n, const int *cnt, const long long *chunk0, const int *stride,
           const unsigned short *loc, unsigned long long *total)
{
    __shared__ int part[256 / CHUNK_LANES];
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int p = t / CHUNK_LANES, sub = t % CHUNK_LANES;
    const bool valid = p < n;
    const int live =
        live_slots<CHUNK_LANES>(loc, valid ? chunk0[p] : 0, valid ? stride[p] : 0,
                   valid ? cnt[p] : 0, sub);
    if (sub == 0)
        part[threadIdx.x / CHUNK_LANES] = live;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0;
        for (int k = 0; k < 256 / CHUNK_LANES; ++k)
            sum += (unsigned long long)part[k];
        atomicAdd(total, sum);
    }
}

// --- exact-order Euler step of the Cython path ----------------------------
//
// peridynamics.pyx:34-99 (bond_force) visits i ascending and, for each live
// j > i of i's row in row order, adds f V_j to F_i and subtracts f V_i from
// F_j.  So F_m is the left fold, from +0.0, of first the bonds to live
// k < m in ascending k, then the bonds to the live j > m of m's current row
// in row order, then the force boundary condition.  Every term is
// (fn (r_j - r_m)) V_j with fn = ((l - l0)/l0 k)/l, l = |r_j - r_m|,
// l0 = |r0_j - r0_m| (spatial.pyx:20-31, 87-97): for a lower neighbour the
// reference subtracts (fn (r_m - r_k)) V_k, which is the same double,
// negated, as r_m - r_k is the exact negation of r_k - r_m.  The fold order
// depends only on node m's own row, so each tile folds its own nodes.
//
// A node's fold list (ford) is its lower slots in ascending order (slot
// order: rows are sorted by caller id; a dead slot adds nothing), then its
// upper neighbours in current row order (slot index << 16 | halo loc, rebuilt
// by compact_tile after every break of the node).  The node's four lanes take
// eight consecutive positions per round, two each, whose evaluations
// interleave (eight lanes, one each): with the reference's operations -- bitwise square roots, IEEE
// divisions, no contraction -- each gives its three force terms and decides
// the break from that exact stretch (peridynamics.pyx:133).  The terms pass
// through the node's 96-byte LDS window, four positions at a time; lanes 0-2
// add the terms of their component in order.  Breaking is applied before the
// force, as in Euler.__call__: a bond that breaks adds nothing, and when any
// bond of the node breaks the row is compacted (peridynamics.pyx:102-156) and
// the part of the list whose order the compaction may change is folded again
// from the sum before it.  Assumes symmetric neighbour lists without repeats,
// as the model builds them.

// LDS of the exact step: the halo (pieces of EXACT_CAP entries), then the
// fold windows (12 doubles per node, tiles of up to EXACT_NODES nodes).
constexpr int EXACT_NODES = 128;
constexpr int EXACT_CAP = (int)((LDS_BYTES - EXACT_NODES * 96u) / 64u);
// Tiles of at most that many nodes run eight lanes per node: they are small
// because the mesh is (set_shape), so that a round's latency bounds it.
constexpr int EXACT_WIDE_NODES = 64;

// Rows of K slots fit compact_tile's groups in the exact step's fold
// windows (its 64 bytes of counts, then at least one row).
__host__ __device__ constexpr bool exact_rows_fit(int K)
{
    return compact_row_bytes(K) + 64u <= EXACT_NODES * 96u;
}

// The exact bond evaluation: the term's components and the stretch.
struct ExactTerm {
    double t0, t1, t2, s;
};

// a / b rounded to nearest, given h ~ 0.5/b (sqrt_core's, relative error
// below 2^-46): one Newton step makes y the reciprocal to within its rounding
// and 2^-92, as the compiler's f64 division does in two from the hardware's
// estimate; then its quotient and residual correction, without its scaling
// steps, which change nothing when a is zero, or when a, b and a/b are
// normal, a >= 2^-969, 1/b is normal and a's exponent exceeds b's by less
// than 768.
__device__ __forceinline__ double div_core(double a, double b, double h)
{
    double y = h + h;
    const double e = __builtin_fma(-b, y, 1.0);
    y = __builtin_fma(y, e, y);
    const double q = a * y;
    const double r = __builtin_fma(-b, q, a);
    return __builtin_fma(r, y, q);
}

// The terms of halo entry e, exactly the reference's while the stretch lies
// strictly in (a.xlo, a.xhi); the caller takes exact_slow otherwise.  The
// interval is empty unless the stiffness is in [2^-100, 2^100], s0 below
// 2^300 and the coordinates in bond_fast's range.  Then q0 is 0 (NaN stretch)
// or in [2^-686, 2^603], s > -1/2 gives q at least 2^-690 (see bond_fast), so
// l and l0 come from sqrt_core exactly and lie in [2^-346, 2^512]; s is 0 or
// at least 2^-54 in magnitude (l - l0 is 0 or at least an ulp of the
// shorter), so every operand and quotient is normal, numerators exceed
// 2^-969 and no exponent gap reaches 768: both quotients are div_core's.  A
// dead or empty position reads entry 0, a far node of volume 0: its terms
// are zero.
__device__ __forceinline__ ExactTerm exact_fast(const StepArgs &a,
                                                const char *ldsb, unsigned e,
                                                const double4 &r0m,
                                                const double4 &rm)
{
    constexpr unsigned PB = 16u * EXACT_CAP;
    const char *pe = ldsb + e;
    const double2 p0 = *reinterpret_cast<const double2 *>(pe);
    const double2 p1 = *reinterpret_cast<const double2 *>(pe + PB);
    const double2 p2 = *reinterpret_cast<const double2 *>(pe + 2 * PB);
    const double p3 = *reinterpret_cast<const double *>(pe + 3 * PB);
    // spatial.pyx:20-31: squares of r_j - r_m summed left to right
    const double dx = p2.x - rm.x, dy = p2.y - rm.y, dz = p3 - rm.z;
    const double q = (dx * dx + dy * dy) + dz * dz;
    const double ex = p0.x - r0m.x, ey = p0.y - r0m.y, ez = p1.x - r0m.z;
    const double q0 = (ex * ex + ey * ey) + ez * ez;
    double l, l0, h, h0;
    sqrt_core(q, l, h);
    sqrt_core(q0, l0, h0);
    ExactTerm t;
    // spatial.pyx:87-97, peridynamics.pyx:75-89
    t.s = div_core(l - l0, l0, h0);
    const double fn = div_core(t.s * a.kx, l, h);
    const double v = p1.y;  // V_j
    t.t0 = (fn * dx) * v;
    t.t1 = (fn * dy) * v;
    t.t2 = (fn * dz) * v;
    return t;
}

// The same with the library's square roots and divisions, and the break
// (peridynamics.pyx:133) of the bond at slot `slot`, position `fold` of its
// node's list; `check` false only evaluates.
__device__ __forceinline__ void exact_slow(const StepArgs &a,
                                           const char *ldsb, unsigned e,
                                           const double4 &r0m,
                                           const double4 &rm, bool check,
                                           size_t slot, size_t fold,
                                           ExactTerm &t, int &nbroken)
{
    if (e == LOC_DEAD) {
        t.t0 = t.t1 = t.t2 = 0.0;
        return;
    }
    constexpr unsigned PB = 16u * EXACT_CAP;
    const char *pe = ldsb + e;
    const double2 p0 = *reinterpret_cast<const double2 *>(pe);
    const double2 p1 = *reinterpret_cast<const double2 *>(pe + PB);
    const double2 p2 = *reinterpret_cast<const double2 *>(pe + 2 * PB);
    const double p3 = *reinterpret_cast<const double *>(pe + 3 * PB);
    const double dx = p2.x - rm.x, dy = p2.y - rm.y, dz = p3 - rm.z;
    const double ex = p0.x - r0m.x, ey = p0.y - r0m.y, ez = p1.x - r0m.z;
    const double l = sqrt((dx * dx + dy * dy) + dz * dz);
    const double l0 = sqrt((ex * ex + ey * ey) + ez * ez);
    t.s = (l - l0) / l0;
    if (check && !(sign_mask(t.s, a.absmask) < 2.0 * a.s0h)) {
        a.loc[slot] = LOC_DEAD;
        a.ford[fold] = LOC_DEAD;
        a.gidx[slot] |= (int)(DEAD | NEWB);
        ++nbroken;
        t.t0 = t.t1 = t.t2 = 0.0;
        return;
    }
    double fn = t.s * a.kx;
    fn = fn / l;
    const double v = p1.y;
    t.t0 = (fn * dx) * v;
    t.t1 = (fn * dy) * v;
    t.t2 = (fn * dz) * v;
}

// The fold window of a node: [component][position of four].
__device__ __forceinline__ void window_put(double *win, int q,
                                          const ExactTerm &t)
{
    win[q] = t.t0;
    win[4 + q] = t.t1;
    win[8 + q] = t.t2;
}

// Between a wavefront's writes of its windows and their reads.
__device__ __forceinline__ void window_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One workgroup per tile of at most EXACT_NODES nodes, four lanes per node or
// eight (small meshes; the same results, as the fold's order does not depend
// on who evaluates a position), on k_step's tiles and halo staging.  Records hold
// (r0, V | r0 + u, 0).
//
// What bounds it: the VALU on large meshes, and on small ones a round's
// latency (gather, two square roots, two divisions, window, ordered adds:
// one chain).  Two positions per lane and round halve the chain's rounds and
// interleave two evaluations; with the list's entries in one array (one
// 8-byte load per lane and round), div_core seeded from the square roots and
// one interval test for everything rare, a bond takes 65 wave instructions
// where it took 115: 150 -> 104 us a step on 270,000 nodes, 20.7 -> 14 on
// the 2560-node bar.  Tiles by bisection and fewer stores 94 on the former;
// small tiles and eight lanes 9.8 on the latter.  On large meshes the VALU is
// busy 60 % of the cycles and the LDS (halo reads and windows) 66 %.
template <int LPN>
__global__ __launch_bounds__(512) void k_exact_step(StepArgs a, double dmag,
                                                    double fmag)
{
    static_assert(LPN == 4 || LPN == 8, "two or one positions per lane");
    __shared__ double2 lds[LDS_BYTES / sizeof(double2)];
    constexpr unsigned PB = 16u * EXACT_CAP;
    const int b = blockIdx.x;
    const int tile = (b % XCDS) * a.tiles_per_xcd + b / XCDS;
    if (tile >= a.ntiles)
        return;
    const TileInfo ti = a.tiles[tile];
    char *ldsb = reinterpret_cast<char *>(lds);
    const int l = threadIdx.x / LPN;
    const int sub = threadIdx.x % LPN;
    const bool valid = l < ti.nodes;
    HaloLoads<> hl;
    hl.request(a.halo + ti.halo_off, (unsigned)ti.halo);
    const uint32_t i = (uint32_t)(ti.node_off + (valid ? l : 0));
    const long long c0 = ti.chunk_off + (valid ? l : 0);
    // the lane's list entries of round r are r * fstep further on; with
    // eight lanes, lanes 4-7 take the second of the pairs
    const char *L = reinterpret_cast<const char *>(a.ford + 4 * ti.chunk_off);
    const unsigned fstep = 8u * 4u * (unsigned)ti.nodes;
    unsigned foff = 8u * ((valid ? (unsigned)l : 0u) +
                          (unsigned)(sub & 3) * (unsigned)ti.nodes) +
                    (LPN == 8 ? (unsigned)(sub & 4) : 0u);
    auto pair_at = [&](unsigned off) {
        if constexpr (LPN == 8)
            return make_uint2(*reinterpret_cast<const unsigned *>(L + off),
                              0u);
        else
            return *reinterpret_cast<const uint2 *>(L + off);
    };
    uint2 qa = pair_at(foff), qb = pair_at(foff + fstep);
    double4 r0m = make_double4(0.0, 0.0, 0.0, 0.0), rm = r0m;
    int cnt = 0, nlow = 0, fl = 0;
    double pu = 0.0;
    if (valid) {
        r0m = a.rec_old[i].a;
        rm = a.rec_old[i].b;
        const int meta = a.meta[i];
        cnt = meta & 0xffff;
        fl = meta >> 16;
        nlow = a.nlow[i];
        if (sub < 3)
            pu = a.u[3 * (size_t)i + sub];
    }
    hl.stage<true>(a.rec_old, a.halo + ti.halo_off, (unsigned)ti.halo, ldsb,
                   PB);
    if (threadIdx.x < 4)
        far_entry<false>(ldsb, PB);
    __syncthreads();

    double *win = reinterpret_cast<double *>(ldsb + 4 * PB) + 12 * l;
    double F = 0.0, Flow = 0.0;  // lane d < 3: component d
    int nbroken = 0;
    // four terms of every lane's component, in order: those of lanes from,
    // from + 1, ...
    auto fold4 = [&](const ExactTerm &t, int from) {
        if (LPN == 4 || (sub & 4) == from)
            window_put(win, sub & 3, t);
        window_sync();
        if (sub < 3) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                F = F + win[4 * sub + q];
        }
        window_sync();
    };
    auto round = [&](uint2 en, int r, bool check) {
        ExactTerm t0 = exact_fast(a, ldsb, en.x & 0xffffu, r0m, rm);
        if constexpr (LPN == 8) {
            if (__builtin_expect(!((t0.s > a.xlo) & (t0.s < a.xhi)), 0))
                exact_slow(a, ldsb, en.x & 0xffffu, r0m, rm, check,
                           slot_of(c0, ti.nodes, (int)(en.x >> 16)),
                           fold_of(ti.chunk_off, ti.nodes, l, 8 * r + sub),
                           t0, nbroken);
            fold4(t0, 0);
            fold4(t0, 4);
            return;
        }
        ExactTerm t1 = exact_fast(a, ldsb, en.y & 0xffffu, r0m, rm);
        const bool ok0 = (t0.s > a.xlo) & (t0.s < a.xhi);
        const bool ok1 = (t1.s > a.xlo) & (t1.s < a.xhi);
        if (__builtin_expect(!(ok0 & ok1), 0)) {
            const int pos = 8 * r + sub;
            if (!ok0)
                exact_slow(a, ldsb, en.x & 0xffffu, r0m, rm, check,
                           slot_of(c0, ti.nodes, (int)(en.x >> 16)),
                           fold_of(ti.chunk_off, ti.nodes, l, pos), t0,
                           nbroken);
            if (!ok1)
                exact_slow(a, ldsb, en.y & 0xffffu, r0m, rm, check,
                           slot_of(c0, ti.nodes, (int)(en.y >> 16)),
                           fold_of(ti.chunk_off, ti.nodes, l, pos + 4), t1,
                           nbroken);
        }
        fold4(t0, 0);
        fold4(t1, 0);
    };
    // the wavefront's first node has its longest list (nodes are sorted by
    // bond count); positions past a list's end are dead
    const int rounds = (__builtin_amdgcn_readfirstlane(cnt) + 7) >> 3;
    const int rlow = nlow >> 3;  // the first round with an upper position
    if (valid) {
        for (int r = 0; r < rounds; r += 2) {
            if (r <= rlow)
                Flow = F;
            round(qa, r, true);
            foff += fstep;
            qa = pair_at(foff + (r + 2 < rounds ? fstep : 0u));
            if (r + 1 >= rounds)
                break;
            if (r + 1 <= rlow)
                Flow = F;
            round(qb, r + 1, true);
            foff += fstep;
            qb = pair_at(foff + (r + 3 < rounds ? fstep : 0u));
        }
        if (rlow >= rounds)
            Flow = F;  // no upper part
    }
    nbroken = node_sum<LPN>(nbroken);
    // the fold windows are free: they hold the rows being compacted, and
    // the lists of those nodes are rebuilt in the new row order
    compact_tile<LPN, true>(a, ti, ldsb + 4 * PB, EXACT_NODES * 96u, valid, l,
                            sub, i, cnt, nbroken);
    if (!valid)
        return;
    if (nbroken > 0) {
        // again from the round in which the upper part begins
        F = Flow;
        const int total = nlow + (int)ld_slot(&a.nup[i]);
        for (int r = rlow; 8 * r < total; ++r) {
            const int *e = reinterpret_cast<const int *>(a.ford) +
                           fold_of(ti.chunk_off, ti.nodes, l, 8 * r + sub);
            round(make_uint2(ld_slot(e), LPN == 8 ? 0u : ld_slot(e + 1)), r,
                  false);
        }
    }
    if (sub < 3) {
        // peridynamics.pyx:93-97, then :179-185
        const size_t k = 3 * (size_t)i + sub;
        const bool fbc = (fl >> (3 + sub)) & 1;
        double Fd = F;
        if (fbc)
            Fd = F + fmag * a.fbcv[k];
        if (a.store & STORE_F) {
            if (fbc)
                a.body_force[k] = F;
            a.force[k] = Fd;
        }
        const double u = (fl >> sub) & 1 ? dmag * a.bcv[k] : pu + a.dt * Fd;
        a.u_out[k] = u;
        const double r0d = sub == 0 ? r0m.x : (sub == 1 ? r0m.y : r0m.z);
        reinterpret_cast<double *>(&a.rec_new[i].b)[sub] = r0d + u;
    }
}

// The fold lists of every node from its row and live bonds (set-up, and when
// the exact order is turned on: the fast step does not keep them).
__global__ void __launch_bounds__(256)
    k_fold_lists(int n, int K, const int *tnode, const int *cnt,
                 const long long *chunk0, const int *stride,
                 const long long *tile0, const int *gidx,
                 const unsigned short *loc, const unsigned short *rslot,
                 const int *n_neigh, const int *nlow, int *nup,
                 unsigned *ford)
{
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n)
        return;
    const int i = tnode[p], st = stride[p], low = nlow[p];
    const long long c0 = chunk0[p];
    const long long t0 = tile0[p];
    const int l = (int)(c0 - t0);
    int pos = 0;
    for (int k = 0; k < low; ++k) {
        const unsigned e = loc[slot_of(c0, st, k)];
        ford[fold_of(t0, st, l, pos++)] =
            e == LOC_DEAD ? LOC_DEAD : ((unsigned)k << 16) | e;
    }
    const int live = n_neigh[i];
    for (int q = 0; q < live; ++q) {
        const int k = rslot[(size_t)i * K + q];
        const size_t s = slot_of(c0, st, k);
        if ((int)((uint32_t)gidx[s] & KEYM) > i)
            ford[fold_of(t0, st, l, pos++)] = ((unsigned)k << 16) | loc[s];
    }
    nup[p] = pos - low;
    for (; pos < cnt[p]; ++pos)
        ford[fold_of(t0, st, l, pos)] = LOC_DEAD;
}

// --- adjoint of the Euler step with a recorded break mask -------------------
//
// Forward (PD_EULER, node stiffness field c): u_{n+1} = u_n + dt F(u_n) on
// free DOFs (prescribed DOFs are set), with
//   F_m = sum_j k_mj V_j phi(d_mj),  phi(d) = (1/l0 - 1/l) d = (s/l) d,
//   d_mj = r_j - r_m, k_mj = (c_m + c_j)/2,
// over the bonds live in step n (broken at a step > n, from brk).  For a
// loss L(u_N) and mu = P_free lambda_{n+1}:
//   lambda_n = mu + dt J_n^T mu,
//   (J^T mu)_m = sum_j k_mj A_mj (V_m mu_j - V_j mu_m),
//   A = dphi/dd = (1/l0 - 1/l) I + d d^T / l^3  (symmetric, even in d),
//   dL/dc_m += dt/2 sum_j (1/l0 - 1/l)_mj d_mj . (V_j mu_m - V_m mu_j).

// Bond state at the start of step n0: alive iff it broke at a step >= n0.
// Slots are taken four at a time, whatever node they belong to (an empty slot
// has brk -1), and gidx is written only where it changes.
__global__ void __launch_bounds__(256)
    k_adj_restore(long long nchunks, int n0, const int *brk,
                  const unsigned short *loc0, unsigned short *loc, int *gidx)
{
    const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
    if (c >= nchunks)
        return;
    const int4 b = reinterpret_cast<const int4 *>(brk)[c];
    ushort4 l = reinterpret_cast<const ushort4 *>(loc0)[c];
    const int4 g = reinterpret_cast<const int4 *>(gidx)[c];
    const int bv[4] = {b.x, b.y, b.z, b.w}, gv[4] = {g.x, g.y, g.z, g.w};
    unsigned short lv[4] = {l.x, l.y, l.z, l.w};
    int w[4];
    bool changed = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool alive = bv[q] >= n0;
        if (!alive)
            lv[q] = LOC_DEAD;
        const uint32_t e = (uint32_t)gv[q] & ~(DEAD | NEWB);
        w[q] = (int)(alive ? e : (e | DEAD));
        changed |= w[q] != gv[q];
    }
    reinterpret_cast<ushort4 *>(loc)[c] =
        make_ushort4(lv[0], lv[1], lv[2], lv[3]);
    if (changed)
        reinterpret_cast<int4 *>(gidx)[c] = make_int4(w[0], w[1], w[2], w[3]);
}

// The bonds back to their state at set-up: loc and the n-linear state from
// their copies, gidx without its marks (a slot that never held a bond has
// loc_init 0 and keeps its own).  One thread per chunk, a stream of 2 + 4 B
// read and at most 2 + 4 written per slot.
__global__ void __launch_bounds__(256)
    k_reset_bonds(long long nchunks, const unsigned short *loc_init,
                  const unsigned short *state_init, unsigned short *loc,
                  unsigned short *state, int *gidx)
{
    const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
    if (c >= nchunks)
        return;
    const ushort4 l = reinterpret_cast<const ushort4 *>(loc_init)[c];
    const int4 g = reinterpret_cast<const int4 *>(gidx)[c];
    const unsigned short lv[4] = {l.x, l.y, l.z, l.w};
    const int gv[4] = {g.x, g.y, g.z, g.w};
    int w[4];
    bool changed = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        w[q] = lv[q] == LOC_DEAD ? gv[q]
                                 : (int)((uint32_t)gv[q] & KEYM);
        changed |= w[q] != gv[q];
    }
    reinterpret_cast<ushort4 *>(loc)[c] = l;
    if (changed)
        reinterpret_cast<int4 *>(gidx)[c] = make_int4(w[0], w[1], w[2], w[3]);
    if (state)
        reinterpret_cast<ushort4 *>(state)[c] =
            reinterpret_cast<const ushort4 *>(state_init)[c];
}

// The compact layout's rows as given at set-up: position pos[s] of the
// caller's row lists slot s, and every bond counts.
__global__ void __launch_bounds__(256)
    k_row_slots(int n, int K, const int *tnode, const int *cnt,
                const long long *chunk0, const int *stride,
                const unsigned short *pos, unsigned short *rslot,
                int *n_neigh)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int p = t / ROW_LANES, sub = t % ROW_LANES;
    if (p >= n)
        return;
    const int i = tnode[p], c = cnt[p];
    for (int k = sub; k < c; k += ROW_LANES)
        rslot[(size_t)i * K + pos[slot_of(chunk0[p], stride[p], k)]] =
            (unsigned short)k;
    if (sub == 0)
        n_neigh[i] = c;
}

// A per-node array in the caller's node order: dst[tnode[p]] = src[p], w
// values per node.
__global__ void k_unperm(int n, int w, const int *tnode, const double *src,
                         double *dst)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n)
        return;
    const size_t c = (size_t)tnode[p] * w, q = (size_t)p * w;
    for (int d = 0; d < w; ++d)
        dst[c + d] = src[q + d];
}

// A per-node array in the library's node order from the caller's:
// dst[p] = src[tnode[p]], w values per node.
__global__ void k_perm(int n, int w, const int *tnode, const double *src,
                       double *dst)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n)
        return;
    const size_t c = (size_t)tnode[p] * w, q = (size_t)p * w;
    for (int d = 0; d < w; ++d)
        dst[q + d] = src[c + d];
}

// loc0 and brk at the start of a recording: brk -1 for bonds already broken
// and empty slots, else "never".
__global__ void __launch_bounds__(256)
    k_adj_init(long long nchunks, const unsigned short *loc,
               unsigned short *loc0, int *brk)
{
    const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
    if (c >= nchunks)
        return;
    const ushort4 l = reinterpret_cast<const ushort4 *>(loc)[c];
    reinterpret_cast<ushort4 *>(loc0)[c] = l;
    constexpr int NEVER = 0x7fffffff;
    reinterpret_cast<int4 *>(brk)[c] =
        make_int4(l.x == LOC_DEAD ? -1 : NEVER, l.y == LOC_DEAD ? -1 : NEVER,
                  l.z == LOC_DEAD ? -1 : NEVER, l.w == LOC_DEAD ? -1 : NEVER);
}

// 1/sqrt(q) for q in [2^-767, 2^767]: the hardware estimate y and one step of
// third order, y (1 + r/2 + 3/8 r^2) with r = 1 - q y^2, whose error is of the
// order of e^3 = 2e-22 for an estimate good to e = 6e-8.  Over 4.3e9 random q
// the relative error is at most 1.4e-16, 5.3e-17 in the mean square (two
// Newton steps, of two instructions more: 2.4e-16 and 7.3e-17).
__device__ __forceinline__ double rsqrt_cubic(double q)
{
    const double y = __builtin_amdgcn_rsq(q);
    const double r = __builtin_fma(-(q * y), y, 1.0);
    return __builtin_fma(y, r * __builtin_fma(r, 0.375, 0.5), y);
}

// 1/l0 of every slot's bond, once per recording (inv: caller id -> internal
// id), 0 where there is none.  The same reciprocal square root
// of the same squared length as the backward kernel's 1/l, so that a bond
// with l == l0 (bitwise, e.g. both ends at rest) gets 1/l0 - 1/l = 0 exactly,
// as its stretch is 0 in the forward step: a one-ulp difference there, times
// k dt, is not small.  A squared length that is 0, infinite or NaN has no
// reciprocal root; the forward step breaks such a bond before its first force,
// and 0 takes the place of 1/l0, which a dead slot multiplies by its zeros.
// Bound by the neighbours' coordinates (four scattered
// reads per bond): 105 us on the 50,820-node bar with one lane per node, 61
// with 4 lanes, 50 with 16.
__global__ void __launch_bounds__(256)
    k_adj_il0(int n, const int *cnt, const long long *chunk0,
              const int *stride, const int *gidx, const unsigned short *loc0,
              const int *inv, const double *r0, double *il0)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int p = t / ROW_LANES, sub = t % ROW_LANES;
    if (p >= n)
        return;
    const int nch = chunks_of(cnt[p]);
    const size_t b = 3 * (size_t)p;
    const double x = r0[b], y = r0[b + 1], z = r0[b + 2];
    for (int c = sub; c < nch; c += ROW_LANES) {
        const size_t k = (size_t)(chunk0[p] + (long long)c * stride[p]);
        const int4 g = reinterpret_cast<const int4 *>(gidx)[k];
        const ushort4 l = reinterpret_cast<const ushort4 *>(loc0)[k];
        const int gv[4] = {g.x, g.y, g.z, g.w};
        const unsigned short lv[4] = {l.x, l.y, l.z, l.w};
        double v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t bj = 3 * (size_t)inv[(uint32_t)gv[q] & KEYM];
            const double ex = r0[bj] - x;
            const double ey = r0[bj + 1] - y;
            const double ez = r0[bj + 2] - z;
            const double q0 = sq3<true>(ex, ey, ez);
            v[q] = lv[q] != LOC_DEAD && q0 > 0.0 && q0 < __builtin_inf()
                       ? rsqrt_cubic(q0)
                       : 0.0;
        }
        double2 *o = reinterpret_cast<double2 *>(il0) + 2 * k;
        o[0] = make_double2(v[0], v[1]);
        o[1] = make_double2(v[2], v[3]);
    }
}

// The per-node inputs of one backward step as 64-byte records, from which
// the tiles stage their halos: a = (rx, ry, rz, V), b = (mux, muy, muz, c/2)
// with r = r0 + u_n and mu = lambda_{n+1} with prescribed DOFs zeroed.
__global__ void k_adj_pack(int n, const double *r0, const double *u,
                           const double *vol, const double *c,
                           const int *flags, const double *lam, NodeRec *rec)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n)
        return;
    const size_t b = 3 * (size_t)p;
    const int f = flags[p];
    NodeRec o;
    o.a = make_double4(r0[b] + u[b], r0[b + 1] + u[b + 1],
                       r0[b + 2] + u[b + 2], vol[p]);
    o.b = make_double4(f & 1 ? 0.0 : lam[b], f & 2 ? 0.0 : lam[b + 1],
                       f & 4 ? 0.0 : lam[b + 2], 0.5 * c[p]);
    rec[p] = o;
}

struct AdjArgs {
    int ntiles, tiles_per_xcd, step;
    double dt;
    const TileInfo *tiles;
    const int *halo, *cnt, *brk;
    const NodeRec *rec;  // the records of this step
    const unsigned short *loc0;  // loc at the start of the recording
    const double *il0;
    double *lam_out, *gradc;
    // if set, the records of the step before (k_adj_pack's, from u_prev =
    // u_{n-1} and lambda_n) are written too
    NodeRec *rec_next;
    const double *u_prev, *r0;
    const int *flags;
};

// One backward step on the step kernel's tiles: the tile's halo records
// (k_adj_pack) are staged into LDS piece-major, as in k_step, and every bond
// of a node reads its neighbour from there.  LPN lanes per node take its
// 4-bond chunks round-robin; a slot is live in step n if it broke at a step
// > n (brk, -1 where it held no bond at the start of the recording), and
// reads the far entry 0, whose terms are zero, otherwise.  They are zero as
// products with 0, so a node whose own values are infinite, NaN or so large
// that they become infinite here skips its dead slots in a loop of its own.
//
// What bounds it: the chunks' streams (14 B a slot: loc0, brk, 1/l0) and the
// latency of each, so they are requested two rounds ahead; the arithmetic is
// contracted (43 issue slots per bond where the plain form took 59): 27.3 ->
// 23.5 us on the 50,820-node bar, and 19.6 with tiles even over the CUs and
// 41 slots, 3.8 TB/s of streams.
template <int LPN>
__global__ __launch_bounds__(1024) void k_adj_tile(AdjArgs a)
{
    __shared__ double2 lds[LDS_BYTES / sizeof(double2)];
    constexpr unsigned PB = 16u * LDS_CAP_PMB;
    const int tile = (blockIdx.x % XCDS) * a.tiles_per_xcd + blockIdx.x / XCDS;
    if (tile >= a.ntiles)
        return;
    const TileInfo ti = a.tiles[tile];
    char *ldsb = reinterpret_cast<char *>(lds);
    const int l = threadIdx.x / LPN;
    const int sub = threadIdx.x % LPN;
    const bool valid = l < ti.nodes;
    HaloLoads<> hl;
    hl.request(a.halo + ti.halo_off, (unsigned)ti.halo);
    // chunk k's streams; chunk rows past the tile's last are not used, and
    // their loads stay at the row before it
    const long long row0 = ti.chunk_off + (valid ? l : 0);
    const ushort4 *L4 = reinterpret_cast<const ushort4 *>(a.loc0) + row0;
    const int4 *B4 = reinterpret_cast<const int4 *>(a.brk) + row0;
    const double2 *I2 = reinterpret_cast<const double2 *>(a.il0) + 2 * row0;
    const int last = max(ti.nch, 1) - 1;
    struct Stream {
        uint2 loc;
        int4 brk;
        double2 ia, ib;
    };
    auto stream_at = [&](int c) {
        const unsigned k = (unsigned)min(c, last) * (unsigned)ti.nodes;
        Stream v;
        v.loc = reinterpret_cast<const uint2 *>(L4)[k];
        v.brk = B4[k];
        v.ia = I2[2u * k];
        v.ib = I2[2u * k + 1u];
        return v;
    };
    Stream qa = stream_at(sub), qb = stream_at(sub + LPN);
    const uint32_t i = (uint32_t)(ti.node_off + (valid ? l : 0));
    const NodeRec own = a.rec[i];
    const int cnt = valid ? a.cnt[i] : 0;
    hl.stage<true>(a.rec, a.halo + ti.halo_off, (unsigned)ti.halo, ldsb, PB);
    if (threadIdx.x < 4)
        far_entry<true>(ldsb, PB);
    __syncthreads();

    const double rm[3] = {own.a.x, own.a.y, own.a.z};
    const double mum[3] = {own.b.x, own.b.y, own.b.z};
    const double vm = own.a.w, cm = own.b.w;
    double jt[3] = {0.0, 0.0, 0.0};
    double gc = 0.0;
    // with r below half of the far entry's coordinate a dead slot's 1/l is at
    // most 2^-299; 1/l0 is at most 2^537
    bool plain = fabs(cm) < 0x1p400 && fabs(vm) < __builtin_inf();
    for (int d = 0; d < 3; ++d)
        plain &= fabs(rm[d]) < 0x1p299 && fabs(mum[d]) < __builtin_inf();
    auto bond = [&](auto skip, unsigned ev, int brk, double il0) {
        if (skip && brk <= a.step)
            return;
        const char *pe = ldsb + (brk > a.step ? ev : (unsigned)LOC_DEAD);
        const double2 p0 = *reinterpret_cast<const double2 *>(pe);
        const double2 p1 = *reinterpret_cast<const double2 *>(pe + PB);
        const double2 p2 = *reinterpret_cast<const double2 *>(pe + 2 * PB);
        const double2 p3 = *reinterpret_cast<const double2 *>(pe + 3 * PB);
        const double dd[3] = {p0.x - rm[0], p0.y - rm[1], p1.x - rm[2]};
        const double muj[3] = {p2.x, p2.y, p3.x};
        const double vj = p1.y;
        double w[3];
#pragma unroll
        for (int d = 0; d < 3; ++d)
            w[d] = __builtin_fma(vm, muj[d], -(vj * mum[d]));
        // 1/l from the reciprocal square root of the squared length: no
        // square root or division in the loop
        const double il = rsqrt_cubic(sq3<true>(dd[0], dd[1], dd[2]));
        const double psi = il0 - il;
        const double kk = cm + p3.y;  // (c_m + c_j)/2
        const double dw = __builtin_fma(
            dd[2], w[2], __builtin_fma(dd[1], w[1], dd[0] * w[0]));
        const double kp = kk * psi;
        const double kd = (kk * dw) * (il * il * il);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            jt[d] = __builtin_fma(kp, w[d], __builtin_fma(kd, dd[d], jt[d]));
        gc = __builtin_fma(psi, dw, gc);
    };
    // rounds as in k_step
    const int cmax = __builtin_amdgcn_readfirstlane(cnt);
    auto round = [&](auto skip, const Stream &v, int k) {
        if (sub + LPN * k > last)
            return;
        bond(skip, v.loc.x & 0xffffu, v.brk.x, v.ia.x);
        bond(skip, v.loc.x >> 16, v.brk.y, v.ia.y);
        if (16 * (LPN * k / 4) + 8 < cmax) {
            bond(skip, v.loc.y & 0xffffu, v.brk.z, v.ib.x);
            bond(skip, v.loc.y >> 16, v.brk.w, v.ib.y);
        }
    };
    const int rounds = (chunks_of(cmax) + LPN - 1) / LPN;
    if (valid && plain) {
        for (int k = 0; k < rounds; k += 2) {
            round(std::false_type{}, qa, k);
            qa = stream_at(sub + LPN * (k + 2));
            if (k + 1 >= rounds)
                break;
            round(std::false_type{}, qb, k + 1);
            qb = stream_at(sub + LPN * (k + 3));
        }
    } else if (valid) {
        for (int k = 0; k < rounds; ++k)
            round(std::true_type{}, stream_at(sub + LPN * k), k);
    }
    gc *= -0.5;
    jt[0] = node_sum<LPN>(jt[0]);
    jt[1] = node_sum<LPN>(jt[1]);
    jt[2] = node_sum<LPN>(jt[2]);
    gc = node_sum<LPN>(gc);
    if (!valid)
        return;
    const size_t b = 3 * (size_t)i;
    const int fl = a.rec_next ? a.flags[i] : 0;
    for (int d = sub; d < 4; d += LPN) {
        if (d < 3) {
            const double lam = mum[d] + a.dt * jt[d];
            a.lam_out[b + d] = lam;
            if (a.rec_next) {
                // as k_adj_pack: r = r0 + u_{n-1}, mu = lambda_n masked
                double *ra = reinterpret_cast<double *>(&a.rec_next[i].a);
                double *rb = reinterpret_cast<double *>(&a.rec_next[i].b);
                ra[d] = a.r0[b + d] + a.u_prev[b + d];
                rb[d] = (fl >> d) & 1 ? 0.0 : lam;
            }
        } else if (a.rec_next) {
            reinterpret_cast<double *>(&a.rec_next[i].a)[3] = vm;
            reinterpret_cast<double *>(&a.rec_next[i].b)[3] = cm;
        }
    }
    if (sub == 0)
        a.gradc[i] += a.dt * gc;
}

}  // namespace pdk

// Device scratch of pd_monitor_noalloc: the per-block partial sums of
// k_monitor_part, then the staged outputs of k_monitor_final (6 model sums
// and 5 per tip group), for at most NOALLOC_MAX_GROUPS tip groups.  File
// scope: every device the library runs on holds its own copy (64 KiB) until
// the process ends.  Host code reaches it only through the address that
// hipGetSymbolAddress returns for the current device.
constexpr int NOALLOC_MAX_GROUPS = 1024;
constexpr size_t NOALLOC_DOUBLES = (size_t)pdk::MON_BLOCKS * pdk::MON_SUMS +
                                   pdk::MON_SUMS + 5 * NOALLOC_MAX_GROUPS;
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

namespace {

using namespace pdk;

template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void release()
    {
        if (p)
            (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    hipError_t alloc(size_t count)
    {
        release();
        if (count == 0)
            return hipSuccess;
        const hipError_t e =
            hipMalloc(reinterpret_cast<void **>(&p), count * sizeof(T));
        if (e == hipSuccess)
            n = count;
        else
            p = nullptr;  // n stays 0: a later call allocates again
        return e;
    }
    // room for count values; what is there is kept if it suffices
    hipError_t reserve(size_t count)
    {
        return p && n >= count ? hipSuccess : alloc(count);
    }
};

}  // namespace

struct pd_sim {
    int device = 0;
    int integrator = PD_EULER, layout = PD_LAYOUT_SLOT;
    double dt = 0.0, damping = 0.0;
    int n = 0, K = 0;
    int tension_only = 0;
    int lpn = 4, tile_nodes = 128;  // pd_set_launch's values
    bool launch_given = false;      // pd_set_launch was called
    int lanes = 4;      // lanes per node of the steps (lpn, unless not given)
    int tile_cap = 128; // most nodes of a tile of the current tiling
    int cus = 256;
    int hmax = 0;           // halo capacity of a tile (LDS budget)
    int hstride = 0;        // largest halo of the current tiles
    size_t lds_budget = 0;  // bytes of LDS a workgroup may use
    int ntiles = 0;
    size_t nslots = 0;  // bond slots of the tiles (loc holds LOC_SLACK more)
    bool coords_core = false;  // coordinates in bond_fast's range
    bool odd_corr = false;     // some bond's correction is not finite
    bool odd_tables = false;   // set_tables
    double tab_scale = 1.0;    // set_tables
    bool retile_pending = false;  // tile_nodes changed since the tiling
    bool has_buffers = false, has_corr = false, has_btypes = false,
         has_cnode = false;
    bool lost = false;  // has_buffers was taken back (run_failed)
    int nregimes = 1, nbond_types = 1;
    double k = 0.0, s0 = 0.0;
    int cur = 0;
    bool exact = false;  // exact-order Euler step (k_exact_step)
    // a replay's u_{n+1} (a slot of the segment buffer); null: u
    double *u_out = nullptr;
    DevBuf<int> nlow, nup;  // exact step: lower slots, upper-list length
    DevBuf<unsigned> ford;  // exact step: fold lists
    DevBuf<long long> tile0;  // compact layout: first chunk of a node's tile
    DevBuf<double> wbuf;  // a per-node array on its way to or from the host
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;

    // build inputs in the caller's node order; uploaded in tile order by
    // pd_create_buffers, which fixes that order
    std::vector<double> h_coords, h_vol, h_bcv, h_fbcv, h_dens, h_cnode;
    std::vector<int> h_flags;
    std::vector<double> h_corr;    // (N,K) as given to build
    std::vector<int> h_btypes;     // (N,K)
    std::vector<int> perm;         // internal node p -> caller's node id
    // the tiling's inputs: a later pd_create_buffers with the same ones
    // (compared value by value) keeps the tiles and slots
    bool plan = false, plan_nlin = false;
    int plan_tile_nodes = 0, plan_lpn = 0, plan_nregimes = 0, plan_types = 0;
    std::unique_ptr<int[]> plan_nlist;  // (N,K)
    std::vector<int> plan_nneigh;       // compact layout
    DevBuf<unsigned short> loc_init, state_init;  // per slot, as set up
    DevBuf<int> inv;  // caller's node id -> internal node (adjoint)
    std::vector<int> h_group;      // tiling groups (empty: one group)

    DevBuf<NodeRec> rec[2];
    DevBuf<TileInfo> tiles;
    DevBuf<double> dens1;
    DevBuf<double> r0, vol, u, ud, udd, force, body_force, bcv, fbcv, dens,
        damage, cnode, corr, k_tab, s_tab, pc_tab;
    DevBuf<double> cnode_caller;  // a field given on the device (caller order)
    DevBuf<int> meta;  // cnt | flags << 16
    DevBuf<int> flags, family, cnt, tnode, halo, gidx, stride, nlist_ref,
        n_neigh, out_nlist, out_nneigh;
    DevBuf<long long> chunk0;
    DevBuf<unsigned short> loc, pos, state, rslot;
    DevBuf<unsigned long long> counter;

    // adjoint recording (Euler, node field): break steps, checkpoints
    bool adj_recording = false, adj_ready = false, adj_replay = false;
    bool adj_keep = true;  // pd_adjoint_keep
    bool adj_all = false;  // u of every recorded step is in seg
    // the model or the launch shape was set anew since the recording began:
    // its steps are replayed with the new ones
    bool adj_changed = false;
    int adj_nsteps = 0, adj_every = 0, step_counter = 0;
    std::vector<double> adj_dmag, adj_fmag;
    DevBuf<int> brk;
    DevBuf<unsigned short> loc0;
    DevBuf<double> il0;    // 1/l0 per slot
    DevBuf<NodeRec> arec[2];  // records of a backward step, ping-pong
    DevBuf<double> ckpt, seg, lam[2], gradc, fin_u, fin_force, fin_bforce;

    // monitored sums: tip entries (caller's node, dof) grouped, in order
    std::vector<int> h_tip_node, h_tip_dof, h_tip_off;
    DevBuf<int> tip_q, tip_off;  // internal DOF index 3p + d; group offsets
    DevBuf<double> mon_part, mon_out;
};

namespace {

void run_parallel(int n, const std::function<void(int, int)> &fn,
                  int min_per_thread = 4096)
{
    const unsigned hw = std::thread::hardware_concurrency();
    int nt = (int)std::min<unsigned>(hw ? hw : 1, 16);
    if (n < min_per_thread)
        nt = 1;
    std::vector<std::thread> th;
    const int chunk = (n + nt - 1) / nt;
    for (int t = 0; t < nt; ++t) {
        const int lo = t * chunk, hi = std::min(n, lo + chunk);
        if (lo >= hi)
            break;
        th.emplace_back(fn, lo, hi);
    }
    for (auto &x : th)
        x.join();
}

template <typename T>
hipError_t upload(DevBuf<T> &d, const T *h, size_t count)
{
    hipError_t e = d.alloc(count);
    if (e != hipSuccess || count == 0)
        return e;
    return hipMemcpy(d.p, h, count * sizeof(T), hipMemcpyHostToDevice);
}

// dst[p] = src[perm[p]] for rows of w values (caller order -> tile order)
template <typename T>
std::vector<T> to_internal(const std::vector<int> &perm, const T *src, int w)
{
    std::vector<T> dst(perm.size() * (size_t)w);
    for (size_t p = 0; p < perm.size(); ++p)
        for (int d = 0; d < w; ++d)
            dst[p * w + d] = src[(size_t)perm[p] * w + d];
    return dst;
}

// Upload rows of w values given in the caller's order into tile order.
template <typename T>
hipError_t upload_perm(DevBuf<T> &d, const std::vector<int> &perm,
                       const T *src, int w)
{
    const std::vector<T> v = to_internal(perm, src, w);
    return upload(d, v.data(), v.size());
}

// Download rows of w values in tile order into the caller's order.
// n*w doubles of an internal-order device array into dst in the caller's
// node order: reordered on the device, then one copy.
int download_caller(pd_sim *s, double *dst, const double *src, int w)
{
    const size_t count = (size_t)s->n * w;
    if (count == 0)
        return PD_OK;
    if (s->wbuf.n < count)
        HIPCHK(s->wbuf.alloc(count));
    hipLaunchKernelGGL(k_unperm, dim3((s->n + 255) / 256), dim3(256), 0,
                       s->stream, s->n, w, s->tnode.p, src, s->wbuf.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(dst, s->wbuf.p, count * sizeof(double),
                          hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    return PD_OK;
}

// Blocks of 256 threads for that many lanes per node.
unsigned row_blocks(int n, int lanes)
{
    return (unsigned)(((long long)n * lanes + 255) / 256);
}

// Blocks of 256 threads for one thread per chunk of slots.
unsigned chunk_blocks(const pd_sim *s)
{
    return (unsigned)((s->nslots / 4 + 255) / 256);
}

hipError_t launch_export(pd_sim *s, int rows, double *damage,
                         double *u_out = nullptr)
{
    const auto go = [&](auto kernel, int lanes) {
        hipLaunchKernelGGL(kernel, dim3(row_blocks(s->n, lanes)), dim3(256),
                           0, s->stream, s->n, s->K, s->layout, rows,
                           s->tnode.p, s->cnt.p, s->chunk0.p, s->stride.p,
                           s->loc.p, s->gidx.p, s->pos.p, s->family.p,
                           s->n_neigh.p, s->out_nlist.p, s->out_nneigh.p,
                           damage, s->u.p, u_out);
    };
    if (s->layout == PD_LAYOUT_COMPACT)
        go(k_export<1>, 1);  // counts are kept: one lane per node
    else if (rows)
        go(k_export<ROW_LANES>, ROW_LANES);
    else
        go(k_export<CHUNK_LANES>, CHUNK_LANES);
    return hipGetLastError();
}

int check_sim(pd_sim *s)
{
    if (!s)
        return fail(PD_E_ARG, "null simulation handle");
    HIPCHK(hipSetDevice(s->device));
    return PD_OK;
}

// What a call that needs the simulation's state says without it.
int no_buffers(const pd_sim *s)
{
    return fail(PD_E_STATE,
                s->lost ? "a call failed on its way and left no whole state: "
                          "call pd_create_buffers"
                        : "pd_create_buffers has not been called");
}

int dm_of(const pd_sim *s)
{
    if (s->nregimes > 1 || s->nbond_types > 1)
        return DM_NLIN;
    return s->has_cnode ? DM_FIELD : DM_PMB;
}

StepArgs make_args(pd_sim *s)
{
    StepArgs a;
    a.K = s->K;
    a.ntiles = s->ntiles;
    a.tiles_per_xcd = (s->ntiles + XCDS - 1) / XCDS;
    a.integrator = s->integrator;
    a.layout = s->layout;
    a.has_corr = s->has_corr ? 1 : 0;
    a.absmask = s->tension_only ? 0xffffffffu : 0x7fffffffu;
    a.nregimes = s->nregimes;
    a.ntab = s->nregimes * s->nbond_types;
    a.dt = s->dt;
    a.damping = s->damping;
    a.s0h = s->s0 * 0.5;
    // coordinates outside the range that bond_fast relies on, or corrections
    // or table values whose product with a dead slot's zeros is not zero:
    // every bond takes the exact path
    a.lim = !s->coords_core || s->odd_corr || s->odd_tables ? -1.0
            : dm_of(s) == DM_NLIN ? 1.0
                                  : fast_limit(a.s0h);
    a.rec_old = s->rec[s->cur].p;
    a.rec_new = s->rec[1 - s->cur].p;
    a.tiles = s->tiles.p;
    a.tnode = s->tnode.p;
    a.halo = s->halo.p;
    a.u = s->u.p;
    a.u_out = s->u_out ? s->u_out : s->u.p;
    a.ud = s->ud.p;
    a.udd = s->udd.p;
    a.force = s->force.p;
    a.body_force = s->body_force.p;
    a.bcv = s->bcv.p;
    a.fbcv = s->fbcv.p;
    a.dens = s->dens.p;
    a.dens1 = s->dens1.p;
    a.meta = s->meta.p;
    a.loc = s->loc.p;
    a.gidx = s->gidx.p;
    a.corr = s->corr.p;
    a.state = s->state.p;
    a.k_tab = s->k_tab.p;
    a.s_tab = s->s_tab.p;
    a.pc_tab = s->pc_tab.p;
    a.rslot = s->rslot.p;
    a.n_neigh = s->n_neigh.p;
    a.cnode = s->cnode.p;
    a.brk = s->adj_recording ? s->brk.p : nullptr;
    a.step = s->step_counter;
    a.nlow = s->nlow.p;
    a.nup = s->nup.p;
    a.ford = s->ford.p;
    a.kx = s->k;
    // exact_fast's interval; empty where its range does not hold
    const double ak = std::fabs(s->k);
    const bool core = s->coords_core && ak >= 0x1p-100 && ak <= 0x1p100 &&
                      s->s0 < 0x1p300;
    a.xhi = core ? s->s0 : -1.0;
    a.xlo = s->tension_only ? -0.5 : std::max(-s->s0, -0.5);
    return a;
}

// Threads of a workgroup: the tiles' nodes, in whole wavefronts.
unsigned block_of(const pd_sim *s, int lanes)
{
    return ((unsigned)(s->tile_cap * lanes) + 63u) & ~63u;
}

// Whether tiles of at most `halo` halo entries run the narrow form at four
// lanes per node: it takes blocks of at most 512, and pays where a CU has
// more than two tiles to run (us a step, wide / narrow: 1,038,230-node beam
// 257 / 247, 263,407 nodes 72.7 / 70.1, 204,800 nodes 57.9 / 56.3, 141,143
// nodes 43.1 / 42.4, 100 steps of a 93,433-node plate 1367 / 1307; with two or
// fewer the wide form's early reads of
// the node's state are worth more).
bool narrow_fits(const pd_sim *s, int ntiles, int halo)
{
    return ntiles > 2 * s->cus && halo < LDS_CAP_NARROW &&
           block_of(s, 4) <= 512;
}

template <int DM, int LPN, bool CLA>
hipError_t launch_cla(pd_sim *s, const StepArgs &a, double dmag, double fmag)
{
    const unsigned grid = (unsigned)XCDS * a.tiles_per_xcd;
    const unsigned block = block_of(s, LPN);
    // the n-linear model breaks by regimes, not by the sign mode
    const bool tens = DM != DM_NLIN && a.absmask == 0xffffffffu;
    if constexpr (DM == DM_PMB && LPN == 4 && CLA) {
        if (!a.has_corr && narrow_fits(s, s->ntiles, s->hstride)) {
            if (tens)
                hipLaunchKernelGGL((k_step<DM, LPN, false, true, CLA, true>),
                                   dim3(grid), dim3(block), 0, s->stream, a,
                                   dmag, fmag);
            else
                hipLaunchKernelGGL((k_step<DM, LPN, false, false, CLA, true>),
                                   dim3(grid), dim3(block), 0, s->stream, a,
                                   dmag, fmag);
            return hipGetLastError();
        }
    }
    if (a.has_corr && tens)
        hipLaunchKernelGGL((k_step<DM, LPN, true, DM != DM_NLIN, CLA, false>),
                           dim3(grid), dim3(block), 0, s->stream, a, dmag,
                           fmag);
    else if (a.has_corr)
        hipLaunchKernelGGL((k_step<DM, LPN, true, false, CLA, false>),
                           dim3(grid), dim3(block), 0, s->stream, a, dmag,
                           fmag);
    else if (tens)
        hipLaunchKernelGGL((k_step<DM, LPN, false, DM != DM_NLIN, CLA, false>),
                           dim3(grid), dim3(block), 0, s->stream, a, dmag,
                           fmag);
    else
        hipLaunchKernelGGL((k_step<DM, LPN, false, false, CLA, false>),
                           dim3(grid), dim3(block), 0, s->stream, a, dmag,
                           fmag);
    return hipGetLastError();
}

// The slot layout steps with the OpenCL arithmetic; the compact layout (the
// Cython path: scalar stiffness, no corrections) with the Cython one.
template <int DM, int LPN>
hipError_t launch_one(pd_sim *s, const StepArgs &a, double dmag, double fmag)
{
    if (a.layout == PD_LAYOUT_SLOT)
        return launch_cla<DM, LPN, true>(s, a, dmag, fmag);
    const unsigned grid = (unsigned)XCDS * a.tiles_per_xcd;
    const unsigned block = block_of(s, LPN);
    if (DM != DM_PMB || a.has_corr)
        return hipErrorInvalidValue;  // rejected before launch
    if (a.absmask == 0xffffffffu)
        hipLaunchKernelGGL((k_step<DM_PMB, LPN, false, true, false, false>),
                           dim3(grid), dim3(block), 0, s->stream, a, dmag,
                           fmag);
    else
        hipLaunchKernelGGL((k_step<DM_PMB, LPN, false, false, false, false>),
                           dim3(grid), dim3(block), 0, s->stream, a, dmag,
                           fmag);
    return hipGetLastError();
}

template <int DM>
hipError_t launch_dm(pd_sim *s, const StepArgs &a, double dmag, double fmag)
{
    switch (s->lanes) {
    case 1:
        return launch_one<DM, 1>(s, a, dmag, fmag);
    case 2:
        return launch_one<DM, 2>(s, a, dmag, fmag);
    case 4:
        return launch_one<DM, 4>(s, a, dmag, fmag);
    default:
        return launch_one<DM, 8>(s, a, dmag, fmag);
    }
}


// One backward step's k_adj_tile, with the step kernel's grid and block.
hipError_t launch_adjoint(pd_sim *s, const AdjArgs &a)
{
    const unsigned grid = (unsigned)XCDS * a.tiles_per_xcd;
    const dim3 block(block_of(s, s->lanes));
    switch (s->lanes) {
    case 1:
        hipLaunchKernelGGL(k_adj_tile<1>, dim3(grid), block, 0, s->stream, a);
        break;
    case 2:
        hipLaunchKernelGGL(k_adj_tile<2>, dim3(grid), block, 0, s->stream, a);
        break;
    case 4:
        hipLaunchKernelGGL(k_adj_tile<4>, dim3(grid), block, 0, s->stream, a);
        break;
    default:
        hipLaunchKernelGGL(k_adj_tile<8>, dim3(grid), block, 0, s->stream, a);
        break;
    }
    return hipGetLastError();
}

// Ends a recording; its memory stays for the next one.
void adjoint_end(pd_sim *s)
{
    s->adj_recording = s->adj_ready = s->adj_replay = false;
    s->adj_all = s->adj_changed = false;
    s->adj_nsteps = s->adj_every = s->step_counter = 0;
    s->adj_dmag.clear();
    s->adj_fmag.clear();
}

void adjoint_release(pd_sim *s)
{
    adjoint_end(s);
    s->brk.release();
    s->loc0.release();
    s->il0.release();
    s->arec[0].release();
    s->arec[1].release();
    s->ckpt.release();
    s->seg.release();
    s->lam[0].release();
    s->lam[1].release();
    s->gradc.release();
    s->fin_u.release();
    s->fin_force.release();
    s->fin_bforce.release();
}

// Bookkeeping of an adjoint recording after each forward step: the step's
// magnitudes, and a checkpoint of u every adj_every steps.
int after_step(pd_sim *s, double dmag, double fmag)
{
    if (s->adj_replay)
        return PD_OK;
    if (!s->adj_recording) {
        s->adj_ready = false;  // stepped past a finished recording
        return PD_OK;
    }
    s->adj_dmag.push_back(dmag);
    s->adj_fmag.push_back(fmag);
    ++s->step_counter;
    const size_t B = 3 * (size_t)s->n;
    if (!s->adj_all && s->step_counter % s->adj_every == 0 &&
        s->step_counter < s->adj_nsteps)
        HIPCHK(hipMemcpyAsync(s->ckpt.p + (s->step_counter / s->adj_every) * B,
                              s->u.p, B * sizeof(double),
                              hipMemcpyDeviceToDevice, s->stream));
    if (s->step_counter == s->adj_nsteps) {
        s->adj_recording = false;
        s->adj_ready = true;
    }
    return PD_OK;
}

int tiles_pending()
{
    return fail(PD_E_STATE, "tile_nodes changed: call pd_create_buffers "
                            "to re-tile before stepping");
}

// One step; `last`: the last of its run, whose u and forces are stored.
int launch_step(pd_sim *s, double dmag, double fmag, bool last)
{
    if (s->retile_pending)
        return tiles_pending();
    if (s->ntiles == 0) {
        s->cur = 1 - s->cur;
        return PD_OK;
    }
    if (s->layout == PD_LAYOUT_COMPACT && dm_of(s) != DM_PMB)
        return fail(PD_E_STATE, "the compact (Cython) layout steps the "
                                "scalar stiffness model only");
    if (s->exact && (s->layout != PD_LAYOUT_COMPACT ||
                     s->integrator != PD_EULER || dm_of(s) != DM_PMB ||
                     s->has_corr || !s->ford.p))
        return fail(PD_E_STATE, "the exact-order step needs the compact "
                                "layout, the Euler integrator and the scalar "
                                "model without corrections");
    if (s->exact && (s->lpn != 4 || s->tile_nodes > EXACT_NODES))
        return fail(PD_E_STATE, "the exact-order step runs 4 lanes per node "
                                "and tiles of at most 128 nodes");
    if (s->exact && !exact_rows_fit(s->K))
        return fail(PD_E_LIMIT, "the exact-order step takes at most 4074 "
                                "neighbours per node");
    StepArgs a = make_args(s);
    a.store = last ? STORE_U | STORE_F : 0;
    // a replay stores every u, a recording those that it keeps: all, each in
    // a slot of its own (and the last step's in u), or its checkpoints'
    double *slot = nullptr;
    if (s->u_out) {
        a.store |= STORE_U;
    } else if (s->adj_recording) {
        const int next = s->step_counter + 1;
        if (next % s->adj_every == 0 || s->adj_all)
            a.store |= STORE_U;
        if (s->adj_all && next < s->adj_nsteps)
            a.u_out = slot = s->seg.p + (size_t)next * 3 * s->n;
    }
    hipError_t e;
    if (s->exact) {
        const dim3 grid(XCDS * a.tiles_per_xcd);
        if (s->tile_cap <= EXACT_WIDE_NODES)
            hipLaunchKernelGGL(k_exact_step<8>, grid, dim3(block_of(s, 8)), 0,
                               s->stream, a, dmag, fmag);
        else
            hipLaunchKernelGGL(k_exact_step<4>, grid, dim3(block_of(s, 4)), 0,
                               s->stream, a, dmag, fmag);
        e = hipGetLastError();
    } else {
        switch (dm_of(s)) {
        case DM_NLIN:
            e = launch_dm<DM_NLIN>(s, a, dmag, fmag);
            break;
        case DM_FIELD:
            e = launch_dm<DM_FIELD>(s, a, dmag, fmag);
            break;
        default:
            e = launch_dm<DM_PMB>(s, a, dmag, fmag);
            break;
        }
    }
    if (e != hipSuccess)
        return fail(PD_E_HIP, std::string("step kernel launch: ") +
                                  hipGetErrorString(e));
    s->cur = 1 - s->cur;
    if (slot && last)
        HIPCHK(hipMemcpyAsync(s->u.p, slot, 3 * (size_t)s->n * sizeof(double),
                              hipMemcpyDeviceToDevice, s->stream));
    return after_step(s, dmag, fmag);
}

// After an error on the way of a run, some of whose steps have moved the
// records and the bonds but stored neither u nor forces, of a replay, or of a
// change of the model, whose records may be of both: there is no state to
// read or to go on from.
void run_failed(pd_sim *s)
{
    s->has_buffers = false;
    s->lost = true;
    adjoint_end(s);
}

// run_failed for a call that leaves while its state is away.
struct StateGuard {
    pd_sim *s;
    bool away;
    ~StateGuard()
    {
        if (away)
            run_failed(s);
    }
};

// The tip entries as internal DOF indices 3p + d for the current tiling.
int upload_tips(pd_sim *s)
{
    if (s->h_tip_off.empty() || s->perm.empty())
        return PD_OK;
    std::vector<int> inv(s->n);
    for (int p = 0; p < s->n; ++p)
        inv[s->perm[p]] = p;
    std::vector<int> q(s->h_tip_node.size());
    for (size_t e = 0; e < q.size(); ++e)
        q[e] = 3 * inv[s->h_tip_node[e]] + s->h_tip_dof[e];
    HIPCHK(upload(s->tip_q, q.data(), q.size()));
    HIPCHK(upload(s->tip_off, s->h_tip_off.data(), s->h_tip_off.size()));
    return PD_OK;
}

// (Re)write both record buffers from r0, V, the device u and c.
int refresh_records(pd_sim *s)
{
    const int blocks = (s->n + 255) / 256;
    const int dm = dm_of(s);
    // the exact-order step reads V itself
    const double wscale =
        s->exact         ? 1.0
        : dm == DM_PMB   ? 4.0 * s->k
        : dm == DM_FIELD ? 2.0
                         : 1.0 / s->tab_scale;
    hipLaunchKernelGGL(k_records, dim3(blocks), dim3(256), 0, s->stream, s->n,
                       wscale, s->layout == PD_LAYOUT_SLOT ? 1 : 0, s->r0.p,
                       s->vol.p, s->u.p,
                       s->has_cnode ? s->cnode.p : nullptr, s->rec[0].p,
                       s->rec[1].p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s->stream));
    s->cur = 0;
    return PD_OK;
}

// The compact layout's fold lists from its rows and live bonds.
int fold_lists(pd_sim *s)
{
    if (s->layout != PD_LAYOUT_COMPACT)
        return PD_OK;
    hipLaunchKernelGGL(k_fold_lists, dim3((s->n + 255) / 256), dim3(256), 0,
                       s->stream, s->n, s->K, s->tnode.p, s->cnt.p,
                       s->chunk0.p, s->stride.p, s->tile0.p, s->gidx.p,
                       s->loc.p, s->rslot.p, s->n_neigh.p, s->nlow.p,
                       s->nup.p, s->ford.p);
    HIPCHK(hipGetLastError());
    return PD_OK;
}

// The launch shape of the next tiling.  Up to WAVES_EVEN tiles per CU the tiles
// are as small as keeps that number, so that every CU gets as many of them: a
// mesh of less than one workgroup per CU is one workgroup's latency, most of
// it the issue of its rounds, and of one and a half the latency of two on half
// of the CUs.  No smaller than 32 nodes at eight lanes, 48 at four (their
// halos then cost more), and eight lanes per node where the caller set no
// shape and the tiles are that small.  Tiles change no result; lanes change
// the order of a node's sum.  us a step, scalar model, tiles of 128 / the
// rule, four lanes, and the rule with eight: 2,560 nodes 10.6 / 8.4, 6.7;
// 5,000 nodes 11.6 / 9.1, 6.8; 20,655 nodes 12.4 / 12.0, 12.4 (not taken).
// Four lanes, 128 / the rule: 35,420 nodes 18.2 / 15.0 (n-linear 19.8 / 15.9,
// exact order 24.0 / 20.0), 50,820 nodes 19.0 / 18.7, 75,900 nodes 25.5 / 24.2
// (28.3 / 26.2, 35.1 / 33.0), 111,320 nodes 32.3 / 31.5 (36.8 / 34.3), 141,143
// nodes 38.9 / 38.7 (43.3 / 41.6, 54.5 / 53.7); from six tiles per CU on
// nothing is gained, or lost to the halos (170,810 nodes, exact order: 64.5 /
// 72.2).  A tile more than a multiple of the CUs costs what the multiple
// gains: 50,820 nodes in 530 tiles 23.1.
constexpr int WAVES_EVEN = 5;

void set_shape(pd_sim *s)
{
    if (!s->launch_given)
        s->lanes = s->n <= 48 * s->cus ? 8 : s->lpn;
    const int least = s->lanes == 8 ? 32 : 48;
    // no tile spans two groups
    std::map<int, int> sizes;
    if (s->h_group.empty())
        sizes[0] = s->n;
    else
        for (int g : s->h_group)
            ++sizes[g];
    auto tiles = [&](int cap) {
        long long m = 0;
        for (const auto &g : sizes)
            m += (g.second + cap - 1) / cap;
        return m;
    };
    const long long per_cu = (tiles(s->tile_nodes) + s->cus - 1) / s->cus;
    s->tile_cap = s->tile_nodes;
    if (per_cu > WAVES_EVEN)
        return;
    while (s->tile_cap > least && tiles(s->tile_cap - 1) <= per_cu * s->cus)
        --s->tile_cap;
}

// Keeps the shape of the current tiling while the next one is worked out: it
// comes back unless the next tiling is taken.
struct ShapeGuard {
    pd_sim *s;
    const int lanes = s->lanes, tile_cap = s->tile_cap, hmax = s->hmax;
    bool taken = false;
    ~ShapeGuard()
    {
        if (taken)
            return;
        s->lanes = lanes;
        s->tile_cap = tile_cap;
        s->hmax = hmax;
    }
};

// Rows of w values given in the caller's order into tile order on the device
// (through wbuf); null clears.  On the library's stream: h is read until the
// next synchronization.
int upload_caller(pd_sim *s, DevBuf<double> &d, const double *h, int w)
{
    const size_t count = (size_t)s->n * w;
    HIPCHK(d.reserve(count));
    if (!h) {
        HIPCHK(hipMemsetAsync(d.p, 0, count * sizeof(double), s->stream));
        return PD_OK;
    }
    HIPCHK(s->wbuf.reserve(count));
    HIPCHK(hipMemcpyAsync(s->wbuf.p, h, count * sizeof(double),
                          hipMemcpyHostToDevice, s->stream));
    hipLaunchKernelGGL(k_perm, dim3((s->n + 255) / 256), dim3(256), 0,
                       s->stream, s->n, w, s->tnode.p, s->wbuf.p, d.p);
    HIPCHK(hipGetLastError());
    return PD_OK;
}

// The state of a (re)start once the bonds are set up: u, ud, udd, no force yet
// (what is there is of the run before, in the order of the tiles before), the
// fold lists and the records.  Synchronizes.
int start_state(pd_sim *s, const double *u, const double *ud,
                const double *udd)
{
    int rc = upload_caller(s, s->u, u, 3);
    if (rc == PD_OK)
        rc = upload_caller(s, s->ud, ud, 3);
    if (rc == PD_OK)
        rc = upload_caller(s, s->udd, udd, 3);
    if (rc == PD_OK)
        rc = upload_caller(s, s->force, nullptr, 3);
    if (rc == PD_OK)
        rc = upload_caller(s, s->body_force, nullptr, 3);
    if (rc == PD_OK)
        rc = fold_lists(s);
    return rc == PD_OK ? refresh_records(s) : rc;
}

// Whether a[0, count) and b[0, count) hold the same values, on as many
// threads as their size is worth.
bool same_values(const int *a, const int *b, size_t count)
{
    constexpr size_t PIECE = (size_t)1 << 19;
    const int pieces = (int)((count + PIECE - 1) / PIECE);
    std::atomic<int> differ{0};
    run_parallel(pieces, [&](int lo, int hi) {
        for (int c = lo; c < hi && !differ; ++c) {
            const size_t first = (size_t)c * PIECE;
            const size_t m = std::min(PIECE, count - first);
            if (std::memcmp(a + first, b + first, m * sizeof(int)) != 0)
                differ = 1;
        }
    }, 2);
    return !differ;
}

// Most values of a neighbour list that are kept for comparison (1 GiB).
constexpr size_t PLAN_MOST = (size_t)1 << 28;

void keep_plan(pd_sim *s, const int *nlist, const int *n_neigh, bool nlin,
               bool regimes_given)
{
    const size_t count = (size_t)s->n * s->K;
    s->plan = false;
    if (count > PLAN_MOST || (nlin && regimes_given))
        return;
    s->plan_nlist.reset(new (std::nothrow) int[count]);
    if (!s->plan_nlist)
        return;
    int *dst = s->plan_nlist.get();
    run_parallel(s->n, [&](int lo, int hi) {
        std::memcpy(dst + (size_t)lo * s->K, nlist + (size_t)lo * s->K,
                    (size_t)(hi - lo) * s->K * sizeof(int));
    });
    s->plan_nneigh.clear();
    if (s->layout == PD_LAYOUT_COMPACT)
        s->plan_nneigh.assign(n_neigh, n_neigh + s->n);
    s->plan_nlin = nlin;
    s->plan_nregimes = s->nregimes;
    s->plan_types = s->nbond_types;
    s->plan_tile_nodes = s->tile_nodes;
    s->plan_lpn = s->lanes;
    s->plan = true;
}

// The n-linear model's tables.  Values that are infinite or NaN are noted: a
// padding slot names row 0 of the tables, whether or not a bond is of that
// type.  Values so large that four times them may be infinite are taken 2^-8
// times, and the records' V_j 2^8 times (a quarter and four times beside volumes
// as large).
hipError_t set_tables(pd_sim *s, const double *k, const double *crit,
                      const double *pc)
{
    const size_t T = (size_t)s->nregimes * s->nbond_types;
    const auto large = [](double v) { return std::fabs(v) > 0x1p1000; };
    s->tab_scale = 1.0;
    if (std::any_of(k, k + T, large) || std::any_of(pc, pc + T, large))
        s->tab_scale = std::any_of(s->h_vol.begin(), s->h_vol.end(), large)
                           ? 0x1p-2
                           : 0x1p-8;
    std::vector<double> ks(k, k + T), ps(pc, pc + T);
    s->odd_tables = false;
    for (size_t t = 0; t < T; ++t) {
        ks[t] *= s->tab_scale;
        ps[t] *= s->tab_scale;
        s->odd_tables |= !std::isfinite(4.0 * ks[t]) ||
                         !std::isfinite(2.0 * ps[t]);
    }
    hipError_t e = upload(s->k_tab, ks.data(), T);
    if (e == hipSuccess)
        e = upload(s->s_tab, crit, T);
    return e == hipSuccess ? upload(s->pc_tab, ps.data(), T) : e;
}

// Whether the tiles and slots made by the last pd_create_buffers serve these
// arguments too: the same bonds, launch shape and damage-model tables' shape
// (node arrays, corrections, bond types and groups cannot have changed).
bool plan_holds(const pd_sim *s, const int *nlist, const int *n_neigh,
                bool nlin, int nregimes, int nbond_types, bool regimes_given)
{
    return s->plan && s->has_buffers && !regimes_given &&
           s->plan_nlin == nlin && s->plan_nregimes == nregimes &&
           s->plan_types == nbond_types &&
           s->plan_tile_nodes == s->tile_nodes && s->plan_lpn == s->lanes &&
           (s->layout != PD_LAYOUT_COMPACT ||
            same_values(s->plan_nneigh.data(), n_neigh, (size_t)s->n)) &&
           same_values(s->plan_nlist.get(), nlist, (size_t)s->n * s->K);
}

// pd_create_buffers on the tiles and slots that are there: every bond live
// again, new state and damage-model values.  What bounds it is PCIe (u, ud,
// udd) and the comparison of the lists; tiling the 50,820-node bar anew took
// 47 ms.
int restart(pd_sim *s, const double *bond_stiffness,
            const double *critical_stretch, const double *plus_cs,
            const double *u, const double *ud, const double *udd)
{
    HIPCHK(hipStreamSynchronize(s->stream));
    s->has_buffers = false;  // until the state is whole again
    adjoint_end(s);
    hipLaunchKernelGGL(k_reset_bonds, dim3(chunk_blocks(s)), dim3(256), 0,
                       s->stream, (long long)(s->nslots / 4), s->loc_init.p,
                       s->state_init.p, s->loc.p, s->state.p, s->gidx.p);
    HIPCHK(hipGetLastError());
    if (s->layout == PD_LAYOUT_COMPACT) {
        hipLaunchKernelGGL(k_row_slots, dim3(row_blocks(s->n, ROW_LANES)),
                           dim3(256), 0, s->stream, s->n, s->K, s->tnode.p,
                           s->cnt.p, s->chunk0.p, s->stride.p, s->pos.p,
                           s->rslot.p, s->n_neigh.p);
        HIPCHK(hipGetLastError());
    }
    if (s->plan_nlin) {
        HIPCHK(set_tables(s, bond_stiffness, critical_stretch, plus_cs));
    } else {
        s->k = bond_stiffness[0];
        s->s0 = critical_stretch[0];
    }
    int rc = start_state(s, u, ud, udd);
    if (rc == PD_OK && !s->tip_q.p)
        rc = upload_tips(s);
    if (rc)
        return rc;
    s->has_buffers = true;
    s->lost = false;
    s->retile_pending = false;
    return PD_OK;
}

// LDS entries of a tile's halo, chosen so that the records the bond loop
// reads together fall into different banks.  One ds_read_b128 over 16
// consecutive lanes reads a 16-byte piece of each lane's neighbour record;
// records whose entries are equal modulo HALO_BANK_GROUPS share banks, and
// distinct records in one bank are read one after another.  A row lists its
// node's neighbours as halo indices in slot order; lane
// t = l * lpn + sub takes the chunks of four slots sub, sub + lpn, ...  Read
// groups are (16 lanes, round, bond of the chunk).  Greedy: records in the
// most groups first, each to the residue least loaded over its groups among
// the entries left (entry 0 is the far node).  Returns entry - 1 for each
// halo index; the order changes no result.
constexpr int HALO_BANK_GROUPS = 16;

// Its scratch, kept from tile to tile of one thread.
struct HaloSpread {
    std::vector<int> seen, first, pairs, order, pos, rank;
    std::vector<std::pair<int, int>> found;  // (record, group)
    std::vector<unsigned short> load;

    // off[l], off[l + 1]: node l's row in nb
    const std::vector<int> &place(const std::vector<int> &off,
                                  const std::vector<int> &nb, int lpn, int H)
    {
        constexpr int NB = HALO_BANK_GROUPS;
        seen.assign(H, -1);
        first.assign(H + 1, 0);
        found.clear();
        const int lanes = ((int)off.size() - 1) * lpn;
        int ngroups = 0;
        for (int q0 = 0; q0 < lanes; q0 += 16) {
            const int q1 = std::min(q0 + 16, lanes);
            int rounds = 0;
            for (int t = q0; t < q1; ++t) {
                const int l = t / lpn;
                const int nch = chunks_of(off[l + 1] - off[l]);
                rounds = std::max(rounds, (nch - t % lpn + lpn - 1) / lpn);
            }
            for (int k = 0; k < rounds; ++k)
                for (int b = 0; b < 4; ++b) {
                    const int g = ngroups++;
                    for (int t = q0; t < q1; ++t) {
                        const int l = t / lpn, c = t % lpn + lpn * k;
                        const int p = off[l] + 16 * (c >> 2) + 8 * (b >> 1) +
                                      2 * (c & 3) + (b & 1);
                        if (p < off[l + 1] && seen[nb[p]] != g) {
                            seen[nb[p]] = g;
                            found.emplace_back(nb[p], g);
                            ++first[nb[p] + 1];
                        }
                    }
                }
        }
        int most = 0;
        for (int h = 0; h < H; ++h) {
            most = std::max(most, first[h + 1]);
            first[h + 1] += first[h];
        }
        pairs.resize(found.size());
        pos.assign(first.begin(), first.end() - 1);
        for (const auto &f : found)
            pairs[pos[f.first]++] = f.second;
        // records by descending number of groups, in index order where equal
        rank.assign(most + 2, 0);
        for (int h = 0; h < H; ++h)
            ++rank[most - (first[h + 1] - first[h]) + 1];
        for (int r = 0; r <= most; ++r)
            rank[r + 1] += rank[r];
        order.resize(H);
        for (int h = 0; h < H; ++h)
            order[rank[most - (first[h + 1] - first[h])]++] = h;
        int avail[NB] = {}, next[NB];
        for (int e = 1; e <= H; ++e)
            ++avail[e % NB];
        load.assign((size_t)ngroups * NB, 0);
        pos.resize(H);
        for (int h : order) {
            int score[NB] = {};
            for (int m = first[h]; m < first[h + 1]; ++m)
                for (int r = 0; r < NB; ++r)
                    score[r] += load[(size_t)pairs[m] * NB + r];
            int best = -1;
            for (int r = 0; r < NB; ++r)
                if (avail[r] > 0 && (best < 0 || score[r] < score[best]))
                    best = r;
            pos[h] = best;
            --avail[best];
            for (int m = first[h]; m < first[h + 1]; ++m)
                ++load[(size_t)pairs[m] * NB + best];
        }
        for (int r = 0; r < NB; ++r)
            next[r] = r == 0 ? NB : r;
        for (int h = 0; h < H; ++h) {
            const int r = pos[h];
            pos[h] = next[r] - 1;
            next[r] += NB;
        }
        return pos;
    }
};

// Tiles by recursive bisection of the initial coordinates: the nodes of each
// group (when given) are halved across their longest extent, in proportion
// to the tiles of at most `cap` nodes that each half needs, until a part is
// one tile.  Such tiles are full and nearly cubes, whose halos are smaller
// and more alike than those of runs of a Morton curve (128 nodes of a
// jittered 200 x 47 x 47 lattice: 804 entries on average and 973 at most,
// against 939 and 1283), and parts that are near in the order are near in
// space.  Returns the order of the nodes; starts gets each tile's first.
struct TilePoint {
    double x[3];
    int id;
};

struct TileRange {
    int lo, hi;
};

// One halving of p[r.lo, r.hi), which needs more than one tile.
int bisect(TilePoint *p, const TileRange &r, int cap)
{
    double lo[3], hi[3];
    for (int d = 0; d < 3; ++d)
        lo[d] = hi[d] = p[r.lo].x[d];
    for (int q = r.lo + 1; q < r.hi; ++q)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], p[q].x[d]);
            hi[d] = std::max(hi[d], p[q].x[d]);
        }
    int ax[3] = {0, 1, 2};
    std::stable_sort(ax, ax + 3, [&](int d, int e) {
        return hi[d] - lo[d] > hi[e] - lo[e];
    });
    const long long n = r.hi - r.lo, m = (n + cap - 1) / cap;
    const int cut = r.lo + (int)(n * (m / 2) / m);
    std::nth_element(p + r.lo, p + cut, p + r.hi,
                     [&](const TilePoint &a, const TilePoint &b) {
                         for (int d : ax)
                             if (a.x[d] != b.x[d])
                                 return a.x[d] < b.x[d];
                         return a.id < b.id;
                     });
    return cut;
}

std::vector<int> tile_order(int n, const double *x, const int *group, int cap,
                            std::vector<int> &starts)
{
    std::vector<int> order(n);
    for (int i = 0; i < n; ++i)
        order[i] = i;
    if (group)
        std::stable_sort(order.begin(), order.end(),
                         [&](int a, int b) { return group[a] < group[b]; });
    std::vector<TilePoint> p(n);
    std::vector<TileRange> parts;
    for (int q = 0; q < n; ++q) {
        const int i = order[q];
        for (int d = 0; d < 3; ++d) {
            // a coordinate that is not a number has no place in the order
            const double v = x[3 * (size_t)i + d];
            p[q].x[d] = std::fabs(v) <= __DBL_MAX__ ? v : 0.0;
        }
        p[q].id = i;
        if (q == 0 || (group && group[i] != group[order[q - 1]]))
            parts.push_back({q, q});
        parts.back().hi = q + 1;
    }
    // the first halvings, each level's side by side, until there is a part
    // for every thread; then each part to its tiles
    while (parts.size() < 64) {
        std::vector<int> cut(parts.size(), -1);
        run_parallel((int)parts.size(), [&](int lo, int hi) {
            for (int k = lo; k < hi; ++k)
                if (parts[k].hi - parts[k].lo > std::max(cap, 2048))
                    cut[k] = bisect(p.data(), parts[k], cap);
        }, 2);
        std::vector<TileRange> next;
        for (size_t k = 0; k < parts.size(); ++k) {
            if (cut[k] < 0) {
                next.push_back(parts[k]);
            } else {
                next.push_back({parts[k].lo, cut[k]});
                next.push_back({cut[k], parts[k].hi});
            }
        }
        const bool done = next.size() == parts.size();
        parts.swap(next);
        if (done)
            break;
    }
    std::vector<std::vector<int>> leaves(parts.size());
    run_parallel((int)parts.size(), [&](int lo, int hi) {
        std::vector<TileRange> todo;
        for (int k = lo; k < hi; ++k) {
            todo.assign(1, parts[k]);
            while (!todo.empty()) {
                const TileRange r = todo.back();
                todo.pop_back();
                if (r.hi - r.lo <= cap) {
                    leaves[k].push_back(r.lo);
                    continue;
                }
                const int cut = bisect(p.data(), r, cap);
                todo.push_back({cut, r.hi});  // the left half first
                todo.push_back({r.lo, cut});
            }
        }
    }, 2);
    starts.clear();
    for (const auto &l : leaves)
        starts.insert(starts.end(), l.begin(), l.end());
    for (int q = 0; q < n; ++q)
        order[q] = p[q].id;
    return order;
}

}  // namespace

extern "C" {

const char *pd_last_error(void) { return g_err.c_str(); }

int pd_device_count(int *count)
{
    if (!count)
        return fail(PD_E_ARG, "count is NULL");
    int c = 0;
    const hipError_t e = hipGetDeviceCount(&c);
    *count = (e == hipSuccess) ? c : 0;
    return PD_OK;
}

int pd_device_name(int device, char *name, int name_len, char *arch,
                   int arch_len)
{
    hipDeviceProp_t p;
    HIPCHK(hipGetDeviceProperties(&p, device));
    if (name && name_len > 0) {
        if (p.name[0])
            snprintf(name, name_len, "%s", p.name);
        else  // the marketing name is not always populated
            snprintf(name, name_len, "HIP device %d, %d CUs", device,
                     p.multiProcessorCount);
    }
    if (arch && arch_len > 0)
        snprintf(arch, arch_len, "%s", p.gcnArchName);
    return PD_OK;
}

int pd_build(pd_sim **out, int device, int integrator, int layout, double dt,
             double damping, int nnodes, int max_neighbours,
             const double *coords, const double *volume, const int *family,
             const int *bc_types, const double *bc_values,
             const int *force_bc_types, const double *force_bc_values,
             const double *stiffness_corrections, const int *bond_types,
             const double *densities)
{
    if (!out)
        return fail(PD_E_ARG, "sim is NULL");
    *out = nullptr;
    if (integrator < PD_EULER || integrator > PD_VELOCITY_VERLET)
        return fail(PD_E_ARG, "integrator must be 0, 1 or 2");
    if (layout != PD_LAYOUT_COMPACT && layout != PD_LAYOUT_SLOT)
        return fail(PD_E_ARG, "layout must be 0 (compact) or 1 (slot)");
    if (nnodes <= 0 || nnodes > MAX_NODES)
        return fail(PD_E_LIMIT, "nnodes must be in 1..2^26");
    if (max_neighbours <= 0 || max_neighbours > 65535)
        return fail(PD_E_LIMIT, "max_neighbours must be in 1..65535");
    if (layout == PD_LAYOUT_COMPACT &&
        compact_row_bytes(max_neighbours) + 64u > LDS_BYTES)
        return fail(PD_E_LIMIT, "the compact layout steps at most 27285 "
                                "neighbours per node");
    if (!coords || !volume || !family || !bc_types || !bc_values ||
        !force_bc_types || !force_bc_values)
        return fail(PD_E_ARG, "a required build array is NULL");
    if (integrator == PD_EULER && densities)
        return fail(PD_E_ARG,
                    "densities are not supported by this integrator: it "
                    "neglects inertial effects");
    if (integrator != PD_EULER && !densities)
        return fail(PD_E_ARG,
                    "densities must be supplied for a dynamic integrator");
    if (layout == PD_LAYOUT_COMPACT && (stiffness_corrections || bond_types))
        return fail(PD_E_ARG,
                    "stiffness_corrections and bond_types need the slot "
                    "(-1 marking) neighbour-list layout");
    for (int i = 0; i < nnodes; ++i)
        if (family[i] <= 0)
            return fail(PD_E_ARG, "family must be > 0 for every node");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(PD_E_NODEV, "no HIP device is available");
    if (device < 0 || device >= ndev)
        return fail(PD_E_ARG, "device index out of range");

    HIPCHK(hipSetDevice(device));
    int lds_max = 0;
    HIPCHK(hipDeviceGetAttribute(&lds_max,
                                 hipDeviceAttributeMaxSharedMemoryPerBlock,
                                 device));
    int cus = 0;
    HIPCHK(hipDeviceGetAttribute(
        &cus, hipDeviceAttributeMultiprocessorCount, device));
    pd_sim *s = new pd_sim();
    s->device = device;
    s->cus = std::max(cus, 1);
    s->integrator = integrator;
    s->layout = layout;
    s->dt = dt;
    s->damping = damping;
    s->n = nnodes;
    s->K = max_neighbours;
    s->lds_budget = (size_t)lds_max;
    if ((size_t)lds_max < LDS_BYTES)
        return fail(PD_E_NODEV, "device has less than 80 KiB of LDS per "
                                "workgroup");
    s->hmax = LDS_CAP_PMB - 1;
    const size_t N = (size_t)nnodes;
    s->h_coords.assign(coords, coords + 3 * N);
    s->coords_core = true;
    for (size_t q = 0; q < 3 * N && s->coords_core; ++q)
        s->coords_core = core_coord(coords[q]);

    std::vector<int> flags(N);
    for (size_t i = 0; i < N; ++i) {
        int f = 0;
        for (int d = 0; d < 3; ++d) {
            if (bc_types[3 * i + d] != 0)
                f |= 1 << d;
            if (force_bc_types[3 * i + d] != 0)
                f |= 1 << (3 + d);
        }
        flags[i] = f;
    }
    int rc = PD_OK;
    auto chk = [&](hipError_t e, const char *what) {
        if (e != hipSuccess && rc == PD_OK)
            rc = fail(PD_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
    };
    s->h_vol.assign(volume, volume + N);
    s->h_flags = std::move(flags);
    s->h_bcv.assign(bc_values, bc_values + 3 * N);
    s->h_fbcv.assign(force_bc_values, force_bc_values + 3 * N);
    if (densities)
        s->h_dens.assign(densities, densities + 3 * N);
    chk(upload(s->family, family, N), "family");
    chk(s->rec[0].alloc(N), "rec");
    chk(s->rec[1].alloc(N), "rec");
    chk(s->u.alloc(3 * N), "u");
    chk(s->ud.alloc(3 * N), "ud");
    chk(s->udd.alloc(3 * N), "udd");
    chk(s->force.alloc(3 * N), "force");
    chk(s->body_force.alloc(3 * N), "body_force");
    chk(s->damage.alloc(N), "damage");
    chk(s->out_nneigh.alloc(N), "n_neigh");
    chk(s->counter.alloc(1), "counter");
    chk(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking), "stream");
    chk(hipEventCreate(&s->ev0), "event");
    chk(hipEventCreate(&s->ev1), "event");
    if (stiffness_corrections) {
        s->h_corr.assign(stiffness_corrections,
                         stiffness_corrections + N * max_neighbours);
        s->has_corr = true;
    }
    if (bond_types) {
        s->h_btypes.assign(bond_types, bond_types + N * max_neighbours);
        s->has_btypes = true;
    }
    if (rc != PD_OK) {
        pd_destroy(s);
        return rc;
    }
    *out = s;
    return PD_OK;
}

int pd_create_buffers(pd_sim *s, const int *nlist, const int *n_neigh,
                      const double *bond_stiffness,
                      const double *critical_stretch, const double *plus_cs,
                      int nregimes, int nbond_types, const double *u,
                      const double *ud, const double *udd,
                      const int *regimes)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!nlist || !bond_stiffness || !critical_stretch)
        return fail(PD_E_ARG, "nlist, bond_stiffness and critical_stretch "
                              "are required");
    if (s->layout == PD_LAYOUT_COMPACT && !n_neigh)
        return fail(PD_E_ARG, "n_neigh is required for the compact layout");
    if (nregimes < 1 || nbond_types < 1)
        return fail(PD_E_ARG, "nregimes and nbond_types must be >= 1");
    const bool nlin = nregimes > 1 || nbond_types > 1;
    if (nlin) {
        if (s->layout == PD_LAYOUT_COMPACT)
            return fail(PD_E_ARG,
                        "n-linear damage models are not supported by this "
                        "integrator (compact layout)");
        if (!s->has_btypes)
            return fail(PD_E_ARG, "bond_types must be given to build for an "
                                  "n-linear or composite damage model");
        if (!plus_cs)
            return fail(PD_E_ARG, "plus_cs is required with nregimes > 1");
        if (nregimes * nbond_types > MAX_TAB || nregimes > 254 ||
            nbond_types > 255)
            return fail(PD_E_LIMIT, "damage model table too large");
    }
    const int N = s->n, K = s->K;
    std::atomic<int> given{0};  // some bond starts past its first regime
    if (nlin) {
        std::atomic<int> bad{0};
        run_parallel(N, [&](int lo, int hi) {
            int found = 0, past = 0;
            for (size_t q = (size_t)lo * K; q < (size_t)hi * K; ++q) {
                if (nlist[q] == -1)
                    continue;
                const int t = s->h_btypes[q];
                if (t < 0 || t >= nbond_types)
                    found = 1;
                if (regimes) {
                    if (regimes[q] < 0 || regimes[q] >= nregimes)
                        found = found == 1 ? 1 : 2;
                    past |= regimes[q];
                }
            }
            if (found)
                bad = bad == 1 ? 1 : found;
            if (past)
                given = 1;
        });
        if (bad == 1)
            return fail(PD_E_ARG, "bond_types value out of range");
        if (bad == 2)
            return fail(PD_E_ARG, "regimes value out of range for a "
                                  "live bond");
    }
    if (plan_holds(s, nlist, n_neigh, nlin, nregimes, nbond_types, given))
        return restart(s, bond_stiffness, critical_stretch, plus_cs, u, ud,
                       udd);

    // bond rows: live entries (j, reference column), sorted ascending by j
    std::vector<int> cnt(N);
    std::vector<long long> rstart(N + 1, 0);
    std::atomic<int> bad{0};
    run_parallel(N, [&](int lo, int hi) {
        for (int i = lo; i < hi; ++i) {
            const int *row = nlist + (size_t)i * K;
            int c = 0;
            if (s->layout == PD_LAYOUT_COMPACT) {
                c = n_neigh[i];
                if (c < 0 || c > K) {
                    bad = 1;
                    c = 0;
                }
                for (int p = 0; p < c; ++p)
                    if (row[p] < 0 || row[p] >= N)
                        bad = 2;
            } else {
                for (int p = 0; p < K; ++p) {
                    if (row[p] == -1)
                        continue;
                    if (row[p] < 0 || row[p] >= N)
                        bad = 2;
                    ++c;
                }
            }
            cnt[i] = c;
        }
    });
    if (bad == 1)
        return fail(PD_E_ARG, "n_neigh out of range [0, max_neighbours]");
    if (bad == 2)
        return fail(PD_E_ARG, "nlist entry out of range [0, nnodes)");
    for (int i = 0; i < N; ++i)
        rstart[i + 1] = rstart[i] + cnt[i];
    std::vector<int> rj(rstart[N]);
    std::vector<unsigned short> rp(rstart[N]);
    run_parallel(N, [&](int lo, int hi) {
        std::vector<std::pair<int, int>> ent;
        for (int i = lo; i < hi; ++i) {
            const int *row = nlist + (size_t)i * K;
            ent.clear();
            if (s->layout == PD_LAYOUT_COMPACT) {
                for (int p = 0; p < cnt[i]; ++p)
                    ent.emplace_back(row[p], p);
            } else {
                for (int p = 0; p < K; ++p)
                    if (row[p] != -1)
                        ent.emplace_back(row[p], p);
            }
            const auto by_key = [](const std::pair<int, int> &x,
                                   const std::pair<int, int> &y) {
                return x.first < y.first;
            };
            if (!std::is_sorted(ent.begin(), ent.end(), by_key))
                std::stable_sort(ent.begin(), ent.end(), by_key);
            for (size_t k = 0; k < ent.size(); ++k) {
                rj[rstart[i] + k] = ent[k].first;
                rp[rstart[i] + k] = (unsigned short)ent[k].second;
            }
        }
    });

    ShapeGuard shape{s};
    // tiles, capped by tile_nodes and by the LDS halo capacity
    // entry 0 of a staged halo is the far node of dead slots
    // the compact layout's tiles leave room for the exact step's windows
    s->hmax = (nlin ? LDS_CAP_NLIN
                    : (s->layout == PD_LAYOUT_COMPACT ? EXACT_CAP
                                                      : LDS_CAP_PMB)) -
              1;
    // blocks: the parts of at most tile_cap nodes.  A block is one tile, or
    // several where the halo capacity cuts it; blocks do not depend on each
    // other, so threads take them side by side.
    set_shape(s);
    const int cap = s->tile_cap;
    std::vector<int> bstart;
    std::vector<int> tnode = tile_order(
        N, s->h_coords.data(), s->h_group.empty() ? nullptr : s->h_group.data(),
        cap, bstart);
    const int nblocks = (int)bstart.size();
    bstart.push_back(N);
    std::vector<std::vector<TileInfo>> cuts(nblocks);
    // each block cut into tiles whose halos hold at most `most` entries;
    // their number, or -1 where a node's own neighbourhood does not fit
    auto cut_blocks = [&](int most) {
        std::atomic<int> wide{0}, count{0};
        run_parallel(nblocks, [&](int lo, int hi) {
            std::vector<int> stamp(N, -1);
            int tid = 0;
            for (int bl = lo; bl < hi; ++bl) {
                cuts[bl].clear();
                TileInfo t{};
                t.node_off = bstart[bl];
                ++tid;
                for (int q = bstart[bl]; q < bstart[bl + 1]; ++q) {
                    const int i = tnode[q];
                    if (1 + cnt[i] > most) {
                        wide = 1;
                        return;
                    }
                    // the distinct nodes that i and its neighbours add (a
                    // row may list a neighbour more than once)
                    auto add = [&]() {
                        int c = 0;
                        auto visit = [&](int j) {
                            c += stamp[j] != tid;
                            stamp[j] = tid;
                        };
                        visit(i);
                        for (long long r = rstart[i]; r < rstart[i + 1]; ++r)
                            visit(rj[r]);
                        return c;
                    };
                    int c = add();
                    if (t.nodes > 0 && t.halo + c > most) {
                        cuts[bl].push_back(t);
                        t = TileInfo{};
                        t.node_off = q;
                        ++tid;
                        c = add();
                    }
                    t.halo += c;
                    ++t.nodes;
                }
                cuts[bl].push_back(t);
                count += (int)cuts[bl].size();
            }
        }, 16);
        return wide ? -1 : (int)count;
    };
    // the narrow form's capacity first, where the step may use it and it
    // costs few more tiles (in 50 at most one: its gain is three times that)
    int ncut = -1;
    if (s->layout == PD_LAYOUT_SLOT && s->lanes == 4 && !nlin &&
        dm_of(s) == DM_PMB && !s->has_corr && narrow_fits(s, nblocks, 0)) {
        ncut = cut_blocks(LDS_CAP_NARROW - 1);
        if (ncut > nblocks + nblocks / 50)
            ncut = -1;
    }
    if (ncut < 0 && cut_blocks(s->hmax) < 0)
        return fail(PD_E_LIMIT, "a node's neighbourhood exceeds the "
                                "LDS halo capacity");
    std::vector<TileInfo> tiles;
    for (const auto &c : cuts)
        tiles.insert(tiles.end(), c.begin(), c.end());
    // within a tile, nodes by descending bond count: the nodes sharing a
    // wavefront then run loops of nearly equal length
    run_parallel((int)tiles.size(), [&](int lo, int hi) {
        for (int t = lo; t < hi; ++t)
            std::stable_sort(tnode.begin() + tiles[t].node_off,
                             tnode.begin() + tiles[t].node_off +
                                 tiles[t].nodes,
                             [&](int y, int z) { return cnt[y] > cnt[z]; });
    }, 16);
    std::vector<int> inv(N);  // caller's node id -> internal id
    for (int q = 0; q < N; ++q)
        inv[tnode[q]] = q;
    const int ntiles = (int)tiles.size();
    long long halo_total = 0, chunk_total = 0;
    for (auto &t : tiles) {
        t.halo_off = (int)halo_total;
        halo_total += t.halo;
        int nch = 0;
        for (int l = 0; l < t.nodes; ++l)
            nch = std::max(nch, chunks_of(cnt[tnode[t.node_off + l]]));
        // the exact step's fold lists take the place of the slots: two rows
        // of pairs per row of chunks, four per round of eight positions
        if (s->layout == PD_LAYOUT_COMPACT && t.nodes > 0)
            nch = std::max(nch, 2 * ((cnt[tnode[t.node_off]] + 7) >> 3));
        t.nch = nch;
        t.pad = 0;
        t.chunk_off = chunk_total;
        // at least one row, which the kernel's clamped loads may read
        chunk_total += (long long)std::max(nch, 1) * t.nodes;
    }
    if (halo_total > 0x7fffffffLL)
        return fail(PD_E_LIMIT, "total halo size exceeds 2^31");
    const size_t S = (size_t)chunk_total * 4;
    std::vector<int> halo(halo_total);
    std::vector<unsigned short> loc(S + LOC_SLACK, LOC_DEAD);
    std::vector<int> gidx(S, (int)DEAD);
    std::vector<unsigned short> pos(S, 0);
    std::vector<double> corr;
    std::vector<unsigned short> state;
    if (s->has_corr)
        corr.assign(S + LOC_SLACK, 0.0);
    if (nlin)
        state.assign(S + LOC_SLACK, 0);
    std::vector<long long> chunk0(N);
    std::vector<int> stride(N);
    const bool compact = s->layout == PD_LAYOUT_COMPACT;
    std::vector<int> nlow_h(compact ? N : 0);
    std::vector<long long> tile0_h(compact ? N : 0);
    std::atomic<int> halo_mismatch{0}, odd{0};
    run_parallel(ntiles, [&](int lo, int hi) {
        std::vector<int> lmap(N, -1);  // internal id -> halo position
        std::vector<int> hl;
        std::vector<int> roff, rows;
        HaloSpread spread;
        for (int t = lo; t < hi; ++t) {
            const TileInfo &ti = tiles[t];
            hl.clear();
            auto visit = [&](int h) {
                if (lmap[h] == -1) {
                    lmap[h] = 0;
                    hl.push_back(h);
                }
            };
            for (int l = 0; l < ti.nodes; ++l) {
                const int i = tnode[ti.node_off + l];
                visit(ti.node_off + l);
                for (long long r = rstart[i]; r < rstart[i + 1]; ++r)
                    visit(inv[rj[r]]);
            }
            std::sort(hl.begin(), hl.end());
            if ((int)hl.size() != ti.halo) {
                halo_mismatch = 1;
                break;
            }
            for (size_t h = 0; h < hl.size(); ++h)
                lmap[hl[h]] = (int)h;
            rows.clear();
            roff.assign(1, 0);
            for (int l = 0; l < ti.nodes; ++l) {
                const int i = tnode[ti.node_off + l];
                for (int k = 0; k < cnt[i]; ++k)
                    rows.push_back(lmap[inv[rj[rstart[i] + k]]]);
                roff.push_back((int)rows.size());
            }
            const std::vector<int> &hpos =
                spread.place(roff, rows, s->lanes, (int)hl.size());
            for (size_t h = 0; h < hl.size(); ++h) {
                lmap[hl[h]] = hpos[h];
                halo[ti.halo_off + hpos[h]] = hl[h];
            }
            for (int l = 0; l < ti.nodes; ++l) {
                const int i = tnode[ti.node_off + l];
                chunk0[ti.node_off + l] = ti.chunk_off + l;
                stride[ti.node_off + l] = ti.nodes;
                for (int k = 0; k < cnt[i]; ++k) {
                    const int j = rj[rstart[i] + k];
                    const int p = rp[rstart[i] + k];
                    const size_t sl = slot_of(ti.chunk_off + l, ti.nodes, k);
                    loc[sl] = (unsigned short)(16 * (lmap[inv[j]] + 1));
                    gidx[sl] = j;
                    pos[sl] = (unsigned short)p;
                    const size_t src = (size_t)i * K + p;
                    if (s->has_corr) {
                        corr[sl] = s->h_corr[src];
                        if (!std::isfinite(corr[sl]))
                            odd = 1;
                    }
                    if (nlin)
                        state[sl] = (unsigned short)(
                            16 * (s->h_btypes[src] * nregimes +
                                  (regimes ? regimes[src] : 0)));
                }
                if (compact) {
                    const int p = ti.node_off + l;
                    const int *rb = rj.data() + rstart[i];
                    nlow_h[p] = (int)(std::lower_bound(rb, rb + cnt[i], i) - rb);
                    tile0_h[p] = ti.chunk_off;
                }
            }
            for (int h : hl)
                lmap[h] = -1;
        }
    }, 16);
    if (halo_mismatch)
        return fail(PD_E_STATE, "internal: tile halo count mismatch");
    for (const auto &t : tiles)
        if (t.halo > s->hmax)
            return fail(PD_E_LIMIT, "internal: tile halo over capacity");

    HIPCHK(hipStreamSynchronize(s->stream));
    // from here the device state is replaced: until it is whole again no
    // step may run (a failure below leaves the simulation without buffers)
    shape.taken = true;
    s->has_buffers = false;
    s->plan = false;
    adjoint_release(s);
    s->inv.release();
    auto chk = [&](hipError_t e, const char *what) {
        if (e != hipSuccess && rc == PD_OK)
            rc = fail(PD_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
    };
    s->ntiles = ntiles;
    s->nslots = S;
    s->odd_corr = odd != 0;
    s->hstride = 1;
    for (const auto &t : tiles)
        s->hstride = std::max(s->hstride, t.halo);
    chk(upload(s->tiles, tiles.data(), tiles.size()), "tiles");
    chk(upload(s->tnode, tnode.data(), tnode.size()), "tnode");
    chk(upload(s->halo, halo.data(), halo.size()), "halo");
    s->perm = tnode;
    chk(upload_perm(s->cnt, s->perm, cnt.data(), 1), "cnt");
    chk(upload_perm(s->r0, s->perm, s->h_coords.data(), 3), "coords");
    chk(upload_perm(s->vol, s->perm, s->h_vol.data(), 1), "volume");
    chk(upload_perm(s->flags, s->perm, s->h_flags.data(), 1), "flags");
    {
        std::vector<int> meta(N);
        for (int i = 0; i < N; ++i)
            meta[i] = cnt[i] | s->h_flags[i] << 16;
        chk(upload_perm(s->meta, s->perm, meta.data(), 1), "flags");
    }
    chk(upload_perm(s->bcv, s->perm, s->h_bcv.data(), 3), "bc_values");
    chk(upload_perm(s->fbcv, s->perm, s->h_fbcv.data(), 3),
        "force_bc_values");
    s->dens1.release();
    if (!s->h_dens.empty()) {
        chk(upload_perm(s->dens, s->perm, s->h_dens.data(), 3), "densities");
        // one density per node (the reference's tiled layout, model.py:
        // 691-702) is read as one value per node
        bool per_node = true;
        for (size_t i = 0; per_node && i < N; ++i)
            per_node = s->h_dens[3 * i] == s->h_dens[3 * i + 1] &&
                       s->h_dens[3 * i] == s->h_dens[3 * i + 2];
        if (per_node) {
            std::vector<double> d1(N);
            for (size_t i = 0; i < N; ++i)
                d1[i] = s->h_dens[3 * i];
            chk(upload_perm(s->dens1, s->perm, d1.data(), 1), "densities");
        }
    }
    if (s->has_cnode && !s->h_cnode.empty()) {
        chk(upload_perm(s->cnode, s->perm, s->h_cnode.data(), 1),
            "node stiffness");
    } else if (s->has_cnode) {
        // given on the device: into the new node order there
        chk(s->cnode.alloc(N), "node stiffness");
        if (rc == PD_OK)
            hipLaunchKernelGGL(k_perm, dim3((N + 255) / 256), dim3(256), 0,
                               s->stream, (int)N, 1, s->tnode.p,
                               s->cnode_caller.p, s->cnode.p);
        chk(hipGetLastError(), "node stiffness");
    }
    chk(upload(s->chunk0, chunk0.data(), (size_t)N), "chunk0");
    chk(upload(s->stride, stride.data(), (size_t)N), "stride");
    chk(upload(s->loc, loc.data(), loc.size()), "loc");
    chk(upload(s->gidx, gidx.data(), gidx.size()), "gidx");
    chk(upload(s->pos, pos.data(), pos.size()), "pos");
    if (s->has_corr)
        chk(upload(s->corr, corr.data(), corr.size()), "corr");
    else
        s->corr.release();
    if (nlin)
        chk(upload(s->state, state.data(), state.size()), "state");
    else
        s->state.release();
    chk(s->loc_init.alloc(S), "loc");
    if (rc == PD_OK)
        chk(hipMemcpyAsync(s->loc_init.p, s->loc.p, S * sizeof(unsigned short),
                           hipMemcpyDeviceToDevice, s->stream),
            "loc");
    s->state_init.release();
    if (nlin && !given) {
        chk(s->state_init.alloc(S), "state");
        if (rc == PD_OK)
            chk(hipMemcpyAsync(s->state_init.p, s->state.p,
                               S * sizeof(unsigned short),
                               hipMemcpyDeviceToDevice, s->stream),
                "state");
    }
    if (s->layout == PD_LAYOUT_COMPACT) {
        chk(upload(s->nlist_ref, nlist, (size_t)N * K), "nlist");
        chk(s->rslot.alloc((size_t)N * K), "nlist");
        chk(s->n_neigh.alloc((size_t)N), "n_neigh");
        if (rc == PD_OK) {
            hipLaunchKernelGGL(k_row_slots, dim3(row_blocks(N, ROW_LANES)),
                               dim3(256), 0, s->stream, N, K, s->tnode.p,
                               s->cnt.p, s->chunk0.p, s->stride.p, s->pos.p,
                               s->rslot.p, s->n_neigh.p);
            chk(hipGetLastError(), "nlist");
        }
        chk(upload(s->nlow, nlow_h.data(), nlow_h.size()), "exact lists");
        chk(upload(s->tile0, tile0_h.data(), tile0_h.size()), "exact lists");
        chk(s->nup.alloc((size_t)N), "exact lists");
        // the rounds' look-ahead reads past a tile's lists, and positions
        // past a list's end are dead
        chk(s->ford.alloc(S + LOC_SLACK), "exact lists");
        if (rc == PD_OK)
            chk(hipMemsetAsync(s->ford.p, 0,
                               (S + LOC_SLACK) * sizeof(unsigned), s->stream),
                "exact lists");
    } else {
        s->nlist_ref.release();
        s->rslot.release();
        s->n_neigh.release();
        s->nlow.release();
        s->nup.release();
        s->ford.release();
        s->tile0.release();
    }
    chk(s->out_nlist.alloc(s->layout == PD_LAYOUT_SLOT ? (size_t)N * K : 0),
        "nlist export");
    s->nregimes = nregimes;
    s->nbond_types = nbond_types;
    s->odd_tables = false;
    if (nlin) {
        chk(set_tables(s, bond_stiffness, critical_stretch, plus_cs),
            "damage model tables");
        s->k = 0.0;
        s->s0 = 0.0;
    } else {
        s->k_tab.release();
        s->s_tab.release();
        s->pc_tab.release();
        s->k = bond_stiffness[0];
        s->s0 = critical_stretch[0];
    }
    if (rc)
        return rc;
    rc = start_state(s, u, ud, udd);
    if (rc)
        return rc;
    rc = upload_tips(s);
    if (rc)
        return rc;
    s->has_buffers = true;
    s->lost = false;
    s->retile_pending = false;
    keep_plan(s, nlist, n_neigh, nlin, given);
    return PD_OK;
}

int pd_set_tips(pd_sim *s, int nentries, const int *node, const int *dof,
                const int *group, int ngroups)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (nentries < 0 || ngroups < 0 ||
        (nentries > 0 && (!node || !dof || !group)))
        return fail(PD_E_ARG, "node, dof and group (nentries) are required");
    std::vector<int> off(ngroups + 1, 0);
    for (int e = 0; e < nentries; ++e) {
        if (node[e] < 0 || node[e] >= s->n || dof[e] < 0 || dof[e] > 2 ||
            group[e] < 0 || group[e] >= ngroups)
            return fail(PD_E_ARG, "a tip entry is out of range");
        off[group[e] + 1]++;
    }
    for (int g = 0; g < ngroups; ++g)
        off[g + 1] += off[g];
    // group the entries, keeping their order inside a group
    std::vector<int> fill(off.begin(), off.end() - 1);
    s->h_tip_node.assign(nentries, 0);
    s->h_tip_dof.assign(nentries, 0);
    for (int e = 0; e < nentries; ++e) {
        const int at = fill[group[e]]++;
        s->h_tip_node[at] = node[e];
        s->h_tip_dof[at] = dof[e];
    }
    s->h_tip_off = off;
    s->tip_q.release();
    s->tip_off.release();
    if (s->has_buffers)
        return upload_tips(s);
    return PD_OK;
}

int pd_monitor(pd_sim *s, double *model, double *tips)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    if (!model)
        return fail(PD_E_ARG, "model (6 doubles) is required");
    const int ngroups =
        s->h_tip_off.empty() ? 0 : (int)s->h_tip_off.size() - 1;
    if (ngroups > 0 && !tips)
        return fail(PD_E_ARG, "tips (5 doubles per group) is required");
    // where pd_set_tips got no memory for them
    if (ngroups > 0 && !s->tip_off.p && (rc = upload_tips(s)) != PD_OK)
        return rc;
    const int N = s->n;
    if (!s->mon_part.p) {
        HIPCHK(s->mon_part.alloc((size_t)MON_BLOCKS * MON_SUMS));
    }
    const size_t nout = MON_SUMS + 5 * (size_t)ngroups;
    if (s->mon_out.n < nout) {
        HIPCHK(s->mon_out.alloc(nout));
    }
    HIPCHK(launch_export(s, 0, s->damage.p));
    hipLaunchKernelGGL(k_monitor_part, dim3(MON_BLOCKS), dim3(256), 0,
                       s->stream, N, s->u.p, s->ud.p, s->udd.p, s->force.p,
                       s->body_force.p, s->flags.p, s->vol.p, s->damage.p,
                       s->mon_part.p);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_monitor_final, dim3(1), dim3(256), 0, s->stream,
                       s->mon_part.p, ngroups, s->tip_off.p, s->tip_q.p,
                       s->u.p, s->ud.p, s->udd.p, s->force.p,
                       s->body_force.p, s->flags.p, s->vol.p, s->mon_out.p);
    HIPCHK(hipGetLastError());
    std::vector<double> h(nout);
    HIPCHK(hipMemcpyAsync(h.data(), s->mon_out.p, nout * sizeof(double),
                          hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    std::copy(h.begin(), h.begin() + MON_SUMS, model);
    if (ngroups > 0)
        std::copy(h.begin() + MON_SUMS, h.end(), tips);
    return PD_OK;
}

namespace {

// The device address of `scratch` for each device, looked up once per
// device with that device current.
constexpr int NOALLOC_DEVICES = 64;
std::mutex g_scratch_mu;
double *g_scratch[NOALLOC_DEVICES] = {};

int scratch_address(int device, double **out)
{
    if (device < 0 || device >= NOALLOC_DEVICES)
        return fail(PD_E_LIMIT, "pd_monitor_noalloc: device index beyond 63");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(PD_E_HIP, std::string("hipGetSymbolAddress(scratch): ") +
                                      hipGetErrorString(e));
        g_scratch[device] = static_cast<double *>(p);
    }
    *out = g_scratch[device];
    return PD_OK;
}

}  // namespace

int pd_monitor_noalloc(pd_sim *s, double *model, double *tips)
{
    int rc = check_sim(s);  // makes the simulation's device current
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    if (!model)
        return fail(PD_E_ARG, "model (6 doubles) is required");
    const int ngroups =
        s->h_tip_off.empty() ? 0 : (int)s->h_tip_off.size() - 1;
    if (ngroups > NOALLOC_MAX_GROUPS)
        return fail(PD_E_LIMIT, "pd_monitor_noalloc: more than 1024 tip "
                                "groups (use pd_monitor)");
    if (ngroups > 0 && !tips)
        return fail(PD_E_ARG, "tips (5 doubles per group) is required");
    // where pd_set_tips got no memory for them
    if (ngroups > 0 && !s->tip_off.p && (rc = upload_tips(s)) != PD_OK)
        return rc;
    double *sp = nullptr;
    rc = scratch_address(s->device, &sp);
    if (rc)
        return rc;
    // every entry of both regions is written by the kernels below before it
    // is read: nothing needs clearing between calls
    double *part = sp;
    double *staged = sp + (size_t)MON_BLOCKS * MON_SUMS;
    const int N = s->n;
    HIPCHK(launch_export(s, 0, s->damage.p));
    hipLaunchKernelGGL(k_monitor_part, dim3(MON_BLOCKS), dim3(256), 0,
                       s->stream, N, s->u.p, s->ud.p, s->udd.p, s->force.p,
                       s->body_force.p, s->flags.p, s->vol.p, s->damage.p,
                       part);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_monitor_final, dim3(1), dim3(256), 0, s->stream,
                       part, ngroups, s->tip_off.p, s->tip_q.p, s->u.p,
                       s->ud.p, s->udd.p, s->force.p, s->body_force.p,
                       s->flags.p, s->vol.p, staged);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(model, staged, MON_SUMS * sizeof(double),
                          hipMemcpyDeviceToHost, s->stream));
    if (ngroups > 0)
        HIPCHK(hipMemcpyAsync(tips, staged + MON_SUMS,
                              5 * (size_t)ngroups * sizeof(double),
                              hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    return PD_OK;
}

int pd_set_node_stiffness(pd_sim *s, const double *c)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    HIPCHK(hipStreamSynchronize(s->stream));
    s->adj_changed = true;
    StateGuard state{s, s->has_buffers};
    if (!c) {
        s->cnode.release();
        s->h_cnode.clear();
        s->has_cnode = false;
    } else {
        s->h_cnode.assign(c, c + s->n);
        s->has_cnode = true;
        // uploaded in tile order, which pd_create_buffers fixes
        if (s->has_buffers)
            HIPCHK(upload_perm(s->cnode, s->perm, c, 1));
    }
    s->cnode_caller.release();
    if (s->has_buffers) {
        // the records carry c: rewrite both from the device u
        rc = refresh_records(s);
        if (rc)
            return rc;
    }
    state.away = false;
    return PD_OK;
}

int pd_set_node_stiffness_device(pd_sim *s, const double *c)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!c)
        return fail(PD_E_ARG, "c is NULL (pd_set_node_stiffness clears)");
    HIPCHK(hipStreamSynchronize(s->stream));
    s->adj_changed = true;
    const size_t N = (size_t)s->n;
    HIPCHK(s->cnode_caller.reserve(N));
    StateGuard state{s, s->has_buffers};
    HIPCHK(hipMemcpyAsync(s->cnode_caller.p, c, N * sizeof(double),
                          hipMemcpyDeviceToDevice, s->stream));
    s->h_cnode.clear();
    s->has_cnode = true;
    if (s->has_buffers) {
        HIPCHK(s->cnode.reserve(N));
        hipLaunchKernelGGL(k_perm, dim3((s->n + 255) / 256), dim3(256), 0,
                           s->stream, s->n, 1, s->tnode.p, s->cnode_caller.p,
                           s->cnode.p);
        HIPCHK(hipGetLastError());
        rc = refresh_records(s);  // synchronizes the stream
        state.away = rc != PD_OK;
        return rc;
    }
    HIPCHK(hipStreamSynchronize(s->stream));
    return PD_OK;
}

int pd_set_break_mode(pd_sim *s, int tension_only)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    s->tension_only = tension_only ? 1 : 0;
    s->adj_changed = true;
    return PD_OK;
}

int pd_set_exact_order(pd_sim *s, int on)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (on && (s->layout != PD_LAYOUT_COMPACT || s->integrator != PD_EULER))
        return fail(PD_E_ARG, "the exact-order step is the Cython path's: "
                              "PD_LAYOUT_COMPACT and PD_EULER only");
    if (on && !exact_rows_fit(s->K))
        return fail(PD_E_LIMIT, "the exact-order step takes at most 4074 "
                                "neighbours per node");
    const bool was = s->exact;
    s->exact = on != 0;
    // the records carry V (exact) or 4kV (default): rewrite them; the fast
    // step does not keep the fold lists
    if (s->has_buffers && was != s->exact) {
        StateGuard state{s, true};
        if (s->exact)
            rc = fold_lists(s);
        if (rc == PD_OK)
            rc = refresh_records(s);
        state.away = rc != PD_OK;
    }
    return rc;
}

int pd_set_launch(pd_sim *s, int lanes_per_node, int tile_nodes)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (lanes_per_node != 1 && lanes_per_node != 2 && lanes_per_node != 4 &&
        lanes_per_node != 8)
        return fail(PD_E_ARG, "lanes_per_node must be 1, 2, 4 or 8");
    if (tile_nodes < 64 || tile_nodes % 64 ||
        tile_nodes * lanes_per_node > 1024)
        return fail(PD_E_ARG, "tile_nodes must be a multiple of 64 with "
                              "tile_nodes * lanes_per_node <= 1024");
    // a new tile size takes effect when pd_create_buffers re-tiles; until
    // then the current tiles (of the old size) cannot be stepped
    if (s->has_buffers && tile_nodes != s->tile_nodes)
        s->retile_pending = true;
    s->lpn = s->lanes = lanes_per_node;
    s->tile_nodes = tile_nodes;
    s->launch_given = true;
    s->adj_changed = true;
    return PD_OK;
}

int pd_set_groups(pd_sim *s, const int *group)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (s->has_buffers)
        return fail(PD_E_STATE, "groups must be set before pd_create_buffers");
    if (!group) {
        s->h_group.clear();
        return PD_OK;
    }
    s->h_group.assign(group, group + s->n);
    return PD_OK;
}

int pd_step(pd_sim *s, double dmag, double fmag)
{
    return pd_run(s, 1, &dmag, &fmag);
}

int pd_run(pd_sim *s, int nsteps, const double *disp_mags,
           const double *force_mags)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    if (nsteps < 0)
        return fail(PD_E_ARG, "nsteps < 0");
    const int cur0 = s->cur;  // of a first step that is not launched
    for (int t = 0; t < nsteps; ++t) {
        rc = launch_step(s, disp_mags ? disp_mags[t] : 0.0,
                         force_mags ? force_mags[t] : 0.0, t + 1 == nsteps);
        if (rc) {
            if (t > 0 || s->cur != cur0)
                run_failed(s);
            return rc;
        }
    }
    return PD_OK;
}

int pd_run_timed(pd_sim *s, int nsteps, const double *disp_mags,
                 const double *force_mags, float *elapsed_ms)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!elapsed_ms)
        return fail(PD_E_ARG, "elapsed_ms is NULL");
    HIPCHK(hipEventRecord(s->ev0, s->stream));
    rc = pd_run(s, nsteps, disp_mags, force_mags);
    if (rc)
        return rc;
    HIPCHK(hipEventRecord(s->ev1, s->stream));
    HIPCHK(hipEventSynchronize(s->ev1));
    HIPCHK(hipEventElapsedTime(elapsed_ms, s->ev0, s->ev1));
    return PD_OK;
}

// The steps go to the device as graphs of GRAPH_STEPS (a first one of two), so
// that it runs one while the host captures the next: a captured and
// instantiated step costs the host about 6 us, which in one graph all came
// before the first step.  Wall clock of 25 steps, one graph / graphs of 4, 8
// and 16: 1,280 nodes 363 / 244, 236, 238 us; 141,143 nodes 1162 / 1024, 1002,
// 1019 (of 400: 18.3 / 16.0, 15.6, 15.6 ms).
// All steps run or none: where the first graph cannot be made nothing has run,
// and where a later one cannot, the steps from there on are launched one by
// one.
constexpr int GRAPH_STEPS = 8;

int pd_run_graph(pd_sim *s, int nsteps, const double *disp_mags,
                 const double *force_mags, float *elapsed_ms)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    if (nsteps < 0)
        return fail(PD_E_ARG, "nsteps < 0");
    if (nsteps == 0) {
        if (elapsed_ms)
            *elapsed_ms = 0.0f;
        return PD_OK;
    }
    if (s->adj_recording)
        return fail(PD_E_STATE, "an adjoint recording runs step by step "
                                "(pd_run), not as a graph");
    HIPCHK(hipStreamSynchronize(s->stream));
    std::vector<hipGraphExec_t> execs;
    hipError_t e = hipSuccess;
    const auto step = [&](int t) {
        return launch_step(s, disp_mags ? disp_mags[t] : 0.0,
                           force_mags ? force_mags[t] : 0.0, t + 1 == nsteps);
    };
    int t0 = 0;  // the steps before it are on their way
    while (t0 < nsteps) {
        const int t1 = std::min(nsteps, t0 == 0 ? 2 : t0 + GRAPH_STEPS);
        const int cur0 = s->cur;
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        e = hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            for (int t = t0; t < t1 && rc == PD_OK; ++t)
                rc = step(t);
            e = hipStreamEndCapture(s->stream, &graph);
        }
        if (rc == PD_OK && e == hipSuccess)
            e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (graph)
            (void)hipGraphDestroy(graph);
        if (exec)
            execs.push_back(exec);
        if (rc == PD_OK && e == hipSuccess && t0 == 0 && elapsed_ms)
            e = hipEventRecord(s->ev0, s->stream);
        const bool made = rc == PD_OK && e == hipSuccess;
        if (made)
            e = hipGraphLaunch(exec, s->stream);
        if (made && e == hipSuccess) {
            t0 = t1;
            continue;
        }
        s->cur = cur0;  // these steps do not run
        (void)hipGetLastError();  // or the next launch would report it
        if (made || t0 == 0)
            break;
        rc = PD_OK;
        e = hipSuccess;
        for (; t0 < nsteps && rc == PD_OK; ++t0)
            rc = step(t0);
        break;
    }
    const bool ran = rc == PD_OK && e == hipSuccess;
    if (ran && elapsed_ms)
        e = hipEventRecord(s->ev1, s->stream);
    const hipError_t es = hipStreamSynchronize(s->stream);
    if (t0 > 0 && !(ran && es == hipSuccess))
        run_failed(s);
    for (hipGraphExec_t x : execs)
        (void)hipGraphExecDestroy(x);
    if (e == hipSuccess)
        e = es;
    if (rc == PD_OK && e == hipSuccess && elapsed_ms)
        e = hipEventElapsedTime(elapsed_ms, s->ev0, s->ev1);
    if (rc != PD_OK)
        return rc;
    if (e != hipSuccess)
        return fail(PD_E_HIP, std::string("graph run: ") +
                                  hipGetErrorString(e));
    return PD_OK;
}

namespace {

// Whether a recording keeps u of all its steps (room for them is then in
// seg), where checkpoints and a segment take `slots` arrays: the backward
// pass then replays nothing (a third of it and of the forward pass together:
// 200 steps and their gradient on 50,820 nodes 12.3 -> 8.8 ms).  At most
// KEEP_TIMES the memory that the caller's checkpoint interval asks for (at an
// interval of 100, recordings of up to 4,700 steps), a 64th of the device's and
// a quarter of what is free (2000 steps of 50,820 nodes: 17 times, 2.4 GB);
// never where the caller holds recordings to their checkpoints
// (pd_adjoint_keep).
constexpr size_t KEEP_TIMES = 32;

bool keep_all(pd_sim *s, int nsteps, size_t slots)
{
    const size_t count = (size_t)nsteps * 3 * s->n;
    if (!s->adj_keep || (size_t)nsteps > KEEP_TIMES * slots)
        return false;
    if (s->seg.p && s->seg.n >= count)
        return true;
    size_t avail = 0, total = 0;
    if (hipMemGetInfo(&avail, &total) != hipSuccess ||
        count * sizeof(double) > std::min(total / 64, avail / 4) ||
        s->seg.alloc(count) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

}  // namespace

int pd_adjoint_keep(pd_sim *s, int every_step)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    s->adj_keep = every_step != 0;
    return PD_OK;
}

int pd_adjoint_start(pd_sim *s, int nsteps, int checkpoint_every)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers || s->retile_pending)
        return no_buffers(s);
    if (s->integrator != PD_EULER || s->layout != PD_LAYOUT_SLOT ||
        !s->has_cnode || s->nregimes > 1 || s->nbond_types > 1)
        return fail(PD_E_ARG, "the adjoint needs the Euler integrator, the "
                              "slot layout and a node stiffness field");
    if (nsteps < 1 || checkpoint_every < 1)
        return fail(PD_E_ARG, "nsteps and checkpoint_every must be >= 1");
    adjoint_end(s);
    const size_t S = s->nslots, N = (size_t)s->n, B = 3 * N;
    const int nck = (nsteps + checkpoint_every - 1) / checkpoint_every;
    if (!s->inv.p) {
        std::vector<int> inv(N);
        for (size_t q = 0; q < N; ++q)
            inv[s->perm[q]] = (int)q;
        HIPCHK(upload(s->inv, inv.data(), N));
    }
    // a recording after one of the same size allocates nothing
    HIPCHK(s->brk.reserve(S));
    HIPCHK(s->il0.reserve(S));
    HIPCHK(s->arec[0].reserve(N));
    HIPCHK(s->arec[1].reserve(N));
    HIPCHK(s->loc0.reserve(S));
    s->adj_all = keep_all(s, nsteps, (size_t)nck + checkpoint_every);
    if (!s->adj_all) {
        // held to the checkpoints, an earlier recording's room goes back
        if (!s->adj_keep && s->seg.n > (size_t)checkpoint_every * B)
            s->seg.release();
        if (!s->adj_keep && s->ckpt.n > (size_t)nck * B)
            s->ckpt.release();
        HIPCHK(s->ckpt.reserve((size_t)nck * B));
        HIPCHK(s->seg.reserve((size_t)checkpoint_every * B));
    }
    HIPCHK(s->lam[0].reserve(B));
    HIPCHK(s->lam[1].reserve(B));
    HIPCHK(s->gradc.reserve(N));
    // rows past a node's own, up to its tile's longest: finite
    HIPCHK(hipMemsetAsync(s->il0.p, 0, S * sizeof(double), s->stream));
    hipLaunchKernelGGL(k_adj_init, dim3(chunk_blocks(s)), dim3(256), 0,
                       s->stream, (long long)(S / 4), s->loc.p, s->loc0.p,
                       s->brk.p);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_adj_il0, dim3(row_blocks(s->n, ROW_LANES)),
                       dim3(256), 0, s->stream, s->n, s->cnt.p, s->chunk0.p, s->stride.p,
                       s->gidx.p, s->loc0.p, s->inv.p, s->r0.p, s->il0.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(s->adj_all ? s->seg.p : s->ckpt.p, s->u.p,
                          B * sizeof(double), hipMemcpyDeviceToDevice,
                          s->stream));
    s->adj_nsteps = nsteps;
    s->adj_every = checkpoint_every;
    s->step_counter = 0;
    s->adj_recording = true;
    return PD_OK;
}

namespace {

// Put the state at the start of step n0 from u (already in s->u): bond
// states from brk, records from u.
int adjoint_restore(pd_sim *s, int n0)
{
    hipLaunchKernelGGL(k_adj_restore, dim3(chunk_blocks(s)), dim3(256), 0,
                       s->stream, (long long)(s->nslots / 4), n0, s->brk.p,
                       s->loc0.p, s->loc.p, s->gidx.p);
    HIPCHK(hipGetLastError());
    return refresh_records(s);
}

// Steps n0 .. n1 - 2 again from u of step n0, the segment's first slot: the
// same kernel from the same state reproduces the recorded steps (and their
// breaks) bitwise; step n writes u_{n+1} to slot n + 1 - n0 of the segment.
int adjoint_replay(pd_sim *s, double *seg, int n0, int n1)
{
    const size_t B = 3 * (size_t)s->n;
    HIPCHK(hipMemcpyAsync(s->u.p, seg, B * sizeof(double),
                          hipMemcpyDeviceToDevice, s->stream));
    const int rc0 = adjoint_restore(s, n0);
    if (rc0)
        return rc0;
    struct ReplayGuard {  // the steps below are replays
        pd_sim *s;
        ~ReplayGuard()
        {
            s->adj_replay = false;
            s->u_out = nullptr;
        }
    } guard{s};
    s->adj_replay = true;
    int rc = PD_OK;
    for (int n = n0; n < n1 - 1 && rc == PD_OK; ++n) {
        s->step_counter = n;
        s->u_out = seg + (size_t)(n - n0 + 1) * B;
        rc = launch_step(s, s->adj_dmag[n], s->adj_fmag[n], false);
    }
    return rc;
}

// pd_adjoint_backward with dL_du and dL_dc in host memory (device false) or
// in device memory (device true), both in the caller's node order.
int adjoint_backward(pd_sim *s, const double *dL_du, double *dL_dc,
                     bool device)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->adj_ready)
        return fail(PD_E_STATE, "no finished adjoint recording: call "
                                "pd_adjoint_start and run its steps");
    if (!dL_du || !dL_dc)
        return fail(PD_E_ARG, "dL_du and dL_dc are required");
    if (!s->has_cnode)
        return fail(PD_E_STATE, "the node stiffness field was cleared after "
                                "the recording: set it again");
    const size_t N = (size_t)s->n, B = 3 * N, BB = B * sizeof(double);
    // with every u kept, the recording is one segment that needs no replay,
    // and the state is not touched
    const bool replay = !s->adj_all || s->adj_changed;
    const int nsteps = s->adj_nsteps, every = replay ? s->adj_every : nsteps;
    // with a checkpoint of every step there is no step to run again
    if (replay && s->retile_pending && std::min(every, nsteps) > 1)
        return tiles_pending();
    const int nck = (nsteps + every - 1) / every;
    hipStream_t st = s->stream;
    HIPCHK(hipStreamSynchronize(st));
    if (replay) {
        HIPCHK(s->fin_u.reserve(B));
        HIPCHK(s->fin_force.reserve(B));
        HIPCHK(s->fin_bforce.reserve(B));
        HIPCHK(hipMemcpyAsync(s->fin_u.p, s->u.p, BB, hipMemcpyDeviceToDevice,
                              st));
        HIPCHK(hipMemcpyAsync(s->fin_force.p, s->force.p, BB,
                              hipMemcpyDeviceToDevice, st));
        HIPCHK(hipMemcpyAsync(s->fin_bforce.p, s->body_force.p, BB,
                              hipMemcpyDeviceToDevice, st));
    }
    if (device) {
        hipLaunchKernelGGL(k_perm, dim3((s->n + 255) / 256), dim3(256), 0, st,
                           s->n, 3, s->tnode.p, dL_du, s->lam[0].p);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemsetAsync(s->gradc.p, 0, N * sizeof(double), st));
    } else {
        const std::vector<double> v = to_internal(s->perm, dL_du, 3);
        HIPCHK(hipMemcpyAsync(s->lam[0].p, v.data(), BB,
                              hipMemcpyHostToDevice, st));
        HIPCHK(hipMemsetAsync(s->gradc.p, 0, N * sizeof(double), st));
        HIPCHK(hipStreamSynchronize(st));
    }
    int cur = 0;
    const int pblocks = (int)((N + 255) / 256);
    AdjArgs aa{};
    aa.ntiles = s->ntiles;
    aa.tiles_per_xcd = (s->ntiles + XCDS - 1) / XCDS;
    aa.dt = s->dt;
    aa.tiles = s->tiles.p;
    aa.halo = s->halo.p;
    aa.cnt = s->cnt.p;
    aa.brk = s->brk.p;
    aa.r0 = s->r0.p;
    aa.flags = s->flags.p;
    aa.loc0 = s->loc0.p;
    aa.il0 = s->il0.p;
    aa.gradc = s->gradc.p;
    // from here on a replay takes the state back to earlier steps
    StateGuard state{s, replay};
    for (int k = nck - 1; k >= 0 && rc == PD_OK; --k) {
        const int n0 = k * every, n1 = std::min(n0 + every, nsteps);
        double *seg = s->seg.p + (s->adj_all ? (size_t)n0 * B : 0);
        if (!s->adj_all)
            HIPCHK(hipMemcpyAsync(seg, s->ckpt.p + (size_t)k * B, BB,
                                  hipMemcpyDeviceToDevice, st));
        if (replay) {
            rc = adjoint_replay(s, seg, n0, n1);
            if (rc)
                break;
        }
        // the records of the segment's last step; each backward step then
        // writes those of the step before it, within the segment
        int ra = 0;
        hipLaunchKernelGGL(k_adj_pack, dim3(pblocks), dim3(256), 0, st, s->n,
                           s->r0.p, seg + (size_t)(n1 - 1 - n0) * B,
                           s->vol.p, s->cnode.p, s->flags.p, s->lam[cur].p,
                           s->arec[ra].p);
        HIPCHK(hipGetLastError());
        for (int n = n1 - 1; n >= n0; --n) {
            aa.step = n;
            aa.rec = s->arec[ra].p;
            aa.lam_out = s->lam[1 - cur].p;
            aa.rec_next = n > n0 ? s->arec[1 - ra].p : nullptr;
            aa.u_prev = n > n0 ? seg + (size_t)(n - 1 - n0) * B : nullptr;
            if (s->ntiles > 0)
                HIPCHK(launch_adjoint(s, aa));
            cur = 1 - cur;
            ra = 1 - ra;
        }
    }
    if (rc)
        return rc;
    if (replay) {
        // back to the end of the recording
        HIPCHK(hipMemcpyAsync(s->u.p, s->fin_u.p, BB, hipMemcpyDeviceToDevice,
                              st));
        HIPCHK(hipMemcpyAsync(s->force.p, s->fin_force.p, BB,
                              hipMemcpyDeviceToDevice, st));
        HIPCHK(hipMemcpyAsync(s->body_force.p, s->fin_bforce.p, BB,
                              hipMemcpyDeviceToDevice, st));
        rc = adjoint_restore(s, nsteps);
        if (rc)
            return rc;
        s->step_counter = nsteps;
        state.away = false;
    }
    if (device) {
        hipLaunchKernelGGL(k_unperm, dim3((s->n + 255) / 256), dim3(256), 0,
                           st, s->n, 1, s->tnode.p, s->gradc.p, dL_dc);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(st));
        return PD_OK;
    }
    return download_caller(s, dL_dc, s->gradc.p, 1);
}

}  // namespace

int pd_adjoint_backward(pd_sim *s, const double *dL_du, double *dL_dc)
{
    return adjoint_backward(s, dL_du, dL_dc, false);
}

int pd_adjoint_backward_device(pd_sim *s, const double *dL_du, double *dL_dc)
{
    return adjoint_backward(s, dL_du, dL_dc, true);
}

int pd_write_device(pd_sim *s, double *u, double *damage)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    if (damage) {
        HIPCHK(launch_export(s, 0, damage, u));
    } else if (u) {
        hipLaunchKernelGGL(k_unperm, dim3((s->n + 255) / 256), dim3(256), 0,
                           s->stream, s->n, 3, s->tnode.p, s->u.p, u);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(s->stream));
    return PD_OK;
}

int pd_adjoint_stop(pd_sim *s)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    HIPCHK(hipStreamSynchronize(s->stream));
    adjoint_release(s);
    return PD_OK;
}

int pd_write(pd_sim *s, double *u, double *ud, double *udd, double *force,
             double *body_force, double *damage, int *nlist, int *n_neigh)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    const int N = s->n;
    if (u)
        HIPCHK(s->wbuf.reserve(3 * (size_t)N));
    HIPCHK(launch_export(s, nlist ? 1 : 0, s->damage.p,
                         u ? s->wbuf.p : nullptr));
    if (nlist && s->layout == PD_LAYOUT_COMPACT) {
        hipLaunchKernelGGL(k_export_rows, dim3(row_blocks(N, ROW_LANES)),
                           dim3(256), 0,
                           s->stream, N, s->K, s->tnode.p, s->cnt.p,
                           s->chunk0.p, s->stride.p, s->gidx.p, s->rslot.p,
                           s->nlist_ref.p);
        HIPCHK(hipGetLastError());
    }
    if (u)
        HIPCHK(hipMemcpyAsync(u, s->wbuf.p, 3 * (size_t)N * sizeof(double),
                              hipMemcpyDeviceToHost, s->stream));
    if (damage)
        HIPCHK(hipMemcpyAsync(damage, s->damage.p, (size_t)N * sizeof(double),
                              hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    const struct {
        double *dst;
        const double *src;
    } fields[] = {{ud, s->ud.p}, {udd, s->udd.p},
                  {force, s->force.p}, {body_force, s->body_force.p}};
    for (const auto &f : fields) {
        if (f.dst) {
            rc = download_caller(s, f.dst, f.src, 3);
            if (rc)
                return rc;
        }
    }
    if (body_force) {
        // stored only on force-BC DOFs; equal to force everywhere else
        std::vector<double> tmp;
        const double *f = force;
        if (!f) {
            tmp.resize(3 * (size_t)N);
            rc = download_caller(s, tmp.data(), s->force.p, 3);
            if (rc)
                return rc;
            f = tmp.data();
        }
        for (size_t q = 0; q < 3 * (size_t)N; ++q)
            if (!((s->h_flags[q / 3] >> (3 + (int)(q % 3))) & 1))
                body_force[q] = f[q];
    }
    if (nlist) {
        const size_t NB = (size_t)N * s->K * sizeof(int);
        if (s->layout == PD_LAYOUT_SLOT)
            HIPCHK(hipMemcpy(nlist, s->out_nlist.p, NB, hipMemcpyDeviceToHost));
        else
            HIPCHK(hipMemcpy(nlist, s->nlist_ref.p, NB, hipMemcpyDeviceToHost));
    }
    if (n_neigh)
        HIPCHK(hipMemcpy(n_neigh, s->out_nneigh.p, (size_t)N * sizeof(int),
                         hipMemcpyDeviceToHost));
    return PD_OK;
}

int pd_get_regimes(pd_sim *s, int *regimes)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!s->has_buffers)
        return no_buffers(s);
    if (!regimes)
        return fail(PD_E_ARG, "regimes is NULL");
    const size_t NK = (size_t)s->n * s->K;
    if (!s->state.p) {
        std::memset(regimes, 0, NK * sizeof(int));
        return PD_OK;
    }
    DevBuf<int> out;
    HIPCHK(out.alloc(NK));
    HIPCHK(hipMemsetAsync(out.p, 0, NK * sizeof(int), s->stream));
    const int blocks = (s->n + 255) / 256;
    hipLaunchKernelGGL(k_export_regimes, dim3(blocks), dim3(256), 0,
                       s->stream, s->n, s->K, s->tnode.p, s->cnt.p,
                       s->chunk0.p, s->stride.p, s->pos.p, s->state.p,
                       s->gidx.p, s->nregimes, out.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s->stream));
    HIPCHK(hipMemcpy(regimes, out.p, NK * sizeof(int), hipMemcpyDeviceToHost));
    return PD_OK;
}

int pd_live_bonds(pd_sim *s, long long *count)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (!count)
        return fail(PD_E_ARG, "count is NULL");
    if (!s->has_buffers)
        return no_buffers(s);
    HIPCHK(hipMemsetAsync(s->counter.p, 0, sizeof(unsigned long long),
                          s->stream));
    hipLaunchKernelGGL(k_live, dim3(row_blocks(s->n, CHUNK_LANES)),
                       dim3(256), 0,
                       s->stream, s->n, s->cnt.p, s->chunk0.p, s->stride.p,
                       s->loc.p, s->counter.p);
    HIPCHK(hipGetLastError());
    unsigned long long h = 0;
    HIPCHK(hipMemcpyAsync(&h, s->counter.p, sizeof(h), hipMemcpyDeviceToHost,
                          s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    *count = (long long)h;
    return PD_OK;
}

int pd_synchronize(pd_sim *s)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    HIPCHK(hipStreamSynchronize(s->stream));
    return PD_OK;
}

int pd_tile_stats(pd_sim *s, int *ntiles, int *hmax, int *hstride,
                  long long *halo_total, long long *slots)
{
    int rc = check_sim(s);
    if (rc)
        return rc;
    if (ntiles)
        *ntiles = s->ntiles;
    if (hmax)
        *hmax = s->hmax;
    if (hstride)
        *hstride = s->hstride;
    if (halo_total)
        *halo_total = (long long)s->halo.n;
    if (slots)
        *slots = (long long)s->nslots;
    return PD_OK;
}

void pd_destroy(pd_sim *s)
{
    if (!s)
        return;
    (void)hipSetDevice(s->device);
    if (s->stream)
        (void)hipStreamSynchronize(s->stream);
    if (s->ev0)
        (void)hipEventDestroy(s->ev0);
    if (s->ev1)
        (void)hipEventDestroy(s->ev1);
    if (s->stream)
        (void)hipStreamDestroy(s->stream);
    delete s;
}

int pd_bond_check(int device, int n, const double *ri, const double *rj,
                  const double *r0i, const double *r0j, double s0,
                  int flags, double *l, double *l0, double *s,
                  double *s_exact, int *broken)
{
    if (n <= 0 || !ri || !rj || !r0i || !r0j || !l || !l0 || !s ||
        !s_exact || !broken)
        return fail(PD_E_ARG, "pd_bond_check: bad arguments");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(PD_E_NODEV, "no HIP device is available");
    HIPCHK(hipSetDevice(device));
    const size_t N = (size_t)n;
    DevBuf<double> d_ri, d_rj, d_r0i, d_r0j, d_l, d_l0, d_s, d_se;
    DevBuf<int> d_b;
    HIPCHK(upload(d_ri, ri, 3 * N));
    HIPCHK(upload(d_rj, rj, 3 * N));
    HIPCHK(upload(d_r0i, r0i, 3 * N));
    HIPCHK(upload(d_r0j, r0j, 3 * N));
    HIPCHK(d_l.alloc(N));
    HIPCHK(d_l0.alloc(N));
    HIPCHK(d_s.alloc(N));
    HIPCHK(d_se.alloc(N));
    HIPCHK(d_b.alloc(N));
    const auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((n + CHECK_BLOCK - 1) / CHECK_BLOCK),
                           dim3(CHECK_BLOCK), 0, 0, n, d_ri.p, d_rj.p,
                           d_r0i.p, d_r0j.p, s0, d_l.p, d_l0.p, d_s.p, d_se.p,
                           d_b.p);
    };
    const bool cla = (flags & PD_CHECK_OPENCL) != 0;
    if (flags & PD_CHECK_TENSION)
        cla ? go(k_bond_check<true, true>) : go(k_bond_check<true, false>);
    else
        cla ? go(k_bond_check<false, true>) : go(k_bond_check<false, false>);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    HIPCHK(hipMemcpy(l, d_l.p, N * sizeof(double), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(l0, d_l0.p, N * sizeof(double), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(s, d_s.p, N * sizeof(double), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(s_exact, d_se.p, N * sizeof(double),
                     hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(broken, d_b.p, N * sizeof(int), hipMemcpyDeviceToHost));
    return PD_OK;
}

int pd_neighbour_list(int n, const double *x, double horizon, int *family,
                      int *nlist, int max_neighbours, int pad_value)
{
    if (n <= 0 || !x || !family)
        return fail(PD_E_ARG, "nnodes, coords and family are required");
    if (!(horizon > 0.0))
        return fail(PD_E_ARG, "horizon must be > 0");
    double lo[3] = {x[0], x[1], x[2]}, hi[3] = {x[0], x[1], x[2]};
    for (int i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], x[3 * (size_t)i + d]);
            hi[d] = std::max(hi[d], x[3 * (size_t)i + d]);
        }
    long dim[3];
    long total = 1;
    for (int d = 0; d < 3; ++d) {
        dim[d] = std::max(1L, (long)std::floor((hi[d] - lo[d]) / horizon) + 1);
        dim[d] = std::min(dim[d], 1L << 20);
        total *= dim[d];
        if (total > (1L << 28))
            return fail(PD_E_LIMIT, "cell grid too large for this horizon");
    }
    auto cell_of = [&](int i, int d) {
        long c = (long)std::floor((x[3 * (size_t)i + d] - lo[d]) / horizon);
        return std::min(std::max(c, 0L), dim[d] - 1);
    };
    std::vector<long> cstart(total + 1, 0);
    std::vector<long> cid(n);
    for (int i = 0; i < n; ++i) {
        cid[i] = (cell_of(i, 0) * dim[1] + cell_of(i, 1)) * dim[2] + cell_of(i, 2);
        cstart[cid[i] + 1]++;
    }
    for (long c = 0; c < total; ++c)
        cstart[c + 1] += cstart[c];
    std::vector<int> members(n);
    {
        std::vector<long> fillp(cstart.begin(), cstart.end() - 1);
        for (int i = 0; i < n; ++i)
            members[fillp[cid[i]]++] = i;
    }
    const double h2 = horizon * horizon;
    std::atomic<int> overflow{0};
    run_parallel(n, [&](int a, int b) {
        std::vector<int> row;
        for (int i = a; i < b; ++i) {
            row.clear();
            const long ci[3] = {cell_of(i, 0), cell_of(i, 1), cell_of(i, 2)};
            for (long c0 = std::max(0L, ci[0] - 1); c0 <= std::min(dim[0] - 1, ci[0] + 1); ++c0)
                for (long c1 = std::max(0L, ci[1] - 1); c1 <= std::min(dim[1] - 1, ci[1] + 1); ++c1)
                    for (long c2 = std::max(0L, ci[2] - 1); c2 <= std::min(dim[2] - 1, ci[2] + 1); ++c2) {
                        const long c = (c0 * dim[1] + c1) * dim[2] + c2;
                        for (long m = cstart[c]; m < cstart[c + 1]; ++m) {
                            const int j = members[m];
                            if (j == i)
                                continue;
                            double d0 = x[3 * (size_t)j] - x[3 * (size_t)i];
                            double d1 = x[3 * (size_t)j + 1] - x[3 * (size_t)i + 1];
                            double d2 = x[3 * (size_t)j + 2] - x[3 * (size_t)i + 2];
                            d0 = d0 * d0;
                            d1 = d1 * d1;
                            d2 = d2 * d2;
                            if ((d0 + d1) + d2 <= h2)
                                row.push_back(j);
                        }
                    }
            std::sort(row.begin(), row.end());
            family[i] = (int)row.size();
            if (nlist) {
                if ((int)row.size() > max_neighbours) {
                    overflow = 1;
                    continue;
                }
                int *dst = nlist + (size_t)i * max_neighbours;
                std::copy(row.begin(), row.end(), dst);
                for (int p = (int)row.size(); p < max_neighbours; ++p)
                    dst[p] = pad_value;
            }
        }
    });
    if (overflow)
        return fail(PD_E_LIMIT, "a node has more than max_neighbours bonds");
    return PD_OK;
}

}  // extern "C"
