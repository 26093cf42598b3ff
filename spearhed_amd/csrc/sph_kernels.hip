// sph_kernels.hip -- hand-written gfx950 kernels of the SPH-MHD particle step.
//
// Stage -> kernels (reference stage in brackets):
//   drift + bin   k_drift_bin        [PushVelocity, PushVelocity.hpp:35-42; + supercell key/histogram; large
//                                     steps store the drift in k_gather]
//   resort        k_scan_local, k_scan_top (large tables), k_scatter, k_gather
//                                    [UpdateVolumes RegionBoundsUpdate.hpp:175-214 and the frame index
//                                     FrameIndex.hpp:209-296, replaced by a counting sort by (cell, id)]
//   density       k_density<CH>      [UpdateDensity, DensitySummation.hpp:104-138]
//   forces        k_forces<CH, MHD>  [UpdateHydroForces, HydroForces.hpp:183-214, + AV/MHD/cleaning]
//   integrate     k_kick, k_finalize (within k_kick for small sets)
//                                    [EulerIntegrate, EulerIntegrate.hpp:43-52, + CFL and FP64 sums]
//
// Pair passes: one wave64 per target supercell. The 27 neighbour supercells form a virtual list
// whose candidates within the support radius of the targets' bounding box are staged chunk by
// chunk into LDS (records pre-shifted by the periodic image or the supercell-origin offset,
// ParticleParticleInteraction.hpp:236-264). The cell's nt targets are
// spread over the wave as (target t, sub-lane k) with K = floor(64/nt) sub-lanes per target, so a
// supercell of ~14 particles still fills the wave; sub-lane k owns candidates v = c*K + k.
// The density pass culls each lane's candidates 32 at a time into a bit mask (strict r2 < H^2,
// ParticleParticleInteraction.hpp:291) and stores the masks; the force pass replays them instead
// of culling again. Each lane then runs the pair physics over its set bits; with pair_balance the
// accepted candidates of a target's K lanes are first compacted into LDS and shared round-robin
// among those K lanes (ceil(accepted/K) iterations instead of the slowest lane's count, at the
// price of a prefix scan and two barriers per 32 candidates). The K partial sums are combined in lane order:
// every summation order depends only on the run's own data, so a run gives bit-identical results
// alone or batched with others.

#include <type_traits>

#include "sph_device.hpp"
#include "sph_launch.hpp"

namespace sph {

// ------------------------------------------------------------------------------------------------
// helpers
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ int find_run_by_cell(const RunDev* runs, int nruns, int cell)
{
    int lo = 0, hi = nruns - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (runs[mid].c0 <= cell) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Inclusive sum over the lanes of a wave by DPP row shifts and row broadcasts (six additions).
__device__ __forceinline__ int dpp_incl_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

// An LDS record at a byte offset from its array: the pair loops keep byte offsets so that a slot's
// address is one 24-bit multiply-add (candidate bit x lane stride + the lane's first slot).
template <class T>
__device__ __forceinline__ const T& lds_at(const T* base, int byte_off)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}

__device__ __forceinline__ int wave_incl_max(int v)
{
    int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int t = __shfl_up(v, off, 64);
        if (lane >= off) v = v > t ? v : t;
    }
    return v;
}

// XCD-aware mapping: the hardware deals consecutive workgroups round-robin to the 8 XCDs; give
// each XCD one contiguous range of supercells so that neighbouring cells share an L2.
__device__ __forceinline__ int xcd_cell(int bid, int nblk_total, int ncell)
{
    int per = nblk_total >> 3;
    int cell = (bid & 7) * per + (bid >> 3);
    return cell < ncell ? cell : -1;
}

// ------------------------------------------------------------------------------------------------
// drift + supercell key + histogram rank (wave-aggregated atomics: particles arrive sorted by
// cell, so runs of equal keys in a wave take one atomicAdd per run)
// ------------------------------------------------------------------------------------------------
// A coordinate after a drift of dt, wrapped into a periodic box.
__device__ __forceinline__ double drifted(const RunDev& R, int a, double x, float v, double dt)
{
#pragma clang fp contract(off)
    x = x + (double)v * dt;
    if (run_periodic(R.flags, a)) {
        const double hi = R.lo[a] + R.L[a];
        if (x >= hi) x = x - R.L[a];
        else if (x < R.lo[a]) x = x + R.L[a];
    }
    return x;
}
__device__ __forceinline__ float drifted(const RunDev& R, int a, float x, float v, double dt)
{
#pragma clang fp contract(off)
    x = x + v * (float)dt;
    if (run_periodic(R.flags, a)) {
        const float hi = R.lo32[a] + R.L32[a];
        if (x >= hi) x = x - R.L32[a];
        else if (x < R.lo32[a]) x = x + R.L32[a];
    }
    return x;
}
// Whether a particle of run r moves in a drift of dt: a run whose next step primes it (fresh initial data) does
// not move in that step, nor does a run without a CFL bound (no live target: dt = +inf).
__device__ __forceinline__ bool moves(int priming, uint8_t species, uint8_t live, double dt)
{
    return is_movable(species, live) && !priming && isfinite(dt);
}

// STORE: the drifted positions are stored; otherwise the gather of the same step drifts them again on their way
// to their sorted place.
template <bool MIXED, bool STORE>
__global__ __launch_bounds__(256) void k_drift_bin(const RunDev* __restrict__ runs, StateBuf S, WorkBuf W,
                                                   double dt_host, int do_drift)
{
    const int b = blockIdx.x;
    const int r = W.blk_run[b];
    const RunDev& R = runs[r];
    const int64_t local = (int64_t)(b - R.kb_first) * 256 + threadIdx.x;
    const bool active = local < R.np;
    const int64_t i = R.p0 + (active ? local : 0);
    uint32_t key = 0xffffffffu;
    if (active) {
        const double dt = dt_host > 0.0 ? dt_host : W.dt[r];
        const bool mov = do_drift && moves(W.prime_flag[r], S.species[i], S.mask[i], dt);
        int c[3];
        for (int a = 0; a < 3; ++a) {
#pragma clang fp contract(off)
            int ci;
            if (MIXED) {
                double x = S.pos64[a][i];
                if (mov) {
                    x = drifted(R, a, x, S.vel[a][i], dt);
                    if (STORE) S.pos64[a][i] = x;
                }
                ci = (int)fmin(fmax(floor((x - R.lo[a]) * R.inv_s[a]), 0.0), (double)(R.n[a] - 1));
            } else {
                float x = S.pos32[a][i];
                if (mov) {
                    x = drifted(R, a, x, S.vel[a][i], dt);
                    if (STORE) S.pos32[a][i] = x;
                }
                ci = (int)fminf(fmaxf(floorf((x - R.lo32[a]) * R.inv_s32[a]), 0.0f), (float)(R.n[a] - 1));
            }
            // clamped before the conversion: outside the box (or not finite) maps to an edge cell
            c[a] = ci;
        }
        key = (uint32_t)(R.c0 + c[0] + R.n[0] * (c[1] + R.n[1] * c[2]));
        W.key[i] = key;
    }
    // segments of equal consecutive keys within the wave
    const int lane = threadIdx.x & 63;
    const uint32_t prev = __shfl_up(key, 1, 64);
    const bool head = lane == 0 || prev != key || !active;
    const int hl = wave_incl_max(head ? lane : 0);
    const uint64_t heads = __ballot(head);
    uint32_t base = 0;
    if (head && active) {
        const uint64_t after = lane == 63 ? 0ull : (heads >> (lane + 1)) << (lane + 1);
        const int next = after ? __builtin_ctzll(after) : 64;
        base = atomicAdd(&W.count[key], (uint32_t)(next - lane));
    }
    base = __shfl(base, hl, 64);
    if (active) W.rank[i] = base + (uint32_t)(lane - hl);
}

// ------------------------------------------------------------------------------------------------
// exclusive scan of the per-cell histogram -> cell starts (absolute particle index): within blocks of
// kScanBlock cells in place (k_scan_local), then the blocks' offsets added by k_scatter, which needs the
// starts first. The offsets of up to kScatterBlocks blocks are scanned by each workgroup of k_scatter for
// itself (half a million supercells: one load per thread and a scan in LDS, against two more launches of
// 4.7 us each at any size, and 1.4 us more in the scatter of 2,097,152 particles); more of them are scanned
// by k_scan_top in between. A table of up to kScatterCells is scanned whole by each workgroup of k_scatter:
// no other launch, for 0.4 us more in the scatter of 131,044 particles in 5,625 supercells (33 KB of LDS
// per workgroup bound the limit: four workgroups per compute unit).
// ------------------------------------------------------------------------------------------------
constexpr int kScanPerThread = 8;
constexpr int kScanBlock = 256 * kScanPerThread;
constexpr int kScatterBlocks = 256;
constexpr int kScatterCells = 8192;

__device__ __forceinline__ uint32_t block_excl_scan256(uint32_t s, uint32_t (&wsum)[4], uint32_t& total)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint32_t incl = (uint32_t)dpp_incl_scan((int)s);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        before += w < wid ? wsum[w] : 0u;
        total += wsum[w];
    }
    return before + incl - s;
}

__global__ __launch_bounds__(256) void k_scan_local(uint32_t* __restrict__ count, uint32_t* __restrict__ bsum, int n)
{
    __shared__ uint32_t wsum[4];
    const int base = blockIdx.x * kScanBlock + threadIdx.x * kScanPerThread;
    uint32_t v[kScanPerThread];
    const bool whole = base + kScanPerThread <= n;  // the table is 256-byte aligned: two 16-byte accesses
    if (whole) {
        const uint4 a = reinterpret_cast<const uint4*>(count + base)[0];
        const uint4 b = reinterpret_cast<const uint4*>(count + base)[1];
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    } else {
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k) v[k] = base + k < n ? count[base + k] : 0u;
    }
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k) {
        const uint32_t c = v[k];
        v[k] = s;
        s += c;
    }
    uint32_t total;
    const uint32_t off = block_excl_scan256(s, wsum, total);
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k) v[k] += off;
    if (whole) {
        reinterpret_cast<uint4*>(count + base)[0] = make_uint4(v[0], v[1], v[2], v[3]);
        reinterpret_cast<uint4*>(count + base)[1] = make_uint4(v[4], v[5], v[6], v[7]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k)
            if (base + k < n) count[base + k] = v[k];
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

// block sums -> exclusive offsets, in place, with the total after the last
__global__ __launch_bounds__(1024) void k_scan_top(uint32_t* __restrict__ bsum, int nb)
{
    __shared__ uint32_t wsum[16];
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < nb; base += 1024) {
        int e = base + threadIdx.x;
        uint32_t s = e < nb ? bsum[e] : 0u;
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        int incl = dpp_incl_scan((int)s);
        if (lane == 63) wsum[wid] = (uint32_t)incl;
        __syncthreads();
        uint32_t woff = carry;
        for (int w = 0; w < wid; ++w) woff += wsum[w];
        if (e < nb) bsum[e] = woff + (uint32_t)incl - s;
        __syncthreads();
        if (threadIdx.x == 1023) carry = woff + (uint32_t)incl;
        __syncthreads();
    }
    if (threadIdx.x == 0) bsum[nb] = carry;
}

// ------------------------------------------------------------------------------------------------
// scatter (histogram slot) and gather (final slot = cell start + rank of id within the cell)
// ------------------------------------------------------------------------------------------------
// The workgroups past the particles' nkb only write cell starts (launch_scatter_gather).
template <bool WHOLE>
__global__ __launch_bounds__(256) void k_scatter(const RunDev* __restrict__ runs, StateBuf S, WorkBuf W, int ncell,
                                                 int nkb)
{
    __shared__ uint32_t wsum[4];
    const int b = blockIdx.x;
    bool active = false;
    int64_t i = 0;
    uint32_t key = 0, rank = 0;
    uint64_t id = 0;
    if (b < nkb) {
        const RunDev& R = runs[W.blk_run[b]];
        const int64_t local = (int64_t)(b - R.kb_first) * 256 + threadIdx.x;
        active = local < R.np;
        i = R.p0 + (active ? local : 0);
    }
    if (active) {
        key = W.key[i];
        rank = W.rank[i];
        id = S.id[i];
    }
    const int first = b * 256 + (int)threadIdx.x, step = (int)gridDim.x * 256;  // the entries of cs to write
    uint32_t slot = 0;
    if constexpr (WHOLE) {
        constexpr int kTile = 1024;  // four supercells per thread
        __shared__ __align__(16) uint32_t start[kScatterCells + 4];
        uint4 v[kScatterCells / kTile];
#pragma unroll
        for (int t = 0; t < kScatterCells / kTile; ++t) {
            const int e = t * kTile + 4 * (int)threadIdx.x;
            v[t] = make_uint4(0u, 0u, 0u, 0u);
            if (e + 4 <= ncell) {
                v[t] = *reinterpret_cast<const uint4*>(W.count + e);  // the table is 256-byte aligned
            } else if (e < ncell) {
                v[t].x = W.count[e];
                if (e + 1 < ncell) v[t].y = W.count[e + 1];
                if (e + 2 < ncell) v[t].z = W.count[e + 2];
            }
        }
        uint32_t carry = 0;
#pragma unroll
        for (int t = 0; t < kScatterCells / kTile; ++t) {
            if (t * kTile > ncell) break;  // the entry at ncell is written too
            uint32_t total;
            const uint32_t x = carry + block_excl_scan256(v[t].x + v[t].y + v[t].z + v[t].w, wsum, total);
            *reinterpret_cast<uint4*>(start + t * kTile + 4 * (int)threadIdx.x) =
                make_uint4(x, x + v[t].x, x + v[t].x + v[t].y, x + v[t].x + v[t].y + v[t].z);
            carry += total;
            __syncthreads();
        }
        if (ncell == kScatterCells && threadIdx.x == 0) start[ncell] = carry;
        __syncthreads();
        slot = start[key] + rank;
        for (int e = first; e <= ncell; e += step) W.cs[e] = start[e];
    } else {
        __shared__ uint32_t pre[kScatterBlocks + 1];  // the scan blocks' offsets, then the total
        const int nb = (ncell + kScanBlock - 1) / kScanBlock;
        const uint32_t* off = W.bsum;
        if (nb <= kScatterBlocks) {
            uint32_t total;
            const uint32_t x = block_excl_scan256((int)threadIdx.x < nb ? W.bsum[threadIdx.x] : 0u, wsum, total);
            pre[threadIdx.x] = x;
            if ((int)threadIdx.x == nb - 1) pre[nb] = total;
            __syncthreads();
            off = pre;
        }
        slot = W.count[key] + off[key / kScanBlock] + rank;
        for (int e = first; e <= ncell; e += step) W.cs[e] = e < ncell ? W.count[e] + off[e / kScanBlock] : off[nb];
    }
    if (active) {
        W.tmp[slot] = (uint32_t)i;
        W.tmpid[slot] = id;
    }
}

// STATE: all of the state is gathered; otherwise only what the density pass of a call without a state needs
// (identity, mass, h and position: 40 bytes per particle read and written less).
template <bool MIXED, bool STATE>
__global__ __launch_bounds__(256) void k_gather(const RunDev* __restrict__ runs, StateBuf Sold, StateBuf Snew,
                                                WorkBuf W, int has_mhd, int ncell, int nkb, double dt_host,
                                                int do_drift)
{
    const int b = blockIdx.x;
    // histogram reset for the next resort
    for (int e = b * 256 + (int)threadIdx.x; e < ncell; e += (int)gridDim.x * 256) W.count[e] = 0u;
    if (b >= nkb) return;  // only there for the histogram (launch_scatter_gather)
    const int r = W.blk_run[b];
    const RunDev& R = runs[r];
    const int64_t local = (int64_t)(b - R.kb_first) * 256 + threadIdx.x;
    if (local >= R.np) return;
    const int64_t q = R.p0 + local;
    if (local == 0) W.chbits[r] = 0u;  // cleaning-speed maximum of the coming density pass
    const uint32_t i = W.tmp[q];
    const uint32_t c = W.key[i];
    const uint64_t myid = W.tmpid[q];
    // the particle's old record is read before the rank search, so its loads overlap the search's
    const double dt = dt_host > 0.0 || !do_drift ? dt_host : W.dt[r];
    const int priming = do_drift ? W.prime_flag[r] : 0;
    const uint8_t live = Sold.mask[i], sp = Sold.species[i];
    const float m = Sold.mass[i], hh = Sold.h[i], uu = STATE ? Sold.u[i] : 0.f, rh = STATE ? Sold.rho[i] : 0.f;
    float vel[3] = {0.f, 0.f, 0.f}, bf[3] = {0.f, 0.f, 0.f}, ps = 0.f;
    double x64[3] = {0.0, 0.0, 0.0};
    float x32[3] = {0.f, 0.f, 0.f};
    for (int a = 0; a < 3; ++a) {
        if (STATE) vel[a] = Sold.vel[a][i];
        if (MIXED) x64[a] = Sold.pos64[a][i];
        else x32[a] = Sold.pos32[a][i];
    }
    if (has_mhd) {
        for (int a = 0; a < 3; ++a) bf[a] = Sold.B[a][i];
        ps = Sold.psi[i];
    }
    const uint32_t cb = W.cs[c], ce = W.cs[c + 1];
    // rank within the supercell = number of smaller ids in it; four independent loads per round
    uint32_t rank = 0, mm = cb;
    for (; mm + 4 <= ce; mm += 4) {
        const uint64_t a0 = W.tmpid[mm], a1 = W.tmpid[mm + 1], a2 = W.tmpid[mm + 2], a3 = W.tmpid[mm + 3];
        rank += (a0 < myid ? 1u : 0u) + (a1 < myid ? 1u : 0u) + (a2 < myid ? 1u : 0u) + (a3 < myid ? 1u : 0u);
    }
    for (; mm < ce; ++mm) rank += (W.tmpid[mm] < myid) ? 1u : 0u;
    if (do_drift) {  // the step's drift, binned but not stored
        if (moves(priming, sp, live, dt))
            for (int a = 0; a < 3; ++a) {
                if (MIXED) x64[a] = drifted(R, a, x64[a], vel[a], dt);
                else x32[a] = drifted(R, a, x32[a], vel[a], dt);
            }
    }
    const uint32_t f = cb + rank;
    if (W.perm) W.perm[f] = (int32_t)i;

    Snew.id[f] = myid;
    Snew.mask[f] = live;
    Snew.species[f] = sp;
    Snew.mass[f] = m;
    Snew.h[f] = hh;
    if (STATE) {
        Snew.u[f] = uu;
        Snew.rho[f] = rh;
    }
    float pc[3];
    const int lc = (int)c - R.c0;
    const int cxyz[3] = {lc % R.n[0], (lc / R.n[0]) % R.n[1], lc / (R.n[0] * R.n[1])};
    for (int a = 0; a < 3; ++a) {
#pragma clang fp contract(off)
        if (STATE) Snew.vel[a][f] = vel[a];
        if (MIXED) {
            const double x = x64[a];
            Snew.pos64[a][f] = x;
            pc[a] = (float)((x - R.lo[a]) - (double)cxyz[a] * R.s[a]);
        } else {
            Snew.pos32[a][f] = x32[a];
            pc[a] = x32[a];
        }
    }
    if (has_mhd) {
        for (int a = 0; a < 3; ++a) Snew.B[a][f] = bf[a];
        Snew.psi[f] = ps;
    }
    float4 p0 = is_source(sp, live) ? make_float4(pc[0], pc[1], pc[2], m)
                                    : make_float4(kSentinel, kSentinel, kSentinel, 0.0f);
    W.P0[f] = p0;
}

// ------------------------------------------------------------------------------------------------
// shared set-up of the supercell stencil's virtual neighbour list (one wave): the (2 reach + 1)^3
// supercells around a cell, x fastest, concatenated. NS = 27 serves supercells of edge >= H (reach
// 1), NS = 125 also those of edge >= H/2 (reach 2: 5^3 stencil, about 58% of the candidates).
// ------------------------------------------------------------------------------------------------
template <int NS>
struct NbListT {
    float4 t[NS];     // staged-position shift of a stencil supercell (x, y, z) and its first particle less its first
                      // list index (int bits): list index v of that supercell is particle v + this
    int off[NS + 1];  // list index of its first candidate; entries past the run's stencil hold the total, so no
                      // search selects them
};
template <int RMAX>
using NbListR = NbListT<RMAX == 1 ? 27 : 125>;
// LDS candidate slot indices of the balanced pair loop
template <int CH>
using ListT = typename std::conditional<(CH <= 256), uint8_t, uint16_t>::type;

// Arguments of the pair passes. The kernels read them where they are used, from the kernel-argument
// segment (the struct is their only parameter, at its start): as plain parameters some fifty pointers are
// loaded at the entry, more than the scalar registers hold, and the spills cost vector instructions
// (350 of a density wave's 2,500).
struct PairArgs {
    const RunDev* runs;
    int nruns, ncell_tot, nblk_total, kmax;
    int dense;  // a particle per supercell on average, or more
    StateBuf S;
    WorkBuf W;
};
__device__ __forceinline__ const PairArgs& pair_args()
{
    return *(const PairArgs*)__builtin_amdgcn_kernarg_segment_ptr();
}

// A run's constants in the constant address space: scalar loads wherever they are used, also after the
// wave's own stores (no pair pass writes the table).
using RunC = const __attribute__((address_space(4))) RunDev;

// A value that is the same in every lane, moved to a scalar register: what follows from it is then
// computed by the scalar unit instead of taking vector issue slots (the pair passes are bound by them).
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// x / d for uniform x, d > 0 (1 / d given to within an ulp or two): the float quotient of x + 1/2 stays at
// least 1/(2 d) away from the next whole number, more than its rounding error below 2^20; larger x divide.
__device__ __forceinline__ int quot(int x, int d, float rd)
{
    return x < (1 << 20) ? (int)(((float)x + 0.5f) * rd) : x / d;
}
__device__ __forceinline__ int uquot(int x, int d, float rd) { return uniform(quot(x, d, rd)); }

// Element at a 32-bit byte offset from a uniform base: the offset is one vector register and the base
// stays in scalar ones (no 64-bit vector address arithmetic). A context holds at most 2^30 particles, so
// columns of up to four bytes are reached from their start; 16-byte records from the wave's first one.
template <class T>
__device__ __forceinline__ T& at32(T* base, uint32_t byte_off)
{
    return *(T*)((char*)base + byte_off);
}

// Particle t (per lane) of the supercell whose first particle is t0 (uniform): offsets of its columns.
struct Slot {
    int t0;
    uint32_t i;    // index in a column
    uint32_t t16;  // byte offset of its record from that of t0

    __device__ __forceinline__ Slot(int t0_, uint32_t t) : t0(t0_), i((uint32_t)t0_ + t), t16(t * 16u) {}
    template <class T>
    __device__ __forceinline__ T& col(T* base) const
    {
        static_assert(sizeof(T) <= 4, "a wider column needs a 64-bit offset");
        return at32(base, i * (uint32_t)sizeof(T));
    }
    __device__ __forceinline__ float4& rec(float4* base) const { return at32(base + t0, t16); }
};

// Maximum over the wave of values whose bits order as unsigned integers (floats >= +0), as a uniform.
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v)
{
    auto step = [&](auto ctrl, auto rows) {
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value,
                                                                 decltype(rows)::value, 0xf, false);
        v = v > o ? v : o;
    };
    step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Neighbour supercell `seg` of cell c in a stencil of side 2 reach + 1 (x fastest, offsets
// d = seg % side - reach, ...): returns false outside a non-periodic axis; else the global cell and
// the staged-position shift (the periodic image for FP32 absolute coordinates, d * cell edge for
// supercell-relative ones). A 1-cell periodic axis is wrapped twice by a reach of 2.
template <bool MIXED, int RMAX>
__device__ __forceinline__ bool nb_cell(RunC& R, const int c[3], int seg, int& cc, float sh[3])
{
    int d[3];
    if (RMAX == 1) {  // seg < 64: quotients by 9 and 3 as multiply-shifts
        const int z = (int)(__umul24((unsigned)seg, 57u) >> 9), yx = seg - 9 * z;
        const int y = (int)(__umul24((unsigned)yx, 11u) >> 5);
        d[0] = yx - 3 * y - 1;
        d[1] = y - 1;
        d[2] = z - 1;
    } else {
        const int r = R.reach, side = 2 * R.reach + 1;
        d[0] = seg % side - r;
        d[1] = (seg / side) % side - r;
        d[2] = seg / (side * side) - r;
    }
    int idx[3];
    bool ok = true;
    for (int a = 0; a < 3; ++a) {
        int x = c[a] + d[a];
        int wrap = 0;
        if (run_periodic(R.flags, a)) {
            if (RMAX == 1) wrap = x < 0 ? -1 : (x >= R.n[a] ? 1 : 0);
            else wrap = x >= 0 ? x / R.n[a] : -((R.n[a] - 1 - x) / R.n[a]);
            x -= wrap * R.n[a];
        } else if (x < 0 || x >= R.n[a]) {
            ok = false;
        }
        idx[a] = x;
        sh[a] = MIXED ? (float)d[a] * R.s32[a] : (float)wrap * R.L32[a];
    }
    cc = R.c0 + idx[0] + R.n[0] * (idx[1] + R.n[1] * idx[2]);
    return ok;
}

// Index of the cell's own supercell in its stencil (the centre).
template <int RMAX>
__device__ __forceinline__ int self_segment(RunC& R)
{
    if (RMAX == 1) return 13;
    const int side = 2 * R.reach + 1;
    return (side * side * side - 1) / 2;
}

// A load that stays where it is written: the compiler otherwise sinks one below the branches that do not need
// it, and its latency adds to that of the loads after them.
__device__ __forceinline__ uint32_t load_early(const uint32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// The stencil of a cell: each lane requests the particle ranges of its supercells (the constructor), then the
// list is built in LDS.
template <bool MIXED, int RMAX>
struct Stencil {
    static constexpr int NS = RMAX == 1 ? 27 : 125, ROUNDS = (NS + 63) / 64;
    uint32_t st[ROUNDS], end[ROUNDS];
    float sh[ROUNDS][3];
    int nseg;

    __device__ __forceinline__ Stencil(RunC& R, int lcell, const uint32_t* __restrict__ cs)
    {
        const int n0 = R.n[0], n1 = R.n[1], n2 = R.n[2];
        const uint32_t div0 = R.div[0], div1 = R.div[1], flags = (uint32_t)R.flags;
        const int c0 = R.c0;
        const uint32_t row = div_by((uint32_t)lcell, (uint32_t)n0, div0);
        const uint32_t plane = div_by(row, (uint32_t)n1, div1);
        const int c[3] = {lcell - (int)row * n0, (int)row - (int)plane * n1, (int)plane};
        const int side = RMAX == 1 ? 3 : 2 * R.reach + 1;
        nseg = RMAX == 1 ? 27 : side * side * side;
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int seg = i * 64 + (int)threadIdx.x;
            st[i] = end[i] = 0;
            sh[i][0] = sh[i][1] = sh[i][2] = 0.f;
            int cc;
            if (seg < nseg && nb_cell<MIXED, RMAX>(R, c, seg, cc, sh[i])) {
                st[i] = load_early(cs + cc);
                end[i] = load_early(cs + cc + 1);
            }
        }
    }
    // Builds the list; returns its total and sets the list index of the cell's own first particle.
    __device__ __forceinline__ int build(RunC& R, NbListR<RMAX>& L, int& self_v0) const
    {
        int carry = 0;
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int seg = i * 64 + (int)threadIdx.x;
            const int cnt = (int)(end[i] - st[i]);
            const int incl = dpp_incl_scan(cnt) + carry;
            if (seg < NS) {
                L.t[seg] = make_float4(sh[i][0], sh[i][1], sh[i][2], __int_as_float((int)st[i] - (incl - cnt)));
                L.off[seg] = seg < nseg ? incl - cnt : 0;  // past the stencil: overwritten with the total below
            }
            if (RMAX == 1) self_v0 = __builtin_amdgcn_readlane(incl - cnt, 13);
            carry = __builtin_amdgcn_readlane(incl, 63);
        }
        // the total after the last stencil entry, and in every entry past the run's stencil
        for (int k = nseg + (int)threadIdx.x; k <= NS; k += 64) L.off[k] = carry;
        __syncthreads();
        if (RMAX != 1) self_v0 = uniform(L.off[self_segment<RMAX>(R)]);
        return carry;
    }
};

// segment of virtual index v (largest k with off[k] <= v, over non-decreasing off[0..NS-1])
template <int NS>
__device__ __forceinline__ int nb_segment(const NbListT<NS>& L, int v)
{
    int k = 0;
#pragma unroll
    for (int step = NS > 64 ? 64 : 16; step >= 1; step >>= 1) {
        int t = k + step;
        if (t < NS && L.off[t] <= v) k = t;
    }
    return k;
}

// ------------------------------------------------------------------------------------------------
// Candidate pre-filter of the chunked pair passes. A candidate farther than the support radius from
// the bounding box of the supercell's targets is farther than that from every target, so the cull
// would reject it for all of them. Both passes drop such candidates before staging and stage the
// others in the same order, so the force pass replays the density pass's masks slot by slot as
// before. With supercells of edge ~H about half of the 27-cell stencil goes (MHD turbulence at 2M
// particles: 381 -> 194 candidates per supercell in a CPU replay), which halves the cull and the
// staging and leaves fewer, fuller chunks for the pair loops. The density pass filters; the force
// pass reads the kept list back from the mask row (recomputing it only where it was not stored).
// ------------------------------------------------------------------------------------------------
constexpr int kPreCap = 768;  // larger stencils, and supercells of more than 64 particles, stage whole

constexpr uint16_t kNoSelf = 0xffff;  // past every staged slot

struct PreList {
    union {
        uint16_t v[kPreCap];       // the kept candidates in list order (pre_entry)
        uint32_t v2[kPreCap / 2];  // the same, two entries per word
    };
    uint16_t self_s[64];  // kept index of each target of the supercell; kNoSelf of one at no finite position
};

// A kept-list entry: the list index (< kPreCap <= 1024) and, for the 27-cell stencil, its segment, so that
// staging needs no search.
template <int NS>
__device__ __forceinline__ uint16_t pre_entry(int v, int sg)
{
    return (uint16_t)(NS == 27 ? v | (sg << 10) : v);
}

// Particle index and position shift of list index v.
template <int NS>
__device__ __forceinline__ int list_candidate(const NbListT<NS>& L, int v, float4& t)
{
    t = L.t[nb_segment(L, v)];
    return v + __float_as_int(t.w);
}

// Particle index and position shift of the kept-list entry e.
template <int NS>
__device__ __forceinline__ int kept_candidate(const NbListT<NS>& L, int e, float4& t)
{
    if (NS != 27) return list_candidate(L, e, t);
    t = L.t[e >> 10];
    return (e & 1023) + __float_as_int(t.w);
}

// Bounding box of the targets among a supercell's nt <= 64 particles (from their position records;
// empty, lo > hi, without targets). Its inputs need no neighbour list: a pass requests them first
// (target_box_load) and reduces them once the list is built (target_box), so the loads overlap.
struct TargetBox {
    float lx, ly, lz, hx, hy, hz;
};

struct TargetBoxInput {
    uint8_t species = 0, mask = 0;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
};

__device__ __forceinline__ TargetBoxInput target_box_load(const StateBuf& S, const WorkBuf& W, int t0, int nt)
{
    const uint32_t lane = threadIdx.x;
    TargetBoxInput in;
    if ((int)lane < nt) {
        in.species = at32(S.species + t0, lane);
        in.mask = at32(S.mask + t0, lane);
        in.o = at32(W.P0 + t0, lane * 16u);  // a target is a source: its record holds its position
    }
    return in;
}

// Minimum or maximum over a wave whose lanes past nt hold the neutral value: rotations within the
// 16-lane rows (every lane reads a valid one, so each is one instruction), then the rows in use.
template <bool MAX>
__device__ __forceinline__ float wave_extreme(float x, int nt)
{
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : fminf(a, b); };
    auto ror = [&](auto n) {
        return __int_as_float(
            __builtin_amdgcn_mov_dpp(__float_as_int(x), 0x120 + decltype(n)::value, 0xf, 0xf, true));
    };
    x = op(x, ror(std::integral_constant<int, 8>{}));
    x = op(x, ror(std::integral_constant<int, 4>{}));
    x = op(x, ror(std::integral_constant<int, 2>{}));
    x = op(x, ror(std::integral_constant<int, 1>{}));
    auto row = [&](int r) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 16 * r)); };
    float m = row(0);
    if (nt > 16) m = op(m, row(1));
    if (nt > 32) m = op(op(m, row(2)), row(3));
    return m;
}

__device__ __forceinline__ TargetBox target_box(const TargetBoxInput& in, int nt)
{
    const bool has = (int)threadIdx.x < nt && is_target(in.species, in.mask);
    TargetBox b;
    b.lx = wave_extreme<false>(has ? in.o.x : INFINITY, nt);
    b.hx = wave_extreme<true>(has ? in.o.x : -INFINITY, nt);
    b.ly = wave_extreme<false>(has ? in.o.y : INFINITY, nt);
    b.hy = wave_extreme<true>(has ? in.o.y : -INFINITY, nt);
    b.lz = wave_extreme<false>(has ? in.o.z : INFINITY, nt);
    b.hz = wave_extreme<true>(has ? in.o.z : -INFINITY, nt);
    return b;
}

// Stencil segments of the list indices [vb, vb + 256) into seg4, one byte each (27-cell stencil): every
// non-empty segment marks its first index with its number, and a running maximum over the bytes (segments
// ascend with the index) fills the rest, `last` being the segment in force at vb. About 25 instructions for
// 256 candidates, where a search per candidate took 20 for each 64.
__device__ __forceinline__ void fill_segments(uint32_t* seg4, int vb, int seg_off, int seg_cnt, uint32_t& last)
{
    const int lane = threadIdx.x;
    seg4[lane] = 0u;
    __syncthreads();
    const int at = seg_off - vb;
    if (seg_cnt > 0 && (unsigned)at < 256u) reinterpret_cast<uint8_t*>(seg4)[at] = (uint8_t)lane;
    __syncthreads();
    const uint32_t w = seg4[lane];
    uint32_t b0 = w & 255u, b1 = (w >> 8) & 255u, b2 = (w >> 16) & 255u, b3 = w >> 24;
    b1 = b0 > b1 ? b0 : b1;
    b2 = b1 > b2 ? b1 : b2;
    b3 = b2 > b3 ? b2 : b3;
    uint32_t m = b3;  // inclusive maximum over the lanes
    auto step = [&](auto ctrl, auto rows) {
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, decltype(ctrl)::value,
                                                                 decltype(rows)::value, 0xf, false);
        m = m > o ? m : o;
    };
    step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x138, 0xf, 0xf, false);  // wave_shr:1
    before = before > last ? before : last;
    b0 = before > b0 ? before : b0;
    b1 = before > b1 ? before : b1;
    b2 = before > b2 ? before : b2;
    b3 = before > b3 ? before : b3;
    seg4[lane] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
    const uint32_t top = (uint32_t)__builtin_amdgcn_readlane((int)m, 63);
    last = top > last ? top : last;
    __syncthreads();
}

// Keeps the candidates of the supercell's list (of `total` <= kPreCap) that lie within the support radius
// of its nt <= 64 targets' bounding box B: their entries go to `list`, in list order, the kept index of each
// target to self_s; returns how many there are. seg4: 64 words for fill_segments. Both pair passes are bound
// by their vector instructions (3.2 to 3.5 cycles each): segments by table instead of a search, medians
// instead of two maxima per axis, uniform work on the scalar unit and candidates consecutive in LDS took a
// density wave from 2,440 to 2,060 of them and a force wave from 3,030 to 2,740; at 2,097,152 particles the
// density pass went from 0.528 to 0.457 ms and the force pass from 0.70 to 0.68 ms.
template <int NS>
__device__ __forceinline__ int prefilter(const NbListT<NS>& L, const WorkBuf& W, const TargetBox& B, int nt,
                                         int total, int self_v0, float H2, uint16_t* list, uint16_t* self_s,
                                         uint32_t* seg4)
{
    const int lane = threadIdx.x;
    // The test cannot drop a candidate the cull accepts, at any coordinate magnitude: per axis the
    // rounded distance to the box is at most the rounded distance to any target in it (rounding is
    // monotone), and both sums of squares round in the same fma order, so the cull's r2 is never
    // below this d2. The 2^-13 margin on H^2 is kept on top of that.
    const float H2m = B.lx <= B.hx ? H2 * (1.0f + 1.0f / 8192.0f) : -1.0f;  // no targets: nothing is kept
    // a target is kept, unless its position is not finite: its distance to the box is not a number then
    self_s[lane] = kNoSelf;
    int count = 0;
    int seg_off = 0, seg_cnt = 0;  // lane's own segment of the 27
    uint32_t last = 0;
    if (NS == 27 && lane < 27) {
        seg_off = L.off[lane];
        seg_cnt = L.off[lane + 1] - seg_off;
    }
    // four candidates per lane and round, all four records requested before any is tested; lanes past the
    // end take the last candidate's place and are cut off from what is kept
    for (int vb = 0; vb < total; vb += 256) {
        if constexpr (NS == 27) fill_segments(seg4, vb, seg_off, seg_cnt, last);
        float4 q[4], t[4];
        int v[4], sg[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int at = vb + 64 * r + lane;
            v[r] = at < total ? at : total - 1;
            sg[r] = NS == 27 ? (int)reinterpret_cast<const uint8_t*>(seg4)[v[r] - vb] : nb_segment(L, v[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = L.t[sg[r]];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (vb + 64 * r < total) q[r] = W.P0[v[r] + __float_as_int(t[r].w)];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int v0 = vb + 64 * r;
            if (v0 >= total) break;
            const float px = q[r].x + t[r].x, py = q[r].y + t[r].y, pz = q[r].z + t[r].z;
            // distance to the box per axis: to the nearest point of it (the median of the coordinate
            // and the two faces), the same rounded value as the difference to the face
            const float dx = px - __builtin_amdgcn_fmed3f(px, B.lx, B.hx);
            const float dy = py - __builtin_amdgcn_fmed3f(py, B.ly, B.hy);
            const float dz = pz - __builtin_amdgcn_fmed3f(pz, B.lz, B.hz);
            const bool near = fmaf(dz, dz, fmaf(dy, dy, dx * dx)) < H2m;  // sentinel records: +inf, dropped
            const uint64_t in = total - v0 >= 64 ? ~0ull : (1ull << (total - v0)) - 1ull;
            const uint64_t b = __ballot(near) & in;
            const int sidx = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)b, (uint32_t)count));
            const bool keep = (b >> lane) & 1ull;
            if (keep) list[sidx] = pre_entry<NS>(v[r], sg[r]);
            if (v0 + 64 > self_v0 && v0 < self_v0 + nt) {  // the targets' own places
                const unsigned ts = (unsigned)(v[r] - self_v0);
                if (keep && ts < (unsigned)nt) self_s[ts] = (uint16_t)sidx;
            }
            count += __popcll(b);
        }
    }
    __syncthreads();
    return count;
}

// Cull lim (<= 32) consecutive lane candidates in the LDS slots from sp on: bit ii set iff r2 < H2, read
// off the sign of |r2| - H2 (exact: the rounded difference has the sign of the exact one; r2 that is not a
// number, a position not being finite, loses the sign that it may have: never a neighbour). Returns
// LSB-first bits. Candidates go four at a time, all four LDS reads issued before any is used, up to
// three slots past lim (the caller's LDS array has them; their bits are cut off).
__device__ __forceinline__ uint32_t cull32(const float4* __restrict__ sp, int lim, float xi, float yi, float zi,
                                           float H2)
{
    uint32_t m = 0;
    int n = 0;
    for (; n < lim; n += 4) {
        const float4 q0 = sp[n], q1 = sp[n + 1], q2 = sp[n + 2], q3 = sp[n + 3];
        __builtin_amdgcn_sched_barrier(0);
        float dx, dy, dz;
        const float r2a = geom_r2(xi, yi, zi, q0, dx, dy, dz);
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(fabsf(r2a) - H2), 31);  // (m << 1) | sign
        const float r2b = geom_r2(xi, yi, zi, q1, dx, dy, dz);
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(fabsf(r2b) - H2), 31);
        const float r2c = geom_r2(xi, yi, zi, q2, dx, dy, dz);
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(fabsf(r2c) - H2), 31);
        const float r2d = geom_r2(xi, yi, zi, q3, dx, dy, dz);
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(fabsf(r2d) - H2), 31);
    }
    const uint32_t bits = __builtin_bitreverse32(m) >> (32 - n);
    return lim == 32 ? bits : bits & ((1u << lim) - 1u);
}

// Staged order of a supercell's candidates in the chunked pair passes. The virtual list (the
// stencil's segments back to back) is cut into blocks of 8 consecutive candidates; the full blocks
// are laid out as 8 rows of consecutive blocks (the first `rem` rows one block longer) and staged
// column by column, the partial last block after them. A chunk of 64 staged slots then holds 8
// blocks from 8 places spread over the whole neighbourhood instead of a few neighbour supercells,
// so the accepted pairs of a chunk spread more evenly over the targets and the chunk's pair loop
// waits less for its busiest lane (a CPU replay of the force pass's lanes at 262,144 particles:
// 41.5 -> 34.0 pair rounds per wave), while the 8 lanes of a block still read 8 consecutive
// records (one candidate per slot, spread that way, made the staging loads uncoalesced and the
// force pass 14% slower). Both passes stage in this order, so the density pass's masks, indexed by
// staged slot, replay unchanged.
struct StageOrder {
    int nfull;  // full blocks of 8
    int cm1;    // blocks per short row - 1 (0 when nfull <= 8: the identity)
    int rem;    // rows of cm1 + 1 blocks

    __device__ __forceinline__ explicit StageOrder(int total)
    {
        nfull = total >> 3;
        const int c = (nfull + 7) >> 3;
        cm1 = c > 0 ? c - 1 : 0;
        rem = nfull - 8 * cm1;
    }
    // list index of staged slot u < total
    __device__ __forceinline__ int list_index(int u) const
    {
        if (u >= 8 * nfull) return u;
        const int b = u >> 3, i = b & 7, j = b >> 3;
        return 8 * (i * cm1 + (i < rem ? i : rem) + j) + (u & 7);
    }
    // staged slot of list index v < total
    __device__ __forceinline__ int slot(int v) const
    {
        if (v >= 8 * nfull) return v;
        const int blk = v >> 3, c = cm1 + 1;
        const bool longrow = blk < rem * c;
        // short rows are only reached when cm1 > 0
        const int num = longrow ? blk : blk - rem * c, den = longrow ? c : cm1;
        const int q = quot(num, den, fast_rcp((float)den));
        const int i = longrow ? q : rem + q;
        const int j = num - q * den;
        return 8 * (8 * j + i) + (v & 7);
    }
};

// Lane layout of a supercell-wave: nt targets, K = floor(64/nt) (capped) lanes per target.
struct LaneMap {
    int K, tpg, tl, k, gfirst, glast;
    float rK;  // 1 / K
    bool inwave;
};

__device__ __forceinline__ LaneMap lane_map(int nt, int kmax)
{
    LaneMap m;
    const int lane = threadIdx.x;
    int K = nt >= 64 ? 1 : uquot(64, nt, fast_rcp((float)nt));
    m.K = K < kmax ? K : kmax;
    m.rK = fast_rcp((float)m.K);
    m.tpg = uquot(64, m.K, m.rK);
    m.tl = (int)(((float)lane + 0.5f) * m.rK);  // lane / K, exact for lane < 64
    m.k = lane - m.tl * m.K;
    m.inwave = m.tl < m.tpg;
    m.gfirst = m.inwave ? m.tl * m.K : 63;
    m.glast = m.inwave ? m.gfirst + m.K - 1 : 63;
    return m;
}

// LDS places of a chunk's slots: lane candidate c of sub-lane k at k * stride + c, so that a lane's
// candidates are consecutive (their addresses are constants off one register in the cull). With few
// sub-lanes the stride is odd, which keeps them off each other's LDS banks. CAP slots hold
// K * stride of them and the three that the cull may read past the last.
struct ChunkMap {
    int per;     // lane candidates per chunk
    int stride;  // >= per

    __device__ __forceinline__ ChunkMap(int cap, const LaneMap& m)
    {
        stride = uquot(cap - 3, m.K, m.rK);
        if (m.K <= 8) stride = (stride - 1) | 1;
        per = stride;
    }
    // place of the slot e = c * K + k of a chunk
    __device__ __forceinline__ int place(int e, const LaneMap& m) const
    {
        const int c = (int)(((float)e + 0.5f) * m.rK);  // e / K, exact for e < 2^20
        return (int)__umul24((unsigned)(e - c * m.K), (unsigned)stride) + c;
    }
};

// Whether a supercell-wave keeps its masks: one target group and every lane's candidates fit.
__device__ __forceinline__ bool masks_fit(int nt, int total, const LaneMap& m, int words = kMaskWords)
{
    return nt <= m.tpg && uquot(total + m.K - 1, m.K, m.rK) <= 32 * words;
}

// The pre-filter's kept list travels from the density pass to the force pass in the top of the
// supercell's mask row (kMaskWords x 64 words): the last word holds the kept count (or kNoList), the
// 16-bit entries lie below it, downwards. With the filter on, masks use at most kMaskWords - 1 words of
// each lane, so the count never shares a word with mask bits, and the list counts as stored only where it
// stays above the words the masks use.
constexpr uint32_t kNoList = 0xffffffffu;
constexpr int kRowWords = kMaskWords * 64;
__device__ __forceinline__ uint16_t* row_entry0(uint32_t* row)
{
    return reinterpret_cast<uint16_t*>(row + kRowWords - 1) - 1;  // entry e at [-e]
}
// entries 2 d and 2 d + 1 of a row, the first in the low half
__device__ __forceinline__ uint32_t row_entries(const uint32_t* row, int d)
{
    const uint32_t w = row[kRowWords - 2 - d];
    return (w << 16) | (w >> 16);
}

__device__ __forceinline__ bool list_fits(int count, int K, float rK)
{
    const int mask_words = (uquot(count + K - 1, K, rK) + 31) / 32;
    return (count + 1) / 2 <= kRowWords - 1 - 64 * mask_words;
}

// Mask words are indexed by lane candidate c (candidate v = c*K + k of sub-lane k), so the two
// passes may stage with different chunk sizes. Bits for [c0, c0 + lim) may straddle two words.
// Words at or past `wlim` (those of candidates past the lane's last one: the last chunk's padding,
// all-zero bits) are not written, so the row above the lane's masks stays free.
struct MaskWriter {
    uint32_t* row = nullptr;
    uint32_t pend = 0;
    int pend_w = -1;
    int wlim = kMaskWords;  // <= kMaskWords
    __device__ __forceinline__ void put(uint32_t bits, int c0, int lim)
    {
        const int w = c0 >> 5, off = c0 & 31;
        if (w >= wlim) return;
        if (w != pend_w) {
            if (pend_w >= 0) row[pend_w * 64] = pend;
            pend = 0;
            pend_w = w;
        }
        pend |= bits << off;
        if (off + lim > 32) {
            row[w * 64] = pend;
            pend = bits >> (32 - off);
            pend_w = w + 1 < wlim ? w + 1 : -1;
        }
    }
    __device__ __forceinline__ void flush()
    {
        if (pend_w >= 0) row[pend_w * 64] = pend;
        pend_w = -1;
    }
};

__device__ __forceinline__ uint32_t mask_get(const uint32_t* row, int c0, int lim, int per_lane)
{
    int nvalid = per_lane - c0;
    if (nvalid <= 0) return 0u;
    if (nvalid > lim) nvalid = lim;
    const int w = c0 >> 5, off = c0 & 31;
    if (w >= kMaskWords) return 0u;
    uint32_t a = row[w * 64] >> off;
    if (off && off + nvalid > 32 && w + 1 < kMaskWords) a |= row[(w + 1) * 64] << (32 - off);
    return nvalid == 32 ? a : (a & ((1u << nvalid) - 1u));
}

// Compact the accepted LDS slots (first + bit) of each target's K lanes into lst[gfirst*32 ...) (in
// sub-lane, then candidate order) and return the target's count; the K lanes then share them round-robin.
template <class LT>
__device__ __forceinline__ int compact_group(uint32_t msk, int first, const LaneMap& m, LT* lst)
{
    const int na = __popc(msk);
    const int incl = dpp_incl_scan(na);
    const int bprev = __shfl(incl, m.gfirst > 0 ? m.gfirst - 1 : 0, 64);
    const int before = m.gfirst > 0 ? bprev : 0;
    const int gtot = __shfl(incl, m.glast, 64) - before;
    int wpos = m.gfirst * 32 + (incl - na - before);
    while (msk) {
        const int ii = __builtin_ctz(msk);
        msk &= msk - 1;
        lst[wpos++] = (LT)(first + ii);
    }
    return m.inwave ? gtot : 0;
}

// Gradient factor of the smoothing kernel (kslope), the h powers and sigma included.
__device__ __forceinline__ float grad_factor(int kern, float sig, float h)
{
#pragma clang fp contract(off)
    return (kern == 2) ? -5.0f * sig / (h * h * h * h * h) : sig / (h * h * h * h);
}

// x of the lane below (DPP wave_shr:1; lane 0 gets zero). K - 1 steps of x = lane_below(x) + v, from x = v,
// leave the sum of K consecutive lanes' v, added in lane order, in the last of them.
__device__ __forceinline__ uint32_t lane_below(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x138, 0xf, 0xf, true);
}
__device__ __forceinline__ float lane_below(float x)
{
    return __uint_as_float(lane_below(__float_as_uint(x)));
}

// K partial sums of a target combined in lane order (deterministic); then one lane per particle
// writes rho, the neighbour count and the interaction records of the force pass, and the run's
// fast-speed maximum (cleaning speed) is raised.
template <bool MHD>
__device__ __forceinline__ void density_finish(RunC& R, int r, const StateBuf& S, const WorkBuf& W, const LaneMap& lm,
                                               float acc, uint32_t cnt, bool valid, bool tgt, uint8_t spc,
                                               uint8_t live, const Slot& s, float m_own, float h, float uu,
                                               float vx, float vy, float vz, float rho_in, float bx, float by,
                                               float bz, float psi, float gam, int kern)
{
    const int K = lm.K, k = lm.k;
    const int lane = threadIdx.x;
    float acc_t = acc;
    uint32_t cnt_t = cnt;
    for (int kk = 1; kk < K; ++kk) {
        acc_t = lane_below(acc_t) + acc;
        cnt_t = lane_below(cnt_t) + cnt;
    }
    const bool writer = k == K - 1;
    // epilogue: one lane per particle writes rho and its interaction records
    float cmax = 0.0f;
    if (writer && valid && is_source(spc, live)) {
#pragma clang fp contract(off)
        const float sig = R.sigma;
        // the divisions by powers of h are the run's own constants where the wave's particles have its h
        float invh = R.inv_h0, wfac = R.wfac0, gfac = R.gfac0;
        if (__ballot(h != R.h0) != 0) {
            invh = 1.0f / h;
            wfac = sig / (h * h * h);
            gfac = grad_factor(kern, sig, h);
        }
        float rho;
        if (tgt) {
            rho = wfac * (acc_t + m_own * kshape0(kern));
            s.col(S.rho) = rho;
            s.col(W.nnb) = cnt_t;
        } else {
            rho = rho_in;
        }
        if (MHD || W.P1 != nullptr) {  // null: no force pass follows
            const float P = (gam - 1.0f) * rho * uu;
            const float invrho = 1.0f / rho;
            const float B2 = bx * bx + by * by + bz * bz;
            const float bdr = invrho * invrho;
            const float ph = P * bdr;
            const float pr = (P + 0.5f * B2) * bdr;
            const float psr = psi * bdr;
            const float c = sqrtf((gam * P + B2) * invrho);
            s.rec(W.P1) = make_float4(vx, vy, vz, c);
            s.rec(W.P2) = make_float4(h, invh, gfac, ph);
            s.rec(W.P3) = make_float4(pr, 0.5f * rho, bdr, psr);
            if (MHD) s.rec(W.P4) = make_float4(bx, by, bz, psi);
            if (tgt) cmax = c;
        }
    }
    if (writer && valid && !tgt) s.col(W.nnb) = 0;
    if (MHD && run_mhd(R.flags) && run_cleaning(R.flags)) {
        const uint32_t bits = dpp_max_u32(__float_as_uint(cmax));
        // every wave of the run targets this one word: test before the atomic, so that only a
        // wave holding a new maximum pays for one (the value only grows, so a stale read costs
        // at most a redundant atomic)
        if (lane == 0 && bits != 0u) {
            if (bits > __atomic_load_n(&W.chbits[r], __ATOMIC_RELAXED)) atomicMax(&W.chbits[r], bits);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// density pass: cull of the 27-supercell candidates staged in LDS, density sum, candidate masks,
// and the per-particle interaction records of the force pass
// ------------------------------------------------------------------------------------------------
// LDS of a density wave (27-cell stencil, 256 slots: 4,768 bytes, so that 32 waves fit a compute unit). sp
// holds the staged candidates, its top the pre-filter's kept list while there is one (160 slots are left for
// a chunk then), and its first slots the segment table while the pre-filter runs. Staging the kept candidates
// straight from the filter, without their list, needs room for all of them (236 on average in a turbulent
// state, 330 at the 95th percentile) and cost more in occupancy than the second pass over their records:
// 0.476 / 0.504 ms with 320 / 384 slots at 7 / 6 waves per SIMD against 0.450 ms at 2,097,152 particles.
template <int CH, int RMAX>
struct DensityLds {
    NbListR<RMAX> L;
    float4 sp[CH];
    uint16_t self_s[64];
};
constexpr int kListSlots = kPreCap * 2 / 16;  // slots that the kept list takes

template <int CH, bool MIXED, bool MHD, int KT, int RMAX>
__device__ __forceinline__ void density_wave(int vb, DensityLds<CH, RMAX>& lds)
{
    const PairArgs& args = pair_args();
    const StateBuf& S = args.S;
    const WorkBuf& W = args.W;
    const RunDev* const runs = args.runs;
    constexpr int NS = RMAX == 1 ? 27 : 125;
    static_assert(CH - kListSlots >= 67, "a chunk beside the kept list needs a slot per lane and the cull's three");
    NbListR<RMAX>& L = lds.L;
    float4(&sp)[CH] = lds.sp;
    const int cell = xcd_cell(vb, args.nblk_total, args.ncell_tot);
    if (cell < 0) return;
    const int t0 = uniform((int)W.cs[cell]);
    const int nt = uniform((int)W.cs[cell + 1]) - t0;
    if (nt == 0) return;
    const int r = find_run_by_cell(runs, args.nruns, cell);
    RunC& R = ((RunC*)runs)[r];
    // the targets' box inputs are requested before the neighbour list, so their loads overlap the list's
    const TargetBoxInput box_in = nt <= 64 ? target_box_load(S, W, t0, nt) : TargetBoxInput{};
    int self_v0;
    const int all = Stencil<MIXED, RMAX>(R, cell - R.c0, W.cs).build(R, L, self_v0);
    const int lane = threadIdx.x;
    const LaneMap lm = lane_map(nt, args.kmax);
    const int K = lm.K, k = lm.k;
    uint32_t* const row = W.nbmask != nullptr ? W.nbmask + (size_t)cell * kRowWords : nullptr;
    // supercells of more than 64 particles or a longer list are not filtered
    const bool pre = nt <= 64 && all <= kPreCap;
    uint16_t* const list = reinterpret_cast<uint16_t*>(sp + CH - kListSlots);
    const ChunkMap cm(pre ? CH - kListSlots : CH, lm);
    int total = all;  // staged candidates
    if (pre)
        total = prefilter<NS>(L, W, target_box(box_in, nt), nt, all, self_v0, R.H2, list, lds.self_s,
                              reinterpret_cast<uint32_t*>(sp));
    const StageOrder so(total);
    const int chk = cm.per * K;  // staged entries per chunk (a multiple of K)
    const int kern = KT >= 0 ? KT : run_kernel(R.flags);  // compile-time when every run uses one kernel
    const float H2 = R.H2;
    const float gam = R.gamma;
    // no mask table: density only; with the filter on the top word of each lane carries the kept list
    const bool keep = masks_fit(nt, total, lm, pre ? kMaskWords - 1 : kMaskWords) && row != nullptr;
    MaskWriter mw;
    mw.row = row + lane;
    mw.pend = 0;
    mw.pend_w = -1;
    mw.wlim = (uquot(total + K - 1, K, lm.rK) + 31) / 32;  // the words the lane's candidates need

    for (int tg = 0; tg < nt; tg += lm.tpg) {
        const int tt = tg + lm.tl;
        const bool valid = lm.inwave && tt < nt;
        // t0 made opaque in the loop (one round for most cells): otherwise the bases of all the columns
        // are formed ahead of it and no scalar registers are left
        int t0l = t0;
        asm volatile("" : "+s"(t0l));
        const Slot s(t0l, valid ? (uint32_t)tt : 0u);
        const uint8_t live = s.col(S.mask), spc = s.col(S.species);
        const bool tgt = valid && is_target(spc, live);
        const float4 own = s.rec(W.P0);
        const float h = s.col(S.h);
        // inputs of the epilogue, loaded early so their latency overlaps the cull
        const float uu = s.col(S.u);
        const float vx = s.col(S.vel[0]), vy = s.col(S.vel[1]),
                    vz = s.col(S.vel[2]);
        const float rho_in = s.col(S.rho);
        float bx = 0.f, by = 0.f, bz = 0.f, psi = 0.f;
        if (MHD && run_mhd(R.flags)) {
            bx = s.col(S.B[0]);
            by = s.col(S.B[1]);
            bz = s.col(S.B[2]);
            psi = s.col(S.psi);
        }
        float invh = R.inv_h0;
        if (__ballot(h != R.h0) != 0) invh = 1.0f / h;
        // the lane candidate that is the self pair: its staged slot is this lane's or no lane candidate
        int self_c = -1;
        if (tgt) {
            const int self_u = so.slot(pre ? (int)lds.self_s[tt] : self_v0 + tt);
            const int c = quot(self_u, K, lm.rK);
            self_c = self_u - c * K == k ? c : -1;
        }
        float acc = 0.0f;
        uint32_t cnt = 0;
        const float4* const mine = sp + __umul24((unsigned)k, (unsigned)cm.stride);  // this lane's slots

        for (int base = 0, cbase = 0; base < total; base += chk, cbase += cm.per) {
            // lane slots of this chunk that hold candidates (the most any lane has): the last chunk's
            // padding is not culled
            const int left = total - base < chk ? total - base : chk;
            const int nval = uquot(left + K - 1, K, lm.rK);
            for (int e = lane; e < nval * K; e += 64) {
                const int u = base + e;
                float4 p = make_float4(kSentinel, kSentinel, kSentinel, 0.0f);
                if (u < total) {
                    float4 t4;
                    const int li = so.list_index(u);
                    const int j = pre ? kept_candidate(L, list[li], t4) : list_candidate(L, li, t4);
                    p = W.P0[j];
                    p.x += t4.x;
                    p.y += t4.y;
                    p.z += t4.z;
                }
                sp[cm.place(e, lm)] = p;
            }
            __syncthreads();
            for (int sb = 0; sb < nval; sb += 32) {
                const int lim = nval - sb < 32 ? nval - sb : 32;
                uint32_t msk = cull32(mine + sb, lim, own.x, own.y, own.z, H2);
                // the self pair (r2 = 0) passes the cull: drop it here; its density term is the
                // self term m_i W(0, h_i) added below, as DensityInitSelf does
                const unsigned bit = (unsigned)(self_c - cbase - sb);
                if (bit < (unsigned)lim) msk &= ~(1u << bit);
                if (!tgt) msk = 0;
                if (keep) mw.put(msk, cbase + sb, lim);
                cnt += (uint32_t)__popc(msk);
                // each lane sums its own accepted candidates (the density pairs are too cheap for
                // sharing them among a target's lanes to pay for the compaction)
                while (msk) {
                    const int ii = __builtin_ctz(msk);
                    msk &= msk - 1;
                    const float4 p = lds_at(mine + sb, ii * (int)sizeof(float4));
                    float dx, dy, dz;
                    const float r2 = geom_r2(own.x, own.y, own.z, p, dx, dy, dz);
                    acc += p.w * kshape(kern, fast_sqrt(r2) * invh);
                }
            }
            __syncthreads();
        }
        if (keep) mw.flush();
        density_finish<MHD>(R, r, S, W, lm, acc, cnt, valid, tgt, spc, live, s, own.w, h, uu, vx, vy, vz, rho_in,
                            bx, by, bz, psi, gam, kern);
    }
    // the kept list for the force pass, stored last: stores count in the same wait counter as the
    // loads, so stored earlier they would delay every later wait for the staging loads
    if (pre && row != nullptr) {
        const bool store = keep && list_fits(total, K, lm.rK);
        if (store)
            for (int e = lane; e < total; e += 64) *(row_entry0(row) - e) = list[e];
        if (lane == 0) row[kRowWords - 1] = store ? (uint32_t)total : kNoList;
    }
}

template <int CH, bool MIXED, bool MHD, int KT, int RMAX = 1, bool GRID = false>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(KT == 2 && RMAX == 1 ? 8 : 1, 8)))  // KT 2: Wendland
void k_density(PairArgs)
{
    __shared__ DensityLds<CH, RMAX> lds;
    if constexpr (GRID) {
        // a persistent grid: each wave walks the supercells at a stride of the grid (a multiple
        // of 8, so every cell a wave visits belongs to its own XCD's range)
        for (int vb = blockIdx.x; vb < pair_args().nblk_total; vb += gridDim.x)
            density_wave<CH, MIXED, MHD, KT, RMAX>(vb, lds);
    } else {
        // one supercell per wave
        density_wave<CH, MIXED, MHD, KT, RMAX>((int)blockIdx.x, lds);
    }
}

// ------------------------------------------------------------------------------------------------
// force pass: pressure gradient, P dV, Monaghan viscosity, SPMHD stress, induction, cleaning
// ------------------------------------------------------------------------------------------------
struct ForceAcc {
    float ax, ay, az, DV, AVU, vmax;
    float Ti, Tj, TBx, TBy, TBz, VBx, VBy, VBz, DB, PSx, PSy, PSz;
};

// Per-run constants of the pair loop. alpha <= 0 switches the viscosity off with both coefficients 0, so
// the loop has no branch for it (the term is then an exact zero).
struct PairConst {
    int kern;
    float beta;               // of the signal speed
    float va, vb;             // alpha / 2 and beta of the viscosity
    float h, invh, gfac, e;   // ONE_H: the run's one smoothing length, 1/h, gradient factor and 0.01 h^2

    __device__ __forceinline__ PairConst(RunC& R, int kern_, float h_)
        : kern(kern_), beta(R.beta), va(R.alpha > 0.0f ? 0.5f * R.alpha : 0.0f), vb(R.alpha > 0.0f ? R.beta : 0.0f),
          h(h_), invh(R.inv_h0), gfac(R.gfac0), e((0.01f * h_) * h_)
    {
        if (uniform(__float_as_int(h_)) != __float_as_int(R.h0)) {
            invh = 1.0f / h_;
            gfac = grad_factor(kern_, R.sigma, h_);
        }
    }
};

// The pair terms of target o and neighbour q, added to A. Records: 0 (x, y, z, m), 1 (v, c),
// 2 (h, 1/h, gfac, ph), 3 (pr, rho / 2, bdr, psr), 4 (B, psi).
// ONE_H: every particle of the run has the same smoothing length, so record 2 of the neighbour is not
// read; the same bits as the general form. The pass is bound by VALU issue, so the pair is a straight
// run of 72 instructions (three transcendental; 77 with the loop's own) with no branch or select in it: the support test is the
// clamp of kslope, the r > 0 guard a lower bound on r2 (every normal r2 is itself; coincident particles have
// r = 0, a finite 1/r and exact zeros in every term), runs without viscosity or cleaning take zeros through
// the same code, and the exact halves and doublings of the viscosity are folded away (rho / 2 in the record:
// 1 / (rho_i/2 + rho_j/2) is the mean density's reciprocal). Every product and fused multiply-add is
// written out, contraction off, so all instantiations round alike. Against the branched form with five
// staged records (85 instructions) the force pass took 0.75 -> 0.69 ms at 2,097,152 particles.
template <bool MHD, bool ONE_H>
__device__ __forceinline__ void force_pair(const float4& o0, const float4& o1, const float4& o2, const float4& o3,
                                           const float4& o4, const float4& q0, const float4& q1, const float4& q2,
                                           const float4& q3, const float4& q4, const PairConst& C, ForceAcc& A)
{
#pragma clang fp contract(off)
    float dx, dy, dz;
    const float r2 = geom_r2(o0.x, o0.y, o0.z, q0, dx, dy, dz);
    const float invR = fast_rsq(fmaxf(r2, 0x1p-126f));  // the least normal number: v_rsq_f32 gives inf below it
    const float rr = r2 * invR;
    const float ms_i = q0.w * kslope(C.kern, invR, rr * (ONE_H ? C.invh : o2.y), ONE_H ? C.gfac : o2.z);
    float ms_j = ms_i;
    // equal smoothing lengths give the same gradient bit for bit: the second evaluation is skipped then
    if (!ONE_H && __builtin_expect(q2.x != o2.x, 0)) ms_j = q0.w * kslope(C.kern, invR, rr * q2.y, q2.z);
    const float dvx = o1.x - q1.x, dvy = o1.y - q1.y, dvz = o1.z - q1.z;
    const float vr = fmaf(dvz, dz, fmaf(dvx, dx, dvy * dy));
    const float fiso = fmaf(o3.x, ms_i, q3.x * ms_j);
    A.ax = fmaf(-fiso, dx, A.ax);
    A.ay = fmaf(-fiso, dy, A.ay);
    A.az = fmaf(-fiso, dz, A.az);
    A.DV = fmaf(ms_i, vr, A.DV);
    const float vrm = fminf(vr, 0.0f);  // receding pairs: no viscosity
    const float cs = o1.w + q1.w;
    const float vs = fmaf(-C.beta, vrm * invR, cs);
    // signal speeds are >= +0, so their float bits order as integers: an integer max is the float
    // max without the NaN-quieting copy fmaxf needs for its loop-carried operand
    A.vmax = __int_as_float(max(__float_as_int(A.vmax), __float_as_int(vs)));
    // Pi = (beta mu - alpha cb) mu / rb, cb and rb the pair's mean sound speed and density, and
    // gv = Pi (m s_i + m s_j) / 2
    const float hb = ONE_H ? C.h : 0.5f * (o2.x + q2.x);
    const float mu = (hb * vrm) * fast_rcp(r2 + (ONE_H ? C.e : (0.01f * hb) * hb));
    const float Pi = (mu * fmaf(C.vb, mu, -(C.va * cs))) * fast_rcp(o3.y + q3.y);
    const float gv = (ONE_H ? ms_i : 0.5f * (ms_i + ms_j)) * Pi;
    A.ax = fmaf(-gv, dx, A.ax);
    A.ay = fmaf(-gv, dy, A.ay);
    A.az = fmaf(-gv, dz, A.az);
    A.AVU = fmaf(gv, vr, A.AVU);
    if constexpr (MHD) {
        const float fps = fmaf(o3.w, ms_i, q3.w * ms_j);
        A.PSx = fmaf(fps, dx, A.PSx);
        A.PSy = fmaf(fps, dy, A.PSy);
        A.PSz = fmaf(fps, dz, A.PSz);
        const float Bir = fmaf(o4.z, dz, fmaf(o4.x, dx, o4.y * dy));
        const float Bjr = fmaf(q4.z, dz, fmaf(q4.x, dx, q4.y * dy));
        const float bj = Bjr * q3.z;
        const float tj = bj * ms_j;
        A.TBx = fmaf(tj, q4.x, A.TBx);
        A.TBy = fmaf(tj, q4.y, A.TBy);
        A.TBz = fmaf(tj, q4.z, A.TBz);
        A.Ti = fmaf(Bir * o3.z, ms_i, A.Ti);
        A.Tj = fmaf(bj, ms_j, A.Tj);
        const float wv = ms_i * Bir;
        A.VBx = fmaf(wv, dvx, A.VBx);
        A.VBy = fmaf(wv, dvy, A.VBy);
        A.VBz = fmaf(wv, dvz, A.VBz);
        A.DB = fmaf(ms_i, Bir - Bjr, A.DB);
    }
}

// One target's derivatives, signal speed and div B from its summed pair terms T.
template <bool MHD>
__device__ __forceinline__ void force_write(RunC& R, const WorkBuf& W, const ForceAcc& T, const Slot& s,
                                            const float4& o1, const float4& o2, const float4& o3, const float4& o4, bool mhd,
                                            bool clean, float borve, float ch)
{
    const float rho = 2.0f * o3.y;
    const float invrho = 1.0f / rho;
    float ax = T.ax, ay = T.ay, az = T.az;
    if (MHD && mhd) {
        const float tcoef = T.Ti - borve * (T.Ti + T.Tj);
        ax = ax + T.TBx + o4.x * tcoef;
        ay = ay + T.TBy + o4.y * tcoef;
        az = az + T.TBz + o4.z * tcoef;
    }
    s.col(W.dvdt[0]) = ax;
    s.col(W.dvdt[1]) = ay;
    s.col(W.dvdt[2]) = az;
    s.col(W.dudt) = o2.w * T.DV + 0.5f * T.AVU;
    s.col(W.vsig) = fmaxf(2.0f * o1.w, T.vmax);
    if (MHD && mhd) {
        const float divB = -T.DB * invrho;
        const float divv = -T.DV * invrho;
        float dbx = -(T.VBx - o4.x * T.DV) * invrho;
        float dby = -(T.VBy - o4.y * T.DV) * invrho;
        float dbz = -(T.VBz - o4.z * T.DV) * invrho;
        float dpsi = 0.0f;
        if (clean) {
            dbx -= rho * T.PSx;
            dby -= rho * T.PSy;
            dbz -= rho * T.PSz;
            const float psi = o4.w;
            dpsi = -ch * ch * divB - psi * R.clean_sigma * ch * o2.y - 0.5f * psi * divv;
        }
        s.col(W.dbdt[0]) = dbx;
        s.col(W.dbdt[1]) = dby;
        s.col(W.dbdt[2]) = dbz;
        s.col(W.dpsidt) = dpsi;
        s.col(W.divb) = divB;
    }
}

// x from the lane D below in the same 16-lane row (DPP row_shr:D; lanes at the row's start read 0)
template <int D>
__device__ __forceinline__ float row_shr(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x110 + D, 0xf, 0xf, true));
}

// K partial force sums of a target combined (deterministic), field by field; then one lane per
// target writes its derivatives, signal speed and div B. For K = 2, 4, 8 or 16 a target's lanes lie
// in one 16-lane row, and log2 K DPP steps (each lane adds the partial of the lane 1, 2, 4, ... below
// it) leave the target's total in its last lane; other K take K - 1 wave shifts by one lane, which add
// the partials in lane order and leave the total there too.
template <bool MHD>
__device__ __forceinline__ void force_finish(RunC& R, const WorkBuf& W, const LaneMap& lm, ForceAcc& A, bool tgt,
                                             const Slot& s, const float4& o1, const float4& o2, const float4& o3,
                                             const float4& o4, bool mhd, bool clean, float borve, float ch)
{
    const int K = lm.K, k = lm.k;
    constexpr int NF = MHD ? 17 : 5;
    float v[NF] = {A.ax, A.ay, A.az, A.DV, A.AVU};
    if constexpr (MHD) {
        const float m[12] = {A.Ti, A.Tj, A.TBx, A.TBy, A.TBz, A.VBx, A.VBy, A.VBz, A.DB, A.PSx, A.PSy, A.PSz};
#pragma unroll
        for (int f = 0; f < 12; ++f) v[5 + f] = m[f];
    }
    float sum[NF];
    float vm;
    if (K == 1 || K == 2 || K == 4 || K == 8 || K == 16) {
        auto step = [&](auto d) {
            constexpr int D = decltype(d)::value;
#pragma unroll
            for (int f = 0; f < NF; ++f) v[f] += row_shr<D>(v[f]);
            // signal speeds are >= +0: an integer max on their bits
            A.vmax = __int_as_float(max(__float_as_int(A.vmax), __float_as_int(row_shr<D>(A.vmax))));
        };
        if (K >= 2) step(std::integral_constant<int, 1>{});
        if (K >= 4) step(std::integral_constant<int, 2>{});
        if (K >= 8) step(std::integral_constant<int, 4>{});
        if (K >= 16) step(std::integral_constant<int, 8>{});
#pragma unroll
        for (int f = 0; f < NF; ++f) sum[f] = v[f];
        vm = A.vmax;
    } else {
        // one step of the sum for all fields, K - 1 times: 17 instructions each. Shuffled through the LDS to
        // every lane of the target it was 18 LDS reads each, and the force pass of a 152,320-particle Sod tube
        // took 61.5 us instead of 50.5 (2,097,152 particles: 0.673 ms instead of 0.660)
#pragma unroll
        for (int f = 0; f < NF; ++f) sum[f] = v[f];
        vm = A.vmax;
        for (int kk = 1; kk < K; ++kk) {
#pragma unroll
            for (int f = 0; f < NF; ++f) sum[f] = lane_below(sum[f]) + v[f];
            vm = fmaxf(lane_below(vm), A.vmax);
        }
    }
    const bool writer = k == K - 1;
    ForceAcc& T = A;
    T.ax = sum[0];
    T.ay = sum[1];
    T.az = sum[2];
    T.DV = sum[3];
    T.AVU = sum[4];
    T.vmax = vm;
    if constexpr (MHD) {
        T.Ti = sum[5];
        T.Tj = sum[6];
        T.TBx = sum[7];
        T.TBy = sum[8];
        T.TBz = sum[9];
        T.VBx = sum[10];
        T.VBy = sum[11];
        T.VBz = sum[12];
        T.DB = sum[13];
        T.PSx = sum[14];
        T.PSy = sum[15];
        T.PSz = sum[16];
    }
    if (writer && tgt) force_write<MHD>(R, W, T, s, o1, o2, o3, o4, mhd, clean, borve, ch);
}

// Records staged per neighbour: P0, P1, P3, P4 with MHD fields, and P2 unless the run has one smoothing
// length (64 instead of 80 bytes per neighbour).
template <bool MHD, bool ONE_H>
constexpr int kForcePlanes = 3 + (MHD ? 1 : 0) + (ONE_H ? 0 : 1);

// LDS slots of a force chunk in each of NP planes: CH and some more for the odd-stride rounding of ChunkMap and
// for the cull's three. With five planes only four more, and the cull reads on into the second plane: the LDS
// then stays within 7,680 bytes (64 slots, MHD, unequal h), 21 waves per compute unit, for which the compiler
// keeps to 96 registers, 5 waves per SIMD. With eight more and the filter's segment table beside them (it lies in
// the slots while the filter runs) it was 8,224 bytes and 98 registers, 4 waves: the cubic force pass of 262,144
// particles took 102.5 us instead of 98.2, the quintic 112.3 instead of 107.9, the Wendland 96.0 instead of 93.3.
template <int CH, int NP>
constexpr int kForceSlots = CH + (NP == 5 ? 4 : 8);
template <int CH, int NP>
constexpr int kForceCap = kForceSlots<CH, NP> + (NP == 5 ? 3 : 0);  // ChunkMap's CAP

template <int CH, bool MIXED, bool MHD, int KT, int BAL, int RMAX, bool ONE_H = false,
          int NP = kForcePlanes<MHD, ONE_H>>
__device__ __forceinline__ void forces_wave(int vb, NbListR<RMAX>& L,
                                            float4 (&sp)[NP][kForceSlots<CH, NP>],
                                            ListT<CH> (&lst)[BAL == 1 ? 64 * 32 : 1], PreList& P)
{
    const PairArgs& args = pair_args();
    const StateBuf& S = args.S;
    const WorkBuf& W = args.W;
    const RunDev* const runs = args.runs;
    constexpr int NS = RMAX == 1 ? 27 : 125;
    const int cell = xcd_cell(vb, args.nblk_total, args.ncell_tot);
    if (cell < 0) return;
    // the supercell's range, the density pass's kept set (stored in its mask row: its count, its first 256
    // entries and the lane's first 64 mask bits) and the stencil's ranges are all requested before any is
    // waited for (the kept set is used only if this step's filter and masks apply to the supercell). Where most
    // supercells are empty the rows wait until the supercell is known not to be: reading them for nothing cost
    // 5% with 200,000 particles in 4.2 M supercells
    const int lane = threadIdx.x;
    const uint32_t first_p = load_early(W.cs + cell), end_p = load_early(W.cs + cell + 1);
    const uint32_t* row = W.nbmask + (size_t)cell * kRowWords;
    const uint32_t* const mrow = row + lane;
    uint32_t row_last = 0, head0 = 0, head1 = 0, mw0 = 0, mw1 = 0;
    auto load_row = [&]() {
        row_last = load_early(row + kRowWords - 1);
        head0 = load_early(row + kRowWords - 2 - lane);
        head1 = load_early(row + kRowWords - 66 - lane);
        mw0 = load_early(mrow);
        mw1 = load_early(mrow + 64);
    };
    if (args.dense) load_row();
    const int r = find_run_by_cell(runs, args.nruns, cell);
    RunC& R = ((RunC*)runs)[r];
    const Stencil<MIXED, RMAX> stencil(R, cell - R.c0, W.cs);
    const int t0 = uniform((int)first_p);
    const int nt = uniform((int)end_p) - t0;
    if (nt == 0) return;
    if (!args.dense) load_row();
    const uint32_t n_row = nt <= 64 ? row_last : kNoList;
    const uint64_t m01 = ((uint64_t)mw1 << 32) | mw0;
    int self_v0;
    const int all = stencil.build(R, L, self_v0);
    const LaneMap lm = lane_map(nt, args.kmax);
    const int K = lm.K, k = lm.k;
    // read back where the density pass stored it, else recomputed
    const bool pre = nt <= 64 && all <= kPreCap;
    int total = all;
    const int n_kept = uniform((int)n_row);
    if (pre && (uint32_t)n_kept != kNoList) {
        if (2 * lane < n_kept) P.v2[lane] = (head0 << 16) | (head0 >> 16);
        if (2 * (lane + 64) < n_kept) P.v2[lane + 64] = (head1 << 16) | (head1 >> 16);
        for (int d = lane + 128; 2 * d < n_kept; d += 64) P.v2[d] = row_entries(row, d);
        __syncthreads();
        total = n_kept;
    } else if (pre) {
        total = prefilter<NS>(L, W, target_box(target_box_load(S, W, t0, nt), nt), nt, all, self_v0, R.H2, P.v,
                              P.self_s, reinterpret_cast<uint32_t*>(sp[0]));
    }
    const StageOrder so(total);  // the density pass's staged order: its masks replay slot by slot
    const ChunkMap cm(kForceCap<CH, NP>, lm);
    const int per_lane = uquot(total + K - 1, K, lm.rK);
    const int kern = KT >= 0 ? KT : run_kernel(R.flags);  // compile-time when every run uses one kernel
    const float H2 = R.H2;
    const float h_own = S.h[t0];  // the run's one smoothing length (ONE_H)
    const PairConst pc(R, kern, h_own);
    const bool mhd = MHD && run_mhd(R.flags);
    const bool clean = mhd && run_cleaning(R.flags);
    const float borve = mhd ? R.borve : 0.0f;
    const float ch = __uint_as_float(W.chbits[r]);
    const bool keep = masks_fit(nt, total, lm, pre ? kMaskWords - 1 : kMaskWords);
    // as few chunks as the slots allow, of about equal size: a chunk's pair loop waits for its busiest lane,
    // so a short last chunk would waste rounds
    const int nch = uquot(per_lane + cm.per - 1, cm.per, fast_rcp((float)cm.per));
    const int per = uquot(per_lane + nch - 1, nch, fast_rcp((float)nch));
    const int chk = per * K;

    for (int tg = 0; tg < nt; tg += lm.tpg) {
        const int tt = tg + lm.tl;
        const bool valid = lm.inwave && tt < nt;
        // t0 made opaque in the loop (one round for most cells): otherwise the bases of all the columns
        // are formed ahead of it and no scalar registers are left
        int t0l = t0;
        asm volatile("" : "+s"(t0l));
        const Slot s(t0l, valid ? (uint32_t)tt : 0u);
        const bool tgt = valid && is_target(s.col(S.species), s.col(S.mask));
        const float4 o0 = s.rec(W.P0), o1 = s.rec(W.P1), o3 = s.rec(W.P3);
        float4 o2 = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (!ONE_H) o2 = s.rec(W.P2);
        float4 o4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (MHD) o4 = s.rec(W.P4);
        // the lane candidate that is the self pair is needed only where the pass culls (a stored list
        // implies stored masks)
        int self_c = -1;
        if (tgt && !keep) {
            const int self_u = so.slot(pre ? (int)P.self_s[tt] : self_v0 + tt);
            const int c = quot(self_u, K, lm.rK);
            self_c = self_u - c * K == k ? c : -1;
        }
        ForceAcc A = {};
        const int first = (int)__umul24((unsigned)k, (unsigned)cm.stride);  // this lane's slots

        for (int base = 0, cbase = 0; base < total; base += chk, cbase += per) {
            const int left = total - base < chk ? total - base : chk;
            const int nval = uquot(left + K - 1, K, lm.rK);
            for (int e = lane; e < nval * K; e += 64) {
                const int u = base + e, at = cm.place(e, lm);
                if (u < total) {
                    float4 t4;
                    const int li = so.list_index(u);
                    const int j = pre ? kept_candidate(L, P.v[li], t4) : list_candidate(L, li, t4);
                    float4 p = W.P0[j];
                    p.x += t4.x;
                    p.y += t4.y;
                    p.z += t4.z;
                    sp[0][at] = p;
                    sp[1][at] = W.P1[j];
                    sp[2][at] = W.P3[j];
                    if constexpr (MHD) sp[3][at] = W.P4[j];
                    if constexpr (!ONE_H) sp[MHD ? 4 : 3][at] = W.P2[j];
                } else {
                    sp[0][at] = make_float4(kSentinel, kSentinel, kSentinel, 0.0f);
                }
            }
            __syncthreads();
            for (int sb = 0; sb < nval; sb += 32) {
                const int lim = nval - sb < 32 ? nval - sb : 32;
                const int c0 = cbase + sb;
                uint32_t msk;
                if (keep) {
                    if (c0 + lim <= 64) msk = (uint32_t)(m01 >> c0) & (0xffffffffu >> (32 - lim));
                    else msk = mask_get(mrow, c0, lim, per_lane);
                } else {
                    msk = cull32(sp[0] + first + sb, lim, o0.x, o0.y, o0.z, H2);
                    const unsigned bit = (unsigned)(self_c - c0);  // the self pair adds exact zeros; drop it anyway
                    if (bit < (unsigned)lim) msk &= ~(1u << bit);
                }
                if (!tgt) msk = 0;
                const int eb0 = (int)sizeof(float4) * (first + sb);  // byte offset of bit 0's slot
                if (BAL == 0) {
                    while (msk) {
                        const int ii = __builtin_ctz(msk);
                        msk &= msk - 1;
                        const int eb = (ii << 4) + eb0;
                        // all of the pair's records read before any is used: one LDS wait per pair
                        // instead of one per record (force pass 3% faster; same arithmetic)
                        const float4 q0 = lds_at(sp[0], eb), q1 = lds_at(sp[1], eb), q3 = lds_at(sp[2], eb);
                        float4 q2 = make_float4(0.f, 0.f, 0.f, 0.f), q4 = q2;
                        if constexpr (MHD) q4 = lds_at(sp[3], eb);
                        if constexpr (!ONE_H) q2 = lds_at(sp[MHD ? 4 : 3], eb);
                        __builtin_amdgcn_sched_barrier(0);
                        force_pair<MHD, ONE_H>(o0, o1, o2, o3, o4, q0, q1, q2, q3, q4, pc, A);
                    }
                } else {
                    const int gtot = compact_group(msk, first + sb, lm, lst);
                    __syncthreads();
                    const ListT<CH>* mine = lst + lm.gfirst * 32;  // this target's accepted slots
                    for (int q = k; q < gtot; q += K) {
                        const int eb = (int)sizeof(float4) * (int)mine[q];
                        const float4 q0 = lds_at(sp[0], eb), q1 = lds_at(sp[1], eb), q3 = lds_at(sp[2], eb);
                        float4 q2 = make_float4(0.f, 0.f, 0.f, 0.f), q4 = q2;
                        if constexpr (MHD) q4 = lds_at(sp[3], eb);
                        if constexpr (!ONE_H) q2 = lds_at(sp[MHD ? 4 : 3], eb);
                        __builtin_amdgcn_sched_barrier(0);
                        force_pair<MHD, ONE_H>(o0, o1, o2, o3, o4, q0, q1, q2, q3, q4, pc, A);
                    }
                    __syncthreads();
                }
            }
            __syncthreads();
        }
        if constexpr (ONE_H) o2 = s.rec(W.P2);
        force_finish<MHD>(R, W, lm, A, tgt, s, o1, o2, o3, o4, mhd, clean, borve, ch);
    }
}

// The default pass over MHD fields and unequal h takes 98 registers, 4 waves per SIMD, unless it is held to 96.
// The balanced loop is held too; its LDS leaves it 4 waves with unequal h, and it takes 100 there.
template <int CH, bool MHD, int BAL, int RMAX, bool GRID, bool ONE_H>
constexpr int kForceWaves = !GRID && (BAL == 1 || (CH == 64 && MHD && !ONE_H && RMAX == 1)) ? 5 : 1;

template <int CH, bool MIXED, bool MHD, int KT, int BAL, int RMAX = 1, bool GRID = false, bool ONE_H = false>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(kForceWaves<CH, MHD, BAL, RMAX, GRID, ONE_H>)))
void k_forces(PairArgs)
{
    __shared__ NbListR<RMAX> L;
    constexpr int NP = kForcePlanes<MHD, ONE_H && !GRID>;
    __shared__ float4 sp[NP][kForceSlots<CH, NP>];
    __shared__ ListT<CH> lst[BAL == 1 ? 64 * 32 : 1];  // compaction lists of the balanced pair loop
    __shared__ PreList P;
    if constexpr (GRID) {
        // a persistent grid: each wave walks the supercells at a stride of the grid (a multiple
        // of 8, so every cell a wave visits belongs to its own XCD's range)
        for (int vb = blockIdx.x; vb < pair_args().nblk_total; vb += gridDim.x)
            forces_wave<CH, MIXED, MHD, KT, BAL, RMAX>(vb, L, sp, lst, P);
    } else {
        // one supercell per wave
        forces_wave<CH, MIXED, MHD, KT, BAL, RMAX, ONE_H>((int)blockIdx.x, L, sp, lst, P);
    }
}

// ------------------------------------------------------------------------------------------------
// Whole-cell pair passes (tuning pair_balance = 2).
//
// Lane (target t, sub-lane k) owns the contiguous candidate range [k*Lr, min((k+1)*Lr, total)) of
// the 27-supercell virtual list, Lr = ceil(total / K). The density pass stages the positions of
// all candidates at once (chunks of CAPD only for very large stencils), culls its range and stores
// the accepted bits of the range (bit b <-> candidate k*Lr + b). Because the ranges of a target's
// K lanes are consecutive, concatenating their accepted candidates gives each target's neighbour
// list sorted by candidate index. The force pass builds these lists once per supercell in LDS, then
// stages the records chunk by chunk: within a chunk a target's pairs are one contiguous run of its
// list, dealt round-robin to its K lanes, with no per-chunk compaction. Cells whose lists do not
// fit (or whose masks were not stored) take a direct per-lane loop over their own bits.
// ------------------------------------------------------------------------------------------------
constexpr int kCellListCap = 2048;  // uint16 entries of the per-supercell neighbour lists

// Popcount of bits [lo, hi) of a lane's mask row (word w at row[w * 64]).
__device__ __forceinline__ int mask_count(const uint32_t* row, int lo, int hi)
{
    int n = 0;
    for (int b = lo; b < hi;) {
        const int w = b >> 5, off = b & 31;
        const int take = (32 - off) < (hi - b) ? (32 - off) : (hi - b);
        uint32_t m = row[w * 64] >> off;
        if (take < 32) m &= (1u << take) - 1u;
        n += __popc(m);
        b += take;
    }
    return n;
}

// Bits [lo, lo + lim) of a lane's mask row, LSB first (lim <= 32).
__device__ __forceinline__ uint32_t mask_bits(const uint32_t* row, int lo, int lim)
{
    const int w = lo >> 5, off = lo & 31;
    uint32_t a = row[w * 64] >> off;
    if (off && off + lim > 32) a |= row[(w + 1) * 64] << (32 - off);
    return lim == 32 ? a : (a & ((1u << lim) - 1u));
}

template <int CAPD, bool MIXED, bool MHD, int KT>
__global__ __launch_bounds__(64) void k_density_cell(PairArgs)
{
    const PairArgs& args = pair_args();
    const StateBuf& S = args.S;
    const WorkBuf& W = args.W;
    const RunDev* const runs = args.runs;
    constexpr int RMAX = 1;
    __shared__ NbListR<RMAX> L;
    __shared__ float4 sp[CAPD + 3];
    const int cell = xcd_cell(blockIdx.x, args.nblk_total, args.ncell_tot);
    if (cell < 0) return;
    const int t0 = (int)W.cs[cell];
    const int nt = (int)W.cs[cell + 1] - t0;
    if (nt == 0) return;
    const int r = find_run_by_cell(runs, args.nruns, cell);
    RunC& R = ((RunC*)runs)[r];
    int self_v0;
    const int total = Stencil<MIXED, RMAX>(R, cell - R.c0, W.cs).build(R, L, self_v0);
    const int lane = threadIdx.x;
    const LaneMap lm = lane_map(nt, args.kmax);
    const int K = lm.K, k = lm.k;
    const int Lr = (total + K - 1) / K;
    const bool keep = nt <= lm.tpg && Lr <= 32 * kMaskWords && W.nbmask != nullptr;
    const int kern = KT >= 0 ? KT : run_kernel(R.flags);  // compile-time when every run uses one kernel
    const float H2 = R.H2;
    const float gam = R.gamma;
    MaskWriter mw;
    mw.row = W.nbmask + (size_t)cell * (kMaskWords * 64) + lane;
    mw.pend = 0;
    mw.pend_w = -1;
    mw.wlim = kMaskWords;

    for (int tg = 0; tg < nt; tg += lm.tpg) {
        const int t = tg + lm.tl;
        const bool valid = lm.inwave && t < nt;
        const int i = t0 + (valid ? t : 0);
        const uint8_t live = S.mask[i], spc = S.species[i];
        const bool tgt = valid && is_target(spc, live);
        const float4 own = W.P0[i];
        const float h = S.h[i];
        const float uu = S.u[i];
        const float vx = S.vel[0][i], vy = S.vel[1][i], vz = S.vel[2][i];
        const float rho_in = S.rho[i];
        float bx = 0.f, by = 0.f, bz = 0.f, psi = 0.f;
        if (MHD && run_mhd(R.flags)) {
            bx = S.B[0][i];
            by = S.B[1][i];
            bz = S.B[2][i];
            psi = S.psi[i];
        }
        const float invh = 1.0f / h;
        const int self_v = self_v0 + t;
        const int v0 = lm.inwave ? k * Lr : total;
        const int v1 = v0 + Lr < total ? v0 + Lr : total;
        float acc = 0.0f;
        uint32_t cnt = 0;
        for (int base = 0; base < total; base += CAPD) {
            const int top = base + CAPD < total ? base + CAPD : total;
            for (int v = base + lane; v < top; v += 64) {
                float4 t4;
                float4 p = W.P0[list_candidate(L, v, t4)];
                p.x += t4.x;
                p.y += t4.y;
                p.z += t4.z;
                sp[v - base] = p;
            }
            __syncthreads();
            const int a = v0 > base ? v0 : base;
            const int b = v1 < top ? v1 : top;
            for (int cc = a; cc < b; cc += 32) {
                const int lim = b - cc < 32 ? b - cc : 32;
                uint32_t msk = cull32(sp + (cc - base), lim, own.x, own.y, own.z, H2);
                // the self pair passes the cull; its density term is the self term added at the end
                if (self_v >= cc && self_v < cc + lim) msk &= ~(1u << (self_v - cc));
                if (!tgt) msk = 0;
                if (keep) mw.put(msk, cc - v0, lim);
                cnt += (uint32_t)__popc(msk);
                while (msk) {
                    const int ii = __builtin_ctz(msk);
                    msk &= msk - 1;
                    const float4 p = sp[cc - base + ii];
                    float dx, dy, dz;
                    const float r2 = geom_r2(own.x, own.y, own.z, p, dx, dy, dz);
                    acc += p.w * kshape(kern, fast_sqrt(r2) * invh);
                }
            }
            __syncthreads();
        }
        if (keep) mw.flush();
        density_finish<MHD>(R, r, S, W, lm, acc, cnt, valid, tgt, spc, live, Slot(t0, (uint32_t)(i - t0)), own.w, h, uu, vx, vy, vz,
                            rho_in, bx, by, bz, psi, gam, kern);
    }
}

template <int CH, bool MIXED, bool MHD, int KT>
__global__ __launch_bounds__(64) void k_forces_cell(PairArgs)
{
    const PairArgs& args = pair_args();
    const StateBuf& S = args.S;
    const WorkBuf& W = args.W;
    const RunDev* const runs = args.runs;
    constexpr int NP = MHD ? 5 : 4;
    constexpr int RMAX = 1;
    __shared__ NbListR<RMAX> L;
    __shared__ float4 sp[NP][CH + 3];
    __shared__ uint16_t lst[kCellListCap];
    const int cell = xcd_cell(blockIdx.x, args.nblk_total, args.ncell_tot);
    if (cell < 0) return;
    const int t0 = (int)W.cs[cell];
    const int nt = (int)W.cs[cell + 1] - t0;
    if (nt == 0) return;
    const int r = find_run_by_cell(runs, args.nruns, cell);
    RunC& R = ((RunC*)runs)[r];
    int self_v0;
    const int total = Stencil<MIXED, RMAX>(R, cell - R.c0, W.cs).build(R, L, self_v0);
    const int lane = threadIdx.x;
    const LaneMap lm = lane_map(nt, args.kmax);
    const int K = lm.K, k = lm.k;
    const int Lr = (total + K - 1) / K;
    const bool keep = nt <= lm.tpg && Lr <= 32 * kMaskWords;  // the density pass stored masks
    const int kern = KT >= 0 ? KT : run_kernel(R.flags);  // compile-time when every run uses one kernel
    const float H2 = R.H2;
    const PairConst pc(R, kern, R.h0);
    const bool mhd = MHD && run_mhd(R.flags);
    const bool clean = mhd && run_cleaning(R.flags);
    const float borve = mhd ? R.borve : 0.0f;
    const float ch = __uint_as_float(W.chbits[r]);
    const uint32_t* mrow = W.nbmask + (size_t)cell * (kMaskWords * 64) + lane;

    for (int tg = 0; tg < nt; tg += lm.tpg) {
        const int t = tg + lm.tl;
        const bool valid = lm.inwave && t < nt;
        const int i = t0 + (valid ? t : 0);
        const bool tgt = valid && is_target(S.species[i], S.mask[i]);
        const float4 o0 = W.P0[i], o1 = W.P1[i], o2 = W.P2[i], o3 = W.P3[i];
        float4 o4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (MHD) o4 = W.P4[i];
        const int self_v = self_v0 + t;
        const int v0 = lm.inwave ? k * Lr : total;
        const int v1 = v0 + Lr < total ? v0 + Lr : total;
        ForceAcc A = {};

        // neighbour lists from the stored masks: lane order = candidate order within a target
        const int mine = (keep && tgt) ? mask_count(mrow, 0, v1 - v0) : 0;
        const int incl = dpp_incl_scan(mine);
        const bool listed = keep && __shfl(incl, 63, 64) <= kCellListCap;
        int lo = 0;
        if (listed) {
            int pos = incl - mine;
            for (int w = 0; w * 32 < v1 - v0 && mine > 0; ++w) {
                const int lim = (v1 - v0) - w * 32 < 32 ? (v1 - v0) - w * 32 : 32;
                uint32_t m = mask_bits(mrow, w * 32, lim);
                while (m) {
                    const int ii = __builtin_ctz(m);
                    m &= m - 1;
                    lst[pos++] = (uint16_t)(v0 + w * 32 + ii);
                }
            }
            // every lane takes part in the shuffle (a lane reading from an inactive lane does not
            // get that lane's value): clamp the source, then select
            const int pre = __shfl(incl, lm.gfirst > 0 ? lm.gfirst - 1 : 0, 64);
            lo = lm.gfirst > 0 ? pre : 0;  // first entry of this target's list
        }

        for (int base = 0; base < total; base += CH) {
            const int top = base + CH < total ? base + CH : total;
            for (int v = base + lane; v < top; v += 64) {
                const int e = v - base;
                float4 t4;
                const int j = list_candidate(L, v, t4);
                float4 p = W.P0[j];
                p.x += t4.x;
                p.y += t4.y;
                p.z += t4.z;
                sp[0][e] = p;
                sp[1][e] = W.P1[j];
                sp[2][e] = W.P2[j];
                sp[3][e] = W.P3[j];
                if constexpr (MHD) sp[4][e] = W.P4[j];
            }
            __syncthreads();
            if (listed) {
                // this target's entries below `top`: counted from each sub-lane's own bits
                const int a = v0 > base ? v0 : base;
                const int b = v1 < top ? v1 : top;
                const int in_chunk = (tgt && b > a) ? mask_count(mrow, a - v0, b - v0) : 0;
                const int ci = dpp_incl_scan(in_chunk);
                const int cpre = __shfl(ci, lm.gfirst > 0 ? lm.gfirst - 1 : 0, 64);
                const int clast = __shfl(ci, lm.glast, 64);
                const int g = lm.inwave ? clast - (lm.gfirst > 0 ? cpre : 0) : 0;
                for (int q = k; q < g; q += K) {
                    const int e = (int)lst[lo + q] - base;
                    float4 q4 = make_float4(0.f, 0.f, 0.f, 0.f);
                    if constexpr (MHD) q4 = sp[4][e];
                    force_pair<MHD, false>(o0, o1, o2, o3, o4, sp[0][e], sp[1][e], sp[2][e], sp[3][e], q4, pc, A);
                }
                lo += g;
            } else {
                const int a = v0 > base ? v0 : base;
                const int b = v1 < top ? v1 : top;
                for (int cc = a; cc < b; cc += 32) {
                    const int lim = b - cc < 32 ? b - cc : 32;
                    uint32_t msk;
                    if (keep) {
                        msk = mask_bits(mrow, cc - v0, lim);
                    } else {
                        msk = cull32(sp[0] + (cc - base), lim, o0.x, o0.y, o0.z, H2);
                        if (self_v >= cc && self_v < cc + lim) msk &= ~(1u << (self_v - cc));
                    }
                    if (!tgt) msk = 0;
                    while (msk) {
                        const int ii = __builtin_ctz(msk);
                        msk &= msk - 1;
                        const int e = cc - base + ii;
                        float4 q4 = make_float4(0.f, 0.f, 0.f, 0.f);
                        if constexpr (MHD) q4 = sp[4][e];
                        force_pair<MHD, false>(o0, o1, o2, o3, o4, sp[0][e], sp[1][e], sp[2][e], sp[3][e], q4, pc, A);
                    }
                }
            }
            __syncthreads();
        }
        force_finish<MHD>(R, W, lm, A, tgt, Slot(t0, (uint32_t)(i - t0)), o1, o2, o3, o4, mhd, clean, borve, ch);
    }
}

// ------------------------------------------------------------------------------------------------
// kick + CFL + FP64 conservation sums (deterministic two-level reduction)
// ------------------------------------------------------------------------------------------------
// Reduce a run's kick-block partials in a fixed tree order (one workgroup), publish the conserved sums, set
// the next dt and advance the time.
__device__ __forceinline__ void finalize_run(const RunDev& R, int r, const WorkBuf& W, double dt_host, int advance,
                                             int priming)
{
    __shared__ double red[6][4];
    double s[6] = {INFINITY, 0, 0, 0, 0, 0};
    const double* base = W.partial + (int64_t)R.kb_first * 6;
    int bb = threadIdx.x;
    for (; bb + 768 < R.kb_count; bb += 1024) {  // four partials per round, loads independent
        double v[4][6];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int q = 0; q < 6; ++q) v[u][q] = base[(int64_t)(bb + 256 * u) * 6 + q];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            s[0] = fmin(s[0], v[u][0]);
            for (int q = 1; q < 6; ++q) s[q] += v[u][q];
        }
    }
    for (; bb < R.kb_count; bb += 256) {
        double v[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) v[q] = base[(int64_t)bb * 6 + q];
        s[0] = fmin(s[0], v[0]);
#pragma unroll
        for (int q = 1; q < 6; ++q) s[q] += v[q];
    }
    // butterfly within each wave (every lane ends with the wave's result), then the four waves in order
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        s[0] = fmin(s[0], __shfl_xor(s[0], off, 64));
#pragma unroll
        for (int q = 1; q < 6; ++q) s[q] += __shfl_xor(s[q], off, 64);
    }
    const int wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 6; ++q) red[q][wid] = s[q];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) {
            red[0][0] = fmin(red[0][0], red[0][w]);
            for (int q = 1; q < 6; ++q) red[q][0] += red[q][w];
        }
        const double dt_used = dt_host > 0.0 ? dt_host : W.dt[r];
        double t = W.time[r];
        if (advance && !priming && isfinite(dt_used)) t += dt_used;
        W.time[r] = t;
        const double dtn = R.dt_fixed > 0.0 ? R.dt_fixed : red[0][0];
        double* c = W.cons + (int64_t)r * 8;
        c[0] = red[1][0];
        c[1] = red[2][0];
        c[2] = red[3][0];
        c[3] = red[4][0];
        c[4] = red[5][0];
        c[5] = dtn;
        c[6] = t;
        c[7] = (double)__uint_as_float(W.chbits[r]);
        // a step sets the next dt; a reduction outside a step (prime, queries) sets it only for
        // runs still waiting for their first dt, so runs already stepping keep their own sequence.
        // A run's first step after new initial data is its priming step: no drift, no kick, no
        // time advance (the same arithmetic as sph_prime), only its first CFL dt
        if (advance || priming) W.dt[r] = dtn;
        // the step that primed the run is done; the count above bit 0 (k_kick) starts again
        __hip_atomic_store(&W.prime_flag[r], advance ? 0 : priming, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Up to this many workgroups in all, the kick finalises its runs itself, one launch less. Each workgroup's
// release writes its XCD's L2 back, so the kick grows with their number: 16 workgroups 7.9 us against 5.6 of the
// kick and 4.5 of the finalising launch, 62 8.0 against 5.6 + 4.7, 128 8.8 against 5.7 + 4.7, 250 12.2 against
// 6.3 + 4.7. A step alone takes 64.1 us against 64.8 with 16, 66.5 against 67.4 with 62, as long either way with
// 128 and 0.5 us longer with 168; contexts in turn with 129 take 1.4% longer a pass.
constexpr int kKickFinalizes = 64;

// LAST: the last workgroup of a run to come here also finalises the run.
template <bool MIXED, bool LAST>
__global__ __launch_bounds__(256) void k_kick(const RunDev* __restrict__ runs, StateBuf S, WorkBuf W, double dt_host,
                                              int do_kick)
{
    __shared__ double red[6][4];
    const int b = blockIdx.x;
    const int r = W.blk_run[b];
    const RunDev& R = runs[r];
    // bit 0; the workgroups count themselves off above it (LAST), so the load is atomic as the count is
    const int priming =
        LAST ? __hip_atomic_load(&W.prime_flag[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 1 : W.prime_flag[r];
    const int64_t local = (int64_t)(b - R.kb_first) * 256 + threadIdx.x;
    double v_dt = INFINITY, v_m = 0, v_px = 0, v_py = 0, v_pz = 0, v_e = 0;
    if (local < R.np) {
        const int64_t i = R.p0 + local;
        if (is_target(S.species[i], S.mask[i])) {
            const double dt = dt_host > 0.0 ? dt_host : W.dt[r];
            const float dtf = (float)dt;
            float vx = S.vel[0][i], vy = S.vel[1][i], vz = S.vel[2][i];
            float u = S.u[i];
            const float ax = W.dvdt[0][i], ay = W.dvdt[1][i], az = W.dvdt[2][i];
            float bx = 0.f, by = 0.f, bz = 0.f;
            const bool kick = do_kick && !priming && isfinite(dt);  // no CFL bound: no kick
            if (kick) {
                vx = vx + ax * dtf;
                vy = vy + ay * dtf;
                vz = vz + az * dtf;
                u = u + W.dudt[i] * dtf;
                S.vel[0][i] = vx;
                S.vel[1][i] = vy;
                S.vel[2][i] = vz;
                S.u[i] = u;
            }
            if (run_mhd(R.flags)) {
                bx = S.B[0][i];
                by = S.B[1][i];
                bz = S.B[2][i];
                if (kick) {
                    bx = bx + W.dbdt[0][i] * dtf;
                    by = by + W.dbdt[1][i] * dtf;
                    bz = bz + W.dbdt[2][i] * dtf;
                    S.B[0][i] = bx;
                    S.B[1][i] = by;
                    S.B[2][i] = bz;
                    S.psi[i] = S.psi[i] + W.dpsidt[i] * dtf;
                }
            }
            const float h = S.h[i], vsg = W.vsig[i];
            if (MIXED) {
                double dti = (double)R.cfl * (double)h / (double)vsg;
                double a2 = (double)ax * ax + (double)ay * ay + (double)az * az;
                if (a2 > 0.0) dti = fmin(dti, (double)R.cfl_force * sqrt((double)h / sqrt(a2)));
                v_dt = dti;
            } else {
                float dti = R.cfl * h / vsg;
                float a2 = ax * ax + ay * ay + az * az;
                if (a2 > 0.0f) dti = fminf(dti, R.cfl_force * sqrtf(h / sqrtf(a2)));
                v_dt = (double)dti;
            }
            const double m = (double)S.mass[i];
            const double dvx = vx, dvy = vy, dvz = vz;
            const double b2 = (double)bx * bx + (double)by * by + (double)bz * bz;
            v_m = m;
            v_px = m * dvx;
            v_py = m * dvy;
            v_pz = m * dvz;
            v_e = m * (0.5 * (dvx * dvx + dvy * dvy + dvz * dvz) + (double)u + 0.5 * b2 / (double)S.rho[i]);
        }
    }
    // wave then block reduction, fixed order
    for (int off = 32; off >= 1; off >>= 1) {
        v_dt = fmin(v_dt, __shfl_xor(v_dt, off, 64));
        v_m += __shfl_xor(v_m, off, 64);
        v_px += __shfl_xor(v_px, off, 64);
        v_py += __shfl_xor(v_py, off, 64);
        v_pz += __shfl_xor(v_pz, off, 64);
        v_e += __shfl_xor(v_e, off, 64);
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        red[0][wid] = v_dt;
        red[1][wid] = v_m;
        red[2][wid] = v_px;
        red[3][wid] = v_py;
        red[4][wid] = v_pz;
        red[5][wid] = v_e;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int q = threadIdx.x;
        double s;
        if (q == 0) s = fmin(fmin(red[0][0], red[0][1]), fmin(red[0][2], red[0][3]));
        else s = (red[q][0] + red[q][1]) + (red[q][2] + red[q][3]);
        W.partial[(int64_t)b * 6 + q] = s;
    }
    if constexpr (LAST) {
        // The partials pass between workgroups, and XCDs with an L2 each, within this kernel: the workgroup's are
        // stored before the barrier, its count-off releases them, and the last one acquires everybody's after its
        // own count-off and before the barrier that its loads come after.
        __shared__ int last;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int before = __hip_atomic_fetch_add(&W.prime_flag[r], 2, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            last = (before >> 1) == R.kb_count - 1;
            if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
        if (last) finalize_run(R, r, W, dt_host, do_kick, priming);
    }
}

// One block per run.
__global__ __launch_bounds__(256) void k_finalize(const RunDev* __restrict__ runs, WorkBuf W, double dt_host,
                                                  int advance)
{
    const int r = blockIdx.x;
    finalize_run(runs[r], r, W, dt_host, advance, W.prime_flag[r]);
}


// Pool compaction: destination particle d belongs to the last kept run whose destination start is
// <= d; every state column is copied from its source slot.
__global__ __launch_bounds__(256) void k_move_runs(StateBuf A, StateBuf B, const int64_t* __restrict__ tab, int n_keep,
                                                   int64_t total, int mixed, int mhd)
{
    const int64_t d = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (d >= total) return;
    int lo = 0, hi = n_keep - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[3 * mid] <= d) lo = mid;
        else hi = mid - 1;
    }
    const int64_t s = tab[3 * lo + 1] + (d - tab[3 * lo]);
    B.id[d] = A.id[s];
    B.mask[d] = A.mask[s];
    B.species[d] = A.species[s];
    for (int a = 0; a < 3; ++a) {
        if (mixed) B.pos64[a][d] = A.pos64[a][s];
        else B.pos32[a][d] = A.pos32[a][s];
        B.vel[a][d] = A.vel[a][s];
        if (mhd) B.B[a][d] = A.B[a][s];
    }
    B.mass[d] = A.mass[s];
    B.h[d] = A.h[s];
    B.u[d] = A.u[s];
    B.rho[d] = A.rho[s];
    if (mhd) B.psi[d] = A.psi[s];
}

// Per-run scalars across a change of the run set: the old runs' dt, time and priming flag are saved,
// then new run r takes those of old run run_src[r], or starts fresh when run_src[r] < 0 (dt = its
// fixed dt or 0 until its priming step sets one, time 0, primed by its next step).
__global__ __launch_bounds__(256) void k_save_run_scalars(WorkBuf W, int n_old)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= n_old) return;
    W.run_tmp[3 * q] = W.dt[q];
    W.run_tmp[3 * q + 1] = W.time[q];
    W.run_tmp[3 * q + 2] = (double)W.prime_flag[q];
}

__global__ __launch_bounds__(256) void k_load_run_scalars(const RunDev* __restrict__ runs, WorkBuf W, int n_new)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n_new) return;
    const int q = W.run_src[r];
    if (q >= 0) {
        W.dt[r] = W.run_tmp[3 * q];
        W.time[r] = W.run_tmp[3 * q + 1];
        W.prime_flag[r] = (int32_t)W.run_tmp[3 * q + 2];
    } else {
        W.dt[r] = runs[r].dt_fixed > 0.0 ? runs[r].dt_fixed : 0.0;
        W.time[r] = 0.0;
        W.prime_flag[r] = 1;
    }
}

// New initial data for one run: time 0, dt its fixed dt or 0, primed by its next step.
__global__ void k_restart_run(const RunDev* __restrict__ runs, WorkBuf W, int run)
{
    W.dt[run] = runs[run].dt_fixed > 0.0 ? runs[run].dt_fixed : 0.0;
    W.time[run] = 0.0;
    W.prime_flag[run] = 1;
}

hipError_t launch_remap_runs(const RunDev* runs, const WorkBuf& W, int n_old, int n_new, hipStream_t s)
{
    if (n_old > 0) k_save_run_scalars<<<(unsigned)((n_old + 255) / 256), 256, 0, s>>>(W, n_old);
    if (n_new > 0) k_load_run_scalars<<<(unsigned)((n_new + 255) / 256), 256, 0, s>>>(runs, W, n_new);
    return hipGetLastError();
}

hipError_t launch_restart_run(const RunDev* runs, const WorkBuf& W, int run, hipStream_t s)
{
    k_restart_run<<<1, 1, 0, s>>>(runs, W, run);
    return hipGetLastError();
}

hipError_t launch_move_runs(const StateBuf& A, const StateBuf& B, const int64_t* tab, int n_keep, int64_t total,
                            int mixed, int mhd, hipStream_t s)
{
    if (total <= 0 || n_keep <= 0) return hipSuccess;
    k_move_runs<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(A, B, tab, n_keep, total, mixed, mhd);
    return hipGetLastError();
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
static inline int nblk_xcd(int ncell) { return ((ncell + 7) / 8) * 8; }

// Blocks of a chunked pair-pass launch: one wave per supercell (persistent_waves 0), or a persistent
// grid of that many waves (a multiple of 8) striding over the supercells when there are more cells
// than waves. The whole-cell passes and the 125-cell stencil launch one wave per supercell.
static inline int pair_grid(const LaunchCtx& c, int nblk)
{
    return (c.persistent_waves > 0 && c.persistent_waves < nblk) ? c.persistent_waves : nblk;
}

// One column per blockIdx.y, copied in the widest units that its addresses allow.
__global__ __launch_bounds__(256) void k_copy_columns(CopyTable t)
{
    char* const dst = static_cast<char*>(t.col[blockIdx.y].dst);
    const char* const src = static_cast<const char*>(t.col[blockIdx.y].src);
    const int64_t bytes = t.col[blockIdx.y].bytes;
    const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
    auto copy = [&](auto unit) {
        using T = decltype(unit);
        const int64_t n = bytes / (int64_t)sizeof(T);
        for (int64_t i = first; i < n; i += step) reinterpret_cast<T*>(dst)[i] = reinterpret_cast<const T*>(src)[i];
        const int64_t at = n * (int64_t)sizeof(T) + first;  // fewer than sizeof(T) bytes are left
        if (at < bytes) dst[at] = src[at];
    };
    const uintptr_t low = reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src);
    if ((low & 15) == 0) copy(uint4{});
    else if ((low & 7) == 0) copy(uint64_t{});
    else if ((low & 3) == 0) copy(uint32_t{});
    else copy(uint8_t{});
}

// The same by kCopyOutWaves waves of one XCD, for larger responses: stores to host memory hold up whatever
// else their XCD writes, so they are kept off the other seven (workgroups are dealt to the XCDs in turn; only
// those of the first work), and few waves, each waiting for its stores, fill the link. Three contexts in turn
// with 3.75 MB each: 101 us against 119 over all XCDs.
constexpr int kCopyOutWaves = 32;
constexpr int kCopyOutUnits = 4;  // 16-byte units per lane in flight

__global__ __launch_bounds__(64) void k_copy_out(CopyTable t)
{
    if (blockIdx.x % 8 != 0) return;
    const int w = (int)blockIdx.x / 8;
    for (int c = 0; c < t.n; ++c) {
        char* const dst = static_cast<char*>(t.col[c].dst);
        const char* const src = static_cast<const char*>(t.col[c].src);
        const int64_t bytes = t.col[c].bytes;
        auto copy = [&](auto unit) {
            using T = decltype(unit);
            const T* const s = reinterpret_cast<const T*>(src);
            T* const d = reinterpret_cast<T*>(dst);
            constexpr int64_t step = (int64_t)kCopyOutWaves * 64 * kCopyOutUnits;
            const int64_t n = bytes / (int64_t)sizeof(T);
            T now[kCopyOutUnits], next[kCopyOutUnits];
            int64_t i = (int64_t)w * 64 * kCopyOutUnits + threadIdx.x;
#pragma unroll
            for (int u = 0; u < kCopyOutUnits; ++u)
                if (i + 64 * u < n) now[u] = s[i + 64 * u];
            for (; i < n; i += step) {
#pragma unroll
                for (int u = 0; u < kCopyOutUnits; ++u)
                    if (i + step + 64 * u < n) next[u] = s[i + step + 64 * u];
#pragma unroll
                for (int u = 0; u < kCopyOutUnits; ++u)
                    if (i + 64 * u < n) d[i + 64 * u] = now[u];
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
                for (int u = 0; u < kCopyOutUnits; ++u) now[u] = next[u];
            }
            const int64_t at = n * (int64_t)sizeof(T) + threadIdx.x;  // fewer than sizeof(T) bytes are left
            if (w == 0 && at < bytes) dst[at] = src[at];
        };
        const uintptr_t low = reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src);
        if ((low & 15) == 0) copy(uint4{});
        else if ((low & 7) == 0) copy(uint64_t{});
        else if ((low & 3) == 0) copy(uint32_t{});
        else copy(uint8_t{});
    }
}

hipError_t launch_copy_columns(const CopyTable& t, hipStream_t s)
{
    if (t.n <= 0) return hipSuccess;
    int64_t most = 0;
    for (int i = 0; i < t.n; ++i) most = most > t.col[i].bytes ? most : t.col[i].bytes;
    const int64_t blocks = (most + 4095) / 4096;  // 16 bytes per thread
    k_copy_columns<<<dim3((unsigned)(blocks < 64 ? blocks : 64), (unsigned)t.n), 256, 0, s>>>(t);
    return hipGetLastError();
}

hipError_t launch_copy_out(const CopyTable& t, hipStream_t s)
{
    int64_t bytes = 0;
    for (int i = 0; i < t.n; ++i) bytes += t.col[i].bytes;
    if (bytes <= kWideCopyBytes) return launch_copy_columns(t, s);
    k_copy_out<<<8 * kCopyOutWaves, 64, 0, s>>>(t);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    k_fill_u32<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(p, v, n);
    return hipGetLastError();
}

template <bool STORE>
static void drift_bin(const LaunchCtx& c, double dt_host, int do_drift)
{
    if (c.mixed)
        k_drift_bin<true, STORE><<<c.nkb, 256, 0, c.stream>>>(c.runs, c.S, c.W, dt_host, do_drift);
    else
        k_drift_bin<false, STORE><<<c.nkb, 256, 0, c.stream>>>(c.runs, c.S, c.W, dt_host, do_drift);
}

hipError_t launch_drift_bin(const LaunchCtx& c, double dt_host, int do_drift, bool store)
{
    if (store) drift_bin<true>(c, dt_host, do_drift);
    else drift_bin<false>(c, dt_host, do_drift);
    return hipGetLastError();
}

hipError_t launch_scan(const LaunchCtx& c)
{
    const int n = c.ncell_tot;
    if (n <= kScatterCells) return hipSuccess;  // k_scatter scans the histogram itself
    const int nb = (n + kScanBlock - 1) / kScanBlock;
    k_scan_local<<<nb, 256, 0, c.stream>>>(c.W.count, c.W.bsum, n);
    if (nb > kScatterBlocks) k_scan_top<<<1, 1024, 0, c.stream>>>(c.W.bsum, nb);
    return hipGetLastError();
}

template <bool STATE>
static void gather(const LaunchCtx& c, const StateBuf& Snew, int grid, double dt_host, int do_drift)
{
    if (c.mixed)
        k_gather<true, STATE><<<grid, 256, 0, c.stream>>>(c.runs, c.S, Snew, c.W, c.has_mhd, c.ncell_tot, c.nkb,
                                                          dt_host, do_drift);
    else
        k_gather<false, STATE><<<grid, 256, 0, c.stream>>>(c.runs, c.S, Snew, c.W, c.has_mhd, c.ncell_tot, c.nkb,
                                                           dt_host, do_drift);
}

hipError_t launch_scatter_gather(const LaunchCtx& c, const StateBuf& Snew, double dt_host, int do_drift)
{
    // both kernels also walk the supercells, at most four per thread: sparse sets need more workgroups for
    // that than for their particles
    const int cells = (c.ncell_tot + 1023) / 1024;
    const int grid = c.nkb > cells ? c.nkb : cells;
    if (c.ncell_tot <= kScatterCells)
        k_scatter<true><<<grid, 256, 0, c.stream>>>(c.runs, c.S, c.W, c.ncell_tot, c.nkb);
    else
        k_scatter<false><<<grid, 256, 0, c.stream>>>(c.runs, c.S, c.W, c.ncell_tot, c.nkb);
    if (!c.has_state) gather<false>(c, Snew, grid, dt_host, do_drift);
    else gather<true>(c, Snew, grid, dt_host, do_drift);
    return hipGetLastError();
}

static inline PairArgs args_of(const LaunchCtx& c, int nblk)
{
    return PairArgs{c.runs, c.nruns, c.ncell_tot, nblk, c.kmax, (int64_t)c.nkb * 256 >= c.ncell_tot, c.S, c.W};
}

#define SPH_COMMA ,
// Instantiate a pair kernel for (precision, MHD fields, smoothing kernel): KT = -1 reads the kernel
// type per run (batches that mix kernel types).
#define SPH_PAIR_DISPATCH(KERNEL, GRIDN, SIZE, EXTRA, ...)                                          \
    do {                                                                                            \
        auto go = [&](auto mixed, auto mhd, auto kt) {                                              \
            KERNEL<SIZE, decltype(mixed)::value, decltype(mhd)::value, decltype(kt)::value EXTRA>    \
                <<<(GRIDN), 64, 0, c.stream>>>(__VA_ARGS__);                                         \
        };                                                                                          \
        auto kt_go = [&](auto mixed, auto mhd) {                                                    \
            switch (c.kern) {                                                                       \
            case 0: go(mixed, mhd, std::integral_constant<int, 0>{}); break;                        \
            case 1: go(mixed, mhd, std::integral_constant<int, 1>{}); break;                        \
            case 2: go(mixed, mhd, std::integral_constant<int, 2>{}); break;                        \
            default: go(mixed, mhd, std::integral_constant<int, -1>{}); break;                      \
            }                                                                                       \
        };                                                                                          \
        if (c.mixed) {                                                                              \
            if (c.has_mhd) kt_go(std::true_type{}, std::true_type{});                               \
            else kt_go(std::true_type{}, std::false_type{});                                        \
        } else {                                                                                    \
            if (c.has_mhd) kt_go(std::false_type{}, std::true_type{});                              \
            else kt_go(std::false_type{}, std::false_type{});                                       \
        }                                                                                           \
    } while (0)

constexpr int kDensitySlots = 256;      // LDS slots of the chunked density pass (DensityLds)
constexpr int kDensityCellSlots = 512;  // and of the whole-cell one

static void density_chunked(const LaunchCtx& c, int nblk)
{
    const int grid = pair_grid(c, nblk);
    if (grid < nblk)
        SPH_PAIR_DISPATCH(k_density, grid, kDensitySlots, SPH_COMMA 1 SPH_COMMA true, args_of(c, nblk));
    else
        SPH_PAIR_DISPATCH(k_density, nblk, kDensitySlots, , args_of(c, nblk));
}

// supercells finer than H somewhere in the context: the chunked lane loop over the 125-cell stencil
static void density_fine(const LaunchCtx& c, int nblk)
{
    SPH_PAIR_DISPATCH(k_density, nblk, kDensitySlots, SPH_COMMA 2, args_of(c, nblk));
}

static void density_cell(const LaunchCtx& c, int nblk)
{
    SPH_PAIR_DISPATCH(k_density_cell, nblk, kDensityCellSlots, , args_of(c, nblk));
}

template <int CH>
static void forces_cell_ch(const LaunchCtx& c, int nblk)
{
    SPH_PAIR_DISPATCH(k_forces_cell, nblk, CH, , args_of(c, nblk));
}

hipError_t launch_density(const LaunchCtx& c)
{
    const int nblk = nblk_xcd(c.ncell_tot);
    if (c.rmax == 2) density_fine(c, nblk);
    else if (c.balance == 2) density_cell(c, nblk);
    else density_chunked(c, nblk);
    return hipGetLastError();
}

template <int CH, int BAL>
static void forces_ch(const LaunchCtx& c, int nblk)
{
    const int grid = pair_grid(c, nblk);
    if (grid < nblk)
        SPH_PAIR_DISPATCH(k_forces, grid, CH, SPH_COMMA BAL SPH_COMMA 1 SPH_COMMA true, args_of(c, nblk));
    else if (c.one_h)  // one smoothing length per run: the pair loop neither tests nor averages h
        SPH_PAIR_DISPATCH(k_forces, nblk, CH, SPH_COMMA BAL SPH_COMMA 1 SPH_COMMA false SPH_COMMA true,
                          args_of(c, nblk));
    else
        SPH_PAIR_DISPATCH(k_forces, nblk, CH, SPH_COMMA BAL, args_of(c, nblk));
}

template <int CH>
static void forces_fine_ch(const LaunchCtx& c, int nblk)
{
    SPH_PAIR_DISPATCH(k_forces, nblk, CH, SPH_COMMA 0 SPH_COMMA 2, args_of(c, nblk));
}

hipError_t launch_forces(const LaunchCtx& c)
{
    const int nblk = nblk_xcd(c.ncell_tot);
    if (c.rmax == 2) {
        if (c.force_chunk >= 128) forces_fine_ch<128>(c, nblk);
        else forces_fine_ch<64>(c, nblk);
    } else if (c.balance == 2) {
        forces_cell_ch<128>(c, nblk);
    } else if (c.force_chunk >= 128) {
        if (c.balance == 1) forces_ch<128, 1>(c, nblk);
        else forces_ch<128, 0>(c, nblk);
    } else {
        if (c.balance == 1) forces_ch<64, 1>(c, nblk);
        else forces_ch<64, 0>(c, nblk);
    }
    return hipGetLastError();
}

hipError_t launch_kick(const LaunchCtx& c, double dt_host, int do_kick)
{
    if (c.nkb <= kKickFinalizes) {
        if (c.mixed)
            k_kick<true, true><<<c.nkb, 256, 0, c.stream>>>(c.runs, c.S, c.W, dt_host, do_kick);
        else
            k_kick<false, true><<<c.nkb, 256, 0, c.stream>>>(c.runs, c.S, c.W, dt_host, do_kick);
        return hipGetLastError();
    }
    if (c.mixed)
        k_kick<true, false><<<c.nkb, 256, 0, c.stream>>>(c.runs, c.S, c.W, dt_host, do_kick);
    else
        k_kick<false, false><<<c.nkb, 256, 0, c.stream>>>(c.runs, c.S, c.W, dt_host, do_kick);
    k_finalize<<<c.nruns, 256, 0, c.stream>>>(c.runs, c.W, dt_host, do_kick);
    return hipGetLastError();
}

}  // namespace sph
