// bsn_kernels.hip -- CDNA4 kernels of the Euler right-hand side, the SSP-RK3
// stage update, the CFL reduction, ghost fills and FMR transfer operators.
//
// Kernel map (reference function -> kernel):
//   fill_ghost_3d_outflow!/periodic!  euler3d.jl:33-62        k_ghost_fill
//   _apply_floors_kernel!             gpu_kernels.jl:26-46    k_floors (and inside k_update)
//   _weno_fluxes_{x,y,z}_kernel!      gpu_kernels.jl:51-154   k_flux<DIR>
//   _flux_divergence_kernel!          gpu_kernels.jl:159-169  k_update (fused)
//   _sg_gradient_kernel!              gpu_kernels.jl:291-319  k_update (fused), k_sg_force
//   _bh_gravity_kernel!               gpu_kernels.jl:199-230  update kernels (fused), k_src
//   _sink_sources_kernel!             gpu_kernels.jl:238-284  update kernels (fused), k_src
//   RK3 stage combines                euler3d.jl:244,250,256  k_update (fused), k_ghost_combine
//   _cfl_speeds_kernel! + maximum     gpu_kernels.jl:174-191  k_update (stage 3), k_cfl
//   _prolong_fine_ghosts!/_prolong_all!  fmr3d.jl:206-255     k_prolong
//   _restrict!                        fmr3d.jl:266-285        k_restrict
//   _accumulate_fr_coarse!/_fine!     fmr3d.jl:292-369        k_fr_coarse, k_fr_fine
//   _bc_correct!                      fmr3d.jl:379-422        k_fmr_correct (with _restrict! and floors)
//
// All work is described by device-resident tile lists (struct Tile) or by
// per-grid prefix offsets, so one launch sweeps any number of grids of any
// shape.  Tile-list kernels are persistent: a workgroup takes a contiguous
// chunk of the list, which keeps neighbouring tiles (shared halo cells) on one
// CU and one XCD L2.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <mutex>
#include "bsn_internal.hpp"
#include "bsn_physics.hpp"
#include "bsn_launch.hpp"

namespace bsn {

#define NG BSN_NG

__device__ __forceinline__ int64_t uidx(const GridDev& G, int i, int j, int k) {
    return ((int64_t)k * G.Ny + j) * G.pitch + BSN_XOFF + i;
}

// Global-address-space view of a device pointer.  The state and flux
// pointers come out of the GridDev table in memory, so the compiler cannot
// infer their address space and would emit flat loads and stores; flat
// operations also count against the scalar-load counter, and every scalar
// reload of a table field would then wait for all HBM loads in flight.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gmem(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}

// base + a 32-bit byte offset.  With a uniform base (scalar registers) and a
// per-lane offset, a store takes the global saddr form and needs no 64-bit
// address arithmetic.  Callers keep the uniform parts (the field, the z plane)
// in the base and only the in-plane part in the offset, so the offset stays
// far below 4 GiB.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* at_off(T* base, uint32_t off) {
    return (__attribute__((address_space(1))) T*)((__attribute__((address_space(1))) char*)base + off);
}

// Load through a raw buffer descriptor: a uniform base (scalar registers, a
// range of 2 GiB) and a 32-bit per-lane byte offset.  The compiler folds
// a plain pointer's per-lane offset into the base and then carries that
// 64-bit per-lane address from one loop iteration to the next, one 64-bit
// VALU addition per load; through the descriptor the base stays scalar.
// The base must be uniform over the wave.  NT: streaming (nontemporal).
template <typename T, bool NT = false>
__device__ __forceinline__ T bld(const T* base, uint32_t off) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4- or 8-byte loads");
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x00020000);
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, NT ? 2 : 0));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, NT ? 2 : 0));
}

// The contiguous tiles of this workgroup.  Where the list does not divide
// evenly the first workgroups take one more: consecutive workgroups go to
// different XCDs and CUs, so the longer chunks spread over the chip.  (Chunks
// cut at b n / G put every longer chunk of, say, 576 tiles over 512 workgroups
// on the one XCD that workgroups 7, 15, 23, ... run on.)
__device__ __forceinline__ void chunk(int ntiles, int& t0, int& t1) {
    const int b = (int)blockIdx.x, q = ntiles / (int)gridDim.x, r = ntiles % (int)gridDim.x;
    t0 = b * q + min(b, r);
    t1 = t0 + q + (b < r ? 1 : 0);
}

// Lane -> (x, row) of a column tile: 64 lanes along x and one row per wave,
// or, in a flat tile (COL_FLAT in a), 256 consecutive columns in row-major
// order from (a, b), wrapping after width columns.  row0: the wave's first row.
__device__ __forceinline__ void col_lane(int width, int a, int b, int& i, int& row, int& row0) {
    const int lx = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a & COL_FLAT) {
        const unsigned s = (unsigned)(a & ~COL_FLAT) + 64u * wv, q0 = s / (unsigned)width;
        const unsigned x = s - q0 * width + lx, q = x / (unsigned)width;
        row0 = b + (int)q0;
        row = row0 + (int)q;
        i = (int)(x - q * width);
    } else {
        row0 = row = b + wv;
        i = a + lx;
    }
}

__device__ __forceinline__ int find_grid(const int64_t* __restrict__ off, int ngrids, int64_t e) {
    int lo = 0, hi = ngrids - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= e) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// Ghost cells.  The set of ghost cells of a grid is split into three disjoint
// slabs: x-slabs (ghost i, all j, k), y-slabs (active i, ghost j, all k) and
// z-slabs (active i, j, ghost k) -- the same partition as the reference's
// fill order (euler3d.jl:36-43, fmr3d.jl:228-254).

__device__ __forceinline__ int64_t ghost_count(const GridDev& G) {
    return 2 * NG * ((int64_t)G.Ny * G.Nz + (int64_t)G.nx * G.Nz + (int64_t)G.nx * G.ny);
}

__device__ __forceinline__ void ghost_decode(const GridDev& G, int64_t t, int& i, int& j, int& k) {
    const int64_t A = 2 * NG * (int64_t)G.Ny * G.Nz;
    const int64_t B = 2 * NG * (int64_t)G.nx * G.Nz;
    if (t < A) {
        int ig = (int)(t % (2 * NG)); t /= 2 * NG;
        j = (int)(t % G.Ny); k = (int)(t / G.Ny);
        i = ig < NG ? ig : G.nx + ig;
    } else if (t < A + B) {
        t -= A;
        i = NG + (int)(t % G.nx); t /= G.nx;
        int jg = (int)(t % (2 * NG)); k = (int)(t / (2 * NG));
        j = jg < NG ? jg : G.ny + jg;
    } else {
        t -= A + B;
        i = NG + (int)(t % G.nx); t /= G.nx;
        j = NG + (int)(t % G.ny);
        int kg = (int)(t / G.ny);
        k = kg < NG ? kg : G.nz + kg;
    }
}

__device__ __forceinline__ int bc_src(int a, int n, bool periodic) {
    if (periodic) return a < NG ? a + n : (a >= NG + n ? a - n : a);
    return a < NG ? NG : (a >= NG + n ? NG + n - 1 : a);
}

// Ghost fill by boundary condition.  A ghost cell takes the value of the
// active cell its index maps to per axis; this equals the reference's
// x -> y -> z sequence of slab copies (each slab copy only moves values that
// an earlier copy placed).  With copy_un, the raw value of every ghost cell
// is first saved to Un (the RK3 base state is a copy of the input).
__global__ void k_ghost_fill(const GridDev* __restrict__ grids, const int64_t* __restrict__ off,
                             int ngrids, int copy_un) {
    const int64_t total = off[ngrids];
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int g = find_grid(off, ngrids, e);
        const GridDev& G = grids[g];
        int i, j, k;
        ghost_decode(G, e - off[g], i, j, k);
        const int si = bc_src(i, G.nx, G.bc & 1), sj = bc_src(j, G.ny, G.bc & 2),
                  sk = bc_src(k, G.nz, G.bc & 4);
        const int64_t d = uidx(G, i, j, k), s = uidx(G, si, sj, sk);
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            if (copy_un) G.Un[q * G.fs + d] = G.U[q * G.fs + d];
            G.U[q * G.fs + d] = G.U[q * G.fs + s];
        }
    }
}

// Stage-3 combination on ghost cells, where the reference's dU is zero
// (euler3d.jl:138 fills dU with zeros; the combine runs over the whole array).
// With ghost mapping the stage input's ghost value is read from the active
// cell it maps to.
// advance: the step ends here, t += dt.
__global__ void k_ghost_combine(const GridDev* __restrict__ grids, const int64_t* __restrict__ off,
                                int ngrids, int stage, int advance) {
    if (advance && blockIdx.x == 0)
        for (int g = threadIdx.x; g < ngrids; g += blockDim.x) {
            double* s = grids[g].scal;
            s[SCAL_T] = s[SCAL_T] + s[SCAL_DT];
        }
    const int64_t total = off[ngrids];
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int g = find_grid(off, ngrids, e);
        const GridDev& G = grids[g];
        int i, j, k;
        ghost_decode(G, e - off[g], i, j, k);
        const int64_t d = uidx(G, i, j, k);
        const int64_t su = (G.lmode & 1) ? uidx(G, bc_src(i, G.nx, G.bc & 1), bc_src(j, G.ny, G.bc & 2),
                                                bc_src(k, G.nz, G.bc & 4))
                                         : d;
        const double dt = G.scal[SCAL_DT];
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const double un = G.Un[q * G.fs + d], u = G.U[q * G.fs + su];
            double v;
            if (stage == 1)      v = un + dt * 0.0;
            else if (stage == 2) v = 0.75 * un + 0.25 * u + (0.25 * dt) * 0.0;
            else                 v = (1.0 / 3.0) * un + (2.0 / 3.0) * u + ((2.0 / 3.0) * dt) * 0.0;
            G.Uout[q * G.fs + d] = v;
        }
    }
}

// a / b: IEEE division for the FP64 form; for the split form (FAST) the
// product with a reciprocal good to a few ulp, which its FP64 state needs for
// range and accuracy, not for bit parity.
template <bool FAST>
__device__ __forceinline__ double ddiv(double a, double b) {
    if (FAST) return a * sp::rcp64(b);
    return a / b;
}

// src/gpu_kernels.jl:26-46 on the five values of one cell.
template <bool FAST = false>
__device__ __forceinline__ bool apply_floor(double (&u)[5], double rho_floor, double P_floor,
                                            double g) {
    const double r = u[0];
    if (r < rho_floor) {
        u[0] = rho_floor; u[1] = 0.0; u[2] = 0.0; u[3] = 0.0;
        u[4] = P_floor / (g - 1.0);
        return true;
    }
    const double KE = ddiv<FAST>(0.5 * (u[1] * u[1] + u[2] * u[2] + u[3] * u[3]), r);
    const double P = (g - 1.0) * (u[4] - KE);
    if (P < P_floor) { u[4] = P_floor / (g - 1.0) + KE; return true; }
    return false;
}

// Loads the five values a stage sees at padded cell (i, j, k) of its input
// U, where only axis AX may be a ghost index.  With lmode bit 0 a ghost cell
// reads the active cell its index maps to (the value the reference's ghost
// fill would have copied there, unfloored: the fill precedes the floors,
// euler3d.jl:189-196); with lmode bit 1 an active cell is floored on load.
// NT: streaming (nontemporal) loads, for callers that read each cell once.
template <int AX, bool FLOOR = true, bool FAST = false, bool NT = false>
__device__ __forceinline__ void load_cell(const GridDev& G, int i, int j, int k, double (&u)[5]) {
    int si = i, sj = j, sk = k;
    if (G.lmode & 1) {
        if (AX == 0) si = bc_src(i, G.nx, G.bc & 1);
        if (AX == 1) sj = bc_src(j, G.ny, G.bc & 2);
        if (AX == 2) sk = bc_src(k, G.nz, G.bc & 4);
    }
    const int64_t o = uidx(G, si, sj, sk);
#pragma unroll
    for (int q = 0; q < 5; ++q)
        u[q] = NT ? __builtin_nontemporal_load(&gmem(G.U)[q * G.fs + o]) : gmem(G.U)[q * G.fs + o];
    // only active cells are floored (callers pass active cross indices; a
    // ghost cell holds the raw value of a ghost fill or a prolongation)
    const bool active = AX == 0 ? (i >= NG && i < NG + G.nx)
                      : AX == 1 ? (j >= NG && j < NG + G.ny) : (k >= NG && k < NG + G.nz);
    if (FLOOR && (G.lmode & 2) && active) apply_floor<FAST>(u, G.rho_floor, G.P_floor, G.gamma);
}

__device__ __forceinline__ void floor_cell(const GridDev& G, int64_t c, bool copy_un) {
    double u[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) u[q] = G.U[q * G.fs + c];
    if (copy_un) {
#pragma unroll
        for (int q = 0; q < 5; ++q) G.Un[q * G.fs + c] = u[q];
    }
    // the split form floors with the same division wherever it floors
    const bool fired = G.prec == 1 ? apply_floor<true>(u, G.rho_floor, G.P_floor, G.gamma)
                                   : apply_floor<false>(u, G.rho_floor, G.P_floor, G.gamma);
    if (fired) {
#pragma unroll
        for (int q = 0; q < 5; ++q) G.U[q * G.fs + c] = u[q];
    }
}

// Floors on active cells (apply_floors_3d!, euler3d.jl:73-80); with copy_un
// the raw value is saved to Un first.
__global__ void k_floors(const GridDev* __restrict__ grids, const int64_t* __restrict__ off,
                         int ngrids, int copy_un) {
    const int64_t total = off[ngrids];
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int g = find_grid(off, ngrids, e);
        const GridDev& G = grids[g];
        int64_t t = e - off[g];
        const int i = NG + (int)(t % G.nx); t /= G.nx;
        const int j = NG + (int)(t % G.ny);
        const int k = NG + (int)(t / G.ny);
        floor_cell(G, uidx(G, i, j, k), copy_un);
    }
}

// ---------------------------------------------------------------------------
// Interface fluxes.  One workgroup stages a pencil tile of cells (five
// conserved values reduced to rho, m, P) in LDS, six cells deep along the
// sweep direction, then each thread computes one interface.
//
//   DIR 0 (x): tile (g, f0, j0, k): interfaces f0..f0+W-1 (f < nx) along x
//              for rows j0..j0+H-1.  Lanes run along x.  A tile with
//              a = -1 instead computes the last interface f = nx for the
//              rows j0..j0+W*H-1, gathering from HBM.  Each wave stages and
//              computes its own rows (64 / W of them), with no block
//              barrier.
//   DIR 1 (y): tile (g, f0, i0, k): interfaces f0..f0+H-1 (f <= ny) along y
//              for cells i0..i0+W-1.  Lanes run along x (coalesced).
//   DIR 2 (z): tile (g, f0, i0, j): as DIR 1 along z.

template <typename T> struct Prec;
template <> struct Prec<double> {
    using Carry = ex::WenoCarry;
    // big: uniform over the wave, set where a stencil holds a value too large
    // for the flux's shared reciprocals (big_cell) or gamma is out of range
    template <int DIR, bool WALK = false>
    __device__ static void flux(const double (&c)[4][6], const double (&p)[6], const GridDev& G,
                                bool big, double F[5], Carry (&w)[5]) {
        if (__builtin_expect(!ex::interface_flux_shared<DIR, WALK>(c, p, G.gamma, G.gfac, big, F, w), 0)) {
            volatile double s[30];
#pragma unroll
            for (int m = 0; m < 6; ++m) {
#pragma unroll
                for (int q = 0; q < 4; ++q) s[6 * q + m] = c[q][m];
                s[24 + m] = p[m];
            }
            ex::interface_flux_plain<DIR>([&](int q, int m) { return s[6 * q + m]; }, G.gamma, G.gfac, F);
            // the carry is formed again, so that it need not be kept here
            if (WALK) ex::interface_walk_start<1>(c, p, w);
        }
    }
    // The same where at(q, m) can read the stencil again from LDS.
    template <int DIR, typename At>
    __device__ static void flux_at(const double (&c)[4][6], const double (&p)[6], const GridDev& G,
                                bool big, double F[5], Carry (&w)[5], At&& at) {
        if (__builtin_expect(!ex::interface_flux_shared<DIR, false>(c, p, G.gamma, G.gfac, big, F, w), 0)) {
            asm volatile("" ::: "memory");      // at reads again: nothing is kept for it
            ex::interface_flux_plain<DIR>(at, G.gamma, G.gfac, F);
        }
    }
    __device__ static void start(const double (&c)[4][6], const double (&p)[6], Carry (&w)[5]) {
        ex::interface_walk_start(c, p, w);
    }
    __device__ static double pressure(const double (&u)[5], double g) {
        return ex::cell_pressure(u[0], u[1], u[2], u[3], u[4], g);
    }
    __device__ static bool big_cell(const double (&u)[5], double p) {
        return ex::cell_big(u[0], u[1], u[2], u[3], p);
    }
    __device__ static bool big_gamma(double g) { return !ex::gamma_ok(g); }
};
template <> struct Prec<float> {
    using Carry = sp::WenoCarry;
    template <int DIR, bool WALK = false>
    __device__ static void flux(const float (&c)[4][6], const float (&p)[6], const GridDev& G, bool,
                                float F[5], Carry (&w)[5]) {
        sp::interface_flux<DIR, WALK>(c, p, G.gf32[0], G.gf32[1], G.gf32[2], F, w);
    }
    template <int DIR, typename At>
    __device__ static void flux_at(const float (&c)[4][6], const float (&p)[6], const GridDev& G, bool big,
                                float F[5], Carry (&w)[5], At&&) {
        flux<DIR>(c, p, G, big, F, w);
    }
    __device__ static void start(const float (&c)[4][6], const float (&p)[6], Carry (&w)[5]) {
        sp::interface_walk_start(c, p, w);
    }
    __device__ static double pressure(const double (&u)[5], double g) {
        return sp::cell_pressure(u[0], u[1], u[2], u[3], u[4], g);
    }
    __device__ static bool big_cell(const double (&)[5], double) { return false; }
    __device__ static bool big_gamma(double) { return false; }
};

// Stores the flux of interface f along DIR with cross indices ci, cj
// (active, 0-based; ci runs along x for DIR 1 and 2, along y for DIR 0).
// Streaming stores: the update reads each face flux once, from HBM (1.2% off
// the split step at 256^3 against cached stores).
template <int DIR, typename T>
__device__ __forceinline__ void store_face(const GridDev& G, const T (&F)[5], int f, int ci, int cj) {
    auto Fp = gmem((T*)G.F[DIR]);
    int64_t o;
    if (DIR == 0)      o = ((int64_t)cj * G.ny + ci) * G.fp[0] + f;
    else if (DIR == 1) o = ((int64_t)cj * (G.ny + 1) + f) * G.fp[1] + ci;
    else               o = ((int64_t)f * G.ny + cj) * G.fp[2] + ci;
#pragma unroll
    for (int q = 0; q < 5; ++q) __builtin_nontemporal_store(F[q], &Fp[q * G.ffs[DIR] + o]);
}

// tiles t0 .. t1 - 1 of a list
template <int DIR, typename T, int W, int H, bool FLAT>
__device__ __forceinline__ void flux_tiles(const GridDev* __restrict__ grids, const Tile* __restrict__ tiles,
                                           int t0, int t1) {
    constexpr int NT = W * H;
    constexpr bool FAST = sizeof(T) == 4;        // split form
    constexpr int SA = DIR == 0 ? H : H + 5;     // LDS rows
    constexpr int SB = DIR == 0 ? W + 5 : W;     // LDS row length
    // x tiles of 256 threads, 64, 32 or 16 wide: each wave stages and
    // computes its own rows, with no block barrier.  The split 64 x 4 tile is
    // held to 80 VGPRs, 6 waves per SIMD (a few values spilled): 0.367 ms
    // against 0.376 at 91 VGPRs, 5 waves.
    constexpr bool WAVE = DIR == 0 && W * H == 256 && (W == 64 || W == 32 || W == 16);
    // FLAT (64 x 4): the list may hold flat tiles.  A kernel of its own, used
    // where a grid of the list has them: 64 x 4 tiles took 0.379 ms in it at
    // 256^3 (split) against 0.363.
    static_assert(!FLAT || (DIR == 0 && W == 64 && H == 4), "flat tiles are 4 waves of 64");
    constexpr int LW = 64 + 5 * XFLAT_ROWS;      // staged cells of a wave, FLAT
    __shared__ T lds[5][FLAT ? H : SA][FLAT ? LW : SB];
    const int tid = threadIdx.x;
    typename Prec<T>::Carry nc[5];               // unused: no indicators are carried between tiles
    for (int t = t0; t < t1; ++t) {
        const Tile tl = tiles[t];
        const GridDev& G = grids[tl.g];
        const int Nx = G.nx + 2 * NG;
        T c[4][6], p[6];
        if (tl.a < 0) {
            // edge tile (x only): the last interface f = nx of NT consecutive
            // rows from b, gathered from HBM.  The tile is uniform, so every
            // thread of the block takes this branch.
            const int ci = tl.b + tid, cj = tl.c;
            const int f = DIR == 0 ? G.nx : DIR == 1 ? G.ny : G.nz;
            if (ci < (DIR == 0 ? G.ny : G.nx)) {
                bool big = Prec<T>::big_gamma(G.gamma);
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    double u[5];
                    if (DIR == 0)      load_cell<0, true, FAST>(G, f + m, NG + ci, NG + cj, u);
                    else if (DIR == 1) load_cell<1, true, FAST>(G, NG + ci, f + m, NG + cj, u);
                    else               load_cell<2, true, FAST>(G, NG + ci, NG + cj, f + m, u);
                    const double pr = Prec<T>::pressure(u, G.gamma);
                    big |= Prec<T>::big_cell(u, pr);
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[q][m] = (T)u[q];
                    p[m] = (T)pr;
                }
                T F[5];
                Prec<T>::template flux<DIR>(c, p, G, __ballot(big) != 0, F, nc);
                store_face<DIR>(G, F, f, ci, cj);
            }
            continue;
        }
        if constexpr (FLAT) {
            // each wave stages and computes 64 consecutive interfaces: of one
            // row, or, in a flat tile, of up to XFLAT_ROWS rows in row-major
            // order, each row's n interfaces with the n + 5 cells they read.
            // Cell t of the wave's sequence goes to slot t; the interface of a
            // lane in the wave's row s reads slots lane + 5 s ...  Both loads
            // of a lane are issued before either is used (indices clamped into
            // the grid), then floors and pressures.  The wave's first row is
            // uniform: its base stays in scalar registers.
            const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
            const bool flat = tl.a & COL_FLAT;
            int x0 = tl.a & ~COL_FLAT, j0 = tl.b, k0 = tl.c;
            // per staged cell: its padded x, byte offset from the first row's
            // start and whether it exists; of the lane's interface: f and s
            int pc[2], f, seg = 0;
            uint32_t ro[2] = {0, 0};
            bool ok[2], mine;
            const double* rowU;
            if (flat) {
                for (x0 += 64 * wv; x0 > G.nx; x0 -= G.nx + 1)
                    if (++j0 == G.ny) { j0 = 0; ++k0; }
                const int n0 = G.nx + 1 - x0;            // interfaces left in the first row
                // t / d as a product: exact for t < 128 and d >= 9
                const uint32_t m6 = 65536u / (uint32_t)(G.nx + 6) + 1, m1 = 65536u / (uint32_t)(G.nx + 1) + 1;
                auto past = [&](int l) { return l < n0 ? 0 : 1 + (int)(((uint32_t)(l - n0) * m1) >> 16); };
                // a row past the first wraps into the next plane at most once
                // (flat tiles come from grids of at least XFLAT_ROWS rows)
                auto row_ok = [&](int s) { return (j0 + s < G.ny ? k0 : k0 + 1) < G.nz; };
                const int tmax = 64 + 5 * (past(63) + 1);
                seg = past(lane);
                f = seg ? lane - n0 - (seg - 1) * (G.nx + 1) : x0 + lane;
                mine = row_ok(seg);
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const int t = lane + 64 * r, v = t - (n0 + 5);
                    const int sg = v < 0 ? 0 : 1 + (int)(((uint32_t)v * m6) >> 16);
                    pc[r] = v < 0 ? x0 + t : v - (sg - 1) * (G.nx + 6);
                    ok[r] = t < tmax && row_ok(sg);
                    // rows of one plane are a pitch apart, the next plane
                    // starts 2 NG rows on
                    ro[r] = ok[r] ? (uint32_t)(sg + (j0 + sg >= G.ny ? 2 * NG : 0)) * (uint32_t)G.pitch * 8u : 0u;
                    pc[r] = ok[r] ? pc[r] : 0;
                }
                rowU = G.U + uidx(G, 0, j0 + NG, min(k0, G.nz - 1) + NG);
            } else {
                // a row's last interface belongs to the edge tiles
                j0 += wv;
                f = x0 + lane;
                const bool row = j0 < G.ny;
                mine = row && f < G.nx;
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    pc[r] = min(x0 + (r ? W + min(lane, 4) : lane), Nx - 1);
                    ok[r] = row && (r == 0 || lane < 5) && x0 + W * r + lane < Nx;
                }
                rowU = G.U + uidx(G, 0, min(j0, G.ny - 1) + NG, k0 + NG);
            }
            double u[2][5];
            bool big = Prec<T>::big_gamma(G.gamma);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int pi = (G.lmode & 1) ? bc_src(pc[r], G.nx, G.bc & 1) : pc[r];
#pragma unroll
                for (int q = 0; q < 5; ++q) u[r][q] = bld(rowU + q * G.fs, ro[r] + (uint32_t)pi * 8u);
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                if (ok[r]) {
                    if ((G.lmode & 2) && pc[r] >= NG && pc[r] < NG + G.nx)
                        apply_floor<FAST>(u[r], G.rho_floor, G.P_floor, G.gamma);
                    const double pr = Prec<T>::pressure(u[r], G.gamma);
                    big |= Prec<T>::big_cell(u[r], pr);
#pragma unroll
                    for (int q = 0; q < 4; ++q) lds[q][wv][lane + 64 * r] = (T)u[r][q];
                    lds[4][wv][lane + 64 * r] = (T)pr;
                }
            }
            // the cells come from other lanes of this wave: the LDS runs one
            // wave's operations in order, and the fences keep the compiler
            // from moving the reads above the writes
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const bool wbig = __ballot(big) != 0;        // any cell of the wave
            if (mine) {
                const int l0 = lane + 5 * seg;
#pragma unroll
                for (int m = 0; m < 6; ++m) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[q][m] = lds[q][wv][l0 + m];
                    p[m] = lds[4][wv][l0 + m];
                }
                T F[5];
                Prec<T>::template flux_at<0>(c, p, G, wbig, F, nc,
                                             [&](int q, int m) { return lds[q][wv][l0 + m]; });
                T* rowF = (T*)G.F[0] + ((int64_t)k0 * G.ny + j0) * G.fp[0];
                const uint32_t fo = (uint32_t)(seg * G.fp[0] + f) * (uint32_t)sizeof(T);
#pragma unroll
                for (int q = 0; q < 5; ++q)
                    __builtin_nontemporal_store(F[q], at_off(rowF + q * G.ffs[0], fo));
            }
            // the next tile's stores follow this tile's reads (same order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            continue;
        } else if constexpr (WAVE) {
            // each wave stages and computes its own RW = 64 / W rows of the
            // tile (lane -> row hb + lane / W, x = lane % W): cells f0 .. f0+W+4
            // of each row, both loads issued before either is used (indices
            // clamped into the grid), then floors and pressures.  The wave's
            // first row is uniform: its base stays in scalar registers, and a
            // lane's row past it goes into its 32-bit load and store offsets.
            constexpr int RW = 64 / W;
            const int hb = __builtin_amdgcn_readfirstlane(tid >> 6) * RW, lane = tid & 63;
            const int x = lane % W, h = hb + lane / W;
            const bool row_ok = tl.b + h < G.ny;
            const int pjb = NG + min(tl.b + hb, G.ny - 1), pk = NG + tl.c;
            const int pj = NG + min(tl.b + h, G.ny - 1);
            const double* rowU = G.U + uidx(G, 0, pjb, pk);
            const uint32_t roff = (uint32_t)((pj - pjb) * G.pitch) * 8u;
            double u[2][5];
            bool big = Prec<T>::big_gamma(G.gamma);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                int pi = min(tl.a + (r ? W + min(x, 4) : x), Nx - 1);
                if (G.lmode & 1) pi = bc_src(pi, G.nx, G.bc & 1);
#pragma unroll
                for (int q = 0; q < 5; ++q) u[r][q] = bld(rowU + q * G.fs, roff + (uint32_t)pi * 8u);
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int b = r ? W + x : x, pi = tl.a + b;
                if ((r == 0 || x < 5) && row_ok && pi < Nx) {
                    if ((G.lmode & 2) && pi >= NG && pi < NG + G.nx)
                        apply_floor<FAST>(u[r], G.rho_floor, G.P_floor, G.gamma);
                    const double pr = Prec<T>::pressure(u[r], G.gamma);
                    big |= Prec<T>::big_cell(u[r], pr);
#pragma unroll
                    for (int q = 0; q < 4; ++q) lds[q][h][b] = (T)u[r][q];
                    lds[4][h][b] = (T)pr;
                }
            }
            // the rows' cells come from other lanes of this wave: the LDS
            // runs one wave's operations in order, and the fences keep the
            // compiler from moving the reads above the writes
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const bool wbig = __ballot(big) != 0;        // any cell of the wave's rows
            const int f = tl.a + x, ci = tl.b + h;
            if (f < G.nx && ci < G.ny) {
#pragma unroll
                for (int m = 0; m < 6; ++m) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[q][m] = lds[q][h][x + m];
                    p[m] = lds[4][h][x + m];
                }
                T F[5];
                Prec<T>::template flux_at<0>(c, p, G, wbig, F, nc,
                                             [&](int q, int m) { return lds[q][h][x + m]; });
                T* rowF = (T*)G.F[0] + ((int64_t)tl.c * G.ny + tl.b + hb) * G.fp[0];
                const uint32_t fo = (uint32_t)((h - hb) * G.fp[0] + f) * (uint32_t)sizeof(T);
#pragma unroll
                for (int q = 0; q < 5; ++q)
                    __builtin_nontemporal_store(F[q], at_off(rowF + q * G.ffs[0], fo));
            }
            // the next tile's stores follow this tile's reads (same order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            continue;
        }
        // stage cells into LDS
        bool big = Prec<T>::big_gamma(G.gamma);
        for (int e = tid; e < SA * SB; e += NT) {
            const int a = e / SB, b = e - a * SB;
            int pi, pj, pk;
            bool ok;
            if (DIR == 0) {
                pi = tl.a + b; pj = NG + tl.b + a; pk = NG + tl.c;
                ok = pi < Nx && tl.b + a < G.ny;
            } else if (DIR == 1) {
                pi = NG + tl.b + b; pj = tl.a + a; pk = NG + tl.c;
                ok = tl.b + b < G.nx && pj < G.ny + 2 * NG;
            } else {
                pi = NG + tl.b + b; pj = NG + tl.c; pk = tl.a + a;
                ok = tl.b + b < G.nx && pk < G.nz + 2 * NG;
            }
            if (ok) {
                double u[5];
                load_cell<DIR, true, FAST>(G, pi, pj, pk, u);
                const double pr = Prec<T>::pressure(u, G.gamma);
                big |= Prec<T>::big_cell(u, pr);
#pragma unroll
                for (int q = 0; q < 4; ++q) lds[q][a][b] = (T)u[q];
                lds[4][a][b] = (T)pr;
            }
        }
        // any cell of the tile (the FP64 form asks; the barrier orders the LDS)
        if constexpr (FAST) __syncthreads();
        else                big = __syncthreads_or(big);
        const int x = tid % W, h = tid / W;
        int f, ci;
        bool valid;
        if (DIR == 0) {
            f = tl.a + x; ci = tl.b + h;
            valid = f < G.nx && ci < G.ny;
        } else {
            f = tl.a + h; ci = tl.b + x;
            valid = f <= (DIR == 1 ? G.ny : G.nz) && ci < G.nx;
        }
        if (valid) {
#pragma unroll
            for (int m = 0; m < 6; ++m) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    c[q][m] = DIR == 0 ? lds[q][h][x + m] : lds[q][h + m][x];
                p[m] = DIR == 0 ? lds[4][h][x + m] : lds[4][h + m][x];
            }
            T F[5];
            Prec<T>::template flux_at<DIR>(c, p, G, big, F, nc, [&](int q, int m) {
                return DIR == 0 ? lds[q][h][x + m] : lds[q][h + m][x];
            });
            store_face<DIR>(G, F, f, ci, tl.c);
        }
        __syncthreads();
    }
}

template <int DIR, typename T, int W, int H, bool FLAT = false>
__global__ __launch_bounds__(W * H, (DIR == 0 && W == 64 && H == 4 && sizeof(T) == 4) ? 6 : 1) void k_flux(const GridDev* __restrict__ grids,
                                                 const Tile* __restrict__ tiles, int ntiles) {
    int t0, t1;
    chunk(ntiles, t0, t1);
    flux_tiles<DIR, T, W, H, FLAT>(grids, tiles, t0, t1);
}

// x interface fluxes as short register walks.  Tile (g, f0, j0, k | n): a
// block of four waves stages rows j0 .. j0+3 of plane k, cells f0 .. f0+n+4
// (padded x), in LDS; lane l of wave w walks row j0+w through its share of
// the n <= 64 KMAX interfaces f0 .. f0+n-1 (KMAX consecutive ones when the
// tile is full) with a six-cell register window read from LDS, and the split
// form carries the smoothness indicators that consecutive interfaces share.
// With OUT the fluxes go back through the row's LDS slots, so that the lanes
// store them to HBM contiguously; without it each lane stores its fluxes
// as they are formed (cached stores: the L2 joins the lanes' strided words
// into whole lines), which needs no flux registers.  Cell b of a row sits at b + b/4: a lane's
// cells start five words after its neighbour's, so the lanes of a wave read
// distinct banks.  Interfaces 0 .. nx-1 are covered by such tiles; an edge
// tile (g, -1, r0, 0) computes the last interface f = nx of the 256 rows
// r0 .. r0+255 (row r = k ny + j), one per thread, gathering from HBM.
template <typename T, int KMAX, bool OUT>
__global__ __launch_bounds__(256) void k_fxwalk(const GridDev* __restrict__ grids,
                                                const Tile* __restrict__ tiles, int ntiles) {
    constexpr bool FAST = sizeof(T) == 4;        // split form
    constexpr int NC = 64 * KMAX + 5;            // staged cells per row
    constexpr int SB = NC + NC / 4 + 1;          // LDS row length after the skew
    __shared__ T lds[5][4][SB];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    auto at = [](int b) { return b + (b >> 2); };
    typename Prec<T>::Carry nw[5];               // of the edge tiles, which carry nothing
    int t0, t1;
    chunk(ntiles, t0, t1);
    for (int t = t0; t < t1; ++t) {
        const Tile tl = tiles[t];
        const GridDev& G = grids[tl.g];
        if (tl.a < 0) {
            // edge tile: uniform over the block, so no thread reaches the
            // barriers below while another takes this branch
            const int r = tl.b + tid;
            if (r < G.ny * G.nz) {
                const int jr = r % G.ny, kr = r / G.ny;
                T c[4][6], p[6];
                bool big = Prec<T>::big_gamma(G.gamma);
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    double u[5];
                    load_cell<0, true, FAST>(G, G.nx + m, NG + jr, NG + kr, u);
                    const double pr = Prec<T>::pressure(u, G.gamma);
                    big |= Prec<T>::big_cell(u, pr);
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[q][m] = (T)u[q];
                    p[m] = (T)pr;
                }
                T F[5];
                Prec<T>::template flux<0>(c, p, G, __ballot(big) != 0, F, nw);
                store_face<0>(G, F, G.nx, jr, kr);
            }
            continue;
        }
        const int f0 = tl.a, j0 = tl.b, k = tl.c & ZT_K0_MASK, n = tl.c >> ZT_LEN_SHIFT;
        const int nc = n + 5;
        bool big = Prec<T>::big_gamma(G.gamma);
        {
            // every thread issues all of its loads before it uses the first
            // (indices clamped into the grid, so the loads need no branch),
            // so that the tile costs one memory round trip, not NE; the floors
            // follow the loads
            constexpr int NE = (4 * NC + 255) / 256;
            double u[NE][5];
#pragma unroll
            for (int r = 0; r < NE; ++r) {
                const int e = min(tid + 256 * r, 4 * nc - 1);
                const int a = e / nc, b = e - a * nc;
                load_cell<0, false, FAST>(G, f0 + b, NG + min(j0 + a, G.ny - 1), NG + k, u[r]);
            }
#pragma unroll
            for (int r = 0; r < NE; ++r) {
                const int e = tid + 256 * r;
                const int a = e / nc, b = e - a * nc;
                if (e < 4 * nc && j0 + a < G.ny) {
                    if ((G.lmode & 2) && f0 + b >= NG && f0 + b < NG + G.nx)
                        apply_floor<FAST>(u[r], G.rho_floor, G.P_floor, G.gamma);
                    const double pr = Prec<T>::pressure(u[r], G.gamma);
                    big |= Prec<T>::big_cell(u[r], pr);
#pragma unroll
                    for (int q = 0; q < 4; ++q) lds[q][a][at(b)] = (T)u[r][q];
                    lds[4][a][at(b)] = (T)pr;
                }
            }
        }
        // any cell of the tile (the FP64 form asks; the barrier orders the LDS)
        if constexpr (FAST) __syncthreads();
        else                big = __syncthreads_or(big);
        const int j = j0 + w;
        const int b0 = (lane * n) >> 6, len = (((lane + 1) * n) >> 6) - b0;
        T Fb[OUT ? KMAX : 1][5];
        if (j < G.ny && len > 0) {
            T c[4][6], p[6];
            auto place = [&](int slot, int b) {
#pragma unroll
                for (int q = 0; q < 4; ++q) c[q][slot] = lds[q][w][at(b)];
                p[slot] = lds[4][w][at(b)];
            };
#pragma unroll
            for (int m = 0; m < 5; ++m) place(m, b0 + m);
            typename Prec<T>::Carry wc[5];
            if constexpr (FAST) Prec<T>::start(c, p, wc);
            auto step = [&](int m, T (&F)[5]) {
                place(5, b0 + m + 5);
                Prec<T>::template flux<0, FAST>(c, p, G, big, F, wc);
#pragma unroll
                for (int s = 0; s < 5; ++s) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[q][s] = c[q][s + 1];
                    p[s] = p[s + 1];
                }
            };
            if constexpr (OUT) {
                // unrolled, so that the flux registers are indexed statically
#pragma unroll
                for (int m = 0; m < KMAX; ++m)
                    if (m < len) step(m, Fb[m]);
            } else {
                auto Fp = gmem((T*)G.F[0]);
                const int64_t o = ((int64_t)k * G.ny + j) * G.fp[0] + f0 + b0;
                for (int m = 0; m < len; ++m) {
                    step(m, Fb[0]);
#pragma unroll
                    for (int q = 0; q < 5; ++q) Fp[q * G.ffs[0] + o + m] = Fb[0][q];
                }
            }
        }
        if (!OUT) {
            __syncthreads();
            continue;
        }
        // every lane of the block has read its cells: the fluxes replace them
        __syncthreads();
        if (j < G.ny) {
#pragma unroll
            for (int m = 0; m < KMAX; ++m)
                if (m < len) {
#pragma unroll
                    for (int q = 0; q < 5; ++q) lds[q][w][at(b0 + m)] = Fb[OUT ? m : 0][q];
                }
        }
        __syncthreads();
        if (j < G.ny) {
            auto Fp = gmem((T*)G.F[0]);
            const int64_t row = ((int64_t)k * G.ny + j) * G.fp[0] + f0;
            // streaming stores, as for the other sweeps
            for (int e = lane; e < n; e += 64) {
#pragma unroll
                for (int q = 0; q < 5; ++q)
                    __builtin_nontemporal_store(lds[q][w][at(e)], &Fp[q * G.ffs[0] + row + e]);
            }
        }
        __syncthreads();
    }
}

// y (DIR 1) and z (DIR 2) interface fluxes as register walks.  Tile
// (g, i0, c0, f0 | len): 64 x 4 threads over (i, c) with c = k for DIR 1 and
// c = j for DIR 2; each thread walks its column along DIR through the
// interfaces f0 .. f0+len-1 with a six-cell register window, loading one new
// cell per interface straight from HBM (lanes along x: coalesced), and the
// split form carries the smoothness indicators that consecutive interfaces
// share.  A run of len interfaces reads len + 5 cells.
// The FP64 form carries them too, with their reciprocals, at 252 VGPRs, 2 waves
// per SIMD.
template <int DIR, typename T>
__device__ __forceinline__ void walk_tiles(const GridDev* __restrict__ grids, const Tile* __restrict__ tiles,
                                           int t0, int t1) {
    constexpr bool FAST = sizeof(T) == 4;        // split form
    for (int t = t0; t < t1; ++t) {
        const Tile tl = tiles[t];
        const GridDev& G = grids[tl.g];
        const int f0 = tl.c & ZT_K0_MASK, len = tl.c >> ZT_LEN_SHIFT;
        // the wave's first row cc0 (uniform) and this lane's row past it: the
        // walk's addresses are a scalar base per cell or face and a lane offset
        // fixed for the tile
        int i, cc, cc0;
        col_lane(col_width(G.nx, FAST), tl.a, tl.b, i, cc, cc0);
        const int dr = cc - cc0;
        if (i >= G.nx || cc >= (DIR == 1 ? G.nz : G.ny)) continue;
        const uint32_t uoff =
            (uint32_t)(((DIR == 1 ? (int64_t)G.Ny * G.pitch : (int64_t)G.pitch) * dr + NG + i) * 8);
        const uint32_t foff =
            (uint32_t)(((DIR == 1 ? (int64_t)(G.ny + 1) * G.fp[1] : (int64_t)G.fp[2]) * dr + i) * sizeof(T));
        T c[4][6], p[6];
        double nxt[5];
        int npf = 0;
        bool big = Prec<T>::big_gamma(G.gamma);
        // cells along the walk are read once (halo cells of neighbouring
        // runs aside): streaming loads.  The load is raw and the floor is
        // applied when the cell is placed, so that the next cell's load stays
        // in flight during the current interface's flux.  A ghost index along
        // the walk reads the active cell it maps to, as load_cell does.
        auto load = [&](int pf, double (&u)[5]) {
            int sp_ = pf;
            if (G.lmode & 1) sp_ = bc_src(pf, DIR == 1 ? G.ny : G.nz, G.bc & (DIR == 1 ? 2 : 4));
            const int64_t base = DIR == 1 ? ((int64_t)(NG + cc0) * G.Ny + sp_) * G.pitch + BSN_XOFF
                                          : ((int64_t)sp_ * G.Ny + NG + cc0) * G.pitch + BSN_XOFF;
#pragma unroll
            for (int q = 0; q < 5; ++q) u[q] = bld<double, true>(G.U + q * G.fs + base, uoff);
        };
        auto fetch = [&](int pf) { npf = pf; load(pf, nxt); };
        auto place = [&](int slot, int pf, double (&u)[5]) {
            if ((G.lmode & 2) && pf >= NG && pf < NG + (DIR == 1 ? G.ny : G.nz))
                apply_floor<FAST>(u, G.rho_floor, G.P_floor, G.gamma);
            const double pr = Prec<T>::pressure(u, G.gamma);
            big |= __ballot(Prec<T>::big_cell(u, pr)) != 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) c[q][slot] = (T)u[q];
            p[slot] = (T)pr;
        };
        {
            // the window's cells in one memory round trip
            double u[5][5];
#pragma unroll
            for (int m = 0; m < 5; ++m) load(f0 + m, u[m]);
            fetch(f0 + 5);
#pragma unroll
            for (int m = 0; m < 5; ++m) place(m, f0 + m, u[m]);
        }
        typename Prec<T>::Carry wc[5];
        Prec<T>::start(c, p, wc);
        const int fend = f0 + len;
        auto step = [&](int f) {
            place(5, npf, nxt);                         // cell f+5 (padded)
            if (f + 1 < fend) fetch(f + 6);             // in flight during the flux
            T F[5];
            Prec<T>::template flux<DIR, true>(c, p, G, big, F, wc);
            // store_face's layout, from the wave's first row
            T* fb = (T*)G.F[DIR] + (DIR == 1 ? ((int64_t)cc0 * (G.ny + 1) + f) * G.fp[1]
                                             : ((int64_t)f * G.ny + cc0) * G.fp[2]);
#pragma unroll
            for (int q = 0; q < 5; ++q) __builtin_nontemporal_store(F[q], at_off(fb + q * G.ffs[DIR], foff));
#pragma unroll
            for (int m = 0; m < 5; ++m) {
#pragma unroll
                for (int q = 0; q < 4; ++q) c[q][m] = c[q][m + 1];
                p[m] = p[m + 1];
            }
        };
        int f = f0;
        if constexpr (FAST) {
            // six interfaces per pass: the window's slots come back to the
            // same registers after six shifts, so the shifts cost no moves
            // (split form: 754 -> 695 VALU instructions per interface; the
            // FP64 form would double its registers).  The split walk is held
            // to 128 VGPRs, 4 waves per SIMD, with a few values spilled: the
            // y sweep took 0.295 ms against 0.305 at 133 VGPRs and 3 waves.
            for (; f + 6 <= fend; f += 6) {
#pragma unroll
                for (int u = 0; u < 6; ++u) step(f + u);
            }
        }
        for (; f < fend; ++f) step(f);
    }
}

template <int DIR, typename T>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2) void k_fwalk(const GridDev* __restrict__ grids,
                                               const Tile* __restrict__ tiles, int ntiles) {
    int t0, t1;
    chunk(ntiles, t0, t1);
    walk_tiles<DIR, T>(grids, tiles, t0, t1);
}

// All three sweeps of small grids in one launch: the list holds nx x tiles (64 x 4
// and flat), then ny y runs and the z runs, one per workgroup.  Such a sweep
// leaves most of the chip idle and takes the latency of its launch and of one
// interface, which this way is paid once (plan_small in bsn_api.cpp has the times).
template <typename T>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2) void k_sweeps(const GridDev* __restrict__ grids,
                                                                        const Tile* __restrict__ tiles, int nx,
                                                                        int ny) {
    const int b = (int)blockIdx.x;
    if (b < nx)           flux_tiles<0, T, 64, 4, true>(grids, tiles, b, b + 1);
    else if (b < nx + ny) walk_tiles<1, T>(grids, tiles, b, b + 1);
    else                  walk_tiles<2, T>(grids, tiles, b, b + 1);
}

// ---------------------------------------------------------------------------
// Fused flux divergence + phi source + SSP-RK3 stage combine + floors
// (+ the CFL wave-speed maximum of the new state on stage 3).
// Tile (g, i0, j0, k0): 64 x 4 threads over (i, j); each thread walks KZ
// cells along z and carries the z-face flux.  stage 0 stores dU instead
// (euler3d_rhs!).

template <bool FAST = false>
__device__ __forceinline__ uint64_t cfl_speed_bits(const double (&u)[5], const GridDev& G) {
    // src/gpu_kernels.jl:180-189
    const double g = G.gamma;
    const double r = jl_max(u[0], 1e-30);
    const double vx = ddiv<FAST>(u[1], r), vy = ddiv<FAST>(u[2], r), vz = ddiv<FAST>(u[3], r);
    const double KE = 0.5 * (vx * vx + vy * vy + vz * vz);
    const double P = jl_max(((g - 1.0) * (ddiv<FAST>(u[4], r) - KE)) * r, 0.0);
    const double cs = sqrt(ddiv<FAST>(g * P, r));
    const double s = jl_max(jl_max((fabs(vx) + cs) * G.idx, (fabs(vy) + cs) * G.idy),
                            (fabs(vz) + cs) * G.idz);
    return (uint64_t)__double_as_longlong(s);
}

__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t w = (uint64_t)__shfl_xor((unsigned long long)v, o, 64);
        v = w > v ? w : v;
    }
    return v;
}

__device__ __forceinline__ void block_max_to(uint64_t v, unsigned long long* dst) {
    __shared__ uint64_t red[16];
    v = wave_max_u64(v);
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t m = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) m = red[w] > m ? red[w] : m;
        if (m) atomicMax(dst, (unsigned long long)m);
    }
    __syncthreads();
}

// Point-mass gravity on active cell (i, j, k) (0-based) with stage-input
// state u: d += (0, rho a, rho v.a) (src/gpu_kernels.jl:199-230).
__device__ __forceinline__ void bh_gravity_add(const SrcDev& S, int i, int j, int k,
                                               const double (&u)[5], double (&d)[5]) {
    const double xc = S.gx0[0] + ((double)(i + 1) - 0.5) * S.dx;
    const double yc = S.gx0[1] + ((double)(j + 1) - 0.5) * S.dy;
    const double zc = S.gx0[2] + ((double)(k + 1) - 0.5) * S.dz;
    const double r = u[0];
    const double vx = u[1] / r, vy = u[2] / r, vz = u[3] / r;
    double ax = 0.0, ay = 0.0, az = 0.0;
    for (int n = 0; n < S.nbh; ++n) {
        const double ddx = xc - S.px[n], ddy = yc - S.py[n], ddz = zc - S.pz[n];
        const double r2 = ddx * ddx + ddy * ddy + ddz * ddz + S.eps[n] * S.eps[n];
        const double r3 = r2 * sqrt(r2);
        const double fac = -S.mass[n] / r3;
        ax += fac * ddx;
        ay += fac * ddy;
        az += fac * ddz;
    }
    d[1] += r * ax;
    d[2] += r * ay;
    d[3] += r * az;
    d[4] += r * (vx * ax + vy * ay + vz * az);
}

// Gas sinks on active cell (i, j, k): torque-free or uniform drain inside
// each sink radius (src/gpu_kernels.jl:238-284).
__device__ __forceinline__ void sink_add(const SrcDev& S, int i, int j, int k,
                                         const double (&u)[5], double (&d)[5]) {
    const double r = u[0], mx = u[1], my = u[2], mz = u[3], E = u[4];
    if (!(r > S.rho_sink_min)) return;
    const double xc = S.sx0[0] + ((double)(i + 1) - 0.5) * S.dx;
    const double yc = S.sx0[1] + ((double)(j + 1) - 0.5) * S.dy;
    const double zc = S.sx0[2] + ((double)(k + 1) - 0.5) * S.dz;
    for (int n = 0; n < S.nsink; ++n) {
        const double ddx = xc - S.spx[n], ddy = yc - S.spy[n], ddz = zc - S.spz[n];
        const double dist = sqrt(ddx * ddx + ddy * ddy + ddz * ddz);
        if (!(dist < S.rs[n])) continue;
        const double t = S.ts[n];
        d[0] -= r / t;
        if (S.torque_free) {
            const double rx = ddx / dist, ry = ddy / dist, rz = ddz / dist;
            const double vx = mx / r, vy = my / r, vz = mz / r;
            const double vrx = vx - S.svx[n], vry = vy - S.svy[n], vrz = vz - S.svz[n];
            const double v_r = vrx * rx + vry * ry + vrz * rz;
            const double e_int = E / r - 0.5 * (vx * vx + vy * vy + vz * vz);
            d[1] -= r * v_r * rx / t;
            d[2] -= r * v_r * ry / t;
            d[3] -= r * v_r * rz / t;
            d[4] -= (0.5 * r * (v_r * v_r) + r * e_int) / t;
        } else {
            d[1] -= mx / t;
            d[2] -= my / t;
            d[3] -= mz / t;
            d[4] -= E / t;
        }
    }
}

// Flux divergence of one conserved field (src/gpu_kernels.jl:165-167).  The
// split form's FP32 face fluxes are differenced in FP64 (exactly) and the
// three terms summed with FMA; the FP64 form keeps the reference's operations.
template <bool FAST>
__device__ __forceinline__ double flux_div(double fx0, double fx1, double fy0, double fy1,
                                           double fz0, double fz1, const GridDev& G) {
    if (FAST) return -__builtin_fma(fx1 - fx0, G.idx, __builtin_fma(fy1 - fy0, G.idy, (fz1 - fz0) * G.idz));
    return (-(fx1 - fx0)) * G.idx - (fy1 - fy0) * G.idy - (fz1 - fz0) * G.idz;
}

// Phi source, stage combination and floors of active cell (i, j, k) with the
// flux divergence d (src/gpu_kernels.jl:291-319, src/euler3d.jl:244-257);
// the result goes to Uout.  Returns the CFL speed bits of the new state.
template <bool FAST = false>
__device__ __forceinline__ void cell_state(const GridDev& G, int64_t c, int stage, double (&u)[5],
                                           double (&un)[5]) {
    const bool need_u = stage > 1 || G.phi != nullptr || G.src != nullptr;
    // each cell's state is read once per launch: streaming loads (the
    // stand-alone update kernel 0.515 -> 0.544 of HBM peak at 256^3)
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        un[q] = __builtin_nontemporal_load(&gmem(G.Un)[q * G.fs + c]);
        u[q] = need_u ? __builtin_nontemporal_load(&gmem(G.U)[q * G.fs + c]) : 0.0;
    }
    if (need_u && (G.lmode & 2)) apply_floor<FAST>(u, G.rho_floor, G.P_floor, G.gamma);
}

template <bool FAST = false>
__device__ __forceinline__ uint64_t finish_cell_with(const GridDev& G, int i, int j, int k, int stage,
                                                     double (&d)[5], const double (&u)[5],
                                                     const double (&un)[5], int do_cfl, double dt) {
    // sources in the order of the reference's coupled step
    // (scripts/run_sn50_fiducial.jl:772-781): point masses, self-gravity, sinks
    if (G.src && G.src->nbh > 0) bh_gravity_add(*G.src, i, j, k, u, d);
    if (G.phi) {
        const auto ph = gmem(G.phi);
        const int ip = min(i + 1, G.nx - 1), im = max(i - 1, 0);
        const int jp = min(j + 1, G.ny - 1), jm = max(j - 1, 0);
        const int kp = min(k + 1, G.nz - 1), km = max(k - 1, 0);
        const double i2x = 0.5 * G.idx, i2y = 0.5 * G.idy, i2z = 0.5 * G.idz;
        const double fxf = ip > im ? i2x : 2.0 * i2x;
        const double fyf = jp > jm ? i2y : 2.0 * i2y;
        const double fzf = kp > km ? i2z : 2.0 * i2z;
        const int64_t row = ((int64_t)k * G.ny + j) * G.nx;
        const double gx = (ph[row + ip] - ph[row + im]) * fxf;
        const double gy = (ph[((int64_t)k * G.ny + jp) * G.nx + i] -
                           ph[((int64_t)k * G.ny + jm) * G.nx + i]) * fyf;
        const double gz = (ph[((int64_t)kp * G.ny + j) * G.nx + i] -
                           ph[((int64_t)km * G.ny + j) * G.nx + i]) * fzf;
        const double r = u[0];
        const double vdotg = (u[1] * gx + u[2] * gy + u[3] * gz) / r;
        d[1] -= r * gx;
        d[2] -= r * gy;
        d[3] -= r * gz;
        d[4] -= r * vdotg;
    }
    if (G.src && G.src->nsink > 0) sink_add(*G.src, i, j, k, u, d);
    double v[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        // the split form combines with FMA (one rounding per term)
        if (FAST) {
            if (stage == 1)      v[q] = __builtin_fma(dt, d[q], un[q]);
            else if (stage == 2) v[q] = __builtin_fma(0.25 * dt, d[q], __builtin_fma(0.25, u[q], 0.75 * un[q]));
            else                 v[q] = __builtin_fma((2.0 / 3.0) * dt, d[q],
                                                      __builtin_fma(2.0 / 3.0, u[q], (1.0 / 3.0) * un[q]));
        } else {
            if (stage == 1)      v[q] = un[q] + dt * d[q];
            else if (stage == 2) v[q] = 0.75 * un[q] + 0.25 * u[q] + (0.25 * dt) * d[q];
            else                 v[q] = (1.0 / 3.0) * un[q] + (2.0 / 3.0) * u[q] + ((2.0 / 3.0) * dt) * d[q];
        }
    }
    apply_floor<FAST>(v, G.rho_floor, G.P_floor, G.gamma);
    // streaming stores: the new state is not read again by this kernel
    // (measured 1.5% faster at 256^3 than cached stores; nontemporal loads of
    // the x and y fluxes were 7% slower and are not used)
    // plane NG + k as the base, the cell's place in it as the offset
    double* const ob = G.Uout + (int64_t)(NG + k) * G.Ny * G.pitch;
    const uint32_t oo = (uint32_t)uidx(G, NG + i, NG + j, 0) * (uint32_t)sizeof(double);
#pragma unroll
    for (int q = 0; q < 5; ++q) __builtin_nontemporal_store(v[q], at_off(ob + q * G.fs, oo));
    return do_cfl ? cfl_speed_bits<FAST>(v, G) : 0;
}

template <typename T, int KZ>
__global__ __launch_bounds__(256) void k_update(const GridDev* __restrict__ grids,
                                                const Tile* __restrict__ tiles, int ntiles,
                                                int stage, int do_cfl, double* __restrict__ dU_out) {
    int t0, t1;
    chunk(ntiles, t0, t1);
    const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
    for (int t = t0; t < t1; ++t) {
        const Tile tl = tiles[t];
        const GridDev& G = grids[tl.g];
        const int i = tl.a + lx, j = tl.b + ly;
        uint64_t smax = 0;
        if (i < G.nx && j < G.ny) {
            const auto Fx = gmem((const T*)G.F[0]);
            const auto Fy = gmem((const T*)G.F[1]);
            const auto Fz = gmem((const T*)G.F[2]);
            const int kend = min(tl.c + KZ, G.nz);
            const double dt = stage != 0 ? G.scal[SCAL_DT] : 0.0;
            double fz0[5];
            {
                const int64_t o = ((int64_t)tl.c * G.ny + j) * G.fp[2] + i;
#pragma unroll
                for (int q = 0; q < 5; ++q) fz0[q] = (double)Fz[q * G.ffs[2] + o];
            }
            for (int k = tl.c; k < kend; ++k) {
                const int64_t ox = ((int64_t)k * G.ny + j) * G.fp[0] + i;
                const int64_t oy = ((int64_t)k * (G.ny + 1) + j) * G.fp[1] + i;
                const int64_t oz = ((int64_t)(k + 1) * G.ny + j) * G.fp[2] + i;
                const int64_t c = uidx(G, NG + i, NG + j, NG + k);
                // the cell's state is loaded with its fluxes: one round trip
                // to HBM per cell
                double u[5], un[5];
                if (stage != 0) cell_state<sizeof(T) == 4>(G, c, stage, u, un);
                double d[5], fz1[5];
#pragma unroll
                for (int q = 0; q < 5; ++q) {
                    const double fx0 = (double)Fx[q * G.ffs[0] + ox];
                    const double fx1 = (double)Fx[q * G.ffs[0] + ox + 1];
                    const double fy0 = (double)Fy[q * G.ffs[1] + oy];
                    const double fy1 = (double)Fy[q * G.ffs[1] + oy + G.fp[1]];
                    fz1[q] = (double)Fz[q * G.ffs[2] + oz];
                    // src/gpu_kernels.jl:165-167
                    d[q] = flux_div<sizeof(T) == 4>(fx0, fx1, fy0, fy1, fz0[q], fz1[q], G);
                }
                if (stage == 0) {
#pragma unroll
                    for (int q = 0; q < 5; ++q) dU_out[q * G.fs + c] = d[q];
                } else {
                    const uint64_t b =
                        finish_cell_with<sizeof(T) == 4>(G, i, j, k, stage, d, u, un, do_cfl, dt);
                    smax = b > smax ? b : smax;
                }
#pragma unroll
                for (int q = 0; q < 5; ++q) fz0[q] = fz1[q];
            }
        }
        if (do_cfl) block_max_to(smax, (unsigned long long*)&G.scal[SCAL_SMAX]);
    }
}

// z sweep fused with the stage update.  Tile (g, i0, j0, k0 | len): 64 x 4
// threads over (i, j); each thread walks its z column from k0 for len cells with a
// six-cell register window, computes the z interface fluxes in order and
// finishes every cell as soon as both of its z faces are known, reading the
// x and y fluxes from HBM.  The z fluxes never leave registers.  The stage
// writes Uout != U, so columns can be walked in any order.
//   PF:   1 = the next window cell and the update operands are loaded before
//         the flux arithmetic (latency overlap, more registers); 2 = only the
//         next window cell is;
//   WB:   minimum waves per SIMD the register allocation must allow;
//   RING: the raw FP64 values of the last four window cells stay in a
//         per-thread LDS ring, so the update reads the cell's own state (and,
//         when Un is the stage input, its base state) from LDS instead of
//         fetching it from HBM a second time.
template <typename T, int PF, int WB, int RING>
__global__ __launch_bounds__(256, WB) void k_zupdate(const GridDev* __restrict__ grids,
                                                     const Tile* __restrict__ tiles, int ntiles,
                                                     int stage, int do_cfl) {
    constexpr bool FAST = sizeof(T) == 4;        // split form
    // the FP64 carry (60 VGPRs) does not fit beside the update's operands in 2
    // waves per SIMD: with it, spilled, the 192^3 step took 5.52 ms against 5.34
    constexpr bool CARRY = FAST;
    __shared__ double ring[RING ? 4 : 1][5][RING ? 256 : 1];
    const int rt = RING ? (int)threadIdx.x : 0;
    int t0, t1;
    chunk(ntiles, t0, t1);
    for (int t = t0; t < t1; ++t) {
        const Tile tl = tiles[t];
        const GridDev& G = grids[tl.g];
        // tile.c packs the first cell k0 (bits 0-20) and the column length (bits 21-30)
        const int k0 = tl.c & ZT_K0_MASK, klen = tl.c >> ZT_LEN_SHIFT;
        int i, j, j0;
        col_lane(col_width(G.nx, FAST), tl.a, tl.b, i, j, j0);
        uint64_t smax = 0;
        if (i < G.nx && j < G.ny) {
            const int kend = min(k0 + klen, G.nz);
            const double dt = G.scal[SCAL_DT];
            T c[4][6], p[6];
            // interface f (between active cells f-1 and f) uses padded z = f .. f+5
            const int64_t col = uidx(G, NG + i, NG + j, 0);
            const int64_t zs = (int64_t)G.Ny * G.pitch;
            // every access below is a uniform base (field, z plane) plus the
            // lane's byte offset in the plane
            const uint32_t uo = (uint32_t)col * (uint32_t)sizeof(double);
            const uint32_t fxo = (uint32_t)(j * G.fp[0] + i) * (uint32_t)sizeof(T);
            const uint32_t fyo = (uint32_t)(j * G.fp[1] + i) * (uint32_t)sizeof(T);
            double nxt[5];
            int npz = 0;
            bool big = Prec<T>::big_gamma(G.gamma);
            // the z window and the base state are read once per launch:
            // streaming loads (2.7 % on this kernel at 256^3 against cached
            // loads; the x and y fluxes, whose faces neighbouring lanes and
            // rows share, stay cached)
            auto load = [&](int pz, double (&v)[5]) {
                // load_cell along z: a ghost plane reads the active plane its
                // index maps to; without the ring an active cell is floored here
                const int sk = (G.lmode & 1) ? bc_src(pz, G.nz, G.bc & 4) : pz;
                const double* const b = G.U + sk * zs;
#pragma unroll
                for (int q = 0; q < 5; ++q) v[q] = bld<double, true>(b + q * G.fs, uo);
                if (!RING && (G.lmode & 2) && pz >= NG && pz < NG + G.nz)
                    apply_floor<FAST>(v, G.rho_floor, G.P_floor, G.gamma);
            };
            auto fetch = [&](int pz) { npz = pz; load(pz, nxt); };
            auto place = [&](int slot, int pz, double (&v)[5]) {
                if (RING) {
                    // raw value (unfloored) into the ring; slot pz & 3 is not
                    // read again before cell pz + 4 replaces it
#pragma unroll
                    for (int q = 0; q < 5; ++q) ring[pz & 3][q][rt] = v[q];
                    if ((G.lmode & 2) && pz >= NG && pz < NG + G.nz)
                        apply_floor<FAST>(v, G.rho_floor, G.P_floor, G.gamma);
                }
                const double pr = Prec<T>::pressure(v, G.gamma);
                big |= __ballot(Prec<T>::big_cell(v, pr)) != 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) c[q][slot] = (T)v[q];
                p[slot] = (T)pr;
            };
            T fx[2][5], fy[2][5];
            double u[5], un[5];
            // the operands of the update of active cell k
            auto operands = [&](int k) {
                const T* const xb = (const T*)G.F[0] + (int64_t)k * G.ny * G.fp[0];
                const T* const yb = (const T*)G.F[1] + (int64_t)k * (G.ny + 1) * G.fp[1];
#pragma unroll
                for (int q = 0; q < 5; ++q) {
                    fx[0][q] = bld(xb + q * G.ffs[0], fxo);
                    fx[1][q] = bld(xb + q * G.ffs[0] + 1, fxo);
                    fy[0][q] = bld(yb + q * G.ffs[1], fyo);
                    fy[1][q] = bld(yb + q * G.ffs[1] + G.fp[1], fyo);
                }
                const int64_t cc = col + (int64_t)(NG + k) * zs;
                if (RING) {
                    const int sl = (NG + k) & 3;
                    const bool un_in_ring = G.Un == G.U;
                    const bool need_u = stage > 1 || G.phi != nullptr || G.src != nullptr;
                    const double* const nb = G.Un + (NG + k) * zs;
#pragma unroll
                    for (int q = 0; q < 5; ++q) {
                        const double r = ring[sl][q][rt];
                        u[q] = r;
                        un[q] = un_in_ring ? r : bld<double, true>(nb + q * G.fs, uo);
                    }
                    if (need_u && (G.lmode & 2)) apply_floor<FAST>(u, G.rho_floor, G.P_floor, G.gamma);
                } else {
                    cell_state<FAST>(G, cc, stage, u, un);
                }
            };
            {
                // the window's cells in one memory round trip
                double v[5][5];
#pragma unroll
                for (int m = 0; m < 5; ++m) load(k0 + m, v[m]);
                fetch(k0 + 5);
#pragma unroll
                for (int m = 0; m < 5; ++m) place(m, k0 + m, v[m]);
            }
            // split form: the smoothness indicators that consecutive
            // interfaces share are carried along the column
            typename Prec<T>::Carry wc[5];
            if constexpr (CARRY) Prec<T>::start(c, p, wc);
            T fz0[5];                                   // the previous interface's z flux
            for (int f = k0; f <= kend; ++f) {
                place(5, npz, nxt);                     // cell f+5
                if (PF >= 1 && f < kend) fetch(f + 6);  // next iteration's cell, in flight during the flux
                const int k = f - 1;                    // the cell finished in this iteration
                if (PF == 1 && f > k0) operands(k);
                T F[5];
                Prec<T>::template flux<2, CARRY>(c, p, G, big, F, wc);
                if (G.nzkeep > 0) {
                    // an interface the flux registers read: store it as the
                    // z-flux sweep would (adjacent tiles both compute their
                    // shared interface and store the same values)
                    bool keep = false;
                    for (int n = 0; n < G.nzkeep; ++n) keep |= G.zkeep[n] == f;
                    if (keep) {
                        const auto Fz = gmem((T*)G.F[2]);
                        const int64_t oz = ((int64_t)f * G.ny + j) * G.fp[2] + i;
#pragma unroll
                        for (int q = 0; q < 5; ++q) Fz[q * G.ffs[2] + oz] = F[q];
                    }
                }
                if (PF == 0 && f < kend) fetch(f + 6);
                if (PF != 1 && f > k0) operands(k);
                if (f > k0) {
                    double d[5];
#pragma unroll
                    for (int q = 0; q < 5; ++q)
                        d[q] = flux_div<FAST>(fx[0][q], fx[1][q], fy[0][q], fy[1][q], fz0[q], F[q], G);
                    const uint64_t b = finish_cell_with<FAST>(G, i, j, k, stage, d, u, un, do_cfl, dt);
                    smax = b > smax ? b : smax;
                }
#pragma unroll
                for (int q = 0; q < 5; ++q) fz0[q] = F[q];
#pragma unroll
                for (int m = 0; m < 5; ++m) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[q][m] = c[q][m + 1];
                    p[m] = p[m + 1];
                }
            }
        }
        if (do_cfl) block_max_to(smax, (unsigned long long*)&G.scal[SCAL_SMAX]);
    }
}

// Stand-alone CFL maximum over active cells (cfl_dt_3d, euler3d.jl:157-169).
template <int KZ>
__global__ __launch_bounds__(256) void k_cfl(const GridDev* __restrict__ grids,
                                             const Tile* __restrict__ tiles, int ntiles) {
    int t0, t1;
    chunk(ntiles, t0, t1);
    const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
    uint64_t smax = 0;
    for (int t = t0; t < t1; ++t) {
        const Tile tl = tiles[t];
        const GridDev& G = grids[tl.g];
        const int i = tl.a + lx, j = tl.b + ly;
        if (i < G.nx && j < G.ny) {
            // several cells' loads in flight (cells past the grid repeat its
            // last).  Bound by memory: 256^3 in 115 us, 5.9 TB/s; 150 with a
            // reduction and an atomic per tile, 171 also one cell after the other.
            constexpr int M = KZ < 4 ? KZ : 4;
            const int kend = min(tl.c + KZ, G.nz);
            for (int k = tl.c; k < kend; k += M) {
                double u[M][5];
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const int64_t c = uidx(G, NG + i, NG + j, NG + min(k + m, G.nz - 1));
#pragma unroll
                    for (int q = 0; q < 5; ++q) u[m][q] = __builtin_nontemporal_load(&gmem(G.U)[q * G.fs + c]);
                }
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const uint64_t b = cfl_speed_bits(u[m], G);
                    smax = b > smax ? b : smax;
                }
            }
        }
        // one reduction and one atomic per grid and workgroup
        if (t + 1 == t1 || tiles[t + 1].g != tl.g) {
            block_max_to(smax, (unsigned long long*)&G.scal[SCAL_SMAX]);
            smax = 0;
        }
    }
}

// dt = cfl / smax (Inf when smax is not > 0), optionally clipped to t_end - t;
// the maximum is reset for the next accumulation.
__device__ __forceinline__ double take_dt(double* s) {
    const uint64_t bits = *(const uint64_t*)&s[SCAL_SMAX];
    const double smax = __longlong_as_double((long long)bits);
    double dt = smax > 0.0 ? s[SCAL_CFL] / smax : __builtin_inf();
    if (s[SCAL_TEND] > 0.0) dt = jl_min(dt, s[SCAL_TEND] - s[SCAL_T]);
    s[SCAL_DT] = dt;
    *(uint64_t*)&s[SCAL_SMAX] = 0;
    return dt;
}

__global__ void k_dt(const GridDev* __restrict__ grids, int ngrids, double* __restrict__ out) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ngrids) return;
    const double dt = take_dt(grids[g].scal);
    if (out) out[g] = dt;
}

// The dts of a hierarchy's levels, then dt_root = min(dt_root, r0 dt_1, r0 r1 dt_2, ...)
// (cfl_dt_fmr3d, fmr3d.jl:615-622; factor[l] the ratios' product up to level l).
__global__ void k_fmr_dt(const GridDev* __restrict__ grids, FmrFactors f) {
    double* root = grids[0].scal;
    double dt = take_dt(root);
    for (int l = 1; l < f.nlev; ++l) dt = jl_min(dt, take_dt(grids[l].scal) * f.factor[l]);
    root[SCAL_DT] = dt;
}

// Start of a CFL accumulation: CFL number, end time and an empty maximum; restart
// also sets t = 0.  One launch for all grids: three per grid were 0.6 of the 14 ms of
// two steps of 48 problems.
__global__ void k_cfl_begin(const GridDev* __restrict__ grids, int ngrids, double cfl, double t_end, int restart) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ngrids) return;
    double* s = grids[g].scal;
    s[SCAL_CFL] = cfl;
    s[SCAL_TEND] = t_end;
    *(uint64_t*)&s[SCAL_SMAX] = 0;
    if (restart) s[SCAL_T] = 0.0;
}

__global__ void k_set_scal(double* scal, int idx, double v) { scal[idx] = v; }

__global__ void k_fill_u64(uint64_t* p, int64_t n, uint64_t v) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        p[e] = v;
}

// ---------------------------------------------------------------------------
// Layout conversion between the reference's (5, Nx, Ny, Nz) column-major
// array and the device layout.  dst/src select the device buffer (U, Un or
// any buffer with U's layout).

__global__ void k_aos_to_soa(GridDev G, const double* __restrict__ aos, double* __restrict__ dst) {
    const int Nx = G.nx + 2 * NG;
    const int64_t n = (int64_t)Nx * G.Ny * G.Nz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % Nx);
        const int64_t r = e / Nx;
        const int j = (int)(r % G.Ny), k = (int)(r / G.Ny);
        const int64_t c = uidx(G, i, j, k);
#pragma unroll
        for (int q = 0; q < 5; ++q) dst[q * G.fs + c] = aos[5 * e + q];
    }
}

__global__ void k_soa_to_aos(GridDev G, const double* __restrict__ src, double* __restrict__ aos) {
    const int Nx = G.nx + 2 * NG;
    const int64_t n = (int64_t)Nx * G.Ny * G.Nz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % Nx);
        const int64_t r = e / Nx;
        const int j = (int)(r % G.Ny), k = (int)(r / G.Ny);
        const int64_t c = uidx(G, i, j, k);
#pragma unroll
        for (int q = 0; q < 5; ++q) aos[5 * e + q] = src[q * G.fs + c];
    }
}

// Fluxes to the reference's F? arrays (zero outside the active-range
// interfaces, as after euler3d.jl:197-202).  Shapes: Fx (5, Nx+1, Ny, Nz),
// Fy (5, Nx, Ny+1, Nz), Fz (5, Nx, Ny, Nz+1).
template <typename T>
__global__ void k_flux_export(GridDev G, int dir, double* __restrict__ out) {
    const int Nx = G.nx + 2 * NG;
    const int Ex = Nx + (dir == 0), Ey = G.Ny + (dir == 1), Ez = G.Nz + (dir == 2);
    const int64_t n = (int64_t)Ex * Ey * Ez;
    const T* F = (const T*)G.F[dir];
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int a = (int)(e % Ex);
        const int64_t r = e / Ex;
        const int b = (int)(r % Ey), c = (int)(r / Ey);
        // reference 0-based index of interface f is NG - 1 + f along dir
        int f = -1, ci = -1, cj = -1;
        bool in;
        if (dir == 0) { f = a - (NG - 1); ci = b - NG; cj = c - NG;
                        in = f >= 0 && f <= G.nx && ci >= 0 && ci < G.ny && cj >= 0 && cj < G.nz; }
        else if (dir == 1) { f = b - (NG - 1); ci = a - NG; cj = c - NG;
                        in = f >= 0 && f <= G.ny && ci >= 0 && ci < G.nx && cj >= 0 && cj < G.nz; }
        else { f = c - (NG - 1); ci = a - NG; cj = b - NG;
               in = f >= 0 && f <= G.nz && ci >= 0 && ci < G.nx && cj >= 0 && cj < G.ny; }
        int64_t o = 0;
        if (in) {
            if (dir == 0)      o = ((int64_t)cj * G.ny + ci) * G.fp[0] + f;
            else if (dir == 1) o = ((int64_t)cj * (G.ny + 1) + f) * G.fp[1] + ci;
            else               o = ((int64_t)f * G.ny + cj) * G.fp[2] + ci;
        }
#pragma unroll
        for (int q = 0; q < 5; ++q) out[5 * e + q] = in ? (double)F[q * G.ffs[dir] + o] : 0.0;
    }
}

// Phi source on a dU buffer with U's layout (_apply_sg_force_level!,
// fmr_gravity.jl:146-156 -> gpu_kernels.jl:291-319).
__global__ void k_sg_force(GridDev G, double* __restrict__ dU) {
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % G.nx);
        const int64_t r = e / G.nx;
        const int j = (int)(r % G.ny), k = (int)(r / G.ny);
        const int64_t c = uidx(G, NG + i, NG + j, NG + k);
        const double* ph = G.phi;
        const int ip = min(i + 1, G.nx - 1), im = max(i - 1, 0);
        const int jp = min(j + 1, G.ny - 1), jm = max(j - 1, 0);
        const int kp = min(k + 1, G.nz - 1), km = max(k - 1, 0);
        const double i2x = 0.5 * G.idx, i2y = 0.5 * G.idy, i2z = 0.5 * G.idz;
        const double fxf = ip > im ? i2x : 2.0 * i2x;
        const double fyf = jp > jm ? i2y : 2.0 * i2y;
        const double fzf = kp > km ? i2z : 2.0 * i2z;
        const double gx = (ph[((int64_t)k * G.ny + j) * G.nx + ip] - ph[((int64_t)k * G.ny + j) * G.nx + im]) * fxf;
        const double gy = (ph[((int64_t)k * G.ny + jp) * G.nx + i] - ph[((int64_t)k * G.ny + jm) * G.nx + i]) * fyf;
        const double gz = (ph[((int64_t)kp * G.ny + j) * G.nx + i] - ph[((int64_t)km * G.ny + j) * G.nx + i]) * fzf;
        const double rr = G.U[c], mx = G.U[G.fs + c], my = G.U[2 * G.fs + c], mz = G.U[3 * G.fs + c];
        const double vdotg = (mx * gx + my * gy + mz * gz) / rr;
        dU[G.fs + c] -= rr * gx;
        dU[2 * G.fs + c] -= rr * gy;
        dU[3 * G.fs + c] -= rr * gz;
        dU[4 * G.fs + c] -= rr * vdotg;
    }
}

// Point-mass gravity (which = 0) or sink (which = 1) source on a dU buffer
// with U's layout, from the grid's state (add_bh_gravity_source!,
// src/gravity_bh.jl:58-78; add_sink_sources!, src/sinks.jl:32-58).
__global__ void k_src(GridDev G, double* __restrict__ dU, int which) {
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % G.nx);
        const int64_t r = e / G.nx;
        const int j = (int)(r % G.ny), k = (int)(r / G.ny);
        const int64_t c = uidx(G, NG + i, NG + j, NG + k);
        double u[5], d[5];
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            u[q] = G.U[q * G.fs + c];
            d[q] = dU[q * G.fs + c];
        }
        if (which == 0) bh_gravity_add(*G.src, i, j, k, u, d);
        else            sink_add(*G.src, i, j, k, u, d);
#pragma unroll
        for (int q = 0; q < 5; ++q) dU[q * G.fs + c] = d[q];
    }
}

// Whole-array RK3 combine with a caller-supplied dU in U's layout
// (rk3.jl:24,28,32 / euler3d.jl:244,250,256), over every padded cell.
__global__ void k_combine_all(GridDev G, int stage, const double* __restrict__ dU, double dt) {
    const int Nx = G.nx + 2 * NG;
    const int64_t n = (int64_t)Nx * G.Ny * G.Nz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % Nx);
        const int64_t r = e / Nx;
        const int j = (int)(r % G.Ny), k = (int)(r / G.Ny);
        const int64_t c = uidx(G, i, j, k);
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const double un = G.Un[q * G.fs + c], u = G.U[q * G.fs + c], d = dU[q * G.fs + c];
            double v;
            if (stage == 1)      v = un + dt * d;
            else if (stage == 2) v = 0.75 * un + 0.25 * u + (0.25 * dt) * d;
            else                 v = (1.0 / 3.0) * un + (2.0 / 3.0) * u + ((2.0 / 3.0) * dt) * d;
            G.U[q * G.fs + c] = v;
        }
    }
}

// Copy every padded cell of src into dst (both with U's layout).
__global__ void k_copy_state(GridDev G, const double* __restrict__ src, double* __restrict__ dst) {
    const int64_t n = 5 * G.fs;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        dst[e] = src[e];
}

// Conservation totals: per-block partial sums over active cells, then a
// fixed-order final sum (deterministic for a fixed launch shape).
__global__ void k_totals_partial(GridDev G, double* __restrict__ part) {
    __shared__ double red[5][256];
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    double acc[5] = {0, 0, 0, 0, 0};
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % G.nx);
        const int64_t r = e / G.nx;
        const int j = (int)(r % G.ny), k = (int)(r / G.ny);
        const int64_t c = uidx(G, NG + i, NG + j, NG + k);
#pragma unroll
        for (int q = 0; q < 5; ++q) acc[q] += G.U[q * G.fs + c];
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) red[q][threadIdx.x] = acc[q];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
#pragma unroll
            for (int q = 0; q < 5; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < 5; ++q) part[5 * blockIdx.x + q] = red[q][0];
}

__global__ void k_totals_final(const double* __restrict__ part, int nblocks, double dV,
                               double* __restrict__ out) {
    const int q = threadIdx.x;
    if (q >= 5) return;
    double s = 0.0;
    for (int b = 0; b < nblocks; ++b) s += part[5 * b + q];
    out[q] = s * dV;
}

// ---------------------------------------------------------------------------
// FMR transfer operators (src/fmr3d.jl).  Fine active cell a (0-based) of a box
// that starts at coarse cell lo has the stencil centre lo + floor(a / ratio) and
// the weights of a mod ratio: what _coarse_stencil (fmr3d.jl:165-170) computes
// in FP64, where no centre is nearer than 1 / (2 ratio) to a tie.

// Fine cells of one axis, 0-based from the first active one, in groups of at most
// two that share a coarse centre: cells a0 .. a1 - 1, coarse cells from c0.
struct FineAxis {
    int a0, a1, c0, p;           // p: groups of a coarse cell
};

__device__ __forceinline__ FineAxis fine_axis(int n, bool ghosts, int r) {
    FineAxis x;
    x.a0 = ghosts ? -NG : 0;
    x.a1 = n + (ghosts ? NG : 0);
    x.c0 = x.a0 < 0 ? -((r - 1 - x.a0) / r) : 0;
    x.p = (r + 1) / 2;
    return x;
}

// Prolongation of up to NX x NY x NZ fine cells around one coarse centre, whose
// 125 coarse values src (at the stencil's first cell; sx, sy, sz: strides, fs:
// field stride) serve them all.  w?: the Lagrange weights of each axis's first
// cell, those of a second one 5 on.  Each cell and field sums its terms in the
// reference's (di, dj, dk) order.  The next 25 values are in flight while the
// last 25 are summed.
template <int NX, int NY, int NZ, typename Put>
__device__ __forceinline__ void prolong_cells(const double* __restrict__ src, int64_t sx, int64_t sy,
                                              int64_t sz, int64_t fs, const double* wx, const double* wy,
                                              const double* wz, Put&& put) {
    double val[NX][NY][NZ][5] = {};
    double nxt[5][5], wi[NX], wj[NY], wk[NZ][5];
    auto load = [&](int di, int dj) {
        const double* b = src + di * sx + dj * sy;
#pragma unroll
        for (int dk = 0; dk < 5; ++dk)
#pragma unroll
            for (int q = 0; q < 5; ++q) nxt[dk][q] = b[dk * sz + q * fs];
#pragma unroll
        for (int x = 0; x < NX; ++x) wi[x] = wx[5 * x + di];
#pragma unroll
        for (int y = 0; y < NY; ++y) wj[y] = wy[5 * y + dj];
    };
#pragma unroll
    for (int z = 0; z < NZ; ++z)
#pragma unroll
        for (int dk = 0; dk < 5; ++dk) wk[z][dk] = wz[5 * z + dk];
    load(0, 0);
    int di = 0, dj = 0;
#pragma unroll 1
    for (int m = 0; m < 25; ++m) {
        double cur[5][5], wij[NX][NY];
#pragma unroll
        for (int dk = 0; dk < 5; ++dk)
#pragma unroll
            for (int q = 0; q < 5; ++q) cur[dk][q] = nxt[dk][q];
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int y = 0; y < NY; ++y) wij[x][y] = wi[x] * wj[y];
        if (++dj == 5) { dj = 0; ++di; }
        if (m < 24) load(di, dj);
#pragma unroll
        for (int dk = 0; dk < 5; ++dk)
#pragma unroll
            for (int x = 0; x < NX; ++x)
#pragma unroll
                for (int y = 0; y < NY; ++y)
#pragma unroll
                    for (int z = 0; z < NZ; ++z) {
                        const double w = wij[x][y] * wk[z][dk];
#pragma unroll
                        for (int q = 0; q < 5; ++q) val[x][y][z][q] += w * cur[dk][q];
                    }
    }
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y)
#pragma unroll
            for (int z = 0; z < NZ; ++z) put(x, y, z, val[x][y][z]);
}

// Prolongation of fine cells from the parent state Uca (fmr3d.jl:551: the one
// interpolated in time).  all_cells = 1 fills every fine cell (_prolong_all!),
// else only ghost cells in the reference's slab partition.  The values go to
// each of the dst.n buffers in the child's layout, or to the child's state when
// dst.n is 0.
//
// Bound by the 625 coarse values a cell gathers through L1 and L2: a thread takes
// the 2 x 2 fine cells in its slab's plane that share a coarse centre, for a
// quarter of the loads, and no wave takes cells of two slabs (it would run
// both).  A child of 128 x 128 x 96 took 100 us per call cell for cell, 71 with waves
// that mix slabs, now 62; with 1 x 2 cells 77 (twice the loads).
__global__ __launch_bounds__(64) void k_prolong(const GridDev* __restrict__ grids, const FmrDev* __restrict__ fmr,
                                                const double* __restrict__ Uca, const double* __restrict__ Ucat,
                                                int all_cells, ProlongDst dst) {
    const FmrDev& M = *fmr;
    const GridDev& C = grids[M.parent];
    const GridDev& Fg = grids[M.child];
    const int r = M.ratio;
    const ProlongWork W = prolong_work(Fg.nx, Fg.ny, Fg.nz, all_cells, r);
    const FineAxis X = fine_axis(Fg.nx, all_cells, r), Yg = fine_axis(Fg.ny, true, r);
    const FineAxis Y = fine_axis(Fg.ny, all_cells, r), Zg = fine_axis(Fg.nz, true, r);
    const int64_t zs = (int64_t)C.Ny * C.pitch;
    // the coarse cell and the weights of fine cell a (a >= -NG)
    auto centre = [&](int a, int& c, const double*& w) {
        c = (a + NG * r) / r - NG;
        w = M.w + 5 * (a - c * r);
    };
    auto group = [&](const FineAxis& x, int g, int& c, int& a, const double*& w) {
        c = x.c0 + g / x.p;
        a = c * r + 2 * (g % x.p);
        w = M.w + 5 * (a - c * r);
    };
    auto in = [&](const FineAxis& x, int a, int c) { return a >= x.a0 && a < min(x.a1, (c + 1) * r); };
    auto ghost = [](int l, int n) { return l < NG ? l - NG : n + l - NG; };
    auto store = [&](int i, int j, int k, const double (&v)[5]) {
        const int64_t d = uidx(Fg, NG + i, NG + j, NG + k);
        if (dst.n == 0) {
#pragma unroll
            for (int q = 0; q < 5; ++q) Fg.U[q * Fg.fs + d] = v[q];
        }
        for (int b = 0; b < dst.n; ++b) {
#pragma unroll
            for (int q = 0; q < 5; ++q) dst.p[b][q * Fg.fs + d] = v[q];
        }
    };
    // the stencil's first cell (padded, 0-based) in the parent
    auto first = [&](int a, int c) { return NG + M.lo[a] + c - 3; };
    for (int64_t blk = blockIdx.x; blk < W.bx + W.by + W.bz; blk += gridDim.x) {
        int cx, cy, cz, i, j, k;
        const double *wx, *wy, *wz;
        if (blk < W.bx) {
            // x slabs: lanes along y, from the transposed box, when there is
            // one, where consecutive y cells are adjacent
            const int64_t e = blk * 64 + threadIdx.x;
            if (e >= W.nx) continue;
            const uint32_t u = (uint32_t)e, t = u / (uint32_t)W.gyg;
            group(Yg, (int)(u % (uint32_t)W.gyg), cy, j, wy);
            group(Zg, (int)(t % (uint32_t)W.gzg), cz, k, wz);
            i = ghost((int)(t / (uint32_t)W.gzg), Fg.nx);
            centre(i, cx, wx);
            const int pi = first(0, cx), pj = first(1, cy), pk = first(2, cz);
            const double* src = Uca + uidx(C, pi, pj, pk);
            int64_t sx = 1, sy = C.pitch, sz = zs, fs = C.fs;
            if (Ucat) {
                sy = 1;
                sz = M.phi[1] - M.plo[1] + 1;
                sx = sz * (M.phi[2] - M.plo[2] + 1);
                fs = sx * (M.phi[0] - M.plo[0] + 1);
                src = Ucat + (pi - M.plo[0]) * sx + (pk - M.plo[2]) * sz + (pj - M.plo[1]);
            }
            prolong_cells<1, 2, 2>(src, sx, sy, sz, fs, wx, wy, wz, [&](int, int y, int z, const double (&v)[5]) {
                if (in(Yg, j + y, cy) && in(Zg, k + z, cz)) store(i, j + y, k + z, v);
            });
        } else if (blk < W.bx + W.by) {
            const int64_t e = (blk - W.bx) * 64 + threadIdx.x;
            if (e >= W.ny) continue;
            const uint32_t u = (uint32_t)e, t = u / (uint32_t)W.gx;
            group(X, (int)(u % (uint32_t)W.gx), cx, i, wx);
            j = ghost((int)(t % (2 * NG)), Fg.ny);
            centre(j, cy, wy);
            group(Zg, (int)(t / (2 * NG)), cz, k, wz);
            prolong_cells<2, 1, 2>(Uca + uidx(C, first(0, cx), first(1, cy), first(2, cz)), 1, C.pitch, zs, C.fs,
                                   wx, wy, wz, [&](int x, int, int z, const double (&v)[5]) {
                if (in(X, i + x, cx) && in(Zg, k + z, cz)) store(i + x, j, k + z, v);
            });
        } else {
            const int64_t e = (blk - W.bx - W.by) * 64 + threadIdx.x;
            if (e >= W.nz) continue;
            const uint32_t u = (uint32_t)e, t = u / (uint32_t)W.gx;
            group(X, (int)(u % (uint32_t)W.gx), cx, i, wx);
            group(Y, (int)(t % (uint32_t)W.gy), cy, j, wy);
            k = all_cells ? (int)(t / (uint32_t)W.gy) - NG : ghost((int)(t / (uint32_t)W.gy), Fg.nz);
            centre(k, cz, wz);
            prolong_cells<2, 2, 1>(Uca + uidx(C, first(0, cx), first(1, cy), first(2, cz)), 1, C.pitch, zs, C.fs,
                                   wx, wy, wz, [&](int x, int y, int, const double (&v)[5]) {
                if (in(X, i + x, cx) && in(Y, j + y, cy)) store(i + x, j + y, k, v);
            });
        }
    }
}

__device__ __forceinline__ bool in_shell(const FmrDev& M, int axis, int p) {
    return p <= M.slo[axis] || p >= M.shi[axis];
}

// U_c_interp = (1 - alpha) * U_c_n + alpha * U_c_np1 (fmr3d.jl:547-551) over
// the parent cells the child's ghost stencils read, once per fine sub-cycle
// (alpha is fixed for its three stages): the x slabs read the transposed copy,
// the others the plain one, none the inside of the box.
__global__ void k_time_interp(const GridDev* __restrict__ grids, const FmrDev* __restrict__ fmr,
                              double alpha) {
    const FmrDev& M = *fmr;
    const GridDev& C = grids[M.parent];
    const int nx = M.phi[0] - M.plo[0] + 1, ny = M.phi[1] - M.plo[1] + 1, nz = M.phi[2] - M.plo[2] + 1;
    const int64_t total = (int64_t)nx * ny * nz;
    const double oma = 1.0 - alpha;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = M.plo[0] + (int)(e % nx);
        const int64_t r = e / nx;
        const int j = M.plo[1] + (int)(r % ny), k = M.plo[2] + (int)(r / ny);
        const bool xs = in_shell(M, 0, i), yz = in_shell(M, 1, j) || in_shell(M, 2, k);
        if (!xs && !yz) continue;
        const int64_t o = uidx(C, i, j, k);
        const int64_t ot = ((int64_t)(i - M.plo[0]) * nz + (k - M.plo[2])) * ny + (j - M.plo[1]);
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const double v = oma * M.Ucn[q * C.fs + o] + alpha * M.Ucnp1[q * C.fs + o];
            if (yz) M.Uci[q * C.fs + o] = v;
            if (xs) M.Ucit[q * total + ot] = v;
        }
    }
}

// Start of a level's fused step: its ghost cells, which the stage-3 combination
// reads after the prolongation has replaced them, are saved to Un (a child, own
// != 0); so is what its child's ghost stencils read of the state at the start,
// the child's flux registers are cleared and its dt is set (a parent, fmr != null).  Copying
// the whole state took 258 of 6270 us per root step of three levels from 192^3,
// now 90.
__global__ void k_level_begin(const GridDev* __restrict__ grids, int level, const FmrDev* __restrict__ fmr,
                              int own) {
    const GridDev& G = grids[level];
    // dt_child = dt_parent / ratio (fmr3d.jl:454)
    if (fmr && blockIdx.x == 0 && threadIdx.x == 0)
        grids[fmr->child].scal[SCAL_DT] = G.scal[SCAL_DT] / (double)fmr->ratio;
    int64_t nb = 0, nr = 0;
    int nx = 1, ny = 1;
    if (fmr) {
        nx = fmr->phi[0] - fmr->plo[0] + 1;
        ny = fmr->phi[1] - fmr->plo[1] + 1;
        nb = (int64_t)nx * ny * (fmr->phi[2] - fmr->plo[2] + 1);
        nr = fmr->froff[6];
    }
    const int64_t ng = own ? ghost_count(G) : 0, total = ng + nb + nr;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        if (e >= ng + nb) {
            fmr->frc[e - ng - nb] = 0.0;
            fmr->frf[e - ng - nb] = 0.0;
            continue;
        }
        int i, j, k;
        if (e < ng) {
            ghost_decode(G, e, i, j, k);
        } else {
            const int64_t t = e - ng;
            i = fmr->plo[0] + (int)(t % nx);
            const int64_t r = t / nx;
            j = fmr->plo[1] + (int)(r % ny);
            k = fmr->plo[2] + (int)(r / ny);
            if (!in_shell(*fmr, 0, i) && !in_shell(*fmr, 1, j) && !in_shell(*fmr, 2, k)) continue;
        }
        const int64_t c = uidx(G, i, j, k);
#pragma unroll
        for (int q = 0; q < 5; ++q) G.Un[q * G.fs + c] = G.U[q * G.fs + c];
    }
}

// _restrict! (fmr3d.jl:266-285)
// _restrict! (fields 0..nq-1; nq = 5) and restrict_density_to_coarse!
// (nq = 1, src/fmr_gravity.jl:40-60): the same sum in the same order.
__global__ void k_restrict(const GridDev* __restrict__ grids, const FmrDev* __restrict__ fmr, int nq) {
    const FmrDev& M = *fmr;
    const GridDev& C = grids[M.parent];
    const GridDev& Fg = grids[M.child];
    const int r = M.ratio;
    const int nic = M.hi[0] - M.lo[0] + 1, njc = M.hi[1] - M.lo[1] + 1, nkc = M.hi[2] - M.lo[2] + 1;
    const int64_t total = (int64_t)nic * njc * nkc;
    const double inv_r3 = 1.0 / (double)(r * r * r);
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int m = (int)(e % nic);
        const int64_t rr = e / nic;
        const int n = (int)(rr % njc), p = (int)(rr / njc);
        const int64_t dc = uidx(C, NG + M.lo[0] + m - 1, NG + M.lo[1] + n - 1, NG + M.lo[2] + p - 1);
        for (int q = 0; q < nq; ++q) {
            double val = 0.0;
            for (int sx = 1; sx <= r; ++sx)
                for (int sy = 1; sy <= r; ++sy)
                    for (int sz = 1; sz <= r; ++sz)
                        val += Fg.U[q * Fg.fs + uidx(Fg, NG + r * m + sx - 1, NG + r * n + sy - 1,
                                                     NG + r * p + sz - 1)];
            C.U[q * C.fs + dc] = val * inv_r3;
        }
    }
}

// _prolong_scalar_trilinear! (src/fmr_gravity.jl:70-106): phi of the fine
// active cells (x fastest) from the coarse active-cell phi, the fine box
// starting at coarse active cell (lo_x, lo_y, lo_z) (1-based), in the
// reference's operation order.
__global__ void k_prolong_scalar(const double* __restrict__ phc, int ncx, int ncy, int ncz,
                                 double* __restrict__ phf, int nfx, int nfy, int nfz, int lox,
                                 int loy, int loz, int r) {
    const int64_t total = (int64_t)nfx * nfy * nfz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % nfx);
        const int64_t rr = e / nfx;
        const int j = (int)(rr % nfy), k = (int)(rr / nfy);
        // fine cell centre in coarse active-cell coordinates (1-based)
        const double xc = ((double)(lox - 1) + ((double)(i + 1) - 0.5) / (double)r) + 0.5;
        const double yc = ((double)(loy - 1) + ((double)(j + 1) - 0.5) / (double)r) + 0.5;
        const double zc = ((double)(loz - 1) + ((double)(k + 1) - 0.5) / (double)r) + 0.5;
        const int ic = min(max((int)floor(xc), 1), ncx - 1);
        const int jc = min(max((int)floor(yc), 1), ncy - 1);
        const int kc = min(max((int)floor(zc), 1), ncz - 1);
        const double fx = xc - ic, fy = yc - jc, fz = zc - kc;
        const double w000 = (1 - fx) * (1 - fy) * (1 - fz);
        const double w100 = fx * (1 - fy) * (1 - fz);
        const double w010 = (1 - fx) * fy * (1 - fz);
        const double w110 = fx * fy * (1 - fz);
        const double w001 = (1 - fx) * (1 - fy) * fz;
        const double w101 = fx * (1 - fy) * fz;
        const double w011 = (1 - fx) * fy * fz;
        const double w111 = fx * fy * fz;
        auto P = [&](int a, int b, int c) {
            return phc[((int64_t)(kc - 1 + c) * ncy + (jc - 1 + b)) * ncx + (ic - 1 + a)];
        };
        phf[e] = w000 * P(0, 0, 0) + w100 * P(1, 0, 0) + w010 * P(0, 1, 0) + w110 * P(1, 1, 0) +
                 w001 * P(0, 0, 1) + w101 * P(1, 0, 1) + w011 * P(0, 1, 1) + w111 * P(1, 1, 1);
    }
}

// a .*= s
__global__ void k_scale(double* __restrict__ a, int64_t n, double s) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        a[e] = a[e] * s;
}

// Flux registers: face f in 0..5 = x_lo, x_hi, y_lo, y_hi, z_lo, z_hi, each
// (5, n1, n2) column-major as FluxReg3D (fmr3d.jl:81-96).
__device__ __forceinline__ void face_dims(const FmrDev& M, int face, int& n1, int& n2) {
    const int nic = M.hi[0] - M.lo[0] + 1, njc = M.hi[1] - M.lo[1] + 1, nkc = M.hi[2] - M.lo[2] + 1;
    if (face < 2)      { n1 = njc; n2 = nkc; }
    else if (face < 4) { n1 = nic; n2 = nkc; }
    else               { n1 = nic; n2 = njc; }
}

template <typename T>
__device__ __forceinline__ double flux_at(const GridDev& G, int dir, int q, int f, int a, int b) {
    // dir 0: (f, j=a, k=b); dir 1: (i=a, f, k=b); dir 2: (i=a, j=b, f)
    const T* F = (const T*)G.F[dir];
    int64_t o;
    if (dir == 0)      o = ((int64_t)b * G.ny + a) * G.fp[0] + f;
    else if (dir == 1) o = ((int64_t)b * (G.ny + 1) + f) * G.fp[1] + a;
    else               o = ((int64_t)f * G.ny + b) * G.fp[2] + a;
    return (double)F[q * G.ffs[dir] + o];
}

// _accumulate_fr_coarse! (fmr3d.jl:292-326); fac = weight * dt of the parent.
template <typename T>
__global__ void k_fr_coarse(const GridDev* __restrict__ grids, const FmrDev* __restrict__ fmr,
                            double weight) {
    const int q = blockIdx.y;                   // one field per grid row
    const FmrDev& M = *fmr;
    const GridDev& C = grids[M.parent];
    const double fac = weight * C.scal[SCAL_DT];
    const int64_t n = M.froff[6] / 5;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        int face = 0;
        while (face < 5 && e >= M.froff[face + 1] / 5) ++face;
        const int64_t loc = e - M.froff[face] / 5;
        int n1, n2;
        face_dims(M, face, n1, n2);
        const int a = (int)(loc % n1), b = (int)(loc / n1);
        const int hi = face & 1;
        // reference interface NG + ci_lo - 1 (lo) or NG + ci_hi (hi) is
        // device interface f = ci_lo - 1 or ci_hi (active-cell faces)
        double F;
        if (face < 2)      F = flux_at<T>(C, 0, q, hi ? M.hi[0] : M.lo[0] - 1, M.lo[1] - 1 + a, M.lo[2] - 1 + b);
        else if (face < 4) F = flux_at<T>(C, 1, q, hi ? M.hi[1] : M.lo[1] - 1, M.lo[0] - 1 + a, M.lo[2] - 1 + b);
        else               F = flux_at<T>(C, 2, q, hi ? M.hi[2] : M.lo[2] - 1, M.lo[0] - 1 + a, M.lo[1] - 1 + b);
        double* R = &M.frc[M.froff[face] + q + 5 * loc];
        *R = *R + fac * F;
    }
}

// _accumulate_fr_fine! (fmr3d.jl:331-369): each register element sums its
// r^2 fine faces in the reference's loop order; fac = weight*dt_f/r^2.
template <typename T>
__global__ void k_fr_fine(const GridDev* __restrict__ grids, const FmrDev* __restrict__ fmr,
                          double weight) {
    const int q = blockIdx.y;                   // one field per grid row
    const FmrDev& M = *fmr;
    const GridDev& Fg = grids[M.child];
    const int r = M.ratio;
    const double fac = (weight * Fg.scal[SCAL_DT]) / (double)(r * r);
    const int64_t n = M.froff[6] / 5;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        int face = 0;
        while (face < 5 && e >= M.froff[face + 1] / 5) ++face;
        const int64_t loc = e - M.froff[face] / 5;
        int n1, n2;
        face_dims(M, face, n1, n2);
        const int a = (int)(loc % n1), b = (int)(loc / n1);
        const int hi = face & 1;
        double* R = &M.frf[M.froff[face] + q + 5 * loc];
        double acc = *R;
        // outer loop over the second register index (kf or jf), inner over
        // the first (jf or ia), as the reference
        for (int ob = 0; ob < r; ++ob)
            for (int oa = 0; oa < r; ++oa) {
                const int fa = a * r + oa, fb = b * r + ob;   // 0-based fine active
                double F;
                if (face < 2)      F = flux_at<T>(Fg, 0, q, hi ? Fg.nx : 0, fa, fb);
                else if (face < 4) F = flux_at<T>(Fg, 1, q, hi ? Fg.ny : 0, fa, fb);
                else               F = flux_at<T>(Fg, 2, q, hi ? Fg.nz : 0, fa, fb);
                acc = acc + fac * F;
            }
        *R = acc;
    }
}

// _restrict! (fmr3d.jl:266-285) into the child's box, _bc_correct! (fmr3d.jl:379-422)
// on the cells around it, each of which receives one face's correction, and the
// floors on both: the parent's other cells were floored by the last stage, and a
// floored cell stays as it is under the floors.
__global__ void k_fmr_correct(const GridDev* __restrict__ grids, const FmrDev* __restrict__ fmr) {
    const FmrDev& M = *fmr;
    const GridDev& C = grids[M.parent];
    const GridDev& Fg = grids[M.child];
    const int r = M.ratio;
    int n[3];
    for (int a = 0; a < 3; ++a) n[a] = M.hi[a] - M.lo[a] + 1;
    const int64_t total = (int64_t)(n[0] + 2) * (n[1] + 2) * (n[2] + 2);
    const double inv_r3 = 1.0 / (double)(r * r * r);
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        // position in the box, -1 and n outside it
        const int64_t t = e / (n[0] + 2);
        const int m[3] = {(int)(e % (n[0] + 2)) - 1, (int)(t % (n[1] + 2)) - 1, (int)(t / (n[1] + 2)) - 1};
        int face = -1, outside = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (m[a] < 0 || m[a] == n[a]) { ++outside; face = 2 * a + (m[a] < 0 ? 0 : 1); }
        if (outside > 1) continue;
        const int i = M.lo[0] - 1 + m[0], j = M.lo[1] - 1 + m[1], k = M.lo[2] - 1 + m[2];   // 0-based active
        const int64_t c = uidx(C, NG + i, NG + j, NG + k);
        double u[5];
        if (outside == 0) {
#pragma unroll
            for (int q = 0; q < 5; ++q) u[q] = 0.0;
            for (int sx = 0; sx < r; ++sx)
                for (int sy = 0; sy < r; ++sy)
                    for (int sz = 0; sz < r; ++sz) {
                        const int64_t o = uidx(Fg, NG + r * m[0] + sx, NG + r * m[1] + sy, NG + r * m[2] + sz);
#pragma unroll
                        for (int q = 0; q < 5; ++q) u[q] += Fg.U[q * Fg.fs + o];
                    }
#pragma unroll
            for (int q = 0; q < 5; ++q) u[q] = u[q] * inv_r3;
        } else {
            const int n1 = face < 2 ? n[1] : n[0];
            const int a = face < 2 ? m[1] : m[0], b = face < 4 ? m[2] : m[1];
            const double inv = face < 2 ? C.idx : face < 4 ? C.idy : C.idz;
            const int64_t o = M.froff[face] + 5 * ((int64_t)b * n1 + a);
#pragma unroll
            for (int q = 0; q < 5; ++q) {
                const double rc = M.frc[o + q], rf = M.frf[o + q];
                u[q] = C.U[q * C.fs + c] + ((face & 1) ? (rf - rc) * inv : (rc - rf) * inv);
            }
        }
        if (i >= 0 && i < C.nx && j >= 0 && j < C.ny && k >= 0 && k < C.nz) {
            if (C.prec == 1) apply_floor<true>(u, C.rho_floor, C.P_floor, C.gamma);
            else             apply_floor<false>(u, C.rho_floor, C.P_floor, C.gamma);
        }
#pragma unroll
        for (int q = 0; q < 5; ++q) C.U[q * C.fs + c] = u[q];
    }
}


// ---------------------------------------------------------------------------
// Launch helpers

static int resident_blocks(const void* fn, int threads, size_t lds) {
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, threads, lds) != hipSuccess || per < 1)
        per = 1;
    return per;
}

static int occupancy_grid(const void* fn, int threads, size_t lds, int ntiles, int cus) {
    int64_t g = (int64_t)resident_blocks(fn, threads, lds) * cus;
    if (g > ntiles) g = ntiles;
    return (int)(g < 1 ? 1 : g);
}

template <int DIR, typename T, int W, int H, bool FLAT = false>
static hipError_t launch_flux_t(const LaunchCtx& L, const GridDev* grids, const Tile* tiles,
                                int ntiles, int max_wg) {
    if (ntiles <= 0) return hipSuccess;
    const void* fn = (const void*)&k_flux<DIR, T, W, H, FLAT>;
    int g = occupancy_grid(fn, W * H, 0, ntiles, L.cus);
    if (max_wg > 0 && g > max_wg) g = max_wg;
    hipLaunchKernelGGL((k_flux<DIR, T, W, H, FLAT>), dim3(g), dim3(W * H), 0, L.stream, grids, tiles, ntiles);
    return hipGetLastError();
}

template <int DIR, typename T>
static hipError_t launch_fwalk_t(const LaunchCtx& L, const GridDev* grids, const Tile* tiles,
                                 int ntiles, int max_wg) {
    if (ntiles <= 0) return hipSuccess;
    const void* fn = (const void*)&k_fwalk<DIR, T>;
    int g = occupancy_grid(fn, 256, 0, ntiles, L.cus);
    if (max_wg > 0 && g > max_wg) g = max_wg;
    hipLaunchKernelGGL((k_fwalk<DIR, T>), dim3(g), dim3(256), 0, L.stream, grids, tiles, ntiles);
    return hipGetLastError();
}

template <typename T, int KMAX, bool OUT>
static hipError_t launch_fxwalk_t(const LaunchCtx& L, const GridDev* grids, const Tile* tiles,
                                  int ntiles, int max_wg) {
    if (ntiles <= 0) return hipSuccess;
    const void* fn = (const void*)&k_fxwalk<T, KMAX, OUT>;
    int g = occupancy_grid(fn, 256, 0, ntiles, L.cus);
    if (max_wg > 0 && g > max_wg) g = max_wg;
    hipLaunchKernelGGL((k_fxwalk<T, KMAX, OUT>), dim3(g), dim3(256), 0, L.stream, grids, tiles, ntiles);
    return hipGetLastError();
}

template <int DIR, typename T>
static hipError_t launch_flux_shape(const LaunchCtx& L, int shape, const GridDev* grids,
                                    const Tile* tiles, int ntiles, int max_wg) {
    if (DIR != 0 && shape >= FLUX_WALK_SHAPE0)
        return launch_fwalk_t<DIR == 0 ? 1 : DIR, T>(L, grids, tiles, ntiles, max_wg);
    if (DIR == 0 && shape >= FLUX_XWALK_SHAPE0 && shape != FLUX_XFLAT)
        switch (shape - FLUX_XWALK_SHAPE0) {
            case 0: return launch_fxwalk_t<T, 2, true>(L, grids, tiles, ntiles, max_wg);
            case 1: return launch_fxwalk_t<T, 4, true>(L, grids, tiles, ntiles, max_wg);
            default: return launch_fxwalk_t<T, 4, false>(L, grids, tiles, ntiles, max_wg);
        }
    // shape ids: x sweep 0: 64x4, 1: 32x8, 2: 16x16;  y/z sweep 0: 64x4, 1: 64x8, 2: 32x8, 3: 64x2,
    // 4: 32x16
    if (DIR == 0) {
        switch (shape) {
            case FLUX_XFLAT: return launch_flux_t<0, T, 64, 4, true>(L, grids, tiles, ntiles, max_wg);
            case 1: return launch_flux_t<DIR, T, 32, 8>(L, grids, tiles, ntiles, max_wg);
            case 2: return launch_flux_t<DIR, T, 16, 16>(L, grids, tiles, ntiles, max_wg);
            default: return launch_flux_t<DIR, T, 64, 4>(L, grids, tiles, ntiles, max_wg);
        }
    } else {
        switch (shape) {
            case 1: return launch_flux_t<DIR, T, 64, 8>(L, grids, tiles, ntiles, max_wg);
            case 2: return launch_flux_t<DIR, T, 32, 8>(L, grids, tiles, ntiles, max_wg);
            case 3: return launch_flux_t<DIR, T, 64, 2>(L, grids, tiles, ntiles, max_wg);
            case 4: return launch_flux_t<DIR, T, 32, 16>(L, grids, tiles, ntiles, max_wg);
            default: return launch_flux_t<DIR, T, 64, 4>(L, grids, tiles, ntiles, max_wg);
        }
    }
}

// W x H of a tiled shape; for the walk shapes W = 64 lanes and H = 4 rows or
// columns, with the run length flux_walk_len(dir, shape).
void flux_shape_dims(int dir, int shape, int& W, int& H) {
    static const int xs[3][2] = {{64, 4}, {32, 8}, {16, 16}};
    static const int ys[5][2] = {{64, 4}, {64, 8}, {32, 8}, {64, 2}, {32, 16}};
    if (flux_walk_len(dir, shape) > 0) { W = 64; H = 4; return; }
    if (dir == 0) { if (shape < 0 || shape > 2) shape = 0; W = xs[shape][0]; H = xs[shape][1]; }
    else          { if (shape < 0 || shape > 4) shape = 0; W = ys[shape][0]; H = ys[shape][1]; }
}

// Run length of a walk shape (interfaces per thread; for x the most one lane
// takes), 0 for a tiled shape.
int flux_walk_len(int dir, int shape) {
    if (shape < 0 || shape >= flux_shape_count(dir)) return 0;
    if (dir == 0) {
        static const int lens[3] = {2, 4, 4};
        return shape >= FLUX_XWALK_SHAPE0 ? lens[shape - FLUX_XWALK_SHAPE0] : 0;
    }
    static const int lens[3] = {16, 32, 64};
    return shape >= FLUX_WALK_SHAPE0 ? lens[shape - FLUX_WALK_SHAPE0] : 0;
}

int flux_slots(int dir, int prec, int shape, int cus) {
    // only the walks' tile lists depend on it
    if (dir == 0 || flux_walk_len(dir, shape) <= 0) return cus;
    const void* fn = prec == 0 ? (dir == 1 ? (const void*)&k_fwalk<1, double> : (const void*)&k_fwalk<2, double>)
                               : (dir == 1 ? (const void*)&k_fwalk<1, float> : (const void*)&k_fwalk<2, float>);
    return resident_blocks(fn, 256, 0) * cus;
}

int flux_shape_count(int dir) { return dir == 0 ? FLUX_XWALK_SHAPE0 + 3 : FLUX_WALK_SHAPE0 + 3; }

hipError_t launch_flux(const LaunchCtx& L, int dir, int prec, int shape, const GridDev* grids,
                       const Tile* tiles, int ntiles, int max_wg) {
    if (prec == 0) {
        if (dir == 0) return launch_flux_shape<0, double>(L, shape, grids, tiles, ntiles, max_wg);
        if (dir == 1) return launch_flux_shape<1, double>(L, shape, grids, tiles, ntiles, max_wg);
        return launch_flux_shape<2, double>(L, shape, grids, tiles, ntiles, max_wg);
    }
    if (dir == 0) return launch_flux_shape<0, float>(L, shape, grids, tiles, ntiles, max_wg);
    if (dir == 1) return launch_flux_shape<1, float>(L, shape, grids, tiles, ntiles, max_wg);
    return launch_flux_shape<2, float>(L, shape, grids, tiles, ntiles, max_wg);
}

template <typename T, int KZ>
static hipError_t launch_update_t(const LaunchCtx& L, const GridDev* grids, const Tile* tiles, int ntiles,
                                  int stage, int do_cfl, double* dU_out) {
    const int g = KZ == 1 ? ntiles : occupancy_grid((const void*)&k_update<T, KZ>, 256, 0, ntiles, L.cus);
    hipLaunchKernelGGL((k_update<T, KZ>), dim3(g), dim3(256), 0, L.stream, grids, tiles, ntiles, stage, do_cfl,
                       dU_out);
    return hipGetLastError();
}

hipError_t launch_update(const LaunchCtx& L, int prec, int kz, const GridDev* grids, const Tile* tiles,
                         int ntiles, int stage, int do_cfl, double* dU_out) {
    if (ntiles <= 0) return hipSuccess;
    if (kz == 1)
        return prec == 0 ? launch_update_t<double, 1>(L, grids, tiles, ntiles, stage, do_cfl, dU_out)
                         : launch_update_t<float, 1>(L, grids, tiles, ntiles, stage, do_cfl, dU_out);
    return prec == 0 ? launch_update_t<double, UPDATE_KZ>(L, grids, tiles, ntiles, stage, do_cfl, dU_out)
                     : launch_update_t<float, UPDATE_KZ>(L, grids, tiles, ntiles, stage, do_cfl, dU_out);
}

hipError_t launch_sweeps(const LaunchCtx& L, int prec, const GridDev* grids, const Tile* tiles, const int n[3]) {
    const int total = n[0] + n[1] + n[2];
    if (total <= 0) return hipSuccess;
    if (prec == 0)
        hipLaunchKernelGGL(k_sweeps<double>, dim3(total), dim3(256), 0, L.stream, grids, tiles, n[0], n[1]);
    else
        hipLaunchKernelGGL(k_sweeps<float>, dim3(total), dim3(256), 0, L.stream, grids, tiles, n[0], n[1]);
    return hipGetLastError();
}

static int flat_blocks(int64_t n, int cus);

template <typename T, int PF, int WB, int RING>
static hipError_t launch_zupdate_t(const LaunchCtx& L, const GridDev* grids, const Tile* tiles,
                                   int ntiles, int stage, int do_cfl) {
    const void* fn = (const void*)&k_zupdate<T, PF, WB, RING>;
    const int g = occupancy_grid(fn, 256, 0, ntiles, L.cus);
    hipLaunchKernelGGL((k_zupdate<T, PF, WB, RING>), dim3(g), dim3(256), 0, L.stream, grids,
                       tiles, ntiles, stage, do_cfl);
    return hipGetLastError();
}

template <typename T, int PF, int WB, int RING>
static int zupdate_slots_t(int cus) {
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)&k_zupdate<T, PF, WB, RING>,
                                                     256, 0) != hipSuccess || per < 1)
        per = 1;
    return per * cus;
}

// Shapes: 3 * variant + segmentation.  Variant 0 plain, 1 operands loaded one
// cell ahead (FP64) or variant 3 without a register cap (split: 2 waves per
// SIMD), 2 LDS ring of the window's raw cells, 3 ring plus an early load of
// the next window cell (split: both capped at 168 VGPRs, 3 waves per SIMD).
// Segmentation 0: at most 16 cells per run, 1: 32, 2: runs balanced by the load of
// a CU (run_counts in bsn_api.cpp).
int zupdate_shape_count() { return 12; }
int zupdate_seg(int shape) { return shape % 3; }

int zupdate_slots(int prec, int shape, int cus) {
    const int v = shape / 3;
    if (prec == 0) {
        switch (v) {
            case 1: return zupdate_slots_t<double, 1, 1, 0>(cus);
            case 2: return zupdate_slots_t<double, 0, 1, 1>(cus);
            case 3: return zupdate_slots_t<double, 2, 1, 1>(cus);
            default: return zupdate_slots_t<double, 0, 1, 0>(cus);
        }
    }
    switch (v) {
        case 1: return zupdate_slots_t<float, 2, 1, 1>(cus);
        case 2: return zupdate_slots_t<float, 0, 3, 1>(cus);
        case 3: return zupdate_slots_t<float, 2, 3, 1>(cus);
        default: return zupdate_slots_t<float, 0, 1, 0>(cus);
    }
}

template <typename T>
static hipError_t launch_zupdate_p(const LaunchCtx& L, int shape, const GridDev* grids,
                                   const Tile* tiles, int ntiles, int stage, int do_cfl) {
    constexpr bool F = sizeof(T) == 4;
    switch (shape / 3) {
        case 1: return F ? launch_zupdate_t<T, 2, 1, 1>(L, grids, tiles, ntiles, stage, do_cfl)
                         : launch_zupdate_t<T, 1, 1, 0>(L, grids, tiles, ntiles, stage, do_cfl);
        case 2: return launch_zupdate_t<T, 0, F ? 3 : 1, 1>(L, grids, tiles, ntiles, stage, do_cfl);
        case 3: return launch_zupdate_t<T, 2, F ? 3 : 1, 1>(L, grids, tiles, ntiles, stage, do_cfl);
        default: return launch_zupdate_t<T, 0, 1, 0>(L, grids, tiles, ntiles, stage, do_cfl);
    }
}

hipError_t launch_zupdate(const LaunchCtx& L, int prec, int shape, const GridDev* grids,
                          const Tile* tiles, int ntiles, int stage, int do_cfl) {
    if (ntiles <= 0) return hipSuccess;
    if (prec == 0) return launch_zupdate_p<double>(L, shape, grids, tiles, ntiles, stage, do_cfl);
    return launch_zupdate_p<float>(L, shape, grids, tiles, ntiles, stage, do_cfl);
}

hipError_t launch_cfl(const LaunchCtx& L, int kz, const GridDev* grids, const Tile* tiles, int ntiles) {
    if (ntiles <= 0) return hipSuccess;
    if (kz == 1) {
        hipLaunchKernelGGL(k_cfl<1>, dim3(ntiles), dim3(256), 0, L.stream, grids, tiles, ntiles);
    } else {
        const int g = occupancy_grid((const void*)&k_cfl<UPDATE_KZ>, 256, 0, ntiles, L.cus);
        hipLaunchKernelGGL(k_cfl<UPDATE_KZ>, dim3(g), dim3(256), 0, L.stream, grids, tiles, ntiles);
    }
    return hipGetLastError();
}

static int flat_blocks(int64_t n, int cus) {
    int64_t b = (n + 255) / 256;
    const int64_t cap = (int64_t)cus * 16;
    if (b > cap) b = cap;
    return (int)(b < 1 ? 1 : b);
}

hipError_t launch_ghost_fill(const LaunchCtx& L, const GridDev* grids, const int64_t* off,
                             int ngrids, int64_t total, int copy_un) {
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ghost_fill, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream, grids,
                       off, ngrids, copy_un);
    return hipGetLastError();
}

hipError_t launch_ghost_combine(const LaunchCtx& L, const GridDev* grids, const int64_t* off,
                                int ngrids, int64_t total, int stage, int advance) {
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ghost_combine, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream,
                       grids, off, ngrids, stage, advance);
    return hipGetLastError();
}

hipError_t launch_floors(const LaunchCtx& L, const GridDev* grids, const int64_t* off, int ngrids,
                         int64_t total, int copy_un) {
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_floors, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream, grids,
                       off, ngrids, copy_un);
    return hipGetLastError();
}

hipError_t launch_fmr_dt(const LaunchCtx& L, const GridDev* grids, const FmrFactors& f) {
    hipLaunchKernelGGL(k_fmr_dt, dim3(1), dim3(1), 0, L.stream, grids, f);
    return hipGetLastError();
}

hipError_t launch_cfl_begin(const LaunchCtx& L, const GridDev* grids, int ngrids, double cfl, double t_end,
                            int restart) {
    hipLaunchKernelGGL(k_cfl_begin, dim3((ngrids + 63) / 64), dim3(64), 0, L.stream, grids, ngrids, cfl, t_end,
                       restart);
    return hipGetLastError();
}

hipError_t launch_fmr_correct(const LaunchCtx& L, const GridDev* grids, const FmrDev* fmr, const FmrDev& hf) {
    int64_t cells = 1;
    for (int a = 0; a < 3; ++a) cells *= hf.hi[a] - hf.lo[a] + 3;
    hipLaunchKernelGGL(k_fmr_correct, dim3(flat_blocks(cells, L.cus)), dim3(256), 0, L.stream, grids, fmr);
    return hipGetLastError();
}

hipError_t launch_dt(const LaunchCtx& L, const GridDev* grids, int ngrids, double* out) {
    hipLaunchKernelGGL(k_dt, dim3((ngrids + 63) / 64), dim3(64), 0, L.stream, grids, ngrids, out);
    return hipGetLastError();
}

hipError_t launch_set_scal(const LaunchCtx& L, double* scal, int idx, double v) {
    hipLaunchKernelGGL(k_set_scal, dim3(1), dim3(1), 0, L.stream, scal, idx, v);
    return hipGetLastError();
}

hipError_t launch_fill_u64(const LaunchCtx& L, uint64_t* p, int64_t n, uint64_t v) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_u64, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, p, n, v);
    return hipGetLastError();
}

hipError_t launch_aos_to_soa(const LaunchCtx& L, const GridDev& G, const double* aos, double* dst) {
    const int64_t n = (int64_t)(G.nx + 2 * NG) * G.Ny * G.Nz;
    hipLaunchKernelGGL(k_aos_to_soa, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, aos, dst);
    return hipGetLastError();
}

hipError_t launch_soa_to_aos(const LaunchCtx& L, const GridDev& G, const double* src, double* aos) {
    const int64_t n = (int64_t)(G.nx + 2 * NG) * G.Ny * G.Nz;
    hipLaunchKernelGGL(k_soa_to_aos, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, src, aos);
    return hipGetLastError();
}

hipError_t launch_flux_export(const LaunchCtx& L, const GridDev& G, int dir, double* out) {
    const int64_t n = (int64_t)(G.nx + 2 * NG + (dir == 0)) * (G.Ny + (dir == 1)) * (G.Nz + (dir == 2));
    if (G.prec == 0)
        hipLaunchKernelGGL(k_flux_export<double>, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, dir, out);
    else
        hipLaunchKernelGGL(k_flux_export<float>, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, dir, out);
    return hipGetLastError();
}

hipError_t launch_sg_force(const LaunchCtx& L, const GridDev& G, double* dU) {
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    hipLaunchKernelGGL(k_sg_force, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, dU);
    return hipGetLastError();
}

hipError_t launch_src(const LaunchCtx& L, const GridDev& G, double* dU, int which) {
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    hipLaunchKernelGGL(k_src, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, dU, which);
    return hipGetLastError();
}

hipError_t launch_combine_all(const LaunchCtx& L, const GridDev& G, int stage, const double* dU, double dt) {
    const int64_t n = (int64_t)(G.nx + 2 * NG) * G.Ny * G.Nz;
    hipLaunchKernelGGL(k_combine_all, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, G, stage, dU, dt);
    return hipGetLastError();
}

hipError_t launch_copy_state(const LaunchCtx& L, const GridDev& G, const double* src, double* dst) {
    hipLaunchKernelGGL(k_copy_state, dim3(flat_blocks(5 * G.fs, L.cus)), dim3(256), 0, L.stream, G, src, dst);
    return hipGetLastError();
}

// Fixed scratch of bsn_conserved_totals_noalloc: the block partial sums of
// one totals launch (TOTALS_BLOCKS x 5) and its five sums, in a file-scope
// device array.  Each device holds its own copy until the process ends; host
// code reaches it only through the address totals_scratch_setup returns
// (the array's name is a host-side stand-in, not a device address).
static __device__ __align__(256) double scratch[TOTALS_SCRATCH_DOUBLES];

static std::mutex s_scratch_mu;
static double* s_scratch_ptr[BSN_MAX_DEVICES] = {};

// Once per device, with that device current: the device address of scratch.
hipError_t totals_scratch_setup(int device, double** ptr) {
    *ptr = nullptr;
    if (device < 0 || device >= BSN_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(s_scratch_mu);
    if (!s_scratch_ptr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        s_scratch_ptr[device] = (double*)p;
    }
    *ptr = s_scratch_ptr[device];
    return hipSuccess;
}

hipError_t launch_totals(const LaunchCtx& L, const GridDev& G, double* part, int nblocks, double dV,
                         double* out) {
    hipLaunchKernelGGL(k_totals_partial, dim3(nblocks), dim3(256), 0, L.stream, G, part);
    hipLaunchKernelGGL(k_totals_final, dim3(1), dim3(64), 0, L.stream, part, nblocks, dV, out);
    return hipGetLastError();
}

hipError_t launch_prolong(const LaunchCtx& L, const GridDev* grids, const FmrDev* fmr, const GridDev& child,
                          int ratio, const double* Uca, const double* Ucat, int all_cells, ProlongDst dst) {
    // blocks of one wave: few threads with much work each, spread over all CUs
    const ProlongWork w = prolong_work(child.nx, child.ny, child.nz, all_cells, ratio);
    hipLaunchKernelGGL(k_prolong, dim3((unsigned)std::min<int64_t>(w.bx + w.by + w.bz, 64LL * L.cus)), dim3(64), 0, L.stream,
                       grids, fmr, Uca, Ucat, all_cells, dst);
    return hipGetLastError();
}

hipError_t launch_time_interp(const LaunchCtx& L, const GridDev* grids, const FmrDev* fmr,
                              int64_t total, double alpha) {
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_time_interp, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream, grids,
                       fmr, alpha);
    return hipGetLastError();
}

hipError_t launch_restrict(const LaunchCtx& L, const GridDev* grids, const FmrDev* fmr, int64_t total,
                           int nfields) {
    hipLaunchKernelGGL(k_restrict, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream, grids, fmr,
                       nfields);
    return hipGetLastError();
}

hipError_t launch_prolong_scalar(const LaunchCtx& L, const double* phc, const int nc[3], double* phf,
                                 const int nf[3], const int lo[3], int ratio) {
    const int64_t total = (int64_t)nf[0] * nf[1] * nf[2];
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_prolong_scalar, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream, phc,
                       nc[0], nc[1], nc[2], phf, nf[0], nf[1], nf[2], lo[0], lo[1], lo[2], ratio);
    return hipGetLastError();
}

hipError_t launch_scale(const LaunchCtx& L, double* a, int64_t n, double s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_scale, dim3(flat_blocks(n, L.cus)), dim3(256), 0, L.stream, a, n, s);
    return hipGetLastError();
}

hipError_t launch_level_begin(const LaunchCtx& L, const GridDev* grids, int level, const GridDev& h,
                              const FmrDev* fmr, const FmrDev* hf, int own) {
    const int64_t ghosts = 2LL * NG * ((int64_t)h.Ny * h.Nz + (int64_t)h.nx * h.Nz + (int64_t)h.nx * h.ny);
    int64_t total = own ? ghosts : 0;
    if (fmr) {
        int64_t box = 1;
        for (int a = 0; a < 3; ++a) box *= hf->phi[a] - hf->plo[a] + 1;
        total += box + hf->froff[6];
    }
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_level_begin, dim3(flat_blocks(total, L.cus)), dim3(256), 0, L.stream, grids, level,
                       fmr, own);
    return hipGetLastError();
}

hipError_t launch_fr_coarse(const LaunchCtx& L, int prec, const GridDev* grids, const FmrDev* fmr,
                            int64_t nelem, double weight) {
    const dim3 grid(flat_blocks(nelem, L.cus), 5);     // one grid row per field
    if (prec == 0)
        hipLaunchKernelGGL(k_fr_coarse<double>, grid, dim3(256), 0, L.stream, grids, fmr, weight);
    else
        hipLaunchKernelGGL(k_fr_coarse<float>, grid, dim3(256), 0, L.stream, grids, fmr, weight);
    return hipGetLastError();
}

hipError_t launch_fr_fine(const LaunchCtx& L, int prec, const GridDev* grids, const FmrDev* fmr,
                          int64_t nelem, double weight) {
    const dim3 grid(flat_blocks(nelem, L.cus), 5);     // one grid row per field
    if (prec == 0)
        hipLaunchKernelGGL(k_fr_fine<double>, grid, dim3(256), 0, L.stream, grids, fmr, weight);
    else
        hipLaunchKernelGGL(k_fr_fine<float>, grid, dim3(256), 0, L.stream, grids, fmr, weight);
    return hipGetLastError();
}

}  // namespace bsn
