// Several time steps of one 2-D shot per launch.
//
// A workgroup takes a tile of every array, its halo included, into workgroup memory and
// advances it up to 8 steps (velocity and stress updates with their CPML memory, rigid
// faces, free surface, sources and receivers) before it writes the cells it owns to the
// model's other state: one update's dependency reaches h = order - 1 cells each way, so a
// halo of steps * h cells keeps the owned ones exact, and the tiles recompute each other's
// halos instead of exchanging them.  A thread owns K consecutive columns of one row and
// keeps its wavefields, coefficients and CPML memory in registers; workgroup memory only
// carries the neighbours' samples, with two barriers per step.  The expressions and their
// order are the passes' (fdtd2d.hip), so the results are the same bit for bit; outside an
// update's range its coefficient is zero and outside a strip the CPML update is the
// identity, which leaves the inner loop without branches.  (The identity holds for finite
// derivatives: where a shot has overflowed, the first step's infinities may be NaN here.  The same
// samples are non-finite and the finite ones equal; a select per derivative that keeps the
// infinities took 2.8 % of an elastic gradient on 251 x 333 cells and 6 % of a shot on 301^2.)
//
// The passes read and write 48 (acoustic) or 72 (elastic) bytes per cell and step and launch
// twice a step, which bounds grids below about 600 cells a side by the launches (3.6 us
// each).  Here a tile's arrays (6 in, 3 out; elastic 10 in, 5 out) move once per launch:
// 2-D elastic 2081^2 takes 16 us a step (269 Gcell-steps/s) against 53, where the inner
// tiles' time is half memory traffic, half arithmetic (the compiled loop has 33 vector and 7
// workgroup-memory instructions per cell and step, for 1.5 times the owned cells); acoustic 241^2 takes 1.4 us a step against 7.3, bound by
// the latency of a launch and of the two barriers per step.
#include "fdtd2d.h"
#include "fdtd2d_steps.h"
#include "gpi_util.h"
#include "stencil.h"

namespace gpi {

namespace {

// first cell of tile k when n cells are dealt evenly to t tiles
__host__ __device__ constexpr int tile_start(int k, int n, int t) { return k * n / t; }
__host__ constexpr int tile_of(int x, int n, int t) { return ((x + 1) * t - 1) / n; }

// element o of a slab by a 32-bit byte offset from its (wave-uniform) base
__device__ __forceinline__ const float& at(const float* base, uint32_t o)
{
    return *(const float*)((const char*)base + 4u * o);
}
__device__ __forceinline__ float& at(float* base, uint32_t o) { return *(float*)((char*)base + 4u * o); }

// strip index of derivative point j of nd, -1 outside the active strips
__device__ __forceinline__ int strip_index(int j, int nd, int npml, bool lo, bool hi)
{
    if (j < 0 || j >= nd) return -1;
    if (lo && j < npml) return j;
    if (hi && j >= nd - npml) return j - nd + 2 * npml;
    return -1;
}

// one CPML memory update (cpml.jl:178-180)
__device__ __forceinline__ float pml_at(float d, float& psi, float a, float b, float k)
{
    psi = b * psi + a * d;
    return d * k + psi;
}

template <int O, int PHYS, int RZ, int WX, int NT>
struct Tile {
    static constexpr int H = O - 1;
    static constexpr int G = NT / RZ;         // column groups
    static constexpr int K = WX / G;          // columns per thread
    static constexpr int A = RZ * WX;         // floats per array
    static constexpr int NF = PHYS ? 5 : 3;   // arrays: stresses, then vx, vz
    static constexpr int ND = PHYS ? 4 : 2;   // derivatives along x (and along z)
    static constexpr int FVX = PHYS ? 3 : 1;
    static constexpr int FVZ = FVX + 1;
    static constexpr int PAD = H * RZ + H;    // stencils of edge cells stay inside the allocation
    static constexpr int FLOATS = NF * A + 2 * PAD;
    static constexpr bool XREG = K == 1;      // x CPML coefficients in registers (else workgroup memory)
    static constexpr int XC = XREG ? 1 : ND * 3 * WX;
    static_assert(WX % G == 0 && NT % RZ == 0 && NT >= MAX_TILE_SOURCES, "tile");
};

// The derivatives along one axis in the order of their updates and the slot of their CPML
// memory; `v`: taken by the velocity update (derivative point = cell - h), cut0 / cut1:
// how much shorter than the stress grid the derivative is along z / x, in h.
struct Deriv {
    int slot, v, cutz, cutx;
};
template <int PHYS>
struct Derivs;
template <>
struct Derivs<0> {
    static constexpr Deriv X[2] = {{0, 1, 2, 1}, {2, 0, 0, 0}};   // dpdx, dvxdx
    static constexpr Deriv Z[2] = {{1, 1, 1, 2}, {3, 0, 0, 0}};   // dpdz, dvzdz
};
template <>
struct Derivs<1> {
    static constexpr Deriv X[4] = {{0, 1, 2, 1}, {2, 1, 1, 2}, {4, 0, 0, 0}, {7, 0, 1, 1}};   // dtauxxdx, dtauxzdx, dvxdx, dvzdx
    static constexpr Deriv Z[4] = {{1, 1, 2, 1}, {3, 1, 1, 2}, {5, 0, 0, 0}, {6, 0, 1, 1}};   // dtauxzdz, dtauzzdz, dvzdz, dvxdz
};

struct TileLds {
    float* f;         // arrays of the tile
    float* xc;        // x CPML coefficients: ND x 3 x WX
    int* kind;        // the tile's sources: kind, two steps' increments
    float* amp;
};

// PX / PZ: the tile reaches the strips or faces of x / z.  Outside the strips the CPML
// update is the identity (a = b = 0, kI = 1, psi = 0), outside an update's range its
// coefficient is zero, so only the stores of tiles on the grid's edge are masked.
// SR: the tile may hold sources and receivers.  KEEP: every step is kept (a ring).  Both cost
// the inner tiles registers, and with them the second tile per CU (KEEP: 21.1 against 15.3 ms
// for 800 steps of 2-D elastic 2081^2), so they are choices at compile time.  FORCE:
// time reversal, p forced on stored planes before every step.
template <int O, int PHYS, int RZ, int WX, int NT, bool PX, bool PZ, bool SR, bool KEEP, bool FORCE>
__device__ __forceinline__ void run_tile(const StepParams2D& P, const TileLds& Q, const TileBox& B)
{
    using T = Tile<O, PHYS, RZ, WX, NT>;
    using D = Derivs<PHYS>;
    constexpr int H = T::H, K = T::K, A = T::A, NF = T::NF, ND = T::ND, FVX = T::FVX, FVZ = T::FVZ;
    constexpr bool PP = PX || PZ;
    const int tid = (int)threadIdx.x;
    const int lr = tid % RZ;
    int g = tid / RZ;
    if (RZ == 64) g = __builtin_amdgcn_readfirstlane(g);
    const int lc0 = g * K;
    const int czl = B.z0, czh = B.z1, cxl = B.x0, cxh = B.x1;
    // Cores are dealt evenly, so a small one's tile reaches past its own halo.  Inner tiles load
    // every cell without a test: their last ones start earlier instead of ending outside the grid
    // (the cells between are further halo, and inner tiles have no table of cells).
    int r0 = czl - P.lead, c0 = cxl - P.lead;
    if constexpr (!SR) {
        r0 = min(r0, P.nz + H - RZ);
        c0 = min(c0, P.nx + H - WX);
    }
    const int r = r0 + lr, cc = c0 + lc0;
    const int ld = P.ld;
    float* const L = Q.f + T::PAD + lr + RZ * lc0;   // this thread's first cell of array 0
    const bool edge = PP && (r0 <= H || r0 + RZ >= P.nz - H || c0 <= H || c0 + WX >= P.nx - H);

    // ---- wavefields, coefficients and CPML memory into registers
    float S[K][NF], C[K][NF];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = cc + k;
        const int o = r + ld * c;
        const bool in = !PP || (r >= 0 && r < P.nz + H && c >= 0 && c < P.nx + H);
#pragma unroll
        for (int f = 0; f < NF; ++f) S[k][f] = in ? at(P.in[f], o) : 0.0f;
#pragma unroll
        for (int f = 0; f < NF; ++f) C[k][f] = in ? at(P.coef[f], o) : 0.0f;
    }
    // stored planes: this thread's offset in one step's values of fx (>= 0) or fz (~offset), or none
    constexpr int NONE = INT32_MIN;
    int foff[FORCE ? K : 1];
    auto forced = [&](int k, int64_t it) __attribute__((always_inline)) {
        const int64_t n = P.fnt - 1 - it;
        const int o = foff[FORCE ? k : 0];
        return o >= 0 ? P.fx[n * (6 * (int64_t)P.nz) + o] : P.fz[n * (6 * (int64_t)P.nx) + ~o];
    };
    if constexpr (FORCE) {
        auto plane = [](int p, int n, int np) { return p >= np && p < np + 3 ? p - np : p >= n - np - 3 && p < n - np ? p - (n - np) + 6 : -1; };
        const int az = r >= 0 && r < P.nz ? plane(r, P.nz, P.fnp[0]) : -1;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = cc + k;
            foff[k] = NONE;
            if (r < 0 || r >= P.nz || c < 0 || c >= P.nx) continue;
            const int ax = plane(c, P.nx, P.fnp[1]);
            if (ax >= 0) foff[k] = r + P.nz * ax;
            else if (az >= 0) foff[k] = ~(az + 6 * c);
            if (foff[k] != NONE) S[k][0] = forced(k, P.it0);
        }
    }
    float px[K][PX ? ND : 1], pz[K][PZ ? ND : 1], za[ND], zb[ND], zk[ND], xa[K][ND], xb[K][ND], xk[K][ND];
    int zi[ND];
    if constexpr (PZ) {
        const bool lo = (P.pml_mask & GPI_FACE(0, 0)) != 0, hi = (P.pml_mask & GPI_FACE(0, 1)) != 0;
#pragma unroll
        for (int q = 0; q < ND; ++q) {
            constexpr auto& DZ = D::Z;
            zi[q] = strip_index(r - H * DZ[q].v, P.nz - H * DZ[q].cutz, P.npml, lo, hi);
            const bool in = zi[q] >= 0;
            za[q] = in ? at(P.pa[DZ[q].slot], zi[q]) : 0.0f;
            zb[q] = in ? at(P.pb[DZ[q].slot], zi[q]) : 0.0f;
            zk[q] = in ? at(P.pk[DZ[q].slot], zi[q]) : 1.0f;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int j = cc + k - H * DZ[q].v;
                pz[k][q] = in && j >= 0 && j < P.nx - H * DZ[q].cutx
                               ? at(P.psi_in[DZ[q].slot], zi[q] + P.ps2[DZ[q].slot] * j) : 0.0f;
            }
        }
    }
    if constexpr (PX) {
        const bool lo = (P.pml_mask & GPI_FACE(2, 0)) != 0, hi = (P.pml_mask & GPI_FACE(2, 1)) != 0;
#pragma unroll
        for (int q = 0; q < ND; ++q) {
            constexpr auto& DX = D::X;
            const int i = r - H * DX[q].v;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int xi = strip_index(cc + k - H * DX[q].v, P.nx - H * DX[q].cutx, P.npml, lo, hi);
                px[k][q] = xi >= 0 && i >= 0 && i < P.nz - H * DX[q].cutz
                               ? at(P.psi_in[DX[q].slot], i + P.ps2[DX[q].slot] * xi) : 0.0f;
                if (T::XREG) {
                    xa[k][q] = xi >= 0 ? at(P.pa[DX[q].slot], xi) : 0.0f;
                    xb[k][q] = xi >= 0 ? at(P.pb[DX[q].slot], xi) : 0.0f;
                    xk[k][q] = xi >= 0 ? at(P.pk[DX[q].slot], xi) : 1.0f;
                }
            }
            if (!T::XREG && tid < WX) {
                const int xi = strip_index(c0 + tid - H * DX[q].v, P.nx - H * DX[q].cutx, P.npml, lo, hi);
                Q.xc[(3 * q) * WX + tid] = xi >= 0 ? at(P.pa[DX[q].slot], xi) : 0.0f;
                Q.xc[(3 * q + 1) * WX + tid] = xi >= 0 ? at(P.pb[DX[q].slot], xi) : 0.0f;
                Q.xc[(3 * q + 2) * WX + tid] = xi >= 0 ? at(P.pk[DX[q].slot], xi) : 1.0f;
            }
        }
    }
    auto pml_z = [&](float d, int q, int k) __attribute__((always_inline)) { return pml_at(d, pz[k][q], za[q], zb[q], zk[q]); };
    auto pml_x = [&](float d, int q, int k) __attribute__((always_inline)) {
        if (T::XREG) return pml_at(d, px[k][q], xa[k][q], xb[k][q], xk[k][q]);
        const float* x = Q.xc + 3 * q * WX + lc0 + k;
        return pml_at(d, px[k][q], x[0], x[WX], x[2 * WX]);
    };

    // ---- sources: first << 16 | count of this thread's cells, through a map over the tile
    const int ns = SR ? B.s1 - B.s0 : 0, nr = SR ? B.r1 - B.r0 : 0;
    int mine[SR ? K : 1];
    const float* amp_next = nullptr;
    if (SR && ns) {
        int* map = (int*)(Q.f + T::PAD);
        for (int e = tid; e < A; e += NT) map[e] = 0;
        TileSource E{};
        if (tid < ns) {
            E = P.src[B.s0 + tid];
            amp_next = P.amp + P.it0 * P.namp + E.target;
            Q.kind[tid] = E.kind;
            Q.amp[tid] = *amp_next;
        }
        __syncthreads();
        if (tid < ns && E.first) map[E.cell] = tid << 16 | E.first;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; ++k) mine[SR ? k : 0] = map[lr + RZ * (lc0 + k)];
        __syncthreads();
    }
    // ---- receivers: one per thread in registers (the rest, if any, read per step)
    TileReceiver R{};
    float* rout = nullptr;
    int rnpts = 0;
    if (SR && tid < nr) {
        R = P.rec[B.r0 + tid];
        rnpts = P.rnpts[R.set];
        rout = P.rout[R.set] + P.it0 * rnpts + R.point;
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int f = 0; f < NF; ++f) L[f * A + RZ * k] = S[k][f];
    __syncthreads();

    // sample of one receiver (tap order of the interpolation column)
    auto sample = [&](const TileReceiver& E) __attribute__((always_inline)) {
        const float* a = Q.f + T::PAD + E.array * A + E.base;
        float t = 0.0f;
        t += E.w[0] * a[0];
        t += E.w[1] * a[1];
        t += E.w[2] * a[RZ];
        t += E.w[3] * a[RZ + 1];
        return t;
    };
    auto gather = [&](bool velocity, int64_t it) __attribute__((always_inline)) {
        if (!SR || !nr) return;
        if (tid < nr && (R.array >= FVX) == velocity) {
            *rout = sample(R);
            rout += rnpts;
        }
        for (int e = tid + NT; e < nr; e += NT) {
            const TileReceiver E = P.rec[B.r0 + e];
            if ((E.array >= FVX) == velocity) P.rout[E.set][it * P.rnpts[E.set] + E.point] = sample(E);
        }
    };

    const bool own = r >= czl && r < czh;
    // the tile's own values of arrays f0 .. f1 - 1 after `n` of the launch's steps
    auto keep = [&](int f0, int f1, int n) __attribute__((always_inline)) {
        int slot = P.hstart + n;
        if (slot >= P.hslots) slot -= P.hslots;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = cc + k;
            if (!own || c < cxl || c >= cxh) continue;
            if (FORCE && f0 == 0 && (r >= P.nz || c >= P.nx)) continue;   // not yet restored there
#pragma unroll
            for (int f = 0; f < NF; ++f)
                if (f >= f0 && f < f1 && P.hist[f]) at(P.hist[f] + P.hslab * slot, r + ld * c) = S[k][f];
        }
    };

#pragma unroll 1
    for (int s = 0; s < P.steps; ++s) {
        const int64_t it = P.it0 + s;
        float anext = 0.0f;
        if (SR && tid < ns && s + 1 < P.steps) anext = *(amp_next += P.namp);
        float fnext[FORCE ? K : 1];
        if constexpr (FORCE) {
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (s + 1 < P.steps && foff[k] != NONE) fnext[k] = forced(k, it + 1);
        }
        const float* amp = Q.amp + (s & 1) * MAX_TILE_SOURCES;
        // columns whose values are still needed: the rest of the halo is stale already
        const int halo = SR ? P.lead : cxl - c0;
        const int need0 = halo - (P.steps - 1 - s) * H;
        const int need1 = halo + (cxh - cxl) + (P.steps - s) * H;
        gather(false, it);
        if (lc0 + K > need0 && lc0 < need1) {
            if (PP && edge) {   // the free surface's row is written by the row below
#pragma unroll
                for (int k = 0; k < K; ++k)
#pragma unroll
                    for (int f = 0; f < FVX; ++f) S[k][f] = L[RZ * k + f * A];
            }
            if (KEEP && !FORCE && s) keep(0, FVX, s);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const float* l = L + RZ * k;
                float v[O];
                // derivative points start H cells before the velocities they update
#pragma unroll
                for (int q = 0; q < O; ++q) v[q] = q == H ? S[k][0] : l[(q - H) * RZ];
                float dx = stencil<O>(v) * P.dxI;
                if constexpr (PX) dx = pml_x(dx, 0, k);
                if (PHYS == 0) {
                    S[k][FVX] = S[k][FVX] + C[k][0] * dx;
                } else {
#pragma unroll
                    for (int q = 0; q < O; ++q) v[q] = l[2 * A + (q - H) - H * RZ];
                    float d2 = stencil<O>(v) * P.dzI;
                    if constexpr (PZ) d2 = pml_z(d2, 0, k);
                    S[k][FVX] = S[k][FVX] - C[k][0] * (dx + d2);
                }
                constexpr int FZ = PHYS ? 1 : 0;   // p or tauzz
#pragma unroll
                for (int q = 0; q < O; ++q) v[q] = q == H ? S[k][FZ] : l[FZ * A + (q - H)];
                float dz = stencil<O>(v) * P.dzI;
                if constexpr (PZ) dz = pml_z(dz, PHYS ? 1 : 0, k);
                if (PHYS == 0) {
                    S[k][FVZ] = S[k][FVZ] + C[k][1] * dz;
                } else {
#pragma unroll
                    for (int q = 0; q < O; ++q) v[q] = l[2 * A - H + (q - H) * RZ];
                    float d2 = stencil<O>(v) * P.dxI;
                    if constexpr (PX) d2 = pml_x(d2, PHYS ? 1 : 0, k);
                    S[k][FVZ] = S[k][FVZ] - C[k][1] * (d2 + dz);
                }
            }
            if (PP && edge) {
                // rigid faces: the mirror of the first / last interior velocity, before its sources
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    float* l = L + RZ * k;
                    const int c = cc + k;
                    const bool ux = r >= H && r < P.nz - H && c >= H && c < P.nx;
                    const bool uz = r >= H && r < P.nz && c >= H && c < P.nx - H;
                    if (ux && (P.rigid_mask & GPI_FACE(2, 0)) && c == H && lc0 + k >= H) l[FVX * A - H * RZ] = -S[k][FVX];
                    if (ux && (P.rigid_mask & GPI_FACE(2, 1)) && c == P.nx - 1 && lc0 + k + H < WX)
                        l[FVX * A + H * RZ] = -S[k][FVX];
                    if (uz && (P.rigid_mask & GPI_FACE(0, 0)) && r == H && lr >= H) l[FVZ * A - H] = -S[k][FVZ];
                    if (uz && (P.rigid_mask & GPI_FACE(0, 1)) && r == P.nz - 1 && lr + H < RZ) l[FVZ * A + H] = -S[k][FVZ];
                }
            }
            if (SR && ns) {
#pragma unroll
                for (int k = 0; k < K; ++k) {
#pragma unroll 1
                    for (int e = mine[SR ? k : 0] >> 16, n = mine[SR ? k : 0] & 0xffff; n > 0; ++e, --n) {
                        const int kind = Q.kind[e];
                        const float a = amp[e];
                        if (kind == 1) S[k][FVX] = S[k][FVX] + a;
                        if (kind == 2) S[k][FVZ] = S[k][FVZ] + a;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                float* l = L + RZ * k;
                const int c = cc + k;
                if (!edge || (r >= H && r < P.nz - H && c >= H && c < P.nx)) l[FVX * A] = S[k][FVX];
                if (!edge || (r >= H && r < P.nz && c >= H && c < P.nx - H)) l[FVZ * A] = S[k][FVZ];
            }
        }
        __syncthreads();
        gather(true, it);
        if (lc0 + K > need0 && lc0 < need1 - H) {
            if (PP && edge) {   // mirrored by a neighbour
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    S[k][FVX] = L[RZ * k + FVX * A];
                    S[k][FVZ] = L[RZ * k + FVZ * A];
                }
            }
            if (KEEP && s + 1 < P.steps) keep(FVX, NF, s + 1);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const float* l = L + RZ * k;
                float v[O];
#pragma unroll
                for (int q = 0; q < O; ++q) v[q] = q == 0 ? S[k][FVX] : l[FVX * A + q * RZ];
                float dvx = stencil<O>(v) * P.dxI;
                if constexpr (PX) dvx = pml_x(dvx, PHYS ? 2 : 1, k);
#pragma unroll
                for (int q = 0; q < O; ++q) v[q] = q == 0 ? S[k][FVZ] : l[FVZ * A + q];
                float dvz = stencil<O>(v) * P.dzI;
                if constexpr (PZ) dvz = pml_z(dvz, PHYS ? 2 : 1, k);
                if (PHYS == 0) {
                    S[k][0] = S[k][0] + (dvx + dvz) * C[k][2];
                } else {
                    const float m = C[k][2], lam = C[k][3 % NF];
                    S[k][0] = (S[k][0] - (m * dvx)) - (lam * dvz);
                    S[k][1] = (S[k][1] - (m * dvz)) - (lam * dvx);
#pragma unroll
                    for (int q = 0; q < O; ++q) v[q] = l[FVX * A + q + H * RZ];
                    float a = stencil<O>(v) * P.dzI;
                    if constexpr (PZ) a = pml_z(a, ND - 1, k);
#pragma unroll
                    for (int q = 0; q < O; ++q) v[q] = l[FVZ * A + H + q * RZ];
                    float b = stencil<O>(v) * P.dxI;
                    if constexpr (PX) b = pml_x(b, ND - 1, k);
                    S[k][2] = S[k][2] - C[k][4 % NF] * (a + b);
                }
            }
            const bool fs = PP && PHYS && edge && (P.free_mask & GPI_FACE(0, 0)) != 0;
            if (fs && r == 1 && lr >= 1) {   // tauzz above the free surface, before the sources
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (cc + k >= 0 && cc + k < P.nx) L[RZ * k + A - 1] = -S[k][1];
            }
            if (SR && ns) {
#pragma unroll
                for (int k = 0; k < K; ++k) {
#pragma unroll 1
                    for (int e = mine[SR ? k : 0] >> 16, n = mine[SR ? k : 0] & 0xffff; n > 0; ++e, --n) {
                        if (Q.kind[e]) continue;
                        const float a = amp[e];
                        S[k][0] = S[k][0] + a;
                        if (PHYS) S[k][1] = S[k][1] + a;
                    }
                }
            }
            if constexpr (FORCE) {   // kept as the step left it, and forced for the next one
                if (s + 1 < P.steps) keep(0, FVX, s + 1);
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (s + 1 < P.steps && foff[k] != NONE) S[k][0] = fnext[k];
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                float* l = L + RZ * k;
                const int c = cc + k;
                const bool un = !edge || (r >= 0 && r < P.nz && c >= 0 && c < P.nx);
                if (un) l[0] = S[k][0];
                if (PHYS) {
                    if (un && !(fs && r == 0)) l[A] = S[k][1];
                    if (!edge || (r >= 0 && r < P.nz - H && c >= 0 && c < P.nx - H))
                        l[2 * A] = (fs && r == 0) ? 0.0f : S[k][2];
                }
            }
        }
        if (SR && tid < ns) Q.amp[((s + 1) & 1) * MAX_TILE_SOURCES + tid] = anext;
        __syncthreads();
    }

    // ---- the tile's own cells out
    if (own) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = cc + k;
            if (c < cxl || c >= cxh) continue;
            const int o = r + ld * c;
#pragma unroll
            for (int f = 0; f < NF; ++f) at(P.out[f], o) = PP && edge ? L[f * A + RZ * k] : S[k][f];
            if constexpr (PZ) {
#pragma unroll
                for (int q = 0; q < ND; ++q) {
                    constexpr auto& DZ = D::Z;
                    const int j = c - H * DZ[q].v;
                    if (zi[q] >= 0 && j >= 0 && j < P.nx - H * DZ[q].cutx)
                        at(P.psi_out[DZ[q].slot], zi[q] + P.ps2[DZ[q].slot] * j) = pz[k][q];
                }
            }
            if constexpr (PX) {
                const bool lo = (P.pml_mask & GPI_FACE(2, 0)) != 0, hi = (P.pml_mask & GPI_FACE(2, 1)) != 0;
#pragma unroll
                for (int q = 0; q < ND; ++q) {
                    constexpr auto& DX = D::X;
                    const int i = r - H * DX[q].v;
                    const int xi = strip_index(c - H * DX[q].v, P.nx - H * DX[q].cutx, P.npml, lo, hi);
                    if (xi >= 0 && i >= 0 && i < P.nz - H * DX[q].cutz)
                        at(P.psi_out[DX[q].slot], i + P.ps2[DX[q].slot] * xi) = px[k][q];
                }
            }
        }
    }
}

template <int O, int PHYS, int RZ, int WX, int NT, bool KEEP, bool FORCE>
__global__ __launch_bounds__(NT) void steps2d_kernel(StepParams2D P)
{
    using T = Tile<O, PHYS, RZ, WX, NT>;
    __shared__ float f[T::FLOATS];
    __shared__ float xc[T::XC];
    __shared__ int kind[MAX_TILE_SOURCES];
    __shared__ float amp[2 * MAX_TILE_SOURCES];
    const TileBox B = P.box[xcd_remap(blockIdx.x, gridDim.x)];
    const TileLds Q{f, xc, kind, amp};
    constexpr int H = O - 1;
    // tiles away from the strips and faces need none of their code
    const int r0 = B.z0 - P.lead, c0 = B.x0 - P.lead, e = H + P.npml + 1;
    const bool pz = r0 < e || r0 + RZ > P.nz - H - e, px = c0 < e || c0 + WX > P.nx - H - e;
    if (px) {
        if (pz) run_tile<O, PHYS, RZ, WX, NT, true, true, true, KEEP, FORCE>(P, Q, B);
        else run_tile<O, PHYS, RZ, WX, NT, true, false, true, KEEP, FORCE>(P, Q, B);
    } else {
        if (pz) run_tile<O, PHYS, RZ, WX, NT, false, true, true, KEEP, FORCE>(P, Q, B);
        else run_tile<O, PHYS, RZ, WX, NT, false, false, true, KEEP, FORCE>(P, Q, B);
    }
}

// Tiles away from the strips and faces, without sources and receivers.
template <int O, int PHYS, int RZ, int WX, int NT, bool KEEP, bool FORCE>
__global__ __launch_bounds__(NT) void steps2d_inner_kernel(StepParams2D P)
{
    using T = Tile<O, PHYS, RZ, WX, NT>;
    __shared__ float f[T::FLOATS];
    run_tile<O, PHYS, RZ, WX, NT, false, false, false, KEEP, FORCE>(P, TileLds{f, nullptr, nullptr, nullptr},
                                                       P.box[xcd_remap(blockIdx.x, gridDim.x)]);
}

// Coefficients of the updates at the cells they update, with the passes' expressions.
template <int PHYS>
__global__ __launch_bounds__(256) void step_coef_kernel(const float* rho, const float* c0, const float* c1, float* o0,
                                                        float* o1, float* o2, float* o3, float* o4, int nz, int nx,
                                                        int ld, int H, float dt)
{
    const int r = blockIdx.x * 64 + threadIdx.x, c = blockIdx.y * 4 + threadIdx.y;
    if (r >= nz + H || c >= nx + H) return;
    const int o = r + ld * c;
    float cx = 0.0f, cz = 0.0f;
    if (r >= H && r < nz - H && c >= H && c < nx) cx = dt_over_av2(dt, rho[r + ld * (c - H)], rho[r + ld * (c - H + 1)]);
    if (r >= H && r < nz && c >= H && c < nx - H) cz = dt_over_av2(dt, rho[r - H + ld * c], rho[r - H + 1 + ld * c]);
    o0[o] = cx;
    o1[o] = cz;
    if (PHYS) {
        float m = 0.0f, l = 0.0f, a = 0.0f;
        if (r < nz && c < nx) {
            m = dtm_of(c0[o], c1[o], dt);
            l = (1.0f / c0[o]) * dt;
        }
        if (r < nz - H && c < nx - H) a = dt_over_av4(dt, c1[o], c1[o + 1], c1[o + ld], c1[o + 1 + ld]);
        o2[o] = m;
        o3[o] = l;
        o4[o] = a;
    }
}

// amp[it][base + t]: what target t adds to its field at step it, the sum of its
// contributions in source order times its scale (source.jl:160-177)
__global__ __launch_bounds__(256) void amplitude_kernel(float* amp, int namp, int base, int ntarget, int64_t nt,
                                                        const int64_t* toff, const int32_t* tptr, const int32_t* tsrc,
                                                        const float* tw, const float* wav, int npts, const float* coef,
                                                        const float* rho, float dt)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= nt * ntarget) return;
    const int64_t it = e / ntarget;
    const int t = (int)(e % ntarget);
    const float* w = wav + it * (int64_t)npts;
    float a = 0.0f;
    for (int c = tptr[t]; c < tptr[t + 1]; ++c) a += tw[c] * w[tsrc[c]];
    if (coef) {
        a = a * coef[toff[t]];
    } else {
        const int64_t* roff = toff + ntarget;
        const float av = (rho[roff[2 * t]] + rho[roff[2 * t + 1]]) * 0.5f;
        a = (a / av) * dt;
    }
    amp[it * namp + base + t] = a;
}

// A rectangle of cells dealt evenly to tz x tx tiles, boxes first .. of a launch.
struct Region {
    int z0, nz, x0, nx, tz, tx, first;
};

template <int O, int PHYS, int RZ, int WX, int NT>
void launch_all(const StepParams2D& P, hipStream_t s)
{
    const dim3 grd(P.ntile), blk(NT);
    if constexpr (PHYS == 0) {
        if (P.fx) {
            hipLaunchKernelGGL((steps2d_kernel<O, PHYS, RZ, WX, NT, true, true>), grd, blk, 0, s, P);
            return;
        }
    }
    if (P.hslots) hipLaunchKernelGGL((steps2d_kernel<O, PHYS, RZ, WX, NT, true, false>), grd, blk, 0, s, P);
    else hipLaunchKernelGGL((steps2d_kernel<O, PHYS, RZ, WX, NT, false, false>), grd, blk, 0, s, P);
}

template <int O, int PHYS, int RZ, int WX, int NT>
void launch_inner(const StepParams2D& P, hipStream_t s)
{
    const dim3 grd(P.ntile), blk(NT);
    if constexpr (PHYS == 0) {
        if (P.fx) {
            hipLaunchKernelGGL((steps2d_inner_kernel<O, PHYS, RZ, WX, NT, true, true>), grd, blk, 0, s, P);
            return;
        }
    }
    if (P.hslots) hipLaunchKernelGGL((steps2d_inner_kernel<O, PHYS, RZ, WX, NT, true, false>), grd, blk, 0, s, P);
    else hipLaunchKernelGGL((steps2d_inner_kernel<O, PHYS, RZ, WX, NT, false, false>), grd, blk, 0, s, P);
}

// The tiles that pick_tiles chooses from.
template <int O, int PHYS>
void launch_o(const StepTile& t, bool inner, const StepParams2D& P, hipStream_t s)
{
    if constexpr (O == 2) {
        if (inner && t.wx == 32) launch_inner<O, PHYS, 64, 32, 1024>(P, s);
        else if (inner) launch_inner<O, PHYS, 64, PHYS ? 48 : 64, PHYS ? 768 : 1024>(P, s);
        else if (t.rz == 32) launch_all<O, PHYS, 32, 32, 1024>(P, s);
        else launch_all<O, PHYS, 64, 32, 1024>(P, s);
    } else if constexpr (O == 4) {
        if (inner) launch_inner<O, PHYS, 64, 64, 1024>(P, s);
        else if (t.rz == 32) launch_all<O, PHYS, 32, 32, 1024>(P, s);
        else if (PHYS == 0 && t.wx == 64) launch_all<O, 0, 64, 64, 1024>(P, s);
        else launch_all<O, PHYS, 64, 32, 1024>(P, s);
    } else {
        launch_all<O, PHYS, 64, 32, 1024>(P, s);
    }
}

// Tiles of a region: cores of at most (rz - 2 lead) x (wx - 2 lead) cells, dealt evenly.
Region region_of(const StepTile& t, int lead, int z0, int z1, int x0, int x1, int first)
{
    Region R{};
    R.z0 = z0;
    R.nz = z1 - z0;
    R.x0 = x0;
    R.nx = x1 - x0;
    const int mz = t.rz - 2 * lead, mx = t.wx - 2 * lead;
    R.tz = (R.nz + mz - 1) / mz;
    R.tx = (R.nx + mx - 1) / mx;
    R.first = first;
    return R;
}

// The whole grid in one launch (inner.rz == 0), or the frame of strips and faces around an
// inner rectangle.
struct Frame {
    int zh, xh, e, zi, xi;   // extents, the inner rectangle [e, zi) x [e, xi)
};

Frame frame_of(const Model& m, int lead)
{
    Frame f{};
    f.zh = (int)m.g.n[0] + m.h;
    f.xh = (int)m.g.n[2] + m.h;
    f.e = lead + m.h + m.g.npml + 1;
    f.zi = f.zh - (f.e + 2 * m.h);
    f.xi = f.xh - (f.e + 2 * m.h);
    return f;
}

bool frame_fits(const Frame& f, const StepTile& inner) { return f.zi - f.e >= inner.rz && f.xi - f.e >= inner.wx; }

int64_t tiles_in(const StepTile& t, int lead, int z, int x)
{
    if (t.rz <= 2 * lead || t.wx <= 2 * lead) return INT32_MAX;
    const Region R = region_of(t, lead, 0, z, 0, x, 0);
    return (int64_t)R.tz * R.tx;
}

int64_t frame_tiles(const Frame& f, const StepTile& t, int lead)
{
    return tiles_in(t, lead, f.e, f.xh) + tiles_in(t, lead, f.zh - f.zi, f.xh) + tiles_in(t, lead, f.zi - f.e, f.e) +
           tiles_in(t, lead, f.zi - f.e, f.xh - f.xi);
}

// Tile and steps per launch by grid size and order; false where the passes are as fast.
// A launch costs about 6 us besides its steps (the wavefields' way through memory and the
// launch itself) and a step about 0.7 (acoustic) or 1 us (elastic) per round of tiles, one
// 1024-thread tile at a time on each of the 256 CUs, so a small grid takes the most steps
// for which its tiles still make one round.  Larger grids are bound by the inner tiles'
// memory traffic and arithmetic; their strips, faces and sources (twice the registers, a
// quarter of the tiles in flight) go to a launch of their own.  us per step, order 2,
// absorbing width 20, against the passes: acoustic 260^2 1.59 / 7.2, 400^2 2.15 / 7.5,
// 700^2 3.4 / 9, 1500^2 6.5 / 25; elastic 260^2 1.91 / 8.3, 700^2 4.8 / 13, 1500^2 10.4 / 31,
// 2001^2 (width 40) 16.1 / 53.  Order 4: acoustic 260^2 3.4 / 7.3, 497x811 (width 43) 6.5 / 9.7,
// 1500^2 13.3 / 25; elastic 260^2 4.3 / 8.4, 1500^2 26 / 34.  Order 6, whose halo is five cells a
// step, gains on small grids only (260^2: 4.9 / 7.4 and 7.0 / 8.5; 400^2 lost), and order 8 nowhere
// (1500^2 one step: 76 / 25).
// The lines between the shapes, us per step on the extended grid:
// - order 2, 6 steps from 3 M cells, 8 below (6 / 8 steps, width 40): acoustic 1650^2 7.8 / 8.1,
//   1760^2 8.0 / 8.2, 1900^2 8.4 / 10.0, 2081^2 9.1 / 10.6, 2400^2 11.8 / 12.1; elastic 1650^2
//   12.3 / 13.1, 1760^2 12.5 / 13.9, 1900^2 13.7 / 16.2, 2081^2 16.4 / 18.8, 2400^2 22.7 / 22.7.
//   Below the line the two are within 7 % (1300^2: 6.7 / 6.9 and 10.1 / 10.3); 7 steps, which the
//   rule does not know, took 6.1 and 9.2 there and 7 to 13 % more than 6 steps from 1900^2 to 2081^2.
// - order 2, one round of 32 x 32 tiles or of 32 x 32 around 64 x 32, and no whole grid of 64 x 32:
//   383x483 acoustic 2.04 and elastic 2.58 against 1.86 and 2.73 in one round of 64 x 32 at 8 steps,
//   450^2 2.09 and 2.69 against 2.42 and 3.39.
// - order 4 acoustic, up to two rounds of 64 x 64 whole tiles at 3 steps where the frame takes more
//   than one: 583x897 6.7 against 8.3 with the frame apart and 8.0 in one round at 2 steps,
//   700^2 6.0 / 8.4 / 8.1; the frame apart gains at the upper end, 760x900 10.0 / 9.2 / 10.6.
bool pick_tiles(const Model& m, StepTile* all, StepTile* inner)
{
    constexpr int CUS = 256;
    const int H = m.h, z = (int)m.g.n[0] + H, x = (int)m.g.n[2] + H;
    const bool ac = m.g.physics == 0;
    *inner = StepTile{};
    auto one_round = [&](int rz, int wx, int steps) {
        *all = StepTile{rz, wx, steps};
        return tiles_in(*all, steps * H, z, x) <= CUS;
    };
    if (m.g.order == 2) {
        for (int t = 8; t >= 5; --t)
            if (one_round(32, 32, t)) return true;
        for (int t = 8; t >= 6; --t) {
            *all = StepTile{32, 32, t};
            *inner = StepTile{64, 32, t};
            const Frame f = frame_of(m, t);
            if (frame_fits(f, *inner) && tiles_in(*inner, t, f.zi - f.e, f.xi - f.e) <= 2 * CUS &&
                frame_tiles(f, *all, t) <= CUS)
                return true;
        }
        const int t = (int64_t)z * x > 3000000 ? 6 : 8;
        *all = StepTile{64, 32, t};
        *inner = StepTile{64, ac ? 64 : 48, t};
        if (!frame_fits(frame_of(m, t), *inner)) {   // little more than its strips
            *all = StepTile{64, 32, 6};
            *inner = StepTile{};
        }
        return true;
    }
    if (m.g.order == 4) {
        if (one_round(32, 32, 3) || one_round(32, 32, 2) || one_round(64, 32, 2)) return true;
        *all = StepTile{64, 32, 3};
        *inner = StepTile{64, 64, 3};
        const Frame f = frame_of(m, 3 * H);
        // wide strips: their tiles take longer than the whole grid in two rounds of larger ones
        if (ac && tiles_in(*inner, 3 * H, z, x) <= 2 * CUS &&
            (!frame_fits(f, *inner) || frame_tiles(f, *all, 3 * H) > CUS)) {
            *all = StepTile{64, 64, 3};
            *inner = StepTile{};
            return true;
        }
        if (!frame_fits(f, *inner)) {
            *all = StepTile{64, 32, 2};
            *inner = StepTile{};
        }
        return true;
    }
    return m.g.order == 6 && one_round(64, 32, 2);
}

}  // namespace
int launch_steps_2d(const Model& m)
{
    StepTile all{}, inner{};
    return m.g.ndim == 2 && pick_tiles(m, &all, &inner) ? all.steps : 0;
}

int plan_steps_2d(gpi_ctx* c, Model& m, Scratch& S, int64_t nt, const Sources& src,
                  const gpi_shot* shot, const std::vector<DevPoints>& rec, StepPlan* plan, bool* ok, bool second)
{
    *ok = false;
    const gpi_grid& g = m.g;
    const bool ac = g.physics == 0;
    const int H = m.h, nz = (int)g.n[0], nx = (int)g.n[2];
    if (g.ndim != 2 || c->arena || nt < 2 || !src.vfall.empty() || !src.sfall.empty()) return GPI_OK;
    if (m.slab >= (1 << 30)) return GPI_OK;   // 32-bit byte offsets
    StepParams2D P{};
    VelParams2D V;
    StrParams2D T;
    if (!vel_params_2d(m, *m.st0, &V) || !str_params_2d(m, *m.st0, &T)) return GPI_OK;
    const int ders[8] = {ac ? GPI_DPDX : GPI_DTAUXXDX, ac ? GPI_DPDZ : GPI_DTAUXZDZ, ac ? GPI_DVXDX : GPI_DTAUXZDX,
                         ac ? GPI_DVZDZ : GPI_DTAUZZDZ, GPI_DVXDX, GPI_DVZDZ, GPI_DVXDZ, GPI_DVZDX};
    const int nder = ac ? 4 : 8;
    for (int q = 0; q < nder; ++q)   // both strips of an axis apart, so a point has one memory variable
        if (g.pml_mask && m.pml[ders[q]].nd < 2 * g.npml) return GPI_OK;
    StepTile t[2];
    if (!pick_tiles(m, &t[0], &t[1])) return GPI_OK;
    const int lead = t[0].steps * H;
    if (t[0].rz <= 2 * (lead + H) || t[0].wx <= 2 * (lead + H)) return GPI_OK;
    P.lead = lead;

    // ---- regions: the whole grid in one launch, or an inner rectangle clear of strips and
    // faces (its tiles' halos included) in a launch of its own and the four around it; inner
    // tiles with sources or receivers are cut into tiles of the other launch
    std::vector<Region> reg;
    Region in{};
    int ntile = 0;
    const Frame fr = frame_of(m, lead);
    const int zh = fr.zh, xh = fr.xh, e = fr.e, zi = fr.zi, xi = fr.xi;
    auto add = [&](int z0, int z1, int x0, int x1) {
        if (z1 <= z0 || x1 <= x0) return;
        reg.push_back(region_of(t[0], lead, z0, z1, x0, x1, ntile));
        ntile += reg.back().tz * reg.back().tx;
    };
    const bool split = t[1].rz > 0;
    if (split) {
        in = region_of(t[1], lead, e, zi, e, xi, 0);
        add(0, e, 0, xh);
        add(zi, zh, 0, xh);
        add(e, zi, 0, e);
        add(e, zi, xi, xh);
    } else {
        add(0, zh, 0, xh);
    }
    const int64_t most = std::max({zh, xh, nz, nx});
    if (most * (most + 1) > INT32_MAX) return GPI_OK;   // tile_start's products
    for (const Region& R : reg)   // a rigid face's mirror cells share their tile with the velocities they mirror
        if (R.nz / R.tz <= H || R.nx / R.tx <= H) return GPI_OK;

    // targets of the sources and first taps of the receivers
    struct Cell {
        int r, x, kind, id;      // kind: source kind, or array sampled
    };
    std::vector<Cell> tg, rv;
    std::vector<const float*> rw;
    int namp = 0, nset = 0;
    for (size_t q = 0; q < src.pts.size(); ++q) {
        const DevPoints& D = src.pts[q];
        const int kind = D.field == GPI_VX ? 1 : D.field == GPI_VZ ? 2 : 0;
        for (int k = 0; k < D.ntarget; ++k)
            tg.push_back(Cell{(int)(src.toff[q][k] % m.pitch0), (int)(src.toff[q][k] / m.pitch0), kind, namp + k});
        namp += D.ntarget;
    }
    if ((int64_t)namp * nt > ((int64_t)1 << 28)) return GPI_OK;
    std::vector<int> rset;
    for (int q = 0; shot && q < shot->nrec; ++q) {
        const DevPoints& D = rec[q];
        const gpi_points& U = shot->rec[q];
        const int f = D.field;
        if (D.npts == 0 || !(f == GPI_P || f == GPI_VX || f == GPI_VZ)) continue;
        if (nset == MAX_STEP_REC) return GPI_OK;
        int64_t n3[3];
        shape_of(g.ndim, g.order, g.physics, g.n, f, n3);
        const int array = f == GPI_P ? 0 : f == GPI_VX ? (ac ? 1 : 3) : (ac ? 2 : 4);
        for (int p = 0; p < D.npts; ++p) {
            const int64_t* ix = U.idx + (size_t)p * 4;
            if (ix[1] != ix[0] + 1 || ix[2] != ix[0] + n3[0] || ix[3] != ix[2] + 1 || ix[0] % n3[0] == n3[0] - 1)
                return GPI_OK;   // not the taps of a linear interpolation
            rv.push_back(Cell{(int)(ix[0] % n3[0]), (int)(ix[0] / n3[0]), array, p});
            rw.push_back(U.w + (size_t)p * 4);
            rset.push_back(nset);
        }
        P.rnpts[nset] = D.npts;
        P.rout[nset] = D.rec;
        ++nset;
    }
    // calls fn(tile) for every tile of region R (tile l) that holds cell (r, x), its halo included
    auto holders = [&](const Region& R, const StepTile& l, int r, int x, auto&& fn) {
        const int bx0 = tile_of(std::min(std::max(x - R.x0 - l.wx, 0), R.nx - 1), R.nx, R.tx);
        const int bz0 = tile_of(std::min(std::max(r - R.z0 - l.rz, 0), R.nz - 1), R.nz, R.tz);
        for (int bx = bx0; bx < R.tx; ++bx) {
            const int lc = x - R.x0 - tile_start(bx, R.nx, R.tx) + lead;
            if (lc < 0) break;
            if (lc >= l.wx) continue;
            for (int bz = bz0; bz < R.tz; ++bz) {
                const int lr = r - R.z0 - tile_start(bz, R.nz, R.tz) + lead;
                if (lr < 0) break;
                if (lr < l.rz) fn(bz + R.tz * bx, lr + l.rz * lc);
            }
        }
    };
    std::vector<char> special((size_t)(in.tz * in.tx), 0);
    if (split) {
        for (const Cell& c : tg) holders(in, t[1], c.r, c.x, [&](int b, int) { special[b] = 1; });
        for (const Cell& c : rv)
            if (c.r >= in.z0 && c.r < in.z0 + in.nz && c.x >= in.x0 && c.x < in.x0 + in.nx)
                special[tile_of(c.r - in.z0, in.nz, in.tz) + in.tz * tile_of(c.x - in.x0, in.nx, in.tx)] = 1;
        for (int b = 0; b < in.tz * in.tx; ++b) {
            if (!special[b]) continue;
            const int bz = b % in.tz, bx = b / in.tz;
            add(in.z0 + tile_start(bz, in.nz, in.tz), in.z0 + tile_start(bz + 1, in.nz, in.tz),
                in.x0 + tile_start(bx, in.nx, in.tx), in.x0 + tile_start(bx + 1, in.nx, in.tx));
        }
    }
    // tables: the boxes of both launches, then the sources and receivers by tile
    std::vector<TileBox> box;
    auto boxes = [&](const Region& R, bool skip) {
        for (int b = 0; b < R.tz * R.tx; ++b) {
            const int bz = b % R.tz, bx = b / R.tz;
            if (skip && special[b]) continue;
            box.push_back(TileBox{R.z0 + tile_start(bz, R.nz, R.tz), R.z0 + tile_start(bz + 1, R.nz, R.tz),
                                  R.x0 + tile_start(bx, R.nx, R.tx), R.x0 + tile_start(bx + 1, R.nx, R.tx), 0, 0, 0, 0});
        }
    };
    for (const Region& R : reg) boxes(R, false);
    if (split) boxes(in, true);
    struct Src {
        int tile;
        TileSource e;
    };
    std::vector<Src> sl;
    std::vector<std::pair<int, TileReceiver>> rl;
    for (const Region& R : reg) {
        for (const Cell& c : tg)
            holders(R, t[0], c.r, c.x, [&](int b, int cell) {
                sl.push_back(Src{R.first + b, TileSource{cell, 0, c.kind, c.id}});
            });
        for (size_t k = 0; k < rv.size(); ++k) {
            const Cell& c = rv[k];
            if (c.r < R.z0 || c.r >= R.z0 + R.nz || c.x < R.x0 || c.x >= R.x0 + R.nx) continue;
            const int bz = tile_of(c.r - R.z0, R.nz, R.tz), bx = tile_of(c.x - R.x0, R.nx, R.tx);
            TileReceiver E{};
            E.base = (c.r - R.z0 - tile_start(bz, R.nz, R.tz) + lead) +
                     t[0].rz * (c.x - R.x0 - tile_start(bx, R.nx, R.tx) + lead);
            E.array = c.kind;
            E.set = rset[k];
            E.point = c.id;
            std::copy(rw[k], rw[k] + 4, E.w);
            rl.push_back({R.first + bz + R.tz * bx, E});
        }
    }
    std::stable_sort(sl.begin(), sl.end(), [](const Src& a, const Src& b) {
        return a.tile != b.tile ? a.tile < b.tile : a.e.cell < b.e.cell;
    });
    for (size_t k = 0, n; k < sl.size(); k = n) {   // entries of one cell, in set order
        for (n = k + 1; n < sl.size() && sl[n].tile == sl[k].tile && sl[n].e.cell == sl[k].e.cell;) ++n;
        sl[k].e.first = (int32_t)(n - k);
    }
    std::stable_sort(rl.begin(), rl.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    for (size_t k = 0, n; k < sl.size(); k = n) {
        for (n = k + 1; n < sl.size() && sl[n].tile == sl[k].tile;) ++n;
        if (n - k > (size_t)MAX_TILE_SOURCES) return GPI_OK;
        box[sl[k].tile].s0 = (int32_t)k;
        box[sl[k].tile].s1 = (int32_t)n;
    }
    for (size_t k = 0, n; k < rl.size(); k = n) {
        for (n = k + 1; n < rl.size() && rl[n].first == rl[k].first;) ++n;
        box[rl[k].first].r0 = (int32_t)k;
        box[rl[k].first].r1 = (int32_t)n;
    }
    const size_t sb = sizeof(TileBox) * box.size(), sr = sb + sizeof(TileSource) * sl.size();
    std::vector<char> tab(sr + sizeof(TileReceiver) * rl.size());
    std::memcpy(tab.data(), box.data(), sb);
    for (size_t k = 0; k < sl.size(); ++k) std::memcpy(&tab[sb + sizeof(TileSource) * k], &sl[k].e, sizeof(TileSource));
    for (size_t k = 0; k < rl.size(); ++k)
        std::memcpy(&tab[sr + sizeof(TileReceiver) * k], &rl[k].second, sizeof(TileReceiver));

    // ---- the second state, the coefficients and the tables, for this call alone: without room for
    // them the passes run
    Optional spare(c);
    Scratch R(c);
    auto alt = std::make_shared<State>();
    float* co[5] = {};
    char* dtab = nullptr;
    float* amp = nullptr;
    int rc = second ? alloc_state(c, m, alt.get(), true) : GPI_OK;
    R.p.swap(alt->allocs);
    std::swap(R.bytes, alt->bytes);
    for (int k = 0; !rc && k < (ac ? 2 : 5); ++k) rc = R.alloc(&co[k], (size_t)m.slab);
    if (!rc && namp) rc = R.alloc(&amp, (size_t)namp * (size_t)nt);
    if (!rc) rc = R.put(&dtab, tab);
    if (rc == GPI_ENOMEM) {
        (void)hipGetLastError();
        c->err.clear();
        return GPI_OK;
    }
    if (rc) return rc;
    P.box = (const TileBox*)dtab;
    P.src = (const TileSource*)(dtab + sb);
    P.rec = (const TileReceiver*)(dtab + sr);
    P.ntile = ntile;
    const dim3 grd((nz + H + 63) / 64, (nx + H + 3) / 4), blk(64, 4);
    if (ac)
        hipLaunchKernelGGL(step_coef_kernel<0>, grd, blk, 0, c->stream, m.coef[GPI_C_RHO], (const float*)nullptr,
                           (const float*)nullptr, co[0], co[1], (float*)nullptr, (float*)nullptr, (float*)nullptr, nz,
                           nx, (int)m.pitch0, H, g.dt);
    else
        hipLaunchKernelGGL(step_coef_kernel<1>, grd, blk, 0, c->stream, m.coef[GPI_C_RHO], m.coef[GPI_C_INVLAMBDA],
                           m.coef[GPI_C_INVMU], co[0], co[1], co[2], co[3], co[4], nz, nx, (int)m.pitch0, H, g.dt);
    P.coef[0] = co[0];
    P.coef[1] = co[1];
    P.coef[2] = ac ? m.coef[GPI_C_DTK] : co[2];
    P.coef[3] = co[3];
    P.coef[4] = co[4];
    if (namp) {
        int base = 0;
        for (const DevPoints& D : src.pts) {
            if (D.ntarget == 0) continue;
            const int64_t n = nt * D.ntarget;
            hipLaunchKernelGGL(amplitude_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, amp, namp,
                               base, D.ntarget, nt, D.toff, D.tptr, D.tsrc, D.tw, D.wav, D.npts,
                               is_velocity(D.field) ? (const float*)nullptr : P.coef[2], m.coef[GPI_C_RHO], g.dt);
            base += D.ntarget;
        }
        P.amp = amp;
        P.namp = namp;
    }
    for (int q = 0; q < nder; ++q) {
        const Pml& D = m.pml[ders[q]];
        P.pa[q] = D.a;
        P.pb[q] = D.b;
        P.pk[q] = D.kI;
        P.ps2[q] = (int)D.ps2;
    }
    P.nz = nz;
    P.nx = nx;
    P.ld = (int)m.pitch0;
    P.npml = g.npml;
    P.pml_mask = g.pml_mask;
    P.rigid_mask = g.rigid_mask;
    P.free_mask = g.free_mask;
    P.dxI = g.dsI[2];
    P.dzI = g.dsI[0];
    P.dt = g.dt;
    plan->steps = t[0].steps;
    plan->launches = 0;
    if (split && box.size() > (size_t)ntile) {   // the larger launch first
        StepParams2D& L = plan->P[plan->launches];
        L = P;
        L.box = P.box + ntile;
        L.ntile = (int)(box.size() - (size_t)ntile);
        plan->tile[plan->launches] = t[1];
        plan->inner[plan->launches++] = true;
    }
    plan->P[plan->launches] = P;
    plan->tile[plan->launches] = t[0];
    plan->inner[plan->launches++] = false;
    plan->st[0] = m.st0;
    plan->alt = alt;
    plan->st[1] = second ? alt.get() : nullptr;
    S.p.insert(S.p.end(), R.p.begin(), R.p.end());
    S.bytes += R.bytes;
    R.p.clear();
    R.bytes = 0;
    plan->cur = 0;
    std::copy(ders, ders + 8, plan->ders);
    *ok = true;
    return GPI_OK;
}

void run_steps_2d(const Model& m, StepPlan& plan, int64_t it0, int steps, hipStream_t s, Ring* ring)
{
    const State& a = *plan.st[plan.cur];
    const State& b = *plan.st[plan.cur ^ 1];
    const bool ac = m.g.physics == 0;
    const int af[3] = {GPI_P, GPI_VX, GPI_VZ}, ef[5] = {GPI_TAUXX, GPI_TAUZZ, GPI_TAUXZ, GPI_VX, GPI_VZ};
    for (int l = 0; l < plan.launches; ++l) {
        StepParams2D& P = plan.P[l];
        for (int k = 0; k < (ac ? 3 : 5); ++k) {
            const int f = ac ? af[k] : ef[k];
            P.in[k] = a.field[f];
            P.out[k] = b.field[f];
            P.hist[k] = ring ? ring->base[f] : nullptr;
            if (P.hist[k]) {
                P.in[k] = P.hist[k] + ring->slab * ring->cur;
                P.out[k] = P.hist[k] + ring->slab * ring->after(steps);
            }
        }
        P.hslots = ring ? ring->slots : 0;
        P.hslab = ring ? ring->slab : 0;
        P.hstart = ring ? ring->cur : 0;
        for (int q = 0; q < (ac ? 4 : 8); ++q) {
            P.psi_in[q] = a.psi[plan.ders[q]];
            P.psi_out[q] = b.psi[plan.ders[q]];
        }
        P.it0 = it0;
        P.steps = steps;
        const StepTile& t = plan.tile[l];
        const bool in = plan.inner[l];
        switch (m.g.order) {
        case 2: ac ? launch_o<2, 0>(t, in, P, s) : launch_o<2, 1>(t, in, P, s); break;
        case 4: ac ? launch_o<4, 0>(t, in, P, s) : launch_o<4, 1>(t, in, P, s); break;
        default: ac ? launch_o<6, 0>(t, in, P, s) : launch_o<6, 1>(t, in, P, s); break;
        }
    }
    plan.cur ^= 1;
    if (ring) ring->cur = ring->after(steps);
}

}  // namespace gpi
