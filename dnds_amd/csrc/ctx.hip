// Device context, arrays and the FP64 kernels of the hot path (gfx950).
//
// The context holds the mesh and the VR setup in device memory, repacked from
// the reference layouts into those of kernels.hpp: the sweep matrices in groups
// of 16 cells as a wave of four lanes per cell loads them (ab_vec), coefficients
// in blocks of 64 cells with the four variables side by side (rec), the other
// arrays of several values per cell or face in blocks of 64 (blk64, quad64).
// All kernels are launched on the context's stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "ctx.hpp"

using namespace dndsmi_dev;
using namespace dndsmi_host;

namespace dndsmi_host {

hipEvent_t prof_event(dndsmi_ctx *c) {
    if (c->ev_used == c->ev_pool.size()) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess)
            return nullptr;
        c->ev_pool.push_back(e);
    }
    return c->ev_pool[c->ev_used++];
}

// brackets a launch with events when profiling is on
void prof_begin(dndsmi_ctx *c, int id) {
    if (!c->prof_on)
        return;
    c->prof_open = id;
    c->prof_open_ev = c->ev_used;
    hipEvent_t e = prof_event(c);
    if (e)
        (void)hipEventRecord(e, c->stream);
}

void prof_end(dndsmi_ctx *c) {
    if (!c->prof_on || c->prof_open < 0)
        return;
    hipEvent_t e = prof_event(c);
    if (e) {
        (void)hipEventRecord(e, c->stream);
        c->prof_recs.push_back({c->prof_open, c->prof_open_ev});
    }
    c->prof_open = -1;
}

} // namespace dndsmi_host

// ========================================================================
// kernels
// ========================================================================

// ---- reconstruction sweeps: four lanes per cell --------------------------
//
// A sweep is bound by its stream of A^-1 B (720 B per cell and face, read
// once) and by the latency of the gathers beside it.  Four neighbouring lanes
// (a quad) own one cell, lane v of the quad variable v, so a wave covers 16
// cells: a lane keeps 9 coefficients instead of 36, which leaves registers
// for the loads of several slots in flight.  Each lane loads a quarter of the
// cell's A^-1 B (one contiguous KiB per wave and load) and the quad passes
// the entries around with DPP moves, so no byte is loaded twice.  Every sum
// runs in the order of a one-lane-per-cell sweep.

// a quad's sum of squares, lane 0's nine in turn, then lane 1's and so on: in
// the last lane
__device__ __forceinline__ double quad_norm2(const double d[9]) {
    double sum = 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int r = 0; r < 9; r++)
            sum += d[r] * d[r];
        if (q < 3)
            sum = quad_get(sum, q);
    }
    return sum;
}

// the neighbouring lane's `a` (lanes 2 k and 2 k + 1 exchange)
__device__ __forceinline__ double pair_swap(double a) {
    const uint64_t w = __builtin_bit_cast(uint64_t, a);
    const uint32_t lo = uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(w)), 0xb1, 0xf, 0xf, true));
    const uint32_t hi = uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(w >> 32)), 0xb1, 0xf, 0xf, true));
    return __builtin_bit_cast(double, uint64_t(lo) | uint64_t(hi) << 32);
}

// 16-byte loads from one group of the stream through a buffer descriptor,
// whose cache policy is part of the instruction (with plain and non-temporal
// pointer loads on two sides of a branch, the compiler makes one plain load)
struct ab_stream {
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ ab_stream(const void *p, int bytes)
        : rs(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00020000)) {}
    template <typename T, bool NT>
    __device__ __forceinline__ T get(uint32_t off, int soff) const {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, NT ? 2 : 0));
    }
};

// A lane's part of the A^-1 B, A^-1 b of one cell and slot (ab_vec's layout)
struct AbPart {
    dbl2 w[kAbVecs / 4], last;
    // groups with (i / 64) mod 64 below `keep` are read with ordinary loads
    __device__ __forceinline__ void load(const double *__restrict__ M, int s, int32_t i, int64_t ldc, int v,
                                         int32_t keep) {
        // a wave holds one group of 16 cells: a scalar base
        const int32_t g = __builtin_amdgcn_readfirstlane(i);
        const double *p = M + 2 * ab_group(s, g, ldc, kAbVecs);
        const uint32_t cl = i & 15;
        const ab_stream rs(p, 256 * kAbVecs);
        if (((g >> 6) & 63) < keep) {
#pragma unroll
            for (int k = 0; k < kAbVecs / 4; k++)
                w[k] = rs.get<dbl2, false>((4 * cl + v) * 16, 1024 * k);
            last = rs.get<dbl2, false>(cl * 16, 256 * (kAbVecs - 1));
        } else {
#pragma unroll
            for (int k = 0; k < kAbVecs / 4; k++)
                w[k] = rs.get<dbl2, true>((4 * cl + v) * 16, 1024 * k);
            last = rs.get<dbl2, true>(cl * 16, 256 * (kAbVecs - 1));
        }
    }
    // the same for lanes of one wave at different slots, ordinary loads
    __device__ __forceinline__ void load_each(const double *__restrict__ M, int s, int32_t i, int64_t ldc, int v) {
        const dbl2 *p = reinterpret_cast<const dbl2 *>(M) + ab_group(s, i, ldc, kAbVecs);
#pragma unroll
        for (int k = 0; k < kAbVecs / 4; k++)
            w[k] = p[64 * k + 4 * (i & 15) + v];
        last = p[16 * (kAbVecs - 1) + (i & 15)];
    }
    // entry d = 10 r + c: A^-1 B (c < 9) or A^-1 b (c = 9) of row r
    __device__ __forceinline__ double get(int d) const {
        const int p = d / 2;
        if (p == kAbVecs - 1)
            return d % 2 ? last.y : last.x;
        return quad_get(d % 2 ? w[p / 4].y : w[p / 4].x, p % 4);
    }
};

// nw[r] += relax ((M xj)_r + du (bmul b_r)), rows in turn
__device__ __forceinline__ void ab_apply(const AbPart &ab, const double xj[9], double du, double bmul, double relax,
                                         double nw[9]) {
#pragma unroll
    for (int r = 0; r < 9; r++) {
        double tt = 0.0;
#pragma unroll
        for (int c = 0; c < 9; c++)
            tt += ab.get(10 * r + c) * xj[c];
        const double b = bmul * ab.get(10 * r + 9);
        nw[r] += relax * (tt + du * b);
    }
}

// doubles 2 P0 .. 2 P1 + 1 of a contiguous run, a quarter per lane of the quad
template <int P0, int P1>
struct QuadPart {
    static constexpr int N = (P1 - P0) / 4 + 1;
    dbl2 w[N];
    __device__ __forceinline__ void load(const double *__restrict__ m, int v) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            w[k] = dbl2{0.0, 0.0};
            if (P0 + 4 * k + v <= P1)
                w[k] = reinterpret_cast<const dbl2 *>(m)[P0 + 4 * k + v];
        }
    }
    __device__ __forceinline__ double get(int e) const {
        const int p = e / 2 - P0;
        return quad_get(e % 2 ? w[p / 4].y : w[p / 4].x, p % 4);
    }
};

// Boundary correction of a Wall_Euler / Wall_NoSlip face to its cell's sweep
// (DNDS_FV_VR.hpp:1577-1657), from the cell's coefficients xi and mean ui of
// this lane's variable v: out = relax A^-1 sum_g w_g |n_g| D0^T W0^2 (uBV -
// u_i).  The four lanes of the cell's quad call it together.
__device__ __forceinline__ void wall_correction(int32_t slot, const double xi[9], double ui, int v,
                                                const double *__restrict__ walls, double relax, int32_t *errw,
                                                double out[9]) {
    const double *wd = walls + kWallEntries * int64_t(wall_of(slot));
    QuadPart<0, 40> ainv;
    QuadPart<0, 13> d0;
    d0.load(wd + kWallD0, v);
    double BCc[9];
#pragma unroll
    for (int r = 0; r < 9; r++)
        BCc[r] = 0.0;
    const double w0 = wd[kWallW0];
#pragma unroll
    for (int g = 0; g < 3; g++) {
        const double gw = g == 1 ? kLine3W1 : kLine3W0;
        const double nx = wd[kWallNrm + 2 * g], ny = wd[kWallNrm + 2 * g + 1];
        double uB = 0;
#pragma unroll
        for (int c = 0; c < 9; c++)
            uB += d0.get(9 * g + c) * xi[c];
        uB += ui;
        double n0, n1;
        stable_normalized(nx, ny, n0, n1);
        const double rho = quad_bcast<0>(uB), m0 = quad_bcast<1>(uB), m1 = quad_bcast<2>(uB);
        double uBV = uB;
        if (!wall_noslip(slot)) {
            const double dd = n0 * m0 + n1 * m1;
            if (v == 1)
                uBV = uB - n0 * dd;
            else if (v == 2)
                uBV = uB - n1 * dd;
        } else if (!(rho > 0)) {
            raise_error(errw, ERR_NONPOSITIVE);
        } else if (v == 1 || v == 2) {
            uBV *= -1;
        }
        const double nl = sqrt(nx * nx + ny * ny);
#pragma unroll
        for (int r = 0; r < 9; r++) {
            double inc = d0.get(9 * g + r) * w0 * w0 * (uBV - ui);
            inc *= nl;
            BCc[r] += inc * gw;
        }
    }
    ainv.load(wd, v);
#pragma unroll
    for (int r = 0; r < 9; r++) {
        double acc = 0;
#pragma unroll
        for (int c = 0; c < 9; c++)
            acc += ainv.get(9 * r + c) * BCc[c];
        out[r] = relax * acc;
    }
}

// where the wave's group of 16 cells starts in a REC array; lane l's variable
// of its cell lies l further on, coefficient c 256 c further on
__device__ __forceinline__ int64_t rec_group(int32_t i) {
    return rec(__builtin_amdgcn_readfirstlane(i) & ~15, 0, 0);
}

// One SOR pass over cells of one colour (SOR_Instead,
// DNDS_FV_VR.hpp:1495-1662), in place on x.  No two cells of a colour are
// neighbours, so the pass equals the reference's sequential in-place scan
// over those cells, and the colours in turn equal its scan in colour-major
// order.  As in the reference, every term is added to the cell's own
// coefficients: the far-field product M x_i and the Wall_Euler / Wall_NoSlip
// corrections take the partial sum after (1 - w) scaling and the faces before
// them.
//
// The cells are the device range [base, base + n): with SOR_Instead the
// device numbering is colour-major.  x and xo are the same array.
template <int NF>
__global__ __launch_bounds__(kBlock, 3) void k_sor(int32_t n, int32_t base, int64_t ldc,
                                                   const int32_t *__restrict__ nbr, const int32_t *__restrict__ sbc,
                                                   const double *__restrict__ M, const double *__restrict__ u,
                                                   const double *x, double *xo, double relax,
                                                   const double *__restrict__ walls, int32_t *errw, int32_t keep) {
    const int32_t t = xcd_block() * blockDim.x + threadIdx.x, v = t & 3;
    // whole groups of 16 cells from the one that holds `base`
    const int32_t i = (base & ~15) + (t >> 2);
    if (i < base || i >= base + n)
        return;
    const uint32_t lane = threadIdx.x & 63;
    int32_t jn[NF];
#pragma unroll
    for (int s = 0; s < NF; s++)
        jn[s] = nbr[s * ldc + i];
    const double ui = u[4 * int64_t(i) + v];
    double nw[9];
#pragma unroll
    for (int r = 0; r < 9; r++)
        nw[r] = (1 - relax) * (x + rec_group(i))[256 * r + lane];
#pragma unroll
    for (int s = 0; s < NF; s++) {
        const int32_t j = jn[s];
        if (j == -2)
            continue;
        AbPart ab;
        ab.load(M, s, i, ldc, v, keep);
        if (j >= 0) {
            double xj[9];
#pragma unroll
            for (int c = 0; c < 9; c++)
                xj[c] = x[rec(j, c, v)];
            ab_apply(ab, xj, u[4 * int64_t(j) + v] - ui, 1.0, relax, nw);
            continue;
        }
        if (is_wall_slot(j)) {
            double cw[9];
            wall_correction(j, nw, ui, v, walls, relax, errw, cw);
#pragma unroll
            for (int r = 0; r < 9; r++)
                nw[r] += cw[r];
            continue;
        }
        const int32_t bc = sbc[s * ldc + i];
        if (bc == BC_WALL) {
#pragma unroll
            for (int r = 0; r < 9; r++)
                nw[r] += relax * ((0.0 - ui) * ab.get(10 * r + 9));
        } else if (is_far(bc)) {
            // M_if times the partial sum, no mean-value term
            double own[9];
#pragma unroll
            for (int c = 0; c < 9; c++)
                own[c] = nw[c];
            ab_apply(ab, own, 0.0, 0.0, relax, nw);
        } else {
            raise_error(errw, ERR_BC);
        }
    }
#pragma unroll
    for (int r = 0; r < 9; r++)
        __builtin_nontemporal_store(nw[r], xo + rec_group(i) + (256 * r + lane));
}

// One block-Jacobi VR sweep, SOR off (ReconstructionJacobiStep,
// DNDS_FV_VR.hpp:1495-1682): new_i = (1-w) x_i + w sum_f [M_if x_j + b_if (u_j - u_i)^T]
// in cell2face order, with the reference's boundary variants: far field
// couples the cell to itself (M_if x_i), a Wall face adds b_if (0 - u_i)^T,
// Wall_Euler / Wall_NoSlip faces add their correction from the old iterate.
//
// diff2 (may be null): receives |x_i - new_i|^2 per cell; the old coefficients
// come from the caches.  With a kernel of its own that reads both arrays again
// (k_rec_diff2) a sweep of dndsmi_reconstruct_to_tolerance takes 49.5 us on 66 k
// cells, 43.5 this way, and 300 / 268 on 524 k.
//
// RESID (the FP64 step of the mixed-precision sweeps): instead of the new
// iterate, writes the increment r = J(x) - x rounded to FP32 into r32 (also the
// start of the FP32 correction sweeps, k_delta32).
template <int NF, bool RESID>
__global__ __launch_bounds__(kBlock, 3) void k_jacobi(int32_t nc, int64_t ldc, const int32_t *__restrict__ nbr,
                                                      const int32_t *__restrict__ sbc,
                                                      const double *__restrict__ M, const double *__restrict__ u,
                                                      const double *__restrict__ x, double *__restrict__ xn,
                                                      double relax, const double *__restrict__ walls, double *corr,
                                                      int32_t *errw, float *__restrict__ r32, int32_t keep,
                                                      double *__restrict__ diff2) {
    __shared__ double tile[9][kBlock];
    const int32_t t = xcd_block() * blockDim.x + threadIdx.x, v = t & 3;
    const bool live = (t >> 2) < nc;
    const int32_t i = live ? t >> 2 : nc - 1;
    const uint32_t lane = threadIdx.x & 63;
    const double *xo = x + rec((t >> 2) & ~15, 0, 0);
    int32_t jn[NF];
    bool wall = false;
#pragma unroll
    for (int s = 0; s < NF; s++) {
        jn[s] = nbr[s * ldc + i];
        wall |= is_wall_slot(jn[s]);
    }
    const double ui = u[4 * int64_t(i) + v];
    // wall corrections first (stored, and read back in their slot), before
    // the loads in flight take the registers
    if (live && wall) {
#pragma unroll 1
        for (int s = 0; s < NF; s++) {
            const int32_t j = s == 0 ? jn[0] : s == 1 ? jn[1] : s == 2 ? jn[2] : jn[NF - 1];
            if (!is_wall_slot(j))
                continue;
            double own[9], cw[9];
#pragma unroll
            for (int r = 0; r < 9; r++)
                own[r] = xo[256 * r + lane];
            wall_correction(j, own, ui, v, walls, relax, errw, cw);
#pragma unroll
            for (int r = 0; r < 9; r++)
                corr[kRec * int64_t(wall_of(j)) + 9 * v + r] = cw[r];
        }
    }
    double nw[9];
#pragma unroll
    for (int r = 0; r < 9; r++) {
        nw[r] = xo[256 * r + lane];
        tile[r][threadIdx.x] = nw[r];
        nw[r] = (1 - relax) * nw[r];
    }
    AbPart ab;
    ab.load(M, 0, i, ldc, v, keep);
    __syncthreads();
    const int32_t i0 = (t - int32_t(threadIdx.x)) >> 2;
#pragma unroll
    for (int s = 0; s < NF; s++) {
        if (s == 3 && jn[s] == -2)
            continue;
        if (s > 0)
            ab.load(M, s, i, ldc, v, keep);
        const int32_t j = jn[s] < 0 ? i : jn[s];
        const double uj = u[4 * int64_t(j) + v];
        double xj[9];
        const uint32_t jl = uint32_t(j - i0);
        if (jl < kBlock / 4) {
#pragma unroll
            for (int c = 0; c < 9; c++)
                xj[c] = tile[c][4 * jl + v];
        } else {
#pragma unroll
            for (int c = 0; c < 9; c++)
                xj[c] = x[rec(j, c, v)];
        }
        const int32_t bc = jn[s] == -1 ? sbc[s * ldc + i] : BC_INNER;
        if (jn[s] >= 0 || is_far(bc)) {
            // far field: M_if x_i (gathered from i), no mean-value term
            const double bmul = jn[s] < 0 ? 0.0 : 1.0;
            ab_apply(ab, xj, bmul * (uj - ui), bmul, relax, nw);
        } else if (bc == BC_WALL) {
#pragma unroll
            for (int r = 0; r < 9; r++)
                nw[r] += relax * ((0.0 - ui) * ab.get(10 * r + 9));
        } else if (is_wall_slot(jn[s])) {
#pragma unroll
            for (int r = 0; r < 9; r++)
                nw[r] += corr[kRec * int64_t(wall_of(jn[s])) + 9 * v + r];
        } else {
            raise_error(errw, ERR_BC);
        }
    }
    if (!live)
        return;
    // the new iterate streams out with non-temporal stores: written once and
    // read by the next launch, it would only displace the neighbours'
    // reconstructions that this sweep still gathers
#pragma unroll
    for (int r = 0; r < 9; r++) {
        if (RESID) {
            const float d = float(nw[r] - xo[256 * r + lane]);
            __builtin_nontemporal_store(d, r32 + rec_group(i) + (256 * r + lane));
        } else
            __builtin_nontemporal_store(nw[r], xn + rec_group(i) + (256 * r + lane));
    }
    if (!RESID && diff2) {
        double d[9];
#pragma unroll
        for (int r = 0; r < 9; r++)
            d[r] = xo[256 * r + lane] - nw[r];
        const double sum = quad_norm2(d);
        if (v == 3)
            diff2[i] = sum;
    }
}

// The sweep of a small mesh: 16 lanes per cell, a quad per slot.  Small sweeps
// are bound by one cell's chain of loads and sums, which k_jacobi runs slot
// after slot (and a corner cell's two walls one after the other, 4 us each);
// here the slots' terms form side by side and the first quad adds them in the
// slots' order.  An absent slot adds -0, which changes no bit.
template <int NF, bool RESID>
__global__ __launch_bounds__(64) void k_jacobi_wide(int32_t nc, int64_t ldc, const int32_t *__restrict__ nbr,
                                                    const int32_t *__restrict__ sbc, const double *__restrict__ M,
                                                    const double *__restrict__ u, const double *__restrict__ x,
                                                    double *__restrict__ xn, double relax,
                                                    const double *__restrict__ walls, int32_t *errw,
                                                    float *__restrict__ r32, double *__restrict__ diff2) {
    const int32_t t = xcd_block() * 64 + threadIdx.x, i = t >> 4;
    const int s = (t >> 2) & 3, v = t & 3;
    if (i >= nc)
        return;
    const int32_t jn = s < NF ? nbr[s * ldc + i] : -2;
    double term[9], own[9];
#pragma unroll
    for (int r = 0; r < 9; r++)
        term[r] = -0.0;
    const double ui = u[4 * int64_t(i) + v];
    if (s == 0 || is_wall_slot(jn))
#pragma unroll
        for (int r = 0; r < 9; r++)
            own[r] = x[rec(i, r, v)];
    if (is_wall_slot(jn)) {
        wall_correction(jn, own, ui, v, walls, relax, errw, term);
    } else if (jn != -2) {
        AbPart ab;
        ab.load_each(M, s, i, ldc, v);
        const int32_t j = jn < 0 ? i : jn;
        const double uj = u[4 * int64_t(j) + v];
        double xj[9];
#pragma unroll
        for (int c = 0; c < 9; c++)
            xj[c] = x[rec(j, c, v)];
        const int32_t bc = jn == -1 ? sbc[s * ldc + i] : BC_INNER;
        if (jn >= 0 || is_far(bc)) {
            const double bmul = jn < 0 ? 0.0 : 1.0, du = bmul * (uj - ui);
#pragma unroll
            for (int r = 0; r < 9; r++) {
                double tt = 0.0;
#pragma unroll
                for (int c = 0; c < 9; c++)
                    tt += ab.get(10 * r + c) * xj[c];
                const double b = bmul * ab.get(10 * r + 9);
                term[r] = relax * (tt + du * b);
            }
        } else if (bc == BC_WALL) {
#pragma unroll
            for (int r = 0; r < 9; r++)
                term[r] = relax * ((0.0 - ui) * ab.get(10 * r + 9));
        } else {
            raise_error(errw, ERR_BC);
        }
    }
    double nw[9];
#pragma unroll
    for (int r = 0; r < 9; r++) {
        nw[r] = (1 - relax) * own[r];
#pragma unroll
        for (int q = 0; q < NF; q++)
            nw[r] += row_ahead(term[r], q);
    }
    if (s > 0)
        return;
#pragma unroll
    for (int r = 0; r < 9; r++) {
        if (RESID)
            r32[rec(i, r, v)] = float(nw[r] - own[r]);
        else
            xn[rec(i, r, v)] = nw[r];
    }
    if (!RESID && diff2) {
        double d[9];
#pragma unroll
        for (int r = 0; r < 9; r++)
            d[r] = own[r] - nw[r];
        const double sum = quad_norm2(d);
        if (v == 3)
            diff2[i] = sum;
    }
}

// the increment's squared norm per cell where the sweep does not give it
__global__ __launch_bounds__(kBlock) void k_rec_diff2(int32_t nc, const double *__restrict__ x,
                                                      const double *__restrict__ xn, double *__restrict__ diff2) {
    const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if ((t >> 2) >= nc)
        return;
    const int64_t o = rec((t >> 2) & ~15, 0, 0) + (threadIdx.x & 63);
    double d[9];
#pragma unroll
    for (int r = 0; r < 9; r++)
        d[r] = x[o + 256 * r] - xn[o + 256 * r];
    const double sum = quad_norm2(d);
    if ((t & 3) == 3)
        diff2[t >> 2] = sum;
}

// sums of the cells' diff2, 256 cells each in a fixed tree, one per wave, into
// pinned host memory: 16 a workgroup, stored as one run of 128 bytes
__global__ __launch_bounds__(1024) void k_diff2_sums(int32_t nc, const double *__restrict__ diff2, double *part) {
    __shared__ double sums[16];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int64_t i = (int64_t(blockIdx.x) * 16 + wave) * 256 + lane;
    double e[4];
#pragma unroll
    for (int q = 0; q < 4; q++)
        e[q] = i + 64 * q < nc ? diff2[i + 64 * q] : 0.0;
    double a = (e[0] + e[2]) + (e[1] + e[3]);
    for (int off = 32; off > 0; off >>= 1)
        a += __shfl_down(a, off, 64);
    if (lane == 0)
        sums[wave] = a;
    __syncthreads();
    if (threadIdx.x < 16)
        part[int64_t(blockIdx.x) * 16 + threadIdx.x] = sums[threadIdx.x];
}

// Read-bandwidth probe of the sweep's dominant stream: every cell streams its
// slots' A^-1 B, A^-1 b with k_jacobi's loads (four lanes per cell, 16 bytes
// each, the same share of the stream kept in the Infinity Cache, the same slots
// skipped) and none of the sweep's gathers, and writes one double per lane.
// Its rate is the ceiling of the sweep's streaming part in this layout; it says
// nothing about another one.
template <int NF>
__global__ __launch_bounds__(kBlock) void k_read_probe(int32_t nc, int64_t ldc, const int32_t *__restrict__ nbr,
                                                       const double *__restrict__ M, double *__restrict__ out,
                                                       int32_t keep) {
    const int32_t t = xcd_block() * blockDim.x + threadIdx.x, i = t >> 2, v = t & 3;
    if (i >= nc)
        return;
    double a = 0.0;
#pragma unroll
    for (int s = 0; s < NF; s++) {
        if (nbr[s * ldc + i] == -2)
            continue;
        AbPart ab;
        ab.load(M, s, i, ldc, v, keep);
#pragma unroll
        for (int k = 0; k < kAbVecs / 4; k++)
            a += ab.w[k].x + ab.w[k].y;
        a += v == 0 ? ab.last.x + ab.last.y : 0.0;
    }
    out[4 * int64_t(i) + v] = a;
}

// Linear part of the Wall_Euler / Wall_NoSlip correction (wall_correction)
// for a correction d of the reconstruction: the wall state is the
// reconstructed value D d with the normal momentum removed (Wall_Euler) or
// the momentum reversed (Wall_NoSlip), both linear, and the cell mean drops
// out.  di: this lane's variable; the cell's quad calls it together.
__device__ __forceinline__ void wall_correction_lin(int32_t slot, const float di[9], int v,
                                                    const double *__restrict__ walls, float relax, float out[9]) {
    const double *wd = walls + kWallEntries * int64_t(wall_of(slot));
    QuadPart<0, 40> ainv;
    QuadPart<0, 13> d0;
    d0.load(wd + kWallD0, v);
    float BCc[9];
#pragma unroll
    for (int r = 0; r < 9; r++)
        BCc[r] = 0.f;
    const float w0 = float(wd[kWallW0]);
#pragma unroll
    for (int g = 0; g < 3; g++) {
        const float gw = float(g == 1 ? kLine3W1 : kLine3W0);
        const double nx = wd[kWallNrm + 2 * g], ny = wd[kWallNrm + 2 * g + 1];
        float uB = 0.f;
#pragma unroll
        for (int c = 0; c < 9; c++)
            uB = fmaf(float(d0.get(9 * g + c)), di[c], uB);
        double n0, n1;
        stable_normalized(nx, ny, n0, n1);
        const float m0 = quad_bcast<1>(uB), m1 = quad_bcast<2>(uB);
        float uBV = uB;
        if (!wall_noslip(slot)) {
            const float dd = float(n0) * m0 + float(n1) * m1;
            if (v == 1)
                uBV = uB - float(n0) * dd;
            else if (v == 2)
                uBV = uB - float(n1) * dd;
        } else if (v == 1 || v == 2) {
            uBV = -uB;
        }
        const float nl = float(sqrt(nx * nx + ny * ny));
#pragma unroll
        for (int r = 0; r < 9; r++)
            BCc[r] += float(d0.get(9 * g + r)) * w0 * w0 * uBV * nl * gw;
    }
    ainv.load(wd, v);
#pragma unroll
    for (int r = 0; r < 9; r++) {
        float acc = 0.f;
#pragma unroll
        for (int c = 0; c < 9; c++)
            acc = fmaf(float(ainv.get(9 * r + c)), BCc[c], acc);
        out[r] = relax * acc;
    }
}

// FP32 correction sweep of the mixed-precision reconstruction.  The Jacobi
// map is affine, J(x) = G x + c with G x = (1-w) x + w sum_f M_if x_j (far
// field faces couple the cell to itself), so with r = J(x) - x the sweeps
//   d_0 = r,  d_{k+1} = G d_k + r
// give x + d_k = J^{k+1}(x) exactly in real arithmetic: n - 1 FP32 sweeps
// after one FP64 step reproduce n FP64 sweeps, with FP32 rounding confined
// to the correction d (iterative refinement).  M is read as FP32.  LAST adds
// the correction to the FP64 iterate in place.  Wall_Euler / Wall_NoSlip
// faces contribute the linear part of their boundary correction (the wall
// state is linear in the reconstructed value there).  Four lanes per cell, as
// in k_jacobi.
template <int NF, bool LAST>
__global__ __launch_bounds__(kBlock, 4) void k_delta32(int32_t nc, int64_t ldc, const int32_t *__restrict__ nbr,
                                                       const int32_t *__restrict__ sbc,
                                                       const float *__restrict__ M32, const float *__restrict__ r32,
                                                       const float *__restrict__ din, float *__restrict__ dout,
                                                       float relax, double *__restrict__ x,
                                                       const double *__restrict__ walls, float *corr, int32_t keep) {
    const int32_t t = xcd_block() * blockDim.x + threadIdx.x, i = t >> 2, v = t & 3;
    if (i >= nc)
        return;
    const uint32_t lane = threadIdx.x & 63;
    const float *xo = din + rec_group(i);
    int32_t jn[NF];
    bool wall = false;
#pragma unroll
    for (int s = 0; s < NF; s++) {
        jn[s] = nbr[s * ldc + i];
        wall |= is_wall_slot(jn[s]);
    }
    // wall corrections first, as in k_jacobi
    if (wall) {
#pragma unroll 1
        for (int s = 0; s < NF; s++) {
            const int32_t j = s == 0 ? jn[0] : s == 1 ? jn[1] : s == 2 ? jn[2] : jn[NF - 1];
            if (!is_wall_slot(j))
                continue;
            float own[9], cw[9];
#pragma unroll
            for (int r = 0; r < 9; r++)
                own[r] = xo[256 * r + lane];
            wall_correction_lin(j, own, v, walls, relax, cw);
#pragma unroll
            for (int r = 0; r < 9; r++)
                corr[kRec * int64_t(wall_of(j)) + 9 * v + r] = cw[r];
        }
    }
    float nw[9];
#pragma unroll
    for (int r = 0; r < 9; r++)
        nw[r] = (1.0f - relax) * xo[256 * r + lane];
    constexpr int kW = kAb32Vecs / 4;
#pragma unroll
    for (int s = 0; s < NF; s++) {
        if (s == 3 && jn[s] == -2)
            continue;
        const int32_t g = __builtin_amdgcn_readfirstlane(i);
        const ab_stream rs(M32 + 4 * ab_group(s, g, ldc, kAb32Vecs), 256 * kAb32Vecs);
        const uint32_t cl = i & 15;
        flt4 w[kW], last;
        if (((g >> 6) & 63) < keep) {
#pragma unroll
            for (int k = 0; k < kW; k++)
                w[k] = rs.get<flt4, false>((4 * cl + v) * 16, 1024 * k);
            last = rs.get<flt4, false>(cl * 16, 256 * (kAb32Vecs - 1));
        } else {
#pragma unroll
            for (int k = 0; k < kW; k++)
                w[k] = rs.get<flt4, true>((4 * cl + v) * 16, 1024 * k);
            last = rs.get<flt4, true>(cl * 16, 256 * (kAb32Vecs - 1));
        }
        const int32_t j = jn[s] < 0 ? i : jn[s];
        float dj[9];
#pragma unroll
        for (int c = 0; c < 9; c++)
            dj[c] = din[rec(j, c, v)];
        const int32_t bc = jn[s] == -1 ? sbc[s * ldc + i] : BC_INNER;
        if (is_wall_slot(jn[s])) {
#pragma unroll
            for (int r = 0; r < 9; r++)
                nw[r] += corr[kRec * int64_t(wall_of(jn[s])) + 9 * v + r];
        } else if (bc != BC_WALL) { // far field: d_i; a Wall face's constant term is in r only
#pragma unroll
            for (int r = 0; r < 9; r++) {
                float tt = 0.f;
#pragma unroll
                for (int c = 0; c < 9; c++) {
                    const int e = 9 * r + c, k = e / 4;
                    const float m = k == kAb32Vecs - 1 ? last[e % 4]
                                                       : quad_get(float(w[k < 20 ? k / 4 : 0][e % 4]), k % 4);
                    tt = fmaf(m, dj[c], tt);
                }
                nw[r] = fmaf(relax, tt, nw[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 9; r++) {
        const float d = nw[r] + (r32 + rec_group(i))[256 * r + lane];
        if (LAST)
            (x + rec_group(i))[256 * r + lane] += double(d);
        else
            __builtin_nontemporal_store(d, dout + rec_group(i) + (256 * r + lane)); // streamed, as in k_jacobi
    }
}

// A^-1 B in FP32, one thread per 16-byte vector of the FP32 stream, in the
// stream's order (with consecutive threads on consecutive cells every 64-byte
// piece was touched four times: 901 us on 264 k cells, 161 now)
__global__ __launch_bounds__(kBlock) void k_m_to_f32(int32_t nfmax, int64_t ldc, const double *__restrict__ M,
                                                     float *__restrict__ M32) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= int64_t(nfmax) * kAb32Vecs * ldc)
        return;
    const int64_t group = t / (16 * kAb32Vecs);
    const int w = int(t % (16 * kAb32Vecs)); // ab_vec's place in a group of 16 cells
    const bool last = w >= 16 * (kAb32Vecs - 1);
    const int q = last ? kAb32Vecs - 1 : 4 * (w / 64) + w % 4;
    const int64_t i = 16 * (group % (ldc / 16)) + (last ? w % 16 : w / 4 % 16);
    const int s = int(group / (ldc / 16));
    flt4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int k = 4 * q + e, d = 10 * (k / 9) + k % 9;
        o[e] = k < 81 ? float(M[ab_vec(s, d / 2, i, ldc, kAbVecs) * 2 + d % 2]) : 0.f;
    }
    reinterpret_cast<flt4 *>(M32)[t] = o;
}

// EvaluateDt face loop (DNDS_FV_EulerEvaluator.cpp:25-137): lambdaFace and
// deltaLambdaFace per face (muGas = 0).
__global__ __launch_bounds__(kBlock) void k_dt_face(int32_t nf, int64_t ldf, const int32_t *__restrict__ f2c,
                                                    const double *__restrict__ fnc, const double *__restrict__ u,
                                                    GasParams gp, const double *__restrict__ farea,
                                                    const double *__restrict__ vol, double *__restrict__ lf,
                                                    double *__restrict__ dlf, int32_t *errw) {
    const double gamma = gp.gamma;
    const int32_t f = xcd_block() * blockDim.x + threadIdx.x;
    if (f >= nf)
        return;
    const int32_t L = f2c[f], R = f2c[ldf + f];
    double n0, n1;
    normalized(fnc[f], fnc[ldf + f], n0, n1);
    double UL[4];
    for (int k = 0; k < 4; k++)
        UL[k] = u[4 * int64_t(L) + k];
    double uMean[4] = {UL[0], UL[1], UL[2], UL[3]};
    double pL, asqrL, HL, pR, asqrR, HR;
    const double vL0 = UL[1] / UL[0], vL1 = UL[2] / UL[0];
    double vR0 = vL0, vR1 = vL1;
    ideal_gas_thermal(UL[3], UL[0], vL0 * vL0 + vL1 * vL1, gamma, pL, asqrL, HL);
    pR = pL, HR = HL, asqrR = asqrL;
    if (R >= 0) {
        double UR[4];
        for (int k = 0; k < 4; k++)
            UR[k] = u[4 * int64_t(R) + k];
        for (int k = 0; k < 4; k++)
            uMean[k] = (uMean[k] + UR[k]) * 0.5;
        vR0 = UR[1] / UR[0], vR1 = UR[2] / UR[0];
        ideal_gas_thermal(UR[3], UR[0], vR0 * vR0 + vR1 * vR1, gamma, pR, asqrR, HR);
    }
    if (!(uMean[0] > 0))
        raise_error(errw, ERR_NONPOSITIVE);
    const double veloNMean = 0.5 * ((vL0 + vR0) * n0 + (vL1 + vR1) * n1);
    const double pMean = (pL + pR) * 0.5;
    const double aMean = sqrt(gamma * pMean / uMean[0]);
    const double lambdaConvection = fabs(veloNMean) + aMean;
    if (gp.mu > 0) { // DNDS_FV_EulerEvaluator.cpp:79-119, NS_2D
        const double lamVis = sutherland_mu(gp, pMean, uMean[0]) / uMean[0] * fmax(4. / 3., gamma / gp.pr);
        const double volL = vol[L], volR = R >= 0 ? vol[R] : volL;
        lf[f] = lambdaConvection + lamVis * farea[f] * (1. / volL + 1. / volR);
    } else {
        lf[f] = lambdaConvection;
    }
    dlf[f] = fabs((vR0 - vL0) * n0 + (vR1 - vL1) * n1) + sqrt(fabs(asqrR - asqrL)) * 0.7071;
}

// EvaluateDt cell loop (DNDS_FV_EulerEvaluator.cpp:132-150): lambdaCell from
// the faces in ascending order, dt_i and the block minimum.
template <int NF>
__global__ __launch_bounds__(kBlock) void k_dt_cell(int32_t nc, int64_t ldc, const int32_t *__restrict__ gat,
                                                    const double *__restrict__ lf, const double *__restrict__ farea,
                                                    const double *__restrict__ vol, double cfl, double max_dt,
                                                    double *__restrict__ dt, double *__restrict__ part) {
    __shared__ double red[kBlock];
    const int32_t i = xcd_block() * blockDim.x + threadIdx.x;
    double d = 3e200;
    if (i < nc) {
        double lam = 0.0;
#pragma unroll
        for (int s = 0; s < NF; s++) {
            const int32_t g = gat[s * ldc + i];
            if (g < 0)
                continue;
            const int32_t f = g >> 1;
            lam += lf[f] * farea[f];
        }
        d = fmin(cfl * vol[i] / (lam + 1e-100), max_dt);
        dt[i] = d;
    }
    red[threadIdx.x] = d;
    __syncthreads();
    if (threadIdx.x >= 64)
        return;
    d = tree256(red, Min());
    if (threadIdx.x == 0)
        part[blockIdx.x] = d;
}

__global__ __launch_bounds__(kBlock) void k_min_final(int32_t n, const double *__restrict__ part,
                                                      double *__restrict__ out, double *host_out, int32_t *errw) {
    __shared__ double red[kBlock];
    double d = 3e200;
    for (int32_t k = threadIdx.x; k < n; k += kBlock)
        d = fmin(d, part[k]);
    red[threadIdx.x] = d;
    __syncthreads();
    if (threadIdx.x >= 64)
        return;
    d = tree256(red, Min());
    if (threadIdx.x == 0) {
        out[0] = d;
        *host_out = d;
        if (!isfinite(d))
            raise_error(errw, ERR_NAN);
    }
}

__global__ __launch_bounds__(kBlock) void k_fill_from(int32_t n, const double *__restrict__ src,
                                                      double *__restrict__ dst) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        dst[i] = src[0];
}

// EvaluateRHS face loop (DNDS_FV_EulerEvaluator.cpp:215-492): left/right
// states at the three LINE_3 points, Riemann flux, flux-balance fluxes,
// Gauss sum.  Stores the integrated F, FLfix, FRfix per face in its cells'
// slots.
//
// MIXED: the face reconstruction D0 . x runs in FP32 (FP32 bases, FP32
// accumulation) and the integrated fluxes are stored in FP32; the Riemann
// solver and the boundary states stay FP64.
//
// VIS (muGas > 0, FP64 only): also the gradients of both sides at each point
// from rows 1, 2 of the DiBj blocks (DNDS_FV_EulerEvaluator.cpp:297-346), the
// face gradient with the jump term over distGRP = 2 min(V) / A, which walls
// push to 3e200 (:356-395, USE_DISABLE_DIST_GRP_FIX_AT_WALL), and fluxFace's
// viscous flux (DNDS_FV_EulerEvaluator.hpp:397-430, 574-577).
struct FaceArgs {
    int64_t ldf;
    int32_t nfmax;
    const int32_t *f2c, *fbc;
    const double *fxy, *cmom, *fn, *fctr, *dlf, *u, *x;
    GasParams gp;
    double t;
    const uint8_t *fpos;
    double *fslot;
    float *fslot32;
    int32_t *errw;
    const double *cscale, *vol, *farea; // VIS
    // the steps' limiter leaves its unlimited cells in x and flags the others
    const double *xalt;
    const uint8_t *limf;

    __device__ const double *rec_of(int32_t cell) const { return (limf && limf[cell]) ? xalt : x; }
};

// reconstructed increments D0 . x of one side's cell at NP of the face's
// points from point g0 on; the bases D0 (row 0 of the DiBj blocks) are
// evaluated from the points' scaled coordinates and the cell's moments, in c
// order as stored bases would be read.  MIXED: the bases are rounded to FP32
// and the products accumulated in FP32.
template <int NP, bool MIXED>
__device__ __forceinline__ void face_increments(const double *xs, const double *cmom, const dbl2 *xy, int32_t cell,
                                                int sd, int g0, double inc[NP][4]) {
    double pX[NP][4], pY[NP][4];
#pragma unroll
    for (int g = 0; g < NP; g++) {
        const dbl2 q = __builtin_nontemporal_load(xy + 64 * (sd * 3 + g0 + g));
        int_powers(q.x, pX[g]);
        int_powers(q.y, pY[g]);
    }
    float acc[NP][4];
#pragma unroll
    for (int g = 0; g < NP; g++)
#pragma unroll
        for (int v = 0; v < 4; v++)
            inc[g][v] = 0.0, acc[g][v] = 0.f;
#pragma unroll
    for (int c = 0; c < 9; c++) {
        const double m = cmom[blk64(cell, 9) + 64 * c];
        const dbl2 *xq = reinterpret_cast<const dbl2 *>(xs + rec(cell, c, 0));
        const dbl2 xa = xq[0], xb = xq[1];
        const double xc[4] = {xa.x, xa.y, xb.x, xb.y};
#pragma unroll
        for (int g = 0; g < NP; g++) {
            const double d = pX[g][kBX[c + 1]] * pY[g][kBY[c + 1]] - m;
            if (MIXED) {
                const float d32 = float(d);
#pragma unroll
                for (int v = 0; v < 4; v++)
                    acc[g][v] = fmaf(d32, float(xc[v]), acc[g][v]);
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    inc[g][v] += d * xc[v];
            }
        }
    }
    if (MIXED)
#pragma unroll
        for (int g = 0; g < NP; g++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                inc[g][v] = double(acc[g][v]);
}

// the gradient of one side's cell at point g
__device__ __forceinline__ void face_gradient(const double *xs, const double *cscale, const dbl2 *xy, int32_t cell,
                                              int sd, int g, double G[2][4]) {
    const dbl2 q = xy[64 * (sd * 3 + g)];
    double px[4], py[4];
    int_powers(q.x, px);
    int_powers(q.y, py);
    const dbl2 sc = reinterpret_cast<const dbl2 *>(cscale)[cell];
    const double isx = 1.0 / sc.x, isy = 1.0 / sc.y; // the rows' scales as reciprocals
#pragma unroll
    for (int d = 0; d < 2; d++)
#pragma unroll
        for (int v = 0; v < 4; v++)
            G[d][v] = 0.0;
    // d/dx: bx X^(bx-1) Y^by / sx, d/dy: by X^bx Y^(by-1) / sy
#pragma unroll
    for (int c = 0; c < 9; c++) {
        const int bx = kBX[c + 1], by = kBY[c + 1];
        const dbl2 *xq = reinterpret_cast<const dbl2 *>(xs + rec(cell, c, 0));
        const dbl2 xa = xq[0], xb = xq[1];
        const double xc[4] = {xa.x, xa.y, xb.x, xb.y};
        if (bx > 0) {
            const double dx = double(bx) * px[bx - 1] * py[by] * isx;
#pragma unroll
            for (int v = 0; v < 4; v++)
                G[0][v] += dx * xc[v];
        }
        if (by > 0) {
            const double dy = double(by) * px[bx] * py[by - 1] * isy;
#pragma unroll
            for (int v = 0; v < 4; v++)
                G[1][v] += dy * xc[v];
        }
    }
}

// adds the viscous flux at a point to F, from the gradients of both sides
// (gR = gL at a boundary face), minVol the smaller volume
__device__ __forceinline__ void add_viscous_flux(const GasParams &gp, const double gL[2][4], const double gR[2][4],
                                                 double minVol, double area, int32_t bc, double n0, double n1,
                                                 const double ULxy[4], const double URxy[4], double F[4]) {
    double distGRP = minVol / area * 2;
    distGRP += (bc == BC_WALL_EULER || bc == BC_WALL_NOSLIP) ? 3e200 : 0.0;
    double GM[2][4], UM[4];
#pragma unroll
    for (int d = 0; d < 2; d++) {
        const double nd = d ? n1 : n0;
#pragma unroll
        for (int v = 0; v < 4; v++)
            GM[d][v] = (gR[d][v] + gL[d][v]) * 0.5 + (1.0 / distGRP) * (nd * (URxy[v] - ULxy[v]));
    }
#pragma unroll
    for (int v = 0; v < 4; v++)
        UM[v] = 0.5 * (ULxy[v] + URxy[v]);
    const double vm0 = UM[1] / UM[0], vm1 = UM[2] / UM[0];
    double pM, aM, HM;
    ideal_gas_thermal(UM[3], UM[0], vm0 * vm0 + vm1 * vm1, gp.gamma, pM, aM, HM);
    const double muf = sutherland_mu(gp, pM, UM[0]);
    const double k = gp.cp * (muf - muf) / 0.9 + gp.cp * muf / gp.pr;
    double vn[4];
    viscous_flux_n(UM, GM, n0, n1, bc == BC_WALL_NOSLIP, gp.gamma, muf, k, gp.cp, vn);
#pragma unroll
    for (int v = 0; v < 4; v++)
        F[v] += vn[v];
}

// A quad per face, lane g at point g (the fourth repeats the third's): the
// flux's long chain of divisions and square roots runs once instead of three
// times in turn.  A few hundred boundary faces on one lane each were a launch
// of 15 to 35 us after the inner faces', all of it that chain; as quads in
// front of the inner faces' workgroups they cost nothing of their own (33 k
// cells: 16 + 20 us before, 17 now; viscous 27 + 27, 26).  Each lane sums the points in order (the others' values from
// their lanes) and stores one of the face's four terms.
template <bool BOUNDARY, bool MIXED, bool VIS>
__device__ __forceinline__ void face_quad(const FaceArgs &fa, int32_t f) {
    const int lane = threadIdx.x & 3, g = lane < 3 ? lane : 2;
    const int32_t L = fa.f2c[f], R = fa.f2c[fa.ldf + f];
    if (!BOUNDARY && R < 0)
        return;
    double uL[4], uR[4], inc[1][4], ULxy[4], URxy[4], URm[4];
    const dbl2 *xy = reinterpret_cast<const dbl2 *>(fa.fxy) + blk64(f, 6);
#pragma unroll
    for (int k = 0; k < 4; k++)
        uL[k] = fa.u[4 * int64_t(L) + k];
    const double nx = fa.fn[blk64(f, 6) + 64 * (2 * g)], ny = fa.fn[blk64(f, 6) + 64 * (2 * g + 1)];
    const double dl = fa.dlf[f];
    const int32_t bc = BOUNDARY ? fa.fbc[f] : BC_INNER;
    const int32_t pos = fa.fpos[f];
    face_increments<1, MIXED>(fa.rec_of(L), fa.cmom, xy, L, 0, g, inc);
    compress_rec_part(uL, inc[0], ULxy);
    double n0, n1;
    normalized(nx, ny, n0, n1);
    const double nl = sqrt(nx * nx + ny * ny);
    bool ok = true;
    if (BOUNDARY) {
        const double px = fa.fctr[f], py = fa.fctr[fa.ldf + f];
        ok &= boundary_value(fa.gp, ULxy, n0, n1, px, py, fa.t, bc, URxy);
        ok &= boundary_value(fa.gp, uL, n0, n1, px, py, fa.t, bc, URm);
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++)
            uR[k] = URm[k] = fa.u[4 * int64_t(R) + k];
        face_increments<1, MIXED>(fa.rec_of(R), fa.cmom, xy, R, 1, g, inc);
        compress_rec_part(uR, inc[0], URxy);
    }
    double F[4], FL[4], FR[4];
    ok = ok && balance_fluxes(fa.gp, uL, URm, n0, n1, FL, FR);
    ok = ok && riemann_face(fa.gp, ULxy, URxy, n0, n1, dl, F);
    if (VIS) {
        double gL[2][4], gR[2][4], minVol = fa.vol[L];
        face_gradient(fa.rec_of(L), fa.cscale, xy, L, 0, g, gL);
        if (!BOUNDARY) {
            face_gradient(fa.rec_of(R), fa.cscale, xy, R, 1, g, gR);
            minVol = fmin(minVol, fa.vol[R]);
        }
        add_viscous_flux(fa.gp, gL, BOUNDARY ? gL : gR, minVol, fa.farea[f], bc, n0, n1, ULxy, URxy, F);
    }
    if (!ok)
        raise_error(fa.errw, ERR_NONPOSITIVE);
    const double w = g == 1 ? kLine3W1 : kLine3W0;
    double term[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const double a = F[v] * nl, b = FL[v] * nl, c = FR[v] * nl;
        const double pa = a * w, pb = b * w, pc = c * w;
        double sa = 0.0, sb = 0.0, sc = 0.0;
#pragma unroll
        for (int q = 0; q < 3; q++)
            sa += quad_get(pa, q), sb += quad_get(pb, q), sc += quad_get(pc, q);
        // signed as the cells apply them
        term[v] = lane == 0 ? sa : lane == 1 ? -sb : lane == 2 ? -sa : sc;
    }
    if (BOUNDARY && lane > 1)
        return;
    const int64_t o = (lane < 2 ? quad64(L, 2 * fa.nfmax, 2 * (pos & 15)) : quad64(R, 2 * fa.nfmax, 2 * (pos >> 4))) +
                      256 * (lane & 1);
    if (MIXED) {
        *reinterpret_cast<flt4 *>(fa.fslot32 + o) =
            flt4{float(term[0]), float(term[1]), float(term[2]), float(term[3])};
    } else {
        dbl2 *p = reinterpret_cast<dbl2 *>(fa.fslot + o);
        p[0] = dbl2{term[0], term[1]}, p[1] = dbl2{term[2], term[3]};
    }
}

// The first nbb workgroups (a multiple of the XCDs) take the nb boundary faces
// of `list`, the others the n faces' inner ones.
template <bool MIXED, bool VIS>
__global__ __launch_bounds__(64) void k_rhs_face_quads(int32_t nb, int32_t nbb, const int32_t *__restrict__ list,
                                                           int32_t n, FaceArgs fa) {
    const int32_t b = blockIdx.x;
    if (b < nbb) {
        const int32_t q = int32_t(b * blockDim.x + threadIdx.x) >> 2;
        if (q < nb)
            face_quad<true, MIXED, VIS>(fa, list[q]);
    } else {
        const int32_t f = int32_t(xcd_block(b - nbb, gridDim.x - nbb) * blockDim.x + threadIdx.x) >> 2;
        if (f < n)
            face_quad<false, MIXED, VIS>(fa, f);
    }
}

// One lane per inner face, for meshes that fill the chip this way; the three
// points in turn.  Boundary faces as in k_rhs_face_quads.
//
// STRAIGHT (a mesh whose face normals are bitwise equal at the three points,
// as on straight edges): the unit normal, |n| and the flux-balance fluxes are
// computed at point 0 and reused, which yields the same bits as recomputing
// them from the same inputs.
//
// The members of `fa` that the inner faces use come once more as parameters
// (the launch takes them from it): pointers inside a struct are not restrict,
// and the kernel took 133 us instead of 112 on 500 k cells.
template <bool MIXED, bool STRAIGHT, bool VIS>
__global__ __launch_bounds__(kBlock, VIS ? 2 : 1) void k_rhs_face(
    int32_t nb, int32_t nbb, const int32_t *__restrict__ list, FaceArgs fa, int32_t n, int64_t ldf, int nfmax,
    const int32_t *__restrict__ f2c, const double *__restrict__ fxy, const double *__restrict__ cmom,
    const double *__restrict__ fn, const double *__restrict__ dlf, const double *__restrict__ u,
    const double *__restrict__ x, GasParams gp, const uint8_t *__restrict__ fpos,
    double *__restrict__ fslot, float *__restrict__ fslot32, int32_t *errw, const double *__restrict__ cscale,
    const double *__restrict__ vol, const double *__restrict__ farea, const double *__restrict__ xalt,
    const uint8_t *__restrict__ limf) {
    static_assert(!(VIS && MIXED), "the viscous terms run in FP64 only");
    const int32_t b = blockIdx.x;
    if (b < nbb) {
        const int32_t q = int32_t(b * blockDim.x + threadIdx.x) >> 2;
        if (q < nb)
            face_quad<true, MIXED, VIS>(fa, list[q]);
        return;
    }
    const int32_t f = xcd_block(b - nbb, gridDim.x - nbb) * blockDim.x + threadIdx.x;
    if (f >= n)
        return;
    const int32_t L = f2c[f], R = f2c[ldf + f];
    if (R < 0)
        return;
    double uL[4], uR[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        uL[k] = u[4 * int64_t(L) + k];
    double incL[3][4], incR[3][4];
    const dbl2 *xy = reinterpret_cast<const dbl2 *>(fxy) + blk64(f, 6);
#pragma unroll 1
    for (int sd = 0; sd < 2; sd++) {
        double inc[3][4];
        const int32_t cell = sd ? R : L;
        face_increments<3, MIXED>((limf && limf[cell]) ? xalt : x, cmom, xy, cell, sd, 0, inc);
#pragma unroll
        for (int g = 0; g < 3; g++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                if (sd)
                    incR[g][v] = inc[g][v];
                else
                    incL[g][v] = inc[g][v];
            }
    }
#pragma unroll
    for (int k = 0; k < 4; k++)
        uR[k] = u[4 * int64_t(R) + k];
    const double dl = dlf[f];
    double acc[12];
#pragma unroll
    for (int k = 0; k < 12; k++)
        acc[k] = 0.0;
    bool ok = true, okb = true;
    double n0, n1, nl, FL[4], FR[4];
    // the viscous variant keeps its points apart: unrolled, their gradient
    // work would be scheduled together and crowd the registers
#pragma unroll(VIS ? 1 : 3)
    for (int g = 0; g < 3; g++) {
        double ULxy[4], URxy[4];
        if (!STRAIGHT || g == 0) {
            const double nx = fn[blk64(f, 6) + 64 * (2 * g)], ny = fn[blk64(f, 6) + 64 * (2 * g + 1)];
            normalized(nx, ny, n0, n1);
            nl = sqrt(nx * nx + ny * ny);
        }
        compress_rec_part(uL, incL[g], ULxy);
        compress_rec_part(uR, incR[g], URxy);
        double F[4];
        if (!STRAIGHT || g == 0)
            okb = ok && balance_fluxes(gp, uL, uR, n0, n1, FL, FR);
        ok &= ok && okb && riemann_face(gp, ULxy, URxy, n0, n1, dl, F);
        if (VIS) {
            // formed here rather than kept for all three points
            double gL[2][4], gR[2][4];
            face_gradient((limf && limf[L]) ? xalt : x, cscale, xy, L, 0, g, gL);
            face_gradient((limf && limf[R]) ? xalt : x, cscale, xy, R, 1, g, gR);
            add_viscous_flux(gp, gL, gR, fmin(vol[L], vol[R]), farea[f], BC_INNER, n0, n1, ULxy, URxy, F);
        }
        const double w = g == 1 ? kLine3W1 : kLine3W0;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const double a = F[v] * nl, b = FL[v] * nl, c = FR[v] * nl;
            acc[v] += a * w;
            acc[4 + v] += b * w;
            acc[8 + v] += c * w;
        }
    }
    if (!ok)
        raise_error(errw, ERR_NONPOSITIVE);
    // each side's two terms go to its cell's slot for this face, signed as
    // the cell applies them (negation is exact, so the cell's sums are
    // unchanged bit for bit)
    const int32_t pos = fpos[f];
    const int64_t oL = quad64(L, 2 * nfmax, 2 * (pos & 15)), oR = quad64(R, 2 * nfmax, 2 * (pos >> 4));
    if (MIXED) {
        auto put = [&](int64_t o, float a, float b, float c, float d) {
            *reinterpret_cast<flt4 *>(fslot32 + o) = flt4{a, b, c, d};
        };
        put(oL, float(acc[0]), float(acc[1]), float(acc[2]), float(acc[3]));
        put(oL + 256, -float(acc[4]), -float(acc[5]), -float(acc[6]), -float(acc[7]));
        put(oR, -float(acc[0]), -float(acc[1]), -float(acc[2]), -float(acc[3]));
        put(oR + 256, float(acc[8]), float(acc[9]), float(acc[10]), float(acc[11]));
        return;
    }
    // plain stores (with non-temporal ones this kernel ran 19 % slower)
    auto put = [&](int64_t o, double a, double b, double c, double d) {
        dbl2 *p = reinterpret_cast<dbl2 *>(fslot + o);
        p[0] = dbl2{a, b}, p[1] = dbl2{c, d};
    };
    put(oL, acc[0], acc[1], acc[2], acc[3]);
    put(oL + 256, -acc[4], -acc[5], -acc[6], -acc[7]);
    put(oR, -acc[0], -acc[1], -acc[2], -acc[3]);
    put(oR + 256, acc[8], acc[9], acc[10], acc[11]);
}

// EvaluateRHS scatter as a per-cell gather in ascending face order
// (DNDS_FV_EulerEvaluator.cpp:501-508): the face kernel has stored each
// face's two terms at the cell's slot for that face, slots in ascending face
// order, signed so that the cell only adds (F/V then -FLfix/V for side 0,
// -F/V then FRfix/V for side 1).  Optionally fused with the SSP-RK3 stage
// update of ExplicitSSPRK3LocalDt::Step (DNDS_ODE.hpp:136-157):
//   stage 0: rhs = gathered value
//   stage 1: xLast = x; x = x + rhs dt
//   stage 2/3: x = ((x + rhs dt) c/(1-c) + xLast)(1-c), c = 1/4, 2/3
template <int NF, typename FT = double>
__global__ __launch_bounds__(kBlock) void k_rhs_cell(int32_t nc, int64_t ldc, const int32_t *__restrict__ gat,
                                                     const FT *__restrict__ fslot,
                                                     const double *__restrict__ vol, double *__restrict__ rhs,
                                                     int stage, double *__restrict__ x,
                                                     double *__restrict__ xlast, const double *__restrict__ dt,
                                                     const double *__restrict__ dtmin, double coefA, double coefB,
                                                     int32_t *errw) {
    const int32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= nc)
        return;
    const FT V = FT(vol[i]);
    // a cell has 3 or 4 faces: only the 4-slot layout has an absent last slot
    const int ns = NF == 4 && gat[3 * ldc + i] < 0 ? 3 : NF;
    FT r[4] = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < NF; s++) {
        if (s >= ns)
            break;
#pragma unroll
        for (int v = 0; v < 4; v++)
            r[v] += fslot[quad64(i, 2 * NF, 2 * s) + v] / V;
#pragma unroll
        for (int v = 0; v < 4; v++)
            r[v] += fslot[quad64(i, 2 * NF, 2 * s + 1) + v] / V;
    }
    bool finite = true;
#pragma unroll
    for (int v = 0; v < 4; v++)
        finite &= isfinite(r[v]);
    if (!finite)
        raise_error(errw, ERR_NAN);
    if (stage == 0) {
#pragma unroll
        for (int v = 0; v < 4; v++)
            rhs[4 * int64_t(i) + v] = double(r[v]);
        return;
    }
    const double d = dt ? dt[i] : dtmin[0];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const double xo = x[4 * int64_t(i) + v];
        double xv = xo + double(r[v]) * d;
        if (stage == 1) {
            xlast[4 * int64_t(i) + v] = xo;
        } else {
            xv *= coefA;
            xv += xlast[4 * int64_t(i) + v];
            xv *= coefB;
        }
        x[4 * int64_t(i) + v] = xv;
    }
}


// WBAP V3 step 0, face part (DNDS_FV_VR.hpp:2084-2126): for each inner face
// the (IJI, ISI) diagonals of the (rho, E) jump functional at the first
// LINE_3 point with the LINE_1 weight 2, for both adjacent cells.  As in the
// reference, a cell evaluates the face's side-0 basis with its own
// coefficients and the side-1 basis with its neighbour's.
//
// Two lanes per face, one per side: each evaluates its side's basis (the
// divisions, which bound this kernel), applies it to both cells'
// coefficients, and finishes its own cell's terms; the coefficients and the
// products that the other side needs change lanes with DPP moves.
__global__ __launch_bounds__(kBlock) void k_wbap_face(int32_t nf, int64_t ldf, int nfmax,
                                                      const int32_t *__restrict__ f2c,
                                                      const double *__restrict__ fxy, const double *__restrict__ cmom,
                                                      const double *__restrict__ cscale,
                                                      const double *__restrict__ fw,
                                                      const double *__restrict__ fn, const double *__restrict__ u,
                                                      const double *__restrict__ x, double tang_weight, int twd_norm,
                                                      const uint8_t *__restrict__ wpos, double *__restrict__ wslot,
                                                      int32_t *__restrict__ lim_count) {
    const int32_t t = xcd_block() * blockDim.x + threadIdx.x, f = t >> 1;
    const bool sd = t & 1;
    if (t == 0)
        *lim_count = 0; // k_wbap_ind, the next launch, counts
    if (f >= nf)
        return;
    const int32_t L = f2c[f], R = f2c[ldf + f];
    if (R < 0)
        return;
    const int32_t cell = sd ? R : L;
    // the cell's rho and E, coefficients and mean, and the other side's
    double xs[9][2], xt[9][2];
#pragma unroll
    for (int c = 0; c < 9; c++)
        xs[c][0] = x[rec(cell, c, 0)], xs[c][1] = x[rec(cell, c, 3)];
    const double us[2] = {u[4 * int64_t(cell)], u[4 * int64_t(cell) + 3]};
    // the DiBj block of this side at point 0, evaluated from the point's
    // scaled coordinates and the cell's scales and moments; zero entries are
    // skipped (adding them would not change any sum).  The rows are taken in
    // the functional's groups {0}, {1, 2}, {3, 4, 5}, {6..9}, whose terms then
    // join the indicator sums in their order.
    const dbl2 p0 = __builtin_nontemporal_load(reinterpret_cast<const dbl2 *>(fxy) + blk64(f, 6) + (sd ? 64 * 3 : 0));
    const dbl2 sc = reinterpret_cast<const dbl2 *>(cscale)[cell];
    double pX[4], pY[4], sX[4], sY[4];
    int_powers(p0.x, pX), int_powers(p0.y, pY), int_powers(sc.x, sX), int_powers(sc.y, sY);
    double W[10];
#pragma unroll
    for (int k = 0; k < 10; k++)
        W[k] = fw[blk64(f, 10) + 64 * k];
    const double gx = fn[blk64(f, 6)], gy = fn[blk64(f, 6) + 64];
    const FFParams P = ff_params(W, gx, gy, tang_weight, twd_norm);
    const double nl = sqrt(gx * gx + gy * gy);
#pragma unroll
    for (int c = 0; c < 9; c++)
        xt[c][0] = pair_swap(xs[c][0]), xt[c][1] = pair_swap(xs[c][1]);
    const double ut[2] = {pair_swap(us[0]), pair_swap(us[1])};
    double sums[2][2] = {{0.0, 0.0}, {0.0, 0.0}}; // [rho, E][IJI, ISI]
    auto pass = [&](auto group) {
        constexpr int G = decltype(group)::value;
        constexpr int r0 = G == 0 ? 0 : G == 1 ? 1 : G == 2 ? 3 : 6, nr = G == 0 ? 1 : G == 1 ? 2 : G == 2 ? 3 : 4;
        double bs[nr][2], bt[nr][2]; // this side's basis times its own and the other cell's coefficients
#pragma unroll
        for (int k = 0; k < nr * 2; k++)
            (&bs[0][0])[k] = 0.0, (&bt[0][0])[k] = 0.0;
#pragma unroll
        for (int c = 0; c < 9; c++) {
            const double m = G == 0 ? cmom[blk64(cell, 9) + 64 * c] : 0.0;
#pragma unroll
            for (int rr = 0; rr < nr; rr++) {
                const int r = r0 + rr;
                const int coef = dibj_coef(r, c + 1);
                if (coef == 0)
                    continue;
                const int ex = kBX[c + 1] - kBX[r], ey = kBY[c + 1] - kBY[r];
                double d = double(coef) * pX[ex] * pY[ey] * 1.0;
                if (r == 0)
                    d -= m;
                else
                    d = d / (sX[kBX[r]] * sY[kBY[r]] * 1.0);
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    bs[rr][q] += d * xs[c][q];
                    bt[rr][q] += d * xt[c][q];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            double val[nr], jmp[nr];
#pragma unroll
            for (int rr = 0; rr < nr; rr++) {
                // cell L: side 0 with its own, side 1 with R's own; cell R:
                // side 0 with R's, side 1 with L's coefficients
                const double other = pair_swap(sd ? bs[rr][q] : bt[rr][q]);
                double vl = sd ? other : bs[rr][q], vr = sd ? bt[rr][q] : other;
                if (r0 + rr == 0) {
                    vl += us[q];
                    vr += ut[q];
                }
                val[rr] = (vl + vr) * 0.5;
                jmp[rr] = (vl - vr) * 0.5;
            }
            ff_group<G>(P, jmp, sums[q][0]);
            ff_group<G>(P, val, sums[q][1]);
        }
    };
    pass(std::integral_constant<int, 0>{});
    pass(std::integral_constant<int, 1>{});
    pass(std::integral_constant<int, 2>{});
    pass(std::integral_constant<int, 3>{});
    double out[4];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        double a = sums[q][0], b = sums[q][1];
        a *= nl, b *= nl;
        out[2 * q] = a * 2.0;
        out[2 * q + 1] = b * 2.0;
    }
    // into the cell's own slot of this face, so that the indicator reads its
    // terms as a coalesced stream
    const int slot = sd ? (wpos[f] >> 4) : (wpos[f] & 15);
    dbl2 *to = reinterpret_cast<dbl2 *>(wslot + quad64(cell, nfmax, slot));
    to[0] = dbl2{out[0], out[1]}, to[1] = dbl2{out[2], out[3]};
}

// WBAP V3 smoothness indicator: sum over the cell's faces in cell2face order
// (DNDS_FV_VR.hpp:2125-2137).  Cells below WBAP_SmoothIndicatorScale (unless
// ifAll) keep their reconstruction; the others are appended to `list`
// (one atomic per wavefront; the order of the list does not affect any
// result, each cell is limited independently).
template <int NF>
__global__ __launch_bounds__(kBlock) void k_wbap_ind(int32_t nc, int64_t ldc, const int32_t *__restrict__ nbr,
                                                     const double *__restrict__ wslot, const double *__restrict__ x,
                                                     double *__restrict__ xo, double *__restrict__ ind, double scale,
                                                     int if_all, int32_t *__restrict__ count,
                                                     int32_t *__restrict__ list, uint8_t *__restrict__ limf) {
    const int32_t i = xcd_block() * blockDim.x + threadIdx.x;
    bool lim = false;
    if (i < nc) {
        double sum[4] = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < NF; s++) {
            const int32_t j = nbr[s * ldc + i];
            if (j < 0)
                continue;
#pragma unroll
            for (int k = 0; k < 4; k++)
                sum[k] += wslot[quad64(i, NF, s) + k];
        }
        const double si0 = sum[0] / (sum[1] + kVerySmallReal);
        const double si1 = sum[2] / (sum[3] + kVerySmallReal);
        const double flag = sqrt(fmax(fabs(si0), fabs(si1))) * (3 * 3);
        ind[i] = flag;
        lim = !(flag < scale && !if_all);
        if (limf)
            limf[i] = uint8_t(lim);
        else if (!lim) {
#pragma unroll
            for (int c = 0; c < 9; c++) {
                const dbl2 *from = reinterpret_cast<const dbl2 *>(x + rec(i, c, 0));
                dbl2 *to = reinterpret_cast<dbl2 *>(xo + rec(i, c, 0));
                to[0] = from[0], to[1] = from[1];
            }
        }
    }
    const uint64_t mask = __ballot(lim);
    if (mask == 0)
        return;
    const int lane = threadIdx.x & 63;
    const int first = __ffsll((unsigned long long)mask) - 1;
    int32_t base = 0;
    if (lane == first)
        base = atomicAdd(count, __popcll(mask));
    base = __shfl(base, first);
    if (lim)
        list[base + __popcll(mask & ((1ull << lane) - 1))] = i;
}

// ---- WBAP limiting: sixteen lanes per limited cell -----------------------
//
// The limited cells are few (a shock's neighbourhood), so what counts is how
// long one cell takes: with one lane per cell the face loop's chain of index
// loads, products, eigenvectors and divisions ran once per neighbour, at one
// wave per SIMD.  A row of 16 lanes now owns a cell, quad s of the row the
// neighbour in slot s, lane v of the quad variable v: the neighbours' terms
// are formed side by side and then combined in slot order by the row's first
// quad.  The secondary matrices are stored face by face ([face][side][82]):
// what a cell reads of them is contiguous.
//
// Measured against one lane per cell, a Mach-3 shock on 24 727 mixed cells:
// V2 (three launches) 140 -> 21 us, V3 354 -> 13; on 393 734 cells 198 -> 32
// and 490 -> 21.  With every cell limited (262 088 triangles) 528 -> 417 and
// 1562 -> 411, on 810 000 quads the whole call 1940 -> 1773 and 6707 -> 1656.
// There the divisions bound it, so that a quad shares them (quad_char_rows):
// with whole matrices formed in every lane V2 took 525 and 2088.

constexpr int kSecEntries = 82; // 81 and a pad, per face and side
constexpr unsigned kLimBlocks = 8192; // workgroups that walk the list (131 072 cells at once)

// a lane's row of the face's eigenvector matrices for neighbour j of cell i
// through face f, and the side of i
__device__ __forceinline__ bool face_char_rows(double gamma, const double *__restrict__ u, int32_t i, int32_t j,
                                               int32_t f, int side, int64_t ldf, const double *__restrict__ fnc, int v,
                                               double ml[4], double mr[4]) {
    const double *uLp = u + 4 * int64_t(side ? j : i), *uRp = u + 4 * int64_t(side ? i : j);
    double UL[4], UR[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        UL[k] = uLp[k], UR[k] = uRp[k];
    return quad_char_rows(gamma, UL, UR, fnc[f], fnc[ldf + f], v, ml, mr);
}

// sum over the quad's lanes b of row[b] a_b, in order
__device__ __forceinline__ double quad_dot(const double row[4], double a) {
    double p = 0;
#pragma unroll
    for (int b = 0; b < 4; b++)
        p += row[b] * quad_get(a, b);
    return p;
}

// WBAP V3 per-order characteristic limiting of the listed cells
// (DNDS_FV_VR.hpp:2152-2317).  Reads x, writes xo.  uF: the limited face
// values of rows 2..8 of the orders already done.
template <int NF>
__global__ __launch_bounds__(kBlock, 2) void k_wbap_lim(int64_t ldc, int64_t ldf, const int32_t *__restrict__ count,
                                                        const int32_t *__restrict__ list,
                                                        const int32_t *__restrict__ nbr,
                                                        const int32_t *__restrict__ sface,
                                                        const int32_t *__restrict__ f2c,
                                                        const double *__restrict__ fnc,
                                                        const double *__restrict__ msec, const double *__restrict__ u,
                                                        const double *__restrict__ x, double *__restrict__ xo,
                                                        double gamma, double nStd, double eps4, int32_t *errw) {
    const int s = (threadIdx.x >> 2) & 3, v = threadIdx.x & 3;
    const int32_t n = count[0];
    for (int32_t q = blockIdx.x * (kBlock / 16) + (threadIdx.x >> 4); q < n; q += gridDim.x * (kBlock / 16)) {
        const int32_t i = list[q];
        const int32_t j = s < NF ? nbr[s * ldc + i] : -1;
        const bool valid = j >= 0;
        double own[9], xj[9], uF[7], ml[4], mr[4];
        QuadPart<0, 40> ms, msO;
#pragma unroll
        for (int r = 0; r < 9; r++)
            own[r] = x[rec(i, r, v)];
        if (valid) {
            const int32_t f = sface[s * ldc + i];
            const int side = f2c[f] == i ? 0 : 1;
            const double *m = msec + 2 * kSecEntries * int64_t(f);
            ms.load(m + kSecEntries * side, v);
            msO.load(m + kSecEntries * (1 - side), v);
#pragma unroll
            for (int c = 0; c < 9; c++)
                xj[c] = x[rec(j, c, v)];
            if (!face_char_rows(gamma, u, i, j, f, side, ldf, fnc, v, ml, mr))
                raise_error(errw, ERR_NONPOSITIVE);
        }
#pragma unroll
        for (int order = 3; order >= 1; order--) {
            const int ls = order == 3 ? 5 : (order == 2 ? 2 : 0);
            const int le = order == 3 ? 8 : (order == 2 ? 4 : 1);
            constexpr int kMaxR = 4;
            const int nr = le - ls + 1;
            double up[kMaxR], down[kMaxR]; // this neighbour's terms
#pragma unroll
            for (int r = 0; r < kMaxR; r++)
                up[r] = down[r] = 0.0;
            if (valid) {
                double oIn[kMaxR];
#pragma unroll
                for (int r = 0; r < kMaxR; r++)
                    oIn[r] = 0.0;
                // uOtherOther rows: the neighbour's coefficients up to le, above
                // le the limited face values of the higher orders mapped to its
                // basis
#pragma unroll
                for (int c = 0; c < 9; c++) {
                    double uoo = xj[c];
                    if (c > le) {
                        uoo = 0;
#pragma unroll
                        for (int cc = 0; cc < 9; cc++)
                            if (cc > le)
                                uoo += msO.get(9 * c + cc) * uF[cc - 2];
                    }
#pragma unroll
                    for (int r = 0; r < kMaxR; r++)
                        if (r < nr)
                            oIn[r] += ms.get(9 * (ls + r) + c) * uoo;
                }
#pragma unroll
                for (int r = 0; r < kMaxR; r++) {
                    if (r >= nr)
                        continue;
                    const double u0 = own[ls + r];
                    const double oC = quad_dot(ml, oIn[r]), tC = quad_dot(ml, u0);
                    // FWBAP_L2_Biway(uThisIn, uOtherIn, 1)
                    const double frac = tC / (fabs(oC) + 1e-12) * sgn(oC);
                    const double th1 = frac * frac * frac;
                    const double th2 = (frac * frac) * (frac * frac);
                    const double xv = quad_dot(mr, tC * (1.0 + th1) / (1.0 + th2));
                    if (ls + r >= 2)
                        uF[ls + r - 2] = xv;
                    // FWBAP_L2_Multiway's terms
                    const double ti = u0 / (fabs(xv) + eps4) * sgn(xv);
                    down[r] = (ti * ti) * (ti * ti);
                    up[r] = ti * ti * ti;
                }
            }
            // the neighbours in cell2face order, in the row's first quad
#pragma unroll
            for (int r = 0; r < kMaxR; r++) {
                if (r >= nr)
                    continue;
                double sd = 0.0, su = 0.0;
#pragma unroll
                for (int t = 0; t < NF; t++) {
                    const double d = row_ahead(down[r], t), p = row_ahead(up[r], t);
                    if (row_ahead(int(valid), t)) {
                        sd += d;
                        su += p;
                    }
                }
                if (s == 0)
                    xo[rec(i, ls + r, v)] = own[ls + r] * (su + nStd) / (sd + nStd);
            }
        }
    }
}

// WBAP V2 limiting of the listed cells for one order (DNDS_FV_VR.hpp:1843-2040,
// rows ls..le of the order).  xo is the reference's uRecNewBuf: before this
// launch it holds x for the unlimited cells and, for the limited ones, the rows
// of the higher orders as limited by the earlier launches; rows ls..le and
// below are still x everywhere.  Each neighbour's full 9-row buffer is mapped
// to this cell's basis (rows <= le read from x, rows > le from xo), so the
// launch reads xo only above le and writes it only at ls..le: no cell reads
// what another writes.  FWBAP_L2_Biway with n = nStd per neighbour, then
// FWBAP_L2_Multiway centred on the first neighbour's result with n1 = 1.
template <int NF, int ORDER>
__global__ __launch_bounds__(kBlock, 3) void k_wbap_lim_v2(int64_t ldc, int64_t ldf, const int32_t *__restrict__ count,
                                                           const int32_t *__restrict__ list,
                                                           const int32_t *__restrict__ nbr,
                                                           const int32_t *__restrict__ sface,
                                                           const int32_t *__restrict__ f2c,
                                                           const double *__restrict__ fnc,
                                                           const double *__restrict__ msec,
                                                           const double *__restrict__ u, const double *__restrict__ x,
                                                           double *__restrict__ xo, double gamma, double nStd,
                                                           double eps4, int32_t *errw,
                                                           const uint8_t *__restrict__ limf) {
    constexpr int ls = ORDER == 3 ? 5 : (ORDER == 2 ? 2 : 0);
    constexpr int le = ORDER == 3 ? 8 : (ORDER == 2 ? 4 : 1);
    constexpr int nr = le - ls + 1;
    const int s = (threadIdx.x >> 2) & 3, v = threadIdx.x & 3;
    const int32_t n = count[0];
    for (int32_t q = blockIdx.x * (kBlock / 16) + (threadIdx.x >> 4); q < n; q += gridDim.x * (kBlock / 16)) {
        const int32_t i = list[q];
        const int32_t j = s < NF ? nbr[s * ldc + i] : -1;
        const bool valid = j >= 0;
        double uC[nr], xv[nr];
#pragma unroll
        for (int r = 0; r < nr; r++) {
            uC[r] = x[rec(i, ls + r, v)];
            xv[r] = 0.0;
        }
        if (valid) {
            const int32_t f = sface[s * ldc + i];
            const int side = f2c[f] == i ? 0 : 1;
            QuadPart<9 * ls / 2, (9 * le + 8) / 2> ms;
            ms.load(msec + kSecEntries * (2 * int64_t(f) + side), v);
            // the neighbour's rows above le: limited (xo) or, with limf, as given (x)
            const double *above = (limf && !limf[j]) ? x : xo;
            double uj[9];
#pragma unroll
            for (int c = 0; c < 9; c++)
                uj[c] = (c <= le ? x : above)[rec(j, c, v)];
            double ml[4], mr[4];
            if (!face_char_rows(gamma, u, i, j, f, side, ldf, fnc, v, ml, mr))
                raise_error(errw, ERR_NONPOSITIVE);
#pragma unroll
            for (int r = 0; r < nr; r++) {
                double oIn = 0.0;
#pragma unroll
                for (int c = 0; c < 9; c++)
                    oIn += ms.get(9 * (ls + r) + c) * uj[c];
                const double oC = quad_dot(ml, oIn), tC = quad_dot(ml, uC[r]);
                // FWBAP_L2_Biway(uThisIn, uOtherIn, nStd)
                const double frac = tC / (fabs(oC) + 1e-12) * sgn(oC);
                const double th1 = frac * frac * frac;
                const double th2 = (frac * frac) * (frac * frac);
                xv[r] = quad_dot(mr, tC * (nStd + th1) / (nStd + th2));
            }
        }
        // the neighbours in cell2face order, in the row's first quad
#pragma unroll
        for (int r = 0; r < nr; r++) {
            double first = 0.0, up = 0.0, down = 0.0;
            bool any = false;
#pragma unroll
            for (int t = 0; t < NF; t++) {
                const double a = row_ahead(xv[r], t);
                if (!row_ahead(int(valid), t))
                    continue;
                if (!any) {
                    first = a;
                } else {
                    const double ti = first / (fabs(a) + eps4) * sgn(a);
                    down += (ti * ti) * (ti * ti);
                    up += ti * ti * ti;
                }
                any = true;
            }
            if (s == 0)
                xo[rec(i, ls + r, v)] = any ? first * (up + 1.0) / (down + 1.0) : uC[r];
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_set(int64_t n, double *__restrict__ p, double v) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

// ========================================================================
// host side
// ========================================================================

namespace dndsmi_host {

int check_errw(dndsmi_ctx *c) {
    DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    volatile int32_t *e = c->host->err;
    const bool nonpositive = e[ERR_NONPOSITIVE], nan = e[ERR_NAN], bc = e[ERR_BC];
    if (!nonpositive && !nan && !bc)
        return DNDSMI_OK;
    for (int k = 0; k < ERR_KINDS; k++)
        e[k] = 0;
    if (nonpositive) {
        c->err = "non-positive density or sound speed in a flux or boundary state";
        return DNDSMI_ERR_NONPOSITIVE_STATE;
    }
    if (nan) {
        c->err = "non-finite value in the right-hand side or time step";
        return DNDSMI_ERR_NAN;
    }
    c->err = "boundary face of an unsupported kind";
    return DNDSMI_ERR_UNSUPPORTED;
}

bool same_ctx(const dndsmi_ctx *c, const dndsmi_array *a, int32_t kind) { return a && a->ctx == c && a->kind == kind; }

} // namespace dndsmi_host

extern "C" int dndsmi_ctx_create(const dndsmi_mesh_view *mesh, const dndsmi_vr_view *vr,
                                 const dndsmi_vr_setting *vs, const dndsmi_euler_setting *es, void *stream,
                                 dndsmi_ctx **out) {
    if (!mesh || !vr || !vs || !es || !out)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    {
        std::string why;
        if (check_mesh_view(mesh, why) != DNDSMI_OK)
            return DNDSMI_ERR_INVALID_ARGUMENT;
    }
    if (vr->n_cell != mesh->n_cell || vr->n_face != mesh->n_face || vr->n_c2f != mesh->cell_ptr[mesh->n_cell] ||
        mesh->n_cell > (int64_t(1) << 30) || mesh->n_face > (int64_t(1) << 30))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (!vr->face_gauss_xy || !vr->cell_scale || !vr->base_moment || !vr->face_d0)
        return DNDSMI_ERR_INVALID_ARGUMENT; // the device evaluates the face bases from these
    if (!vr->volume || !vr->face_area || !vr->face_center || !vr->face_norm_center || !vr->face_norm ||
        !vr->face_weight || !vr->ainv || !vr->ainv_b || !vr->ainv_bvec)
        return DNDSMI_ERR_INVALID_ARGUMENT; // matrix_secondary alone may be absent (no WBAP then)
    if (es->riemann_solver != DNDSMI_RS_ROE && es->riemann_solver != DNDSMI_RS_HLLC &&
        es->riemann_solver != DNDSMI_RS_HLLEP &&
        !(es->riemann_solver >= DNDSMI_RS_ROE_M1 && es->riemann_solver <= DNDSMI_RS_ROE_M5))
        return DNDSMI_ERR_UNSUPPORTED;
    // local coordinates: the kernels evaluate the bases' values only
    if (vr->cell_frame && (es->mu_gas > 0 || vr->matrix_secondary))
        return DNDSMI_ERR_UNSUPPORTED;
    if (!(es->mu_gas >= 0) ||
        (es->mu_gas > 0 && !(es->pr_gas > 0 && es->r_gas > 0 && es->t_ref > 0 && es->c_sutherland >= 0)))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    dndsmi_ctx *c = new (std::nothrow) dndsmi_ctx();
    if (!c)
        return DNDSMI_ERR_OUT_OF_MEMORY;
    auto fail = [&](int rc) {
        dndsmi_ctx_destroy(c);
        return rc;
    };
    if (hipGetDevice(&c->device) != hipSuccess)
        return fail(DNDSMI_ERR_HIP);
    if (noalloc_scratch_init(c) != DNDSMI_OK)
        return fail(DNDSMI_ERR_HIP);
    if (stream) {
        c->stream = static_cast<hipStream_t>(stream);
    } else {
        if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
            return fail(DNDSMI_ERR_HIP);
        c->own_stream = true;
    }
    const int64_t nc = mesh->n_cell, nf = mesh->n_face;
    c->nc = nc, c->nf = nf, c->ldc = pad64(nc), c->ldf = pad64(nf);
    c->relax = vs->jacobi_relax;
    c->sor = vs->sor_instead != 0;
    c->sor_inverse = c->sor && vs->sor_inverse_scanning != 0;
    c->gas.gamma = es->gamma;
    for (int k = 0; k < 4; k++)
        c->gas.far[k] = es->far_field[k];
    c->gas.rs = es->riemann_solver;
    c->gas.mu = es->mu_gas;
    c->gas.pr = es->pr_gas;
    c->gas.cp = es->r_gas * es->gamma / (es->gamma - 1);
    c->gas.tref = es->t_ref;
    c->gas.csuth = es->c_sutherland;
    int nfmax = 0;
    for (int64_t i = 0; i < nc; i++)
        nfmax = std::max<int>(nfmax, int(mesh->cell_ptr[i + 1] - mesh->cell_ptr[i]));
    if (nfmax != 3 && nfmax != 4)
        return fail(DNDSMI_ERR_INVALID_ARGUMENT);
    c->nfmax = nfmax;
    const int64_t ldc = c->ldc, ldf = c->ldf;
    try {
        // ---- device numbering.  Every device array is indexed through c2d /
        // f2d (host arrays keep the mesh numbering).  The mesh's own order is
        // kept: on the structured-as-unstructured meshes it is row-major, and
        // measured faster for the sweeps than Morton or strip orders (whose
        // neighbour loads coalesce worse); a mesh read in a scattered order
        // would be renumbered here.  On a mesh of triangles and quads, each
        // window of 64 consecutive cells (one wavefront) puts its triangles
        // before its quads, keeping their order: the fourth slot's A^-1 B
        // vectors of a block are then contiguous over its quads, and the
        // 128-byte lines of that stream hold no unused triangle slots.
        //
        // With SOR_Instead the numbering is colour-major instead: each colour
        // is a contiguous range (its cells in mesh order), so that a colour's
        // pass streams whole lines of the A^-1 B stream and the coefficients; in
        // each colour the cells with terms on their own partial sum (far
        // field, Wall_Euler, Wall_NoSlip) come last, so that their longer
        // waves are few.  The windows of 64 then start at each range's start.
        //
        // Colouring (multicolour LU-SGS and SOR): each cell takes the
        // smallest colour that no lower-numbered neighbour holds.
        std::vector<int32_t> col(size_t(nc), -1);
        int32_t ncol = 0;
        for (int64_t i = 0; i < nc; i++) { // mesh numbering
            uint32_t used = 0;
            for (int64_t q = mesh->cell_ptr[i]; q < mesh->cell_ptr[i + 1]; q++) {
                const int64_t f = mesh->cell2face[q];
                const int64_t L = mesh->face2cell[2 * f], R = mesh->face2cell[2 * f + 1];
                const int64_t j = L == i ? R : L;
                if (j != DNDSMI_NO_CELL && j < i && col[j] < 32)
                    used |= 1u << col[j];
            }
            int32_t k = 0;
            while (used & (1u << k))
                k++;
            col[i] = k;
            ncol = std::max(ncol, k + 1);
        }
        std::vector<int32_t> &c2d = c->c2d, &f2d = c->f2d;
        {
            // the numbering's segments (mesh cells in order) and their ends
            std::vector<int64_t> seq(static_cast<size_t>(nc)), seg_end;
            if (c->sor) {
                std::vector<uint8_t> self(size_t(nc), 0);
                for (int64_t i = 0; i < nc; i++)
                    for (int64_t q = mesh->cell_ptr[i]; q < mesh->cell_ptr[i + 1]; q++) {
                        const int64_t f = mesh->cell2face[q];
                        const int64_t L = mesh->face2cell[2 * f], R = mesh->face2cell[2 * f + 1];
                        if ((L == i ? R : L) == DNDSMI_NO_CELL && mesh->face_bc[f] != DNDSMI_BC_WALL)
                            self[size_t(i)] = 1;
                    }
                std::vector<int64_t> cnt(2 * size_t(ncol) + 1, 0);
                for (int64_t i = 0; i < nc; i++)
                    cnt[2 * col[i] + self[size_t(i)] + 1]++;
                for (size_t g = 0; g + 1 < cnt.size(); g++)
                    cnt[g + 1] += cnt[g];
                seg_end.assign(cnt.begin() + 1, cnt.end());
                std::vector<int64_t> fill(cnt.begin(), cnt.end() - 1);
                for (int64_t i = 0; i < nc; i++)
                    seq[fill[2 * col[i] + self[size_t(i)]]++] = i;
                c->sor_start.assign(size_t(ncol) + 1, nc);
                for (int32_t k = 0; k < ncol; k++)
                    c->sor_start[k] = cnt[2 * k];
            } else {
                for (int64_t i = 0; i < nc; i++)
                    seq[i] = i;
                seg_end.push_back(nc);
            }
            c2d.resize(static_cast<size_t>(nc));
            int64_t a = 0;
            for (const int64_t b : seg_end) {
                for (int64_t w0 = a; w0 < b; w0 += 64) {
                    const int64_t w1 = std::min<int64_t>(b, w0 + 64);
                    int64_t d = w0;
                    for (int pass = 0; pass < 2; pass++)
                        for (int64_t p = w0; p < w1; p++) {
                            const int64_t i = seq[p];
                            const bool quad = mesh->cell_ptr[i + 1] - mesh->cell_ptr[i] == 4;
                            if (quad == (pass == 1))
                                c2d[i] = int32_t(d++);
                        }
                }
                a = b;
            }
            c->d2c.resize(static_cast<size_t>(nc));
            for (int64_t i = 0; i < nc; i++)
                c->d2c[c2d[i]] = int32_t(i);
            // faces in the order of their first cell in the mesh (the
            // partition of a window above moves cells by less than a
            // wavefront, and the face kernels gather best in mesh order)
            std::vector<std::pair<int64_t, int64_t>> fk(static_cast<size_t>(nf));
            for (int64_t f = 0; f < nf; f++)
                fk[f] = {mesh->face2cell[2 * f], f};
            std::sort(fk.begin(), fk.end());
            f2d.assign(static_cast<size_t>(nf), 0);
            for (int64_t d = 0; d < nf; d++)
                f2d[fk[d].second] = int32_t(d);
        }
        // ---- cell streams
        std::vector<int32_t> nbr(size_t(nfmax) * ldc, -2), sbc(size_t(nfmax) * ldc, 0), sface(size_t(nfmax) * ldc, -1);
        std::vector<int32_t> gat(size_t(nfmax) * ldc, -1);
        std::vector<uint8_t> wpos(ldf, 0);
        std::vector<double> M(size_t(nfmax) * kAbVecs * 2 * ldc, 0.0), vol(ldc, 1.0);
        std::vector<double> cmom(9 * size_t(ldc), 0.0), cscale(2 * size_t(ldc), 1.0);
        std::vector<int64_t> wall_cell, wall_face, wall_c2f;
        for (int64_t i = 0; i < nc; i++) {
            const int64_t b0 = mesh->cell_ptr[i];
            const int n = int(mesh->cell_ptr[i + 1] - b0);
            const int64_t ci = c2d[i]; // device column of mesh cell i
            vol[ci] = vr->volume[i];
            for (int k = 0; k < 9; k++)
                cmom[blk64(ci, 9) + 64 * k] = vr->base_moment[10 * i + 1 + k];
            cscale[2 * ci] = vr->cell_scale[2 * i], cscale[2 * ci + 1] = vr->cell_scale[2 * i + 1];
            std::vector<std::pair<int64_t, int>> order;
            for (int s = 0; s < n; s++) {
                const int64_t f = mesh->cell2face[b0 + s];
                const int64_t L = mesh->face2cell[2 * f], R = mesh->face2cell[2 * f + 1];
                const int side = L == i ? 0 : 1;
                const int64_t j = side == 0 ? R : L;
                nbr[s * ldc + ci] = j == DNDSMI_NO_CELL ? -1 : c2d[j];
                sbc[s * ldc + ci] = mesh->face_bc[f];
                sface[s * ldc + ci] = f2d[f];
                if (j != DNDSMI_NO_CELL)
                    wpos[f2d[f]] |= uint8_t(s << (4 * side));
                for (int d = 0; d < 90; d++)
                    M[size_t(ab_vec(s, d / 2, ci, ldc, kAbVecs)) * 2 + d % 2] =
                        d % 10 < 9 ? vr->ainv_b[81 * (b0 + s) + 9 * (d / 10) + d % 10]
                                   : vr->ainv_bvec[9 * (b0 + s) + d / 10];
                order.push_back({f, side});
                if (j == DNDSMI_NO_CELL &&
                    (mesh->face_bc[f] == DNDSMI_BC_WALL_EULER || mesh->face_bc[f] == DNDSMI_BC_WALL_NOSLIP)) {
                    nbr[s * ldc + ci] = wall_slot(int32_t(wall_cell.size()), mesh->face_bc[f]);
                    wall_cell.push_back(i), wall_face.push_back(f), wall_c2f.push_back(b0 + s);
                }
            }
            // the gather visits the faces in the mesh's face order (the
            // reference's scatter order), whatever their device numbers
            std::sort(order.begin(), order.end());
            for (int s = 0; s < n; s++)
                gat[s * ldc + ci] = int32_t((int64_t(f2d[order[s].first]) << 1) | order[s].second);
        }
        DNDSMI_TRY(c->alloc(c->nbr, nfmax * ldc));
        DNDSMI_TRY(c->upload(c->nbr, nbr));
        DNDSMI_TRY(c->alloc(c->sbc, nfmax * ldc));
        DNDSMI_TRY(c->upload(c->sbc, sbc));
        DNDSMI_TRY(c->alloc(c->sface, nfmax * ldc));
        DNDSMI_TRY(c->upload(c->sface, sface));
        DNDSMI_TRY(c->alloc(c->gat, nfmax * ldc));
        DNDSMI_TRY(c->upload(c->gat, gat));
        DNDSMI_TRY(c->alloc(c->wpos, ldf));
        DNDSMI_TRY(c->upload(c->wpos, wpos));
        {
            std::vector<uint8_t> fpos(ldf, 0);
            for (int s = 0; s < nfmax; s++)
                for (int64_t ci = 0; ci < nc; ci++) {
                    const int32_t g = gat[s * ldc + ci];
                    if (g >= 0)
                        fpos[g >> 1] |= uint8_t(s << (4 * (g & 1)));
                }
            DNDSMI_TRY(c->alloc(c->fpos, ldf));
            DNDSMI_TRY(c->upload(c->fpos, fpos));
        }
        DNDSMI_TRY(c->alloc(c->M, int64_t(nfmax) * kAbVecs * 2 * ldc));
        DNDSMI_TRY(c->upload(c->M, M));
        M.clear(), M.shrink_to_fit();
        DNDSMI_TRY(c->alloc(c->vol, ldc));
        DNDSMI_TRY(c->upload(c->vol, vol));
        DNDSMI_TRY(c->alloc(c->cmom, 9 * ldc));
        DNDSMI_TRY(c->upload(c->cmom, cmom));
        DNDSMI_TRY(c->alloc(c->cscale, 2 * ldc));
        DNDSMI_TRY(c->upload(c->cscale, cscale));
        // wall faces (Wall_Euler / Wall_NoSlip): compact arrays
        const int64_t nw = int64_t(wall_cell.size());
        c->n_wall = std::max<int64_t>(nw, 1);
        {
            std::vector<double> wd(kWallEntries * size_t(c->n_wall), 0.0);
            for (int64_t w = 0; w < nw; w++) {
                const int64_t i = wall_cell[w], f = wall_face[w];
                double *p = &wd[kWallEntries * size_t(w)];
                std::copy_n(vr->ainv + 81 * i, 81, p);
                for (int g = 0; g < 3; g++)
                    std::copy_n(vr->face_d0 + 54 * f + 18 * g, 9, p + kWallD0 + 9 * g);
                std::copy_n(vr->face_norm + 6 * f, 6, p + kWallNrm);
                p[kWallW0] = vr->face_weight[10 * f];
            }
            DNDSMI_TRY(c->alloc(c->walls, kWallEntries * c->n_wall));
            DNDSMI_TRY(c->upload(c->walls, wd));
            DNDSMI_TRY(c->alloc(c->wall_corr, kRec * c->n_wall));
            c->n_wall_faces = nw;
        }
        // ---- face streams
        std::vector<int32_t> f2c(2 * size_t(ldf), -1), fbc(ldf, DNDSMI_BC_INNER);
        bool straight = true;
        std::vector<double> fxy(12 * size_t(ldf), 0.0), fn(6 * size_t(ldf), 0.0), fnc(2 * size_t(ldf), 0.0),
            farea(ldf, 0.0), fctr(2 * size_t(ldf), 0.0);
        for (int64_t fo = 0; fo < nf; fo++) {
            const int64_t f = f2d[fo]; // device column of mesh face fo
            f2c[f] = c2d[mesh->face2cell[2 * fo]];
            const int64_t R = mesh->face2cell[2 * fo + 1];
            f2c[ldf + f] = R == DNDSMI_NO_CELL ? -1 : c2d[R];
            fbc[f] = mesh->face_bc[fo];
            for (int g = 0; g < 3; g++) // rows [side][g] of (X, Y) pairs
                for (int sd = 0; sd < 2; sd++)
                    for (int k = 0; k < 2; k++)
                        fxy[(blk64(f, 6) + 64 * (sd * 3 + g)) * 2 + k] =
                            vr->face_gauss_xy[12 * fo + 4 * g + 2 * sd + k];
            for (int k = 0; k < 6; k++)
                fn[blk64(f, 6) + 64 * k] = vr->face_norm[6 * fo + k];
            for (int k = 2; k < 6; k++)
                straight &= std::memcmp(&vr->face_norm[6 * fo + k], &vr->face_norm[6 * fo + k % 2], 8) == 0;
            fnc[f] = vr->face_norm_center[2 * fo], fnc[ldf + f] = vr->face_norm_center[2 * fo + 1];
            farea[f] = vr->face_area[fo];
            fctr[f] = vr->face_center[2 * fo], fctr[ldf + f] = vr->face_center[2 * fo + 1];
        }
        DNDSMI_TRY(c->alloc(c->f2c, 2 * ldf));
        DNDSMI_TRY(c->upload(c->f2c, f2c));
        DNDSMI_TRY(c->alloc(c->fbc, ldf));
        DNDSMI_TRY(c->upload(c->fbc, fbc));
        DNDSMI_TRY(c->alloc(c->fxy, 12 * ldf));
        DNDSMI_TRY(c->upload(c->fxy, fxy));
        DNDSMI_TRY(c->alloc(c->fn, 6 * ldf));
        DNDSMI_TRY(c->upload(c->fn, fn));
        c->straight_faces = straight;
        DNDSMI_TRY(c->alloc(c->fnc, 2 * ldf));
        DNDSMI_TRY(c->upload(c->fnc, fnc));
        DNDSMI_TRY(c->alloc(c->farea, ldf));
        DNDSMI_TRY(c->upload(c->farea, farea));
        DNDSMI_TRY(c->alloc(c->fctr, 2 * ldf));
        DNDSMI_TRY(c->upload(c->fctr, fctr));
        std::vector<int32_t> bfl;
        for (int64_t f = 0; f < nf; f++)
            if (mesh->face2cell[2 * f + 1] == DNDSMI_NO_CELL)
                bfl.push_back(f2d[f]);
        std::sort(bfl.begin(), bfl.end());
        c->n_bface = int64_t(bfl.size());
        if (bfl.empty())
            bfl.push_back(0);
        DNDSMI_TRY(c->alloc(c->bfaces, int64_t(bfl.size())));
        DNDSMI_TRY(c->upload(c->bfaces, bfl));
        // ---- WBAP data
        c->tang_weight = vs->tang_weight;
        c->twd_norm = vs->tang_weight_direction == 0;
        c->wbap_scale = vs->wbap_smooth_indicator_scale;
        c->wbap_nstd = vs->wbap_n_std;
        if (vr->matrix_secondary) {
            c->has_limiter = true;
            std::vector<double> buf;
            buf.assign(2 * kSecEntries * size_t(ldf), 0.0);
            for (int64_t f = 0; f < nf; f++)
                for (int k = 0; k < 162; k++)
                    buf[kSecEntries * (2 * size_t(f2d[f]) + k / 81) + k % 81] = vr->matrix_secondary[162 * f + k];
            DNDSMI_TRY(c->alloc(c->msec, 2 * kSecEntries * ldf));
            DNDSMI_TRY(c->upload(c->msec, buf));
            buf.assign(10 * size_t(ldf), 0.0);
            for (int64_t f = 0; f < nf; f++)
                for (int k = 0; k < 10; k++)
                    buf[blk64(f2d[f], 10) + 64 * k] = vr->face_weight[10 * f + k];
            DNDSMI_TRY(c->alloc(c->fw, 10 * ldf));
            DNDSMI_TRY(c->upload(c->fw, buf));
            DNDSMI_TRY(c->alloc(c->wslot, int64_t(nfmax) * 4 * ldc));
            DNDSMI_TRY(c->alloc(c->ind, ldc));
            DNDSMI_TRY(c->alloc(c->xlim, 36 * ldc));
            DNDSMI_TRY(c->alloc(c->limf, ldc));
            DNDSMI_TRY(c->alloc(c->lim_list, ldc));
            DNDSMI_TRY(c->alloc(c->lim_count, 1));
        }
        // ---- multicolour scan lists (col and ncol from before the numbering)
        {
            c->n_colour = ncol;
            c->col_start.assign(size_t(ncol) + 1, 0);
            for (int64_t i = 0; i < nc; i++)
                c->col_start[col[i] + 1]++;
            for (int32_t k = 0; k < ncol; k++)
                c->col_start[k + 1] += c->col_start[k];
            std::vector<int32_t> cells(static_cast<size_t>(nc)), fill(c->col_start.begin(), c->col_start.end() - 1);
            for (int64_t i = 0; i < nc; i++) // ascending mesh index within a colour
                cells[fill[col[i]]++] = c2d[i];
            std::vector<int32_t> colp(size_t(ldc), 0);
            for (int64_t i = 0; i < nc; i++)
                colp[c2d[i]] = col[i];
            c->colour_host = col;
            DNDSMI_TRY(c->alloc(c->colour, ldc));
            DNDSMI_TRY(c->upload(c->colour, colp));
            DNDSMI_TRY(c->alloc(c->col_cells, nc));
            DNDSMI_TRY(c->upload(c->col_cells, cells));
            DNDSMI_TRY(c->alloc(c->jinv, ldc));
        }
        // ---- scratch
        DNDSMI_TRY(c->alloc(c->lambda_face, ldf));
        DNDSMI_TRY(c->alloc(c->dlambda_face, ldf));
        DNDSMI_TRY(c->alloc(c->fslot, int64_t(nfmax) * 8 * ldc));
        DNDSMI_TRY(c->alloc(c->dt_part, int64_t(grid_for(nc)) + 1));
        DNDSMI_TRY(c->alloc(c->dt_min, 1));
        DNDSMI_TRY(c->hip(hipHostMalloc(&c->host, sizeof(HostWords), hipHostMallocCoherent), "hipHostMalloc"));
        std::memset(static_cast<void *>(c->host), 0, sizeof(HostWords));
        c->errw = c->host->err;
        DNDSMI_TRY(c->alloc(c->xlast, 4 * ldc));
        DNDSMI_TRY(c->alloc(c->dt_tmp, ldc));
        hipLaunchKernelGGL(k_set, dim3(grid_for(ldf)), dim3(kBlock), 0, c->stream, ldf, c->dlambda_face, 0.0);
        DNDSMI_TRY(c->launch_check("init kernels"));
        DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    } catch (const std::bad_alloc &) {
        return fail(DNDSMI_ERR_OUT_OF_MEMORY);
    }
    *out = c;
    return DNDSMI_OK;
}

// defined with the warm start (warmstart.hip) and the BDF integrator
// (lusgs.hip): forget the context
void dndsmi_warmstart_detach(dndsmi_warmstart *w);
void dndsmi_bdf_detach(dndsmi_bdf *b);

extern "C" void dndsmi_ctx_destroy(dndsmi_ctx *c) {
    if (!c)
        return;
    if (c->stream)
        (void)hipStreamSynchronize(c->stream);
    // arrays and warm starts may outlive their context (any destruction
    // order is allowed): free the arrays' storage and detach them
    for (dndsmi_array *a : c->arrays) {
        (void)hipFree(a->d);
        a->d = nullptr;
        a->ctx = nullptr;
    }
    c->arrays.clear();
    for (dndsmi_warmstart *w : c->warmstarts)
        dndsmi_warmstart_detach(w);
    c->warmstarts.clear();
    for (dndsmi_bdf *b : c->bdfs)
        dndsmi_bdf_detach(b);
    c->bdfs.clear();
    for (void *p : c->allocs)
        (void)hipFree(p);
    if (c->host)
        (void)hipHostFree(c->host);
    if (c->host_sums)
        (void)hipHostFree(c->host_sums);
    for (hipEvent_t e : c->ev_pool)
        (void)hipEventDestroy(e);
    if (c->own_stream && c->stream)
        (void)hipStreamDestroy(c->stream);
    delete c;
}

extern "C" int dndsmi_last_error(const dndsmi_ctx *c, char *buf, size_t n) {
    if (!c || !buf || n == 0)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    std::snprintf(buf, n, "%s", c->err.c_str());
    return DNDSMI_OK;
}

extern "C" int dndsmi_sync(dndsmi_ctx *c) {
    if (!c)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    return check_errw(c);
}

extern "C" int64_t dndsmi_ctx_device_bytes(const dndsmi_ctx *c) { return c ? c->bytes : -1; }

extern "C" int dndsmi_array_create(dndsmi_ctx *c, int32_t kind, dndsmi_array **out) {
    if (!c || !out || kind < DNDSMI_ARRAY_DOF || kind > DNDSMI_ARRAY_SCALAR)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    dndsmi_array *a = new (std::nothrow) dndsmi_array();
    if (!a)
        return DNDSMI_ERR_OUT_OF_MEMORY;
    a->ctx = c;
    a->kind = kind;
    a->elems = kind == DNDSMI_ARRAY_DOF ? 4 * c->ldc : (kind == DNDSMI_ARRAY_REC ? 36 * c->ldc : c->ldc);
    void *p = nullptr;
    if (hipMalloc(&p, sizeof(double) * a->elems) != hipSuccess) {
        (void)hipGetLastError();
        delete a;
        c->err = "hipMalloc of an array failed";
        return DNDSMI_ERR_OUT_OF_MEMORY;
    }
    a->d = static_cast<double *>(p);
    hipLaunchKernelGGL(k_set, dim3(grid_for(a->elems)), dim3(kBlock), 0, c->stream, a->elems, a->d, 0.0);
    int rc = c->launch_check("k_set");
    if (rc) {
        (void)hipFree(a->d);
        delete a;
        return rc;
    }
    c->arrays.insert(a);
    *out = a;
    return DNDSMI_OK;
}

extern "C" void dndsmi_array_destroy(dndsmi_array *a) {
    if (!a)
        return;
    if (a->ctx) { // else its context was destroyed first and freed the storage
        (void)hipStreamSynchronize(a->ctx->stream);
        (void)hipFree(a->d);
        a->ctx->arrays.erase(a);
    }
    delete a;
}

// REC arrays between the host's rows of 36 and the device's blocks of 64 cells.
// Both are bound by the host's memory.  Into the blocks they are written as
// they lie, from the block's rows (which stay in the first-level cache); out of
// them the rows are written in turn, and each cell of 288 bytes asks for as
// much of the block after its own, whose elements of 32 bytes no prefetcher
// follows.  Whole calls, ms, element by element through rec() -> now: 810 k
// cells 76 -> 51 up, 100 -> 73 down, 45 k 1.3 -> 0.75, 2.8 -> 1.1 (with planes
// of one element, the layout before: 64, 74; 15, 2.2).
static void rec_to_device(const dndsmi_ctx *c, const double *host, double *buf) {
    for (int64_t b = 0; b < c->nc; b += 64) {
        double *blk = buf + rec(b, 0, 0);
        const int n = int(std::min<int64_t>(64, c->nc - b));
        if (n < 64) // the padding
            std::fill_n(blk, 64 * kRec, 0.0);
        for (int r = 0; r < 9; r++)
            for (int l = 0; l < n; l++) {
                const double *from = host + 36 * int64_t(c->d2c[b + l]) + r;
                double *to = blk + 256 * r + 4 * l;
                to[0] = from[0], to[1] = from[9], to[2] = from[18], to[3] = from[27];
            }
    }
}

static void rec_to_host(const dndsmi_ctx *c, const double *buf, double *host) {
    const int64_t last = kRec * c->ldc - 40;
    for (int64_t i = 0; i < c->nc; i++) {
        const double *ahead = buf + std::min(kRec * (i + 64), last);
        for (int q = 0; q < 5; q++)
            __builtin_prefetch(ahead + 8 * q);
        const double *from = buf + rec(c->c2d[i], 0, 0);
        double *to = host + 36 * i;
        for (int v = 0; v < 4; v++)
            for (int r = 0; r < 9; r++)
                to[r + 9 * v] = from[256 * r + v];
    }
}

extern "C" int dndsmi_array_upload(dndsmi_array *a, const double *host) {
    if (!a || !host || !a->ctx) // no context: it was destroyed before the array
        return DNDSMI_ERR_INVALID_ARGUMENT;
    dndsmi_ctx *c = a->ctx;
    const int64_t nc = c->nc, ldc = c->ldc;
    const std::vector<int32_t> &c2d = c->c2d;
    if (a->kind == DNDSMI_ARRAY_REC) {
        const size_t n = kRec * size_t(ldc);
        const std::unique_ptr<double[]> buf(new double[n]); // written below, the padding too
        rec_to_device(c, host, buf.get());
        DNDSMI_TRY(c->hip(hipMemcpyAsync(a->d, buf.get(), sizeof(double) * n, hipMemcpyHostToDevice, c->stream),
                          "upload"));
        return c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    }
    const int w = a->kind == DNDSMI_ARRAY_DOF ? 4 : 1;
    std::vector<double> buf(size_t(w) * ldc, 0.0);
    for (int64_t i = 0; i < nc; i++)
        for (int v = 0; v < w; v++)
            buf[size_t(w) * c2d[i] + v] = host[w * i + v];
    return c->upload(a->d, buf);
}

extern "C" int dndsmi_array_download(const dndsmi_array *a, double *host) {
    if (!a || !host || !a->ctx)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    dndsmi_ctx *c = a->ctx;
    const int64_t nc = c->nc, ldc = c->ldc;
    if (a->kind == DNDSMI_ARRAY_REC) {
        const size_t n = kRec * size_t(ldc);
        const std::unique_ptr<double[]> buf(new double[n]);
        DNDSMI_TRY(c->hip(hipMemcpyAsync(buf.get(), a->d, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream),
                          "download"));
        DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
        rec_to_host(c, buf.get(), host);
        return DNDSMI_OK;
    }
    const int w = a->kind == DNDSMI_ARRAY_DOF ? 4 : 1;
    std::vector<double> buf(size_t(w) * ldc);
    DNDSMI_TRY(c->hip(hipMemcpyAsync(buf.data(), a->d, sizeof(double) * buf.size(), hipMemcpyDeviceToHost, c->stream),
                      "download"));
    DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    for (int64_t i = 0; i < nc; i++)
        for (int v = 0; v < w; v++)
            host[w * i + v] = buf[size_t(w) * c->c2d[i] + v];
    return DNDSMI_OK;
}

extern "C" int dndsmi_array_copy(dndsmi_array *dst, const dndsmi_array *src) {
    if (!dst || !src || !dst->ctx || dst->ctx != src->ctx || dst->kind != src->kind)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    return dst->ctx->hip(hipMemcpyAsync(dst->d, src->d, sizeof(double) * dst->elems, hipMemcpyDeviceToDevice,
                                        dst->ctx->stream),
                         "copy");
}

extern "C" int dndsmi_array_set_constant(dndsmi_array *a, double value) {
    if (!a || !a->ctx)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    hipLaunchKernelGGL(k_set, dim3(grid_for(a->elems)), dim3(kBlock), 0, a->ctx->stream, a->elems, a->d, value);
    return a->ctx->launch_check("k_set");
}

namespace dndsmi_host {

// How many of every 64 blocks of the A^-1 B stream (`vecs` 16-byte vectors per
// cell and face) a sweep reads with ordinary loads.  The Infinity Cache (256
// MB) then still holds those at the next sweep, while the others, loaded
// non-temporally, pass it by; a stream read by ordinary loads throughout
// evicts itself once it is larger.  112 MB is what stays; small streams stay
// as a whole, and beyond `largest` bytes the rest of the traffic wins.
// Jacobi sweeps, us, none / 112 MB / all kept: 97 k triangles 52.7 / 49.4 /
// 46.2 (209 MB), 131 k 69.5 / 60.4 / 73.4 (283 MB), 218 k 105 / 93 / 116 (470),
// 320 k 152 / 143 / 168 (691), 405 k 200 / 194 / 215 (874), 524 k 255 / 254 / 274
// (1132), 1.0 M mixed cells 571 / 573 (2400).  FP32 sweeps: 264 k 76.6 / 69 / 87
// (265 MB), 524 k 147 / 142 / 163 (528), 980 k 268 / 276 / 289 (987).
int32_t keep_share(const dndsmi_ctx *c, int vecs, int64_t largest) {
    const int64_t stream = (2 * c->nf - c->n_bface) * 16 * vecs;
    constexpr int64_t kKept = 112000000;
    if (stream > largest)
        return 0;
    return stream <= kKept * 3 / 2 ? 64 : int32_t(kKept * 64 / stream);
}
constexpr int64_t kKeepLargest = 900000000, kKeepLargest32 = 600000000;
// the FP64 sweep of a mixed-precision stage shares the cache with the FP32 ones
constexpr int64_t kKeepLargestMixed = 450000000;

// A sweep takes 16 lanes per cell (k_jacobi_wide) while its whole stream stays
// in the Infinity Cache.  us, four lanes per cell / 16: FP64 triangles 1.8 k
// cells 8.9 / 7.2, 8 k 10.0 / 10.1, 33 k 20.0 / 20.1, 66 k 35.3 / 31.7, 80 k
// (173 MB) 40.4 / 36.8, 97 k (209 MB) 46.2 / 48.9, 180 k 76.6 / 104; mixed
// cells with walls 0.9 k 17.0 / 10.2, 9.5 k 20.8 / 18.3, 39 k 42.6 / 36.0.
bool wide_sweep(const dndsmi_ctx *c) { return keep_share(c, kAbVecs, kKeepLargest) == 64; }

// Workgroup size of an SOR pass or FP32 sweep over `lanes` lanes.  Waves are
// independent; small sweeps take one wave per workgroup, so that their waves
// spread over all CUs.  FP32 sweep, us, 64 / 256 threads: 1.8 k cells 7.4 / 8.4,
// 8 k 7.8 / 8.2, 33 k 12.2 / 12.1, 80 k 23.4 / 23.4, 146 k 39.1 / 38.3, 259 k
// 67.0 / 65.1; SOR colour of 1.8 k cells 8.5 / 9.2, of 131 k 22.9 / 23.6.
int sweep_block(int64_t lanes) { return lanes < 300000 ? 64 : kBlock; }

// SOR_Instead: colour by colour in place on x (forward; with
// SOR_InverseScanning then backward, DNDS_FV_VR.hpp:1493-1502)
int launch_sor(dndsmi_ctx *c, const double *u, double *x, double t) {
    const int passes = c->sor_inverse ? 2 : 1;
    for (int pass = 0; pass < passes; pass++)
        for (int32_t kk = 0; kk < c->n_colour; kk++) {
            const int32_t col = pass == 0 ? kk : c->n_colour - 1 - kk;
            // whole groups of 16 cells around the colour's range
            const int64_t b = c->sor_start[col], n = c->sor_start[col + 1] - b;
            if (n == 0)
                continue;
            const int64_t lanes = 4 * ((b & 15) + n);
            const int block = sweep_block(lanes);
            auto kern = c->nfmax == 3 ? k_sor<3> : k_sor<4>;
            prof_begin(c, DNDSMI_K_JACOBI);
            hipLaunchKernelGGL(kern, dim3(grid_for(lanes, block)), dim3(block), 0,
                               c->stream, int32_t(n), int32_t(b), c->ldc, c->nbr, c->sbc, c->M, u, x, x,
                               c->relax, c->walls, c->errw, keep_share(c, kAbVecs, kKeepLargest));
            prof_end(c);
            DNDSMI_TRY(c->launch_check("k_sor"));
        }
    return DNDSMI_OK;
}

int step_sweep(dndsmi_ctx *c, const double *u, double *&x, double *&xn, double t) {
    if (c->sor)
        return launch_sor(c, u, x, t);
    DNDSMI_TRY(launch_jacobi(c, u, x, xn, t));
    std::swap(x, xn);
    return DNDSMI_OK;
}

int launch_jacobi(dndsmi_ctx *c, const double *u, const double *x, double *xn, double t, double *diff2) {
    if (c->sor) {
        // the steps expect the new iterate in xn: start it from x, then update in place
        DNDSMI_TRY(c->hip(hipMemcpyAsync(xn, x, sizeof(double) * 36 * c->ldc, hipMemcpyDeviceToDevice, c->stream),
                          "copy uRec"));
        DNDSMI_TRY(launch_sor(c, u, xn, t));
        if (diff2)
            hipLaunchKernelGGL(k_rec_diff2, dim3(grid_for(4 * c->nc)), dim3(kBlock), 0, c->stream, int32_t(c->nc), x,
                               xn, diff2);
        return c->launch_check("k_rec_diff2");
    }
    if (wide_sweep(c)) {
        prof_begin(c, DNDSMI_K_JACOBI);
        hipLaunchKernelGGL((c->nfmax == 3 ? k_jacobi_wide<3, false> : k_jacobi_wide<4, false>),
                           dim3(grid_for(16 * c->nc, 64)), dim3(64), 0, c->stream, int32_t(c->nc), c->ldc, c->nbr,
                           c->sbc, c->M, u, x, xn, c->relax, c->walls, c->errw, nullptr, diff2);
        prof_end(c);
        return c->launch_check("k_jacobi_wide");
    }
    prof_begin(c, DNDSMI_K_JACOBI);
    hipLaunchKernelGGL((c->nfmax == 3 ? k_jacobi<3, false> : k_jacobi<4, false>), dim3(grid_for(4 * c->nc)),
                       dim3(kBlock), 0, c->stream, int32_t(c->nc), c->ldc, c->nbr, c->sbc, c->M, u, x, xn, c->relax,
                       c->walls, c->wall_corr, c->errw, nullptr, keep_share(c, kAbVecs, kKeepLargest), diff2);
    prof_end(c);
    return c->launch_check("k_jacobi");
}

int ensure_increment(dndsmi_ctx *c) {
    if (!c->rec_diff)
        DNDSMI_TRY(c->alloc(c->rec_diff, c->ldc));
    if (!c->host_sums)
        DNDSMI_TRY(c->hip(hipHostMalloc(&c->host_sums, sizeof(double) * 16 * size_t(grid_for(c->nc, 16 * 256)),
                                        hipHostMallocCoherent),
                          "hipHostMalloc"));
    return DNDSMI_OK;
}

int launch_increment(dndsmi_ctx *c, const double *u, const double *x, double *xn, double t) {
    DNDSMI_TRY(launch_jacobi(c, u, x, xn, t, c->rec_diff));
    hipLaunchKernelGGL(k_diff2_sums, dim3(grid_for(c->nc, 16 * 256)), dim3(1024), 0, c->stream, int32_t(c->nc),
                       c->rec_diff, c->host_sums);
    return c->launch_check("k_diff2_sums");
}

int launch_dt(dndsmi_ctx *c, const double *u, double cfl, double max_dt, double *dt_out) {
    const int nc = int(c->nc), nf = int(c->nf);
    prof_begin(c, DNDSMI_K_DT_FACE);
    hipLaunchKernelGGL(k_dt_face, dim3(grid_for(nf)), dim3(kBlock), 0, c->stream, nf, c->ldf, c->f2c, c->fnc, u,
                       c->gas, c->farea, c->vol, c->lambda_face, c->dlambda_face, c->errw);
    prof_end(c);
    const unsigned g = grid_for(nc);
    prof_begin(c, DNDSMI_K_DT_CELL);
    if (c->nfmax == 3)
        hipLaunchKernelGGL(k_dt_cell<3>, dim3(g), dim3(kBlock), 0, c->stream, nc, c->ldc, c->gat, c->lambda_face,
                           c->farea, c->vol, cfl, max_dt, dt_out, c->dt_part);
    else
        hipLaunchKernelGGL(k_dt_cell<4>, dim3(g), dim3(kBlock), 0, c->stream, nc, c->ldc, c->gat, c->lambda_face,
                           c->farea, c->vol, cfl, max_dt, dt_out, c->dt_part);
    prof_end(c);
    hipLaunchKernelGGL(k_min_final, dim3(1), dim3(kBlock), 0, c->stream, int32_t(g), c->dt_part, c->dt_min,
                       &c->host->dt_min, c->errw);
    return c->launch_check("dt kernels");
}

// Meshes with fewer faces take a quad per face.  EvaluateRHS with EvaluateDt,
// quads / one lane per face, us: Euler 8 k cells (12 k faces) 43 / 47, 16 k
// 45 / 49, 33 k (49 k faces) 52 / 49, 131 k 90 / 80; viscous 8 k 45 / 55, 16 k
// 48 / 56, 33 k 60 / 60, 131 k 116 / 114.
constexpr int64_t kQuadFaces = 40000;

// the face fluxes into fslot (MIXED: fslot32)
template <bool MIXED, bool VIS>
int launch_rhs_faces(dndsmi_ctx *c, const double *u, const double *x, double t, const double *xalt,
                     const uint8_t *limf) {
    const int32_t nf = int32_t(c->nf), nb = int32_t(c->n_bface);
    const FaceArgs fa{c->ldf,   c->nfmax, c->f2c,     c->fbc,  c->fxy,    c->cmom, c->fn,
                      c->fctr,  c->dlambda_face, u,   x,       c->gas,    t,
                      c->fpos,  c->fslot, c->fslot32, c->errw, c->cscale, c->vol,  c->farea, xalt, limf};
    const bool quads = nf < kQuadFaces;
    const int block = quads ? 64 : kBlock;
    const unsigned nbb = (grid_for(4 * int64_t(nb), block) + kNumXCD - 1) / kNumXCD * kNumXCD;
    prof_begin(c, MIXED ? DNDSMI_K_RHS_FACE32 : DNDSMI_K_RHS_FACE);
    if (quads)
        hipLaunchKernelGGL((k_rhs_face_quads<MIXED, VIS>), dim3(nbb + grid_for(4 * int64_t(nf), block)), dim3(block), 0,
                           c->stream, nb, int32_t(nbb), c->bfaces, nf, fa);
    else
        hipLaunchKernelGGL((c->straight_faces ? k_rhs_face<MIXED, true, VIS> : k_rhs_face<MIXED, false, VIS>),
                           dim3(nbb + grid_for(nf, block)), dim3(block), 0, c->stream, nb, int32_t(nbb), c->bfaces, fa,
                           nf, fa.ldf, fa.nfmax, fa.f2c, fa.fxy, fa.cmom, fa.fn, fa.dlf, fa.u, fa.x, fa.gp, fa.fpos,
                           fa.fslot, fa.fslot32, fa.errw, fa.cscale, fa.vol, fa.farea, fa.xalt, fa.limf);
    prof_end(c);
    return c->launch_check("k_rhs_face");
}

int launch_rhs(dndsmi_ctx *c, const double *u, const double *x, double t, double *rhs, int stage, double *xs,
               const double *dt, double coefA, double coefB, const double *xalt, const uint8_t *limf) {
    const int nc = int(c->nc);
    DNDSMI_TRY((c->gas.mu > 0 ? launch_rhs_faces<false, true> : launch_rhs_faces<false, false>)(c, u, x, t, xalt,
                                                                                               limf));
    prof_begin(c, DNDSMI_K_RHS_CELL);
    if (c->nfmax == 3)
        hipLaunchKernelGGL(k_rhs_cell<3>, dim3(grid_for(nc)), dim3(kBlock), 0, c->stream, nc, c->ldc, c->gat,
                           c->fslot, c->vol, rhs, stage, xs, c->xlast, dt, c->dt_min, coefA, coefB, c->errw);
    else
        hipLaunchKernelGGL(k_rhs_cell<4>, dim3(grid_for(nc)), dim3(kBlock), 0, c->stream, nc, c->ldc, c->gat,
                           c->fslot, c->vol, rhs, stage, xs, c->xlast, dt, c->dt_min, coefA, coefB, c->errw);
    prof_end(c);
    return c->launch_check("rhs kernels");
}

int launch_wbap(dndsmi_ctx *c, const double *u, const double *x, double *xo, double *ind, int if_all,
                int procedure, bool full_copy) {
    c->wbap_full_copy = full_copy;
    if (!c->has_limiter) {
        c->err = "WBAP needs a setup built with build_limiter_data";
        return DNDSMI_ERR_UNSUPPORTED;
    }
    const int nc = int(c->nc), nf = int(c->nf);
    const double eps4 = std::pow(1e-200, 1.0 / 4); // verySmallReal_pDiP, DNDS_FV_Limiters.hpp:345
    prof_begin(c, DNDSMI_K_WBAP_FACE);
    hipLaunchKernelGGL(k_wbap_face, dim3(grid_for(2 * int64_t(nf))), dim3(kBlock), 0, c->stream, nf, c->ldf,
                       c->nfmax, c->f2c, c->fxy, c->cmom, c->cscale, c->fw, c->fn, u, x, c->tang_weight, c->twd_norm,
                       c->wpos, c->wslot, c->lim_count);
    prof_end(c);
    prof_begin(c, DNDSMI_K_WBAP_CELL);
    if (c->nfmax == 3)
        hipLaunchKernelGGL(k_wbap_ind<3>, dim3(grid_for(nc)), dim3(kBlock), 0, c->stream, nc, c->ldc, c->nbr,
                           c->wslot, x, xo, ind ? ind : c->ind, c->wbap_scale, if_all, c->lim_count, c->lim_list,
                           full_copy ? nullptr : c->limf);
    else
        hipLaunchKernelGGL(k_wbap_ind<4>, dim3(grid_for(nc)), dim3(kBlock), 0, c->stream, nc, c->ldc, c->nbr,
                           c->wslot, x, xo, ind ? ind : c->ind, c->wbap_scale, if_all, c->lim_count, c->lim_list,
                           full_copy ? nullptr : c->limf);
    prof_end(c);
    prof_begin(c, DNDSMI_K_WBAP_LIM);
    // rows of 16 lanes walk the list, whose length only the device knows
    const dim3 grid(std::min(grid_for(16 * int64_t(nc)), kLimBlocks));
    if (procedure == 1) {
        hipLaunchKernelGGL((c->nfmax == 3 ? k_wbap_lim<3> : k_wbap_lim<4>), grid, dim3(kBlock), 0, c->stream, c->ldc,
                           c->ldf, c->lim_count, c->lim_list, c->nbr, c->sface, c->f2c, c->fnc, c->msec, u, x, xo,
                           c->gas.gamma, c->wbap_nstd, eps4, c->errw);
    } else {
        // orders 3, 2, 1 in stream order: each launch reads the rows the
        // previous ones wrote
        auto order = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(kBlock), 0, c->stream, c->ldc, c->ldf, c->lim_count, c->lim_list,
                               c->nbr, c->sface, c->f2c, c->fnc, c->msec, u, x, xo, c->gas.gamma, c->wbap_nstd, eps4,
                               c->errw, full_copy ? nullptr : c->limf);
        };
        order(c->nfmax == 3 ? k_wbap_lim_v2<3, 3> : k_wbap_lim_v2<4, 3>);
        order(c->nfmax == 3 ? k_wbap_lim_v2<3, 2> : k_wbap_lim_v2<4, 2>);
        order(c->nfmax == 3 ? k_wbap_lim_v2<3, 1> : k_wbap_lim_v2<4, 1>);
    }
    prof_end(c);
    return c->launch_check("wbap kernels");
}

int ensure_mixed(dndsmi_ctx *c) {
    if (c->M32)
        return DNDSMI_OK;
    const int64_t nm = int64_t(c->nfmax) * kAb32Vecs * 4 * c->ldc;
    DNDSMI_TRY(c->ensure(c->r32, 36 * c->ldc));
    DNDSMI_TRY(c->ensure(c->dA32, 36 * c->ldc));
    DNDSMI_TRY(c->ensure(c->dB32, 36 * c->ldc));
    DNDSMI_TRY(c->ensure(c->fslot32, int64_t(c->nfmax) * 8 * c->ldc));
    DNDSMI_TRY(c->ensure(c->wcorr32, kRec * c->n_wall));
    DNDSMI_TRY(c->alloc(c->M32, nm)); // the last: all are there where it is
    hipLaunchKernelGGL(k_m_to_f32, dim3(grid_for(nm / 4)), dim3(kBlock), 0, c->stream, int32_t(c->nfmax), c->ldc,
                       c->M, c->M32);
    DNDSMI_TRY(c->launch_check("k_m_to_f32"));
    return c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
}

// one FP64 step that yields r = J(x) - x, then n - 1 FP32 correction sweeps,
// the last adding the correction to x in place
int launch_jacobi_mixed(dndsmi_ctx *c, const double *u, double *x, int n_sweeps, double t) {
    const int64_t lanes = 4 * c->nc;
    const int block = sweep_block(lanes), nc = int(c->nc);
    const dim3 grid(grid_for(lanes, block));
    prof_begin(c, DNDSMI_K_JACOBI);
    if (wide_sweep(c)) {
        hipLaunchKernelGGL((c->nfmax == 3 ? k_jacobi_wide<3, true> : k_jacobi_wide<4, true>),
                           dim3(grid_for(16 * c->nc, 64)), dim3(64), 0, c->stream, nc, c->ldc, c->nbr, c->sbc, c->M, u,
                           x, nullptr, c->relax, c->walls, c->errw, c->r32, nullptr);
    } else {
        hipLaunchKernelGGL((c->nfmax == 3 ? k_jacobi<3, true> : k_jacobi<4, true>), dim3(grid_for(lanes)), dim3(kBlock),
                           0, c->stream, nc, c->ldc, c->nbr, c->sbc, c->M, u, x, nullptr, c->relax, c->walls,
                           c->wall_corr, c->errw, c->r32, keep_share(c, kAbVecs, kKeepLargestMixed), nullptr);
    }
    prof_end(c);
    DNDSMI_TRY(c->launch_check("k_jacobi (residual)"));
    const int32_t keep = keep_share(c, kAb32Vecs, kKeepLargest32);
    // d_0 = r: the first correction sweep reads r itself
    float *din = c->r32, *dout = c->dA32, *next = c->dB32;
    for (int k = 1; k < n_sweeps; k++) {
        auto kern = k == n_sweeps - 1 ? (c->nfmax == 3 ? k_delta32<3, true> : k_delta32<4, true>)
                                      : (c->nfmax == 3 ? k_delta32<3, false> : k_delta32<4, false>);
        prof_begin(c, DNDSMI_K_DELTA32);
        hipLaunchKernelGGL(kern, grid, dim3(block), 0, c->stream, nc, c->ldc, c->nbr, c->sbc, c->M32,
                           c->r32, din, dout, float(c->relax), x, c->walls,
                           c->wcorr32, keep);
        prof_end(c);
        DNDSMI_TRY(c->launch_check("k_delta32"));
        din = dout;
        std::swap(dout, next);
    }
    return DNDSMI_OK;
}

int launch_rhs_mixed(dndsmi_ctx *c, const double *u, const double *x, double t, double *rhs, int stage, double *xs,
                     const double *dt, double coefA, double coefB, const double *xalt, const uint8_t *limf) {
    const int nc = int(c->nc);
    DNDSMI_TRY((launch_rhs_faces<true, false>(c, u, x, t, xalt, limf)));
    prof_begin(c, DNDSMI_K_RHS_CELL32);
    if (c->nfmax == 3)
        hipLaunchKernelGGL((k_rhs_cell<3, float>), dim3(grid_for(nc)), dim3(kBlock), 0, c->stream, nc, c->ldc,
                           c->gat, c->fslot32, c->vol, rhs, stage, xs, c->xlast, dt, c->dt_min, coefA, coefB,
                           c->errw);
    else
        hipLaunchKernelGGL((k_rhs_cell<4, float>), dim3(grid_for(nc)), dim3(kBlock), 0, c->stream, nc, c->ldc,
                           c->gat, c->fslot32, c->vol, rhs, stage, xs, c->xlast, dt, c->dt_min, coefA, coefB,
                           c->errw);
    prof_end(c);
    return c->launch_check("mixed rhs kernels");
}

} // namespace dndsmi_host

namespace {

int wbap_entry(dndsmi_ctx *c, const dndsmi_array *u, const dndsmi_array *uRec, dndsmi_array *uRecNewBuf,
               dndsmi_array *uRecNewBuf1, dndsmi_array *ifUseLimiter, int32_t ifAll, int procedure) {
    if (!c || !same_ctx(c, u, DNDSMI_ARRAY_DOF) || !same_ctx(c, uRec, DNDSMI_ARRAY_REC) ||
        !same_ctx(c, uRecNewBuf, DNDSMI_ARRAY_REC) || uRec == uRecNewBuf ||
        (uRecNewBuf1 && (!same_ctx(c, uRecNewBuf1, DNDSMI_ARRAY_REC) || uRecNewBuf1 == uRec ||
                         uRecNewBuf1 == uRecNewBuf)) ||
        (ifUseLimiter && !same_ctx(c, ifUseLimiter, DNDSMI_ARRAY_SCALAR)))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(launch_wbap(c, u->d, uRec->d, uRecNewBuf->d, ifUseLimiter ? ifUseLimiter->d : nullptr, ifAll,
                           procedure));
    if (uRecNewBuf1)
        DNDSMI_TRY(c->hip(hipMemcpyAsync(uRecNewBuf1->d, uRecNewBuf->d, sizeof(double) * uRecNewBuf->elems,
                                         hipMemcpyDeviceToDevice, c->stream),
                          "copy"));
    return DNDSMI_OK;
}

} // namespace

extern "C" int dndsmi_wbap_limit_facial_v3(dndsmi_ctx *c, const dndsmi_array *u, const dndsmi_array *uRec,
                                           dndsmi_array *uRecNewBuf, dndsmi_array *uRecNewBuf1,
                                           dndsmi_array *ifUseLimiter, int32_t ifAll) {
    return wbap_entry(c, u, uRec, uRecNewBuf, uRecNewBuf1, ifUseLimiter, ifAll, 1);
}

extern "C" int dndsmi_wbap_limit_facial_v2(dndsmi_ctx *c, const dndsmi_array *u, const dndsmi_array *uRec,
                                           dndsmi_array *uRecNewBuf, dndsmi_array *uRecNewBuf1,
                                           dndsmi_array *ifUseLimiter, int32_t ifAll) {
    return wbap_entry(c, u, uRec, uRecNewBuf, uRecNewBuf1, ifUseLimiter, ifAll, 0);
}

extern "C" int dndsmi_set_limiter_procedure(dndsmi_ctx *c, int32_t limiterProcedure) {
    if (!c || (limiterProcedure != 0 && limiterProcedure != 1))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    c->limiter_procedure = limiterProcedure;
    return DNDSMI_OK;
}

extern "C" int dndsmi_set_limiter_if_all(dndsmi_ctx *c, int32_t ifAll) {
    if (!c)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    c->limiter_if_all = ifAll != 0;
    return DNDSMI_OK;
}

extern "C" int dndsmi_reconstruction_jacobi_step(dndsmi_ctx *c, const dndsmi_array *u, dndsmi_array *uRec,
                                                 dndsmi_array *uRecNewBuf, double t) {
    if (!c || !same_ctx(c, u, DNDSMI_ARRAY_DOF) || !same_ctx(c, uRec, DNDSMI_ARRAY_REC) ||
        !same_ctx(c, uRecNewBuf, DNDSMI_ARRAY_REC) || uRec == uRecNewBuf)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (c->sor) // in place on uRec; uRecNewBuf is not touched (DNDS_FV_VR.hpp:1507-1510, 1707)
        return launch_sor(c, u->d, uRec->d, t);
    DNDSMI_TRY(launch_jacobi(c, u->d, uRec->d, uRecNewBuf->d, t));
    // uRec = uRecNewBuf (DNDS_FV_VR.hpp:1707-1711): afterwards both arrays
    // hold the new iterate, as in the reference.
    return c->hip(hipMemcpyAsync(uRec->d, uRecNewBuf->d, sizeof(double) * uRec->elems, hipMemcpyDeviceToDevice,
                                 c->stream),
                  "copy uRecNewBuf to uRec");
}

extern "C" int dndsmi_evaluate_dt(dndsmi_ctx *c, dndsmi_array *dt, const dndsmi_array *u, double CFL,
                                  double *dtMinall, double MaxDt, int32_t UseLocaldt) {
    if (!c || !same_ctx(c, dt, DNDSMI_ARRAY_SCALAR) || !same_ctx(c, u, DNDSMI_ARRAY_DOF))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(launch_dt(c, u->d, CFL, MaxDt, dt->d));
    if (!UseLocaldt) {
        hipLaunchKernelGGL(k_fill_from, dim3(grid_for(c->nc)), dim3(kBlock), 0, c->stream, int32_t(c->nc), c->dt_min,
                           dt->d);
        DNDSMI_TRY(c->launch_check("k_fill_from"));
    }
    if (dtMinall) {
        const int rc = check_errw(c);
        *dtMinall = c->host->dt_min;
        return rc;
    }
    return DNDSMI_OK;
}

extern "C" int dndsmi_evaluate_rhs(dndsmi_ctx *c, dndsmi_array *rhs, const dndsmi_array *u, const dndsmi_array *uRec,
                                   double t) {
    if (!c || !same_ctx(c, rhs, DNDSMI_ARRAY_DOF) || !same_ctx(c, u, DNDSMI_ARRAY_DOF) ||
        !same_ctx(c, uRec, DNDSMI_ARRAY_REC))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    return launch_rhs(c, u->d, uRec->d, t, rhs->d, 0, nullptr, nullptr, 0, 0);
}

extern "C" int dndsmi_ssprk3_step(dndsmi_ctx *c, dndsmi_array *u, dndsmi_array *uRec, dndsmi_array *uRecNew,
                                  int32_t n_sweeps, int32_t use_limiter, double CFL, double MaxDt, int32_t UseLocaldt,
                                  double t, double *dt_out) {
    if (!c || !same_ctx(c, u, DNDSMI_ARRAY_DOF) || !same_ctx(c, uRec, DNDSMI_ARRAY_REC) ||
        !same_ctx(c, uRecNew, DNDSMI_ARRAY_REC) || uRec == uRecNew || n_sweeps < 0)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (use_limiter && !c->has_limiter) {
        c->err = "WBAP needs a setup built with build_limiter_data";
        return DNDSMI_ERR_UNSUPPORTED;
    }
    // fdt: EvaluateDt; the stage update reads dt_i (local) or the device minimum
    DNDSMI_TRY(launch_dt(c, u->d, CFL, MaxDt, c->dt_tmp));
    // the global minimum sets the stage times (one host read per step)
    DNDSMI_TRY(check_errw(c));
    const double dtmin = c->host->dt_min;
    if (dt_out)
        *dt_out = dtmin;
    const double Coef[3] = {1.0, 0.25, 2.0 / 3.0};
    const double ct[3] = {1, 0.25, 2. / 3.};
    for (int stage = 0; stage < 3; stage++) {
        const double ts = t + ct[stage] * dtmin;
        for (int k = 0; k < n_sweeps; k++) {
            DNDSMI_TRY(step_sweep(c, u->d, uRec->d, uRecNew->d, ts));
        }
        const double cA = stage ? Coef[stage] / (1 - Coef[stage]) : 0.0;
        const double cB = stage ? 1 - Coef[stage] : 0.0;
        // the RHS sees the limited cells from xlim (flagged), the others from
        // uRec, which keeps the unlimited iterate
        if (use_limiter)
            DNDSMI_TRY(launch_wbap(c, u->d, uRec->d, c->xlim, nullptr, c->limiter_if_all, c->limiter_procedure, false));
        DNDSMI_TRY(launch_rhs(c, u->d, uRec->d, ts, nullptr, stage + 1, u->d, UseLocaldt ? c->dt_tmp : nullptr, cA,
                              cB, use_limiter ? c->xlim : nullptr, use_limiter ? c->limf : nullptr));
    }
    return DNDSMI_OK;
}

namespace {

// the three stages of a mixed-precision SSP-RK3 step on (u, x) after
// EvaluateDt (c->dt_tmp and dtmin set); `ws`: the stages run the learned
// warm start's hook, adding its correction when `correct`
int mixed_stages(dndsmi_ctx *c, double *u, double *x, int32_t n_sweeps, int32_t use_limiter, int32_t UseLocaldt,
                 double t, double dtmin, bool ws, bool correct) {
    const double Coef[3] = {1.0, 0.25, 2.0 / 3.0};
    const double ct[3] = {1, 0.25, 2. / 3.};
    for (int stage = 0; stage < 3; stage++) {
        const double ts = t + ct[stage] * dtmin;
        if (ws)
            DNDSMI_TRY(ws_stage_begin(c, u, x, correct));
        DNDSMI_TRY(launch_jacobi_mixed(c, u, x, n_sweeps, ts));
        const double cA = stage ? Coef[stage] / (1 - Coef[stage]) : 0.0;
        const double cB = stage ? 1 - Coef[stage] : 0.0;
        if (use_limiter)
            DNDSMI_TRY(launch_wbap(c, u, x, c->xlim, nullptr, c->limiter_if_all, c->limiter_procedure, false));
        DNDSMI_TRY(launch_rhs_mixed(c, u, x, ts, nullptr, stage + 1, u, UseLocaldt ? c->dt_tmp : nullptr, cA, cB,
                                    use_limiter ? c->xlim : nullptr, use_limiter ? c->limf : nullptr));
    }
    return DNDSMI_OK;
}

} // namespace

extern "C" int dndsmi_ssprk3_step_mixed(dndsmi_ctx *c, dndsmi_array *u, dndsmi_array *uRec, dndsmi_array *uRecNew,
                                        int32_t n_sweeps, int32_t use_limiter, double CFL, double MaxDt,
                                        int32_t UseLocaldt, double t, double *dt_out) {
    if (!c || !same_ctx(c, u, DNDSMI_ARRAY_DOF) || !same_ctx(c, uRec, DNDSMI_ARRAY_REC) ||
        !same_ctx(c, uRecNew, DNDSMI_ARRAY_REC) || uRec == uRecNew || n_sweeps < 2)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (use_limiter && !c->has_limiter) {
        c->err = "WBAP needs a setup built with build_limiter_data";
        return DNDSMI_ERR_UNSUPPORTED;
    }
    if (c->sor) {
        c->err = "the mixed-precision step iterates the Jacobi map (SOR_Instead must be off)";
        return DNDSMI_ERR_UNSUPPORTED;
    }
    if (c->gas.mu > 0) {
        c->err = "the mixed-precision step covers the Euler model (muGas = 0) only";
        return DNDSMI_ERR_UNSUPPORTED;
    }
    DNDSMI_TRY(ensure_mixed(c));
    // the learned warm start: is this step in a check window (the plain run
    // on shadow copies beside the corrected one)?
    const bool ws = c->step_ws && !c->ws_rejected;
    bool window = false;
    if (ws) {
        if (c->ws_win_left == 0 && (c->ws_first || (c->ws_recheck > 0 && c->ws_since_check >= c->ws_recheck))) {
            DNDSMI_TRY(ws_window_begin(c, u->d, uRec->d));
            c->ws_win_left = c->ws_check_steps;
            c->ws_first = false;
        }
        window = c->ws_win_left > 0;
    }
    // the step's dt: from the plain run's state in a window, used by both runs
    DNDSMI_TRY(launch_dt(c, window ? c->ws_sh_u : u->d, CFL, MaxDt, c->dt_tmp));
    DNDSMI_TRY(check_errw(c));
    const double dtmin = c->host->dt_min;
    if (dt_out)
        *dt_out = dtmin;
    if (!window) {
        if (ws)
            c->ws_since_check++;
        return mixed_stages(c, u->d, uRec->d, n_sweeps, use_limiter, UseLocaldt, t, dtmin, ws, ws);
    }
    DNDSMI_TRY(mixed_stages(c, c->ws_sh_u, c->ws_sh_x, n_sweeps, use_limiter, UseLocaldt, t, dtmin, false, false));
    DNDSMI_TRY(check_errw(c)); // the plain run's own failures are the method's
    int rc = mixed_stages(c, u->d, uRec->d, n_sweeps, use_limiter, UseLocaldt, t, dtmin, true, true);
    if (rc == DNDSMI_OK)
        rc = check_errw(c);
    const bool failed = rc == DNDSMI_ERR_NONPOSITIVE_STATE || rc == DNDSMI_ERR_NAN;
    if (rc != DNDSMI_OK && !failed)
        return rc;
    c->ws_win_left--;
    if (failed || c->ws_win_left == 0) {
        DNDSMI_TRY(ws_window_end(c, u->d, uRec->d, failed));
        c->ws_since_check = 0;
        c->ws_win_left = 0;
    }
    return DNDSMI_OK;
}

// ---- profiling ---------------------------------------------------------

extern "C" int dndsmi_read_probe(dndsmi_ctx *c, int32_t reps) {
    if (!c || reps < 1)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (!c->probe_out)
        DNDSMI_TRY(c->alloc(c->probe_out, 4 * c->ldc));
    for (int k = 0; k < reps; k++) {
        prof_begin(c, DNDSMI_K_READ_PROBE);
        hipLaunchKernelGGL((c->nfmax == 3 ? k_read_probe<3> : k_read_probe<4>), dim3(grid_for(4 * c->nc)),
                           dim3(kBlock), 0, c->stream, int32_t(c->nc), c->ldc, c->nbr, c->M, c->probe_out,
                           keep_share(c, kAbVecs, kKeepLargest));
        prof_end(c);
        DNDSMI_TRY(c->launch_check("k_read_probe"));
    }
    return DNDSMI_OK;
}

extern "C" int dndsmi_profile_enable(dndsmi_ctx *c, int32_t on) {
    if (!c)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    c->prof_on = on != 0;
    c->prof_recs.clear();
    c->ev_used = 0;
    return DNDSMI_OK;
}

extern "C" int dndsmi_profile_query(dndsmi_ctx *c, int32_t kernel, int64_t *count, double *total_ms) {
    if (!c || !count || !total_ms || kernel < 0 || kernel >= DNDSMI_K_COUNT)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    int64_t n = 0;
    double tot = 0;
    for (auto &r : c->prof_recs) {
        if (r.first != kernel)
            continue;
        float ms = 0;
        DNDSMI_TRY(c->hip(hipEventElapsedTime(&ms, c->ev_pool[r.second], c->ev_pool[r.second + 1]),
                          "hipEventElapsedTime"));
        tot += ms;
        n++;
    }
    *count = n;
    *total_ms = tot;
    return DNDSMI_OK;
}

// Algorithmic (unique) HBM bytes of one launch of a kernel: every stream the
// kernel needs read once and every output written once, from mesh counts.
extern "C" int64_t dndsmi_kernel_bytes(const dndsmi_ctx *c, int32_t kernel) {
    if (!c)
        return -1;
    const int64_t nc = c->nc, nf = c->nf, nif = nf - c->n_bface, nbf = c->n_bface;
    int64_t c2f = 0; // sum of faces per cell = 2 nif + nbf
    c2f = 2 * nif + nbf;
    switch (kernel) {
    case DNDSMI_K_JACOBI: // M + b per slot, slot neighbour index, x read + x_new write, u
        return c2f * (81 + 9) * 8 + c2f * 4 + nc * (36 * 8 * 2 + 4 * 8);
    case DNDSMI_K_DT_FACE: // f2c, centre normal, lambda + dlambda out; u once per cell
        return nf * (8 + 16 + 16) + nc * 32;
    case DNDSMI_K_DT_CELL: // gather index, lambda + area per slot, volume, dt out
        return c2f * (4 + 16) + nc * (8 + 8);
    case DNDSMI_K_RHS_FACE: // f2c, slot positions, point coordinates, normals, dlambda, 2 x 8 terms out;
        // x, u and the moments once per cell; viscous: face area, both volumes and cell scales; boundary faces:
        // index, f2c, slot position, kind, one side's point coordinates, normals, centre, dlambda, 8 terms out
        return c->n_bface * (4 + 8 + 1 + 4 + 48 + 48 + 16 + 8 + 64 + (c->gas.mu > 0 ? 8 + 8 + 16 : 0)) +
               nif * (8 + 1 + 96 + (c->straight_faces ? 16 : 48) + 8 + 128 + (c->gas.mu > 0 ? 8 + 16 + 32 : 0)) +
               nc * (36 * 8 + 32 + 72);
    case DNDSMI_K_RHS_CELL: // 8 terms per slot, volume, x read+write, xLast (+ last-slot index for 4 slots)
        return c2f * 64 + nc * (8 + 32 * 3 + (c->nfmax == 4 ? 4 : 0));
    case DNDSMI_K_WBAP_FACE: // point-0 coordinates of both sides, f2c, slot positions, weights, normal, 8 terms
        // out; x (rho, E), u (rho, E), moments and scales once per cell
        return nif * (32 + 8 + 1 + 80 + 16 + 64) + nc * (18 * 8 + 16 + 72 + 16);
    case DNDSMI_K_WBAP_CELL: // terms and neighbour index per slot, indicator out; x read and copied out for the
        // unlimited cells of a full copy (an upper bound: as if no cell were limited), else a flag per cell
        return c2f * (32 + 4) + nc * (8 + (c->wbap_full_copy ? 36 * 8 * 2 : 1));
    case DNDSMI_K_WBAP_LIM: // depends on the number of limited cells; not a bandwidth kernel
        return 0;
    case DNDSMI_K_LUSGS_MATVEC: // per scan position cell, D, x own in, Ax out; per slot both neighbour indices,
        // normal, c_f, lambda, u and x of the neighbour
        return nc * (4 + 8 + 32 + 32) + c2f * (8 + 16 + 16 + 32 + 32);
    case DNDSMI_K_LUSGS_SWEEP: // one whole forward (or backward) sweep, all colours together: per scan position
        // cell, 1/D, rhs (or the increment) in, increment out; per slot the neighbour index, and per used slot
        // (half of them) normal, c_f, lambda, u and the increment of the neighbour
        return nc * (4 + 8 + 32 + 32) + c2f * 4 + c2f / 2 * (16 + 16 + 32 + 32);
    case DNDSMI_K_DELTA32: // FP32 M per slot + slot index; d read + r read + d write (FP32)
        return c2f * (81 * 4 + 4) + nc * (36 * 4 * 3);
    case DNDSMI_K_RHS_FACE32: // as DNDSMI_K_RHS_FACE with 2 x 8 FP32 terms out
        return c->n_bface * (4 + 8 + 1 + 4 + 48 + 48 + 16 + 8 + 32) +
               nif * (8 + 1 + 96 + (c->straight_faces ? 16 : 48) + 8 + 64) + nc * (36 * 8 + 32 + 72);
    case DNDSMI_K_RHS_CELL32: // 8 FP32 terms per slot, volume, x read+write, xLast (+ last-slot index)
        return c2f * 32 + nc * (8 + 32 * 3 + (c->nfmax == 4 ? 4 : 0));
    case DNDSMI_K_READ_PROBE: // the sweep's A^-1 B, A^-1 b (45 x 16 B per slot) and slot index, four doubles out
        return c2f * (kAbVecs * 16 + 4) + nc * 32;
    default:
        return 0;
    }
}
