// gfx950 kernels of the PME variable group: OpenMM's NonbondedForce with
// particle-mesh Ewald evaluated on x and on x + d, then the ATM combine.
//
// Direct space and charge spreading of x:
//   k_pme_begin      inputs from the host's memory; clear the cell counts, charge grids and force sums
//   k_pme_bin        (form x + d) wrap into the box, cell of edge >= rc, rank in the cell
//   k_pme_scan       cell starts (one block)
//   k_pme_scatter    atom indices into cell order
//   k_pme_cellsort   each cell ordered by atom index (deterministic sums), and
//                    positions / parameters / exclusion keys / displacement
//                    classes gathered into cell order
//   k_pme_direct     erfc(alpha r)/r Coulomb + LJ over minimum-image pairs with
//                    r < rc that are not exceptions; one block per (64 atoms of a
//                    cell, the cell or one of its 13 forward neighbours): each pair once
//   k_pme_spread_tiles  order-5 B-spline charge spreading per cell into an LDS
//                    tile of the grid, 64-bit fixed point (k_pme_spread: the
//                    same straight into the grid, when a tile does not fit)
// x + d differs from x at the displaced atoms only.  When they are few (at most one in
// 16) k_pme_direct takes the pairs whose separation d leaves alone, once for both
// states, k_pme_displaced the others at x and at x + d, and the charges move on a
// difference grid; otherwise the same kernels run on x + d.  Then for both states at
// once (blockIdx.y):
//   k_pme_planes     two axes of the forward transform per plane of the grid, in LDS
//   k_pme_lines      the third axis forward, influence function, reciprocal energy,
//                    convolution, the third axis back
//   k_pme_planes     the other two axes back, to the real potential
//                    (k_pme_dft_lines / k_pme_convolve, one pass per axis, where a plane
//                    does not fit a block; k_pme_q2c + k_pme_dft for lines too long for LDS)
//   k_pme_gather     reciprocal forces from the potential grid; exception pairs:
//                    own Coulomb + LJ, minus erf(alpha r)/r
// and once per evaluation:
//   k_pme_finish     fixed-order sums of every energy slot, U1, U2, combine
//   k_pme_blend      F += (1 - sp) F1 + sp F2 (direction-aware), FP64 out
//
// Everything is FP64: positions, pair function, grid, transforms.  Forces are
// summed in 64-bit fixed point (2^-24 kJ/mol/nm) with integer atomics, energies
// in per-block slots reduced in a fixed order, so results are bit-reproducible.
//
// The model restated is OpenMM's PME NonbondedForce as the reference's
// end-to-end test builds it (python/tests/test_abfe.py:42-43, through
// AmberPrmtopFile.createSystem), cloned into the ATM inner contexts at
// openmmapi/src/ATMMetaForceImpl.cpp:58-63 and combined by
// platforms/reference/src/ReferenceATMMetaForceKernels.cpp:56-110.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "atm_pme.h"
#include "atm_math.h"
#include "atm_wrap.h"

namespace atm {

namespace {

constexpr double kFix = 16777216.0;          // 2^24 force units per kJ/mol/nm
constexpr double kGridFix = 68719476736.0;   // 2^36 charge-grid units per e
constexpr int kOrder = 5;

__device__ __forceinline__ unsigned long long fixed_force(double f) { return (unsigned long long)__double2ll_rn(f * kFix); }

__device__ __forceinline__ void add_fixed(unsigned long long* p, double f) { atomicAdd(p, fixed_force(f)); }

// Integer add in LDS (workgroup scope, no result).
__device__ __forceinline__ void lds_add(unsigned long long* p, unsigned long long v) {
    typedef __attribute__((address_space(3))) unsigned long long LdsU64;
    __hip_atomic_fetch_add((LdsU64*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// A whole number below 2^51 as an integer: the low bits of its sum with 1.5 2^52.
__device__ __forceinline__ long long whole(double v) {
    return __double_as_longlong(v + 6755399441055744.0) - 0x4338000000000000LL;
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over each aligned octet of lanes (xor 1, xor 2, half-row mirror by DPP).
__device__ __forceinline__ double oct_sum(double v) {
    v += dpp_f64<0xB1>(v);
    v += dpp_f64<0x4E>(v);
    v += dpp_f64<0x141>(v);
    return v;
}

// Grid index v in [-K, 2K) wrapped into [0, K) (no integer division).
__device__ __forceinline__ int wrap_index(int v, int K) {
    v = v < 0 ? v + K : v;
    return v >= K ? v - K : v;
}

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block sum (fixed order) of one value per thread; valid in thread 0.
template <int NT>
__device__ double block_sum(double v, double* red) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[w] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int k = 0; k < NT / 64; ++k) s += red[k];
    __syncthreads();
    return s;
}

// Order-5 cardinal B-spline weights M5(w + j) and derivatives M5'(w + j),
// j = 0..4, for w in [0, 1) (two-term recursion M_k(t) = t/(k-1) M_{k-1}(t)
// + (k-t)/(k-1) M_{k-1}(t-1), from M_2(w) = w, M_2(w+1) = 1 - w).
__device__ __forceinline__ void bspline5(double w, double th[kOrder], double dth[kOrder]) {
    double a[kOrder] = {w, 1.0 - w, 0.0, 0.0, 0.0};
    for (int k = 3; k <= kOrder; ++k) {
        double nw[kOrder];
        const double inv = 1.0 / (k - 1);
        for (int j = 0; j < kOrder; ++j) {
            const double am1 = j > 0 ? a[j - 1] : 0.0;
            nw[j] = j < k ? ((w + j) * a[j] + (k - w - j) * am1) * inv : 0.0;
        }
        if (k == kOrder)
            for (int j = 0; j < kOrder; ++j) dth[j] = a[j] - (j > 0 ? a[j - 1] : 0.0);
        for (int j = 0; j < kOrder; ++j) a[j] = nw[j];
    }
    for (int j = 0; j < kOrder; ++j) th[j] = a[j];
}

}  // namespace

// Cell of every atom and its rank among the cell's atoms (any order: the cell
// sort fixes it).  Ranks come from a block histogram in LDS and one global
// atomic per (block, occupied cell), so the few hundred atoms of a cell do not
// serialise on one counter; grids with more than kPmeBinLds cells use global
// atomics directly.
// d: when not null, x + d (the displaced state) is written to P.x2 for the kernels
// after this one; shifted: those positions are the ones binned.
__global__ void __launch_bounds__(256) k_pme_bin(PmeDesc D, PmePtrs P, const double* x, const double* d, int shifted) {
    __shared__ int hist[kPmeBinLds];
    __shared__ int base[kPmeBinLds];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool lds = D.ncell <= kPmeBinLds;
    if (lds) {
        for (int c = threadIdx.x; c < D.ncell; c += blockDim.x) hist[c] = 0;
        __syncthreads();
    }
    int c = -1, r = 0;
    if (i < D.n) {
        double w[3], xi[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
        if (d) {
            for (int k = 0; k < 3; ++k) {
                const double v = xi[k] + d[3 * i + k];
                P.x2[3 * i + k] = v;
                if (shifted) xi[k] = v;
            }
        }
        const int cx = wrap_cell(xi[0], D.L[0], D.invL[0], D.m[0], &w[0]);
        const int cy = wrap_cell(xi[1], D.L[1], D.invL[1], D.m[1], &w[1]);
        const int cz = wrap_cell(xi[2], D.L[2], D.invL[2], D.m[2], &w[2]);
        c = (cx * D.m[1] + cy) * D.m[2] + cz;
        P.cellOf[i] = c;
        P.wpos[i] = make_double4(w[0], w[1], w[2], 0.0);
        r = lds ? atomicAdd(&hist[c], 1) : atomicAdd(&P.cellCount[c], 1);
    }
    if (lds) {
        __syncthreads();
        for (int k = threadIdx.x; k < D.ncell; k += blockDim.x)
            base[k] = hist[k] ? atomicAdd(&P.cellCount[k], hist[k]) : 0;
        __syncthreads();
        if (c >= 0) r += base[c];
    }
    if (i < D.n) P.rankOf[i] = r;
}

__global__ void __launch_bounds__(1024) k_pme_scan(PmeDesc D, PmePtrs P) {
    __shared__ int part[1024];
    const int t = threadIdx.x;
    const int per = (D.ncell + 1023) / 1024;
    const int b0 = t * per, b1 = min(b0 + per, D.ncell);
    int s = 0, mx = 0;
    for (int c = b0; c < b1; ++c) { s += P.cellCount[c]; mx = max(mx, P.cellCount[c]); }
    part[t] = s;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = part[t] - s;
    for (int c = b0; c < b1; ++c) { P.cellStart[c] = run; run += P.cellCount[c]; }
    if (t == 1023) P.cellStart[D.ncell] = part[1023];
    if (mx > D.cellCap) atomicOr(P.overflow, 1);
}

__global__ void k_pme_scatter(PmeDesc D, PmePtrs P) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D.n) return;
    P.cellAtoms[P.cellStart[P.cellOf[i]] + P.rankOf[i]] = i;
}

// One block per cell: order its atoms by index and gather them into cell order.
__global__ void __launch_bounds__(256) k_pme_cellsort(PmeDesc D, PmePtrs P) {
    __shared__ int ids[kPmeCellMax];
    const int c = blockIdx.x;
    const int s0 = P.cellStart[c], cnt = min(P.cellStart[c + 1] - s0, kPmeCellMax);
    for (int k = threadIdx.x; k < cnt; k += blockDim.x) ids[k] = P.cellAtoms[s0 + k];
    __syncthreads();
    for (int k = threadIdx.x; k < cnt; k += blockDim.x) {
        const int a = ids[k];
        int r = 0;
        for (int l = 0; l < cnt; ++l) r += ids[l] < a;
        const int slot = s0 + r;
        const double4 w = P.wpos[a];
        const double2 pr = P.prm[a];
        P.cpos[slot] = make_double4(w.x, w.y, w.z, pr.x);
        P.cprm[slot] = make_double2(P.prm2[a].x, P.prm2[a].y);
        const int4 ex = P.exkey[a];
        P.cex[slot] = make_int4(ex.x, ex.y, ex.z, a | ex.w << kPmeClassShift);
    }
}

// erfc(alpha r)/r Coulomb + LJ of one pair from r^2 (qq = k_e q q', sg = mixed sigma,
// e4 = 4 eps): the energy; fs, the force over the separation.
__device__ __forceinline__ double direct_pair(const PmeDesc& D, double r2, double qq, double sg, double e4, double& fs) {
    const double a = D.alpha;
    // 1/r: hardware estimate and two Newton steps on the residual 1 - r2 y^2 (an FMA)
    double rinv = __builtin_amdgcn_rsq(r2);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const double t = r2 * rinv;
        rinv = fma(0.5 * rinv, fma(-t, rinv, 1.0), rinv);
    }
    const double r = r2 * rinv, r2inv = rinv * rinv;
    const double ec = qq * erfc(a * r) * rinv;
    const double s2 = sg * sg * r2inv, s6 = s2 * s2 * s2;
    const double t = e4 * s6;
    const double elj = fma(t, s6, -t);
    fs = (ec + qq * D.twoAlphaSqrtPi * exp(-a * a * r2) + fma(12.0, elj, 6.0 * t)) * r2inv;
    return ec + elj;
}

// Half shell: neighbour 0 is cell c itself (pairs with the j slot above the i slot), 1..13
// its forward neighbour cells (all pairs).  Every pair is visited once: +f on i, -f on j,
// the whole pair energy.
//
// One block of 4 waves per (cell c, fastest; kPmeIBlock atoms of c; neighbour): those atoms
// and, kPmeJBlock at a time, the neighbour cell's are staged in LDS with their force sums.
// Each wave takes its share of the staged j-atoms against every i-atom:
//  test:  lane il + n2 jg tests i-atom il of a chunk of up to 64 against j-atom k G + jg (a
//         chunk of n2 = 8, 16, 32 or 64 i-atoms takes G = 64 / n2 j-atoms a step, so the 5
//         atoms left of a cell of 133 cost an eighth of a full chunk).  FP64 r^2, the
//         image shift known from the cell offset, exclusion bitmap for atoms of one
//         exclusion group; in-range pairs are appended to the wave's ring in LDS (ballot +
//         mbcnt, so the order is fixed);  shared: pairs of atoms displaced differently are left
//         out (looked up only where a wave's atoms hold a displaced one);
//  dense: whenever 64 pairs are pending, each lane evaluates one of them
//         (erfc Coulomb + LJ in FP64); forces go to the block's LDS sums in 64-bit fixed
//         point (integer atomics: order-independent).
// The dense steps bound it (some 230 VALU instructions and six 64-bit LDS adds each):
// pairs of one j-atom sit in consecutive lanes and their adds queue on one address, so an
// octet of lanes of one j-atom adds up first (LDS conflict cycles halved, 85 -> 73 us with
// blocks of 8 waves).  59 -> 48 us for 8,479 atoms, 151 -> 120 for 25,437, against one wave
// per (64 atoms, neighbour, quarter of its atoms) with its own sums.
__global__ void __launch_bounds__(64 * kPmeDirectWaves, 4) k_pme_direct(PmeDesc D, PmePtrs P, unsigned long long* F,
                                                                       double* eslot, int shared) {
    constexpr int IB = kPmeIBlock, JB = kPmeJBlock, W = kPmeDirectWaves, NT = 64 * W;
    static_assert(JB + W - 1 <= 64 * W, "a wave's j-atoms are looked over one per lane");
    __shared__ double4 sI[IB], sJ[JB];       // x, y, z, q sqrt(k_e); i-atoms shifted to the neighbour's image
    __shared__ double2 sIp[IB], sJp[JB];
    __shared__ int4 sIx[IB], sJx[JB];        // exclusion group, rank, row offset, atom and displacement class
    __shared__ uint32_t sIw[kPmeExWords][IB]; // first words of the i-atoms' exclusion rows
    __shared__ unsigned long long sIF[3][IB], sJF[3][JB];
    __shared__ uint32_t sQ[W][128];
    __shared__ double sE[W];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // the cell itself, its face, edge and corner neighbours: most pairs first
    constexpr unsigned long long order = 0xDB75CA86429310ull;
    const int nb = (int)((order >> (4 * blockIdx.z)) & 15ull), c = blockIdx.x;
    const int i0 = P.cellStart[c] + blockIdx.y * IB, ni = min(P.cellStart[c + 1] - i0, IB);
    const int blockSlot = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + c;
    if (ni <= 0) {  // no atom in this part of the cell
        if (threadIdx.x == 0) eslot[blockSlot] = 0.0;
        return;
    }
    const int cz = c % D.m[2], cy = (c / D.m[2]) % D.m[1], cx = c / (D.m[1] * D.m[2]);
    // forward offsets: (a, b, e) lexicographically above (0, 0, 0); nb = 0 is the cell itself
    int ox = 0, oy = 0, oz = 0;
    if (nb > 0) {
        const int f = nb + 13;  // 14..26 in the 3x3x3 numbering (a + 1) 9 + (b + 1) 3 + (e + 1)
        ox = f / 9 - 1; oy = (f / 3) % 3 - 1; oz = f % 3 - 1;
    }
    int nx = cx + ox, ny = cy + oy, nz = cz + oz;
    double sx = 0.0, sy = 0.0, sz = 0.0;  // image of the neighbour cell: x_j + s
    if (nx < 0) { nx += D.m[0]; sx = -D.L[0]; } else if (nx >= D.m[0]) { nx -= D.m[0]; sx = D.L[0]; }
    if (ny < 0) { ny += D.m[1]; sy = -D.L[1]; } else if (ny >= D.m[1]) { ny -= D.m[1]; sy = D.L[1]; }
    if (nz < 0) { nz += D.m[2]; sz = -D.L[2]; } else if (nz >= D.m[2]) { nz -= D.m[2]; sz = D.L[2]; }
    const int cn = (nx * D.m[1] + ny) * D.m[2] + nz;
    const int jend = P.cellStart[cn + 1];
    // in the cell itself only j slots above the block's first slot can pair with it
    const int jstart = nb == 0 ? i0 + 1 : P.cellStart[cn];
    for (int k = threadIdx.x; k < ni; k += NT) {
        double4 p = P.cpos[i0 + k];
        p.x -= sx; p.y -= sy; p.z -= sz;  // (x_i - s) - x_j = x_i - (x_j + s)
        sI[k] = p;
        sIp[k] = P.cprm[i0 + k];
        const int4 xk = P.cex[i0 + k];
        sIx[k] = xk;
#pragma unroll
        for (int w = 0; w < kPmeExWords; ++w) sIw[w][k] = P.exbits[xk.z + w];  // (padded past the last row)
        sIF[0][k] = 0ull; sIF[1][k] = 0ull; sIF[2][k] = 0ull;
    }
    const double rc2 = D.rc2;
    double e = 0.0;
    int head = 0, tail = 0;  // the wave's ring [head, tail) of pending pairs (wave-uniform)
    uint32_t* Q = sQ[wave];

    // evaluate `count` queued pairs, one per lane
    auto dense = [&](int count) __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < count) {
            const uint32_t code = Q[(head + lane) & 127];
            const int i = code >> 16, k = (int)(code & 0xFFFFu);
            const double4 p = sI[i];
            const double2 ip = sIp[i];
            const double4 pj = sJ[k];
            const double2 jp = sJp[k];
            const double dx = p.x - pj.x, dy = p.y - pj.y, dz = p.z - pj.z;
            const double r2 = dx * dx + dy * dy + dz * dz;
            double fs;
            e += direct_pair(D, r2, p.w * pj.w, ip.x + jp.x, ip.y * jp.y, fs);
            const double vx = fs * dx * kFix, vy = fs * dy * kFix, vz = fs * dz * kFix;
            const double mx = fmax(fabs(vx), fmax(fabs(vy), fabs(vz)));
            // the pairs of one j-atom sit in consecutive lanes (up to 64 of them: the adds to its
            // sums would queue on one address): an octet of one j-atom adds up first, exactly (whole
            // numbers below 2^48, whose sum whole() takes), and issues one add per component
            const int k0 = __shfl(k, lane & 56, 64);
            uint64_t oct = __ballot(k == k0 && mx < 281474976710656.0);
            oct &= oct >> 1; oct &= oct >> 2; oct &= oct >> 4;
            oct &= 0x0101010101010101ull;
            oct = (oct << 8) - oct;  // all 8 lanes of such octets
            double rx = rint(vx), ry = rint(vy), rz = rint(vz);
            const bool big = !(mx < 2251799813685248.0);
            const long long fx = big ? __double2ll_rn(vx) : whole(rx);
            const long long fy = big ? __double2ll_rn(vy) : whole(ry);
            const long long fz = big ? __double2ll_rn(vz) : whole(rz);
            lds_add(&sIF[0][i], (unsigned long long)fx);
            lds_add(&sIF[1][i], (unsigned long long)fy);
            lds_add(&sIF[2][i], (unsigned long long)fz);
            rx = oct_sum(rx); ry = oct_sum(ry); rz = oct_sum(rz);
            const bool full = __builtin_amdgcn_inverse_ballot_w64(oct);
            const bool idle = full && (lane & 7) != 0;
            const long long gx = idle ? 0ll : -(full ? whole(rx) : fx);
            const long long gy = idle ? 0ll : -(full ? whole(ry) : fy);
            const long long gz = idle ? 0ll : -(full ? whole(rz) : fz);
            if (gx != 0) lds_add(&sJF[0][k], (unsigned long long)gx);
            if (gy != 0) lds_add(&sJF[1][k], (unsigned long long)gy);
            if (gz != 0) lds_add(&sJF[2][k], (unsigned long long)gz);
        }
        head += count;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    for (int jb = jstart; jb < jend; jb += JB) {
        const int nj = min(JB, jend - jb);
        for (int k = threadIdx.x; k < nj; k += NT) {
            sJ[k] = P.cpos[jb + k];
            sJp[k] = P.cprm[jb + k];
            sJx[k] = P.cex[jb + k];
            sJF[0][k] = 0ull; sJF[1][k] = 0ull; sJF[2][k] = 0ull;
        }
        __syncthreads();
        const int ka = nj * wave / W, kb = nj * (wave + 1) / W;  // this wave's j-atoms
        for (int ic = 0; ic < ni; ic += 64) {
            const int cnt = min(64, ni - ic);
            const int lg = cnt > 32 ? 6 : (cnt > 16 ? 5 : (cnt > 8 ? 4 : 3)), G = 64 >> lg;
            const int il = lane & ((1 << lg) - 1), jg = lane >> lg;
            const bool active = il < cnt;
            const int i = ic + (active ? il : 0);
            const double px = sI[i].x, py = sI[i].y, pz = sI[i].z;
            const int4 xi = sIx[i];
            const uint64_t act = __ballot(active);
            const uint32_t codeI = (uint32_t)i << 16;
            const int jself = jb - (i0 + i);  // the cell itself: j slots above the i slot only
            const int clsI = xi.w >> kPmeClassShift;
            const bool mixed = shared && __ballot((active && clsI != 0) || (ka + lane < kb && sJx[ka + lane].w > kPmeAtomMask)) != 0ull;
            for (int k0 = ka; k0 < kb; k0 += G) {
                const int k = min(k0 + jg, kb - 1);
                const double dx = px - sJ[k].x, dy = py - sJ[k].y, dz = pz - sJ[k].z;
                const double r2 = dx * dx + dy * dy + dz * dz;
                uint64_t m = __ballot(r2 < rc2) & act;
                if (G > 1) m &= __ballot(k0 + jg < kb);
                if (nb == 0) m &= __ballot(jself + k > 0);
                if (mixed) m &= __ballot((sJx[k].w >> kPmeClassShift) == clsI);
                if (m == 0ull) continue;
                const uint64_t same = __ballot(sJx[k].x == xi.x) & m;
                if (same != 0ull) {  // atoms of one exclusion group: look the pairs up
                    bool ex = false;
                    if (__builtin_amdgcn_inverse_ballot_w64(same)) {
                        const int rank = sJx[k].y;
                        uint32_t bits = sIw[min(rank >> 5, kPmeExWords - 1)][i];
                        if (rank >= 32 * kPmeExWords) bits = P.exbits[xi.z + (rank >> 5)];
                        ex = (bits >> (rank & 31)) & 1u;
                    }
                    m &= ~__ballot(ex);
                }
                const int at = tail + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
                if (__builtin_amdgcn_inverse_ballot_w64(m)) Q[at & 127] = codeI | (uint32_t)k;
                tail += __popcll(m);
                if (tail - head >= 64) dense(64);
            }
        }
        if (tail > head) dense(tail - head);  // the staged j-atoms are replaced or flushed next
        __syncthreads();
        for (int k = threadIdx.x; k < nj; k += NT) {  // j forces of the batch
            const int atom = sJx[k].w & kPmeAtomMask;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const unsigned long long v = sJF[q][k];
                if (v) atomicAdd(F + (long long)q * D.n + atom, v);
            }
        }
        __syncthreads();
    }
    for (int k = threadIdx.x; k < ni; k += NT) {
        const int atom = sIx[k].w & kPmeAtomMask;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const unsigned long long v = sIF[q][k];
            if (v) atomicAdd(F + (long long)q * D.n + atom, v);
        }
    }
    e = wave_sum(e);
    if (lane == 0) sE[wave] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < W; ++w) e += sE[w];
        eslot[blockSlot] = e;
    }
}

// The pairs that d changes, at each state by themselves (the displaced atoms are few): one
// wave per (displaced atom k, neighbour cell, state): the pairs of atom k at that state
// with the cell's atoms that are not displaced; the first cell's wave also takes the
// displaced atoms after k that are displaced differently.  Energies and forces go to the
// state's own sums (per pair in fixed point, as k_pme_direct adds them), so nothing cancels:
// a pair that clashes at x, up to the last bit it has, leaves x + d alone.  (k_pme_direct with
// these pairs at x and this kernel taking them off again for x + d left 1e-16 of the clash in
// U2 and, past the fixed-point range of a force, thousands of kJ/mol/nm.)  10 us for the
// 21-atom ligand of an 8,479-atom system, where a second cell list and direct pass took 79;
// one wave per neighbour cell because a wave walking all 27 waits on memory 50 times in a row.
__global__ void __launch_bounds__(64) k_pme_displaced(PmeDesc D, PmePtrs P) {
    const int lane = threadIdx.x, cellOff = blockIdx.x >> 1, st = blockIdx.x & 1, k = blockIdx.y;
    const int a = P.lig[k];
    const double* X = st ? P.x2 : P.x;
    unsigned long long* F = P.F + 3ll * D.n * st;
    double w[3];
    const int c0 = wrap_cell(X[3 * a], D.L[0], D.invL[0], D.m[0], &w[0]);
    const int c1 = wrap_cell(X[3 * a + 1], D.L[1], D.invL[1], D.m[1], &w[1]);
    const int c2 = wrap_cell(X[3 * a + 2], D.L[2], D.invL[2], D.m[2], &w[2]);
    int nx = c0 + cellOff / 9 - 1, ny = c1 + (cellOff / 3) % 3 - 1, nz = c2 + cellOff % 3 - 1;
    double px = w[0], py = w[1], pz = w[2];  // the atom's image next to the neighbour cell
    if (nx < 0) { nx += D.m[0]; px += D.L[0]; } else if (nx >= D.m[0]) { nx -= D.m[0]; px -= D.L[0]; }
    if (ny < 0) { ny += D.m[1]; py += D.L[1]; } else if (ny >= D.m[1]) { ny -= D.m[1]; py -= D.L[1]; }
    if (nz < 0) { nz += D.m[2]; pz += D.L[2]; } else if (nz >= D.m[2]) { nz -= D.m[2]; pz -= D.L[2]; }
    const int cn = (nx * D.m[1] + ny) * D.m[2] + nz;
    const int4 xa = P.exkey[a];
    const double2 pa = P.prm2[a];
    const double qa = P.prm[a].x;
    double e = 0.0;
    unsigned long long fx = 0ull, fy = 0ull, fz = 0ull;
    auto pair = [&](int b, double dx, double dy, double dz, double r2, int grp, int rank, double qb, double2 pb) {
        if (grp == xa.x && ((P.exbits[xa.z + (rank >> 5)] >> (rank & 31)) & 1u)) return;
        double fs;
        e += direct_pair(D, r2, qa * qb, pa.x + pb.x, pa.y * pb.y, fs);
        const unsigned long long gx = fixed_force(fs * dx), gy = fixed_force(fs * dy), gz = fixed_force(fs * dz);
        fx += gx; fy += gy; fz += gz;
        atomicAdd(F + b, 0ull - gx);
        atomicAdd(F + D.n + b, 0ull - gy);
        atomicAdd(F + 2ll * D.n + b, 0ull - gz);
    };
    const int j0 = P.cellStart[cn], j1 = min(P.cellStart[cn + 1], j0 + kPmeCellMax);
    for (int j = j0 + lane; j < j1; j += 64) {
        const double4 pj = P.cpos[j];
        const double dx = px - pj.x, dy = py - pj.y, dz = pz - pj.z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (!(r2 < D.rc2)) continue;
        const int4 xj = P.cex[j];
        if (xj.w > kPmeAtomMask) continue;  // displaced itself: below
        pair(xj.w, dx, dy, dz, r2, xj.x, xj.y, pj.w, P.cprm[j]);
    }
    if (cellOff == 0)
        for (int q = k + 1 + lane; q < D.nlig; q += 64) {
            const int b = P.lig[q];
            const int4 xb = P.exkey[b];
            if (xb.w == xa.w) continue;  // displaced alike: in the shared sums
            double v[3];
            wrap_cell(X[3 * b], D.L[0], D.invL[0], D.m[0], &v[0]);
            wrap_cell(X[3 * b + 1], D.L[1], D.invL[1], D.m[1], &v[1]);
            wrap_cell(X[3 * b + 2], D.L[2], D.invL[2], D.m[2], &v[2]);
            double dx = w[0] - v[0], dy = w[1] - v[1], dz = w[2] - v[2];
            dx -= D.L[0] * rint(dx * D.invL[0]);
            dy -= D.L[1] * rint(dy * D.invL[1]);
            dz -= D.L[2] * rint(dz * D.invL[2]);
            const double r2 = dx * dx + dy * dy + dz * dz;
            if (!(r2 < D.rc2)) continue;
            pair(b, dx, dy, dz, r2, xb.x, xb.y, P.prm[b].x, P.prm2[b]);
        }
    e = wave_sum(e);
    fx = wave_sum(fx); fy = wave_sum(fy); fz = wave_sum(fz);
    if (lane == 0) {
        P.eslot[(long long)D.nslot * st + D.nslotPairs + 27 * k + cellOff] = e;
        if (fx != 0ull) atomicAdd(F + a, fx);
        if (fy != 0ull) atomicAdd(F + D.n + a, fy);
        if (fz != 0ull) atomicAdd(F + 2ll * D.n + a, fz);
    }
}

// One axis' place on the grid of a position: scaled coordinate u (grid index floor(u)).
// tiles: from the wrapped position, as the tile kernel spreads; otherwise as k_pme_spread.
__device__ __forceinline__ double grid_coord(const PmeDesc& D, double x, int d, bool tiles) {
    if (tiles) {
        double w;
        wrap_cell(x, D.L[d], D.invL[d], D.m[d], &w);
        return w * D.invL[d] * D.K[d];
    }
    return grid_fraction(x, D.invL[d]) * D.K[d];
}

// The displaced atoms' charges off the grid at x and onto it at x + d, into the
// difference grid: by the formulas of the spreading kernels, so that grid + difference is
// the grid of x + d.  One task per (atom, state, first B-spline index).
__device__ void spread_difference(const PmeDesc& D, const PmePtrs& P, int task) {
    const int a = task % kOrder, st = (task / kOrder) & 1, i = P.lig[task / (2 * kOrder)];
    const double q = P.prm[i].y;
    if (q == 0.0) return;
    const double* X = st ? P.x2 : P.x;
    double th[3][kOrder], dth[kOrder];
    int g0[3];
    for (int d = 0; d < 3; ++d) {
        const double u = grid_coord(D, X[3 * i + d], d, D.tileBytes > 0);
        g0[d] = (int)floor(u);
        bspline5(u - g0[d], th[d], dth);
    }
    unsigned long long* G = reinterpret_cast<unsigned long long*>(P.qgrid) + D.ngrid;
    const int ia = wrap_index(g0[0] - a, D.K[0]);
    for (int b = 0; b < kOrder; ++b) {
        const int ib = wrap_index(g0[1] - b, D.K[1]);
        const double qab = q * th[0][a] * th[1][b];
        for (int cc = 0; cc < kOrder; ++cc) {
            const int ic = wrap_index(g0[2] - cc, D.K[2]);
            const long long v = __double2ll_rn(qab * th[2][cc] * kGridFix);
            atomicAdd(G + ((long long)ia * D.K[1] + ib) * D.K[2] + ic, (unsigned long long)(st ? v : -v));
        }
    }
}

__global__ void k_pme_spread_difference(PmeDesc D, PmePtrs P) {
    const int task = blockIdx.x * blockDim.x + threadIdx.x;
    if (task < D.nlig * 2 * kOrder) spread_difference(D, P, task);
}

__global__ void k_pme_spread(PmeDesc D, PmePtrs P, const double* x, unsigned long long* grid) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D.n) return;
    const double q = P.prm[i].y;
    if (q == 0.0) return;
    double th[3][kOrder], dth[kOrder];
    int g0[3];
    for (int d = 0; d < 3; ++d) {
        const double u = grid_fraction(x[3 * i + d], D.invL[d]) * D.K[d];
        int g = (int)floor(u);
        const double w = u - g;
        g0[d] = g;
        bspline5(w, th[d], dth);
    }
    for (int a = 0; a < kOrder; ++a) {
        const int ia = ((g0[0] - a) % D.K[0] + D.K[0]) % D.K[0];
        for (int b = 0; b < kOrder; ++b) {
            const int ib = ((g0[1] - b) % D.K[1] + D.K[1]) % D.K[1];
            const double qab = q * th[0][a] * th[1][b];
            for (int cc = 0; cc < kOrder; ++cc) {
                const int ic = ((g0[2] - cc) % D.K[2] + D.K[2]) % D.K[2];
                atomicAdd(grid + ((long long)ia * D.K[1] + ib) * D.K[2] + ic,
                          (unsigned long long)__double2ll_rn(qab * th[2][cc] * kGridFix));
            }
        }
    }
}

// Charge at grid point k of a state, in fixed-point units.
__device__ __forceinline__ long long grid_charge(const PmeDesc& D, const long long* q, int state, int k) {
    return state == 0 ? q[k] : q[D.ngrid + k] + (D.delta ? q[k] : 0ll);
}

__global__ void k_pme_q2c(PmeDesc D, PmePtrs P) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= D.ngrid) return;
    const int st = blockIdx.y;
    P.g0[(long long)st * D.ngrid + k] = make_double2((double)grid_charge(D, P.qgrid, st, k) * (1.0 / kGridFix), 0.0);
}

// One axis of an unnormalised complex DFT: out[..k..] = sum_j in[..j..] e^{sign 2 pi i j k / K}.
__global__ void k_pme_dft(PmeDesc D, const double2* in, double2* out, const double2* tw, int axis, double sign) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= D.ngrid) return;
    in += (long long)blockIdx.y * D.ngrid;  // blockIdx.y: state
    out += (long long)blockIdx.y * D.ngrid;
    const int K = D.K[axis];
    const int stride = axis == 2 ? 1 : (axis == 1 ? D.K[2] : D.K[1] * D.K[2]);
    const int k = (idx / stride) % K;
    const int base = idx - k * stride;
    double re = 0.0, im = 0.0;
    int t = 0;
    for (int j = 0; j < K; ++j) {
        const double2 v = in[base + j * stride];
        const double2 w = tw[t];
        const double s = sign * w.y;
        re += v.x * w.x - v.y * s;
        im += v.y * w.x + v.x * s;
        t += k;
        if (t >= K) t -= K;
    }
    out[idx] = make_double2(re, im);
}

// One wave per grid line along `axis` (four lines per block): the line and the
// axis' twiddles are staged in LDS, then lane k (k + 64, ...) forms output k.
// Dynamic LDS: 5 K complex values.
// qfix: when not null, the input is the fixed-point charge grid (real), read in
// place of `in` (the first forward pass needs no separate conversion kernel).
__global__ void __launch_bounds__(256) k_pme_dft_lines(PmeDesc D, const double2* in, double2* out, const double2* tw,
                                                      int axis, double sign, const long long* qfix) {
    extern __shared__ double2 sm[];
    in += (long long)blockIdx.y * D.ngrid;  // blockIdx.y: state
    out += (long long)blockIdx.y * D.ngrid;
    const int K = D.K[axis];
    const int stride = axis == 2 ? 1 : (axis == 1 ? D.K[2] : D.K[1] * D.K[2]);
    const int nlines = D.ngrid / K;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double2* stw = sm;
    double2* line = sm + K + w * K;
    for (int t = threadIdx.x; t < K; t += 256) stw[t] = tw[t];
    const int L = blockIdx.x * 4 + w;
    int base = 0;
    if (L < nlines) {
        base = (L / stride) * K * stride + L % stride;
        if (qfix)
            for (int j = lane; j < K; j += 64) 
                line[j] = make_double2((double)grid_charge(D, qfix, blockIdx.y, base + j * stride) * (1.0 / kGridFix), 0.0);
        else
            for (int j = lane; j < K; j += 64) line[j] = in[base + j * stride];
    }
    __syncthreads();
    if (L >= nlines) return;
    for (int k = lane; k < K; k += 64) {
        double re = 0.0, im = 0.0;
        int t = 0;
        for (int j = 0; j < K; ++j) {
            const double2 v = line[j];
            const double2 c = stw[t];
            const double sn = sign * c.y;
            re += v.x * c.x - v.y * sn;
            im += v.y * c.x + v.x * sn;
            t += k;
            if (t >= K) t -= K;
        }
        out[base + k * stride] = make_double2(re, im);
    }
}

// Charge spreading of one cell's atoms into an LDS tile of the grid (64-bit
// fixed point, integer LDS atomics), then one global atomic per nonzero tile
// point.  The tile covers grid indices [o, o + T) per axis with
// o = floor(c K / m) - 5 and T = D.tile[axis]; a point outside it (rounding at
// the cell edge) goes straight to the global grid.
__global__ void __launch_bounds__(256) k_pme_spread_tiles(PmeDesc D, PmePtrs P, unsigned long long* grid) {
    extern __shared__ unsigned long long tile[];
    if ((int)blockIdx.x >= D.ncell * kPmeSpreadSplit) {  // the last blocks: the displaced atoms
        const int task = ((int)blockIdx.x - D.ncell * kPmeSpreadSplit) * 256 + threadIdx.x;
        if (task < D.nlig * 2 * kOrder) spread_difference(D, P, task);
        return;
    }
    // block (c, part): part `part` of kPmeSpreadSplit contiguous parts of cell c's atoms
    const int c = blockIdx.x / kPmeSpreadSplit, part = blockIdx.x % kPmeSpreadSplit;
    const int cz = c % D.m[2], cy = (c / D.m[2]) % D.m[1], cx = c / (D.m[1] * D.m[2]);
    const int o[3] = {(cx * D.K[0]) / D.m[0] - 5, (cy * D.K[1]) / D.m[1] - 5, (cz * D.K[2]) / D.m[2] - 5};
    const int T0 = D.tile[0], T1 = D.tile[1], T2 = D.tile[2], TT = T0 * T1 * T2;
    for (int k = threadIdx.x; k < TT; k += 256) tile[k] = 0ull;
    __syncthreads();
    const int cs = P.cellStart[c], call = min(P.cellStart[c + 1] - cs, D.cellCap);
    const int s0 = cs + (call * part) / kPmeSpreadSplit, cnt = cs + (call * (part + 1)) / kPmeSpreadSplit - s0;
    // task = (atom, first B-spline index a): 25 points each
    for (int task = threadIdx.x; task < cnt * kOrder; task += 256) {
        const int sl = s0 + task / kOrder, a = task % kOrder;
        const double4 p = P.cpos[sl];
        const double q = P.prm[P.cex[sl].w & kPmeAtomMask].y;
        if (q == 0.0) continue;
        double th[3][kOrder], dth[kOrder];
        int g0[3];
        const double pv[3] = {p.x, p.y, p.z};
        for (int d = 0; d < 3; ++d) {
            const double u = pv[d] * D.invL[d] * D.K[d];
            const int g = (int)floor(u);
            g0[d] = g;
            bspline5(u - g, th[d], dth);
        }
        const int la = g0[0] - a - o[0];
        for (int b = 0; b < kOrder; ++b) {
            const int lb = g0[1] - b - o[1];
            const double qab = q * th[0][a] * th[1][b];
            for (int cc = 0; cc < kOrder; ++cc) {
                const int lc = g0[2] - cc - o[2];
                const unsigned long long v = (unsigned long long)__double2ll_rn(qab * th[2][cc] * kGridFix);
                if (la >= 0 && la < T0 && lb >= 0 && lb < T1 && lc >= 0 && lc < T2) {
                    atomicAdd(&tile[(la * T1 + lb) * T2 + lc], v);
                } else {
                    const int ia = wrap_index(g0[0] - a, D.K[0]);
                    const int ib = wrap_index(g0[1] - b, D.K[1]);
                    const int ic = wrap_index(g0[2] - cc, D.K[2]);
                    atomicAdd(grid + ((long long)ia * D.K[1] + ib) * D.K[2] + ic, v);
                }
            }
        }
    }
    __syncthreads();
    // tile index o + l lies in [-5, K + 3): one wrap per axis
    for (int k = threadIdx.x; k < TT; k += 256) {
        const unsigned long long v = tile[k];
        if (v == 0ull) continue;
        const int lc = k % T2, lb = (k / T2) % T1, la = k / (T1 * T2);
        const int ia = wrap_index(o[0] + la, D.K[0]);
        const int ib = wrap_index(o[1] + lb, D.K[1]);
        const int ic = wrap_index(o[2] + lc, D.K[2]);
        atomicAdd(grid + ((long long)ia * D.K[1] + ib) * D.K[2] + ic, v);
    }
}

// The influence function at frequency indices (a, b, c): exp(-pi^2 m^2 / alpha^2) / (m^2 B),
// 0 at m = 0.
__device__ __forceinline__ double influence(const PmeDesc& D, const PmePtrs& P, int a, int b, int c) {
    const double mx = (a <= D.K[0] / 2 ? a : a - D.K[0]) * D.invL[0];
    const double my = (b <= D.K[1] / 2 ? b : b - D.K[1]) * D.invL[1];
    const double mz = (c <= D.K[2] / 2 ? c : c - D.K[2]) * D.invL[2];
    const double m2 = mx * mx + my * my + mz * mz;
    if ((a | b | c) == 0) return 0.0;
    const double B = P.bmod[a] * P.bmod[D.K[0] + b] * P.bmod[D.K[0] + D.K[1] + c];
    return exp(-D.pi2OverAlpha2 * m2) / (m2 * B);
}

__global__ void __launch_bounds__(256) k_pme_convolve(PmeDesc D, PmePtrs P, double2* g, double* eslot) {
    __shared__ double red[4];
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    g += (long long)blockIdx.y * D.ngrid;  // blockIdx.y: state
    eslot += (long long)blockIdx.y * D.nslot;
    double e = 0.0;
    if (idx < D.ngrid) {
        const int c = idx % D.K[2], b = (idx / D.K[2]) % D.K[1], a = idx / (D.K[1] * D.K[2]);
        const double w = influence(D, P, a, b, c);
        const double2 f = g[idx];
        e = w * (f.x * f.x + f.y * f.y);
        g[idx] = make_double2(w * f.x, w * f.y);
    }
    const double s = block_sum<256>(e, red);
    if (threadIdx.x == 0) eslot[blockIdx.x] = s * D.recipEnergyScale;
}

// ------------------------------------------------ fused transforms
// A length-K axis, K = A B, is transformed in two short steps over an array in LDS
// (positions `as` elements apart), in place: with n = B n1 + n2 and k = k1 + A k2,
//   y[k1, n2] = W_K^{n2 k1} sum_{n1} x[B n1 + n2] W_K^{B n1 k1}   (at position B k1 + n2)
//   X[k1, k2] =             sum_{n2} y[k1, n2]    W_K^{A n2 k2}   (at position B k1 + k2)
// and backwards the same two steps in reverse order with conjugate twiddles, so
// frequency k1 + A k2 sits at position B k1 + k2 between the two transforms and no
// reordering pass is needed.  Each output costs A or B products instead of K.  Results
// wait in registers while the block still reads the inputs.
// Three launches for both states instead of seven per state (35 x 40 x 35: 34 us instead
// of 70, 105 x 40 x 35: 44 instead of 90); what is left is LDS reads (two 16-byte reads
// per product) and launches that fill a quarter of the chip.
__device__ __forceinline__ int div_small(int v, float inv) { return (int)(((float)v + 0.5f) * inv); }

// stepA: sums over n1 (or k1); otherwise over n2 (or k2).  twiddle: times W_K^{n2 k1}.
__device__ __forceinline__ void dft_step(double2* buf, const double2* tw, int total, int K, int A, int as, bool stepA,
                                         bool twiddle, double sign) {
    const int B = K / A;
    const float invAs = 1.0f / as, invK = 1.0f / K, invB = 1.0f / B;
    double2 out[kPmeFuseMax / kPmeFuseNT];
#pragma unroll
    for (int u = 0; u < kPmeFuseMax / kPmeFuseNT; ++u) {
        const int e = threadIdx.x + u * kPmeFuseNT;
        if (e < total) {
            const int row = div_small(e, invAs);
            const int pos = row - div_small(row, invK) * K;
            const int hi = div_small(pos, invB), lo = pos - hi * B;  // position B hi + lo
            // summed positions: stepA B n + lo (n < A), else B hi + n (n < B)
            const double2* v = buf + e - (stepA ? hi * B : lo) * as;
            const int R = stepA ? A : B, es = stepA ? B * as : as, dt = stepA ? B * hi : A * lo;
            double re = 0.0, im = 0.0;
            int t = 0;
            for (int n = 0; n < R; ++n) {
                const double2 x = v[n * es], c = tw[t];
                const double sn = sign * c.y;
                re += x.x * c.x - x.y * sn;
                im += x.y * c.x + x.x * sn;
                t += dt;
                if (t >= K) t -= K;
            }
            if (twiddle) {
                const double2 c = tw[hi * lo];  // hi < A, lo < B: below K
                const double sn = sign * c.y, r2 = re * c.x - im * sn;
                im = im * c.x + re * sn;
                re = r2;
            }
            out[u] = make_double2(re, im);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPmeFuseMax / kPmeFuseNT; ++u) {
        const int e = threadIdx.x + u * kPmeFuseNT;
        if (e < total) buf[e] = out[u];
    }
    __syncthreads();
}

__device__ __forceinline__ void dft_axis(double2* buf, const double2* tw, int total, int K, int A, int as, bool forward) {
    if (forward) {
        if (A > 1) dft_step(buf, tw, total, K, A, as, true, true, -1.0);
        dft_step(buf, tw, total, K, A, as, false, false, -1.0);
    } else {
        dft_step(buf, tw, total, K, A, as, false, A > 1, 1.0);
        if (A > 1) dft_step(buf, tw, total, K, A, as, true, false, 1.0);
    }
}

// Axis strides of the grid arrays.
__device__ __forceinline__ int axis_stride(const PmeDesc& D, int ax) {
    return ax == 2 ? 1 : (ax == 1 ? D.K[2] : D.K[1] * D.K[2]);
}

// One plane (axes pAx, qAx) at position blockIdx.x of the line axis, state blockIdx.y, in LDS.
// FORWARD: from the fixed-point charges to g0; otherwise from g0 to the real potential.
template <bool FORWARD>
__global__ void __launch_bounds__(kPmeFuseNT) k_pme_planes(PmeDesc D, PmePtrs P) {
    extern __shared__ double2 sm[];
    const int Kp = D.K[D.pAx], Kq = D.K[D.qAx], total = Kp * Kq, st = blockIdx.y;
    double2 *twp = sm + total, *twq = twp + Kp;
    for (int t = threadIdx.x; t < Kp; t += kPmeFuseNT) twp[t] = P.tw[D.twOff[D.pAx] + t];
    for (int t = threadIdx.x; t < Kq; t += kPmeFuseNT) twq[t] = P.tw[D.twOff[D.qAx] + t];
    const int sP = axis_stride(D, D.pAx), sQ = axis_stride(D, D.qAx);
    const int base = blockIdx.x * axis_stride(D, D.lineAx);
    const float invKq = 1.0f / Kq;
    double2* g = P.g0 + (long long)st * D.ngrid;
    for (int e = threadIdx.x; e < total; e += kPmeFuseNT) {
        const int p = div_small(e, invKq), at = base + p * sP + (e - p * Kq) * sQ;
        sm[e] = FORWARD ? make_double2((double)grid_charge(D, P.qgrid, st, at) * (1.0 / kGridFix), 0.0) : g[at];
    }
    __syncthreads();
    dft_axis(sm, twq, total, Kq, D.fA[D.qAx], 1, FORWARD);
    dft_axis(sm, twp, total, Kp, D.fA[D.pAx], Kq, FORWARD);
    double* phi = reinterpret_cast<double*>(P.g1) + (long long)st * D.ngrid;
    for (int e = threadIdx.x; e < total; e += kPmeFuseNT) {
        const int p = div_small(e, invKq), at = base + p * sP + (e - p * Kq) * sQ;
        if (FORWARD) g[at] = sm[e]; else phi[at] = sm[e].x;
    }
}

// lineTile lines along the line axis (blockIdx.x), state blockIdx.y: forward transform,
// convolution with the influence function (reciprocal energy into the block's slot),
// backward transform.
__global__ void __launch_bounds__(kPmeFuseNT) k_pme_lines(PmeDesc D, PmePtrs P, double* eslot) {
    extern __shared__ double2 sm[];
    __shared__ double red[kPmeFuseNT / 64];
    const int K = D.K[D.lineAx], T = D.lineTile, Kq = D.K[D.qAx], nl = D.K[D.pAx] * Kq, st = blockIdx.y;
    double2* tw = sm + K * T;
    for (int t = threadIdx.x; t < K; t += kPmeFuseNT) tw[t] = P.tw[D.twOff[D.lineAx] + t];
    const int sL = axis_stride(D, D.lineAx), sP = axis_stride(D, D.pAx), sQ = axis_stride(D, D.qAx);
    const float invT = 1.0f / T, invKq = 1.0f / Kq;
    double2* g = P.g0 + (long long)st * D.ngrid;
    const int l0 = blockIdx.x * T, total = K * T;
    for (int e = threadIdx.x; e < total; e += kPmeFuseNT) {
        const int pos = div_small(e, invT), l = l0 + e - pos * T;
        const int p = l / Kq;
        sm[e] = l < nl ? g[p * sP + (l - p * Kq) * sQ + pos * sL] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const int A = D.fA[D.lineAx];
    dft_axis(sm, tw, total, K, A, T, true);
    // the frequency at position B hi + lo is hi + A lo
    auto freq = [&](int ax, int pos) {
        const int a = D.fA[ax], b = D.K[ax] / a;
        return pos / b + a * (pos % b);
    };
    double e0 = 0.0;
    for (int e = threadIdx.x; e < total; e += kPmeFuseNT) {
        const int pos = div_small(e, invT), l = l0 + e - pos * T;
        if (l < nl) {
            const int p = div_small(l, invKq);
            int f[3];
            const int fl = freq(D.lineAx, pos), fp = freq(D.pAx, p), fq = freq(D.qAx, l - p * Kq);
            f[0] = D.lineAx == 0 ? fl : (D.pAx == 0 ? fp : fq);
            f[1] = D.lineAx == 1 ? fl : (D.pAx == 1 ? fp : fq);
            f[2] = D.lineAx == 2 ? fl : (D.pAx == 2 ? fp : fq);
            const double w = influence(D, P, f[0], f[1], f[2]);
            const double2 v = sm[e];
            e0 += w * (v.x * v.x + v.y * v.y);
            sm[e] = make_double2(w * v.x, w * v.y);
        }
    }
    const double s = block_sum<kPmeFuseNT>(e0, red);  // (its barriers also order the products above)
    if (threadIdx.x == 0) eslot[(long long)st * D.nslot + blockIdx.x] = s * D.recipEnergyScale;
    dft_axis(sm, tw, total, K, A, T, false);
    for (int e = threadIdx.x; e < total; e += kPmeFuseNT) {
        const int pos = div_small(e, invT), l = l0 + e - pos * T;
        const int p = l / Kq;
        if (l < nl) g[p * sP + (l - p * Kq) * sQ + pos * sL] = sm[e];
    }
}

// Reciprocal forces, 8 lanes per atom: lane a < 5 of the octet sums the 25 grid
// points of B-spline index a, then the octet adds its partial gradients
// (xor shuffles 1, 2, 4; lanes 5-7 add zeros).  Eight atoms per wave.
// phi: the potentials of the states, ps doubles apart per point (1: real, 2: complex).
__device__ __forceinline__ void gather_forces(const PmeDesc& D, const PmePtrs& P, const double* x, const double* phi,
                                              int ps, unsigned long long* F) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = t >> 3, a = t & 7;
    const bool on = i < D.n;
    const double q = on ? P.prm[i].y : 0.0;
    double gx = 0.0, gy = 0.0, gz = 0.0;
    if (on && q != 0.0 && a < kOrder) {
        double th[3][kOrder], dth[3][kOrder];
        int g0[3];
        for (int d = 0; d < 3; ++d) {
            const double u = grid_fraction(x[3 * i + d], D.invL[d]) * D.K[d];
            const int g = (int)floor(u);
            g0[d] = g;
            bspline5(u - g, th[d], dth[d]);
        }
        int ic[kOrder];  // g0 in [0, K]: g0 - k in [-4, K]
#pragma unroll
        for (int cc = 0; cc < kOrder; ++cc) ic[cc] = wrap_index(g0[2] - cc, D.K[2]);
        // th[0][a], dth[0][a] with a run-time a: select from the unrolled values
        double t0 = th[0][0], dt0 = dth[0][0];
#pragma unroll
        for (int k = 1; k < kOrder; ++k)
            if (a == k) { t0 = th[0][k]; dt0 = dth[0][k]; }
        const int ia = wrap_index(g0[0] - a, D.K[0]);
#pragma unroll
        for (int b = 0; b < kOrder; ++b) {
            const int ib = wrap_index(g0[1] - b, D.K[1]);
            const long long row = ((long long)ia * D.K[1] + ib) * D.K[2];
#pragma unroll
            for (int cc = 0; cc < kOrder; ++cc) {
                const double p = phi[(row + ic[cc]) * ps];
                gx += dt0 * th[1][b] * th[2][cc] * p;
                gy += t0 * dth[1][b] * th[2][cc] * p;
                gz += t0 * th[1][b] * dth[2][cc] * p;
            }
        }
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        gx += __shfl_xor(gx, o, 64);
        gy += __shfl_xor(gy, o, 64);
        gz += __shfl_xor(gz, o, 64);
    }
    if (on && q != 0.0 && a < 3) {
        const double s = -q * D.recipPhiScale;
        const double g = a == 0 ? gx * D.K[0] * D.invL[0] : (a == 1 ? gy * D.K[1] * D.invL[1] : gz * D.K[2] * D.invL[2]);
        add_fixed(F + (long long)a * D.n + i, s * g);
    }
}

// Exception pairs, one per thread of block `blk`.
__device__ __forceinline__ void exception_pairs(const PmeDesc& D, const PmePtrs& P, const double* x, int blk,
                                                unsigned long long* F, double* eslot) {
    __shared__ double red[4];
    const int k = blk * 256 + threadIdx.x;
    double e = 0.0;
    if (k < D.nex) {
        const int2 pr = P.expairs[k];
        const double4 ep = P.exprm[k];  // (k_e qq', sigma', 4 eps', k_e q_i q_j)
        const double dx = x[3 * pr.x] - x[3 * pr.y];
        const double dy = x[3 * pr.x + 1] - x[3 * pr.y + 1];
        const double dz = x[3 * pr.x + 2] - x[3 * pr.y + 2];
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double rinv = 1.0 / sqrt(r2), r = r2 * rinv, r2inv = rinv * rinv;
        double fs = 0.0;
        if (ep.x != 0.0) { e += ep.x * rinv; fs += ep.x * rinv * r2inv; }
        if (ep.z != 0.0) {
            const double s2 = ep.y * ep.y * r2inv, s6 = s2 * s2 * s2;
            e += ep.z * (s6 * s6 - s6);
            fs += ep.z * (12.0 * s6 * s6 - 6.0 * s6) * r2inv;
        }
        if (ep.w != 0.0) {
            const double ar = D.alpha * r;
            const double ec = ep.w * erf(ar) * rinv;
            e -= ec;
            fs -= (ec - ep.w * D.twoAlphaSqrtPi * exp(-ar * ar)) * r2inv;
        }
        if (fs != 0.0) {
            add_fixed(F + pr.x, fs * dx); add_fixed(F + D.n + pr.x, fs * dy); add_fixed(F + 2 * D.n + pr.x, fs * dz);
            add_fixed(F + pr.y, -fs * dx); add_fixed(F + D.n + pr.y, -fs * dy); add_fixed(F + 2 * D.n + pr.y, -fs * dz);
        }
    }
    const double s = block_sum<256>(e, red);
    if (threadIdx.x == 0) eslot[blk] = s;
}

// Reciprocal forces (the first gatherBlocks blocks) and exception pairs of state blockIdx.y.
__global__ void __launch_bounds__(256) k_pme_gather(PmeDesc D, PmePtrs P, const double* phi, int ps, int gatherBlocks) {
    const int st = blockIdx.y;
    const double* x = st ? P.x2 : P.x;
    unsigned long long* F = P.F + 3ll * D.n * st;
    if ((int)blockIdx.x < gatherBlocks)
        gather_forces(D, P, x, phi + (long long)st * D.ngrid * ps, ps, F);
    else
        exception_pairs(D, P, x, (int)blockIdx.x - gatherBlocks, F, P.eslot + (long long)st * D.nslot + D.nslotDirect);
}

// Fixed-order sums of the energy slots of both states; U = sum + constants;
// combine.  parts[s][0..4]: direct, exceptions, reciprocal, self, dispersion.
// single: state 0 only (W = U1, hybrid weight 0).
__global__ void __launch_bounds__(1024) k_pme_finish(PmeDesc D, PmePtrs P, int single) {
    __shared__ double red[16];
    double U[2] = {0.0, 0.0};
    auto sum = [&](const double* sl, int first, int last) {
        // four independent partial sums per thread (fixed order): their loads overlap
        double v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
        int k = first + (int)threadIdx.x;
        for (; k + 3 * 1024 < last; k += 4 * 1024) {
            v0 += sl[k];
            v1 += sl[k + 1024];
            v2 += sl[k + 2 * 1024];
            v3 += sl[k + 3 * 1024];
        }
        for (; k < last; k += 1024) v0 += sl[k];
        return block_sum<1024>((v0 + v1) + (v2 + v3), red);
    };
    const bool own = D.delta && !single;  // the pairs of both states in state 0's slots, then each state's own
    const double shared = own ? sum(P.eslot, 0, D.nslotPairs) : 0.0;
    for (int s = 0; s < (single ? 1 : 2); ++s) {
        const double* sl = P.eslot + (long long)s * D.nslot;
        double parts[3];
        parts[0] = own ? shared + sum(sl, D.nslotPairs, D.nslotDirect) : sum(sl, 0, D.nslotPairs);
        parts[1] = sum(sl, D.nslotDirect, D.nslotDirect + D.nslotEx);
        parts[2] = sum(sl, D.nslotDirect + D.nslotEx, D.nslot);
        if (threadIdx.x == 0) {
            P.parts[5 * s + 0] = parts[0];
            P.parts[5 * s + 1] = parts[1];
            P.parts[5 * s + 2] = parts[2];
            P.parts[5 * s + 3] = D.selfEnergy;
            P.parts[5 * s + 4] = D.dispersionEnergy;
            U[s] = parts[0] + parts[1] + parts[2] + D.selfEnergy + D.dispersionEnergy + (P.eoff && !single ? P.eoff[s] : 0.0);
        }
    }
    if (threadIdx.x == 0) {
        SysResult r;
        if (single) {
            r.W = U[0]; r.usc = 0.0; r.U1 = U[0]; r.U2 = 0.0; r.u = 0.0; r.fp = 1.0; r.bfp = 0.0; r.sp = 0.0;
        } else {
            atm_combine(*P.params, U[0], U[1], r);
        }
        *P.result = r;
        PmeHostRecord& h = *P.record;
        h.result = r;
        for (int k = 0; k < 10; ++k) h.parts[k] = P.parts[k];
        h.overflow = *P.overflow;
    }
}

// Writes straight to the host's page-locked memory, consecutive lanes consecutive doubles;
// with the inputs' copy in k_pme_begin and the record of k_pme_finish this replaces two copies in
// and four out, 274 -> 208 us (8k atoms) and 435 -> 360 us (25k).
__global__ void k_pme_blend(PmeDesc D, PmePtrs P, int single) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= 3 * D.n) return;
    const int i = j / 3, k = (j - 3 * i) * D.n + i;  // the sums are SoA
    const SysResult r = *P.result;
    const double a = single ? 0.0 : (P.params->direction > 0.0 ? r.sp : 1.0 - r.sp);  // weight of state 2 (x + d)
    const unsigned long long both = P.F[6ll * D.n + k];
    const double f1 = (double)(long long)(P.F[k] + both) * (1.0 / kFix);
    const double f2 = single ? 0.0 : (double)(long long)(P.F[3ll * D.n + k] + both) * (1.0 / kFix);
    P.hostF[j] = (1.0 - a) * f1 + a * f2;
}

__global__ void k_pme_fill(unsigned long long* p, long long n) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = 0ull;
}

// The first kernel of an evaluation: its inputs from the host's page-locked memory and three
// buffers and the overflow flag cleared by one launch (each launch of a graph costs a few us).
// Thread k copies word k of the inputs (first: they arrive while the rest is cleared) or
// clears one of the concatenation a | b | c.
__global__ void k_pme_begin(PmePtrs P, long long nin, unsigned long long* a, long long na, unsigned long long* b,
                            long long nb, unsigned long long* c, long long nc) {
    long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) *P.overflow = 0;
    if (k < nin) { P.in[k] = P.hostIn[k]; return; }
    k -= nin;
    if (k < na) { a[k] = 0ull; return; }
    k -= na;
    if (k < nb) { b[k] = 0ull; return; }
    k -= nb;
    if (k < nc) c[k] = 0ull;
}

static inline unsigned blocks_of(long long n, int t) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_pme_fill(unsigned long long* p, long long n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_pme_fill<<<blocks_of(n, 256), 256, 0, st>>>(p, n);
    return hipGetLastError();
}

hipError_t launch_pme_states(const PmeDesc& D, const PmePtrs& P, bool single, hipStream_t st) {
    const int ns = single ? 1 : 2;
    unsigned long long* q0 = reinterpret_cast<unsigned long long*>(P.qgrid);
    const bool delta = D.delta && !single;
    // cell list of the positions of `state`, its direct space into F
    auto cells = [&](int state, bool first) {
        if (first) {
            const long long nin = kPmeInHead + 3ll * D.n, nc = (D.ncell + 1) / 2, ng = (long long)ns * D.ngrid, nf = 9ll * D.n;
            k_pme_begin<<<blocks_of(nin + nc + ng + nf, 256), 256, 0, st>>>(
                P, nin, reinterpret_cast<unsigned long long*>(P.cellCount), nc, q0, ng, P.F, nf);
        } else {
            launch_pme_fill(reinterpret_cast<unsigned long long*>(P.cellCount), (D.ncell + 1) / 2, st);
        }
        // 256 threads: the histogram loops assume it; the first call forms x + d
        k_pme_bin<<<blocks_of(D.n, 256), 256, 0, st>>>(D, P, P.x, single ? nullptr : P.displ, state);
        k_pme_scan<<<1, 1024, 0, st>>>(D, P);
        k_pme_scatter<<<blocks_of(D.n, 256), 256, 0, st>>>(D, P);
        k_pme_cellsort<<<D.ncell, 256, 0, st>>>(D, P);
    };
    auto spread = [&](int state) {
        unsigned long long* grid = q0 + (long long)state * D.ngrid;
        const unsigned lb = delta && state == 0 ? blocks_of((long long)D.nlig * 2 * kOrder, 256) : 0u;
        if (D.tileBytes > 0) {  // the cell's grid tile fits in LDS
            k_pme_spread_tiles<<<D.ncell * kPmeSpreadSplit + lb, 256, D.tileBytes, st>>>(D, P, grid);
        } else {
            k_pme_spread<<<blocks_of(D.n, 256), 256, 0, st>>>(D, P, state ? P.x2 : P.x, grid);
            if (lb) k_pme_spread_difference<<<lb, 256, 0, st>>>(D, P);
        }
    };
    // cell fastest, neighbour slowest and the fullest first (the cell itself holds three times
    // the pairs of an edge neighbour): the launch ends on the short blocks
    const dim3 gridDirect(D.ncell, D.chunks, kPmeHalfShell);
    cells(0, true);
    k_pme_direct<<<gridDirect, 64 * kPmeDirectWaves, 0, st>>>(D, P, delta ? P.F + 6ll * D.n : P.F, P.eslot, delta ? 1 : 0);
    spread(0);
    if (delta) {
        if (D.nlig > 0) k_pme_displaced<<<dim3(54, D.nlig), 64, 0, st>>>(D, P);
    } else if (!single) {
        cells(1, false);
        k_pme_direct<<<gridDirect, 64 * kPmeDirectWaves, 0, st>>>(D, P, P.F + 3ll * D.n, P.eslot + D.nslot, 0);
        spread(1);
    }
    const unsigned gatherBlocks = blocks_of(8ll * D.n, 256);
    const dim3 gridGather(gatherBlocks + D.nslotEx, ns);
    double* erec = P.eslot + D.nslotDirect + D.nslotEx;
    if (D.fused) {
        const int Kp = D.K[D.pAx], Kq = D.K[D.qAx], Kl = D.K[D.lineAx];
        const size_t ldsPlane = (size_t)(Kp * Kq + Kp + Kq) * sizeof(double2);
        k_pme_planes<true><<<dim3(Kl, ns), kPmeFuseNT, ldsPlane, st>>>(D, P);
        k_pme_lines<<<dim3(D.lineBlocks, ns), kPmeFuseNT, (size_t)(D.lineTile + 1) * Kl * sizeof(double2), st>>>(D, P, erec);
        k_pme_planes<false><<<dim3(Kl, ns), kPmeFuseNT, ldsPlane, st>>>(D, P);
        k_pme_gather<<<gridGather, 256, 0, st>>>(D, P, reinterpret_cast<const double*>(P.g1), 1, gatherBlocks);
        return hipGetLastError();
    }
    const unsigned gb = blocks_of(D.ngrid, 256);
    auto dft = [&](const double2* in, double2* out, int axis, double sign, const long long* qfix = nullptr) {
        const int K = D.K[axis];
        if (K <= kPmeDftLdsMax) {
            k_pme_dft_lines<<<dim3(blocks_of(D.ngrid / K, 4), ns), 256, 5 * K * sizeof(double2), st>>>(
                D, in, out, P.tw + D.twOff[axis], axis, sign, qfix);
        } else {
            if (qfix) k_pme_q2c<<<dim3(gb, ns), 256, 0, st>>>(D, P);  // into g0 = in
            k_pme_dft<<<dim3(gb, ns), 256, 0, st>>>(D, in, out, P.tw + D.twOff[axis], axis, sign);
        }
    };
    // first pass straight from the fixed-point charge grid
    dft(P.g0, P.g1, 2, -1.0, P.qgrid);
    dft(P.g1, P.g0, 1, -1.0);
    dft(P.g0, P.g1, 0, -1.0);
    k_pme_convolve<<<dim3(gb, ns), 256, 0, st>>>(D, P, P.g1, erec);
    dft(P.g1, P.g0, 0, 1.0);
    dft(P.g0, P.g1, 1, 1.0);
    dft(P.g1, P.g0, 2, 1.0);
    k_pme_gather<<<gridGather, 256, 0, st>>>(D, P, reinterpret_cast<const double*>(P.g0), 2, gatherBlocks);
    return hipGetLastError();
}

hipError_t launch_pme_finish(const PmeDesc& D, const PmePtrs& P, bool single, bool forces, hipStream_t st) {
    k_pme_finish<<<1, 1024, 0, st>>>(D, P, single ? 1 : 0);
    if (forces) k_pme_blend<<<blocks_of(3ll * D.n, 256), 256, 0, st>>>(D, P, single ? 1 : 0);
    return hipGetLastError();
}

// ------------------------------------------------------------------ bonded terms
// HarmonicBondForce, HarmonicAngleForce and PeriodicTorsionForce of the
// system's group 0 (the AMBER terms test_abfe.py keeps beside the ATM force).

__global__ void __launch_bounds__(256) k_bonded(BondedPtrs B, double* eslot) {
    __shared__ double red[4];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    double eb = 0.0, ea = 0.0, et = 0.0;
    const double* x = B.x;
    auto diff = [&](int i, int j, double d[3]) {
        for (int c = 0; c < 3; ++c) d[c] = x[3 * i + c] - x[3 * j + c];
    };
    auto addf = [&](int i, double s, const double d[3]) {
        for (int c = 0; c < 3; ++c) add_fixed(B.F + 3ll * i + c, s * d[c]);
    };
    if (k < B.nb) {
        const int2 a = B.bonds[k];
        const double2 p = B.bprm[k];  // r0, k
        double d[3];
        diff(a.x, a.y, d);
        const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        const double dr = r - p.x;
        eb = 0.5 * p.y * dr * dr;
        const double s = -p.y * dr / r;
        addf(a.x, s, d);
        addf(a.y, -s, d);
    } else if (k < B.nb + B.na) {
        const int4 a = B.angles[k - B.nb];
        const double2 p = B.aprm[k - B.nb];  // theta0, k
        double v1[3], v2[3];
        diff(a.x, a.y, v1);
        diff(a.z, a.y, v2);
        const double r1 = sqrt(v1[0] * v1[0] + v1[1] * v1[1] + v1[2] * v1[2]);
        const double r2 = sqrt(v2[0] * v2[0] + v2[1] * v2[1] + v2[2] * v2[2]);
        double c = (v1[0] * v2[0] + v1[1] * v2[1] + v1[2] * v2[2]) / (r1 * r2);
        c = fmin(1.0, fmax(-1.0, c));
        const double th = acos(c);
        const double dth = th - p.x;
        ea = 0.5 * p.y * dth * dth;
        const double sn = fmax(sqrt(1.0 - c * c), 1e-300);
        const double g = p.y * dth / sn;  // -dE/dtheta * (-1/sin)
        double f1[3], f3[3];
        for (int q = 0; q < 3; ++q) {
            f1[q] = g * (v2[q] / (r1 * r2) - c * v1[q] / (r1 * r1));
            f3[q] = g * (v1[q] / (r1 * r2) - c * v2[q] / (r2 * r2));
        }
        const double one[3] = {1.0, 1.0, 1.0};
        for (int q = 0; q < 3; ++q) {
            add_fixed(B.F + 3ll * a.x + q, f1[q]);
            add_fixed(B.F + 3ll * a.z + q, f3[q]);
            add_fixed(B.F + 3ll * a.y + q, -(f1[q] + f3[q]) * one[q]);
        }
    } else if (k < B.nb + B.na + B.nt) {
        const int t = k - B.nb - B.na;
        const int4 a = B.torsions[t];
        const double4 p = B.tprm[t];  // periodicity, phase, k
        double rij[3], rkj[3], rkl[3];
        diff(a.x, a.y, rij);
        diff(a.z, a.y, rkj);
        diff(a.z, a.w, rkl);
        const double m[3] = {rij[1] * rkj[2] - rij[2] * rkj[1], rij[2] * rkj[0] - rij[0] * rkj[2],
                             rij[0] * rkj[1] - rij[1] * rkj[0]};
        const double nv[3] = {rkj[1] * rkl[2] - rkj[2] * rkl[1], rkj[2] * rkl[0] - rkj[0] * rkl[2],
                              rkj[0] * rkl[1] - rkj[1] * rkl[0]};
        const double m2 = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
        const double n2 = nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2];
        const double rkj2 = rkj[0] * rkj[0] + rkj[1] * rkj[1] + rkj[2] * rkj[2];
        const double nrkj = sqrt(rkj2);
        double cp = (m[0] * nv[0] + m[1] * nv[1] + m[2] * nv[2]) / sqrt(m2 * n2);
        cp = fmin(1.0, fmax(-1.0, cp));
        const double sgn = rij[0] * nv[0] + rij[1] * nv[1] + rij[2] * nv[2];
        const double phi = sgn < 0.0 ? -acos(cp) : acos(cp);
        et = p.z * (1.0 + cos(p.x * phi - p.y));
        const double dV = -p.z * p.x * sin(p.x * phi - p.y);
        double fi[3], fl[3], fj[3], fk[3];
        const double pp = (rij[0] * rkj[0] + rij[1] * rkj[1] + rij[2] * rkj[2]) / rkj2;
        const double qq = (rkl[0] * rkj[0] + rkl[1] * rkj[1] + rkl[2] * rkj[2]) / rkj2;
        for (int q = 0; q < 3; ++q) {
            fi[q] = -dV * nrkj / m2 * m[q];
            fl[q] = dV * nrkj / n2 * nv[q];
        }
        for (int q = 0; q < 3; ++q) {
            const double sv = pp * fi[q] - qq * fl[q];
            fj[q] = fi[q] - sv;
            fk[q] = fl[q] + sv;
        }
        for (int q = 0; q < 3; ++q) {
            add_fixed(B.F + 3ll * a.x + q, fi[q]);
            add_fixed(B.F + 3ll * a.y + q, -fj[q]);
            add_fixed(B.F + 3ll * a.z + q, -fk[q]);
            add_fixed(B.F + 3ll * a.w + q, fl[q]);
        }
    }
    const double sb = block_sum<256>(eb, red);
    const double sa = block_sum<256>(ea, red);
    const double stt = block_sum<256>(et, red);
    if (threadIdx.x == 0) {
        eslot[3 * blockIdx.x] = sb;
        eslot[3 * blockIdx.x + 1] = sa;
        eslot[3 * blockIdx.x + 2] = stt;
    }
}

hipError_t launch_bonded(const BondedPtrs& B, double* eslot, int nblocks, hipStream_t st) {
    if (nblocks <= 0) return hipSuccess;
    k_bonded<<<nblocks, 256, 0, st>>>(B, eslot);
    return hipGetLastError();
}

}  // namespace atm
