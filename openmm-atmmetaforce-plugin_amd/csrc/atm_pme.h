// Device-side layout of the PME variable-group evaluation and of the bonded
// terms (kernels in atm_pme.hip, host side in atm_pme_capi.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "atm_internal.h"

namespace atm {

constexpr int kPmeCellMax = 1024;  // atoms per cell the cell sort holds
// Block of the direct kernel: atoms of a cell, atoms of its neighbour cell staged at a time, waves.
// 48 us for 8,479 atoms and 120 for 25,437 (cells of some 133); (64, 160, 8) 55 / 156,
// (64, 160, 2) 70 / 133, (128, 160, 8) 73 / 151, (192, 192, 8) 74 / 152.  Staged atoms 96 / 160 / 224 at other
// cell sizes, whole calls of 16,958 atoms in us: cells of 39 295 / 294 / 294, 68 284 / 285 / 283, 132 296 / 287 /
// 286, 202 318 / 310 / 300, 314 355 / 341 / 337.
constexpr int kPmeIBlock = 64;
constexpr int kPmeJBlock = 160;
constexpr int kPmeDirectWaves = 4;
// Displacement classes: 0 not displaced, 1 .. kPmeClassMax the same for atoms displaced alike; with the
// atom (below 2^24) in one word.
constexpr int kPmeClassShift = 24, kPmeClassMax = 127, kPmeAtomMask = (1 << kPmeClassShift) - 1;
constexpr int kPmeExWords = 4;       // words of each i-atom's exclusion row it stages (groups of up to 128 atoms)
constexpr int kPmeSpreadSplit = 4; // parts of a cell's atoms spread by separate blocks (own LDS tiles)
constexpr int kPmeHalfShell = 14;  // the cell itself and its 13 forward neighbour cells
constexpr int kPmeBinLds = 4096;   // cell grids up to this size are binned through LDS histograms
constexpr int kPmeDftLdsMax = 600; // grid lines up to this length are transformed from LDS
constexpr int kPmeTileLdsMax = 49152;  // bytes of LDS for one cell's charge-grid tile
constexpr int kPmeFuseNT = 512;    // threads of the fused transform kernels ...
constexpr int kPmeFuseMax = 4096;  // ... and complex points they hold (8 per thread in registers between steps)
constexpr int kPmeLineTile = 16;   // grid lines per block of the fused line kernel (fewer when lines are long)

// Scalars of one evaluation (by value in the kernel arguments).
struct PmeDesc {
    int n;                       // atoms
    int m[3], ncell;             // cell grid (edge >= rc, at least 3 per axis)
    int cellCap, chunks;         // atoms per cell the direct kernel covers (chunks of kPmeIBlock)
    int K[3], ngrid;             // PME grid
    int twOff[3];                // offset of each axis' twiddle table
    int nex;                     // exception pairs
    int nslot, nslotDirect, nslotEx;  // energy slots per state (direct | exceptions | reciprocal)
    int nslotPairs;              // direct slots of the cell pairs (delta: of state 0, for both states); the displaced
                                 // atoms' own follow in each state
    int delta;                   // x + d shares the direct space that d leaves alone, and its charges are the difference
                                 // from x (few displaced atoms)
    int nlig;                    // displaced atoms
    // fused transforms (fused != 0): planes over axes pAx, qAx in LDS, then lines along lineAx with the
    // convolution; every axis length K = fA (K / fA) in two short steps
    int fused, lineAx, pAx, qAx, fA[3], lineTile, lineBlocks;
    int tile[3], tileBytes;      // per-cell charge-grid tile (0 bytes: spread without tiles)
    double L[3], invL[3];
    double rc2, alpha, twoAlphaSqrtPi, pi2OverAlpha2;
    double recipEnergyScale;     // k_e / (2 pi V)
    double recipPhiScale;        // k_e / (pi V)
    double selfEnergy;           // -k_e alpha / sqrt(pi) sum q^2
    double dispersionEnergy;     // long-range LJ correction / V
};

struct PmePtrs {
    const double* x;        // [3n] positions (state 0)
    double* x2;             // [3n] x + d (state 1)
    const double* displ;    // [3n]
    int* cellOf;            // [n]
    int* rankOf;            // [n]
    int* cellCount;         // [ncell]
    int* cellStart;         // [ncell + 1]
    int* cellAtoms;         // [n]
    double4* wpos;          // [n] wrapped positions
    const double2* prm;     // [n] (q sqrt(k_e), q)
    const double2* prm2;    // [n] (sigma/2, 2 sqrt(eps))
    const int4* exkey;      // [n] (exclusion group, rank in group, bitmap row offset, displacement class)
    double4* cpos;          // [n] cell order: wrapped x, y, z, q sqrt(k_e)
    double2* cprm;          // [n] cell order: sigma/2, 2 sqrt(eps)
    int4* cex;              // [n] cell order: group, rank, row offset, atom | class << kPmeClassShift
    const uint32_t* exbits; // exclusion bitmaps
    const int2* expairs;    // [nex]
    const double4* exprm;   // [nex] (k_e qq', sigma', 4 eps', k_e q_i q_j)
    long long* qgrid;       // [2][ngrid] fixed-point charge grids (delta: the second is the difference)
    double2* g0;            // [2][ngrid]
    double2* g1;            // [2][ngrid] (fused: the potentials, [2][ngrid] doubles)
    const double2* tw;      // twiddles of the three axes
    const double* bmod;     // B-spline moduli of the three axes, concatenated
    unsigned long long* F;  // [3][3][n] fixed-point forces (SoA): of state 0, of state 1, and the part both share
    const int* lig;         // [nlig] displaced atoms
    double* eslot;          // [2][nslot]
    double* parts;          // [2][5]
    SysResult* result;
    const AtmParamsDev* params;  // the nine ATM parameters (in the input block)
    const double* eoff;          // [2] energies of other variable-group forces added to U1, U2 (in the input block)
    int* overflow;
    // page-locked host memory the kernels read and write in place: the parameters, offsets and
    // positions of this evaluation, copied by the first kernel to `in`, and its results (every address
    // the kernels use is in here: a captured evaluation is made again when one of them changes)
    const double* hostIn;   // [kPmeInHead + 3n]
    double* in;             // [kPmeInHead + 3n] (params, eoff and x point into it)
    struct PmeHostRecord* record;
    double* hostF;          // [3n] the force, atom by atom
};

// The head of the input block: the nine ATM parameters and the two offsets, padded.
constexpr int kPmeInHead = 16;

struct PmeHostRecord {
    SysResult result;
    double parts[10];
    int overflow;
};

struct BondedPtrs {
    const double* x;          // [3n]
    unsigned long long* F;    // [3n] fixed point (AoS)
    const int2* bonds;
    const double2* bprm;      // r0, k
    const int4* angles;       // i, j (vertex), k, -
    const double2* aprm;      // theta0, k
    const int4* torsions;
    const double4* tprm;      // periodicity, phase, k, -
    int nb, na, nt;
};

hipError_t launch_pme_fill(unsigned long long* p, long long n, hipStream_t st);
// Every kernel of one evaluation (single: state 0 only) up to the energy sums.
hipError_t launch_pme_states(const PmeDesc& D, const PmePtrs& P, bool single, hipStream_t st);
// Energy sums and combine; forces: the hybrid force into P.hostF
hipError_t launch_pme_finish(const PmeDesc& D, const PmePtrs& P, bool single, bool forces, hipStream_t st);
hipError_t launch_bonded(const BondedPtrs& B, double* eslot, int nblocks, hipStream_t st);

}  // namespace atm
