// Device-side building blocks for the gfx950 transport engine: the
// per-particle Philox4x32-10 stream, 64-wide wavefront helpers, and the
// layouts of tables, phantoms, jobs and particle queues in HBM.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "omc_dev.h"

namespace omc {

// Global-memory view of a pointer.  A pointer read from LDS or from memory
// carries no address space, so the compiler reaches it with FLAT
// instructions, which also wait on the LDS counter; the cast makes the loads
// and atomics through it global ones.
template <typename T> using gmem = __attribute__((address_space(1))) T;
template <typename T> __device__ __forceinline__ gmem<T> *glob(T *p) { return (gmem<T> *)p; }

constexpr double RM = OMC_RM;
constexpr int MXGE = OMC_MXGE;
constexpr int MXEKE = OMC_MXEKE;
constexpr int MAXMED = OMC_MXMED;
constexpr int MAX_PHANTOMS = 16;     // resident phantoms per context

// ---------------------------------------------------------------- RNG -----
// Philox4x32-10 (Salmon et al., SC'11).  Each particle owns a stream: key
// (k0,k1) and a draw counter `ctr`; draw d uses word d&3 of block d>>2 and
// becomes the 24-bit uniform (w >> 8) * 2^-24, the same granularity as the
// RANMAR numbers ompMC uses.  A secondary's key is the Philox block
// (parent ctr, 1, 0, 0) under the parent key, taken after the interaction's
// last draw, so every history is independent of processing order.
//
// One round: the two 32x32 products as 64-bit multiplications, which the
// compiler turns into one v_mad_u64_u32 each instead of a v_mul_lo and a
// v_mul_hi (all of them quarter rate), and the two xors of a word as one
// v_bitop3_b32, which it does not find by itself.  The kernels are bound by
// VALU issue where pipelines overlap: FP32 slab of 1e8 histories 302 -> 296 ms,
// 400 beamlets 399 -> 392 ms.
__device__ __forceinline__ void philox_round(uint32_t &c0, uint32_t &c1, uint32_t &c2, uint32_t &c3, uint32_t k0,
                                             uint32_t k1)
{
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    constexpr unsigned XOR3 = 0x96;     // truth table of a ^ b ^ c
    const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, XOR3);
    const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, XOR3);
    c0 = n0; c1 = (uint32_t)p1; c2 = n2; c3 = (uint32_t)p0;
}

__device__ __forceinline__ void philox10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                         uint32_t k0, uint32_t k1, uint32_t out[4])
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        philox_round(c0, c1, c2, c3, k0, k1);
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// The same function with its rounds kept as a loop: for the rare paths
// inlined at every draw site (a block the ring does not hold, a secondary's
// key), where ten unrolled rounds would be most of the kernel's code.
__device__ __forceinline__ void philox10_rolled(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                uint32_t k0, uint32_t k1, uint32_t out[4])
{
#pragma unroll 1
    for (int r = 0; r < 10; ++r) {
        philox_round(c0, c1, c2, c3, k0, k1);
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// The uniform of a Philox word: (w >> 8) * 2^-24, exact in FP32.
__device__ __forceinline__ float philox_uniform(uint32_t w) { return (float)(w >> 8) * (1.0f / 16777216.0f); }

// Look-ahead of a lane's stream in LDS: RNG_RING Philox blocks per lane as
// ready uniforms, draw d in row d % (4 * RNG_RING) of the lane's column (rows
// are a block's threads wide, so any mix of rows is free of bank conflicts).
// A draw is then one 4-byte LDS read behind a wavefront-wide test that the
// ring holds it: about 8 instructions.  Holding the current block's four
// words in registers instead, as this engine did before, took about 50 per
// draw: the compiler carried the words, the block number and the ring's end
// through every divergent region of some fifty draw sites (2200 of the FP32
// charged-particle kernel's 13400 vector instructions were such copies).
// ring_fill() tops the rings of a wavefront up where its lanes are converged
// (the head of each trip).  The words and their order are those of the stream
// itself.  The ring is the launch's dynamic LDS (RNG_RING_BYTES).
constexpr uint32_t RNG_RING = 8;
constexpr int RNG_LANES = 256;           // threads per transport block
constexpr size_t RNG_RING_BYTES = (size_t)RNG_RING * 4 * RNG_LANES * sizeof(float);
extern __shared__ float rng_ring[];      // [4 * RNG_RING][RNG_LANES]

// Computes block b of stream (k0, k1) into the ring column `col`.
template <bool ROLLED>
__device__ __forceinline__ void ring_block(uint32_t b, uint32_t k0, uint32_t k1, uint32_t col)
{
    uint32_t o[4];
    if (ROLLED) philox10_rolled(b, 0u, 0u, 0u, k0, k1, o);
    else philox10(b, 0u, 0u, 0u, k0, k1, o);
    float *r = rng_ring + (b % RNG_RING) * (4 * RNG_LANES) + col;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i * RNG_LANES] = philox_uniform(o[i]);
}

// Blocks b and, if `both`, b + 1, whose rounds share one key schedule and
// overlap each other's multiplications.
__device__ __forceinline__ void ring_two_blocks(uint32_t b, bool both, uint32_t k0, uint32_t k1, uint32_t col)
{
    uint32_t c0 = b, c1 = 0u, c2 = 0u, c3 = 0u, d0 = b + 1u, d1 = 0u, d2 = 0u, d3 = 0u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        philox_round(c0, c1, c2, c3, k0, k1);
        philox_round(d0, d1, d2, d3, k0, k1);
    }
    float *r = rng_ring + (b % RNG_RING) * (4 * RNG_LANES) + col;
    r[0] = philox_uniform(c0); r[RNG_LANES] = philox_uniform(c1);
    r[2 * RNG_LANES] = philox_uniform(c2); r[3 * RNG_LANES] = philox_uniform(c3);
    if (both) {
        r = rng_ring + ((b + 1u) % RNG_RING) * (4 * RNG_LANES) + col;
        r[0] = philox_uniform(d0); r[RNG_LANES] = philox_uniform(d1);
        r[2 * RNG_LANES] = philox_uniform(d2); r[3 * RNG_LANES] = philox_uniform(d3);
    }
}

struct Rng {
    uint32_t k0, k1, ctr;
    uint32_t tail;           // draws [ctr, tail) are in this thread's ring column (multiple of 4)

    // Nothing in the ring (secondaries, particles read from a queue).  Only
    // the stream of the particle a transport lane owns is drawn from, so the
    // thread's column holds that stream only.
    __device__ __forceinline__ void reset_cache() { tail = 0u; }

    // Next uniform.  The test is taken by the wavefront's active lanes
    // together (a scalar branch); a stream that ran past its ring computes
    // its next block on the spot.
    __device__ __forceinline__ float next()
    {
        const uint32_t c = ctr;
        if (__ballot(c >= tail) != 0) {
            if (c >= tail) {
                ring_block<true>(c >> 2, k0, k1, threadIdx.x);
                tail = (c & ~3u) + 4u;
            }
        }
        ctr = c + 1u;
        return rng_ring[(c % (4 * RNG_RING)) * RNG_LANES + threadIdx.x];
    }
    // Makes the next n draws available to at() (n <= 4 * RNG_RING - 3).
    __device__ __forceinline__ void ensure(uint32_t n)
    {
        const uint32_t end = ctr + n;
        if (__ballot(end > tail) != 0) {
            if (end > tail) {
                uint32_t t = max(tail, ctr & ~3u);
                do {
                    ring_block<true>(t >> 2, k0, k1, threadIdx.x);
                    t += 4u;
                } while (t < end);
                tail = t;
            }
        }
    }
    // Draw ctr + k, without taking it.
    __device__ __forceinline__ float at(uint32_t k) const
    {
        return rng_ring[((ctr + k) % (4 * RNG_RING)) * RNG_LANES + threadIdx.x];
    }
    // Key of a secondary: the Philox block (ctr, tag, 0, 0) under this key.
    // Interactions use tag 1 for the particles they create; tag 2 is for a
    // copy of the stream's own particle handed on while the stream goes on
    // (photon splitting), so the two never share a key.
    __device__ __forceinline__ void child(uint32_t &c0, uint32_t &c1, uint32_t tag = 1u) const
    {
        uint32_t o[4];
        philox10_rolled(ctr, tag, 0u, 0u, k0, k1, o);
        c0 = o[0]; c1 = o[1];
    }
};

// A stream read in order by one thread without a ring (the source kernel).
struct SeqRng {
    uint32_t k0, k1, ctr;
    uint32_t w[4];

    __device__ __forceinline__ float next()
    {
        if ((ctr & 3u) == 0u) philox10(ctr >> 2, 0u, 0u, 0u, k0, k1, w);
        const float even = philox_uniform((ctr & 2u) ? w[2] : w[0]), odd = philox_uniform((ctr & 2u) ? w[3] : w[1]);
        const float x = (ctr & 1u) ? odd : even;
        ctr++;
        return x;
    }
};

// next uniform of a particle stream, in [0,1) with 24-bit granularity
template <typename R, typename S> __device__ __forceinline__ R urand(S &r) { return (R)r.next(); }

__device__ __forceinline__ void primary_key(uint32_t s0, uint32_t s1, uint64_t hid, uint32_t &k0, uint32_t &k1)
{
    uint32_t o[4];
    philox10((uint32_t)hid, (uint32_t)(hid >> 32), 2u, 0u, s0, s1, o);
    k0 = o[0]; k1 = o[1];
}

// ------------------------------------------------------------ wavefront ----
__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ uint32_t lanes_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// One atomic per wavefront for all active lanes that call it together; every
// calling lane gets a distinct index.  Works in divergent code (only the
// currently active lanes take part).
__device__ __forceinline__ uint32_t wave_reserve(uint32_t *counter, uint32_t n_per_lane)
{
    uint64_t m = __ballot(1);
    int leader = __ffsll((unsigned long long)m) - 1;
    uint32_t total = (uint32_t)__popcll(m) * n_per_lane;
    uint32_t base = 0;
    if (lane_id() == leader) base = atomicAdd(counter, total);
    base = __shfl(base, leader);
    return base + lanes_below(m) * n_per_lane;
}

// Between LDS accesses of lanes of one wavefront to each other's words.  LDS
// executes a wavefront's accesses in order; this keeps the compiler to it (no
// instruction).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Tops up the Philox rings of a wavefront's live lanes; every lane of the
// wavefront calls it, converged (`mask` is the ballot of `live`).
//
// With at most half of the lanes live, the idle lanes compute blocks too:
// each live lane gets 2, 4 or 8 consecutive lanes of the wavefront, which
// share its missing blocks (8 helpers do all of them in one pass).  A lone
// particle's trip spent a fifth of its time on four or five passes of one
// lane each.
//
// In a fuller wavefront each lane computes its own, two blocks a pass (one
// where it has room for one only), as long as RNG_FILL_LANES lanes have room
// for two or a lane holds fewer than RNG_FILL_MIN: the few lanes that drew most
// in the last trip catch up over the next ones instead of costing the wavefront
// a pass each.
#ifndef OMC_RNG_FILL_LANES
#define OMC_RNG_FILL_LANES 24
#endif
#ifndef OMC_RNG_FILL_MIN
#define OMC_RNG_FILL_MIN 6
#endif
__device__ __forceinline__ void ring_fill(Rng &r, bool live, uint64_t mask)
{
    wave_lds_fence();                  // the owners' reads so far before the helpers' writes
    const uint32_t cur = r.ctr >> 2;
    uint32_t tb = max(r.tail >> 2, cur);                    // first block not in the ring
    uint32_t room = live ? cur + RNG_RING - tb : 0u;
    const int nlive = __popcll(mask);
    if (nlive <= 32) {
        const int sh = nlive <= 8 ? 3 : nlive <= 16 ? 2 : 1;
        const int lane = lane_id();
        const int rank = (int)lanes_below(mask);            // among the live lanes
        // lane i learns the live lane of rank i: a permutation, live lanes first
        const int at = live ? rank : nlive + lane - rank;
        const int of_rank = __builtin_amdgcn_ds_permute(at << 2, lane);
        const int own = __builtin_amdgcn_ds_bpermute((lane >> sh) << 2, of_rank);
        const uint32_t k0 = (uint32_t)__builtin_amdgcn_ds_bpermute(own << 2, (int)r.k0);
        const uint32_t k1 = (uint32_t)__builtin_amdgcn_ds_bpermute(own << 2, (int)r.k1);
        const uint32_t first = (uint32_t)__builtin_amdgcn_ds_bpermute(own << 2, (int)tb);
        // (every lane takes part in the exchange: a lane that is masked off
        // has no value to give)
        const uint32_t want = (uint32_t)__builtin_amdgcn_ds_bpermute(own << 2, (int)room);
        const uint32_t n = (lane >> sh) < nlive ? want : 0u;
        const uint32_t col = (threadIdx.x & ~63u) + (uint32_t)own;
        for (uint32_t j = (uint32_t)lane & ((1u << sh) - 1u); __ballot(j < n) != 0; j += 1u << sh)
            if (j < n) ring_block<false>(first + j, k0, k1, col);
        tb += room;
    } else {
        while (__popcll(__ballot(room > 1u)) >= OMC_RNG_FILL_LANES ||
               __ballot(room > RNG_RING - OMC_RNG_FILL_MIN) != 0) {
            if (room) {
                const uint32_t n = min(room, 2u);
                ring_two_blocks(tb, n == 2u, r.k0, r.k1, threadIdx.x);
                tb += n;
                room -= n;
            }
        }
    }
    if (live) r.tail = tb << 2;
    wave_lds_fence();                  // the helpers' writes before the owners' reads
}

// ------------------------------------------------------------- layouts ----
template <typename R> struct R2 { R c1, c0; };           // pwlf slope / intercept
template <typename R> struct R4 { R a1, a0, b1, b0; };   // two pwlf pairs

// Per (medium, charge, bin) electron step data used at every CH step
// (sig, tmxs, eta, blcce) and by msdist / the interaction choice.
template <typename R> struct ElecBin {
    R sig1, sig0, tmxs1, tmxs0;
    R eta1, eta0, blc1, blc0;
    R q1c1, q1c0, q2c1, q2c0;
    R br11, br10, br21, br20;
};

// CSDA data, FP64 in every precision mode: restricted stopping power,
// range to the first table energy, and that energy.
struct ElecCsda {
    double dedx1, dedx0, range, earr;
};

// multiple-scattering surface entry: alias threshold, alias index, u node
// One node of a multiple-scattering alias table (mscatSample tables): the
// alias weight, the node's value and the value of the node it aliases
// (same row), so that a draw is one load.
template <typename R> struct MsAlias {
    R wms, ums, ualias, pad;
};

// Per-medium scalars and the small tables.
struct MediumScalars {
    double ge0, ge1, eke0, eke1, blcc, xcc, esig_e, psig_e;
    double te, thmoll, ap, delcm, zbrang, bpar0, bpar1, pad;
    int mono_e, mono_p, meke;
    int nregular;            // leading electron bins in which zero_ustep's shortcut holds
    double dl1[8], dl2[8], dl3[8], dl4[8], dl5[8], dl6[8];
};

struct SmallTables {
    int nmed;
    int pad;
    double b2spin_min, dbeta2i, espml, dleneri, dqq1i, dllambi, dqmsi;
    // Rayleigh: ompMC samples with medium-0 form factors (ompmc.c:1120-1131)
    double xgrid[OMC_MXRAYFF], fcum[OMC_MXRAYFF], b_array[OMC_MXRAYFF], c_array[OMC_MXRAYFF];
    int i_array[OMC_RAYCDFSIZE];
    MediumScalars med[MAXMED];
};

// Device tables for precision R.  Photon bins are interleaved so one voxel
// step reads one 32-byte record.
template <typename R> struct DevTables {
    const SmallTables *small;
    const R4<R> *ph_mfp;     // {gmfp1, gmfp0, cohe1, cohe0} [imed*MXGE + bin]
    const R4<R> *ph_br;      // {gbr11, gbr10, gbr21, gbr20}
    const R2<R> *ph_pmax;    // {pmax1, pmax0}
    const ElecBin<R> *el;    // [(imed*2 + qel)*MXEKE + bin]
    const ElecCsda *csda;    // [(imed*2 + qel)*MXEKE + bin]
    const R *spin;           // [imed*32768 + qel*16384 + i*512 + j*32 + k]
    const MsAlias<R> *ms;    // [i*256 + j*32 + k]
};

// Resident phantom: region r = voxel + 1, region 0 = outside.
// Delta tracking of photon flights in a phantom with a uniform voxel grid
// whose media share one photon energy grid: mu[bin] bounds the attenuation
// coefficient (1/cm) of every voxel at every energy of that bin.
template <typename R> struct Woodcock {
    const R *mu;             // [MXGE] majorant; null = voxel stepping only
    double ge0, ge1;         // lgle = ge1 * log(E) + ge0 for every medium
    double x0, y0, z0;       // lower corner of the grid
    R idx, idy, idz;         // inverse voxel sizes
    int pad;
};

template <typename R> struct Side2 { R lo, hi; };        // lower and upper bound of a voxel on one axis

template <typename R> struct DevPhantom {
    int isize, jsize, ksize, nreg;
    const double *xb, *yb, *zb;
    // lower and upper bound of every voxel of each axis, rounded to R: x
    // voxels, then y, then z.  One load gives both sides of a voxel.
    const Side2<R> *sides;
    const uint8_t *med;      // [nreg] medium index, 0xff = vacuum / outside
    const R *rhof;           // [nreg]
    double ecut[MAXMED + 1]; // [imed + 1]; entry 0 is vacuum / outside
    double pcut[MAXMED + 1];
    Woodcock<R> wc;
};

// The medium scalars a charged particle's step reads, copied to LDS at kernel
// start (values in R where every use converts them): read from the table
// record in memory they were a chain of dependent loads in every step.
template <typename R> struct MedRec {
    double eke0, eke1, te;
    R keke0, keke1, blcc, xcc, sig_e, sig_p;
    R ap, thmoll, delcm, zbrang;
    R dl[6][4];              // screening coefficients of bremsstrahlung (dl1..dl6)
    int mono;                // bit 0 electrons, bit 1 positrons
    int nregular;

    __device__ __forceinline__ void stage(const MediumScalars &m)
    {
        eke0 = m.eke0; eke1 = m.eke1; te = m.te;
        keke0 = (R)m.eke0; keke1 = (R)m.eke1; blcc = (R)m.blcc; xcc = (R)m.xcc;
        sig_e = (R)m.esig_e; sig_p = (R)m.psig_e;
        ap = (R)m.ap; thmoll = (R)m.thmoll; delcm = (R)m.delcm; zbrang = (R)m.zbrang;
        for (int l = 0; l < 4; ++l) {
            dl[0][l] = (R)m.dl1[l]; dl[1][l] = (R)m.dl2[l]; dl[2][l] = (R)m.dl3[l];
            dl[3][l] = (R)m.dl4[l]; dl[4][l] = (R)m.dl5[l]; dl[5][l] = (R)m.dl6[l];
        }
        mono = (m.mono_e ? 1 : 0) | (m.mono_p ? 2 : 0);
        nregular = m.nregular;
    }
};

// The scalars of the elastic scattering tables, likewise.  Each test and index
// of a rejection loop waited for its own load of one of them (all lanes the
// same address); with these and the interactions' scalars (ap to dl) in LDS
// the charged-particle kernel of 2e7 FP32 slab histories takes 75.9 ms against
// 78.7, the slab of 1e8 289 against 297, 400 beamlets 381 against 391.
template <typename R> struct ScatRec {
    R b2spin_min, dbeta2i, espml, dleneri, dqq1i, dllambi, dqmsi;

    __device__ __forceinline__ void stage(const SmallTables &t)
    {
        b2spin_min = (R)t.b2spin_min; dbeta2i = (R)t.dbeta2i; espml = (R)t.espml; dleneri = (R)t.dleneri;
        dqq1i = (R)t.dqq1i; dllambi = (R)t.dllambi; dqmsi = (R)t.dqmsi;
    }
};

// What a charged-particle kernel keeps in LDS of the small tables.
template <typename R> struct ElectronRec {
    MedRec<R> med[MAXMED];
    ScatRec<R> scat;

    // (every thread of the block calls it)
    __device__ __forceinline__ void stage(const SmallTables &t)
    {
        const int k = (int)threadIdx.x - 64;
        if (k >= 0 && k < MAXMED) med[k].stage(t.med[k]);
        else if (threadIdx.x == 0) scat.stage(t);
    }
};

// The part of a phantom record a transport kernel's lanes read, copied to
// LDS at kernel start (cut-offs in R, as every use converts them).
template <typename R> struct GeoRec {
    int isize, jsize, ksize, nreg;
    const Side2<R> *sides;
    const uint8_t *med;
    const R *rhof;
    R ecut[MAXMED + 1];      // [imed + 1]; entry 0 is vacuum / outside

    __device__ __forceinline__ void stage(const DevPhantom<R> &p)
    {
        isize = p.isize; jsize = p.jsize; ksize = p.ksize; nreg = p.nreg;
        sides = p.sides; med = p.med; rhof = p.rhof;
        for (int m = 0; m <= MAXMED; ++m) ecut[m] = (R)p.ecut[m];
    }
};

template <typename R> struct PhotonGeoRec : GeoRec<R> {
    R pcut[MAXMED + 1];
    Woodcock<R> wc;

    __device__ __forceinline__ void stage(const DevPhantom<R> &p)
    {
        GeoRec<R>::stage(p);
        for (int m = 0; m <= MAXMED; ++m) pcut[m] = (R)p.pcut[m];
        wc = p.wc;
    }
};

// One source job (a dosxyz field, one beamlet, one serving request).
struct DevJob {
    int phantom;             // index into the phantom table
    int kind;                // 0 dosxyz field, 1 beamlet
    int charge;
    int spectrum;
    double energy;           // mono energy
    const double *cdf1, *cdf2;   // [1000] inverse CDF (device)
    double deltak;
    // dosxyz field
    double ssd, xinl, yinl, xsize, ysize;
    int ixinl, iyinl;
    // beamlet
    double src[3], corner[3], side1[3], side2[3];
    // histories
    uint64_t hist0;          // stream index of the first history
    int64_t nperbatch;
    uint32_t s0, s1;         // seed
    int nsplit;              // photon splitting (vrt.nsplit); 0 or 1 = off
    int pad_nsplit;
    double *tally;           // [slot*nreg + region], slot = batch
    double *ledger;          // optional [3*nhist]
};

// A run of consecutive histories [first, first + n) of one job, placed at
// thread offset `off` of a source launch and at entry `slot` of the queue of
// its particles' type.
struct SourceSeg {
    uint64_t first;
    uint32_t job, n, off, slot;
};

// Structure-of-arrays particle queue.  A particle that gave up its lane in
// the middle of its transport (a yield) also carries the lane's state, so
// the next launch resumes it exactly where it stopped.
//
// One allocation per queue: QR_N arrays of R (e x y z u v w wt, then the five
// real-valued resume variables), then QU_N arrays of uint32 (ir, meta =
// job << 3 | resume << 2 | (iq + 1), history index within the job, Philox
// key and counter, packed integer resume variables, loop trips taken so
// far), each `cap` long.  A queue is then three scalars -- base, tail
// counter, capacity -- and a kernel's three queues fit its scalar
// registers; with one pointer per array they took 135 of them and the
// compiler spilled pointers into vector-register lanes, reading them back
// before every table or queue access.
enum { QR_E, QR_X, QR_Y, QR_Z, QR_U, QR_V, QR_W, QR_WT, QR_ST, QR_N = QR_ST + 5 };
enum { QU_IR, QU_META, QU_HIST, QU_K0, QU_K1, QU_CTR, QU_SFLAGS, QU_TRIPS, QU_N };

template <typename R> struct Queue {
    char *base;
    uint32_t *count;         // device tail counter
    uint32_t cap;

    __host__ __device__ R *r(int f) const { return reinterpret_cast<R *>(base) + (size_t)f * cap; }
    __host__ __device__ uint32_t *u(int f) const
    {
        return reinterpret_cast<uint32_t *>(base + sizeof(R) * (size_t)QR_N * cap) + (size_t)f * cap;
    }
    __host__ __device__ R *e() const { return r(QR_E); }
    __host__ __device__ R *x() const { return r(QR_X); }
    __host__ __device__ R *y() const { return r(QR_Y); }
    __host__ __device__ R *z() const { return r(QR_Z); }
    __host__ __device__ R *uu() const { return r(QR_U); }
    __host__ __device__ R *v() const { return r(QR_V); }
    __host__ __device__ R *w() const { return r(QR_W); }
    __host__ __device__ R *wt() const { return r(QR_WT); }
    __host__ __device__ R *st(int k) const { return r(QR_ST + k); }
    __host__ __device__ int32_t *ir() const { return reinterpret_cast<int32_t *>(u(QU_IR)); }
    __host__ __device__ uint32_t *meta() const { return u(QU_META); }
    __host__ __device__ uint32_t *hist() const { return u(QU_HIST); }
    __host__ __device__ uint32_t *k0() const { return u(QU_K0); }
    __host__ __device__ uint32_t *k1() const { return u(QU_K1); }
    __host__ __device__ uint32_t *ctr() const { return u(QU_CTR); }
    __host__ __device__ uint32_t *sflags() const { return u(QU_SFLAGS); }
    __host__ __device__ uint32_t *trips() const { return u(QU_TRIPS); }
};

constexpr uint32_t META_RESUME = 4u;

// energy-ordered fetch of charged-particle launches (kernels_impl.h)
constexpr int SORT_BUCKETS = 64;
constexpr int SORT_BLOCKS = 128;

template <typename R> struct Particle {
    R e, x, y, z, u, v, w, wt;
    int ir, iq;
    uint32_t job, hist;
    Rng rng;
};

// Returns true if the entry carries a resume state.
template <typename R>
__device__ __forceinline__ bool q_load(const Queue<R> &q, uint32_t i, Particle<R> &p)
{
    p.e = q.e()[i]; p.x = q.x()[i]; p.y = q.y()[i]; p.z = q.z()[i];
    p.u = q.uu()[i]; p.v = q.v()[i]; p.w = q.w()[i]; p.wt = q.wt()[i];
    p.ir = q.ir()[i];
    uint32_t m = q.meta()[i];
    p.job = m >> 3;
    p.iq = (int)(m & 3u) - 1;
    p.hist = q.hist()[i];
    p.rng.k0 = q.k0()[i]; p.rng.k1 = q.k1()[i]; p.rng.ctr = q.ctr()[i];
    p.rng.reset_cache();
    return (m & META_RESUME) != 0u;
}

template <typename R>
__device__ __forceinline__ void q_store(const Queue<R> &q, uint32_t i, const Particle<R> &p, uint32_t resume = 0u)
{
    q.e()[i] = p.e; q.x()[i] = p.x; q.y()[i] = p.y; q.z()[i] = p.z;
    q.uu()[i] = p.u; q.v()[i] = p.v; q.w()[i] = p.w; q.wt()[i] = p.wt;
    q.ir()[i] = p.ir;
    q.meta()[i] = (p.job << 3) | resume | (uint32_t)(p.iq + 1);
    q.hist()[i] = p.hist;
    q.k0()[i] = p.rng.k0; q.k1()[i] = p.rng.k1; q.ctr()[i] = p.rng.ctr;
}

// Physics events counted by the transport kernels, in the order of the
// omc_dev_stats fields.  The rare ones (interactions) are counted per block
// with LDS atomics; the frequent ones (every condensed history step) in a
// per-thread LDS slot, so neither holds a register.
enum EvKind {
    EV_COMPTON, EV_PHOTO, EV_PAIR, EV_RAYLEIGH, EV_BREMS, EV_MOLLER, EV_BHABHA, EV_ANNIH, EV_RANNIH, EV_FICT,
    EV_NRARE,
    EV_MSDIST = EV_NRARE, EV_SSCAT, EV_HOWFAR_E,
    EV_N
};

// Counters and error flags of a pipeline.  The device keeps STATUS_COPIES of
// them, each on lines of its own, and a block adds to the copy of its number:
// all blocks of a launch end with some ten additions each, and one address
// serves an atomic every 11 to 12 ns.  k_gen_end sums the copies.
constexpr int STATUS_COPIES = 16;
struct alignas(256) DevStatus {
    uint32_t overflow;       // a push found its queue full
    uint32_t killed;         // particles stopped by the per-particle step limit
    unsigned long long yields;                         // particles handed to the next launch
    unsigned long long photon_steps, electron_steps;   // transport loop trips
    unsigned long long photon_cross, electron_cross;   // voxel boundaries crossed
    unsigned long long photon_dep, electron_dep;       // ausgab calls
    unsigned long long wc_over;                        // delta-tracking sites above the majorant
    unsigned long long ev[EV_N];                       // physics events (EvKind)
};

// Words between the counters of a pipeline's queues: each on a line of its own,
// since tail and fetch counters on one line wait for each other's atomics.  With
// the status' copies and one addition per block at a launch's end instead of
// one per wavefront, the photon kernel of 2e7 FP32 slab histories went from
// 14.5 to 9.5 ms, that of 400 beamlets from 86 to 62 ms.
constexpr int COUNT_STRIDE = 64;

// Sums of a launch that every thread adds to once, at its end.
enum { SUM_STEPS, SUM_CROSS, SUM_DEP, SUM_YIELDS, SUM_LONGEST, SUM_N };
static __shared__ uint32_t ev_sums[SUM_N];
static __shared__ uint32_t ev_block[EV_NRARE];
static __shared__ uint32_t ev_lane[EV_N - EV_NRARE][RNG_LANES];

// Zeroes the block's event counters (the per-thread slots only where the
// kernel counts frequent events); the caller synchronises the block before
// the first count.
template <bool LANES> __device__ __forceinline__ void events_begin()
{
    if (threadIdx.x < EV_NRARE) ev_block[threadIdx.x] = 0u;
    if (threadIdx.x < SUM_N) ev_sums[threadIdx.x] = 0u;
    if (LANES)
        for (int k = 0; k < EV_N - EV_NRARE; ++k) ev_lane[k][threadIdx.x] = 0u;
}

// A rare event in this lane: an LDS atomic (same-address lanes of a
// wavefront are serialised by the LDS, which costs little for events that
// come a few times per history).
__device__ __forceinline__ void count_event(int k) { atomicAdd(&ev_block[k], 1u); }

// A frequent event of this thread's lane.
// (An LDS atomic without a result: a read, an addition and a write would wait
// for the read.)
__device__ __forceinline__ void count_lane_event(int k) { atomicAdd(&ev_lane[k - EV_NRARE][threadIdx.x], 1u); }

// Largest of v over a wavefront, sums of the others: into the block's sums.
__device__ __forceinline__ void sum_up(int k, uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t w = (uint32_t)__shfl_xor((int)v, o);
        v = k == SUM_LONGEST ? max(v, w) : v + w;
    }
    if (lane_id() == 0 && v) {
        if (k == SUM_LONGEST) atomicMax(&ev_sums[k], v);
        else atomicAdd(&ev_sums[k], v);
    }
}

// Adds the block's counts to its copy of the status, and the trips of its
// longest track to *longest (every thread of the block calls it once, after
// its transport loop, with its own counts).
template <bool LANES>
__device__ __forceinline__ void events_end(DevStatus *st, uint32_t *longest, uint32_t steps, uint32_t cross,
                                           uint32_t dep, uint32_t yields, uint32_t trips)
{
    sum_up(SUM_STEPS, steps);
    sum_up(SUM_CROSS, cross);
    sum_up(SUM_DEP, dep);
    sum_up(SUM_YIELDS, yields);
    sum_up(SUM_LONGEST, trips);
    __syncthreads();
    const int k = threadIdx.x;
    if (k < EV_NRARE) {
        if (ev_block[k]) atomicAdd(&st->ev[k], (unsigned long long)ev_block[k]);
    } else if (LANES && k < EV_N) {
        unsigned long long n = 0;
        for (int t = 0; t < RNG_LANES; ++t) n += ev_lane[k - EV_NRARE][t];
        if (n) atomicAdd(&st->ev[k], n);
    } else if (k >= 64 && k < 64 + SUM_N && ev_sums[k - 64]) {
        const uint32_t v = ev_sums[k - 64];
        if (k - 64 == SUM_STEPS) atomicAdd(LANES ? &st->electron_steps : &st->photon_steps, (unsigned long long)v);
        else if (k - 64 == SUM_CROSS) atomicAdd(LANES ? &st->electron_cross : &st->photon_cross, (unsigned long long)v);
        else if (k - 64 == SUM_DEP) atomicAdd(LANES ? &st->electron_dep : &st->photon_dep, (unsigned long long)v);
        else if (k - 64 == SUM_YIELDS) atomicAdd(&st->yields, (unsigned long long)v);
        else atomicMax(longest, v);
    }
}

}  // namespace omc
