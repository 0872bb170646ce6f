// Persistent forced-scattering life-cycle kernel (the benchmarked engine): one photon packet
// per lane at a time, run as a small state machine -- peel-off traversal, forced path first
// pass, second pass to the interaction point, scattering.  Every loop iteration advances each
// busy lane by one cell crossing; lanes whose traversal ended wait until enough lanes of the
// wavefront are waiting (the transition threshold), then the wave runs one transition round
// together, so the divergent event code is amortised over many lanes.  Lanes whose packet
// terminated refill from a global history counter with one atomic per wavefront (ballot +
// mbcnt prefix), which stream-compacts packets of very uneven path length without a
// separate compaction pass.  The order of operations within each packet is the reference's
// (MonteCarloSimulation.cpp:614-694, :1492-1544, :2034-2092).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "../../include/skirt_mi355x.h"
#include "guide.hpp"
#include "lifecycle.hpp"
#include "pipeline.hpp"
#include "traverse.hpp"

namespace skg
{
    // ------------------------------------------------------------------ the life cycle
    struct SimParams
    {
        GridView grid;
        const double* dens;
        const float* dens32;
        int nlambda;
        int nframes;
        const double* lambda;
        const double* sext;
        const double* ssca;
        const double* gpar;
        const double* lpack;
        double src[3];
        double xi, min_weight_reduction;
        int min_scatt;
        int threshold;
        int lanes;  // packets that each wavefront takes at a time (lanes per packet: L)
        uint64_t seed;
        uint64_t first, count;
        unsigned long long* queue;     // next history offset (work queue head)
        unsigned long long* counters;  // kNumCounters event counters
        double* frame;
        const FrameGeom* frames;  // device copy of the instrument geometry
        const Instance* inst;     // batched instances (ninst > 0) or none
        int ninst;
        const double* ilpack;     // launch luminosities per instance (ninst x nlambda)
        GuideNet net;             // guided variant: the network, its input frame and the mixture
        GuideFrame gframe;
        double guideMix;
        uint32_t contKey;         // nonzero: histories continue on Philox tag contKey from their first
                                  // scattering on (same emission and first interaction, independent
                                  // continuations)
        int32_t srcHint;          // the cell (octree: leaf node) of the point source (the start hint of its packets), -1: none
        double* rf;               // radiation-field variant: ncells x nlambda table
        int persp;                // some instruments are perspective instruments
        int nent;                 // particle-source variant: number of entities (0: the point source)
        int entKernel;            // smoothing kernel: 0 uniform, 1 cubic spline
        const double* ent;        // per entity: x, y, z, smoothing length h
        const int64_t* entFirst;  // first history index of each entity (nent + 1 entries)
        const double* entLpack;   // launch luminosity per packet, nent x nlambda
        const double* entX;       // cubic spline: cumulative mass at u = k / kSplineN, k = 0..kSplineN
    };

    // kernel variants of the life cycle
    enum Variant : int
    {
        kPlain = 0,      // one run
        kBatched = 1,    // batched independent instances
        kGuided = 2,     // scattering directions from the defensive guide / HG mixture
        kStoreRF = 3,    // one run that also stores the radiation field of the forced paths (perspective
                         // instruments allowed)
        kPersp = 4,      // one run with perspective instruments among the instruments
        kParticles = 5   // one run whose source is a set of imported particles
    };
    constexpr int kSplineN = 400;  // CubicSplineSmoothingKernel's table size (CubicSplineSmoothingKernel.cpp:18)

    // SpecialFunctions::lnmean(x1, x2, lnx1, lnx2) (SpecialFunctions.cpp:860-880): the
    // logarithmic mean (x2 - x1) / ln(x2 / x1), by its series for nearly equal arguments
    __device__ __forceinline__ double ln_mean(double x1, double x2, double lnx1, double lnx2)
    {
        if (x1 > x2)
        {
            const double t = x1, lt = lnx1;
            x1 = x2;
            x2 = t;
            lnx1 = lnx2;
            lnx2 = lt;
        }
        if (x1 <= 0) return 0.;
        const double x = x2 / x1 - 1.;
        if (x < 1e-3)
        {
            const double c3 = 1. / 3., c5 = 1. / 5., c6 = 1. / 6.;
            return x1 / (1. - 0.5 * x + c3 * x * x - 0.25 * x * x * x + c5 * x * x * x * x - c6 * x * x * x * x * x);
        }
        return (x2 - x1) / (lnx2 - lnx1);
    }

    enum Phase : int
    {
        kFetch = 0,
        kPeel = 1,
        kFwd1 = 2,
        kFwd2 = 3,
        kDone = 4,
        kScatter = 5  // guided variant: peel-offs done, waiting for the wave's guided scattering
    };

#ifndef SKG_GUIDE_LANES
#define SKG_GUIDE_LANES 16
#endif
    constexpr int kGuideLanes = SKG_GUIDE_LANES;  // guided variant: lanes per network evaluation round
    constexpr int kMaxScatterings = 1 << 20;  // guard against non-terminating histories (NaN weights)
    constexpr int kMaxSteps = 1 << 26;        // guard against non-terminating traversals

    // Packet state that only the event transitions read and write.  Between transitions it
    // lives in LDS as a structure of arrays over the workgroup's lanes (conflict-free, one
    // 8-byte or 4-byte word per lane and field), so the crossing loop keeps only the
    // traversal state in registers.
    enum ColdF64 : int
    {
        cRx, cRy, cRz, cKx, cKy, cKz, cW, cLam, cLthr, cTaupath, cTauCached, cWp, kColdF64
    };
    enum ColdU32 : int
    {
        cHist0, cHist1, cDraw, cEll, cNscatt, cF, cPix, cFlags, cInst, cHint, kColdU32
    };
    constexpr int kLcThreads = 256;
    constexpr int kColdBytes = kLcThreads * (8 * kColdF64 + 4 * kColdU32);  // 34 KB per workgroup

    // LDS pointers: the event function, a call of its own, then reads the packet with LDS
    // instructions (a generic pointer would make them flat ones)
    typedef __attribute__((address_space(3))) double LdsF64;
    typedef __attribute__((address_space(3))) uint32_t LdsU32;

    __device__ __forceinline__ void lds_count(LdsU32* c, uint32_t v = 1u)
    {
        __hip_atomic_fetch_add(c, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    struct Packet
    {
        Philox rng;
        double rx, ry, rz, kx, ky, kz;
        double W, lam, Lthr, taupath, tauCached, Wp;
        int ell, nscatt, f, pix, inst;
        int hint;  // a cell (octree: a leaf's node) that probably holds the packet's position (-1: none)
        bool scat, haveTau;

        template<bool INST>
        __device__ __forceinline__ void load(const LdsF64* cd, const LdsU32* cu, int t, const SimParams& p)
        {
            rx = cd[cRx * kLcThreads + t];
            ry = cd[cRy * kLcThreads + t];
            rz = cd[cRz * kLcThreads + t];
            kx = cd[cKx * kLcThreads + t];
            ky = cd[cKy * kLcThreads + t];
            kz = cd[cKz * kLcThreads + t];
            W = cd[cW * kLcThreads + t];
            lam = cd[cLam * kLcThreads + t];
            Lthr = cd[cLthr * kLcThreads + t];
            taupath = cd[cTaupath * kLcThreads + t];
            tauCached = cd[cTauCached * kLcThreads + t];
            Wp = cd[cWp * kLcThreads + t];
            uint64_t h = static_cast<uint64_t>(cu[cHist0 * kLcThreads + t])
                         | (static_cast<uint64_t>(cu[cHist1 * kLcThreads + t]) << 32);
            inst = static_cast<int>(cu[cInst * kLcThreads + t]);
            hint = static_cast<int>(cu[cHint * kLcThreads + t]);
            nscatt = static_cast<int>(cu[cNscatt * kLcThreads + t]);
            rng.init(INST ? p.inst[inst].seed : p.seed, h, p.contKey != 0u && nscatt > 0 ? p.contKey : 0u);
            rng.draw = cu[cDraw * kLcThreads + t];
            ell = static_cast<int>(cu[cEll * kLcThreads + t]);
            f = static_cast<int>(cu[cF * kLcThreads + t]);
            pix = static_cast<int>(cu[cPix * kLcThreads + t]);
            uint32_t fl = cu[cFlags * kLcThreads + t];
            scat = fl & 1u;
            haveTau = (fl >> 1) & 1u;
        }

        __device__ __forceinline__ void store(LdsF64* cd, LdsU32* cu, int t) const
        {
            cd[cRx * kLcThreads + t] = rx;
            cd[cRy * kLcThreads + t] = ry;
            cd[cRz * kLcThreads + t] = rz;
            cd[cKx * kLcThreads + t] = kx;
            cd[cKy * kLcThreads + t] = ky;
            cd[cKz * kLcThreads + t] = kz;
            cd[cW * kLcThreads + t] = W;
            cd[cLam * kLcThreads + t] = lam;
            cd[cLthr * kLcThreads + t] = Lthr;
            cd[cTaupath * kLcThreads + t] = taupath;
            cd[cTauCached * kLcThreads + t] = tauCached;
            cd[cWp * kLcThreads + t] = Wp;
            cu[cHist0 * kLcThreads + t] = rng.h0;
            cu[cHist1 * kLcThreads + t] = rng.h1;
            cu[cDraw * kLcThreads + t] = rng.draw;
            cu[cEll * kLcThreads + t] = static_cast<uint32_t>(ell);
            cu[cNscatt * kLcThreads + t] = static_cast<uint32_t>(nscatt);
            cu[cF * kLcThreads + t] = static_cast<uint32_t>(f);
            cu[cPix * kLcThreads + t] = static_cast<uint32_t>(pix);
            cu[cFlags * kLcThreads + t] = (scat ? 1u : 0u) | (haveTau ? 2u : 0u);
            cu[cInst * kLcThreads + t] = static_cast<uint32_t>(inst);
            cu[cHint * kLcThreads + t] = static_cast<uint32_t>(hint);
        }
    };

    // What an event (life_event) returns: the packet's next phase and traversal -- direction, start
    // cell, section, the optical depth that ends it early (lim), the path length that does (slim) --
    // and the event's detector deposit (off < 0: none).  The traversal starts at the packet's
    // position.
    struct EventOut
    {
        int phase, hint, ell;
        double kx, ky, kz;
        double section, lim, slim, rfL;
        int64_t off;
        double v;

        // the traversal of the first of each group of L lanes to the whole group
        template<int L, int V> __device__ __forceinline__ void share()
        {
            if constexpr (L > 1)
            {
                phase = group_first<L>(phase);
                hint = group_first<L>(hint);
                kx = group_first<L>(kx);
                ky = group_first<L>(ky);
                kz = group_first<L>(kz);
                section = group_first<L>(section);
                lim = group_first<L>(lim);
                if constexpr (V == kPersp || V == kStoreRF) slim = group_first<L>(slim);
                if constexpr (V == kStoreRF)
                {
                    ell = group_first<L>(ell);
                    rfL = group_first<L>(rfL);
                }
            }
        }
    };

    // traversal state of one lane: the generator, the running sums and the phase (L lanes per packet)
    template<int GT, int FP, int L> struct Trav
    {
        Gen<GT, L> gen;
        int phase;
        bool ended;
        int steps;
        double tau, s;         // FP64 sums (s of a finished forced path: the distance of the interaction
                               // or of the path's end)
        Kahan32 tau32, s32;    // FP32 sums
        int last;              // cell (octree: node) of the last stored segment; the interaction's
        double section;
        double lim;            // the traversal ends where the optical depth exceeds it: the early-out
                               // of a peel-off, the interaction of a second forced pass
        int ell;        // radiation-field variant: the packet's bin, luminosity and the
        double rfL;     // extinction factor at the start of the current segment
        double rfExt;
        double slim;    // perspective variant: path length after which a peel-off ends

        __device__ __forceinline__ double tau_value() const
        {
            return FP == SKG_FP64 ? tau : static_cast<double>(tau32.sum);
        }
        __device__ __forceinline__ double s_value() const
        {
            return FP == SKG_FP64 ? s : static_cast<double>(s32.sum);
        }
        // the distance a finished forced path reached
        __device__ __forceinline__ double s_end(bool interaction) const
        {
            return FP == SKG_FP64 || interaction ? s : static_cast<double>(s32.sum);
        }
        __device__ __forceinline__ void add_length(double ds)
        {
            if (FP == SKG_FP64)
                s += ds;
            else
                s32.add(static_cast<float>(ds));
        }

        // the lane that acts for its packet (events, counts, sums in memory); the packet's other lanes
        // have the same traversal state
        static __device__ __forceinline__ bool lead() { return L == 1 || threadIdx.x % L == 0; }

        __device__ __forceinline__ void finish(LdsU32* lds)
        {
            ended = true;
            gen.idle();
            if (!lead()) return;
            // the crossing counters are added once, where a traversal ends
            lds_count(lds + 4, static_cast<uint32_t>(steps));
            if (phase == kFwd2) lds_count(lds + 7, static_cast<uint32_t>(steps));
        }

        // starts the traversal an event asked for and enters the domain; the path's length before
        // the domain, if any, is its first segment
        template<bool PERSP>
        __device__ __forceinline__ void start(const GridView& grid, const EventOut& io, LdsF64* cd, LdsU32* cu, LdsU32* lds,
                                              int t)
        {
            gen.start(cd[cRx * kLcThreads + t], cd[cRy * kLcThreads + t], cd[cRz * kLcThreads + t], io.kx, io.ky, io.kz,
                      io.hint);
            phase = io.phase;
            ended = false;
            steps = 0;
            tau = 0.;
            s = 0.;
            tau32.reset();
            s32.reset();
            last = -1;
            section = io.section;
            lim = io.lim;
            // radiation-field variant: the luminosity at the start of a forced path and the
            // extinction factor before its first segment (unused, and removed, elsewhere)
            ell = io.ell;
            rfL = io.rfL;
            rfExt = 1.;
            slim = io.slim;
            double entry;
            bool fin = !gen.begin(grid, entry);
            // every traversal starts at the packet's position: its start cell is the hint for the
            // next traversal from there
            if (gen.hint >= 0) cu[cHint * kLcThreads + t] = static_cast<uint32_t>(gen.hint);
            if (!fin && entry > 0.)
            {
                steps = 1;
                if (phase != kPeel)
                    add_length(entry);
                else if (PERSP)
                {
                    s += entry;
                    fin = s > slim;
                }
            }
            if (fin) finish(lds);
        }

        // one cell crossing of the current traversal; with RF, the first forced pass also
        // stores the radiation field (MonteCarloSimulation::storeRadiationField, :909-925):
        // L * lnmean(e^-tau_end, e^-tau_begin) * ds per stored segment in a cell
        template<bool RF, bool PERSP>
        __device__ __forceinline__ void step(const GridView& grid, LdsU32* lds, double* rf, int nl)
        {
            const int at = gen.i;  // the octree's leaves are named by their node, Voronoi cells by their run, others by m
            int m;
            double ds, nd;
            const int r = gen.cross(grid, m, ds, nd);
            if (r == 0) return;  // one level of the octree's descent
            // the traversal ends at the path's end (r < 0, or r == 2 after its last segment), where
            // its optical depth exceeds lim, or past a perspective peel-off's distance
            bool fin = r < 0 || ++steps > kMaxSteps;
            if (!fin)
            {
                const bool peel = phase == kPeel;
                const double tprev = tau_value(), sprev = s_value();
                // a peel-off's optical depth counts every segment, a forced path stores those of
                // positive length
                if (peel || ds > 0.)
                {
                    if (FP == SKG_FP64)
                        tau += section * nd * ds;
                    else
                        tau32.add(static_cast<float>(section) * static_cast<float>(nd) * static_cast<float>(ds));
                    if (!peel)
                    {
                        add_length(ds);
                        last = GT == kOctree || GT == kVoronoi ? at : m;
                        if constexpr (RF)
                        {
                            if (phase == kFwd1)
                            {
                                const double lnEnd = -tau_value();
                                const double extEnd = exp(lnEnd);
                                const double em = ln_mean(extEnd, rfExt, lnEnd, -tprev);
                                if (lead()) unsafeAtomicAdd(rf + static_cast<int64_t>(m) * nl + ell, rfL * em * ds);
                                rfExt = extEnd;
                            }
                        }
                    }
                }
                if (__builtin_expect(tau_value() > lim, 0))
                {
                    fin = true;
                    if (peel)
                    {
                        if (FP == SKG_FP64)
                            tau = INFINITY;
                        else
                            tau32.sum = INFINITY;
                    }
                    else
                    {
                        // the second pass stops at the first segment whose exit optical depth
                        // exceeds the interaction's
                        s = sprev + ((lim - tprev) / (tau_value() - tprev)) * (s_value() - sprev);
                    }
                }
                if constexpr (PERSP)
                {
                    // MediumSystem::getExtinctionOpticalDepth(pp, distance) (MediumSystem.cpp:
                    // 2376-2382): the segment that passes the distance still counts
                    if (peel)
                    {
                        s += ds;
                        if (s > slim) fin = true;
                    }
                }
            }
            if (__builtin_expect(fin || r == 2, 0)) finish(lds);
        }
    };

    // The deposits of one transition round into the frames (FluxRecorder::detect,
    // FluxRecorder.cpp:414-418, with LockFree::add, LockFree.hpp:23-36), combined across the
    // wavefront: the deposits into the pixel of the first depositing lane are summed by a
    // shuffle reduction over the whole (converged) wave into one FP64 atomic, the others are
    // added directly.  off < 0: no deposit.  Counter 5 counts the atomics issued.
    __device__ __forceinline__ void flush_deposits(double* frame, int64_t off, double val, LdsU32* lds)
    {
        const bool has = off >= 0;
        const unsigned long long m = __ballot(has);
        if (!m) return;
        const int leader = __ffsll(static_cast<long long>(m)) - 1;
        const int64_t key = __shfl(off, leader);
        const bool same = has && off == key;
        double v = same ? val : 0.;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (__lane_id() == leader)
        {
            unsafeAtomicAdd(frame + key, v);
            lds_count(lds + 5);
        }
        if (has && !same)
        {
            unsafeAtomicAdd(frame + off, val);
            lds_count(lds + 5);
        }
    }

    // The guided scattering direction (defensive mixture of the guide's lobes and HG) and its
    // weight factor Phi_HG / ((1 - mix) Phi_HG + mix q), from the network outputs o.  Not
    // inlined: its registers are then not added to those of the traversal state that is live
    // around the call in the persistent kernel.
    __device__ __attribute__((noinline)) double guided_direction(const float* o, double g, double mix, Philox& rng,
                                                                 double& kx, double& ky, double& kz)
    {
        LobesF Lb;
        guide_lobes_f(o, Lb);
        const double kxo = kx, kyo = ky, kzo = kz;
        const bool useGuide = rng.uniform() < mix;
        if (useGuide)
            guide_sample_f(Lb, rng, kx, ky, kz);
        else
            scatter_hg(rng, g, kx, ky, kz);
        const double c = kxo * kx + kyo * ky + kzo * kz;
        const double phi = (fabs(g) < 1e-6 ? 1.0 : value_hg(g, c)) / (4 * M_PI);
        const double q = guide_pdf_f(Lb, kx, ky, kz);
        return phi / ((1.0 - mix) * phi + mix * q);
    }

    // The event transitions of the life cycle, on a packet loaded from LDS.
    template<int GT, int V> struct Events
    {
        static constexpr bool INST = V == kBatched;
        const SimParams& p;
        EventOut& io;
        Packet& pk;
        LdsU32* lds;

        __device__ __forceinline__ void finish()
        {
            lds_count(lds + 0);
            io.phase = kFetch;
        }

        // the packet's next traversal, from its position
        __device__ __forceinline__ void travel(double dx, double dy, double dz, int ph, double lim)
        {
            io.phase = ph;
            io.kx = dx;
            io.ky = dy;
            io.kz = dz;
            io.hint = pk.hint;
            io.section = INST ? p.sext[pk.ell] * p.inst[pk.inst].scale : p.sext[pk.ell];
            io.lim = lim;
            io.slim = INFINITY;
            io.ell = pk.ell;
            io.rfL = pk.W / pk.lam;
        }

        // a peel-off of luminosity L: it ends at the optical depth log(L) + 745 (MediumSystem.cpp:
        // 2335), that is where the sum exceeds the next smaller number
        __device__ __forceinline__ void peel(double dx, double dy, double dz, double L)
        {
            lds_count(lds + 1);
            travel(dx, dy, dz, kPeel, nextafter(log(L) + 745, -INFINITY));
        }

        __device__ __forceinline__ void forced()
        {
            lds_count(lds + 2);
            travel(pk.kx, pk.ky, pk.kz, kFwd1, INFINITY);
        }

        // L exp(-tau) into the packet's pixel: held for the wave's combined flush at the end of
        // the round (a lane's second deposit in one round adds its first one directly)
        __device__ __forceinline__ void deposit(const FrameGeom& fg, double L, double t)
        {
            double v = L * exp(-t);
            if (io.off >= 0)
            {
                unsafeAtomicAdd(p.frame + io.off, io.v);
                lds_count(lds + 5);
            }
            io.off = fg.offset + pk.pix + static_cast<int64_t>(pk.ell) * fg.nx * fg.ny;
            io.v = v;
            lds_count(lds + 8);
        }

        // MonteCarloSimulation::performLifeCycle launch + SourceSystem::launch; in a batched
        // launch, history h is history h - offset of its instance
        __device__ __forceinline__ bool launch(uint64_t h)
        {
            uint64_t seed = p.seed;
            const double* lp = p.lpack;
            pk.inst = 0;
            if constexpr (INST)
            {
                int lo = 0, hi = p.ninst - 1;  // last instance whose offset is <= h
                while (lo < hi)
                {
                    int mid = (lo + hi + 1) >> 1;
                    if (p.inst[mid].offset <= h)
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                pk.inst = lo;
                h -= p.inst[lo].offset;
                seed = p.inst[lo].seed;
                lp = p.ilpack + static_cast<int64_t>(lo) * p.nlambda;
            }
            pk.rng.init(seed, h);
            pk.ell = static_cast<int>(pk.rng.uniform() * p.nlambda);
            if (pk.ell >= p.nlambda) pk.ell = p.nlambda - 1;
            pk.lam = p.lambda[pk.ell];
            // the particle launch: its own variant, and a run-time branch of the radiation-field
            // and perspective variants
            bool particles = false;
            if constexpr (V == kParticles)
                particles = true;
            else if constexpr (V == kStoreRF || V == kPersp)
                particles = p.nent > 0;
            if (particles)
            {
                // ImportedSource::launch: the entity whose history index range holds h
                // (ImportedSource.cpp:466-471), its luminosity for the bin (:653-705, the
                // oligochromatic bias weight folded into entLpack), a position from its smoothing
                // kernel (ParticleSnapshot::generatePosition, ParticleSnapshot.cpp:275-286)
                int lo = 0, hi = p.nent - 1;
                while (lo < hi)
                {
                    int mid = (lo + hi + 1) >> 1;
                    if (p.entFirst[mid] <= static_cast<int64_t>(h))
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                const int m = lo;
                pk.W = p.entLpack[static_cast<int64_t>(m) * p.nlambda + pk.ell] * pk.lam;
                const double X = pk.rng.uniform();
                double u;
                if (p.entKernel == 1)
                {
                    // CubicSplineSmoothingKernel::generateRadius (:78-85): NR::locateClip on the table
                    int a = 0, b = kSplineN;
                    while (b - a > 1)
                    {
                        int mid = (a + b) >> 1;
                        if (X >= p.entX[mid])
                            a = mid;
                        else
                            b = mid;
                    }
                    const double f = (X - p.entX[a]) / (p.entX[a + 1] - p.entX[a]);
                    u = (a + f) / kSplineN;
                }
                else
                    u = pow(X, 1.0 / 3.0);  // UniformSmoothingKernel::generateRadius (:27-31)
                double dx, dy, dz;
                isotropic(pk.rng, dx, dy, dz);
                const double hm = p.ent[4 * m + 3];
                pk.rx = p.ent[4 * m + 0] + dx * u * hm;
                pk.ry = p.ent[4 * m + 1] + dy * u * hm;
                pk.rz = p.ent[4 * m + 2] + dz * u * hm;
            }
            else
            {
                pk.W = lp[pk.ell] * pk.lam;
                pk.rx = p.src[0];
                pk.ry = p.src[1];
                pk.rz = p.src[2];
            }
            // (srcHint is the point source's cell: on a mesh, a particle far from it would first have that
            // cell rejected, after a round's wait)
            const int startHint = particles ? -1 : p.srcHint;
            isotropic(pk.rng, pk.kx, pk.ky, pk.kz);
            pk.nscatt = 0;
            pk.taupath = 0.;
            pk.tauCached = 0.;
            pk.Wp = 0.;
            pk.pix = -1;
            pk.hint = startHint;
            pk.haveTau = false;
            if (!(pk.W / pk.lam > 0))
            {
                finish();
                return false;
            }
            pk.Lthr = (pk.W / pk.lam) / p.min_weight_reduction;
            begin_peel(false);
            return true;
        }

        __device__ __forceinline__ void begin_peel(bool scattering)
        {
            pk.scat = scattering;
            pk.f = (INST ? p.inst[pk.inst].fbeg : 0) - 1;
        }

        // peel-off toward each instrument in turn (MonteCarloSimulation.cpp:698-715, :2034-2092;
        // FluxRecorder::detect skips the optical depth for packets outside the frame, :375)
        __device__ __forceinline__ void next_peel()
        {
            int fb = 0, fe = p.nframes;
            if constexpr (INST)
            {
                fb = p.inst[pk.inst].fbeg;
                fe = p.inst[pk.inst].fend;
            }
            while (++pk.f < fe)
            {
                const FrameGeom& fg = p.frames[pk.f];
                if constexpr (V == kPersp || V == kStoreRF)
                {
                    if (fg.persp)
                    {
                        // PerspectiveInstrument: toward the eye from this position
                        // (PerspectiveInstrument.cpp:93-101), luminosity / zp^2 and the
                        // optical depth over the path length zp (FluxRecorder.cpp:372-405)
                        double zp;
                        pk.pix = fg.persp_pixel(pk.rx, pk.ry, pk.rz, zp);
                        const double dx = fg.eye[0] - pk.rx, dy = fg.eye[1] - pk.ry, dz = fg.eye[2] - pk.rz;
                        const double D = sqrt(dx * dx + dy * dy + dz * dz);
                        const double ox = dx / D, oy = dy / D, oz = dz / D;
                        if (!fg.same_as_prev || pk.f == fb)
                        {
                            pk.haveTau = false;
                            pk.Wp = pk.W;
                            if (pk.scat) pk.Wp = pk.W * peel_phase(p.gpar[pk.ell], pk.kx * ox + pk.ky * oy + pk.kz * oz);
                        }
                        if (pk.pix < 0) continue;
                        const double L = pk.Wp / pk.lam;
                        if (pk.haveTau)
                        {
                            deposit(fg, L / (zp * zp), pk.tauCached);
                            continue;
                        }
                        if (L <= 0)
                        {
                            pk.haveTau = true;
                            pk.tauCached = INFINITY;
                            continue;
                        }
                        peel(ox, oy, oz, L);
                        io.slim = zp;
                        return;
                    }
                }
                if (!fg.same_as_prev || pk.f == fb)
                {
                    pk.haveTau = false;
                    pk.Wp = pk.W;
                    if (pk.scat)
                    {
                        double c = pk.kx * fg.kobs[0] + pk.ky * fg.kobs[1] + pk.kz * fg.kobs[2];
                        pk.Wp = pk.W * peel_phase(p.gpar[pk.ell], c);
                    }
                }
                pk.pix = fg.pixel(pk.rx, pk.ry, pk.rz);
                if (pk.pix < 0) continue;
                double L = pk.Wp / pk.lam;
                if (pk.haveTau)
                {
                    deposit(fg, L, pk.tauCached);
                    continue;
                }
                if (L <= 0)
                {
                    pk.haveTau = true;
                    pk.tauCached = INFINITY;
                    continue;
                }
                peel(fg.kobs[0], fg.kobs[1], fg.kobs[2], L);
                return;
            }
            // all instruments done: scatter (after a scattering peel-off) and start a forced path
            if (pk.scat)
            {
                if constexpr (V == kGuided)
                {
                    // the wave's guided scattering round follows (guided_scatter)
                    io.phase = kScatter;
                    return;
                }
                if (p.contKey != 0u && pk.nscatt == 0) pk.rng.retag(p.contKey);
                scatter_hg(pk.rng, p.gpar[pk.ell], pk.kx, pk.ky, pk.kz);
                pk.nscatt++;
                lds_count(lds + 3);
            }
            forced();
        }

        // Guided scattering with the network outputs o of this packet's event: a direction from
        // the defensive mixture (1 - mix) HG + mix guide, and the weight factor
        // Phi_HG / p_mix that keeps the estimator unbiased.  The termination threshold takes the
        // same factor, so the rule (MonteCarloSimulation.cpp:643-660) applies to the weight
        // without the guide's factors (packets the guide down-weights are not cut early).
        __device__ __forceinline__ void guided_scatter(const float* o)
        {
            if (p.contKey != 0u && pk.nscatt == 0) pk.rng.retag(p.contKey);
            const double ratio = guided_direction(o, p.gpar[pk.ell], p.guideMix, pk.rng, pk.kx, pk.ky, pk.kz);
            pk.W *= ratio;
            pk.Lthr *= ratio;
            pk.nscatt++;
            lds_count(lds + 3);
            forced();
        }

        // event handling once a traversal ended; true when the packet peels off next
        __device__ __forceinline__ bool transition(int phase, int last, double tau, double s)
        {
            if (phase == kPeel)
            {
                pk.haveTau = true;
                pk.tauCached = tau;
                const FrameGeom& fg = p.frames[pk.f];
                double L = pk.Wp / pk.lam;
                if constexpr (V == kPersp || V == kStoreRF)
                {
                    if (fg.persp)
                    {
                        double zp;
                        fg.persp_pixel(pk.rx, pk.ry, pk.rz, zp);
                        L /= zp * zp;
                    }
                }
                deposit(fg, L, pk.tauCached);
                return true;
            }
            if (phase == kFwd1)
            {
                // MonteCarloSimulation::simulateForcedPropagation (:1492-1544)
                pk.taupath = tau;
                if (pk.taupath <= 0.)
                {
                    pk.W *= 0.;
                    finish();
                    return false;
                }
                double xi = p.xi;
                double tint;
                if (xi == 0.)
                    tint = expon_cutoff(pk.rng, pk.taupath);
                else
                {
                    tint = pk.rng.uniform() < xi ? pk.rng.uniform() * pk.taupath : expon_cutoff(pk.rng, pk.taupath);
                    double pp = -exp(-tint) / expm1(-pk.taupath);
                    double q = (1.0 - xi) * pp + xi / pk.taupath;
                    pk.W *= pp / q;
                }
                lds_count(lds + 6);
                travel(pk.kx, pk.ky, pk.kz, kFwd2, tint);
                return false;
            }
            // the second pass: SpatialGridPath::findInteractionPoint (SpatialGridPath.cpp:161-203):
            // the interaction's cell and distance, or beyond the last segment that segment's
            const int m = last;
            double n = 0.;
            if (m >= 0)
                n = GT == kOctree    ? p.grid.node[m].dens
                    : GT == kVoronoi ? reinterpret_cast<const VorHead*>(p.grid.vnb + m)->dens
                                     : p.dens[m];
            double ss = INST ? p.ssca[pk.ell] * p.inst[pk.inst].scale : p.ssca[pk.ell];
            double se = INST ? p.sext[pk.ell] * p.inst[pk.inst].scale : p.sext[pk.ell];
            double ksca = n > 0. ? n * ss : 0.;
            double kext = n > 0. ? n * se : 0.;
            double albedo = kext > 0. ? ksca / kext : 0.;
            pk.W *= -expm1(-pk.taupath) * albedo;
            pk.hint = GT == kCartesian ? -1 : m;  // the interaction point lies in the cell of its segment
            pk.rx += s * pk.kx;
            pk.ry += s * pk.ky;
            pk.rz += s * pk.kz;
            double L = pk.W / pk.lam;
            if (L <= 0 || (L <= pk.Lthr && pk.nscatt >= p.min_scatt) || pk.nscatt >= kMaxScatterings)
            {
                finish();
                return false;
            }
            begin_peel(true);
            return true;
        }
    };

    // The kernel's parameter block, passed to a function in vector registers, as the uniform
    // address it is: its fields are then read with scalar loads
    __device__ __forceinline__ const SimParams& uniform_params(const SimParams* q)
    {
        const uint64_t a = reinterpret_cast<uint64_t>(q);
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
        const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
        typedef const __attribute__((address_space(4))) SimParams* KernargPtr;
        return *(const SimParams*)(KernargPtr)(static_cast<uint64_t>(hi) << 32 | lo);
    }

    // One event of one packet: the launch of history `hist` (phase kFetch) or what follows the
    // traversal of phase `phase` that ended with optical depth tau, cell `last` and distance s, up to
    // the packet's next traversal, its end, or (guided) the wait for the network.  A call of its
    // own, with the packet in LDS: its FP64 transcendentals need far more registers than the
    // crossing loop, and inlined they spilled the loop's traversal state.
    template<int GT, int V>
    __device__ __attribute__((noinline)) void life_event(const SimParams* params, int phase, int last, double tau, double s,
                                                         uint64_t hist, EventOut& out, LdsF64* cd, LdsU32* cu, LdsU32* lds,
                                                         int t)
    {
        const SimParams& p = uniform_params(params);
        EventOut io;
        io.off = -1;
        Packet pk;
        Events<GT, V> E{p, io, pk, lds};
        bool peels;
        if (phase == kFetch)
            peels = E.launch(hist);
        else
        {
            pk.template load<V == kBatched>(cd, cu, t, p);
            peels = E.transition(phase, last, tau, s);
        }
        if (peels) E.next_peel();
        pk.store(cd, cu, t);
        out = io;
    }

    // The guided scattering of one packet from the network outputs o (guided_scatter), likewise.
    template<int GT>
    __device__ __attribute__((noinline)) void life_guided(const SimParams* params, const float* o, EventOut& out,
                                                          LdsF64* cd, LdsU32* cu, LdsU32* lds, int t)
    {
        const SimParams& p = uniform_params(params);
        EventOut io;
        io.off = -1;
        Packet pk;
        pk.template load<false>(cd, cu, t, p);
        Events<GT, kGuided> E{p, io, pk, lds};
        E.guided_scatter(o);
        pk.store(cd, cu, t);
        out = io;
    }

    __device__ __forceinline__ int lane_id() { return __lane_id(); }

    // Minimum waves per SIMD, with the measured alternatives (ms at 2 / 3 / 4 waves):
    //   Cartesian 64^3, 2^21 packets               23.2 / 22.5 / 21.8
    //   Cartesian 44^3, 2e5 packets                 3.3 /  3.3 /  3.6 (one packet per lane)
    //   octree disk, ten levels, tau_V 50, 2^21    50.1 / 43.3 / 46.0 (at four, spills around the
    //   octree, nine levels, 40 wavelengths, 3e5    8.4 /  8.4 /  8.1  events double the writes)
    //   octree with the radiation field, 2e5        7.8 / 11.6 / 13.2 (bound by its atomics, whose
    //   Cartesian with the field, 7e5              targets collide more with more waves)
    //   Voronoi, 400 000 sites, 2^18 packets       39.9 / 39.6 / 44.4
    //   tetra, 150 000 vertices, 64 instances, 2^20   - / 61.2 / 57.8
    // The guided variant's network call holds whole layers' weights in registers, and its four-wave build does not compile for the mesh grids.
    template<int GT, int V> constexpr int lifecycle_waves()
    {
        return V == kGuided || V == kStoreRF ? 2 : GT == kOctree ? 3 : GT == kTetra ? 4 : 3;
    }

    // The kernel's parameter block where it lies in the kernarg segment, behind a pointer the
    // compiler cannot see through: fields read through the returned reference are loaded again
    // (scalar loads through the constant cache) instead of being held in registers across the
    // whole loop, which keeps the register pressure of the uniform values down.
    __device__ __forceinline__ const SimParams& kernel_params()
    {
        typedef const __attribute__((address_space(4))) SimParams* KernargPtr;
        KernargPtr q = (KernargPtr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(q));
        return *(const SimParams*)q;
    }

    template<int GT, int FP, int V, int L>
    __global__ void __launch_bounds__(kLcThreads, (lifecycle_waves<GT, V>())) lifecycle(SimParams p)
    {
        constexpr bool PERSP = V == kPersp || V == kStoreRF;
        __shared__ uint32_t wgcnt[kNumCounters];
        __shared__ double coldD[kColdF64 * kLcThreads];
        __shared__ uint32_t coldU[kColdU32 * kLcThreads];
        LdsF64* const cd = (LdsF64*)coldD;
        LdsU32* const cu = (LdsU32*)coldU;
        LdsU32* const cnt = (LdsU32*)wgcnt;
        if (threadIdx.x < kNumCounters) wgcnt[threadIdx.x] = 0;
        stage_planes<GT>(p.grid);
        __syncthreads();  // the counters are zero before any wave adds to them
        const int t = threadIdx.x / L;
        const int lane = lane_id();
        const bool lead = Trav<GT, FP, L>::lead();
        Trav<GT, FP, L> T;
        // the lanes that take packets (all of them unless the run is small); a lane without one
        // waits in kFetch
        T.phase = lane / L < p.lanes ? kFetch : kDone;
        T.ended = false;
        T.gen.idle();
        T.last = -1;
        T.tau = T.s = T.lim = 0.;
        T.tau32.reset();
        T.s32.reset();
        bool busy = false;  // the lane's traversal is under way
        while (true)
        {
            // A transition round of the wave: events for the lanes whose traversal ended, new
            // histories, the traversals that follow.
            {
                const SimParams& kp = kernel_params();
                EventOut io;
                int64_t off = -1;  // this round's deposit
                double v = 0.;
                uint64_t hist = 0;
                bool event = T.ended, go = false;
                // new histories for the lanes without one, with one atomic per wavefront
                const unsigned long long need = __ballot(T.phase == kFetch && lead);
                if (need)
                {
                    const int leader = __ffsll(static_cast<long long>(need)) - 1;
                    unsigned long long base = 0;
                    if (lane == leader) base = atomicAdd(kp.queue, static_cast<unsigned long long>(__popcll(need)));
                    base = __shfl(base, leader);
                    if (T.phase == kFetch)
                    {
                        const unsigned long long mine = base + __popcll(need & ((1ull << (lane & -L)) - 1ull));
                        hist = kp.first + mine;
                        event = mine < kp.count;
                        if (!event) T.phase = kDone;
                    }
                }
                if (event)
                {
                    if (lead)
                    {
                        life_event<GT, V>(&kp, T.phase, T.last, T.tau_value(), T.s_end(T.tau_value() > T.lim), hist, io, cd,
                                          cu, cnt, t);
                        off = io.off;
                        v = io.v;
                    }
                    io.template share<L, V>();
                    T.phase = io.phase;
                    T.ended = false;
                    go = io.phase == kPeel || io.phase == kFwd1 || io.phase == kFwd2;
                }
                if constexpr (V == kGuided)
                {
                    // one network evaluation for the lanes of the wave that wait to scatter, once
                    // there are kGuideLanes of them or no lane of the wave is still traversing
                    const bool sc = T.phase == kScatter && lead;
                    const unsigned long long scm = __ballot(sc);
                    if (scm && (__popcll(scm) >= kGuideLanes / L || __ballot(go || busy) == 0))
                    {
                        float feat[kGuideIn];
                        for (int q = 0; q < kGuideIn; ++q) feat[q] = 0.f;
                        if (sc)
                            guide_features(kp.gframe, cd[cRx * kLcThreads + t], cd[cRy * kLcThreads + t],
                                           cd[cRz * kLcThreads + t], cd[cKx * kLcThreads + t], cd[cKy * kLcThreads + t],
                                           cd[cKz * kLcThreads + t], cd[cLam * kLcThreads + t], feat);
                        float o[kGuideOut];
                        guide_wave_infer_regs(kp.net, feat, sc, o);
                        if (T.phase == kScatter)
                        {
                            if (sc) life_guided<GT>(&kp, o, io, cd, cu, cnt, t);
                            io.template share<L, V>();
                            T.phase = io.phase;
                            go = true;
                        }
                    }
                }
                flush_deposits(kp.frame, off, v, cnt);  // the wave is converged here
                if (!go && T.gen.asks() && !T.ended)
                {
                    T.gen.resolve(kp.grid);
                    busy = true;
                }
                if (go)
                {
                    T.template start<PERSP>(kp.grid, io, cd, cu, cnt, t);
                    busy = !T.ended;
                }
            }
            // Crossings until enough lanes wait for a round.  The threshold is a share of the lanes
            // that still take part: in a small run, and at the end of every run, a fixed number of
            // waiting lanes would never come together and each packet would wait for the longest
            // traversal of the wave.  Guided: the lanes that wait for the network do not count as
            // waiting (they call no round with few events to handle).  A loop of its own, so that
            // the registers' spills lie outside it.
            const SimParams& sp = kernel_params();
            const int nact = __popcll(__ballot(T.phase != kDone));
            if (nact == 0) break;
            const int nscat = V == kGuided ? __popcll(__ballot(T.phase == kScatter)) : 0;
            const int stop = max(0, nact - nscat - ((sp.threshold * nact + 63) >> 6));
            while (__popcll(__ballot(busy)) > stop)
            {
                if (busy)
                {
                    T.template step<V == kStoreRF, PERSP>(kernel_params().grid, cnt, kernel_params().rf, kernel_params().nlambda);
                    busy = !T.ended && !T.gen.asks();
                }
            }
        }
        // workgroup event counters to the global counters
        __syncthreads();
        if (threadIdx.x < kNumCounters && wgcnt[threadIdx.x])
            atomicAdd(p.counters + threadIdx.x, static_cast<unsigned long long>(wgcnt[threadIdx.x]));
    }
}
