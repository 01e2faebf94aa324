// sg_split.hpp -- the photon-packet life cycle (MonteCarloSimulation::dostellaremissionchunk,
// MonteCarloSimulation.cpp:259-297) as two alternating kernels over device-resident queues:
//
//   k_events: one thread per in-flight packet slot runs the packet's state machine from the end of
//             its propagation (or its launch) to its next own path -- launch, peel-offs, the new
//             direction -- and appends the walks it needs (peel-offs and the own path) to the queue;
//   k_walks:  persistent lanes take walk requests from the queue and run the cell walks, with the
//             same ballot-compacted refill as the lane pipeline; a peel-off walk ends with its
//             detection (FrameInstrument::detect); a lane that ends an own path draws the packet's
//             escape, absorption, stop test and biased path length, and walks on to the interaction
//             point itself (own_path_end), whose place goes to the packet slot.
//
// The walk kernel carries only the walker and the running sums, so it keeps several times more
// waves in flight than a kernel that also holds the event logic; the event kernel's FP64 and libm
// work runs at full width over the slots. Each packet still draws from its own Philox stream in the
// same order, and every walk repeats the same arithmetic, so results equal the lane pipeline's up
// to the order of the tally additions.
#pragma once
#include "sg_mc.hpp"

namespace sg {

enum SlotR { SR_RX = 0, SR_RY, SR_RZ, SR_KX, SR_KY, SR_KZ, SR_L, SR_RES, SR_NR };
// SU_MCELL: several dust components: the cell of the interaction point (-1: none).
// SU_HINT: the leaf (tree node, or Voronoi cell) the packet's position lies in, as the last
// propagation walk left it (-1: unknown), handed to the walks that start there.
enum SlotU { SU_PLO = 0, SU_PHI, SU_DRAW, SU_W0, SU_W1, SU_W2, SU_W3, SU_NSCATT, SU_HINT,
             SU_MCELL, SU_STATE, SU_NU };
// PS_OWN: the packet's own path is in the walk queue; the walk kernel leaves it at its interaction point
// (PS_PROP) or finished (PS_FRESH: the slot takes a new packet).
enum PacketState : uint32_t { PS_FRESH = 0, PS_OWN, PS_PROP, PS_DEAD };
enum WalkKind : uint32_t { WK_PEEL = 0, WK_OWN = 1 };

// Packet slots: structure of arrays, n slots.
template <typename R> struct Slots {
    R* r;
    uint32_t* u;
    int64_t n;
    __device__ __forceinline__ R& fr(int f, int64_t i) const { return r[f * n + i]; }
    __device__ __forceinline__ uint32_t& fu(int f, int64_t i) const { return u[f * n + i]; }
};
template <typename R> __host__ __device__ constexpr size_t slot_bytes(int64_t n)
{
    return (size_t)n * (SR_NR * sizeof(R) + SU_NU * sizeof(uint32_t));
}

// Walk requests: origin (3), direction (3, unused for peel-offs: the instrument's direction is
// taken from its record) and a value (peel-off or own-path luminosity) in the run's real type; a tag
// (kind | instrument << 2), an index (packet slot, or pixel for a peel-off) and the start cell hint of the
// walker. One record per request, so that a request moved to its sorted place, or read by a lane, is one
// contiguous block.
template <typename R> struct alignas(16) WalkReq {
    R o[3], d[3], val;
    uint32_t tag, idx, hint;
};
static_assert(sizeof(WalkReq<float>) == 48 && sizeof(WalkReq<double>) == 80, "walk request records");

constexpr int kXcdSegs = 8;
// Progress of one pass of a slot group. A group's passes use a ring of these records; the event kernel of
// a pass clears the next one, so that no fill runs between the kernels.
struct PassCtl {
    unsigned long long tail;            // requests appended by the event kernel
    unsigned long long claim;           // requests taken by the walk kernel
    unsigned long long seg[kXcdSegs];   // the same per XCD segment
    unsigned long long t0;              // walk kernel: its start (clock ticks; 0: it had no requests)
};
constexpr int kPassRing = 4;
struct GroupCtl {
    PassCtl pass[kPassRing];
    unsigned long long ticks;           // walk kernels' durations, summed over the finished passes
    unsigned long long start;           // the first pass's start (clock ticks)
};
// What each wave of the walk kernel keeps from pass to pass in a record of its own: the end of its last pass
// (clock ticks) and its counts. (Added up with atomics at the end of every pass, on one cache line at about 10 ns
// each, they took 100 us of it.)
struct WaveRec {
    unsigned long long t1, own, peel, re, stuck, recompute;
};
// A group's count records, added up at the end of a run.
struct GroupTally {
    WaveRec* waves;                     // per wave of the walk kernel
    int nwaves;
    unsigned long long* events;         // per workgroup of the event kernel: packets, scatterings, peel-offs, walks
    int64_t nevents;
    int64_t slot0;                      // the group's first slot among all groups' (its first packet in a batch)
};

// Walk order. The walks of a pass are sorted by a coherence key before the walk kernel takes them:
// peel-offs by instrument and the Morton order of their pixel (rays toward one instrument through
// neighbouring pixels cross the same cells), own paths by the Morton order of their start point. Lanes and waves that run at the same time then touch a small part of the grid,
// which the L2 cache of their XCD holds. A counting sort: the event kernel counts each request into
// its key's bin and keeps its rank there, a one-block scan turns the counts into bin offsets (and
// clears them), and a scatter moves each request to offset + rank. Histories do not depend on the
// order (only the order of the tally additions changes).
constexpr int kKeyBits = 16;
constexpr uint32_t kKeyBins = 1u << kKeyBits;
template <typename R> struct WalkQueue {
    WalkReq<R>* req;            // requests in the order the event kernel appended them
    WalkReq<R>* sorted;         // the same in key order (null: the walk kernel reads req)
    uint32_t* key;              // per request: its bin, and its rank within the bin
    uint32_t* rank;
    uint32_t* hist;             // kKeyBins counts (zero between passes; a buffer of its own, cleared once)
    uint32_t* off;              // kKeyBins bin offsets
    int64_t cap;
    unsigned long long* tail;   // requests appended by the event kernel
};
// requests, sorted requests, keys and ranks (the bin counts and offsets are held apart)
template <typename R> __host__ __device__ constexpr size_t queue_bytes(int64_t cap, bool sort)
{
    return (size_t)cap * sizeof(WalkReq<R>) * (sort ? 2 : 1) + (sort ? (size_t)cap * 8 : 0);
}

// 2-D and 3-D Morton codes (bit interleaving) of small integer coordinates.
__device__ __forceinline__ uint32_t spread2(uint32_t v)   // 8 bits -> every second bit
{
    v &= 0xffu;
    v = (v | (v << 4)) & 0x0f0fu;
    v = (v | (v << 2)) & 0x3333u;
    v = (v | (v << 1)) & 0x5555u;
    return v;
}
__device__ __forceinline__ uint32_t spread3(uint32_t v)   // 5 bits -> every third bit
{
    v &= 0x1fu;
    v = (v | (v << 8)) & 0x100fu;
    v = (v | (v << 4)) & 0x10c3u;
    v = (v | (v << 2)) & 0x1249u;
    return v;
}
// The coherence key of a request: 4 bits of class (peel-off instrument 0-7, own path 8) above 12 bits of Morton order (a peel-off's pixel on a 64 x 64 raster of its frame; a start
// point on a 16 x 16 x 16 raster of the grid box).
template <typename R>
__device__ __forceinline__ uint32_t walk_key(const McArgs& a, const InstrDev* instr, uint32_t tag, uint32_t idx, R ox,
                                             R oy, R oz)
{
    const uint32_t kind = tag & 3u;
    if (kind == WK_PEEL) {
        const InstrDev& in = instr[tag >> 2];
        const uint32_t i = idx % (uint32_t)in.Nx, j = idx / (uint32_t)in.Nx;
        const uint32_t qi = (uint32_t)(((uint64_t)i << 6) / (uint32_t)in.Nx);
        const uint32_t qj = (uint32_t)(((uint64_t)j << 6) / (uint32_t)in.Ny);
        return ((tag >> 2) << 12) | spread2(qi) | (spread2(qj) << 1);
    }
    auto q = [](double v, double lo, double sc) {
        const double t = (v - lo) * sc;
        return (uint32_t)(!(t > 0.0) ? 0.0 : t > 15.0 ? 15.0 : t);   // NaN to 0
    };
    const uint32_t qx = q((double)ox, a.key_lo[0], a.key_scale[0]);
    const uint32_t qy = q((double)oy, a.key_lo[1], a.key_scale[1]);
    const uint32_t qz = q((double)oz, a.key_lo[2], a.key_scale[2]);
    return (8u << 12) | spread3(qx) | (spread3(qy) << 1) | (spread3(qz) << 2);
}

// An instrument as the event kernel uses it, in the run's real type: pixel_on_detector's products of two angle
// functions taken once.
template <typename R> struct EventInstr {
    R sinphi, cosphi, c1, c2, sintheta, cospa, sinpa, xpmin, xpsiz, ypmin, ypsiz, k[3];
    int Nx, Ny;
    double* frame;
};
template <typename R> __device__ __forceinline__ EventInstr<R> event_instr(const InstrDev& in)
{
    EventInstr<R> e;
    e.sinphi = (R)in.sinphi; e.cosphi = (R)in.cosphi;
    e.c1 = -(R)in.cosphi * (R)in.costheta; e.c2 = (R)in.sinphi * (R)in.costheta; e.sintheta = (R)in.sintheta;
    e.cospa = (R)in.cospa; e.sinpa = (R)in.sinpa;
    e.xpmin = (R)in.xpmin; e.xpsiz = (R)in.xpsiz; e.ypmin = (R)in.ypmin; e.ypsiz = (R)in.ypsiz;
    for (int a = 0; a < 3; a++) e.k[a] = (R)in.kobs[a];
    e.Nx = in.Nx; e.Ny = in.Ny; e.frame = in.frame;
    return e;
}
// SingleFrameInstrument::pixelondetector (SingleFrameInstrument.cpp:130-147), operation for operation as
// pixel_on_detector
template <typename R> __device__ __forceinline__ int event_pixel(const EventInstr<R>& in, R x, R y, R z)
{
    const R xpp = -in.sinphi * x + in.cosphi * y;
    const R ypp = in.c1 * x - in.c2 * y + in.sintheta * z;
    const R xp = in.cospa * xpp - in.sinpa * ypp;
    const R yp = in.sinpa * xpp + in.cospa * ypp;
    const R fi = floor((xp - in.xpmin) / in.xpsiz);
    const R fj = floor((yp - in.ypmin) / in.ypsiz);
    if (!(fi >= (R)0 && fi < (R)in.Nx && fj >= (R)0 && fj < (R)in.Ny)) return -1;
    return (int)fi + in.Nx * (int)fj;
}

// Henyey-Greenstein scattering direction (DustMix.cpp:596-601) and Random::direction(k, cos)
// (Random.cpp:189-223).
template <typename R>
__device__ __forceinline__ void hg_scatter(PacketRng& rng, R gg, R& kx, R& ky, R& kz)
{
    R nkx, nky, nkz;
    if (fabs((double)gg) < 1e-6) {
        double a0, a1, a2;
        iso_direction(rng, a0, a1, a2);
        nkx = (R)a0; nky = (R)a1; nkz = (R)a2;
    } else {
        R f = (((R)1.0 - gg) * ((R)1.0 + gg)) / ((R)1.0 - gg + (R)2.0 * gg * uni<R>(rng));
        R costheta = ((R)1.0 + gg * gg - f * f) / ((R)2.0 * gg);
        R phi = (R)(2.0 * M_PI) * uni<R>(rng);
        R cosphi = cos(phi), sinphi = sin(phi);
        R sintheta = sqrt(fabs(((R)1.0 - costheta) * ((R)1.0 + costheta)));
        if (kz > (R)0.99999) { nkx = cosphi * sintheta; nky = sinphi * sintheta; nkz = costheta; }
        else if (kz < (R)-0.99999) { nkx = cosphi * sintheta; nky = sinphi * sintheta; nkz = -costheta; }
        else {
            R root = sqrt(((R)1.0 - kz) * ((R)1.0 + kz));
            nkx = sintheta / root * (-kx * kz * cosphi + ky * sinphi) + kx * costheta;
            nky = -sintheta / root * (ky * kz * cosphi + kx * sinphi) + ky * costheta;
            nkz = root * sintheta * cosphi + kz * costheta;
        }
    }
    kx = nkx; ky = nky; kz = nkz;
}

// A launched packet's state and random stream, which continues where the emission left it; false when every
// packet has been claimed (*p then not set), or for a packet without luminosity.
template <typename R>
__device__ __forceinline__ bool take_packet(const McArgs& a, uint64_t p, PacketRng& rng, R& rx, R& ry, R& rz, R& kx, R& ky,
                                            R& kz, R& L, int32_t& hint)
{
    const R* e = reinterpret_cast<const R*>(a.emitted);
    const size_t n = a.count;
    L = e[6 * n + p];
    if (!(L > (R)0)) return false;
    rx = e[p]; ry = e[n + p]; rz = e[2 * n + p];
    kx = e[3 * n + p]; ky = e[4 * n + p]; kz = e[5 * n + p];
    rng.start(a.seed, a.member, a.first + p, a.ell);
    rng.draw = a.emit_draw[p];
    if (rng.draw & 3u) {
        rng.w0 = rng.plo; rng.w1 = rng.phi; rng.w2 = rng.draw >> 2; rng.w3 = rng.ell;
        philox10(rng.w0, rng.w1, rng.w2, rng.w3, rng.k0, rng.k1);
    }
    hint = a.emit_hint ? a.emit_hint[p] : -1;
    return true;
}

// Event pass: every slot advances its packet to its next own path (or takes a new packet): peel-offs toward every
// instrument (MonteCarloSimulation::peeloffemission/peeloffscattering, MonteCarloSimulation.cpp:299-357), the
// scattered direction, and the requests for their walks. The requests are counted first (one ballot per kind and
// wave), the workgroup takes its part of the queue with one atomic, and each lane writes its own requests, so
// that only the counts pass through LDS: staged whole there (51 KB a workgroup in FP64) they left three workgroups
// on a CU. Within the workgroup's part the requests lie instrument by instrument, own paths last: neighbours in
// the queue walk in the same direction. gc/pass: the group's progress ring; this pass's record is q.tail's.
// The device adds to one address about once in 10 ns, so atomics are few: one per workgroup for its part of the
// queue, and one per wave that needs packets while there are unclaimed ones, none in a batch's first pass (`first`:
// every slot is free and takes the packet of its own number, slot0 + i).
constexpr int kEventBlock = 512;
template <typename R, bool MULTI>
__global__ void __launch_bounds__(kEventBlock) k_events(const McArgs a, Slots<R> sl, WalkQueue<R> q, GroupCtl* gc, int pass,
                                                        int first, const GroupTally ta)
{
    constexpr int kKinds = SG_MAX_INSTR + 1, nw = kEventBlock / 64;
    __shared__ EventInstr<R> s_instr[SG_MAX_INSTR];
    __shared__ uint32_t s_n[kKinds * nw];                 // requests per kind and wave, then their places in the part
    __shared__ uint32_t s_stat[4 * nw];
    __shared__ unsigned long long s_base;
    const int wave = (int)threadIdx.x >> 6, lane = __lane_id();
    if ((int)threadIdx.x < a.ni) s_instr[threadIdx.x] = event_instr<R>(a.scene->instr[threadIdx.x]);
    if (blockIdx.x == gridDim.x - 1) {
        // a workgroup of its own for the bookkeeping. The previous pass's walk kernel has ended: its duration, from
        // its start to its last wave's end; the next pass's record, last used three passes ago, is cleared
        const PassCtl& pv = gc->pass[(pass + kPassRing - 1) % kPassRing];
        if (threadIdx.x == 0) {
            s_base = 0;
            if (pass == 0) gc->start = wall_clock64();
            PassCtl& nx = gc->pass[(pass + 1) % kPassRing];
            nx.tail = 0; nx.claim = 0; nx.t0 = 0;
            for (int k = 0; k < kXcdSegs; k++) nx.seg[k] = 0;
        }
        __syncthreads();
        unsigned long long t1 = 0;
        for (int w = (int)threadIdx.x; w < ta.nwaves; w += kEventBlock) t1 = max(t1, ta.waves[w].t1);
        atomicMax(&s_base, t1);
        __syncthreads();
        if (threadIdx.x == 0 && pv.t0 && s_base > pv.t0) gc->ticks += s_base - pv.t0;
        return;
    }
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t state0 = i < sl.n ? sl.fu(SU_STATE, i) : (uint32_t)PS_DEAD;
    uint32_t state = state0;
    R rx = 0, ry = 0, rz = 0, kx = 0, ky = 0, kz = 0, L = 0;
    int32_t hint = -1;
    PacketRng rng;
    rng.k0 = a.seed; rng.k1 = a.member; rng.ell = (uint32_t)a.ell;
    rng.plo = 0; rng.phi = 0; rng.draw = 0; rng.w0 = 0; rng.w1 = 0; rng.w2 = 0; rng.w3 = 0;
    uint32_t c_pk = 0, c_peel = 0;   // wave totals
    bool acts = false;               // the lane makes peel-offs and requests an own path
    const bool scatters = state0 == PS_PROP;
    int mcell = -1;
    if (scatters) {
        // PhotonPackage::propagate (PhotonPackage.cpp:93-96) by pathlength(tau)
        const R d = sl.fr(SR_RES, i);
        kx = sl.fr(SR_KX, i); ky = sl.fr(SR_KY, i); kz = sl.fr(SR_KZ, i);
        rx = sl.fr(SR_RX, i) + d * kx; ry = sl.fr(SR_RY, i) + d * ky; rz = sl.fr(SR_RZ, i) + d * kz;
        L = sl.fr(SR_L, i);
        rng.plo = sl.fu(SU_PLO, i); rng.phi = sl.fu(SU_PHI, i); rng.draw = sl.fu(SU_DRAW, i);
        rng.w0 = sl.fu(SU_W0, i); rng.w1 = sl.fu(SU_W1, i); rng.w2 = sl.fu(SU_W2, i); rng.w3 = sl.fu(SU_W3, i);
        hint = (int32_t)sl.fu(SU_HINT, i);
        if (MULTI) mcell = (int)sl.fu(SU_MCELL, i);
        acts = true;
    }
    // without a dust system the peel-offs are detected here, and a slot takes up to four packets per pass
    for (int turn = 0; turn < (a.has_dust ? 1 : 4); turn++) {
        uint64_t p = 0;
        bool got = false;
        if (state == PS_FRESH) {
            if (first && turn == 0) {
                p = (uint64_t)(ta.slot0 + i);
                got = p < a.count;
            } else if (__hip_atomic_load(a.next_packet, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < a.count)
                got = wave_claim(a.next_packet, a.count, p);
            if (!got) state = PS_DEAD;
        }
        c_pk += (uint32_t)__popcll(__ballot(got));
        const bool lit = got && take_packet<R>(a, p, rng, rx, ry, rz, kx, ky, kz, L, hint);
        if (a.has_dust) {
            acts = acts | lit;
            break;
        }
        for (int k = 0; k < a.ni; k++) {
            const int pix = lit ? event_pixel<R>(s_instr[k], rx, ry, rz) : -1;
            if (pix >= 0) unsafeAtomicAdd(s_instr[k].frame + (size_t)a.ell * s_instr[k].Nx * s_instr[k].Ny + pix, (double)L);
            c_peel += (uint32_t)__popcll(__ballot(pix >= 0));
        }
    }
    // peel-off pixels and luminosities (the phase-function weight of a scattering)
    int pix[SG_MAX_INSTR];
    R Lp[SG_MAX_INSTR];
    const R gg = (R)a.g;
    // peeloffscattering aborts when the scattering point has no scattering dust (MonteCarloSimulation.cpp:321-327)
    const bool peels = acts && !(MULTI && scatters && !peel_weights_ok<R>(a, mcell));
#pragma unroll
    for (int k = 0; k < SG_MAX_INSTR; k++) {
        pix[k] = -1;
        Lp[k] = L;
        if (k >= a.ni) continue;   // the same for every lane
        if (peels) {
            const EventInstr<R>& in = s_instr[k];
            pix[k] = event_pixel<R>(in, rx, ry, rz);
            if (scatters) {
                // DustMix::phaseFunctionValue, Henyey-Greenstein (DustMix.cpp:648-653)
                const R cosalpha = kx * in.k[0] + ky * in.k[1] + kz * in.k[2];
                if (MULTI) Lp[k] = L * mixed_phase<R>(a, mcell, cosalpha);
                else {
                    const R t = (R)1.0 + gg * gg - (R)2 * gg * cosalpha;
                    Lp[k] = L * (((R)1.0 - gg) * ((R)1.0 + gg) / sqrt(t * t * t));
                }
            }
        }
        const uint32_t n = (uint32_t)__popcll(__ballot(pix[k] >= 0));
        c_peel += n;
        if (lane == 0) s_n[k * nw + wave] = n;
    }
    const uint64_t own = __ballot(acts), scattered = __ballot(scatters);
    if (lane == 0) {
        s_n[a.ni * nw + wave] = (uint32_t)__popcll(own);
        s_stat[wave] = c_pk;
        s_stat[nw + wave] = (uint32_t)__popcll(scattered);
        s_stat[2 * nw + wave] = c_peel;
        s_stat[3 * nw + wave] = a.has_dust ? c_peel + (uint32_t)__popcll(own) : 0u;
    }
    __syncthreads();
    // places of the (kind, wave) runs in the workgroup's part of the queue, kind by kind
    const int runs = (a.ni + 1) * nw;
    static_assert(kKinds * nw <= 128, "two runs per lane");
    if (wave == 0) {
        const bool dust = a.has_dust != 0;
        const uint32_t n0 = dust && 2 * lane < runs ? s_n[2 * lane] : 0u;
        const uint32_t n1 = dust && 2 * lane + 1 < runs ? s_n[2 * lane + 1] : 0u;
        uint32_t x = n0 + n1;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (2 * lane < runs) s_n[2 * lane] = x - n0 - n1;
        if (2 * lane + 1 < runs) s_n[2 * lane + 1] = x - n1;
        if (lane == 63) s_base = x ? atomicAdd(q.tail, (unsigned long long)x) : 0ull;
    }
    if (threadIdx.x >= 64 && threadIdx.x < 68) {
        const int k = (int)threadIdx.x & 3;
        unsigned long long t = 0;
        for (int w = 0; w < nw; w++) t += s_stat[k * nw + w];
        if (t) ta.events[4 * (size_t)blockIdx.x + k] += t;
    }
    // the scattered direction meanwhile (several components: the mix drawn first, DustSystem.cpp:855-869)
    R nx = kx, ny = ky, nz = kz;
    int nscatt = 0;
    if (scatters) {
        const R gs = MULTI ? (R)a.scene->gc[random_mix(a, mcell, rng)] : gg;
        hg_scatter<R>(rng, gs, nx, ny, nz);
        nscatt = (int)sl.fu(SU_NSCATT, i) + 1;
    }
    if (acts) {
        state = PS_OWN;
        sl.fr(SR_RX, i) = rx; sl.fr(SR_RY, i) = ry; sl.fr(SR_RZ, i) = rz;
        sl.fr(SR_KX, i) = nx; sl.fr(SR_KY, i) = ny; sl.fr(SR_KZ, i) = nz;
        sl.fu(SU_PLO, i) = rng.plo; sl.fu(SU_PHI, i) = rng.phi; sl.fu(SU_DRAW, i) = rng.draw;
        sl.fu(SU_W0, i) = rng.w0; sl.fu(SU_W1, i) = rng.w1; sl.fu(SU_W2, i) = rng.w2; sl.fu(SU_W3, i) = rng.w3;
        sl.fu(SU_NSCATT, i) = (uint32_t)nscatt;
        sl.fu(SU_HINT, i) = (uint32_t)hint;
    }
    if (state != state0) sl.fu(SU_STATE, i) = state;
    __syncthreads();
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
    auto put = [&](bool has, int k, const WalkReq<R>& w) {
        const uint64_t mask = __ballot(has);
        if (!has) return;
        const uint64_t at = s_base + s_n[k * nw + wave] + (uint64_t)__popcll(mask & below);
        q.req[at] = w;
        if (q.sorted) {
            const uint32_t key = walk_key<R>(a, a.scene->instr, w.tag, w.idx, w.o[0], w.o[1], w.o[2]);
            q.key[at] = key;
            q.rank[at] = atomicAdd(q.hist + key, 1u);
        }
    };
#pragma unroll
    for (int k = 0; k < SG_MAX_INSTR; k++) {
        if (k >= a.ni) continue;
        put(pix[k] >= 0, k, WalkReq<R>{{rx, ry, rz}, {(R)0, (R)0, (R)0}, Lp[k], (uint32_t)WK_PEEL | (uint32_t)k << 2,
                                       (uint32_t)pix[k], (uint32_t)hint});
    }
    put(acts, a.ni, WalkReq<R>{{rx, ry, rz}, {nx, ny, nz}, L, (uint32_t)WK_OWN, (uint32_t)i, (uint32_t)hint});
}

// Bin offsets of the walk order: exclusive prefix sum of the bin counts, which are cleared for the
// next pass. One block of 1024 threads; each thread sums kKeyBins / 1024 consecutive bins.
__global__ void __launch_bounds__(1024) k_key_scan(uint32_t* hist, uint32_t* off)
{
    constexpr int per = (int)(kKeyBins / 1024);
    __shared__ uint32_t s_wave[16];
    const int t = threadIdx.x;
    uint32_t v[per];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < per; k++) { v[k] = hist[t * per + k]; sum += v[k]; }
    // inclusive scan of the per-thread sums: within each wave, then across the 16 waves
    uint32_t x = sum;
    const int lane = __lane_id(), w = t >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[w] = x;
    __syncthreads();
    if (t < 64) {
        uint32_t z = t < 16 ? s_wave[t] : 0u;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const uint32_t y = __shfl_up(z, o);
            if (lane >= o) z += y;
        }
        if (t < 16) s_wave[t] = z;
    }
    __syncthreads();
    uint32_t run = x - sum + (w ? s_wave[w - 1] : 0u);
#pragma unroll
    for (int k = 0; k < per; k++) {
        off[t * per + k] = run;
        run += v[k];
        hist[t * per + k] = 0u;
    }
}

// Moves each request of the pass to its place in the walk order. A place beyond the pass's requests
// (bin counts that were not zero when the pass began) is reported through the error flag (bit 2)
// and not written.
template <typename R>
__global__ void __launch_bounds__(256) k_key_scatter(WalkQueue<R> q, int* error)
{
    const uint64_t n = *q.tail;
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t k = q.key[j];
        const uint64_t pos = (uint64_t)q.off[k < kKeyBins ? k : 0] + q.rank[j];
        if (k < kKeyBins && pos < n) q.sorted[pos] = q.req[j];
        else atomicOr(error, 2);
    }
}

// Start of a run: what its kernels expect to be zero, the packet claims, the scene, the clock.
struct RunBegin {
    struct Fill { uint32_t* p; int64_t words; } zero[11];
    int nzero;
    const uint32_t* scene_host;         // pinned host memory
    uint32_t* scene;
    unsigned long long* next;
    unsigned long long first_claim;
    unsigned long long* begin;          // clock ticks
};
// One launch: the scene's blocking copy, eleven fills and the event records took about 250 us of a run between them
// (a run of 5e3 packets on 24^3 cells: 1.05 ms with them, 0.95 ms now).
__global__ void __launch_bounds__(256) k_run_begin(const RunBegin b)
{
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, n = (int64_t)gridDim.x * blockDim.x;
    if (blockIdx.x == 0) {
        for (int i = (int)threadIdx.x; i < (int)(sizeof(SceneDev) / 4); i += (int)blockDim.x) b.scene[i] = b.scene_host[i];
        if (threadIdx.x == 0) {
            *b.next = b.first_claim;
            *b.begin = wall_clock64();
        }
    }
    for (int k = 0; k < b.nzero; k++)
        for (int64_t i = i0; i < b.zero[k].words; i += n) b.zero[k].p[i] = 0;
}

// What a run leaves in pinned host memory: its counters, error bits, and on the device clock its walk kernels'
// duration, its span from the start, and the times of its first pass's start and of its end.
struct RunResult {
    unsigned long long counters[SG_NCOUNTERS];
    unsigned long long err, walk, span, first, last;
};
struct RunEnd {
    GroupTally tally[2];
    GroupCtl* ctl[2];
    int n;
    unsigned long long* counters;
    const int* err;
    const unsigned long long* begin;
    unsigned int* ticket;               // zero at the run's start
    RunResult* out;                     // or null: the counters alone
};
// End of a run: the event workgroups' and the walk waves' counts into the run counters, by the last workgroup to
// finish written to the host with the rest of the result.
__global__ void __launch_bounds__(256) k_run_end(const RunEnd e)
{
    __shared__ unsigned long long s_sum[9];
    __shared__ bool s_last;
    if (threadIdx.x < 9) s_sum[threadIdx.x] = 0;
    __syncthreads();
    unsigned long long v[9] = {};
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, n = (int64_t)gridDim.x * blockDim.x;
    for (int g = 0; g < e.n; g++) {
        for (int64_t b = i0; b < e.tally[g].nevents; b += n)
            for (int k = 0; k < 4; k++) v[k] += e.tally[g].events[4 * b + k];
        for (int64_t w = i0; w < e.tally[g].nwaves; w += n) {
            const WaveRec& r = e.tally[g].waves[w];
            v[4] += r.own; v[5] += r.peel; v[6] += r.re; v[7] += r.stuck; v[8] += r.recompute;
        }
    }
#pragma unroll
    for (int k = 0; k < 9; k++) add_wave(&s_sum[k], v[k]);
    __syncthreads();
    const int dst[9] = {0, 3, 4, 7, 1, 2, 8, 5, 9};
#pragma unroll
    for (int k = 0; k < 9; k++)
        if ((int)threadIdx.x == k && s_sum[k]) atomicAdd(e.counters + dst[k], s_sum[k]);
    if (!e.out) return;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(e.ticket, 1u) == gridDim.x - 1;
    __syncthreads();
    if (!s_last) return;
    __threadfence();
    if (threadIdx.x < SG_NCOUNTERS)
        e.out->counters[threadIdx.x] = __hip_atomic_load(e.counters + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x == SG_NCOUNTERS) {
        unsigned long long walk = 0, start = ~0ull;
        for (int g = 0; g < e.n; g++) {
            walk += e.ctl[g]->ticks;
            start = min(start, e.ctl[g]->start);
        }
        const unsigned long long now = wall_clock64();
        e.out->err = (unsigned long long)*e.err;
        e.out->walk = walk;
        e.out->span = now - *e.begin;
        e.out->first = min(start, now);
        e.out->last = now;
    }
}

// Request claims of one wave: chunks of requests by one global atomic each, handed out in order to the lanes
// that ask. Called by the whole wave; cur/end is the wave's current chunk and last the place of its latest
// claim (wave-uniform). The chunk follows what is left of the queue, half of a wave's even share of it and at
// most kClaimChunk: large while the queue is long (few atomics), small near its end and for short queues, so
// that the last walks are spread over the waves instead of queueing up in a few. Returns whether this lane
// got request r; a lane that did not finds the queue exhausted.
constexpr uint64_t kClaimChunk = 128, kClaimMin = 16;
__device__ __forceinline__ bool chunk_claim(unsigned long long* ctr, uint64_t nq, uint64_t nwaves, bool want,
                                            uint64_t& cur, uint64_t& end, uint64_t& last, uint64_t& r)
{
    bool served = false;
    const int lane = __lane_id();
    for (;;) {
        const uint64_t mask = __ballot(want && !served);
        const uint64_t k = (uint64_t)__popcll(mask);
        if (k == 0) break;
        if (cur == end) {
            if (last >= nq) break;
            const uint64_t chunk = min(max((nq - last) / (2 * nwaves), kClaimMin), kClaimChunk);
            unsigned long long b = 0;
            if (lane == 0) b = atomicAdd(ctr, (unsigned long long)chunk);
            const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
            const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
            last = ((uint64_t)hi << 32) | lo;
            cur = min(last, nq);
            end = min(last + chunk, nq);
            if (cur == end) break;
        }
        const uint64_t take = min(k, end - cur);
        const uint64_t rank = (uint64_t)__popcll(mask & (lane ? (~0ull >> (64 - lane)) : 0ull));
        if (want && !served && rank < take) {
            r = cur + rank;
            served = true;
        }
        cur += take;
    }
    return served;
}

// Request claims by XCD segment: the requests [0, nq) of a pass, in walk order, are cut into kXcdSegs
// contiguous segments; a wave takes chunks from the segment of its workgroup's XCD (workgroups are dispatched
// to the XCDs in turn, so blockIdx.x mod 8 names the XCD) and moves on to the following segments once that one
// is exhausted. Walks that are neighbours in the walk order (start points or pixels close together) thus meet
// in the same XCD's L2. ctr holds one counter per segment. Lanes the wave's chunk does not serve stay idle
// until the next claim; exhausted (wave-uniform) becomes true when every segment is exhausted.
__device__ __forceinline__ bool seg_claim(unsigned long long* ctr, uint64_t nq, bool want, int& seg, int& tried,
                                          uint64_t& cur, uint64_t& end, uint64_t& r, bool& exhausted)
{
    const uint64_t mask = __ballot(want);
    const uint64_t k = (uint64_t)__popcll(mask);
    if (k == 0 || exhausted) return false;
    const int lane = __lane_id();
    const uint64_t rank = (uint64_t)__popcll(mask & (lane ? (~0ull >> (64 - lane)) : 0ull));
    if (end == cur) {
        while (tried < kXcdSegs) {
            const uint64_t s0 = nq * (uint64_t)seg / kXcdSegs, s1 = nq * (uint64_t)(seg + 1) / kXcdSegs;
            unsigned long long b = 0;
            if (lane == 0) b = atomicAdd(ctr + seg, (unsigned long long)kClaimChunk);
            const uint32_t lo = __shfl((uint32_t)b, 0), hi = __shfl((uint32_t)(b >> 32), 0);
            const uint64_t nb = s0 + (((uint64_t)hi << 32) | lo);
            if (nb < s1) {
                cur = nb;
                end = min(nb + kClaimChunk, s1);
                break;
            }
            seg = (seg + 1) % kXcdSegs;
            tried++;
        }
        if (end == cur) {
            exhausted = true;
            return false;
        }
    }
    const uint64_t take = min(k, end - cur);
    const bool ok = rank < take;
    if (ok) r = cur + rank;
    cur += take;
    return ok && want;
}

// Occupancy target of the walk kernel (waves per SIMD), by measurement; registers and spills as the compiler reports
// them. Four for the mixed tree walk: 128 registers, 2 to 4 spilled (4e6 packets on 7e5 leaves 51.9 ms; three 55.2,
// five, which spill more, 54.7). Three for the exact tree walk: 168 registers, 68 to 112 spilled (3e5 packets of optical
// depth 5: 13.0 ms; two 12.8, four 30.4). Four for the others.
#ifndef SG_WALK_WAVES_PER_EU
#define SG_WALK_WAVES_PER_EU 4
#endif
template <class W> struct WalkWaves { static constexpr int value = SG_WALK_WAVES_PER_EU; };
#ifndef SG_W32_WAVES
#define SG_W32_WAVES 4
#endif
template <> struct WalkWaves<TreeW32> { static constexpr int value = SG_W32_WAVES; };
#ifndef SG_W64_WAVES
#define SG_W64_WAVES 3
#endif
template <> struct WalkWaves<TreeW64> { static constexpr int value = SG_W64_WAVES; };
// the exact Cartesian walk at three: 168 registers, 2 to 4 spilled (1e6 packets on 50^3 cells: 9.2 ms; 9.4 at four, 11.1
// at five)
template <> struct WalkWaves<CartW64> { static constexpr int value = 3; };
// Lanes per Voronoi walk and entries per lane and step: 8 x 3 = 24 entries a step, which most lists (19 on average
// along the walks) fit, at three waves per SIMD: 168 registers, of which the mixed walk spills 5 to 6. On 1e5 sites with
// 3 x 1e5 packets: 33 ms a run; four lanes x 6 42 ms, 8 x 2 50 ms and 8 x 3 51 ms at four waves (spills), 16 x 2 50 ms; one lane x 16
// entries (VoroW, as the lane pipeline walks) spilled and took 106 ms. These are mixed runs; the FP64 walk takes the same
// shape, where it spills 78 to 91 registers (3e4 packets on 3e4 sites 14.1 ms; VoroW in the passes 61, in the lane
// pipeline 28).
#ifndef SG_VORO_LANES
#define SG_VORO_LANES 8
#endif
#ifndef SG_VORO_EACH
#define SG_VORO_EACH 3
#endif
#ifndef SG_VORO_WAVES
#define SG_VORO_WAVES 3
#endif
template <typename R> using VoroWalk = VoroC<R, SG_VORO_LANES, SG_VORO_EACH>;
template <typename R> struct WalkWaves<VoroWalk<R>> { static constexpr int value = SG_VORO_WAVES; };

// The end of an own path (lane's walk of slot idx, request w): DustSystem::fillOpticalDepth's check
// (DustSystem.cpp:952-955), simulateescapeandabsorption (MonteCarloSimulation.cpp:432-508), the stop test
// and simulatepropagation (:513-531). Either the packet is finished or scatters where it is, which the slot's
// state tells the next event pass, or the lane goes on with the walk to the interaction point (ST_PROP).
// Done here rather than in the event kernel, the re-walk shares this pass with the long walks: as a pass of
// its own it took a fifth of the walk time for 3% of the crossings, and each scattering took two event
// passes.
template <class W, bool MULTI>
__device__ __forceinline__ void own_path_end(Hot<W>& h, const typename W::View& g, const int32_t* lds, int nlds,
                                             const McArgs& a, const Slots<typename W::Real>& sl, uint32_t idx,
                                             const WalkReq<typename W::Real>* w)
{
    using R = typename W::Real;
    const R taupath = h.tau;
    h.stage = ST_NEWPKT;
    if (taupath < (R)0 || isnan(taupath) || isinf(taupath)) {
        atomicOr(a.error, 1);
        sl.fu(SU_STATE, idx) = PS_FRESH;
        return;
    }
    // one component, or the sum of each cell's albedo times its interacting luminosity, gathered along the walk
    R L;
    if (MULTI) L = h.lsca;
    else {
        const R expfactor = -rexpm1<R>(-taupath);
        L = h.L0 * (R)a.albedo * expfactor;
    }
    if (L <= (R)0 || (L <= (R)a.Lthreshold && (int)sl.fu(SU_NSCATT, idx) >= a.minfs)) {
        sl.fu(SU_STATE, idx) = PS_FRESH;
        return;
    }
    sl.fu(SU_STATE, idx) = PS_PROP;
    if (taupath == (R)0) {
        // zero optical depth along the path: scattering in place
        sl.fr(SR_L, idx) = L;
        sl.fr(SR_RES, idx) = (R)0;
        if (MULTI) sl.fu(SU_MCELL, idx) = (uint32_t)-1;
        return;
    }
    PacketRng rng;
    rng.k0 = a.seed; rng.k1 = a.member; rng.ell = (uint32_t)a.ell;
    rng.plo = sl.fu(SU_PLO, idx); rng.phi = sl.fu(SU_PHI, idx); rng.draw = sl.fu(SU_DRAW, idx);
    rng.w0 = sl.fu(SU_W0, idx); rng.w1 = sl.fu(SU_W1, idx); rng.w2 = sl.fu(SU_W2, idx); rng.w3 = sl.fu(SU_W3, idx);
    // one deviate, or (biased) one for the choice of distribution and one for the depth
    R tt, u = 0;
    bool uniform = false;
    for (int k = a.xi == 0.0 ? 1 : 0; k < 2; k++) {
        uniform = k == 1 && a.xi != 0.0 && u < (R)a.xi;
        u = uni<R>(rng);
    }
    if (uniform) tt = u * taupath;
    else tt = exponcutoff_from(rng, u, taupath);
    if (a.xi != 0.0) {
        const R pp = -rexp<R>(-tt) / rexpm1<R>(-taupath);
        const R qq = ((R)1.0 - (R)a.xi) * pp + (R)a.xi / taupath;
        L = L * (pp / qq);
    }
    sl.fr(SR_L, idx) = L;
    sl.fu(SU_DRAW, idx) = rng.draw;
    sl.fu(SU_W0, idx) = rng.w0; sl.fu(SU_W1, idx) = rng.w1; sl.fu(SU_W2, idx) = rng.w2; sl.fu(SU_W3, idx) = rng.w3;
    if constexpr (W::kHint) h.w.init_hinted(g, lds, nlds, w->o[0], w->o[1], w->o[2], w->d[0], w->d[1], w->d[2], (int)w->hint);
    else h.w.init(g, lds, nlds, w->o[0], w->o[1], w->o[2], w->d[0], w->d[1], w->d[2]);
    h.start_walk(ST_PROP, tt);
}

// A finished walk's result: a peel-off's detection (FrameInstrument::detect, FrameInstrument.cpp:33-47), an own
// path's end, or the interaction point's distance and leaf for the packet slot. Afterwards the lane is idle, or
// walks on to the interaction point.
template <class W, bool MULTI>
__device__ __forceinline__ void walk_end(Hot<W>& h, const typename W::View& g, const int32_t* lds, int nlds,
                                         const McArgs& a, const Slots<typename W::Real>& sl, const InstrDev* instr,
                                         uint32_t inst, uint32_t idx, const WalkReq<typename W::Real>* w)
{
    if (h.stage == ST_PEELW_DONE) {
        const InstrDev& in = instr[inst];
        if (leads<W>())
            unsafeAtomicAdd(in.frame + (size_t)a.ell * in.Nx * in.Ny + idx, (double)(h.L0 * rexp<typename W::Real>(-h.tau)));
        h.stage = ST_NEWPKT;
    } else if (h.stage == ST_PROP_DONE) {
        using R = typename W::Real;
        const R d = prop_length(h);
        sl.fr(SR_RES, idx) = d;
        if (MULTI) sl.fu(SU_MCELL, idx) = (uint32_t)h.mcell;
        h.stage = ST_NEWPKT;
        // the leaf holding the interaction point, where the packet's next walks start: the last segment's, or
        // (a walker whose start cells are exact) looked for by this lane, once for all of those walks, at the
        // point that the event kernel computes by the same formula
        if constexpr (W::kLocates) {
            h.w.locate_next(g, (double)(w->o[0] + d * w->d[0]), (double)(w->o[1] + d * w->d[1]),
                            (double)(w->o[2] + d * w->d[2]));
            h.start_walk(ST_LOC, (R)0);
        } else if constexpr (W::kHint) sl.fu(SU_HINT, idx) = (uint32_t)h.w.hint();
    } else if (h.stage == ST_LOC_DONE) {
        if constexpr (W::kLocates) sl.fu(SU_HINT, idx) = (uint32_t)h.w.hint();
        h.stage = ST_NEWPKT;
    } else if (h.stage == ST_OWN_DONE) own_path_end<W, MULTI>(h, g, lds, nlds, a, sl, idx, w);
}

// Walk kernel bookkeeping of a pass: its first wave's start and, by block 0, the host's progress word (bit 63:
// written, bit 62: every packet claimed, below: requests of the pass).
__device__ __forceinline__ void pass_begin(PassCtl* pc, const McArgs& a, uint64_t nq, unsigned long long* progress)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const bool claimed = *a.next_packet >= a.count;
    pc->t0 = nq ? (unsigned long long)wall_clock64() : 0ull;
    __hip_atomic_store(progress, (1ull << 63) | (claimed ? 1ull << 62 : 0ull) | (unsigned long long)nq, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// Walk pass: persistent lanes over the requests [0, *q.tail). A queue with fewer requests than the launch
// has chunks needs only the first workgroups.
template <class W, bool ABS, bool MULTI>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WalkWaves<W>::value, 8))) k_walks(const typename W::View g, const McArgs a, WalkQueue<typename W::Real> q,
                                              Slots<typename W::Real> sl, PassCtl* pc, unsigned long long* progress,
                                              const GroupTally ta, int nlds_req, int xcd_segments)
{
    using R = typename W::Real;
    __shared__ InstrDev s_instr[SG_MAX_INSTR];
    extern __shared__ __align__(16) unsigned char smem[];
    const uint64_t nq = *q.tail;
    pass_begin(pc, a, nq, progress);
    if ((uint64_t)blockIdx.x * (blockDim.x >> 6) * kClaimMin >= nq) return;
    int32_t* s_nodes = reinterpret_cast<int32_t*>(smem);
    int nlds = 0;
    if (nlds_req > 0) stage_view<W>(g, s_nodes, nlds_req, threadIdx.x, blockDim.x, nlds);
    if (threadIdx.x < SG_MAX_INSTR) s_instr[threadIdx.x] = a.scene->instr[threadIdx.x];
    __syncthreads();
    const WalkReq<R>* reqs = q.sorted ? q.sorted : q.req;
    const uint64_t nwaves = (uint64_t)gridDim.x * (blockDim.x >> 6);
    Hot<W> h;
    h.stage = ST_NEWPKT;   // idle: needs a request
    h.nseg = 0; h.nent = 0;
    h.w.nrecompute = 0; h.w.nstuck = 0;
    uint32_t idx = 0, inst = 0, req = 0;
    uint32_t n_own = 0, n_peel = 0, n_re = 0;   // the lane's crossings by walk kind
    uint64_t ccur = 0, cend = 0, clast = 0;      // the wave's chunk of requests
    int seg = blockIdx.x % kXcdSegs, tried = 0;  // XCD segments: the wave's segment, segments left behind
    bool exhausted = false;
    const int thr = a.compact;
    for (;;) {
        if (finished_stage(h.stage)) {
            if (leads<W>()) count_walk(h, n_own, n_peel, n_re);
            walk_end<W, MULTI>(h, g, s_nodes, nlds, a, sl, s_instr, inst, idx, reqs + req);
        }
        const bool want = h.stage == ST_NEWPKT;
        uint64_t r = 0;
        // a walk's lanes (neighbours, all in the same stage) share the request that their first lane claims
        const bool asks = want && leads<W>();
        bool got = xcd_segments ? seg_claim(pc->seg, nq, asks, seg, tried, ccur, cend, r, exhausted)
                                : chunk_claim(&pc->claim, nq, nwaves, asks, ccur, cend, clast, r);
        if constexpr (W::kLanes > 1) {
            const uint32_t first = __lane_id() & ~(uint32_t)(W::kLanes - 1);
            got = __shfl((int)got, first) != 0;
            r = __shfl((uint32_t)r, first);   // requests number fewer than 2^32
        }
        if (want && !got && xcd_segments && !exhausted) {
            // not served by this claim: the lane stays idle and claims again
        } else if (want) {
            const WalkReq<R> w = got ? reqs[r] : WalkReq<R>{};
            const uint32_t kind = w.tag & 3u;
            const uint32_t wi = w.tag >> 2;
            // a request that names no pixel of an instrument or no packet slot is reported (error bit 2)
            // and dropped, never followed; the lane stays idle and takes the next one
            const uint32_t npix = wi < (uint32_t)a.ni ? (uint32_t)(s_instr[wi].Nx * s_instr[wi].Ny) : 0u;
            const bool valid = kind == WK_PEEL ? w.idx < npix : kind == WK_OWN && (int64_t)w.idx < sl.n;
            if (!got) h.stage = ST_DEAD;
            else if (!valid) atomicOr(a.error, 4);
            else {
                idx = w.idx;
                inst = wi;
                req = (uint32_t)r;
                const R ox = w.o[0], oy = w.o[1], oz = w.o[2];
                double dx, dy, dz;
                if (kind == WK_PEEL) {
                    const InstrDev& in = s_instr[inst];
                    dx = in.kobs[0]; dy = in.kobs[1]; dz = in.kobs[2];
                } else {
                    dx = w.d[0]; dy = w.d[1]; dz = w.d[2];
                }
                if constexpr (W::kHint)
                    h.w.init_hinted(g, s_nodes, nlds, ox, oy, oz, dx, dy, dz, (int)w.hint);
                else
                    h.w.init(g, s_nodes, nlds, ox, oy, oz, dx, dy, dz);
                h.L0 = w.val;
                h.lsca = (R)0;
                if (kind == WK_PEEL) h.start_walk(ST_PEELW, (R)a.tau_cut);
                else h.start_walk(ST_OWN, (R)0);
            }
        }
        const uint64_t alive = __ballot(h.stage != ST_DEAD);
        if (!alive) break;
        // wave-uniform, kept in a scalar register
        const int need_n = __builtin_amdgcn_readfirstlane(max(1, min(thr, __popcll(alive) >> 1)));
        bool walk = walking_stage(h.stage);
        for (;;) {
            if (walk) walk = crossing<W, ABS, MULTI>(h, g, s_nodes, nlds, a);
            // lanes alive and not walking are idle (alive is fixed while the wave walks)
            const uint64_t wm = __ballot(walk);
            if (__popcll(alive & ~wm) >= need_n || !wm) break;
        }
    }
    // the wave's record: only this wave writes it
    WaveRec& rec = ta.waves[blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)];
    const unsigned long long own = wave_sum(n_own), peel = wave_sum(n_peel), re = wave_sum(n_re);
    const unsigned long long stuck = wave_sum(leads<W>() ? h.w.nstuck : 0u);
    const unsigned long long recompute = wave_sum(leads<W>() ? h.w.nrecompute : 0u);
    if (__lane_id() == 0) {
        rec.own += own; rec.peel += peel; rec.re += re; rec.stuck += stuck; rec.recompute += recompute;
        rec.t1 = (unsigned long long)wall_clock64();
    }
}

} // namespace sg
