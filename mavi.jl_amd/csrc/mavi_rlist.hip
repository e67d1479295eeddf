// mavi_rlist.hip -- Verlet lists for Rings step! (src/rings/integration.jl:
// 522-543) of a fixed population of rings (of 3 to 32 particles) on a periodic
// chunk grid whose chunks are at least the interaction range wide: one kernel per
// step instead of a binning (three launches), the pair gather and the ring update.
//
// State.  While the lists run the state lies in ring order (slot = position of
// the particle's id among the active ids), so a ring's particles are
// consecutive and every kernel reads and writes them with unit stride; the two
// state copies ping-pong, because a ring's neighbours read its old positions.
//
// Pairs.  Each particle lists the others within range + skin that it can
// interact with (not its bonded neighbours), found on a grid of cells at least
// that wide.  The lists stay complete while no particle has moved more than
// half the skin since the build; the host checks that once per block of steps
// (the same bound as the neighbour lists of plain systems, mavi_nlist.hip) and
// rolls an overrun block back.
//
// Same bits as the gather.  calc_forces! visits the pairs of adjacent chunks
// of the step's own binning; every pair within range is among them, and the
// gather adds a particle's pairs by chunk row, chunk column (the visiting order
// at the periodic edges included) and id.  One or two pairs in range add to
// the same value in any order; for three or more the contributions are put in
// that order first, from the exact chunks of the positions.  Everything else
// of the step is ring_lanes' arithmetic term by term, so a trajectory does not
// depend on whether the lists run, when they were built or how it was split
// into calls, and a batch replica stays bit-identical to the system alone.
//
// Errors.  Chunks and chunk counts of the reference grid follow every particle
// (out of box, non-finite); a count that may have passed the capacity, or a
// list that is too long, hands the block to the gather, which checks exactly.
//
// Handing over.  The lists give a state to the gather for a while when a list
// would serve at most two of its steps or a chunk may be full (rl_back_off), and
// until a new state or skin when a list is too long; the gather's steps are the
// same bits.
#include <math.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "mavi_batch.h"
#include "mavi_device.h"
#include "mavi_host.h"

namespace {

constexpr int kRlHead = 4;    // list entries in the particle's int4
constexpr int kRlMax = 16;    // list entries per particle
// Step workgroup: waves of floor(64 / nmax) rings.  us a step at 2k / 800k
// particles: 4 waves 11.7 / 48.6, 8 waves 12.8 / 51.7, 12 waves 14.0 / 54.8
// (one wave does the ring stage of all while the others' places stay empty).
constexpr int kRlWaves = 4, kRlWG = 64 * kRlWaves;
constexpr uint32_t kRlOverflow = 1u;  // a list longer than kRlMax
constexpr uint32_t kRlCapacity = 2u;  // a chunk count may have passed the capacity

// A list entry: partner slot (26 bits), its ring type (5 bits); the sign bit
// marks the end (-1).  Same-ring partners are told apart by their slots.
constexpr int kRlSlotBits = 26;
constexpr int32_t kRlSlotMask = (1 << kRlSlotBits) - 1;

struct RLArgs {
    const double2 *Pin;
    double2 *Pout;
    double2 *F;                 // last step of a call only
    const int32_t *slot_of;     // null: slot = id (every ring full)
    const int4 *head;
    const int32_t *more;        // entries kRlHead.. of slot q: more[e * na + q]
    const uint8_t *count;
    int32_t *key;               // reference chunk (row << 16 | col) of each slot
    int32_t *ccnt;
    double *pol;
    double2 *polcs;             // cos, sin of each ring's polarisation
    double *areas;
    double2 *cms, *cms_next, *cpos;
    const int32_t *rtype;
    const RingType *types;
    const RingInter *inter;     // matrix of interactions; null: `uni` for every pair
    RingInter uni;
    uint32_t *bmax;             // per workgroup: high word of the largest squared step, rounded up
    uint32_t *flags, *status;
    uint64_t seed;
    const unsigned long long *cin;  // the step counter before this step
    unsigned long long *cout;
    int64_t stride;             // slots (stride of `more`)
    int32_t per;                // most rings of a wave
    // a batch: replicas by wave of the step kernel, and their table
    const Replica *reps;
    const int32_t *wave_rep;
    int32_t nwaves;
};

// Where a system's arrays start in a batch (0 for a system alone).
struct RLBase {
    int32_t slot = 0, id = 0, chunk = 0, ring = 0, type = 0, inter = 0, flag = 0;
    int64_t cpos = 0;
};
__device__ __forceinline__ RLBase rl_base(const Replica &Q, int rep) {
    return RLBase{Q.pbase, Q.nbase, Q.cbase, Q.rbase, Q.tbase, Q.ibase, rep, Q.cpbase};
}

__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// calc_diff with the image arithmetic only where some lane of the wave needs
// it (min_image is the identity for |dr| <= half the box).
__device__ __forceinline__ double2 wave_diff(const SysParams &P, double2 a, double2 b) {
    double dx = a.x - b.x, dy = a.y - b.y;
    if (__any(fabs(dx) > P.halfL || fabs(dy) > P.halfH)) {
        dx = min_image(dx, P.L, P.halfL);
        dy = min_image(dy, P.H, P.halfH);
    }
    return make_double2(dx, dy);
}

// Place of partner chunk (rj, cj) in the gather's order around (ri, ci): its
// rows from -1 to 1, in a row the columns in slot order, except that at the
// periodic column edges the wrapped column comes last.
__device__ __forceinline__ uint32_t visit_rank(const SysParams &P, int ri, int ci, int rj, int cj) {
    int d = rj - ri + 1;
    if (d < 0) d += P.rows;
    else if (d > 2) d -= P.rows;
    int c = cj - ci + 1;
    if (ci == 0) c = cj > 1 ? 2 : cj;                                     // 0, 1, then cols - 1
    else if (ci == P.cols - 1) c = cj == 0 ? 2 : cj - (P.cols - 2);        // cols - 2, cols - 1, then 0
    return (uint32_t)(d * 3 + c);
}

// The interaction of type ti with entry e's type (mat null: `uni` for every pair).
__device__ __forceinline__ RingInter rl_inter(const SysParams &P, const RingInter *mat, const RingInter &uni, int ti,
                                              int32_t e) {
    return mat ? mat[ti + P.ntypes * (e >> kRlSlotBits)] : uni;
}

// calc_interaction_force (src/rings/integration.jl:47-77) of a listed pair in
// range (never bonded neighbours).
__device__ __forceinline__ double2 rl_force(const RingInter &I, double2 d, double r2, bool same) {
    const double dist = sqrt(r2);
    double fmod;
    double u = dist;
    if (I.dist_eq != 1.0) u = dist / I.dist_eq;  // discs of unit diameter need no division
    if (r2 < I.eq2) fmod = -I.k_rep * (u - 1.0);
    else fmod = same ? 0.0 : -I.k_atr * (u - 1.0);
    const double q = fmod / dist;
    return make_double2(q * d.x, q * d.y);
}

__device__ __forceinline__ unsigned long long visit_key(const SysParams &P, int ri, int ci, double2 pj, int j) {
    uint32_t flag = 0;
    int32_t rj, cj;
    cell_rc(P, P.rows, P.cols, P.cl, P.ch, pj.x, pj.y, &flag, MAVI_FLAG_OUT_OF_BOX, &rj, &cj);
    return ((unsigned long long)visit_rank(P, ri, ci, rj, cj) << 32) | (uint32_t)j;
}

// The sums of the wave's particles with long lists (`longer`), into their f: four
// particles at a time, a row of 16 lanes to each, a lane to each entry.  A lane's
// pair in range goes to its place in the gather's order (the number of its row's
// smaller keys) in the row's part of `place`, which the particle's own lane sums
// from the front.  Bound: the trip of a row's entries and positions to memory, once
// per four particles; with each such lane selecting its pairs one by one, its list
// walked for every pair, it was that trip for every entry of every walk.  us a step
// of jammed mixtures, before -> after: 20k particles 25.2 -> 16.4, 200k 41.4 ->
// 24.1; 2k pressed to 0.6 of the box's side 59 -> 25 (the gather 47).  Out of the
// way of the step's straight line (builtin_expect): 1 % of a step where no list is long.
__device__ __forceinline__ void rl_long_sums(const SysParams &P, const RLArgs &A, const RingInter *mat,
                                             const RingInter &uni, bool longer, int q, int cnt, int t0, int np, int ti,
                                             int32_t ko, const double2 *xs, double2 *place, double2 &f) {
    static_assert(kRlMax == 16, "a lane of a row per entry");
    const int lane = (int)lane_id(), e = lane & 15, row = lane >> 4;
    for (unsigned long long m = __ballot(longer); m;) {
        // the next four
        int l[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            l[k] = m ? __ffsll(m) - 1 : -1;
            m &= m - 1;
        }
        const int from = row == 0 ? l[0] : row == 1 ? l[1] : row == 2 ? l[2] : l[3];
        const int src = max(from, 0);
        const int qs = __shfl(q, src, 64), cs = __shfl(cnt, src, 64), n = from < 0 ? 0 : cs;
        const int ts = __shfl(t0, src, 64), nps = __shfl(np, src, 64), tis = __shfl(ti, src, 64);
        const int32_t ks = __shfl(ko, src, 64);
        bool in = false;
        unsigned long long key = ~0ull;
        double2 c = make_double2(0.0, 0.0);
        if (e < n) {
            const int32_t w = e < kRlHead ? ((const int32_t *)A.head)[(int64_t)kRlHead * qs + e]
                                          : A.more[(int64_t)(e - kRlHead) * A.stride + qs];
            const int j = w & kRlSlotMask;
            const double2 pj = A.Pin[j];
            const double2 d = cdiff(P, xs[src], pj);
            const double r2 = d.x * d.x + d.y * d.y;
            const RingInter I = rl_inter(P, mat, uni, tis, w);
            in = !(r2 > I.max2);
            if (in) {
                key = visit_key(P, ks >> 16, ks & 0xffff, pj, j);
                c = rl_force(I, d, r2, j >= ts && j < ts + nps);
            }
        }
        int at = 0;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const unsigned long long o = __shfl(key, (lane & 48) + k, 64);
            at += o < key ? 1 : 0;
        }
        if (in) place[(lane & 48) + at] = c;
        const unsigned long long hits = __ballot(in);
        lds_sync();
        if (lane == l[0] || lane == l[1] || lane == l[2] || lane == l[3]) {
            const int r = lane == l[0] ? 0 : lane == l[1] ? 1 : lane == l[2] ? 2 : 3;
            const int k1 = __popcll((hits >> (16 * r)) & 0xffffull);
            double2 s = make_double2(0.0, 0.0);
            for (int k = 0; k < k1; k++) {
                s.x += place[16 * r + k].x;
                s.y += place[16 * r + k].y;
            }
            f = s;
        }
        lds_sync();  // before the places are written again
    }
}

// What the polarisation update of ring k of a workgroup (place k % per of wave
// k / per, per the most rings of a wave) needs from memory, and its noise.  np 0: no ring there.
struct RingScalars {
    double pol, cs, sn, rate, dt, noise;
    int32_t np, rg;
};
template <bool BATCH>
__device__ __forceinline__ RingScalars ring_scalars(const SysParams &P0, const RLArgs &A, int block, int k,
                                                    unsigned long long step) {
    const int w = k / A.per, wl = block * kRlWaves + w;
    RingScalars R{};
    if (BATCH && wl >= A.nwaves) return R;
    const Replica *Q = BATCH ? A.reps + A.wave_rep[wl] : nullptr;
    const SysParams &P = BATCH ? Q->P : P0;
    const int own = BATCH ? 64 / P.nmax : A.per;  // rings of that wave
    const int g = k - w * A.per;
    const int ring = (BATCH ? wl - Q->rwbase : wl) * own + g;
    if (g >= own || ring >= P.nrings) return R;
    R.rg = (BATCH ? Q->rbase : 0) + ring;
    const RingType *T = A.types + (BATCH ? Q->tbase : 0) + (P.typed ? A.rtype[R.rg] : 0);
    const double2 cs = A.polcs[R.rg];
    R.pol = A.pol[R.rg];
    R.cs = cs.x;
    R.sn = cs.y;
    R.np = T->np;
    R.dt = P.dt;
    R.rate = 1.0 / T->relax;
    const double rot = T->rot;
    const double z = rot != 0.0 ? philox_normal(BATCH ? Q->seed : A.seed, step, (uint32_t)ring) : 0.0;
    R.noise = sqrt(2.0 * rot * R.dt) * z;
    return R;
}

// Largest value of the wave, in lane 63.
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
#define MAVI_DPP_MAX(ctrl, rows) \
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false))
    MAVI_DPP_MAX(0x111, 0xf);  // row_shr 1, 2, 4, 8: lane 15 of a row holds the row's
    MAVI_DPP_MAX(0x112, 0xf);
    MAVI_DPP_MAX(0x114, 0xf);
    MAVI_DPP_MAX(0x118, 0xf);
    MAVI_DPP_MAX(0x142, 0xa);  // row_bcast 15, 31
    MAVI_DPP_MAX(0x143, 0xc);
#undef MAVI_DPP_MAX
    return v;
}

// One Rings step! of the rings of this workgroup.  LAST: the last step of a
// call, which leaves the forces and the continuous positions (every step
// recomputes both before it uses them).
//
// Bound: FP64 VALU issue (817 instructions a wave, 45 % of the issue cycles at 800k
// particles) and the length of its dependent chain.  The ring's
// left-to-right sums (unwrap, centre of mass, shoelace, mean velocity) run
// once per ring and component on a few lanes (2 or 3 per ring) instead of as
// masked loops of every lane, and the scalar work of a ring (noise, asin,
// sincos of the new angle) once per workgroup on one lane per ring: as part of
// every wave it was a third of the ring kernel's instructions.  That lane takes
// its inputs and the noise, which do not depend on the forces, while the pairs'
// positions are on their way.  With the rebuilds 46.3 us a step at 800k
// particles (49.0 with the ring stage's loads at its end) against 97 us for the
// five launches it replaces (scan 12.1, scatter 8.7, finalize 11.1, pairs 26.2,
// ring update 38.1); 11.3 against 33 us at 2k particles.
template <bool LAST, bool BATCH>
__global__ __launch_bounds__(kRlWG) __attribute__((amdgpu_waves_per_eu(4))) void k_rl_step(SysParams P0, RLArgs A) {
    __shared__ double2 s_a[kRlWG + 32], s_b[kRlWG + 32], s_c[kRlWG + 32];
    __shared__ double s_t[kRlWG + 32];
    __shared__ double s_r[kRlWaves][64 * 3];  // per ring of a wave: sums
    __shared__ uint32_t s_max[kRlWaves];
    __shared__ RingScalars s_ring[64];  // wave 0: of the workgroup's first 64 rings
    const int lane = (int)lane_id(), wave = uniform((int)(threadIdx.x >> 6));
    const int block = xcd_block();
    const int wl = block * kRlWaves + wave;
    const int rep = BATCH ? uniform(A.wave_rep[min(wl, A.nwaves - 1)]) : 0;
    const SysParams P = BATCH ? A.reps[rep].P : P0;
    const RLBase B = BATCH ? rl_base(A.reps[rep], rep) : RLBase{};
    const RingInter *mat = BATCH ? (A.reps[rep].uniform ? nullptr : A.inter + B.inter) : A.inter;
    const RingInter &uni = BATCH ? A.inter[B.inter] : A.uni;
    const int per = 64 / P.nmax;
    const int grp = lane / P.nmax, i = lane - grp * P.nmax;
    const int first = (BATCH ? wl - A.reps[rep].rwbase : wl) * per;  // the wave's first ring
    const int r = first + grp;
    const bool ring_ok = (!BATCH || wl < A.nwaves) && grp < per && r < P.nrings;
    const int rr = ring_ok ? r : 0;
    const int t = P.typed ? A.rtype[B.ring + rr] : 0;
    const RingType *T = A.types + B.type + t;
    const bool full = !A.slot_of;  // every ring has nmax particles
    const int np = full ? P.nmax : T->np;
    const bool act = ring_ok && i < np;
    const int id = rr * P.nmax + i;
    const int q = act ? (full ? B.slot + id : A.slot_of[B.id + id]) : B.slot;
    const int t0 = q - i, t1 = t0 + np;  // the ring's slots
    const double2 x = act ? A.Pin[q] : make_double2(0.0, 0.0);
    int4 h = act ? A.head[q] : make_int4(-1, -1, -1, -1);
    const int32_t ko = act ? A.key[q] : 0;
    const double2 pcs = A.polcs[B.ring + rr];
    const unsigned long long step = A.cin[0] + 1ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) A.cout[0] = step;

    // ---- pairs within range: the head's four entries
    const int32_t ent[kRlHead] = {h.x, h.y, h.z, h.w};
    double2 pj[kRlHead];
#pragma unroll
    for (int e = 0; e < kRlHead; e++)
        pj[e] = ent[e] >= 0 ? A.Pin[ent[e] & kRlSlotMask] : x;
    int cnt = 0;  // of a list that the head may not hold
    if (ent[kRlHead - 1] >= 0) cnt = A.count[q];

    // meanwhile: what the ring stage of wave 0 takes from memory and its noise
    uint32_t hi0 = 0u;
    if (wave == 0) {
        hi0 = A.bmax[block];
        if (lane < kRlWaves * A.per) s_ring[lane] = ring_scalars<BATCH>(P0, A, block, lane, step);
    }

    // neighbours along the ring and the unwrap's steps, meanwhile
    const int me = (int)threadIdx.x, tb = me - i, wb = wave * 64;
    const int inext = (i == np - 1) ? 0 : i + 1;
    const int iprev = (i == 0) ? np - 1 : i - 1;
    s_a[me] = x;
    lds_sync();
    const double2 xn = s_a[tb + inext];
    const double2 xp = s_a[tb + iprev];
    const double2 dprev = wave_diff(P, x, xp);
    s_b[me] = i == 0 ? x : dprev;
    lds_sync();
    // ring sizes for the serial lanes: lane l < 3 per (<= 63: rl_fits) works for
    // ring l / 2 or l / 3
    const int np2 = __shfl(np, min(lane >> 1, per - 1) * P.nmax, 64);
    const int np3 = __shfl(np, min(lane / 3, per - 1) * P.nmax, 64);
    if (lane < 2 * per) {
        // c_0 = x_0, c_k = c_{k-1} + calc_diff(x_k, x_{k-1}), one lane per component
        const int o = 2 * (wb + (lane >> 1) * P.nmax) + (lane & 1);
        const double *src = (const double *)s_b + o;
        double *dst = (double *)s_c + o;
        double c = src[0];
        dst[0] = c;
#pragma unroll 4
        for (int k = 1; k < np2; k++) {
            c = c + src[2 * k];
            dst[2 * k] = c;
        }
    }
    lds_sync();
    const double2 c = s_c[me], cn = s_c[tb + inext];
    if (LAST && act) A.cpos[B.cpos + id] = c;
    s_t[me] = c.x * cn.y - c.y * cn.x;
    lds_sync();
    if (lane < 3 * per) {
        // centre of mass and shoelace sums in ring order, one lane per sum
        const int g = lane / 3, which = lane - 3 * g;
        const double *src = which == 2 ? s_t + wb + g * P.nmax : (const double *)(s_c + wb + g * P.nmax) + which;
        const int stride = which == 2 ? 1 : 2;
        double s = 0.0;
#pragma unroll 4
        for (int k = 0; k < np3; k++) s += src[k * stride];
        s_r[wave][lane] = s;
    }

    // ---- pair forces
    double2 f[kRlHead];
    bool in[kRlHead];
    int m = 0;
#pragma unroll
    for (int e = 0; e < kRlHead; e++) {
        f[e] = make_double2(0.0, 0.0);
        in[e] = false;
        if (!__any(ent[e] >= 0)) continue;
        const double2 d = wave_diff(P, x, pj[e]);
        const double r2 = d.x * d.x + d.y * d.y;
        const RingInter I = rl_inter(P, mat, uni, t, ent[e] >= 0 ? ent[e] : 0);
        in[e] = ent[e] >= 0 && !(r2 > I.max2);
        if (in[e]) {
            const int j = ent[e] & kRlSlotMask;
            f[e] = rl_force(I, d, r2, j >= t0 && j < t1);
            m++;
        }
    }
    const bool longer = cnt > kRlHead;
    const bool order = m > 2 && !longer;
    if (__builtin_expect(__any(order), 0)) {
        if (order) {
            const int ri = ko >> 16, ci = ko & 0xffff;
            unsigned long long k[kRlHead];
#pragma unroll
            for (int e = 0; e < kRlHead; e++)
                k[e] = in[e] ? visit_key(P, ri, ci, pj[e], ent[e] & kRlSlotMask) : ~0ull;
            auto cmpx = [&](int a, int b) {
                const bool sw = k[b] < k[a];
                const unsigned long long ka = sw ? k[b] : k[a], kb = sw ? k[a] : k[b];
                const double2 fa = sw ? f[b] : f[a], fb = sw ? f[a] : f[b];
                k[a] = ka;
                k[b] = kb;
                f[a] = fa;
                f[b] = fb;
            };
            cmpx(0, 1);
            cmpx(2, 3);
            cmpx(0, 2);
            cmpx(1, 3);
            cmpx(1, 2);
        }
    }
    double2 Fi = make_double2(0.0, 0.0);
#pragma unroll
    for (int e = 0; e < kRlHead; e++) {
        Fi.x += f[e].x;
        Fi.y += f[e].y;
    }
    if (__builtin_expect(__any(longer), 0)) rl_long_sums(P, A, mat, uni, longer, q, cnt, t0, np, t, ko, s_a + wb, s_b + wb, Fi);

    // ---- springs and area force
    const double2 ds = wave_diff(P, x, xn);
    const double dist = sqrt(ds.x * ds.x + ds.y * ds.y);
    const double sq = -T->kspring * (dist - T->lspring) / dist;
    const double2 fi = make_double2(sq * ds.x, sq * ds.y);
    s_b[me] = fi;  // the unwrap's reads of s_b are done
    lds_sync();
    const double2 fprev = s_b[tb + iprev];
    const double area = s_r[wave][min(grp, per - 1) * 3 + 2] / 2.0;
    if (ring_ok && i == 0) {
        const double *s = &s_r[wave][grp * 3];
        const int g = B.ring + r;
        A.cms[g] = A.cms_next[g];  // update_cms! reads the previous continuous positions
        A.cms_next[g] = make_double2(s[0] / (double)np, s[1] / (double)np);
        A.areas[g] = area;
    }
    double area0 = (double)np * T->lspring / T->p0;
    area0 = area0 * area0;
    const double fa = T->karea * (area - area0);
    const double2 da = wave_diff(P, xn, xp);
    if (i == 0) {
        Fi.x += fi.x;
        Fi.y += fi.y;
        Fi.x -= fprev.x;
        Fi.y -= fprev.y;
    } else {
        Fi.x -= fprev.x;
        Fi.y -= fprev.y;
        Fi.x += fi.x;
        Fi.y += fi.y;
    }
    Fi.x -= fa * (da.y / 2.0);
    Fi.y -= fa * (-da.x / 2.0);
    if (LAST && act) A.F[q] = Fi;

    // ---- update!
    const double vx = T->vo * pcs.x + T->mu * Fi.x;
    const double vy = T->vo * pcs.y + T->mu * Fi.y;
    s_a[me] = make_double2(vx, vy);  // the neighbour reads of s_a are done
    lds_sync();
    if (lane < 2 * per) {
        const double *src = (const double *)s_a + 2 * (wb + (lane >> 1) * P.nmax) + (lane & 1);
        double s = 0.0;
#pragma unroll 4
        for (int k = 0; k < np2; k++) s += src[2 * k];
        s_r[wave][lane] = s;  // the area's reads are done
    }
    double l2 = 0.0;
    if (act) {
        double px = x.x + vx * P.dt, py = x.y + vy * P.dt;
        const double lx = px - x.x, ly = py - x.y;
        l2 = lx * lx + ly * ly;
        periodic_wrap(P, px, py);
        A.Pout[q] = make_double2(px, py);
        // the chunk of the new position; still clear inside the old one (by
        // more than the rounding of the chunk edges): the same
        const int r0 = ko >> 16, c0 = ko & 0xffff;
        const double ax = px - P.blx, ay = (-py + P.bly) + P.H;
        const double mg = 1e-12 * (P.L + P.H);
        if (!(ax >= (double)c0 * P.cl + mg && ax <= (double)(c0 + 1) * P.cl - mg && ay >= (double)r0 * P.ch + mg &&
              ay <= (double)(r0 + 1) * P.ch - mg)) {
            uint32_t flag = 0;
            int32_t rn, cc;
            cell_rc(P, P.rows, P.cols, P.cl, P.ch, px, py, &flag, MAVI_FLAG_OUT_OF_BOX, &rn, &cc);
            if (flag) atomicOr(A.flags + B.flag, flag);
            const int32_t kn = (rn << 16) | cc;
            if (kn != ko) {
                A.key[q] = kn;
                atomicSub(&A.ccnt[B.chunk + r0 * P.cols + c0], 1);
                if (atomicAdd(&A.ccnt[B.chunk + rn * P.cols + cc], 1) + 1 > P.nc) atomicOr(A.status, kRlCapacity);
            }
        }
    }

    // largest squared step (high word, rounded up; a non-finite step gives the
    // largest word)
    const uint32_t hi =
        wave_umax(l2 == l2 ? min((uint32_t)__double2hiint(l2) + 1u, 0x7ff00000u) : 0x7ff00000u);
    if (lane == 63) s_max[wave] = hi;

    // ---- polarisations: one lane per ring of the workgroup
    __syncthreads();
    if (wave != 0) return;
    if (lane == 0) {  // the largest since the block began
        uint32_t m = hi0;
#pragma unroll
        for (int w = 0; w < kRlWaves; w++) m = max(m, s_max[w]);
        if (m > hi0) A.bmax[block] = m;
    }
    for (int k = lane; k < kRlWaves * A.per; k += 64) {
        const RingScalars R = k < 64 ? s_ring[k] : ring_scalars<BATCH>(P0, A, block, k, step);
        if (R.np == 0) continue;  // no ring
        const int w = k / A.per, g = k - w * A.per;
        const double vcx = s_r[w][2 * g] / (double)R.np, vcy = s_r[w][2 * g + 1] / (double)R.np;
        const double speed = sqrt(vcx * vcx + vcy * vcy);
        double cr = 0.0;
        if (speed != 0.0) {
            cr = (R.cs * vcy - R.sn * vcx) / speed;
            if (fabs(cr) > 1.0) cr = cr > 0.0 ? 1.0 : -1.0;
        }
        const double d_theta = R.rate * asin(cr) * R.dt + R.noise;
        const double th = R.pol + d_theta;
        double sn, cn2;
        sincos(th, &sn, &cn2);
        A.pol[R.rg] = th;
        A.polcs[R.rg] = make_double2(cn2, sn);
    }
}

// The lists: one thread per particle, in cell order of the list grid (src[t]:
// the slot at place t), over the 3x3 cells around its own.  A batch's places
// lie in their replica's slot range (waves of one replica), greps holds the
// list grids and radii.
struct RLBuild {
    const double2 *pos;
    const int32_t *ID, *rtype;
    const RingType *types;
    const int32_t *src, *scell, *start;
    int32_t nslots;
    double rl2;
    int4 *head;
    int32_t *more;
    uint8_t *count;
    uint32_t *status;
    const Replica *reps, *greps;
    const int32_t *wave_rep;  // replica of 64 slots
};
template <bool BATCH>
__global__ __launch_bounds__(256) void k_rl_build(SysParams G0, SysParams P0, RLBuild A) {
    const int t = xcd_block() * blockDim.x + threadIdx.x;
    if (t >= A.nslots) return;
    const int rep = BATCH ? uniform(A.wave_rep[t >> 6]) : 0;
    const SysParams &P = BATCH ? A.reps[rep].P : P0;
    const SysParams &G = BATCH ? A.greps[rep].P : G0;
    const RLBase B = BATCH ? rl_base(A.reps[rep], rep) : RLBase{};
    const double rl2 = BATCH ? A.greps[rep].list2 : A.rl2;
    const int gbase = BATCH ? A.greps[rep].cbase : 0;
    const int32_t *start = A.start + gbase;
    const int q = A.src[t], c = A.scell[t] - gbase;
    const int id = A.ID[q] - B.id;
    if (id < 0) return;  // a padding slot
    const double2 x = A.pos[q];
    const int ring = id / P.nmax;
    const int np = A.types[B.type + (P.typed ? A.rtype[B.ring + ring] : 0)].np;
    const int row = c / G.cols, col = c - row * G.cols;
    int32_t h[kRlHead] = {-1, -1, -1, -1};
    int n = 0;
    auto run = [&](int a, int b) {
        for (int u = a; u < b; u++) {
            const int j = A.src[u];
            if (j == q) continue;
            const double2 d = cdiff(P, x, A.pos[j]);
            if (!(d.x * d.x + d.y * d.y <= rl2)) continue;
            const int idj = A.ID[j] - B.id, rj = idj / P.nmax;
            if (rj == ring) {
                const int diff = abs(id - idj);
                if (diff == 1 || diff == np - 1) continue;  // bonded neighbours do not interact
            }
            const int32_t e = j | ((P.typed ? A.rtype[B.ring + rj] : 0) << kRlSlotBits);
#pragma unroll
            for (int s = 0; s < kRlHead; s++) h[s] = n == s ? e : h[s];
            if (n >= kRlHead && n < kRlMax) A.more[(int64_t)(n - kRlHead) * A.nslots + q] = e;
            n++;
        }
    };
    for (int d = -1; d <= 1; d++) {
        int rw = row + d;
        rw = rw < 0 ? rw + G.rows : (rw >= G.rows ? rw - G.rows : rw);
        const int32_t *sr = start + rw * G.cols;
        if (col > 0 && col < G.cols - 1) {
            run(sr[col - 1], sr[col + 2]);
        } else {
            run(sr[col == 0 ? 0 : col - 1], sr[col == 0 ? 2 : G.cols]);
            run(sr[col == 0 ? G.cols - 1 : 0], sr[col == 0 ? G.cols : 1]);
        }
    }
    if (n > kRlMax) {
        atomicOr(A.status, kRlOverflow);
        n = kRlMax;
    }
    A.head[q] = make_int4(h[0], h[1], h[2], h[3]);
    A.count[q] = (uint8_t)n;
}

// After a build: reference chunks and counts (capacity as the binning checks
// it), the build positions, cos and sin of the polarisations.
template <bool BATCH>
__global__ void k_rl_keys(SysParams P0, int32_t nslots, int32_t nrings, const Replica *__restrict__ reps,
                          const int32_t *__restrict__ wave_rep, const double2 *__restrict__ pos,
                          int32_t *__restrict__ key, int32_t *__restrict__ ccnt, double2 *__restrict__ xb,
                          const double *__restrict__ pol, double2 *__restrict__ polcs, uint32_t *__restrict__ flags) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nrings) {
        double sn, cs;
        sincos(pol[s], &sn, &cs);
        polcs[s] = make_double2(cs, sn);
    }
    if ((s & ~63) >= nslots) return;  // whole waves
    const int rep = BATCH ? uniform(wave_rep[s >> 6]) : 0;
    const SysParams &P = BATCH ? reps[rep].P : P0;
    const RLBase B = BATCH ? rl_base(reps[rep], rep) : RLBase{};
    const bool valid = s - B.slot < P.na;
    uint32_t flag = 0;
    int32_t r = 0, c = 0, k = -1;
    double2 p = make_double2(0.0, 0.0);
    if (valid) {
        p = pos[s];
        cell_rc(P, P.rows, P.cols, P.cl, P.ch, p.x, p.y, &flag, MAVI_FLAG_OUT_OF_BOX, &r, &c);
        k = B.chunk + r * P.cols + c;
    }
    const int32_t rank = wave_arrival_rank(valid, k, ccnt);
    if (valid && rank + 1 > P.nc) flag |= MAVI_FLAG_OVERFLOW;
    if (flag) atomicOr(flags + B.flag, flag);
    if (!valid) return;
    key[s] = (r << 16) | c;
    xb[s] = p;
}

// Block start: the state to roll back to, the step maxima cleared, the step
// counter taken over.
struct RLSnap {
    double2 *pos, *cms, *cms_next;
    double *pol;
    uint32_t *flags;
};
__global__ void k_rl_block_start(int32_t na, int32_t nrings, const double2 *__restrict__ pos,
                                 const double *__restrict__ pol, const double2 *__restrict__ cms,
                                 const double2 *__restrict__ cms_next, RLSnap S, uint32_t *__restrict__ bmax,
                                 int32_t nbmax, unsigned long long *__restrict__ out,
                                 const uint32_t *__restrict__ flags, int32_t nflags, const unsigned long long *__restrict__ counter,
                                 unsigned long long *__restrict__ c0) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < na) S.pos[i] = pos[i];
    if (i < nrings) {
        S.pol[i] = pol[i];
        S.cms[i] = cms[i];
        S.cms_next[i] = cms_next[i];
    }
    if (i < nbmax) bmax[i] = 0u;
    if (i < nflags) S.flags[i] = flags[i];
    if (i == 0) {
        out[0] = out[1] = 0ull;
        *c0 = *counter;
    }
}

// Block end: out[0] <- the largest squared step (bits), out[1] <- the largest
// squared displacement from the build, out[2] <- the status.  At most 64
// workgroups, so the maxima of one word take few atomics.
constexpr int kRlMeasureBlocks = 64;
template <bool BATCH>
__global__ __launch_bounds__(1024) void k_rl_measure(SysParams P0, int32_t nslots, const Replica *__restrict__ reps,
                                                     const int32_t *__restrict__ wave_rep,
                                                     const double2 *__restrict__ pos,
                                                     const double2 *__restrict__ xb,
                                                     const uint32_t *__restrict__ bmax, int32_t nbmax,
                                                     const uint32_t *__restrict__ status,
                                                     unsigned long long *__restrict__ out) {
    double d2 = 0.0;
    uint32_t hi = 0u;
    const int g = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    for (int s = g; s < nslots; s += stride) {
        const Replica *Q = BATCH ? reps + uniform(wave_rep[s >> 6]) : nullptr;
        if (BATCH && s - Q->pbase >= Q->P.na) continue;  // padding
        const double2 d = cdiff(BATCH ? Q->P : P0, pos[s], xb[s]);
        const double v = d.x * d.x + d.y * d.y;
        d2 = v == v ? fmax(d2, v) : INFINITY;
    }
    for (int s = g; s < nbmax; s += stride) hi = max(hi, bmax[s]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        d2 = fmax(d2, __shfl_xor(d2, o, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
    }
    // one atomic per workgroup and word (one per wave, 1024 on an address: 30 us)
    __shared__ double s_d[16];
    __shared__ uint32_t s_h[16];
    if (lane_id() == 0) {
        s_d[threadIdx.x >> 6] = d2;
        s_h[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) {
            d2 = fmax(d2, s_d[w]);
            hi = max(hi, s_h[w]);
        }
        atomicMax(&out[0], (unsigned long long)hi << 32);
        atomicMax(&out[1], (unsigned long long)__double_as_longlong(d2));
    }
    if (g == 0) out[2] = *status;
}

__global__ void k_rl_copy_counter(const unsigned long long *__restrict__ src, unsigned long long *__restrict__ dst) {
    if (threadIdx.x == 0 && blockIdx.x == 0) dst[0] = src[0];
}

__global__ void k_rl_restore(int32_t na, int32_t nrings, RLSnap S, double2 *__restrict__ pos, double *__restrict__ pol,
                             double2 *__restrict__ cms, double2 *__restrict__ cms_next, uint32_t *__restrict__ flags,
                             int32_t nflags, uint32_t *__restrict__ status) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < na) pos[i] = S.pos[i];
    if (i < nrings) {
        pol[i] = S.pol[i];
        cms[i] = S.cms[i];
        cms_next[i] = S.cms_next[i];
    }
    if (i < nflags) flags[i] = S.flags[i];
    if (i == 0) *status = 0u;
}

int rl_blocks(const SysParams &P) { return nblk(nblk(P.nrings, 64 / P.nmax), kRlWaves); }

RLSnap rl_snap(const RList &N) { return RLSnap{N.psnap, N.csnap, N.nsnap, N.polsnap, N.fsnap}; }

// What the block loop needs of a system alone or of a batch's rings replicas.
struct RLSys {
    mavi_ctx *ctx;
    RList *N;
    SysParams P;  // alone; a batch: unused
    int32_t nslots, nrings, nflags;
    double2 **Pc;
    int *cur;
    double *pol;
    double2 *cms, *cms_next;
    uint32_t *flags;
    unsigned long long *counter;
    const Replica *reps;       // batch: replica table, replica of 64 slots
    const int32_t *wave_rep;
    bool graphs;
    mavi_sys *s;
    BatchSub *b;
};
RLSys rl_env(mavi_sys *s) {
    return RLSys{s->ctx, s->rl, s->P, s->P.na, s->P.nrings, 1, s->P_, &s->cur, s->pol, s->cms, s->cms_next, s->flags,
                 s->counter, nullptr, nullptr, s->use_graphs && !s->prof, s, nullptr};
}
RLSys rl_env(BatchSub *b) {
    return RLSys{b->ctx, b->rl, SysParams{}, (int32_t)b->nslots, (int32_t)b->nrings, (int32_t)b->reps.size(), b->P_,
                 &b->cur, b->pol, b->cms, b->cms_next, b->flags, b->counter, b->d_reps, b->wave_rep,
                 b->use_graphs && !b->prof, nullptr, b};
}

hipError_t rl_step(const RLSys &E, bool last, hipStream_t st) {
    RList &N = *E.N;
    const int c = *E.cur;
    RLArgs A{};
    A.Pin = E.Pc[c];
    A.Pout = E.Pc[1 - c];
    A.head = (const int4 *)N.head;
    A.more = N.more;
    A.count = N.count;
    A.key = N.key;
    A.ccnt = N.ccnt;
    A.pol = E.pol;
    A.polcs = N.polcs;
    A.cms = E.cms;
    A.cms_next = E.cms_next;
    A.bmax = N.bmax;
    A.flags = E.flags;
    A.status = N.status;
    A.cin = N.counter + N.ph;
    A.cout = N.counter + (1 - N.ph);
    A.stride = E.nslots;
    A.per = N.per;
    const dim3 grid(N.nbmax);
    if (mavi_sys *s = E.s) {
        ProfScope ps(s, MAVI_PROF_RINGS, st);
        A.F = s->F;
        A.slot_of = N.full ? nullptr : s->slot_of;
        A.areas = s->areas;
        A.cpos = s->cpos;
        A.rtype = s->rtype;
        A.types = s->types;
        A.inter = N.uniform ? nullptr : s->inter;
        A.uni = s->host_inter[0];
        A.seed = s->seed;
        if (last) hipLaunchKernelGGL((k_rl_step<true, false>), grid, dim3(kRlWG), 0, st, s->P, A);
        else hipLaunchKernelGGL((k_rl_step<false, false>), grid, dim3(kRlWG), 0, st, s->P, A);
    } else {
        BatchSub *b = E.b;
        BatchProf ps(b, MAVI_PROF_RINGS, st);
        A.F = b->F;
        A.slot_of = N.full ? nullptr : b->slot_of;
        A.areas = b->areas;
        A.cpos = b->cpos;
        A.rtype = b->rtype;
        A.types = b->types;
        A.inter = b->inter;
        A.reps = b->d_reps;
        A.wave_rep = b->ring_wave_rep;
        A.nwaves = b->nring_waves;
        if (last) hipLaunchKernelGGL((k_rl_step<true, true>), grid, dim3(kRlWG), 0, st, SysParams{}, A);
        else hipLaunchKernelGGL((k_rl_step<false, true>), grid, dim3(kRlWG), 0, st, SysParams{}, A);
    }
    N.ph = 1 - N.ph;
    *E.cur = 1 - c;
    return hipGetLastError();
}

// Eight steps from (copy, counter word) captured once.
hipError_t rl_graph(const RLSys &E, hipStream_t st, hipGraphExec_t *out) {
    RList &N = *E.N;
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return e;
    const int c0 = *E.cur, ph0 = N.ph;
    hipError_t e1 = hipSuccess;
    for (int k = 0; k < kRlGraphSteps && e1 == hipSuccess; k++) e1 = rl_step(E, false, st);
    e = hipStreamEndCapture(st, &g);
    *E.cur = c0;
    N.ph = ph0;
    if (e1 != hipSuccess) e = e1;
    if (e == hipSuccess) e = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
    if (g) (void)hipGraphDestroy(g);
    return e;
}

// State in ring order (both copies' ids, slot_of the identity over active ids).
hipError_t rl_ring_order(const RLSys &E, hipStream_t st) {
    RList &N = *E.N;
    if (N.ordered) return hipSuccess;
    hipError_t e;
    if (mavi_sys *s = E.s) {
        e = mavi::launch_unpermute(s, false, false, st);
        s->cur = 0;
        if (e == hipSuccess) e = mavi::launch_iota_state(s, st);
        if (e == hipSuccess)
            e = hipMemcpyAsync(s->ID_[1], s->ID_[0], sizeof(int32_t) * (size_t)s->P.na, hipMemcpyDeviceToDevice, st);
        s->sorted = false;
    } else {
        e = mavi::launch_batch_ring_order(E.b, st);
    }
    N.ordered = e == hipSuccess;
    return e;
}

hipError_t rl_rebuild(const RLSys &E, hipStream_t st) {
    RList &N = *E.N;
    mavi_sys *s = E.s;
    BatchSub *b = E.b;
    hipError_t e = s ? mavi::drop_keys(s, st) : hipSuccess;
    if (N.scan_stale) {
        if (e == hipSuccess) e = mavi::launch_fill_i32((int32_t *)N.scan_ticket, 0, 2, st);
        if (e == hipSuccess) e = mavi::launch_fill_i32((int32_t *)N.scan_state, 0, 2 * (int64_t)N.scan_words, st);
        N.scan_stale = e != hipSuccess;
    }
    if (e == hipSuccess) e = rl_ring_order(E, st);
    if (e == hipSuccess)
        e = s ? mavi::launch_cell_order(s, N.G, N.scan_ticket, N.scan_state, st)
              : mavi::launch_batch_cell_order(b, (const Replica *)N.greps, N.gcells, N.scan_ticket, N.scan_state, st);
    if (e != hipSuccess) return e;
    const int c = *E.cur;
    RLBuild A{};
    A.pos = E.Pc[c];
    A.ID = s ? s->ID_[c] : b->ID_[c];
    A.rtype = s ? s->rtype : b->rtype;
    A.types = s ? s->types : b->types;
    A.src = s ? s->src : b->src;
    A.scell = s ? s->scell : b->scell;
    A.start = s ? s->start : b->start;
    A.nslots = E.nslots;
    A.rl2 = N.rl2;
    A.head = (int4 *)N.head;
    A.more = N.more;
    A.count = N.count;
    A.status = N.status;
    A.reps = E.reps;
    A.greps = (const Replica *)N.greps;
    A.wave_rep = E.wave_rep;
    const dim3 gb(nblk(E.nslots, 256)), gk(nblk(std::max(E.nslots, E.nrings), 256));
    if (s) hipLaunchKernelGGL(k_rl_build<false>, gb, dim3(256), 0, st, N.G, s->P, A);
    else hipLaunchKernelGGL(k_rl_build<true>, gb, dim3(256), 0, st, SysParams{}, SysParams{}, A);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = mavi::launch_fill_i32(N.ccnt, 0, s ? s->P.ncell : b->ncells, st)) != hipSuccess) return e;
    if (s)
        hipLaunchKernelGGL(k_rl_keys<false>, gk, dim3(256), 0, st, s->P, E.nslots, E.nrings, nullptr, nullptr,
                           E.Pc[c], N.key, N.ccnt, N.xb, E.pol, N.polcs, E.flags);
    else
        hipLaunchKernelGGL(k_rl_keys<true>, gk, dim3(256), 0, st, SysParams{}, E.nslots, E.nrings, E.reps, E.wave_rep,
                           E.Pc[c], N.key, N.ccnt, N.xb, E.pol, N.polcs, E.flags);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    N.valid = true;
    N.d_start = 0.0;
    N.rebuilds++;
    return hipSuccess;
}

double rl_step_est(const RList &N) { return std::max(N.step_hist[0], std::max(N.step_hist[1], N.step_hist[2])); }

// Steps from a block start that keep d + (steps - 1) x step within half_skin, at
// a step 1.08 times the estimate; d: the largest displacement there.
int64_t rl_fit(const RList &N, double d) {
    const double r = (N.half_skin - d) / (1.08 * rl_step_est(N));
    if (!(r < 1e9)) return INT64_MAX;
    return (int64_t)floor(r) + 1;
}
int64_t rl_room(const RList &N) { return rl_fit(N, N.d_start); }

// A state whose lists would serve no more steps than this goes to the gather.  us for
// 200 steps of jammed mixtures with 6, 3, 2 and 1 here (gather: 6890 .. 11470): 2k particles
// at dt 0.01 6060, 6040, 3970, 4360; 20k at 0.005 6590, 4910, 4940, 5090, at 0.02
// 6780, 6770, 6760, 8420; 200k at 0.005 10560, 7490, 7440, 7650.
constexpr int64_t kRlMinFit = 2;
constexpr int64_t kRlMinBlock = 6;  // shorter blocks cost more than the rebuild they put off
constexpr int64_t kRlNewBlock = 8;  // most steps of the first block on a new state

// The lists give the state to the gather for a while.
void rl_back_off(RList &N) {
    N.backoff = N.ran > 4 * N.backoff ? kRlWaitMin : std::clamp(2 * N.backoff, kRlWaitMin, kRlWaitMax);
    N.wait = N.backoff;
    N.ran = 0;
}

// Blocks of steps with one read back each (see the top); *left > 0: the chunk
// gather runs the rest.
int rl_run(const RLSys &E, int64_t nsteps, int64_t *left) {
    mavi_ctx *ctx = E.ctx;
    hipStream_t st = ctx->stream;
    RList &N = *E.N;
    *left = 0;
    const int span = std::max(std::max(E.nslots, E.nrings), std::max(N.nbmax, E.nflags));
    int64_t k = 0;
    bool first = N.first;  // on a new state
    N.first = false;
    while (k < nsteps) {
        const double est = rl_step_est(N);
        if (N.block == 0 && N.valid && est > 0.0) {
            // lists that serve few more steps are rebuilt, unless these are the
            // call's last or new ones would serve few
            const int64_t few = std::min(std::min(kRlMinBlock, nsteps - k), std::max<int64_t>(1, rl_fit(N, 0.0) / 4));
            if (rl_room(N) < few) N.valid = false;
        }
        if (N.block == 0 && !N.valid && !first && est > 0.0 && rl_fit(N, 0.0) <= kRlMinFit) {
            rl_back_off(N);
            *left = nsteps - k;
            return MAVI_OK;
        }
        if (!N.valid) HIPCHK(ctx, rl_rebuild(E, st));
        int64_t want = N.block_now;
        if (N.block == 0) {
            if (first || !(est > 0.0)) want = std::min<int64_t>(want, kRlNewBlock);
            if (est > 0.0) want = std::min(want, std::max<int64_t>(1, rl_room(N)));
        }
        const int64_t blk = std::min<int64_t>(want, nsteps - k);
        const int cur0 = *E.cur;
        N.ph = 0;
        hipLaunchKernelGGL(k_rl_block_start, dim3(nblk(span, 256)), dim3(256), 0, st, E.nslots, E.nrings, E.Pc[cur0],
                           E.pol, E.cms, E.cms_next, rl_snap(N), N.bmax, N.nbmax, N.out, E.flags, E.nflags, E.counter,
                           N.counter);
        HIPCHK(ctx, hipGetLastError());
        const bool ends = k + blk == nsteps;  // the block's last step leaves the call's outputs
        const int64_t plain = ends ? blk - 1 : blk;
        int64_t done = 0;
        while (done < plain) {
            if (E.graphs && done + kRlGraphSteps <= plain) {
                hipGraphExec_t &g = N.graph[*E.cur][N.ph];
                if (!g) HIPCHK(ctx, rl_graph(E, st, &g));
                HIPCHK(ctx, hipGraphLaunch(g, st));
                done += kRlGraphSteps;  // an even number: the copies and the counter words are where they were
            } else {
                HIPCHK(ctx, rl_step(E, false, st));
                done++;
            }
        }
        if (ends) HIPCHK(ctx, rl_step(E, true, st));
        const int mb = std::min(nblk(std::max(E.nslots, N.nbmax), 1024), kRlMeasureBlocks);
        auto measure = E.reps ? &k_rl_measure<true> : &k_rl_measure<false>;
        hipLaunchKernelGGL(measure, dim3(mb), dim3(1024), 0, st, E.P, E.nslots, E.reps, E.wave_rep, E.Pc[*E.cur], N.xb,
                           N.bmax, N.nbmax, N.status, N.out);
        HIPCHK(ctx, hipGetLastError());
        HIPCHK(ctx, hipMemcpyAsync(N.host, N.out, 3 * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
        HIPCHK(ctx, hipStreamSynchronize(st));
        const double step = sqrt(__builtin_bit_cast(double, N.host[0]));
        const double d_end = sqrt(__builtin_bit_cast(double, N.host[1]));
        const uint32_t status = (uint32_t)N.host[2];
        if (first) N.step_hist[0] = N.step_hist[1] = N.step_hist[2] = 0.0;  // of the state before
        first = false;
        N.step_hist[N.step_i] = step;
        N.step_i = (N.step_i + 1) % 3;
        // The block evaluated y_0 .. y_{T-1} and moved to y_T: y_t is within
        // min(d_start + t step, d_end + (T - t) step) of its build position.
        const double T = (double)blk;
        const bool finite = std::isfinite(step) && std::isfinite(d_end);
        const double bound = std::min(N.d_start + (T - 1.0) * step, 0.5 * (N.d_start + d_end + T * step));
        if (status || !finite || !(bound <= N.half_skin)) {
            *E.cur = cur0;
            hipLaunchKernelGGL(k_rl_restore, dim3(nblk(span, 256)), dim3(256), 0, st, E.nslots, E.nrings, rl_snap(N),
                               E.Pc[cur0], E.pol, E.cms, E.cms_next, E.flags, E.nflags, N.status);
            HIPCHK(ctx, hipGetLastError());
            N.valid = false;
            N.rollbacks++;
            // (one step from a fresh build evaluates the build positions: its
            // bound is 0, so a block can always shrink to one that passes)
            if (status || !finite) {
                // the chunk gather takes over: until a new state if a list
                // overflowed, for a while if a chunk may have (it checks
                // exactly: a particle may have been counted in before another
                // of its step was counted out), for this call if the state is
                // not finite
                *left = nsteps - k;
                if (status & kRlOverflow) {
                    N.disabled = true;
                    N.skip = N.skip_next;
                    N.skip_next = std::min(2 * N.skip_next, 64);
                } else if (!finite) {
                    N.wait = *left;
                } else {
                    rl_back_off(N);
                }
                if (!finite) N.step_hist[0] = N.step_hist[1] = N.step_hist[2] = 0.0;
                return MAVI_OK;
            }
            if (N.block != 0 && N.block_now > 1) N.block_now = std::max(1, N.block_now / 2);
            continue;
        }
        hipLaunchKernelGGL(k_rl_copy_counter, dim3(1), dim3(64), 0, st, N.counter + N.ph, E.counter);
        HIPCHK(ctx, hipGetLastError());
        k += blk;
        N.ran += blk;
        N.skip_next = 1;
        N.d_start = d_end;
        if (N.block != 0 && d_end + 1.2 * step * (double)N.block_now > N.half_skin) N.valid = false;
        const int32_t cap = N.block == 0 ? kNlBlockCap : N.block;
        if (N.block_now < cap) N.block_now = std::min(cap, 2 * N.block_now);
    }
    return MAVI_OK;
}

}  // namespace

namespace mavi {

// Whether a rings system can run on lists.
static bool rl_fits(const SysParams &P, double list2) {
    if (P.potential != MAVI_POT_RINGS || P.nwalls > 0 || !P.periodic || P.na <= 0) return false;
    // k_rl_step has a lane for each of a wave's three sums a ring, which rings of
    // two (32 to a wave) have more of than lanes; taking turns cost all others
    // up to 0.8 % of a step
    if (P.nmax < 3 || P.nmax > 32) return false;
    if (P.na > kRlSlotMask || P.ntypes > 32) return false;
    if (P.cols < 3 || P.rows < 3 || P.rows > 32767 || P.cols > 65535) return false;
    const double range = sqrt(list2);
    if (!(range > 0.0) || !(range < INFINITY)) return false;
    // every pair within range is in adjacent chunks at the binned positions
    return P.cl >= range * (1.0 + 1e-12) && P.ch >= range * (1.0 + 1e-12);
}

// The list grid: cells at least range + skin wide.  false: the box holds fewer
// than three a side.
static bool rl_grid(const SysParams &P, double range, double skin_frac, SysParams &G, double &rl2, double &half_skin) {
    const double skin = skin_frac * range;
    const double rl = (range + skin) * (1.0 + 1e-9);
    rl2 = rl * rl;
    half_skin = 0.5 * skin * (1.0 - 1e-9);
    G = P;
    G.cols = P.cl >= rl ? P.cols : (int32_t)floor(P.L / rl);
    G.rows = P.ch >= rl ? P.rows : (int32_t)floor(P.H / rl);
    G.cl = P.L / (double)std::max(G.cols, 1);
    G.ch = P.H / (double)std::max(G.rows, 1);
    G.ncell = G.cols * G.rows;
    G.nc = P.na;
    return G.cols >= 3 && G.rows >= 3;
}

bool rl_eligible(const mavi_sys *s) { return rl_fits(s->P, s->list2); }

// skin as a fraction of the range
bool rl_set_skin(mavi_sys *s, double skin_frac) {
    RList &N = *s->rl;
    N.fits = rl_grid(s->P, sqrt(s->list2), skin_frac, N.G, N.rl2, N.half_skin);
    N.valid = false;
    rl_reset(N);
    N.scan_stale = true;
    return N.fits;
}

static hipError_t rl_buffers(RList &N, int64_t nslots, int64_t nrings, int64_t ncells, int64_t nflags,
                             hipStream_t st) {
    N.scan_words = (int32_t)((ncells + 1 + kScanTileMin - 1) / kScanTileMin) + 1;
    // one allocation for all: a system is made with few calls
    struct Part {
        void **p;
        size_t bytes;
    } parts[] = {
        {(void **)&N.head, sizeof(int32_t) * 4 * nslots},
        {(void **)&N.more, sizeof(int32_t) * (kRlMax - kRlHead) * nslots},
        {(void **)&N.count, sizeof(*N.count) * nslots},
        {(void **)&N.key, sizeof(*N.key) * nslots},
        {(void **)&N.ccnt, sizeof(*N.ccnt) * ncells},
        {(void **)&N.xb, sizeof(*N.xb) * nslots},
        {(void **)&N.psnap, sizeof(*N.psnap) * nslots},
        {(void **)&N.csnap, sizeof(*N.csnap) * nrings},
        {(void **)&N.nsnap, sizeof(*N.nsnap) * nrings},
        {(void **)&N.polsnap, sizeof(*N.polsnap) * nrings},
        {(void **)&N.fsnap, sizeof(*N.fsnap) * nflags},
        {(void **)&N.polcs, sizeof(*N.polcs) * nrings},
        {(void **)&N.bmax, sizeof(*N.bmax) * N.nbmax},
        {(void **)&N.status, sizeof(*N.status)},
        {(void **)&N.counter, sizeof(*N.counter) * 2},
        {(void **)&N.out, sizeof(*N.out) * 3},
        {(void **)&N.scan_ticket, sizeof(*N.scan_ticket)},
        {(void **)&N.scan_state, sizeof(*N.scan_state) * N.scan_words},
    };
    size_t total = 0;
    for (const Part &q : parts) total += (q.bytes + 255) / 256 * 256;
    hipError_t e = dalloc(&N.arena, (int64_t)total, st);
    size_t at = 0;
    for (const Part &q : parts) {
        if (e == hipSuccess) *q.p = N.arena + at;
        at += (q.bytes + 255) / 256 * 256;
    }
    return e;
}

static bool rl_uniform(const RingInter *I, int n) {
    for (int k = 1; k < n; k++)
        if (I[k].k_rep != I[0].k_rep || I[k].k_atr != I[0].k_atr || I[k].dist_eq != I[0].dist_eq ||
            I[k].dist_max != I[0].dist_max)
            return false;
    return true;
}

static void rl_drop_graphs(RList &N, hipStream_t st) {
    for (auto &row : N.graph)
        for (auto &g : row) {
            if (!g) continue;
            (void)hipStreamSynchronize(st);
            (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
}

static void rl_release(RList *&rl, hipStream_t st) {
    if (!rl) return;
    RList &N = *rl;
    rl_drop_graphs(N, st);
    dfree(N.arena);
    if (N.greps) (void)hipFree(N.greps);
    delete rl;
    rl = nullptr;
}

hipError_t rl_alloc(mavi_sys *s, hipStream_t st) {
    s->rl = new RList();
    RList &N = *s->rl;
    rl_set_skin(s, kRlSkin);
    N.uniform = rl_uniform(s->host_inter.data(), (int)s->host_inter.size());
    N.full = s->P.na == s->P.n;
    N.per = 64 / s->P.nmax;
    N.nbmax = rl_blocks(s->P);
    if ((N.host = pin_words(s->ctx, s->pin)) == nullptr) return hipErrorOutOfMemory;
    return rl_buffers(N, s->P.na, s->P.nrings, s->P.ncell, 1, st);
}

void rl_drop_graph(mavi_sys *s) {
    if (s->rl) rl_drop_graphs(*s->rl, s->ctx->stream);
}

void rl_free(mavi_sys *s) { rl_release(s->rl, s->ctx->stream); }

void rlb_drop_graph(BatchSub *b) {
    if (b->rl) rl_drop_graphs(*b->rl, b->ctx->stream);
}

void rlb_free(BatchSub *b) { rl_release(b->rl, b->ctx->stream); }

// The lists of a batch's rings replicas: one block length and one displacement
// bound for all (the smallest half skin), a list grid per replica.  No lists
// if some replica is not eligible.
hipError_t rlb_alloc(BatchSub *b, hipStream_t st) {
    if (b->nslots > kRlSlotMask) return hipSuccess;
    std::vector<Replica> g(b->reps);
    int64_t gcells = 0;
    double half = INFINITY;
    bool full = true;
    int per = 1;
    for (Replica &Q : g) {
        const double range = sqrt(Q.list2);
        SysParams G = Q.P;
        double rl2, hs;
        if (!rl_fits(Q.P, Q.list2) || !rl_grid(Q.P, range, kRlSkin, G, rl2, hs)) return hipSuccess;
        full = full && Q.P.na == Q.P.n;
        per = std::max(per, 64 / Q.P.nmax);
        half = std::min(half, hs);
        Q.P = G;
        Q.list2 = rl2;
        Q.cbase = (int32_t)gcells;
        gcells += G.ncell + 1;  // and its pad cell
    }
    b->rl = new RList();
    RList &N = *b->rl;
    N.half_skin = half;
    N.per = per;
    N.gcells = gcells;
    N.fits = true;
    N.full = full;
    N.nbmax = nblk(b->nring_waves, kRlWaves);
    N.host = pin_words(b->ctx, *b->pin);
    hipError_t e = N.host ? hipSuccess : hipErrorOutOfMemory;
    if (e == hipSuccess) e = rl_buffers(N, b->nslots, b->nrings, b->ncells, (int64_t)b->reps.size(), st);
    if (e == hipSuccess) e = hipMalloc(&N.greps, sizeof(Replica) * g.size());
    if (e == hipSuccess) e = hipMemcpyAsync(N.greps, g.data(), sizeof(Replica) * g.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    return e;
}

bool rl_allowed(const mavi_sys *s) { return s->rl && s->rl->on && s->rl->fits && !s->neigh_on && !s->var; }

bool rl_active(const mavi_sys *s) { return rl_allowed(s) && !s->rl->disabled; }

bool rl_take(RList &N, int64_t n) {
    if (N.renewed) {
        N.renewed = false;
        N.first = true;
        N.wait = std::min(N.wait, kRlWaitNew);
        if (N.disabled && --N.skip <= 0) N.disabled = false;
    }
    if (N.disabled || N.wait > 0) return false;
    return n >= kRlMinCall || (N.valid && (N.block != 0 || rl_room(N) >= n));
}

int64_t rl_turn(RList &N, int64_t n, int64_t unit) {
    if (N.disabled || N.wait <= 0) return n;
    n = std::min(n, (N.wait + unit - 1) / unit * unit);
    N.wait -= n;
    return n;
}

void rl_reset(RList &N) {
    N.disabled = false;
    N.skip_next = 1;
    N.wait = N.backoff = 0;
}

int rl_steps(mavi_sys *s, int64_t nsteps, int64_t *left) {
    const int rc = rl_run(rl_env(s), nsteps, left);
    s->sorted = false;  // not in chunk order
    return rc;
}

int rlb_steps(BatchSub *b, int64_t nsteps, int64_t *left) { return rl_run(rl_env(b), nsteps, left); }

}  // namespace mavi
