// mavi_batch.h -- replica batches: the replica table and one sub-batch (the
// plain replicas or the rings replicas) with its device arrays.
#pragma once
#include <vector>

#include "mavi_internal.h"

struct Replica {
    SysParams P;
    int32_t pbase, npad;  // first sorted slot (multiple of 64), padded slot count
    int32_t nbase;        // first particle id
    int32_t cbase;        // first chunk; cbase + P.ncell is the pad chunk
    int32_t rbase;        // first ring (even; rings only)
    int32_t tbase, ibase; // first ring type / interaction entry
    int32_t abase;        // first entry of the active id list (rings only)
    int64_t cpbase;       // first continuous position (rings only)
    double list2;         // squared candidate-list range
    uint64_t seed;
    float inv_nmax;
    int32_t kind;         // 0 LJ, 1 HarmTrunc, 2 rings
    int32_t rwbase;       // first wave of the ring kernel (rings only)
    int32_t uniform;      // one interaction for all type pairs (rings only)
};

enum { KIND_LJ = 0, KIND_HT = 1, KIND_RINGS = 2, NKIND = 3 };

// The replicas of one family, with their own slots, ids, chunks and rings
// numbered from 0.
struct BatchSub {
    mavi_ctx *ctx = nullptr;
    PinBuf *pin = nullptr;  // the batch's
    bool rings = false;
    std::vector<int32_t> global;  // batch index of each replica
    std::vector<Replica> reps;
    int64_t nids = 0, nactive = 0, nslots = 0, ncells = 0, nrings = 0;
    SysParams G{};  // na = nslots, ncell = ncells: the sort over all replicas
    std::vector<uint8_t *> blocks;  // the allocations that hold all device arrays below
    // per-kind wave lists
    int2 *items[NKIND] = {nullptr, nullptr, nullptr};
    int32_t nitems[NKIND] = {0, 0, 0};
    int32_t *ring_wave_rep = nullptr;
    int32_t nring_waves = 0;
    Replica *d_reps = nullptr;
    int32_t *wave_rep = nullptr;
    // state (same roles as in mavi_sys)
    double2 *P_[2] = {nullptr, nullptr}, *V_[2] = {nullptr, nullptr};
    int32_t *ID_[2] = {nullptr, nullptr};
    double2 *F = nullptr, *P2 = nullptr, *F1 = nullptr;
    int32_t *key = nullptr, *rank = nullptr, *src = nullptr, *scell = nullptr, *sid = nullptr, *slot_of = nullptr;
    int32_t *cnt = nullptr, *start = nullptr;
    unsigned long long *scan_state = nullptr, *scan_ticket = nullptr;
    uint32_t *flags = nullptr;
    // force reuse
    int32_t *perm = nullptr, *needc = nullptr;
    uint32_t *epoch = nullptr, *rvalid = nullptr;
    bool keys_ready = false;  // the last second evaluation did the next binning's first pass
    unsigned long long *counter = nullptr;
    int32_t *active_ids = nullptr;
    double2 *pos_id = nullptr, *vel_id = nullptr, *force_id = nullptr;
    double *pol = nullptr, *areas = nullptr;
    double2 *cms = nullptr, *cms_next = nullptr, *cpos = nullptr;
    int32_t *rtype = nullptr;
    RingType *types = nullptr;
    RingInter *inter = nullptr;
    int cur = 0;
    // execution shape
    int32_t wg = 256, listed = 0, graph_steps = 100;
    bool use_graphs = true;
    hipGraphExec_t graph = nullptr;
    RList *rl = nullptr;  // lists of the rings replicas, null if some replica is not eligible
    // profiling
    bool prof = false;
    ProfSlot profs[MAVI_PROF_NCLASS];
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
};

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

struct BatchProf {
    BatchSub *b;
    int which;
    hipStream_t st;
    BatchProf(BatchSub *b_, int w, hipStream_t st_) : b(b_), which(w), st(st_) {
        if (b->prof) (void)hipEventRecord(b->ev0, st);
    }
    ~BatchProf() {
        if (!b->prof) return;
        (void)hipEventRecord(b->ev1, st);
        if (hipEventSynchronize(b->ev1) == hipSuccess) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, b->ev0, b->ev1) == hipSuccess) {
                b->profs[which].ms += ms;
                b->profs[which].launches += 1;
            }
        }
    }
};

namespace mavi {
// Lists of the rings replicas (mavi_rlist.hip), as rl_* for a single system.
hipError_t rlb_alloc(BatchSub *b, hipStream_t st);
void rlb_free(BatchSub *b);
void rlb_drop_graph(BatchSub *b);
int rlb_steps(BatchSub *b, int64_t nsteps, int64_t *left);
// Counting sort of the slots on the list grids (greps: the replicas with their
// list grid as P and cbase), the state left where it is.
hipError_t launch_batch_cell_order(BatchSub *b, const Replica *greps, int64_t gcells, unsigned long long *ticket,
                                   unsigned long long *state, hipStream_t st);
// The state from wherever it is into ring order, both copies' ids too.
hipError_t launch_batch_ring_order(BatchSub *b, hipStream_t st);
}  // namespace mavi
