// Batched execution of many independent cases on one device.
//
// Every case keeps its own lattice, parameters and buffers resident in HBM.
// A batch step runs, for each group of cases of one tile shape, the phase pass
// of its cases and then their collide pass, one launch each: workgroups read a
// work item (case, tile origin) from a table built in XCD order, then a
// CaseView from a device array. Cases never exchange data, so each case's
// numbers do not depend on what else is in the batch, and the groups advance
// independently: they run side by side on a few streams (lanes), where one
// group's drain and its phase pass overlap another's collide pass.
#pragma once
#include <map>
#include <memory>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "fused.hpp"
#include "readback.hpp"
#include "state.hpp"

namespace mcb {

struct CaseState {
    mcb_params p{};
    Geo geo{};
    Phys phys{};
    int storage = MCB_STORE_FP32;
    int mode = COLLIDE_STEP;       // COLLIDE_STEP or COLLIDE_STEP_BGK
    Tiling tiling{64, 8, 16};
    bool own_tiling = false;        // set by the library's caller
    bool alone = false;             // a context's only case
    Tiling phase{64, 8, 16};        // tiles of the phase pass (phase_tiling16)
    Tiling sum{64, 8, 16};          // tiles of the sum of phi of stored 16-bit g (build_own_table)
    int cur = 0;                    // population buffer of the current state
    int parity_offset = 0;          // cur = batch parity ^ parity_offset
    long long steps = 0;            // steps taken since init
    void* f[2] = {nullptr, nullptr};
    void* g[2] = {nullptr, nullptr};
    float* phi[2] = {nullptr, nullptr};
    float* phi_last = nullptr;      // written by the most recent phase pass
    int gm = GM_POPULATIONS;        // FP32 at tau_g = 1: g in moment form (GMode)
    float* gmu[3] = {nullptr, nullptr, nullptr};
    float* gmn[3] = {nullptr, nullptr, nullptr};   // FP32 moment form: n, stored by the collide pass
    MassCell* mass = nullptr;       // 16-bit storage: mass-drift correction state
    MassQ* massq = nullptr;         // 16-bit storage in moment form: its correction state
    double* partial = nullptr;      // one FP64 partial per phase work item
    size_t partial_cap = 0;
    std::vector<std::pair<void*, size_t>> allocs;   // device blocks and their sizes
    size_t bytes = 0;
    int slot = 0;                   // index in the batch's view arrays
    // This case's tiles with case index 0 (its macro pass): [0, n_work) collide,
    // [n_work, n_work + n_phase) phase where its tiles differ.
    WorkItem* d_work = nullptr;
    size_t work_cap = 0;
    unsigned n_work = 0, n_phase = 0;

    // Buffers seen by the kernels at A/B parity q (q = cur before a step).
    CaseView view(int q) const;

    CaseState() = default;
    CaseState(const CaseState&) = delete;
    CaseState& operator=(const CaseState&) = delete;
    // Frees the device memory still listed in allocs (the owning batch makes
    // its device current and drains its stream first).
    ~CaseState();
};

// Host-side constants of a parameter set (host.cpp).
Phys host_phys(const mcb_params& p);
mcb_status host_validate(const mcb_params* p, std::string* why);

// Geometry of a lattice on the fused kernels: populations (not f as moments)
// in blocks (FP32) and, if asked for and worth it (pads_rows), in padded rows,
// as far as they fit the kernels' 32-bit buffers. 16-bit rows that one collide tile spans stay
// unpadded: the tile is one contiguous piece of memory (FP16, rows padded
// against not: 176^3 187 against 154 us per step, 144^3 134 against 125).
Geo fused_geo(const mcb_params& p, bool pad_rows);

// Device bytes of a case with these parameters (populations, phase field(s)
// and, at tau_g = 1, the moment form of g).
size_t case_bytes(const mcb_params& p, bool pad_rows = false);

class Batch {
public:
    Batch(int device, hipStream_t stream);
    ~Batch();
    Batch(const Batch&) = delete;
    Batch& operator=(const Batch&) = delete;

    // Allocate a case and set its initial state from phi (host, nx*ny*nz
    // floats), or from bubbles on the device (serving; bubble_phi_cell, the
    // bits of the host initialisation).
    // alone: a context's only case, on the tiles and rows of a lattice that has
    // the device to itself; case_bytes(p, true) of device memory where its rows
    // are padded (Geo::pitch), case_bytes(p) otherwise and where that does not fit.
    mcb_status add(const mcb_params& p, const float* phi_host, int* id, bool alone = false);
    mcb_status add_bubbles(const mcb_params& p, const mcb_bubble* bubbles, int n, float width, int* id,
                           bool alone = false);
    mcb_status remove(int id);
    mcb_status step(int nsteps);
    mcb_status macros(int id);
    mcb_status read(int id, int field, float* host, size_t n);
    mcb_status write(int id, int field, const float* host, size_t n);
    mcb_status reduce(int id, double* sum_phi, double* kinetic);
    mcb_status set_tiling(int id, const Tiling& t, bool by_caller = true);
    // State image of a case at a step boundary (state.hpp): size, save, load
    // into a case of the same parameters, or a new case from an image.
    mcb_status state_size(int id, size_t* bytes);
    mcb_status save_state(int id, void* buf, size_t bytes);
    mcb_status load_state(int id, const void* buf, size_t bytes);
    mcb_status add_state(const void* buf, size_t bytes, int* id);
    mcb_status synchronize();
    // Keep up to limit bytes of freed case buffers for reuse by later cases
    // of the same sizes (0: free them at once). trim_pool frees cached blocks
    // until at most keep bytes remain cached.
    void set_pool_limit(size_t limit) { pool_limit_ = limit; }
    mcb_status trim_pool(size_t keep);
    size_t pool_bytes() const { return pool_bytes_; }
    CaseState* get(int id);
    int count() const { return (int)cases_.size(); }
    size_t bytes() const;
    const std::string& error() const { return err_; }
    long long batch_steps() const { return batch_steps_; }
    hipStream_t stream() const { return stream_; }

private:
    mcb_status fail(mcb_status s, const std::string& m);
    mcb_status add_impl(const mcb_params& p, const float* phi_host, const BubbleSet* bubbles, int* id, bool alone);
    mcb_status add_case(const mcb_params& p, const float* phi_host, const BubbleSet* bubbles, int* id, bool alone,
                        bool pad_rows);
    mcb_status dev_alloc(size_t bytes, void** out);
    void dev_release(void* ptr, size_t bytes);
    mcb_status build_own_table(CaseState* c);
    mcb_status rebuild();
    // n steps from parity q for every group, on the lanes; stream_ waits for all.
    mcb_status launch_steps(int q, int n);
    // 16-bit storage: reset the mass target and the pending corrections.
    mcb_status set_mass_target(CaseState* c, double target);
    // Keep g as populations from here on (arbitrary g has no moment form):
    // allocates the g buffers and, for 16 bits, the mass-drift state.
    mcb_status to_populations(CaseState* c);
    mcb_status set_form(CaseState* c, int gm);
    // The arrays of a case's state image; mass receives / supplies (5 slots)
    // the 16-bit mass target and pending correction of stored g (0, 1) and
    // of the moment form (2: fixed-point target, 3: target recorded, 4:
    // pending correction).
    std::vector<StatePart> state_parts(CaseState* c, int gm, double* mass);
    hipError_t stage_pops(CaseState* c, bool to_image);
    // One set of macro fields per batch, sized for its largest case; it holds
    // the observables of the case of the most recent macros() call.
    mcb_status ensure_macro_scratch();
    mcb_status ensure_partial();

    int device_;
    hipStream_t stream_;
    std::shared_ptr<Readback> readback_ = Readback::shared();
    std::string err_;
    std::map<int, std::unique_ptr<CaseState>> cases_;
    std::vector<int> order_;          // case ids in view-array order (by group)
    int next_id_ = 1;
    int parity_ = 0;
    long long batch_steps_ = 0;
    bool dirty_ = true;
    int storage_ = -1;                // all cases of a batch share one storage form
    // device arrays
    CaseView* d_views_[2] = {nullptr, nullptr};
    size_t views_cap_ = 0;
    // Cases that step on one tile shape in one collide mode: views
    // [first, first + cases) of the arrays, one work table, one lane.
    struct Group {
        Tiling t{}, pt{};                // tiles of the collide and phase passes
        int mode = COLLIDE_STEP;
        size_t at = 0;                   // its items in d_work_: [at, at + n) collide, then n_phase of the phase
        unsigned n = 0, n_phase = 0;     // pass where its tiles differ
        unsigned first = 0, cases = 0;
        Tiling sum{};                    // zc > 0: its only case sums phi on tiles of its own (launch_mass_sum)
        Geo geo{};                       // of that case
        bool mass = false;               // a case keeps a mass-drift correction (MassCell or MassQ)
        int lane = 0;                    // 0: stream_, i: lane_[i - 1]
    };
    // The first n_groups_ serve calls of one step, the n_long_ behind them (if any)
    // longer ones.
    std::vector<Group> groups_;
    size_t n_groups_ = 0, n_long_ = 0;
    WorkItem* d_work_ = nullptr;         // the groups' work tables
    size_t work_cap_ = 0;
    static constexpr int kLanes = 4;     // hardware queues of a process
    hipStream_t lane_[kLanes - 1] = {};  // created when a batch first needs them
    hipEvent_t fork_ = nullptr, join_[kLanes - 1] = {};
    int lanes_[2] = {1, 1};              // lanes that either list uses
    std::vector<CaseView> hv_[2];     // host copies of the view arrays
    bool any_initial_ = false;        // a moment-form case has not stepped yet
    double* d_partial_ = nullptr;     // reduction scratch (2 * kReduceBlocks + 2 doubles)
    std::vector<void*> macro_bufs_;
    size_t macro_plane_ = 0;
    size_t macro_bytes_ = 0;
    int macro_id_ = 0;
    std::multimap<size_t, void*> pool_;
    size_t pool_bytes_ = 0;
    size_t pool_limit_ = 0;
};

// The tiling of a single-case context: the autotuned choice, else a rule for a
// lattice that has the device to itself (rule_tiling_single).
Tiling choose_tiling_single(const mcb_params& p);
Tiling rule_tiling_single(const mcb_params& p);
// The tiling of a batch case, where the batch fills the device: by row length
// in FP32, else the autotuned choice (tau_g = 1) or a rule.
Tiling batch_tiling(const mcb_params& p);
// Autotuning: the tiles to measure for a context (alone) or a batch case, the
// rule's own first, and the choice for later ones of these sides, storage and
// form of g.
std::vector<Tiling> tune_candidates(const mcb_params& p, bool alone);
void remember_tiling(const mcb_params& p, bool alone, const Tiling& t);

}  // namespace mcb
