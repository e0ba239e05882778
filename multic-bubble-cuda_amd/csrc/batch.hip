// Batched execution (batch.hpp) and the tile autotuner.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <tuple>

#include "batch.hpp"
#include "state.hpp"
#include "tile.hpp"

namespace mcb {

namespace {

unsigned pop_bytes(int storage) { return storage == MCB_STORE_FP32 ? 4u : 2u; }

constexpr int kMacroFields = 10;

// A batch of one group steps as two halves side by side, in calls of two steps
// or more, from kSplitCells on: below, each half is a chain of launches too short
// to fill the device (5.8M cells in FP16: 199 us per step against 155). FP32 up
// to 24M cells, 16M with stored g (us per step, halves against whole, tau_g 1: 20
// cubes of 80 493 against 523, 32 of 32 to 128, 18M cells, 777 against 793, 13 of
// 144 1914 against 1884; tau_g 0.8: 775 against 811, 1357 against 1359, 10 of 128
// 1527 against 1508); FP16 13 of 144 1254 and 3824 against 1327 and 3908. A call
// of one step pays for the join (33 cubes of 72: 888 against 875), and next to
// other groups the halves of the largest one hold up the rest (16 FP16 cubes of
// 48 to 128: 467 against 433).
constexpr long long kSplitCells = 8LL << 20, kSplitCellsFp32 = 24LL << 20, kSplitCellsFp32Bgk = 16LL << 20;
// FP32 cases of different shapes step shape by shape, side by side, in calls of
// two steps or more, where a shape has kShapeCases cases on average; otherwise,
// and in calls of one step, all on 64x8 tiles in one group (us per step, by shape
// against one group, 20 steps a call: 16 cubes of 32 to 64 cells 87 against 108,
// 32 of 32 to 128 825 and with stored g 1396 against 843 and 1435, 30 of 48 to 112
// 1065 against 1143; but 6 cubes of 5 shapes 168 against 160, 8 of 48 to 192 with
// stored g 2540 against 2510, 12 of 24 and 33, 0.3M cells, 55 against 49; one step
// a call 16 of 32 to 64 122 against 108).
constexpr size_t kShapeCases = 5;
constexpr long long kShapeCells = 1LL << 20;
// What a group's launches of a step cost on their lane beside its cells, in
// cells (about 25 us).
constexpr long long kGroupCells = 1LL << 20;

bool same_tiling(const Tiling& a, const Tiling& b) { return a.tx == b.tx && a.ty == b.ty && a.zc == b.zc; }

// Work items of a case (x fastest, then y, then z chunks), renumbered by
// xcd_runs: each XCD takes runs of 8 consecutive tiles, so x-neighbouring
// tiles meet in one L2 while the device works on one contiguous stretch of
// the list (against xcd_order, where each XCD walks its own range: the 64
// FP32 'batch' presets 22.0k -> 22.4k MLUPS, FP16 at 256^3 41.5k -> 42.7k,
// 128^3 and 144^3 within 0.5%; without renumbering FP16 ran 2-7% slower).
std::vector<WorkItem> tiles_of(const CaseState& c, int slot, const Tiling& t) {
    std::vector<WorkItem> v;
    for (int z0 = 0; z0 < c.p.nz; z0 += t.zc)
        for (int y0 = 0; y0 < c.p.ny; y0 += t.ty)
            for (int x0 = 0; x0 < c.p.nx; x0 += t.tx) v.push_back(WorkItem{slot, x0, y0, z0});
    return v;
}

std::vector<WorkItem> xcd_permute(const std::vector<WorkItem>& in) {
    std::vector<WorkItem> out(in.size());
    const unsigned n = (unsigned)in.size();
    for (unsigned lid = 0; lid < n; ++lid) out[lid] = in[xcd_runs(lid, n, 8)];
    return out;
}

}  // namespace

// Whether a 16-bit lattice alone steps on tiles of whole rows (plain rows, then;
// see fused_geo): where one is instantiated, rows are not whole lines, and its
// workgroups fill 11 of a CU's 16 waves (48, 80, 112, 176: 80x230x160 106 us per
// step against 120 with the next best tile, 176^3 155 against 187; not 144, one
// 9-wave workgroup a CU: 125 against 116 with 64x4).
static bool keeps_row_tile16(int nx) {
    const int waves = nx / 16;
    return tiling_supported16(Tiling{nx, 4, 1}) && nx % 32 != 0 && 16 / waves * waves >= 11;
}

// Rows of a lattice alone that are worth padding to whole lines (us per step,
// plain against padded). Above 64 cells: FP32 65x200x150 157 against 132,
// 65x256x256 388 against 261, 200x256x256 815 against 596; FP16 84x256x256 288
// against 204, 200x256x256 583 against 401. Shorter rows fill few lines, and
// what the padding adds is read and written with them: FP32 tau_g 0.8
// 20x256x256 173 against 267, 50x256x256 260 against 402, FP16 tau_g 0.8
// 33x256x256 234 against 314; only rows just below 32 gain (FP32 30x256x256 147
// against 121). 16 bits with stored g, whose traffic is mostly populations, gain
// up to a sixth of padding (144 of 160: 413 against 406, 200x200x150 624
// against 581; 65x200x150 224 against 235, 98x200x150 259 against 273).
static bool pads_rows(const mcb_params& p) {
    const int pitch = (p.nx + 31) / 32 * 32;
    if (p.nx <= 64) return p.nx < 32 && pitch - p.nx <= 2;
    if (p.storage == MCB_STORE_FP32) return true;
    return !keeps_row_tile16(p.nx) && (p.tau_g == 1.0f || 5 * pitch <= 6 * p.nx);
}

Geo fused_geo(const mcb_params& p, bool pad_rows) {
    Geo g{p.nx, p.ny, p.nz, p.nx * p.ny, (long long)p.nx * p.ny * p.nz, 0, 0, p.nx, p.nx * p.ny};
    g.plane = plane_stride_cells(g.n);
    if (p.f_form != MCB_F_POPULATIONS) return g;
    const bool fp32 = p.storage == MCB_STORE_FP32;
    const int group = fp32 ? 64 : 1;
    for (const int pitch : {(p.nx + 31) / 32 * 32, p.nx}) {
        if (pitch != p.nx && !(pad_rows && pads_rows(p))) continue;
        const long long zp = ((long long)pitch * p.ny + group - 1) / group * group, plane = plane_stride_cells(zp * p.nz);
        if (plane * 19 * pop_bytes(p.storage) > 0xFFFFFFFFLL) continue;
        g.blocked = fp32;
        g.pitch = pitch;
        g.zpop = (int)zp;
        g.plane = plane;
        break;
    }
    return g;
}

// Tiles of the 16-bit (phi, B) phase pass of a lattice alone that collides on
// t. The pass stages a halo of one cell: 4-row tiles of 64 stage 1.55 cells for
// each of theirs, 8 rows 1.29 (256^3 FP16: 117 against 103 VALU and 37 against 34
// LDS instructions a cell, 92 us a pass against 85),
// while the collide pass wants the many small workgroups. Where 8 rows and
// longer chunks leave three workgroups a CU (us per step, 8 rows against 4, FP16
// and BF16 alike): 256^3 380 against 390, 256x256x128 197 against 203, 250^3 414
// against 429; 192^3, 224^3 and 256x200x130 the same. Below that 4 rows keep more
// of the device busy (117x90x133 57 against 59). The fixed-point sums of phi do
// not depend on the tiles.
static Tiling phase_tiling16(const mcb_params& p, const Tiling& t) {
    if (t.tx != 64 || t.ty != 4) return t;
    auto groups = [&](int zc) { return (long long)((p.nx + 63) / 64) * ((p.ny + 7) / 8) * ((p.nz + zc - 1) / zc); };
    for (int zc = std::min(32, p.nz); zc > t.zc; zc /= 2)
        if (groups(zc) >= 768) return Tiling{64, 8, zc};
    return t;
}

size_t case_bytes(const mcb_params& p, bool pad_rows) {
    const size_t P = (size_t)fused_geo(p, pad_rows).plane;
    const size_t S = (size_t)plane_stride_cells((long long)p.nx * p.ny * p.nz);
    const bool moments = p.tau_g == 1.0f;
    size_t b = (moments ? 2 : 4) * 19 * P * pop_bytes(p.storage);          // f (and g) A/B
    b += (moments || p.storage != MCB_STORE_FP32 ? 2 : 1) * S * sizeof(float);   // phi
    if (moments) b += p.storage == MCB_STORE_FP32 ? 6 * S * sizeof(float) : 3 * S * 2;   // u, n (FP32) or B (FP16)
    return b;
}

CaseView CaseState::view(int q) const {
    CaseView v{};
    v.geo = geo;
    v.phys = phys;
    v.zc = tiling.zc;
    v.tx = tiling.tx;
    v.ty = tiling.ty;
    v.ptx = phase.tx;
    v.pty = phase.ty;
    v.pzc = phase.zc;
    v.stx = sum.tx;
    v.sty = sum.ty;
    v.szc = sum.zc;
    v.fsrc = f[q];
    v.fdst = f[q ^ 1];
    v.gsrc = g[q];
    v.gdst = g[q ^ 1];
    v.phi = phi[q];
    v.phi_prev = phi[q ^ 1];
    v.mslot = q;
    v.mass = gm == GM_POPULATIONS ? mass : nullptr;
    v.massq = massq;
    v.partial = partial;
    // Moment form: only the parity of the initial state (cur = 0 before the
    // first step) sees GM_INITIAL.
    v.gm = gm == GM_INITIAL && q != cur ? GM_MOMENTS : gm;
    for (int k = 0; k < 3; ++k) {
        v.gm_u[k] = gmu[k];
        v.gm_n[k] = gmn[k];
    }
    return v;
}

CaseState::~CaseState() {
    for (auto& a : allocs) (void)hipFree(a.first);
    if (d_work) (void)hipFree(d_work);
    if (partial) (void)hipFree(partial);
}

// ---------------------------------------------------------------- tilings

namespace {
// Tuned tiles by sides, storage, form of g and whether the lattice is alone.
std::mutex g_tune_mu;
using TuneKey = std::tuple<int, int, int, int, bool, bool>;
std::map<TuneKey, Tiling> g_tuned;

TuneKey tune_key(const mcb_params& p, bool alone) {
    return TuneKey{p.nx, p.ny, p.nz, p.storage, p.tau_g == 1.0f, alone};
}

bool tuned(const mcb_params& p, bool alone, Tiling* t) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(tune_key(p, alone));
    if (it != g_tuned.end()) *t = it->second;
    return it != g_tuned.end();
}

bool supported_for(const Tiling& t, int storage) {
    return storage == MCB_STORE_FP32 ? tiling_supported(t) : tiling_supported16(t);
}
}  // namespace

static Tiling choose_tiling(const mcb_params& p) {
    Tiling t = p.nx >= 64 ? Tiling{64, 8, 16} : (p.nx >= 32 ? Tiling{32, 8, 16} : Tiling{16, 16, 16});
    // 16-bit forms: half the bytes per cell, so longer z runs pay off
    // (measured at 256^3: 64x8x32 fastest, 64x4x32 4% and 32x8x32 17%
    // slower); a 32-wide tile where it pads x less, since padded lanes do no
    // work. Measured per x side on batches of equal cubes (48 ... 192): a tile
    // spanning the whole row where one is instantiated (48, 80, 96, 112, 144,
    // 176; 1.1-1.9x), 64x4 for the other multiples of 32 up to 192; both with
    // z-chunks of 16, which give a lattice of this size alone enough
    // workgroups to fill the GPU (serving at 20 requests/s: p99 0.13 s
    // against 0.28 s with chunks of 32, and the same throughput at saturation).
    if (p.storage != MCB_STORE_FP32 && p.nx >= 48) {
        const int pad64 = (p.nx + 63) / 64 * 64, pad32 = (p.nx + 31) / 32 * 32;
        t = pad32 < pad64 ? Tiling{32, 8, 32} : Tiling{64, 8, 32};
        const Tiling row{p.nx, 4, 16};
        if (tiling_supported16(row)) t = row;
        else if (p.nx <= 192 && p.nx % 32 == 0) t = Tiling{64, 4, 16};
    }
    t.zc = std::min(t.zc, p.nz);
    return t;
}

Tiling batch_tiling(const mcb_params& p) {
    // FP32, batches of equal cubes (k MLUPS, tau_g 1 and 0.8), all in 8-plane
    // chunks: 64x8 tiles (64: 23.3); 32x8 where rows are too short for them (24:
    // 21.1 against 12.8 and 12.9 against 9.7) or end in half of one (32: 24.3
    // against 17.5, 96: 22.7 against 21.8, 160: 22.6 against 21.9, 224: 13.8
    // against 13.3), but not where they end in less (72: 12.0 against 14.4 with
    // 64x8, 136: 12.8 against 15.8, 144: 19.5 against 20.5); whole rows that are
    // odd multiples of 16 (48: 23.6 against 21.7, 80: 20.9 against 18.6, 112: 22.8
    // against 21.6), of which the long ones pay with stored g only (144: 19.7
    // against 20.5, but 13.3 against 12.6; 176: 20.9 against 22.0, 13.6 against 12.9).
    if (p.storage == MCB_STORE_FP32) {
        Tiling t = p.nx <= 32 || p.nx % 64 == 32 ? Tiling{32, 8, 8} : Tiling{64, 8, 8};
        const Tiling row{p.nx, 4, 8};
        if (p.nx >= 48 && p.nx % 32 == 16 && (p.nx < 128 || p.tau_g != 1.0f) && tiling_supported(row)) t = row;
        t.zc = std::min(t.zc, p.nz);
        return t;
    }
    // Stored 16-bit g: the sums of phi follow these tiles (build_own_table), and
    // so do a run's bits; they don't depend on what was tuned before.
    Tiling t;
    return p.tau_g == 1.0f && tuned(p, false, &t) ? t : choose_tiling(p);
}

Tiling choose_tiling_single(const mcb_params& p) {
    Tiling t;
    return p.f_form == MCB_F_POPULATIONS && tuned(p, true, &t) ? t : rule_tiling_single(p);
}

Tiling rule_tiling_single(const mcb_params& p) {
    Tiling t = choose_tiling(p);
    const bool fp32 = p.storage == MCB_STORE_FP32;
    // A lattice alone on the device (us per step, this rule against 64x8x16,
    // 16 bits 32x8x32 and 64x8x32): 4-row tiles, so that twice the workgroups
    // share the CUs, and short chunks, so that the planes that neighbouring
    // chunks read twice are still in L2. FP32 64x4x8 192^3 298 (319), 180^3 279
    // (300); stored g, with twice the planes, 64x4x2 250^3 1152 (1265), 180^3
    // 459 (524), 96x220x200 308 (356). 16 bits 64x4x8 240x250x100 170 (207),
    // 200^3 264 (304), 180^3 167 (186); 16 planes once they fill the device four
    // times over (256^3 397, 8 planes 406). 16-bit stored g, whose sums have
    // tiles of their own (build_own_table): 117x90x133 121 (315), 64^3 30 (101),
    // 200^3 756 (987).
    const int pad64 = (p.nx + 63) / 64 * 64, pad32 = (p.nx + 31) / 32 * 32;
    const bool moments = p.tau_g == 1.0f;
    bool row = false;
    // One 32-wide tile for rows that two of 16 would half fill (plain rows, 16x16
    // against this: FP32 28x256x256 125 against 93, tau_g 0.8 252 against 141;
    // FP16 24x256x256 86 against 61).
    if (p.nx > 16 && p.nx < 32 && p.f_form == MCB_F_POPULATIONS) t = Tiling{32, 8, t.zc};
    if (p.nx > 32 && p.f_form == MCB_F_POPULATIONS) {
        row = !fp32 && keeps_row_tile16(p.nx);
        // 32-wide tiles where 64-wide ones would pad more lanes: FP32 80x230x160
        // 156 against 204, 160^3 196 against 226, 224^3 453 against 501; in 16
        // bits, whose 64 lanes of a row are two lines, only where they pad a
        // fourth, or a sixth with whole 32-cell rows (96^3 41 against 42, 160^3
        // 128 against 137, but 150x105x77 56 against 54, 224^3 331 against 319).
        const bool narrow =
            p.nx > 64 && (fp32 ? pad32 < pad64 : pad32 * 6 < pad64 * 5 + (p.nx % 32 == 0 ? 1 : 0));
        if (row) t = Tiling{p.nx, 4, 16};
        else if (narrow) t = Tiling{32, 8, fp32 ? (moments ? 4 : 2) : 16};
        else t = Tiling{64, 4, fp32 ? (moments ? 8 : 2) : 16};
        t.zc = std::min(t.zc, p.nz);
    }
    auto lanes = [&](const Tiling& q) {
        return (long long)((p.nx + q.tx - 1) / q.tx) * ((p.ny + q.ty - 1) / q.ty) * ((p.nz + q.zc - 1) / q.zc) * q.tx *
               q.ty;
    };
    const long long wave_per_cu = 256 * 64;   // lanes: one wave on each of 256 CUs
    if (!fp32 && !row && t.zc > 8 && lanes(t) < 4 * 16 * wave_per_cu) t.zc = 8;
    // Shorter chunks until most of a CU's 16 waves (what 128 VGPRs allow) are
    // there: 13 in FP32 (112^3 64x4x8, 12.3 waves, 85.7 us, 4 planes 79; 96^3
    // 32x8x4, 13.5 waves, 50.8, 2 planes 52.7), 11 in 16 bits (117x90x133 8
    // planes, 12.2 waves, 54.8, 4 planes 56.1) and before single planes
    // (40x100x60 64x4x2, 11.7 waves, 25.9, 1 plane 31); 7 with whole rows, whose
    // halo is small (112^3 8 planes 58.9, 4 planes 60.8). One plane is the
    // least, 2 in 16 bits but where 3 planes are halved (lattices of 3, 6 and 7:
    // 64x64x6 14.1 with 1, 17.7 with 2).
    auto want = [&] { return (row ? 7 : (fp32 && t.zc > 2 ? 13 : 11)) * wave_per_cu; };
    while (t.zc > (fp32 ? 1 : 2) && lanes(t) < want()) t.zc /= 2;
    // Single planes restage their own halo: 8 rows where they pad no more
    // (64^3 with stored g 23.2 against 25.6), in 32-wide tiles where 64 lanes
    // do not fill (48^3 18.2 against 19.1).
    if (t.zc == 1 && t.tx == 64 && t.ty == 4 && p.ny % 8 == 0) t = Tiling{p.nx % 64 == 0 ? 64 : 32, 8, 1};
    return t;
}

// ------------------------------------------------------------------ Batch

Batch::Batch(int device, hipStream_t stream) : device_(device), stream_(stream) {}

Batch::~Batch() {
    (void)hipSetDevice(device_);
    (void)hipStreamSynchronize(stream_);
    for (auto& l : lane_)
        if (l) {
            (void)hipStreamSynchronize(l);
            (void)hipStreamDestroy(l);
        }
    if (fork_) (void)hipEventDestroy(fork_);
    for (auto& e : join_)
        if (e) (void)hipEventDestroy(e);
    if (d_work_) (void)hipFree(d_work_);
    for (auto& v : d_views_)
        if (v) (void)hipFree(v);
    if (d_partial_) (void)hipFree(d_partial_);
    cases_.clear();
    for (auto& q : macro_bufs_) (void)hipFree(q);
    for (auto& kv : pool_) (void)hipFree(kv.second);
}

mcb_status Batch::fail(mcb_status s, const std::string& m) {
    err_ = m;
    return s;
}

#define B_HIP(call)                                                                         \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess) return fail(hip_status(e_), std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

CaseState* Batch::get(int id) {
    auto it = cases_.find(id);
    return it == cases_.end() ? nullptr : it->second.get();
}

size_t Batch::bytes() const {
    size_t b = 0;
    for (auto& kv : cases_) b += kv.second->bytes;
    return b + macro_bytes_;
}

mcb_status Batch::dev_alloc(size_t bytes, void** out) {
    auto it = pool_.find(bytes);
    if (it != pool_.end()) {
        *out = it->second;
        pool_.erase(it);
        pool_bytes_ -= bytes;
        return MCB_OK;
    }
    hipError_t e = hipMalloc(out, bytes);
    if (e == hipErrorOutOfMemory && !pool_.empty()) {
        (void)hipGetLastError();
        mcb_status st = trim_pool(0);
        if (st != MCB_OK) return st;
        e = hipMalloc(out, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(hip_status(e), "hipMalloc failed for a case");
    }
    return MCB_OK;
}

void Batch::dev_release(void* ptr, size_t bytes) {
    if (pool_bytes_ + bytes <= pool_limit_) {
        pool_.emplace(bytes, ptr);
        pool_bytes_ += bytes;
    } else {
        (void)hipFree(ptr);
    }
}

mcb_status Batch::trim_pool(size_t keep) {
    B_HIP(hipSetDevice(device_));
    while (pool_bytes_ > keep && !pool_.empty()) {
        auto it = std::prev(pool_.end());   // largest first
        pool_bytes_ -= it->first;
        void* q = it->second;
        pool_.erase(it);
        B_HIP(hipFree(q));
    }
    return MCB_OK;
}

mcb_status Batch::ensure_partial() {
    if (!d_partial_) B_HIP(hipMalloc(reinterpret_cast<void**>(&d_partial_), (2 * kReduceBlocks + 2) * sizeof(double)));
    return MCB_OK;
}

mcb_status Batch::add(const mcb_params& p, const float* phi_host, int* id, bool alone) {
    if (!phi_host) return fail(MCB_ERR_INVALID_ARG, "null argument");
    return add_impl(p, phi_host, nullptr, id, alone);
}

mcb_status Batch::add_bubbles(const mcb_params& p, const mcb_bubble* bubbles, int n, float width, int* id,
                              bool alone) {
    if (!bubbles || n < 1 || n > kMaxBubbleSet || !(width > 0.0f) || !std::isfinite(width))
        return fail(MCB_ERR_INVALID_ARG, "invalid bubble set");
    BubbleSet s{};
    for (int i = 0; i < n; ++i) {
        const mcb_bubble& b = bubbles[i];
        if (!std::isfinite(b.cx) || !std::isfinite(b.cy) || !std::isfinite(b.cz) || !std::isfinite(b.r) || b.r < 0.0f)
            return fail(MCB_ERR_INVALID_ARG, "invalid bubble");
        s.b[i] = b;
    }
    s.n = n;
    s.width = width;
    return add_impl(p, nullptr, &s, id, alone);
}

mcb_status Batch::add_impl(const mcb_params& p, const float* phi_host, const BubbleSet* bubbles, int* id, bool alone) {
    mcb_status st = add_case(p, phi_host, bubbles, id, alone, alone);
    // Plain rows, which take less, where padded ones do not fit.
    if (st == MCB_ERR_OUT_OF_MEMORY && alone && fused_geo(p, true).pitch != p.nx)
        st = add_case(p, phi_host, bubbles, id, alone, false);
    return st;
}

mcb_status Batch::add_case(const mcb_params& p, const float* phi_host, const BubbleSet* bubbles, int* id, bool alone,
                           bool pad_rows) {
    if (!id) return fail(MCB_ERR_INVALID_ARG, "null argument");
    std::string why;
    if (host_validate(&p, &why) != MCB_OK) return fail(MCB_ERR_INVALID_ARG, why);
    if (p.bc_mode != MCB_BC_PERIODIC) return fail(MCB_ERR_UNSUPPORTED, "batched cases are periodic");
    if (p.f_form != MCB_F_POPULATIONS) return fail(MCB_ERR_UNSUPPORTED, "batched cases keep f as populations");
    if (storage_ >= 0 && p.storage != storage_) return fail(MCB_ERR_UNSUPPORTED, "one storage form per batch");
    const Geo geo = fused_geo(p, pad_rows);
    const long long P = geo.plane;
    if (19LL * P * pop_bytes(p.storage) > 0xFFFFFFFFLL) return fail(MCB_ERR_UNSUPPORTED, "lattice too large");
    Tiling t = batch_tiling(p);
    if (!supported_for(t, p.storage)) return fail(MCB_ERR_UNSUPPORTED, "no tiling for this lattice");
    B_HIP(hipSetDevice(device_));

    // On any failure below, cs goes out of scope and frees what was allocated.
    auto cs = std::make_unique<CaseState>();
    CaseState* c = cs.get();
    c->p = p;
    c->storage = p.storage;
    c->mode = p.tau_g == 1.0f ? COLLIDE_STEP : COLLIDE_STEP_BGK;
    c->tiling = t;
    c->alone = alone;
    // FP32 populations in 64-cell blocks (16-bit ones stay in planes: with
    // blocks the FP16 batch ran 3% slower).
    c->geo = geo;
    c->phys = host_phys(p);
    auto alloc = [&](size_t bytes, void** out) -> mcb_status {
        mcb_status s = dev_alloc(bytes, out);
        if (s != MCB_OK) return s;
        c->allocs.emplace_back(*out, bytes);
        c->bytes += bytes;
        return MCB_OK;
    };
    mcb_status st;
    const size_t pops = 19 * (size_t)P * pop_bytes(p.storage), S = (size_t)plane_stride_cells(geo.n);
    // At tau_g = 1 g is kept in moment form instead of two sets of 19
    // planes, for every storage form.
    const bool moments = c->mode == COLLIDE_STEP;
    for (int b = 0; b < 2; ++b) {
        if ((st = alloc(pops, &c->f[b])) != MCB_OK) return st;
        if (!moments && (st = alloc(pops, &c->g[b])) != MCB_OK) return st;
    }
    void* q = nullptr;
    if ((st = alloc(S * sizeof(float), &q)) != MCB_OK) return st;
    c->phi[0] = c->phi[1] = static_cast<float*>(q);
    if (moments || p.storage != MCB_STORE_FP32) {
        // phi[1] holds the state's phi (moment form) or the g anchor (16 bits).
        if ((st = alloc(S * sizeof(float), &q)) != MCB_OK) return st;
        c->phi[1] = static_cast<float*>(q);
    }
    if (moments) {
        // FP32: u and n (collisionPhase's inputs, bit-exact; a batch's
        // 8-plane chunks are too short for the phase pass to recompute n
        // profitably); 16 bits: the vector B = 3 phi u + phi_n n in FP16
        // (phase_tile_ab).
        const bool fp32 = p.storage == MCB_STORE_FP32;
        for (int k = 0; k < (fp32 ? 6 : 3); ++k) {
            if ((st = alloc(S * (fp32 ? sizeof(float) : 2), &q)) != MCB_OK) return st;
            (k < 3 ? c->gmu[k] : c->gmn[k - 3]) = static_cast<float*>(q);
        }
        if (!fp32) {
            // Mass-drift correction of the 16-bit moment form (MassQ).
            if ((st = alloc(sizeof(MassQ), &q)) != MCB_OK) return st;
            c->massq = static_cast<MassQ*>(q);
            const MassQ zero{0, 0, 0, {0.0, 0.0}};
            B_HIP(hipMemcpyAsync(c->massq, &zero, sizeof(zero), hipMemcpyHostToDevice, stream_));
        }
        c->gm = GM_INITIAL;
    } else if (p.storage != MCB_STORE_FP32) {
        // 16-bit phase populations: per-step FP64 mass-drift correction.
        if ((st = alloc(sizeof(MassCell), &q)) != MCB_OK) return st;
        c->mass = static_cast<MassCell*>(q);
        double target = 0.0;
        if (phi_host)
            for (long long i = 0; i < c->geo.n; ++i) target += (double)phi_host[i];
        if ((st = set_mass_target(c, target)) != MCB_OK) return st;
    }
    // Initial state: the current populations are in buffer 0, the initial
    // phi (state or g anchor) in phi[1].
    if (phi_host) {
        B_HIP(hipMemcpyAsync(c->phi[1], phi_host, (size_t)c->geo.n * sizeof(float), hipMemcpyHostToDevice, stream_));
    } else {
        B_HIP(launch_bubble_phi(c->phi[1], c->geo, *bubbles, stream_));
        if (c->mass) {
            if ((st = ensure_partial()) != MCB_OK) return st;
            B_HIP(launch_sum(c->phi[1], c->geo.n, d_partial_, &c->mass->target, stream_));
        }
    }
    if (p.storage == MCB_STORE_FP32) {
        B_HIP(launch_init_pull(c->phi[1], static_cast<float*>(c->f[0]), static_cast<float*>(c->g[0]), c->geo, c->phys,
                               stream_));
    } else {
        B_HIP(launch_init16(c->phi[1], c->f[0], c->g[0], c->geo, c->phys, p.storage, stream_));
    }
    c->cur = 0;
    c->parity_offset = parity_;
    c->phi_last = c->phi[1];
    c->steps = 0;
    if ((st = build_own_table(c)) != MCB_OK) return st;
    B_HIP(hipStreamSynchronize(stream_));
    storage_ = p.storage;
    *id = next_id_++;
    cases_[*id] = std::move(cs);
    dirty_ = true;
    return MCB_OK;
}

// The case's own work table (case index 0, used with the case's entry of the
// view arrays as the base) and its partial-sum buffer, for its tiling: the
// collide pass's items, then the phase pass's where its tiles differ.
mcb_status Batch::build_own_table(CaseState* c) {
    // Stored 16-bit g adds its FP64 sums tile by tile. In a context they
    // keep the tiles of a batch case, whatever the context steps on: a state
    // image continues with the same bits in either.
    const bool holds_g = c->gm == GM_POPULATIONS, ruled = c->alone && !c->own_tiling && c->storage != MCB_STORE_FP32;
    c->sum = ruled && holds_g ? batch_tiling(c->p) : c->tiling;
    c->phase = ruled && !holds_g ? phase_tiling16(c->p, c->tiling) : c->tiling;
    auto own = xcd_permute(tiles_of(*c, 0, c->tiling));
    c->n_work = (unsigned)own.size();
    c->n_phase = 0;
    if (!same_tiling(c->phase, c->tiling)) {
        const auto phase = xcd_permute(tiles_of(*c, 0, c->phase));
        c->n_phase = (unsigned)phase.size();
        own.insert(own.end(), phase.begin(), phase.end());
    }
    auto over = [](int n, int t) { return (size_t)((n + t - 1) / t); };
    auto count = [&](const Tiling& t) { return over(c->p.nx, t.tx) * over(c->p.ny, t.ty) * over(c->p.nz, t.zc); };
    const size_t sums = std::max(count(c->sum), count(c->phase));
    if (own.size() > c->work_cap) {
        if (c->d_work) B_HIP(hipFree(c->d_work));
        c->d_work = nullptr;
        c->work_cap = 0;
        B_HIP(hipMalloc(reinterpret_cast<void**>(&c->d_work), own.size() * sizeof(WorkItem)));
        c->work_cap = own.size();
    }
    B_HIP(hipMemcpyAsync(c->d_work, own.data(), own.size() * sizeof(WorkItem), hipMemcpyHostToDevice, stream_));
    const size_t parts = std::max<size_t>(c->n_work, sums);
    if ((c->mass || c->massq) && parts > c->partial_cap) {
        if (c->partial) B_HIP(hipFree(c->partial));
        c->partial = nullptr;
        c->partial_cap = 0;
        B_HIP(hipMalloc(reinterpret_cast<void**>(&c->partial), parts * sizeof(double)));
        c->partial_cap = parts;
    }
    B_HIP(hipStreamSynchronize(stream_));   // own is a host temporary
    return MCB_OK;
}

mcb_status Batch::remove(int id) {
    auto it = cases_.find(id);
    if (it == cases_.end()) return fail(MCB_ERR_INVALID_ARG, "no such case");
    B_HIP(hipSetDevice(device_));
    B_HIP(hipStreamSynchronize(stream_));
    CaseState* c = it->second.get();
    for (auto& a : c->allocs) dev_release(a.first, a.second);
    c->allocs.clear();
    cases_.erase(it);   // frees the case's tables
    if (cases_.empty()) storage_ = -1;
    if (macro_id_ == id) macro_id_ = 0;
    dirty_ = true;
    return MCB_OK;
}

mcb_status Batch::set_mass_target(CaseState* c, double target) {
    const MassCell m{target, {0.0, 0.0}};
    B_HIP(hipMemcpyAsync(c->mass, &m, sizeof(m), hipMemcpyHostToDevice, stream_));
    B_HIP(hipStreamSynchronize(stream_));
    return MCB_OK;
}

mcb_status Batch::ensure_macro_scratch() {
    size_t need = 0;
    for (auto& kv : cases_) need = std::max(need, (size_t)plane_stride_cells(kv.second->geo.n));
    if (need <= macro_plane_) return MCB_OK;
    for (void* q : macro_bufs_) B_HIP(hipFree(q));
    macro_bufs_.clear();
    macro_bytes_ = 0;
    macro_plane_ = 0;
    macro_id_ = 0;
    for (int k = 0; k < kMacroFields; ++k) {
        void* q = nullptr;
        B_HIP(hipMalloc(&q, need * sizeof(float)));
        macro_bufs_.push_back(q);
        macro_bytes_ += need * sizeof(float);
    }
    macro_plane_ = need;
    return MCB_OK;
}

mcb_status Batch::rebuild() {
    B_HIP(hipSetDevice(device_));
    B_HIP(hipStreamSynchronize(stream_));
    mcb_status st = ensure_macro_scratch();
    if (st != MCB_OK) return st;
    // FP32 cases whose rules name different shapes can step on 64x8 tiles all
    // together, one launch per pass for a mode (kShapeCases). All the rules'
    // chunks are 8 planes, so the views serve either shape.
    auto ruled = [&](const CaseState* c) { return storage_ == MCB_STORE_FP32 && !c->own_tiling; };
    bool mixed = false;
    const CaseState* some = nullptr;
    long long total = 0;
    for (auto& kv : cases_) {
        const CaseState* c = kv.second.get();
        total += c->geo.n;
        if (!ruled(c)) continue;
        if (!some) some = c;
        mixed |= c->tiling.tx != some->tiling.tx || c->tiling.ty != some->tiling.ty;
    }
    auto merged = [&](const CaseState* c) { return mixed && ruled(c) ? Tiling{64, 8, c->tiling.zc} : c->tiling; };
    // Cases in the order of their groups: collide mode, then tile shapes, merged
    // ones together.
    auto key = [&](int id) {
        const CaseState* c = cases_[id].get();
        const Tiling m = merged(c);
        return std::make_tuple(c->mode, m.tx, m.ty, c->phase.tx * (mixed && ruled(c) ? 0 : 1),
                               c->phase.ty * (mixed && ruled(c) ? 0 : 1));
    };
    auto shape_key = [&](int id) {
        const CaseState* c = cases_[id].get();
        return std::tuple_cat(key(id), std::make_tuple(c->tiling.tx, c->tiling.ty));
    };
    order_.clear();
    for (auto& kv : cases_) order_.push_back(kv.first);
    std::stable_sort(order_.begin(), order_.end(), [&](int a, int b) { return shape_key(a) < shape_key(b); });
    const size_t n = order_.size();
    if (n > views_cap_) {
        for (auto& v : d_views_) {
            if (v) B_HIP(hipFree(v));
            v = nullptr;
        }
        views_cap_ = 0;
        const size_t cap = std::max<size_t>(n, 2 * n);
        for (auto& v : d_views_) B_HIP(hipMalloc(reinterpret_cast<void**>(&v), cap * sizeof(CaseView)));
        views_cap_ = cap;
    }
    any_initial_ = false;
    for (int q = 0; q < 2; ++q) hv_[q].clear();
    for (size_t i = 0; i < n; ++i) {
        CaseState* c = cases_[order_[i]].get();
        for (int q = 0; q < 2; ++q) {
            CaseView v = c->view(q ^ c->parity_offset);
            float** m = reinterpret_cast<float**>(&v.rho);
            for (int k = 0; k < kMacroFields; ++k) m[k] = static_cast<float*>(macro_bufs_[k]);
            hv_[q].push_back(v);
        }
        if (c->gm == GM_INITIAL) any_initial_ = true;
        c->slot = (int)i;
    }
    for (int q = 0; q < 2; ++q)
        if (n) B_HIP(hipMemcpyAsync(d_views_[q], hv_[q].data(), n * sizeof(CaseView), hipMemcpyHostToDevice, stream_));
    // The groups of short calls, then those of longer ones where they differ: by
    // shape, or the halves of a large one.
    std::vector<std::pair<size_t, size_t>> range;
    auto ranges_by = [&](auto&& of) {
        for (size_t i = 0; i < n; ++i) {
            if (i == 0 || of(order_[i]) != of(order_[i - 1])) range.emplace_back(i, i);
            range.back().second = i + 1;
        }
    };
    auto cells = [&](size_t i) { return cases_[order_[i]]->geo.n; };
    ranges_by(key);
    n_groups_ = range.size();
    bool by_shape = false;
    if (mixed && total >= kShapeCells) {
        ranges_by(shape_key);
        by_shape = n >= kShapeCases * (range.size() - n_groups_);
        if (!by_shape) range.resize(n_groups_);
    }
    const bool one = n_groups_ == 1 && !by_shape;
    if (one || by_shape) {
        // The largest group in two, if it holds most of the work.
        size_t at = 0;
        long long work = 0;
        for (size_t k = one ? 0 : n_groups_; k < range.size(); ++k) {
            long long w = 0;
            for (size_t i = range[k].first; i < range[k].second; ++i) w += cells(i);
            if (w > work) {
                work = w;
                at = k;
            }
        }
        const size_t begin = range[at].first, end = range[at].second;
        const long long most = cases_[order_[0]]->mode == COLLIDE_STEP ? kSplitCellsFp32 : kSplitCellsFp32Bgk;
        if (end - begin > 1 && work >= kSplitCells && (one ? (storage_ != MCB_STORE_FP32 || work < most) : 2 * work > total)) {
            long long half = 0;
            size_t cut = begin;
            while (cut < end - 1 && 2 * half < work) half += cells(cut++);
            if (one) range.emplace_back(begin, cut);
            else range[at].second = cut;
            range.emplace_back(cut, end);
        }
    }
    n_long_ = range.size() - n_groups_;
    if (groups_.size() < range.size()) groups_.resize(range.size());
    std::vector<WorkItem> tables;
    std::vector<std::pair<long long, size_t>> load[2];   // cost and index of a group, of either list
    for (size_t k = 0; k < range.size(); ++k) {
        Group& gr = groups_[k];
        const size_t begin = range[k].first, end = range[k].second;
        gr.first = (unsigned)begin;
        gr.cases = (unsigned)(end - begin);
        const CaseState* c0 = cases_[order_[begin]].get();
        const bool own = by_shape && k >= n_groups_;   // each case's own shape
        auto shape = [&](const CaseState* c) { return own ? c->tiling : merged(c); };
        auto phase_shape = [&](const CaseState* c) { return own || !(mixed && ruled(c)) ? c->phase : merged(c); };
        gr.t = shape(c0);
        gr.pt = phase_shape(c0);
        gr.mode = c0->mode;
        gr.mass = false;
        gr.sum = c0->sum;   // of its own: a case alone (a context) only
        if (c0->gm != GM_POPULATIONS || same_tiling(c0->sum, c0->tiling)) gr.sum.zc = 0;
        gr.geo = c0->geo;
        std::vector<WorkItem> items, phase;
        bool differ = false;
        long long work = 0;
        for (size_t i = begin; i < end; ++i) {
            const CaseState* c = cases_[order_[i]].get();
            gr.mass |= c->massq || c->mass;
            differ |= !same_tiling(phase_shape(c), shape(c));
            work += c->geo.n;
        }
        for (size_t i = begin; i < end; ++i) {
            const CaseState* c = cases_[order_[i]].get();
            const auto tl = tiles_of(*c, (int)i, shape(c));
            items.insert(items.end(), tl.begin(), tl.end());
            if (!differ) continue;
            const auto pl = tiles_of(*c, (int)i, phase_shape(c));
            phase.insert(phase.end(), pl.begin(), pl.end());
        }
        items = xcd_permute(items);
        phase = xcd_permute(phase);
        gr.n = (unsigned)items.size();
        gr.n_phase = (unsigned)phase.size();
        gr.at = tables.size();
        tables.insert(tables.end(), items.begin(), items.end());
        tables.insert(tables.end(), phase.begin(), phase.end());
        load[k >= n_groups_].emplace_back(work + kGroupCells, k);
    }
    if (tables.size() > work_cap_) {
        if (d_work_) B_HIP(hipFree(d_work_));
        d_work_ = nullptr;
        work_cap_ = 0;
        const size_t cap = 2 * tables.size();
        B_HIP(hipMalloc(reinterpret_cast<void**>(&d_work_), cap * sizeof(WorkItem)));
        work_cap_ = cap;
    }
    if (!tables.empty())
        B_HIP(hipMemcpyAsync(d_work_, tables.data(), tables.size() * sizeof(WorkItem), hipMemcpyHostToDevice, stream_));
    B_HIP(hipStreamSynchronize(stream_));   // the copies of hv_ and tables
    // Lanes: each group to the least loaded one, largest first.
    for (int j = 0; j < 2; ++j) {
        std::sort(load[j].rbegin(), load[j].rend());
        lanes_[j] = (int)std::max<size_t>(1, std::min<size_t>(kLanes, load[j].size()));
        long long lane_load[kLanes] = {};
        for (const auto& l : load[j]) {
            const int at = (int)(std::min_element(lane_load, lane_load + lanes_[j]) - lane_load);
            groups_[l.second].lane = at;
            lane_load[at] += l.first;
        }
    }
    const int lanes = std::max(lanes_[0], lanes_[1]);
    if (lanes > 1 && !fork_) B_HIP(hipEventCreateWithFlags(&fork_, hipEventDisableTiming));
    for (int i = 0; i + 1 < lanes; ++i) {
        if (!lane_[i]) B_HIP(hipStreamCreateWithFlags(&lane_[i], hipStreamNonBlocking));
        if (!join_[i]) B_HIP(hipEventCreateWithFlags(&join_[i], hipEventDisableTiming));
    }
    dirty_ = false;
    return MCB_OK;
}

mcb_status Batch::launch_steps(int q, int n) {
    // A caller capturing stream_ gets everything recorded there.
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (std::max(lanes_[0], lanes_[1]) > 1) B_HIP(hipStreamIsCapturing(stream_, &cap));
    const bool captured = cap != hipStreamCaptureStatusNone, longer = n_long_ > 0 && n > 1 && !captured;
    const int lanes = captured ? 1 : lanes_[longer];
    const bool fork = lanes > 1;
    const size_t first = longer ? n_groups_ : 0, last = longer ? n_groups_ + n_long_ : n_groups_;
    if (fork) {
        B_HIP(hipEventRecord(fork_, stream_));
        for (int i = 0; i + 1 < lanes; ++i) B_HIP(hipStreamWaitEvent(lane_[i], fork_, 0));
    }
    hipError_t e = hipSuccess;
    for (int k = 0; k < n && e == hipSuccess; ++k, q ^= 1)
        for (size_t i = first; i < last && e == hipSuccess; ++i) {
            const Group& gr = groups_[i];
            const hipStream_t s = fork && gr.lane ? lane_[gr.lane - 1] : stream_;
            const WorkItem* const work = d_work_ + gr.at;
            e = gr.n_phase ? launch_phase_batch(d_views_[q], work + gr.n, gr.n_phase, gr.pt, storage_, s)
                           : launch_phase_batch(d_views_[q], work, gr.n, gr.t, storage_, s);
            if (e == hipSuccess && gr.sum.zc) e = launch_mass_sum(d_views_[q] + gr.first, gr.geo, gr.sum, s);
            if (e == hipSuccess && gr.mass) e = launch_mass_finish(d_views_[q] + gr.first, gr.cases, s);
            if (e == hipSuccess) e = launch_collide_batch(d_views_[q], work, gr.n, gr.t, gr.mode, storage_, s);
        }
    // Also after an error: whatever was launched is ordered before stream_'s next work.
    for (int i = 0; fork && i + 1 < lanes; ++i) {
        hipError_t j = hipEventRecord(join_[i], lane_[i]);
        if (j == hipSuccess) j = hipStreamWaitEvent(stream_, join_[i], 0);
        if (j != hipSuccess) (void)hipStreamSynchronize(lane_[i]);
        if (e == hipSuccess) e = j;
    }
    B_HIP(e);
    return MCB_OK;
}

mcb_status Batch::step(int nsteps) {
    if (nsteps < 0) return fail(MCB_ERR_INVALID_ARG, "negative step count");
    if (cases_.empty()) return MCB_OK;
    B_HIP(hipSetDevice(device_));
    if (dirty_) {
        mcb_status st = rebuild();
        if (st != MCB_OK) return st;
    }
    if (nsteps == 0) return MCB_OK;
    int left = nsteps;
    if (any_initial_) {
        // The first step of moment-form cases reads their initial state; the
        // view of that parity then switches to the moment form (stream-ordered
        // copy from the persistent host array).
        mcb_status st = launch_steps(parity_, 1);
        if (st != MCB_OK) return st;
        const int q = parity_;
        parity_ ^= 1;
        left -= 1;
        for (size_t i = 0; i < order_.size(); ++i) {
            CaseState* c = cases_[order_[i]].get();
            if (c->gm != GM_INITIAL) continue;
            c->gm = GM_MOMENTS;
            hv_[q][i].gm = GM_MOMENTS;
            B_HIP(hipMemcpyAsync(d_views_[q] + i, &hv_[q][i], sizeof(CaseView), hipMemcpyHostToDevice, stream_));
        }
        any_initial_ = false;
    }
    if (left > 0) {
        mcb_status st = launch_steps(parity_, left);
        if (st != MCB_OK) return st;
        parity_ ^= left & 1;
    }
    batch_steps_ += nsteps;
    macro_id_ = 0;  // the macro fields no longer match any case's state
    for (auto& kv : cases_) {
        CaseState* c = kv.second.get();
        c->cur = parity_ ^ c->parity_offset;
        c->steps += nsteps;
        c->phi_last = c->phi[c->cur ^ 1];
    }
    return MCB_OK;
}

mcb_status Batch::macros(int id) {
    CaseState* c = get(id);
    if (!c) return fail(MCB_ERR_INVALID_ARG, "no such case");
    B_HIP(hipSetDevice(device_));
    if (dirty_) {
        mcb_status st = rebuild();
        if (st != MCB_OK) return st;
    }
    // The case's own table indexes case 0 of a view array based at its slot.
    const CaseView* views = d_views_[parity_] + c->slot;
    const bool own_phase = c->n_phase != 0;
    B_HIP(launch_phase_batch(views, own_phase ? c->d_work + c->n_work : c->d_work, own_phase ? c->n_phase : c->n_work,
                             c->phase, storage_, stream_));
    B_HIP(launch_collide_batch(views, c->d_work, c->n_work, c->tiling, COLLIDE_MACROS, storage_, stream_));
    c->phi_last = c->phi[c->cur];
    macro_id_ = id;
    return MCB_OK;
}

mcb_status Batch::read(int id, int field, float* host, size_t n) {
    CaseState* c = get(id);
    if (!c || !host) return fail(MCB_ERR_INVALID_ARG, "no such case or null buffer");
    B_HIP(hipSetDevice(device_));
    const size_t cells = (size_t)c->geo.n;
    const size_t P = (size_t)c->geo.plane;
    if (field == MCB_FIELD_F || field == MCB_FIELD_G) {
        if (n != 19 * cells) return fail(MCB_ERR_INVALID_ARG, "population buffer must hold 19*nx*ny*nz floats");
        const bool isf = field == MCB_FIELD_F;
        float* tmp = nullptr;
        B_HIP(hipMalloc(reinterpret_cast<void**>(&tmp), 19 * P * sizeof(float)));
        hipError_t e;
        if (!isf && c->gm != GM_POPULATIONS)
            e = c->storage == MCB_STORE_FP32 ? launch_gm_to_ref(c->view(c->cur), tmp, stream_)
                                             : launch_ab_to_ref(c->view(c->cur), tmp, stream_);
        else if (c->storage == MCB_STORE_FP32)
            e = launch_link_shift(static_cast<const float*>(isf ? c->f[c->cur] : c->g[c->cur]), 1, tmp, 0,
                                  c->geo, +1, stream_);
        else
            e = launch_decode16(isf ? c->f[c->cur] : c->g[c->cur], isf ? nullptr : c->phi[c->cur ^ 1], tmp, c->geo,
                                c->phys, c->storage, stream_);
        if (e == hipSuccess)
            e = Readback::copy_rows(readback_.get(), host, tmp, cells * sizeof(float), P * sizeof(float), 19, stream_);
        (void)hipFree(tmp);
        B_HIP(e);
        return MCB_OK;
    }
    if (n != cells) return fail(MCB_ERR_INVALID_ARG, "field buffer must hold nx*ny*nz floats");
    const float* src = nullptr;
    if (field == MCB_FIELD_PHI) {
        src = c->phi_last;
    } else if (field >= MCB_FIELD_RHO && field <= MCB_FIELD_NORMZ) {
        if (macro_id_ != id) return fail(MCB_ERR_INVALID_ARG, "compute the macros of this case first");
        src = static_cast<const float*>(macro_bufs_[field - MCB_FIELD_RHO]);
    } else {
        return fail(MCB_ERR_INVALID_ARG, "unknown field");
    }
    B_HIP(Readback::copy(readback_.get(), host, src, cells * sizeof(float), stream_));
    return MCB_OK;
}

mcb_status Batch::to_populations(CaseState* c) {
    B_HIP(hipStreamSynchronize(stream_));
    // A case that went back to the moment form (load_state) still has these.
    const size_t pops = 19 * (size_t)c->geo.plane * pop_bytes(c->storage);
    for (int b = 0; b < 2; ++b) {
        if (c->g[b]) continue;
        void* q = nullptr;
        mcb_status st = dev_alloc(pops, &q);
        if (st != MCB_OK) return st;
        c->g[b] = q;
        c->allocs.emplace_back(q, pops);
        c->bytes += pops;
    }
    if (c->storage != MCB_STORE_FP32 && !c->mass) {
        void* q = nullptr;
        mcb_status st = dev_alloc(sizeof(MassCell), &q);
        if (st != MCB_OK) return st;
        c->allocs.emplace_back(q, sizeof(MassCell));
        c->mass = static_cast<MassCell*>(q);
    }
    return set_form(c, GM_POPULATIONS);
}

// The form of g that the case's next step reads; its phase and sum tiles go
// with it.
mcb_status Batch::set_form(CaseState* c, int gm) {
    const bool other = (gm == GM_POPULATIONS) != (c->gm == GM_POPULATIONS);
    c->gm = gm;
    dirty_ = true;
    return other ? build_own_table(c) : MCB_OK;
}

// --------------------------------------------------------------- state

// What the next step of a case reads (view(cur)): f of the current buffer;
// g as populations, or its moment form (u in FP32; B in 16 bits); the
// state's phi (the moment form's phi, the 16-bit g anchor; with FP32 g
// populations the phi the last step reported, which the populations do not
// give back); the 16-bit mass target and the correction pending for the next
// phase pass. n is not part of an image: it is gradCalc of the state's phi,
// rebuilt on loading. FP32 images have the parts of a single context's (same
// form), so either resumes in the other. gm: the form of g, which alone decides
// the parts (a case may hold buffers of the other form besides).
std::vector<StatePart> Batch::state_parts(CaseState* c, int gm, double* mass) {
    const size_t N = (size_t)c->geo.n, P = (size_t)c->geo.plane;
    const unsigned eb = pop_bytes(c->storage);
    // Images keep populations in plain planes: other layouts pass through the
    // idle A/B buffers (stage_pops), which the next step overwrites.
    const int side = pops_relaid(c->geo) ? c->cur ^ 1 : c->cur;
    std::vector<StatePart> parts;
    parts.push_back({"f", c->f[side], 19, N, P, eb, false});
    if (gm == GM_POPULATIONS) parts.push_back({"g", c->g[side], 19, N, P, eb, false});
    parts.push_back({"phi", c->phi[c->cur ^ 1], 1, N, N, 4, false});
    if (gm != GM_POPULATIONS) {
        static const char* const un[3] = {"u0", "u1", "u2"};
        for (int k = 0; k < 3; ++k)
            if (c->gmu[k]) parts.push_back({un[k], c->gmu[k], 1, N, N, c->storage == MCB_STORE_FP32 ? 4u : 2u, false});
    }
    if (c->storage != MCB_STORE_FP32 && gm == GM_POPULATIONS) parts.push_back({"mass", mass, 1, 2, 2, 8, true});
    if (c->massq) parts.push_back({"massq", mass + 2, 1, 3, 3, 8, true});
    return parts;
}

mcb_status Batch::state_size(int id, size_t* bytes) {
    CaseState* c = get(id);
    if (!c || !bytes) return fail(MCB_ERR_INVALID_ARG, "no such case or null size pointer");
    double m5[5];
    *bytes = state_image_bytes(state_parts(c, c->gm, m5));
    return MCB_OK;
}

mcb_status Batch::save_state(int id, void* buf, size_t bytes) {
    CaseState* c = get(id);
    if (!c) return fail(MCB_ERR_INVALID_ARG, "no such case");
    B_HIP(hipSetDevice(device_));
    B_HIP(hipStreamSynchronize(stream_));
    double m5[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (c->mass && c->gm == GM_POPULATIONS) {
        MassCell m;
        B_HIP(hipMemcpy(&m, c->mass, sizeof(m), hipMemcpyDeviceToHost));
        m5[0] = m.target;
        m5[1] = m.delta[c->cur];
    }
    if (c->massq) {
        MassQ m;
        B_HIP(hipMemcpy(&m, c->massq, sizeof(m), hipMemcpyDeviceToHost));
        std::memcpy(&m5[2], &m.target, sizeof(double));   // the integer's bits
        m5[3] = (double)m.set;
        m5[4] = m.delta[c->cur];
    }
    StateHeader h{};
    h.params = c->p;
    h.path = MCB_PATH_FUSED;
    h.gm = c->gm;
    h.steps = c->steps;
    if (pops_relaid(c->geo)) B_HIP(stage_pops(c, true));
    return state_image_save(stream_, h, state_parts(c, c->gm, m5), buf, bytes, &err_);
}

// Populations in another layout around a state image: the current f (and g
// populations) into the idle buffers in planes, or back.
hipError_t Batch::stage_pops(CaseState* c, bool to_image) {
    const int cur = c->cur, idle = c->cur ^ 1;
    void* const* bufs[2] = {c->f, c->gm == GM_POPULATIONS ? c->g : nullptr};
    for (void* const* b : bufs) {
        if (!b) continue;
        const hipError_t e = to_image ? launch_pop_relayout(b[cur], 1, b[idle], 0, c->geo, pop_bytes(c->storage), stream_)
                                      : launch_pop_relayout(b[idle], 0, b[cur], 1, c->geo, pop_bytes(c->storage), stream_);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

mcb_status Batch::load_state(int id, const void* buf, size_t bytes) {
    CaseState* c = get(id);
    if (!c) return fail(MCB_ERR_INVALID_ARG, "no such case");
    StateHeader h;
    mcb_status st = state_image_header(buf, bytes, &h, &err_);
    if (st != MCB_OK) return st;
    if (!same_state_params(h.params, c->p) || h.path != MCB_PATH_FUSED)
        return fail(MCB_ERR_INVALID_ARG, "state image of another lattice or parameter set");
    if (h.gm < GM_POPULATIONS || h.gm > GM_INITIAL || (h.gm != GM_POPULATIONS && c->mode != COLLIDE_STEP))
        return fail(MCB_ERR_INVALID_ARG, "state image with an invalid g form");
    B_HIP(hipSetDevice(device_));
    B_HIP(hipStreamSynchronize(stream_));
    // A refused image leaves the case as it was.
    double m5[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if ((st = state_image_check(buf, bytes, state_parts(c, h.gm, m5), &err_)) != MCB_OK) return st;
    // A case that holds populations and gets a moment-form image keeps its
    // g buffers (unused) and reads the moment fields again.
    if ((st = h.gm == GM_POPULATIONS ? to_populations(c) : set_form(c, h.gm)) != MCB_OK) return st;
    if ((st = state_image_load(stream_, buf, bytes, state_parts(c, h.gm, m5), &err_)) != MCB_OK) return st;
    if (pops_relaid(c->geo)) {
        B_HIP(stage_pops(c, false));
        B_HIP(hipStreamSynchronize(stream_));
    }
    if (c->mass && c->gm == GM_POPULATIONS) {
        MassCell m{m5[0], {0.0, 0.0}};
        m.delta[c->cur] = m5[1];
        B_HIP(hipMemcpy(c->mass, &m, sizeof(m), hipMemcpyHostToDevice));
    }
    if (c->massq) {
        MassQ m{0, m5[3] != 0.0 ? 1 : 0, 0, {0.0, 0.0}};
        std::memcpy(&m.target, &m5[2], sizeof(double));
        m.delta[c->cur] = m5[4];
        B_HIP(hipMemcpy(c->massq, &m, sizeof(m), hipMemcpyHostToDevice));
    }
    if (c->gm != GM_POPULATIONS && c->gmn[0]) {
        B_HIP(launch_normals(c->view(c->cur), stream_));
        B_HIP(hipStreamSynchronize(stream_));
    }
    c->steps = h.steps;
    c->phi_last = c->phi[c->cur ^ 1];
    if (macro_id_ == id) macro_id_ = 0;
    dirty_ = true;
    return MCB_OK;
}

mcb_status Batch::add_state(const void* buf, size_t bytes, int* id) {
    StateHeader h;
    mcb_status st = state_image_header(buf, bytes, &h, &err_);
    if (st != MCB_OK) return st;
    if (h.path != MCB_PATH_FUSED) return fail(MCB_ERR_INVALID_ARG, "state image of a staged-path context");
    mcb_params p = h.params;
    p.device = device_;
    std::string why;
    if (host_validate(&p, &why) != MCB_OK) return fail(MCB_ERR_INVALID_ARG, "state image: " + why);
    std::vector<float> zero;
    try {
        zero.assign((size_t)p.nx * p.ny * p.nz, 0.0f);
    } catch (const std::bad_alloc&) {
        return fail(MCB_ERR_OUT_OF_MEMORY, "host memory for the case's placeholder phi");
    }
    int nid = 0;
    if ((st = add(p, zero.data(), &nid)) != MCB_OK) return st;
    if ((st = load_state(nid, buf, bytes)) != MCB_OK) {
        const std::string keep = err_;
        (void)remove(nid);
        err_ = keep;
        return st;
    }
    if (id) *id = nid;
    return MCB_OK;
}

mcb_status Batch::write(int id, int field, const float* host, size_t n) {
    CaseState* c = get(id);
    if (!c || !host) return fail(MCB_ERR_INVALID_ARG, "no such case or null buffer");
    B_HIP(hipSetDevice(device_));
    const size_t cells = (size_t)c->geo.n;
    const size_t P = (size_t)c->geo.plane;
    if (field == MCB_FIELD_F || field == MCB_FIELD_G) {
        if (n != 19 * cells) return fail(MCB_ERR_INVALID_ARG, "population buffer must hold 19*nx*ny*nz floats");
        const bool isf = field == MCB_FIELD_F;
        if (!isf && c->gm != GM_POPULATIONS) {
            // Arbitrary g populations have no moment form: the case keeps g as
            // populations from here on (16 bits: anchored to the state's phi,
            // with the mass-drift correction).
            mcb_status st = to_populations(c);
            if (st != MCB_OK) return st;
        }
        float* tmp = nullptr;
        B_HIP(hipMalloc(reinterpret_cast<void**>(&tmp), 19 * P * sizeof(float)));
        hipError_t e = hipSuccess;
        for (int l = 0; l < 19 && e == hipSuccess; ++l)
            e = hipMemcpyAsync(tmp + l * P, host + l * cells, cells * sizeof(float), hipMemcpyHostToDevice, stream_);
        if (e == hipSuccess) {
            if (c->storage == MCB_STORE_FP32)
                e = launch_link_shift(tmp, 0, static_cast<float*>(isf ? c->f[c->cur] : c->g[c->cur]), 1,
                                      c->geo, -1, stream_);
            else
                e = launch_encode16(tmp, isf ? nullptr : c->phi[c->cur ^ 1], isf ? c->f[c->cur] : c->g[c->cur], c->geo,
                                    c->phys, c->storage, stream_);
        }
        if (e == hipSuccess) e = hipStreamSynchronize(stream_);
        (void)hipFree(tmp);
        B_HIP(e);
        if (c->mass && !isf) {
            // The written phase populations define the mass to keep.
            double target = 0.0;
            for (size_t i = 0; i < 19 * cells; ++i) target += (double)host[i];
            return set_mass_target(c, target);
        }
        return MCB_OK;
    }
    if (field != MCB_FIELD_PHI) return fail(MCB_ERR_INVALID_ARG, "only PHI, F and G can be written");
    if (c->storage != MCB_STORE_FP32 && c->gm == GM_POPULATIONS)
        return fail(MCB_ERR_UNSUPPORTED, "with 16-bit populations phi anchors the g populations; write G instead");
    if (n != cells) return fail(MCB_ERR_INVALID_ARG, "field buffer must hold nx*ny*nz floats");
    // In moment form phi of the state is phi[cur ^ 1]; like a write with
    // populations, the written phi is what the next phase pass replaces.
    if (c->gm != GM_POPULATIONS) c->phi_last = c->phi[c->cur];
    B_HIP(hipMemcpyAsync(c->phi_last, host, cells * sizeof(float), hipMemcpyHostToDevice, stream_));
    B_HIP(hipStreamSynchronize(stream_));
    return MCB_OK;
}

mcb_status Batch::reduce(int id, double* sum_phi, double* kinetic) {
    CaseState* c = get(id);
    if (!c) return fail(MCB_ERR_INVALID_ARG, "no such case");
    if (macro_id_ != id) return fail(MCB_ERR_INVALID_ARG, "compute the macros of this case first");
    B_HIP(hipSetDevice(device_));
    mcb_status st = ensure_partial();
    if (st != MCB_OK) return st;
    float* const* m = reinterpret_cast<float* const*>(macro_bufs_.data());
    B_HIP(launch_reduce(c->phi_last, m[0], m[1], m[2], m[3], c->geo.n, d_partial_, d_partial_ + 2 * kReduceBlocks,
                        stream_));
    double h[2] = {0.0, 0.0};
    B_HIP(hipMemcpyAsync(h, d_partial_ + 2 * kReduceBlocks, sizeof(h), hipMemcpyDeviceToHost, stream_));
    B_HIP(hipStreamSynchronize(stream_));
    if (sum_phi) *sum_phi = h[0];
    if (kinetic) *kinetic = h[1];
    if (!std::isfinite(h[0]) || !std::isfinite(h[1])) return fail(MCB_ERR_NONFINITE, "non-finite diagnostic");
    return MCB_OK;
}

mcb_status Batch::set_tiling(int id, const Tiling& t, bool by_caller) {
    CaseState* c = get(id);
    if (!c) return fail(MCB_ERR_INVALID_ARG, "no such case");
    if (!supported_for(t, c->storage) || t.zc > c->p.nz) return fail(MCB_ERR_INVALID_ARG, "unsupported tiling");
    B_HIP(hipSetDevice(device_));
    B_HIP(hipStreamSynchronize(stream_));
    c->tiling = t;
    c->own_tiling = by_caller;
    mcb_status st = build_own_table(c);
    if (st != MCB_OK) return st;
    dirty_ = true;
    return MCB_OK;
}

mcb_status Batch::synchronize() {
    B_HIP(hipSetDevice(device_));
    B_HIP(hipStreamSynchronize(stream_));
    return MCB_OK;
}

// --------------------------------------------------------------- autotune

void remember_tiling(const mcb_params& p, bool alone, const Tiling& t) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[tune_key(p, alone)] = t;
}

std::vector<Tiling> tune_candidates(const mcb_params& p, bool alone) {
    std::vector<Tiling> v{alone ? rule_tiling_single(p) : choose_tiling(p)};
    for (int i = 0; i < tiling_count(); ++i)
        for (int zc : {1, 2, 4, 8, 16, 32}) {
            const Tiling t{tiling_at(i).tx, tiling_at(i).ty, zc};
            if (zc <= p.nz && supported_for(t, p.storage) && t.tx <= 2 * p.nx && t.ty <= 2 * p.ny && !same_tiling(t, v[0]))
                v.push_back(t);
        }
    return v;
}

}  // namespace mcb
