// Host-side state of one device ensemble and the launchers of each phase.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "../host/device_api.h"
#include "../host/engine.h"
#include "../host/errors.h"
#include "common.h"

namespace tfg {

#define TFG_HIP(call)                                                                   \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess)                                                           \
            return set_error(TFG_E_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Device buffers of one ensemble: hipMalloc'd one by one, or carved in
// 256-byte steps from a caller's arena (no allocation; nothing to free).
struct Buffers {
    std::vector<void *> ptrs;
    unsigned char *arena = nullptr;
    size_t arena_cap = 0, arena_used = 0;
    ~Buffers() {
        for (void *p : ptrs) (void)hipFree(p);
    }
    template <typename T> int alloc(T **out, size_t n) {
        if (n == 0) n = 1;
        if (arena) {
            const size_t bytes = (n * sizeof(T) + 255) & ~static_cast<size_t>(255);
            if (bytes > arena_cap - arena_used)
                return set_error(TFG_E_RANGE, "the system needs more device memory than the " +
                                                  std::to_string(arena_cap >> 20) + " MiB scratch array holds");
            *out = reinterpret_cast<T *>(arena + arena_used);
            arena_used += bytes;
            return TFG_OK;
        }
        void *p = nullptr;
        TFG_HIP(hipMalloc(&p, n * sizeof(T)));
        ptrs.push_back(p);
        *out = static_cast<T *>(p);
        return TFG_OK;
    }
};

// Launch shape of the pair kernel and the streaming kernels.
struct LaunchShape {
    int nonbond_blocks = 0;   // workgroups of the pair kernel (0 = one cell per wave)
    int stream_threads = 256;
    int stream_blocks = 0;
};

// A member's last read: none since its host record, of the state it has now,
// of an earlier state that is kept.
constexpr char kReadNone = 0, kReadCurrent = 1, kReadKept = 2;

struct DeviceEnsemble {
    int precision = PREC_MIXED;
    int device = 0;
    int cus = 256;
    std::vector<Engine *> engines;
    std::vector<SysDesc> sys;
    int nsys = 0, np = 0, ncells = 0, S = 0;
    int max_sys_blocks = 1;   // energy partial blocks per system
    // has_ext: some pair potential needs the extended dispatch (radius
    // transforms, sums, periodic images)
    bool has_dpd = false, has_flux = false, has_ext = false;
    bool lean_advance = false;   // no bonds, angles, active walls or species: the lean update kernel
    int integrator = INTEG_FORWARD_EULER;   // shared by every system of the ensemble
    int nr_fluxsteps = 1;                   // shared as well
    int coef_lds_bytes = 0;   // table bytes cached in LDS by the pair kernel (0: read from global)
    NbLayout nb{};            // LDS layout of the pair kernel
    NbLayout nbs{};           // its staging area as one region, for cells that a workgroup shares
    NbLayout nbb{};           // LDS layout of the list-build variant
    NbLayout nbl{};           // LDS of the list pair kernel (off_coef: tables, off_waves: cell offsets)
    bool list_mode = false;   // neighbour lists in use (every member asked for them and can use them)
    // no_alloc: buffers from an arena, the null stream, no events, no lists
    bool no_alloc = false;
    int lcap = 0;
    int lpp = 1, lpp_log2 = 0;  // list pass lanes per particle
    int nlblocks = 0;
    int4 *d_lblock = nullptr;
    unsigned char *d_limage = nullptr;
    int *d_list = nullptr, *d_lcount = nullptr, *d_cid0 = nullptr, *d_lflags = nullptr, *d_sflags = nullptr;
    int *d_ncount = nullptr;
    void *xb = nullptr, *x0 = nullptr, *xn = nullptr;
    int max_stencil = 0;      // cells of the largest neighbour stencil
    int nb_cells = 4;         // cells of a pair-kernel workgroup
    int nonbond_resident = 0; // pair-kernel workgroups resident on the device at once
    LaunchShape shape;
    Buffers buf;
    hipStream_t stream = nullptr;
    hipEvent_t ev[8];
    int nev = 0;
    float last_ms = 0.0f;
    // phases: bin, list build, pair pass, advance (events 0..4 of a step)
    double kernel_ms[4] = {0, 0, 0, 0};
    hipGraphExec_t graph = nullptr;
    bool profile = false;
    std::vector<hipEvent_t> prof_ev;
    double prof_ms[4] = {0, 0, 0, 0};
    int prof_steps = 0;

    SysDesc *d_sys = nullptr;
    int *d_cell_sys = nullptr, *d_stencil = nullptr, *d_fluxmap = nullptr;
    int2 *d_slots = nullptr;
    int *d_wallmap = nullptr;
    void *d_pots = nullptr, *d_coef = nullptr, *d_flux = nullptr;
    TypeDesc *d_types = nullptr;
    void *pos[2] = {nullptr, nullptr}, *vel[2] = {nullptr, nullptr}, *imass[2] = {nullptr, nullptr};
    void *sp[2] = {nullptr, nullptr}, *qq[2] = {nullptr, nullptr};
    void *rk[2][5] = {{nullptr}};   // Runge-Kutta p0, v0, sx, sv, vk per buffer
    int4 *meta[2] = {nullptr, nullptr};
    void *force = nullptr;
    int *slot_of = nullptr, *cnt = nullptr, *fill = nullptr, *start = nullptr, *bsum = nullptr;
    int2 *tmp = nullptr;
    double *e_part = nullptr, *e_nb = nullptr, *e_vir = nullptr, *e_kin = nullptr, *e_bond = nullptr,
           *e_ang = nullptr;
    double *d_energy = nullptr, *d_spec_tot = nullptr, *sp_part = nullptr;
    int *inc_off = nullptr, *inc = nullptr;
    int4 *d_bonds = nullptr, *d_angles = nullptr;
    int4 *d_bslot = nullptr, *d_aslot = nullptr;
    void *d_tforce = nullptr;
    int nbonds = 0, nangles = 0;
    long long *d_step = nullptr;
    int *d_err = nullptr;

    // What the host needs to know after a call, written by k_report into
    // pinned memory as the call's last kernel; then each system's 5 sums.
    struct Status {
        long long step;
        int err[2];
        int due;      // some system waits for a full step
        int served;   // full steps that were waited for
    };
    Status *status = nullptr;
    double *status_sums() const { return reinterpret_cast<double *>(status + 1); }
    int light_run = 4;   // light steps between two full ones
    bool full_only = false;   // no light steps: almost every step waits (of the last sample, counted here)
    int sample_steps = 0, sample_waits = 0;

    // Readback: a pinned buffer and an event per reading thread.  read_lock is
    // held over a read: host threads may read several members, or one engine
    // in several ways, at once, and share the buffers and the kept state.
    std::mutex read_lock;
    struct ReadSlot {
        unsigned char *ptr = nullptr;
        size_t bytes = 0;
        hipEvent_t done = nullptr;
    };
    ReadSlot read_slot[8];
    // keep_reads: what was last read of a member is what its host engine holds
    // when it leaves the ensemble without a download.  kept: that state by id
    // on the device, for the members whose state has changed since (kept_sys).
    bool keep_reads = false;
    ReadRows kept;
    std::vector<char> kept_sys;   // kReadNone ..

    ~DeviceEnsemble() {
        if (status) (void)hipHostFree(status);
        for (ReadSlot &r : read_slot) {
            if (r.ptr) (void)hipHostFree(r.ptr);
            if (r.done) (void)hipEventDestroy(r.done);
        }
        for (hipEvent_t e : prof_ev) (void)hipEventDestroy(e);
        if (graph) (void)hipGraphExecDestroy(graph);
        for (int k = 0; k < nev; k++) (void)hipEventDestroy(ev[k]);
        if (stream) (void)hipStreamDestroy(stream);
    }

    int stream_grid() const {
        const int want = (np + shape.stream_threads - 1) / shape.stream_threads;
        const int cap = shape.stream_blocks > 0 ? shape.stream_blocks : cus * 8;
        return want < 1 ? 1 : (want < cap ? want : cap);
    }
    // Default: one cell per wave, or per workgroup of crowded cells (the hardware dispatcher balances the uneven
    // cells; measured faster than persistent ranges on 2M- and 2.6M-particle
    // systems).
    int nonbond_grid() const { return grid_of((ncells + nb_cells - 1) / nb_cells); }
    int build_grid() const { return grid_of((ncells + nb.waves - 1) / (nb.waves > 0 ? nb.waves : 1)); }   // one cell per wave
    int grid_of(int want) const {
        const int g = shape.nonbond_blocks > 0 && shape.nonbond_blocks < want ? shape.nonbond_blocks : want;
        return g < 1 ? 1 : g;
    }
};

int launch_error(const char *what);
Energies energies_of(const double *e);

template <typename real> KP<real> make_params(DeviceEnsemble *E, int energy);

// engine_force for one host engine with every device buffer carved from
// arena (cap bytes): upload, binning, nonbonded and bonded passes, energies;
// forces and number density by particle id into f (n*4).  The engine's own
// state is not changed.  Allocates no device memory, creates no stream or
// event; runs on the null stream and returns after it has drained.
int ensemble_force_arena(Engine *e, int precision, void *arena, size_t cap, double *f, Energies *en);

// Readback (readback.hip): system s from the device into its host engine's
// particles; for keep_reads the members read are kept before their state
// changes, and put back at the end.
int read_into_engine(DeviceEnsemble *E, int s);
int keep_reads(DeviceEnsemble *E);
int restore_kept(DeviceEnsemble *E);

// Binning: scan of the cell counts, placement, per-cell order and move of
// buffer B into buffer A.  Cell counts come from the previous advance.  begin:
// the first kernel of a step without lists, which also counts the step.
template <typename real> int run_bin(DeviceEnsemble *E, const KP<real> &P, bool begin);
template <typename real> int run_sync(DeviceEnsemble *E, const KP<real> &P, bool force);
// Counts particles per cell from buffer B (after an upload).
int run_count(DeviceEnsemble *E);
template <typename real> int run_nonbond(DeviceEnsemble *E, const KP<real> &P);
// Chooses the LDS layout and the resident grid of the pair kernel.
template <typename real> int nonbond_setup(DeviceEnsemble *E, int max_types, int max_coef);
// update: 0 forces only, 1 forward-Euler update, 2..5 Runge-Kutta stage 1..4.
template <typename real> int run_advance(DeviceEnsemble *E, const KP<real> &P, int update);
// Neighbour lists: the build (a variant of the pair kernel over the wider
// stencil, run when the step rebuilds) and the list pair kernel.
template <typename real> int run_list_build(DeviceEnsemble *E, const KP<real> &P);
// The pair pass's LDS contents of every system, once after the upload.
template <typename real> int run_list_image(DeviceEnsemble *E, const KP<real> &P);
template <typename real> int run_near(DeviceEnsemble *E, const KP<real> &P);
template <typename real> int run_list_force(DeviceEnsemble *E, const KP<real> &P);
// The flux-only list pass of a flux sub-step (pending flux, no forces).
template <typename real> int run_list_flux(DeviceEnsemble *E, const KP<real> &P);
// Fluxes_integrate over every particle of buffer A (the flux sub-steps).
template <typename real> int run_flux_integrate(DeviceEnsemble *E, const KP<real> &P);
template <typename real> int run_energy(DeviceEnsemble *E, const KP<real> &P);

}  // namespace tfg
