// Host-side state of one case: parsed dictionaries, lattice tables, device buffers.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <string>
#include <vector>

#include "../../include/mplb.h"
#include "dict.h"
#include "kernels.h"
#include "mesh.h"
#include "passes.h"

namespace mplb {

struct FieldCfg {
    bool present = false;
    ModelParams mp{};
    std::vector<int> bctype;                    // bdType per boundary list
    std::vector<std::array<double, 3>> bcval;   // value entry
    std::vector<double> pert;                   // fixedRandomT pert (percent)
    std::vector<int> psteps;                    // fixedRandomT duration
    std::vector<int> localT;                    // fixedRandomT localTStep
    std::vector<std::string> bcname;            // type string as read
};

struct DevBd {
    int* nodes = nullptr;
    int n = 0;
    int sequential[2] = {0, 0};                 // per field
    int* rnd_off[2] = {nullptr, nullptr};       // fixedRandomT draw offsets per field
};

struct Timer {
    const char* name;
    double ms = 0;
    int launches = 0;
};

}  // namespace mplb

namespace mplb {
struct HostStage;
struct Tiles;

// Makes dev the calling thread's device, and its own again at the end: events and
// allocations belong to the current device, which need not be the case's.
class DeviceScope {
public:
    explicit DeviceScope(int dev) {
        if (hipGetDevice(&before_) != hipSuccess || before_ == dev) before_ = -1;
        err = hipSetDevice(dev);
    }
    ~DeviceScope() {
        if (before_ >= 0) (void)hipSetDevice(before_);
    }
    DeviceScope(const DeviceScope&) = delete;
    DeviceScope& operator=(const DeviceScope&) = delete;
    hipError_t err;

private:
    int before_ = -1;
};

// Device memory that a case can do without: a failure is no error of the call
inline bool device_alloc(void** p, size_t bytes) {
    if (hipMalloc(p, bytes ? bytes : 1) == hipSuccess) return true;
    (void)hipGetLastError();
    *p = nullptr;
    return false;
}
}

struct mplb_case {
    mplb_opts opts{};
    std::string dir;
    std::string err;
    mplb::Mesh mesh;
    mplb::EosParams eos{};
    double rho0 = 0;
    double rho0_dict = 0;                       // EOS/rho_0 as the dictionary gives it
    mplb::FieldCfg fc[2];
    int update[2] = {1, 1};
    int start = 0, end = 0, write_interval = 1, current = 0, stp = 0;
    std::string data_format = "asciiRaw";
    bool initialized = false;
    bool psi_valid = false;
    int ss_first = 1;

    // device
    int dev = 0;
    hipStream_t stream = nullptr;
    size_t scalar_bytes = 8;
    void* f[2] = {nullptr, nullptr};
    void* f_alt[2] = {nullptr, nullptr};
    void* rho = nullptr;
    void* temp = nullptr;
    void* p = nullptr;
    void* U = nullptr;
    void* Fi = nullptr;
    void* Ft = nullptr;
    void* ss = nullptr;
    void* psi = nullptr;
    int* nb = nullptr;
    uint8_t* onbnd = nullptr;
    std::vector<mplb::DevBd> bd;
    double* rnd = nullptr;                      // fixedRandomT draws r = rand()/RAND_MAX
    double* red = nullptr;                      // reduction result + partials
    unsigned int* nanc = nullptr;
    void* rho_snap = nullptr;                   // density snapshot of mplb_density_change
    bool snap_valid = false;

    // fused passes of the per-routine arithmetic (kernels_passes.hip)
    bool passes = false;
    int pass_faces = 0;                         // faces read through the neighbour table
    uint8_t* order[2] = {nullptr, nullptr};     // per field: each node's boundary list (255: none)
    void* sumg = nullptr;
    mplb::PassMarch march;                      // the single-pass march (isothermal periodic D3Q15)

    // several steps per launch on small lattices (tiles.hip): rho, T, U, Fi, Ft, ss and psi
    // of the level being written
    mplb::Tiles* tiles = nullptr;
    bool tiles_tried = false;                   // at the first init
    void* alt[7] = {nullptr};

    // fused structured-box path
    bool fused = false;
    void* fz = nullptr;                         // fused-state handle (kernels_fused.hip)

    mplb::HostStage* stage = nullptr;           // pinned buffers of large field transfers

    // timers
    bool timing = false;
    std::vector<mplb::Timer> timers;
    std::vector<hipEvent_t> ev_pool;
};

namespace mplb {
// resolve the device address of warm.hip's allocation-free scratch array for the
// case's device (once per device; the device must be current)
int warm_scratch_setup(mplb_case* c);
}  // namespace mplb
