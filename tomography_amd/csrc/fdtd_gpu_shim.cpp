// fdtd_gpu_shim.cpp — the reference's objective entry points with their exact
// C++ signatures, so that a search driver written against FDTD_GPU.cuh:8 and
// FDTD_CPU.h:8 (e.g. test.cxx:94-121, which passes them to TAO as function
// pointers) links against libtomo.so unchanged.
//
//   double FDTD_GPU(const std::vector<double>&)  : REF_GPU preset, 27 parameters,
//       fitness -sum (D - m)^2 / 40 (FDTD_GPU.cu:1004-1008);
//   double FDTD_CPU(const std::vector<double>&)  : REF_CPU preset, 162 parameters,
//       fitness -sum (D - m)^2 / (m^2 40) (FDTD_CPU.cxx:841-845), evaluated by
//       the same gfx950 kernels with the CPU-path semantics.
//
// The "measurement" m is read from a file (the reference hard-codes it at
// FDTD_GPU.cu:996 and FDTD_CPU.cxx:789): $TOMO_MEASUREMENT_GPU /
// $TOMO_MEASUREMENT_CPU, else data/measurement_{gpu,cpu}.f32 next to the
// package (raw little-endian float32, D[exc][freq][angle] then, for the GPU
// file, the phase P in the same layout).
//
// Differences from the reference, by design: a HIP failure throws
// std::runtime_error instead of exit(-1) (FDTD_GPU.cu:35-48); a short vector
// throws std::out_of_range exactly like its vector::at; the device context
// persists between calls (the reference mallocs and frees per call).
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/tomo.h"

namespace {

std::mutex g_mu;
tomo_ctx* g_ctx = nullptr;

std::string data_dir() {
    Dl_info info;
    if (dladdr((void*)&data_dir, &info) && info.dli_fname) {
        std::string p(info.dli_fname);
        const size_t k = p.find_last_of('/');
        return (k == std::string::npos ? std::string(".") : p.substr(0, k)) + "/data";
    }
    return "data";
}

std::vector<float> load_measurement(const char* env, const char* name, size_t n) {
    const char* e = std::getenv(env);
    const std::string path = e ? std::string(e) : data_dir() + "/" + name;
    std::vector<float> v;
    FILE* f = std::fopen(path.c_str(), "rb");
    if (!f) throw std::runtime_error("cannot open measurement file " + path);
    v.resize(n);
    const size_t got = std::fread(v.data(), sizeof(float), n, f);
    std::fclose(f);
    if (got < n) throw std::runtime_error("measurement file " + path + " is shorter than expected");
    return v;
}

tomo_ctx* ctx() {
    if (!g_ctx) {
        const char* d = std::getenv("TOMO_DEVICE");
        if (tomo_ctx_create(d ? std::atoi(d) : 0, 0, &g_ctx) != TOMO_OK)
            throw std::runtime_error(std::string("tomo_ctx_create: ") + tomo_last_error());
        // the schedule whose DFT chunk the drop-in's results are compared under
        const tomo_schedule s = TOMO_DROPIN_SCHEDULE;
        if (tomo_set_schedule(g_ctx, &s) != TOMO_OK)
            throw std::runtime_error(std::string("tomo_set_schedule: ") + tomo_last_error());
    }
    return g_ctx;
}

// Packaged measurement of a reference preset (loaded once).
const std::vector<float>& packaged_measurement(int preset) {
    static std::vector<float> meas_gpu, meas_cpu;
    const bool gpu = preset == TOMO_PRESET_REF_GPU;
    std::vector<float>& m = gpu ? meas_gpu : meas_cpu;
    if (m.empty()) {
        tomo_sim_config cfg;
        if (tomo_preset(preset, 0, &cfg) != TOMO_OK) throw std::runtime_error(tomo_last_error());
        const size_t L = (size_t)tomo_farfield_len(&cfg);
        m = gpu ? load_measurement("TOMO_MEASUREMENT_GPU", "measurement_gpu.f32", 2 * L)
                : load_measurement("TOMO_MEASUREMENT_CPU", "measurement_cpu.f32", L);
    }
    return m;
}

double run(int preset, const std::vector<double>& arguments, const char* label) {
    std::lock_guard<std::mutex> g(g_mu);
    double fit = 0;
    const int rc = tomo_fitness(ctx(), preset, 0, arguments.data(), arguments.size(), nullptr, 0, &fit);
    if (rc == TOMO_E_SHORT) throw std::out_of_range("vector::_M_range_check");
    if (rc != TOMO_OK) throw std::runtime_error(std::string("tomo_fitness: ") + tomo_last_error());
    std::cout << label << fit << std::endl;
    return fit;
}

}  // namespace

extern "C" int tomo_fitness(tomo_ctx* c, int preset, int32_t flags, const double* params, size_t n_params,
                            const float* measurement, size_t n_measurement, double* fitness_out) {
    tomo_sim_config cfg;
    int rc = tomo_preset(preset, 0, &cfg);
    if (rc) return rc;
    cfg.flags |= flags;
    if (!measurement && cfg.mode == TOMO_MODE_REF_COMPAT) {
        try {
            const std::vector<float>& m = packaged_measurement(preset);
            measurement = m.data();
            n_measurement = m.size();
        } catch (const std::exception&) {
            return TOMO_E_INVALID;
        }
    }
    // The vector's excitations are independent simulations: they advance
    // together (the batched form, whose results equal tomo_eval's bit for bit).
    return tomo_eval_batch(c, &cfg, params, 1, n_params, measurement, n_measurement, fitness_out, nullptr);
}

double FDTD_GPU(const std::vector<double>& arguments) { return run(TOMO_PRESET_REF_GPU, arguments, "fitness is: "); }

double FDTD_CPU(const std::vector<double>& arguments) { return run(TOMO_PRESET_REF_CPU, arguments, " fitness = "); }
