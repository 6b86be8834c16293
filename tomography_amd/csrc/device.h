// device.h — small device helpers shared by the kernel files.
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "tomo_internal.h"

// Global-address-space views: loads and stores through these compile to
// global_* instructions (not flat_*), so LDS waits never wait on HBM.
#define GAS __attribute__((address_space(1)))
// Constant-address-space views of data that is read-only for a whole launch
// (row spans, the source waveform): wave-uniform loads through these become
// scalar loads (s_load_*), which are tracked by lgkmcnt and so never force a
// wait on the vector loads prefetched rows ahead.
#define CAS __attribute__((address_space(4)))

namespace tomo {
typedef GAS float gfloat;
typedef GAS const float gcfloat;
typedef GAS const uint8_t gcu8;
typedef GAS const int gcint;
typedef CAS const int kcint;
typedef CAS const float kcfloat;

// Events armed for the calling thread's next timed launch (arm_launch_events);
// taking them disarms.
void take_launch_events(hipEvent_t* start, hipEvent_t* stop);
}  // namespace tomo

// A launch whose dispatch packet carries the armed start/stop events (none
// when nothing is armed); the events are consumed by this launch.
#define TIMED_LAUNCH(K, G, B, SHM, ST, ...)                                 \
    do {                                                                    \
        hipEvent_t ea_, eb_;                                                \
        ::tomo::take_launch_events(&ea_, &eb_);                             \
        hipExtLaunchKernelGGL(K, G, B, SHM, ST, ea_, eb_, 0u, __VA_ARGS__); \
    } while (0)
