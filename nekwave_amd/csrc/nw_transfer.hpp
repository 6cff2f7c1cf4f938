// nw_transfer.hpp -- states between the caller's host arrays and the device.
#pragma once

#include <type_traits>

#include "nw_internal.hpp"

namespace nw {

// One state on the device: component c of node p at c * cs + p * ns, in FP64 or FP32.
struct DeviceState {
    void* data;
    bool f64;
    long long cs, ns;
};

// Pinned staging, per device: up to kStageSlots slots of kStageBytes for a large transfer,
// kSmallSlots for small ones, made when a transfer first needs them and freed when the
// device's last solver is gone.  Large transfers of one device take turns (they share its
// link); small ones and other devices' do not wait for them.
constexpr int kStageSlots = 8, kSmallSlots = 4;
constexpr size_t kStageBytes = size_t(2) << 20;
void stage_retain(int device);
void stage_release(int device);

// host (6 component blocks of P values, FP64) -> device, or back.  Returns when
// the host array has been read (the device then holds the state in stream
// order) or written.
int upload_state(int device, hipStream_t s, const double* host, long long P, const DeviceState& d);
int download_state(int device, hipStream_t s, double* host, long long P, const DeviceState& d);
// `bytes` (any number) from device memory to the caller's array (host or device memory),
// in stream order, waited for.
int download_bytes(int device, hipStream_t s, void* host, const void* dev, size_t bytes);

// Whether p is memory of a device (then the plain copies are used).
bool device_pointer(const void* p);

}  // namespace nw
