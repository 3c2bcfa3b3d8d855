#include "resident_seat.h"

#include <stdlib.h>

#include <map>
#include <mutex>
#include <string>

#include "forge_hip.h"

namespace fh {

int32_t fail(int32_t code, const std::string& msg);       // common.h, which a host compiler does not take

bool resident_cooperative() {
    const char* e = getenv("FORGE_HIP_PD_COOP");
    return e && e[0] == '1';
}
hipError_t resident_launch(const void* kernel, uint32_t grid, uint32_t threads, void** args, uint32_t lds, bool cooperative, hipStream_t s) {
    return cooperative ? hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(threads), args, lds, s) : hipLaunchKernel(kernel, dim3(grid), dim3(threads), args, lds, s);
}

struct ResidentSeat::Device {
    std::mutex mutex;
    uint32_t seats = 0;
    hipEvent_t event = nullptr;               // behind the launch before; null until there was a second seat
    hipStream_t stream = nullptr;             // that launch's, or null if it has ended
};

ResidentSeat::Lock::Lock(Device* device) : d(device) { d->mutex.lock(); }
ResidentSeat::Lock::~Lock() { d->mutex.unlock(); }
ResidentSeat::ResidentSeat() {
    // never destroyed: a model may outlive the statics of its process
    static std::mutex* mutex = new std::mutex;
    static auto* devices = new std::map<int, Device>;
    int id = 0;
    (void)hipGetDevice(&id);
    {
        const std::lock_guard<std::mutex> one(*mutex);
        dev = &(*devices)[id];
    }
    const Lock lock(dev);
    if (++dev->seats != 2) return;
    // launches made while there was one seat left no event: they end here.  An event belongs to the device that is current when it is made.
    (void)hipDeviceSynchronize();
    if (!dev->event && hipEventCreateWithFlags(&dev->event, hipEventDisableTiming) != hipSuccess) { dev->event = nullptr; (void)hipGetLastError(); }
}
ResidentSeat::~ResidentSeat() {
    const Lock lock(dev);
    if (--dev->seats > 0) return;
    if (dev->event) (void)hipEventDestroy(dev->event);
    dev->event = nullptr;
    dev->stream = nullptr;
}
int32_t ResidentSeat::before(hipStream_t s) {
    if (dev->seats < 2 || !dev->stream || dev->stream == s) return FORGE_HIP_OK;
    const hipError_t e = hipStreamWaitEvent(s, dev->event, 0);
    return e == hipSuccess ? FORGE_HIP_OK : fail(FORGE_HIP_ERR_HIP, std::string("resident decode: the wait for another model's step: ") + hipGetErrorString(e));
}
// The step is on its way, whatever happens here: where nothing can be left for the next launch to wait for, this one is waited for at once.
void ResidentSeat::after(hipStream_t s) {
    if (dev->seats < 2) return;
    dev->stream = s;
    if (dev->event && hipEventRecord(dev->event, s) == hipSuccess) return;
    (void)hipGetLastError();
    (void)hipStreamSynchronize(s);
    dev->stream = nullptr;
}

}  // namespace fh
