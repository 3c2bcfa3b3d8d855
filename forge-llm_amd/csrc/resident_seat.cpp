#include "resident_seat.h"

#include <mutex>
#include <string>

#include "forge_hip.h"

namespace fh {

int32_t fail(int32_t code, const std::string& msg);       // common.h, which a host compiler does not take

namespace {
std::mutex seat_mutex;
uint32_t seats = 0;
hipEvent_t seat_event = nullptr;          // behind the launch before; null until there was a second seat
hipStream_t seat_stream = nullptr;        // that launch's, or null if it has ended
}  // namespace

ResidentSeat::Lock::Lock() { seat_mutex.lock(); }
ResidentSeat::Lock::~Lock() { seat_mutex.unlock(); }
ResidentSeat::ResidentSeat() {
    const Lock lock;
    // launches made while there was one seat left no event: they end here
    if (++seats == 2) (void)hipDeviceSynchronize();
}
ResidentSeat::~ResidentSeat() {
    const Lock lock;
    if (--seats > 0) return;
    if (seat_event) (void)hipEventDestroy(seat_event);
    seat_event = nullptr;
    seat_stream = nullptr;
}
int32_t ResidentSeat::before(hipStream_t s) {
    if (seats < 2 || !seat_stream || seat_stream == s) return FORGE_HIP_OK;
    const hipError_t e = hipStreamWaitEvent(s, seat_event, 0);
    return e == hipSuccess ? FORGE_HIP_OK : fail(FORGE_HIP_ERR_HIP, std::string("resident decode: the wait for another model's step: ") + hipGetErrorString(e));
}
// The step is on its way, whatever happens here: where nothing can be left for the next launch to wait for, this one is waited for at once.
void ResidentSeat::after(hipStream_t s) {
    if (seats < 2) return;
    seat_stream = s;
    if (!seat_event && hipEventCreateWithFlags(&seat_event, hipEventDisableTiming) != hipSuccess) seat_event = nullptr;
    if (seat_event && hipEventRecord(seat_event, s) == hipSuccess) return;
    (void)hipGetLastError();
    (void)hipStreamSynchronize(s);
    seat_stream = nullptr;
}

}  // namespace fh
