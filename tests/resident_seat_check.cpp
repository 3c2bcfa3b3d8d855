// Launches and turns of resident kernels over a stand-in for the runtime: what is called is printed, and an event is recorded on, and waited for by, streams as HIP has it
// (recording: only on a stream of the event's own device).  Argument: the scenario.
#include <hip/hip_runtime_api.h>
#include <stdio.h>

#include <string>

#include "forge_hip.h"
#include "resident_seat.h"

namespace {
struct Stream { int device; const char* name; };
struct Event { int device; };
int current = 0;
bool record_fails = false, wait_fails = false;
hipStream_t handle(Stream& s) { return reinterpret_cast<hipStream_t>(&s); }
const char* name(hipStream_t s) { return reinterpret_cast<Stream*>(s)->name; }
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipDeviceSynchronize() { printf("sync device %d\n", current); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(new Event{current}); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (record_fails) return hipErrorOutOfMemory;
    if (reinterpret_cast<Event*>(e)->device != reinterpret_cast<Stream*>(s)->device) return hipErrorInvalidHandle;
    printf("record %s\n", name(s));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) {
    if (wait_fails) return hipErrorUnknown;
    printf("wait %s\n", name(s));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { printf("sync %s\n", name(s)); return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3 block, void**, size_t lds, hipStream_t s) {
    printf("ordinary %s %u %u %zu\n", name(s), grid.x, block.x, lds);
    return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void*, dim3 grid, dim3 block, void**, unsigned lds, hipStream_t s) {
    printf("cooperative %s %u %u %u\n", name(s), grid.x, block.x, lds);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace fh {
int32_t fail(int32_t code, const std::string&) { return code; }
}  // namespace fh

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    Stream a{0, "a"}, b{0, "b"};
    auto step = [](fh::ResidentSeat& seat, Stream& s) {
        const int32_t rc = seat.turn(handle(s), [&] { printf("launch %s\n", s.name); return (int32_t)FORGE_HIP_OK; });
        printf("-> %d\n", rc);
    };
    if (what == "offsets") {
        // the last row of a cache and of an output matrix that 32 bits reach, and the first that they do not
        printf("%d %d %d %d %d %d\n", fh::decode_ahead_offsets_fit((1u << 21) - 1, 1024, 128256, 2048, false), fh::decode_ahead_offsets_fit(1u << 21, 1024, 128256, 2048, false),
               fh::decode_ahead_offsets_fit(4096, 512, (1u << 21) - 1, 2048, false), fh::decode_ahead_offsets_fit(4096, 512, 1u << 21, 2048, false),
               fh::decode_ahead_offsets_fit(4096, 512, (1u << 22) - 1, 2048, true), fh::decode_ahead_offsets_fit(4096, 512, 1u << 22, 2048, true));
    } else if (what == "copy") {
        // the 1B shape: 1.236e9 weights, 1.39 GB; free memory that just suffices, and a byte less
        const uint64_t blocks = 1235746816ull / 32, need = fh::decode_ahead_copy_bytes(blocks) * 8;
        printf("%d %d %d\n", fh::decode_ahead_copy_fits(blocks, need), fh::decode_ahead_copy_fits(blocks, need - 1), fh::decode_ahead_copy_fits(blocks, 0));
    } else if (what == "launch") {
        (void)fh::resident_launch(nullptr, 256, 768, nullptr, 1000, fh::resident_cooperative(), handle(a));
    } else if (what == "one") {
        fh::ResidentSeat seat;
        step(seat, a);
        step(seat, a);
    } else if (what == "two") {
        fh::ResidentSeat one, other;
        step(one, a);
        step(one, a);
        step(other, b);
        step(one, a);
    } else if (what == "devices") {
        // a model on each of two devices, then a second one on the second; steps come while the first device is current
        Stream c{1, "c"}, d{1, "d"};
        fh::ResidentSeat one;
        current = 1;
        fh::ResidentSeat other;
        current = 0;
        step(one, a);
        step(other, c);
        step(one, a);
        current = 1;
        fh::ResidentSeat third;
        current = 0;
        step(other, c);
        step(one, a);
        step(third, d);
    } else if (what == "record fails") {
        fh::ResidentSeat one, other;
        record_fails = true;
        step(one, a);
        record_fails = false;
        step(other, b);
        step(one, a);
    } else if (what == "wait fails") {
        fh::ResidentSeat one, other;
        step(one, a);
        wait_fails = true;
        step(other, b);
    } else {
        return 2;
    }
    return 0;
}
