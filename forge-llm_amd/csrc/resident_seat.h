// Whose turn it is to launch a resident kernel.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace fh {

// The workgroups of a resident kernel wait for each other, so all of them have to be on the device at once.  One such kernel takes every compute unit; were two launched
// side by side (models of two threads), each could get a part and wait for the rest until its polls run out.  A model that launches one holds a seat: while there are
// several seats in the process, a launch on another stream than the one before it waits for that one to end.  With a single seat nothing is recorded.
class ResidentSeat {
public:
    ResidentSeat();
    ~ResidentSeat();
    ResidentSeat(const ResidentSeat&) = delete;
    ResidentSeat& operator=(const ResidentSeat&) = delete;
    // launch(): enqueues on s.  Fails only where nothing was launched.
    template <typename F>
    int32_t turn(hipStream_t s, F launch) {
        const Lock lock;
        int32_t rc = before(s);
        if (!rc) rc = launch();
        if (!rc) after(s);
        return rc;
    }

private:
    struct Lock { Lock(); ~Lock(); };
    static int32_t before(hipStream_t s);
    static void after(hipStream_t s);
};

}  // namespace fh
