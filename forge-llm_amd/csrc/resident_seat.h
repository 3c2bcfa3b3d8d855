// The host's side of the resident kernels: what they can reach, how they are launched, and whose turn it is.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace fh {

// decode_ahead_kernel finds a layer's cached rows and the blocks of a matrix by 32-bit byte offsets.  (Its other matrices are smaller than the output matrix can be:
// at most 8192 by 2048 twice.)
constexpr bool decode_ahead_offsets_fit(uint64_t max_seq, uint64_t kv_channels, uint64_t vocab, uint64_t hidden, bool lm_head_q4) {
    return max_seq * kv_channels * 2 <= 0xFFFFFFFFull && vocab * hidden / (lm_head_q4 ? 2 : 1) <= 0xFFFFFFFFull;
}

// A K-quant model's matrices as decode_ahead_kernel reads them are a copy of `blocks` blocks of 36 bytes.  It buys time only (decode_persistent_kernel runs the same models), so
// it takes an eighth of the free memory at most: a model of up to 2048 channels next to others finds room for what it cannot do without.
constexpr uint64_t decode_ahead_copy_bytes(uint64_t blocks) { return blocks * 36; }
constexpr bool decode_ahead_copy_fits(uint64_t blocks, uint64_t free_bytes) { return decode_ahead_copy_bytes(blocks) <= free_bytes / 8; }

// All workgroups are co-resident by construction (one per compute unit, checked when the model is created) and every wait in the kernel is bounded, so an ordinary launch
// is enough; it costs ~7 us less per step than a cooperative one, which checks again.  FORGE_HIP_PD_COOP=1 asks for that one.
bool resident_cooperative();
hipError_t resident_launch(const void* kernel, uint32_t grid, uint32_t threads, void** args, uint32_t lds, bool cooperative, hipStream_t s);

// The workgroups of a resident kernel wait for each other, so all of them have to be on the device at once.  One such kernel takes every compute unit; were two launched
// side by side (models of two threads), each could get a part and wait for the rest until its polls run out.  A model that launches one holds a seat of its device: while
// there are several seats of a device, a launch on another stream than the one before it waits for that one to end.  With a single seat nothing is recorded.
// (What recording costs a model beside an idle one, us a token alone / with it: SmolLM2-135M 387 / 387, 1B shape 434 / 434.)
class ResidentSeat {
public:
    ResidentSeat();                           // of the current device
    ~ResidentSeat();
    ResidentSeat(const ResidentSeat&) = delete;
    ResidentSeat& operator=(const ResidentSeat&) = delete;
    // launch(): enqueues on s.  Fails only where nothing was launched.
    template <typename F>
    int32_t turn(hipStream_t s, F launch) {
        const Lock lock(dev);
        int32_t rc = before(s);
        if (!rc) rc = launch();
        if (!rc) after(s);
        return rc;
    }

private:
    struct Device;                            // what the seats of one device share
    struct Lock {
        Device* d;
        explicit Lock(Device* device);
        ~Lock();
    };
    Device* dev;
    int32_t before(hipStream_t s);
    void after(hipStream_t s);
};

}  // namespace fh
