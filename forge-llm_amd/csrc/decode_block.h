// What decode_block.hip is made of: a block network's layer runs as it sees them.
#pragma once

#include <vector>

#include "checkpoint.h"
#include "common.h"

namespace fh {

// decode_block.hip — the decode step of a bfloat16 block network as one resident kernel.  The functions are the pd_ ones' counterparts.
struct PbMixer {
    MixerKind kind;
    LatentShape latent;                      // the kind's own is filled, the others are as constructed
    GroupedShape grouped;
    LinearShape linear;
    DenseWeight in, o, uq, ukv;
    const float *wa = nullptr, *wb = nullptr, *wc = nullptr;      // latent: norms of the query and of the key / value latent; grouped: of q and k; linear: W2, its bias, the heads' norm
    const float *cos_t = nullptr, *sin_t = nullptr;
    size_t values_at = 0;                    // grouped: from a run's cache to its values
};
struct PbLayerIn {                           // one layer run
    const PbMixer* mixer;
    DenseWeight gate_up, down;
    DynTanh norm1, norm2, post1, post2;      // elementwise norms
    LayerNorm ln1, ln2;                      // else these
    void* cache;
    bool pass_start;
    Act act;
    uint32_t ff;                             // padded; 0: none
};
struct PbModelIn {
    std::vector<PbLayerIn> layers;
    bool elementwise;
    uint32_t width, ln_n, max_seq;
    DenseWeight head, loop;
    DynTanh final_norm;
    const float* ln_final;
    float ln_eps, embed_scale, cap;
    const void* table;
    uint32_t table_ld, table_n;
    float* logits;
    uint32_t *state, *counts;
};
struct PbState;
int32_t pb_create(const PbModelIn& in, PbState** out);
void pb_destroy(PbState* st);
bool pb_covers(const PbState* st, int64_t pos);
void pb_set_repeat_penalty(PbState* st, float penalty);
void pb_set_poll_limit(PbState* st, uint32_t n);
int32_t pb_enqueue(PbState* st, int64_t pos, bool profile, uint32_t token, uint32_t step_seq, hipStream_t s);
bool pb_wait_token(PbState* st, uint32_t* next);
int32_t pb_after_sync(PbState* st, uint32_t abort_flag, hipStream_t s);
int32_t pb_phase_ms(PbState* st, std::vector<float>* out, hipStream_t s);

}  // namespace fh
