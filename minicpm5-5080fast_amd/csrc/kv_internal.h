// kv_internal.h - declarations shared by the host-side translation units.
#pragma once

#include "kv_common.h"

namespace mckv {

// Validates an mc_kv_layout_t (power-of-two page size, non-zero sizes) and
// fills the device view.
bool layout_valid(const mc_kv_layout_t& l, DevLayout* out);

}  // namespace mckv

namespace mckv {

// Deterministic synthetic qkv rows (synth.hip).
mc_status_t launch_synth_qkv(uint16_t* rows, uint32_t n, const int32_t* tokens,
                             const uint32_t* base_pos, uint32_t layer, hipStream_t st);
mc_status_t launch_synth_qkv_batch(uint16_t* rows, uint32_t n,
                                   const int32_t* const* slot_tok,
                                   const uint32_t* const* slot_pos, uint32_t layer,
                                   hipStream_t st);

// Prefill half-barrier status (attention_prefill.hip): after the caller's
// prefill work has been synchronized, reads and clears the device's timeout
// count; MC_E_INTERNAL (with a message) when it is non-zero.
mc_status_t prefill_barrier_check(const char* who);


// mc_kv_attention_prefill for a caller that knows on the host how many keys
// the chunk's last row attends (keys; 0 = not known): they decide the workgroup
// shape and how many of the S_kv splits are used.
mc_status_t prefill_attention(const uint16_t* d_q_rows, uint32_t tokens,
                              const uint32_t* d_base_pos, uint32_t layer,
                              const uint32_t* d_page_table, const uint16_t* d_kv_pool,
                              mc_kv_layout_t layout, uint16_t* d_out, float* d_partials,
                              uint32_t S_kv, uint32_t keys, void* stream);

}  // namespace mckv
