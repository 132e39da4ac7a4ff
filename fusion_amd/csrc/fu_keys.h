// What relocalisation (reloc.hip) uses of the keypoint map (keymap.hip) beside its C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/fusion_amd.h"

namespace fu {

// a fu_surf without its descriptor
struct alignas(16) SurfHead {
    unsigned char valid;
    unsigned char pad[3];
    float pos[3];
    float normal[4];
};

uint32_t keymap_count(const fu_keymap* k);
fu_status keymap_pack(fu_keymap* k, float* desc, int32_t* slot, uint32_t n, hipStream_t s);
const SurfHead* keymap_heads(const fu_keymap* k);  // of the map's slots, kSlotHeads apart
constexpr int kSlotHeads = sizeof(fu_surf) / sizeof(SurfHead);
int keymap_device(const fu_keymap* k);
fu_status build_adjacency(const SurfHead* frame, const SurfHead* map, int stride, const float* dist, int n, float* matrix,
                          hipStream_t s);

}  // namespace fu
