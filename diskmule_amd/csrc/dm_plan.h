// dm_plan.h -- launch arithmetic that a kernel and its host code share, or
// that decides which kernel takes a call.  Plain constexpr functions without
// any HIP, so that a CPU program can check them over every size.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace dm {

// The grouped-experts launch of `pairs` (token, selection) pairs: its entries
// (an expert and up to 8 of its tokens) are found on the device, and each
// workgroup works on one entry.  Two workgroups per CU, and never fewer than
// the entries, of which there are at most as many as pairs: a partition of 32
// CUs has 64 workgroups where 16 tokens can make 128 entries.
constexpr uint32_t experts_grid(uint32_t cus, uint32_t pairs) { return 2 * cus > pairs ? 2 * cus : pairs; }
// Workgroups per entry; workgroup b works on entry b / share, if there is one.
constexpr uint32_t experts_share(uint32_t grid, uint32_t entries) { return grid > entries ? grid / entries : 1u; }

}  // namespace dm
