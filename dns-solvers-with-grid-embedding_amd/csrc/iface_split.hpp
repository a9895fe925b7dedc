// iface_split.hpp -- how the interface fill shares a tile's directions out over workgroups.
#pragma once
#include <algorithm>

namespace dnsg {

constexpr int IF_UNITS = 10;  // pairs of directions, and the rest direction alone

// Workgroups per tile, for `tiles` tiles of a kernel of which the GPU holds `slots`
// workgroups at once (CUs x resident workgroups per CU): a launch whose tiles alone fill them
// (the Re_tau=180 bands: 1024 tiles) takes 1, a launch of small channels (the serving queue)
// shortens its chains.  Only the numbers that shorten the longest chain are taken: 2, 3, 5,
// 10 (7 to 9 give the chain of 5 with more work: gratio 2, FP64, 90 tiles 26.2 us with 8,
// 22.9 with 5; FP32, 192 tiles 23.0 and 19.8), but 7 where 5 gives fewer than half of the
// CUs a second workgroup and the launch waits for those (gratio 4, FP64, 64 tiles: 35.9 us
// with 5, 34.6 with 8, 32.9 with 7).
// 19, one direction each, where every workgroup then has a CU of its own (gratio 3, 4 tiles:
// 11.4 and 10.0 us a launch against 13.2 and 11.6 with 10; gratio 2, 16 tiles, whose 304
// workgroups share CUs: 12.5 and 11.4 against 11.8 and 10.2), and up to 2.5 a CU where they
// fit with FP32 planes at gratio 3 and 4 (16 tiles 13.5 and 14.5 us against 14.3 and 16.3
// with 10; 30 tiles 14.3 against 14.8; 64 tiles 19.8 against 16.9).
inline int iface_groups(long tiles, long slots, long cus, bool fp32_gr34) {
    if (tiles >= slots) return 1;
    if (tiles * 19 <= (fp32_gr34 ? std::min(slots, 5 * cus / 2) : cus)) return 19;
    const long most = slots / tiles;
    if (most >= 10) return 10;
    if (most >= 7 && 2 * tiles * 5 < 3 * cus) return 7;
    return most >= 5 ? 5 : (most >= 3 ? 3 : (int)most);
}

}  // namespace dnsg
