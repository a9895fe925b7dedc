// The sharing of the interface fill's directions over workgroups (csrc/iface_split.hpp)
// against measured fills, on the host.
#include "../../dns-solvers-with-grid-embedding_amd/csrc/iface_split.hpp"

#include <cstdio>

using namespace dnsg;

// us a fill (with its share of the injection) of `tiles` tiles by workgroups per tile, of a
// kernel with `slots` workgroups resident on 256 CUs; and with up to 19 single directions a
// tile, the form before units of two
static const int by[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 19};
static const struct {
    int tiles, slots;
    bool fp32_gr34;
    double before, us[11];
} measured[] = {
    {4, 512, false, 14.4, {45.0, 29.3, 23.9, 22.4, 19.4, 19.1, 20.3, 18.9, 17.4, 15.8, 14.3}},     // gratio 3, FP64
    {16, 512, false, 20.0, {62.4, 40.2, 31.8, 29.9, 24.7, 24.7, 24.3, 24.5, 21.7, 19.7, 19.6}},    // gratio 4, FP64
    {16, 768, true, 15.1, {48.7, 31.8, 24.9, 23.8, 20.2, 20.8, 19.7, 19.5, 17.2, 16.4, 14.5}},     // gratio 4, FP32
    {16, 768, false, 17.5, {36.0, 24.7, 21.5, 20.0, 17.6, 17.7, 17.9, 17.5, 16.5, 15.3, 16.5}},    // gratio 2, FP64
    {30, 1024, true, 15.7, {37.3, 25.1, 21.0, 19.4, 16.9, 16.9, 16.8, 16.8, 16.0, 14.8, 14.3}},    // gratio 3, FP32
    {32, 768, true, 17.8, {48.9, 32.2, 25.7, 24.1, 20.9, 20.5, 20.3, 20.1, 18.5, 16.9, 16.6}},     // gratio 4, FP32
    {64, 512, false, 33.0, {68.2, 47.4, 37.2, 34.4, 35.9, 35.3, 32.9, 34.6, 42.1, 37.9, 43.6}},    // gratio 4, FP64
    {64, 512, false, 34.1, {66.1, 47.6, 37.7, 35.6, 35.5, 35.0, 33.5, 35.3, 40.9, 38.9, 44.2}},    // gratio 4, FP64
    {64, 768, true, 22.1, {52.9, 32.6, 26.9, 24.2, 22.8, 22.8, 22.1, 22.6, 23.4, 21.2, 25.3}},     // gratio 4, FP32
    {64, 1024, true, 20.0, {37.9, 25.7, 21.6, 20.2, 18.5, 18.5, 18.3, 18.6, 18.2, 16.9, 19.9}},    // gratio 3, FP32
    {90, 768, false, 27.7, {37.8, 26.7, 26.9, 25.6, 22.9, 25.0, 24.4, 26.2, 27.4, 25.9, 31.4}},    // gratio 2, FP64
    {96, 768, true, 26.3, {52.9, 37.2, 30.6, 28.9, 25.8, 27.3, 27.0, 28.2, 32.5, 31.6, 34.5}},     // gratio 4, FP32
    {132, 1024, true, 25.5, {38.7, 27.4, 24.3, 24.4, 22.2, 22.9, 22.9, 27.5, 25.4, 25.7, 28.6}},   // gratio 3, FP32
    {192, 1536, false, 24.6, {30.1, 22.8, 21.1, 20.4, 19.8, 21.2, 21.9, 23.0, 22.8, 22.8, 27.1}},  // gratio 2, FP32
    {256, 512, false, 69.6, {80.6, 67.2, 79.7, 81.2, 80.3, 86.2, 92.3, 102.8, 98.1, 99.1, 132.1}}, // gratio 4, FP64
    {256, 768, true, 40.2, {53.5, 42.0, 39.2, 50.1, 45.7, 46.9, 52.6, 57.1, 54.4, 56.5, 69.6}},    // gratio 4, FP32
    {256, 2048, false, 25.1, {22.4, 18.3, 17.9, 18.0, 17.3, 17.9, 18.5, 20.8, 20.4, 20.1, 24.6}},  // gratio 1, FP32
};

int main() {
    int bad = 0;
    for (const auto &m : measured) {
        const int g = iface_groups(m.tiles, m.slots, 256, m.fp32_gr34);
        double us = 0., best = m.us[0];
        for (int i = 0; i < 11; i++) {
            if (by[i] == g) us = m.us[i];
            best = std::min(best, m.us[i]);
        }
        if (us == 0. || us > 1.03 * best || us > m.before) {
            printf("%d tiles, %d slots: %d workgroups a tile take %.1f us, the best %.1f, before %.1f\n", m.tiles, m.slots, g, us,
                   best, m.before);
            bad = 1;
        }
    }
    // the units are shared out whole, or one by one in single directions
    for (long tiles = 1; tiles < 4000; tiles += 7)
        for (long slots : {256L, 512L, 768L, 1024L, 2048L})
            for (bool w : {false, true}) {
                const int g = iface_groups(tiles, slots, 256, w);
                if (g != 19 && (g < 1 || g > IF_UNITS)) {
                    printf("%ld tiles, %ld slots: %d workgroups a tile\n", tiles, slots, g);
                    bad = 1;
                }
            }
    return bad;
}
