// The tiles of a grid of several matrices (qmmh_tile_at): each is some workgroup's, and the XCDs, every eighth workgroup, have their
// share of each matrix.
#include "aq_qmm.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

int main() {
    srand(1);
    for (int round = 0; round < 3000; round++) {
        aq::QmmSegment seg[aq::kQmmSegments] = {};
        const int count = 1 + rand() % aq::kQmmSegments, bands = rand() % 12;
        std::vector<int> first(count + 1, 0);
        for (int i = 0; i < count; i++) {
            seg[i].strips = 1 + rand() % 20;
            seg[i].ksplit = 1 + rand() % 6;
            first[i + 1] = first[i] + bands * seg[i].strips * seg[i].ksplit;
        }
        std::vector<int> taken(first[count], 0), on_xcd((count + 1) * 8, 0);
        for (int place = 0; place < (first[count] + 7) / 8 * 8; place++) {
            const aq::QmmTileAt at = aq::qmmh_tile_at(seg, count, bands, place);
            if (at.seg < 0) continue;
            const int units = seg[at.seg].strips * seg[at.seg].ksplit;
            if (at.id < 0 || at.id >= bands * units || at.units != units || taken[first[at.seg] + at.id]++) {
                printf("round %d, workgroup %d: tile %d of matrix %d\n", round, place, at.id, at.seg);
                return 1;
            }
            on_xcd[at.seg * 8 + place % 8]++, on_xcd[count * 8 + place % 8]++;
        }
        for (int i = 0; i <= count; i++) {
            const int tiles = i < count ? first[i + 1] - first[i] : first[count];
            for (int x = 0; x < 8; x++)
                if (on_xcd[i * 8 + x] != tiles / 8 && on_xcd[i * 8 + x] != (tiles + 7) / 8) {
                    printf("round %d: %d of the %d tiles of matrix %d on XCD %d\n", round, on_xcd[i * 8 + x], tiles, i, x);
                    return 1;
                }
        }
    }
    puts("ok");
    return 0;
}
