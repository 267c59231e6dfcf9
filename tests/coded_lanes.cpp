// Replays on the CPU what every lane of a coded kernel's grid reads: a banded
// matrix's codes and table as codes_build lays them out, then the words, table
// entries and byte offsets of each lane as k_coded forms them.
// argv: n, words of a row, bytes of a vector's entry, then the band's offsets.
// Prints the entries read outside the vector or off its entries' grid, the rows
// whose entries are not the matrix's, and the lanes without a row that read
// another entry than padding.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "coded_lane.h"

int main(int argc, char **argv) {
    const int n = std::atoi(argv[1]), words = std::atoi(argv[2]);
    const unsigned int bytes = (unsigned int)std::atoi(argv[3]);
    std::vector<int> off;   // the table: code = place
    for (int k = 4; k < argc; ++k) off.push_back(std::atoi(argv[k]));
    const int nslices = (n + hz::kCodeRows - 1) / hz::kCodeRows;
    std::vector<unsigned int> code((size_t)nslices * words * hz::kCodeRows, hz::kCodePadWord);
    std::vector<int> count(n, 0);
    for (int r = 0; r < n; ++r) {
        int k = 0;
        for (int c = 0; c < (int)off.size(); ++c) {
            if (r + off[c] < 0 || r + off[c] >= n) continue;
            unsigned int &w = code[((size_t)(r / hz::kCodeRows) * words + k / 4) * hz::kCodeRows + r % hz::kCodeRows];
            w = (w & ~(0xFFu << (8 * (k % 4)))) | ((unsigned int)c << (8 * (k % 4)));
            ++k;
        }
        count[r] = k;
    }
    long outside = 0, wrong = 0, stray = 0;
    const int blocks = (nslices + 3) / 4;   // four wavefronts a workgroup, a slice each
    for (int s = 0; s < 4 * blocks; ++s)
        for (int lane = 0; lane < hz::kCodeRows; ++lane) {
            const hz::CodedLane l = hz::coded_lane(s, lane, n, nslices, words, bytes);
            int entries = 0;
            for (int k = 0; k < words + 3; ++k)   // a round reads up to three words past the last
                for (int u = 0; u < 4; ++u) {
                    if (k < words && l.first + (size_t)k * hz::kCodeRows >= code.size()) {
                        ++outside;
                        continue;
                    }
                    const unsigned int h = hz::coded_entry(hz::coded_word(l, code.data(), k, words), u);
                    const bool pad = h == (unsigned int)hz::kCodePad;
                    const unsigned int at = l.base + (unsigned int)(pad ? 0 : off[h] * (int)bytes);
                    if (at >= (unsigned long long)n * bytes || at % bytes) ++outside;
                    entries += !pad;
                }
            if (l.in) wrong += entries != count[l.row];
            else stray += entries != 0;
        }
    std::printf("outside %ld wrong %ld stray %ld\n", outside, wrong, stray);
    return outside || wrong || stray;
}
