// coded_lane.h -- what a lane of a kernel over entry codes reads (coded.hpp):
// its row, its place in the codes, its words, and the byte offset of the row's
// own entry in a vector, to which the table's offsets are added.  Plain
// constexpr functions, so that host code can replay every lane of a grid.
#pragma once
#include <cstddef>

namespace hz {

constexpr int kCodes = 256, kCodePad = 255;   // codes of a byte, and the one of padding (offset 0, value 0)
constexpr int kCodeRows = 64;                 // rows of a slice
constexpr unsigned int kCodePadWord = 0xFFFFFFFFu;   // four paddings

struct CodedLane {
    int row;
    bool in;               // the lane has a row of the matrix
    size_t first;          // its first word; the next ones follow kCodeRows apart
    unsigned int base;     // byte offset of its row (without one: of the last row)
};

// Lane `lane` of the wavefront that takes slice s.  The grid is whole
// workgroups, so the last one can have wavefronts past the last slice (s >=
// nslices): none of their lanes has a row.
constexpr CodedLane coded_lane(int s, int lane, int n, int nslices, int words, unsigned int bytes) {
    const int r = s * kCodeRows + lane;
    return {r, r < n, (size_t)(s < nslices ? s : nslices - 1) * words * kCodeRows + lane,
            (unsigned int)(r < n ? r : n - 1) * bytes};
}

// Word k of a lane: padding past the last word, and everywhere in a lane without
// a row, whose slice's real offsets would lead past the vector from base.
template <class W>
constexpr unsigned int coded_word(const CodedLane &l, const W *code, int k, int words) {
    return l.in && k < words ? (unsigned int)code[l.first + (size_t)k * kCodeRows] : kCodePadWord;
}

constexpr unsigned int coded_entry(unsigned int word, int u) { return (word >> (8 * u)) & 0xFFu; }

}  // namespace hz
