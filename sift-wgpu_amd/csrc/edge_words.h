// edge_words.h -- which word of a row of w pixels holds the four columns xw .. xw + 3
// (xw a multiple of 4) when columns outside [0, w) take the nearest pixel, and which
// of its bytes they are. Plain C++, so that the CPU tests compile it too.
//
// No word reaches past the row's last pixel, but for rows of fewer than 4 pixels: the
// columns that include it come from the row's last four pixels, by a word that need not
// be aligned, and not from the aligned word, of which up to 3 bytes lie past the row.
// After a caller's last row those are not the caller's.
#pragma once

namespace sh {

struct EdgeRow {
    int last_word;                // columns from here on take in the row's last pixel
    int last_at;                  // the word of the last four pixels
    unsigned sel_last, sel_past;  // its bytes for last_word and for the columns past it

    // where the word of columns xw .. xw + 3 begins, and the bytes to take of it (a
    // v_perm selector of one word)
    constexpr int at(int xw) const { return xw < 0 ? 0 : xw < last_at ? xw : last_at; }
    constexpr unsigned sel(int xw) const {
        return xw < 0 ? 0u : xw < last_word ? 0x03020100u : xw == last_word ? sel_last : sel_past;
    }
};

constexpr EdgeRow edge_row(int w) {
    const int last = (w - 1) & 3;             // the last pixel's column, modulo 4
    const int shift = w >= 4 ? 3 - last : 0;  // last_word less last_at
    const unsigned bytes = last == 3 ? 0x03020100u : last == 2 ? 0x02020100u : last == 1 ? 0x01010100u : 0u;
    return {(w - 1) & ~3, w >= 4 ? w - 4 : 0, bytes + (unsigned)shift * 0x01010101u,
            (unsigned)(last + shift) * 0x01010101u};
}

}  // namespace sh
