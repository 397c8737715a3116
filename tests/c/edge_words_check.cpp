// Every word that the one-launch blur loads at an image's edges, for rows of 1 to 400
// pixels: with 4 pixels or more it lies in the row, and its selected bytes are the
// columns' pixels, those outside the row as the nearest one inside.
#include <algorithm>
#include <cstdio>

#include "edge_words.h"

int main() {
    for (int w = 1; w <= 400; w++) {
        constexpr int kMargin = 320;  // a tile's columns and halo past the image
        const sh::EdgeRow row = sh::edge_row(w);
        for (int xw = -kMargin; xw < w + kMargin; xw += 4) {
            const int at = row.at(xw);
            if (at < 0 || (w >= 4 && at + 4 > w)) return printf("w %d xw %d: word at %d\n", w, xw, at), 1;
            for (int b = 0; b < 4; b++) {
                const int byte = (int)(row.sel(xw) >> (8 * b)) & 255;
                const int want = std::min(std::max(xw + b, 0), w - 1);
                if (byte > 3 || at + byte != want)
                    return printf("w %d column %d: byte %d of the word at %d\n", w, xw + b, byte, at), 1;
            }
        }
    }
    printf("EDGE_WORDS_OK\n");
    return 0;
}
