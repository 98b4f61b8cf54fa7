// A product in pieces, for the kernels that sum whole rows of it.
#pragma once

#include "common.h"

namespace fi {

// parts of `total` units of `unit` stages over `n` workgroups
struct Cut {
  int per, rem, unit;
  FI_DEV Cut(int total, int n, int unit)
      : per(total / n), rem(total % n), unit(unit) {}
  FI_DEV int start(int i) const { return (i * per + min(i, rem)) * unit; }
  // the part that holds a stage (unit 1)
  FI_DEV int holder(int stage) const {
    const int wide = rem * (per + 1);
    return stage < wide ? stage / (per + 1) : rem + (stage - wide) / per;
  }
};

// Tiles of tn columns in sk stages each, cut into parts of which none is more
// than a tile long: the first piece of a tile is its part's start of one (its
// second place), the others are ends (the first). A piece has `rows` rows, one
// after another or (columns) 16 columns of all rows after one another.
struct PieceRows {
  const void* pieces;
  const u16* bias;             // [N] or nullptr
  int tn, sk, tiles, parts, rows;
  bool columns;
};

// the row of x that a workgroup has: two rows that share the lines of pieces go
// to the same XCD, whose turn comes every eight workgroups
FI_DEV int piece_row(bool columns) {
  const int xcd = blockIdx.x % 8, turn = blockIdx.x / 8;
  return columns ? (turn / 2 * 8 + xcd) * 2 + turn % 2
                 : static_cast<int>(blockIdx.x);
}

// Where a thread's columns n on of row m lie (as many as share 16): requests
// of pieces from `next` on, zeros and no fetch beyond the last.
struct PieceReader {
  BufferRsrc from;
  u32 at, piece_b;
  int first, last, next;
  FI_DEV PieceReader(const PieceRows& p, int m, int n) {
    const int tile = n / p.tn, of = n - tile * p.tn;
    const Cut cut(p.tiles * p.sk, p.parts, 1);
    first = cut.holder(tile * p.sk);
    last = cut.holder(tile * p.sk + p.sk - 1);
    next = first;
    piece_b = p.tn * p.rows * 4;
    from = buffer_of(p.pieces, p.parts * 2 * piece_b);
    at = p.columns ? (of / 16 * p.rows + m) * 64 + of % 16 * 4
                   : (m * p.tn + of) * 4;
  }
  // four columns of piece next + i, `more` bytes on
  FI_DEV u32x4 get(int i, u32 more) const {
    const int q = next + i;
    return buffer_load16(
        from, q > last ? ~0u : at + more + (q * 2 + (q == first)) * piece_b, 0);
  }
};

}  // namespace fi
