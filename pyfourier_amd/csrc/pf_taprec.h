// Shape of a sample's tap record: 4 header words (first tap z, y, x, frame),
// then the weights of the three axes, padded to whole 16-byte pieces.  2 pieces
// (width-1 plans, 1-D up to W = 2) to 7 (3-D, W = 8).  The records are
// allocated back to back with nothing behind the last one.
#pragma once

constexpr int PF_REC_HEAD = 4;

// words of a record for kernel widths wz, wy, wx (1 on axes a plan does not have)
constexpr int pf_rec_words(int wz, int wy, int wx) { return (PF_REC_HEAD + wz + wy + wx + 3) & ~3; }

// the piece a lane copies when a fixed number of lanes stages a record of rec4
// pieces: its own, or piece 0 again past the record's end
constexpr int pf_rec_piece(int c, int rec4) { return c < rec4 ? c : 0; }
