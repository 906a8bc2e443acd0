// chunk_rule.h -- how the planes of 3D ideal-gas blocks are divided among workgroups where
// no timing has been done.  Free of HIP, so that a host program can check it.
#pragma once
#include <algorithm>

namespace e4 {

// Chunks of a launch over `cols` tile columns of `nk` planes where nothing has been
// tuned: 2048 workgroups (8 a compute unit).  In FP64, where that leaves fewer than
// eight planes to a chunk, one round of what the chip holds (768 workgroups, three a
// compute unit; 650 come close enough) if that is the shorter by the model: a chunk
// takes its planes and 1.5 for its ends, and the last one, alone, `tail` of that again
// (0: the first choice always, as in mixed precision).
// A step of ausmdv, many or few: 128^3 (4 planes, 11) 269, 262 us; 96^3 (2, 5) 139,
// 133; 160 x 160 x 20 (1, 3) 100, 93; 48 x 56 x 500 (4, 10) 261, 255; joined blocks,
// 3 of 90 x 70 x 33 (2, 4) 205, 155; 16 of 64 x 64 x 40 (5, 14) 425, 364; many is the
// better, and taken, for 300 x 300 x 40 (7, 20) 476, 495 and 400 x 380 x 12 (3, 12)
// 257, 291.  The reference arithmetic gains less: 3 of 90 x 70 x 33 258, 212, but 128^3
// 404, 422 and 8 of 48 x 56 x 50 (3, 9) 397, 419 (many taken; few for 48 x 56 x 500, 400,
// 411, all the same).
constexpr double CHUNK_TAIL_FP64 = 0.4, CHUNK_TAIL_EXACT = 0.6;
inline long untuned_chunks(long cols, long nk, double tail)
{
    const long many = (2048 + cols - 1) / cols, few = std::max(1L, 768 / cols);
    if (tail == 0.0 || (nk + many - 1) / many >= 8) return many;
    auto height = [&](long chunks) { return (nk + chunks - 1) / chunks; };
    auto groups = [&](long chunks) { return cols * ((nk + height(chunks) - 1) / height(chunks)); };
    auto time = [&](long chunks) {
        return ((double)height(chunks) + 1.5) * ((double)((groups(chunks) + 767) / 768) + tail);
    };
    return (groups(few) >= 650 && time(few) < time(many)) ? few : many;
}

} // namespace e4
