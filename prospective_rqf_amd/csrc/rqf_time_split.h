// rqf_time_split.h -- sequences of the (B,T,F) scans cut into chunks.
//
// A block of those scans owns 16 filters of one batch element and walks its sequence in
// passes, so few sequences leave most of the 256 CUs idle: one recording of 128
// filters makes 8 blocks.  There a sequence is cut into chunks of whole passes, a block
// each, in two launches: the first scans every chunk from a zero state for its end
// state only (its pair at its start, for an adjoint), the second forms each chunk's
// entry from the chunks before (after) it, in fp64 with the power of the chunk's
// length, and runs the chunk.  An unstable filter's power may overflow (|c1| = 1.2 at 4096
// steps), so there the entry starts from the first state that is not zero: silence before a
// chunk stays silence, as it does in a whole sequence.  The input is read twice, so large
// grids, which memory bounds, run whole sequences.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace rqf {

// What a launch does: whole sequences, or, of a time split, the chunks' end states or
// the chunks themselves.
enum Phase { kWhole, kTotals, kChunks };
struct Split {
  int64_t chunks;  // per sequence
  int64_t steps;   // per chunk: whole passes (the last chunk may be shorter)
};

// Up to `most` sequences (`most_long` of twelve passes and more) of at least `least`
// passes: as many chunks as fill the CUs.
inline Split time_split(int64_t sequences, int64_t T, int64_t pass, int64_t least, int64_t most,
                        int64_t most_long) {
  const int64_t passes = (T + pass - 1) / pass;
  Split s{1, T};
  if (sequences < 1 || passes < least || sequences > (passes >= 12 ? most_long : most)) return s;
  const int64_t want = std::min(passes, std::max<int64_t>(2, 256 / sequences));
  const int64_t per = (passes + want - 1) / want;
  s.steps = per * pass;
  s.chunks = (passes + per - 1) / per;
  return s;
}

}  // namespace rqf
