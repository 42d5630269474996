// Host-side helpers shared by libmpm_hip and its host check library (plain
// C++, no HIP types).
#pragma once
#include <algorithm>
#include <cstddef>

namespace mpm {

// Bytes per part when a host copy of `bytes` bytes is split over `nt`
// threads: ceil(bytes / nt) rounded up to a multiple of 64, so parts start
// on cache-line boundaries and nt of them cover every byte.  Part t spans
// [min(bytes, t * part), t + 1 == nt ? bytes : min(bytes, (t + 1) * part)).
inline size_t readback_part_bytes(size_t bytes, unsigned nt) {
  const size_t per = (bytes + nt - 1) / nt;
  return (per + 63) / 64 * 64;
}

// A copy of `total` bytes to the caller through pinned memory: pieces of up to
// 1 MiB, two in flight per host thread, up to four threads; `ring` bytes of
// pinned memory hold the pieces in flight.
struct XferPlan {
  unsigned threads;
  size_t piece, ring;
};
constexpr size_t XFER_PIECE = size_t(1) << 20, XFER_PIECE_MIN = size_t(1) << 17;
constexpr unsigned XFER_THREADS = 4;
inline XferPlan xfer_plan(size_t total) {
  XferPlan p;
  p.threads = (unsigned)std::min<size_t>(XFER_THREADS, std::max<size_t>(1, total / (2 * XFER_PIECE)));
  p.piece = std::min(XFER_PIECE, std::max(XFER_PIECE_MIN, readback_part_bytes(total, 4 * p.threads)));
  p.piece = std::min(p.piece, std::max<size_t>(64, readback_part_bytes(total, 1)));
  p.ring = 2 * p.threads * p.piece;
  return p;
}

// The pieces of `count` parts of the given bytes, each piece inside one part:
// their number, and piece i (`at`: the bytes of the pieces before it).  Worked
// out per piece, not listed: a read through the C interface allocates nothing
// on the heap but its threads, whose failure it survives.
struct XferPiece {
  int part;
  size_t offset, bytes, at;
};
inline size_t xfer_pieces(const size_t* bytes, int count, size_t piece) {
  size_t n = 0;
  for (int k = 0; k < count; ++k) n += (bytes[k] + piece - 1) / piece;
  return n;
}
inline XferPiece xfer_piece(const size_t* bytes, int count, size_t piece, size_t i) {
  size_t at = 0;
  for (int k = 0; k < count; ++k) {
    const size_t n = (bytes[k] + piece - 1) / piece;
    if (i < n) return {k, i * piece, std::min(piece, bytes[k] - i * piece), at + i * piece};
    i -= n;
    at += bytes[k];
  }
  return {count, 0, 0, at};
}

}  // namespace mpm
