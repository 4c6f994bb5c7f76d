// Which tiles of keys a workgroup of chunk_attention.hip walks and which keys of gathered rows it may read: plain integers, so
// that a host program checks the very arithmetic that the kernels use.
#pragma once

namespace mxs {

constexpr int kWalkPage = 16;  // keys that a stager takes or leaves together

// first key of a sequence's gathered rows: the page of its first query's oldest visible key
constexpr int first_gathered(int past, int window) {
  return window > 0 && past - window + 1 > 0 ? (past - window + 1) / kWalkPage * kWalkPage : 0;
}

// Tiles of kt keys: nA of the kept first tokens below the window, then from the window's first, t0, to the diagonal's.
struct ChunkWalk {
  int t0, nA, ntile, kt;
  constexpr int start(int it) const { return (it < nA ? it : t0 + it - nA) * kt; }
};
// first, last: positions of the workgroup's first and last query
constexpr ChunkWalk chunk_walk(int first, int last, int window, int keep, int kt) {
  const int t0 = window > 0 && first - window + 1 > 0 ? (first - window + 1) / kt : 0;
  const int kept = window > 0 ? (keep + kt - 1) / kt : 0, nA = kept < t0 ? kept : t0;
  return ChunkWalk{t0, nA, nA + last / kt - t0 + 1, kt};
}

// The last key of the page from key0 on that may be read of gathered rows, counted from key0 (negative: none of them).  A tile
// can begin a page or more before the rows do: those keys are outside every query's window.
constexpr int gathered_left(int key0, int low, int kmax) { return key0 < low ? -1 : kmax - key0; }

}  // namespace mxs
