// Device kd-tree build: the records one level of the breadth-first build
// works on.  The build makes the same decisions as the host builder
// (host/kdtree.cpp) with the same floating-point operations, so the tree it
// produces is identical, entry for entry.
#pragma once

#include "re_math.hpp"

namespace re {
namespace kdb {

// A triangle reference inside a node: its id and the box of the part of the
// triangle inside the node.
struct Ref {
  int32_t prim;
  float lo[3], hi[3];
};

// Node modes of a level: a leaf by size or depth, every candidate plane
// (at most kExactMax references), binned by one wave (at most kWaveBinMax),
// binned by many blocks.
enum : int32_t { kModeLeaf = 0, kModeExact = 1, kModeBinned = 2, kModeBig = 3 };

// An active node of the current level.
struct LNode {
  float lo[3], hi[3];
  int64_t rbegin;    // first reference in the level's reference array
  int32_t n;         // references
  int32_t depth;     // root = 1
  int32_t gid;       // breadth-first node id
  int32_t mode;      // kMode*
  int32_t axis;      // chosen split axis, -1 none
  float pos;         // chosen split position
  int32_t nl, nr;    // counts the split was costed with
  int32_t cl, cr;    // references that actually go below / above (after clipping)
  int32_t split;     // 1 if the node becomes an inner node
  int32_t child;     // index of its below child in the next level (above = child + 1)
  int64_t crbegin;   // first reference of its below child in the next level's array
  int64_t pool;      // leaves: first slot in the leaf-reference pool
};

// A node of the finished tree, in breadth-first order.
struct GNode {
  float lo[3], hi[3];
  int32_t axis;      // -1 for a leaf
  float split;
  int32_t child0, child1;
  int32_t depth;
  int32_t pool_n;    // leaves: references
  int64_t pool;      // leaves: first slot in the leaf-reference pool
};

struct Params {
  int32_t max_leaf, max_depth, n_bins, clip;
  float ct, ci, eb;
};

constexpr int kExactMax = 64;  // nodes with at most this many references test every candidate plane
constexpr int kMaxBins = 64;
// References per block of the many-block binning, and the most that one wave
// bins by itself.  Equal, so that a chunk's references belong to at most two
// big nodes (its first and its last) and each chunk index is at most one big
// node's rbegin / kBinChunk, which numbers the histograms.
constexpr int kBinChunk = 1024;
constexpr int kWaveBinMax = kBinChunk;

RE_HD int32_t mode_of(int32_t n, int32_t depth, const Params& P) {
  if (n <= P.max_leaf || depth >= P.max_depth) return kModeLeaf;
  return n <= kExactMax ? kModeExact : (n <= kWaveBinMax ? kModeBinned : kModeBig);
}

// What a node adds to the next level and to the leaf pool, scanned together:
// next-level references, leaf-pool references, next-level nodes; and, in
// `last`, the largest leaf in the low 31 bits, with bit 31 set when a
// next-level node is to be binned by bin_count_kernel (their maximum and or).
// The references are summed in 64 bits: a reference that straddles a plane
// counts twice, so a level of 2^31 - 1 may ask for twice as many.
struct Adds {
  int64_t refs, leaf;
  int32_t kids;
  uint32_t last;
};
constexpr uint32_t kBigBit = 0x80000000u;
struct AddsSum {
  RE_HD Adds operator()(const Adds& a, const Adds& b) const {
    const uint32_t m = a.last & ~kBigBit, n = b.last & ~kBigBit;
    return Adds{a.refs + b.refs, a.leaf + b.leaf, a.kids + b.kids, ((a.last | b.last) & kBigBit) | (m > n ? m : n)};
  }
};
// Of a node whose split is decided.
RE_HD Adds node_adds(const LNode& nd, const Params& P) {
  if (!nd.split) return Adds{0, nd.n, 0, (uint32_t)nd.n};
  const bool big = mode_of(nd.cl, nd.depth + 1, P) == kModeBig || mode_of(nd.cr, nd.depth + 1, P) == kModeBig;
  return Adds{(int64_t)nd.cl + nd.cr, 0, 2, big ? kBigBit : 0u};
}

// Whether the level after one with `nodes` tree nodes up to its end and
// `records` leaf-pool references up to its end can be built: node indices have
// 30 bits, references and triangle records are indexed with 31.
inline bool level_fits(int64_t nodes, int64_t records, const Adds& total) {
  return nodes + total.kids <= (int64_t)0x3fffffff && total.refs <= (int64_t)0x7fffffff &&
         records + total.leaf <= (int64_t)0x7fffffff;
}

// Device and pinned host memory that a context keeps between its device
// builds: one chunk of what the last build took, at most kKeepBytes, and the
// totals of a level.  A build that needs more takes and frees the rest itself;
// an allocation of the context that finds the device full frees the chunk.
constexpr size_t kKeepBytes = (size_t)256 << 20;
struct Workspace {
  char* chunk = nullptr;
  size_t bytes = 0;
  Adds* totals = nullptr;  // pinned
};

}  // namespace kdb
}  // namespace re
