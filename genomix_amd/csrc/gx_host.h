// Rules of the graph build that the host decides by, free of HIP so that they
// can be checked without a GPU.
#pragma once

#include <cstddef>
#include <cstdint>

namespace gx {

// A buffer that is filled once and kept.  It counts as filled only after its
// fill returned: one that threw (a failed launch) is run again.
template <class Buf>
struct FilledOnce {
  Buf buf;
  bool filled = false;
  template <class Fill>
  void* get(size_t bytes, Fill&& fill) {
    if (!buf.p) filled = false;
    void* p = buf.ensure(bytes);
    if (!filled) {
      fill(p);
      filled = true;
    }
    return p;
  }
};

// Items (records, nodes) of the fullest key bucket among n whose keys' top
// byte lies in [tlo, thi); a bucket is the keys that share their top `bytes`
// bytes.  top: k-mer occurrences by the key's top byte, or nothing counted
// (all zero): the canonical choice then makes the lowest keys, which the whole
// range holds, twice as full as the mean.  Inside one top byte the buckets
// are taken as even.
inline double fullest_bucket(uint64_t n, int bytes, const uint64_t* top, uint32_t tlo, uint32_t thi) {
  uint64_t sum = 0, most = 0;
  for (uint32_t t = tlo; t < thi; t++) {
    sum += top[t];
    if (top[t] > most) most = top[t];
  }
  double x = (double)n * (sum ? (double)most / (double)sum : 2.0 / 256);
  for (int b = 1; b < bytes; b++) x /= 256;
  return x;
}

// Bytes of a record-sort bucket: two while the fullest bucket stays well
// inside what a block sorts in LDS (16384 one-word, 8192 two-word records; a
// larger bucket goes through the global radix sort).  A third byte costs a
// radix pass (320 M one-word records: 2.7 ms) and 16 M buckets of a few
// records; one-word buckets fuller than 10240 have not been measured.  The
// limit holds for the buckets the range covers: taken from the range's size
// as if it filled all 65536, three passes over 576 M two-word records sent
// 448 M of them through the global sort (build 190.7 ms, now 107.0), four
// over 720 M one-word records 317 M (105.4 ms, now 91.2).
inline int record_bucket_bytes(int words, int key_bytes, uint64_t n, const uint64_t* top, uint32_t tlo, uint32_t thi) {
  if (key_bytes < 2) return 1;
  return key_bytes >= 4 && fullest_bucket(n, 2, top, tlo, thi) > (words == 1 ? 10240 : 8192) ? 3 : 2;
}

// LDS slots of k_nix_build: 32 KB (512 threads), 64 KB (1024).
constexpr int kNixSmall = 8192, kNixLarge = 16384;

// Bytes of a node index bucket: two while the larger LDS table holds the two
// slots per node of a bucket a quarter above the fullest; a larger bucket
// claims its slots in HBM (the indexes of those three passes 23.9 ms, now
// 7.7).
inline int index_bucket_bytes(int key_bytes, uint64_t n, const uint64_t* top, uint32_t tlo, uint32_t thi) {
  if (key_bytes < 2) return 1;
  return key_bytes >= 4 && 2.5 * fullest_bucket(n, 2, top, tlo, thi) > kNixLarge ? 3 : 2;
}

// Nodes one walk from a path's end may claim; a graph with a longer path is
// ranked again as a whole by walks between splitters.  A walk's step takes
// 0.4 us and the splitters 0.1-0.2 ns a node, so a walk stops when it has cost
// about what they will: at most about twice the better of the two.  Merge of
// graphs of short paths and one of 3000, 4000, 7900 and 9000 nodes: 18.6 M
// nodes 9.7, 9.7, 9.7, 9.7 ms under a cap of 1024 and 6.2, 6.6, 8.1, 12.1
// under 4096; 3.7 M nodes 2.4, 2.4, 2.4, 2.4 and 2.0, 2.3, 3.6, 4.4; 0.5 M
// nodes 1.3, 1.3, 1.4, 1.3 and 1.5, 1.8, 3.4, 3.5.
inline uint32_t walk_cap(uint64_t nodes) {
  const uint64_t n = nodes / 4096;
  return n < 1024 ? 1024 : n > 4096 ? 4096 : (uint32_t)n;
}

}  // namespace gx
