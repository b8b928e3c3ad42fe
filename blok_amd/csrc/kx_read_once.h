// kx_read_once.h -- what is copied nontemporally (kx_copy16_to_lds_once of kx_lds_copy.h): host code on sizes alone, in plain C++.  Nontemporal copies of whole
// lines arrive faster from HBM, but leave nothing in the memory-side cache of 256 MB for the next pass, and a launch with little to read is done before
// their rate counts.
#pragma once
#include <stddef.h>

namespace kxonce {

// A cache of latent rows that `seqs` sequences attend once, `bytes` of it in all.  us, plain / nontemporal, the same cache again and caches of 1.4 GB in turn:
// 8 x 4096 (36 MB) 29.4 / 32.3 and 30.0 / 32.2, 1 x 32768 35.4 / 38.7 and 36.6 / 39.0, 1 x 131072 (144 MB) 63.6 / 66.1 and 65.0 / 66.4, 16 x 8192 47.8 / 48.7 and
// 49.5 / 49.0; 16 x 14000 (246 MB) 69.7 / 67.9 and 72.1 / 68.5, 1 x 262144 (288 MB) 89.4 / 88.5 and 89.3 / 89.3, 16 x 32768 135.9 / 129.4 and 135.2 / 128.2.
constexpr size_t LATENT = (size_t)240 << 20;
inline bool latent(size_t bytes) { return bytes >= LATENT; }

}  // namespace kxonce
