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

// Matrices of a model, all of which a step goes through: `model` bytes lie between two passes over one.  Up to 256 MB they stay where they are from step to step.
// us, plain / nontemporal, 8 tokens and copies of one matrix in turn, about 190 MB in all and then 1.2 GB: 12288 x 1024 7.3 / 7.8 and 8.3 / 8.2, 16384 x 1024
// 8.3 / 8.7 and 9.6 / 9.1, 8192 x 2048 10.3 / 11.6 and 12.1 / 11.8, 16384 x 2048 13.0 / 15.0 and 17.2 / 15.8.  24 steps of Kimi-K2 layers of 2048 columns, 32 sequences,
// 189 MB 3.19 / 3.58 ms, 314 MB 6.17 / 6.11; of 7168 columns, 2.1 GB, 12 sequences 13.71 / 12.69.
constexpr size_t MODEL = (size_t)256 << 20;
inline int megabytes(size_t bytes) { return (int)((bytes + ((size_t)1 << 20) - 1) >> 20); }
inline bool layers(size_t model) { return model > MODEL; }
// Of larger models of the hybrid decoder the smaller matrices are left to the cache, which the larger ones pass by.  32 steps, all plain / all nontemporal / by the
// matrix: Kagalorn, 8 sequences, 333 MB 9.30 / 9.22 / 9.02 ms, 568 MB 11.01 / 10.48 / 10.37; Rapitar, 265 MB 8.24 / 8.43 / 8.22, 1 GB 13.26 / 12.25 / 12.25.
constexpr size_t MATRIX = (size_t)24 << 20, EXPERTS = (size_t)192 << 20;  // bytes of a matrix, of a layer's experts
inline bool matrix(size_t bytes, size_t model) { return bytes >= MATRIX && layers(model > bytes ? model : bytes); }
inline bool experts(size_t bytes, size_t model) { return bytes >= EXPERTS && layers(model > bytes ? model : bytes); }

}  // namespace kxonce
