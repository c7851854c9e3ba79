// Tile shapes of the plain multisplit, shared by host code and kernels.
//
// One workgroup of 256 threads (4 waves of 64) owns one tile of 256*K keys.
// K keys per thread are held in registers in blocked order; the local stable
// reorder ranks digits of at most LEVEL_BITS bits per LDS pass.  The prescan
// uses the same tile so that both kernels agree on the histogram matrix.
#pragma once

#include <stdint.h>

namespace gms {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

// Keys per thread, by log2(bucket count), key-value-ness and input size
// (measured on MI355X).  24 everywhere, except for inputs of at least
// kLongTileMin keys where longer tiles -- longer per-bucket output runs --
// measured faster: 64- and 256-bucket key-value (28: at 2^27 pairs the
// 256-bucket call takes 0.564 ms against 0.571 at 24, 0.576 at 20, 0.586 at
// 32; the 64-bucket one 0.515 against 0.523 at 24 and 0.532 at 32), 512 and
// 1024 buckets key-value (36, the longest tile that keeps two workgroups per
// CU: 1024 buckets 0.820 ms against 0.939 at 24, 0.882 at 28, 0.901 at 32)
// and key-only: 128 and 256 buckets 56 (256 buckets 0.379 ms against 0.388
// at 48 and 0.394 at 40), 512 and 1024 buckets 48 (at 56 a 1024-bucket
// workgroup no longer fits twice in a CU: 0.705 against 0.521 ms).  Below that
// size the longer tiles leave too few tiles per CU, except for 1024-bucket
// key-value, whose long tiles pay from 2^24 keys (0.116 ms against 0.132 at
// 2^24, 0.229 against 0.266 at 2^25; 512 buckets there are within 2 % either
// way, 256 buckets at 2^25 0.161 against 0.156).
constexpr uint32_t kLongTileMin = 1u << 26;
constexpr uint32_t long_tile_min(int log_b, bool kv) {
    return kv && log_b >= 10 ? kLongTileMin / 4 : kLongTileMin;
}
// The prescan streams its key loads past the caches from this many keys;
// smaller inputs are re-read by the postscan while still in the last-level
// cache.
constexpr uint32_t kStreamLoadMin = 1u << 26;

constexpr int tune_items(int log_b, bool kv, bool large) {
    if (!large) return 24;
    if (!kv) return log_b >= 9 ? 48 : (log_b >= 7 ? 56 : 24);
    return log_b >= 9 ? 36 : (log_b == 6 || log_b == 8 ? 28 : 24);
}

// Widest digit ranked in one LDS pass (2^w x 256 u32 counters): 1..4 bits in
// one pass; 5 bits as 3+2, 6 as 3+3, 7 as 4+3, 8 as 4+4.
constexpr int tune_level_bits(int log_b) {
    return log_b <= 4 ? (log_b < 1 ? 1 : log_b) : (log_b <= 6 ? 3 : 4);
}

// Digit counters of a ranking pass with D digits: logically D x 256 u32,
// digit-major (word d*256 + t), and each thread scans the D consecutive
// logical words [t*D, t*D+D) -- its "row".  Rows are padded in LDS to
// D + cnt_pad(D) words so that the rows of 8 consecutive lanes start on
// different banks (row stride / 4 odd for 16-byte accesses; stride 3 for
// D = 2): unpadded, the 16-byte row reads of D = 16 are 16-way bank conflicts.
constexpr int cnt_pad(int D) { return D % 4 == 0 ? (((D / 4) & 1) ? 0 : 4) : (D == 2 ? 1 : 0); }
constexpr int cnt_row(int D) { return D + cnt_pad(D); }
// LDS words of the counters of passes of up to level_bits bits.
constexpr uint32_t cnt_words(int level_bits) { return (uint32_t)cnt_row(1 << level_bits) * kThreads; }

// Whether a key-value postscan keeps its digit counters inside the value
// staging area (fewer LDS bytes, more resident workgroups).  Not for 128/256
// buckets with short tiles: three resident workgroups per CU then keep more
// partially written output lines open than L2 merges well, which measured
// 35 % slower than two.
constexpr bool tune_alias(int log_b, int items, bool kv, int level_bits) {
    return kv && cnt_row(1 << level_bits) <= items && !(log_b >= 7 && items < 28);
}

// Keys from which a class always loads a postscan tile through LDS and ranks it
// with register counters (ms_postscan_reg_kernel) instead of blocked loads and
// LDS counters; 0: no such size.  On MI355X, whole call, LDS counters against
// registers (us):
//   key-value  2 buckets 10M 48.7 / 47.0, 13M 60.3 / 55.9, 2^24 73.1 / 68.9, 2^25
//              134 / 132, 2^26 240 / 238; 16 buckets 13M 66.6 / 62.0, 2^25 139 / 134,
//              2^26 257 / 238, 90M 347 / 336; 32 buckets 20M 86.7 / 90.6, 2^26 258 / 243
//   key-only   2 buckets 10M 29.1 / 27.5, 13M 35.7 / 32.6, 2^25 85.2 / 84.2, 2^26 143 /
//              140; 8 buckets 13M 36.6 / 34.1, 2^26 144 / 137
// At 3M to 8M keys both are the same or the LDS counters up to 5 % faster.  With
// more buckets it depends on the identifier and on what wrote the input: 2^25 pairs
// in 256 buckets 157 / 149 by range but 153 / 154 by division, passes of an 8-bit
// sort of 2^25 keys 98 / 107, of 2^26 pairs 277 / 413.
constexpr uint32_t reg_rank_from(int log_b, bool kv) {
    return log_b <= (kv ? 4 : 3) ? 9u << 20 : (kv && log_b == 5 ? kLongTileMin : 0u);
}

// Keys below which it does so in a call that wants the bucket starts: this form
// writes them, the other leaves them to a launch of about 4 us and the gap before
// it.  Range / division / digit identifier, as above:
//   key-only   16 buckets 2.2M 19.9 / 18.2, 21.8 / 20.1, 20.8 / 18.7; 64 buckets 6M
//              27.2 / 23.5, 29.5 / 26.1, 27.4 / 24.9, at 9.5M 35.9 / 32.6, 39.2 / 37.5,
//              36.5 / 35.8, at 24M by digit 63 / 68; 256 buckets 4M 27.8 / 23.3, 29.6 /
//              25.9, 28.4 / 25.0
//   key-value  2 buckets 4M 24.9 / 18.9 by range, 8M 32.8 / 31.2; 16 buckets 6M 35.6 /
//              34.2, 36.0 / 35.1, 35.5 / 34.0; 64 buckets 6M 34.5 / 32.7, 36.0 / 34.9,
//              34.7 / 33.0, at 9.5M 44.1 / 45.3, 46.8 / 48.8, 45.1 / 45.4; 256 buckets 6M
//              42.4 / 37.0, 43.9 / 38.9, 42.9 / 36.6
constexpr uint32_t reg_rank_starts_below(int log_b, bool kv) {
    return log_b > 8 ? 0u : (kv && log_b > 3 ? 7u << 20 : 9u << 20);
}

constexpr bool reg_rank(int log_b, bool kv, uint32_t n, bool starts) {
    const uint32_t from = reg_rank_from(log_b, kv);
    return (from && n >= from) || (starts && n < reg_rank_starts_below(log_b, kv));
}

// Bucket counts up to this run in one prescan/scan/postscan pass (three LDS
// ranking passes of at most 4 bits above 256); more take LSD passes over
// 8-bit digits of the bucket id.
constexpr uint32_t kSinglePassBuckets = 1024;

// Keys per tile for an input of n keys.  The shortest tile, used to size the
// histogram matrix for every n up to a capacity, is tile_keys(log_b, kv, 0).
constexpr uint32_t tile_keys(int log_b, bool kv, uint32_t n) {
    return (uint32_t)(kThreads * tune_items(log_b, kv, n >= long_tile_min(log_b, kv)));
}

inline int ceil_log2_u32(uint32_t x) {
    int l = 0;
    while ((1u << l) < x && l < 31) ++l;
    return l;
}

}  // namespace gms
