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

// Choices between forms of the same results.  The tests of the CPU emulation build
// force them (gms_emu_force; short_calls only off), as its sizes stay below most limits;
// the GPU library always goes by the rule.
enum class Form { short_calls, reg_postscan, range_table, batch_lds };
#ifdef GMS_HOST_EMULATION
extern int emu_forced[4];  // per Form: -1 by the rule, 0 or 1
inline bool form(Form f, bool rule) {
    const int v = emu_forced[(int)f];
    return v < 0 ? rule : v != 0;
}
#else
constexpr bool form(Form, bool rule) { return rule; }
#endif

// Few buckets: the classes whose postscan loads its tile through LDS and ranks it with
// register counters (ms_postscan_reg_kernel), instead of blocked loads and LDS
// counters, whenever the call wants the bucket starts, and from some size on without.
constexpr bool reg_rank_few(int log_b, bool kv) { return log_b <= (kv ? 4 : 3); }

// Keys from which a class takes it in every call; 0: no such size.  On MI355X, whole
// call without starts, registers / LDS counters, the worst of uniform, sorted and
// one-key-in-ten keys and of range, division and digit identifiers, then the best:
//   key-value  2 buckets 9.5M 1.00 .98, 2^24 .96 .95, 50M 1.02 .99, 2^26 .96 .94; 8 buckets
//              9.5M 1.04 1.00, 13.5M 1.03 1.00, 2^24 .98 .94, 2^25 .98 .94, 2^26 .96 .89; 16
//              buckets 9.5M 1.08 1.04, 15M 1.05 1.00, 20M 1.05 .98, 2^25 1.00 .96, 2^26 .93 .89
//   key-only   2 buckets 13.5M 1.03 .97, 2^25 1.00 .98, 2^26 .85 .82; 4 buckets 9.5M 1.06
//              1.02, 13.5M 1.07 .99, 20M 1.04 .99, 2^26 .88 .84; 8 buckets 13.5M 1.06 .99, 50M
//              1.04 1.00, 2^26 .94 .87
// With 32 buckets of pairs at 2^26 uniform keys gain (258 / 243 us) what sorted ones
// lose (256 / 281); with more it depends on the identifier and on what wrote the
// input: 2^25 pairs in 256 buckets 157 / 149 by range but 153 / 154 by division,
// passes of an 8-bit sort of 2^25 keys 98 / 107, of 2^26 pairs 277 / 413.
constexpr uint32_t reg_rank_from(int log_b, bool kv) {
    if (!reg_rank_few(log_b, kv)) return 0u;
    return kv ? (log_b <= 3 ? 1u << 24 : 1u << 25) : 1u << 26;
}

// Keys below which a class takes it in a call that wants the bucket starts: this form
// writes them, the other leaves them to a launch of about 4 us and the gap before
// it.  As above (the other form with its launch):
//   key-value  2 buckets 2.3M .87 .84, 9.5M .96 .94, 2^25 .97 .96; 16 buckets 4.2M 1.01 .99, 6.3M
//              1.04 1.00, 9.5M 1.04 .99, 2^24 .98 .94; 64 buckets 4.2M .98 .96, 6.3M 1.03 .98, 8.5M
//              1.02 .97; 256 buckets 4.2M .88 .83, 6.3M 1.00 .93; at 9.5M 64 buckets 44.1 / 45.3 us
//              by range, 46.8 / 48.8 by division
//   key-only   2 buckets 6.3M .92 .87; 8 buckets 6.3M .95 .92, 50M 1.01 .97; 64 buckets 6.3M .98
//              .93, 8.5M .97 .89, at 24M by digit 63 / 68 us; 256 buckets 4.2M .88 .84, 8.5M .96 .90
constexpr uint32_t reg_rank_starts_below(int log_b, bool kv) {
    if (reg_rank_few(log_b, kv)) return 0xFFFFFFFFu;
    return log_b > 8 ? 0u : (kv ? 7u << 20 : 9u << 20);
}

// The form of one call; `pass`: of one digit pass of a sort or of a multisplit into
// many buckets.  Those read what a kernel has just written: pairs gain only where the
// loads stream (4-bit sort of 2^26 2030 / 1817 us, 5-bit 1803 / 1664, of 2^25 1021 / 988;
// but 2^25 sorted pairs into 500,000 buckets, last pass 3 bits, 478 / 490), key-only
// ones lose (2048 buckets, last pass 3 bits: 2^25 keys 199 / 203, 2^26 368 / 377).
constexpr bool reg_rank(int log_b, bool kv, uint32_t n, bool starts, bool pass) {
    const uint32_t from = reg_rank_from(log_b, kv);
    if (pass) return kv && from && n >= kStreamLoadMin;
    return (from && n >= from) || (starts && n < reg_rank_starts_below(log_b, kv));
}

// Bucket counts up to this run in one prescan/scan/postscan pass (three LDS
// ranking passes of at most 4 bits above 256); more take LSD passes over
// digits of the bucket id (large_passes).
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
