// Which kernels the stages of a job run on: plain arithmetic on its sizes, so that a host compiler can take it as well.
#pragma once

#include <limits.h>

#include <algorithm>

namespace {

constexpr int BLOCK = 256;            // lanes of the block-per-row kernels and counting workgroups
#ifndef MOE_A2A_ROWS
#define MOE_A2A_ROWS 4
#endif
constexpr int ROWS = MOE_A2A_ROWS;    // rows (= waves) per workgroup of a ranked row move

bool items_fit(long long rows, int chunks) { return rows * chunks <= INT_MAX / 2; }

// ---------------------------------------------------------------- streams beyond the caches
//
// Streams that do not stay in L2 (32 MB) on their way from one stage to the next, nor in the 256 MB behind it, are bound by what memory
// takes at a time. Rows of them are read with nontemporal loads, which push nothing of what is being written out of the caches, and
// in small pieces along the stream, so that fewer places of it are open at once: a plain copy of 470 MB runs at 5.4 TB/s with 14 vectors per
// lane, 5.7 with four, 6.1 with one, and 6.5 with nontemporal loads and one; of 28 MB, at 6.1 to 6.4 with any of them.
// us of a graph of stages 1, 2, expert, 3 and 4, plain / nontemporal loads in one stage (8 entries per token, 14 KB but where said):
//  - expert, four vectors per lane / two and nontemporal: 2.3 MB 17.8 / 17.8, 15 MB 29.9 / 30.0, 29 MB 49.5 / 47.0, 46 MB 78.8 / 74.3, 134
//    MB of 4 KB 214 / 198, 235 MB 377 / 348, 470 MB 720 / 716 (its rows then fill the cache behind L2 for stage 3 to push out: below)
//  - stage 3: 15 MB 29.7 / 30.2, 29 MB 47.2 / 47.0, 46 MB 72.1 / 71.0, 69 MB 99.8 / 98.3, 134 MB of 4 KB 193.9 / 189.0, 235 MB 340 / 329.
//    That is one set of buffers again and again, most of which the caches keep. Whole calls of a rank on six sets in turn, and by themselves between
//    fills of 700 MB: 29 MB 53.1 / 50.8, 64.3 / 61.4, compact and skewed 53.0 / 51.7, 59.7 / 57.3, 24 MB of 5.8 KB 54.7 / 53.3, 65.1 / 62.3, 31 MB of 4
//    KB 66.9 / 65.4, 78.5 / 75.3, 47 MB of 2 KB 103.1 / 100.4, 112.7 / 105.2, 45 MB 78.2 / 74.8, 94.2 / 91.7; on one set 46.3 / 46.3, 55.2 / 55.3,
//    48.0 / 47.9, 59.2 / 59.5, 96.5 / 96.7, 68.9 / 69.1. What loses is a stage 3 whose rows no expert has written since it last read them, which the
//    cache behind L2 then still holds: the graph of stages 1, 2, 3 and 4 alone, 28 MB 35.4 / 38.4, 43 MB 55.3 / 58.3, 54 MB 69.5 / 69.4. A job has an
//    expert there. (Loads of another scope, sc0 and sc1, take the same as without, with and without nt.)
//  - stage 2, four vectors per lane / two / two and nontemporal: 29 MB 47.2 / 46.6 / 47.2, 46 MB - / 74.2 / 72.0, 69 MB 102.2 / 102.1 /
//    101.1, 134 MB of 8 KB 196.0 / 194.2 / 192.7, 275 MB 395 / 393 / 378, 470 MB 682 / 676 / 663; of rows of up to 4 KB one vector per lane:
//    134 MB of 4 KB, two / one 195.2 / 193.5, 67 MB of 2 KB 128.0 / 123.9, 16 MB of 2 KB 48.8 / 47.8.
constexpr long long EXPERT_PAST_BYTES = 24ll << 20, RECV_PAST_BYTES = 40ll << 20;

// The expert's results go past the cache behind L2 only where it could hold little of them, else through it (Store):
// 134 MB 198 / 205, 268 MB 497 / 510, 336 MB 708 / 685 and, the other stages at their best, 658 / 664; 470 MB 716 / 682 and 649 / 637.
constexpr long long EXPERT_STREAM_BYTES = 384ll << 20;

// Vectors per lane of the movers of a planned stage 2: one for rows of up to 4 KB, and for those of more than 8 KB that the cache behind L2 holds
// none of; us of stages 1, 2, 3 and 4, and of a whole step, two / one: 14 KB 185 MB 216.5 / 219.1, 318.3 / 319.4, 240 MB 279.6 / 285.7, 411.6 / 413.3,
// 294 MB 366.9 / 362.1, 531.8 / 533.1, 348 MB 435.8 / 425.8, 634.8 / 638.2, 446 MB 549.1 / 538.6, 803.5 / 802.6; 10 KB 319 MB 389.5 / 385.9, 510.6 /
// 511.9; 8 KB 312 MB 389.6 / 390.8, 513.3 / 515.8; 6 KB 328 MB 429.8 / 427.1, 557.4 / 559.7.
int planned_recv_vecs(long long bytes, int row_vecs) { return row_vecs > BLOCK && (row_vecs <= 2 * BLOCK || bytes < 288ll << 20) ? 2 : 1; }

// Vectors per lane of a planned stage 3: four (a 256-vector piece per wave) made a whole step 0.5 us shorter at 2048 rows of 14 KB than the
// 14 of the scan path; 2, 6 and 8 were no better than 14. Long rows beyond the cache take eight: 470 MB 660 / 654 us as above, 336 MB of 10 KB
// 670 / 665, 275 MB 378 / 376, but 235 MB 329 / 331 and, a whole row in eight, 268 MB of 8 KB 485 / 497.
int planned_send_vecs(long long bytes, int row_vecs) { return bytes >= 256ll << 20 && row_vecs > 2 * BLOCK ? 8 : 4; }

// ---------------------------------------------------------------- stage 1

constexpr int FANOUT_MIN_K = 4;
constexpr int FEW_ENTRIES = 64 * 16;
constexpr int FEW_MAX_K = 64;            // a lane of the wave for each
constexpr int BLOCK_RANKS = 8;
constexpr int BLOCK_MAX_ENTRIES = 255 * BLOCK;  // keys that 256 lanes count in bytes
constexpr int LONG_BLOCK = 1024;                // lanes of dispatch_long_kernel
constexpr int LONG_ENTRIES = 5120, LONG_MAX_ENTRIES = 255 * LONG_BLOCK;

enum SendWay {
  SEND_BY_ENTRY,     // dispatch_send_kernel
  SEND_FEW,          // dispatch_few_kernel
  SEND_BLOCK,        // dispatch_block_kernel
  SEND_FANOUT,       // dispatch_fanout_kernel
  SEND_FANOUT_WIDE   // dispatch_fanout_wide_kernel: rows of more than one 256-lane chunk
};

// Keys per lane of a wave that holds all of a stream: the smallest of the numbers that there are kernels for.
// (12 beside 16 is worth 4 to 7 %, us with 12 / 16: stage 1, 65 tokens of 14 KB, 8 per token 4.06 / 4.22, 190 of 1 KB, 4 each 3.06 / 3.26; stage 2, 530
// rows of 5.8 KB 3.51 / 3.70, 600 of 512 bytes 2.86 / 3.08.)
int few_keys(long long entries) {
  for (const int keys : {2, 4, 8, 12})
    if (entries <= 64 * keys) return keys;
  return 16;
}

// `row_vecs`: vectors of 16 bytes in a row, or its elements where those cannot be used (vec16).
//
// With one entry per token a wave per entry only scans what lies ahead in the stream, where the other kernel's passes take 2048 keys.
// Behind the first pass that is ahead up to 3000 entries, before its end on rows of 4 to 10 KB (shorter ones leave it idle, and of longer
// ones the scan is little), on elements up to 2700. us, a wave per entry / four tokens in a pass: 1967 tokens of 5.8 KB 5.5 / 6.2, 2303 of 4.9
// KB 6.6 / 7.6, 2440 of 768 bytes 5.3 / 5.6, 2862 of 3.7 KB 6.8 / 7.3, 2067 of 1452 elements 7.6 / 8.5; but 1823 of 1.4 KB 4.5 / 4.2, 1326
// of 16 KB 9.1 / 8.7, 3642 of 1.2 KB 6.9 / 6.7, 3735 of 7.4 KB 11.3 / 10.2.
bool stays_by_entry(long long entries, int row_vecs, bool vec16) {
  if (!vec16) return entries <= 2700;
  return entries <= 3000 && row_vecs <= 640 && (entries > 2048 || row_vecs > 256);
}

// Up to 1024 entries every wave holds all keys. That costs each workgroup, which moves a piece of 256 vectors, as many loads and
// compares as there are keys per lane, and pays up to about 16000 of them over all pieces, 12000 where a vector is one
// element. Beyond (many tokens with long rows and few entries) a wave per entry is ahead; only tokens with four and more
// entries of whole vectors then have as much to store per piece. us, held by every wave / a wave per entry: 1 per token, 500 of
// 14 KB (16000) 4.4 / 4.6, 728 of 4.6 KB (17472) 4.5 / 4.0, 918 of 13 KB (58752) 8.1 / 5.9; of single elements 60 tokens of 7167,
// 2 each (3360) 3.6 / 4.1, 179 of 1971, 2 each (11456) 4.1 / 4.2, 126 of 6277, 2 each (12600) 5.0 / 4.6, 500 of 7167 (112000) 14.1 /
// 5.4, 200 of 4097, 4 each (54400) 8.8 / 6.3.
//
// Longer streams go to the kernel that ranks four tokens in one pass over the keys, but for two kinds of short ones, where
// a pass is little beside the rows and the others store them faster: fewer than four entries per token up to
// 1280 of them (600 tokens of 14 KB, 2 per token 6.2 / 6.4 us), with one entry per token further (stays_by_entry), and long rows as long as a pass over the keys is short
// beside the rows of a token, which the tokens and the vectors of a row measure: the others / that kernel 8 per token of 14 KB, 1024
// tokens 26.2 / 27.8, 1400 34.3 / 36.9, 1800 43.7 / 48.9, 4096 118.9 / 102.5; 4 of 10 KB, 1000 tokens 10.7 / 11.1, 1500
// 16.2 / 16.3; 6 of 13.7 KB, 600 tokens 12.0 / 13.0; but 3 of 9.2 KB, 500 tokens 5.6 / 5.4, and rows moved by elements 18.1 /
// 10.2 (6 of 4111, 500 tokens). Rows of 7 KB (6.4 of seven entries) are long in that sense beyond 4096 entries, where the others rank eight at a
// time: 8 per token of 8 KB, 997 tokens 15.0 / 16.9, 1518 23.0 / 26.0, 5 per token, 919 10.5 / 11.8, 8 of 7.7 KB, 953 14.1 / 16.1, 7 of 6.7 KB, 648
// 9.0 / 10.0; but 399 of 8 KB, 8 per token 8.2 / 7.8, and not with four entries (1156 of 7 KB 11.4 / 10.1), of which
// rows of more than 4 KB up to 2048 of them: 492 tokens of 4.5 KB 4.4 / 4.7, 509 of 8 KB 4.8 / 5.4; but 523 of 5.1 KB 5.7 / 5.2.
//
// The others: tokens with several entries have one workgroup per (token, 256-vector chunk) that stores the chunk to
// all of the token's slots (measured at K = 8, H = 7168: 8.4 us against 8.8 us with a wave per
// entry; one chunk per workgroup beats two or four). With one or two entries per token the
// wave-per-entry kernel scans fewer keys per byte moved.
SendWay send_way(long long tokens, int per_token, int ranks, int row_vecs, bool vec16) {
  const long long entries = tokens * per_token;
  const int pieces = (row_vecs + BLOCK - 1) / BLOCK;
  // (a job without tokens goes to the kernels below, which then read nothing)
  if (entries > 0 && entries <= FEW_ENTRIES && per_token <= FEW_MAX_K && tokens * pieces <= 1 << 20) {
    if (vec16 && per_token >= FANOUT_MIN_K) return SEND_FEW;
    return tokens * pieces * few_keys(entries) <= (vec16 ? 16000 : 12000) ? SEND_FEW : SEND_BY_ENTRY;
  }
  const bool few_entries = (per_token < FANOUT_MIN_K && entries <= 1280) || (per_token == 1 && stays_by_entry(entries, row_vecs, vec16));
  const bool long_rows = per_token >= FANOUT_MIN_K && vec16 && tokens <= 3ll * row_vecs &&
                         (row_vecs > 2 * BLOCK || (per_token > 4 && row_vecs >= (per_token > 6 ? 400 : 448) && entries > 4096) ||
                          (per_token == 4 && row_vecs > BLOCK && entries <= 2048));
  if (entries > 0 && entries <= BLOCK_MAX_ENTRIES && ranks <= BLOCK_RANKS && per_token * ROWS <= 64 && !few_entries && !long_rows)
    return SEND_BLOCK;
  if (per_token >= FANOUT_MIN_K && (ranks + 2ll) * entries <= INT_MAX && items_fit(tokens, pieces))
    return row_vecs > BLOCK && entries < 65536 && ranks < 16384 ? SEND_FANOUT_WIDE : SEND_FANOUT;
  return SEND_BY_ENTRY;
}

// Tokens of a workgroup of dispatch_long_kernel, or 0 where a stream stays with its choice above. From 5120 entries on it takes whole vectors over from
// dispatch_block_kernel, and from 65281 on from all others, which compare every key with every entry. It stays behind
//  - below 5120 entries (4900, 613 tokens of 900 bytes, 6.2 / 6.4 us) and with few tokens and entries, of which a workgroup then holds three or four (722 of
//    272 bytes, 8 per token 5.4 / 6.1, 1005 of 5.6 KB, 6 each 11.1 / 12.2),
//  - with five and more entries per token, of which a workgroup holds few tokens, just past a batch of 8192 keys, which is another pass: rows of 1 to 6.4 KB,
//    8193 to 10240 entries, 107 streams 1.03 on average (1836 of 2.3 KB, 5 each 9.2 / 10.1, 1627 of 2.7 KB, 6 each 10.3 / 11.3, 1046 of 1.9 KB, 8 each
//    8.0 / 8.7; of up to 8192 entries 0.96, of up to 1 KB 0.99), and past two batches and the entries that a workgroup per unit holds rows of up to 3 KB
//    (2803 of 1.9 KB, 6 each 14.8 / 15.7, 2235 of 1.5 KB, 8 each 14.1 / 15.0, 2225 of 272 bytes 12.7 / 13.4).
// Over 700 streams of 5120 to 32768 entries, one to eight per token, rows of 128 bytes to 14 KB, one launch after another, the choice takes 0.74 of the
// time of dispatch_block_kernel; 26 are more than 3 % behind, the worst by 10 % (4108 tokens of 11 KB, 3 each 35.3 / 39.0).
//
// Short rows have one workgroup per unit, which leaves the passes over the keys to the fewest, as long as those hold all tokens (64 entries each);
// others two, and where a row takes longer than a pass four. us, with 256 / 512 / 768 / 1024 workgroups: 3590 tokens of 1 KB, 3 per token 7.5 / 10.6 /
// 14.4; 2675 of 2.1 KB, 6 each 15.4 / 13.0 / 15.7; 2055 of 5.8 KB, 4 each 14.2 / 15.2 / 16.8; 3594 of 6.3 KB, 8 each 40.5 / 40.7 / 41.1 / 44.4; 3212 of
// 5 KB, 5 each 28.6 / 24.5 / 24.1 / 25.0; 3731 of 14.3 KB, 4 each 63.9 / 62.5 / 59.1 / 57.2; 4084 of 11.2 KB, 6 each 60.9 / 60.3 / 60.2 / 56.6; 4096 of
// 14 KB, 8 each, with the other stages, - / 809 / 815 / 807.
int long_tokens(SendWay way, long long tokens, int per_token, int ranks, int row_vecs, bool vec16) {
  const long long entries = tokens * per_token;
  if (!vec16 || ranks > BLOCK_RANKS || per_token > 64 || entries < LONG_ENTRIES || entries > LONG_MAX_ENTRIES ||
      (way != SEND_BLOCK && entries <= BLOCK_MAX_ENTRIES))
    return 0;
  if (tokens < 1024 && entries < 6400) return 0;
  if (per_token >= 5 && row_vecs > 64 && row_vecs <= 400 && entries > 8192 && entries <= 10240) return 0;
  if (per_token >= 6 && row_vecs <= 192 && entries >= 16800 && entries <= 18432) return 0;
  const bool one_each = row_vecs <= (entries <= 9216 ? 400 : 256) && tokens <= 64 / per_token * 264;
  const int workgroups = one_each ? 256 : row_vecs > 512 && entries >= 7500 ? 1024 : 512;
  return (int)std::min<long long>(64 / per_token, (tokens + workgroups - 1) / workgroups);
}

// Vectors per lane of a wave of dispatch_block_kernel, for rows that a wave has in one go with `nvw`. Rows
// are cut into pieces of two vectors per lane where there are few workgroups otherwise, else of four: pieces of 2 / 4 /
// whole rows: 250 tokens of 5.8 KB, 8 per token 4.8 / 5.1 / 5.5 us. (Whole vectors come here with up to 5119 entries, and with some more of rows of up to
// 6.4 KB: long_tokens.) With one entry a piece would do little but rank: 2000 of 14 KB 13.4 / 10.7 / 9.6. Two and three
// entries pay for a piece of long rows only, two for one of four vectors: 1292 of 5 KB, 2 per token 7.1 / 6.6 / 5.9, 1380 of 15 KB 14.0 /
// 12.6 / 12.4, 1001 of 13.7 KB 8.5 / 8.0 / 9.2, 671 of 10.8 KB 6.1 / 5.5 / 5.8; 893 of 4.5 KB, 3 per token 6.1 / 5.5 / 5.3, 537 of 13.6 KB
// 6.5 / 7.0 / 7.2.
int block_piece(long long tokens, int per_token, int nvw, bool vec16) {
  if (!vec16 || per_token == 1 || (per_token < FANOUT_MIN_K && nvw <= 8)) return nvw;
  if (per_token == 2) return std::min(nvw, 4);
  return std::min(nvw, (tokens + ROWS - 1) / ROWS <= 400 ? 2 : 4);
}

// ---------------------------------------------------------------- stage 2

constexpr int STAGE2_THROUGH_ROWS = 1024;
constexpr long long STAGE2_THROUGH_BYTES = 8 << 20;

bool recv_through(long long rows_hint, long long row_bytes) {
  return rows_hint >= STAGE2_THROUGH_ROWS || rows_hint * row_bytes >= STAGE2_THROUGH_BYTES;
}

enum RecvFew { RECV_NOT_FEW, RECV_FEW_PLAIN, RECV_FEW_THROUGH };

// Whether a planned stage 2 runs on dispatch_recv_few_kernel, where every wave holds all keys, and how that stores its rows
// (Store). `nvw`: vectors per lane of the wave that moves a row, or a piece of one.
//
// Up to 1024 rows, but for two kinds. Elements: each of a row's pieces of 1024 ranks the row again, which costs more than
// the other kernel's shared scan above 512 rows (padded; in the compact layout the scan is as long). us, held by every wave / scan: 900
// rows of 5001 elements 8.3 / 6.6, 1000 of 2049 5.8 / 5.0, 700 of 7167 7.4 / 6.6; 512 of 2049 4.2 / 4.2, 256 4.1 / 4.4.
// And 8 MB of rows of 13 or 14 vectors per lane: those and the keys leave room for fewer waves. us, held and plain / held and
// past L2 / scan and past L2, 14 KB: 600 rows 5.15 / 4.93 / 4.78, 800 6.06 / 5.51 / 5.18, 900 6.44 / 5.94 / 5.42, 1024
// 6.94 / 6.71 / 5.86; compact 900 6.62 / 6.03 / 5.93. Rows of other lengths stay, from 8 MB on past L2 as there: 900 of 10 KB 5.27 /
// 4.77 / 5.31, 800 of 12 KB 5.49 / 5.20 / 5.59, 600 of 16 KB 5.67 / 5.43 / 6.20; longer ones, of several pieces, with plain
// stores (800 of 28 KB 9.10 / 9.65 / 9.11, 500 of 56 KB 9.98 / 10.92 / 10.80).
RecvFew recv_few(long long rows_hint, int row_vecs, int nvw, bool vec16, bool compact) {
  if (rows_hint > FEW_ENTRIES) return RECV_NOT_FEW;
  const bool pieces = row_vecs > 64 * nvw;
  if (!vec16) return pieces && !compact && rows_hint > 512 ? RECV_NOT_FEW : RECV_FEW_PLAIN;
  if (rows_hint * row_vecs * 16 < STAGE2_THROUGH_BYTES) return RECV_FEW_PLAIN;
  return nvw == 14 ? RECV_NOT_FEW : pieces ? RECV_FEW_PLAIN : RECV_FEW_THROUGH;
}

// ---------------------------------------------------------------- stage 4

// Vectors per lane of combine_recv_mapped_kernel, and whether it reads rows past the caches. One vector with more than two entries per token, or
// four of a large stream: of fewer a wave has little to do but to find them. us of the graph of stages as above, one / two: 8 per token
// of 14 KB, 69 MB 100.8 / 101.8; 4 of 5.8 KB, 18 MB 38.6 / 39.3; 3 of 8 KB, 20 MB 40.7 / 41.2, 101 MB 143.2 / 142.3; 2 of 8 KB, 67 MB 105.7 / 103.4; 1
// of 8 KB, 34 MB 69.2 / 67.3. Plain / nontemporal loads (rows and results): 78 MB 100.8 / 101.4, 100 MB (2 per token) 111.4 / 103.4, 118 MB
// 151.1 / 148.0, 134 MB 149.2 / 142.3, 528 MB 652.7 / 641.6; of 67 MB (1 per token) 67.3 / 65.7, of 52 MB 72.5 / 73.6.
constexpr long long COMBINE_PAST_BYTES = 80ll << 20;
int mapped_vecs(int per_token, int row_vecs, bool past) { return row_vecs > 64 && per_token <= (past ? 4 : 2) ? 2 : 1; }

// Tokens of a workgroup of combine_recv_block_kernel, or 0 where a workgroup looks for the rows of one token: up to as many tokens as there are units
// that has no less to share (256 of 14 KB, 8 per token 8.1 / 8.7 us, 128 of 11 KB, 7 each 5.1 / 5.4; 278 of 8.6 KB, 4 each 5.4 / 5.4). One workgroup
// per unit, two where there are three tokens for each. us, with 256 / 512 / 1024 of them: 377 of 10 KB, 6 each 7.4 / 8.0 / 8.0; 531 of 6.4
// KB, 2 each 4.9 / 5.2 / 5.6; 885 of 5.8 KB, 4 each 7.5 / 7.2 / 9.3; 1428 of 7.6 KB, 2 each 8.8 / 7.8 / 9.2; 1622 of 1 KB 4.5 / 4.4 / 5.2.
constexpr int COMBINE_BLOCK = 1024, COMBINE_TOKENS = 64;  // lanes, and most tokens, of a workgroup
int combine_block(long long tokens, long long rows_hint, int per_token) {
  if (tokens <= 256 || rows_hint <= 512 || per_token > 8) return 0;
  const int workgroups = tokens >= 768 ? 512 : 256;
  return (int)std::min<long long>(COMBINE_TOKENS, (tokens + workgroups - 1) / workgroups);
}

// ---------------------------------------------------------------- jobs on one GPU

// Tokens of a workgroup of local_dispatch_long_kernel, or 0 where a launch of its own plans the rows: more ranks than its tables have, more experts than
// it counts in 36 KB, or so many keys that what 256 workgroups read of them (of 128 KB, 32 MB out of L2) is not little beside the rows. One
// workgroup per unit: us of whole calls, plan / with 256 / 512 / 1024 workgroups, 8 ranks of 238 tokens of 4.5 KB, 6 each 34.8 / 32.8 / 33.6 / 46, of
// 65 of 8.6 KB, 5 each 18.4 / 15.7 / 16.7 / 27; one rank of 3084 of 1.6 KB, 2 each 24.8 / 21.0 / 22.6 / 26.
constexpr int LOCAL_LONG_KEYS = 32768, LOCAL_LONG_MAX_K = 64;
constexpr int LOCAL_LONG_ENTRIES = LOCAL_LONG_KEYS / 256 + LOCAL_LONG_MAX_K;  // most entries of a workgroup
int local_long_tokens(long long tokens, int per_token, int ranks, int experts) {
  const long long entries = tokens * per_token;
  if (entries < 1 || entries > LOCAL_LONG_KEYS || per_token > LOCAL_LONG_MAX_K || ranks > 8 || experts > 512) return 0;
  return (int)((tokens + 255) / 256);
}
// Vectors per lane of its pieces: two, of many long rows four (235 MB 58.9 / 56.4 us, 146 MB 39.8 / 39.0, but 92 MB 41.5 / 41.6, 24 MB 15.6 / 16.9).
int local_long_vecs(long long bytes, int row_vecs) { return row_vecs <= 64 ? 1 : row_vecs > 128 && bytes >= 128ll << 20 ? 4 : 2; }

// Vectors of a row that a lane of local_dispatch_few_kernel moves: one, two or four, of single elements one, four or eight. Every
// workgroup holds all keys, so that many pieces of rows cost more than the rows: beyond two workgroups per unit with tables of
// several ranks or more than 1024 keys, else beyond four, a lane moves more. (Up to 256 keys are so few that pieces of
// whole vectors stay as they are.) us, one / two / four / eight vectors (ranks x tokens x entries, hidden): 8 x 60 x 2, 7168 8.1 / 6.7 / 5.8 / 6.6,
// 8 x 100 x 1, 7168 9.9 / 7.7 / 6.5 / 8.3, 8 x 16 x 4, 7168 5.1 / 5.2 / 6.2, 1 x 900 x 1, 7168 7.1 / 5.6 / 5.1 / 6.9, 1 x 128 x 8,
// 7168 5.7 / 6.0 / 8.1; single elements 8 x 64 x 2, 7167 30.0 / 18.2 / 12.4 / 10.3, 8 x 16 x 8, 3001 9.3 / 7.3 / 7.2 / 8.2, 1 x 250 x 8, 5001
// 24.3 / 15.9 / 11.7 / 11.2, 1 x 1000 x 1, 513 5.1 / 4.5 / 3.6 / 4.0, 1 x 16 x 8, 7167 3.8 / 4.4 / 5.1 / 6.3.
int local_few_vecs(long long tokens, long long entries, int ranks, int row_vecs, bool vec16) {
  if (row_vecs <= BLOCK || (vec16 && entries <= 64 * 4)) return 1;
  auto workgroups = [&](int vecs) { return tokens * ((row_vecs + BLOCK * vecs - 1) / (BLOCK * vecs)); };
  const int limit = entries > 64 * 16 || (ranks > 1 && entries > 64 * 4) ? 512 : 1024;
  if (workgroups(1) <= limit) return 1;
  const int more = vec16 ? 2 : 4;
  return row_vecs <= BLOCK * more || workgroups(more) <= (vec16 ? limit : 1024) ? more : 2 * more;
}

}  // namespace
