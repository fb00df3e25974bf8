// wave_dp.h -- the gapped X-drop with one wave per extension and the DP row
// in registers.
//
// Lane l holds the C consecutive columns base + l C .. base + l C + C - 1 of
// a window of 64 C columns that moves along with the band; everything that
// belongs to the extension as a whole (band ends, best score, row) is
// wave-uniform and lives in scalar registers.  A row is about 90
// instructions with no memory access but the score lookups, which are read a
// row ahead; what bounds it is their issue and the scans' dependent steps:
// 280 ns a row for a wave that has its SIMD to itself, where a lane that
// walks the row's 20 to 30 cells one by one takes 0.5 to 1.3 us.  This is the
// form for calls with too few jobs to fill the chip with a lane each, and
// for bands that outgrow the lanes' first LDS ring.  Measured per call
// against the lane forms: 300 read extensions 310 -> 25 us, 20,011 of
// proteins of 100-500 residues 4.0 -> 0.31 ms, 3,001 of Pareto lengths up to
// 35,000 99.8 -> 10 ms; 1,000,003 of reads (first ring on lanes, its
// overflow here) 1.38 -> 1.24 ms.  C is 1 and widens to 2 and 4 when a band
// needs it: with one column per lane nothing inside a lane is serial, and bands
// at the presearch's cutoff are 15 to 30 columns wide.  The result build
// (traceback.hip) records the operations of the same rows, in windows of up
// to 4 columns per lane at its higher cutoff.
//
// The row recurrence is GappedOneSide's (src/gapped_extender.cpp:306-471),
// with the two values that it carries from column to column as scans:
//   * the horizontal gap g: a gap opened from a cell that a gap itself
//     reached is never better (gap opening >= 0), so with sp(a) the cell's
//     score before the horizontal gap, g(a) = max over b < a of
//     sp(b) - (open + ext) - (a - 1 - b) ext.  The reference resets g to
//     kInitScore after a pruned cell; without the reset g through a pruned
//     cell stays below the running best less the cutoff from there on, so
//     it neither keeps a cell nor sets a kept cell's score;
//   * the running best: an exclusive max-scan of the row's scores, needed
//     only in rows that raise the best score.
// Columns outside the band hold kInitScore in both values, which (cutoffs
// up to kWaveDpMaxCutoff) no diagonal step of up to 127 lifts back to a kept
// score; so the band's ends need no tests of their own:
//   * column array_start is a cell whose diagonal is such a dead column;
//   * the columns that the reference appends behind a kept last column while
//     the gap holds are those whose g passes the prune test (all of the
//     row's cells lie before them, so the running best there is the row's);
//   * a live diagonal step into column array_end happens only where the
//     reference appends no pruned column behind a kept one: at the query's
//     end, where `limit` cuts it, and in the row after the band has shrunk
//     from there, which `bare` marks.
#pragma once

#include <hip/hip_runtime.h>

#include <limits.h>

#include "gz_common.h"
#include "gz_device.h"

namespace gz {

// A delimiter column scores kWall, which takes at least 128 off a score:
// more than any cutoff the form serves.
constexpr int kWaveDpMaxCutoff = 120;
constexpr int kWaveDpMaxGap = 512;    // gap open + extension
constexpr int kWall = -128;
constexpr int kWallCode = 32;
constexpr int kScoreStride = 64;      // bytes per score row (32 codes, the wall)
constexpr int kNoScore = -(1 << 28);  // below every score

// Whether the form is exact for these parameters.
inline bool WaveDpServes(int cutoff, int gap_open, int gap_ext) {
  return cutoff >= 0 && cutoff <= kWaveDpMaxCutoff && gap_open >= 0 && gap_ext >= 0 &&
         gap_open <= kWaveDpMaxGap && gap_open + gap_ext <= kWaveDpMaxGap;
}

// The score table: kScoreStride bytes per database code, [code] the score,
// the wall behind the 32 codes.
__device__ __forceinline__ void StageWaveDpScores(int8_t *lds, const int *matrix, uint32_t nl) {
  for (uint32_t i = threadIdx.x; i < kTableDim * kScoreStride; i += blockDim.x) {
    const uint32_t r = i / kScoreStride, c = i % kScoreStride;
    lds[i] = c >= kTableDim ? (int8_t)kWall
                            : (r < nl && c < nl) ? (int8_t)matrix[r * nl + c] : (int8_t)0;
  }
}

struct WaveDpParams {
  const uint64_t *queries;
  const uint64_t *database;
  uint32_t delim;
  int gap_init;  // gap open + extension
  int gap_ext;
  int cutoff;
  // columns kept free behind the band while its query side goes on past the
  // window (a row whose gap fills more is noticed at the next one)
  int margin;
};

// What the presearch's parameters (26, 12, 1) need: a row's gap fills at most
// (cutoff - gap_init) / gap_ext + 1 columns.  At higher cutoffs gaps that
// fill more are rare; a side that loses a row to one starts again in a wider
// window.  A margin for all of them would leave the windows no room: the
// result build of 3,001 proteins at cutoff 90 takes 46 ms with it (bands that
// fit 256 columns run on lanes) and 0.92 ms with this one.
constexpr int kWaveDpMargin = 16;

// Most columns per lane that a call's jobs take in the score-only form, 0
// where lanes are the better form.  `wide`: the longest query side, as the
// power of two of columns that it is given.
//   * Two serve sides of up to 62 residues, which end inside the first
//     window; sides of up to 126, which end inside the second, if their first
//     row stays below 64 columns; and cutoffs that pay for few gaps, whose
//     bands stay below 128.  The kernel for four keeps 84 registers instead of
//     47 and is 2 to 5% slower where two are enough (20,011 of 100-500
//     residues at cutoff 26, gaps 11/1: 309 us and 325; at 42 485 and 497;
//     60,000 frames of 100 residues at 60 677 and 693); where they are not,
//     jobs run again on the global ring (20,011 at 46 762 and 553, at 60 1,367
//     and 648; 3,001 of Pareto lengths at 60 70 ms and 19).
//   * Long sides whose bands outgrow 256 columns too pay for both forms, and
//     the longest one's rows are the call's time: 3,001 of Pareto lengths at
//     110 88 ms so and 68 on lanes, at 120 94 and 73, at 100 32 and 65; 3,000 of
//     2,000-4,000 residues at 120 9.9 and 9.3.  Shorter sides gain anyway (3,000
//     of 1,000-2,000 at 120 4.2 and 5.5).
inline int RowColumnsFor(int cutoff, int gap_open, int gap_ext, uint32_t wide) {
  if (!WaveDpServes(cutoff, gap_open, gap_ext)) return 0;
  const int gap_init = gap_open + gap_ext;
  if (wide <= 64 || cutoff < gap_init) return 2;
  if (gap_ext == 0) return 4;
  const int span = (cutoff - gap_init) / gap_ext + 1;  // columns that one gap can pass
  if (wide <= 128 && span < kWave - 1) return 2;
  if (wide > 2048 && span * cutoff > 800 * gap_init) return 0;
  return span > 16 && 2 * cutoff > 7 * gap_init ? 4 : 2;
}

// The value of a wave-uniform expression as a scalar.
__device__ __forceinline__ int Uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t Uniform(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ uint64_t Uniform(uint64_t v) {
  return (uint64_t)Uniform((uint32_t)v) | ((uint64_t)Uniform((uint32_t)(v >> 32)) << 32);
}

// Inclusive max-scan over the wave (INT_MIN as the identity lets every step
// be one v_max with a DPP operand).
__device__ __forceinline__ int WaveMaxScan(int v) { return WaveInclusiveMaxDpp(v, INT_MIN); }

// kWaveDpWiden: the band does not fit the window (the state is that before
// the row); kWaveDpLost: the row's gap went on outside the window.
enum : int { kWaveDpDone = 1, kWaveDpWiden = 2, kWaveDpLost = 3 };

// What a wave holds of an extension besides the row: all of it uniform.
struct WaveDpBand {
  int base;              // the window's first column
  int start, end;        // array_start, array_end, less base
  int last_col;          // the query side's last residue column (INT_MAX: not seen)
  int best, best_col, best_row, row, cells;
  int widest;            // most columns of a row's band
  int bare;              // -1: no pruned column behind a kept last one, else 0
  uint32_t qpos;
  // the database walk: unread codes of the current word, the next word
  uint64_t word, ahead;
  uint32_t index;        // of the next word
  int left;              // unread codes in the current one
  uint32_t d;            // the row's code
};

template <bool kReverse, int C>
struct WaveDp {
  static constexpr int W = kWave * C;
  // A read of C <= 12 codes touches two packed words, 24 codes from the
  // first's word on; new columns are read at most this far past a residue,
  // which keeps the words inside the delimiter padding.
  static constexpr int kReach = (int)kPackPadCodes - 2 * (int)kCodesPerWord;
  static_assert(C <= 12, "a lane's codes lie in two words");

  // the lane's columns of the row
  int h[C], e[C];    // score and vertical gap
  int code[C];       // query codes (kWallCode where there is no residue)
  int limit[C];      // INT_MAX, or kNoScore past the query side's last residue

  static __device__ __forceinline__ int Lane() { return (int)__lane_id(); }
  static __device__ __forceinline__ int Offset(int j) { return Lane() * C + j; }

  // Whether the query side ends inside the window (with room for the shifts
  // by `start`, which then is at most W - C - 2).
  static __device__ __forceinline__ bool EndsInside(const WaveDpBand &B) {
    return B.last_col - B.base < W - C;
  }

  // The codes of the lane's columns (column c >= 1 is the query code at
  // qpos + (c - 1) inc); every one must lie within kReach of a residue.
  static __device__ __forceinline__ void ReadCodes(const WaveDpParams &P, const WaveDpBand &B,
                                                   int (&out)[C]) {
    const int c0 = B.base + Offset(0);
    const uint32_t first = kReverse ? B.qpos - (uint32_t)(c0 - 1) - (uint32_t)(C - 1)
                                    : B.qpos + (uint32_t)(c0 - 1);
    const uint32_t p = first + kPackPadCodes, w = p / kCodesPerWord, k = p - w * kCodesPerWord;
    const uint64_t lo = P.queries[w], hi = P.queries[w + 1];
    const uint64_t mask = (1ull << (kCodeBits * kCodesPerWord)) - 1;
    const uint64_t win = ((lo & mask) >> (kCodeBits * k)) |
                         ((hi & mask) << (kCodeBits * (kCodesPerWord - k)));
#pragma unroll
    for (int j = 0; j < C; ++j)
      out[j] = (int)(win >> (kCodeBits * (kReverse ? C - 1 - j : j))) & 31;
  }

  // Reads columns base + [from, to) (to - from <= kReach, every column
  // before them a residue) and notes the first delimiter.
  __device__ __forceinline__ void ReadColumns(const WaveDpParams &P, WaveDpBand &B, int from,
                                              int to) {
    int first = INT_MAX;
    const int c0 = Offset(0);
    if (c0 + C > from && c0 < to) {
      int v[C];
      ReadCodes(P, B, v);
#pragma unroll
      for (int j = C - 1; j >= 0; --j) {
        if (c0 + j >= from && c0 + j < to) {
          code[j] = v[j];
          if ((uint32_t)v[j] == P.delim) first = c0 + j;
        }
      }
    }
    const uint64_t seen = __ballot(first != INT_MAX);
    if (seen)
      B.last_col = B.base - 1 +
                   __builtin_amdgcn_readlane(first, __ffsll((unsigned long long)seen) - 1);
  }

  // Reads the window's columns from `from` on, in steps of kReach, the later
  // ones where the earlier ones hold no delimiter.
  __device__ __forceinline__ void ReadWindow(const WaveDpParams &P, WaveDpBand &B, int from) {
    for (int c = from; c < W && B.last_col == INT_MAX; c += kReach)
      ReadColumns(P, B, c, c + kReach < W ? c + kReach : W);
  }

  // After the window or last_col changed: wall codes and limits.
  __device__ __forceinline__ void Limits(const WaveDpBand &B) {
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int a = B.base + Offset(j);
      limit[j] = a <= B.last_col ? INT_MAX : kNoScore;
      if (a > B.last_col || a == 0) code[j] = kWallCode;
    }
  }

  __device__ __forceinline__ void LoadScores(const int8_t *sm, int (&m)[C], uint32_t d) const {
    const int8_t *r = sm + d * kScoreStride;
#pragma unroll
    for (int j = 0; j < C; ++j) m[j] = r[code[j]];
  }

  static __device__ __forceinline__ uint32_t NextCode(const WaveDpParams &P, WaveDpBand &B) {
    uint32_t c;
    if (kReverse) {
      c = (uint32_t)(B.word >> (kCodeBits * (kCodesPerWord - 1))) & 31u;
      B.word <<= kCodeBits;
    } else {
      c = (uint32_t)B.word & 31u;
      B.word >>= kCodeBits;
    }
    if (--B.left == 0) {
      B.word = Uniform(B.ahead);
      B.left = (int)kCodesPerWord;
      // the word before holds residues or the walk's delimiter, so the word
      // after the next lies inside the padding
      B.index = kReverse ? B.index - 1 : B.index + 1;
      B.ahead = P.database[B.index];
    }
    return c;
  }

  // Moves the window up by `lanes` lanes.
  __device__ __forceinline__ void Rebase(const WaveDpParams &P, WaveDpBand &B, int lanes) {
    const int from = Lane() + lanes;
    const bool inside = from < kWave;
    const int at = 4 * (inside ? from : Lane());
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int vh = __builtin_amdgcn_ds_bpermute(at, h[j]);
      const int ve = __builtin_amdgcn_ds_bpermute(at, e[j]);
      const int vc = __builtin_amdgcn_ds_bpermute(at, code[j]);
      h[j] = inside ? vh : kInitScore;
      e[j] = inside ? ve : kInitScore;
      code[j] = inside ? vc : kWallCode;
    }
    B.base += lanes * C;
    B.start -= lanes * C;
    B.end -= lanes * C;
    // new columns follow residues only (a delimiter in the old window ends
    // the query side)
    ReadWindow(P, B, W - lanes * C);
    Limits(B);
  }

  // The seed (q, dp) and its first row.
  __device__ __forceinline__ int Begin(const WaveDpParams &P, WaveDpBand &B, uint32_t q,
                                       uint32_t dp) {
    const int gi = P.gap_init, ge = P.gap_ext;
    B.qpos = q;
    B.base = B.start = B.row = B.cells = B.widest = 0;
    B.end = 1;
    B.best = 0;
    B.best_col = 0;
    B.best_row = -1;
    B.bare = 0;
    const uint32_t p = dp + kPackPadCodes, w = p / kCodesPerWord, k = p - w * kCodesPerWord;
    B.index = kReverse ? w - 1 : w + 1;
    const uint64_t word = P.database[w];
    B.ahead = P.database[B.index];
#pragma unroll
    for (int j = 0; j < C; ++j) code[j] = kWallCode;
    B.last_col = INT_MAX;
    ReadColumns(P, B, 1, kReach);
    ReadWindow(P, B, kReach);
    Limits(B);
    B.word = Uniform(word);
    if (kReverse) {
      B.word <<= kCodeBits * (kCodesPerWord - 1 - k);
      B.left = (int)k + 1;
    } else {
      B.word >>= kCodeBits * k;
      B.left = (int)(kCodesPerWord - k);
    }
    B.d = NextCode(P, B);
    if (B.last_col == 0 || B.d == P.delim) return kWaveDpDone;
    // the first row: gap scores down to the cutoff or the last residue, and
    // a pruned column behind them
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int a = Offset(j);
      const int s = -gi - (a - 1) * ge;
      const bool on = a <= B.last_col && s >= -P.cutoff;
      h[j] = a == 0 ? 0 : on ? s : kInitScore;
      e[j] = a == 0 ? -gi : on ? s - gi : kInitScore;
    }
    int stop = P.cutoff < gi ? 1 : ge > 0 ? (P.cutoff - gi) / ge + 2 : INT_MAX;
    if (B.last_col < stop) stop = B.last_col + 1;  // the delimiter's column comes first
    if (stop >= W) return kWaveDpLost;
    B.end = stop <= B.last_col ? stop + 1 : stop;
    return 0;
  }

  // Rows until the extension ends or the band needs a wider window.  `ops`
  // records the operations (NoOps: none).  Every branch is wave-uniform; the
  // row loop has one exit, and what it tests and carries is integer
  // arithmetic (uniform booleans cost several scalar instructions each).
  template <class Ops>
  __device__ __forceinline__ int Rows(const WaveDpParams &P, const int8_t *sm, WaveDpBand &B,
                                      Ops &ops) {
    const int gi = P.gap_init, ge = P.gap_ext, cutoff = P.cutoff;
    const int rel = Offset(0);
    const int key_add = (rel + C - 1) * ge - gi, key_sub = (rel - 1) * ge;
    int score[C];
    LoadScores(sm, score, B.d);
    for (;;) {
      // what a row rarely needs: room behind the band, unless the query side
      // ends inside the window (the band then ends with it)
      int room = W - P.margin;
      while (!EndsInside(B) && B.end > room) {
        // a live column at the window's end: the gap may go on outside
        if (B.end > W) return kWaveDpLost;
        int lanes = B.start / C;
        lanes = lanes < kReach / C ? lanes : kReach / C;
        if (lanes == 0) return kWaveDpWiden;
        Rebase(P, B, lanes);
        LoadScores(sm, score, B.d);
      }
      if (EndsInside(B)) room = W;
      // and a cleared diagonal
      if (B.bare) {
#pragma unroll
        for (int j = 0; j < C; ++j) score[j] = Offset(j) == B.end ? kNoScore : score[j];
      }
      const int last_rel = B.last_col - B.base;
      uint64_t any;
      int stop;
      do {
        if (!ops.Row(B)) return kWaveDpLost;
        // the next row's code and scores
        const uint32_t dn = NextCode(P, B);
        int next[C];
        LoadScores(sm, next, dn);
        int sp[C], s[C], diag[C], gap[C];
        {
          int prev = WaveShiftUp1(h[C - 1], kInitScore);
          int total = 0;  // the best gap source, as the gap into the lane's following column
#pragma unroll
          for (int j = 0; j < C; ++j) {
            diag[j] = prev + score[j];
            prev = h[j];
            sp[j] = diag[j] > e[j] ? diag[j] : e[j];
            const int t = total - ge;
            total = j == 0 || t < sp[j] ? sp[j] : t;
          }
          // as a key that does not depend on the column it is scanned over
          // the lanes
          int g = WaveShiftUp1(WaveMaxScan(total + key_add), kNoScore) - key_sub;
#pragma unroll
          for (int j = 0; j < C; ++j) {
            gap[j] = g;
            // max(sp, g), or at most sp (a wall) past the last residue
            asm("v_med3_i32 %0, %1, %2, %3" : "=v"(s[j]) : "v"(sp[j]), "v"(g), "v"(limit[j]));
            if (j + 1 < C) {
              const int t = g - ge, o = sp[j] - gi;
              g = t > o ? t : o;
            }
          }
        }
        uint64_t live[C];
        if constexpr (C == 1) {
          // the columns that raise the best score, one after the other; the
          // columns behind each are pruned against it
          live[0] = __ballot(s[0] >= B.best - cutoff);
          uint64_t up = __ballot(s[0] > B.best);
          if (up) {
            int c;
            do {
              c = __ffsll((unsigned long long)up) - 1;
              B.best = __builtin_amdgcn_readlane(s[0], c);
              live[0] &= ~(~1ull << c) | __ballot(s[0] >= B.best - cutoff);
              up = __ballot(s[0] > B.best);
            } while (up);
            B.best_col = B.base + c;
            B.best_row = B.row;
          }
        } else {
          int top = s[0];
#pragma unroll
          for (int j = 1; j < C; ++j) top = s[j] > top ? s[j] : top;
          int run = B.best;
          if (__ballot(top > B.best)) {
            const int incl = WaveMaxScan(top);
            const int before = WaveShiftUp1(incl, kNoScore);
            run = before > run ? before : run;
            B.best = __builtin_amdgcn_readlane(incl, kWave - 1);
            B.best_col = INT_MAX;
            B.best_row = B.row;
#pragma unroll
            for (int j = 0; j < C; ++j) {
              const uint64_t at = __ballot(s[j] == B.best);
              const int c =
                  at ? B.base + (__ffsll((unsigned long long)at) - 1) * C + j : INT_MAX;
              B.best_col = c < B.best_col ? c : B.best_col;
            }
          }
#pragma unroll
          for (int j = 0; j < C; ++j) {
            live[j] = __ballot(s[j] >= run - cutoff);
            run = s[j] > run ? s[j] : run;
          }
        }
        // the first kept column past `start`, and the last live one
        uint64_t past[C];
        int first = INT_MAX, last = -1;
        any = 0;
#pragma unroll
        for (int j = 0; j < C; ++j) {
          // lanes l with l C + j > start (start <= end - 2 or the band's only
          // column, so the shift is below 64)
          past[j] = live[j] & (~0ull << ((B.start - j + C) / C & 63));
          any |= past[j];
          const int lo = (__ffsll((unsigned long long)past[j]) - 1) * C + j;
          const int hi = (63 - __clzll((long long)past[j])) * C + j;
          if (C == 1) {
            first = lo;
            last = hi;
          } else {
            first = past[j] && lo < first ? lo : first;
            last = past[j] && hi > last ? hi : last;
          }
        }
        ops.Cells(*this, P, B, live, s, diag, sp, gap);
        // the old first column leaves the band when the band's start moves
        // (nothing kept: the row is the last one)
        const bool moved = first - 1 != B.start;
#pragma unroll
        for (int j = 0; j < C; ++j) {
          const bool on = __builtin_amdgcn_inverse_ballot_w64(moved ? past[j] : live[j]);
          const int v = s[j] - gi, x = e[j] - ge;
          const int ve = v > x ? v : x;
          h[j] = on ? s[j] : kInitScore;
          e[j] = on ? ve : kInitScore;
        }
        const int columns = B.end - B.start;
        B.cells += columns - 1;
        B.widest = columns > B.widest ? columns : B.widest;
        ++B.row;
        // the band's end: a pruned column behind the last live one, unless
        // the query side ends there (after a band that shrinks: at the old
        // end)
        const int after = last + 1;
        const int ends = (last_rel - (after > B.end ? after : B.end)) >> 31;  // -1: no column
        B.bare = (ends & (after - B.end)) >> 31;
        B.start = first - 1;
        B.end = after + 1 + ends;
        B.d = dn;
#pragma unroll
        for (int j = 0; j < C; ++j) score[j] = next[j];
        // the loop's exits: nothing kept, the database's delimiter, no room,
        // or a diagonal to clear
        stop = ((int)(dn ^ P.delim) - 1) | (room - B.end) | B.bare;
        if (any == 0) stop = -1;
        ops.End(*this, B, any != 0);
      } while (stop >= 0);
      if (any == 0 || B.d == P.delim) return kWaveDpDone;
    }
  }

  // Takes over the row of a window of C / 2 columns per lane: column c of the
  // window moves from lane c / (C / 2) to lane c / C.
  __device__ __forceinline__ void Widen(const WaveDpParams &P, WaveDpBand &B,
                                        const WaveDp<kReverse, C / 2> &x) {
    constexpr int H = C / 2;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int from = 2 * Lane() + j / H;
      const bool inside = from < kWave;
      const int at = 4 * (inside ? from : 0);
      const int vh = __builtin_amdgcn_ds_bpermute(at, x.h[j % H]);
      const int ve = __builtin_amdgcn_ds_bpermute(at, x.e[j % H]);
      const int vc = __builtin_amdgcn_ds_bpermute(at, x.code[j % H]);
      h[j] = inside ? vh : kInitScore;
      e[j] = inside ? ve : kInitScore;
      code[j] = inside ? vc : kWallCode;
    }
    ReadWindow(P, B, kWave * H);
    Limits(B);
  }

  // Goes on from a narrower window that ended with r: at its row, or from the
  // seed when it lost that row.
  __device__ __forceinline__ int TakeOver(const WaveDpParams &P, WaveDpBand &B,
                                          const WaveDp<kReverse, C / 2> &x, int r, uint32_t q,
                                          uint32_t dp) {
    if (r != kWaveDpWiden) return Begin(P, B, q, dp);
    Widen(P, B, x);
    return 0;
  }
};

// No operations recorded.
struct NoOps {
  __device__ __forceinline__ bool Row(const WaveDpBand &) { return true; }
  template <class Dp, int C>
  __device__ __forceinline__ void Cells(const Dp &, const WaveDpParams &, const WaveDpBand &,
                                        const uint64_t (&)[C], const int (&)[C],
                                        const int (&)[C], const int (&)[C], const int (&)[C]) {}
  template <class Dp>
  __device__ __forceinline__ void End(const Dp &, const WaveDpBand &, bool) {}
};

constexpr int kWaveDpBlock = 256;

// Jobs out of the first ring up to which they run one wave per job: beyond,
// the 64-column ring's lanes fill the chip.
constexpr uint32_t kWaveDpJobs = 1u << 16;
constexpr uint32_t kWaveDpWaves = 8192;  // resident at once: 8 per SIMD

// The jobs of a block of the one-wave-per-job form: block b of B has jobs b,
// b + B, b + 2 B, ... (an order by length spreads evenly), which its waves
// take one by one from a counter in LDS.  Blocks that end early leave their
// issue slots to the others of the CU.  A counter in memory that all waves
// share costs 12 ns a request, and every wave makes at least the one that finds
// no job: 10,000 read extensions took 135 us with it and take 58 so, 45,000
// 539 and 180; with a quarter of the jobs left to such a counter 135 and 197.
struct BlockJobs {
  uint32_t *next;  // in LDS
  uint32_t k;
  // by every thread, before the block's next barrier
  __device__ __forceinline__ void Begin(uint32_t *lds_next) {
    next = lds_next;
    k = Uniform(threadIdx.x / kWave);
    if (threadIdx.x == 0) *next = blockDim.x / kWave;
  }
  // the wave's job, or one past the jobs
  __device__ __forceinline__ uint64_t Job(uint32_t block, uint32_t blocks) const {
    return (uint64_t)block + (uint64_t)k * blocks;
  }
  __device__ __forceinline__ void Advance() {
    uint32_t v = 0;
    if (__lane_id() == 0) v = atomicAdd(next, 1u);
    k = Uniform(v);
  }
};

// One wave per job: jobs k (order[k] when `order` is set), or the
// *list_count jobs of `list` when that is set and they are at most
// kWaveDpJobs.  A job whose band outgrows 64 kMostColumns columns is appended
// to overflow_list; narrow_count and wide_count (either may be null) count
// those past narrow_columns and past 64 columns.
template <bool kReverse, int kMostColumns>
__global__ void __launch_bounds__(kWaveDpBlock)
    GappedRowKernel(uint32_t n, const uint32_t *list, const uint32_t *list_count,
                    const uint32_t *order, uint32_t limit, WaveDpParams P, const int *matrix,
                    uint32_t nl, uint32_t *qpos, uint32_t *dpos, int *scores, uint32_t *cells,
                    uint32_t *overflow_count, uint32_t *overflow_list, int narrow_columns,
                    uint32_t *narrow_count, uint32_t *wide_count, uint32_t *failed) {
  __shared__ int8_t sm[kTableDim * kScoreStride];
  __shared__ uint32_t next, counts[2];
  if (list) {
    n = Uniform(*list_count);
    if (n > kWaveDpJobs) return;
  }
  if (blockIdx.x >= n) return;  // no job for the block
  BlockJobs jobs;
  jobs.Begin(&next);
  if (threadIdx.x < 2) counts[threadIdx.x] = 0;
  StageWaveDpScores(sm, matrix, nl);
  __syncthreads();
  const int inc = kReverse ? -1 : 1;
  const bool leads = __lane_id() == 0;
  for (uint64_t k; (k = jobs.Job(blockIdx.x, gridDim.x)) < n; jobs.Advance()) {
    const uint32_t i = Uniform(list ? list[k] : order ? order[k] : (uint32_t)k);
    if (i >= limit) {  // an order entry out of range: counted, never read
      if (leads) atomicAdd(failed, 1u);
      continue;
    }
    const uint32_t q = Uniform(qpos[i]), d = Uniform(dpos[i]);
    WaveDpBand B;
    WaveDp<kReverse, 1> x;
    NoOps none;
    int r = x.Begin(P, B, q, d);
    if (r == 0) r = x.Rows(P, sm, B, none);
    if constexpr (kMostColumns == 2) {
      if (r == kWaveDpWiden) {
        WaveDp<kReverse, 2> y;
        y.Widen(P, B, x);
        r = y.Rows(P, sm, B, none);
      }
    } else if (r != kWaveDpDone) {
      WaveDp<kReverse, 2> y;
      r = y.TakeOver(P, B, x, r, q, d);
      if (r == 0) r = y.Rows(P, sm, B, none);
      if (r != kWaveDpDone) {
        WaveDp<kReverse, 4> z;
        r = z.TakeOver(P, B, y, r, q, d);
        if (r == 0) r = z.Rows(P, sm, B, none);
      }
    }
    if (leads) {
      const bool done = r == kWaveDpDone;
      if (done) {
        scores[i] = B.best;
        qpos[i] = (uint32_t)((int)q + (B.best_col - 1) * inc);
        dpos[i] = (uint32_t)((int)d + B.best_row * inc);
        if (cells) cells[i] = (uint32_t)B.cells;
      } else {
        overflow_list[atomicAdd(overflow_count, 1u)] = i;
      }
      if (!done || B.widest > narrow_columns) atomicAdd(&counts[0], 1u);
      if (!done || B.widest > 64) atomicAdd(&counts[1], 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (narrow_count && counts[0]) atomicAdd(narrow_count, counts[0]);
    if (wide_count && counts[1]) atomicAdd(wide_count, counts[1]);
  }
}

// Blocks of a GappedRowKernel launch over at most `jobs` jobs: as many waves
// as jobs up to the resident ones.
inline uint32_t WaveDpBlocksFor(size_t jobs) {
  const size_t per = kWaveDpBlock / kWave;
  const size_t waves = jobs < kWaveDpWaves ? (jobs > 0 ? jobs : 1) : (size_t)kWaveDpWaves;
  return (uint32_t)((waves + per - 1) / per);
}

}  // namespace gz
