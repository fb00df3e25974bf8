// traceback.hip -- the result build (AlignerBuildResultsThread) on the device.
//
// For every presearched result the reference re-extends both sides with the
// result cutoff and a traceback (GappedExtender::ExtendOneSide with
// EditBlocks, src/gapped_extender.cpp:70-304,473-531), then counts length,
// mismatches and gap openings / extensions over the joined edit script
// (AlignerCommon::BuildResult, src/aligner_common.h:276-343).  One wave runs
// one side of a result (TracebackWaveKernel: the DP of wave_dp.h with the
// operations recorded); a lane runs a result where that form does not serve
// (TracebackKernel).  The op store follows the reference's gap_states_ layout:
// rows are laid back to back in one byte arena ([0] holds the first op, row r
// starts where row r-1 ends), so the traceback's reads outside a row's band
// see the same neighbouring bytes.  Cells an extension does not write hold a
// marker; reading one (or reading outside the written range) means the
// reference would have read a byte left by an earlier extension, and the
// result is flagged so the host replays the chunk in the reference order.
// Results whose op rows exceed the arena are flagged for the host as well.
#include <hip/hip_runtime.h>

#include <climits>

#include <algorithm>

#include "gz_common.h"
#include "gz_device.h"
#include "gz_runtime.h"
#include "traceback.h"
#include "ungapped.h"
#include "wave_dp.h"

namespace gz {

namespace {

constexpr uint8_t kSub = 0, kGap0 = 1, kGap1 = 2, kExt0 = 4, kExt1 = 8;
constexpr uint8_t kEditGap0 = 0, kEditSub = 1, kEditGap1 = 2;
constexpr uint8_t kUnwritten = 0xFF;
constexpr int kTbThreads = 64;
// Query sides of up to kTbLdsCols - 2 residues keep their DP columns in LDS,
// column-major over the block's lanes ([column][lane]): 16-bit cells (16 KB
// per block) when the cutoff and gap costs allow them, else 32-bit ones.
constexpr uint32_t kTbLdsCols = 64;
constexpr int kTbLow = -16384;

__shared__ int2 tb_dp[kTbLdsCols * kTbThreads];
// 16-bit columns.  Exact when the cutoff is at most 8192 and gap open +
// extension at most 1024 (the launch checks): a side of at most 62 residues
// scores at most 62 x 127, and values stored below -16384 (the band's first
// gap column keeps decreasing) are clamped there, which changes no comparison
// and no recorded op, since every value compared with them is above
// -16384 + the gap extension.
__shared__ short2 tb_dp16[kTbLdsCols * kTbThreads];
// The query side's codes by DP column: column a (a >= 1) holds the code at
// q0 + (a - 1) inc, the delimiter closing the side included.
__shared__ uint8_t tb_qc[kTbLdsCols * kTbThreads];

// DP column access: the lane's LDS column set (32- or 16-bit cells), or its
// global scratch.
template <bool kLds, bool kShort>
struct DpCells {
  int2 *global;
  __device__ __forceinline__ int2 Get(int i) const {
    if constexpr (kLds && kShort) {
      const short2 v = tb_dp16[i * kTbThreads + (int)threadIdx.x];
      return make_int2(v.x, v.y);
    } else if constexpr (kLds) {
      return tb_dp[i * kTbThreads + (int)threadIdx.x];
    } else {
      return global[i];
    }
  }
  __device__ __forceinline__ void Set(int i, int2 v) const {
    if constexpr (kLds && kShort) {
      tb_dp16[i * kTbThreads + (int)threadIdx.x] =
          make_short2((short)(v.x > kTbLow ? v.x : kTbLow), (short)(v.y > kTbLow ? v.y : kTbLow));
    } else if constexpr (kLds) {
      tb_dp[i * kTbThreads + (int)threadIdx.x] = v;
    } else {
      global[i] = v;
    }
  }
};

struct Lane {
  int2 *dp;
  uint8_t *arena;
  int2 *rows;  // (base, off)
  uint8_t *ops;
  uint32_t dp_cap, arena_cap, row_cap, op_cap;
};

struct Side {
  int score, p0, p1;
  uint32_t nops;  // ops generated (traceback order), in ops[base ..)
};

__device__ __forceinline__ uint32_t CodeAt(const uint64_t *packed, int64_t pos) {
  return PackedCodeAt(packed, (uint32_t)pos);
}

// GappedExtender::ExtendOneSide with traceback (the DP and band bookkeeping
// after the delimiter checks); ops are generated from the best cell back to
// the origin.  Returns flags (kTracebackStale/Overflow).
template <bool kLds, bool kShort>
__device__ __forceinline__ uint32_t ExtendBody(const uint64_t *pq, int64_t q0, uint32_t s0len,
                                               const uint64_t *pd, int64_t d0, int inc,
                                               const int8_t *sm, int gap_open, int gap_ext,
                                               int cutoff, Lane &L, uint32_t op_base,
                                               Side *out) {
  const DpCells<kLds, kShort> dp{L.dp};
  // the query code at q0 + p, p = (a - 1) inc for DP column a
  auto qcode = [&](int p) -> uint32_t {
    if constexpr (kLds) return tb_qc[(p * inc + 1) * kTbThreads + (int)threadIdx.x];
    else return CodeAt(pq, q0 + p);
  };
  const uint32_t extra =
      (gap_ext > 0 && cutoff != INT_MAX) ? (uint32_t)(cutoff / gap_ext + 3) : s0len + 3;
  uint32_t used = 0;
  int64_t written = 0;  // highest arena index written
  {
    const uint32_t l = extra + extra / 3;
    if ((uint64_t)used + l >= L.arena_cap) return kTracebackOverflow;
  }
  L.arena[0] = kSub;
  const int gi = gap_open + gap_ext;
  int as = 0, ae = 0, ai = 0, last = 0;
  int score = -gi;
  dp.Set(0, make_int2(0, -gi));
  int p0 = 0;
  for (ai = 1; qcode(p0) != kDelimiter; ++ai, p0 += inc) {
    if (score < -cutoff) break;
    dp.Set(ai, make_int2(score, score - gi));
    score -= gap_ext;
  }
  if (qcode(p0) != kDelimiter) {
    dp.Set(ai, make_int2(kInitScore, kInitScore));
    ae = ai + 1;
  } else {
    ae = ai;
  }
  int max_score = 0, mp0 = -inc, mp1 = -inc;
  uint32_t nrows = 0;
  uint32_t c1_next = CodeAt(pd, d0);
  for (int p1 = 0;; p1 += inc) {
    const uint32_t c1 = c1_next;
    if (c1 == kDelimiter) break;
    // the next row's code, read ahead (in bounds: c1 is a residue)
    c1_next = CodeAt(pd, d0 + p1 + inc);
    const uint32_t length = gap_ext > 0 ? (uint32_t)(ae - as) + extra : extra - (uint32_t)as;
    const uint32_t l = length + length / 3;
    if ((uint64_t)used + l >= L.arena_cap || nrows >= L.row_cap) return kTracebackOverflow;
    const int base = (int)used + 1;
    const int off = as;
    L.rows[nrows++] = make_int2(base, off);
    const int zero = base - off;
    const int8_t *row = sm + c1 * kTableDim;
    p0 = as * inc;
    int prev = dp.Get(as).x;
    {
      int2 c = dp.Get(as);
      c.x = (max_score - c.y > cutoff) ? kInitScore : c.y;
      dp.Set(as, make_int2(c.x, c.y - gap_ext));
    }
    int gap_row = dp.Get(as).x - gi;
    L.arena[zero + as] = kGap0 + kExt0;
    written = max(written, (int64_t)(zero + as));
    last = as;
    for (ai = as + 1; ai < ae; ++ai, p0 += inc) {
      int s = prev + row[qcode(p0)];
      const int2 cell = dp.Get(ai);
      prev = cell.x;
      int gap_col = cell.y;
      uint8_t op = kSub;
      if (s < gap_col) {
        op = kGap0;
        s = gap_col;
      }
      if (s < gap_row) {
        op = kGap1;
        s = gap_row;
      }
      if (max_score - s > cutoff) {
        if (as + 1 == ai) ++as;
        dp.Set(ai, make_int2(kInitScore, kInitScore));
        gap_row = kInitScore;
        L.arena[zero + ai] = kUnwritten;
      } else {
        last = ai;
        if (s > max_score) {
          max_score = s;
          mp0 = p0;
          mp1 = p1;
        }
        gap_col -= gap_ext;
        gap_row -= gap_ext;
        int gap_keep;
        if (gap_col < s - gi) {
          gap_keep = s - gi;
        } else {
          gap_keep = gap_col;
          op += kExt0;
        }
        if (gap_row < s - gi) gap_row = s - gi; else op += kExt1;
        L.arena[zero + ai] = op;
        dp.Set(ai, make_int2(s, gap_keep));
      }
      written = max(written, (int64_t)(zero + ai));
    }
    if (as + 1 == ae) break;
    if (last < ae - 1) {
      ae = last + 1;
    } else {
      while (gap_row >= (max_score - cutoff) && qcode(p0) != kDelimiter) {
        dp.Set(ae, make_int2(gap_row, gap_row - gi));
        L.arena[zero + ae] = kGap0 + kExt0;
        written = max(written, (int64_t)(zero + ae));
        gap_row -= gap_ext;
        ++ae;
        p0 += inc;
      }
    }
    if (qcode(p0) != kDelimiter) {
      dp.Set(ae, make_int2(kInitScore, kInitScore));
      L.arena[zero + ae] = kUnwritten;
      written = max(written, (int64_t)(zero + ae));
      ++ae;
    }
    used += (uint32_t)(ae - off);
  }
  out->score = max_score;
  out->p0 = mp0;
  out->p1 = mp1;
  // PickOptimalPath: generated from the best cell back to the origin
  uint32_t flags = 0;
  uint32_t n = op_base;
  int q = mp0, d = mp1;
  uint8_t op = kSub;
  auto emit = [&](uint8_t e, int count) {
    for (int k = 0; k < count; ++k) {
      if (n >= L.op_cap) {
        flags |= kTracebackOverflow;
        return;
      }
      L.ops[n++] = e;
    }
  };
  while (d * inc >= 0 && q * inc >= 0) {
    const int r = d * inc;
    const int2 rb = L.rows[r];
    const int64_t idx = (int64_t)rb.x + q * inc - rb.y + 1;
    uint8_t next = 0;
    if (idx < 0 || idx > written) {
      flags |= kTracebackStale;
    } else {
      next = L.arena[idx];
      if (next == kUnwritten) {
        flags |= kTracebackStale;
        next = 0;
      }
    }
    if (op == kGap0) {
      op = next & 3;
      if (next & kExt0) op = kGap0;
    } else if (op == kGap1) {
      op = next & 3;
      if (next & kExt1) op = kGap1;
    } else {
      op = next & 3;
    }
    if (op == kGap0) {
      emit(kEditGap0, 1);
      d -= inc;
    } else if (op == kGap1) {
      emit(kEditGap1, 1);
      q -= inc;
    } else {
      emit(kEditSub, 1);
      d -= inc;
      q -= inc;
    }
    if (flags & kTracebackOverflow) return flags;
  }
  if (d * inc >= 0) emit(kEditGap0, d * inc + 1);
  else if (q * inc >= 0) emit(kEditGap1, q * inc + 1);
  out->nops = n - op_base;
  return flags;
}

template <bool kShort>
__device__ uint32_t Extend(const uint64_t *pq, int64_t q0, uint32_t s0len, const uint64_t *pd,
                           int64_t d0, bool reversed, const int8_t *sm, int gap_open,
                           int gap_ext, int cutoff, Lane &L, uint32_t op_base, Side *out) {
  const int inc = reversed ? -1 : 1;
  out->score = 0;
  out->p0 = -inc;
  out->p1 = -inc;
  out->nops = 0;
  if (CodeAt(pq, q0) == kDelimiter || CodeAt(pd, d0) == kDelimiter) return 0;
  // n0 = residues before the delimiter, twelve codes per packed word pair;
  // the codes go to the side's LDS columns on the way.  A window starts at a
  // residue, so its words lie inside the padded array.
  uint32_t n0 = 0;
  bool found = false;
  for (uint32_t base = 0; !found; base += kCodesPerWord) {
    const uint32_t first =
        (uint32_t)(reversed ? q0 - (int64_t)base - (int64_t)(kCodesPerWord - 1)
                            : q0 + (int64_t)base) + kPackPadCodes;
    const uint32_t w = first / kCodesPerWord;
    const uint64_t win = Window12(pq[w] & kCodeBitsMask, pq[w + 1] & kCodeBitsMask,
                                  first - w * kCodesPerWord);
#pragma unroll
    for (int j = 0; j < (int)kCodesPerWord; ++j) {
      const uint32_t code =
          (uint32_t)(win >> (kCodeBits * (reversed ? (int)kCodesPerWord - 1 - j : j))) & 31u;
      if (!found) {
        const uint32_t a = base + (uint32_t)j + 1;
        if (a < kTbLdsCols) tb_qc[a * kTbThreads + threadIdx.x] = (uint8_t)code;
        if (code == kDelimiter) {
          found = true;
          n0 = base + (uint32_t)j;
        }
      }
    }
  }
  // columns 0 .. n0 + 1 are touched (the band may step one past the last
  // residue); s0len, the distance to the query's far end, can exceed n0 when
  // the query holds several frames
  if (n0 + 2 <= kTbLdsCols)
    return ExtendBody<true, kShort>(pq, q0, s0len, pd, d0, inc, sm, gap_open, gap_ext, cutoff,
                                    L, op_base, out);
  if (max(s0len + 1, n0 + 2) > L.dp_cap) return kTracebackOverflow;
  return ExtendBody<false, false>(pq, q0, s0len, pd, d0, inc, sm, gap_open, gap_ext, cutoff,
                                  L, op_base, out);
}

template <bool kShort>
__global__ void __launch_bounds__(kTbThreads)
    TracebackKernel(const uint64_t *pq, const uint64_t *pd, const TracebackJob *jobs,
                    uint32_t n, const uint32_t *list, const int *matrix, uint32_t nl,
                    int gap_open, int gap_ext, int cutoff, uint8_t *scratch, LaneCaps caps,
                    TracebackOut *outs) {
  __shared__ int8_t sm[kTableDim * kTableDim];
  StageScoreTable(sm, matrix, nl);
  __syncthreads();
  const uint32_t lane_id = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lanes = gridDim.x * blockDim.x;
  Lane L;
  uint8_t *mine = scratch + (size_t)lane_id * caps.bytes_per_lane;
  L.dp = reinterpret_cast<int2 *>(mine);
  L.rows = reinterpret_cast<int2 *>(mine + caps.dp * sizeof(int2));
  L.arena = mine + (caps.dp + caps.rows) * sizeof(int2);
  L.ops = L.arena + caps.arena;
  L.dp_cap = caps.dp;
  L.row_cap = caps.rows;
  L.arena_cap = caps.arena;
  L.op_cap = caps.ops;
  for (uint32_t k = lane_id; k < n; k += lanes) {
    const uint32_t j = list ? list[k] : k;
    const TracebackJob job = jobs[j];
    TracebackOut o = {};
    Side rev, fwd;
    // reverse side from (hit - 1), forward side from the hit
    uint32_t flags = Extend<kShort>(pq, (int64_t)job.query_offset + job.hit_q - 1, job.hit_q - 1, pd,
                            (int64_t)job.hit_d - 1, true, sm, gap_open, gap_ext, cutoff, L, 0,
                            &rev);
    if (!(flags & kTracebackOverflow))
      flags |= Extend<kShort>(pq, (int64_t)job.query_offset + job.hit_q, job.query_length - job.hit_q,
                      pd, (int64_t)job.hit_d, false, sm, gap_open, gap_ext, cutoff, L, rev.nops,
                      &fwd);
    o.flags = flags;
    if (!(flags & kTracebackOverflow)) {
      o.score = rev.score + fwd.score;
      o.start_q = job.hit_q - 1 + rev.p0;
      o.start_d = job.hit_d - 1 + rev.p1;
      o.end_q = job.hit_q + fwd.p0;
      o.end_d = job.hit_d + fwd.p1;
      // the joined script: both generated sequences reversed, reverse side first
      uint32_t qp = o.start_q, dp = o.start_d, m = 0, op_open = 0, ext = 0, len = 0;
      uint8_t prev = kEditSub;
      for (int part = 0; part < 2; ++part) {
        const uint32_t b = part == 0 ? 0 : rev.nops;
        const uint32_t cnt = part == 0 ? rev.nops : fwd.nops;
        for (uint32_t k = cnt; k-- > 0;) {
          const uint8_t e = L.ops[b + k];
          if (e == kEditSub) {
            if (CodeAt(pq, (int64_t)job.query_offset + qp) != CodeAt(pd, dp)) ++m;
            ++qp;
            ++dp;
          } else if (e == kEditGap0) {
            if (prev != kEditGap0) ++op_open; else ++ext;
            ++dp;
          } else {
            if (prev != kEditGap1) ++op_open; else ++ext;
            ++qp;
          }
          prev = e;
          ++len;
        }
      }
      o.length = len;
      o.mismatches = m;
      o.gap_openings = op_open;
      o.gap_extensions = ext;
    }
    outs[j] = o;
  }
}

// ---------------------------------------------------------------------------
// one wave per side
// ---------------------------------------------------------------------------
// What a side's wave leaves for its result.
struct TracebackHalf {
  int score;
  uint32_t q, d;  // where the extension ends
  uint32_t length, mismatches, gap_openings, gap_extensions;
  uint32_t flags;  // kTracebackStale / Overflow / kNeedsLane
};
constexpr uint32_t kNeedsLane = 4;

constexpr int kTbWaveBlock = 256;
// Results of one call from which sides that fit the lanes' LDS columns take a
// lane each again, where the lanes' scratch (11 GB) is kept: on read results a
// call takes 24 ns each on waves, and 1.4 ms and 13 ns each on lanes (843,199
// in one call: 20.3 ms on waves, 12.5 on lanes).
constexpr uint32_t kLaneResults = 131072;
// Waves resident at once: four per SIMD, enough to hide a row's dependent
// steps behind the other waves' instructions.
constexpr uint32_t kTbWaves = 4096;

struct WaveCaps {
  uint32_t arena, rows, ops;     // a wave's bytes of the arena, rows, ops
  uint32_t max_rows, max_query;  // rows the side may have, longest query
  uint32_t stride;               // bytes per wave
};

// Records the operations of WaveDp's rows in the reference's layout.  A row's
// cells past its new band end are overwritten by the following rows or never
// read but as unwritten, so a row stores the columns [start, new end) only
// and every byte has one writer.  The horizontal gap lacks the reference's
// reset after a pruned cell, so kExt1 of a kept cell may be set where the
// reference's is not.  No path reads it there: a path comes to a cell in a
// horizontal gap only from the cell's right neighbour in the same row, and the
// gap into that neighbour is at least the running best less the cutoff, which
// a gap through a pruned cell is below.
struct ArenaOps {
  uint8_t *arena;
  int2 *rows;  // (base, off)
  uint32_t max_rows, extra;
  int gap_init, gap_ext;
  uint32_t used = 0;
  int start = 0;  // the row's first column in the window
  bool full = false;
  int op[4];

  static __device__ __forceinline__ uint32_t Need(uint32_t length) { return length + length / 3; }

  __device__ __forceinline__ bool Row(const WaveDpBand &B) {
    const uint32_t as = (uint32_t)(B.base + B.start);
    const uint32_t length = gap_ext > 0 ? (uint32_t)(B.end - B.start) + extra : extra - as;
    if ((uint64_t)used + Need(length) >= kTracebackArena || (uint32_t)B.row >= max_rows) {
      full = true;
      return false;
    }
    if (__lane_id() == 0) rows[B.row] = make_int2((int)used + 1, (int)as);
    start = B.start;
    return true;
  }

  template <class Dp, int C>
  __device__ __forceinline__ void Cells(const Dp &dp, const WaveDpParams &P, const WaveDpBand &B,
                                        const uint64_t (&live)[C], const int (&s)[C],
                                        const int (&diag)[C], const int (&sp)[C],
                                        const int (&gap)[C]) {
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int a = Dp::Offset(j), opened = s[j] - gap_init;
      int x = diag[j] < dp.e[j] ? kGap0 : kSub;
      x = sp[j] < gap[j] ? kGap1 : x;
      x += dp.e[j] - gap_ext >= opened ? kExt0 : 0;
      x += gap[j] - gap_ext >= opened ? kExt1 : 0;
      // the band's first column and those a row's gap appends
      const bool fixed = a == B.start || a >= B.end;
      x = fixed ? kGap0 + kExt0 : x;
      const bool kept = __builtin_amdgcn_inverse_ballot_w64(live[j]) || a == B.start;
      op[j] = kept ? x : kUnwritten;
    }
  }

  template <class Dp>
  __device__ __forceinline__ void End(const Dp &, const WaveDpBand &B, bool any) {
    constexpr int C = Dp::W / kWave;
    // nothing kept: the side's last row; only its first column can be read
    const int columns = any ? B.end - start : 1;
    uint8_t *row = arena + used + 1;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int k = Dp::Offset(j) - start;
      if (k >= 0 && k < columns) row[k] = (uint8_t)op[j];
    }
    used += (uint32_t)columns;
  }
};

// One side: q0 / d0 the positions of its first residues, s0len the distance
// to the query's end.
template <bool kReverse>
__device__ void WaveSide(const WaveDpParams &P, const int8_t *sm, uint32_t q0, uint32_t s0len,
                         uint32_t d0, uint8_t *mine, const WaveCaps &caps, TracebackHalf *out) {
  const int lane = (int)__lane_id();
  ArenaOps ops;
  ops.arena = mine;
  ops.rows = reinterpret_cast<int2 *>(mine + caps.arena);
  ops.max_rows = caps.max_rows;
  ops.gap_init = P.gap_init;
  ops.gap_ext = P.gap_ext;
  ops.extra = P.gap_ext > 0 ? (uint32_t)(P.cutoff / P.gap_ext + 3) : s0len + 3;
  uint8_t *script = mine + caps.arena + caps.rows;
  TracebackHalf h = {};
  // a window of 64 columns serves a query side that ends inside it, wider
  // ones a band that moves along its query side
  WaveDpBand B;
  WaveDp<kReverse, 1> x;
  int r = x.Begin(P, B, q0, d0);
  const bool begun = r != kWaveDpDone;
  if (begun && ArenaOps::Need(ops.extra) >= kTracebackArena) {
    h.flags = kTracebackOverflow;
    if (lane == 0) *out = h;
    return;
  }
  if (begun) {
    if (r == 0 && x.EndsInside(B)) {
      r = x.Rows(P, sm, B, ops);
    } else {
      WaveDp<kReverse, 2> y;
      r = y.Begin(P, B, q0, d0);
      if (r == 0) r = y.Rows(P, sm, B, ops);
      if (r != kWaveDpDone && !ops.full) {
        // a lost row's side starts again, its operations with it
        WaveDp<kReverse, 4> z;
        if (r == kWaveDpLost) ops.used = 0;
        r = z.TakeOver(P, B, y, r, q0, d0);
        if (r == 0) r = z.Rows(P, sm, B, ops);
      }
    }
  }
  if (r != kWaveDpDone) {
    h.flags = ops.full ? kTracebackOverflow : kNeedsLane;
    if (lane == 0) *out = h;
    return;
  }
  if (lane == 0) ops.arena[0] = kSub;
  // the wave's stores are read by its other lanes from here on
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  // the path from the best cell back: while the state (a substitution run, a
  // vertical or a horizontal gap) lasts, lane l looks l cells ahead
  const int best_row = B.best_row, best_col = B.best_col;
  int row = best_row, col = best_col, state = kSub;
  uint32_t nops = 0;
  while (row >= 0 && col >= 1) {
    const int lr = row - (state != kGap1 ? lane : 0), lc = col - (state != kGap0 ? lane : 0);
    const bool on = lr >= 0 && lc >= 1;
    int byte = 0;
    bool stale = false;
    if (on) {
      const int2 at = ops.rows[lr];
      const int idx = at.x + lc - at.y;
      stale = idx < 0 || idx > (int)ops.used;
      if (!stale) {
        byte = ops.arena[idx];
        stale = byte == kUnwritten;
        byte = stale ? 0 : byte;
      }
    }
    const bool go = on && (state == kSub ? (byte & 3) == 0
                                         : (byte & (state == kGap0 ? kExt0 : kExt1)) != 0);
    const uint64_t stops = __ballot(!go), inside = __ballot(on);
    const int f = stops ? __ffsll((unsigned long long)stops) - 1 : kWave;
    const bool turns = f < kWave && ((inside >> f) & 1ull) != 0;
    // the cells that the path visits
    const uint64_t seen = f >= kWave - 1 ? ~0ull : (2ull << f) - 1ull;
    if (__ballot(stale) & seen) h.flags |= kTracebackStale;
    const int next = turns ? __builtin_amdgcn_readlane(byte, f) & 3 : 0;
    auto edit = [](int op) { return op == kGap0 ? kEditGap0 : op == kGap1 ? kEditGap1 : kEditSub; };
    if (lane < f || (lane == f && turns)) script[nops + lane] = edit(lane < f ? state : next);
    row -= state != kGap1 ? f : 0;
    col -= state != kGap0 ? f : 0;
    nops += (uint32_t)f;
    if (turns) {
      ++nops;
      row -= next != kGap1 ? 1 : 0;
      col -= next != kGap0 ? 1 : 0;
      state = next;
    }
  }
  const int tail = row >= 0 ? row + 1 : col >= 1 ? col : 0;
  for (int k = lane; k < tail; k += kWave) script[nops + k] = row >= 0 ? kEditGap0 : kEditGap1;
  nops += (uint32_t)tail;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  // The joined script holds both generated sequences reversed, the reverse
  // side's first: each side's counts stand alone, since a side consumes
  // exactly its stretch of both sequences and the reverse side's last op (its
  // first generated one, at the best cell) is never a gap.
  const int inc = kReverse ? -1 : 1;
  h.score = B.best;
  h.q = q0 + (uint32_t)((best_col - 1) * inc);
  h.d = d0 + (uint32_t)(best_row * inc);
  uint32_t q = kReverse ? h.q : q0, d = kReverse ? h.d : d0;
  uint64_t last0 = 0, last1 = 0;  // whether the pass before ended in a gap
  const uint64_t below = (1ull << lane) - 1ull;
  for (uint32_t k = 0; k < nops; k += kWave) {
    const bool on = k + (uint32_t)lane < nops;
    const int e = on ? script[nops - 1 - k - (uint32_t)lane] : -1;
    const uint64_t subs = __ballot(e == kEditSub), gap0 = __ballot(e == kEditGap0),
                   gap1 = __ballot(e == kEditGap1);
    bool differs = false;
    if (e == kEditSub)
      differs = CodeAt(P.queries, q + (uint32_t)__popcll((subs | gap1) & below)) !=
                CodeAt(P.database, d + (uint32_t)__popcll((subs | gap0) & below));
    h.mismatches += (uint32_t)__popcll(__ballot(differs));
    const uint32_t opens = (uint32_t)(__popcll(gap0 & ~(gap0 << 1 | last0)) +
                                      __popcll(gap1 & ~(gap1 << 1 | last1)));
    h.gap_openings += opens;
    h.gap_extensions += (uint32_t)(__popcll(gap0) + __popcll(gap1)) - opens;
    last0 = gap0 >> 63;
    last1 = gap1 >> 63;
    q += (uint32_t)__popcll(subs | gap1);
    d += (uint32_t)__popcll(subs | gap0);
  }
  h.length = nops;
  if (lane == 0) *out = h;
}

// Sides of the jobs, one wave each: blocks of even index the reverse sides
// (from hit - 1), of odd index the forward sides.  A wave takes `batch` jobs
// at a time, its first without asking, the others from heads[direction]
// (zero at the launch).
//
// Bound: the issue of a row's instructions (with the operations about 120,
// against 90 without), then the path's dependent loads, a table entry and an
// op per run of equal operations.  A call with its copies and without
// allocations, against a lane per result that walks the cells one by one with
// its op rows strided over the chip's memory: 50,021 results of reads 5.9 ->
// 1.34 ms (1.18 of it this kernel), 3,001 of proteins of 100-500 residues 26 ->
// 0.64 ms; at cutoffs of 90 and 120 the latter 48 -> 0.92 and 63 -> 63 ms
// (bands past 256 columns take a lane each).
__global__ void __launch_bounds__(kTbWaveBlock)
    TracebackWaveKernel(WaveDpParams P, const TracebackJob *jobs, uint32_t n, uint32_t batch,
                        uint32_t *heads, const int *matrix, uint32_t nl, uint8_t *scratch,
                        WaveCaps caps, TracebackHalf *halves) {
  __shared__ int8_t sm[kTableDim * kScoreStride];
  StageWaveDpScores(sm, matrix, nl);
  __syncthreads();
  const uint32_t side = blockIdx.x & 1u, per = kTbWaveBlock / kWave;
  const uint32_t in_block = Uniform(threadIdx.x / kWave);
  const uint32_t wave = (blockIdx.x >> 1) * per + in_block;
  const uint32_t waves = (gridDim.x >> 1) * per;
  uint8_t *mine = scratch + (size_t)(blockIdx.x * per + in_block) * caps.stride;
  for (uint32_t first = wave * batch; first < n;) {
    const uint32_t stop = first + batch < n ? first + batch : n;
    for (uint32_t j = first; j < stop; ++j) {
      const uint32_t offset = Uniform(jobs[j].query_offset), length = Uniform(jobs[j].query_length);
      const uint32_t hit_q = Uniform(jobs[j].hit_q), hit_d = Uniform(jobs[j].hit_d);
      TracebackHalf *out = halves + 2 * (size_t)j + side;
      // the buffers hold any side between the query's two delimiters
      const bool framed = hit_q >= 1 && hit_q < length && length <= caps.max_query &&
                          CodeAt(P.queries, offset) == kDelimiter &&
                          CodeAt(P.queries, (int64_t)offset + length - 1) == kDelimiter;
      if (!Uniform(framed ? 1 : 0)) {
        if (__lane_id() == 0) {
          TracebackHalf h = {};
          h.flags = kNeedsLane;
          *out = h;
        }
      } else if (side == 0) {
        WaveSide<true>(P, sm, offset + hit_q - 1, hit_q - 1, hit_d - 1, mine, caps, out);
      } else {
        WaveSide<false>(P, sm, offset + hit_q, length - hit_q, hit_d, mine, caps, out);
      }
    }
    if ((uint64_t)waves * batch >= n) break;  // no jobs past the first ones
    uint32_t b = 0;
    if (__lane_id() == 0) b = atomicAdd(&heads[side], batch);
    first = waves * batch + Uniform(b);
  }
}

// Both sides' halves as results; jobs that a wave could not serve are listed.
__global__ void __launch_bounds__(256)
    TracebackJoinKernel(const TracebackJob *jobs, uint32_t n, const TracebackHalf *halves,
                        TracebackOut *outs, uint32_t *count, uint32_t *list) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const TracebackHalf rev = halves[2 * (size_t)j], fwd = halves[2 * (size_t)j + 1];
  if ((rev.flags | fwd.flags) & kNeedsLane) {
    list[atomicAdd(count, 1u)] = j;
    return;
  }
  TracebackOut o = {};
  o.flags = rev.flags | (rev.flags & kTracebackOverflow ? 0u : fwd.flags);
  if (!(o.flags & kTracebackOverflow)) {
    const uint32_t offset = jobs[j].query_offset;
    o.score = rev.score + fwd.score;
    o.start_q = rev.q - offset;
    o.start_d = rev.d;
    o.end_q = fwd.q - offset;
    o.end_d = fwd.d;
    o.length = rev.length + fwd.length;
    o.mismatches = rev.mismatches + fwd.mismatches;
    o.gap_openings = rev.gap_openings + fwd.gap_openings;
    o.gap_extensions = rev.gap_extensions + fwd.gap_extensions;
  }
  outs[j] = o;
}

__global__ void ClearKernel(uint32_t *p, uint32_t n) {
  if (threadIdx.x < n) p[threadIdx.x] = 0;
}

size_t Align256(size_t b) { return (b + 255) / 256 * 256; }

// A lane's scratch capacities.
LaneCaps TracebackCaps(uint32_t max_query_length, uint32_t max_subject_length) {
  LaneCaps c;
  c.dp = max_query_length + 4;
  c.rows = max_subject_length + 4;
  c.arena = kTracebackArena;
  c.ops = 2 * (max_query_length + max_subject_length) + 16;
  c.bytes_per_lane = Align256((size_t)(c.dp + c.rows) * sizeof(int2) + c.arena + c.ops);
  return c;
}

// Lanes of n results: those resident at once (up to seven 64-lane blocks per
// CU), within a 12 GB scratch budget.
size_t TracebackLanes(uint32_t n, const LaneCaps &caps) {
  const size_t budget = (size_t)12 << 30;
  const size_t lanes = std::min<size_t>(((size_t)n + 63) / 64 * 64, (size_t)7 * 64 * 256);
  return std::max<size_t>(64, std::min(lanes, budget / caps.bytes_per_lane / 64 * 64));
}

// A wave's: an arena that holds the rows a side can have, up to the limit.
WaveCaps TracebackWaveCaps(uint32_t max_query_length, uint32_t max_subject_length) {
  WaveCaps c;
  const uint64_t rows = (uint64_t)max_subject_length + 4, cols = (uint64_t)max_query_length + 4;
  c.max_rows = (uint32_t)rows;
  c.max_query = max_query_length;
  c.arena = (uint32_t)Align256(std::min<uint64_t>(kTracebackArena, rows * cols + 16));
  c.rows = (uint32_t)(rows * sizeof(int2));
  c.ops = (uint32_t)(rows + cols + 16);
  c.stride = (uint32_t)Align256((size_t)c.arena + c.rows + c.ops);
  return c;
}

}  // namespace

TracebackRunner::~TracebackRunner() {
  Release(&ws_, &cap_);
  Release(&lane_ws_, &lane_cap_);
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
}

void TracebackRunner::Release(void **p, size_t *capacity) {
  if (*p && pooled_) WorkspacePool::Give(*p, *capacity);
  else if (*p) (void)gz::Free(*p);
  *p = nullptr;
  *capacity = 0;
}

hipError_t TracebackRunner::Reserve(size_t bytes, void **p, size_t *capacity) {
  if (*capacity >= bytes) return hipSuccess;
  Release(p, capacity);
  hipError_t e;
  if (pooled_) {
    e = WorkspacePool::Take(bytes, p, capacity);
  } else {
    e = gz::Malloc(p, bytes);
    *capacity = bytes;
  }
  if (e != hipSuccess) {
    *p = nullptr;
    *capacity = 0;
  }
  return e;
}

hipError_t TracebackRunner::ReserveLanes(size_t before, size_t lanes, size_t bytes_per_lane,
                                         void **p, size_t *capacity) {
  for (;;) {
    const hipError_t e = Reserve(before + lanes * bytes_per_lane, p, capacity);
    if (e != hipErrorOutOfMemory || lanes <= 64) return e;
    (void)hipGetLastError();
    lanes = lanes / 2 / 64 * 64;
  }
}

hipError_t TracebackRunner::Lanes(const TracebackInputs &in, const TracebackJob *d_jobs,
                                  uint32_t n, const uint32_t *d_list, TracebackOut *d_outs,
                                  uint8_t *scratch, size_t bytes, hipStream_t s) {
  const LaneCaps caps = TracebackCaps(in.max_query_length, in.max_subject_length);
  const size_t lanes = std::min(TracebackLanes(n, caps), bytes / caps.bytes_per_lane / 64 * 64);
  const uint32_t blocks = (uint32_t)(lanes / kTbThreads);
  const bool short_cells =
      in.cutoff <= 8192 && in.gap_ext >= 0 && in.gap_open + in.gap_ext <= 1024;
  if (short_cells)
    hipLaunchKernelGGL(TracebackKernel<true>, dim3(blocks), dim3(kTbThreads), 0, s, in.queries,
                       in.database, d_jobs, n, d_list, in.matrix, in.nl, in.gap_open, in.gap_ext,
                       in.cutoff, scratch, caps, d_outs);
  else
    hipLaunchKernelGGL(TracebackKernel<false>, dim3(blocks), dim3(kTbThreads), 0, s, in.queries,
                       in.database, d_jobs, n, d_list, in.matrix, in.nl, in.gap_open, in.gap_ext,
                       in.cutoff, scratch, caps, d_outs);
  return hipGetLastError();
}

hipError_t TracebackRunner::Run(const TracebackInputs &in, const TracebackJob *jobs, uint32_t n,
                                TracebackOut *outs, hipStream_t s, float *kernel_ms) {
  if (n == 0) return hipSuccess;
  const hipError_t e = Queue(in, jobs, n, outs, s, kernel_ms);
  // after an error nothing of the call may still use the workspace
  if (e != hipSuccess) (void)hipStreamSynchronize(s);
  return e;
}

hipError_t TracebackRunner::Queue(const TracebackInputs &in, const TracebackJob *jobs, uint32_t n,
                                  TracebackOut *outs, hipStream_t s, float *kernel_ms) {
  for (hipEvent_t &x : ev_)
    if (!x) {
      const hipError_t c = hipEventCreate(&x);
      if (c != hipSuccess) return c;
    }
  // the wave form's rows of the longest subject must fit 32-bit offsets
  const bool many_short = !pooled_ && n > kLaneResults && in.longest_side + 2 <= kTbLdsCols;
  const bool waves = !many_short && WaveDpServes(in.cutoff, in.gap_open, in.gap_ext) &&
                     in.max_subject_length < (1u << 27) && in.max_query_length < (1u << 27);
  const uint32_t per = kTbWaveBlock / kWave;
  WaveCaps wc = {};
  uint32_t side_blocks = 0, batch = 1;
  if (waves) {
    wc = TracebackWaveCaps(in.max_query_length, in.max_subject_length);
    // blocks of a side: for as many waves as jobs up to half the resident
    // ones, within a 4 GB scratch budget, but at least one (subjects of tens
    // of millions of residues: up to 10 GB)
    const uint64_t side_waves = std::min<uint64_t>(n, kTbWaves / 2);
    const uint64_t fit = ((uint64_t)4 << 30) / 2 / ((uint64_t)per * wc.stride);
    side_blocks = (uint32_t)std::max<uint64_t>(1, std::min((side_waves + per - 1) / per, fit));
    const uint64_t b = n / ((uint64_t)side_blocks * per * 8) + 1;
    batch = (uint32_t)std::min<uint64_t>(b, 4);
  }
  const size_t a_jobs = Align256(n * sizeof(TracebackJob));
  const size_t a_outs = Align256(n * sizeof(TracebackOut));
  const size_t a_half = waves ? Align256(2 * (size_t)n * sizeof(TracebackHalf)) : 0;
  const size_t a_list = waves ? Align256((size_t)n * 4) : 0;
  const size_t before = a_jobs + a_outs + 256 + a_half + a_list;
  const LaneCaps lc = TracebackCaps(in.max_query_length, in.max_subject_length);
  hipError_t e = waves ? Reserve(before + (size_t)side_blocks * 2 * per * wc.stride, &ws_, &cap_)
                       : ReserveLanes(before, TracebackLanes(n, lc), lc.bytes_per_lane, &ws_,
                                      &cap_);
  if (e != hipSuccess) return e;
  char *w = (char *)ws_;
  TracebackJob *d_jobs = (TracebackJob *)w;
  TracebackOut *d_outs = (TracebackOut *)(w + a_jobs);
  uint32_t *d_counters = (uint32_t *)(w + a_jobs + a_outs);  // heads, listed jobs
  TracebackHalf *d_halves = (TracebackHalf *)(w + a_jobs + a_outs + 256);
  uint32_t *d_list = (uint32_t *)(w + a_jobs + a_outs + 256 + a_half);
  uint8_t *scratch = (uint8_t *)(w + before);
  e = hipMemcpyAsync(d_jobs, jobs, n * sizeof(TracebackJob), hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipEventRecord(ev_[0], s);
  if (e != hipSuccess) return e;
  uint32_t listed = 0;
  if (waves) {
    const WaveDpParams P = {in.queries, in.database, kDelimiter, in.gap_open + in.gap_ext,
                            in.gap_ext, in.cutoff, kWaveDpMargin};
    hipLaunchKernelGGL(ClearKernel, dim3(1), dim3(64), 0, s, d_counters, 3u);
    hipLaunchKernelGGL(TracebackWaveKernel, dim3(2 * side_blocks), dim3(kTbWaveBlock), 0, s, P,
                       d_jobs, n, batch, d_counters, in.matrix, in.nl, scratch, wc, d_halves);
    hipLaunchKernelGGL(TracebackJoinKernel, dim3((n + 255) / 256), dim3(256), 0, s, d_jobs, n,
                       d_halves, d_outs, d_counters + 2, d_list);
    e = hipGetLastError();
  } else {
    e = Lanes(in, d_jobs, n, nullptr, d_outs, scratch, cap_ - before, s);
  }
  if (e == hipSuccess) e = hipEventRecord(ev_[1], s);
  // the copies back are queued once the kernels are done: a device-to-host
  // copy queued behind a running kernel holds up other streams' copies
  if (e == hipSuccess) e = hipEventSynchronize(ev_[1]);
  if (e == hipSuccess && waves) {
    e = hipMemcpyAsync(&listed, d_counters + 2, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e == hipSuccess && listed > 0) {
      // bands past 256 columns and jobs whose frame is not as described, in
      // the waves' scratch, which is idle by now, where it has room for them
      const size_t lanes = TracebackLanes(listed, lc);
      size_t bytes = cap_ - before;
      if (bytes < lanes * lc.bytes_per_lane) {
        e = ReserveLanes(0, lanes, lc.bytes_per_lane, &lane_ws_, &lane_cap_);
        if (e == hipSuccess) {
          scratch = (uint8_t *)lane_ws_;
          bytes = lane_cap_;
        } else if (bytes >= 64 * lc.bytes_per_lane) {
          (void)hipGetLastError();
          e = hipSuccess;
        }
      }
      if (e == hipSuccess) e = Lanes(in, d_jobs, listed, d_list, d_outs, scratch, bytes, s);
      if (e == hipSuccess) e = hipEventRecord(ev_[1], s);
      if (e == hipSuccess) e = hipEventSynchronize(ev_[1]);
    }
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(outs, d_outs, n * sizeof(TracebackOut), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess && kernel_ms) e = hipEventElapsedTime(kernel_ms, ev_[0], ev_[1]);
  return e;
}

}  // namespace gz
