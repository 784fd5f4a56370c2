// Where the walks of a launch with few rows are split over more waves.  (Host arithmetic, no device code.)
#pragma once

namespace omni_attn {

// Slabs are dealt to the XCDs round-robin.  Where their number leaves some XCDs with more than 6 % less
// than others (4 slabs on 8 XCDs: half the device idle), each is dealt in parts of its tiles instead.
inline int slab_parts(int n_slabs, int n_xcd) {
  int parts = 1;
  while (parts < n_xcd) {
    const long long n = (long long)n_slabs * parts, most = (n + n_xcd - 1) / n_xcd;
    if (most * n_xcd * 100 <= n * 106) break;
    parts *= 2;
  }
  return parts;
}
// ... and what that makes of slabs of S rows (a multiple of 64): the 128-row tiles of the XCD that has most, and
// whether none has more than 6 % above the mean.
struct Dealing {
  int parts;
  long long busiest;
  bool even;
};
inline Dealing fwd_dealing(int n_slabs, int S, int n_xcd) {
  const int parts = slab_parts(n_slabs, n_xcd);
  const long long busiest = ((long long)n_slabs * parts + n_xcd - 1) / n_xcd * ((S / 128 + parts - 1) / parts);
  return {parts, busiest, 100 * 4 * busiest * n_xcd <= 106 * ((long long)n_slabs * (S / 32))};
}

// How the walk of a query block is split over waves (FwdShape says what the numbers are).
enum class FwdSplit : int {
  kNone,       // one workgroup per query block
  kRows32x4,   // 32-row tiles, four groups of one wave (steps without barriers)
  kRows64x2,   // 64-row tiles, two groups of two waves
  kRows64x4,   // 64-row tiles, four groups of two waves (head_dim 128)
  kRows128x2,  // 128-row tiles, two groups of four waves (head_dim 128)
};
constexpr int fwd_split_rows(FwdSplit s, int QB) {
  return s == FwdSplit::kNone ? QB : (s == FwdSplit::kRows32x4 ? 32 : (s == FwdSplit::kRows128x2 ? 128 : 64));
}
// Workgroups of an XCD from which on the longest lists of a batch's slabs go first (the caller says why).  With two waves
// on every SIMD, the others wait for a place (head_dim 32 has registers for three; the second and the third share
// the vector pipe all the same: B=3 H=5 S=2500, 64-row blocks, one element of three unmasked, 25.6 -> 26.2 us from the third).
// Four lone waves at head_dim 128 take longest over a list, and one such workgroup beside another is what
// a launch ends with: from the second workgroup of a compute unit (of two that fit), B=3 H=2 S=2048, one of
// three unmasked, 22.8 -> 20.4 us, causal 19.04 -> 19.20, spans 19.26 -> 19.45.  Elsewhere that costs nearly as often: head_dim 64,
// B=3 H=2 S=2304, 15.5 -> 13.8, causal 12.7 -> 12.95, spans 15.9 -> 16.1; B=3 H=4 S=2500 27.9 -> 27.9, 21.1 -> 21.4, 27.5 -> 27.7.
constexpr int fwd_waves(FwdSplit s, int QB) {
  const int groups = s == FwdSplit::kNone ? 1 : (s == FwdSplit::kRows32x4 || s == FwdSplit::kRows64x4 ? 4 : 2);
  return fwd_split_rows(s, QB) / 32 * groups;
}
constexpr int fwd_order_line(FwdSplit s, int D, int QB, int cus) {
  return s == FwdSplit::kRows32x4 && D == 128 ? cus : cus * (8 / fwd_waves(s, QB));
}

// Which split?  `rows32`: 32-row tiles of the whole launch, S: rows per slab; `busiest`: 128-row tiles dealt
// to the XCD that has most, `cus`: compute units of an XCD.  A wave walks a list of up
// to S / 64 steps of 1.2 us (alone on its SIMD, head_dim 128) to 1.7 us (two per SIMD); the device
// holds 2048 such waves.  With fewer tiles than that the longest list is the time of the launch, and
// sharing its steps shortens it; with more, the split costs K/V loads per row (a tile of 32 rows
// loads four times what one of 128 rows does, against 64 bytes per cycle and compute unit) and the
// merge, and whole blocks are faster.  A workgroup of eight waves (kRows64x4, kRows128x2) has a compute
// unit to itself: what does not start in the first round starts late, so those need one round, or
// lists long against the start and end of a workgroup.  The lines lie where the split gains on some masks
// and costs none of them more than runs differ by, as a rule (causal, two layouts of unaligned spans, and
// images of 1024 tokens; B H = 4 .. 64, S = 512 .. 8192).  Whole blocks, us, and the split against them:
//   D=128  kRows32x4   against kRows64x4: B H=8 S=1536 19-20 (-9 .. -17 %), B H=12 S=1024 15-16 (-12 .. -18), B H=5
//                      S=3000 30-43 (-3 .. -7), B H=2 S=8192 66-71 (-3 .. -5); beyond: B H=8 S=2048 23-24 (-3 .. +12)
//          kRows64x4   B H=16 S=1024 22-24 (-20 .. -23 %), S=1152 24 (-21, one layout +5); B H=12 S=2048 38-41
//                      (-23 .. +3), B H=8 S=3072 54-58 (-21 .. -36); beyond: B H=20 S=1152 24 (-3 .. +24)
//          kRows64x2   B H=20 S=1152 24 (0 .. -7), B H=24 S=1024 22-24 (-4 .. -10); beyond: B H=32 S=1237 30-35
//                      (-6 .. -12), but S=1280 30 (-11 .. +11) and S=1408 32 (-6 .. +25); where an XCD has a few more blocks
//                      than compute units: B H=26 S=1152 24 (-10 .. +1), B H=32 S=1100 24-29 (-8 .. -11), B H=48 S=700 19-22
//                      (-3 .. -14), with as many: B H=32 S=1024 21-24 (-8 .. +3)
//          kRows128x2  B H=20 S=1300 28-34 (-7 .. -17), B H=16 S=2048 38-42 (-8 .. -11), B H=14 S=2500 48-61 (-15
//                      .. -23), B H=12 S=4096 79-85 (-18 .. 0), B H=8 S=8192 169-175 (-2 .. -14); beyond: B H=26
//                      S=1152 26 (+10 .. +26; 39 workgroups for 32 compute units), B H=16 S=4096 89-96 (-9 .. +14)
//   64-row blocks: kRows64x4  B H=16 S=1237 31-40 (-34 .. -40), B H=12 S=2048 48 (-20 .. -38); kRows64x2  B H=40
//                      S=512 16 (-12), B H=24 S=1024 27 (-23), B H=20 S=2048 50-56 (-18 .. -26)
//   D=64   kRows32x4   against kRows64x2: B H=16 S=1024 11 (-10), B H=8 S=2048 17 (-22), B H=4 S=4096 29 (-25);
//                      B H=8 S=2304 19-22 (-10 .. -15), B H=10 S=2000 18-22 (0 .. -17), B H=4 S=5000 35-46 (-25 .. -32);
//                      beyond: B H=20 S=1024 12 (+31), B H=16 S=1237 13-16 (+3 .. +21), B H=6 S=4096 30-33 (-5 .. +8)
//          kRows64x2   B H=64 S=512 11-13 (-11 .. +3), B H=32 S=1024 18-20 (-4 .. -21), S=1237 21-28 (-14 .. -27),
//                      B H=20 S=2048 31-34 (-6 .. -24), B H=16 S=3072 45-49 (-8 .. -23), S=4096 60-65 (-8 .. +3);
//                      beyond: B H=40 S=1024 18-20 (0 .. +19), B H=24 S=2048 32-34 (-10 .. +16)
//   D=32   kRows32x4   against kRows64x2: B H=16 S=1237 11-16 (-17 .. -29), B H=6 S=4096 25-27 (-17 .. -26); beyond: B H=8
//                      S=4096 25-27 (-3 .. +7).  (Sparse lists of a single block each take longer so: B H=16 S=1152
//                      5.7 -> 6.2, of half the blocks 9.6 -> 7.8.)
//          kRows64x2   B H=40 S=1024 16-18 (-3 .. -16), B H=32 S=1536 21-24 (-10 .. -21), S=2048 28-33 (-14 .. +1)
// `ragged`: the sequence ends inside a query block.  With PARTIAL tiles every block of that list is one then (its last
// rows attend nothing): the longest list of a slab also has the slowest steps, and sharing it gains in larger
// launches.  `even`: no XCD has more than 6 % above the mean.  `batched`: more than one batch element; one in three may
// attend everything, and a launch of many long lists is bound by K/V loads.  Whole blocks, us, and the split against
// them, causal, two layouts of spans and images, then "mixed" (such a batch):
//   D=128  one batch element
//          kRows64x2   B H=32 S=1153 22-32 (-10 .. -15 %; the layouts with most work, one in four, +5), S=1237 and
//                      S=1270 28-32 (-3 .. -9; one in four, +4); beyond: S=1400 28-34 (-10 .. +16),
//                      B H=40 S=1000 22-26 (-15 .. +20), uneven B H=36 S=1100 24-29 (-9 .. +13)
//          kRows128x2  B H=24 S=1600 31-38 (-1 .. -19), S=1900 37-43 (-2 .. -17), B H=20 S=2100 39-48 (-8 .. -18), B H=16
//                      S=2600 47-58 (-11 .. -23), S=3700 70-89 (-18 .. +1); beyond: B H=24 S=2100 42-50 (-5 .. +10), B H=16
//                      S=4200 83-103 (-13 .. +4), uneven B H=22 S=1800 36-46 (-9 .. +15)
//          batched
//          kRows64x2   B H=24 S=1600 31-38 (-5 .. -14), mixed 41-43 (-15 .. +1), B H=20 S=2000 37-45 (-5 .. -13), mixed
//                      49 (-5); kRows128x2 there: mixed +10; beyond: B H=24 S=1750 mixed 45 (+13), B H=20 S=2100 39-48
//                      (-14 .. +7), B H=32 S=1237, four elements' spans 31 (+13)
//   D=64   kRows64x2   B H=32 S=1500 22-29 (-4 .. -25), mixed 30 (-5), B H=24 S=1900 26-34 (-15 .. -33), mixed 36 (-21);
//                      one batch element: B H=24 S=2700 38-52 (-3 .. -21), B H=16 S=4500 60-80 (-5 .. -18), B H=12 S=6000
//                      76-103 (-6 .. -21); beyond: B H=32 S=2000 mixed 39 (+11), B H=24 S=2000 mixed 38 (+8), B H=32 S=2300
//                      33-43 (-5 .. +10), B H=40 S=1237 19-25 (-13 .. +8), B H=20 S=4000 55-78 (-8 .. +8)
//   D=32   kRows64x2   B H=48 S=1237 16-23 (-5 .. -18), mixed 23 (-16), B H=40 S=1700 22-31 (-8 .. -27), B H=32 S=2300 27-37
//                      (-17 .. -24), S=3000 38-50 (-3 .. -18), mixed 57 (-1 .. -5), B H=16 S=6000 68-93 (-7 .. -28); beyond:
//                      B H=48 S=1500 20-27 (-18 .. +3)
//   64-row blocks (every head_dim: half the waves per workgroup, so half of the device stands by longer)
//          kRows64x2   D=128 B H=32 S=1237 30-38 (-16 .. -31), B H=24 S=1500 35-44 (-28 .. -33), B H=20 S=2300 50-64 (-15 ..
//                      -32); D=64 B H=32 S=1700 25-32 (-5 .. -26), B H=16 S=5000 72-91 (-2 .. -20), B H=12 S=6000 81-104 (-10 ..
//                      -26); batched B H=24 S=1500 22-29 (-12 .. -34), S=1700 24-32 (-4 .. -30), B H=16 S=5000 72-104
//                      (-2 .. -12); D=32 B H=32 S=2000 24-31 (-7 .. -32), batched B H=40 S=1300 17-22 (-2 .. -28); beyond:
//                      batched, D=64 B H=32 S=1700 mixed 33 (+15), S=1237 mixed 25 (+3)
inline FwdSplit fwd_ragged_split_64(int D, long long rows32, int S, bool even, bool batched) {
  if (!even || S < 1152) return FwdSplit::kNone;
  bool two;
  if (batched) {
    two = rows32 <= 1344 && (D == 32 || 5 * rows32 <= 4LL * S);
  } else {
    two = rows32 <= (D == 128 ? 1440 : (D == 64 ? 1792 : 2048));
  }
  return two || (D != 128 && rows32 <= 2560 && S >= 2 * rows32) ? FwdSplit::kRows64x2 : FwdSplit::kNone;
}
inline FwdSplit fwd_ragged_split(int D, long long rows32, int S, bool even, bool batched) {
  bool two;
  if (D == 128) {
    if (!even) return FwdSplit::kNone;
    if (!batched && ((rows32 <= 1440 && S >= 1600) || (rows32 <= 1856 && S >= 2 * rows32))) return FwdSplit::kRows128x2;
    two = rows32 <= 1280 && S >= (batched ? 1600 : 1152);
  } else if (D == 64) {
    if (S < 1408 || S < rows32) return FwdSplit::kNone;
    two = batched ? (rows32 <= 1440 && 4 * rows32 >= 3LL * S) || (rows32 <= 1792 && rows32 >= S)
                  : rows32 <= 2112 || (rows32 <= 2304 && S >= 2 * rows32);
  } else {
    two = (rows32 <= 1920 && S >= 1280) || (rows32 <= 2304 && S >= 1792) || (rows32 <= 3072 && S >= rows32);
  }
  return two ? FwdSplit::kRows64x2 : FwdSplit::kNone;
}
inline FwdSplit fwd_choose_split(int D, int QB, long long rows32, int S, long long busiest, int cus,
                                 bool ragged = false, bool even = true, bool batched = true) {
  const int one_round_32 = D == 128 ? 384 : (D == 64 ? 512 : 768);
  if (rows32 <= one_round_32 || (D == 128 && rows32 <= 512 && S >= 2560) || (D == 64 && rows32 <= 672 && S >= 2000))
    return FwdSplit::kRows32x4;
  const bool some = (rows32 <= 1024 && S >= 512) || (rows32 <= 1280 && S >= 2048) || (rows32 <= 2048 && S >= 2 * rows32);
  const bool lone = (rows32 <= 512 && S >= 512) || (rows32 <= 640 && S >= 1152) || (rows32 <= 768 && S >= 1536);
  if (QB != 128) {
    if (D == 128 && (lone || (rows32 <= 768 && S >= 1152))) return FwdSplit::kRows64x4;
    if (some) return FwdSplit::kRows64x2;
    return ragged ? fwd_ragged_split_64(D, rows32, S, even, batched) : FwdSplit::kNone;
  }
  if (D != 128) {
    const bool more = D == 64 ? rows32 <= 1280 && S >= 1152
                              : (rows32 <= 1280 && S >= 1024) || (rows32 <= 1536 && S >= 1536) || (rows32 <= 2048 && S >= 2048);
    if (some || more) return FwdSplit::kRows64x2;
    return ragged ? fwd_ragged_split(D, rows32, S, even, batched) : FwdSplit::kNone;
  }
  if (lone) return FwdSplit::kRows64x4;
  if (rows32 <= 768 && S >= 1024) return FwdSplit::kRows64x2;
  const bool one_round = busiest <= cus || (S >= 1280 && 8 * busiest <= 9LL * cus);
  const bool long_lists = S >= 2048 && (rows32 <= 1152 || (rows32 <= 1280 && S >= 2 * rows32) ||
                                        (rows32 <= 2048 && 5LL * S >= 13 * rows32));
  if ((rows32 <= 1152 && S >= 1152 && one_round) || long_lists) return FwdSplit::kRows128x2;
  if (rows32 <= 1152 && S >= 640 && busiest > cus && 4 * busiest < 5LL * cus) return FwdSplit::kRows64x2;
  return ragged ? fwd_ragged_split(D, rows32, S, even, batched) : FwdSplit::kNone;
}

// How the walk of a KV block is split over waves in the dK/dV kernel.
enum class DkdvSplit : int {
  kNone,      // one workgroup per KV block
  kKeys64x2,  // 64 keys, two groups of waves that share the query steps
  kKeys32x4,  // 32 keys, four groups (head_dim <= 64)
};

// Which splits?  The reasons are the forward's (fwd_choose_split): with few rows the longest walk is the
// time of a launch.  rows32: 32-row tiles of the launch, S: rows per slab.  The lines lie where a split gains
// on some masks and costs none more than runs differ by, as a rule (causal, unaligned spans, images of 1024
// tokens; B H = 4 .. 64, S = 512 .. 4096).  Both kernels together, causal, us, whole blocks -> chosen:
//   D=128  B H=8  S=512 37.9 -> 29.5, S=1024 59.7 -> 41.0, S=2048 102.9 -> 71.7, S=4096 192.3 -> 154.9
//   D=64   B H=8  S=512 29.4 -> 20.2, S=1024 46.2 -> 26.5, S=2048  79.7 -> 51.1, S=4096 146.9 -> 103.0
// The operator's backward at the lines (causal, spans, images), whole blocks, us, and the split of that kernel:
//   dQ     D=128  B H=20 S=1024 62 (-2 .. -10 %), B H=8 S=4096 177-217 (-12 .. +3); with the forward, B H=8 S=3000 173-222
//                 (-9 .. -14), B H=12 S=1700 112-125 (-12 .. -13), S=2048 131-152 (-1 .. -12), B H=16 S=1700 117-130 (-6
//                 .. -8); beyond: B H=20 S=1408 104 (-5 .. +1), B H=28 S=1152 95-101 (-2 .. +5); 64-row blocks (against
//                 steps of 64 keys, bwd_dq_step): B H=16 S=2048 107-140 (-7 .. +1), S=1024 beyond: B H=32 68-85 (+1 .. +5)
//          D=64   B H=40 S=1024 52-59 (-3 .. +1), B H=32 S=1237 58-72 (-6 .. -12), B H=24 S=2048 87-106 (-7 .. +3), B H=16
//                 S=4096 167-211 (-3 .. +2); 64-row blocks B H=32 S=1237 57-69 (-7 .. -13), B H=16 S=4096 172-225 (-8 .. 0)
//   dK/dV  D=128  B H=16 S=1237 62-73 (-1 .. -13), B H=8 S=4096 176-216 (-10 .. +2); 64-key blocks B H=12 S=1237 62-71
//                 (-8 .. -12), B H=8 S=4096 184-226 (-10 .. +1); beyond: B H=20 S=1237 69-86 (+1 .. +9)
//          D=64   B H=16 S=1237 51-60 (-4 .. -15), soft-capped 68-77 (-10), B H=12 S=2048 71-81 (-4 .. -17), B H=20 S=2048
//                 75-95 (0 .. -13); 64-key blocks 73-90 (-3 .. +9); beyond: B H=24 S=2048 78-106 (-2 .. +9), B H=12
//                 S=4096 136-170 (-7 .. +6)
//   dQ, D=64, lengths that end inside a block, where the forward is split for that if dealt evenly: B H=24 S=2300 127-172 (-2 .. -5), B H=16
//          S=4500 248-317 (0 .. -5), soft-capped 437 (-10), 64-row blocks B H=32 S=1700 97-117 (-3 .. -13), B H=24 S=2300
//          123-158 (-6 .. -10), B H=16 S=4500 258-327 (-3 .. -5); beyond: B H=40 S=1700 107-134 (-3 .. +4); D=128 gains
//          nowhere: B H=32 S=1237 101-130 (0 .. +4), B H=24 S=1700 128-171 (-2 .. +4).  However the slabs
//          are dealt, where the forward with 64-row blocks looks at that too: 64-row blocks with 7 - 17 % more on one XCD,
//          B H=37 S=1300 90-111 (0 .. -4, one layout +1), B H=35 S=1400 83-102 (-4 .. -8), B H=28 S=1900 105-131 (-6 .. -11)
//   dQ, D=64, soft-capped (three exponentials and a reciprocal per score: twice the vector work against a list's
//          loads), lengths that end inside a block: B H=32 S=2300 188-237 (-1 .. -9), S=2500 212-366 (-1 .. -5), B H=24 S=3000
//          242-356 (-2 .. -7), B H=20 S=4000 322-388 (-1 .. -9); beyond: S=3000 279-455 (0 .. -2), whole blocks B H=32
//          S=2048 161-230 (-5 .. +5), S=3072 286-406 (0 .. +2); D=128 B H=32 S=1500 148-208 (+3 .. +6)
//   dQ, D=32, lengths that end inside a block: B H=32 S=1700 76-125 (-7 .. -10), S=3000 152-267 (-1 .. -9), B H=40 S=2000 98-181 (0 ..
//          -8), B H=16 S=4500 184-234 (-6 .. -16), S=6000 274-354 (-2 .. -17), soft-capped B H=32 S=2000 135-211 (-4 .. -7),
//          64-row blocks B H=40 S=1700 83-148 (-3 .. -5), B H=16 S=4500 200-384 (-10 .. -14); beyond: B H=48 S=1237 67-96
//          (-8 .. +3); whole blocks B H=32 S=2048 90-129 (-7 .. +6), S=3072 157-215 (-1 .. +1)
inline FwdSplit bwd_choose_dq_split(int D, int QB, long long rows32, int S, bool ragged = false, bool batched = true,
                                    bool capped = false) {
  if (rows32 <= (D == 128 ? 256 : 512)) return FwdSplit::kRows32x4;
  bool two;
  if (D == 128) {
    two = rows32 <= 640 || (rows32 <= 1024 && S >= (QB == 128 ? 4096 : 2048)) ||
          (QB == 128 && ((rows32 <= 768 && S >= 1024) || (rows32 <= 896 && S >= 1536)));
  } else {
    two = (rows32 <= 1024 && S >= 512) || (rows32 <= 1536 && S >= 1024) || (rows32 <= 2048 && S >= 4096) ||
          (D == 32 && ragged && ((rows32 <= 2560 && S >= 1664) || (rows32 <= 3072 && S >= rows32))) ||
          (D == 64 && capped && ragged && QB == 128 && rows32 <= 2688 && S >= 2048 && S >= rows32) ||
          (D == 64 && ragged &&
           (QB == 128 ? fwd_ragged_split(D, rows32, S, true, batched)
                      : fwd_ragged_split_64(D, rows32, S, true, batched)) != FwdSplit::kNone);
  }
  return two ? FwdSplit::kRows64x2 : FwdSplit::kNone;
}
// Keys per step of a dQ launch without a split.  A 64-row block is two waves, and at head_dim 128 its tiles of 64 keys leave room
// for two workgroups on a compute unit, one wave per SIMD; with 32 keys four fit, but a step's halves no longer overlap inside
// a wave, and barriers come twice as often.  The second wave of a SIMD is worth more than that where the launch is bound by its
// total work; where the longest lists are its time, they take longer with 32 keys.  That changes at nearly two rounds of
// 512 workgroups; later for a length that ends inside a block, whose last list has the slowest steps, and where the
// rows belong to few slabs, with lists that differ more.  Both backward kernels, causal, spans, images (and `mixed` batches), us
// with 64 keys (and what 32 change):
//   lengths of whole blocks: B H=28 S=2048 150-255 (-6 .. +1 %), B H=64 S=896 81-121 (-3 .. +3), B H=32 S=1792 129-196 (-1 ..
//          +4), from 1920 row tiles B H=32 S=1920 144-239 (-2 .. -8), batched 145-265 (-2 .. -11), B H=24 S=2560 184-294 (-4 .. +8),
//          batched 185-370 (-12 .. +4), B H=40 S=1536 124-184 (-3 .. +5), B H=120 S=512 65-97 (-2 .. -8), B H=32 S=2048 162-261
//          (-8 .. +1), B H=16 S=4096 288-452 (-2 .. -4); below: B H=32 S=1024 65-92 (+5 .. +8), B H=48 S=1024 80-120 (+1 .. +7)
//   others: B H=20 S=1100 69-101 (+4 .. +11), B H=32 S=1400 95 (+6 .. +13), B H=24 S=2600 192-296 (-2 .. +10), B H=48 S=1400 126-190
//          (-3 .. +6); from 2208 row tiles B H=24 S=2900 229-365 (0 .. -3), B H=32 S=2500 230-364 (-6 .. +3), B H=64 S=1237
//          139-236 (-3 .. -9), B H=24 S=3700 346-559 (-6 .. +1); fewer than 20 slabs B H=16 S=5000 432-644 (-4 .. +3), B H=8
//          S=9000 711-1010 (-2 .. +11), S=12000 1184-1598 (-7 .. +3), from 3072 B H=8 S=14000 1671-2193 (0 .. -9), B H=16
//          S=7000 797-1101 (-4 .. -10)
inline int bwd_dq_step(int D, int QB, long long rows32, int S, bool ragged) {
  if (D != 128 || QB != 64) return 64;
  const long long from = !ragged ? 1920 : (5LL * S <= 8 * rows32 ? 2208 : 3072);
  return rows32 >= from ? 32 : 64;
}
inline DkdvSplit bwd_choose_dkdv_split(int D, bool capped, long long rows32, int S) {
  if (D != 128 && rows32 <= 256) return DkdvSplit::kKeys32x4;
  bool two = rows32 <= 512 || (rows32 <= 640 && S >= 1152);
  if (D == 128) {
    two = two || (rows32 <= 1024 && S >= 4096);
  } else if (!capped) {
    two = two || (rows32 <= 768 && S >= 1152) || (rows32 <= 1280 && S >= 2048);
  }
  return two ? DkdvSplit::kKeys64x2 : DkdvSplit::kNone;
}

}  // namespace omni_attn
