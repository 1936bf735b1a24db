// gq_gemm_plan.h -- which kernel a batched product takes, how it is cut into
// blocks, and the workspace it needs.  Host code without HIP, so that the
// rules are tested against measured times on the CPU.
#pragma once
#include <stddef.h>

#include <algorithm>

namespace gq {

// ----------------------------------------------------------- workspace
// The batch that an eager call of n tokens takes workspace for: n rounded up
// to 256 and, past 1024, to a quarter of a power of two.  Superseded workspaces
// are kept, so a growing batch must not grow its workspace with every token:
// the sizes are a third or more apart, and the kept ones at most 3 times the
// last.
inline long gemm_room_tokens(int n) {
  long step = 256;
  while (4 * step < n) step *= 2;
  return (n + step - 1) / step * step;
}

// A workspace of `held` bytes (at `p`), a call that needs `need` of them and
// would take `room`: what to use.  The room is for other calls to come, so
// where alloc(room) gives nothing the call goes on with its own bytes, and
// that much room is not asked for again (`denied`).  False: not even those.
template <class Alloc>
bool take_workspace(void *&p, size_t &held, size_t &denied, size_t need, size_t room, Alloc alloc) {
  if (room > held && room < denied) {
    if (void *q = alloc(room)) {
      p = q;
      held = room;
    } else {
      denied = room;
    }
  }
  if (need <= held) return true;
  void *q = alloc(need);
  if (!q) return false;
  p = q;
  held = need;
  return true;
}

// ----------------------------------------------------------- bf16 mode
// (gq_gemm_quad.hip.)  Batches of up to GEMM_QUAD_MAX tokens in blocks of
// GEMM_QUAD_ROWS weight rows by all the tokens; a step of its K loop is a quad of
// units.
constexpr int GEMM_QUAD_MAX = 128, GEMM_QUAD_ROWS = 112;

// Token tiles of a batch of n <= 128: 1, 2, 3, 4, 6 or 8.
inline int gemm_quad_nt(int n) {
  const int t = (n + 15) / 16;
  return t <= 4 ? t : t <= 6 ? 6 : 8;
}

// Estimated time of a short batch's call, us, on `tiles` row tiles (`rows` rows
// in all) with K in ks parts: rounds of blocks (one a CU), each a start, its
// quads' dequant and MFMAs, and what of their weights' way from HBM these do not
// cover (longer the more of the CUs load at once); a split adds the reduction's
// launch and writes and reads ks partial products.  The constants (the types
// differ in the dequant and in what a block's first loads wait for) are those that
// choose best, here and in gemm_quad_faster, over every split of 4100 calls of 1 to
// 128 tokens on 64 x 256 to 130000 x 256 weights: the chosen ones take 0.1% longer
// than the best on average, 22 of them more than 5%, the worst 12%.  Of the times
// themselves they miss 11%.
inline double gemm_quad_time(int dtype, int tiles, long rows, int units, int n, int ks, int num_cus) {
  const int nt = gemm_quad_nt(n), quads = ((units + 3) / 4 + ks - 1) / ks;
  const double rounds = (double)(((long)tiles * ks + num_cus - 1) / num_cus), fill = tiles * ks / (rounds * num_cus);
  const double bits = dtype == 12 ? 4.5 : dtype == 13 ? 5.5 : dtype == 14 ? 6.5625 : 8.5;
  const double hbm = fill * num_cus * GEMM_QUAD_ROWS * 256 * bits / 8 / 4.7e6;  // a unit of every block
  const double start = dtype == 12 ? 0.76 : dtype == 14 ? 1.34 : 0.91;
  const double step = (dtype == 13 ? 2.56 : dtype == 8 ? 2.81 : 2.7) + 0.683 * nt;
  const double out = (double)rows * n * 8e-6 / 4.5;  // a result written and read
  return 4.76 + rounds * (start + 0.135 * hbm * std::min(4 * quads, units) + step * quads) +
         (ks > 1 ? 2.23 + 0.053 * ks + 1.03 * ks * out : 0.0) + 0.463 * out;
}

// The K split (over quads) of such a call: the least estimated time.  Up to 32
// tokens (two token tiles) many splits lie closer together than the estimates'
// error, and the split with the least rounds of quads, a start and a reduction
// counted as parts of one, is right more often: there that one, unless another's
// time is 3% less.  (Of 5700 calls 13 took 3% to 13% longer by the estimates alone
// than by the count; now three do, by up to 5%.)  Measured unsplit / in 2, us a
// call: 3584 x 2048 Q8_0 at 128 tokens 22.0 / 18.4, 14336 x 2048 Q4_K at 128 22.8 /
// 26.4, 65536 x 3584 Q6_K at 128 128.6 / 136.7 (the partial products' traffic);
// 3584 x 18944 Q6_K at 37 107 unsplit, 50 in 3, 36 in 5, 32 in 8, 41 in 10 (a second
// round); 12071 x 6912 Q6_K at 24 40.1 unsplit, 30.5 in 2, 36.3 in 7 (three rounds
// of single quads).
inline int gemm_quad_ksplit(int dtype, int tiles, long rows, int units, int n, int num_cus) {
  const int quads = (units + 3) / 4;
  int best = 1, count = 1;
  double best_t = 1e30, count_t = 1e30, time_of_count = 0.0;
  for (int ks = 1; ks <= std::min(quads, 16); ks++) {
    const double t = gemm_quad_time(dtype, tiles, rows, units, n, ks, num_cus);
    const long rounds = ((long)tiles * ks + num_cus - 1) / num_cus;
    const double c = rounds * (0.5 + (quads + ks - 1) / ks) + (ks > 1 ? 0.7 + 0.05 * ks : 0.0);
    if (t < best_t - 1e-9) {
      best_t = t;
      best = ks;
    }
    if (c < count_t - 1e-9) {
      count_t = c;
      count = ks;
      time_of_count = t;
    }
  }
  return n > 32 || best_t < 0.97 * time_of_count ? best : count;
}

// The 160 x 256 kernel's K split of a launch with this many row x token tiles and
// 64-element stages.
inline int gemm_ksplit(int tiles, int stages, int num_cus) {
  // The split with the least time per unit of work, rounds / ks (a block
  // per CU per round; 45 tiles x 6 = 270 blocks would run a second round
  // of 14), the smaller on ties; at most 8, at least 4 stages per split.
  if (tiles >= num_cus) return 1;
  const int kmax = std::max(1, std::min(8, stages / 4));
  int best = 1;
  double best_t = 1.0;
  for (int ks = 2; ks <= kmax; ks++) {
    const double t = (double)((tiles * ks + num_cus - 1) / num_cus) / ks;
    if (t < best_t - 1e-9) {
      best_t = t;
      best = ks;
    }
  }
  return best;
}

// Its estimated time at up to 256 tokens, us (error 5%): its stages take the same
// however few the tokens.  A ragged last tile waits on its one last row.
inline double gemm_direct_time(int dtype, int rows, int units, int n, int num_cus) {
  const int tiles = (rows + 159) / 160, ks = gemm_ksplit(tiles, 4 * units, num_cus);
  const double stage = dtype == 12 ? 1.13 : dtype == 13 ? 1.5 : dtype == 14 ? 1.36 : 1.15;
  const double out = (double)rows * n * 8e-6 / 4.5;
  const long rounds = ((long)tiles * ks + num_cus - 1) / num_cus;
  return 3.1 + rounds * (3.4 + stage * ((4 * units + ks - 1) / ks)) + (ks > 1 ? 3.2 + 0.78 * ks * out : 0.0) +
         0.22 * out + 2.4 * n / 128 + 1.6 * (tiles * 160 - rows) / 160;
}

// Whether a batch of n <= 128 tokens is faster on the short-batch kernel.  It is,
// up to four times, but where a row is one unit, and three quarters of the MFMA
// depth its zeros, or where its lower tiles take one round of blocks more; then
// the estimates decide.  Measured short / 160 x 256, us a call: 4800 x 256 Q4_K
// at 64 tokens 10.8 / 12.0, at 97 13.8 / 12.1; 37888 x 256 Q8_0 (339 and 237
// tiles) at 1 token 13.9 / 10.9, at 128 27.3 / 15.0; 37888 x 512 Q6_K at 128 28.1 /
// 21.3; 18944 x 512 Q4_K at 128 15.5 / 25.9.
inline bool gemm_quad_faster(int dtype, int rows, int units, int n, int num_cus) {
  const int tiles = (rows + GEMM_QUAD_ROWS - 1) / GEMM_QUAD_ROWS;
  const int rounds = (tiles + num_cus - 1) / num_cus, direct = ((rows + 159) / 160 + num_cus - 1) / num_cus;
  if (units > 1 && rounds <= direct) return true;
  const int ks = gemm_quad_ksplit(dtype, tiles, rows, units, n, num_cus);
  return gemm_quad_time(dtype, tiles, rows, units, n, ks, num_cus) <= gemm_direct_time(dtype, rows, units, n, num_cus);
}

// ----------------------------------------------------------- int8 mode
// (gq_gemm_q8.hip.)  small: 64 x 64 blocks, no K split; else 160 rows x 128 nj
// tokens.
constexpr int Q8_ROWS = 160, Q6S = 64;
struct Q8Plan {
  bool small;
  int nj, npad, ntiles, tiles, ksplit;
};

// The K split with the least estimated time of a token tile, us: rounds of
// blocks, each a start and its units (6.5 or 10 us each), and the reduction's
// launch and traffic.  Measured with 128- / 256-token tiles, us a call: 18944
// x 3584 Q4_K at 512 tokens 177 / 124, at 128 57 / 72; 3584 x 18944 Q6_K at
// 200 135 / 94; 9000 x 512 Q6_K at 300 23 / 30; 3584 x 3584 Q4_K at 512 58 / 47
// (in 2 / 5 splits).
inline double q8_split(int rows, int units, int nj, int n, int num_cus, int &ksplit) {
  const double out = (double)n * rows * 8e-6 / 4.5;  // one partial product written and read
  const int bn = 128 * nj;
  const long tiles = (long)((rows + Q8_ROWS - 1) / Q8_ROWS) * ((n + bn - 1) / bn);
  double best = 1e30;
  for (int ks = 1; ks <= std::min(units, 16); ks++) {
    const long rounds = (tiles * ks + num_cus - 1) / num_cus;
    const double t =
        rounds * (3.0 + (nj == 1 ? 6.5 : 10.0) * ((units + ks - 1) / ks)) + (ks > 1 ? 4.0 + ks * out : 0.0);
    if (t < best - 1e-9) {
      best = t;
      ksplit = ks;
    }
  }
  return best;
}

// Whether a Q6_K product takes the small kernel: where its estimated time is
// less by more than the estimates' error (about 4%), us a call.  Its
// blocks wait on latency, 4 us a unit, until they are more than the CUs; the
// other kernel pays a longer start, its 160-row stages and (in p's split) a
// reduction.  Measured small / 160-row, at 256 CUs: 600 x 256 at 200 tokens 11 /
// 16, 4800 x 512 at 200 17 / 23, 2400 x 768 at 700 25 / 33, 9000 x 256 at 512
// 27 / 19, 9000 x 512 at 700 44 / 32, 600 x 1024 at 16 21 / 16.
inline bool q6_small(int rows, int units, int n, const Q8Plan &p, int num_cus) {
  const double out = (double)n * rows * 8e-6 / 4.5;
  const long blocks = (long)((rows + Q6S - 1) / Q6S) * ((n + Q6S - 1) / Q6S);
  if ((n + Q6S - 1) / Q6S > 65535) return false;  // (the launch's second dimension)
  const double small =
      5.7 + units * (4.0 + (blocks > num_cus ? 0.65 + 1.46 * (blocks - num_cus) / num_cus : 0.0)) +
      std::min(n, Q6S) / (double)Q6S + 0.95 * out;
  const int bn = 128 * p.nj;
  const long tiles = (long)((rows + Q8_ROWS - 1) / Q8_ROWS) * ((n + bn - 1) / bn) * p.ksplit;
  const double rounds = (double)((tiles + num_cus - 1) / num_cus), upb = (units + p.ksplit - 1) / p.ksplit;
  const double used = std::min(n, 128) / 128.0 * std::min(rows, Q8_ROWS) / Q8_ROWS;
  const double big = 6.7 + 0.85 * tiles / (rounds * num_cus) +
                     rounds * (3.85 + upb * ((p.nj == 1 ? 5.3 : 7.0) + 2.6 * used)) +
                     (p.ksplit > 1 ? 1.2 + 1.06 * p.ksplit * out : 0.0) + 0.3 * out;
  return small < 0.97 * big;
}

inline Q8Plan q8_plan(int dtype, int rows, int units, int n, int num_cus) {
  int k1 = 1, k2 = 1;
  const double t1 = q8_split(rows, units, 1, n, num_cus, k1), t2 = q8_split(rows, units, 2, n, num_cus, k2);
  Q8Plan p{};
  p.nj = t2 < t1 - 1e-9 ? 2 : 1;
  p.ksplit = p.nj == 2 ? k2 : k1;
  p.small = dtype == 14 && q6_small(rows, units, n, p, num_cus);
  if (p.small) p.ksplit = 1;
  const int bm = p.small ? Q6S : Q8_ROWS, bn = p.small ? Q6S : 128 * p.nj;
  p.ntiles = (n + bn - 1) / bn;
  p.npad = p.ntiles * bn;
  p.tiles = (rows + bm - 1) / bm;
  return p;
}

// Workspace: codes, scales, thirds, partial products.
struct Q8Bytes {
  size_t xq, xs, xm, part;
  size_t total() const { return xq + xs + xm + part + 256; }
};
inline Q8Bytes q8_bytes(const Q8Plan &p, int rows, int units, int n) {
  const auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
  const size_t tu = (size_t)(p.npad / 16) * units;
  return {up256(tu * (p.small ? 4096 : 8192)), up256(tu * 512), up256(tu * 1024),
          p.ksplit > 1 ? (size_t)p.ksplit * n * rows * 4 : 0};
}

// A bound for every batch of up to n tokens.  A token tile's batches share
// their block counts, so the shortest has the largest split of each tile size.
inline size_t q8_bytes_bound(int rows, int units, int n, int num_cus) {
  Q8Plan p{};
  p.npad = (n + 255) / 256 * 256;
  p.ksplit = 1;
  Q8Bytes b = q8_bytes(p, rows, units, n);
  for (int n0 = 0; n0 < n; n0 += 128) {
    int ks = 1;
    for (int nj = 1; nj <= 2; nj++) {
      int k = 1;
      (void)q8_split(rows, units, nj, n0 + 1, num_cus, k);
      ks = std::max(ks, k);
    }
    if (ks > 1) b.part = std::max(b.part, (size_t)ks * std::min(n, n0 + 128) * rows * 4);
  }
  return b.total();
}

}  // namespace gq
