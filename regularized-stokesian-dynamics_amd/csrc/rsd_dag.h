// rsd_dag.h -- the order of the dataflow Cholesky's tasks (rsd_dense.hip) and
// the number of workgroups of a launch, apart from the kernel so that the order
// can be played through on the CPU (tests/host/dag_host.cpp).
//
// Ticket 0 is the walker; tickets 1 .. dag_tickets() are the lower tiles (i,j)
// of nt block columns, or, with macro tasks, 2x2 blocks of them; behind them
// come X = inv(L_S)'s tiles, when a launch forms it.  Which tile a ticket is
// stands in rsd_dag_tile.inc and rsd_dag_x.inc.
#pragma once

#if defined(__HIPCC__) || defined(__HIP__)
#define RSD_DAG_HD __host__ __device__
#else
#define RSD_DAG_HD
#endif

namespace rsd {

constexpr int kAhead = 6;  // columns by which the early tiles start ahead
constexpr int kEarly = 3;  // early tiles per column: (c,c), (c+1,c), (c+2,c)

// Block columns from which macro tasks take the place of the single tiles away
// from the diagonal.  Below, a launch has too few of them to fill the CUs near
// its end; single / macro ms for the 11N launch and the W_PP product after it:
// N = 640 (110 block columns) 3.71 / 3.76, N = 720 (124) 5.15 / 5.27, N = 800
// (138) 6.74 / 6.70, N = 900 (155) 9.57 / 9.33, N = 997 (172) 12.6 / 12.3,
// N = 1400 (242) 35.9 / 33.0.
constexpr int kMacroTiles = 136;

// Workgroups that have to run at once beside the walker's for every order to
// finish, by playing the orders through task by task (with macro tasks; single
// tiles alone finish with 16).  A launch has that many, or one per task
// (dag_workgroups).  What counts is how many are resident: concurrent launches
// share the CUs, a workgroup to a CU.  A launch that holds as many as it needs
// runs to its end and gives its CUs back; while none does, each holds 19 at
// most, three of an XCD's 32 CUs (a launch's workgroups go to the eight XCDs in
// turn), so that up to ten launches at once leave each of them a CU for its
// next workgroup.  HIP runs a process's launches from four hardware queues by
// default, one at a time each.
constexpr int kDagBeside = 19;

RSD_DAG_HD inline int dag_early(int nt, int c) { return c < nt ? (kEarly < nt - c ? kEarly : nt - c) : 0; }

// Ticket order with macro tasks, per pair J of block columns: the early tiles
// of columns 2J + kAhead and 2J + 1 + kAhead; tile (2J+3, 2J) alone; the macro
// tasks (I, J), I >= J + 2; and, when nt is odd, the last block row's two tiles.
struct MacroCounts {
  int e0, e1, single, macros, last;
};
RSD_DAG_HD inline MacroCounts macro_counts(int nt, int J) {
  const int m = nt / 2 - (J + 2);
  return {dag_early(nt, 2 * J + kAhead), dag_early(nt, 2 * J + 1 + kAhead), 2 * J + 3 < nt ? 1 : 0, m > 0 ? m : 0,
          (nt & 1) && nt - 1 >= 2 * J + 4 ? 2 : 0};
}

// the factorization's tickets after the walker's
inline int dag_tickets(int nt, bool macro) {
  if (!macro) return nt * (nt + 1) / 2;
  int n = 0;
  for (int c = 0; c < kAhead; ++c) n += dag_early(nt, c);
  for (int J = 0; J < (nt + 1) / 2; ++J) {
    const MacroCounts k = macro_counts(nt, J);
    n += k.e0 + k.e1 + k.single + k.macros + k.last;
  }
  return n;
}

// The persistent workgroups of a launch of nt block columns: at most one per CU,
// and no more than its tile work keeps busy beside the diagonal chain, so that
// concurrent suspensions' factorisations share the chip (a workgroup takes all
// of a CU's registers).  Launches alone, us with 16 + nt^2/24 / 20 + nt^2/16 / 64 +
// nt^2/6: 19 block columns (N = 108) 420 / 360 / 362, 35 (N = 200) 681 / 600 / 606,
// 58 (N = 333) 1118 / 1009 / 1015, 88 (N = 512) 2105 / 2075 / 2079 with the
// inverse; a batch of 12 suspensions of N = 108..640 takes 53.5 / 54.4 / 56.0 ms.
inline int dag_workgroups(int nt, int tickets, int cus) {
  const int most = 1 + kDagBeside + nt * nt / 16;
  return tickets < most ? (tickets < cus ? tickets : cus) : (most < cus ? most : cus);
}

}  // namespace rsd
