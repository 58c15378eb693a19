// Plays the dataflow Cholesky's order of tasks (csrc/rsd_dag.h and the lines that
// the kernel includes) through on the CPU: which tasks finish when a given number
// of workgroups run at once.
//
// A task is the list of flags that it waits for, in its order, with the flags
// that it sets between them, as dag_walker, dag_task and macro_task have them.
// Workgroups take tickets in order, each the next one as soon as it is free.
// What a workgroup can do never depends on how far another one has gone beyond
// the flags that it has set, and flags are never cleared, so the outcome does
// not depend on who goes first.
#include <stddef.h>

#include <set>
#include <utility>
#include <vector>

#include "../../regularized-stokesian-dynamics_amd/csrc/rsd_dag.h"

using namespace rsd;

namespace {

// the tile of a ticket; macro: the macro task (i, j)
struct DagTile {
  int i, j;
  bool macro;
};
DagTile dag_tile(int nt, bool MACRO, int t) {
  int i, j;
#define MACRO_TASK(I, J) return {I, J, true}
#include "../../regularized-stokesian-dynamics_amd/csrc/rsd_dag_tile.inc"
#undef MACRO_TASK
  return {i, j, false};
}
DagTile dag_x_tile(int ns, int r) {
  if (r < ns) return {r, r, false};
  int i, j;
#include "../../regularized-stokesian-dynamics_amd/csrc/rsd_dag_x.inc"
  return {i, j, false};
}

struct Play {
  int nt, s0, ns;
  bool macro;
  // flags: tiles (i,j), partial tiles 0 .. 2 nt - 1, X's tiles
  std::vector<char> tile, part, x;

  Play(int nt_, bool macro_, int s0_)
      : nt(nt_), s0(s0_), ns(s0_ >= 0 ? nt_ - s0_ : 0), macro(macro_), tile((size_t)nt_ * nt_), part(2 * nt_),
        x((size_t)ns * ns) {}
  char* L(int i, int j) { return &tile[(size_t)i + (size_t)nt * j]; }
  char* P(int q) { return &part[q]; }
  char* X(int i, int j) { return &x[(size_t)i + (size_t)ns * j]; }

  struct Op {
    char* flag;
    bool set;
  };
  using Task = std::vector<Op>;
  static void wait(Task& t, char* f) { t.push_back({f, false}); }
  static void set(Task& t, char* f) { t.push_back({f, true}); }

  Task walker() {
    Task t;
    wait(t, P(0));
    for (int j = 0; j < nt; ++j) {
      if (j > 0) set(t, L(j, j - 1));
      if (j + 1 < nt) {
        wait(t, P(2 * j + 1));
        wait(t, P(2 * (j + 1)));
      }
      set(t, L(j, j));
    }
    return t;
  }
  Task tile_task(const DagTile& q) {
    Task t;
    if (q.macro) {
      const int i0 = 2 * q.i, j0 = 2 * q.j;
      for (int k = 0; k < j0; ++k)
        for (int r : {i0, i0 + 1, j0, j0 + 1}) wait(t, L(r, k));
      wait(t, L(j0, j0));
      set(t, L(i0, j0));
      set(t, L(i0 + 1, j0));
      wait(t, L(j0 + 1, j0));
      wait(t, L(j0 + 1, j0 + 1));
      set(t, L(i0, j0 + 1));
      set(t, L(i0 + 1, j0 + 1));
      return t;
    }
    const int kend = q.i == q.j ? q.j - 1 : q.j;
    for (int k = 0; k < kend; ++k) {
      wait(t, L(q.i, k));
      wait(t, L(q.j, k));
    }
    if (q.i - q.j <= 1) {
      set(t, P(2 * q.j + q.i - q.j));
    } else {
      wait(t, L(q.j, q.j));
      set(t, L(q.i, q.j));
    }
    return t;
  }
  Task x_task(const DagTile& q) {
    Task t;
    for (int k = q.j; k < q.i; ++k) {
      wait(t, X(k, q.j));
      wait(t, L(s0 + q.i, s0 + k));
    }
    wait(t, L(s0 + q.i, s0 + q.i));
    set(t, X(q.i, q.j));
    return t;
  }
  Task task(int t, int nfac) {
    if (t == 0) return walker();
    return t <= nfac ? tile_task(dag_tile(nt, macro, t)) : x_task(dag_x_tile(ns, t - nfac - 1));
  }
};

}  // namespace

extern "C" {

// the tickets that are left over with `workgroups` at once (0: all finish)
int dag_play(int nt, int macro, int s0, int workgroups) {
  Play p(nt, macro, s0);
  const int nfac = dag_tickets(nt, macro), total = nfac + p.ns * (p.ns + 1) / 2;  // the last ticket
  struct Worker {
    Play::Task task;
    size_t at = 0;
  };
  std::vector<Worker> w(workgroups);
  int next = 0, left = total + 1;
  for (bool moved = true; moved && left > 0;) {
    moved = false;
    for (Worker& k : w) {
      if (k.at == k.task.size()) {
        if (next > total) continue;
        k.task = p.task(next++, nfac);
        k.at = 0;
        moved = true;
      }
      while (k.at < k.task.size()) {
        const Play::Op& op = k.task[k.at];
        if (op.set) *op.flag = 1;
        else if (!*op.flag) break;
        moved = true;
        if (++k.at == k.task.size()) --left;
      }
    }
  }
  return left;
}

// whether every lower tile is one ticket's, and every flag of a tile is set by
// one task (0: yes)
int dag_covers(int nt, int macro) {
  std::set<std::pair<int, int>> seen;
  size_t tiles = 0;
  for (int t = 1; t <= dag_tickets(nt, macro); ++t) {
    const DagTile q = dag_tile(nt, macro, t);
    const int f = q.macro ? 2 : 1;
    for (int a = 0; a < f; ++a)
      for (int b = 0; b < f; ++b, ++tiles) {
        const int i = f * q.i + a, j = f * q.j + b;
        if (i >= nt || j < 0 || j > i || !seen.insert({i, j}).second) return 1;
      }
  }
  return tiles == (size_t)nt * (nt + 1) / 2 ? 0 : 2;
}

int dag_x_covers(int ns) {
  std::set<std::pair<int, int>> seen;
  for (int r = 0; r < ns * (ns + 1) / 2; ++r) {
    const DagTile q = dag_x_tile(ns, r);
    if (q.j < 0 || q.j > q.i || q.i >= ns || !seen.insert({q.i, q.j}).second) return 1;
  }
  return 0;
}

int dag_beside() { return kDagBeside; }
int dag_macro_tiles() { return kMacroTiles; }
int dag_launch(int nt, int macro, int s0, int cus) {
  const int ns = s0 >= 0 ? nt - s0 : 0;
  return dag_workgroups(nt, 1 + dag_tickets(nt, macro) + ns * (ns + 1) / 2, cus);
}
int dag_total(int nt, int macro, int s0) {
  const int ns = s0 >= 0 ? nt - s0 : 0;
  return 1 + dag_tickets(nt, macro) + ns * (ns + 1) / 2;
}
}
