// simt.cpp -- TEST HARNESS: one workgroup of 64-lane wavefronts on the CPU.
//
// Each lane runs the kernel's per-lane code on its own fiber (ucontext).
// The wavefront primitives of ccd_core.h (ballot, shuffles, cross-lane
// reductions) are barriers of a wavefront: a lane that reaches one parks;
// when the wavefront's lanes have parked, the results are computed from
// their inputs and they run on, in lane order.  lane_sync and mem_sync are
// barriers of the workgroup: a wavefront runs on until all its lanes wait
// there, then the next one runs, in an order the caller picks, so that
// wavefronts are as far apart as the barriers let them.  Between barriers
// the lanes therefore run one after another, not in lockstep, so code that
// passes data between lanes or wavefronts through memory without a barrier
// reads stale values here; lanes that reach different primitives, or finish
// while others wait, are reported.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

namespace c2a {
namespace simt {

namespace {

constexpr int NL = 64;       // lanes of a wavefront
constexpr int NW_MAX = 4;    // wavefronts of a workgroup
constexpr size_t kStack = 8u << 20;
enum Kind : int { NONE = 0, SYNC, BALLOT, BCAST, BCASTD, PMAX, MIND, MAXI, LANE0, DONE };
const char* const kName[] = {"none", "sync", "ballot", "bcast", "bcastd",
                             "excl_prefix_max", "mind", "maxi", "lane0", "done"};

struct Lane {
  ucontext_t ctx;
  char* stack = nullptr;
  int kind = NONE;
  int64_t iv = 0, oi = 0;
  double dv = 0.0, od = 0.0;
  int src = 0;
};

Lane group[NW_MAX * NL];
Lane* lanes = group;   // the wavefront that runs
ucontext_t sched;
int cur = -1;          // its lane
void (*g_body)(int, void*) = nullptr;
void* g_arg = nullptr;
int64_t g_barriers = 0;

void arrive(int k) {
  Lane& l = lanes[cur];
  l.kind = k;
  swapcontext(&l.ctx, &sched);
}

void trampoline(int lane) {
  g_body(lane, g_arg);
  group[lane].kind = DONE;
}

void resolve(int k) {
  g_barriers++;
  switch (k) {
    case BALLOT: {
      uint64_t m = 0;
      for (int i = 0; i < NL; i++)
        if (lanes[i].iv) m |= 1ull << i;
      for (int i = 0; i < NL; i++) lanes[i].oi = (int64_t)m;
      break;
    }
    case BCAST:
      for (int i = 0; i < NL; i++) lanes[i].oi = lanes[lanes[i].src & (NL - 1)].iv;
      break;
    case BCASTD:
      for (int i = 0; i < NL; i++) lanes[i].od = lanes[lanes[i].src & (NL - 1)].dv;
      break;
    case PMAX: {
      int64_t run = 0;
      for (int i = 0; i < NL; i++) {
        const int64_t v = lanes[i].iv;
        lanes[i].oi = i == 0 ? 0 : run;
        run = (i == 0 || v > run) ? v : run;
      }
      break;
    }
    case MIND: {
      double m = lanes[0].dv;
      for (int i = 1; i < NL; i++) m = lanes[i].dv < m ? lanes[i].dv : m;
      for (int i = 0; i < NL; i++) lanes[i].od = m;
      break;
    }
    case MAXI: {
      int64_t m = lanes[0].iv;
      for (int i = 1; i < NL; i++) m = lanes[i].iv > m ? lanes[i].iv : m;
      for (int i = 0; i < NL; i++) lanes[i].oi = m;
      break;
    }
    case LANE0:
      for (int i = 0; i < NL; i++) lanes[i].oi = lanes[0].iv;
      break;
    default:
      break;
  }
  for (int i = 0; i < NL; i++) lanes[i].kind = NONE;
}

}  // namespace

int lane_id() { return (int)(lanes - group) + cur; }
int64_t barriers() { return g_barriers; }

void sync() { arrive(SYNC); }
uint64_t ballot(bool p) {
  lanes[cur].iv = p ? 1 : 0;
  arrive(BALLOT);
  return (uint64_t)lanes[cur].oi;
}
int bcast(int v, int src) {
  lanes[cur].iv = v;
  lanes[cur].src = src;
  arrive(BCAST);
  return (int)lanes[cur].oi;
}
double bcastd(double v, int src) {
  lanes[cur].dv = v;
  lanes[cur].src = src;
  arrive(BCASTD);
  return lanes[cur].od;
}
int excl_prefix_max(int v) {
  lanes[cur].iv = v;
  arrive(PMAX);
  return (int)lanes[cur].oi;
}
double mind(double v) {
  lanes[cur].dv = v;
  arrive(MIND);
  return lanes[cur].od;
}
int maxi(int v) {
  lanes[cur].iv = v;
  arrive(MAXI);
  return (int)lanes[cur].oi;
}
long long lane0(long long v) {
  lanes[cur].iv = v;
  arrive(LANE0);
  return (long long)lanes[cur].oi;
}

// Runs wavefront w until its lanes wait at a workgroup barrier or have
// finished; the kind they wait at, or -1 when they diverged.
static int run_wave(int w) {
  lanes = group + w * NL;
  for (;;) {
    for (int i = 0; i < NL; i++) {
      if (lanes[i].kind != NONE) continue;
      cur = i;
      swapcontext(&sched, &lanes[i].ctx);
    }
    cur = -1;
    const int k = lanes[0].kind;
    for (int i = 1; i < NL; i++)
      if (lanes[i].kind != k) {
        fprintf(stderr, "simt: wavefront %d: lane %d at %s while lane 0 is at %s (barrier %lld)\n",
                w, i, kName[lanes[i].kind], kName[k], (long long)g_barriers);
        return -1;
      }
    if (k == SYNC || k == DONE) return k;
    resolve(k);
  }
}

// Runs body(lane, arg) on `waves` wavefronts, the last one first when
// `backward`; 0 when every lane finished together, else the lanes diverged
// (the message names the primitives).
int launch(void (*body)(int, void*), void* arg, int waves, bool backward) {
  if (waves < 1 || waves > NW_MAX) return 4;
  g_body = body;
  g_arg = arg;
  g_barriers = 0;
  for (int i = 0; i < waves * NL; i++) {
    Lane& l = group[i];
    if (!l.stack) l.stack = (char*)malloc(kStack);
    if (!l.stack) return 3;
    getcontext(&l.ctx);
    l.ctx.uc_stack.ss_sp = l.stack;
    l.ctx.uc_stack.ss_size = kStack;
    l.ctx.uc_link = &sched;
    makecontext(&l.ctx, (void (*)())trampoline, 1, i);
    l.kind = NONE;
  }
  for (;;) {
    int ndone = 0;
    for (int i = 0; i < waves; i++) {
      const int k = run_wave(backward ? waves - 1 - i : i);
      if (k < 0) return 1;
      if (k == DONE) ndone++;
    }
    if (ndone == waves) return 0;
    if (ndone > 0) {
      fprintf(stderr, "simt: %d wavefronts finished while %d wait (barrier %lld)\n", ndone,
              waves - ndone, (long long)g_barriers);
      return 2;
    }
    g_barriers++;
    for (int i = 0; i < waves * NL; i++) group[i].kind = NONE;
  }
}

}  // namespace simt
}  // namespace c2a
