// Host-side replay of the DMA issue order of the pipelined MFMA kernels, with the kernels' own instruction counts and
// wait values (zluda_amd/csrc/kernels/mfma_wait_counts.hpp) and the planner's table of instantiated tile variants:
// at every counted s_waitcnt vmcnt(N) of every variant
//   * the stage the wait is there for has landed, given that a wave's loads retire in the order they were issued,
//   * N is exactly the number of DATA instructions issued after that stage's last one (one more would let the wait pass
//     early, one less would wait for a stage that should stay in flight),
//   * the MX scale chunk a stage reads landed before the barrier in front of the read.
// For the transposing kernel, which leaves the counting to the compiler: every trip whose younger stage in flight can
// hold lanes past the end of K is one that waits for everything.
// usage: mfma_wait_check   (prints the number of waits checked, exits non-zero on the first violation)
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../zluda_amd/csrc/kernels/mfma_wait_counts.hpp"
#include "../../zluda_amd/csrc/planner.hpp"

using namespace zluda_amd;

enum { DATA, SCALE, SURPLUS };
struct Ins { int kind, id; };  // DATA: stage; SCALE: chunk; SURPLUS: -

static long checked = 0;

static void fail(const char *what, int variant, int mx, int wave, int kt, int KT) {
  printf("variant %d mx %d wave %d stage %d of %d: %s\n", variant, mx, wave, kt, KT, what);
  exit(1);
}

// the youngest `n` of `log` are outstanding: has every instruction of (kind, id) landed?
static bool landed(const std::vector<Ins> &log, size_t issued, int n, int kind, int id) {
  for (size_t i = issued > (size_t)n ? issued - n : 0; i < issued; i++)
    if (log[i].kind == kind && log[i].id == id) return false;
  return true;
}
// DATA instructions issued after the last one of `stage`
static int data_after(const std::vector<Ins> &log, int stage) {
  int last = -1;
  for (size_t i = 0; i < log.size(); i++)
    if (log[i].kind == DATA && log[i].id == stage) last = (int)i;
  if (last < 0) return -1;
  int n = 0;
  for (size_t i = last + 1; i < log.size(); i++) n += log[i].kind == DATA;
  return n;
}

// gemm_mfma_pipe_kernel: prologue, then per stage [reads of the next stage's scales] wait, barrier, scale instructions,
// data of stage kt + nstage
static void check_pipe(const MfmaVariant &v, int variant, bool mx, int ks) {
  const PipeCounts c = pipe_counts(mx, v.bp, v.bq, v.wp, v.wq, v.bkb, v.stages);
  if ((v.stages - 1) * c.nload >= 64) fail("vmcnt range", variant, mx, 0, 0, 0);
  for (int KT = 1; KT <= 3 * c.ch + v.stages + 2; KT++)
    for (int wave = 0; wave < c.nwv; wave++) {
      std::vector<Ins> log;
      auto scale_part = [&](int chunk, int part) { log.push_back(part < c.sparts ? Ins{SCALE, chunk} : Ins{SURPLUS, 0}); };
      auto data = [&](int stage) { for (int i = 0; i < c.ndata; i++) log.push_back(Ins{DATA, stage}); };
      for (int i = 0; i < c.pro_s; i++) scale_part(0, i * c.nwv + wave);
      for (int s = 0; s < v.stages; s++) {
        for (int i = 0; i < c.ls; i++) scale_part(0, c.sparts);
        data(s);
      }
      size_t wait_at = log.size();  // instructions issued at the last wait, and its N
      int wait_n = c.wait_prologue;
      if (!landed(log, wait_at, wait_n, DATA, 0)) fail("prologue: stage 0 still in flight", variant, mx, wave, 0, KT);
      if (data_after(log, 0) != wait_n) fail("prologue: N is not the count of younger data instructions", variant, mx, wave, 0, KT);
      if (mx && !landed(log, wait_at, wait_n, SCALE, 0)) fail("prologue: first scale chunk still in flight", variant, mx, wave, 0, KT);
      checked++;
      for (int kt = 0; kt < KT; kt++) {
        const int next_chunk = (kt + 1) / c.ch;
        // several sub-steps: the scales of stage kt + 1 are read in the first one, under the previous barrier
        if (mx && ks > 1 && kt + 1 < KT && !landed(log, wait_at, wait_n, SCALE, next_chunk))
          fail("scale chunk read before it landed", variant, mx, wave, kt, KT);
        wait_at = log.size();
        wait_n = c.wait_stage;
        if (!landed(log, wait_at, wait_n, DATA, kt + 1)) fail("next stage still in flight", variant, mx, wave, kt, KT);
        if (data_after(log, kt + 1) != wait_n) fail("N is not the count of younger data instructions", variant, mx, wave, kt, KT);
        if (mx && ks == 1 && kt + 1 < KT && !landed(log, wait_at, wait_n, SCALE, next_chunk))
          fail("scale chunk read before it landed", variant, mx, wave, kt, KT);
        checked++;
        for (int i = 0; i < c.ls; i++) scale_part(kt / c.ch + 1, ((kt % c.ch) * c.ls + i) * c.nwv + wave);
        data(kt + v.stages);
      }
      // every part of every chunk that a stage reads was issued by some wave: parts [0, sparts) over the waves
      if (mx && wave == 0) {
        std::vector<int> seen(c.sparts, 0);
        for (int w = 0; w < c.nwv; w++)
          for (int kt = 0; kt < c.ch; kt++)
            for (int i = 0; i < c.ls; i++) {
              const int part = ((kt % c.ch) * c.ls + i) * c.nwv + w;
              if (part < c.sparts) {
                if (kt >= c.ch - v.stages) fail("a scale part is issued too late in its chunk", variant, mx, w, kt, KT);
                seen[part]++;
              }
            }
        for (int p = 0; p < c.sparts; p++)
          if (seen[p] != 1) fail("scale parts of a chunk not issued exactly once", variant, mx, 0, p, KT);
      }
    }
}

// gemm_mfma_pipe16_kernel: stages 0 and 1, wait; per stage wait, barrier, data of stage kt + 2
static void check_pipe16(int variant) {
  const MfmaVariant &v = kMfmaVariants[variant];
  const Pipe16Counts c = pipe16_counts(v.bp, v.bq, v.wp, v.wq);
  if (v.stages != 2 || v.bkb != 128) fail("two stages of 128 bytes", variant, 0, 0, 0, 0);
  for (int KT = 1; KT <= 9; KT++) {
    std::vector<Ins> log;
    auto data = [&](int stage) { for (int i = 0; i < c.nload; i++) log.push_back(Ins{DATA, stage}); };
    data(0); data(1);
    if (!landed(log, log.size(), c.wait_prologue, DATA, 0)) fail("prologue: stage 0 still in flight", variant, 0, 0, 0, KT);
    if (data_after(log, 0) != c.wait_prologue) fail("prologue: N is not the count of younger data instructions", variant, 0, 0, 0, KT);
    checked++;
    for (int kt = 0; kt < KT; kt++) {
      if (!landed(log, log.size(), c.wait_stage, DATA, kt + 1)) fail("next stage still in flight", variant, 0, 0, kt, KT);
      if (data_after(log, kt + 1) != c.wait_stage) fail("N is not the count of younger data instructions", variant, 0, 0, kt, KT);
      checked++;
      data(kt + 2);
    }
  }
}

// The form of gemm_mfma_pipe16_kernel for operands along their row index, on tiles of bp x bq: what the prologue counts on --
// stage 0 landed with stage 1's instructions outstanding -- holds only while neither stage can retire ahead of its turn, i.e.
// neither is the last one, whose K tail an instruction may miss altogether.  (The waits of the loop count nothing.)
static void check_pipe16_mc(int bp, int bq, int wp, int wq) {
  const Pipe16Counts c = pipe16_counts(bp, bq, wp, wq);
  if (c.wait_stage != 0) fail("a wait of the loop that counts", -1, 0, 0, 0, 0);
  for (int KT = 1; KT <= 9; KT++) {
    const int last = KT - 1;
    if (last <= 1 && !pipe16_drains_prologue(true, KT)) fail("the prologue counts past a stage that can retire early", -1, 0, 0, 0, KT);
    if (last > 1 && pipe16_drains_prologue(true, KT)) fail("needless wait in the prologue", -1, 0, 0, 0, KT);
    if (pipe16_drains_prologue(false, KT)) fail("needless wait in the prologue", -1, 0, 0, 0, KT);
    checked++;
  }
}

// The same on a ring of more than two stages: a wait of the loop leaves those behind the next one in flight, but nothing where the
// last stage of K is among them; nothing behind that one is requested.
static void check_pipe16_ring(int bp, int bq, int wp, int wq, int nstage) {
  const Pipe16Counts c = pipe16_counts(bp, bq, wp, wq, nstage);
  if ((nstage - 1) * c.nload >= 64) fail("vmcnt range", -1, 0, 0, 0, 0);
  for (int KT = 0; KT <= 5 * nstage + 2; KT++) {
    std::vector<Ins> log;
    auto data = [&](int stage) { for (int i = 0; i < c.nload; i++) log.push_back(Ins{DATA, stage}); };
    for (int s = 0; s < nstage && s < KT; s++) data(s);
    const bool drained = pipe16_drains_prologue(true, KT, nstage);
    if (drained != (nstage - 1 >= KT - 1)) fail("the prologue's drain", -1, 0, 0, 0, KT);
    if (!drained && !landed(log, log.size(), c.wait_prologue, DATA, 0)) fail("prologue: stage 0 still in flight", -1, 0, 0, 0, KT);
    if (!drained && data_after(log, 0) != c.wait_prologue) fail("prologue: N is not the count of younger data instructions", -1, 0, 0, 0, KT);
    // the turns at compile time: none of their stages drains, or requests what is not a whole stage
    int inside = 0;
    for (; pipe16_inside(inside, KT, nstage); inside += pipe16_turn(nstage))
      for (int kt = inside; kt < inside + pipe16_turn(nstage); kt++)
        if (pipe16_drains_stage(kt, KT, nstage) || kt + nstage >= KT - 1) fail("a turn reaches the last stage", -1, 0, 0, kt, KT);
    if (inside % nstage || inside % 2) fail("a turn leaves the ring inside it", -1, 0, 0, inside, KT);
    if (inside + pipe16_turn(nstage) + nstage + 1 <= KT) fail("a turn is left out", -1, 0, 0, inside, KT);
    for (int kt = 0; kt < KT; kt++) {
      const bool drains = pipe16_drains_stage(kt, KT, nstage);
      if (drains != (kt + nstage - 1 >= KT - 1)) fail("a stage's drain", -1, 0, 0, kt, KT);
      checked++;
      if (drains) continue;  // (and requests nothing)
      if (kt + nstage >= KT) fail("a stage behind the last one is requested", -1, 0, 0, kt, KT);
      if (!landed(log, log.size(), c.wait_stage, DATA, kt + 1)) fail("next stage still in flight", -1, 0, 0, kt, KT);
      if (data_after(log, kt + 1) != c.wait_stage) fail("N is not the count of younger data instructions", -1, 0, 0, kt, KT);
      data(kt + nstage);
    }
  }
}

// gemm_mfma_tr_kernel: the stages are requested in order, nothing past the last one, kl.  The prologue stores stage 0's registers
// with stage 1 in flight, trip kt those of stage kt + 1 with stage kt + 2 in flight.
static void check_tr(int esz) {
  for (int kbytes = esz; kbytes <= 64 * 9; kbytes += esz) {
    const int KT = (kbytes + 63) / 64, KL = KT - 1;
    const int tail_from = tr_tail_from(kbytes, esz);
    const bool last_retires_early = (kbytes & 63) != 0 || esz == 2;  // lanes past the end of K; the extra loads of 2-byte elements
    std::vector<int> in_flight;  // stages, oldest first
    auto request = [&](int stage) { if (stage <= KL) in_flight.push_back(stage); };
    auto store = [&](int stage, bool waits_for_all, const char *where, int kt) {
      // counted: everything but the stages younger than `stage` has landed -- unless one of those can be done before its turn
      for (int s : in_flight)
        if (s > stage && s == KL && last_retires_early && !waits_for_all) {
          printf("transposing kernel, K = %d bytes of %d-byte elements, %s %d: counts past a stage that can retire early\n", kbytes, esz, where, kt);
          exit(1);
        }
      if (waits_for_all) in_flight.clear();
      while (!in_flight.empty() && in_flight[0] <= stage) in_flight.erase(in_flight.begin());
      checked++;
    };
    request(0); request(1);
    store(0, tail_from < 0, "prologue", 0);
    request(2);
    for (int kt = 0; kt + 1 <= KL; kt++) {  // trips that still store a stage
      store(kt + 1, kt >= tail_from, "trip", kt);
      request(kt + 3);
    }
    if (!last_retires_early && tail_from != 0x7fffffff) { printf("transposing kernel, K = %d bytes: needless waits\n", kbytes); exit(1); }
    if (last_retires_early && KL >= 3 && KL - 3 >= tail_from) { printf("transposing kernel, K = %d bytes: waits a trip early\n", kbytes); exit(1); }
  }
}

// gemm_mfma_short_kernel: runs of tiles of every length and start in small grids, whose last tiles along P and Q hang over the ends or
// not.  Counted by hand here: a wave's 64 x 64 part of a 128 x 128 tile has 16 tiles of 16 x 16 and stores two of them (16-bit D) or one
// (32 bits) with an instruction; a panel is 128 rows in chunks of 128 bytes, 32 rows per instruction of the four waves.
static void check_short(int chunks, bool wide) {
  const ShortCounts c = short_counts(chunks);
  enum { PANEL, STORE, LOOSE };  // LOOSE: stores that can be dropped, and retire early
  const int panel_ins = chunks * 128 / 32, store_ins = wide ? 16 : 8;
  if (short_wait_n(c, 0) >= 64) fail("vmcnt range", -2, 0, 0, 0, 0);
  long widest = 0;
  for (int tp = 1; tp <= 3; tp++)
    for (int tq = 1; tq <= 4; tq++)
      for (int edges = 0; edges < 4; edges++)
        for (int first = 0; first < 2 * tp * tq; first++)
          for (int count = 1; count <= 9; count++) {
            std::vector<Ins> log;
            ShortPos use{first / tq % tp, first % tq, first / (tp * tq), count, true}, ask = use;
            int asked = 0, read = 0, panels = 0, st1 = 0, st2 = 0, tiles = 0, row = -1;  // (row of tiles whose P panel is in registers)
            auto request = [&]() {
              if (ask.left == 0) return;
              for (int i = 0; i < panel_ins; i++) log.push_back(Ins{PANEL, asked});
              asked++; panels++;
              short_advance(ask, tp, tq);
            };
            request(); request();
            while (use.left > 0) {
              const int which = short_wait(c, panels == 2, st1 + st2), n = short_wait_n(c, which);
              // in order: everything but the loose stores; those may be gone already, so only the others count as outstanding
              int younger = 0;
              for (size_t i = log.size(); i-- > 0 && !(log[i].kind == PANEL && log[i].id == read);) younger += log[i].kind != LOOSE;
              if (n > younger) fail("short K: a panel may still be in flight", -2, 0, chunks, read, count);
              // the waits are as lax as the kernel has them: between whole tiles of a run nothing younger is waited for
              if (which == 0) widest++;
              if (!wide && panels == 2 && st1 + st2 == 2 * store_ins && n != younger) fail("short K: a needless wait", -2, 0, chunks, read, count);
              checked++;
              const ShortPos now = use;
              read++; panels--;
              request();
              short_advance(use, tp, tq);
              st2 = st1;
              st1 = 0;
              if (now.p_due) { row = now.bt * tp + now.p; continue; }
              if (now.bt * tp + now.p != row || row * tq + now.q != first + tiles) fail("short K: another tile's turn", -2, 0, chunks, tiles, count);
              const bool whole = !((edges & 1) && now.p == tp - 1) && !((edges & 2) && now.q == tq - 1);
              for (int i = 0; i < store_ins; i++) log.push_back(Ins{whole ? STORE : LOOSE, 0});
              if (whole) st1 = c.stores;
              tiles++;
            }
            if (tiles != count || asked != read) fail("short K: a run does not hold its tiles", -2, 0, chunks, tiles, count);
          }
  if (widest == 0) fail("short K: the widest wait is never reached", -2, 0, chunks, 0, 0);
}

int main() {
  for (int variant = 0; variant < kNumMfmaVariants; variant++) {
    const MfmaVariant &v = kMfmaVariants[variant];
    if (v.w4) continue;  // every wait of the four-wave kernel is vmcnt(0) (checked on its source)
    if (v.m16) { check_pipe16(variant); continue; }
    // sub-steps per stage: 32 K bytes each, fp8 64; with and without MX scales where the variant serves MXFP4
    for (int ks : {v.bkb / 32, v.bkb / 64}) check_pipe(v, variant, false, ks);
    if (variant < kNumMfmaVariants32) check_pipe(v, variant, true, v.bkb / 32);
  }
  for (int ks : {2, 4}) check_pipe(kMfmaEightWaves, 2, false, ks);
  for (int chunks : {1, 2})
    for (bool wide : {false, true}) check_short(chunks, wide);
  for (int v : {1, 3}) check_pipe16_mc(kTrVariants[v].bp, kTrVariants[v].bq, kTrVariants[v].wp, kTrVariants[v].wq);
  check_pipe16_ring(kTrVariants[1].bp, kTrVariants[1].bq, kTrVariants[1].wp, kTrVariants[1].wq, kTrDeepStages);
  for (int nstage : kTr64Stages) {
    if (nstage > 2) check_pipe16_ring(kTrVariants[2].bp, kTrVariants[2].bq, kTrVariants[2].wp, kTrVariants[2].wq, nstage);
    else check_pipe16_mc(kTrVariants[2].bp, kTrVariants[2].bq, kTrVariants[2].wp, kTrVariants[2].wq);
  }
  for (int esz : {1, 2, 4}) check_tr(esz);
  printf("%ld waits checked\n", checked);
  return 0;
}
