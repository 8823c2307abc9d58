// Instruction counts of the pipelined MFMA kernels' DMA side, and the s_waitcnt vmcnt(N) values derived from them:
// one definition for the kernels (gemm_mfma_pipe.hpp, gemm_mfma_pipe16.hpp) and for the host program that replays
// their issue order on the CPU and checks every count (tests/host_c/mfma_wait_check.cpp).
//
// The rule behind every N: the vector memory instructions of one wave that make a round trip to memory retire in the
// order they were issued, so "at most N outstanding" means "everything but the youngest N has landed".  An
// instruction whose lanes are ALL out of range makes no round trip and can retire ahead of older ones, so no kernel
// that counts issues one: padding stages and surplus scale instructions are real loads of one cache line, and an
// instruction of a K tail always holds the lane of its row's first chunk.  A wait that cannot be counted that way
// is vmcnt(0).
#pragma once

namespace zluda_amd {

struct PipeCounts {
  int cpr;      // 16-byte chunks per LDS row
  int rpw;      // rows filled by one wave DMA instruction
  int rpp;      // rows filled per DMA pass of the workgroup
  int lp, lq;   // data DMA instructions per thread, stage and operand
  int ndata;    // lp + lq
  int nwv;      // waves
  // MX block scales (zero without them): chunks of 32 scale bytes per tile row = ch stages, sparts instructions per
  // chunk, ls of them issued by every wave in front of every stage's data, pro_s per wave for the first chunk
  int sb, ch, sparts, ls, pro_s;
  int nload;    // ndata + ls: vector memory instructions per stage
  // Counted waits.  They count the DATA instructions of the younger stages only: the scale instructions of a stage
  // are issued in front of its data, so a wait that also covers them costs nothing.
  int wait_prologue;  // after the prologue (stages 0 .. nstage-1 issued): stage 0 has landed
  int wait_stage;     // in stage kt, before its slot is refilled: stage kt + 1 has landed
};

constexpr PipeCounts pipe_counts(bool mx, int bp, int bq, int wp, int wq, int bkb, int nstage) {
  PipeCounts c{};
  c.nwv = wp * wq;
  c.cpr = bkb / 16;
  c.rpw = 64 / c.cpr;
  c.rpp = c.nwv * c.rpw;
  c.lp = bp / c.rpp;
  c.lq = bq / c.rpp;
  c.ndata = c.lp + c.lq;
  c.sb = bkb / 16;
  c.ch = 32 / c.sb;
  c.sparts = (bp + bq) / 32;
  c.ls = mx ? (c.sparts + c.nwv * (c.ch - nstage) - 1) / (c.nwv * (c.ch - nstage)) : 0;
  c.pro_s = mx ? (c.sparts + c.nwv - 1) / c.nwv : 0;
  c.nload = c.ndata + c.ls;
  c.wait_prologue = (nstage - 1) * c.ndata;
  c.wait_stage = (nstage - 2) * c.ndata;
  return c;
}

// gemm_mfma_pipe16.hpp: `nstage` stages of 128 K bytes (two; up to six in the forms for operands along their row index), eight
// rows per DMA instruction, no scale instructions
struct Pipe16Counts {
  int rpp, lp, lq, nload;
  int wait_prologue;  // stages 0 .. nstage - 1 issued: stage 0 has landed
  int wait_stage;     // in stage kt, before its slot is refilled: stage kt + 1 has landed (of two stages, nothing younger is in flight)
};

constexpr Pipe16Counts pipe16_counts(int bp, int bq, int wp, int wq, int nstage = 2) {
  Pipe16Counts c{};
  c.rpp = wp * wq * 8;
  c.lp = bp / c.rpp;
  c.lq = bq / c.rpp;
  c.nload = c.lp + c.lq;
  c.wait_prologue = c.nload;
  c.wait_stage = 0;
  c.wait_prologue += (nstage - 2) * c.nload;
  c.wait_stage += (nstage - 2) * c.nload;
  return c;
}

// The form of gemm_mfma_pipe16.hpp whose operands lie along their row index ("MC"): an instruction of the last stage may hold
// no K row that exists.  Where that stage is in flight the prologue waits for everything, and so does a stage of a ring of more than two
// slots, which then requests no further one: what lies behind the last stage is never asked for there.
constexpr bool pipe16_drains_prologue(bool mc, int kt) { return mc && kt <= 2; }
constexpr bool pipe16_drains_prologue(bool mc, int kt, int nstage) { return pipe16_drains_prologue(mc, kt - (nstage - 2)); }
constexpr bool pipe16_drains_stage(int stage, int kt, int nstage) { return stage + nstage >= kt; }
// Rings of more than two slots are walked in turns of pipe16_turn() stages (whole turns of the ring, an even number of stages) from `stage`
// on while none of them requests the last stage or one behind it; those waits drain nothing.
constexpr int pipe16_turn(int nstage) { return nstage % 2 ? 2 * nstage : nstage; }
constexpr bool pipe16_inside(int stage, int kt, int nstage) { return stage + pipe16_turn(nstage) + nstage < kt; }

// gemm_mfma_tr.hpp leaves its waits to the compiler, which counts: before the LDS stores of trip kt (stage kt + 1's
// registers) it waits until only stage kt + 2's loads are outstanding.  Stages hold 64 K bytes; nothing past the last one that
// holds data, stage kl = ceil(kbytes / 64) - 1, is fetched.  Instructions of that stage can have all of their lanes out of
// range when kbytes is no multiple of 64, and with 2-byte elements always (the last element of a row, fetched on its own by
// the lanes that have one).  From the first trip whose younger stage is that one, the kernel waits for
// everything instead: the value below, compared with kt (0x7fffffff: never; negative: the prologue waits as well).
constexpr int tr_tail_from(int kbytes, int esz) {
  const int kt = (kbytes + 63) / 64, kl = kt > 0 ? kt - 1 : 0;
  return (kbytes & 63) || esz == 2 ? kl - 2 : 0x7fffffff;
}

// gemm_mfma_short.hpp: panels (128 rows of P or Q, all of K) come through a ring of two LDS slots in the order in which they are
// used: a run of tiles along Q needs a panel of Q each, behind one of P where the run starts or turns to the next tile of P.
// In flight at the wait for a panel, younger than it: the panel behind it (if the run has one), and the stores of the tile
// before and of the one before that, as far as those can be counted -- the stores of a tile that hangs over an end may be
// dropped and retire early.
struct ShortPos { int p, q, bt, left; bool p_due; };  // the next tile, how many are left, and whether its P panel comes first
constexpr void short_advance(ShortPos &c, int tiles_p, int tiles_q) {  // to the panel after this one
  if (c.p_due) { c.p_due = false; return; }
  c.left--;
  if (++c.q == tiles_q) {
    c.q = 0;
    c.p_due = true;
    if (++c.p == tiles_p) { c.p = 0; c.bt++; }
  }
}

struct ShortCounts {
  int panel;   // DMA instructions per wave and panel
  int stores;  // counted stores per wave and whole tile: those of a 16-bit D; one of 32 bits has twice as many
};
constexpr ShortCounts short_counts(int chunks) { return ShortCounts{chunks * 4, 8}; }

// The kernel's waits, N = short_wait_n(c, 0 .. 3); the one for a panel is the first whose N does not exceed what is younger than it
constexpr int short_wait_n(const ShortCounts &c, int which) {
  return which == 0 ? c.panel + 2 * c.stores : which == 1 ? c.panel + c.stores : which == 2 ? c.panel : 0;
}
constexpr int short_wait(const ShortCounts &c, bool panel_behind, int counted_stores) {
  const int younger = (panel_behind ? c.panel : 0) + counted_stores;
  return younger >= short_wait_n(c, 0) ? 0 : younger >= short_wait_n(c, 1) ? 1 : younger >= short_wait_n(c, 2) ? 2 : 3;
}

} // namespace zluda_amd
