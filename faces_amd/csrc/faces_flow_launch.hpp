// faces_flow_launch.hpp -- the launches of the one-item kernel (faces_flow.hpp)
// for one element size n: the kernel instantiations (elements per item S,
// load width, mode, tree order) of each n are compiled in the translation
// unit of its group of sizes (faces_flow_g*.hip), beside one another.
#pragma once

#include "faces_common.hpp"
#include "faces_flow.hpp"

namespace faces {

template <int N, int S>
int launch_flow_ns(int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st)
{
  constexpr int T = kFlowThreads<N, S>;
  // load widths 0 to 2 and mode 3 hold 8-byte slots: 256-thread items of n <= 12
  constexpr bool narrow = flow_narrow(N, S);
  if (!narrow && (lw != 3 || mode == 3))
    return fail(FACES_ERR_ARG, "one-item kernel: n=%d S=%d is compiled with load width 3 and modes 0 to 2", N, S);
  SurfWork sw = {};
  unsigned nblk = 0;
  if (mode == 3 && (!W || W->nblk || lw != 2 || tree))
    return fail(FACES_ERR_ARG, "one-item kernel: mode 3 takes the receive slots, load width 2, no surface blocks");
  if (W) {
    if (mode != 1 && mode != 3) return fail(FACES_ERR_ARG, "one-item kernel: surface blocks need mode 1");
    sw = *W;
    // leading surface blocks: a multiple of 8, so that item block b still
    // runs on XCD b % 8
    nblk = W->lead ? (W->nblk + 7u) & ~7u : W->nblk;
    sw.nblk = nblk;
  }
  sw.sfirst = W && W->lead ? 0u : nb;
  sw.item0 = W && W->lead ? nblk : 0u;
  if ((unsigned long)nb + nblk > 0x7fffffffUL) return fail(FACES_ERR_ARG, "one-item kernel: grid too large");
  const dim3 grid(nb + nblk), blk(T);
  // the footprint, and for mode 1 the marks of the rank-surface copies
#define FACES_LAUNCH_FLOW(LW, MODE, TREE)                                                      \
  k_flow<N, S, LW, MODE, TREE>                                                                 \
      <<<grid, blk,                                                                            \
         (size_t)StreamShape<N, S>::P * sizeof(double) +                                       \
             (MODE == 1 ? (size_t)kFlowMarkWords<N, S> * sizeof(unsigned) : 0),                \
         st>>>(G, F, sw)
#define FACES_LAUNCH_PAIRS(MODE, TREE)                                                         \
  k_pairs<N, S, MODE, TREE>                                                                    \
      <<<grid, blk,                                                                            \
         (size_t)PairShape<N, S>::P * sizeof(double) +                                         \
             (MODE == 1 ? (size_t)PairShape<N, S>::kMarkWords * sizeof(unsigned) : 0),         \
         st>>>(G, F, sw)
  if (tree) {
    // the 6-message schedule's tree: owned runs in 16-byte pairs (any
    // alignment; load width 3: the partner regions' too), periodic or open
    if (lw < 2 || mode == 1 || mode == 3)
      return fail(FACES_ERR_ARG, "one-item kernel: tree order z,y,x needs load width 2 or 3 and mode 0 or 2");
    if (lw == 3) {
      if (mode == 2) FACES_LAUNCH_PAIRS(2, 1);
      else FACES_LAUNCH_PAIRS(0, 1);
    }
    if constexpr (narrow) {
      if (lw == 2 && mode == 2) FACES_LAUNCH_FLOW(2, 2, 1);
      else if (lw == 2) FACES_LAUNCH_FLOW(2, 0, 1);
    }
  } else if (lw == 3) {
    // the partner regions in 16-byte pairs too
    if (mode == 2) FACES_LAUNCH_PAIRS(2, 0);
    else if (mode == 1) FACES_LAUNCH_PAIRS(1, 0);
    else FACES_LAUNCH_PAIRS(0, 0);
  } else if constexpr (narrow) {
    if (mode == 3) {
      FACES_LAUNCH_FLOW(2, 3, 0);
    } else if (mode == 2) {
      if (lw == 2) FACES_LAUNCH_FLOW(2, 2, 0);
      else if (lw == 1) FACES_LAUNCH_FLOW(1, 2, 0);
      else FACES_LAUNCH_FLOW(0, 2, 0);
    } else if (mode == 1) {
      if (lw == 2) FACES_LAUNCH_FLOW(2, 1, 0);
      else if (lw == 1) FACES_LAUNCH_FLOW(1, 1, 0);
      else FACES_LAUNCH_FLOW(0, 1, 0);
    } else {
      if (lw == 2) FACES_LAUNCH_FLOW(2, 0, 0);
      else if (lw == 1) FACES_LAUNCH_FLOW(1, 0, 0);
      else FACES_LAUNCH_FLOW(0, 0, 0);
    }
  }
#undef FACES_LAUNCH_FLOW
#undef FACES_LAUNCH_PAIRS
  FACES_HIP(hipGetLastError());
  return FACES_OK;
}

template <int N>
int launch_flow_n(int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                  const SurfWork *W, hipStream_t st)
{
#define FACES_FLOW_LEN(SS)                                                                         \
  if constexpr (flow_case(N, SS))                                                                  \
    if (S == SS) return launch_flow_ns<N, SS>(lw, mode, tree, G, F, nb, W, st);
  FACES_FLOW_LEN(1) FACES_FLOW_LEN(2) FACES_FLOW_LEN(3) FACES_FLOW_LEN(4) FACES_FLOW_LEN(5) FACES_FLOW_LEN(6)
  FACES_FLOW_LEN(8) FACES_FLOW_LEN(10) FACES_FLOW_LEN(12) FACES_FLOW_LEN(16) FACES_FLOW_LEN(24) FACES_FLOW_LEN(32)
  FACES_FLOW_LEN(64)
#undef FACES_FLOW_LEN
  return fail(FACES_ERR_ARG, "one-item kernel has no n=%d S=%d specialisation", N, S);
}


// The n of one group, dispatched to launch_flow_n<N>.
#define FACES_FLOW_GROUP(NAME, ...)                                                                       \
  int NAME(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb, \
           const SurfWork *W, hipStream_t st)                                                          \
  {                                                                                                    \
    switch (n) {                                                                                       \
      __VA_ARGS__                                                                                      \
      default: return fail(FACES_ERR_ARG, "one-item kernel has no n=%d specialisation", n);       \
    }                                                                                                  \
  }
#define FACES_FLOW_CASE(NN) \
  case NN: return launch_flow_n<NN>(S, lw, mode, tree, G, F, nb, W, st);

int launch_flow_g0(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st);  // n = 2, 3
int launch_flow_g1(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st);  // n = 4, 5
int launch_flow_g2(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st);  // n = 6, 7, 8
int launch_flow_g3(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st);  // n = 9, 10
int launch_flow_g4(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st);  // n = 11, 12
int launch_flow_g5(int n, int S, int lw, int mode, int tree, const Geom &G, const FlowItems &F, unsigned nb,
                   const SurfWork *W, hipStream_t st);  // n = 13 to 16

}  // namespace faces
