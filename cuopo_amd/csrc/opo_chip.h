// opo_chip.h -- the interior of one large instance's crystal pass as one launch
// over the whole chip.
//
// From 2^15 samples one XCD's 32 CUs are too few for an instance, and the
// two-launch path leaves a kernel boundary of about 4 us in a stage of 5.7 us
// (2^16, FP32C) to 13.5 us (2^18, FP64).  Here one block per CU, over all
// XCDs, runs every slice with a barrier in place of the boundary; each row (a
// field's team of N2/ER threads) and each column tile (a wavefront per field)
// keeps to one block.  Per slice, two-launch -> this, three equations: 2^15
// 10.2 -> 8.5 us FP64, 9.9 -> 8.0 FP32C (one XCD's team: 9.4 FP64); 2^16 13.3
// -> 9.7, 11.7 -> 8.6; 2^17 17.7 -> 13.0, 14.7 -> 10.3; 2^18 28.5 -> 20.7,
// 20.7 -> 14.7; with 4 samples per thread in the columns 10.4 -> 7.6 at 2^15,
// 13.3 -> 9.6 at 2^16, 28.9 -> 25.2 at 2^18 (FP64).  What bounds it: a stage
// at 2^16 is 2.9 us of exchange (below) beside 1.4 to 1.9 us of transforms
// with one wavefront per SIMD; at 2^18 12.6 MB pass through the fabric twice
// per stage (3.7 to 4.0 us) beside the transforms (4 us of FP64 on the CUs
// that hold two of the 384 rows).
//
// Memory order.  Blocks read what other XCDs wrote, so the fields are stored at
// agent scope as well as loaded (sc1: past the XCD's L2); a block waits for its
// stores (vmcnt), then adds one to one of 64 counters, which a wavefront of
// every waiting block polls, a counter a lane.  What that rests on, in the
// AMDGPU backend's memory model for gfx942 and gfx950: stores and loads marked
// sc1 are the model's relaxed atomic accesses of agent scope, coherent at every
// address over all L2s of the device; and vmcnt reaches zero when a store is
// complete at its scope, so the counter moves after the data.  The model's
// agent fences add a write-back and an invalidation of the L2, for accesses
// without sc1, which the fields do not have here.  It names accesses of up to 8
// bytes; a 16-byte one carries the same bits and is taken as two of those: no
// more is needed, as the counter orders them.  The tests compare every grid,
// type and equation set with the stage launches bit for bit.  Load, store and barrier of 3 MB
// of fields (2^16, FP64) take 2.9 us on 192 blocks so; with one counter per XCD
// and one for the XCDs 3.3, with a flag per block 3.2 to 4.1, with one counter
// 6.8 (256 blocks).
//
// No block waits for one that is not running: the first block to start closes
// the launch's team once all have joined, or after a short window, and the
// rows and tiles are dealt over the blocks that joined (as in opo_resident.h).
#pragma once

#include "opo_resident.h"

namespace opo {

// One word per XCD: valid, blocks in all, first rank of this XCD.
constexpr unsigned kChipValid = 1u << 31;
static_assert(kChipBlocks < 512, "nine bits each");

static_assert(kChipCounters <= kMaxTeams * kXcds, "one line each of ResSync::team");
constexpr int kChipThreads = 512;

// Teams per block: enough for all rows (tiles) in one turn of the full chip, if they fit.
template <int N1, int N2, int NF, int ER> __host__ __device__ constexpr int chip_rows() {
  const int units = NF * N1, need = (units + kChipBlocks - 1) / kChipBlocks, fit = kChipThreads / (N2 / ER);
  return need < fit ? need : fit;
}
template <int N1, int N2, int NF, int EC> __host__ __device__ constexpr int chip_cols() {
  const int tiles = N1 * N2 / (64 * EC), need = (tiles + kChipBlocks - 1) / kChipBlocks, fit = kChipThreads / (64 * NF);
  return need < fit ? need : fit;
}
template <int N1, int N2, int NF, int EC, int ER> __host__ __device__ constexpr int chip_threads() {
  const int r = chip_rows<N1, N2, NF, ER>() * (N2 / ER), c = chip_cols<N1, N2, NF, EC>() * 64 * NF;
  return r > c ? r : c;
}
template <int N1, int N2, int NF, int EC, int ER> __host__ __device__ constexpr int chip_lds_elems() {
  const int r = chip_rows<N1, N2, NF, ER>() * 2 * (N2 + N2 / 8), c = chip_cols<N1, N2, NF, EC>() * NF * 64 * EC;
  return N1 + (r > c ? r : c);
}

template <typename T, int N1, int N2, int NF, int EC, int ER>
__global__ __launch_bounds__((chip_threads<N1, N2, NF, EC, ER>())) void chip_pass(const OpoInst *__restrict__ insts,
                                                                                 ResArgs a) {
  using V = typename vec2<T>::type;
  constexpr int T2 = N2 / ER;
  constexpr int GR = chip_rows<N1, N2, NF, ER>(), GC = chip_cols<N1, N2, NF, EC>();
  constexpr int NROW = NF * N1, NTC = N1 * N2 / (64 * EC);
  constexpr unsigned N = N1 * N2;
  constexpr int NP2 = N2 + N2 / 8;
  static_assert(T2 % 64 == 0 && N1 / EC <= 64, "rows of whole wavefronts, columns of one");
  extern __shared__ __align__(16) unsigned char smem_raw[];  // (the static words before it are not a multiple of 16 bytes)
  __shared__ unsigned sh_rank, sh_word;
  __shared__ int sh_ok;
  V *ltw = reinterpret_cast<V *>(smem_raw);  // N1-point root table
  V *lds = ltw + N1;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);

  // ---- join ----
  const unsigned x = xcc_id();
  ResSync *S = reinterpret_cast<ResSync *>(a.sync);
  if (tid == 0) {
    unsigned word = 0;
    const unsigned old = agent_add(&S->join[x].v, 1u);
    if (old < kTeamClosed) {
      if (agent_add(&S->next.v, 1u) == 0) {
        const unsigned long long t0 = wall_clock64();
        for (;;) {
          unsigned n = 0;
#pragma unroll
          for (int i = 0; i < kXcds; ++i) n += agent_load(&S->join[i].v);
          if (n >= (unsigned)a.expect || wall_clock64() - t0 >= kJoinTicks) break;
        }
        unsigned nx[kXcds], total = 0;
#pragma unroll
        for (int i = 0; i < kXcds; ++i) {
          nx[i] = __hip_atomic_fetch_or(&S->join[i].v, kTeamClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          total += nx[i];
        }
        unsigned at = 0;
#pragma unroll
        for (int i = 0; i < kXcds; ++i) {
          agent_store(&S->size[i].v, kChipValid | (total << 9) | at);
          at += nx[i];
        }
      }
      if (!poll_until(&S->size[x].v, a.polls, [](unsigned v) { return v != 0; }, &word)) agent_store(&a.err[0], 1);
    }
    sh_rank = old;
    sh_word = word;
  }
  {
    const auto tw1 = gp(reinterpret_cast<const V *>(a.tw1));
    for (int e = tid; e < N1; e += blockDim.x) ltw[e] = tw1[e];
  }
  __syncthreads();
  const unsigned word = __builtin_amdgcn_readfirstlane(sh_word);
  if (word == 0) return;
  const int rank = (int)(__builtin_amdgcn_readfirstlane(sh_rank) + (word & 511u));
  const int size = (int)((word >> 9) & 511u);
  unsigned *mine_cnt = &S->team[rank & (kChipCounters - 1)].part[0].v;

  const auto I = cp_scalar(insts);
  if (!a.always && I->active_v == 0) return;
  const FieldBuf<V> in(reinterpret_cast<V *>(I->state), NF * N * (unsigned)sizeof(V));
  const double *nl = I->nl;
  const double h6 = I->h6;
  unsigned stages = 0;  // finished

  auto wait_all = [&]() -> bool {
    if (stages == 0) return true;
    if (tid < kChipCounters) {
      const unsigned need = stages * (unsigned)((size + kChipCounters - 1 - tid) / kChipCounters);
      bool ok = false;
      for (unsigned n = 0; n < a.polls && !ok; ++n) {
        ok = __all((int)(agent_load(&S->team[tid].part[0].v) - need) >= 0);
        if (!ok) __builtin_amdgcn_s_sleep(1);
      }
      if (tid == 0) {
        if (!ok) agent_store(&a.err[0], 3);
        sh_ok = ok;
      }
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(sh_ok) != 0;
  };
  auto arrive = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    ++stages;
    if (tid == 0) agent_add(mine_cnt, 1u);
  };

  for (int s = 0; s < a.NZ; ++s) {
    // ---- row stage ----
    {
      const int l = opaque(tid);
      const int t = l & (T2 - 1);
      const int grp = __builtin_amdgcn_readfirstlane(tid / T2);
      const bool mine = grp < GR;
      bool waited = false;
      auto wait = [&]() { return waited || (waited = wait_all()); };
      // consecutive rows on different blocks: a last turn of few rows spreads out
      for (int u0 = 0; u0 < NROW; u0 += size * GR) {
        const int u = u0 + grp * size + rank;
        const bool on = mine && u < NROW;
        const int f = on ? u / N1 : 0, k1 = on ? u % N1 : 0;
        if (!row_tile<N1, N2, ER, true>(in, a, I, f, k1, t, on, mine, lds, (mine ? grp : 0) * NP2, GR * NP2, wait)) return;
        __syncthreads();  // the next row's first pass writes the buffer that this one read last
      }
      if (!wait()) return;
      arrive();
    }
    if (s == a.NZ - 1) break;
    // ---- column stage ----
    {
      const int l = opaque(tid & 63);
      const int sub = wave / NF, f = wave - sub * NF;
      const bool mine = sub < GC;
      const NlCoef<NF, V> nle = load_nl_at<NF, V>(cp_scalar(nl) + 16 * s, h6);
      const NlCoef<NF, V> nls = load_nl_at<NF, V>(cp_scalar(nl) + 16 * (s + 1), h6);
      bool waited = false;
      auto wait = [&]() { return waited || (waited = wait_all()); };
      // neighbouring columns on one block: they share cache lines
      for (int t0 = 0; t0 < NTC; t0 += size * GC) {
        const int tile = t0 + rank * GC + sub;
        const bool on = mine && tile < NTC;
        V *buf = lds + (mine ? sub : 0) * (NF * 64 * EC);
        if (!col_tile<N1, N2, NF, EC, true>(in, a, f, tile, l, on, mine, buf, ltw, nle, nls, wait)) return;
      }
      if (!wait()) return;
      arrive();
    }
  }
}

template <typename T, int N1, int N2, int NF, int EC, int ER>
int launch_chip_k(const OpoInst *insts, ResArgs a, hipStream_t s) {
  using V = typename vec2<T>::type;
  constexpr int threads = chip_threads<N1, N2, NF, EC, ER>();
  constexpr size_t lds = (size_t)chip_lds_elems<N1, N2, NF, EC, ER>() * sizeof(V);
  static_assert(lds <= (size_t)kMaxDynLds, "LDS");
  // blocks that have a row or a tile
  constexpr int gr = (NF * N1 + chip_rows<N1, N2, NF, ER>() - 1) / chip_rows<N1, N2, NF, ER>();
  constexpr int gc = (N1 * N2 / (64 * EC) + chip_cols<N1, N2, NF, EC>() - 1) / chip_cols<N1, N2, NF, EC>();
  constexpr int work = gr > gc ? gr : gc;
  constexpr int grid = work < kChipBlocks ? work : kChipBlocks;
  auto kern = &chip_pass<T, N1, N2, NF, EC, ER>;
  static std::once_flag big_lds[kMaxDevices];
  if (lds > 64 * 1024 - 64) {
    const int rc = opt_in_big_lds(reinterpret_cast<const void *>(kern), big_lds, kMaxDynLds);
    if (rc != 0) return rc;
  }
  a.expect = grid;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, s, insts, a);
  return (int)hipGetLastError();
}

// 8 samples per thread in rows (with 4 their teams would not fit a block), 8 or 4 in columns
template <typename T, int N1, int N2>
int launch_chip_n(int NF, int ce, const OpoInst *insts, const ResArgs &a, hipStream_t s) {
  if (ce == 8)
    return NF == 3 ? launch_chip_k<T, N1, N2, 3, 8, 8>(insts, a, s) : launch_chip_k<T, N1, N2, 2, 8, 8>(insts, a, s);
  return NF == 3 ? launch_chip_k<T, N1, N2, 3, 4, 8>(insts, a, s) : launch_chip_k<T, N1, N2, 2, 4, 8>(insts, a, s);
}

}  // namespace opo
