// opo_resident.h -- the interior of a crystal pass as one launch.
//
// Two launches per slice pay a kernel boundary per stage: about 3.8 us on an
// idle MI355X for a 2^14-sample instance whose stages need 1-2 us of work, and
// a batch streams every field through the fabric twice per slice.  Here the
// blocks of one XCD form teams; a team takes an instance from a queue and runs
// all of its slices (row stage, column stage, ...) with a counter barrier in
// place of the kernel boundary.  The instance's fields stay in that XCD's
// 4 MiB L2 between stages.
//
// Barrier and memory order.  Blocks of one team share an L2.  Stores go
// through the L1 to the L2, so a block waits for its stores (vmcnt) and then
// adds one to a counter of the team; the readers poll the counters and load the
// fields with agent scope (sc1), which passes the L1 over.  Eight counters a
// team, a lane of one wavefront polling each: atomic adds to one line follow
// each other (2^14, three equations, six handles: 7.33 us per slice with
// one counter, 7.14 with eight; sixteen are no better).  No fence is
// needed: agent-scope acquire (buffer_inv sc1) takes 5 us per stage here and
// the release's write-back of the L2 more.  Measured for 0.75 MB per stage,
// load + store only, one block per CU: 1.6 us a stage on one XCD, 1.65 us with
// all eight XCDs busy, 7.0 us with the fences.
//
// No block waits for one that is not running.  A block joins its XCD's team by
// an atomic add; the first one waits until all expected blocks have joined, or
// a short window has passed, and closes the team with the size it has then.
// Later blocks leave at once.  Tiles are dealt over the blocks that did join,
// so any number of them finishes the work.  Every wait is bounded by a count
// as well: on a time-out the blocks leave and the host reports an error.
//
// Which XCD a block runs on is read from the hardware (XCC_ID), never assumed
// from the block index.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "opo_device.h"
#include "opo_handoff.h"
#include "opo_internal.h"

namespace opo {

constexpr unsigned kTeamClosed = 1u << 20;
constexpr unsigned long long kJoinTicks = 2000;          // 20 us of the 100 MHz clock

__device__ __forceinline__ unsigned xcc_id() {
  return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & (kXcds - 1);  // hwreg(HW_REG_XCC_ID, 0, 4)
}
template <typename T> __device__ __forceinline__ T agent_add(T *p, T v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ T agent_load(T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void agent_store(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polls until f(value) holds, then *got is that value; false after `polls` reads.
template <typename T, typename F> __device__ __forceinline__ bool poll_until(T *p, unsigned polls, F f, T *got) {
  for (unsigned n = 0; n < polls; ++n) {
    const T v = agent_load(p);
    if (f(v)) {
      *got = v;
      return true;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}

// The launch's queue and a team's word, for hand_out and hand_in.
struct TeamQueue {
  ResSync *S;
  ResTeam *tm;
  unsigned polls;
  __device__ __forceinline__ unsigned take() { return agent_add(&S->next.v, 1u); }
  __device__ __forceinline__ void publish(unsigned long long w) { agent_store(&tm->cur, w); }
  __device__ __forceinline__ bool await(unsigned turn, unsigned long long *w) {
    return poll_until(&tm->cur, polls, [turn](unsigned long long v) { return is_turn(v, turn); }, w);
  }
};

// Coherent loads of the instance's fields: 16- (8-) byte buffer loads at agent
// scope.  `off` in elements.
template <typename V> struct FieldBuf {
  __amdgpu_buffer_rsrc_t r;
  V *base;
  __device__ __forceinline__ FieldBuf(V *p, unsigned bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00020000)), base(p) {}
  __device__ __forceinline__ V load(unsigned off) const {
    constexpr int kAgent = 16;  // sc1
    if constexpr (sizeof(V) == 16) {
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      const u4 w = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off * 16), 0, kAgent);
      return __builtin_bit_cast(V, w);
    } else {
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      const u2 w = __builtin_amdgcn_raw_buffer_load_b64(r, (int)(off * 8), 0, kAgent);
      return __builtin_bit_cast(V, w);
    }
  }
  // WIDE: past this XCD's L2 as well (agent scope), for readers on the others
  template <bool WIDE> __device__ __forceinline__ void store(unsigned off, V v) const {
    if constexpr (!WIDE) {
      gp(base)[off] = v;
    } else if constexpr (sizeof(V) == 16) {
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, (int)(off * 16), 0, 16);
    } else {
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, (int)(off * 8), 0, 16);
    }
  }
};

// The same value, as far as the compiler can see a new one each time: keeps
// the offsets and addresses formed from it inside a stage instead of hoisted
// out of the slice loop into registers that the transforms need.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// One wavefront per field of a tile: 64*E samples of each field, as 64*EC/N1
// columns or 64*ER/N2 rows.  A block holds `sub` tiles side by side.
template <int NF, int EC, int ER> __host__ __device__ constexpr int res_tile_elems() {
  return NF * (64 * EC > 72 * ER ? 64 * EC : 72 * ER);  // rows carry one pad slot per 8 samples
}

// Row k1 of field f by the thread's team of N2/ER threads (t: its index):
// FFT, linear phase, inverse FFT.  `on`: there is such a row; `mine`: the
// thread has a part of the LDS.  `wait` returns once the stage before is
// complete; phases and twiddles are constant, so their loads go out before.
template <int N1, int N2, int ER, bool WIDE, typename V, typename D, typename Wait>
__device__ __forceinline__ bool row_tile(const FieldBuf<V> &in, const ResArgs &a, D I, int f, int k1, int t, bool on,
                                         bool mine, V *buf, int gbase, int bufstride, Wait wait) {
  constexpr unsigned N = N1 * N2;
  constexpr int T2 = N2 / ER;
  constexpr bool wave = team_in_wave(T2);
  const unsigned row = f * N + N2 * k1;
  constexpr int NTW = tw_count(N2, ER, tw_pow<V>());
  V v[ER], ph_tab[ER], treg[NTW > 0 ? NTW : 1];
  V xr = mk<V>(0, 0);
  const auto lfac = gp(reinterpret_cast<const V *>(I->lfac_spt[ER == 8 ? 0 : 1]));
  const bool use_fac = (bool)lfac;
  if (use_fac) {
    const int L = a.xl_bits;
    const long long FB = (long long)ER * N1 + N2 + ((N / ER) >> L) + (1LL << L);
    const auto F = lfac + f * FB;
    const auto Sx = F + ER * N1;
    const auto XH = Sx + N2;
    const auto XL = XH + ((N / ER) >> L);
    const unsigned e = (unsigned)k1 * (unsigned)t;
    xr = cmul(V(XL[e & ((1u << L) - 1u)]), V(XH[e >> L]));
#pragma unroll
    for (int m = 0; m < ER; ++m) ph_tab[m] = cmul(V(Sx[t + m * T2]), V(F[ER * k1 + m]));
  } else {
    const auto lin = gp(reinterpret_cast<const V *>(I->lin));
#pragma unroll
    for (int m = 0; m < ER; ++m) ph_tab[m] = lin[row + t + m * T2];
  }
  load_twiddles<N2, ER>(treg, t, gp(reinterpret_cast<const V *>(a.tw2)));
  if (!wait()) return false;
#pragma unroll
  for (int m = 0; m < ER; ++m) v[m] = in.load(row + t + m * T2);
  if (use_fac) {
#pragma unroll
    for (int m = 0; m < ER; ++m) ph_tab[m] = cmul(xr, ph_tab[m]);
  }
  int ph = 0;
  team_fft<N2, +1, true, true, ER>(v, mine, buf, ph, t, gbase, 1, bufstride, treg, wave);
#pragma unroll
  for (int m = 0; m < ER; ++m) v[m] = cmul(v[m], ph_tab[m]);
  team_fft<N2, -1, true, true, ER>(v, mine, buf, ph, t, gbase, 1, bufstride, treg, wave);
  if (on) {
#pragma unroll
    for (int m = 0; m < ER; ++m) in.template store<WIDE>(row + t + m * T2, v[m]);
  }
  return true;
}

// Field f of one tile of 64*EC/N1 columns, one wavefront: inverse FFT, NL end
// of slice s, NL start of s + 1 (over the tile's NF wavefronts), FFT.
template <int N1, int N2, int NF, int EC, bool WIDE, typename V, typename Wait>
__device__ __forceinline__ bool col_tile(const FieldBuf<V> &in, const ResArgs &a, int f, int tile, int lane, bool on,
                                         bool mine, V *lds, const V *ltw, const NlCoef<NF, V> &nle,
                                         const NlCoef<NF, V> &nls, Wait wait) {
  constexpr bool F64 = sizeof(V) == 16;
  constexpr unsigned N = N1 * N2;
  constexpr int T1 = N1 / EC, CT = 64 / T1;
  constexpr int fstride = 64 * EC;
  const int c = lane & (CT - 1), t = lane / CT;
  const int n2 = (on ? tile : 0) * CT + c;
  const unsigned at = f * N + n2;
  const auto twlo = gp(reinterpret_cast<const V *>(a.twlo));
  const auto twhi = gp(reinterpret_cast<const V *>(a.twhi));
  const unsigned lm = (1u << a.lobits) - 1u;
  // four-step twiddles as col_stage forms them (same products)
  V gh[F64 ? 1 : EC], gl[F64 ? 1 : EC], W[EC];
  V x0{}, b1{};
  if constexpr (F64) {
    const unsigned e0 = (unsigned)(n2 * t) & (N - 1), e1 = (unsigned)(n2 * T1) & (N - 1);
    const V x0h = twhi[e0 >> a.lobits], x0l = twlo[e0 & lm];
    const V b1h = twhi[e1 >> a.lobits], b1l = twlo[e1 & lm];
    x0 = cmul(x0h, x0l);
    b1 = cmul(b1h, b1l);
  } else {
#pragma unroll
    for (int m = 0; m < EC; ++m) {
      const unsigned e = (unsigned)(n2 * (t + m * T1)) & (N - 1);
      gh[m] = twhi[e >> a.lobits];
      gl[m] = twlo[e & lm];
    }
#pragma unroll
    for (int m = 0; m < EC; ++m) W[m] = cmul(gh[m], gl[m]);
  }
  if (!wait()) return false;
  V v[EC];
#pragma unroll
  for (int m = 0; m < EC; ++m) v[m] = in.load(at + N2 * (t + m * T1));
  auto roots = [&]() {
    if constexpr (F64) {
      const V b2 = cmul(b1, b1), b4 = cmul(b2, b2);
#pragma unroll
      for (int m = 0; m < EC; ++m) {
        V w = x0;
        if (m & 4) w = cmul(w, b4);
        if (m & 2) w = cmul(w, b2);
        if (m & 1) w = cmul(w, b1);
        W[m] = w;
      }
    }
  };
  roots();
  int ph = 0;
  V *own = lds + f * fstride;
#pragma unroll
  for (int m = 0; m < EC; ++m) v[m] = cmul(v[m], cconj(W[m]));
  team_fft<N1, -1, false, false, EC>(v, mine, own, ph, t, c, CT, 0, ltw, true);
#pragma unroll
  for (int m = 0; m < EC; ++m)
    if (mine) own[c + (t + m * T1) * CT] = v[m];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < EC; ++m) {
    if (mine && m % NF == f) {
      const int o = c + (t + m * T1) * CT;
      V xp[1] = {lds[o]}, xq[1] = {lds[fstride + o]};
      V xi[1] = {NF == 3 ? lds[2 * fstride + o] : mk<V>(0, 0)};
      nl_half_pt<NF, 1>(xp, xq, xi, nle);
      nl_half_pt<NF, 1>(xp, xq, xi, nls);
      lds[o] = xp[0];
      lds[fstride + o] = xq[0];
      if constexpr (NF == 3) lds[2 * fstride + o] = xi[0];
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < EC; ++m) v[m] = own[c + (t + m * T1) * CT];
  team_fft<N1, +1, false, false, EC>(v, mine, own, ph, t, c, CT, 0, ltw, true);
  if constexpr (F64) {
    // W again from its two roots (see col_stage)
    asm volatile("" : "+v"(x0.x), "+v"(x0.y), "+v"(b1.x), "+v"(b1.y));
    roots();
  }
#pragma unroll
  for (int m = 0; m < EC; ++m) v[m] = cmul(v[m], W[m]);
  if (on) {
#pragma unroll
    for (int m = 0; m < EC; ++m) in.template store<WIDE>(at + N2 * (t + m * T1), v[m]);
  }
  return true;
}

template <typename T, int N1, int N2, int NF, int EC, int ER>
__global__ __launch_bounds__(kResThreads) void resident_pass(const OpoInst *__restrict__ insts, ResArgs a) {
  using V = typename vec2<T>::type;
  constexpr int T1 = N1 / EC, T2 = N2 / ER;
  constexpr int CT = 64 / T1, RT = 64 / T2;
  constexpr int NTC = N2 / CT, NTR = N1 / RT;
  constexpr unsigned N = N1 * N2;
  static_assert(T1 <= 64 && T2 <= 64 && NTC >= 1 && NTR >= 1, "one wavefront per field");
  extern __shared__ __align__(16) unsigned char smem_raw[];  // (the static words before it are not a multiple of 16 bytes)
  __shared__ unsigned sh_next[2];
  __shared__ int sh_rank, sh_size, sh_ok;
  V *ltw = reinterpret_cast<V *>(smem_raw);  // N1-point root table
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int sub = wave / NF, f = wave - sub * NF;  // uniform over the wavefront
  const int lane = tid & 63;
  V *lds = ltw + N1 + sub * res_tile_elems<NF, EC, ER>();

  // ---- join this XCD's blocks ----
  const unsigned x = xcc_id();
  ResSync *S = reinterpret_cast<ResSync *>(a.sync);
  if (tid == 0) {
    const unsigned old = agent_add(&S->join[x].v, 1u);
    int size = 0;
    if (old >= kTeamClosed) {
      size = -1;
    } else if (old == 0) {
      const unsigned long long t0 = wall_clock64();
      while (agent_load(&S->join[x].v) < (unsigned)a.expect && wall_clock64() - t0 < kJoinTicks) {
      }
      size = (int)__hip_atomic_fetch_or(&S->join[x].v, kTeamClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      agent_store(&S->size[x].v, (unsigned)size);
    } else {
      unsigned closed = 0;
      if (!poll_until(&S->size[x].v, a.polls, [](unsigned v) { return v != 0; }, &closed)) {
        agent_store(&a.err[0], 1);
        size = -1;
      } else {
        size = (int)closed;
      }
    }
    sh_rank = (int)old;
    sh_size = size;
  }
  {
    const auto tw1 = gp(reinterpret_cast<const V *>(a.tw1));
    for (int e = tid; e < N1; e += blockDim.x) ltw[e] = tw1[e];
  }
  __syncthreads();
  const int xs = __builtin_amdgcn_readfirstlane(sh_size);
  if (xs < 0) return;
  // teams of consecutive ranks: blocks that start together sit on different
  // CUs, so each CU holds blocks of several teams and one team's waits are
  // filled by another's arithmetic
  const int per = (xs + a.teams - 1) / a.teams;
  const int rank = __builtin_amdgcn_readfirstlane(sh_rank);
  const int team = rank / per, r0 = rank - team * per;
  const int size = min(per, xs - team * per);
  ResTeam *tm = &S->team[team * kXcds + x];
  const int nsub = a.sub, workers = size * nsub;
  const unsigned total = (unsigned)(a.count + a.count2);
  TeamQueue queue{S, tm, a.polls};
  auto inst = [&](unsigned i) { return i < (unsigned)a.count ? insts + i : a.insts2 + (i - (unsigned)a.count); };
  unsigned arrived = 0;  // stages finished

  for (unsigned epoch = 1;; ++epoch) {
    // ---- the team's next instance ----
    if (tid == 0) {
      unsigned i = ~0u;
      if (r0 == 0) {
        if (epoch == 1 && a.spread) {
          // fewer instances than teams: each launch prefers an XCD of its own,
          // so that solvers running side by side do not share one
          const unsigned long long t0 = wall_clock64();
          const unsigned long long d = ((x - (unsigned)a.prefer) & (kXcds - 1)) * 30ull + team * 240ull;
          while (wall_clock64() - t0 < d) {
          }
        }
        i = hand_out(queue, epoch, total, [&](unsigned k) { return a.always || inst(k)->active_v != 0; });
      } else if (!hand_in(queue, epoch, &i)) {
        agent_store(&a.err[0], 2);  // (i stays past the end: the block leaves)
      }
      sh_next[epoch & 1] = i;
    }
    __syncthreads();
    const unsigned idx = __builtin_amdgcn_readfirstlane(sh_next[epoch & 1]);
    if (idx >= total) return;
    const auto I = cp_scalar(inst(idx));
    V *state = reinterpret_cast<V *>(I->state);
    const FieldBuf<V> in(state, NF * N * (unsigned)sizeof(V));
    const double *nl = I->nl;
    const double h6 = I->h6;
    bool first = true;

    // Waits until every block of the team has finished the stage before.
    auto wait_team = [&]() -> bool {
      if (first) {
        first = false;
        return true;
      }
      if (tid < 64) {
        const int c = lane & (kTeamCounters - 1);
        const unsigned need = arrived * (unsigned)((size + kTeamCounters - 1 - c) / kTeamCounters);
        bool ok = false;
        for (unsigned n = 0; n < a.polls && !ok; ++n) {
          ok = lane >= kTeamCounters || (int)(agent_load(&tm->part[c].v) - need) >= 0;
          ok = __all(ok);
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
    // This block's stores have reached the L2: one arrival.
    auto arrive = [&]() {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) agent_add(&tm->part[r0 & (kTeamCounters - 1)].v, 1u);
      ++arrived;
    };

    for (int s = 0; s < a.NZ; ++s) {
      // ---- row stage: FFT, linear phase, inverse FFT of each row ----
      {
        const int l = opaque(lane);
        const int t = l & (T2 - 1), r = l / T2;
        bool waited = false;
        auto wait = [&]() { return waited || (waited = wait_team()); };
        for (int t0 = 0; t0 < NTR; t0 += workers) {
          const int tile = t0 + r0 * nsub + sub;
          const bool on = tile < NTR;
          const int k1 = (on ? tile : 0) * RT + r;
          V *buf = lds + f * (64 * ER + 8 * ER);
          constexpr int NP2 = N2 + N2 / 8;
          if (!row_tile<N1, N2, ER, false>(in, a, I, f, k1, t, on, true, buf, r * NP2, 0, wait)) return;
        }
        if (!wait()) return;  // (a block without a tile still keeps step)
        arrive();
      }
      if (s == a.NZ - 1) break;
      // ---- column stage: inverse FFT, NL end of slice s, NL start of s + 1, FFT ----
      {
        const int l = opaque(lane);
        const NlCoef<NF, V> nle = load_nl_at<NF, V>(cp_scalar(nl) + 16 * s, h6);
        const NlCoef<NF, V> nls = load_nl_at<NF, V>(cp_scalar(nl) + 16 * (s + 1), h6);
        bool waited = false;
        auto wait = [&]() { return waited || (waited = wait_team()); };
        for (int t0 = 0; t0 < NTC; t0 += workers) {
          const int tile = t0 + r0 * nsub + sub;
          const bool on = tile < NTC;
          if (!col_tile<N1, N2, NF, EC, false>(in, a, f, tile, l, on, true, lds, ltw, nle, nls, wait)) return;
        }
        if (!wait()) return;
        arrive();
      }
    }
    if (ends_with_wait(a.NZ) && !wait_team()) return;
  }
}

template <typename T, int N1, int N2, int NF, int EC, int ER>
int launch_resident_k(const OpoInst *insts, const ResArgs &a, int grid, hipStream_t s) {
  using V = typename vec2<T>::type;
  const int threads = 64 * NF * a.sub;
  const size_t lds = ((size_t)N1 + (size_t)a.sub * res_tile_elems<NF, EC, ER>()) * sizeof(V);
  if (a.sub < 1 || threads > kResThreads || lds > kMaxDynLds || grid < kXcds || a.teams < 1 ||
      a.teams > kMaxTeams)
    return (int)hipErrorInvalidValue;
  auto kern = &resident_pass<T, N1, N2, NF, EC, ER>;
  static std::once_flag big_lds[kMaxDevices];
  if (lds > 64 * 1024 - 64) {
    const int rc = opt_in_big_lds(reinterpret_cast<const void *>(kern), big_lds, kMaxDynLds);
    if (rc != 0) return rc;
  }
  hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, s, insts, a);
  return (int)hipGetLastError();
}

// Samples per thread: every pair that fits a wavefront, as the group is set.
template <typename T, int N1, int N2, int NF>
int launch_resident_n(int ce, int re, const OpoInst *insts, const ResArgs &a, int grid, hipStream_t s) {
  if (ce == 8 && re == 8) return launch_resident_k<T, N1, N2, NF, 8, 8>(insts, a, grid, s);
  if (ce == 4 && re == 8) return launch_resident_k<T, N1, N2, NF, 4, 8>(insts, a, grid, s);
  if constexpr (N2 <= 256) {
    if (ce == 4 && re == 4) return launch_resident_k<T, N1, N2, NF, 4, 4>(insts, a, grid, s);
    if (ce == 8 && re == 4) return launch_resident_k<T, N1, N2, NF, 8, 4>(insts, a, grid, s);
  }
  return (int)hipErrorInvalidValue;
}

template <typename T, int NF>
int launch_resident_t(int N1, int N2, int ce, int re, const OpoInst *insts, const ResArgs &a, int grid, hipStream_t s) {
  if (N1 == 32 && N2 == 32) return launch_resident_n<T, 32, 32, NF>(ce, re, insts, a, grid, s);
  if (N1 == 32 && N2 == 64) return launch_resident_n<T, 32, 64, NF>(ce, re, insts, a, grid, s);
  if (N1 == 64 && N2 == 64) return launch_resident_n<T, 64, 64, NF>(ce, re, insts, a, grid, s);
  if (N1 == 64 && N2 == 128) return launch_resident_n<T, 64, 128, NF>(ce, re, insts, a, grid, s);
  if (N1 == 64 && N2 == 256) return launch_resident_n<T, 64, 256, NF>(ce, re, insts, a, grid, s);
  if (N1 == 64 && N2 == 512) return launch_resident_n<T, 64, 512, NF>(ce, re, insts, a, grid, s);
  return (int)hipErrorInvalidValue;
}

}  // namespace opo
