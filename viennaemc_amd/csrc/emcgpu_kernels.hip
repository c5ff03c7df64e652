// emcgpu_kernels.hip -- gfx950 kernels of the EMC particle step.
//
// A wave owns 64 * PPT particles and keeps them on the chip for all steps fused
// into a launch, so HBM sees the SoA state once per launch: in LDS
// (k_bulk_fused), or, where a launch has one or a few steps, in registers
// (k_bulk_lanes) or streamed through (k_bulk_once).  Each step is the
// free-flight / scatter loop of basicBulkParticleHandler::moveParticles
// (examples/bulkSimulation/basicBulkParticleHandler.hpp:195-221):
//   drift min(tau, dt); while (dt - tau > 0) { scatter; tau += tau';
//   drift min(rem, tau'); rem -= tau' }; tau -= dt
// followed by the per-step ensemble sums (FP64 per lane, wave reductions,
// one FP64 partial per wave per step, combined by the compensated reduction
// k_reduce_chunks, with k_reduce_final where there are several chunks).
//
// Random numbers:
//   production: Philox-4x32-10 keyed by the seed, counter
//               (block, step, particle, instance); one counter block per
//               scatter event (4 words -> selection, two final-state
//               uniforms, free-flight time), 24-bit uniforms that FP64
//               widens, so both precisions follow the same random path.
//   replay:     the reference engine's recorded raw 64-bit draws, consumed
//               in the reference's order and mapped like libstdc++'s
//               generate_canonical (FP64 only).
#include <hip/hip_runtime.h>

#include "emcgpu_particle.h"

namespace emcgpu {

// ---------------------------------------------------------------------------
// wave-level reductions (wave64)
// ---------------------------------------------------------------------------
// DPP moves (GCN/CDNA data-parallel primitives): quad_perm [1,0,3,2] and
// [2,3,0,1], row_shr:4 and :8 within rows of 16 lanes, row_bcast:15 (rows 1
// and 3) and row_bcast:31 (rows 2 and 3); lanes without a source read 0, so
// after the six steps lane 63 holds the wave's sum, which readlane makes
// uniform.  VALU moves instead of LDS permutes.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_d(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = dpp_i<CTRL, ROWS>((int)(b & 0xffffffffll));
  const int hi = dpp_i<CTRL, ROWS>((int)(b >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double wave_sum(double x) {
  x = x + dpp_d<0xb1, 0xf>(x);
  x = x + dpp_d<0x4e, 0xf>(x);
  x = x + dpp_d<0x114, 0xf>(x);
  x = x + dpp_d<0x118, 0xf>(x);
  x = x + dpp_d<0x142, 0xa>(x);
  x = x + dpp_d<0x143, 0xc>(x);
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), 63);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ int wave_sum_i(int x) {
  x = x + dpp_i<0xb1, 0xf>(x);
  x = x + dpp_i<0x4e, 0xf>(x);
  x = x + dpp_i<0x114, 0xf>(x);
  x = x + dpp_i<0x118, 0xf>(x);
  x = x + dpp_i<0x142, 0xa>(x);
  x = x + dpp_i<0x143, 0xc>(x);
  return __builtin_amdgcn_readlane(x, 63);
}

// the wave's sums of e and v at once: the first stage leaves each lane one of
// them (v in the lanes whose parity is `vpar`, e in the others), the others
// reduce lanes of one parity, so two sums cost 26 instructions instead of 40
__device__ __forceinline__ double wave_sum_pair(double e, double v, int vpar) {
  const bool has_v = (int)(threadIdx.x & 1u) == vpar;
  double x = (has_v ? v : e) + dpp_d<0xb1, 0xf>(has_v ? e : v);  // with lane ^ 1
  x = x + dpp_d<0x4e, 0xf>(x);                                   // lane ^ 2
  x = x + dpp_d<0x124, 0xf>(x);                                  // rows rotated by 4, by 8
  x = x + dpp_d<0x128, 0xf>(x);
#pragma unroll
  for (int half = 0; half < 2; ++half) {  // across the rows of 16, then the halves
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    unsigned long long p, q;
    if (half == 0) {
      const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
      p = ((unsigned long long)h[0] << 32) | l[0];
      q = ((unsigned long long)h[1] << 32) | l[1];
    } else {
      const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
      p = ((unsigned long long)h[0] << 32) | l[0];
      q = ((unsigned long long)h[1] << 32) | l[1];
    }
    x = __builtin_bit_cast(double, p) + __builtin_bit_cast(double, q);
  }
  return x;
}

constexpr int kObsMax = 2 + kMaxV * (3 + kMaxDeg);
static_assert(kObsMax <= 64, "one lane per observable of a wave");

// Per-step ensemble sums of one wave (each lane holds PPT particles): event
// counts, per-valley count / sum E / sum v.dir, per-(valley, subvalley)
// counts.  Lanes sum their own particles in FP64, the wave reduces with
// shuffles and ballots, and lane o writes value o of the wave's partial:
// partial[step][obs][tile * kSubs + wave].  No block barrier: the waves of a
// block run their steps independently.
template <typename R, int PPT>
__device__ __forceinline__ void tile_observables(const StepArgs<R> &a, const InstDev<R> *P,
                                                 int tile, int s, const bool (&valid)[PPT],
                                                 const int (&v)[PPT], const int (&sub)[PPT],
                                                 const R (&kx)[PPT], const R (&ky)[PPT],
                                                 const R (&kz)[PPT], const R (&E)[PPT], int nev,
                                                 int nreal) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nv = P->n_valleys;
  double mine = 0.0;  // the value this lane writes
  const int ev = wave_sum_i(nev);
  const int re = wave_sum_i(nreal);
  mine = (lane == 0) ? (double)ev : mine;
  mine = (lane == 1) ? (double)re : mine;
  for (int vv = 0; vv < a.max_v; ++vv) {
    double se = 0.0, sv = 0.0;
    int cnt = 0;
    if (vv < nv) {
      double de = 0.0, dv = 0.0;
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const bool in = valid[j] && v[j] == vv;
        de += in ? (double)E[j] : 0.0;
        dv += in ? (double)vdir_of(kane_of(P->valley[vv]), P->valley[vv].wdir[sub[j]], kx[j], ky[j],
                                   kz[j], E[j])
                 : 0.0;
        cnt += (int)__popcll(__ballot(in));
      }
      se = wave_sum(de);
      sv = wave_sum(dv);
    }
    mine = (lane == 2 + 3 * vv) ? (double)cnt : mine;
    mine = (lane == 3 + 3 * vv) ? se : mine;
    mine = (lane == 4 + 3 * vv) ? sv : mine;
    for (int ss = 0; ss < a.max_deg; ++ss) {
      int c2 = 0;
#pragma unroll
      for (int j = 0; j < PPT; ++j)
        c2 += (int)__popcll(__ballot(valid[j] && v[j] == vv && sub[j] == ss));
      mine = (lane == 2 + 3 * a.max_v + vv * a.max_deg + ss) ? (double)c2 : mine;
    }
  }
  if (lane < a.n_obs)
    a.partial[((long long)s * a.n_obs + lane) * ((long long)a.n_tiles * kSubs) +
              (long long)tile * kSubs + wave] = mine;
}

// instance of a kernel tile of tile_size particles (tiles never straddle
// instances: instances start on kUnit boundaries and kUnit % tile_size == 0)
__device__ __forceinline__ int tile_instance(const int *unit_inst, long long tile, int tile_size) {
  return unit_inst[(tile * tile_size) / kUnit];
}

// ---------------------------------------------------------------------------
// phonon-bath tallies: each block counts its events in an LDS histogram of
// its instance's bins and adds the non-zero counts to the global 64-bit
// tallies once at the end
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ void tally_clear(const InstDev<R> *P, uint32_t *lds_tally) {
  for (int i = threadIdx.x; i < 2 * P->total_bins; i += kTile)
    lds_tally[i] = 0u;
  // the baths' window sums, read by the bisection of the q-resolved angle,
  // from LDS: they change only between steps (one step per launch here)
  if (P->win_lds) {
    R *dst = lds_window<R>(P, lds_tally);
    const R *src = P->bath_win[0];
    for (int i = threadIdx.x; i < 2 * (P->total_bins + P->n_baths); i += kTile)
      dst[i] = src[i];
  }
  __syncthreads();
}

template <typename R>
__device__ __forceinline__ void tally_flush(const InstDev<R> *P, const uint32_t *lds_tally,
                                            unsigned long long *tally, long long tally_bins) {
  __syncthreads();
  unsigned long long *g =
      tally + 2 * ((long long)(blockIdx.x % kTallyCopies) * tally_bins + P->gbin_off);
  for (int i = threadIdx.x; i < 2 * P->total_bins; i += kTile) {
    const uint32_t c = lds_tally[i];
    if (c)
      atomicAdd(&g[i], (unsigned long long)c);
  }
}

// ---------------------------------------------------------------------------
// production step kernel
//
// A wave owns 64 * PPT particles (particle j * 64 + l of wave w in a tile of
// 256 * PPT is tile_first + j * 256 + w * 64 + l, so every load and store is
// a contiguous 64-wide access) and keeps their state in LDS for all steps of
// the launch.  Each step every particle drifts min(tau, dt) on its own lane.
// A particle with time left (about a fifth of them per 1 fs step in Si) is
// queued; the wave's 64 lanes then work on queued particles, one scatter
// event each per pass, whichever lane the particles belong to.  A particle
// that has a further event in the step keeps its worker lane and goes on in
// the next step's pass, behind the others (at most kRing - 1 steps); the sums
// of a step are complete, and written, when no particle lags behind it.  The
// random numbers are indexed by (event, step, particle), so the order of the
// work does not change a history.  No barriers are involved.
//
// Bound by vector-ALU issue.  An event loop on the lane that owns the particle
// runs the scatter body while any lane has an event left: 3.8 passes per step
// of 256 Si particles (50 kV/cm, 1 fs) at a quarter of the lanes, 1300 VALU
// instructions; here 1.1 passes and 600.  10M particles FP32, 64 steps,
// with the step sums: 4.39 -> 2.42 ms; 4M of the two-valley model FP64 (0.03
// events per particle and step, a pass every fourth step), 16 steps: 1.12 ->
// 0.57 ms.
// ---------------------------------------------------------------------------
// steps that a particle may lag behind, plus one: the sums of this many
// steps are held in LDS
constexpr int kRing = 8;
// a pass is run while this many particles have an event pending (a wave has
// 64 lanes); fewer wait for the next step's.  us per step, 10M Si FP32 (64
// steps) / 4M two-valley FP64 (16 steps): 8 pending 42.3 / 37.3, 16 40.5 /
// 34.4, 24 40.1 / 33.4, 28 40.3 / 33.6, 32 39.8 / 33.4, 40 40.0 / 33.4, 48
// 40.7 / 33.4, 64 48.1 / 33.5
constexpr int kPass = 28;
// valley/subvalley word in LDS: not with its home lane, in step at kAtShift
constexpr uint32_t kAway = 0x80000000u;
constexpr int kAtShift = 24;
constexpr uint32_t kVsMask = 0x00FFFFFFu;
static_assert(kMaxV <= 256 && kRing <= 128, "valley, step tag and kAway share a word");

// a wave's particles in LDS: k, tau (and the position), the valley/subvalley
// word, the queue's index; the energy follows from k.  Its kRing * n_obs
// sums come after.  Less LDS is more waves: Si FP32 with the energy and a
// ring of 16 leaves 4 blocks per CU (2.91 ms at 10M), with a ring of 8 five
// (2.62 ms).
template <int PPT>
struct QueueIndex {
  typedef uint8_t type;
};
template <>
struct QueueIndex<8> {
  typedef uint16_t type;
};
template <typename R, int PPT, bool POS>
constexpr size_t fused_state_bytes() {
  return (size_t)64 * PPT *
         ((POS ? 7 : 4) * sizeof(R) + sizeof(uint32_t) + sizeof(typename QueueIndex<PPT>::type));
}

// the instance's parameters: valleys and mechanisms come last in InstDev, so
// a prefix holds what the instance uses
template <typename R>
__device__ __forceinline__ const InstDev<R> *stage_params(unsigned char *lds, const InstDev<R> *src,
                                                          int bytes) {
  static_assert(sizeof(InstDev<R>) % 8 == 0, "8-byte copy");
  const unsigned long long *s = reinterpret_cast<const unsigned long long *>(src);
  unsigned long long *d = reinterpret_cast<unsigned long long *>(lds);
  const int n = bytes < (int)sizeof(InstDev<R>) ? bytes : (int)sizeof(InstDev<R>);
  for (int i = threadIdx.x; i < n / 8; i += kTile)
    d[i] = s[i];
  __syncthreads();
  return reinterpret_cast<const InstDev<R> *>(lds);
}

__device__ __forceinline__ int lanes_below(unsigned long long mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                        __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// energy and velocity sums of one step over the particles in step with the
// wave, per lane in FP64
template <typename R, int NV>
struct StepSums {
  double e[NV], v[NV];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < NV; ++k)
      e[k] = v[k] = 0.0;
  }
  // the active lanes enter a particle each
  __device__ __forceinline__ void add(const InstDev<R> *P, const Kane<R> &K, int vv, int ss, R kx,
                                      R ky, R kz, R E) {
    const double de = (double)E;
    const double dv = (double)vdir_of(K, P->valley[NV == 1 ? 0 : vv].wdir[ss], kx, ky, kz, E);
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (NV == 1 || vv == k) {
        e[k] += de;
        v[k] += dv;
      }
  }
  // value `lane` of the step's sums, events and real events included; the
  // counts are kept apart
  __device__ __forceinline__ double total(const StepArgs<R> &a, int nev, int nreal) const {
    const int lane = threadIdx.x & 63;
    double mine = 0.0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (k < a.max_v) {
        const double x = wave_sum_pair(e[k], v[k], k & 1);  // lane 3 + 3 k: e, the next: v
        mine = (unsigned)(lane - 3 - 3 * k) < 2u ? x : mine;
      }
    }
    mine = (lane == 0) ? (double)nev : mine;
    return (lane == 1) ? (double)nreal : mine;
  }
};

// the lanes' common value, in scalar registers
__device__ __forceinline__ float uniform_value(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
__device__ __forceinline__ double uniform_value(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}
template <typename R, int NV>
__device__ __forceinline__ auto kane_source(const InstDev<R> *P) {
  if constexpr (NV == 1) {
    const ValleyDev<R> &V = P->valley[0];
    return KaneOne<R>{{uniform_value(V.c2), uniform_value(V.alpha), uniform_value(V.cv)}};
  } else {
    return KaneAny<R>{P};
  }
}

// orders the wave's LDS accesses: lanes exchange particles through it
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// waves per SIMD that the registers leave room for: as many as the LDS does in
// the large ensembles (FP64 two-valley: 173 VGPRs allow two waves, 168 three,
// 0.68 -> 0.57 ms with the 16 VGPRs that it then spills, four per lane; 2 to 24
// in the other FP64 kernels)
template <typename R, int PPT, bool HOT, bool POS, int NV>
__global__ __launch_bounds__(kTile, PPT == 1 ? 1 : sizeof(R) == 8 ? 3 : 6) void k_bulk_fused(StepArgs<R> a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int TS = kTile * PPT, W = 64 * PPT;
  const int tile = blockIdx.x;
  const int inst = tile_instance(a.unit_inst, tile, TS);
  const InstDev<R> *P = stage_params(lds, a.inst + inst, a.lds_params);
  uint32_t *lds_tally = reinterpret_cast<uint32_t *>(lds + a.lds_params);
  if constexpr (HOT)
    tally_clear(P, lds_tally);
  const long long base = a.inst_start[inst];
  const long long count = a.inst_count[inst];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // local index of the wave's particle 0; particle i is (i / 64) * 256 + i % 64 further on
  const long long first = (long long)tile * TS - base + wave * 64;

  unsigned char *mem = lds + a.lds_params + a.lds_hot + (size_t)wave * a.lds_wave;
  R *const skx = reinterpret_cast<R *>(mem);
  R *const sky = skx + W, *const skz = sky + W, *const stau = skz + W;
  R *const spos = stau + W;  // [3][W], POS only
  uint32_t *const svs = reinterpret_cast<uint32_t *>(stau + (POS ? 4 : 1) * W);
  typedef typename QueueIndex<PPT>::type Index;
  Index *const list = reinterpret_cast<Index *>(svs + W);
  double *const ring = reinterpret_cast<double *>(list + W);

#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    const int i = j * 64 + lane;
    const long long local = first + (long long)j * kTile + lane;
    uint32_t vs = 0xFFFFFFFFu;  // no particle: away for good
    if (local < count) {
      const long long gi = base + local;
      skx[i] = a.kx[gi];
      sky[i] = a.ky[gi];
      skz[i] = a.kz[gi];
      stau[i] = a.tau[gi];
      vs = a.vs[gi];
      if constexpr (POS) {
        spos[i] = a.px[gi];
        spos[W + i] = a.py[gi];
        spos[2 * W + i] = a.pz[gi];
      }
    }
    svs[i] = vs;
  }
  for (int i = lane; i < kRing * a.n_obs; i += 64)
    ring[i] = 0.0;
  wave_lds_fence();
  // the particles per valley and (valley, subvalley): lane o holds count o of
  // the layout, the ring its change in each step
  const int sub0 = 2 + 3 * a.max_v;
  bool counts = lane >= sub0;
  double held = 0.0;
  for (int k = 0; k < a.max_v; ++k) {
    int n = 0;
    for (int d = 0; d < a.max_deg; ++d) {
      int c = 0;
#pragma unroll
      for (int j = 0; j < PPT; ++j)
        c += (int)__popcll(__ballot(svs[j * 64 + lane] == (((uint32_t)k << 16) | (uint32_t)d)));
      n += c;
      held = (lane == sub0 + k * a.max_deg + d) ? (double)c : held;
    }
    counts = counts || lane == 2 + 3 * k;
    held = (lane == 2 + 3 * k) ? (double)n : held;
  }

  StepRng<R, 0> rng;
  rng.inst = (uint32_t)inst;
  rng.k0 = a.key0;
  rng.k1 = a.key1;
  const R dt = P->dt;
  const auto kane = kane_source<R, NV>(P);
  double *const out = a.partial + (long long)tile * kSubs + wave;
  const long long out_stride = (long long)a.n_tiles * kSubs;
  // the sums of step r, complete, leave the ring
  auto retire = [&](int r) {
    if (lane < a.n_obs) {
      double *const q = ring + (r & (kRing - 1)) * a.n_obs + lane;
      held = *q + (counts ? held : 0.0);
      out[((long long)r * a.n_obs + lane) * out_stride] = held;
      *q = 0.0;
    }
  };

  // the worker lane's particle
  bool busy = false;
  R kx = 0, ky = 0, kz = 0, E = 0, tau = 0, rem = 0;
  R pos[3] = {0, 0, 0};
  int v = 0, sub = 0, idx = 0, at = 0;  // its index in the wave, its step
  uint32_t ev = 0;
  uint32_t head = 0, tail = 0;  // queue of particle indices (positions modulo W)
  int emptied = 0;         // last step whose passes emptied the queue
  StepSums<R, NV> sums;

  for (int s = 0; s < a.n_steps; ++s) {
    int nev = 0, nreal = 0;
    sums.clear();
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      const int i = j * 64 + lane;
      const uint32_t vs = svs[i];
      const bool here = !(vs & kAway);
      R x = skx[i], y = sky[i], z = skz[i], en = R(0), ta = stau[i];
      R wp[3] = {0, 0, 0};
      const int vv = (int)(vs >> 16), ss = (int)(vs & 0xffffu);
      bool pend = false;
      if (here) {
        if constexpr (POS) {
          wp[0] = spos[i];
          wp[1] = spos[W + i];
          wp[2] = spos[2 * W + i];
        }
        // std::min(tau, dt), then tRemaining
        drift<R, POS>(P, kane(vv), (dt < ta) ? dt : ta, x, y, z, en, NV == 1 ? 0 : vv, ss, wp);
        pend = dt - ta > R(0);
        skx[i] = x;
        sky[i] = y;
        skz[i] = z;
        stau[i] = pend ? ta : ta - dt;
        if constexpr (POS) {
          spos[i] = wp[0];
          spos[W + i] = wp[1];
          spos[2 * W + i] = wp[2];
        }
      }
      const unsigned long long m = __ballot(pend);
      if (pend) {
        svs[i] = vs | kAway | ((uint32_t)(s & (kRing - 1)) << kAtShift);
        list[(tail + lanes_below(m)) & (W - 1)] = (Index)i;
      }
      tail += (uint32_t)__popcll(m);
      if (here && !pend)
        sums.add(P, kane(vv), vv, ss, x, y, z, en);
    }
    wave_lds_fence();

    const bool last = s + 1 == a.n_steps;
    for (;;) {
      // enough pending events for a pass, or the last step of the launch,
      // which ends with every particle, or particles that must not lag
      // further (the queue holds none older than the step after `emptied`)
      const unsigned long long at_work = __ballot(busy);
      const int waiting = (int)(tail - head);
      if (!((int)__popcll(at_work) + waiting >= kPass || (last && (waiting > 0 || at_work)) ||
            (waiting > 0 && s - emptied >= kRing / 2) || __ballot(busy && at + (kRing - 1) <= s)))
        break;
      // idle lanes take the particles at the head of the queue
      const unsigned long long idle = __ballot(!busy);
      const int r = lanes_below(idle);
      if (!busy && r < waiting) {
        idx = list[(head + r) & (W - 1)];
        kx = skx[idx];
        ky = sky[idx];
        kz = skz[idx];
        tau = stau[idx];
        const uint32_t vs = svs[idx];
        at = s - ((s - (int)(vs >> kAtShift)) & (kRing - 1));
        v = (int)((vs & kVsMask) >> 16);
        sub = (int)(vs & 0xffffu);
        E = energy_of(kane(v), kx, ky, kz);
        if constexpr (POS) {
          pos[0] = spos[idx];
          pos[1] = spos[W + idx];
          pos[2] = spos[2 * W + idx];
        }
        rem = dt - tau;
        ev = 0;
        busy = true;
      }
      const int n_idle = (int)__popcll(idle);
      head += (uint32_t)(n_idle < waiting ? n_idle : waiting);
      if (tail == head)
        emptied = s;

      // one scatter event per particle
      int real = 0;
      const int v0 = v, sub00 = sub;
      if (busy) {
        rng.step = a.step0 + (uint32_t)at;
        rng.pid = (uint32_t)(first + (long long)(idx >> 6) * kTile + (idx & 63));
        event_once<R, 0, HOT, HOT, POS>(P, kane, a.cum, kx, ky, kz, E, tau, rem, v, sub, ev, rng, real,
                                        lds_tally, pos);
      }
      nev += (int)__popcll(__ballot(busy && at == s));
      nreal += (int)__popcll(__ballot(real && at == s));
      double *q = ring + (at & (kRing - 1)) * a.n_obs;
      if (busy && at < s) {
        atomicAdd(q, 1.0);
        if (real)
          atomicAdd(q + 1, 1.0);
      }
      if (v != v0 || sub != sub00) {
        atomicAdd(q + sub0 + v0 * a.max_deg + sub00, -1.0);
        atomicAdd(q + sub0 + v * a.max_deg + sub, 1.0);
        if (NV > 1 && v != v0) {
          atomicAdd(q + 2 + 3 * v0, -1.0);
          atomicAdd(q + 2 + 3 * v, 1.0);
        }
      }
      // particles at the end of their step: those of this step go home, those
      // behind enter their step's sums and start the next one
      for (;;) {
        const bool done = busy && (!(rem > R(0)) || ev >= kMaxEventsPerStep);
        const bool home = done && at == s, next = done && at < s;
        if (__ballot(home)) {
          if (home) {
            skx[idx] = kx;
            sky[idx] = ky;
            skz[idx] = kz;
            stau[idx] = tau - dt;
            svs[idx] = ((uint32_t)v << 16) | (uint32_t)sub;
            if constexpr (POS) {
              spos[idx] = pos[0];
              spos[W + idx] = pos[1];
              spos[2 * W + idx] = pos[2];
            }
            busy = false;
            sums.add(P, kane(v), v, sub, kx, ky, kz, E);
          }
        }
        if (!__ballot(next))
          break;
        if (next) {
          q = ring + (at & (kRing - 1)) * a.n_obs;
          atomicAdd(q + 3 + 3 * v, (double)E);
          atomicAdd(q + 4 + 3 * v,
                    (double)vdir_of(kane(v), P->valley[NV == 1 ? 0 : v].wdir[sub], kx, ky, kz, E));
          tau -= dt;
          ++at;
          ev = 0;
          drift<R, POS>(P, kane(v), (dt < tau) ? dt : tau, kx, ky, kz, E, NV == 1 ? 0 : v, sub, pos);
          rem = dt - tau;
        }
      }
    }
    if (tail == head)
      emptied = s;
    wave_lds_fence();
    const double mine = sums.total(a, nev, nreal);
    if (lane < a.n_obs)
      ring[(s & (kRing - 1)) * a.n_obs + lane] += mine;
    wave_lds_fence();
    if (s >= kRing - 1)
      retire(s - (kRing - 1));
  }
  for (int r = a.n_steps > kRing - 1 ? a.n_steps - (kRing - 1) : 0; r < a.n_steps; ++r)
    retire(r);
  if constexpr (HOT)
    tally_flush(P, lds_tally, a.tally, a.tally_bins);

#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    const int i = j * 64 + lane;
    const long long local = first + (long long)j * kTile + lane;
    if (local < count) {
      const long long gi = base + local;
      const R x = skx[i], y = sky[i], z = skz[i];
      const uint32_t vs = svs[i];
      a.kx[gi] = x;
      a.ky[gi] = y;
      a.kz[gi] = z;
      a.E[gi] = energy_of(kane((int)(vs >> 16)), x, y, z);
      a.tau[gi] = stau[i];
      a.vs[gi] = vs;
      if constexpr (POS) {
        a.px[gi] = spos[i];
        a.py[gi] = spos[W + i];
        a.pz[gi] = spos[2 * W + i];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// production step kernel of launches with one step (phonon baths and plasma
// screening, and callers that step one at a time): the particles stream
// through, 64 of the wave's 64 * PPT at a time with the next 64 on their way;
// those without an event are done after their flight, the others wait in LDS
// until a pass fills the wave's lanes.  Only a wave's last passes are partly
// filled, so more particles per lane mean fewer idle lanes, and the particles
// take no LDS.  Used in FP64, whose scatter body is long (screened cooling
// with 0.13 events per particle and step, 1M: 53.6 -> 41.8 us per step with
// 8 per lane, 4M: 134.7 -> 106.6), and in FP32 with two per lane.  With more
// the stores of single particles cost more than the passes they save (4M Si:
// 47.4 us with the particles in LDS, 55.5 streamed).  For models of one
// valley without positions: with more, the passes' and the stream's registers
// do not fit side by side (FP64, two valleys, 8M: 242 us in LDS with 4 per
// lane, 318 streamed with 8; positions: 48 spilled VGPRs, 8M Si 490 us against
// 377 in registers).
// ---------------------------------------------------------------------------
template <typename R>
constexpr bool streams_one_step(int ppt) {
  return sizeof(R) == 8 || ppt <= 2;
}
// queue entries of a wave: less than a pass's worth waits when 64 more arrive
constexpr int kOnceQueue = 128;
constexpr int kOncePass = 60;  // pending events that make a pass worth its while

template <typename R>
constexpr size_t once_wave_bytes() {
  return (size_t)kOnceQueue * (4 * sizeof(R) + sizeof(uint32_t) + sizeof(uint16_t));
}

template <typename R, int PPT, bool HOT>
__global__ __launch_bounds__(kTile, sizeof(R) == 8 ? 3 : 6) void k_bulk_once(StepArgs<R> a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int TS = kTile * PPT, Q = kOnceQueue, NV = 1;
  const int tile = blockIdx.x;
  const int inst = tile_instance(a.unit_inst, tile, TS);
  const InstDev<R> *P = stage_params(lds, a.inst + inst, a.lds_params);
  uint32_t *lds_tally = reinterpret_cast<uint32_t *>(lds + a.lds_params);
  if constexpr (HOT)
    tally_clear(P, lds_tally);
  const long long base = a.inst_start[inst];
  const long long count = a.inst_count[inst];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // local index of the wave's particle 0; particle i is (i / 64) * 256 + i % 64 further on
  const long long first = (long long)tile * TS - base + wave * 64;

  unsigned char *mem = lds + a.lds_params + a.lds_hot + (size_t)wave * a.lds_wave;
  R *const qx = reinterpret_cast<R *>(mem);
  R *const qy = qx + Q, *const qz = qy + Q, *const qtau = qz + Q;
  uint32_t *const qvs = reinterpret_cast<uint32_t *>(qtau + Q);
  uint16_t *const qidx = reinterpret_cast<uint16_t *>(qvs + Q);
  double *const delta = reinterpret_cast<double *>(qidx + Q);  // changes of the counts [n_obs]
  for (int i = lane; i < a.n_obs; i += 64)
    delta[i] = 0.0;

  StepRng<R, 0> rng;
  rng.inst = (uint32_t)inst;
  rng.step = a.step0;
  rng.k0 = a.key0;
  rng.k1 = a.key1;
  const R dt = P->dt;
  const auto kane = kane_source<R, NV>(P);
  const int sub0 = 2 + 3 * a.max_v;

  struct Part {
    R x, y, z, tau;
    uint32_t vs;
    bool valid;
  };
  auto load = [&](int j, Part &p) {
    const long long local = first + (long long)j * kTile + lane;
    p.valid = j < PPT && local < count;
    p.vs = 0xFFFFFFFFu;
    if (p.valid) {
      const long long gi = base + local;
      p.x = a.kx[gi];
      p.y = a.ky[gi];
      p.z = a.kz[gi];
      p.tau = a.tau[gi];
      p.vs = a.vs[gi];
    }
  };
  auto store = [&](int i, R x, R y, R z, R E, R tau) {
    const long long gi = base + first + (long long)(i >> 6) * kTile + (i & 63);
    a.kx[gi] = x;
    a.ky[gi] = y;
    a.kz[gi] = z;
    a.E[gi] = E;
    a.tau[gi] = tau;
    return gi;
  };

  // the worker lane's particle
  bool busy = false;
  R kx = 0, ky = 0, kz = 0, E = 0, tau = 0, rem = 0;
  int v = 0, sub = 0, idx = 0;
  uint32_t ev = 0, head = 0, tail = 0;
  int nev = 0, nreal = 0;
  double held = 0.0;  // lane o: count o of the layout before the step's events
  StepSums<R, NV> sums;
  sums.clear();

  // passes while `enough` events are pending
  auto passes = [&](int enough) {
    for (;;) {
      const int waiting = (int)(tail - head);
      if ((int)__popcll(__ballot(busy)) + waiting < enough)
        break;
      const unsigned long long idle = __ballot(!busy);
      const int r = lanes_below(idle);
      if (!busy && r < waiting) {
        const int q = (int)((head + (uint32_t)r) & (Q - 1));
        idx = qidx[q];
        kx = qx[q];
        ky = qy[q];
        kz = qz[q];
        tau = qtau[q];
        const uint32_t vs = qvs[q];
        v = (int)(vs >> 16);
        sub = (int)(vs & 0xffffu);
        E = energy_of(kane(v), kx, ky, kz);
        rem = dt - tau;
        ev = 0;
        busy = true;
      }
      const int n_idle = (int)__popcll(idle);
      head += (uint32_t)(n_idle < waiting ? n_idle : waiting);
      int real = 0;
      const int v0 = v, sub00 = sub;
      if (busy) {
        rng.pid = (uint32_t)(first + (long long)(idx >> 6) * kTile + (idx & 63));
        event_once<R, 0, HOT, HOT>(P, kane, a.cum, kx, ky, kz, E, tau, rem, v, sub, ev, rng, real,
                                   lds_tally);
      }
      nev += (int)__popcll(__ballot(busy));
      nreal += (int)__popcll(__ballot(real));
      if (v != v0 || sub != sub00) {
        atomicAdd(delta + sub0 + v0 * a.max_deg + sub00, -1.0);
        atomicAdd(delta + sub0 + v * a.max_deg + sub, 1.0);
      }
      if (busy && (!(rem > R(0)) || ev >= kMaxEventsPerStep)) {
        const long long gi = store(idx, kx, ky, kz, E, tau - dt);
        a.vs[gi] = ((uint32_t)v << 16) | (uint32_t)sub;
        sums.add(P, kane(v), v, sub, kx, ky, kz, E);
        busy = false;
      }
    }
  };

  Part next;
  load(0, next);
#pragma unroll 1
  for (int j = 0; j < PPT; ++j) {
    Part p = next;
    load(j + 1, next);
    const int vv = (int)(p.vs >> 16), ss = (int)(p.vs & 0xffffu);
    int n = 0;
    for (int d = 0; d < a.max_deg; ++d) {
      const int c = (int)__popcll(__ballot(p.valid && ss == d));
      n += c;
      held += (lane == sub0 + d) ? (double)c : 0.0;
    }
    held += (lane == 2) ? (double)n : 0.0;
    bool pend = false;
    R en = R(0);
    if (p.valid) {
      drift<R>(P, kane(vv), (dt < p.tau) ? dt : p.tau, p.x, p.y, p.z, en, 0, ss);
      pend = dt - p.tau > R(0);
      if (!pend) {
        store(j * 64 + lane, p.x, p.y, p.z, en, p.tau - dt);
        sums.add(P, kane(vv), vv, ss, p.x, p.y, p.z, en);
      }
    }
    const unsigned long long m = __ballot(pend);
    if (pend) {
      const int q = (int)((tail + (uint32_t)lanes_below(m)) & (Q - 1));
      qx[q] = p.x;
      qy[q] = p.y;
      qz[q] = p.z;
      qtau[q] = p.tau;
      qvs[q] = p.vs;
      qidx[q] = (uint16_t)(j * 64 + lane);
    }
    tail += (uint32_t)__popcll(m);
    wave_lds_fence();
    passes(kOncePass);
    wave_lds_fence();
  }
  passes(1);
  wave_lds_fence();
  const double mine = sums.total(a, nev, nreal);
  if (lane < a.n_obs) {
    a.partial[((long long)lane * a.n_tiles + tile) * kSubs + wave] = mine + held + delta[lane];
  }
  if constexpr (HOT)
    tally_flush(P, lds_tally, a.tally, a.tally_bins);
}

// ---------------------------------------------------------------------------
// production step kernel of short launches: a lane keeps its PPT particles in
// registers and works through their events itself, one at a time, pulling the
// state of its next particle that has time left.  No particle passes through
// LDS, so the first step costs no more than the others and more waves fit a
// SIMD, while the scatter body runs for as many passes as the wave's busiest
// lane has events.  Bound by HBM at few events, by vector-ALU issue at many.
// Which launches take it is keeps_lanes below.
// ---------------------------------------------------------------------------
template <typename R, int PPT, bool HOT, bool POS, int NV>
__global__ __launch_bounds__(kTile) void k_bulk_lanes(StepArgs<R> a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int TS = kTile * PPT;
  const int tile = blockIdx.x;
  const int inst = tile_instance(a.unit_inst, tile, TS);
  const InstDev<R> *P = stage_params(lds, a.inst + inst, a.lds_params);
  uint32_t *lds_tally = reinterpret_cast<uint32_t *>(lds + a.lds_params);
  if constexpr (HOT)
    tally_clear(P, lds_tally);
  const long long base = a.inst_start[inst];
  const long long count = a.inst_count[inst];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long first = (long long)tile * TS - base + threadIdx.x;  // local index, j = 0

  R kx[PPT], ky[PPT], kz[PPT], E[PPT], tau[PPT], rem[PPT];
  R pos[PPT][3];  // POS only
  int v[PPT], sub[PPT];
  uint32_t ev[PPT];
  bool valid[PPT];
#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    const long long local = first + (long long)j * kTile;
    valid[j] = local < count;
    kx[j] = ky[j] = kz[j] = E[j] = tau[j] = R(0);
    pos[j][0] = pos[j][1] = pos[j][2] = R(0);
    v[j] = sub[j] = 0;
    if (valid[j]) {
      const long long gi = base + local;
      kx[j] = a.kx[gi];
      ky[j] = a.ky[gi];
      kz[j] = a.kz[gi];
      tau[j] = a.tau[gi];
      const uint32_t vs = a.vs[gi];
      v[j] = (int)(vs >> 16);
      sub[j] = (int)(vs & 0xffffu);
      if constexpr (POS) {
        pos[j][0] = a.px[gi];
        pos[j][1] = a.py[gi];
        pos[j][2] = a.pz[gi];
      }
    }
  }
  StepRng<R, 0> rng;
  rng.inst = (uint32_t)inst;
  rng.k0 = a.key0;
  rng.k1 = a.key1;
  const R dt = P->dt;
  const auto kane = kane_source<R, NV>(P);

  for (int s = 0; s < a.n_steps; ++s) {
    rng.step = a.step0 + (uint32_t)s;
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      ev[j] = 0;
      rem[j] = R(0);
      if (valid[j]) {
        // std::min(tau, dt), then tRemaining
        drift<R, POS>(P, kane(v[j]), (dt < tau[j]) ? dt : tau[j], kx[j], ky[j], kz[j], E[j],
                      NV == 1 ? 0 : v[j], sub[j], pos[j]);
        rem[j] = dt - tau[j];
      }
    }
    int nreal = 0;
    for (;;) {
      int sel = -1;  // the lane's first particle with time left in the step
#pragma unroll
      for (int j = PPT - 1; j >= 0; --j)
        if (rem[j] > R(0) && ev[j] < kMaxEventsPerStep)
          sel = j;
      if (sel < 0)
        break;
      R x = kx[0], y = ky[0], z = kz[0], en = E[0], ta = tau[0], rm = rem[0];
      R wp[3] = {pos[0][0], pos[0][1], pos[0][2]};
      int vv = v[0], ss = sub[0];
      uint32_t ee = ev[0];
#pragma unroll
      for (int j = 1; j < PPT; ++j)
        if (sel == j) {
          x = kx[j];
          y = ky[j];
          z = kz[j];
          en = E[j];
          ta = tau[j];
          rm = rem[j];
          vv = v[j];
          ss = sub[j];
          ee = ev[j];
          if constexpr (POS) {
            wp[0] = pos[j][0];
            wp[1] = pos[j][1];
            wp[2] = pos[j][2];
          }
        }
      rng.pid = (uint32_t)(first + (long long)sel * kTile);
      event_once<R, 0, HOT, HOT, POS>(P, kane, a.cum, x, y, z, en, ta, rm, vv, ss, ee, rng, nreal,
                                      lds_tally, wp);
#pragma unroll
      for (int j = 0; j < PPT; ++j)
        if (sel == j) {
          kx[j] = x;
          ky[j] = y;
          kz[j] = z;
          E[j] = en;
          tau[j] = ta;
          rem[j] = rm;
          v[j] = vv;
          sub[j] = ss;
          ev[j] = ee;
          if constexpr (POS) {
            pos[j][0] = wp[0];
            pos[j][1] = wp[1];
            pos[j][2] = wp[2];
          }
        }
    }
    int nev = 0;
    StepSums<R, NV> sums;
    sums.clear();
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      nev += (int)ev[j];
      if (valid[j]) {
        tau[j] -= dt;
        sums.add(P, kane(v[j]), v[j], sub[j], kx[j], ky[j], kz[j], E[j]);
      }
    }
    double mine = sums.total(a, wave_sum_i(nev), wave_sum_i(nreal));
    for (int k = 0; k < a.max_v; ++k) {
      int n = 0;
      for (int d = 0; d < a.max_deg; ++d) {
        int c = 0;
#pragma unroll
        for (int j = 0; j < PPT; ++j)
          c += (int)__popcll(__ballot(valid[j] && v[j] == k && sub[j] == d));
        n += c;
        mine = (lane == 2 + 3 * a.max_v + k * a.max_deg + d) ? (double)c : mine;
      }
      mine = (lane == 2 + 3 * k) ? (double)n : mine;
    }
    if (lane < a.n_obs)
      a.partial[(((long long)s * a.n_obs + lane) * a.n_tiles + tile) * kSubs + wave] = mine;
  }
  if constexpr (HOT)
    tally_flush(P, lds_tally, a.tally, a.tally_bins);

#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    if (valid[j]) {
      const long long gi = base + first + (long long)j * kTile;
      a.kx[gi] = kx[j];
      a.ky[gi] = ky[j];
      a.kz[gi] = kz[j];
      a.E[gi] = E[j];
      a.tau[gi] = tau[j];
      a.vs[gi] = ((uint32_t)v[j] << 16) | (uint32_t)sub[j];
      if constexpr (POS) {
        a.px[gi] = pos[j][0];
        a.py[gi] = pos[j][1];
        a.pz[gi] = pos[j][2];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// replay step kernel (FP64): one particle per lane, the reference engine's
// recorded draws consumed in the reference's order, optional per-step trace
// ---------------------------------------------------------------------------
template <typename R, bool HOT, bool POS>
__global__ __launch_bounds__(kTile) void k_bulk_replay(StepArgs<R> a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds_tally[];
  const int tile = blockIdx.x;
  const int inst = tile_instance(a.unit_inst, tile, kTile);
  const InstDev<R> *P = a.inst + inst;
  if constexpr (HOT)
    tally_clear(P, lds_tally);
  const long long base = a.inst_start[inst];
  const long long local = (long long)tile * kTile + threadIdx.x - base;
  bool valid[1] = {local < a.inst_count[inst]};
  const long long gi = base + local;

  R kx[1] = {0}, ky[1] = {0}, kz[1] = {0}, E[1] = {0}, tau = 0;
  R pos[3] = {0, 0, 0};
  int v[1] = {0}, sub[1] = {0};
  if (valid[0]) {
    kx[0] = a.kx[gi];
    ky[0] = a.ky[gi];
    kz[0] = a.kz[gi];
    E[0] = a.E[gi];
    tau = a.tau[gi];
    const uint32_t vs = a.vs[gi];
    v[0] = (int)(vs >> 16);
    sub[0] = (int)(vs & 0xffffu);
    if constexpr (POS) {
      pos[0] = a.px[gi];
      pos[1] = a.py[gi];
      pos[2] = a.pz[gi];
    }
  }
  StepRng<R, 1> rng;
  rng.rs.p = a.draws + (valid[0] ? local : 0) * a.draw_stride;
  rng.rs.len = a.draw_stride;
  rng.rs.pos = valid[0] ? (long long)a.cursor[local] : 0;
  rng.rs.over = false;
  double grain = (valid[0] && a.grain_tau) ? a.grain_tau[local] : 1.0;

  for (int s = 0; s < a.n_steps; ++s) {
    int nev = 0, nreal = 0;
    if (valid[0]) {
      move_one<R, 1, HOT, HOT, POS>(P, a.cum, kx[0], ky[0], kz[0], E[0], tau, v[0], sub[0], rng,
                                    nev, nreal, lds_tally, pos);
      // grain bookkeeping (basicBulkParticleHandler.hpp:213-220), no grain
      // mechanism: a new grainTau of -ln U[1e-6,1) * 1 s
      grain -= a.dt_s;
      if (grain <= 0)
        grain = -::log(rng.rs.uniform(1e-6, 1.)) * 1.0;
      if (a.tr_valley && inst == 0) {
        const long long o = (long long)s * a.tr_n + local;
        a.tr_valley[o] = v[0];
        a.tr_sub[o] = sub[0];
        a.tr_events[o] = nev;
        a.tr_k[3 * o] = (double)kx[0];
        a.tr_k[3 * o + 1] = (double)ky[0];
        a.tr_k[3 * o + 2] = (double)kz[0];
        a.tr_E[o] = (double)E[0];
        if (a.tr_pos) {
          a.tr_pos[3 * o] = (double)pos[0];
          a.tr_pos[3 * o + 1] = (double)pos[1];
          a.tr_pos[3 * o + 2] = (double)pos[2];
        }
      }
    }
    tile_observables<R, 1>(a, P, tile, s, valid, v, sub, kx, ky, kz, E, nev, nreal);
  }
  if constexpr (HOT)
    tally_flush(P, lds_tally, a.tally, a.tally_bins);

  if (valid[0]) {
    a.kx[gi] = kx[0];
    a.ky[gi] = ky[0];
    a.kz[gi] = kz[0];
    a.E[gi] = E[0];
    a.tau[gi] = tau;
    a.vs[gi] = ((uint32_t)v[0] << 16) | (uint32_t)sub[0];
    if constexpr (POS) {
      a.px[gi] = pos[0];
      a.py[gi] = pos[1];
      a.pz[gi] = pos[2];
    }
    a.cursor[local] = (uint64_t)rng.rs.pos;
    if (a.grain_tau)
      a.grain_tau[local] = grain;
    if (rng.rs.over)
      atomicAdd(a.overflow, 1);
  }
}

// the ensemble sums of the current state, without a step: one particle per
// lane, the partials of "step 0" (the getAvg* calls right after
// generateInitialParticles, bulkSimulation.cpp:143-146)
template <typename R>
__global__ __launch_bounds__(kTile) void k_observe(StepArgs<R> a) {
  const int tile = blockIdx.x;
  const int inst = tile_instance(a.unit_inst, tile, kTile);
  const InstDev<R> *P = a.inst + inst;
  const long long base = a.inst_start[inst];
  const long long local = (long long)tile * kTile + threadIdx.x - base;
  bool valid[1] = {local < a.inst_count[inst]};
  const long long gi = base + local;
  R kx[1] = {0}, ky[1] = {0}, kz[1] = {0}, E[1] = {0};
  int v[1] = {0}, sub[1] = {0};
  if (valid[0]) {
    kx[0] = a.kx[gi];
    ky[0] = a.ky[gi];
    kz[0] = a.kz[gi];
    E[0] = a.E[gi];
    const uint32_t vs = a.vs[gi];
    v[0] = (int)(vs >> 16);
    sub[0] = (int)(vs & 0xffffu);
  }
  tile_observables<R, 1>(a, P, tile, 0, valid, v, sub, kx, ky, kz, E, 0, 0);
}

// ---------------------------------------------------------------------------
// per-(step, observable, instance) compensated reduction of the tile partials
// partial layout [step][obs][tile].  Two passes, both deterministic (fixed
// order for a given tile count): chunks of kChunk tiles per block with
// Neumaier summation per thread and a TwoSum tree across the block, then
// the chunk (sum, compensation) pairs of each output value.
// ---------------------------------------------------------------------------
constexpr int kChunk = 2048;

__device__ __forceinline__ void neumaier_add(double &sum, double &comp, double x) {
  const double y = sum + x;
  if (fabs(sum) >= fabs(x))
    comp += (sum - y) + x;
  else
    comp += (x - y) + sum;
  sum = y;
}

// TwoSum tree over 256 (sum, comp) pairs in LDS; result in ss[0] + sc[0]
__device__ __forceinline__ void block_twosum(double *ss, double *sc) {
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      const double x = ss[threadIdx.x], y0 = ss[threadIdx.x + w];
      const double y = x + y0;
      const double bb = y - x;
      const double err = (x - (y - bb)) + (y0 - bb);
      ss[threadIdx.x] = y;
      sc[threadIdx.x] += sc[threadIdx.x + w] + err;
    }
    __syncthreads();
  }
}

// With out (an output whose partials fit one chunk) the sum is finished here:
// the second pass would add one pair to zero.  A pass less is about 5 us of
// every call on an ensemble of up to 2048 waves.
__global__ __launch_bounds__(256) void k_reduce_chunks(const double *__restrict__ partial,
                                                       int n_tiles, int tile_size,
                                                       const long long *__restrict__ inst_start,
                                                       const long long *__restrict__ inst_count,
                                                       int n_chunks, double *__restrict__ chunk_out,
                                                       double *__restrict__ out, int n_obs,
                                                       int out_step0, int out_total) {
  __shared__ double ss[256], sc[256];
  const int chunk = blockIdx.x, so = blockIdx.y, inst = blockIdx.z;
  // the wave partials of the instance's tiles (tiles start on instance
  // boundaries; every wave of a tile with particles wrote one)
  const long long t0 = inst_start[inst] / tile_size * kSubs;
  const long long nt = (inst_count[inst] + tile_size - 1) / tile_size * kSubs;
  const long long lo = (long long)chunk * kChunk;
  const long long hi = (lo + kChunk < nt) ? lo + kChunk : nt;
  const double *src = partial + (long long)so * ((long long)n_tiles * kSubs) + t0;
  double sum = 0.0, comp = 0.0;
  for (long long t = lo + threadIdx.x; t < hi; t += 256)
    neumaier_add(sum, comp, src[t]);
  ss[threadIdx.x] = sum;
  sc[threadIdx.x] = comp;
  block_twosum(ss, sc);
  if (threadIdx.x == 0) {
    if (out) {
      out[((long long)inst * out_total + out_step0) * n_obs + so] = ss[0] + sc[0];
    } else {
      double *o = chunk_out + (((long long)inst * gridDim.y + so) * n_chunks + chunk) * 2;
      o[0] = ss[0];
      o[1] = sc[0];
    }
  }
}

__global__ __launch_bounds__(256) void k_reduce_final(const double *__restrict__ chunk_out,
                                                      int n_chunks, int n_obs,
                                                      double *__restrict__ out, int out_step0,
                                                      int out_total) {
  __shared__ double ss[256], sc[256];
  const int so = blockIdx.x, inst = blockIdx.y;
  const int s = so / n_obs, o = so % n_obs;
  const double *src = chunk_out + ((long long)inst * gridDim.x + so) * n_chunks * 2;
  double sum = 0.0, comp = 0.0;
  for (int c = threadIdx.x; c < n_chunks; c += 256) {
    neumaier_add(sum, comp, src[2 * c]);
    comp += src[2 * c + 1];
  }
  ss[threadIdx.x] = sum;
  sc[threadIdx.x] = comp;
  block_twosum(ss, sc);
  if (threadIdx.x == 0)
    out[((long long)inst * out_total + out_step0 + s) * n_obs + o] = ss[0] + sc[0];
}

// ---------------------------------------------------------------------------
// End of a hot-phonon step, one block per instance with baths:
//   every bath of the instance is updated (emcPhononBath::update,
//   emcPhononBath.hpp:264-358) and its mean occupation taken (getMeanNq,
//   :461-470); then, on rebuild steps, the instance's scatter tables are
//   rebuilt from the baths (reinitScatterTables: fillScatterTables +
//   renormalizeTables, emcScatterHandler.hpp:100-108, 220-272).
// The per-bin update runs on all lanes; the DOS-weighted sums that the
// reference takes sequentially over the bins are taken in that order by
// lane 0 from LDS, so the FP64 results match the reference operation for
// operation.  Hot-phonon rates are scatterConst * N / kI * ln (absorption)
// and scatterConst * (N + 1) / kI * ln (emission) with the per-level kI and
// ln of emcHotPhononFroehlichMechanism.hpp:79-91 / :159-173 precomputed in
// FP64 on the host (kI = 0 marks a zero rate); other mechanisms keep their
// FP64 rates.  Cumulative sums run over the tables in registration order and
// are normalised by the largest total rate; the FP64 result is stored in the
// precision of the kinematics and in an FP64 copy.
// ---------------------------------------------------------------------------
constexpr double kPi = 3.14159265358979323846;
constexpr double kQ = 1.60219e-19, kKB = 1.38066e-23;  // include/emcConstants.hpp
constexpr double kEps0 = 8.85419e-12;
constexpr int kBathThreads = 1024;

__device__ double bath_planck(double energy_ev, double temp_k) {
#pragma clang fp contract(off)
  const double x = kQ * energy_ev / (kKB * temp_k);
  return 1.0 / (::exp(x) - 1.0);
}
__device__ double bath_planck_temp(double energy_ev, double n) {
#pragma clang fp contract(off)
  if (n <= 0.0)
    return 0.0;
  return kQ * energy_ev / (kKB * ::log(1.0 + 1.0 / n));
}

// one lane per bin in the bath update; the per-bin LDS arrays double as
// per-lane reduction buffers
static_assert(kMaxBins == kBathThreads, "bath block: one lane per bin");

struct BathShared {
  double old_n[kMaxBins];
  double new_n[kMaxBins];
  double w[kMaxBins];
  double vmax[kBathThreads];
  // terms of the energy record: net emissions, LO population change, decay
  double e_em[kMaxBins], e_lo[kMaxBins], e_dec[kMaxBins];
  double target;
  double qs2;  // the instance's q_s^2, broadcast to the block
};

template <typename R>
__device__ void bath_update_one(const BathDev &B, BathVar &V, double *__restrict__ nq,
                                const double *__restrict__ tau_prof,
                                unsigned long long *__restrict__ tally, long long tally_bins,
                                double dt, double *__restrict__ hist,
                                double *__restrict__ energy, BathShared &sh,
                                double qs2, double *__restrict__ win64, R *__restrict__ win) {
#pragma clang fp contract(off)
  const int nb = B.n_bins;
  if (threadIdx.x == 0) {
    // decay target: N0 unless a daughter reservoir is hot (:269-286)
    double target = B.n0;
    if (B.has_ac) {
      double n_klemens = B.n0;
      if (V.n_ac > B.n_ac_eq)
        n_klemens = bath_planck(B.lo_e, bath_planck_temp(B.ac_e, V.n_ac));
      if (B.has_ridley) {
        double n_ridley = B.n0;
        if (V.n_to > B.n_to_eq)
          n_ridley = bath_planck(B.lo_e, bath_planck_temp(B.to_e, V.n_to));
        target = (1.0 - B.w_r) * n_klemens + B.w_r * n_ridley;
      } else {
        target = n_klemens;
      }
    }
    sh.target = target;
  }
  // the event counts of this step: the sum of the tally copies, which are
  // cleared.  G = blockDim / nb lane groups share the copies of a bin
  // (copies g, g + G, ...), their integer partial sums meet in LDS (exact as
  // doubles: far below 2^53)
  const int G = (nb > 0 && (int)blockDim.x >= nb) ? (int)blockDim.x / nb : 1;
  if ((int)threadIdx.x < G * nb) {
    const int i = (int)threadIdx.x % nb, g = (int)threadIdx.x / nb;
    const long long gi = B.off + i;
    unsigned long long c_em = 0ull, c_abs = 0ull;
#pragma unroll 16
    for (int r = g; r < kTallyCopies; r += G) {
      unsigned long long *t = tally + 2 * ((long long)r * tally_bins + gi);
      c_em += t[0];
      c_abs += t[1];
      t[0] = 0ull;
      t[1] = 0ull;
    }
    sh.vmax[threadIdx.x] = (double)c_em;
    sh.old_n[threadIdx.x] = (double)c_abs;
  }
  __syncthreads();
  double cnt_em[kMaxBins / kBathThreads + 1], cnt_abs[kMaxBins / kBathThreads + 1];
  {
    int u = 0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x, ++u) {
      double e = 0.0, b = 0.0;
      for (int g = 0; g < G; ++g) {
        e = e + sh.vmax[g * nb + i];
        b = b + sh.old_n[g * nb + i];
      }
      cnt_em[u] = e;
      cnt_abs[u] = b;
    }
  }
  __syncthreads();
  const double target = sh.target;
  int u = 0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x, ++u) {
    const long long gi = B.off + i;
    const double q = ((double)i + 0.5) * B.dq;
    const double dph = q * q * B.dq * B.vsim / (2.0 * kPi * kPi);
    const double n_em = cnt_em[u], n_abs = cnt_abs[u];
    const double g = (dph > 0.0) ? (n_em - n_abs) / (dph * dt) : 0.0;
    const double tau_i = B.has_profile ? tau_prof[gi] : B.tau_lo;
    const double n_old = nq[gi];
    const double w = q * q;
    double n = n_old;
    n += g * dt - (dt / tau_i) * (n - target);
    if (n < 0.0)
      n = 0.0;
    nq[gi] = n;
    if (energy) {
      sh.e_em[i] = n_em - n_abs;
      sh.e_lo[i] = dph * (n - n_old);
      sh.e_dec[i] = dph * (dt / tau_i) * (n_old - target);
    }
    // the terms of the bin-order sums, formed on all lanes: the reservoir
    // source from the start-of-step occupations (:291-355), getMeanNq
    // (:461-470) and, when read, the window sums (:109-124)
    sh.old_n[i] = B.has_profile ? w * (n_old - target) / tau_i : w * (n_old - target);
    sh.new_n[i] = w * n;
    if (win64) {
      const double denom = q * q + qs2;
      const double ww = (denom > 0.0) ? q / denom : 0.0;
      sh.w[i] = ww;
      sh.vmax[i] = ww * n;
    }
  }
  __syncthreads();
  // the sums themselves in bin order (the reference's), one lane each of
  // four waves side by side
  const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  if (lane == 0 && wave == 0 && B.has_ac) {
    {
      // sum of the weights q^2: a constant of the bath, summed on the host
      // in the same order
      const double sum_w = B.sum_w;
      double sum_t = 0.0;
#pragma unroll 16
      for (int i = 0; i < nb; ++i)
        sum_t += sh.old_n[i];
      const double f_klemens = B.has_ridley ? (1.0 - B.w_r) : 1.0;
      const double src = (sum_w > 0.0) ? sum_t / sum_w : 0.0;
      double n_ac = V.n_ac, n_to = V.n_to;
      if (!B.has_profile) {
        n_ac += dt * f_klemens * src / B.tau_lo - dt * (n_ac - B.n_ac_eq) / B.tau_ac;
        if (n_ac < B.n_ac_eq)
          n_ac = B.n_ac_eq;
        if (B.has_ridley) {
          n_to += dt * B.w_r * src / B.tau_lo - dt * (n_to - B.n_to_eq) / B.tau_to;
          if (n_to < B.n_to_eq)
            n_to = B.n_to_eq;
        }
      } else {
        n_ac += dt * f_klemens * src - dt * (n_ac - B.n_ac_eq) / B.tau_ac;
        if (n_ac < B.n_ac_eq)
          n_ac = B.n_ac_eq;
        if (B.has_ridley) {
          n_to += dt * B.w_r * src - dt * (n_to - B.n_to_eq) / B.tau_to;
          if (n_to < B.n_to_eq)
            n_to = B.n_to_eq;
        }
      }
      V.n_ac = n_ac;
      V.n_to = n_to;
    }
  } else if (lane == 0 && wave == 1) {
    // getMeanNq over the updated occupations
    double sum_wn = 0.0;
#pragma unroll 16
    for (int i = 0; i < nb; ++i)
      sum_wn += sh.new_n[i];
    const double mean = (B.sum_w > 0.0) ? sum_wn / B.sum_w : B.n0;
    V.mean = mean;
    if (hist)
      *hist = mean;
  } else if (lane == 0 && (wave == 2 || wave == 3) && win64) {
    double *t = (wave == 2) ? sh.w : sh.vmax;
    double acc = 0.0;
#pragma unroll 16
    for (int i = 0; i < nb; ++i) {
      acc = acc + t[i];
      t[i] = acc;
    }
  } else if (lane == 0 && wave >= 4 && wave <= 6 && energy) {
    // the energy record in bin order, x hbar w_LO [eV]
    const double *t = (wave == 4) ? sh.e_em : (wave == 5) ? sh.e_lo : sh.e_dec;
    double acc = 0.0;
#pragma unroll 16
    for (int i = 0; i < nb; ++i)
      acc += t[i];
    energy[wave - 4] = B.lo_e * acc;
  }
  __syncthreads();
  if (win64) {
    // the window sums leave from all lanes: one lane's serial
    // stores took as long as its adds
    double *cw = win64 + B.woff, *cwn = cw + nb + 1;
    R *rw = win + B.woff, *rwn = rw + nb + 1;
    for (int i = threadIdx.x; i <= nb; i += blockDim.x) {
      const double sw = i ? sh.w[i - 1] : 0.0, sn = i ? sh.vmax[i - 1] : 0.0;
      cw[i] = sw;
      cwn[i] = sn;
      rw[i] = (R)sw;
      rwn[i] = (R)sn;
    }
    __syncthreads();
  }
}

// getNqInWindow (emcPhononBath.hpp:378-394) over the FP64 window sums
__device__ __forceinline__ double window_nq(const BathDev &B, const double *__restrict__ win64,
                                           double mean, double qmin, double qmax) {
#pragma clang fp contract(off)
  if (B.n_bins < 2 || qmax <= qmin)
    return mean;
  long lo = (long)::floor(qmin / B.dq);
  long hi = (long)::ceil(qmax / B.dq);
  if (lo < 0)
    lo = 0;
  if (hi > (long)B.n_bins)
    hi = (long)B.n_bins;
  if (hi - lo < 1)
    return mean;
  const double *cw = win64 + B.woff, *cwn = cw + B.n_bins + 1;
  const double wsum = cw[hi] - cw[lo];
  if (wsum <= 0.0)
    return mean;
  return (cwn[hi] - cwn[lo]) / wsum;
}

// screenedFroehlichLogFactor (emcScreenedFroehlichInteraction.hpp:52-62)
__device__ __forceinline__ double screened_log(double ki, double kf, double qs2) {
#pragma clang fp contract(off)
  const double p2 = (ki + kf) * (ki + kf), m2 = (ki - kf) * (ki - kf);
  if (qs2 <= 0.0)
    return (m2 <= 0.0) ? 0.0 : 0.5 * ::log(p2 / m2);
  return 0.5 * ::log((p2 + qs2) / (m2 + qs2));
}

__device__ __forceinline__ double rebuild_rate(const RebuildJob &J, int j, int l,
                                               const double *__restrict__ arena,
                                               const BathVar *__restrict__ var,
                                               const BathDev *__restrict__ baths,
                                               const double *__restrict__ win64, double qs2) {
#pragma clang fp contract(off)
  const long long o = J.rate_off[j];
  if (J.kind[j] == kRateConst)
    return arena[o + l];
  const double ki = arena[o + l];
  if (!(ki > 0.0))
    return 0.0;
  if (J.kind[j] == kRateScrAb || J.kind[j] == kRateScrEm) {
    // emcScreenedFroehlichInteraction.hpp:128-138 / :184-196 (constant N)
    // and :257-269 / :333-348 (bath mean or window mean)
    const double kf = arena[o + J.n_levels + l];
    double n = J.nconst[j];
    if (J.nsrc[j] == kNMean) {
      n = var[J.bath[j]].mean;
    } else if (J.nsrc[j] == kNWindow) {
      const double d = ki - kf;
      n = window_nq(baths[J.bath[j]], win64, var[J.bath[j]].mean, (d < 0.0) ? -d : d, ki + kf);
    }
    const double lf = screened_log(ki, kf, qs2);
    return (J.kind[j] == kRateScrAb) ? J.C[j] * n / ki * lf : J.C[j] * (n + 1.0) / ki * lf;
  }
  const double ln = arena[o + J.n_levels + l];
  const double n = var[J.bath[j]].mean;
  return (J.kind[j] == kRateHotAb) ? J.C[j] * n / ki * ln : J.C[j] * (n + 1.0) / ki * ln;
}

template <typename R>
__device__ void rebuild_one(const RebuildJob &J, const BathStepArgs<R> &a, double qs2,
                            BathShared &sh) {
#pragma clang fp contract(off)
  const double *__restrict__ arena = a.arena;
  const BathVar *__restrict__ var = a.var;
  const BathDev *__restrict__ baths = a.baths;
  const double *__restrict__ win64 = a.win64;
  R *__restrict__ cum = a.cum;
  double *__restrict__ cum64 = a.cum64;
  const int nt = J.n_tables, nl = J.n_levels;
  // pass 1: the cumulative rates of each level, kept unnormalised in the
  // FP64 copy by the lane that normalises them in pass 2
  double mx = -1.0;
  for (int l = threadIdx.x; l < nl; l += blockDim.x) {
    double c = 0.0;
    for (int j = 0; j < nt; ++j) {
      const double r = rebuild_rate(J, j, l, arena, var, baths, win64, qs2);
      c = (j == 0) ? r : r + c;
      cum64[J.cum_off + (long long)l * nt + j] = c;
    }
    mx = (mx < c) ? c : mx;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double x = __shfl_xor(mx, o, 64);
    mx = (mx < x) ? x : mx;
  }
  if ((threadIdx.x & 63) == 0)
    sh.vmax[threadIdx.x >> 6] = mx;
  __syncthreads();
  for (int w = 0; w < (int)blockDim.x / 64; ++w)
    mx = (mx < sh.vmax[w]) ? sh.vmax[w] : mx;
  __syncthreads();
  if (!(mx > 0.0))
    return;  // no rate at any level: the kinematics keep the previous tables
  for (int l = threadIdx.x; l < nl; l += blockDim.x) {
    for (int j = 0; j < nt; ++j) {
      const long long e = J.cum_off + (long long)l * nt + j;
      const double x = cum64[e] / mx;
      put_row_entry(cum + J.tab_off + (long long)l * row_stride(nt), nt, j, (R)x);
      cum64[e] = x;
    }
  }
  if (threadIdx.x == 0) {
    const double tau = 1. / mx;
    a.inst[J.inst].tau0[J.valley] = (R)(tau * 1e15);
    a.tau0_64[J.inst * kMaxV + J.valley] = tau;
  }
}

// updateScreening (examples/hotCarrierMHP/hotCarrierMHP.cpp:563-581) of one
// instance from the partials of the step just taken: N over all valleys,
// the valley-0 energy sum and count, the Debye q_s^2 at the temperature of
// the valley-0 mean energy (getMBTemp, emcHotCarrierOutput.hpp:89-92)
template <typename R>
__device__ void screening_update(const BathInstDev &I, const BathStepArgs<R> &a, BathShared &sh) {
#pragma clang fp contract(off)
  double vals[3] = {0.0, 0.0, 0.0};  // N, sum E valley 0, count valley 0
  // the instance's tiles: it starts on a tile boundary, tiles past its
  // count hold zeros
  const long long ts = a.tile_size, nsub = (long long)a.n_tiles * kSubs;
  const long long tile0 = a.inst_start[I.inst] / ts * kSubs;
  const long long tile1 = (a.inst_start[I.inst] + a.inst_count[I.inst] + ts - 1) / ts * kSubs;
  const long long tend = (tile1 < nsub) ? tile1 : nsub;
#pragma unroll 4
  for (long long t = tile0 + threadIdx.x; t < tend; t += blockDim.x) {
    for (int v = 0; v < I.n_valleys; ++v)
      vals[0] += a.partial[(long long)(2 + 3 * v) * nsub + t];
    vals[1] += a.partial[3LL * nsub + t];
    vals[2] += a.partial[2LL * nsub + t];
  }
  // the three sums, a wave each, as trees over the lanes that halve the
  // distance from 512 to 1 (fixed order, deterministic); one barrier instead
  // of eleven.  With the window sums' stores (bath_update_one) the screened
  // FP64 bath step went from 16.8 to 13.7 us (1 M carriers, 256 bins)
  static_assert(kBathThreads == 1024, "sixteen terms per lane below");
  sh.vmax[threadIdx.x] = vals[0];
  sh.old_n[threadIdx.x] = vals[1];
  sh.new_n[threadIdx.x] = vals[2];
  __syncthreads();
  const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  if (wave < 3) {
    const double *r = wave == 0 ? sh.vmax : wave == 1 ? sh.old_n : sh.new_n;
    double x[16];
#pragma unroll
    for (int m = 0; m < 16; ++m)
      x[m] = r[lane + 64 * m];
#pragma unroll
    for (int w = 8; w > 0; w >>= 1)
#pragma unroll
      for (int m = 0; m < w; ++m)
        x[m] = x[m] + x[m + w];
#pragma unroll
    for (int w = 32; w > 0; w >>= 1)
      x[0] = x[0] + __shfl_down(x[0], w, 64);
    if (lane == 0)
      sh.w[wave] = x[0];
  }
  __syncthreads();
  const double tot[3] = {sh.w[0], sh.w[1], sh.w[2]};
  if (threadIdx.x == 0) {
    double qs2 = 0.0;
    if (tot[0] != 0.0) {
      const double ns = tot[0] / I.scr_vol;
      const double avg = (tot[2] != 0.0) ? tot[1] / tot[2] : 0.0;
      const double ts = 2.0 * avg * kQ / (3.0 * kKB);
      if (ts > 0.0)
        qs2 += ns * kQ * kQ / (I.scr_eps * kEps0 * kKB * ts);
    }
    a.scr[I.inst] = qs2;
    a.inst[I.inst].qs2 = (R)(qs2 * 1e-18);
    sh.qs2 = qs2;
  }
  __syncthreads();
}

// rebuildWindowSums (emcPhononBath.hpp:109-124) of one bath with the
// instance's q_s^2: weights on all lanes, the prefix sums by lane 0 in bin
// order (FP64, as the reference adds them) and a copy in the precision of
// the kinematics
template <typename R>
__device__ void window_sums_one(const BathDev &B, double qs2, const BathStepArgs<R> &a,
                                BathShared &sh) {
#pragma clang fp contract(off)
  const int nb = B.n_bins;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) {
    const double q = ((double)i + 0.5) * B.dq;
    const double denom = q * q + qs2;
    const double w = (denom > 0.0) ? q / denom : 0.0;
    sh.old_n[i] = w;
    sh.new_n[i] = w * a.nq[B.off + i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double *cw = a.win64 + B.woff, *cwn = cw + nb + 1;
    R *rw = a.win + B.woff, *rwn = rw + nb + 1;
    double s = 0.0, sn = 0.0;
    cw[0] = 0.0;
    cwn[0] = 0.0;
    rw[0] = R(0);
    rwn[0] = R(0);
#pragma unroll 16
    for (int i = 0; i < nb; ++i) {
      s = s + sh.old_n[i];
      sn = sn + sh.new_n[i];
      cw[i + 1] = s;
      cwn[i + 1] = sn;
      rw[i + 1] = (R)s;
      rwn[i + 1] = (R)sn;
    }
  }
  __syncthreads();
}

// the instance's q_s^2 into LDS: from the step's partials (plasma
// screening) or as held
template <typename R>
__device__ void group_screening(const BathInstDev &I, const BathStepArgs<R> &a, bool plasma,
                                BathShared &sh) {
  if (plasma && I.plasma) {
    screening_update(I, a, sh);
    return;
  }
  if (threadIdx.x == 0)
    sh.qs2 = a.scr ? a.scr[I.inst] : 0.0;
  __syncthreads();
}

template <typename R>
__device__ void rebuild_group(const BathInstDev &I, const BathStepArgs<R> &a, BathShared &sh) {
  const double qs2 = sh.qs2;
  for (int j = I.job0; j < I.job0 + I.n_jobs; ++j)
    rebuild_one<R>(a.jobs[j], a, qs2, sh);
}

// One block per instance with baths or plasma screening: the baths' update,
// the screening from the step's partials, the window sums, the tables (the
// order of hotCarrierMHP.cpp:693-703).  Window sums and screening follow
// the values the reference's setScreeningQ2 / update leave behind.
// The screening depends on the carriers only, so it is taken first; the
// window sums then see the updated occupations and the new q_s^2, as after
// the reference's update + setScreeningQ2.
template <typename R>
__global__ __launch_bounds__(kBathThreads) void k_bath_step(BathStepArgs<R> a) {
  __shared__ BathShared sh;
  const BathInstDev &I = a.groups[blockIdx.x];
  group_screening<R>(I, a, a.partial != nullptr, sh);
  const double qs2 = sh.qs2;
  double *win64 = (a.win64 && I.need_win) ? a.win64 : nullptr;
  for (int b = I.bath0; b < I.bath0 + I.n_baths; ++b)
    bath_update_one<R>(a.baths[b], a.var[b], a.nq, a.tau_prof, a.tally, a.tally_bins, a.dt,
                       a.hist ? a.hist + (long long)b * a.hist_steps + a.hist_step : nullptr,
                       a.energy ? a.energy + 3 * ((long long)b * a.hist_steps + a.hist_step)
                                : nullptr,
                       sh, qs2, win64, a.win);
  // the tables follow in k_rebuild_rates / k_rebuild_norm
}

// The per-step table rebuild over (level chunk, job) blocks, one level per
// lane: the cumulative FP64 rates of the level (kept unnormalised in the
// FP64 copy) and the block's maximum ...
template <typename R>
__global__ __launch_bounds__(kRebuildChunk) void k_rebuild_rates(BathStepArgs<R> a) {
#pragma clang fp contract(off)
  __shared__ double red[kRebuildChunk];
  const RebuildJob &J = a.jobs[blockIdx.y];
  if (!(a.rebuild || J.every_step))
    return;
  const int nl = J.n_levels, nt = J.n_tables;
  const int l0 = (int)blockIdx.x * kRebuildChunk;
  if (l0 >= nl)
    return;  // the whole block leaves: no barrier below is reached
  const double qs2 = a.scr ? a.scr[J.inst] : 0.0;
  const int l = l0 + (int)threadIdx.x;
  double c = -1.0;
  if (l < nl) {
    for (int j = 0; j < nt; ++j) {
      const double r = rebuild_rate(J, j, l, a.arena, a.var, a.baths, a.win64, qs2);
      c = (j == 0) ? r : r + c;
      a.cum64[J.cum_off + (long long)l * nt + j] = c;
    }
  }
  red[threadIdx.x] = c;
  __syncthreads();
  for (int w = kRebuildChunk / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w && red[threadIdx.x] < red[threadIdx.x + w])
      red[threadIdx.x] = red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    a.rb_max[(long long)blockIdx.y * kRebuildChunks + blockIdx.x] = red[0];
}

// ... then the largest total rate of the job over its chunks, the
// normalised tables and tau0 (renormalizeTables, emcScatterHandler.hpp:
// 248-272); with no rate at any level the kinematics keep the previous tables
template <typename R>
__global__ __launch_bounds__(kRebuildChunk) void k_rebuild_norm(BathStepArgs<R> a) {
#pragma clang fp contract(off)
  const RebuildJob &J = a.jobs[blockIdx.y];
  if (!(a.rebuild || J.every_step))
    return;
  const int nl = J.n_levels, nt = J.n_tables;
  const int l0 = (int)blockIdx.x * kRebuildChunk;
  if (l0 >= nl)
    return;
  const int nc = (nl + kRebuildChunk - 1) / kRebuildChunk;
  double mx = -1.0;
  for (int k = 0; k < nc; ++k) {
    const double m = a.rb_max[(long long)blockIdx.y * kRebuildChunks + k];
    mx = (mx < m) ? m : mx;
  }
  if (!(mx > 0.0))
    return;
  const int l = l0 + (int)threadIdx.x;
  if (l < nl) {
    for (int j = 0; j < nt; ++j) {
      const long long e = J.cum_off + (long long)l * nt + j;
      const double x = a.cum64[e] / mx;
      put_row_entry(a.cum + J.tab_off + (long long)l * row_stride(nt), nt, j, (R)x);
      a.cum64[e] = x;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const double tau = 1. / mx;
    a.inst[J.inst].tau0[J.valley] = (R)(tau * 1e15);
    a.tau0_64[J.inst * kMaxV + J.valley] = tau;
  }
}

// window sums and tables alone (after the model, the field, a bath state or
// the screening changed)
template <typename R>
__global__ __launch_bounds__(kBathThreads) void k_bath_refresh(BathStepArgs<R> a) {
  __shared__ BathShared sh;
  const BathInstDev &I = a.groups[blockIdx.x];
  group_screening<R>(I, a, false, sh);
  if (a.win64 && I.need_win)
    for (int b = I.bath0; b < I.bath0 + I.n_baths; ++b)
      window_sums_one(a.baths[b], sh.qs2, a, sh);
  rebuild_group<R>(I, a, sh);
}

// ---------------------------------------------------------------------------
// scatter rates from descriptors: one lane per (level, mechanism), the
// FP64 formulas of emcgpuPhysics.hpp (the reference's operation order; the
// device's pow / sqrt / log are within an ulp of the host's)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_rates_desc(const RateDescJob *__restrict__ jobs,
                                                    int n_levels, double dE,
                                                    double *__restrict__ out) {
#pragma clang fp contract(off)
  const RateDescJob &J = jobs[blockIdx.y];
  const int l = (int)blockIdx.x * 256 + (int)threadIdx.x;
  if (l >= n_levels)
    return;
  const double E = (double)(unsigned long long)(l + 1) * dE;
  const bool ab = J.absorption != 0;
  double r = 0.0;
  switch (J.kind) {
  case EMCGPU_MECH_ACOUSTIC:
    r = phys::acousticRate(J.C, J.iv, E);
    break;
  case EMCGPU_MECH_ZERO_IV_AB:
  case EMCGPU_MECH_ZERO_IV_EM:
    r = phys::zeroOrderRate(J.C, J.fv, E, J.hw, J.delta, ab);
    break;
  case EMCGPU_MECH_FIRST_IV_AB:
  case EMCGPU_MECH_FIRST_IV_EM:
    r = phys::firstOrderRate(J.C, J.iv, J.fv, E, J.hw, J.delta, ab);
    break;
  case EMCGPU_MECH_SCREENED_FROEHLICH_AB:
  case EMCGPU_MECH_SCREENED_FROEHLICH_EM:
    r = phys::screenedFroehlichRate(J.C, J.nq, J.meff, J.iv, E, J.hw, J.qs2, ab);
    break;
  default:
    r = phys::froehlichRate(J.C, J.nq, J.meff, J.iv, E, J.hw, ab);
    break;
  }
  out[J.out_off + l] = r;
}

hipError_t launch_rates_desc(const RateDescJob *jobs, int n_jobs, int n_levels, double dE,
                             double *out, hipStream_t st) {
  if (n_jobs <= 0 || n_levels <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_rates_desc, dim3((n_levels + 255) / 256, n_jobs), dim3(256), 0, st, jobs,
                     n_levels, dE, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// thermal initialisation (emcElectron.hpp:75-90, emcParticleInitialization.hpp:36-51)
// ---------------------------------------------------------------------------
// init_mean > 0 selects the prescribed-energy initialiser: E = mean +
// sigma * sqrt(-2 ln u2) cos(2 pi u6) (u2 in [1e-6, 1)), |E| if negative,
// the mean if zero; sigma = 0 is the fixed-energy photoexcitation
// (emcParticleInitialization.hpp:57-71)
template <typename R>
__global__ __launch_bounds__(kTile) void k_init_thermal(StepArgs<R> a, double init_mean,
                                                        double init_sigma) {
  const long long tile = (long long)a.tile_base + blockIdx.x;
  const int inst = tile_instance(a.unit_inst, tile, kTile);
  const InstDev<R> *P = a.inst + inst;
  const long long base = a.inst_start[inst];
  const long long local = tile * kTile + threadIdx.x - base;
  if (local >= a.inst_count[inst])
    return;
  const long long gi = base + local;
  const uint32_t st = 0xFFFFFFFFu, pid = (uint32_t)local, in = (uint32_t)inst;
  const R lo = R(1e-6), sc = R(1 - 1e-6);
  const R uv = stream_uniform<R>(0, st, pid, in, a.key0, a.key1) * sc + lo;
  const R us = stream_uniform<R>(1, st, pid, in, a.key0, a.key1) * sc + lo;
  const R ue = stream_uniform<R>(2, st, pid, in, a.key0, a.key1) * sc + lo;
  const R uphi = stream_uniform<R>(3, st, pid, in, a.key0, a.key1);
  const R ucos = stream_uniform<R>(4, st, pid, in, a.key0, a.key1);
  const R ut = stream_uniform<R>(5, st, pid, in, a.key0, a.key1) * sc + lo;
  int v = (int)Math<R>::floor((R)P->n_valleys * uv);
  v = v < P->n_valleys ? v : P->n_valleys - 1;
  const ValleyDev<R> &V = P->valley[v];
  int sub = (int)Math<R>::floor((R)V.deg * us);
  sub = sub < V.deg ? sub : V.deg - 1;
  R E;
  if (init_mean > 0.0) {
    E = (R)init_mean;
    if (init_sigma > 0.0) {
      const R u6 = stream_uniform<R>(6, st, pid, in, a.key0, a.key1);
      R sn, cs;
      Math<R>::sincos2pi(u6, &sn, &cs);
      E = (R)init_mean + (R)init_sigma * (Math<R>::sqrt(R(-2) * Math<R>::log(ue)) * cs);
      E = (E < R(0)) ? -E : E;
      E = (E == R(0)) ? (R)init_mean : E;
    }
  } else {
    E = R(-1.5) * P->vt * Math<R>::log(ue);
  }
  R kx, ky, kz;
  random_direction(normk_of(kane_of(V), E), uphi, ucos, kx, ky, kz);
  a.kx[gi] = kx;
  a.ky[gi] = ky;
  a.kz[gi] = kz;
  a.E[gi] = E;
  a.tau[gi] = -Math<R>::log(ut) * P->tau0[v];
  a.vs[gi] = ((uint32_t)v << 16) | (uint32_t)sub;
  if (a.px) {
    // positions uniform in the periodic box: the density of the bulk
    // handler's initParticlePos per node (emcParticleInitialization.hpp:
    // 13-29) over nodes weighted by their cells
    a.px[gi] = stream_uniform<R>(8, st, pid, in, a.key0, a.key1) * P->box[0];
    a.py[gi] = stream_uniform<R>(9, st, pid, in, a.key0, a.key1) * P->box[1];
    a.pz[gi] = stream_uniform<R>(10, st, pid, in, a.key0, a.key1) * P->box[2];
  }
}

// ---------------------------------------------------------------------------
// launch wrappers (called by the C ABI layer)
// ---------------------------------------------------------------------------
// particles per tile of a step-kernel variant (1 = replay / one per lane)
int tile_size_of(int ppt) { return kTile * ppt; }

// the extended kernels: bath tallies and the screened final states
template <typename R>
bool extended(const StepArgs<R> &a) {
  return (a.tally && a.lds_bins > 0) || a.ext_kinds;
}

// LDS of a block of the production kernel: the parameters, tallies and
// (8-byte aligned) staged window sums, then per wave the particles, the queue
// and the step sums
template <typename R, int PPT, bool POS>
size_t fused_lds(StepArgs<R> &a) {
  a.lds_hot = extended(a) ? (int)((sizeof(uint32_t) * 2 * (size_t)a.lds_bins + 8 +
                                   sizeof(R) * (size_t)a.lds_win + 15) & ~size_t(15))
                          : 0;
  a.lds_wave = (int)((fused_state_bytes<R, PPT, POS>() +
                      sizeof(double) * kRing * (size_t)a.n_obs + 15) & ~size_t(15));
  return (size_t)a.lds_params + a.lds_hot + (size_t)kSubs * a.lds_wave;
}

// the particles per lane that a block's LDS holds, at most ppt
template <typename R, bool POS>
int fitting_ppt_t(StepArgs<R> a, int ppt) {
  if (!POS && ppt >= 8 && fused_lds<R, 8, POS>(a) <= kMaxBulkLds)
    return 8;
  if (ppt >= 4 && fused_lds<R, 4, POS>(a) <= kMaxBulkLds)
    return 4;
  if (ppt >= 2 && fused_lds<R, 2, POS>(a) <= kMaxBulkLds)
    return 2;
  return 1;
}
template <typename R>
int fitting_ppt(StepArgs<R> a, int ppt) {
  return a.px ? fitting_ppt_t<R, true>(a, ppt) : fitting_ppt_t<R, false>(a, ppt);
}
template int fitting_ppt<float>(StepArgs<float>, int);
template int fitting_ppt<double>(StepArgs<double>, int);

// the same for the kernel of one-step launches
template <typename R>
size_t once_lds(StepArgs<R> &a) {
  a.lds_wave =
      (int)((once_wave_bytes<R>() + sizeof(double) * (size_t)a.n_obs + 15) & ~size_t(15));
  return (size_t)a.lds_params + a.lds_hot + (size_t)kSubs * a.lds_wave;
}

// Launches that keep the particles in the lanes' registers (k_bulk_lanes) where
// k_bulk_fused would hold them in LDS or k_bulk_once stream them.  us per step
// here / there, si: one valley of 13 mechanisms, tv: two valleys, 1 fs:
// - one per lane: up to four steps.  10k FP32 si, 1 / 4 steps: 9.4 / 11.6,
//   4.5 / 5.0; 8M FP64: si 313 / 368, 214 / 230, tv 279 / 447, 176 / 231; a tie
//   at 4 steps of tv in FP32 (1M: 13.9 / 13.9).  Where the waves fill the chip
//   and the registers of k_bulk_fused leave two waves per SIMD, longer ones
//   too: FP64 tv to 32 steps (8M: 148 / 161; where events are frequent a tie by
//   then, 10 fs 279 / 282, 1M 38.2 / 37.4); with positions any number (1M si, 64
//   steps: FP64 30.4 / 38.0, FP32 12.6 / 13.8; FP32 tv to 8: 13.6 / 13.7)
// - one step of two or four per lane, several valleys: while events are rare
//   (at 0.044 expected per particle 4M FP64 100 / 102, 10M 279 / 305, 8M FP32
//   74 / 84; at 0.088 4M FP64 112 / 109; with baths at 0.2 204 / 170 at 1M;
//   two per lane in FP64 up to a million particles: 250k 17 / 20, 4M 123 / 116),
//   always for two in FP32 (4M: 49 / 58, 0.35 events 63 / 76) and with
//   positions (8M FP64: 283 / 358)
// - one step with positions of one valley, two per lane (k_bulk_once spills):
//   300k FP32 20.3 / 21.0
// events: expected per particle and step
template <typename R>
bool keeps_lanes(const StepArgs<R> &a, int ppt, double events) {
  const bool fp64 = sizeof(R) == 8;
  if (ppt == 1) {
    if (a.n_steps <= 4)
      return true;
    if ((long long)a.n_tiles * kSubs < 2048)  // two waves on each of the 1024 SIMDs
      return false;
    if (a.px)
      return fp64 || a.max_v == 1 || a.n_steps <= 8;
    return fp64 && a.max_v > 1 && a.n_steps <= 32;
  }
  if (a.n_steps > 1 || ppt > 4)
    return false;
  if (a.max_v == 1)
    return a.px && ppt == 2;
  if (a.px || (!fp64 && ppt == 2))
    return true;
  return events < 0.05 && (ppt == 4 || (long long)a.n_tiles * kSubs <= 8192);
}

template <typename R, int PPT, bool HOT, bool POS>
hipError_t launch_fused(StepArgs<R> a, double events, hipStream_t st) {
  size_t lds = fused_lds<R, PPT, POS>(a);
  const void *f = a.max_v == 1 ? (const void *)k_bulk_fused<R, PPT, HOT, POS, 1>
                               : (const void *)k_bulk_fused<R, PPT, HOT, POS, kMaxV>;
  if constexpr (!POS && PPT > 1 && streams_one_step<R>(PPT)) {
    if (a.n_steps == 1 && a.max_v == 1) {
      lds = once_lds<R>(a);
      f = (const void *)k_bulk_once<R, PPT, HOT>;
    }
  }
  if (keeps_lanes(a, PPT, events)) {
    lds = (size_t)a.lds_params + a.lds_hot;
    if constexpr (PPT == 1 || (PPT == 2 && POS))
      if (a.max_v == 1)
        f = (const void *)k_bulk_lanes<R, PPT, HOT, POS, 1>;
    if constexpr (PPT <= 4)
      if (a.max_v > 1)
        f = (const void *)k_bulk_lanes<R, PPT, HOT, POS, kMaxV>;
  }
  if (lds > kMaxBulkLds)
    return hipErrorInvalidValue;
  if (lds > 64 * 1024) {
    // the limit is the kernel's, not the launch's: every context sets the same
    // one, whichever thread comes between this call and the launch
    const hipError_t e =
        hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxBulkLds);
    if (e != hipSuccess)
      return e;
  }
  void *args[] = {&a};
  return hipLaunchKernel(f, dim3(a.n_tiles), dim3(kTile), args, lds, st);
}

template <typename R, bool HOT>
hipError_t launch_steps_t(const StepArgs<R> &a, int mode, int ppt, double events, hipStream_t st) {
  if (mode == 1) {
    // tallies, then (8-byte aligned) the staged window sums
    const dim3 g(a.n_tiles), b(kTile);
    const size_t lds = HOT ? sizeof(uint32_t) * 2 * (size_t)a.lds_bins + 8 +
                                 sizeof(R) * (size_t)a.lds_win
                           : 0;
    if (a.px)
      hipLaunchKernelGGL((k_bulk_replay<R, HOT, true>), g, b, lds, st, a);
    else
      hipLaunchKernelGGL((k_bulk_replay<R, HOT, false>), g, b, lds, st, a);
    return hipGetLastError();
  }
  if (a.px) {  // positions tracked
    switch (ppt) {
    case 1:
      return launch_fused<R, 1, HOT, true>(a, events, st);
    case 2:
      return launch_fused<R, 2, HOT, true>(a, events, st);
    case 4:
      return launch_fused<R, 4, HOT, true>(a, events, st);
    default:
      return hipErrorInvalidValue;
    }
  }
  switch (ppt) {
  case 1:
    return launch_fused<R, 1, HOT, false>(a, events, st);
  case 2:
    return launch_fused<R, 2, HOT, false>(a, events, st);
  case 4:
    return launch_fused<R, 4, HOT, false>(a, events, st);
  case 8:
    return launch_fused<R, 8, HOT, false>(a, events, st);
  default:
    return hipErrorInvalidValue;
  }
}

template <typename R>
hipError_t launch_steps(const StepArgs<R> &a, int mode, int ppt, double events, hipStream_t st) {
  if (a.n_tiles <= 0)
    return hipSuccess;
  if (extended(a))
    return launch_steps_t<R, true>(a, mode, ppt, events, st);
  return launch_steps_t<R, false>(a, mode, ppt, events, st);
}

template <typename R>
hipError_t launch_observe(const StepArgs<R> &a, hipStream_t st) {
  if (a.n_tiles <= 0)
    return hipSuccess;
  hipLaunchKernelGGL((k_observe<R>), dim3(a.n_tiles), dim3(kTile), 0, st, a);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_init(const StepArgs<R> &a, double init_mean, double init_sigma,
                       hipStream_t st) {
  if (a.n_tiles <= 0)
    return hipSuccess;
  hipLaunchKernelGGL((k_init_thermal<R>), dim3(a.n_tiles), dim3(kTile), 0, st, a, init_mean,
                     init_sigma);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_bath_step(const BathStepArgs<R> &a, int n_groups, hipStream_t st) {
  if (n_groups <= 0)
    return hipSuccess;
  hipLaunchKernelGGL((k_bath_step<R>), dim3(n_groups), dim3(kBathThreads), 0, st, a);
  if (a.n_jobs > 0) {
    const dim3 g(kRebuildChunks, a.n_jobs);
    hipLaunchKernelGGL((k_rebuild_rates<R>), g, dim3(kRebuildChunk), 0, st, a);
    hipLaunchKernelGGL((k_rebuild_norm<R>), g, dim3(kRebuildChunk), 0, st, a);
  }
  return hipGetLastError();
}

template <typename R>
hipError_t launch_rebuild(const BathStepArgs<R> &a, int n_jobs, hipStream_t st) {
  if (n_jobs <= 0)
    return hipSuccess;
  hipLaunchKernelGGL((k_bath_refresh<R>), dim3(n_jobs), dim3(kBathThreads), 0, st, a);
  return hipGetLastError();
}

// number of chunk pairs per output value for the largest instance
int reduce_chunks(long long max_count, int tile_size) {
  const long long nt = (max_count + tile_size - 1) / tile_size * kSubs;
  return (int)((nt + kChunk - 1) / kChunk > 0 ? (nt + kChunk - 1) / kChunk : 1);
}

hipError_t launch_reduce(const double *partial, int n_steps, int n_tiles, int n_obs, int tile_size,
                         const long long *inst_start, const long long *inst_count, int n_inst,
                         int n_chunks, double *chunk_buf, double *out, int out_step0,
                         int out_total, hipStream_t st) {
  if (n_steps <= 0 || n_inst <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_reduce_chunks, dim3(n_chunks, n_steps * n_obs, n_inst), dim3(256), 0, st,
                     partial, n_tiles, tile_size, inst_start, inst_count, n_chunks, chunk_buf,
                     n_chunks == 1 ? out : nullptr, n_obs, out_step0, out_total);
  if (n_chunks > 1)
    hipLaunchKernelGGL(k_reduce_final, dim3(n_steps * n_obs, n_inst), dim3(256), 0, st, chunk_buf,
                     n_chunks, n_obs, out, out_step0, out_total);
  return hipGetLastError();
}

template hipError_t launch_steps<float>(const StepArgs<float> &, int, int, double, hipStream_t);
template hipError_t launch_steps<double>(const StepArgs<double> &, int, int, double, hipStream_t);
template hipError_t launch_observe<float>(const StepArgs<float> &, hipStream_t);
template hipError_t launch_observe<double>(const StepArgs<double> &, hipStream_t);
template hipError_t launch_init<float>(const StepArgs<float> &, double, double, hipStream_t);
template hipError_t launch_init<double>(const StepArgs<double> &, double, double, hipStream_t);
template hipError_t launch_bath_step<float>(const BathStepArgs<float> &, int, hipStream_t);
template hipError_t launch_bath_step<double>(const BathStepArgs<double> &, int, hipStream_t);
template hipError_t launch_rebuild<float>(const BathStepArgs<float> &, int, hipStream_t);
template hipError_t launch_rebuild<double>(const BathStepArgs<double> &, int, hipStream_t);

}  // namespace emcgpu
