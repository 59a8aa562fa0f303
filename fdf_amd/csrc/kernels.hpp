// kernels.hpp -- gfx950 kernels of the per-step particle loop.
//
// One thread per particle (or node / cell / face).  Block size 256 = four
// 64-wide wavefronts.  All FP64 arithmetic that must match the reference is
// written in the reference's operation order; the build uses
// -ffp-contract=off, and FP32 code asks for fused multiply-adds explicitly.
// More than one source file includes this header: its kernels are templates
// or static.
#pragma once
#include "picgpu_internal.hpp"

namespace picgpu {

constexpr int kBlock = 256;

__device__ __forceinline__ void unpack_cell(int32_t c, int IM, int JM, int &i, int &j, int &k) {
  i = c % IM;
  int r = c / IM;
  j = r % JM;
  k = r / JM;
}

// The same decoding without integer division, given rI = fl(1/IM) and
// rIJ = fl(1/(IM*JM)) in FP64: (c + 0.5) * rIJ lies within (c/(IM*JM)) * 2^-51
// of (c + 0.5)/(IM*JM), which is at least 0.5/(IM*JM) from an integer, so the
// truncation is floor(c / (IM*JM)) for every c < 2^31 (likewise for j).
struct CellIdx {
  int IM, JM;
  double rI, rIJ;
};
__device__ __forceinline__ void unpack_cell(int32_t c, const CellIdx &x, int &i, int &j, int &k) {
  k = (int)(((double)c + 0.5) * x.rIJ);
  const int r = c - k * (x.IM * x.JM);
  j = (int)(((double)r + 0.5) * x.rI);
  i = r - j * x.IM;
}
__device__ __forceinline__ CellIdx cell_idx(const GridView &g) { return CellIdx{g.IM, g.JM, g.rI, g.rIJ}; }
__device__ __forceinline__ int32_t pack_cell(int i, int j, int k, int IM, int JM) {
  return (int32_t)(i + IM * (j + JM * k));
}

// Cycle detection for the walk (Brent).  For a fixed point the walk is a
// deterministic map cell -> next cell (walkingsearch.c:882-959), so a
// revisited cell means the walk is periodic: it will never accept a cell
// and the reference ends it LOST at MAX_TRAVERSAL (:1206-1212).  Warped
// k-faces leave thin gaps in which walks cycle among two or three cells;
// concluding them at the first revisit gives the reference's outcome
// without holding a 64-lane wavefront for up to 1000 iterations.
struct CycleGuard {
  int32_t saved = -1;
  int power = 1, lam = 0;
  __device__ __forceinline__ bool revisit(int32_t c) {
    if (c == saved) return true;
    if (++lam == power) {
      saved = c;
      power <<= 1;
      lam = 0;
    }
    return false;
  }
};

// ---------------------------------------------------------------------------
// ResetAllParticleStatuses (ParticleMotion.c:2149-2176) fused with
// UpdateAllParticlePositions (ParticleMotion.c:19-95): x += v*dt.
// ---------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(kBlock) void k_reset_advect(int64_t n, double *__restrict__ pos,
                                                         const R *__restrict__ vel,
                                                         int32_t *__restrict__ status, double dt,
                                                         int do_reset, int do_advect) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  if (do_reset && status[p] == ST_LOCATED) status[p] = ST_NEEDS;
  if (do_advect) {
#pragma unroll
    for (int c = 0; c < 3; ++c) pos[3 * p + c] += (double)vel[3 * p + c] * dt;
  }
}

// ---------------------------------------------------------------------------
// Walking search.  Each wavefront owns `chunk` consecutive particles and keeps
// its 64 lanes busy: a lane whose walk ends takes the next unassigned
// particle of the chunk (ballot + prefix count), so long and short walks are
// regrouped instead of idling until the wave's longest walk ends.
//
// A walk is a chain of dependent record loads, so its time is iterations times
// the latency of one load and its evaluation, and a large launch's is the
// record lines it touches.  In FP64 the steps of a walk are therefore decided
// on the 128-byte FP32 record (a.filter): where the filter certifies every
// face (planes_fp32_certified), the reference's FP64 distances have those
// signs and lie outside the zero band, so the step is the reference's.  The
// 304-byte FP64 record (3 or 4 lines) is read where the filter certifies the
// owner, for the weights, and where it certifies nothing.  Lanes wait for that
// evaluation (ph 2) until kExactGroup of them can make it together: walks end
// at different iterations, and a wavefront would otherwise pay for the FP64
// path in nearly every one (groups of 8, 24 and 48 measure alike).
// 8,388,608 particles moved by up to 1.5 cells an axis in 128x128x256 cells, in
// random order, FP64: 2.60 -> 1.33 ms (about 9.1 -> 6.3 GB of record lines).
//
// Long walks are bound by instructions (four wavefronts a SIMD, about 300 an
// iteration), so the iterations run in a loop of their own, branch-free but for
// the walk's ends (about 120): the wavefront turns to ended walks, new particles
// and full evaluations when kStopped lanes have stopped.  10,000 particles from
// cell (0,0,0) of 128x128x192, FP64: 395 -> 242 us; of 24x24x24: 60 -> 44.
// ---------------------------------------------------------------------------
template <typename R>
struct LocateArgs {
  GridView g;
  const void *planes;  // CellPlanes64 (FP64) or CellPlanes32 (FP32) per cell
  const CellPlanes32 *filter;  // FP64: the FP32 records (null: every evaluation is made in FP64)
  int64_t n;
  int64_t chunk;
  const double *pos;
  int32_t *cell;
  R *w;
  int32_t *status;
  const int32_t *guess;  // may be null
  const int32_t *order;  // may be null: the q-th particle visited is order[q]
  int32_t *steps_out;    // may be null
  unsigned long long *walk_hist;  // null, or [kCounterStripes][64] walk-iteration histogram
  unsigned long long *counters;
  int max_traversal;
  double thresh_scale;
  R clamp;
  int skip_lost;
};

// Particles per wavefront: few where the launch would otherwise leave SIMDs
// idle (each SIMD holds 4 of its wavefronts, 4096 on the chip), 256 where
// there are enough, so that a wavefront's last, long walks weigh little.
// 3,000 particles, FP32, call and wait: 63 us at 256 a wavefront, 42 us at 16.
constexpr int64_t kLocateWaves = 4096;
inline int64_t locate_chunk(int64_t n, int lanes) {
  const int64_t c = (n + kLocateWaves - 1) / kLocateWaves, least = lanes > 1 ? 64 / lanes : 16;
  return c < least ? least : c > 256 ? 256 : c;
}
inline int64_t locate_blocks(int64_t n, int64_t chunk) {
  const int64_t waves = (n + chunk - 1) / chunk;
  return (waves * 64 + kBlock - 1) / kBlock;
}
constexpr int kExactGroup = 24;
// FP32: the lanes at a face that is not certified for which a wavefront leaves its
// iterations.  They are few, and a lane that waits for others of its kind holds up
// its own walk: of 24, as in FP64, and with the last ones left to the end of the
// wavefront's walks, 16.8M out of cell (0,0,0) of a 128x128x1024 tube, the lines
// in LDS 16.8 ms, without 19.0; of 2, 15.3 and 17.5 (17.6 with fallbacks in
// place).  One at a time: 14.2 and 16.3, but 300,000 in a 48x48x250 tube 293 ->
// 328 us and 2M in 24x24x24 cells 413 -> 456.
constexpr int kFallbacks = 2;
constexpr int kHeld = 2;      // full evaluations that took a walk on before it is taken on by them alone
constexpr int kStopped = 16;  // lanes without a walk at which a wavefront turns to them

// Walks that all start in cell (0,0,0) are long.  In a grid of at least
// kLocateLong cells along some axis, lanes a particle (k_locate_ahead): 16 up to
// 16,384 particles, 4 up to 131,072, while the evaluations that no walk reaches
// still find idle lanes.  The locate in FP64, us, one lane / 16 / 4:
//   n          20x20x280          63x47x129        24x24x24
//   10,000     221 /  74 / 106    166 / 108 / 125   44 / 53 / 52
//   60,000     452 /   - / 247    245 /   - / 202   70 /  - / 76
//   100,000    499 /   - / 344    271 /   - / 271   76 /  - / 101
// and before both, 342, 265 and 60 at 10,000.
constexpr int kLocateLong = 48;
inline int locate_ahead(int64_t n) { return n <= kLocateWaves * 4 ? 16 : n <= kLocateWaves * 32 ? 4 : 1; }
// From kLocateLines particles on, the records' lines through LDS (wave_records)
// in the iterations that at least kLinesLanes lanes of the wavefront evaluate.
// The staging costs a wavefront the same for one walk as for 64, so that a few
// long walks among lanes that have ended (the bent pipe from cell (0,0,0): most
// walks leave the grid after two or three iterations, the others take hundreds)
// are better off with loads of their own.  The locate, us, own loads / all
// iterations staged / those of 32 lanes:
//   n            48x48x250 tube     63x47x129 cube     128x128x192 cube
//   300,000 FP64  202 /  274 / 206   440 /  419 / 369   740 /  718 / 676
//   300,000 FP32  274 /  341 / 287   461 /  428 / 379   839 /  756 / 722
//   2M FP64       665 /  617 / 537  2107 / 1686 / 1574 3473 / 3026 / 2931
//   2M FP32       640 /  629 / 576  2330 / 1772 / 1695 4180 / 3358 / 3170
// 16.8M FP32 in a 128x128x1024 tube: 18.95 / 19.24 / 16.74 ms.  (FP32 with lanes that
// wait for 24 uncertified faces; kFallbacks takes off up to 7 %, here 17.4 / - / 15.3.)
// 16 or 48 lanes in place of 32 measure within 5 %.  Below the line the LDS gains less than it costs
// where walks are short: 262,144 particles, own loads / 32 lanes, the tube 177 / 192
// in FP32, the cubes 366 / 319 and 619 / 482; 140,000: 185 / 204, 297 / 308, 452 / 438.
constexpr int64_t kLocateLines = 1 << 18;
constexpr int kLinesLanes = 32;

// The FP32 record of cell l for each lane of a wavefront (l < 0: none), all
// lanes taking part; stage: 64 records of LDS, the wavefront's own.
// A lane that reads the 128 bytes of its own record makes 8 loads that each
// touch a line of its own in every lane.  Here 8 lanes read one record's line
// together and LDS turns it round; the chunks of record r are stored XORed
// with r mod 8, so that neither the writes (8 chunks of a record) nor the
// reads (a chunk of 8 records) meet in a bank.
__device__ __forceinline__ CellPlanes32 wave_records(const CellPlanes32 *__restrict__ recs, int32_t l, float4 *stage,
                                                     int lane) {
  const int row = lane >> 3, col = lane & 7;
  const float4 *src = reinterpret_cast<const float4 *>(recs);
  float4 v[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int32_t lr = __shfl(l, 8 * b + row);
    v[b] = src[(int64_t)(lr < 0 ? 0 : lr) * 8 + col];
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int b = 0; b < 8; ++b) stage[(8 * b + row) * 8 + (col ^ row)] = v[b];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  CellPlanes32 r;
#pragma unroll
  for (int c = 0; c < 6; ++c) r.plane[c] = stage[lane * 8 + (c ^ col)];
  const float4 t0 = stage[lane * 8 + (6 ^ col)], t1 = stage[lane * 8 + (7 ^ col)];
  r.v0[0] = __hiloint2double(__float_as_int(t0.y), __float_as_int(t0.x));
  r.v0[1] = __hiloint2double(__float_as_int(t0.w), __float_as_int(t0.z));
  r.v0[2] = __hiloint2double(__float_as_int(t1.y), __float_as_int(t1.x));
  r.thr = t1.z;
  r.amax = t1.w;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  return r;
}

// Statistics of a locate launch: one atomic a wavefront and word, and the
// workgroup's histogram of walk iterations.
template <typename R>
__device__ __forceinline__ void locate_tally(const LocateArgs<R> &a, int64_t base, int lane,
                                             unsigned long long my_iters, unsigned long long my_fb, unsigned my_max,
                                             unsigned my_loc, unsigned my_lost, int my_err,
                                             const int32_t *shist) {
  if (base < a.n) {
    for (int off = 32; off > 0; off >>= 1) {
      my_iters += __shfl_xor(my_iters, off);
      const unsigned om = __shfl_xor(my_max, off);
      my_max = my_max > om ? my_max : om;
      my_fb += __shfl_xor(my_fb, off);
      my_loc += __shfl_xor(my_loc, off);
      my_lost += __shfl_xor(my_lost, off);
      my_err |= __shfl_xor(my_err, off);
    }
    if (lane == 0) {
      unsigned long long *ctr = counter_stripe(a.counters);
      atomicAdd(&ctr[C_WALK_ITERS], my_iters);
      atomicMax(&ctr[C_WALK_MAX], (unsigned long long)my_max);
      if (my_fb) atomicAdd(&ctr[C_FALLBACKS], my_fb);
      if (my_loc) atomicAdd(&ctr[C_LOCATED], (unsigned long long)my_loc);
      if (my_lost) atomicAdd(&ctr[C_LOST], (unsigned long long)my_lost);
      if (my_err) atomicOr(&ctr[C_ERROR], 1ull);
    }
  }
  if (a.walk_hist) {
    __syncthreads();
    if (threadIdx.x < 64 && shist[threadIdx.x] > 0)
      atomicAdd(&a.walk_hist[(blockIdx.x & (kCounterStripes - 1)) * 64 + threadIdx.x],
                (unsigned long long)shist[threadIdx.x]);
  }
}

template <typename R, bool EXACT, bool LINES>
__global__ __launch_bounds__(kBlock, 4) void k_locate(LocateArgs<R> a) {
  __shared__ int32_t shist[64];
  __shared__ float4 stage[LINES ? kBlock * 8 : 1];
  float4 *const my_stage = stage + (LINES ? (threadIdx.x & ~63) * 8 : 0);
  if (threadIdx.x < 64) shist[threadIdx.x] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t base = wave * a.chunk;
  const int64_t end = base + a.chunk < a.n ? base + a.chunk : a.n;
  int64_t cursor = base;
  // a lane's state: no particle; walking; at a cell whose evaluation waits
  // (kHold: FP64's owner, and what the filter does not certify); ended
  enum : int { kIdle = 0, kWalk = 1, kHold = 2, kOwner = 3, kLost = 4 };
  int ph = kIdle;
  int32_t p = 0;  // n < 2^31
  int ci = 0, cj = 0, ck = 0, steps = 0;
  int32_t lc = 0;  // ci + IM (cj + JM ck); used only inside the grid
  const int32_t sj = a.g.IM, sk = a.g.IM * a.g.JM;
  const CellPlanes32 *const recs = EXACT ? a.filter : static_cast<const CellPlanes32 *>(a.planes);
  int32_t saved = -1;  // the walk's cell at iteration 1, 3, 7, 15 ... (CycleGuard's test)
  int held = 0;        // full evaluations of the walk that took it on
  double x[3] = {0.0, 0.0, 0.0};
  float d[6];
  unsigned long long my_iters = 0;
  unsigned long long my_fb = 0;
  unsigned my_max = 0, my_loc = 0, my_lost = 0;
  int my_err = 0;
  const unsigned long long lane_mask_lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  auto step = [&](const auto dist[6]) {
    int di, dj, dk;
    step_of(dist, di, dj, dk);
    ci += di;
    cj += dj;
    ck += dk;
    lc += di + dj * sj + dk * sk;
    ph = steps >= a.max_traversal ? kLost : kWalk;  // MAX_TRAVERSAL (:1206-1212)
  };
  // an iteration's tests before its evaluation (walkingsearch.c:1123-1132)
  auto arrive = [&]() {
    steps++;
    if ((unsigned)ci >= (unsigned)a.g.IM || (unsigned)cj >= (unsigned)a.g.JM || (unsigned)ck >= (unsigned)a.g.KM) {
      ph = kLost;  // walked outside the global domain: LOST
    } else if (lc == saved) {
      ph = kLost;  // periodic walk: LOST at MAX_TRAVERSAL (:1206-1212)
      steps = a.max_traversal;
    } else {
      if ((steps & (steps + 1)) == 0) saved = lc;
      ph = kHold;
    }
  };
  while (true) {
    const unsigned long long idle = __ballot(ph == kIdle);
    if (idle != 0ull && cursor < end) {
      if (ph == kIdle) {
        const int64_t q = cursor + __popcll(idle & lane_mask_lt);
        if (q < end) {
          const int32_t pq = a.order ? a.order[q] : (int32_t)q;
          const int32_t st = a.status[pq];
          int32_t c = a.cell[pq];
#pragma unroll
          for (int t = 0; t < 3; ++t) x[t] = a.pos[3 * (int64_t)pq + t];
          if (!(st == ST_LOCATED || (a.skip_lost && st == ST_LOST))) {
            p = pq;
            ph = kWalk;
            if (c < 0 && a.guess) c = a.guess[pq];
            ci = cj = ck = 0;  // (info.xs, info.ys, info.zs) on one rank, walkingsearch.c:611-616
            if (c >= 0) unpack_cell(c, cell_idx(a.g), ci, cj, ck);
            lc = c >= 0 ? c : 0;
            steps = 0;
            saved = -1;
            held = 0;
          } else if (a.steps_out) {
            a.steps_out[pq] = 0;
          }
        }
      }
      cursor += __popcll(idle);
    }
    unsigned long long walking = __ballot(ph == kWalk);
    if (walking != 0ull) {
      // iterations of the walk (walkingsearch.c:1123-1203) until kStopped lanes have stopped
      const int least = cursor < end ? 64 - kStopped : 0;
      do {
        bool eval = false;
        if (ph == kWalk) {
          arrive();
          eval = ph == kHold;
        }
        auto decide = [&](const CellPlanes32 &rec) {
          if (planes_fp32_certified(rec, x, d)) {
            if (certified_outside(d))
              step(d);
            else if (!EXACT)
              ph = kOwner;
          }
        };
        if (LINES && __popcll(__ballot(eval)) >= kLinesLanes) {
          const CellPlanes32 rec = wave_records(recs, eval ? lc : -1, my_stage, lane);
          if (eval) decide(rec);
        } else {
          if (eval && (!EXACT || recs)) decide(recs[lc]);
        }
        walking = __ballot(ph == kWalk);
      } while (__popcll(walking) > least && (EXACT || __popcll(__ballot(ph == kHold)) < kFallbacks));
    }
    const unsigned long long waiting = __ballot(ph == kHold);
    if ((walking | waiting) == 0ull && __ballot(ph != kIdle) == 0ull && cursor >= end) break;
    if (waiting != 0ull && (walking == 0ull || __popcll(waiting) >= (EXACT ? kExactGroup : kFallbacks))) {
      // the last walks of a wavefront that are certified nowhere (a point within
      // the filter's bound of a plane along the grid) stay here to their end
      const bool last = walking == 0ull && cursor >= end;
      while (ph == kHold) {
        R df[6];
        unsigned long long fb = 0;
        if (!eval_cell_planes<R, EXACT>(a.planes, a.g, ci, cj, ck, x, a.thresh_scale, df, fb)) {
          my_err = 1;
          ph = kLost;
        } else if (point_accepted<R>(df)) {
          if constexpr (EXACT) {
            R wv[3];
            weights_from_distances<R>(df, a.clamp, wv);
#pragma unroll
            for (int t = 0; t < 3; ++t) a.w[3 * (int64_t)p + t] = wv[t];
          } else {
#pragma unroll
            for (int t = 0; t < 6; ++t) d[t] = df[t];
          }
          ph = kOwner;
        } else {
          step(df);
          if (++held > kHeld && last && ph == kWalk) arrive();
        }
        my_fb += fb;
      }
    }
    if (ph >= kOwner) {
      if (ph == kOwner) {
        if constexpr (!EXACT) {
          float wv[3];
          weights_from_distances<float>(d, a.clamp, wv);
#pragma unroll
          for (int t = 0; t < 3; ++t) a.w[3 * (int64_t)p + t] = wv[t];
        }
        a.cell[p] = lc;
        a.status[p] = ST_LOCATED;
        my_loc++;
      } else if (!my_err) {
        a.cell[p] = -1;
        a.status[p] = ST_LOST;
        my_lost++;
      }
      if (a.steps_out) a.steps_out[p] = steps;
      if (a.walk_hist) atomicAdd(&shist[steps < 63 ? steps : 63], 1);
      my_iters += steps;
      my_max = my_max > (unsigned)steps ? my_max : (unsigned)steps;
      ph = kIdle;
    }
  }
  locate_tally(a, base, lane, my_iters, my_fb, my_max, my_loc, my_lost, my_err, shist);
}

// The walk of few particles: G lanes a particle, which evaluate the next G
// cells of its walk at once.  A launch of few particles is bound by the
// latency of a walk's record loads, one after another, while most lanes of the
// chip have no particle.  A walk mostly goes on in the direction of its last
// step: lane m evaluates the cell m such steps ahead, and the walk takes the
// lanes' steps as long as each is the predicted one, up to and with the first
// that is not.  These are the cells, steps and iterations of the walk taken
// one by one; an evaluation that the walk does not reach is dropped.
// The group looks twice as far ahead as the row it has just taken, so that a
// walk with many turns costs few loads.
template <typename R, bool EXACT, int G>
__global__ __launch_bounds__(kBlock, 4) void k_locate_ahead(LocateArgs<R> a) {
  static_assert(G >= 2 && G <= 16 && (G & (G - 1)) == 0, "G lanes a particle");
  constexpr unsigned kGroupMask = (1u << G) - 1u;
  __shared__ int32_t shist[64];
  if (threadIdx.x < 64) shist[threadIdx.x] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int m = lane & (G - 1), first = lane & ~(G - 1);  // place in the group, the group's first lane
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t base = wave * a.chunk;
  const int64_t end = base + a.chunk < a.n ? base + a.chunk : a.n;
  int64_t cursor = base;
  // the same in every lane of a group, but for d in the lane of the owner
  enum : int { kIdle = 0, kWalk = 1, kHold = 2, kOwner = 3, kLost = 4 };
  int ph = kIdle;
  int32_t p = 0;  // n < 2^31
  int ci = 0, cj = 0, ck = 0, steps = 0;
  int di = 0, dj = 0, dk = 0;  // the last step
  int32_t lc = 0, dl = 0;      // cell and step in the linear index
  int reach = 1;               // lanes that look ahead
  int owner = 0;               // the lane (of the group) that holds the owner's distances
  const int32_t sj = a.g.IM, sk = a.g.IM * a.g.JM;
  const CellPlanes32 *const recs = EXACT ? a.filter : static_cast<const CellPlanes32 *>(a.planes);
  int32_t saved = -1;  // cell of an earlier round (CycleGuard's test)
  int round = 0;
  int held = 0;        // full evaluations of the walk that took it on
  double x[3] = {0.0, 0.0, 0.0};
  float d[6];
  unsigned long long my_iters = 0;
  unsigned long long my_fb = 0;
  unsigned my_max = 0, my_loc = 0, my_lost = 0;
  int my_err = 0;
  const unsigned long long groups_lt = first == 0 ? 0ull : (~0ull >> (64 - first));
  auto move = [&](int count) {
    ci += count * di;
    cj += count * dj;
    ck += count * dk;
    lc += count * dl;
  };
  auto turn = [&]() {
    dl = di + dj * sj + dk * sk;
    move(1);
    ph = steps >= a.max_traversal ? kLost : kWalk;  // MAX_TRAVERSAL (:1206-1212)
  };
  while (true) {
    const unsigned long long idle = __ballot(ph == kIdle);
    if (idle != 0ull && cursor < end) {
      if (ph == kIdle) {
        const int64_t q = cursor + __popcll(idle & groups_lt) / G;
        if (q < end) {
          const int32_t st = a.status[q];
          int32_t c = a.cell[q];
#pragma unroll
          for (int t = 0; t < 3; ++t) x[t] = a.pos[3 * q + t];
          if (!(st == ST_LOCATED || (a.skip_lost && st == ST_LOST))) {
            p = (int32_t)q;
            ph = kWalk;
            if (c < 0 && a.guess) c = a.guess[q];
            ci = cj = ck = 0;  // (info.xs, info.ys, info.zs) on one rank, walkingsearch.c:611-616
            if (c >= 0) unpack_cell(c, cell_idx(a.g), ci, cj, ck);
            lc = c >= 0 ? c : 0;
            di = dj = dk = 0;
            dl = 0;
            reach = 1;
            steps = 0;
            saved = -1;
            round = 0;
            held = 0;
          } else if (a.steps_out && m == 0) {
            a.steps_out[q] = 0;
          }
        }
      }
      cursor += __popcll(idle) / G;
    }
    unsigned long long walking = __ballot(ph == kWalk);
    if (walking != 0ull) {
      const int least = cursor < end ? 64 - kStopped : 0;
      do {
        // up to G iterations of each group's walk (walkingsearch.c:1123-1203)
        enum : int { STEP = 0, OUT = 1, HOLD = 2, OWNER = 3 };
        int kind = HOLD, si = 0, sj_ = 0, sk_ = 0;
        bool periodic = false;
        if (ph == kWalk) {
          const int i = ci + m * di, j = cj + m * dj, k = ck + m * dk;
          if ((unsigned)i >= (unsigned)a.g.IM || (unsigned)j >= (unsigned)a.g.JM ||
              (unsigned)k >= (unsigned)a.g.KM) {
            kind = OUT;  // walked outside the global domain: LOST (:1127-1132)
          } else if (m < reach && planes_fp32_certified(recs[lc + m * dl], x, d)) {
            if (certified_outside(d)) {
              kind = STEP;
              step_of<float>(d, si, sj_, sk_);
            } else if (!EXACT) {
              kind = OWNER;
            }
          }
        }
        // (the lanes beyond reach break the row of predicted steps)
        const bool predicted = m + 1 < reach && kind == STEP && si == di && sj_ == dj && sk_ == dk;
        const unsigned go = (unsigned)(__ballot(predicted) >> first) & kGroupMask;
        const int len = __ffs(~go) - 1;  // < reach
        // the evaluation after the predicted ones, one number for its kind and step
        const int at = __shfl(kind | (si + 1) << 2 | (sj_ + 1) << 4 | (sk_ + 1) << 6, first + len);
        if (ph == kWalk) {
          // out of the domain, lc is no cell (the kind tells)
          periodic = lc == saved && !(len == 0 && (at & 3) == OUT);
          if (((round + 1) & (round + 2)) == 0) saved = (len == 0 && (at & 3) == OUT) ? -1 : lc;
          ++round;
          if (periodic || len >= a.max_traversal - steps) {
            steps = a.max_traversal;  // LOST there, and a periodic walk at once (:1206-1212)
            ph = kLost;
          } else {
            steps += len + 1;
            move(len);
            reach = 2 * len + 2 < G ? 2 * len + 2 : G;
            if ((at & 3) == STEP) {
              di = ((at >> 2) & 3) - 1;
              dj = ((at >> 4) & 3) - 1;
              dk = ((at >> 6) & 3) - 1;
              turn();
            } else {
              ph = (at & 3) == OUT ? kLost : (at & 3) == HOLD ? kHold : kOwner;
              owner = len;
            }
          }
        }
        walking = __ballot(ph == kWalk);
      } while (__popcll(walking) > least);
    }
    const unsigned long long waiting = __ballot(ph == kHold);
    if ((walking | waiting) == 0ull && __ballot(ph != kIdle) == 0ull && cursor >= end) break;
    if (waiting != 0ull && (walking == 0ull || __popcll(waiting) >= kExactGroup)) {
      // what the filter does not certify (and in FP64 the owner) in full, one
      // cell, or G ahead once that has taken the walk on
      R df[6];
      unsigned long long fb = 0;
      enum : int { STEP = 0, OUT = 1, ERROR = 2, OWNER = 3 };
      int kind = ERROR, si = 0, sj_ = 0, sk_ = 0;
      const int i = ci + m * di, j = cj + m * dj, k = ck + m * dk;
      const bool reached = m == 0 || held > 0;
      if (ph == kHold) {
        if ((unsigned)i >= (unsigned)a.g.IM || (unsigned)j >= (unsigned)a.g.JM || (unsigned)k >= (unsigned)a.g.KM) {
          kind = OUT;
        } else if (reached &&
                   eval_cell_planes<R, EXACT>(a.planes, a.g, i, j, k, x, a.thresh_scale, df, fb)) {
          kind = OWNER;
          if (!point_accepted<R>(df)) {
            kind = STEP;
            step_of<R>(df, si, sj_, sk_);
          }
        }
      }
      const bool predicted = m + 1 < G && held > 0 && kind == STEP && si == di && sj_ == dj && sk_ == dk;
      const unsigned go = (unsigned)(__ballot(predicted) >> first) & kGroupMask;
      const int len = __ffs(~go) - 1;
      const int at = __shfl(kind | (si + 1) << 2 | (sj_ + 1) << 4 | (sk_ + 1) << 6, first + len);
      if (ph == kHold) {
        if (m <= len) my_fb += fb;
        if (len > a.max_traversal - steps) {  // (the first of these iterations is counted in steps)
          steps = a.max_traversal;
          ph = kLost;
        } else {
          steps += len;
          move(len);
          const int kd = at & 3;
          if (kd == STEP) {
            di = ((at >> 2) & 3) - 1;
            dj = ((at >> 4) & 3) - 1;
            dk = ((at >> 6) & 3) - 1;
            reach = 1;
            ++held;
            turn();
          } else if (kd == OWNER) {
            if (m == len) {
              R wv[3];
              weights_from_distances<R>(df, a.clamp, wv);
#pragma unroll
              for (int t = 0; t < 3; ++t) a.w[3 * (int64_t)p + t] = wv[t];
            }
            owner = -1;
            ph = kOwner;
          } else {
            if (kd == ERROR) my_err = 1;
            ph = kLost;
          }
        }
      }
    }
    if (ph >= kOwner) {
      if constexpr (!EXACT) {
        if (ph == kOwner && m == owner) {
          float wv[3];
          weights_from_distances<float>(d, a.clamp, wv);
#pragma unroll
          for (int t = 0; t < 3; ++t) a.w[3 * (int64_t)p + t] = wv[t];
        }
      }
      if (m == 0) {
        if (ph == kOwner) {
          a.cell[p] = lc;
          a.status[p] = ST_LOCATED;
          my_loc++;
        } else if (!my_err) {
          a.cell[p] = -1;
          a.status[p] = ST_LOST;
          my_lost++;
        }
        if (a.steps_out) a.steps_out[p] = steps;
        if (a.walk_hist) atomicAdd(&shist[steps < 63 ? steps : 63], 1);
        my_iters += steps;
        my_max = my_max > (unsigned)steps ? my_max : (unsigned)steps;
      }
      ph = kIdle;
    }
  }
  locate_tally(a, base, lane, my_iters, my_fb, my_max, my_loc, my_lost, my_err, shist);
}

// ---------------------------------------------------------------------------
// Centre -> corner (interpolation.c:598-680): node (i,j,k) = mean of the
// valid cells (i-1..i, j-1..j, k-1..k), summed dk, dj, di in that nesting.
// ucat is compact [KM][JM][IM][3].
//
// A thread takes the node column (i, j) over `chunk` consecutive k (grid: x
// over columns, y over chunks of k).  The four cells of plane k that node k
// sums last are the four that node k+1 sums first, so a long chunk loads four
// cells a node, not eight; the next plane is requested while a node is summed.
// Neighbouring threads take neighbouring i, so loads and stores are
// contiguous.  A chunk is a serial chain of loads, so its length is cut
// (c2c_chunk) until the launch has kC2CWaves wavefronts: the reloaded planes
// come from L2.
// Chunks of 32 planes -> cut: 20x20x280 FP64 29.6 -> 5.3 us, 48x48x250 FP64
// 36 -> 10.5 us, 61x45x131 FP32 28.7 -> 5.9 us; 128x128x512 FP32 keeps 32
// planes, 53 us (201 MB at 3.8 TB/s).
//
// zero [nzero] is cleared by the same launch (the counters and the key
// histogram of the fused step that follows), which saves that step two fill
// launches of about 4 us.
// ---------------------------------------------------------------------------
constexpr int kC2CChunk = 32;
constexpr int64_t kC2CWaves = 4096;
inline int c2c_chunk(int64_t columns, int64_t planes) {
  const int64_t waves = (columns + 63) / 64;
  int chunk = kC2CChunk;
  while (chunk > 1 && waves * ((planes + chunk - 1) / chunk) < kC2CWaves) chunk /= 2;
  return chunk;
}

// the cells (i-1,j-1), (i,j-1), (i-1,j), (i,j) of plane ck (the (dj, di)
// order of the sum); v[c] false for a cell outside the grid
template <typename R>
__device__ __forceinline__ void c2c_plane(int IM, int JM, int KM, const R *__restrict__ ucat, int i, int j, int ck,
                                          R u[4][3], bool v[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int ci = i - 1 + (c & 1), cj = j - 1 + (c >> 1);
    v[c] = ci >= 0 && ci < IM && cj >= 0 && cj < JM && ck >= 0 && ck < KM;
    if (v[c]) {
      const R *p = ucat + 3 * ((int64_t)ci + (int64_t)IM * (cj + (int64_t)JM * ck));
      u[c][0] = p[0];
      u[c][1] = p[1];
      u[c][2] = p[2];
    } else {
      u[c][0] = u[c][1] = u[c][2] = (R)0;
    }
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_center_to_corner(int IM, int JM, int KM, int chunk,
                                                             const R *__restrict__ ucat, R *__restrict__ corner,
                                                             int32_t *__restrict__ zero, int64_t nzero) {
  for (int64_t q = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x; q < nzero;
       q += (int64_t)gridDim.x * gridDim.y * blockDim.x)
    zero[q] = 0;
  const uint32_t col = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nI = (uint32_t)IM + 1u;
  if (col >= nI * ((uint32_t)JM + 1u)) return;
  const int i = (int)(col % nI), j = (int)(col / nI);
  const int64_t plane = (int64_t)nI * (JM + 1);
  // chunks blockIdx.y, blockIdx.y + gridDim.y, ... (one per block unless the
  // grid's y limit binds)
  for (int64_t kc = (int64_t)blockIdx.y * chunk; kc < (int64_t)KM + 1; kc += (int64_t)gridDim.y * chunk) {
  const int k0 = (int)kc;
  const int k1 = k0 + chunk < KM + 1 ? k0 + chunk : KM + 1;
  R lo[4][3], hi[4][3];
  bool vlo[4], vhi[4];
  c2c_plane(IM, JM, KM, ucat, i, j, k0 - 1, lo, vlo);
  c2c_plane(IM, JM, KM, ucat, i, j, k0, hi, vhi);
  for (int k = k0; k < k1; ++k) {
    R nx[4][3];
    bool vnx[4];
    if (k + 1 < k1) c2c_plane(IM, JM, KM, ucat, i, j, k + 1, nx, vnx);
    R s0 = 0, s1 = 0, s2 = 0;
    int cnt = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (vlo[c]) {
        s0 += lo[c][0];
        s1 += lo[c][1];
        s2 += lo[c][2];
        cnt++;
      }
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (vhi[c]) {
        s0 += hi[c][0];
        s1 += hi[c][1];
        s2 += hi[c][2];
        cnt++;
      }
    R *o = corner + 3 * ((int64_t)k * plane + col);
    if (cnt > 0) {
      o[0] = s0 / (R)cnt;
      o[1] = s1 / (R)cnt;
      o[2] = s2 / (R)cnt;
    } else {
      o[0] = o[1] = o[2] = (R)0;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      vlo[c] = vhi[c];
      vhi[c] = vnx[c];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        lo[c][d] = hi[c][d];
        hi[c][d] = nx[c][d];
      }
    }
  }
  }
}

// ---------------------------------------------------------------------------
// Trilinear interpolation (interpolation.c:839-864, 957-1042) per particle
// (interpolation.c:1341-1385): a cell outside the grid gives zero velocity.
// ---------------------------------------------------------------------------
// Trilinear interpolation from the corner values C (interpolation.c:957-1042
// with the weights of :839-864): clamp to [0,1], the eight corner weights in
// the order of :851-858 / 990-999, accumulate corner by corner, divide by the
// weight sum when it exceeds 1e-14.  FP64 mode: the reference operations.
// FP32 mode: fused multiply-adds and one hardware reciprocal.
template <typename R>
__device__ __forceinline__ void trilinear_vals(const R C[8][3], R a1, R a2, R a3, R out[3]) {
  a1 = ((R)0 < ((R)1 < a1 ? (R)1 : a1)) ? ((R)1 < a1 ? (R)1 : a1) : (R)0;
  a2 = ((R)0 < ((R)1 < a2 ? (R)1 : a2)) ? ((R)1 < a2 ? (R)1 : a2) : (R)0;
  a3 = ((R)0 < ((R)1 < a3 ? (R)1 : a3)) ? ((R)1 < a3 ? (R)1 : a3) : (R)0;
  const R oa1 = (R)1 - a1, oa2 = (R)1 - a2, oa3 = (R)1 - a3;
  R wc[8];
  wc[0] = oa1 * oa2 * oa3;
  wc[1] = a1 * oa2 * oa3;
  wc[2] = oa1 * a2 * oa3;
  wc[3] = a1 * a2 * oa3;
  wc[4] = oa1 * oa2 * a3;
  wc[5] = a1 * oa2 * a3;
  wc[6] = oa1 * a2 * a3;
  wc[7] = a1 * a2 * a3;
  R sw = 0, ax = 0, ay = 0, az = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    if constexpr (sizeof(R) == 4) {
      ax = __builtin_fmaf(wc[c], C[c][0], ax);
      ay = __builtin_fmaf(wc[c], C[c][1], ay);
      az = __builtin_fmaf(wc[c], C[c][2], az);
    } else {
      ax += wc[c] * C[c][0];
      ay += wc[c] * C[c][1];
      az += wc[c] * C[c][2];
    }
    sw += wc[c];
  }
  if (sw > (R)1.0e-14) {
    if constexpr (sizeof(R) == 4) {
      const R rs = __builtin_amdgcn_rcpf(sw);
      out[0] = ax * rs;
      out[1] = ay * rs;
      out[2] = az * rs;
    } else {
      out[0] = ax / sw;
      out[1] = ay / sw;
      out[2] = az / sw;
    }
  } else {
    out[0] = out[1] = out[2] = (R)0;
  }
}

template <typename R>
__device__ __forceinline__ void trilinear(int IM, int JM, const R *__restrict__ corner, int i, int j, int k, R a1,
                                          R a2, R a3, R out[3]) {
  const int64_t sy = IM + 1, sz = (int64_t)(JM + 1) * (IM + 1);
  const int64_t b = (int64_t)k * sz + (int64_t)j * sy + i;
  R C[8][3];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int64_t q = b + (c & 1) + ((c >> 1) & 1) * sy + ((c >> 2) & 1) * sz;
    C[c][0] = corner[3 * q];
    C[c][1] = corner[3 * q + 1];
    C[c][2] = corner[3 * q + 2];
  }
  trilinear_vals<R>(C, a1, a2, a3, out);
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_interp(int64_t n, int IM, int JM, int KM, const R *__restrict__ corner,
                                                   const int32_t *__restrict__ cell, const R *__restrict__ w,
                                                   R *__restrict__ vel) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int32_t c = cell[p];
  R out[3] = {(R)0, (R)0, (R)0};
  if (c >= 0) {
    int i, j, k;
    unpack_cell(c, IM, JM, i, j, k);
    trilinear<R>(IM, JM, corner, i, j, k, w[3 * p], w[3 * p + 1], w[3 * p + 2], out);
  }
  vel[3 * p] = out[0];
  vel[3 * p + 1] = out[1];
  vel[3 * p + 2] = out[2];
}

// ---------------------------------------------------------------------------
// Removal flags (ParticleMotion.c:532-625 LOST; :283-383 bounding box with
// IsParticleInBox :106-110).  keep[p] = 1 for survivors.
// ---------------------------------------------------------------------------
static __global__ __launch_bounds__(kBlock) void k_keep_flags(int64_t n, const double *__restrict__ pos,
                                                       const int32_t *__restrict__ status, int check_lost,
                                                       int check_box, double bx0, double by0, double bz0,
                                                       double bx1, double by1, double bz1,
                                                       int32_t *__restrict__ keep,
                                                       unsigned long long *counters) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int k = 0, rl = 0, ro = 0;
  if (p < n) {
    k = 1;
    if (check_lost && status[p] == ST_LOST) {
      k = 0;
      rl = 1;
    } else if (check_box) {
      const double x = pos[3 * p], y = pos[3 * p + 1], z = pos[3 * p + 2];
      bool in = x >= bx0 && x <= bx1 && y >= by0 && y <= by1 && z >= bz0 && z <= bz1;
      if (!in) {
        k = 0;
        ro = 1;
      }
    }
    keep[p] = k;
  }
  // wave totals
  unsigned long long bl = __ballot(rl != 0), bo = __ballot(ro != 0);
  if ((threadIdx.x & 63) == 0) {
    unsigned long long *ctr = counter_stripe(counters);
    if (bl) atomicAdd(&ctr[C_REMOVED_LOST], (unsigned long long)__popcll(bl));
    if (bo) atomicAdd(&ctr[C_REMOVED_OOB], (unsigned long long)__popcll(bo));
  }
}

// Moves every particle p with keep[p] to slot off[p] of the destination
// arrays (off = exclusive scan of keep), preserving order.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_compact(int64_t n, const int32_t *__restrict__ keep,
                                                    const int32_t *__restrict__ off, int64_t base, const double *pos,
                                                    const R *vel, const R *w, const int32_t *cell,
                                                    const int32_t *status, const int64_t *pid, const R *P,
                                                    double *pos2, R *vel2, R *w2, int32_t *cell2,
                                                    int32_t *status2, int64_t *pid2, R *P2) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || !keep[p]) return;
  int64_t q = base + off[p];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    pos2[3 * q + c] = pos[3 * p + c];
    vel2[3 * q + c] = vel[3 * p + c];
    w2[3 * q + c] = w[3 * p + c];
  }
  cell2[q] = cell[p];
  status2[q] = status[p];
  pid2[q] = pid[p];
  P2[q] = P[p];
}

// ---------------------------------------------------------------------------
// Counting sort by owning cell, in PID order within a cell: histogram with a
// provisional slot for each particle, its number and short fields scattered to
// start[c] + slot, then one thread a slot ranks its PID among its cell's and
// moves the particle to start[c] + rank.  Particles with cell < 0 are dropped.
//
// Each access to a particle in arbitrary order costs a line, whatever it takes
// of it, so these go together, in a record: 6M FP32 particles as below, 307 +
// 770 us with the number and the PID in two arrays and the rest gathered,
// 174 + 677 with number, cell and PID in a record, 226 + 494 with status and P too.
//
// The rank costs a cell of L particles L reads by each of L threads, of the
// same few lines; in return every consumer of a cell walks its segment once.
// (Consumers that each looked for the next PID read L^2 serially, in one
// thread, for every face of the cell.)
// 6M FP32 particles in 64x64x256 cells of the bent pipe, in random order: sort
// and P averages 2.1 -> 1.4 ms, face sums of the three directions 3.36 -> 0.16;
// 800,000 FP64 in 80x72x100: face sums 140 -> 30 us.
// ---------------------------------------------------------------------------
static __global__ __launch_bounds__(kBlock) void k_cell_histogram(int64_t n, const int32_t *__restrict__ cell,
                                                           int32_t *__restrict__ count, int32_t *__restrict__ rank) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int32_t c = cell[p];
  rank[p] = c >= 0 ? atomicAdd(&count[c], 1) : -1;
}

template <typename R>
struct alignas(32) SortRec {
  int32_t p, cell;
  int64_t pid;
  R P;
  int32_t status;
};
template <typename R>
__global__ __launch_bounds__(kBlock) void k_slot_scatter(int64_t n, const int32_t *__restrict__ rank,
                                                         const int32_t *__restrict__ start,
                                                         const int32_t *__restrict__ cell,
                                                         const int64_t *__restrict__ pid, const R *__restrict__ P,
                                                         const int32_t *__restrict__ status,
                                                         SortRec<R> *__restrict__ rec) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int32_t c = cell[p];
  if (c < 0) return;
  rec[(int64_t)start[c] + rank[p]] = SortRec<R>{(int32_t)p, c, pid[p], P[p], status[p]};
}

// lane t's value in every lane (t the same in all)
template <typename V>
__device__ __forceinline__ V lane_value(V v, int t) {
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(V, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), t));
  } else {
    const int2 w = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(V, make_int2(__builtin_amdgcn_readlane(w.x, t), __builtin_amdgcn_readlane(w.y, t)));
  }
}

// For each lane with `on`, the number of the PIDs of slots [s, e) that come before
// slot q's, id: the smaller ones, and of equal ones those in slots before q.  q
// is the wavefront's first slot plus the lane; all lanes take part.  Lanes of a
// cell of up to kAlone particles read its PIDs one by one; those of a larger one
// 64 at a load, and pass them round (a staged step without deposition, which
// sorts all the same, FP64: 200,000 in 8x8x8 cells 517 -> 442 us, 2M in 32x32x32
// 778 -> 678; with the order in a cell left to chance 370 and 732).
constexpr int32_t kAlone = 64;
template <typename Pid>
__device__ __forceinline__ int32_t pid_rank(bool on, int32_t s, int32_t e, int64_t q, int64_t id, Pid pid) {
  int32_t r = 0;
  if (on && e - s <= kAlone)
    for (int32_t t = s; t < e; ++t) {
      const int64_t o = pid(t);
      r += (o < id || (o == id && t < q)) ? 1 : 0;
    }
  const int lane = threadIdx.x & 63;
  unsigned long long rest = __ballot(on && e - s > kAlone);
  while (rest != 0ull) {
    const int h = __ffsll(rest) - 1;
    const int32_t hs = __builtin_amdgcn_readlane(s, h), he = __builtin_amdgcn_readlane(e, h);
    const bool mine = on && s == hs;
    const int64_t first = q - lane, last = first + 63;  // the wavefront's slots
    int32_t n = 0;
    for (int32_t t0 = hs; t0 < he; t0 += 64) {
      const int64_t own = pid(t0 + lane < he ? t0 + lane : hs);
      const int32_t m = he - t0 < 64 ? he - t0 : 64;
      if (t0 > last || t0 + 63 < first) {  // slots behind, or before, every lane's
        const bool ahead = t0 < first;
#pragma unroll 8
        for (int32_t x = 0; x < m; ++x) {
          const int64_t o = lane_value(own, x);
          n += ahead ? !(id < o) : o < id;
        }
      } else {
        for (int32_t x = 0; x < m; ++x) {
          const int64_t o = lane_value(own, x);
          n += (o < id || (o == id && t0 + x < q)) ? 1 : 0;
        }
      }
    }
    if (mine) r = n;
    rest &= ~__ballot(mine && e - s > kAlone);
  }
  return r;
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_sort_gather(const int32_t *__restrict__ located,
                                                        const int32_t *__restrict__ start,
                                                        const SortRec<R> *__restrict__ rec,
                                                        const double *__restrict__ pos, const R *__restrict__ vel,
                                                        const R *__restrict__ w, double *__restrict__ pos2, R *__restrict__ vel2,
                                                        R *__restrict__ w2, int32_t *__restrict__ cell2,
                                                        int32_t *__restrict__ status2, int64_t *__restrict__ pid2,
                                                        R *__restrict__ P2) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool on = q < *located;
  SortRec<R> own = {};
  double x[3] = {};
  R v[3] = {}, ww[3] = {};
  int32_t s = 0, e = 0;
  if (on) {
    own = rec[q];
    const int64_t p = own.p;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      x[k] = pos[3 * p + k];
      v[k] = vel[3 * p + k];
      ww[k] = w[3 * p + k];
    }
    s = start[own.cell];
    e = start[own.cell + 1];
  }
  const int32_t r = pid_rank(on, s, e, q, own.pid, [&](int32_t t) { return rec[t].pid; });
  if (!on) return;
  const int64_t d = (int64_t)s + r;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    pos2[3 * d + k] = x[k];
    vel2[3 * d + k] = v[k];
    w2[3 * d + k] = ww[k];
  }
  cell2[d] = own.cell;
  status2[d] = own.status;
  pid2[d] = own.pid;
  P2[d] = own.P;
}

// The same sort without memory for the records: the swarm moved to its
// provisional slots (start given), each slot's rank among its cell's PIDs, and
// the swarm moved to the ranks (start null).  What lies from *located on stays.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_move_swarm(
    int64_t n, const int32_t *__restrict__ start, const int32_t *__restrict__ rank, const double *__restrict__ pos,
    const R *__restrict__ vel, const R *__restrict__ w, const int32_t *__restrict__ cell,
    const int32_t *__restrict__ status, const int64_t *__restrict__ pid, const R *__restrict__ P,
    double *__restrict__ pos2, R *__restrict__ vel2, R *__restrict__ w2, int32_t *__restrict__ cell2,
    int32_t *__restrict__ status2, int64_t *__restrict__ pid2, R *__restrict__ P2) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int32_t c = cell[p];
  if (start && c < 0) return;
  const int64_t q = (start ? (int64_t)start[c] : 0) + rank[p];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    pos2[3 * q + k] = pos[3 * p + k];
    vel2[3 * q + k] = vel[3 * p + k];
    w2[3 * q + k] = w[3 * p + k];
  }
  cell2[q] = c;
  status2[q] = status[p];
  pid2[q] = pid[p];
  P2[q] = P[p];
}
static __global__ __launch_bounds__(kBlock) void k_pid_rank(int64_t n, const int32_t *__restrict__ located,
                                                            const int32_t *__restrict__ start,
                                                            const int32_t *__restrict__ cell,
                                                            const int64_t *__restrict__ pid,
                                                            int32_t *__restrict__ rank) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool on = q < n && q < *located;
  int64_t id = 0;
  int32_t s = 0, e = 0;
  if (on) {
    id = pid[q];
    s = start[cell[q]];
    e = start[cell[q] + 1];
  }
  const int32_t r = pid_rank(on, s, e, q, id, [&](int32_t t) { return pid[t]; });
  if (q < n) rank[q] = on ? s + r : (int32_t)q;
}

// Neumaier-compensated accumulator of the P averages in FP32 (a cell's sum of
// equal P values stays exact at any count); plain sum in FP64.
template <typename R>
struct Acc {
  R s = 0, c = 0;
  __device__ __forceinline__ void add(R v) {
    if constexpr (sizeof(R) == 4) {
      // Neumaier: c collects the rounding error of every s + v, computed
      // exactly and without a branch by Knuth's TwoSum (the same value the
      // |s| >= |v| ordered form gives)
      const R t = s + v;
      const R bv = t - s;
      c += (s - (t - bv)) + (v - bv);
      s = t;
    } else {
      s += v;
    }
  }
  __device__ __forceinline__ R value() const { return s + c; }
};

// Accumulator of the face deposition: a plain sum in R, in the fixed order
// (one cell's particles in PID order).  A face sums a few dozen
// terms at most, so in FP32 its error stays within n * 2^-24 of the summed
// magnitudes, far inside the FP32 mode's 1e-5; a compensated sum costs seven
// instructions an addition instead of one.
template <typename R>
struct FaceAcc {
  R s = 0;
  __device__ __forceinline__ void add(R v) { s += v; }
  __device__ __forceinline__ R value() const { return s; }
};

// P average per cell: sum (interpolation.c:1838-1923) / count
// (interpolation.c:1943-2036), summed in PID order (the order of the swarm
// within a cell after the sort).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_scatter_P(int64_t ncell, const int32_t *__restrict__ start,
                                                      const R *__restrict__ P, R *__restrict__ avg) {
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const int32_t s = start[c], e = start[c + 1];
  Acc<R> acc;
  for (int32_t t = s; t < e; ++t) acc.add(P[t]);
  R cnt = (R)(e - s);
  avg[c] = cnt > (R)0.5 ? acc.value() / cnt : (R)0;
}

// Hexahedron volume as six tetrahedra around the diagonal V0-V5.
__device__ __forceinline__ double cell_volume(const GridView &g, int i, int j, int k) {
  double V[8][3];
  load_vertices(g, i, j, k, V);
  const int T[6][2] = {{1, 2}, {1, 6}, {3, 2}, {3, 4}, {7, 6}, {7, 4}};
  double s = 0.0;
  for (int t = 0; t < 6; ++t) {
    const double *a = V[0], *b = V[T[t][0]], *c = V[T[t][1]], *d = V[5];
    double x0 = b[0] - a[0], x1 = b[1] - a[1], x2 = b[2] - a[2];
    double y0 = c[0] - a[0], y1 = c[1] - a[1], y2 = c[2] - a[2];
    double z0 = d[0] - a[0], z1 = d[1] - a[1], z2 = d[2] - a[2];
    double det = x0 * (y1 * z2 - y2 * z1) + x1 * (y2 * z0 - y0 * z2) + x2 * (y0 * z1 - y1 * z0);
    s += fabs(det);
  }
  return s / 6.0;
}

// Face volume fraction = count * V_p / V_dual with V_dual = half the summed
// volumes of the adjacent cells (lower cell first).
template <typename R>
__device__ __forceinline__ double face_volfrac(int dir, const GridView &g, const R *__restrict__ face, double vp,
                                               int64_t f) {
  const int fI = g.IM + (dir == 0), fJ = g.JM + (dir == 1);
  const int i = (int)(f % fI);
  const int64_t r = f / fI;
  const int j = (int)(r % fJ);
  const int k = (int)(r / fJ);
  double s = 0.0;
  const int li = i - (dir == 0), lj = j - (dir == 1), lk = k - (dir == 2);
  if (li >= 0 && lj >= 0 && lk >= 0) s += cell_volume(g, li, lj, lk);
  if (i < g.IM && j < g.JM && k < g.KM) s += cell_volume(g, i, j, k);
  const double vd = 0.5 * s;
  return ((double)face[4 * f] * vp) / vd;
}

// ---------------------------------------------------------------------------
// Device-side input preparation.
// ---------------------------------------------------------------------------
// per-block min/max of node coordinates: out[6*b .. 6*b+5] = (min xyz, max xyz)
static __global__ __launch_bounds__(kBlock) void k_bbox_partial(int64_t nnode, const double *__restrict__ coor,
                                                         double *__restrict__ out) {
  __shared__ double sh[6][kBlock];
  double lo[3] = {1.7976931348623157e308, 1.7976931348623157e308, 1.7976931348623157e308};
  double hi[3] = {-1.7976931348623157e308, -1.7976931348623157e308, -1.7976931348623157e308};
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nnode; q += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      double x = coor[3 * q + a];
      lo[a] = x < lo[a] ? x : lo[a];
      hi[a] = x > hi[a] ? x : hi[a];
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    sh[a][threadIdx.x] = lo[a];
    sh[3 + a][threadIdx.x] = hi[a];
  }
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        double o = sh[a][threadIdx.x + s];
        sh[a][threadIdx.x] = o < sh[a][threadIdx.x] ? o : sh[a][threadIdx.x];
        double h = sh[3 + a][threadIdx.x + s];
        sh[3 + a][threadIdx.x] = h > sh[3 + a][threadIdx.x] ? h : sh[3 + a][threadIdx.x];
      }
    }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[6 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}

// node-slot ucat (double) -> compact [KM][JM][IM][3] in the working precision
template <typename R>
__global__ __launch_bounds__(kBlock) void k_ucat_compact(int IM, int JM, int KM, const double *__restrict__ in,
                                                         R *__restrict__ out) {
  const int64_t ncell = (int64_t)IM * JM * KM;
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  int i = (int)(c % IM);
  int64_t r = c / IM;
  int j = (int)(r % JM);
  int k = (int)(r / JM);
  const double *u = in + 3 * (((int64_t)k * (JM + 1) + j) * (IM + 1) + i);
  out[3 * c] = (R)u[0];
  out[3 * c + 1] = (R)u[1];
  out[3 * c + 2] = (R)u[2];
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_init_particles(int64_t n, const double *__restrict__ pos_in,
                                                           int64_t pid_base, double *__restrict__ pos,
                                                           R *__restrict__ vel, R *__restrict__ w,
                                                           int32_t *__restrict__ cell, int32_t *__restrict__ status,
                                                           int64_t *__restrict__ pid, R *__restrict__ P) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    pos[3 * p + c] = pos_in[3 * p + c];
    vel[3 * p + c] = (R)0;
    w[3 * p + c] = (R)0;
  }
  cell[p] = -1;
  status[p] = ST_UNINIT;
  pid[p] = pid_base + p;
  P[p] = (R)101325.0;
}

static __global__ __launch_bounds__(kBlock) void k_keep_unlocated(int64_t n, const int32_t *__restrict__ cell,
                                                           int32_t *__restrict__ keep) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) keep[p] = cell[p] < 0 ? 1 : 0;
}

// ---------------------------------------------------------------------------
// Heun (RK2) predictor and corrector (no reference counterpart; the
// reference advects with forward Euler, ParticleMotion.c:19-95).
//   predictor: x* = x + u dt            (particles LOST at step start skip)
//   corrector: x1 = x + (u + u*) (dt/2) (particles located at x*)
// ---------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(kBlock) void k_rk2_predict(int64_t n, double *__restrict__ pos, const R *__restrict__ vel,
                                                        const int32_t *__restrict__ status, double *__restrict__ pos0,
                                                        R *__restrict__ vel0, double dt) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const bool lost = status[p] == ST_LOST;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double x = pos[3 * p + c];
    R u = vel[3 * p + c];
    pos0[3 * p + c] = x;
    vel0[3 * p + c] = u;
    if (!lost) pos[3 * p + c] = x + (double)u * dt;
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_rk2_correct(int64_t n, double *__restrict__ pos, const R *__restrict__ vel,
                                                        int32_t *__restrict__ status, const double *__restrict__ pos0,
                                                        const R *__restrict__ vel0, double h) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  if (status[p] != ST_LOCATED) return;
#pragma unroll
  for (int c = 0; c < 3; ++c)
    pos[3 * p + c] = pos0[3 * p + c] + ((double)vel0[3 * p + c] + (double)vel[3 * p + c]) * h;
  status[p] = ST_NEEDS;
}

}  // namespace picgpu
