// emd_comm.hip -- serial periodic-image exchange (CommSerial on one GPU).
//
// exchange       : wrap local positions back into the box once per dimension
// exchange_halo  : every ghost of the six phases (+x,-x,+y,-y,+z,-z faces)
//                  from one pass over the local atoms, in phase and ascending
//                  source order; every ghost also records its owning local
//                  atom ("root") and its periodic shift
// update_halo    : one gather kernel over all ghosts: x_g = x_root + shift,
//                  one addition per shifted dimension (the same single
//                  rounding the phase-by-phase copy performs)
// update_force   : phases 5..0, f[pack] += f[ghost] (targets unique per phase)
#include "emd_internal.hpp"

// CommSerial::TagExchangeSelf, src/comm_types/comm_serial.h:95-108
__global__ void k_wrap(double *__restrict__ x, int n, double lx, double ly, double lz) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double L[3] = {lx, ly, lz};
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const double xd = x[3 * (size_t)i + d];
    double r = xd;
    if (xd > L[d]) r -= L[d];
    if (xd < 0) r += L[d];
    x[3 * (size_t)i + d] = r;
  }
}

extern "C" emd_status emd_comm_exchange(emd_ctx *ctx, emd_system *s) {
  if (!ctx || !s) return EMD_ERR_ARG;
  if (s->n_local <= 0) return EMD_OK;
  EMD_LAUNCH(ctx, "comm_exchange", k_wrap, emd_blocks(s->n_local, 256), 256, 0, s->x, s->n_local,
             s->domain[0], s->domain[1], s->domain[2]);
  return EMD_OK;
}

// CommSerial::exchange_halo (comm_serial.h:112-181) in one pass over the
// local atoms.  Phase +d takes every atom and every ghost of an earlier
// dimension with x_d >= hi_d - depth and shifts it by -L_d, phase -d those
// with x_d <= lo_d + depth (by +L_d); the -d phase does not take the +d
// phase's ghosts.  A ghost keeps its owner's coordinate in every dimension
// not yet shifted, so an atom's six face tests decide all of its ghosts: it
// has the ghost (sx, sy, sz), s_d in {0 none, 1 -L_d, 2 +L_d}, exactly if
// its test for every non-zero s_d holds.  Ghosts are ordered by phase, within
// a phase by ascending source index, and the sources of a phase are the
// locals followed by the earlier phases' ghosts; that order is the list
// number q = sx + 3 sy + 9 sz (1..26), then the owner's index.  So 26 counts
// per block of atoms, one exclusive scan of them and one emit pass give the
// halo, with one message to the host (the six phase counts), where one scan
// per phase needed six rounds of kernels and six host waits.  Bound: launch
// and wait latency up to ~100k atoms, then two reads of the positions.
//   k_halo_one     up to HALO_ONE_MAX local atoms: all of it in one workgroup
//   k_halo_count, k_halo_offsets, k_halo_emit   larger systems
// Capacities (system arrays, pack lists, root/image tables) are compared with
// the counts before anything is written: a halo that does not fit is counted
// only, the host grows and runs it again.
constexpr int HALO_LISTS = 27;  // list 0 (the atom itself) unused

struct halo_args {
  double *x, *vel, *q;
  int *type, *id;
  int *pack[6], *root, *image;
  double hi_thr[3], lo_thr[3], L[3];
  int cap_pack[6];
  int n_local, n_max, root_cap;
  emd_mail mail;  // payload: ghosts per phase [6], 1 if all fit
};

// first list of each phase (phase of list q: the last p with first <= q)
__device__ __forceinline__ constexpr int halo_first_list(int p) {
  return p == 0 ? 1 : p == 1 ? 2 : p == 2 ? 3 : p == 3 ? 6 : p == 4 ? 9 : p == 5 ? 18 : 27;
}
__device__ __forceinline__ constexpr int halo_phase_of(int q) {
  return q < 2 ? 0 : q < 3 ? 1 : q < 6 ? 2 : q < 9 ? 3 : q < 18 ? 4 : 5;
}
// the list of the ghost that list q's ghost is an image of (0: the atom)
__device__ __forceinline__ constexpr int halo_parent(int q) {
  return q >= 9 ? q % 9 : q >= 3 ? q % 3 : 0;
}

// the six face tests of atom i: bits 2d (x_d >= hi - depth) and 2d + 1
__device__ __forceinline__ unsigned halo_flags(const halo_args &a, int i) {
  unsigned fl = 0;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const double xd = a.x[3 * (size_t)i + d];
    if (xd >= a.hi_thr[d]) fl |= 1u << (2 * d);
    if (xd <= a.lo_thr[d]) fl |= 2u << (2 * d);
  }
  return fl;
}

// the wavefront's atoms in list `lane` (lanes 1..26; 0 in other lanes):
// the AND of the face-test ballots that the list asks for
__device__ __forceinline__ unsigned long long halo_lane_mask(unsigned fl) {
  unsigned long long m[6];
#pragma unroll
  for (int k = 0; k < 6; k++) m[k] = __ballot((fl >> k) & 1u);
  const int q = __lane_id();
  if (q < 1 || q >= HALO_LISTS) return 0ull;
  unsigned long long r = ~0ull;
  const int s[3] = {q % 3, (q / 3) % 3, q / 9};
#pragma unroll
  for (int d = 0; d < 3; d++) r &= s[d] == 0 ? ~0ull : (s[d] == 1 ? m[2 * d] : m[2 * d + 1]);
  return r;
}

// value of another lane with a uniform lane number
__device__ __forceinline__ int halo_lane_int(int v, int lane) {
  return __builtin_amdgcn_readlane(v, lane);
}
__device__ __forceinline__ unsigned long long halo_lane_u64(unsigned long long v, int lane) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), lane);
  return ((unsigned long long)hi << 32) | lo;
}

// the ghosts of the wavefront's 64 atoms (atom i in this lane): `mask` and
// `pos` are list lane's members and the ghost index of its first one,
// phase0[p] the first ghost index of phase p
__device__ __forceinline__ void halo_emit_wave(const halo_args &a, int i, unsigned long long mask,
                                               int pos, const int *phase0) {
  if (__ballot(mask != 0ull) == 0ull) return;  // no atom of the wavefront near a face
  const unsigned long long lt = emd_lanemask_lt();
  const int lane = __lane_id();
  double xi[3], vi[3], qi = 0;
  int ti = 0, di = 0;
  bool loaded = false;
  int mine[HALO_LISTS];  // this atom's ghost index in each list
#pragma unroll
  for (int q = 1; q < HALO_LISTS; q++) {
    const unsigned long long m = halo_lane_u64(mask, q);
    mine[q] = 0;
    if (m == 0ull) continue;
    const int gi = halo_lane_int(pos, q) + __popcll(m & lt);
    mine[q] = gi;
    if ((m >> lane) & 1ull) {
      if (!loaded) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
          xi[d] = a.x[3 * (size_t)i + d];
          vi[d] = a.vel[3 * (size_t)i + d];
        }
        qi = a.q[i];
        ti = a.type[i];
        di = a.id[i];
        loaded = true;
      }
      const int ph = halo_phase_of(q), par = halo_parent(q);
      const int s[3] = {q % 3, (q / 3) % 3, q / 9};
      a.pack[ph][gi - phase0[ph]] = par == 0 ? i : a.n_local + mine[par];
      a.root[gi] = i;
      a.image[gi] = s[0] | (s[1] << 2) | (s[2] << 4);
      const size_t g = (size_t)a.n_local + gi;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        a.x[3 * g + d] = s[d] == 0 ? xi[d] : xi[d] + (s[d] == 1 ? -a.L[d] : a.L[d]);
        a.vel[3 * g + d] = vi[d];
      }
      a.q[g] = qi;
      a.id[g] = di;
      a.type[g] = ti;
    }
  }
}

// list sizes (tot, lane q of one wavefront) -> first ghost index of every
// list (returned, same lane), phase counts and whether they fit; lane 0 posts
// them to the host
__device__ __forceinline__ int halo_bases(const halo_args &a, int tot, int *s_phase0, int *s_fits,
                                          int post) {
  const int lane = __lane_id();
  const int inc = emd_wave_incl_scan(tot);
  const int base = inc - tot;
  int fits = 1, num[6];
#pragma unroll
  for (int p = 0; p < 6; p++) {
    const int b0 = halo_lane_int(base, halo_first_list(p));
    const int b1 = halo_lane_int(base, halo_first_list(p + 1));  // lane 27: the total
    num[p] = b1 - b0;
    if (lane == 0) s_phase0[p] = b0;
    if (num[p] > a.cap_pack[p]) fits = 0;
  }
  const int total = halo_lane_int(base, HALO_LISTS);
  if (total > a.root_cap || total > a.n_max - a.n_local) fits = 0;
  if (lane == 0) {
    *s_fits = fits;
    if (post) {
#pragma unroll
      for (int p = 0; p < 6; p++) a.mail.box[EMD_MAIL_DATA + p] = num[p];
      a.mail.box[EMD_MAIL_DATA + 6] = fits;
      emd_mail_post(a.mail);
    }
  }
  return base;
}

constexpr int HALO_ONE_THREADS = 1024;
// local atoms in one workgroup: a whole call takes 14 / 20 / 30 us there with
// 864 / 2048 / 4000 atoms of an LJ melt and 20 / 20 / 19 us with the three
// kernels (host wait included, early counts; 60 / 68 / 76 us with one pass per phase, and
// 194 us from 16 384 atoms on where the three kernels take 19-22)
constexpr int HALO_ONE_MAX = 2048;
constexpr int HALO_ONE_WAVES = HALO_ONE_THREADS / EMD_WAVE;
constexpr int HALO_ONE_GROUPS = HALO_ONE_MAX / EMD_WAVE;  // 64-atom groups, in index order
static_assert(HALO_ONE_GROUPS <= EMD_WAVE, "one wavefront scans a list's group counts");

__global__ void __launch_bounds__(HALO_ONE_THREADS) k_halo_one(halo_args a) {
  __shared__ int s_cnt[HALO_LISTS][HALO_ONE_GROUPS + 1];  // + 1: lanes are lists in pass 1
  __shared__ int s_base[EMD_WAVE], s_phase0[6], s_fits;
  const int wid = threadIdx.x / EMD_WAVE, lane = __lane_id();
  const int n = a.n_local, ng = (n + EMD_WAVE - 1) / EMD_WAVE;
  for (int k = wid; k < ng; k += HALO_ONE_WAVES) {
    const int i = k * EMD_WAVE + lane;
    const unsigned long long m = halo_lane_mask(i < n ? halo_flags(a, i) : 0u);
    if (lane < HALO_LISTS) s_cnt[lane][k] = __popcll(m);
  }
  __syncthreads();
  for (int q = 1 + wid; q < HALO_LISTS; q += HALO_ONE_WAVES) {
    const int c = lane < ng ? s_cnt[q][lane] : 0;
    const int inc = emd_wave_incl_scan(c);
    if (lane < ng) s_cnt[q][lane] = inc - c;
    if (lane == EMD_WAVE - 1) s_base[q] = inc;
  }
  __syncthreads();
  if (wid == 0) {
    const int tot = lane >= 1 && lane < HALO_LISTS ? s_base[lane] : 0;
    s_base[lane] = halo_bases(a, tot, s_phase0, &s_fits, 1);
  }
  __syncthreads();
  if (!s_fits) return;
  for (int k = wid; k < ng; k += HALO_ONE_WAVES) {
    const int i = k * EMD_WAVE + lane;
    const unsigned long long m = halo_lane_mask(i < n ? halo_flags(a, i) : 0u);
    const int pos = lane < HALO_LISTS ? s_base[lane] + s_cnt[lane][k] : 0;
    halo_emit_wave(a, i, m, pos, s_phase0);
  }
}

constexpr int HALO_THREADS = 256;
constexpr int HALO_WAVES = HALO_THREADS / EMD_WAVE;
constexpr int HALO_ITEMS = 4;                                // 64-atom groups per wavefront
constexpr int HALO_GROUPS = HALO_WAVES * HALO_ITEMS;         // groups per block
constexpr int HALO_TILE = HALO_GROUPS * EMD_WAVE;            // atoms per block

// list sizes of each block of HALO_TILE atoms: cnt[q * nb + block]
__global__ void __launch_bounds__(HALO_THREADS) k_halo_count(halo_args a, int nb,
                                                             int *__restrict__ cnt) {
  __shared__ int s_w[HALO_WAVES][HALO_LISTS];
  const int wid = threadIdx.x / EMD_WAVE, lane = __lane_id();
  int c = 0;
#pragma unroll
  for (int k = 0; k < HALO_ITEMS; k++) {
    const int i = (blockIdx.x * HALO_GROUPS + k * HALO_WAVES + wid) * EMD_WAVE + lane;
    c += __popcll(halo_lane_mask(i < a.n_local ? halo_flags(a, i) : 0u));
  }
  if (lane < HALO_LISTS) s_w[wid][lane] = c;
  __syncthreads();
  if (threadIdx.x >= 1 && threadIdx.x < HALO_LISTS) {
    int t = 0;
#pragma unroll
    for (int w = 0; w < HALO_WAVES; w++) t += s_w[w][threadIdx.x];
    cnt[(size_t)threadIdx.x * nb + blockIdx.x] = t;
  }
}

// one workgroup: each list's block counts scanned in place by one wavefront,
// then the lists' first ghost indices into out[0..26], the phases' into
// out[32..37], out[38] = all fit
constexpr int HALO_OUT = 40;
__global__ void __launch_bounds__(1024) k_halo_offsets(halo_args a, int nb, int *__restrict__ cnt,
                                                       int *__restrict__ out) {
  __shared__ int s_tot[EMD_WAVE], s_phase0[6], s_fits;
  const int wid = threadIdx.x / EMD_WAVE, lane = __lane_id();
  for (int q = 1 + wid; q < HALO_LISTS; q += 1024 / EMD_WAVE) {
    int *c = cnt + (size_t)q * nb;
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += 4 * EMD_WAVE) {
      int v[4], s = 0;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int b = b0 + 4 * lane + k;
        v[k] = b < nb ? c[b] : 0;
        s += v[k];
      }
      const int inc = emd_wave_incl_scan(s);
      int run = carry + inc - s;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int b = b0 + 4 * lane + k;
        if (b < nb) c[b] = run;
        run += v[k];
      }
      carry += halo_lane_int(inc, EMD_WAVE - 1);
    }
    if (lane == 0) s_tot[q] = carry;
  }
  __syncthreads();
  if (wid != 0) return;
  const int tot = lane >= 1 && lane < HALO_LISTS ? s_tot[lane] : 0;
  const int base = halo_bases(a, tot, s_phase0, &s_fits, 1);
  if (lane < HALO_LISTS) out[lane] = base;
  if (lane == 0) {
    for (int p = 0; p < 6; p++) out[32 + p] = s_phase0[p];
    out[38] = s_fits;
  }
}

__global__ void __launch_bounds__(HALO_THREADS) k_halo_emit(halo_args a, int nb,
                                                            const int *__restrict__ cnt,
                                                            const int *__restrict__ out) {
  __shared__ int s_w[HALO_GROUPS][HALO_LISTS];
  if (!out[38]) return;
  const int wid = threadIdx.x / EMD_WAVE, lane = __lane_id();
  unsigned long long m[HALO_ITEMS];
#pragma unroll
  for (int k = 0; k < HALO_ITEMS; k++) {
    const int i = (blockIdx.x * HALO_GROUPS + k * HALO_WAVES + wid) * EMD_WAVE + lane;
    m[k] = halo_lane_mask(i < a.n_local ? halo_flags(a, i) : 0u);
    if (lane < HALO_LISTS) s_w[k * HALO_WAVES + wid][lane] = __popcll(m[k]);
  }
  __syncthreads();
  const bool ql = lane >= 1 && lane < HALO_LISTS;
  int pos = ql ? out[lane] + cnt[(size_t)lane * nb + blockIdx.x] : 0, next = 0;
#pragma unroll
  for (int k = 0; k < HALO_ITEMS; k++) {
    const int mygroup = k * HALO_WAVES + wid;
    for (; next < mygroup; next++) pos += ql ? s_w[next][lane] : 0;
    const int i = mygroup * EMD_WAVE + blockIdx.x * HALO_TILE + lane;
    halo_emit_wave(a, i, m[k], pos, out + 32);
  }
}

extern "C" emd_status emd_comm_exchange_halo(emd_ctx *ctx, emd_system *s, double comm_depth,
                                             emd_halo *h) {
  if (!ctx || !s || !h) return EMD_ERR_ARG;
  const int n = s->n_local;
  if (n <= 0) {
    for (int p = 0; p < 6; p++) h->num_ghost[p] = 0;
    s->n_ghost = h->n_ghost = 0;
    return EMD_OK;
  }
  // the first attempt may only count; the second has room for those counts
  for (int attempt = 0; attempt < 2; attempt++) {
    halo_args a;
    a.x = s->x; a.vel = s->v; a.q = s->q; a.type = s->type; a.id = s->id;
    a.root = h->root;
    a.image = h->image;
    for (int p = 0; p < 6; p++) {
      a.pack[p] = h->pack[p];
      a.cap_pack[p] = h->pack[p] ? h->cap[p] : 0;
    }
    for (int d = 0; d < 3; d++) {
      a.hi_thr[d] = s->hi[d] - comm_depth;
      a.lo_thr[d] = s->lo[d] + comm_depth;
      a.L[d] = s->domain[d];
    }
    a.n_local = n;
    a.n_max = s->n_max;
    a.root_cap = (h->root && h->image) ? h->root_cap : 0;
    a.mail = emd_mail_next(ctx);
    if (ctx->halo_one && n <= HALO_ONE_MAX) {
      EMD_LAUNCH(ctx, "comm_exchange_halo", k_halo_one, 1, HALO_ONE_THREADS, 0, a);
    } else {
      const int nb = emd_blocks(n, HALO_TILE);
      EMD_TRY(emd_ensure(ctx, &ctx->d_tmp2, &ctx->tmp2_cap,
                         ((size_t)HALO_LISTS * nb + HALO_OUT) * sizeof(int)));
      int *out = (int *)ctx->d_tmp2, *cnt = out + HALO_OUT;
      EMD_LAUNCH(ctx, "comm_exchange_halo", k_halo_count, nb, HALO_THREADS, 0, a, nb, cnt);
      EMD_LAUNCH(ctx, "comm_exchange_halo", k_halo_offsets, 1, 1024, 0, a, nb, cnt, out);
      EMD_LAUNCH(ctx, "comm_exchange_halo", k_halo_emit, nb, HALO_THREADS, 0, a, nb, cnt, out);
    }
    const int *got = nullptr;
    EMD_TRY(emd_count_wait(ctx, a.mail, &got));
    int num[6], total = 0;
    for (int p = 0; p < 6; p++) total += num[p] = got[p];
    if (got[6]) {
      for (int p = 0; p < 6; p++) h->num_ghost[p] = num[p];
      s->n_ghost = h->n_ghost = total;
      return EMD_OK;
    }
    if ((long)n + total > s->n_max) {
      const long want = (long)n + total;
      EMD_TRY(emd_system_grow(ctx, s, (int)(want + want / 10 + 64)));
    }
    for (int p = 0; p < 6; p++) EMD_TRY(emd_ensure_int(ctx, &h->pack[p], &h->cap[p], num[p]));
    // root and image grow together and share root_cap
    int rcap = h->root ? h->root_cap : 0, icap = h->image ? h->root_cap : 0;
    EMD_TRY(emd_grow_keep_int(ctx, &h->root, &rcap, total, 0));
    EMD_TRY(emd_grow_keep_int(ctx, &h->image, &icap, total, 0));
    h->root_cap = rcap < icap ? rcap : icap;
  }
  return emd_set_error(ctx, EMD_ERR_STATE, "emd_comm_exchange_halo: capacities did not settle");
}

// CommSerial::TagHaloUpdateSelf (comm_serial.h:184-197) for all six phases at
// once, positions only: ghost velocities/charges/ids are copies made at
// exchange_halo time and no kernel reads them afterwards
__global__ void k_halo_update(double *__restrict__ x, const int *__restrict__ root,
                              const int *__restrict__ image, int n_local, int n_ghost, double lx,
                              double ly, double lz) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_ghost) return;
  emd_halo_update_at(g, x, root, image, n_local, lx, ly, lz);
}

extern "C" emd_status emd_comm_update_halo(emd_ctx *ctx, emd_system *s, const emd_halo *h) {
  if (!ctx || !s || !h) return EMD_ERR_ARG;
  if (h->n_ghost <= 0) return EMD_OK;
  EMD_LAUNCH(ctx, "comm_update_halo", k_halo_update, emd_blocks(h->n_ghost, 256), 256, 0, s->x,
             h->root, h->image, s->n_local, h->n_ghost, s->domain[0], s->domain[1],
             s->domain[2]);
  return EMD_OK;
}

// CommSerial::TagHaloForceSelf, comm_serial.h:200-213, for the ghosts off ..
// off + n0 + n1 - 1 of both phases of a dimension, the first n0 owned by pack0
// (or, n1 = 0, of one phase).  Neither phase's owners are among the other's
// ghosts, and where no atom owns a ghost in each (emd_comm_update_force's rule)
// an address gets one addition per launch: the sequential fold's result.
// (Atomic for a halo put together by the caller that has such atoms all the
// same.)  Bound by the launch, so three of them where one per phase took six
// (86 000 atoms: 20 us a step).
template <class T>
__global__ void k_halo_fold(T *__restrict__ f, const int *__restrict__ pack0, int n0,
                            const int *__restrict__ pack1, int n1, int off) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 3 * (n0 + n1)) return;
  const int ii = t / 3, d = t - 3 * ii;
  const int i = ii < n0 ? pack0[ii] : pack1[ii - n0];
  atomicAdd(&f[3 * (size_t)i + d], f[3 * (size_t)off + t]);
}

// all six phases in one launch of one workgroup (emd_fold_phases_one): per
// atom the same additions in the same order as the launches per dimension
template <class T>
__global__ void __launch_bounds__(FOLD_ONE_THREADS)
k_halo_fold_one(T *__restrict__ f, fold_phases ph) {
  emd_fold_phases_one<T, FOLD_ONE_THREADS>(f, ph);
}

long emd_fold_phases_of(const emd_system *s, const emd_halo *h, fold_phases &ph) {
  long total = 0;
  for (int p = 0; p < 6; p++) {
    ph.pack[p] = h->pack[p];
    ph.num[p] = h->num_ghost[p] > 0 ? h->num_ghost[p] : 0;
    ph.off[p] = p == 0 ? s->n_local : ph.off[p - 1] + h->num_ghost[p - 1];
    total += ph.num[p];
  }
  return total;
}

extern "C" emd_status emd_comm_update_force(emd_ctx *ctx, emd_system *s, const emd_halo *h,
                                            int precision) {
  if (!ctx || !s || !h) return EMD_ERR_ARG;
  fold_phases ph;
  const long total = emd_fold_phases_of(s, h, ph);
  if (total == 0) return EMD_OK;
  if (total <= (precision == EMD_MIXED ? FOLD_ONE_MAX_F32 : FOLD_ONE_MAX_F64) && ctx->fold_one) {
    if (precision == EMD_MIXED)
      EMD_LAUNCH(ctx, "comm_update_force", k_halo_fold_one<float>, 1, FOLD_ONE_THREADS, 0,
                 s->f32, ph);
    else
      EMD_LAUNCH(ctx, "comm_update_force", k_halo_fold_one<double>, 1, FOLD_ONE_THREADS, 0, s->f,
                 ph);
    return EMD_OK;
  }
  auto fold = [&](int p, int n0, int n1) -> emd_status {
    if (n0 + n1 <= 0) return EMD_OK;
    const int blocks = emd_blocks(3l * (n0 + n1), 256);
    if (precision == EMD_MIXED)
      EMD_LAUNCH(ctx, "comm_update_force", k_halo_fold<float>, blocks, 256, 0, s->f32, ph.pack[p],
                 n0, n1 ? ph.pack[p + 1] : nullptr, n1, ph.off[p]);
    else
      EMD_LAUNCH(ctx, "comm_update_force", k_halo_fold<double>, blocks, 256, 0, s->f, ph.pack[p],
                 n0, n1 ? ph.pack[p + 1] : nullptr, n1, ph.off[p]);
    return EMD_OK;
  };
  // An atom owns a ghost in both phases of a dimension only where the halo is
  // deeper than half the box, hi - depth <= lo + depth; every source then passes
  // at least one of the two face tests, so the phases have at least as many
  // ghosts as there are sources.  Fewer: one launch; else one per phase, in the
  // sequential fold's order.
  for (int p = 4; p >= 0; p -= 2) {
    const int n0 = ph.num[p], n1 = ph.num[p + 1];
    if ((long)n0 + n1 < ph.off[p]) {
      EMD_TRY(fold(p, n0, n1));
    } else {
      EMD_TRY(fold(p + 1, n1, 0));
      EMD_TRY(fold(p, n0, 0));
    }
  }
  return EMD_OK;
}

extern "C" emd_status emd_halo_free(emd_ctx *ctx, emd_halo *h) {
  if (!ctx || !h) return EMD_ERR_ARG;
  hipStreamSynchronize(ctx->stream);
  for (int p = 0; p < 6; p++) {
    if (h->pack[p]) hipFree(h->pack[p]);
    h->pack[p] = nullptr;
    h->cap[p] = 0;
    h->num_ghost[p] = 0;
  }
  if (h->root) hipFree(h->root);
  if (h->image) hipFree(h->image);
  h->root = h->image = nullptr;
  h->root_cap = 0;
  h->n_ghost = 0;
  return EMD_OK;
}
