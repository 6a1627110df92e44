// emd_snap.hip -- linear SNAP forces and energy on the GPU.
//
// The reference (ForceSNAP + SNA) computes, per atom, U_tot, the full Z
// array, and per neighbour dU/dr and dB_k/dr for all 55 components before
// contracting with beta.  Here the same force is evaluated in adjoint form:
// the beta-weighted sum over the three symmetry roles of dB/dr (the three
// half-plane sums of SNA::compute_dbidrj, sna_impl.hpp:329-539) is folded
// into one array Y_J(ma,mb) per atom, so each neighbour needs only
// dU_J/dr contracted with Y_J:
//
//   F_ij = sum_J sum'_{ma,mb} Re( conj(dU_J(ma,mb)/dr_j) Y_J(ma,mb) )
//   Y_J  = sum_{a>=b} c_{abJ} Z_{abJ},  c collects 2 beta_k, 2 beta_k (j+1)/(j1+1)
//          and 2 beta_k (j+1)/(j2+1) for the roles in which (a,b,J) appears
//
// (sum' is the reference's half plane: mb < J/2, plus for even J the middle
// column ma <= J/2 with weight 1/2 on the diagonal).
//
// Kernels (T = double, or float for the mixed path):
//   k_snap_neigh_ui  one wavefront per atom: compacts the in-cutoff neighbours
//                 (FP64 distance test, list order kept) with ballots, writes
//                 each neighbour's Cayley-Klein parameters, switching function
//                 and derivative factors (snap_par) once, and sums sfac*U over
//                 the neighbours with the layer recursion in registers (nine
//                 lanes per neighbour, seven neighbours at a time at twojmax
//                 <= 8); U_tot (285 complex at twojmax 8) written with its
//                 mirror entries.  k_snap_ui_rg: U_tot alone
//   k_snap_yflat  one block per atom: U_tot staged in LDS, Y (155 half-plane
//                 entries at twojmax 8) from a host-built flat stream of
//                 weighted U_a U_b products, two to a slot
//   k_snap_fij_rev  the force as the gradient of sum Re(conj(U) sfac w Y): U
//                 forward in registers (same layout), adjoints backward, two
//                 complex sums per lane, atomic scatter to f_i / f_j
//   k_snap_energy a third of Re(conj(U_tot) Y) per atom, and the repulsion
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <map>
#include <set>
#include <tuple>
#include <vector>

#include "emd_internal.hpp"

namespace {

// Two size classes: twojmax <= 8 (the kernels tuned for SNAP-2k, whose
// twojmax is 8) and twojmax <= 12 (the same kernels with larger tables and
// more registers, four neighbours per wavefront).  Per class J:
constexpr int SNAP_MAXJ = 8;                 // the first class
constexpr int SNAP_JBIG = 12;                // the second class: the largest twojmax
constexpr double SNAP_PI = 3.14159265358979323846;

// U entries sum_j (j+1)^2, half-plane entries sum_j (j+1)(j/2+1), (a,b,J)
// triples and bispectrum components (diagonalstyle 3) up to twojmax J
constexpr int snap_nu(int J) { return J < 0 ? 0 : snap_nu(J - 1) + (J + 1) * (J + 1); }
constexpr int snap_ny(int J) { return J < 0 ? 0 : snap_ny(J - 1) + (J + 1) * (J / 2 + 1); }
constexpr int snap_counts(int J, bool coeff) {
  int n = 0;
  for (int j1 = 0; j1 <= J; j1++)
    for (int j2 = 0; j2 <= j1; j2++)
      for (int j = j1 - j2; j <= (J < j1 + j2 ? J : j1 + j2); j += 2)
        if (!coeff || j >= j1) n++;
  return n;
}
template <int J>
struct snap_dim {
  static constexpr int NU = snap_nu(J);
  static constexpr int NY = snap_ny(J);
};
constexpr int SNAP_MAXT = snap_counts(SNAP_JBIG, false);  // (a,b,J) triples: 343
constexpr int SNAP_MAXC = snap_counts(SNAP_JBIG, true);   // components: 140
constexpr int SNAP_NU_BIG = snap_nu(SNAP_JBIG);
static_assert(snap_nu(8) == 285 && snap_ny(8) == 155 && snap_counts(8, false) == 125 &&
                  snap_counts(8, true) == 55,
              "SNAP table sizes at twojmax 8");

// device tables (filled by emd_snap_create)
struct snap_dev_tables {
  int twojmax;
  int nu, ny;                      // number of U entries / half-plane entries
  int ustart[SNAP_JBIG + 2];       // full layer offsets: ustart[j] + ma*(j+1) + mb
  int ystart[SNAP_JBIG + 2];       // half-plane offsets: ystart[J] + mb*(J+1) + ma
  double rfac0, rmin0, rcut, wj, wself;
  int switchflag;
};

struct etab_entry {
  int j1, j2, j, cgoff;
  double beta;
};

struct stab_entry {
  int a, b, cgoff, tid;
};

template <class T>
struct cplx {
  T r, i;
};

__device__ __forceinline__ void snap_sincos(float a, float &s, float &c) { sincosf(a, &s, &c); }
__device__ __forceinline__ void snap_sincos(double a, double &s, double &c) { sincos(a, &s, &c); }

// ------------------------------------------------------------- switching
template <class T>
__device__ __forceinline__ void sfac_dsfac(const snap_dev_tables &t, T r, T &sfac, T &dsfac) {
  if (t.switchflag == 0) {
    sfac = 1;
    dsfac = 0;
  } else if (r <= (T)t.rmin0) {
    sfac = 1;
    dsfac = 0;
  } else if (r > (T)t.rcut) {
    sfac = 0;
    dsfac = 0;
  } else {
    const T rcutfac = (T)(SNAP_PI / (t.rcut - t.rmin0));
    T cs, sn;
    snap_sincos((r - (T)t.rmin0) * rcutfac, sn, cs);
    sfac = (T)0.5 * (cs + (T)1);
    dsfac = (T)-0.5 * sn * rcutfac;
  }
}

// Per in-cutoff neighbour, computed once by the neighbour compaction: the
// Cayley-Klein parameters a = (z0 - i z)/r0, b = (y - i x)/r0 of rij, the
// switching function and its derivative (times wj), the unit vector and the
// factors of da/dr and db/dr, which are rank one in the unit vector u:
//   da_r = c1 u, da_i = c2 u - r0inv e_z, db_r = c3 u + r0inv e_y,
//   db_i = c4 u - r0inv e_x
// (SNA::compute_uarray / compute_duarray, sna_impl.hpp:640-700, 728-790)
template <class T>
struct alignas(16) snap_par {
  T a_r, a_i, b_r, b_i;
  T sfac, dsfac;
  T u[3];
  T c1, c2, c3, c4;
  T r0inv;
  T pad[2];
};

template <class T>
__device__ __forceinline__ void snap_par_of(const snap_dev_tables &t, double dx, double dy,
                                            double dz, snap_par<T> &p) {
  const T x = (T)dx, y = (T)dy, z = (T)dz;
  const T rsq = x * x + y * y + z * z;
  const T r = sqrt(rsq);
  const T rscale0 = (T)t.rfac0 * (T)SNAP_PI / ((T)t.rcut - (T)t.rmin0);
  const T theta0 = (r - (T)t.rmin0) * rscale0;
  T cs, sn;
  snap_sincos(theta0, sn, cs);
  const T z0 = r * cs / sn;
  const T dz0dr = z0 / r - (r * rscale0) * (rsq + z0 * z0) / rsq;
  const T rinv = (T)1 / r;
  const T r0inv = (T)1 / sqrt(r * r + z0 * z0);
  const T dr0invdr = -(r0inv * r0inv * r0inv) * (r + z0 * dz0dr);
  p.a_r = z0 * r0inv;
  p.a_i = -z * r0inv;
  p.b_r = y * r0inv;
  p.b_i = -x * r0inv;
  T sfac, dsfac;
  sfac_dsfac(t, r, sfac, dsfac);
  p.sfac = sfac * (T)t.wj;
  p.dsfac = dsfac * (T)t.wj;
  p.u[0] = x * rinv;
  p.u[1] = y * rinv;
  p.u[2] = z * rinv;
  p.c1 = dz0dr * r0inv + z0 * dr0invdr;
  p.c2 = -z * dr0invdr;
  p.c3 = y * dr0invdr;
  p.c4 = -x * dr0invdr;
  p.r0inv = r0inv;
  p.pad[0] = p.pad[1] = 0;
}

// the reference's ad-hoc pair repulsion as F/r, force_snap_neigh_impl.h:705-711
__device__ __forceinline__ double snap_fdivr(double dx, double dy, double dz) {
  const double r2 = dx * dx + dy * dy + dz * dz, r4 = r2 * r2;
  return -1.5e6 / (r4 * r4 * r4 * r2);
}

}  // namespace

// ================================================================ kernels
// in-cutoff neighbours of each atom, ForceSNAP::operator() lines 612-656
// (rij = x_j - x_i, test rsq < rcutmax^2); slot k of atom i at i*maxn + k.
// With a force array given (f64 or f32), block i also zeroes its rows
// i, i + n, i + 2n, ... below ntot (deep_copy(f, 0), src/examinimd.cpp:232,
// done here instead of in a launch of its own: the force kernels that add
// into f come after this one).  The slot's neighbour parameters (par, in T) and
// the repulsion F/r (fdv) are written as well.
// (for atom i by one wavefront, in k_snap_neigh_ui; returns the count)
template <class T>
__device__ __forceinline__ int snap_compact(const snap_dev_tables &t, int i, const double *__restrict__ x,
                                            const int *__restrict__ row, const int *__restrict__ num,
                                            const int *__restrict__ entries, int pitch, int n,
                                            double cutsq, int maxn, int *__restrict__ nin,
                                            int *__restrict__ nj, double *__restrict__ nr,
                                            double *__restrict__ f64, float *__restrict__ f32,
                                            int ntot, snap_par<T> *__restrict__ par,
                                            double *__restrict__ fdv) {
#pragma clang fp contract(off)  // the distance test as the reference (the parameters are
                                // computed in functions of their own)
  const int lane = threadIdx.x % 64;
  if (f64 || f32) {
    for (int r = i + n * (lane / 3); r < ntot; r += n * 21) {  // lanes 0..62: 21 rows of 3
      if (lane < 63) {
        if (f64) f64[3 * (size_t)r + lane % 3] = 0.0;
        else f32[3 * (size_t)r + lane % 3] = 0.0f;
      }
    }
  }
  const double x_i = x[3 * (size_t)i], y_i = x[3 * (size_t)i + 1], z_i = x[3 * (size_t)i + 2];
  const int *rp = entries + (row ? (size_t)row[i] : (size_t)i * (size_t)pitch);
  const int cnt = num[i];
  const unsigned long long lt = emd_lanemask_lt();
  int run = 0;
  for (int c0 = 0; c0 < cnt; c0 += 64) {
    const int c = c0 + lane;
    bool keep = false;
    int j = 0;
    double dx = 0, dy = 0, dz = 0;
    if (c < cnt) {
      j = rp[c];
      dx = x[3 * (size_t)j] - x_i;
      dy = x[3 * (size_t)j + 1] - y_i;
      dz = x[3 * (size_t)j + 2] - z_i;
      const double rsq = dx * dx + dy * dy + dz * dz;
      keep = rsq < cutsq;
    }
    const unsigned long long m = __ballot(keep);
    if (keep) {
      const int k = run + __popcll(m & lt);
      if (k < maxn) {
        const size_t o = (size_t)i * maxn + k;
        nj[o] = j;
        nr[3 * o] = dx;
        nr[3 * o + 1] = dy;
        nr[3 * o + 2] = dz;
        snap_par_of<T>(t, dx, dy, dz, par[o]);
        fdv[o] = snap_fdivr(dx, dy, dz);
      }
    }
    run += __popcll(m);
  }
  if (lane == 0) nin[i] = run < maxn ? run : maxn;
  return run < maxn ? run : maxn;
}

// the neighbour parameters in FP64 (and the repulsion F/r) from the compacted
// neighbours, for FP64 U_tot after a compaction that wrote FP32
__global__ void __launch_bounds__(64)
k_snap_par(snap_dev_tables t, const int *__restrict__ nin, const double *__restrict__ nr,
           int maxn, int n, snap_par<double> *__restrict__ par, double *__restrict__ fdv) {
  const int i = blockIdx.x;
  if (i >= n) return;
  for (int k = threadIdx.x; k < nin[i]; k += 64) {
    const size_t o = (size_t)i * maxn + k;
    snap_par_of<double>(t, nr[3 * o], nr[3 * o + 1], nr[3 * o + 2], par[o]);
    fdv[o] = snap_fdivr(nr[3 * o], nr[3 * o + 1], nr[3 * o + 2]);
  }
}

// ordering of LDS traffic among the lanes of one wavefront (no block barrier)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Z_{abJ}(ma,mb) = sum_ma1 cg(ma1,ma2) sum_mb1 cg(mb1,mb2) U_a(ma1,mb1) U_b(ma2,mb2)
// (SNA::compute_zi, sna_impl.hpp:221-274) from U_tot staged in LDS
template <class T>
__device__ __forceinline__ cplx<T> z_entry(const snap_dev_tables &t, const double *__restrict__ cg,
                                           const T *su_r, const T *su_i, int a, int b, int J,
                                           int cgoff, int ma, int mb) {
  cplx<T> z{0, 0};
  const int ma1lo = max(0, (2 * ma - J - b + a) / 2), ma1hi = min(a, (2 * ma - J + b + a) / 2);
  const int mb1lo = max(0, (2 * mb - J - b + a) / 2), mb1hi = min(a, (2 * mb - J + b + a) / 2);
  const int ua = t.ustart[a], ub = t.ustart[b];
  for (int ma1 = ma1lo; ma1 <= ma1hi; ma1++) {
    const int ma2 = (2 * ma - J - (2 * ma1 - a) + b) / 2;
    T s_r = 0, s_i = 0;
    for (int mb1 = mb1lo; mb1 <= mb1hi; mb1++) {
      const int mb2 = (2 * mb - J - (2 * mb1 - a) + b) / 2;
      const T c = (T)cg[cgoff + mb1 * (b + 1) + mb2];
      const T u1r = su_r[ua + ma1 * (a + 1) + mb1], u1i = su_i[ua + ma1 * (a + 1) + mb1];
      const T u2r = su_r[ub + ma2 * (b + 1) + mb2], u2i = su_i[ub + ma2 * (b + 1) + mb2];
      s_r += c * (u1r * u2r - u1i * u2i);
      s_i += c * (u1r * u2i + u1i * u2r);
    }
    const T c = (T)cg[cgoff + ma1 * (b + 1) + ma2];
    z.r += s_r * c;
    z.i += s_i * c;
  }
  return z;
}

// half-plane entry e (0..ny-1) -> (J, ma, mb)
__device__ __forceinline__ void y_entry(const snap_dev_tables &t, int e, int &J, int &ma,
                                        int &mb) {
  J = 0;
  while (J < t.twojmax && e >= t.ystart[J + 1]) J++;
  const int k = e - t.ystart[J];
  mb = k / (J + 1);
  ma = k - mb * (J + 1);
}

// Y of AT atoms per block from a flat stream of products.  Every half-plane
// entry e = (J, ma, mb) is the sum over its (a, b) keys and (ma1, mb1) of
//   w * U_a(ma1, mb1) * U_b(ma2, mb2),  w = coef(a,b,J) cg(ma1,ma2) cg(mb1,mb2)
// (the double sum of SNA::compute_zi, sna_impl.hpp:221-274, weighted as in
// compute_dbidrj's three roles).  The host pairs an entry's products that
// share a U entry (yf_pairs): a slot of the stream is
//   U_c (w_x U_x + w_y U_y),
// three LDS byte offsets (its code), two weights, eight multiply-adds and
// three LDS reads for two products, where one product at a time takes twelve
// and four.  Entries of half-plane weight 0 (the middle columns' ma > mb)
// have no products.  The slots come entry by entry, each entry's list
// padded with zero-weight slots to whole chunks of YF_CHUNK, and thread t gets the
// chunks [t P, (t+1) P) of that sequence, interleaved so that step s of every
// thread is one coalesced load.  Chunk boundaries are the same for every
// lane, so the slot loop carries no branch.  Once per chunk a
// thread whose run of one entry's chunks ends stores the run's sum in LDS;
// each entry adds its runs in thread order (fixed order: deterministic).
// With AT atoms per block (U_tot of each in LDS) every code and weight load
// serves AT atoms.
// Arithmetic (54 % of its issue rate at 16 000 atoms in FP64), LDS reads (65
// %) and the stream from L2 (76 % of the address units, 18 TB/s) bound it
// about equally, so all three had to shrink: one product at a time with the
// middle columns in full took 303 us for 16 000 atoms (FP64, twojmax 8), 24.4
// for 2000 (mixed), 222 / 109 for 1024 atoms at twojmax 12 (FP64 / mixed); this
// takes 222, 18, 137 and 69.
//
// LDS banks: the LDS serves 256 bytes per cycle, so a wavefront's
// ds_read_b64 is served 32 lanes per cycle, and two lanes of one cycle that
// read different 8-byte words at the same bank residue (word index mod 32)
// are served in turn.  (Measured: 5.15 LDS-active cycles per wavefront read
// of an earlier FP32 term order, for which this model gives 5.19.)  A
// ds_read_b128 of 16-byte FP64 pairs measured 8 cycles: its 8-byte halves
// are served like two b64 reads, and a 16-byte stride leaves only 16
// residues.  So FP32 U_tot is stored as (re, im) pairs and FP64 U_tot as an
// array of real parts and one of imaginary parts, each read with b64 loads
// at word residue u mod 32.  U_tot is staged four times,
// copy c at word offset c * stride + shift(c), and the host gives every
// read of every term the copy whose residue no other address of its
// 32-lane group takes (a matching per group; with the shifts 0, 5, 11, 19
// about 4 % of the groups keep one conflict).

// threads per Y block (the stream is split this many ways): 512, at twojmax
// above 8, where one block's LDS fills a CU, 1024
template <int J>
constexpr int yf_threads() { return J <= SNAP_MAXJ ? 512 : 1024; }
constexpr int SF_THREADS = 512;
constexpr int YF_CHUNK = 8;   // slots
constexpr int SF_CHUNK = 16;  // products (the beta adjoint's stream)

template <class T>
struct alignas(2 * sizeof(T)) cpair {
  T r, i;
};

// U_tot copies in the Y kernel's LDS, in 8-byte words: an FP32 pair is one
// word, an FP64 entry a word in the real array and one in the imaginary
// array (IMB bytes further)
template <class T, int J>
struct yf_layout {
  static constexpr bool SOA = sizeof(T) == 8;
  static constexpr int NCOPY = 4;
  static constexpr int MOD = 32;    // bank residues of an 8-byte word
  static constexpr int GROUP = 32;  // lanes served per cycle
  static constexpr int STRIDE = (snap_dim<J>::NU + MOD - 1) / MOD * MOD;
  __host__ __device__ static constexpr int shift(int c) {
    return c == 0 ? 0 : c == 1 ? 5 : c == 2 ? 11 : 19;
  }
  __host__ __device__ static constexpr int base(int c) { return c * STRIDE + shift(c); }
  static constexpr int NUC = base(NCOPY - 1) + snap_dim<J>::NU;  // words the copies span
  // an odd number of 256-byte rows: at a multiple of 512 bytes the compiler
  // joins the real and imaginary (or two atoms') reads into ds_read2st64_b64,
  // which takes twice as long as the two
  static constexpr int NUC_PAD = ((NUC + MOD - 1) / MOD | 1) * MOD;
  static constexpr int IMB = SOA ? NUC_PAD * 8 : 0;            // imaginary array (FP64)
  static constexpr int UBYTES = SOA ? 2 * NUC_PAD * 8 : NUC_PAD * 8;
};

// the byte offsets of a slot's U_tot entries in LDS
struct alignas(8) yf_code {
  unsigned short c, x, y, pad;
};
template <class T, int J>
__device__ __forceinline__ cpair<T> yf_u(const unsigned char *ub, unsigned off) {
  using L = yf_layout<T, J>;
  if constexpr (L::SOA)
    return cpair<T>{*reinterpret_cast<const T *>(ub + off),
                    *reinterpret_cast<const T *>(ub + L::IMB + off)};
  else
    return *reinterpret_cast<const cpair<T> *>(ub + off);
}

// meta[c][t]: the LDS slot of the
// run that ends with thread t's chunk c, or YF_NO_RUN.  A thread's runs are
// the entries its chunk range touches, so there are at most ny + threads - 1.
constexpr unsigned short YF_NO_RUN = 0xFFFFu;
template <int J>
constexpr int yf_maxruns() { return snap_dim<J>::NY + yf_threads<J>(); }
static_assert(yf_layout<double, SNAP_JBIG>::NUC * 8 < 65536 &&
                  yf_layout<float, SNAP_JBIG>::NUC * 8 < 65536,
              "U_tot byte offsets fit 16 bits");

// Place of slot k of (chunk c, thread t) in the stream: a wavefront's slots lie
// together, one step of its lanes in a row, so all loads of a chunk have one
// address and constant offsets.  Codes and FP32 weights take two slots
// per 16-byte load.
__host__ __device__ constexpr size_t yf_place(int P, int c, int k, int t) {
  return ((size_t)(t / 64 * P + c) * YF_CHUNK + k) * 64 + t % 64;
}
__host__ __device__ constexpr size_t yf_place2(size_t place) {  // two slots of a lane together
  return (place / 128 * 64 + place % 64) * 2 + place / 64 % 2;
}

// four slots of the stream in registers
template <class T>
struct yf_regs {
  yf_code c[4];
  cpair<T> w[4];
  __device__ __forceinline__ void load(const yf_code *__restrict__ code,
                                       const cpair<T> *__restrict__ wt, int step, int l) {
    typedef unsigned v4 __attribute__((ext_vector_type(4)));
    const v4 *cp = reinterpret_cast<const v4 *>(code) + ((size_t)step * 2 * 64 + l);
    reinterpret_cast<v4 *>(c)[0] = cp[0];
    reinterpret_cast<v4 *>(c)[1] = cp[64];
    if constexpr (sizeof(T) == 4) {
      const v4 *wp = reinterpret_cast<const v4 *>(wt) + ((size_t)step * 2 * 64 + l);
      reinterpret_cast<v4 *>(w)[0] = wp[0];
      reinterpret_cast<v4 *>(w)[1] = wp[64];
    } else {
      const cpair<T> *wp = wt + ((size_t)step * 4 * 64 + l);
#pragma unroll
      for (int k = 0; k < 4; k++) w[k] = wp[64 * k];
    }
  }
};

template <class T, int J, int AT>
__global__ void __launch_bounds__(yf_threads<J>())
k_snap_yflat(int nu, int ny, int nch, const yf_code *__restrict__ code,
             const cpair<T> *__restrict__ w, const unsigned short *__restrict__ meta,
             const int *__restrict__ rstart, int n, const T *__restrict__ utot_r,
             const T *__restrict__ utot_i, T *__restrict__ y_r, T *__restrict__ y_i) {
  // the copies of U_tot from byte 0 (a static array: its LDS address is
  // known when the kernel is compiled, so a code's offset is the whole LDS
  // address), then the run sums
  using L = yf_layout<T, J>;
  constexpr int NT = yf_threads<J>();
  static_assert(L::UBYTES % sizeof(cpair<T>) == 0, "run sums aligned");
  constexpr int UP = L::UBYTES / sizeof(cpair<T>);  // pairs per atom's U_tot copies
  constexpr int MR = yf_maxruns<J>();
  __shared__ cpair<T> s_yf[AT * (UP + MR)];
  unsigned char *sb = reinterpret_cast<unsigned char *>(s_yf);
  cpair<T> *part = s_yf + AT * UP;
  const int i0 = blockIdx.x * AT;
  if (i0 >= n) return;
  const int l = threadIdx.x % 64;
  const size_t wv = (size_t)(threadIdx.x / 64) * nch * YF_CHUNK * 64;  // the wavefront's slots
  code += wv;
  w += wv;
  yf_regs<T> b0, b1;
  b0.load(code, w, 0, l);  // under way while U_tot is staged
#pragma unroll
  for (int k0 = 0; k0 < snap_dim<J>::NU; k0 += NT) {
    const int k = k0 + (int)threadIdx.x;
    if (k < nu) {
      T vr[AT], vi[AT];
#pragma unroll
      for (int a = 0; a < AT; a++) {
        const size_t i = i0 + a < n ? i0 + a : i0;
        vr[a] = utot_r[i * nu + k];
        vi[a] = utot_i[i * nu + k];
      }
#pragma unroll
      for (int a = 0; a < AT; a++) {
        unsigned char *ub = sb + a * L::UBYTES;
#pragma unroll
        for (int c = 0; c < L::NCOPY; c++) {
          if (L::SOA) {
            reinterpret_cast<T *>(ub)[L::base(c) + k] = vr[a];
            reinterpret_cast<T *>(ub + L::IMB)[L::base(c) + k] = vi[a];
          } else {
            reinterpret_cast<cpair<T> *>(ub)[L::base(c) + k] = cpair<T>{vr[a], vi[a]};
          }
        }
      }
    }
  }
  __syncthreads();
  T ar[AT], ai[AT];
#pragma unroll
  for (int a = 0; a < AT; a++) ar[a] = ai[a] = 0;
  auto add = [&](const yf_regs<T> &b) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
#pragma unroll
      for (int a = 0; a < AT; a++) {
        const unsigned char *ub = sb + a * L::UBYTES;
        const cpair<T> uc = yf_u<T, J>(ub, b.c[k].c), ux = yf_u<T, J>(ub, b.c[k].x),
                       uy = yf_u<T, J>(ub, b.c[k].y);
        const T vr = b.w[k].r * ux.r + b.w[k].i * uy.r;
        const T vi = b.w[k].r * ux.i + b.w[k].i * uy.i;
        ar[a] += uc.r * vr;  // two multiply-adds each, not a sum of products
        ar[a] -= uc.i * vi;
        ai[a] += uc.r * vi;
        ai[a] += uc.i * vr;
      }
    }
  };
  static_assert(YF_CHUNK == 8, "two halves");
#pragma unroll 1
  for (int c = 0; c < nch; c++) {
    // the next half's loads are under way while one half is added up
    b1.load(code, w, 2 * c + 1, l);
    const unsigned short m = meta[(size_t)c * NT + threadIdx.x];
    add(b0);
    b0.load(code, w, c + 1 < nch ? 2 * c + 2 : 0, l);
    add(b1);
    if (m != YF_NO_RUN) {
#pragma unroll
      for (int a = 0; a < AT; a++) {
        part[a * MR + m] = cpair<T>{ar[a], ai[a]};
        ar[a] = 0;
        ai[a] = 0;
      }
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < AT * ny; q += NT) {
    const int a = q / ny, e = q - a * ny;
    if (i0 + a >= n) break;
    T yr = 0, yi = 0;
    for (int r = rstart[e]; r < rstart[e + 1]; r++) {
      yr += part[a * MR + r].r;
      yi += part[a * MR + r].i;
    }
    y_r[(size_t)(i0 + a) * ny + e] = yr;
    y_i[(size_t)(i0 + a) * ny + e] = yi;
  }
}

// the slots' weights for the current coefficients (two products per slot)
__global__ void k_yf_weights(int nslots, const unsigned short *__restrict__ key,
                             const double *__restrict__ cgw, const double *__restrict__ kcoef,
                             double *__restrict__ w64, float *__restrict__ w32) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= 2 * nslots) return;
  const double v = kcoef[key[s]] * cgw[s];
  w64[s] = v;
  w32[2 * yf_place2(s / 2) + s % 2] = (float)v;
}

// ------------------------------------------- register-resident recursion
// A neighbour's layer j fits the J + 1 lanes of its group: lane ma holds the
// entries (ma, mb) of every half-plane column mb = 0..j/2 in registers.
// The kernels carry V rather than U,
//   U_j(ma,mb) = norm_j(ma,mb) V_j(ma,mb),
//   norm_j(ma,mb) = sqrt(ma! (j-ma)! / (mb! (j-mb)!)),
// because the factors sqrt((j-ma)/(j-mb)) and sqrt(ma/(j-mb)) of the
// recursion of SNA::compute_uarray (sna_impl.hpp:663-695) cancel in V:
//   V_j(ma,mb)  = conj(a) V_{j-1}(ma,mb)   - conj(b) V_{j-1}(ma-1,mb)
// and, its mirror image (the norm is the same at (j-ma, j-mb)),
//   V_j(ma,j/2) = b V_{j-1}(ma,j/2-1) + a V_{j-1}(ma-1,j/2-1)
// for the middle column of an even layer, whose first form would need
// columns outside the half plane.  So an entry takes 8 multiply-adds (12 and
// a table record with the factors), V(ma-1) comes from the lane below by a
// DPP shift and nothing is permuted.  V is exactly 0 where the entry does
// not exist (ma > j): the borders need no test, and what the lane shifts
// carry over a group's edge meets only such zeros.  The norm is applied once
// per atom, to the sums over the neighbours or to Y.
// FP64 (FP32) arithmetic bounds all three kernels (75 % of its issue rate in
// the force kernel and W, 70 % in U_tot).  Against U with its factors, FP64, 16 000 atoms of 26
// neighbours, twojmax 8: U_tot 174 -> 82 us, force 232 -> 144 us; W of 64 BCC
// configurations of 128 to 1024 atoms 820 -> 262 us; mixed, 2000 atoms:
// 24.4 -> 15.9 and 28.6 -> 14.9 us.  Twojmax 12,
// 1024 atoms, against one neighbour per wavefront with the layers in LDS:
// U_tot 140 -> 27 us (FP64), force 141 -> 28 us (mixed).
// Groups of 9 lanes, seven per wavefront (one lane idle), for twojmax <= 8;
// of 13 lanes, four per wavefront, up to 12.
__host__ __device__ constexpr int rg_slot0(int j) { return j <= 0 ? 0 : j + (j - 1) * (j - 1) / 4; }
template <int J>
struct rg {
  static constexpr int W = J + 1;                // lanes per neighbour (ma = 0..J)
  static constexpr int NB = 64 / W;              // neighbours per wavefront
  static constexpr int COLS = J / 2 + 1;         // columns of the top layer
  static constexpr int SLOTS = rg_slot0(J + 1);  // (layer, column) pairs of layers 0..J
};
// first column slot of layer j: sum over layers j' < j of (j'/2 + 1) columns
static_assert(rg_slot0(1) == 1 && rg_slot0(2) == 2 && rg_slot0(3) == 4 && rg_slot0(8) == 20 &&
                  rg<8>::SLOTS == 25 && rg<12>::SLOTS == 49,
              "column slots");

template <class T>
struct alignas(2 * sizeof(T)) rg_rec {
  T yr, yi;  // weighted Y of (j, ma, mb), in V's norm
};

// value of lane l - 1 (0 in lane 0): DPP wavefront shift right by one
// (bound_ctrl: the lane without a source reads 0)
__device__ __forceinline__ float lane_below(float v) {
  return __builtin_bit_cast(float,
                            __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_below(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x138, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x138, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// value of lane l + 1 (0 in lane 63): DPP wavefront shift left by one
__device__ __forceinline__ float lane_above(float v) {
  return __builtin_bit_cast(float,
                            __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_above(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x130, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x130, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Per (column slot s, lane ma), k = s * W + ma, built on the host once:
//   norm norm_j(ma, mb)
//   ey   the half-plane index of Y (or -1: the entry does not exist), wgt its
//        half-plane weight
//   uo   the U_tot index of (ma, mb), um that of the mirror (j-ma, j-mb) off
//        the middle column (or -1), neg its sign (-1)^(ma+mb) and diag for
//        ma == mb (wself)
struct rg_map {
  double norm;
  int ey, uo, um;
  unsigned char wq, neg, diag, pad;  // wgt = wq / 2
};

// body(j) for j = FIRST .. LAST (up or down), each j a constant of its own:
// the register arrays are indexed by it, and the unroller gives up on a loop
// over the layers at twojmax 12
template <int FIRST, int LAST, class F>
__device__ __forceinline__ void rg_layers(const F &body) {
  body(std::integral_constant<int, FIRST>{});
  if constexpr (FIRST < LAST) rg_layers<FIRST + 1, LAST>(body);
  else if constexpr (FIRST > LAST) rg_layers<FIRST - 1, LAST>(body);
}

// layer j from layer j-1, in place
template <int j, class T, int COLS>
__device__ __forceinline__ void rg_layer(T a_r, T a_i, T b_r, T b_i, T (&c)[COLS][2]) {
  T q[COLS][2];
#pragma unroll
  for (int mb = 0; mb <= (j - 1) / 2; mb++) {
    q[mb][0] = lane_below(c[mb][0]);
    q[mb][1] = lane_below(c[mb][1]);
  }
  if constexpr ((j & 1) == 0) {
    constexpr int m = j / 2 - 1;
    c[m + 1][0] = b_r * c[m][0] - b_i * c[m][1] + a_r * q[m][0] - a_i * q[m][1];
    c[m + 1][1] = b_r * c[m][1] + b_i * c[m][0] + a_r * q[m][1] + a_i * q[m][0];
  }
#pragma unroll
  for (int mb = 0; 2 * mb < j; mb++) {
    const T p0 = c[mb][0], p1 = c[mb][1];
    c[mb][0] = a_r * p0 + a_i * p1 - b_r * q[mb][0] - b_i * q[mb][1];
    c[mb][1] = a_r * p1 - a_i * p0 - b_r * q[mb][1] + b_i * q[mb][0];
  }
}

// Sums over the neighbours (NB at a time) of atom i of sfac * V for the
// lane's entries (ma, mb) of every column of every layer (SNA::compute_ui,
// sna_impl.hpp:152-190), added to acc[column slot].  The recursion is linear:
// it starts from sfac.
template <class T, int J>
__device__ __forceinline__ void rg_u_sums(const snap_dev_tables &t,
                                          const snap_par<T> *__restrict__ par, int i, int maxn,
                                          int cnt, int g, int ma, T (&acc)[rg<J>::SLOTS][2]) {
  using R = rg<J>;
  for (int base = 0; base < cnt; base += R::NB) {
    const int jj = base + g;
    const bool act = g < R::NB && jj < cnt;
    const size_t o = (size_t)i * maxn + (act ? jj : base);
    const T a_r = par[o].a_r, a_i = par[o].a_i, b_r = par[o].b_r, b_i = par[o].b_i;
    T c[R::COLS][2];
#pragma unroll
    for (int mb = 0; mb < R::COLS; mb++) c[mb][0] = c[mb][1] = 0;
    c[0][0] = act && ma == 0 ? par[o].sfac : (T)0;  // an idle group adds nothing
    acc[0][0] += c[0][0];
    rg_layers<1, J>([&](auto jc) {
      constexpr int j = jc;
      if (j > t.twojmax) return;
      rg_layer<j>(a_r, a_i, b_r, b_i, c);
#pragma unroll
      for (int mb = 0; mb <= j / 2; mb++) {
        acc[rg_slot0(j) + mb][0] += c[mb][0];
        acc[rg_slot0(j) + mb][1] += c[mb][1];
      }
    });
  }
}

// acc summed over the groups of the wavefront in group order (in TA) and
// handed to out(column slot * W + ma, sum_r, sum_i), one entry per lane at a
// time.  Through LDS, RG_CHUNK slots at a time: a row of the buffer holds one
// value of every lane, and the pitch of 64 + W keeps the W-wide pieces that
// one read takes from successive rows in successive banks.
template <int J>
struct rg_sum {
  static constexpr int CH = 63 / rg<J>::W;      // column slots at a time
  static constexpr int PITCH = 64 + rg<J>::W;   // of a row of the buffer
  static constexpr int BUF = 2 * CH * PITCH;    // values of T
};
template <class TA, int J, class T, class F>
__device__ __forceinline__ void rg_group_sum(const T (&acc)[rg<J>::SLOTS][2], int l, T *buf,
                                             const F &out) {
  using R = rg<J>;
  using S = rg_sum<J>;
#pragma unroll
  for (int s0 = 0; s0 < R::SLOTS; s0 += S::CH) {
    const int ns = R::SLOTS - s0 < S::CH ? R::SLOTS - s0 : S::CH;
    wave_sync();  // the previous slots have been read
#pragma unroll
    for (int s = 0; s < ns; s++) {
      buf[s * S::PITCH + l] = acc[s0 + s][0];
      buf[(S::CH + s) * S::PITCH + l] = acc[s0 + s][1];
    }
    wave_sync();
    if (l < ns * R::W) {
      const T *b = buf + (l / R::W) * S::PITCH + l % R::W;
      TA vr = 0, vi = 0;
#pragma unroll
      for (int g = 0; g < R::NB; g++) {
        vr += (TA)b[g * R::W];
        vi += (TA)b[S::CH * S::PITCH + g * R::W];
      }
      out(s0 * R::W + l, vr, vi);
    }
  }
}

// U_tot of atom i from the lanes' sums: wself * I + norm * sum, own entries
// and mirrors
template <class T, int J>
__device__ __forceinline__ void rg_store_u(const snap_dev_tables &t,
                                           const rg_map *__restrict__ rgm,
                                           const T (&acc)[rg<J>::SLOTS][2], int l, T *buf,
                                           T *__restrict__ ur, T *__restrict__ ui) {
  rg_group_sum<T, J>(acc, l, buf, [&](int k, T vr, T vi) {
    const rg_map m = rgm[k];
    if (m.ey < 0) return;
    vr *= (T)m.norm;
    vi *= (T)m.norm;
    if (m.diag) vr += (T)t.wself;
    ur[m.uo] = vr;
    ui[m.uo] = vi;
    if (m.um >= 0) {
      ur[m.um] = m.neg ? -vr : vr;
      ui[m.um] = m.neg ? vi : -vi;
    }
  });
}

// U_tot from the neighbour parameters of the last compaction, one wavefront
// per atom; every sum in a fixed order: deterministic.
template <class T, int J>
__global__ void __launch_bounds__(64)
k_snap_ui_rg(snap_dev_tables t, const rg_map *__restrict__ rgm, const int *__restrict__ nin,
             const snap_par<T> *__restrict__ par, int maxn, int n, T *__restrict__ utot_r,
             T *__restrict__ utot_i) {
  __shared__ T s_buf[rg_sum<J>::BUF];
  const int i = blockIdx.x;
  if (i >= n) return;
  const int l = threadIdx.x;
  const int g = l / rg<J>::W, ma = l - g * rg<J>::W;  // g = NB only for idle lanes
  T acc[rg<J>::SLOTS][2];
#pragma unroll
  for (int s = 0; s < rg<J>::SLOTS; s++) acc[s][0] = acc[s][1] = 0;
  rg_u_sums<T, J>(t, par, i, maxn, nin[i], g, ma, acc);
  rg_store_u<T, J>(t, rgm, acc, l, s_buf, utot_r + (size_t)i * t.nu, utot_i + (size_t)i * t.nu);
}

// The compaction (with the neighbour parameters in T's precision) followed by
// U_tot in the same wavefront, one wavefront per atom as k_snap_ui_rg: one
// launch less per force evaluation, and the parameters just written are read
// back from the cache.
template <class T, int J>
__global__ void __launch_bounds__(64)
k_snap_neigh_ui(snap_dev_tables t, const rg_map *__restrict__ rgm,
                const double *__restrict__ x, const int *__restrict__ row,
                const int *__restrict__ num, const int *__restrict__ entries, int pitch, int n,
                double cutsq, int maxn, int *__restrict__ nin, int *__restrict__ nj,
                double *__restrict__ nr, double *__restrict__ f64, float *__restrict__ f32,
                int ntot, snap_par<T> *__restrict__ par, double *__restrict__ fdv,
                T *__restrict__ utot_r, T *__restrict__ utot_i) {
  __shared__ T s_buf[rg_sum<J>::BUF];
  const int i = blockIdx.x;
  if (i >= n) return;
  const int cnt = snap_compact<T>(t, i, x, row, num, entries, pitch, n, cutsq, maxn, nin, nj, nr,
                                  f64, f32, ntot, par, fdv);
  __syncthreads();  // the wavefront's parameter writes are visible
  const int l = threadIdx.x;
  const int g = l / rg<J>::W, ma = l - g * rg<J>::W;
  T acc[rg<J>::SLOTS][2];
#pragma unroll
  for (int q = 0; q < rg<J>::SLOTS; q++) acc[q][0] = acc[q][1] = 0;
  rg_u_sums<T, J>(t, par, i, maxn, cnt, g, ma, acc);
  rg_store_u<T, J>(t, rgm, acc, l, s_buf, utot_r + (size_t)i * t.nu, utot_i + (size_t)i * t.nu);
}

// Blocks of RG_WAVES wavefronts take NB * RG_WAVES neighbours of one atom in
// the force kernel (grid.y over the neighbour slots).
constexpr int RG_WAVES = 4;

// F_ij in reverse mode.  With G_j(e) = w(e) norm_j(e) Y_j(e) (w the
// half-plane weight) the force on the pair is the gradient with respect to
// r_ij of sfac * L,
//   L = sum_j sum_e Re(conj(V_j(e)) G_j(e)).
// V is linear in V_{j-1} and r enters only through a, b and sfac.  So, with
// the adjoints A_j(e) = dL/dRe V + i dL/dIm V propagated from the top layer
// down and A'_j(ma) = A_j(ma+1) from the lane above,
//   A_{j-1}(ma,mb) = G_{j-1} + a A_j - b A'_j               (2 mb < j)
//                  + conj(b) A_j(m) + conj(a) A'_j(m)       (mb = j/2-1, m = j/2)
//   dL/dr_k = Re(conj(da_k) Sa) - Re(conj(db_k) Sb),
//   Sa = sum conj(A_j) V_{j-1} + sum_m A'_j conj(V_{j-1}(j/2-1)),
//   Sb = sum conj(A'_j) V_{j-1} - sum_m A_j conj(V_{j-1}(j/2-1)),
// and L itself is A_0 (V_0 = 1), so the forward pass does not read Y.  It
// keeps V of layers 0..J-1 in registers; what the lane shifts carry past a
// group's edge stays in entries with ma > j, where V is 0.  24 multiply-adds,
// 4 lane shifts of a value and one LDS read of Y per entry (about 44, 6 and
// three records with the factors in U).  The
// force on i is added up over the wavefront before its atomics, and a
// component takes a lane: 2 atomic instructions per seven neighbours (6 each).
template <class T, class TF, int J>
__global__ void __launch_bounds__(64 * RG_WAVES, J <= SNAP_MAXJ ? 3 : 1)
k_snap_fij_rev(snap_dev_tables t, const rg_map *__restrict__ rgm, const int *__restrict__ nin,
               const int *__restrict__ nj, const double *__restrict__ nr,
               const snap_par<T> *__restrict__ par, const double *__restrict__ fdv, int maxn, int n,
               const T *__restrict__ y_r, const T *__restrict__ y_i, TF *__restrict__ f) {
  using R = rg<J>;
  constexpr int NT = 64 * RG_WAVES, RP = 64 + 3;  // RP: the components' rows in different banks
  __shared__ rg_rec<T> s_rec[R::SLOTS * R::W];
  __shared__ T s_red[RG_WAVES][3][RP];
  __shared__ TF s_f[RG_WAVES][3][R::NB];
  const int i = blockIdx.x;
  if (i >= n) return;
  const int cnt_i = nin[i];
  const int row0 = blockIdx.y * (RG_WAVES * R::NB);
  if (row0 >= cnt_i) return;  // no neighbour for this block
#pragma unroll
  for (int q = 0; q < (R::SLOTS * R::W + NT - 1) / NT; q++) {
    const int k = q * NT + (int)threadIdx.x;
    if (k < R::SLOTS * R::W) {
      const rg_map m = rgm[k];
      rg_rec<T> r{0, 0};
      if (m.ey >= 0) {
        const T wgt = (T)(0.5 * m.wq * m.norm);
        r.yr = wgt * y_r[(size_t)i * t.ny + m.ey];
        r.yi = wgt * y_i[(size_t)i * t.ny + m.ey];
      }
      s_rec[k] = r;
    }
  }
  __syncthreads();
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  const int g = l / R::W, ma = l - g * R::W;  // g = NB only for idle lanes
  const int jj0 = row0 + w * R::NB;
  if (jj0 >= cnt_i) return;  // uniform over the wavefront; no block barrier follows
  const int jj = jj0 + g;
  const bool act = g < R::NB && jj < cnt_i;
  const size_t o = (size_t)i * maxn + (act ? jj : jj0);
  const T a_r = par[o].a_r, a_i = par[o].a_i, b_r = par[o].b_r, b_i = par[o].b_i;
  const int tj = t.twojmax;

  // forward: V of layers 0..J-1 (column slot rg_slot0(j) + mb)
  T vs[rg_slot0(J)][2];
#pragma unroll
  for (int s = 0; s < rg_slot0(J); s++) vs[s][0] = vs[s][1] = 0;
  {
    T c[R::COLS][2];
#pragma unroll
    for (int mb = 0; mb < R::COLS; mb++) c[mb][0] = c[mb][1] = 0;
    c[0][0] = ma == 0 ? (T)1 : (T)0;
    vs[0][0] = c[0][0];
    rg_layers<1, J - 1>([&](auto jc) {
      constexpr int j = jc;
      if (j >= tj) return;
      rg_layer<j>(a_r, a_i, b_r, b_i, c);
#pragma unroll
      for (int mb = 0; mb <= j / 2; mb++) {
        vs[rg_slot0(j) + mb][0] = c[mb][0];
        vs[rg_slot0(j) + mb][1] = c[mb][1];
      }
    });
  }

  // backward: adjoints of layer j (columns 0..j/2), from the top layer down
  T ad[R::COLS][2];
#pragma unroll
  for (int mb = 0; mb < R::COLS; mb++) ad[mb][0] = ad[mb][1] = 0;
  T sa_r = 0, sa_i = 0, sb_r = 0, sb_i = 0;
  if (tj == 0) ad[0][0] = s_rec[ma].yr;  // no layer below the top one
  rg_layers<J, 1>([&](auto jc) {
    constexpr int j = jc;
    if (j > tj) return;
    if (j == tj) {  // the top layer's adjoint is its own term
#pragma unroll
      for (int mb = 0; mb <= j / 2; mb++) {
        const rg_rec<T> q = s_rec[(rg_slot0(j) + mb) * R::W + ma];
        ad[mb][0] = q.yr;
        ad[mb][1] = q.yi;
      }
    }
    T up[R::COLS][2];
#pragma unroll
    for (int mb = 0; mb <= j / 2; mb++) {
      up[mb][0] = lane_above(ad[mb][0]);
      up[mb][1] = lane_above(ad[mb][1]);
    }
    constexpr int m = j / 2;
#pragma unroll
    for (int mb = 0; 2 * mb < j; mb++) {
      const rg_rec<T> q = s_rec[(rg_slot0(j - 1) + mb) * R::W + ma];
      const T p0 = vs[rg_slot0(j - 1) + mb][0], p1 = vs[rg_slot0(j - 1) + mb][1];
      const T u0 = ad[mb][0], u1 = ad[mb][1], w0 = up[mb][0], w1 = up[mb][1];
      // (one multiply-add per product: a sum of products would round twice)
      sa_r += u0 * p0;
      sa_r += u1 * p1;
      sa_i += u0 * p1;
      sa_i -= u1 * p0;
      sb_r += w0 * p0;
      sb_r += w1 * p1;
      sb_i += w0 * p1;
      sb_i -= w1 * p0;
      T z0 = q.yr + a_r * u0 - a_i * u1 - b_r * w0 + b_i * w1;
      T z1 = q.yi + a_r * u1 + a_i * u0 - b_r * w1 - b_i * w0;
      if (2 * mb + 2 == j) {  // this column also feeds the middle one
        const T c0 = ad[m][0], c1 = ad[m][1], d0 = up[m][0], d1 = up[m][1];
        sa_r += d0 * p0;
        sa_r += d1 * p1;
        sa_i += d1 * p0;
        sa_i -= d0 * p1;
        sb_r -= c0 * p0;
        sb_r -= c1 * p1;
        sb_i -= c1 * p0;
        sb_i += c0 * p1;
        z0 = z0 + b_r * c0 + b_i * c1 + a_r * d0 + a_i * d1;
        z1 = z1 + b_r * c1 - b_i * c0 + a_r * d1 - a_i * d0;
      }
      ad[mb][0] = z0;
      ad[mb][1] = z1;
    }
  });
  const T auy = ma == 0 ? ad[0][0] : (T)0;
  // the lane's share of F_ij
  const T u3[3] = {par[o].u[0], par[o].u[1], par[o].u[2]};
  const T c1 = par[o].c1, c2 = par[o].c2, c3 = par[o].c3, c4 = par[o].c4, r0i = par[o].r0inv;
  const T sfac = par[o].sfac, dsfac = par[o].dsfac;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const T da_r = c1 * u3[k], da_i = c2 * u3[k] - (k == 2 ? r0i : (T)0);
    const T db_r = c3 * u3[k] + (k == 1 ? r0i : (T)0), db_i = c4 * u3[k] - (k == 0 ? r0i : (T)0);
    s_red[w][k][l] = dsfac * auy * u3[k] +
                     sfac * ((da_r * sa_r + da_i * sa_i) - (db_r * sb_r + db_i * sb_i));
  }
  wave_sync();
  if (ma < 3 && g < R::NB) {  // lane ma adds up component ma over its group
    T s = 0;
#pragma unroll
    for (int m = 0; m < R::W; m++) s += s_red[w][ma][g * R::W + m];
    // ad-hoc repulsion of the reference, force_snap_neigh_impl.h:705-711
    const TF F = act ? (TF)s + (TF)(nr[3 * o + ma] * fdv[o]) : (TF)0;
    if (act) atomicAdd(&f[3 * (size_t)nj[o] + ma], -F);
    s_f[w][ma][g] = F;
  }
  wave_sync();
  if (l < 3) {
    TF s = 0;
#pragma unroll
    for (int q = 0; q < R::NB; q++) s += s_f[w][l][q];
    atomicAdd(&f[3 * (size_t)i + l], s);
  }
}

// per-atom energy: beta_0 + sum_k beta_k B_k + pair repulsion (FP64), one
// wavefront per atom.  The energy is a cubic form of U_tot whose variation is
// dE = sum' w Re(conj(dU) Y) (the identity the forces rest on), so by Euler's
// theorem for homogeneous functions sum_k beta_k B_k = 1/3 sum' w Re(conj(U)
// Y): one pass of the Y stream and a 155- (434- at twojmax 12) term dot
// product instead of every component's Z double sum (164 us for 420 atoms at
// twojmax 8, 713 us for 1024 at 12).
struct snap_edot {
  int u;      // U_tot index of half-plane entry e
  float wgt;  // its half-plane weight (1, 1/2 or 0)
};
constexpr int ENERGY_WAVES = 4;

__global__ void __launch_bounds__(64 * ENERGY_WAVES)
k_snap_energy(int nu, int ny, const snap_edot *__restrict__ dot, double e0, double rcut,
              const int *__restrict__ nin, const double *__restrict__ nr, int maxn, int n,
              const double *__restrict__ utot_r, const double *__restrict__ utot_i,
              const double *__restrict__ y_r, const double *__restrict__ y_i,
              double *__restrict__ eatom) {
  const int i = blockIdx.x * ENERGY_WAVES + threadIdx.x / 64, l = threadIdx.x % 64;
  if (i >= n) return;
  const double *ur = utot_r + (size_t)i * nu, *ui = utot_i + (size_t)i * nu;
  const double *yr = y_r + (size_t)i * ny, *yi = y_i + (size_t)i * ny;
  double e = 0.0;
  for (int k = l; k < ny; k += 64) {
    const snap_edot d = dot[k];
    e += (double)d.wgt * (ur[d.u] * yr[k] + ui[d.u] * yi[k]);
  }
  e *= 1.0 / 3.0;
  // the rc-shifted repulsion of the atom's neighbours
  const double rc2 = rcut * rcut, rc12 = 1.0 / (rc2 * rc2 * rc2 * (rc2 * rc2 * rc2));
  for (int k = l; k < nin[i]; k += 64) {
    const double *r = nr + 3 * ((size_t)i * maxn + k);
    const double r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2], r6 = r2 * r2 * r2;
    e += 1.25e5 * (1.0 / (r6 * r6) - rc12);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, 64);
  if (l == 0) eatom[i] = e0 + e;
}

// sum of n values in double-double, to the host
__global__ void __launch_bounds__(1024) k_snap_energy_sum(const double *__restrict__ v, int n,
                                                          emd_mail mail) {
#pragma clang fp contract(off)
  __shared__ double s_out[2];
  double hi = 0.0, lo = 0.0;
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    double s, e;
    two_sum(hi, v[k], s, e);
    hi = s;
    lo += e;
  }
  block_dd_sum(hi, lo, s_out);
  if (threadIdx.x == 0) {
    *reinterpret_cast<double *>(mail.box + EMD_MAIL_DATA) = s_out[0] + s_out[1];
    emd_mail_post(mail);
  }
}

// ============================================================ host side
struct emd_snap {
  snap_dev_tables t;
  int ncoeff;
  std::vector<double> beta;            // beta_0 .. beta_ncoeff
  std::vector<int> idxj;               // 3 per component
  std::map<std::tuple<int, int, int>, int> cgoff;
  std::vector<double> cg_h;
  double *cg = nullptr;
  etab_entry *etab = nullptr;
  size_t etab_cap = 0;  // entries allocated (kept across coefficient updates)
  // host sources of the last coefficient upload's stream-ordered copies
  // (kept until the next upload, which first waits for the stream)
  std::vector<etab_entry> h_etab;
  std::vector<double> h_kcoef;
  int bzeroflag = 0;
  double rcutfac = 0, radelem = 0;
  // per-system scratch
  int cap_n = 0, cap_maxn = 0;
  int *nin = nullptr, *nj = nullptr;
  double *nr = nullptr;
  // neighbour parameters (snap_par<float> or <double>, per slot) and the
  // repulsion F/r, with the precision the parameters were last written in
  void *par = nullptr;
  double *fdv = nullptr;
  rg_map *rg_map_d = nullptr;  // the register layout's index map, per (column slot, lane)
  size_t cap_par = 0, cap_fdv = 0;
  int par_prec = -1;
  void *u_r = nullptr, *u_i = nullptr, *y_r = nullptr, *y_i = nullptr;
  size_t cap_u = 0, cap_y = 0, cap_ui = 0, cap_yi = 0;
  double *eatom = nullptr;
  int cap_e = 0;
  snap_edot *edot = nullptr;  // energy dot product: U index and weight of each entry
  // slot stream of k_snap_yflat: LDS byte offsets, keys and cg products of
  // its two products per slot, their weights for the current coefficients,
  // run slot per (chunk, thread), first run per entry
  yf_code *yf_codes = nullptr;
  unsigned short *yf_key = nullptr, *yf_meta = nullptr;
  // product stream of k_snap_s_flat (twojmax <= 8): LDS byte offsets, key and
  // cg product of each, entry of each (chunk, thread) (0 if none)
  uint32_t *sf_code = nullptr;
  unsigned short *sf_key = nullptr, *sf_centry = nullptr;
  double *sf_cgw = nullptr;
  int sf_nch = 0;
  unsigned short *yf_keytid = nullptr;  // adjoint triple id of each key
  double *s_part = nullptr;  // the beta adjoint's per-block key sums (k_snap_s_flat)
  size_t cap_spart = 0;
  // emd_snap_static_geometry: the compaction, neighbour parameters and U_tot
  // of the last force or adjoint call (twojmax <= 8) are reused while the
  // caller keeps positions and list fixed: their precision (-1: none), atom
  // count, and the position and list arrays they came from
  int geom_static = 0, geom_prec = -1, geom_n = -1;
  const double *geom_x = nullptr;
  const int *geom_ent = nullptr;
  double *yf_cgw = nullptr, *yf_w64 = nullptr, *yf_kcoef = nullptr;
  float *yf_w32 = nullptr;
  int *yf_rstart = nullptr;
  int yf_nslots = 0, yf_nch = 0;
  std::vector<std::tuple<int, int, int>> yf_keys;  // (a, b, J), sorted
  // adjoint: every (a,b,J) triple grouped by J, with its id
  std::map<std::tuple<int, int, int>, int> tid;
  std::vector<int> sjstart;
  stab_entry *stab = nullptr;
  double *w_r = nullptr, *w_i = nullptr, *sbuf = nullptr;
  size_t cap_w = 0, cap_wi = 0, cap_s = 0;
};

static double host_factorial(int n) {
  struct table {
    double v[2 * SNAP_JBIG + 2];
    table() {
      v[0] = 1.0;
      for (int k = 1; k < 2 * SNAP_JBIG + 2; k++) v[k] = v[k - 1] * k;
    }
  };
  static const table f;
  return f.v[n];
}

// Clebsch-Gordan <j1/2 m1; j2/2 m2 | j/2 m1+m2> by the Racah formula
// (integer-doubled arguments; m1 = k1 - j1/2, m2 = k2 - j2/2)
static double host_cg(int j1, int j2, int j, int k1, int k2) {
  const int aa2 = 2 * k1 - j1, bb2 = 2 * k2 - j2;
  const int cc2 = aa2 + bb2;
  if (cc2 < -j || cc2 > j) return 0.0;
  double sum = 0.0;
  const int zmin = std::max(0, std::max(-(j - j2 + aa2) / 2, -(j - j1 - bb2) / 2));
  const int zmax = std::min((j1 + j2 - j) / 2, std::min((j1 - aa2) / 2, (j2 + bb2) / 2));
  for (int z = zmin; z <= zmax; z++) {
    const double sgn = (z % 2) ? -1.0 : 1.0;
    sum += sgn / (host_factorial(z) * host_factorial((j1 + j2 - j) / 2 - z) *
                  host_factorial((j1 - aa2) / 2 - z) * host_factorial((j2 + bb2) / 2 - z) *
                  host_factorial((j - j2 + aa2) / 2 + z) * host_factorial((j - j1 - bb2) / 2 + z));
  }
  const double delta = std::sqrt(host_factorial((j1 + j2 - j) / 2) * host_factorial((j1 - j2 + j) / 2) *
                                 host_factorial((-j1 + j2 + j) / 2) /
                                 host_factorial((j1 + j2 + j) / 2 + 1));
  const double norm = std::sqrt(host_factorial((j1 + aa2) / 2) * host_factorial((j1 - aa2) / 2) *
                                host_factorial((j2 + bb2) / 2) * host_factorial((j2 - bb2) / 2) *
                                host_factorial((j + cc2) / 2) * host_factorial((j - cc2) / 2) *
                                (j + 1));
  return sum * delta * norm;
}

// Copies of U_tot for one read of a lane group served in one LDS cycle: the
// group's distinct U entries are matched to distinct bank residues (u + shift(c))
// mod MOD, each entry choosing one copy c (augmenting paths, a free residue
// taken before any is freed); an entry left unmatched takes the least loaded
// residue among its copies.  Lanes reading the same entry read the same copy.
// Bit sets, as this is most of emd_snap_create: 55 of its 113 ms at twojmax 12
// with arrays of flags (one core of an EPYC host).
template <class L>
struct yf_matching {
  static_assert(L::MOD == 32, "residues in a 32-bit set");
  int addr[L::GROUP], copy_of[L::GROUP], owner[L::MOD];
  uint32_t open, seen;  // residues without an owner; visited by the path
  bool take(int a, int c, int b) {
    open &= ~(1u << b);
    owner[b] = a;
    copy_of[a] = c;
    return true;
  }
  bool augment(int a) {
    for (int c = 0; c < L::NCOPY; c++) {
      const int b = (addr[a] + L::shift(c)) % L::MOD;
      if (open >> b & 1) return take(a, c, b);
    }
    for (int c = 0; c < L::NCOPY; c++) {
      const int b = (addr[a] + L::shift(c)) % L::MOD;
      if (seen >> b & 1) continue;
      seen |= 1u << b;
      if (augment(owner[b])) return take(a, c, b);
    }
    return false;
  }
  // copies of the group's entries u[0 .. GROUP)
  void assign(const int *u, int *cp, std::vector<int> &index) {
    int na = 0;
    for (int l = 0; l < L::GROUP; l++)
      if (index[u[l]] < 0) {
        index[u[l]] = na;
        addr[na++] = u[l];
      }
    open = ~0u;
    bool all = true;
    for (int a = 0; a < na; a++) {
      seen = 0;
      copy_of[a] = -1;
      all &= augment(a);
    }
    int load[L::MOD] = {0};
    for (int a = 0; a < na && !all; a++)
      if (copy_of[a] >= 0) load[(addr[a] + L::shift(copy_of[a])) % L::MOD]++;
    for (int a = 0; a < na && !all; a++)
      if (copy_of[a] < 0) {
        int best = 0;
        for (int c = 1; c < L::NCOPY; c++)
          if (load[(addr[a] + L::shift(c)) % L::MOD] < load[(addr[a] + L::shift(best)) % L::MOD])
            best = c;
        copy_of[a] = best;
        load[(addr[a] + L::shift(best)) % L::MOD]++;
      }
    for (int l = 0; l < L::GROUP; l++) cp[l] = copy_of[index[u[l]]];
    for (int a = 0; a < na; a++) index[addr[a]] = -1;
  }
};

// LDS byte offsets of one read (of U entry u) of every slot of a stream
template <class L>
static std::vector<unsigned short> yf_offsets(const std::vector<int> &u, int nu) {
  std::vector<int> cp(u.size(), 0), index(nu, -1);
  std::vector<unsigned short> off(u.size());
  yf_matching<L> m;
  for (size_t g0 = 0; g0 < u.size(); g0 += L::GROUP) m.assign(&u[g0], &cp[g0], index);
  for (size_t k = 0; k < u.size(); k++) off[k] = (unsigned short)((L::base(cp[k]) + u[k]) * 8);
  return off;
}
static std::vector<unsigned short> yf_offsets(const std::vector<int> &u, const snap_dev_tables &t) {
  // (the same word offsets serve FP32 and FP64, there into the real array)
  return t.twojmax <= SNAP_MAXJ ? yf_offsets<yf_layout<float, SNAP_MAXJ>>(u, t.nu)
                                : yf_offsets<yf_layout<float, SNAP_JBIG>>(u, t.nu);
}

struct yf_term {
  int i1, i2, key;
  double cgw;
};
struct yf_slot {
  int c, x, y;        // U_c (w_x U_x + w_y U_y)
  int kx, ky;
  double cx, cy;
};

// The products of one entry as slots of two that share a U entry: the
// products are the edges of a graph over the U entries, and a connected graph
// splits into pairs of adjacent edges but for one edge when their number is
// odd (depth first: a vertex pairs the edges its subtree left to it, and takes
// the edge to its parent for an odd one).
struct yf_pairs {
  const yf_term *t = nullptr;
  std::vector<yf_slot> *out = nullptr;
  std::vector<int> first, at, adj;  // edges of vertex v: adj[first[v] .. first[v + 1])
  std::vector<char> used, seen;
  explicit yf_pairs(int nu) : first(nu + 1), at(nu), seen(nu) {}
  void split(const std::vector<yf_term> &terms, std::vector<yf_slot> &slots) {
    t = terms.data();
    out = &slots;
    std::fill(first.begin(), first.end(), 0);
    std::fill(seen.begin(), seen.end(), 0);
    for (const yf_term &q : terms) {
      first[q.i1 + 1]++;
      if (q.i2 != q.i1) first[q.i2 + 1]++;
    }
    for (size_t v = 1; v < first.size(); v++) first[v] += first[v - 1];
    std::copy(first.begin(), first.end() - 1, at.begin());
    adj.resize(first.back());
    for (size_t e = 0; e < terms.size(); e++) {
      adj[at[t[e].i1]++] = (int)e;
      if (t[e].i2 != t[e].i1) adj[at[t[e].i2]++] = (int)e;
    }
    used.assign(terms.size(), 0);
    slots.reserve(terms.size() / 2 + 8);
    for (const yf_term &q : terms)
      if (!seen[q.i1]) visit(q.i1, -1);
  }
  int other(int e, int v) const { return t[e].i1 == v ? t[e].i2 : t[e].i1; }
  void emit(int v, int e1, int e2) {
    yf_slot s{v, other(e1, v), 0, t[e1].key, 0, t[e1].cgw, 0.0};
    if (e2 >= 0) {
      s.y = other(e2, v);
      s.ky = t[e2].key;
      s.cy = t[e2].cgw;
    } else {
      s.y = s.x;  // weight 0
      s.ky = s.kx;
    }
    out->push_back(s);
  }
  // true if v took the edge to its parent
  bool visit(int v, int parent) {
    seen[v] = 1;
    int left = -1;
    for (int k = first[v]; k < first[v + 1]; k++) {
      const int e = adj[k];
      if (used[e]) continue;
      used[e] = 1;
      const int w = other(e, v);
      if (w != v && !seen[w] && visit(w, e)) continue;
      if (left < 0) {
        left = e;
      } else {
        emit(v, left, e);
        left = -1;
      }
    }
    if (left < 0) return false;
    emit(v, left, parent);
    return parent >= 0;
  }
};

// Entries' lists of the given lengths in chunks of `chunk`, in entry order:
// (entry, first element) of each, `threads` threads taking P each
struct yf_chunks {
  std::vector<std::pair<int, int>> at;
  int P = 0;
  yf_chunks(const std::vector<int> &len, int chunk, int threads) {
    for (int e = 0; e < (int)len.size(); e++)
      for (int f = 0; f < len[e]; f += chunk) at.push_back(std::make_pair(e, f));
    P = ((int)at.size() + threads - 1) / threads;
  }
};

template <class V>
static emd_status yf_upload(emd_ctx *ctx, V **dst, const std::vector<V> &v) {
  EMD_HIP(ctx, hipMalloc(dst, std::max<size_t>(1, v.size()) * sizeof(V)));
  if (!v.empty()) EMD_HIP(ctx, hipMemcpy(*dst, v.data(), v.size() * sizeof(V), hipMemcpyHostToDevice));
  return EMD_OK;
}

// the stream of k_snap_s_flat (see there)
static emd_status snap_build_sflat(emd_ctx *ctx, emd_snap *sn,
                                   const std::vector<std::vector<yf_term>> &eterms) {
  const snap_dev_tables &t = sn->t;
  std::vector<int> len(t.ny);
  for (int e = 0; e < t.ny; e++) len[e] = (int)eterms[e].size();
  const yf_chunks ch(len, SF_CHUNK, SF_THREADS);
  const int nchunks = (int)ch.at.size(), P = ch.P;
  const size_t nslots = (size_t)P * SF_CHUNK * SF_THREADS;
  std::vector<int> u1(nslots, 0), u2(nslots, 0);
  std::vector<unsigned short> key(nslots, 0), centry((size_t)P * SF_THREADS, 0);
  std::vector<double> cgw(nslots, 0.0);
  // A chunk's terms all belong to one entry, so their order within the
  // chunk is free (it changes rounding only): by key, padding last, so that
  // runs of one key are summed before the atomic add (1.8 runs per chunk at
  // twojmax 8).  LDS bank conflicts are left to the copy assignment (offline:
  // 1.08 cycles per read against 1.04 with a bank-greedy order).
  for (int g = 0; g < nchunks; g++) {
    const int e = ch.at[g].first, th = g / P, c = g % P;
    const int f = ch.at[g].second, m = std::min(SF_CHUNK, len[e] - f);
    std::vector<yf_term> pool(eterms[e].begin() + f, eterms[e].begin() + f + m);
    std::stable_sort(pool.begin(), pool.end(), [](const yf_term &x, const yf_term &y) {
      if (x.key != y.key) return x.key < y.key;
      return x.i1 != y.i1 ? x.i1 < y.i1 : x.i2 < y.i2;
    });
    for (int k = 0; k < m; k++) {
      const size_t slot = ((size_t)c * SF_CHUNK + k) * SF_THREADS + th;
      u1[slot] = pool[k].i1;
      u2[slot] = pool[k].i2;
      key[slot] = (unsigned short)pool[k].key;
      cgw[slot] = pool[k].cgw;
    }
    centry[(size_t)c * SF_THREADS + th] = (unsigned short)e;
  }
  const std::vector<unsigned short> o1 = yf_offsets(u1, t), o2 = yf_offsets(u2, t);
  std::vector<uint32_t> code(nslots);
  for (size_t k = 0; k < nslots; k++) code[k] = o1[k] | (uint32_t)o2[k] << 16;
  sn->sf_nch = P;
  EMD_TRY(yf_upload(ctx, &sn->sf_code, code));
  EMD_TRY(yf_upload(ctx, &sn->sf_key, key));
  EMD_TRY(yf_upload(ctx, &sn->sf_cgw, cgw));
  EMD_TRY(yf_upload(ctx, &sn->sf_centry, centry));
  return EMD_OK;
}

// the beta-independent part of the flat Y stream (see k_snap_yflat)
static emd_status snap_build_yflat(emd_ctx *ctx, emd_snap *sn) {
  const snap_dev_tables &t = sn->t;
  const int nk = (int)sn->idxj.size() / 3;
  std::set<std::tuple<int, int, int>> keyset;
  for (int k = 0; k < nk; k++) {
    const int j1 = sn->idxj[3 * k], j2 = sn->idxj[3 * k + 1], j = sn->idxj[3 * k + 2];
    keyset.insert(std::make_tuple(std::max(j1, j2), std::min(j1, j2), j));
    keyset.insert(std::make_tuple(std::max(j, j2), std::min(j, j2), j1));
    keyset.insert(std::make_tuple(std::max(j1, j), std::min(j1, j), j2));
  }
  sn->yf_keys.assign(keyset.begin(), keyset.end());
  std::vector<std::vector<yf_term>> eterms(t.ny);
  std::vector<int> seen;
  for (int J = 0; J <= t.twojmax; J++)
    for (int mb = 0; 2 * mb <= J; mb++)
      for (int ma = 0; ma <= J; ma++) {
        if (2 * mb == J && ma > mb) continue;  // half-plane weight 0
        const int e = t.ystart[J] + mb * (J + 1) + ma;
        for (size_t q = 0; q < sn->yf_keys.size(); q++) {
          int a, b, JJ;
          std::tie(a, b, JJ) = sn->yf_keys[q];
          if (JJ != J) continue;
          // a == b: (i1, i2) -> the term of this key and entry that holds it
          const int key0 = (int)eterms[e].size();
          if (a == b) seen.assign((size_t)(a + 1) * (a + 1) * (a + 1) * (a + 1), -1);
          const int cgoff = sn->cgoff.at(sn->yf_keys[q]);
          const int ma1lo = std::max(0, (2 * ma - J - b + a) / 2);
          const int ma1hi = std::min(a, (2 * ma - J + b + a) / 2);
          const int mb1lo = std::max(0, (2 * mb - J - b + a) / 2);
          const int mb1hi = std::min(a, (2 * mb - J + b + a) / 2);
          for (int ma1 = ma1lo; ma1 <= ma1hi; ma1++) {
            const int ma2 = (2 * ma - J - (2 * ma1 - a) + b) / 2;
            const double cma = sn->cg_h[cgoff + ma1 * (b + 1) + ma2];
            for (int mb1 = mb1lo; mb1 <= mb1hi; mb1++) {
              const int mb2 = (2 * mb - J - (2 * mb1 - a) + b) / 2;
              const double cw = cma * sn->cg_h[cgoff + mb1 * (b + 1) + mb2];
              if (cw == 0.0) continue;
              int i1 = t.ustart[a] + ma1 * (a + 1) + mb1, i2 = t.ustart[b] + ma2 * (b + 1) + mb2;
              // a == b: (i1, i2) and (i2, i1) are the same product
              if (a == b) {
                if (i1 < i2) std::swap(i1, i2);
                int &at = seen[(size_t)(i1 - t.ustart[a]) * (a + 1) * (a + 1) + (i2 - t.ustart[a])];
                if (at >= key0) {
                  eterms[e][at].cgw += cw;
                  continue;
                }
                at = (int)eterms[e].size();
              }
              eterms[e].push_back(yf_term{i1, i2, (int)q, cw});
            }
          }
        }
      }
  // ---- the slot stream of k_snap_yflat
  std::vector<std::vector<yf_slot>> eslots(t.ny);
  std::vector<int> len(t.ny);
  yf_pairs pairs(t.nu);
  for (int e = 0; e < t.ny; e++) {
    pairs.split(eterms[e], eslots[e]);
    len[e] = (int)eslots[e].size();
  }
  const bool small = t.twojmax <= SNAP_MAXJ;
  const int nt = small ? yf_threads<SNAP_MAXJ>() : yf_threads<SNAP_JBIG>();
  const yf_chunks ch(len, YF_CHUNK, nt);
  const int nchunks = (int)ch.at.size(), P = ch.P;
  // runs: a thread's consecutive chunks of one entry; run slots numbered
  // entry by entry, in thread order within an entry (= slot order)
  std::vector<unsigned short> meta((size_t)P * nt, YF_NO_RUN);
  std::vector<int> rstart(t.ny + 1, 0);
  int nruns = 0, done = 0;
  for (int g = 0; g < nchunks; g++) {
    const int e = ch.at[g].first;
    while (done <= e) rstart[done++] = nruns;
    if (g % P == P - 1 || g + 1 == nchunks || ch.at[g + 1].first != e)
      meta[(size_t)(g % P) * nt + g / P] = (unsigned short)nruns++;
  }
  while (done <= t.ny) rstart[done++] = nruns;
  if (nruns > (small ? yf_maxruns<SNAP_MAXJ>() : yf_maxruns<SNAP_JBIG>()) ||
      t.nu > (small ? snap_nu(SNAP_MAXJ) : snap_nu(SNAP_JBIG)))
    return emd_set_error(ctx, EMD_ERR_ARG, "emd_snap_create: Y stream too large");
  const size_t nslots = (size_t)P * YF_CHUNK * nt;
  std::vector<int> uc(nslots, 0), ux(nslots, 0), uy(nslots, 0);
  std::vector<unsigned short> key(2 * nslots, 0);
  std::vector<double> cgw(2 * nslots, 0.0);
  for (int g = 0; g < nchunks; g++) {
    const std::vector<yf_slot> &es = eslots[ch.at[g].first];
    for (int k = 0; k < YF_CHUNK && ch.at[g].second + k < (int)es.size(); k++) {
      const yf_slot &q = es[ch.at[g].second + k];
      const size_t slot = yf_place(P, g % P, k, g / P);
      uc[slot] = q.c;
      ux[slot] = q.x;
      uy[slot] = q.y;
      key[2 * slot] = (unsigned short)q.kx;
      key[2 * slot + 1] = (unsigned short)q.ky;
      cgw[2 * slot] = q.cx;
      cgw[2 * slot + 1] = q.cy;
    }
  }
  {
    const std::vector<unsigned short> oc = yf_offsets(uc, t), ox = yf_offsets(ux, t),
                                      oy = yf_offsets(uy, t);
    std::vector<yf_code> code(nslots);
    for (size_t k = 0; k < nslots; k++) code[yf_place2(k)] = yf_code{oc[k], ox[k], oy[k], 0};
    EMD_TRY(yf_upload(ctx, &sn->yf_codes, code));
  }
  sn->yf_nslots = (int)nslots;
  sn->yf_nch = P;
  std::vector<unsigned short> keytid(sn->yf_keys.size(), 0);
  for (size_t q = 0; q < sn->yf_keys.size(); q++) keytid[q] = (unsigned short)sn->tid.at(sn->yf_keys[q]);
  EMD_TRY(yf_upload(ctx, &sn->yf_keytid, keytid));
  EMD_TRY(yf_upload(ctx, &sn->yf_key, key));
  EMD_TRY(yf_upload(ctx, &sn->yf_meta, meta));
  EMD_TRY(yf_upload(ctx, &sn->yf_cgw, cgw));
  EMD_TRY(yf_upload(ctx, &sn->yf_rstart, rstart));
  EMD_HIP(ctx, hipMalloc(&sn->yf_w64, std::max<size_t>(1, 2 * nslots) * sizeof(double)));
  EMD_HIP(ctx, hipMalloc(&sn->yf_w32, std::max<size_t>(1, 2 * nslots) * sizeof(float)));
  EMD_HIP(ctx, hipMalloc(&sn->yf_kcoef, std::max<size_t>(1, sn->yf_keys.size()) * sizeof(double)));
  return small ? snap_build_sflat(ctx, sn, eterms) : EMD_OK;
}

// the index map of the register layout (see rg_map)
template <int J>
static emd_status snap_build_rg(emd_ctx *ctx, emd_snap *sn) {
  using R = rg<J>;
  const snap_dev_tables &t = sn->t;
  double fact[J + 1];
  fact[0] = 1.0;
  for (int k = 1; k <= J; k++) fact[k] = fact[k - 1] * k;
  std::vector<rg_map> mp(R::SLOTS * R::W);
  for (int sl = 0; sl < R::SLOTS; sl++)
    for (int ma = 0; ma < R::W; ma++) {
      int j = 0;
      while (j < J && rg_slot0(j + 1) <= sl) j++;
      const int mb = sl - rg_slot0(j);
      rg_map m{0.0, -1, -1, -1, 0, 0, 0, 0};
      if (j <= t.twojmax && ma <= j) {
        m.norm = std::sqrt(fact[ma] * fact[j - ma] / (fact[mb] * fact[j - mb]));
        // the reference's half plane: middle column ma < mb, diagonal 1/2
        m.wq = 2 * mb == j ? (ma < mb ? 2 : (ma == mb ? 1 : 0)) : 2;
        m.ey = t.ystart[j] + mb * (j + 1) + ma;
        m.uo = t.ustart[j] + ma * (j + 1) + mb;
        m.um = 2 * mb != j ? t.ustart[j] + (j - ma) * (j + 1) + (j - mb) : -1;
        m.neg = (ma + mb) & 1;
        m.diag = ma == mb;
      }
      mp[sl * R::W + ma] = m;
    }
  EMD_HIP(ctx, hipMalloc(&sn->rg_map_d, mp.size() * sizeof(mp[0])));
  EMD_HIP(ctx, hipMemcpy(sn->rg_map_d, mp.data(), mp.size() * sizeof(mp[0]), hipMemcpyHostToDevice));
  return EMD_OK;
}

static emd_status snap_upload_coeff(emd_ctx *ctx, emd_snap *sn) {
  const int twojmax = sn->t.twojmax;
  // Y weights: the three roles of each component (compute_dbidrj)
  std::map<std::tuple<int, int, int>, double> coef;
  const int nk = (int)sn->idxj.size() / 3;
  for (int k = 0; k < nk; k++) {
    const int j1 = sn->idxj[3 * k], j2 = sn->idxj[3 * k + 1], j = sn->idxj[3 * k + 2];
    const double b = sn->beta[k + 1];
    coef[std::make_tuple(std::max(j1, j2), std::min(j1, j2), j)] += 2.0 * b;
    coef[std::make_tuple(std::max(j, j2), std::min(j, j2), j1)] += 2.0 * b * (j + 1) / (j1 + 1.0);
    coef[std::make_tuple(std::max(j1, j), std::min(j1, j), j2)] += 2.0 * b * (j + 1) / (j2 + 1.0);
  }
  EMD_HIP(ctx, hipStreamSynchronize(ctx->stream));  // the previous upload's copies are done
  std::vector<etab_entry> &et = sn->h_etab;
  et.clear();
  for (int k = 0; k < nk; k++) {
    etab_entry e;
    e.j1 = sn->idxj[3 * k]; e.j2 = sn->idxj[3 * k + 1]; e.j = sn->idxj[3 * k + 2];
    e.cgoff = sn->cgoff.at(std::make_tuple(e.j1, e.j2, e.j));
    e.beta = sn->beta[k + 1];
    et.push_back(e);
  }
  // the tables keep their allocation while they fit (coefficient updates
  // in a force-matching loop do not reallocate); copies are stream-ordered
  if (et.size() > sn->etab_cap || !sn->etab) {
    EMD_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (sn->etab) EMD_HIP(ctx, hipFree(sn->etab));
    sn->etab = nullptr;
    sn->etab_cap = std::max<size_t>(1, et.size());
    EMD_HIP(ctx, hipMalloc(&sn->etab, sn->etab_cap * sizeof(etab_entry)));
  }
  if (!et.empty())
    EMD_HIP(ctx, hipMemcpyAsync(sn->etab, et.data(), et.size() * sizeof(etab_entry),
                                hipMemcpyHostToDevice, ctx->stream));
  if (sn->yf_codes) {
    std::vector<double> &kc = sn->h_kcoef;
    kc.assign(sn->yf_keys.size(), 0.0);
    for (size_t q = 0; q < kc.size(); q++) {
      auto it = coef.find(sn->yf_keys[q]);
      if (it != coef.end()) kc[q] = it->second;
    }
    if (!kc.empty())
      EMD_HIP(ctx, hipMemcpyAsync(sn->yf_kcoef, kc.data(), kc.size() * sizeof(double),
                                  hipMemcpyHostToDevice, ctx->stream));
    const int nslots = sn->yf_nslots;
    if (nslots > 0)
      EMD_LAUNCH(ctx, "snap_coeff", k_yf_weights, emd_blocks(2 * nslots, 256), 256, 0, nslots,
                 sn->yf_key, sn->yf_cgw, sn->yf_kcoef, sn->yf_w64, sn->yf_w32);
  }
  return EMD_OK;
}

extern "C" emd_status emd_snap_create(emd_ctx *ctx, const emd_snap_params *p, emd_snap **out) {
  if (!ctx || !p || !out) return EMD_ERR_ARG;
  *out = nullptr;
  if (p->twojmax < 0 || p->twojmax > SNAP_JBIG)
    return emd_set_error(ctx, EMD_ERR_ARG, "emd_snap_create: twojmax must be in 0..%d", SNAP_JBIG);
  if (!p->coeff) return emd_set_error(ctx, EMD_ERR_ARG, "emd_snap_create: no coefficients");
  emd_snap *sn = new emd_snap();
  snap_dev_tables &t = sn->t;
  memset(&t, 0, sizeof(t));
  const int twojmax = p->twojmax;
  t.twojmax = twojmax;
  int nu = 0, ny = 0;
  for (int j = 0; j <= twojmax; j++) {
    t.ustart[j] = nu;
    t.ystart[j] = ny;
    nu += (j + 1) * (j + 1);
    ny += (j + 1) * (j / 2 + 1);
  }
  t.ustart[twojmax + 1] = nu;
  t.ystart[twojmax + 1] = ny;
  t.nu = nu;
  t.ny = ny;
  t.rfac0 = p->rfac0;
  t.rmin0 = p->rmin0;
  t.rcut = (p->radelem + p->radelem) * p->rcutfac;
  t.wj = p->wjelem;
  t.wself = 1.0;
  t.switchflag = p->switchflag;
  sn->bzeroflag = p->bzeroflag;
  sn->rcutfac = p->rcutfac;
  sn->radelem = p->radelem;
  // component list (SNA::build_indexlist, diagonalstyle 3) and CG blocks
  for (int j1 = 0; j1 <= twojmax; j1++)
    for (int j2 = 0; j2 <= j1; j2++)
      for (int j = j1 - j2; j <= std::min(twojmax, j1 + j2); j += 2) {
        if (j >= j1) {
          sn->idxj.push_back(j1);
          sn->idxj.push_back(j2);
          sn->idxj.push_back(j);
        }
        sn->cgoff[std::make_tuple(j1, j2, j)] = (int)sn->cg_h.size();
        for (int k1 = 0; k1 <= j1; k1++)
          for (int k2 = 0; k2 <= j2; k2++) sn->cg_h.push_back(host_cg(j1, j2, j, k1, k2));
      }
  sn->ncoeff = (int)sn->idxj.size() / 3;
  {
    // all (a,b,J) triples grouped by J for the adjoint contraction
    std::vector<stab_entry> st;
    for (int J = 0; J <= twojmax; J++) {
      sn->sjstart.push_back((int)st.size());
      for (auto &kv : sn->cgoff) {
        int a, b, JJ;
        std::tie(a, b, JJ) = kv.first;
        if (JJ != J) continue;
        const int id = (int)sn->tid.size();
        sn->tid[kv.first] = id;
        st.push_back(stab_entry{a, b, kv.second, id});
      }
    }
    sn->sjstart.push_back((int)st.size());
    if (st.size() > (size_t)SNAP_MAXT) {
      delete sn;
      return emd_set_error(ctx, EMD_ERR_ARG, "emd_snap_create: too many (a,b,J) triples");
    }
    EMD_HIP(ctx, hipMalloc(&sn->stab, st.size() * sizeof(stab_entry)));
    EMD_HIP(ctx, hipMemcpy(sn->stab, st.data(), st.size() * sizeof(stab_entry), hipMemcpyHostToDevice));
  }
  if (p->ncoeff != sn->ncoeff) {
    const int want = sn->ncoeff;
    emd_snap_destroy(ctx, sn);
    return emd_set_error(ctx, EMD_ERR_ARG, "emd_snap_create: ncoeff %d but twojmax %d has %d",
                         p->ncoeff, twojmax, want);
  }
  sn->beta.assign(p->coeff, p->coeff + sn->ncoeff + 1);
  if (hipMalloc(&sn->cg, sn->cg_h.size() * sizeof(double)) != hipSuccess) {
    delete sn;
    return emd_set_error(ctx, EMD_ERR_ALLOC, "emd_snap_create: hipMalloc failed");
  }
  EMD_HIP(ctx, hipMemcpy(sn->cg, sn->cg_h.data(), sn->cg_h.size() * sizeof(double),
                         hipMemcpyHostToDevice));
  {
    std::vector<snap_edot> dot(std::max(1, t.ny));
    for (int j = 0; j <= twojmax; j++)
      for (int mb = 0; 2 * mb <= j; mb++)
        for (int ma = 0; ma <= j; ma++)
          dot[t.ystart[j] + mb * (j + 1) + ma] =
              snap_edot{t.ustart[j] + ma * (j + 1) + mb,
                        2 * mb != j || ma < mb ? 1.0f : (ma == mb ? 0.5f : 0.0f)};
    EMD_HIP(ctx, hipMalloc(&sn->edot, dot.size() * sizeof(snap_edot)));
    EMD_HIP(ctx, hipMemcpy(sn->edot, dot.data(), dot.size() * sizeof(snap_edot),
                           hipMemcpyHostToDevice));
  }
  emd_status st = snap_build_yflat(ctx, sn);
  if (st == EMD_OK)
    st = twojmax <= SNAP_MAXJ ? snap_build_rg<SNAP_MAXJ>(ctx, sn) : snap_build_rg<SNAP_JBIG>(ctx, sn);
  if (st == EMD_OK) st = snap_upload_coeff(ctx, sn);
  if (st != EMD_OK) {
    emd_snap_destroy(ctx, sn);
    return st;
  }
  *out = sn;
  return EMD_OK;
}

extern "C" emd_status emd_snap_destroy(emd_ctx *ctx, emd_snap *sn) {
  if (!sn) return EMD_OK;
  if (ctx) hipStreamSynchronize(ctx->stream);
  void *ptrs[] = {sn->cg, sn->etab, sn->nin, sn->nj, sn->nr, sn->par, sn->fdv,
                  sn->rg_map_d,
                  sn->stab, sn->w_r, sn->edot,
                  sn->w_i, sn->sbuf,
                  sn->u_r, sn->u_i, sn->y_r, sn->y_i, sn->eatom,
                  sn->yf_codes, sn->yf_key, sn->yf_meta, sn->yf_cgw, sn->sf_code, sn->sf_key,
                  sn->sf_cgw, sn->sf_centry, sn->yf_keytid, sn->s_part,
                  sn->yf_w64, sn->yf_w32, sn->yf_rstart, sn->yf_kcoef};
  for (void *q : ptrs)
    if (q) hipFree(q);
  delete sn;
  return EMD_OK;
}

extern "C" emd_status emd_snap_static_geometry(emd_ctx *ctx, emd_snap *sn, int on) {
  if (!ctx || !sn) return EMD_ERR_ARG;
  sn->geom_static = on != 0;
  sn->geom_prec = -1;
  return EMD_OK;
}

extern "C" emd_status emd_snap_set_coeff(emd_ctx *ctx, emd_snap *sn, const double *coeff) {
  if (!ctx || !sn || !coeff) return EMD_ERR_ARG;
  EMD_HIP(ctx, hipStreamSynchronize(ctx->stream));
  sn->beta.assign(coeff, coeff + sn->ncoeff + 1);
  return snap_upload_coeff(ctx, sn);
}

static emd_status snap_scratch(emd_ctx *ctx, emd_snap *sn, int n, int maxn) {
  if (n > sn->cap_n || maxn > sn->cap_maxn || !sn->nin) {
    EMD_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (sn->nin) EMD_HIP(ctx, hipFree(sn->nin));
    if (sn->nj) EMD_HIP(ctx, hipFree(sn->nj));
    if (sn->nr) EMD_HIP(ctx, hipFree(sn->nr));
    const int cn = n + n / 8 + 16, cm = maxn + 8;
    EMD_HIP(ctx, hipMalloc(&sn->nin, (size_t)cn * sizeof(int)));
    EMD_HIP(ctx, hipMalloc(&sn->nj, (size_t)cn * cm * sizeof(int)));
    EMD_HIP(ctx, hipMalloc(&sn->nr, (size_t)cn * cm * 3 * sizeof(double)));
    sn->cap_n = cn;
    sn->cap_maxn = cm;
  }
  const size_t slots = (size_t)n * sn->cap_maxn;
  EMD_TRY(emd_ensure(ctx, &sn->par, &sn->cap_par, slots * sizeof(snap_par<double>)));
  EMD_TRY(emd_ensure(ctx, (void **)&sn->fdv, &sn->cap_fdv, slots * sizeof(double)));
  EMD_TRY(emd_ensure(ctx, &sn->u_r, &sn->cap_u, (size_t)n * sn->t.nu * sizeof(double)));
  EMD_TRY(emd_ensure(ctx, &sn->u_i, &sn->cap_ui, (size_t)n * sn->t.nu * sizeof(double)));
  EMD_TRY(emd_ensure(ctx, &sn->y_r, &sn->cap_y, (size_t)n * sn->t.ny * sizeof(double)));
  EMD_TRY(emd_ensure(ctx, &sn->y_i, &sn->cap_yi, (size_t)n * sn->t.ny * sizeof(double)));
  return EMD_OK;
}

// The compaction with the neighbour parameters in precision prec and U_tot of
// every atom, in one launch.  zero_prec: EMD_FP64 or EMD_MIXED to zero that
// precision's force array (all n_local + n_ghost rows) in the same launch, or -1.
template <class T>
static emd_status snap_neigh_ui_as(emd_ctx *ctx, const emd_system *s, const emd_neigh *nl,
                                   emd_snap *sn, int zero_prec) {
  const int n = s->n_local;
  const double rcutmax = 2.0 * sn->radelem * sn->rcutfac;
  const int *row = nl->layout == EMD_NEIGH_CSR ? nl->row : nullptr;
  double *f64 = zero_prec == EMD_FP64 ? s->f : nullptr;
  float *f32 = zero_prec == EMD_MIXED ? s->f32 : nullptr;
  if (sn->t.twojmax <= SNAP_MAXJ)
    EMD_LAUNCH(ctx, "snap_ui", (k_snap_neigh_ui<T, SNAP_MAXJ>), n, 64, 0, sn->t, sn->rg_map_d,
               s->x, row, nl->num, nl->entries, nl->maxneighs, n, rcutmax * rcutmax, sn->cap_maxn,
               sn->nin, sn->nj, sn->nr, f64, f32, s->n_local + s->n_ghost, (snap_par<T> *)sn->par,
               sn->fdv, (T *)sn->u_r, (T *)sn->u_i);
  else
    EMD_LAUNCH(ctx, "snap_ui", (k_snap_neigh_ui<T, SNAP_JBIG>), n, 64, 0, sn->t, sn->rg_map_d,
               s->x, row, nl->num, nl->entries, nl->maxneighs, n, rcutmax * rcutmax, sn->cap_maxn,
               sn->nin, sn->nj, sn->nr, f64, f32, s->n_local + s->n_ghost, (snap_par<T> *)sn->par,
               sn->fdv, (T *)sn->u_r, (T *)sn->u_i);
  return EMD_OK;
}

static emd_status snap_neigh_ui(emd_ctx *ctx, const emd_system *s, const emd_neigh *nl,
                                emd_snap *sn, int zero_prec, int prec) {
  EMD_TRY(snap_scratch(ctx, sn, s->n_local, nl->maxneighs > 0 ? nl->maxneighs : 1));
  if (prec == EMD_MIXED) EMD_TRY(snap_neigh_ui_as<float>(ctx, s, nl, sn, zero_prec));
  else EMD_TRY(snap_neigh_ui_as<double>(ctx, s, nl, sn, zero_prec));
  sn->par_prec = prec;
  return EMD_OK;
}

// U_tot of every atom in FP64 from the last compaction
static emd_status launch_ui(emd_ctx *ctx, emd_snap *sn, int n) {
  snap_par<double> *par = (snap_par<double> *)sn->par;
  if (sn->par_prec != EMD_FP64)
    EMD_LAUNCH(ctx, "snap_neigh", k_snap_par, n, 64, 0, sn->t, sn->nin, sn->nr, sn->cap_maxn, n,
               par, sn->fdv);
  sn->par_prec = EMD_FP64;
  if (sn->t.twojmax <= SNAP_MAXJ)
    EMD_LAUNCH(ctx, "snap_ui", (k_snap_ui_rg<double, SNAP_MAXJ>), n, 64, 0, sn->t, sn->rg_map_d,
               sn->nin, par, sn->cap_maxn, n, (double *)sn->u_r, (double *)sn->u_i);
  else
    EMD_LAUNCH(ctx, "snap_ui", (k_snap_ui_rg<double, SNAP_JBIG>), n, 64, 0, sn->t, sn->rg_map_d,
               sn->nin, par, sn->cap_maxn, n, (double *)sn->u_r, (double *)sn->u_i);
  return EMD_OK;
}

template <class T>
static emd_status snap_y(emd_ctx *ctx, emd_snap *sn, int n) {
  T *ur = (T *)sn->u_r, *ui = (T *)sn->u_i, *yr = (T *)sn->y_r, *yi = (T *)sn->y_i;
  const cpair<T> *w = std::is_same<T, float>::value ? (const cpair<T> *)sn->yf_w32
                                                    : (const cpair<T> *)sn->yf_w64;
  // Atoms per block: more of them share each code and weight load, but take
  // LDS from other blocks, and leave CUs without a block in small systems.
  // us at twojmax 8 with 1 / 2 / 3 atoms per block: FP64 250 atoms 11.4 / 12.5 /
  // 15.2, 300: 15.1 / 12.7 / 15.2, 2000: 51 / 34 / 39, 16 000: 348 / 223 / 272;
  // mixed 250 atoms 9.4 / 9.5 / 11.1, 300: 11.8 / 9.6 / 11.1, 1024: 18.4 / 13.8 /
  // 15.2, 1620: 27.4 / 20.6 / 20.6, 1800: 30.1 / 20.8 / 20.1, 16 000: 214 / 128 / 107:
  // one while every atom can have a CU (256 of them), in FP32 three from six
  // atoms per CU on.  Twojmax 12, where a block fills a CU's LDS, with 1 / 2 / 4:
  // FP64 250 atoms 54 / 58, 300: 95 / 59, 1024: 204 / 139; mixed 250 atoms 34 / 32 /
  // 54, 300: 54 / 33 / 54, 504: 62 / 42 / 57, 588: 81 / 63 / 58, 1024: 116 / 78 / 69:
  // in FP32 four once blocks of two no longer have a CU each.
  auto launch = [&](auto jc, auto ac) -> emd_status {
    constexpr int J = jc, AT = ac;
    EMD_LAUNCH(ctx, "snap_y", (k_snap_yflat<T, J, AT>), (n + AT - 1) / AT, yf_threads<J>(), 0,
               sn->t.nu, sn->t.ny, sn->yf_nch, sn->yf_codes, w, sn->yf_meta, sn->yf_rstart, n, ur,
               ui, yr, yi);
    return EMD_OK;
  };
  using J8 = std::integral_constant<int, SNAP_MAXJ>;
  using J12 = std::integral_constant<int, SNAP_JBIG>;
  using A1 = std::integral_constant<int, 1>;
  using A2 = std::integral_constant<int, 2>;
  constexpr bool f32 = std::is_same<T, float>::value;
  const int cus = ctx->num_cu;
  if (sn->t.twojmax > SNAP_MAXJ) {
    if (n <= cus) return launch(J12{}, A1{});
    if (f32 && n > 2 * cus) return launch(J12{}, std::integral_constant<int, f32 ? 4 : 2>{});
    return launch(J12{}, A2{});
  }
  if (n <= cus) return launch(J8{}, A1{});
  if (f32 && n > 6 * cus) return launch(J8{}, std::integral_constant<int, f32 ? 3 : 2>{});
  return launch(J8{}, A2{});
}

// F_ij for every (atom, neighbour)
template <class T, class TF>
static emd_status launch_fij(emd_ctx *ctx, emd_snap *sn, int n, const T *yr, const T *yi,
                             TF *f) {
  const snap_par<T> *par = (const snap_par<T> *)sn->par;
  const int nb = RG_WAVES * (sn->t.twojmax <= SNAP_MAXJ ? rg<SNAP_MAXJ>::NB : rg<SNAP_JBIG>::NB);
  const dim3 grid(n, (sn->cap_maxn + nb - 1) / nb);
  if (sn->t.twojmax <= SNAP_MAXJ)
    EMD_LAUNCH(ctx, "snap_fij", (k_snap_fij_rev<T, TF, SNAP_MAXJ>), grid, 64 * RG_WAVES, 0, sn->t,
               sn->rg_map_d, sn->nin, sn->nj, sn->nr, par, sn->fdv, sn->cap_maxn, n, yr, yi, f);
  else
    EMD_LAUNCH(ctx, "snap_fij", (k_snap_fij_rev<T, TF, SNAP_JBIG>), grid, 64 * RG_WAVES, 0, sn->t,
               sn->rg_map_d, sn->nin, sn->nj, sn->nr, par, sn->fdv, sn->cap_maxn, n, yr, yi, f);
  return EMD_OK;
}

// with static geometry on: are the compaction, neighbour parameters and U_tot
// in precision prec those of this system and list?
static bool snap_geom_cached(const emd_snap *sn, const emd_system *s, const emd_neigh *nl,
                             int prec) {
  return sn->geom_static && sn->t.twojmax <= SNAP_MAXJ && sn->geom_prec == prec && sn->par_prec == prec &&
         sn->geom_n == s->n_local && sn->geom_x == s->x && sn->geom_ent == nl->entries;
}

static void snap_geom_record(emd_snap *sn, const emd_system *s, const emd_neigh *nl, int prec) {
  if (!sn->geom_static) return;
  sn->geom_prec = prec;
  sn->geom_n = s->n_local;
  sn->geom_x = s->x;
  sn->geom_ent = nl->entries;
}

static emd_status snap_force(emd_ctx *ctx, emd_system *s, const emd_neigh *nl, emd_snap *sn,
                             int precision, bool zero) {
  if (!ctx || !s || !nl || !sn) return EMD_ERR_ARG;
  EMD_ARG(ctx, nl->n == s->n_local, "neighbour list does not match the system");
  const int n = s->n_local;
  if (n <= 0) return zero ? emd_force_zero(ctx, s, precision) : EMD_OK;
  const int prec = precision == EMD_MIXED ? EMD_MIXED : EMD_FP64;
  // compaction, neighbour parameters and U_tot in one launch (or, with
  // static geometry, those of the previous call), then Y
  if (snap_geom_cached(sn, s, nl, prec)) {
    if (zero) EMD_TRY(emd_force_zero(ctx, s, prec));
  } else {
    EMD_TRY(snap_neigh_ui(ctx, s, nl, sn, zero ? prec : -1, prec));
    snap_geom_record(sn, s, nl, prec);
  }
  if (precision == EMD_MIXED) EMD_TRY(snap_y<float>(ctx, sn, n));
  else EMD_TRY(snap_y<double>(ctx, sn, n));
  if (precision == EMD_MIXED) {
    EMD_TRY((launch_fij<float, float>(ctx, sn, n, (const float *)sn->y_r,
                                      (const float *)sn->y_i, s->f32)));
  } else {
    EMD_TRY((launch_fij<double, double>(ctx, sn, n, (const double *)sn->y_r,
                                        (const double *)sn->y_i, s->f)));
  }
  return EMD_OK;
}

extern "C" emd_status emd_snap_force(emd_ctx *ctx, emd_system *s, const emd_neigh *nl,
                                     emd_snap *sn, int precision) {
  return snap_force(ctx, s, nl, sn, precision, false);
}

extern "C" emd_status emd_snap_force_zeroed(emd_ctx *ctx, emd_system *s, const emd_neigh *nl,
                                            emd_snap *sn, int precision) {
  return snap_force(ctx, s, nl, sn, precision, true);
}

extern "C" emd_status emd_snap_energy(emd_ctx *ctx, const emd_system *s, const emd_neigh *nl,
                                      emd_snap *sn, double *energy, double *eatom) {
  if (!ctx || !s || !nl || !sn || !energy) return EMD_ERR_ARG;
  const int n = s->n_local;
  *energy = 0.0;
  if (n <= 0) return EMD_OK;
  // the static geometry serves force and adjoint calls: an energy is that of
  // the positions as they are, and the compaction and U_tot are rewritten
  sn->geom_prec = -1;
  EMD_TRY(snap_neigh_ui(ctx, s, nl, sn, -1, EMD_FP64));
  EMD_TRY(snap_y<double>(ctx, sn, n));
  double *ea = eatom;
  if (!ea) {
    EMD_TRY(emd_ensure_int(ctx, (int **)&sn->eatom, &sn->cap_e, 2l * n));
    ea = sn->eatom;
  }
  double e0 = sn->beta[0];
  if (sn->bzeroflag)
    for (int k = 0; k < sn->ncoeff; k++)
      e0 -= sn->beta[k + 1] * sn->t.wself * sn->t.wself * sn->t.wself * (sn->idxj[3 * k + 2] + 1);
  EMD_LAUNCH(ctx, "snap_energy", k_snap_energy, emd_blocks(n, ENERGY_WAVES), 64 * ENERGY_WAVES, 0,
             sn->t.nu, sn->t.ny, sn->edot, e0, sn->t.rcut, sn->nin, sn->nr, sn->cap_maxn, n,
             (const double *)sn->u_r, (const double *)sn->u_i, (const double *)sn->y_r,
             (const double *)sn->y_i, ea);
  const emd_mail mail = emd_mail_next(ctx);
  EMD_LAUNCH(ctx, "snap_energy", k_snap_energy_sum, 1, 1024, 0, ea, n, mail);
  const int *got = nullptr;
  EMD_TRY(emd_mail_wait(ctx, mail, &got));
  memcpy(energy, got, sizeof(double));
  return EMD_OK;
}

// ====================================================== adjoint (dL/dbeta)
// F is affine in beta: F_ij = sum_J sum' Re(conj(dU_J) Y_J(beta)) + repulsion.
// For a cotangent g = dL/dF, sum_i g_i . dF_i/dbeta_k
//   = sum_i sum_J sum' Re(conj(W^i_J) dY^i_J/dbeta_k),
//   W^i_J = sum_{j in N(i)} w(ma,mb) sum_d (g_i - g_j)_d dU_J/dr_d
// (ghost j carries the cotangent of its owner), and dY_J/dbeta_k is the
// three-role combination of Z_{abJ}; so per triple (a,b,J) only
// S_{abJ} = sum_i sum' Re(conj(W^i_J) Z^i_{abJ}) is needed.

// W^i for every atom with the register-resident recursion:
//   W^i_J(e) = sum_{j in N(i)} w(e) [dsfac (g . u) U_J(e) + sfac dU_J(e)/dr . g],
// g = g_i - g_j (a ghost j carries its owner's cotangent): the derivative
// of sfac U along g.  Each lane carries sfac V and its derivative X (4 values
// per entry), whose recursions are linear: they start from sfac and dsfac (g.u),
//   X_j = conj(a) X_{j-1}(ma) - conj(b) X_{j-1}(ma-1)
//       + conj(da_g) sfac V_{j-1}(ma) - conj(db_g) sfac V_{j-1}(ma-1)
// with da_g = g . da/dr and db_g = g . db/dr, both rank one in u plus constants:
//   da_g = c1 (g.u) + i (c2 (g.u) - r0inv g_z),  db_g = c3 (g.u) + r0inv g_y
//                                                   + i (c4 (g.u) - r0inv g_x).
// One wavefront per atom, a group of lanes per neighbour; each lane sums its
// group's neighbours (in TS), the groups are added in FP64 in order:
// deterministic.
template <class T, class TS, int J>
__global__ void __launch_bounds__(64)
k_snap_w_rg(snap_dev_tables t, const rg_map *__restrict__ rgm, const int *__restrict__ nin,
            const int *__restrict__ nj, const snap_par<T> *__restrict__ par, int maxn, int n,
            const int *__restrict__ root, const double *__restrict__ g, double *__restrict__ w_r,
            double *__restrict__ w_i) {
  using R = rg<J>;
  __shared__ TS s_buf[rg_sum<J>::BUF];
  const int i = blockIdx.x;
  if (i >= n) return;
  const int l = threadIdx.x;
  const int gr = l / R::W, ma = l - gr * R::W;  // gr = NB only for idle lanes
  TS acc[R::SLOTS][2];
#pragma unroll
  for (int s = 0; s < R::SLOTS; s++) acc[s][0] = acc[s][1] = 0;
  const double gi0 = g[3 * (size_t)i], gi1 = g[3 * (size_t)i + 1], gi2 = g[3 * (size_t)i + 2];
  const int cnt = nin[i];
  for (int base = 0; base < cnt; base += R::NB) {
    const int jj = base + gr;
    const bool act = gr < R::NB && jj < cnt;
    const size_t o = (size_t)i * maxn + (act ? jj : base);
    const snap_par<T> pp = par[o];
    const int jn = nj[o];
    const int own_j = jn < n ? jn : root[jn - n];
    const T g0 = (T)(gi0 - g[3 * (size_t)own_j]);
    const T g1 = (T)(gi1 - g[3 * (size_t)own_j + 1]);
    const T g2 = (T)(gi2 - g[3 * (size_t)own_j + 2]);
    const T gu = g0 * pp.u[0] + g1 * pp.u[1] + g2 * pp.u[2];
    const T a_r = pp.a_r, a_i = pp.a_i, b_r = pp.b_r, b_i = pp.b_i;
    const T da_r = pp.c1 * gu, da_i = pp.c2 * gu - pp.r0inv * g2;
    const T db_r = pp.c3 * gu + pp.r0inv * g1, db_i = pp.c4 * gu - pp.r0inv * g0;
    const bool first = act && ma == 0;  // an idle group adds nothing
    T c[R::COLS][2], d[R::COLS][2];     // sfac V and X of (ma, mb)
#pragma unroll
    for (int mb = 0; mb < R::COLS; mb++) c[mb][0] = c[mb][1] = d[mb][0] = d[mb][1] = 0;
    c[0][0] = first ? pp.sfac : (T)0;
    d[0][0] = first ? pp.dsfac * gu : (T)0;
    acc[0][0] += (TS)d[0][0];
    rg_layers<1, J>([&](auto jc) {
      constexpr int j = jc;
      if (j > t.twojmax) return;
      // X first: it needs V_{j-1}
      T q[R::COLS][4];
#pragma unroll
      for (int mb = 0; 2 * mb < j; mb++) {
        q[mb][0] = lane_below(c[mb][0]);
        q[mb][1] = lane_below(c[mb][1]);
        q[mb][2] = lane_below(d[mb][0]);
        q[mb][3] = lane_below(d[mb][1]);
      }
#pragma unroll
      for (int mb = j / 2; mb >= 0; mb--) {
        const bool mid = 2 * mb == j;
        const int k = mid ? mb - 1 : mb;  // the middle column comes from the one beside it
        const T p0 = c[k][0], p1 = c[k][1], x0 = d[k][0], x1 = d[k][1];
        const T q0 = q[k][0], q1 = q[k][1], y0 = q[k][2], y1 = q[k][3];
        if (mid) {
          d[mb][0] = db_r * p0 - db_i * p1 + da_r * q0 - da_i * q1 + b_r * x0 - b_i * x1 +
                     a_r * y0 - a_i * y1;
          d[mb][1] = db_r * p1 + db_i * p0 + da_r * q1 + da_i * q0 + b_r * x1 + b_i * x0 +
                     a_r * y1 + a_i * y0;
          c[mb][0] = b_r * p0 - b_i * p1 + a_r * q0 - a_i * q1;
          c[mb][1] = b_r * p1 + b_i * p0 + a_r * q1 + a_i * q0;
        } else {
          d[mb][0] = da_r * p0 + da_i * p1 - db_r * q0 - db_i * q1 + a_r * x0 + a_i * x1 -
                     b_r * y0 - b_i * y1;
          d[mb][1] = da_r * p1 - da_i * p0 - db_r * q1 + db_i * q0 + a_r * x1 - a_i * x0 -
                     b_r * y1 + b_i * y0;
          c[mb][0] = a_r * p0 + a_i * p1 - b_r * q0 - b_i * q1;
          c[mb][1] = a_r * p1 - a_i * p0 - b_r * q1 + b_i * q0;
        }
      }
#pragma unroll
      for (int mb = 0; mb <= j / 2; mb++) {
        acc[rg_slot0(j) + mb][0] += (TS)d[mb][0];
        acc[rg_slot0(j) + mb][1] += (TS)d[mb][1];
      }
    });
  }
  rg_group_sum<double, J>(acc, l, s_buf, [&](int k, double vr, double vi) {
    const rg_map m = rgm[k];
    if (m.ey < 0) return;
    const double wgt = 0.5 * m.wq * m.norm;
    w_r[(size_t)i * t.ny + m.ey] = wgt * vr;
    w_i[(size_t)i * t.ny + m.ey] = wgt * vi;
  });
}

// S_{abJ} += sum' Re(conj(W^i_J) Z^i_{abJ}) over atoms (FP64 accumulation)
template <class T>
__global__ void __launch_bounds__(192)
k_snap_s(snap_dev_tables t, const double *__restrict__ cg, const stab_entry *__restrict__ stab,
         const int *__restrict__ sjstart, int ntrip, int n, const T *__restrict__ utot_r,
         const T *__restrict__ utot_i, const double *__restrict__ w_r,
         const double *__restrict__ w_i, double *__restrict__ S) {
  __shared__ T su_r[SNAP_NU_BIG], su_i[SNAP_NU_BIG];
  __shared__ double sS[SNAP_MAXT];
  const int i = blockIdx.x;
  if (i >= n) return;
  for (int k = threadIdx.x; k < t.nu; k += blockDim.x) {
    su_r[k] = utot_r[(size_t)i * t.nu + k];
    su_i[k] = utot_i[(size_t)i * t.nu + k];
  }
  for (int k = threadIdx.x; k < ntrip; k += blockDim.x) sS[k] = 0.0;
  __syncthreads();
  for (int e = threadIdx.x; e < t.ny; e += blockDim.x) {
    int J, ma, mb;
    y_entry(t, e, J, ma, mb);
    const double wr = w_r[(size_t)i * t.ny + e], wi = w_i[(size_t)i * t.ny + e];
    if (wr != 0.0 || wi != 0.0) {
      for (int q = sjstart[J]; q < sjstart[J + 1]; q++) {
        const stab_entry te = stab[q];
        const cplx<T> z = z_entry<T>(t, cg, su_r, su_i, te.a, te.b, J, te.cgoff, ma, mb);
        atomicAdd(&sS[te.tid], wr * (double)z.r + wi * (double)z.i);
      }
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < ntrip; k += blockDim.x) atomicAdd(&S[k], sS[k]);
}

// S_{abJ} from a stream of single products (twojmax <= 8): a term of entry
// e and key (a, b, J) adds cgw * Re(conj(W_e) U_a U_b) to S of its key (the
// double sum of k_snap_s, term by term).  Its codes address the
// same bank-shifted U_tot copies as k_snap_yflat; AT atoms per block share
// each term's loads, W of the chunk's entry is read once per chunk, a run of
// one key within a chunk is summed in a register and added to the block's
// LDS sums by one atomic, and the block stores its key sums to its row of
// part (k_snap_s_reduce adds the rows up: no global atomics on the few key
// addresses, and a fixed order).
template <class T, int J, int AT>
__global__ void __launch_bounds__(SF_THREADS)
k_snap_s_flat(int nu, int ny, int nch, const uint32_t *__restrict__ code,
              const unsigned short *__restrict__ key, const double *__restrict__ cgw,
              const unsigned short *__restrict__ centry, const unsigned short *__restrict__ keytid,
              int nkeys, int n, const T *__restrict__ utot_r, const T *__restrict__ utot_i,
              const double *__restrict__ w_r, const double *__restrict__ w_i,
              double *__restrict__ part) {
  using L = yf_layout<T, J>;
  static_assert(L::UBYTES % sizeof(cpair<T>) == 0, "copies aligned");
  constexpr int UP = L::UBYTES / sizeof(cpair<T>);
  constexpr int NY = snap_dim<J>::NY;
  __shared__ cpair<T> s_u[AT * UP];
  __shared__ double s_w[AT][2][NY];
  __shared__ double s_S[SNAP_MAXT];
  unsigned char *sb = reinterpret_cast<unsigned char *>(s_u);
  const int i0 = blockIdx.x * AT;
  if (i0 >= n) return;
  for (int a = 0; a < AT; a++) {
    const int i = i0 + a < n ? i0 + a : i0;
    unsigned char *ub = sb + a * L::UBYTES;
    for (int k = threadIdx.x; k < nu; k += SF_THREADS) {
      const T vr = utot_r[(size_t)i * nu + k], vi = utot_i[(size_t)i * nu + k];
#pragma unroll
      for (int c = 0; c < L::NCOPY; c++) {
        if (L::SOA) {
          reinterpret_cast<T *>(ub)[L::base(c) + k] = vr;
          reinterpret_cast<T *>(ub + L::IMB)[L::base(c) + k] = vi;
        } else {
          reinterpret_cast<cpair<T> *>(ub)[L::base(c) + k] = cpair<T>{vr, vi};
        }
      }
    }
    // the second atom of an odd-sized last block adds nothing
    for (int e = threadIdx.x; e < ny; e += SF_THREADS) {
      s_w[a][0][e] = i0 + a < n ? w_r[(size_t)i * ny + e] : 0.0;
      s_w[a][1][e] = i0 + a < n ? w_i[(size_t)i * ny + e] : 0.0;
    }
  }
  for (int k = threadIdx.x; k < nkeys; k += SF_THREADS) s_S[k] = 0.0;
  __syncthreads();
  for (int c = 0; c < nch; c++) {
    const int e = centry[(size_t)c * SF_THREADS + threadIdx.x];  // 0 for padding chunks
    double wr[AT], wi[AT];
#pragma unroll
    for (int a = 0; a < AT; a++) {
      wr[a] = s_w[a][0][e];
      wi[a] = s_w[a][1][e];
    }
    // a chunk's terms come in runs of one key (padding, weight 0, last):
    // each run is summed here and added to S once
    int run_key = key[(size_t)c * SF_CHUNK * SF_THREADS + threadIdx.x];
    double run = 0.0;
#pragma unroll 4
    for (int k = 0; k < SF_CHUNK; k++) {
      const size_t slot = ((size_t)c * SF_CHUNK + k) * SF_THREADS + threadIdx.x;
      const uint32_t cc = code[slot];
      const double cw = cgw[slot];
      const int kk = key[slot];
      if (kk != run_key && cw != 0.0) {
        atomicAdd(&s_S[run_key], run);
        run = 0.0;
        run_key = kk;
      }
      double v = 0.0;
#pragma unroll
      for (int a = 0; a < AT; a++) {
        const unsigned char *ub = sb + a * L::UBYTES;
        const cpair<T> u1 = yf_u<T, J>(ub, cc & 0xFFFFu), u2 = yf_u<T, J>(ub, cc >> 16);
        const T pr = u1.r * u2.r - u1.i * u2.i;
        const T pi = u1.r * u2.i + u1.i * u2.r;
        v += wr[a] * (double)pr + wi[a] * (double)pi;
      }
      run += cw * v;
    }
    atomicAdd(&s_S[run_key], run);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < nkeys; k += SF_THREADS) part[(size_t)blockIdx.x * nkeys + k] = s_S[k];
}

// S of each key: its column of the per-block sums, added by one block in a
// fixed order (strided partial sums, then a tree)
__global__ void __launch_bounds__(256)
k_snap_s_reduce(const double *__restrict__ part, int nrows, int nkeys,
                const unsigned short *__restrict__ keytid, double *__restrict__ S) {
  __shared__ double s_v[256];
  const int k = blockIdx.x;
  double v = 0.0;
  for (int r = threadIdx.x; r < nrows; r += 256) v += part[(size_t)r * nkeys + k];
  s_v[threadIdx.x] = v;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s_v[threadIdx.x] += s_v[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) S[keytid[k]] += s_v[0];  // one key per block: no other writer
}

// sum over atoms of every bispectrum component B_k (dE/dbeta_k), FP64
__global__ void __launch_bounds__(256)
k_snap_bsum(snap_dev_tables t, const double *__restrict__ cg, const etab_entry *__restrict__ etab,
            int ne, int bzero, int n, const double *__restrict__ utot_r,
            const double *__restrict__ utot_i, double *__restrict__ bsum,
            double *__restrict__ brow) {
  __shared__ double su_r[SNAP_NU_BIG], su_i[SNAP_NU_BIG];
  __shared__ double sB[SNAP_MAXC];
  const int i = blockIdx.x;
  if (i >= n) return;
  for (int k = threadIdx.x; k < t.nu; k += blockDim.x) {
    su_r[k] = utot_r[(size_t)i * t.nu + k];
    su_i[k] = utot_i[(size_t)i * t.nu + k];
  }
  for (int k = threadIdx.x; k < ne; k += blockDim.x) sB[k] = 0.0;
  __syncthreads();
  for (int k = 0; k < ne; k++) {
    const etab_entry te = etab[k];
    const int J = te.j;
    const int nyj = t.ystart[J + 1] - t.ystart[J];
    for (int q = threadIdx.x; q < nyj; q += blockDim.x) {
      const int mb = q / (J + 1), ma = q - mb * (J + 1);
      double wgt = 1.0;
      if (2 * mb == J) wgt = (ma < mb) ? 1.0 : ((ma == mb) ? 0.5 : 0.0);
      if (wgt == 0.0) continue;
      const cplx<double> z = z_entry<double>(t, cg, su_r, su_i, te.j1, te.j2, J, te.cgoff, ma, mb);
      const int u = t.ustart[J] + ma * (J + 1) + mb;
      atomicAdd(&sB[k], 2.0 * wgt * (su_r[u] * z.r + su_i[u] * z.i));
    }
  }
  __syncthreads();
  // the atom's B_k into row i of brow, or added into bsum
  for (int k = threadIdx.x; k < ne; k += blockDim.x) {
    double b = sB[k];
    if (bzero) b -= t.wself * t.wself * t.wself * (etab[k].j + 1);
    if (brow) brow[(size_t)i * ne + k] = b;
    else atomicAdd(&bsum[k], b);
  }
}

__global__ void k_zero_d(double *p, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = 0.0;
}

template <class T>
static emd_status snap_adjoint_impl(emd_ctx *ctx, const emd_system *s, const emd_halo *h,
                                    emd_snap *sn, const double *g, double *S) {
  const int n = s->n_local;
  // the neighbour parameters (in T) and U_tot came with the compaction
  const snap_par<T> *par = (const snap_par<T> *)sn->par;
  if (sn->t.twojmax <= SNAP_MAXJ)
    EMD_LAUNCH(ctx, "snap_adjoint_w", (k_snap_w_rg<T, T, SNAP_MAXJ>), n, 64, 0, sn->t, sn->rg_map_d,
               sn->nin, sn->nj, par, sn->cap_maxn, n, h ? h->root : nullptr, g, sn->w_r, sn->w_i);
  else
    EMD_LAUNCH(ctx, "snap_adjoint_w", (k_snap_w_rg<T, double, SNAP_JBIG>), n, 64, 0, sn->t,
               sn->rg_map_d, sn->nin, sn->nj, par, sn->cap_maxn, n, h ? h->root : nullptr, g,
               sn->w_r, sn->w_i);
  const int ntrip = (int)sn->tid.size();
  if (sn->t.twojmax <= SNAP_MAXJ) {
    const int nb = (n + 1) / 2, nkeys = (int)sn->yf_keys.size();
    EMD_TRY(emd_ensure(ctx, (void **)&sn->s_part, &sn->cap_spart,
                       (size_t)nb * nkeys * sizeof(double)));
    EMD_LAUNCH(ctx, "snap_adjoint_s", (k_snap_s_flat<T, SNAP_MAXJ, 2>), nb, SF_THREADS, 0,
               sn->t.nu, sn->t.ny, sn->sf_nch, sn->sf_code, sn->sf_key, sn->sf_cgw, sn->sf_centry,
               sn->yf_keytid, nkeys, n, (const T *)sn->u_r, (const T *)sn->u_i, sn->w_r, sn->w_i,
               sn->s_part);
    if (nkeys > 0)
      EMD_LAUNCH(ctx, "snap_adjoint_s", k_snap_s_reduce, nkeys, 256, 0, sn->s_part, nb, nkeys,
                 sn->yf_keytid, S);
  } else {
    EMD_LAUNCH(ctx, "snap_adjoint_s", k_snap_s<T>, n, 192, 0, sn->t, sn->cg, sn->stab,
               (const int *)(sn->sbuf + SNAP_MAXT + SNAP_MAXC), ntrip, n, (const T *)sn->u_r,
               (const T *)sn->u_i, sn->w_r, sn->w_i, S);
  }
  return EMD_OK;
}

extern "C" emd_status emd_snap_adjoint_beta(emd_ctx *ctx, const emd_system *s, const emd_neigh *nl,
                                            const emd_halo *h, emd_snap *sn, const double *dLdF,
                                            double dLdE, int precision, double *dLdbeta) {
  if (!ctx || !s || !nl || !sn || !dLdF || !dLdbeta) return EMD_ERR_ARG;
  const int n = s->n_local;
  for (int k = 0; k <= sn->ncoeff; k++) dLdbeta[k] = 0.0;
  if (n <= 0) return EMD_OK;
  EMD_ARG(ctx, s->n_ghost == 0 || (h && h->root && h->n_ghost == s->n_ghost),
          "ghost atoms need the halo (owner of each ghost)");
  const int aprec = precision == EMD_MIXED ? EMD_MIXED : EMD_FP64;
  if (!snap_geom_cached(sn, s, nl, aprec)) {
    EMD_TRY(snap_neigh_ui(ctx, s, nl, sn, -1, aprec));
    snap_geom_record(sn, s, nl, aprec);
  }
  EMD_TRY(emd_ensure(ctx, (void **)&sn->w_r, &sn->cap_w, (size_t)n * sn->t.ny * sizeof(double)));
  EMD_TRY(emd_ensure(ctx, (void **)&sn->w_i, &sn->cap_wi, (size_t)n * sn->t.ny * sizeof(double)));
  // sbuf: S[SNAP_MAXT] | Bsum[SNAP_MAXC] | sjstart ints (twojmax + 2 of them)
  constexpr int SB_D = SNAP_MAXT + SNAP_MAXC;
  EMD_TRY(emd_ensure(ctx, (void **)&sn->sbuf, &sn->cap_s, (SB_D + SNAP_JBIG + 2) * sizeof(double)));
  double *S = sn->sbuf, *B = sn->sbuf + SNAP_MAXT;
  EMD_HIP(ctx, hipMemcpyAsync(sn->sbuf + SB_D, sn->sjstart.data(),
                              sn->sjstart.size() * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  EMD_LAUNCH(ctx, "snap_adjoint_s", k_zero_d, emd_blocks(SB_D, 256), 256, 0, sn->sbuf, SB_D);
  if (precision == EMD_MIXED) EMD_TRY(snap_adjoint_impl<float>(ctx, s, h, sn, dLdF, S));
  else EMD_TRY(snap_adjoint_impl<double>(ctx, s, h, sn, dLdF, S));
  // dE/dbeta_k = sum_i B_k^i in FP64
  if (dLdE != 0.0) {
    sn->geom_prec = -1;  // U_tot is rewritten in FP64
    EMD_TRY(launch_ui(ctx, sn, n));
    EMD_LAUNCH(ctx, "snap_adjoint_bsum", k_snap_bsum, n, 256, 0, sn->t, sn->cg, sn->etab,
               sn->ncoeff, sn->bzeroflag, n, (const double *)sn->u_r, (const double *)sn->u_i, B,
               nullptr);
  }
  std::vector<double> hS(SB_D);
  EMD_HIP(ctx, hipMemcpyAsync(hS.data(), sn->sbuf, hS.size() * sizeof(double),
                              hipMemcpyDeviceToHost, ctx->stream));
  EMD_TRY(emd_wait(ctx));
  dLdbeta[0] = dLdE * n;
  for (int k = 0; k < sn->ncoeff; k++) {
    const int j1 = sn->idxj[3 * k], j2 = sn->idxj[3 * k + 1], j = sn->idxj[3 * k + 2];
    const double s1 = hS[sn->tid.at(std::make_tuple(std::max(j1, j2), std::min(j1, j2), j))];
    const double s2 = hS[sn->tid.at(std::make_tuple(std::max(j, j2), std::min(j, j2), j1))];
    const double s3 = hS[sn->tid.at(std::make_tuple(std::max(j1, j), std::min(j1, j), j2))];
    dLdbeta[k + 1] = 2.0 * s1 + 2.0 * (j + 1) / (j1 + 1.0) * s2 + 2.0 * (j + 1) / (j2 + 1.0) * s3 +
                     dLdE * hS[SNAP_MAXT + k];
  }
  return EMD_OK;
}

extern "C" emd_status emd_snap_descriptors(emd_ctx *ctx, const emd_system *s, const emd_neigh *nl,
                                           emd_snap *sn, double *B) {
  if (!ctx || !s || !nl || !sn || !B) return EMD_ERR_ARG;
  const int n = s->n_local;
  if (n <= 0) return EMD_OK;
  sn->geom_prec = -1;  // the compaction and U_tot are rewritten
  EMD_TRY(snap_neigh_ui(ctx, s, nl, sn, -1, EMD_FP64));
  EMD_LAUNCH(ctx, "snap_descriptors", k_snap_bsum, n, 256, 0, sn->t, sn->cg, sn->etab,
             sn->ncoeff, sn->bzeroflag, n, (const double *)sn->u_r, (const double *)sn->u_i,
             nullptr, B);
  return EMD_OK;
}
