// Batched kernels outside the channel context, on caller-owned device
// arrays:
//   k_cn_solve   complex tridiagonal systems of the Crank-Nicolson form
//                (channel.f:914-963) with per-system coefficients, the work
//                of THOMAS_FORWARD/BACKWARD_COMPLEX_MPI (mpi.f:708-865) on
//                many systems at once;
//   k_fft512_*   2-D real transforms of 512 x 512 planes in the directions
//                and normalisation of FFT_XZ_TO_FOURIER/PHYSICAL
//                (mpi.f:1477-1606): a real-to-complex x pass and a complex z
//                pass, full spectra (no de-aliasing truncation).
// FP64 (double2) or FP32 (float2) storage and arithmetic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "dh_fft_dev.h"

namespace dh {

// ---------------------------------------------------------------------------
// Batched Crank-Nicolson solve.  System s, row j (0..ny-1):
//   a_j x_{j-1} + b_j x_j + c_j x_{j+1} = d_j,
//   a_j = -alpha_s sl_j, c_j = -alpha_s su_j, b_j = 1 + alpha_s (sl_j + su_j),
// the rows of channel.f:914-963 with alpha_s = NU T1 / h^2 and sl, su the
// metric factors h^2/(DY(J) DYF(J)), h^2/(DY(J+1) DYF(J)); sl = su = 0 gives
// an identity (Dirichlet) row.  The couplings a_0 and c_{ny-1} reach outside
// the system and are dropped, as the reference's sweeps never read them.
// Layout [row][system], systems fastest.
//
// A block of four waves solves 256/SEG systems, SEG lanes each: wave w, lane
// (256/SEG) p + s holds segment w SEG/4 + p of system s, so that a wave's
// access to one row of each of its segments is whole cache lines (128 B per
// segment for SEG = 32 in FP64).  A lane holds rows [R p', R p' + R) of its
// system, p' its segment, in registers (rows at or beyond ny are identity
// rows with zero right-hand side, which leave the others alone) and
// eliminates them locally, Thomas on the segment with its outer couplings
// dropped, so that
//   x_r = y_r - v_r X_L - w_r X_R,
// X_L, X_R the solution just outside the segment (the partition or SPIKE
// method): y = T^-1 d, v = T^-1 a_0 e_0, w = T^-1 c_{R-1} e_{R-1}.  The first
// and last rows of the segments give a 2 x 2 block-tridiagonal system over
// the interfaces, reduced cyclically across the wave's segments and then
// joined over the four waves through LDS.  Each lane then sweeps its rows
// again with the boundary terms moved to the right-hand side.  The
// forward-swept right-hand side, c/pivot and 1/pivot stay in registers
// between the sweeps (4 reals per row); the spike's forward values are
// formed again when needed.  Loads and stores are the right-hand side and
// the solution only (the diagonals come from alpha and the row tables): 32
// bytes per row in FP64.
//
// What bounds it: in FP64 memory (257 rows of 131584 systems, 1.08 GB, in
// 0.252 ms: 4.3 TB/s, where a plain copy of that size reaches 4.9), in FP32
// (0.197 ms, 2.8 TB/s) and below some 10^4 systems the chain of each lane's
// sweeps.  With one lane per system for the interfaces (31 dependent
// eliminations while 31 lanes wait) and 32 B row segments per wave it took
// 0.481 and 0.274 ms; the cyclic reduction alone took FP64 to 0.284, row
// tables that need no tests to 0.271, whole cache lines per wave the rest.
// ---------------------------------------------------------------------------
constexpr int kCnThreads = 256;
constexpr int kCnRows = 9;  // rows per lane: 36 + 36 registers of a segment in FP64, three waves per SIMD
constexpr int kCnMaxNy = 32 * kCnRows;
constexpr int cn_systems(int seg) { return 256 / seg; }  // systems per block

// SEG segments (lanes) per system: the fewest of 4, 8, 16, 32 whose 9 rows
// per lane hold ny, so that short systems do not pay for identity rows (60
// rows of 99999 systems: 44 us with 8 segments, 64 with 16; 30 rows of 90001
// in FP32: 12 us with 4, 67 with 16 segments before).
template <int R, int SEG, class C>
__device__ __forceinline__ void cn_solve_block(const double *__restrict__ alpha, const C *__restrict__ rhs,
                                              C *__restrict__ x, int ny, long long nsys, const Sc<C> *tab, Sc<C> *xch) {
  using S = Sc<C>;
  constexpr int kRows = SEG * R, kCnSys = cn_systems(SEG), kCnSeg = 64 / kCnSys;  // systems and segments per wave
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int p = lane / kCnSys, sw = lane % kCnSys;
  // a block's row segment is one or two whole cache lines in FP64 (half of
  // that in FP32) only where nsys keeps it aligned: blocks that share a line
  // share an L2
  const long long sys = (long long)xcd_range_block() * kCnSys + sw;
  const bool live = sys < nsys;
  const long long sysc = live ? sys : nsys - 1;  // loads of idle lanes stay in bounds
  const int r0 = (w * kCnSeg + p) * R;
  const S al = S(alpha[sysc]);
  const S *ta = tab + r0, *tc = ta + kRows, *tb = tc + kRows;
  auto coef = [&](int r, S &a, S &b, S &c) {
    a = -al * ta[r];
    c = -al * tc[r];
    b = S(1) + al * tb[r];
  };

  C d[R];
  {
    // rows at stride nsys from the segment's first: the per-row offsets are
    // multiples of a scalar, so no per-row address stays live in registers
    const C *rp = rhs + (long long)r0 * nsys + sysc;
#pragma unroll
    for (int r = 0; r < R; ++r) d[r] = (r0 + r < ny) ? rp[(long long)r * nsys] : mkc<C>(S(0), S(0));
  }
  // forward: cp_r = c_r / piv_r, d'_r; the left spike v'_r = -a_r v'_{r-1} / piv_r
  // (v'_0 = a_0 / piv_0) is carried only to its last value
  S cp[R], ip[R];  // c_r / piv_r and 1 / piv_r
  S a0 = S(0), vlast = S(0);
  {
    S cprev = S(0), vprev = S(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S a, b, c;
      coef(r, a, b, c);
      if (r == 0) a0 = a;
      const S piv = (r == 0) ? b : b - a * cprev;
      const S inv = S(1) / piv;
      ip[r] = inv;
      cp[r] = c * inv;
      if (r > 0) d[r] = mkc<C>(d[r].x - a * d[r - 1].x, d[r].y - a * d[r - 1].y);
      d[r] = mkc<C>(d[r].x * inv, d[r].y * inv);
      vprev = ((r == 0) ? a : -a * vprev) * inv;
      cprev = cp[r];
    }
    vlast = vprev;
  }
  // first-row values: y_0 and w_0 by the backward recurrences (no storage),
  // v_0 = a_0 (T^-1)_00 = a_0 / q_0 with q the pivots of an elimination from
  // the bottom: q_{R-1} = b_{R-1}, q_r = b_r - c_r a_{r+1} / q_{r+1} (formed
  // from the top's pivots instead, without these divisions, v_0 raised the
  // FP32 solution's error by 3%)
  // (the empty asm makes every sweep read its row tables from LDS again
  // rather than keep the previous sweep's coefficients in registers)
  asm volatile("" ::: "memory");
  C yf, yl = d[R - 1];
  S wf, wl = cp[R - 1], vf, vl = vlast;
  {
    C yy = d[R - 1];
    S ww = cp[R - 1], q, anext, c;
    coef(R - 1, anext, q, c);
#pragma unroll
    for (int r = R - 2; r >= 0; --r) {
      S a, b;
      coef(r, a, b, c);
      yy = mkc<C>(d[r].x - cp[r] * yy.x, d[r].y - cp[r] * yy.y);
      ww = -cp[r] * ww;
      q = b - c * anext / q;
      anext = a;
    }
    yf = yy;
    wf = ww;
    vf = a0 / q;
  }
  // The segments' first and last values F_p, L_p satisfy
  //   F_p = yf - vf L_{p-s} - wf F_{p+s},   L_p = yl - vl L_{p-s} - wl F_{p+s}
  // with s = 1.  Each step eliminates a = L_{p-s} and b = F_{p+s} with the
  // equations of the lanes p - s (') and p + s (''):
  //   (1 - wl' vf) a - wl' wf b   = yl' - wl' yf   - vl' L_{p-2s}
  //   -vf'' vl a + (1 - vf'' wl) b = yf'' - vf'' yl - wf'' F_{p+2s}
  // which doubles s.  A neighbour outside the wave's segments stays an
  // unknown, the same one for every lane (the equations a = A, b = B: vl' =
  // -1, wf'' = -1), so after log2(segments per wave) steps with all lanes at
  // work F and L depend on X_l and X_r alone, the values just outside the
  // wave's segments.
#pragma unroll
  for (int s = 1; s < kCnSeg; s *= 2) {
    const int ds = kCnSys * s;
    const bool lo = p >= s, hi = p + s < kCnSeg;
    C yl1 = mkc<C>(__shfl_up(yl.x, ds), __shfl_up(yl.y, ds));
    S vl1 = __shfl_up(vl, ds), wl1 = __shfl_up(wl, ds);
    C yf2 = mkc<C>(__shfl_down(yf.x, ds), __shfl_down(yf.y, ds));
    S vf2 = __shfl_down(vf, ds), wf2 = __shfl_down(wf, ds);
    yl1 = mkc<C>(lo ? yl1.x : S(0), lo ? yl1.y : S(0));
    yf2 = mkc<C>(hi ? yf2.x : S(0), hi ? yf2.y : S(0));
    vl1 = lo ? vl1 : S(-1);
    wl1 = lo ? wl1 : S(0);
    vf2 = hi ? vf2 : S(0);
    wf2 = hi ? wf2 : S(-1);
    const S m00 = S(1) - wl1 * vf, m01 = -(wl1 * wf), m10 = -(vf2 * vl), m11 = S(1) - vf2 * wl;
    const S id = S(1) / (m00 * m11 - m01 * m10);
    // [a b] = (constant) - (A) L_{p-2s} - (B) F_{p+2s}
    const C ca = mkc<C>(yl1.x - wl1 * yf.x, yl1.y - wl1 * yf.y), cb = mkc<C>(yf2.x - vf2 * yl.x, yf2.y - vf2 * yl.y);
    const S i00 = m11 * id, i01 = -m01 * id, i10 = -m10 * id, i11 = m00 * id;
    const C ka = mkc<C>(i00 * ca.x + i01 * cb.x, i00 * ca.y + i01 * cb.y);
    const C kb = mkc<C>(i10 * ca.x + i11 * cb.x, i10 * ca.y + i11 * cb.y);
    const S aA = i00 * vl1, bA = i10 * vl1, aB = i01 * wf2, bB = i11 * wf2;
    yf = mkc<C>(yf.x - vf * ka.x - wf * kb.x, yf.y - vf * ka.y - wf * kb.y);
    yl = mkc<C>(yl.x - vl * ka.x - wl * kb.x, yl.y - vl * ka.y - wl * kb.y);
    const S nvf = -(vf * aA + wf * bA), nwf = -(vf * aB + wf * bB);
    const S nvl = -(vl * aA + wl * bA), nwl = -(vl * aB + wl * bB);
    vf = nvf;
    wf = nwf;
    vl = nvl;
    wl = nwl;
  }
  // The four waves' first and last values, joined the same way by every lane
  // for its system: P_i = last value of wave i, Q_i = first of wave i + 1,
  //   P_i + vl_i P_{i-1} + wl_i Q_i         = yl_i
  //   vf_{i+1} P_i + Q_i + wf_{i+1} Q_{i+1} = yf_{i+1}
  // with P_{-1} = Q_3 = 0 (no rows outside the system).
  constexpr int kW = kCnThreads / 64;
  if (p == 0) {
    S *q = xch + (w * kCnSys + sw) * 8;
    q[0] = yf.x; q[1] = yf.y; q[2] = vf; q[3] = wf;
  }
  if (p == kCnSeg - 1) {
    S *q = xch + (w * kCnSys + sw) * 8;
    q[4] = yl.x; q[5] = yl.y; q[6] = vl; q[7] = wl;
  }
  __syncthreads();
  C Xl = mkc<C>(S(0), S(0)), Xr = Xl;
  {
    S c0[kW - 1], c1[kW - 1];
    C r0v[kW - 1], r1v[kW - 1];
    S pc0 = S(0);
    C prP = mkc<C>(S(0), S(0));
#pragma unroll
    for (int i = 0; i < kW - 1; ++i) {
      const S *qi = xch + (i * kCnSys + sw) * 8, *qn = qi + kCnSys * 8;
      const C ylv = mkc<C>(qi[4], qi[5]), yfv = mkc<C>(qn[0], qn[1]);
      const S vli = qi[6], wli = qi[7], vfn = qn[2], wfn = qn[3];
      const S m01 = wli - vli * pc0;
      const S idet = S(1) / (S(1) - m01 * vfn);
      const C t0 = mkc<C>(ylv.x - vli * prP.x, ylv.y - vli * prP.y);
      c0[i] = -m01 * wfn * idet;
      c1[i] = wfn * idet;
      r0v[i] = mkc<C>((t0.x - m01 * yfv.x) * idet, (t0.y - m01 * yfv.y) * idet);
      r1v[i] = mkc<C>((yfv.x - vfn * t0.x) * idet, (yfv.y - vfn * t0.y) * idet);
      pc0 = c0[i];
      prP = r0v[i];
    }
    C qn = mkc<C>(S(0), S(0));
#pragma unroll
    for (int i = kW - 2; i >= 0; --i) {
      const C P = mkc<C>(r0v[i].x - c0[i] * qn.x, r0v[i].y - c0[i] * qn.y);
      qn = mkc<C>(r1v[i].x - c1[i] * qn.x, r1v[i].y - c1[i] * qn.y);
      if (w == i + 1) Xl = P;
      if (w == i) Xr = qn;
    }
  }
  // X_L = L_{p-1}, X_R = F_{p+1}, at the wave's ends X_l and X_r
  yf = mkc<C>(yf.x - vf * Xl.x - wf * Xr.x, yf.y - vf * Xl.y - wf * Xr.y);
  yl = mkc<C>(yl.x - vl * Xl.x - wl * Xr.x, yl.y - vl * Xl.y - wl * Xr.y);
  C XL = mkc<C>(__shfl_up(yl.x, kCnSys), __shfl_up(yl.y, kCnSys));
  C XR = mkc<C>(__shfl_down(yf.x, kCnSys), __shfl_down(yf.y, kCnSys));
  XL = mkc<C>(p > 0 ? XL.x : Xl.x, p > 0 ? XL.y : Xl.y);
  XR = mkc<C>(p < kCnSeg - 1 ? XR.x : Xr.x, p < kCnSeg - 1 ? XR.y : Xr.y);
  asm volatile("" ::: "memory");
  // the segment's system with the boundary terms on the right: forward-swept
  // d''_r = d'_r - X_L v'_r - X_R w'_r (w'_r = 0 below the last row, cp_{R-1}
  // there), then the backward sweep x_r = d''_r - cp_r x_{r+1}
  {
    S vprev = S(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S a, b, c;
      coef(r, a, b, c);
      vprev = ((r == 0) ? a : -a * vprev) * ip[r];
      d[r] = mkc<C>(d[r].x - vprev * XL.x, d[r].y - vprev * XL.y);
    }
    d[R - 1] = mkc<C>(d[R - 1].x - cp[R - 1] * XR.x, d[R - 1].y - cp[R - 1] * XR.y);
  }
#pragma unroll
  for (int r = R - 2; r >= 0; --r) d[r] = mkc<C>(d[r].x - cp[r] * d[r + 1].x, d[r].y - cp[r] * d[r + 1].y);
  if (!live) return;
  C *xp = x + (long long)r0 * nsys + sys;
  asm volatile("" : "+v"(xp));  // a fresh base: the loads' addresses are not kept for the stores
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r0 + r < ny) xp[(long long)r * nsys] = d[r];
}

template <int SEG, class C>
__global__ void __launch_bounds__(kCnThreads) k_cn_solve(const double *__restrict__ sl, const double *__restrict__ su,
                                                       const double *__restrict__ alpha, const C *__restrict__ rhs,
                                                       C *__restrict__ x, int ny, long long nsys) {
  using S = Sc<C>;
  // rows of the three coefficients over alpha: sl without the coupling of row
  // 0, su without that of row ny-1, and sl + su; zero rows (identity) from ny
  // to the segments' end, so that no sweep tests its row
  constexpr int kRows = SEG * kCnRows;
  __shared__ S tab[3 * kRows];
  __shared__ S xch[(kCnThreads / 64) * cn_systems(SEG) * 8];
  for (int j = threadIdx.x; j < kRows; j += blockDim.x) {
    const S l = j < ny ? S(sl[j]) : S(0), u = j < ny ? S(su[j]) : S(0);
    tab[j] = j == 0 ? S(0) : l;
    tab[kRows + j] = j == ny - 1 ? S(0) : u;
    tab[2 * kRows + j] = l + u;
  }
  __syncthreads();
  cn_solve_block<kCnRows, SEG, C>(alpha, rhs, x, ny, nsys, tab, xch);
}

// ---------------------------------------------------------------------------
// 512-point complex DFT, 512 = 8 x 8 x 8, over 64 lanes l with x_{l + 64 j}
// in v[j] (j < 8), ending with X_{l + 64 j} in v[j]:
//   an 8-point DFT over j, twiddle W512^{l k1};
//   transpose (lane l1 + 8 k1 takes the values of l = l1 + 8 l2), an
//   8-point DFT over l2, twiddle W64^{l1 k2a};
//   transpose (lane k1 + 8 k2a takes the values of l1), an 8-point DFT
//   over l1, giving X_{k1 + 8 k2a + 64 k2b} in v[k2b].
// The exchanges go through LDS slots (fft512_slot; every 64th slot is
// followed by a padding slot, without which the second transpose's reads,
// 64 slots apart, fall on one bank group).  tw holds exp(-2 pi i m/512),
// m < 512.
// ---------------------------------------------------------------------------
constexpr int kFftN = 512, kFftK = 257;
constexpr int kFftSlots = kFftN + 8;
__device__ __forceinline__ int fft512_slot(int i) { return i + (i >> 6); }

template <bool INV, class C>
__device__ __forceinline__ C tw_of(const C *tw, int m) {
  const C w = tw[m & 511];
  return INV ? cconj(w) : w;
}

// the three stages; put(i, v) and get(i) exchange slot i < 512 of the
// transform, sync1 orders the first transpose, sync2 the slots' reuse within
// the 8 lanes 8 k1 + (0..7), sync3 the second transpose
template <bool INV, class C, class Put, class Get, class S1, class S2, class S3>
__device__ __forceinline__ void fft512_stages(C (&v)[8], int l, const C *tw, Put put, Get get, S1 sync1, S2 sync2,
                                              S3 sync3) {
  dft_small<8, INV>(v);
#pragma unroll
  for (int k1 = 1; k1 < 8; ++k1) v[k1] = cmul(v[k1], tw_of<INV>(tw, l * k1));
#pragma unroll
  for (int k1 = 0; k1 < 8; ++k1) put(64 * k1 + l, v[k1]);
  sync1();
  {
    const int l1 = l & 7, k1 = l >> 3;
#pragma unroll
    for (int l2 = 0; l2 < 8; ++l2) v[l2] = get(64 * k1 + l1 + 8 * l2);
    dft_small<8, INV>(v);  // v[k2a]
#pragma unroll
    for (int k2a = 1; k2a < 8; ++k2a) v[k2a] = cmul(v[k2a], tw_of<INV>(tw, 8 * l1 * k2a));
    sync2();
#pragma unroll
    for (int k2a = 0; k2a < 8; ++k2a) put(64 * k1 + 8 * k2a + l1, v[k2a]);
  }
  sync3();
  {
    const int k1 = l & 7, k2a = l >> 3;
#pragma unroll
    for (int l1 = 0; l1 < 8; ++l1) v[l1] = get(64 * k1 + 8 * k2a + l1);
    dft_small<8, INV>(v);  // v[k2b] = X_{k1 + 8 k2a + 64 k2b} = X_{l + 64 k2b}
  }
}

// one transform per wave in the wave's own slots s[kFftSlots]
template <bool INV, class C>
__device__ __forceinline__ void fft512_wave(C (&v)[8], C *s, const C *tw) {
  fft512_stages<INV>(
      v, threadIdx.x & 63, tw, [&](int i, C x) { s[fft512_slot(i)] = x; }, [&](int i) { return s[fft512_slot(i)]; },
      [] { wave_lds_sync(); }, [] { wave_lds_sync(); }, [] { wave_lds_sync(); });
  wave_lds_sync();
}

// x pass, forward: two rows z, z+1 of a plane per wave as one complex
// transform of x_n + i y_n; X_k = (Z_k + conj Z_{512-k})/2, Y_k = (Z_k -
// conj Z_{512-k})/(2i), k = 0..256, each divided by NX = 512 (mpi.f:1490-1500
// scales by 1/NX; a power of two, so a multiplication).  phys
// [plane][512][512], four [plane][512][257].
template <class C>
__global__ void __launch_bounds__(256) k_fft512_rows_fwd(const Sc<C> *__restrict__ phys, C *__restrict__ four,
                                                       const C *__restrict__ tw, long long np) {
  using S = Sc<C>;
  __shared__ C sm[4][kFftSlots];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long long pair = (long long)blockIdx.x * 4 + w;  // rows 2 pair, 2 pair + 1 of all planes' rows
  if (pair >= np * (kFftN / 2)) return;                  // whole waves exit together
  const S *ra = phys + 2 * pair * kFftN, *rb = ra + kFftN;
  C v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = mkc<C>(ra[lane + 64 * j], rb[lane + 64 * j]);
  fft512_wave<false>(v, sm[w], tw);
  // Z_k is this lane's v[j], k = lane + 64 j <= 256; Z_{512-k} comes from
  // slots 0 and 256..511
  if (lane == 0) sm[w][0] = v[0];
#pragma unroll
  for (int j = 4; j < 8; ++j) sm[w][fft512_slot(lane + 64 * j)] = v[j];
  wave_lds_sync();
  C *oa = four + 2 * pair * kFftK, *ob = oa + kFftK;
  const S h = S(0.5 / kFftN);
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const int k = lane + 64 * j;
    if (k <= kFftN / 2) {
      const C zk = v[j], zm = sm[w][fft512_slot((kFftN - k) & (kFftN - 1))];
      oa[k] = mkc<C>(h * (zk.x + zm.x), h * (zk.y - zm.y));
      ob[k] = mkc<C>(h * (zk.y + zm.y), h * (zm.x - zk.x));
    }
  }
}

// A value of type C at a real's alignment: the caller's physical planes are
// arrays of reals (the wide load and store need 4-byte alignment only).
template <class C>
using AtReal __attribute__((aligned(sizeof(Sc<C>)))) = C;

// x pass, inverse (the c2r of mpi.f:1600-1604, unnormalised): rows
// z, z+1 of the half spectra X, Y to x_n + i y_n = sum_k (X_k + i Y_k) e^{+2
// pi i nk/512}, with X_{512-k} = conj X_k and the imaginary parts of X_0,
// X_256 ignored as a c2r ignores them.  A row's 512 reals hold its X_k, k =
// 1..255, as 256 complex values with (Re X_0, Re X_256) in the first, as the
// z pass leaves them.  It runs in place (in == phys; a wave reads its two rows
// before it writes them) or from planes elsewhere.
template <class C>
__global__ void __launch_bounds__(256) k_fft512_rows_inv(const Sc<C> *in, Sc<C> *phys, const C *__restrict__ tw,
                                                       long long np) {
  using S = Sc<C>;
  __shared__ C sm[4][kFftSlots];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long long pair = (long long)blockIdx.x * 4 + w;
  if (pair >= np * (kFftN / 2)) return;
  S *oa = phys + 2 * pair * kFftN, *ob = oa + kFftN;
  const AtReal<C> *ia = reinterpret_cast<const AtReal<C> *>(in + 2 * pair * kFftN), *ib = ia + kFftN / 2;
  // Z_k = X_k + i Y_k for this lane's k = lane + 64 j < 256, and its mirror
  // Z_{512-k} = conj X_k + i conj Y_k through LDS to the lane that holds it
  // (each coefficient read once); Z_256 is lane 0's v[4]
  C v[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int k = lane + 64 * j;
    C X = ia[k], Y = ib[k];
    if (k == 0) {
      sm[w][fft512_slot(kFftN / 2)] = mkc<C>(X.y, Y.y);
      X.y = Y.y = S(0);
    }
    v[j] = mkc<C>(X.x - Y.y, X.y + Y.x);
    if (k != 0) sm[w][fft512_slot(kFftN - k)] = mkc<C>(X.x + Y.y, Y.x - X.y);
  }
  wave_lds_sync();
#pragma unroll
  for (int j = 4; j < 8; ++j) v[j] = sm[w][fft512_slot(lane + 64 * j)];
  wave_lds_sync();
  fft512_wave<true>(v, sm[w], tw);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    oa[lane + 64 * j] = v[j].x;
    ob[lane + 64 * j] = v[j].y;
  }
}

// z pass: the columns (plane, kx) of [plane][512][257] in one sequence, CT
// consecutive ones per block of 64 CT threads, thread CT l + c lane l of
// column c's transform.  Loads and stores go between memory and the first
// and last stage's registers, CT columns (128 B) side by side per row; LDS
// holds the two exchanges only, [slot][CT].  Forward divides by NZ = 512
// (mpi.f:1529-1531, a multiplication by 2^-9) and runs in place (a column is
// read before any of it is written); inverse is unnormalised and leaves the
// rows of k_fft512_rows_inv in the physical planes, which needs no memory of
// its own between the passes.
//
// What bounds it and the row pass: memory.  257 FP64 planes (1.08 GB in and
// out per pass) take 0.24 ms forward per pass, 4.5 TB/s where a plain copy of
// that size reaches 4.9, and 0.43 / 0.50 ms for the whole forward / inverse
// transform; 0.82 / 0.78 ms with the tile filled and drained around three
// exchanges and 16 planes per launch pair.  Keeping the planes between the
// passes in the last-level cache, 16 to 128 MB at a time, lost more to the
// launches' ends than it saved, also with one chunk's rows beside the
// columns of the chunk before.
template <bool INV, class C, int CT>
__global__ void __launch_bounds__(64 * CT) k_fft512_cols(const C *src, C *dst, Sc<C> *phys,
                                                               const C *__restrict__ tw, long long np) {
  using S = Sc<C>;
  extern __shared__ double2 smraw[];
  C *tile = reinterpret_cast<C *>(smraw);
  const int c = threadIdx.x % CT, l = threadIdx.x / CT;
  const long long col = (long long)xcd_range_block() * CT + c;
  const bool live = col < np * kFftK;
  const long long plane = live ? col / kFftK : 0;
  const int kx = live ? (int)(col - plane * kFftK) : 0;
  const C *in = src + (plane * kFftN + l) * kFftK + kx;
  C v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = live ? in[64 * j * kFftK] : mkc<C>(S(0), S(0));
  // the slots 64 k1 + (0..63) are written and read by lanes 8 k1 + (0..7),
  // one wave for CT = 8
  fft512_stages<INV>(
      v, l, tw, [&](int i, C x) { tile[fft512_slot(i) * CT + c] = x; },
      [&](int i) { return tile[fft512_slot(i) * CT + c]; }, [] { lds_barrier(); },
      [] {
        if constexpr (CT == 8)
          wave_lds_sync();
        else
          lds_barrier();
      },
      [] { lds_barrier(); });
  if (!live) return;
  if constexpr (INV) {
    S *row = phys + (plane * kFftN + l) * kFftN;
    const bool edge = kx == 0 || kx == kFftN / 2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      S *r = row + 64 * j * kFftN;
      if (edge)
        r[kx == 0 ? 0 : 1] = v[j].x;
      else
        *reinterpret_cast<AtReal<C> *>(r + 2 * kx) = v[j];
    }
  } else {
    C *out = dst + (plane * kFftN + l) * kFftK + kx;
    const S sc = S(1.0 / kFftN);
#pragma unroll
    for (int j = 0; j < 8; ++j) out[64 * j * kFftK] = mkc<C>(sc * v[j].x, sc * v[j].y);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {
// Twiddles exp(-2 pi i m/512), m < 512, in file-scope device arrays (one
// copy per device), filled from the host at the first call on each device.
__device__ double2 g_tw64_dev[kFftN];
__device__ float2 g_tw32_dev[kFftN];

std::mutex g_mu;
const void *g_tw64[64] = {nullptr}, *g_tw32[64] = {nullptr};  // their addresses, per device

// the twiddle tables of the current device (computed in long double and
// rounded once; no device memory is allocated)
hipError_t twiddles(bool fp32, const void **out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_tw64[dev]) {
    double2 h64[kFftN];
    float2 h32[kFftN];
    for (int m = 0; m < kFftN; ++m) {
      const long double a = -2.0L * 3.141592653589793238462643383279502884L * (long double)m / (long double)kFftN;
      const long double cr = cosl(a), ci = sinl(a);
      h64[m] = make_double2((double)cr, (double)ci);
      h32[m] = make_float2((float)cr, (float)ci);
    }
    void *p64 = nullptr, *p32 = nullptr;
    if ((e = hipGetSymbolAddress(&p64, HIP_SYMBOL(g_tw64_dev))) != hipSuccess) return e;
    if ((e = hipGetSymbolAddress(&p32, HIP_SYMBOL(g_tw32_dev))) != hipSuccess) return e;
    if ((e = hipMemcpy(p64, h64, sizeof(h64), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(p32, h32, sizeof(h32), hipMemcpyHostToDevice)) != hipSuccess) return e;
    g_tw32[dev] = p32;
    g_tw64[dev] = p64;
  }
  *out = fp32 ? g_tw32[dev] : g_tw64[dev];
  return hipSuccess;
}

thread_local std::string g_err;
int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}
}  // namespace

// the column tile (66.6 KB) is beyond the default dynamic-LDS limit, which is
// raised per device, at the first call on it
hipError_t fft512_lds_limits() {
  static bool raised[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_mu);
  if (raised[dev]) return hipSuccess;
  const void *k[] = {(const void *)k_fft512_cols<false, double2, 8>, (const void *)k_fft512_cols<true, double2, 8>,
                     (const void *)k_fft512_cols<false, float2, 16>, (const void *)k_fft512_cols<true, float2, 16>};
  for (const void *f : k)
    if ((e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax)) != hipSuccess) return e;
  raised[dev] = true;
  return hipSuccess;
}

// planes per launch pair: all of them up to a grid's 2^32 threads
constexpr long long kFftChunk = 65536;

static unsigned fft512_row_blocks(long long np) { return (unsigned)((np * (kFftN / 2) + 3) / 4); }

template <bool INV, class C, int CT>
static void launch_fft512_cols_t(const C *src, C *dst, Sc<C> *phys, const C *tw, long long np, hipStream_t st) {
  const unsigned lds = kFftSlots * CT * sizeof(C);
  hipLaunchKernelGGL((k_fft512_cols<INV, C, CT>), dim3((unsigned)((np * kFftK + CT - 1) / CT)), dim3(64 * CT), lds, st,
                     src, dst, phys, tw, np);
}
template <bool INV, class C>
static void launch_fft512_cols(const C *src, C *dst, Sc<C> *phys, const C *tw, long long np, hipStream_t st) {
  // FP32: 16 columns make a cache line (257 planes forward 0.234 ms, 0.257
  // with 8); fewer planes take 8 per block, twice the blocks (5 planes 12.1
  // us against 13.4, 64 planes 56 against 57)
  if (sizeof(C) == sizeof(float2) && np >= 96)
    launch_fft512_cols_t<INV, C, sizeof(C) == sizeof(float2) ? 16 : 8>(src, dst, phys, tw, np, st);
  else
    launch_fft512_cols_t<INV, C, 8>(src, dst, phys, tw, np, st);
}

template <class C>
static hipError_t fft512_forward_t(const void *phys, void *four, long long nplanes, hipStream_t st, const C *tw) {
  for (long long p0 = 0; p0 < nplanes; p0 += kFftChunk) {
    const long long np = std::min(kFftChunk, nplanes - p0);
    C *fo = (C *)four + p0 * kFftN * kFftK;
    hipLaunchKernelGGL(k_fft512_rows_fwd<C>, dim3(fft512_row_blocks(np)), dim3(256), 0, st,
                       (const Sc<C> *)phys + p0 * kFftN * kFftN, fo, tw, np);
    launch_fft512_cols<false, C>(fo, fo, nullptr, tw, np, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// mid: where the planes lie between the passes, chunk of them (null: in phys)
template <class C>
static hipError_t fft512_inverse_t(const void *four, void *phys, long long nplanes, hipStream_t st, const C *tw,
                                   Sc<C> *mid, long long chunk) {
  for (long long p0 = 0; p0 < nplanes; p0 += chunk) {
    const long long np = std::min(chunk, nplanes - p0);
    Sc<C> *ph = (Sc<C> *)phys + p0 * kFftN * kFftN, *q = mid ? mid : ph;
    launch_fft512_cols<true, C>((const C *)four + p0 * kFftN * kFftK, nullptr, q, tw, np, st);
    hipLaunchKernelGGL(k_fft512_rows_inv<C>, dim3(fft512_row_blocks(np)), dim3(256), 0, st, q, ph, tw, np);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// An inverse whose phys shares memory with its four: the column pass must not
// write where other blocks still read, so the planes between the passes lie in
// a static array, kOverlapPlanes at a time (33.6 MB on each device the library
// runs on).  Calls on several streams take the array in turn; under capture,
// where an event from outside cannot be waited for, a graph's calls are in
// order with one another only.
constexpr long long kOverlapPlanes = 16;
__device__ __align__(256) double g_overlap_dev[kOverlapPlanes * kFftN * kFftN];
static struct {
  std::mutex mu;
  void *at[64];         // the array's address on each device
  hipEvent_t done[64];  // its last call there
} g_overlap;

static bool fft512_overlap(const void *four, const void *phys, long long nplanes, bool fp32) {
  const size_t real = fp32 ? sizeof(float) : sizeof(double);
  const char *f = (const char *)four, *p = (const char *)phys;
  return f < p + nplanes * kFftN * kFftN * real && p < f + nplanes * kFftN * kFftK * 2 * real;
}

template <class C>
static hipError_t fft512_inverse_overlap(const void *four, void *phys, long long nplanes, hipStream_t st, const C *tw) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);  // below 64: twiddles has checked it
  if (e != hipSuccess) return e;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if ((e = hipStreamIsCapturing(st, &cap)) != hipSuccess) return e;
  const bool order = cap == hipStreamCaptureStatusNone;
  std::lock_guard<std::mutex> lk(g_overlap.mu);
  void *&mid = g_overlap.at[dev];
  hipEvent_t &ev = g_overlap.done[dev];
  if (!mid && (e = hipGetSymbolAddress(&mid, HIP_SYMBOL(g_overlap_dev))) != hipSuccess) return e;
  if (order && ev && (e = hipStreamWaitEvent(st, ev, 0)) != hipSuccess) return e;
  if (order && !ev && (e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return e;
  e = fft512_inverse_t<C>(four, phys, nplanes, st, tw, static_cast<Sc<C> *>(mid), kOverlapPlanes);
  if (order) {
    const hipError_t r = hipEventRecord(ev, st);
    if (e == hipSuccess) e = r;
  }
  return e;
}

static hipError_t fft512_transform(bool inverse, const void *src, void *dst, long long nplanes, bool fp32,
                                   hipStream_t st) {
  const void *tw = nullptr;
  hipError_t e = fft512_lds_limits();
  if (e != hipSuccess) return e;
  e = twiddles(fp32, &tw);
  if (e != hipSuccess) return e;
  const float2 *t32 = static_cast<const float2 *>(tw);
  const double2 *t64 = static_cast<const double2 *>(tw);
  if (inverse && fft512_overlap(src, dst, nplanes, fp32))
    return fp32 ? fft512_inverse_overlap<float2>(src, dst, nplanes, st, t32)
                : fft512_inverse_overlap<double2>(src, dst, nplanes, st, t64);
  if (inverse)
    return fp32 ? fft512_inverse_t<float2>(src, dst, nplanes, st, t32, nullptr, kFftChunk)
                : fft512_inverse_t<double2>(src, dst, nplanes, st, t64, nullptr, kFftChunk);
  return fp32 ? fft512_forward_t<float2>(src, dst, nplanes, st, t32) : fft512_forward_t<double2>(src, dst, nplanes, st, t64);
}

}  // namespace dh

using namespace dh;

extern "C" {

const char *dh_batched_last_error(void) { return g_err.c_str(); }

int dh_cn_solve_batched_dev(const double *sl, const double *su, const double *alpha, const void *rhs, void *x,
                            int32_t ny, int64_t nsys, int32_t fp32, void *stream) {
  if (!sl || !su || !alpha || !rhs || !x) return fail(DH_EARG, "null pointer");
  if (ny < 2 || ny > kCnMaxNy) return fail(DH_EARG, "ny must lie in 2..288");
  if (nsys <= 0) return fail(DH_EARG, "nsys must be positive");
  if ((nsys + 7) / 8 > 0x7fffffffLL || (long long)ny * nsys > (1LL << 40)) return fail(DH_EARG, "too many systems");
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto launch = [&](auto seg) {
    constexpr int SEG = decltype(seg)::value, per = cn_systems(SEG);
    const dim3 g((unsigned)((nsys + per - 1) / per)), b(kCnThreads);
    if (fp32)
      hipLaunchKernelGGL((k_cn_solve<SEG, float2>), g, b, 0, st, sl, su, alpha, (const float2 *)rhs, (float2 *)x,
                         (int)ny, (long long)nsys);
    else
      hipLaunchKernelGGL((k_cn_solve<SEG, double2>), g, b, 0, st, sl, su, alpha, (const double2 *)rhs, (double2 *)x,
                         (int)ny, (long long)nsys);
  };
  if (ny <= 4 * kCnRows)
    launch(std::integral_constant<int, 4>{});
  else if (ny <= 8 * kCnRows)
    launch(std::integral_constant<int, 8>{});
  else if (ny <= 16 * kCnRows)
    launch(std::integral_constant<int, 16>{});
  else
    launch(std::integral_constant<int, 32>{});
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(DH_EHIP, hipGetErrorString(e));
  return DH_OK;
}

int dh_fft512_xz_to_fourier_dev(const void *phys, void *four, int64_t nplanes, int32_t fp32, void *stream) {
  if (!phys || !four) return fail(DH_EARG, "null pointer");
  if (nplanes <= 0) return fail(DH_EARG, "nplanes must be positive");
  const hipError_t e = fft512_transform(false, phys, four, nplanes, fp32 != 0, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(DH_EHIP, hipGetErrorString(e));
  return DH_OK;
}

int dh_fft512_xz_to_physical_dev(const void *four, void *phys, int64_t nplanes, int32_t fp32, void *stream) {
  if (!phys || !four) return fail(DH_EARG, "null pointer");
  if (nplanes <= 0) return fail(DH_EARG, "nplanes must be positive");
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(DH_EHIP, hipGetErrorString(e));
  if (dev < 0 || dev >= 64) return fail(DH_EARG, "device index beyond 63");
  e = fft512_transform(true, four, phys, nplanes, fp32 != 0, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(DH_EHIP, hipGetErrorString(e));
  return DH_OK;
}

int dh_fft512_xz_to_physical_noalloc_dev(const void *four, void *phys, int64_t nplanes, int32_t fp32, void *stream) {
  return dh_fft512_xz_to_physical_dev(four, phys, nplanes, fp32, stream);
}

}  // extern "C"
