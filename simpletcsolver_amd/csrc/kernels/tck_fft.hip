/*
 * tck_fft.hip -- batched FFTs of the Poisson solve (gfx950), replacing the FFTW plans of
 * src/fluid/compute_potential.c:247-309 and the pencil transposes around them (:517-581).
 *
 * Spectrum layout in HBM: S[kz][ky][i] (complex, i fastest, row pitch nx), ky = 0..ny/2.
 * With i innermost, the theta and z transforms read and write rows of a few consecutive i
 * (coalesced), and the radial solve reads each (ky, kz) line contiguously: no transpose
 * pass is needed anywhere.
 *
 *  tck_div_yfft   assign_input (:382-425: divergence / (gamma dt ny nz)) fused with the
 *                 real-to-complex theta transform; a real length-N transform is done as a
 *                 complex length-N/2 transform of (x_2m + i x_2m+1) plus the usual split.
 *  tck_zfft       complex axial transforms, forward or backward, in place.
 *  tck_yifft_psi  complex-to-real theta transform fused with extract_output (:427-443): psi
 *                 with its periodic halos and Neumann wall copies (boundary/psi.c:13-45).
 * The first pass of a tile takes its butterflies from memory and the last pass stores from
 * registers, so a tile crosses LDS only between passes (tck_div_yfft's split and
 * tck_yifft_psi's pairing each add one crossing).  tck_zfft and tck_yifft_psi have a persistent
 * form (suffix _p) for launches whose tiles cover the data exactly: a block loops over tiles and
 * issues the next tile's loads before the current tile's passes.  Tiles whose LDS leaves few
 * blocks per CU run with half the elements per thread (twice the threads), so that a CU still
 * holds 16 waves.  Every form computes the same bits.
 * Transforms are unnormalised, as FFTW's; the imaginary parts of the DC and Nyquist bins are
 * ignored by the complex-to-real transform, as FFTW's c2r does with a Hermitian input.
 *
 * The in-LDS transform is a Stockham autosort FFT (Govindaraju et al., "High performance
 * discrete Fourier transforms on graphics processors", SC 2008) with radix 8, 7, 5, 4, 3
 * and 2 passes; each pass reads all its butterfly inputs into registers, synchronises, and
 * writes in place.
 */
#include "tck_common.h"

#define FFT_MAXST 16
#define FFT_EPT 16   /* complex elements per thread per pass */
#define FFT_MAXTHREADS 1024

/* complex pair of the transform's arithmetic type T (double, or float in the mixed step) */
template <typename T> struct cvec;
template <> struct cvec<double> { typedef double2 type; };
template <> struct cvec<float> { typedef float2 type; };
template <typename T> __device__ __forceinline__ typename cvec<T>::type mk2(T x, T y);
template <> __device__ __forceinline__ double2 mk2<double>(double x, double y){ return make_double2(x, y); }
template <> __device__ __forceinline__ float2 mk2<float>(float x, float y){ return make_float2(x, y); }

struct FftPlan {
  int M;
  int nst;
  int rad[FFT_MAXST];
  /* per stage: multipliers that divide by M / rad and by the stage's span Ns with one high
   * multiply (floor(2^32 / d) + 1, exact for dividends below 2^16; 0 for d = 1) */
  unsigned mper[FFT_MAXST], mns[FFT_MAXST];
  /* threads per block of the launch.  The kernels read the block size from here (a kernel
   * argument, in scalar registers) rather than from blockDim.x, whose 16-bit read from the
   * dispatch packet is a vector memory load that the compiler may repeat inside the passes:
   * a wait for it there would also wait for every global load and store issued before it. */
  int nt;
};

/* log2 of a tile width (tile widths are powers of two, at most 64) */
__device__ __forceinline__ int fft_lg(int x){ return __builtin_ctz((unsigned)x); }

/* x / d for the multiplier m of d (see FftPlan) */
__device__ __forceinline__ unsigned fft_div(unsigned x, unsigned m){
  return m ? __umulhi(x, m) : x;
}

template <typename V> __device__ __forceinline__ V cmul(V a, V b){
  V r; r.x = a.x * b.x - a.y * b.y; r.y = a.x * b.y + a.y * b.x; return r;
}
template <typename V> __device__ __forceinline__ V cadd(V a, V b){ V r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }
template <typename V> __device__ __forceinline__ V csub(V a, V b){ V r; r.x = a.x - b.x; r.y = a.y - b.y; return r; }
/* s i a */
template <typename V, typename T> __device__ __forceinline__ V crot(V a, T s){ V r; r.x = - s * a.y; r.y = s * a.x; return r; }
template <typename V> __device__ __forceinline__ V cconj(V a){ V r; r.x = a.x; r.y = - a.y; return r; }

/* R-point DFTs, y_k = sum_n x_n exp(s 2 pi i n k / R) */
template <int R, typename T> struct dftr;

template <typename T> struct dftr<2, T> {
  typedef typename cvec<T>::type V;
  static __device__ __forceinline__ void run(V * x, T s){
    (void)s;
    const V a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
  }
};

template <typename T> struct dftr<4, T> {
  typedef typename cvec<T>::type V;
  static __device__ __forceinline__ void run(V * x, T s){
    const V a0 = cadd(x[0], x[2]), a1 = csub(x[0], x[2]);
    const V b0 = cadd(x[1], x[3]), b1 = crot(csub(x[1], x[3]), s);
    x[0] = cadd(a0, b0);
    x[2] = csub(a0, b0);
    x[1] = cadd(a1, b1);
    x[3] = csub(a1, b1);
  }
};

template <typename T> struct dftr<3, T> {
  typedef typename cvec<T>::type V;
  static __device__ __forceinline__ void run(V * x, T s){
    const T h = T(0.86602540378443864676);   /* sqrt(3) / 2 */
    const V t1 = cadd(x[1], x[2]);
    const V t2 = crot(csub(x[1], x[2]), s * h);
    const V m = mk2<T>(x[0].x - T(0.5) * t1.x, x[0].y - T(0.5) * t1.y);
    x[0] = cadd(x[0], t1);
    x[1] = cadd(m, t2);
    x[2] = csub(m, t2);
  }
};

/* odd R-point DFT by conjugate pairs (R = 5, 7): with a_n = x_n + x_{R-n} and
 * b_n = x_n - x_{R-n}, n = 1..h = (R-1)/2,
 *   y_0 = x_0 + sum a_n,  y_k, y_{R-k} = x_0 + sum_n a_n cos(2 pi n k / R)
 *                                     +- s i sum_n b_n sin(2 pi n k / R),  k = 1..h */
template <int R> struct oddtab;
template <> struct oddtab<5> {
  static __device__ __forceinline__ double c(int m){
    return m == 1 ? 0.3090169943749474241023 : -0.8090169943749474241023;
  }
  static __device__ __forceinline__ double sn(int m){
    return m == 1 ? 0.9510565162951535721164 : 0.5877852522924731291687;
  }
};
template <> struct oddtab<7> {
  static __device__ __forceinline__ double c(int m){
    return m == 1 ? 0.6234898018587335305250 : m == 2 ? -0.2225209339563144042889 : -0.9009688679024191262361;
  }
  static __device__ __forceinline__ double sn(int m){
    return m == 1 ? 0.7818314824680298087084 : m == 2 ? 0.9749279121818236070181 : 0.4338837391175581204758;
  }
};

template <int R, typename T> struct dftodd {
  typedef typename cvec<T>::type V;
  static __device__ __forceinline__ void run(V * x, T s){
    constexpr int h = (R - 1) / 2;
    V a[h], b[h];
    #pragma unroll
    for(int n = 1; n <= h; n++){ a[n - 1] = cadd(x[n], x[R - n]); b[n - 1] = csub(x[n], x[R - n]); }
    V y0 = x[0];
    #pragma unroll
    for(int n = 0; n < h; n++) y0 = cadd(y0, a[n]);
    V re[h], im[h];
    #pragma unroll
    for(int k = 1; k <= h; k++){
      V r = x[0];
      V q = mk2<T>(T(0.), T(0.));
      #pragma unroll
      for(int n = 1; n <= h; n++){
        /* m = n k mod R, folded into 1..h with the sign of the sine */
        const int m0 = (n * k) % R;
        const int m = m0 <= h ? m0 : R - m0;
        const T cv = T(oddtab<R>::c(m));
        const T sv = T(m0 <= h ? oddtab<R>::sn(m) : - oddtab<R>::sn(m));
        r = mk2<T>(r.x + cv * a[n - 1].x, r.y + cv * a[n - 1].y);
        q = mk2<T>(q.x + sv * b[n - 1].x, q.y + sv * b[n - 1].y);
      }
      re[k - 1] = r;
      im[k - 1] = crot(q, s);
    }
    x[0] = y0;
    #pragma unroll
    for(int k = 1; k <= h; k++){
      x[k] = cadd(re[k - 1], im[k - 1]);
      x[R - k] = csub(re[k - 1], im[k - 1]);
    }
  }
};
template <typename T> struct dftr<5, T> : dftodd<5, T> {};
template <typename T> struct dftr<7, T> : dftodd<7, T> {};

template <typename T> struct dftr<8, T> {
  typedef typename cvec<T>::type V;
  static __device__ __forceinline__ void run(V * x, T s){
    const T r = T(0.70710678118654752440);   /* sqrt(1/2) */
    V e[4] = {x[0], x[2], x[4], x[6]};
    V o[4] = {x[1], x[3], x[5], x[7]};
    dftr<4, T>::run(e, s);
    dftr<4, T>::run(o, s);
    /* o_k *= w8^k, w8 = r (1 + s i) */
    o[1] = mk2<T>(r * (o[1].x - s * o[1].y), r * (o[1].y + s * o[1].x));
    o[2] = crot(o[2], s);
    o[3] = mk2<T>(r * (- o[3].x - s * o[3].y), r * (- o[3].y + s * o[3].x));
    #pragma unroll
    for(int k = 0; k < 4; k++){
      x[k] = cadd(e[k], o[k]);
      x[k + 4] = csub(e[k], o[k]);
    }
  }
};

/* block barrier that orders the LDS accesses only: global loads issued before it stay in
 * flight and pending global stores are not waited for */
__device__ __forceinline__ void fft_lds_barrier(){
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* the same, and no instruction is scheduled across it: the loads of the pass after it (its
 * twiddle factors) are not hoisted into the pass before it, which would hold more registers */
__device__ __forceinline__ void fft_pass_barrier(){
  __builtin_amdgcn_sched_barrier(0);
  fft_lds_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

/* padded position of element n of a line in LDS: one spare slot after every 8 elements, so
 * that the first Stockham pass, which writes elements R apart from consecutive threads, and
 * the row-wise fills spread over all banks */
__host__ __device__ __forceinline__ int fpad(int n){ return n + (n >> 3); }

template <int R, typename T, int EPT = FFT_EPT>
__device__ __forceinline__ void fft_stage(typename cvec<T>::type * buf, int M, int ld, int nb, int Ns,
    const typename cvec<T>::type * __restrict__ tw, T s, unsigned mper, unsigned mns, int nt){
  typedef typename cvec<T>::type V;
  constexpr int BPT = (EPT + R - 1) / R;
  const int tid = threadIdx.x;
  const int per = M / R;
  const int nbf = nb * per;
  const int twstep = M / (Ns * R);
  V v[BPT][R];
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = tid + q * nt;
    if(bf < nbf){
      const int b = (int)fft_div((unsigned)bf, mper);
      const int jj = bf - b * per;
      const int jm = jj - (int)fft_div((unsigned)jj, mns) * Ns;
      const V * src = buf + b * ld;
      #pragma unroll
      for(int r = 0; r < R; r++){
        V x = src[fpad(jj + r * per)];
        if(r > 0){
          V w = tw[jm * r * twstep];
          if(s > T(0.)) w.y = - w.y;
          x = cmul(x, w);
        }
        v[q][r] = x;
      }
      dftr<R, T>::run(v[q], s);
    }
  }
  fft_pass_barrier();
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = tid + q * nt;
    if(bf < nbf){
      const int b = (int)fft_div((unsigned)bf, mper);
      const int jj = bf - b * per;
      const int jm = jj - (int)fft_div((unsigned)jj, mns) * Ns;
      V * dst = buf + b * ld;
      const int d0 = (jj - jm) * R + jm;
      #pragma unroll
      for(int r = 0; r < R; r++) dst[fpad(d0 + r * Ns)] = v[q][r];
    }
  }
  fft_pass_barrier();
}

/* The first and last passes with the tile's memory accesses in them.  The inputs of a first
 * pass's butterfly jj are the elements jj + r M / R, and the outputs of a last pass's the same,
 * so a thread loads its butterflies' inputs straight into registers and stores the last
 * pass's results from there: a transform of n passes crosses LDS n - 1 times instead of n + 1.
 * Butterflies are numbered with the line fastest, so that a row access covers consecutive
 * lines.  The first pass's twiddle factors are all 1 and are left out; otherwise the operations
 * are fft_stage's. */
template <int R, typename T, int EPT, typename LD>
__device__ __forceinline__ void fft_load_pass(typename cvec<T>::type (*v)[R], int M, int lg, int nbf, T s, int nt, LD load){
  constexpr int BPT = (EPT + R - 1) / R;
  const int per = M / R, nb1 = (1 << lg) - 1;
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = (int)threadIdx.x + q * nt;
    #pragma unroll
    for(int r = 0; r < R; r++) v[q][r] = load(bf & nb1, (bf >> lg) + r * per, bf < nbf);
  }
  #pragma unroll
  for(int q = 0; q < BPT; q++) dftr<R, T>::run(v[q], s);
}

template <int R, typename T, int EPT, typename LD>
__device__ __forceinline__ void fft_first_r(typename cvec<T>::type * buf, int M, int ld, int lg, T s, int nt, LD load){
  constexpr int BPT = (EPT + R - 1) / R;
  const int nbf = (M / R) << lg, nb1 = (1 << lg) - 1;
  typename cvec<T>::type v[BPT][R];
  fft_load_pass<R, T, EPT>(v, M, lg, nbf, s, nt, load);
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = (int)threadIdx.x + q * nt;
    if(bf < nbf){
      typename cvec<T>::type * dst = buf + (bf & nb1) * ld;
      const int d0 = (bf >> lg) * R;
      #pragma unroll
      for(int r = 0; r < R; r++) dst[fpad(d0 + r)] = v[q][r];
    }
  }
}

template <typename T, int EPT, bool W, typename LD>
__device__ __forceinline__ void fft_first(typename cvec<T>::type * buf, int ld, int lg, const FftPlan & P, T s, LD load){
  const int R = P.rad[0];
  if(R == 8) fft_first_r<8, T, EPT>(buf, P.M, ld, lg, s, P.nt, load);
  else if(R == 4) fft_first_r<4, T, EPT>(buf, P.M, ld, lg, s, P.nt, load);
  else if(R == 2) fft_first_r<2, T, EPT>(buf, P.M, ld, lg, s, P.nt, load);
  else if(W && R == 5) fft_first_r<5, T, EPT>(buf, P.M, ld, lg, s, P.nt, load);
  else if(W && R == 7) fft_first_r<7, T, EPT>(buf, P.M, ld, lg, s, P.nt, load);
  else fft_first_r<3, T, EPT>(buf, P.M, ld, lg, s, P.nt, load);
  fft_pass_barrier();
}

/* passes st0..st1 - 1, in LDS, of nb transforms of length P.M stored at buf + b * ld; tw[t] =
 * exp(-2 pi i t / M); each pass keeps at most EPT elements per thread in registers, so
 * P.nt * EPT >= nb * P.M.  W: the plan may hold radix 5 and 7 passes (compiled only into the
 * kernels of such lengths, so that the 2^a 3^b kernels keep their register budget) */
template <typename T, int EPT, bool W>
__device__ __forceinline__ void fft_mid(typename cvec<T>::type * buf, int ld, int nb, const FftPlan & P,
    const typename cvec<T>::type * __restrict__ tw, T s, int st0, int st1){
  int Ns = 1;
  for(int st = 0; st < st0; st++) Ns *= P.rad[st];
  for(int st = st0; st < st1; st++){
    const int R = P.rad[st];
    const unsigned mp = P.mper[st], mn = P.mns[st];
    if(R == 8) fft_stage<8, T, EPT>(buf, P.M, ld, nb, Ns, tw, s, mp, mn, P.nt);
    else if(R == 4) fft_stage<4, T, EPT>(buf, P.M, ld, nb, Ns, tw, s, mp, mn, P.nt);
    else if(R == 3) fft_stage<3, T, EPT>(buf, P.M, ld, nb, Ns, tw, s, mp, mn, P.nt);
    else if(W && R == 5) fft_stage<5, T, EPT>(buf, P.M, ld, nb, Ns, tw, s, mp, mn, P.nt);
    else if(W && R == 7) fft_stage<7, T, EPT>(buf, P.M, ld, nb, Ns, tw, s, mp, mn, P.nt);
    else if(R == 2) fft_stage<2, T, EPT>(buf, P.M, ld, nb, Ns, tw, s, mp, mn, P.nt);
    Ns *= R;
  }
}

template <int R, typename T, int EPT, typename ST>
__device__ __forceinline__ void fft_last_r(const typename cvec<T>::type * buf, int M, int ld, int lg,
    const typename cvec<T>::type * __restrict__ tw, T s, int nt, ST store){
  typedef typename cvec<T>::type V;
  constexpr int BPT = (EPT + R - 1) / R;
  const int per = M / R, nbf = per << lg, nb1 = (1 << lg) - 1;
  V v[BPT][R];
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = (int)threadIdx.x + q * nt;
    if(bf < nbf){
      const int jj = bf >> lg;
      const V * src = buf + (bf & nb1) * ld;
      #pragma unroll
      for(int r = 0; r < R; r++){
        V x = src[fpad(jj + r * per)];
        if(r > 0){
          V w = tw[jj * r];
          if(s > T(0.)) w.y = - w.y;
          x = cmul(x, w);
        }
        v[q][r] = x;
      }
      dftr<R, T>::run(v[q], s);
    }
  }
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = (int)threadIdx.x + q * nt;
    #pragma unroll
    for(int r = 0; r < R; r++) store(bf & nb1, (bf >> lg) + r * per, v[q][r], bf < nbf);
  }
}

template <typename T, int EPT, bool W, typename ST>
__device__ __forceinline__ void fft_last(const typename cvec<T>::type * buf, int ld, int lg, const FftPlan & P,
    const typename cvec<T>::type * __restrict__ tw, T s, ST store){
  const int R = P.rad[P.nst - 1];
  if(R == 8) fft_last_r<8, T, EPT>(buf, P.M, ld, lg, tw, s, P.nt, store);
  else if(R == 4) fft_last_r<4, T, EPT>(buf, P.M, ld, lg, tw, s, P.nt, store);
  else if(R == 2) fft_last_r<2, T, EPT>(buf, P.M, ld, lg, tw, s, P.nt, store);
  else if(W && R == 5) fft_last_r<5, T, EPT>(buf, P.M, ld, lg, tw, s, P.nt, store);
  else if(W && R == 7) fft_last_r<7, T, EPT>(buf, P.M, ld, lg, tw, s, P.nt, store);
  else fft_last_r<3, T, EPT>(buf, P.M, ld, lg, tw, s, P.nt, store);
}

/* a transform of one pass (lengths 2, 3, 4, 5, 7 and 8): no LDS at all */
template <int R, typename T, int EPT, typename LD, typename ST>
__device__ __forceinline__ void fft_only_r(int M, int lg, T s, int nt, LD load, ST store){
  constexpr int BPT = (EPT + R - 1) / R;
  const int per = M / R, nbf = per << lg, nb1 = (1 << lg) - 1;
  typename cvec<T>::type v[BPT][R];
  fft_load_pass<R, T, EPT>(v, M, lg, nbf, s, nt, load);
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = (int)threadIdx.x + q * nt;
    #pragma unroll
    for(int r = 0; r < R; r++) store(bf & nb1, (bf >> lg) + r * per, v[q][r], bf < nbf);
  }
}

/* the whole transform of a tile of 1 << lg lines: load(t, n, ok) gives element n of line t (ok
 * false: any value, from a valid address), store(t, n, v, ok) takes it (ok false: nothing) */
template <typename T, int EPT, bool W, typename LD, typename ST>
__device__ __forceinline__ void fft_tile_run(typename cvec<T>::type * buf, int ld, int lg, const FftPlan & P,
    const typename cvec<T>::type * __restrict__ tw, T s, LD load, ST store){
  if(P.nst == 1){
    const int R = P.rad[0];
    if(R == 8) fft_only_r<8, T, EPT>(P.M, lg, s, P.nt, load, store);
    else if(R == 4) fft_only_r<4, T, EPT>(P.M, lg, s, P.nt, load, store);
    else if(R == 2) fft_only_r<2, T, EPT>(P.M, lg, s, P.nt, load, store);
    else if(W && R == 5) fft_only_r<5, T, EPT>(P.M, lg, s, P.nt, load, store);
    else if(W && R == 7) fft_only_r<7, T, EPT>(P.M, lg, s, P.nt, load, store);
    else fft_only_r<3, T, EPT>(P.M, lg, s, P.nt, load, store);
    return;
  }
  fft_first<T, EPT, W>(buf, ld, lg, P, s, load);
  fft_mid<T, EPT, W>(buf, ld, 1 << lg, P, tw, s, 1, P.nst - 1);
  fft_last<T, EPT, W>(buf, ld, lg, P, tw, s, store);
}

__constant__ double c_fft_rka[3] = {32. / 60., 25. / 60., 45. / 60.};
__constant__ double c_fft_rkb[3] = { 0. / 60., -17. / 60., -25. / 60.};

/* tile of this block among ntiles: blocks that run on the same XCD (consecutive slots of the
 * round-robin dispatch) take consecutive tiles, whose rows share 128 B lines in its L2 */
__device__ __forceinline__ long long fft_tile_of(long long ntiles){
  long long t = blockIdx.x;
  if(ntiles % TCK_NXCD == 0) t = (t % TCK_NXCD) * (ntiles / TCK_NXCD) + t / TCK_NXCD;
  return t;
}

/* ------------------------------------------------------------------------------------- */
struct YFwdArgs {
  tc_geom_t g;
  tc_coef_t c;
  const double * ux; const double * uy; const double * uz;
  const double * dt;
  int rkstep;
  void * S;                      /* spectrum of the transform type */
  int nky, ti, ld;               /* ld: LDS row pitch of a padded line (fft_ld) */
  FftPlan P;                     /* length M = ny / 2 */
  const void * twM;              /* exp(-2 pi i t / M) */
  const void * twN;              /* exp(-2 pi i k / ny), k = 0..M */
};

/* the divergence is formed in FP64 (assign_input :404-423) and rounded to the transform
 * type T only when it enters the transform */
/* the first pass of a tile: packed element n of a line is the divergence at rows 2 n + 1 and
 * 2 n + 2, whose common face is read once; GD elements' loads are issued together (out-of-field
 * elements read cell (1, 1) of the plane and are put as 0, so that no load is conditional) */
template <int R, typename T, int EPT, int GD>
__device__ __forceinline__ void div_first_r(typename cvec<T>::type * buf, const YFwdArgs & A, int i0, int k, double prefactor){
  typedef typename cvec<T>::type V;
  constexpr int BPT = (EPT + R - 1) / R;
  const tc_geom_t & g = A.g;
  const tc_coef_t & c = A.c;
  const int lg = fft_lg(A.ti), nt = A.P.nt;
  const int per = A.P.M / R, nbf = per << lg;
  const long long sy = g.px, sz = g.plane;
  V v[BPT][R];
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    const int bf = (int)threadIdx.x + q * nt;
    const int i = i0 + (bf & (A.ti - 1)), jj = bf >> lg;
    const bool ok = bf < nbf && i <= g.nx;
    const int ii = ok ? i : 1;
    #pragma unroll
    for(int r0 = 0; r0 < R; r0 += GD){
      /* one batch of loads at a time: more would not fit in registers beside v */
      asm volatile("" ::: "memory");
      double P[GD][11];
      #pragma unroll
      for(int u = 0; u < GD; u++) if(r0 + u < R){
        const long long o = tck_idx(g, ii, ok ? 2 * (jj + (r0 + u) * per) + 1 : 1, k);
        P[u][0] = A.ux[o]; P[u][1] = A.ux[o + 1]; P[u][2] = A.ux[o + sy]; P[u][3] = A.ux[o + sy + 1];
        P[u][4] = A.uy[o]; P[u][5] = A.uy[o + sy]; P[u][6] = A.uy[o + 2 * sy];
        P[u][7] = A.uz[o]; P[u][8] = A.uz[o + sz]; P[u][9] = A.uz[o + sy]; P[u][10] = A.uz[o + sy + sz];
      }
      #pragma unroll
      for(int u = 0; u < GD; u++) if(r0 + u < R){
        const double d0 = c.ijdxc[ii] * (
            - c.jhxf[ii] * P[u][0] + c.jhxf[ii + 1] * P[u][1]
            - c.jhyc[ii] * P[u][4] + c.jhyc[ii] * P[u][5]
            - c.jhzc[ii] * P[u][7] + c.jhzc[ii] * P[u][8]);
        const double d1 = c.ijdxc[ii] * (
            - c.jhxf[ii] * P[u][2] + c.jhxf[ii + 1] * P[u][3]
            - c.jhyc[ii] * P[u][5] + c.jhyc[ii] * P[u][6]
            - c.jhzc[ii] * P[u][9] + c.jhzc[ii] * P[u][10]);
        v[q][r0 + u] = mk2<T>(ok ? T(prefactor * d0) : T(0.), ok ? T(prefactor * d1) : T(0.));
        asm volatile("" : "+v"(v[q][r0 + u].x), "+v"(v[q][r0 + u].y));
      }
    }
  }
  #pragma unroll
  for(int q = 0; q < BPT; q++){
    dftr<R, T>::run(v[q], T(-1.));
    const int bf = (int)threadIdx.x + q * nt;
    if(bf < nbf){
      V * dst = buf + (bf & (A.ti - 1)) * A.ld;
      const int d0 = (bf >> lg) * R;
      #pragma unroll
      for(int r = 0; r < R; r++) dst[fpad(d0 + r)] = v[q][r];
    }
  }
}

/* NTMAX, the block size the kernel is compiled for, sets how many elements' loads are issued at a
 * time beside the pass's registers: 1024 two (four in FP32), 512 three (at four waves per SIMD),
 * 256 all eight, for launches of so few waves that their latency is what counts */
template <typename T, int EPT, bool W, int NTMAX>
__global__ void __launch_bounds__(NTMAX) tck_div_yfft(const YFwdArgs A){
  constexpr int GD = NTMAX == 256 ? 8 : (sizeof(T) == 4 ? 4 : (NTMAX == 512 ? 3 : 2));
  typedef typename cvec<T>::type V;
  extern __shared__ __align__(16) unsigned char fft_smem[];
  V * sm = (V *)fft_smem;
  const tc_geom_t & g = A.g;
  const int ti = A.ti;
  const int M = A.P.M;
  const int ntx = (g.nx + ti - 1) / ti;
  const long long tile = fft_tile_of((long long)ntx * g.nz);
  const int i0 = 1 + (int)(tile % ntx) * ti;
  const int k = 1 + (int)(tile / ntx);
  const double dt = *A.dt;
  const double gamma = c_fft_rka[A.rkstep] + c_fft_rkb[A.rkstep];
  const double norm = 1. * g.ny * g.nz;
  const double prefactor = 1. / (gamma * dt) / norm;
  const V * twM = (const V *)A.twM;
  const V * twN = (const V *)A.twN;
  const int R = A.P.rad[0];
  if(R == 8) div_first_r<8, T, EPT, GD>(sm, A, i0, k, prefactor);
  else if(R == 4) div_first_r<4, T, EPT, GD>(sm, A, i0, k, prefactor);
  else if(R == 2) div_first_r<2, T, EPT, GD>(sm, A, i0, k, prefactor);
  else if(W && R == 5) div_first_r<5, T, EPT, GD>(sm, A, i0, k, prefactor);
  else if(W && R == 7) div_first_r<7, T, EPT, GD>(sm, A, i0, k, prefactor);
  else div_first_r<3, T, EPT, GD>(sm, A, i0, k, prefactor);
  fft_pass_barrier();
  fft_mid<T, EPT, W>(sm, A.ld, ti, A.P, twM, T(-1.), 1, A.P.nst);
  /* split: X_k = (Z_k + conj Z_{M-k}) / 2 - i W^k (Z_k - conj Z_{M-k}) / 2, k = 0..M */
  V * S = (V *)A.S;
  for(int e = threadIdx.x; e < ti * (M + 1); e += A.P.nt){
    const int t = (e & (ti - 1));
    const int kk = (e >> fft_lg(ti));
    const int i = i0 + t;
    if(i > g.nx) continue;
    const V zk = sm[t * A.ld + fpad(kk == M ? 0 : kk)];
    const V zc = cconj(sm[t * A.ld + fpad(kk == 0 ? 0 : M - kk)]);
    const V w = twN[kk];
    const V ev = mk2<T>(T(0.5) * (zk.x + zc.x), T(0.5) * (zk.y + zc.y));
    const V od = mk2<T>(T(0.5) * (zk.x - zc.x), T(0.5) * (zk.y - zc.y));
    /* - i w od */
    const V wo = cmul(w, od);
    const V X = mk2<T>(ev.x + wo.y, ev.y - wo.x);
    tck_st(&S[(long long)(i - 1) + (long long)g.nx * ((long long)kk + (long long)A.nky * (k - 1))], X);
  }
}

/* ------------------------------------------------------------------------------------- */
struct ZArgs {
  int nx, nky, nz, tz, ld;
  void * S;
  FftPlan P;               /* length nz */
  const void * tw;
  double sign;
};

/* one block per tile of tz consecutive i at one ky */
template <typename T, int EPT, bool W>
__global__ void __launch_bounds__(FFT_MAXTHREADS) tck_zfft(const ZArgs A){
  typedef typename cvec<T>::type V;
  extern __shared__ __align__(16) unsigned char fft_smem[];
  V * sm = (V *)fft_smem;
  const int tz = A.tz;
  const int ntx = (A.nx + tz - 1) / tz;
  const long long tile = fft_tile_of((long long)ntx * A.nky);
  const int i0 = (int)(tile % ntx) * tz;
  const int ky = (int)(tile / ntx);
  const long long kstride = (long long)A.nx * A.nky;
  V * base = (V *)A.S + (long long)A.nx * ky + i0;
  const int nl = A.nx - i0;   /* lines of this tile inside the spectrum */
  fft_tile_run<T, EPT, W>(sm, A.ld, fft_lg(tz), A.P, (const V *)A.tw, T(A.sign),
      [&](int t, int kz, bool ok){ return tck_ld(ok && t < nl ? &base[t + kstride * kz] : (const V *)A.S); },
      [&](int t, int kz, V v, bool ok){ if(ok && t < nl) tck_st(&base[t + kstride * kz], v); });
}

/* Persistent exact form: the tiles cover the spectrum exactly (nx a multiple of tz, blockDim.x EPTK
 * = tz nz), so no access is conditional; the first radix is 8 and the last one RL (2, 3, 4 or 8).
 * The twiddle factors are read from LDS (after the tile's lines), so that the passes issue no
 * global loads.  The inputs of the next tile's first pass are loaded into registers before the
 * current tile's middle passes, and the last pass stores its results from registers, so a tile
 * crosses LDS once between passes.  Outstanding global loads and stores complete in issue order
 * as far as the wait counter is concerned, so a wait for a load issued after a store also waits
 * for the store: here the loads of tile n+1 are issued before the stores of tile n, and the
 * first pass of tile n+1 waits only for its loads.  The stores into a zero-size buffer before the
 * loop (they write nothing) give the loop's entry the same outstanding loads-then-stores
 * sequence as the end of an iteration, so that the compiler's wait there is the same counted
 * wait on both paths into it.  Bound by HBM (the spectrum read and written once).  Against a
 * persistent form that went through LDS for the first loads and the last stores, ms per step
 * (six launches): FP64 512x1024x512 6.02 -> 5.17, 256x512x512 1.60 -> 1.38; FP32 256x512x512
 * 0.82 -> 0.74 */
template <typename T, int EPTK, int RL>
__global__ void __launch_bounds__(FFT_MAXTHREADS) tck_zfft_p(const ZArgs A){
  typedef typename cvec<T>::type V;
  extern __shared__ __align__(16) unsigned char fft_smem[];
  V * sm = (V *)fft_smem;
  constexpr int NB = EPTK / 8, NL = (EPTK + RL - 1) / RL;     /* butterflies per thread: first, last pass */
  constexpr bool ALL = NL * RL == EPTK;             /* every thread has NL in the last pass */
  const int tz = A.tz, nz = A.nz, nt = A.P.nt, lg = fft_lg(tz);
  const int ntx = A.nx / tz;
  const int ntiles = ntx * A.nky;
  const long long kstride = (long long)A.nx * A.nky;
  V * twl = sm + tz * A.ld;
  for(int t = threadIdx.x; t < nz; t += nt) twl[t] = ((const V *)A.tw)[t];
  /* butterfly q of this thread: line t0, index j0 + q dr */
  const int t0 = threadIdx.x & (tz - 1), j0 = (int)threadIdx.x >> lg, dr = nt >> lg;
  const int perf = nz / 8, perl = nz / RL;
  /* FP32: the spectrum spans under 4 GB (checked on the host), so a tile's accesses are a buffer
   * resource at the tile's first column plus 32-bit offsets */
  const unsigned vz = (unsigned)sizeof(V) * (unsigned)(t0 + kstride * j0);
  const unsigned ks = (unsigned)sizeof(V) * (unsigned)kstride;
  #define ZX_COL(tl) ((V *)A.S + (long long)A.nx * ((tl) / ntx) + (long long)(((tl) % ntx) * tz))
  #define ZX_RS(tl) tck_rsrc_u(ZX_COL(tl), ks * (unsigned)nz)
  #define ZX_LOAD(tl) \
    if constexpr (sizeof(T) == 4){ \
      const __amdgpu_buffer_rsrc_t rs = ZX_RS(tl); \
      _Pragma("unroll") for(int q = 0; q < NB; q++) \
        _Pragma("unroll") for(int r = 0; r < 8; r++) pre[q][r] = tck_bldf2(rs, vz, ks * (unsigned)(q * dr + r * perf)); \
    }else{ \
      const V * col = ZX_COL(tl) + (t0 + kstride * j0); \
      _Pragma("unroll") for(int q = 0; q < NB; q++) \
        _Pragma("unroll") for(int r = 0; r < 8; r++) pre[q][r] = tck_ld(col + kstride * (q * dr + r * perf)); \
    }
  int tile = blockIdx.x;             /* the launch has at least four tiles per block */
  const T s = T(A.sign);
  V pre[NB][8];
  ZX_LOAD(tile)
  {
    const __amdgpu_buffer_rsrc_t nul = tck_rsrc(A.S, 0u);
    #pragma unroll
    for(int q = 0; q < EPTK; q++) tck_bst0(nul, 16u * q);
  }
  for(;;){
    /* the LDS offsets are recomputed in every tile rather than held across the passes */
    int tt = t0, jj0 = j0;
    asm volatile("" : "+v"(tt), "+v"(jj0));
    #pragma unroll
    for(int q = 0; q < NB; q++){
      dftr<8, T>::run(pre[q], s);
      V * dst = sm + tt * A.ld;
      #pragma unroll
      for(int r = 0; r < 8; r++) dst[fpad(8 * (jj0 + q * dr) + r)] = pre[q][r];
    }
    fft_pass_barrier();
    const int nxt = tile + (int)gridDim.x < ntiles ? tile + (int)gridDim.x : tile;
    ZX_LOAD(nxt)
    fft_mid<T, EPTK, false>(sm, A.ld, tz, A.P, twl, s, 1, A.P.nst - 1);
    {
      const __amdgpu_buffer_rsrc_t rs = ZX_RS(tile);
      V * col = ZX_COL(tile) + (tt + kstride * jj0);
      const V * src = sm + tt * A.ld;
      #pragma unroll
      for(int q = 0; q < NL; q++){
        const int jj = jj0 + q * dr;
        if(!ALL && jj >= perl) break;
        V v[RL];
        #pragma unroll
        for(int r = 0; r < RL; r++){
          V x = src[fpad(jj + r * perl)];
          if(r > 0){
            V w = twl[jj * r];
            if(s > T(0.)) w.y = - w.y;
            x = cmul(x, w);
          }
          v[r] = x;
        }
        dftr<RL, T>::run(v, s);
        #pragma unroll
        for(int r = 0; r < RL; r++){
          if constexpr (sizeof(T) == 4) tck_bstf2(rs, vz, ks * (unsigned)(q * dr + r * perl), v[r]);
          else tck_st(col + kstride * (q * dr + r * perl), v[r]);
        }
      }
    }
    tile += (int)gridDim.x;
    if(tile >= ntiles) break;
    fft_lds_barrier();
  }
  #undef ZX_COL
  #undef ZX_RS
  #undef ZX_LOAD
}

/* ------------------------------------------------------------------------------------- */
struct YInvArgs {
  tc_geom_t g;
  const void * S;
  void * psi;              /* of the transform type */
  int nky, ti, ld;
  FftPlan P;
  const void * twM;
  const void * twN;
};

/* Z'_k = (X_k + conj X_{M-k}) + i W^{-k} (X_k - conj X_{M-k}) so that
 * IFFT_M(Z')_m = x_2m + i x_2m+1 (unnormalised, as FFTW's c2r) */
template <typename V>
__device__ __forceinline__ V c2r_pre(V xk, V xmk, V w){
  const V xc = cconj(xmk);
  const V a = cadd(xk, xc);
  const V d = csub(xk, xc);
  const V wd = cmul(cconj(w), d);
  V r;
  r.x = a.x - wd.y;
  r.y = a.y + wd.x;
  return r;
}

template <typename T, int EPT, bool W>
__global__ void __launch_bounds__(FFT_MAXTHREADS) tck_yifft_psi(const YInvArgs A){
  typedef typename cvec<T>::type V;
  extern __shared__ __align__(16) unsigned char fft_smem[];
  V * sm = (V *)fft_smem;
  const tc_geom_t & g = A.g;
  const int ti = A.ti, lg = fft_lg(ti);
  const int M = A.P.M;
  const int ntx = (g.nx + ti - 1) / ti;
  const long long tile = fft_tile_of((long long)ntx * g.nz);
  const int i0 = 1 + (int)(tile % ntx) * ti;
  const int k = 1 + (int)(tile / ntx);
  const int nl = g.nx + 1 - i0;   /* lines of this tile inside the field */
  const V * S = (const V *)A.S;
  const V * row = S + (long long)g.nx * (long long)A.nky * (k - 1) + (i0 - 1);
  const V * twN = (const V *)A.twN;
  /* Z'_k and Z'_{M-k} from X_k and X_{M-k}, k = 1..M/2, put in LDS as they are formed: EPT / 2
   * pairs per thread, whose loads are issued together; and Z'_0 from X_0 and X_M by the first
   * ti threads */
  constexpr int GP = EPT / 2;
  const int npair = (M / 2) * ti;
  const bool ok0 = (int)threadIdx.x < ti && (int)threadIdx.x < nl;
  V x0 = tck_ld(ok0 ? &row[threadIdx.x] : S), xm = tck_ld(ok0 ? &row[threadIdx.x + (long long)g.nx * M] : S);
  for(int e0 = threadIdx.x; e0 < npair; e0 += GP * A.P.nt){
    V xa[GP], xb[GP];
    #pragma unroll
    for(int u = 0; u < GP; u++){
      const int e = e0 + u * A.P.nt;
      const int t = e & (ti - 1), k1 = 1 + (e >> lg);
      const bool ok = e < npair && t < nl;
      xa[u] = tck_ld(ok ? &row[t + (long long)g.nx * k1] : S);
      xb[u] = tck_ld(ok ? &row[t + (long long)g.nx * (M - k1)] : S);
    }
    #pragma unroll
    for(int u = 0; u < GP; u++){
      const int e = e0 + u * A.P.nt;
      if(e >= npair) break;
      const int t = e & (ti - 1), k1 = 1 + (e >> lg), k2 = M - k1;
      const V z1 = c2r_pre(xa[u], xb[u], twN[k1]);
      if(k2 != k1) sm[t * A.ld + fpad(k2)] = c2r_pre(xb[u], xa[u], twN[k2]);
      sm[t * A.ld + fpad(k1)] = z1;
    }
  }
  if((int)threadIdx.x < ti){
    x0.y = T(0.);
    xm.y = T(0.);
    sm[threadIdx.x * A.ld + fpad(0)] = c2r_pre(x0, xm, twN[0]);
  }
  fft_lds_barrier();
  /* element n of a line is psi at rows 2 n + 1 and 2 n + 2.  A thread's line is the same for all
   * its butterflies (the block size is a multiple of the tile width), so its wall copy is one
   * offset, and the z image of the first and last planes a uniform one; the y images are those
   * of elements 0 and M - 1 */
  const int i = i0 + ((int)threadIdx.x & (ti - 1));
  T * col = (T *)A.psi + tck_idx(g, i, 0, k);
  const int wall = i == 1 ? -1 : (i == g.nx ? 1 : 0);
  const long long dk = k == 1 ? g.plane * g.nz : (k == g.nz ? - g.plane * g.nz : 0);
  const auto put = [&](int j, T v){
    T * p = col + (long long)g.px * j;
    tck_st(p, v);
    if(wall) tck_st(&p[wall], v);
    if(dk){
      p[dk] = v;
      if(wall) p[dk + wall] = v;
    }
  };
  const auto store = [&](int t, int n, V v, bool ok){
    if(ok && t < nl){
      put(2 * n + 1, v.x);
      put(2 * n + 2, v.y);
      if(n == 0) put(g.ny + 1, v.x);
      if(n == M - 1) put(0, v.y);
    }
  };
  fft_mid<T, EPT, W>(sm, A.ld, ti, A.P, (const V *)A.twM, T(1.), 0, A.P.nst - 1);
  fft_last<T, EPT, W>(sm, A.ld, lg, A.P, (const V *)A.twM, T(1.), store);
}

/* Persistent exact form: the tiles cover the field exactly (nx a multiple of ti,
 * blockDim.x EPTK = ti M), so no load is conditional and the loops have fixed counts; the last
 * radix is RL.  The twiddle factors are read from LDS (after the
 * tile's lines); the pairs (X_k, X_{M-k}) of the next tile are loaded into registers before the
 * current tile's passes and stores, and forming Z' from them waits only for those loads (the
 * zero-size stores before the loop give its entry the outstanding loads-then-stores sequence of
 * an iteration's end, as in tck_zfft_p).  Bound by HBM (a read of the spectrum and a write of
 * psi).  One-tile form against this one, ms per step (three launches): FP64 512x1024x512
 * 4.07 -> 3.06, 256x512x512 0.82 -> 0.77, 128x1024x256 0.574 -> 0.448; FP32 512x1024x512
 * 2.26 -> 1.72, 128x1024x256 0.363 -> 0.297 */
template <typename T, int EPTK, int RL>
__global__ void __launch_bounds__(FFT_MAXTHREADS) tck_yifft_psi_p(const YInvArgs A){
  typedef typename cvec<T>::type V;
  extern __shared__ __align__(16) unsigned char fft_smem[];
  V * sm = (V *)fft_smem;
  constexpr int NP = EPTK / 2, NL = (EPTK + RL - 1) / RL;   /* pairs, last-pass butterflies per thread */
  constexpr bool ALL = NL * RL == EPTK;
  const tc_geom_t & g = A.g;
  const int ti = A.ti, lg = fft_lg(ti);
  const int M = A.P.M;
  const int nt = A.P.nt;
  const int ntx = g.nx / ti;
  const int ntiles = ntx * g.nz;
  const V * S = (const V *)A.S;
  T * psi = (T *)A.psi;
  V * twl = sm + ti * A.ld;
  V * twnl = twl + M;
  for(int t = threadIdx.x; t < M; t += nt){ twl[t] = ((const V *)A.twM)[t]; twnl[t] = ((const V *)A.twN)[t]; }
  fft_lds_barrier();   /* twnl is read for the first tile before any of the barriers of the loop */
  /* pair u of this thread: line t0, k1 = 1 + r0 + u dr; last-pass butterfly q: index r0 + q dr */
  const int t0i = (int)threadIdx.x & (ti - 1), r0i = (int)threadIdx.x >> lg, dr = nt >> lg;
  const int perl = M / RL;
  /* the thread row whose last-pass butterflies include the last one, perl - 1, whose last output
   * is element M - 1 and with it row ny (dr - 1 only where RL divides EPTK) */
  const int rlast = (perl - 1) % dr;
  int tile = blockIdx.x;               /* the launch has at least four tiles per block */
  /* buffer addressing: a tile's spectrum values lie in one plane of S (nky nx complex values) and
   * its psi values in one plane of the field, so each access is a per-thread byte offset that does
   * not change between tiles plus a uniform one */
  constexpr unsigned CB = sizeof(V), RB = sizeof(T);                 /* complex, real bytes */
  const unsigned ss = CB * (unsigned)(g.nx * dr);                    /* per u */
  const unsigned va = CB * (unsigned)(t0i + g.nx * (1 + r0i));       /* X_k1, u = 0 */
  const unsigned vb = CB * (unsigned)(t0i + g.nx * (M - 1 - r0i - (NP - 1) * dr));   /* X_{M-k1}, u = NP - 1 */
  const unsigned v0 = CB * (unsigned)t0i, vm = CB * (unsigned)(t0i + g.nx * M);
  const unsigned sbytes = CB * (unsigned)(g.nx * A.nky);
  const unsigned vp = RB * (unsigned)(t0i + 2 * g.px * r0i);         /* psi row 2 r0 + 1 */
  const unsigned sp = RB * (unsigned)g.px;
  const unsigned pbytes = RB * (unsigned)(g.px * g.ny);
  V xa[NP], xb[NP], x0, xm;
  #define YX_LOAD(tl) { \
    const __amdgpu_buffer_rsrc_t rs = tck_rsrc(S + (long long)((tl) % ntx * ti) + (long long)g.nx * A.nky * ((tl) / ntx), sbytes); \
    _Pragma("unroll") for(int u = 0; u < NP; u++){ xa[u] = tck_bldc<V>(rs, va, ss * u); xb[u] = tck_bldc<V>(rs, vb, ss * (NP - 1 - u)); } \
    x0 = tck_bldc<V>(rs, v0, 0u); \
    xm = tck_bldc<V>(rs, vm, 0u); }
  YX_LOAD(tile)
  {
    const __amdgpu_buffer_rsrc_t nul = tck_rsrc(A.S, 0u);
    #pragma unroll
    for(int q = 0; q < 2 * EPTK; q++) tck_bst0(nul, 16u * q);
  }
  for(;;){
    /* the LDS offsets are recomputed in every tile rather than held across the passes */
    int t0 = t0i, r0 = r0i;
    asm volatile("" : "+v"(t0), "+v"(r0));
    const int k = 1 + tile / ntx;
    const int i = 1 + (tile % ntx) * ti + t0;
    V * ln = sm + t0 * A.ld;
    #pragma unroll
    for(int u = 0; u < NP; u++){
      const int k1 = 1 + r0 + u * dr, k2 = M - k1;
      const V z1 = c2r_pre(xa[u], xb[u], twnl[k1]);
      if(k2 != k1) ln[fpad(k2)] = c2r_pre(xb[u], xa[u], twnl[k2]);
      ln[fpad(k1)] = z1;
    }
    if(r0 == 0){
      x0.y = T(0.);
      xm.y = T(0.);
      ln[fpad(0)] = c2r_pre(x0, xm, twnl[0]);
    }
    fft_lds_barrier();
    const int nxt = tile + (int)gridDim.x < ntiles ? tile + (int)gridDim.x : tile;
    YX_LOAD(nxt)
    fft_mid<T, EPTK, false>(sm, A.ld, ti, A.P, twl, T(1.), 0, A.P.nst - 1);
    V v[NL][RL];
    const __amdgpu_buffer_rsrc_t rp = tck_rsrc(psi + tck_idx(g, 1 + (tile % ntx) * ti, 1, k), pbytes);
    #pragma unroll
    for(int q = 0; q < NL; q++){
      const int jj = r0 + q * dr;
      if(!ALL && jj >= perl) break;
      #pragma unroll
      for(int r = 0; r < RL; r++){
        V x = ln[fpad(jj + r * perl)];
        if(r > 0){
          V w = twl[jj * r];
          w.y = - w.y;
          x = cmul(x, w);
        }
        v[q][r] = x;
      }
      dftr<RL, T>::run(v[q], T(1.));
      #pragma unroll
      for(int r = 0; r < RL; r++){
        tck_bstn<T>(rp, vp, sp * (unsigned)(2 * (q * dr + r * perl)), v[q][r].x);
        tck_bstn<T>(rp, vp, sp * (unsigned)(2 * (q * dr + r * perl) + 1), v[q][r].y);
      }
    }
    /* the halo images and wall copies of the threads that have any */
    if(i == 1 || i == g.nx || k == 1 || k == g.nz || r0 == 0 || r0 == rlast){
      T * col = psi + tck_idx(g, i, 0, k);
      const int wall = i == 1 ? -1 : (i == g.nx ? 1 : 0);
      const long long dk = k == 1 ? g.plane * g.nz : (k == g.nz ? - g.plane * g.nz : 0);
      const auto img = [&](int j, T x, bool self){
        T * p = col + (long long)g.px * j;
        if(self) *p = x;
        if(wall) tck_st(&p[wall], x);
        if(dk){
          p[dk] = x;
          if(wall) p[dk + wall] = x;
        }
      };
      #pragma unroll
      for(int q = 0; q < NL; q++){
        const int jj = r0 + q * dr;
        if(!ALL && jj >= perl) break;
        #pragma unroll
        for(int r = 0; r < RL; r++){
          const int n = jj + r * perl;
          img(2 * n + 1, v[q][r].x, false);
          img(2 * n + 2, v[q][r].y, false);
          if(r == 0 && n == 0) img(g.ny + 1, v[q][r].x, true);
          if(r == RL - 1 && n == M - 1) img(0, v[q][r].y, true);
        }
      }
    }
    tile += (int)gridDim.x;
    if(tile >= ntiles) break;
    fft_lds_barrier();
  }
  #undef YX_LOAD
}

/* ------------------------------------------------------------------------------------- */
extern "C" {

static int make_plan(int M, FftPlan * P){
  P->M = M;
  P->nst = 0;
  int n = M;
  while(n > 1){
    int r;
    if(n % 8 == 0) r = 8;
    else if(n % 4 == 0) r = 4;
    else if(n % 2 == 0) r = 2;
    else if(n % 3 == 0) r = 3;
    else if(n % 5 == 0) r = 5;
    else if(n % 7 == 0) r = 7;
    else return -1;
    if(P->nst >= FFT_MAXST) return -1;
    P->rad[P->nst++] = r;
    n /= r;
  }
  /* division multipliers of each stage (dividends stay below 16 * 4096 = 2^16) */
  int ns = 1;
  for(int st = 0; st < P->nst; st++){
    const unsigned per = (unsigned)(M / P->rad[st]);
    P->mper[st] = per > 1 ? (unsigned)(0x100000000ULL / per + 1) : 0u;
    P->mns[st] = ns > 1 ? (unsigned)(0x100000000ULL / (unsigned)ns + 1) : 0u;
    ns *= P->rad[st];
  }
  return 0;
}

int tck_fft_supported(int n){
  FftPlan P;
  return make_plan(n, &P) == 0;
}

/* the plan holds a radix 5 or 7 pass: the launch takes the kernels compiled with them */
static int plan_wide(const FftPlan * P){
  for(int q = 0; q < P->nst; q++) if(P->rad[q] == 5 || P->rad[q] == 7) return 1;
  return 0;
}

/* Tile of TB transforms of length M per block: TB = 16 (one 128 B line of doubles, or two
 * lines of complex values, per row access) when the LDS allows it, fewer for very long
 * transforms; threads = TB * M / FFT_EPT, or TB * M / (FFT_EPT / 2) for tiles so large that
 * the LDS holds too few blocks per CU (measured on the FP64 transforms of 512x1024x1024:
 * 7.2 -> 5.6 ms for the divergence + theta transform, 4.6 -> 3.7 ms for the inverse theta
 * transform; the FP32 tiles, already at 16 waves per CU, were slower with twice the
 * threads). */
#ifndef TCK_FFT_HALFEPT
#define TCK_FFT_HALFEPT 1    /* LDS-bound tiles: FFT_EPT / 2 elements per thread */
#endif
#ifndef TCK_FFT_YSHARE
#define TCK_FFT_YSHARE 1     /* theta transforms: blocks per CU the tiles are sized for */
#endif
#ifndef TCK_FFT_ZSHARE
#define TCK_FFT_ZSHARE 1     /* axial transforms */
#endif
static size_t g_lds_limit = 0;

static size_t lds_limit(void){
  if(g_lds_limit == 0){
    int dev = 0;
    if(hipGetDevice(&dev) != hipSuccess) dev = 0;
    int v = 0;
    if(hipDeviceGetAttribute(&v, hipDeviceAttributeSharedMemPerBlockOptin, dev) != hipSuccess || v <= 0){
      if(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0) v = 65536;
    }
    g_lds_limit = (size_t)v;
  }
  return g_lds_limit;
}

static int g_fft_ncu = 0;

static int fft_ncu(void){
  if(g_fft_ncu == 0){
    int dev = 0, v = 0;
    if(hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    g_fft_ncu = v;
  }
  return g_fft_ncu;
}

/* share: tiles sized to leave room for `share` blocks per CU in the LDS (while at least 4
 * transforms, 64 B of contiguous FP64 complex values, remain per row access).  lines: the
 * transforms of the launch; small launches take narrower tiles, so that there are at least
 * two blocks per CU, while a tile keeps 16 butterflies of 8 (a thread takes whole ones) */
/* LDS pitch of one padded line of M elements, odd so that the rows of a tile start in
 * different banks */
static int fft_ld(int M){
  const int ld = fpad(M - 1) + 1;
  return ld | 1;
}

/* the tile width b is a power of two (16 halved or doubled, capped at a power of two): the
 * kernels divide by it with shifts.  most: elements of a tile at most.  FFT_MOST is what a block
 * takes at all; the FP64 axial transforms keep to half of it, eight elements per thread: with
 * 16, which only tiles of 513 to 568, 1025 to 1137 and 2049 to 2275 rows would have, their first and
 * last passes spill, and narrower tiles are the quicker ones, ms per step of both directions (16
 * elements, 8): 128x256x540 0.948 / 0.690, 64x1120x560 1.83 / 1.29, 128x256x1080 2.01 / 1.78.
 * The theta transforms are not: 128x1080x256 divergence + theta 1.27 / 1.37, inverse 0.83 / 0.89 */
#define FFT_MOST (FFT_EPT * FFT_MAXTHREADS)
static int fft_tile(int M, int cap, size_t csize, int * threads, int share, long long lines, int most){
  int b = 16;
  const size_t lb = (size_t)fft_ld(M) * csize;
  while(b > 1 && ((size_t)b * lb > lds_limit() || b * M > most)) b /= 2;
  while(share > 1 && b > 4 && (size_t)b * lb * share > lds_limit()) b /= 2;
  while(b * 2 <= cap && b * 2 * M <= FFT_EPT * 64) b *= 2;   /* short transforms: wider tiles */
  while(b > 1 && b * M > 128 && lines / b < 2LL * fft_ncu()) b /= 2;
  if(b > cap) b = cap < 1 ? 1 : cap;
  /* elements per thread: FFT_EPT, or half that where the LDS holds so few blocks per CU that
   * FFT_EPT would leave fewer than 16 waves on it (FP64 tiles of long transforms: one block
   * per CU), and for every FP64 tile that 1024 threads cover so, because 16 elements do not fit in
   * a thread's registers beside a pass that loads or stores them.  The device passes loop over their
   * butterflies, so any count up to FFT_EPT computes the same bits. */
  int ept = FFT_EPT;
  const long long per = (long long)(lds_limit() / ((size_t)b * lb));
  const int w16 = ((b * M + FFT_EPT - 1) / FFT_EPT + 63) / 64;
  if(TCK_FFT_HALFEPT && (csize == sizeof(double2) || per * w16 < 16) && (b * M + FFT_EPT / 2 - 1) / (FFT_EPT / 2) <= FFT_MAXTHREADS) ept = FFT_EPT / 2;
  int t = (b * M + ept - 1) / ept;
  t = (t + 63) / 64 * 64;
  if(t < 64) t = 64;
  *threads = t;
  return b;
}

/* raises a kernel's dynamic LDS limit once per (kernel, size): later launches, including
 * those recorded into a graph, make no attribute call */
#define FFT_LDS_CACHE 32
static const void * g_lds_fn[FFT_LDS_CACHE];
static size_t g_lds_bytes[FFT_LDS_CACHE];
static int g_lds_n = 0;

static int set_lds(const void * fn, size_t bytes){
  if(bytes <= 65536) return 0;
  for(int q = 0; q < g_lds_n; q++) if(g_lds_fn[q] == fn && g_lds_bytes[q] >= bytes) return 0;
  if(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return -1;
  if(g_lds_n < FFT_LDS_CACHE){
    g_lds_fn[g_lds_n] = fn;
    g_lds_bytes[g_lds_n] = bytes;
    g_lds_n++;
  }
  return 0;
}

/* Persistent launches.  The kernels are compiled for ept elements per thread per pass
 * (FFT_EPT / 2, or FFT_EPT for the FP32 axial transforms); a launch qualifies when its threads
 * cover the tile at that count and it has at least four tiles per resident block.
 * Returns 1 when launched (the caller checks the launch), 0 when the caller should launch the
 * one-tile form, < 0 when the LDS limit could not be raised.  Resident blocks per CU are
 * queried once per (kernel, threads, LDS), so launches recorded into a graph make no query. */
#define PERSIST_EPT (FFT_EPT / 2)
#define PERSIST_CACHE 32
static const void * g_pc_fn[PERSIST_CACHE];
static int g_pc_nt[PERSIST_CACHE], g_pc_per[PERSIST_CACHE];
static size_t g_pc_lds[PERSIST_CACHE];
static int g_pc_n = 0;

}   /* extern "C" */

/* sets the kernel's LDS limit, then launches (lambda) */
template <typename F>
static int fft_one(const void * fn, F launch, size_t lds){
  if(set_lds(fn, lds)) return 1;
  launch();
  return 0;
}

template <typename Args>
static int launch_persistent(void (*kern)(const Args), const Args & A, int nt, size_t lds,
    long long elems, long long ntiles, hipStream_t stream, int ept = PERSIST_EPT){
  if((long long)nt * ept < elems || nt > FFT_MAXTHREADS) return 0;
  const void * fn = (const void *)kern;
  int per = 0;
  for(int q = 0; q < g_pc_n; q++) if(g_pc_fn[q] == fn && g_pc_nt[q] == nt && g_pc_lds[q] == lds) per = g_pc_per[q];
  if(per == 0){
    if(set_lds(fn, lds)) return -1;
    if(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, nt, lds) != hipSuccess || per < 1) per = 1;
    if(g_pc_n < PERSIST_CACHE){
      g_pc_fn[g_pc_n] = fn; g_pc_nt[g_pc_n] = nt; g_pc_lds[g_pc_n] = lds; g_pc_per[g_pc_n] = per;
      g_pc_n++;
    }
  }
  const long long nb = (long long)per * fft_ncu();
  if(ntiles < 4 * nb) return 0;
  if(set_lds(fn, lds)) return -1;
  hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(nt), lds, stream, A);
  return 1;
}

extern "C" {

/* the one-tile form of kernel K, compiled for E elements per thread per pass, for the transform
 * type T (E: float when mixed, else double) and radix set; nonzero when the LDS limit could not be
 * raised */
#define FFT_ONE_T(K, T, E, wide) ( \
  (wide) ? fft_one((const void *)K<T, E, true>, [&]{ hipLaunchKernelGGL((K<T, E, true>), grd, dim3(nt), lds, stream, A); }, lds) \
         : fft_one((const void *)K<T, E, false>, [&]{ hipLaunchKernelGGL((K<T, E, false>), grd, dim3(nt), lds, stream, A); }, lds))
#define FFT_ONE_E(K, E, mixed, wide) ((mixed) ? FFT_ONE_T(K, float, E, wide) : FFT_ONE_T(K, double, E, wide))

/* mixed: spectrum, transforms and psi in FP32 (twiddles twM, twN, tw as float2) */
int tck_launch_div_yfft(const tc_geom_t * g, const tc_coef_t * c, const double * ux,
    const double * uy, const double * uz, const double * dt, int rkstep, void * S,
    const void * twM, const void * twN, int mixed, hipStream_t stream){
  YFwdArgs A;
  A.g = *g; A.c = *c; A.ux = ux; A.uy = uy; A.uz = uz; A.dt = dt; A.rkstep = rkstep;
  A.S = S; A.nky = g->ny / 2 + 1;
  if(make_plan(g->ny / 2, &A.P) != 0) return (int)hipErrorInvalidValue;
  const size_t cs = mixed ? sizeof(float2) : sizeof(double2);
  int nt;
  A.ti = fft_tile(A.P.M, 64, cs, &nt, TCK_FFT_YSHARE, (long long)g->nx * g->nz, FFT_MOST);
  A.P.nt = nt;
  A.twM = twM; A.twN = twN;
  A.ld = fft_ld(A.P.M);
  const size_t lds = cs * (size_t)A.ti * A.ld;
  const long long ntiles = (long long)((g->nx + A.ti - 1) / A.ti) * g->nz;
  const dim3 grd((unsigned)ntiles);
  const long long el = (long long)A.ti * A.P.M;
  const bool wide = plan_wide(&A.P);
  if(mixed && (el + FFT_EPT / 2 - 1) / (FFT_EPT / 2) <= FFT_MAXTHREADS){
    nt = (int)(((el + FFT_EPT / 2 - 1) / (FFT_EPT / 2) + 63) / 64 * 64);
    A.P.nt = nt;
  }
  const bool half = (long long)nt * (FFT_EPT / 2) >= el;
  /* at most two waves per SIMD */
  const bool few = nt <= 256 && ntiles * (nt / 64) <= 8LL * fft_ncu();
  #define DIV_ONE(T, E, W, N) fft_one((const void *)tck_div_yfft<T, E, W, N>, [&]{ hipLaunchKernelGGL((tck_div_yfft<T, E, W, N>), grd, dim3(nt), lds, stream, A); }, lds)
  #define DIV_N(T, W) (half ? (few ? DIV_ONE(T, FFT_EPT / 2, W, 256) : nt <= 512 ? DIV_ONE(T, FFT_EPT / 2, W, 512) : DIV_ONE(T, FFT_EPT / 2, W, FFT_MAXTHREADS)) : DIV_ONE(T, FFT_EPT, W, FFT_MAXTHREADS))
  if(mixed ? (wide ? DIV_N(float, true) : DIV_N(float, false)) : (wide ? DIV_N(double, true) : DIV_N(double, false))) return (int)hipErrorInvalidValue;
  #undef DIV_N
  #undef DIV_ONE
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_launch_zfft(int nx, int nky, int nz, void * S, const void * tw, int sign, int mixed, int exact, hipStream_t stream){
  ZArgs A;
  A.nx = nx; A.nky = nky; A.nz = nz; A.S = S; A.tw = tw;
  A.sign = sign < 0 ? -1. : 1.;
  if(make_plan(nz, &A.P) != 0) return (int)hipErrorInvalidValue;
  const size_t cs = mixed ? sizeof(float2) : sizeof(double2);
  int nt;
  A.tz = fft_tile(nz, 64, cs, &nt, TCK_FFT_ZSHARE, (long long)nx * nky, mixed ? FFT_MOST : FFT_MOST / 2);
  A.P.nt = nt;
  A.ld = fft_ld(nz);
  const size_t lds = cs * (size_t)A.tz * A.ld;
  const long long ntiles = (long long)((nx + A.tz - 1) / A.tz) * nky;
  {
    const long long el = (long long)A.tz * nz;
    /* the exact form when the tiles cover the spectrum exactly, the plan starts with radix 8, has
     * two passes at least and no radix 5 or 7, and its twiddle factors fit in the LDS beside the
     * tile.  Where it does not hold (300x512x512), the one-tile form took 2.35 ms per step against
     * 2.79 ms of a persistent one with conditional accesses */
    const size_t ldsx = lds + cs * (size_t)nz;
    const int rl = A.P.rad[A.P.nst - 1];
    const bool x = exact && !plan_wide(&A.P) && A.P.nst >= 2 && A.P.rad[0] == 8 && nx % A.tz == 0 && ldsx <= lds_limit() && (long long)nt * (mixed ? FFT_EPT : PERSIST_EPT) == el
        && (!mixed || (long long)sizeof(float2) * nx * nky * nz < (1LL << 32));
    #define ZX(T, E) (rl == 8 ? launch_persistent(tck_zfft_p<T, E, 8>, A, nt, ldsx, el, ntiles, stream, E) \
        : rl == 4 ? launch_persistent(tck_zfft_p<T, E, 4>, A, nt, ldsx, el, ntiles, stream, E) \
        : rl == 3 ? launch_persistent(tck_zfft_p<T, E, 3>, A, nt, ldsx, el, ntiles, stream, E) \
                  : launch_persistent(tck_zfft_p<T, E, 2>, A, nt, ldsx, el, ntiles, stream, E))
    const int r = !x ? 0 : mixed ? ZX(float, FFT_EPT) : ZX(double, PERSIST_EPT);
    #undef ZX
    if(r < 0) return (int)hipErrorInvalidValue;
    if(r > 0){ TCK_CHECK_LAUNCH(); return 0; }
  }
  const dim3 grd((unsigned)ntiles);
  const bool wide = plan_wide(&A.P);
  /* FP64 tiles always have FFT_EPT / 2 elements per thread (fft_tile) */
  const bool half = !mixed || (long long)nt * (FFT_EPT / 2) >= (long long)A.tz * nz;
  if((long long)nt * (half ? FFT_EPT / 2 : FFT_EPT) < (long long)A.tz * nz) return (int)hipErrorInvalidValue;
  if(half ? FFT_ONE_E(tck_zfft, FFT_EPT / 2, mixed, wide) : FFT_ONE_T(tck_zfft, float, FFT_EPT, wide)) return (int)hipErrorInvalidValue;
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_launch_yifft_psi(const tc_geom_t * g, const void * S, void * psi, const void * twM,
    const void * twN, int mixed, int exact, hipStream_t stream){
  YInvArgs A;
  A.g = *g; A.S = S; A.psi = psi; A.nky = g->ny / 2 + 1;
  if(make_plan(g->ny / 2, &A.P) != 0) return (int)hipErrorInvalidValue;
  const size_t cs = mixed ? sizeof(float2) : sizeof(double2);
  int nt;
  A.ti = fft_tile(A.P.M, 64, cs, &nt, TCK_FFT_YSHARE, (long long)g->nx * g->nz, FFT_MOST);
  A.P.nt = nt;
  A.twM = twM; A.twN = twN;
  A.ld = fft_ld(A.P.M);
  const size_t lds = cs * (size_t)A.ti * A.ld;
  const long long ntiles = (long long)((g->nx + A.ti - 1) / A.ti) * g->nz;
  {
    const long long el = (long long)A.ti * A.P.M;
    /* the persistent form when the tiles cover the field exactly, the plan has two passes at least
     * and no radix 5 or 7, both twiddle tables fit in the LDS beside the tile and a plane's byte
     * offsets fit in 31 bits.  It is the faster one at every such FP64 size measured (128 to 1024
     * rows, one to four blocks per CU: by 1 to 25 %; with a last radix of 3, one-tile against
     * persistent, ms per step: 128x192x1024 0.333 and 0.332, 256x384x768 0.981 and 0.922,
     * 512x768x768 4.98 and 4.19), and in FP32 with a last radix other than 3 (1 to 24 %); with radix
     * 3, whose three butterflies per thread do not divide its 8 elements, FP32 256x384x768 takes
     * 0.654 ms against 0.596 ms per step */
    const size_t ldsx = lds + cs * (size_t)(2 * A.P.M);
    const int rl = A.P.rad[A.P.nst - 1];
    const int ntx = (int)(el / PERSIST_EPT);
    const bool x = exact && !plan_wide(&A.P) && A.P.nst >= 2 && A.P.M % 2 == 0 && g->nx % A.ti == 0
        && (!mixed || rl != 3) && ntx <= FFT_MAXTHREADS && ntx % 64 == 0 && (long long)ntx * PERSIST_EPT == el && ldsx <= lds_limit()
        && 16LL * g->plane < (1LL << 31) && 16LL * g->nx * A.nky < (1LL << 31);
    YInvArgs X = A;
    X.P.nt = ntx;
    #define YX(T) (rl == 8 ? launch_persistent(tck_yifft_psi_p<T, PERSIST_EPT, 8>, X, ntx, ldsx, el, ntiles, stream) \
        : rl == 4 ? launch_persistent(tck_yifft_psi_p<T, PERSIST_EPT, 4>, X, ntx, ldsx, el, ntiles, stream) \
                  : launch_persistent(tck_yifft_psi_p<T, PERSIST_EPT, 2>, X, ntx, ldsx, el, ntiles, stream))
    const int r = !x ? 0 : mixed ? YX(float)
        : rl == 3 ? launch_persistent(tck_yifft_psi_p<double, PERSIST_EPT, 3>, X, ntx, ldsx, el, ntiles, stream) : YX(double);
    #undef YX
    if(r < 0) return (int)hipErrorInvalidValue;
    if(r > 0){ TCK_CHECK_LAUNCH(); return 0; }
  }
  const dim3 grd((unsigned)ntiles);
  const bool half = (long long)nt * (FFT_EPT / 2) >= (long long)A.ti * A.P.M;
  if(half ? FFT_ONE_E(tck_yifft_psi, FFT_EPT / 2, mixed, plan_wide(&A.P)) : FFT_ONE_E(tck_yifft_psi, FFT_EPT, mixed, plan_wide(&A.P))) return (int)hipErrorInvalidValue;
  TCK_CHECK_LAUNCH();
  return 0;
}

}
