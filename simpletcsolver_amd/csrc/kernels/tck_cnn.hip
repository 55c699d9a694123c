/*
 * tck_cnn.hip -- the learned subgrid closure: a small 3-D CNN on the coarse grid (gfx950).
 *
 * No reference counterpart: the reference solves the flow on one grid only.  The network
 * maps (u, v, w, T, r) at the coarse cell centres to a 4-component correction of the
 * right-hand sides of ux, uy, uz and T.  Layers: 3x3x3 convolutions, 16 (padded inputs) ->
 * 32 -> 32 -> 4 channels, ReLU between; the x direction (walls) is zero-padded, y and z are
 * periodic like the flow.
 *
 * Activations are channels-last BF16 rows act[v][C], v = x + NX (y + NY (z + NZ b)) for
 * sample b of a batch.  The convolution is an implicit GEMM on the matrix cores
 * (v_mfma_f32_16x16x32_bf16, FP32 accumulation) over activation tiles staged in LDS with
 * their halo; so is the weight gradient, on tiles transposed in LDS.  Weights are
 * W[tap][co][ci] BF16 with FP32 master copies; biases FP32.
 *
 * Training: the backward data pass is the same convolution with the kernel flipped and its
 * channel roles exchanged (the adjoint of zero padding is zero padding, of periodic wrapping
 * periodic wrapping), so tck_cnn_conv serves both; the weight gradient is an FP32 reduction
 * over cells (per-block partial sums, then a fixed-order sum, so gradients are reproducible);
 * Adam updates the FP32 masters and re-rounds the BF16 copies.
 */
#include "tck_common.h"
#include <stdint.h>

typedef float cnn_f4 __attribute__((ext_vector_type(4)));

/* FP32 -> BF16, round to nearest even (inputs here are finite) */
__device__ __forceinline__ unsigned short cnn_bf16(float x){
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float cnn_f32(unsigned short h){
  return __uint_as_float(((uint32_t)h) << 16);
}

/* nb samples of nx x ny x nz cells, v = x + nx (y + ny (z + nz b)) */
struct CnnGrid { int nx, ny, nz, nb; long long nv; };

/* ---------------------------------------------------------------------------------------
 * convolution: out[v][co] = bias[co] + sum_tap sum_ci W[tap][co][ci] in[v + tap][ci]
 *   CI input channels (16 or 32), CO output channels (16 or 32) of which the first co_store
 *   are written, as the launch's mode says.
 *
 * Implicit GEMM on v_mfma_f32_16x16x32_bf16: A = 16 output channels by 32 K entries, B = 32 K
 * entries by 16 cells of an x row.  K is the 32 input channels of one tap (CI = 32), or the
 * 16 input channels of two taps (CI = 16, the 27th tap paired with zeros).  Lane l holds the
 * eight K entries 8 (l / 16) .. +7 of A row l % 16 and of B column l % 16 (the same K order on
 * both sides, which is all the product needs); the accumulator holds four consecutive
 * channels 4 (l / 16) .. +3 of cell l % 16, which go out as one 8- or 16-byte store.
 *
 * A block stages the kernel once (rows of CI BF16 padded by 16 bytes, so that the 16 lanes
 * reading one K group hit distinct banks) and loops over a run of tiles of 16 x CNN_TY x CNN_TZ
 * cells of one sample: each tile's activations with a one-cell halo (zero outside the walls in
 * x, periodic images in y and z) are staged in LDS with the same padded rows, the next tile's
 * on their way into registers during the products.  A wave takes the CNN_TY rows of one z; the
 * 18 input pieces (six rows, three x shifts) that a plane of taps needs are read once and
 * used by all rows and taps they reach, so that the plane's 72 products of a 32 -> 32 layer
 * read 36 pieces from LDS instead of 72.  The taps are added in the order of their index
 * whatever the tile, so the result does not depend on the tiling.
 *
 * Measured on a million cells (64 x 128 x 128): 86 us for 32 -> 32 channels (675 TFLOP/s), 58
 * us for 32 -> 16 and 63 us for 16 -> 32; reading each tap's operands from LDS again for every
 * row, with the halo images found by runtime division, took 149, 111 and 73 us.  LDS reads
 * and, on small grids, the staging bound it: 16, 11 and 13 us at 32 x 64 x 64, where each CU
 * has one tile (23, 18 and 14 us before; 18.5, 11.3 and 13.7 with the kernel's pieces in scratch).
 * ------------------------------------------------------------------------------------- */
struct ConvArgs {
  CnnGrid G;
  const unsigned short * in;     /* [nv][CI] bf16 */
  const unsigned short * w;      /* [27][CO][CI] bf16 */
  const float * bias;            /* [CO] or null */
  unsigned short * out_bf;       /* [nv][co_store] bf16 (CNN_RELU, CNN_RELU_BWD) */
  float * out_f;                 /* [nv][co_store] fp32 (CNN_PLAIN) */
  const unsigned short * act;    /* CNN_RELU_BWD: [nv][co_store] bf16, the layer's stored activations */
  float * bpart;                 /* CNN_RELU_BWD: [blocks][CO], sums of the gradient over a block's cells */
  int co_store;                  /* a multiple of 4 */
  int mode;
};

/* what becomes of an output value: stored FP32; max(0, .) stored BF16; or, in the backward data
 * pass, the gradient through the layer's ReLU (kept where its stored activation is positive),
 * stored BF16 for the next products, with the FP32 values summed for the bias gradient */
enum { CNN_PLAIN = 0, CNN_RELU = 1, CNN_RELU_BWD = 2 };

#define CNN_TY 4
/* depth of a tile, one wave per z: a block of 155 KB (32 input channels) or 93 KB (16) per CU.
 * For 16 input channels two blocks of depth 4 per CU were no faster (66 against 63 us for a
 * million cells) and slower where each CU has one tile (17.0 against 13.6 us at 32 x 64 x 64) */
#define CNN_TZ 8
#define CNN_HX 18                             /* halo'd tile: 16 + 2 cells in x */
#define CNN_HCELLS (CNN_HX * (CNN_TY + 2) * (CNN_TZ + 2))

typedef __bf16 cnn_b8 __attribute__((ext_vector_type(8)));

/* LDS bytes of the convolution of CI -> CO channels: the kernel and one halo'd tile */
__host__ __device__ constexpr int cnn_conv_lds(int ci, int co){
  return (27 * co + CNN_HCELLS) * (2 * ci + 16);
}

/* periodic image of a position at most one cell below the grid or some cells above it (the
 * halo and the unused rows of a tile); only grids thinner than a tile need the division */
__device__ __forceinline__ int cnn_wrap(int a, int n){
  if(a < 0) return a + n;
  if(a >= n){
    a -= n;
    if(a >= n) a %= n;
  }
  return a;
}

template <int CI, int CO>
__global__ void __launch_bounds__(CNN_TZ * TCK_WAVE) tck_cnn_conv(const ConvArgs A){
  constexpr int TZ = CNN_TZ, NTH = TZ * TCK_WAVE, HC = CNN_HCELLS;
  constexpr int RS = 2 * CI + 16;                 /* padded row: bytes per cell or per co */
  constexpr int NT = CO / 16;                     /* 16-channel output blocks */
  constexpr int PC = CI / 8;                      /* 16-byte pieces per row */
  constexpr int NP = (HC * PC + NTH - 1) / NTH;   /* tile pieces per thread */
  constexpr int NW = (27 * CO * PC + NTH - 1) / NTH;      /* kernel pieces per thread */
  extern __shared__ __align__(16) unsigned char cnn_smem[];
  unsigned char * wl = cnn_smem;                  /* [27][CO] rows */
  unsigned char * al = cnn_smem + 27 * CO * RS;   /* [HZ][HY][HX] rows */
  const int lane = threadIdx.x % TCK_WAVE;
  const int wv = threadIdx.x / TCK_WAVE;          /* z within the tile */
  const int kg = lane / 16;                       /* this lane's K group */
  const int cl = lane % 16;                       /* A row (channel) / B column (cell in x) */
  const CnnGrid & G = A.G;
  const int ntx = (G.nx + 15) / 16, nty = (G.ny + CNN_TY - 1) / CNN_TY, ntz = (G.nz + TZ - 1) / TZ;
  const int ntiles = ntx * nty * ntz * G.nb;
  /* a contiguous run of tiles per block, neighbouring runs on the same XCD */
  const int per = (ntiles + (int)gridDim.x - 1) / (int)gridDim.x;
  int run = blockIdx.x;
  if(gridDim.x % TCK_NXCD == 0) run = (run % TCK_NXCD) * ((int)gridDim.x / TCK_NXCD) + run / TCK_NXCD;
  const int t0 = run * per, t1 = min(t0 + per, ntiles);
  uint4 pre[NP];
  auto fetch = [&](int tile){
    int r = tile / ntx;
    const int x0 = 16 * (tile % ntx), y0 = CNN_TY * (r % nty);
    r /= nty;
    const int z0 = TZ * (r % ntz), b = r / ntz;
    #pragma unroll
    for(int q = 0; q < NP; q++){
      const int e = threadIdx.x + q * NTH;
      const int c = e / PC, pc = e % PC;
      const int hx = c % CNN_HX, hy = (c / CNN_HX) % (CNN_TY + 2), hz = c / (CNN_HX * (CNN_TY + 2));
      const int xx = x0 + hx - 1;
      pre[q] = uint4{0u, 0u, 0u, 0u};
      if(c < HC && xx >= 0 && xx < G.nx){
        const int yy = cnn_wrap(y0 + hy - 1, G.ny), zz = cnn_wrap(z0 + hz - 1, G.nz);
        const long long src = (long long)xx + (long long)G.nx * ((long long)yy + (long long)G.ny * ((long long)zz + (long long)G.nz * b));
        pre[q] = *(const uint4 *)(A.in + src * CI + 8 * pc);
      }
    }
  };
  if(t0 < t1) fetch(t0);
  {
    /* loaded without a condition: an element written only under one stays in scratch memory */
    uint4 wp[NW];
    #pragma unroll
    for(int q = 0; q < NW; q++){
      const int e = threadIdx.x + q * NTH;
      wp[q] = *(const uint4 *)(A.w + 8LL * (e < 27 * CO * PC ? e : 0));
    }
    #pragma unroll
    for(int q = 0; q < NW; q++){
      const int e = threadIdx.x + q * NTH;
      if(e < 27 * CO * PC) *(uint4 *)(wl + (e / PC) * RS + 16 * (e % PC)) = wp[q];
    }
  }
  cnn_f4 bsum[NT];
  #pragma unroll
  for(int t = 0; t < NT; t++) bsum[t] = cnn_f4{0.f, 0.f, 0.f, 0.f};
  for(int tile = t0; tile < t1; tile++){
    int r = tile / ntx;
    const int x0 = 16 * (tile % ntx), y0 = CNN_TY * (r % nty);
    r /= nty;
    const int z0 = TZ * (r % ntz), b = r / ntz;
    __syncthreads();                              /* the previous tile's reads are done */
    #pragma unroll
    for(int q = 0; q < NP; q++){
      const int e = threadIdx.x + q * NTH;
      if(e < HC * PC) *(uint4 *)(al + (e / PC) * RS + 16 * (e % PC)) = pre[q];
    }
    __syncthreads();
    if(tile + 1 < t1) fetch(tile + 1);
    /* the stored activations of the wave's cells, in flight during the products */
    ushort4 act[CNN_TY][NT];
    if(A.mode == CNN_RELU_BWD){
      #pragma unroll
      for(int q = 0; q < CNN_TY; q++){
        const int x = x0 + cl, y = y0 + q, z = z0 + wv;
        const bool in = x < G.nx && y < G.ny && z < G.nz;
        const long long v = in ? (long long)x + (long long)G.nx * ((long long)y + (long long)G.ny * ((long long)z + (long long)G.nz * b)) : 0;
        #pragma unroll
        for(int t = 0; t < NT; t++){
          const int co = 16 * t + 4 * kg;
          act[q][t] = *(const ushort4 *)(A.act + v * A.co_store + (co < A.co_store ? co : 0));
        }
      }
    }
    cnn_f4 acc[CNN_TY][NT];
    #pragma unroll
    for(int q = 0; q < CNN_TY; q++)
      #pragma unroll
      for(int t = 0; t < NT; t++) acc[q][t] = cnn_f4{0.f, 0.f, 0.f, 0.f};
    if constexpr (CI == 32){
      #pragma unroll 1
      for(int dz = 0; dz < 3; dz++){
        const unsigned char * ap = al + (cl + CNN_HX * ((CNN_TY + 2) * (wv + dz))) * RS + 16 * kg;
        const unsigned char * wp = wl + (9 * dz * CO + cl) * RS + 16 * kg;
        cnn_b8 av[CNN_TY + 2][3];
        #pragma unroll
        for(int hy = 0; hy < CNN_TY + 2; hy++)
          #pragma unroll
          for(int dx = 0; dx < 3; dx++) av[hy][dx] = *(const cnn_b8 *)(ap + (dx + CNN_HX * hy) * RS);
        #pragma unroll
        for(int tp = 0; tp < 9; tp++){
          cnn_b8 bw[NT];
          #pragma unroll
          for(int t = 0; t < NT; t++) bw[t] = *(const cnn_b8 *)(wp + (tp * CO + 16 * t) * RS);
          #pragma unroll
          for(int q = 0; q < CNN_TY; q++)
            #pragma unroll
            for(int t = 0; t < NT; t++)
              acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[t], av[q + tp / 3][tp % 3], acc[q][t], 0, 0, 0);
        }
      }
    }else{
      /* K group kg reads tap 2 s + (kg >> 1), channels 8 (kg & 1) .. +7: fully unrolled, so that
       * a step's input offset is one select between two constants */
      const int odd = kg >> 1;
      const unsigned char * ap = al + (cl + CNN_HX * ((CNN_TY + 2) * wv)) * RS + 16 * (kg & 1);
      const unsigned char * wp = wl + (odd * CO + cl) * RS + 16 * (kg & 1);
      #pragma unroll
      for(int s = 0; s < 14; s++){
        constexpr int HP = CNN_HX * (CNN_TY + 2);
        const int ta = 2 * s, tb = 2 * s + 1 < 27 ? 2 * s + 1 : 26;
        const int oa = (ta % 3 + CNN_HX * ((ta / 3) % 3) + HP * (ta / 9)) * RS;
        const int ob = (tb % 3 + CNN_HX * ((tb / 3) % 3) + HP * (tb / 9)) * RS;
        const unsigned char * as = ap + (odd ? ob : oa);
        cnn_b8 bw[NT];
        #pragma unroll
        for(int t = 0; t < NT; t++){
          /* the last step's odd half has no tap: zeros (its read stays on tap 26) */
          if(s == 13){
            bw[t] = *(const cnn_b8 *)(wl + (26 * CO + cl + 16 * t) * RS + 16 * (kg & 1));
            if(odd) bw[t] = cnn_b8{};
          }else bw[t] = *(const cnn_b8 *)(wp + (ta * CO + 16 * t) * RS);
        }
        #pragma unroll
        for(int q = 0; q < CNN_TY; q++){
          const cnn_b8 av = *(const cnn_b8 *)(as + CNN_HX * q * RS);
          #pragma unroll
          for(int t = 0; t < NT; t++) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[t], av, acc[q][t], 0, 0, 0);
        }
      }
    }
    /* accumulator: channels 16 t + 4 kg .. +3 of cell x0 + cl of the row */
    #pragma unroll
    for(int q = 0; q < CNN_TY; q++){
      const int x = x0 + cl, y = y0 + q, z = z0 + wv;
      if(x >= G.nx || y >= G.ny || z >= G.nz) continue;
      const long long v = (long long)x + (long long)G.nx * ((long long)y + (long long)G.ny * ((long long)z + (long long)G.nz * b));
      #pragma unroll
      for(int t = 0; t < NT; t++){
        const int co = 16 * t + 4 * kg;
        if(co >= A.co_store) continue;
        cnn_f4 val = acc[q][t];
        if(A.bias) val += *(const cnn_f4 *)(A.bias + co);
        if(A.mode == CNN_PLAIN){
          *(cnn_f4 *)(A.out_f + v * A.co_store + co) = val;
          continue;
        }
        if(A.mode == CNN_RELU){
          #pragma unroll
          for(int u = 0; u < 4; u++) val[u] = val[u] > 0.f ? val[u] : 0.f;
        }else{
          const ushort4 a = act[q][t];
          val[0] = cnn_f32(a.x) > 0.f ? val[0] : 0.f;
          val[1] = cnn_f32(a.y) > 0.f ? val[1] : 0.f;
          val[2] = cnn_f32(a.z) > 0.f ? val[2] : 0.f;
          val[3] = cnn_f32(a.w) > 0.f ? val[3] : 0.f;
          bsum[t] += val;
        }
        *(ushort4 *)(A.out_bf + v * A.co_store + co) = make_ushort4(cnn_bf16(val[0]), cnn_bf16(val[1]), cnn_bf16(val[2]), cnn_bf16(val[3]));
      }
    }
  }
  if(A.mode != CNN_RELU_BWD) return;
  /* the block's sums: over the 16 cells of a wave's lanes, then over the waves in order */
  __syncthreads();
  float * red = (float *)al;                      /* [waves][CO] */
  #pragma unroll
  for(int t = 0; t < NT; t++)
    #pragma unroll
    for(int u = 0; u < 4; u++){
      float v = bsum[t][u];
      for(int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, TCK_WAVE);
      if(cl == 0) red[wv * CO + 16 * t + 4 * kg + u] = v;
    }
  __syncthreads();
  if((int)threadIdx.x < CO){
    float v = 0.f;
    for(int w = 0; w < TZ; w++) v += red[w * CO + threadIdx.x];
    A.bpart[(long long)blockIdx.x * CO + threadIdx.x] = v;
  }
}

/* ---------------------------------------------------------------------------------------
 * weight gradient on the matrix cores: for each tap a GEMM over cells,
 *   part[blk][tap][co][ci] = sum over the block's cells v of g[v][co] * in[v + tap][ci]
 * (FP32), then a fixed-order sum over blocks.
 *
 * K of the product is the cells, while activations are channels-last, so a block transposes
 * a tile of 16 x 4 x 4 cells into LDS rows of one channel along x: g without a halo, the inputs
 * with a one-cell halo (periodic images in y and z, zeros past the walls; cells outside the
 * grid have g = 0).  A lane then reads its eight K entries (consecutive x of one channel) as one
 * 16-byte piece; the taps dx = -1 and +1 are the same piece shifted by one element, formed from
 * its neighbour words in registers, so one read of the inputs serves the three taps of a
 * (dy, dz) pair.  One wave per (dy, dz), nine per block, each holding the accumulators of its
 * three taps; a block loops over a contiguous run of tiles with the next tile's loads in
 * flight during the products.  An input row of a channel is 16 cells, the cell past them and,
 * at the end of the row's 24 slots, the cell before the next row's; the channel pitches
 * are 4 and 52 mod 64 words, so that the 16 lanes of a K group read distinct banks.
 *
 * Measured on a batch of 4 of 32 x 64 x 64 cells (29 GFLOP for 32 -> 32 channels): 50 us for
 * 32 -> 32 (580 TFLOP/s), 39 us for 32 -> 16 and 30 us for 16 -> 32; gathering every tap's
 * operands from memory as 2-byte loads took 675, 745 and 741 us.
 * ------------------------------------------------------------------------------------- */
struct WgradArgs {
  CnnGrid G;
  const unsigned short * in;   /* [nv][CI] bf16 */
  const unsigned short * g;    /* [nv][CO] bf16 */
  float * part;                /* [nblk][27][CO][CI] */
};

#define CNN_WG_THREADS 576                    /* nine waves */
#define CNN_WG_ROWS 36                        /* halo'd rows of a tile: 6 in y, 6 in z */
#define CNN_WG_PITCH (8 + 24 * CNN_WG_ROWS)   /* elements per channel of the input tile */
#define CNN_WG_GPITCH (256 + 8)               /* elements per channel of the gradient tile */
#define CNN_WG_PAIRS (10 * CNN_WG_ROWS)       /* x pairs of the input tile */

__host__ __device__ constexpr int cnn_wgrad_lds(int ci, int co){
  return 2 * (ci * CNN_WG_PITCH + co * CNN_WG_GPITCH);
}

/* the same channel of two neighbouring cells, as one word */
__device__ __forceinline__ uint32_t cnn_pair(uint32_t a, uint32_t b, int hi){
  return hi ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
}

/* a and b: eight channels of two neighbouring cells -> the word at slot `at` of each of the
 * eight channel rows */
__device__ __forceinline__ void cnn_put_pair(uint32_t * at, int pitch_words, uint4 a, uint4 b){
  const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
  #pragma unroll
  for(int q = 0; q < 8; q++) at[q * pitch_words] = cnn_pair(aw[q >> 1], bw[q >> 1], q & 1);
}

template <int CI, int CO>
__global__ void __launch_bounds__(CNN_WG_THREADS) tck_cnn_wgrad(const WgradArgs A){
  constexpr int NT = CO / 16, NS = CI / 16;
  constexpr int NI = (CNN_WG_PAIRS * (CI / 8) + CNN_WG_THREADS - 1) / CNN_WG_THREADS;   /* input pieces per thread */
  constexpr int NG = (128 * (CO / 8) + CNN_WG_THREADS - 1) / CNN_WG_THREADS;
  extern __shared__ __align__(16) unsigned char cnn_smem[];
  unsigned short * il = (unsigned short *)cnn_smem;     /* [CI][CNN_WG_PITCH] */
  unsigned short * gl = il + CI * CNN_WG_PITCH;         /* [CO][CNN_WG_GPITCH] */
  const CnnGrid & G = A.G;
  const int lane = threadIdx.x % TCK_WAVE, wv = threadIdx.x / TCK_WAVE;
  const int dy = wv % 3, dz = wv / 3;                   /* halo offsets 0..2 */
  const int kg = lane / 16, cl = lane % 16;
  const int ntx = (G.nx + 15) / 16, nty = (G.ny + 3) / 4, ntz = (G.nz + 3) / 4;
  const int ntiles = ntx * nty * ntz * G.nb;
  const int per = (ntiles + (int)gridDim.x - 1) / (int)gridDim.x;
  const int t0 = blockIdx.x * per, t1 = min(t0 + per, ntiles);
  cnn_f4 acc[3][NT][NS];
  #pragma unroll
  for(int d = 0; d < 3; d++)
    #pragma unroll
    for(int t = 0; t < NT; t++)
      #pragma unroll
      for(int u = 0; u < NS; u++) acc[d][t][u] = cnn_f4{0.f, 0.f, 0.f, 0.f};
  const uint4 zero = {0u, 0u, 0u, 0u};
  uint4 ia[NI], ib[NI], ga[NG], gb[NG];
  /* a tile's pieces into registers: pairs of neighbouring cells, eight channels each */
  auto fetch = [&](int tile){
    const int tx = tile % ntx;
    int r = tile / ntx;
    const int ty = r % nty; r /= nty;
    const int tz = r % ntz, b = r / ntz;
    const int x0 = 16 * tx, y0 = 4 * ty, z0 = 4 * tz;
    #pragma unroll
    for(int q = 0; q < NI; q++){
      const int e = threadIdx.x + q * CNN_WG_THREADS;
      const int c = e % (CI / 8), pr = e / (CI / 8);
      const int p = pr % 10, row = pr / 10;
      ia[q] = zero; ib[q] = zero;
      if(row < CNN_WG_ROWS){
        const int y = cnn_wrap(y0 + row % 6 - 1, G.ny), z = cnn_wrap(z0 + row / 6 - 1, G.nz);
        const int xa = x0 + 2 * p - 2;                  /* the pair's cells: xa, xa + 1 */
        const unsigned short * src = A.in + (long long)G.nx * ((long long)y + (long long)G.ny * ((long long)z + (long long)G.nz * b)) * CI + 8 * c;
        if(p > 0 && xa < G.nx) ia[q] = *(const uint4 *)(src + (long long)xa * CI);
        if(p < 9 && xa + 1 >= 0 && xa + 1 < G.nx) ib[q] = *(const uint4 *)(src + (long long)(xa + 1) * CI);
      }
    }
    #pragma unroll
    for(int q = 0; q < NG; q++){
      const int e = threadIdx.x + q * CNN_WG_THREADS;
      const int c = e % (CO / 8), pr = e / (CO / 8);
      const int x = x0 + 2 * (pr % 8), y = y0 + (pr / 8) % 4, z = z0 + pr / 32;
      ga[q] = zero; gb[q] = zero;
      if(pr < 128 && y < G.ny && z < G.nz){
        const unsigned short * src = A.g + ((long long)x + (long long)G.nx * ((long long)y + (long long)G.ny * ((long long)z + (long long)G.nz * b))) * CO + 8 * c;
        if(x < G.nx) ga[q] = *(const uint4 *)src;
        if(x + 1 < G.nx) gb[q] = *(const uint4 *)(src + CO);
      }
    }
  };
  if(t0 < t1) fetch(t0);
  for(int tile = t0; tile < t1; tile++){
    __syncthreads();                                    /* the previous tile's reads are done */
    #pragma unroll
    for(int q = 0; q < NI; q++){
      const int e = threadIdx.x + q * CNN_WG_THREADS;
      const int c = e % (CI / 8), pr = e / (CI / 8);
      const int p = pr % 10, row = pr / 10;
      if(row < CNN_WG_ROWS)
        cnn_put_pair((uint32_t *)il + (8 * c * CNN_WG_PITCH + 8 + 24 * row + 2 * p - 2) / 2, CNN_WG_PITCH / 2, ia[q], ib[q]);
    }
    #pragma unroll
    for(int q = 0; q < NG; q++){
      const int e = threadIdx.x + q * CNN_WG_THREADS;
      const int c = e % (CO / 8), pr = e / (CO / 8);
      if(pr < 128) cnn_put_pair((uint32_t *)gl + (8 * c * CNN_WG_GPITCH + 2 * pr) / 2, CNN_WG_GPITCH / 2, ga[q], gb[q]);
    }
    __syncthreads();
    if(tile + 1 < t1) fetch(tile + 1);
    /* 32 cells (two rows) per product: K entries 8 kg .. +7 are cells 8 (kg % 2) .. +7 of row
     * kg / 2 of the two */
    #pragma unroll 2
    for(int s = 0; s < 8; s++){
      const int ry = (2 * s + (kg >> 1)) % 4, rz = (2 * s) / 4;
      const int at = 8 + 24 * (ry + dy + 6 * (rz + dz)) + 8 * (kg & 1);
      cnn_b8 av[NT];
      #pragma unroll
      for(int t = 0; t < NT; t++) av[t] = *(const cnn_b8 *)(gl + (16 * t + cl) * CNN_WG_GPITCH + 32 * s + 8 * kg);
      #pragma unroll
      for(int u = 0; u < NS; u++){
        const unsigned short * row = il + (16 * u + cl) * CNN_WG_PITCH + at;
        const uint4 w = *(const uint4 *)row;
        const uint32_t before = *(const uint32_t *)(row - 2), after = *(const uint32_t *)(row + 8);
        uint4 m, n;                                     /* the cells one to the left and one to the right */
        m.x = __builtin_amdgcn_alignbit(w.x, before, 16);
        m.y = __builtin_amdgcn_alignbit(w.y, w.x, 16);
        m.z = __builtin_amdgcn_alignbit(w.z, w.y, 16);
        m.w = __builtin_amdgcn_alignbit(w.w, w.z, 16);
        n.x = m.y; n.y = m.z; n.z = m.w;
        n.w = __builtin_amdgcn_alignbit(after, w.w, 16);
        const cnn_b8 bl = __builtin_bit_cast(cnn_b8, m), b0 = __builtin_bit_cast(cnn_b8, w), br = __builtin_bit_cast(cnn_b8, n);
        #pragma unroll
        for(int t = 0; t < NT; t++){
          acc[0][t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t], bl, acc[0][t][u], 0, 0, 0);
          acc[1][t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t], b0, acc[1][t][u], 0, 0, 0);
          acc[2][t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t], br, acc[2][t][u], 0, 0, 0);
        }
      }
    }
  }
  /* accumulator [d][t][u][q]: tap d + 3 dy + 9 dz, co = 16 t + 4 kg + q, ci = 16 u + cl */
  #pragma unroll
  for(int d = 0; d < 3; d++){
    float * out = A.part + ((long long)blockIdx.x * 27 + d + 3 * dy + 9 * dz) * (CO * CI);
    #pragma unroll
    for(int t = 0; t < NT; t++)
      #pragma unroll
      for(int u = 0; u < NS; u++)
        #pragma unroll
        for(int q = 0; q < 4; q++) out[(16 * t + 4 * kg + q) * CI + 16 * u + cl] = acc[d][t][u][q];
  }
}

/* The fixed-order sums of the per-block partial results of all layers in one launch:
 * out[e] = sum_b part[b][e].  A block takes 64 entries of one segment; its four waves sum a
 * quarter of the partials each, in order, eight loads at a time, and the quarters are added
 * in order. */
#define CNN_NSEG 6
struct ReduceArgs {
  const float * part[CNN_NSEG];
  float * out[CNN_NSEG];
  int n[CNN_NSEG], nblk[CNN_NSEG];
  int first[CNN_NSEG + 1];     /* first block of each segment */
};

__global__ void __launch_bounds__(256) tck_cnn_reduce(const ReduceArgs A){
  __shared__ float red[4][64];
  int sg = 0;
  while(sg + 1 < CNN_NSEG && (int)blockIdx.x >= A.first[sg + 1]) sg++;
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  const int n = A.n[sg], nblk = A.nblk[sg];
  const int e = ((int)blockIdx.x - A.first[sg]) * 64 + lane;
  const int q = (nblk + 3) / 4;
  const int b1 = min((w + 1) * q, nblk);
  int b = w * q;
  float s = 0.f;
  if(e < n){
    const float * p = A.part[sg] + e;
    for(; b + 8 <= b1; b += 8){
      float v[8];
      #pragma unroll
      for(int u = 0; u < 8; u++) v[u] = p[(long long)(b + u) * n];
      #pragma unroll
      for(int u = 0; u < 8; u++) s += v[u];
    }
    for(; b < b1; b++) s += p[(long long)b * n];
  }
  red[w][lane] = s;
  __syncthreads();
  if(w == 0 && e < n) A.out[sg][e] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

/* ---------------------------------------------------------------------------------------
 * elementwise pieces
 * ------------------------------------------------------------------------------------- */
/* loss = mean over cells and the four channels of (pred - target)^2, and its gradient: one
 * cell per thread and iteration.  g: the gradient as BF16 rows of 16 channels (4 used, the
 * others zero), the operand of the backward products; bpart, lpart: per-block sums of the FP32
 * gradient (16 entries) and of the squares */
__global__ void __launch_bounds__(256) tck_cnn_mse(const float4 * pred, const float4 * target, long long nv,
    float scale, unsigned short * g, float * bpart, float * lpart){
  __shared__ float red[256][5];
  float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
  for(long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (long long)gridDim.x * blockDim.x){
    const float4 p = pred[v], t = target[v];
    const float d[4] = {p.x - t.x, p.y - t.y, p.z - t.z, p.w - t.w};
    uint32_t h[4];
    #pragma unroll
    for(int c = 0; c < 4; c++){
      const float gr = 2.f * d[c] * scale;
      h[c] = cnn_bf16(gr);
      s[c] += gr;
      s[4] += d[c] * d[c];
    }
    uint4 * row = (uint4 *)(g + v * 16);
    row[0] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), 0u, 0u);
    row[1] = make_uint4(0u, 0u, 0u, 0u);
  }
  #pragma unroll
  for(int c = 0; c < 5; c++) red[threadIdx.x][c] = s[c];
  __syncthreads();
  for(int h = 128; h > 0; h >>= 1){
    if((int)threadIdx.x < h){
      #pragma unroll
      for(int c = 0; c < 5; c++) red[threadIdx.x][c] += red[threadIdx.x + h][c];
    }
    __syncthreads();
  }
  if(threadIdx.x < 16) bpart[blockIdx.x * 16 + threadIdx.x] = threadIdx.x < 4 ? red[0][threadIdx.x] : 0.f;
  if(threadIdx.x == 16) lpart[blockIdx.x] = red[0][4];
}

/* network inputs as the caller gives them, [nv][5] FP32, to the BF16 rows of 16 channels the
 * first convolution reads (channels 5..15 zero).  One cell per thread: the rows are formed
 * here rather than on the host, which took 5.5 ms for a million cells against 20 us, and 20
 * bytes per cell cross PCIe instead of 32 */
__global__ void __launch_bounds__(256) tck_cnn_pack(const float * x, long long nv, unsigned short * out){
  for(long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (long long)gridDim.x * blockDim.x){
    uint32_t h[5];
    #pragma unroll
    for(int q = 0; q < 5; q++) h[q] = cnn_bf16(x[v * 5 + q]);
    uint4 * row = (uint4 *)(out + v * 16);
    row[0] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4], 0u);
    row[1] = make_uint4(0u, 0u, 0u, 0u);
  }
}

/* FP32 -> BF16 copy */
__global__ void tck_cnn_to_bf16(const float * x, long long n, unsigned short * y){
  for(long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x)
    y[e] = cnn_bf16(x[e]);
}

/* adjoint kernel for the backward data pass: Wt[26 - tap][ci][co] = W[tap][co][ci]
 * (co, ci padded in the transposed tensor to co_p, ci_p with zeros) */
__global__ void tck_cnn_flip(const unsigned short * w, int co_n, int ci_n, int ci_p, int co_p, unsigned short * wt){
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = 27 * ci_p * co_p;
  if(e >= n) return;
  const int co = e % co_p;                /* wt's input channel */
  const int ci = (e / co_p) % ci_p;       /* wt's output channel */
  const int tap = e / (co_p * ci_p);
  unsigned short v = 0;
  if(co < co_n && ci < ci_n) v = w[((long long)(26 - tap) * co_n + co) * ci_n + ci];
  wt[e] = v;
}

/* Adam on the FP32 masters of all layers in one launch (one segment per blockIdx.y); weights
 * are re-rounded to their BF16 copies, the plain one and the flipped one of the backward data
 * pass (tck_cnn_flip) */
struct AdamArgs {
  float * w[CNN_NSEG]; float * m[CNN_NSEG]; float * v[CNN_NSEG];
  const float * g[CNN_NSEG];
  unsigned short * wbf[CNN_NSEG]; unsigned short * wt[CNN_NSEG];   /* or null */
  int n[CNN_NSEG], co[CNN_NSEG], ci[CNN_NSEG];
  float lr, b1, b2, eps, c1, c2;
};

__global__ void __launch_bounds__(256) tck_cnn_adam(const AdamArgs A){
  const int sg = blockIdx.y;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if(e >= A.n[sg]) return;
  const float gg = A.g[sg][e];
  const float mm = A.b1 * A.m[sg][e] + (1.f - A.b1) * gg;
  const float vv = A.b2 * A.v[sg][e] + (1.f - A.b2) * gg * gg;
  A.m[sg][e] = mm;
  A.v[sg][e] = vv;
  const float upd = A.lr * (mm / A.c1) / (sqrtf(vv / A.c2) + A.eps);
  const float w = A.w[sg][e] - upd;
  A.w[sg][e] = w;
  if(A.wbf[sg]){
    const unsigned short h = cnn_bf16(w);
    A.wbf[sg][e] = h;
    if(A.wt[sg]){
      const int ci = A.ci[sg], co = A.co[sg];
      const int ic = e % ci, oc = (e / ci) % co, tap = e / (ci * co);
      A.wt[sg][((26 - tap) * ci + ic) * co + oc] = h;
    }
  }
}

/* ---------------------------------------------------------------------------------------
 * coupling with the flow (device layout of tc_shared.h)
 * ------------------------------------------------------------------------------------- */
struct GatherArgs {
  tc_geom_t g;
  const double * ux; const double * uy; const double * uz; const double * t;
  const double * xc;        /* XC(i) at [i] */
  float mean[5], inv_std[5];
  unsigned short * out;     /* [nv][16] bf16: u v w T r, channels 5..15 zero */
};

/* network input at cell centres: u = (UX(i) + UX(i+1)) / 2, v = UY, w = UZ, T, r = XC(i) */
__global__ void tck_cnn_gather(const GatherArgs A){
  const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 1 + blockIdx.y;
  const int k = 1 + blockIdx.z;
  if(i > A.g.nx) return;
  const long long o = tck_idx(A.g, i, j, k);
  float c[5];
  c[0] = (float)(0.5 * A.ux[o] + 0.5 * A.ux[o + 1]);
  c[1] = (float)A.uy[o];
  c[2] = (float)A.uz[o];
  c[3] = A.t ? (float)A.t[o] : 0.f;
  c[4] = (float)A.xc[i];
  const long long v = (long long)(i - 1) + (long long)A.g.nx * ((long long)(j - 1) + (long long)A.g.ny * (k - 1));
  unsigned short * p = A.out + v * 16;
  #pragma unroll
  for(int q = 0; q < 5; q++) p[q] = cnn_bf16((c[q] - A.mean[q]) * A.inv_std[q]);
  #pragma unroll
  for(int q = 5; q < 16; q++) p[q] = 0;
}

struct ScatterArgs {
  tc_geom_t g;
  const float * pred;       /* [nv][4] network output */
  float scale[4];           /* output de-normalisation */
  float * cx; float * cy; float * cz; float * ct;   /* corrections, field layout */
};

/* corrections at the variables' own positions: ux faces i = 2..nx average the two centres,
 * uy, uz, T at centres */
__global__ void tck_cnn_scatter(const ScatterArgs A){
  const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 1 + blockIdx.y;
  const int k = 1 + blockIdx.z;
  if(i > A.g.nx) return;
  const long long o = tck_idx(A.g, i, j, k);
  const long long v = (long long)(i - 1) + (long long)A.g.nx * ((long long)(j - 1) + (long long)A.g.ny * (k - 1));
  const float * p = A.pred + v * 4;
  A.cy[o] = A.scale[1] * p[1];
  A.cz[o] = A.scale[2] * p[2];
  if(A.ct) A.ct[o] = A.scale[3] * p[3];
  if(i >= 2) A.cx[o] = A.scale[0] * (0.5f * A.pred[(v - 1) * 4] + 0.5f * p[0]);
  else A.cx[o] = 0.f;
}

/* ------------------------------------------------------------------------------------- */
/* a convolution launch; the first one of an instantiation raises its dynamic LDS limit */
template <int CI, int CO>
static int cnn_conv_launch(const ConvArgs & A, dim3 grd, int lds, hipStream_t stream){
  static int ready = 0;
  if(!ready){
    const hipError_t e = hipFuncSetAttribute((const void *)tck_cnn_conv<CI, CO>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if(e != hipSuccess) return (int)e;
    ready = 1;
  }
  hipLaunchKernelGGL((tck_cnn_conv<CI, CO>), grd, dim3(CNN_TZ * TCK_WAVE), lds, stream, A);
  return 0;
}

template <int CI, int CO>
static int cnn_wgrad_launch(const WgradArgs & A, int nblk, hipStream_t stream){
  static int ready = 0;
  constexpr int lds = cnn_wgrad_lds(CI, CO);
  if(!ready){
    const hipError_t e = hipFuncSetAttribute((const void *)tck_cnn_wgrad<CI, CO>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if(e != hipSuccess) return (int)e;
    ready = 1;
  }
  hipLaunchKernelGGL((tck_cnn_wgrad<CI, CO>), dim3((unsigned)nblk), dim3(CNN_WG_THREADS), lds, stream, A);
  return 0;
}

static int g_cnn_ncu = 0;

static int cnn_ncu(void){
  if(g_cnn_ncu == 0){
    int dev = 0, v = 0;
    if(hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    g_cnn_ncu = v;
  }
  return g_cnn_ncu;
}

static long long cnn_conv_tiles(int nx, int ny, int nz, int nb){
  return (long long)((nx + 15) / 16) * ((ny + CNN_TY - 1) / CNN_TY) * ((nz + CNN_TZ - 1) / CNN_TZ) * nb;
}

/* blocks of a convolution: persistent, as many as the LDS holds per CU (the kernel and a
 * halo'd tile) */
static int cnn_conv_blocks(int nx, int ny, int nz, int nb, int ci, int co){
  const long long ntiles = cnn_conv_tiles(nx, ny, nz, nb);
  long long per_cu = (160LL * 1024) / cnn_conv_lds(ci, co);
  per_cu = per_cu < 1 ? 1 : (per_cu > 4 ? 4 : per_cu);
  const long long cap = per_cu * cnn_ncu();
  return (int)(ntiles < cap ? ntiles : cap);
}

extern "C" {

/* the most blocks a backward convolution has (entries of its bias partial sums: 32 each) */
int tck_cnn_bgrad_blocks(int nx, int ny, int nz, int nb){
  const int a = cnn_conv_blocks(nx, ny, nz, nb, 16, 32), b = cnn_conv_blocks(nx, ny, nz, nb, 32, 32);
  return a > b ? a : b;
}

/* out_bf set and act null: CNN_RELU; act set: CNN_RELU_BWD, *nblk the blocks of its partial
 * sums; else CNN_PLAIN into out_f */
int tck_cnn_launch_conv(int nx, int ny, int nz, int nb, const unsigned short * in, int ci,
    const unsigned short * w, int co, const float * bias, int co_store,
    unsigned short * out_bf, float * out_f, const unsigned short * act, float * bpart, int * nblk,
    hipStream_t stream){
  ConvArgs A;
  A.G.nx = nx; A.G.ny = ny; A.G.nz = nz; A.G.nb = nb; A.G.nv = (long long)nx * ny * nz * nb;
  A.in = in; A.w = w; A.bias = bias; A.out_bf = out_bf; A.out_f = out_f;
  A.act = act; A.bpart = bpart;
  A.co_store = co_store;
  A.mode = act ? CNN_RELU_BWD : (out_bf ? CNN_RELU : CNN_PLAIN);
  if(co_store % 4 != 0 || co_store > co || cnn_conv_tiles(nx, ny, nz, nb) > 0x7fffffffLL) return (int)hipErrorInvalidValue;
  const int lds = cnn_conv_lds(ci, co);
  const int blocks = cnn_conv_blocks(nx, ny, nz, nb, ci, co);
  if(nblk) *nblk = blocks;
  const dim3 grd((unsigned)blocks);
  int rc;
  if(ci == 16 && co == 32) rc = cnn_conv_launch<16, 32>(A, grd, lds, stream);
  else if(ci == 32 && co == 32) rc = cnn_conv_launch<32, 32>(A, grd, lds, stream);
  else if(ci == 32 && co == 16) rc = cnn_conv_launch<32, 16>(A, grd, lds, stream);
  else return (int)hipErrorInvalidValue;
  if(rc) return rc;
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_wgrad(int nx, int ny, int nz, int nb, const unsigned short * in, int ci_n,
    const unsigned short * g, int co_n, float * part, int * nblk_io, hipStream_t stream){
  int nblk = *nblk_io;
  WgradArgs A;
  A.G.nx = nx; A.G.ny = ny; A.G.nz = nz; A.G.nb = nb; A.G.nv = (long long)nx * ny * nz * nb;
  A.in = in; A.g = g; A.part = part;
  const long long ntiles = (long long)((nx + 15) / 16) * ((ny + 3) / 4) * ((nz + 3) / 4) * nb;
  if(ntiles > 0x7fffffffLL) return (int)hipErrorInvalidValue;
  if(nblk > ntiles) nblk = (int)ntiles;
  int rc;
  if(ci_n == 16 && co_n == 32) rc = cnn_wgrad_launch<16, 32>(A, nblk, stream);
  else if(ci_n == 32 && co_n == 32) rc = cnn_wgrad_launch<32, 32>(A, nblk, stream);
  else if(ci_n == 32 && co_n == 16) rc = cnn_wgrad_launch<32, 16>(A, nblk, stream);
  else return (int)hipErrorInvalidValue;
  if(rc) return rc;
  *nblk_io = nblk;
  TCK_CHECK_LAUNCH();
  return 0;
}

/* nseg sums of per-block partials, in one launch */
int tck_cnn_launch_reduce(int nseg, const float * const * part, const int * nblk, const int * n,
    float * const * out, hipStream_t stream){
  if(nseg < 1 || nseg > CNN_NSEG) return (int)hipErrorInvalidValue;
  ReduceArgs A;
  int first = 0;
  for(int q = 0; q < CNN_NSEG; q++){
    const int m = q < nseg ? q : nseg - 1;
    A.part[q] = part[m]; A.out[q] = out[m]; A.n[q] = n[m]; A.nblk[q] = nblk[m];
    A.first[q] = first;
    if(q < nseg) first += (n[q] + 63) / 64;
  }
  A.first[CNN_NSEG] = first;
  hipLaunchKernelGGL(tck_cnn_reduce, dim3((unsigned)first), dim3(256), 0, stream, A);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_mse(const float * pred, const float * target, long long nv, float scale,
    unsigned short * g, float * bpart, float * lpart, int nblk, hipStream_t stream){
  hipLaunchKernelGGL(tck_cnn_mse, dim3(nblk), dim3(256), 0, stream, (const float4 *)pred, (const float4 *)target,
      nv, scale, g, bpart, lpart);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_pack(const float * x, long long nv, unsigned short * out, hipStream_t stream){
  const long long nb = (nv + 255) / 256;
  hipLaunchKernelGGL(tck_cnn_pack, dim3((unsigned)(nb < 4096 ? nb : 4096)), dim3(256), 0, stream, x, nv, out);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_to_bf16(const float * x, long long n, unsigned short * y, hipStream_t stream){
  hipLaunchKernelGGL(tck_cnn_to_bf16, dim3(2048), dim3(256), 0, stream, x, n, y);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_flip(const unsigned short * w, int co_n, int ci_n, int ci_p, int co_p,
    unsigned short * wt, hipStream_t stream){
  const int n = 27 * ci_p * co_p;
  hipLaunchKernelGGL(tck_cnn_flip, dim3((n + 255) / 256), dim3(256), 0, stream, w, co_n, ci_n, ci_p, co_p, wt);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_adam(int nseg, float * const * w, float * const * m, float * const * v,
    float * const * g, unsigned short * const * wbf, unsigned short * const * wt, const int * n,
    const int * co, const int * ci, float lr, float b1, float b2, float eps, float c1, float c2,
    hipStream_t stream){
  if(nseg < 1 || nseg > CNN_NSEG) return (int)hipErrorInvalidValue;
  AdamArgs A;
  int nmax = 0;
  for(int q = 0; q < nseg; q++){
    A.w[q] = w[q]; A.m[q] = m[q]; A.v[q] = v[q]; A.g[q] = g[q]; A.wbf[q] = wbf[q]; A.wt[q] = wt[q];
    A.n[q] = n[q]; A.co[q] = co[q]; A.ci[q] = ci[q];
    if(n[q] > nmax) nmax = n[q];
  }
  A.lr = lr; A.b1 = b1; A.b2 = b2; A.eps = eps; A.c1 = c1; A.c2 = c2;
  hipLaunchKernelGGL(tck_cnn_adam, dim3((nmax + 255) / 256, nseg), dim3(256), 0, stream, A);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_gather(const tc_geom_t * g, const double * ux, const double * uy,
    const double * uz, const double * t, const double * xc, const float mean[5],
    const float inv_std[5], unsigned short * out, hipStream_t stream){
  GatherArgs A;
  A.g = *g; A.ux = ux; A.uy = uy; A.uz = uz; A.t = t; A.xc = xc; A.out = out;
  for(int q = 0; q < 5; q++){ A.mean[q] = mean[q]; A.inv_std[q] = inv_std[q]; }
  hipLaunchKernelGGL(tck_cnn_gather, dim3((g->nx + 63) / 64, g->ny, g->nz), dim3(64), 0, stream, A);
  TCK_CHECK_LAUNCH();
  return 0;
}

int tck_cnn_launch_scatter(const tc_geom_t * g, const float * pred, const float scale[4],
    float * cx, float * cy, float * cz, float * ct, hipStream_t stream){
  ScatterArgs A;
  A.g = *g; A.pred = pred; A.cx = cx; A.cy = cy; A.cz = cz; A.ct = ct;
  for(int q = 0; q < 4; q++) A.scale[q] = scale[q];
  hipLaunchKernelGGL(tck_cnn_scatter, dim3((g->nx + 63) / 64, g->ny, g->nz), dim3(64), 0, stream, A);
  TCK_CHECK_LAUNCH();
  return 0;
}

}
