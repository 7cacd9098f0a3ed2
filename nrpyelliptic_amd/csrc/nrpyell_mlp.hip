// nrpyell_mlp.hip -- the learned initial guess: a coordinate MLP u(x; punctures), trained on
// solutions this solver produced, run on hand-written BF16 MFMA kernels (CDNA4
// v_mfma_f32_32x32x16_bf16) with FP32 accumulation. No reference counterpart.
//
// Network: 23 input features (zero-padded to K0 = 64) -> 5 x [Linear(256) + SiLU] -> Linear(1).
// Activations between layers are stored in BF16 (MFMA operands), pre-activations in FP32;
// master weights, gradients and Adam moments are FP32, weights are re-rounded to BF16 after
// every update.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <math.h>
#include <string.h>

#include <chrono>
#include <memory>
#include <string>
#include <vector>

#include "nrpyell_internal.h"

typedef __bf16 bf16_t;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

#define MLP_K0 64  // input features, zero-padded so every GEMM dimension is a multiple of 64
#define MLP_NFEAT 23
#define MLP_W 256
#define MLP_HIDDEN 5  // hidden layers of width 256 (6 linear layers in total)

// Parameter offsets (elements) of W_l and b_l, l = 1..5, and of the output layer (index 6).
struct MlpOffsets {
  long w[MLP_HIDDEN + 2], b[MLP_HIDDEN + 2];
};

// 1 / (1 + e^-z). The reciprocal is v_rcp_f32 (1 ulp) with one Newton step: 4 instructions in the
// place of the 10 of an FP32 division. It is taken of (1 + e^-z) / 4, and the Newton step brings the 4
// back, because v_rcp_f32 gives 0 for a denormal reciprocal (z below -87.3); powers of two change no
// other bit. Where e^-z is infinite the Newton step is NaN, which the clamp to [0, 1], an output modifier
// of its last FMA, makes 0 (a NaN z stays NaN in z * sigmoidf_(z)).
// Measured over 4 million z in [-100, 30]: z * sigmoidf_(z) is the same float as with the division for z
// above -30; below, 0.4 % differ in a denormal's last bit, at the same error against FP64 (rms 1.6e-6,
// largest 4.1e-6, from the exponential).
__device__ __forceinline__ float sigmoidf_(float z) {
  const float d = fmaf(0.25f, __expf(-z), 0.25f);
  const float r = __builtin_amdgcn_rcpf(d), q = 0.25f * r;
  return __builtin_amdgcn_fmed3f(fmaf(fmaf(-d, r, 1.0f), q, q), 0.0f, 1.0f);
}
__device__ __forceinline__ bf16_t to_bf16(float x) { return (bf16_t)x; }

// splitmix64 of (seed, m): the dataset row of minibatch row m (uniform, with replacement)
__device__ __forceinline__ long draw_row(unsigned long long seed, int m, long N) {
  unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (unsigned long long)(m + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (long)(z % (unsigned long long)N);
}

// ---------------------------------------------------------------------------------------
// Training: one minibatch step is three launches.
//
// 1. mlp_train_rows_kernel: a block takes TR_R rows through the forward pass (activations in
//    LDS, ping-pong), the output layer and the loss, then back through the data-gradient chain
//    dZ_{l-1} = (dZ_l W_l) * silu'(Z_{l-1}). Every product is row-local, so nothing crosses
//    blocks. silu'(z) stays with the lane that produces z in the forward epilogue: it holds the
//    same (row, column) entries of dZ in the backward one. H_l (l = 0..5) and dZ_l (l = 1..5)
//    leave the block transposed ([width x M], rows contiguous), which is the layout the weight
//    gradients consume as MFMA operands.
// 2. mlp_grad_kernel, mlp_small_kernel: dW_l = dZ_l^T H_{l-1}, db_l = column sums of dZ_l, and the output layer's
//    gradients, as sums over TR_SPLITS row ranges in range order (deterministic), then Adam and
//    the BF16 weight copies (W_l and, for l >= 2, W_l transposed, the data-gradient chain's
//    operand).
//
// Arithmetic per entry matches the network definition: FP32 accumulation of BF16 products in
// ascending inner index, z = acc + b, h = bf16(silu(z)), y = sum_k h_k w_k + b (FP32),
// dy = 2 (y - t) / M, dZ_5 = bf16(dy w_out silu'(z_5)), dZ_{l-1} = bf16(acc silu'(z_{l-1})).
// ---------------------------------------------------------------------------------------
constexpr int TR_R = 32;        // rows per block
constexpr int TR_WAVES = 8;     // wave w owns columns 32w .. 32w+31 of every 256-wide layer
constexpr int TR_LD = MLP_W + 8;
constexpr int TR_SPLITS = 32;   // row ranges of the weight-gradient reduction

// Operand layout of a matrix X[rows][inner] (rows a multiple of 32, inner a multiple of 16):
// lane (li, lj) of a wave feeds the 32x32x16 MFMA for rows 32 t .. 32 t + 31 and inner step q
// with X[32 t + li][16 q + 8 lj .. 16 q + 8 lj + 7]; the layout keeps those 8 elements at
// ((t * (inner / 16) + q) * 64 + 32 lj + li) * 8, so a wave's operand load is 1 KB of
// consecutive bytes (a row-major load would touch 32 rows, 32 bytes each).
__device__ __forceinline__ long swz(int row, int col, int inner16) {
  return ((long)((row >> 5) * inner16 + (col >> 4)) * 64 + ((col >> 3) & 1) * 32 + (row & 31)) * 8 + (col & 7);
}

// Where the BF16 weight copies live in pws: W_l (rows n, inner k; l = 1..5) and W_l^T (rows k,
// inner n; l = 2..5) in the operand layout.
struct WeightCopies {
  long w_off[MLP_HIDDEN + 1];  // W_l in the FP32 parameters
  long fs[MLP_HIDDEN + 1];     // W_l in pws
  long ts[MLP_HIDDEN + 1];     // W_l^T in pws
};

struct TrainArgs {
  const bf16_t *X;  // dataset features [N x 64]
  const float *t;   // dataset targets [N]
  long N;
  unsigned long long seed;
  int gather;  // 1: minibatch row m is dataset row draw_row(seed, m, N); 0: row m
  int M;       // minibatch rows (multiple of 64)
  const bf16_t *pws;  // weights in the operand layout (WeightCopies)
  const float *p;
  MlpOffsets off;
  WeightCopies wc;
  bf16_t *Ht[MLP_HIDDEN + 1];      // H_l^T [width_l x M], l = 0..5
  bf16_t *dZt[MLP_HIDDEN + 1];     // dZ_l^T [256 x M], l = 1..5
  float *dy;                       // [M]
  double *loss;                    // += sum over the block's rows of (y - t)^2 / M
};

// The 32 x 32 MFMA tile of columns 32 ct .. and the block's rows r0 .. r0+31 to the transposed
// global [width x M] in the operand layout (rows = columns of the layer, inner = minibatch rows),
// straight from the accumulators' layout: v[g] holds column li, rows 8 g + 4 lj .. + 3, half of an
// 8-element chunk; lanes lj = 0, 1 fill it, so a wave's store is 512 consecutive bytes.
__device__ __forceinline__ void store_tile_transposed(const bf16x4 (&v)[4], bf16_t *__restrict__ out, int ct, int r0,
                                                      int M, int li, int lj) {
  bf16_t *o = out + ((long)(ct * (M / 16) + r0 / 16) * 64 + li) * 8 + 4 * lj;
#pragma unroll
  for (int g = 0; g < 4; g++) *(bf16x4 *)(o + ((g >> 1) * 64 + (g & 1) * 32) * 8) = v[g];
}

// 256 blocks at the production minibatch of 8192 rows, one per CU: each of the ten dependent
// products is 16 MFMAs of latency behind 128 KB of weights from L2, so what counts is the work
// between them. silu' of four layers stays in registers (of all five it does not fit 256), the
// transposed copies go to memory from the accumulators, and the sigmoid has no division: 28.0 us
// (silu' of three layers in LDS, the copies read back from the LDS tiles, divisions: 31.1 us).
__global__ void __launch_bounds__(512) mlp_train_rows_kernel(TrainArgs a) {
  __shared__ __attribute__((aligned(16))) bf16_t Hb[2][TR_R * TR_LD];
  __shared__ float s_part[TR_WAVES][TR_R];
  __shared__ float s_t[TR_R], s_dy[TR_R];
  __shared__ float s_dsl[16][64 * TR_WAVES];  // silu' of layer 1, read back by the thread that wrote it
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lj = lane >> 5;
  const int r0 = blockIdx.x * TR_R;
  // this lane's column of every 256-wide layer; the eight 32-column slices are rotated by the
  // block index so that concurrent blocks read different weight rows (no change to any sum)
  const int ct = (wave + blockIdx.x) & (TR_WAVES - 1);
  const int c = ct * 32 + li;
  // the weight operands of the next product are loaded (all of them, 16 B per lane per
  // 16-wide inner step) as soon as the current product's MFMAs are issued, so their latency
  // overlaps the epilogue and the barrier
  bf16x8 bv[MLP_W / 16];
#pragma unroll
  for (int q = 0; q < MLP_K0 / 16; q++)
    bv[q] = *(const bf16x8 *)(a.pws + a.wc.fs[1] + ((long)ct * (MLP_K0 / 16) + q) * 512 + 8 * lane);
  if (tid < TR_R * 8) {  // 32 rows x 64 BF16 features = 256 chunks of 16 B
    const int row = tid >> 3, ch = tid & 7;
    const long src = a.gather ? draw_row(a.seed, r0 + row, a.N) : (long)(r0 + row);
    if (ch == 0) s_t[row] = a.t[src];
    *(bf16x8 *)(&Hb[0][row * TR_LD + 8 * ch]) = *(const bf16x8 *)(a.X + src * MLP_K0 + 8 * ch);
  }
  __syncthreads();
  {  // H_0 transposed: 4 rows of one column per thread
    const int col = tid % MLP_K0, m = 4 * (tid / MLP_K0);
    bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = Hb[0][(m + i) * TR_LD + col];
    *(bf16x4 *)(a.Ht[0] + swz(col, r0 + m, a.M / 16)) = v;
  }
  // accumulator r of lane (li, lj): row 8*(r/4) + 4*lj + r%4 of the block, column c
  float dsl[MLP_HIDDEN][16];  // silu'(z); layer 1's waits in s_dsl
  int cur = 0;
#pragma unroll
  for (int l = 1; l <= MLP_HIDDEN; l++) {
    const int Kl = l == 1 ? MLP_K0 : MLP_W;
    const bf16_t *Hin = Hb[cur] + li * TR_LD + 8 * lj;
    const float bc = a.p[a.off.b[l] + c];
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
    for (int q = 0; q < Kl / 16; q++)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8 *)(Hin + 16 * q), bv[q], acc, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    // next: W_{l+1}, or W_5^T for the first step of the data-gradient chain
    const bf16_t *Wn = a.pws + (l < MLP_HIDDEN ? a.wc.fs[l + 1] : a.wc.ts[MLP_HIDDEN]) + (long)ct * 16 * 512 + 8 * lane;
#pragma unroll
    for (int q = 0; q < MLP_W / 16; q++) bv[q] = *(const bf16x8 *)(Wn + 512 * q);
    __builtin_amdgcn_sched_barrier(0);
    bf16_t *Hout = Hb[cur ^ 1] + 4 * lj * TR_LD + c;
    bf16x4 hb[4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      floatx4 h;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float z = acc[4 * g + i] + bc, s = sigmoidf_(z);
        const float ds = s * (1.0f + z * (1.0f - s));
        if (l == 1)
          s_dsl[4 * g + i][tid] = ds;
        else
          dsl[l - 1][4 * g + i] = ds;
        h[i] = z * s;
      }
      hb[g] = __builtin_convertvector(h, bf16x4);
#pragma unroll
      for (int i = 0; i < 4; i++) Hout[(8 * g + i) * TR_LD] = hb[g][i];
    }
    __syncthreads();
    store_tile_transposed(hb, a.Ht[l], ct, r0, a.M, li, lj);
    cur ^= 1;
  }
  // output layer: wave w sums columns 32w .. 32w+31 of every row, then the 8 partials in a fixed order
  const float *wout = a.p + a.off.w[MLP_HIDDEN + 1];
  if (lane < TR_R) {
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; k += 8) {
      const bf16x8 h = *(const bf16x8 *)(Hb[cur] + lane * TR_LD + wave * 32 + k);
#pragma unroll
      for (int i = 0; i < 8; i++) acc += (float)h[i] * wout[wave * 32 + k + i];
    }
    s_part[wave][lane] = acc;
  }
  const float wc_ = wout[c];
  __syncthreads();
  if (tid < 64) {
    double l2 = 0.0;
    if (tid < TR_R) {
      const float y = (((s_part[0][tid] + s_part[1][tid]) + (s_part[2][tid] + s_part[3][tid])) +
                       ((s_part[4][tid] + s_part[5][tid]) + (s_part[6][tid] + s_part[7][tid]))) +
                      a.p[a.off.b[MLP_HIDDEN + 1]];
      const float diff = y - s_t[tid];
      const float dy = 2.0f * diff / (float)a.M;
      s_dy[tid] = dy;
      a.dy[r0 + tid] = dy;
      l2 = (double)diff * (double)diff / (double)a.M;
    }
    for (int o = 32; o > 0; o >>= 1) l2 += __shfl_down(l2, o, 64);
    if (tid == 0) atomicAdd(a.loss, l2);
  }
  __syncthreads();
  // dZ_5 into the other buffer (H_4 there is no longer read), then dZ_{l-1} = (dZ_l W_l) *
  // silu'(Z_{l-1}), l = 5..2: A = dZ_l (LDS), B(k, n) = W_l^T[k][n]
#pragma unroll
  for (int l = MLP_HIDDEN + 1; l >= 2; l--) {
    floatx16 acc;
    if (l > MLP_HIDDEN) {
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] = s_dy[8 * (r >> 2) + 4 * lj + (r & 3)] * wc_;
    } else {
      const bf16_t *Din = Hb[cur] + li * TR_LD + 8 * lj;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
      for (int q = 0; q < MLP_W / 16; q++)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8 *)(Din + 16 * q), bv[q], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (l > 2) {
        const bf16_t *WT = a.pws + a.wc.ts[l - 1] + (long)ct * 16 * 512 + 8 * lane;
#pragma unroll
        for (int q = 0; q < MLP_W / 16; q++) bv[q] = *(const bf16x8 *)(WT + 512 * q);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    bf16_t *Dout = Hb[cur ^ 1] + 4 * lj * TR_LD + c;
    bf16x4 db[4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      floatx4 d;
#pragma unroll
      for (int i = 0; i < 4; i++) d[i] = acc[4 * g + i] * (l == 2 ? s_dsl[4 * g + i][tid] : dsl[l - 2][4 * g + i]);
      db[g] = __builtin_convertvector(d, bf16x4);
      if (l > 2) {
#pragma unroll
        for (int i = 0; i < 4; i++) Dout[(8 * g + i) * TR_LD] = db[g][i];
      }
    }
    if (l > 2) __syncthreads();
    store_tile_transposed(db, a.dZt[l - 1], ct, r0, a.M, li, lj);
    cur ^= 1;
  }
}

// The BF16 copies of parameter k (see WeightCopies).
__device__ __forceinline__ void store_weight(const WeightCopies &wc, long k, float v, bf16_t *__restrict__ pws) {
  const bf16_t b = to_bf16(v);
#pragma unroll
  for (int l = 1; l <= MLP_HIDDEN; l++) {
    const int Kl = l == 1 ? MLP_K0 : MLP_W;
    const long d = k - wc.w_off[l];
    if (d >= 0 && d < (long)MLP_W * Kl) {
      const int n = (int)(d / Kl), kk = (int)(d % Kl);
      pws[wc.fs[l] + swz(n, kk, Kl / 16)] = b;
      if (l >= 2) pws[wc.ts[l] + swz(kk, n, MLP_W / 16)] = b;
    }
  }
}

__global__ void refresh_weights_kernel(long n, const float *__restrict__ p, WeightCopies wc,
                                       bf16_t *__restrict__ pws) {
  const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) store_weight(wc, k, p[k], pws);
}

// Adam on one parameter, in the state arrays p, mo (first moment), ve (second); c1, c2 the bias
// corrections 1 - beta^t.
struct AdamArgs {
  float *p, *mo, *ve;
  bf16_t *pws;
  float lr, c1, c2;
  WeightCopies wc;
};
__device__ __forceinline__ void adam_update(const AdamArgs &o, long k, float gk) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float m = b1 * o.mo[k] + (1.0f - b1) * gk;
  const float v = b2 * o.ve[k] + (1.0f - b2) * gk * gk;
  o.mo[k] = m;
  o.ve[k] = v;
  const float pk = o.p[k] - o.lr * (m / o.c1) / (sqrtf(v / o.c2) + eps);
  o.p[k] = pk;
  store_weight(o.wc, k, pk, o.pws);
}

struct GradArgs {
  const bf16_t *Ht[MLP_HIDDEN + 1];
  const bf16_t *dZt[MLP_HIDDEN + 1];
  const float *dy;
  int M, chunk;  // rows per range (multiple of 16)
  MlpOffsets off;
  float *g;      // [n_params]
  float *part;   // [TR_SPLITS x GR_PART]: layer 1 and the output layer by ranges
  int update;    // 1: also an Adam step
  AdamArgs adam;
};

// The partials of one range: dW_1 as 16 tiles of 32 x 32, db_1, the output layer's weights and bias.
constexpr int GR_PB1 = MLP_W * MLP_K0, GR_PW = GR_PB1 + MLP_W, GR_PB = GR_PW + MLP_W, GR_PART = GR_PB + 1;

__device__ __forceinline__ void finish_gradient(const GradArgs &a, long k, float gk) {
  a.g[k] = gk;
  if (a.update) adam_update(a.adam, k, gk);
}

// 2. The gradients of one minibatch and the Adam step on them. A gradient is the sum over TR_SPLITS
// row ranges, in range order, of FP32 partials: dW_l = dZ_l^T H_{l-1} by MFMA in ascending rows,
// db_l the column sums of dZ_l, the output layer's by rows.
//
// Layers 2..5: block b owns one 32 x 32 tile of a dW_l through all ranges. Its eight waves take four
// ranges each, the partials meet in LDS (132 KB) and every thread adds the 32 of its two entries. So
// no partial leaves the chip (as global arrays they were 36 MB written and read again). A tile costs its reads of dZ_l and H_{l-1}, 1 MB at 8192 rows, and L1's rate sets the
// kernel's time: 256 tiles, one per CU, is the split with the least per CU. GR_D inner steps of 16
// rows are in flight per wave, across the ranges' ends. XCD x (where workgroups with b % 8 = x
// run) has half the rows of one layer, so its L2 serves their reuse.
// Layer 1 and the output layer would be a second block on a few CUs, which doubles the time;
// instead a ninth wave of every block takes a share of their ranges, and mlp_small_kernel adds
// those partials (2 MB). 8192 rows: 23.6 us and 4.8 us (gradients by row ranges 20.4 us, then
// reduction and Adam 9.8 us).
constexpr int GR_D = 8;
constexpr int GR_BLOCKS = 8 * (MLP_W / 32) * (MLP_HIDDEN - 1);
constexpr int GR_THREADS = 9 * 64;
static_assert(GR_BLOCKS == 8 * TR_SPLITS, "the ninth waves cover every range of layer 1 and the output layer");

// GR_D inner steps of a pair of operand tiles from step t on, at a uniform address. A group that
// starts past the last row reads the end of the tile's rows and the arrays' padding: not used.
struct GradRing {
  bf16x8 a[GR_D], b[GR_D];
};
__device__ __forceinline__ void grad_load(GradRing &r, int i, const bf16_t *A, const bf16_t *B, int t, int M16) {
  const long o = (long)min(t, M16) * 512;
  const unsigned v = 16 * (threadIdx.x & 63) + 1024 * i;
  r.a[i] = *(const bf16x8 *)((const char *)(A + o) + v);
  r.b[i] = *(const bf16x8 *)((const char *)(B + o) + v);
}
__device__ __forceinline__ void grad_fill(GradRing &r, const bf16_t *A, const bf16_t *B, int t, int M16) {
#pragma unroll
  for (int i = 0; i < GR_D; i++) {
    grad_load(r, i, A, B, t, M16);
    __builtin_amdgcn_sched_barrier(0);  // issued in the order of use: a wait for one leaves the later ones in flight
  }
}
// One range of a tile: its cs steps from s0 on (ns of them real), the group of (A1, B1) at `then`
// loaded as the last one is used; acc += A B^T, bsum += this lane's elements of A where `bias`.
__device__ __forceinline__ void grad_range(GradRing &r, const bf16_t *A, const bf16_t *B, int s0, int cs, int ns,
                                           const bf16_t *A1, const bf16_t *B1, int then, int M16, bool bias,
                                           floatx16 &acc, float &bsum) {
  for (int q0 = 0; q0 < cs; q0 += GR_D) {
    const bool more = q0 + GR_D < cs;
    const int next = more ? s0 + q0 + GR_D : then;
    const bf16_t *An = more ? A : A1, *Bn = more ? B : B1;
#pragma unroll
    for (int i = 0; i < GR_D; i++) {
      if (q0 + i < ns) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(r.a[i], r.b[i], acc, 0, 0, 0);
        if (bias) {
#pragma unroll
          for (int e = 0; e < 8; e++) bsum += (float)r.a[i][e];
        }
      }
      grad_load(r, i, An, Bn, next, M16);
    }
  }
}
// accumulator r of lane (li, lj) is row 8*(r/4) + 4*lj + r%4, column li of the 32 x 32 tile
__device__ __forceinline__ void store_tile(float *P, const floatx16 &acc, int li, int lj) {
#pragma unroll
  for (int r = 0; r < 16; r++) P[(8 * (r >> 2) + 4 * lj + (r & 3)) * 32 + li] = acc[r];
}

// The ninth wave of block b: two tiles of dW_1 for one range, and for b < 4 TR_SPLITS 64 of the output
// layer's inputs for one range.
__device__ __forceinline__ void grad_small_layers(const GradArgs &a, int b, int nrange, int M16, int cs) {
  const int lane = threadIdx.x & 63, li = lane & 31, lj = lane >> 5;
  const int s = b >> 3, t0 = (2 * b) & 15;  // tiles t0, t0 + 1: the same 32 rows n, both column halves
  if (s < nrange) {
    GradRing ring;
    const bf16_t *A = a.dZt[1] + (long)(t0 >> 1) * M16 * 512, *B = a.Ht[0], *B1 = B + (long)M16 * 512;
    float *P = a.part + (long)s * GR_PART;
    grad_fill(ring, A, B, s * cs, M16);
#pragma unroll
    for (int u = 0; u < 2; u++) {
      floatx16 acc;
      float bsum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] = 0.0f;
      grad_range(ring, A, u == 0 ? B : B1, s * cs, cs, min(cs, M16 - s * cs), A, B1, u == 0 ? s * cs : M16, M16, u == 0,
                 acc, bsum);
      store_tile(P + 1024 * (t0 + u), acc, li, lj);
      bsum += __shfl_xor(bsum, 32, 64);
      if (u == 0 && lj == 0) P[GR_PB1 + 32 * (t0 >> 1) + li] = bsum;
    }
  }
  const int so = b >> 2, q = b & 3;
  if (b < 4 * TR_SPLITS && so < nrange) {
    // gw[k] = sum_m dy[m] H_5[m][k], gb = sum_m dy[m]; a lane reads one row k of H_5^T, GR_D chunks of
    // 8 rows in flight
    const bf16_t *h = a.Ht[MLP_HIDDEN] + ((long)(2 * q + lj) * M16 * 64 + li) * 8;
    const int m1 = min(a.M, (so + 1) * a.chunk);
    float gw = 0.0f, gb = 0.0f;
    for (int m = so * a.chunk; m < m1; m += 8 * GR_D) {
      bf16x8 hv[GR_D];
      floatx4 dv[GR_D][2];
#pragma unroll
      for (int u = 0; u < GR_D; u++) {
        const int c = min(m + 8 * u, m1 - 8);
        hv[u] = *(const bf16x8 *)(h + ((long)(c >> 4) * 64 + ((c >> 3) & 1) * 32) * 8);
        dv[u][0] = *(const floatx4 *)(a.dy + c);
        dv[u][1] = *(const floatx4 *)(a.dy + c + 4);
      }
#pragma unroll
      for (int u = 0; u < GR_D; u++)
        if (m + 8 * u < m1) {
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const float d = dv[u][i >> 2][i & 3];
            gw += d * (float)hv[u][i];
            gb += d;
          }
        }
    }
    a.part[(long)so * GR_PART + GR_PW + 64 * q + lane] = gw;
    if (q == 0 && lane == 0) a.part[(long)so * GR_PART + GR_PB] = gb;
  }
}

__global__ void __launch_bounds__(GR_THREADS) mlp_grad_kernel(GradArgs a) {
  __shared__ float s_p[TR_SPLITS][32 * 32];
  __shared__ float s_b[TR_SPLITS][32];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lj = lane >> 5;
  const int b = blockIdx.x;
  const int nrange = (a.M + a.chunk - 1) / a.chunk;  // ranges with rows; the others add zero
  const int M16 = a.M / 16, cs = a.chunk / 16;       // inner steps: in all, per range
  const int x = b & 7, j = b >> 3;
  const int l = 2 + (x >> 1), nt = 4 * (x & 1) + (j >> 3), kt = j & 7;
  if (wave == 8) {
    grad_small_layers(a, b, nrange, M16, cs);
  } else {
    const bf16_t *A = a.dZt[l] + (long)nt * M16 * 512, *B = a.Ht[l - 1] + (long)kt * M16 * 512;
    GradRing ring;
    grad_fill(ring, A, B, wave * cs, M16);
    // this wave's ranges wave, wave + 8, ..: one accumulator each, so the waves run free of each other
    // until every range is done
    constexpr int NPH = TR_SPLITS / 8;
    floatx16 acc[NPH];
    float bsum[NPH];
#pragma unroll
    for (int ph = 0; ph < NPH; ph++) {
#pragma unroll
      for (int r = 0; r < 16; r++) acc[ph][r] = 0.0f;
      bsum[ph] = 0.0f;
      const int s0 = (8 * ph + wave) * cs;
      if (8 * ph < nrange)
        grad_range(ring, A, B, s0, cs, min(cs, M16 - s0), A, B, s0 + 8 * cs, M16, kt == 0, acc[ph], bsum[ph]);
    }
#pragma unroll
    for (int ph = 0; ph < NPH; ph++) {
      store_tile(s_p[8 * ph + wave], acc[ph], li, lj);
      if (kt == 0) {
        const float t = bsum[ph] + __shfl_xor(bsum[ph], 32, 64);
        if (lj == 0) s_b[8 * ph + wave][li] = t;
      }
    }
  }
  __syncthreads();
  if (tid >= 512) return;
  float gw[2] = {0.0f, 0.0f}, gb = 0.0f;
#pragma unroll
  for (int s = 0; s < TR_SPLITS; s++) {
#pragma unroll
    for (int e = 0; e < 2; e++) gw[e] += s_p[s][tid + 512 * e];
  }
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int k = tid + 512 * e;
    finish_gradient(a, a.off.w[l] + (long)(32 * nt + (k >> 5)) * MLP_W + 32 * kt + (k & 31), gw[e]);
  }
  if (kt == 0 && tid < 32) {
    for (int s = 0; s < TR_SPLITS; s++) gb += s_b[s][tid];
    finish_gradient(a, a.off.b[l] + 32 * nt + tid, gb);
  }
}

// Layer 1 and the output layer: the ranges' partials of mlp_grad_kernel in range order, Adam.
__global__ void __launch_bounds__(256) mlp_small_kernel(GradArgs a) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= GR_PART) return;
  const int nrange = (a.M + a.chunk - 1) / a.chunk;
  float v[TR_SPLITS], gk = 0.0f;
#pragma unroll
  for (int s = 0; s < TR_SPLITS; s++) v[s] = s < nrange ? a.part[(long)s * GR_PART + j] : 0.0f;
#pragma unroll
  for (int s = 0; s < TR_SPLITS; s++) gk += v[s];
  long k;
  if (j < GR_PB1) {
    const int t = j >> 10, e = j & 1023;
    k = a.off.w[1] + (32 * (t >> 1) + (e >> 5)) * MLP_K0 + 32 * (t & 1) + (e & 31);
  } else if (j < GR_PW) {
    k = a.off.b[1] + (j - GR_PB1);
  } else {
    k = j < GR_PB ? a.off.w[MLP_HIDDEN + 1] + (j - GR_PW) : a.off.b[MLP_HIDDEN + 1];
  }
  finish_gradient(a, k, gk);
}

// An Adam step with the gradient of an earlier mlp_grad_kernel launch.
__global__ void mlp_adam_kernel(long n, const float *__restrict__ g, AdamArgs o) {
  const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) adam_update(o, k, g[k]);
}

// Inference, all six layers in one launch: a block takes FI_R rows through the five hidden
// layers with the activations held in LDS (one FI_R x 256 BF16 buffer, overwritten layer by
// layer), so nothing but the 64 input features and the output leave the chip. Arithmetic of an
// entry: FP32 accumulation over BF16 products in ascending K, z = acc + b, h = bf16(silu(z)),
// output y = sum_k h_k w_k + b in FP32.
//
// Each of the 4 waves owns 64 output columns of the 64 rows, as 2 x 2 MFMA accumulators of
// Z^T = W H^T: with the weights as the first operand a lane ends up with 4 consecutive columns of
// one row, i.e. one 8-byte LDS store instead of four 2-byte ones, and the weights (544 KB of
// BF16, shared by every block) come from the operand layout, 1 KB of consecutive bytes per wave
// and load, FI_PF inner steps ahead of their use and across the layer boundary. The kernel is
// bound by the activations' vector instructions (1280 per row, each an exponential, a reciprocal
// and about 8 more; the MFMAs need 58 us of the 186 at 2.5 PFLOP/s) and overlaps them with other
// waves' MFMAs: four blocks per CU, which the single buffer (40 KB of LDS) and 125 registers per
// lane allow (one body for all five layers takes 160: layer 1 stands by itself). 262 144 rows: 186 us,
// 786 TFLOP/s (two ping-pong buffers, row-major weights loaded where they are used and FP32 divisions:
// 390 us, 375 TFLOP/s; the same outputs).
constexpr int FI_R = 64, FI_LD = MLP_W + 8;  // rows per block; LDS row stride (528 B)
constexpr int FI_PF = 4;                     // inner steps of weights in flight

// One hidden layer of K inputs: acc[x][y] (columns 64 wave + 32 x .., rows 32 y ..) from the
// activations in H, with the first FI_PF weight steps of this wave's two column tiles already in wv.
template <int K>
__device__ __forceinline__ void fi_layer(const bf16_t *H, const bf16_t *__restrict__ W, bf16x8 (&wv)[FI_PF][2],
                                         floatx16 (&acc)[2][2]) {
  constexpr int Q = K / 16;
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[x][y][r] = 0.0f;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    bf16x8 h[2];
#pragma unroll
    for (int y = 0; y < 2; y++) h[y] = *(const bf16x8 *)(H + 32 * y * FI_LD + 16 * q);
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 2; y++)
        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[q % FI_PF][x], h[y], acc[x][y], 0, 0, 0);
    if (q + FI_PF < Q) {
#pragma unroll
      for (int x = 0; x < 2; x++) wv[q % FI_PF][x] = *(const bf16x8 *)(W + ((long)x * Q + q + FI_PF) * 512);
    }
  }
}

__global__ void __launch_bounds__(256, 4) mlp_forward_fused_kernel(const bf16_t *__restrict__ X,
                                                                   const bf16_t *__restrict__ pws,
                                                                   const float *__restrict__ p, MlpOffsets off,
                                                                   WeightCopies wc, long M, float *__restrict__ y) {
  __shared__ __attribute__((aligned(16))) bf16_t Hbuf[FI_R * FI_LD];
  __shared__ __attribute__((aligned(16))) float s_b[MLP_HIDDEN][MLP_W];
  __shared__ float s_out[4][FI_R];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 31, lj = lane >> 5;
  const long r0 = (long)blockIdx.x * FI_R;
  bf16x8 wv[FI_PF][2];
  const bf16_t *W = pws + wc.fs[1] + (long)(2 * wave) * (MLP_K0 / 16) * 512 + 8 * lane;
#pragma unroll
  for (int q = 0; q < FI_PF; q++)
#pragma unroll
    for (int x = 0; x < 2; x++) wv[q][x] = *(const bf16x8 *)(W + (x * (MLP_K0 / 16) + q) * 512);
  // input features: 64 rows x 64 BF16 = 512 chunks of 16 B, 2 per thread (rows past M clamped)
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int e = tid + 256 * q, row = e >> 3, ch = e & 7;
    const long m = min(r0 + row, M - 1);
    *(bf16x8 *)(&Hbuf[row * FI_LD + 8 * ch]) = *(const bf16x8 *)(X + m * MLP_K0 + 8 * ch);
  }
#pragma unroll
  for (int l = 0; l < MLP_HIDDEN; l++) s_b[l][tid] = p[off.b[l + 1] + tid];
  __syncthreads();
  const bf16_t *H = Hbuf + li * FI_LD + 8 * lj;
  // the activations of layer l from its accumulators, between the layer's products and the next one's
  auto activate = [&](int l, const floatx16 (&acc)[2][2]) {
    if (l < MLP_HIDDEN) {  // the next layer's first weights, in flight during the activations
      W = pws + wc.fs[l + 1] + (long)(2 * wave) * (MLP_W / 16) * 512 + 8 * lane;
#pragma unroll
      for (int q = 0; q < FI_PF; q++)
#pragma unroll
        for (int x = 0; x < 2; x++) wv[q][x] = *(const bf16x8 *)(W + (x * (MLP_W / 16) + q) * 512);
    }
    __syncthreads();  // every wave has read this layer's input
    // accumulator r of lane (li, lj) in tile (x, yy): column 8*(r/4) + 4*lj + r%4, row li
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int c = 64 * wave + 32 * x + 8 * g + 4 * lj;
        const float4 b = *(const float4 *)(&s_b[l - 1][c]);
        const float bb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int yy = 0; yy < 2; yy++) {
          floatx4 h;
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float z = acc[x][yy][4 * g + i] + bb[i];
            h[i] = z * sigmoidf_(z);
          }
          *(bf16x4 *)(&Hbuf[(32 * yy + li) * FI_LD + c]) = __builtin_convertvector(h, bf16x4);
        }
      }
    __syncthreads();
  };
  floatx16 z[2][2];
  fi_layer<MLP_K0>(H, W, wv, z);
  activate(1, z);
#pragma unroll 1
  for (int l = 2; l <= MLP_HIDDEN; l++) {
    fi_layer<MLP_W>(H, W, wv, z);
    activate(l, z);
  }
  // output layer: wave w sums columns 64w..64w+63 of every row, then the 4 partials are added
  const float *wout = p + off.w[MLP_HIDDEN + 1] + 64 * wave;
  float acc = 0.0f;
#pragma unroll
  for (int c = 0; c < 64; c += 8) {
    const bf16x8 h = *(const bf16x8 *)(&Hbuf[lane * FI_LD + 64 * wave + c]);
#pragma unroll
    for (int i = 0; i < 8; i++) acc += (float)h[i] * wout[c + i];
  }
  s_out[wave][lane] = acc;
  __syncthreads();
  if (tid < FI_R && r0 + tid < M)
    y[r0 + tid] = ((s_out[0][tid] + s_out[1][tid]) + (s_out[2][tid] + s_out[3][tid])) + p[off.b[MLP_HIDDEN + 1]];
}

__global__ void gather_rows_kernel(const bf16_t *__restrict__ X, const float *__restrict__ t, long N, int M,
                                   unsigned long long seed, bf16_t *__restrict__ Xb, float *__restrict__ tb) {
  const int m = blockIdx.x;
  // splitmix64 of (seed, m): uniform row index
  unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (unsigned long long)(m + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  const long row = (long)(z % (unsigned long long)N);
  for (int k = threadIdx.x; k < MLP_K0; k += blockDim.x) Xb[(long)m * MLP_K0 + k] = X[row * MLP_K0 + k];
  if (threadIdx.x == 0) tb[m] = t[row];
}

// ---------------------------------------------------------------------------------------
// Features of the learned initial guess at every interior and pure outer point of a grid.
// With b the SinhSymTP focus (bScale), r = |X|, r_n = |X - x_n|:
//   point: X/(r+b), Y/(r+b), Z/(r+b), r/(r+b), log(1+r/b)/10, b/(r_0+b), b/(r_1+b)
//   configuration: m_0, m_1, D/20, 10 P_0, 10 P_1, S_0/m_0^2, S_1/m_1^2, b/10
// (23 numbers, zero-padded to 64). The network predicts t = log(50 u (r+b)): u > 0 everywhere
// (lap u = -AA^2/(8 psi^7) <= 0 with u -> 0 far away), and u (r+b) stays within a few
// decades over the grid, so t is O(1) at every point; u = exp(t)/(50 (r+b)).
// ---------------------------------------------------------------------------------------
struct FeatureParams {
  double AMAX, w, b, D;
  double m[2], pos[2][3], P[2][3], S[2][3];
};

__device__ inline void point_features(const FeatureParams &f, double x0, double x1, double x2,
                                      float out[MLP_NFEAT], double &scale) {
  const double f0 = f.AMAX * (exp(x0 / f.w) - exp(-x0 / f.w)) / f.D;
  const double X = f0 * sin(x1) * cos(x2), Y = f0 * sin(x1) * sin(x2), Z = sqrt(f0 * f0 + f.b * f.b) * cos(x1);
  const double r = sqrt(X * X + Y * Y + Z * Z), rb = r + f.b;
  double rn[2];
  for (int n = 0; n < 2; n++) {
    const double dx = X - f.pos[n][0], dy = Y - f.pos[n][1], dz = Z - f.pos[n][2];
    rn[n] = sqrt(dx * dx + dy * dy + dz * dz);
  }
  const double sep = sqrt((f.pos[0][0] - f.pos[1][0]) * (f.pos[0][0] - f.pos[1][0]) +
                          (f.pos[0][1] - f.pos[1][1]) * (f.pos[0][1] - f.pos[1][1]) +
                          (f.pos[0][2] - f.pos[1][2]) * (f.pos[0][2] - f.pos[1][2]));
  int k = 0;
  out[k++] = (float)(X / rb);
  out[k++] = (float)(Y / rb);
  out[k++] = (float)(Z / rb);
  out[k++] = (float)(r / rb);
  out[k++] = (float)(log1p(r / f.b) / 10.0);
  out[k++] = (float)(f.b / (rn[0] + f.b));
  out[k++] = (float)(f.b / (rn[1] + f.b));
  out[k++] = (float)f.m[0];
  out[k++] = (float)f.m[1];
  out[k++] = (float)(sep / 20.0);
  for (int n = 0; n < 2; n++)
    for (int d = 0; d < 3; d++) out[k++] = (float)(10.0 * f.P[n][d]);
  for (int n = 0; n < 2; n++)
    for (int d = 0; d < 3; d++) out[k++] = (float)(f.S[n][d] / fmax(f.m[n] * f.m[n], 1e-12));
  out[k++] = (float)(f.b / 10.0);
  scale = 1.0 / (50.0 * rb);
}

// One thread per interior or pure-outer point (i0 in [NG, G0), i1, i2 interior) and per padding
// row (zeros). The block's 256 rows of 128 B leave through LDS, so that a wave's store is 1 KB of
// consecutive bytes: 272 384 rows in 18.7 us, now bound by the FP64 closed forms (64 two-byte
// stores per thread, 128 B apart, after a clearing pass over X: 26 us and 10 us).
constexpr int FEAT_C = (MLP_NFEAT + 7) / 8;  // 16-byte chunks of a row that hold features
__global__ void __launch_bounds__(256) features_kernel(GridDims g, FeatureParams f, const double *__restrict__ xx0,
                                                       const double *__restrict__ xx1, const double *__restrict__ xx2,
                                                       long rows, bf16_t *__restrict__ X, double *__restrict__ scale,
                                                       long *__restrict__ idx) {
  __shared__ __attribute__((aligned(16))) bf16_t s_x[256][8 * FEAT_C];
  const int n0 = g.G0 - NRPYELL_NG, tid = threadIdx.x;
  const long k0 = (long)blockIdx.x * 256, k = k0 + tid;
  const long npts = (long)n0 * g.N1 * g.N2;
  float out[MLP_NFEAT] = {};
  if (k < npts) {
    const int i0 = NRPYELL_NG + (int)(k % n0);
    const int i1 = NRPYELL_NG + (int)((k / n0) % g.N1);
    const int i2 = NRPYELL_NG + (int)(k / ((long)n0 * g.N1));
    double s;
    point_features(f, xx0[i0], xx1[i1], xx2[i2], out, s);
    scale[k] = s;
    idx[k] = idx3(g, i0, i1, i2);
  }
#pragma unroll
  for (int q = 0; q < 8 * FEAT_C; q++) s_x[tid][q] = to_bf16(q < MLP_NFEAT ? out[q] : 0.0f);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MLP_K0 / 8; q++) {
    const int e = tid + 256 * q, row = e / (MLP_K0 / 8), ch = e % (MLP_K0 / 8);
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = to_bf16(0.0f);
    if (ch < FEAT_C) v = *(const bf16x8 *)(&s_x[row][8 * ch]);
    if (k0 + row < rows) *(bf16x8 *)(X + (k0 + row) * MLP_K0 + 8 * ch) = v;
  }
}

// u = e^t * scale at the listed points. FINAL: also v = eta u, and both at every parity image;
// otherwise u and its images in the interior phi planes, which is what the smoothing reads.
template <bool FINAL>
__global__ void seed_state_kernel(GridDims g, long npts, const float *__restrict__ t, const double *__restrict__ scale,
                                  const long *__restrict__ idx, double eta, double *__restrict__ yn) {
  const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npts) return;
  const double u = exp((double)t[k]) * scale[k];
  const long p = idx[k];
  yn[p] = u;
  if (FINAL) yn[g.ntot + p] = eta * u;
  const int i0 = (int)(p % g.G0), i1 = (int)((p / g.G0) % g.G1), i2 = (int)(p / ((long)g.G0 * g.G1));
  if (FINAL)
    for_each_image(g, i0, i1, i2, [&](long d) {
      yn[d] = u;
      yn[g.ntot + d] = eta * u;
    });
  else
    for_each_image_in_planes(g, i0, i1, i2, [&](long d) { yn[d] = u; });
}

// One binomial smoothing pass of u over the interior points, (f[-1] + 2 f + f[+1]) / 4 along i0,
// then i1, then i2 (phi neighbours through the periodic map), pure outer points copied. It removes
// the grid-scale part of the network's pointwise error (BF16 activations round independently at
// neighbouring points), which the Laplacian in the residual would otherwise amplify by 1/dx^2.
// Every thread forms the i0 averages of its 3 x 3 (i1, i2) neighbours itself: on a ghost row they
// are those of the row's source point, because `in` holds the parity images there and the average
// is symmetric. So the three directions are one pass over memory (5.8 us at 128x128x16, LAST 8.5;
// as three 5.1 + 5.3 + 6.2 us and a copy back, then 7 us for v and the ghost planes). Every point
// writes its images: those in the interior phi planes for the next pass, LAST all of them and
// v = eta u beside u.
template <bool LAST>
__global__ void smooth_kernel(GridDims g, double eta, const double *__restrict__ in, double *__restrict__ out) {
  const int i0 = NRPYELL_NG + blockIdx.x * blockDim.x + threadIdx.x;
  const int i1 = NRPYELL_NG + blockIdx.y, i2 = NRPYELL_NG + blockIdx.z;
  if (i0 >= g.G0) return;
  const long p = idx3(g, i0, i1, i2);
  double v = in[p];
  if (i0 < g.N0 + NRPYELL_NG) {
    double f2[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const int j2 = wrap2(g, i2 + k - 1);
      double f1[3];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const double *f = in + idx3(g, i0, i1 + j - 1, j2);
        f1[j] = 0.25 * (f[-1] + f[1]) + 0.5 * f[0];
      }
      f2[k] = 0.25 * (f1[0] + f1[2]) + 0.5 * f1[1];
    }
    v = 0.25 * (f2[0] + f2[2]) + 0.5 * f2[1];
  }
  out[p] = v;
  if (LAST) {
    out[g.ntot + p] = eta * v;
    for_each_image(g, i0, i1, i2, [&](long d) {
      out[d] = v;
      out[g.ntot + d] = eta * v;
    });
  } else {
    for_each_image_in_planes(g, i0, i1, i2, [&](long d) { out[d] = v; });
  }
}

// log(u / scale) at the listed points: the network's training target from a solved state
// (u / scale floored at 1e-8).
__global__ void target_kernel(long npts, const double *__restrict__ yn, const double *__restrict__ scale,
                              const long *__restrict__ idx, float *__restrict__ t) {
  const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < npts) t[k] = (float)log(fmax(yn[idx[k]] / scale[k], 1e-8));
}

// ---------------------------------------------------------------------------------------
// Host object
// ---------------------------------------------------------------------------------------
template <typename T>
static T *mlp_alloc(size_t n) {
  void *p = nullptr;
  HIPCHK(hipMalloc(&p, n * sizeof(T) > 0 ? n * sizeof(T) : 1));
  return (T *)p;
}

struct nrpyell_mlp {
  // parameter layout (FP32, concatenated): for l = 1..5: W_l [256 x K_l], b_l [256]; then w_out [256], b_out [1]
  std::vector<long> w_off, b_off, w_size;
  long n_params = 0;
  // the network's arrays, in one allocation
  char *params = nullptr;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  float *part = nullptr;  // gradient partials of layer 1 and the output layer [TR_SPLITS x GR_PART]
  bf16_t *pws = nullptr;  // BF16 W_l and W_l^T in the MFMA operand layout (WeightCopies)
  long adam_t = 0;
  int cap = 0;                       // minibatch arrays allocated for this many rows
  bf16_t *ws = nullptr;              // ... in one allocation
  bf16_t *Ht[MLP_HIDDEN + 1] = {};   // H_l^T [width_l x M], l = 0..5
  bf16_t *dZt[MLP_HIDDEN + 1] = {};  // dZ_l^T [256 x M], l = 1..5
  float *dy = nullptr;               // per-row output gradient
  double *loss = nullptr;
  // seeding workspace (features, per-row scale and point index, network output), grown on demand
  // and kept between seeds so a seed allocates nothing after the first one on a grid this large
  long seed_cap = 0;
  bf16_t *seedX = nullptr;
  double *seed_scale = nullptr;
  long *seed_idx = nullptr;
  float *seed_y = nullptr;
  int seed_nxx = 0;           // coordinates seed_xx has room for
  double *seed_xx = nullptr;
  hipStream_t st = nullptr;
  ~nrpyell_mlp() {
    (void)hipFree(params);
    release_seed_rows();
    release_seed_xx();
    release();
    if (st) (void)hipStreamDestroy(st);
  }
  int K(int l) const { return l == 1 ? MLP_K0 : MLP_W; }
  void alloc_params() {
    const size_t np = (size_t)(n_params + 63) / 64 * 64, nw = (size_t)pws_size(), ng = (size_t)TR_SPLITS * GR_PART;
    params = mlp_alloc<char>(sizeof(double) * 32 + sizeof(float) * (4 * np + ng) + sizeof(bf16_t) * nw);
    loss = (double *)params;
    p = (float *)(params + sizeof(double) * 32);
    g = p + np;
    m = g + np;
    v = m + np;
    pws = (bf16_t *)(v + np);
    part = (float *)(pws + nw);
  }
  void release() {
    (void)hipFree(ws);
    ws = nullptr;
    cap = 0;
  }
  void release_seed_rows() {
    (void)hipFree(seedX); (void)hipFree(seed_scale); (void)hipFree(seed_idx); (void)hipFree(seed_y);
    seedX = nullptr; seed_scale = nullptr; seed_idx = nullptr; seed_y = nullptr;
    seed_cap = 0;
  }
  void release_seed_xx() {
    (void)hipFree(seed_xx);
    seed_xx = nullptr;
    seed_nxx = 0;
  }
  // The rows' arrays and the coordinates' grow apart: a grid with more of one and fewer of the other takes
  // nothing away from the next. A failed allocation leaves the size 0: the next seed allocates again.
  void ensure_seed(long rows, int nxx) {
    if (rows > seed_cap) {
      release_seed_rows();
      seedX = mlp_alloc<bf16_t>((size_t)rows * MLP_K0);
      seed_scale = mlp_alloc<double>((size_t)rows);
      seed_idx = mlp_alloc<long>((size_t)rows);
      seed_y = mlp_alloc<float>((size_t)rows);
      seed_cap = rows;
    }
    if (nxx > seed_nxx) {
      release_seed_xx();
      seed_xx = mlp_alloc<double>((size_t)nxx);
      seed_nxx = nxx;
    }
  }
  void ensure(int M) {
    if (M <= cap) return;
    // release first; a failed allocation below (HipFailure) leaves cap 0, so the next call
    // allocates again. mlp_grad_kernel loads whole groups of GR_D steps: up to a group past an
    // array's end, which is in the next array or the padding behind the last one.
    release();
    const size_t m0 = (size_t)M * MLP_K0, m1 = (size_t)M * MLP_W, pad = GR_D * 512;
    ws = mlp_alloc<bf16_t>(m0 + 2 * MLP_HIDDEN * m1 + pad + 2 * (size_t)M);
    Ht[0] = ws;
    for (int l = 1; l <= MLP_HIDDEN; l++) {
      Ht[l] = ws + m0 + (l - 1) * m1;
      dZt[l] = ws + m0 + (MLP_HIDDEN + l - 1) * m1;
    }
    dy = (float *)(ws + m0 + 2 * MLP_HIDDEN * m1 + pad);
    cap = M;
  }
  MlpOffsets offsets() const {
    MlpOffsets off;
    for (int l = 1; l <= MLP_HIDDEN + 1; l++) {
      off.w[l] = w_off[l];
      off.b[l] = b_off[l];
    }
    return off;
  }
  WeightCopies copies() const {
    WeightCopies wc;
    long o = 0;
    for (int l = 1; l <= MLP_HIDDEN; l++) {
      wc.w_off[l] = w_off[l];
      wc.fs[l] = o;
      o += (long)MLP_W * K(l);
    }
    for (int l = 2; l <= MLP_HIDDEN; l++) {
      wc.ts[l] = o;
      o += (long)MLP_W * MLP_W;
    }
    wc.w_off[0] = wc.fs[0] = wc.ts[0] = wc.ts[1] = 0;
    return wc;
  }
  static long pws_size() { return (long)MLP_W * MLP_K0 + (2L * MLP_HIDDEN - 2) * MLP_W * MLP_W; }
  void refresh_bf16() {
    hipLaunchKernelGGL(refresh_weights_kernel, dim3((n_params + 255) / 256), dim3(256), 0, st, n_params, p, copies(),
                       pws);
  }
  // forward, loss (added to *loss_out) and gradient of M minibatch rows (M a multiple of 64):
  // rows drawn from the dataset (gather) or its first M rows; with update, one Adam step at
  // learning rate lr
  void step(const bf16_t *X, const float *t, long N, unsigned long long seed, int gather, int M, double *loss_out,
            int update, float lr) {
    ensure(M);
    TrainArgs a;
    a.X = X;
    a.t = t;
    a.N = N;
    a.seed = seed;
    a.gather = gather;
    a.M = M;
    a.pws = pws;
    a.wc = copies();
    a.p = p;
    a.off = offsets();
    for (int l = 0; l <= MLP_HIDDEN; l++) {
      a.Ht[l] = Ht[l];
      a.dZt[l] = dZt[l];
    }
    a.dy = dy;
    a.loss = loss_out;
    hipLaunchKernelGGL(mlp_train_rows_kernel, dim3(M / TR_R), dim3(64 * TR_WAVES), 0, st, a);
    GradArgs w;
    for (int l = 0; l <= MLP_HIDDEN; l++) {
      w.Ht[l] = Ht[l];
      w.dZt[l] = dZt[l];
    }
    w.dy = dy;
    w.M = M;
    w.chunk = ((M + TR_SPLITS - 1) / TR_SPLITS + 15) / 16 * 16;
    w.off = a.off;
    w.g = g;
    w.update = update;
    w.adam = update ? next_adam(lr) : AdamArgs{};
    w.part = part;
    hipLaunchKernelGGL(mlp_grad_kernel, dim3(GR_BLOCKS), dim3(GR_THREADS), 0, st, w);
    hipLaunchKernelGGL(mlp_small_kernel, dim3((GR_PART + 255) / 256), dim3(256), 0, st, w);
  }
  // outputs of M feature rows (M a multiple of 64) on a stream
  void forward(const bf16_t *X, long M, float *y, hipStream_t stream) {
    hipLaunchKernelGGL(mlp_forward_fused_kernel, dim3((unsigned)((M + FI_R - 1) / FI_R)), dim3(256), 0, stream, X, pws,
                       p, offsets(), copies(), M, y);
  }
  // the arguments of the next Adam step (counts it)
  AdamArgs next_adam(float lr) {
    adam_t++;
    return {p, m, v, pws, lr, 1.0f - powf(0.9f, (float)adam_t), 1.0f - powf(0.999f, (float)adam_t), copies()};
  }
};

extern "C" int nrpyell_mlp_create(unsigned long long seed, nrpyell_mlp **out) {
  return api_call([&]() -> int {
    auto s = std::make_unique<nrpyell_mlp>();
    s->w_off.assign(7, 0);
    s->b_off.assign(7, 0);
    s->w_size.assign(7, 0);
    long off = 0;
    for (int l = 1; l <= MLP_HIDDEN; l++) {
      s->w_off[l] = off;
      s->w_size[l] = (long)MLP_W * s->K(l);
      off += s->w_size[l];
      s->b_off[l] = off;
      off += MLP_W;
    }
    s->w_off[6] = off;
    s->w_size[6] = MLP_W;
    off += MLP_W;
    s->b_off[6] = off;
    off += 1;
    s->n_params = off;
    // He-style initialisation (uniform, splitmix64 stream), biases zero
    std::vector<float> h(off, 0.0f);
    unsigned long long z = seed;
    auto rnd = [&]() {
      z += 0x9E3779B97F4A7C15ull;
      unsigned long long x = z;
      x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
      x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
      x ^= x >> 31;
      return (double)(x >> 11) / 9007199254740992.0;
    };
    for (int l = 1; l <= 6; l++) {
      const int fan_in = l == 1 ? MLP_NFEAT : MLP_W;
      const double a = sqrt(6.0 / fan_in) * (l == 6 ? 0.1 : 1.0);
      for (long k = 0; k < s->w_size[l]; k++) h[s->w_off[l] + k] = (float)((2 * rnd() - 1) * a);
    }
    s->alloc_params();
    HIPCHK(hipMemcpy(s->p, h.data(), off * sizeof(float), hipMemcpyHostToDevice));
    HIPCHK(hipMemset(s->m, 0, off * sizeof(float)));
    HIPCHK(hipMemset(s->v, 0, off * sizeof(float)));
    HIPCHK(hipStreamCreateWithFlags(&s->st, hipStreamNonBlocking));
    s->refresh_bf16();
    HIPCHK(hipStreamSynchronize(s->st));
    *out = s.release();
    return NRPYELL_OK;
  });
}

extern "C" int nrpyell_mlp_destroy(nrpyell_mlp *s) {
  return api_call([&]() -> int {
    if (s) {
      (void)hipStreamSynchronize(s->st);
      delete s;
    }
    return NRPYELL_OK;
  });
}

extern "C" long nrpyell_mlp_num_params(nrpyell_mlp *s) { return s->n_params; }

extern "C" int nrpyell_mlp_get_params(nrpyell_mlp *s, float *host) {
  return api_call([&]() -> int {
    HIPCHK(hipStreamSynchronize(s->st));
    HIPCHK(hipMemcpy(host, s->p, s->n_params * sizeof(float), hipMemcpyDeviceToHost));
    return NRPYELL_OK;
  });
}

extern "C" int nrpyell_mlp_set_params(nrpyell_mlp *s, const float *host) {
  return api_call([&]() -> int {
    HIPCHK(hipMemcpy(s->p, host, s->n_params * sizeof(float), hipMemcpyHostToDevice));
    s->refresh_bf16();
    HIPCHK(hipStreamSynchronize(s->st));
    return NRPYELL_OK;
  });
}

static int check_rows(int M) {
  if (M <= 0 || M % 64) {
    set_last_error("MLP row count must be a positive multiple of 64");
    return NRPYELL_EINVAL;
  }
  return NRPYELL_OK;
}

// Forward pass on M rows of device BF16 features [M x 64]; y (device, FP32) gets M outputs.
extern "C" int nrpyell_mlp_forward(nrpyell_mlp *s, const void *x, int M, float *y_out) {
  return api_call([&]() -> int {
    if (check_rows(M)) return NRPYELL_EINVAL;
    s->forward((const bf16_t *)x, M, y_out, s->st);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s->st));
    return NRPYELL_OK;
  });
}

// Loss (mean squared error) and its gradient for M rows; grads copied to host when non-null.
// Loss (mean squared error) and its gradient for M rows (device BF16 features [M x 64], FP32
// targets); grads copied to host when non-null.
extern "C" int nrpyell_mlp_loss_grad(nrpyell_mlp *s, const void *x, const float *t, int M, double *loss,
                                     float *grads_host) {
  return api_call([&]() -> int {
    if (check_rows(M)) return NRPYELL_EINVAL;
    HIPCHK(hipMemsetAsync(s->loss, 0, sizeof(double), s->st));
    s->step((const bf16_t *)x, t, M, 0, 0, M, s->loss, 0, 0.0f);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(loss, s->loss, sizeof(double), hipMemcpyDeviceToHost, s->st));
    if (grads_host) HIPCHK(hipMemcpyAsync(grads_host, s->g, s->n_params * sizeof(float), hipMemcpyDeviceToHost, s->st));
    HIPCHK(hipStreamSynchronize(s->st));
    return NRPYELL_OK;
  });
}

// nsteps of Adam on minibatches of `batch` rows drawn uniformly from a device dataset
// (features BF16 [N x 64], targets FP32 [N]); cosine learning-rate decay from lr to lr/100.
// losses (host, nsteps entries, may be null) receives each step's minibatch loss. Three
// launches per step; the seed of step k's draw is
// seed + 0x632BE59BD9B4E019 (k + 1).
extern "C" int nrpyell_mlp_train(nrpyell_mlp *s, const void *X, const float *t, long N, int batch, int nsteps,
                                 float lr, unsigned long long seed, double *losses) {
  return api_call([&]() -> int {
    if (check_rows(batch) || N <= 0 || nsteps < 0) return NRPYELL_EINVAL;
    DevBuf<double> dlb(nsteps > 0 ? nsteps : 1);
    double *dl = dlb.p;
    HIPCHK(hipMemsetAsync(dl, 0, (nsteps > 0 ? nsteps : 1) * sizeof(double), s->st));
    for (int k = 0; k < nsteps; k++) {
      const float frac = nsteps > 1 ? (float)k / (float)(nsteps - 1) : 0.0f;
      const float lrk = lr * (0.01f + 0.99f * 0.5f * (1.0f + cosf(3.14159265f * frac)));
      s->step((const bf16_t *)X, t, N, seed + 0x632BE59BD9B4E019ull * (unsigned long long)(k + 1), 1, batch, dl + k, 1,
              lrk);
    }
    HIPCHK(hipGetLastError());
    if (losses && nsteps > 0)
      HIPCHK(hipMemcpyAsync(losses, dl, nsteps * sizeof(double), hipMemcpyDeviceToHost, s->st));
    HIPCHK(hipStreamSynchronize(s->st));
    return NRPYELL_OK;
  });
}

// n_take rows drawn uniformly (with replacement) from device rows (x_src [n_src x 64],
// t_src [n_src]) into x_dst/t_dst: the per-configuration sample of the training set.
extern "C" int nrpyell_mlp_sample_rows(const void *x_src, const float *t_src, long n_src, long n_take,
                                       unsigned long long seed, void *x_dst, float *t_dst) {
  return api_call([&]() -> int {
    if (n_src <= 0 || n_take <= 0 || n_take > (1L << 30)) {
      set_last_error("sample_rows: bad sizes");
      return NRPYELL_EINVAL;
    }
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)n_take), dim3(64), 0, 0, (const bf16_t *)x_src, t_src, n_src,
                       (int)n_take, seed, (bf16_t *)x_dst, t_dst);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    return NRPYELL_OK;
  });
}

// One Adam step with the gradient of the last nrpyell_mlp_loss_grad call.
extern "C" int nrpyell_mlp_adam_step(nrpyell_mlp *s, float lr) {
  return api_call([&]() -> int {
    hipLaunchKernelGGL(mlp_adam_kernel, dim3((s->n_params + 255) / 256), dim3(256), 0, s->st, s->n_params, s->g,
                       s->next_adam(lr));
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s->st));
    return NRPYELL_OK;
  });
}

static FeatureParams feature_params(const paramstruct *p) {
  FeatureParams f;
  f.AMAX = p->AMAX;
  f.w = p->SINHWAA;
  f.b = p->bScale;
  f.D = exp(1.0 / p->SINHWAA) - exp(-1.0 / p->SINHWAA);
  f.m[0] = p->bare_mass_0;
  f.m[1] = p->bare_mass_1;
  const double pos[2][3] = {{p->puncture_0_x, p->puncture_0_y, p->puncture_0_z},
                            {p->puncture_1_x, p->puncture_1_y, p->puncture_1_z}};
  const double P[2][3] = {{p->P0_x, p->P0_y, p->P0_z}, {p->P1_x, p->P1_y, p->P1_z}};
  const double S[2][3] = {{p->S0_x, p->S0_y, p->S0_z}, {p->S1_x, p->S1_y, p->S1_z}};
  memcpy(f.pos, pos, sizeof(pos));
  memcpy(f.P, P, sizeof(P));
  memcpy(f.S, S, sizeof(S));
  return f;
}

// Number of feature rows of a grid (interior + pure outer points), rounded up to 64.
extern "C" long nrpyell_mlp_feature_rows(const griddata_struct *gd) {
  const GridDims g = dims_from_params(&gd->params);
  const long n = (long)(g.G0 - NRPYELL_NG) * g.N1 * g.N2;
  return (n + 63) / 64 * 64;
}

// The feature kernel on the default stream; xx is device memory for the G0 + G1 + G2 coordinates.
static void launch_features(const griddata_struct *gd, const GridDims &g, double *xx, void *X, double *scale,
                            long *idx) {
  const long rows = nrpyell_mlp_feature_rows(gd);
  std::vector<double> h(gd->xx[0], gd->xx[0] + g.G0);
  h.insert(h.end(), gd->xx[1], gd->xx[1] + g.G1);
  h.insert(h.end(), gd->xx[2], gd->xx[2] + g.G2);
  HIPCHK(hipMemcpy(xx, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(features_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, 0, g,
                     feature_params(&gd->params), xx, xx + g.G0, xx + g.G0 + g.G1, rows, (bf16_t *)X, scale, idx);
}

// Features (device BF16 [rows x 64], padding rows zero), per-row u scale and grid index.
extern "C" int nrpyell_mlp_features(const griddata_struct *gd, void *X, double *scale, long *idx) {
  return api_call([&]() -> int {
    const GridDims g = dims_from_params(&gd->params);
    DevBuf<double> xx(g.G0 + g.G1 + g.G2);
    launch_features(gd, g, xx.p, X, scale, idx);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    return NRPYELL_OK;
  });
}

// Training targets t = u/scale from the solved y_n of a griddata at the feature rows.
extern "C" int nrpyell_mlp_targets(const griddata_struct *gd, const double *scale, const long *idx, float *t) {
  return api_call([&]() -> int {
    const GridDims g = dims_from_params(&gd->params);
    const long n = (long)(g.G0 - NRPYELL_NG) * g.N1 * g.N2;
    hipLaunchKernelGGL(target_kernel, dim3((n + 255) / 256), dim3(256), 0, 0, n, gd->gridfuncs.y_n_gfs, scale, idx, t);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    return NRPYELL_OK;
  });
}

// Seed griddata's y_n from the network: u = e^t scale at interior and pure outer points,
// smoothed by smooth_passes binomial passes (each along i0, i1, i2), v = eta u (the steady
// state of du/dt = v - eta u), parity images written in every ghost point. k_odd_gfs is the
// scratch of the smoothing.
extern "C" int nrpyell_mlp_seed(nrpyell_mlp *s, griddata_struct *gd, int smooth_passes) {
  return api_call([&]() -> int {
    if (smooth_passes < 0 || smooth_passes > 64) {
      set_last_error("mlp_seed: smooth_passes must be in [0, 64]");
      return NRPYELL_EINVAL;
    }
    const GridDims g = dims_from_params(&gd->params);
    const long n = (long)(g.G0 - NRPYELL_NG) * g.N1 * g.N2, rows = nrpyell_mlp_feature_rows(gd);
    s->ensure_seed(rows, g.G0 + g.G1 + g.G2);
    launch_features(gd, g, s->seed_xx, s->seedX, s->seed_scale, s->seed_idx);
    s->forward(s->seedX, rows, s->seed_y, 0);
    const double eta = gd->params.eta_damping;
    double *yn = gd->gridfuncs.y_n_gfs, *other = gd->gridfuncs.k_odd_gfs;
    const dim3 sg((g.G0 - NRPYELL_NG + 63) / 64, g.N1, g.N2), pg((unsigned)((n + 255) / 256));
    if (smooth_passes == 0) {
      hipLaunchKernelGGL(seed_state_kernel<true>, pg, dim3(256), 0, 0, g, n, s->seed_y, s->seed_scale, s->seed_idx,
                         eta, yn);
    } else {
      // u alternates between the two arrays so that the last pass writes y_n
      double *from = smooth_passes % 2 ? other : yn, *to = smooth_passes % 2 ? yn : other;
      hipLaunchKernelGGL(seed_state_kernel<false>, pg, dim3(256), 0, 0, g, n, s->seed_y, s->seed_scale, s->seed_idx,
                         eta, from);
      for (int k = 1; k < smooth_passes; k++) {
        hipLaunchKernelGGL(smooth_kernel<false>, sg, dim3(64), 0, 0, g, eta, from, to);
        std::swap(from, to);
      }
      hipLaunchKernelGGL(smooth_kernel<true>, sg, dim3(64), 0, 0, g, eta, from, to);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    return NRPYELL_OK;
  });
}
