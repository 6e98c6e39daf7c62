// mlp_net.hpp -- the warm-start network's fused kernels (gfx950), for widths
// up to 256: the whole forward pass, and for training the whole backward
// data pass with it, in one launch; the hidden layers' weight gradients in a
// second.  Included by mlp.hip.
//
// What bounds the layer-by-layer form: each 256 x 256 layer is 8.6 GFLOP at
// a 65,536-row batch (7 us at the matrix rate) but moves 100 MB of
// activations and runs one launch; forward took 231 us, a training step
// 1190 us.  Here a wavefront carries 32 rows through every layer in
// registers, so inference moves only inputs and outputs and is bound by the
// SiLU's vector arithmetic (an exponential and a reciprocal per value):
// 75 us forward at 65,536 rows of the 5-256x6-4 network, 372 us a step.
//
// Layout.  A layer computes Z^T = W A^T: the 32x32x16 MFMA takes a 32 x 16
// piece of W and 16 x 32 of A^T and leaves lane l with batch row l % 32 and
// outputs n = 8 (r/4) + 4 (l/32) + r%4 (r = 0..15).  Rounded to BF16 pairs
// and with one v_permlane32_swap per pair of registers, those are exactly
// the next layer's operand (8 consecutive k per lane): no LDS and no barrier
// between layers but for the weights, which stream through LDS in chunks of
// 32 outputs shared by the block's wavefronts.  Every product sum is the one
// the layer-by-layer kernels form, in the same order; SiLU's reciprocal
// (sigm_fast) may differ from their division in the last place.
//
// For the weight gradients A and dZ are needed with batch rows along k; a
// product with the identity (exact) turns a 32 x 32 piece, and it is stored
// as the operand the weight-gradient kernel reads, 1 KB per wavefront store.
#pragma once

namespace dgbgk {
namespace mlp {

constexpr int kMaxFused = 256;  // widest network of the fused kernels

typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bfx2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

struct NetArgs {
  const float* X;     // [n][fin]; row r of the batch is X's row r, or a drawn one
  const float* T;     // targets [n][fout] (training)
  long n;             // rows of X (rows at and past n read as zero)
  unsigned seed, step;
  int gather;         // draw rows by the hash of (seed, step, row)
  int rows, fin, fout, hidden;
  const bf16* pb;     // parameters, BF16 and FP32, packed per layer
  const float* p;
  const bf16* wf;     // hidden weights as forward operands (pack_index)
  const bf16* wb;     // and as backward operands
  float* Y;           // [rows][fout] (inference)
  float* loss_part;   // per block
  uintx4* Z;          // [hidden][rows W/8]: this kernel's own order, piece by
                      // piece where dZ's go
  uintx4* A;          // [hidden-1][rows W/8]: weight-gradient operands
  size_t act4;        // uintx4 per layer of Z, A
  float* pin;         // per block: [W][fin+1]  dW, db of the input layer
  float* pout;        //            [fout][W+1] of the output layer
  float* pbias;       // [hidden-1][blocks][W]  db of layers 1..hidden-1
};

// Where weight (o, k) of a hidden layer lies in the operand packs: pieces of
// 32 x 16 as the MFMA's lanes hold them, the pieces of 32 outputs (forward)
// or inputs (backward) contiguous.
__host__ __device__ inline size_t pack_index(int row, int k, int W) {
  return ((size_t)(row >> 5) * (W / 16) + (k >> 4)) * 512 +
         ((row & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

__device__ __forceinline__ unsigned pk_bf16(float a, float b) {  // round to nearest even
  const floatx2 v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bfx2));
}
__device__ __forceinline__ float lo_bf(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_bf(unsigned u) { return __uint_as_float(u & 0xffff0000u); }

// 1 / (1 + exp(-z)): the hardware reciprocal (1 ulp) and one Newton step,
// which rounds as the division does but for rare last-place ties, at 3
// instructions instead of the division's 10.  fmaxf: d = inf gives 0, as the
// division does (fma(-inf, 0, 1) is NaN), and a NaN stays NaN.
__device__ __forceinline__ float sigm_fast(float z) {
  const float d = 1.0f + __expf(-z);
  const float y = __builtin_amdgcn_rcpf(d);
  return fmaf(y, fmaxf(fmaf(-d, y, 1.0f), -1.0f), y);
}

// An empty constraint on running sums: without it the scheduler finishes one
// sum of several first and keeps (spills) what the others wait for.
template <int N>
__device__ __forceinline__ void pin(float (&s)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(s[i]));
}

// p: 8 BF16 pairs of a 32 x 32 accumulator (register order); to the two
// 16-deep MFMA operands with 8 consecutive k per lane
__device__ __forceinline__ void to_operands(unsigned (&p)[8], uintx4& k0, uintx4& k1) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uintx2 s = __builtin_amdgcn_permlane32_swap(p[i], p[i + 2], false, false);
    p[i] = s.x;
    p[i + 2] = s.y;
    s = __builtin_amdgcn_permlane32_swap(p[i + 4], p[i + 6], false, false);
    p[i + 4] = s.x;
    p[i + 6] = s.y;
  }
  k0 = uintx4{p[0], p[1], p[2], p[3]};
  k1 = uintx4{p[4], p[5], p[6], p[7]};
}

__device__ __forceinline__ floatx16 mfma(uintx4 a, uintx4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// batch row of this step: a counter-based hash of (seed, step, row)
__device__ __forceinline__ long drawn_row(unsigned seed, unsigned step, int r, long ns) {
  unsigned long long h = ((unsigned long long)seed << 32) ^ ((unsigned long long)step << 20) ^
                         (unsigned long long)r;
  h ^= h >> 33; h *= 0xff51afd7ed558ccdULL; h ^= h >> 33; h *= 0xc4ceb9fe1a85ec53ULL;
  h ^= h >> 33;
  return (long)(h % (unsigned long long)ns);
}

// NW wavefronts of 32 rows per block.  Training: forward, loss, backward
// data, the small layers' gradients and all bias gradients.  FI, FO: inputs
// and outputs computed (at least fin, fout; the rest are zeros).
template <int W, int NW, bool kTrain, int FI, int FO>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_net(NetArgs a) {
  constexpr int NT = W / 32, KS = W / 16, QK = W / 64;
  constexpr int kThreads = 64 * NW;
  constexpr int kChunk4 = 32 * W / 8;           // uintx4 per weight chunk
  constexpr int kStage = kChunk4 / kThreads;    // per thread
  static_assert(kChunk4 % kThreads == 0, "chunk split");
  __shared__ uintx4 s_ring[2][kChunk4];
  __shared__ __align__(16) bf16 s_win[W][kMaxIO];
  __shared__ __align__(16) float s_wout[W][kMaxIO];
  __shared__ float s_tmp[kTrain ? 2 : 1][kTrain ? NW : 1][kTrain ? 32 : 1][kMaxIO + 1];
  __shared__ __align__(16) float s_dy[kTrain ? NW : 1][kTrain ? 32 : 1][kMaxIO];
  __shared__ __align__(16) float s_x[kTrain ? NW : 1][kTrain ? 32 : 1][kMaxIO];
  __shared__ float s_loss[NW];
  const int t = threadIdx.x, lane = t & 63, half = lane >> 5, c = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wave = blockIdx.x * NW + wv;
  const int row = wave * 32 + c;
  const bool live = wave * 32 < a.rows;  // rows is a multiple of 64 in training
  const int H = a.hidden, fin = a.fin, fout = a.fout;
  const int nfwd = (H - 1) * NT;
  const size_t per = (size_t)W * W + W;         // parameters of a hidden layer
  const size_t base = (size_t)W * fin + W;      // those of the input layer
  const size_t wout = base + (size_t)(H - 1) * per;

  uintx4 stage[kStage];
  auto stage_load = [&](const bf16* src) {
#pragma unroll
    for (int i = 0; i < kStage; ++i)
      stage[i] = reinterpret_cast<const uintx4*>(src)[i * kThreads + t];
  };
  auto stage_store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kStage; ++i) s_ring[buf][i * kThreads + t] = stage[i];
  };
  stage_load(a.wf);
  for (int i = t; i < W * kMaxIO; i += kThreads) {
    const int j = i / kMaxIO, k = i % kMaxIO;
    s_win[j][k] = k < fin ? a.pb[j * fin + k] : (bf16)0;
    s_wout[j][k] = k < fout ? bf2f(a.pb[wout + (size_t)k * W + j]) : 0.0f;
  }
  long src = row;
  if (kTrain && a.gather) src = drawn_row(a.seed, a.step, row, a.n);
  const bool have = live && src < a.n;
  float x[FI];
#pragma unroll
  for (int k = 0; k < FI; ++k) {
    x[k] = have && k < fin ? bf2f(f2bf(a.X[(size_t)src * fin + k])) : 0.0f;
    if (kTrain && half == 0) s_x[wv][c][k] = x[k];
  }
  stage_store(0);
  __syncthreads();

  // identity operands of the 32 x 32 turn
  uintx4 id0 = {0, 0, 0, 0}, id1 = {0, 0, 0, 0};
  if (kTrain) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const unsigned one = 0x3F80u << (16 * (j & 1));
      if (c == 8 * half + j) id0[j >> 1] |= one;
      if (c == 16 + 8 * half + j) id1[j >> 1] |= one;
    }
  }
  auto turn = [&](uintx4 k0, uintx4 k1) {  // lane: column, registers: rows
    floatx16 d = {};
    d = mfma(k0, id0, d);
    return mfma(k1, id1, d);
  };
  // this lane's place in a layer: rows 0-15 of piece nt (16-31: 64 NT on)
  auto piece = [&](int nt) { return ((size_t)(2 * wave) * NT + nt) * 64 + lane; };
  // a turned piece as the weight-gradient operands of rows 0-15 and 16-31
  auto put = [&](const floatx16& d, uintx4* dst, int nt) {
    unsigned q[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = pk_bf16(d[2 * j], d[2 * j + 1]);
    uintx4 r0, r1;
    to_operands(q, r0, r1);
    if (live) {
      dst[piece(nt)] = r0;
      dst[piece(nt) + 64 * NT] = r1;
    }
  };

  uintx4 act[KS], nxt[KS];
  // bias added: keep the rounded pre-activation, round SiLU, hand it on
  auto finish = [&](int l, int nt, const float (&z)[16]) {
    unsigned p[8];
    if constexpr (kTrain) {
#pragma unroll
      for (int j = 0; j < 8; ++j) p[j] = pk_bf16(z[2 * j], z[2 * j + 1]);
      if (live) {
        uintx4* zd = a.Z + (size_t)l * a.act4 + piece(nt);
        zd[0] = uintx4{p[0], p[1], p[2], p[3]};
        zd[64 * NT] = uintx4{p[4], p[5], p[6], p[7]};
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      p[j] = pk_bf16(z[2 * j] * sigm_fast(z[2 * j]), z[2 * j + 1] * sigm_fast(z[2 * j + 1]));
    to_operands(p, nxt[2 * nt], nxt[2 * nt + 1]);
    if constexpr (kTrain)
      if (l < H - 1) put(turn(nxt[2 * nt], nxt[2 * nt + 1]), a.A + (size_t)l * a.act4, nt);
  };

  // input layer: FP32 on the rounded operands
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float z[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int n = 32 * nt + 8 * (r >> 2) + 4 * half + (r & 3);
      const uintx4 w = *reinterpret_cast<const uintx4*>(s_win[n]);
      float s = a.p[(size_t)W * fin + n];
#pragma unroll
      for (int k = 0; k < FI; ++k)
        s += ((k & 1) ? hi_bf(w[k >> 1]) : lo_bf(w[k >> 1])) * x[k];
      z[r] = s;
    }
    finish(0, nt, z);
  }
#pragma unroll
  for (int k = 0; k < KS; ++k) act[k] = nxt[k];

  // hidden layers
  for (int l = 1; l < H; ++l) {
    const float* bl = a.p + base + (size_t)(l - 1) * per + (size_t)W * W;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int cf = (l - 1) * NT + nt;
      const bool more = kTrain || cf + 1 < nfwd;
      if (more)
        stage_load(cf + 1 < nfwd ? a.wf + (size_t)(cf + 1) * 32 * W
                                 : a.wb + (size_t)(H - 2) * W * W);
      const uintx4* wl = s_ring[nt & 1];
      floatx16 acc = {};
#pragma unroll
      for (int k = 0; k < KS; ++k) acc = mfma(wl[k * 64 + lane], act[k], acc);
      float z[16];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 b = *reinterpret_cast<const float4*>(bl + 32 * nt + 8 * g + 4 * half);
        z[4 * g] = acc[4 * g] + b.x;
        z[4 * g + 1] = acc[4 * g + 1] + b.y;
        z[4 * g + 2] = acc[4 * g + 2] + b.z;
        z[4 * g + 3] = acc[4 * g + 3] + b.w;
      }
      finish(l, nt, z);
      if (more) stage_store((nt + 1) & 1);
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) act[k] = nxt[k];
  }

  // output layer, in four quarters of the width summed in order (the lower
  // lanes the first two, the upper lanes the last two; the partner lane's 8
  // of each 16 come by the swap), then pairwise
  float y[FO];
  {
    float q[2][FO];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int o = 0; o < FO; ++o) q[h][o] = 0.0f;
#pragma unroll
      for (int s = 0; s < QK; ++s) {
        const int lo = h * QK + s, hi = (2 + h) * QK + s;
        unsigned v[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uintx2 u = __builtin_amdgcn_permlane32_swap(act[lo][j], act[hi][j], false, false);
          v[j] = u.x;
          v[4 + j] = u.y;
        }
        const float(*w)[kMaxIO] = &s_wout[16 * (half ? hi : lo)];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float av = (j & 1) ? hi_bf(v[j >> 1]) : lo_bf(v[j >> 1]);
#pragma unroll
          for (int o = 0; o < FO; ++o) q[h][o] += w[j][o] * av;
        }
        pin(q[h]);
      }
    }
#pragma unroll
    for (int o = 0; o < FO; ++o) {
      float s = q[0][o] + q[1][o];
      s += __shfl_xor(s, 32, 64);
      y[o] = o < fout ? a.p[wout + (size_t)fout * W + o] + s : 0.0f;
    }
  }
  if constexpr (!kTrain) {
    if (half == 0 && row < a.n)
#pragma unroll
      for (int o = 0; o < FO; ++o)
        if (o < fout) a.Y[(size_t)row * fout + o] = y[o];
    return;
  } else {
    // mean squared error and its gradient at the output
    float dy[FO], loss = 0.0f;
#pragma unroll
    for (int o = 0; o < FO; ++o) {
      dy[o] = 0.0f;
      if (live && o < fout) {
        const float d = y[o] - a.T[(size_t)src * fout + o];
        loss += d * d;
        dy[o] = 2.0f * d / (float)(a.rows * fout);
      }
      if (half == 0) s_dy[wv][c][o] = dy[o];
    }
    for (int o = 16; o > 0; o >>= 1) loss += __shfl_down(loss, o, 32);
    if (lane == 0) s_loss[wv] = loss;
    __syncthreads();
    if (t == 0) {
      float s = 0.0f;
      for (int i = 0; i < NW; ++i) s += s_loss[i];
      a.loss_part[blockIdx.x] = s / (float)(a.rows * fout);
    }
    // sums over the block's rows: each wavefront leaves nv values per column
    // of a piece in s_tmp[buf]; after the next barrier they are added in
    // wavefront order and written
    auto leave = [&](int buf, int v, float s) {
      s += __shfl_xor(s, 32, 64);
      if (half == 0) s_tmp[buf][wv][c][v] = s;
    };
    auto collect = [&](int buf, int v) {  // of column t % 32
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < NW; ++i) s += s_tmp[buf][i][t & 31][v];
      return s;
    };
    // output layer's gradients and dZ of the last hidden layer
    // (dZ of a layer takes the place of its Z, each lane's values read before
    // it writes there)
    uintx4* dl = a.Z + (size_t)(H - 1) * a.act4;
    float* po = a.pout + (size_t)blockIdx.x * fout * (W + 1);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uintx4* zs = dl + piece(nt);
      uintx4 z0 = {0, 0, 0, 0}, z1 = z0;
      if (live) {
        z0 = zs[0];
        z1 = zs[64 * NT];
      }
      const floatx16 d = turn(act[2 * nt], act[2 * nt + 1]);
      {
        float s[FO];
#pragma unroll
        for (int o = 0; o < FO; ++o) s[o] = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float* g = s_dy[wv][8 * (r >> 2) + 4 * half + (r & 3)];
#pragma unroll
          for (int o = 0; o < FO; ++o) s[o] += g[o] * d[r];
          if ((r & 3) == 3) pin(s);
        }
#pragma unroll
        for (int o = 0; o < FO; ++o) leave(nt & 1, o, s[o]);
      }
      unsigned p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = 2 * j + i;
          const float* w = s_wout[32 * nt + 8 * (r >> 2) + 4 * half + (r & 3)];
          float g = 0.0f;
#pragma unroll
          for (int o = 0; o < FO; ++o) g += dy[o] * w[o];
          const unsigned zw = j < 4 ? z0[j & 3] : z1[j & 3];
          const float z = i ? hi_bf(zw) : lo_bf(zw), s = sigm_fast(z);
          v[i] = g * (s * (1.0f + z * (1.0f - s)));
        }
        p[j] = pk_bf16(v[0], v[1]);
      }
      to_operands(p, nxt[2 * nt], nxt[2 * nt + 1]);
      const floatx16 e = turn(nxt[2 * nt], nxt[2 * nt + 1]);
      put(e, dl, nt);
      float s = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) s += e[r];
      leave(nt & 1, kMaxIO, s);
      __syncthreads();
      for (int i = t; i < 32 * (fout + 1); i += kThreads) {  // t % 32 is the column
        const int o = i >> 5, n = 32 * nt + (i & 31);
        if (o < fout)
          po[(size_t)o * (W + 1) + n] = collect(nt & 1, o);
        else
          a.pbias[((size_t)(H - 2) * gridDim.x + blockIdx.x) * W + n] = collect(nt & 1, kMaxIO);
      }
    }
    if (t < fout) {
      float s = 0.0f;
      for (int i = 0; i < NW; ++i)
        for (int j = 0; j < 32; ++j) s += s_dy[i][j][t];
      po[(size_t)t * (W + 1) + W] = s;
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) act[k] = nxt[k];

    // dZ_{l-1} = (dZ_l W_l) SiLU'(Z_{l-1})
    for (int l = H - 1; l >= 1; --l) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const bool more = nt + 1 < NT || l > 1;
        if (more)
          stage_load(nt + 1 < NT ? a.wb + (size_t)(l - 1) * W * W + (size_t)(nt + 1) * 32 * W
                                 : a.wb + (size_t)(l - 2) * W * W);
        const uintx4* zs = a.Z + (size_t)(l - 1) * a.act4 + piece(nt);
        uintx4 z0 = {0, 0, 0, 0}, z1 = z0;
        if (live) {
          z0 = zs[0];
          z1 = zs[64 * NT];
        }
        const uintx4* wl = s_ring[nt & 1];
        floatx16 acc = {};
#pragma unroll
        for (int k = 0; k < KS; ++k) acc = mfma(wl[k * 64 + lane], act[k], acc);
        unsigned p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const unsigned zw = j < 4 ? z0[j & 3] : z1[j & 3];
          const float za = lo_bf(zw), zb = hi_bf(zw);
          const float sa = sigm_fast(za), sb = sigm_fast(zb);
          p[j] = pk_bf16(acc[2 * j] * (sa * (1.0f + za * (1.0f - sa))),
                         acc[2 * j + 1] * (sb * (1.0f + zb * (1.0f - sb))));
        }
        to_operands(p, nxt[2 * nt], nxt[2 * nt + 1]);
        const floatx16 e = turn(nxt[2 * nt], nxt[2 * nt + 1]);
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) s += e[r];
        leave(nt & 1, kMaxIO, s);
        if (l > 1) {
          put(e, a.Z + (size_t)(l - 1) * a.act4, nt);
        } else {
          float v[FI];
#pragma unroll
          for (int k = 0; k < FI; ++k) v[k] = 0.0f;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float* g = s_x[wv][8 * (r >> 2) + 4 * half + (r & 3)];
#pragma unroll
            for (int k = 0; k < FI; ++k) v[k] += e[r] * g[k];
            if ((r & 3) == 3) pin(v);
          }
#pragma unroll
          for (int k = 0; k < FI; ++k) leave(nt & 1, k, v[k]);
        }
        if (more) stage_store((nt + 1) & 1);
        __syncthreads();
        if (l > 1) {
          if (t < 32)
            a.pbias[((size_t)(l - 2) * gridDim.x + blockIdx.x) * W + 32 * nt + t] =
                collect(nt & 1, kMaxIO);
        } else {
          for (int i = t; i < 32 * (fin + 1); i += kThreads) {
            const int k = i >> 5, n = 32 * nt + (i & 31);
            a.pin[((size_t)blockIdx.x * W + n) * (fin + 1) + k] =
                collect(nt & 1, k < fin ? k : kMaxIO);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < KS; ++k) act[k] = nxt[k];
    }
  }
}

// dW_l[o][i] = sum over rows of dZ_l[row][o] A_{l-1}[row][i] for the hidden
// layers: block (split, layer) sums a run of rows into P[layer][split], four
// wavefronts of W/2 x W/2 outputs.  The operands are stored as the MFMA
// reads them (k_net), so they go from memory to registers; bound by reading
// dZ and A once (67 MB a layer at 65,536 rows of width 256).  kPre pieces of
// 16 rows are in flight per wavefront: 116 us for five such layers, 155 with
// the loads left to the scheduler, which moves them to their use, and 147
// with four blocks of a quarter of the outputs each, which read all twice.
template <int W>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4)))
k_wgrad(const uintx4* __restrict__ D, const uintx4* __restrict__ A, size_t act4, int rows_per,
        float* __restrict__ P) {
  constexpr int NT = W / 32, M = W / 64, kPre = 2;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int om = (wv >> 1) * M, im = (wv & 1) * M;
  const size_t l = blockIdx.y;
  const int nb = rows_per / 16;
  const uintx4* d = D + l * act4 + ((size_t)blockIdx.x * nb * NT + om) * 64 + lane;
  const uintx4* b = A + l * act4 + ((size_t)blockIdx.x * nb * NT + im) * 64 + lane;
  floatx16 acc[M][M];
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j) acc[i][j] = floatx16{};
  uintx4 qd[kPre][M], qa[kPre][M];
#pragma unroll
  for (int s = 0; s < kPre; ++s)
#pragma unroll
    for (int i = 0; i < M; ++i) {  // nb is even: rows_per is a multiple of 32
      qd[s][i] = d[((size_t)s * NT + i) * 64];
      qa[s][i] = b[((size_t)s * NT + i) * 64];
    }
  for (int r = 0; r < nb; r += kPre) {
#pragma unroll
    for (int s = 0; s < kPre; ++s) {
      const size_t rn = (size_t)min(r + s + kPre, nb - 1) * NT;
#pragma unroll
      for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) acc[i][j] = mfma(qd[s][i], qa[s][j], acc[i][j]);
      // the set's registers are free again: its next piece, kPre on
#pragma unroll
      for (int i = 0; i < M; ++i) {
        qd[s][i] = d[(rn + i) * 64];
        qa[s][i] = b[(rn + i) * 64];
      }
      __builtin_amdgcn_sched_barrier(0);  // the loads stay here, not at their use
    }
  }
  float* o = P + (l * gridDim.x + blockIdx.x) * (size_t)W * W;
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[(size_t)(32 * (om + i) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * W + 32 * (im + j) +
          (lane & 31)] = acc[i][j][r];
}

// All partial sums of a step to the packed gradient: kRedCols outputs per
// block, as k_reduce_splits, eight of a thread's partials in flight (46 -> 21
// us for 84 MB; one after the other they were latency).  Blocks: the hidden weights, the hidden
// biases, the input layer, the output layer.
struct NetReduce {
  const float *pw, *pbias, *pin, *pout;
  float* g;
  int W, hidden, fin, fout, splits, blocks;
};
__global__ void __launch_bounds__(256) k_reduce_net(NetReduce a) {
  __shared__ float s_sum[kRedGroups][kRedCols];
  const int c = threadIdx.x % kRedCols, grp = threadIdx.x / kRedCols;
  const int W = a.W, L1 = a.hidden - 1;
  const size_t per = (size_t)W * W + W, base = (size_t)W * a.fin + W;
  const int bw = W * W / kRedCols, bb = W / kRedCols;
  int b = blockIdx.x;
  const float* P;
  float* dst;
  int n, splits, i;
  if (b < L1 * bw) {
    const int l = b / bw;
    n = W * W;
    splits = a.splits;
    P = a.pw + (size_t)l * splits * n;
    i = (b % bw) * kRedCols + c;
    dst = a.g + base + l * per + i;
  } else if ((b -= L1 * bw) < L1 * bb) {
    const int l = b / bb;
    n = W;
    splits = a.blocks;
    P = a.pbias + (size_t)l * splits * n;
    i = (b % bb) * kRedCols + c;
    dst = a.g + base + l * per + (size_t)W * W + i;
  } else if ((b -= L1 * bb) < W * (a.fin + 1) / kRedCols) {
    n = W * (a.fin + 1);
    splits = a.blocks;
    P = a.pin;
    i = b * kRedCols + c;
    const int o = i / (a.fin + 1), k = i % (a.fin + 1);
    dst = a.g + (k < a.fin ? o * a.fin + k : W * a.fin + o);
  } else {
    b -= W * (a.fin + 1) / kRedCols;
    n = a.fout * (W + 1);
    splits = a.blocks;
    P = a.pout;
    i = b * kRedCols + c;
    const int o = i / (W + 1), k = i % (W + 1);
    dst = a.g + base + L1 * per + (k < W ? o * W + k : a.fout * W + o);
  }
  float s = 0.0f;
  if (i < n)
    for (int z = grp; z < splits; z += 8 * kRedGroups) {
      float x[8];  // in flight together, added in order (past the end: 0)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int zj = z + j * kRedGroups;
        x[j] = zj < splits ? P[(size_t)zj * n + i] : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) s += x[j];
    }
  s_sum[grp][c] = s;
  __syncthreads();
  if (grp != 0 || i >= n) return;
  float t = 0.0f;
#pragma unroll
  for (int g = 0; g < kRedGroups; ++g) t += s_sum[g][c];
  *dst = t;
}

}  // namespace mlp
}  // namespace dgbgk
