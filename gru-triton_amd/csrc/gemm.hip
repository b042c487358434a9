// fp32 GEMM on v_mfma_f32_16x16x4f32 (gfx950) for the products around the
// scans: the backward's recomputation of the hidden projection for all steps
// at once, gh = q_in([h0; out[0..T-2]]) Wh^T + bh (NT), and the weight
// gradient dWh = dgh^T q_in([h0; out[0..T-2]]) (TN) -- the per-step products
// of the reference backward (src/gru_qat/triton_kernels/scan.py:388-421 and
// :576-619), batched over every step because neither depends on the reverse
// recurrence.
//
// Tiling: a workgroup of 4 waves computes a T x T tile of C, T = 128 or 64
// (big_tiles says which); wave (wy, wx) owns a quarter as MFMA tiles of
// 16 x 16 (4 x 4 or 2 x 2 of them). K advances in slices of 2048 / T, so that
// a thread loads 8 floats of each operand whatever T is. A slice's products
// take the operands read from LDS during the slice before, while the next is
// read, the one after it goes from registers to LDS and the one two further is
// loaded: nothing the matrix pipe does waits for memory, and the schedule
// below puts all of it between the MFMAs. Loads are raw buffer loads along
// each operand's contiguous dimension, 16 bytes where its extent is a multiple
// of 4 floats (whatever the base and the row stride: gfx950 loads 16 bytes
// from any 4-byte address) and single words where it is not; per-lane offsets
// stay put while the uniform base walks K, and lanes past an edge carry an
// offset past the buffer, which reads zeros. Operands land in LDS without
// transposition:
//   k-contiguous operand: S[row][k], row stride BK + 8;
//   row-contiguous operand: S[k][row], row stride T + 4 (NN) or T + 16 (TN).
// A k-contiguous operand is read as float4s: lane (row r, k-group q) reads
// k = 4 q + 16 h, and MFMA s takes k = 4 q + 16 (s / 4) + s % 4.
// gfx950 serves a 16-byte LDS read in 16-lane passes that pair 8-lane groups
// {0, 3}, {1, 2}, {4, 7}, {5, 6}, i.e. rows r < 8 of one k-group with rows
// r >= 8 of the next; with stride 24 or 40 (6 or 10 four-bank groups) every row
// starts on an even group and the two k-groups of a pass sit one group apart,
// so a pass covers all 64 banks. A row-contiguous operand is read as single
// words (32 banks, 32-lane passes covering k-groups q and q + 1): under the NN
// mapping those rows are 4 k apart, 4 (T + 4) = 16 mod 32 words; under TN's
// k = q + 4 s they are 1 k apart, T + 16 = 16 mod 32. Any bijection between
// (MFMA step, k-group) and k is valid as long as A and B use the same one; an
// element's MFMAs run over the same k in the same order for both T.
//
// Bound: the fp32 MFMA rate (16x16x4: 130-145 TFLOP/s with nothing else on
// this chip), and for small products the last round of workgroups and the
// 8 us or so that first loads and last stores take. Measured against one
// 64 x 64 tile kernel that staged a slice, met at a barrier, and then issued
// its 32 MFMAs: M = 32768, N = 3072, K = 1024 (128 x 128) NT 2101 -> 1470 us
// (140 TFLOP/s), NN 2052 -> 1414, TN 2309 -> 1404; M = 2048, N = 1536, K = 512
// (64 x 64) NT 42.2 -> 34.9, NN 43.2 -> 35.1, TN 42.3 -> 36.7; single words,
// M = 32768, N = 1503, K = 301: NT 449 -> 362, NN 454 -> 338, TN 517 -> 351.
// Rows of any length in 16-byte loads (the last one moved back to the row's
// end, its floats shifted on their way to LDS) were slower than single words
// where rows are off 64-byte lines: 480 against 446 us at M = 8192, N = 3072,
// K = 1023.
//
// MFMA operand layout (16x16x4 f32): lane l supplies A[i = l % 16][k-group
// l / 16] and B[k-group l / 16][j = l % 16]; D VGPR v of lane l is
// C[4 (l / 16) + v][l % 16].
#include "gs_gemm.h"
#include "gs_mfma.h"

namespace gs {
namespace {

constexpr int kGemmThreads = 256;
constexpr int kSmallT = 64, kBigT = 128;
constexpr int kSplitK = 32;  // K splits start at multiples of this: whole slices of either tile

// How an operand's tile is loaded: 16 bytes or one float per buffer load, or
// (rows too far apart for 32-bit offsets) one float at a 64-bit address.
enum { kLoadVec = 0, kLoadWord = 1, kLoadFar = 2 };

// One operand's tile of a slice: T rows of the output dimension x BK k, from
// memory to 8 registers of each thread, then into LDS. KC: contiguous along k.
template <bool KC, int T, int LOAD, int RS>
struct TileLoader {
  static constexpr int BK = 2048 / T, KS = BK + 8;
  static constexpr int kStage = KC ? T * KS : BK * RS;
  static constexpr int W = LOAD == kLoadVec ? 4 : 1, NV = 8 / W;
  static constexpr int PR = (KC ? BK : T) / W;  // loads per contiguous run
  const float* base;  // LOAD != kLoadFar: the first slice's first k, the tile's first row
  int64_t ld, step;   // floats to the next row (k, if not KC); to the next slice
  uint32_t off[NV], tail[NV];

  static __device__ __forceinline__ void at(int e, int* row, int* k) {
    const int idx = threadIdx.x + kGemmThreads * e, run = idx / PR, in = (idx % PR) * W;
    *row = KC ? run : in;
    *k = KC ? in : run;
  }
  // rows row0 .. lim_row - 1, k from kbeg; klast: the first k of the last slice
  __device__ __forceinline__ void init(const float* p, int64_t ld_, int row0, int lim_row, int kbeg, int klast,
                                       int kend) {
    ld = ld_;
    base = KC ? p + (int64_t)row0 * ld + kbeg : p + (int64_t)kbeg * ld + row0;
    step = KC ? BK : BK * ld;
#pragma unroll
    for (int e = 0; e < NV; ++e) {
      int row, k;
      at(e, &row, &k);
      off[e] = row0 + row >= lim_row ? kOffNone
               : LOAD == kLoadFar    ? 0u
                                     : (uint32_t)(4 * (KC ? row * (int)ld + k : k * (int)ld + row));
      tail[e] = klast + k < kend ? 0u : kOffNone;
    }
  }
  // slice s of n; past the last one: zeros, without touching memory
  __device__ __forceinline__ void load(int s, int n, float (&x)[8]) const {
    const uint32_t m = s == n - 1 ? ~0u : 0u, past = s >= n ? kOffNone : 0u;
    const float* b = base + s * step;
    if constexpr (LOAD == kLoadFar) {
#pragma unroll
      for (int e = 0; e < NV; ++e) {
        int row, k;
        at(e, &row, &k);
        x[e] = (off[e] | (tail[e] & m) | past) ? 0.0f : b[KC ? row * ld + k : k * ld + row];
      }
    } else {
      const auto r = bounded_rsrc(b, 0x7fffffffu);
#pragma unroll
      for (int e = 0; e < NV; ++e) {
        const uint32_t o = off[e] | (tail[e] & m) | past;
        if constexpr (LOAD == kLoadVec) {
          typedef unsigned int u4 __attribute__((ext_vector_type(4)));
          const u4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) x[4 * e + i] = __uint_as_float(v[i]);
        } else {
          x[e] = buf_ld(r, o, 0);
        }
      }
    }
  }
  template <bool QUANT>
  __device__ __forceinline__ void stage(float* d, const float (&x)[8], const Quant& q) const {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = QUANT ? fake_quant(x[i], q) : x[i];  // fake_quant(0) == 0: the padding stays
#pragma unroll
    for (int e = 0; e < NV; ++e) {
      int row, k;
      at(e, &row, &k);
      float* o = d + (KC ? row * KS + k : k * RS + row);
      if constexpr (LOAD == kLoadVec)
        *reinterpret_cast<f4*>(o) = f4{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
      else
        *o = v[e];
    }
  }
};

// A wave's MT operand tiles of one slice: v[t][h][e] feeds MFMA 4 h + e.
template <bool KC, bool TN, int BK, int RS, int MT>
__device__ __forceinline__ void read_operand(const float* s, int row, int kq, f4 (&v)[MT][BK / 16]) {
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int h = 0; h < BK / 16; ++h) {
      if constexpr (KC) {
        v[t][h] = *reinterpret_cast<const f4*>(s + (row + 16 * t) * (BK + 8) + 4 * kq + 16 * h);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[t][h][e] = s[(16 * h + (TN ? kq + 4 * e : 4 * kq + e)) * RS + row + 16 * t];
      }
    }
}

// The schedule of a slice's NM MFMAs: NR LDS reads from the first on, NS LDS
// writes and as many loads towards the last (left alone, the scheduler puts
// them all in front, where the matrix pipe idles).
template <int NM, int NR, int NS>
__device__ __forceinline__ void interleave() {
  constexpr int kRead = (NR + NM - 1) / NM, kPut = (4 * NS + NM - 1) / NM;  // puts: over the last half
  static_for<0, NM>([&](auto I) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                             // MFMA
    if constexpr (I * kRead < NR) __builtin_amdgcn_sched_group_barrier(0x100, kRead, 0);  // LDS read
    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);                             // VALU
    if constexpr (I >= NM / 2 && (I - NM / 2) * kPut < NS) __builtin_amdgcn_sched_group_barrier(0x200, kPut, 0);
    if constexpr (I >= NM / 2 && (I - NM / 2) * kPut >= NS) __builtin_amdgcn_sched_group_barrier(0x020, kPut, 0);
  });
}

// Q: fake-quantizes A (NT) or B (TN) on its way to LDS.
// Four workgroups of NT's small tiles fit a CU, which short products, bound by
// their stores, are the faster for (M = 16384, N = 1536, K = 64: 60 -> 53 us);
// NN and TN lose more to the registers (their backward 112 -> 116 us).
template <int LAYOUT, int T, int LOAD, bool Q>
__global__ __launch_bounds__(kGemmThreads, T == kBigT || LOAD == kLoadFar                ? 2
                                           : LAYOUT == kGemmNT && LOAD == kLoadVec ? 4
                                                                                   : 3) void gemm_kernel(GemmArgs g) {
  constexpr bool A_KC = LAYOUT != kGemmTN, B_KC = LAYOUT == kGemmNT, TN = LAYOUT == kGemmTN;
  constexpr bool QA = Q && LAYOUT == kGemmNT, QB = Q && LAYOUT == kGemmTN;
  constexpr int RS = T + (LAYOUT == kGemmNN ? 4 : 16);
  typedef TileLoader<A_KC, T, LOAD, RS> LA;
  typedef TileLoader<B_KC, T, LOAD, RS> LB;
  constexpr int BK = LA::BK, MT = T / 32, KH = BK / 16;
  __shared__ __attribute__((aligned(16))) float As[2][LA::kStage];
  __shared__ __attribute__((aligned(16))) float Bs[2][LB::kStage];
  // this workgroup's tile: patches of 1024 rows; of big tiles, each XCD
  // (workgroup mod 8) takes a run, whose operands its L2 then holds
  const int mt = (g.M + T - 1) / T, nt = (g.N + T - 1) / T, total = mt * nt;
  const int wg = blockIdx.y * gridDim.x + blockIdx.x, per = (total + 7) / 8;
  const int tile = T == kBigT ? (wg & 7) * per + (wg >> 3) : wg;
  if ((T == kBigT && (wg >> 3) >= per) || tile >= total) return;  // uniform
  constexpr int kPatch = 1024 / T;
  const int patch = tile / (kPatch * nt), in_patch = tile - patch * kPatch * nt;
  const int pm = min(kPatch, mt - patch * kPatch);
  const int i0 = (patch * kPatch + in_patch % pm) * T, j0 = in_patch / pm * T;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wy = wave >> 1, wx = wave & 1;
  const int kper = ((g.K + g.ksplit - 1) / g.ksplit + kSplitK - 1) / kSplitK * kSplitK;
  const int z = blockIdx.z / g.ksplit, split = blockIdx.z - z * g.ksplit;
  const int kbeg = split * kper, kend = min(g.K, kbeg + kper);
  const int n = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
  const int klast = kbeg + (n - 1) * BK;

  LA la;
  LB lb;
  la.init(g.a + (int64_t)(z % g.a_mod) * g.a_bs, g.lda, i0, g.M, kbeg, klast, kend);
  lb.init(g.b + (int64_t)(z % g.b_mod) * g.b_bs, g.ldb, j0, g.N, kbeg, klast, kend);
  float xa[2][8], xb[2][8];
  la.load(0, n, xa[0]);
  lb.load(0, n, xb[0]);
  la.load(1, n, xa[1]);
  lb.load(1, n, xb[1]);

  f4 acc[MT][MT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, kq = lane >> 4;
  f4 oa[2][MT][KH], ob[2][MT][KH];
  auto read = [&](auto I) __attribute__((always_inline)) {
    read_operand<A_KC, TN, BK, RS, MT>(As[I], 16 * MT * wy + r16, kq, oa[I]);
    read_operand<B_KC, TN, BK, RS, MT>(Bs[I], 16 * MT * wx + r16, kq, ob[I]);
  };
  auto put = [&](int s, auto I) __attribute__((always_inline)) {  // slice s to LDS; its registers take s + 2
    la.template stage<QA>(As[I], xa[I], g.qa);
    lb.template stage<QB>(Bs[I], xb[I], g.qb);
    la.load(s + 2, n, xa[I]);
    lb.load(s + 2, n, xb[I]);
  };
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  auto products = [&](auto I) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4 * KH; ++e)
#pragma unroll
      for (int ti = 0; ti < MT; ++ti)
#pragma unroll
        for (int tj = 0; tj < MT; ++tj)
          acc[ti][tj] = __builtin_amdgcn_mfma_f32_16x16x4f32(oa[I][ti][e >> 2][e & 3], ob[I][tj][e >> 2][e & 3],
                                                             acc[ti][tj], 0, 0, 0);
  };
  put(0, I0);
  if (n > 1) put(1, I1);
  lds_barrier();
  read(I0);
  lds_barrier();  // slice 0 is read: its half of the LDS takes slice 2
  // slice s + 2 is staged where slice s was: every wave read that one before
  // the barrier that ended slice s - 1
  auto slice = [&](int s, auto I, auto J) __attribute__((always_inline)) {
    read(J);
    put(s + 2, I);
    products(I);
    interleave<4 * KH * MT * MT, MT * KH * ((A_KC ? 1 : 4) + (B_KC ? 1 : 4)), LA::NV + LB::NV>();
    lds_barrier();
  };
  int s = 0;
  for (; s + 2 < n; s += 2) {  // in pairs, so that the loop has one exit
    slice(s, I0, I1);
    slice(s + 1, I1, I0);
  }
  // the last one or two: nothing further to stage
  if (s + 1 < n) read(I1);
  if (s < n) products(I0);
  if (s + 1 < n) products(I1);

  float* c = g.c + (int64_t)z * g.c_bs + (int64_t)split * g.split_stride;
  const float* biasp = g.bias ? g.bias + (int64_t)z * g.bias_bs : nullptr;
  const bool add_bias = biasp != nullptr && split == 0;
#pragma unroll
  for (int tj = 0; tj < MT; ++tj) {
    const int j = j0 + 16 * (MT * wx + tj) + r16;
    if (j >= g.N) continue;
    const float bias = add_bias ? biasp[j] : 0.0f;
#pragma unroll
    for (int ti = 0; ti < MT; ++ti)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = i0 + 16 * (MT * wy + ti) + 4 * kq + v;
        if (i < g.M) c[(int64_t)i * g.ldc + j] = acc[ti][tj][v] + bias;
      }
  }
}

// ---- int8 NT product (gemm_i8_nt) -----------------------------------------------
// A 64 x 64 tile of C per workgroup of 4 waves, each wave 2 x 2 tiles of
// v_mfma_i32_16x16x64_i8; K advances by 64, double-buffered through LDS. Each
// thread loads 16 consecutive k (16 bytes) of one row of each operand and
// stores them with one 16-byte LDS write; a row holds 64 bytes in a stride of
// 20 words, so the 16 rows that a 16-lane pass of the operand reads start on
// distinct 4-bank groups (20 r mod 64) and the 16-byte reads are free of
// conflicts. MFMA operand layout: lane l supplies the 16 bytes of row l % 16
// at k-group l / 16 for A and for B alike, so whatever k the hardware assigns
// a byte, A's and B's bytes at one position are the same k; D VGPR v of lane
// l is C[4 (l / 16) + v][l % 16].
constexpr int kI8Tile = 64, kI8BK = 64, kI8RowWords = 20;
typedef int i4v __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(kGemmThreads) void gemm_i8_nt_kernel(GemmI8Args g) {
  __shared__ __attribute__((aligned(16))) int As[2][kI8Tile * kI8RowWords];
  __shared__ __attribute__((aligned(16))) int Bs[2][kI8Tile * kI8RowWords];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wy = wave >> 1, wx = wave & 1;
  const int i0 = blockIdx.x * kI8Tile, j0 = blockIdx.y * kI8Tile;
  // loader: row lr of the tile, k = 16 lk .. 16 lk + 15 of the slice
  const int lr = threadIdx.x >> 2, lk = threadIdx.x & 3;
  const int ra = i0 + lr, rb = j0 + lr;
  const bool oka = ra < g.M, okb = rb < g.N;
  const int8_t* pa = g.a + (int64_t)(oka ? ra : 0) * g.lda + 16 * lk;
  const int8_t* pb = g.b + (int64_t)(okb ? rb : 0) * g.ldb + 16 * lk;
  i4v va, vb;
  auto load = [&](int k0) {
    const bool in = k0 + 16 * lk < g.K;  // K % 16 == 0: 16 bytes wholly inside or outside
    va = (oka && in) ? *reinterpret_cast<const i4v*>(pa + k0) : i4v{0, 0, 0, 0};
    vb = (okb && in) ? *reinterpret_cast<const i4v*>(pb + k0) : i4v{0, 0, 0, 0};
  };
  auto stage = [&](int buf) {
    *reinterpret_cast<i4v*>(&As[buf][lr * kI8RowWords + 4 * lk]) = va;
    *reinterpret_cast<i4v*>(&Bs[buf][lr * kI8RowWords + 4 * lk]) = vb;
  };
  i4v acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = i4v{0, 0, 0, 0};
  const int r16 = lane & 15, kg = lane >> 4;
  int buf = 0;
  load(0);
  stage(0);
  __syncthreads();
  for (int k0 = 0; k0 < g.K; k0 += kI8BK) {
    const bool more = k0 + kI8BK < g.K;
    if (more) load(k0 + kI8BK);
    i4v a[2], b[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      a[t] = *reinterpret_cast<const i4v*>(&As[buf][(32 * wy + 16 * t + r16) * kI8RowWords + 4 * kg]);
      b[t] = *reinterpret_cast<const i4v*>(&Bs[buf][(32 * wx + 16 * t + r16) * kI8RowWords + 4 * kg]);
    }
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
      for (int tj = 0; tj < 2; ++tj) acc[ti][tj] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[ti], b[tj], acc[ti][tj], 0, 0, 0);
    if (more) stage(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
#pragma unroll
  for (int tj = 0; tj < 2; ++tj) {
    const int j = j0 + 32 * wx + 16 * tj + r16;
    if (j >= g.N) continue;
    const float sc = g.sa * g.b_scale[j];
    const float bias = g.bias ? g.bias[j] : 0.0f;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = i0 + 32 * wy + 16 * ti + 4 * kg + v;
        if (i < g.M) g.c[(int64_t)i * g.ldc + j] = (float)acc[ti][tj][v] * sc + bias;
      }
  }
}

__global__ void quant_codes_kernel(float* dst_q, int8_t* codes, const float* src, int64_t ld, int rows, int cols,
                                   Quant q) {
  const int64_t n = (int64_t)rows * cols;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = e / cols;
    const int i = (int)(e - m * cols);
    const float lv = quant_level(src[m * ld + i], q);
    if (dst_q != nullptr) dst_q[e] = lv * q.scale;
    codes[e] = (int8_t)(int)lv;
  }
}

__global__ void sum_partials_kernel(float* dst, const float* src, int64_t n, int parts, int64_t stride) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    float s = src[e];
    for (int p = 1; p < parts; ++p) s += src[p * stride + e];
    dst[e] = s;
  }
}

// Two independent sums of partials in one launch: element e < a.n of job a,
// then the elements of job b.
__global__ void sum_partials2_kernel(SumJob a, SumJob b) {
  const int64_t n = a.n + b.n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const bool first = e < a.n;
    const SumJob& j = first ? a : b;
    const int64_t i = first ? e : e - a.n;
    float s = j.src[i];
    for (int p = 1; p < j.parts; ++p) s += j.src[p * j.stride + i];
    j.dst[i] = s;
  }
}

// Column sums: a workgroup takes 64 columns x kColRows rows; its 256 threads
// are 64 columns x 4 row lanes, each lane summing every 4th row (8 loads in
// flight), and the 4 lanes are combined through LDS into partial[chunk][j].
constexpr int kColRows = 256;
__global__ __launch_bounds__(256) void colsum_kernel(const float* src, int64_t ld, int rows, int cols,
                                                     float* partial) {
  __shared__ float red[4][64];
  const int jl = threadIdx.x & 63, lane_r = threadIdx.x >> 6;
  const int j = blockIdx.x * 64 + jl;
  const int r0 = blockIdx.y * kColRows;
  const int r1 = min(rows, r0 + kColRows);
  float s = 0.0f;
  if (j < cols) {
    int r = r0 + lane_r;
    for (; r + 28 < r1; r += 32) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[(int64_t)(r + 4 * u) * ld + j];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; r < r1; r += 4) s += src[(int64_t)r * ld + j];
  }
  red[lane_r][jl] = s;
  __syncthreads();
  if (lane_r == 0 && j < cols)
    partial[(int64_t)blockIdx.y * cols + j] = ((red[0][jl] + red[1][jl]) + red[2][jl]) + red[3][jl];
}

__global__ void quant_copy_kernel(float* dst, const float* src, int64_t ld, int rows, int cols, Quant q) {
  const int64_t n = (int64_t)rows * cols;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = e / cols;
    const int i = (int)(e - m * cols);
    dst[e] = fake_quant(src[m * ld + i], q);
  }
}

__global__ void prev_state_kernel(float* hq, const float* h0, int64_t sh0_b, const float* out, int64_t so_b,
                                  int64_t rows, int B, int H, Quant q) {
  const int64_t n = rows * H;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = e / H;
    const int k = (int)(e - m * H);
    float v = m < B ? h0[m * sh0_b + k] : out[(m - B) * so_b + k];
    if (q.on) v = fake_quant(v, q);
    hq[e] = v;
  }
}

typedef void (*GemmFn)(GemmArgs);

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int64_t tile_count(int M, int N, int T) { return (int64_t)((M + T - 1) / T) * ((N + T - 1) / T); }

// Microseconds that a product takes beyond what both tile sizes spend, from
// runs on the chip: the CUs take tiles in rounds of 256; a 128 x 128 tile does
// one k in 0.059 us of its CU, a 64 x 64 one in 0.0158 (TN, whose operands come
// from LDS in single words: 0.0165); first loads and last stores, during which
// the matrix pipes idle, take 25 us more with big tiles.
double tiles_us(int T, int layout, int64_t tiles, int64_t kper) {
  const double rounds = (double)((tiles + 255) / 256);
  return T == kBigT ? rounds * kper * 0.059 + 25.0 : rounds * kper * (layout == kGemmTN ? 0.0165 : 0.0158);
}

// 128 x 128 tiles read each operand word half as often, but come in quarters
// of the number: they pay where there are many rounds of long tiles. M = 32768,
// N = 3072, K = 1024, NT: 1501 us with 64 x 64, 1463 with 128 x 128 (its TN in
// four splits 1594 and 1404); M = 2048, N = 1536, K = 512: 33 and 46;
// M = 8192, N = 1536, K = 512: 114 and 122.
bool big_tiles(const GemmArgs& g) {
  const int64_t kper = (g.K + g.ksplit - 1) / g.ksplit, n = (int64_t)g.batch * g.ksplit;
  return tiles_us(kBigT, g.layout, tile_count(g.M, g.N, kBigT) * n, kper) <
         tiles_us(kSmallT, g.layout, tile_count(g.M, g.N, kSmallT) * n, kper);
}

}  // namespace

// K split of a product. For 64 x 64 tiles: at least two workgroups per CU of
// the MI355X (256 CUs) where K allows it (at least 256 terms per split, at
// most 16 splits), and among those splits the one whose last round of
// workgroups fills the CUs best (smallest on ties). The dense backward's dWh
// at T=64, B=32, H=512 (192 tiles) then splits K in 4 (768 workgroups, 3 per
// CU) rather than 3 (576, a last round a quarter full): 51.5 -> 42.1 us.
// Then any split in 128 x 128 tiles that is faster, each costing its partials'
// way to memory and back (4.5 TB/s) and the launch that adds them: M = 3072,
// N = 1024, K = 32768 takes 1404 us in 192 big tiles and four splits, and took
// 2309 in 768 small ones unsplit (1660 now). Never fewer splits than the small
// tiles would have: each fp32 accumulator would sum a longer chain for it (K = 4282
// in one chain instead of 16: relative error 1.2e-6 instead of 3.2e-7).
int gemm_pick_split(int M, int N, int K) {
  constexpr int kCUs = 256;
  const int64_t tiles = tile_count(M, N, kSmallT);
  const int smax = std::max(1, std::min(16, (K + 255) / 256));
  int best = 1;
  int64_t best_num = -1, best_den = 1;  // fill fraction best_num / best_den
  for (int s = 1; s <= smax; ++s) {
    const int64_t n = (int64_t)tiles * s;
    if (n < 2 * kCUs && s < smax) continue;
    const int64_t den = (int64_t)kCUs * ((n + kCUs - 1) / kCUs);
    if (n * best_den > best_num * den) {
      best = s;
      best_num = n;
      best_den = den;
    }
  }
  auto us = [&](int T, int s) {
    const double sum = s > 1 ? 4.0 + (s + 1.0) * M * N * 4e-6 / 4.5 : 0.0;
    return tiles_us(T, kGemmTN, tile_count(M, N, T) * s, (K + s - 1) / s) + sum;
  };
  double least = us(kSmallT, best);
  for (int s = best; s <= smax; ++s)
    if (us(kBigT, s) < least) {
      best = s;
      least = us(kBigT, s);
    }
  return best;
}

int gemm_f32(const GemmArgs& g, hipStream_t stream, const char* who) {
  if (g.M < 1 || g.N < 1 || g.K < 1 || g.ksplit < 1)
    return set_error(GS_ERR_INVALID, "%s: GEMM dims must be positive (M=%d, N=%d, K=%d, ksplit=%d)", who, g.M, g.N,
                     g.K, g.ksplit);
  if (g.batch < 1 || g.a_mod < 1 || g.b_mod < 1 || (int64_t)g.batch * g.ksplit > 65535)
    return set_error(GS_ERR_INVALID, "%s: bad GEMM batch (batch=%d, a_mod=%d, b_mod=%d, ksplit=%d)", who, g.batch,
                     g.a_mod, g.b_mod, g.ksplit);
  if (g.layout != kGemmNT && g.layout != kGemmTN && g.layout != kGemmNN)
    return set_error(GS_ERR_INVALID, "%s: unknown GEMM layout %d", who, g.layout);
  const bool a_kc = g.layout != kGemmTN, b_kc = g.layout == kGemmNT;
  const bool vec = (a_kc ? g.K % 4 == 0 : g.M % 4 == 0) && (b_kc ? g.K % 4 == 0 : g.N % 4 == 0);
  // the farthest float of a slice's tile from its first, for 32-bit byte offsets
  auto reach = [](bool kc, int64_t ld, int T) { return (kc ? T : 2048 / T) * ld + (kc ? 2048 / T : T); };
  auto near = [&](int T) {
    return std::max(reach(a_kc, g.lda, T), reach(b_kc, g.ldb, T)) < (int64_t(1) << 29);
  };
  const bool big = near(kBigT) && big_tiles(g);
  const int load = !near(kSmallT) ? kLoadFar : vec ? kLoadVec : kLoadWord;
#define GS_GEMM_ROW(L, T, V) {gemm_kernel<L, T, V, false>, gemm_kernel<L, T, V, L != kGemmNN>}
#define GS_GEMM_LAYOUT(L) \
  {GS_GEMM_ROW(L, kSmallT, kLoadVec), GS_GEMM_ROW(L, kSmallT, kLoadWord), GS_GEMM_ROW(L, kSmallT, kLoadFar), \
   GS_GEMM_ROW(L, kBigT, kLoadVec), GS_GEMM_ROW(L, kBigT, kLoadWord)}
  static const GemmFn table[3][5][2] = {GS_GEMM_LAYOUT(kGemmNT), GS_GEMM_LAYOUT(kGemmTN), GS_GEMM_LAYOUT(kGemmNN)};
#undef GS_GEMM_LAYOUT
#undef GS_GEMM_ROW
  const bool quant = g.layout == kGemmNT ? g.qa.on : g.qb.on;
  if ((g.qa.on || g.qb.on) && (!quant || g.layout == kGemmNN || (g.qa.on && g.qb.on)))
    return set_error(GS_ERR_INVALID, "%s: GEMM layout %d quantizes no such operand", who, g.layout);
  GemmFn fn = table[g.layout][big ? 3 + load : load][quant ? 1 : 0];
  int64_t tiles = tile_count(g.M, g.N, big ? kBigT : kSmallT);
  if (big) tiles = 8 * ((tiles + 7) / 8);
  const int64_t gx = std::min<int64_t>(tiles, 1 << 20);  // for big tiles a multiple of 8
  if (tiles > INT32_MAX || (tiles + gx - 1) / gx > 65535)
    return set_error(GS_ERR_INVALID, "%s: GEMM of too many tiles (M=%d, N=%d)", who, g.M, g.N);
  const dim3 grid((unsigned)gx, (unsigned)((tiles + gx - 1) / gx), (unsigned)(g.batch * g.ksplit));
  hipLaunchKernelGGL(fn, grid, dim3(kGemmThreads), 0, stream, g);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

bool gemm_i8_applies(const GemmI8Args& g) {
  return g.K >= 1 && g.K <= 65536 && g.K % 16 == 0 && g.lda % 16 == 0 && g.ldb % 16 == 0 && aligned16(g.a) &&
         aligned16(g.b) && g.b_scale != nullptr;
}

int gemm_i8_nt(const GemmI8Args& g, hipStream_t stream, const char* who) {
  if (g.M < 1 || g.N < 1 || !gemm_i8_applies(g))
    return set_error(GS_ERR_INVALID, "%s: int8 GEMM operands out of its contract (M=%d, N=%d, K=%d)", who, g.M, g.N,
                     g.K);
  const dim3 grid((unsigned)((g.M + kI8Tile - 1) / kI8Tile), (unsigned)((g.N + kI8Tile - 1) / kI8Tile));
  hipLaunchKernelGGL(gemm_i8_nt_kernel, grid, dim3(kGemmThreads), 0, stream, g);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

int quant_copy_codes(float* dst_q, int8_t* codes, const float* src, int64_t ld, int rows, int cols, const Quant& q,
                     hipStream_t stream, const char* who) {
  (void)who;
  const int64_t n = (int64_t)rows * cols;
  hipLaunchKernelGGL(quant_codes_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)), dim3(256), 0,
                     stream, dst_q, codes, src, ld, rows, cols, q);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

int sum_partials(float* dst, const float* src, int64_t n, int parts, int64_t stride, hipStream_t stream,
                 const char* who) {
  (void)who;
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(sum_partials_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, stream, dst,
                     src, n, parts, stride);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

int sum_partials2(const SumJob& a, const SumJob& b, hipStream_t stream, const char* who) {
  (void)who;
  const int64_t blocks = (a.n + b.n + 255) / 256;
  if (blocks == 0) return GS_OK;
  hipLaunchKernelGGL(sum_partials2_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, stream, a,
                     b);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

int64_t colsum_partial_floats(int rows, int cols) { return (int64_t)((rows + kColRows - 1) / kColRows) * cols; }

int colsum(float* dst, const float* src, int64_t ld, int rows, int cols, float* partials, hipStream_t stream,
           const char* who) {
  const int chunks = (rows + kColRows - 1) / kColRows;
  hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((cols + 63) / 64), (unsigned)chunks), dim3(256), 0, stream, src,
                     ld, rows, cols, partials);
  GS_CHECK_HIP(hipGetLastError());
  return sum_partials(dst, partials, cols, chunks, cols, stream, who);
}

int quant_copy(float* dst, const float* src, int64_t ld, int rows, int cols, const Quant& q, hipStream_t stream,
               const char* who) {
  (void)who;
  const int64_t n = (int64_t)rows * cols;
  hipLaunchKernelGGL(quant_copy_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)), dim3(256), 0, stream,
                     dst, src, ld, rows, cols, q);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

int build_prev_state(float* hq, const float* h0, int64_t sh0_b, const float* out, int64_t so_b, int T, int B, int H,
                     const Quant& q, hipStream_t stream, const char* who) {
  (void)who;
  const int64_t n = (int64_t)T * B * H;
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(prev_state_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream, hq, h0,
                     sh0_b, out, so_b, (int64_t)T * B, B, H, q);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

}  // namespace gs
