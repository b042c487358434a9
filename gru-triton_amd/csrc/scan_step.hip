// Dense GRU scan with one launch per step (gfx950): every step is a product of
// the whole batch with the whole of Wh plus the gate epilogue, spread over all
// CUs, and the stream order between launches is the only synchronisation. No
// workgroup waits for another, so there is no co-residency requirement and no
// workspace; the state of step t - 1 is read back from out (the forward) or
// from D (the backward's recurrence).
//
// These kernels serve the barrier-free entry points (gs_dense_fwd_tiled,
// gs_dense_bwd_tiled; reference gru_scan_fwd_kernel and gru_scan_bwd_kernel,
// LarocheC/gru-triton src/gru_qat/triton_kernels/scan.py:755-913, :916-1352)
// and every dense recurrence with H > 1024, where scan_tiled.hip's kernels run
// a batch tile's steps on one CU and stream all of Wh through it each step.
//
// Arithmetic. The products are those of the persistent and batch-tiled kernels
// bit for bit: 16 K slices (slice s takes k = 64 c + 4 s + e), each an fp32
// chain over c in two accumulators by the parity of e, the slices summed as
// reduce16 does. v_mfma_f32_16x16x1_4b_f32 is one fma per output element and
// block, so a wave that gives its four blocks the slices 4 w .. 4 w + 3 forms
// exactly the sixteen-block 4x4x1 instruction's chains of those slices, for 16
// rows x 16 columns instead of 4 x 4; the four waves of a workgroup cover the
// sixteen slices and meet once, in LDS, at the end of the step. The 4x4x1 form
// needs one weight operand register per instruction (4 rows x 4 columns x 16
// slices); this one reuses each operand register over 16 rows and 16 columns,
// which is what lets a whole batch share one read of the weights.
//
// MFMA layout (16x16x1, 4 blocks): lane l supplies A[block l / 16][row l % 16]
// and B[block l / 16][col l % 16]; D VGPR 4 b + v of lane l is block b's element
// (row 4 (l / 16) + v, col l % 16).
//
// Bound: with few rows the launch itself (kernel start, first loads, the LDS
// exchange and the epilogue, about 3.3 us a step), then Wh from the caches (12
// KiB a 64-k chunk and workgroup, 16 KiB with the state), and from a few hundred
// rows x 1024 units the fp32 MFMA rate: at B = 256, H = 1024 a forward step's
// products take 12.5 us at the measured 129 TFLOP/s and the step 19.9. Measured us a
// step, batch-tiled -> here: forward H = 512, B = 32: 59.6 -> 5.4; H = 2048, B = 32:
// 991 -> 12.6 (int8 codes 364 -> 7.6); whole backward per step: H = 512 37.6 -> 8.9,
// H = 2048 556 -> 35.0 (23 of it the recurrence); at B = 256, H = 1024 the recurrence takes
// 28 us a step and the whole backward 56.
#include "gs_gemm.h"
#include "gs_mfma.h"

namespace gs {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kStepThreads = 256;  // 4 waves, 4 K slices each
// LDS row stride (words) of a staged 64-word chunk row: a 16-lane pass of the
// operand reads (rows r < 8 of one slice, r >= 8 of the next, as gfx950 pairs
// them) then covers all 64 banks.
constexpr int kStepRS = 64 + 8;

struct SFParams {
  const float* gi;  // of step t
  const float* hprev;
  const float* w;  // [3H, H]
  const float* bh;
  float* out;      // of step t
  float* gh_save;  // of step t: [B, 3H], or NULL
  const int8_t* wq;
  const float* wsc;
  float pscale;
  int64_t sg_b, sh_b, so_b;
  int B, H, nch;
  Quant qin, qout;
};

// Elements k .. k + 3 of a row of H floats (the int8 kernel's state loads); those
// past its end repeat its start: the weights' codes are 0 there. (A select of the
// value right behind the load would make every load wait for its data.)
template <bool VEC>
__device__ __forceinline__ f4 load_row4(const float* row, int k, int H) {
  f4 v;
  if constexpr (VEC) {
    v = *reinterpret_cast<const f4*>(row + (k < H ? k : 0));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = row[k + e < H ? k + e : 0];
  }
  return v;
}

// Operand loads of the fp32 kernels: 16-byte raw buffer loads, whose per-lane
// offset stays put while the uniform one walks K, so a chunk costs no address
// arithmetic. Every lane of a chunk past the last, and the lanes that the last
// chunk of a row does not reach, take kOffNone and read zeros without a branch.
// gfx950 loads 16 bytes from any 4-byte address, so rows of any length and base
// are read like this (H = 501 took 12.3 us a step with single-word loads). Only
// where H is not a multiple of 4 (RAG) one lane of the last chunk has a row's
// last 1 to 3 elements: it loads the row's last four instead, and fix() moves
// them to their places. (Its offset in the chunk may then be negative, which the
// hardware would read as past the end: row_rsrc and row_off keep 16 bytes below.)
constexpr uint32_t kBufBytes = 0x7fffffffu;

template <bool RAG>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const float* p) {
  return bounded_rsrc(RAG ? p - 4 : p, kBufBytes);
}
template <bool RAG>
__device__ __forceinline__ uint32_t row_off(int64_t elems) {
  return 4u * (uint32_t)elems + (RAG ? 16u : 0u);
}

template <bool RAG> struct RowTail {
  uint32_t none;  // kOffNone for the lanes that the last chunk of a row does not reach
  uint32_t back;  // bytes by which the lane across the row's end starts earlier in the last chunk, else 0
  __device__ __forceinline__ RowTail(int k, int H)
      : none(k < H ? 0u : kOffNone), back(RAG && k < H && k + 4 > H ? 4u * (k + 4 - H) : 0u) {}
  // at_last / past_last (uniform): this is a row's last chunk / past it
  __device__ __forceinline__ f4 load(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff, bool at_last,
                                     bool past_last) const {
    const uint32_t m = at_last ? ~0u : 0u;
    if constexpr (RAG) off -= back & m;
    off |= (none & m) | (past_last ? kOffNone : 0u);
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(f4, (u4)__builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0));
  }
  // a value loaded from a row's last chunk; rem = H % 4 (uniform, not 0)
  __device__ __forceinline__ f4 fix(f4 x, int rem) const {
    const f4 y = rem == 3 ? f4{x[1], x[2], x[3], 0.f} : rem == 2 ? f4{x[2], x[3], 0.f, 0.f} : f4{x[3], 0.f, 0.f, 0.f};
    return back != 0u ? y : x;
  }
};

// step(c, I) for c = 0 .. n - 1 with I = c mod 4 at compile time. The loop runs
// whole groups of four and has one exit: leaving it in the middle of a group
// would join that path with the loop's own, and the compiler's waits for one
// register set's loads would then cover every set's.
template <typename F>
__device__ __forceinline__ void by_four(int n, F&& step) {
  const int full = n & ~3;
  for (int c = 0; c < full; c += 4) static_for<0, 4>([&](auto I) __attribute__((always_inline)) { step(c + I, I); });
  if (full + 0 < n) step(full + 0, std::integral_constant<int, 0>{});
  if (full + 1 < n) step(full + 1, std::integral_constant<int, 1>{});
  if (full + 2 < n) step(full + 2, std::integral_constant<int, 2>{});
}

// Interleaves the staging of a later chunk (vector ops, NR LDS reads, NW LDS
// writes, NL buffer loads) with a chunk's NM products: left alone, the
// scheduler puts them in front, where the matrix pipe idles (a wave issues in
// order, and the waves of a workgroup run the same phase at once).
template <int NM, int NR, int NW, int NL>
__device__ __forceinline__ void interleave() {
  static_for<0, NM>([&](auto I) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                  // MFMA
    if constexpr (I < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);            // LDS read
    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);                                  // VALU
    if constexpr (I >= NM - NW) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);      // LDS write
    if constexpr (I >= NM - NL) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);      // load
  });
}

// The in-wave part of reduce16 for one element: the two parities, then the
// wave's four slices in its order.
__device__ __forceinline__ float slice_sum(const f16v& p0, const f16v& p1, int v) {
  const float x0 = p0[v] + p1[v], x1 = p0[4 + v] + p1[4 + v];
  const float x2 = p0[8 + v] + p1[8 + v], x3 = p0[12 + v] + p1[12 + v];
  return (x0 + x2) + (x1 + x3);
}

// One step. A workgroup owns 16 RT RW batch rows x 16 hidden units (all three
// gates): RW row groups of four waves, each wave 16 RT rows. K advances in
// chunks of 64, loaded coalesced (16 lanes a row) into PD register sets in
// flight and staged through two LDS buffers.
template <int RT, int RW, bool RAG, bool SAVE, bool QA>
__global__ __launch_bounds__(kStepThreads* RW, RT == 1 ? 2 : RW) void step_fwd_kernel(SFParams p) {
  constexpr int NA = RT * RW;                // 16-row blocks of h
  constexpr int NB = NA + 3;                 // and one per gate of Wh
  constexpr int NL = (NB + RW - 1) / RW;     // blocks per thread
  constexpr int NO = RT + 3;                 // operands per wave
  constexpr int PD = RW > 1 ? 1 : 4;         // RW 1: by_four's register sets
  constexpr bool kLateGates = RW > 1;        // no registers to hold the gate inputs across the loop
  __shared__ __attribute__((aligned(16))) float lds[2][NL * RW * 16 * kStepRS];
  static_assert(sizeof(lds) >= 4 * NA * 3 * 256 * sizeof(float), "slice sums fit the staging buffers");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = (tid >> 6) & 3;           // K slices 4 wave .. 4 wave + 3
  const int rw = __builtin_amdgcn_readfirstlane(tid >> 8);  // row group
  const int H = p.H;
  const int u0 = 16 * blockIdx.x, row0 = 16 * NA * blockIdx.y;
  const int r16 = (tid >> 4) & 15, k4 = 4 * (tid & 15);

  // operand rows of this thread's loads (rows past the end repeat the last one: their products are not stored)
  const auto rh = row_rsrc<RAG>(p.hprev + (int64_t)row0 * p.sh_b);
  const auto rwt = row_rsrc<RAG>(p.w);
  const int last = p.nch - 1;
  uint32_t off[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int blk = i * RW + rw;
    off[i] = row_off<RAG>((blk < NA ? (int64_t)min(16 * blk + r16, p.B - 1 - row0) * p.sh_b
                                    : ((int64_t)min(blk - NA, 2) * H + min(u0 + r16, H - 1)) * H) +
                          k4);
  }
  const RowTail<RAG> tail(64 * last + k4, H);
  f4 reg[PD][NL];
  auto load = [&](int c, f4 (&x)[NL]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) x[i] = tail.load(i * RW + rw < NA ? rh : rwt, off[i], 256u * c, c == last, c > last);
  };
  static_for<0, PD>([&](auto I) { load(I, reg[I]); });

  // the epilogue's element i of this thread: row 16 i + 4 (lane / 16) + wave of its row group, unit lane % 16
  const int unit = u0 + (lane & 15), uc = min(unit, H - 1);
  const int erow = row0 + 16 * RT * rw + 4 * (lane >> 4) + wave;
  float gin[RT][3], hp[RT], bb[3];
  auto load_gates = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int64_t row = min(erow + 16 * i, p.B - 1);
#pragma unroll
      for (int g = 0; g < 3; ++g) gin[i][g] = p.gi[row * p.sg_b + g * H + uc];
      hp[i] = p.hprev[row * p.sh_b + uc];
    }
#pragma unroll
    for (int g = 0; g < 3; ++g) bb[g] = p.bh[g * H + uc];
  };
  if constexpr (!kLateGates) load_gates();

  f16v acc[2][RT][3];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int g = 0; g < 3; ++g)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][i][g][v] = 0.0f;

  const int st = r16 * kStepRS + k4;
  const int rd = (lane & 15) * kStepRS + 16 * wave + 4 * (lane >> 4);
  auto write = [&](int c, f4 (&x)[NL]) __attribute__((always_inline)) {
    float* buf = lds[c & 1];
    if (RAG && c == last) {  // uniform
#pragma unroll
      for (int i = 0; i < NL; ++i) x[i] = tail.fix(x[i], H & 3);
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int blk = i * RW + rw;
      f4 v = x[i];
      if constexpr (QA) {
        f4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = fake_quant(v[e], p.qin);
        v = blk < NA ? w : v;
      }
      *reinterpret_cast<f4*>(buf + blk * 16 * kStepRS + st) = v;  // (a block past NB is never read)
    }
  };
  auto read = [&](int c, f4 (&o)[NO]) __attribute__((always_inline)) {
    const float* buf = lds[c & 1];
#pragma unroll
    for (int i = 0; i < NO; ++i)
      o[i] = *reinterpret_cast<const f4*>(buf + (i < RT ? rw * RT + i : NA - RT + i) * 16 * kStepRS + rd);
  };
  auto mfma = [&](const f4 (&o)[NO]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int g = 0; g < 3; ++g)
          acc[e & 1][i][g] = __builtin_amdgcn_mfma_f32_16x16x1f32(o[i][e], o[RT + g][e], acc[e & 1][i][g], 0, 0, 0);
  };
  if constexpr (RW == 1) {
    // While chunk c's products run, chunk c + 1's operands come from LDS and
    // chunk c + 2 is staged into the buffer that chunk c's operands left (their
    // reads ended before the last barrier: lds_barrier waits for them).
    f4 o[2][NO];
    write(0, reg[0]);
    load(PD, reg[0]);
    write(1, reg[1 % PD]);
    load(PD + 1, reg[1 % PD]);
    lds_barrier();
    read(0, o[0]);
    lds_barrier();
    auto step = [&](int c, auto I) __attribute__((always_inline)) {
      read(c + 1, o[(I + 1) & 1]);
      write(c + 2, reg[(I + 2) % PD]);
      load(c + 2 + PD, reg[(I + 2) % PD]);
      mfma(o[I & 1]);
      interleave<12 * RT, NO, NL, NL>();
      lds_barrier();
    };
    by_four(p.nch, step);
  } else {
    // the second wave of each SIMD covers a wave's operand reads, so one operand set and one register set do
    write(0, reg[0]);
    load(1, reg[0]);
    lds_barrier();
    f4 o[NO];
    for (int c = 0; c < p.nch; ++c) {
      read(c, o);
      write(c + 1, reg[0]);
      load(c + 2, reg[0]);
      mfma(o);
      interleave<12 * RT, NO, NL, NL>();
      lds_barrier();
    }
  }

  if constexpr (kLateGates) load_gates();
  lds_barrier();  // every wave's operand reads are over: the buffers take the slice sums
  float* red = &lds[0][0] + rw * 4 * RT * 3 * 256;  // [wave][RT * 3][v][lane] of this row group
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int g = 0; g < 3; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[((wave * RT * 3 + i * 3 + g) * 4 + v) * 64 + lane] = slice_sum(acc[0][i][g], acc[1][i][g], v);
  lds_barrier();

  constexpr float kR = -kLog2e, kN = 2.0f * kLog2e;
  constexpr int WS = RT * 3 * 256;  // floats per wave
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    float gh[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const float* r = red + ((i * 3 + g) * 4 + wave) * 64 + lane;
      gh[g] = (r[0] + r[WS]) + (r[2 * WS] + r[3 * WS]);
    }
    const int row = erow + 16 * i;
    if (row >= p.B || unit >= H) continue;
    const float cr = __builtin_fmaf(kR, gin[i][0], kR * bb[0]);
    const float cz = __builtin_fmaf(kR, gin[i][1], kR * bb[1]), an2 = kN * gin[i][2];
    float hn = gru_update_l2(__builtin_fmaf(kR, gh[0], cr), __builtin_fmaf(kR, gh[1], cz),
                             __builtin_fmaf(kN, gh[2], kN * bb[2]), an2, hp[i]);
    if (p.qout.on) hn = fake_quant(hn, p.qout);
    p.out[(int64_t)row * p.so_b + unit] = hn;
    if constexpr (SAVE) {
      float* o = p.gh_save + (int64_t)row * 3 * H + unit;
#pragma unroll
      for (int g = 0; g < 3; ++g) __builtin_nontemporal_store(gh[g], o + g * H);
    }
  }
}

// The same step on int8 weight codes: the h levels and the codes on
// v_mfma_i32_16x16x64_i8 (exact integer sums, so any K order gives the other
// kernels' result), gh = sum * (row scale * q_in scale). K chunks of 256: wave w
// takes bytes 64 w .. 64 w + 63 of each staged row.
template <int RT, bool VEC>
__global__ __launch_bounds__(kStepThreads) void step_fwd_i8_kernel(SFParams p) {
  constexpr int NP = RT + 3;
  constexpr int PD = RT == 1 ? 3 : 2;
  __shared__ __attribute__((aligned(16))) int lds[2][NP * 16 * kStepRS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = p.H;
  const int u0 = 16 * blockIdx.x, row0 = 16 * RT * blockIdx.y;
  const int r16 = tid >> 4, c16 = tid & 15;

  const float* srch[RT];
  const int8_t* srcw[3];
#pragma unroll
  for (int i = 0; i < RT; ++i) srch[i] = p.hprev + (int64_t)min(row0 + 16 * i + r16, p.B - 1) * p.sh_b;
#pragma unroll
  for (int g = 0; g < 3; ++g) srcw[g] = p.wq + ((int64_t)g * H + min(u0 + r16, H - 1)) * H;
  struct Set {
    i4 w[3];
    f4 h[RT][4];  // words c16 + 16 j of the chunk
  };
  Set reg[PD];
  auto load = [&](int c, Set& x) __attribute__((always_inline)) {
    const int kw = 256 * c + 16 * c16;  // H % 16 == 0: 16 codes wholly inside or outside
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      x.w[g] = *reinterpret_cast<const i4*>(srcw[g] + (kw < H ? kw : 0));
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) x.h[i][j] = load_row4<VEC>(srch[i], 256 * c + 64 * j + 4 * c16, H);
  };
  const int nch = (H + 255) >> 8;
  const int last = nch - 1;
  static_for<0, PD>([&](auto I) { load(min((int)I, last), reg[I]); });

  const int unit = u0 + (lane & 15), uc = min(unit, H - 1);
  const int erow = row0 + 4 * (lane >> 4) + wave;
  float gin[RT][3], hp[RT], bb[3], sc[3];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int64_t row = min(erow + 16 * i, p.B - 1);
#pragma unroll
    for (int g = 0; g < 3; ++g) gin[i][g] = p.gi[row * p.sg_b + g * H + uc];
    hp[i] = p.hprev[row * p.sh_b + uc];
  }
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    bb[g] = p.bh[g * H + uc];
    sc[g] = p.wsc[g * H + uc] * p.pscale;
  }

  i4 acc[RT][3];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int g = 0; g < 3; ++g) acc[i][g] = i4{0, 0, 0, 0};
  const int rd = (lane & 15) * kStepRS + 16 * wave + 4 * (lane >> 4);
  auto chunk = [&](int c, Set& x, auto more) __attribute__((always_inline)) {
    int* buf = lds[c & 1];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t wd = 0;  // any level past H: W's codes are 0 there
#pragma unroll
        for (int e = 0; e < 4; ++e) wd |= ((uint32_t)(int)quant_level(x.h[i][j][e], p.qin) & 0xffu) << (8 * e);
        buf[(i * 16 + r16) * kStepRS + c16 + 16 * j] = (int)wd;
      }
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const bool in = 256 * c + 16 * c16 < H;
      *reinterpret_cast<i4*>(buf + ((RT + g) * 16 + r16) * kStepRS + 4 * c16) = in ? x.w[g] : i4{0, 0, 0, 0};
    }
    if constexpr (more) load(min(c + PD, last), x);
    lds_barrier();
    i4 o[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) o[i] = *reinterpret_cast<const i4*>(buf + i * 16 * kStepRS + rd);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int g = 0; g < 3; ++g) acc[i][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[i], o[RT + g], acc[i][g], 0, 0, 0);
  };
  const int nfull = nch / PD * PD;
  for (int c = 0; c < nfull; c += PD)
    static_for<0, PD>([&](auto I) { chunk(c + I, reg[I], std::true_type{}); });
  static_for<0, PD - 1>([&](auto I) {
    if (nfull + I < nch) chunk(nfull + I, reg[I], std::false_type{});
  });

  lds_barrier();
  int* red = &lds[0][0];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int g = 0; g < 3; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((wave * RT * 3 + i * 3 + g) * 4 + v) * 64 + lane] = acc[i][g][v];
  lds_barrier();

  constexpr float kR = -kLog2e, kN = 2.0f * kLog2e;
  constexpr int WS = RT * 3 * 256;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    float gh[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const int* r = red + ((i * 3 + g) * 4 + wave) * 64 + lane;
      gh[g] = (float)(r[0] + r[WS] + r[2 * WS] + r[3 * WS]) * sc[g];
    }
    const int row = erow + 16 * i;
    if (row >= p.B || unit >= H) continue;
    const float cr = __builtin_fmaf(kR, gin[i][0], kR * bb[0]);
    const float cz = __builtin_fmaf(kR, gin[i][1], kR * bb[1]), an2 = kN * gin[i][2];
    float hn = gru_update_l2(__builtin_fmaf(kR, gh[0], cr), __builtin_fmaf(kR, gh[1], cz),
                             __builtin_fmaf(kN, gh[2], kN * bb[2]), an2, hp[i]);
    if (p.qout.on) hn = fake_quant(hn, p.qout);
    p.out[(int64_t)row * p.so_b + unit] = hn;
  }
}

// ---- the backward's recurrence --------------------------------------------------------
//   D_{t-1} = dout[t-1] + Zm_t D_t + Mi_t (dgh_t Wh),   dgh_t = D_t (Cr, Cz, Chn)_t,
//   dh0 = Zm_0 D_0 + Mi_0 (dgh_0 Wh)
// one launch per step: M = B rows, N = H units, K = 3H over the rows of Wh (the
// gates one after the other, 64-chunks of each, as the persistent kernel's
// chain runs). Wh is read k-contiguous from a transposed copy, written once per
// call: wt[u][g][k], k zero-padded to 64 nch.
struct SBParams {
  const float* wt;
  const float* d;      // D_t [B, H]
  const float* cg;     // [B, 3H] (Cr, Cz, Chn) of step t
  const float* zm;     // [B, H] of step t
  const float* mi;     // [B, H] of step t
  const float* dprev;  // dout[t-1] (t > 0)
  float* dst;          // D_{t-1}, or dh0 at t = 0
  float* dfirst;       // t = T - 1: D_{T-1} = dout[T-1] is written here, else NULL
  int B, H, nch, last;  // last: t = 0
};

template <int RT, int CT, bool RAG>
__global__ __launch_bounds__(kStepThreads) void step_bwd_kernel(SBParams p) {
  constexpr int NP = RT + CT;
  constexpr int QS = RT * CT == 1 ? 2 : 1;  // 64-chunks per stage
  constexpr int PD = 4;                     // stages in flight
  constexpr int RS = 64 * QS + 8;
  __shared__ __attribute__((aligned(16))) float lds[2][NP * 16 * RS];
  static_assert(sizeof(lds) >= 4 * RT * CT * 256 * sizeof(float), "slice sums fit the staging buffers");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = p.H, nk = 3 * p.nch;
  const int u0 = 16 * CT * blockIdx.x, row0 = 16 * RT * blockIdx.y;
  const int r16 = tid >> 4, k4 = 4 * (tid & 15);
  const int ldw = 64 * nk;

  const auto rd_ = row_rsrc<RAG>(p.d + (int64_t)row0 * H);
  const auto rc_ = row_rsrc<RAG>(p.cg + (int64_t)row0 * 3 * H);
  const auto rw_ = row_rsrc<false>(p.wt);
  uint32_t offd[RT], offc[RT], offw[CT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const uint32_t row = min(16 * i + r16, p.B - 1 - row0);
    offd[i] = row_off<RAG>(row * H + k4);
    offc[i] = row_off<RAG>(row * 3 * H + k4);
  }
#pragma unroll
  for (int j = 0; j < CT; ++j) offw[j] = row_off<false>((int64_t)min(u0 + 16 * j + r16, H - 1) * ldw + k4);
  const RowTail<RAG> tail(64 * (p.nch - 1) + k4, H);
  const RowTail<false> whole(0, 64);  // wt's rows are padded to whole chunks
  struct Set {
    f4 d[QS][RT], c[QS][RT], w[QS][CT];
  };
  Set reg[PD];
  const int nst = (nk + QS - 1) / QS;
  auto load = [&](int s, Set& x) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < QS; ++q) {
      const int cc = s * QS + q;
      const int g = cc >= 2 * p.nch ? 2 : cc >= p.nch ? 1 : 0;
      const int kc = cc - g * p.nch;  // chunk of the gate
      const bool at_last = kc == p.nch - 1, past = cc >= nk;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        x.d[q][i] = tail.load(rd_, offd[i], 256u * kc, at_last, past);
        x.c[q][i] = tail.load(rc_, offc[i], 256u * kc + 4u * g * H, at_last, past);
      }
#pragma unroll
      for (int j = 0; j < CT; ++j) x.w[q][j] = whole.load(rw_, offw[j], 256u * cc, false, past);
    }
  };
  static_for<0, PD>([&](auto I) { load(I, reg[I]); });

  const int erow = row0 + 4 * (lane >> 4) + wave;
  float zm[RT][CT], mi[RT][CT], dn[RT][CT], dt[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int64_t e = (int64_t)min(erow + 16 * i, p.B - 1) * H + min(u0 + 16 * j + (lane & 15), H - 1);
      zm[i][j] = p.zm[e];
      mi[i][j] = p.mi[e];
      dt[i][j] = p.d[e];
      dn[i][j] = p.last ? 0.0f : p.dprev[e];
    }

  f16v acc[2][RT][CT];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][i][j][v] = 0.0f;

  const int st = r16 * RS + k4;
  const int rd = (lane & 15) * RS + 16 * wave + 4 * (lane >> 4);
  auto write = [&](int s, Set& x) __attribute__((always_inline)) {
    float* buf = lds[s & 1];
#pragma unroll
    for (int q = 0; q < QS; ++q) {
      if (RAG) {
        const int cc = s * QS + q;
        if (cc == p.nch - 1 || cc == 2 * p.nch - 1 || cc == nk - 1) {  // a gate's last chunk (uniform)
#pragma unroll
          for (int i = 0; i < RT; ++i) {
            x.d[q][i] = tail.fix(x.d[q][i], H & 3);
            x.c[q][i] = tail.fix(x.c[q][i], H & 3);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < RT; ++i) *reinterpret_cast<f4*>(buf + i * 16 * RS + st + 64 * q) = x.d[q][i] * x.c[q][i];
#pragma unroll
      for (int j = 0; j < CT; ++j) *reinterpret_cast<f4*>(buf + (RT + j) * 16 * RS + st + 64 * q) = x.w[q][j];
    }
  };
  auto read = [&](int s, f4 (&o)[QS][NP]) __attribute__((always_inline)) {
    const float* buf = lds[s & 1];
#pragma unroll
    for (int q = 0; q < QS; ++q)
#pragma unroll
      for (int i = 0; i < NP; ++i) o[q][i] = *reinterpret_cast<const f4*>(buf + i * 16 * RS + rd + 64 * q);
  };
  // (a chunk past the end adds zeros: D and C read 0 there)
  auto mfma = [&](const f4 (&o)[QS][NP]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < QS; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < CT; ++j)
            acc[e & 1][i][j] =
                __builtin_amdgcn_mfma_f32_16x16x1f32(o[q][i][e], o[q][RT + j][e], acc[e & 1][i][j], 0, 0, 0);
  };
  // the forward's pipeline, by stages
  f4 o[2][QS][NP];
  write(0, reg[0]);
  load(PD, reg[0]);
  write(1, reg[1 % PD]);
  load(PD + 1, reg[1 % PD]);
  lds_barrier();
  read(0, o[0]);
  lds_barrier();
  auto step = [&](int s, auto I) __attribute__((always_inline)) {
    read(s + 1, o[(I + 1) & 1]);
    write(s + 2, reg[(I + 2) % PD]);
    load(s + 2 + PD, reg[(I + 2) % PD]);
    mfma(o[I & 1]);
    interleave<4 * QS * RT * CT, QS * NP, QS * NP, QS * (NP + RT)>();
    lds_barrier();
  };
  by_four(nst, step);

  lds_barrier();
  float* red = &lds[0][0];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[((wave * RT * CT + i * CT + j) * 4 + v) * 64 + lane] = slice_sum(acc[0][i][j], acc[1][i][j], v);
  lds_barrier();

  constexpr int WS = RT * CT * 256;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const float* r = red + ((i * CT + j) * 4 + wave) * 64 + lane;
      const float via_w = (r[0] + r[WS]) + (r[2 * WS] + r[3 * WS]);
      const int row = erow + 16 * i, u = u0 + 16 * j + (lane & 15);
      if (row >= p.B || u >= H) continue;
      const int64_t e = (int64_t)row * H + u;
      float carry;
      {
#pragma clang fp contract(off)
        carry = zm[i][j] * dt[i][j] + mi[i][j] * via_w;
      }
      if (p.dfirst != nullptr) p.dfirst[e] = dt[i][j];
      p.dst[e] = p.last ? carry : dn[i][j] + carry;
    }
}

// wt[u][g][k] = Wh[g H + k][u], zero for k in [H, 64 nch). One workgroup per
// 64 x 64 tile of a gate, transposed through LDS.
__global__ __launch_bounds__(256) void step_transpose_kernel(const float* __restrict__ w, float* __restrict__ wt,
                                                             int H, int nch) {
  __shared__ float tile[64][65];
  const int g = blockIdx.z, k0 = 64 * blockIdx.x, u0 = 64 * blockIdx.y;
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  for (int i = y; i < 64; i += 4)
    tile[i][x] = (k0 + i < H && u0 + x < H) ? w[((int64_t)g * H + k0 + i) * H + u0 + x] : 0.0f;
  __syncthreads();
  for (int i = y; i < 64; i += 4)
    if (u0 + i < H) wt[((int64_t)(u0 + i) * 3 + g) * 64 * nch + k0 + x] = tile[x][i];
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Whether [a, a + an) and [b, b + bn) (floats) share memory.
bool overlap(const float* a, int64_t an, const float* b, int64_t bn) { return a < b + bn && b < a + an; }

// Smallest H that takes a launch per step: below, a batch tile's step on one CU
// (scan_tiled.hip) is not longer than a launch on the GPU and its 2.5 us on the
// host. B = 32, T = 64, us a step, one CU against a launch: forward 2.9 / 3.6 at
// H = 64, 5.7 / 3.8 at 128, 12.2 / 4.1 at 192; backward (all its passes) 3.5 / 4.6 at 64,
// 6.4 / 5.0 at 128, 9.7 / 6.2 at 192.
constexpr int64_t kStepMinH = 129;
constexpr int64_t kStepMaxB = 16 * 65535;  // 16-row tiles in the grid's second dimension

// A training step is some 120 to 160 us of host time, behind which a few steps
// of few units run on one CU for nothing, while a launch each adds 2.5 us to it.
// Forward and backward, us, one-CU kernels / launches: T = 8, B = 4, H = 140
// 152 / 173; T = 6, B = 32, H = 200 176 / 189; T = 10, B = 16, H = 160 208 / 212;
// T = 3, B = 16, H = 320 164 / 171 (T H^2 = 157000 to 307000); T = 10, B = 2, H = 361
// 1120 / 204. So training scans take launches from T H^2 = 400000 on, or for one step.
bool enough_steps(int64_t T, int64_t H) { return T == 1 || T * H * H >= 400000; }

}  // namespace

// The step kernels address a workgroup's state rows (at most 64) with 32-bit
// byte offsets, and read all of a step's previous state while they write its
// next: h0 (and gi) must not share memory with out, which one CU running a
// batch tile's steps by itself allows (scan_tiled.hip).
bool step_fwd_applies(const gs_args* a) {
  if (a->H < kStepMinH || a->B > kStepMaxB) return false;
  if (a->gh_save != nullptr && !enough_steps(a->T, a->H)) return false;
  if (a->B > 1 && std::max(a->sh0_b, a->so_b) > int64_t(1) << 22) return false;
  const int64_t n_out = (a->T - 1) * a->so_t + (a->B - 1) * a->so_b + a->H;
  const int64_t n_gi = (a->T - 1) * a->sg_t + (a->B - 1) * a->sg_b + 3 * a->H;
  return !overlap(a->out, n_out, a->h0, (a->B - 1) * a->sh0_b + a->H) && !overlap(a->out, n_out, a->gi, n_gi) &&
         !overlap(a->out, n_out, a->w, 3 * a->H * a->H);
}

namespace {
// 4-row blocks that a group of the persistent dense kernels (KC 16 and up) takes
// in turn: one workgroup of 16 units per CU.
int64_t persistent_rounds(int64_t B, int64_t H) {
  const int64_t groups = std::max<int64_t>(1, 256 / ((H + 15) / 16));
  return ((B + 3) / 4 + groups - 1) / groups;
}
// T launches cost the host 2.5 us each, which shows while the whole recurrence
// is only some 50 us of a call that the host bounds.
bool pays_launches(int64_t T, int64_t rounds) { return T == 1 || T * rounds >= 32; }
}  // namespace

// The persistent kernels take about 1.2 us (H <= 256), 1.65 (<= 512) or 2.9 (<= 1024)
// a round, with the packed exchange (pack) 1.3, 1.55 or 2.5, int8 codes 0.8, 1.1 or
// 1.0; a step here 4 to 8 us plus its products, more where rows are not whole
// 64-byte lines (H % 16) and where gh is saved along such rows. So each of them moves
// the number of rounds from which a step here is shorter. Measured at T = 40, us a
// step, persistent / here: H = 256, B = 384 (6 rounds) 6.7 / 5.5; H = 384, B = 160 (4)
// 6.8 / 5.4; H = 512, B = 128 (4) 6.2 / 5.9, packed 5.8 / 5.8; H = 500, B = 128 (4) 6.1 / 6.2,
// B = 160 (5) packed 7.2 / 7.4, packed with gh 7.4 / 8.2; H = 640, B = 72 (3) 8.6 / 6.3;
// H = 900, B = 48 (3) 8.6 / 7.8, packed 7.6 / 7.8; H = 1000, B = 48 (3) 8.7 / 8.9, packed
// 7.6 / 8.9, B = 64 (4) packed 10.0 / 11.0, B = 80 (5) packed with gh 12.7 / 12.3; H = 1024,
// B = 48 (3) 8.7 / 8.0, packed 7.6 / 7.9, B = 256 (16) 44.3 / 19.6. int8 codes: H = 256,
// B = 384 (6) 4.5 / 4.4; H = 384, B = 160 (4) 5.1 / 4.1; H = 768, B = 96 (5) 5.9 / 6.5,
// B = 160 (8) 8.6 / 6.5; H = 1024, B = 160 (10) 9.7 / 11.3, B = 256 (16) 15.2 / 11.7.
static int64_t least_rounds(int64_t H, int kc, bool i8, bool pack, bool save) {
  if (i8) return kc == 16 ? 7 : kc == 32 ? 4 : H <= 768 ? 7 : 12;
  if (kc == 16) return 6;
  const bool lines = H % 16 == 0;
  if (kc == 32) {
    if (lines || H <= 320) return 4;
    return save ? (H <= 384 ? 5 : 6) : H <= 448 ? 4 : pack ? 6 : 5;
  }
  if (lines) return pack && H > 896 ? 4 : 3;
  return H <= (pack || save ? 832 : 928) ? 3 : pack && H > 960 ? 5 : 4;
}

bool step_fwd_beats_persistent(const gs_args* a, bool i8, bool pack) {
  const int kc = a->H <= kPersistentMaxH ? choose_kc((int)a->H) : 0;
  const int64_t rounds = kc < 16 ? 0 : persistent_rounds(a->B, a->H);
  return kc >= 16 && rounds >= least_rounds(a->H, kc, i8, pack, a->gh_save != nullptr) &&
         pays_launches(a->T, rounds) && step_fwd_applies(a);
}

// The whole backward, us a step, persistent / here: H = 256, B = 384 (6 rounds)
// 14.4 / 14.2, B = 512 (8) 18.4 / 16.3; H = 512, B = 160 (5) 17.1 / 18.4, B = 256 (8)
// 27 / 23; H = 1024, B = 32 (2) 17.2 / 18.4, B = 48 (3) 24.1 / 20.6, B = 256 (16) 122 / 63.
bool step_bwd_beats_persistent(int64_t T, int64_t B, int64_t H) {
  const int kc = H <= kPersistentMaxH ? choose_kc((int)H) : 0;
  const int64_t least = kc == 16 ? 7 : kc == 32 ? 7 : 3;
  const int64_t rounds = kc < 16 ? 0 : persistent_rounds(B, H);
  return kc >= 16 && B <= kStepMaxB && rounds >= least && pays_launches(T, rounds);
}

// dh0 is written by the launch that reads D_0, and dout is D_{T-1}.
bool step_bwd_applies(const float* dout, const float* dh0, int64_t T, int64_t B, int64_t H) {
  return H >= kStepMinH && B <= kStepMaxB && enough_steps(T, H) && !overlap(dh0, B * H, dout, T * B * H);
}

// The forward, one launch per step (see the header comment).
int run_step_fwd(const gs_args* a, hipStream_t stream, const int8_t* codes, const float* scales) {
  const int B = (int)a->B, H = (int)a->H;
  SFParams p;
  p.w = a->w;
  p.bh = a->bh;
  p.sg_b = a->sg_b;
  p.so_b = a->so_b;
  p.B = B;
  p.H = H;
  p.nch = (H + 63) / 64;
  p.qin = to_quant(a->q_in);
  p.qout = to_quant(a->q_out);
  const bool i8 = codes != nullptr && dense_i8_applies(a) && al16(codes);
  p.wq = i8 ? codes : nullptr;
  p.wsc = i8 ? scales : nullptr;
  p.pscale = a->q_in.scale;
  const bool save = a->gh_save != nullptr;
  const int nut = (H + 15) / 16;
  // Rows a workgroup: 16, 32 or 64. A CU takes its workgroups of one kind in
  // turn (or overlaps them, at much the same cost each): relative cost of one
  // 64-k chunk 0.30 us for 16 rows, 0.48 for the first and 0.61 for each further
  // workgroup of 32, 0.95 and 1.05 of 64 (H = 1024, B = 64 ... 512). int8 (its time
  // is the level conversion, per row): 32 rows where that still fills the CUs.
  auto rounds = [&](int r) { return (double)(((int64_t)((B + r - 1) / r) * nut + 255) / 256); };
  int rt = 1;
  if (i8) {
    rt = B > 16 && (int64_t)((B + 31) / 32) * nut >= 224 ? 2 : 1;
  } else {
    const double c1 = 0.30 * rounds(16), c2 = 0.48 + 0.61 * (rounds(32) - 1), c4 = 0.95 + 1.05 * (rounds(64) - 1);
    rt = c1 <= c2 && c1 <= c4 ? 1 : c2 <= c4 ? 2 : 4;
  }
  const dim3 grid((unsigned)nut, (unsigned)((B + 16 * rt - 1) / (16 * rt)));
  typedef void (*Fn)(SFParams);
#define GS_STEP_FWD_Q(R, S, Q) {step_fwd_kernel<1, 1, R, S, Q>, step_fwd_kernel<1, 2, R, S, Q>, step_fwd_kernel<2, 2, R, S, Q>}
#define GS_STEP_FWD(R, S) {GS_STEP_FWD_Q(R, S, false), GS_STEP_FWD_Q(R, S, true)}
  static const Fn f32[2][2][2][3] = {{GS_STEP_FWD(false, false), GS_STEP_FWD(false, true)},
                                  {GS_STEP_FWD(true, false), GS_STEP_FWD(true, true)}};
#undef GS_STEP_FWD
#undef GS_STEP_FWD_Q
  static const Fn q8[2][2] = {{step_fwd_i8_kernel<1, false>, step_fwd_i8_kernel<2, false>},
                              {step_fwd_i8_kernel<1, true>, step_fwd_i8_kernel<2, true>}};
  const int ri = rt == 4 ? 2 : rt == 2 ? 1 : 0;
  for (int64_t t = 0; t < a->T; ++t) {
    p.gi = a->gi + t * a->sg_t;
    p.hprev = t == 0 ? a->h0 : a->out + (t - 1) * a->so_t;
    p.sh_b = t == 0 ? a->sh0_b : a->so_b;
    p.out = a->out + t * a->so_t;
    p.gh_save = save ? a->gh_save + t * B * 3 * H : nullptr;
    const bool quant_a = a->q_in.enabled && (t == 0 || !same_quant(a->q_in, a->q_out));
    const bool vec = al16(p.hprev) && (B == 1 || p.sh_b % 4 == 0);
    const Fn fn = i8 ? q8[vec ? 1 : 0][ri] : f32[H % 4 != 0 ? 1 : 0][save ? 1 : 0][quant_a ? 1 : 0][ri];
    hipLaunchKernelGGL(fn, grid, dim3(rt > 1 && !i8 ? 2 * kStepThreads : kStepThreads), 0, stream, p);
    GS_CHECK_HIP(hipGetLastError());
  }
  return GS_OK;
}

// Step 3 of the dense backward, one launch per step. wt: tiled_bwd_wt_bytes of scratch.
int run_step_bwd_recurrence(const float* w, float* wt, const float* dout, const float* cg, const float* zm,
                            const float* mi, float* dsum, float* dh0, int64_t T, int64_t B, int64_t H,
                            hipStream_t stream) {
  const int nch = (int)((H + 63) / 64);
  hipLaunchKernelGGL(step_transpose_kernel, dim3((unsigned)nch, (unsigned)nch, 3), dim3(256), 0, stream, w, wt, (int)H,
                     nch);
  GS_CHECK_HIP(hipGetLastError());
  const int64_t BH = B * H;
  SBParams p;
  p.wt = wt;
  p.B = (int)B;
  p.H = (int)H;
  p.nch = nch;
  // 16 x 16, 32 x 16 or 32 x 32 (rows x units) a workgroup, by rounds of 256 workgroups; relative cost of a
  // workgroup 6.5, 10 and 17 us at K = 3 x 1024
  auto rounds = [&](int rt, int ct) {
    return (double)((((B + 16 * rt - 1) / (16 * rt)) * ((H + 16 * ct - 1) / (16 * ct)) + 255) / 256);
  };
  const double c0 = 6.5 * rounds(1, 1), c1 = 10.0 * rounds(2, 1), c2 = 17.0 * rounds(2, 2);
  const int sel = c0 <= c1 && c0 <= c2 ? 0 : c1 <= c2 ? 1 : 2;
  const int rt = sel >= 1 ? 2 : 1, ct = sel == 2 ? 2 : 1;
  typedef void (*Fn)(SBParams);
  static const Fn table[2][3] = {
      {step_bwd_kernel<1, 1, false>, step_bwd_kernel<2, 1, false>, step_bwd_kernel<2, 2, false>},
      {step_bwd_kernel<1, 1, true>, step_bwd_kernel<2, 1, true>, step_bwd_kernel<2, 2, true>}};
  const dim3 grid((unsigned)((H + 16 * ct - 1) / (16 * ct)), (unsigned)((B + 16 * rt - 1) / (16 * rt)));
  for (int64_t t = T - 1; t >= 0; --t) {
    const bool first = t == T - 1;
    p.d = first ? dout + t * BH : dsum + t * BH;
    p.cg = cg + t * 3 * BH;
    p.zm = zm + t * BH;
    p.mi = mi + t * BH;
    p.dprev = t > 0 ? dout + (t - 1) * BH : nullptr;
    p.dst = t > 0 ? dsum + (t - 1) * BH : dh0;
    p.dfirst = first ? dsum + t * BH : nullptr;
    p.last = t == 0;
    hipLaunchKernelGGL(table[H % 4 != 0 ? 1 : 0][sel], grid, dim3(kStepThreads), 0, stream, p);
    GS_CHECK_HIP(hipGetLastError());
  }
  return GS_OK;
}

}  // namespace gs
