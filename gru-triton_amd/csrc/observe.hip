// Observer path (gfx950): the GRU scan and a tensor quantizer with per-tensor
// fake-quants whose scale is computed on the device from the tensor itself,
// and whose running statistics are updated, as GRULayer.calibrate runs them.
//
// Reference: the per-step path GRULayer.forward takes with use_triton off
// (LarocheC/gru-triton src/gru_qat/gru_layer.py:205-223) over step_with_gi
// (gru_cell.py:437-464), with FakeQuantize.forward (quantizers.py:84-96) in
// the dynamic or min_max mode: _compute_scale_zp of FakeQuantizePerTensor
// (quantizers.py:176-181) through _scale_zp_from_min_max (:124-134), then
// _update_observer (:136-156) in min_max mode, then fake_quant_ste
// (ste.py:65-95). calibrate (calibration.py:31-126, gru_layer.py:308-336)
// switches the activation quantizers to min_max and runs such forwards.
//
// A quantizer's scale depends on the min and max of the whole tensor it sees,
// so every step has a grid-wide reduction between computing h_t and
// quantizing it. The steps therefore run as one launch each on the stream, with
// all scales kept on the device:
//   once:      the map as a dense [3H, H] matrix (gs_hidden_map_dense) unless
//              the kind is dense or diagonal; (min, max) partials of h0.
//   step t:    every workgroup reduces the partials of the pre-quant h_{t-1}
//              itself and derives q_out's and q_in's scales (workgroup 0 alone
//              updates the statistics and the trace), applies both to the rows
//              it multiplies, and runs the product, the gates and the (min, max)
//              partial of its part of the pre-quant h_t. out[t-1] = q_out(h_{t-1})
//              is written on the way by the workgroup that owns the element.
//   at last:   out[T-1] = q_out(h_{T-1}).
// Batches whose step would be several rounds of workgroups take three launches a
// step instead (one_launch): the product by gemm.hip with K split, the gates, and a
// quantizer pass, which fill the CUs better there. Same bits either way.
// fq is monotone, so the min and max of q_out(h_{t-1}), which q_in sees at step
// t, are q_out of the pre-quant min and max: one reduction per step covers
// both quantizers.
#include "gs_gemm.h"
#include "gs_mfma.h"

namespace gs {

int validate_map(const gs_map_args* a, const char* who);
int64_t hidden_map_scratch(const gs_map_args* a);
int materialize_map(const gs_map_args* a, hipStream_t stream, const char* who);

namespace {

constexpr int kRedThreads = 256;
constexpr int kMaxParts = 512;  // (min, max) partials of one reduction
constexpr int kMaxSplit = 8;    // K splits of a step's product (one wave each in observe_step_kernel)
// _update_observer's mixing weights as the fp32 values torch multiplies by.
constexpr float kKeep = (float)0.99;
constexpr float kMix = (float)(1.0 - 0.99);

struct Obs {
  int mode, sym;
  float qmin, qmax, scale, zp;
  float* stats;
};

struct ObsPair {
  Obs in, out;
};

// (Only min_max keeps statistics: elsewhere a stats pointer, which may be the other observer's, is nobody's.)
Obs to_obs(const gs_observer& o) {
  return Obs{o.mode, o.symmetric, (float)o.qmin, (float)o.qmax, o.scale, o.zero_point,
             o.mode == GS_OBS_MIN_MAX ? o.stats : nullptr};
}

__host__ __device__ inline bool is_dynamic(const Obs& o) {
  return o.mode == GS_OBS_DYNAMIC || o.mode == GS_OBS_MIN_MAX;
}

// fake_quant_ste's forward: clamp(round(x / s + zp), qmin, qmax), then (q - zp) s.
__device__ __forceinline__ float fq(float x, float s, float zp, float qmin, float qmax) {
#pragma clang fp contract(off)
  float v = __builtin_rintf(x / s + zp);
  v = __builtin_fminf(__builtin_fmaxf(v, qmin), qmax);
  return (v - zp) * s;
}

__device__ __forceinline__ void scale_zp(const Obs& o, float mn, float mx, float* s, float* zp) {
#pragma clang fp contract(off)
  if (o.sym) {
    const float a = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(mx), __builtin_fabsf(mn)), 1e-8f);
    *s = a / o.qmax;
    *zp = 0.0f;
  } else {
    *s = __builtin_fmaxf(mx - mn, 1e-8f) / (o.qmax - o.qmin);
    *zp = __builtin_rintf(o.qmin - mn / *s);
  }
}

__device__ __forceinline__ void observe(const Obs& o, float mn, float mx) {
  if (o.mode != GS_OBS_MIN_MAX) return;
  float* st = o.stats;
  if (st[2] == 0.0f) {
    st[0] = mn;
    st[1] = mx;
    st[2] = 1.0f;
  } else {
#pragma clang fp contract(off)
    st[0] = kKeep * st[0] + kMix * mn;
    st[1] = kKeep * st[1] + kMix * mx;
  }
}

// (min, max) over the workgroup, written by thread 0 to *dst.
__device__ __forceinline__ void block_minmax(float mn, float mx, float2* dst) {
  __shared__ float red[2][kRedThreads / 64];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    mn = __builtin_fminf(mn, __shfl_xor(mn, o));
    mx = __builtin_fmaxf(mx, __shfl_xor(mx, o));
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][wave] = mn;
    red[1][wave] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kRedThreads / 64; ++w) {
      mn = __builtin_fminf(mn, red[0][w]);
      mx = __builtin_fmaxf(mx, red[1][w]);
    }
    *dst = float2{mn, mx};
  }
}

__global__ __launch_bounds__(kRedThreads) void minmax_partials(const float* x, int64_t rows, int cols, int64_t ld,
                                                               float2* part) {
  float mn = __builtin_inff(), mx = -__builtin_inff();
  const int64_t n = rows * cols;
  for (int64_t e = blockIdx.x * (int64_t)kRedThreads + threadIdx.x; e < n; e += (int64_t)gridDim.x * kRedThreads) {
    const int64_t r = e / cols;
    const float v = x[r * ld + (e - r * cols)];
    mn = __builtin_fminf(mn, v);
    mx = __builtin_fmaxf(mx, v);
  }
  block_minmax(mn, mx, part + blockIdx.x);
}

// One quantizer pass. Every workgroup first reduces the np (min, max)
// partials (np = 0: no dynamic quantizer needs them) and derives the scales
// itself; workgroup 0 alone writes them back to st, the trace and the running
// statistics. phase 0: the partials are of what c.in sees (h0, or the tensor of
// gs_observe_tensor), and hq = q_in(x). phase 1: they are of step t's
// pre-quant h_t in x, which c.out sees; then y = q_out(x) goes to dst (when
// apply_out) and, for step t + 1, hq = q_in(y), with q_in's scale from the min
// and max of y (q_out of the pre-quant ones). A word of st is written in a
// phase-1 launch only when its quantizer is dynamic, and read then by
// workgroup 0 alone (for the trace).
__global__ __launch_bounds__(kRedThreads) void quant_step(const float2* part, int np, ObsPair c, float* st,
                                                          float* trace, int t, int T, int phase, const float* x,
                                                          int64_t ldx, float* dst, int64_t ldd, float* hq,
                                                          int64_t rows, int cols, int apply_out) {
  __shared__ float2 tot;
  __shared__ float sc[4];
  float mn = __builtin_inff(), mx = -__builtin_inff();
  if (np > 0) {
    for (int i = threadIdx.x; i < np; i += kRedThreads) {
      mn = __builtin_fminf(mn, part[i].x);
      mx = __builtin_fmaxf(mx, part[i].y);
    }
    block_minmax(mn, mx, &tot);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const bool writer = blockIdx.x == 0;
    const bool din = is_dynamic(c.in), dout = is_dynamic(c.out);
    if (np > 0) {
      mn = tot.x;
      mx = tot.y;
    }
    float s_in = 1.0f, zp_in = 0.0f, s_out = 1.0f, zp_out = 0.0f;
    if (!din && c.in.mode == GS_OBS_FROZEN) {
      s_in = c.in.scale;
      zp_in = c.in.zp;
    }
    if (!dout && c.out.mode == GS_OBS_FROZEN) {
      s_out = c.out.scale;
      zp_out = c.out.zp;
    }
    if (phase == 0) {
      if (din) scale_zp(c.in, mn, mx, &s_in, &zp_in);
      if (writer) {
        if (din) observe(c.in, mn, mx);
        st[0] = s_in;  // no workgroup reads st in phase 0
        st[1] = zp_in;
      }
    } else {
      if (dout) {
        scale_zp(c.out, mn, mx, &s_out, &zp_out);
        if (writer) observe(c.out, mn, mx);
      }
      if (writer && trace != nullptr) {
        float* tr = trace + (int64_t)t * 4;
        tr[0] = din ? st[0] : s_in;  // the q_in scale step t used
        tr[1] = din ? st[1] : zp_in;
        tr[2] = s_out;
        tr[3] = zp_out;
      }
      if (din && t + 1 < T) {
        float a = mn, b = mx;
        if (c.out.mode != GS_OBS_OFF) {
          a = fq(mn, s_out, zp_out, c.out.qmin, c.out.qmax);
          b = fq(mx, s_out, zp_out, c.out.qmin, c.out.qmax);
        }
        scale_zp(c.in, a, b, &s_in, &zp_in);
        if (writer) {
          observe(c.in, a, b);
          st[0] = s_in;
          st[1] = zp_in;
        }
      }
    }
    sc[0] = s_in;
    sc[1] = zp_in;
    sc[2] = s_out;
    sc[3] = zp_out;
  }
  __syncthreads();
  const float s_in = sc[0], zp_in = sc[1], s_out = sc[2], zp_out = sc[3];
  const int64_t n = rows * cols;
  for (int64_t e = blockIdx.x * (int64_t)kRedThreads + threadIdx.x; e < n; e += (int64_t)gridDim.x * kRedThreads) {
    const int64_t r = e / cols;
    const int k = (int)(e - r * cols);
    float v = x[r * ldx + k];
    if (apply_out) v = fq(v, s_out, zp_out, c.out.qmin, c.out.qmax);
    if (dst != nullptr) dst[r * ldd + k] = v;
    if (hq != nullptr) hq[e] = fq(v, s_in, zp_in, c.in.qmin, c.in.qmax);
  }
}

// The gates of one step of the three-launch form; writes the pre-quant h_t to
// out_t and a (min, max) partial per workgroup. gh comes from `nsplit` GEMM
// partials [B, 3H] (split 0 holds the bias).
__global__ __launch_bounds__(kRedThreads) void gates_step(const float* gi_t, int64_t sg_b, const float* gh, int nsplit,
                                                          int64_t split_stride, const float* hprev, int64_t shp_b,
                                                          float* out_t, int64_t so_b, int B, int H, float2* part) {
  float mn = __builtin_inff(), mx = -__builtin_inff();
  const int64_t n = (int64_t)B * H;
  for (int64_t e = blockIdx.x * (int64_t)kRedThreads + threadIdx.x; e < n; e += (int64_t)gridDim.x * kRedThreads) {
    const int b = (int)(e / H), k = (int)(e - (int64_t)b * H);
    const float* p = gh + (int64_t)b * 3 * H + k;
    float v[kMaxSplit][3], g3[3];
#pragma unroll
    for (int q = 0; q < kMaxSplit; ++q)
#pragma unroll
      for (int g = 0; g < 3; ++g) v[q][g] = q < nsplit ? p[q * split_stride + g * H] : 0.0f;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      float sum = v[0][g];
#pragma unroll
      for (int q = 1; q < kMaxSplit; ++q)
        if (q < nsplit) sum += v[q][g];
      g3[g] = sum;
    }
    const float* gr = gi_t + (int64_t)b * sg_b + k;
    const float h = gru_update(gr[0], gr[H], gr[2 * H], g3[0], g3[1], g3[2], hprev[(int64_t)b * shp_b + k]);
    out_t[(int64_t)b * so_b + k] = h;
    mn = __builtin_fminf(mn, h);
    mx = __builtin_fmaxf(mx, h);
  }
  block_minmax(mn, mx, part + blockIdx.x);
}

// ---- one step ------------------------------------------------------------------------

// fq at a scale found at run time. A symmetric one in quant_code's range takes
// its division-free quotient, which equals the IEEE one (gs_device.h). Codes stay
// within kQuickCodes there: the bound under which q_in repeats q_out (same_quant,
// gs_host.h), inside the 2^24 up to which the quotient holds.
constexpr int kQuickCodes = 1 << 22;
struct DynQuant {
  Quant q;
  float zp;
  int on, fast;
  __device__ __forceinline__ float operator()(float x) const {
#pragma clang fp contract(off)
    if (fast) {
      float v = quant_code(x, q);
      v = __builtin_fminf(__builtin_fmaxf(v, q.qmin), q.qmax);
      return v * q.scale;
    }
    return on ? fq(x, q.scale, zp, q.qmin, q.qmax) : x;
  }
};

// WIDE: the range may exceed kQuickCodes.
template <bool WIDE>
__device__ __forceinline__ DynQuant dyn_quant(const Obs& o, float s, float zp) {
  DynQuant d{{s, o.qmin, o.qmax, 1, 1.0f / s}, zp, o.mode != GS_OBS_OFF, 0};
  d.fast = d.on && zp == 0.0f && s >= 0x1p-126f && s <= 0x1p64f;
  if constexpr (WIDE) d.fast = d.fast && o.qmin >= (float)-kQuickCodes && o.qmax <= (float)kQuickCodes;
  return d;
}

struct OStep {
  const float* gi;     // of step t
  const float* hprev;  // pre-quant h_{t-1}, or h0
  const float* w;      // the map [3H, H], or the diagonal kind's [3, H]
  const float* bh;
  float* hnext;        // pre-quant h_t
  float* out_prev;     // out[t-1], or NULL at t = 0
  const float2* part_in;
  float2* part_out;
  float* st;     // the scale and zero point of q_in at step t (written here; read for step t - 1's trace)
  float* trace;  // of step t - 1, or NULL
  ObsPair c;
  int64_t sg_b, sh_b, sn_b, so_b;
  int B, H, first, np, nsplit;
};

// (min, max) over the wave, in every lane, with VALU lane moves.
__device__ __forceinline__ void wave_minmax(float& mn, float& mx) {
  static_for<0, 6>([&](auto I) {
    mn = __builtin_fminf(mn, lane_xor_c<(1 << I)>(mn));
    mx = __builtin_fmaxf(mx, lane_xor_c<(1 << I)>(mx));
  });
}

// What step_scales reads, loaded by every thread before anything else: memory
// returns in order, and behind the operand loads these would wait for all of
// them (workgroup 0 for a second trip, in front of everyone else's step t + 1).
struct StepIn {
  float2 part[4];  // lanes past the last partial repeat it
  float in[3], out[3], st[2];
};

__device__ __forceinline__ StepIn load_step_in(const OStep& p) {
  StepIn v;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < 4; ++j) v.part[j] = p.part_in[min(lane + 64 * j, max(p.np, 1) - 1)];
  const float* si = p.c.in.mode == GS_OBS_MIN_MAX ? p.c.in.stats : p.st;
  const float* so = p.c.out.mode == GS_OBS_MIN_MAX ? p.c.out.stats : p.st;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    v.in[j] = si[j];
    v.out[j] = so[j];
  }
  v.st[0] = p.st[0];
  v.st[1] = p.st[1];
  return v;
}

// observe() on statistics already in registers.
__device__ __forceinline__ void observe_in(const Obs& o, float (&s)[3], float mn, float mx) {
#pragma clang fp contract(off)
  if (o.mode != GS_OBS_MIN_MAX) return;
  s[0] = s[2] == 0.0f ? mn : kKeep * s[0] + kMix * mn;
  s[1] = s[2] == 0.0f ? mx : kKeep * s[1] + kMix * mx;
  s[2] = s[2] == 0.0f ? 1.0f : s[2];
#pragma unroll
  for (int j = 0; j < 3; ++j) o.stats[j] = s[j];
}

// Reduces the partials (each wave by itself: no barrier) and derives the scales
// of step t: q_out for h_{t-1} (none at t = 0: h0 is not quantized) and q_in.
// Workgroup 0 updates the statistics, the scale words and the trace.
template <bool WIDE>
__device__ __forceinline__ void step_scales(const OStep& p, StepIn& v, DynQuant* qout, DynQuant* qin) {
  float mn = v.part[0].x, mx = v.part[0].y;
#pragma unroll
  for (int j = 1; j < 4; ++j) {
    mn = __builtin_fminf(mn, v.part[j].x);
    mx = __builtin_fmaxf(mx, v.part[j].y);
  }
  for (int i = 256 + (threadIdx.x & 63); i < p.np; i += 64) {
    const float2 w = p.part_in[i];
    mn = __builtin_fminf(mn, w.x);
    mx = __builtin_fmaxf(mx, w.y);
  }
  wave_minmax(mn, mx);
  const bool writer = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
  const bool din = is_dynamic(p.c.in), dout = is_dynamic(p.c.out);
  float s_out = p.c.out.mode == GS_OBS_FROZEN ? p.c.out.scale : 1.0f;
  float zp_out = p.c.out.mode == GS_OBS_FROZEN ? p.c.out.zp : 0.0f;
  float s_in = p.c.in.mode == GS_OBS_FROZEN ? p.c.in.scale : 1.0f;
  float zp_in = p.c.in.mode == GS_OBS_FROZEN ? p.c.in.zp : 0.0f;
  if (!p.first) {
    if (dout) {
      scale_zp(p.c.out, mn, mx, &s_out, &zp_out);
      if (writer) {
        observe_in(p.c.out, v.out, mn, mx);
        if (p.c.in.stats == p.c.out.stats) {  // one quantizer in both places
#pragma unroll
          for (int j = 0; j < 3; ++j) v.in[j] = v.out[j];
        }
      }
    }
    if (writer && p.trace != nullptr) {
      p.trace[0] = din ? v.st[0] : s_in;  // what step t - 1 used
      p.trace[1] = din ? v.st[1] : zp_in;
      p.trace[2] = s_out;
      p.trace[3] = zp_out;
    }
    if (p.c.out.mode != GS_OBS_OFF) {
      mn = fq(mn, s_out, zp_out, p.c.out.qmin, p.c.out.qmax);
      mx = fq(mx, s_out, zp_out, p.c.out.qmin, p.c.out.qmax);
    }
  }
  if (din) {
    scale_zp(p.c.in, mn, mx, &s_in, &zp_in);
    if (writer) {
      observe_in(p.c.in, v.in, mn, mx);
      p.st[0] = s_in;
      p.st[1] = zp_in;
    }
  }
  *qout = dyn_quant<WIDE>(p.c.out, s_out, zp_out);
  if (p.first) qout->on = qout->fast = 0;
  *qin = dyn_quant<WIDE>(p.c.in, s_in, zp_in);
  // q_in repeats q_out: the levels it sees are its own (same_quant, gs_host.h)
  if (qout->fast && qin->fast && s_in == s_out && p.c.in.qmin == p.c.out.qmin && p.c.in.qmax == p.c.out.qmax)
    qin->on = qin->fast = 0;
}

// (min, max) over the workgroup into *dst; red holds two floats per wave.
template <int NW>
__device__ __forceinline__ void wg_minmax(float mn, float mx, float2* red, float2* dst) {
  wave_minmax(mn, mx);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = float2{mn, mx};
  lds_barrier();  // (not the stores of the step: their acknowledgements would be waited for)
  if (threadIdx.x == 0) {
    for (int w = 1; w < NW; ++w) {
      mn = __builtin_fminf(mn, red[w].x);
      mx = __builtin_fmaxf(mx, red[w].y);
    }
    *dst = float2{mn, mx};
  }
}

// A workgroup of 8 waves owns 16 RT batch rows x 16 units (three gates); wave q
// runs K split q of the product (gemm.hip's NT kernel with K split in up to 8:
// 16x16x4 MFMAs over 32-k slices in its k order, the splits added in order, so
// gh is that GEMM's bit for bit) from an LDS staging of its own, without a
// barrier, NS slices in flight, quantizing the state's rows as it stages them; the
// splits meet in LDS once. Bound: one launch of about 3.3 us, two dependent trips
// to memory (partials, then operands to use) and the product. us a step at B = 32,
// H = 512: GEMM 7.0, gates 3.8 and quantizers 3.8 as three launches, 13.8 together
// -> 8.0; B = 256, H = 512 23.0 -> 11.2; B = 32, H = 1024 18.7 -> 11.2; H = 64 12.7 -> 5.9.
constexpr int kObsRS = 40;  // LDS row stride of a 32-k slice (gemm.hip)

template <int RT, bool RAG, int NS>
__global__ __launch_bounds__(512) void observe_step_kernel(OStep p) {
  extern __shared__ __attribute__((aligned(16))) float olds[];
  __shared__ float2 red2[8];
  constexpr int NR = 16 * RT + 48;  // staged rows: the state's, then 16 units of each gate
  constexpr int NL = NR / 8;        // 16-byte loads a lane and slice (8 lanes a row)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = p.H;
  const int u0 = 16 * blockIdx.x, row0 = 16 * RT * blockIdx.y;
  float* mine = olds + wave * NR * kObsRS;
  StepIn in = load_step_in(p);
  __builtin_amdgcn_sched_barrier(0);

  const int kper = ((H + p.nsplit - 1) / p.nsplit + 31) / 32 * 32;
  const int kbeg = wave * kper, kend = wave < p.nsplit ? min(H, kbeg + kper) : 0;
  const int r8 = lane >> 3, k4 = 4 * (lane & 7);
  const float* src[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int r = 8 * i + r8;
    src[i] = i < 2 * RT ? p.hprev + (int64_t)min(row0 + r, p.B - 1) * p.sh_b
                        : p.w + ((int64_t)((r - 16 * RT) >> 4) * H + min(u0 + (r & 15), H - 1)) * H;
  }
  // elements k .. k + 3 of each row; what lies past the end is zeroed at staging
  // (RAG: the lane across a row's end loads its last four)
  f4 x[NS][NL];  // slices in flight
  auto load = [&](int k0, f4 (&v)[NL]) __attribute__((always_inline)) {
    const int k = k0 + k4;
    if (RAG && H < 4) {
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = src[i][k + e < H ? k + e : 0];
      return;
    }
    const int kk = RAG ? min(k, H - 4) : k < H ? k : 0;
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int i = 0; i < NL; ++i) v[i] = *reinterpret_cast<const f4u*>(src[i] + kk);
  };
  static_for<0, NS>([&](auto I) { load(kbeg + 32 * I, x[I]); });

  // the epilogue's element: row 16 (wave / 4) + 4 (lane / 16) + wave % 4, unit lane % 16
  const int er = row0 + 16 * (wave >> 2) + 4 * (lane >> 4) + (wave & 3), eu = u0 + (lane & 15);
  const bool mineq = wave < 4 * RT;
  const bool live = mineq && er < p.B && eu < H;
  const int64_t erc = min(er, p.B - 1);
  const int euc = min(eu, H - 1);
  float gin[3], bb[3];
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    gin[g] = p.gi[erc * p.sg_b + g * H + euc];
    bb[g] = p.bh[g * H + euc];
  }
  const float hraw = p.hprev[erc * p.sh_b + euc];

  DynQuant qout, qin;
  step_scales<false>(p, in, &qout, &qin);

  // one division-free quantizer for the state (the common case): applied as the rows are staged
  const bool one_quant = (qout.fast && !qin.on) || (qin.fast && !qout.on);
  const Quant q1 = qout.on ? qout.q : qin.q;

  f4 acc[RT][3];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int g = 0; g < 3; ++g) acc[i][g] = f4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, kq = lane >> 4;
  auto slice = [&](int k0, f4 (&v)[NL]) __attribute__((always_inline)) {
    const int k = k0 + k4;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      f4 y = v[i];
      if (RAG && k0 + 32 > H && H >= 4) {  // (uniform)
        const int s = k - (H - 4);  // 1 .. 3: the lane across the end, its last four loaded
        if (s == 1) y = f4{y[1], y[2], y[3], 0.f};
        if (s == 2) y = f4{y[2], y[3], 0.f, 0.f};
        if (s == 3) y = f4{y[3], 0.f, 0.f, 0.f};
      }
      if (i < 2 * RT && one_quant) {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = quant_level(y[e], q1) * q1.scale;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = k + (RAG ? e : 0) < kend ? y[e] : 0.0f;
      *reinterpret_cast<f4*>(mine + (8 * i + r8) * kObsRS + k4) = y;
    }
    if (!one_quant) {  // affine, off or different quantizers: in place, a loop to keep the code short
#pragma unroll 1
      for (int i = 0; i < 8 * RT; ++i) {
        float* h = mine + (8 * (i >> 2) + r8) * kObsRS + k4 + (i & 3);
        *h = k + (RAG ? i & 3 : 0) < kend ? qin(qout(*h)) : 0.0f;
      }
    }
    // (a wave's LDS accesses complete in order: no barrier within the wave's own staging)
    f4 a[RT][2], b[3][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
        a[i][h] = *reinterpret_cast<const f4*>(mine + (16 * i + r16) * kObsRS + 4 * kq + 16 * h);
#pragma unroll
      for (int g = 0; g < 3; ++g)
        b[g][h] = *reinterpret_cast<const f4*>(mine + (16 * (RT + g) + r16) * kObsRS + 4 * kq + 16 * h);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int g = 0; g < 3; ++g)
          acc[i][g] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s >> 2][s & 3], b[g][s >> 2][s & 3], acc[i][g], 0, 0, 0);
  };
  for (int k0 = kbeg; k0 < kend; k0 += 32 * NS) {
    const bool more = k0 + 32 * NS < kend;
    static_for<0, NS>([&](auto I) {
      if (I < 2 || k0 + 32 * I < kend) slice(k0 + 32 * I, x[I]);  // (a slice past kend adds zeros)
      if (more) load(k0 + 32 * (NS + I), x[I]);
    });
  }

  float* red = mine;  // [RT * 3][v][lane] in the wave's own staging
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int g = 0; g < 3; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((i * 3 + g) * 4 + v) * 64 + lane] = acc[i][g][v];
  lds_barrier();
  float mn = __builtin_inff(), mx = -__builtin_inff();
  if (mineq) {
    float g3[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const float* q = olds + (((wave >> 2) * 3 + g) * 4 + (wave & 3)) * 64 + lane;
      float sum = q[0] + bb[g];
#pragma unroll
      for (int w = 1; w < kMaxSplit; ++w)
        if (w < p.nsplit) sum += q[w * NR * kObsRS];
      g3[g] = sum;
    }
    if (live) {
      const float h = qout(hraw);
      if (p.out_prev != nullptr) p.out_prev[er * p.so_b + eu] = h;
      const float v = gru_update(gin[0], gin[1], gin[2], g3[0], g3[1], g3[2], h);
      p.hnext[er * p.sn_b + eu] = v;
      mn = mx = v;
      if (!(v == v)) {  // a NaN takes no part, as in the other reductions
        mn = __builtin_inff();
        mx = -__builtin_inff();
      }
    }
  }
  wg_minmax<8>(mn, mx, red2, p.part_out + (int64_t)blockIdx.y * gridDim.x + blockIdx.x);
}

// The diagonal kind's step: every element is its own, so the pre-quant h_t goes
// to out[t] and is quantized in place a launch later. As two launches a step
// (gates 3.8 us, quantizers 3.8) it took 6.4 us at B = 32, H = 512, here 4.0.
__global__ __launch_bounds__(kRedThreads) void observe_diag_kernel(OStep p) {
  __shared__ float2 red2[kRedThreads / 64];
  StepIn in = load_step_in(p);
  DynQuant qout, qin;
  step_scales<true>(p, in, &qout, &qin);
  const int H = p.H;
  float mn = __builtin_inff(), mx = -__builtin_inff();
  const int64_t n = (int64_t)p.B * H;
  for (int64_t e = blockIdx.x * (int64_t)kRedThreads + threadIdx.x; e < n; e += (int64_t)gridDim.x * kRedThreads) {
    const int b = (int)(e / H), k = (int)(e - (int64_t)b * H);
    const float h = qout(p.hprev[(int64_t)b * p.sh_b + k]);
    if (p.out_prev != nullptr && qout.on) p.out_prev[(int64_t)b * p.so_b + k] = h;
    const float hq = qin(h);
    float g3[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
#pragma clang fp contract(off)
      g3[g] = p.w[g * H + k] * hq + p.bh[g * H + k];
    }
    const float* gr = p.gi + (int64_t)b * p.sg_b + k;
    const float v = gru_update(gr[0], gr[H], gr[2 * H], g3[0], g3[1], g3[2], h);
    p.hnext[(int64_t)b * p.sn_b + k] = v;
    mn = __builtin_fminf(mn, v);
    mx = __builtin_fmaxf(mx, v);
  }
  wg_minmax<kRedThreads / 64>(mn, mx, red2, p.part_out + blockIdx.x);
}

int validate_observer(const gs_observer& o, const char* name, const char* who) {
  if (o.mode < GS_OBS_OFF || o.mode > GS_OBS_MIN_MAX)
    return set_error(GS_ERR_INVALID, "%s: %s mode %d is not a GS_OBS_* value", who, name, o.mode);
  if (o.mode == GS_OBS_OFF) return GS_OK;
  if (o.qmin > o.qmax)
    return set_error(GS_ERR_INVALID, "%s: %s qmin (%d) must be <= qmax (%d)", who, name, o.qmin, o.qmax);
  if (o.symmetric && o.qmax <= 0)
    return set_error(GS_ERR_INVALID, "%s: symmetric %s needs qmax > 0; got %d", who, name, o.qmax);
  if (!o.symmetric && o.qmax == o.qmin)
    return set_error(GS_ERR_INVALID, "%s: affine %s needs qmax > qmin", who, name);
  if (o.mode == GS_OBS_FROZEN && !(std::isfinite(o.scale) && o.scale > 0.0f && std::isfinite(o.zero_point)))
    return set_error(GS_ERR_INVALID, "%s: frozen %s needs a finite scale > 0 and a finite zero point", who, name);
  if (o.mode == GS_OBS_MIN_MAX && o.stats == nullptr)
    return set_error(GS_ERR_INVALID, "%s: %s in min_max mode needs its stats buffer", who, name);
  return GS_OK;
}

int check_plain_scratch(void* p, int64_t have, int64_t need, const char* who) {
  if (need <= 0) return GS_OK;
  if (p == nullptr || have < need)
    return set_error(GS_ERR_INVALID, "%s: scratch of %lld bytes required; got %lld", who, (long long)need,
                     (long long)have);
  if ((reinterpret_cast<uintptr_t>(p) & 255u) != 0)
    return set_error(GS_ERR_INVALID, "%s: scratch must be 256-byte aligned", who);
  return GS_OK;
}

unsigned parts_for(int64_t n) { return (unsigned)std::min<int64_t>((n + kRedThreads - 1) / kRedThreads, kMaxParts); }

dim3 grid1d(int64_t n) { return dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)); }

// Scratch of gs_observe_scan, each region 256-byte aligned:
// scales [4] | partials of two steps | pre-quant h of two steps [2][B, H] (not
// the diagonal kind), or with three launches a step hq [B, H] and gh [split][B, 3H] |
// map [3H, H] (Monarch, butterfly, circulant) | map construction scratch.
struct OPlan {
  bool gemm, own_map;
  bool three;   // three launches a step
  int split;
  int rt;       // 16-row tiles a workgroup (1 or 2)
  int64_t nwg;  // workgroups, and partials, of a step
  int64_t st, part, hpre, gh, map, map_tmp;
  int64_t total() const { return st + 2 * part + (three ? 1 : 2) * hpre + gh + map + map_tmp; }
};

// Whether a step of the kinds with a product is one launch. Up to a workgroup per
// CU always; a further round costs as much again (an 8-wave workgroup holds a CU's
// LDS), which pays while the eight waves share K without a rest and the product is
// short. us a step, three launches / one: one round 13 to 83 / 6 to 48; two rounds
// H = 64, B = 4096 18.6 / 16.5, H = 512, B = 512 31.9 / 22.9, H = 2048, B = 128 57 / 52, but
// H = 100, B = 2048 18.1 / 22.3, H = 640, B = 256 27.0 / 29.8, H = 3072, B = 64 50 / 70; three
// H = 192, B = 2048 28.6 / 26.7, H = 1024, B = 384 53.5 / 47.4, but H = 16, B = 20000 19.1 / 22.9;
// four and more H = 64, B = 20000 38 / 62, H = 127, B = 8192 37 / 83, H = 512, B = 1024 46.9 / 46.1.
bool one_launch(int64_t H, int split, int64_t nwg) {
  const int64_t rounds = (nwg + 255) / 256;
  if (rounds <= 1) return true;
  if (H % (64 * split) != 0) return false;
  return rounds == 2 ? H <= 2048 : rounds == 3 && H >= 192 && H <= 1024;
}

// Codes past kQuickCodes take three: a check in the one-launch kernel costs every
// step 0.07 us of its 7.9.
bool wide_codes(const gs_observer& o) {
  return o.mode != GS_OBS_OFF && (o.qmin < -kQuickCodes || o.qmax > kQuickCodes);
}

gs_map_args map_view(const gs_observe_args* a) {
  gs_map_args m{};
  m.kind = a->kind;
  m.w = a->w;
  m.w2 = a->w2;
  m.H = a->H;
  m.nblocks = a->nblocks;
  m.blksz = a->blksz;
  m.log_n = a->log_n;
  m.bfly_nblocks = a->bfly_nblocks;
  return m;
}

int plan_observe(const gs_observe_args* a, OPlan* p, const char* who) {
  if (a == nullptr) return set_error(GS_ERR_INVALID, "%s: args is NULL", who);
  gs_args f{};
  f.gi = a->gi;
  f.h0 = a->h0;
  f.w = a->w;
  f.bh = a->bh;
  f.out = a->out;
  f.T = a->T;
  f.B = a->B;
  f.H = a->H;
  f.sg_t = a->sg_t;
  f.sg_b = a->sg_b;
  f.sh0_b = a->sh0_b;
  f.so_t = a->so_t;
  f.so_b = a->so_b;
  int rc = validate_common(&f, who);
  if (rc) return rc;
  const gs_map_args m = map_view(a);
  rc = validate_map(&m, who);
  if (rc) return rc;
  rc = validate_observer(a->q_in, "h_in observer", who);
  if (rc) return rc;
  rc = validate_observer(a->q_out, "h_out observer", who);
  if (rc) return rc;
  const int64_t B = a->B, H = a->H;
  if (B * 3 * H > INT32_MAX / 4)
    return set_error(GS_ERR_INVALID, "%s: B * 3H = %lld is too large", who, (long long)(B * 3 * H));
  p->gemm = a->kind != GS_KIND_DIAGONAL;
  p->own_map = a->kind == GS_KIND_MONARCH || a->kind == GS_KIND_BUTTERFLY || a->kind == GS_KIND_CIRCULANT;
  // gh has only B rows: split K in up to 8 parts of >= 64 terms
  p->split = p->gemm ? (int)std::max<int64_t>(1, std::min<int64_t>(kMaxSplit, H / 64)) : 1;
  // 32 rows a workgroup (Wh read half as often) once 16 give every CU one
  const int64_t nut = (H + 15) / 16;
  p->rt = ((B + 15) / 16) * nut > 256 ? 2 : 1;
  p->nwg = p->gemm ? ((B + 16 * p->rt - 1) / (16 * p->rt)) * nut : parts_for(B * H);
  p->three = p->gemm && (wide_codes(a->q_in) || wide_codes(a->q_out) || !one_launch(H, p->split, p->nwg));
  if (p->three) p->nwg = parts_for(B * H);
  p->st = 256;
  p->part = align256(std::max<int64_t>(p->nwg, kMaxParts) * 8);
  p->hpre = p->gemm ? align256(B * H * 4) : 0;
  p->gh = p->three ? align256((int64_t)p->split * B * 3 * H * 4) : 0;
  p->map = p->own_map ? align256(3 * H * H * 4) : 0;
  p->map_tmp = p->own_map ? hidden_map_scratch(&m) : 0;
  return GS_OK;
}

// The steps as three launches each: gh by the K-split GEMM from hq = q_in(h_{t-1}),
// the gates (pre-quant h_t into out[t]), and a quantizer pass that finishes out[t]
// and writes the next step's hq. part: kMaxParts partials; those of h0 are in it.
int three_launches(const gs_observe_args* a, const OPlan& p, const ObsPair& c, const float* W, float* st, float2* part,
                   float* hq, float* gh, hipStream_t stream, const char* who) {
  const int T = (int)a->T, B = (int)a->B, H = (int)a->H;
  const int64_t BH = (int64_t)B * H;
  const bool in_on = c.in.mode != GS_OBS_OFF, out_on = c.out.mode != GS_OBS_OFF;
  const int np = is_dynamic(c.in) || is_dynamic(c.out) ? (int)p.nwg : 0;
  if (in_on) {
    hipLaunchKernelGGL(quant_step, grid1d(BH), dim3(kRedThreads), 0, stream, part, is_dynamic(c.in) ? (int)p.nwg : 0,
                       c, st, a->trace, 0, T, 0, a->h0, a->sh0_b, nullptr, (int64_t)0, hq, (int64_t)B, H, 0);
    GS_CHECK_HIP(hipGetLastError());
  }
  for (int t = 0; t < T; ++t) {
    const float* hprev = t == 0 ? a->h0 : a->out + (int64_t)(t - 1) * a->so_t;
    const int64_t shp = t == 0 ? a->sh0_b : a->so_b;
    float* out_t = a->out + (int64_t)t * a->so_t;
    GemmArgs g;
    g.a = in_on ? hq : hprev;  // the matmul-side h
    g.lda = in_on ? H : shp;
    g.b = W;  // B(k, n) = W[n][k]
    g.ldb = H;
    g.c = gh;
    g.ldc = 3 * H;
    g.split_stride = 3 * BH;
    g.bias = a->bh;
    g.M = B;
    g.N = 3 * H;
    g.K = H;
    g.ksplit = p.split;
    g.layout = kGemmNT;
    const int rc = gemm_f32(g, stream, who);
    if (rc) return rc;
    hipLaunchKernelGGL(gates_step, dim3((unsigned)p.nwg), dim3(kRedThreads), 0, stream,
                       a->gi + (int64_t)t * a->sg_t, a->sg_b, gh, p.split, 3 * BH, hprev, shp, out_t, a->so_b, B, H,
                       part);
    GS_CHECK_HIP(hipGetLastError());
    // every step: it also writes the trace
    hipLaunchKernelGGL(quant_step, grid1d(BH), dim3(kRedThreads), 0, stream, part, np, c, st, a->trace, t, T, 1, out_t,
                       a->so_b, out_on ? out_t : nullptr, a->so_b, in_on && t + 1 < T ? hq : nullptr, (int64_t)B, H,
                       out_on ? 1 : 0);
    GS_CHECK_HIP(hipGetLastError());
  }
  return GS_OK;
}

int64_t tensor_scratch(const gs_observe_tensor_args*) { return 256 + align256((int64_t)kMaxParts * 8); }

}  // namespace
}  // namespace gs

extern "C" int64_t gs_observe_scan_scratch_bytes(const gs_observe_args* a) {
  using namespace gs;
  OPlan p;
  const int rc = plan_observe(a, &p, "gs_observe_scan_scratch_bytes");
  if (rc) return rc;
  return p.total();
}

extern "C" int gs_observe_scan(const gs_observe_args* a, hipStream_t stream) {
  using namespace gs;
  clear_error();
  const char* who = "gs_observe_scan";
  OPlan p;
  int rc = plan_observe(a, &p, who);
  if (rc) return rc;
  rc = check_plain_scratch(a->scratch, a->scratch_bytes, p.total(), who);
  if (rc) return rc;
  char* cur = static_cast<char*>(a->scratch);
  auto take = [&](int64_t bytes) {
    char* r = cur;
    cur += bytes;
    return r;
  };
  float* st = reinterpret_cast<float*>(take(p.st));
  float2* part[2];
  for (float2*& q : part) q = reinterpret_cast<float2*>(take(p.part));
  float* hpre[2] = {};
  for (int i = 0; i < (p.three ? 1 : 2); ++i) hpre[i] = reinterpret_cast<float*>(take(p.hpre));
  float* gh = reinterpret_cast<float*>(take(p.gh));
  float* map = reinterpret_cast<float*>(take(p.map));
  void* map_tmp = take(p.map_tmp);

  const int T = (int)a->T, B = (int)a->B, H = (int)a->H;
  const ObsPair c{to_obs(a->q_in), to_obs(a->q_out)};
  const bool out_on = a->q_out.mode != GS_OBS_OFF;
  const int64_t BH = (int64_t)B * H;

  const float* W = a->w;
  if (p.own_map) {
    gs_map_args m = map_view(a);
    m.m = map;
    m.scratch = map_tmp;
    m.scratch_bytes = p.map_tmp;
    rc = materialize_map(&m, stream, who);
    if (rc) return rc;
    W = map;
  }
  const bool any_dyn = is_dynamic(c.in) || is_dynamic(c.out);
  int np = 0;
  if (is_dynamic(c.in)) {
    np = (int)parts_for(BH);
    hipLaunchKernelGGL(minmax_partials, dim3((unsigned)np), dim3(kRedThreads), 0, stream, a->h0, (int64_t)B, H,
                       a->sh0_b, part[1]);
    GS_CHECK_HIP(hipGetLastError());
  }

  if (p.three) return three_launches(a, p, c, W, st, part[1], hpre[0], gh, stream, who);

  const unsigned nut = (unsigned)((H + 15) / 16);
  const dim3 grid = p.gemm ? dim3(nut, (unsigned)(p.nwg / nut)) : dim3((unsigned)p.nwg);
  const bool rag = H % 4 != 0;
  void (*fn)(OStep) = !p.gemm ? observe_diag_kernel
                      : p.rt == 2 ? (rag ? observe_step_kernel<2, true, 2> : observe_step_kernel<2, false, 2>)
                      : H > 64 * p.split ? (rag ? observe_step_kernel<1, true, 4> : observe_step_kernel<1, false, 4>)
                                         : (rag ? observe_step_kernel<1, true, 2> : observe_step_kernel<1, false, 2>);
  const int lds = p.gemm ? 8 * (16 * p.rt + 48) * kObsRS * 4 : 0;
  if (lds > 65536) GS_CHECK_HIP(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  OStep s;
  s.w = W;
  s.bh = a->bh;
  s.st = st;
  s.c = c;
  s.sg_b = a->sg_b;
  s.so_b = a->so_b;
  s.B = B;
  s.H = H;
  s.nsplit = p.split;
  for (int t = 0; t < T; ++t) {
    s.gi = a->gi + (int64_t)t * a->sg_t;
    float* out_t = a->out + (int64_t)t * a->so_t;
    s.out_prev = t == 0 ? nullptr : out_t - a->so_t;
    s.hprev = t == 0 ? a->h0 : p.gemm ? hpre[(t - 1) & 1] : s.out_prev;
    s.sh_b = t == 0 ? a->sh0_b : p.gemm ? H : a->so_b;
    s.hnext = p.gemm ? hpre[t & 1] : out_t;
    s.sn_b = p.gemm ? H : a->so_b;
    s.part_in = part[(t + 1) & 1];
    s.part_out = part[t & 1];
    s.trace = t > 0 && a->trace != nullptr ? a->trace + (int64_t)(t - 1) * 4 : nullptr;
    s.first = t == 0;
    s.np = np;
    hipLaunchKernelGGL(fn, grid, dim3(p.gemm ? 512 : kRedThreads), (size_t)lds, stream, s);
    GS_CHECK_HIP(hipGetLastError());
    np = any_dyn ? (int)p.nwg : 0;
  }
  // out[T-1] and the last trace entry
  float* out_t = a->out + (int64_t)(T - 1) * a->so_t;
  const float* x = p.gemm ? hpre[(T - 1) & 1] : out_t;
  hipLaunchKernelGGL(quant_step, grid1d(BH), dim3(kRedThreads), 0, stream, part[(T - 1) & 1], np, c, st, a->trace,
                     T - 1, T, 1, x, p.gemm ? (int64_t)H : a->so_b, p.gemm || out_on ? out_t : nullptr, a->so_b,
                     nullptr, (int64_t)B, H, out_on ? 1 : 0);
  GS_CHECK_HIP(hipGetLastError());
  return GS_OK;
}

extern "C" int64_t gs_observe_tensor_scratch_bytes(const gs_observe_tensor_args* a) {
  if (a == nullptr) return gs::set_error(GS_ERR_INVALID, "gs_observe_tensor_scratch_bytes: args is NULL");
  return gs::tensor_scratch(a);
}

extern "C" int gs_observe_tensor(const gs_observe_tensor_args* a, hipStream_t stream) {
  using namespace gs;
  clear_error();
  const char* who = "gs_observe_tensor";
  if (a == nullptr) return set_error(GS_ERR_INVALID, "%s: args is NULL", who);
  if (a->rows < 1 || a->cols < 1 || a->cols > INT32_MAX || a->rows > (int64_t(1) << 40))
    return set_error(GS_ERR_INVALID, "%s: rows and cols must be > 0; got %lld, %lld", who, (long long)a->rows,
                     (long long)a->cols);
  if (a->rows > 1 && a->ld < a->cols)
    return set_error(GS_ERR_INVALID, "%s: row stride ld=%lld < cols=%lld", who, (long long)a->ld, (long long)a->cols);
  if (!a->x || !a->y) return set_error(GS_ERR_INVALID, "%s: x and y must be non-NULL device pointers", who);
  int rc = validate_observer(a->q, "observer", who);
  if (rc) return rc;
  rc = check_plain_scratch(a->scratch, a->scratch_bytes, tensor_scratch(a), who);
  if (rc) return rc;
  float* st = static_cast<float*>(a->scratch);
  float2* part = reinterpret_cast<float2*>(static_cast<char*>(a->scratch) + 256);
  // The tensor's quantizer takes the "in" slot of the scale words.
  const ObsPair c{to_obs(a->q), Obs{GS_OBS_OFF, 1, 0.f, 0.f, 1.f, 0.f, nullptr}};
  const int64_t n = a->rows * a->cols;
  const unsigned np = parts_for(n);
  if (is_dynamic(c.in)) {
    hipLaunchKernelGGL(minmax_partials, dim3(np), dim3(kRedThreads), 0, stream, a->x, a->rows, (int)a->cols, a->ld,
                       part);
    GS_CHECK_HIP(hipGetLastError());
  }
  // identity (observer off): y = x through the dst path; otherwise y = q(x)
  const bool off = c.in.mode == GS_OBS_OFF;
  hipLaunchKernelGGL(quant_step, grid1d(n), dim3(kRedThreads), 0, stream, part, is_dynamic(c.in) ? (int)np : 0, c, st,
                     nullptr, 0, 1, 0, a->x, a->ld, off ? a->y : nullptr, a->cols, off ? nullptr : a->y, a->rows,
                     (int)a->cols, 0);
  GS_CHECK_HIP(hipGetLastError());
  if (a->used != nullptr) GS_CHECK_HIP(hipMemcpyAsync(a->used, st, 2 * sizeof(float), hipMemcpyDeviceToDevice, stream));
  return GS_OK;
}
