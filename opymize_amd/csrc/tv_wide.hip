// K fused TV iterations per pass over HBM for one-channel FP32 images, streamed
// down column strips with two columns per lane; see tv_common.h for the model
// and tv_stream.hip for the pipeline.
#include "tv_common.h"

namespace opy {
namespace {

// Work unit: one wavefront per (strip, chunk) of an instance, as in
// tv_stream_kernel; the chunks of an instance share its rows evenly.  The wavefront walks down R + 2K rows, loads each row of x,
// f and y once and runs the K iterations as a pipeline skewed by one row per
// level.  Lane l holds the columns 2l and 2l + 1 of a strip of 128 columns, of
// which 128 - 2K are exact.
//
// With 8 iterations per launch the one-column kernel is bound by VALU issue:
// 213 instructions per row of 64 columns, of which 48 are exact.  Here:
// - 112 of 128 columns are exact: 1024 columns take 9 strips of 128 instead of
//   21 of 64, 14% fewer lanes.
// - One neighbour of either column is in the lane itself; only every second
//   horizontal difference goes through a DPP shift, folded into its subtraction.
// - The unmasked steps run in pairs, so that the state that moves from step to
//   step (x, x_bar, and y of the row above, per level) alternates between two
//   sets of registers instead of being copied: 320 instructions per row of 128
//   columns, 13 of them copies.
// - The two columns' chains alternate instruction by instruction (a dependent
//   instruction has to wait, an independent one does not), so two wavefronts per
//   SIMD keep it issuing and the state of 8 levels fits without spilling: 191
//   registers, where three wavefronts (168, with spills in the edge strips'
//   loops) took 313 us per launch on 32 images of 1024^2 against 251.
// - min(1, s) of the projection is the clamp modifier of the product that forms
//   s (s >= 0; a NaN gives 0 instead of 1, and NaN results either way).
// - The step coefficients of the launch's iterations come from a table
//   (tv_steps_kernel) through scalar loads; no wavefront advances the FP64
//   schedule itself.
// - A block is one wavefront: the units of the strips at the image edges, with
//   their masks, take longer than the others, and a block of four held its slots
//   until the last had ended (313 against 251 us).
// 8 iterations on 32 / 128 images of 1024^2: 350 -> 251 us / 1200 -> 1027 us
// (3.8 / 3.7 TB/s of 28 B per pixel, clock 1.9 GHz under this load); 4
// iterations, where HBM bounds both, 216 -> 206 us on 32.
// A row's loads go out a whole step before they are used: the step starts by
// waiting for its row (an empty asm statement takes the registers, so that the
// wait stands before anything is issued), then stores the previous step's
// result, then loads the next row.  The wait therefore never covers a store or
// load of its own step.  Rows and columns beyond the image load the nearest
// ones inside; the masks keep their values out of every exact one.
//
// The arithmetic per pixel, and the rounding of every product and sum, is that
// of primal_px / overrelax / dual_px, so the iterates equal those of
// tv_stream_kernel, tv_multi_kernel and K single launches bit for bit.

// one iteration's coefficients (FoldedStep<float, 1> and 1 + theta)
struct alignas(32) WideStep {
  float a, b, theta, theta1;
  float p0, p1, q0, q1;
};

constexpr int kWideCols = 128;

__host__ __device__ inline int wide_strips_ext(int W, int sw) {
  return W <= kWideCols ? 1 : (W - kWideCols + sw - 1) / sw + 1;
}
// the strips at the image edges need no halo beyond it (tv_stream.hip)
__host__ __device__ inline int wide_strips(int W, int sw) {
  return min((W + sw - 1) / sw, wide_strips_ext(W, sw));
}

// iteration i (< n) of every running instance's step schedule: its coefficients
// to tab[b * n + i], and the instance's state n iterations on (the FP64
// operations of tv_accel_kernel and fold_step).  One wavefront per instance: the
// schedule is a serial chain of square roots and divisions, the coefficients
// that hang off it are formed by one lane per iteration.
__global__ void __launch_bounds__(64) tv_steps_kernel(const opy_tv_inst_t* __restrict__ insts,
                                                      opy_adapt_state_t* __restrict__ st,
                                                      const opy_tv_check_t* __restrict__ chk, Cfg cfg, int n,
                                                      WideStep* __restrict__ tab) {
  const int b = blockIdx.x;
  if (chk[b].status != 0) return;
  const opy_tv_inst_t I = insts[b];
  double tau = st[b].tau, sigma = st[b].sigma;
  for (int i0 = 0; i0 < n; i0 += 64) {
    // every lane walks the chain and keeps its own iteration's values
    double mt = 0.0, ms = 0.0, mth = 1.0;
    const int m = min(64, n - i0);
    for (int i = 0; i < m; ++i) {
      const double th = accel_theta(cfg.steps, I, tau);
      const double so = sigma / th;
      if ((int)threadIdx.x == i) {
        mt = tau;
        ms = so;
        mth = th;
      }
      tau *= th;
      sigma = so;
    }
    if ((int)threadIdx.x < m) {
      const FoldedStep<float, 1> s = fold_step<float, 1>(mt, ms, mth, I, cfg);
      tab[(int64_t)b * n + i0 + threadIdx.x] = {s.a,       s.b,       s.theta,   1.0f + s.theta,
                                                s.p[0][0], s.p[1][0], s.q[0][0], s.q[1][0]};
    }
  }
  if (cfg.steps == OPY_TV_STEPS_ACCEL && threadIdx.x == 0) {
    st[b].tau = tau;
    st[b].sigma = sigma;
  }
}

// two or four FP32 values at an address that is only known to be element aligned
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

template <typename T>
__device__ inline T* at_byte(T* p, uint32_t bytes) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(p) + (size_t)bytes);
}
template <typename T>
__device__ inline const T* at_byte(const T* p, uint32_t bytes) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + (size_t)bytes);
}

template <int K>
__global__ void __launch_bounds__(64, K >= 7 ? 2 : (K >= 5 ? 3 : 4)) tv_wide_kernel(const float* __restrict__ xin, float* __restrict__ xout,
                                                      const float* __restrict__ yin, float* __restrict__ yout,
                                                      const float* __restrict__ f,
                                                      const opy_tv_inst_t* __restrict__ insts,
                                                      const WideStep* __restrict__ tab, int tab_n, int it0,
                                                      const int32_t* __restrict__ active_inst,
                                                      const int32_t* __restrict__ unit_off,
                                                      const int32_t* __restrict__ nact_p, int rows) {
  constexpr int SW = kWideCols - 2 * K;
  const int nact = *nact_p;
  if (nact <= 0) return;
  const int total = unit_off[nact];
  const int lane = threadIdx.x;
  for (int u = xcd_block(); u < total; u += gridDim.x) {
    const TileRef tr = locate(u, active_inst, unit_off, nact, insts, SW, rows);
    const opy_tv_inst_t I = insts[tr.b];
    const int H = I.H, W = I.W;
    const int nc = (H + rows - 1) / rows, R = (H + nc - 1) / nc;  // chunks, and their rows (at most `rows`)
    const int NSTEP = R + 2 * K;
    const int ns = wide_strips(W, SW), ty = tr.j / ns;
    const bool ext = ns < (W + SW - 1) / SW;
    const int r0 = ty * R - K;  // image row of pipeline row 0
    const int c0 = (tr.j - ty * ns) * SW - (ext ? 0 : K);
    // exact columns of the strip, stored: [slo, shi)
    const int slo = (ext && c0 == 0) ? 0 : K, shi = (ext && c0 + kWideCols >= W) ? kWideCols : kWideCols - K;
    const int c = c0 + 2 * lane;
    const bool cedge = !(c0 >= 1 && c0 + kWideCols < W);  // the strip's columns reach an image edge
    WideStep fs[K];
#pragma unroll
    for (int i = 0; i < K; ++i) fs[i] = tab[(int64_t)tr.b * tab_n + it0 + i];
    const float tvw = (float)I.tvw;
    const float* xb = xin + I.off;
    const float* fb = f + I.off;
    const float* yb = yin + 2 * I.off;
    float* xob = xout + I.off;
    float* yob = yout + 2 * I.off;
    // L1: data kind; MC: column masks, per-column accesses (uniform over the unit)
    auto run = [&](auto l1_tag, auto mc_tag) {
      constexpr bool L1 = decltype(l1_tag)::value, MC = decltype(mc_tag)::value;
      // per level: x^(i+1) and x_bar^(i+1) of its last row, y^i of the row above its current one, f
      // delayed by i rows
      float Xo[K][2], XB[K][2], YL[K][4], F[K][2];
#pragma unroll
      for (int i = 0; i < K; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) Xo[i][j] = XB[i][j] = F[i][j] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) YL[i][e] = 0.f;
      }
      float nx[2], nf[2], ny[4];  // the next row (y: the pairs of the two columns)
      float rx_[2], ry_[4];       // the last step's result, not stored yet
#pragma unroll
      for (int j = 0; j < 2; ++j) rx_[j] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) ry_[e] = 0.f;
      const uint32_t ca = MC ? (uint32_t)min(max(c, 0), W - 1) : (uint32_t)c;
      const uint32_t cb = MC ? (uint32_t)min(max(c + 1, 0), W - 1) : 0u;
      auto load_row = [&](int n) {
        const int r = min(max(r0 + n, 0), H - 1);
        const float* xr = xb + (int64_t)r * W;
        const float* fr = fb + (int64_t)r * W;
        const float* yr = yb + 2 * (int64_t)r * W;
        if constexpr (MC) {
          const f32x2u y0 = *reinterpret_cast<const f32x2u*>(at_byte(yr, ca * 8u));
          const f32x2u y1 = *reinterpret_cast<const f32x2u*>(at_byte(yr, cb * 8u));
          ny[0] = y0.x;
          ny[1] = y0.y;
          ny[2] = y1.x;
          ny[3] = y1.y;
          nx[0] = *at_byte(xr, ca * 4u);
          nx[1] = *at_byte(xr, cb * 4u);
          nf[0] = *at_byte(fr, ca * 4u);
          nf[1] = *at_byte(fr, cb * 4u);
        } else {
          const f32x4u y = *reinterpret_cast<const f32x4u*>(at_byte(yr, ca * 8u));
          const f32x2u x = *reinterpret_cast<const f32x2u*>(at_byte(xr, ca * 4u));
          const f32x2u fv = *reinterpret_cast<const f32x2u*>(at_byte(fr, ca * 4u));
          ny[0] = y.x;
          ny[1] = y.y;
          ny[2] = y.z;
          ny[3] = y.w;
          nx[0] = x.x;
          nx[1] = x.y;
          nf[0] = fv.x;
          nf[1] = fv.y;
        }
      };
      const bool s0 = 2 * lane >= slo && 2 * lane < shi && (!MC || c < W);
      const bool s1 = 2 * lane + 1 >= slo && 2 * lane + 1 < shi && (!MC || c + 1 < W);
      auto store_row = [&](int r) {  // the exact columns of image row r
        float* xr = xob + (int64_t)r * W;
        float* yr = yob + 2 * (int64_t)r * W;
        if (!MC && K % 2 == 0) {  // s0 == s1
          if (s0) {
            *reinterpret_cast<f32x2u*>(at_byte(xr, (uint32_t)c * 4u)) = f32x2u{rx_[0], rx_[1]};
            *reinterpret_cast<f32x4u*>(at_byte(yr, (uint32_t)c * 8u)) = f32x4u{ry_[0], ry_[1], ry_[2], ry_[3]};
          }
        } else {
          if (s0) {
            *at_byte(xr, (uint32_t)c * 4u) = rx_[0];
            *reinterpret_cast<f32x2u*>(at_byte(yr, (uint32_t)c * 8u)) = f32x2u{ry_[0], ry_[1]};
          }
          if (s1) {
            *at_byte(xr, (uint32_t)(c + 1) * 4u) = rx_[1];
            *reinterpret_cast<f32x2u*>(at_byte(yr, (uint32_t)(c + 1) * 8u)) = f32x2u{ry_[2], ry_[3]};
          }
        }
      };
      // one pipeline step; MR: row masks; ST: the store of the last step's result (0 none, 1 stored,
      // 2 stored where it is a row of the chunk)
      auto step = [&](auto mr_tag, auto st_tag, int n) {
        constexpr bool MR = decltype(mr_tag)::value;
        constexpr int ST = decltype(st_tag)::value;
        asm volatile("" : "+v"(nx[0]), "+v"(nx[1]), "+v"(nf[0]), "+v"(nf[1]), "+v"(ny[0]), "+v"(ny[1]), "+v"(ny[2]),
                     "+v"(ny[3]));
        float xcur[2], ycur[4];
#pragma unroll
        for (int i = K - 1; i > 0; --i)
#pragma unroll
          for (int j = 0; j < 2; ++j) F[i][j] = F[i - 1][j];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          xcur[j] = nx[j];
          F[0][j] = nf[j];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) ycur[e] = ny[e];
        {
          const int m = n - 1 - K, r = r0 + m;  // pipeline and image row of the pending result
          if (ST == 1 || (ST == 2 && m >= K && r < H)) store_row(r);
        }
        load_row(n + 1);
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the step
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int rx = r0 + n - i, ry = rx - 1;  // rows of x^(i+1) and y^(i+1) of this step
          const WideStep& s = fs[i];
          // operation by operation for the lane's two columns: their chains are independent, and a result
          // takes twice as long as an instruction
#define OPY_J _Pragma("unroll") for (int j = 0; j < 2; ++j)
          float y0[2], y1[2], yu[2], y1l[2], v[2], xnew[2], xbar[2], xbr[2], gd[2], gr[2], w0[2], w1[2], n2[2], yp[4];
          y1l[0] = dpp_shr1(0.f, ycur[3]);  // y1 of the columns to the left
          xbr[1] = dpp_shl1(0.f, XB[i][0]);  // x_bar of the columns to the right
          y1l[1] = ycur[1];
          xbr[0] = XB[i][1];
          OPY_J {
            y0[j] = ycur[2 * j];
            y1[j] = ycur[2 * j + 1];
            yu[j] = YL[i][2 * j];
          }
          if (MR) OPY_J {
            if (!(rx < H - 1)) y0[j] = 0.f;
            if (!(rx > 0)) yu[j] = 0.f;
          }
          if (MC) OPY_J {
            if (!(c + j < W - 1)) y1[j] = 0.f;
            if (!(c + j > 0)) y1l[j] = 0.f;
          }
          OPY_J v[j] = y0[j] - yu[j];
          OPY_J y1[j] = y1[j] - y1l[j];
          OPY_J v[j] = __builtin_fmaf(v[j], s.p0, xcur[j]);
          OPY_J v[j] = __builtin_fmaf(y1[j], s.p1, v[j]);
          if constexpr (L1) {
            // soft_rest, the clamp as one median (a NaN stays one in the difference)
            float cl[2];
            OPY_J v[j] = v[j] - F[i][j];
            OPY_J cl[j] = __builtin_amdgcn_fmed3f(v[j], -s.b, s.b);
            OPY_J v[j] = v[j] - cl[j];
            OPY_J xnew[j] = F[i][j] + v[j];
          } else {
            OPY_J v[j] = __builtin_fmaf(s.b, F[i][j], v[j]);
            OPY_J xnew[j] = mul_rn(s.a, v[j]);
          }
          OPY_J xbar[j] = overrelax(s.theta1, s.theta, xnew[j], xcur[j]);
          OPY_J gr[j] = xbr[j] - XB[i][j];
          OPY_J gd[j] = xbar[j] - XB[i][j];
          if (MR && !(ry < H - 1)) OPY_J gd[j] = 0.f;
          if (MC) OPY_J {
            if (!(c + j < W - 1)) gr[j] = 0.f;
          }
          OPY_J w1[j] = __builtin_fmaf(gr[j], s.q1, YL[i][2 * j + 1]);
          OPY_J w0[j] = __builtin_fmaf(gd[j], s.q0, YL[i][2 * j]);
          OPY_J n2[j] = mul_rn(w1[j], w1[j]);
          OPY_J n2[j] = __builtin_fmaf(w0[j], w0[j], n2[j]);
          OPY_J n2[j] = ball_scale(tvw, n2[j]);
          OPY_J n2[j] = __builtin_amdgcn_fmed3f(n2[j], 0.f, 1.f);
          OPY_J yp[2 * j] = mul_rn(w0[j], n2[j]);
          OPY_J yp[2 * j + 1] = mul_rn(w1[j], n2[j]);
#undef OPY_J
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            YL[i][e] = ycur[e];
            ycur[e] = yp[e];
          }
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            XB[i][j] = xbar[j];
            const float xo = Xo[i][j];
            Xo[i][j] = xnew[j];
            xcur[j] = xo;
          }
        }
        // x^K and y^K at pipeline row n - K
#pragma unroll
        for (int j = 0; j < 2; ++j) rx_[j] = xcur[j];
#pragma unroll
        for (int e = 0; e < 4; ++e) ry_[e] = ycur[e];
      };
      using TT = std::true_type;
      using FF = std::false_type;
      using S0 = std::integral_constant<int, 0>;
      using S1 = std::integral_constant<int, 1>;
      using S2 = std::integral_constant<int, 2>;
      load_row(0);
      int n = 0;
      {
        // steps [nA, nB): every level's rows lie inside the image with one to spare, no row masks; the
        // result of step n - 1 is a row of the chunk from n = 2K + 1 on (and inside the image up to nB)
        const int nA = max(0, K - r0), nB = min(NSTEP, H - 1 - r0);
        const int nS = min(nB, 2 * K + 1);
#pragma unroll 1
        for (; n < min(nA, NSTEP); ++n) step(TT{}, S2{}, n);
#pragma unroll 1
        for (; n < nS; ++n) step(FF{}, S0{}, n);
        if (n == 2 * K + 1) {
#pragma unroll 1
          for (; n + 1 < nB; n += 2) {
            step(FF{}, S1{}, n);
            step(FF{}, S1{}, n + 1);
          }
        }
      }
#pragma unroll 1
      for (; n < NSTEP; ++n) step(TT{}, S2{}, n);
      if (r0 + NSTEP - 1 - K < H) store_row(r0 + NSTEP - 1 - K);
    };
    using TT = std::true_type;
    using FF = std::false_type;
    if (I.data == OPY_TV_DATA_L1) {
      if (cedge) run(TT{}, TT{});
      else run(TT{}, FF{});
    } else {
      if (cedge) run(FF{}, TT{});
      else run(FF{}, FF{});
    }
  }
}

// Units of the running instances before a (exclusive prefix) in wide_off[a], all of them in
// wide_off[nact], and the same of tv_stream_kernel's units in stream_off; one block
__global__ void __launch_bounds__(kTB) tv_wide_units_kernel(const opy_tv_inst_t* __restrict__ insts,
                                                            const int32_t* __restrict__ active_inst,
                                                            const int32_t* __restrict__ nact_p, int k,
                                                            int32_t* __restrict__ stream_off, int stream_rows,
                                                            int32_t* __restrict__ wide_off, int wide_rows) {
  __shared__ int part[2][kTB];
  const int nact = *nact_p;
  const int per = (nact + kTB - 1) / kTB;
  const int lo = threadIdx.x * per, hi = min(nact, lo + per);
  auto units = [&](int a, int& ns, int& nw) {
    const opy_tv_inst_t& I = insts[active_inst[a]];
    ns = stream_strips(I.W, 64 - 2 * k) * ((I.H + stream_rows - 1) / stream_rows);
    nw = wide_strips(I.W, kWideCols - 2 * k) * ((I.H + wide_rows - 1) / wide_rows);
  };
  int n[2] = {0, 0};
  for (int a = lo; a < hi; ++a) {
    int ns, nw;
    units(a, ns, nw);
    n[0] += ns;
    n[1] += nw;
  }
  part[0][threadIdx.x] = n[0];
  part[1][threadIdx.x] = n[1];
  __syncthreads();
  if (threadIdx.x < 2) {
    int t = 0;
    for (int i = 0; i < kTB; ++i) {
      const int v = part[threadIdx.x][i];
      part[threadIdx.x][i] = t;
      t += v;
    }
    (threadIdx.x == 0 ? stream_off : wide_off)[nact > 0 ? nact : 0] = t;
  }
  __syncthreads();
  int ts = part[0][threadIdx.x], tw = part[1][threadIdx.x];
  for (int a = lo; a < hi; ++a) {
    stream_off[a] = ts;
    wide_off[a] = tw;
    int ns, nw;
    units(a, ns, nw);
    ts += ns;
    tw += nw;
  }
}

constexpr int kWideMaxRows = 1 << 20;
constexpr int kWideMaxK = 8;

}  // namespace
}  // namespace opy

using namespace opy;

OPY_API int opy_tv_wide_units(const opy_tv_inst_t* insts, const int32_t* active_inst, const int32_t* nact, int k,
                              int32_t* stream_off, int stream_rows, int32_t* wide_off, int wide_rows, void* s) {
  if (!insts || !active_inst || !nact || !stream_off || !wide_off) return fail(kInvalid, "tv_wide_units: null pointer");
  if (k < 2 || k > kWideMaxK) return fail(kInvalid, "tv_wide_units: k = %d not in [2, %d]", k, kWideMaxK);
  if (stream_rows < 1 || stream_rows > kWideMaxRows || wide_rows < 1 || wide_rows > kWideMaxRows)
    return fail(kInvalid, "tv_wide_units: rows = %d, %d not in [1, %d]", stream_rows, wide_rows, kWideMaxRows);
  hipLaunchKernelGGL(tv_wide_units_kernel, dim3(1), dim3(kTB), 0, as_stream(s), insts, active_inst, nact, k, stream_off,
                     stream_rows, wide_off, wide_rows);
  return check_launch("tv_wide_units");
}

OPY_API int opy_tv_wide_steps(const opy_tv_inst_t* insts, opy_adapt_state_t* st, const opy_tv_check_t* chk, int B,
                              const opy_tv_cfg_t* cfg, int n, float* table, void* s) {
  if (int rc = check_cfg(cfg)) return rc;
  if (cfg->C != 1) return fail(kInvalid, "tv_wide_steps: one channel only (got C = %d)", cfg->C);
  if (cfg->steps == OPY_TV_STEPS_PRECOND) return fail(kInvalid, "tv_wide_steps: preconditioned steps vary per pixel");
  if (!insts || !st || !chk || !table || B < 1 || n < 1) return fail(kInvalid, "tv_wide_steps: bad arguments");
  if ((reinterpret_cast<uintptr_t>(table) & 31) != 0)
    return fail(kInvalid, "tv_wide_steps: the table must be 32-byte aligned");
  hipLaunchKernelGGL(tv_steps_kernel, dim3(B), dim3(64), 0, as_stream(s), insts, st, chk, make_cfg(cfg), n,
                     reinterpret_cast<WideStep*>(table));
  return check_launch("tv_wide_steps");
}

OPY_API int opy_tv_wide_f32(const float* xi, float* xo, const float* yi, float* yo, const float* f,
                            const opy_tv_inst_t* insts, const float* table, int n, int it0,
                            const int32_t* active_inst, const int32_t* unit_off, const int32_t* nact, int k, int rows,
                            int grid, void* s) {
  if (k < 2 || k > kWideMaxK) return fail(kInvalid, "tv_wide: k = %d not in [2, %d]", k, kWideMaxK);
  if (rows < 1 || rows > kWideMaxRows) return fail(kInvalid, "tv_wide: rows = %d not in [1, %d]", rows, kWideMaxRows);
  if (!xi || !xo || !yi || !yo || !f || !insts || !table || !active_inst || !unit_off || !nact || grid < 0)
    return fail(kInvalid, "tv_wide: null pointer or negative grid");
  if (n < 1 || it0 < 0 || it0 + k > n) return fail(kInvalid, "tv_wide: iterations %d..%d outside the table of %d", it0, it0 + k, n);
  if ((reinterpret_cast<uintptr_t>(table) & 31) != 0) return fail(kInvalid, "tv_wide: the table must be 32-byte aligned");
  if (xi == xo || yi == yo) return fail(kInvalid, "tv_wide: ping-pong buffers must differ");
  const WideStep* tab = reinterpret_cast<const WideStep*>(table);
#define OPY_W(KK)                                                                                              \
  hipLaunchKernelGGL((tv_wide_kernel<KK>), dim3(launch_grid(KF(tv_wide_kernel<KK>), grid, 64)), dim3(64), 0,    \
                     as_stream(s), xi, xo, yi, yo, f, insts, tab, n, it0, active_inst, unit_off, nact, rows)
  switch (k) {
    case 2: OPY_W(2); break;
    case 3: OPY_W(3); break;
    case 4: OPY_W(4); break;
    case 5: OPY_W(5); break;
    case 6: OPY_W(6); break;
    case 7: OPY_W(7); break;
    default: OPY_W(8); break;
  }
#undef OPY_W
  return check_launch("tv_wide");
}
