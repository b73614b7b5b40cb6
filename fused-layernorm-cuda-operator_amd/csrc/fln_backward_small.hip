// fln_backward_small.hip -- the backward of small problems in one launch, without a workspace.
//
// With few rows the two-stage backward is bound by latency: stage 1, the hand-over of its partial
// rows through memory, a second launch to sum them, and, for rows past the register tiles, a third
// for their statistics.  dx needs sums over a row and dgamma / dbeta sums over the columns, but
// neither needs the other, and a small x and dy are served from L2 the second time.  So the blocks
// of one launch take two roles:
//   dx blocks (the first p.dx_blocks): whole rows, each in the registers of `wpr` waves, up to 8
//     vectors per lane in the I/O type (65536 16-bit or 32768 fp32 columns: without column sums to
//     carry, a 1024-thread block holds x and dy of a row that wide); as bwd_reg_kernel otherwise.
//   column blocks: `cw` vector columns each (8 to 64, one per lane) over every row: the block's
//     1024 / cw row slices take the rows in turn, 4 in flight each, then the slices' partial sums
//     of a column are added through LDS.
// Both roles take unaligned vectors (RaggedRow), so any width of at least one vector runs here.
//
// Taken for at most one row per CU, where no width that it takes loses.  Backward calls, us, before -> here: fp32 32 x 768 6.4 -> 3.6, 128
// x 768 6.9 -> 3.8, 256 x 768 7.7 -> 4.7, 256 x 16384 27.4 -> 18.2, 256 x 32768 36.8 -> 36.5; bf16 64 x
// 4096 8.1 -> 4.3, 256 x 1024 8.4 -> 4.8, 256 x 8192 19.5 -> 8.1, 200 x 12288 19.9 -> 7.6, 100 x 40000
// 25.3 -> 14.7, 1 x 32768 11.5 -> 6.7; erf GELU 64 x 4096 9.5 -> 8.0, 100 x 30000
// 32.3 -> 15.2; residual gradient 200 x 50000 41.1 -> 28.2.  More rows amortize the two stages'
// overhead and read x and dy once: wide ones soon (us, two stages / here: bf16 512 x 4097 15.5 / 13.8,
// 768 x 4097 17.7 / 18.8; fp32 768 x 2048 10.8 / 9.7, 1000 x 2048 11.2 / 12.0), narrow ones only past
// 1000 (fp32 512 x 768 7.8 / 6.2, 1000 x 768 10.8 / 8.7, 1500 x 768 9.6 / 11.9; bf16 1000 x 4096 14.8 /
// 13.7, 1500 x 4096 16.4 / 19.1), so that a limit by rows and columns would serve more calls.  What
// bounds it: one launch and two dependent round trips to memory
// for narrow rows; the bandwidth of the few CUs that hold a row for wide ones.
#include <type_traits>

#include "fln_device.h"
#include "fln_internal.h"

namespace fln {
namespace {

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;

struct SmallArgs {
  BwdParams p;
  int dx_blocks;  // blocks of the dx role (0: dx not requested)
  int groups;     // row groups per dx block
  int cw;         // vector columns of a column block
};

template <class T, bool DRES, int GELU, int VEC, int VPL>
__global__ __launch_bounds__(kSmallThreads) void bwd_small_kernel(const SmallArgs a) {
  using P = Pack<T, VEC>;
  const BwdParams& p = a.p;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t N = p.cols;
  const uint32_t row_bytes = static_cast<uint32_t>(N * sizeof(T));
  const RaggedRow<T, VEC> rag(static_cast<uint32_t>(N));
  const T* X = static_cast<const T*>(p.x);
  const T* DY = static_cast<const T*>(p.dy);
  const rsrc_t g_rs = make_rsrc(p.gamma, row_bytes);
  const rsrc_t b_rs = make_rsrc(p.beta, row_bytes);  // GELU only; absent beta reads as zeros
  const bool has_g = p.gamma != nullptr;
  __shared__ float4 gelu_tab[GELU != 0 ? kGeluTabN : 1];
  if constexpr (GELU != 0) {
    if (threadIdx.x < kGeluTabN)
      gelu_tab[threadIdx.x] = reinterpret_cast<const float4*>(
          GELU == 1 ? kGeluTabData : kGeluTanhTabData)[threadIdx.x];
  }
  // Gradient at the LayerNorm output of one element: dy, or dy GELU'(xhat gamma + beta).
  auto upstream = [&](float d, float xh, float g, float b) -> float {
    if constexpr (GELU != 0) {
      const float u = kGeluTabInvH * fmaf(xh, g, b);
      d = 0.5f * fmaf(d, gelu_grad2_sign_tab(gelu_tab, u), d);
    }
    (void)xh, (void)g, (void)b;
    return d;
  };

  if (static_cast<int>(blockIdx.x) < a.dx_blocks) {
    __shared__ float red[2][kSmallWaves + 16];  // padded for combine_partials
    const int wpr = p.wpr;
    const int rg = wave / wpr;
    const int t = (wave - rg * wpr) * kWave + lane;
    const int tpr = kWave * wpr;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * a.groups + rg;
    const bool in = rg < a.groups && row < p.rows;
    const uint32_t nb = in ? row_bytes : 0u;  // no row: reads zeros, stores nothing
    const int64_t r = in ? row : 0;
    // Up to 2 vectors per lane gamma, beta and the residual gradient are loaded with the row; wider
    // tiles have no registers for them and read them where they are used.
    constexpr bool PRELOAD = VPL <= 2;
    const rsrc_t xr = make_rsrc(X + r * N, nb), dr = make_rsrc(DY + r * N, nb);
    const rsrc_t rr = make_rsrc(DRES ? static_cast<const T*>(p.dres) + r * N : nullptr, nb);
    uint32_t off[VPL];
    P xv[VPL], dv[VPL], gp[PRELOAD ? VPL : 1], bp[PRELOAD && GELU ? VPL : 1],
        rp[PRELOAD && DRES ? VPL : 1];
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      off[i] = rag.off(static_cast<uint32_t>(t + i * tpr));
      xv[i] = buf_load_at<P>(xr, off[i]);
      dv[i] = buf_load_at<P>(dr, off[i]);
      if constexpr (PRELOAD) {
        gp[i] = buf_load_at<P>(g_rs, off[i]);
        if constexpr (GELU != 0) bp[i] = buf_load_at<P>(b_rs, off[i]);
        if constexpr (DRES) rp[i] = buf_load_at<P>(rr, off[i]);
      }
    }
    const uint32_t sb = in ? 4u : 0u;
    const float mu = __builtin_bit_cast(
        float, BufIO<4>::load(make_rsrc(p.rms ? nullptr : p.mean + r, sb), 0));
    const float rs = __builtin_bit_cast(float, BufIO<4>::load(make_rsrc(p.rstd + r, sb), 0));
    if constexpr (GELU != 0) __syncthreads();  // the table
    auto gamma = [&](int i) -> P {
      if constexpr (PRELOAD)
        return gp[i];
      else
        return buf_load_at<P>(g_rs, off[i]);
    };
    auto beta = [&](int i) -> P {
      if constexpr (GELU == 0)
        return P{};
      else if constexpr (PRELOAD)
        return bp[i];
      else
        return buf_load_at<P>(b_rs, off[i]);
    };
    float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const P gv = gamma(i), bv = beta(i);
      const int lo = rag.lo(static_cast<uint32_t>(t + i * tpr));
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float xh = (to_f32(xv[i].v[e]) - mu) * rs;
        const float gm = has_g ? to_f32(gv.v[e]) : 1.0f;
        const float g = upstream(to_f32(dv[i].v[e]), xh, gm, GELU ? to_f32(bv.v[e]) : 0.0f) * gm;
        if (e >= lo) {  // the last vector's own elements
          s1 += g;
          s2 = fmaf(g, xh, s2);
        }
      }
    }
    s1 = wave_allreduce<SumOp>(s1);
    s2 = wave_allreduce<SumOp>(s2);
    if (wpr > 1) {
      if (lane == 0) {
        red[0][wave] = s1;
        red[1][wave] = s2;
      }
      __syncthreads();
      s1 = combine_partials<SumOp>(red[0], rg * wpr, wpr, lane, 0.0f);
      s2 = combine_partials<SumOp>(red[1], rg * wpr, wpr, lane, 0.0f);
    }
    const float inv_n = 1.0f / static_cast<float>(N);
    const float cb = p.rms ? 0.0f : -rs * (s1 * inv_n);
    const float cx = -rs * (s2 * inv_n);
    const rsrc_t xo = make_rsrc(static_cast<T*>(p.dx) + r * N, nb);
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      if constexpr (!PRELOAD) {  // widened again from the packs, not kept in fp32 across the sums
        keep_packed(xv[i]);
        keep_packed(dv[i]);
      }
      const P gv = gamma(i), bv = beta(i);
      P rv{};
      if constexpr (DRES) {
        if constexpr (PRELOAD)
          rv = rp[i];
        else
          rv = buf_load_at<P>(rr, off[i]);
      }
      P o;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float xh = (to_f32(xv[i].v[e]) - mu) * rs;
        const float gm = has_g ? to_f32(gv.v[e]) : 1.0f;
        const float d = upstream(to_f32(dv[i].v[e]), xh, gm, GELU ? to_f32(bv.v[e]) : 0.0f);
        float dxv = fmaf(rs, d * gm, fmaf(cx, xh, cb));
        if constexpr (DRES) dxv += to_f32(rv.v[e]);
        o.v[e] = from_f32<T>(dxv);
      }
      buf_store_at<P>(o, xo, off[i]);
    }
    return;
  }

  // Column role: lane = (row slice of the wave, vector column).
  constexpr int kRows = 4;               // rows in flight per lane
  constexpr int kMostCols = kWave * VEC; // columns of a block at most
  __shared__ float part[2][kSmallWaves * kMostCols];
  const int cw = a.cw;
  const int col = lane & (cw - 1), slices = kSmallWaves * (kWave / cw);
  const int slice = wave * (kWave / cw) + lane / cw;
  const uint32_t v0 = (blockIdx.x - static_cast<uint32_t>(a.dx_blocks)) * cw;
  const uint32_t off = rag.off(v0 + col);
  // One resource over each tensor (under 2 GiB here): the lanes of a wave take different rows.
  const uint32_t rows = static_cast<uint32_t>(p.rows);
  const rsrc_t xr = make_rsrc(X, rows * row_bytes), dr = make_rsrc(DY, rows * row_bytes);
  const rsrc_t mr = make_rsrc(p.rms ? nullptr : p.mean, rows * 4u), sr = make_rsrc(p.rstd, rows * 4u);
  const P gv = buf_load_at<P>(g_rs, off);
  P bv{};
  if constexpr (GELU != 0) {
    bv = buf_load_at<P>(b_rs, off);
    __syncthreads();  // the table
  }
  float acc_g[VEC], acc_b[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc_g[e] = acc_b[e] = 0.0f;
  for (uint32_t row0 = 0; row0 < rows; row0 += kRows * slices) {
    P xv[kRows], dv[kRows];
    float mu[kRows], rs[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      // Rows past the tensor read as zeros, statistics included: they add exact zeros.
      const uint32_t r = row0 + u * slices + slice;
      const bool in = r < rows;
      const uint32_t o = in && off != kOutOfRange ? r * row_bytes + off : kOutOfRange;
      const uint32_t so = in ? r * 4u : kOutOfRange;
      xv[u] = buf_load_at<P>(xr, o);
      dv[u] = buf_load_at<P>(dr, o);
      mu[u] = __builtin_bit_cast(float, BufIO<4>::load(mr, so));
      rs[u] = __builtin_bit_cast(float, BufIO<4>::load(sr, so));
    }
    // The rows in flight are summed by themselves first: shorter chains, smaller rounding errors.
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      float sum_g = 0.0f, sum_b = 0.0f;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        const float xh = (to_f32(xv[u].v[e]) - mu[u]) * rs[u];
        const float d = upstream(to_f32(dv[u].v[e]), xh, has_g ? to_f32(gv.v[e]) : 1.0f,
                                 GELU ? to_f32(bv.v[e]) : 0.0f);
        sum_g = fmaf(d, xh, sum_g);
        sum_b += d;
      }
      acc_g[e] += sum_g;
      acc_b[e] += sum_b;
    }
  }
  const int cols = cw * VEC;  // columns of this block
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    part[0][slice * cols + col * VEC + e] = acc_g[e];
    part[1][slice * cols + col * VEC + e] = acc_b[e];
  }
  __syncthreads();
  if (static_cast<int>(threadIdx.x) >= 2 * cols) return;
  const int which = static_cast<int>(threadIdx.x) / cols, c = static_cast<int>(threadIdx.x) % cols;
  const uint32_t v = v0 + static_cast<uint32_t>(c / VEC);
  void* out = which == 0 ? p.out_g : p.out_b;
  if (out == nullptr || c % VEC < rag.lo(v)) return;  // (lo = VEC past the row)
  // Eight sums and a tree over them (slices is a multiple of 16): shorter chains, closer to the
  // exact sum than the slices in turn.
  float s[8] = {};
  for (int k = 0; k < slices; k += 8)
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] += part[which][(k + j) * cols + c];
  const float sum = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
  store_param(out, p.out_dtype, rag.off(v) / static_cast<uint32_t>(sizeof(T)) + c % VEC, sum);
}

template <class T, int VPL>
int launch_vpl(const SmallArgs& a, int blocks, hipStream_t s) {
  constexpr int VEC = 16 / sizeof(T);
  if (a.p.gelu == FLN_GELU_ERF) {
    static std::atomic<void*> cache[64];
    return launch_cached(bwd_small_kernel<T, false, 1, VEC, VPL>, cache, dim3(blocks),
                         dim3(kSmallThreads), s, a);
  }
  if (a.p.gelu == FLN_GELU_TANH) {
    static std::atomic<void*> cache[64];
    return launch_cached(bwd_small_kernel<T, false, 2, VEC, VPL>, cache, dim3(blocks),
                         dim3(kSmallThreads), s, a);
  }
  if (a.p.dres) {
    static std::atomic<void*> cache[64];
    return launch_cached(bwd_small_kernel<T, true, 0, VEC, VPL>, cache, dim3(blocks),
                         dim3(kSmallThreads), s, a);
  }
  static std::atomic<void*> cache[64];
  return launch_cached(bwd_small_kernel<T, false, 0, VEC, VPL>, cache, dim3(blocks),
                       dim3(kSmallThreads), s, a);
}

struct SmallPlan {
  int wpr, vpl, groups, dx_blocks, col_blocks, cw;
};

// Waves per row (1..16) and vectors per lane (1, 2, 4 or 8) of the dx role; vpl 0: too wide.
SmallPlan plan(const BwdParams& p, int es) {
  SmallPlan s{};
  const int64_t vec = 16 / es, nvec = (p.cols + vec - 1) / vec;
  const int64_t cus = device_cu_count();
  const int64_t slots = (nvec + kWave - 1) / kWave;  // wave-wide vectors of a row
  s.vpl = slots <= 16 ? 1 : slots <= 32 ? 2 : slots <= 64 ? 4 : slots <= 128 ? 8 : 0;
  if (s.vpl == 0) return s;
  s.wpr = static_cast<int>((slots + s.vpl - 1) / s.vpl);
  // Column blocks: fewer columns and more row slices each while a slice has more than 4 rows, the
  // blocks leaving most CUs to the rows.
  s.cw = kWave;
  while (s.cw > 8 && p.rows * s.cw > 4 * kSmallThreads && nvec <= 64 * (s.cw / 2)) s.cw /= 2;
  if (p.out_g || p.out_b) s.col_blocks = static_cast<int>((nvec + s.cw - 1) / s.cw);
  if (p.dx) {
    // One row per block while the blocks still fit the CUs, then as many as a block holds.
    const int64_t room = cus > 2 * s.col_blocks ? cus - s.col_blocks : cus / 2;
    int64_t groups = (p.rows + room - 1) / room;
    const int most = kSmallWaves / s.wpr;
    if (groups > most) groups = most;
    s.groups = static_cast<int>(groups);
    s.dx_blocks = static_cast<int>((p.rows + groups - 1) / groups);
  }
  return s;
}

}  // namespace

bool backward_is_small(const BwdParams& p, const void* dgamma, const void* dbeta, int dtype) {
  const Tuning& tun = tuning();
  if (tun.bwd_small_rows < 0 || tun.bwd_epl > 0 || tun.bwd_wpr > 0 || tun.bwd_threads > 0 ||
      tun.bwd_grid_mult > 0 || tun.bwd_no_lds || tun.bwd_no_two_pass || tun.bwd_stat_splits > 0 ||
      tun.bwd_colpass_per_cu > 0)
    return false;
  const int es = element_size(dtype);
  const int64_t vec = 16 / es;
  if (p.cols < vec || p.cols > 16 * kWave * 8 * vec) return false;
  const int64_t limit = tun.bwd_small_rows > 0 ? tun.bwd_small_rows : device_cu_count();
  if (p.rows > limit || p.rows * p.cols * es >= int64_t(1) << 31) return false;
  // The widest rows (8 vectors per lane) are bound by the one CU that holds a row: with a few rows
  // the two passes spread each over many CUs (backward calls, us, here / two passes: bf16 LN 4 x
  // 50000 11.8 / 8.4, 16 x 50000 12.6 / 11.6, 20 x 50000 12.8 / 12.8, 40 x 50000 13.6 / 15.8; widths
  // that are no whole vectors 4 x 60001 15.4 / 9.4, 16 x 60001 15.8 / 13.2, 32 x 60001 16.8 / 15.5, 40
  // x 60001 17.2 / 16.9; fp32 4 x 32768 8.5 / 7.2, 16 x 20001 8.2 / 10.3, 16 x 32768 9.4 / 9.9).  The
  // rule looks at the width, not at the pointers.
  // So are 16-bit rows with GELU, whose derivative is taken twice per element: 8 vectors per lane
  // never (64 x 50000 24.5 / 21.2, 128 x 50000 28.3 / 28), 4 only while every block has its own CU
  // (200 x 20000 23.1 / 31.6, but 256 x 20000 35.4 / 34.2, 256 x 32768 38.1 / 33.1).
  const int64_t nvec = (p.cols + vec - 1) / vec;
  if (nvec > 64 * kWave) {
    if (p.gelu && es == 2) return false;
    if (p.rows < (es == 2 && p.cols % vec != 0 ? 32 : 16)) return false;
  } else if (nvec > 32 * kWave && p.gelu && es == 2 &&
             p.rows + (nvec + kWave - 1) / kWave > device_cu_count()) {
    return false;
  }
  // The roles run at the same time: an output in place of an input (dx over dy, say) would be
  // written while other blocks still read it.
  const int64_t bytes = p.rows * p.cols * es, param = p.cols * es, stat = p.rows * 4;
  const std::pair<const void*, int64_t> in[] = {{p.x, bytes},    {p.dy, bytes},  {p.dres, bytes},
                                                {p.gamma, param}, {p.beta, param}, {p.mean, stat},
                                                {p.rstd, stat}};
  const std::pair<const void*, int64_t> out[] = {
      {p.dx, bytes}, {dgamma, 4 * p.cols}, {dbeta, 4 * p.cols}};
  for (const auto& o : out)
    for (const auto& i : in)
      if (overlaps(o.first, o.second, i.first, i.second)) return false;
  return true;
}

int launch_backward_small(const BwdParams& p, int dtype, hipStream_t s) {
  SmallArgs a{};
  a.p = p;
  const SmallPlan pl = plan(p, element_size(dtype));
  if (pl.vpl == 0) return FLN_ERR_INVALID;
  a.p.wpr = pl.wpr;
  a.dx_blocks = pl.dx_blocks;
  a.groups = pl.groups;
  a.cw = pl.cw;
  const int blocks = pl.dx_blocks + pl.col_blocks;
  if (blocks == 0) return FLN_OK;
  auto go = [&](auto t) {
    using T = decltype(t);
    switch (pl.vpl) {
      case 1: return launch_vpl<T, 1>(a, blocks, s);
      case 2: return launch_vpl<T, 2>(a, blocks, s);
      case 4: return launch_vpl<T, 4>(a, blocks, s);
      default: return launch_vpl<T, 8>(a, blocks, s);
    }
  };
  switch (dtype) {
    case FLN_F32: return go(float{});
    case FLN_BF16: return go(__bf16{});
    case FLN_F16: return go(_Float16{});
    default: return FLN_ERR_INVALID;
  }
}

}  // namespace fln
