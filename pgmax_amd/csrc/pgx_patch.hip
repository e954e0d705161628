// Small graphs of 2x2 factors (variables of at most 4 edges): several BP
// iterations per launch on patches of the graph held in LDS.
//
// A launch per iteration takes 5 to 6 us on a graph that does not fill the
// chip, whatever its size: the launch itself, three dependent loads (tile,
// positions, messages) and one factor update, of which only the last is work.
// A workgroup here takes a patch: its own factors and, around them, the
// factors within a few steps (rings). It loads the patch's messages, tables
// and evidence once, runs as many iterations as it has rings -- each leaves
// one ring fewer up to date -- and writes its own factors' messages. Graphs
// of components that fit a workgroup need no rings and run to the last
// iteration in one launch. Every factor update, own or repeated in a
// neighbour's rings, is the same operations in the same order on the same
// values as in the per-phase kernels, so the messages are equal bit for bit.
//
// One thread per edge: it sums the messages of its variable, exchanges the
// result with its factor's other edge (the neighbouring lane) and does half
// of the factor's log-sum-exps. A variable's four messages are LDS reads at
// indices kept in registers. An iteration costs a workgroup of 1,024 edges
// about 0.7 us at T = 0 and 1.3 at T = 1, a launch of four with its loads 7.6.
// 16 x 16 torus, 20 iterations at T = 0: 102 us in 20 launches, 19.5 in one;
// 50 x 50, 200 at T = 1: 1,164 us in 200 launches, 379 in 50. The workgroup
// folds a step's delta into one address once: an atomic per wavefront took
// the 50 x 50 torus 12.3 us a launch.

#include "pgx_launch.h"

namespace pgx {
namespace {

// The other lane of a pair (lanes 2k and 2k + 1).
__device__ __forceinline__ float pair_lane(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xb1, 0xf, 0xf, false));
}

// Max of a wavefront's u (in every lane), by lane shifts in the vector unit.
__device__ __forceinline__ uint32_t wave_umax(uint32_t u) {
  auto step = [&](auto ctrl) {
    u = max(u, uint32_t(__builtin_amdgcn_update_dpp(0, int(u), decltype(ctrl)::value, 0xf, 0xf,
                                                    false)));
  };
  step(std::integral_constant<int, 0x111>{});  // row_shr:1, 2, 4, 8
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});  // row_bcast:15
  step(std::integral_constant<int, 0x143>{});  // row_bcast:31
  return uint32_t(__builtin_amdgcn_readlane(int(u), 63));
}

struct PatchIO {
  const float* in;   // the caller's messages (first launch), else null
  int64_t in_stride;
  const float* src;  // one float per edge, num_edges per batch element
  float* dst;
  float* out;        // the caller's result (last launch), else null
  int32_t it0, steps;
};

// The normalised, clipped one-float message of edge e.
__device__ __forceinline__ float patch_load(const PatchIO& io, int32_t b, int32_t num_edges,
                                            int32_t e) {
  if (!io.in) return io.src[int64_t(b) * num_edges + e];
  float x[2];
  ldv<2>(io.in + b * io.in_stride + 2 * int64_t(e), x);
  const float mx = nmax(x[0], x[1]);
  return pair_encode(nmax(x[0] - mx, kMsgNegInf), nmax(x[1] - mx, kMsgNegInf));
}

template <bool kT0>
__device__ __forceinline__ void patch_body(const DevGraph& g, const DevPatches& p,
                                           const RunBufs& r, const PatchIO& io, float t) {
  __shared__ float m[2][kPatchSlots];
  __shared__ uint32_t red[4];  // the patch's delta of steps j, j - 1, ..
  const int32_t b = blockIdx.y, tid = threadIdx.x;
  const int4 d0 = p.desc[2 * blockIdx.x], d1 = p.desc[2 * blockIdx.x + 1];
  const int32_t nt = d0.y, own = d1.x;
  const bool on = tid < nt;
  int32_t e = 0, ring = 0;
  uint32_t s01 = ~0u, s23 = ~0u;
  float l00 = 0.f, l01 = 0.f, l10 = 0.f, l11 = 0.f, e0 = 0.f, e1 = 0.f;
  if (on) {
    const int4 th = p.thr[d0.x + tid];
    e = th.x & kPatchEdgeMask;
    ring = int32_t(uint32_t(th.x) >> kPatchRingShift);
    s01 = uint32_t(th.z);
    s23 = uint32_t(th.w);
    float lp[4], ev[2];
    ldv<4>(r.lp + b * r.lp_stride + p.lp[d0.x + tid], lp);
    ldv<2>(r.ev + b * r.ev_stride + th.y, ev);
    m[0][tid] = patch_load(io, b, g.num_edges, e);
    e0 = ev[0];
    e1 = ev[1];
    // the edge's own states are rows: the second edge reads the transpose
    l00 = clip_lp(lp[0]);
    l01 = clip_lp((tid & 1) ? lp[2] : lp[1]);
    l10 = clip_lp((tid & 1) ? lp[1] : lp[2]);
    l11 = clip_lp(lp[3]);
  }
  for (int32_t k = tid; k < d0.w; k += blockDim.x)
    m[0][nt + k] = patch_load(io, b, g.num_edges, p.extra[d0.z + k]);
  if (tid < 4) red[tid] = 0;
  __syncthreads();
  for (int32_t j = 0; j < io.steps; ++j) {
    const float* cur = m[j & 1];
    float* nxt = m[(j & 1) ^ 1];
    float dl = 0.f;
    // both edges of a factor share its ring, so a pair of lanes stays together
    if (on && ring < io.steps - j) {
      const uint32_t s[4] = {s01 & 0xffffu, s01 >> 16, s23 & 0xffffu, s23 >> 16};
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = s[u] != 0xffffu ? cur[s[u]] : 0.f;
      const float2 o = pair_decode(cur[tid]);
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s[u] != 0xffffu) {
          const float2 q = pair_decode(v[u]);
          a0 += q.x;
          a1 += q.y;
        }
      const float x0 = (a0 + e0) - o.x, x1 = (a1 + e1) - o.y;
      const float y0 = pair_lane(x0), y1 = pair_lane(x1);
      const float s00 = (x0 + y0) + l00, s01f = (x0 + y1) + l01;
      const float s10 = (x1 + y0) + l10, s11 = (x1 + y1) + l11;
      const float f0 = (kT0 ? nmax(s00, s01f) : lse2(s00, s01f, t)) - x0;
      const float f1 = (kT0 ? nmax(s10, s11) : lse2(s10, s11, t)) - x1;
      float n0, n1;
      damp_norm2(r.d, r.omd, o.x, o.y, f0, f1, n0, n1, dl);
      nxt[tid] = pair_encode(n0, n1);
    }
    if ((tid & ~63) < own) {  // whole wavefronts; repeated factors leave dl to their owner
      const uint32_t u = wave_umax(tid < own ? __float_as_uint(fabsf(dl)) : 0u);
      if ((tid & 63) == 0) atomicMax(&red[j & 3], u);
    }
    __syncthreads();
    if (tid == 0) {  // (four steps pass before red[j & 3] is folded into again)
      atomicMax(delta_slot(r, b, io.it0 + j), red[j & 3]);
      red[j & 3] = 0;
    }
  }
  if (tid < own) {
    const float v = m[io.steps & 1][tid];
    if (io.out) {
      const float2 q = pair_decode(v);
      const float x[2] = {q.x, q.y};
      stv<2>(io.out + b * g.num_es + 2 * int64_t(e), x);
    } else {
      io.dst[int64_t(b) * g.num_edges + e] = v;
    }
  }
}

template <bool kT0>
__global__ void __launch_bounds__(kPatchThreads)
    k_patch(DevGraph g, DevPatches p, RunBufs r, PatchIO io) {
  if (!kT0 && r.t == 1.f)
    patch_body<kT0>(g, p, r, io, 1.f);
  else
    patch_body<kT0>(g, p, r, io, r.t);
}

}  // namespace

int launch_patches(pgx_graph* g, const RunBufs& r, const float* ftov_in, int64_t in_stride,
                   float* out, float* buf, int32_t batch, bool t0, hipStream_t s) {
  const DevPatches& p = g->patches;
  const int32_t steps = p.depth ? p.depth : r.n_it;
  float* const half[2] = {buf, buf + size_t(batch) * size_t(g->dev.num_edges)};
  const dim3 grid(p.count, batch), block(p.threads);
  for (int32_t it = 0, n = 0; it < r.n_it; it += steps, ++n) {
    PatchIO io;
    io.in = it == 0 ? ftov_in : nullptr;
    io.in_stride = in_stride;
    io.src = half[n & 1];
    io.dst = half[(n & 1) ^ 1];
    io.it0 = it;
    io.steps = std::min(steps, r.n_it - it);
    io.out = it + io.steps == r.n_it ? out : nullptr;
    if (t0)
      hipLaunchKernelGGL((k_patch<true>), grid, block, 0, s, g->dev, p, r, io);
    else
      hipLaunchKernelGGL((k_patch<false>), grid, block, 0, s, g->dev, p, r, io);
  }
  PGX_HIP(hipGetLastError());
  return PGX_OK;
}

}  // namespace pgx
