// Adjoint of the path tracer for differentiable hair appearance: gradients of
// L(mean image) w.r.t. per-strand sigma_a and global beta_m, beta_n, alpha,
// given dL/d(image).
//
// The wavefront tracer renders the paths of up to 16 passes (the reference's
// per-pixel streams, cuda/path_tracing.cu:29) into its radiance ring and
// records every hair vertex on a tape: ray, hit, throughput, random state,
// radiance gathered before it and the visibility of its two light samples, 81
// bytes. The vertices are then independent: one thread per record evaluates
// the vertex again from its random state and differentiates every factor that
// depends on the parameters, with adj = dL/dI / spp:
//   direct-lighting sample k:  c_k = f_k * w_k * (parameter-free factor), so
//     dc_k = (c_k / f_k) * df_k + c_k * dw_k / w_k, where w_k is the
//     power-heuristic MIS weight through the BSDF pdf (1 for delta lights);
//   continuation: the radiance still to come after the vertex is
//     proportional to f, so it contributes rem * df / f.
// Sampled directions, the sampling pdfs in the estimators' denominators and
// Russian roulette are held fixed (detached): the estimator stays unbiased
// for the derivative of the expected image.
// Per-strand gradients are reduced with FP64 atomics.
//
// Tracing the paths once more instead of taping them (one lane per path, all
// its rays included) took 39 ms of a 73 ms step at 512 x 512, 16 passes, 3.2 M
// segments. The tape is sequential memory, 2 GB there, on a GPU of 288 GB.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/hmsnn.h"
#include "hm_api_util.h"
#include "hm_context.h"
#include "hm_hair_ad.h"

namespace hm {

namespace {

struct AdjArgs {
  HairConstsAD hcd;
  const float4* dl_dimg;  // w*h
  float inv_spp;
  int dl_zero, dl_from, max_vertex;
  const float4* ring;  // primal radiance of pass p of the run at ring[p * npx + pixel]
  double* g_sigma;  // num_strands * 3
  double* g_glob;   // 3
  float* g_px;      // optional: w*h*3 per-pixel d/d(beta_m, beta_n, alpha)
};

HM_D int strand_of(const SceneView& sc, int prim) { return (int)sc.seg_by_id[8 * (size_t)prim + 7]; }

HM_D V3 strand_sigma_of(const SceneView& sc, int prim) {
  if (!sc.strand_sigma) return sc.sigma_a;
  const int s = strand_of(sc, prim);
  return v3(sc.strand_sigma[3 * s], sc.strand_sigma[3 * s + 1], sc.strand_sigma[3 * s + 2]);
}

// g[k] = sum_c wk_c * f_c'[k] + wc * r[k]; the global part goes to gg, the
// sigma part to the strand's FP64 slots.
HM_D void add_grad(const SceneView& sc, const AdjArgs& a, int prim, const Dual f[3], V3 wk, float wc, const float r[kAdParams],
                   float* gg) {
  float g[kAdParams];
  bool ok = true;
#pragma unroll
  for (int k = 0; k < kAdParams; ++k) {
    g[k] = wk.x * f[0].d[k] + wk.y * f[1].d[k] + wk.z * f[2].d[k] + wc * r[k];
    ok = ok && isfinite(g[k]);
  }
  if (!ok) return;
  gg[0] += g[0];
  gg[1] += g[1];
  gg[2] += g[2];
  const int strand = strand_of(sc, prim);
#pragma unroll
  for (int c = 0; c < 3; ++c)
    if (g[3 + c] != 0.f) atomicAdd(&a.g_sigma[3 * (size_t)strand + c], (double)g[3 + c]);
}

HM_D V3 safe_ratio(V3 c, V3 f) {
  return v3(f.x != 0.f ? c.x / f.x : 0.f, f.y != 0.f ? c.y / f.y : 0.f, f.z != 0.f ? c.z / f.z : 0.f);
}

// One taped vertex: the gradient of its direct lighting (shadow rays visible
// per vis) and of its continuation, which the radiance still to come, Lt - L,
// is proportional to. The operations and random draws are those the tracer's
// shading makes from the same random state. gg receives the global part.
HM_D void adj_vertex(const SceneView& sc, const AdjArgs& a, V3 o, V3 d, float t, int prim, float u, V3 beta,
                     uint32_t rng, V3 L, V3 Lt, V3 adj, int depth, int vis, float gg[3]) {
  Hit h;
  setup_hit(sc, o, d, t, prim, u, h);
  const V3 sigma = strand_sigma_of(sc, prim);
  if (depth == 0 ? a.dl_zero != 0 : depth >= a.dl_from) {
    DirectOut dl;
    direct_lighting(sc, h, rng, dl);
    const bool v1 = dl.has1 && (vis & 1), v2 = dl.has2 && (vis & 2);
    V3 sum = v3(0.f);
    if (v1) sum = sum + dl.c1;
    if (v2) sum = sum + dl.c2;
    if (any_nan(sum)) {
      sum = v3(0.f);
    } else {
      const V3 W = adj * beta;  // dLoss / dc per channel
      // one copy of the derivative code for both light samples
#pragma unroll 1
      for (int k = 0; k < 2; ++k) {
        if (!(k ? v2 : v1)) continue;
        Dual f[3], pd;
        hair_eval_dual(a.hcd, h.wo_local, k ? dl.wl2 : dl.wl1, h.hw.h, sigma, f, &pd);
        const float pb = k ? dl.bp2 : dl.bp1, pl = k ? dl.lp2 : dl.lp1;
        // d(weight) / weight through the BSDF pdf: of the light sample's weight
        // pl^2 / (pl^2 + pb^2), of the BSDF sample's pb^2 / (pb^2 + pl^2)
        float c = 0.f;
        if (k == 0) c = dl.mis1 ? -2.f * pb / (pl * pl + pb * pb) : 0.f;
        else c = pb > 0.f ? 2.f * pl * pl / (pb * (pb * pb + pl * pl)) : 0.f;
        float r[kAdParams];
#pragma unroll
        for (int q = 0; q < kAdParams; ++q) r[q] = c * pd.d[q];
        const V3 cc = k ? dl.c2 : dl.c1;
        add_grad(sc, a, prim, f, W * safe_ratio(cc, k ? dl.f2 : dl.f1), dot(W, cc), r, gg);
      }
    }
    L = L + beta * sum;
  }
  if (depth >= 1) {
    const float rr = fmaxf(0.05f, 1.f - luminance(beta));
    if (draw(rng) < rr) return;
  }
  if (depth + 1 > a.max_vertex) return;
  const BsdfSample bs = sample_bsdf(sc, h, rng);
  if (any_nan((bs.pdf == 0.f) ? bs.f : bs.f / bs.pdf)) return;
  const V3 rem = Lt - L;  // radiance gathered after this vertex
  Dual fd[3], pd;
  hair_eval_dual(a.hcd, h.wo_local, bs.wl, h.hw.h, sigma, fd, &pd);
  float r[kAdParams];
#pragma unroll
  for (int k = 0; k < kAdParams; ++k) r[k] = 0.f;
  add_grad(sc, a, prim, fd, adj * safe_ratio(rem, bs.f), 0.f, r, gg);
}

// Bound by its vector arithmetic (the dual-number evaluations carry six
// tangents): 6.7 ms for the 20 M records (4.85 a path) of a 512 x 512, 16-pass
// step. Two waves per SIMD keep its registers (1, 2, 3 and 4 waves: 42.7, 40.9,
// 42.4 and 42.2 ms for the whole step).
__global__ void __launch_bounds__(256, 2) k_adjoint(SceneView sc, AdjArgs a, VertexTape tape,
                                                                   const long long* count) {
  const int npx = sc.width * sc.height;
  const long long n = min(*count, tape.cap);
  const long long stride = (long long)gridDim.x * blockDim.x;
  float gg[3] = {0.f, 0.f, 0.f};
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float4 l = tape.L[i];
    const int prim = __float_as_int(l.w);
    if (prim < 0) continue;
    const int4 m = tape.meta[i];
    const float4 g4 = a.dl_dimg[m.x];
    const V3 adj = a.inv_spp * v3(g4.x, g4.y, g4.z);
    if (adj.x == 0.f && adj.y == 0.f && adj.z == 0.f) continue;
    const float4 lt = a.ring[(size_t)m.y * npx + m.x];
    const V3 Lt = v3(lt.x, lt.y, lt.z);
    if (any_nan(Lt)) continue;  // writePixel drops NaN samples (utils.cuh:20-21)
    const float4 o = tape.o[i], d = tape.d[i], b = tape.beta[i];
    float gv[3] = {0.f, 0.f, 0.f};
    adj_vertex(sc, a, v3(o.x, o.y, o.z), v3(d.x, d.y, d.z), o.w, prim, d.w, v3(b.x, b.y, b.z), __float_as_uint(b.w),
               v3(l.x, l.y, l.z), Lt, adj, m.z, tape.vis[i], gv);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      gg[k] += gv[k];
      if (a.g_px && gv[k] != 0.f) atomicAdd(&a.g_px[3 * (size_t)m.x + k], gv[k]);
    }
  }
  // the global gradients: wave sums, block sums in LDS, one FP64 atomic per
  // block and parameter
  __shared__ float part[4][3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float v = gg[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (__lane_id() == 0) part[threadIdx.x >> 6][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = 0.0;
    for (int w = 0; w < 4; ++w) v += (double)part[w][threadIdx.x];
    if (v != 0.0) atomicAdd(&a.g_glob[threadIdx.x], v);
  }
}

// Records a path is expected to leave (its hair vertices and its last, missed
// ray): what the context's last run left and an eighth more (tape_per_path), at
// least kTapePerPath. A run that leaves more than its tape holds is repeated
// with a larger one, or, where that would pass kTapeBytes, as two runs of half
// the passes; only a single pass may take more, and gives the tape back when
// the call ends.
constexpr double kTapePerPath = 10.0;
constexpr size_t kTapeBytes = (size_t)8 << 30;

void tape_release(Context& c) {
  for (void* p : c.tape_allocs) dev_free(p);
  c.tape_allocs.clear();
  c.tape = VertexTape{};
}

// Records for `paths` paths.
long long tape_records(const Context& c, long long paths) {
  return (long long)std::ceil(std::max(kTapePerPath, c.tape_per_path) * (double)paths) + 64;
}

// Makes the context's tape hold at least `records`.
int tape_ensure(Context& c, long long records, std::string& err) {
  if (c.tape.cap >= records) return kOk;
  tape_release(c);
  const size_t n = (size_t)records;
  auto A = [&](void** p, size_t bytes) -> int {
    HM_TRY(dev_alloc(p, bytes, err));
    c.tape_allocs.push_back(*p);
    return kOk;
  };
  for (float4** p : {&c.tape.o, &c.tape.d, &c.tape.beta, &c.tape.L}) HM_TRY(A((void**)p, sizeof(float4) * n));
  HM_TRY(A((void**)&c.tape.meta, sizeof(int4) * n));
  HM_TRY(A((void**)&c.tape.vis, n));
  c.tape.cap = records;
  return kOk;
}

// Group g of K's share of the tape.
VertexTape tape_share(const VertexTape& t, int g, int K) {
  VertexTape v = t;
  v.cap = t.cap / K;
  const size_t off = (size_t)v.cap * g;
  v.o += off;
  v.d += off;
  v.beta += off;
  v.L += off;
  v.meta += off;
  v.vis += off;
  return v;
}

// Passes p0 .. p0 + np - 1 (at most kStreamRing): traced with the tape, then
// differentiated.
int adjoint_passes(Context& c, const AdjArgs& a, int p0, int np, float4* tmp_acc, std::string& err) {
  const size_t npx = (size_t)c.scene.width * c.scene.height;
  const int K = stream_groups(c, np);
  const long long paths = (long long)npx * np;
  long long want = tape_records(c, paths);
  for (;;) {
    const bool fits = np == 1 || (size_t)want * kTapeRecordBytes <= kTapeBytes;
    const int rc = fits ? tape_ensure(c, want, err) : kENoMem;
    if (rc && np > 1) {  // no room: half the passes at a time
      err.clear();
      (void)hipGetLastError();
      HM_TRY(adjoint_passes(c, a, p0, np / 2, tmp_acc, err));
      return adjoint_passes(c, a, p0 + np / 2, np - np / 2, tmp_acc, err);
    }
    HM_TRY(rc);
    StreamTape st{};
    for (int g = 0; g < K; ++g) st.tape[g] = tape_share(c.tape, g, K);
    HM_TRY(stream_passes(c, p0, np, tmp_acc, tmp_acc + npx, nullptr, err, &st));
    long long count[kStreamGroups] = {};
    for (int g = 0; g < K; ++g)
      HM_HIP(hipMemcpyAsync(&count[g], st.count[g], sizeof(long long), hipMemcpyDeviceToHost, c.stream), err);
    HM_HIP(hipStreamSynchronize(c.stream), err);
    long long most = 0;
    for (int g = 0; g < K; ++g) most = std::max(most, count[g]);
    c.tape_per_path = 1.125 * (double)(K * most) / (double)paths;
    if (most > st.tape[0].cap) {
      want = K * (most + most / 8);
      continue;
    }
    AdjArgs x = a;
    x.ring = c.stream_ring;
    for (int g = 0; g < K; ++g) {
      const int blocks = (int)std::min<long long>(c.num_cus * 8ll, std::max<long long>(1, (count[g] + 255) / 256));
      hipLaunchKernelGGL(k_adjoint, dim3(blocks), dim3(256), 0, c.stream, c.view, x, st.tape[g], st.count[g]);
    }
    return check_launch("adjoint", err);
  }
}

}  // namespace

}  // namespace hm

using namespace hm;

struct hmsnn_ctx {
  Context c;
};

extern "C" {

int hmsnn_set_hair_params(hmsnn_ctx* ctx, float beta_m, float beta_n, float alpha) {
  if (!ctx || !(beta_m > 0.f) || !(beta_n > 0.f)) return fail(HMSNN_EINVAL, "hmsnn_set_hair_params: bad arguments");
  Context& c = ctx->c;
  c.scene.beta_m = beta_m;
  c.scene.beta_n = beta_n;
  c.scene.alpha = alpha;
  const float gains[4] = {c.scene.R_G, c.scene.TT_G, c.scene.TRT_G, c.scene.TRRT_G};
  c.view.hc = make_hair_consts(beta_m, beta_n, alpha, gains);
  return HMSNN_OK;
}

int hmsnn_adjoint_render(hmsnn_ctx* ctx, int spp, const float* dl_dimg, double* grad_sigma, double grad_glob[3],
                         float* grad_px) {
  if (!ctx || spp <= 0 || !dl_dimg || !grad_glob) return fail(HMSNN_EINVAL, "hmsnn_adjoint_render: bad arguments");
  Context& c = ctx->c;
  if (!c.scene.has_hair) return fail(HMSNN_EINVAL, "scene has no hair");
  std::string err;
  int rc = c.ensure_image(err);
  if (rc) return fail(rc, err);
  const size_t npx = (size_t)c.scene.width * c.scene.height;
  const size_t ns = (size_t)c.hair.num_strands;
  float4* d_adj = nullptr;
  double* d_gs = nullptr;
  double* d_gg = nullptr;
  float* d_px = nullptr;
  rc = dev_alloc((void**)&d_adj, sizeof(float4) * npx, err);
  if (!rc) rc = dev_alloc((void**)&d_gs, sizeof(double) * 3 * ns, err);
  if (!rc) rc = dev_alloc((void**)&d_gg, sizeof(double) * 4, err);
  if (!rc && grad_px) rc = dev_alloc((void**)&d_px, sizeof(float) * 3 * npx, err);
  auto cleanup = [&]() {
    (void)hipStreamSynchronize(c.stream);
    dev_free(d_adj);
    dev_free(d_gs);
    dev_free(d_gg);
    dev_free(d_px);
  };
  if (rc) {
    cleanup();
    return fail(rc, err);
  }
  hipError_t e = hipMemcpyAsync(d_adj, dl_dimg, sizeof(float4) * npx, hipMemcpyHostToDevice, c.stream);
  if (e == hipSuccess) e = hipMemsetAsync(d_gs, 0, sizeof(double) * 3 * ns, c.stream);
  if (e == hipSuccess) e = hipMemsetAsync(d_gg, 0, sizeof(double) * 4, c.stream);
  if (e == hipSuccess && d_px) e = hipMemsetAsync(d_px, 0, sizeof(float) * 3 * npx, c.stream);
  if (e != hipSuccess) {
    cleanup();
    return fail(HMSNN_EDEVICE, hipGetErrorString(e));
  }
  AdjArgs a;
  const float gains[4] = {c.scene.R_G, c.scene.TT_G, c.scene.TRT_G, c.scene.TRRT_G};
  a.hcd = make_hair_consts_ad(c.scene.beta_m, c.scene.beta_n, c.scene.alpha, gains);
  a.dl_dimg = d_adj;
  a.inv_spp = 1.f / (float)spp;
  const PassConfig pc = c.pt_pass_config();
  a.dl_zero = pc.dl_zero;
  a.dl_from = pc.dl_from;
  a.max_vertex = pc.max_vertex;
  a.g_sigma = d_gs;
  a.g_glob = d_gg;
  a.g_px = d_px;
  float4* tmp_acc = nullptr;
  rc = dev_alloc((void**)&tmp_acc, 2 * sizeof(float4) * (size_t)npx, err);
  for (int p0 = 0; !rc && p0 < spp;) {
    // as many passes as a tape of kTapeBytes is expected to hold
    const size_t pass_bytes = (size_t)tape_records(c, (long long)npx) * kTapeRecordBytes;
    const int chunk = (int)std::max<size_t>(1, std::min<size_t>(kStreamRing, kTapeBytes / pass_bytes));
    const int np = std::min(chunk, spp - p0);
    rc = adjoint_passes(c, a, p0, np, tmp_acc, err);
    p0 += np;
  }
  (void)hipStreamSynchronize(c.stream);
  dev_free(tmp_acc);
  if ((size_t)c.tape.cap * kTapeRecordBytes > kTapeBytes) tape_release(c);
  if (!rc) {
    double gg[4];
    e = hipMemcpyAsync(gg, d_gg, sizeof(gg), hipMemcpyDeviceToHost, c.stream);
    if (e == hipSuccess && grad_sigma)
      e = hipMemcpyAsync(grad_sigma, d_gs, sizeof(double) * 3 * ns, hipMemcpyDeviceToHost, c.stream);
    if (e == hipSuccess && grad_px)
      e = hipMemcpyAsync(grad_px, d_px, sizeof(float) * 3 * npx, hipMemcpyDeviceToHost, c.stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
    if (e != hipSuccess) rc = HMSNN_EDEVICE, err = hipGetErrorString(e);
    else for (int k = 0; k < 3; ++k) grad_glob[k] = gg[k];
  }
  cleanup();
  return rc ? fail(rc, err) : HMSNN_OK;
}

}  // extern "C"
