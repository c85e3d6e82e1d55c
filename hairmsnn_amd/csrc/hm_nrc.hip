// Neural radiance caching, the reference's comparator renderer
// (render_nrc.cu:116-701, cuda/nrc.cu:18-398). Per frame:
//   shuffle  : the training-pixel indices (one pixel in every_nth)
//   G_BUFFER : every pixel's path until its spread exceeds the camera
//              footprint, where it queries the cache; training pixels go on
//              with a suffix that ends in a second query (or, for every 16th,
//              runs to the end unbiased) and record every vertex
//   infer    : the cache at all queries (frame + training suffixes)
//   RENDER   : pixel = radiance before the query + throughput x cache;
//              training targets = suffix radiance sums + throughput x cache
//   train    : one Adam step on the training records
// The cache network is the fused MLP of hm_mlp.hip (12-float records; NRC
// fills position / scene scale, wo and the shading normal, channels 9-11 0).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <vector>

#include "../../include/hmsnn.h"
#include "hm_api_util.h"
#include "hm_context.h"
#include "hm_mlp.h"

namespace hm {

// State of one pipeline slot: path buffers, the G_BUFFER arrays and training
// records of up to `frames` consecutive frames, and the stream their G_BUFFER
// pass runs on. The pass does not depend on the network, so consecutive
// frames are traced as one pass and consecutive batches' passes run on
// consecutive slots and overlap; inference, RENDER and training run in frame
// order on the context stream.
struct NrcSlot {
  int frames = 0;  // capacity
  PathBuffers pb{};
  std::vector<void*> allocs;
  hipStream_t st = nullptr;
  int* train_idx = nullptr;
  int* idx_host = nullptr;  // pinned staging of train_idx
  float* query = nullptr;   // n_query x 12
  float4* gb_beta = nullptr;
  uint8_t* gb_hit = nullptr;
  float4* state = nullptr;
  float4* prev = nullptr;
  float4* tb[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};  // pos, wo, n, rad, beta
  int* tb_bounces = nullptr;
  uint8_t* tb_hit = nullptr;
  hipEvent_t ev_gb = nullptr;    // the slot's G_BUFFER pass is done
  hipEvent_t ev_done = nullptr;  // the context stream has consumed the slot
  hipEvent_t ev_copy = nullptr;  // idx_host has been read
  bool used = false;
  void release() {
    if (st) (void)hipStreamSynchronize(st);
    for (void* p : allocs) dev_free(p);
    allocs.clear();
    frames = 0;
    used = false;
    if (idx_host) (void)hipHostFree(idx_host);
    idx_host = nullptr;
    for (hipEvent_t* e : {&ev_gb, &ev_done, &ev_copy})
      if (*e) (void)hipEventDestroy(*e), *e = nullptr;
    if (st) (void)hipStreamDestroy(st);
    st = nullptr;
  }
};

// The buffers and streams stay with the context from one hmsnn_nrc_begin to
// the next (allocating and freeing them took 47 ms of a begin at 512 x 512,
// several times the 8 frames that followed); everything a run computes starts
// over.
struct NrcState {
  MlpState* mlp = nullptr;
  bool ready = false;  // fully built (a failed setup is not reused)
  int n_rec = 0;       // training records per step (numTrainingRecords)
  int n_tpx = 0;       // training pixels (numTrainingPixels)
  int every_nth = 1;
  int frame_size = 0;  // pixels
  int n_query = 0;     // nnFrameSize: frame + training queries, a multiple of 128
  float c = 0.01f;
  int all_unbiased = 0;
  int loss = HMSNN_LOSS_RELATIVE_L2_LUMINANCE;
  float lr = 1e-2f;
  int train_steps = 0;
  int frame = 0;
  uint64_t rng_state = 0;
  std::vector<int> idx;  // current permutation of the training indices
  // Frames of one pass: a pass's 40 depths are bound by their longest rays'
  // chains, about 0.14 ms each at any path count past the tenth, so frames
  // share them (20 frames of 256 x 256: 11.8 ms one by one on four slots, 4.4
  // ms at 8 to a pass, 3.5 ms at 16, 4.0 ms at 32). A call of more than
  // kBatch frames or kBatchPaths paths is several passes, on two slots that
  // overlap one pass's last depths with the next one's first. Splitting smaller
  // calls for that overlap is not worth it: 8 frames of 512 x 512 took 9.6 ms
  // in two passes and 10.1 in one, but the first ones of a scene 23.4 against
  // 20.5 (the second slot's buffers), and 14.5 where the two slots' streams got
  // one hardware queue; half a million paths 6.6 and 6.9, a quarter level.
  static constexpr int kSlots = 2, kBatch = 16;
  static constexpr int kBatchPaths = 4 << 20;
  NrcSlot slots[kSlots];
  int next_slot = 0, last_slot = -1, last_frame = 0;  // the last frame: its slot and place there
  // shared, used in frame order on the context stream
  std::vector<void*> allocs;
  float* cache = nullptr;    // n_query x 3
  float4* gb_rad = nullptr;  // radiance before the query (RENDER pass input), per pixel
  float* train_in = nullptr;   // n_rec x 12
  float* train_tgt = nullptr;  // n_rec x 3
  float4* acc = nullptr;
  float4* avg = nullptr;
  int* counts_dev = nullptr;   // [0] frame cache queries, [1] training records with data
  hipStream_t ctx_stream = nullptr;
  ~NrcState() {
    if (ctx_stream) (void)hipStreamSynchronize(ctx_stream);
    for (NrcSlot& sl : slots) sl.release();
    for (void* p : allocs) dev_free(p);
    if (mlp) mlp_destroy(mlp);
  }
  // Waits for the last run's work and forgets its results; the buffers stay.
  int restart(std::string& err) {
    HM_HIP(hipStreamSynchronize(ctx_stream), err);
    for (NrcSlot& sl : slots) {
      if (sl.st) HM_HIP(hipStreamSynchronize(sl.st), err);
      sl.used = false;
    }
    mlp_destroy(mlp);
    mlp = nullptr;
    train_steps = frame = next_slot = 0;
    last_slot = -1;
    return kOk;
  }
  uint64_t next_u64() {
    uint64_t z = (rng_state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  }
};

void nrc_release(NrcState* s) { delete s; }

namespace {

// Adds v, summed over a 256-thread block, to *counter with one atomic per
// block (every wave of a frame-sized launch adding to the one counter
// serialised there). Every thread of the block calls it.
__device__ __forceinline__ void block_count(int* counter, int v) {
  __shared__ int part[4];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if (__lane_id() == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int sum = part[0] + part[1] + part[2] + part[3];
    if (sum) atomicAdd(counter, sum);
  }
}

// RENDER pass, pixel side (cuda/nrc.cu:378-392): radiance before the query
// plus throughput x max(cache, 0), a NaN cache counting as 0; accumulated
// like writePixel (utils.cuh:13-35, NaN scrub). Also stores the G-buffer
// radiance for inspection and counts the frame's cache queries.
// first: the frame's first slot in pb; nr holds the frame's own arrays.
__global__ void k_nrc_render(PathBuffers pb, int first, NrcPassArgs nr, const float* cache, float4* gb_rad, float4* acc,
                             float4* avg, int accum_id, int* counts) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool in = i < nr.frame_size;
  bool queried = false;
  if (in) {
    const float4 l4 = (pb.flags[first + i] & kNrcSuffix) ? pb.L_short[first + i] : pb.L[first + i];
    const float4 b4 = nr.gb_beta[i];
    V3 cr = v3(cache[3 * (size_t)i], cache[3 * (size_t)i + 1], cache[3 * (size_t)i + 2]);
    if (any_nan(cr)) cr = v3(0.f);
    cr = v3(fmaxf(cr.x, 0.f), fmaxf(cr.y, 0.f), fmaxf(cr.z, 0.f));
    V3 col = v3(l4.x, l4.y, l4.z) + v3(b4.x, b4.y, b4.z) * cr;
    gb_rad[i] = make_float4(l4.x, l4.y, l4.z, 0.f);
    queried = b4.x != 0.f || b4.y != 0.f || b4.z != 0.f;
    if (any_nan(col)) col = v3(0.f);
    if (accum_id > 0) {
      const float4 a = acc[i];
      col = col + v3(a.x, a.y, a.z);
    }
    acc[i] = make_float4(col.x, col.y, col.z, 1.f);
    const float inv = 1.f / (float)(accum_id + 1);
    avg[i] = make_float4(col.x * inv, col.y * inv, col.z * inv, 1.f);
  }
  block_count(&counts[0], queried ? 1 : 0);
}

// RENDER pass, training side (nrcGenerateTrainingData, cuda/nrc.cu:69-133):
// for training pixel tr (whose camera ray hit) and each recorded vertex b <
// bounces, target = sum over the later vertices of their direct light times
// the throughput from b, plus that throughput times the suffix's cache value
// (0 for unbiased suffixes or suffixes without a query); NaN targets become
// 0. The sums run in the reference's order. Records beyond `bounces` stay 0.
// One lane per record: with a lane per training pixel (1638 of them: 7 blocks
// with up to 820 dependent sums a lane) this took 93 us a frame, half of what
// follows the G_BUFFER pass; 8 frames went from 12.1 to 11.4 ms.
__global__ void k_nrc_train_data(NrcPassArgs nr, const int* train_idx, const float* cache, float* train_in,
                                 float* train_tgt, int n_rec, int* counts) {
  const int rec = blockIdx.x * blockDim.x + threadIdx.x;
  const int tr = rec / kNrcMaxBounces, b = rec - tr * kNrcMaxBounces;
  int used = 0;
  if (tr < nr.n_tpx && rec < n_rec) {
    const int px = tr * nr.every_nth + train_idx[tr] % nr.every_nth;
    const int B = min(nr.tb_bounces[tr], kNrcMaxBounces);
    if (b < B && px < nr.frame_size && nr.gb_hit[px]) {
      V3 cr = v3(0.f);
      if (nr.tb_hit[tr] && tr % 16 != 0 && !nr.all_unbiased) {
        const size_t qi = (size_t)nr.frame_size + tr;
        cr = v3(cache[3 * qi], cache[3 * qi + 1], cache[3 * qi + 2]);
      }
      V3 color = v3(0.f), beta = v3(1.f);
      for (int sub = rec; sub < rec - b + B; ++sub) {
        const float4 r = nr.tb_rad[sub], vb = nr.tb_beta[sub];
        color = color + beta * v3(r.x, r.y, r.z);
        beta = beta * v3(vb.x, vb.y, vb.z);
      }
      const float4 p = nr.tb_pos[rec], wo = nr.tb_wo[rec], n = nr.tb_n[rec];
      float* in = train_in + (size_t)rec * kNnInputCh;
      in[0] = p.x; in[1] = p.y; in[2] = p.z;
      in[3] = wo.x; in[4] = wo.y; in[5] = wo.z;
      in[6] = n.x; in[7] = n.y; in[8] = n.z;
      in[9] = 0.f; in[10] = 0.f; in[11] = 0.f;
      V3 t = color + beta * cr;
      if (any_nan(t)) t = v3(0.f);
      train_tgt[3 * (size_t)rec] = t.x;
      train_tgt[3 * (size_t)rec + 1] = t.y;
      train_tgt[3 * (size_t)rec + 2] = t.z;
      used = 1;
    }
  }
  block_count(&counts[1], used);  // the records written
}

struct NrcTimer {
  hipEvent_t e[6];
  NrcTimer() {
    for (auto& x : e) (void)hipEventCreate(&x);
  }
  NrcTimer(const NrcTimer&) = delete;
  NrcTimer& operator=(const NrcTimer&) = delete;
  ~NrcTimer() {
    for (auto& x : e) (void)hipEventDestroy(x);
  }
  static double ms(hipEvent_t a, hipEvent_t b) {
    float t = 0.f;
    (void)hipEventElapsedTime(&t, a, b);
    return t;
  }
};

float nrc_lr_at(float base, int step) {
  if (step < 4000) return base;
  return base * std::pow(0.33f, (float)((step - 4000) / 4000 + 1));
}

// Buffers and events of a slot, which has its stream, for passes of `frames`
// frames.
int nrc_alloc_slot(Context& c, const NrcState& m, NrcSlot& sl, int frames, std::string& err) {
  const size_t npx = (size_t)m.frame_size * frames, tpx = (size_t)m.n_tpx * frames;
  auto S = [&](void** p, size_t bytes) -> int {
    HM_TRY(dev_alloc(p, bytes, err));
    sl.allocs.push_back(*p);
    return kOk;
  };
  for (hipEvent_t* e : {&sl.ev_gb, &sl.ev_done, &sl.ev_copy})
    HM_HIP(hipEventCreateWithFlags(e, hipEventDisableTiming), err);
  HM_TRY(alloc_path_buffers(sl.pb, sl.allocs, npx, true, c.stack_levels(), c.trace_blocks * kTraceBlock, sl.st, err));
  HM_TRY(S((void**)&sl.train_idx, sizeof(int) * tpx));
  HM_TRY(S((void**)&sl.query, sizeof(float) * kNnInputCh * (size_t)m.n_query * frames));
  HM_TRY(S((void**)&sl.gb_beta, sizeof(float4) * npx));
  HM_TRY(S((void**)&sl.gb_hit, npx));
  HM_TRY(S((void**)&sl.state, sizeof(float4) * npx));
  HM_TRY(S((void**)&sl.prev, sizeof(float4) * npx));
  for (float4*& t : sl.tb) HM_TRY(S((void**)&t, sizeof(float4) * tpx * kNrcMaxBounces));
  HM_TRY(S((void**)&sl.tb_bounces, sizeof(int) * tpx));
  HM_TRY(S((void**)&sl.tb_hit, tpx));
  HM_HIP(hipHostMalloc((void**)&sl.idx_host, sizeof(int) * tpx), err);
  HM_HIP(hipStreamSynchronize(sl.st), err);  // the set-up work
  sl.frames = frames;
  return kOk;
}

// The frames of one pass in a call of `frames` frames, and the slots for it.
// Without the memory for larger or more slots the ones that are there serve
// (nrc_setup made one for single frames). No slot has work in flight.
int nrc_batch(Context& c, NrcState& m, int frames) {
  const int cap = std::clamp(NrcState::kBatchPaths / m.frame_size, 1, NrcState::kBatch);
  const int batches = (frames - 1) / cap + 1, want = (frames - 1) / batches + 1;
  for (int k = 0; k < std::min(NrcState::kSlots, batches); ++k) {
    NrcSlot& sl = m.slots[k];
    if (sl.frames >= want) continue;
    NrcSlot grown;
    std::string err;
    grown.st = sl.st;  // the stream stays, and with it the hardware queue it got
    if (nrc_alloc_slot(c, m, grown, want, err)) {
      (void)hipStreamSynchronize(grown.st);
      grown.st = nullptr;
      grown.release();
      (void)hipGetLastError();
      break;
    }
    (void)hipStreamSynchronize(sl.st);
    sl.st = nullptr;
    sl.release();
    sl = std::move(grown);
    if (m.last_slot == k) m.last_slot = -1;
  }
  return std::min(want, m.slots[0].frames);
}

// The buffers that the frames share (the sizes in m are set), and a slot.
int nrc_alloc(Context& c, NrcState& m, std::string& err) {
  const int npx = m.frame_size;
  auto A = [&](void** p, size_t bytes) -> int {
    HM_TRY(dev_alloc(p, bytes, err));
    m.allocs.push_back(*p);
    return kOk;
  };
  // The slots' passes overlap only on hardware queues of their own, and which
  // one a stream gets is settled when it is made: two streams made in a row
  // mostly get different ones (two of 24 histories of scenes opened, rendered
  // and closed before did not; seven where the second stream was made with its
  // slot's first pass. One queue for both costs two passes of 4M paths 19.4 ms
  // against 15.4).
  for (NrcSlot& sl : m.slots) HM_HIP(hipStreamCreateWithFlags(&sl.st, hipStreamNonBlocking), err);
  HM_TRY(nrc_alloc_slot(c, m, m.slots[0], 1, err));
  HM_TRY(A((void**)&m.cache, sizeof(float) * 3 * (size_t)m.n_query));
  HM_TRY(A((void**)&m.gb_rad, sizeof(float4) * (size_t)npx));
  HM_TRY(A((void**)&m.train_in, sizeof(float) * kNnInputCh * (size_t)m.n_rec));
  HM_TRY(A((void**)&m.train_tgt, sizeof(float) * 3 * (size_t)m.n_rec));
  HM_TRY(A((void**)&m.acc, sizeof(float4) * (size_t)npx));
  HM_TRY(A((void**)&m.avg, sizeof(float4) * (size_t)npx));
  HM_TRY(A((void**)&m.counts_dev, sizeof(int) * 4));
  return kOk;
}

int nrc_setup(Context& c, std::string& err) {
  const Scene& s = c.scene;
  const int npx = s.width * s.height;
  const int n_rec = std::max(128, s.nrc_train_records / 128 * 128);
  NrcState* m = c.nrc;
  const bool fresh = !m || !m->ready || m->frame_size != npx || m->n_rec != n_rec;
  if (fresh) {
    nrc_release(m);
    c.nrc = nullptr;
    m = c.nrc = new NrcState();
  } else {
    HM_TRY(m->restart(err));
  }
  m->ready = false;
  m->frame_size = npx;
  m->n_rec = n_rec;
  // render_nrc.cu:130-146, integer divisions as in the reference
  m->n_tpx = std::max(1, m->n_rec / kNrcMaxBounces);
  m->every_nth = std::max(1, npx / m->n_tpx);
  m->n_query = npx + m->n_tpx - m->n_tpx % 128 + 128;
  m->c = s.nrc_c;
  m->all_unbiased = s.nrc_all_unbiased ? 1 : 0;
  m->lr = s.msnn_lr;
  m->loss = s.msnn_loss == "RelativeL2" ? HMSNN_LOSS_RELATIVE_L2
            : s.msnn_loss == "L2"        ? HMSNN_LOSS_L2
                                         : HMSNN_LOSS_RELATIVE_L2_LUMINANCE;
  m->rng_state = s.msnn_seed * 0x2545F4914F6CDD1Dull + 5;
  const int prec = s.msnn_precision == "bf16" ? HMSNN_BF16 : s.msnn_precision == "fp8" ? HMSNN_FP8 : HMSNN_FP16;
  HM_TRY(mlp_create(prec, s.msnn_seed, &m->mlp, err));
  // tcnn.init_weights (scene.cpp:330-331 -> render_nrc.cu:149-150)
  if (!s.nrc_weights.empty()) HM_TRY(mlp_load(*m->mlp, scene_path(s, s.nrc_weights), err));
  m->ctx_stream = c.stream;
  if (fresh) HM_TRY(nrc_alloc(c, *m, err));
  HM_HIP(hipMemsetAsync(m->avg, 0, sizeof(float4) * (size_t)npx, c.stream), err);
  m->idx.resize(m->n_tpx);
  for (int i = 0; i < m->n_tpx; ++i) m->idx[i] = i;  // thrust::sequence (render_nrc.cu:170-173)
  HM_HIP(hipStreamSynchronize(c.stream), err);  // the first passes start after the set-up work
  m->ready = true;
  return kOk;
}

// The pass's arguments, its arrays from frame f of the slot on.
NrcPassArgs nrc_args(const Context& c, const NrcState& m, const NrcSlot& sl, int f) {
  const size_t npx = (size_t)f * m.frame_size, tpx = (size_t)f * m.n_tpx, nv = tpx * kNrcMaxBounces;
  NrcPassArgs a{};
  a.enabled = 1;
  a.all_unbiased = m.all_unbiased;
  a.c = m.c;
  a.scene_scale = c.scene_scale;
  a.frame_size = m.frame_size;
  a.n_tpx = m.n_tpx;
  a.every_nth = m.every_nth;
  a.n_query = m.n_query;
  a.query = sl.query + (size_t)f * m.n_query * kNnInputCh;
  a.gb_beta = sl.gb_beta + npx;
  a.gb_hit = sl.gb_hit + npx;
  a.state = sl.state + npx;
  a.prev = sl.prev + npx;
  a.tb_pos = sl.tb[0] + nv;
  a.tb_wo = sl.tb[1] + nv;
  a.tb_n = sl.tb[2] + nv;
  a.tb_rad = sl.tb[3] + nv;
  a.tb_beta = sl.tb[4] + nv;
  a.tb_bounces = sl.tb_bounces + tpx;
  a.tb_hit = sl.tb_hit + tpx;
  return a;
}

// `frames` consecutive frames (render_nrc.cu:640-701): their shuffles and
// G_BUFFER passes, as one pass, on the next slot, then inference, RENDER and
// training in frame order on the context stream. tm, when given, is the
// frames' timers, whose events mark: [0], [1] (the first frame's only) the
// G_BUFFER pass on the slot's stream; [2] inference start, [3] RENDER start,
// [4] training start and [5] end on the context stream.
int nrc_frames(Context& c, NrcState& m, int frames, NrcTimer* tm, std::string& err) {
  const int npx = m.frame_size;
  NrcSlot& sl = m.slots[m.next_slot];
  m.last_slot = m.next_slot;
  m.last_frame = frames - 1;
  m.next_slot = (m.next_slot + 1) % NrcState::kSlots;
  if (m.slots[m.next_slot].frames < frames) m.next_slot = 0;
  hipStream_t st = sl.st, cs = c.stream;
  if (sl.used) HM_HIP(hipStreamWaitEvent(st, sl.ev_done, 0), err);
  sl.used = true;
  if (tm) (void)hipEventRecord(tm[0].e[0], st);
  // ---- shuffles (render_nrc.cu:652-655): seeded, applied to the previous order ----
  HM_HIP(hipEventSynchronize(sl.ev_copy), err);  // the slot's staging buffer is free again
  const size_t tpx = (size_t)m.n_tpx * frames, nv = tpx * kNrcMaxBounces;
  for (int f = 0; f < frames; ++f) {
    for (int i = m.n_tpx - 1; i > 0; --i) std::swap(m.idx[i], m.idx[(int)(m.next_u64() % (uint64_t)(i + 1))]);
    std::copy(m.idx.begin(), m.idx.end(), sl.idx_host + (size_t)f * m.n_tpx);
  }
  HM_HIP(hipMemcpyAsync(sl.train_idx, sl.idx_host, sizeof(int) * tpx, hipMemcpyHostToDevice, st), err);
  HM_HIP(hipEventRecord(sl.ev_copy, st), err);
  // ---- clear the frames' buffers (owlBufferClear + RESET, render_nrc.cu:684-692) ----
  HM_HIP(hipMemsetAsync(sl.query, 0, sizeof(float) * kNnInputCh * (size_t)m.n_query * frames, st), err);
  HM_HIP(hipMemsetAsync(sl.gb_beta, 0, sizeof(float4) * (size_t)npx * frames, st), err);
  HM_HIP(hipMemsetAsync(sl.gb_hit, 0, (size_t)npx * frames, st), err);
  for (float4* t : sl.tb) HM_HIP(hipMemsetAsync(t, 0, sizeof(float4) * nv, st), err);
  HM_HIP(hipMemsetAsync(sl.tb_bounces, 0, sizeof(int) * tpx, st), err);
  HM_HIP(hipMemsetAsync(sl.tb_hit, 0, tpx, st), err);
  // ---- G_BUFFER ----
  PassConfig cfg = c.pt_pass_config();
  cfg.accum_id = m.frame;
  cfg.frames = frames;
  cfg.dl_zero = 1;  // nrcTracePaths lights every vertex (nrc.cu:166-169)
  cfg.dl_from = 1;
  cfg.max_vertex = kNrcMaxBounces - 1;
  cfg.train_idx = sl.train_idx;
  cfg.every_nth = m.every_nth;
  cfg.nrc = nrc_args(c, m, sl, 0);
  HM_TRY(pt_run_pass(c.view_no_caps(), sl.pb, cfg, st, err));
  if (tm) (void)hipEventRecord(tm[0].e[1], st);
  HM_HIP(hipEventRecord(sl.ev_gb, st), err);
  HM_HIP(hipStreamWaitEvent(cs, sl.ev_gb, 0), err);
  for (int f = 0; f < frames; ++f) {
    const NrcPassArgs nr = nrc_args(c, m, sl, f);
    hipEvent_t* e = tm ? tm[f].e : nullptr;
    // ---- infer (context stream, frame order) ----
    if (e) (void)hipEventRecord(e[2], cs);
    HM_HIP(hipMemsetAsync(m.train_in, 0, sizeof(float) * kNnInputCh * (size_t)m.n_rec, cs), err);
    HM_HIP(hipMemsetAsync(m.train_tgt, 0, sizeof(float) * 3 * (size_t)m.n_rec, cs), err);
    HM_HIP(hipMemsetAsync(m.counts_dev, 0, sizeof(int) * 4, cs), err);
    HM_TRY(mlp_forward(*m.mlp, nr.query, m.n_query, m.cache, cs, err));
    if (e) (void)hipEventRecord(e[3], cs);
    // ---- RENDER ----
    hipLaunchKernelGGL(k_nrc_render, dim3((npx + 255) / 256), dim3(256), 0, cs, sl.pb, f * npx, nr, m.cache, m.gb_rad,
                       m.acc, m.avg, m.frame, m.counts_dev);
    hipLaunchKernelGGL(k_nrc_train_data, dim3((m.n_tpx * kNrcMaxBounces + 255) / 256), dim3(256), 0, cs, nr,
                       sl.train_idx + (size_t)f * m.n_tpx, m.cache, m.train_in, m.train_tgt, m.n_rec, m.counts_dev);
    HM_TRY(check_launch("nrc render", err));
    if (e) (void)hipEventRecord(e[4], cs);
    // ---- train ----
    if (c.scene.nrc_train) {
      const float lr = nrc_lr_at(m.lr, m.train_steps);
      HM_TRY(mlp_loss_grad_step(*m.mlp, m.train_in, m.train_tgt, m.n_rec, m.loss, nullptr, nullptr, true, lr, cs,
                                err));
      m.train_steps++;
    }
    if (e) (void)hipEventRecord(e[5], cs);
    m.frame++;
  }
  HM_HIP(hipEventRecord(sl.ev_done, cs), err);
  return kOk;
}

}  // namespace

}  // namespace hm

using namespace hm;

struct hmsnn_ctx {
  Context c;
};

extern "C" {

int hmsnn_nrc_begin(hmsnn_ctx* ctx) {
  if (!ctx) return fail(HMSNN_EINVAL, "NULL context");
  std::string err;
  Context& c = ctx->c;
  int rc = nrc_setup(c, err);
  if (!rc && hipStreamSynchronize(c.stream) != hipSuccess) rc = HMSNN_EDEVICE, err = "NRC setup failed";
  return rc ? fail(rc, err) : HMSNN_OK;
}

int hmsnn_nrc_set_params(hmsnn_ctx* ctx, float c_spread, int all_unbiased) {
  if (!ctx || !(c_spread >= 0.f)) return fail(HMSNN_EINVAL, "hmsnn_nrc_set_params: bad arguments");
  if (!ctx->c.nrc) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  ctx->c.nrc->c = c_spread;
  ctx->c.nrc->all_unbiased = all_unbiased ? 1 : 0;
  return HMSNN_OK;
}

int hmsnn_nrc_frames(hmsnn_ctx* ctx, int frames, hmsnn_nrc_stats* stats) {
  if (!ctx || frames < 0) return fail(HMSNN_EINVAL, "hmsnn_nrc_frames: bad arguments");
  Context& c = ctx->c;
  if (!c.nrc || !c.nrc->ready) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  std::string err;
  std::vector<NrcTimer> timers(stats ? (size_t)frames : 0);
  const auto t0 = std::chrono::steady_clock::now();
  const int batch = frames > 0 ? nrc_batch(c, *c.nrc, frames) : 1;
  c.nrc->next_slot = 0;
  for (int k = 0; k < frames; k += batch) {
    int rc = nrc_frames(c, *c.nrc, std::min(batch, frames - k), stats ? &timers[k] : nullptr, err);
    if (rc) return fail(rc, err);
  }
  hipError_t e = hipStreamSynchronize(c.stream);
  if (e != hipSuccess) return fail(HMSNN_EDEVICE, hipGetErrorString(e));
  const auto t1 = std::chrono::steady_clock::now();
  if (stats) {
    hmsnn_nrc_stats local{};
    for (int k = 0; k < frames; k += batch) local.gbuffer_ms += NrcTimer::ms(timers[k].e[0], timers[k].e[1]);
    for (NrcTimer& tm : timers) {
      local.infer_ms += NrcTimer::ms(tm.e[2], tm.e[3]);
      local.render_ms += NrcTimer::ms(tm.e[3], tm.e[4]);
      local.train_ms += NrcTimer::ms(tm.e[4], tm.e[5]);
    }
    local.total_ms = std::chrono::duration<double, std::milli>(t1 - t0).count();
    local.frames = frames;
    local.train_steps = c.nrc->train_steps;
    int counts[4] = {0, 0, 0, 0};
    e = hipMemcpy(counts, c.nrc->counts_dev, sizeof(counts), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fail(HMSNN_EDEVICE, hipGetErrorString(e));
    local.cache_queries = counts[0];
    local.train_records_used = counts[1];
    *stats = local;
  }
  return HMSNN_OK;
}

int hmsnn_nrc_get_image(hmsnn_ctx* ctx, float* rgba) {
  if (!ctx || !rgba) return fail(HMSNN_EINVAL, "hmsnn_nrc_get_image: bad arguments");
  Context& c = ctx->c;
  if (!c.nrc || !c.nrc->ready) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  const size_t bytes = sizeof(float4) * (size_t)c.scene.width * c.scene.height;
  hipError_t e = hipMemcpyAsync(rgba, c.nrc->avg, bytes, hipMemcpyDeviceToHost, c.stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
  return e == hipSuccess ? HMSNN_OK : fail(HMSNN_EDEVICE, hipGetErrorString(e));
}

int hmsnn_nrc_get_sizes(hmsnn_ctx* ctx, int sizes[4]) {
  if (!ctx || !sizes) return fail(HMSNN_EINVAL, "hmsnn_nrc_get_sizes: bad arguments");
  const NrcState* m = ctx->c.nrc;
  if (!m) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  sizes[0] = m->n_tpx;
  sizes[1] = m->every_nth;
  sizes[2] = m->n_query;
  sizes[3] = m->n_rec;
  return HMSNN_OK;
}

int hmsnn_nrc_get_buffer(hmsnn_ctx* ctx, int which, void* host, size_t bytes) {
  if (!ctx || !host) return fail(HMSNN_EINVAL, "hmsnn_nrc_get_buffer: bad arguments");
  const NrcState* m = ctx->c.nrc;
  if (!m) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  const size_t npx = (size_t)m->frame_size;
  if (m->last_slot < 0) return fail(HMSNN_EINVAL, "hmsnn_nrc_get_buffer: no frame rendered yet");
  const NrcSlot& sl = m->slots[m->last_slot];
  const NrcPassArgs nr = nrc_args(ctx->c, *m, sl, m->last_frame);
  const void* src = nullptr;
  size_t need = 0;
  switch (which) {
    case HMSNN_NRC_QUERY: src = nr.query, need = sizeof(float) * kNnInputCh * (size_t)m->n_query; break;
    case HMSNN_NRC_CACHE: src = m->cache, need = sizeof(float) * 3 * (size_t)m->n_query; break;
    case HMSNN_NRC_GB_RADIANCE: src = m->gb_rad, need = sizeof(float4) * npx; break;
    case HMSNN_NRC_GB_BETA: src = nr.gb_beta, need = sizeof(float4) * npx; break;
    case HMSNN_NRC_GB_HIT: src = nr.gb_hit, need = npx; break;
    case HMSNN_NRC_TRAIN_INPUT: src = m->train_in, need = sizeof(float) * kNnInputCh * (size_t)m->n_rec; break;
    case HMSNN_NRC_TRAIN_TARGET: src = m->train_tgt, need = sizeof(float) * 3 * (size_t)m->n_rec; break;
    case HMSNN_NRC_TRAIN_IDX: src = sl.train_idx + (size_t)m->last_frame * m->n_tpx, need = sizeof(int) * (size_t)m->n_tpx; break;
    case HMSNN_NRC_TRAIN_BOUNCES: src = nr.tb_bounces, need = sizeof(int) * (size_t)m->n_tpx; break;
    case HMSNN_NRC_TRAIN_HIT: src = nr.tb_hit, need = (size_t)m->n_tpx; break;
    default: return fail(HMSNN_EINVAL, "hmsnn_nrc_get_buffer: unknown buffer");
  }
  if (bytes != need) return fail(HMSNN_EINVAL, "hmsnn_nrc_get_buffer: size mismatch");
  hipError_t e = hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, ctx->c.stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->c.stream);
  return e == hipSuccess ? HMSNN_OK : fail(HMSNN_EDEVICE, hipGetErrorString(e));
}

int hmsnn_nrc_get_mlp_weights(hmsnn_ctx* ctx, float* w_host, int n) {
  if (!ctx || !w_host || n != kMlpWeightCount) return fail(HMSNN_EINVAL, "hmsnn_nrc_get_mlp_weights: bad arguments");
  if (!ctx->c.nrc || !ctx->c.nrc->ready) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  std::string err;
  if (hipStreamSynchronize(ctx->c.stream) != hipSuccess) return fail(HMSNN_EDEVICE, "stream failed");
  int rc = mlp_get_weights(*ctx->c.nrc->mlp, w_host, err);
  return rc ? fail(rc, err) : HMSNN_OK;
}

int hmsnn_nrc_save_weights(hmsnn_ctx* ctx, const char* path) {
  if (!ctx || !path) return fail(HMSNN_EINVAL, "hmsnn_nrc_save_weights: bad arguments");
  if (!ctx->c.nrc || !ctx->c.nrc->ready) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  std::string err;
  if (hipStreamSynchronize(ctx->c.stream) != hipSuccess) return fail(HMSNN_EDEVICE, "stream failed");
  int rc = mlp_save(*ctx->c.nrc->mlp, path, err);
  return rc ? fail(rc, err) : HMSNN_OK;
}

int hmsnn_nrc_set_mlp_weights(hmsnn_ctx* ctx, const float* w_host, int n) {
  if (!ctx || !w_host || n != kMlpWeightCount) return fail(HMSNN_EINVAL, "hmsnn_nrc_set_mlp_weights: bad arguments");
  if (!ctx->c.nrc || !ctx->c.nrc->ready) return fail(HMSNN_EINVAL, "call hmsnn_nrc_begin first");
  std::string err;
  if (hipStreamSynchronize(ctx->c.stream) != hipSuccess) return fail(HMSNN_EDEVICE, "stream failed");
  int rc = mlp_set_weights(*ctx->c.nrc->mlp, w_host, err);
  return rc ? fail(rc, err) : HMSNN_OK;
}

int hmsnn_render_nrc(hmsnn_ctx* ctx, int spp, float* rgba, hmsnn_nrc_stats* stats) {
  if (!ctx || spp <= 0) return fail(HMSNN_EINVAL, "hmsnn_render_nrc: bad arguments");
  int rc = hmsnn_nrc_begin(ctx);
  if (rc) return rc;
  rc = hmsnn_nrc_frames(ctx, spp, stats);
  if (rc) return rc;
  return rgba ? hmsnn_nrc_get_image(ctx, rgba) : HMSNN_OK;
}

}  // extern "C"
