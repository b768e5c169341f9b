// sovits_decoder.cpp — the SoVITS decoder (Generator::forward, src/sovits/dec.hpp:264-345) issued
// through the C ABI as a fixed sequence of fused convolution launches, eager or recorded into a HIP
// graph (gsvk_sovits_decoder_*).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <vector>

#include "gsvk.h"
#include "gsvk_conv_group.hpp"
#include "gsvk_sovits.h"

namespace {

constexpr size_t kAlign = 256;  // bytes: alignment of every workspace region

size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Workspace layout: the folded bias (c0 floats), then 8 activation slots of `slot` elements of the
// activation dtype each: X (stage input, then the stage output), Y (upsampler output, the first
// residual), TA0..TA2 (each ResBlock's pair middle activation, so the three ResBlocks can run
// side by side; where a pair is one launch, the second pair's sum) and CUR0..CUR2 (the three branch accumulators). The pairs' LeakyReLU inputs are
// not stored: the first conv of a pair reads lrelu(cur) as it loads (GSVK_CONV_X_LRELU).
enum Slot {
  kX,
  kY,
  kTa0,
  kCur0 = kTa0 + GSVK_SOVITS_RESBLOCKS,
  kSlots = kCur0 + GSVK_SOVITS_RESBLOCKS
};

// Where one launch for the three ResBlocks' m-th convolutions does not pay (conv1d_group_pays),
// two of them run on two more streams, concurrent with the first on the main one (they share only the upsampler's output, which they read); the branch mean waits for all
// three. In a recorded graph the streams and events are the capture's; eagerly, the side streams
// are the device's own (below) and the events the call's.
constexpr int kSide = GSVK_SOVITS_RESBLOCKS - 1;
struct Branches {
  const hipStream_t* side;  // kSide streams
  hipEvent_t fork;
  const hipEvent_t* join;
};

struct Layout {
  size_t vec_bytes = 0;   // bytes of the folded bias (c0 floats, rounded up)
  size_t slot_bytes = 0;  // bytes of one activation slot
  size_t t_out = 0;       // samples of the output
  size_t bytes = 0;
};

// The shapes a valid descriptor must have (no buffer pointers needed) and the workspace layout.
int shapes(const gsvk_sovits_decoder_desc* d, Layout* lay) {
  if (!d || !d->stage) return GSVK_E_NULL;
  if (d->dtype != GSVK_F32 && d->dtype != GSVK_F16) return GSVK_E_DTYPE;
  if (d->frames == 0 || d->c_z == 0 || d->c0 == 0 || d->pre_k == 0 || d->post_k == 0 ||
      d->n_stages == 0 || d->n_stages > GSVK_SOVITS_MAX_STAGES)
    return GSVK_E_SIZE;
  size_t c = d->c0, T = d->frames, slot = d->c0 * d->frames;
  for (size_t s = 0; s < d->n_stages; ++s) {
    const gsvk_sovits_stage& S = d->stage[s];
    if (S.c_in != c || S.c_out == 0 || S.ups_k == 0 || S.ups_u == 0) return GSVK_E_SIZE;
    for (size_t j = 0; j < GSVK_SOVITS_RESBLOCKS; ++j)
      if (S.res_k[j] == 0) return GSVK_E_SIZE;
    for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m)
      if (S.res_dil[m] == 0) return GSVK_E_SIZE;
    if (T > SIZE_MAX / S.ups_u) return GSVK_E_SIZE;
    c = S.c_out;
    T *= S.ups_u;
    if (T > SIZE_MAX / c) return GSVK_E_SIZE;
    if (c * T > slot) slot = c * T;
  }
  const size_t esz = d->dtype == GSVK_F32 ? 4 : 2;
  if (slot > (SIZE_MAX / 2) / esz / kSlots) return GSVK_E_SIZE;
  lay->vec_bytes = round_up(d->c0 * sizeof(float), kAlign);
  lay->slot_bytes = round_up(slot * esz, kAlign);
  lay->t_out = T;
  lay->bytes = lay->vec_bytes + kSlots * lay->slot_bytes;
  return GSVK_OK;
}

// Shapes, every weight and buffer pointer, and the workspace; the convolutions check the rest
// (aliasing, strides) themselves.
int check_workspace(const gsvk_sovits_decoder_desc* d, Layout* lay) {
  const int rc = shapes(d, lay);
  if (rc) return rc;
  if (!d->pre_w || !d->post_w || !d->z || !d->out) return GSVK_E_NULL;
  if (d->g_in && (!d->cond_w || !d->ge)) return GSVK_E_NULL;
  for (size_t s = 0; s < d->n_stages; ++s) {
    const gsvk_sovits_stage& S = d->stage[s];
    if (!S.ups_w) return GSVK_E_NULL;
    for (size_t j = 0; j < GSVK_SOVITS_RESBLOCKS; ++j)
      for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m)
        if (!S.w1[j][m] || !S.w2[j][m]) return GSVK_E_NULL;
  }
  if (!d->workspace) return GSVK_E_NULL;
  if (reinterpret_cast<uintptr_t>(d->workspace) % 16 != 0) return GSVK_E_ARG;
  if (d->workspace_bytes < lay->bytes) return GSVK_E_SIZE;
  return GSVK_OK;
}

// The passes of the decoder; three convolutions grouped into one launch count as three.
int count_launches(const gsvk_sovits_decoder_desc* d) {
  // cond with the bias fold (with conditioning), conv_pre, 20 per stage, conv_post
  return (d->g_in ? 1 : 0) + 1 + 20 * static_cast<int>(d->n_stages) + 1;
}

// Where the pairs of the three ResBlocks share a launch instead of running on branches. A recorded
// graph: the branches' fork and join cost about 20 us a stage, but a branch runs into its next pair
// while another's last workgroups drain. Whole decoder, us, branches against shared up to 1.2 M / 2.4 M
// elements: 75 frames fp16 586 / 565 / 568, exact 744 / 725 / 733, 150 frames 757 / 751 / 770 and 966 /
// 967 / 987. Issued eagerly the branches also cost host calls and cross-stream waits. One stage, us:
// 96 x 16006 exact 244 -> 166, 24 x 40000 117 -> 66, 24 x 120000 171 -> 139 (level above 5 M).
constexpr size_t kTogetherGraph = 1200000, kTogetherEager = 5000000;

// One Generator stage (dec.hpp:283-336): out = lrelu(mean_j ResBlock_j(ups(x)), slope_next). x
// [c_in, T] with row stride ldx arrives LeakyReLU'd; buf[kY .. kSlots - 1] hold c_out x T ups_u
// elements each. br: the streams ResBlocks 1 and 2 may run on (nullptr: all on st). together: the
// three ResBlocks' m-th pairs share a launch up to this many elements of one activation.
int issue_stage(int dt, int rx, const gsvk_sovits_stage& S, const void* x, size_t ldx, size_t T,
                void* const* buf, float slope_next, void* out, void* st, const Branches* br,
                size_t together) {
  const float slope = 0.1f;  // LRELU_SLOPE (dec.hpp:284, 322, 324)
  const size_t C = S.c_out, Tu = T * S.ups_u;
  // y = ups(x)  (dec.hpp:285)
  if (int rc = gsvk_convt1d(dt, rx, x, ldx, S.ups_w, S.ups_b, GSVK_CONV_EPI_BIAS, 0.f, nullptr,
                            nullptr, 0, buf[kY], Tu, S.c_in, C, T, S.ups_k, S.ups_u, st))
    return rc;
  T = Tu;
  const void* curs[GSVK_SOVITS_RESBLOCKS];
  gsvk::ConvItem c1[GSVK_SOVITS_PAIRS][GSVK_SOVITS_RESBLOCKS];
  gsvk::ConvItem c2[GSVK_SOVITS_PAIRS][GSVK_SOVITS_RESBLOCKS];
  size_t ord[GSVK_SOVITS_RESBLOCKS];  // ResBlocks, largest k first
  for (size_t j = 0; j < GSVK_SOVITS_RESBLOCKS; ++j) ord[j] = j, curs[j] = buf[kCur0 + j];
  std::sort(ord, ord + GSVK_SOVITS_RESBLOCKS,
            [&](size_t p, size_t q) { return S.res_k[p] > S.res_k[q]; });
  for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m)
    for (size_t i = 0; i < GSVK_SOVITS_RESBLOCKS; ++i) {
      const size_t j = ord[i];
      void* cur = buf[kCur0 + j];
      void* ta = buf[kTa0 + j];
      // cur_j starts as a copy of y (dec.hpp:316): the first pair reads y in place
      const void* src = m == 0 ? buf[kY] : cur;
      // t_a = lrelu(convs1[m](lrelu(cur_j)))  (dec.hpp:322-324: leaky_relu_write as the
      // convolution reads its input, leaky_relu_io in its store)
      c1[m][i] = {src, S.w1[j][m], S.b1[j][m], nullptr, nullptr, ta, S.res_k[j], S.res_dil[m]};
      // cur_j = res + convs2[m](t_a)  (dec.hpp:325-326)
      c2[m][i] = {ta, S.w2[j][m], S.b2[j][m], cur, src, nullptr, S.res_k[j], 1};
    }
  // Narrow stages run a pair as one launch, from one buffer into another: y -> cur -> t_a -> cur.
  const bool grouped = gsvk::conv1d_group_pays(C, T);
  bool pairs = !grouped;
  for (size_t j = 0; j < GSVK_SOVITS_RESBLOCKS; ++j)
    for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m)
      pairs = pairs && gsvk::conv1d_pair_fits(C, T, S.res_k[j], S.res_dil[m], dt == GSVK_F32 ? 4 : 2);
  // The convolutions of ResBlocks i .. i + n - 1 (in that order) on stream bst.
  auto blocks = [&](size_t i, int n, void* bst) -> int {
    for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m) {
      if (pairs) {
        gsvk::ConvItem p1[GSVK_SOVITS_RESBLOCKS], p2[GSVK_SOVITS_RESBLOCKS];
        for (int e = 0; e < n; ++e) {
          const size_t j = ord[i + e];
          p1[e] = c1[m][i + e], p2[e] = c2[m][i + e];
          p1[e].x = p2[e].res = m == 0 ? buf[kY] : m == 1 ? buf[kCur0 + j] : buf[kTa0 + j];
          p2[e].cur = m == 1 ? buf[kTa0 + j] : buf[kCur0 + j];
        }
        if (int e = gsvk::conv1d_pairs(dt, rx, p1, p2, n, slope, T, C, T, bst)) return e;
        continue;
      }
      if (int e = gsvk::conv1d_group(dt, rx, &c1[m][i], n,
                                     GSVK_CONV_EPI_LRELU | GSVK_CONV_X_LRELU, slope, T, C, T,
                                     bst))
        return e;
      if (int e = gsvk::conv1d_group(dt, rx, &c2[m][i], n, GSVK_CONV_EPI_RES, slope, T, C, T,
                                     bst))
        return e;
    }
    return GSVK_OK;
  };
  static_assert(GSVK_SOVITS_PAIRS == 3, "the buffers the pairs alternate between");
  if (grouped || (pairs && C * T <= together)) {
    if (int rc = blocks(0, GSVK_SOVITS_RESBLOCKS, st)) return rc;
  } else if (!br) {
    for (size_t i = 0; i < GSVK_SOVITS_RESBLOCKS; ++i)
      if (int rc = blocks(i, 1, st)) return rc;
  } else {
    int rc = GSVK_OK;  // (a failed wait still reaches the joins below)
    if (hipEventRecord(br->fork, static_cast<hipStream_t>(st)) != hipSuccess) return GSVK_E_HIP;
    for (int i = 0; i < kSide; ++i)
      if (hipStreamWaitEvent(br->side[i], br->fork, 0) != hipSuccess) rc = GSVK_E_HIP;
    // (the longest ResBlock last: on the main stream it measured 1-2% slower at 192 channels)
    for (size_t i = GSVK_SOVITS_RESBLOCKS; i-- > 0 && rc == GSVK_OK;)
      rc = blocks(i, 1, i + 1 < GSVK_SOVITS_RESBLOCKS ? br->side[kSide - 1 - i] : st);
    // every side stream joins back, also after an error (a capture must end joined)
    for (int i = 0; i < kSide; ++i)
      if ((hipEventRecord(br->join[i], br->side[i]) != hipSuccess ||
           hipStreamWaitEvent(static_cast<hipStream_t>(st), br->join[i], 0) != hipSuccess) &&
          rc == GSVK_OK)
        rc = GSVK_E_HIP;
    if (rc) return rc;
  }
  // x = lrelu(mean_j cur_j): mul_write / add_scaled_inplace (dec.hpp:328-333) with the next
  // stage's leaky_relu_io (dec.hpp:284, 0.1) or the final one (dec.hpp:342, 0.01).
  return gsvk_resblock_branch_mean(dt, curs, nullptr, GSVK_SOVITS_RESBLOCKS, out, C * T, 1,
                                   slope_next, st);
}

// The launches of one decoder pass in Generator::forward's order.
int issue(const gsvk_sovits_decoder_desc* d, const Layout& lay, void* st, const Branches* br,
          size_t together) {
  const int dt = d->dtype, rx = d->round_x;
  const float slope = 0.1f;  // LRELU_SLOPE (dec.hpp:284, 322, 324)
  char* ws = static_cast<char*>(d->workspace);
  float* bias = reinterpret_cast<float*>(ws);
  void* slot[kSlots];
  for (int i = 0; i < kSlots; ++i)
    slot[i] = ws + lay.vec_bytes + static_cast<size_t>(i) * lay.slot_bytes;
  int rc = GSVK_OK;

  // x = lrelu(conv_pre(z) + b_pre + cond(ge)[:, 0], 0.1): the broadcast add of dec.hpp:275-279
  // folded into the bias, the stage-0 leaky_relu_io (dec.hpp:284) into the store. cond is a k = 1
  // convolution of one frame, i.e. a GEMV; b_pre enters as its residual, so one launch leaves
  // bias = (W_cond ge + b_cond) + b_pre in fp32.
  const float* pre_bias = d->pre_b;
  if (d->g_in) {
    if ((rc = gsvk_gemv_f16w(GSVK_F32, rx, d->ge, d->g_in, d->cond_w, d->cond_b, GSVK_ACT_NONE, 0.f,
                             d->pre_b, GSVK_F32, bias, d->c0, 1, d->c0, d->g_in, st)))
      return rc;
    pre_bias = bias;
  }
  size_t T = d->frames;
  if ((rc = gsvk_conv1d(dt, rx, d->z, T, d->pre_w, pre_bias, GSVK_CONV_EPI_LRELU, slope, nullptr,
                        nullptr, 0, slot[kX], T, d->c_z, d->c0, T, d->pre_k, 1, st)))
    return rc;

  for (size_t s = 0; s < d->n_stages; ++s) {
    const float next_slope = s + 1 < d->n_stages ? slope : 0.01f;
    if ((rc = issue_stage(dt, rx, d->stage[s], slot[kX], T, T, slot, next_slope, slot[kX], st, br,
                          together)))
      return rc;
    T *= d->stage[s].ups_u;
  }
  // out = tanh(conv_post(x))  (dec.hpp:343-344; conv_post has no bias)
  return gsvk_conv1d(dt, rx, slot[kX], T, d->post_w, nullptr, GSVK_CONV_EPI_TANH, 0.f, nullptr,
                     nullptr, 0, d->out, T, d->stage[d->n_stages - 1].c_out, 1, T, d->post_k, 1,
                     st);
}

// The eager form's side streams: two per device, created on its first eager call and kept for the
// process (default priority, non-blocking). Calls that overlap on one device share them; each
// call's own events order its launches, so sharing only serializes the calls' side work.
constexpr int kMaxDevices = 64;
int device_side_streams(hipStream_t (&side)[kSide]) {
  static std::mutex mu;
  static hipStream_t streams[kMaxDevices][kSide];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return GSVK_E_HIP;
  std::lock_guard<std::mutex> lock(mu);
  for (int i = 0; i < kSide; ++i) {
    if (!streams[dev][i] &&
        hipStreamCreateWithFlags(&streams[dev][i], hipStreamNonBlocking) != hipSuccess) {
      streams[dev][i] = nullptr;
      return GSVK_E_HIP;
    }
    side[i] = streams[dev][i];
  }
  return GSVK_OK;
}

// The fork and join events of an eager call, kept between calls (creating and destroying three on each
// call costs more host time than their records): taken for the issue of one call and given back after
// it, when every wait on them has been enqueued. At most kKeptEvents sets per device are kept.
struct EventSet {
  hipEvent_t fork = nullptr, join[kSide] = {};
};
constexpr size_t kKeptEvents = 8;
std::mutex events_mu;
std::vector<EventSet> events[kMaxDevices];

void destroy(EventSet& e) {
  if (e.fork) (void)hipEventDestroy(e.fork);
  for (int i = 0; i < kSide; ++i)
    if (e.join[i]) (void)hipEventDestroy(e.join[i]);
  e = EventSet{};
}

// Issues f(Branches) on the side streams with events of its own (fresh: none that are kept).
template <class F>
int with_branches(const hipStream_t* side, bool fresh, F f) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return GSVK_E_HIP;
  EventSet e;
  if (!fresh) {
    std::lock_guard<std::mutex> lock(events_mu);
    if (!events[dev].empty()) e = events[dev].back(), events[dev].pop_back();
  }
  int rc = GSVK_OK;
  if (!e.fork) {
    if (hipEventCreateWithFlags(&e.fork, hipEventDisableTiming) != hipSuccess) rc = GSVK_E_HIP;
    for (int i = 0; i < kSide && rc == GSVK_OK; ++i)
      if (hipEventCreateWithFlags(&e.join[i], hipEventDisableTiming) != hipSuccess) rc = GSVK_E_HIP;
  }
  if (rc == GSVK_OK) rc = f(Branches{side, e.fork, e.join});
  if (rc == GSVK_OK && !fresh) {
    std::lock_guard<std::mutex> lock(events_mu);
    if (events[dev].size() < kKeptEvents) {
      events[dev].push_back(e);
      return rc;
    }
  }
  destroy(e);  // (an event destroyed while its record is pending is released once that completes)
  return rc;
}

// Whether a call on st is being captured: its events are then the capture's, and not kept.
bool capturing(void* st) {
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(static_cast<hipStream_t>(st), &s) != hipSuccess ||
         s != hipStreamCaptureStatusNone;
}

}  // namespace

// The graph handle and its recorder live in t2s_decode_step.cpp.
__attribute__((visibility("hidden"))) int gsvk_record_graph_branches_(
    int (*issue_fn)(const void*, hipStream_t, const hipStream_t*, hipEvent_t, const hipEvent_t*),
    const void* ctx, int nside, int launches, gsvk_t2s_step** out);

extern "C" size_t gsvk_sovits_decoder_workspace_bytes(const gsvk_sovits_decoder_desc* desc) {
  Layout lay;
  return shapes(desc, &lay) == GSVK_OK ? lay.bytes : 0;
}

// A stage alone: its shapes, and the bytes of one of its 7 buffers (0: invalid).
static size_t stage_slot_bytes(int dtype, const gsvk_sovits_stage* S, size_t T) {
  if (!S || (dtype != GSVK_F32 && dtype != GSVK_F16)) return 0;
  if (T == 0 || S->c_in == 0 || S->c_out == 0 || S->ups_k == 0 || S->ups_u == 0) return 0;
  for (size_t j = 0; j < GSVK_SOVITS_RESBLOCKS; ++j)
    if (S->res_k[j] == 0) return 0;
  for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m)
    if (S->res_dil[m] == 0) return 0;
  const size_t esz = dtype == GSVK_F32 ? 4 : 2;
  if (T > SIZE_MAX / S->ups_u || T * S->ups_u > (SIZE_MAX / 2) / esz / kSlots / S->c_out) return 0;
  return round_up(T * S->ups_u * S->c_out * esz, kAlign);
}

extern "C" size_t gsvk_sovits_stage_workspace_bytes(int dtype, const gsvk_sovits_stage* stage,
                                                    size_t T) {
  return (kSlots - kY) * stage_slot_bytes(dtype, stage, T);
}

extern "C" int gsvk_sovits_stage_eager(int dtype, int round_x, const gsvk_sovits_stage* stage,
                                       const void* x, size_t ldx, size_t T, float slope_next,
                                       void* out, void* workspace, size_t workspace_bytes,
                                       void* const* side, void* stream) {
  if (!stage || !x || !out || !workspace || !stage->ups_w) return GSVK_E_NULL;
  for (size_t j = 0; j < GSVK_SOVITS_RESBLOCKS; ++j)
    for (size_t m = 0; m < GSVK_SOVITS_PAIRS; ++m)
      if (!stage->w1[j][m] || !stage->w2[j][m]) return GSVK_E_NULL;
  if (side && (!side[0] || !side[1])) return GSVK_E_NULL;
  if (dtype != GSVK_F32 && dtype != GSVK_F16) return GSVK_E_DTYPE;
  const size_t slot = stage_slot_bytes(dtype, stage, T);
  if (slot == 0 || workspace_bytes < (kSlots - kY) * slot) return GSVK_E_SIZE;
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return GSVK_E_ARG;
  void* buf[kSlots] = {};
  for (int i = kY; i < kSlots; ++i) buf[i] = static_cast<char*>(workspace) + (i - kY) * slot;
  if (!side || gsvk::conv1d_group_pays(stage->c_out, T * stage->ups_u))
    return issue_stage(dtype, round_x, *stage, x, ldx, T, buf, slope_next, out, stream, nullptr,
                       kTogetherEager);
  hipStream_t sd[kSide];
  for (int i = 0; i < kSide; ++i) sd[i] = static_cast<hipStream_t>(side[i]);
  return with_branches(sd, capturing(stream), [&](const Branches& br) {
    return issue_stage(dtype, round_x, *stage, x, ldx, T, buf, slope_next, out, stream, &br,
                       kTogetherEager);
  });
}

extern "C" int gsvk_sovits_decoder_eager(const gsvk_sovits_decoder_desc* desc, void* stream) {
  Layout lay;
  int rc = check_workspace(desc, &lay);
  if (rc) return rc;
  hipStream_t side[kSide];
  if ((rc = device_side_streams(side))) return rc;
  return with_branches(side, capturing(stream), [&](const Branches& br) {
    return issue(desc, lay, stream, &br, kTogetherEager);
  });
}

extern "C" int gsvk_sovits_decoder_create(const gsvk_sovits_decoder_desc* desc,
                                          gsvk_t2s_step** out) {
  if (!out) return GSVK_E_NULL;
  *out = nullptr;
  Layout lay;
  const int rc = check_workspace(desc, &lay);
  if (rc) return rc;
  struct Ctx {
    const gsvk_sovits_decoder_desc* d;
    Layout lay;
  } ctx{desc, lay};
  return gsvk_record_graph_branches_(
      [](const void* c, hipStream_t st, const hipStream_t* side, hipEvent_t fork,
         const hipEvent_t* join) {
        const Ctx* x = static_cast<const Ctx*>(c);
        const Branches br{side, fork, join};
        return issue(x->d, x->lay, st, &br, kTogetherGraph);
      },
      &ctx, GSVK_SOVITS_RESBLOCKS - 1, count_launches(desc), out);
}
