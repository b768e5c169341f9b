// gsvk_t2s_attn.hip — QKV projection, KV append and attention of one T2S decode layer in one launch,
// for few sequences.
//
// At small batches every launch of a decode layer is latency: the QKV GEMV, the key scan and the
// merge of its chunks move at most a few hundred kilobytes per CU, and each pays a launch, a
// round of loads and a write-back that the next one reads. A head of one sequence needs only its own
// 3 x 32 rows of W_qkv and its own 64-byte slices of the cached keys and values, so one workgroup
// per (sequence, head) does all of it:
//   x   = LN(z)                    (norm2 of the layer before; layer 0 reads x as it is)
//   q, k, v = W_qkv[its 96 rows] x + b       fp32
//   append k, v (rounded to fp16); out = softmax(q K^T / sqrt(32)) V
// The weights, z, the LayerNorm vectors and the first keys are all asked for before anything is
// waited for. The batch multiplies the reads of the weights (96 KiB per head and workgroup, from
// L2: the two heads that share the cache's 128-byte lines run on one XCD), which is why large batches
// keep the separate launches.
//
// Bound by latency: one layer's three launches (LN + QKV, attention, merge) took 4.9 + 6.6 + 3.2 us
// at one sequence and 300 keys, this one about 7; the line and both sides' times on the whole step
// stand at kFusedKeys in host/t2s_decode_step.cpp.
#include <cmath>

#include "gsvk_common.hpp"
#include "gsvk_t2s_attn.hpp"

namespace gsvk {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kHD = 32;             // head width
constexpr int kQWaves = 8;
constexpr int kQThreads = kQWaves * kWave;
constexpr int kTiles = 3 * kHD / 16;  // 16-row tiles of the head's q, k, v rows
constexpr int kQuarters = 4;          // K quarters of the projection
constexpr int kUnits = kTiles * kQuarters / kQWaves;  // (tile, quarter) units per wave
static_assert(kTiles * kQuarters % kQWaves == 0, "units per wave");
constexpr int kSlots = 4;           // key rounds in flight
constexpr int kKeysPerRound = 16 * kQWaves;

// Projection of S x 128 inputs (D = 128 S). Matrix-core operands: A = 16 rows of W x 32 k, B = the
// same 32 values of x in all 16 columns, so every column of the result holds the 16 dot products.
// Unit u = wave + 8 i is tile u % 6 (q, q, k, k, v, v) over quarter u / 6 of K.
template <int S, bool LN>
__global__ __launch_bounds__(kQThreads)
__attribute__((amdgpu_waves_per_eu(2))) void t2s_qkv_attn(T2sAttnArgs a) {
  constexpr int D = 128 * S;
  __shared__ __attribute__((aligned(16))) _Float16 xs[kQWaves][D];
  __shared__ f4v red[kQuarters][kTiles][4];
  __shared__ float qkv[3 * kHD];
  __shared__ float st_m[4 * kQWaves], st_l[4 * kQWaves], st_o[4 * kQWaves][kHD + 1];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r16 = lane & 15, grp = lane >> 4;
  // heads 2 p and 2 p + 1 on one XCD when there are 16 (blockIdx round-robin over 8 XCDs)
  const int hi = blockIdx.x % a.heads, b = blockIdx.x / a.heads;
  const int head = a.heads == 16 ? 2 * (hi & 7) + (hi >> 3) : hi;
  const int64_t pos = a.pos[b];

  // ---- every load that depends on nothing -------------------------------------------------------
  const bool on = 8 * lane < D;
  const size_t zc = static_cast<size_t>(b) * D + (on ? 8 * lane : 0);
  const u32x4 zraw = ld16<false>(static_cast<const uint16_t*>(a.z) + zc);
  u32x4 graw[2], braw[2];
  if constexpr (LN) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = (on ? 8 * lane : 0) + 4 * q;
      graw[q] = ld16<false>(a.ln_g ? a.ln_g + c : kOnes8);
      braw[q] = ld16<false>(a.ln_b ? a.ln_b + c : kZeros8);
    }
  }
  u32x4 w[kUnits][S];
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int u = wave + kQWaves * i, t = u % kTiles, kq = u / kTiles;
    const size_t row = static_cast<size_t>((t / 2) * D + head * kHD + (t & 1) * 16 + r16);
#pragma unroll
    for (int s = 0; s < S; ++s)
      w[i][s] = ld16<false>(a.wqkv + row * D + kq * (32 * S) + 32 * s + 8 * grp);
  }
  // output tid < 96 of the head: row part tid / 32, dim tid % 32
  const int orow = min(tid, 3 * kHD - 1);
  const float* bp = a.bqkv ? a.bqkv + (orow / kHD) * D + head * kHD + orow % kHD : kNegZeros8;
  const float bias = *bp;

  // Cached keys (the ones before the new token): lane holds dims 8 (lane & 3) .. + 7 of key
  // 128 r + 16 wave + lane / 4 in round r; past the end it rereads the last one with weight 0.
  const bool valid = pos >= 0 && pos < a.max_len;
  const int past = valid ? static_cast<int>(pos) : 0;
  const int rounds = (past + kKeysPerRound - 1) / kKeysPerRound;
  const int key0 = 16 * wave + (lane >> 2);
  const size_t seq = (static_cast<size_t>(b) * a.max_len) * D + head * kHD + 8 * (lane & 3);
  h8 kr[kSlots], vr[kSlots];
  auto kv_at = [&](int r) {
    return seq + static_cast<size_t>(max(0, min(key0 + kKeysPerRound * r, past - 1))) * D;
  };
  auto k_load = [&](int s, int r) {
    kr[s] = __builtin_bit_cast(h8, ld16<false>(static_cast<const uint16_t*>(a.kc) + kv_at(r)));
  };
  auto v_load = [&](int s, int r) {
    vr[s] = __builtin_bit_cast(h8, ld16<false>(static_cast<const uint16_t*>(a.vc) + kv_at(r)));
  };
#pragma unroll
  for (int s = 0; s < kSlots; ++s) k_load(s, s);
#pragma unroll
  for (int s = 0; s < kSlots; ++s) v_load(s, s);

  // ---- x, in this wave's own copy (its LDS accesses execute in order: no barrier) ----------------
  u32x4 xraw = zraw;
  if constexpr (LN) {
    float v[8];
    Store<GSVK_F16>::unpack(zraw, v);
    if (!on) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = 0.f;
    }
    const float mean =
        static_cast<float>(static_cast<double>(wave_sum(chunk_sum<8>(v))) * a.inv_n);
    const float sq = on ? chunk_sumsq<8>(v, mean) : 0.f;
    const float var = static_cast<float>(static_cast<double>(wave_sum(sq)) * a.inv_n);
    const float rstd = __builtin_amdgcn_rsqf(var + a.eps);
    const f4v g0 = __builtin_bit_cast(f4v, graw[0]), g1 = __builtin_bit_cast(f4v, graw[1]);
    const f4v b0 = __builtin_bit_cast(f4v, braw[0]), b1 = __builtin_bit_cast(f4v, braw[1]);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      v[k] = __builtin_fmaf((v[k] - mean) * rstd, k < 4 ? g0[k & 3] : g1[k & 3],
                            k < 4 ? b0[k & 3] : b1[k & 3]);
    xraw = Store<GSVK_F16>::pack(v);
    if (hi == 0 && wave == 0 && on) st16<false>(static_cast<uint16_t*>(a.x) + zc, xraw);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  if (on) *reinterpret_cast<u32x4*>(&xs[wave][8 * lane]) = xraw;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int u = wave + kQWaves * i, t = u % kTiles, kq = u / kTiles;
    f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const h8 xf = *reinterpret_cast<const h8*>(&xs[wave][kq * (32 * S) + 32 * s + 8 * grp]);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, w[i][s]), xf, acc, 0, 0, 0);
    }
    if (r16 == 0) red[kq][t][grp] = acc;  // rows 4 grp .. + 3
  }
  lds_barrier();
  if (tid < 3 * kHD) {
    const int t = tid / 16, e = tid & 15;
    float s = red[0][t][e / 4][e & 3];
#pragma unroll
    for (int q = 1; q < kQuarters; ++q) s += red[q][t][e / 4][e & 3];
    s += bias;
    if (tid >= kHD) {  // the new key and value as the cache holds them
      const uint16_t h = static_cast<uint16_t>(f2h(s));
      s = h2f(h);
      if (valid) {
        uint16_t* c = static_cast<uint16_t*>(tid < 2 * kHD ? a.kc : a.vc);
        c[(static_cast<size_t>(b) * a.max_len + static_cast<size_t>(pos)) * D + head * kHD +
          tid % kHD] = h;
      }
    }
    qkv[tid] = s;
  }
  lds_barrier();

  // ---- the keys -----------------------------------------------------------------------------------
  // Running maxima start at the lowest finite value, not -inf: every difference below is then a
  // number (or -inf, weight 0) without a test, and a sum without keys is 0.
  const int d0 = 8 * (lane & 3);
  float q[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = qkv[d0 + i];
  float m = -3.4028234663852886e38f, l = 0.f, o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = 0.f;
  if (wave == 0 && valid) {  // the new token: one four-lane group of wave 0, from the projection
    float d = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) d = __builtin_fmaf(q[i], qkv[kHD + d0 + i], d);
    d += dpp_f32<0xB1>(d);
    d += dpp_f32<0x4E>(d);
    if (lane < 4) {
      m = fmaxf(m, d * a.scale);
      l = __expf(d * a.scale - m);
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = l * qkv[2 * kHD + d0 + i];
    }
  }
  for (int r0 = 0; r0 < rounds; r0 += kSlots) {
    float sc[kSlots], mn = m;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      float d = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) d = __builtin_fmaf(q[i], static_cast<float>(kr[s][i]), d);
      d += dpp_f32<0xB1>(d);
      d += dpp_f32<0x4E>(d);
      sc[s] = key0 + kKeysPerRound * (r0 + s) < past ? d * a.scale : -INFINITY;
      mn = fmaxf(mn, sc[s]);
    }
    // the next rounds' keys (clamped past the last) travel while these are weighed
#pragma unroll
    for (int s = 0; s < kSlots; ++s) k_load(s, r0 + kSlots + s);
    const float corr = __expf(m - mn);
    m = mn;
    l *= corr;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] *= corr;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const float p = __expf(sc[s] - mn);
      l += p;
      if (key0 + kKeysPerRound * (r0 + s) < past) {  // (0 times an infinite reread value is NaN)
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = __builtin_fmaf(p, static_cast<float>(vr[s][i]), o[i]);
      }
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s) v_load(s, r0 + kSlots + s);
  }

  // ---- merge: the four key groups of each 16-lane row, then the 32 rows of the workgroup ----------
  auto rot_max = [](float v) {
    v = fmaxf(v, dpp_f32<0x124>(v));  // row_ror:4
    return fmaxf(v, dpp_f32<0x128>(v));
  };
  auto rot_sum = [](float v) {
    v += dpp_f32<0x124>(v);
    return v + dpp_f32<0x128>(v);
  };
  const float M = rot_max(m);
  const float f = __expf(m - M);
  l = rot_sum(l * f);
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = rot_sum(o[i] * f);
  const int st = 4 * wave + grp;
  if (r16 < 4) {
    if (r16 == 0) st_m[st] = M, st_l[st] = l;
#pragma unroll
    for (int i = 0; i < 8; ++i) st_o[st][d0 + i] = o[i];
  }
  lds_barrier();
  if (wave != 0) return;
  // wave 0: lane k % 32 weighs state k; then lane (half, dim) adds 16 states
  constexpr int kStates = 4 * kQWaves;
  static_assert(kStates == 32 && kHD == 32, "one state, one dim per lane of half a wave");
  const int half = lane >> 5, k = lane & 31;
  const float mk = st_m[k];
  float mx = rot_max(mk);
  mx = fmaxf(mx, dpp_f32<0xB1>(mx));
  mx = fmaxf(mx, dpp_f32<0x4E>(mx));   // of the 16-lane row
  mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
  const float e = __expf(mk - mx);
  const float L = wave_sum(half ? 0.f : st_l[k] * e);
  st_m[k] = e;  // (both halves write the same value; this wave reads it back in order)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float O = 0.f;
#pragma unroll
  for (int i = 0; i < kStates / 2; ++i)
    O = __builtin_fmaf(st_o[16 * half + i][k], st_m[16 * half + i], O);
  O += __shfl_xor(O, 32, kWave);
  const float y = L > 0.f ? O * (1.f / L) : __builtin_nanf("");  // L = 0: an invalid position
  if (half == 0)
    static_cast<uint16_t*>(a.out)[static_cast<size_t>(b) * D + head * kHD + k] =
        static_cast<uint16_t>(f2h(y));
  if (!valid && hi == 0 && lane == 0 && a.err) *a.err = 1;
}

template <int S>
void launch(const T2sAttnArgs& a, size_t batch, bool ln, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(batch * a.heads));
  if (ln) hipLaunchKernelGGL((t2s_qkv_attn<S, true>), grid, dim3(kQThreads), 0, st, a);
  else hipLaunchKernelGGL((t2s_qkv_attn<S, false>), grid, dim3(kQThreads), 0, st, a);
}

}  // namespace

__attribute__((visibility("hidden"))) bool t2s_qkv_attention_ok(const T2sAttnArgs& a, size_t batch,
                                                                size_t D) {
  if (D == 0 || D % 128 || D > 512 || static_cast<size_t>(a.heads) * kHD != D) return false;
  if (batch == 0 || a.max_len <= 0 || a.max_len > (1l << 30)) return false;
  if (!(a.eps >= 0.f) || !std::isfinite(a.eps)) return false;
  const void* al[] = {a.z, a.x, a.ln_g, a.ln_b, a.wqkv, a.kc, a.vc, a.out};
  for (const void* p : al)
    if (!aligned16(p)) return false;
  // what the separate launches refuse, and what they allow only because they run one after another
  const size_t rb = batch * D * 2, cb = batch * static_cast<size_t>(a.max_len) * D * 2;
  const size_t wb = 3 * D * D * 2;
  const struct { const void* p; size_t n; } out[] = {{a.x, rb}, {a.kc, cb}, {a.vc, cb}, {a.out, rb}};
  const struct { const void* p; size_t n; } in[] = {
      {a.z, rb}, {a.wqkv, wb}, {a.ln_g, D * 4}, {a.ln_b, D * 4}, {a.bqkv, 3 * D * 4},
      {a.pos, batch * 8}};
  for (int i = 0; i < 4; ++i) {
    if (!out[i].p) continue;
    for (const auto& r : in)
      if (overlaps(out[i].p, out[i].n, r.p, r.n)) return false;
    for (int j = i + 1; j < 4; ++j)
      if (overlaps(out[i].p, out[i].n, out[j].p, out[j].n)) return false;
  }
  return true;
}

__attribute__((visibility("hidden"))) int t2s_qkv_attention(const T2sAttnArgs& a, size_t batch,
                                                            size_t D, bool ln, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (D / 128) {
    case 1: launch<1>(a, batch, ln, st); break;
    case 2: launch<2>(a, batch, ln, st); break;
    case 3: launch<3>(a, batch, ln, st); break;
    default: launch<4>(a, batch, ln, st); break;
  }
  return launch_status();
}

}  // namespace gsvk
