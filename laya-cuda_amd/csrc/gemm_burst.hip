// GEMM for few rows (batch-1 requests): whole K panels loaded at once, waves splitting K.
//
// At 16-2,000 rows a projection is bound by latency and by how fast each CU pulls its operands: an
// empty kernel costs 1.67 us per graph node, a cold weight panel another 0.9 us before its first
// byte, and a CU streams about 45 bytes per clock from L2 (64-row x 768 panels: +0.45 us per 48 KB,
// from 4, 8 or 16 waves alike, as long as an instruction covers whole 128-byte lines; 64-byte row
// segments run at half of that).  So a workgroup owns a BM x BN tile small enough that every CU has
// one, moves its operands with direct global-to-LDS loads in stages of SL 64-deep slabs, S stages
// (at K = 768 usually all of K) in flight before the first wait, and takes one barrier per stage, not
// per slab.  Its waves are WM x WN x KG: KG groups split the k-steps of a stage, so eight waves have
// work on a 32x32 tile; the groups' fp32 partial tiles are added in group order through LDS.
//
// 96 rows, weights cold in every cache, graph replays, against the 64-row tiles it replaced: QKV 6.6 ->
// 4.7 us, with RoPE 9.9 -> 4.9, GELU up 7.2 -> 5.7, 768 x 768 with fp32 output 4.1 -> 3.5.  A form without
// LDS (each wave loading its own MFMA fragments, 64-byte row segments) ran QKV in 6.0; touching the
// later slabs' lines ahead to pull them into L2 cost 0.1-0.5 us.
//
// LDS holds each slab as rows of 128 bytes, the 16-byte chunk index XOR-swizzled by (row / 2) % 8
// (conflict-free 16-byte reads of one chunk position of 16 consecutive rows).  The MFMA is
// v_mfma_f32_16x16x32 with the weights as its A operand: lane l supplies row l % 16 and the
// k 8 (l / 16) .. +7 of a step, and ends with output columns 4 (l / 16) .. +3 of row l % 16.
#include "gemm_burst.hpp"
#include "tiles.hpp"

namespace laya {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));

template <int BM, int BN, int SL, int S>
constexpr int burst_stage_bytes() { return (BM + BN) * 128 * SL; }
// LDS: the S stages, reused for the KG partial tiles, then the tile's bias.
template <int BM, int BN, int KG, int SL, int S>
constexpr int burst_lds() {
  const int stages = S * burst_stage_bytes<BM, BN, SL, S>(), parts = KG * BM * (BN + 4) * 4;
  return (stages > parts ? stages : parts) + BN * 4;
}

template <typename T, int BM, int BN, int WM, int WN, int KG, int SL, int S, Epi E>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_burst_kernel(GemmArgs a) {
  constexpr int NW = WM * WN * KG, NT = 64 * NW;
  constexpr int WTM = BM / WM, WTN = BN / WN, MB = WTM / 16, NB = WTN / 16;
  static_assert(MB >= 1 && NB >= 1 && WTM % 16 == 0 && WTN % 16 == 0, "16x16 MFMA blocks");
  constexpr int PITCH = BN + 4;  // floats per row of a partial tile: 16-byte rows, spread over the banks
  constexpr int STAGE = burst_stage_bytes<BM, BN, SL, S>();
  constexpr int GROUPS = (BM + BN) / 8 * SL;        // 1 KB loads (8 rows x 128 B) of a stage
  constexpr int NLD = (GROUPS + NW - 1) / NW;       // per wave; past the last, the last again
  static_assert((S - 1) * NLD < 64, "vmcnt range");
  typedef typename Vec8<T>::type T8;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float* const red = reinterpret_cast<float*>(smem_raw);  // [KG][BM][PITCH], after the main loop
  float* const sbias = reinterpret_cast<float*>(smem_raw + burst_lds<BM, BN, KG, SL, S>() - BN * 4);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tx, ty, z;
  tile_of_even(blockIdx.x, a.N / BN, (a.M + BM - 1) / BM, a.splits, &tx, &ty, &z);
  const int n0 = tx * BN, m0 = ty * BM;

  // Weight row of tile column n.  With RoPE, tiles narrower than a head hold 16 dims of a head and
  // the 16 dims 32 further on, so that both halves of every rotated pair are in one tile.
  auto column = [&](int n) {
    if constexpr (E == Epi::QKV_ROPE && BN == 32) return (n0 & ~63) + ((n0 & 32) >> 1) + (n & 15) + ((n & 16) << 1);
    else return n0 + n;
  };

  // This split's slabs and stages.
  const int slabs = a.K / 64;
  const int per = (slabs + a.splits - 1) / a.splits;
  const int kb = z * per, n = max(min(slabs, kb + per) - kb, 0);
  const int stages = (n + SL - 1) / SL;

  // Direct loads of a stage: group q of this wave is 8 rows of slab `slab` of the stage.
  const i32x4 rsA = buffer_resource(a.a, static_cast<unsigned>(static_cast<size_t>(a.M) * a.lda * 2));
  const i32x4 rsB = buffer_resource(a.b, static_cast<unsigned>(static_cast<size_t>(a.N) * a.ldb * 2));
  const unsigned lds_base = lds_address(smem_raw);
  constexpr int RG = (BM + BN) / 8;  // row groups of a slab: A's, then B's
  unsigned src[NLD];
#pragma unroll
  for (int q = 0; q < NLD; ++q) {
    const int g = min(wave + NW * q, GROUPS - 1), rg = g % RG, r = rg * 8 + (lane >> 3);
    const int ch = (lane & 7) ^ ((r >> 1) & 7);
    src[q] = r < BM ? (static_cast<unsigned>(min(m0 + r, a.M - 1)) * static_cast<unsigned>(a.lda) + ch * 8u) * 2u
                    : (static_cast<unsigned>(column(r - BM)) * static_cast<unsigned>(a.ldb) + ch * 8u) * 2u;
  }
  auto issue = [&](int stage, int buf) {
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      const int g = min(wave + NW * q, GROUPS - 1), rg = g % RG, slab = g / RG;
      const unsigned k = static_cast<unsigned>(kb + min(stage * SL + slab, n - 1)) * 128u;
      lds_load16_buffer(rg * 8 < BM ? rsA : rsB, src[q], k, lds_base + static_cast<unsigned>(buf * STAGE + g * 1024));
    }
  };

  float early_bias = 0.f;
  const bool with_bias = (E != Epi::F32 || a.splits == 1) && a.bias;
  if (with_bias && tid < BN) early_bias = a.bias[column(tid)];
  // RoPE: the positions of this thread's output rows.
  constexpr int kRopeIt = E == Epi::QKV_ROPE ? (BM * BN / 4 + NT - 1) / NT : 1;
  int pos[kRopeIt];
  if constexpr (E == Epi::QKV_ROPE) {
#pragma unroll
    for (int i = 0; i < kRopeIt; ++i) pos[i] = a.positions[min(m0 + (tid + i * NT) / (BN / 4), a.M - 1)];
  }

  const int kg = wave / (WM * WN), wm0 = (wave % (WM * WN)) / WN * WTM, wn0 = wave % WN * WTN;
  const int r16 = lane & 15, kq = lane >> 4;
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // k-steps (32 deep, two per slab) of a stage, dealt to the wave groups in turn.
  auto compute = [&](int buf, int steps) {
    constexpr int PS = (2 * SL + KG - 1) / KG;
#pragma unroll
    for (int u = 0; u < PS; ++u) {
      const int st = kg + u * KG;
      if (st < steps) {
        const T* const slab = reinterpret_cast<const T*>(smem_raw + buf * STAGE) + (st >> 1) * (BM + BN) * 64;
        T8 fa[MB], fb[NB];
        const int ch = (st & 1) * 4 + kq;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const int r = wm0 + i * 16 + r16;
          fa[i] = *reinterpret_cast<const T8*>(slab + r * 64 + ((ch ^ ((r >> 1) & 7)) << 3));
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int r = BM + wn0 + j * 16 + r16;
          fb[j] = *reinterpret_cast<const T8*>(slab + r * 64 + ((ch ^ ((r >> 1) & 7)) << 3));
        }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j) acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
      }
    }
  };

  // Every stage's barrier makes its loads visible and ends the reads of the stage before it, whose
  // buffer then takes stage it + S - 1.
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < stages) issue(s, s);
  int buf = 0;
  for (int it = 0; it < stages; ++it) {
    const int younger = min(it ? S - 2 : S - 1, stages - 1 - it);  // stages in flight behind this one
    if (S >= 4 && younger >= 3) publish_stage<waitcnt_vm(S >= 4 ? 3 * NLD : 0)>();
    else if (S >= 3 && younger >= 2) publish_stage<waitcnt_vm(S >= 3 ? 2 * NLD : 0)>();
    else if (S >= 2 && younger >= 1) publish_stage<waitcnt_vm(NLD)>();
    else publish_stage<waitcnt_vm(0)>();
    if (it && it + S - 1 < stages) issue(it + S - 1, buf ? buf - 1 : S - 1);
    compute(buf, 2 * min(SL, n - it * SL));
    buf = buf + 1 == S ? 0 : buf + 1;
  }
  f32x2 rcos[kRopeIt], rsin[kRopeIt];
  if constexpr (E == Epi::QKV_ROPE) {
#pragma unroll
    for (int i = 0; i < kRopeIt; ++i) {
      const size_t at = static_cast<size_t>(pos[i]) * 32 + (column((tid + i * NT) % (BN / 4) * 2) & 31);
      rcos[i] = *reinterpret_cast<const f32x2*>(a.rope_cos + at);
      rsin[i] = *reinterpret_cast<const f32x2*>(a.rope_sin + at);
    }
  }
  __syncthreads();  // the partial tiles reuse the stages

  float* const own = red + kg * BM * PITCH;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
      *reinterpret_cast<f32x4*>(own + (wm0 + i * 16 + r16) * PITCH + wn0 + j * 16 + 4 * kq) = acc[i][j];
  if (tid < BN) sbias[tid] = early_bias;
  __syncthreads();

  // Sum of the groups' partials of tile columns n, n + 1 of row r, in group order, and with the bias.
  auto total2 = [&](int r, int n) {
    f32x2 v = *reinterpret_cast<const f32x2*>(red + r * PITCH + n);
#pragma unroll
    for (int w = 1; w < KG; ++w) {
      const f32x2 t = *reinterpret_cast<const f32x2*>(red + (w * BM + r) * PITCH + n);
      v[0] = v[0] + t[0];
      v[1] = v[1] + t[1];
    }
    return v;
  };
  auto biased2 = [&](int r, int n) {
    f32x2 v = total2(r, n);
    if (with_bias) {
      v[0] = v[0] + sbias[n];
      v[1] = v[1] + sbias[n + 1];
    }
    return v;
  };
  typedef T T2 __attribute__((ext_vector_type(2)));
  auto half2 = [](float x, float y) {
    T2 h;
    h[0] = to_half<T>(x);
    h[1] = to_half<T>(y);
    return h;
  };

  if constexpr (E == Epi::QKV || E == Epi::QKV_ROPE) {
    const int part = n0 / a.width, head = (n0 - part * a.width) >> 6;  // a tile lies in one head (64 % BN == 0)
    auto dim = [&](int n) { return column(n) & 63; };
    if (part == 2) {
      // V^T [head][64][M]: a thread takes two tokens of one dim; M is a multiple of 8, so both are in or out.
      T* const vt = static_cast<T*>(a.vt) + static_cast<size_t>(head) * 64 * a.M;
      for (int c = tid; c < BM * BN / 2; c += NT) {
        const int r = (c % (BM / 2)) * 2, n = c / (BM / 2);
        float v0 = red[r * PITCH + n], v1 = red[(r + 1) * PITCH + n];
#pragma unroll
        for (int w = 1; w < KG; ++w) {
          v0 = v0 + red[(w * BM + r) * PITCH + n];
          v1 = v1 + red[(w * BM + r + 1) * PITCH + n];
        }
        if (with_bias) {
          v0 = v0 + sbias[n];
          v1 = v1 + sbias[n];
        }
        if (m0 + r < a.M) store_through(vt + static_cast<size_t>(dim(n)) * a.M + m0 + r, half2(v0, v1));
      }
      return;
    }
    T* const qk = static_cast<T*>(part == 0 ? a.q : a.k) + static_cast<size_t>(head) * a.M * 64;
    if constexpr (E == Epi::QKV) {
      for (int c = tid; c < BM * BN / 2; c += NT) {
        const int r = c / (BN / 2), n = (c % (BN / 2)) * 2, row = m0 + r;
        if (row >= a.M) continue;
        const f32x2 v = biased2(r, n);
        store_through(qk + static_cast<size_t>(row) * 64 + dim(n), half2(v[0], v[1]));
      }
    } else {
#pragma unroll
      for (int i = 0; i < kRopeIt; ++i) {
        const int c = tid + i * NT;
        const int r = c / (BN / 4), n = (c % (BN / 4)) * 2, row = m0 + r, d = dim(n);
        if (c >= BM * BN / 4 || row >= a.M) continue;
        const f32x2 cs = rcos[i], sn = rsin[i];
        const f32x2 lo = biased2(r, n), hi = biased2(r, n + BN / 2);
        T* const out = qk + static_cast<size_t>(row) * 64 + d;
        store_through(out, half2(lo[0] * cs[0] - hi[0] * sn[0], lo[1] * cs[1] - hi[1] * sn[1]));
        store_through(out + 32, half2(hi[0] * cs[0] + lo[0] * sn[0], hi[1] * cs[1] + lo[1] * sn[1]));
      }
    }
  } else if constexpr (E == Epi::GEGLU) {
    // Groups of 32 columns: 16 gate columns, then their 16 value columns.
    T* const out = static_cast<T*>(a.out);
    for (int c = tid; c < BM * BN / 4; c += NT) {
      const int r = c / (BN / 4), f = (c % (BN / 4)) * 2, row = m0 + r;
      if (row >= a.M) continue;
      const int n = (f / 16) * 32 + f % 16;
      const f32x2 g = biased2(r, n), v = biased2(r, n + 16);
      store_through(out + static_cast<long long>(row) * a.ldo + n0 / 2 + f,
                    half2(gelu16_rational(g[0]) * v[0], gelu16_rational(g[1]) * v[1]));
    }
  } else {
    for (int c = tid; c < BM * BN / 2; c += NT) {
      const int r = c / (BN / 2), n = (c % (BN / 2)) * 2, row = m0 + r;
      if (row >= a.M) continue;
      const f32x2 v = biased2(r, n);
      const long long at = static_cast<long long>(row) * a.ldo + n0 + n;
      if constexpr (E == Epi::F32) {
        store_through(static_cast<float*>(a.out) + z * a.split_stride + at, v);
      } else {
        auto act = [](float x) { return E == Epi::GELU ? gelu16(x) : E == Epi::RELU ? fmaxf(x, 0.f) : x; };
        store_through(static_cast<T*>(a.out) + at, half2(act(v[0]), act(v[1])));
      }
    }
  }
}

template <typename T, Epi E>
hipError_t launch_t(const GemmArgs& a, int variant, hipStream_t stream) {
  switch (variant) {
#define LAYA_BURST(ID, BM, BN, WM, WN, KG, SL, S)                                                   \
  case ID:                                                                                          \
    LAYA_LAUNCH((gemm_burst_kernel<T, BM, BN, WM, WN, KG, SL, S, E>),                               \
                dim3(a.N / BN * ((a.M + BM - 1) / BM) * a.splits), dim3(64 * WM * WN * KG),         \
                (burst_lds<BM, BN, KG, SL, S>()), stream, a);                                       \
    break;
    LAYA_BURST_TILES
#undef LAYA_BURST
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T, Epi E>
hipError_t set_lds() {
  hipError_t e = hipSuccess;
#define LAYA_BURST(ID, BM, BN, WM, WN, KG, SL, S)                                                     \
  if (e == hipSuccess)                                                                                \
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_burst_kernel<T, BM, BN, WM, WN, KG, SL, S, E>), \
                            hipFuncAttributeMaxDynamicSharedMemorySize, burst_lds<BM, BN, KG, SL, S>());
  LAYA_BURST_TILES
#undef LAYA_BURST
  return e;
}

template <typename F>
hipError_t for_epilogue(Epi epi, F&& f) {
  switch (epi) {
#define LAYA_EPI(E) case Epi::E: return f(std::integral_constant<Epi, Epi::E>());
    LAYA_EPI(F32) LAYA_EPI(HALF) LAYA_EPI(GELU) LAYA_EPI(QKV) LAYA_EPI(QKV_ROPE) LAYA_EPI(RELU) LAYA_EPI(GEGLU)
#undef LAYA_EPI
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t burst_prepare() {
  for (Epi epi : {Epi::F32, Epi::HALF, Epi::GELU, Epi::QKV, Epi::QKV_ROPE, Epi::RELU, Epi::GEGLU}) {
    const hipError_t e = for_epilogue(epi, [](auto c) {
      const hipError_t h = set_lds<f16, decltype(c)::value>();
      return h == hipSuccess ? set_lds<bf16, decltype(c)::value>() : h;
    });
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_burst(const GemmArgs& a, Epi epi, DType t, int variant, hipStream_t stream) {
  return for_epilogue(epi, [&](auto c) {
    return t == DType::F16 ? launch_t<f16, decltype(c)::value>(a, variant, stream)
                           : launch_t<bf16, decltype(c)::value>(a, variant, stream);
  });
}

}  // namespace laya
