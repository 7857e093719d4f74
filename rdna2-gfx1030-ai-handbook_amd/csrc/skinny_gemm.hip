// GEMM of few activation rows (M <= 16) against quantized weights on gfx950:
// out = A @ W^T with W [N, K] int8 (A int8, dequant epilogues of the INT8
// GEMM), fp8 e4m3fn / e5m2 or grouped INT4 in the nk layout (A fp16 / bf16).
//
// Such a call reads each weight byte once; what bounds it is how many bytes
// the chip keeps requested, and how many clocks a CU spends on each request.
//  * A workgroup of 8 waves owns 16 CT output columns and all rows. K is cut
//    into 128-element chunks; wave w takes chunks w, w + 8, ..., so the
//    workgroup reads every weight row front to back.
//  * Each wave copies its chunks (weights, activations, INT4 group
//    parameters) HBM -> LDS into a ring of its own, D chunks deep, with direct
//    copies: no barrier until the last one, and every wait is an exact count.
//    Loading the MFMA fragments into registers instead (16 bytes per lane,
//    neighbouring lanes in different rows) costs one request per lane, about
//    72 clocks per KB, whatever the depth in flight: M 16, N 3072, K 12288 fp8
//    took 19 us that way. A copy's neighbouring lanes read neighbouring bytes.
//  * A lane reads 16 weight bytes of one column per k-step group and puts them
//    into K order with two-input row exchanges (swap16 / swap32), so that the
//    activations are used as they lie in memory.
//  * LDS rows hold 16-byte chunks permuted by an XOR with the row (lds_row_xor).
//  * The 8 partial tiles are summed through LDS in wave order.
// fp8, N 12288, K 3072 (37.7 MB of weights, one box, rotated weight copies):
// 9.6 us at M 16 and 8.0 us at M <= 4 = 3.9 and 4.7 TB/s, against 40.9 us for
// the 128-row tiles of k_wd_gemm, whose 96 workgroups walk 24 stages with one
// stage of lookahead. What is left at M 16 is the copies of the activations
// (every workgroup reads all of them, about 33 clocks per KB): N 3072, K 12288
// 13.5 us against 9.1 us at M <= 4.
#include "qg_common.h"
#include "qg_epilogue.h"
#include "qg_internal.h"
#include "qg_w4_params.h"
#include "qg_wformat.h"

namespace qg {

namespace {

// RP: activation rows held in LDS (4, 8 or 16 >= M; fragment rows past RP
// repeat row RP - 1). G: INT4 group size. D: ring depth.
template <int FMT_, bool F16A_, int RP_, int CT_, int D_, int G_ = 128, int NW_ = 8>
struct SkinnyCfg {
  static constexpr int FMT = FMT_, RP = RP_, CT = CT_, D = D_, G = G_;
  static constexpr bool F16A = F16A_;
  static constexpr bool I8 = FMT == SK_I8, W4 = FMT >= SK_W4, UINT4 = FMT == SK_UINT4;
  static constexpr int NW = NW_, KS = 128;
  static constexpr int AROW = I8 ? KS : 2 * KS;           // LDS bytes of an activation row and chunk
  static constexpr int WROW = W4 ? KS / 2 : KS;           // of a weight row
  static constexpr int A_COPIES = RP * AROW / 1024, W_COPIES = 16 * CT * WROW / 1024;
  static constexpr int SPC = W4 ? KS / G : 0;             // groups per chunk
  static constexpr int COPIES = A_COPIES + W_COPIES;      // copies of a chunk
  static constexpr int W_AT = A_COPIES * 1024, STAGE = COPIES * 1024;
  static constexpr int PITCH = 16 * CT + 1;               // words per row of a partial tile
  static constexpr int RED = NW * 16 * PITCH * 4;
  static constexpr int PAR_AT = NW * D * STAGE;           // INT4 group parameters after the rings
  static constexpr int LDS = PAR_AT > RED ? PAR_AT : RED;
  static_assert(RP * AROW % 1024 == 0 && A_COPIES >= 1, "activation copies of whole waves");
  static_assert(D * COPIES < 64 && D >= 2 && D <= 4, "vmcnt range");
  static_assert(LDS <= 160 * 1024, "LDS per CU");
};

inline int skinny_par_bytes(const SkinnyArgs& p, int cols) {
  const int s = cols * w4_scale_pitch(p.ng, p.scale_f32);
  const int z = cols * w4_zero_pitch(p.ng, p.zw, p.flags & QG_W4_ZEROS_PACKED);
  return 4 * (((s + 63) & ~63) + ((z + 63) & ~63));
}

template <typename C>
__global__ __launch_bounds__(64 * C::NW) void k_skinny_gemm(SkinnyArgs p) {
#pragma clang fp contract(off)
  using acc_t = std::conditional_t<C::I8, i32x4, f32x4>;
  constexpr int CT = C::CT, D = C::D;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * 16 * CT;
  char* const ring = smem + wave * D * C::STAGE;
  const uint32_t ring_addr = lds_addr_of(ring);

  // ---- copy plan: per-lane byte offsets from the operand bases -------------
  // Copy i of the activations covers 1024 / AROW rows; lane l lands in 16-byte
  // slot l of it and fetches the chunk that the row's XOR stores there.
  constexpr int APC = 1024 / C::AROW, ASL = C::AROW / 16;  // rows per copy, slots per row
  constexpr int WPC = 1024 / C::WROW, WSL = C::WROW / 16;
  uint32_t aoff[C::A_COPIES], woff[C::W_COPIES];
  auto a_xor = [&](int row) __attribute__((always_inline)) { return lds_row_xor<C::AROW>(row); };
  auto w_xor = [&](int c) __attribute__((always_inline)) { return lds_row_xor<C::WROW>(c); };
  const int a_slot = lane % ASL, w_slot = lane % WSL;
  static_for<0, C::A_COPIES>([&](auto i) {
    const int row = APC * i + lane / ASL;
    aoff[i] = static_cast<uint32_t>(min(row, p.M - 1)) * static_cast<uint32_t>((C::I8 ? 1 : 2) * p.a_sm);
  });
  static_for<0, C::W_COPIES>([&](auto i) {
    const int c = WPC * i + lane / WSL;
    woff[i] = static_cast<uint32_t>(min(n0 + c, p.N - 1)) * static_cast<uint32_t>(p.w_sn);
  });
  const uint32_t a_end = static_cast<uint32_t>((C::I8 ? 1 : 2) * p.K) - 16;  // last 16 bytes of a row
  const uint32_t w_end = static_cast<uint32_t>(C::W4 ? p.K / 2 : p.K) - 16;
  const int chunks = (p.K + C::KS - 1) / C::KS;
  auto issue = [&](int c, int slot) __attribute__((always_inline)) {
    const uint32_t at = ring_addr + slot * C::STAGE;
    static_for<0, C::W_COPIES>([&](auto i) {
      const int r = (WPC * i + lane / WSL) & 15;
      const uint32_t k = static_cast<uint32_t>(C::WROW) * c + 16u * (w_slot ^ w_xor(r));
      dma16s_nt(p.w, woff[i] + min(k, w_end), at + C::W_AT + 1024 * i);
    });
    static_for<0, C::A_COPIES>([&](auto i) {
      const int r = APC * i + lane / ASL;
      const uint32_t k = static_cast<uint32_t>(C::AROW) * c + 16u * (a_slot ^ a_xor(r));
      dma16s(p.a, aoff[i] + min(k, a_end), at + 1024 * i);
    });
  };
  // INT4: the scales and zero points of the workgroup's columns are contiguous
  // (rows n0 .. of [N, ng] / [N, zw]): copied as dwords by all waves before
  // anything else. One copy per column, group and chunk instead (64 scattered
  // dwords) costs more clocks than the chunk's weights (M 16, N 4096, K 14336:
  // 19 us).
  const bool zpacked = C::UINT4 || (p.flags & QG_W4_ZEROS_PACKED);
  const bool sf32 = !C::UINT4 && p.scale_f32;
  const int sper = w4_scale_pitch(p.ng, sf32), zper = w4_zero_pitch(p.ng, p.zw, zpacked);
  const int spart = (16 * CT * sper + 63) & ~63;  // words of the scale part
  if constexpr (C::W4) {
    const uint32_t par_addr = lds_addr_of(smem + C::PAR_AT);
    // word e: word e % pitch of column e / pitch
    auto copy_words = [&](int pitch, auto copy) __attribute__((always_inline)) {
      for (int w0 = 64 * wave; w0 < 16 * CT * pitch; w0 += 64 * C::NW) {
        const int e = w0 + lane, cc = e / pitch;
        copy(static_cast<uint32_t>(min(n0 + cc, p.N - 1)), static_cast<uint32_t>(e - cc * pitch), 4u * w0);
      }
    };
    if (!sf32 && (p.N * p.ng & 1)) {  // the last scale is half a word
      copy_words(sper, [&](uint32_t n, uint32_t w, uint32_t to) __attribute__((always_inline)) {
        const W4Read r = w4_scale_read(n, p.N, p.ng, false, w);
        if (r.bytes == 2) dma2s(p.scales, r.offset, par_addr + to);
        else dma4s(p.scales, r.offset, par_addr + to);
      });
    } else {
      copy_words(sper, [&](uint32_t n, uint32_t w, uint32_t to) __attribute__((always_inline)) {
        dma4s(p.scales, w4_scale_read(n, p.N, p.ng, sf32, w).offset, par_addr + to);
      });
    }
    copy_words(zper, [&](uint32_t n, uint32_t w, uint32_t to) __attribute__((always_inline)) {
      dma4s(p.zeros, w4_zero_read(n, zpacked ? p.zw : p.ng, w).offset, par_addr + 4 * spart + to);
    });
  }

  acc_t acc[CT];
  f32x4 total[C::W4 ? CT : 1];
  static_for<0, CT>([&](auto t) {
    acc[t] = acc_t{0, 0, 0, 0};
    if constexpr (C::W4) total[t] = f32x4{0, 0, 0, 0};
  });
  const NibbleExpand<C::F16A> expand(C::W4 && !C::UINT4 && (p.flags & QG_W4_ORDER_HIGH));
  const uint32_t wxor = (C::W4 && !C::UINT4 && (p.flags & QG_W4_SIGNED_NIBBLES)) ? 0x88888888u : 0u;
  uint32_t one2 = C::F16A ? 0x3C003C00u : 0x3F803F80u;
  asm volatile("" : "+v"(one2));
  const i32x4 ones = {static_cast<int>(one2), static_cast<int>(one2), static_cast<int>(one2), static_cast<int>(one2)};
  const int arow = min(col, C::RP - 1);

  // tail: the chunk holds K elements past the end, which are zeroed (byte
  // formats; INT4 groups past the end get scale 0)
  auto compute = [&](int c, int slot, bool tail) __attribute__((always_inline)) {
    const char* const st = ring + slot * C::STAGE;
    auto a_frag = [&](int chunk) __attribute__((always_inline)) {
      return *reinterpret_cast<const i32x4*>(st + arow * C::AROW + 16 * (chunk ^ a_xor(arow)));
    };
    auto w_frag = [&](int t, int chunk) __attribute__((always_inline)) {
      return *reinterpret_cast<const i32x4*>(st + C::W_AT + (16 * t + col) * C::WROW + 16 * (chunk ^ w_xor(col)));
    };
    const i32x4 zero4 = {0, 0, 0, 0};
    if constexpr (C::I8) {
      static_for<0, 2>([&](auto u) {
        const bool in = !tail || C::KS * c + 64 * u + 16 * q < p.K;
        const i32x4 a = in ? a_frag(4 * u + q) : zero4;
        static_for<0, CT>([&](auto t) {
          acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, w_frag(t, 4 * u + q), acc[t], 0, 0, 0);
        });
      });
    } else if constexpr (!C::W4) {
      static_for<0, 2>([&](auto u) {
        i32x4 w[CT];
        static_for<0, CT>([&](auto t) {
          w[t] = w_frag(t, 4 * u + q);
          if (tail && C::KS * c + 64 * u + 16 * q >= p.K) w[t] = zero4;
          w[t] = k_order_bytes(w[t]);
        });
        static_for<0, 2>([&](auto h) {
          constexpr int H = decltype(h)::value;
          const bool in = !tail || C::KS * c + 64 * u + 32 * H + 8 * q < p.K;
          const i32x4 a = in ? a_frag(8 * u + 4 * H + q) : zero4;
          static_for<0, CT>([&](auto t) {
            const i32x4 b = fp8x8<C::F16A, C::FMT == SK_E5M2>(static_cast<uint32_t>(w[t][2 * H]),
                                                              static_cast<uint32_t>(w[t][2 * H + 1]));
            acc[t] = mfma_half<C::F16A>(a, b, acc[t]);
          });
        });
      });
    } else {
      constexpr int SPG = 4 / C::SPC;  // k-steps per group
      constexpr float MAGIC = C::F16A ? 256.0f : 128.0f, UNIT = C::F16A ? 4.0f : 1.0f;
      const char* const par = smem + C::PAR_AT;
      const uint32_t* const zpar = reinterpret_cast<const uint32_t*>(par) + spart;
      i32x4 w[CT];
      static_for<0, CT>([&](auto t) {
        w[t] = k_order_words(w_frag(t, q));
      });
      f32x4 asum = {0, 0, 0, 0};
      static_for<0, 4>([&](auto j) {
        constexpr int J = decltype(j)::value;
        if constexpr (J % SPG == 0) {
          asum = f32x4{0, 0, 0, 0};
          static_for<0, CT>([&](auto t) { acc[t] = acc_t{0, 0, 0, 0}; });
        }
        const i32x4 a = a_frag(4 * J + q);
        asum = mfma_half<C::F16A>(a, ones, asum);
        static_for<0, CT>([&](auto t) {
          acc[t] = mfma_half<C::F16A>(a, expand(static_cast<uint32_t>(w[t][J]) ^ wxor), acc[t]);
        });
        if constexpr (J % SPG == SPG - 1) {
          constexpr int gi = J / SPG;
          const int g = c * C::SPC + gi;
          static_for<0, CT>([&](auto t) {
            const int cc = 16 * t + col, gl = min(g, p.ng - 1);
            const uint32_t odd = static_cast<uint32_t>(min(n0 + cc, p.N - 1)) * p.ng & 1u;  // of the first bf16 scale
            const float sc = sf32 ? reinterpret_cast<const float*>(par)[cc * sper + gl]
                                  : bf16_to_f32(reinterpret_cast<const uint16_t*>(par)[cc * 2 * sper + odd + gl]);
            const float s = g < p.ng ? sc / UNIT : 0.0f;
            const uint32_t rz = zpacked ? zpar[cc * zper + (gl >> 3)] : zpar[cc * zper + gl];
            const int z = zpacked ? static_cast<int>((rz >> (4 * (gl & 7))) & 15u) : static_cast<int>(rz);
            const int zu = (!C::UINT4 && (p.flags & QG_W4_SIGNED_NIBBLES)) ? (zpacked ? (z ^ 8) : z + 8) : z;
            const float zb = MAGIC + UNIT * static_cast<float>(zu);
            static_for<0, 4>([&](auto e) {
              const float v = __builtin_fmaf(-zb, asum[int(e)], acc[t][int(e)]);
              total[t][int(e)] = __builtin_fmaf(s, v, total[t][int(e)]);
            });
          });
        }
      });
    }
  };

  // ---- this wave's chunks --------------------------------------------------
  const int n = chunks > wave ? (chunks - wave + C::NW - 1) / C::NW : 0;
  static_for<0, D>([&](auto d) {
    if (d < n) issue(wave + C::NW * d, d);
  });
  if constexpr (C::W4) {  // the parameters have landed (the chunks may still fly)
    if (n >= D) wait_vm_barrier<D * C::COPIES>();
    else wait_vm_barrier<0>();
  }
  const bool ragged = p.K % C::KS != 0;
  int slot = 0;
  for (int i = 0; i < n; ++i) {
    const int after = n - 1 - i;  // chunks issued after this one: min(after, D - 1)
    if (after >= D - 1) wait_vm<(D - 1) * C::COPIES>();
    else if (D > 2 && after == D - 2) wait_vm<(D > 2 ? D - 2 : 0) * C::COPIES>();
    else if (D > 3 && after == D - 3) wait_vm<(D > 3 ? D - 3 : 0) * C::COPIES>();
    else wait_vm<0>();
    const int c = wave + C::NW * i;
    if (!C::W4 && ragged && c == chunks - 1) compute(c, slot, true);
    else compute(c, slot, false);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's reads are done
    if (i + D < n) issue(c + C::NW * D, slot);
    slot = slot + 1 == D ? 0 : slot + 1;
  }

  // ---- partial tiles: row 4 q + i, column 16 t + col -------------------------
  uint32_t* const red = reinterpret_cast<uint32_t*>(smem);
  __syncthreads();  // every ring is done with
  static_for<0, CT>([&](auto t) {
    static_for<0, 4>([&](auto i) {
      uint32_t v;
      if constexpr (C::W4) v = __float_as_uint(total[t][int(i)]);
      else if constexpr (C::I8) v = static_cast<uint32_t>(acc[t][int(i)]);
      else v = __float_as_uint(acc[t][int(i)]);
      red[(wave * 16 + 4 * q + i) * C::PITCH + 16 * t + col] = v;
    });
  });
  __syncthreads();
  for (int e = threadIdx.x; e < C::RP * 16 * CT; e += 64 * C::NW) {
    const int row = e / (16 * CT), cc = e % (16 * CT);
    const int nn = n0 + cc;
    if (row >= p.M || nn >= p.N) continue;
    if constexpr (C::I8) {
      int v = static_cast<int>(red[row * C::PITCH + cc]);
#pragma unroll
      for (int w = 1; w < C::NW; ++w) v += static_cast<int>(red[(w * 16 + row) * C::PITCH + cc]);
      i8_store_out(p.i8, row, nn, v);
    } else {
      const int64_t idx = static_cast<int64_t>(row) * p.N + nn;
      float v = __uint_as_float(red[row * C::PITCH + cc]);
#pragma unroll
      for (int w = 1; w < C::NW; ++w) v = v + __uint_as_float(red[(w * 16 + row) * C::PITCH + cc]);
      if (!C::W4 && p.b_scale) v = v * p.b_scale[nn];
      if (p.bias) v = v + bias_value(load_bias_bits(p.bias, p.bias_dtype, nn), p.bias_dtype);
      if (p.out_dtype == QG_F32) store_elem<QG_F32>(p.out, idx, __float_as_uint(v));
      else if (p.out_dtype == QG_F16) store_elem<QG_F16>(p.out, idx, f32_to_f16(v));
      else store_elem<QG_BF16>(p.out, idx, f32_to_bf16(v));
    }
  }
}

template <typename C>
hipError_t launch_skinny_c(const SkinnyArgs& p, hipStream_t stream) {
  int lds = C::LDS;
  if constexpr (C::W4) {
    const int with_par = C::PAR_AT + skinny_par_bytes(p, 16 * C::CT);
    lds = with_par > lds ? with_par : lds;
  }
  hipLaunchKernelGGL(k_skinny_gemm<C>, dim3(ceil_div(p.N, 16 * C::CT)), dim3(64 * C::NW), lds, stream, p);
  return hipGetLastError();
}

constexpr int kCUs = 256;  // MI355X
constexpr int kMaxLds = 160 * 1024;

// Column tiles per workgroup: the copies a CU issues decide the time once the
// weights are in flight, ceil(workgroups / CUs) x (activation copies + CT x
// weight copies) of a chunk; the smallest CT among equals. fp8, M 16, K 3072:
// N 12288 13.2 / 12.2 / 9.6 us with 1 / 2 / 3 tiles (18 / 16 / 10 by this
// count), N 3072 5.3 / 6.3 / 7.7 us (6 / 8 / 10).
int skinny_tiles(int n, int a_copies, int w_copies, int max_tiles, const int* allowed, int count) {
  int best = allowed[0];
  long best_cost = -1;
  for (int i = 0; i < count && allowed[i] <= max_tiles; ++i) {
    const int ct = allowed[i];
    const long groups = ceil_div(n, 16 * ct);
    const long cost = (groups + kCUs - 1) / kCUs * (a_copies + ct * w_copies);
    if (best_cost < 0 || cost < best_cost) {
      best = ct;
      best_cost = cost;
    }
  }
  return best;
}

// Ring depth 2: the 8 waves of a workgroup keep 48 to 160 KB in flight, and
// depths 3 and 4 measured the same or slower (fewer workgroups per CU).
template <int FMT, bool F16A, int RP>
hipError_t launch_skinny_bytes(const SkinnyArgs& p, hipStream_t stream) {
  using C1 = SkinnyCfg<FMT, F16A, RP, 1, 2>;
  const int allowed[] = {1, 2, 3};
  switch (skinny_tiles(p.N, C1::A_COPIES, C1::W_COPIES, 3, allowed, 3)) {
    case 1: return launch_skinny_c<C1>(p, stream);
    case 2: return launch_skinny_c<SkinnyCfg<FMT, F16A, RP, 2, 2>>(p, stream);
    default: return launch_skinny_c<SkinnyCfg<FMT, F16A, RP, 3, 2>>(p, stream);
  }
}

template <int FMT, bool F16A>
hipError_t launch_skinny_fp8_rows(const SkinnyArgs& p, hipStream_t stream) {
  if (p.M <= 4) return launch_skinny_bytes<FMT, F16A, 4>(p, stream);
  if (p.M <= 8) return launch_skinny_bytes<FMT, F16A, 8>(p, stream);
  return launch_skinny_bytes<FMT, F16A, 16>(p, stream);
}

// INT4 column tiles: four pay only at 16 rows (uint4, N 14336, K 4096: 19 / 14
// / 17 / 12 us with 1 / 2 / 3 / 4), one or two below. The same rule holds for a
// short K (16 rows, N 14336, K 256: group 32 7.8 us against 10.5 with one tile,
// group 64, N 28672, K 512 10.1 against 12.5 with two). The parameters of K / G
// groups have to fit next to the rings.
template <typename C1>
int skinny_w4_tiles(const SkinnyArgs& p) {
  const int allowed[] = {1, 2, 4};
  int ct = skinny_tiles(p.N, C1::A_COPIES, C1::W_COPIES, C1::RP == 16 && C1::G != 32 ? 4 : 2, allowed, 3);
  while (ct > 1 && C1::RP * 4096 + ct * 16384 + skinny_par_bytes(p, 16 * ct) > kMaxLds) ct >>= 1;
  return ct;
}

template <int FMT, bool F16A, int RP, int G>
hipError_t launch_skinny_w4_rows(const SkinnyArgs& p, hipStream_t stream) {
  using C1 = SkinnyCfg<FMT, F16A, RP, 1, 2, G>;
  const int ct = skinny_w4_tiles<C1>(p);
  if (C1::PAR_AT + skinny_par_bytes(p, 16) > kMaxLds) return hipErrorInvalidValue;
  if constexpr (RP == 16 && G != 32) {
    if (ct == 4) return launch_skinny_c<SkinnyCfg<FMT, F16A, RP, 4, 2, G>>(p, stream);
  }
  if (ct == 2) return launch_skinny_c<SkinnyCfg<FMT, F16A, RP, 2, 2, G>>(p, stream);
  return launch_skinny_c<C1>(p, stream);
}

template <int FMT, bool F16A, int G>
hipError_t launch_skinny_w4_g(const SkinnyArgs& p, hipStream_t stream) {
  if (p.M <= 4) return launch_skinny_w4_rows<FMT, F16A, 4, G>(p, stream);
  if (p.M <= 8) return launch_skinny_w4_rows<FMT, F16A, 8, G>(p, stream);
  return launch_skinny_w4_rows<FMT, F16A, 16, G>(p, stream);
}

template <bool F16A>
hipError_t launch_skinny_w4_t(const SkinnyArgs& p, int group, hipStream_t stream) {
  switch (group) {
    case 128:
      if (!p.scale_f32 && p.flags == QG_W4_ZEROS_PACKED) return launch_skinny_w4_g<SK_UINT4, F16A, 128>(p, stream);
      return launch_skinny_w4_g<SK_W4, F16A, 128>(p, stream);
    case 64: return launch_skinny_w4_g<SK_W4, F16A, 64>(p, stream);
    default: return launch_skinny_w4_g<SK_W4, F16A, 32>(p, stream);
  }
}

}  // namespace

bool skinny_w4_applies(const W4Args& p) {
  if (p.M < 1 || p.M > kSkinnyMaxRows || (p.flags & QG_W4_LAYOUT_KN)) return false;
  if (((reinterpret_cast<uintptr_t>(p.scales) | reinterpret_cast<uintptr_t>(p.zeros)) & 3) != 0) return false;
  SkinnyArgs t{};
  t.flags = p.flags;
  t.ng = p.ng;
  t.zw = p.zw;
  t.scale_f32 = p.scale_f32;
  // one column tile next to the rings of 16 rows (8 waves x 2 chunks x 5 KB)
  return 80 * 1024 + skinny_par_bytes(t, 16) <= kMaxLds;
}

hipError_t launch_skinny_w4(const W4Args& p, hipStream_t stream) {
  if (!skinny_w4_applies(p)) return hipErrorInvalidValue;
  const SkinnyArgs t = skinny_args(p);
  return p.a_f16 ? launch_skinny_w4_t<true>(t, p.group, stream) : launch_skinny_w4_t<false>(t, p.group, stream);
}

hipError_t launch_skinny_fp8(const SkinnyArgs& p, bool f16a, bool e5, hipStream_t stream) {
  if (p.M < 1 || p.M > kSkinnyMaxRows || p.K % 16 != 0 || p.K < 16) return hipErrorInvalidValue;
  if (f16a) return e5 ? launch_skinny_fp8_rows<SK_E5M2, true>(p, stream) : launch_skinny_fp8_rows<SK_E4M3, true>(p, stream);
  return e5 ? launch_skinny_fp8_rows<SK_E5M2, false>(p, stream) : launch_skinny_fp8_rows<SK_E4M3, false>(p, stream);
}

hipError_t launch_skinny_i8(const I8GemmArgs& p, hipStream_t stream) {
  if (p.M < 1 || p.M > kSkinnyMaxRows || p.K % 16 != 0 || p.K < 16) return hipErrorInvalidValue;
  SkinnyArgs t{};
  t.a = p.a;
  t.a_sm = p.a_sm;
  t.w = p.w;
  t.w_sn = p.w_sn;
  t.M = p.M;
  t.N = p.N;
  t.K = p.K;
  t.i8 = p;
  return p.M <= 8 ? launch_skinny_bytes<SK_I8, false, 8>(t, stream) : launch_skinny_bytes<SK_I8, false, 16>(t, stream);
}

}  // namespace qg
