// GEMM of a middling number of activation rows (17 to 2048, K from 1024)
// against quantized weights on gfx950: out = A @ W^T with W [N, K] int8 (A
// int8), fp8 or grouped INT4 in the nk layout (A fp16 / bf16).
//
// These grids fill the chip once or not at all, so a call lasts as long as one
// workgroup's K loop: what counts is the time per stage. A tile of BM x 128 and
// a K stage of 128 elements:
//  * every operand reaches LDS by direct copies in a ring of R slots, R - 1
//    stages ahead, with one barrier per stage (the copies of stage s + R - 1 go
//    into the slot that stage s - 1 left, which the barrier shows to be read).
//    With one stage of lookahead (k_wd_gemm, 128 rows) a stage takes 1.4 to 2.2
//    us, an L2 / HBM round trip; here, with tiles of 32 / 64 / 128 rows, fp8
//    0.50 / 0.67 / 1.42 us, INT4 0.64 / 0.95 / 1.60 us at group 128, 0.74 / 1.25
//    / 1.70 at 64, 0.97 / 1.35 at 32, int8 (64 rows) 0.50 us;
//  * 8 waves, fragments read half a stage ahead of their MFMAs. What is left
//    of a stage (N 3072, K 12288, M 64, parts removed): fp8 0.73 us, of which
//    0.60 without the copies (conversions) and 0.57 without the compute (40 to
//    50 clocks per KB copied); int8 0.57, 0.29 and 0.54 us;
//  * INT4 group scales and zero points of the workgroup's K range are decoded
//    to fp32 pairs [group][column] in LDS before the loop;
//  * where the tiles leave CUs idle, K is split over `splits` workgroups whose
//    partial tiles (fp32, int32) a second launch sums in order.
#include "qg_common.h"
#include "qg_epilogue.h"
#include "qg_internal.h"
#include "qg_wformat.h"

namespace qg {

namespace {

// NWM x 8 / NWM waves.
template <int FMT_, bool F16A_, int BM_, int R_, int G_ = 128, int NWM_ = 2>
struct MidCfg {
  static constexpr int FMT = FMT_, BM = BM_, R = R_, G = G_;
  static constexpr bool F16A = F16A_;
  static constexpr bool I8 = FMT == SK_I8, W4 = FMT >= SK_W4, UINT4 = FMT == SK_UINT4;
  static constexpr int BN = 128, KS = 128, NWM = NWM_, NWN = 8 / NWM, NW = 8;
  static constexpr int FM = BM / 16 / NWM, FN = BN / 16 / NWN;
  static constexpr int AROW = I8 ? KS : 2 * KS, WROW = W4 ? KS / 2 : KS;
  static constexpr int A_COPIES = BM * AROW / 1024 / NW, W_COPIES = BN * WROW / 1024 / NW;  // per wave and stage
  static constexpr int COPIES = A_COPIES + W_COPIES;
  static constexpr int W_AT = BM * AROW, STAGE = W_AT + BN * WROW;
  static constexpr int SPC = W4 ? KS / G : 0;  // groups per stage
  static constexpr int PAR_AT = R * STAGE;     // INT4: float2 (scale, zero term) [group][BN]
  static constexpr int GROUP_BYTES = 8 * BN;
  static_assert(BM * AROW % (1024 * NW) == 0 && BN * WROW % (1024 * NW) == 0 && A_COPIES >= 1, "whole copies per wave");
  static_assert(R >= 3 && (R - 1) * COPIES < 64, "ring");
  static_assert(PAR_AT <= 160 * 1024, "LDS per CU");
};

template <typename C>
__global__ __launch_bounds__(64 * C::NW, 1) void k_mid_gemm(MidArgs p) {
#pragma clang fp contract(off)
  using acc_t = std::conditional_t<C::I8, i32x4, f32x4>;
  constexpr int FM = C::FM, FN = C::FN, R = C::R;
  constexpr int AES = C::I8 ? 1 : 2;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const SkinnyArgs& o = p.op;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave / C::NWN, wc = wave % C::NWN;
  const int col = lane & 15, q = lane >> 4;
  // consecutive workgroups share the weight columns (and their L2 lines) of
  // one column tile; each of the 8 XCDs takes a contiguous range of tiles
  const int nbm = ceil_div(o.M, C::BM), nbn = ceil_div(o.N, C::BN);
  const int total_tiles = nbm * nbn;
  int bid = blockIdx.x;
  if ((total_tiles & 7) == 0) bid = (bid & 7) * (total_tiles >> 3) + (bid >> 3);
  const int m0 = (bid % nbm) * C::BM, n0 = (bid / nbm) * C::BN;
  // stages of this workgroup's K range
  const int all = ceil_div(o.K, C::KS);
  const int per = ceil_div(all, p.splits);
  const int first = min(static_cast<int>(blockIdx.y) * per, all);
  const int S = min(per, all - first);

  const uint32_t base = lds_addr_of(smem);
  constexpr int APC = 1024 / C::AROW, ASL = C::AROW / 16;
  constexpr int WPC = 1024 / C::WROW, WSL = C::WROW / 16;
  uint32_t aoff[C::A_COPIES], woff[C::W_COPIES], achunk, wchunk[C::W_COPIES];
  // copy i of wave w is copy w + 8 i of the stage; the XOR of a lane's row is
  // the same in every activation copy (8 copies are a multiple of its period)
  static_for<0, C::A_COPIES>([&](auto i) {
    const int row = APC * (wave + C::NW * i) + lane / ASL;
    aoff[i] = static_cast<uint32_t>(min(m0 + row, o.M - 1)) * static_cast<uint32_t>(AES * o.a_sm);
  });
  achunk = 16u * ((lane % ASL) ^ lds_row_xor<C::AROW>((APC * wave + lane / ASL) & 15));
  static_for<0, C::W_COPIES>([&](auto i) {
    const int c = WPC * (wave + C::NW * i) + lane / WSL;
    woff[i] = static_cast<uint32_t>(min(n0 + c, o.N - 1)) * static_cast<uint32_t>(o.w_sn);
    wchunk[i] = 16u * ((lane % WSL) ^ lds_row_xor<C::WROW>(c & 15));
  });
  const uint32_t a_end = static_cast<uint32_t>(AES * o.K) - 16;
  const uint32_t w_end = static_cast<uint32_t>(C::W4 ? o.K / 2 : o.K) - 16;
  // copy i (activations, then weights) of stage s into its slot
  auto copy = [&](auto i_c, int s, int slot) __attribute__((always_inline)) {
    constexpr int i = decltype(i_c)::value;
    const uint32_t at = base + slot * C::STAGE;
    const uint32_t c = first + s;
    if constexpr (i < C::A_COPIES)
      dma16s_free(o.a, aoff[i] + min(C::AROW * c + achunk, a_end), at + 1024 * (wave + C::NW * i));
    else
      dma16s_free(o.w, woff[i - C::A_COPIES] + min(C::WROW * c + wchunk[i - C::A_COPIES], w_end),
                  at + C::W_AT + 1024 * (wave + C::NW * (i - C::A_COPIES)));
  };

  static_for<0, R - 1>([&](auto d) {
    if (d < S) static_for<0, C::COPIES>([&](auto i) { copy(i, d, d); });
  });
  // ---- INT4 group parameters of the K range, decoded ------------------------
  constexpr float MAGIC = C::F16A ? 256.0f : 128.0f, UNIT = C::F16A ? 4.0f : 1.0f;
  const int g0 = first * C::SPC;
  if constexpr (C::W4) {
    const bool zpacked = C::UINT4 || (o.flags & QG_W4_ZEROS_PACKED);
    const bool sgn = !C::UINT4 && (o.flags & QG_W4_SIGNED_NIBBLES);
    const bool sf32 = !C::UINT4 && o.scale_f32;
    const int ngl = S * C::SPC;  // groups past ng: scale 0
    float2* const par = reinterpret_cast<float2*>(smem + C::PAR_AT);
    for (int e = threadIdx.x; e < C::BN * ngl; e += 64 * C::NW) {
      const int cc = e / ngl, gl = e - cc * ngl, g = min(g0 + gl, o.ng - 1);
      const uint32_t n = static_cast<uint32_t>(min(n0 + cc, o.N - 1));
      const uint32_t gi = n * o.ng + g;
      const float sc = sf32 ? static_cast<const float*>(o.scales)[gi]
                            : bf16_to_f32(static_cast<const uint16_t*>(o.scales)[gi]);
      const uint32_t rz = static_cast<const uint32_t*>(o.zeros)[zpacked ? n * o.zw + (g >> 3) : gi];
      const int z = zpacked ? static_cast<int>((rz >> (4 * (g & 7))) & 15u) : static_cast<int>(rz);
      const int zu = sgn ? (zpacked ? (z ^ 8) : z + 8) : z;
      par[gl * C::BN + cc] = make_float2(g0 + gl < o.ng ? sc / UNIT : 0.0f, MAGIC + UNIT * static_cast<float>(zu));
    }
  }

  acc_t acc[FM][FN];
  f32x4 total[C::W4 ? FM : 1][C::W4 ? FN : 1], asum[C::W4 ? FM : 1];
  static_for<0, FM>([&](auto f) {
    static_for<0, FN>([&](auto t) {
      acc[f][t] = acc_t{0, 0, 0, 0};
      if constexpr (C::W4) total[f][t] = f32x4{0, 0, 0, 0};
    });
  });
  const NibbleExpand<C::F16A> expand(C::W4 && !C::UINT4 && (o.flags & QG_W4_ORDER_HIGH));
  const uint32_t wxor = (C::W4 && !C::UINT4 && (o.flags & QG_W4_SIGNED_NIBBLES)) ? 0x88888888u : 0u;
  uint32_t one2 = C::F16A ? 0x3C003C00u : 0x3F803F80u;
  asm volatile("" : "+v"(one2));
  const i32x4 ones = {static_cast<int>(one2), static_cast<int>(one2), static_cast<int>(one2), static_cast<int>(one2)};
  const int axor = lds_row_xor<C::AROW>(col), wxr = lds_row_xor<C::WROW>(col);
  const int arow = (wr * 16 * FM + col) * C::AROW, wrow = C::W_AT + (wc * 16 * FN + col) * C::WROW;

  // Fragments of one half stage (64 K elements): two 32-element steps of
  // 2-byte activations, or one 64-element step of int8. The 16 weight bytes of
  // a lane cover a half stage of int8 / fp8 and the whole stage of INT4.
  constexpr int AC = C::I8 ? 1 : 2;
  struct Half {
    i32x4 a[FM][AC], w[FN];
  };
  auto read_half = [&](Half& x, int slot, auto h_c) __attribute__((always_inline)) {
    constexpr int H = decltype(h_c)::value;
    const char* const st = smem + slot * C::STAGE;
    if constexpr (!C::W4 || H == 0) {
      static_for<0, FN>([&](auto t) {
        const int chunk = C::W4 ? q : 4 * H + q;
        x.w[t] = *reinterpret_cast<const i32x4*>(st + wrow + t * 16 * C::WROW + 16 * (chunk ^ wxr));
      });
    }
    static_for<0, AC>([&](auto j) {
      static_for<0, FM>([&](auto f) {
        const int chunk = 4 * (AC * H + j) + q;
        x.a[f][j] = *reinterpret_cast<const i32x4*>(st + arow + f * 16 * C::AROW + 16 * (chunk ^ axor));
      });
    });
  };
  // Zeroes what lies past K (byte formats, the last stage of a ragged K).
  auto trim = [&](Half& x, int k0) __attribute__((always_inline)) {
    const i32x4 zero4 = {0, 0, 0, 0};
    static_for<0, FN>([&](auto t) {
      if (k0 + 16 * q >= o.K) x.w[t] = zero4;
    });
    static_for<0, AC>([&](auto j) {
      static_for<0, FM>([&](auto f) {
        if (k0 + (C::I8 ? 16 * q : 32 * j + 8 * q) >= o.K) x.a[f][j] = zero4;
      });
    });
  };
  // MFMAs of half H of stage s from x (INT4: weights in w4), with `copies`
  // called after each group.
  auto mfma_half_stage = [&](const Half& x, const i32x4 (&w4)[FN], int s, auto h_c, auto&& copies)
      __attribute__((always_inline)) {
    constexpr int H = decltype(h_c)::value;
    if constexpr (C::I8) {
      static_for<0, FM>([&](auto f) {
        static_for<0, FN>([&](auto t) {
          acc[f][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.a[f][0], x.w[t], acc[f][t], 0, 0, 0);
        });
        copies(f, std::integral_constant<int, FM>{});
      });
    } else {
      i32x4 wk[FN];
      if constexpr (!C::W4) static_for<0, FN>([&](auto t) { wk[t] = k_order_bytes(x.w[t]); });
      static_for<0, 2>([&](auto j) {
        constexpr int J = 2 * H + decltype(j)::value;  // step of the stage
        constexpr int SPG = C::W4 ? 4 / (C::W4 ? C::SPC : 1) : 4;
        i32x4 b[FN];
        static_for<0, FN>([&](auto t) {
          if constexpr (C::W4) b[t] = expand(static_cast<uint32_t>(w4[t][J]) ^ wxor);
          else b[t] = fp8x8<C::F16A, C::FMT == SK_E5M2>(static_cast<uint32_t>(wk[t][2 * int(j)]),
                                                        static_cast<uint32_t>(wk[t][2 * int(j) + 1]));
        });
        if constexpr (C::W4 && J % SPG == 0) {
          static_for<0, FM>([&](auto f) {
            asum[f] = f32x4{0, 0, 0, 0};
            static_for<0, FN>([&](auto t) { acc[f][t] = acc_t{0, 0, 0, 0}; });
          });
        }
        static_for<0, FM>([&](auto f) {
          if constexpr (C::W4) asum[f] = mfma_half<C::F16A>(x.a[f][j], ones, asum[f]);
          static_for<0, FN>([&](auto t) { acc[f][t] = mfma_half<C::F16A>(x.a[f][j], b[t], acc[f][t]); });
          copies(std::integral_constant<int, FM * int(j) + int(f)>{}, std::integral_constant<int, 2 * FM>{});
        });
        if constexpr (C::W4 && J % SPG == SPG - 1) {
          constexpr int gi = J / SPG;
          const float2* const par =
              reinterpret_cast<const float2*>(smem + C::PAR_AT) + (s * C::SPC + gi) * C::BN + wc * 16 * FN + col;
          static_for<0, FN>([&](auto t) {
            const float2 sz = par[16 * t];
            static_for<0, FM>([&](auto f) {
              static_for<0, 4>([&](auto e) {
                const float v = __builtin_fmaf(-sz.y, asum[f][int(e)], acc[f][t][int(e)]);
                total[f][t][int(e)] = __builtin_fmaf(sz.x, v, total[f][t][int(e)]);
              });
            });
          });
        }
      });
    }
  };

  // ---- main loop ------------------------------------------------------------
  // Top of stage s: stage s + 1 has landed everywhere and every wave has read
  // stage s - 1, whose slot takes stage s + R - 1; its copies are spread over
  // the MFMAs (a wave that issues a copy waits until the CU takes it, about 28
  // clocks per copy and wave). Half 1 of stage s is read under the MFMAs of
  // half 0, half 0 of stage s + 1 under those of half 1.
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  const bool ragged = !C::W4 && o.K % C::KS != 0;
  if (S > 0) {
    Half x0, x1;
    if (S > 1) wait_vm_barrier<(R - 2) * C::COPIES>();
    else wait_vm_barrier<0>();
    // fewer than R - 1 stages: the count above waits for nothing, so drain
    if (S < R - 1) wait_vm_barrier<0>();
    read_half(x0, 0, H0{});
    int slot = 0;
    for (int s = 0; s < S; ++s) {
      const int after = S - 2 - s;  // stages after s + 1, at most R - 3 of them issued
      if (after >= R - 3) wait_vm_barrier<(R - 3) * C::COPIES>();
      else wait_vm_barrier<0>();
      const bool fill = s + R - 1 < S;
      const int into = slot == 0 ? R - 1 : slot - 1;
      const int next = slot + 1 == R ? 0 : slot + 1;
      const bool last = ragged && first + s == all - 1;
      // copies [from, to) of COPIES for group g of n of half H
      auto spread = [&](auto h_c) __attribute__((always_inline)) {
        return [&, h_c](auto g_c, auto n_c) __attribute__((always_inline)) {
          constexpr int H = decltype(h_c)::value, g = decltype(g_c)::value, n = decltype(n_c)::value;
          constexpr int a = (H * n + g) * C::COPIES / (2 * n), b = (H * n + g + 1) * C::COPIES / (2 * n);
          if constexpr (b > a) {
            if (fill) static_for<a, b>([&](auto i) { copy(i, s + R - 1, into); });
          }
          __builtin_amdgcn_sched_barrier(0);
        };
      };
      read_half(x1, slot, H1{});
      __builtin_amdgcn_sched_barrier(0);
      i32x4 w4[FN];
      if constexpr (C::W4) static_for<0, FN>([&](auto t) { w4[t] = k_order_words(x0.w[t]); });
      if (last) trim(x0, C::KS * (first + s));
      mfma_half_stage(x0, w4, s, H0{}, spread(H0{}));
      if (s + 1 < S) read_half(x0, next, H0{});
      __builtin_amdgcn_sched_barrier(0);
      if (last) trim(x1, C::KS * (first + s) + 64);
      mfma_half_stage(x1, w4, s, H1{}, spread(H1{}));
      slot = next;
    }
  }

  // ---- INT4: elements that are not finite ------------------------------------
  // The loop sums a (MAGIC + UNIT u) and takes the zero point's share off each
  // group's sum, which turns an infinite activation, or a sum past fp32's range,
  // into NaN in every column. Such elements are summed again with the weights
  // u - z themselves, the products that the dequantized weights give (finite
  // elements keep their bits; the loop above is as it was without this).
  if constexpr (C::W4) {
    float off = 0.0f;  // NaN if some element of the lane is not finite
    static_for<0, FM>([&](auto f) {
      static_for<0, FN>([&](auto t) {
        static_for<0, 4>([&](auto e) { off = __builtin_fmaf(total[f][t][int(e)], 0.0f, off); });
      });
    });
    if (__builtin_expect(__any(off != 0.0f), 0)) static_for<0, FM>([&](auto f) {
      static_for<0, FN>([&](auto t) {
        bool lost[4];
        static_for<0, 4>([&](auto e) { lost[int(e)] = !(fabsf(total[f][t][int(e)]) < __builtin_inff()); });
        if (!__any(lost[0] || lost[1] || lost[2] || lost[3])) return;
        constexpr int STEPS = C::G / 32;  // of a group
        const int cc = wc * 16 * FN + 16 * t + col;
        const char* const ar = static_cast<const char*>(o.a) +
                               2 * static_cast<int64_t>(min(m0 + (wr * FM + f) * 16 + col, o.M - 1)) * o.a_sm;
        const uint32_t* const wr32 = reinterpret_cast<const uint32_t*>(static_cast<const char*>(o.w) +
                                                                       min(n0 + cc, o.N - 1) * o.w_sn);
        const float2* const par = reinterpret_cast<const float2*>(smem + C::PAR_AT) + cc;
        const int groups = min(S * C::SPC, o.ng - g0);
        f32x4 again = {0, 0, 0, 0};
        for (int g = 0; g < groups; ++g) {
          const float2 sz = par[g * C::BN];
          f32x4 sum = {0, 0, 0, 0};
          static_for<0, STEPS>([&](auto j) {
            const int step = (g0 + g) * STEPS + j;
            const i32x4 a = *reinterpret_cast<const i32x4*>(ar + 64 * step + 16 * q);
            i32x4 b = expand(wr32[4 * step + q] ^ wxor);
            static_for<0, 4>([&](auto i) {
              const uint32_t x = static_cast<uint32_t>(b[int(i)]);
              const uint16_t lo = static_cast<uint16_t>(x), hi = static_cast<uint16_t>(x >> 16);
              uint32_t l, h;  // u - z (times UNIT), exact
              if constexpr (C::F16A) {
                l = f32_to_f16(f16_to_f32(lo) - sz.y);
                h = f32_to_f16(f16_to_f32(hi) - sz.y);
              } else {
                l = f32_to_bf16(bf16_to_f32(lo) - sz.y);
                h = f32_to_bf16(bf16_to_f32(hi) - sz.y);
              }
              b[int(i)] = static_cast<int>(l | h << 16);
            });
            sum = mfma_half<C::F16A>(a, b, sum);
          });
          static_for<0, 4>([&](auto e) { again[int(e)] = __builtin_fmaf(sz.x, sum[int(e)], again[int(e)]); });
        }
        static_for<0, 4>([&](auto e) { total[f][t][int(e)] = lost[int(e)] ? again[int(e)] : total[f][t][int(e)]; });
      });
    });
  }

  // ---- output: row 4 q + e of block f, column col of block t -----------------
  static_for<0, FN>([&](auto t) {
    const int nn = n0 + wc * 16 * FN + 16 * t + col;
    if (nn >= o.N) return;
    float ws = 1.0f, bv = 0.0f;
    if constexpr (!C::I8) {
      if (p.splits == 1) {
        if (!C::W4 && o.b_scale) ws = o.b_scale[nn];
        if (o.bias) bv = bias_value(load_bias_bits(o.bias, o.bias_dtype, nn), o.bias_dtype);
      }
    }
    static_for<0, FM>([&](auto f) {
      static_for<0, 4>([&](auto e) {
        const int row = m0 + wr * 16 * FM + 16 * f + 4 * q + e;
        if (row >= o.M) return;
        const int64_t idx = static_cast<int64_t>(row) * o.N + nn;
        const int64_t at = static_cast<int64_t>(blockIdx.y) * o.M * o.N + idx;
        if constexpr (C::I8) {
          if (p.splits > 1) static_cast<int*>(p.partial)[at] = acc[f][t][int(e)];
          else i8_store_out(o.i8, row, nn, acc[f][t][int(e)]);
        } else {
          float v;
          if constexpr (C::W4) v = total[f][t][int(e)];
          else v = acc[f][t][int(e)];
          if (p.splits > 1) {
            static_cast<float*>(p.partial)[at] = v;
          } else {
            if (!C::W4 && o.b_scale) v = v * ws;
            if (o.bias) v = v + bv;
            if (o.out_dtype == QG_F32) store_elem<QG_F32>(o.out, idx, __float_as_uint(v));
            else if (o.out_dtype == QG_F16) store_elem<QG_F16>(o.out, idx, f32_to_f16(v));
            else store_elem<QG_BF16>(o.out, idx, f32_to_bf16(v));
          }
        }
      });
    });
  });
}

// Sums the partial tiles in split order and applies the epilogue: one row per
// blockIdx.y, VEC columns per thread.
template <bool I8, int VEC>
__global__ __launch_bounds__(256) void k_mid_reduce(MidArgs p) {
#pragma clang fp contract(off)
  const SkinnyArgs& o = p.op;
  const int nn = (blockIdx.x * 256 + threadIdx.x) * VEC;
  if (nn >= o.N) return;
  const int row = blockIdx.y;
  const int64_t total = static_cast<int64_t>(o.M) * o.N, at = static_cast<int64_t>(row) * o.N + nn;
  typedef uint32_t vec_t __attribute__((ext_vector_type(VEC)));
  const uint32_t* const src = static_cast<const uint32_t*>(p.partial) + at;
  vec_t x = *reinterpret_cast<const vec_t*>(src);
  for (int s = 1; s < p.splits; ++s) {
    const vec_t y = *reinterpret_cast<const vec_t*>(src + s * total);
    static_for<0, VEC>([&](auto e) {
      if constexpr (I8) x[int(e)] += y[int(e)];
      else x[int(e)] = __float_as_uint(__uint_as_float(x[int(e)]) + __uint_as_float(y[int(e)]));
    });
  }
  static_for<0, VEC>([&](auto e) {
    const int n = nn + e;
    const uint32_t bits = x[int(e)];
    if constexpr (I8) {
      i8_store_out(o.i8, row, n, static_cast<int>(bits));
    } else {
      float v = __uint_as_float(bits);
      if (o.b_scale) v = v * o.b_scale[n];
      if (o.bias) v = v + bias_value(load_bias_bits(o.bias, o.bias_dtype, n), o.bias_dtype);
      const int64_t i = at + e;
      if (o.out_dtype == QG_F32) store_elem<QG_F32>(o.out, i, __float_as_uint(v));
      else if (o.out_dtype == QG_F16) store_elem<QG_F16>(o.out, i, f32_to_f16(v));
      else store_elem<QG_BF16>(o.out, i, f32_to_bf16(v));
    }
  });
}

constexpr int kCUs = 256;  // MI355X
constexpr int kMaxLds = 160 * 1024;

template <typename C>
hipError_t launch_mid_c(const MidArgs& p, hipStream_t stream) {
  const int tiles = ceil_div(p.op.M, C::BM) * ceil_div(p.op.N, C::BN);
  int lds = C::PAR_AT;
  if constexpr (C::W4) lds += ceil_div(ceil_div(p.op.K, C::KS), p.splits) * C::SPC * C::GROUP_BYTES;
  if (lds > kMaxLds) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mid_gemm<C>, dim3(tiles, p.splits), dim3(64 * C::NW), lds, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.splits == 1) return e;
  if (p.op.N % 4 == 0)
    hipLaunchKernelGGL((k_mid_reduce<C::I8, 4>), dim3(ceil_div(p.op.N, 1024), p.op.M), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((k_mid_reduce<C::I8, 1>), dim3(ceil_div(p.op.N, 256), p.op.M), dim3(256), 0, stream, p);
  return hipGetLastError();
}

// Wave grids: 1 x 8 expands every weight once (fp8 N 3072, K 3072, M 64: 15.5
// against 19.1 us for 2 x 4 with 32-row tiles); int8 has nothing to expand and
// 2 x 4 reads fewer LDS bytes, as do the 128-row INT4 tiles, where 1 x 8 spills
// (57 against 97 us at M 1024, N = K = 4096). Ring depths: what LDS holds.
template <int FMT, bool F16A, int G>
hipError_t launch_mid_w4(const MidArgs& p, int bm, hipStream_t stream) {
  if (bm == 32) return launch_mid_c<MidCfg<FMT, F16A, 32, 4, G, 1>>(p, stream);
  if (bm == 64) return launch_mid_c<MidCfg<FMT, F16A, 64, G == 128 ? 4 : 3, G, 1>>(p, stream);
  if constexpr (G != 32) {
    if (bm == 128) return launch_mid_c<MidCfg<FMT, F16A, 128, 3, G, 2>>(p, stream);
  }
  return hipErrorInvalidValue;
}

template <int FMT, bool F16A>
hipError_t launch_mid_fp8_t(const MidArgs& p, int bm, hipStream_t stream) {
  if (bm == 32) return launch_mid_c<MidCfg<FMT, F16A, 32, 4, 128, 1>>(p, stream);
  if (bm == 64) return launch_mid_c<MidCfg<FMT, F16A, 64, 4, 128, 1>>(p, stream);
  if (bm == 128) return launch_mid_c<MidCfg<FMT, F16A, 128, 3, 128, 1>>(p, stream);
  return hipErrorInvalidValue;
}

template <bool F16A>
hipError_t launch_mid_w4_t(const MidArgs& p, int group, int bm, hipStream_t stream) {
  switch (group) {
    case 128:
      if (!p.op.scale_f32 && p.op.flags == QG_W4_ZEROS_PACKED) return launch_mid_w4<SK_UINT4, F16A, 128>(p, bm, stream);
      return launch_mid_w4<SK_W4, F16A, 128>(p, bm, stream);
    case 64: return launch_mid_w4<SK_W4, F16A, 64>(p, bm, stream);
    default: return launch_mid_w4<SK_W4, F16A, 32>(p, bm, stream);
  }
}

}  // namespace

// Time model (us) behind the choice of tile and split, from a sweep over M 32
// to 1024 and (N, K) of 1024 x 4096 to 12288 x 3072 and 3072 x 12288 on one
// box, which it meets within about 10 % (over 840 calls, M 17 to 2048, other
// boxes and weights from HBM take 1.1 to 1.35 times as long, tiles and splits
// alike): 3.5 us plus the stages of one
// workgroup times the rounds of 256 workgroups times the time of a stage
// (128 K elements; 15 % more where rounds overlap); a split adds 2.5 us and
// its partial tiles at 4 TB/s. A split has to win by 10 %, and its partial tiles
// to fit in `room` bytes.
MidPlan plan_mid(int kind, int group, int64_t m, int64_t n, int64_t k, size_t room) {
  MidPlan best{0, 1, 0.0};
  if (m <= kSkinnyMaxRows || m > kMidMaxRows || n < 1 || k < kMidMinK) return best;
  struct Tile {
    int bm;
    double stage_us;
    int ring_kb;
  };
  static const Tile fp8[] = {{32, 0.50, 96}, {64, 0.67, 128}, {128, 1.42, 144}};
  static const Tile i8[] = {{64, 0.50, 144}};
  static const Tile g128[] = {{32, 0.64, 64}, {64, 0.95, 96}, {128, 1.60, 120}};
  static const Tile g64[] = {{32, 0.74, 64}, {64, 1.25, 72}, {128, 1.70, 120}};
  static const Tile g32[] = {{32, 0.97, 64}, {64, 1.35, 72}};
  const Tile* tiles = kind == MID_FP8 ? fp8 : kind == MID_I8 ? i8 : group == 128 ? g128 : group == 64 ? g64 : g32;
  const int count = kind == MID_I8 ? 1 : (kind == MID_W4 && group == 32) ? 2 : 3;
  const int64_t stages = (k + 127) / 128;
  for (int splits = 1; splits <= 8; splits *= 2) {
    if (splits > 1 && (m > 1024 || stages < 4 * splits || splits * m * n * 4 > (int64_t(256) << 20) ||
                       mid_partial_bytes(splits, m, n) > room))
      break;
    for (int i = 0; i < count; ++i) {
      const int64_t per = (stages + splits - 1) / splits;
      if (kind == MID_W4 && tiles[i].ring_kb * 1024 + per * (128 / group) * 1024 > kMaxLds) continue;
      const int64_t wgs = ((m + tiles[i].bm - 1) / tiles[i].bm) * ((n + 127) / 128) * splits;
      const int64_t rounds = (wgs + kCUs - 1) / kCUs;
      double us = 3.5 + rounds * per * tiles[i].stage_us * (rounds > 1 ? 1.15 : 1.0);
      if (splits > 1) us += 2.5 + (splits + 0.5) * m * n * 4 / 4.0e6;
      const double bar = best.splits < splits && best.bm != 0 ? 0.9 * best.us : best.us;
      if (best.bm == 0 || us < bar) best = MidPlan{tiles[i].bm, splits, us};
    }
  }
  return best;
}

hipError_t launch_mid_fp8(const MidArgs& p, int bm, bool f16a, bool e5, hipStream_t stream) {
  if (p.op.K % 16 != 0 || p.splits < 1) return hipErrorInvalidValue;
  if (f16a) return e5 ? launch_mid_fp8_t<SK_E5M2, true>(p, bm, stream) : launch_mid_fp8_t<SK_E4M3, true>(p, bm, stream);
  return e5 ? launch_mid_fp8_t<SK_E5M2, false>(p, bm, stream) : launch_mid_fp8_t<SK_E4M3, false>(p, bm, stream);
}

hipError_t launch_mid_i8(const MidArgs& p, hipStream_t stream) {
  if (p.op.K % 16 != 0 || p.splits < 1) return hipErrorInvalidValue;
  return launch_mid_c<MidCfg<SK_I8, false, 64, 6>>(p, stream);
}

hipError_t launch_mid_w4(const W4Args& a, int bm, int splits, void* partial, hipStream_t stream) {
  if ((a.flags & QG_W4_LAYOUT_KN) || splits < 1) return hipErrorInvalidValue;
  const MidArgs p{skinny_args(a), splits, partial};
  return a.a_f16 ? launch_mid_w4_t<true>(p, a.group, bm, stream) : launch_mid_w4_t<false>(p, a.group, bm, stream);
}

}  // namespace qg
