// Grouped (MoE) INT8 GEMM for a few routed rows per expert (a decode step) on
// gfx950: the contract, tile table and epilogues of k_i8_moe_pp (int8_gemm.hip),
// bit for bit.
//
// Such a call reads each used expert's weights once and is bound by that read.
// The persistent 192 x 256 tiles leave a tail (64 experts x 6 or 8 column tiles
// over 256 CUs, one workgroup each) and spend their stages on empty rows. Here
// a workgroup of 4 waves owns 32 columns of one table entry, wave w takes K
// chunks w, w + 4, ... into a ring of its own (no barrier until the partial
// tiles are summed, as in k_skinny_gemm), and three workgroups per CU overlap
// one another's table reads, copies and epilogues. Up to 8 rows copy half of
// the activation bytes that up to 16 do. An entry of more rows (a skewed router)
// takes 64 at a time, 16 a wave, all waves on one chunk of the weights: passes of
// 16 rows over the weights instead cost 162.9 us at 64 tokens on the same 8 of 64
// experts, hidden 4096, inter 2048, where the tiles take 98.6 and this 75. 16
// tokens, 64 experts, top-8, hidden 2048, inter 768 (56 of the experts in use):
// gate/up 176 MB 50.5 -> 31.3 us (5.6 TB/s), down 88 MB 32.7 -> 20.0 us (4.4
// TB/s).
#include "qg_common.h"
#include "qg_epilogue.h"
#include "qg_internal.h"
#include "qg_wformat.h"

namespace qg {

namespace {

constexpr int kMoeRowsWaves = 4, kMoeRowsDepth = 2, kMoeRowsCT = 2;
constexpr int kMoeTallSlots = 4;  // ring of the tall form

template <int RP_, int CT_>
struct MoeRowsCfg {
  static constexpr int RP = RP_, CT = CT_, D = kMoeRowsDepth, NW = kMoeRowsWaves, KS = 128;
  static constexpr int A_COPIES = RP * KS / 1024, W_COPIES = 16 * CT * KS / 1024;
  static constexpr int COPIES = A_COPIES + W_COPIES;
  static constexpr int W_AT = A_COPIES * 1024, STAGE = COPIES * 1024;
  static constexpr int PITCH = 16 * CT + 1;  // words per row of a partial tile
  static constexpr int RING = NW * D * STAGE, RED = NW * 16 * PITCH * 4;
  static_assert(RP * KS % 1024 == 0 && (RP == 8 || RP == 16), "activation copies of whole waves");
  static_assert(RED <= RING && D == 2, "partial tiles reuse the rings; two-deep waits");
};

struct MoeRowsTile {
  const int8_t* w;   // the expert's weights
  const float* sb;   // and column scales
  int first, stop;   // rows
  int n0;
};

// Rows [t.first, t.stop) of one table entry and column block, RP at a time, the
// K chunks spread over the waves. TALL (entries of many rows): 16 rows a wave
// and all waves on the same chunk, in a ring of kMoeTallSlots chunks that they
// fill together, one barrier per chunk; the weights are copied once for 64 rows.
template <int MOE, int RP, int CT, bool TALL>
__device__ __forceinline__ void moe_rows_body(const I8GemmArgs& p, const MoeRowsTile& t, char* smem) {
#pragma clang fp contract(off)
  using C = MoeRowsCfg<RP, CT>;
  constexpr int NW = C::NW, D = C::D;
  constexpr int PASS = TALL ? 16 * NW : RP;  // rows per pass
  // copies of a wave and chunk, 8 rows of 128 bytes each
  constexpr int A_COPIES = TALL ? PASS / 8 / NW : C::A_COPIES, W_COPIES = TALL ? 2 * CT / NW : C::W_COPIES;
  constexpr int STAGE = TALL ? (PASS + 16 * CT) * C::KS : C::STAGE, W_AT = PASS * C::KS;
  static_assert(!TALL || (2 * CT % NW == 0 && kMoeTallSlots * STAGE <= C::RING), "copies and ring of the tall form");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, q = lane >> 4;
  char* const ring = TALL ? smem : smem + wave * D * STAGE;
  const uint32_t ring_addr = lds_addr_of(ring);
  const int slot16 = lane & 7;  // 16-byte slot of a lane in its 128-byte LDS row
  const int row8 = lane >> 3;   // row of a lane in a copy
  // copy i of a wave: rows 8 copy_of(i) .. + 7 of the operand
  auto copy_of = [&](int i) __attribute__((always_inline)) { return TALL ? wave + NW * i : i; };
  auto source = [&](int row) __attribute__((always_inline)) {
    return min(max(p.row_token ? p.row_token[row] : row, 0), p.a_rows - 1);
  };

  uint32_t woff[W_COPIES];
  static_for<0, W_COPIES>([&](auto i) {
    const int c = 8 * copy_of(i) + row8;
    woff[i] = static_cast<uint32_t>(min(t.n0 + c, p.N - 1)) * static_cast<uint32_t>(p.w_sn) +
              16u * (slot16 ^ lds_row_xor<C::KS>(c & 15));
  });
  const int chunks = p.K / C::KS;
  const int n = TALL ? chunks : chunks > wave ? (chunks - wave + NW - 1) / NW : 0;

  for (int r0 = t.first; r0 < t.stop; r0 += PASS) {
    // everything that is read through registers is requested before the copies
    uint32_t aoff[A_COPIES];
    static_for<0, A_COPIES>([&](auto i) {
      const int r = 8 * copy_of(i) + row8;
      aoff[i] = static_cast<uint32_t>(source(min(r0 + r, t.stop - 1))) * static_cast<uint32_t>(p.a_sm) +
                16u * (slot16 ^ lds_row_xor<C::KS>(r & 15));
    });
    // output elements of this thread: (row, column), or (row, feature) for SiLU * mul
    constexpr int OC = MOE == QG_MOE_EPI_SILU_MUL ? 8 * CT : 16 * CT;
    constexpr int PER = (PASS * OC + 64 * NW - 1) / (64 * NW);
    float sa[PER], sb[PER], sb2[PER], rw[PER];
    int dst[PER], at[PER];
    static_for<0, PER>([&](auto i) {
      const int e = threadIdx.x + 64 * NW * i;
      const int rr = e / OC, oc = e % OC;
      // gate column of feature oc; its up column is 16 further on
      const int cc = MOE == QG_MOE_EPI_SILU_MUL ? 32 * (oc >> 4) + (oc & 15) : oc;
      const int row = r0 + rr;
      const bool in = rr < PASS && row < t.stop && t.n0 + cc < p.N;
      at[i] = rr * C::PITCH + cc;
      dst[i] = in ? row : -1;
      sa[i] = sb[i] = sb2[i] = rw[i] = 0.0f;
      if (in) {
        if constexpr (MOE != QG_MOE_EPI_I32) {
          sa[i] = p.a_scale[source(row)];
          sb[i] = t.sb[t.n0 + cc];
        }
        if constexpr (MOE == QG_MOE_EPI_SILU_MUL) sb2[i] = t.sb[t.n0 + cc + 16];
        if constexpr (MOE == QG_MOE_EPI_ROUTE) {
          rw[i] = p.row_weight[row];
          dst[i] = p.row_slot[row];
        }
      }
    });

    auto issue = [&](int c, int slot) __attribute__((always_inline)) {
      const uint32_t to = ring_addr + slot * STAGE;
      static_for<0, W_COPIES>([&](auto i) {
        if constexpr (TALL) dma16s(t.w, woff[i] + static_cast<uint32_t>(C::KS * c), to + W_AT + 1024 * copy_of(i));
        else dma16s_nt(t.w, woff[i] + static_cast<uint32_t>(C::KS * c), to + W_AT + 1024 * i);
      });
      static_for<0, A_COPIES>([&](auto i) {
        dma16s(p.a, aoff[i] + static_cast<uint32_t>(C::KS * c), to + 1024 * copy_of(i));
      });
    };
    i32x4 acc[CT];
    static_for<0, CT>([&](auto j) { acc[j] = i32x4{0, 0, 0, 0}; });
    const int arow = TALL ? 16 * wave + col : min(col, RP - 1);
    auto product = [&](int slot) __attribute__((always_inline)) {
      const char* const st = ring + slot * STAGE;
      static_for<0, 2>([&](auto u) {
        const i32x4 a = *reinterpret_cast<const i32x4*>(st + arow * C::KS +
                                                        16 * ((4 * u + q) ^ lds_row_xor<C::KS>(arow & 15)));
        static_for<0, CT>([&](auto j) {
          const i32x4 w = *reinterpret_cast<const i32x4*>(st + W_AT + (16 * j + col) * C::KS +
                                                          16 * ((4 * u + q) ^ lds_row_xor<C::KS>(col)));
          acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, w, acc[j], 0, 0, 0);
        });
      });
    };
    if constexpr (TALL) {
      // top of chunk i: it has landed everywhere and every wave has read chunk
      // i - 1, whose slot takes chunk i + R - 1
      constexpr int R = kMoeTallSlots, COPIES = A_COPIES + W_COPIES;
      static_assert(R == 4, "waits below");
      static_for<0, R - 1>([&](auto d) {
        if (d < n) issue(d, d);
      });
      for (int i = 0; i < n; ++i) {
        const int after = n - 1 - i;  // chunks issued after this one: min(after, R - 2)
        if (after >= 2) wait_vm_barrier<2 * COPIES>();
        else if (after == 1) wait_vm_barrier<COPIES>();
        else wait_vm_barrier<0>();
        if (i + R - 1 < n) issue(i + R - 1, (i + R - 1) % R);
        product(i % R);
      }
    } else {
      static_for<0, D>([&](auto d) {
        if (d < n) issue(wave + NW * d, d);
      });
      for (int i = 0; i < n; ++i) {
        if (i + 1 < n) wait_vm<C::COPIES>();
        else wait_vm<0>();
        product(i & 1);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's reads are done
        if (i + D < n) issue(wave + NW * (i + D), i & 1);
      }
    }

    int* const red = reinterpret_cast<int*>(smem);
    __syncthreads();  // every ring is done with
    static_for<0, CT>([&](auto j) {
      static_for<0, 4>([&](auto e) {
        red[(wave * 16 + 4 * q + e) * C::PITCH + 16 * j + col] = acc[j][int(e)];
      });
    });
    __syncthreads();
    static_for<0, PER>([&](auto i) {
      if (dst[i] < 0 || dst[i] >= p.out_rows) return;
      auto sum = [&](int word) __attribute__((always_inline)) {
        int v = red[word];
        if constexpr (!TALL) {
#pragma unroll
          for (int w = 1; w < NW; ++w) v += red[w * 16 * C::PITCH + word];
        }
        return v;
      };
      const int e = threadIdx.x + 64 * NW * i;
      const int64_t o = static_cast<int64_t>(dst[i]) * p.out_sm +
                        (MOE == QG_MOE_EPI_SILU_MUL ? t.n0 / 2 : t.n0) + e % OC;
      const int v = sum(at[i]);
      if constexpr (MOE == QG_MOE_EPI_I32) {
        static_cast<int32_t*>(p.out)[o] = v;
      } else if constexpr (MOE == QG_MOE_EPI_SILU_MUL) {
        const float g = static_cast<float>(v) * (sa[i] * sb[i]);
        const float u = static_cast<float>(sum(at[i] + 16)) * (sa[i] * sb2[i]);
        static_cast<uint16_t*>(p.out)[o] = f32_to_bf16(silu(g) * u);
      } else {
        const float y = static_cast<float>(v) * (sa[i] * sb[i]);
        static_cast<uint16_t*>(p.out)[o] = f32_to_bf16(y * rw[i]);
      }
    });
    if (r0 + PASS < t.stop) __syncthreads();  // the partial tiles have been read
  }
}

template <int MOE, int CT>
__global__ __launch_bounds__(64 * kMoeRowsWaves) void k_moe_rows(I8GemmArgs p) {
  __shared__ __attribute__((aligned(1024))) char smem[MoeRowsCfg<16, CT>::RING];
  const int cols = ceil_div(p.N, 16 * CT);
  const int tile = blockIdx.x / cols;
  if (tile >= min(max(p.tiles[3], 0), p.tiles_max)) return;
  const int e = __builtin_amdgcn_readfirstlane(p.tiles[4 * tile]);
  const int m0 = __builtin_amdgcn_readfirstlane(p.tiles[4 * tile + 1]);
  const int m_end = __builtin_amdgcn_readfirstlane(p.tiles[4 * tile + 2]);
  if (e < 0 || e >= p.n_experts || m0 < 0 || m0 >= p.M || m_end <= m0 || m_end > p.M) return;
  const MoeRowsTile t{p.w + e * p.w_estride, p.b_scale ? p.b_scale + static_cast<int64_t>(e) * p.N : nullptr, m0,
                      min(m_end, m0 + QG_MOE_TILE_ROWS), (static_cast<int>(blockIdx.x) - tile * cols) * 16 * CT};
  const int rows = t.stop - t.first;
  if (rows <= 8) moe_rows_body<MOE, 8, CT, false>(p, t, smem);
  else if (rows <= 16) moe_rows_body<MOE, 16, CT, false>(p, t, smem);
  else moe_rows_body<MOE, 16, CT, true>(p, t, smem);
}

template <int MOE>
hipError_t launch_moe_rows_e(const I8GemmArgs& p, hipStream_t stream) {
  const int64_t blocks = static_cast<int64_t>(p.tiles_max) * ceil_div(p.N, 16 * kMoeRowsCT);
  hipLaunchKernelGGL((k_moe_rows<MOE, kMoeRowsCT>), dim3(static_cast<unsigned>(blocks)), dim3(64 * kMoeRowsWaves), 0,
                     stream, p);
  return hipGetLastError();
}

}  // namespace

// Few rows per expert. A gathered operand of up to 32 tokens (a token takes an
// expert at most once), or of up to 64 where rows_max leaves 16 rows per expert
// on average after the dispatch's default padding to 64; up to 16 slots per
// expert behind the route epilogue, however the router spreads them (the tall
// form keeps even all tokens on the same experts within 4 % of the tiles).
// Whole MoE calls against the persistent tiles (us, tiles / here):
//   tokens, experts, top-k, hidden, inter    even routing     the same experts
//   16, 64, 8, 2048, 768                     104.5    66.7     59.8    32.8
//   64, 64, 8, 2048, 768                     104.8    78.5     59.7    37.5
//   32, 16, 8, 4096, 2048                    121.2    94.6     91.4    64.4
//   64, 8, 2, 2048, 768                       56.4    33.4     56.8    30.5
//   128, 64, 8, 4096, 2048 (down here only)  387.3   367.4    100.7   104.3
//   512, 64, 1, 2048, 768 (down here only)   103.3    93.2     59.5    56.0
//   1000, 64, 1, 2048, 768 (down here only)  114.3   103.9     63.0    61.3
bool moe_rows_applies(const I8GemmArgs& p) {
  const int64_t few = static_cast<int64_t>(kMoeFewRows) * p.n_experts;
  if (p.moe_epi == QG_MOE_EPI_ROUTE) return p.out_rows <= few;
  return p.a_rows <= 2 * kMoeFewRows ||
         (p.a_rows <= 4 * kMoeFewRows && p.M <= few + 63 * static_cast<int64_t>(p.n_experts));
}

hipError_t launch_moe_rows(const I8GemmArgs& p, hipStream_t stream) {
  switch (p.moe_epi) {
    case QG_MOE_EPI_I32: return launch_moe_rows_e<QG_MOE_EPI_I32>(p, stream);
    case QG_MOE_EPI_SILU_MUL: return launch_moe_rows_e<QG_MOE_EPI_SILU_MUL>(p, stream);
    default: return launch_moe_rows_e<QG_MOE_EPI_ROUTE>(p, stream);
  }
}

}  // namespace qg
