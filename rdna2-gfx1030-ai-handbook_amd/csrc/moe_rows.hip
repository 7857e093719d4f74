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
// the activation bytes that up to 16 do; more rows of an entry repeat the walk
// over its weights. 16 tokens, 64 experts, top-8, hidden 2048, inter 768 (56 of
// the experts in use): gate/up 176 MB 50.5 -> 31.3 us (5.6 TB/s), down 88 MB
// 32.7 -> 20.0 us (4.4 TB/s).
#include "qg_common.h"
#include "qg_epilogue.h"
#include "qg_internal.h"
#include "qg_wformat.h"

namespace qg {

namespace {

constexpr int kMoeRowsWaves = 4, kMoeRowsDepth = 2, kMoeRowsCT = 2;

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

// Rows [t.first, t.stop), RP at a time, of one table entry and column block.
template <int MOE, int RP, int CT>
__device__ __forceinline__ void moe_rows_body(const I8GemmArgs& p, const MoeRowsTile& t, char* smem) {
#pragma clang fp contract(off)
  using C = MoeRowsCfg<RP, CT>;
  constexpr int NW = C::NW, D = C::D;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, q = lane >> 4;
  char* const ring = smem + wave * D * C::STAGE;
  const uint32_t ring_addr = lds_addr_of(ring);
  const int slot16 = lane & 7;  // 16-byte slot of a lane in its 128-byte LDS row
  auto source = [&](int row) __attribute__((always_inline)) {
    return min(max(p.row_token ? p.row_token[row] : row, 0), p.a_rows - 1);
  };

  uint32_t woff[C::W_COPIES];
  static_for<0, C::W_COPIES>([&](auto i) {
    const int c = 8 * i + (lane >> 3);
    woff[i] = static_cast<uint32_t>(min(t.n0 + c, p.N - 1)) * static_cast<uint32_t>(p.w_sn) +
              16u * (slot16 ^ lds_row_xor<C::KS>(c & 15));
  });
  const int chunks = p.K / C::KS;
  const int n = chunks > wave ? (chunks - wave + NW - 1) / NW : 0;

  for (int r0 = t.first; r0 < t.stop; r0 += RP) {
    // everything that is read through registers is requested before the copies
    uint32_t aoff[C::A_COPIES];
    static_for<0, C::A_COPIES>([&](auto i) {
      const int r = 8 * i + (lane >> 3);
      aoff[i] = static_cast<uint32_t>(source(min(r0 + r, t.stop - 1))) * static_cast<uint32_t>(p.a_sm) +
                16u * (slot16 ^ lds_row_xor<C::KS>(r));
    });
    // output elements of this thread: (row, column), or (row, feature) for SiLU * mul
    constexpr int OC = MOE == QG_MOE_EPI_SILU_MUL ? 8 * CT : 16 * CT;
    constexpr int PER = (RP * OC + 64 * NW - 1) / (64 * NW);
    float sa[PER], sb[PER], sb2[PER], rw[PER];
    int dst[PER], at[PER];
    static_for<0, PER>([&](auto i) {
      const int e = threadIdx.x + 64 * NW * i;
      const int rr = e / OC, oc = e % OC;
      // gate column of feature oc; its up column is 16 further on
      const int cc = MOE == QG_MOE_EPI_SILU_MUL ? 32 * (oc >> 4) + (oc & 15) : oc;
      const int row = r0 + rr;
      const bool in = rr < RP && row < t.stop && t.n0 + cc < p.N;
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
      const uint32_t to = ring_addr + slot * C::STAGE;
      static_for<0, C::W_COPIES>([&](auto i) {
        dma16s_nt(t.w, woff[i] + static_cast<uint32_t>(C::KS * c), to + C::W_AT + 1024 * i);
      });
      static_for<0, C::A_COPIES>([&](auto i) {
        dma16s(p.a, aoff[i] + static_cast<uint32_t>(C::KS * c), to + 1024 * i);
      });
    };
    i32x4 acc[CT];
    static_for<0, CT>([&](auto j) { acc[j] = i32x4{0, 0, 0, 0}; });
    static_for<0, D>([&](auto d) {
      if (d < n) issue(wave + NW * d, d);
    });
    const int arow = min(col, RP - 1);
    for (int i = 0; i < n; ++i) {
      if (i + 1 < n) wait_vm<C::COPIES>();
      else wait_vm<0>();
      const char* const st = ring + (i & 1) * C::STAGE;
      static_for<0, 2>([&](auto u) {
        const i32x4 a = *reinterpret_cast<const i32x4*>(st + arow * C::KS + 16 * ((4 * u + q) ^ lds_row_xor<C::KS>(arow)));
        static_for<0, CT>([&](auto j) {
          const i32x4 w = *reinterpret_cast<const i32x4*>(st + C::W_AT + (16 * j + col) * C::KS +
                                                          16 * ((4 * u + q) ^ lds_row_xor<C::KS>(col)));
          acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, w, acc[j], 0, 0, 0);
        });
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's reads are done
      if (i + D < n) issue(wave + NW * (i + D), i & 1);
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
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[w * 16 * C::PITCH + word];
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
    if (r0 + RP < t.stop) __syncthreads();  // the partial tiles have been read
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
  if (t.stop - t.first <= 8) moe_rows_body<MOE, 8, CT>(p, t, smem);
  else moe_rows_body<MOE, 16, CT>(p, t, smem);
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
// expert at most once, so up to two passes), or of up to 64 where rows_max
// leaves 16 rows per expert on average after the dispatch's default padding to
// 64 (with another padding at most four passes); up to 16 slots per expert
// behind the route epilogue. Whole MoE calls against the persistent tiles (us):
//   tokens, experts, top-k, hidden, inter    tiles   here
//   16, 64, 8, 2048, 768                     104.0   67.8   2 rows an expert
//   64, 64, 8, 2048, 768                     105.9   77.4   8
//   16, 8, 8, 2048, 1024                      59.6   34.8   16
//   32, 16, 8, 3072, 1024                     78.6   64.7   16
//   32, 8, 8, 2048, 1024                      59.7   49.4   32, gate/up here only
//   64, 16, 8, 3072, 1024                     79.3   83.0   32, gate/up here only
//   64, 8, 8, 2048, 1024                      59.4   58.8   64, gate/up here only
//   1000, 64, 1, 1024, 512                    58.6   57.8   16, down here only
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
