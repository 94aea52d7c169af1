// fewrows_softmax.hip -- the chain for a few query rows against long key
// matrices (attention scores in decode: batch of heads x sequences,
//   out[b] = softmax_row(scale * Q[b] . K[b]^T), Q of at most 32 rows, K <= 128),
// one workgroup per batch, all rows and columns.
//
// What bounds it is reading B once: 128 batches x 4 rows x 2048 columns x 128
// are 64 MiB of B and 2 MiB of output.  The row-block kernel reads B twice and
// computes 128 rows, the tiles stage and store 128 rows per 128 columns; here a
// workgroup streams B once through a ring of direct-to-LDS loads, keeps the
// logits (m x n f32) in LDS and normalises from there, so nothing else goes to
// memory and no workgroup waits for another.
//
// 8 waves in two roles while B streams, in units of 64 k-rows x 128 columns
// (16 KiB): 4 I/O waves request unit u + S - 1 while 4 compute waves, 32
// columns each, run unit u's MFMAs (32 x 32 x 16, D = B^T . A^T: a lane's
// accumulators belong to one row).  A wave that issues loads waits until the
// memory pipeline takes them, so the streaming does not depend on the compute
// waves' pace.  A few KiB at most, A goes straight to registers as fragments.
// Then all 8 waves share the rows.
//
// Bytes in flight per CU set the rate (about 2 us from HBM under load): the
// ring takes what the logits leave, S = 6 units (80 KiB in flight) with up to
// 64 KiB of logits; small problems of more batches than CUs run two workgroups
// per CU (S = 4, up to 16 KiB), so that one streams while the other starts or
// normalises.
//
// Measured against the split path's 128-row tiles (us a call): 128 x 4 x 2048 x
// 128 37.4 -> 14.3 (68 MB: 4.8 TB/s), 256 x 1 x 2048 x 128 41 -> 23 (5.8 TB/s),
// 512 x 2 x 1720 x 96 114 -> 28.5, 64 x 8 x 1024 x 64 12.8 -> 7.2.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"
#include "tile_layout.h"
#include "wtc_kernels.h"

namespace wtc {

namespace few {
constexpr int BN = 128;         // columns per tile
constexpr int UNIT = 64 * 256;  // 64 k-rows of a tile: 16 KiB
constexpr int NCW = 4;          // compute waves, then 4 I/O waves
constexpr int NT = 512;
constexpr int BPW = 4;          // 1 KiB load blocks per I/O wave and unit
constexpr int KS = 8;           // k-steps of 16: K <= 128
constexpr int NC = 7;           // 8-column chunks a lane holds of a row, at most
// S ring stages and the logits' floats; 160 KiB over the workgroups of a CU
template <int S> struct Lds {
  static constexpr int RING = S * UNIT;
  static constexpr int LOGITS = S == 6 ? kFewRowsMaxLogits : kFewRowsPairLogits;
  static constexpr int BYTES = RING + LOGITS * 4;
};
static_assert(Lds<6>::BYTES <= 160 * 1024 && 2 * Lds<4>::BYTES <= 160 * 1024, "LDS");

// Waves that share a row in the last phase: 8 over the rows' next power of two.
__host__ __device__ constexpr int waves_per_row(int m) { return m == 1 ? 8 : (m == 2 ? 4 : (m <= 4 ? 2 : 1)); }
// The most chunks a lane holds, over every number of rows with the longest rows
// that the logits' limit lets in: the last phase reads, sums and stores NC.
constexpr int most_chunks() {
  int most = 0;
  for (int m = 1; m <= kFewRowsMax; ++m) {
    const int tiles = (kFewRowsMaxLogits / m - kFewRowsPad) / BN, lanes = 64 * waves_per_row(m);
    const int chunks = (tiles * (BN / 8) + lanes - 1) / lanes;
    most = chunks > most ? chunks : most;
  }
  return most;
}
static_assert(most_chunks() == NC && kFewRowsMax <= 32, "chunks of a row in a lane's registers; 32 rows per MFMA");
static_assert(kFewRowsPairLogits <= kFewRowsMaxLogits, "the pair limit is the smaller one");
}  // namespace few

template <int IN_DT, int OUT_DT, int S>
__global__ void __launch_bounds__(few::NT, S == 6 ? 2 : 4)
chain_few_rows_kernel(const ChainParams p) {
  using namespace few;
  using L = Lds<S>;
  __shared__ __attribute__((aligned(16))) uint8_t smem[L::BYTES];
  float* logits = reinterpret_cast<float*>(smem + L::RING);  // [m][pitch], raw accumulators

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave_u = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t bt = blockIdx.x;
  const uint32_t M = (uint32_t)p.M, N = (uint32_t)p.N, K = (uint32_t)p.K;
  const int nT = p.nT;
  const int pitch = nT * BN + kFewRowsPad;
  const int upt = K > 64 ? 2 : 1;  // units per tile
  const int units = nT * upt;

  if (wave_u >= NCW) {
    // ---- I/O waves: barrier B(u) says that unit u has landed and that every
    // compute wave is done with unit u-1, whose stage unit u+S-1 then takes.
    const int v = wave_u - NCW;
    const uint32_t ldb = (uint32_t)p.ldb_bytes;
    const i32x4 rbv = raw_rsrc(p.b + bt * p.b_bstride, (uint32_t)p.b_bstride);
    // Block q of this wave: k-rows 16v + 4q .. +3 of the unit.  k-rows past K are
    // clamped to K, whose offset lies past the buffer descriptor (one batch
    // slice of B): they read zero.
    const uint32_t krow0 = (uint32_t)dma_b_row(dma_block(v, 0, BPW), lane);
    const uint32_t bcol = 8u * (uint32_t)dma_b_chunk(dma_block(v, 0, BPW), lane);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(WTC_LDS uint8_t*)smem + (uint32_t)dma_block(v, 0, BPW) * 1024u;
    auto issue = [&](int u) {
      const uint32_t tile = (uint32_t)u >> (upt - 1), kb = upt == 2 ? 64u * ((uint32_t)u & 1u) : 0u;
      const uint32_t col = tile * BN + bcol;
      const bool in = u < units && col < N;
#pragma unroll
      for (int q = 0; q < BPW; ++q) {
        const uint32_t off = min(kb + krow0 + 4u * (uint32_t)q, K) * ldb + col * 2u;
        dma16(rbv, in ? off : kOutOfRange, lds0 + (uint32_t)(u % S) * UNIT + (uint32_t)q * 1024u);
      }
    };
#pragma unroll
    for (int u = 0; u < S - 1; ++u) issue(u);
    for (int u = 0; u < units; ++u) {
      wait_loads_barrier<BPW*(S - 2)>();  // B(u)
      issue(u + S - 1);
    }
    // every load has landed before the ring is used for the reductions
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    // ---- compute waves: columns nw .. nw+31 of every tile
    const int nw = wave_u * 32;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a + bt * p.a_bstride, (uint32_t)p.a_bstride);
    const uint32_t row = (uint32_t)frag_row(lane);
    u32x4 af[KS];  // row lane % 32, k = 16 s + 8 (lane / 32) .. +7; zero past M and K
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t k = 16u * s + 8u * (uint32_t)(lane >> 5);
      af[s] = bload16(ra, row < M && k < K ? row * (uint32_t)p.lda_bytes + 2u * k : kOutOfRange);
    }
    f32x16 acc;
    auto products = [&](const uint8_t* st, int s0) {  // the four k-steps of a unit
      u32x4 bf[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const u32x2 lo = tr_read(st + btr_offset(btr_k(s, 0, lane), btr_n(nw, lane)));
        const u32x2 hi = tr_read(st + btr_offset(btr_k(s, 1, lane), btr_n(nw, lane)));
        bf[s] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const u32x4 a = s0 ? af[4 + s] : af[s];
        if constexpr (IN_DT == DT_F16)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, bf[s]), __builtin_bit_cast(f16x8, a),
                                                       acc, 0, 0, 0);
        else
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bf[s]),
                                                        __builtin_bit_cast(bf16x8, a), acc, 0, 0, 0);
      }
    };
    float* mine = logits + (int)row * pitch + nw + 4 * (lane >> 5);
    int u = 0;
    for (int tile = 0; tile < nT; ++tile) {
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // B(u)
      products(smem + (u % S) * UNIT, 0);
      ++u;
      if (upt == 2) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        products(smem + (u % S) * UNIT, 4);
        ++u;
      }
      if (row < M) {
#pragma unroll
        for (int g = 0; g < 4; ++g)  // columns nw + 8g + 4 (lane / 32) .. +3
          *reinterpret_cast<f32x4*>(mine + tile * BN + 8 * g) =
              f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
      }
    }
  }
  __syncthreads();

  // ---- all waves: row r0 + wave / P, chunks (8 columns) part * 64 + lane, in
  // steps of 64 P.  A row's statistics meet in the ring's first words.
  const int P = waves_per_row((int)M);
  const int par = 8 / P;  // rows at a time
  const int part = wave_u % P;
  float* red = reinterpret_cast<float*>(smem);  // [2][8 waves]
  const int nch = (int)N / 8;
  const float c2 = p.c2;
  uint8_t* o_base = p.out + (int64_t)bt * p.o_bstride;
  constexpr int OSZ = OutTraits<OUT_DT>::SZ;
  for (int r0 = 0; r0 < (int)M; r0 += par) {
    const int r = r0 + wave_u / P;
    const bool live = r < (int)M;
    const float* src = logits + (live ? r : 0) * pitch;
    f32x4 x[NC][2];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = part * 64 + lane + i * 64 * P;
      const bool in = c < nch;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[i][h] = *reinterpret_cast<const f32x4*>(src + (in ? 8 * c : 0) + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, in ? x[i][h][e] * c2 : -INFINITY);
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if (P > 1) {
      if (lane == 0) red[wave_u] = mx;
      __syncthreads();
      for (int w = 0; w < P; ++w) mx = fmaxf(mx, red[wave_u - part + w]);
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = part * 64 + lane + i * 64 * P;
      float s = 0.0f;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(x[i][h][e], c2, -mx));
          x[i][h][e] = y;
          s += y;
        }
      sum += c < nch ? s : 0.0f;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (P > 1) {
      if (lane == 0) red[8 + wave_u] = sum;
      __syncthreads();
      sum = 0.0f;
      for (int w = 0; w < P; ++w) sum += red[8 + wave_u - part + w];
    }
    const float inv = 1.0f / sum;
    uint8_t* dst = o_base + (int64_t)r * p.ldo_bytes;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = part * 64 + lane + i * 64 * P;
      if (!live || c >= nch) continue;
      if constexpr (OSZ == 4) {
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<f32x4*>(dst + (int64_t)c * 32 + 16 * h) = x[i][h] * inv;
      } else {
        uint32_t w0, w1, w2, w3;
        pack4_product<OUT_DT>(x[i][0], inv, &w0, &w1);
        pack4_product<OUT_DT>(x[i][1], inv, &w2, &w3);
        *reinterpret_cast<u32x4*>(dst + (int64_t)c * 16) = u32x4{w0, w1, w2, w3};
      }
    }
  }
}

namespace {
template <int IN_DT, int S> const void* few_by_out(int out_dt) {
  switch (out_dt) {
    case DT_F32: return reinterpret_cast<const void*>(&chain_few_rows_kernel<IN_DT, DT_F32, S>);
    case DT_F16: return reinterpret_cast<const void*>(&chain_few_rows_kernel<IN_DT, DT_F16, S>);
    case DT_BF16: return reinterpret_cast<const void*>(&chain_few_rows_kernel<IN_DT, DT_BF16, S>);
  }
  return nullptr;
}
}  // namespace

const void* few_rows_kernel_symbol(int in_dt, int out_dt, int stages) {
  if (in_dt == DT_F16) return stages == 6 ? few_by_out<DT_F16, 6>(out_dt) : few_by_out<DT_F16, 4>(out_dt);
  if (in_dt == DT_BF16) return stages == 6 ? few_by_out<DT_BF16, 6>(out_dt) : few_by_out<DT_BF16, 4>(out_dt);
  return nullptr;
}
int few_rows_kernel_threads() { return few::NT; }

}  // namespace wtc
