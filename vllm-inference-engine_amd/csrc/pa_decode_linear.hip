// Projections of a decode step's transformer layer for gfx950 (MI355X).
//
// Y = X W^T for the few hundred rows of a decode batch (modeling_qwen2's
// q/k/v, o, gate/up and down projections), with the elementwise neighbours of
// each product in the same launch: the RMSNorm before it, and the bias, the
// residual add or silu(gate) * up after it. A decoder layer is then four of
// these launches around the attention launch instead of four library GEMMs,
// two norm launches and a SwiGLU launch.
//
// What bounds it. At these sizes a launch is a chain of latencies -- about 1.6
// us for an empty launch in a captured graph, then the memory round trips from
// the first loads to the last store -- plus the weight stream (1.6 to 17 MB at
// hidden 896) and every workgroup's reads of X through its L1. So the kernel
// keeps one round trip where it can and makes every load a whole-line one:
//   * Operands are packed (pack_index): the fragment a wavefront feeds to
//     one v_mfma_f32_16x16x32_f16 (16 rows x 32 of K) is 1 KB of consecutive
//     memory. Row-major operands make each 16-byte load touch 16 rows; the
//     same kernel on row-major weights and activations took 9.2 us instead of
//     5.4 (down projection 4864 -> 896 at 8 rows) and 16.2 instead of 7.9 us
//     (128 rows). Weights are packed once; activations are written packed by
//     the launch that produces them.
//   * Weights that a program may change in place (o and down, which are not
//     merged with others) are read where they are, row-major (WROW). A fragment
//     takes its 8 values of row lane % 16 from every lane; loaded so, 16
//     neighbouring lanes touch 16 rows. Instead two loads fetch two K steps of a tile,
//     eight lanes to 128 consecutive bytes of a row, and the wavefront exchanges them
//     through LDS of its own. Us per launch as below, cold weights and from L2: down at
//     8 rows packed 5.5 and 4.4, row-major loads 7.8, this 6.2 and 5.2; o 3.2 and 2.9,
//     3.7, 3.5 and 3.1; at 128 rows down 7.0 and 5.9, 13.4, 7.8 and 6.9, o 3.8 and 3.5,
//     5.7, 4.3 and 3.9. Four steps at a time, 64 bytes of a row to four lanes and a
//     transpose in registers: down 6.5 and 5.4, 8.1 and 7.3. A packed copy would be
//     faster but would not follow the parameter.
//   * K is split over the workgroup's wavefronts: each loads its own weight
//     and X fragments straight into registers, DEPTH steps ahead, multiplies,
//     and the wavefronts' tiles are summed through LDS in wavefront order (the
//     same bits on every run). Nothing is staged, and there is no barrier
//     before the sum.
//   * The norm needs each row's sum of squares. The launch that writes a
//     residual row also leaves the sum over each of its 16-column tiles
//     (ss_out), so the next launch adds a row's few dozen partial sums, loaded
//     ahead of the fragments, instead of reading the row twice. The scale
//     rsqrt(mean + eps) is split into a power of two, applied to the fp16
//     values exactly, and a factor in [1, 2) applied to the fp32 sums: the
//     product's operand fp16(x * 2^e * weight) is rounded once, where the
//     unfused norm rounds twice.
//
// Measured on MI355X inside captured graphs, each launch on another layer's
// weights (hidden 896, MLP 4864, 14 / 2 heads of 64), against the library GEMM
// (row-major, without norm and SwiGLU), us per launch: 8 rows: q/k/v 3.7
// against 5.5, o 3.3 / 5.4, gate/up 6.6 / 8.5, down 5.5 / 9.3; 128 rows: 4.5 /
// 7.5, 3.9 / 7.4, 11.1 / 12.6, 7.0 / 10.0; 256 rows: 5.6 / 7.7, 4.7 / 7.5,
// 19.3 / 15.5, 8.9 / 11.3 (the norms and SwiGLU it saves are three more launches
// of about 3.5 us); 512 rows: 7.9 / 8.0, 6.6 / 7.8, 34 / 20, 18 / 16.
#include "pa_tiles.h"

namespace pa {

using namespace tiles;

// One workgroup: TO = TN output tiles of 16 columns (SILU: TN / 2, with the
// gate and the up rows of the merged weight) by TM tiles of 16 rows, K split
// over NW wavefronts. Tiles past the end of N or M repeat the last one and are
// not stored; K steps past a wavefront's range load zeros (empty resources),
// so no branch separates the loads. WROW: row-major weights.
template <int NW, int TN, int TM, int DEPTH, bool NORM, bool SILU, bool XPACK, bool WROW>
__global__ __launch_bounds__(64 * NW) void decode_linear_kernel(LinearArgs a) {
  constexpr int TO = SILU ? TN / 2 : TN;
  constexpr int ROWS = 16 * TM;
  constexpr int PARTS = 64 * NW / ROWS;  // threads that add one row's partial sums
  static_assert(!SILU || TN % 2 == 0, "a gate tile goes with its up tile");
  static_assert(!WROW || DEPTH % 2 == 0, "row-major weights come two steps at a time");
  static_assert(PARTS * ROWS == 64 * NW, "threads must split evenly over the rows");
  __shared__ __attribute__((aligned(16))) float s_red[NW * TN * TM * 256];
  __shared__ float s_ss[NORM ? PARTS * ROWS : 1];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int row = lane & 15;
  const int grp = lane >> 4;
  // Row tiles of one column tile are neighbours on one XCD, whose L2 then
  // serves the weights to all but the first.
  const int wg = xcd_order(blockIdx.x, gridDim.x);
  const int nt = wg / a.mtiles;
  const int mt0 = (wg - nt * a.mtiles) * TM;  // first 16-row tile
  const int m0 = mt0 * 16;
  const int o0 = nt * TO;  // first 16-column output tile
  const int mrows = min(a.M - m0, ROWS);
  const int ntiles = a.N / 16;

  const int steps = a.K / 32;
  const int u0 = steps * wave / NW;  // this wavefront's K steps [u0, u1)
  const int u1 = steps * (wave + 1) / NW;

  // Partial sums of squares first: loads return in order, so waiting for these
  // does not wait for the fragments.
  float ssum = 0.f;
  if constexpr (NORM) {
    constexpr int U = 16;  // loads in flight
    const float* sp = a.ss + m0 + min(tid % ROWS, mrows - 1);
    for (int p0 = tid / ROWS; p0 < a.ss_parts; p0 += U * PARTS) {
      float v[U];
#pragma unroll
      for (int i = 0; i < U; ++i)
        v[i] = sp[(int64_t)min(p0 + i * PARTS, a.ss_parts - 1) * a.M];
#pragma unroll
      for (int i = 0; i < U; ++i) ssum += p0 + i * PARTS < a.ss_parts ? v[i] : 0.f;
    }
  }

  const f16* wt[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int t = min(o0 + (SILU ? i % TO : i), ntiles - 1) + (SILU && i >= TO ? ntiles : 0);
    wt[i] = a.w + (int64_t)t * 16 * (WROW ? a.ldw : a.K);
  }
  const f16* xt[TM];
  uint32_t x_lane[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    if constexpr (XPACK) {
      xt[t] = a.x + (int64_t)min(mt0 + t, (a.M - 1) / 16) * a.K * 16;
      x_lane[t] = lane * 16;
    } else {
      xt[t] = a.x + (int64_t)m0 * a.ldx;
      x_lane[t] = (uint32_t)min(t * 16 + row, mrows - 1) * (uint32_t)(a.ldx * 2) + grp * 16;
    }
  }

  u32x4 wf[DEPTH][TN], xf[DEPTH][TM], nf[NORM ? DEPTH : 1];
  // Row-major weights: load j of a pair holds rows 8 (j % 2) + lane / 8 of the tile, piece (8
  // values of K) lane % 8 of the pair's two steps. In LDS a piece's 16 rows are consecutive,
  // pieces 32 bytes further apart than they need be, so that neither the stores (two rows by
  // eight pieces per 16 lanes) nor the loads (16 rows) meet in a bank.
  constexpr int kPiece = 16 * 16 + 32;
  constexpr int kTile = 8 * kPiece;
  constexpr int kEnd = 0x7ff00000;  // past every tile: loads return zero
  __shared__ __attribute__((aligned(16))) char s_w[WROW ? NW * TN * kTile : 16];
  const int w_lane = (lane >> 3) * (int)a.ldw * 2 + (lane & 7) * 16;
  const int w_put = wave * TN * kTile + (lane & 7) * kPiece + (lane >> 3) * 16;
  const int w_get = wave * TN * kTile + grp * kPiece + row * 16;
  auto load_rows = [&](int j, int u, const f16* w) {
    const int pair = u - (j & 1);  // the pair's first step
    const bool in = pair + ((lane >> 2) & 1) < u1;
    return __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(w, kEnd), in ? w_lane : kEnd,
                                                 (j & 1) * 16 * (int)a.ldw + pair * 64, 0);
  };
  // The fragments of loads j and j + 1, in place.
  auto exchange = [&](int j) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      *reinterpret_cast<u32x4*>(&s_w[w_put + i * kTile]) = wf[j][i];
      *reinterpret_cast<u32x4*>(&s_w[w_put + i * kTile + 8 * 16]) = wf[j + 1][i];
    }
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      wf[j][i] = *reinterpret_cast<const u32x4*>(&s_w[w_get + i * kTile]);
      wf[j + 1][i] = *reinterpret_cast<const u32x4*>(&s_w[w_get + i * kTile + 4 * kPiece]);
    }
    wave_lds_fence();
  };
  auto load = [&](int j, int u) {
    const int nb = u < u1 ? 0x7fffffff : 0;
#pragma unroll
    for (int t = 0; t < TM; ++t)
      xf[j][t] = __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(xt[t], nb), (int)x_lane[t],
                                                       u * (XPACK ? 1024 : 64), 0);
#pragma unroll
    for (int i = 0; i < TN; ++i)
      wf[j][i] = WROW ? load_rows(j, u, wt[i])
                      : __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(wt[i], nb), lane * 16,
                                                              u * 1024, 0);
    if constexpr (NORM)
      nf[j] = __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(a.norm, nb), grp * 16, u * 64, 0);
  };
#pragma unroll
  for (int j = 0; j < DEPTH; ++j) {
    load(j, u0 + j);
    __builtin_amdgcn_sched_barrier(0);
  }

  // Row scales: rsqrt(mean + eps) = pow2 * rest.
  float rest[TM];
  f16 pow2[TM];
  if constexpr (NORM) {
    s_ss[tid] = ssum;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      float tot = 0.f;
#pragma unroll
      for (int p = 0; p < PARTS; ++p) tot += s_ss[p * ROWS + t * 16 + row];
      const float inv = rsqrtf(tot * a.inv_k + a.eps);
      // Rounded down: the fp16 operand never exceeds the normed value it stands for.
      const uint32_t e = __builtin_bit_cast(uint32_t, inv) & 0x7f800000u;
      const float p2 = fminf(fmaxf(__builtin_bit_cast(float, e), 0x1p-24f), 0x1p15f);  // fp16's range
      pow2[t] = (f16)p2;
      rest[t] = inv / p2;
    }
  }

  f32x4 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto product = [&](int j) {
    if constexpr (WROW) {
      if (j % 2 == 0) exchange(j);
    }
    f16x8 xv[TM];
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      xv[t] = __builtin_bit_cast(f16x8, xf[j][t]);
      if constexpr (NORM) xv[t] = xv[t] * pow2[t] * __builtin_bit_cast(f16x8, nf[j]);
    }
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int t = 0; t < TM; ++t)
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, wf[j][i]),
                                                           xv[t], acc[i][t], 0, 0, 0);
  };
  for (int u = u0; u + DEPTH < u1; u += DEPTH) {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      product(j);
      if (WROW && j % 2 == 0) continue;  // the pair's registers are free after its second step
      __builtin_amdgcn_sched_barrier(0);
      if (WROW) load(j - 1, u + DEPTH + j - 1);
      load(j, u + DEPTH + j);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int j = 0; j < DEPTH; ++j) product(j);

  // Sum over the wavefronts: lane (row, grp) of tile (i, t) holds columns 4
  // grp .. + 3 of row `row`.
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int t = 0; t < TM; ++t)
      *reinterpret_cast<f32x4*>(&s_red[((wave * TN + i) * TM + t) * 256 + lane * 4]) =
          NORM ? acc[i][t] * rest[t] : acc[i][t];
  __syncthreads();
  for (int j = wave; j < TO * TM; j += NW) {
    const int o = j / TM, t = j - o * TM;
    if (o0 + o >= ntiles || t * 16 >= mrows) continue;  // wavefront-uniform
    auto total = [&](int i) {
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
        s += *reinterpret_cast<const f32x4*>(&s_red[((w * TN + i) * TM + t) * 256 + lane * 4]);
      return s;
    };
    f32x4 y = total(o);
    const int n = (o0 + o) * 16 + grp * 4;
    const int m = m0 + t * 16 + row;
    const bool ok = t * 16 + row < mrows;
    if constexpr (SILU) {
      const f32x4 up = total(TO + o);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = y[r] / (1.f + expf(-y[r])) * up[r];
    }
    if (a.bias) {
      const f16x4 b4 = *reinterpret_cast<const f16x4*>(a.bias + n);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] += (float)b4[r];
    }
    const int64_t packed = pack_index(m, n, a.N);
    if (a.res && ok) {
      const f16x4 r4 = *reinterpret_cast<const f16x4*>(a.res + packed);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] += (float)r4[r];
    }
    f16x4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = (f16)y[r];
    if (ok) *reinterpret_cast<f16x4*>(a.y + (a.y_packed ? packed : m * a.ldy + n)) = h;
    if (a.ss_out) {
      float s = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) s = __builtin_fmaf((float)h[r], (float)h[r], s);
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (grp == 0 && ok) a.ss_out[(int64_t)(o0 + o) * a.M + m] = s;
    }
  }
}

// Row-major rows to the packed layout, with each row's sum of squares: one
// workgroup per row.
__global__ __launch_bounds__(256) void pack_rows_kernel(const f16* __restrict__ x, int64_t ldx,
                                                        f16* __restrict__ y, float* __restrict__ ss,
                                                        int K) {
  const int m = blockIdx.x;
  float s = 0.f;
  for (int k = threadIdx.x * 8; k < K; k += 256 * 8) {
    const f16x8 v = *reinterpret_cast<const f16x8*>(x + m * ldx + k);
    *reinterpret_cast<f16x8*>(y + pack_index(m, k, K)) = v;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf((float)v[e], (float)v[e], s);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  __shared__ float part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) ss[m] = part[0] + part[1] + part[2] + part[3];
}

template <int NW, int TN, int TM, int DEPTH, bool NORM, bool SILU, bool XPACK, bool WROW = false>
static hipError_t launch_tile(LinearArgs a, hipStream_t s) {
  constexpr int TO = SILU ? TN / 2 : TN;
  a.mtiles = (a.M + 16 * TM - 1) / (16 * TM);
  const int64_t grid = (int64_t)a.mtiles * ((a.N / 16 + TO - 1) / TO);
  if (grid > 0x7fffffff) return hipErrorInvalidValue;
  decode_linear_kernel<NW, TN, TM, DEPTH, NORM, SILU, XPACK, WROW>
      <<<(unsigned)grid, 64 * NW, 0, s>>>(a);
  return hipGetLastError();
}

// Tiles. The smallest tile whose workgroups all run at once (at most one per
// CU): a second round costs a whole chain of latencies, and a larger tile
// leaves CUs idle and gives each workgroup more X to read. Measured as above,
// us: q/k/v at 64 rows 2 x 1 tiles (144 workgroups) 4.0, 1 x 2 4.1, 2 x 2 4.5;
// at 128 rows 2 x 2 (144) 4.5, 2 x 1 (288) 4.8, 1 x 2 (288) 4.9; gate/up at
// 128 rows 6 x 4 (204) 11.1, 4 x 4 (304) 12.4, 6 x 2 (408) 12.5, 8 x 4 (152)
// 12.8; at 64 rows 6 x 2 (204) 9.1, 4 x 4 (152) 9.4, 4 x 2 (304) 10.4; down at
// 192 rows 2 x 2 (168) 8.7, 1 x 2 (336) 11.4, 2 x 1 (336) 11.7. Four
// wavefronts hold K up to 896 in one round of loads; longer rows take eight
// (down at 8 rows: eight 5.5, sixteen 5.8).
template <bool NORM, bool XPACK>
static hipError_t launch_plain(const LinearArgs& a, int cus, hipStream_t s) {
  const int64_t mt = (a.M + 15) / 16, nt = a.N / 16;
  const bool wide = a.K > 32 * 4 * 14;
  if (mt * nt <= cus)
    return wide ? launch_tile<8, 1, 1, 10, NORM, false, XPACK>(a, s)
                : launch_tile<4, 1, 1, 7, NORM, false, XPACK>(a, s);
  if (mt == 1 || mt * ((nt + 1) / 2) <= cus)
    return wide ? launch_tile<8, 2, 1, 10, NORM, false, XPACK>(a, s)
                : launch_tile<4, 2, 1, 7, NORM, false, XPACK>(a, s);
  return wide ? launch_tile<8, 2, 2, 7, NORM, false, XPACK>(a, s)
              : launch_tile<4, 2, 2, 7, NORM, false, XPACK>(a, s);
}

// Row-major weights: as launch_plain, but a long K pays for each weight tile's
// exchange, so two row tiles share one before two column tiles do (down, us, cold and
// from L2, 128 rows: 1 x 2 7.8 and 6.9, 2 x 1 9.7 and 9.1, 2 x 2 11.3 and 9.3; o at 128
// rows 2 x 1 4.3 and 3.9, 1 x 2 4.6 and 4.2).
template <bool XPACK>
static hipError_t launch_row(const LinearArgs& a, int cus, hipStream_t s) {
  const int64_t mt = (a.M + 15) / 16, nt = a.N / 16;
  const bool wide = a.K > 32 * 4 * 14;
  if (mt * nt <= cus)
    return wide ? launch_tile<8, 1, 1, 10, false, false, XPACK, true>(a, s)
                : launch_tile<4, 1, 1, 8, false, false, XPACK, true>(a, s);
  if (wide && mt > 1 && (mt + 1) / 2 * nt <= cus)
    return launch_tile<8, 1, 2, 10, false, false, XPACK, true>(a, s);
  if (mt == 1 || (!wide && mt * ((nt + 1) / 2) <= cus))
    return wide ? launch_tile<8, 2, 1, 10, false, false, XPACK, true>(a, s)
                : launch_tile<4, 2, 1, 8, false, false, XPACK, true>(a, s);
  return wide ? launch_tile<8, 2, 2, 8, false, false, XPACK, true>(a, s)
              : launch_tile<4, 2, 2, 8, false, false, XPACK, true>(a, s);
}

hipError_t launch_decode_linear(const LinearArgs& a, bool x_packed, bool silu, int cus,
                                hipStream_t s) {
  if (a.ldw) return x_packed ? launch_row<true>(a, cus, s) : launch_row<false>(a, cus, s);
  if (!silu) {
    if (a.norm) return launch_plain<true, true>(a, cus, s);
    return x_packed ? launch_plain<false, true>(a, cus, s) : launch_plain<false, false>(a, cus, s);
  }
  const int64_t mt = (a.M + 15) / 16, nt = a.N / 16;
  const int64_t by2 = (nt + 1) / 2, by3 = (nt + 2) / 3;
  if (mt == 1 || mt * by2 <= cus) return launch_tile<4, 4, 1, 7, true, true, true>(a, s);
  if (mt == 2 || (mt + 1) / 2 * by2 <= cus) return launch_tile<4, 4, 2, 4, true, true, true>(a, s);
  if (mt == 3 || (mt + 1) / 2 * by3 <= cus) return launch_tile<4, 6, 2, 4, true, true, true>(a, s);
  return launch_tile<4, 6, 4, 2, true, true, true>(a, s);
}

hipError_t launch_pack_rows(const f16* x, int64_t ldx, f16* y, float* ss, int rows, int K,
                            hipStream_t s) {
  pack_rows_kernel<<<rows, 256, 0, s>>>(x, ldx, y, ss, K);
  return hipGetLastError();
}

}  // namespace pa
