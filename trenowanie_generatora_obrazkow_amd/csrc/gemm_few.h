// Grouped GEMM for few rows per expert (prompts and small batches over many experts), forward projections with the
// weights N-contiguous: the launch streams every weight once and is bound by how many of their bytes are in flight.
//
// The persistent kernel (gemm.hip) gives a CU one 256x256 tile or two 128x128 ones: most of its ring and copy slots hold
// rows of A, of which there are few here, and each tile's prologue (counts, expert scan, row ids), short main loop and
// epilogue follow one another.  Here a workgroup is one tile of 32 FR rows x 64 columns per wave (two waves with 32 rows,
// four otherwise; SwiGLU: half of the columns are gate columns, half the matching up ones) and a CU holds two to six of
// them, so one fills its ring while another multiplies or stores; what a tile's epilogue reads (row scatter index, routing
// weight, column scales) is loaded ahead of its first copy.  Four waves side by side give 256-byte (16-bit) or 128-byte
// (int8) pieces of a gate row: half-line pieces measured up to 25% slower.  A shallow ring and more workgroups per CU beat a
// deep ring (d 2048, h 320, 128 int8 experts, 4 rows per expert, down: rings of 12, 8, 6, 5 and 4 slices with 32 rows 50.6,
// 36.4, 28.9, 23.8 and 22.7 us), but only with that many workgroups: with one per CU and a long reduction the two or three
// slices in flight do not cover their latency, and the rule (gemm.hip) leaves such launches to the persistent kernel.
// The ring is NS slices of 32 k deep with NS - 1 in flight; every iteration issues a whole slice (past K: copies outside
// the range, which move nothing), so the wait counts are constants.
//
// The products and their order in k are those of the persistent kernel (the same 32x32x16 MFMAs in k order from zero), and
// so are the roundings of the epilogues: the results are bit-identical.
//
// Measured inside whole calls whose weights come from HBM (GB/s of weights): 24 tokens, top-6 of 64 int8 experts, d 2048,
// h 1408: gate/up 126 -> 66.7 us (5000), down 63 -> 36.4 (4600); 64 tokens, top-8 of 128, h 320: 68.8 -> 43.2 (3900) and
// 37.2 -> 27.3 (3070).
#pragma once
#include "gemm_common.h"

namespace hmoe {

template <int FR_, int W_, int NS_, int BE_>
struct FewCfg {
  static constexpr int FR = FR_, NWAVES = W_, NS = NS_, BE = BE_;  // row fragments, waves, ring slices, bytes per weight
  static constexpr int BM = 32 * FR, BN = 64 * NWAVES, NT = 64 * NWAVES;
  static constexpr int A_BYTES = BM * kBK * 2, B_BYTES = BN * kBK * BE, STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int LDS_BYTES = NS * STAGE_BYTES;
};
constexpr int kFewMaxE = 256;           // experts: four per lane in the scan of the counts
constexpr int64_t kFewMaxM = 1 << 20;  // rows (32-bit row arithmetic)
static_assert(kFewMaxE * kFewMaxM < INT32_MAX, "sums of counts, each at most M");

template <class C, int EPI, bool F16>
__global__ __launch_bounds__(C::NT, 2) void few_rows_gemm_kernel(GemmParams p, int nb_n) {
  static_assert(EPI == EPI_STORE || EPI == EPI_SWIGLU, "forward epilogues");
  using X = Elt<F16>;
  using TA = KTile<C::BM, C::NWAVES>;
  using TB = typename TileSel<true, C::BN, C::NWAVES, C::BE, C::NWAVES, F16>::type;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int E = p.E;

  // ---- the workgroup's tile.  The tiles, m-tiles in expert order and each with all its n-tiles in a row, are dealt to the 8
  // XCDs in runs of equal length (workgroups go to the XCDs in turn, so those with the same id modulo 8 share one): the XCDs
  // have equal shares whichever and however few experts the tokens picked, an expert's further m-tiles read its weights
  // again soon after its first one and from the same L2, and so do two n-tiles that share a weight line (64-byte halves with
  // int8 gate / up columns).  Same tile against whole m-tiles dealt to the XCDs in runs, 16-bit gate/up, geometric means:
  // fewer than 8 rows per expert 0.92-0.97, 8 to 64 rows 0.95-0.99, 64 on 0.97 (one expert on one token, K 1024, h 4096: 19
  // us, now 10); down projections within 1%.  (Every expert's first m-tile ahead of all further ones: 0.5-2.5% slower.)
  // Each wave scans the counts by itself, up to four experts per lane.
  const int M = (int)p.M, per = (E + 63) / 64;
  int cnt[4], rs = 0, tl = 0;  // counts of the lane's experts; their rows and m-tiles
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = lane * per + i;
    int64_t c = 0;
    if (i < per && e < E) c = read_count(p.counts, p.counts64, e);
    cnt[i] = (int)(c < 0 ? 0 : (c > M ? M : c));
    rs += cnt[i];  // (at most kFewMaxE * kFewMaxM, also where the counts name more rows than there are)
    tl += (cnt[i] + C::BM - 1) / C::BM;
  }
  int irs = rs, itl = tl;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const int a = __shfl_up(irs, s, 64), b = __shfl_up(itl, s, 64);
    if (lane >= s) {
      irs += a;
      itl += b;
    }
  }
  int st = irs - rs;  // the lane's first row
  if (__builtin_amdgcn_readfirstlane(__shfl(irs, 63, 64)) > M) {  // more rows counted than there are: only those below M
    tl = 0;
#pragma unroll
    for (int i = 0, r = st; i < 4; ++i) {
      cnt[i] = max(0, min(cnt[i], M - r));
      r += cnt[i];
      tl += (cnt[i] + C::BM - 1) / C::BM;
    }
    itl = tl;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const int b = __shfl_up(itl, s, 64);
      if (lane >= s) itl += b;
    }
  }
  const int total = __builtin_amdgcn_readfirstlane(__shfl(itl, 63, 64));
  const int share = (total * nb_n + 7) >> 3, at = (int)blockIdx.x >> 3;  // tiles per XCD, and the workgroup's in its run
  const int tile = ((int)blockIdx.x & 7) * share + at;
  if (at >= share || tile >= total * nb_n) return;
  const int mt = tile / nb_n, nb = tile - mt * nb_n;
  const int ol = __builtin_ctzll(__ballot(itl > mt));  // lanes are in expert order: the first one holds the tile
  int left = mt - __shfl(itl - tl, ol, 64), first = __shfl(st, ol, 64), e = -1, row0 = 0, row_end = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = __shfl(cnt[i], ol, 64), t = (c + C::BM - 1) / C::BM;
    if (e < 0 && left < t) {
      e = ol * per + i;
      row0 = first + left * C::BM;
      row_end = min(first + c, row0 + C::BM);
    }
    left -= t;
    first += c;
  }
  e = __builtin_amdgcn_readfirstlane(e);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  row_end = __builtin_amdgcn_readfirstlane(row_end);
  const int n0 = nb * (EPI == EPI_SWIGLU ? C::BN / 2 : C::BN);

  // ---- copy sources ----
  TA ta;
  TB tb;
  ta.K = p.K;
  ta.rsrc = make_rsrc(p.a_idx ? p.A : p.A + (int64_t)row0 * p.lda);
#pragma unroll
  for (int i = 0; i < TA::PER_WAVE; ++i) {
    const int rr = TA::row_of(wave, lane, i);
    const int c = (lane & 3) ^ swz_k(rr);
    ta.voff[i] = kOOB;
    if (row0 + rr < row_end) {
      const int64_t src = p.a_idx ? (int64_t)p.a_idx[row0 + rr] : (int64_t)rr;
      ta.voff[i] = (uint32_t)(src * p.lda * 2 + c * 16);
    }
    ta.chunk[i] = c;
  }
  tb.rsrc = make_rsrc(static_cast<const char*>(p.B) + (int64_t)e * p.strideBe * C::BE);
  tb.kstep = (uint32_t)(p.ldb * C::BE);
  tb.Kvalid = p.K;
#pragma unroll
  for (int i = 0; i < TB::PER_WAVE; ++i) {
    int k, nn;
    TB::slot(wave, lane, i, k, nn);
    int col = n0 + nn;
    bool ok = col < p.N;
    if (EPI == EPI_SWIGLU) {  // tile columns [0, BN / 2) gate, [BN / 2, BN) the matching up
      const int ac = n0 + nn % (C::BN / 2);
      col = nn / (C::BN / 2) * p.h + ac;
      ok = ac < p.N;
    }
    tb.krow[i] = k;
    tb.voff[i] = ok ? (uint32_t)(((int64_t)k * p.ldb + col) * C::BE) : kOOB;
  }

  // ---- epilogue inputs, loaded ahead of the copies: the lane's rows' scatter index and scale (row a*32 + lane%32), and
  // with int8 weights its columns' scales (halves b of BN / 2 columns, groups g; a lane holds 4 consecutive columns per group) ----
  [[maybe_unused]] int yr[C::FR];
  [[maybe_unused]] float sc[C::FR];
  if constexpr (EPI == EPI_STORE) {
#pragma unroll
    for (int a = 0; a < C::FR; ++a) {
      const int row = row0 + a * 32 + (lane & 31);
      yr[a] = row;
      sc[a] = 1.0f;  // the product is then exact
      if (row < row_end) {
        if (p.y_idx) yr[a] = p.y_idx[row];
        if (p.scale)
          sc[a] = p.scale_f32 ? static_cast<const float*>(p.scale)[row]
                              : X::one(static_cast<const uint16_t*>(p.scale)[row]);
      }
    }
  }
  [[maybe_unused]] float cs[2][4][4];
  if constexpr (C::BE == 1) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int lc = wave * 32 + 8 * g + 4 * (lane >> 5);
        const int col = EPI == EPI_SWIGLU ? b * p.h + n0 + lc : n0 + C::BN / 2 * b + lc;
        const bool ok = (EPI == EPI_SWIGLU ? n0 + lc : col) < p.N;
        const int64_t at = (int64_t)e * p.ldws + col;
        float* v = cs[b][g];
        if (p.w_scale_f32) {
          const float4 w = ok ? *reinterpret_cast<const float4*>(static_cast<const float*>(p.w_scale) + at)
                              : make_float4(0.f, 0.f, 0.f, 0.f);
          v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
        } else {
          const uint2 w = ok ? *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p.w_scale) + at)
                             : make_uint2(0u, 0u);
          v[0] = bf_lo(w.x); v[1] = bf_hi(w.x); v[2] = bf_lo(w.y); v[3] = bf_hi(w.y);
        }
      }
  }

  // ---- main loop ----
  constexpr int LOADS = TA::PER_WAVE + TB::PER_WAVE;
  const int nk = (p.K + kBK - 1) / kBK;
  auto issue = [&](int s) {  // slice s into its slot; past the last slice copies that move nothing
    char* slot = smem + (s % C::NS) * C::STAGE_BYTES;
    if (s < nk) {
      ta.issue(slot, wave, lane, s * kBK);
      tb.issue(slot + C::A_BYTES, wave, lane, s * kBK);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) buf2lds(kOOB, tb.rsrc, 0u, slot + (wave * LOADS + i) * 1024);
    }
  };
  const int loff_a = TA::lane_off(0, lane), loff_b = TB::lane_off(wave & 1, lane);
  f32x16 acc[C::FR][2];
#pragma unroll
  for (int a = 0; a < C::FR; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
  auto main_loop = [&](auto fe_tag) {  // FE: row fragments holding rows (of FR)
    constexpr int FE = decltype(fe_tag)::value;
#pragma unroll
    for (int s = 0; s < C::NS - 1; ++s) issue(s);
    uint32_t cons = 0, fill = (C::NS - 1) * C::STAGE_BYTES;  // ring offsets: the slot filled is that of slice kt - 1
    const uint32_t pa = lds_addr(smem) + wave * (TA::PER_WAVE * 1024);
    const uint32_t pb = lds_addr(smem) + C::A_BYTES + wave * (TB::PER_WAVE * 1024);
    auto iter = [&](int kt, auto fast_tag) {
      wait_vm<(C::NS - 2) * LOADS>();  // this wave's copies of slice kt have landed
      lds_barrier();                   // and the others'; all have read slice kt - 1, whose slot is filled next
      if constexpr (decltype(fast_tag)::value) {
        const int k0 = (kt + C::NS - 1) * kBK;
        const uint32_t sa = ta.soff_of(k0), sb = tb.soff_of(k0);
        static_for<TA::PER_WAVE>([&](auto l) { ta.template issue_inner<decltype(l)::value>(pa + fill, sa); });
        static_for<TB::PER_WAVE>([&](auto l) { tb.template issue_inner<decltype(l)::value>(pb + fill, sb); });
      } else {
        issue(kt + C::NS - 1);
      }
      const char* slot = smem + cons;
      fill = cons;
      cons += C::STAGE_BYTES;
      if (cons == C::LDS_BYTES) cons = 0;
      bf16x8 xa[2][FE], wb[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int b = 0; b < 2; ++b) wb[ks][b] = TB::frag(slot + C::A_BYTES, b * (C::BN / 2) + 64 * (wave >> 1), loff_b, ks);
#pragma unroll
        for (int a = 0; a < FE; ++a) xa[ks][a] = TA::frag(slot, 32 * a, loff_a, ks);
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int a = 0; a < FE; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = mfma16<F16>(wb[ks][b], xa[ks][a], acc[a][b]);
    };
    const int nfast = max(0, p.K / kBK - (C::NS - 1));
    int kt = 0;
    for (; kt < nfast; ++kt) iter(kt, std::true_type{});
    for (; kt < nk; ++kt) iter(kt, std::false_type{});
  };
  const int live = row_end - row0;
  if (C::FR >= 2 && live <= 32)
    main_loop(std::integral_constant<int, 1>{});
  else if (C::FR >= 4 && live <= 64)
    main_loop(std::integral_constant<int, 2>{});
  else
    main_loop(std::integral_constant<int, C::FR>{});
  wait_vm<0>();

  // ---- epilogue: a lane holds row a*32 + lane%32 and, per group g, 4 consecutive columns; it stores them itself (8
  // bytes: with few rows the outputs are a few percent of the weights' bytes) ----
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int lc = wave * 32 + 8 * g + 4 * (lane >> 5);  // column within a half (BN / 2) of the tile
    if constexpr (EPI == EPI_SWIGLU) {
      const int col = n0 + lc;
      if (col >= p.N) continue;
#pragma unroll
      for (int a = 0; a < C::FR; ++a) {
        const int64_t row = row0 + a * 32 + (lane & 31);
        if (row >= row_end) continue;
        float gs[4], us[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          gs[t] = acc[a][0][4 * g + t];
          us[t] = acc[a][1][4 * g + t];
          if constexpr (C::BE == 1) {
            gs[t] *= cs[0][g][t];
            us[t] *= cs[1][g][t];
          }
        }
        // act = R(R(silu(g)) * u) with g, u the rounded projections (R: to bf16, or fp16 with F16)
        uint32_t o[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const uint32_t gb = X::pack2(gs[2 * t], gs[2 * t + 1]), ub = X::pack2(us[2 * t], us[2 * t + 1]);
          const uint32_t sl = X::pack2(silu_f(X::lo(gb)), silu_f(X::hi(gb)));
          o[t] = X::pack2(X::lo(sl) * X::lo(ub), X::hi(sl) * X::hi(ub));
        }
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.C) + row * p.ldc + col) = make_uint2(o[0], o[1]);
      }
    } else {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int col = n0 + C::BN / 2 * b + lc;
        if (col >= p.N) continue;
#pragma unroll
        for (int a = 0; a < C::FR; ++a) {
          const int64_t row = row0 + a * 32 + (lane & 31);
          if (row >= row_end) continue;
          float v[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            v[t] = acc[a][b][4 * g + t];
            if constexpr (C::BE == 1) v[t] *= cs[b][g][t];  // the column scale first, then the row scale
            v[t] *= sc[a];
          }
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.C) + (int64_t)yr[a] * p.ldc + col) =
              make_uint2(X::pack2(v[0], v[1]), X::pack2(v[2], v[3]));
        }
      }
    }
  }
}

}  // namespace hmoe
