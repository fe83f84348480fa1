// Grouped GEMM for copies with few rows, included by grouped_gemm.hip.
//
// With some tens of rows per copy a 256 x 256 tile multiplies mostly padding
// and the call is bound by reading every copy's weights once.  What the
// 256-row kernels lack there is bytes in flight: one block per CU with one
// 64-deep K-tile (32 KB of weights) on its way at a time.  This kernel keeps
// more of the stream in flight on a smaller footprint: BM x BN tiles, K in
// steps of KT, through a ring of NST stages filled by buffer->LDS loads
// NST - 1 K-tiles ahead (waited for by count), small enough for several
// blocks per CU, whose epilogues and tile switches overlap each other's loads.
//
// The ragged tile walk is that of the other kernels (m-tiles of BM rows per
// group), n fastest, so that the m-tiles of a group, which share weight
// strips, run close together on one XCD.  LDS operand layouts, the MFMA
// (16x16x32) and the rounding points are those of the four-wave kernel.  The
// accumulator holds output tiles transposed (lane l: row l%16, columns
// 4*(l/16) .. +3), so outputs leave as 8-byte row pieces straight from
// registers; the L2 merges them into lines.
namespace fr {

constexpr int kMaxG = 1024;  // groups (the m-tile prefix in LDS)

// WM x WN waves, each FM x FN tiles of 16 x 16; NST stages; BPC blocks per CU.
template <int WM_, int WN_, int FM_, int FN_, int NST_, int BPC_>
struct Cfg {
  static constexpr int WM = WM_, WN = WN_, FM = FM_, FN = FN_, NST = NST_, BPC = BPC_;
  static constexpr int KS = 2;                     // k-steps (the MFMA's 32) of a K-tile
  static constexpr int KT = 32 * KS;               // depth of a K-tile
  static constexpr int CHK = KT / 8;               // 16-byte chunks of a K-contiguous row
  static constexpr int RPL = 64 / CHK;             // such rows per load
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int BM = WM * FM * 16, BN = WN * FN * 16;
  static constexpr int A_BYTES = BM * KT * 2, B_BYTES = BN * KT * 2, STAGE = A_BYTES + B_BYTES;
  static constexpr int PA = A_BYTES / 1024, PB = B_BYTES / 1024;    // 1 KB loads per K-tile
  static constexpr int QA = PA / NW, QB = PB / NW;                  // ... of one wave
  static_assert(PB % NW == 0 && PA % NW == 0, "whole loads per wave");
  static_assert(FN % 2 == 0 && NST >= 2 && (NST - 2) * (QA + QB) <= 63, "configuration");
};

// Operand loads of one wave for one output tile: the lane's byte offset of
// load q0 (kOOB: outside the operand's rows or columns), and whether the lane
// lies within K in the partial last K-tile (bit q0 of tmask).
template <int Q>
struct Op {
  __amdgpu_buffer_rsrc_t r0, r1;  // r1: k-rows from `split` on (NN with two weight tensors)
  uint32_t off[Q];
  uint32_t tmask;
  uint32_t kstep;  // offset per K-tile
};

// K-contiguous operand rows (row, KT k): load q fills rows RPL*q .. +RPL-1,
// lane i row RPL*q + i/CHK, physical chunk i%CHK = logical chunk ^ kc_swz(row).
// `src(row)` is the row's index in the operand, negative past its end.
template <class CF, int Q, typename F>
__device__ __forceinline__ void kc_setup(Op<Q>& op, int wave, int lane, int64_t ldb, int krem, F src) {
  op.tmask = 0;
  op.kstep = CF::KT * 2;
#pragma unroll
  for (int q0 = 0; q0 < Q; ++q0) {
    const int row = (q0 * CF::NW + wave) * CF::RPL + lane / CF::CHK;
    const int c = (lane % CF::CHK) ^ kc_swz(row);
    const int64_t r = src(row);
    op.off[q0] = r >= 0 ? (uint32_t)(r * ldb) + (uint32_t)c * 16u : kOOB;
    op.tmask |= (c * 8 < krem ? 1u : 0u) << q0;
  }
}

template <int KIND, class CF>
struct Tile {
  TileInfo i;
  Op<CF::QA> A;
  Op<CF::QB> B;
};

template <int KIND, class CF>
__device__ __forceinline__ void setup(const GemmParams& P, Tile<KIND, CF>& tc, int wave, int lane) {
  asm volatile("" : "+v"(lane));  // keep the per-lane arithmetic here
  const TileInfo& ti = tc.i;
  const int krem = (int)(P.K - (P.K - 1) / CF::KT * CF::KT);  // k of the last K-tile
  const int64_t left = ti.row_end - ti.row0;
  const int64_t rows = left < CF::BM ? left : CF::BM;
  tc.A.r0 = tc.A.r1 = make_rsrc(P.a.p0 + (int64_t)ti.row0 * P.a.ld, (uint64_t)rows * P.a.ld * 2);
  kc_setup<CF>(tc.A, wave, lane, P.a.ld * 2, krem, [&](int row) { return row < rows ? (int64_t)row : -1; });
  const bf16_t* b0 = P.b.p0 + (int64_t)ti.g * P.b.gs0;
  const bf16_t* b1 = P.b.p1 + (int64_t)ti.g * P.b.gs1;
  if constexpr (KIND == KIND_FC1) {
    // Virtual B rows alternate 16 gate rows (r0) and the matching 16 up rows (r1).
    tc.B.r0 = make_rsrc(b0, (uint64_t)P.I * P.K * 2);
    tc.B.r1 = make_rsrc(b1, (uint64_t)P.I * P.K * 2);
    const int64_t j0 = (int64_t)ti.ntile * (CF::BN / 2);
    kc_setup<CF>(tc.B, wave, lane, P.K * 2, krem, [&](int row) {
      const int64_t j = j0 + (row >> 5) * 16 + (row & 15);
      return j < P.I ? j : (int64_t)-1;
    });
  } else if constexpr (KIND == KIND_NT) {
    const int64_t n0 = (int64_t)ti.ntile * CF::BN;
    tc.B.r0 = tc.B.r1 = make_rsrc(b0 + n0 * P.K, (uint64_t)(P.N - n0) * P.K * 2);
    kc_setup<CF>(tc.B, wave, lane, P.K * 2, krem, [&](int row) { return n0 + row < P.N ? (int64_t)row : (int64_t)-1; });
  } else {
    // B[g] is [K][N]: load q fills k-rows q*ROWS .. +ROWS-1 of the K-tile, lane
    // i k-row q*ROWS + i/CH, physical chunk i%CH = logical chunk ^ mn_swz.
    constexpr int CH = CF::BN / 8, ROWS = 64 / CH;
    const int64_t split = P.b.split < P.K ? P.b.split : P.K;
    tc.B.r0 = make_rsrc(b0, (uint64_t)split * P.N * 2);
    tc.B.r1 = make_rsrc(b1, (uint64_t)(P.K - split) * P.N * 2);
    tc.B.kstep = (uint32_t)(CF::KT * P.N * 2);
    tc.B.tmask = 0;
#pragma unroll
    for (int q0 = 0; q0 < CF::QB; ++q0) {
      const int krow = (q0 * CF::NW + wave) * ROWS + lane / CH;
      const int c = (lane % CH) ^ w4::mn_swz(krow);
      const int64_t col = (int64_t)ti.ntile * CF::BN + c * 8;
      tc.B.off[q0] = col < P.N ? (uint32_t)(krow * P.N * 2 + col * 2) : kOOB;
      tc.B.tmask |= (krow < krem ? 1u : 0u) << q0;
    }
  }
}

// Load J of this wave's share of K-tile kt into `stage` (A: 0 .. QA-1, B: QA ..
// QA+QB-1).
template <int KIND, class CF, int J>
__device__ __forceinline__ void issue(const GemmParams& P, char* stage, const Tile<KIND, CF>& tc, int32_t kt, int wave) {
  const bool tail = (int64_t)(kt + 1) * CF::KT > P.K;
  if constexpr (J < CF::QA) {
    const int q = J * CF::NW + wave;
    dma16(tc.A.r0, stage + q * 1024, tail && !((tc.A.tmask >> J) & 1u) ? kOOB : tc.A.off[J], (uint32_t)kt * tc.A.kstep);
  } else {
    constexpr int q0 = J - CF::QA;
    const int q = q0 * CF::NW + wave;
    __amdgpu_buffer_rsrc_t rb = tc.B.r0;
    uint32_t soff = (uint32_t)kt * tc.B.kstep;
    if constexpr (KIND == KIND_FC1) rb = ((q * CF::RPL) >> 4) & 1 ? tc.B.r1 : tc.B.r0;
    if constexpr (KIND == KIND_NN) {
      // the host sends two weight tensors here only when the split is a whole number of K-tiles
      const int32_t ksplit = (int32_t)((P.b.split < P.K ? P.b.split : P.K + CF::KT - 1) / CF::KT);
      if (kt >= ksplit) {
        rb = tc.B.r1;
        soff = (uint32_t)(kt - ksplit) * tc.B.kstep;
      }
    }
    dma16(rb, stage + CF::A_BYTES + q * 1024, tail && !((tc.B.tmask >> q0) & 1u) ? kOOB : tc.B.off[q0], soff);
  }
}

template <class CF>
struct Frags {
  bf16x8_t a[CF::FM], b[CF::FN];
};

// The I-th fragment read of a k-step, in the order its (mt-major) MFMAs use
// them: A0, B0 .. B(FN-1), A1 .. ; ids as in the reads (A first, then B).
template <class CF>
constexpr int order(int i) { return i == 0 ? 0 : i <= CF::FN ? CF::FM + i - 1 : i - CF::FN; }

// Four consecutive outputs of a row (8 bytes).
__device__ __forceinline__ void st4(bf16_t* p, uint2 v) { *reinterpret_cast<uint2*>(p) = v; }
__device__ __forceinline__ uint2 ld4(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }

template <int KIND, class CF>
__device__ __forceinline__ void epilogue(const GemmParams& P, const TileInfo& ti, int wm, int wn, int lane,
                                         const f32x4_t (&acc)[CF::FM][CF::FN]) {
  asm volatile("" : "+v"(lane));
  const int c4 = (lane >> 4) * 4;
#pragma unroll
  for (int mt = 0; mt < CF::FM; ++mt) {
    const int64_t r = (int64_t)ti.row0 + (wm * CF::FM + mt) * 16 + (lane & 15);
    if (r >= ti.row_end) continue;
    if constexpr (KIND == KIND_FC1) {
      const int64_t I = P.I;
      const float wt = P.row_w != nullptr ? Elt::to_f32(P.row_w[r]) : 0.f;
#pragma unroll
      for (int nt = 0; nt < CF::FN; nt += 2) {
        const int64_t j = (int64_t)ti.ntile * (CF::BN / 2) + (wn * CF::FN + nt) * 8 + c4;
        if (j >= I) continue;
        const f32x4_t g4 = acc[mt][nt], u4 = acc[mt][nt + 1];
        st4(P.gu + r * 2 * I + j, pack4(g4[0], g4[1], g4[2], g4[3]));
        st4(P.gu + r * 2 * I + I + j, pack4(u4[0], u4[1], u4[2], u4[3]));
        float g[4], u[4];
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          g[e] = g4[e], g[e + 1] = g4[e + 1], u[e] = u4[e], u[e + 1] = u4[e + 1];
          Elt::round2(g[e], g[e + 1]);
          Elt::round2(u[e], u[e + 1]);
          g[e] = silu_f32(g[e]), g[e + 1] = silu_f32(g[e + 1]);
          Elt::round2(g[e], g[e + 1]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] *= u[e];
        if (P.row_w != nullptr) {  // the weight on the rounded activation (non-EP fc2 input)
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            Elt::round2(g[e], g[e + 1]);
            g[e] *= wt, g[e + 1] *= wt;
          }
        }
        st4(P.act + r * I + j, pack4(g[0], g[1], g[2], g[3]));
      }
    } else if constexpr (KIND == KIND_NNS) {
      const int64_t I = P.I;
#pragma unroll
      for (int nt = 0; nt < CF::FN; nt += 2) {
        const int64_t ja = (int64_t)ti.ntile * CF::BN + (wn * CF::FN + nt) * 16 + c4, jb = ja + 16;
        // columns past I: read column ja's place again, write nothing
        const bool ina = ja < I, inb = jb < I;
        const bf16_t* gr = P.gin + r * 2 * I;
        const int64_t la = ina ? ja : 0, lb = inb ? jb : 0;
        const uint2 ga = ld4(gr + la), gb = ld4(gr + lb), ua = ld4(gr + I + la), ub = ld4(gr + I + lb);
        const uint2 da = w4::bf16x4(acc[mt][nt]), db = w4::bf16x4(acc[mt][nt + 1]);
        float d[8], g[8], u[8], dg[8], du[8];
        unpack8e<Elt>(make_uint4(da.x, da.y, db.x, db.y), d);
        unpack8e<Elt>(make_uint4(ga.x, ga.y, gb.x, gb.y), g);
        unpack8e<Elt>(make_uint4(ua.x, ua.y, ub.x, ub.y), u);
        swiglu_bwd8<Elt>(d, g, u, dg, du);
        const uint4 pg = pack8e<Elt>(dg), pu = pack8e<Elt>(du);
        bf16_t* o = P.c0 + r * 2 * I;
        if (ina) st4(o + ja, make_uint2(pg.x, pg.y)), st4(o + I + ja, make_uint2(pu.x, pu.y));
        if (inb) st4(o + jb, make_uint2(pg.z, pg.w)), st4(o + I + jb, make_uint2(pu.z, pu.w));
      }
    } else {
      const bool mapped = P.row_tok != nullptr;
      const int32_t tok = mapped ? P.row_tok[r] : -1;
      const bool to = mapped && (uint32_t)tok < (uint32_t)P.M;
      const float wt = KIND == KIND_NT && mapped ? Elt::to_f32(P.row_w[r]) : 0.f;
#pragma unroll
      for (int nt = 0; nt < CF::FN; ++nt) {
        const int64_t col = (int64_t)ti.ntile * CF::BN + (wn * CF::FN + nt) * 16 + c4;
        if (col >= P.N) continue;
        const uint2 v = w4::bf16x4(acc[mt][nt]);
        if (KIND == KIND_NN && mapped) {
          if (to) st4(P.c0 + (int64_t)tok * P.ldc + col, v);
          continue;
        }
        st4(P.c0 + r * P.ldc + col, v);
        if (to) {
          // the combine kernel's rounding: 0 + bf16(f * w), as fma(f, w, 0)
          float f[4];
          Elt::unpack2(v.x, f[0], f[1]);
          Elt::unpack2(v.y, f[2], f[3]);
#pragma unroll
          for (int e = 0; e < 4; ++e) f[e] = __builtin_fmaf(f[e], wt, 0.f);
          st4(P.cout + (int64_t)tok * P.ldc + col, pack4(f[0], f[1], f[2], f[3]));
        }
      }
    }
  }
}

template <int KIND, class CF>
__global__ __launch_bounds__(CF::NT, CF::NW * CF::BPC / 4) void few_rows_grouped_gemm_kernel(GemmParams P) {
  static_assert(KIND != KIND_TN, "ragged rows only");
  constexpr int NW = CF::NW, L = CF::QA + CF::QB;
  __shared__ __attribute__((aligned(1024))) char lds[CF::NST * CF::STAGE];
  __shared__ int32_t tpre[kMaxG + 1];
  __shared__ int32_t wsum[NW];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = uni(t >> 6);
  const int wm = wave / CF::WN, wn = wave % CF::WN;
  const int G = P.G;

  // Exclusive prefix of the groups' m-tiles in tpre[0..G]: consecutive groups
  // per thread, a wave scan of the threads' sums, then the waves' sums.
  {
    const int per = (G + CF::NT - 1) / CF::NT;
    const int g0 = t * per, g1 = g0 + per < G ? g0 + per : G;
    int32_t sum = 0;
    for (int g = g0; g < g1; ++g) sum += (P.offsets[g + 1] - P.offsets[g] + CF::BM - 1) / CF::BM;
    int32_t inc = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t v = __shfl_up(inc, off, 64);
      if (lane >= off) inc += v;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int32_t run = inc - sum;
    for (int w = 0; w < wave; ++w) run += wsum[w];
    for (int g = g0; g < g1; ++g) {
      tpre[g] = run;
      run += (P.offsets[g + 1] - P.offsets[g] + CF::BM - 1) / CF::BM;
    }
    if (t == CF::NT - 1) tpre[G] = run;
    __syncthreads();
  }
  const int32_t ntn = (int32_t)(KIND == KIND_FC1 ? (P.I + CF::BN / 2 - 1) / (CF::BN / 2) : (P.N + CF::BN - 1) / CF::BN);
  const int64_t total = (int64_t)uni(tpre[G]) * ntn;
  const int32_t nk = (int32_t)((P.K + CF::KT - 1) / CF::KT);
  // Blocks go round-robin over the XCDs: each XCD walks its own eighth of the
  // tile list (so a weight strip's tiles meet in one L2), its blocks
  // round-robin within it.
  int64_t first = blockIdx.x, step = gridDim.x, end = total;
  if (gridDim.x % kNumXcd == 0) {
    const int64_t x = blockIdx.x % kNumXcd;
    step = gridDim.x / kNumXcd;
    end = total * (x + 1) / kNumXcd;
    first = total * x / kNumXcd + blockIdx.x / kNumXcd;
  }
  if (first >= end) return;

  // Tile order: group by group, within a group n-tile by n-tile with its
  // m-tiles (which read the same weight strip) next to each other.
  auto decode = [&](int64_t tile, TileInfo& ti) {
    const int32_t m = (int32_t)(tile / ntn);
    int lo = 0, hi = G - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (uni(tpre[mid]) <= m) lo = mid;
      else hi = mid - 1;
    }
    const int32_t m0 = uni(tpre[lo]), gm = uni(tpre[lo + 1]) - m0;
    const int32_t local = (int32_t)(tile - (int64_t)m0 * ntn);
    ti.g = lo;
    ti.ntile = local / gm;
    ti.mtile = local - ti.ntile * gm;
    ti.row0 = uni(P.offsets[lo]) + ti.mtile * CF::BM;
    ti.row_end = uni(P.offsets[lo + 1]);
    ti.nk = nk;
  };

  // Issue cursor: NST - 1 K-tiles in front of the one being multiplied.
  Tile<KIND, CF> it;
  int64_t i_tile = first;
  // Every tile walks K from 0 as the 256-row kernels do: an output's bits depend
  // on its row and its copy's weights alone, not on the slot that holds the copy
  // or on how many rows the call has.  (Tiles that start at K-tiles of their own
  // spread the K-contiguous weights' reads over the memory channels, but sum in an
  // order of the slot; fc1 183 -> 178 us at 160 copies of 5 rows of 2048 x 768,
  // 158 -> 149 at 32 of 20 rows of 4096 x 1536.)
  int32_t i_kt = 0;
  bool i_live = true;
  auto set_tile = [&]() {
    decode(i_tile, it.i);
    setup<KIND, CF>(P, it, wave, lane);
  };
  set_tile();
  int i_stage = 0;
  auto advance_issue = [&]() {
    i_stage = i_stage + 1 == CF::NST ? 0 : i_stage + 1;
    if (!i_live || ++i_kt < nk) return;
    i_kt = 0;
    i_tile += step;
    if (i_tile < end) {
      set_tile();
    } else {
      // past the block's last K-tile: loads out of range, so that every
      // K-tile issues the same number
      i_live = false;
#pragma unroll
      for (int q = 0; q < CF::QA; ++q) it.A.off[q] = kOOB;
#pragma unroll
      for (int q = 0; q < CF::QB; ++q) it.B.off[q] = kOOB;
    }
  };
#pragma unroll
  for (int s = 0; s < CF::NST - 1; ++s) {
    static_for<0, L>([&](auto j) __attribute__((always_inline)) {
      issue<KIND, CF, decltype(j)::value>(P, lds + i_stage * CF::STAGE, it, i_kt, wave);
    });
    advance_issue();
  }

  // K-contiguous fragments: lane l reads row rb + l%16, chunk ks*4 + l/16
  int32_t sa[CF::KS];
#pragma unroll
  for (int ks = 0; ks < CF::KS; ++ks) {
    const int r = lane & 15;
    sa[ks] = r * (CF::KT * 2) + (((ks * 4 + (lane >> 4)) ^ kc_swz(r)) << 4);
  }
  // fragments of [KT][BN] tiles: the lane's offset of each column block
  int32_t sb[CF::FN];
  if constexpr (b_is_mn<KIND>()) {
    const int g = lane >> 4, i = lane & 15;
    const int s = w4::mn_swz(g * 8 + (i >> 2));
#pragma unroll
    for (int n = 0; n < CF::FN; ++n) {
      const int c = (wn * CF::FN + n) * 2 + ((i & 3) >> 1);
      sb[n] = (g * 8 + (i >> 2)) * (2 * CF::BN) + (i & 1) * 8 + ((c ^ s) << 4);
    }
  }
  // Fragment J of k-step ks of `stage`: A 0 .. FM-1, then B.
  auto read = [&](auto jj, const char* stage, int ks, Frags<CF>& f) __attribute__((always_inline)) {
    constexpr int J = decltype(jj)::value;
    if constexpr (J < CF::FM) {
      f.a[J] = *reinterpret_cast<const bf16x8_t*>(stage + (wm * CF::FM + J) * 16 * (CF::KT * 2) + sa[ks]);
    } else if constexpr (b_is_mn<KIND>()) {
      const char* p = stage + CF::A_BYTES + ks * 32 * (2 * CF::BN) + sb[J - CF::FM];
      const bf16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_TR_PTR(p));
      const bf16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_TR_PTR(p + 4 * (2 * CF::BN)));
      f.b[J - CF::FM] = bf16x8_t{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
    } else {
      f.b[J - CF::FM] = *reinterpret_cast<const bf16x8_t*>(
          stage + CF::A_BYTES + (wn * CF::FN + J - CF::FM) * 16 * (CF::KT * 2) + sa[ks]);
    }
  };

  f32x4_t acc[CF::FM][CF::FN];
  Frags<CF> f0, f1;
  constexpr int NM = CF::FM * CF::FN, NR = CF::FM + CF::FN;
  // One k-step of MFMAs from `fm`, in NR groups: each reads one fragment of
  // k-step ks of `stage` into `fr`, and (loads) issues its share of the loads
  // of the K-tile NST - 1 ahead.
  auto kstep = [&](auto first, auto loads, const Frags<CF>& fm, const char* stage, int ks, Frags<CF>& fr)
      __attribute__((always_inline)) {
    char* refill = lds + i_stage * CF::STAGE;
    static_for<0, NR>([&](auto jj) __attribute__((always_inline)) {
      constexpr int j = decltype(jj)::value;
      if constexpr (decltype(loads)::value) {
        static_for<j * L / NR, (j + 1) * L / NR>([&](auto l) __attribute__((always_inline)) {
          issue<KIND, CF, decltype(l)::value>(P, refill, it, i_kt, wave);
        });
      }
      read(Int<order<CF>(j)>{}, stage, ks, fr);
      static_for<j * NM / NR, (j + 1) * NM / NR>([&](auto xx) __attribute__((always_inline)) {
        constexpr int x = decltype(xx)::value, m = x / CF::FN, n = x % CF::FN;
        acc[m][n] = mfma16(fm.b[n], fm.a[m], decltype(first)::value ? f32x4_t{} : acc[m][n]);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // The end of a K-tile: the next one has landed (at most the loads of the
  // NST - 2 K-tiles issued after it are outstanding), and every wave has read
  // this one.
  auto turn = [&]() __attribute__((always_inline)) {
    wait_loads_lds<(CF::NST - 2) * L>();
    block_barrier();
  };

  turn();
  int c_stage = 0;
  for (int64_t tile = first; tile < end; tile += step) {
    // K-tile 0 of the tile: its first k-step has no MFMAs of this tile to run behind.
    {
      const char* stage = lds + c_stage * CF::STAGE;
      static_for<0, NR>([&](auto j) __attribute__((always_inline)) { read(Int<order<CF>(decltype(j)::value)>{}, stage, 0, f0); });
      kstep(Int<1>{}, Int<1>{}, f0, stage, 1, f1);
      advance_issue();
      turn();
      c_stage = c_stage + 1 == CF::NST ? 0 : c_stage + 1;
    }
    for (int32_t kt = 1; kt < nk; ++kt) {
      const char* stage = lds + c_stage * CF::STAGE;
      kstep(Int<0>{}, Int<1>{}, f1, stage, 0, f0);
      kstep(Int<0>{}, Int<0>{}, f0, stage, 1, f1);
      advance_issue();
      turn();
      c_stage = c_stage + 1 == CF::NST ? 0 : c_stage + 1;
    }
#pragma unroll
    for (int m = 0; m < CF::FM; ++m)
#pragma unroll
      for (int n = 0; n < CF::FN; ++n) acc[m][n] = mfma16(f1.b[n], f1.a[m], acc[m][n]);
    TileInfo ti;
    decode(tile, ti);
    epilogue<KIND, CF>(P, ti, wm, wn, lane, acc);
  }
  wait_loads<0>();
}

// Weight gradient of copies with few rows: C[g] = A[rows g]^T B[rows g] with
// one or two 64-row K-tiles, bound by writing C.  The persistent 256 x 256
// kernel spends a tile there on one K-tile and then on an epilogue during
// which the CU does nothing else; here a block computes one 128 x 128 tile
// (4 waves of 64 x 64, 32 KB of LDS, four blocks per CU), so that the blocks
// of a CU load, multiply and store beside each other.  Operands, both
// [64 k][128] in LDS, and fragments as in the other kernels; the output goes
// through the same LDS and leaves as whole 128-byte row pieces.
constexpr int kWgT = 128, kWgNT = 256;

__global__ __launch_bounds__(kWgNT, 4) void few_rows_wgrad_grouped_gemm_kernel(GemmParams P) {
  constexpr int QL = 4;  // 1 KB loads per wave and operand
  __shared__ __attribute__((aligned(1024))) char lds[2 * kWgT * BK * 2];
  char* As = lds;
  char* Bs = lds + kWgT * BK * 2;
  const int lane = threadIdx.x & 63;
  const int wave = uni(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // Copy by copy, each XCD (blocks go round-robin over them) takes an eighth of
  // the copy's tiles, n fastest: a copy with many more rows than the others
  // is spread over the whole chip.  (With whole copies per XCD the one with
  // the hot copies worked alone: 128 copies of 2560 x 1920, 101 rows on
  // average under Zipf(1.0), 784 + 1669 us against 404 + 996 on the persistent
  // kernel.)
  const int64_t ntn = (P.N + kWgT - 1) / kWgT, per_g = (P.M + kWgT - 1) / kWgT * ntn;
  const int64_t per_x = (per_g + kNumXcd - 1) / kNumXcd;
  const int64_t j = blockIdx.x / kNumXcd, g = j / per_x;
  const int64_t tile = (blockIdx.x + g) % kNumXcd * per_x + j % per_x;
  if (tile >= per_g) return;
  const int64_t m0 = tile / ntn * kWgT, n0 = tile % ntn * kWgT;
  const int64_t row0 = P.offsets[g], row_end = P.offsets[g + 1];

  f32x4_t acc[4][4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = f32x4_t{};

  // Load q covers k-rows 4q .. 4q+3, lane i k-row 4q + i/16, physical chunk
  // i%16 = logical chunk ^ mn_swz; k-rows past the copy fail the range check.
  uint32_t oa[QL], ob[QL];
#pragma unroll
  for (int q = 0; q < QL; ++q) {
    const int krow = (q * 4 + wave) * 4 + (lane >> 4);
    const int c = (lane & 15) ^ w4::mn_swz(krow);
    oa[q] = m0 + c * 8 < P.M ? (uint32_t)(krow * P.a.ld * 2 + (m0 + c * 8) * 2) : kOOB;
    ob[q] = n0 + c * 8 < P.N ? (uint32_t)(krow * P.b.ld * 2 + (n0 + c * 8) * 2) : kOOB;
  }
  const int gq = lane >> 4, i16 = lane & 15;
  const int base = (gq * 8 + (i16 >> 2)) * (2 * kWgT) + (i16 & 1) * 8;
  const int sw = w4::mn_swz(gq * 8 + (i16 >> 2));
  auto frag = [&](const char* t, int cb, int ks) __attribute__((always_inline)) {
    const char* p = t + ks * 32 * (2 * kWgT) + base + ((((cb >> 3) + ((i16 & 3) >> 1)) ^ sw) << 4);
    const bf16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_TR_PTR(p));
    const bf16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_TR_PTR(p + 4 * (2 * kWgT)));
    return bf16x8_t{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
  };
  for (int64_t r = row0; r < row_end; r += BK) {
    const int64_t rows = uni64(row_end - r < BK ? row_end - r : BK);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(P.a.p0 + uni64(r) * P.a.ld, (uint64_t)rows * P.a.ld * 2);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(P.b.p0 + uni64(r) * P.b.ld, (uint64_t)rows * P.b.ld * 2);
#pragma unroll
    for (int q = 0; q < QL; ++q) {
      dma16(ra, As + (q * 4 + wave) * 1024, oa[q], 0);
      dma16(rb, Bs + (q * 4 + wave) * 1024, ob[q], 0);
    }
    wait_loads<0>();
    block_barrier();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (ks * 32 >= rows) break;
      bf16x8_t a[4], b[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = frag(As, wm * 64 + m * 16, ks);
#pragma unroll
      for (int n = 0; n < 4; ++n) b[n] = frag(Bs, wn * 64 + n * 16, ks);
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = mfma16(b[n], a[m], acc[m][n]);
    }
    wait_lds();
    block_barrier();  // every wave has read the stage
  }

  // The wave's 64 x 64 tile through its own 8 KB: row r at 128 bytes, 16-byte
  // chunk c at c ^ ((r >> 1) & 7); then 8 rows x 128 bytes per store.
  char* st = lds + wave * 8192;
  const int h = lane >> 4;
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int r = m * 16 + (lane & 15), x = n * 32 + h * 8;
      *reinterpret_cast<uint2*>(st + r * 128 + (((x >> 4) ^ kc_swz(r)) << 4) + (x & 15)) = w4::bf16x4(acc[m][n]);
    }
  wait_lds();
  const int64_t col = n0 + wn * 64 + (lane & 7) * 8;
  const bool whole_lines = P.ldc % 64 == 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = q * 8 + (lane >> 3);
    const uint4 v = *reinterpret_cast<const uint4*>(st + r * 128 + (((lane & 7) ^ kc_swz(r)) << 4));
    const int64_t m = m0 + wm * 64 + r;
    if (m < P.M && col < P.N) {
      bf16_t* crow = m < P.csplit ? P.c0 + g * P.cgs + m * P.ldc : P.c1 + g * P.cgs + (m - P.csplit) * P.ldc;
      // Streaming stores of whole lines; rows off the 128-byte lines leave
      // partial ones, which the L2 must merge before they go to memory (fc2
      // wgrad of 40 copies of 2048 x 1416: 48 us with plain stores, 107 with
      // streaming ones; of 160 of 2048 x 768, whole lines: 115 and 86).
      if (whole_lines) st_stream(crow + col, v);
      else *reinterpret_cast<uint4*>(crow + col) = v;
    }
  }
}

}  // namespace fr
