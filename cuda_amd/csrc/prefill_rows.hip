// Prefill for launches whose 256-row query tiles leave the chip idle (16-bit,
// head dim 64 and 128, softmax scale >= 0): waves of a workgroup share rows.
//
// Same contract and math as prefill.hip. One workgroup = 32 QG query rows of
// one (b, h) (or a causal pair of such tiles) = 8 waves: QG row groups of 32
// rows, KS = 8 / QG waves ("parts") per group, each walking every KS-th key
// tile with an online softmax of its own; the parts' (m, l, O) meet in LDS at
// the end, each part combining and storing its share of the head dims. The
// walks are KS times shorter and the workgroups 256 / (32 QG) times as many
// as in the 256-row kernels, whose rate per CU is the higher one: they stay
// wherever they fill the chip (launch_prefill).
//
// K and V tiles (kBN keys) travel HBM -> LDS by buffer loads into a ring of
// groups of KS tiles, one tile per part, shared by the row groups; one barrier
// per group. Tile layout, fragment reads and register layouts are those of
// prefill.hip: S^T = K Q^T with the rho row permutation, whose accumulators
// are the B operand of O^T += V^T P^T.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "launch.h"
#include "lds_dma.h"
#include "prefill_common.h"

namespace ca {
namespace {

constexpr int kRowsWaves = 8;

struct RowsArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;
  int S, Hq, Hkv;
  float scale_log2;
  int n_qt, n_bh, n_work, order;
};

template <typename Tr, int D, bool CAUSAL, int QG>
__device__ CA_INLINE void prefill_rows_tile(const RowsArgs& a, int bh, int qt) {
  using Gm = PfGeom<D>;
  using vec8 = typename Tr::vec8;
  using vec4 = typename Tr::vec4;
  using vec2 = typename Tr::vec2;
  constexpr int kNW = kRowsWaves, KS = kNW / QG;
  // 64 keys per tile; 32 where four 64-key tiles would fill the ring
  constexpr int kBN = D == 128 && KS == 4 ? 32 : 64;
  constexpr int kMB = kBN / 32;                  // 32-key blocks per tile
  constexpr int kKK = kBN / 16;                  // PV k-steps per tile
  constexpr int kRowB = Gm::kRowB, kNKS = Gm::kNKS, kNOB = Gm::kNOB;
  constexpr int kTileB = kBN * kRowB;            // K (or V) tile
  constexpr int kGroupB = KS * 2 * kTileB;       // one K and one V tile per part
  constexpr int kGroups = 128 * 1024 / kGroupB;  // ring, groups
  static_assert(kGroups >= 2, "a group loads while another is read");
  constexpr int kT = kTileB / 1024;              // 1-KB loads per tile
  constexpr int kLoads = KS * 2 * kT / kNW;  // loads per wave per group
  static_assert(kT % kNW == 0, "a tile's loads are dealt to all waves");
  constexpr int NR = 16 * kNOB / KS;             // O^T registers a part combines
  constexpr int kMeetB = QG * KS * (KS - 1) * NR * 256;  // the others' registers
  constexpr int kRowsB = QG * 32 * kRowB;        // output rows, packed
  static_assert(kMeetB + kRowsB <= kGroups * kGroupB, "the meeting fits the ring");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kGroups * kGroupB];
  __shared__ float red_m[QG][KS][32], red_l[QG][KS][32];

  const int S = a.S;
  const int lane = lane_here();  // (not hoisted out of the pair's loop: registers)
  const int wave = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_workitem_id_x() >> 6);
  const int qg = wave % QG, part = wave / QG;
  const int l32 = lane & 31, hl = lane >> 5;
  const int q0 = qt * 32 * QG, qw0 = q0 + 32 * qg, myq = qw0 + l32;
  const bool q_in = myq < S;
  const int h = bh % a.Hq;
  const size_t khead = (size_t)((bh / a.Hq) * a.Hkv + h / (a.Hq / a.Hkv)) * S;
  const uint16_t* Kp = a.k + khead * D;
  const uint16_t* Vp = a.v + khead * D;

  const int kv_end = CAUSAL ? min(S, q0 + 32 * QG) : S;
  const int n_tiles = (kv_end + kBN - 1) / kBN, n_groups = (n_tiles + KS - 1) / KS;
  // tiles this row group computes; the last holds the diagonal or the end
  const int w_end = CAUSAL ? min(kv_end, qw0 + 32) : kv_end;
  const int w_tiles = qw0 < S ? (w_end + kBN - 1) / kBN : 0;

  // load j of this wave: 1 KB of tile `sub` of the group, K or V, rows from
  // kRpk * piece (rows past kv_end read as zero)
  uint32_t off0;
  {
    const int row = Gm::kRpk * wave + lane / Gm::kLpr;
    off0 = row * kRowB + 16 * ((lane % Gm::kLpr) ^ Gm::swz(row));
  }
  auto issue = [&](int g) CA_INLINE {
    unsigned char* st = lds + (g % kGroups) * kGroupB;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      constexpr int kPer = kT / kNW;  // loads of a wave per tile
      const int sub = j / (2 * kPer), is_v = (j / kPer) % 2, p = j % kPer;
      const uint32_t t = (uint32_t)(g * KS + sub);
      dma16_buf(make_rsrc_at(is_v ? Vp : Kp, t * kTileB, (uint32_t)kv_end * kRowB),
                (CA_LDS void*)(st + (2 * sub + is_v) * kTileB + 1024 * (kNW * p + wave)),
                off0 + 1024u * kNW * p);  // swz repeats every 16 rows
    }
  };
#pragma unroll
  for (int g = 0; g < kGroups - 1; ++g) issue(g);

  // Q as the B operand of S^T = K Q^T: k-step ks holds d = 16 ks + 8 hl + [0, 8).
  // Lanes past S take row S - 1 of their own tile, whose vote in the tiles below
  // is that row's (q may be o itself: other tiles' rows may be written already).
  vec8 qv[kNKS];
  {
    const uint16_t* Qr = a.q + ((size_t)bh * S + min(myq, S - 1)) * D;
#pragma unroll
    for (int ks = 0; ks < kNKS; ++ks) qv[ks] = *(const vec8*)(Qr + 16 * ks + 8 * hl);
  }

  // LDS read offsets (prefill.hip): K row rho(l32), chunk hl (^ 32 ks bytes);
  // V^T source rows tr_row and tr_row + 4, chunks c0 (^ 64 ob bytes)
  const int krow = (l32 & 0x13) | ((l32 & 4) << 1) | ((l32 & 8) >> 1);
  const uint32_t kofs = krow * kRowB + 16 * (hl ^ Gm::swz(krow));
  const int g16 = lane >> 4, s16 = lane & 15;
  const int tr_row = 8 * (g16 >> 1) + (s16 >> 2), c0 = 2 * (g16 & 1) + ((s16 & 3) >> 1);
  const uint32_t vofs1 = kTileB + tr_row * kRowB + 16 * (c0 ^ Gm::swz(tr_row)) + 8 * (s16 & 1);
  const uint32_t vofs2 =
      kTileB + (tr_row + 4) * kRowB + 16 * (c0 ^ Gm::swz(tr_row + 4)) + 8 * (s16 & 1);
  const uint32_t lds0 = lds_off(lds);

  f32x16 o[kNOB];
#pragma unroll
  for (int i = 0; i < kNOB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m_run = kNegInf, l_run = 0.f;
  constexpr float kStaleMax = std::is_same<Tr, BF16>::value ? 0x1p48f : 0x1p15f;

  // One key tile at LDS byte `st`, keys from k0. FIRST: the part's first tile,
  // which takes the row max before its exponentials; later ones take theirs
  // against the running max as it stands, and again with their own only when a
  // lane's sum passes what P's type and O hold (stale_softmax in prefill.hip).
  // MASK: the row group's last tile (diagonal, end of the keys).
  auto tile = [&](uint32_t st, int k0, auto first_tag, auto mask_tag) CA_INLINE {
    constexpr bool FIRST = decltype(first_tag)::value, MASK = decltype(mask_tag)::value;
    f32x16 s[kMB];
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[mb][r] = 0.f;
    const uint32_t ka = st + kofs;
    u32x4 kr[kNKS][kMB];
    auto kread = [&](int ks) CA_INLINE {
      kr[ks][0] = lds_read_b128<0>(ka ^ (32 * ks));
      if constexpr (kMB == 2) kr[ks][kMB - 1] = lds_read_b128<32 * kRowB>(ka ^ (32 * ks));
    };
    constexpr int KD = 2;  // k-steps read ahead
#pragma unroll
    for (int ks = 0; ks < KD; ++ks) kread(ks);
#pragma unroll
    for (int ks = 0; ks < kNKS; ++ks) {
      if (ks + KD < kNKS) kread(ks + KD);
      wait_lgkm_n(kMB * (KD < kNKS - 1 - ks ? KD : kNKS - 1 - ks));
#pragma unroll
      for (int mb = 0; mb < kMB; ++mb) {
        after_wait(kr[ks][mb]);
        s[mb] = Tr::mfma32(__builtin_bit_cast(vec8, kr[ks][mb]), qv[ks], s[mb]);
      }
    }
    // the first V^T fragments land under the softmax
    constexpr int NST = kNOB * kKK, VD = 2;  // PV steps: O^T block st / kKK, k-step st % kKK
    u32x2 vr[NST][2];
    auto vread = [&](auto i) CA_INLINE {
      constexpr int st_ = decltype(i)::value, ob = st_ / kKK, kk = st_ % kKK;
      vr[st_][0] = lds_read_tr16<16 * kRowB * kk>((st + vofs1) ^ (64 * ob));
      vr[st_][1] = lds_read_tr16<16 * kRowB * kk>((st + vofs2) ^ (64 * ob));
    };
    for_const<VD>(vread);

    // a masked tile scales its logits before the mask, so that a masked one's
    // weight is 0 for scale 0 too
    vec8 pb[kKK];
    float sv[16 * kMB];
    // register i is key k0 + 8 hl + off
    const int last = (CAUSAL ? min(S - 1, myq) : S - 1) - k0 - 8 * hl;
#pragma unroll
    for (int i = 0; i < 16 * kMB; ++i) {
      sv[i] = s[i >> 4][i & 15];
      if (MASK) {
        const int off = 32 * (i >> 4) + 16 * ((i >> 3) & 1) + (i & 7);
        sv[i] = off > last ? kNegInf : sv[i] * a.scale_log2;
      }
    }
    auto settle_max = [&]() CA_INLINE {
      float t0 = kNegInf, t1 = kNegInf;
#pragma unroll
      for (int i = 0; i < 16 * kMB; i += 4) {
        t0 = max3(t0, sv[i], sv[i + 1]);
        t1 = max3(t1, sv[i + 2], sv[i + 3]);
      }
      const float t2 = __builtin_fmaxf(t0, t1);
      const float m_new = __builtin_fmaxf(m_run, pair32_max(MASK ? t2 : t2 * a.scale_log2));
      if (!FIRST) {
        const float alpha = m_new == kNegInf ? 1.f : fast_exp2(m_run - m_new);
#pragma unroll
        for (int i = 0; i < kNOB; ++i) o[i] *= alpha;
        l_run *= alpha;
      }
      m_run = m_new;
    };
    float sum[2];
    auto exp_all = [&]() CA_INLINE {
      const float msub = m_run == kNegInf ? 0.f : m_run;
#pragma unroll
      for (int i = 0; i < 16 * kMB; i += 2) {
        const float p0 = fast_exp2(MASK ? sv[i] - msub : __builtin_fmaf(sv[i], a.scale_log2, -msub));
        const float p1 = fast_exp2(MASK ? sv[i + 1] - msub : __builtin_fmaf(sv[i + 1], a.scale_log2, -msub));
        const vec2 pk = Tr::pack2(p0, p1);
        pb[i / 8][i % 8] = pk[0];
        pb[i / 8][i % 8 + 1] = pk[1];
        sum[(i / 2) & 1] = i < 4 ? p0 + p1 : sum[(i / 2) & 1] + (p0 + p1);
      }
    };
    if (FIRST) settle_max();
    exp_all();
    if (!FIRST && __builtin_expect(wave_any(!(sum[0] + sum[1] <= kStaleMax)), 0)) {
      settle_max();
      exp_all();
    }
    l_run += sum[0] + sum[1];

    // O^T += V^T P^T
    auto step = [&](auto i) CA_INLINE {
      constexpr int st_ = decltype(i)::value;
      if constexpr (st_ + VD < NST) vread(std::integral_constant<int, st_ + VD>{});
      wait_lgkm<2 * (VD < NST - 1 - st_ ? VD : NST - 1 - st_)>();
      after_wait(vr[st_][0]);
      after_wait(vr[st_][1]);
      const u32x4 w = {vr[st_][0][0], vr[st_][0][1], vr[st_][1][0], vr[st_][1][1]};
      o[st_ / kKK] = Tr::mfma32(__builtin_bit_cast(vec8, w), pb[st_ % kKK], o[st_ / kKK]);
    };
    for_const<NST>(step);
  };

  // one iteration per group: the part's tile of group g is g KS + part
  auto sync = [&](int g) CA_INLINE {
    wait_vmcnt<kLoads * (kGroups - 2)>();  // this wave's loads of group g landed
    __builtin_amdgcn_s_barrier();          // ... and every wave's; group g - 1 is read
    issue(g + kGroups - 1);
    return lds0 + (uint32_t)((g % kGroups) * kGroupB + part * 2 * kTileB);
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  int g = 0;
  if (part < w_tiles - 1) {
    tile(sync(0), part * kBN, T_{}, F_{});
#pragma clang loop unroll(disable)
    for (g = 1; g * KS + part < w_tiles - 1; ++g) tile(sync(g), (g * KS + part) * kBN, F_{}, F_{});
  }
  if (g * KS + part == w_tiles - 1) {
    const uint32_t st = sync(g);
    if (g == 0) tile(st, (g * KS + part) * kBN, T_{}, T_{});
    else tile(st, (g * KS + part) * kBN, F_{}, T_{});
    ++g;
  }
  for (; g < n_groups; ++g) sync(g);
  wait_vmcnt<0>();
  const float l_part = pair32_sum(l_run);
  if (hl == 0) {
    red_m[qg][part][l32] = m_run;
    red_l[qg][part][l32] = l_part;
  }
  __syncthreads();  // the ring is read: the parts' registers and the rows go there
  // Register r of 16 kNOB goes to part r / NR. Block (qg, dst, j), j counting
  // the other parts: [NR / 4][64 lanes] x 4 floats.
  auto block = [&](int dst, int j) CA_INLINE {
    return (f32x4*)lds + ((qg * KS + dst) * (KS - 1) + j) * (NR * 16) + lane;
  };
  f32x4 own[NR / 4];
#pragma unroll
  for (int dst = 0; dst < KS; ++dst) {
    f32x4 x[NR / 4];
#pragma unroll
    for (int j = 0; j < NR / 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = dst * NR + 4 * j + e;
        x[j][e] = o[i / 16][i % 16];
      }
    if (dst == part) {
#pragma unroll
      for (int j = 0; j < NR / 4; ++j) own[j] = x[j];
    } else {
      f32x4* blk = block(dst, part < dst ? part : part - 1);
#pragma unroll
      for (int j = 0; j < NR / 4; ++j) blk[64 * j] = x[j];
    }
  }
  __syncthreads();
  float M = kNegInf, L = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) M = __builtin_fmaxf(M, red_m[qg][s][l32]);
  auto weight = [&](int s) CA_INLINE { return M == kNegInf ? 0.f : fast_exp2(red_m[qg][s][l32] - M); };
#pragma unroll
  for (int s = 0; s < KS; ++s) L += weight(s) * red_l[qg][s][l32];
  const float inv = L > 0.f ? 1.f / L : 0.f;
  if (a.lse && part == 0 && hl == 0 && q_in) a.lse[(size_t)bh * S + myq] = row_lse(M, L);
  const float w_own = weight(part);
#pragma unroll
  for (int j = 0; j < NR / 4; ++j) own[j] *= w_own;
#pragma unroll
  for (int p = 0; p < KS - 1; ++p) {
    const float w = weight(p < part ? p : p + 1);
    const f32x4* blk = block(part, p);
#pragma unroll
    for (int j = 0; j < NR / 4; ++j) own[j] += blk[64 * j] * w;
  }
  // packed into the group's rows: register r of a 32-d block is d = 8 (r / 4) +
  // 4 hl + r % 4
  unsigned char* rows = lds + kMeetB + qg * 32 * kRowB;
#pragma unroll
  for (int j = 0; j < NR / 4; ++j) {
    const vec2 lo = Tr::pack2(own[j][0] * inv, own[j][1] * inv), hi = Tr::pack2(own[j][2] * inv, own[j][3] * inv);
    vec4 y;
    y[0] = lo[0]; y[1] = lo[1]; y[2] = hi[0]; y[3] = hi[1];
    const int c = part * (NR / 4) + j;  // 16-byte chunk: d = 8 c + 4 hl
    *(u32x2*)(rows + l32 * kRowB + 16 * (c ^ (l32 % Gm::kLpr)) + 8 * hl) = __builtin_bit_cast(u32x2, y);
  }
  __syncthreads();
  // the group's KS waves store its 32 rows, 16 bytes a lane
#pragma unroll
  for (int j = 0; j < 32 * kRowB / 1024 / KS; ++j) {
    const int p = 64 * (j * KS + part) + lane, r = p / Gm::kLpr, c = p % Gm::kLpr;
    const int row = qw0 + r;
    if (row < S)
      *(u32x4*)(a.o + ((size_t)bh * S + row) * D + 8 * c) =
          *(const u32x4*)(rows + r * kRowB + 16 * (c ^ (r % Gm::kLpr)));
  }
}

template <typename Tr, int D, bool CAUSAL, int QG>
__global__ __launch_bounds__(64 * kRowsWaves) void prefill_rows_kernel(RowsArgs a) {
  const int wg = __builtin_amdgcn_workgroup_id_x();
  const QTileWork wk = prefill_item(wg, a.n_work, a.n_qt, a.n_bh, a.order);
  const int n_pass = wk.qt1 < 0 ? 1 : 2;
#pragma clang loop unroll(disable)
  for (int pass = 0; pass < n_pass; ++pass) {
    if (pass) __syncthreads();  // every wave has stored its rows from LDS
    prefill_rows_tile<Tr, D, CAUSAL, QG>(a, pass ? wk.bh1 : wk.bh0, pass ? wk.qt1 : wk.qt0);
  }
}

template <typename Tr, int D, bool CAUSAL>
hipError_t launch_t(RowsArgs a, int groups, long long grid, hipStream_t stream) {
  const auto kernel = groups == 4 ? &prefill_rows_kernel<Tr, D, CAUSAL, 4>
                                  : &prefill_rows_kernel<Tr, D, CAUSAL, 2>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * kRowsWaves), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

// The times behind the rule, in 0.1 us (fitted to 31 shapes on one MI355X): a
// key step of a workgroup, and what a query tile costs beside its steps (first
// loads, meeting, store; the 256-row kernels overlap part of it with the tile
// before).
//   groups  keys per step   step (D = 128, 64)   tile
//   8       64              11, 9                30     (256-row kernels)
//   4       128             17, 12               28
//   2       128, 256        13, 10.5             39
// A launch takes its busiest CU's time: tiles in rounds (equal tiles, pairs), or
// the longest walk or the mean load, with a tenth for its end (2 groups: 45 %,
// they fetch K and V most often: 12 heads x 3500 x 64, 660 tiles, 38 us against
// 34 with 4). Waves share rows where that is estimated a
// tenth or more shorter, as measured for 32/8 heads, one sequence, causal: 333
// keys 12.3 -> 9.4 us at D = 128, 10.0 -> 7.1 at 64; 1000 keys 23.6 -> 20.5, 18.9
// -> 13.6; 8 heads of 2500 keys 44.5 -> 28.5, 35.6 -> 17.4; for 2048 keys of 32
// heads (D = 128) the 256-row kernel is the faster one (43.8 us against 46.5).
int prefill_rows_groups(int B, int Hq, int S, int D, float scale, bool causal) {
  const float sl2 = scale * kLog2e;
  if (!(sl2 >= 0.f && sl2 <= 3.0e38f)) return 0;
  const double cus = std::max(device_cus(), 1);
  const double bh = (double)B * Hq;
  auto estimate = [&](int groups, int keys, double step, double tile, double slack = 1.1) {
    const int rows = 32 * groups, n_qt = (S + rows - 1) / rows;
    int order = 0;
    const double grid = (double)prefill_grid(B, Hq, n_qt, causal, 1, &order);
    auto walk = [&](int n) { return tile + step * ((n + keys - 1) / keys); };
    const double longest = walk(S);
    if (!causal) return std::ceil(grid / cus) * longest;
    // the mean of a causal tile's steps: half the longest's and a half step
    const double mean = tile + step * (0.5 * S / keys + 0.5);
    if (order == kOrderPairs) return std::ceil(grid / cus) * 2 * mean;
    return std::max(longest, slack * bh * n_qt * mean / cus);
  };
  const bool d64 = D == 64;
  const double base = estimate(8, 64, d64 ? 9 : 11, 30);
  const double four = estimate(4, 128, d64 ? 12 : 17, 28);
  const double two = estimate(2, d64 ? 256 : 128, d64 ? 10.5 : 13, 39, 1.45);
  if (std::min(four, two) > 0.9 * base) return 0;
  const int groups = two < four ? 2 : 4;
  // a workgroup per tile here, and a launch's threads are 32-bit (the 256-row
  // kernels' launches of equal tiles are persistent)
  const int rows = 32 * groups;
  return bh * ((S + rows - 1) / rows) * (64 * kRowsWaves) > 4294967295.0 ? 0 : groups;
}

hipError_t launch_prefill_rows(int groups, bool f16, const void* q, const void* k, const void* v,
                               void* o, float* lse, int B, int Hq, int Hkv, int S, int D,
                               float scale, bool causal, hipStream_t stream) {
  RowsArgs a{(const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)o, lse, S, Hq,
             Hkv, scale * kLog2e, 0, B * Hq, 0, 0};
  a.n_qt = (S + 32 * groups - 1) / (32 * groups);
  const long long grid = prefill_grid(B, Hq, a.n_qt, causal, 1, &a.order);
  if (grid == 0) return hipSuccess;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  a.n_work = (int)grid;
#define CA_ROWS_CASE(TR, DD)                                              \
  if (D == DD)                                                            \
    return causal ? launch_t<TR, DD, true>(a, groups, grid, stream)       \
                  : launch_t<TR, DD, false>(a, groups, grid, stream);
  if (f16) {
    CA_ROWS_CASE(F16, 64)
    CA_ROWS_CASE(F16, 128)
  } else {
    CA_ROWS_CASE(BF16, 64)
    CA_ROWS_CASE(BF16, 128)
  }
#undef CA_ROWS_CASE
  return hipErrorInvalidValue;
}

}  // namespace ca
