// Final-norm output → LM head → shifted cross-entropy → dH, streaming the
// vocabulary in chunks: no [rows, vocab] logits or dlogits ever exist in
// memory, only a bf16 [rows, chunk] probability tile per chunk (over few rows
// several chunks, or all, are taken as one: head_group).
//
// Semantics: deltaserve-plugin/deltaserve/bwd_services/common/head.py:42-100
//   loss = sum_rows CE(logits, target) / n_valid, dlogits = (softmax - onehot)/n_valid,
//   grad_rows = dlogits · W. Rows that predict nothing (the last token of each
//   sequence) carry label -1 and contribute neither loss nor gradient.
//
// Two vocabulary-wide products, with the softmax taken against a per-row
// reference M that is known before the first product:
//   ce_init: M = the row's target logit (a dot of the row with W[target]);
//   per chunk c: logits = H·W_cᵀ (GEMM; its epilogue writes P = bf16(exp(logit
//     − M)) and, per wave-wide run of vocabulary columns, Σ exp(logit − M),
//     both over the columns other than the target's, whose logit x_t goes out
//     by itself, and the sum of the rounded P beside it. Any reference within
//     a few tens of the row maximum serves: bf16 and fp32 keep their relative
//     precision over that range. Only where
//     a sum passes 2^57 (a logit more than about 40 above M) does the run take
//     its own maximum m_t as its reference instead);
//   ce_rescale: per row L += Σ_t s_t·e^(m_t − M), the rounded sum R likewise,
//     and, on the rows where some m_t differs from M, M' = max_t m_t, α =
//     e^(M − M') and P scaled in place to M';
//   dH = dH·α + P·W_c (GEMM, fp32 accumulate with the per-row α);
//   after the last chunk, with e_t = exp(x_t − M): loss_row = ln(1 + L/e_t),
//   dH = (dH − R·W[target]) · L/R / (e_t + L) / n_valid, LSE = M + ln(e_t + L),
//   and a single-block deterministic sum gives the cycle loss.
// L/R takes the common part of P's rounding out of dH: one column that
// dominates the others' sum is rounded by up to 2^-9 (its exponential is 1 only
// against a reference that is its own), and L/R restores it to fp32. 300 rows
// with one column 17 above the sum of 2000 others: dH off by up to 2.5e-3 without
// it, 1e-7 with. R comes from the matrix cores (P times ones, a row's values
// being in the operand layout already): the logits products of 2048 × 2048 and
// 8192 × 4096 take 689 µs on average, 698 with dot products of two values, 684
// without R and the target's column kept apart.
// The target's term stays out of the sums because softmax − onehot cancels
// there: with p_t near 1 the row's loss and its coefficient of W[target],
// p_t − 1, are L/e_t and −L/(e_t + L), full precision in L, while e_t + L
// rounds L away and M, the dot, differs from x_t by the order of its sum. At
// 1 − p_t = 5e-5 on average (298 rows, target logits near 18, 4096 wide, 2000
// words) sums over all columns gave each row's dH an error of 29 % on average
// and the loss one of 1 %; now 6e-5 and 6e-7.
// With the tile maxima as references (every row of the first chunk rescaled,
// later ones where the row maximum lay in the chunk) the rescale took 48 µs
// per chunk at 8192 rows and 14 µs at 504, whose rows' serial passes over P
// set the time; reading the statistics alone takes 8.6 and 5.4 µs, and ce_init,
// once per cycle, 24 and 4 µs.
// Against the reference's 2 passes (logits for the LSE, then dlogits, both
// chunked, head.py:78-80, :92-94) this keeps its 2·M·D·V of logits and
// 2·M·D·V of dH and needs no third product. P passes through bf16 (the MFMA
// operand type) where the reference keeps probabilities in fp32; dH
// accumulates in fp32. The chunk is the reference's VOCAB_CHUNK unit; the
// caller can pause between a chunk's two products and between chunks.
#include "gemm_nt.h"
#include "kernels.h"

namespace dsb {

namespace {

// A run's sum of exp(logit − M) up to which M stays its reference: every term
// is then at most 2^57, far inside fp32 and bf16 range, and so are the sums
// and the dH accumulators (V and the weights add at most 2^30).
constexpr float kSumLimit = 0x1p57f;

// Per run of TN vocabulary columns (a wave tile's width) of chunk [c0, c0 + Vc)
// and row: (reference m_t, Σ exp(logit − m_t), Σ of those values as P holds
// them) into stats[m, (c0 + column) / TN] and P[m, j] = bf16(exp(logit[m, c0 +
// j] − m_t)) for the chunk's columns j < Vc; the row's target column counts as
// zero in all, its logit goes to tgt_logit[m]. Columns [Vc, Nc8) (Nc8 = round_up(Vc, 8)) are written as zero so
// the dH product runs its K loop over whole 16-byte chunks. m_t is run_m[m]
// unless the run's sum passes kSumLimit (or is NaN), then the run's maximum.
// Runs that hold a target (one in V / TN of a row's) or pass the limit take the
// exponentials a second time; the others test neither per element.
// A lane holds 4·FN values of a row, so the exponentials and the row sums are
// taken in the accumulator layout (two shuffles per row) and only bf16 values
// are staged for the row-contiguous stores; no barrier, each wave its own
// rows and columns. The epilogue it replaces (a maximum pass, an exchange
// between the waves of a row, fp32 staging and four shuffles per 8 values)
// made the product of a 16384-column chunk take 951 µs at 8192 rows × 4096
// against 791 now (the chunk's dH product, whose code did not change, 873 and
// 798 µs in the same two runs), 147 → 116 µs at 2048 × 2048 and 30.5 → 25.3 µs
// at 504 × 1024.
struct EpiCEProb {
  CEStat* stats;
  int ntn;
  bf16* P;
  long ldp;
  int c0, Vc, Nc8;
  const float* run_m;
  const int* labels;
  float* tgt_logit;
  template <int FM, int FN, int WM, int WN>
  DSB_DEV void run(const f32x4 (&acc)[FM][FN], int mw, int nw, int M, int lane, int wave,
                   void* smem) const {
    constexpr int TN = FN * 16, PITCH = TN + 8, CG = TN / 8;
    if (nw >= Vc || mw >= M) return;  // no live column or row in the wave tile
    const int l16 = lane & 15, lq = lane >> 4;
    const bool whole = nw + TN <= Vc;
    const int run = (c0 + nw) / TN;
    bf16* buf = reinterpret_cast<bf16*>(smem) + wave * 32 * PITCH;
    // the rows' references and target columns, all loaded before the first is
    // used (rows past M read row M − 1 and are not stored)
    float ref0[FM];
    int tcol[FM];  // within the run; outside [0, TN): not in it (label −1: negative)
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      const int m = min(mw + fm * 16 + l16, M - 1);
      ref0[fm] = run_m[m];
      tcol[fm] = labels[m] - (c0 + nw);
    }
#pragma unroll
    for (int b = 0; b < FM / 2; ++b) {
      if (mw + b * 32 >= M) break;  // uniform: the rest of the wave tile is past M
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int fm = 2 * b + h;
        bf16x4 pk[FN];
        // lane: row l16, columns 16·fn + 4·lq + i; with `skips` column 4·lq + tl
        // counts as zero (a factor min(|column − target|, 1): as per-element
        // tests the masks of 128 columns spill)
        const float tl = (float)(tcol[fm] - 4 * lq);
        auto take = [&](float ref, auto skips) {
          float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float e = __expf(acc[fm][fn][i] - ref);
              if (!whole) e = nw + fn * 16 + 4 * lq + i < Vc ? e : 0.f;
              if (decltype(skips)::value) e *= fminf(fabsf((float)(fn * 16 + i) - tl), 1.f);
              part[i] += e;
              pk[fn][i] = (bf16)e;
            }
          // the rounded values' row sums: products with ones, in which the order
          // of a row's values among its four lanes does not matter
          f32x4 r = {0.f, 0.f, 0.f, 0.f};
          const bf16 o = (bf16)1.f;
          const bf16x8 ones = {o, o, o, o, o, o, o, o};
#pragma unroll
          for (int fn = 0; fn < FN; fn += 2)
            r = mfma16(ones, __builtin_shufflevector(pk[fn], pk[fn + 1], 0, 1, 2, 3, 4, 5, 6, 7), r);
          float v = (part[0] + part[1]) + (part[2] + part[3]);
          v += __shfl_xor(v, 16, 64);
          return CEStat{ref, v + __shfl_xor(v, 32, 64), r[0]};
        };
        const int m = mw + fm * 16 + l16;
        CEStat st = take(ref0[fm], std::false_type{});
        if (__any(!(st.sum <= kSumLimit) || (unsigned)tcol[fm] < (unsigned)TN)) {
          // rare: rows with their target in this run, without it; rows past
          // the limit, against their run's own maximum
          float v = -INFINITY, xt = 0.f;
#pragma unroll
          for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
              const float x = acc[fm][fn][i];
              v = whole || nw + fn * 16 + 4 * lq + i < Vc ? fmaxf(v, x) : v;
              xt = (float)(fn * 16 + i) == tl ? x : xt;
            }
          const int tc = tcol[fm];
          if ((unsigned)tc < (unsigned)TN && ((tc >> 2) & 3) == lq && m < M) tgt_logit[m] = xt;
          v = fmaxf(v, __shfl_xor(v, 16, 64));
          v = fmaxf(v, __shfl_xor(v, 32, 64));
          st = take(st.sum <= kSumLimit ? st.ref : fmaxf(st.ref, v), std::true_type{});
        }
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
          *reinterpret_cast<bf16x4*>(buf + (16 * h + l16) * PITCH + fn * 16 + 4 * lq) = pk[fn];
        if (lq == 0 && m < M) stats[(long)m * ntn + run] = st;
      }
#pragma unroll
      for (int it = 0; it < 32 * CG / 64; ++it) {
        const int c = lane + 64 * it, row = c / CG, m = mw + b * 32 + row;
        const int n = nw + (c % CG) * 8;
        const u32x4 v = *reinterpret_cast<const u32x4*>(buf + row * PITCH + (c % CG) * 8);
        if (m < M && n < Nc8) stg128(P + (long)m * ldp + n, v);
      }
    }
  }
};

// Width of the runs the logits product's statistics cover: its wave tile's.
constexpr int ce_run(int cfg) {
  return cfg == GEMM_BIG ? 128 : cfg == GEMM_NARROW ? 32 : 64;
}

}  // namespace

// One wave per live row: the label (ids[t + 1] where row t predicts, −1
// elsewhere; an id outside [0, V) raises err bit 1), the row's first softmax
// reference, a dot of the row with W[target] (0 for rows without a target), and
// L = R = 0, α = 1.
__global__ __launch_bounds__(256) void ce_init_kernel(HeadArgs a) {
  int N = a.n;
  if (a.n_dev) N = min(N, *a.n_dev);
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (m >= N) return;
  int lab = -1;
  if (a.pred[m]) {
    const int64_t id = a.ids[m + 1];
    if (id >= 0 && id < a.V)
      lab = (int)id;
    else if (l == 0)
      atomicOr(a.err, 1);
  }
  float dot = 0.f;
  if (lab >= 0) {
    const bf16 *x = a.normed + (long)m * a.ldh, *w = a.W + (long)lab * a.D;
    for (int k = l; k < a.D / 8; k += 64) {
      float xf[8], wf[8];
      unpack8(ldg128(x + 8 * k), xf);
      unpack8(ldg128(w + 8 * k), wf);
#pragma unroll
      for (int e = 0; e < 8; ++e) dot += xf[e] * wf[e];
    }
    dot = wave_sum(dot);
  }
  if (l == 0) {
    a.labels[m] = lab;
    a.run_m[m] = dot;
    a.run_l[m] = a.run_r[m] = 0.f;
    a.alpha[m] = 1.f;
  }
}

// Chunk [c0, c0 + Vc) after its logits product, one wave per live row: the
// runs' largest reference M_c, the row's reference M and sums L and R moved to
// M' = max(M, M_c), α = e^(M − M') for the dH accumulator, and, on rows where
// some run's reference is not M', P scaled in place by e^(m_t − M') so that
// P = bf16(exp(logit − M')), R then taking the sum of the rounded products. Rows without a target keep their P: the finalize
// sets their dH to zero whatever the product accumulated.
__global__ __launch_bounds__(256) void ce_rescale_kernel(HeadArgs a, int c0) {
  int N = a.n;
  if (a.n_dev) N = min(N, *a.n_dev);
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (m >= N) return;
  const int bn = a.ce_bn, Vc = min(a.vchunk, a.V - c0), Nc8 = (Vc + 7) / 8 * 8;
  const int nt = (Vc + bn - 1) / bn;
  const CEStat* st = a.stats + (long)m * a.ntn + c0 / bn;
  const float mo = a.run_m[m];
  float mc = -INFINITY;
  for (int j = l; j < nt; j += 64) mc = fmaxf(mc, st[j].ref);
  mc = wave_max(mc);
  const float mn = fmaxf(mo, mc);
  float sc = 0.f, rs = 0.f;
  bool scaled = false;
  for (int j = l; j < nt; j += 64) {
    const CEStat s = st[j];
    sc += s.sum * __expf(s.ref - mn);
    rs += s.rsum;
    scaled |= s.ref != mn;
  }
  sc = wave_sum(sc);
  rs = wave_sum(rs);
  const float al = __expf(mo - mn);
  if (l == 0) {
    a.run_m[m] = mn;
    a.run_l[m] = a.run_l[m] * al + sc;
    a.alpha[m] = al;
  }
  if (a.labels[m] < 0) return;
  if (!__any(scaled)) {
    if (l == 0) a.run_r[m] = a.run_r[m] * al + rs;
    return;
  }
  rs = 0.f;
  bf16* pr = a.dlog + (long)m * a.vchunk;
#pragma unroll 4
  for (int k = l; k < Nc8 / 8; k += 64) {
    u32x4* q = reinterpret_cast<u32x4*>(pr + 8 * k);
    const float f = __expf(st[(8 * k) / bn].ref - mn);
    float v[8];
    unpack8(*q, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = (float)(bf16)(v[e] * f);
      rs += v[e];
    }
    *q = pack8(v);
  }
  rs = wave_sum(rs);
  if (l == 0) a.run_r[m] = a.run_r[m] * al + rs;
}

// After the last chunk, one wave per live row: with e_t = exp(x_t − M) and the
// other columns' sum L, loss_row = ln((e_t + L) / e_t), LSE = x_t + loss_row and
// dH = (dH − R·W[target]) · L/R / (e_t + L) / n_valid (R: the sum of P), with dH
// the sum in order of the `ks` accumulated K-slice partials when the product
// was split; rows without a target get dH = 0 and no loss.
__global__ __launch_bounds__(256) void ce_finalize_kernel(HeadArgs a, int ks) {
  int N = a.n;
  if (a.n_dev) N = min(N, *a.n_dev);
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (m >= N) return;
  const int t = a.labels[m];
  float* dr = a.dH + (long)m * a.D;
  if (t < 0) {
    for (int k = l; k < a.D / 4; k += 64)
      reinterpret_cast<f32x4*>(dr)[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (l == 0) a.loss_row[m] = 0.f;
    return;
  }
  const float L = a.run_l[m], xt = a.tgt_logit[m], d = xt - a.run_m[m], et = __expf(d);
  if (l == 0) {
    // ln(1 + L/e_t) where the sum would round L away; log1pf of a large ratio
    // is off by a bias of 1e-7 (the loss of 2048 rows at 128256 words: 1.2e-7
    // on average over six inputs, 4e-8 this way)
    const float loss = L < et ? log1pf(L / et) : logf(et + L) - d;
    a.lse[m] = xt + loss;
    a.loss_row[m] = loss;
  }
  // R = 0: P is all zeros
  const float R = a.run_r[m], f = R == 0.f ? 0.f : L / (et + L) / R * *a.inv_nvalid;
  const bf16* w = a.W + (long)t * a.D;
  const float* src = ks > 1 ? a.part + (long)m * a.D : dr;
  const long plane = (long)a.n * a.D;
  for (int k = l; k < a.D / 8; k += 64) {
    float wf[8];
    unpack8(ldg128(w + 8 * k), wf);
    f32x4 x0 = *reinterpret_cast<const f32x4*>(src + 8 * k);
    f32x4 x1 = *reinterpret_cast<const f32x4*>(src + 8 * k + 4);
#pragma unroll 4
    for (int z = 1; z < ks; ++z) {
      x0 += *reinterpret_cast<const f32x4*>(src + z * plane + 8 * k);
      x1 += *reinterpret_cast<const f32x4*>(src + z * plane + 8 * k + 4);
    }
    f32x4* d = reinterpret_cast<f32x4*>(dr + 8 * k);
    d[0] = f32x4{(x0[0] - wf[0] * R) * f, (x0[1] - wf[1] * R) * f,
                 (x0[2] - wf[2] * R) * f, (x0[3] - wf[3] * R) * f};
    d[1] = f32x4{(x1[0] - wf[4] * R) * f, (x1[1] - wf[5] * R) * f,
                 (x1[2] - wf[6] * R) * f, (x1[3] - wf[7] * R) * f};
  }
}

// Deterministic single-block sum of loss_row[0:n) times 1/n_valid.
__global__ __launch_bounds__(1024) void ce_loss_kernel(const float* __restrict__ loss_row,
                                                       int n, const int* n_dev,
                                                       const float* inv_nvalid,
                                                       float* __restrict__ out) {
  int N = n;
  if (n_dev) N = min(N, *n_dev);
  __shared__ float red[16];
  float s = 0.f;
  for (int i = threadIdx.x; i < N; i += 1024) s += loss_row[i];
  s = block_sum<1024>(s, red);
  if (threadIdx.x == 0) out[0] = s * (*inv_nvalid);
}

int head_num_chunks(const HeadArgs& a) { return (a.V + a.vchunk - 1) / a.vchunk; }

int head_group(int n, int V, int vchunk) {
  // A chunk's products over few rows are short: at 504 rows × 1024 the ten
  // pairs of a 151936-word head took 25 + 31 µs each, launch gaps, half-filled
  // last rounds and the accumulators' read and write included. Chunks are
  // taken together while the probability tile stays within the 2^27 elements
  // (268 MB) that 8192 rows have with one chunk, which also keeps the time
  // between two pause points with work at that of such a cycle's chunk; the
  // units are made equal. Cycles in µs by the bound 2^20 (one chunk each) /
  // 2^25 / 2^26 / 2^27 / 2^28: 504 rows × 1024 × 151936: 1600 / 1442 / 1433 /
  // 1399 / 1398; 256 × 5120 × 151936: 3540 / 3267 / 3104 / 3100 / 3109; 2048 ×
  // 2048 × 128256: 4470 / 4470 / 4311 / 4231 / 4150 (the head alone 1880 /
  // 1870 / 1814 / 1769 / 2021).
  if (n <= 0) return 1;
  const long kGroupElems = 1L << 27;
  const long nch = ((long)V + vchunk - 1) / vchunk;
  const long most = std::max(1L, kGroupElems / ((long)n * vchunk));
  const long units = (nch + most - 1) / most;
  return (int)((nch + units - 1) / units);
}

static GemmProblem chunk_logits_problem(const HeadArgs& a, int c0) {
  const int Vc = min(a.vchunk, a.V - c0);
  return GemmProblem{a.normed, a.ldh, a.W + (long)c0 * a.D, (long)a.D, nullptr, 0, nullptr, 0,
                     a.n, Vc, a.D, 0, a.n_dev};
}

void head_plan(HeadArgs& a, int gemm_cfg, bool can_split) {
  // The logits product's tile (the 64-wide one has no epilogue here): by cost,
  // over a full chunk, 2 bytes per element out.
  a.ce_cfg = GEMM_BIG;
  double bt = 0;
  for (int cfg : {GEMM_BIG, GEMM_WIDE, GEMM_MID, GEMM_NARROW}) {
    const double c = gemm_cost(a.n, a.vchunk, a.D, 2.0, cfg, 1);
    if (bt == 0 || c < bt) {
      bt = c;
      a.ce_cfg = cfg;
    }
  }
  a.ce_bn = ce_run(a.ce_cfg);
  a.ntn = (a.V + a.ce_bn - 1) / a.ce_bn;
  // The dH product's tile and K slices, the same for every chunk. A split
  // keeps one fp32 accumulator per slice across the chunks (read and written
  // by the product's epilogue) and the finalize adds the slices once, so a
  // chunk has no reduction launch: 8 bytes per slice's element and a share of
  // that one pass. 504 rows × 1024, K = 16384: 48 + 7.5 µs (256×256 tiles in 8
  // slices, 64 blocks, and a reduction per chunk) → 30 µs (128×128 in 8, 256
  // blocks); 256 rows × 5120: 55 + 13.7 → 48 µs.
  a.dh_cfg = gemm_cfg >= 0 ? gemm_cfg : GEMM_BIG;
  a.dh_ks = 1;
  if (gemm_cfg >= 0) return;
  bt = 0;
  const int nk = (a.vchunk + 63) / 64, nch = head_num_chunks(a);
  for (int cfg = 0; cfg < kGemmCfgs; ++cfg) {
    const GemmTile t = gemm_tile(cfg);
    const long tiles = (long)((a.n + t.bm - 1) / t.bm) * ((a.D + t.bn - 1) / t.bn);
    for (int ks = 1; ks <= (can_split && a.D % 8 == 0 ? std::min(16, nk / 3) : 1); ++ks) {
      if (ks > 1 && tiles * ks > kGemmCus * t.occ) break;
      // ks blocks per tile run as ks · tiles plain ones of a K / ks product
      // whose epilogue reads and writes the accumulator
      double c = gemm_cost(a.n, a.D, (nk + ks - 1) / ks * 64, 0.0, cfg, 1);
      const double blocks = (double)tiles * ks;
      if (ks > 1) {
        const double steps = (nk + ks - 1) / ks, operands = 2.0 * a.vchunk * ((double)a.n + a.D);
        c = 5.0 + std::max(std::ceil(blocks / kGemmCus) * steps * t.step + 0.5, operands / 6.8e6) +
            4.0 * ks * a.n * a.D / 3.9e6 / nch;
      }
      c += std::ceil(blocks / kGemmCus) * t.bm * t.bn * 8.0 *
           std::min(blocks, (double)kGemmCus) / 7.8e6;
      if (bt == 0 || c < bt) {
        bt = c;
        a.dh_cfg = cfg;
        a.dh_ks = ks;
      }
    }
  }
}

long head_part_elems(const HeadArgs& a) { return gemm_part_elems(a.n, a.D, a.dh_ks); }

hipError_t head_init(const HeadArgs& a, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(ce_init_kernel, dim3((a.n + 3) / 4), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t head_prob(const HeadArgs& a, int c0, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  const int Vc = min(a.vchunk, a.V - c0), Nc8 = (Vc + 7) / 8 * 8;
  EpiCEProb epi{a.stats, a.ntn,   a.dlog,  (long)a.vchunk, c0,
                Vc,      Nc8,     a.run_m, a.labels,       a.tgt_logit};
  const GemmProblem p = chunk_logits_problem(a, c0);
  switch (a.ce_cfg) {
    case GEMM_BIG: return launch_gemm_cfg<256, 256, 2, 2, 2, 3>(p, epi, s);
    case GEMM_WIDE: return launch_gemm_cfg<256, 128, 2, 2, 3, 3>(p, epi, s);
    case GEMM_MID: return launch_gemm_cfg<128, 128, 2, 2, 2, 3>(p, epi, s);
    case GEMM_NARROW: return launch_gemm_cfg<128, 64, 2, 2, 3, 3>(p, epi, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t head_rescale(const HeadArgs& a, int c0, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(ce_rescale_kernel, dim3((a.n + 3) / 4), dim3(256), 0, s, a, c0);
  return hipGetLastError();
}

hipError_t head_finalize(const HeadArgs& a, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(ce_finalize_kernel, dim3((a.n + 3) / 4), dim3(256), 0, s, a, a.dh_ks);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ce_loss_kernel, dim3(1), dim3(1024), 0, s, a.loss_row, a.n, a.n_dev,
                     a.inv_nvalid, a.loss_out);
  return hipGetLastError();
}

int head_dh_tail(const HeadArgs& a, int c0, int* tail) {
  *tail = 0;
  if (!a.tail_part || a.dh_ks > 1 || a.dh_cfg != GEMM_BIG) return 1;
  const int Nc8 = (min(a.vchunk, a.V - c0) + 7) / 8 * 8;
  const int kt = gemm_tail_split(a.n, a.D, Nc8, a.ncu, tail);
  return kt > 1 && (long)kt * *tail * 65536 <= a.tail_elems ? kt : 1;
}

hipError_t head_chunk_dh(const HeadArgs& a, int c0, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  const int Nc8 = (min(a.vchunk, a.V - c0) + 7) / 8 * 8;
  // dH = dH·α + P[:, chunk] · W[chunk, :]: the head read in place as the
  // [K, N] operand, rows past the vocabulary loading as zeros
  GemmProblem q{a.dlog, (long)a.vchunk, a.W + (long)c0 * a.D, (long)a.D, nullptr, 0, nullptr, 0,
                a.n, a.D, Nc8, 0, a.n_dev};
  q.b_kn = 1;
  q.kb_rows = min(a.vchunk, a.V - c0);
  EpiF32 ef{a.dH, (long)a.D, a.D, c0 > 0 ? 1 : 0, a.alpha};
  if (a.dh_ks > 1) {
    // each K slice accumulates its own partial; a slice past a short last
    // chunk's K only applies α
    if (!a.part || a.D % 8) return hipErrorInvalidValue;
    q.part = a.part;
    q.part_acc = c0 > 0 ? 1 : 0;
    q.part_scale = a.alpha;
    return launch_gemm(q, ef, s, a.dh_cfg, a.dh_ks);
  }
  int tail = 0;
  const int kt = head_dh_tail(a, c0, &tail);
  if (kt > 1) return launch_gemm_tail(q, ef, kt, tail, a.tail_part, s);
  return launch_gemm(q, ef, s, a.dh_cfg);
}

hipError_t head_fwd_bwd(const HeadArgs& a, hipStream_t s) {
  hipError_t e;
  if (a.n <= 0) return hipSuccess;
  if ((e = head_init(a, s)) != hipSuccess) return e;
  for (int c0 = 0; c0 < a.V; c0 += a.vchunk) {
    if ((e = head_prob(a, c0, s)) != hipSuccess) return e;
    if ((e = head_rescale(a, c0, s)) != hipSuccess) return e;
    if ((e = head_chunk_dh(a, c0, s)) != hipSuccess) return e;
  }
  return head_finalize(a, s);
}

}  // namespace dsb
