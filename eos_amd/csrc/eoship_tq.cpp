// TurboQuant half of the eoship C ABI: corpus binding and top-k scoring.
//
// Replaces the host loop topTurboQuantRetrievalScoresWithStats
// (runtime/retrieval_turboquant.go:1853-1887) and its per-document
// q.InnerProductPrepared calls with a device pipeline per batch of <= 64
// queries, enqueued on the runtime stream without host synchronisation:
//   1. eos_tq_rotate /  rotate (f64), round to int16, split into int8 hi/lo
//      eos_tq_quantize  MFMA fragments (PrepareQuery)
//   2. sample scan      exact scores of every s-th tile of 32 vectors
//   3. eos_tq_threshold per query, a score below the r-th best sample
//   4. filter scan      one pass over the corpus, keep score >= threshold
//   5. eos_tq_finalize  select + order the kept candidates (score desc,
//                       id asc), emit top-k, or flag the query
//   6. exact fallback   gated on the flags: exhaustive scores + exact radix
//                       selection for any query whose kept set is too small
//                       or overflowed.
// Step 6 makes the result exact whatever the data; steps 2-3 only decide how
// much work step 4 saves.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "eoship_internal.h"
#include "kernels/tq_args.h"

namespace {
// The finalize variant for k: up to 1024 the one with the small selection
// buffer (it fits beside a running filter scan on a CU), else the full one.
const char* finalize_kernel(int k) {
  return k <= 1024 ? "eos_tq_finalize_k1024" : "eos_tq_finalize";
}
}  // namespace

using eoship::hip_err;
using eoship::set_err;

namespace {

constexpr int kBatch = 64;          // queries per scan (two 32-column groups)
constexpr int kMaxCols = 128;       // MFMA query columns per pass (MaxSim: four 32-token groups)
constexpr int kCap = 8192;          // kept candidates per query
constexpr int kRescoreBlocks = 16;  // workgroups per query rescoring kept ids (64 ids each)
constexpr int kSortCap = 8192;      // largest k the device sort handles
constexpr int kSampleStride = 16;     // sample every 16th tile (at least)
constexpr int kMaxSampleTiles = 2048;  // tile maxima per query (the threshold kernel holds 4096)
// Candidates the sample threshold aims to keep per query, as a multiple of k:
// on the benchmark's c2 corpus a 1/16 sample at 3 k keeps ~320 for k = 100, with the
// fewest kept over 256 queries still ~1.8 k (fewer than k triggers the exact
// fallback, which stays correct but costs a dense pass).
constexpr double kKeepFactor = 3.0;
constexpr int kTile = 32;
constexpr int kQmaxLimit = 127 * 256 + 127;  // largest int16 with int8 hi/lo halves
const int kSupportedKs[] = {1, 2, 4, 8, 12, 16, 24, 32};

int ks_for_dim(int d) {
  for (int ks : kSupportedKs)
    if (ks * 32 >= d) return ks;
  return 0;
}

inline uint8_t sext(uint8_t b) { return (b & 0x80) ? 0xff : 0x00; }

// Emulates v_perm_b32 (byte select with sign-replicate/zero/0xFF selectors).
uint32_t perm_emul(uint32_t s0, uint32_t s1, uint32_t sel) {
  const uint64_t in = ((uint64_t)s0 << 32) | s1;
  uint32_t out = 0;
  for (int b = 0; b < 4; ++b) {
    const uint32_t s = (sel >> (8 * b)) & 0xff;
    uint32_t v;
    if (s >= 13) v = 0xff;
    else if (s == 12) v = 0x00;
    else if (s == 11) v = ((in >> 63) & 1) ? 0xff : 0;
    else if (s == 10) v = ((in >> 47) & 1) ? 0xff : 0;
    else if (s == 9) v = ((in >> 31) & 1) ? 0xff : 0;
    else if (s == 8) v = ((in >> 15) & 1) ? 0xff : 0;
    else v = (uint32_t)((in >> (8 * s)) & 0xff);
    out |= v << (8 * b);
  }
  return out;
}

// Solves the two XOR-combined 8-byte tables of the 4-bit decode so that
// perm(A, x) ^ perm(B, x ^ 8) == C[x] for every 4-bit x.
int solve_lut4(const int8_t* cb, uint32_t lut[4], char** err) {
  uint8_t c[16];
  for (int i = 0; i < 16; ++i) c[i] = (uint8_t)cb[i];
  uint8_t kb[8] = {0}, ka[16] = {0};
  kb[4] = 0x00;
  kb[5] = kb[6] = kb[7] = 0xff;
  ka[12] = 0x00;
  ka[13] = ka[14] = ka[15] = 0xff;
  kb[2] = sext((uint8_t)~c[13]);
  kb[3] = sext((uint8_t)~c[15]);
  ka[10] = sext((uint8_t)~c[5]);
  ka[11] = sext((uint8_t)~c[7]);
  ka[9] = sext(c[3] ^ kb[3]);
  kb[1] = sext(c[11] ^ ka[11]);
  kb[0] = sext(c[9] ^ ka[9]);
  ka[8] = sext(c[1] ^ kb[1]);
  uint8_t ta[8], tb[8];
  for (int u = 0; u < 8; ++u) {
    ta[u] = c[u] ^ kb[u];
    tb[u] = c[u + 8] ^ ka[u + 8];
  }
  lut[0] = ta[0] | (ta[1] << 8) | (ta[2] << 16) | ((uint32_t)ta[3] << 24);
  lut[1] = ta[4] | (ta[5] << 8) | (ta[6] << 16) | ((uint32_t)ta[7] << 24);
  lut[2] = tb[0] | (tb[1] << 8) | (tb[2] << 16) | ((uint32_t)tb[3] << 24);
  lut[3] = tb[4] | (tb[5] << 8) | (tb[6] << 16) | ((uint32_t)tb[7] << 24);
  for (uint32_t x = 0; x < 16; ++x) {
    const uint32_t sel = x * 0x01010101u;
    const uint32_t r = perm_emul(lut[1], lut[0], sel) ^ perm_emul(lut[3], lut[2], sel ^ 0x08080808u);
    if (r != (uint32_t)c[x] * 0x01010101u)
      return set_err(err, "eoship: 4-bit codebook lookup table self-check failed at code %u", x);
  }
  return 0;
}

}  // namespace

struct EosHipTQ {
  EosHipRuntime* rt = nullptr;
  int d = 0, bits = 0, ks = 0, nload = 0, row_bytes = 0, qmax = 0;
  int64_t n = 0, ntiles = 0;
  float cb_scale = 0.f;
  int8_t codebook[16] = {0};
  uint32_t lut[4] = {0, 0, 0, 0};
  void* packed = nullptr;
  float* norms = nullptr;
  float* rot_t = nullptr;
  // Encoding: the split operand fragments of R and, in the same allocation, R
  // row-major (rot_frag NULL: no rotation, or scales outside the split
  // product's bound), the largest row norm of R and the decision distance in
  // half level steps.
  float* rot_r = nullptr;
  void* rot_frag = nullptr;
  float rot_rmax = 0.f, enc_delta2 = 0.f;
  double* qrot = nullptr;  // [kMaxCols][d] rotated query columns
  // per-batch device scratch
  int8_t* bfrag = nullptr;
  float* alpha = nullptr;
  float* tau = nullptr;
  unsigned long long* cand = nullptr;
  uint32_t* cand_count = nullptr;
  int* status = nullptr;
  float* samp = nullptr;
  int64_t samp_tiles = 0;
  float* dense = nullptr;
  size_t dense_bytes = 0;
  // MaxSim query preparation for a whole chunk of queries (every pass reads
  // its column blocks from it): fragments [ks][ms_ncb][64][16], alpha and the
  // f64 rotated columns of 32 * ms_ncb / 2 token columns
  int8_t* ms_bfrag = nullptr;
  size_t ms_bfrag_bytes = 0;
  float* ms_alpha = nullptr;
  size_t ms_alpha_bytes = 0;
  double* ms_qrot = nullptr;
  size_t ms_qrot_bytes = 0;
  int ms_ncb = 0;
  float* ms_lonorm = nullptr;  // [token columns] ||lo||_2 (bound filter)
  size_t ms_lonorm_bytes = 0;
  // bound-filtered MaxSim top-k of a chunk (carved by maxsim_filtered)
  void* ms_ws = nullptr;
  size_t ms_ws_bytes = 0;
  // chunked row selection: per-chunk top-k keys, then per row the list
  // length and finalize status
  unsigned long long* sel_keys = nullptr;
  size_t sel_keys_bytes = 0;
  uint32_t* sel_aux = nullptr;
  size_t sel_aux_bytes = 0;
  int32_t* dense_dots = nullptr;
  size_t dense_dots_bytes = 0;
  int16_t* qs_buf = nullptr;
  // high-half filter bounds: per query column ||lo||_2, per tile max ||C||_2
  float* lonorm = nullptr;
  float* tile_cn = nullptr;
  // reference-layout code rows padded to rs16 16-byte chunks (rescoring)
  uint8_t* codes_rm = nullptr;
  int rs16 = 0;
  // host-API staging
  void* io = nullptr;
  size_t io_bytes = 0;
  // Corpus bound with an ID order (EosHipTQBindOptions::id_rank): vector i
  // sits at position rank[i], so position order is the string-ID order the
  // ties follow; id_map[p] (device) is the vector index at position p,
  // reported in its place. Empty / nullptr for index order.
  long long* id_map = nullptr;
  std::vector<int64_t> rank_host;
  // Handles sharing the corpus arrays (packed, norms, rot_t, rot_frag,
  // tile_cn, codes_rm, id_map) through eoship_tq_share; nullptr while this is the only one.
  int* corpus_refs = nullptr;

  void free_all() {
    void* scratch[] = {qrot, bfrag, alpha, tau, cand, cand_count, status, samp, dense, dense_dots,
                       qs_buf, lonorm, io, sel_keys, sel_aux, ms_bfrag, ms_alpha, ms_qrot,
                       ms_lonorm, ms_ws};
    for (void* p : scratch)
      if (p) hipFree(p);
    if (corpus_refs != nullptr && --*corpus_refs > 0) return;
    delete corpus_refs;
    corpus_refs = nullptr;
    void* corpus[] = {packed, norms, rot_t, rot_frag, tile_cn, codes_rm, id_map};
    for (void* p : corpus)
      if (p) hipFree(p);
  }

  // Per-call device scratch (the corpus arrays are allocated by the bind).
  int alloc_scratch(char** err) {
    const size_t bfrag_bytes = (size_t)ks * 8 * 64 * 16;
    samp_tiles = std::min<int64_t>((ntiles + kSampleStride - 1) / kSampleStride, kMaxSampleTiles);
    if (rt->alloc(bfrag_bytes, reinterpret_cast<void**>(&bfrag), err) != 0 ||
        rt->alloc((size_t)kMaxCols * d * sizeof(double), reinterpret_cast<void**>(&qrot), err) != 0 ||
        rt->alloc(kMaxCols * sizeof(float), reinterpret_cast<void**>(&alpha), err) != 0 ||
        rt->alloc(kMaxCols * sizeof(float), reinterpret_cast<void**>(&lonorm), err) != 0 ||
        rt->alloc((size_t)kBatch * d * sizeof(int16_t), reinterpret_cast<void**>(&qs_buf), err) != 0 ||
        rt->alloc(kMaxCols * sizeof(float), reinterpret_cast<void**>(&tau), err) != 0 ||
        rt->alloc(kMaxCols * sizeof(uint32_t), reinterpret_cast<void**>(&cand_count), err) != 0 ||
        rt->alloc(kMaxCols * sizeof(int), reinterpret_cast<void**>(&status), err) != 0 ||
        rt->alloc((size_t)kBatch * kCap * sizeof(unsigned long long), reinterpret_cast<void**>(&cand),
                  err) != 0 ||
        rt->alloc((size_t)kBatch * std::max<int64_t>(samp_tiles, 1) * sizeof(float),
                  reinterpret_cast<void**>(&samp), err) != 0)
      return 1;
    return 0;
  }

  // 32-coordinate tiles and 32-wide K chunks (an even number) of the encode's
  // split product.
  int enc_tiles() const { return (d + 31) / 32; }
  int enc_chunks() const { return (d + 63) / 64 * 2; }

  // The rotation's operands of eos_tq_encode_split_* and the bound that
  // gives its decision distance: with R = Rh + Rl + Re and x = xh + xl + xe in
  // bf16 pairs, |u~ - u| / |x| <=
  //   |R_j| 2^-18 + max|Re_j| + max|Rl_j| 2^-9     (R xe, Re x, Rl xl dropped)
  // + |R_j| 33 * 2^-23     (32 products of a chunk summed in f32, an ulp lost
  //                         at each addition whatever the order)
  // + |R_j| chunks * 2^-24 (the sum over the chunks)
  // with 5 % on top for the second-order terms (d = 384: 1.1e-5). How the MFMA
  // adds inside a chunk is not documented; an ulp of the running sum per
  // addition is assumed. Measured with rows and vectors whose every dropped
  // part and rounding has one sign, next to decision points, d 32 to 768: at most
  // 3.3e-6, a quarter of the bound.
  // Scales that would put the distance over a quarter of a half step, or leave
  // f32 and bf16 no room, keep the f64 kernels (rot_frag stays NULL).
  // R is uploaded once; its transpose and the sums come from the device. Two
  // uploads and passes over d^2 values on the host were most of binding a small
  // corpus (no vectors: d = 384 1.06 ms, d = 1024 7.1, now 0.12 and 0.24).
  int prepare_rotation(const float* rot, char** err) {
    const size_t bytes = (size_t)d * d * sizeof(float);
    const size_t frag_bytes = (size_t)enc_tiles() * enc_chunks() * 4096;
    if (rt->alloc(bytes, reinterpret_cast<void**>(&rot_t), err) != 0 ||
        rt->alloc(frag_bytes + bytes, &rot_frag, err) != 0)
      return 1;
    rot_r = reinterpret_cast<float*>(static_cast<char*>(rot_frag) + frag_bytes);
    hipError_t e = rt->copy_async(rot_r, rot, bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(rotation)", e);
    static_assert(kMaxCols >= 3, "qrot holds the sums");
    TqRotFragArgs f{rot_r, rot_frag, rot_t, qrot, d, enc_tiles(), enc_chunks()};
    const unsigned threads = (unsigned)(f.jtiles * f.nchunk) * 128u;
    std::vector<double> sums(3 * (size_t)d);
    if (rt->launch("eos_tq_rot_transpose", dim3((unsigned)(d * d + 255) / 256), dim3(256), 0, &f,
                   err) != 0 ||
        rt->launch("eos_tq_rot_frag", dim3((threads + 255) / 256), dim3(256), 0, &f, err) != 0 ||
        rt->launch("eos_tq_rot_rows", dim3((unsigned)(d + 3) / 4), dim3(256), 0, &f, err) != 0)
      return 1;
    e = rt->copy_async(sums.data(), qrot, sums.size() * sizeof(double), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(rotation sums)", e);
    if (rt->sync(err) != 0) return 1;
    double rmax = 0.0, lmax = 0.0, emax = 0.0;
    bool finite = true;
    for (int j = 0; j < d; ++j) {
      finite = finite && std::isfinite(sums[j]);
      rmax = std::max(rmax, sums[j]);
      lmax = std::max(lmax, sums[d + j]);
      emax = std::max(emax, sums[2 * d + j]);
    }
    rmax = std::sqrt(rmax) * (1.0 + 1e-6);
    const double bound = 1.05 * (rmax * (0x1p-18 + 33 * 0x1p-23 + enc_chunks() * 0x1p-24) +
                                 std::sqrt(emax) + std::sqrt(lmax) * 0x1p-9);
    const double delta2 = 2.0 * bound / (double)cb_scale + 1e-4;
    if (finite && rmax >= 0x1p-20 && rmax <= 0x1p20 && cb_scale <= 0x1p20f && delta2 < 0.25) {
      rot_rmax = (float)(rmax * (1.0 + 1e-6));
      enc_delta2 = (float)(delta2 * (1.0 + 1e-6));
      return 0;
    }
    hipFree(rot_frag);
    rot_r = nullptr;
    rot_frag = nullptr;
    return 0;
  }

  int ensure(void** p, size_t* have, size_t need, char** err) {
    if (*have >= need && *p != nullptr) return 0;
    if (*p) hipFree(*p);
    *p = nullptr;
    *have = 0;
    if (rt->alloc(need, p, err) != 0) return 1;
    *have = need;
    return 0;
  }

  int nqg_for(int qb) const { return (qb <= 32 || ks > 24) ? 1 : 2; }
  int batch_cap() const { return ks > 24 ? 32 : kBatch; }

  void scan_base(TqScanArgs* s, int qb) const {
    memset(s, 0, sizeof(*s));
    s->packed = static_cast<const int32_t*>(packed);
    s->norms = norms;
    s->bfrag = bfrag;
    s->alpha = alpha;
    s->tau = tau;
    s->cand = cand;
    s->cand_count = cand_count;
    s->n = n;
    s->tile_step = 1;
    s->q = qb;
    s->cap = kCap;
    s->lut0 = lut[0];
    s->lut1 = lut[1];
    s->lut2 = lut[2];
    s->lut3 = lut[3];
    s->lonorm = lonorm;
    s->tile_cn = tile_cn;
  }

  int launch_scan(TqScanArgs* s, int qb, char** err) {
    // The scan kernels assume at least one tile (their first loads are clamped
    // to the last tile); with none there is nothing to scan or keep.
    if (s->ntiles <= 0) return 0;
    static const char* const labels[4] = {"tq_scan_dense", "tq_scan_filter", "tq_scan_sample",
                                          "tq_scan_filter"};
    const int nqg = nqg_for(qb);
    char name[64];
    const char kind = s->mode == 1 ? 'f' : s->mode == 3 ? 'h' : 'w';
    snprintf(name, sizeof(name), "eos_tq_scan_b%d_k%d_g%d_%c", bits, ks, nqg, kind);
    // One workgroup per CU (eight waves; twelve for the high-half filter up to
    // 16 K-steps, matching the kernels' launch bounds),
    // each owning a contiguous tile range of at least one tile (the kernel
    // clamps its loads to the range).
    const int threads = s->mode == 3 && ks <= 16 ? 768 : 512;
    int64_t blocks = (s->ntiles + threads / 64 - 1) / (threads / 64);
    if (blocks > rt->compute_units) blocks = rt->compute_units;
    if (blocks < 1) blocks = 1;
    return rt->launch(name, dim3((unsigned)blocks), dim3(threads), 0, s, err, labels[s->mode]);
  }

  // Rotates and quantizes nsrc source rows into ncols = 32 * nqg MFMA columns:
  // column c reads source row (c / group) * group_live + c % group when
  // c % group < group_live, else it is a zero column.
  int prepare_cols(const float* d_src, int nsrc, int nqg, int group, int group_live,
                   int16_t* qs_out, char** err) {
    TqPrepArgs p;
    memset(&p, 0, sizeof(p));
    p.bfrag = bfrag;
    p.alpha = alpha;
    p.tau = tau;
    p.cand_count = cand_count;
    p.qrot = qrot;
    p.lonorm = lonorm;
    return prepare_into(&p, d_src, nsrc, nqg, group, group_live, qs_out, err);
  }

  // prepare_cols into the output buffers p already names (tau, cand_count
  // and lonorm may be NULL).
  int prepare_into(TqPrepArgs* pp, const float* d_src, int nsrc, int nqg, int group,
                   int group_live, int16_t* qs_out, char** err) {
    TqPrepArgs& p = *pp;
    p.queries = d_src;
    p.rot_t = rot_t;
    p.qs_out = qs_out;
    p.q = nsrc;
    p.d = d;
    p.ks = ks;
    p.ncb = 2 * nqg;
    p.qmax = qmax;
    p.cb_scale = cb_scale;
    p.group = group;
    p.group_live = group_live;
    const unsigned cblocks = (unsigned)(32 * nqg / 8);  // 8 columns per workgroup
    if (rot_t != nullptr) {
      const unsigned jblocks = (unsigned)((d + 31) / 32);
      if (rt->launch("eos_tq_rotate", dim3(jblocks, cblocks), dim3(256), 0, &p, err) != 0) return 1;
    }
    return rt->launch(d <= 384 ? "eos_tq_quantize_m12" : "eos_tq_quantize", dim3(cblocks), dim3(256),
                      0, &p, err, "eos_tq_quantize");
  }

  int prepare(const float* d_queries, int qb, int16_t* qs_out, char** err) {
    return prepare_cols(d_queries, qb, nqg_for(qb), 1, 1, qs_out, err);
  }

  int maxsim_nqg() const { return ks <= 8 ? 4 : ks <= 24 ? 2 : 1; }

  // Prepares nq queries of tq tokens (source rows [nq * tq][d]) at once: query
  // g is the 32-column group g (tokens past tq are zero columns), rounded up
  // to whole passes of the kernels that read them.
  // With `bounds` also each column's ||lo||_2 (ms_lonorm) for the high-half
  // bound filter.
  int maxsim_prepare(const float* d_src, int nq, int tq, char** err, bool bounds = false) {
    const int per = bounds && maxsim_wide(nq) ? 8 : maxsim_nqg();
    const int groups = (nq + per - 1) / per * per;
    const size_t cols = (size_t)groups * 32;
    if (ensure(reinterpret_cast<void**>(&ms_bfrag), &ms_bfrag_bytes, (size_t)ks * 2 * groups * 64 * 16,
               err) != 0 ||
        ensure(reinterpret_cast<void**>(&ms_alpha), &ms_alpha_bytes, cols * sizeof(float), err) != 0 ||
        (bounds && ensure(reinterpret_cast<void**>(&ms_lonorm), &ms_lonorm_bytes,
                          cols * sizeof(float), err) != 0) ||
        (rot_t != nullptr && ensure(reinterpret_cast<void**>(&ms_qrot), &ms_qrot_bytes,
                                    cols * (size_t)d * sizeof(double), err) != 0))
      return 1;
    ms_ncb = 2 * groups;
    TqPrepArgs p;
    memset(&p, 0, sizeof(p));
    p.bfrag = ms_bfrag;
    p.alpha = ms_alpha;
    p.qrot = ms_qrot;
    p.lonorm = bounds ? ms_lonorm : nullptr;
    return prepare_into(&p, d_src, nq * tq, groups, 32, tq, nullptr, err);
  }

  // Arguments of a MaxSim launch over the prepared chunk's groups [g0, g0 +
  // groups) (maxsim_launch splits them into passes on blockIdx.y).
  TqMaxsimArgs maxsim_args(int g0, int groups, int doc_len) const {
    TqMaxsimArgs m;
    memset(&m, 0, sizeof(m));
    m.packed = static_cast<const int32_t*>(packed);
    m.norms = norms;
    m.bfrag = ms_bfrag;
    m.alpha = ms_alpha + (size_t)g0 * 32;
    m.frag_ncb = ms_ncb;
    m.frag_cb0 = 2 * g0;
    m.tiles_per_doc = doc_len / kTile;
    m.groups = groups;
    m.lut0 = lut[0];
    m.lut1 = lut[1];
    m.lut2 = lut[2];
    m.lut3 = lut[3];
    return m;
  }

  // The bound filter over 8 groups a pass: at short K its per-tile work
  // (decode, norms) is a third of the instructions at 4 groups. Not where the
  // rounding up to 8 adds a group pass to three or fewer. Whole calls over
  // 100,000 documents x 128 rows of dim 128, 32 tokens, 4 groups / 8 a pass: 5
  // queries 642 / 512 us, 9 846 / 906, 12 904 / 943, 13 1,146 / 962, 17 1,443 /
  // 1,427, 20 1,462 / 1,456, 25 2,023 / 1,928, 32 2,299 / 2,000.
  bool maxsim_wide(int groups) const {
    const int p4 = (groups + 3) / 4;
    return ks <= 4 && p4 > 1 && (p4 % 2 == 0 || p4 >= 5);
  }

  // Launches MaxSim kernel `hi` (bound filter) or exact over `docs` documents
  // per pass, for m.groups groups; listed documents are scored one group a
  // pass (each group has its own list).
  int maxsim_launch(TqMaxsimArgs* m, bool hi, int64_t docs, const char* label, char** err) {
    int nqg = maxsim_nqg();
    if (hi && maxsim_wide(m->groups)) nqg = 8;
    if (m->doc_list != nullptr) nqg = 1;
    char name[64];
    snprintf(name, sizeof(name), "eos_tq_maxsim_b%d_k%d_g%d%s", bits, ks, nqg, hi ? "_h" : "");
    // As many resident workgroups as the kernel's registers allow (three
    // waves per SIMD for most variants), each wave striding over documents;
    // the passes share them.
    int per_cu = 2;
    if (rt->blocks_per_cu(name, 256, 0, &per_cu, err) != 0) return 1;
    const int passes = (m->groups + nqg - 1) / nqg;
    int64_t blocks = (docs + 3) / 4;
    const int64_t maxb = std::max<int64_t>(1, (int64_t)rt->compute_units * per_cu / passes);
    if (blocks > maxb) blocks = maxb;
    if (blocks < 1) blocks = 1;
    return rt->launch(name, dim3((unsigned)blocks, (unsigned)passes), dim3(256), 0, m, err, label);
  }

  // Doc scores of the prepared queries [q0, q0 + qp) (qp <= maxsim_nqg(),
  // q0 a multiple of it) for documents [doc_begin, doc_begin + ndocs) into
  // out [qp][ndocs].
  int maxsim_pass(int q0, int qp, int doc_len, int64_t doc_begin, int64_t ndocs, float* out,
                  char** err) {
    TqMaxsimArgs m = maxsim_args(q0, qp, doc_len);
    m.out = out;
    m.doc_begin = doc_begin;
    m.ndocs = ndocs;
    m.out_stride = ndocs;
    return maxsim_launch(&m, false, ndocs, "tq_maxsim", err);
  }

  // Exhaustive scores of all queries of the batch into dense [qb][count].
  int dense_scores(int qb, int64_t begin, int64_t count, bool want_dots, char** err) {
    const size_t need = (size_t)qb * (size_t)count * sizeof(float);
    if (ensure(reinterpret_cast<void**>(&dense), &dense_bytes, need, err) != 0) return 1;
    if (want_dots &&
        ensure(reinterpret_cast<void**>(&dense_dots), &dense_dots_bytes,
               (size_t)qb * (size_t)count * sizeof(int32_t), err) != 0)
      return 1;
    TqScanArgs s;
    scan_base(&s, qb);
    s.mode = 0;
    s.out_scores = dense;
    s.out_dots = want_dots ? dense_dots : nullptr;
    s.out_begin = begin;
    s.out_count = count;
    s.out_stride = count;
    s.tile_begin = begin / kTile;
    const int64_t tile_end = (begin + count + kTile - 1) / kTile;
    s.ntiles = (int)(tile_end - s.tile_begin);
    return launch_scan(&s, qb, err);
  }

  // Enqueues one batch on the runtime stream (no host synchronisation):
  // prepare, sample + threshold, filter scan, finalize. Finalize writes each
  // query's status to d_status (0: its row is final; 1: fewer than k kept;
  // 2: the kept set overflowed). With `gated` the exact fallback follows on
  // the device, gated by those flags, so the rows are exact when the stream
  // reaches that point; otherwise flagged rows wait for fallback_batch.
  int topk_batch(const float* d_queries, int qb, int kk, int64_t* d_ids, float* d_scores,
                 int* d_status, bool gated, char** err) {
    if (prepare(d_queries, qb, qs_buf, err) != 0) return 1;
    if (n > kCap) {
      const int64_t stride = std::max<int64_t>(kSampleStride, (ntiles + kMaxSampleTiles - 1) / kMaxSampleTiles);
      const int64_t ns = (ntiles + stride - 1) / stride;
      int64_t nsv = 0;
      for (int64_t j = 0; j < ns; ++j) nsv += std::min<int64_t>(kTile, n - j * stride * kTile);
      const double target = std::min<double>(kKeepFactor * kk, kCap / 4.0);
      int64_t r = (int64_t)std::ceil(target * (double)nsv / (double)n);
      r = std::max<int64_t>(1, std::min<int64_t>(r, ns));  // r-th best of ns tile maxima
      TqScanArgs s;
      scan_base(&s, qb);
      s.mode = 2;
      s.out_scores = samp;
      s.out_stride = ns;
      s.tile_begin = 0;
      s.tile_step = stride;
      s.ntiles = (int)ns;
      if (launch_scan(&s, qb, err) != 0) return 1;
      TqSelectArgs sel;
      memset(&sel, 0, sizeof(sel));
      sel.rows = samp;
      sel.tau = tau;
      sel.n = ns;
      sel.stride = ns;
      sel.kk = (int)r;
      sel.nrows = qb;
      if (rt->launch("eos_tq_threshold", dim3(qb), dim3(256), 0, &sel, err) != 0) return 1;
    }
    // High-half filter (ids whose score bound reaches tau), then their exact
    // scores: the kept set equals the exact filter's.
    TqScanArgs s;
    scan_base(&s, qb);
    s.mode = 3;
    s.tile_begin = 0;
    s.ntiles = (int)ntiles;
    if (launch_scan(&s, qb, err) != 0) return 1;
    TqRescoreArgs rs;
    memset(&rs, 0, sizeof(rs));
    rs.codes = codes_rm;
    rs.norms = norms;
    rs.qs = qs_buf;
    rs.alpha = alpha;
    rs.tau = tau;
    rs.cand = cand;
    rs.cand_count = cand_count;
    rs.n = n;
    rs.q = qb;
    rs.d = d;
    rs.rs = rs16;
    rs.cap = kCap;
    rs.lut0 = lut[0];
    rs.lut1 = lut[1];
    rs.lut2 = lut[2];
    rs.lut3 = lut[3];
    if (rt->launch(bits == 4 ? "eos_tq_rescore_b4" : "eos_tq_rescore_b2", dim3(qb, kRescoreBlocks),
                   dim3(256), 0, &rs, err, "tq_rescore") != 0)
      return 1;
    TqFinalizeArgs f;
    memset(&f, 0, sizeof(f));
    f.cand = cand;
    f.cand_count = cand_count;
    f.ids = reinterpret_cast<long long*>(d_ids);
    f.scores = d_scores;
    f.status = d_status;
    f.cap = kCap;
    f.kk = kk;
    f.q = qb;
    f.id_map = id_map;
    if (rt->launch(finalize_kernel(f.kk), dim3(qb), dim3(256), 0, &f, err, "eos_tq_finalize") != 0)
      return 1;
    if (gated) return fallback_batch(d_queries, qb, kk, d_ids, d_scores, d_status, false, err);
    return 0;
  }

  // Exact fallback of one batch, gated on the device by d_status: exhaustive
  // scores of the batch (skipped by every workgroup when no query is
  // flagged) and an exact radix selection for each flagged row. `reprepare`
  // rebuilds the query fragments first (another batch may have used them).
  int fallback_batch(const float* d_queries, int qb, int kk, int64_t* d_ids, float* d_scores,
                     const int* d_status, bool reprepare, char** err) {
    if (ensure(reinterpret_cast<void**>(&dense), &dense_bytes, (size_t)qb * (size_t)n * sizeof(float),
               err) != 0)
      return 1;
    if (reprepare && prepare(d_queries, qb, nullptr, err) != 0) return 1;
    TqScanArgs ds;
    scan_base(&ds, qb);
    ds.mode = 0;
    ds.gate = d_status;
    ds.out_scores = dense;
    ds.out_begin = 0;
    ds.out_count = n;
    ds.out_stride = n;
    ds.tile_begin = 0;
    ds.ntiles = (int)ntiles;
    if (launch_scan(&ds, qb, err) != 0) return 1;
    TqSelectArgs sel;
    memset(&sel, 0, sizeof(sel));
    sel.rows = dense;
    sel.status = d_status;
    sel.ids = reinterpret_cast<long long*>(d_ids);
    sel.scores = d_scores;
    sel.n = n;
    sel.stride = n;
    sel.kk = kk;
    sel.mode = 1;
    sel.nrows = qb;
    sel.id_map = id_map;
    return rt->launch("eos_tq_row_select", dim3(qb), dim3(1024), 0, &sel, err, "tq_fallback_select");
  }

  // Waits for the batch and reads its per-query status (and kept counts for
  // the statistics); returns the number of flagged queries in *flagged.
  int batch_status(int qb, const int* d_status, EosHipTQStats* st, int* flagged, char** err) {
    int hstatus[kBatch];
    uint32_t hcount[kBatch];
    hipError_t e = rt->copy_async(hstatus, d_status, sizeof(int) * qb, hipMemcpyDeviceToHost);
    if (e == hipSuccess && st)
      e = rt->copy_async(hcount, cand_count, sizeof(uint32_t) * qb, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(status)", e);
    if (rt->sync(err) != 0) return 1;
    int nf = 0;
    for (int i = 0; i < qb; ++i) {
      if (hstatus[i] != 0) ++nf;
      if (st) st->candidates_kept += std::min<uint32_t>(hcount[i], (uint32_t)kCap);
    }
    if (st) {
      st->fallback_queries += nf;
      st->candidate_count += (int64_t)qb * n;
      st->batches += 1;
    }
    *flagged = nf;
    return 0;
  }
};

extern "C" {

int eoship_tq_bind_corpus(EosHipRuntime* rt, const EosHipTQDesc* desc, const uint8_t* codes,
                          const float* norms, int64_t n, EosHipTQ** out, char** err) {
  return eoship_tq_bind_corpus_opts(rt, desc, codes, norms, n, nullptr, out, err);
}

int eoship_tq_bind_corpus_opts(EosHipRuntime* rt, const EosHipTQDesc* desc, const uint8_t* codes,
                               const float* norms, int64_t n, const EosHipTQBindOptions* opts,
                               EosHipTQ** out, char** err) {
  if (rt == nullptr || desc == nullptr || out == nullptr)
    return set_err(err, "eoship_tq_bind_corpus: NULL argument");
  *out = nullptr;
  if (desc->bits != 2 && desc->bits != 4)
    return set_err(err, "eoship_tq_bind_corpus: bits must be 2 or 4 (got %d)", desc->bits);
  const int ks = ks_for_dim(desc->dim);
  if (desc->dim < 1 || ks == 0)
    return set_err(err, "eoship_tq_bind_corpus: dim must be in [1, 1024] (got %d)", desc->dim);
  if (!(desc->codebook_scale > 0.f) || !std::isfinite(desc->codebook_scale))
    return set_err(err, "eoship_tq_bind_corpus: codebook_scale must be finite and > 0");
  if (desc->codebook == nullptr) return set_err(err, "eoship_tq_bind_corpus: codebook is NULL");
  if (n < 0 || n >= (int64_t)0xffffffffLL)
    return set_err(err, "eoship_tq_bind_corpus: n must be in [0, 2^32-1) (got %lld)", (long long)n);
  if (n > 0 && (codes == nullptr || norms == nullptr))
    return set_err(err, "eoship_tq_bind_corpus: codes/norms are NULL");
  // validateEosQuantizedVectorNorm (runtime/turboquant_quantized_vector.go:
  // 25-34): Norm > 0 is accepted, Norm == 0 only for a vector the caller
  // confirms as the genuine zero vector, anything else is refused. Infinite
  // norms are refused too (the reference would score them as +-inf or NaN).
  const uint8_t* zero_ok = opts != nullptr ? opts->zero_vector_allowed : nullptr;
  for (int64_t i = 0; i < n; ++i) {
    const float nv = norms[i];
    if (nv > 0.f && std::isfinite(nv)) continue;
    if (nv == 0.f && zero_ok != nullptr && zero_ok[i] != 0) continue;
    if (nv == 0.f)
      return set_err(err,
                     "eoship_tq_bind_corpus: vector %lld has Norm 0; refusing to score a vector that "
                     "dropped its input-norm field (set zero_vector_allowed only for a confirmed "
                     "genuine zero-vector input)",
                     (long long)i);
    return set_err(err,
                   "eoship_tq_bind_corpus: vector %lld has non-positive or non-finite Norm %g",
                   (long long)i, (double)nv);
  }
  // Optional ID order: a permutation of 0..n-1, checked before anything is
  // allocated; codes and norms are laid out in that order.
  const int64_t* id_rank = opts != nullptr ? opts->id_rank : nullptr;
  std::vector<uint8_t> codes_perm;
  std::vector<float> norms_perm;
  std::vector<long long> map_host;
  const size_t row_bytes_in = (size_t)(desc->dim * desc->bits + 7) / 8;
  if (id_rank != nullptr && n > 0) {
    std::vector<uint8_t> seen((size_t)n, 0);
    map_host.resize((size_t)n);
    for (int64_t i = 0; i < n; ++i) {
      const int64_t r = id_rank[i];
      if (r < 0 || r >= n || seen[(size_t)r])
        return set_err(err, "eoship_tq_bind_corpus: id_rank is not a permutation of 0..n-1 (entry %lld = %lld)",
                       (long long)i, (long long)r);
      seen[(size_t)r] = 1;
      map_host[(size_t)r] = (long long)i;
    }
    codes_perm.resize((size_t)n * row_bytes_in);
    norms_perm.resize((size_t)n);
    for (int64_t i = 0; i < n; ++i) {
      const size_t r = (size_t)id_rank[i];
      memcpy(&codes_perm[r * row_bytes_in], codes + (size_t)i * row_bytes_in, row_bytes_in);
      norms_perm[r] = norms[i];
    }
    codes = codes_perm.data();
    norms = norms_perm.data();
  }
  auto* tq = new EosHipTQ();
  if (id_rank != nullptr && n > 0) tq->rank_host.assign(id_rank, id_rank + n);
  tq->rt = rt;
  tq->d = desc->dim;
  tq->bits = desc->bits;
  tq->ks = ks;
  const int spl = 8 / desc->bits;
  tq->nload = (ks + spl - 1) / spl;
  tq->row_bytes = (desc->dim * desc->bits + 7) / 8;
  tq->n = n;
  tq->ntiles = (n + kTile - 1) / kTile;
  tq->cb_scale = desc->codebook_scale;
  const int levels = 1 << desc->bits;
  int cmax = 0;
  for (int v = 0; v < levels; ++v) {
    tq->codebook[v] = desc->codebook[v];
    cmax = std::max(cmax, std::abs((int)desc->codebook[v]));
  }
  if (cmax == 0) {
    tq->qmax = kQmaxLimit;
  } else {
    const int64_t lim = (int64_t)2147483647 / ((int64_t)cmax * desc->dim) - 128;
    tq->qmax = (int)std::min<int64_t>(kQmaxLimit, lim);
  }
  if (tq->qmax < 1) {
    delete tq;
    return set_err(err, "eoship_tq_bind_corpus: dim too large for exact int32 dots");
  }
  if (desc->bits == 4) {
    if (solve_lut4(tq->codebook, tq->lut, err) != 0) {
      delete tq;
      return 1;
    }
  } else {
    tq->lut[0] = (uint8_t)tq->codebook[0] | ((uint8_t)tq->codebook[1] << 8) |
                 ((uint8_t)tq->codebook[2] << 16) | ((uint32_t)(uint8_t)tq->codebook[3] << 24);
  }
  auto fail = [&](void) {
    tq->free_all();
    delete tq;
    return 1;
  };
  hipError_t e = hipSetDevice(rt->device);
  if (e != hipSuccess) {
    hip_err(err, "hipSetDevice", e);
    return fail();
  }
  const int64_t padded = tq->ntiles * kTile;
  const size_t packed_bytes = (size_t)tq->ntiles * tq->nload * 64 * 16;
  if (rt->alloc(packed_bytes, &tq->packed, err) != 0) return fail();
  if (rt->alloc((size_t)std::max<int64_t>(padded, 1) * sizeof(float),
                reinterpret_cast<void**>(&tq->norms), err) != 0)
    return fail();
  e = hipMemsetAsync(tq->norms, 0, (size_t)std::max<int64_t>(padded, 1) * sizeof(float), rt->stream);
  if (e != hipSuccess) {
    hip_err(err, "hipMemsetAsync(norms)", e);
    return fail();
  }
  if (n > 0) {
    e = rt->copy_async(tq->norms, norms, (size_t)n * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      hip_err(err, "hipMemcpyAsync(norms)", e);
      return fail();
    }
    void* dcodes = nullptr;
    const size_t code_bytes = (size_t)n * tq->row_bytes;
    if (rt->alloc(code_bytes, &dcodes, err) != 0) return fail();
    e = rt->copy_async(dcodes, codes, code_bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      hipFree(dcodes);
      hip_err(err, "hipMemcpyAsync(codes)", e);
      return fail();
    }
    if (rt->alloc((size_t)tq->ntiles * 2 * sizeof(float), reinterpret_cast<void**>(&tq->tile_cn), err) != 0) {
      hipFree(dcodes);
      return fail();
    }
    TqTileNormArgs tn;
    memset(&tn, 0, sizeof(tn));
    tn.codes = static_cast<const uint8_t*>(dcodes);
    tn.norms = tq->norms;
    tn.tile_cn = tq->tile_cn;
    tn.n = n;
    tn.d = tq->d;
    tn.bits = tq->bits;
    tn.row_bytes = tq->row_bytes;
    for (int v = 0; v < levels; ++v) tn.cb[v] = tq->codebook[v];
    if (rt->launch("eos_tq_tile_cnorm", dim3((unsigned)((n + 255) / 256)), dim3(256), 0, &tn, err) != 0) {
      rt->sync(nullptr);
      hipFree(dcodes);
      return fail();
    }
    TqPackArgs p;
    memset(&p, 0, sizeof(p));
    p.codes = static_cast<const uint8_t*>(dcodes);
    p.packed = static_cast<uint32_t*>(tq->packed);
    p.n = n;
    p.total_dwords = (long long)(packed_bytes / 4);
    p.d = tq->d;
    p.bits = tq->bits;
    p.row_bytes = tq->row_bytes;
    p.ks = tq->ks;
    p.nload = tq->nload;
    const int64_t blocks = (p.total_dwords + 255) / 256;
    if (rt->launch("eos_tq_pack", dim3((unsigned)blocks), dim3(256), 0, &p, err) != 0) {
      rt->sync(nullptr);
      hipFree(dcodes);
      return fail();
    }
    const int rc = rt->sync(err);
    if (rc != 0) {
      hipFree(dcodes);
      return fail();
    }
    // The reference-layout rows stay resident for the exact rescoring of
    // kept ids, padded to whole 16-byte chunks (at most 32: 1024 dims at 4
    // bits); rows that already are whole chunks are kept as uploaded.
    tq->rs16 = (tq->row_bytes + 15) / 16;
    const size_t pitch = (size_t)tq->rs16 * 16;
    if (pitch == (size_t)tq->row_bytes) {
      tq->codes_rm = static_cast<uint8_t*>(dcodes);
    } else {
      if (rt->alloc((size_t)n * pitch, reinterpret_cast<void**>(&tq->codes_rm), err) != 0) {
        hipFree(dcodes);
        return fail();
      }
      e = hipMemsetAsync(tq->codes_rm, 0, (size_t)n * pitch, rt->stream);
      if (e == hipSuccess)
        e = hipMemcpy2DAsync(tq->codes_rm, pitch, dcodes, tq->row_bytes, tq->row_bytes, (size_t)n,
                             hipMemcpyDeviceToDevice, rt->stream);
      if (e == hipSuccess) {
        ++rt->n_syncs;
        e = hipStreamSynchronize(rt->stream);
      }
      hipFree(dcodes);
      if (e != hipSuccess) {
        hip_err(err, "hipMemcpy2DAsync(code rows)", e);
        return fail();
      }
    }
  }
  if (tq->alloc_scratch(err) != 0) return fail();
  if (desc->rotation != nullptr && tq->prepare_rotation(desc->rotation, err) != 0) return fail();
  if (!map_host.empty()) {
    if (rt->alloc(map_host.size() * sizeof(long long), reinterpret_cast<void**>(&tq->id_map), err) != 0)
      return fail();
    e = rt->copy_sync(tq->id_map, map_host.data(), map_host.size() * sizeof(long long), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      hip_err(err, "hipMemcpy(id_map)", e);
      return fail();
    }
  }
  *out = tq;
  return 0;
}

int eoship_tq_vector_bytes(int32_t dim, int32_t bit_width, int64_t* bytes, char** err) {
  if (bytes == nullptr) return set_err(err, "eoship_tq_vector_bytes: NULL output");
  if (dim < 1 || bit_width < 1 || bit_width > 8)
    return set_err(err, "eoship_tq_vector_bytes: dim must be >= 1 and bit_width in [1, 8]");
  const int64_t mse = ((int64_t)dim * (bit_width - 1) + 7) / 8;
  const int64_t signs = ((int64_t)dim + 7) / 8;
  *bytes = mse + signs + 8;
  return 0;
}

int eoship_tq_mse_vector_bytes(int32_t dim, int32_t bits, int64_t* bytes, char** err) {
  if (bytes == nullptr) return set_err(err, "eoship_tq_mse_vector_bytes: NULL output");
  if (dim < 1 || bits < 1 || bits > 8)
    return set_err(err, "eoship_tq_mse_vector_bytes: dim must be >= 1 and bits in [1, 8]");
  *bytes = ((int64_t)dim * bits + 7) / 8 + 4;
  return 0;
}

int eoship_tq_share(EosHipRuntime* rt, EosHipTQ* src, EosHipTQ** out, char** err) {
  if (rt == nullptr || src == nullptr || out == nullptr)
    return set_err(err, "eoship_tq_share: NULL argument");
  *out = nullptr;
  if (rt->device != src->rt->device)
    return set_err(err, "eoship_tq_share: runtime is on device %d, the corpus on device %d",
                   rt->device, src->rt->device);
  // The corpus arrays are complete: the bind synchronised its stream.
  auto* tq = new EosHipTQ();
  tq->rt = rt;
  tq->d = src->d;
  tq->bits = src->bits;
  tq->ks = src->ks;
  tq->nload = src->nload;
  tq->row_bytes = src->row_bytes;
  tq->qmax = src->qmax;
  tq->n = src->n;
  tq->ntiles = src->ntiles;
  tq->cb_scale = src->cb_scale;
  memcpy(tq->codebook, src->codebook, sizeof(tq->codebook));
  memcpy(tq->lut, src->lut, sizeof(tq->lut));
  tq->rs16 = src->rs16;
  tq->rank_host = src->rank_host;
  if (tq->alloc_scratch(err) != 0) {
    tq->free_all();  // scratch only: the corpus arrays are not attached yet
    delete tq;
    return 1;
  }
  if (src->corpus_refs == nullptr) src->corpus_refs = new int(1);
  tq->corpus_refs = src->corpus_refs;
  ++*tq->corpus_refs;
  tq->packed = src->packed;
  tq->norms = src->norms;
  tq->rot_t = src->rot_t;
  tq->rot_r = src->rot_r;
  tq->rot_frag = src->rot_frag;
  tq->rot_rmax = src->rot_rmax;
  tq->enc_delta2 = src->enc_delta2;
  tq->tile_cn = src->tile_cn;
  tq->codes_rm = src->codes_rm;
  tq->id_map = src->id_map;
  *out = tq;
  return 0;
}

int eoship_tq_release(EosHipTQ* tq, char** err) {
  (void)err;
  if (tq == nullptr) return 0;
  (void)tq->rt->sync(nullptr);
  tq->free_all();
  delete tq;
  return 0;
}

static int check_common(EosHipRuntime* rt, EosHipTQ* tq, int32_t q, const char* what, char** err) {
  if (rt == nullptr || tq == nullptr) return set_err(err, "%s: NULL runtime or corpus", what);
  if (tq->rt != rt) return set_err(err, "%s: corpus was bound on another runtime", what);
  if (q < 0) return set_err(err, "%s: negative query count", what);
  return 0;
}

// Batches of <= 64 queries through the pipeline. mode 0: the device-gated
// exact fallback follows every batch (no host wait). mode 1: statuses go to
// d_status_out and flagged rows are left for eoship_tq_topk_repair_device.
// mode 2 (host API): each batch is awaited and the fallback runs only for a
// batch with a flagged query.
static int topk_device_impl(EosHipRuntime* rt, EosHipTQ* tq, const float* d_queries, int32_t q,
                            int32_t k, int64_t* d_ids, float* d_scores, EosHipTQStats* stats,
                            int mode, int32_t* d_status_out, char** err) {
  if (stats) memset(stats, 0, sizeof(*stats));
  const int64_t kk64 = (k <= 0 || (int64_t)k > tq->n) ? tq->n : k;
  if (q == 0 || kk64 == 0) return 0;
  if (kk64 > kSortCap)
    return set_err(err, "eoship_tq_topk: k=%lld exceeds the device top-k limit of %d",
                   (long long)kk64, kSortCap);
  const int kk = (int)kk64;
  const int cap = tq->batch_cap();
  for (int q0 = 0; q0 < q; q0 += cap) {
    const int qb = std::min(cap, q - q0);
    const float* dq = d_queries + (size_t)q0 * tq->d;
    int64_t* di = d_ids + (size_t)q0 * kk;
    float* ds = d_scores + (size_t)q0 * kk;
    int* st = mode == 1 ? d_status_out + q0 : tq->status;
    if (tq->topk_batch(dq, qb, kk, di, ds, st, mode == 0, err) != 0) return 1;
    if (mode == 2 || stats) {
      int flagged = 0;
      if (tq->batch_status(qb, st, stats, &flagged, err) != 0) return 1;
      if (mode == 2 && flagged > 0 && tq->fallback_batch(dq, qb, kk, di, ds, st, false, err) != 0)
        return 1;
    }
  }
  return 0;
}

int eoship_tq_topk_device(EosHipRuntime* rt, EosHipTQ* tq, const float* d_queries, int32_t q,
                          int32_t k, int64_t* d_ids, float* d_scores, EosHipTQStats* stats,
                          char** err) {
  if (check_common(rt, tq, q, "eoship_tq_topk_device", err) != 0) return 1;
  if (q > 0 && (d_queries == nullptr || d_ids == nullptr || d_scores == nullptr))
    return set_err(err, "eoship_tq_topk_device: NULL buffer");
  return topk_device_impl(rt, tq, d_queries, q, k, d_ids, d_scores, stats, 0, nullptr, err);
}

int eoship_tq_topk_device_deferred(EosHipRuntime* rt, EosHipTQ* tq, const float* d_queries,
                                   int32_t q, int32_t k, int64_t* d_ids, float* d_scores,
                                   int32_t* d_status, char** err) {
  if (check_common(rt, tq, q, "eoship_tq_topk_device_deferred", err) != 0) return 1;
  if (q > 0 && (d_queries == nullptr || d_ids == nullptr || d_scores == nullptr || d_status == nullptr))
    return set_err(err, "eoship_tq_topk_device_deferred: NULL buffer");
  return topk_device_impl(rt, tq, d_queries, q, k, d_ids, d_scores, nullptr, 1, d_status, err);
}

int eoship_tq_topk_repair_device(EosHipRuntime* rt, EosHipTQ* tq, const float* d_queries, int32_t q,
                                 int32_t k, int64_t* d_ids, float* d_scores,
                                 const int32_t* d_status, char** err) {
  if (check_common(rt, tq, q, "eoship_tq_topk_repair_device", err) != 0) return 1;
  const int64_t kk64 = (k <= 0 || (int64_t)k > tq->n) ? tq->n : k;
  if (q == 0 || kk64 == 0) return 0;
  if (d_queries == nullptr || d_ids == nullptr || d_scores == nullptr || d_status == nullptr)
    return set_err(err, "eoship_tq_topk_repair_device: NULL buffer");
  if (kk64 > kSortCap)
    return set_err(err, "eoship_tq_topk_repair_device: k=%lld exceeds the device top-k limit of %d",
                   (long long)kk64, kSortCap);
  const int kk = (int)kk64;
  const int cap = tq->batch_cap();
  for (int q0 = 0; q0 < q; q0 += cap) {
    const int qb = std::min(cap, q - q0);
    if (tq->fallback_batch(d_queries + (size_t)q0 * tq->d, qb, kk, d_ids + (size_t)q0 * kk,
                           d_scores + (size_t)q0 * kk, d_status + q0, true, err) != 0)
      return 1;
  }
  return 0;
}

int eoship_tq_topk(EosHipRuntime* rt, EosHipTQ* tq, const float* queries, int32_t q, int32_t k,
                   int64_t* ids, float* scores, EosHipTQStats* stats, char** err) {
  if (check_common(rt, tq, q, "eoship_tq_topk", err) != 0) return 1;
  const int64_t kk = (k <= 0 || (int64_t)k > tq->n) ? tq->n : k;
  if (stats) memset(stats, 0, sizeof(*stats));
  if (q == 0 || kk == 0) return 0;
  if (queries == nullptr || ids == nullptr || scores == nullptr)
    return set_err(err, "eoship_tq_topk: NULL buffer");
  const size_t qbytes = (size_t)q * tq->d * sizeof(float);
  const size_t ibytes = (size_t)q * kk * sizeof(int64_t);
  const size_t sbytes = (size_t)q * kk * sizeof(float);
  if (tq->ensure(&tq->io, &tq->io_bytes, qbytes + ibytes + sbytes + 256, err) != 0) return 1;
  char* base = static_cast<char*>(tq->io);
  float* dq = reinterpret_cast<float*>(base);
  int64_t* di = reinterpret_cast<int64_t*>(base + ((qbytes + 15) & ~(size_t)15));
  float* ds = reinterpret_cast<float*>(reinterpret_cast<char*>(di) + ibytes);
  hipError_t e = rt->copy_async(dq, queries, qbytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(queries)", e);
  if (topk_device_impl(rt, tq, dq, q, k, di, ds, stats, 2, nullptr, err) != 0) return 1;
  e = rt->copy_async(ids, di, ibytes, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = rt->copy_async(scores, ds, sbytes, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(results)", e);
  return rt->sync(err);
}

int eoship_tq_scores(EosHipRuntime* rt, EosHipTQ* tq, const float* queries, int32_t q,
                     int64_t begin, int64_t count, int32_t* dots, float* scores, char** err) {
  if (check_common(rt, tq, q, "eoship_tq_scores", err) != 0) return 1;
  if (begin < 0 || count < 0 || begin + count > tq->n)
    return set_err(err, "eoship_tq_scores: range [%lld, %lld) outside [0, %lld)", (long long)begin,
                   (long long)(begin + count), (long long)tq->n);
  if (q == 0 || count == 0) return 0;
  if (queries == nullptr) return set_err(err, "eoship_tq_scores: queries is NULL");
  const size_t qbytes = (size_t)q * tq->d * sizeof(float);
  if (tq->ensure(&tq->io, &tq->io_bytes, qbytes, err) != 0) return 1;
  float* dq = static_cast<float*>(tq->io);
  hipError_t e = rt->copy_async(dq, queries, qbytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(queries)", e);
  const int cap = tq->batch_cap();
  if (tq->id_map != nullptr) {
    // Ranked corpus: vector i sits at position rank[i]; every position is
    // scored and the requested vectors are picked out on the host.
    const int64_t n = tq->n;
    std::vector<float> hs(scores ? (size_t)cap * n : 0);
    std::vector<int32_t> hd(dots ? (size_t)cap * n : 0);
    for (int q0 = 0; q0 < q; q0 += cap) {
      const int qb = std::min(cap, q - q0);
      if (tq->prepare(dq + (size_t)q0 * tq->d, qb, nullptr, err) != 0) return 1;
      if (tq->dense_scores(qb, 0, n, dots != nullptr, err) != 0) return 1;
      if (scores) e = rt->copy_async(hs.data(), tq->dense, (size_t)qb * n * sizeof(float), hipMemcpyDeviceToHost);
      if (e == hipSuccess && dots)
        e = rt->copy_async(hd.data(), tq->dense_dots, (size_t)qb * n * sizeof(int32_t), hipMemcpyDeviceToHost);
      if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(scores)", e);
      if (rt->sync(err) != 0) return 1;
      for (int r = 0; r < qb; ++r)
        for (int64_t j = 0; j < count; ++j) {
          const size_t src = (size_t)r * n + (size_t)tq->rank_host[(size_t)(begin + j)];
          const size_t dst = (size_t)(q0 + r) * count + (size_t)j;
          if (scores) scores[dst] = hs[src];
          if (dots) dots[dst] = hd[src];
        }
    }
    return 0;
  }
  for (int q0 = 0; q0 < q; q0 += cap) {
    const int qb = std::min(cap, q - q0);
    if (tq->prepare(dq + (size_t)q0 * tq->d, qb, nullptr, err) != 0) return 1;
    if (tq->dense_scores(qb, begin, count, dots != nullptr, err) != 0) return 1;
    const size_t rows = (size_t)qb * count;
    if (scores) {
      e = rt->copy_async(scores + (size_t)q0 * count, tq->dense, rows * sizeof(float), hipMemcpyDeviceToHost);
      if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(scores)", e);
    }
    if (dots) {
      e = rt->copy_async(dots + (size_t)q0 * count, tq->dense_dots, rows * sizeof(int32_t), hipMemcpyDeviceToHost);
      if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(dots)", e);
    }
    if (rt->sync(err) != 0) return 1;
  }
  return 0;
}

int eoship_tq_prepare(EosHipRuntime* rt, EosHipTQ* tq, const float* queries, int32_t q,
                      int16_t* qs, float* alpha, char** err) {
  if (check_common(rt, tq, q, "eoship_tq_prepare", err) != 0) return 1;
  if (q == 0) return 0;
  if (queries == nullptr) return set_err(err, "eoship_tq_prepare: queries is NULL");
  const size_t qbytes = (size_t)q * tq->d * sizeof(float);
  if (tq->ensure(&tq->io, &tq->io_bytes, qbytes, err) != 0) return 1;
  if (tq->qs_buf == nullptr &&
      tq->rt->alloc((size_t)kBatch * tq->d * sizeof(int16_t), reinterpret_cast<void**>(&tq->qs_buf),
                    err) != 0)
    return 1;
  float* dq = static_cast<float*>(tq->io);
  hipError_t e = rt->copy_async(dq, queries, qbytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(queries)", e);
  const int cap = tq->batch_cap();
  for (int q0 = 0; q0 < q; q0 += cap) {
    const int qb = std::min(cap, q - q0);
    if (tq->prepare(dq + (size_t)q0 * tq->d, qb, tq->qs_buf, err) != 0) return 1;
    if (qs) {
      e = rt->copy_async(qs + (size_t)q0 * tq->d, tq->qs_buf, (size_t)qb * tq->d * sizeof(int16_t), hipMemcpyDeviceToHost);
      if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(qs)", e);
    }
    if (alpha) {
      e = rt->copy_async(alpha + q0, tq->alpha, (size_t)qb * sizeof(float), hipMemcpyDeviceToHost);
      if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(alpha)", e);
    }
    if (rt->sync(err) != 0) return 1;
  }
  return 0;
}

}  // extern "C"

namespace {

int maxsim_check(EosHipRuntime* rt, EosHipTQ* tq, int32_t doc_len, int32_t q, int32_t tq_tokens,
                 const char* what, char** err) {
  if (rt == nullptr || tq == nullptr) return set_err(err, "%s: NULL runtime or corpus", what);
  if (tq->rt != rt) return set_err(err, "%s: corpus was bound on another runtime", what);
  if (q < 0) return set_err(err, "%s: negative query count", what);
  if (tq->id_map != nullptr)
    return set_err(err, "%s: documents need their vectors in index order (corpus bound with id_rank)",
                   what);
  if (doc_len <= 0 || doc_len % kTile != 0)
    return set_err(err, "%s: doc_len must be a positive multiple of %d (got %d)", what, kTile, doc_len);
  if (tq->n % doc_len != 0)
    return set_err(err, "%s: corpus size %lld is not a whole number of %d-vector documents", what,
                   (long long)tq->n, doc_len);
  if (tq_tokens < 1 || tq_tokens > 32)
    return set_err(err, "%s: query tokens must be in [1, 32] (got %d)", what, tq_tokens);
  return 0;
}

// Chunks each of `rows` score rows of n splits into for its top kk: about one
// workgroup per CU in all, at least 2048 (and 4 kk) elements each, lists that
// eos_tq_finalize can merge.
int rank_chunks(EosHipRuntime* rt, int rows, int64_t n, int kk) {
  int64_t chunks = std::max<int64_t>(1, rt->compute_units / rows);
  chunks = std::min<int64_t>(chunks, kSortCap / kk);
  return (int)std::min<int64_t>(chunks, n / std::max<int64_t>(4 * (int64_t)kk, 2048));
}

// Top kk of each of `rows` score rows [rows][n] by (score desc, index asc)
// into ids / scores [rows][kk]. With few rows, each row is split into
// rank_chunks: every chunk's exact top kk (keys unique, so exactly kk or the
// whole chunk) into keys [rows][chunks * kk], then eos_tq_finalize merges
// each row's (counts and status [rows] are its scratch); with many rows (or
// a kk too large to merge) one workgroup ranks each row.
int rank_rows(EosHipRuntime* rt, const float* d_rows, int rows, int64_t n, int kk, int64_t* d_ids,
              float* d_scores, unsigned long long* keys, uint32_t* counts, int* status,
              const char* label, char** err, bool split = true) {
  TqSelectArgs sel;
  memset(&sel, 0, sizeof(sel));
  sel.rows = d_rows;
  sel.ids = reinterpret_cast<long long*>(d_ids);
  sel.scores = d_scores;
  sel.n = n;
  sel.stride = n;
  sel.kk = kk;
  sel.nrows = rows;
  const int nch = split ? rank_chunks(rt, rows, n, kk) : 1;
  if (nch < 2) {
    sel.mode = 1;
    return rt->launch("eos_tq_row_select", dim3(rows), dim3(1024), 0, &sel, err, label);
  }
  sel.mode = 2;
  sel.nchunks = nch;
  sel.keys_out = keys;
  sel.counts_out = counts;
  if (rt->launch("eos_tq_row_select", dim3(rows, nch), dim3(1024), 0, &sel, err, label) != 0)
    return 1;
  TqFinalizeArgs f;
  memset(&f, 0, sizeof(f));
  f.cand = keys;
  f.cand_count = counts;
  f.ids = reinterpret_cast<long long*>(d_ids);
  f.scores = d_scores;
  f.status = status;
  f.cap = nch * kk;
  f.kk = kk;
  f.q = rows;
  return rt->launch(finalize_kernel(f.kk), dim3(rows), dim3(256), 0, &f, err, label);
}

// Bound-filtered MaxSim top-k of one prepared chunk of cq queries (kk <=
// kMsMaxK, ndocs >= kMsMinDocs), all passes in each launch:
//  1. exact scores of every stride-th document (at most kMsSampleDocs), and
//     per query tau = the r-th best of them, r chosen so that about
//     min(3 kk, kMsTarget) documents of the corpus are expected above it;
//  2. the high-half bound filter over every document: a document is listed
//     for a query when its score bound reaches the query's tau (a bound >=
//     the exact score, so every document scoring >= tau is listed);
//  3. exact scores of the listed documents, the rank keys of those >= tau
//     kept per query, and the top kk of them (eos_tq_finalize): final when
//     there are at least kk, since every unlisted document scores below tau;
//  4. otherwise (too few, the list overflowed kMsList or the kept keys
//     kMsCap) the query is flagged and its row recomputed exhaustively, gated
//     on the device. The list holds the documents that only the bound lets
//     through too (at 100,000 documents x 128 rows of dim 128 about 2,000 for
//     430 above tau), so it has twice the keys' capacity.
// Results equal the exhaustive path's: the same exact scores, ranked by
// (score desc, document index asc).
constexpr int kMsCap = 8192;
constexpr int kMsList = 16384;
constexpr int kMsTarget = 1024;
constexpr int kMsSampleDocs = 2048;
constexpr int kMsMinDocs = 16384;
constexpr int kMsMaxK = 512;
// Least r with P(N >= r) <= 1 / 3000 for a Poisson count N of this mean.
int64_t maxsim_safe_rank(double mean) {
  double p = std::exp(-mean), below = p;  // P(N = r - 1), P(N < r)
  int64_t r = 1;
  while (1.0 - below > 1.0 / 3000 && r < kMsSampleDocs) {
    p *= mean / (double)r;
    below += p;
    ++r;
  }
  return r;
}

int maxsim_filtered(EosHipRuntime* rt, EosHipTQ* tq, int doc_len, int64_t ndocs, int cq, int kk,
                    int64_t* d_ids, float* d_scores, char** err) {
  const int64_t stride = std::max<int64_t>(16, (ndocs + kMsSampleDocs - 1) / kMsSampleDocs);
  const int64_t ns = (ndocs + stride - 1) / stride;
  const double target = std::min<double>(3.0 * kk, kMsTarget);
  int64_t r = (int64_t)std::ceil(target * (double)ns / (double)ndocs);
  // Fewer than kk documents score >= tau when r or more of the sample are
  // among the best kk - 1, a Poisson count of mean (kk - 1) ns / ndocs: r is
  // raised until that is one query in 3,000 or rarer (at 100,000 documents and
  // k = 100 3 kk alone, r = 7, gives one in 200: with 32 queries every seventh
  // call paid an exhaustive pass, 1.5 ms, where two more list entries in seven
  // cost 40 us), unless so many documents above tau would crowd the kept keys.
  // The best of the sample (r = 1) always does for kk = 1.
  const int64_t safe = maxsim_safe_rank((double)(kk - 1) * (double)ns / (double)ndocs);
  const int64_t room = (int64_t)((double)(kMsCap / 2) * (double)ns / (double)ndocs);
  r = std::max(r, std::min(safe, room));
  r = std::max<int64_t>(1, std::min<int64_t>(r, ns));
  // workspace: samples [cq][ns] f32, tau [cq], lists [cq][kMsList] u32, list
  // counts [cq][EOS_MS_COUNT] and key counts likewise (cleared together), rank
  // keys [cq][kMsCap] u64, status [cq]
  auto al = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t o_samp = 0;
  const size_t o_tau = o_samp + al((size_t)cq * ns * 4);
  const size_t o_list = o_tau + al((size_t)cq * 4);
  const size_t o_lcnt = o_list + al((size_t)cq * kMsList * 4);
  const size_t count_bytes = (size_t)cq * EOS_MS_COUNT * 4;
  const size_t o_ccnt = o_lcnt + count_bytes;
  const size_t o_cand = o_ccnt + count_bytes;
  const size_t o_stat = o_cand + al((size_t)cq * kMsCap * 8);
  const size_t total = o_stat + al((size_t)cq * 4);
  if (tq->ensure(&tq->ms_ws, &tq->ms_ws_bytes, total, err) != 0) return 1;
  char* w = static_cast<char*>(tq->ms_ws);
  float* samp = reinterpret_cast<float*>(w + o_samp);
  float* tau = reinterpret_cast<float*>(w + o_tau);
  uint32_t* list = reinterpret_cast<uint32_t*>(w + o_list);
  uint32_t* lcnt = reinterpret_cast<uint32_t*>(w + o_lcnt);
  unsigned long long* cand = reinterpret_cast<unsigned long long*>(w + o_cand);
  uint32_t* ccnt = reinterpret_cast<uint32_t*>(w + o_ccnt);
  int* status = reinterpret_cast<int*>(w + o_stat);
  // 1. sample and threshold
  TqMaxsimArgs m = tq->maxsim_args(0, cq, doc_len);
  m.out = samp;
  m.doc_begin = 0;
  m.doc_stride = stride;
  m.ndocs = ns;
  m.out_stride = ns;
  if (tq->maxsim_launch(&m, false, ns, "tq_maxsim_sample", err) != 0) return 1;
  TqSelectArgs sel;
  memset(&sel, 0, sizeof(sel));
  sel.rows = samp;
  sel.tau = tau;
  sel.n = ns;
  sel.stride = ns;
  sel.kk = (int)r;
  sel.nrows = cq;
  if (rt->launch("eos_tq_threshold", dim3((unsigned)cq), dim3(256), 0, &sel, err, "tq_maxsim_threshold") != 0)
    return 1;
  // 2. bound filter
  hipError_t e = hipMemsetAsync(lcnt, 0, 2 * count_bytes, rt->stream);
  if (e != hipSuccess) return hip_err(err, "hipMemsetAsync(list counts)", e);
  m = tq->maxsim_args(0, cq, doc_len);
  m.doc_begin = 0;
  m.ndocs = ndocs;
  m.tau = tau;
  m.lonorm = tq->ms_lonorm;
  m.tile_cn = tq->tile_cn;
  m.list = list;
  m.list_count = lcnt;
  m.list_cap = kMsList;
  if (tq->maxsim_launch(&m, true, ndocs, "tq_maxsim_filter", err) != 0) return 1;
  // 3. exact scores of the listed documents, then the top kk of each query
  m = tq->maxsim_args(0, cq, doc_len);
  m.ndocs = std::min<int64_t>(kMsList, ndocs);
  m.doc_list = list;
  m.list_count = lcnt;
  m.list_cap = kMsList;
  m.cand_cap = kMsCap;
  m.cand = cand;
  m.cand_count = ccnt;
  m.tau = tau;
  if (tq->maxsim_launch(&m, false, m.ndocs, "tq_maxsim_rescore", err) != 0) return 1;
  TqFinalizeArgs f;
  memset(&f, 0, sizeof(f));
  f.cand = cand;
  f.cand_count = ccnt;
  f.ids = reinterpret_cast<long long*>(d_ids);
  f.scores = d_scores;
  f.status = status;
  f.cap = kMsCap;
  f.kk = kk;
  f.q = cq;
  f.count_stride = EOS_MS_COUNT;
  if (rt->launch(finalize_kernel(f.kk), dim3((unsigned)cq), dim3(256), 0, &f, err, "tq_maxsim_finalize") != 0)
    return 1;
  // 4. exhaustive rows of the flagged queries (both launches return at once
  // when none is flagged)
  if (tq->ensure(reinterpret_cast<void**>(&tq->dense), &tq->dense_bytes,
                 (size_t)cq * (size_t)ndocs * sizeof(float), err) != 0)
    return 1;
  m = tq->maxsim_args(0, cq, doc_len);
  m.out = tq->dense;
  m.doc_begin = 0;
  m.ndocs = ndocs;
  m.out_stride = ndocs;
  m.gate = status;
  if (tq->maxsim_launch(&m, false, ndocs, "tq_maxsim_fallback", err) != 0) return 1;
  memset(&sel, 0, sizeof(sel));
  sel.rows = tq->dense;
  sel.status = status;
  sel.ids = reinterpret_cast<long long*>(d_ids);
  sel.scores = d_scores;
  sel.n = ndocs;
  sel.stride = ndocs;
  sel.kk = kk;
  sel.mode = 1;
  sel.nrows = cq;
  return rt->launch("eos_tq_row_select", dim3((unsigned)cq), dim3(1024), 0, &sel, err,
                    "tq_maxsim_fallback_select");
}

int maxsim_topk_impl(EosHipRuntime* rt, EosHipTQ* tq, int32_t doc_len, const float* d_queries,
                     int32_t q, int32_t tq_tokens, int32_t k, int64_t* d_ids, float* d_scores,
                     char** err) {
  const int64_t ndocs = tq->n / doc_len;
  const int64_t kk64 = (k <= 0 || (int64_t)k > ndocs) ? ndocs : k;
  if (q == 0 || kk64 == 0) return 0;
  if (kk64 > kSortCap)
    return set_err(err, "eoship_tq_maxsim_topk: k=%lld exceeds the device top-k limit of %d",
                   (long long)kk64, kSortCap);
  const int kk = (int)kk64;
  const int per = tq->maxsim_nqg();
  if (ndocs >= kMsMinDocs && kk <= kMsMaxK) {
    // Chunks of whole passes whose exhaustive fallback rows stay under 1 GiB.
    const int64_t by_mem = std::max<int64_t>(1, ((int64_t)1 << 30) / (ndocs * 4));
    const int chunk = (int)std::max<int64_t>(per, std::min<int64_t>(256, by_mem) / per * per);
    for (int c0 = 0; c0 < q; c0 += chunk) {
      const int cq = std::min(chunk, q - c0);
      if (tq->maxsim_prepare(d_queries + (size_t)c0 * tq_tokens * tq->d, cq, tq_tokens, err,
                             true) != 0 ||
          maxsim_filtered(rt, tq, doc_len, ndocs, cq, kk, d_ids + (size_t)c0 * kk,
                          d_scores + (size_t)c0 * kk, err) != 0)
        return 1;
    }
    return 0;
  }
  // The document scores of a chunk of queries (all of its scan passes) are
  // kept, so one select launch ranks every row of the chunk in parallel (one
  // workgroup per row; a select per pass ran only `per` workgroups at once).
  // Chunks are whole passes, and their score block stays under 1 GiB.
  const int64_t by_mem = std::max<int64_t>(1, ((int64_t)1 << 30) / (ndocs * 4));
  const int chunk = (int)std::max<int64_t>(per, std::min<int64_t>(256, by_mem) / per * per);
  const int rows = std::min(chunk, q);
  if (tq->ensure(reinterpret_cast<void**>(&tq->dense), &tq->dense_bytes,
                 (size_t)rows * (size_t)ndocs * sizeof(float), err) != 0)
    return 1;
  for (int c0 = 0; c0 < q; c0 += chunk) {
    const int cq = std::min(chunk, q - c0);
    // One preparation for every pass of the chunk.
    if (tq->maxsim_prepare(d_queries + (size_t)c0 * tq_tokens * tq->d, cq, tq_tokens, err) != 0)
      return 1;
    for (int q0 = 0; q0 < cq; q0 += per) {
      const int qp = std::min(per, cq - q0);
      if (tq->maxsim_pass(q0, qp, doc_len, 0, ndocs, tq->dense + (size_t)q0 * ndocs, err) != 0)
        return 1;
    }
    const int nch = std::max(1, rank_chunks(rt, cq, ndocs, kk));
    if (tq->ensure(reinterpret_cast<void**>(&tq->sel_keys), &tq->sel_keys_bytes,
                   (size_t)cq * nch * kk * sizeof(unsigned long long), err) != 0 ||
        tq->ensure(reinterpret_cast<void**>(&tq->sel_aux), &tq->sel_aux_bytes,
                   (size_t)cq * 2 * sizeof(uint32_t), err) != 0 ||
        rank_rows(rt, tq->dense, cq, ndocs, kk, d_ids + (size_t)c0 * kk,
                  d_scores + (size_t)c0 * kk, tq->sel_keys, tq->sel_aux,
                  reinterpret_cast<int*>(tq->sel_aux + cq), "tq_maxsim_select", err) != 0)
      return 1;
  }
  return 0;
}

}  // namespace

extern "C" {

int eoship_tq_maxsim_topk_device(EosHipRuntime* rt, EosHipTQ* tq, int32_t doc_len,
                                 const float* d_queries, int32_t q, int32_t tq_tokens, int32_t k,
                                 int64_t* d_ids, float* d_scores, char** err) {
  if (maxsim_check(rt, tq, doc_len, q, tq_tokens, "eoship_tq_maxsim_topk_device", err) != 0) return 1;
  if (q > 0 && (d_queries == nullptr || d_ids == nullptr || d_scores == nullptr))
    return set_err(err, "eoship_tq_maxsim_topk_device: NULL buffer");
  return maxsim_topk_impl(rt, tq, doc_len, d_queries, q, tq_tokens, k, d_ids, d_scores, err);
}

int eoship_tq_maxsim_topk(EosHipRuntime* rt, EosHipTQ* tq, int32_t doc_len, const float* queries,
                          int32_t q, int32_t tq_tokens, int32_t k, int64_t* ids, float* scores,
                          char** err) {
  if (maxsim_check(rt, tq, doc_len, q, tq_tokens, "eoship_tq_maxsim_topk", err) != 0) return 1;
  const int64_t ndocs = tq->n / doc_len;
  const int64_t kk = (k <= 0 || (int64_t)k > ndocs) ? ndocs : k;
  if (q == 0 || kk == 0) return 0;
  if (queries == nullptr || ids == nullptr || scores == nullptr)
    return set_err(err, "eoship_tq_maxsim_topk: NULL buffer");
  const size_t qbytes = (size_t)q * tq_tokens * tq->d * sizeof(float);
  const size_t ibytes = (size_t)q * kk * sizeof(int64_t);
  const size_t sbytes = (size_t)q * kk * sizeof(float);
  if (tq->ensure(&tq->io, &tq->io_bytes, qbytes + ibytes + sbytes + 256, err) != 0) return 1;
  char* base = static_cast<char*>(tq->io);
  float* dq = reinterpret_cast<float*>(base);
  int64_t* di = reinterpret_cast<int64_t*>(base + ((qbytes + 15) & ~(size_t)15));
  float* ds = reinterpret_cast<float*>(reinterpret_cast<char*>(di) + ibytes);
  hipError_t e = rt->copy_async(dq, queries, qbytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(queries)", e);
  if (maxsim_topk_impl(rt, tq, doc_len, dq, q, tq_tokens, k, di, ds, err) != 0) return 1;
  e = rt->copy_async(ids, di, ibytes, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = rt->copy_async(scores, ds, sbytes, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(results)", e);
  return rt->sync(err);
}

int eoship_tq_maxsim_scores(EosHipRuntime* rt, EosHipTQ* tq, int32_t doc_len, const float* queries,
                            int32_t q, int32_t tq_tokens, int64_t doc_begin, int64_t doc_count,
                            float* scores, char** err) {
  if (maxsim_check(rt, tq, doc_len, q, tq_tokens, "eoship_tq_maxsim_scores", err) != 0) return 1;
  const int64_t ndocs = tq->n / doc_len;
  if (doc_begin < 0 || doc_count < 0 || doc_begin + doc_count > ndocs)
    return set_err(err, "eoship_tq_maxsim_scores: documents [%lld, %lld) outside [0, %lld)",
                   (long long)doc_begin, (long long)(doc_begin + doc_count), (long long)ndocs);
  if (q == 0 || doc_count == 0) return 0;
  if (queries == nullptr || scores == nullptr) return set_err(err, "eoship_tq_maxsim_scores: NULL buffer");
  const size_t qbytes = (size_t)q * tq_tokens * tq->d * sizeof(float);
  if (tq->ensure(&tq->io, &tq->io_bytes, qbytes, err) != 0) return 1;
  float* dq = static_cast<float*>(tq->io);
  hipError_t e = rt->copy_async(dq, queries, qbytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(queries)", e);
  const int per = tq->maxsim_nqg();
  if (tq->ensure(reinterpret_cast<void**>(&tq->dense), &tq->dense_bytes,
                 (size_t)per * (size_t)doc_count * sizeof(float), err) != 0)
    return 1;
  for (int q0 = 0; q0 < q; q0 += per) {
    const int qp = std::min(per, q - q0);
    if (tq->maxsim_prepare(dq + (size_t)q0 * tq_tokens * tq->d, qp, tq_tokens, err) != 0 ||
        tq->maxsim_pass(0, qp, doc_len, doc_begin, doc_count, tq->dense, err) != 0)
      return 1;
    e = rt->copy_async(scores + (size_t)q0 * doc_count, tq->dense,
                       (size_t)qp * doc_count * sizeof(float), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(scores)", e);
    if (rt->sync(err) != 0) return 1;
  }
  return 0;
}

}  // extern "C"

// ------------------------------------------------------ parent aggregation

// A parent layout over a bound corpus: parent p owns the corpus vectors
// [off[p], off[p+1]) -- the children of topTurboQuantMultiVectorParentScores
// (runtime/retrieval_multivector_turboquant.go:746-758), grouped by parent.
struct EosHipTQParents {
  EosHipTQ* tq = nullptr;
  int64_t np = 0, live = 0;
  long long* off = nullptr;   // [np + 1]
  double* l1p = nullptr;      // [np] log1p(child count)
  long long* long_ids = nullptr;  // [nlong] parents of more than EOS_PARENT_SHORT children
  int64_t nlong = 0;
  float* pscores = nullptr;   // [per][np]
  size_t pscores_bytes = 0;
  void* io = nullptr;         // host-API staging
  size_t io_bytes = 0;
  ~EosHipTQParents() {
    void* ptrs[] = {off, l1p, long_ids, pscores, io};
    for (void* p : ptrs)
      if (p) hipFree(p);
  }
};

namespace {

// Whether a parent row's ranking is split. The merge of the chunks' best costs
// a launch and, at large k, a sort of k keys; one workgroup a row costs about
// 1 us per 1,000 parents. Whole calls, split against one workgroup a row:
// 8,320 parents, k = 50, 2 queries 36 / 36 us; 16,384 37 / 42, 64 queries
// 58 / 63; 40,000, 16 queries, k = 100 54 / 76, k = 1,000 131 / 99; 64 queries,
// k = 100 87 / 111. The second line passes through the sizes at which both cost
// the same: 16,000 parents at k = 300, 24,000 at 400, 41,000 at 600, 60,000 at
// 800, 76,000 at 1,000.
bool parents_split(int64_t np, int kk) { return np >= 16384 && np >= 84 * (int64_t)kk - 9600; }

// Queries per pass: the dense child-score block [per][n] stays under 4 GiB.
int parent_batch(const EosHipTQParents* P) {
  const int64_t by_mem = ((int64_t)1 << 32) / std::max<int64_t>(1, P->tq->n * 4);
  return (int)std::max<int64_t>(1, std::min<int64_t>(P->tq->batch_cap(), by_mem));
}

int parent_check(EosHipRuntime* rt, EosHipTQParents* P, int32_t q, int32_t top_n, double penalty,
                 const char* what, char** err) {
  if (rt == nullptr || P == nullptr) return set_err(err, "%s: NULL runtime or parents", what);
  if (P->tq->rt != rt) return set_err(err, "%s: parents were bound on another runtime", what);
  if (q < 0) return set_err(err, "%s: negative query count", what);
  if (top_n != 1 && top_n != 2 && top_n != 3 && top_n != 5)
    return set_err(err, "%s: aggregation must be max (1), top2-mean, top3-mean or top5-mean (got top_n %d)",
                   what, top_n);
  if (!(penalty >= 0.0) || std::isinf(penalty))
    return set_err(err, "%s: child-count-penalty must be non-negative and finite", what);
  return 0;
}

int parent_topk_impl(EosHipRuntime* rt, EosHipTQParents* P, const float* d_queries, int32_t q,
                     int32_t k, int32_t top_n, double penalty, int64_t* d_ids, float* d_scores,
                     int64_t* d_best, float* d_best_score, char** err) {
  EosHipTQ* tq = P->tq;
  const int64_t kk64 = (k <= 0 || (int64_t)k > P->live) ? P->live : k;
  if (q == 0 || kk64 == 0) return 0;
  if (kk64 > kSortCap)
    return set_err(err, "eoship_tq_parent_topk: k=%lld exceeds the device top-k limit of %d",
                   (long long)kk64, kSortCap);
  const int kk = (int)kk64;
  const int per = parent_batch(P);
  if (tq->ensure(reinterpret_cast<void**>(&P->pscores), &P->pscores_bytes,
                 (size_t)per * (size_t)P->np * sizeof(float), err) != 0)
    return 1;
  for (int q0 = 0; q0 < q; q0 += per) {
    const int qb = std::min(per, q - q0);
    if (tq->prepare(d_queries + (size_t)q0 * tq->d, qb, nullptr, err) != 0) return 1;
    if (tq->dense_scores(qb, 0, tq->n, false, err) != 0) return 1;
    TqParentArgs ag;
    memset(&ag, 0, sizeof(ag));
    ag.scores = tq->dense;
    ag.off = P->off;
    ag.l1p = P->l1p;
    ag.out = P->pscores;
    ag.np = P->np;
    ag.out_stride = P->np;
    ag.stride = tq->n;
    ag.penalty = penalty;
    ag.top_n = top_n;
    ag.qb = qb;
    // Short parents by a lane each, the others (listed at bind) by a wavefront.
    if (P->nlong < P->np &&
        rt->launch("eos_tq_parent_agg_short", dim3((unsigned)((P->np + 255) / 256), qb), dim3(256),
                   0, &ag, err, "tq_parent_agg") != 0)
      return 1;
    if (P->nlong > 0) {
      ag.np = P->nlong;
      ag.list = P->long_ids;
      if (rt->launch("eos_tq_parent_agg", dim3((unsigned)((P->nlong + 3) / 4), qb), dim3(256), 0,
                     &ag, err, "tq_parent_agg") != 0)
        return 1;
    }
    // The flat scan's candidate lists (kBatch x kCap keys) hold the chunks'.
    if (rank_rows(rt, P->pscores, qb, P->np, kk, d_ids + (size_t)q0 * kk, d_scores + (size_t)q0 * kk,
                  tq->cand, tq->cand_count, tq->status, "tq_parent_select", err,
                  parents_split(P->np, kk)) != 0)
      return 1;
    TqParentBestArgs bb;
    memset(&bb, 0, sizeof(bb));
    bb.scores = tq->dense;
    bb.off = P->off;
    bb.parents = reinterpret_cast<const long long*>(d_ids + (size_t)q0 * kk);
    bb.best_child = reinterpret_cast<long long*>(d_best + (size_t)q0 * kk);
    bb.best_score = d_best_score + (size_t)q0 * kk;
    bb.stride = tq->n;
    bb.kk = kk;
    bb.qb = qb;
    if (rt->launch("eos_tq_parent_best", dim3((unsigned)((kk + 3) / 4), qb), dim3(256), 0, &bb, err,
                   "tq_parent_best") != 0)
      return 1;
  }
  return 0;
}

}  // namespace

extern "C" {

int eoship_tq_parents_bind(EosHipRuntime* rt, EosHipTQ* tq, const int64_t* offsets,
                           int64_t nparents, EosHipTQParents** out, char** err) {
  const char* what = "eoship_tq_parents_bind";
  if (rt == nullptr || tq == nullptr || offsets == nullptr || out == nullptr)
    return set_err(err, "%s: NULL argument", what);
  *out = nullptr;
  if (tq->rt != rt) return set_err(err, "%s: corpus was bound on another runtime", what);
  if (tq->id_map != nullptr)
    return set_err(err, "%s: parents need their children in index order (corpus bound with id_rank)",
                   what);
  if (nparents <= 0 || nparents > ((int64_t)1 << 31))
    return set_err(err, "%s: parent count must be in 1..2^31 (got %lld)", what, (long long)nparents);
  if (offsets[0] != 0 || offsets[nparents] != tq->n)
    return set_err(err, "%s: offsets must start at 0 and end at the corpus size %lld", what,
                   (long long)tq->n);
  std::vector<double> l1p((size_t)nparents);
  std::vector<long long> longs;
  int64_t live = 0;
  for (int64_t p = 0; p < nparents; ++p) {
    const int64_t c = offsets[p + 1] - offsets[p];
    if (c < 0) return set_err(err, "%s: offsets decrease at parent %lld", what, (long long)p);
    live += c > 0 ? 1 : 0;
    if (c > EOS_PARENT_SHORT) longs.push_back((long long)p);
    l1p[(size_t)p] = std::log1p((double)c);
  }
  auto* P = new EosHipTQParents();
  P->tq = tq;
  P->np = nparents;
  P->live = live;
  const size_t ob = (size_t)(nparents + 1) * sizeof(long long), lb = (size_t)nparents * sizeof(double);
  hipError_t e = hipSuccess;
  if (rt->alloc(ob, reinterpret_cast<void**>(&P->off), err) ||
      rt->alloc(lb, reinterpret_cast<void**>(&P->l1p), err) ||
      rt->alloc(longs.size() * sizeof(long long), reinterpret_cast<void**>(&P->long_ids), err)) {
    delete P;
    return 1;
  }
  P->nlong = (int64_t)longs.size();
  e = rt->copy_sync(P->off, offsets, ob, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = rt->copy_sync(P->l1p, l1p.data(), lb, hipMemcpyHostToDevice);
  if (e == hipSuccess && !longs.empty())
    e = rt->copy_sync(P->long_ids, longs.data(), longs.size() * sizeof(long long), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    delete P;
    return hip_err(err, "hipMemcpy(parent offsets)", e);
  }
  *out = P;
  return 0;
}

int eoship_tq_parents_release(EosHipTQParents* parents, char** err) {
  (void)err;
  if (parents == nullptr) return 0;
  (void)parents->tq->rt->sync(nullptr);
  delete parents;
  return 0;
}

int eoship_tq_parent_topk_device(EosHipRuntime* rt, EosHipTQParents* parents,
                                 const float* d_queries, int32_t q, int32_t k, int32_t top_n,
                                 double child_count_penalty, int64_t* d_parent_ids,
                                 float* d_scores, int64_t* d_best_child, float* d_best_child_score,
                                 char** err) {
  const char* what = "eoship_tq_parent_topk_device";
  if (parent_check(rt, parents, q, top_n, child_count_penalty, what, err) != 0) return 1;
  if (q > 0 && (d_queries == nullptr || d_parent_ids == nullptr || d_scores == nullptr ||
                d_best_child == nullptr || d_best_child_score == nullptr))
    return set_err(err, "%s: NULL buffer", what);
  return parent_topk_impl(rt, parents, d_queries, q, k, top_n, child_count_penalty, d_parent_ids,
                          d_scores, d_best_child, d_best_child_score, err);
}

int eoship_tq_parent_topk(EosHipRuntime* rt, EosHipTQParents* parents, const float* queries,
                          int32_t q, int32_t k, int32_t top_n, double child_count_penalty,
                          int64_t* parent_ids, float* scores, int64_t* best_child,
                          float* best_child_score, char** err) {
  const char* what = "eoship_tq_parent_topk";
  if (parent_check(rt, parents, q, top_n, child_count_penalty, what, err) != 0) return 1;
  const int64_t kk = (k <= 0 || (int64_t)k > parents->live) ? parents->live : k;
  if (q == 0 || kk == 0) return 0;
  if (queries == nullptr || parent_ids == nullptr || scores == nullptr || best_child == nullptr ||
      best_child_score == nullptr)
    return set_err(err, "%s: NULL buffer", what);
  const int d = parents->tq->d;
  const size_t qbytes = ((size_t)q * d * sizeof(float) + 15) & ~(size_t)15;
  const size_t rows = (size_t)q * (size_t)kk;
  const size_t need = qbytes + rows * (8 + 4 + 8 + 4) + 64;
  if (parents->tq->ensure(&parents->io, &parents->io_bytes, need, err) != 0) return 1;
  char* base = static_cast<char*>(parents->io);
  float* dq = reinterpret_cast<float*>(base);
  int64_t* di = reinterpret_cast<int64_t*>(base + qbytes);
  int64_t* db = di + rows;
  float* ds = reinterpret_cast<float*>(db + rows);
  float* dbs = ds + rows;
  hipError_t e = rt->copy_async(dq, queries, (size_t)q * d * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(queries)", e);
  if (parent_topk_impl(rt, parents, dq, q, k, top_n, child_count_penalty, di, ds, db, dbs, err) != 0)
    return 1;
  e = rt->copy_async(parent_ids, di, rows * 8, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = rt->copy_async(scores, ds, rows * 4, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = rt->copy_async(best_child, db, rows * 8, hipMemcpyDeviceToHost);
  if (e == hipSuccess)
    e = rt->copy_async(best_child_score, dbs, rows * 4, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(results)", e);
  return rt->sync(err);
}

}  // extern "C"

// ----------------------------------------------------------------- encode

namespace {

// Rotated encodes on the matrix cores (see eos_tq_encode_split_*).
int encode_split(EosHipRuntime* rt, EosHipTQ* tq, const float* d_x, int64_t n, uint8_t* d_codes,
                 float* d_norms, char** err) {
  constexpr int kRows = 96;  // vectors per workgroup
  TqEncSplitArgs a;
  memset(&a, 0, sizeof(a));
  a.rot_r = tq->rot_r;
  a.rfrag = tq->rot_frag;
  a.d = tq->d;
  a.bits = tq->bits;
  a.row_bytes = tq->row_bytes;
  a.nchunk = tq->enc_chunks();
  a.jtiles = tq->enc_tiles();
  a.cb_scale = tq->cb_scale;
  a.delta2 = tq->enc_delta2;
  a.rmax = tq->rot_rmax;
  const bool vec = tq->d % 4 == 0 && (reinterpret_cast<uintptr_t>(d_x) & 15) == 0;
  a.words = tq->row_bytes % 4 == 0 && (reinterpret_cast<uintptr_t>(d_codes) & 3) == 0 ? 1 : 0;
  const int levels = 1 << tq->bits;
  for (int v = 0; v < levels; ++v) a.cb[v] = tq->codebook[v];
  // Distinct levels ascending, each with the first code that has it (ties go
  // to the lower code).
  std::vector<std::pair<int, int>> lv;
  for (int v = 0; v < levels; ++v) lv.emplace_back(a.cb[v], v);
  std::sort(lv.begin(), lv.end());
  for (const auto& l : lv) {
    if (a.m > 0 && a.lv[a.m - 1] == l.first) continue;
    a.lv[a.m] = l.first;
    a.li[a.m++] = l.second;
  }
  // The fewest workgroups side by side that 12 multiplying wavefronts (32
  // coordinates each) cover, and the smallest of 4, 8, 12 that then do: each
  // workgroup side by side splits the same vectors again (d = 384, 10^6
  // vectors: 12 wavefronts 1.35 ms, 2 x 8 1.88, 3 x 4 1.55; d = 768, 300,000:
  // 2 x 12 1.38 ms, 3 x 8 1.54), and wavefronts without coordinates idle
  // (d = 128: 4 wavefronts 0.29 ms, 8 0.43).
  a.jblocks = (a.jtiles + 11) / 12;
  const int per = (a.jtiles + a.jblocks - 1) / a.jblocks;
  const int nw = per <= 4 ? 4 : per <= 8 ? 8 : 12;
  char name[40];
  snprintf(name, sizeof(name), "eos_tq_encode_split_w%d%s", nw, vec ? "_v" : "");
  // At most 2^24 vectors per launch (grid size).
  const int64_t step = (int64_t)1 << 24;
  for (int64_t i0 = 0; i0 < n; i0 += step) {
    a.n = std::min(step, n - i0);
    a.x = d_x + (size_t)i0 * tq->d;
    a.codes = d_codes + (size_t)i0 * tq->row_bytes;
    a.norms = d_norms + i0;
    const int64_t vblocks = ((a.n + kRows - 1) / kRows + 7) / 8 * 8;
    if (rt->launch(name, dim3((unsigned)(vblocks * a.jblocks)), dim3(64 * (nw + 4)), 0, &a, err,
                   "tq_encode") != 0)
      return 1;
  }
  return 0;
}

int encode_impl(EosHipRuntime* rt, EosHipTQ* tq, const float* d_x, int64_t n, uint8_t* d_codes,
                float* d_norms, char** err) {
  if (n == 0) return 0;
  if (tq->rot_frag != nullptr) return encode_split(rt, tq, d_x, n, d_codes, d_norms, err);
  TqEncodeArgs a;
  memset(&a, 0, sizeof(a));
  a.rot_t = tq->rot_t;
  a.d = tq->d;
  a.bits = tq->bits;
  a.row_bytes = tq->row_bytes;
  a.cb_scale = tq->cb_scale;
  for (int v = 0; v < (1 << tq->bits); ++v) a.cb[v] = tq->codebook[v];
  const bool small = tq->d <= 512;
  const int per_wg = small ? 32 : 16;
  // At most 2^24 vectors per launch (grid size).
  const int64_t step = (int64_t)1 << 24;
  for (int64_t i0 = 0; i0 < n; i0 += step) {
    const int64_t cnt = std::min(step, n - i0);
    a.x = d_x + (size_t)i0 * tq->d;
    a.codes = d_codes + (size_t)i0 * tq->row_bytes;
    a.norms = d_norms + i0;
    a.n = cnt;
    if (rt->launch(small ? "eos_tq_encode_d512" : "eos_tq_encode_d1024",
                   dim3((unsigned)((cnt + per_wg - 1) / per_wg)), dim3(256), 0, &a, err,
                   "tq_encode") != 0)
      return 1;
  }
  return 0;
}

}  // namespace

extern "C" {

int eoship_tq_encode_device(EosHipRuntime* rt, EosHipTQ* tq, const float* d_x, int64_t n,
                            uint8_t* d_codes, float* d_norms, char** err) {
  if (rt == nullptr || tq == nullptr) return set_err(err, "eoship_tq_encode_device: NULL argument");
  if (tq->rt != rt) return set_err(err, "eoship_tq_encode_device: quantizer bound on another runtime");
  if (n < 0) return set_err(err, "eoship_tq_encode_device: negative vector count");
  if (n > 0 && (d_x == nullptr || d_codes == nullptr || d_norms == nullptr))
    return set_err(err, "eoship_tq_encode_device: NULL buffer");
  return encode_impl(rt, tq, d_x, n, d_codes, d_norms, err);
}

int eoship_tq_encode(EosHipRuntime* rt, EosHipTQ* tq, const float* x, int64_t n, uint8_t* codes,
                     float* norms, char** err) {
  if (rt == nullptr || tq == nullptr) return set_err(err, "eoship_tq_encode: NULL argument");
  if (tq->rt != rt) return set_err(err, "eoship_tq_encode: quantizer bound on another runtime");
  if (n < 0) return set_err(err, "eoship_tq_encode: negative vector count");
  if (n == 0) return 0;
  if (x == nullptr || codes == nullptr || norms == nullptr)
    return set_err(err, "eoship_tq_encode: NULL buffer");
  // Host rows go through the staging buffer in chunks of at most 2^18 vectors.
  const int64_t chunk = std::min<int64_t>(n, (int64_t)1 << 18);
  const size_t xb = ((size_t)chunk * tq->d * sizeof(float) + 255) & ~(size_t)255;
  const size_t cb = ((size_t)chunk * tq->row_bytes + 255) & ~(size_t)255;
  const size_t nb = (size_t)chunk * sizeof(float);
  if (tq->ensure(&tq->io, &tq->io_bytes, xb + cb + nb, err) != 0) return 1;
  char* base = static_cast<char*>(tq->io);
  float* dx = reinterpret_cast<float*>(base);
  uint8_t* dc = reinterpret_cast<uint8_t*>(base + xb);
  float* dn = reinterpret_cast<float*>(base + xb + cb);
  for (int64_t i0 = 0; i0 < n; i0 += chunk) {
    const int64_t cnt = std::min(chunk, n - i0);
    hipError_t e = rt->copy_async(dx, x + (size_t)i0 * tq->d, (size_t)cnt * tq->d * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(vectors)", e);
    if (encode_impl(rt, tq, dx, cnt, dc, dn, err) != 0) return 1;
    e = rt->copy_async(codes + (size_t)i0 * tq->row_bytes, dc, (size_t)cnt * tq->row_bytes, hipMemcpyDeviceToHost);
    if (e == hipSuccess)
      e = rt->copy_async(norms + i0, dn, (size_t)cnt * sizeof(float), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_err(err, "hipMemcpyAsync(codes)", e);
    if (rt->sync(err) != 0) return 1;
  }
  return 0;
}

}  // extern "C"

// ------------------------------------------------- two-stage retrieval (f16)

namespace eoship {

int tq_fp16_rerank_check(const Runtime* rt, const float* d_queries, int32_t q, int32_t d,
                         const uint16_t* d_rows, int64_t n, const int64_t* d_cand_ids,
                         const float* d_cand_scores, int32_t c, int64_t* d_ids, float* d_scores,
                         const char* what, char** err) {
  if (rt == nullptr) return set_err(err, "%s: NULL runtime", what);
  if (q < 0 || c < 0 || n < 0) return set_err(err, "%s: negative size", what);
  if (d < 1 || d > 4096) return set_err(err, "%s: dim must be in [1, 4096]", what);
  if (c > 4096)
    return set_err(err, "%s: at most 4096 candidates per query (got %d; the reference takes any overfetch)",
                   what, c);
  if (q > 65535) return set_err(err, "%s: at most 65535 queries per call", what);
  if (n >= ((int64_t)1 << 32) - 1)
    return set_err(err, "%s: corpus must hold fewer than 2^32 - 1 rows", what);
  if (q == 0 || c == 0) return 0;
  if (d_queries == nullptr || d_rows == nullptr || d_cand_ids == nullptr || d_cand_scores == nullptr ||
      d_ids == nullptr || d_scores == nullptr)
    return set_err(err, "%s: NULL buffer", what);
  return 0;
}

int tq_fp16_rerank_launch(Runtime* rt, const float* d_queries, int32_t q, int32_t d,
                          const uint16_t* d_rows, int64_t n, const int64_t* d_cand_ids,
                          const float* d_cand_scores, int32_t c, int32_t k, int32_t bit_width,
                          int32_t overfetch, const int64_t* d_id_rank, int64_t* d_ids,
                          float* d_scores, float* scratch, const char* what, char** err) {
  (void)what;
  TqRerankArgs a;
  memset(&a, 0, sizeof(a));
  a.queries = d_queries;
  a.rows = reinterpret_cast<const unsigned short*>(d_rows);
  a.cand_ids = reinterpret_cast<const long long*>(d_cand_ids);
  a.cand_scores = d_cand_scores;
  a.out_ids = reinterpret_cast<long long*>(d_ids);
  a.out_scores = d_scores;
  a.dots = scratch;
  a.n = n;
  a.d = d;
  a.c = c;
  a.kk = (k <= 0 || k > c) ? c : k;
  a.id_rank = reinterpret_cast<const long long*>(d_id_rank);
  a.vec = (d % 8 == 0 && (reinterpret_cast<uintptr_t>(d_rows) & 15) == 0) ? 1 : 0;
  // shouldApplyTurboQuantFP16RerankRescue (runtime/retrieval_turboquant.go:1664-1669).
  a.rescue = (bit_width == 4 && k == 100 && overfetch == 200 && c >= 120) ? 1 : 0;
  if (rt->launch("eos_tq_rr_dots", dim3((unsigned)((c + 63) / 64), (unsigned)q), dim3(64), 0, &a,
                 err, "tq_fp16_rerank_dots") != 0)
    return 1;
  return rt->launch("eos_tq_rr_sort", dim3((unsigned)q), dim3(256), 0, &a, err, "tq_fp16_rerank_sort");
}

// Shared checks of the dense and reconstruct reranks.
static int rerank_sizes_check(const Runtime* rt, const float* d_queries, int32_t q, int32_t d,
                              int64_t n, const int64_t* d_cand_ids, int32_t c, int64_t* d_ids,
                              float* d_scores, const char* what, char** err) {
  if (rt == nullptr) return set_err(err, "%s: NULL runtime", what);
  if (q < 0 || c < 0 || n < 0) return set_err(err, "%s: negative size", what);
  if (d < 1 || d > 4096) return set_err(err, "%s: dim must be in [1, 4096]", what);
  if (c > 4096)
    return set_err(err, "%s: at most 4096 candidates per query (got %d; the reference takes any overfetch)",
                   what, c);
  if (q > 65535) return set_err(err, "%s: at most 65535 queries per call", what);
  if (n >= ((int64_t)1 << 32) - 1)
    return set_err(err, "%s: corpus must hold fewer than 2^32 - 1 rows", what);
  if (q == 0 || c == 0) return 0;
  if (d_queries == nullptr || d_cand_ids == nullptr || d_ids == nullptr || d_scores == nullptr)
    return set_err(err, "%s: NULL buffer", what);
  return 0;
}

}  // namespace eoship

extern "C" {

int eoship_tq_dense_rerank_device(EosHipRuntime* rt, const float* d_queries, int32_t q, int32_t d,
                                  const float* d_rows, int64_t n, const int64_t* d_cand_ids,
                                  int32_t c, int32_t k, const int64_t* d_id_rank, int64_t* d_ids,
                                  float* d_scores, char** err) {
  const char* what = "eoship_tq_dense_rerank_device";
  if (eoship::rerank_sizes_check(rt, d_queries, q, d, n, d_cand_ids, c, d_ids, d_scores, what,
                                 err) != 0)
    return 1;
  if (q == 0 || c == 0) return 0;
  if (d_rows == nullptr) return set_err(err, "%s: NULL rows", what);
  void* ws = nullptr;
  if (rt->workspace((size_t)q * (size_t)c * sizeof(float), &ws, err) != 0) return 1;
  TqRerankArgs a;
  memset(&a, 0, sizeof(a));
  a.queries = d_queries;
  a.rows_f32 = d_rows;
  a.cand_ids = reinterpret_cast<const long long*>(d_cand_ids);
  a.out_ids = reinterpret_cast<long long*>(d_ids);
  a.out_scores = d_scores;
  a.dots = static_cast<float*>(ws);
  a.n = n;
  a.d = d;
  a.c = c;
  a.kk = (k <= 0 || k > c) ? c : k;
  a.id_rank = reinterpret_cast<const long long*>(d_id_rank);
  a.vec = (d % 4 == 0 && (reinterpret_cast<uintptr_t>(d_rows) & 15) == 0) ? 1 : 0;
  if (rt->launch("eos_tq_rr_dots_f32", dim3((unsigned)((c + 63) / 64), (unsigned)q), dim3(64), 0,
                 &a, err, "tq_dense_rerank_dots") != 0)
    return 1;
  return rt->launch("eos_tq_rr_sort", dim3((unsigned)q), dim3(256), 0, &a, err,
                    "tq_dense_rerank_sort");
}

int eoship_tq_reconstruct_rerank_device(EosHipRuntime* rt, const EosHipTQCodes* codes,
                                        const float* d_queries, int32_t q,
                                        const int64_t* d_cand_ids, int32_t c, int32_t k,
                                        const int64_t* d_id_rank, int64_t* d_ids,
                                        float* d_scores, char** err) {
  const char* what = "eoship_tq_reconstruct_rerank_device";
  if (codes == nullptr) return set_err(err, "%s: NULL codes", what);
  const int d = codes->dim, bits = codes->bits;
  if (bits != 1 && bits != 2 && bits != 3 && bits != 4 && bits != 8)
    return set_err(err, "%s: bits must be 1, 2, 3, 4 or 8 (got %d)", what, bits);
  if (d > 1024) return set_err(err, "%s: dim must be in [1, 1024] (got %d)", what, d);
  if (eoship::rerank_sizes_check(rt, d_queries, q, d, codes->n, d_cand_ids, c, d_ids, d_scores,
                                 what, err) != 0)
    return 1;
  if (q == 0 || c == 0) return 0;
  if (codes->codes == nullptr || codes->norms == nullptr || codes->codebook == nullptr)
    return set_err(err, "%s: NULL codes, norms or codebook", what);
  const bool ip = codes->signs != nullptr;
  if (ip && (codes->resnorms == nullptr || codes->qjl_t == nullptr))
    return set_err(err, "%s: an inner-product code set needs resnorms and qjl_t", what);
  if (!ip && (codes->resnorms != nullptr || codes->qjl_t != nullptr))
    return set_err(err, "%s: resnorms and qjl_t without signs", what);
  // Dequantized vectors [q][c][d] and the f32 scores share one workspace block.
  const size_t x_bytes = (size_t)q * (size_t)c * (size_t)d * sizeof(float);
  void* ws = nullptr;
  if (rt->workspace(x_bytes + (size_t)q * (size_t)c * sizeof(float), &ws, err) != 0) return 1;
  TqReconArgs r;
  memset(&r, 0, sizeof(r));
  r.rot_t = codes->rotation_t;
  r.codes = codes->codes;
  r.norms = codes->norms;
  r.codebook = codes->codebook;
  r.signs = codes->signs;
  r.resnorms = codes->resnorms;
  r.qjl_t = codes->qjl_t;
  r.cand_ids = reinterpret_cast<const long long*>(d_cand_ids);
  r.xhat = static_cast<float*>(ws);
  r.n = codes->n;
  r.d = d;
  r.c = c;
  r.bits = bits;
  r.row_bytes = (d * bits + 7) / 8;
  if (rt->launch("eos_tq_rr_dequant", dim3((unsigned)((c + 7) / 8), (unsigned)q), dim3(256), 0, &r,
                 err, "tq_reconstruct_dequant") != 0)
    return 1;
  TqRerankArgs a;
  memset(&a, 0, sizeof(a));
  a.queries = d_queries;
  a.rows_f32 = r.xhat;
  a.rows_by_pos = 1;
  a.cand_ids = r.cand_ids;
  a.out_ids = reinterpret_cast<long long*>(d_ids);
  a.out_scores = d_scores;
  a.dots = reinterpret_cast<float*>(static_cast<char*>(ws) + x_bytes);
  a.n = codes->n;
  a.d = d;
  a.c = c;
  a.kk = (k <= 0 || k > c) ? c : k;
  a.id_rank = reinterpret_cast<const long long*>(d_id_rank);
  a.vec = d % 4 == 0 ? 1 : 0;
  if (rt->launch("eos_tq_rr_dots_f32", dim3((unsigned)((c + 63) / 64), (unsigned)q), dim3(64), 0,
                 &a, err, "tq_reconstruct_dots") != 0)
    return 1;
  return rt->launch("eos_tq_rr_sort", dim3((unsigned)q), dim3(256), 0, &a, err,
                    "tq_reconstruct_sort");
}

// ------------------------------------------------------ inner-product layout

// Query preparation of the inner-product layout into qs / ys / alpha / beta:
// qr = R q and y = S qr as tiled f64 matrix-vector launches (eos_tq_ip_matvec),
// then one quantize workgroup per column (eos_tq_ip_quant); with `frag` the
// quantize also writes the scan's query fragments, ysum and the filter state
// of frag->ncols columns (qs / ys may then be NULL).
// qr, y: device scratch of q * d doubles each.
struct IpFragOut {
  int8_t* bfrag;
  int* ysum;
  float* tau;
  uint32_t* cand_count;
  int ks, nqg;
  float* lonorm;
  int* kq;
};
static int ip_prepare_launch(EosHipRuntime* rt, const TqIpArgs& a, int q, double* qr, double* y,
                             const IpFragOut* frag, char** err) {
  if (q <= 0) return 0;
  const dim3 grid((unsigned)((a.d + 31) / 32), (unsigned)((q + 7) / 8));
  TqIpMatArgs m1{a.rot_t, a.queries, nullptr, qr, q, a.d};
  TqIpMatArgs m2{a.qjl_t, nullptr, qr, y, q, a.d};
  TqIpQuantArgs qa;
  memset(&qa, 0, sizeof(qa));
  qa.qr = qr;
  qa.y = y;
  qa.qs = a.qs;
  qa.ys = a.ys;
  qa.alpha = a.alpha;
  qa.beta = a.beta;
  qa.q = q;
  qa.d = a.d;
  qa.qmax = a.qmax;
  qa.qmax2 = a.qmax2;
  qa.cb_scale = a.cb_scale;
  int ncols = q;
  if (frag != nullptr) {
    qa.bfrag = frag->bfrag;
    qa.ysum = frag->ysum;
    qa.tau = frag->tau;
    qa.cand_count = frag->cand_count;
    qa.ks = frag->ks;
    qa.nqg = frag->nqg;
    qa.lonorm = frag->lonorm;
    qa.kq = frag->kq;
    ncols = 32 * frag->nqg;
  }
  if (rt->launch("eos_tq_ip_matvec", grid, dim3(256), 0, &m1, err, "tq_ip_prepare") != 0 ||
      rt->launch("eos_tq_ip_matvec", grid, dim3(256), 0, &m2, err, "tq_ip_prepare") != 0)
    return 1;
  return rt->launch("eos_tq_ip_quant", dim3((unsigned)ncols), dim3(256), 0, &qa, err,
                    "tq_ip_prepare");
}

static int ip_spec_check(EosHipRuntime* rt, const EosHipTQIPSpec* spec, TqIpArgs* a,
                         const char* what, char** err) {
  if (rt == nullptr || spec == nullptr) return set_err(err, "%s: NULL argument", what);
  const int d = spec->dim, bits = spec->bits;
  if (d < 1 || d > 1024) return set_err(err, "%s: dim must be in [1, 1024]", what);
  if (bits != 1 && bits != 2 && bits != 3 && bits != 4)
    return set_err(err, "%s: MSE bits must be 1, 2, 3 or 4 (got %d)", what, bits);
  if (spec->codebook == nullptr || spec->qjl_t == nullptr)
    return set_err(err, "%s: NULL codebook or QJL matrix", what);
  if (!(spec->codebook_scale > 0.f) || std::isinf(spec->codebook_scale))
    return set_err(err, "%s: codebook_scale must be finite and > 0", what);
  memset(a, 0, sizeof(*a));
  const int levels = 1 << bits;
  int cmax = 0;
  for (int v = 0; v < levels; ++v) {
    a->cb[v] = spec->codebook[v];
    cmax = std::max(cmax, std::abs((int)spec->codebook[v]));
  }
  // The MSE query grid keeps |D_mse| < 2^31 as the flat scan's does; the QJL
  // grid |D_qjl| <= d * qmax2 < 2^31, and both stay within the int8 high /
  // low split (127 * 256 + 127) of the MFMA scan.
  const int64_t lim = cmax == 0 ? kQmaxLimit : (int64_t)2147483647 / ((int64_t)cmax * d) - 128;
  a->qmax = (int)std::min<int64_t>(kQmaxLimit, lim);
  a->qmax2 = (int)std::min<int64_t>(kQmaxLimit, (int64_t)2147483647 / d - 1);
  if (a->qmax < 1) return set_err(err, "%s: codebook too wide for dim %d", what, d);
  a->rot_t = spec->rotation_t;
  a->qjl_t = spec->qjl_t;
  a->d = d;
  a->bits = bits;
  a->row_bytes = (d * bits + 7) / 8;
  a->sign_bytes = (d + 7) / 8;
  a->cb_scale = spec->codebook_scale;
  return 0;
}

int eoship_tq_ip_encode_device(EosHipRuntime* rt, const EosHipTQIPSpec* spec, const float* d_x,
                               int64_t n, uint8_t* d_codes, uint8_t* d_signs, float* d_resnorms,
                               float* d_norms, char** err) {
  const char* what = "eoship_tq_ip_encode_device";
  TqIpArgs a;
  if (ip_spec_check(rt, spec, &a, what, err) != 0) return 1;
  if (n < 0) return set_err(err, "%s: negative n", what);
  if (n == 0) return 0;
  if (!d_x || !d_codes || !d_signs || !d_resnorms || !d_norms)
    return set_err(err, "%s: NULL buffer", what);
  a.x = d_x;
  a.codes = d_codes;
  a.signs = d_signs;
  a.resnorms = d_resnorms;
  a.norms = d_norms;
  a.n = n;
  // 128 coordinates per tile row of the kernel (TJ); 32 vectors per workgroup
  // while their residuals fit the LDS beside the stages (d <= 512), else 16.
  // At d <= 512, up to 16 vectors a CU, a workgroup's own latency is the call:
  // half the vectors and twice the load depth (us, 32 vectors / 16: d = 256
  // 53 / 35, d = 384 101 / 65, d = 512 170 / 104 at any n up to 4,096). From
  // 4,097 on the smaller workgroups share CUs (d = 384: 4,097 106 / 126, 8,192
  // 112 / 132, 65,536 805 / 962; where 32 vectors just begin a second round
  // they would win again, 8,193 206 / 185). Above d = 512 both take 16 vectors
  // and the deeper loads only cost registers (d = 768: 205 / 222).
  const int tj = (a.d + 127) / 128;
  const bool small = tj <= 4 && n <= 16 * (int64_t)rt->compute_units;
  const int per = tj <= 4 && !small ? 32 : 16;
  char name[32];
  snprintf(name, sizeof(name), "eos_tq_encode_ip_%c%d", small ? 's' : 't', tj);
  return rt->launch(name, dim3((unsigned)((n + per - 1) / per)), dim3(512), 0, &a, err,
                    "tq_encode_ip");
}

int eoship_tq_ip_scores_device(EosHipRuntime* rt, const EosHipTQIPSpec* spec,
                               const float* d_queries, int32_t q, const uint8_t* d_codes,
                               const uint8_t* d_signs, const float* d_resnorms,
                               const float* d_norms, int64_t n, float* d_scores, int32_t k,
                               int64_t* d_top_ids, float* d_top_scores, char** err) {
  const char* what = "eoship_tq_ip_scores_device";
  TqIpArgs a;
  if (ip_spec_check(rt, spec, &a, what, err) != 0) return 1;
  if (q < 0 || n < 0) return set_err(err, "%s: negative size", what);
  if (n >= ((int64_t)1 << 31)) return set_err(err, "%s: n must be below 2^31", what);
  if (k < 0 || k > 8192) return set_err(err, "%s: k must be in 0..8192", what);
  if (k > 0 && (d_top_ids == nullptr || d_top_scores == nullptr))
    return set_err(err, "%s: top-k outputs are NULL", what);
  if (q == 0 || n == 0) return 0;
  if (!d_queries || !d_codes || !d_signs || !d_resnorms || !d_norms || !d_scores)
    return set_err(err, "%s: NULL buffer", what);
  const size_t grid_bytes = (size_t)q * (size_t)a.d * sizeof(int);
  const size_t f64_bytes = (size_t)q * (size_t)a.d * sizeof(double);
  void* ws = nullptr;
  if (rt->workspace(2 * f64_bytes + 2 * grid_bytes + (size_t)q * 8, &ws, err) != 0) return 1;
  char* w = static_cast<char*>(ws);
  double* qr = reinterpret_cast<double*>(w);
  double* yv = reinterpret_cast<double*>(w + f64_bytes);
  w += 2 * f64_bytes;
  a.queries = d_queries;
  a.qs = reinterpret_cast<int*>(w);
  a.ys = reinterpret_cast<int*>(w + grid_bytes);
  a.alpha = reinterpret_cast<float*>(w + 2 * grid_bytes);
  a.beta = a.alpha + q;
  a.codes = const_cast<uint8_t*>(d_codes);
  a.signs = const_cast<uint8_t*>(d_signs);
  a.resnorms = const_cast<float*>(d_resnorms);
  a.norms = const_cast<float*>(d_norms);
  a.scores = d_scores;
  a.n = n;
  a.q = q;
  if (ip_prepare_launch(rt, a, q, qr, yv, nullptr, err) != 0 ||
      rt->launch("eos_tq_ip_scores", dim3((unsigned)((n + 255) / 256), (unsigned)((q + 7) / 8)),
                 dim3(256), 0, &a, err, "tq_ip_scores") != 0)
    return 1;
  if (k == 0) return 0;
  TqSelectArgs sel;
  memset(&sel, 0, sizeof(sel));
  sel.rows = d_scores;
  sel.ids = reinterpret_cast<long long*>(d_top_ids);
  sel.scores = d_top_scores;
  sel.n = n;
  sel.stride = n;
  sel.kk = (int64_t)k > n ? (int)n : k;
  sel.mode = 1;
  sel.nrows = q;
  return rt->launch("eos_tq_row_select", dim3((unsigned)q), dim3(1024), 0, &sel, err, "tq_ip_topk");
}

int eoship_f16_sidecar_device(EosHipRuntime* rt, const float* d_x, int64_t count, uint16_t* d_half,
                              char** err) {
  if (rt == nullptr) return set_err(err, "eoship_f16_sidecar_device: NULL runtime");
  if (count < 0) return set_err(err, "eoship_f16_sidecar_device: negative count");
  if (count == 0) return 0;
  if (d_x == nullptr || d_half == nullptr) return set_err(err, "eoship_f16_sidecar_device: NULL buffer");
  TqHalfArgs a;
  a.x = d_x;
  a.h = reinterpret_cast<unsigned short*>(d_half);
  a.count = count;
  const int64_t blocks = std::min<int64_t>((count + 1023) / 1024, 8192);
  return rt->launch("eos_tq_f16_sidecar", dim3((unsigned)blocks), dim3(256), 0, &a, err,
                    "f16_sidecar");
}

int eoship_tq_fp16_rerank_device(EosHipRuntime* rt, const float* d_queries, int32_t q, int32_t d,
                                 const uint16_t* d_rows, int64_t n, const int64_t* d_cand_ids,
                                 const float* d_cand_scores, int32_t c, int32_t k,
                                 int32_t bit_width, int32_t overfetch, const int64_t* d_id_rank,
                                 int64_t* d_ids, float* d_scores, char** err) {
  const char* what = "eoship_tq_fp16_rerank_device";
  if (eoship::tq_fp16_rerank_check(rt, d_queries, q, d, d_rows, n, d_cand_ids, d_cand_scores, c,
                                   d_ids, d_scores, what, err) != 0)
    return 1;
  if (q == 0 || c == 0) return 0;
  void* ws = nullptr;
  if (rt->workspace((size_t)q * (size_t)c * sizeof(float), &ws, err) != 0) return 1;
  return eoship::tq_fp16_rerank_launch(rt, d_queries, q, d, d_rows, n, d_cand_ids, d_cand_scores,
                                       c, k, bit_width, overfetch, d_id_rank, d_ids, d_scores,
                                       static_cast<float*>(ws), what, err);
}

}  // extern "C"

// ---------------------------------------- inner-product first stage (top-k)
//
// The promoted serving profile's first stage (turboquant_ip_b4_overfetch200_
// fp16_rerank, runtime/retrieval_turboquant.go:1500-1556): the top-k of the
// inner-product estimate over IPQuantized documents, as
// topTurboQuantRetrievalScoresWithStats computes it with InnerProductPrepared
// (:1853-1887). Per batch of <= 64 queries (32 when the dimension needs more
// than 12 K-steps): eos_tq_ip_matvec (R q, S R q) + eos_tq_ip_quant (their int
// grids as MFMA fragments), a sample scan of tile maxima and
// eos_tq_threshold, the filter scan (exact scores, keep >= tau),
// eos_tq_finalize, and the exact fallback gated on its flags (dense scan +
// eos_tq_row_select).
struct EosHipTQIP {
  EosHipRuntime* rt = nullptr;
  int d = 0, bits = 0, ks = 0, nqg = 0, qmax = 0, qmax2 = 0;
  int64_t n = 0, ntiles = 0;
  float cb_scale = 0.f;
  int cb[16] = {0};
  uint32_t lut0 = 0, lut1 = 0;
  const float* rot_t = nullptr;  // caller's device matrices
  const float* qjl_t = nullptr;
  int32_t* packed = nullptr;
  float* norms = nullptr;
  float* resnorms = nullptr;
  float* tile_cn = nullptr;  // [ntiles][4] code-norm bound per tile
  // per-batch scratch
  float* alpha = nullptr;
  float* beta = nullptr;
  float* lonorm = nullptr;  // [cols] bound filter constants
  int* kq = nullptr;
  int* ysum = nullptr;
  int8_t* bfrag = nullptr;
  float* tau = nullptr;
  unsigned long long* cand = nullptr;
  uint32_t* cand_count = nullptr;
  int* status = nullptr;
  float* samp = nullptr;
  float* dense = nullptr;
  size_t dense_bytes = 0;
  double* qr = nullptr;  // [cols][d] R q
  double* yv = nullptr;  // [cols][d] S R q

  int batch_cap() const { return 32 * nqg; }

  ~EosHipTQIP() {
    void* p[] = {packed, norms, resnorms, alpha, beta, ysum, bfrag, tau, cand, cand_count, status,
                 samp, dense, qr, yv, tile_cn, lonorm, kq};
    for (void* x : p)
      if (x) (void)hipFree(x);
  }

  // mode 3: the high-half bound filter (mode 1 of the _h kernel).
  int scan(int mode, int qb, int64_t tile_begin, int64_t tile_step, int64_t ntl, float* out,
           int64_t out_stride, const int* gate, char** err) {
    if (ntl <= 0) return 0;
    const bool hi = mode == 3;
    TqIpScanArgs s;
    memset(&s, 0, sizeof(s));
    s.packed = packed;
    s.norms = norms;
    s.resnorms = resnorms;
    s.bfrag = bfrag;
    s.alpha = alpha;
    s.beta = beta;
    s.ysum = ysum;
    s.tau = tau;
    s.cand = cand;
    s.cand_count = cand_count;
    s.out_scores = out;
    s.gate = gate;
    s.n = n;
    s.out_begin = 0;
    s.out_count = n;
    s.out_stride = out_stride;
    s.tile_begin = tile_begin;
    s.tile_step = tile_step;
    s.ntiles = (int)ntl;
    s.q = qb;
    s.cap = kCap;
    s.mode = hi ? 1 : mode;
    s.lut0 = lut0;
    s.lut1 = lut1;
    s.lonorm = lonorm;
    s.kq = kq;
    s.tile_cn = tile_cn;
    char name[48];
    snprintf(name, sizeof(name), "eos_tq_ipscan_k%d_g%d%s", ks, nqg, hi ? "_h" : "");
    static const char* const labels[4] = {"tq_ipscan_dense", "tq_ipscan_filter", "tq_ipscan_sample",
                                          "tq_ipscan_filter"};
    int64_t blocks = (ntl + 7) / 8;
    if (blocks > rt->compute_units) blocks = rt->compute_units;
    if (blocks < 1) blocks = 1;
    return rt->launch(name, dim3((unsigned)blocks), dim3(512), 0, &s, err, labels[mode]);
  }

  int prepare(const float* d_queries, int qb, char** err) {
    TqIpArgs a;
    memset(&a, 0, sizeof(a));
    a.queries = d_queries;
    a.rot_t = rot_t;
    a.qjl_t = qjl_t;
    a.alpha = alpha;
    a.beta = beta;
    a.d = d;
    a.q = qb;
    a.qmax = qmax;
    a.qmax2 = qmax2;
    a.cb_scale = cb_scale;
    const IpFragOut f{bfrag, ysum, tau, cand_count, ks, nqg, lonorm, kq};
    return ip_prepare_launch(rt, a, qb, qr, yv, &f, err);
  }

  int topk_batch(const float* d_queries, int qb, int kk, int64_t* d_ids, float* d_scores,
                 char** err) {
    if (prepare(d_queries, qb, err) != 0) return 1;
    if (n > kCap) {
      const int64_t stride =
          std::max<int64_t>(kSampleStride, (ntiles + kMaxSampleTiles - 1) / kMaxSampleTiles);
      const int64_t ns = (ntiles + stride - 1) / stride;
      int64_t nsv = 0;
      for (int64_t j = 0; j < ns; ++j) nsv += std::min<int64_t>(kTile, n - j * stride * kTile);
      const double target = std::min<double>(kKeepFactor * kk, kCap / 4.0);
      int64_t r = (int64_t)std::ceil(target * (double)nsv / (double)n);
      r = std::max<int64_t>(1, std::min<int64_t>(r, ns));
      if (scan(2, qb, 0, stride, ns, samp, ns, nullptr, err) != 0) return 1;
      TqSelectArgs sel;
      memset(&sel, 0, sizeof(sel));
      sel.rows = samp;
      sel.tau = tau;
      sel.n = ns;
      sel.stride = ns;
      sel.kk = (int)r;
      sel.nrows = qb;
      if (rt->launch("eos_tq_threshold", dim3(qb), dim3(256), 0, &sel, err, "tq_ip_threshold") != 0)
        return 1;
    }
    if (n > kCap) {
      // High-half bound filter (ids), then their exact scores.
      if (scan(3, qb, 0, 1, ntiles, nullptr, 0, nullptr, err) != 0) return 1;
      TqIpRescoreArgs rs;
      memset(&rs, 0, sizeof(rs));
      rs.packed = packed;
      rs.norms = norms;
      rs.resnorms = resnorms;
      rs.bfrag = bfrag;
      rs.nqg = nqg;
      rs.alpha = alpha;
      rs.beta = beta;
      rs.ysum = ysum;
      rs.tau = tau;
      rs.cand = cand;
      rs.cand_count = cand_count;
      rs.n = n;
      rs.q = qb;
      rs.d = d;
      rs.ks = ks;
      rs.cap = kCap;
      rs.lut0 = lut0;
      rs.lut1 = lut1;
      if (rt->launch("eos_tq_ip_rescore", dim3((unsigned)qb, 2 * kRescoreBlocks), dim3(256), 0, &rs,
                     err, "tq_ip_rescore") != 0)
        return 1;
    } else if (scan(1, qb, 0, 1, ntiles, nullptr, 0, nullptr, err) != 0) {
      return 1;
    }
    TqFinalizeArgs f;
    memset(&f, 0, sizeof(f));
    f.cand = cand;
    f.cand_count = cand_count;
    f.ids = reinterpret_cast<long long*>(d_ids);
    f.scores = d_scores;
    f.status = status;
    f.cap = kCap;
    f.kk = kk;
    f.q = qb;
    if (rt->launch(finalize_kernel(f.kk), dim3(qb), dim3(256), 0, &f, err, "tq_ip_finalize") != 0)
      return 1;
    // Exact fallback, gated on the device by the finalize flags.
    const size_t need = (size_t)qb * (size_t)n * sizeof(float);
    if (dense_bytes < need) {
      if (dense != nullptr) {
        if (rt->sync(err) != 0) return 1;
        (void)hipFree(dense);
      }
      dense = nullptr;
      dense_bytes = 0;
      if (rt->alloc(need, reinterpret_cast<void**>(&dense), err) != 0) return 1;
      dense_bytes = need;
    }
    if (scan(0, qb, 0, 1, ntiles, dense, n, status, err) != 0) return 1;
    TqSelectArgs sel;
    memset(&sel, 0, sizeof(sel));
    sel.rows = dense;
    sel.status = status;
    sel.ids = reinterpret_cast<long long*>(d_ids);
    sel.scores = d_scores;
    sel.n = n;
    sel.stride = n;
    sel.kk = kk;
    sel.mode = 1;
    sel.nrows = qb;
    return rt->launch("eos_tq_row_select", dim3(qb), dim3(1024), 0, &sel, err,
                      "tq_ip_fallback_select");
  }
};

extern "C" {

int eoship_tq_ip_bind_corpus(EosHipRuntime* rt, const EosHipTQIPSpec* spec,
                             const uint8_t* d_codes, const uint8_t* d_signs,
                             const float* d_resnorms, const float* d_norms, int64_t n,
                             const EosHipTQBindOptions* opts, EosHipTQIP** out, char** err) {
  const char* what = "eoship_tq_ip_bind_corpus";
  if (out == nullptr) return set_err(err, "%s: NULL output", what);
  *out = nullptr;
  TqIpArgs a;
  if (ip_spec_check(rt, spec, &a, what, err) != 0) return 1;
  if (spec->bits > 3)
    return set_err(err, "%s: the scan takes MSE codes of 1, 2 or 3 bits (bit widths 2..4; got %d)",
                   what, spec->bits);
  if (n < 1 || n >= ((int64_t)1 << 31) - 64)
    return set_err(err, "%s: n must be in [1, 2^31 - 64)", what);
  if (!d_codes || !d_signs || !d_resnorms || !d_norms) return set_err(err, "%s: NULL buffer", what);
  if (opts != nullptr && opts->id_rank != nullptr)
    return set_err(err, "%s: id_rank is not supported for the inner-product layout", what);
  int ks = 0;
  for (int k : {4, 8, 12, 16, 24, 32})
    if (ks == 0 && k * 32 >= spec->dim) ks = k;
  // Norm policy of validateEosQuantizedVectorNorm (runtime/
  // turboquant_quantized_vector.go:25-49), as the MSE bind applies it.
  {
    std::vector<float> hn((size_t)n);
    hipError_t e = rt->copy_sync(hn.data(), d_norms, (size_t)n * 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_err(err, "hipMemcpy(norms)", e);
    for (int64_t i = 0; i < n; ++i) {
      const float v = hn[(size_t)i];
      if (!(v >= 0.f) || std::isinf(v))
        return set_err(err, "%s: vector %lld has an invalid norm %g", what, (long long)i, (double)v);
      if (v == 0.f && (opts == nullptr || opts->zero_vector_allowed == nullptr ||
                       opts->zero_vector_allowed[i] == 0))
        return set_err(err, "%s: vector %lld has Norm 0 and is not marked as a zero vector", what,
                       (long long)i);
    }
  }
  auto* ip = new EosHipTQIP();
  ip->rt = rt;
  ip->d = spec->dim;
  ip->bits = spec->bits;
  ip->ks = ks;
  ip->nqg = ks <= 12 ? 2 : 1;
  ip->qmax = a.qmax;
  ip->qmax2 = a.qmax2;
  ip->n = n;
  ip->ntiles = (n + kTile - 1) / kTile;
  ip->cb_scale = spec->codebook_scale;
  ip->rot_t = spec->rotation_t;
  ip->qjl_t = spec->qjl_t;
  uint8_t t8[8] = {0};
  for (int v = 0; v < (1 << spec->bits); ++v) {
    ip->cb[v] = spec->codebook[v];
    t8[v] = (uint8_t)spec->codebook[v];
  }
  ip->lut0 = t8[0] | (t8[1] << 8) | (t8[2] << 16) | ((uint32_t)t8[3] << 24);
  ip->lut1 = t8[4] | (t8[5] << 8) | (t8[6] << 16) | ((uint32_t)t8[7] << 24);
  const int cols = 32 * ip->nqg;
  const int64_t samp_tiles =
      std::min<int64_t>((ip->ntiles + kSampleStride - 1) / kSampleStride, kMaxSampleTiles);
  auto fail = [&]() {
    delete ip;
    return 1;
  };
  if (rt->alloc((size_t)ip->ntiles * (ks / 2) * 64 * 16, reinterpret_cast<void**>(&ip->packed), err) ||
      rt->alloc((size_t)ip->ntiles * kTile * 4, reinterpret_cast<void**>(&ip->norms), err) ||
      rt->alloc((size_t)ip->ntiles * kTile * 4, reinterpret_cast<void**>(&ip->resnorms), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->alpha), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->beta), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->ysum), err) ||
      rt->alloc((size_t)ks * 4 * ip->nqg * 64 * 16, reinterpret_cast<void**>(&ip->bfrag), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->tau), err) ||
      rt->alloc((size_t)cols * kCap * 8, reinterpret_cast<void**>(&ip->cand), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->cand_count), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->status), err) ||
      rt->alloc((size_t)cols * std::max<int64_t>(samp_tiles, 1) * 4,
                reinterpret_cast<void**>(&ip->samp), err) ||
      rt->alloc((size_t)cols * ip->d * 8, reinterpret_cast<void**>(&ip->qr), err) ||
      rt->alloc((size_t)cols * ip->d * 8, reinterpret_cast<void**>(&ip->yv), err) ||
      rt->alloc((size_t)ip->ntiles * 16, reinterpret_cast<void**>(&ip->tile_cn), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->lonorm), err) ||
      rt->alloc((size_t)cols * 4, reinterpret_cast<void**>(&ip->kq), err))
    return fail();
  TqIpTileNormArgs tn;
  memset(&tn, 0, sizeof(tn));
  tn.codes = d_codes;
  tn.tile_cn = ip->tile_cn;
  tn.n = n;
  tn.d = ip->d;
  tn.bits = ip->bits;
  tn.row_bytes = a.row_bytes;
  for (int v = 0; v < (1 << spec->bits); ++v) tn.cb[v] = spec->codebook[v];
  if (rt->launch("eos_tq_ip_tile_cnorm", dim3((unsigned)((n + 255) / 256)), dim3(256), 0, &tn, err,
                 "tq_ip_pack") != 0)
    return fail();
  TqIpPackArgs p;
  memset(&p, 0, sizeof(p));
  p.codes = d_codes;
  p.signs = d_signs;
  p.norms = d_norms;
  p.resnorms = d_resnorms;
  p.packed = ip->packed;
  p.norms_out = ip->norms;
  p.resnorms_out = ip->resnorms;
  p.n = n;
  p.ntiles = ip->ntiles;
  p.d = ip->d;
  p.ks = ks;
  p.bits = ip->bits;
  p.row_bytes = a.row_bytes;
  p.sign_bytes = a.sign_bytes;
  const int64_t threads = ip->ntiles * (ks / 2) * 64;
  if (rt->launch("eos_tq_ip_pack", dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, &p, err,
                 "tq_ip_pack") != 0 ||
      rt->sync(err) != 0)
    return fail();
  *out = ip;
  return 0;
}

int eoship_tq_ip_topk_device(EosHipRuntime* rt, EosHipTQIP* ip, const float* d_queries,
                             int32_t q, int32_t k, int64_t* d_ids, float* d_scores, char** err) {
  const char* what = "eoship_tq_ip_topk_device";
  if (rt == nullptr || ip == nullptr) return set_err(err, "%s: NULL runtime or corpus", what);
  if (ip->rt != rt) return set_err(err, "%s: corpus was bound on another runtime", what);
  if (q < 0) return set_err(err, "%s: negative query count", what);
  const int64_t kk64 = (k <= 0 || (int64_t)k > ip->n) ? ip->n : k;
  if (q == 0) return 0;
  if (kk64 > kSortCap)
    return set_err(err, "%s: k=%lld exceeds the device top-k limit of %d", what, (long long)kk64,
                   kSortCap);
  if (d_queries == nullptr || d_ids == nullptr || d_scores == nullptr)
    return set_err(err, "%s: NULL buffer", what);
  const int kk = (int)kk64;
  const int cap = ip->batch_cap();
  for (int q0 = 0; q0 < q; q0 += cap) {
    const int qb = std::min(cap, q - q0);
    if (ip->topk_batch(d_queries + (size_t)q0 * ip->d, qb, kk, d_ids + (size_t)q0 * kk,
                       d_scores + (size_t)q0 * kk, err) != 0)
      return 1;
  }
  return 0;
}

int eoship_tq_ip_release(EosHipTQIP* ip, char** err) {
  (void)err;
  if (ip == nullptr) return 0;
  (void)ip->rt->sync(nullptr);
  delete ip;
  return 0;
}

}  // extern "C"
