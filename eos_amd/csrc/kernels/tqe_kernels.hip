// TurboQuant corpus encoders on gfx950: f32 vectors -> codes and norms, with
// the rotation (and the residual sketch) on the matrix cores.
//
// The contract is the f64 one of eos_tq_encode_* (tq_kernels.hip): u_j one
// fma chain over k, norm from the f64 chain of x^2, code_j the first level
// nearest u_j. eos_tq_encode_split reaches the same codes and norms from
// bounded approximations and decides in f64 only what the bound leaves open.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tq_args.h"

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef double v4d __attribute__((ext_vector_type(4)));

#define EOS_DEV __device__ __forceinline__

namespace {

EOS_DEV uint32_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
EOS_DEV float bf16_val(uint32_t b) { return __uint_as_float(b << 16); }

// Barrier for LDS data only: global loads in flight stay in flight.
EOS_DEV void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace

// R (row-major) as the split product's first operand: per 32 coordinates jt
// and 32-wide K chunk, [K step of 16][high, low][lane][8 bf16], lane l holding
// row 32 jt + l % 32 and K values 16 step + 8 (l / 32) .. + 7; zero past d.
// high = bf16(R), low = bf16(R - high). One thread per 8 values.
extern "C" __global__ __launch_bounds__(256) void eos_tq_rot_frag(TqRotFragArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.jtiles * a.nchunk * 2 * 64) return;
  const int lane = i & 63, ks = (i >> 6) & 1, jc = i >> 7;
  const int c = jc % a.nchunk, jt = jc / a.nchunk;
  const int j = 32 * jt + (lane & 31), k0 = 32 * c + 16 * ks + 8 * (lane >> 5);
  uint32_t h[8], lo[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = (j < a.d && k0 + e < a.d) ? a.rot_r[(size_t)j * a.d + k0 + e] : 0.0f;
    h[e] = bf16_bits(v);
    lo[e] = bf16_bits(v - bf16_val(h[e]));
  }
  v4i* out = reinterpret_cast<v4i*>(a.frag) + (size_t)(jc * 2 + ks) * 128 + lane;
  v4i hv, lv;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    hv[p] = (int)(h[2 * p] | (h[2 * p + 1] << 16));
    lv[p] = (int)(lo[2 * p] | (lo[2 * p + 1] << 16));
  }
  out[0] = hv;
  out[64] = lv;
}

// R^T, the layout of the f64 chains and of query preparation.
extern "C" __global__ __launch_bounds__(256) void eos_tq_rot_transpose(TqRotFragArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < a.d * a.d) a.rot_t[i] = a.rot_r[(size_t)(i % a.d) * a.d + i / a.d];
}

// Squared norms of R's rows and of what the split leaves of them, for its error
// bound: out[0..2][j] = sum over k of R^2, of low^2 and of (R - high - low)^2.
// One wavefront per row.
extern "C" __global__ __launch_bounds__(256) void eos_tq_rot_rows(TqRotFragArgs a) {
  const int lane = threadIdx.x & 63, j = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (j >= a.d) return;
  double t[3] = {0.0, 0.0, 0.0};
  for (int k = lane; k < a.d; k += 64) {
    const float v = a.rot_r[(size_t)j * a.d + k];
    const float rest = v - bf16_val(bf16_bits(v));
    const float low = bf16_val(bf16_bits(rest)), left = rest - low;
    t[0] = fma((double)v, (double)v, t[0]);
    t[1] = fma((double)low, (double)low, t[1]);
    t[2] = fma((double)left, (double)left, t[2]);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) t[i] += __shfl_xor(t[i], o);
    if (lane == 0) a.sums[(size_t)i * a.d + j] = t[i];
  }
}

namespace {

constexpr int kSplitRows = 96;     // vectors per workgroup
constexpr int kSplitItems = 1024;  // undecided (vector, coordinate) pairs listed per workgroup
constexpr int kSplitStage = 4;     // staging wavefronts

// Workgroup: 96 vectors x 32 NW coordinates, wavefront w < NW the coordinates
// [32 w, + 32). K advances in chunks of 32 through two LDS stages; each staged
// f32 value becomes a bf16 pair high + low, and
//   u~ = sum over chunks of (Rh xl + Rl xh + Rh xh)
// on bf16 MFMA, every chunk into a fresh accumulator that is then added in
// f32. The host's bound E on |u~ - u| / |x| (prepare_rotation) covers the split,
// the 32 large products of a chunk summed in f32 in any order and the sum over
// the chunks. In half steps of the integer level grid, w = 2 u~ / (nrm s_c),
// the decision points are whole numbers (sums of neighbouring levels): a
// 512-entry table indexed by the nearest whole number gives the codes on its
// two sides and whether it is a decision point. Values closer to one than
// delta2 = 2 E / s_c (+ 1e-4 for the rounding of w) go to a list and are
// decided in f64: first from a sum in another order with its own bound, then,
// if that is not enough (exact ties), by the contract's fma chain, a thread
// each. The list holds about 1 of 600 coordinates at d = 384, 4 bits. When it
// overflows (sparse vectors under a rotation of few nonzeros: every zero is a
// tie of a symmetric codebook) the tile is decided on the f64 matrix cores:
// 20,000 x 384 under a signed permutation, half of the values zero, 218 us
// (f64 VALU chains for every vector 678; each pair by 16 lanes and then one
// 22,748), a hundredth of them zero, a list of ties, 107 (686; 434).
// The norm's f64 sum is taken in another order too: it is kept when the f32
// norms of its two error bounds agree, else recomputed as the chain.
// A vector of norm 0 has u = 0 and every distance 0, one of infinite or NaN
// norm no finite distance: both take code 0. Norms outside [2^-90, 2^100]
// leave every coordinate to the list (bf16 over- and underflow).
//
// Bound: 10^6 x 384, 4 bits: 1.35-1.43 ms (the f64 kernel 27.3 ms, 14 % of
// the f64 rate), of which the chunk loop takes about 0.83 ms (0.88 PFLOP of
// bf16 products, 1.06 PFLOP/s), the listed pairs 0.14 ms and the start, norms,
// decisions and stores of a workgroup the rest; the vectors read at 1.2 TB/s.
// 96 rows keep R's fragments (590 KB per workgroup from L2) at 9 MFMAs a KB
// within the 128 registers of four wavefronts per SIMD. Workgroups that stay
// for many tiles, with the list left to the staging wavefronts, measured
// slower (1.58 ms: those four then pace the chunks), as did splitting by the
// multiplying wavefronts themselves (1.44).
//
// Wavefronts [0, NW) multiply and decide; the other four stage: while a chunk
// is multiplied out of one LDS stage they split the next into the other, with
// the two after it in flight. One barrier per chunk, at which both sides meet;
// then all wavefronts decide the listed pairs and write the codes.
template <int NW, bool VEC>
struct EncodeSplit {
  static constexpr int PT = 64 * kSplitStage;   // staging threads
  static constexpr int NT = 64 * NW + PT;
  static constexpr int BM = kSplitRows, RT = BM / 32;
  static constexpr int U = BM * 8 / PT;         // 16-byte loads per staging thread per chunk
  static_assert(BM * 8 % PT == 0, "staging split");
  static constexpr int CST = NW * 16 + 4;       // code bytes per vector (4 bits), padded
  struct Lds {
    uint32_t xs[2][2][BM * 16];
    uint8_t cbuf[BM * CST];
    double s64[BM];
    float inv2[BM], dlim[BM];
    uint32_t items[kSplitItems];
    uint32_t nitems, nties;
    uint16_t lut[512];
  };
  const TqEncSplitArgs& a;
  Lds& s;
  // The tile: nv vectors from v0 on, 32-coordinate tiles from jt0 on.
  long long v0;
  int nv, jt0;

  EOS_DEV void multiply(int wave, int lane) {
    const int g = lane >> 5, l32 = lane & 31, d = a.d;
    const bool active = jt0 + wave < a.jtiles;
    const v4i* src = reinterpret_cast<const v4i*>(a.rfrag) +
                     (size_t)min(jt0 + wave, a.jtiles - 1) * a.nchunk * 256 + lane;
    auto load_r = [&](v4i (&rf)[4], int c) {
#pragma unroll
      for (int i = 0; i < 4; ++i) rf[i] = src[(size_t)c * 256 + 64 * i];
    };
    v16f tot[RT];
    auto compute = [&](int st, const v4i (&rf)[4]) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        // The cross products first: the accumulator is small while they add.
        v16f acc = v16f{0};
        v8bf bh[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const int o = (32 * rt + l32) * 16 + ((2 * ks + g) ^ ((l32 >> 2) & 3)) * 4;
          bh[ks] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(&s.xs[st][0][o]));
          const v8bf bl = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(&s.xs[st][1][o]));
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, rf[2 * ks]), bl, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, rf[2 * ks + 1]), bh[ks], acc, 0, 0, 0);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, rf[2 * ks]), bh[ks], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) tot[rt][i] += acc[i];
      }
    };
    v4i rfa[4], rfb[4];
    load_r(rfa, 0);
    // The decision table: cell c = nearest whole number of w, [-256, 255].
    for (int i = 64 * wave + lane; i < 512; i += 64 * NW) {
      const int c = i - 256;
      int below = 0, upto = 0;
      for (int l = 0; l + 1 < a.m; ++l) {
        const int p = a.lv[l] + a.lv[l + 1];
        below += p < c ? 1 : 0;
        upto += p <= c ? 1 : 0;
      }
      s.lut[i] = (uint16_t)(a.li[below] | (a.li[upto] << 4) | (upto != below ? 0x1000 : 0));
    }
    if (wave == 0 && lane == 0) s.nitems = s.nties = 0u;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) tot[rt] = v16f{0};
    lds_barrier();
    for (int c = 0; c < a.nchunk; c += 2) {
      load_r(rfb, c + 1);
      if (active) compute(0, rfa);
      lds_barrier();
      load_r(rfa, min(c + 2, a.nchunk - 1));
      if (active) compute(1, rfb);
      lds_barrier();
    }
    // Codes of the wavefront's 32 coordinates: element 4 q + e of a lane
    // is coordinate 8 q + 4 g + e of vector 32 rt + l32.
    if (active) {
      const int left = d - 32 * (jt0 + wave);  // coordinates from the wavefront's first
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int v = 32 * rt + l32;
        const float iv = s.inv2[v], dl = s.dlim[v];
        const uint32_t keep = dl < -1.0f ? 0u : 0xffffu;
        const uint32_t force = dl > 1.0f ? 0xf000u : 0u;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t pk = 0, fl = force;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // c = w to the nearest whole number, through the low mantissa
            // bits of w + 1.5 * 2^23, clamped to the table; r = w - c.
            constexpr float kM = 12582912.0f;
            const float x = tot[rt][4 * q + e];
            const float f = __builtin_amdgcn_fmed3f(__builtin_fmaf(x, iv, kM), kM - 256.0f, kM + 255.0f);
            const float r = __builtin_fmaf(x, iv, kM - f);
            const uint32_t ent = s.lut[__float_as_uint(f) - (0x4b400000u - 256u)];
            pk |= ((ent >> (r > 0.0f ? 4 : 0)) & 15u) << (e * a.bits);
            fl |= (fabsf(r) > dl ? 0u : ent) << e;
          }
          pk &= keep;
          fl &= 0xf000u;
          const int valid = left - (8 * q + 4 * g);
          if (left < 32 && valid < 4) {
            const int m = valid < 0 ? 0 : valid;
            pk &= (1u << (m * a.bits)) - 1u;
            fl &= ((1u << m) - 1u) << 12;
          }
          if (fl != 0u) {
#pragma unroll 1
            for (fl >>= 12; fl != 0u; fl &= fl - 1u) {
              const uint32_t pos = atomicAdd(&s.nitems, 1u);
              if (pos < (uint32_t)kSplitItems)
                s.items[pos] =
                    (uint32_t)v << 16 | (uint32_t)(32 * wave + 8 * q + 4 * g + (__ffs(fl) - 1));
            }
          }
          if (a.bits == 4)
            *reinterpret_cast<uint16_t*>(&s.cbuf[v * CST + wave * 16 + 4 * q + 2 * g]) = (uint16_t)pk;
          else
            s.cbuf[v * CST + wave * 8 + 2 * q + g] = (uint8_t)pk;
        }
      }
    }
  }

  EOS_DEV void put_code(int v, int jl, int code) {
    const int bit = jl * a.bits;
    const int off = v * CST + (bit >> 3), sh = (off & 3) * 8 + (bit & 7);
    uint32_t* word = reinterpret_cast<uint32_t*>(&s.cbuf[off & ~3]);
    atomicAnd(word, ~(((1u << a.bits) - 1u) << sh));
    atomicOr(word, (uint32_t)code << sh);
  }

  // The contract's decisions for N values u of a vector of norm ne.
  template <int N>
  EOS_DEV void nearest(const double (&u)[N], double ne, int (&code)[N]) {
    double bd[N];
#pragma unroll 1
    for (int l = 0; l < (1 << a.bits); ++l) {
      const double nc = ne * ((double)a.cb_scale * (double)a.cb[l]);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double dv = fabs(u[i] - nc);
        if (l == 0 || dv < bd[i]) {
          bd[i] = dv;
          code[i] = l;
        }
      }
    }
  }

  // Pair i of the list by 16 lanes: every lane's 16-byte pieces of the two
  // rows are requested six at a time. Pairs that this leaves open go to the
  // ties (in xs, which nothing reads any more).
  EOS_DEV void decide(int i, int sub) {
    const int d = a.d;
    const uint32_t item = s.items[i];
    const int v = (int)(item >> 16), jl = (int)(item & 0xffffu);
    if (s.dlim[v] < -1.0f) return;
    const float* xv = a.x + (size_t)(v0 + v) * d;
    const float* rj = a.rot_r + (size_t)(32 * jt0 + jl) * d;
    double u = 0.0;
    if constexpr (VEC) {
      for (int k0 = 4 * sub; k0 < d; k0 += 384) {
        float4 xk[6], rk[6];
#pragma unroll
        for (int p = 0; p < 6; ++p) {
          const int k = min(k0 + 64 * p, d - 4);
          xk[p] = *reinterpret_cast<const float4*>(xv + k);
          rk[p] = *reinterpret_cast<const float4*>(rj + k);
        }
#pragma unroll
        for (int p = 0; p < 6; ++p) {
          double w = (double)rk[p].x * (double)xk[p].x;
          w = fma((double)rk[p].y, (double)xk[p].y, w);
          w = fma((double)rk[p].z, (double)xk[p].z, w);
          w = fma((double)rk[p].w, (double)xk[p].w, w);
          u += k0 + 64 * p < d ? w : 0.0;
        }
      }
    } else {
      for (int k0 = sub; k0 < d; k0 += 192) {
        float xk[12], rk[12];
#pragma unroll
        for (int p = 0; p < 12; ++p) {
          const int k = min(k0 + 16 * p, d - 1);
          xk[p] = xv[k];
          rk[p] = rj[k];
        }
#pragma unroll
        for (int p = 0; p < 12; ++p)
          u = fma(k0 + 16 * p < d ? (double)rk[p] : 0.0, (double)xk[p], u);
      }
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) u += __shfl_xor(u, o);
    if (sub != 0) return;
    const double nrm = __builtin_sqrt(s.s64[v]);
    double d1 = __builtin_inf(), d2 = __builtin_inf();
    int code = 0;
#pragma unroll 1
    for (int l = 0; l < a.m; ++l) {
      const double dv = fabs(u - nrm * ((double)a.cb_scale * (double)a.lv[l]));
      if (dv < d1) {
        d2 = d1;
        d1 = dv;
        code = a.li[l];
      } else if (dv < d2) {
        d2 = dv;
      }
    }
    const double err = (4.0 * d + 32.0) * 2.220446049250313e-16 * nrm *
                       ((double)a.rmax + 128.0 * (double)a.cb_scale);
    if (d2 - d1 > 2.0 * err)
      put_code(v, jl, code);
    else
      (&s.xs[0][0][0])[atomicAdd(&s.nties, 1u)] = item;
  }

  // A tie by the contract's own chains, one thread each: 16 values of either
  // row are requested at a time.
  EOS_DEV void tie(uint32_t item) {
    const int d = a.d, v = (int)(item >> 16), jl = (int)(item & 0xffffu);
    const float* xv = a.x + (size_t)(v0 + v) * d;
    const float* rj = a.rot_r + (size_t)(32 * jt0 + jl) * d;
    double u[1] = {0.0}, ss = 0.0;
#pragma unroll 1
    for (int k0 = 0; k0 < d; k0 += 16) {
      float xk[16], rk[16];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        load4(xk + 4 * p, xv, k0 + 4 * p);
        load4(rk + 4 * p, rj, k0 + 4 * p);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if (k0 + e < d) {
          u[0] = fma((double)rk[e], (double)xk[e], u[0]);
          ss = fma((double)xk[e], (double)xk[e], ss);
        }
      }
    }
    int code[1];
    nearest(u, __builtin_sqrt(ss), code);
    put_code(v, jl, code[0]);
  }

  // Values k .. k + 3 of a row (positions clamped to its end).
  EOS_DEV void load4(float* out, const float* row, int k) {
    if constexpr (VEC) {
      const float4 f = *reinterpret_cast<const float4*>(row + min(k, a.d - 4));
      out[0] = f.x;
      out[1] = f.y;
      out[2] = f.z;
      out[3] = f.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = row[min(k + e, a.d - 1)];
    }
  }
  // The operands of four v_mfma_f64_16x16x4_f64 steps, K values k0 .. k0 + 15
  // (zero past d) of the lane's row: lane group g loads values 4 g .. + 3 and
  // needs value g of each step, a 4 x 4 transposition across the groups.
  EOS_DEV void load_steps(float (&f)[4], const float* row, int k0, int g) {
    load4(f, row, k0 + 4 * g);
    uint32_t u[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = k0 + 4 * g + e < a.d ? __float_as_uint(f[e]) : 0u;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const auto r = __builtin_amdgcn_permlane32_swap(u[e], u[e + 2], false, false);
      u[e] = r[0];
      u[e + 2] = r[1];
    }
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      const auto r = __builtin_amdgcn_permlane16_swap(u[e], u[e + 1], false, false);
      u[e] = r[0];
      u[e + 1] = r[1];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = __uint_as_float(u[e]);
  }

  // Every pair of the tile by the contract, for a list that overflowed: u on
  // v_mfma_f64_16x16x4_f64, whose chain over K is the contract's fma chain
  // (see EncodeIp), 3 x 3 tiles of 16 coordinates x 16 vectors a wavefront;
  // the vectors' norms by a thread each. Bound by the f64 matrix rate.
  EOS_DEV void exact_tile(int tid) {
    const int d = a.d, lane = tid & 63, lr = lane & 15, g = lane >> 4;
    for (int v = tid; v < nv; v += NT) {
      const float* xv = a.x + (size_t)(v0 + v) * d;
      double ss = 0.0;
#pragma unroll 1
      for (int k0 = 0; k0 < d; k0 += 16) {
        float xk[16];
#pragma unroll
        for (int p = 0; p < 4; ++p) load4(xk + 4 * p, xv, k0 + 4 * p);
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (k0 + e < d) ss = fma((double)xk[e], (double)xk[e], ss);
      }
      s.s64[v] = __builtin_sqrt(ss);
    }
    lds_barrier();
    const int jn = min(32 * NW, d - 32 * jt0);
    const int jg = (jn + 47) / 48, vg = (nv + 47) / 48;
#pragma unroll 1
    for (int it = tid >> 6; it < jg * vg; it += NT / 64) {
      const int jb = it % jg * 48 + lr, vb = it / jg * 48 + lr;
      const float *rj[3], *xv[3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        rj[t] = a.rot_r + (size_t)(32 * jt0 + min(jb + 16 * t, jn - 1)) * d;
        xv[t] = a.x + (size_t)(v0 + min(vb + 16 * t, nv - 1)) * d;
      }
      v4d acc[3][3];
#pragma unroll
      for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int t = 0; t < 3; ++t) acc[n][t] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
      for (int k0 = 0; k0 < d; k0 += 16) {
        float rf[3][4], xf[3][4];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          load_steps(rf[t], rj[t], k0, g);
          load_steps(xf[t], xv[t], k0, g);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int n = 0; n < 3; ++n)
#pragma unroll
            for (int t = 0; t < 3; ++t)
              acc[n][t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)rf[t][e], (double)xf[n][e],
                                                               acc[n][t], 0, 0, 0);
      }
      // Element r of a lane: coordinate jb - lr + g + 4 r, vector vb.
#pragma unroll
      for (int n = 0; n < 3; ++n) {
        const int v = vb + 16 * n;
        if (v >= nv) continue;
        const double ne = s.s64[v];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const double u[4] = {acc[n][t][0], acc[n][t][1], acc[n][t][2], acc[n][t][3]};
          int code[4];
          nearest(u, ne, code);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int jl = jb - lr + 16 * t + g + 4 * r;
            if (jl < jn) put_code(v, jl, code[r]);
          }
        }
      }
    }
  }

  // Code rows: the tile's bytes of each vector.
  EOS_DEV void write(int tid) {
    const int rb0 = 4 * jt0 * a.bits;
    const int nb = min(a.row_bytes - rb0, 4 * NW * a.bits);
    uint8_t* out = a.codes + (size_t)v0 * a.row_bytes + rb0;
    if (a.words) {
      const int nw = nb >> 2;
      for (int i = tid; i < nv * nw; i += NT) {
        const int v = i / nw, b = i - v * nw;
        *reinterpret_cast<uint32_t*>(out + (size_t)v * a.row_bytes + 4 * b) =
            *reinterpret_cast<const uint32_t*>(&s.cbuf[v * CST + 4 * b]);
      }
    } else {
      for (int i = tid; i < nv * nb; i += NT) {
        const int v = i / nb, b = i - v * nb;
        out[(size_t)v * a.row_bytes + b] = s.cbuf[v * CST + b];
      }
    }
  }

  EOS_DEV void stage(int tid) {
    const int d = a.d;
    // Thread t stages 4 values (16 bytes) of rows t / 8 + u PT / 8 per chunk.
    // Loads come from clamped positions; what lies past d or n is cleared
    // when the values are stored, so that no load is waited for before that.
    const int slot = tid & 7, row0 = tid >> 3;
    auto load = [&](float (&xr)[U][4], int c) {
      const int k = 32 * c + 4 * slot;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float* src = a.x + (size_t)min(v0 + row0 + u * (PT / 8), a.n - 1) * d;
        if constexpr (VEC) {
          const float4 v = *reinterpret_cast<const float4*>(src + min(k, d - 4));
          xr[u][0] = v.x;
          xr[u][1] = v.y;
          xr[u][2] = v.z;
          xr[u][3] = v.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) xr[u][e] = src[min(k + e, d - 1)];
        }
      }
    };
    double ss[U];
    // Row r's 64 bytes of a stage are four 16-byte groups of 8 K values; group
    // q sits at q ^ ((r >> 2) & 3), so that a fragment read covers all banks.
    auto store = [&](const float (&xr)[U][4], int st, int c) {
      const int k = 32 * c + 4 * slot;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = row0 + u * (PT / 8);
        uint32_t h[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = (r < nv && k + (VEC ? 0 : e) < d) ? xr[u][e] : 0.0f;
          ss[u] = fma((double)v, (double)v, ss[u]);
          h[e] = bf16_bits(v);
          lo[e] = bf16_bits(v - bf16_val(h[e]));
        }
        const int o = r * 16 + (((slot >> 1) ^ ((r >> 2) & 3)) * 4) + (slot & 1) * 2;
        *reinterpret_cast<uint2*>(&s.xs[st][0][o]) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
        *reinterpret_cast<uint2*>(&s.xs[st][1][o]) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
      }
    };
    // Norms, and each vector's scale of w and decision distance.
    auto norms = [&](bool out) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        double sq = ss[u];
        sq += __shfl_xor(sq, 1);
        sq += __shfl_xor(sq, 2);
        sq += __shfl_xor(sq, 4);
        const int r = row0 + u * (PT / 8);
        if (slot != 0) continue;
        const double nrm = __builtin_sqrt(sq);
        if (out && r < nv) {
          const double eps = (double)(d + 8) * 2.220446049250313e-16;
          float nf = (float)nrm;
          if (!((float)__builtin_sqrt(sq * (1.0 - eps)) == (float)__builtin_sqrt(sq * (1.0 + eps)))) {
            const float* src = a.x + (size_t)(v0 + r) * d;
            double w = 0.0;
#pragma unroll 1
            for (int k = 0; k < d; ++k) w = fma((double)src[k], (double)src[k], w);
            nf = (float)__builtin_sqrt(w);
          }
          a.norms[v0 + r] = nf;
        }
        float iv = 0.0f, dl = -2.0f;  // code 0 throughout
        if (nrm > 0.0 && nrm < __builtin_inf()) {
          if (nrm >= 0x1p-90 && nrm <= 0x1p100) {
            iv = (float)(2.0 / (nrm * (double)a.cb_scale));
            dl = a.delta2;
          } else {
            dl = __builtin_inff();  // every coordinate to the list
          }
        }
        s.s64[r] = sq;
        s.inv2[r] = iv;
        s.dlim[r] = dl;
      }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) ss[u] = 0.0;
    float xa[U][4], xb[U][4];
    load(xa, 0);
    load(xb, 1);
    store(xa, 0, 0);
    load(xa, 2);
    lds_barrier();
    for (int c = 0; c + 2 < a.nchunk; c += 2) {
      store(xb, 1, c + 1);
      load(xb, c + 3);
      lds_barrier();
      store(xa, 0, c + 2);
      load(xa, c + 4);
      lds_barrier();
    }
    store(xb, 1, a.nchunk - 1);
    lds_barrier();
    norms(jt0 == 0);  // while the last chunk is multiplied out
    lds_barrier();
  }

  EOS_DEV void run() {
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup w runs on XCD w % 8: the coordinate blocks of a vector block
    // run back to back on one XCD, so its vectors are read into that L2 once.
    const int l = blockIdx.x >> 3;
    v0 = ((long long)(l / a.jblocks) * 8 + (blockIdx.x & 7)) * BM;
    if (v0 >= a.n) return;
    nv = (int)min((long long)BM, a.n - v0);
    jt0 = l % a.jblocks * NW;
    if (wave < NW)
      multiply(wave, tid & 63);
    else
      stage(tid - 64 * NW);
    lds_barrier();
    if (s.nitems > (uint32_t)kSplitItems) {
      exact_tile(tid);
    } else {
      const int total = (int)s.nitems;
#pragma unroll 1
      for (int i = tid >> 4; i < total; i += NT / 16) decide(i, tid & 15);
      lds_barrier();
      const uint32_t* ties = &s.xs[0][0][0];
      for (int i = tid; i < (int)s.nties; i += NT) tie(ties[i]);
    }
    lds_barrier();
    write(tid);
  }
};

}  // namespace

// NW multiplying wavefronts; x rows 16-byte aligned (_v) or not.
#define EOS_TQ_ENCODE_SPLIT(NW)                                                            \
  extern "C" __global__ __launch_bounds__(64 * (NW + kSplitStage)) __attribute__((amdgpu_waves_per_eu(4))) \
  void eos_tq_encode_split_w##NW(TqEncSplitArgs a) {                                      \
    __shared__ __attribute__((aligned(16))) EncodeSplit<NW, false>::Lds lds;              \
    EncodeSplit<NW, false>{a, lds, 0, 0, 0}.run();                                              \
  }                                                                                       \
  extern "C" __global__ __launch_bounds__(64 * (NW + kSplitStage)) __attribute__((amdgpu_waves_per_eu(4))) \
  void eos_tq_encode_split_w##NW##_v(TqEncSplitArgs a) {                                  \
    __shared__ __attribute__((aligned(16))) EncodeSplit<NW, true>::Lds lds;               \
    EncodeSplit<NW, true>{a, lds, 0, 0, 0}.run();                                               \
  }
EOS_TQ_ENCODE_SPLIT(4)
EOS_TQ_ENCODE_SPLIT(8)
EOS_TQ_ENCODE_SPLIT(12)
#undef EOS_TQ_ENCODE_SPLIT

// ------------------------------------------------------- inner-product layout

namespace {

// The inner-product encode (the contract of eos_tq_ip_encode_device) with
// both matrix products on v_mfma_f64_16x16x4_f64. That instruction adds its
// four products to the accumulator one fma after another in K order, so a
// chain of them over K is the contract's fma chain bit for bit (lane l of the
// operands holds row or column l % 16 and K value l / 16; result element r
// is row l / 16 + 4 r, column l % 16).
// Workgroup: 16 NV vectors, all coordinates; wavefront w owns the 16-row tiles
// w, w + 8, ... (at most TJ) of both products. Rotation: x in chunks of 64 K
// values through two LDS stages, R^T fragments from global memory 16 K
// values ahead. The residuals r = u - nrm c then stay in LDS as f64, the
// second product's right operand, and one wavefront runs the ResNorm chains
// over them beside its tiles. Rows of rs are 4 (mod 32) doubles apart: the 16
// vectors x 4 K values of an operand read fall into different banks.
// 200,000 x 384 at 3 bits: 10.96 -> 2.47 ms against f64 VALU chains (one workgroup
// of 8 vectors per CU); bound by the f64 matrix rate (118
// GFLOP; dependent chains of this instruction reach 62 TFLOP/s at two
// wavefronts per SIMD).
// P: steps (of four K values) a fragment load brings. Up to 16 vectors a CU
// nothing hides a load's latency but the chain itself, so those calls take NV
// = 1 and P = 8 at d <= 512 (see the dispatch for both sides).
template <int NV, int TJ, int P>
struct EncodeIp {
  static constexpr int BV = 16 * NV, KC = 64, XST = KC + 4, RST = 128 * TJ + 4;
  static constexpr int kCodeRow = 64 * TJ;  // bytes: 8 TJ tiles x 16 codes of 4 bits
  static constexpr int kSignRow = 16 * TJ;
  static constexpr int kStage = 2 * BV * XST * 4;
  static constexpr int kOut = BV * (kCodeRow + kSignRow);
  struct Lds {
    double rs[BV * RST];
    double ncs[BV * 17];
    double nrms[BV];
    // x stages, then the packed codes and signs
    uint32_t buf[(kStage > kOut ? kStage : kOut) / 4];
  };

  EOS_DEV static void run(const TqIpArgs& a, Lds& s) {
    const int tid = threadIdx.x, lane = tid & 63, d = a.d, levels = 1 << a.bits;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    const long long v0 = (long long)blockIdx.x * BV;
    const int nv = (int)min((long long)BV, a.n - v0);
    const int tiles = (d + 15) / 16;
    float* const xs = reinterpret_cast<float*>(s.buf);

    v4d acc[NV][TJ];
    auto clear = [&]() {
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int t = 0; t < TJ; ++t) acc[n][t] = v4d{0.0, 0.0, 0.0, 0.0};
    };
    // 4 P K values (P steps) of the wavefront's rows of m [k][row].
    auto load_m = [&](float (&f)[P][TJ], const float* m, int k0) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = k0 + 4 * p + lk;
        const float* row = m + (size_t)min(k, d - 1) * d;
#pragma unroll
        for (int t = 0; t < TJ; ++t) f[p][t] = row[min(16 * (wave + 8 * t) + lr, d - 1)];
      }
    };
    auto steps = [&](const float (&f)[P][TJ], int k0, auto&& right) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = k0 + 4 * p + lk;
        double b[NV];
#pragma unroll
        for (int n = 0; n < NV; ++n) b[n] = right(n, k);
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
          const double r = (double)(k < d ? f[p][t] : 0.0f);
#pragma unroll
          for (int n = 0; n < NV; ++n)
            acc[n][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(r, b[n], acc[n][t], 0, 0, 0);
        }
      }
    };

    // Staging thread t: values 4 (t % 16) .. + 3 of chunk c of vector t / 16.
    const int sv = tid >> 4, sk = 4 * (tid & 15);
    const bool stager = sv < BV;
    float xr[4];
    auto load_x = [&](int c) {
      const float* src = a.x + (size_t)(v0 + min(sv, nv - 1)) * d;
#pragma unroll
      for (int e = 0; e < 4; ++e) xr[e] = src[min(KC * c + sk + e, d - 1)];
    };
    auto store_x = [&](int c) {
      if (!stager) return;
      float4 v;
      v.x = (sv < nv && KC * c + sk < d) ? xr[0] : 0.0f;
      v.y = (sv < nv && KC * c + sk + 1 < d) ? xr[1] : 0.0f;
      v.z = (sv < nv && KC * c + sk + 2 < d) ? xr[2] : 0.0f;
      v.w = (sv < nv && KC * c + sk + 3 < d) ? xr[3] : 0.0f;
      *reinterpret_cast<float4*>(&xs[((c & 1) * BV + sv) * XST + sk]) = v;
    };
    const int nchunk = (d + KC - 1) / KC;
    load_x(0);
    store_x(0);
    load_x(1);
    clear();
    double ss = 0.0;
    float fa[P][TJ], fb[P][TJ];
    const bool rot = a.rot_t != nullptr;
    if (rot) load_m(fa, a.rot_t, 0);
    lds_barrier();
    for (int c = 0; c < nchunk; ++c) {
      const float* xc = xs + (c & 1) * BV * XST;
      auto right = [&](int n, int k) { return (double)xc[(16 * n + lr) * XST + (k - KC * c)]; };
      if (rot) {
#pragma unroll
        for (int h = 0; h < KC / (8 * P); ++h) {
          load_m(fb, a.rot_t, KC * c + 8 * P * h + 4 * P);
          steps(fa, KC * c + 8 * P * h, right);
          load_m(fa, a.rot_t, KC * c + 8 * P * h + 8 * P);
          steps(fb, KC * c + 8 * P * h + 4 * P, right);
        }
      }
      // The norms' chains (vector = thread).
      if (tid < BV) {
#pragma unroll 4
        for (int k = 0; k < KC; k += 4) {
          const float4 v = *reinterpret_cast<const float4*>(&xc[tid * XST + k]);
          ss = fma((double)v.x, (double)v.x, ss);
          ss = fma((double)v.y, (double)v.y, ss);
          ss = fma((double)v.z, (double)v.z, ss);
          ss = fma((double)v.w, (double)v.w, ss);
        }
      }
      store_x(c + 1);  // (past the last chunk: zeros nobody reads)
      load_x(c + 2);
      lds_barrier();
    }
    if (tid < BV) {
      const double nrm = __builtin_sqrt(ss);
      s.nrms[tid] = nrm;
      if (tid < nv) a.norms[v0 + tid] = (float)nrm;
      for (int l = 0; l < levels; ++l) s.ncs[tid * 17 + l] = nrm * ((double)a.cb_scale * (double)a.cb[l]);
    }
    if (!rot) {
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int t = 0; t < TJ; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int v = 16 * n + lr, j = 16 * (wave + 8 * t) + lk + 4 * r;
            acc[n][t][r] = v < nv && j < d ? (double)a.x[(size_t)(v0 + v) * d + j] : 0.0;
          }
    }
    lds_barrier();

    // Codes (the first level nearest u) and residuals.
    uint8_t* const cbuf = reinterpret_cast<uint8_t*>(s.buf);
    uint8_t* const sbuf = cbuf + BV * kCodeRow;
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const double* nc = &s.ncs[(16 * n + lr) * 17];
#pragma unroll
      for (int t = 0; t < TJ; ++t) {
        if (wave + 8 * t >= tiles) continue;
        double bd[4];
        int best[4];
        const double n0 = nc[0];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          bd[r] = fabs(acc[n][t][r] - n0);
          best[r] = 0;
        }
        for (int l = 1; l < levels; ++l) {
          const double nl = nc[l];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double dv = fabs(acc[n][t][r] - nl);
            if (dv < bd[r]) {
              bd[r] = dv;
              best[r] = l;
            }
          }
        }
        uint64_t pk = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * (wave + 8 * t) + lk + 4 * r;
          const double res = acc[n][t][r] - nc[best[r]];
          s.rs[(16 * n + lr) * RST + j] = j < d ? res : 0.0;
          if (j < d) pk |= (uint64_t)best[r] << (a.bits * (lk + 4 * r));
        }
        // The tile's 16 codes are 2 bits-many bytes: group lk writes two.
        uint32_t lo = (uint32_t)pk, hi = (uint32_t)(pk >> 32);
        lo |= (uint32_t)__shfl_xor((int)lo, 16);
        hi |= (uint32_t)__shfl_xor((int)hi, 16);
        lo |= (uint32_t)__shfl_xor((int)lo, 32);
        hi |= (uint32_t)__shfl_xor((int)hi, 32);
        if (lk < a.bits)
          *reinterpret_cast<uint16_t*>(&cbuf[(16 * n + lr) * kCodeRow + (wave + 8 * t) * 2 * a.bits + 2 * lk]) =
              (uint16_t)((lk & 2 ? hi : lo) >> (lk & 1 ? 16 : 0));
      }
    }
    lds_barrier();

    if (wave == 7 && lane < nv) {
      double rn = 0.0;
      const double* r = &s.rs[lane * RST];
#pragma unroll 8
      for (int j = 0; j < d; ++j) rn = fma(r[j], r[j], rn);
      const double nrm = s.nrms[lane];
      a.resnorms[v0 + lane] = nrm > 0.0 ? (float)(__builtin_sqrt(rn) / nrm) : 0.0f;
    }
    clear();
    auto right = [&](int n, int k) { return k < d ? s.rs[(16 * n + lr) * RST + k] : 0.0; };
    load_m(fa, a.qjl_t, 0);
    for (int k0 = 0; k0 < d; k0 += 8 * P) {
      load_m(fb, a.qjl_t, k0 + 4 * P);
      steps(fa, k0, right);
      load_m(fa, a.qjl_t, k0 + 8 * P);
      if (k0 + 4 * P < d) steps(fb, k0 + 4 * P, right);
    }
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int t = 0; t < TJ; ++t) {
        if (wave + 8 * t >= tiles) continue;
        uint32_t m = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * (wave + 8 * t) + lk + 4 * r;
          m |= (i < d && acc[n][t][r] >= 0.0 ? 1u : 0u) << (lk + 4 * r);
        }
        m |= (uint32_t)__shfl_xor((int)m, 16);
        m |= (uint32_t)__shfl_xor((int)m, 32);
        if (lk == 0)
          *reinterpret_cast<uint16_t*>(&sbuf[(16 * n + lr) * kSignRow + (wave + 8 * t) * 2]) = (uint16_t)m;
      }
    lds_barrier();
    auto put = [&](uint8_t* dst, int bytes, const uint8_t* src, int pitch) {
      if ((bytes & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 3) == 0) {
        const int nw = bytes >> 2;
        for (int i = tid; i < nv * nw; i += 512) {
          const int v = i / nw, b = i - v * nw;
          reinterpret_cast<uint32_t*>(dst + (size_t)v * bytes)[b] =
              *reinterpret_cast<const uint32_t*>(src + v * pitch + 4 * b);
        }
      } else {
        for (int i = tid; i < nv * bytes; i += 512) {
          const int v = i / bytes, b = i - v * bytes;
          dst[(size_t)v * bytes + b] = src[v * pitch + b];
        }
      }
    };
    put(a.codes + (size_t)v0 * a.row_bytes, a.row_bytes, cbuf, kCodeRow);
    put(a.signs + (size_t)v0 * a.sign_bytes, a.sign_bytes, sbuf, kSignRow);
  }
};

}  // namespace

// 16 NV vectors per workgroup, up to 128 TJ coordinates.
#define EOS_TQ_ENCODE_IP(NAME, NV, TJ, P)                                               \
  extern "C" __global__ __launch_bounds__(512) void eos_tq_encode_ip_##NAME##TJ(TqIpArgs a) { \
    __shared__ __attribute__((aligned(16))) EncodeIp<NV, TJ, P>::Lds lds;               \
    EncodeIp<NV, TJ, P>::run(a, lds);                                                   \
  }
EOS_TQ_ENCODE_IP(t, 2, 1, 4)
EOS_TQ_ENCODE_IP(t, 2, 2, 4)
EOS_TQ_ENCODE_IP(t, 2, 3, 4)
EOS_TQ_ENCODE_IP(t, 2, 4, 4)
EOS_TQ_ENCODE_IP(t, 1, 5, 4)
EOS_TQ_ENCODE_IP(t, 1, 6, 4)
EOS_TQ_ENCODE_IP(t, 1, 7, 4)
EOS_TQ_ENCODE_IP(t, 1, 8, 4)
EOS_TQ_ENCODE_IP(s, 1, 1, 8)
EOS_TQ_ENCODE_IP(s, 1, 2, 8)
EOS_TQ_ENCODE_IP(s, 1, 3, 8)
EOS_TQ_ENCODE_IP(s, 1, 4, 8)
#undef EOS_TQ_ENCODE_IP
