// Vector-ALU SRGEMM kernel for outputs too small to give the 64 x 64 staged tile a workgroup per compute unit.
//
// One WAVE owns a 32 x 32 block of the output (8 x 8 lanes of 4 x 4) and a share of k; the W waves of a workgroup
// work on the same block, wave w on the k-chunks w, w + W, ...  A wave stages its own chunk of A and B through its
// own piece of LDS, so the main loop has no barrier: a wave's LDS accesses complete in order, and its next chunk
// waits in registers while it computes.  After the loop the W accumulators of every output meet in LDS and each
// thread folds and finishes 1024 / (64 W) outputs of a row-contiguous run.
//
// Why: an output of 256 x 256 is 16 blocks of 64 x 64, which left 240 of 256 compute units idle; 32 x 32 blocks
// spread it over 64 of them, with four to sixteen waves each by the length of k (launch_small).
#pragma once

namespace cuasr_amd {

// KC: k per chunk.
template <typename T, int ADD, int MUL, int KC, int W> struct SmallTile {
  using Ops = ValuTile<T, ADD, MUL, 4, 4, 32, true, false>;   // its operators, masks and zero-sign lookup
  using S = typename Ops::S;
  static constexpr int VW = 16 / sizeof(T);
  static constexpr int R = 4, BLOCK = 8 * R;       // outputs per lane and per wave along either direction
  // rows of 36 floats (40 doubles) more than a multiple of 32: the four k-groups that neighbouring lanes of a
  // k-contiguous load write lie 16 (doubles: 32) banks apart, so the transposing stores do not collide
  static constexpr int PAD = sizeof(S) == 8 ? 8 : 4;
  static constexpr int ASTRIDE = 64 + 8;           // accumulator e of all lanes; the fold reads e = 0..3 of 8 lanes at once
  static constexpr int OUTS = 1024 / (64 * W);     // outputs per thread of a folded 32 x 32 block
  typedef T gvec_t __attribute__((ext_vector_type(VW), aligned(sizeof(T))));
  static constexpr int SV = 16 / sizeof(S);
  typedef S s4_t __attribute__((ext_vector_type(SV)));

  struct alignas(16) Panels { S a[KC][BLOCK + PAD], b[KC][BLOCK + PAD]; };
  union Smem {
    Panels p[W];
    S acc[W][16 * ASTRIDE];
  };

  static constexpr int PER = BLOCK * KC / 64;      // elements of a chunk per lane and operand
  static constexpr int XV = BLOCK / VW, KV = KC / VW, DK = 64 / XV, DX = 64 / KV;   // DK of k (DX of x): what one load of the wave covers

  // One operand's chunk, BLOCK x KC, into registers.  VEC: the block lies inside the matrix (the caller moved its origin
  // back where it would not) and the chunk is whole, so 16-byte loads at element alignment.  A matrix narrower than a block
  // still takes them along k, from clamped rows.  Otherwise element by element with clamped indices (what lands past an edge
  // is never stored, k past the end never used).
  static __device__ __forceinline__ void load(T (&r)[PER], const T *base, long long s_x, long long s_k, int x_end, int k0, int k_end, bool xc,
                                              bool vec, int lane) {
    if (vec && (xc || x_end >= BLOCK)) {
      const int xx = xc ? lane % XV * VW : lane / KV, kk = xc ? lane / XV : lane % KV * VW;
      const T *src = base + (long long)xx * s_x + (long long)(k0 + kk) * s_k;
      const long long next = xc ? DK * s_k : DX * s_x;
#pragma unroll
      for (int p = 0; p < PER / VW; ++p) {
        const gvec_t t = *reinterpret_cast<const gvec_t *>(src + p * next);
#pragma unroll
        for (int e = 0; e < VW; ++e) r[p * VW + e] = t[e];
      }
    } else if (vec) {
      int l = lane;   // (as below)
      asm volatile("" : "+v"(l));
#pragma unroll
      for (int p = 0; p < PER / VW; ++p) {
        const gvec_t t = *reinterpret_cast<const gvec_t *>(base + (long long)min(l / KV + p * DX, x_end - 1) * s_x + (k0 + l % KV * VW));
#pragma unroll
        for (int e = 0; e < VW; ++e) r[p * VW + e] = t[e];
      }
    } else {
      // (worked out again each time: kept from chunk to chunk, these addresses take the main loop's registers)
      int l = lane;
      asm volatile("" : "+v"(l));
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int el = l + 64 * p;
        const int xx = min(xc ? el % BLOCK : el / KC, x_end - 1), kk = min(k0 + (xc ? el / BLOCK : el % KC), k_end - 1);
        r[p] = base[(long long)xx * s_x + (long long)kk * s_k];
      }
    }
  }
  static __device__ __forceinline__ void store(const T (&r)[PER], S (*dst)[BLOCK + PAD], bool xc, bool vec, int lane) {
    if (vec) {
      if (xc) {
#pragma unroll
        for (int p = 0; p < PER / VW; ++p) {
          typedef S svec_t __attribute__((ext_vector_type(VW)));
          svec_t t;
#pragma unroll
          for (int e = 0; e < VW; ++e) t[e] = Ops::staged(r[p * VW + e]);
          *reinterpret_cast<svec_t *>(&dst[lane / XV + p * DK][lane % XV * VW]) = t;
        }
      } else {
#pragma unroll
        for (int p = 0; p < PER / VW; ++p)
#pragma unroll
          for (int e = 0; e < VW; ++e) dst[lane % KV * VW + e][lane / KV + p * DX] = Ops::staged(r[p * VW + e]);
      }
    } else {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int el = lane + 64 * p;
        dst[xc ? el / BLOCK : el % KC][xc ? el % BLOCK : el / KC] = Ops::staged(r[p]);
      }
    }
  }

  template <int U> struct Frag { S a[U][R], b[U][R]; };
  template <int U> static __device__ __forceinline__ void fragment(Frag<U> &f, const Panels &pn, int kk, int ly, int lx) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int h = 0; h < R / SV; ++h) {
        const s4_t t = *reinterpret_cast<const s4_t *>(&pn.a[kk + u][ly * R + h * SV]);
#pragma unroll
        for (int e = 0; e < SV; ++e) f.a[u][h * SV + e] = t[e];
      }
#pragma unroll
      for (int h = 0; h < R / SV; ++h) {
        const s4_t t = *reinterpret_cast<const s4_t *>(&pn.b[kk + u][lx * R + h * SV]);
#pragma unroll
        for (int e = 0; e < SV; ++e) f.b[u][h * SV + e] = t[e];
      }
    }
  }
  template <int U> static __device__ __forceinline__ void compute(S (&acc)[R][R], const Frag<U> &f) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if constexpr (U == 2 && !(Ops::MASKED || Ops::ZERO_SIGN || Ops::FUSED)) {
          const T t0 = Op<MUL>::apply(f.a[0][i], f.b[0][j]), t1 = Op<MUL>::apply(f.a[1][i], f.b[1][j]);
          acc[i][j] = fold<ADD, MUL>(t1, fold<ADD, MUL>(t0, acc[i][j]));   // one three-input minimum
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) acc[i][j] = Ops::term(acc[i][j], f.a[u][i], f.b[u][j]);
        }
      }
    }
  }

  static __device__ __forceinline__ void run(const Problem &p, const Operands &ops, Smem &sm) {
    constexpr int U = sizeof(S) == 8 ? 1 : 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lx = lane & 7, ly = lane >> 3;
    const int tiles_m = (p.m + BLOCK - 1) / BLOCK, tiles_n = (p.n + BLOCK - 1) / BLOCK;
    int bm, bn;
    Ops::tile_coords(blockIdx.x, tiles_m, tiles_n, bm, bn);
    const int first_m = bm * BLOCK, first_n = bn * BLOCK;       // the first row and column this workgroup stores
    // blocks at the far edges start earlier instead of reaching past the matrix: what they compute twice is not stored
    const int m0 = p.m >= BLOCK ? min(first_m, p.m - BLOCK) : first_m, n0 = p.n >= BLOCK ? min(first_n, p.n - BLOCK) : first_n;
    int kb = 0, ke = p.k;
    if (p.workspace) {
      const int parts = p.k_sub > 1 ? p.k_sub : 1, slice = blockIdx.y / parts, part = blockIdx.y % parts;
      const int sb = min(p.k, slice * p.k_per_slice), se = min(p.k, sb + p.k_per_slice);
      const int per = ((se - sb + KC - 1) / KC + parts - 1) / parts * KC;
      kb = min(se, sb + part * per);
      ke = min(se, kb + per);
    }
    const T *A = reinterpret_cast<const T *>(ops.A) + (long long)m0 * p.sa_m, *B = reinterpret_cast<const T *>(ops.B) + (long long)n0 * p.sb_n;
    const bool a_xc = p.sa_m == 1, b_xc = p.sb_n == 1;
    const T ident = scalar_as<T>(p.add_identity);

    const bool partial = p.workspace != nullptr;
    EpilogueScalars<T> e;
    e.alpha = e.beta = e.ident = ident;
    e.source_needed = false;
    if (!partial) e = resolve_scalars<T>(p, MUL);
    const T *C = reinterpret_cast<const T *>(ops.C);
    const int oc = threadIdx.x & 31, orow0 = threadIdx.x >> 5;   // this thread's outputs of the block: column oc, rows orow0 + 2 W o
    T src[OUTS];
    if (e.source_needed) {   // it arrives under the product
#pragma unroll
      for (int o = 0; o < OUTS; ++o)
        src[o] = C[(long long)min(m0 + orow0 + 2 * W * o, p.m - 1) * p.ldc + min(n0 + oc, p.n - 1)];
    }

    S acc[R][R];
    const S init = Ops::start(p, wave == 0 && p.k_sub <= 1);
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) acc[i][j] = init;
    // an output narrower than a block gives up the vectors along its narrow side, and no others (or-and, 1 x 65536 x 256: 42.7
    // us with every operand element by element, 23.5 now; 10 x 60000 x 200: 38.6 and 24.5)
    const bool vec_a = p.m >= BLOCK || !a_xc, vec_b = p.n >= BLOCK || !b_xc;
    Panels &pn = sm.p[wave];
    T ra[PER], rb[PER];
    int k0 = kb + wave * KC;
    if (k0 < ke) {
      const bool whole = k0 + KC <= ke;
      load(ra, A, p.sa_m, p.sa_k, p.m - m0, k0, ke, a_xc, vec_a && whole, lane);
      load(rb, B, p.sb_n, p.sb_k, p.n - n0, k0, ke, b_xc, vec_b && whole, lane);
    }
    for (; k0 < ke; k0 += W * KC) {
      const bool whole = k0 + KC <= ke;
      store(ra, pn.a, a_xc, vec_a && whole, lane);
      store(rb, pn.b, b_xc, vec_b && whole, lane);
      wave_lds_order();   // other lanes read what a lane has stored
      const int kn = k0 + W * KC;
      if (kn < ke) {
        const bool whole_next = kn + KC <= ke;
        load(ra, A, p.sa_m, p.sa_k, p.m - m0, kn, ke, a_xc, vec_a && whole_next, lane);
        load(rb, B, p.sb_n, p.sb_k, p.n - n0, kn, ke, b_xc, vec_b && whole_next, lane);
      }
      if (k0 + KC <= ke) {
        Frag<U> f[2];
        fragment<U>(f[0], pn, 0, ly, lx);
#pragma unroll
        for (int s = 0; s < KC / U; ++s) {
          if (s + 1 < KC / U) fragment<U>(f[(s + 1) & 1], pn, U * (s + 1), ly, lx);
          __builtin_amdgcn_sched_barrier(0);
          compute<U>(acc, f[s & 1]);
        }
      } else {
#pragma unroll 1
        for (int kk = 0; kk < ke - k0; ++kk) {
          Frag<1> f;
          fragment<1>(f, pn, kk, ly, lx);
          compute<1>(acc, f);
        }
      }
      wave_lds_order();   // ... before the next chunk takes its place
    }
    T *out = reinterpret_cast<T *>(ops.D);
    long long ld_out = p.ldd;
    if (partial) {
      out = reinterpret_cast<T *>(p.workspace) + (long long)(p.k_sub > 1 ? blockIdx.y / p.k_sub : blockIdx.y) * p.m * p.n;
      ld_out = p.n;
    }
    __syncthreads();   // the panels are dead: their space takes the accumulators
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) sm.acc[wave][(i * R + j) * ASTRIDE + lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int o = 0; o < OUTS; ++o) {
      const int orow = orow0 + 2 * W * o, row = m0 + orow, col = n0 + oc;
      const int at = ((orow & 3) * 4 + (oc & 3)) * ASTRIDE + (orow >> 2) * 8 + (oc >> 2);
      S s = sm.acc[0][at];
#pragma unroll
      for (int w = 1; w < W; ++w) {
        if constexpr (Ops::MASKED) s |= sm.acc[w][at];
        else s = Op<ADD>::apply(s, sm.acc[w][at]);
      }
      if (row < first_m || row >= p.m || col < first_n || col >= p.n) continue;
      T v;
      if constexpr (Ops::MASKED) v = s ? T(1) : T(0);
      else v = s;
      if constexpr (Ops::ZERO_SIGN) {
        if (v == T(0) && ke > kb)
          v = Ops::last_zero_product(A + (long long)(row - m0) * p.sa_m + (long long)kb * p.sa_k, p.sa_k,
                                     B + (long long)(col - n0) * p.sb_n + (long long)kb * p.sb_k, p.sb_k, ke - kb, v);
      }
      T *dst = out + (long long)row * ld_out + col;
      if constexpr (Ops::SUB_SLICES) {
        if (partial && p.k_sub > 1) {
          native_fold<ADD>(dst, v);
          continue;
        }
      }
      if (!partial) {
        v = Op<MUL>::apply(e.alpha, v);
        if (e.source_needed) v = fold_epilogue<ADD, MUL>(v, Op<MUL>::apply(e.beta, src[o]));
      }
      *dst = v;
    }
  }
};

template <typename T, int ADD, int MUL, int KC, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4))) void small_srgemm_kernel(const Problem p) {
  using Tile = SmallTile<T, ADD, MUL, KC, W>;
  __shared__ typename Tile::Smem sm;
  Tile::run(p, batch_operands<T>(p), sm);
}

// The 64 x 64 staged tile with its k range shared out over 1024 threads is the better one from about 176 workgroups on
// (min-plus f32, 60 % of the chip's compute units: 832^3, 169 of them, 30.3 against 26.8 us here; 896^3, 196, 31.5
// against 36.5), for 8-byte elements from 128 (640^3, 100: 47.9 against 34.3 us; 768^3, 144: 56.8 against 56.1; 832^3:
// 60.8 against 62.5; this kernel's double figures are 6 - 10 % lower since, 512^3 17.6 -> 15.7).  Integer plus-times stays there at every size (its multiply-adds spill here: 512^3 30.9 against 48 us).
template <typename T, int ADD> static bool small_preferred(const Problem &p) {
  if (ADD == kPlus || p.k < 1) return false;
  const long long groups64 = (long long)((p.m + 63) / 64) * ((p.n + 63) / 64) * slice_groups(p) * p.batch;
  if (groups64 <= (sizeof(T) == 8 ? 128 : 176)) return true;
  // ... and where 64 x 64 tiles would cover 1.6 times as much as 32 x 32 blocks, which is more than their better rate is
  // worth on 4-byte elements (1000 products of 32^3: 10.5 us there, 6.8 here; 100 of 80^3, 1.78 times: 13.0 and 9.6;
  // 64 of 100^3, the same cover: 11.2 and 11.4)
  const long long groups32 = (long long)((p.m + 31) / 32) * ((p.n + 31) / 32) * slice_groups(p) * p.batch;
  return sizeof(T) == 4 && groups32 * 10 <= groups64 * 25;
}
template <typename T, int ADD, int MUL, int KC, int W> static hipError_t launch_small_as(const Problem &p, hipStream_t s) {
  const long long tiles = (long long)((p.m + 31) / 32) * ((p.n + 31) / 32);
  if (tiles > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)tiles, slice_groups(p), p.batch);
  launch_kernel((small_srgemm_kernel<T, ADD, MUL, KC, W>), grid, dim3(64 * W), 0, s, p);
  return take_launch_status();
}

template <typename T, int ADD, int MUL> static hipError_t launch_small(const Problem &p, hipStream_t s) {
  if (p.m == 0 || p.n == 0) return hipSuccess;
  constexpr int KC = 64 / sizeof(T);
  const long long tiles = (long long)((p.m + 31) / 32) * ((p.n + 31) / 32);
  const long long groups = tiles * slice_groups(p) * p.batch;
  const long long k_range = p.workspace ? p.k_per_slice / (p.k_sub > 1 ? p.k_sub : 1) : p.k;
  const long long chunks = (k_range + KC - 1) / KC;
  // Waves per block: as many as keep the workgroups resident together (1024 threads: one per compute unit, 512: two,
  // 256: four) and leave each wave chunks enough to carry the fold: sixteen waves want four chunks each (256 x 256 x
  // 2048: 21.8 us against 24.1 with eight; 512^3, two chunks each: 10.3 against 9.6), eight want two (900 x 900 x 200,
  // 841 blocks: 16.5 us against 14.6 with four; 832^3, 676 blocks of 52 chunks: 26.8 against 29.5).
  const int w = groups <= 256 && chunks >= 64 ? 16 : (groups <= 512 && chunks >= 8) || chunks >= 32 ? 8 : 4;
  if (w == 16) return launch_small_as<T, ADD, MUL, KC, 16>(p, s);
  if (w == 8) return launch_small_as<T, ADD, MUL, KC, 8>(p, s);
  return launch_small_as<T, ADD, MUL, KC, 4>(p, s);
}

}  // namespace cuasr_amd
