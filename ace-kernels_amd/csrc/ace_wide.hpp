// Wide kernels: the loss's forward and backward for any channel count up to
// 64, softmax or sigmoid, class labels or per-channel targets, hard binning
// and soft binning in the moments layout.  They serve every such call that
// the fast kernels (softmax, class labels, C in {2, 3, 4, 16}) do not, but for
// the soft forwards of few voxels with many bins, where the generic kernels are
// the faster ones (wide_soft_forward_pays).
//
// A lane takes one to four voxels a step (wide_vec), one after the other, all
// channels of a voxel in registers.  The channel count is a compile-time CMAX with
// the channels C .. CMAX - 1 padded: they repeat the last row (cache hits)
// and add 0 to the softmax's sum, so the voxel loop has no branch per
// channel and every load, exponential and table read of a voxel is in flight
// together; only the adds and stores of the few channels that may be padding
// are skipped by a uniform branch.  (A guard per channel, as in the generic
// kernels, makes each channel a serial chain of waits: 970 cycles per
// (wave, channel) at C = 21 against the ~100 of its arithmetic.)  Kernel times
// on MI355X, generic -> wide, forward / backward, and the time of a large copy's
// rate (5.1 TB/s) for the bytes:
//   hard 8 x 21 x 512^2 bf16          258 / 245 -> 46 / 49 us    20 / 34
//   hard 1 x 14 x 97 x 159 x 161      105 / 173 -> 44 / 58 us    31 / 54
//   soft 2 x 5 x 112 x 128 x 96        64 /  59 -> 29 / 26 us    15 / 23
//   soft 2 x 4 x 112^2 x 80, targets   43 /  29 -> 25 / 18 us    13 / 19
//   hard 2 x 3 x 128^3, sigmoid        38 /  24 -> 30 / 20 us    20 / 20
// What is left of the forwards is issue (~25-45 VALU instructions and an
// exponential per value) and the 6-7 us of the cross-block tail.
//
// The probabilities and bins are those of the generic kernels to the bit, and
// so are the hard sums; the soft sums are the exact ones (exact_moment_scale),
// where the generic kernels round each voxel's terms to 2^-41.
#pragma once

#include "ace_core.hpp"

namespace ace {

// The `right` convention is folded into the bucket table (TableRegs::store),
// so every comparison here is the left one.

// VEC consecutive elements of one row as loaded: converting at the load would
// wait for it there, and 16-bit pairs take half the registers.
template <typename T, int VEC>
struct RawRow {
  static constexpr int kBytes = VEC * (int)sizeof(T);
  uint32_t w[(kBytes + 3) / 4];
  __device__ __forceinline__ void load(const T* p, uint32_t bytes) {
    using R = typename RawVec<kBytes, sizeof(T)>::type;
    const R raw = *reinterpret_cast<const R*>(reinterpret_cast<const char*>(p) + bytes);
    w[0] = 0;
    __builtin_memcpy(w, &raw, kBytes);
  }
  __device__ __forceinline__ float get(int j) const {
    if constexpr (sizeof(T) == 4) return __uint_as_float(w[j]);
    const uint32_t pair = w[j >> 1];
    if constexpr (std::is_same<T, __hip_bfloat16>::value) {
      return __uint_as_float((j & 1) ? pair & 0xffff0000u : pair << 16);
    } else {
      const unsigned short half = (unsigned short)((j & 1) ? pair >> 16 : pair);
      T v;
      __builtin_memcpy(&v, &half, 2);
      return to_f32<T>(v);
    }
  }
};

// One step's voxels of a lane.
template <typename T, int C, int VEC, bool LABELS>
struct WideTile {
  RawRow<T, VEC> x[C];
  long long lab[LABELS ? VEC : 1];
  RawRow<float, VEC> y[LABELS ? 1 : C];
};

// The row stride, above 12 channels opaque to the optimiser, so that row
// pointers are formed with two scalar adds where they are used.  Known to be
// the same in every step, the pointers of all rows (and of their gradients)
// were kept across the loop instead, spilled from the scalar registers into
// vector lanes, and read back with 2-3 vector instructions per row and access
// (hard 8 x 21 x 512^2 bf16: 47.6 / 53.0 -> 45.7 / 49.4 us).  Up to 12 channels
// they fit and keeping them is the cheaper way (eval hard 2 x 7 x 0.4 M: 16.6
// us against 17.4).
template <int C>
__device__ __forceinline__ int64_t row_stride(int64_t n) {
  if constexpr (C > 12) asm volatile("" : "+s"(n));
  return n;
}

// The VEC voxels at v - VEC of every row (v at least 1, and the pointers VEC
// elements before the tile); rows C .. CMAX - 1 repeat row nc - 1.  A row's
// uniform pointer plus an unsigned 32-bit byte offset is the address form that
// takes the row from scalar registers: no vector arithmetic per row.
template <typename T, int C, int CMIN, int VEC, bool LABELS>
__device__ __forceinline__ void wide_load(WideTile<T, C, VEC, LABELS>& t, const T* xt,
                                          const long long* lt, const float* yt, int64_t N, uint32_t v,
                                          int nc, bool targets) {
  N = row_stride<C>(N);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    t.x[c].load(xt, v * (uint32_t)sizeof(T));
    xt += (c < CMIN || c + 1 < nc) ? N : 0;
  }
  if (!targets) return;
  if constexpr (LABELS) {
    const char* lb = reinterpret_cast<const char*>(lt) + v * 8u;
    if constexpr (VEC % 2 == 0) {
#pragma unroll
      for (int j = 0; j < VEC; j += 2) {
        const xi64x2 q = *reinterpret_cast<const xi64x2*>(lb + 8 * j);
        t.lab[j] = q.x;
        t.lab[j + 1] = q.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) t.lab[j] = *reinterpret_cast<const long long*>(lb + 8 * j);
    }
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      t.y[c].load(yt, v * 4u);
      yt += (c < CMIN || c + 1 < nc) ? N : 0;
    }
  }
}

// In place: one voxel's logits -> probabilities, the arithmetic of `activate`.
// Padding repeats the last channel (the maximum is unchanged) and adds 0 to
// the sum.
template <int C, int CMIN>
__device__ __forceinline__ void wide_activate(float (&x)[C], int nc, int act) {
  if (act == kActSoftmax) {
    const float m = max_of<C>(x);
    x[0] = exp_neg(x[0] - m);
    float s = x[0];
#pragma unroll
    for (int c = 1; c < C; ++c) {
      x[c] = exp_neg(x[c] - m);
      if (c > CMIN) x[c] = c < nc ? x[c] : 0.0f;
      s += x[c];
    }
    const float y = rcp_rn(s);
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = div_rn(x[c], s, y);
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = sigmoid(x[c]);
  }
}

// Channels of one group whose table reads are issued together, one group
// ahead of the adds (an LDS read cannot pass an LDS atomic).
constexpr int kWideGroup = 4;

// One voxel (logits x, label or targets y) into the histogram copies.
template <int C, int CMIN, bool SOFT, bool LABELS>
__device__ __forceinline__ void wide_accumulate(const FwdParams& P, const Hist& H, const float* tab,
                                                const float* repl, int nc, int copy, int lsh,
                                                float (&x)[C], long long rawlab,
                                                const float (&y)[LABELS ? 1 : C]) {
  const int K = P.K;
  const int off = P.off;
  const int NB = SOFT ? 2 * K : K;
  const float nf = (float)NB;
  const float nw = -(float)P.mw;
  wide_activate<C, CMIN>(x, nc, P.act);
  const uint32_t lab = LABELS ? fast_label<C>(rawlab) : 0u;
  // byte offsets from this lane's copy of channel 0's first bin
  const uint32_t row = (uint32_t)NB << lsh;  // one channel
  unsigned char* const ha = reinterpret_cast<unsigned char*>(H.a + copy);
  const ptrdiff_t dm2 = reinterpret_cast<unsigned char*>(H.m2) - reinterpret_cast<unsigned char*>(H.a);
  constexpr int G = kWideGroup;
  constexpr int NG = (C + G - 1) / G;
  int g[2][G];
  float e[2][G];
  auto guess = [&](int grp) {
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int c = grp * G + i;
      if (c < C) {
        g[grp & 1][i] = bucket_guess(x[c], nf);
        e[grp & 1][i] = tab[g[grp & 1][i] + 1];
      }
    }
  };
  guess(0);
  uint32_t gaddr = 0, gu = 0;
#pragma unroll
  for (int grp = 0; grp < NG; ++grp) {
    if (grp + 1 < NG) guess(grp + 1);
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int c = grp * G + i;
      if (c >= C || (c > CMIN && c >= nc) || (c == 0 && off != 0)) continue;
      const int k = bucket_fix<false>(g[grp & 1][i], e[grp & 1][i], x[c]);
      const uint32_t at = ((uint32_t)k << lsh) + (uint32_t)(c - off) * row;
      const bool hit = LABELS ? lab == (uint32_t)c : y[LABELS ? 0 : c] == 1.0f;
      if constexpr (!SOFT) {
        const uint32_t q = (uint32_t)fx(x[c]);
        const uint32_t hi = hit ? ((1u << (kShiftN - 32)) | (1u << (kShiftG - 32))) : (1u << (kShiftN - 32));
        lds_add(reinterpret_cast<unsigned long long*>(ha + at), ((unsigned long long)hi << 32) | q);
        if constexpr (!LABELS) {
          const float t = y[c];
          if (t != 0.0f && t != 1.0f)
            lds_add(reinterpret_cast<long long*>(reinterpret_cast<unsigned char*>(H.g1 + copy) + at), fx(t));
        }
      } else {
        // a NaN (sigmoid only) counts as 0, as in hard binning
        const float uf = fmaxf(fmaf(x[c], P.msc, (float)k * nw), 0.0f);
        const uint32_t u = cvt_u32(uf);
        const uint32_t hi = hit ? ((1u << (kMomShiftN - 32)) | (1u << (kMomShiftG - 32)))
                                : (1u << (kMomShiftN - 32));
        lds_add(reinterpret_cast<unsigned long long*>(ha + at), ((unsigned long long)hi << 32) | u);
        lds_add(reinterpret_cast<unsigned long long*>(ha + at + dm2), square_word(uf, k == 0));
        if constexpr (LABELS) {
          gaddr = hit ? at : gaddr;
          gu = hit ? u : gu;
        } else {
          if (hit) lds_add(reinterpret_cast<unsigned long long*>(ha + at + 2 * dm2), (unsigned long long)u);
          const float t = y[c];
          if (t != 0.0f && t != 1.0f) {
            // the exact-arithmetic weights of soft_assign64 at half-bin k, a NaN
            // as 0 here too (its weights' bits would land in the sums)
            const double p = (double)fmaxf(x[c], 0.0f);
            const double ld = p - (double)repl[k];
            const double rd = (double)repl[k + 2] - p;
            const double inv = 1.0 / (ld + rd);
            const int l = max(k - 1, 0) >> 1, r = min(k + 1, NB - 1) >> 1;
            long long* gf = H.gf + copy;
            const int R = 1 << (lsh - 3);
            lds_add(gf + ((c - off) * K + l) * R, fx_soft(rd * inv * (double)t, P.sfx));
            lds_add(gf + ((c - off) * K + r) * R, fx_soft(ld * inv * (double)t, P.sfx));
          }
        }
      }
    }
  }
  // without a labelled loss channel gu is 0: the add changes nothing
  if constexpr (SOFT && LABELS)
    lds_add(reinterpret_cast<unsigned long long*>(ha + gaddr + 2 * dm2), (unsigned long long)gu);
}

// VGPRs: at least 4 waves per SIMD up to 16 channels, 3 up to 32, else 2.
constexpr int wide_min_waves(int C) { return C <= 16 ? 4 : (C <= 32 ? 3 : 2); }

template <typename T, int C, int CMIN, int VEC, bool SOFT, bool LABELS>
__global__ void __launch_bounds__(kThreads, (wide_min_waves(C))) fwd_kernel_wide(const FwdParams P) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* tabs = reinterpret_cast<float*>(smem);
  const int K = P.K;
  const int n = SOFT ? 2 * K : K;
  const int nc = CMIN + 1 == C ? C : P.C;
  const int off = P.off;
  const int CL = nc - off;
  const int CK = CL * K;
  const int R = P.copies;
  const int lsh = __builtin_ctz((unsigned)R) + 3;
  const int tid = threadIdx.x;
  const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
  const int b = (int)(blk / P.tiles);
  const int64_t tile = blk - (int64_t)b * P.tiles;
  const int nrepl = SOFT ? 2 * K + 2 : 0;

  const size_t tab_floats = (size_t)((n + 2 + nrepl + 3) / 4 * 4);
  unsigned char* hist = smem + tab_floats * 4;
  const size_t words = (size_t)CL * n * R;
  Hist H;
  H.a = reinterpret_cast<unsigned long long*>(hist);
  H.g1 = reinterpret_cast<long long*>(H.a + words);
  H.m2 = H.a + words;
  H.mg = H.a + 2 * words;
  H.gf = reinterpret_cast<long long*>(H.a + 3 * words);
  const size_t hist_words = (hist_bytes_per_copy(CK, SOFT, LABELS, SOFT) * (size_t)R + 7) / 8;

  const int64_t N = P.N;
  const int64_t t0 = tile * P.tile_vox;
  const int nvox = (int)min(P.tile_vox, N - t0);
  const T* xt = reinterpret_cast<const T*>(P.x) + (int64_t)b * nc * N + t0 - VEC;
  const long long* lt = reinterpret_cast<const long long*>(P.tgt) + (int64_t)b * N + t0 - VEC;
  const float* yt = reinterpret_cast<const float*>(P.tgt) + (int64_t)b * nc * N + t0 - VEC;
  constexpr int stride = kThreads * VEC;

  TableRegs treg;
  treg.load(P.btab, P.rtab, n, nrepl, kThreads);
  // Two tiles in rotation.  A vector that would pass the tile's end moves back
  // to end there (rows hold at least VEC voxels, and earlier tiles more); its
  // first voxels then belong to another lane and are skipped.
  using Tile = WideTile<T, C, VEC, LABELS>;
  Tile ta, tb;
  const int v0 = tid * VEC;
  const int vlast = nvox - VEC;
  auto load = [&](Tile& t, int v) {
    wide_load<T, C, CMIN, VEC, LABELS>(t, xt, lt, yt, N, (uint32_t)(min(v, vlast) + VEC), nc, true);
    keep_order<C>();
  };
  load(ta, v0);
  load(tb, v0 + stride);
  treg.store(tabs, P.btab, P.rtab, n, nrepl, kThreads, 1.0f, P.right);
  {
    unsigned long long* h64 = reinterpret_cast<unsigned long long*>(hist);
    for (size_t i = tid; i < hist_words; i += kThreads) h64[i] = 0ull;
  }
  __syncthreads();
  const float* repl = tabs + n + 2;
  const int copy = tid & (R - 1);
  auto bin = [&](Tile& t, int v) {
    if (v >= nvox) return;
    const int skip = max(v - vlast, 0);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      if (j < skip) continue;
      float x[C], y[LABELS ? 1 : C];
#pragma unroll
      for (int c = 0; c < C; ++c) x[c] = t.x[c].get(j);
      if constexpr (!LABELS) {
#pragma unroll
        for (int c = 0; c < C; ++c) y[c] = t.y[c].get(j);
      }
      wide_accumulate<C, CMIN, SOFT, LABELS>(P, H, tabs, repl, nc, copy, lsh, x,
                                             LABELS ? t.lab[LABELS ? j : 0] : 0, y);
    }
  };
  for (int v = v0; v - v0 < nvox; v += 2 * stride) {
    bin(ta, v);
    load(ta, v + 2 * stride);
    bin(tb, v + stride);
    load(tb, v + 3 * stride);
  }
  __syncthreads();
  constexpr int kMom = !SOFT ? kMomNone : (LABELS ? kMomExact : kMomExactTargets);
  fwd_finish<SOFT, kMom, kMaxWideCopies>(P, H, hist, repl, CK, CL, b, tile, LABELS);
}

// ------------------------------------------------------------ backward

// dL/dx of one voxel, in place in x (logits in, gradient out).  Hard: both
// candidate coefficients (of the guessed bin and the next) are read with the
// table entry that chooses between them, one round trip instead of two.
template <int C, int CMIN, bool SOFT, bool LABELS>
__device__ __forceinline__ void wide_backward(const BwdParams& P, const float* tab, const float* sab,
                                              const float* scg, int nc, float (&x)[C],
                                              long long rawlab, const float (&y)[LABELS ? 1 : C]) {
  const int K = P.K;
  const int off = P.off;
  const float nf = (float)(SOFT ? 2 * K : K);
  wide_activate<C, CMIN>(x, nc, P.act);
  const uint32_t lab = (SOFT && LABELS) ? fast_label<C>(rawlab) : 0u;
  float gp[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    gp[c] = 0.0f;
    if ((c > CMIN && c >= nc) || (c == 0 && off != 0)) continue;
    const int cl = c - off;
    const int g = bucket_guess(x[c], nf);
    const float e = tab[g + 1];
    if constexpr (!SOFT) {
      const float* cg = scg + cl * K + g;
      const float c0 = cg[0], c1 = cg[1];
      gp[c] = e < x[c] ? c1 : c0;
    } else {
      const int h = bucket_fix<false>(g, e, x[c]);
      const int hb = cl * 2 * K + h;
      const float t1 = LABELS ? 0.0f : y[LABELS ? 0 : c];
      const bool hit = LABELS ? lab == (uint32_t)c : t1 == 1.0f;
      const float4 ab = *reinterpret_cast<const float4*>(sab + 8 * hb + (hit ? 4 : 0));
      const float bl = sab[8 * (nc - off) * 2 * K + hb];
      const float t = x[c] - ab.w;
      gp[c] = fmaf(ab.z, t, ab.x) + fmaf(bl, t, ab.y);
      if constexpr (!LABELS) {
        // a fractional target: A_y = A_0 - B y / 2
        if (t1 != 0.0f && !hit)
          gp[c] = (float)(((double)ab.x + (double)ab.y) +
                          ((double)ab.z + (double)bl) * ((double)t - 0.5 * (double)t1));
      }
    }
  }
  if (P.act == kActSoftmax) {
    float dot = 0.0f;
#pragma unroll
    for (int c = 0; c < C; ++c) dot += gp[c] * x[c];
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = x[c] * (gp[c] - dot);
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = gp[c] * x[c] * (1.0f - x[c]);
  }
}

// One vector of every row's gradient.
template <typename T, int C, int CMIN, int VEC, bool NT>
__device__ __forceinline__ void wide_store(T* d, uint32_t v, int64_t N, const float (&out)[C][VEC],
                                           int nc) {
  const uint32_t bytes = v * (uint32_t)sizeof(T);
  N = row_stride<C>(N);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (c <= CMIN || c < nc)
      store_dx<T, VEC, NT>(reinterpret_cast<T*>(reinterpret_cast<char*>(d) + bytes), out[c]);
    d += N;
  }
}

template <typename T, int C, int CMIN, int VEC, bool SOFT, bool LABELS>
__global__ void __launch_bounds__(kThreads, (wide_min_waves(C))) bwd_kernel_wide(const BwdParams P) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* tabs = reinterpret_cast<float*>(smem);
  const int K = P.K;
  const int n = SOFT ? 2 * K : K;
  const int nc = CMIN + 1 == C ? C : P.C;
  const int off = P.off;
  const int CL = nc - off;
  const int CK = CL * K;
  const int tid = threadIdx.x;
  const int64_t blk = xcd_block_back(blockIdx.x, gridDim.x);
  const int b = (int)(blk / P.tiles);
  const int64_t tile = blk - (int64_t)b * P.tiles;
  const int nrepl = SOFT ? 2 * K + 2 : 0;

  const size_t tab_floats = (size_t)((n + 2 + nrepl + 3) / 4 * 4);
  float* scoef = tabs + tab_floats;  // hard: coef times g, and one word past the last bin
  float* sdd = scoef + CK;
  float* sdl = sdd + CK;
  float* sg = sdd + (SOFT ? 2 * CK : 0);
  float* sab = tabs + ((tab_floats + (size_t)CK * (SOFT ? 3 : 1) + CL + 3) & ~(size_t)3);

  const int64_t N = P.N;
  const int64_t t0 = tile * P.tile_vox;
  const int nvox = (int)min(P.tile_vox, N - t0);
  const T* xt = reinterpret_cast<const T*>(P.x) + (int64_t)b * nc * N + t0 - VEC;
  T* dt = reinterpret_cast<T*>(P.dx) + (int64_t)b * nc * N + t0 - VEC;
  const long long* lt = reinterpret_cast<const long long*>(P.tgt) + (int64_t)b * N + t0 - VEC;
  const float* yt = reinterpret_cast<const float*>(P.tgt) + (int64_t)b * nc * N + t0 - VEC;
  constexpr int stride = kThreads * VEC;

  TableRegs treg;
  treg.load(P.btab, P.rtab, n, nrepl, kThreads);
  // as in the forward; a vector moved back computes its first voxels as their
  // own lane does and stores the same bits
  using Tile = WideTile<T, C, VEC, LABELS>;
  Tile ta, tb;
  const int v0 = tid * VEC;
  const int vlast = nvox - VEC;
  auto load = [&](Tile& t, int v) {
    wide_load<T, C, CMIN, VEC, LABELS>(t, xt, lt, yt, N, (uint32_t)(min(v, vlast) + VEC), nc, SOFT);
    keep_order<C>();
  };
  load(ta, v0);
  load(tb, v0 + stride);
  treg.store(tabs, P.btab, P.rtab, n, nrepl, kThreads, 1.0f, P.right);
  const float* cb = P.coef + (int64_t)b * CK;
  const float* db = P.d + (int64_t)b * CK;
  const float* dlb = db + (int64_t)P.B * CK;
  auto g_of = [&](int cl) { return P.jac[b * CL + cl] * P.go[P.go_per_class ? b * CL + cl : 0]; };
  for (int i = tid; i < CK; i += kThreads) {
    if constexpr (SOFT) {
      scoef[i] = cb[i];
      sdd[i] = db[i];
      sdl[i] = dlb[i];
    } else {
      scoef[i] = cb[i] * g_of(i / K);
    }
  }
  if constexpr (SOFT) {
    for (int i = tid; i < CL; i += kThreads) sg[i] = g_of(i);
  } else {
    if (tid == 0) scoef[CK] = 0.0f;  // read beside the last bin, never chosen
  }
  __syncthreads();
  if constexpr (SOFT) {
    soft_half_bin_coefficients(sab, tabs, tabs + n + 2, scoef, sdd, sdl, sg, K, CL);
    __syncthreads();
  }
  auto grad = [&](Tile& t, int v) {
    if (v >= nvox) return;
    float out[C][VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      float x[C], y[LABELS ? 1 : C];
#pragma unroll
      for (int c = 0; c < C; ++c) x[c] = t.x[c].get(j);
      if constexpr (!LABELS) {
#pragma unroll
        for (int c = 0; c < C; ++c) y[c] = t.y[c].get(j);
      }
      wide_backward<C, CMIN, SOFT, LABELS>(P, tabs, sab, scoef, nc, x, LABELS ? t.lab[LABELS ? j : 0] : 0, y);
#pragma unroll
      for (int c = 0; c < C; ++c) out[c][j] = x[c];
    }
    // one kernel for both kinds of store; the empty asm statements keep the
    // compiler from merging the two branches into plain stores
    const uint32_t at = (uint32_t)(min(v, vlast) + VEC);
    if (P.stream) {
      asm volatile("" ::: "memory");
      wide_store<T, C, CMIN, VEC, true>(dt, at, N, out, nc);
      asm volatile("" ::: "memory");
    } else {
      wide_store<T, C, CMIN, VEC, false>(dt, at, N, out, nc);
    }
  };
  for (int v = v0; v - v0 < nvox; v += 2 * stride) {
    grad(ta, v);
    load(ta, v + 2 * stride);
    grad(tb, v + stride);
    load(tb, v + 3 * stride);
  }
}

// ------------------------------------------------------------ launchers

template <typename T, bool SOFT>
hipError_t launch_wide_fwd(const Geometry& g, const FwdParams& p, hipStream_t s);
template <typename T, bool SOFT>
hipError_t launch_wide_bwd(const Geometry& g, const BwdParams& p, hipStream_t s);

template <typename Kern>
hipError_t allow_lds(Kern kern, size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

template <typename T, bool SOFT, int I>
hipError_t wide_fwd_variant(const Geometry& g, const FwdParams& p, hipStream_t s) {
  constexpr WideVariant v = kWideVariants[I];
  constexpr int vl = wide_vec(v.cmax, sizeof(T), SOFT, true, false);
  constexpr int vt = wide_vec(v.cmax, sizeof(T), SOFT, false, false);
  const bool labels = p.tk == kTgtLabels;
  if (g.var.vec != (labels ? vl : vt)) return hipErrorInvalidConfiguration;
  auto kern = labels ? fwd_kernel_wide<T, v.cmax, v.cmin, vl, SOFT, true>
                     : fwd_kernel_wide<T, v.cmax, v.cmin, vt, SOFT, false>;
  const hipError_t e = allow_lds(kern, g.lds_fwd);
  return e != hipSuccess ? e : launch(kern, g.nblk, g.lds_fwd, s, p);
}
template <typename T, bool SOFT, int I>
hipError_t wide_bwd_variant(const Geometry& g, const BwdParams& p, hipStream_t s) {
  constexpr WideVariant v = kWideVariants[I];
  constexpr int vl = wide_vec(v.cmax, sizeof(T), SOFT, true, true);
  constexpr int vt = wide_vec(v.cmax, sizeof(T), SOFT, false, true);
  // the hard gradient reads no targets
  const bool labels = !SOFT || p.tk == kTgtLabels;
  if (g.var.vec != (labels ? vl : vt)) return hipErrorInvalidConfiguration;
  auto kern = bwd_kernel_wide<T, v.cmax, v.cmin, vl, SOFT, true>;
  if constexpr (SOFT)
    if (!labels) kern = bwd_kernel_wide<T, v.cmax, v.cmin, vt, SOFT, false>;
  const hipError_t e = allow_lds(kern, g.lds_bwd);
  return e != hipSuccess ? e : launch(kern, g.nblk, g.lds_bwd, s, p);
}

constexpr int kWideCount = (int)(sizeof(kWideVariants) / sizeof(kWideVariants[0]));
template <typename T, bool SOFT, int I = 0>
hipError_t wide_fwd_switch(const Geometry& g, const FwdParams& p, hipStream_t s) {
  if constexpr (I < kWideCount) {
    if (kWideVariants[I].cmax == g.var.cmax)
      return wide_fwd_variant<T, SOFT, I>(g, p, s);
    return wide_fwd_switch<T, SOFT, I + 1>(g, p, s);
  } else {
    return hipErrorInvalidValue;
  }
}
template <typename T, bool SOFT, int I = 0>
hipError_t wide_bwd_switch(const Geometry& g, const BwdParams& p, hipStream_t s) {
  if constexpr (I < kWideCount) {
    if (kWideVariants[I].cmax == g.var.cmax)
      return wide_bwd_variant<T, SOFT, I>(g, p, s);
    return wide_bwd_switch<T, SOFT, I + 1>(g, p, s);
  } else {
    return hipErrorInvalidValue;
  }
}

#define ACE_DEFINE_WIDE(T, SOFT)                                                                 \
  template <>                                                                                    \
  hipError_t launch_wide_fwd<T, SOFT>(const Geometry& g, const FwdParams& p, hipStream_t s) {    \
    return wide_fwd_switch<T, SOFT>(g, p, s);                                                    \
  }                                                                                              \
  template <>                                                                                    \
  hipError_t launch_wide_bwd<T, SOFT>(const Geometry& g, const BwdParams& p, hipStream_t s) {    \
    return wide_bwd_switch<T, SOFT>(g, p, s);                                                    \
  }

}  // namespace ace
