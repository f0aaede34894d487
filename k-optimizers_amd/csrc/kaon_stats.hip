// kaon_stats.hip -- phase 1 of the step: GC row means, the factored second
// moment's row EMA and the column partials of G^2 and of the clip's G^2 / row
// (src/kaon/_backend.py:147-177, src/kaon/_factored.py:26-83).  All sums follow
// the canonical order of include/kaon_amd.h; there are no floating-point atomics.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kaon_common.h"

using namespace kaon;

namespace kaon {
using StatsFn = void (*)(const KaonTensor*, const KaonItem*, Ws, KaonHyper, int);
StatsFn rag_bf16(int cls);
StatsFn rag_f16(int cls);
StatsFn rag_f32(int cls);
}  // namespace kaon

namespace {

// Columns per LDS segment of the streamed rows' column fold (phase 1).
constexpr int kSeg = 4096;

// KProdigy's coupled decay folded into the gradient its second moment sees,
// g' = fma(wd, p, GC(g)) (_collect_grad, kprodigy.py:406-414; torch's add with
// alpha is one fused multiply-add), for the generic phase-1 kernel.
__device__ __forceinline__ void add_coupled_wd(const KaonTensor& T, const KaonHyper& hp, int64_t e0, int cnt, bool vv,
                                               float x[8]) {
  float p[8];
  if (hp.p_dtype == KAON_BF16) ld8<KAON_BF16>(T.p, e0, cnt, vv, p);
  else if (hp.p_dtype == KAON_F16) ld8<KAON_F16>(T.p, e0, cnt, vv, p);
  else ld8<KAON_F32>(T.p, e0, cnt, vv, p);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = __fmaf_rn(hp.wdl, p[i], x[i]);
}

// mode 0 (Adakaon): GC row mean (stored), row EMA of mean_C(G^2), column
// partial of the slice (wave groups folded in order in LDS); 1-D tensors: v
// EMA.  mode 1 (Lion): GC row means only.  CPL == 0 streams the row from memory
// (rows longer than 24 chunks per lane, fp32 and fp16 grads of more than 10, and
// 1-D).  CPL > 0 keeps a row of up to CPL chunks per lane in registers: KProdigy's
// coupled decay (KAON_F_PD_COUPLED, factored) of every shorter row.  There G is the
// decayed gradient fma(wd, p, GC(g)); the GC mean is still the raw gradient's.
template <int GT, int CPL>
__global__ __launch_bounds__(KAON_WG) void k_stats(const KaonTensor* __restrict__ D,
                                                   const KaonItem* __restrict__ items, Ws ws, KaonHyper hp,
                                                   int mode) {
  extern __shared__ float lds_col[];
  __shared__ float winv_s[4][KAON_ROW_BUDGET];  // 1 / row (the new row) of each wave's rows
  __shared__ float red4[4];
  const KaonItem it = items[blockIdx.x];
  const KaonTensor& T = D[it.tensor];
  // KProdigy's per-element v and its block-factored tensors: their own pass 1 kernels
  if (T.full_v || T.fb_r) return;
  zero_accumulators(T, it, ws, hp.codec);
  const void* gsrc = ws.src(T, hp.flags);
  const int64_t C = T.C;
  const int64_t nch = (C + 7) >> 3;
  const int cpl = (int)((nch + 63) >> 6);
  const bool vec = T.vec_rows != 0;
  const bool eps = (hp.flags & KAON_F_EPS) != 0;
  if constexpr (CPL > 0) mode = 0;
  const bool alg = CPL == 0 && clip_alg(hp, mode);  // KProdigy does not clip
  const bool cwd = CPL > 0 || (mode == 0 && (hp.flags & KAON_F_PD_COUPLED) != 0);

  if constexpr (CPL == 0) {
    if (!T.factored) {
      if (mode == 0) stats_1d<GT>(T, gsrc, hp, alg ? ws.scal(T) : nullptr, red4);
      return;
    }
  }

  const bool gc = (hp.flags & KAON_F_GC) != 0;
  if (mode == 1 && !gc) return;
  KAON_G float* mu_arr = ws.mu(T);
  const int RW = it.kind;
  KAON_G float* part = run_part(ws, T, it);
  const int nsl = run_slices(it);
#pragma clang loop unroll(disable)
  for (int sl = 0; sl < nsl; ++sl) {
  const WaveRows wr = wave_rows(slice_item(it, sl));

  // registers: row buffer (CPL chunks) and the wave-group column partial
  constexpr int NB = CPL > 0 ? CPL : 1;
  float xb[NB][8];
  float colacc[NB][8];
#pragma unroll
  for (int k = 0; k < NB; ++k)
#pragma unroll
    for (int i = 0; i < 8; ++i) colacc[k][i] = 0.0f;

  for (int64_t r = wr.rb; r < wr.re; ++r) {
    const int64_t rowoff = r * C;
    float mu = 0.0f;
    if (CPL > 0) {
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const int64_t c = wr.lane + 64 * k;
        const int cnt = k < cpl ? chunk_cnt(c, C) : 0;
        if (cnt > 0) ld8<GT>(gsrc, rowoff + c * 8, cnt, vec && cnt == 8, xb[k]);
        else
#pragma unroll
          for (int i = 0; i < 8; ++i) xb[k][i] = 0.0f;
      }
      if (gc) {
        float a = 0.0f;
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int cnt = k < cpl ? chunk_cnt(wr.lane + 64 * k, C) : 0;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (i < cnt) a = a + xb[k][i];
        }
        mu = round_to<GT>(wave_csum(a) / (float)C);
        if (wr.lane == 0) mu_arr[r] = mu;
#pragma unroll
        for (int k = 0; k < NB; ++k) {
#pragma unroll
          for (int i = 0; i < 8; i += 2) {
            float a0 = xb[k][i] - mu, a1 = xb[k][i + 1] - mu;
            round_pair<GT>(a0, a1);
            xb[k][i] = a0;
            xb[k][i + 1] = a1;
          }
        }
      }
      if (mode == 1) continue;
      if (cwd) {
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int64_t c = wr.lane + 64 * k;
          const int cnt = k < cpl ? chunk_cnt(c, C) : 0;
          if (cnt > 0) add_coupled_wd(T, hp, rowoff + c * 8, cnt, vec && cnt == 8, xb[k]);
        }
      }
      float a2 = 0.0f;
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const int cnt = k < cpl ? chunk_cnt(wr.lane + 64 * k, C) : 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i < cnt) {
            float q = xb[k][i] * xb[k][i];
            if (eps) q = q + hp.eps1;
            a2 = a2 + q;
            if (RW > 1) colacc[k][i] = colacc[k][i] + q;
          }
      }
      const float s2 = wave_csum(a2);
      const float nr = klerp(T.row[r], s2 / (float)C, hp.w2);
      if (wr.lane == 0) {
        T.row[r] = nr;
        if (alg) winv_s[wr.w][r - wr.rb] = 1.0f / nr;
      }
    } else {
      // streaming: sweep A (GC sum), sweep B (q and the row sum)
      if (gc) {
        float a = 0.0f;
        for (int k = 0; k < cpl; ++k) {
          const int64_t c = wr.lane + 64 * k;
          const int cnt = chunk_cnt(c, C);
          if (cnt <= 0) continue;
          float x[8];
          ld8<GT>(gsrc, rowoff + c * 8, cnt, vec && cnt == 8, x);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (i < cnt) a = a + x[i];
        }
        mu = round_to<GT>(wave_csum(a) / (float)C);
        if (wr.lane == 0) mu_arr[r] = mu;
      }
      if (mode == 1) continue;
      float a2 = 0.0f;
      for (int k = 0; k < cpl; ++k) {
        const int64_t c = wr.lane + 64 * k;
        const int cnt = chunk_cnt(c, C);
        if (cnt <= 0) continue;
        float x[8];
        ld8<GT>(gsrc, rowoff + c * 8, cnt, vec && cnt == 8, x);
        if (gc) {
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = round_to<GT>(x[i] - mu);
        }
        if (cwd) add_coupled_wd(T, hp, rowoff + c * 8, cnt, vec && cnt == 8, x);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i < cnt) {
            float q = x[i] * x[i];
            if (eps) q = q + hp.eps1;
            a2 = a2 + q;
          }
      }
      const float s2 = wave_csum(a2);
      const float nr = klerp(T.row[r], s2 / (float)C, hp.w2);
      if (wr.lane == 0) {
        T.row[r] = nr;
        if (alg) winv_s[wr.w][r - wr.rb] = 1.0f / nr;
      }
    }
  }
  if (mode == 1) continue;

  // fold the wave-group partials in group order into the slice partial
  const bool has_rows = wr.re > wr.rb;
  if (CPL == 0) {
    // streamed rows (RW == 1, any length): the slice partial is folded kSeg
    // columns at a time through LDS.  Per column the order is the one below:
    // wave 0 + wave 1 + wave 2 + wave 3, then the slice added to the run partial.
    for (int64_t c0 = 0; c0 < C; c0 += kSeg) {
      const int64_t c1 = min(C, c0 + (int64_t)kSeg);
      for (int wf = 0; wf < 4; ++wf) {
        if (wr.w == wf && has_rows) {
          const int64_t r = wr.rb;
          const float mu = gc ? mu_arr[r] : 0.0f;
          for (int64_t c = (c0 >> 3) + wr.lane; c * 8 < c1; c += 64) {
            const int cnt = chunk_cnt(c, C);
            float x[8];
            ld8<GT>(gsrc, r * C + c * 8, cnt, vec && cnt == 8, x);
            if (gc) {
#pragma unroll
              for (int i = 0; i < 8; ++i) x[i] = round_to<GT>(x[i] - mu);
            }
            if (cwd) add_coupled_wd(T, hp, r * C + c * 8, cnt, vec && cnt == 8, x);
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (i < cnt) {
                float v = x[i] * x[i];
                if (eps) v = v + hp.eps1;
                const int64_t j = c * 8 + i - c0;
                lds_col[j] = wf == 0 ? v : lds_col[j] + v;
              }
          }
        }
        __syncthreads();
      }
      for (int64_t j = c0 + threadIdx.x; j < c1; j += KAON_WG)
        part[j] = sl == 0 ? lds_col[j - c0] : part[j] + lds_col[j - c0];
      __syncthreads();  // lds_col is reused by the next segment
    }
  } else {
  for (int wf = 0; wf < 4; ++wf) {
    if (wr.w == wf && has_rows) {
      if (CPL > 0) {
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int64_t c = wr.lane + 64 * k;
          const int cnt = k < cpl ? chunk_cnt(c, C) : 0;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (i < cnt) {
              float v;
              if (RW > 1) {
                v = colacc[k][i];
              } else {
                v = xb[k][i] * xb[k][i];
                if (eps) v = v + hp.eps1;
              }
              const int64_t j = c * 8 + i;
              lds_col[j] = wf == 0 ? v : lds_col[j] + v;
            }
        }
      }
    }
    __syncthreads();
  }
  // the run partial: the slice partials added in slice order
  for (int64_t j = threadIdx.x; j < C; j += KAON_WG) part[j] = sl == 0 ? lds_col[j] : part[j] + lds_col[j];
  __syncthreads();  // lds_col is reused by the next slice
  }
  if (!alg) continue;
  // The clip's second column partial, t = (G * G) / row (the new row; no
  // eps1), in the same wave-group / slice / run order, the rows read again
  KAON_G float* part2 = part + (int64_t)T.ngroups * C;
  for (int64_t c0 = 0; c0 < C; c0 += kSeg) {
    const int64_t c1 = min(C, c0 + (int64_t)kSeg);
    for (int wf = 0; wf < 4; ++wf) {
      if (wr.w == wf && has_rows) {
        for (int64_t c = (c0 >> 3) + wr.lane; c * 8 < c1; c += 64) {
          const int cnt = chunk_cnt(c, C);
          float acc[8];
          for (int64_t r = wr.rb; r < wr.re; ++r) {
            const float mu = gc ? mu_arr[r] : 0.0f;
            const float w = winv_s[wf][r - wr.rb];
            float x[8];
            ld8<GT>(gsrc, r * C + c * 8, cnt, vec && cnt == 8, x);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const float gv = gc ? round_to<GT>(x[i] - mu) : x[i];
              const float t = (gv * gv) * w;
              acc[i] = r == wr.rb ? t : acc[i] + t;
            }
          }
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (i < cnt) {
              const int64_t j = c * 8 + i - c0;
              lds_col[j] = wf == 0 ? acc[i] : lds_col[j] + acc[i];
            }
        }
      }
      __syncthreads();
    }
    for (int64_t j = c0 + threadIdx.x; j < c1; j += KAON_WG)
      part2[j] = sl == 0 ? lds_col[j - c0] : part2[j] + lds_col[j - c0];
    __syncthreads();  // lds_col is reused by the next segment or slice
  }
  }
}

// =============================================================== row kernels
// Phase 1 for factored rows of at most 24 chunks per lane (fp32: 10).  A wave
// loads its whole wave group (RW rows, RW * CPL <= 24 chunks per lane) into
// registers as stored, every load issued before the first use, so each lane
// keeps up to 24 x 16 bytes in flight; the row reductions and the column fold
// then run from registers.  RAG false: bf16 rows of whole 16-byte chunks (row
// classes 0-2).  RAG true: any gradient type, row length and alignment (classes
// 3-5): gfx950 loads 16 bytes from any address, a row's partial last chunk reads
// on into the next row (the tensor's last row: the 8 elements before its end,
// shifted down) and its missing elements are masked out of the row sums; the
// column partials past the row's end are never read.  The arithmetic and its
// order are those of k_stats.
//
// k_stats walked such rows one at a time, each row (and each chunk of an
// unaligned row, element by element) a memory round trip, and read them again
// for the clip's partial.  Rows of 771 / 2057 bf16 elements (52 M params): 557 +
// 550 -> 51 + 64 us; fp32 rows of 768 / 3072 (124 M params, 494 MB): 540 + 296 ->
// 140 + 65 us.  Unaligned and 32-byte chunks share cache lines between loads:
// plain loads, non-temporal ones cost 72 + 64 us in the odd rows.
template <int GT>
constexpr int gt_words() {
  return GT == KAON_F32 ? 8 : 4;
}
template <int GT>
struct Raw {
  uint32_t w[gt_words<GT>()];
};

template <int GT, bool RAG>
__device__ __forceinline__ void ld_raw(Raw<GT>& v, const KAON_G uint8_t* a) {
#pragma unroll
  for (int h = 0; h < gt_words<GT>() / 4; ++h) {
    ku4 x;
    if (RAG) x = ((const KAON_G ku4_any*)a)[h];
    else x = ld_stream<true>((const KAON_G ku4*)a + h);
    v.w[4 * h] = x.x;
    v.w[4 * h + 1] = x.y;
    v.w[4 * h + 2] = x.z;
    v.w[4 * h + 3] = x.w;
  }
}
template <int GT>
__device__ __forceinline__ void raw_floats(const Raw<GT>& v, float x[8]) {
  if constexpr (GT == KAON_F32) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(v.w[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = GT == KAON_BF16 ? __uint_as_float(v.w[i] << 16) : h2f(v.w[i] & 0xFFFFu);
      x[2 * i + 1] = GT == KAON_BF16 ? __uint_as_float(v.w[i] & 0xFFFF0000u) : h2f(v.w[i] >> 16);
    }
  }
}
// The chunk moved down by d elements (zeros above).
template <int GT>
__device__ __forceinline__ Raw<GT> raw_down(Raw<GT> v, int d) {
  for (int s = 0; s < d; ++s) {
    if constexpr (GT == KAON_F32) {
#pragma unroll
      for (int i = 0; i < 7; ++i) v.w[i] = v.w[i + 1];
      v.w[7] = 0u;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v.w[i] = (v.w[i] >> 16) | (i < 3 ? v.w[i + 1] << 16 : 0u);
    }
  }
  return v;
}

// Chunk k of the lane in each of the wave group's rows.  Every load is
// issued unconditionally from a valid address (rows past the group and
// chunks past the row end load the last ones again, and a wave without rows
// loads row `rsafe`), so no load waits behind a divergent branch; the caller
// ignores the extra values.
template <int GT, int CPL, int RW, bool RAG>
__device__ __forceinline__ void load_group(const void* g, int64_t rb, int nrows, int64_t rsafe, int64_t R,
                                           int64_t C, int nch, int lane, Raw<GT> (&raw)[RW][CPL]) {
  constexpr int ES = GT == KAON_F32 ? 4 : 2;
  uint32_t off[CPL];
#pragma unroll
  for (int k = 0; k < CPL; ++k) off[k] = 8u * ES * (uint32_t)min(lane + 64 * k, nch - 1);
  // RAG: the elements the last chunk lacks, and that chunk's lanes
  const int d = RAG ? 8 * nch - (int)C : 0;
  const bool tail = RAG && lane + 64 * (CPL - 1) >= nch - 1;
  const uint32_t off_last = off[CPL - 1] - (tail ? (uint32_t)(ES * d) : 0u);
#pragma unroll
  for (int j = 0; j < RW; ++j) {
    const int64_t r = nrows > 0 ? rb + min(j, nrows - 1) : rsafe;
    const KAON_G uint8_t* rowp = (const KAON_G uint8_t*)G((const uint8_t*)g + ES * (r * C));
#pragma unroll
    for (int k = 0; k < CPL; ++k)
      ld_raw<GT, RAG>(raw[j][k], rowp + (RAG && k == CPL - 1 && r == R - 1 ? off_last : off[k]));
  }
  if (RAG && d > 0) {
#pragma unroll
    for (int j = 0; j < RW; ++j) {
      const int64_t r = nrows > 0 ? rb + min(j, nrows - 1) : rsafe;
      if (r == R - 1) {
        const Raw<GT> v = raw_down<GT>(raw[j][CPL - 1], d);
        if (tail) raw[j][CPL - 1] = v;
      }
    }
  }
}

// q = (G - mu)^2 + e1 of one chunk, G - mu rounded to the grad type (GC in the
// grad dtype); e1 is eps1, or 0 without it (x*x + 0 is x*x: a square is never
// -0).  EPS 2: x*x + e1 rounded twice; 1: the same as one fused multiply-add,
// which gives the same bits for every bf16-valued x when e1 is 0 or at least
// 2^-100: x*x is exact unless |x| < 2^-67, and then x*x < 2^-134 lies below half
// an ulp of e1, so both forms give e1.
// With gc the chunk's GC'd values replace it in `v` (as stored), for the clip
// partial's second pass over the row registers.
template <int EPS>
__device__ __forceinline__ float sq1(float x, float e1) {
  return EPS == 1 ? __fmaf_rn(x, x, e1) : x * x + e1;
}
template <int GT, int EPS>
__device__ __forceinline__ void sq_chunk(Raw<GT>& v, float mu, bool gc, float e1, float q[8]) {
  float x[8];
  raw_floats<GT>(v, x);
  if (gc) {
    if constexpr (GT == KAON_BF16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v.w[i] = f2bf2(x[2 * i] - mu, x[2 * i + 1] - mu);
        x[2 * i] = __uint_as_float(v.w[i] << 16);
        x[2 * i + 1] = __uint_as_float(v.w[i] & 0xFFFF0000u);
      }
    } else if constexpr (GT == KAON_F16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v.w[i] = f2h(x[2 * i] - mu) | (f2h(x[2 * i + 1] - mu) << 16);
      raw_floats<GT>(v, x);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[i] = x[i] - mu;
        v.w[i] = __float_as_uint(x[i]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = sq1<EPS>(x[i], e1);
}
// Squares of a chunk whose values are final (GC'd in place by sq_chunk).
template <int GT>
__device__ __forceinline__ void sq_plain(const Raw<GT>& v, float q[8]) {
  float x[8];
  raw_floats<GT>(v, x);
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = x[i] * x[i];
}

// Column partial of a slice, segment by segment: segment k is chunk k of
// every lane (columns 512k .. 512k+511).  Each wave writes its wave group's
// partial for the segment into its LDS slot, and after one barrier every
// thread forms the ordered sum ((w0 + w1) + w2) + w3 of two columns and
// stores it (two LDS buffers alternate, so one barrier per segment suffices).
__device__ __forceinline__ void seg_put(float (*seg)[512], int w, int lane, const float v[8]) {
  kf4* d = (kf4*)(&seg[w][lane * 8]);
  d[0] = kf4{v[0], v[1], v[2], v[3]};
  d[1] = kf4{v[4], v[5], v[6], v[7]};
}
// Two neighbouring columns of a partial: one 8-byte store where the partial's rows
// are 8-byte aligned, column by column where they may be of odd length.
template <bool RAG>
__device__ __forceinline__ void put2(KAON_G float* dst, bool two, float a0, float a1) {
  if (RAG) {
    dst[0] = a0;
    if (two) dst[1] = a1;
  } else {
    *(KAON_G ku2*)dst = ku2{__float_as_uint(a0), __float_as_uint(a1)};
  }
}
// The run partial (the slice partials added in slice order) is kept in
// `racc` (LDS, C floats; each thread owns its two columns) and stored to
// `part` after the last slice, or, with racc == nullptr, accumulated in
// `part` itself.
template <bool RAG>
__device__ __forceinline__ void seg_fold(float (*seg)[512], int nw, int64_t col0, int64_t C, KAON_G float* part,
                                         bool acc, bool last, int tid, float* racc) {
  const int c = 2 * tid;
  if (col0 + c >= C) return;
  const bool two = !RAG || col0 + c + 1 < C;  // C % 8 == 0: both columns are in range or neither
  float a0 = seg[0][c], a1 = seg[0][c + 1];
  for (int w = 1; w < nw; ++w) {
    a0 = a0 + seg[w][c];
    a1 = a1 + seg[w][c + 1];
  }
  KAON_G ku2* dst = (KAON_G ku2*)(part + col0 + c);
  if (racc) {
    float* r = racc + col0 + c;
    if (acc) {
      a0 = r[0] + a0;
      a1 = r[1] + a1;
    }
    if (!last) {
      r[0] = a0;
      r[1] = a1;
      return;
    }
  } else if (acc) {
    if (RAG) {
      a0 = part[col0 + c] + a0;
      if (two) a1 = part[col0 + c + 1] + a1;
    } else {
      const ku2 o = *dst;
      a0 = __uint_as_float(o.x) + a0;
      a1 = __uint_as_float(o.y) + a1;
    }
  }
  put2<RAG>(part + col0 + c, two, a0, a1);
}
// seg_fold with the run partial of the thread's two columns of segment k in
// registers (r0, r1) instead of LDS; the order is the same.
template <bool RAG>
__device__ __forceinline__ void seg_fold_reg(float (*seg)[512], int nw, int64_t col0, int64_t C,
                                             KAON_G float* part, bool acc, bool last, int tid, float& r0,
                                             float& r1) {
  const int c = 2 * tid;
  if (col0 + c >= C) return;
  float a0 = seg[0][c], a1 = seg[0][c + 1];
  for (int w = 1; w < nw; ++w) {
    a0 = a0 + seg[w][c];
    a1 = a1 + seg[w][c + 1];
  }
  if (acc) {
    a0 = r0 + a0;
    a1 = r1 + a1;
  }
  if (!last) {
    r0 = a0;
    r1 = a1;
    return;
  }
  put2<RAG>(part + col0 + c, !RAG || col0 + c + 1 < C, a0, a1);
}

// The second (clip) partial's run accumulator: racc2 in LDS (REG2 false), or
// the thread's two columns per segment in registers rr2 (REG2 true).
template <int CPL, int RW, int GT, int EPS, bool REG2, bool RAG>
__device__ __forceinline__ void pf_stats_body(const KaonTensor& T, const KaonItem& it, const Ws& ws,
                                              const KaonHyper& hp, int mode, float (*seg)[4][512],
                                              KAON_G float* part, bool acc, bool last, float* racc,
                                              KAON_G float* part2, float* racc2, float (&rr2)[48]) {
  const int64_t C = T.C;
  const int nch = (int)((C + 7) >> 3);
  WaveRows wr = wave_rows(it);
  // recomputed per slice: values derived from the lane are not kept live
  // across the slice loop
  asm volatile("" : "+v"(wr.lane));
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int nrows = (int)(wr.re - wr.rb);
  const bool gc = (hp.flags & KAON_F_GC) != 0;
  const float e1 = (hp.flags & KAON_F_EPS) ? hp.eps1 : 0.0f;
  if (mode == 1 && (!gc || nrows <= 0)) return;
  const int64_t rl = lane_row(wr.rb, nrows, wr.lane);
  const float row_old = (mode == 0 && nrows > 0) ? G(T.row)[rl] : 0.0f;
  const void* gsrc = ws.src(T, hp.flags);
  Raw<GT> raw[RW][CPL];
  load_group<GT, CPL, RW, RAG>(gsrc, wr.rb, nrows, it.row0, T.R, C, nch, wr.lane, raw);
  // RAG: how many elements of the lane's last chunk exist
  const int vc = RAG ? (int)C - 8 * (wr.lane + 64 * (CPL - 1)) : 8;
  // GC means of the wave's rows; both per-row divisions by C are exact
  // through the fp64 reciprocal (div_r64)
  const double rc = rcp64((float)C);
  float mu[RW];
  KAON_G float* mu_arr = ws.mu(T);
#pragma unroll
  for (int j = 0; j < RW; ++j) {
    mu[j] = 0.0f;
    if (j >= nrows || !gc) continue;
    float a = 0.0f;
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
      if (k < CPL - 1 || wr.lane + 64 * k < nch) {
        float x[8];
        raw_floats<GT>(raw[j][k], x);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          // a masked element adds +0, which leaves a sum that started from +0
          a = a + (RAG && k == CPL - 1 && i >= vc ? 0.0f : x[i]);
      }
    }
    mu[j] = round_to<GT>(div_r64(wave_csum(a), rc));
    if (wr.lane == 0) mu_arr[wr.rb + j] = mu[j];
  }
  if (mode == 1) return;
  // q = (G - mu)^2 (+eps1) once per element: into the row sums (lane order:
  // chunk by chunk) and the wave group's column partial (row order)
  const int nw = (int)min<int64_t>(4, ((int64_t)it.nrows + RW - 1) / RW);
  // Segments per barrier: the wide class (REG2: the clip's run partial in
  // registers) has the LDS for two, so it waits half as often.  The buffer
  // sets alternate from one barrier group to the next, across both passes;
  // each column's partials are added in the same order either way.
  constexpr int SEGG = REG2 ? 2 : 1;
  constexpr int NG = (CPL + SEGG - 1) / SEGG;  // barrier groups per pass
  auto sbuf = [&](int pass, int k) { return seg[((pass * NG + k / SEGG) & 1) * SEGG + k % SEGG]; };
  float a2[RW];
#pragma unroll
  for (int j = 0; j < RW; ++j) a2[j] = 0.0f;
#pragma unroll
  for (int k = 0; k < CPL; ++k) {
    if (nrows > 0) {
      float v[8];
      const bool in = wr.lane + 64 * k < nch;
#pragma unroll
      for (int j = 0; j < RW; ++j) {
        if (j < nrows) {
          float q[8];
          sq_chunk<GT, EPS>(raw[j][k], mu[j], gc, e1, q);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (RAG && k == CPL - 1) a2[j] = a2[j] + (i < vc ? q[i] : 0.0f);
            else if (in) a2[j] = a2[j] + q[i];
            v[i] = j == 0 ? q[i] : v[i] + q[i];
          }
        }
      }
      seg_put(sbuf(0, k), wr.w, wr.lane, v);
    }
    if (k % SEGG == SEGG - 1 || k == CPL - 1) {
      lds_barrier();  // only LDS is handed over; run partials stay with their thread
#pragma unroll
      for (int kk = k - k % SEGG; kk <= k; ++kk)
        seg_fold<RAG>(sbuf(0, kk), nw, (int64_t)kk * 512, C, part, acc, last, tid, racc);
    }
  }
  float wr_inv[RW];  // 1 / row_j (the new row) for the clip partial
#pragma unroll
  for (int j = 0; j < RW; ++j) {
    wr_inv[j] = 0.0f;
    if (j >= nrows) continue;
    const float s2 = wave_csum(a2[j]);
    const float rv = lane_val(row_old, j);
    const float nr = klerp(rv, div_r64(s2, rc), hp.w2);
    if (wr.lane == 0) G(T.row)[wr.rb + j] = nr;
    wr_inv[j] = 1.0f / nr;
  }
  if (!clip_alg(hp, mode)) return;
  // The clip's second column partial, t = (G * G) / row (no eps1: rows of
  // zeros add nothing), from the registers (GC'd in place by the first pass),
  // in the same wave-group / slice / run order.  The LDS segment buffers keep
  // alternating from the first pass's.
#pragma unroll
  for (int k = 0; k < CPL; ++k) {
    if (nrows > 0) {
      float v[8];
#pragma unroll
      for (int j = 0; j < RW; ++j) {
        if (j < nrows) {
          float q[8];
          sq_plain<GT>(raw[j][k], q);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float t = q[i] * wr_inv[j];
            v[i] = j == 0 ? t : v[i] + t;
          }
        }
      }
      seg_put(sbuf(1, k), wr.w, wr.lane, v);
    }
    if (k % SEGG == SEGG - 1 || k == CPL - 1) {
      lds_barrier();
#pragma unroll
      for (int kk = k - k % SEGG; kk <= k; ++kk) {
        if (REG2)
          seg_fold_reg<RAG>(sbuf(1, kk), nw, (int64_t)kk * 512, C, part2, acc, last, tid, rr2[2 * kk], rr2[2 * kk + 1]);
        else
          seg_fold<RAG>(sbuf(1, kk), nw, (int64_t)kk * 512, C, part2, acc, last, tid, racc2);
      }
    }
  }
}

// Row class 0: 1-4 chunks per lane, 1 class 1: 5-10, class 2: 11-24; the
// body is specialized on the exact chunks per lane and its rows per wave
// group (RW = max(1, KAON_ROW_BUDGET / CPL)).
#define KAON_COMMA ,
#define KAON_PF_SWITCH(CLS, BODY, X, ...)                                                      \
  switch (cpl) {                                                                                \
    case 1: if (CLS == 0) BODY<1, 20 X>(__VA_ARGS__); break;                                   \
    case 2: if (CLS == 0) BODY<2, 10 X>(__VA_ARGS__); break;                                   \
    case 3: if (CLS == 0) BODY<3, 6 X>(__VA_ARGS__); break;                                    \
    case 4: if (CLS == 0) BODY<4, 5 X>(__VA_ARGS__); break;                                    \
    case 5: if (CLS == 1) BODY<5, 4 X>(__VA_ARGS__); break;                                    \
    case 6: if (CLS == 1) BODY<6, 3 X>(__VA_ARGS__); break;                                    \
    case 7: if (CLS == 1) BODY<7, 2 X>(__VA_ARGS__); break;                                    \
    case 8: if (CLS == 1) BODY<8, 2 X>(__VA_ARGS__); break;                                    \
    case 9: if (CLS == 1) BODY<9, 2 X>(__VA_ARGS__); break;                                    \
    case 10: if (CLS == 1) BODY<10, 2 X>(__VA_ARGS__); break;                                  \
    case 11: if (CLS == 2) BODY<11, 1 X>(__VA_ARGS__); break;                                  \
    case 12: if (CLS == 2) BODY<12, 1 X>(__VA_ARGS__); break;                                  \
    case 13: if (CLS == 2) BODY<13, 1 X>(__VA_ARGS__); break;                                  \
    case 14: if (CLS == 2) BODY<14, 1 X>(__VA_ARGS__); break;                                  \
    case 15: if (CLS == 2) BODY<15, 1 X>(__VA_ARGS__); break;                                  \
    case 16: if (CLS == 2) BODY<16, 1 X>(__VA_ARGS__); break;                                  \
    case 17: if (CLS == 2) BODY<17, 1 X>(__VA_ARGS__); break;                                  \
    case 18: if (CLS == 2) BODY<18, 1 X>(__VA_ARGS__); break;                                  \
    case 19: if (CLS == 2) BODY<19, 1 X>(__VA_ARGS__); break;                                  \
    case 20: if (CLS == 2) BODY<20, 1 X>(__VA_ARGS__); break;                                  \
    case 21: if (CLS == 2) BODY<21, 1 X>(__VA_ARGS__); break;                                  \
    case 22: if (CLS == 2) BODY<22, 1 X>(__VA_ARGS__); break;                                  \
    case 23: if (CLS == 2) BODY<23, 1 X>(__VA_ARGS__); break;                                  \
    case 24: if (CLS == 2) BODY<24, 1 X>(__VA_ARGS__); break;                                  \
  }

template <int CLS, int GT, int EPS, bool REG2, bool RAG>
__device__ __forceinline__ void pf_stats_run(const KaonTensor& T, const KaonItem& it, const Ws& ws,
                                             const KaonHyper& hp, int mode, float (*seg)[4][512], float* racc,
                                             float* racc2) {
  const int cpl = (int)((((T.C + 7) >> 3) + 63) >> 6);
  KAON_G float* part = run_part(ws, T, it);
  KAON_G float* part2 = part + (int64_t)T.ngroups * T.C;
  const int nsl = run_slices(it);
  float rr2[48];
#pragma unroll
  for (int i = 0; i < 48; ++i) rr2[i] = 0.0f;
#pragma clang loop unroll(disable)
  for (int sl = 0; sl < nsl; ++sl) {
    if (sl > 0 && mode == 0) lds_barrier();  // the LDS fold buffers are reused
    const KaonItem si = slice_item(it, sl);
    KAON_PF_SWITCH(CLS, pf_stats_body, KAON_COMMA GT KAON_COMMA EPS KAON_COMMA REG2 KAON_COMMA RAG, T, si, ws, hp, mode,
                   seg, part, sl > 0, sl + 1 == nsl, racc, part2, racc2, rr2)
  }
}

// Short rows (at most 16 chunks, RW = 20 rows per wave group): the run's rows
// as a grid of L = 2^ceil(log2(chunks)) lanes per row over the whole workgroup,
// NS slices at a time, each thread loading its (at most five) chunks at once.
// A row per wave kept 2 of 64 lanes busy on rows of 16 elements: the adapters of
// a UNet (758 pairs [16, in], [out, 16], 44 M params) took 423 us in this class,
// 64 us so; 512 fp32 tensors of [8, 16] 9.7 -> 6.6 us.  The row sums
// are the lane group's butterfly; the squares go through LDS, where one thread
// per (wave group, column) adds the group's 20 rows in row order and one thread
// per column folds the groups, slices and run in their order: every sum in the
// order of k_stats.
//
// The canonical row sum of a row held by an aligned group of 2^lsh lanes (lane
// cl of the group holding the sum of its chunk cl, 0 past the row's chunks): the
// 64-lane butterfly of the one-row-per-wave layout adds, at offsets 32 ...
// 2^lsh, only the +0 of lanes past the row, which leaves each lane sum x as
// x + 0 (-0 becomes +0); its offsets 2^(lsh-1) ... 1 pair lanes of the group.
__device__ __forceinline__ float group_csum(float a, int lsh) {
  float v = a + 0.0f;
  for (int o = (1 << lsh) >> 1; o >= 1; o >>= 1) v = v + __shfl_xor(v, o, 64);
  return v;
}
// Longest row of the short-row body: 80 rows (a slice) of 16 chunks fill its 40 KB
// tile, the LDS that four workgroups per CU leave each.
constexpr int kThinChunks = 16;
constexpr int kThinTile = 80 * 16 * 8;      // floats of its LDS tile (80 rows of 16 chunks)
template <int GT, int EPS>
__device__ __forceinline__ void thin_stats(const KaonTensor& T, const KaonItem& it, const Ws& ws,
                                           const KaonHyper& hp, int mode, float* tile) {
  constexpr int ES = GT == KAON_F32 ? 4 : 2;
  const int C = (int)T.C;
  const int nch = (C + 7) >> 3;
  const int lsh = nch <= 1 ? 0 : 32 - __builtin_clz((uint32_t)(nch - 1));
  const int Cp = 8 * nch;
  const int batch = 80 * (nch <= 4 ? 4 : nch <= 8 ? 2 : 1);  // rows per pass: batch * 2^lsh <= 5 * 256
  const bool gc = (hp.flags & KAON_F_GC) != 0;
  if (mode == 1 && !gc) return;
  const bool alg = clip_alg(hp, mode);
  const float e1 = (hp.flags & KAON_F_EPS) ? hp.eps1 : 0.0f;
  const double rc = rcp64((float)C);
  const KAON_G uint8_t* g = (const KAON_G uint8_t*)G((const uint8_t*)ws.src(T, hp.flags));
  KAON_G float* part = run_part(ws, T, it);
  KAON_G float* part2 = part + (int64_t)T.ngroups * C;
  KAON_G float* mu_arr = ws.mu(T);
  const int tid = (int)threadIdx.x, cl = tid & ((1 << lsh) - 1), rstep = KAON_WG >> lsh;
  const int cnt = max(0, min(8, C - 8 * cl));
  float racc = 0.0f, racc2 = 0.0f;
#pragma clang loop unroll(disable)
  for (int b0 = 0; b0 < it.nrows; b0 += batch) {
    const int nr = min(batch, it.nrows - b0);
    const int64_t row0 = (int64_t)it.row0 + b0;
    const int K = (nr + rstep - 1) / rstep;  // passes over the lane grid (workgroup-uniform)
    Raw<GT> raw[5];
    float old[5];
    // loads, all issued first: rows past the batch read the first row
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const int rr = (tid >> lsh) + k * rstep;
      const int64_t r = row0 + (rr < nr ? rr : 0);
      const int64_t e0 = r * C + 8 * min(cl, nch - 1);
      if (k < K) {
        if (T.n >= 8) {
          ld_raw<GT, true>(raw[k], g + ES * min(e0, T.n - 8));
        } else {
#pragma unroll
          for (int i = 0; i < gt_words<GT>(); ++i) raw[k].w[i] = 0u;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (e0 + i >= T.n) continue;
            if constexpr (GT == KAON_F32) raw[k].w[i] = ((const KAON_G uint32_t*)g)[e0 + i];
            else raw[k].w[i >> 1] |= (uint32_t)((const KAON_G uint16_t*)g)[e0 + i] << (16 * (i & 1));
          }
        }
        old[k] = mode == 0 ? T.row[r] : 0.0f;
      }
    }
    float winv[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      if (k >= K) continue;
      const int rr = (tid >> lsh) + k * rstep;
      const bool rv = rr < nr;
      const int64_t r = row0 + (rv ? rr : 0);
      if (T.n >= 8) {
        const int64_t e0 = r * C + 8 * min(cl, nch - 1);
        const int d = (int)(e0 - min(e0, T.n - 8));
        if (__builtin_amdgcn_ballot_w64(d > 0)) {  // the tensor's last chunk, one element at a time
          for (int s = 1; s < 8; ++s) {
            const Raw<GT> v = raw_down<GT>(raw[k], 1);
            if (d >= s) raw[k] = v;
          }
        }
      }
      float x[8], q[8], a = 0.0f;
      raw_floats<GT>(raw[k], x);
      const int m = rv ? cnt : 0;
      if (gc) {
#pragma unroll
        for (int i = 0; i < 8; ++i) a = a + (i < m ? x[i] : 0.0f);
        const float mu = round_to<GT>(div_r64(group_csum(a, lsh), rc));
        if (rv && cl == 0) mu_arr[r] = mu;
        sq_chunk<GT, EPS>(raw[k], mu, true, e1, q);
      } else {
        sq_chunk<GT, EPS>(raw[k], 0.0f, false, e1, q);
      }
      if (mode == 1) continue;
      float a2 = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) a2 = a2 + (i < m ? q[i] : 0.0f);
      const float s2 = group_csum(a2, lsh);
      const float nrow = klerp(old[k], div_r64(s2, rc), hp.w2);
      if (rv && cl == 0) T.row[r] = nrow;
      winv[k] = 1.0f / nrow;
      if (m > 0) {
        kf4* d = (kf4*)(tile + rr * Cp + 8 * cl);
        d[0] = kf4{q[0], q[1], q[2], q[3]};
        d[1] = kf4{q[4], q[5], q[6], q[7]};
      }
    }
    if (mode == 1) continue;
    const int ng = (nr + 19) / 20;  // wave groups of the pass
    auto fold = [&](float& acc) {
      __syncthreads();
      for (int p = tid; p < ng * C; p += KAON_WG) {
        const int gi = p / C, j = p - gi * C;
        float* t = tile + gi * 20 * Cp + j;
        const int nrow = min(20, nr - gi * 20);
        float s = t[0];
        if (nrow == 20) {
#pragma unroll
          for (int i = 1; i < 20; ++i) s = s + t[i * Cp];
        } else {
          for (int i = 1; i < nrow; ++i) s = s + t[i * Cp];
        }
        t[0] = s;  // read by this thread only until the barrier
      }
      __syncthreads();
      if (tid < C) {
        for (int sg = 0; sg < ng; sg += 4) {
          float s = tile[sg * 20 * Cp + tid];
          for (int k = 1; k < 4 && sg + k < ng; ++k) s = s + tile[(sg + k) * 20 * Cp + tid];
          acc = b0 == 0 && sg == 0 ? s : acc + s;
        }
      }
      __syncthreads();  // the tile is written again
    };
    fold(racc);
    if (!alg) continue;
    // the clip's second column partial, t = (G * G) / row (the new row; no eps1)
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      if (k >= K) continue;
      const int rr = (tid >> lsh) + k * rstep;
      if (rr < nr && cnt > 0) {
        float q[8];
        sq_plain<GT>(raw[k], q);
        kf4* d = (kf4*)(tile + rr * Cp + 8 * cl);
        d[0] = kf4{q[0] * winv[k], q[1] * winv[k], q[2] * winv[k], q[3] * winv[k]};
        d[1] = kf4{q[4] * winv[k], q[5] * winv[k], q[6] * winv[k], q[7] * winv[k]};
      }
    }
    fold(racc2);
  }
  if (mode == 0 && tid < C) {
    part[tid] = racc;
    if (alg) part2[tid] = racc2;
  }
}

// The run's tensor, unless KProdigy steps it in its own pass-1 kernels (a
// per-element v, block factoring); clears what phase 5 accumulates.
__device__ __forceinline__ bool stats_begin(const KaonTensor& T, const KaonItem& it, const Ws& ws, const KaonHyper& hp) {
  if (T.full_v || T.fb_r) return false;
  zero_accumulators(T, it, ws, hp.codec);
  return true;
}

// Classes 0 and 1 are held to 4 waves per SIMD (128 VGPRs).  Every class
// keeps its run partial in LDS (rows of at most 2048, 5120 and 12288
// elements) and stores it once per run.  The clip's second run partial is
// kept in LDS too in class 0, accumulated in the workspace in class 1 (in
// registers it would cost class 1 a wave per SIMD, measured slower) and kept
// in registers in class 2, whose LDS already limits it to 2 waves per SIMD.
// The short rows of class 0 (thin_stats) use the same LDS, 40 KB of the 40 that
// four workgroups per CU leave each.
template <int CLS, int EPS>
__global__ __launch_bounds__(KAON_WG, 4) void k_pf_stats(const KaonTensor* __restrict__ D,
                                                         const KaonItem* __restrict__ items, Ws ws, KaonHyper hp,
                                                         int mode) {
  constexpr int kAcc = CLS == 0 ? 4 * 512 : 10 * 512;
  __shared__ __attribute__((aligned(16))) float lds[CLS == 0 ? kThinTile : 4096 + kAcc];
  const KaonItem it = items[blockIdx.x];
  const KaonTensor& T = D[it.tensor];
  if (!stats_begin(T, it, ws, hp)) return;
  if constexpr (CLS == 0) {
    if (T.C <= 8 * kThinChunks) {
      thin_stats<KAON_BF16, EPS>(T, it, ws, hp, mode, lds);
      return;
    }
  }
  pf_stats_run<CLS, KAON_BF16, EPS, false, false>(T, it, ws, hp, mode, (float(*)[4][512])lds, lds + 4096,
                                                  CLS == 0 ? lds + 4096 + kAcc : nullptr);
}
template <int EPS>
__global__ __launch_bounds__(KAON_WG) void k_pf_stats_wide(const KaonTensor* __restrict__ D,
                                                           const KaonItem* __restrict__ items, Ws ws, KaonHyper hp,
                                                           int mode) {
  __shared__ __attribute__((aligned(16))) float seg[4][4][512];  // two buffer sets of two segments
  __shared__ __attribute__((aligned(16))) float racc[24 * 512];
  const KaonItem it = items[blockIdx.x];
  const KaonTensor& T = D[it.tensor];
  if (!stats_begin(T, it, ws, hp)) return;
  pf_stats_run<2, KAON_BF16, EPS, true, false>(T, it, ws, hp, mode, seg, racc, nullptr);
}
// Lion's row means alone (mode 1): the rows' loads and one butterfly each.  The UNet set
// (2.66 G params): class 0 takes 622 us in the kernel above, where the registers and LDS
// of the sums and of the short rows are held too, 595 here.
template <int CLS>
__global__ __launch_bounds__(KAON_WG, CLS == 2 ? 2 : 4) void k_pf_mean(
    const KaonTensor* __restrict__ D, const KaonItem* __restrict__ items, Ws ws, KaonHyper hp, int) {
  const KaonItem it = items[blockIdx.x];
  const KaonTensor& T = D[it.tensor];
  if (!stats_begin(T, it, ws, hp)) return;
  if constexpr (CLS == 0) {
    if (T.C <= 8 * kThinChunks) {
      thin_stats<KAON_BF16, 1>(T, it, ws, hp, 1, nullptr);
      return;
    }
  }
  pf_stats_run<CLS, KAON_BF16, 1, CLS == 2, false>(T, it, ws, hp, 1, nullptr, nullptr, nullptr);
}
// Classes 3-5 (CLS - 3 as above): the rows of any type, length and alignment.
// fp32 rows take twice the registers: 2 waves per SIMD.
template <int GT, int CLS>
__global__ __launch_bounds__(KAON_WG, GT == KAON_F32 || CLS == 5 ? 2 : 3) void k_rag_stats(
    const KaonTensor* __restrict__ D, const KaonItem* __restrict__ items, Ws ws, KaonHyper hp, int mode) {
  constexpr int kSegs = CLS == 5 ? 16 * 512 : 8 * 512, kAcc = CLS == 3 ? 4 * 512 : CLS == 4 ? 10 * 512 : 24 * 512;
  __shared__ __attribute__((aligned(16))) float lds[CLS == 3 ? kThinTile : kSegs + kAcc];
  const KaonItem it = items[blockIdx.x];
  const KaonTensor& T = D[it.tensor];
  if (!stats_begin(T, it, ws, hp)) return;
  if constexpr (CLS == 3) {
    if (T.C <= 8 * kThinChunks) {
      thin_stats<GT, 2>(T, it, ws, hp, mode, lds);
      return;
    }
  }
  pf_stats_run<CLS - 3, GT, 2, CLS == 5, true>(T, it, ws, hp, mode, (float(*)[4][512])lds, lds + kSegs,
                                                 CLS == 3 ? lds + kSegs + kAcc : nullptr);
}

#undef KAON_PF_SWITCH
#undef KAON_COMMA

template <int GT>
StatsFn rag_fn(int cls) {
  switch (cls) {
    case 3: return k_rag_stats<GT, 3>;
    case 4: return k_rag_stats<GT, 4>;
    case 5:  // planned for bf16 gradients only
      if constexpr (GT == KAON_BF16) return k_rag_stats<GT, 5>;
  }
  return nullptr;
}

}  // namespace

// One object per gradient type of the classes 3-5, one for the rest (the build
// compiles them side by side).
namespace kaon {
#if KAON_STATS_PART == 1
StatsFn rag_bf16(int cls) { return rag_fn<KAON_BF16>(cls); }
#elif KAON_STATS_PART == 2
StatsFn rag_f16(int cls) { return rag_fn<KAON_F16>(cls); }
#elif KAON_STATS_PART == 3
StatsFn rag_f32(int cls) { return rag_fn<KAON_F32>(cls); }
#else
namespace {
// fused: eps1 is 0 or at least 2^-100 (sq1)
StatsFn pf_fn(int cls, bool fused) {
  switch (cls) {
    case 0: return fused ? k_pf_stats<0, 1> : k_pf_stats<0, 2>;
    case 1: return fused ? k_pf_stats<1, 1> : k_pf_stats<1, 2>;
    case 2: return fused ? k_pf_stats_wide<1> : k_pf_stats_wide<2>;
  }
  return nullptr;
}
StatsFn mean_fn(int cls) { return cls == 0 ? k_pf_mean<0> : cls == 1 ? k_pf_mean<1> : k_pf_mean<2>; }
// The register variants (classes 3-5) only for KProdigy's coupled decay.
template <int GT>
StatsFn streamed_fn(int cls) {
  switch (cls) {
    case 3: return k_stats<GT, 4>;
    case 4: return k_stats<GT, 10>;
    case 5:  // planned for bf16 gradients only
      if constexpr (GT == KAON_BF16) return k_stats<GT, 24>;
      return nullptr;
    case 6: return k_stats<GT, 0>;
  }
  return nullptr;
}
// coupled: KProdigy's decay inside the gradient (k_stats for every row length)
StatsFn stats_fn(int gt, int cls, bool fused, bool coupled) {
  if (cls < 3 && !coupled) return gt == KAON_BF16 ? pf_fn(cls, fused) : nullptr;
  if (cls < 6 && !coupled) return gt == KAON_F16 ? rag_f16(cls) : gt == KAON_BF16 ? rag_bf16(cls) : rag_f32(cls);
  if (cls < 3) cls += 3;
  return gt == KAON_F16 ? streamed_fn<KAON_F16>(cls) : gt == KAON_BF16 ? streamed_fn<KAON_BF16>(cls) : streamed_fn<KAON_F32>(cls);
}
}  // namespace

// Phase-1 launches, one per register class run (slices are sorted by class).
// KProdigy's coupled decay reads p beside g (k_stats): the same sums, the row
// classes 0-2 as the classes 3-5 of the same chunks per lane.
const char* launch_stats(const KaonLaunch& L, Ws ws, const KaonHyper& hp, int mode, hipStream_t st) {
  // k_stats's dynamic LDS: one slice column partial
  constexpr int kClassMaxC[KAON_ROW_CLASSES] = {4 * 512, 10 * 512, 24 * 512, 4 * 512, 10 * 512, 24 * 512, kSeg};
  int32_t off = 0;
  const bool coupled = mode == 0 && (hp.flags & KAON_F_PD_COUPLED) != 0;
  for (int cls = 0; cls < KAON_ROW_CLASSES; ++cls) {
    const int32_t cnt = L.row_runs[cls];
    if (cnt <= 0) continue;
    if (cls < 3 && hp.g_dtype != KAON_BF16) return "kaon: prefetching row class planned for non-bf16 grads";
    const bool fused = !(hp.flags & KAON_F_EPS) || hp.eps1 == 0.0f || hp.eps1 >= 0x1p-100f;
    StatsFn fn = mode == 1 && cls < 3 ? mean_fn(cls) : stats_fn(hp.g_dtype, cls, fused, coupled);
    if (!fn) return "kaon: no row-statistics kernel for this grad dtype and row class";
    const size_t lds = mode == 0 && (coupled || cls == 6) ? sizeof(float) * (size_t)kClassMaxC[cls] : 0;
    hipLaunchKernelGGL(fn, dim3(cnt), dim3(KAON_WG), lds, st, L.descs, L.row_items + off, ws, hp, mode);
    off += cnt;
  }
  if (off != L.n_row_items) return "kaon: slice class runs do not add up to n_row_items";
  return nullptr;
}

#endif
}  // namespace kaon
