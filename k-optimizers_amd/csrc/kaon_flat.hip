// kaon_flat.hip -- phases 5 and 6 (keep count + momentum absmax, apply) for
// everything outside the specialized kernels of kaon_fast.hip: fp32 and fp16
// params, fp32 gradients, RN and kahan writes, fp32 momenta, 4-bit blocks of any
// size, rows that start at any alignment and 1-D tensors; and any slice of the
// specialized kernels whose configuration has no compiled variant.  Semantics per
// element: src/kaon/adakaon.py:968-1014, src/kaon/lion.py:454-485,
// src/kaon/msam.py:202-235, src/kaon/adapnm.py:1209-1275,
// src/kaon/adamuon.py:557-593.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kaon_common.h"

using namespace kaon;

namespace {

// Rows a slice can hold: 4 waves of 20 rows, or of 24 for the specialized
// kernel's slices (rounded up to a multiple of 8); a chunk that starts in the
// slice's last row can reach 7 rows further (rows of one element).
constexpr int kMaxRows = 4 * 24 + 8;

// Words of a chunk (8 elements) of a stored type / momentum codec.
template <int DT>
constexpr int dt_words() {
  return DT == KAON_F32 ? 8 : 4;
}
template <int CODEC>
constexpr int mom_words() {
  return CODEC == KAON_MOM_F32 ? 8 : CODEC == KAON_MOM_BF16 ? 4 : CODEC == KAON_MOM_INT8 ? 2 : 1;
}

// NW words at a chunk's address, at any alignment: 16-, 8- or 4-byte accesses when
// `vec` (the chunk is whole), otherwise byte by byte, `nbytes` of them (the rest
// reads as 0 / is not written).
template <int NW>
__device__ __forceinline__ void ld_words(const KAON_G uint8_t* a, bool vec, int nbytes, uint32_t (&w)[NW]) {
  if (vec) {
    if constexpr (NW == 1) {
      w[0] = __builtin_nontemporal_load((const KAON_G ku1_any*)a);
    } else if constexpr (NW == 2) {
      const ku2 v = __builtin_nontemporal_load((const KAON_G ku2_any*)a);
      w[0] = v.x;
      w[1] = v.y;
    } else {
#pragma unroll
      for (int k = 0; k < NW / 4; ++k) {
        const KAON_G ku4_any* q = (const KAON_G ku4_any*)a + k;
        const ku4 v = NW == 4 ? __builtin_nontemporal_load(q) : *q;
        w[4 * k] = v.x;
        w[4 * k + 1] = v.y;
        w[4 * k + 2] = v.z;
        w[4 * k + 3] = v.w;
      }
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    w[k] = 0u;
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (4 * k + b < nbytes) w[k] |= (uint32_t)a[4 * k + b] << (8 * b);
  }
}
template <int NW>
__device__ __forceinline__ void st_words(KAON_G uint8_t* a, bool vec, int nbytes, const uint32_t (&w)[NW]) {
  if (vec) {
    if constexpr (NW == 1) {
      __builtin_nontemporal_store(w[0], (KAON_G ku1_any*)a);
    } else if constexpr (NW == 2) {
      __builtin_nontemporal_store(ku2{w[0], w[1]}, (KAON_G ku2_any*)a);
    } else {
#pragma unroll
      for (int k = 0; k < NW / 4; ++k) {
        const ku4 v = ku4{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
        if (NW == 4) __builtin_nontemporal_store(v, (KAON_G ku4_any*)a + k);
        else ((KAON_G ku4_any*)a)[k] = v;
      }
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < NW; ++k)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (4 * k + b < nbytes) a[4 * k + b] = (uint8_t)(w[k] >> (8 * b));
}

template <int DT>
__device__ __forceinline__ void unpack_dt(const uint32_t (&w)[dt_words<DT>()], float o[8]) {
  if constexpr (DT == KAON_F32) {
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = __uint_as_float(w[i]);
  } else if constexpr (DT == KAON_BF16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = __uint_as_float(w[i] << 16);
      o[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = h2f(w[i] & 0xFFFFu);
      o[2 * i + 1] = h2f(w[i] >> 16);
    }
  }
}
// Eight values already rounded to DT, as stored.
template <int DT>
__device__ __forceinline__ void pack_dt(const float x[8], uint32_t (&w)[dt_words<DT>()]) {
  if constexpr (DT == KAON_F32) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = __float_as_uint(x[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = f2lp<DT>(x[2 * i]) | (f2lp<DT>(x[2 * i + 1]) << 16);
  }
}
// fp32 -> bf16 / fp16 storage (RNE, NaN canonical).
template <int DT>
__device__ __forceinline__ void pack_lp(const float x[8], uint32_t (&w)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = f2lp<DT>(x[2 * i]) | (f2lp<DT>(x[2 * i + 1]) << 16);
}
// A rounding to DT whose NaN payload is not observed (pairs: one instruction in bf16).
template <int DT>
__device__ __forceinline__ void round8(float x[8]) {
#pragma unroll
  for (int i = 0; i < 8; i += 2) round_pair<DT>(x[i], x[i + 1]);
}

// A lane's chunk of a window: clamped into the slice, so that its loads are
// unconditional.
struct Pos {
  int64_t wb;   // the window's first element (wave-uniform)
  uint32_t lo;  // the chunk's first element in the window
  uint32_t r, j0;  // its row (relative to the slice) and column
  int cnt;      // existing elements (0 for a lane outside the slice)
  bool vec;     // wave-uniform: whole chunks
};

// What a chunk reads from memory, loaded a window ahead of its arithmetic.
template <int OPT, int PHASE, int PT, int GT, int CODEC>
struct FlatIn {
  uint32_t g[dt_words<GT>()], p[dt_words<PT>()], m[mom_words<CODEC>()], n[mom_words<CODEC>()], o[4], sh[4];
  float f[8];
};

// A tensor's values, read from its descriptor once per workgroup.
struct FlatCtx {
  const KAON_G uint8_t *g, *p, *m, *n, *o, *sh, *f;
  const KAON_G uint8_t *msc, *nsc;  // scales of m (per row or block), of AdaPNM's negative buffer
  const uint16_t* nz[3];
  uint32_t tid;
  bool factored;
};

// Bytes of `cnt` (<= 8) elements of a momentum codec.
template <int CODEC>
__host__ __device__ constexpr int mom_bytes(int cnt) {
  return CODEC == KAON_MOM_F32 ? 4 * cnt : CODEC == KAON_MOM_BF16 ? 2 * cnt : CODEC == KAON_MOM_INT8 ? cnt : (cnt + 1) / 2;
}

// Which streams a kernel reads.  XF: phase 5 reads the weights (weight decay);
// phase 6 writes through the kahan compensation.
template <int OPT, int PHASE, int CODEC, bool XF>
struct FlatCfg {
  static constexpr bool PNM = OPT == KAON_OPT_ADAPNM, MUON = OPT == KAON_OPT_ADAMUON, LION = OPT == KAON_OPT_LION;
  static constexpr bool INT8 = CODEC == KAON_MOM_INT8, Q4 = CODEC == KAON_MOM_4BIT, QUANT = INT8 || Q4;
  static constexpr bool NEEDP = PHASE == 6 || (XF && !PNM);
  static constexpr bool KAHAN = PHASE == 6 && XF;
  // AdaMuon's momentum is the raw grad's: float codecs were stored by the
  // momentum pass; int8 / 4-bit codes are requantized here in phase 6
  static constexpr bool MOM = CODEC != KAON_MOM_NONE && (!MUON || (PHASE == 6 && QUANT));
  // phase 5 takes the absmax of the new momentum, except where an earlier pass did
  static constexpr bool ABSMAX = PHASE == 5 && QUANT && MOM && !PNM && !MUON;
};

// VEC: the slice's chunks are whole and the tensor is factored, so that no load sits behind a branch: a load in a branch, or one
// whose successors are conditional, would make the compiler wait for every load
// in flight at its use, the next window's included.
template <int OPT, int PHASE, int PT, int GT, int CODEC, bool XF, bool VEC>
__device__ __forceinline__ void flat_load(FlatIn<OPT, PHASE, PT, GT, CODEC>& in, const FlatCtx& X, const Pos& q) {
  using F = FlatCfg<OPT, PHASE, CODEC, XF>;
  constexpr int GB = GT == KAON_F32 ? 4 : 2, PB = PT == KAON_F32 ? 4 : 2, MB = mom_bytes<CODEC>(8);
  const bool vec = VEC || q.vec;
  const int cnt = q.cnt;
  ld_words(X.g + GB * q.wb + GB * q.lo, vec, GB * cnt, in.g);
  if constexpr (F::NEEDP) ld_words(X.p + PB * q.wb + PB * q.lo, vec, PB * cnt, in.p);
  if constexpr (F::MOM) ld_words(X.m + MB * (q.wb >> 3) + MB * (q.lo >> 3), vec, mom_bytes<CODEC>(cnt), in.m);
  if constexpr (F::PNM) ld_words(X.n + MB * (q.wb >> 3) + MB * (q.lo >> 3), vec, mom_bytes<CODEC>(cnt), in.n);
  if constexpr (F::MUON) ld_words(X.o + 2 * q.wb + 2 * q.lo, vec, 2 * cnt, in.o);
  if constexpr (F::KAHAN) ld_words(X.sh + 2 * q.wb + 2 * q.lo, vec, 2 * cnt, in.sh);
  if constexpr (!F::LION) {
    if (VEC || X.factored) {
      // the column factors wrap around past C (put_cf), so a chunk that runs
      // into the next row reads on; 4-byte aligned
      typedef kf4 kf4u __attribute__((aligned(4)));
      const KAON_G kf4u* c = (const KAON_G kf4u*)(X.f + 4 * (uint64_t)q.j0);
      const kf4 a = c[0], b = c[1];
      in.f[0] = a.x; in.f[1] = a.y; in.f[2] = a.z; in.f[3] = a.w;
      in.f[4] = b.x; in.f[5] = b.y; in.f[6] = b.z; in.f[7] = b.w;
    } else {
      uint32_t w[8];
      ld_words(X.f + 4 * q.wb + 4 * q.lo, vec, 4 * cnt, w);
#pragma unroll
      for (int i = 0; i < 8; ++i) in.f[i] = __uint_as_float(w[i]);
    }
  }
}

// Phases 5 and 6 over a slice, by flat chunks: the slice's elements are
// contiguous, so its waves walk it in windows of 64 aligned 8-element chunks
// whatever the row length, each chunk going to the slice that holds its first
// element.  Every stream is then 16-byte accesses, one Philox draw serves a
// chunk and every lane has a whole chunk, where a row-by-row walk leaves
// lanes idle past each row's end (rows of 16 elements: 62 of 64), reads
// odd-length rows element by element and draws Philox once per element.
// Row values come from LDS, read there once per slice.  A chunk inside one row
// takes them as one set (STR false); a window in which some lane's chunk runs
// into the next row looks them up per element (STR true).  The keep count and
// the int8 row / 4-bit block absmax do not depend on the order.
//
// Bound by HBM where the rows are aligned: fp32 params and gradients with bf16
// momentum, 123.6 M params: apply 516 -> 490 us (20 B/param, 5.05 TB/s, the copy
// kernel's rate), keep count 169 -> 129 us; bf16 with kahan writes: 591 -> 410 us
// (16 B/param) and 237 -> 138 us.  Rows of 771 and 2057 bf16 elements with int8
// momentum, 52.2 M params: 420 -> 138 us and 263 -> 74 us (the row-by-row walk in
// front of each arrow).  Streams of 32 bytes per chunk (fp32) are ordinary
// accesses (the apply took 578 us with non-temporal stores of two 16-byte halves
// with a stride of 32, 490 so).  Storage that is not 16-byte aligned takes the same
// accesses (whole steps with the gradients one element into their storage, read
// byte by byte before the arrow: fp32, 58 M params, 1313 -> 442 us, aligned 433;
// bf16 kahan 1167 -> 431, aligned 391; the odd rows 765 -> 345, aligned 335; plain
// instead of non-temporal accesses 462, 428 and 333, but 454, 405 and 321 aligned).
// Phase 5 fits 4 waves per SIMD (128 VGPRs); the apply spills
// there (int8 201 us), so it takes 3.
template <int OPT, int PHASE, int PT, int GT, int CODEC, bool XF>
__global__ __launch_bounds__(KAON_WG, PHASE == 5 ? 4 : 3) void k_flat(const KaonTensor* __restrict__ D,
                                                     const KaonItem* __restrict__ items, Ws ws, KaonHyper hp) {
  using F = FlatCfg<OPT, PHASE, CODEC, XF>;
  constexpr bool PNM = F::PNM, MUON = F::MUON, LION = F::LION, INT8 = F::INT8, Q4 = F::Q4;
  constexpr bool MOM = F::MOM, ABSMAX = F::ABSMAX, NEEDP = F::NEEDP, KAHAN = F::KAHAN;
  constexpr bool LOWP = PT == KAON_BF16;
  using In = FlatIn<OPT, PHASE, PT, GT, CODEC>;
  __shared__ kf4 row4[kMaxRows];                      // mu, r, the old scale, the new scale
  __shared__ double rowr[INT8 ? kMaxRows : 1];        // 1 / new scale
  __shared__ float rown[PNM && INT8 ? kMaxRows : 1];  // AdaPNM: the negative buffer's scale
  __shared__ uint32_t smax[INT8 ? kMaxRows : 1];
  __shared__ uint32_t keep_s[4];
  const KaonItem it = items[blockIdx.x];
  const KaonTensor& T = D[it.tensor];
  if (PNM && PHASE == 5 && !keep_late(T, ws)) return;
  const int64_t n = T.n;
  const uint32_t C = (uint32_t)T.C;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool factored = T.factored != 0;
  const bool gc = (hp.flags & KAON_F_GC) && factored;
  const bool gcw = PHASE == 6 && gc && (hp.flags & KAON_F_GC_WRITE) && T.gc_write &&
                   (OPT == KAON_OPT_ADAKAON || LION || PNM);
  const bool cautious = (hp.flags & KAON_F_CAUTIOUS) != 0;
  const bool wd = (hp.flags & KAON_F_WD) != 0;
  const bool nk_remove = OPT == KAON_OPT_ADAKAON && MOM && (hp.flags & KAON_F_NK_REMOVE);
  const bool nk_climb = OPT == KAON_OPT_ADAKAON && MOM && (hp.flags & KAON_F_NK_CLIMB);
  const float nf_old = msam_nanfill(hp.nk_bound_old), nf_new = msam_nanfill(hp.nk_bound_new);
  const bool swap = PNM && (hp.step & 1u) == 0u;  // AdaPNM: m is the positive buffer on odd steps
  const uint32_t B = Q4 ? (uint32_t)T.block4 : 8u;
  const int64_t nb = Q4 ? nblocks4(T) : 0;

  FlatCtx X;
  X.g = (const KAON_G uint8_t*)G(T.g);
  X.p = (const KAON_G uint8_t*)G(T.p);
  X.m = (const KAON_G uint8_t*)G(swap ? T.m2 : T.m);
  X.n = (const KAON_G uint8_t*)G(swap ? T.m : T.m2);
  X.msc = (const KAON_G uint8_t*)G(swap ? T.m2_scale : T.m_scale);
  X.nsc = (const KAON_G uint8_t*)G(swap ? T.m_scale : T.m2_scale);
  X.o = MUON ? (const KAON_G uint8_t*)G(ws.mo(T)) : nullptr;
  X.sh = (const KAON_G uint8_t*)G(T.shift);
  X.f = factored ? (const KAON_G uint8_t*)ws.cf(T)
                 : (const KAON_G uint8_t*)G(PNM && (hp.flags & KAON_F_AMS) && T.max_v ? T.max_v : T.v);
#pragma unroll
  for (int s = 0; s < 3; ++s) X.nz[s] = T.noise[s];
  X.tid = (uint32_t)T.tensor_id;
  X.factored = factored;

  // the slice's chunks [cb, ce) and their windows of 64
  const int64_t ebeg = (int64_t)it.row0 * C;
  const int64_t cb = (ebeg + 7) >> 3, ce = (ebeg + (int64_t)it.nrows * C + 7) >> 3;
  const int64_t w0 = cb >> 6, wend = (ce + 63) >> 6;
  const float rcpC = (1.0f / (float)C) * (1.0f - 0x1p-21f);

  auto locate = [&](int64_t win) {
    Pos q;
    q.wb = win << 9;
    const int64_t c0 = win << 6;
    const int lo = max((int)(cb - c0), 0), hi = (int)min<int64_t>(ce - c0, 64) - 1;
    const int cc = min(max(lane, lo), hi);
    q.lo = (uint32_t)cc << 3;
    q.cnt = (int)min<int64_t>(8, n - (q.wb + q.lo));
    q.vec = __builtin_amdgcn_ballot_w64(q.cnt < 8) == 0;
    const uint32_t rel = (uint32_t)(q.wb - ebeg) + q.lo;
    if (it.nrows == 1) {
      q.r = 0u;
      q.j0 = rel;
    } else {
      // floor(rel / C): the estimate is at most one below it (rel / C < kMaxRows, the
      // factor keeps it from going above)
      q.r = (uint32_t)((float)rel * rcpC);
      q.j0 = rel - q.r * C;
      if (q.j0 >= C) {
        q.r += 1u;
        q.j0 -= C;
      }
    }
    if (cc != lane) q.cnt = 0;
    return q;
  };

  // ---- the slice's row values into LDS; phase 5 keeps the old int8 scales for
  // phase 6, which stores the new ones (each row by the slice that owns it)
  const int nctx = (int)min<int64_t>(T.R - it.row0, (int64_t)it.nrows + 8);
  auto load_rows = [&]() {
    for (int k = threadIdx.x; k < nctx; k += KAON_WG) {
      const int64_t r = (int64_t)it.row0 + k;
      kf4 v = kf4{0.0f, 0.0f, 1.0f, 1.0f};
      if (gc) v.x = ws.mu(T)[r];
      if (!LION && factored) v.y = ws.rf(T)[r];
      if (INT8 && MOM) {
        v.z = PHASE == 6 ? ws.roldsc(T)[r] : ((const KAON_G float*)X.msc)[r];
        if (PNM) rown[k] = ((const KAON_G float*)X.nsc)[r];
        if (PHASE == 6) {
          v.w = fmaxf(__uint_as_float(ws.ramax(T)[r]), 1e-12f) / 127.0f;
          rowr[k] = rcp64(v.w);
          if (k < it.nrows) ((KAON_G float*)X.msc)[r] = v.w;
        } else if (ABSMAX && k < it.nrows) {
          ws.roldsc(T)[r] = v.z;
        }
      }
      row4[k] = v;
      if (ABSMAX && INT8) smax[k] = 0u;
    }
  };
  // clip divisor of the tensor, the cautious rescale
  const float fac = !LION ? clip_div(T, ws, hp) : 1.0f;
  const double rfac = rcp64(fac);
  double rden = 1.0;
  if (PHASE == 6 && cautious) {
    const uint32_t cnt = ((const KAON_G uint32_t*)ws.scal(T))[1];
    rden = rcp64(fmaxf((float)cnt / (float)n, 1e-8f));
  }
  const bool wlo = fabsf(hp.w1) < 0.5f;
  const float wlerp = wlo ? hp.w1 : hp.w1 - 1.0f;
  // torch's lerp with the branch of its weight taken once (klerp)
  auto lerp = [&](float a, float b) { return __fmaf_rn(wlerp, b - a, wlo ? a : b); };
  const int bsh = Q4 && (B & (B - 1)) == 0 ? __builtin_ctz(B) : -1;

  uint32_t keep = 0;
  constexpr int GB = GT == KAON_F32 ? 4 : 2, PB = PT == KAON_F32 ? 4 : 2, MB = mom_bytes<CODEC>(8);

  // The rows of a chunk's elements relative to the chunk's own, four bits each.
  auto row_steps = [&](const Pos& q) -> uint32_t {
    if (C >= 8u) return C - q.j0 < 8u ? 0x11111111u << (4u * (C - q.j0)) : 0u;
    uint32_t pk = 0u, rr = 0u, jj = q.j0;
    for (int i = 0; i < 8; ++i) {
      pk |= rr << (4 * i);
      if (++jj == C) {
        jj = 0u;
        ++rr;
      }
    }
    return pk;
  };
  // One chunk: its arithmetic and, in phase 6, its writes.  Returns the |m|
  // maxima (int8: of the chunk's first row and of the next; 4-bit: of its block).
  auto chunk = [&](const In& in, const Pos& q, auto str_c, auto vec_c, auto&& prefetch) -> kaon_f32x2 {
    constexpr bool STR = decltype(str_c)::value, VEC = decltype(vec_c)::value;
    const int cnt = q.cnt;
    const uint32_t e0 = (uint32_t)q.wb + q.lo;  // < 2^32
    const bool vec = VEC || q.vec;
    const uint32_t steps = STR ? row_steps(q) : 0u;
    // elements past the tensor's end stay on its last row
    auto row_i = [&](int i) -> uint32_t {
      return STR ? min(q.r + ((steps >> (4 * i)) & 7u), (uint32_t)nctx - 1u) : q.r;
    };
    float g[8], p[8];
    unpack_dt<GT>(in.g, g);
    if (gc) {
#pragma unroll
      for (int i = 0; i < 8; ++i) g[i] = g[i] - (STR ? row4[row_i(i)].x : row4[q.r].x);
      round8<GT>(g);
    }
    // the centralized gradient over p.grad (already rounded to the grad dtype),
    // before the next window's loads: a conditional store after them would
    // make the wait for those loads cover it too
    if (gcw && cnt > 0) {
      uint32_t gw[dt_words<GT>()];
      pack_dt<GT>(g, gw);
      st_words((KAON_G uint8_t*)X.g + GB * q.wb + GB * q.lo, vec, GB * cnt, gw);
    }
    prefetch();
    if constexpr (NEEDP) unpack_dt<PT>(in.p, p);
    const kf4 rv = row4[q.r];
    const double rnew = INT8 && PHASE == 6 ? rowr[q.r] : 1.0;
    const float ngs = PNM && INT8 ? rown[q.r] : 1.0f;
    // 4-bit: the block of a whole-chunk block size, or of the chunk's first element
    uint32_t blk = 0, woff = 0;
    float b_old = 1.0f, b_new = 1.0f, b_neg = 1.0f;
    double b_r = 1.0;
    const bool walk = Q4 && (B & 7u) != 0;
    auto blk_ctx = [&](uint32_t b) {
      b_old = PHASE == 5 ? ((const KAON_G float*)X.msc)[b] : ws.boldsc(T, nb)[b];
      if (PNM) b_neg = ((const KAON_G float*)X.nsc)[b];
      if (PHASE == 6) {
        b_new = fmaxf(__uint_as_float(ws.bamax(T)[b]), 1e-12f) / 7.0f;
        b_r = rcp64(b_new);
      }
    };
    if constexpr (Q4 && MOM) {
      blk = bsh >= 0 ? e0 >> bsh : e0 / B;
      woff = e0 - blk * B;
      blk_ctx(blk);
    }
    // ---- noise (bf16 weights)
    uint32_t nz0[8], nz1[8], nz2[8];
    if (LOWP && nk_remove && NEEDP) noise8(hp.seed, hp.step, X.tid, 0u, e0, X.nz[0], cnt, nz0);
    if (LOWP && PHASE == 6 && !KAHAN && hp.bf16_method == KAON_SR)
      noise8(hp.seed, hp.step, X.tid, 1u, e0, X.nz[1], cnt, nz1);
    if (LOWP && PHASE == 6 && nk_climb) noise8(hp.seed, hp.step, X.tid, 2u, e0, X.nz[2], cnt, nz2);
    auto code = [&](const uint32_t (&wd_)[mom_words<CODEC>()], int i) -> float {
      if constexpr (INT8) return (float)(int8_t)(uint8_t)(wd_[i >> 2] >> (8 * (i & 3)));
      else if constexpr (Q4) return (float)((wd_[0] >> (4 * i)) & 0xFu) - 8.0f;
      else if constexpr (CODEC == KAON_MOM_F32) return __uint_as_float(wd_[i]);
      else if constexpr (CODEC == KAON_MOM_BF16)
        return (i & 1) ? __uint_as_float(wd_[i >> 1] & 0xFFFF0000u) : __uint_as_float(wd_[i >> 1] << 16);
      else return 0.0f;
    };
    // ---- the update u / clip * lr
    float ud[8];
    if constexpr (OPT == KAON_OPT_ADAKAON || MUON) {
      float ov[8];
      if constexpr (MUON) unpack_dt<KAON_BF16>(in.o, ov);
      if (VEC || factored) {
#pragma unroll
        for (int i = 0; i < 8; ++i) ud[i] = ((MUON ? ov[i] : g[i]) * (STR ? row4[row_i(i)].y : rv.y)) * in.f[i];
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) ud[i] = (MUON ? ov[i] : g[i]) * (1.0f / sqrtf(in.f[i]));
      }
      if (fac != 1.0f) {
#pragma unroll
        for (int i = 0; i < 8; ++i) ud[i] = div_r64(ud[i], rfac);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) ud[i] = ud[i] * hp.lr;
      if (OPT == KAON_OPT_ADAKAON && CODEC == KAON_MOM_BF16) round8<KAON_BF16>(ud);  // lerped in bf16
    }
    float mdq[8], dout[8];
    uint32_t mw[mom_words<CODEC>()];
#pragma unroll
    for (int k = 0; k < mom_words<CODEC>(); ++k) mw[k] = 0u;
    float cmaxA = 0.0f, cmaxB = 0.0f;
    uint32_t bcur = blk;
    float bmax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool in_t = VEC ? cnt > 0 : i < cnt;
      if (Q4 && MOM && walk && i > 0 && woff == 0u && in_t) blk_ctx(blk);
      kf4 ri = rv;
      if constexpr (STR && INT8 && MOM) ri = row4[row_i(i)];
      float mold = 0.0f;
      if constexpr (MOM) mold = INT8 ? code(in.m, i) * ri.z : Q4 ? code(in.m, i) * b_old : code(in.m, i);
      float pw = 0.0f;  // the weight the inner step sees (after the Nekaon removal)
      if constexpr (NEEDP) {
        pw = p[i];
        if (nk_remove) {
          const float ev = msam_e(mold * hp.nk_k, hp.nk_bound_old, nf_old);
          pw = LOWP ? bf2f(sr_bf16(pw + ev, nz0[i])) : pw + ev;
        }
      }
      const float gv = g[i];
      float d, mfv = 0.0f;  // the update, the new momentum in fp32
      if constexpr (OPT == KAON_OPT_ADAKAON) {
        if constexpr (MOM) {
          mfv = lerp(mold, ud[i]);
          if (CODEC == KAON_MOM_BF16) mfv = rbf(mfv);
          d = mfv;
        } else {
          d = ud[i];
        }
      } else if constexpr (MUON) {
        d = ud[i];
        if (MOM) mfv = lerp(mold, gv);
      } else if constexpr (PNM) {
        const float mng = INT8 ? code(in.n, i) * (STR ? rown[row_i(i)] : ngs)
                               : Q4 ? code(in.n, i) * b_neg : code(in.n, i);
        mfv = __fmaf_rn(hp.a1, gv, mold * hp.b1);
        const float pn = __fmaf_rn(hp.pn_neg, mng, mfv * hp.pn_pos) * hp.pn_rnorm;
        const float rf = STR ? row4[row_i(i)].y : rv.y;
        const float u = VEC || factored ? pn * ((rf * in.f[i]) * hp.bc2)
                                        : pn / ((sqrtf(in.f[i] + 1e-15f) + hp.eps1) / hp.bc2);
        d = (fac == 1.0f ? u : div_r64(u, rfac)) * hp.lr;
      } else {  // Lion
        d = ksign(__fmaf_rn(hp.a1, gv, mold * hp.b1));
        mfv = __fmaf_rn(hp.a2, gv, mold * hp.b2);
      }
      if (wd && !PNM) d = __fmaf_rn(hp.wdl, pw, d);
      const bool kp = d * gv > 0.0f;
      if constexpr (PHASE == 5) {
        keep += kp && in_t ? 1u : 0u;
        if (ABSMAX && in_t) {
          const float ax = fabsf(mfv);
          if constexpr (INT8) {
            const uint32_t st = (steps >> (4 * i)) & 7u;
            if (STR && st != 0u) {
              if (C < 8u) atomicMax(&smax[q.r + st], __float_as_uint(fmaxf(ax, 0.0f)));
              else cmaxB = fmaxf(cmaxB, ax);
            } else {
              cmaxA = fmaxf(cmaxA, ax);
            }
          } else {
            if (walk && blk != bcur) {
              if (bmax > 0.0f) atomicMax((uint32_t*)&ws.bamax(T)[bcur], __float_as_uint(bmax));
              bcur = blk;
              bmax = 0.0f;
            }
            bmax = fmaxf(bmax, ax);
            if (woff == 0u) ws.boldsc(T, nb)[blk] = b_old;
          }
        }
      } else {
        mdq[i] = mfv;
        if constexpr (INT8 && MOM) {
          float x = rintf(div_r64(mfv, STR ? rowr[row_i(i)] : rnew));
          x = fminf(fmaxf(x, -127.0f), 127.0f);
          mw[i >> 2] |= ((uint32_t)(int)x & 0xFFu) << (8 * (i & 3));
          mdq[i] = x * ri.w;
        } else if constexpr (Q4 && MOM) {
          float x = rintf(div_r64(mfv, b_r));
          x = fminf(fmaxf(x, -7.0f), 7.0f);
          if (in_t) {
            mw[0] |= ((uint32_t)((int)x + 8) & 0xFu) << (4 * i);
            if (woff == 0u) ((KAON_G float*)X.msc)[blk] = b_new;
          }
          mdq[i] = x * b_new;
        }
        float dd = d;
        if (cautious) dd = div_r64(d * (kp ? 1.0f : 0.0f), rden);
        if (LION) dd = dd * hp.lr;
        dout[i] = dd;
        p[i] = PNM && wd ? round_to<PT>(pw * hp.wdl) : pw;
      }
      if (Q4 && MOM) {
        ++woff;
        if (woff == B) {
          woff = 0u;
          ++blk;
        }
      }
    }
    if constexpr (PHASE == 5) {
      if (Q4 && ABSMAX && (walk || bsh < 0) && cnt > 0 && bmax > 0.0f)
        atomicMax((uint32_t*)&ws.bamax(T)[bcur], __float_as_uint(bmax));
      return Q4 ? kaon_f32x2{bmax, 0.0f} : kaon_f32x2{cmaxA, cmaxB};
    } else {
      if (cnt <= 0) return kaon_f32x2{0.0f, 0.0f};
      // ---------------- phase 6 writes
      if constexpr (MOM) {
        if constexpr (CODEC == KAON_MOM_F32) {
#pragma unroll
          for (int i = 0; i < 8; ++i) mw[i] = __float_as_uint(mdq[i]);
        } else if constexpr (CODEC == KAON_MOM_BF16) {
          pack_lp<KAON_BF16>(mdq, mw);
        }
        st_words((KAON_G uint8_t*)X.m + MB * (q.wb >> 3) + MB * (q.lo >> 3), vec, mom_bytes<CODEC>(cnt), mw);
      }
      uint32_t pwords[dt_words<PT>()];
      if constexpr (PT == KAON_F32) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float x = p[i] - dout[i];
          if (nk_climb) x = x + msam_e(mdq[i] * (-hp.nk_k), hp.nk_bound_new, nf_new);
          pwords[i] = __float_as_uint(x);
        }
      } else {
        if constexpr (KAHAN) {
          // shift -= lp(delta); p0 = p; p += shift; shift += p0 - p, in the
          // param dtype (_backend.py:90-94); only the stored roundings need a
          // canonical NaN
          float sh[8], s[8], p1[8];
          unpack_dt<PT>(in.sh, sh);
          round8<PT>(dout);
#pragma unroll
          for (int i = 0; i < 8; ++i) s[i] = sh[i] - dout[i];
          round8<PT>(s);
#pragma unroll
          for (int i = 0; i < 8; ++i) p1[i] = p[i] + s[i];
          pack_lp<PT>(p1, pwords);
          unpack_dt<PT>(pwords, p1);
#pragma unroll
          for (int i = 0; i < 8; ++i) p1[i] = p[i] - p1[i];
          round8<PT>(p1);
          uint32_t shw[4];
#pragma unroll
          for (int i = 0; i < 8; ++i) s[i] = s[i] + p1[i];
          pack_lp<PT>(s, shw);
          st_words((KAON_G uint8_t*)X.sh + 2 * q.wb + 2 * q.lo, vec, 2 * cnt, shw);
        } else if (hp.bf16_method == KAON_RN || PT == KAON_F16) {
          // fp16 params are written by RN under "stochastic_rounding" too: the
          // reference's SR write is bf16-only (_backend.py:95-98)
          round8<PT>(dout);
#pragma unroll
          for (int i = 0; i < 8; ++i) p[i] = p[i] - dout[i];
          pack_lp<PT>(p, pwords);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            pwords[i] = pack_hi16(sr_word(p[2 * i] - dout[2 * i], nz1[2 * i]),
                                  sr_word(p[2 * i + 1] - dout[2 * i + 1], nz1[2 * i + 1]));
        }
        if (nk_climb) {
          float o[8];
          unpack_dt<PT>(pwords, o);
#pragma unroll
          for (int i = 0; i < 8; ++i) o[i] = o[i] + msam_e(mdq[i] * (-hp.nk_k), hp.nk_bound_new, nf_new);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            pwords[i] = pack_hi16(sr_word(o[2 * i], nz2[2 * i]), sr_word(o[2 * i + 1], nz2[2 * i + 1]));
        }
      }
      st_words((KAON_G uint8_t*)X.p + PB * q.wb + PB * q.lo, vec, PB * cnt, pwords);
      return kaon_f32x2{0.0f, 0.0f};
    }
  };
  // The maxima of a window's lanes into the row / block maxima.
  auto take_max = [&](const Pos& pc, bool str, kaon_f32x2 am) {
    if (ABSMAX && Q4 && bsh >= 3) {
      // blocks of 2^(bsh-3) consecutive chunks, windows start on multiples of 64
      // chunks: a block is an aligned lane group (or part of it is in the next
      // window or slice, hence the atomic)
      const int gl = min(1 << (bsh - 3), 64);
      float a = am[0];
      for (int o = gl >> 1; o >= 1; o >>= 1) a = fmaxf(a, __shfl_xor(a, o, 64));
      if ((lane & (gl - 1)) == 0 && a > 0.0f)
        atomicMax((uint32_t*)&ws.bamax(T)[((uint32_t)pc.wb + 8u * (uint32_t)lane) >> bsh], __float_as_uint(a));
    }
    if (ABSMAX && INT8) {
      // row maxima: a wave maximum for each row of the window, a lane's own
      // LDS maximum where the window spans many
      const uint32_t ra = __builtin_amdgcn_readfirstlane(pc.r);
      const uint32_t rl = (uint32_t)__builtin_amdgcn_readlane((int)pc.r, 63);
      if (rl - ra < 3u) {
        for (uint32_t r = ra; r <= rl + (str ? 1u : 0u); ++r) {
          const float x = pc.r == r ? am[0] : pc.r + 1u == r ? am[1] : 0.0f;
          const float m = wave_max(x);
          if (lane == 0 && m > 0.0f) atomicMax(&smax[r], __float_as_uint(m));
        }
      } else if (pc.cnt > 0) {
        if (am[0] > 0.0f) atomicMax(&smax[pc.r], __float_as_uint(am[0]));
        if (am[1] > 0.0f) atomicMax(&smax[pc.r + 1u], __float_as_uint(am[1]));
      }
    }
  };

  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  const int64_t first = w0 + w;
  if (factored && ce * 8 <= n) {
    // each window's loads are issued inside the previous window's arithmetic,
    // into two buffers in turn (a copy would wait for the loads in flight)
    In buf0, buf1;
    Pos pos0{}, pos1{};
    if (first < wend) {
      pos0 = locate(first);
      flat_load<OPT, PHASE, PT, GT, CODEC, XF, true>(buf0, X, pos0);
    }
    load_rows();
    __syncthreads();
    auto step = [&](int64_t win, const In& cur, const Pos& pc, In& nxt, Pos& pn) {
      // past the last window: this one's chunks again
      auto prefetch = [&]() {
        pn = locate(min(win + 4, wend - 1));
        flat_load<OPT, PHASE, PT, GT, CODEC, XF, true>(nxt, X, pn);
      };
      const bool str = __builtin_amdgcn_ballot_w64(pc.j0 + 8u > C) != 0;
      kaon_f32x2 am;
      if (str) am = chunk(cur, pc, Yes{}, Yes{}, prefetch);
      else am = chunk(cur, pc, No{}, Yes{}, prefetch);
      take_max(pc, str, am);
    };
    for (int64_t win = first; win < wend; win += 8) {
      step(win, buf0, pos0, buf1, pos1);
      if (win + 4 < wend) step(win + 4, buf1, pos1, buf0, pos0);
    }
  } else {
    load_rows();
    __syncthreads();
    // a vector is one row: no lookups per element (200 vectors of 1280 and 200 of 77,
    // int8: Lion's keep count 5.8 -> 5.3 us and apply 7.4 -> 6.9, Adakaon's 9.9 -> 9.5
    // and 10.5 -> 10.1; four of 4 M elements, whole Adakaon steps 12.8 -> 10.6 ms)
    const bool str = nctx > 1;
    for (int64_t win = first; win < wend; win += 4) {
      In in;
      const Pos q = locate(win);
      flat_load<OPT, PHASE, PT, GT, CODEC, XF, false>(in, X, q);
      kaon_f32x2 am;
      if (str) am = chunk(in, q, Yes{}, No{}, [] {});
      else am = chunk(in, q, No{}, No{}, [] {});
      take_max(q, str, am);
    }
  }

  if (PHASE == 5) {
    if (cautious) {
      const uint32_t wsum = wave_sum_u32(keep);
      if (lane == 0) keep_s[w] = wsum;
    }
    __syncthreads();
    if (cautious && threadIdx.x == 0) {
      const uint32_t tot = keep_s[0] + keep_s[1] + keep_s[2] + keep_s[3];
      if (tot) atomicAdd(ws.keep_ctr(T), tot);
    }
    if (ABSMAX && INT8) {
      for (int k = threadIdx.x; k < nctx; k += KAON_WG)
        if (smax[k]) atomicMax((uint32_t*)&ws.ramax(T)[it.row0 + k], smax[k]);
    }
  }
}

// xf: phase 5 with weight decay, phase 6 with kahan writes (16-bit params).
template <int OPT, int PHASE, int PT, int GT, int CODEC>
ElemFn flat_by_xf(bool xf) {
  if constexpr (CODEC == KAON_MOM_NONE && OPT != KAON_OPT_ADAKAON && OPT != KAON_OPT_ADAMUON) return nullptr;
  else if constexpr ((PHASE == 5 && OPT == KAON_OPT_ADAPNM) || (PHASE == 6 && PT == KAON_F32))
    return k_flat<OPT, PHASE, PT, GT, CODEC, false>;
  else return xf ? k_flat<OPT, PHASE, PT, GT, CODEC, true> : k_flat<OPT, PHASE, PT, GT, CODEC, false>;
}

template <int OPT, int PHASE, int PT, int GT>
ElemFn flat_by_codec(int codec, bool xf) {
  switch (codec) {
    case KAON_MOM_NONE: return flat_by_xf<OPT, PHASE, PT, GT, KAON_MOM_NONE>(xf);
    case KAON_MOM_F32: return flat_by_xf<OPT, PHASE, PT, GT, KAON_MOM_F32>(xf);
    case KAON_MOM_BF16: return flat_by_xf<OPT, PHASE, PT, GT, KAON_MOM_BF16>(xf);
    case KAON_MOM_INT8: return flat_by_xf<OPT, PHASE, PT, GT, KAON_MOM_INT8>(xf);
    case KAON_MOM_4BIT: return flat_by_xf<OPT, PHASE, PT, GT, KAON_MOM_4BIT>(xf);
  }
  return nullptr;
}

template <int OPT, int PHASE>
ElemFn flat_fn(const KaonHyper& h, int codec) {
  const int pt = h.p_dtype, gt = h.g_dtype;
  const bool xf = PHASE == 5 ? (h.flags & KAON_F_WD) != 0 : h.bf16_method == KAON_KAHAN;
  if (pt == KAON_BF16 && gt == KAON_BF16) return flat_by_codec<OPT, PHASE, KAON_BF16, KAON_BF16>(codec, xf);
  if (pt == KAON_BF16 && gt == KAON_F32) return flat_by_codec<OPT, PHASE, KAON_BF16, KAON_F32>(codec, xf);
  if (pt == KAON_F32 && gt == KAON_BF16) return flat_by_codec<OPT, PHASE, KAON_F32, KAON_BF16>(codec, xf);
  if (pt == KAON_F32 && gt == KAON_F32) return flat_by_codec<OPT, PHASE, KAON_F32, KAON_F32>(codec, xf);
  if (pt == KAON_F16 && gt == KAON_F16) return flat_by_codec<OPT, PHASE, KAON_F16, KAON_F16>(codec, xf);
  return nullptr;
}

}  // namespace

// One object per optimizer and phase (the build compiles them side by side).
namespace kaon {
#define KAON_FLAT_FN(NAME, OPT, PHASE) \
  ElemFn NAME(const KaonHyper& h, int codec) { return flat_fn<OPT, PHASE>(h, codec); }
#if KAON_FLAT_PART == 0
KAON_FLAT_FN(flat_ada5, KAON_OPT_ADAKAON, 5)
#elif KAON_FLAT_PART == 1
KAON_FLAT_FN(flat_ada6, KAON_OPT_ADAKAON, 6)
#elif KAON_FLAT_PART == 2
KAON_FLAT_FN(flat_lion5, KAON_OPT_LION, 5)
KAON_FLAT_FN(flat_lion6, KAON_OPT_LION, 6)
#elif KAON_FLAT_PART == 3
KAON_FLAT_FN(flat_muon5, KAON_OPT_ADAMUON, 5)
KAON_FLAT_FN(flat_muon6, KAON_OPT_ADAMUON, 6)
#elif KAON_FLAT_PART == 4
KAON_FLAT_FN(flat_pnm5, KAON_OPT_ADAPNM, 5)
KAON_FLAT_FN(flat_pnm6, KAON_OPT_ADAPNM, 6)
#endif
#undef KAON_FLAT_FN
}  // namespace kaon
