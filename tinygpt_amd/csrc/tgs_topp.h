// tgs_topp.h -- what the two top-p kernels share: a row (or a chunk of one)
// as a view over its allowed ids, and the tail of a sampling row from its
// bucket histogram to the drawn id (one workgroup per row: tgs_topp.hip; a
// row over several workgroups: tgs_topp_split.hip).
//
// The contract keeps the smallest prefix of the allowed ids in (y desc,
// id asc) order whose exact mass reaches P = floor(S p24 / 2^24) and draws
// the first id whose inclusive prefix exceeds t = floor(S' u24 / 2^24);
// masses are q = floor(exp(y - m) 2^40).  Only ids with q > 0 can be the cut
// or the draw (both are where the prefix grows), and those lie within 32 of
// the maximum m.  Counts and masses per bucket below m (width 1/32,
// tgs_bucket.h) locate the cut's and the draw's bucket; only those buckets'
// ids are gathered and ranked.
#pragma once

#include "tgs_bucket.h"
#include "tgs_device.h"
#include "tgs_kernels.h"
#include "tgs_row.h"

namespace tgs {
namespace topp {

constexpr int NB = bucket::NB; // mass buckets below the maximum
constexpr int CAPL = TOPP_CAP; // ids gathered in LDS
constexpr int RES_EPT = 32;    // ids per thread kept in registers

// BT threads per workgroup throughout.
template <int BT>
struct Scratch {
  u64 red64[BT / 64];
  u64 red64b[BT / 64];
  unsigned red32[BT / 64];
  unsigned ng;    // gathered ids: list A's in the low 16 bits, list B's above
  int sel[3];     // buckets of the cut, and of the lowest and the highest draw target
  int first;      // first rank meeting a mass target
  int first2;     // the same for the draw, in the one-gather tail
  unsigned nsel;  // select_list: members of the last bin
};

// The canonical logits of ids [r.v0, r.v1) of a row (r.v0 a multiple of 32):
// y after penalties and temperature, -inf where the id is not allowed (mask
// bit clear, -inf or NaN).  RES: held in registers (RES_EPT ids per thread,
// loaded once).  Otherwise every walk streams them again from L2 / MALL: the
// fallback of a workgroup that finishes a row, or a partner's chunk, whose ids
// it does not hold.
template <typename Tin, bool RES, int BT>
struct RowView {
  static constexpr int EPV = Elem<Tin>::EPV;
  static constexpr int NV = RES ? RES_EPT / EPV : 1;  // vectors per thread held
  const SampleArgs& a;
  const Row& r;
  const int2* hash;
  const uint32_t* hbits;
  const Tin* rowp;
  float y[RES ? RES_EPT : 1];
  unsigned nallowed = 0;  // this thread's allowed ids among y (set by load)

  __device__ __forceinline__ RowView(const SampleArgs& a_, const Row& r_, const int2* h_, const uint32_t* hb_,
                                     const Tin* p_)
      : a(a_), r(r_), hash(h_), hbits(hb_), rowp(p_) {}

  // y of the EPV ids of vector v from its loaded bits
  __device__ __forceinline__ void vec_y(int v, const uint4& raw, float (&yv)[EPV]) const {
    const bool in = v < r.v1;  // a vector past the row end reads no mask or history word
    const uint32_t mw = !in ? 0u : r.mrow ? r.mrow[v >> 5] : 0xFFFFFFFFu;
    const uint32_t hw = (in && r.use_pen) ? hbits[v >> 5] : 0u;
#pragma unroll
    for (int e = 0; e < EPV; e++) {
      const int id = v + e;
      float z = Elem<Tin>::get(raw, e);
      if ((hw >> (id & 31)) & 1u) z = penalise(z, hash_count(hash, a.TS, a.ts_shift, id), r);
      const float yy = row_y(r, z);
      yv[e] = (((mw >> (id & 31)) & 1u) && yy > -__builtin_inff() && id < r.v1) ? yy : -__builtin_inff();
    }
  }

  // vectors J0 .. J1 - 1 of this thread's share of ids [v0, v1).  Whole
  // vectors are read with one unconditional load each (a vector past the end
  // reads the last one again; its mask word is 0), so no load waits for an
  // earlier one: a divergent fallback beside the loads makes the compiler
  // wait for the loads already issued before reusing their registers.  Rows
  // need not be aligned (load_row16); fix_tail puts the ids of a partial
  // last vector in place.
  template <int J0, int J1>
  __device__ __forceinline__ static void fetch(const Tin* p, int v0, int v1, uint4 (&raw)[NV]) {
    if constexpr (RES) {
      const int last = (v1 - v0) / EPV - 1;
      if (last >= 0) {
#pragma unroll
        for (int j = J0; j < J1; j++) {
          const int vi = (int)threadIdx.x + j * BT;
          raw[j] = load_row16<true>(p + v0 + (vi < last ? vi : last) * EPV);
        }
      } else {
#pragma unroll
        for (int j = J0; j < J1; j++) raw[j] = make_uint4(0u, 0u, 0u, 0u);  // fix_tail reads the only vector
      }
    }
  }
  __device__ __forceinline__ static void fix_tail(const Tin* p, int v0, int v1, uint4 (&raw)[NV]) {
    if constexpr (RES) {
      const int n = v1 - v0;
      if (n % EPV != 0) {  // (uniform)
#pragma unroll
        for (int j = 0; j < NV; j++)
          if ((int)threadIdx.x + j * BT == n / EPV) raw[j] = load_vec<Tin>(p, v0 + n / EPV * EPV, v1, false);
      }
    }
  }

  // the mask word of each of this thread's register-resident vectors (all
  // ones without a mask row, 0 past the end)
  __device__ __forceinline__ static void mask_words(const Row& r, int v0, int v1, uint32_t (&mw)[NV]) {
    if constexpr (RES) {
#pragma unroll
      for (int j = 0; j < NV; j++) {
        const int v = v0 + ((int)threadIdx.x + j * BT) * EPV;
        mw[j] = v >= v1 ? 0u : r.mrow ? r.mrow[v >> 5] : 0xFFFFFFFFu;
      }
    }
  }

  // y of the register-resident vectors, specialised on what is uniform over
  // the row (penalties present, a power-of-two temperature, T = 1: y = z
  // exactly) so that the per-element code carries no branch or operation for
  // the cases the row does not have
  template <bool PEN, bool POW2, bool ONE = false>
  __device__ __forceinline__ void load_t(const uint4 (&raw)[NV], const uint32_t (&mw)[NV]) {
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int v = r.v0 + ((int)threadIdx.x + j * BT) * EPV;
      const uint32_t hw = (PEN && v < r.v1) ? hbits[v >> 5] : 0u;
#pragma unroll
      for (int e = 0; e < EPV; e++) {
        const int id = v + e;
        float z = Elem<Tin>::get(raw[j], e);
        if constexpr (PEN) {
          if ((hw >> (id & 31)) & 1u) z = penalise(z, hash_count(hash, a.TS, a.ts_shift, id), r);
        }
        // (an id past the end needs no test: its vector's mask word is 0, or,
        // in a vector that straddles the end, load_vec read it as NaN)
        const float yy = ONE ? z : POW2 ? z * r.rT : row_y(r, z);
        const bool ok = ((mw[j] >> (id & 31)) & 1u) && yy > -__builtin_inff();
        y[j * EPV + e] = ok ? yy : -__builtin_inff();
        nallowed += ok ? 1u : 0u;
      }
    }
  }

  __device__ __forceinline__ void load(const uint4 (&raw)[NV], const uint32_t (&mw)[NV]) {
    if constexpr (RES) {
      if (r.use_pen) load_t<true, false>(raw, mw);
      else if (r.tdiv == TDIV_POW2 && r.rT == 1.0f) load_t<false, true, true>(raw, mw);
      else if (r.tdiv == TDIV_POW2) load_t<false, true>(raw, mw);
      else load_t<false, false>(raw, mw);
    }
  }

  // f(id, y) for every allowed id of the row, read again from L2 / MALL
  // (a rolled loop: no register-held state besides the caller's)
  template <class F>
  __device__ __forceinline__ void each_stream(F f) const {
    const int nvec = (r.v1 - r.v0 + EPV - 1) / EPV;
#pragma unroll 1
    for (int vi = threadIdx.x; vi < nvec; vi += BT) {
      const int v = r.v0 + vi * EPV;
      const uint4 raw = load_vec<Tin>(rowp, v, r.v1, a.aligned);
      float yv[EPV];
      vec_y(v, raw, yv);
#pragma unroll
      for (int e = 0; e < EPV; e++)
        if (yv[e] > -__builtin_inff()) f(v + e, yv[e]);
    }
  }

  // f(id, y) for every allowed id of the row
  template <class F>
  __device__ __forceinline__ void each(F f) const {
    if constexpr (RES) {
#pragma unroll
      for (int j = 0; j < NV; j++)
#pragma unroll
        for (int e = 0; e < EPV; e++) {
          const float yy = y[j * EPV + e];
          if (yy > -__builtin_inff()) f(r.v0 + ((int)threadIdx.x + j * BT) * EPV + e, yy);
        }
    } else {
      const int nvec = (r.v1 - r.v0 + EPV - 1) / EPV;
      for (int vi = threadIdx.x; vi < nvec; vi += BT) {
        const int v = r.v0 + vi * EPV;
        const uint4 raw = load_vec<Tin>(rowp, v, r.v1, a.aligned);
        float yv[EPV];
        vec_y(v, raw, yv);
#pragma unroll
        for (int e = 0; e < EPV; e++)
          if (yv[e] > -__builtin_inff()) f(v + e, yv[e]);
      }
    }
  }
};

// One allowed id and its canonical logit, packed in LDS.
struct alignas(8) Packed {
  float y;
  int id;
};

// The allowed ids of a row packed in LDS: E[0, n).
template <int BT>
struct CompactView {
  const Packed* E;
  int n;
  template <class F>
  __device__ __forceinline__ void each(F f) const {
#pragma unroll 2
    for (int i = threadIdx.x; i < n; i += BT) {
      const Packed e = E[i];
      f(e.id, e.y);
    }
  }
  template <class F>
  __device__ __forceinline__ void each_stream(F f) const {
    each(f);
  }
};

template <int BT, typename T>
__device__ __forceinline__ T block_reduce_max(T x, T* red) {
  x = wave_max(x);
  if (lane_id() == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  T t = red[0];
#pragma unroll
  for (int i = 1; i < BT / 64; i++) t = red[i] > t ? red[i] : t;
  __syncthreads();
  return t;
}

// The row's tail state: the bucket prefixes, the gathered lists and two
// ranked ones of at most 64 ids.
struct Tail {
  unsigned* CI;  // NB + 1 inclusive counts
  u64* MI;       // NB + 1 inclusive masses
  u64* L;        // CAPL gathered composites (list A, then list B from Plan::ob)
  u64 *R, *Q;    // 64 ranked composites and their inclusive masses (list A's)
  u64 *R2, *Q2;  // the same for list B
  Packed* E;     // a.topp_cap packed allowed ids
  float m;
};

// The element of the distinct composites L[0, n) (n > 0; a barrier after the
// gather) whose inclusive mass prefix in descending order first reaches
// target (>= 1): the composite, the mass ahead of it and its rank.  At most
// 64 are ranked by one wave; more are narrowed first by mass-weighted radix
// digits from the highest bit in which they differ (one or two passes over
// the list: counting every entry's rank read n^2 / 2 entries, 5 us at 400).
// BYCOUNT: the target-th element (target in [1, n]) instead.  R, Q: 64
// entries of scratch.  Ends with a barrier.
template <int BT, bool BYCOUNT = false>
__device__ __forceinline__ u64 select_list(const u64* L, unsigned n, float m, u64 target, u64* before, unsigned* rank,
                                           u64* R, u64* Q, Scratch<BT>& ts, BlockScratch& bs) {
  u64 bm = 0;
  unsigned br = 0;
  if (n > 64u) {
    u64 d = 0;
    const u64 x0 = L[0];
    for (unsigned i = threadIdx.x; i < n; i += BT) d |= L[i] ^ x0;
    d = wave_or64(d);
    if (lane_id() == 0) ts.red64b[threadIdx.x >> 6] = d;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < BT / 64; v++) d |= ts.red64b[v];
    int shift = 56 - __clzll((long long)d);
    u64 prefix = 0, pmask = 0;
#pragma unroll 1
    for (;;) {
      if (shift < 0) shift = 0;
      for (int i = threadIdx.x; i < 256; i += BT) {
        bs.hc[i] = 0;
        bs.hm[i] = 0;
      }
      if (threadIdx.x == 0) ts.nsel = 0;
      __syncthreads();
      for (unsigned i = threadIdx.x; i < n; i += BT) {
        const u64 x = L[i];
        if ((x & pmask) == prefix) {
          const unsigned g = (unsigned)(x >> shift) & 255u;
          atomicAdd(&bs.hc[g], 1u);
          const u64 q = bucket::mass_c(x, m);
          if (q) atomicAdd(&bs.hm[g], q);
        }
      }
      __syncthreads();
      if (threadIdx.x < 64) mass_digit_scan<BYCOUNT>(bs, target, bm, br);
      __syncthreads();
      bm = bs.mass_above;
      br = bs.cnt_above;
      prefix |= (u64)bs.sel << shift;
      pmask |= 255ull << shift;
      if (bs.binc_i <= 64) break;  // (composites are distinct: at the latest at shift 0)
      shift -= 8;
    }
    for (unsigned i = threadIdx.x; i < n; i += BT) {
      const u64 x = L[i];
      if ((x & pmask) == prefix) R[atomicAdd(&ts.nsel, 1u)] = x;
    }
    __syncthreads();
    n = ts.nsel;
    L = R;
  }
  if (threadIdx.x < 64) bucket::wave_rank64(L, n, m, R, Q);
  __syncthreads();
  const int i = BYCOUNT ? (int)((unsigned)target - br) - 1 : bucket::first_rank_once(Q, n, target - bm, &ts.first);
  *before = bm + (i > 0 ? Q[i - 1] : 0ull);
  *rank = br + (unsigned)i;
  const u64 x = R[i];
  __syncthreads();
  return x;
}

// The bits that the composites en(f) enumerates share, and where the first
// digit that tells them apart starts (block_select_kth).  The ids of a
// crowded bucket agree in most of their keys' bits, and a digit in which they
// agree costs a pass whose LDS atomics all go to one bin: 64 top-p rows of
// 128,256 equal fp32 logits took 5.9 ms from bit 63 down.
struct Digits {
  u64 prefix, pmask;
  int shift;
};
template <int BT, class Enum>
__device__ __forceinline__ Digits shared_digits(Enum en, Scratch<BT>& ts) {
  u64 any = 0, all = ~0ull;
  en([&](u64 x) {
    any |= x;
    all &= x;
  });
  any = wave_or64(any);
  all = ~wave_or64(~all);
  __syncthreads();
  if (lane_id() == 0) {
    ts.red64[threadIdx.x >> 6] = any;
    ts.red64b[threadIdx.x >> 6] = all;
  }
  __syncthreads();
  any = 0;
  all = ~0ull;
#pragma unroll
  for (int v = 0; v < BT / 64; v++) {
    any |= ts.red64[v];
    all &= ts.red64b[v];
  }
  const u64 d = any ^ all;
  if (d == 0ull) return Digits{all, ~0ull, 0};  // one composite
  const int h = 63 - __clzll((long long)d);
  const u64 pmask = h == 63 ? 0ull : ~0ull << (h + 1);
  return Digits{all & pmask, pmask, h - 7};
}

// Bucket bq's ids (at most CAPL) into tl.L, from the row.  Starts and ends
// with a barrier.
template <int BT, class View>
__device__ __forceinline__ void gather_bucket(const View& rv, Tail& tl, int bq, Scratch<BT>& ts) {
  const float m = tl.m;
  if (threadIdx.x == 0) ts.ng = 0;
  __syncthreads();
  rv.each_stream([&](int id, float y) {
    if (bucket::of(y, m) == bq) tl.L[atomicAdd(&ts.ng, 1u)] = comp_key(tg_key(y), id);
  });
  __syncthreads();
}

// The element of bucket bq whose within-bucket inclusive prefix first
// reaches target (>= 1): its composite, the mass ahead of it in the bucket
// and its rank there.  The bucket's members are gathered from the row; a
// bucket of more than CAPL ids is resolved by a mass-weighted radix
// selection over the row restricted to it instead.
template <int BT, class View>
__device__ __forceinline__ u64 resolve_mass(const View& rv, Tail& tl, int bq, u64 target, u64* before,
                                            unsigned* rank, Scratch<BT>& ts, BlockScratch& bs) {
  const float m = tl.m;
  const unsigned n = tl.CI[bq] - bucket::count_before(tl.CI, bq);
  if (n <= (unsigned)CAPL) {
    gather_bucket<BT>(rv, tl, bq, ts);
    return select_list<BT>(tl.L, n, m, target, before, rank, tl.R, tl.Q, ts, bs);
  }
  auto each_of = [&](auto f) {
    rv.each_stream([&](int id, float y) {
      if (bucket::of(y, m) == bq) f(id, y);
    });
  };
  const Digits d = shared_digits<BT>([&](auto f) { each_of([&](int id, float y) { f(comp_key(tg_key(y), id)); }); }, ts);
  return block_mass_select<BT>(
      [&](auto f) { each_of([&](int id, float y) { f(comp_key(tg_key(y), id), bucket::mass(y, m)); }); }, target, bs,
      before, rank, d.shift, d.prefix, d.pmask);
}

// The ik-th largest (1-based) of bucket bq's ids and the mass of the ik
// largest; as resolve_mass.
template <int BT, class View>
__device__ __forceinline__ u64 resolve_count(const View& rv, Tail& tl, int bq, unsigned ik, u64* mass,
                                             Scratch<BT>& ts, BlockScratch& bs) {
  const float m = tl.m;
  const unsigned n = tl.CI[bq] - bucket::count_before(tl.CI, bq);
  if (n <= (unsigned)CAPL) {
    gather_bucket<BT>(rv, tl, bq, ts);
    u64 before;
    unsigned rank;
    const u64 x = select_list<BT, true>(tl.L, n, m, ik, &before, &rank, tl.R, tl.Q, ts, bs);
    *mass = before + bucket::mass_c(x, m);
    return x;
  }
  auto en = [&](auto f) {
    rv.each_stream([&](int id, float y) {
      if (bucket::of(y, m) == bq) f(comp_key(tg_key(y), id));
    });
  };
  const Digits d = shared_digits<BT>(en, ts);
  const u64 T = block_select_kth<u64, 64, BT>(en, ik, bs, d.shift, d.prefix, d.pmask);
  u64 S = 0, minc = ~0ull;
  en([&](u64 x) {
    if (x < T) return;
    S += bucket::mass_c(x, m);
    minc = x < minc ? x : minc;
  });
  *mass = block_sum<u64, BT>(S, ts.red64);
  return ~block_max<u64, BT>(~minc, ts.red64b);
}

// Pass 2: every allowed id of the view into the count and exact-mass
// histogram over the buckets below m (CI, MI zeroed before).  With
// a finite maximum, x = y - m is +-0 exactly at y == m, where bucket 0 and
// weight 1 follow from x itself (tg_expf_nonpos(+-0) = 1), so the test for
// y == m that an infinite maximum needs is left out.
template <class View>
__device__ __forceinline__ void histogram(const View& rv, Tail& tl) {
  const float m = tl.m;
  if (m < __builtin_inff()) {
    rv.each([&](int, float y) {
      const float x = y - m;
      const int bq = !(x > -32.0f) ? NB : (int)(-x * 32.0f);
      atomicAdd(&tl.CI[bq], 1u);
      if (bq < NB) {  // -32 < x <= 0
        const u64 q = tg_q40(tg_expf_nonpos_in(x));
        if (q) atomicAdd(&tl.MI[bq], q);
      }
    });
  } else {
    rv.each([&](int, float y) {
      const int bq = bucket::of(y, m);
      atomicAdd(&tl.CI[bq], 1u);
      if (bq < NB) {
        const u64 q = bucket::mass(y, m);
        if (q) atomicAdd(&tl.MI[bq], q);
      }
    });
  }
}

// Where a row's cut and draw lie, from the inclusive prefixes.
struct Plan {
  u64 S = 0, P = 0, Sp = 0;  // kept mass, the top-p target, S' (final unless cut_search)
  u64 cutc = 0;  // the cut's composite (final unless cut_search)
  unsigned ntopp = 0, nv = 0;  // size of the top-p set (final unless cut_search), of the top-k set (all allowed ids without one)
  uint32_t uq = 0;  // floor(u 2^24)
  bool cut_search = false;  // the cut is an element of bucket bp still to be found
  bool cut_last = false;  // top-p off: the cut is the top-k set's last element
  bool k_search = false;  // the top-k set ends inside list A: S, and what follows from it, is settled there
  bool one = false;  // lists A and B fit: one gather settles the row
  int bp = 0;  // the cut's bucket (k_search: the top-k set's last)
  int a0 = 0, a1 = 0;  // list A's buckets
  int b0 = 1, b1 = 0;  // list B's buckets (b0 > b1: none)
  unsigned na = 0, nb = 0;  // their ids
  unsigned ob = 0;  // list B's offset in the lists
  // which list bucket q belongs to: 0 A, 1 B, -1 neither
  __device__ __forceinline__ int list(int q) const {
    return q >= a0 && q <= a1 ? 0 : q >= b0 && q <= b1 ? 1 : -1;
  }
};

// The draw: first element with inclusive prefix > t = floor(S' u24 / 2^24).
// While the cut is open, S' lies in [P, MI[bp]] (the cut's inclusive prefix
// reaches P and ends inside bucket bp), so t lies in [tlo, thi] and the draw
// in the buckets that hold the targets tlo + 1 .. thi + 1, few and none past
// bp.  One gather collects them and the cut's bucket: as list A alone when
// they meet it, else as list B (a run of buckets ranks like one).  Zeroes the
// list counters; ends with a barrier.
template <int BT>
__device__ __forceinline__ void plan_row(Plan& pl, const Row& r, const Tail& tl, u64 Mc, unsigned nv, Scratch<BT>& ts) {
  const u64 S = tl.MI[NB - 1];
  u64 P = 0, Sp = S, low = S;  // low: the least S' can be
  pl.cutc = 0;
  pl.ntopp = nv;
  pl.nv = nv;
  pl.cut_last = false;
  pl.cut_search = false;
  pl.k_search = false;
  if (r.top_p < 1.0f) {
    P = mul_shr24(S, (uint32_t)(r.top_p * 16777216.0f));
    if (P == 0) {
      pl.cutc = Mc;
      low = Sp = tg_q40(1.0f);
      pl.ntopp = 1;
    } else {
      pl.cut_search = true;
      low = P;
    }
  } else {
    pl.cut_last = true;
  }
  pl.S = S;
  pl.P = P;
  pl.Sp = Sp;
  pl.uq = (uint32_t)(r.u * 16777216.0f);
  const u64 tlo = mul_shr24(low, pl.uq);
  if (threadIdx.x == 0) ts.ng = 0;
  bucket::find_mass2<BT>(tl.MI, pl.cut_search ? low : tlo + 1, tlo + 1, &ts.sel[0], &ts.sel[1]);
  pl.bp = ts.sel[0];
  const int btl = ts.sel[1];
  int bth = btl;
  if (pl.cut_search) {
    const u64 thi = mul_shr24(tl.MI[pl.bp], pl.uq);
    if (tl.MI[btl] < thi + 1) bth = bucket::find_mass<BT>(tl.MI, thi + 1, &ts.sel[2]);
  }
  const bool join = !pl.cut_search || bth == pl.bp;
  pl.a0 = join ? btl : pl.bp;
  pl.a1 = pl.cut_search ? pl.bp : btl;
  pl.b0 = join ? 1 : btl;
  pl.b1 = join ? 0 : bth;
  pl.na = tl.CI[pl.a1] - bucket::count_before(tl.CI, pl.a0);
  pl.nb = join ? 0u : tl.CI[bth] - bucket::count_before(tl.CI, btl);
  pl.ob = pl.na;
  pl.one = pl.na + pl.nb <= (unsigned)CAPL;
}

// The same for a row whose top-k set (its kk first allowed ids, kk below the
// allowed count) ends in bucket bk < NB.  S lies in [slo, MI[bk]] (all of the
// buckets before bk, and the maximum's own mass), and P, S' and the draw's
// target follow with it, so list A runs from the lowest bucket the cut can
// lie in to bk, joined by the draw's run when they meet.  Ends with a
// barrier.
template <int BT>
__device__ __forceinline__ void plan_topk(Plan& pl, const Row& r, const Tail& tl, u64 Mc, unsigned kk,
                                          Scratch<BT>& ts) {
  pl.nv = kk;
  pl.ntopp = kk;
  pl.cutc = 0;
  pl.k_search = true;
  pl.cut_search = pl.cut_last = false;
  if (threadIdx.x == 0) ts.ng = 0;
  const int bk = bucket::find_count<BT>(tl.CI, kk, &ts.sel[0]);
  pl.bp = bk;
  const u64 one = tg_q40(1.0f), sb = bucket::mass_before(tl.MI, bk);
  const u64 slo = sb > one ? sb : one, shi = tl.MI[bk];
  pl.S = shi;
  pl.uq = (uint32_t)(r.u * 16777216.0f);
  const uint32_t pq = r.top_p < 1.0f ? (uint32_t)(r.top_p * 16777216.0f) : 0u;
  pl.P = 0;
  pl.Sp = one;
  u64 plo = slo, phi = shi;  // the range of S'
  int lo = bk;
  if (r.top_p < 1.0f && pq == 0u) {
    pl.cutc = Mc;
    pl.ntopp = 1;
    plo = phi = one;
  } else if (r.top_p < 1.0f) {
    pl.cut_search = true;
    plo = mul_shr24(slo, pq);  // >= 1: slo >= 2^40
    phi = mul_shr24(shi, pq);
    bucket::find_mass2<BT>(tl.MI, plo, phi, &ts.sel[1], &ts.sel[2]);
    lo = ts.sel[1] < bk ? ts.sel[1] : bk;
    phi = tl.MI[ts.sel[2] < bk ? ts.sel[2] : bk];
    __syncthreads();  // before the slots are written again
  } else {
    pl.cut_last = true;
  }
  bucket::find_mass2<BT>(tl.MI, mul_shr24(plo, pl.uq) + 1, mul_shr24(phi, pl.uq) + 1, &ts.sel[1], &ts.sel[2]);
  const int dl = ts.sel[1], dh = ts.sel[2] < bk ? ts.sel[2] : bk;
  const bool join = dh >= lo;
  if (join && dl < lo) lo = dl;
  pl.a0 = lo;
  pl.a1 = bk;
  pl.b0 = join ? 1 : dl;
  pl.b1 = join ? 0 : dh;
  pl.na = tl.CI[bk] - bucket::count_before(tl.CI, lo);
  pl.nb = pl.b0 <= pl.b1 ? tl.CI[pl.b1] - bucket::count_before(tl.CI, pl.b0) : 0u;
  pl.ob = pl.na;
  pl.one = pl.na + pl.nb <= (unsigned)CAPL;
}

// The allowed ids of the lists' buckets, in no particular order, into their
// list (sink(list, place, composite)); ts.ng counts them (zero before).
// From registers: a bit per slot and list from the position below the
// maximum (the same float the bucket is the integer part of), one wave scan
// and one LDS atomic per wave for the places, then the marked slots written
// (an atomic per id waited for its result in every slot, 5 us).
template <typename Tin, int BT, class F>
__device__ __forceinline__ void gather(const RowView<Tin, true, BT>& rv, const Plan& pl, float m, Scratch<BT>& ts,
                                       F sink) {
  constexpr int EPV = Elem<Tin>::EPV;
  const float a0 = (float)pl.a0, a1 = (float)(pl.a1 + 1), b0 = (float)pl.b0, b1 = (float)(pl.b1 + 1);
  uint32_t ma = 0u, mb = 0u;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) {
    const float y = rv.y[q];
    const float f = y == m ? 0.0f : (m - y) * 32.0f;  // -inf: +inf, in no list
    ma |= (f >= a0 && f < a1) ? 1u << q : 0u;
    mb |= (f >= b0 && f < b1) ? 1u << q : 0u;
  }
  const unsigned n = (unsigned)__popc(ma) | (unsigned)__popc(mb) << 16;
  const unsigned incl = wave_incl_scan(n);
  const unsigned tot = readlane_u32(incl, 63);
  if (tot == 0u) return;
  unsigned at = 0u;
  if (lane_id() == 0) at = atomicAdd(&ts.ng, tot);
  at = readlane_u32(at, 0) + incl - n;
  unsigned oa = at & 0xFFFFu, ob = at >> 16;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) {
    if (!(((ma | mb) >> q) & 1u)) continue;
    const u64 x = comp_key(tg_key(rv.y[q]), rv.r.v0 + ((int)threadIdx.x + (q / EPV) * BT) * EPV + q % EPV);
    if ((ma >> q) & 1u) sink(0, oa++, x);
    else sink(1, ob++, x);
  }
}
// The thread's slots that hold an allowed id with y >= yb, a bit each.
template <typename Tin, int BT>
__device__ __forceinline__ uint32_t floor_marks(const RowView<Tin, true, BT>& rv, float yb) {
  uint32_t ma = 0u;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) ma |= (rv.y[q] >= yb && rv.y[q] > -__builtin_inff()) ? 1u << q : 0u;
  return ma;
}
// Places for the marked slots of the wave's threads (the first of this
// thread's): one wave scan and one LDS atomic; ts.ng counts them.
template <int BT>
__device__ __forceinline__ unsigned mark_places(uint32_t ma, Scratch<BT>& ts) {
  const unsigned n = (unsigned)__popc(ma);
  const unsigned incl = wave_incl_scan(n);
  const unsigned tot = readlane_u32(incl, 63);
  unsigned at = 0u;
  if (lane_id() == 0 && tot) at = atomicAdd(&ts.ng, tot);
  return readlane_u32(at, 0) + incl - n;
}
// sink(place, composite) for the marked slots.
template <typename Tin, int BT, class F>
__device__ __forceinline__ void each_marked(const RowView<Tin, true, BT>& rv, uint32_t ma, unsigned at, F sink) {
  constexpr int EPV = Elem<Tin>::EPV;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++)
    if ((ma >> q) & 1u)
      sink(at++, comp_key(tg_key(rv.y[q]), rv.r.v0 + ((int)threadIdx.x + (q / EPV) * BT) * EPV + q % EPV));
}
// From any other view: one at a time.
template <class View, int BT, class F>
__device__ __forceinline__ void gather(const View& rv, const Plan& pl, float m, Scratch<BT>& ts, F sink) {
  rv.each([&](int id, float y) {
    const int l = pl.list(bucket::of(y, m));
    if (l < 0) return;
    const unsigned at = atomicAdd(&ts.ng, l == 0 ? 1u : 0x10000u);
    sink(l, l == 0 ? at & 0xFFFFu : at >> 16, comp_key(tg_key(y), id));
  });
}

// The drawn composite once tl.L holds lists A and B (every thread; a barrier
// between the gather and the call); settles the cut.  Lists of at most 64
// ids are ranked side by side by two waves.
template <int BT>
__device__ __forceinline__ u64 pick_gathered(Plan& pl, float top_p, Tail& tl, Scratch<BT>& ts, BlockScratch& bs) {
  const float m = tl.m;
  u64 P = pl.P, Sp = pl.Sp;
  const int w = (int)threadIdx.x >> 6;
  const bool ra = pl.na <= 64u, rb = pl.nb <= 64u;  // (uniform)
  if (ra && w == 0) bucket::wave_rank64(tl.L, pl.na, m, tl.R, tl.Q);
  if (rb && w == 1) bucket::wave_rank64(tl.L + pl.ob, pl.nb, m, tl.R2, tl.Q2);
  __syncthreads();
  u64 before;
  unsigned rank;
  const u64 before_a = bucket::mass_before(tl.MI, pl.a0);
  if (pl.k_search) {
    // the top-k set's last element: S, then P or S'
    const unsigned ik = pl.nv - bucket::count_before(tl.CI, pl.a0);  // its place in list A
    u64 last;
    if (ra) {
      last = tl.R[ik - 1];
      pl.S = before_a + tl.Q[ik - 1];
    } else {
      last = select_list<BT, true>(tl.L, pl.na, m, ik, &before, &rank, tl.R, tl.Q, ts, bs);
      pl.S = before_a + before + bucket::mass_c(last, m);
    }
    if (pl.cut_last) {
      pl.cutc = last;
      Sp = pl.S;
    } else if (pl.cut_search) {
      P = mul_shr24(pl.S, (uint32_t)(top_p * 16777216.0f));
    }
  }
  if (pl.cut_search) {
    const u64 target = P - before_a;
    if (ra) {
      const int i = bucket::first_rank_once(tl.Q, pl.na, target, &ts.first2);
      pl.cutc = tl.R[i];
      before = i > 0 ? tl.Q[i - 1] : 0ull;
      rank = (unsigned)i;
    } else {
      pl.cutc = select_list<BT>(tl.L, pl.na, m, target, &before, &rank, tl.R, tl.Q, ts, bs);
    }
    Sp = before_a + before + bucket::mass_c(pl.cutc, m);
    pl.ntopp = bucket::count_before(tl.CI, pl.a0) + rank + 1u;
  }
  pl.Sp = Sp;
  const u64 t = mul_shr24(Sp, pl.uq);
  if (pl.nb > 0u) {
    const u64 target = t + 1 - bucket::mass_before(tl.MI, pl.b0);
    if (rb) return tl.R2[bucket::first_rank_once(tl.Q2, pl.nb, target, &ts.first)];
    return select_list<BT>(tl.L + pl.ob, pl.nb, m, target, &before, &rank, tl.R2, tl.Q2, ts, bs);
  }
  const u64 target = t + 1 - before_a;
  if (ra) return tl.R[bucket::first_rank_once(tl.Q, pl.na, target, &ts.first)];
  return select_list<BT>(tl.L, pl.na, m, target, &before, &rank, tl.R2, tl.Q2, ts, bs);
}

// The same without the one-gather guarantee: the top-k set's end (when it
// lies inside a bucket), the cut, then the draw, each one's bucket gathered
// from the view (or radix selected beyond CAPL ids): three passes over the
// row.  (Radix selections over the whole row, for rows with a top-k, read it
// about twenty times: 1024 rows of 128,256 fp32 ids with k above 1024 took
// 9.6 ms.)
template <int BT, class View>
__device__ __forceinline__ u64 pick_resolved(Plan& pl, float top_p, const View& rv, Tail& tl, Scratch<BT>& ts,
                                             BlockScratch& bs) {
  u64 before;
  unsigned rank;
  if (pl.k_search) {
    u64 mass;
    const u64 last = resolve_count<BT>(rv, tl, pl.bp, pl.nv - bucket::count_before(tl.CI, pl.bp), &mass, ts, bs);
    pl.S = bucket::mass_before(tl.MI, pl.bp) + mass;
    if (pl.cut_last) {
      pl.cutc = last;
      pl.Sp = pl.S;
    } else if (pl.cut_search) {
      pl.P = mul_shr24(pl.S, (uint32_t)(top_p * 16777216.0f));
      pl.bp = bucket::find_mass<BT>(tl.MI, pl.P, &ts.sel[0]);
    }
  }
  if (pl.cut_search) {
    pl.cutc = resolve_mass<BT>(rv, tl, pl.bp, pl.P - bucket::mass_before(tl.MI, pl.bp), &before, &rank, ts, bs);
    pl.Sp = bucket::mass_before(tl.MI, pl.bp) + before + bucket::mass_c(pl.cutc, tl.m);
    pl.ntopp = bucket::count_before(tl.CI, pl.bp) + rank + 1;
  }
  const u64 t = mul_shr24(pl.Sp, pl.uq);
  const int bt = bucket::find_mass<BT>(tl.MI, t + 1, &ts.sel[1]);
  return resolve_mass<BT>(rv, tl, bt, t + 1 - bucket::mass_before(tl.MI, bt), &before, &rank, ts, bs);
}

// The id and the diagnostics of a settled sampling row without a top-k, or
// with one above KMAX (no kept list).
template <int BT, class View>
__device__ __forceinline__ void write_row(const SampleArgs& a, int b, Plan& pl, u64 pick, const View& rv,
                                          Scratch<BT>& ts) {
  if (pl.cut_last && !pl.k_search && a.dbg.cut_ids) {
    u64 x = 0;
    rv.each([&](int id, float y) {
      const u64 v = ~comp_key(tg_key(y), id);
      x = v > x ? v : x;
    });
    pl.cutc = ~block_reduce_max<BT>(x, ts.red64);
  }
  if (threadIdx.x == 0) {
    a.out[b] = comp_id(pick);
    write_row_diag(a, b, (int)pl.nv, (int)pl.ntopp, pl.S, pl.Sp, comp_id(pl.cutc));
  }
  if (a.dbg.kept_ids)
    for (int i = threadIdx.x; i < a.dbg.kept_cap; i += BT) a.dbg.kept_ids[(long long)b * a.dbg.kept_cap + i] = -1;
  if (a.dbg.kept_probs)
    for (int i = threadIdx.x; i < a.dbg.kept_cap; i += BT) a.dbg.kept_probs[(long long)b * a.dbg.kept_cap + i] = 0.0f;
}

// The kept list of a row with 1 <= top_k <= KMAX: sorted[0, n) its top-k set
// in order, the first ntopp of them with their probabilities.
template <int BT>
__device__ __forceinline__ void write_kept(const SampleArgs& a, int b, const u64* sorted, int n, int ntopp, u64 Sp,
                                           float m) {
  if (a.dbg.kept_ids) {
    int32_t* kid = a.dbg.kept_ids + (long long)b * a.dbg.kept_cap;
    for (int i = threadIdx.x; i < a.dbg.kept_cap; i += BT) kid[i] = i < n ? comp_id(sorted[i]) : -1;
  }
  if (a.dbg.kept_probs) {
    float* kp = a.dbg.kept_probs + (long long)b * a.dbg.kept_cap;
    const float fs = tg_u64_to_f32(Sp);
    for (int i = threadIdx.x; i < a.dbg.kept_cap; i += BT)
      kp[i] = i < ntopp ? kept_prob(comp_y(sorted[i]), m, fs) : 0.0f;
  }
}

// A greedy row (the largest composite Mc), or a row with nothing allowed
// (Mc 0: id -1).
template <int BT>
__device__ __forceinline__ void write_greedy(const SampleArgs& a, const Row& r, u64 Mc) {
  const int b = r.b;
  const int id = Mc ? comp_id(Mc) : -1;
  if (threadIdx.x == 0) {
    a.out[b] = id;
    write_row_diag(a, b, id >= 0, id >= 0, 0, 0, id);
  }
  if (a.dbg.kept_ids)
    for (int i = threadIdx.x; i < a.dbg.kept_cap; i += BT)
      a.dbg.kept_ids[(long long)b * a.dbg.kept_cap + i] = (i == 0 && r.mode == 0) ? id : -1;
  if (a.dbg.kept_probs)
    for (int i = threadIdx.x; i < a.dbg.kept_cap; i += BT)
      a.dbg.kept_probs[(long long)b * a.dbg.kept_cap + i] = (i == 0 && r.mode == 0 && id >= 0) ? 1.0f : 0.0f;
}

// The dynamic LDS both kernels carve up: the row's history bits and hash,
// then the tail's arrays.
__device__ __forceinline__ Tail carve(const SampleArgs& a, unsigned char* smem, uint32_t*& hbits, int2*& hash, int& bw) {
  bw = a.TS > 0 ? (a.V + 31) / 32 : 0;
  hbits = (uint32_t*)smem;
  hash = (int2*)(smem + ((bw * 4 + 15) / 16) * 16);
  Tail tl;
  tl.L = (u64*)((unsigned char*)hash + (size_t)a.TS * 8);  // CAPL
  tl.R = tl.L + CAPL;                                       // 64 each
  tl.Q = tl.R + 64;
  tl.R2 = tl.Q + 64;
  tl.Q2 = tl.R2 + 64;
  tl.CI = (unsigned*)(tl.Q2 + 64);                          // NB + 1 (+ pad)
  tl.MI = (u64*)(tl.CI + NB + 4);                           // NB + 1
  tl.E = (Packed*)(tl.MI + NB + 1);                         // a.topp_cap
  return tl;
}

// Pass 1 over the register-resident ids: the thread's largest composite (0:
// nothing allowed).  Branch free: a thread's ids rise with the slot, so a
// strict > keeps the smallest id among its equal maxima (the slot is
// tracked, and its id formed once).
template <typename Tin, int BT>
__device__ __forceinline__ u64 thread_best(const RowView<Tin, true, BT>& rv) {
  constexpr int EPV = Elem<Tin>::EPV;
  float mx = -__builtin_inff();
  int mq = 0;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) {
    const float y = rv.y[q];
    const bool gt = y > mx;
    mq = gt ? q : mq;
    mx = gt ? y : mx;
  }
  const int mid = rv.r.v0 + ((int)threadIdx.x + (mq / EPV) * BT) * EPV + mq % EPV;
  return mx > -__builtin_inff() ? comp_key(tg_key(mx), mid) : 0ull;
}

// The key of the thread's second largest id (0: fewer than two allowed).
template <typename Tin, int BT>
__device__ __forceinline__ uint32_t thread_second(const RowView<Tin, true, BT>& rv) {
  float m1 = -__builtin_inff(), m2 = -__builtin_inff();
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) {
    const float y = rv.y[q];
    m2 = fmaxf(m2, fminf(m1, y));
    m1 = fmaxf(m1, y);
  }
  return m2 > -__builtin_inff() ? tg_key(m2) : 0u;
}

}  // namespace topp
}  // namespace tgs
