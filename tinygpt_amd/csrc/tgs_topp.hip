// tgs_topp.hip -- rows that sample with top-p over the whole vocabulary (top_k
// disabled: k <= 0 or k >= V) and fit one workgroup's registers (V <= 32768;
// tgs_topp_split.hip takes longer ones), one workgroup of 1024 threads per row; in a
// launch that serves the whole batch (every sampling row without a top-k),
// the greedy rows too.
//
// The contract keeps the smallest prefix of the allowed ids in (y desc,
// id asc) order whose exact mass reaches P = floor(S p24 / 2^24) and draws
// the first id whose inclusive prefix exceeds t = floor(S' u24 / 2^24);
// masses are q = floor(exp(y - m) 2^40).  Only ids with q > 0 can be the cut
// or the draw (both are where the prefix grows), and those lie within 32 of
// the maximum.  So:
//
//   pass 1  y (mask, penalties, 1/T): the largest composite (its y is the
//           maximum m; it is the answer of a greedy row) and the allowed
//           count;
//   pass 2  per allowed id its bucket below m (width 1/32, tgs_bucket.h)
//           and mass q, into a count and mass histogram; block prefixes
//           over the buckets locate the bucket of the cut and then of the
//           draw;
//   pass 3  gather the ids of the cut's bucket and of the buckets the draw
//           can fall into (S' lies in the cut's bucket, so its targets span
//           one or two) into LDS, rank them (a wave sort for at most 64),
//           scan their masses in rank order and pick the elements.
//
// The row is held in registers (32 ids per thread) after one read; only the
// rare paths below stream it again from L2 / MALL.
//
// More than CAPL ids in those buckets (a flat row: ties, tiny temperature
// spreads): the cut is resolved first and the draw after it, a crowded
// bucket by a mass-weighted radix selection restricted to it (a few more
// passes).  exp runs once per id (plus once per ranked id).
#include "tgs_topp.h"

namespace tgs {
namespace topp {

constexpr int BT = TOPP_NT;    // threads per workgroup
constexpr int WT = BT / 64;    // waves

// The row after pass 1 (m, the largest composite Mc, nv allowed ids): the
// mass histogram, the cut and the draw over the allowed ids of view v.
template <class View>
__device__ __forceinline__ void topp_rest(const SampleArgs& a, const Row& r, const View& rv, Tail& tl, u64 Mc,
                                          unsigned nv, Scratch<BT>& ts, BlockScratch& bs) {
  histogram(rv, tl);
  __syncthreads();
  bucket::prefix<BT>(tl.CI, tl.MI, ts.red32, ts.red64);
  Plan pl;
  plan_row<BT>(pl, r, tl, Mc, nv, ts);
  u64 pick;
  if (pl.one) {
    gather(rv, pl, tl.m, ts, [&](int l, unsigned o, u64 x) { tl.L[l ? pl.ob + o : o] = x; });
    __syncthreads();
    pick = pick_gathered<BT>(pl, r.top_p, tl, ts, bs);
  } else {
    pick = pick_resolved<BT>(pl, r.top_p, rv, tl, ts, bs);
  }
  write_row<BT>(a, r.b, pl, pick, rv, ts);
}

template <typename Tin>
__device__ __forceinline__ void topp_row(const SampleArgs& a, Row& r, unsigned char* smem, Scratch<BT>& ts,
                                         BlockScratch& bs, const uint4 (&raw)[RowView<Tin, true, BT>::NV],
                                         const uint32_t (&mw)[RowView<Tin, true, BT>::NV]) {
  const int b = r.b;
  uint32_t* hbits;
  int2* hash;
  int bw;
  Tail tl = carve(a, smem, hbits, hash, bw);
  r.v0 = 0;
  r.v1 = a.V;
  if (r.use_pen) hash_build<BT>(a, r, hash, hbits, bw);
  RowView<Tin, true, BT> rv(a, r, hash, hbits, (const Tin*)a.logits + (long long)b * a.row_stride);
  rv.load(raw, mw);
  if (a.dbg.post_logits) {
    float* post = a.dbg.post_logits + (long long)b * a.V;
    for (int v = threadIdx.x; v < a.V; v += BT) post[v] = -__builtin_inff();
    __syncthreads();
    rv.each([&](int id, float y) { post[id] = y; });
  }

  // pass 1: the largest composite (the greedy answer; its y is the maximum m)
  // and the allowed count
  u64 mcl = thread_best<Tin, BT>(rv);
  for (int i = threadIdx.x; i < NB + 1; i += BT) {
    tl.CI[i] = 0u;
    tl.MI[i] = 0ull;
  }
  const unsigned nown = rv.nallowed;  // this thread's allowed ids
  const unsigned wincl = wave_incl_scan(nown);  // lane 63: the wave's allowed ids
  mcl = wave_max(mcl);
  if (lane_id() == 63) {
    ts.red64[threadIdx.x >> 6] = mcl;
    ts.red32[threadIdx.x >> 6] = wincl;
  }
  __syncthreads();
  u64 Mc = 0;
  unsigned nv = 0, wbase = 0;  // wbase: allowed ids of the waves before this one
#pragma unroll
  for (int i = 0; i < WT; i++) {
    Mc = ts.red64[i] > Mc ? ts.red64[i] : Mc;
    wbase += i < (int)(threadIdx.x >> 6) ? ts.red32[i] : 0u;
    nv += ts.red32[i];
  }
  if (nv == 0 || r.mode == 0) {
    write_greedy<BT>(a, r, nv ? Mc : 0ull);
    return;
  }
  tl.m = comp_y(Mc);
  if (nv <= (unsigned)a.topp_cap) {
    // few allowed ids (a grammar mask): they alone, packed into LDS, feed
    // every later pass (the exact exp and the bucket gathers run on allowed
    // ids only), in wave order: a thread's slots follow the allowed ids of
    // the waves and lanes before it
    Packed* dst = tl.E + (wbase + wincl - nown);
    rv.each([&](int id, float y) { *dst++ = Packed{y, id}; });
    __syncthreads();
    topp_rest(a, r, CompactView<BT>{tl.E, (int)nv}, tl, Mc, nv, ts, bs);
    return;
  }
  topp_rest(a, r, rv, tl, Mc, nv, ts, bs);
}

template <typename Tin>
__global__ __launch_bounds__(BT) void topp_kernel(SampleArgs a) {
  TGS_DYN_SMEM(smem);
  __shared__ Scratch<BT> ts;
  __shared__ BlockScratch bs;
  const int b = blockIdx.x;
  if (b >= a.B) return;
  // the row's parameters (scalar loads) requested before its vectors, so
  // that they arrive first.  The mask words wait for them (the first request
  // takes about a microsecond): the row's first NPRE vectors go out before
  // the words, the rest after them, so that neither the row's stream waits
  // for the parameters nor the words for the whole row (the vectors are
  // evaluated in order, each with its word).
  using RV = RowView<Tin, true, BT>;
  constexpr int NPRE = RV::NV < TOPP_MASK_PRE ? RV::NV : TOPP_MASK_PRE;
  const tgs_row_params p = a.params[b];
  const float ub = a.u[b];
  const int hl = a.hist_len ? a.hist_len[b] : a.hist_cap;
  const Tin* rowp = (const Tin*)a.logits + (long long)b * a.row_stride;
  uint4 raw[RV::NV];
  RV::template fetch<0, NPRE>(rowp, 0, a.V, raw);
  Row r;
  const bool valid = row_setup_from(a, b, 0, p, ub, hl, r);
  const bool mine = valid && (r.mode == 2 ? !(r.k >= 1 && r.k < a.V) : (r.mode == 0 && a.topp_all));
  if (!mine) {
    // other kernels' rows; in a launch that serves the whole batch, invalid
    // rows (-2) and rows outside the hint (-3)
    if (a.topp_all && threadIdx.x == 0) {
      a.out[b] = valid ? -3 : -2;
      write_row_diag(a, b, 0, 0, 0, 0, -1);
    }
    return;
  }
  uint32_t mw[RV::NV];
  RV::mask_words(r, 0, a.V, mw);
  RV::template fetch<NPRE, RV::NV>(rowp, 0, a.V, raw);
  RV::fix_tail(rowp, 0, a.V, raw);
  topp_row<Tin>(a, r, smem, ts, bs, raw, mw);
}

}  // namespace topp

int topp_resident_ids() { return TOPP_NT * topp::RES_EPT; }

size_t topp_lds_bytes(int V, int TS) {
  const int bw = TS > 0 ? (V + 31) / 32 : 0;
  return (size_t)((bw * 4 + 15) / 16) * 16 + (size_t)TS * 8 + (size_t)(TOPP_CAP + 4 * 64) * 8 +
         (size_t)(bucket::NB + 4) * 4 + (size_t)(bucket::NB + 1) * 8;
}

int topp_pack_cap(int V, int TS, size_t lds_avail) {
  const size_t base = topp_lds_bytes(V, TS);
  if (lds_avail <= base) return 0;
  const size_t n = (lds_avail - base) / sizeof(topp::Packed);
  return (int)(n < (size_t)V ? n : (size_t)V);
}

hipError_t launch_topp(const SampleArgs& a, int dtype, hipStream_t st) {
  const size_t lds = topp_lds_bytes(a.V, a.TS) + (size_t)a.topp_cap * sizeof(topp::Packed);
  const dim3 g(a.B), blk(TOPP_NT);
  if (dtype == 1) hipLaunchKernelGGL((topp::topp_kernel<uint16_t>), g, blk, lds, st, a);
  else hipLaunchKernelGGL((topp::topp_kernel<float>), g, blk, lds, st, a);
  return hipGetLastError();
}

hipError_t set_topp_lds_limit(size_t bytes) {
  const void* fns[] = {(const void*)topp::topp_kernel<float>, (const void*)topp::topp_kernel<uint16_t>};
  hipError_t e = hipSuccess;
  for (const void* f : fns) {
    hipError_t e2 = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e2 != hipSuccess) e = e2;
  }
  return e;
}

}  // namespace tgs
