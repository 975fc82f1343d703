// tgs_topp_split.hip -- every kind of row over S workgroups of 512 threads, in
// one launch: rows without a top-k too long for one workgroup's registers
// (tgs_topp.hip holds the others), with the batch's greedy rows where the hint
// says so, and whole batches of every kind from 4,097 ids on (split_takes,
// tgs_api.hip).  A row of one chunk skips the exchanges.
//
// What bounds it: one workgroup streams a row at one CU's rate and evaluates
// every id's exact mass (about 40 VALU operations) on one CU, three passes
// over the row from L2: 130 - 150 us for a row of 128,256 fp32 or 151,936
// bf16 ids, whatever the batch, on a chip of 256 CUs.  Here workgroup (b, c)
// reads ids [c L, (c + 1) L) of row b once, into registers (32 per thread at
// most), and the row's workgroups meet three times through device memory:
//
//   1. Each publishes its chunk's largest composite and polls the row's S of
//      them: m, the row's maximum.  A poll that runs out (its partners are
//      not running yet) reads the other chunks itself instead.
//   2. Each builds the count and mass histogram of its chunk below m in LDS
//      (tgs_topp.h), stores it to its slab of the workspace, waits for the
//      stores and counts itself in the row's arrival counter.  The last to
//      arrive owns the row: it sums the S slabs, places the cut's and the
//      draw's buckets, and publishes them.
//   3. The others poll that decision, gather the buckets' ids of their
//      chunk from registers, publish them and their counts, and leave.  One
//      whose poll runs out says so and leaves, and the owner reads that
//      chunk itself (as it does for a chunk with more ids of a bucket than a
//      list holds).  The owner ranks the lists and finishes the row.
//
// No wait depends on a workgroup that has not started: the polls of steps 1
// and 3 are bounded, and the owner waits only for workgroups that have
// arrived, whose polls are bounded.  So any grid is safe, whatever else runs
// on the device; the rows of a group of 8 are consecutive workgroups, so a row's
// chunks run together.
//
// The exchange uses agent-scope loads and stores throughout (they pass the
// per-XCD L2s, which are not coherent with each other) and plain waits for
// the issuing wave's stores; no fence is issued (an agent-scope fence writes
// back or invalidates a whole L2).  Words carry the call's epoch, and the
// row's owner leaves none behind that a later call could take for its own
// (reset_line).
//
// Measured against one workgroup per row streaming it three times (per call):
// 1 row of 151,936 bf16 ids with penalties 137 -> 31 us, 32 rows of 128,256
// fp32 ids 141 -> 27 us.  What bounds it now is the chain (stamps of the
// second, us from the first workgroup's entry): logits in registers 4.7,
// row's maximum 7.1, histogram 12.1 (the exact exp and two LDS atomics per
// id), slabs out and counted 13.8, slabs summed 16.0, decision 17.6, lists in
// 23.2, row written 25.5.  Chunks: at most 16384 ids (32 per thread; more
// spill), about one workgroup per CU, at least 4096 ids.
#include <algorithm>

#include "tgs_topp.h"

namespace tgs {
namespace topp {

constexpr int SBT = TOPPS_NT;
constexpr uint32_t STAG = 0x3FFFu;    // epoch bits a maximum carries
constexpr uint32_t SIDM = 0x3FFFFu;   // its id bits (V <= 2^18)
constexpr uint32_t DONE_LEFT = 1u << 30;  // the chunk's lists were not published

struct SplitShared {
  Scratch<SBT> ts;
  BlockScratch bs;
  u64 rowmax;
  uint32_t done[TOPPS_MAX_SPLIT];
  uint32_t wkey[2][SBT / 64][SBT / 64];  // per bound: [m - 1][wave]: the wave's ceil(k / m)-th largest thread maximum
  u64 slots[SBT / 64][64];               // wave lists (the ranked top-k of at most 64)
  uint32_t floor;
  u64 word;
  uint32_t arrived;
  int flag;
};

// Stores of this wave have reached device memory (an agent-scope store is
// written through, and counts as outstanding until then).
__device__ __forceinline__ void wait_stores() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

template <typename T>
__device__ __forceinline__ T ld(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The decision word (see pack_plan) without lists to gather.
__device__ __forceinline__ u64 decision_tag(uint32_t ep) { return (u64)(ep & 0xFFFFFFu) << 40; }

// A chunk's largest composite with the epoch's low bits between key and id
// (never 0; entries of one call order as their composites; key 0: nothing
// allowed).
__device__ __forceinline__ u64 max_entry(u64 x, uint32_t ep) {
  const uint32_t id = x ? (uint32_t)comp_id(x) : 0u;
  return (x & 0xFFFFFFFF00000000ull) | ((u64)(ep & STAG) << 18) | (u64)(SIDM - id);
}
__device__ __forceinline__ bool max_current(u64 e, uint32_t ep) {
  return e != 0ull && (uint32_t)((e >> 18) & STAG) == (ep & STAG);
}

// The composite of the largest entry (0: nothing allowed).
__device__ __forceinline__ u64 max_comp(u64 e) {
  return (e >> 32) ? comp_key((uint32_t)(e >> 32), (int)(SIDM - (uint32_t)(e & SIDM))) : 0ull;
}

// Ready for the next call: counter zero, maxima and done words cleared, epoch
// advanced (every workgroup of the row has arrived, so nothing polls the maxima), and
// a decision of this epoch with nothing to gather.  Every ending of a row
// leaves one, so the word that a call finds is always its predecessor's, one
// epoch back: a word left from before (or never written, which reads as epoch
// 0) would pass for current once the 24 bits of the tag come round, after
// 2^24 calls whose rows had nothing to decide.  A workgroup that still polls
// finds what the owner published: one whose lists the owner waits for has
// left by now, and without lists the word is the same.  The done words are
// cleared for the same reason (the epoch itself comes round after 2^32
// calls); only one that says its workgroup left without lists can still be on
// its way, and the owner reads that chunk itself, which is right at any time.
__device__ __forceinline__ void reset_line(const SampleArgs& a, u64* line, uint32_t ep) {
  unsigned* cnt = (unsigned*)line;
  if (threadIdx.x < (unsigned)a.S) {
    st(line + 2 + threadIdx.x, (u64)0);
    st(line + 2 + TOPPS_MAX_SPLIT + threadIdx.x, (u64)0);
  }
  if (threadIdx.x == 0) {
    st(line + 1, decision_tag(ep));
    st(cnt, 0u);
    st(cnt + 1, ep == 0xFFFFFFFFu ? 0u : ep);
  }
}

// A wave polls the row's S words (one per chunk) until each is current;
// false after max_spins polls.  *e: lane c's word.
__device__ __forceinline__ bool poll_words(const u64* words, int S, uint32_t ep, int max_spins, u64* e) {
  const bool act = lane_id() < S;
  u64 x = 0ull;
  bool ok = false;
  for (int spins = 0;; spins++) {
    if (act && !max_current(x, ep)) x = ld(words + lane_id());
    ok = __ballot(act && !max_current(x, ep)) == 0ull;
    if (ok || spins >= max_spins) break;
    __builtin_amdgcn_s_sleep(1);
  }
  *e = act ? x : 0ull;
  return ok;
}

// Two floor keys (their top 23 bits: a floor may be lower) in one word with
// the epoch's tag where max_current looks for it.
__device__ __forceinline__ u64 floor_entry(uint32_t k1, uint32_t k2, uint32_t ep) {
  return (u64)(k1 >> 9) << 41 | (u64)((k2 >> 9) >> 14) << 32 | (u64)(ep & STAG) << 18 | (u64)(((k2 >> 9) & 0x3FFFu) << 4) | 1ull;
}
__device__ __forceinline__ uint32_t floor_key1(u64 e) { return (uint32_t)(e >> 41) << 9; }
__device__ __forceinline__ uint32_t floor_key2(u64 e) {
  return (((uint32_t)(e >> 32) & 0x1FFu) << 14 | ((uint32_t)e >> 4 & 0x3FFFu)) << 9;
}

// The sorted top 64 of L[0, n) in wave 0's lanes (slots: the waves' lists).
// Ends with a barrier.
__device__ __forceinline__ u64 top64(const u64* L, unsigned n, u64 (*slots)[64]) {
  u64 acc = 0ull;
  bool first = true;
  for (unsigned s0 = threadIdx.x & ~63u; s0 < n; s0 += SBT) {
    u64 x = s0 + lane_id() < n ? L[s0 + lane_id()] : 0ull;
    x = wave_sort_desc(x);
    acc = first ? x : wave_merge_top64(acc, x);
    first = false;
  }
  return merge_waves<SBT / 64>(acc, slots);
}

// A row with 1 <= top_k <= KMAX from L[0, n), which holds its top-k set (n <=
// CAPL; every allowed id when fewer than k are): finished by one wave up to
// 64 kept ids; otherwise the set is cut out of the list by its k-th element,
// and the cut and the draw selected by mass.
__device__ __forceinline__ void finish_topk(const SampleArgs& a, const Row& r, u64* L, unsigned n, Tail& tl,
                                            SplitShared& sh) {
  const unsigned k = (unsigned)r.k, kk = k < n ? k : n;
  if (kk <= 64u) {
    const u64 x = top64(L, n, sh.slots);
    if (threadIdx.x < 64) wave_finalize(a, r, (unsigned)lane_id() < kk ? x : 0ull, (int)kk);
    return;
  }
  constexpr int PER = (CAPL + SBT - 1) / SBT;
  u64 mx = 0ull;
  for (unsigned i = threadIdx.x; i < n; i += SBT) mx = L[i] > mx ? L[i] : mx;
  const u64 Mc = block_reduce_max<SBT>(mx, sh.ts.red64);
  const float m = comp_y(Mc);
  u64 before = 0;
  unsigned rank = 0;
  unsigned ntopp = kk;
  u64 T = 0ull;
  if (kk < n) T = select_list<SBT, true>(L, n, m, kk, &before, &rank, tl.R, tl.Q, sh.ts, sh.bs);
  u64 keep[PER];
  u64 S = 0, mn = ~0ull;
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const unsigned i = threadIdx.x + j * SBT;
    keep[j] = i < n ? L[i] : 0ull;
    if (keep[j] < T) keep[j] = 0ull;
    if (keep[j]) {
      S += bucket::mass_c(keep[j], m);
      mn = keep[j] < mn ? keep[j] : mn;
    }
  }
  if (threadIdx.x == 0) sh.ts.ng = 0;
  const u64 St = block_sum<u64, SBT>(S, sh.ts.red64);  // (its barriers also end the reads of L)
  u64 cutc = ~block_max<u64, SBT>(~mn, sh.ts.red64b);
#pragma unroll
  for (int j = 0; j < PER; j++)
    if (keep[j]) L[atomicAdd(&sh.ts.ng, 1u)] = keep[j];
  __syncthreads();
  u64 Sp = St;
  if (r.top_p < 1.0f) {
    const u64 P = mul_shr24(St, (uint32_t)(r.top_p * 16777216.0f));
    if (P == 0) {
      cutc = Mc;
      Sp = tg_q40(1.0f);
      ntopp = 1;
    } else {
      cutc = select_list<SBT>(L, kk, m, P, &before, &rank, tl.R, tl.Q, sh.ts, sh.bs);
      Sp = before + bucket::mass_c(cutc, m);
      ntopp = rank + 1;
    }
  }
  const u64 t = mul_shr24(Sp, (uint32_t)(r.u * 16777216.0f));
  const u64 pick = select_list<SBT>(L, kk, m, t + 1, &before, &rank, tl.R, tl.Q, sh.ts, sh.bs);
  if (threadIdx.x == 0) {
    a.out[r.b] = comp_id(pick);
    write_row_diag(a, r.b, (int)kk, (int)ntopp, St, Sp, comp_id(cutc));
  }
  if (a.dbg.kept_ids || a.dbg.kept_probs) {
    int n2 = 1;
    while (n2 < (int)kk) n2 <<= 1;
    for (int i = (int)kk + (int)threadIdx.x; i < n2; i += SBT) L[i] = 0ull;
    __syncthreads();
    block_bitonic_desc<SBT>(L, n2);
    write_kept<SBT>(a, r.b, L, (int)kk, (int)ntopp, Sp, m);
  }
}

// A y below the k-th largest (k <= the allowed ids, or -inf) of a row held by
// one workgroup, from counts per bucket of 1/32 below its maximum: for k
// above the thread count, which no thread maxima bound.  RN(m - y) <
// (q + 1) / 32 gives y > m - (q + 2) / 32, and so y >= its rounding.  CI and
// MI are zero before; ends with a barrier.
template <typename Tin>
__device__ __forceinline__ float counted_floor(const RowView<Tin, true, SBT>& rv, u64 mc, unsigned k, Tail& tl,
                                               SplitShared& sh) {
  const u64 Mc = block_reduce_max<SBT>(mc, sh.ts.red64);
  const float m = Mc ? comp_y(Mc) : 0.0f;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) {
    const float y = rv.y[q];
    const float f = y == m ? 0.0f : (m - y) * 32.0f;
    if (y > -__builtin_inff()) atomicAdd(&tl.CI[f < (float)NB ? (int)f : NB], 1u);
  }
  __syncthreads();
  bucket::prefix<SBT>(tl.CI, tl.MI, sh.ts.red32, sh.ts.red64);
  if (tl.CI[NB - 1] < k) return -__builtin_inff();
  const int q = bucket::find_count<SBT>(tl.CI, k, &sh.ts.sel[0]);
  return m - (float)(q + 2) * 0.03125f;
}

// The slots of a chunk's k largest composites, a bit each (floor_marks); the
// chunk holds at least k ids with y >= yb.  From its registers by bisection:
// first over the keys, until exactly k ids are at or above the middle, then,
// where several ids share the k-th key, over their ids.  mc: the thread's
// largest composite.  At most 32 and 18 rounds of one barrier each; radix
// digits over the chunk read again sent ties to one LDS bin (1 row of 128,256
// equal fp32 logits, k = 1000: 376 us).  ts.ng is 0 after it; starts and ends
// with a barrier.
template <typename Tin>
__device__ __forceinline__ uint32_t kth_marks(const RowView<Tin, true, SBT>& rv, u64 mc, unsigned k, float yb,
                                              SplitShared& sh) {
  constexpr int EPV = Elem<Tin>::EPV;
  const int w = threadIdx.x >> 6;
  unsigned turn = 0;
  // the workgroup's sum of n (two sets of words in turn: one barrier)
  auto sum = [&](unsigned n) -> unsigned {
    n = wave_sum(n);
    uint32_t* words = sh.wkey[turn & 1u][0];
    turn++;
    if (lane_id() == 0) words[w] = n;
    __syncthreads();
    n = 0;
#pragma unroll
    for (int v = 0; v < SBT / 64; v++) n += words[v];
    return n;
  };
  const uint32_t mx = (uint32_t)(block_reduce_max<SBT>(mc, sh.ts.red64) >> 32);
  if (threadIdx.x == 0) sh.ts.ng = 0;
  // the largest key with k ids at or above it: in [lo, hi)
  uint32_t lo = yb > -__builtin_inff() ? tg_key(yb) : 0x00800000u, hi = mx + 1u;
  unsigned above = 0;  // ids at or above hi
  bool met = false;    // exactly k ids at or above lo
  while (hi - lo > 1u && !met) {
    const uint32_t mid = lo + (hi - lo) / 2u;
    const float ym = tg_unkey(mid);
    unsigned n = 0;
#pragma unroll
    for (int q = 0; q < RES_EPT; q++) n += rv.y[q] >= ym ? 1u : 0u;
    n = sum(n);
    if (n >= k) {
      lo = mid;
      met = n == k;
    } else {
      hi = mid;
      above = n;
    }
  }
  const float yk = tg_unkey(lo);
  uint32_t gt = 0u, eq = 0u;
#pragma unroll
  for (int q = 0; q < RES_EPT; q++) {
    gt |= rv.y[q] > yk ? 1u << q : 0u;
    eq |= rv.y[q] == yk ? 1u << q : 0u;
  }
  // the least offset in the chunk up to which the ids of that key make up the
  // rest, in (a, z]: a thread's offsets rise with the slot
  int a = -1, z = rv.r.v1 - rv.r.v0 - 1;
  auto upto = [&](int last) -> uint32_t {
    const int o = last - (int)threadIdx.x * EPV;  // slot q: offset (q / EPV) SBT EPV + q % EPV
    if (o < 0) return 0u;
    const int n = o / (SBT * EPV) * EPV + min(o % (SBT * EPV) + 1, EPV);
    return n >= 32 ? eq : eq & ((1u << n) - 1u);
  };
  while (z - a > 1 && !met) {
    const int mid = a + (z - a) / 2;
    if (above + sum((unsigned)__popc(upto(mid))) >= k) z = mid;
    else a = mid;
  }
  __syncthreads();
  return gt | upto(z);
}

// The decision word: the epoch's low 24 bits over the list buckets in 40
// (bit 0: they are to be gathered; a run of 512 buckets or more for list B is
// settled by the owner alone).  Every ending of a row leaves the word with
// its epoch (reset_line), so a stale one is the previous call's.
__device__ __forceinline__ bool packs(const Plan& pl) { return pl.one && pl.b1 - pl.b0 < 511; }
__device__ __forceinline__ u64 pack_plan(const Plan& pl) {
  return 1ull | (u64)pl.a0 << 1 | (u64)pl.a1 << 11 | (u64)pl.b0 << 21 | (u64)(pl.b1 - pl.b0 + 1) << 31;
}
__device__ __forceinline__ Plan unpack_plan(u64 d) {
  Plan pl;
  pl.a0 = (int)((d >> 1) & 0x3FFu);
  pl.a1 = (int)((d >> 11) & 0x3FFu);
  pl.b0 = (int)((d >> 21) & 0x3FFu);
  pl.b1 = pl.b0 + (int)((d >> 31) & 0x1FFu) - 1;
  return pl;
}
__device__ __forceinline__ bool decided(u64 d, uint32_t ep) { return (uint32_t)(d >> 40) == (ep & 0xFFFFFFu); }

template <typename Tin>
__global__ __launch_bounds__(SBT) void topps_kernel(SampleArgs a) {
  TGS_DYN_SMEM(smem);
  TGS_STATIC_SMEM(SplitShared, sh);
  using RV = RowView<Tin, true, SBT>;
  using SV = RowView<Tin, false, SBT>;
  constexpr int NPRE = RV::NV < TOPP_MASK_PRE ? RV::NV : TOPP_MASK_PRE;
  // Workgroups are dealt out to the 8 XCDs in turn: the rows of a group of 8
  // alternate, so that a row's chunks share an XCD and the rows' owners (most
  // often the last chunk's workgroup) are on all of them.  Row by row, with 8
  // chunks, nearly all owners were on one XCD: 300 rows of 128,256 fp32 with
  // k up to 1024 under masks of one chunk's ids took 276 us, now 179; with k
  // above 1024 (the owner reads the row many times) 4845 and 2837.
  // (The divisions by 8 S and by the last group's rows are multiplications:
  // one integer division is 40 dependent operations ahead of the first load.)
  const int g0 = (int)__umulhi(blockIdx.x, a.div8s) * 8, p8 = (int)blockIdx.x - g0 * a.S;
  const bool full = g0 + 8 <= a.rows;
  const int c = full ? p8 >> 3 : (int)((unsigned)p8 * a.divg >> 16);
  const int lb = g0 + p8 - c * (full ? 8 : a.rows - g0);
  const int b = a.row0 + lb;
  if (b >= a.B) return;
  const int w = threadIdx.x >> 6, lane = lane_id();
  const int v0 = c * a.L, v1 = min(a.V, v0 + a.L);  // a.L a multiple of 64
  const tgs_row_params p = a.params[b];
  const float ub = a.u[b];
  const int hl = a.hist_len ? a.hist_len[b] : a.hist_cap;
  const Tin* rowp = (const Tin*)a.logits + (long long)b * a.row_stride;
  // the row's exchange line: counter and epoch, the decision, the chunk
  // maxima, the done words
  u64* line = a.tp_lines + (long long)b * TOPPS_LINE;
  unsigned* cnt = (unsigned*)line;
  u64* decision = line + 1;
  u64* maxima = line + 2;
  u64* done = line + 2 + TOPPS_MAX_SPLIT;
  const uint32_t epw = ld(cnt + 1);
  uint4 raw[RV::NV];
  RV::template fetch<0, NPRE>(rowp, v0, v1, raw);
  Row r;
  const bool valid = row_setup_from(a, b, c, p, ub, hl, r);
  const bool has_k = r.k >= 1 && r.k < a.V;
  const bool mine = valid && (a.topp_all ? r.mode == 0 || (r.mode == 2 && !has_k) : !outside_hint(a, r));
  if (!mine) {  // invalid rows (-2) and rows outside the hint (-3)
    if (c == 0 && threadIdx.x == 0) {
      a.out[b] = valid ? -3 : -2;
      write_row_diag(a, b, 0, 0, 0, 0, -1);
    }
    return;
  }
  uint32_t mw[RV::NV];
  RV::mask_words(r, v0, v1, mw);
  RV::template fetch<NPRE, RV::NV>(rowp, v0, v1, raw);
  RV::fix_tail(rowp, v0, v1, raw);
  const uint32_t ep = epw + 1u;  // never 0: the epoch word never holds ~0
  uint32_t* hbits;
  int2* hash;
  int bw;
  Tail tl = carve(a, smem, hbits, hash, bw);
  r.v0 = 0;
  r.v1 = a.V;
  if (r.use_pen) hash_build<SBT>(a, r, hash, hbits, bw);  // the whole row's: a chunk read again needs them
  for (int i = threadIdx.x; i < NB + 1; i += SBT) {
    tl.CI[i] = 0u;
    tl.MI[i] = 0ull;
  }
  Row rc = r;
  rc.v0 = v0;
  rc.v1 = v1;
  RV rv(a, rc, hash, hbits, rowp);
  rv.load(raw, mw);
  if (a.dbg.post_logits) {
    constexpr int EPV = RV::EPV;
    float* post = a.dbg.post_logits + (long long)b * a.V;
#pragma unroll
    for (int q = 0; q < RES_EPT; q++) {
      const int id = v0 + ((int)threadIdx.x + (q / EPV) * SBT) * EPV + q % EPV;
      if (id < v1) post[id] = rv.y[q];
    }
  }

  // a top-k past one wave's lists (of one chunk), or past what S short lists
  // hold, whose kept list nobody asked for goes through the histograms like a
  // larger one: the list's cut, mass and draw each select by digits, and lists
  // beyond CAPL select the set first.  Lists alone, now that a chunk's exact top
  // k is a bisection, are about level: 223 rows of 7,325 bf16 ids with k up to
  // 1024 31.1 us (30.3 with this rule), 41 mixed rows of 11,008 fp32 35.4
  // (32.0), 41 of 11,008 with k up to 1024 31.9 (35.2)
  const bool hist_k = r.k > (a.S == 1 ? 64 : 256 * a.S) && !a.dbg.kept_ids && !a.dbg.kept_probs;
  u64 mc = thread_best<Tin, SBT>(rv);
  u64* slab = a.ws + ((long long)lb * a.S + c) * TOPPS_PAIR;
  const u64* slabs = a.ws + (long long)lb * a.S * TOPPS_PAIR;
  if (threadIdx.x == 0) sh.ts.ng = 0;

  if (r.mode == 1 && !hist_k) {
    // ---- a top-k of at most KMAX: the chunk's ids that reach a floor under
    // the row's k-th largest y, and no more meetings.  Floors from the thread
    // maxima (bound_key): the chunk's own k-th largest, or, when S lists of
    // that many would be too long (meet), the lowest over the chunks of each
    // one's ceil(k / S)-th largest, or the highest of their k-th (the better one
    // where a mask or an order leaves the row's largest ids to few chunks).
    const bool counted = a.S == 1 && 4 * r.k > 3 * SBT;
    const bool meet = a.S > 1 && (2 * a.S * r.k > CAPL || 2 * r.k > SBT);
    const int k2 = (r.k + a.S - 1) / a.S;
    // (k > SBT: the ceil(k / 2)-th largest of the threads' second maxima has k
    // ids at or above it)
    const bool two = r.k > SBT;
    const int k1 = two ? (r.k + 1) / 2 : r.k;
    const uint32_t srt = wave_sort_desc((uint32_t)(mc >> 32));
    const uint32_t srt1 = two ? wave_sort_desc(thread_second(rv)) : srt;
#pragma unroll
    for (int q = 1; q <= SBT / 64; q++) {
      const int at = (k1 + q - 1) / q - 1, at2 = (k2 + q - 1) / q - 1;
      const uint32_t x = readlane_u32(srt1, at & 63), x2 = readlane_u32(srt, at2 & 63);
      if (lane == 0) {
        sh.wkey[0][q - 1][w] = at < 64 ? x : 0u;
        sh.wkey[1][q - 1][w] = at2 < 64 ? x2 : 0u;
      }
    }
    __syncthreads();
    uint32_t kb = bound_key<SBT / 64>(sh.wkey[0], lane);
    if (meet) {
      if (w == 0) {
        const uint32_t kb2 = bound_key<SBT / 64>(sh.wkey[1], lane);
        if (lane == 0) st(maxima + c, floor_entry(kb2, kb, ep));
        u64 e;
        const bool ok = poll_words(maxima, a.S, ep, a.key_spins, &e);
        const uint32_t lo = ~wave_max(lane < a.S ? ~floor_key1(e) : 0u), hi = wave_max(lane < a.S ? floor_key2(e) : 0u);
        if (lane == 0) sh.floor = ok ? (lo > hi ? lo : hi) : 0u;
      }
      __syncthreads();
      kb = sh.floor > kb ? sh.floor : kb;
    }
    float yb = kb ? tg_unkey(kb) : -__builtin_inff();
    if (counted) yb = counted_floor<Tin>(rv, mc, (unsigned)r.k, tl, sh);
    uint32_t ma = floor_marks(rv, yb);
    unsigned at = mark_places(ma, sh.ts);
    __syncthreads();
    unsigned n = sh.ts.ng;
    if (n > (unsigned)TOPPS_PAIR) {
      // more ids than the list holds (ties at the floor, no floor): the
      // chunk's exact top k
      ma = kth_marks(rv, mc, (unsigned)r.k, yb, sh);
      at = mark_places(ma, sh.ts);
      n = (unsigned)r.k;
    }
    each_marked(rv, ma, at, [&](unsigned o, u64 x) { st(slab + o, x); });
    wait_stores();
    __syncthreads();
    if (threadIdx.x == 0) {
      st(done + c, ((u64)ep << 32) | n);
      wait_stores();
      sh.arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (sh.arrived != (unsigned)(a.S - 1)) return;
    // the owner: every list has been published
    if (w == 0) {
      const bool act = lane < a.S;
      const uint32_t incl = wave_incl_scan(act ? (uint32_t)ld(done + lane) : 0u);
      if (act) sh.done[lane] = incl;
    }
    __syncthreads();
    n = sh.done[a.S - 1];
    // f(entry i) for this thread's share of the lists laid end to end
    auto each_entry = [&](auto f) {
      for (unsigned i = threadIdx.x; i < n; i += SBT) {
        int cc = 0;
        unsigned base = 0u;
        for (int q = 0; q < a.S - 1; q++)
          if (i >= sh.done[q]) {
            cc = q + 1;
            base = sh.done[q];
          }
        f(i, ld(slabs + (long long)cc * TOPPS_PAIR + (i - base)));
      }
    };
    if (n == 0u) {
      write_greedy<SBT>(a, r, 0ull);
    } else {
      if (n <= (unsigned)CAPL) {
        each_entry([&](unsigned i, u64 x) { tl.L[i] = x; });
      } else {
        // (ties again: the row's top k out of the lists)  The lists are long
        // and many passes follow: a list per group of threads, eight entries'
        // loads in flight (through each_entry 1 row of 128,256 equal fp32
        // logits, k = 1000, took 317 us, now 50).
        int per = SBT;  // threads per list
        while (per * a.S > SBT) per >>= 1;
        const int lc = (int)threadIdx.x / per;
        const unsigned ln = lc < a.S ? sh.done[lc] - (lc ? sh.done[lc - 1] : 0u) : 0u;
        const u64* list = slabs + (long long)lc * TOPPS_PAIR;
        auto en = [&](auto f) {
          constexpr int FLY = 8;
#pragma unroll 1
          for (unsigned i0 = threadIdx.x % (unsigned)per; i0 < ln; i0 += FLY * per) {
            u64 x[FLY];
#pragma unroll
            for (int j = 0; j < FLY; j++) x[j] = i0 + j * per < ln ? ld(list + i0 + j * per) : 0ull;
#pragma unroll
            for (int j = 0; j < FLY; j++)
              if (x[j]) f(x[j]);
          }
        };
        const Digits d = shared_digits<SBT>(en, sh.ts);
        const u64 T = block_select_kth<u64, 64, SBT>(en, (unsigned)r.k, sh.bs, d.shift, d.prefix, d.pmask);
        if (threadIdx.x == 0) sh.ts.ng = 0;
        __syncthreads();
        en([&](u64 x) {
          if (x >= T) tl.L[atomicAdd(&sh.ts.ng, 1u)] = x;
        });
        n = (unsigned)r.k;
      }
      __syncthreads();
      finish_topk(a, r, tl.L, n, tl, sh);
    }
    reset_line(a, line, ep);
    return;
  }

  // ---- 1. the row's maximum
  mc = wave_max(mc);
  if (lane == 0) sh.ts.red64[w] = mc;
  __syncthreads();
  if (r.mode == 0) {
    // a greedy row: the last chunk to arrive takes the largest of them all
    if (w == 0) {
      mc = wave_max(lane < SBT / 64 ? sh.ts.red64[lane] : 0ull);
      if (lane == 0) {
        st(maxima + c, max_entry(mc, ep));
        wait_stores();
        sh.arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    if (sh.arrived != (unsigned)(a.S - 1)) return;
    if (w == 0) {
      const u64 x = wave_max(lane < a.S ? ld(maxima + lane) : 0ull);
      if (lane == 0) sh.rowmax = max_comp(x);
    }
    __syncthreads();
    write_greedy<SBT>(a, r, sh.rowmax);
    reset_line(a, line, ep);
    return;
  }
  if (w == 0) {
    mc = wave_max(lane < SBT / 64 ? sh.ts.red64[lane] : 0ull);
    bool ok = true;
    if (a.S > 1) {
      if (lane == 0) st(maxima + c, max_entry(mc, ep));
      u64 e;
      ok = poll_words(maxima, a.S, ep, a.key_spins, &e);
      // (entries of the call order as their composites)
      mc = max_comp(wave_max(ok ? e : 0ull));
    }
    if (lane == 0) {
      sh.rowmax = mc;
      sh.flag = ok;
    }
  }
  __syncthreads();
  u64 Mc = sh.rowmax;
  if (!sh.flag) {
    // the partners are not running: the whole row's maximum from memory
    SV sv(a, r, hash, hbits, rowp);
    u64 best = 0ull;
    sv.each([&](int id, float y) {
      const u64 x = comp_key(tg_key(y), id);
      best = x > best ? x : best;
    });
    Mc = block_reduce_max<SBT>(best, sh.ts.red64);
  }
  tl.m = Mc ? comp_y(Mc) : 0.0f;
  const bool sampling = Mc != 0ull;

  // ---- 2. the chunk's histogram, its slab, and the arrival
  if (sampling) {
    histogram(rv, tl);
    if (a.S > 1) {
      __syncthreads();
      unsigned* sc = (unsigned*)(slab + NB);
      for (int i = threadIdx.x; i < NB; i += SBT) {
        st(slab + i, tl.MI[i]);
        st(sc + i, tl.CI[i]);
      }
      if (threadIdx.x == 0) st(sc + NB, tl.CI[NB]);
      wait_stores();
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // (its maximum too: a row with nothing allowed has stored only that, and
    // the owner clears it once all have arrived)
    wait_stores();
    sh.arrived = a.S > 1 ? __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
  }
  __syncthreads();
  const bool owner = sh.arrived == (unsigned)(a.S - 1);
  if (!owner && !sampling) return;

  if (!owner) {
    // ---- 3. the decision, and this chunk's ids of its buckets
    if (w == 0) {
      u64 d = 0ull;
      int spins = 0;
      for (; spins <= a.key_spins; spins++) {
        d = ld(decision);
        if (decided(d, ep)) break;
        __builtin_amdgcn_s_sleep(1);
      }
      if (lane == 0) {
        sh.flag = decided(d, ep);
        sh.word = d;
        sh.ts.ng = 0;
      }
    }
    __syncthreads();
    if (!sh.flag) {
      if (threadIdx.x == 0) st(done + c, ((u64)ep << 32) | DONE_LEFT);
      return;
    }
    if (!(sh.word & 1ull)) return;  // the owner settles the row by itself
    const Plan pl = unpack_plan(sh.word);
    u64* list = slab + TOPPS_SLAB;
    gather(rv, pl, tl.m, sh.ts, [&](int l, unsigned o, u64 x) {
      if (o < (unsigned)TOPPS_LIST) st(list + l * TOPPS_LIST + o, x);
    });
    wait_stores();
    __syncthreads();
    if (threadIdx.x == 0) {
      const unsigned na = sh.ts.ng & 0xFFFFu, nb = sh.ts.ng >> 16;
      const bool fit = na <= (unsigned)TOPPS_LIST && nb <= (unsigned)TOPPS_LIST;
      st(done + c, ((u64)ep << 32) | (fit ? (na << 10) | nb : DONE_LEFT));
    }
    return;
  }

  // ---- the owner: the row's histogram, the cut and the draw
  if (!sampling) {
    write_greedy<SBT>(a, r, Mc);
  } else {
    if (a.S > 1) {
      // thread t sums buckets t and t + 512, eight slabs' words in flight
      u64 ms[2] = {0ull, 0ull};
      unsigned cs[2] = {0u, 0u};
#pragma unroll 1
      for (int c0 = 0; c0 < a.S; c0 += 8) {
        u64 mq[8][2];
        unsigned cq[8][2];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const u64* s = slabs + (long long)min(c0 + j, a.S - 1) * TOPPS_PAIR;
#pragma unroll
          for (int h = 0; h < 2; h++) {
            mq[j][h] = ld(s + threadIdx.x + h * SBT);
            cq[j][h] = ld((const unsigned*)(s + NB) + threadIdx.x + h * SBT);
          }
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
          for (int h = 0; h < 2; h++) {
            ms[h] += c0 + j < a.S ? mq[j][h] : 0ull;
            cs[h] += c0 + j < a.S ? cq[j][h] : 0u;
          }
      }
      static_assert(NB == 2 * SBT, "two buckets per thread");
#pragma unroll
      for (int h = 0; h < 2; h++) {
        tl.MI[threadIdx.x + h * SBT] = ms[h];
        tl.CI[threadIdx.x + h * SBT] = cs[h];
      }
    }
    if (a.S > 1 && w == 0) {
      unsigned x = lane < a.S ? ld((const unsigned*)(slabs + (long long)lane * TOPPS_PAIR + NB) + NB) : 0u;
      x = wave_sum(x);
      if (lane == 0) tl.CI[NB] = x;
    }
    __syncthreads();
    bucket::prefix<SBT>(tl.CI, tl.MI, sh.ts.red32, sh.ts.red64);
    const unsigned nall = tl.CI[NB];
    const unsigned kk = has_k && (unsigned)r.k < nall ? (unsigned)r.k : nall;
    Plan pl;
    // a top-k set that reaches the mass-0 bucket carries the whole row's mass:
    // only its last element (a cut with top-p off) is still its own
    const bool whole = kk == nall || kk > tl.CI[NB - 1];
    if (whole) plan_row<SBT>(pl, r, tl, Mc, kk, sh.ts);
    else plan_topk<SBT>(pl, r, tl, Mc, kk, sh.ts);
    const bool lists = packs(pl);
    if (threadIdx.x == 0) st(decision, decision_tag(ep) | (lists ? pack_plan(pl) : 0ull));
    SV sv(a, r, hash, hbits, rowp);
    u64 pick;
    if (lists) {
      auto take = [&](int l, unsigned o, u64 x) { tl.L[l ? pl.ob + o : o] = x; };
      gather(rv, pl, tl.m, sh.ts, take);
      if (w == 0) {
        // every other workgroup of the row has arrived: it publishes its
        // lists or says that it left, within its own bounded poll
        const bool act = lane < a.S && lane != c;
        u64 e = 0ull;
        for (;;) {
          if (act && (uint32_t)(e >> 32) != ep) e = ld(done + lane);
          if (__ballot(act && (uint32_t)(e >> 32) != ep) == 0ull) break;
          __builtin_amdgcn_s_sleep(1);
        }
        if (lane < a.S) sh.done[lane] = act ? (uint32_t)e : 0u;
      }
      __syncthreads();
      // the published lists behind the owner's own, entry t of chunk cc's by
      // thread cc TPC + t (one round of requests for short lists)
      const unsigned own = sh.ts.ng;
      __syncthreads();
      unsigned pa = own & 0xFFFFu, pb = own >> 16;
      constexpr unsigned TPC = SBT / TOPPS_MAX_SPLIT;
      const int mc2 = (int)(threadIdx.x / TPC);
      unsigned mna = 0u, mnb = 0u, mpa = 0u, mpb = 0u;
      bool left = false;
      for (int cc = 0; cc < a.S; cc++) {
        const uint32_t e = sh.done[cc];
        if (e & DONE_LEFT) {
          left = true;
          continue;
        }
        const unsigned na = e >> 10, nb = e & 0x3FFu;
        if (cc == mc2) {
          mna = na;
          mnb = nb;
          mpa = pa;
          mpb = pl.ob + pb;
        }
        pa += na;
        pb += nb;
      }
      {
        const u64* list = slabs + (long long)mc2 * TOPPS_PAIR + TOPPS_SLAB;
        for (unsigned t = threadIdx.x % TPC; t < max(mna, mnb); t += TPC) {
          const u64 x = t < mna ? ld(list + t) : 0ull;
          const u64 y = t < mnb ? ld(list + TOPPS_LIST + t) : 0ull;
          if (t < mna) tl.L[mpa + t] = x;
          if (t < mnb) tl.L[mpb + t] = y;
        }
      }
      if (left) {  // (uniform)
        if (threadIdx.x == 0) sh.ts.ng = pa | pb << 16;
        __syncthreads();
        for (int cc = 0; cc < a.S; cc++) {
          if (!(sh.done[cc] & DONE_LEFT)) continue;
          Row rl = r;
          rl.v0 = cc * a.L;
          rl.v1 = min(a.V, rl.v0 + a.L);
          const SV lv(a, rl, hash, hbits, rowp);
          gather(lv, pl, tl.m, sh.ts, take);
        }
      }
      __syncthreads();
      pick = pick_gathered<SBT>(pl, r.top_p, tl, sh.ts, sh.bs);
    } else {
      pick = pick_resolved<SBT>(pl, r.top_p, sv, tl, sh.ts, sh.bs);
    }
    if (kk < nall && whole && pl.cut_last && a.dbg.cut_ids) {
      const u64 T = block_select_kth<u64, 64, SBT>(
          [&](auto f) { sv.each([&](int id, float y) { f(comp_key(tg_key(y), id)); }); }, kk, sh.bs);
      u64 x = 0ull;
      sv.each([&](int id, float y) {
        const u64 v = comp_key(tg_key(y), id);
        if (v >= T) x = ~v > x ? ~v : x;
      });
      pl.cutc = ~block_max<u64, SBT>(x, sh.ts.red64);
      pl.cut_last = false;
    }
    write_row<SBT>(a, b, pl, pick, sv, sh.ts);
  }
  reset_line(a, line, ep);
}

}  // namespace topp

hipError_t launch_topps(SampleArgs a, int dtype, int rows, hipStream_t st) {
  const size_t lds = topp_lds_bytes(a.V, a.TS);
  for (a.row0 = 0; a.row0 < a.B; a.row0 += rows) {
    a.rows = rows < a.B - a.row0 ? rows : a.B - a.row0;
    a.div8s = (unsigned)((1ull << 32) / (unsigned)(8 * a.S) + 1);  // exact below 2^32 / (8 S)
    a.divg = 65536u / (unsigned)std::max(a.rows % 8, 1) + 1u;       // exact below 2^16 / g
    const dim3 g((unsigned)(a.rows * a.S)), blk(TOPPS_NT);
    if (dtype == 1) hipLaunchKernelGGL((topp::topps_kernel<uint16_t>), g, blk, lds, st, a);
    else hipLaunchKernelGGL((topp::topps_kernel<float>), g, blk, lds, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

size_t topps_static_lds() { return sizeof(topp::SplitShared); }

hipError_t set_topps_lds_limit(size_t bytes) {
  const hipError_t e1 = hipFuncSetAttribute((const void*)topp::topps_kernel<float>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  const hipError_t e2 = hipFuncSetAttribute((const void*)topp::topps_kernel<uint16_t>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  return e1 != hipSuccess ? e1 : e2;
}

}  // namespace tgs
