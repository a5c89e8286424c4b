// dK / dV of the tiled keys, wave-specialised (included by attn_kernels.hip).
//
// One workgroup = KB keys x `heads` query heads of one K/V head, eight waves, two per SIMD that run different
// halves of the work, so that each SIMD has a wave for the matrix pipe while the other is in its vector phase:
//   producers (waves 0-3): wave (row half rh, key half kh) keeps the K / V fragments of KB / 2 keys; per query tile of
//     32 rows it forms, for ITS 16 rows, S = Q' K^T - lse and dP = dO V^T - delta, P = exp2(S), dS = P dP and hands
//     both over, rounded to bf16, through an LDS slot in the layout of the second products' B operand;
//   consumers (waves 4-7): wave (dV or dK, half) keeps 64 keys x min(D, 128) dims of ONE of the two gradients (the
//     half is a key half at head_dim <= 128, a half of the dims at 256) and adds dO^T P resp. Q'^T dS from the slot.
// v_mfma_f32_16x16x32_bf16 reads a 1 KB A fragment (8 cycles of LDS) for 16 cycles of work, so a fragment has to serve
// several products: a producer's fragment of Q' / dO serves 4 (head_dim 64, 256: 2) blocks of 16 keys, a consumer's of
// dO^T / Q'^T serves 4.  Over whole launches the counters read: head_dim 128, 4096 rows, matrix pipe busy 46 % at 1.95 GHz,
// LDS 31 %, waves waiting 23 % of their cycles; head_dim 256, 32760 rows, 50 % at 2.19 GHz, 43 %, 34 %.  What is left is the
// chain barrier -> soft-max -> scores of a producer and the consumers' wait for it.  At head_dim 64 a key block of 64 leaves room for two workgroups on a compute unit, which fill each other's gaps.
// Measured, kernel + sum of the partial results (us), against waves split by key with two 32 x 32 score tiles each:
// 512 rows, 32 heads of 64: 37 -> 18; 4096 rows, 32 heads of 128: 387 -> 300; 8192 rows, 64 heads of 128: 2370 -> 1915;
// 16384 rows, 16 heads of 256 (one wave per SIMD before): 5080 -> 3900.
// Both roles read the SAME row-major query tile: the consumers' A operands come through transposing LDS reads
// (ds_read_b64_tr_b16), so no transposed copy of the queries exists in memory.  Everything a step needs comes
// global -> LDS directly, kAhead tiles ahead, into a ring of kStages buffers: the tile, and the per-row scalars (-lse,
// -delta: the C operands of the score products; the mask interval ends).  In step b the producers turn the scores of
// tile b (computed one step earlier) into P and dS and compute the scores of tile b + 1, while the consumers work on
// tile b - 1.  One workgroup barrier per step; slots are double buffered.
#pragma once

namespace spx {

// How the dK / dV work of a call is cut into workgroups (dkv_plan, on the host).
struct DkvPlan {
  int heads;    // query heads of one K/V head a workgroup takes, one after the other (sums stay in registers)
  int n_hu;     // Hq / heads
  int paired;   // 1: key blocks i and n_kb - 1 - i go to one workgroup (about equal work under a causal mask)
  int windows;  // ranges of kListCap query tiles (rows beyond the first: unpaired only)
  int n_kb, n_k;  // key blocks; workgroups per head unit
  // a workgroup has all query heads of its K/V head and all their rows: it stores the gradients, and there is nothing to add up
  bool whole(int Hkv) const { return n_hu == Hkv && windows == 1; }
  int parts(int Hkv) const { return whole(Hkv) ? 0 : n_hu * windows; }  // fp32 partial results of dK and of dV
};

template <int D>
struct DkvCfg {
  static constexpr int KB = D == 128 ? 128 : 64;       // keys per workgroup
  static constexpr bool kByDim = KB == 64;             // the two consumers of a gradient share its dims, not its keys
  static constexpr int NKP = KB / 32;                  // blocks of 16 keys per producer
  static constexpr int NDC = (kByDim ? D / 2 : D) / 16;  // blocks of 16 dims per consumer (of 4 key blocks)
  static constexpr int kStages = D <= 128 ? 6 : 4;
  static constexpr int kAhead = kStages - 2;           // tile b + kAhead is issued in step b
  static constexpr int RB = D * 2, CK = RB / 16;       // bytes / 16-byte chunks per row of Q' and dO
  static constexpr int kTile = 2 * 32 * RB;            // Q', dO: 32 rows each
  static constexpr int kSlot = 32 * KB * 2;            // P or dS of a tile
  static constexpr int kOffSlot = kStages * kTile;     // [parity][P, dS]
  static constexpr int kOffSmall = kOffSlot + 4 * kSlot;
  static constexpr int kSmall = 6 * 32 * 4;            // -lse, -delta, a1, b1, a2, b2 of 32 rows
  static constexpr int kSets = 8;                      // sets of per-row scalars (tile k: set k % 8)
  static constexpr int kOffList = kOffSmall + kSets * kSmall + 256;  // (+ a spare area)
  static constexpr int kListCap = 2048;                // 64-row query tiles a workgroup looks at
  static constexpr int kOffTot = kOffList + kListCap * 4;
  static constexpr int kBytes = kOffTot + 64;
  // position of 16-byte chunk c of row r inside its LDS row: c ^ swz(r).  16-byte reads of 16 rows at one chunk (the
  // producers) and transposing 8-byte reads of 8 rows at one pair of chunks (the consumers) both fill 256 bytes.
  static __device__ __forceinline__ int swz(int r) {
    if (CK == 8) { const int t = (r >> 1) & 7; return ((t & 3) << 1) | (t >> 2); }
    return ((r & 7) << 1) | ((r >> 3) & 1);
  }
};

typedef __attribute__((ext_vector_type(4))) int i32x4;

__device__ __forceinline__ f32x4 mfma16b(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <typename T>
__device__ __forceinline__ T lds_get(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>((uintptr_t)addr);
}
template <typename T>
__device__ __forceinline__ void lds_put(uint32_t addr, T v) {
  *reinterpret_cast<__attribute__((address_space(3))) T*>((uintptr_t)addr) = v;
}

// What both roles know about the workgroup's work; every value is wave-uniform.
struct DkvJob {
  uint32_t lds;    // LDS address of the workgroup's memory
  uint32_t list;   // ... of its first list entry
  int n_vis;       // visible 64-row query tiles
  int n0;          // first key
  int h0, nh, kvh; // query heads, K/V head
};

// The producers' part: see above.  K/V fragments 2 x NKP x D / 32 x 4 registers.
template <int D>
__device__ __forceinline__ void dkv_produce(const AttnParams& p, const DkvJob& job, int pw, int lane) {
  using C = DkvCfg<D>;
  constexpr int NKP = C::NKP, NKK = D / 32;
  const int rh = pw & 1, kh = pw >> 1;
  const int G = lane >> 4, li = lane & 15;
  const int key0 = job.n0 + kh * (C::KB / 2) + li;
  bf16x8 kf[NKP][NKK], vf[NKP][NKK];
#pragma unroll
  for (int kb = 0; kb < NKP; ++kb) {
    const int c = min(key0 + kb * 16, p.NKV - 1);
    const uint16_t* krow = p.K + (int64_t)job.kvh * p.k_hs + (int64_t)c * D + G * 8;
    const uint16_t* vrow = p.V + (int64_t)job.kvh * p.v_hs + (int64_t)c * D + G * 8;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      kf[kb][kk] = as_bf16x8(*reinterpret_cast<const u32x4*>(krow + kk * 32));
      vf[kb][kk] = as_bf16x8(*reinterpret_cast<const u32x4*>(vrow + kk * 32));
    }
  }
  const int n_steps = job.n_vis * 2 * job.nh;
  const uint32_t rd = job.lds + (rh * 16 + li) * C::RB + ((G ^ C::swz(li)) * 16);
  const uint32_t sm = job.lds + C::kOffSmall + (rh * 16 + 4 * G) * 4;
  const uint32_t slot = job.lds + C::kOffSlot + (kh * NKP * 2 + rh) * 512 + lane * 8;

  f32x4 st[NKP], dp[NKP];
  bf16x8 qa[NKK], da[NKK];
  f32x4 ci, di;
  // operands of the score products of the tile in ring buffer `buf`
  auto fetch = [&](int buf, int set) __attribute__((always_inline)) {
    const uint32_t t = rd + buf * C::kTile;
    ci = lds_get<f32x4>(sm + set * C::kSmall);
    di = lds_get<f32x4>(sm + set * C::kSmall + 128);
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      qa[kk] = as_bf16x8(lds_get<u32x4>(t ^ (kk * 64)));
      da[kk] = as_bf16x8(lds_get<u32x4>((t ^ (kk * 64)) + 32 * C::RB));
    }
  };
  // scores and dP of key blocks kb, kb + 1: four independent chains
  auto score2 = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      st[kb] = mfma16b(qa[kk], kf[kb][kk], kk == 0 ? ci : st[kb]);
      dp[kb] = mfma16b(da[kk], vf[kb][kk], kk == 0 ? di : dp[kb]);
      st[kb + 1] = mfma16b(qa[kk], kf[kb + 1][kk], kk == 0 ? ci : st[kb + 1]);
      dp[kb + 1] = mfma16b(da[kk], vf[kb + 1][kk], kk == 0 ? di : dp[kb + 1]);
    }
  };
  // P and dS of key block kb.  kMask: only the rows whose intervals [lo, lo + len) hold the key keep their value
  // (bitwise on purpose: short-circuit tests would become branches on the lane mask).
  i32x4 lo1, len1, lo2, len2;
  auto soft = [&](int kb, auto mask, uint32_t out) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = fast_exp2(st[kb][r]);
      if constexpr (decltype(mask)::value) {
        const int c = key0 + kb * 16;
        const bool ok = ((uint32_t)(c - lo1[r]) < (uint32_t)len1[r]) | ((uint32_t)(c - lo2[r]) < (uint32_t)len2[r]);
        v = ok ? v : 0.f;
      }
      st[kb][r] = v;
    }
    dp[kb] *= st[kb];
    const u32x2 pw_ = {pack_bf16x2(st[kb][0], st[kb][1]), pack_bf16x2(st[kb][2], st[kb][3])};
    const u32x2 sw_ = {pack_bf16x2(dp[kb][0], dp[kb][1]), pack_bf16x2(dp[kb][2], dp[kb][3])};
    lds_put<u32x2>(out + kb * 1024, pw_);
    lds_put<u32x2>(out + kb * 1024 + C::kSlot, sw_);
  };

  // list entry of step b: position b / 2 (modulo the list, once per head); bit 31 = no mask needed
  int pos = 0;
  uint32_t e = n_steps ? lds_get<uint32_t>(job.list) : 0u;
  __syncthreads();  // the first kAhead tiles are in LDS
  fetch(0, 0);
#pragma unroll
  for (int kb = 0; kb < NKP; kb += 2) score2(kb);
  int nb = 1;  // ring buffer of tile b + 1
  auto step = [&](auto mask, int b) __attribute__((always_inline)) {
    if constexpr (decltype(mask)::value) {
      const uint32_t m = sm + (b & (C::kSets - 1)) * C::kSmall;
      lo1 = lds_get<i32x4>(m + 256);
      len1 = lds_get<i32x4>(m + 384) - lo1;
      lo2 = lds_get<i32x4>(m + 512);
      len2 = lds_get<i32x4>(m + 640) - lo2;
#pragma unroll
      for (int r = 0; r < 4; ++r) { len1[r] = max(len1[r], 0); len2[r] = max(len2[r], 0); }
    }
    // (behind the last tile the scores of whatever the ring holds are formed and left unused)
    fetch(nb, (b + 1) & (C::kSets - 1));
    const uint32_t out = slot + (b & 1) * 2 * C::kSlot;
#pragma unroll
    for (int kb = 0; kb < NKP; kb += 2) {
      soft(kb, mask, out);
      soft(kb + 1, mask, out);
      score2(kb);
    }
  };
  for (int b = 0; b < n_steps; ++b) {
    __syncthreads();
    const bool full = (__builtin_amdgcn_readfirstlane(e) >> 31) != 0;
    pos += b & 1;
    pos = pos == job.n_vis ? 0 : pos;
    e = lds_get<uint32_t>(job.list + pos * 4);
    if (full) step(std::false_type{}, b);
    else step(std::true_type{}, b);
    nb = nb + 1 == C::kStages ? 0 : nb + 1;
  }
  __syncthreads();
}

// The consumers' part, and all loads of the tiles (they have issue slots to spare, the producers do not).
// WHOLE (DkvPlan::whole): out_k, out_v are the gradients of the K/V head, bf16 (accumulate: added to what is there, in fp32, one rounding).
template <int D, bool WHOLE>
__device__ __forceinline__ void dkv_consume(const AttnParams& p, const DkvJob& job, const uint16_t* __restrict__ dO,
                                            int NQp, const float* __restrict__ neg,
                                            const int32_t* __restrict__ mrows, float* __restrict__ out_k,
                                            float* __restrict__ out_v, int accumulate, int cw, int lane) {
  using C = DkvCfg<D>;
  constexpr int NDC = C::NDC, NLQ = 32 * C::RB / 1024, LPW = 2 * NLQ / 4, AH = C::kAhead, NS = C::kStages;
  constexpr int kLoads = LPW + 1;
  const bool is_k = (cw & 1) != 0;
  const int half = cw >> 1;
  const int G = lane >> 4, li = lane & 15;
  const int n_steps = job.n_vis * 2 * job.nh;

  // this wave's loads of a tile: li_ = cw + 4 j of the 2 * NLQ that make it (Q' first, then dO); rows past the last
  // query read as zeros (and contribute nothing).  Per-row scalars: -lse | -delta, a1 | b1, a2 | b2 (32 values each),
  // one 256-byte load by each of waves 0 - 2 (the fourth repeats the first into a spare area so that all count alike).
  int ld_off[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int l_ = cw + 4 * j, l = l_ >= NLQ ? l_ - NLQ : l_;
    const int r = l * (1024 / C::RB) + lane / C::CK;
    ld_off[j] = r * (l_ >= NLQ ? p.Hq * C::RB : C::RB) + ((lane % C::CK) ^ C::swz(r & 15)) * 16;
  }
  const bool sm_mask = cw == 1 || cw == 2;
  const int sm_off = (lane & 31) * 4 + (lane >> 5) * (sm_mask ? NQp * 4 : p.Hq * NQp * 4) + (cw == 2 ? 2 * NQp * 4 : 0);
  const uint32_t q_bytes = (uint32_t)((int64_t)p.NQ * C::RB);
  const uint32_t d_bytes = (uint32_t)((((int64_t)p.NQ - 1) * p.Hq * D + D) * 2);
  const uint32_t n_bytes = (uint32_t)((((int64_t)p.Hq + 1) * NQp) * 4);
  const u32x4 mres = make_rsrc(mrows, (uint32_t)(4 * (int64_t)NQp * 4));
  u32x4 qres, dres, sres;
  auto at_head = [&](int h) __attribute__((always_inline)) {
    qres = make_rsrc(p.Q + (int64_t)h * p.q_hs, q_bytes);
    dres = make_rsrc(dO + (int64_t)h * D, d_bytes);
    sres = sm_mask ? mres : make_rsrc(neg + (int64_t)h * NQp, n_bytes);
  };
  // load j of a tile (j < LPW), or its per-row scalars (j = LPW)
  auto issue = [&](int j, int mq, int buf, int set) __attribute__((always_inline)) {
    if (j < LPW) {
      const bool is_do = 4 * j >= NLQ;  // (NLQ is a multiple of four)
      load_to_lds16<0>(is_do ? dres : qres, job.lds + buf * C::kTile + cw * 1024 + j * 4096,
                       (int)((uint32_t)ld_off[j < LPW ? j : 0] + (uint32_t)mq * (uint32_t)(is_do ? p.Hq * C::RB : C::RB)), 0);
    } else {
      const uint32_t s = job.lds + C::kOffSmall + (cw == 3 ? C::kSets * C::kSmall : set * C::kSmall + cw * 256);
      load_to_lds4(sres, s, sm_off + mq * 4, 0);
    }
  };

  f32x4 acc[NDC][4];
#pragma unroll
  for (int db = 0; db < NDC; ++db)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc[db][kb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // lane s of 16-lane group G points at row 4 G + (s >> 2) (second read: + 16), bytes 8 (s & 3) of dim block db.  k index
  // of the products: elements 0-3 of the lanes of group G are query rows 4 G .. 4 G + 3, elements 4-7 rows 16 + 4 G ..
  const int trow = 4 * G + (li >> 2);
  const int dim0 = C::kByDim ? half * (D / 2) : 0;
  const uint32_t rt = job.lds + (is_k ? 0 : 32 * C::RB) + trow * C::RB +
                      ((((li & 3) >> 1) ^ C::swz(trow) ^ (dim0 / 8)) * 16) + (li & 1) * 8;
  const uint32_t slot = job.lds + C::kOffSlot + (is_k ? C::kSlot : 0) + (C::kByDim ? 0 : half * 4096) + lane * 8;

  // the first fragments of a tile are read ahead, in the step before: they do not depend on the producers
  constexpr int RG = NDC < 4 ? NDC : 4;
  static_assert(NDC % RG == 0 && NDC >= RG, "the ring of fragments starts over with every tile");
  i16x4 lo[RG], hi[RG];
  auto fread = [&](int db, uint32_t t) __attribute__((always_inline)) {
    lo[db % RG] = lds_tr16(t ^ (db % NDC * 32));
    hi[db % RG] = lds_tr16((t ^ (db % NDC * 32)) + 16 * C::RB);
  };
  bf16x8 pb[4];
  auto slot_read = [&](int par) __attribute__((always_inline)) {
    const uint32_t s = slot + par * 2 * C::kSlot;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      pb[kb] = join_bf16x4(lds_get<u32x2>(s + kb * 1024), lds_get<u32x2>(s + kb * 1024 + 512));
  };
  // The loads of a later tile go out one by one between the matrix instructions: in a row they hold the
  // wave for as long as all of them take to issue.
  auto consume = [&](uint32_t t, uint32_t next, int mq, int buf, int set) __attribute__((always_inline)) {
    SPX_DKV_PRIO_MFMA();
#pragma unroll
    for (int db = 0; db < NDC; ++db) {
      const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo[db % RG], hi[db % RG], 0, 1, 2, 3, 4, 5, 6, 7));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) acc[db][kb] = mfma16b(a, pb[kb], acc[db][kb]);
      __builtin_amdgcn_sched_barrier(0);
      fread(db + RG, db + RG < NDC ? t : next);
#pragma unroll
      for (int j = db * kLoads / NDC; j < (db + 1) * kLoads / NDC; ++j) issue(j, mq, buf, set);
    }
    SPX_DKV_PRIO_VALU();
  };

  // ---- the sequence of loads: step k is half k & 1 of list entry (k / 2) % n_vis, head h0 + (k / 2) / n_vis.  Behind the
  // last one its tile is loaded again (nobody reads it): the number of loads in flight is then the same in every step.
  int i_pos = 0, i_head = job.h0, i_left = n_steps - 1;
  at_head(i_head);
  uint32_t e = n_steps ? lds_get<uint32_t>(job.list) : 0u;
  auto row_of = [&](int k) __attribute__((always_inline)) {
    return (int)(__builtin_amdgcn_readfirstlane(e) & 0x7fffffffu) * 64 + (k & 1) * 32;
  };
  auto advance = [&](int k) __attribute__((always_inline)) {
    i_pos += (k & 1) & (i_left > 0);
    i_left -= 1;
    if (i_pos == job.n_vis) {
      i_pos = 0;
      at_head(++i_head);
    }
    e = lds_get<uint32_t>(job.list + i_pos * 4);
  };
  auto issue_all = [&](int k, int buf) __attribute__((always_inline)) {
    const int mq = row_of(k);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) issue(j, mq, buf, k & (C::kSets - 1));
    advance(k);
  };
  if (n_steps > 0) {
    for (int i = 0; i < AH; ++i) issue_all(i, i);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int db = 0; db < RG; ++db) fread(db, rt);
  int bb = 0;  // ring buffer of tile b
  if (n_steps > 0) {
    __syncthreads();
    issue_all(AH, AH);
    bb = 1;
  }
  for (int b = 1; b <= n_steps; ++b) {
    // tile b + 1 has landed when at most the loads of tiles b + 2 .. b + kAhead - 1 are in flight
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AH - 2) * kLoads) : "memory");
    __syncthreads();
    slot_read((b - 1) & 1);
    // tile b + kAhead into the buffer tile b - 2 left behind
    consume(rt + (bb == 0 ? NS - 1 : bb - 1) * C::kTile, rt + bb * C::kTile, row_of(b + AH),
            bb + AH >= NS ? bb + AH - NS : bb + AH, (b + AH) & (C::kSets - 1));
    advance(b + AH);
    bb = bb + 1 == NS ? 0 : bb + 1;
  }
  if (n_steps == 0) __syncthreads();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in memory the next job uses

  if constexpr (WHOLE) {
    uint16_t* const out = reinterpret_cast<uint16_t*>(is_k ? out_k : out_v);
    const float scale = is_k ? kLn2 : 1.f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int c = job.n0 + (C::kByDim ? 0 : half * 64) + kb * 16 + li;
      if (c >= p.NKV) continue;
#pragma unroll
      for (int db = 0; db < NDC; ++db) {
        u32x2* const at = reinterpret_cast<u32x2*>(out + (int64_t)c * D + dim0 + 4 * G + db * 16);
        f32x4 v = acc[db][kb] * scale;
        if (accumulate) {
          const u32x2 old = *at;
          v.x += bf16_lo(old.x); v.y += bf16_hi(old.x); v.z += bf16_lo(old.y); v.w += bf16_hi(old.y);
        }
        *at = u32x2{pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)};
      }
    }
    return;
  }
  float* const out = is_k ? out_k : out_v;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int c = job.n0 + (C::kByDim ? 0 : half * 64) + kb * 16 + li;
    if (c < p.NKV) {
      float* row = out + (int64_t)c * D + dim0 + 4 * G;
#pragma unroll
      for (int db = 0; db < NDC; ++db) *reinterpret_cast<f32x4*>(row + db * 16) = acc[db][kb];
    }
  }
}

// WHOLE: dKp, dVp are dK and dV, dk_hs and dv_hs elements from K/V head to K/V head
template <int D, bool WHOLE>
__global__ __launch_bounds__(512, D == 64 ? 4 : 2) void attn_bwd_dkv_kernel(
    AttnParams p, const uint16_t* __restrict__ dO, int NQp, const float* __restrict__ neg,
    const int32_t* __restrict__ mrows, const int32_t* __restrict__ tile_bounds, DkvPlan pl,
    float* __restrict__ dKp, float* __restrict__ dVp, int64_t dk_hs, int64_t dv_hs, int accumulate) {
  using C = DkvCfg<D>;
  extern __shared__ __attribute__((aligned(16))) uint8_t dkv_smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)dkv_smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroups go to the eight XCDs round robin.  The query tiles a workgroup streams belong to its query heads, so
  // the workgroups that share an XCD (and its L2) at a time get the same heads and consecutive key blocks; heavy key
  // blocks first (under a causal mask the early ones are seen by most rows).
  int hu, ki;
  if (pl.n_hu % 8 == 0) {
    const int xcd = blockIdx.x & 7, s = blockIdx.x >> 3;
    hu = xcd + 8 * (s / pl.n_k);
    ki = s % pl.n_k;
  } else {
    hu = blockIdx.x % pl.n_hu;
    ki = blockIdx.x / pl.n_hu;
  }
  const int win = ki % pl.windows, kb0 = ki / pl.windows;
  const int n_qt = (p.NQ + 63) / 64;
  const int q_lo = win * C::kListCap, q_hi = min(q_lo + C::kListCap, n_qt);
  DkvJob job;
  job.lds = lds0;
  job.h0 = hu * pl.heads;
  job.nh = pl.heads;
  job.kvh = job.h0 / (p.Hq / p.Hkv);
  const int64_t part = ((int64_t)win * pl.n_hu + hu) * p.NKV * D;

  for (int turn = 0; turn < 1 + pl.paired; ++turn) {
    const int kb = turn == 0 ? kb0 : pl.n_kb - 1 - kb0;
    if (turn == 1) {
      if (kb == kb0) break;  // the middle block of an odd count has no partner
      __syncthreads();       // everybody is done with the list, the ring, the slots and the sets
    }
    const int n0 = kb * C::KB, key_last = min(n0 + C::KB - 1, p.NKV - 1);
    // ---- the visible query tiles, in order, into LDS; bit 31: every key of the block is visible to all rows
    int n_all = 0;
    for (int q0 = q_lo; q0 < q_hi; q0 += 512) {
      const int qt = q0 + tid;
      bool vis = false, full = false;
      if (qt < q_hi) {
        const i32x4 t1 = *reinterpret_cast<const i32x4*>(tile_bounds + qt * 8);
        const i32x4 t2 = *reinterpret_cast<const i32x4*>(tile_bounds + qt * 8 + 4);
        vis = (t1[0] <= key_last && t1[3] > n0) || (t2[0] <= key_last && t2[3] > n0);
        full = (t1[1] <= n0 && t1[2] >= n0 + C::KB) || (t2[1] <= n0 && t2[2] >= n0 + C::KB);
      }
      const unsigned long long m = __ballot(vis);
      const int before = __popcll(m & ((1ull << lane) - 1));
      if (lane == 0) lds_put<int>(lds0 + C::kOffTot + wave * 4, __popcll(m));
      __syncthreads();
      int off = n_all;
      for (int w = 0; w < 8; ++w) {
        const int t = __builtin_amdgcn_readfirstlane(lds_get<int>(lds0 + C::kOffTot + w * 4));
        if (w < wave) off += t;
        n_all += t;
      }
      if (vis) lds_put<uint32_t>(lds0 + C::kOffList + (off + before) * 4, (uint32_t)qt | (full ? 0x80000000u : 0u));
      __syncthreads();
    }
    job.list = lds0 + C::kOffList;
    job.n_vis = n_all;
    job.n0 = n0;
    if (wave < 4) dkv_produce<D>(p, job, wave, lane);
    else if constexpr (WHOLE)
      dkv_consume<D, true>(p, job, dO, NQp, neg, mrows, reinterpret_cast<float*>(reinterpret_cast<uint16_t*>(dKp) + job.kvh * dk_hs),
                           reinterpret_cast<float*>(reinterpret_cast<uint16_t*>(dVp) + job.kvh * dv_hs), accumulate, wave - 4, lane);
    else dkv_consume<D, false>(p, job, dO, NQp, neg, mrows, dKp + part, dVp + part, 0, wave - 4, lane);
  }
}

}  // namespace spx
