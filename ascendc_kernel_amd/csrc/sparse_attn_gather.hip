// Task1, true-gather variant (any n_kv): each token attends to the kv rows its
// topk slots select, gathered from the batch's kv block (reference semantics
// of sparse_attn_ref, reference/task1_v0_ref.py:5-24; duplicates and masked
// slots handled exactly like the gather there).
//
// Two kernels, chosen by gather_split: sa_gather_kernel (many tokens of more than 32
// heads) and sa_gather_split_kernel (few tokens, or at most 32 heads). The former:
// one workgroup per token, one wave per 32 heads (ceil(h/32) waves). The slots are
// processed in blocks of 32. The selected kv rows (256 B each) of a block are
// copied straight from global memory into LDS by global_load_lds_dwordx4 (no
// register staging), into a ring of kRing block buffers: one or two blocks are in flight while
// the scores of the next and the products of the current one are computed. Every wave then runs
//   S^T[32 keys x 32 heads]  = K[32 x 128] . Q^T[128 x 32]   (8 x mfma 32x32x16)
//   online softmax with the sink as the initial maximum (log2 domain)
//   O^T[128 x 32 heads]     += V^T[128 x 32] . (P_hi + P_lo)^T (16 x mfma 32x32x16)
// K fragments are 16-byte LDS reads of the swizzled rows; V^T fragments come
// from the same rows through ds_read_b64_tr_b16, which transposes 4x16-bit
// elements across each 16-lane group. The running maximum is only raised when
// a block exceeds it by more than 2^8 (then O and the sum are rescaled), which
// keeps exp2 arguments <= 8 and makes the rescale rare. P is split into a bf16
// high part and a bf16 residual so that the PV product keeps ~16 bits of P.
#include "dsa_common.h"

#include <float.h>

using namespace dsa;

namespace {

constexpr int kD = 128;
constexpr int kKB = 32;          // slots per block
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kRaise = 8.0f;   // log2 headroom before the running max is raised
// bf16 pairs (-1, 0) and (0, -1) as bit patterns: dot2(h, neg_lo, p0) = p0 - h.lo,
// dot2(h, neg_hi, p1) = p1 - h.hi.
constexpr uint32_t kNegLoBits = 0x0000bf80u;
constexpr uint32_t kNegHiBits = 0xbf800000u;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

struct GatherParams {
  const uint16_t* q;     // [B, M, H, 128]
  const uint16_t* kv;    // [B, NKV, 128]
  const void* idx;       // [B, M, TOPK] int32 or int64 (the kernel's IdxT)
  const float* sink;     // [H]
  uint16_t* out;         // [B, M, H, 128]
  int64_t M;
  int32_t B, H, NKV, TOPK;
  int32_t xpb;           // XCDs per batch for the block -> token map (0: identity)
  float scale_log2;      // softmax_scale * log2(e)
};

// Output channel of row i of d-tile dt (O^T rows): lane half hf = (i >> 2) & 1
// gets the contiguous channels 64*hf .. 64*hf + 63 across the four d-tiles.
__device__ __forceinline__ int out_ch(int dt, int i) {
  const int q = i >> 3, hf = (i >> 2) & 1, c = i & 3;
  return 64 * hf + 16 * dt + 4 * q + c;
}

// LDS row r (256 B = 16 chunks of 16 B): chunk c lives at r*16 + (c ^ (r & 15)).
__device__ __forceinline__ int swz(int r, int c) { return r * 16 + (c ^ (r & 15)); }

// Bound by the matrix cores and the VALU (per block and wave 24 products, ~770 cycles, and
// ~700 cycles of softmax), which overlap only across the waves of a SIMD. Two forms, chosen by
// gather_ring:
//  kRing 3: three waves per SIMD, so at most 168 VGPRs (fragment addresses come from one
//    register each by xor, mask bits and copy offsets are formed at their use, V fragments are
//    read one ahead in a pinned order) and a ring of three. 4 x 4096 tokens x 64 heads, 512
//    slots 397-412 -> 383-388 us (1.0 PFLOP/s of issued products), 3 x 421 tokens x 48 heads,
//    333 slots 31.0 -> 26.6, 4096 tokens x 96 heads, 256 slots 103 -> 83-85;
//  kRing 4: two waves per SIMD (196 VGPRs) with the offsets held, the order of the V reads
//    left to the compiler and one more block in flight, for grids that leave two waves or
//    fewer on a SIMD: 300 tokens x 64 heads, 1024 slots 35.2 -> 33.3 us.
// The three-wave form's registers at two waves per SIMD: no change. No s_setprio, or the raised
// priority on the products instead: 1-3 % slower.
template <int NW, typename IdxT, int kRing>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(kRing == 3 ? 3 : 2, kRing == 3 ? 3 : 2)))
void sa_gather_kernel(GatherParams p) {
  static_assert(kRing == 3 || kRing == 4, "one or two blocks in flight beside the two in use");
  const IdxT* const idx = static_cast<const IdxT*>(p.idx);
  // kRing blocks of 32 gathered rows (8 KB each); at the end one 8 KB area per wave. 1 KB
  // alignment: fragment addresses inside a block are formed by xor.
  __shared__ __align__(1024) u32x4 ring[kRing > NW ? kRing : NW][kKB * 16];
  __shared__ int32_t nblk_w[NW];  // per wave: blocks up to its last valid slot
  extern __shared__ int32_t slot[];         // the token's slot indices (masked -> -1)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wi = tid >> 6;
  // Blocks are dispatched to the 8 XCDs round-robin; map them so that XCD x
  // only serves batch x % B and its L2 keeps that batch's kv block.
  int64_t tok;
  if (p.xpb > 0) {
    const int xcd = blockIdx.x & 7;
    const int64_t slotno = blockIdx.x >> 3;
    tok = (int64_t)(xcd % p.B) * p.M + slotno * p.xpb + xcd / p.B;
  } else {
    tok = blockIdx.x;
  }
  const int b = (int)(tok / p.M);
  const int hbase = 32 * wi;             // this wave's heads
  const int col = lane & 31;             // head hbase + col (MFMA column)
  const int hf = lane >> 5;              // lane half: contraction slice 8*hf..8*hf+7
  const bool hvalid = hbase + col < p.H;  // the last wave may cover fewer than 32 heads
  const uint16_t* kvb = p.kv + (int64_t)b * p.NKV * kD;

  // The token's global reads (Q^T, the sink, the slot indices) are all issued
  // before any of them is waited for: one memory latency instead of one per
  // round of the slot loop.
  // Q^T fragments (B operand of the first product): head hbase+col, channels
  // 16ks + 8hf .. +7.
  // Lanes of heads >= H (the last wave when H % 32 != 0) load head 0's row: their
  // MFMA columns and softmax stay separate from the valid heads' and are never
  // stored; loading unconditionally keeps the loads out of branches (whose joins
  // would make the compiler wait for them at once).
  bf16x8 qf[8];
  {
    const uint16_t* qrow = p.q + (tok * p.H + (hvalid ? hbase + col : 0)) * kD + 8 * hf;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      qf[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qrow + 16 * ks));
  }
  const float sink_raw = p.sink[hvalid ? hbase + col : 0];  // unconditional: no wait in a branch
  // Slot indices -> LDS, 8 per thread in flight at a time; out-of-range indices
  // count as masked. Blocks after the last one holding a valid slot are neither
  // loaded nor computed.
  const int nblk = (p.TOPK + kKB - 1) / kKB;
  int last = 0;
  auto slot_chunk = [&](const int s0) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int s = s0 + 64 * NW * u + tid;
      v[u] = slot_index(idx, tok * p.TOPK + min(s, p.TOPK - 1));  // unconditional (see q)
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int s = s0 + 64 * NW * u + tid;
      if (s < nblk * kKB) {
        const int w = (s < p.TOPK && v[u] < p.NKV) ? v[u] : -1;
        slot[s] = w;
        if (w >= 0) last = s / kKB + 1;
      }
    }
  };
  // the first chunk outside the loop, so that nothing waits for Q^T before its loads issue
  slot_chunk(0);
  for (int s0 = 8 * 64 * NW; s0 < nblk * kKB; s0 += 8 * 64 * NW) slot_chunk(s0);
  // Blocks to compute: the maximum of `last` over the wave, then over the waves.
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) last = max(last, __shfl_xor(last, m, 64));
  if (lane == 0) nblk_w[wi] = last;
  __syncthreads();
  int nb = nblk_w[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) nb = max(nb, nblk_w[w]);

  // A block is 8 units of 4 rows (1 KB); one global_load_lds_dwordx4 moves a
  // unit: lane l writes LDS chunk 64u + l, i.e. row 4u + l/16, swizzled chunk
  // position l%16, which holds logical chunk (l%16) ^ (row & 15). Wave wi moves
  // units wi, wi + NW, ...; with NW = 3 the last wave reloads unit 0 (same bytes).
  constexpr int kUnits = (8 + NW - 1) / NW;
  const int wis = __builtin_amdgcn_readfirstlane(wi);
  const i32x4 rsrc = make_rsrc(kvb, (uint32_t)p.NKV * (uint32_t)(kD * 2));
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4*)&ring[0][0];
  // Per lane and unit u: tile row 4u + lane/16 and byte offset 16 ((lane%16) ^ (row%16)) in
  // the row, the unit entering as a scalar. They are recomputed from the lane id at each
  // use: held across the block loop they would spill.
  const uint32_t slot_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int32_t*)slot;
  auto lane_id = [&] {
    if constexpr (kRing == 4) {
      return lane;
    } else {
      int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
      asm volatile("" : "+v"(ln));
      return ln;
    }
  };
  auto unit = [&](int i) {
    const int u = wis + NW * i;
    return u >= 8 ? u - 8 : u;
  };
  // Slot values (kv rows) of this lane's units of block blk.
  auto rows_of = [&](int blk, int (&rv)[kUnits]) {
    const uint32_t srow = slot_lds + 4u * (uint32_t)(lane_id() >> 4);
#pragma unroll
    for (int i = 0; i < kUnits; ++i)
      rv[i] = *(__attribute__((address_space(3))) const int32_t*)(uintptr_t)(srow + (uint32_t)(blk * kKB + 4 * unit(i)) * 4u);
  };
  // Copy block blk (rows rv) into ring buffer rs. A masked row (-1) gives an
  // offset beyond the resource, which reads zeros.
  auto issue = [&](int rs, const int (&rv)[kUnits]) {
    const int ln = lane_id();
    const uint32_t ubase = 16u * (uint32_t)((ln & 15) ^ (ln >> 4));
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
      const int u = unit(i);
      lds_dma16(rsrc, ((uint32_t)rv[i] * (uint32_t)(kD * 2)) + (ubase ^ (64u * (uint32_t)(u & 3))),
                ring_lds + 1024u * (uint32_t)u + 8192u * (uint32_t)rs);
    }
  };
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x16{};
  const float sink_l2 = hvalid ? sink_raw * kLog2e : 0.f;
  const float c2 = p.scale_log2;  // > 0 (checked by the host)
  // Running max (log2 units) incl. the sink, floored at -FLT_MAX so that a -inf
  // sink with a fully masked first block gives exp2(-inf) = 0, not NaN.
  float m_run = fmaxf(sink_l2, -FLT_MAX);
  float l_run = 0.f;       // this lane's partial sum of exp2(s - m_run)

  // S^T = K . Q^T for the block in LDS buffer j: A = K rows (key = lane%32,
  // channels 16ks + 8hf ..). Lane holds keys 8(r/4) + 4hf + (r%4) of head col.
  // Chunk 2ks + hf of the row sits at (2ks + hf) ^ (row%16) = 2ks ^ (hf ^ row%16), so the
  // eight addresses are kbase with a constant xored in.
  typedef __attribute__((address_space(3))) const u32x4* lds_cu32x4_ptr;
  const uint32_t kbase = ring_lds + 16u * (uint32_t)swz(lane & 31, hf);
  auto qk = [&](const int j) {
    f32x16 acc = {};
    uint32_t kb_ = kbase;
    if constexpr (kRing == 3) asm volatile("" : "+v"(kb_));
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const bf16x8 a = __builtin_bit_cast(bf16x8, *(lds_cu32x4_ptr)(uintptr_t)((kb_ ^ (32u * ks)) + 8192u * j));
      acc = mfma32x32x16(a, qf[ks], acc);
    }
    return acc;
  };
  // V^T reads: supplier lane u of a 16-lane group reads 4 channels of one key row, key =
  // base + (u >> 2), channels out_ch(dt, 16*g16 + 4*(u & 3)) .. +3. The chunk's bits are
  // dt (2..1) and the lane's (3, 0), so dt is a xor, and 8 rows on flip the swizzle's bit 3.
  const int u = lane & 15, g16 = (lane >> 4) & 1;
  const int vch = out_ch(0, 16 * g16 + 4 * (u & 3));
  const uint32_t vbase = ring_lds + 16u * (uint32_t)swz(4 * hf + (u >> 2), vch >> 3) + 2u * (uint32_t)(vch & 7);

  int rv[kUnits];
#pragma unroll
  for (int j = 0; j < kRing - 1; ++j) {
    if (j < nb) {
      rows_of(j, rv);
      issue(j, rv);
    }
  }
  // The LDS reads that feed the next iteration are issued one iteration early,
  // so their latency hides behind the wait and the compute: the rows of the
  // block to copy next and this lane's slot of the block to compute next.
  if (nb > 0) rows_of(min(kRing - 1, nb - 1), rv);
  int vslot = slot[lane & 31];
  // The compiler-tracked loads (q, sink) are consumed here, so its own waitcnt
  // (a vmcnt(0), which also covers the copies just issued) stays out of the loop.
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) asm volatile("" ::"v"(qf[ks]));
  asm volatile("" ::"v"(m_run));

  // Two-stage pipeline: iteration kb computes S of block kb+1 on the matrix
  // cores while the VALU runs the softmax of block kb, then O += P(kb) V(kb).
  // Block kb+1 must be in LDS at the start of iteration kb, block kb is read
  // until its end; the copy issued in iteration kb (block kb + kRing - 1) goes to
  // the buffer of block kb-1, released by the barrier.
  // One iteration for block kb, which sits in ring buffer j = kb % kRing (the
  // loop is unrolled by kRing so that j, and with it every LDS offset below,
  // is a compile-time constant).
  uint32_t vm_cur = 0u;
  f32x16 s_cur = {};
  // The two dot2 operands live in SGPRs: as a literal, the compiler encodes the
  // pair (-1, 0) as the inline constant -1.0, which v_dot2c_f32_bf16 reads as the
  // fp32 bit pattern, i.e. the pair (0, -1).
  uint32_t neg_lo_bits = kNegLoBits, neg_hi_bits = kNegHiBits;
  asm volatile("" : "+s"(neg_lo_bits), "+s"(neg_hi_bits));
  const bf16v2 neg_lo = __builtin_bit_cast(bf16v2, neg_lo_bits);
  const bf16v2 neg_hi = __builtin_bit_cast(bf16v2, neg_hi_bits);
  auto step = [&](const int kb, const int j) {
    uint32_t vm_next = 0u;
    if (kb + 1 < nb) {
      // Block kb+1 has landed once at most the younger blocks issued so far are outstanding.
      if (kRing == 4 && kb + 2 < nb) wait_vmcnt<kUnits>();
      else wait_vmcnt<0>();
      __syncthreads();  // block kb+1 is in LDS for every wave; block kb-1 is consumed
      if (kb + kRing - 1 < nb) issue((j + kRing - 1) % kRing, rv);
      vm_next = (uint32_t)__ballot(vslot >= 0);
      rows_of(min(kb + kRing, nb - 1), rv);
      vslot = slot[min(kb + 2, nb - 1) * kKB + (lane_id() & 31)];
    }
    // Masked slots of block kb -> -inf (uniform branch; full blocks skip it).
    if (vm_cur != 0xffffffffu) {
      const uint32_t vmh = vm_cur >> (4 * hf);  // bit 8(r/4) + r%4: the lane's key of register r
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if ((vmh & (1u << (8 * (r >> 2) + (r & 3)))) == 0u) s_cur[r] = -INFINITY;
    }
    // max(s) * c2 == max(s * c2) for c2 > 0; the other lane half holds the
    // other 16 keys of the same head.
    float bmax = s_cur[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) bmax = fmaxf(bmax, s_cur[r]);
    bmax *= c2;
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(bmax), __float_as_uint(bmax),
                                                       false, false);
      bmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    // Raise the running max only when this block exceeds it by > kRaise.
    const bool raise = bmax > m_run + kRaise;
    if (__ballot(raise) != 0) {
      const float m_new = raise ? bmax : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      m_run = m_new;
    }

    // S of the next block (after the last block this reads a stale buffer and
    // the result is unused), independent of the softmax below.
    // The wave runs at raised priority from here to the PV products: on a SIMD
    // shared with another workgroup's wave, the softmax (VALU) of one wave then
    // tends to issue while the other's products occupy the matrix cores (~4 %).
    __builtin_amdgcn_s_setprio(1);
    const f32x16 s_next = qk((j + 1) % kRing);

    float pe[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) pe[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[r], c2, -m_run));
#pragma unroll
    for (int r = 0; r < 16; ++r) l_run += pe[r];
    // B operands of the second product, hi + lo bf16: K-step st uses the
    // lane's registers 8st..8st+7 (keys 16st + 8(j/4) + 4hf + j%4).
    bf16x8 phi[2], plo[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      u32x4 wh, wl;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float p0 = pe[8 * st + 2 * w], p1 = pe[8 * st + 2 * w + 1];
        const uint32_t h = pack_bf2(p0, p1);
        wh[w] = h;
        // residuals p - bf16(p), exact in fp32: one v_dot2c each
        const bf16v2 hv = __builtin_bit_cast(bf16v2, h);
        wl[w] = pack_bf2(__builtin_amdgcn_fdot2_f32_bf16(hv, neg_lo, p0, false),
                         __builtin_amdgcn_fdot2_f32_bf16(hv, neg_hi, p1, false));
      }
      phi[st] = __builtin_bit_cast(bf16x8, wh);
      plo[st] = __builtin_bit_cast(bf16x8, wl);
    }
    // O^T += V^T . P^T. A operand rows: channel out_ch(dt, lane%32); the two
    // transposed reads give keys 16st + 4hf + (0..3) and 16st + 8 + 4hf + (0..3).
    // One fragment is read ahead of its two products (the order is pinned below).
    __builtin_amdgcn_s_setprio(0);
    uint32_t vb_ = vbase;
    if constexpr (kRing == 3) asm volatile("" : "+v"(vb_));
    auto rdv = [&](int i) {
      const int st = i >> 2, dt = i & 3;
      const uint32_t at = 8192u * j + 4096u * st;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_s16x4_ptr)(uintptr_t)((vb_ ^ (32u * dt)) + at));
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_s16x4_ptr)(uintptr_t)((vb_ ^ (32u * dt + 128u)) + at + 2048u));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    bf16x8 va = rdv(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      bf16x8 vn = va;
      if (i + 1 < 8) vn = rdv(i + 1);
      o[i & 3] = mfma32x32x16(va, plo[i >> 2], o[i & 3]);
      o[i & 3] = mfma32x32x16(va, phi[i >> 2], o[i & 3]);
      va = vn;
    }
    if constexpr (kRing == 3) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
      for (int i = 0; i < 7; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
    s_cur = s_next;
    vm_cur = vm_next;
  };

  if (nb > 0) {
    if (kRing == 4 && nb >= 3) wait_vmcnt<2 * kUnits>();
    else if (nb >= 2) wait_vmcnt<kUnits>();
    else wait_vmcnt<0>();
    __syncthreads();
    vm_cur = (uint32_t)__ballot(vslot >= 0);
    vslot = slot[min(1, nb - 1) * kKB + (lane & 31)];
    s_cur = qk(0);
    for (int kb0 = 0; kb0 < nb; kb0 += kRing) {
#pragma unroll
      for (int j = 0; j < kRing; ++j) {
        if (kb0 + j >= nb) break;
        step(kb0 + j, j);
      }
    }
  }
  __syncthreads();  // every wave is done with the ring; it is reused below

  // Normalise: Z = sum over both lane halves + exp2(sink - m_run).
  l_run += __shfl_xor(l_run, 32, 64);
  const float rz = 1.0f / (l_run + __builtin_amdgcn_exp2f(sink_l2 - m_run));
  // O^T lane data: head col, channels out_ch(dt, 8(r/4) + 4hf + r%4) =
  // 64hf + 16dt + 4(r/4) + r%4 -> the lane owns channels 64hf .. 64hf+63.
  // Transpose through LDS (ring buffer wi; 32 heads x 16 chunks = 8 KB) for
  // coalesced stores.
  u32x4* obuf = ring[wi];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
    for (int hc = 0; hc < 2; ++hc) {
      // channels 64hf + 16dt + 8hc .. +7 = registers r = 8hc .. 8hc+7
      u32x4 w;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = pack_bf2(o[dt][8 * hc + 2 * k] * rz, o[dt][8 * hc + 2 * k + 1] * rz);
      const int chunk = 8 * hf + 2 * dt + hc;
      obuf[swz(col, chunk)] = w;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  u32x4* dst = reinterpret_cast<u32x4*>(p.out + (tok * p.H + hbase) * kD);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r = 4 * k + (lane >> 4), c = lane & 15;
    if (hbase + r < p.H) st_nt(dst + r * 16 + c, obuf[swz(r, c)]);
  }
}

// One workgroup per (token, 32 heads), whose slot blocks are divided among SP waves: wave
// w takes blocks w, w + SP, ... . Every wave copies its own blocks into its own two LDS
// buffers, so the block loop has no barrier; blocks without a valid slot are skipped.
// Each wave starts its running max at the sink and keeps its own sum and O^T; at the end
// these go to LDS (O^T over the wave's own buffers) and every wave adds up and normalises
// 64 / SP of the 64 register rows over all SP states (in fp32, one rounding to bf16).
//
// What bounds it: with few tokens the latency of the slot list, the rows and one block
// after the other (~0.8 us each), which the split divides; 8 tokens of 64 heads, 512 slots
// of 8192 rows: 16.4 us with the blocks in sequence (sa_gather_kernel), 8.3 us with SP 4;
// 2048 slots: 52.9 us, 17.1 us with SP 8. With many tokens SP 1 serves up to 32 heads:
// 17 KB of LDS per wave instead of a 4-buffer ring's 33 KB keeps two waves on each SIMD
// (4,800 tokens of 16 heads, 256 slots: 57.1 -> 42.4 us). SP 2 was the best choice
// nowhere by more than 8 %.
constexpr int kSplitRing = 2;

template <int SP, typename IdxT>
__global__ __launch_bounds__(64 * SP) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sa_gather_split_kernel(GatherParams p) {
  static_assert(SP == 1 || SP == 4 || SP == 8, "slot ranges per workgroup");
  const IdxT* const idx = static_cast<const IdxT*>(p.idx);
  __shared__ u32x4 ring[SP][kSplitRing][kKB * 16];
  __shared__ float ml[SP][2][64];   // per wave and lane: running max, partial sum
  extern __shared__ int32_t slot[];  // the token's slot indices (masked -> -1)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wi = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ngrp = (p.H + 31) >> 5;  // head groups of 32 (the last may be half full)
  // Blocks go to the 8 XCDs round-robin: the head groups of a token, which read the same
  // rows, take blocks of one XCD, and where sa_gather_kernel pins a batch to an XCD so
  // does this map. The grid is rounded up to 8 tokens; surplus blocks leave at once.
  const unsigned xcd = blockIdx.x & 7u, slotno = (blockIdx.x >> 3) / (unsigned)ngrp;
  const int hbase = 32 * (int)((blockIdx.x >> 3) - slotno * (unsigned)ngrp);
  const int64_t tok = p.xpb > 0
      ? (int64_t)(xcd % (unsigned)p.B) * p.M + (int64_t)slotno * p.xpb + xcd / (unsigned)p.B
      : (int64_t)slotno * 8 + xcd;
  if (tok >= p.B * p.M) return;
  const int b = (int)(tok / p.M);
  const int col = lane & 31;
  const int hf = lane >> 5;
  const bool hvalid = hbase + col < p.H;

  // As in sa_gather_kernel: every global read of the token is issued before the first wait.
  bf16x8 qf[8];
  {
    const uint16_t* qrow = p.q + (tok * p.H + (hvalid ? hbase + col : 0)) * kD + 8 * hf;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      qf[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qrow + 16 * ks));
  }
  const float sink_raw = p.sink[hvalid ? hbase + col : 0];
  const int nblk = (p.TOPK + kKB - 1) / kKB;
  auto slot_chunk = [&](const int s0) {
    int v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + 64 * SP * u + tid;
      v[u] = slot_index(idx, tok * p.TOPK + min(s, p.TOPK - 1));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + 64 * SP * u + tid;
      if (s < nblk * kKB) slot[s] = (s < p.TOPK && v[u] < p.NKV) ? v[u] : -1;
    }
  };
  slot_chunk(0);
  for (int s0 = 4 * 64 * SP; s0 < nblk * kKB; s0 += 4 * 64 * SP) slot_chunk(s0);
  __syncthreads();

  const i32x4 rsrc = make_rsrc(p.kv + (int64_t)b * p.NKV * kD, (uint32_t)p.NKV * (uint32_t)(kD * 2));
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4*)&ring[wi][0][0];
  // Copy block blk into buffer rs: unit u holds rows 4u .. 4u+3, lane l row 4u + l/16, chunk
  // position l%16 (logical chunk (l%16) ^ (row & 15)); a masked row reads zeros.
  auto issue = [&](const int blk, const int rs) {
    int rv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) rv[u] = slot[blk * kKB + 4 * u + (lane >> 4)];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int r = 4 * u + (lane >> 4);
      lds_dma16(rsrc, (uint32_t)rv[u] * (uint32_t)(kD * 2) + 16u * (uint32_t)((lane & 15) ^ (r & 15)),
                ring_lds + 8192u * (uint32_t)rs + 1024u * (uint32_t)u);
    }
  };
  // The first block from blk on (in steps of SP) that holds a valid slot, or nblk; its
  // valid slots in vm.
  auto next_block = [&](int blk, uint32_t& vm) {
    for (; blk < nblk; blk += SP) {
      vm = (uint32_t)__ballot(slot[blk * kKB + (lane & 31)] >= 0);
      if (vm != 0u) return blk;
    }
    vm = 0u;
    return nblk;
  };
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x16{};
  const float sink_l2 = hvalid ? sink_raw * kLog2e : 0.f;
  const float c2 = p.scale_log2;
  float m_run = fmaxf(sink_l2, -FLT_MAX);  // floored as in sa_gather_kernel
  float l_run = 0.f;
  uint32_t neg_lo_bits = kNegLoBits, neg_hi_bits = kNegHiBits;
  asm volatile("" : "+s"(neg_lo_bits), "+s"(neg_hi_bits));
  const bf16v2 neg_lo = __builtin_bit_cast(bf16v2, neg_lo_bits);
  const bf16v2 neg_hi = __builtin_bit_cast(bf16v2, neg_hi_bits);

  uint32_t vm_cur, vm_nxt = 0u;
  int cur = next_block(wi, vm_cur);
  int nxt = nblk;
  if (cur < nblk) {
    issue(cur, 0);
    nxt = next_block(cur + SP, vm_nxt);
    if (nxt < nblk) issue(nxt, 1);
  }
  // The compiler-tracked loads are consumed here, so that its own vmcnt(0) for them (which
  // also covers the copies just issued) stays out of the loop.
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) asm volatile("" ::"v"(qf[ks]));
  asm volatile("" ::"v"(m_run));

  // One block, which sits in buffer j.
  auto step = [&](const int j) {
    if (nxt < nblk) wait_vmcnt<8>();  // only the next block's copies may be outstanding
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    const u32x4* kvl = ring[wi][j];
    f32x16 s = {};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const bf16x8 a = __builtin_bit_cast(bf16x8, kvl[swz(lane & 31, 2 * ks + hf)]);
      s = mfma32x32x16(a, qf[ks], s);
    }
    if (vm_cur != 0xffffffffu) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = 8 * (r >> 2) + 4 * hf + (r & 3);
        if (!((vm_cur >> key) & 1u)) s[r] = -INFINITY;
      }
    }
    float bmax = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) bmax = fmaxf(bmax, s[r]);
    bmax *= c2;
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(bmax), __float_as_uint(bmax),
                                                       false, false);
      bmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    const bool raise = bmax > m_run + kRaise;
    if (__ballot(raise) != 0) {
      const float m_new = raise ? bmax : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      m_run = m_new;
    }
    float pe[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) pe[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -m_run));
#pragma unroll
    for (int r = 0; r < 16; ++r) l_run += pe[r];
    bf16x8 phi[2], plo[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      u32x4 wh, wl;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float p0 = pe[8 * st + 2 * w], p1 = pe[8 * st + 2 * w + 1];
        const uint32_t h = pack_bf2(p0, p1);
        wh[w] = h;
        const bf16v2 hv = __builtin_bit_cast(bf16v2, h);
        wl[w] = pack_bf2(__builtin_amdgcn_fdot2_f32_bf16(hv, neg_lo, p0, false),
                         __builtin_amdgcn_fdot2_f32_bf16(hv, neg_hi, p1, false));
      }
      phi[st] = __builtin_bit_cast(bf16x8, wh);
      plo[st] = __builtin_bit_cast(bf16x8, wl);
    }
    const int u = lane & 15, g16 = (lane >> 4) & 1;
    const uint16_t* kvh = reinterpret_cast<const uint16_t*>(kvl);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const int ch = out_ch(dt, 16 * g16 + 4 * (u & 3));
        const int r0 = 16 * st + 4 * hf + (u >> 2);
        const int r1 = r0 + 8;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4_ptr)(kvh + swz(r0, ch >> 3) * 8 + (ch & 7)));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4_ptr)(kvh + swz(r1, ch >> 3) * 8 + (ch & 7)));
        const s16x8 v01 = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        const bf16x8 a = __builtin_bit_cast(bf16x8, v01);
        o[dt] = mfma32x32x16(a, plo[st], o[dt]);
        o[dt] = mfma32x32x16(a, phi[st], o[dt]);
      }
    }
    // Buffer j is free once its last reads have returned: refill it with the block
    // after the next.
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    uint32_t vm_2 = 0u;
    int nxt2 = nblk;
    if (nxt < nblk) {
      nxt2 = next_block(nxt + SP, vm_2);
      if (nxt2 < nblk) issue(nxt2, j);
    }
    cur = nxt;
    vm_cur = vm_nxt;
    nxt = nxt2;
    vm_nxt = vm_2;
  };
  while (cur < nblk) {
    step(0);
    if (cur >= nblk) break;
    step(1);
  }

  if constexpr (SP == 1) {
    // One state: normalise it and transpose it through the wave's own buffers (chunk c of
    // head col at swz(col, c)), so that every store writes four whole rows.
    l_run += __shfl_xor(l_run, 32, 64);
    const float rz = 1.0f / (l_run + __builtin_amdgcn_exp2f(sink_l2 - m_run));
    u32x4* obuf = &ring[0][0][0];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      u32x4 w;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = pack_bf2(o[c >> 1][8 * (c & 1) + 2 * k] * rz, o[c >> 1][8 * (c & 1) + 2 * k + 1] * rz);
      obuf[swz(col, 8 * hf + c)] = w;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    u32x4* dst = reinterpret_cast<u32x4*>(p.out + (tok * p.H + hbase) * kD);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int r = 4 * k + (lane >> 4), c = lane & 15;
      if (hbase + r < p.H) st_nt(dst + r * 16 + c, obuf[swz(r, c)]);
    }
    return;
  }
  // The states of all waves: O^T register rows 4k .. 4k+3 of a lane at [k][lane].
  u32x4* mine = &ring[wi][0][0];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x4 v = {o[dt][4 * k], o[dt][4 * k + 1], o[dt][4 * k + 2], o[dt][4 * k + 3]};
      mine[(4 * dt + k) * 64 + lane] = __builtin_bit_cast(u32x4, v);
    }
  ml[wi][0][lane] = m_run;
  ml[wi][1][lane] = l_run;
  __syncthreads();
  float mx = m_run;
#pragma unroll
  for (int w = 0; w < SP; ++w) mx = fmaxf(mx, ml[w][0][lane]);
  float z = __builtin_amdgcn_exp2f(sink_l2 - mx);
  float f[SP];
#pragma unroll
  for (int w = 0; w < SP; ++w) {
    f[w] = __builtin_amdgcn_exp2f(ml[w][0][lane] - mx);
    z += (ml[w][1][col] + ml[w][1][col + 32]) * f[w];
  }
  const float rz = 1.0f / z;
  // Wave wi finishes 8 / SP chunks of 8 channels per lane (chunk c = register rows
  // 8c .. 8c+7 = channels 64 hf + 8 c .. +7 of head col).
#pragma unroll
  for (int i = 0; i < 8 / SP; ++i) {
    const int c = (8 / SP) * wi + i;
    f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < SP; ++w) {
      const f32x4 v0 = __builtin_bit_cast(f32x4, (&ring[w][0][0])[(2 * c) * 64 + lane]);
      const f32x4 v1 = __builtin_bit_cast(f32x4, (&ring[w][0][0])[(2 * c + 1) * 64 + lane]);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        a0[k] += v0[k] * f[w];
        a1[k] += v1[k] * f[w];
      }
    }
    const u32x4 w = {pack_bf2(a0[0] * rz, a0[1] * rz), pack_bf2(a0[2] * rz, a0[3] * rz),
                     pack_bf2(a1[0] * rz, a1[1] * rz), pack_bf2(a1[2] * rz, a1[3] * rz)};
    if (hvalid)
      *reinterpret_cast<u32x4*>(p.out + (tok * p.H + hbase + col) * kD + 64 * hf + 8 * c) = w;
  }
}

// Waves per (token, 32 heads) of sa_gather_split_kernel, or 0 for sa_gather_kernel, for
// `groups` = tokens x head groups of nblk slot blocks on cu CUs. Measured at 16 .. 128
// heads, 32 .. 2048 slots and 8 .. 8192 groups (256 CUs; us, sequential -> split):
//  up to one group per CU the split takes the CU's waves: 8 from 32 blocks on (1024 slots:
//    35.0 -> 12.5, four waves 13.3), 4 from 4 blocks on (128 slots: 7.3 -> 5.5), else one
//    (64 slots: 5.8 -> 5.1);
//  up to two groups per CU, 4 waves from 8 blocks on (512 slots, 512 groups: 16.8 -> 13.1);
//    with fewer blocks the states cost what the split saves (128 slots: 7.7 -> 8.4);
//  beyond that, more than 32 heads stay sequential, where the waves of a token share each
//    row's copy (512 slots, 1536 groups: 23.3, one wave 27.6), and up to 32 heads take one
//    wave (512 slots, 8192 groups: 153.8 -> 108), or 4 where the slot list would leave
//    room for fewer than 7 one-wave workgroups per CU (2048 slots, 3072 groups: one wave
//    181, four 169).
// Masked slots are not known here: where one block of a long list is valid the split costs up to
// 1.7 us (8 tokens x 64 heads, 10 of 1024 slots 5.7 -> 7.3; 100 of them 7.9 -> 7.4).
int gather_split(int64_t groups, int nw, int64_t nblk, int cu) {
  if (groups <= cu) return nblk >= 32 ? 8 : nblk >= 4 ? 4 : 1;
  if (groups <= 2 * (int64_t)cu && nblk >= 8) return 4;
  if (nw > 1) return 0;
  return nblk >= 48 ? 4 : 1;
}

// The form of sa_gather_kernel (kRing) for `tokens` workgroups of nw waves on cu CUs. The
// three-wave form holds 12 waves per CU (6, 4, 3 workgroups of 2, 3, 4 waves) and the two-wave
// form 8 (4, 2, 2), which a CU works off in 1.2 (32 slots) to 1.5 times (from 512) less time, so
// what counts is in how many rounds the grid fits. Measured at 300 .. 8000 tokens and 32 .. 2048
// slots (256 CUs; us, two waves -> three):
//  one round of the two-wave form: that one (300 tokens x 64 heads, 1024 slots 33.3 -> 35.2;
//    400 x 96, 512 20.7 -> 21.5; 400 x 128, 256 14.2 -> 14.9);
//  4 waves, 3 to 4 tokens per CU: two rounds of either, two-wave (900 x 128, 2048 slots 157 ->
//    169), else three waves (640: 136 -> 116; 4000, 512 slots: 197 -> 184);
//  3 waves: three waves (900 x 96, 512 slots: 43 -> 38);
//  2 waves: above 544 slots the slot list leaves LDS for five workgroups of the three-wave
//    form, unevenly over the four SIMDs: two-wave (4000 x 64, 1024 slots: 184 -> 198; 1500: 81 ->
//    89), but for the last block count, where it has room for three workgroups only and the
//    three-wave form for four (900 x 64, 2048 slots: 126 -> 87; 1200: 136 -> 160). Up to 544
//    slots three waves (1500 x 64, 512 slots: 47 -> 41; 8000: 201 -> 194) but where their second
//    round is nearly empty (2000, 512 slots: 54 -> 58; 4 x 500 causal, 32 slots: 17.5 -> 20.9).
int gather_ring(int64_t tokens, int nw, int64_t nblk, int cu) {
  const auto rounds = [&](int per_cu) { return (tokens + per_cu * (int64_t)cu - 1) / (per_cu * (int64_t)cu); };
  if (nw > 2) return tokens <= 2 * (int64_t)cu || (nw == 4 && rounds(3) == 2 && rounds(4) == 1) ? 4 : 3;
  if (nblk == 64) return 4 * rounds(4) < 3 * rounds(3) ? 3 : 4;
  if (nblk > 17 || rounds(4) == 1) return 4;
  return rounds(6) == 2 && tokens < 8 * (int64_t)cu ? 4 : 3;
}

template <typename IdxT>
int launch_split(const GatherParams& p, int sp, unsigned blocks, size_t smem, hipStream_t stream) {
  switch (sp) {
#define DSA_GATHER_CASE(n)                                                                          \
  case n:                                                                                           \
    if (dsa_host::ensure_dyn_lds((const void*)sa_gather_split_kernel<n, IdxT>, (int)smem) != DSA_OK) \
      return DSA_ERR_LAUNCH;                                                                        \
    hipLaunchKernelGGL((sa_gather_split_kernel<n, IdxT>), dim3(blocks), dim3(64 * n), smem, stream, p); \
    break;
    DSA_GATHER_CASE(1)
    DSA_GATHER_CASE(4)
    DSA_GATHER_CASE(8)
#undef DSA_GATHER_CASE
    default:
      return DSA_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? DSA_OK : DSA_ERR_LAUNCH;
}

template <typename IdxT>
int launch_ring(const GatherParams& p, int ring, int nw, unsigned tokens, size_t smem, hipStream_t stream) {
  switch (4 * nw + ring) {
#define DSA_GATHER_CASE(n, r)                                                                          \
  case 4 * n + r:                                                                                      \
    hipLaunchKernelGGL((sa_gather_kernel<n, IdxT, r>), dim3(tokens), dim3(64 * n), smem, stream, p);   \
    break;
    DSA_GATHER_CASE(2, 3)
    DSA_GATHER_CASE(3, 3)
    DSA_GATHER_CASE(4, 3)
    DSA_GATHER_CASE(2, 4)
    DSA_GATHER_CASE(3, 4)
    DSA_GATHER_CASE(4, 4)
#undef DSA_GATHER_CASE
    default:
      return DSA_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? DSA_OK : DSA_ERR_LAUNCH;
}

}  // namespace

int dsa_sparse_attn_gather_launch(const void* q, const void* kv, const void* idx, bool idx64,
                                  const float* sink, void* out, int64_t b, int64_t m, int64_t h,
                                  int64_t n_kv, int64_t topk, float scale, hipStream_t stream) {
  if (h % 16 != 0 || h > 128) return DSA_ERR_UNSUPPORTED;
  if (topk > 2048) return DSA_ERR_UNSUPPORTED;
  if (!(scale > 0.f) || !(scale < INFINITY)) return DSA_ERR_UNSUPPORTED;  // the kernel's max uses scale > 0
  if (n_kv > (INT64_C(1) << 23)) return DSA_ERR_UNSUPPORTED;  // byte offsets of kv rows fit 32 bits
  const int64_t tokens = b * m;
  if (tokens > INT32_MAX) return DSA_ERR_SHAPE;
  GatherParams p;
  p.q = (const uint16_t*)q;
  p.kv = (const uint16_t*)kv;
  p.idx = idx;
  p.sink = sink;
  p.out = (uint16_t*)out;
  p.M = m;
  p.B = (int32_t)b;
  p.H = (int32_t)h;
  p.NKV = (int32_t)n_kv;
  p.TOPK = (int32_t)topk;
  p.scale_log2 = scale * kLog2e;
  p.xpb = (b <= 8 && 8 % b == 0 && m % (8 / b) == 0) ? (int32_t)(8 / b) : 0;
  // Dynamic LDS: the slot list, padded to whole blocks.
  const int64_t nblk = (topk + kKB - 1) / kKB;
  const size_t smem = (size_t)nblk * kKB * sizeof(int32_t);
  const int nw = (int)((h + 31) / 32);
  if (nw < 1 || nw > 4) return DSA_ERR_UNSUPPORTED;
  int cu = 0;
  if (dsa_host::device_cu_count(&cu) != DSA_OK) return DSA_ERR_DEVICE;
  const int sp = gather_split(tokens * nw, nw, nblk, cu);
  if (sp > 0) {
    const int64_t blocks = (tokens + 7) / 8 * 8 * nw;
    if (blocks > INT32_MAX) return DSA_ERR_SHAPE;
    return idx64 ? launch_split<int64_t>(p, sp, (unsigned)blocks, smem, stream)
                 : launch_split<int32_t>(p, sp, (unsigned)blocks, smem, stream);
  }
  const int ring = gather_ring(tokens, nw, nblk, cu);
  return idx64 ? launch_ring<int64_t>(p, ring, nw, (unsigned)tokens, smem, stream)
               : launch_ring<int32_t>(p, ring, nw, (unsigned)tokens, smem, stream);
}
