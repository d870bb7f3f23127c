// Attention for few queries per sequence over long keys (decoding steps) on
// gfx950: flash_varlen_fwd_kernel's contract (ops/suite/dev/
// flash_varlen_fwd_kernel.py:22-320) for calls whose query rows of one KV
// head -- seqlen_q queries x (h / hk) heads -- fit 16 or 32 MFMA columns.
//
// Such a call is bound by reading K and V once.  The prefill kernel gives
// every query head a workgroup of 256 query rows: it multiplies 255 rows of
// padding, reads each KV head once per query head and leaves a sequence's
// keys to one workgroup, however long it is.  Here
//   * a workgroup owns one (sequence, KV head, key range): the queries of all
//     heads sharing the KV head are the columns of one MFMA tile, so K and V
//     leave HBM once.  The host cuts the keys into `splits` ranges when the
//     (sequence, KV head) pairs alone would not fill the chip or would leave
//     it waiting for the longest sequence; attn_decode_merge joins them.
//     Without a workspace for their records (captured graphs, no-alloc
//     calls) one workgroup takes a pair's ranges in turn and joins them in
//     registers by the same operations in the same order (DecRow), so both
//     forms of a call give the same bits;
//   * its 4 waves take 16-key tiles in turn and share nothing until the end:
//     each has its own LDS ring filled by direct global->LDS DMA and waits
//     for its own loads only, so there is no barrier in the loop.  64 KiB of
//     LDS per workgroup: two workgroups per CU, 64-128 KiB in flight;
//   * S^T = K.Q^T on v_mfma_f32_16x16x32 (keys x query rows): a lane holds
//     four scores of one query row, and those four keys are exactly the k
//     slots of that lane in v_mfma_f32_16x16x16, so P feeds O^T = V^T.P^T
//     from registers; V^T comes from ds_read_b64_tr_b16;
//   * the running maximum and sum of a row live in the four lanes holding it,
//     exchanged only when some lane's tile maximum exceeds the reference by
//     more than 8 (attention.hip's rule, exact since l and O share it).
// A K or V row is 16 (8 at d = 64) chunks of 16 bytes; K's chunk index is
// XOR-swizzled by the key so the 16 keys of a fragment read cover the 64
// banks once, V's by 32-byte pieces so a transposing read does.
namespace g950 {

constexpr int DEC_WAVES = 4;
constexpr int DEC_TK = 16;          // keys per tile of one wave
constexpr int DEC_RING = 16384;     // LDS bytes of one wave's ring

__device__ __forceinline__ f32x4 mfma16x16x16(const u32x2& a, const u32x2& b, const f32x4& c, std::true_type) {
  typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
  return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0,
                                               0);
}
__device__ __forceinline__ f32x4 mfma16x16x16(const u32x2& a, const u32x2& b, const f32x4& c, std::false_type) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0,
                                                   0, 0);
}

// a wave-uniform address as a scalar (the DMA's base)
__device__ __forceinline__ const char* uniform_ptr(const char* p) {
  const uint64_t a = (uint64_t)p;
  return (const char*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)a));
}

// value of `v` combined over the four lanes holding one query row
template <class Op>
__device__ __forceinline__ float row4(float v) {
  v = Op::apply(v, __shfl_xor(v, 16));
  return Op::apply(v, __shfl_xor(v, 32));
}

// A query row's key ranges joined one after the other: maximum (log2 units)
// and sum so far.  join() takes the next range's and gives the weights of
// what was gathered before (was) and of the range's own O (now); a range in
// which the row saw no key has weight 0 and is to be left out (its O may hold
// anything).  Both users apply them as fmaf(now, range, was * gathered).
struct DecRow {
  float m = -__builtin_huge_valf(), l = 0.0f;
  __device__ __forceinline__ bool join(float mr, float lr, float& was, float& now) {
    if (mr == -__builtin_huge_valf() && lr == 0.0f) return false;
    const float to = fmaxf(m, mr);
    // no finite score yet on a side: its sum is 0, or NaN and kept
    was = m == -__builtin_huge_valf() ? 1.0f : __builtin_amdgcn_exp2f(m - to);
    now = mr == -__builtin_huge_valf() ? 1.0f : __builtin_amdgcn_exp2f(mr - to);
    l = fmaf(now, lr, was * l);
    m = to;
    return true;
  }
};

// RT: 16-row query tiles per workgroup (1 or 2).  PG: 0 contiguous K/V rows,
// 1 pages of a multiple of 16 keys (a tile lies in one page).  PART: this
// workgroup takes one of a pair's ranges and leaves its record, else all of
// them.
template <int D, bool F16, int RT, int PG, bool PART>
__device__ __forceinline__ void attn_decode_body(const AttnDecArgs& g) {
  constexpr int ROW = D * 2, CH = ROW / 16;      // row bytes, 16-byte chunks per row
  constexpr int KT = DEC_TK * ROW;               // K (or V) bytes of one tile
  constexpr int ST = DEC_RING / (2 * KT);        // tiles in flight per wave
  constexpr int DPT = 2 * KT / 1024;             // DMA instructions per tile
  constexpr int KPI = 64 / CH;                   // keys per DMA instruction
  constexpr int DS = D / 32, DB = D / 16;        // k-steps of S^T, 16-d blocks of O^T
  constexpr int ROWS = 16 * RT;
  static_assert(ROWS * D * 4 <= DEC_RING, "a wave's partial O fits its ring");
  __shared__ __attribute__((aligned(1024))) char lds[DEC_WAVES * DEC_RING];
  __shared__ float ml[DEC_WAVES][ROWS][2];
  if (blockDim.x != DEC_WAVES * 64) return;  // launch shape must match the kernel
  const AttnArgs& p = g.a;
  const VarlenArgs& vl = g.v;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, l16 = lane & 15;
  const int pairs = p.Z * p.Hkv;
  const int split = PART ? blockIdx.x / pairs : 0, pair = blockIdx.x % pairs;
  const int z = pair / p.Hkv, hk = pair % p.Hkv;
  const int G = p.group;
  const SeqGeom sg = varlen_geom(p, vl, z);
  const int Sq = sg.q_len, Sk = sg.k_len;
  const bool has_hi = p.causal || vl.local, has_lo = vl.local;
  const int hi_off = Sk - Sq + vl.wr, lo_off = Sk - Sq - vl.wl;
  const char* kbase = (const char*)p.k + 2 * (sg.k_off + (long long)hk * p.k_sh);
  const char* vbase = (const char*)p.v + 2 * (sg.v_off + (long long)hk * p.v_sh);
  const long long kstride = 2 * p.k_ss, vstride = PG ? kstride : 2 * p.v_ss;
  char* ring = lds + wave * DEC_RING;  // this wave's
  const uint32_t ring32 = lds_addr(ring);
  // queries per pass: seqlen_q (the host: seqlen_q * group <= ROWS), so a
  // pass's rows are those a pair's partial records have room for
  const int qpass = g.rows / G;

  // lane's share of a DMA instruction: key u * KPI + dkey, LDS chunk slot dpos
  const int dkey = lane / CH, dpos = lane % CH;
  auto kswz = [](int key) { return D == 128 ? key & 15 : (key >> 1) & 7; };
  auto vswz = [](int key) { return D == 128 ? key & 7 : (key >> 1) & 3; };
  // LDS offsets: K chunk 4 ks + g4 of key l16; V 16-d block b of the four
  // keys 4 g4 .. + 3 (lane l16: key 4 g4 + l16 / 4, 8 bytes l16 % 4)
  int koff[DS];
#pragma unroll
  for (int ks = 0; ks < DS; ++ks) koff[ks] = l16 * ROW + (((4 * ks + g4) ^ kswz(l16)) << 4);
  const int vkey = 4 * g4 + (l16 >> 2);
  const int voff = KT + vkey * ROW + (vswz(vkey) << 5) + (l16 & 3) * 8;

  // A sequence holding more queries than seqlen_q (outside the contract, but
  // in reach of a device-held length): the further passes run over all keys
  // in one range, by the workgroup of the first.
  for (int q0 = 0; q0 < Sq && q0 < 256; q0 += qpass) {
    const bool ranged = q0 == 0 && g.splits > 1;
    if (PART && !ranged && split != 0) break;
    const int qn = min(qpass, Sq - q0);  // queries of this pass
    int kend = Sk;
    if (has_hi) kend = min(kend, q0 + qn - 1 + hi_off + 1);
    const int kbeg = has_lo ? max(0, q0 + lo_off) / DEC_TK * DEC_TK : 0;

    // query fragments (B port): row rt*16 + l16 = query qi of head hk*G + hg
    u32x4 qf[RT][DS];
    int qi[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int r = rt * 16 + l16;
      const int qr = min(r / G, qn - 1), hg = r % G;
      qi[rt] = q0 + qr;
      const char* src = (const char*)p.q +
                        2 * (sg.q_off + (long long)(hk * G + hg) * p.q_sh + (long long)(q0 + qr) * p.q_ss);
#pragma unroll
      for (int ks = 0; ks < DS; ++ks) qf[rt][ks] = *(const u32x4*)(src + (ks * 32 + g4 * 8) * 2);
    }

    // keys lo .. hi - 1 (of the pass's window) into the waves' partial rows
    auto attend = [&](int lo, int hi) {
      const int ntiles = hi > lo ? (hi - lo + DEC_TK - 1) / DEC_TK : 0;
      const int nloc = ntiles > wave ? (ntiles - wave + DEC_WAVES - 1) / DEC_WAVES : 0;

      // page numbers of this wave's next 64 tiles, one per lane
      int pages = 0;
      auto issue = [&](int j) {
        const int kv0 = lo + DEC_TK * (wave + DEC_WAVES * j);
        long long row0 = 0;  // byte offset of the tile's first key row
        if constexpr (PG == 1) {
          if ((j & 63) == 0) {
            const int key = kv0 + DEC_TK * DEC_WAVES * lane;
            const long long e = (long long)z * vl.pt_stride + key / vl.block_size;
            int ph = key < hi && e < vl.pt_elems ? vl.page_table[e] : 0;
            pages = ph < 0 || ph >= vl.pages ? 0 : ph;
          }
          const int ph = __builtin_amdgcn_readlane(pages, j & 63);
          row0 = 2 * (long long)ph * vl.page_stride + (long long)(kv0 % vl.block_size) * kstride;
        }
        const char* ks0 = uniform_ptr(kbase + (PG ? row0 : (long long)kv0 * kstride));
        const char* vs0 = uniform_ptr(vbase + (PG ? row0 : (long long)kv0 * vstride));
        const uint32_t dst = ring32 + (j % ST) * 2 * KT;
        const int last = Sk - 1 - kv0;  // keys past the end repeat the last one
#pragma unroll
        for (int u = 0; u < DPT / 2; ++u) {
          const int key = u * KPI + dkey;
          dma16_asm(ks0, (uint32_t)(min(key, last) * (int)kstride) + ((dpos ^ kswz(key)) << 4), dst + u * 1024);
        }
#pragma unroll
        for (int u = 0; u < DPT / 2; ++u) {
          const int key = u * KPI + dkey;
          dma16_asm(vs0, (uint32_t)(min(key, last) * (int)vstride) + ((dpos ^ (vswz(key) << 1)) << 4),
                    dst + KT + u * 1024);
        }
      };

      f32x4 o[RT][DB];
      float ms[RT], l[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        ms[rt] = -__builtin_huge_valf();
        l[rt] = 0.0f;
#pragma unroll
        for (int b = 0; b < DB; ++b) o[rt][b] = (f32x4){};
      }
      const float c2 = p.scale_log2;
      for (int j = 0; j < ST && j < nloc; ++j) issue(j);
      for (int i = 0; i < nloc; ++i) {
        // tile i has landed once at most the later tiles' loads are in flight
        if (i + ST <= nloc) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 1) * DPT) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const char* st = ring + (i % ST) * 2 * KT;
        const int kv0 = lo + DEC_TK * (wave + DEC_WAVES * i);
        f32x4 s[RT];
        i32x4 unused;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) s[rt] = (f32x4){};
#pragma unroll
        for (int ks = 0; ks < DS; ++ks) {
          const u32x4 kf = *(const u32x4*)(st + koff[ks]);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) mfma16_step<F16 ? GEMM_F16 : GEMM_BF16>(kf, qf[rt][ks], s[rt], unused);
        }
        // keys kv0 + 4 g4 .. + 3 of query row l16
        const bool mask = kv0 + DEC_TK > Sk || (has_hi && kv0 + DEC_TK - 1 > q0 + hi_off) ||
                          (has_lo && kv0 < q0 + qn - 1 + lo_off);
        if (mask) {
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = kv0 + 4 * g4 + e;
              if (key >= Sk || (has_hi && key > qi[rt] + hi_off) || (has_lo && key < qi[rt] + lo_off))
                s[rt][e] = -__builtin_huge_valf();
            }
        }
        u32x2 pf[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const float mh = vmax3(vmax3(s[rt][0], s[rt][1], s[rt][2]), s[rt][3], s[rt][3]) * c2;
          if (__any(mh > ms[rt] + 8.0f)) {
            const float mt = row4<OpMax>(mh);
            const bool move = mt > ms[rt] + 8.0f;
            const float alpha = move ? __builtin_amdgcn_exp2f(ms[rt] - mt) : 1.0f;
            l[rt] *= alpha;
#pragma unroll
            for (int b = 0; b < DB; ++b) o[rt][b] *= alpha;
            ms[rt] = move ? mt : ms[rt];
          }
          // rows without a visible key so far: exponent base 0, exp2(-inf) = 0
          const float mb = (ms[rt] == -__builtin_huge_valf()) ? 0.0f : ms[rt];
          float pe[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) pe[e] = __builtin_amdgcn_exp2f(fmaf(s[rt][e], c2, -mb));
          l[rt] += (pe[0] + pe[1]) + (pe[2] + pe[3]);
          pf[rt] = (u32x2){pack2(pe[0], pe[1], F16), pack2(pe[2], pe[3], F16)};
        }
#pragma unroll
        for (int b = 0; b < DB; ++b) {
          typedef short s16x4 __attribute__((ext_vector_type(4)));
          const s16x4 vf = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(st + (voff ^ (b << 5))));
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            o[rt][b] = mfma16x16x16(__builtin_bit_cast(u32x2, vf), pf[rt], o[rt][b], std::bool_constant<F16>{});
        }
        // this tile's LDS reads have returned before its slot is refilled
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (i + ST < nloc) issue(i + ST);
      }

      // ---- the four waves' partial rows: O through each wave's own ring
      // (16-byte chunks XOR-swizzled by the row), maxima and sums beside it
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int r = rt * 16 + l16;
        const float ls = row4<OpSum>(l[rt]);
#pragma unroll
        for (int b = 0; b < DB; ++b) *(f32x4*)(ring + r * D * 4 + (((4 * b + g4) ^ l16) << 4)) = o[rt][b];
        if (g4 == 0) {
          ml[wave][r][0] = ms[rt];
          ml[wave][r][1] = ls;
        }
      }
      __syncthreads();
    };
    // chunk c of row r over the four waves: O unnormalised, maximum m, sum lt
    auto waves = [&](int r, int c, float& m, float& lt) {
      m = ml[0][r][0];
#pragma unroll
      for (int w = 1; w < DEC_WAVES; ++w) m = fmaxf(m, ml[w][r][0]);
      f32x4 sum = {};
      lt = 0.0f;
#pragma unroll
      for (int w = 0; w < DEC_WAVES; ++w) {
        const float mw = ml[w][r][0], lw = ml[w][r][1];
        // no finite score: no key of this row (l = 0), or only NaN ones
        const float f = mw == -__builtin_huge_valf() ? 1.0f : __builtin_amdgcn_exp2f(mw - m);
        lt = fmaf(f, lw, lt);
        const f32x4 ow = *(const f32x4*)(lds + w * DEC_RING + r * D * 4 + ((c ^ (r & 15)) << 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = fmaf(f, ow[e], sum[e]);
      }
      return sum;
    };
    auto store = [&](int r, int c, const f32x4& sum, float m, float lt) {
      const int h = hk * G + r % G, q = q0 + r / G;
      const bool empty = !(lt > 0.0f);  // zero or NaN
      const float inv = empty ? 1.0f : 1.0f / lt;
      char* dst = (char*)p.o + 2 * (sg.o_off + (long long)h * p.o_sh + (long long)q * p.o_ss + c * 4);
      *(u32x2*)dst = (u32x2){pack2(sum[0] * inv, sum[1] * inv, F16), pack2(sum[2] * inv, sum[3] * inv, F16)};
      if (c == 0)
        p.lse[sg.lse_off + (long long)h * p.lse_sh + q] =
            empty ? __builtin_huge_valf() : (m + __log2f(lt)) * 0.69314718055994530942f;
    };

    // range n of the pass: its keys, of the pass's window
    auto bounds = [&](int n, int& lo, int& hi) {
      lo = ranged ? max(kbeg, n * g.chunk) : kbeg;
      hi = ranged && n + 1 < g.splits ? min(kend, (n + 1) * g.chunk) : kend;
    };
    constexpr int CPR = D / 4;  // 16-byte chunks (4 d) per row
    constexpr int NT = DEC_WAVES * 64;
    int lo, hi;
    if constexpr (PART) {
      bounds(split, lo, hi);
      attend(lo, hi);
      for (int it = tid; it < qn * G * CPR; it += NT) {
        const int r = it / CPR, c = it % CPR;
        float m, lt;
        const f32x4 sum = waves(r, c, m, lt);
        if (!ranged) {
          store(r, c, sum, m, lt);
          continue;
        }
        // record (pair, row, split): O unnormalised at the row's D floats,
        // maximum and sum behind all the O rows
        const long long rec = ((long long)pair * g.rows + r) * g.splits + split;
        *(f32x4*)(g.part + rec * D + c * 4) = sum;
        if (c == 0) {
          g.ml[2 * rec] = m;
          g.ml[2 * rec + 1] = lt;
        }
      }
      __syncthreads();  // the rings are free for a further pass
    } else {
      // thread tid's chunks tid + NT i gather the ranges
      constexpr int OUT = (ROWS * CPR + NT - 1) / NT;
      DecRow row[OUT];
      f32x4 acc[OUT];
#pragma unroll
      for (int i = 0; i < OUT; ++i) acc[i] = (f32x4){};
      for (int n = 0; n < (ranged ? g.splits : 1); ++n) {
        bounds(n, lo, hi);
        if (lo >= hi) continue;  // no key: nothing to join
        attend(lo, hi);
#pragma unroll
        for (int i = 0; i < OUT; ++i) {
          const int it = tid + NT * i;
          if (it >= qn * G * CPR) continue;
          float m, lt, was, now;
          const f32x4 sum = waves(it / CPR, it % CPR, m, lt);
          if (!row[i].join(m, lt, was, now)) continue;
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] = fmaf(now, sum[e], was * acc[i][e]);
        }
        __syncthreads();  // the rings are free for the next range or pass
      }
#pragma unroll
      for (int i = 0; i < OUT; ++i) {
        const int it = tid + NT * i;
        if (it < qn * G * CPR) store(it / CPR, it % CPR, acc[i], row[i].m, row[i].l);
      }
    }
  }
}

// Joins the key ranges of attn_decode_body: one wave per (sequence, head,
// query), D / 64 outputs per lane.  Lane s holds range s's maximum and sum and
// works out DecRow's weights at range s (its maximum so far is the greatest
// of the ranges up to s); they are applied in the ranges' order.
template <int D, bool F16>
__device__ __forceinline__ void attn_decode_merge_body(const AttnDecArgs& g) {
  const AttnArgs& p = g.a;
  const int lane = threadIdx.x & 63;
  const int item = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (item >= p.Z * p.Hkv * g.rows) return;
  const int pair = item / g.rows, r = item % g.rows;
  const int z = pair / p.Hkv, hk = pair % p.Hkv;
  const int h = hk * p.group + r % p.group, q = r / p.group;
  // eight records' O in flight, the first of them beside the maxima and sums
  constexpr int E = D / 64, U = 8;
  const long long rec = (long long)item * g.splits;
  float v[U][E];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) v[u][e] = g.part[(rec + min(s0 + u, g.splits - 1)) * D + lane * E + e];
  };
  load(0);
  float m = -__builtin_huge_valf(), l = 0.0f;
  if (lane < g.splits) {
    m = g.ml[2 * (rec + lane)];
    l = g.ml[2 * (rec + lane) + 1];
  }
  const SeqGeom sg = varlen_geom(p, g.v, z);
  if (q >= sg.q_len) return;
  // greatest maximum of ranges 0 .. lane (row_shr 1, 2, 4, 8, then across rows)
  constexpr float none = -__builtin_huge_valf();
  float to = fmaxf(m, dpp_f32<0x111, 0xF>(none, m));
  to = fmaxf(to, dpp_f32<0x112, 0xF>(none, to));
  to = fmaxf(to, dpp_f32<0x114, 0xF>(none, to));
  to = fmaxf(to, dpp_f32<0x118, 0xF>(none, to));
  to = fmaxf(to, dpp_f32<0x142, 0xA>(none, to));
  to = fmaxf(to, dpp_f32<0x143, 0xC>(none, to));
  const float before = __shfl_up(to, 1);  // by all lanes
  auto of = [](float x, int s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), s));
  };
  const float mt = of(to, 63);  // (read here, where every lane has worked its part out)
  DecRow row;
  row.m = lane ? before : none;
  float was, now;
  const bool seen = row.join(m, l, was, now);
  // a range left out: 0 x -0 + 1 x what was gathered, without a branch
  const uint64_t live = __ballot(seen);
  was = seen ? was : 1.0f;
  now = seen ? now : 0.0f;
  float acc[E] = {}, lt = 0.0f;
  for (int s0 = 0; s0 < g.splits; s0 += U) {
    if (s0) load(s0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;  // (a lane past the ranges is one left out)
      const float w = of(was, s), n = of(now, s);
      lt = fmaf(n, of(l, s), w * lt);
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] = fmaf(n, (live >> s) & 1 ? v[u][e] : -0.0f, w * acc[e]);
    }
  }
  const bool empty = !(lt > 0.0f);  // zero or NaN
  const float inv = empty ? 1.0f : 1.0f / lt;
  uint16_t* dst = (uint16_t*)p.o + sg.o_off + (long long)h * p.o_sh + (long long)q * p.o_ss + lane * E;
#pragma unroll
  for (int e = 0; e < E; ++e) dst[e] = F16 ? f32_to_f16(acc[e] * inv) : f32_to_bf16(acc[e] * inv);
  if (lane == 0)
    p.lse[sg.lse_off + (long long)h * p.lse_sh + q] =
        empty ? __builtin_huge_valf() : (mt + __log2f(lt)) * 0.69314718055994530942f;
}

}  // namespace g950

// _part: one of a pair's key ranges per workgroup; without it all of them.
// Two waves per SIMD (256 registers), so that two workgroups share a CU: left
// to itself the compiler gave the paged 32-row form at d = 128 264 and the
// forms that gather all ranges up to 305; bounded they take 185 to 233 without
// a spill.  Groups of 8, 4 queries, 64-key pages: 64 sequences of 2048 keys
// (32/4 heads) 72.3 -> 58.2 us, 64 of 4096..300 (8/1) 40.9 -> 29.6.
#define G950_DEC_BODY(NAME, D, F16, RT, PG)                                                     \
  extern "C" __global__ __launch_bounds__(256, 2) void NAME(const g950::AttnDecArgs g) {        \
    g950::attn_decode_body<D, F16, RT, PG, false>(g);                                           \
  }                                                                                             \
  extern "C" __global__ __launch_bounds__(256, 2) void NAME##_part(const g950::AttnDecArgs g) { \
    g950::attn_decode_body<D, F16, RT, PG, true>(g);                                            \
  }
#define G950_DEC(NAME, D, F16)                                                                     \
  G950_DEC_BODY(NAME##_r16, D, F16, 1, 0)                                                          \
  G950_DEC_BODY(NAME##_r16_pg, D, F16, 1, 1)                                                       \
  G950_DEC_BODY(NAME##_r32, D, F16, 2, 0)                                                          \
  G950_DEC_BODY(NAME##_r32_pg, D, F16, 2, 1)                                                       \
  extern "C" __global__ __launch_bounds__(256) void NAME##_merge(const g950::AttnDecArgs g) {      \
    g950::attn_decode_merge_body<D, F16>(g);                                                       \
  }
G950_DEC(g950_attn_dec_bf16_d128, 128, false)
G950_DEC(g950_attn_dec_bf16_d64, 64, false)
G950_DEC(g950_attn_dec_f16_d128, 128, true)
G950_DEC(g950_attn_dec_f16_d64, 64, true)
