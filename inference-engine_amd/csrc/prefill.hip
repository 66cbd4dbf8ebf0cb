// prefill.hip -- chunked-prefill attention (include/paged_kv.h: pkv_paged_prefill*): the
// argument checks and launches of the matrix-core kernel (prefill_kernels.h, also
// cascade decode's prefix pass), and the fp32 matrix-core kernel for fp32 K/V and
// head_dim 16.

#include "cascade.h"
#include "prefill_kernels.h"

namespace {

using namespace pkv;

// ---------------------------------------------------------------------------------
// Chunked-prefill attention in fp32 arithmetic, for the shapes the 16-bit matrix-core kernel
// does not take: fp32 K/V (any supported head_dim) and 16-bit K/V at head_dim 16 (widened as
// they are staged). Same contract and arguments as paged_prefill_kernel (causal /
// non-causal, q_rows, rows, lse); keys whose slot lies outside the pool are left out.
//
// A workgroup of 8 waves takes 64 query rows (token, head of one KV head's group), so every
// K/V tile it stages serves 64 of them, and two halves of its waves take the two halves of
// the key tiles; wave w of a half holds rows 16 w .. 16 w + 15. Per tile of TK keys:
//   * S^T = K . Q^T with v_mfma_f32_16x16x4_f32 (fp32 products and sums). The four k-slots of
//     MFMA j of a 16-dim step are dims 16 i + 4 grp + j for lane group grp, so a lane reads
//     its K operands as one 16-byte row piece and holds Q in registers the same way. Lane
//     (row col, grp) gets keys 16 beta + 4 grp + r of query row col.
//   * fp32 online softmax per row in that layout.
//   * O^T += V^T . P^T with k-slot grp = key 16 beta + 4 grp + j: P's operand is the lane's
//     own p, V's one dword of row 4 grp + j.
// The next tile's K and V come from memory into registers while this one is used, its block
// ids one tile earlier still. LDS rows are padded by 16 bytes: K's 16-byte reads of 16 keys
// and V's dwords of 4 rows x 16 dims then fall on distinct banks. The halves' states merge
// through LDS at the end.
// Bound by the MFMAs where the rows fill the GPU, by the tiles' latency below that. us per call,
// before (16 tokens per workgroup, scores and P.V on the VALU, no load in flight under the
// arithmetic) and now, fp32: 8 x 300 tokens behind up to 1,500, 32 / 8 heads, hd 128: 3,154 ->
// 547; 3 x 100-300 behind up to 700, hd 128: 371 -> 83; 1,000 tokens, hd 64: 234 -> 62; 20
// behind 2,000: 54 -> 17; 2 x 100-300, hd 256: 144 -> 68; bf16 at hd 16, 4 x 100-400: 93 -> 16;
// with one query head per KV head, where 64 rows are 64 tokens: 64 tokens, 4 heads, hd 64 9.2 ->
// 8.9, 32 heads, hd 128 13.4 -> 12.5; 256 chunks of 4, 4 heads, hd 64 55 -> 42.
// Error against 64 bits on 3 chunks of 60-300 tokens, hd 64: 3.5e-7 -> 3.2e-7.
// ---------------------------------------------------------------------------------

template <int HD> struct F32Shape {
  static constexpr int TK = HD <= 64 ? 64 : (HD == 128 ? 32 : 16);  // keys per tile
  static constexpr int NB = TK / 16;    // 16-key blocks per tile
  static constexpr int LDW = HD + 4;    // floats per staged row
  static constexpr int DTL = HD / 16;   // 16-dim tiles of O^T
  static constexpr int BM = 64;         // query rows per workgroup
};

template <int DT, int HD>
__global__ void __launch_bounds__(512)
paged_prefill_f32_kernel(const PrefillArgs a) {
  using SH = F32Shape<HD>;
  constexpr int TK = SH::TK, NB = SH::NB, LDW = SH::LDW, DTL = SH::DTL, BM = SH::BM;
  constexpr int VEC = vec16<DT>();
  constexpr int CPR = HD / VEC;                       // 16-byte chunks per K/V row
  constexpr int NL = (TK * CPR + 255) / 256;          // chunks per thread of a half, K and V each
  using S = typename Elt<DT>::S;
  __shared__ __align__(16) float kv[2][2][TK][LDW];   // [half][K, V]
  __shared__ __align__(16) int live[2][TK];
  __shared__ float xml[4][2][kWave];                  // the merge's (m, l)

  const int tid = threadIdx.x, htid = tid & 255;
  const int half = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(htid / kWave);
  const int col = lane & 15, grp = lane >> 4;
  const unsigned item = blockIdx.y * gridDim.x + blockIdx.x;
  if (item >= (unsigned)(a.row_blocks * a.nkv * a.n_chunks)) return;  // of < 2^31 items
  const PrefillItem it = pick_item(a, (int)item);
  const int c = it.c, q0 = it.q0, n = it.n, kvh = it.kvh;
  const int qlen = it.q1 - q0, G = a.groups, nrows = qlen * G;
  const int rho0 = (a.row_blocks - 1 - it.rbi) * BM;
  if (qlen <= 0 || rho0 >= nrows) return;  // uniform per workgroup
  const int base_pos = n - qlen;

  // This lane's query row: its token, head, place in q and out, and its visible keys.
  const int rho = rho0 + 16 * wave + col;
  const int tok = min(rho, nrows - 1) / G, head = kvh * G + min(rho, nrows - 1) % G;
  int64_t qrow = q0 + tok;
  if (a.rows) qrow = token_row(a, qrow);
  else if (a.q_rows) qrow = a.q_rows[q0 + tok];
  const bool row_ok = rho < nrows && qrow >= 0;  // no query: nothing read or written
  const int64_t orow = a.rows ? qrow : q0 + tok;
  const int last_row = min(nrows - 1, rho0 + BM - 1);
  const int kend = a.causal ? min(n, base_pos + last_row / G + 1) : n;  // keys any row sees
  const int limit = a.causal ? min(n - 1, base_pos + tok) : n - 1;      // last key of this row
  // The last key of any row of this wave (its lane 15 holds the last row), -1 without rows: tiles
  // past it are only staged.
  const int wlimit = rho0 + 16 * wave < nrows ? __builtin_amdgcn_readlane(limit, 15) : -1;
  const int ntiles = kend > 0 ? (kend + TK - 1) / TK : 0;
  const int ns = (ntiles + 1) / 2;
  const int tbeg = half ? ns : 0, nt = half ? ntiles - ns : ns;

  // Staging: chunk e = htid + 256 i of a tile is 16 bytes of row e / CPR.
  const int32_t* trow = a.tables + (int64_t)c * a.table_stride;
  auto blk_of = [&](int p) { return a.bs_shift >= 0 ? p >> a.bs_shift : p / a.bs; };
  int bid[NL];
  auto load_ids = [&](int m) {  // block ids of local tile m's rows
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int p = (tbeg + m) * TK + (htid + 256 * i) / CPR;
      bid[i] = m < nt && p < kend ? trow[blk_of(p)] : -1;
    }
  };
  uint4 kr[NL], vr[NL];
  bool ok[NL];
  auto load_kv = [&](int m) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = htid + 256 * i;
      const int p = (tbeg + m) * TK + e / CPR;
      const int64_t sl = (int64_t)bid[i] * a.bs + (p - blk_of(p) * a.bs);
      ok[i] = (TK * CPR % 256 == 0 || e < TK * CPR) && m < nt && p < kend && bid[i] >= 0 &&
              sl < a.num_slots;
      kr[i] = vr[i] = make_uint4(0, 0, 0, 0);
      if (ok[i]) {
        const int64_t off = sl * a.kv_ss + (int64_t)kvh * a.kv_sh + (e % CPR) * VEC;
        kr[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const S*>(a.k) + off);
        vr[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const S*>(a.v) + off);
      }
    }
  };
  auto store_kv = [&]() {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = htid + 256 * i;
      if (TK * CPR % 256 != 0 && e >= TK * CPR) break;
      const int r = e / CPR, ch = e % CPR;
      float f[VEC];
      unpack16<DT>(kr[i], f);
      store_vec<PKV_F32, VEC>(&kv[half][0][r][ch * VEC], f);
      unpack16<DT>(vr[i], f);
      store_vec<PKV_F32, VEC>(&kv[half][1][r][ch * VEC], f);
      if (ch == 0) live[half][r] = ok[i];
    }
  };

  float m_run = -INFINITY, l_run = 0.f;  // of row col (l: this lane's keys)
  f32x4 ov[DTL];                         // O^T: dims 16 d + 4 grp + r of row col
#pragma unroll
  for (int d = 0; d < DTL; ++d) ov[d] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The first ids and the queries are one memory trip, the first tile the next.
  load_ids(0);
  S qx[HD / 16][4];
  {
    const S* qp = reinterpret_cast<const S*>(a.q) + (row_ok ? qrow : 0) * a.q_st +
                  (int64_t)head * a.q_sh + 4 * grp;
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) {
      if constexpr (DT == PKV_F32) *reinterpret_cast<float4*>(qx[i]) = *reinterpret_cast<const float4*>(qp + 16 * i);
      else *reinterpret_cast<uint2*>(qx[i]) = *reinterpret_cast<const uint2*>(qp + 16 * i);
    }
  }
  load_kv(0);
  load_ids(1);
  float qf[HD / 16][4];
#pragma unroll
  for (int i = 0; i < HD / 16; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) qf[i][j] = row_ok ? Elt<DT>::to_f32(qx[i][j]) * a.scale_log2 : 0.f;
  for (int m = 0; m < ns; ++m) {  // both halves pass every barrier
    __syncthreads();              // the previous tile's readers are done
    if (m < nt) store_kv();
    __syncthreads();
    if (m >= nt) continue;
    load_kv(m + 1);
    load_ids(m + 2);
    if ((tbeg + m) * TK > wlimit) continue;  // wave-uniform
    f32x4 sc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) sc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) {
      f32x4 kf[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b)
        kf[b] = *reinterpret_cast<const f32x4*>(&kv[half][0][16 * b + col][16 * i + 4 * grp]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][j], qf[i][j], sc[b], 0, 0, 0);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int4 lv = *reinterpret_cast<const int4*>(&live[half][16 * b + 4 * grp]);
      const int on[4] = {lv.x, lv.y, lv.z, lv.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kpos = (tbeg + m) * TK + 16 * b + 4 * grp + r;
        sc[b][r] = on[r] && kpos <= limit ? sc[b][r] : -INFINITY;
        mx = fmaxf(mx, sc[b][r]);
      }
    }
    const float mn = fmaxf(m_run, rows_max(mx));
    const float mref = mn == -INFINITY ? 0.f : mn;  // nothing visible yet: stay at 0
    const float alpha = __builtin_amdgcn_exp2f(m_run - mref);
    m_run = mn;
    l_run *= alpha;
#pragma unroll
    for (int d = 0; d < DTL; ++d) ov[d] *= alpha;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[b][r] = __builtin_amdgcn_exp2f(sc[b][r] - mref);
        l_run += sc[b][r];
      }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int d = 0; d < DTL; ++d)
          ov[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[half][1][16 * b + 4 * grp + j][16 * d + col],
                                                       sc[b][j], ov[d], 0, 0, 0);
  }
  float l_tot = rows_sum(l_run);

  // Merge the halves: half 1 leaves (m, l, O^T) per lane, half 0's same lane takes them.
  static_assert(4 * DTL * 4 * kWave <= 2 * 2 * TK * LDW, "the exchange fits the staged tiles");
  float* x = &kv[0][0][0][0] + wave * DTL * 4 * kWave + lane;
  __syncthreads();
  if (half) {
    xml[wave][0][lane] = m_run;
    xml[wave][1][lane] = l_tot;
#pragma unroll
    for (int d = 0; d < DTL; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) x[(4 * d + r) * kWave] = ov[d][r];
  }
  __syncthreads();
  if (half) return;
  const float mb = xml[wave][0][lane];
  const float mn = fmaxf(m_run, mb);
  const float mref = mn == -INFINITY ? 0.f : mn;  // both empty: weights 0
  const float sa = __builtin_amdgcn_exp2f(m_run - mref), sb = __builtin_amdgcn_exp2f(mb - mref);
  l_tot = l_tot * sa + xml[wave][1][lane] * sb;
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;  // nothing visible: 0
  const int64_t e0 = orow * a.out_st + (int64_t)head * a.out_sh;
  bool nan = false;
#pragma unroll
  for (int d = 0; d < DTL; ++d) {
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[r] = (ov[d][r] * sa + x[(4 * d + r) * kWave] * sb) * inv;
      nan = nan || o[r] != o[r];
    }
    if (!row_ok) continue;
    if (a.out_f32) store_vec<PKV_F32, 4>((float*)a.out + e0 + 16 * d + 4 * grp, o);
    else store_vec<DT, 4>((S*)a.out + e0 + 16 * d + 4 * grp, o);
  }
  if (a.lse && row_ok && grp == 0)
    a.lse[(int64_t)(q0 + tok) * a.nh + head] = l_tot > 0.f ? mn + __log2f(l_tot) : -INFINITY;

  // Keys past a row's last one enter its P.V with P = 0, and 0 x inf is NaN: a row that holds a NaN,
  // with an infinite or NaN V among those keys of its tiles, is computed again without them, by the
  // whole wave, 64 keys at a time. Rare (V is finite in practice), so it is only kept small.
  uint64_t redo = __ballot(nan && row_ok);
  redo = (redo | redo >> 16 | redo >> 32 | redo >> 48) & 0xFFFF;
  const int kused = min(kend, (wlimit / TK + 1) * TK);
  const S* kb = reinterpret_cast<const S*>(a.k) + (int64_t)kvh * a.kv_sh;
  const S* vb = reinterpret_cast<const S*>(a.v) + (int64_t)kvh * a.kv_sh;
  auto slot_of = [&](int p, int last) -> int64_t {  // key p's slot, -1 past `last` or the pool
    if (p > last) return -1;
    const int blk = blk_of(p), id = trow[blk];
    const int64_t sl = (int64_t)id * a.bs + (p - blk * a.bs);
    return id >= 0 && sl < a.num_slots ? sl : -1;
  };
  for (; redo; redo &= redo - 1) {
    const int row = __builtin_ctzll(redo);  // lane `row` holds it (and + 16, 32, 48)
    const int last = __builtin_amdgcn_readlane(limit, row);
    bool bad = false;
    for (int p = last + 1 + lane; p < kused; p += kWave) {
      const int64_t sl = slot_of(p, kused);
      for (int e = 0; sl >= 0 && e < HD; ++e) {
        const float v = Elt<DT>::to_f32(vb[sl * a.kv_ss + e]);
        bad = bad || !(fabsf(v) < INFINITY);
      }
    }
    if (!__ballot(bad)) continue;
    auto score = [&](int64_t sl) {
      float sc1 = 0.f;
#pragma unroll
      for (int i = 0; i < HD / 16; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float qv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(qf[i][j]), row + 16 * g));
            sc1 = __builtin_fmaf(qv, Elt<DT>::to_f32(kb[max(sl, (int64_t)0) * a.kv_ss + 16 * i + 4 * g + j]), sc1);
          }
        __builtin_amdgcn_sched_barrier(0);  // few loads in flight: few registers
      }
      return sl >= 0 ? sc1 : -INFINITY;
    };
    float mr = -INFINITY, lr = 0.f, acc[(HD + kWave - 1) / kWave] = {};
    for (int p = 0; p <= last; p += kWave) mr = fmaxf(mr, score(slot_of(p + lane, last)));
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) mr = fmaxf(mr, __shfl_xor(mr, off));
    for (int p = 0; p <= last; p += kWave) {
      const int64_t sl = slot_of(p + lane, last);
      const float pr = __builtin_amdgcn_exp2f(score(sl) - (mr == -INFINITY ? 0.f : mr));
      lr += pr;
      for (int t = 0; t < kWave && p + t <= last; ++t) {
        const int64_t st = __shfl(sl, t);
        const float pt = __shfl(pr, t);
#pragma unroll
        for (int k = 0; k < (HD + kWave - 1) / kWave; ++k)
          if (st >= 0 && lane + kWave * k < HD)
            acc[k] = __builtin_fmaf(pt, Elt<DT>::to_f32(vb[st * a.kv_ss + lane + kWave * k]), acc[k]);
      }
    }
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) lr += __shfl_xor(lr, off);
    const float invr = lr > 0.f ? 1.f / lr : 0.f;
    const int64_t er = __shfl(e0, row);
#pragma unroll
    for (int k = 0; k < (HD + kWave - 1) / kWave; ++k) {
      const int d = lane + kWave * k;
      if (d >= HD) break;
      if (a.out_f32) reinterpret_cast<float*>(a.out)[er + d] = acc[k] * invr;
      else reinterpret_cast<S*>(a.out)[er + d] = Elt<DT>::from_f32(acc[k] * invr);
    }
  }
}

// ---------------------------------------------------------------------------------
// Host-side dispatch.
// ---------------------------------------------------------------------------------

template <int DT, int HD, bool ROWS>
hipError_t launch_prefill_hd(PrefillArgs a, int64_t rows, hipStream_t st) {
  constexpr int BM = PrefillShape<HD>::BM;
  a.row_blocks = (int)((rows + BM - 1) / BM);
  const int64_t items = (int64_t)a.row_blocks * a.nkv * a.n_chunks;
  if (items > 0x7FFFFFFF) return hipErrorInvalidValue;
  const dim3 grid((unsigned)items), block(512);
  if constexpr (DT == PKV_BF16) {
    if (a.v16) {  // P.V in fp16 against the copy of V
      if (a.bs_shift >= 0)
        hipLaunchKernelGGL((paged_prefill_kernel<DT, HD, true, true, ROWS>), grid, block, 0, st, a);
      else
        hipLaunchKernelGGL((paged_prefill_kernel<DT, HD, false, true, ROWS>), grid, block, 0, st, a);
      return hipGetLastError();
    }
  }
  if (a.bs_shift >= 0)
    hipLaunchKernelGGL((paged_prefill_kernel<DT, HD, true, false, ROWS>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((paged_prefill_kernel<DT, HD, false, false, ROWS>), grid, block, 0, st, a);
  return hipGetLastError();
}

template <int DT, bool ROWS>
hipError_t launch_prefill(const PrefillArgs& a, int hd, int64_t rows, hipStream_t st) {
  switch (hd) {
    case 32: return launch_prefill_hd<DT, 32, ROWS>(a, rows, st);
    case 64: return launch_prefill_hd<DT, 64, ROWS>(a, rows, st);
    case 128: return launch_prefill_hd<DT, 128, ROWS>(a, rows, st);
    default: return launch_prefill_hd<DT, 256, ROWS>(a, rows, st);
  }
}

// The fp16 V copy ahead of a bf16 matrix-core prefill: one workgroup per (region tile of
// the widest possible context, KV head, chunk), KV head innermost; workgroups past their
// chunk's context leave.
hipError_t launch_v16(const PrefillArgs& a, int hd, hipStream_t st) {
  const int64_t tiles = ((int64_t)a.max_blocks * a.bs + kV16Rows - 1) / kV16Rows;
  const int64_t wgs = tiles * a.nkv * a.n_chunks;
  if (wgs < 1) return hipSuccess;
  if (wgs > 0x7FFFFFFF) return hipErrorInvalidValue;
  const dim3 grid((unsigned)wgs), block(kV16Threads);
  switch (hd) {
    case 32: hipLaunchKernelGGL((prefill_v16_kernel<32>), grid, block, 0, st, a); break;
    case 64: hipLaunchKernelGGL((prefill_v16_kernel<64>), grid, block, 0, st, a); break;
    case 128: hipLaunchKernelGGL((prefill_v16_kernel<128>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((prefill_v16_kernel<256>), grid, block, 0, st, a); break;
  }
  return hipGetLastError();
}

// The fp32 kernel: one workgroup per item (chunk, 64-row block, KV head). On two grid dimensions:
// a bound on the chunks' lengths that few of them reach makes many empty items, and HIP launches
// fewer than 2^32 threads along x.
template <int DT, int HD> hipError_t launch_f32_hd(PrefillArgs a, int64_t rows, hipStream_t st) {
  a.row_blocks = (int)((rows + F32Shape<HD>::BM - 1) / F32Shape<HD>::BM);
  const int64_t items = (int64_t)a.row_blocks * a.nkv * a.n_chunks;
  if (items > 0x7FFFFFFF) return hipErrorInvalidValue;
  const int64_t gx = items < (1 << 20) ? items : (1 << 20);
  // Head_dim 64 fits a CU twice. Up to two items per CU it runs once there (the LDS keeps a second
  // workgroup out): the heaviest items come first, and a second one beside them would end last (700
  // tokens, 32 / 8 heads, 352 items: 40.8 us against 46.2; 12 chunks of 3-599, 960: 452.6 against
  // 535 with one).
  const unsigned lds = HD == 64 && items < 512 ? 16384 : 0;
  hipLaunchKernelGGL((paged_prefill_f32_kernel<DT, HD>),
                     dim3((unsigned)gx, (unsigned)((items + gx - 1) / gx)), dim3(512), lds, st, a);
  return hipGetLastError();
}
hipError_t launch_f32(const PrefillArgs& a, int hd, int64_t rows, hipStream_t st) {
  switch (hd) {
    case 16: return launch_f32_hd<PKV_F32, 16>(a, rows, st);
    case 32: return launch_f32_hd<PKV_F32, 32>(a, rows, st);
    case 64: return launch_f32_hd<PKV_F32, 64>(a, rows, st);
    case 128: return launch_f32_hd<PKV_F32, 128>(a, rows, st);
    default: return launch_f32_hd<PKV_F32, 256>(a, rows, st);
  }
}

}  // namespace

namespace pkv {

int prefill_args(PrefillArgs* out_args, int64_t* rows_out, void* out, int out_dtype,
                 int64_t out_stride_tok, int64_t out_stride_h, const void* q,
                 int64_t q_stride_tok, int64_t q_stride_h, const void* k_cache,
                 const void* v_cache, int kv_dtype, int64_t kv_stride_slot,
                 int64_t kv_stride_head, int64_t num_slots, const int32_t* block_tables,
                 int64_t table_stride, int32_t max_blocks, const int32_t* context_lens,
                 const int32_t* cu_seqlens_q, int32_t n_chunks, int32_t max_query_len,
                 int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                 float scale, int32_t causal, const int32_t* q_rows, float* lse) {
  if (!valid_dtype(kv_dtype)) return PKV_E_DTYPE;
  if (!(out_dtype == kv_dtype || out_dtype == PKV_F32)) return PKV_E_DTYPE;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || block_size <= 0 ||
      max_blocks < 0 || n_chunks < 0 || n_chunks > 65535 || max_query_len < 0 ||
      num_kv_heads > 65535)
    return PKV_E_SHAPE;
  if (!(head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128 ||
        head_dim == 256))
    return PKV_E_SHAPE;
  if ((int64_t)max_blocks * block_size > (int64_t)1 << 30) return PKV_E_SHAPE;
  if (!(scale > 0.f && scale < INFINITY)) return PKV_E_SHAPE;  // softmax scale
  const int64_t rows = (int64_t)max_query_len * (num_heads / num_kv_heads);
  if (rows > (int64_t)1 << 30) return PKV_E_SHAPE;
  if (n_chunks == 0 || max_query_len == 0) return 1;
  if (!out || !q || !k_cache || !v_cache || !context_lens || !cu_seqlens_q ||
      (max_blocks > 0 && !block_tables))
    return PKV_E_NULL;
  const int vec = kv_dtype == PKV_F32 ? 4 : 8;
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out) ||
      q_stride_tok % vec || q_stride_h % vec || kv_stride_slot % vec || kv_stride_head % vec ||
      out_stride_tok % vec || out_stride_h % vec)
    return PKV_E_ALIGN;
  *rows_out = rows;
  PrefillArgs& a = *out_args;
  a.out = out;
  a.out_st = out_stride_tok;
  a.out_sh = out_stride_h;
  a.q = q;
  a.q_st = q_stride_tok;
  a.q_sh = q_stride_h;
  a.k = k_cache;
  a.v = v_cache;
  a.kv_ss = kv_stride_slot;
  a.kv_sh = kv_stride_head;
  a.num_slots = num_slots;
  a.tables = block_tables;
  a.table_stride = table_stride;
  a.max_blocks = max_blocks;
  a.ctx = context_lens;
  a.cu_q = cu_seqlens_q;
  a.n_chunks = n_chunks;
  a.nh = num_heads;
  a.nkv = num_kv_heads;
  a.groups = num_heads / num_kv_heads;
  a.bs = block_size;
  a.bs_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  a.row_blocks = 0;  // set per head_dim at launch
  a.causal = causal != 0;
  a.q_rows = q_rows;
  a.lse = lse;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.out_f32 = out_dtype == PKV_F32;
  a.v16 = nullptr;
  a.v16_k = nullptr;
  a.v16_kstride = 0;
  a.rows = nullptr;
  a.rows_len = a.num_rows = 0;
  return 0;
}

}  // namespace pkv

namespace {

// Launches for checked arguments: the 16-bit matrix-core kernel takes 16-bit K/V at head_dim
// 32..256 (a bf16 call with a.v16 set converts the chunks' V first), the fp32 kernel the rest.
int run_prefill(const PrefillArgs& a, int64_t rows, int kv_dtype, int head_dim, hipStream_t st) {
  if (kv_dtype == PKV_F32) return (int)launch_f32(a, head_dim, rows, st);
  if (head_dim == 16)
    return (int)(kv_dtype == PKV_BF16 ? launch_f32_hd<PKV_BF16, 16>(a, rows, st)
                                      : launch_f32_hd<PKV_F16, 16>(a, rows, st));
  if (kv_dtype == PKV_F16)
    return (int)(a.rows ? launch_prefill<PKV_F16, true>(a, head_dim, rows, st)
                        : launch_prefill<PKV_F16, false>(a, head_dim, rows, st));
  if (a.v16) {
    const hipError_t e = launch_v16(a, head_dim, st);
    if (e != hipSuccess) return (int)e;
  }
  return (int)(a.rows ? launch_prefill<PKV_BF16, true>(a, head_dim, rows, st)
                      : launch_prefill<PKV_BF16, false>(a, head_dim, rows, st));
}

// Whether a call of these shapes can use the fp16 V copy: bf16 at head_dim 32..256,
// tables of at most kV16MaxTokens tokens, slot indices within 31 bits.
bool v16_shapes(int kv_dtype, int head_dim, int32_t max_blocks, int32_t block_size,
                int64_t num_slots) {
  return kv_dtype == PKV_BF16 && head_dim >= 32 && head_dim <= 256 &&
         (int64_t)max_blocks * block_size <= kV16MaxTokens && num_slots <= 0x7FFFFFFF;
}

// Workspace of the fp16 V copy: the scale exponents (a row of kstride bytes per chunk and
// KV head, the area rounded up to 256 bytes), then every chunk's region at its widest.
struct V16Layout {
  int64_t kstride, k_bytes, total;
};
V16Layout v16_layout(int32_t head_dim, int32_t num_kv_heads, int32_t n_chunks,
                     int32_t max_blocks, int32_t block_size) {
  const int64_t pad = v16_pad(max_blocks * block_size);
  V16Layout l;
  l.kstride = (pad / kV16Rows + 3) / 4 * 4;
  l.k_bytes = ((int64_t)n_chunks * num_kv_heads * l.kstride + 255) / 256 * 256;
  l.total = l.k_bytes + (int64_t)n_chunks * pad * num_kv_heads * head_dim * 2;
  return l;
}

}  // namespace

extern "C" {

int pkv_paged_prefill(void* out, int out_dtype, int64_t out_stride_tok, int64_t out_stride_h,
                      const void* q, int64_t q_stride_tok, int64_t q_stride_h,
                      const void* k_cache, const void* v_cache, int kv_dtype,
                      int64_t kv_stride_slot, int64_t kv_stride_head, int64_t num_slots,
                      const int32_t* block_tables, int64_t table_stride, int32_t max_blocks,
                      const int32_t* context_lens, const int32_t* cu_seqlens_q, int32_t n_chunks,
                      int32_t max_query_len, int32_t num_heads, int32_t num_kv_heads,
                      int32_t head_dim, int32_t block_size, float scale, void* stream) {
  return pkv_paged_prefill_ex(out, out_dtype, out_stride_tok, out_stride_h, q, q_stride_tok,
                              q_stride_h, k_cache, v_cache, kv_dtype, kv_stride_slot,
                              kv_stride_head, num_slots, block_tables, table_stride, max_blocks,
                              context_lens, cu_seqlens_q, n_chunks, max_query_len, num_heads,
                              num_kv_heads, head_dim, block_size, scale, 1, nullptr, nullptr,
                              stream);
}

int pkv_paged_prefill_ex(void* out, int out_dtype, int64_t out_stride_tok, int64_t out_stride_h,
                         const void* q, int64_t q_stride_tok, int64_t q_stride_h,
                         const void* k_cache, const void* v_cache, int kv_dtype,
                         int64_t kv_stride_slot, int64_t kv_stride_head, int64_t num_slots,
                         const int32_t* block_tables, int64_t table_stride, int32_t max_blocks,
                         const int32_t* context_lens, const int32_t* cu_seqlens_q,
                         int32_t n_chunks, int32_t max_query_len, int32_t num_heads,
                         int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale,
                         int32_t causal, const int32_t* q_rows, float* lse, void* stream) {
  PrefillArgs a;
  int64_t rows = 0;
  const int bad = prefill_args(&a, &rows, out, out_dtype, out_stride_tok, out_stride_h, q,
                               q_stride_tok, q_stride_h, k_cache, v_cache, kv_dtype,
                               kv_stride_slot, kv_stride_head, num_slots, block_tables,
                               table_stride, max_blocks, context_lens, cu_seqlens_q, n_chunks,
                               max_query_len, num_heads, num_kv_heads, head_dim, block_size,
                               scale, causal, q_rows, lse);
  if (bad) return bad == 1 ? 0 : bad;
  return run_prefill(a, rows, kv_dtype, head_dim, (hipStream_t)stream);
}

int64_t pkv_prefill_workspace_bytes(int kv_dtype, int32_t head_dim, int32_t num_kv_heads,
                                    int32_t n_chunks, int32_t max_blocks, int32_t block_size) {
  if (!valid_dtype(kv_dtype)) return PKV_E_DTYPE;
  if (!(head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128 ||
        head_dim == 256) ||
      num_kv_heads <= 0 || n_chunks < 0 || max_blocks < 0 || block_size <= 0 ||
      (int64_t)max_blocks * block_size > (int64_t)1 << 30)
    return PKV_E_SHAPE;
  if (!v16_shapes(kv_dtype, head_dim, max_blocks, block_size, 0)) return 0;
  return v16_layout(head_dim, num_kv_heads, n_chunks, max_blocks, block_size).total;
}

int pkv_paged_prefill_ws(void* out, int out_dtype, int64_t out_stride_tok, int64_t out_stride_h,
                         const void* q, int64_t q_stride_tok, int64_t q_stride_h,
                         const void* k_cache, const void* v_cache, int kv_dtype,
                         int64_t kv_stride_slot, int64_t kv_stride_head, int64_t num_slots,
                         const int32_t* block_tables, int64_t table_stride, int32_t max_blocks,
                         const int32_t* context_lens, const int32_t* cu_seqlens_q,
                         int32_t n_chunks, int32_t max_query_len, int32_t num_heads,
                         int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale,
                         void* workspace, int64_t workspace_bytes, void* stream) {
  return pkv_paged_prefill_rows(out, out_dtype, out_stride_tok, out_stride_h, q, q_stride_tok,
                                q_stride_h, k_cache, v_cache, kv_dtype, kv_stride_slot,
                                kv_stride_head, num_slots, block_tables, table_stride, max_blocks,
                                context_lens, cu_seqlens_q, n_chunks, max_query_len, num_heads,
                                num_kv_heads, head_dim, block_size, scale, workspace,
                                workspace_bytes, nullptr, 0, 0, stream);
}

int pkv_paged_prefill_rows(void* out, int out_dtype, int64_t out_stride_tok, int64_t out_stride_h,
                           const void* q, int64_t q_stride_tok, int64_t q_stride_h,
                           const void* k_cache, const void* v_cache, int kv_dtype,
                           int64_t kv_stride_slot, int64_t kv_stride_head, int64_t num_slots,
                           const int32_t* block_tables, int64_t table_stride, int32_t max_blocks,
                           const int32_t* context_lens, const int32_t* cu_seqlens_q,
                           int32_t n_chunks, int32_t max_query_len, int32_t num_heads,
                           int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                           float scale, void* workspace, int64_t workspace_bytes,
                           const int64_t* rows, int64_t rows_len, int64_t num_rows,
                           void* stream) {
  if (rows_len < 0 || num_rows < 0 || num_rows > 0x7FFFFFFF) return PKV_E_SHAPE;
  PrefillArgs a;
  int64_t qrows = 0;  // query rows of the longest chunk for one KV head
  const int bad = prefill_args(&a, &qrows, out, out_dtype, out_stride_tok, out_stride_h, q,
                               q_stride_tok, q_stride_h, k_cache, v_cache, kv_dtype,
                               kv_stride_slot, kv_stride_head, num_slots, block_tables,
                               table_stride, max_blocks, context_lens, cu_seqlens_q, n_chunks,
                               max_query_len, num_heads, num_kv_heads, head_dim, block_size,
                               scale, 1, nullptr, nullptr);
  if (bad) return bad == 1 ? 0 : bad;
  if (rows) {
    a.rows = rows;
    a.rows_len = rows_len;
    a.num_rows = num_rows;
  }
  if (workspace_bytes < 0 || (workspace_bytes > 0 && !workspace)) return PKV_E_WORKSPACE;
  if (workspace && !aligned16(workspace)) return PKV_E_ALIGN;
  if (workspace && v16_shapes(kv_dtype, head_dim, max_blocks, block_size, num_slots)) {
    const V16Layout l = v16_layout(head_dim, num_kv_heads, n_chunks, max_blocks, block_size);
    if (workspace_bytes >= l.total) {
      a.v16_k = static_cast<const uint8_t*>(workspace);
      a.v16_kstride = (int32_t)l.kstride;
      a.v16 = static_cast<const char*>(workspace) + l.k_bytes;
    }
  }
  return run_prefill(a, qrows, kv_dtype, head_dim, (hipStream_t)stream);
}

}  // extern "C"
