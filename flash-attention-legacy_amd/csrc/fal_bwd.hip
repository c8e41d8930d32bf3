// Attention backward for gfx950.
//
// Math follows the reference backward (csrc/kernels/flash_attn_bwd.cu:76-107 for the
// preprocess, :425-647 for the KV-outer kernel): D = rowsum(dO * O);
// P = exp(S*scale - L); dV += P^T dO; dP = dO V^T; dS = P (dP - D) * scale;
// dK += dS^T Q; dQ = dS K; dK/dV of a KV head sum over all query heads of its GQA group.
// Every sum is in a fixed order, in fp32.
//
// Kernels:
// * FA2's split form (no atomics):
//   - bwd_dq_kernel (query-outer, runs first): a workgroup owns 128 query rows;
//     Q and dO stay in VGPRs, K/V tiles stream through LDS; it computes D for its
//     rows, P, dS and dQ = dS K, written once in fp16;
//   - bwd2_kernel (KV-outer): a workgroup owns 64 keys of one KV head and walks every
//     (query head of the group, query tile) that can see them; P and dS leave the
//     accumulators straight into the B operands of dV^T += dO^T P and
//     dK^T += Q^T dS (dO^T and Q^T from the Q/dO tiles via ds_read_b64_tr_b16);
//     dK/dV stay in registers until the end.
// * head_dim 128 and 256 (packed head_dim 128: of longer sequences) run both as
//   software-pipelined asm loops (bwd_kv_pipe_kernel, bwd_dq_kernel with PIPE).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "fal_kernels.h"
#include "fal_bwd_pipe.inc"
#include "fal_dq_pipe.inc"

namespace fal {

#ifndef FAL_PRESCALE_FP16
#define FAL_PRESCALE_FP16 0
#endif

// Scheduling fence between MFMA steps of the head_dim-128 kernel: keeps the compiler
// from hoisting every operand read of a phase at once (which overflows the 256-register
// budget of two waves per SIMD).
#ifndef FAL_BWD_FENCES
#define FAL_BWD_FENCES 1
#endif
#if FAL_BWD_FENCES
#define FAL_BWD_FENCE() __builtin_amdgcn_sched_barrier(0)
#else
#define FAL_BWD_FENCE() ((void)0)
#endif

// --------------------------------------------------------------------------
// KV-outer dK/dV kernel for head_dim 32, 64, 96 and 128 (the dQ kernel below runs first and
// stores D = rowsum(dO * O)).
//
// A 4-wave workgroup owns BN = 64 keys of one KV head: wave w takes keys
// 32*(w%2) .. +32 and query half w/2 of each 64-row query tile.  It walks every
// (query head of the GQA group, query tile) item; per item each wave forms
// S = Q K^T and dP = dO V^T for its 32 keys x 32 rows, P = exp2(S - L*log2e),
// dS = P (dP - D), then dV^T += dO^T P and dK^T += Q^T dS in registers (Q^T, dO^T
// read transposed from LDS, P and dS taken from the accumulators as B operands).
//   - The S accumulator starts at -L*log2e / c (c = scale*log2e) and the dP
//     accumulator at -D, so the MFMAs produce the exponent of P over c and dP - D
//     directly: one multiply and an exp2 per element.
//   - Operands of MFMA step t+1 are read before the MFMAs of step t.
//   - Only tiles that straddle the diagonal apply the causal mask.
//   - MFMA phases run at raised wave priority, so a SIMD's other wave fills their
//     gaps rather than delaying them.
// K/V tiles and the single-buffered Q/dO tile are staged in swizzled LDS by direct
// buffer loads (66 KB, two workgroups per CU).  For causal attention a workgroup
// takes key tiles kt and n-1-kt, so all workgroups do the same work.  The two query
// halves' dK/dV partials are summed in LDS, in a fixed order.
// --------------------------------------------------------------------------
#ifndef FAL_BWD2_NW
#define FAL_BWD2_NW 4   // waves per workgroup: 4 (64 keys, 2 workgroups per CU) or 8 (128 keys, double-buffered Q/dO)
#endif
template <class T, int D, bool CAUSAL>
__global__ void __launch_bounds__(FAL_BWD2_NW * 64) __attribute__((amdgpu_waves_per_eu(2, 8)))
bwd2_kernel(BwdParams p) {
  using V8 = vec8<T>;
  using V4 = vec4<T>;
  // K stays exact and scale*log2(e) is applied to the fp32 scores (one multiply).
  // FAL_PRESCALE_FP16 instead pre-multiplies an fp16 K tile in LDS
  // (rounded once) and starts the S accumulator at -L*log2e; that rounding costs
  // accuracy at large logits, so it is off.
  constexpr bool PRESCALE = FAL_PRESCALE_FP16 && std::is_same<T, half_t>::value;
  using TL = SwizzledTile<D>;
  constexpr int NW = FAL_BWD2_NW, BN = NW * 16, BMQ = 64;
  constexpr int NKG = NW / 2;             // key groups of 32 (x 2 query halves)
  constexpr bool DBUF = NW == 8;          // Q/dO double buffer (else one buffer, 2 WG/CU)
  constexpr int KS = D / 16;
  constexpr int DWB = D / 32;
  constexpr int CPR = TL::CPR;
  constexpr int KPART = BN * CPR * 8;     // elements of the K (or V) tile
  constexpr int QPART = BMQ * CPR * 8;    // elements of one Q (or dO) tile
  constexpr int KIPT = BN * CPR / (NW * 64);
  constexpr int QIPT = BMQ * CPR / (NW * 64);
  static_assert(BMQ * CPR % (NW * 64) == 0, "Q tile must split evenly over the waves");
  static_assert((DBUF ? 2 : 1) * 2 * QPART * 2 >= NKG * 32 * D * 4, "dK/dV reduction reuses the Q/dO buffers");

  __shared__ __attribute__((aligned(1024))) T ks_s[KPART];
  __shared__ __attribute__((aligned(1024))) T vs_s[KPART];
  __shared__ __attribute__((aligned(1024))) T qd_s[(DBUF ? 2 : 1) * 2 * QPART];   // [buffer][Q, dO]
  __shared__ float l_s[2][BMQ];
  __shared__ float d_s[2][BMQ];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int ws = __builtin_amdgcn_readfirstlane(w);
  const int kg = w % NKG;                 // key group
  const int qh = w / NKG;                 // query half
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  // ---- work item: up to two key tiles of one (batch, KV head) ----
  int b, hkv, q_off, k_off, nq, nk, kt_a, kt_b;
  if (p.cu_q) {
    // 1-D grid, KV head fastest: block i runs on XCD i % 8, so for a multiple of 8 KV
    // heads each XCD walks one KV head's items in list order (grouped by sequence) and
    // the query tiles they all read stay in its L2
    const int2 wk = p.work[blockIdx.x / p.Hkv];
    if (wk.x < 0) return;
    hkv = blockIdx.x % p.Hkv;
    b = 0;
    kt_a = wk.y;
    kt_b = -1;
    seg_bounds(p.cu_q, wk.x, p.total_q, q_off, nq);
    seg_bounds(p.cu_k, wk.x, p.total_k, k_off, nk);
  } else {
    const int total = gridDim.x;
    int id = blockIdx.x;
    if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    const int nitems = CAUSAL ? (p.n_ktiles + 1) / 2 : p.n_ktiles;
    const int it = id % nitems;
    const int bh = id / nitems;
    b = bh / p.Hkv;
    hkv = bh % p.Hkv;
    kt_a = it;
    kt_b = (CAUSAL && p.n_ktiles - 1 - it != it) ? p.n_ktiles - 1 - it : -1;
    q_off = 0;
    k_off = 0;
    nq = p.Nq;
    nk = p.Nk;
  }
  const int G = p.Hq / p.Hkv;
  const float c = p.scale_log2;
  const T* kbase = (const T*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh + (int64_t)k_off * p.k_ss;
  const T* vbase = (const T*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh + (int64_t)k_off * p.v_ss;

  // per-lane direct-load byte offsets from a tile's first row (instruction i of wave ws
  // fills chunks [(i*NW+ws)*64, +64)); one buffer resource per tile bounds the rows
  auto dl_offset = [&](int i, int64_t ss) {
    const int I = i * NW + ws;
    const int pch = I * 64 + lane;
    const int r = pch / CPR;
    return (r * (int)ss + TL::logical_chunk(r, pch % CPR) * 8) * 2;
  };
  // Fragment reads (row l32 of a 32-row block, chunk 2t+hh) and transposed reads
  // (rows hf*8 + hh*4 + i/4 of a 16-row step, 32-column block db) of the swizzled
  // tiles.  The swizzle is an XOR on the chunk index, so every address is a lane
  // base XOR a compile-time chunk offset; keeping only the bases saves registers.
  const int fbase = TL::offset(l32, hh);
  int trb[2];
  {
    const int i = lane & 15;
    const int rl = hh * 4 + (i >> 2);
    const int cl = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      trb[hf] = TL::offset(hf * 8 + rl, cl);
    }
  }
  const int tr_lo = 4 * (lane & 1);
  // (The XOR form needs a power-of-two row length in chunks; head_dim 96 has 12 and
  // takes the full offsets.)
  constexpr bool POW2 = (CPR & (CPR - 1)) == 0;
  auto faddr = [&](int t) { return POW2 ? (fbase ^ ((2 * t) << 3)) : TL::offset(l32, 2 * t + hh); };
  const int trl = hh * 4 + ((lane & 15) >> 2);
  const int trc = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
  auto tra = [&](int hf, int db) {
    return POW2 ? (trb[hf] ^ ((db * 4) << 3)) : TL::offset(hf * 8 + trl, db * 4 + trc);
  };
  // 8 k-slots for rows row0.. (multiple of 16) of a swizzled D-column tile, block db
  auto trk = [&](const T* base, int db, int row0) {
    const V4 lo = lds_tr(base + tra(0, db) + tr_lo + row0 * CPR * 8);
    const V4 hi = lds_tr(base + tra(1, db) + tr_lo + row0 * CPR * 8);
    return join8(lo, hi);
  };
  const int nqt = cdiv(nq, BMQ);

  for (int tile_i = 0; tile_i < 2; ++tile_i) {
    const int kt = tile_i == 0 ? kt_a : kt_b;
    if (kt < 0) break;
    const int n0 = kt * BN;
    if (n0 >= nk) continue;
    const int kw0 = n0 + kg * 32;
    const int key = kw0 + l32;

    __syncthreads();   // previous tile's readers of the LDS tiles are done
    {
      const int64_t left = (int64_t)max(nk - n0, 0);
      const __amdgpu_buffer_rsrc_t krs =
          make_rsrc(kbase + (int64_t)n0 * p.k_ss, (uint32_t)min(left * p.k_ss * 2, (int64_t)0x7fffffff));
      const __amdgpu_buffer_rsrc_t vrs =
          make_rsrc(vbase + (int64_t)n0 * p.v_ss, (uint32_t)min(left * p.v_ss * 2, (int64_t)0x7fffffff));
#pragma unroll
      for (int i = 0; i < KIPT; ++i) {
        const int I = i * NW + ws;
        buffer_to_lds16(krs, dl_offset(i, p.k_ss), ks_s + I * 64 * 8);
        buffer_to_lds16(vrs, dl_offset(i, p.v_ss), vs_s + I * 64 * 8);
      }
    }

    f32x16 dk_acc[DWB], dv_acc[DWB];
#pragma unroll
    for (int i = 0; i < DWB; ++i) {
      dk_acc[i] = zero_f16();
      dv_acc[i] = zero_f16();
    }
    // (FAL_PRESCALE_FP16 only) K tile *= scale*log2e, rounded once to fp16, so that S
    // comes out of the MFMAs in log2 units and its accumulator can start at -L*log2e
    wait_vmcnt0();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (PRESCALE ? KPART / (NW * 64 * 8) : 0); ++i) {
      T* ptr = ks_s + (i * NW * 64 + tid) * 8;
      V8 v = ld8(ptr);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (T)((float)v[e] * c);
      *reinterpret_cast<V8*>(ptr) = v;
    }
    const int qt0 = CAUSAL ? (n0 / BMQ) : 0;
    // (query head, query tile) items of this key tile, in one sequence so the Q/dO
    // double buffer alternates across head boundaries too: the fetch of item it+1
    // goes to the buffer item it-1 used, which every wave has finished with once it
    // passes item it's barrier.
    const int ntq = nqt > qt0 ? nqt - qt0 : 0;
    const int nitems_q = G * ntq;
    float lpre = 0.f, dpre = 0.f;
    // the next item to fetch, (query head, query tile), walked with counters: the
    // scalar unit has no divide
    int f_hq = hkv * G, f_qt = qt0;
    auto fetch = [&](int buf) {
      const int hq = f_hq;
      const int q0 = f_qt * BMQ;
      if (++f_qt == nqt) {
        f_qt = qt0;
        ++f_hq;
      }
      const T* qbase = (const T*)p.q + (int64_t)b * p.q_sb + (int64_t)hq * p.q_sh + (int64_t)(q_off + q0) * p.q_ss;
      const T* dobase =
          (const T*)p.dout + (int64_t)b * p.do_sb + (int64_t)hq * p.do_sh + (int64_t)(q_off + q0) * p.do_ss;
      const int64_t left = (int64_t)max(nq - q0, 0);
      const __amdgpu_buffer_rsrc_t qrs = make_rsrc(qbase, (uint32_t)min(left * p.q_ss * 2, (int64_t)0x7fffffff));
      const __amdgpu_buffer_rsrc_t dors = make_rsrc(dobase, (uint32_t)min(left * p.do_ss * 2, (int64_t)0x7fffffff));
#pragma unroll
      for (int i = 0; i < QIPT; ++i) {
        const int I = i * NW + ws;
        buffer_to_lds16(qrs, dl_offset(i, p.q_ss), qd_s + (buf * 2 + 0) * QPART + I * 64 * 8);
        buffer_to_lds16(dors, dl_offset(i, p.do_ss), qd_s + (buf * 2 + 1) * QPART + I * 64 * 8);
      }
      // -L*log2e and -D, the initial values of the S and dP accumulators; a row
      // past the end (or with no keys) gets -inf, so its P is 0
      if (tid < BMQ) {
        float nl = -INFINITY, nd = 0.f;
        if (q0 + tid < nq) {
          const int64_t o = (int64_t)b * p.l_sb + (int64_t)hq * p.l_sh + (int64_t)(q_off + q0 + tid) * p.l_ss;
          const float L = p.lse[o];
          nl = (L == -INFINITY) ? -INFINITY : -L * kLog2e;
          nd = -p.delta[o];
        }
        // without the K pre-scale the S accumulator starts at -L*log2e / c, so that
        // c * S is the exponent (a row with L = -inf keeps exponent -inf for either sign of c)
        if (!PRESCALE) nl /= c;
        lpre = nl;
        dpre = nd;
      }
    };

    if (nitems_q > 0) fetch(0);
    int c_qt = qt0;   // query tile of the current item
    int c_hq = 0;     // its query head within the group
    for (int item = 0; item < nitems_q; ++item) {
      {
        const int buf = DBUF ? (item & 1) : 0;
        const int q0 = c_qt * BMQ;
        const int cur_hq = c_hq;
        if (++c_qt == nqt) {
          c_qt = qt0;
          ++c_hq;
        }
        (void)cur_hq;
        wait_vmcnt0();
        if (tid < BMQ) {
          l_s[buf][tid] = lpre;
          d_s[buf][tid] = dpre;
        }
        __syncthreads();                  // barrier A: item in LDS; readers of item-1 done
        if (DBUF && item + 1 < nitems_q) fetch(buf ^ 1);
        const T* q_s = qd_s + (buf * 2 + 0) * QPART + qh * 32 * CPR * 8;
        const T* do_s = qd_s + (buf * 2 + 1) * QPART + qh * 32 * CPR * 8;
        const int qr0 = q0 + qh * 32;     // first query row of this wave's half
        if (!CAUSAL || qr0 + 31 >= kw0) {
          // S = Q K^T - L*log2e/c and dP = dO V^T - D
          f32x16 s, dp;
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) {
            const f32x4 ln = *reinterpret_cast<const f32x4*>(&l_s[buf][qh * 32 + g4 * 8 + hh * 4]);
            const f32x4 dn = *reinterpret_cast<const f32x4*>(&d_s[buf][qh * 32 + g4 * 8 + hh * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              s[g4 * 4 + e] = ln[e];
              dp[g4 * 4 + e] = dn[e];
            }
          }
          __builtin_amdgcn_s_setprio(1);
          // operands of step t+1 are read before the MFMAs of step t
          const T* kw_s = ks_s + kg * 32 * CPR * 8;
          const T* vw_s = vs_s + kg * 32 * CPR * 8;
          V8 oq = ld8(q_s + faddr(0)), ok = ld8(kw_s + faddr(0));
          V8 od = ld8(do_s + faddr(0)), ov = ld8(vw_s + faddr(0));
#pragma unroll
          for (int t = 0; t < KS; ++t) {
            V8 nq = oq, nk = ok, nd = od, nv = ov;   // (unused after the last step)
            if (t + 1 < KS) {
              const int fa = faddr(t + 1);
              nq = ld8(q_s + fa);
              nk = ld8(kw_s + fa);
              nd = ld8(do_s + fa);
              nv = ld8(vw_s + fa);
            }
            s = mfma32(oq, ok, s);
            dp = mfma32(od, ov, dp);
            FAL_BWD_FENCE();
            oq = nq; ok = nk; od = nd; ov = nv;
          }
          __builtin_amdgcn_s_setprio(0);
          // P = exp2(S) and dS = P dP; element i: query qr0 + (i/4)*8 + hh*4 + i%4, key `key`.
          // Query rows past the end carry L = +inf (P = 0), and keys past the end only
          // feed dK/dV rows that are never written, so the causal test is the only mask:
          // key > query  <=>  key - qr0 - hh*4 > (i/4)*8 + i%4, a constant per element.
          const int cthr = key - qr0 - hh * 4;
          auto grad = [&](auto masked) {
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int i = g4 * 4 + e;
                float pv = fast_exp2(PRESCALE ? s[i] : s[i] * c);
                if (decltype(masked)::value && cthr > g4 * 8 + e) pv = 0.f;
                s[i] = pv;
                dp[i] = pv * dp[i];
              }
            }
          };
          // only a tile that straddles the diagonal has keys past some of its queries
          if (CAUSAL && kw0 + 31 > qr0) grad(std::integral_constant<bool, true>{});
          else grad(std::integral_constant<bool, false>{});
          // dV^T += dO^T P ; dK^T += Q^T dS
          __builtin_amdgcn_s_setprio(1);
          {
            V8 pb[2], sb[2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
              pb[ks] = cvt8t<T>(s, ks);
              sb[ks] = cvt8t<T>(dp, ks);
            }
            V8 ao = trk(do_s, 0, 0), aq = trk(q_s, 0, 0);
#pragma unroll
            for (int st = 0; st < 2 * DWB; ++st) {
              const int ks = st / DWB, db = st % DWB;
              V8 no = ao, nq = aq;   // (unused after the last step)
              if (st + 1 < 2 * DWB) {
                no = trk(do_s, (st + 1) % DWB, (st + 1) / DWB * 16);
                nq = trk(q_s, (st + 1) % DWB, (st + 1) / DWB * 16);
              }
              dv_acc[db] = mfma32(ao, pb[ks], dv_acc[db]);
              dk_acc[db] = mfma32(aq, sb[ks], dk_acc[db]);
              FAL_BWD_FENCE();
              ao = no; aq = nq;
            }
          }
          __builtin_amdgcn_s_setprio(0);
        }
        if (!DBUF && item + 1 < nitems_q) {
          __syncthreads();                // barrier B: every wave is done with this item's tile
          fetch(0);
        }
      }
    }

    // ---- sum the two query halves' dK/dV and write this tile's rows ----
    __syncthreads();
    // The partner waves (same key group, same lane layout) meet in LDS: the second
    // query half stages its accumulators lane-contiguous, [kg][db][i][lane], and the
    // first adds them element by element (bank-conflict free, no transpose).
    float* red = reinterpret_cast<float*>(qd_s);
    auto reduce_write = [&](f32x16 (&acc)[DWB], T* row, float sc) {
      float* mine = red + (size_t)kg * DWB * 16 * 64 + lane;
      if (qh == 1) {
#pragma unroll
        for (int db = 0; db < DWB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) mine[(db * 16 + i) * 64] = acc[db][i];
      }
      __syncthreads();
      if (qh == 0 && key < nk) {
#pragma unroll
        for (int db = 0; db < DWB; ++db)
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) {
            const int col = db * 32 + g4 * 8 + hh * 4;
            V4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (T)((acc[db][g4 * 4 + e] + mine[(db * 16 + g4 * 4 + e) * 64]) * sc);
            *reinterpret_cast<V4*>(row + col) = h;
          }
      }
      __syncthreads();
    };
    const int64_t krow = (int64_t)(k_off + min(key, max(nk - 1, 0)));
    reduce_write(dk_acc, (T*)p.dk + (int64_t)b * p.dk_sb + (int64_t)hkv * p.dk_sh + krow * p.dk_ss, p.scale);
    reduce_write(dv_acc, (T*)p.dv + (int64_t)b * p.dv_sb + (int64_t)hkv * p.dv_sh + krow * p.dv_ss, 1.f);
  }
}


// --------------------------------------------------------------------------
// dK/dV kernel for head_dim 128 and 256 (bwd_kv_pipe_kernel): one wave per SIMD and
// a software-pipelined query-tile loop written as one inline-asm block (fal_bwd_pipe.inc,
// generated by gen_bwd_pipe.py).  A workgroup owns 128 keys of one KV head, each wave
// 32 keys whose K and V fragments stay in registers; the items (query head of the
// group, query tile of 64 rows, or of 32 for head_dim 256) stream through a 4-slot LDS ring
// of Q/dO tiles copied two items ahead.  Per item the S and dP accumulators start at
// -L*log2(e)/c and -D, read from the tile-major array `lsd` that bwd_dq_kernel writes, so
// P = exp2(c*S) and dS = P*dP.  The products of item i-1 (dV^T += dO^T P, dK^T += Q^T dS),
// the exponentials of item i and the products of item i+1 (S = Q K^T, dP = dO V^T)
// overlap inside the wave; no cross-wave sum is needed.  Same math as bwd2_kernel.
// Bound by the MFMA stream (64 per item; 916 TFLOP/s of products at head_dim 128).  Head dim
// 256 replaced the fp32-atomic form, which its atomics bound at 1 TB/s: both kernels of
// B2 x 16/8 heads x 2048 causal 957 -> 322 us, B2 x 16 x 4096 2147 -> 942 (non-causal
// 4053 -> 1709).
// --------------------------------------------------------------------------
constexpr int kPipeBN = 128;    // keys per workgroup
// dK/dV hand-off in LDS after the loop: per wave, dV then dK*scale, D/8 pieces of 512
// bytes each, kKvOStr apart so the row-wise reads of the epilogue spread over the banks
constexpr int kKvOStr = 528;
template <int D>
constexpr int pipe_bm() { return D == 256 ? 32 : 64; }   // query rows per item

enum KvForm { kKvWhole, kKvSplit, kKvPacked };
template <class T, int D, bool CAUSAL, KvForm FORM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
bwd_kv_pipe_kernel(BwdParams p) {
  constexpr bool SPLIT = FORM == kKvSplit, PACKED = FORM == kKvPacked;
  using V8 = vec8<T>;
  using TL = SwizzledTile<D>;
  constexpr int CPR = TL::CPR, KS = D / 16, kPipeBM = pipe_bm<D>();
  constexpr int kKvOPart = (D / 8) * kKvOStr, kKvOWave = 2 * kKvOPart;
  // 4 slots of (Q tile, dO tile) and 4 slots of Ls and Dn values; then the hand-off
  constexpr int kRing = 4 * 32768 + 4 * 512;
  __shared__ __attribute__((aligned(1024))) char smem[kRing > 4 * kKvOWave ? kRing : 4 * kKvOWave];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int ws = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  // work item: one or two 128-key tiles of one (batch, KV head); causal tiles are
  // paired (kt, n-1-kt) so every workgroup has the same number of items.  SPLIT (kv_run set):
  // one run of one key tile's items.  PACKED: one key tile of one sequence; KV heads fastest,
  // so for a multiple of 8 of them an XCD walks one head's list, grouped by sequence, and the
  // query tiles it reads stay in its L2.
  const int nkt = cdiv(p.Nk, kPipeBN);
  const int total = gridDim.x;
  int id = blockIdx.x, run = 0, kit, bh, q_off = 0, k_off = 0, nq = p.Nq, nk = p.Nk, lsd0 = 0;
  if (PACKED) {
    const int2 wk = p.work[id / p.Hkv];
    if (wk.x < 0) return;
    bh = id % p.Hkv;
    kit = wk.y;
    seg_bounds(p.cu_q, wk.x, p.total_q, q_off, nq);
    seg_bounds(p.cu_k, wk.x, p.total_k, k_off, nk);
    lsd0 = p.lsd_seq[wk.x] * (128 / kPipeBM);
  } else if (SPLIT) {
    // the first key tiles of all heads first (an XCD keeps whole heads when they divide by 8):
    // under a causal mask they have the most items
    int units = p.B * p.Hkv, u = 0;
    if ((units & 7) == 0) {
      units >>= 3;
      u = (id & 7) * units;
      id >>= 3;
    }
    kit = id / (units * p.kv_runs);
    id -= kit * units * p.kv_runs;
    bh = u + id / p.kv_runs;
    run = id % p.kv_runs;
  } else {
    if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    const int nk_items = CAUSAL ? (nkt + 1) / 2 : nkt;
    kit = id % nk_items;
    bh = id / nk_items;
  }
  const int slot = (bh * nkt + kit) * p.kv_runs + run;   // (SPLIT) of this workgroup's sums
  const int b = bh / p.Hkv, hkv = bh % p.Hkv;
  const int kt_b = (CAUSAL && FORM == kKvWhole && nkt - 1 - kit != kit) ? nkt - 1 - kit : -1;
  const int G = p.Hq / p.Hkv;
  const int nqt = cdiv(nq, kPipeBM);
  int run_len = 0, nruns = 1;
  if (SPLIT) {
    kv_runs_of(G * max(nqt - (CAUSAL ? kit * kPipeBN / kPipeBM : 0), 0), p.kv_run, &run_len, &nruns);
    // (uniform values: the pipelined loop takes them as scalar operands)
    run_len = __builtin_amdgcn_readfirstlane(run_len);
    nruns = __builtin_amdgcn_readfirstlane(nruns);
    if (run >= nruns) return;
  }

  typedef __attribute__((address_space(3))) char lds_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)((lds_t*)smem);
  // per-lane LDS addresses: fragment (row l32, chunk 2t+hh) and transposed reads
  // (rows hf*8 + hh*4 + i/4 of a 16-row step, 32-column block db) of a slot's tiles
  uint32_t p_qa[8], p_ta[2][4];
#pragma unroll
  for (int t = 0; t < 8; ++t) p_qa[t] = lds0 + 2 * TL::offset(l32, 2 * t + hh);
  {
    const int i = lane & 15;
    const int rl = hh * 4 + (i >> 2);
    const int cl = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int db = 0; db < 4; ++db) p_ta[hf][db] = lds0 + 2 * (TL::offset(hf * 8 + rl, db * 4 + cl) + 4 * (lane & 1));
  }
  const uint32_t p_la = lds0 + 131072 + 16 * hh;
  // copy offsets: load i of wave ws fills chunks [(4i + ws)*64, +64) of a tile
  int p_qo[4], p_do[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int pch = (i * 4 + ws) * 64 + lane;
    const int r = pch / CPR;
    const int cc = TL::logical_chunk(r, pch % CPR);
    p_qo[i] = (int)(r * p.q_ss + cc * 8) * 2;
    p_do[i] = (int)(r * p.do_ss + cc * 8) * 2;
  }
  const int p_lo4 = lane * 4, p_lo4b = 256 + lane * 4;
  const int p_lk = l32 - 4 * hh;
  const uint32_t p_olds = lds0 + ws * kKvOWave + lane * 8;
  const uint32_t p_lbase = __builtin_amdgcn_readfirstlane(lds0 + ws * 1024);
  const uint32_t p_ldbase = __builtin_amdgcn_readfirstlane(lds0 + 131072);
  const float p_c = p.scale_log2;
  const float p_negc = p.scale_log2 > 0.f ? -INFINITY : INFINITY;   // c * negc = -inf
  const float p_scale = p.scale;
  const uint32_t p_qrb = (uint32_t)(p.q_ss * 2), p_drb = (uint32_t)(p.do_ss * 2);
  // (head_dim 256) how far a tile's last row reaches past rows * stride
  const int p_qx = 2 * D - (int)p_qrb, p_dx = 2 * D - (int)p_drb;
  (void)p_qx, (void)p_dx;
  const int p_nq = nq, p_nqt = nqt;
  const int64_t qstep = (int64_t)kPipeBM * p.q_ss * 2, dstep = (int64_t)kPipeBM * p.do_ss * 2;
  // head_dim 256: an item's copies leave the resources 16 rows on
  const int64_t qhalf = D == 256 ? 16 * p.q_ss * 2 : 0, dhalf = D == 256 ? 16 * p.do_ss * 2 : 0;

  // K and V of this wave's 32 keys of key tile kt (B operands), buffer loads: keys past
  // the end read as zeros.  The second tile's are loaded right after the first tile's
  // loop, so their latency overlaps that tile's epilogue.
  V8 kreg[KS], vreg[KS];
  auto load_kv = [&](int kt) {
    // one resource per key tile: its rows inside the sequence, offsets from its first row
    const int n0 = kt * kPipeBN;
    const int64_t rows = min(max((int64_t)nk - n0, (int64_t)0), (int64_t)kPipeBN);
    const __amdgpu_buffer_rsrc_t krs =
        make_rsrc((const T*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh + (int64_t)(k_off + n0) * p.k_ss,
                  rows_bytes<D>(rows, p.k_ss));
    const __amdgpu_buffer_rsrc_t vrs =
        make_rsrc((const T*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh + (int64_t)(k_off + n0) * p.v_ss,
                  rows_bytes<D>(rows, p.v_ss));
    const int r = ws * 32 + l32;
    const int ko = (int)(r * p.k_ss * 2) + hh * 16, vo = (int)(r * p.v_ss * 2) + hh * 16;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      kreg[t] = __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(krs, ko + t * 32, 0, 0));
      vreg[t] = __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(vrs, vo + t * 32, 0, 0));
    }
  };
  // (head_dim 256: its 128 registers of K and V would be spilled around the epilogue, so
  // each tile loads its own first)
  constexpr bool AHEAD = D == 128;
  if (AHEAD) load_kv(kit);
  for (int tile_i = 0; tile_i < (FORM != kKvWhole || !CAUSAL ? 1 : 2); ++tile_i) {
    const int kt = tile_i == 0 ? kit : kt_b;
    if (kt < 0) break;
    const int n0 = kt * kPipeBN;
    const int kw0 = n0 + ws * 32;
    const int qt0 = CAUSAL ? n0 / kPipeBM : 0;
    const int ntq = max(nqt - qt0, 0);
    if (!AHEAD) load_kv(kt);
    // this workgroup's items: all of the key tile's, or a run of them from item i0 on
    const bool part = SPLIT && nruns > 1;
    const int i0 = part ? run * run_len : 0;
    const int nitems = part ? min(run_len, G * ntq - i0) : G * ntq;
    __syncthreads();   // the previous tile's epilogue readers are done with the LDS
    if (nitems > 0) {
      const int h0 = part ? __builtin_amdgcn_readfirstlane(i0 / ntq) : 0;
      const int hq0 = hkv * G + h0, q0 = qt0 + i0 - h0 * ntq;
      const uint64_t qb = (uint64_t)(uintptr_t)((const T*)p.q + (int64_t)b * p.q_sb + (int64_t)hq0 * p.q_sh +
                                                ((int64_t)q0 * kPipeBM + q_off) * p.q_ss);
      const uint64_t dob = (uint64_t)(uintptr_t)((const T*)p.dout + (int64_t)b * p.do_sb +
                                                 (int64_t)hq0 * p.do_sh + ((int64_t)q0 * kPipeBM + q_off) * p.do_ss);
      const uint64_t lb =
          (uint64_t)(uintptr_t)(p.lsd + (((int64_t)b * p.Hq + hq0) * p.lsd_tiles + lsd0 + q0) * 2 * kPipeBM);
      const int64_t qwrap = p.q_sh * 2 - (int64_t)(ntq - 1) * qstep - qhalf;
      const int64_t dwrap = p.do_sh * 2 - (int64_t)(ntq - 1) * dstep - dhalf;
      const uint32_t p_qb_lo = (uint32_t)qb, p_qb_hi = (uint32_t)(qb >> 32) & 0xffffu;
      const uint32_t p_db_lo = (uint32_t)dob, p_db_hi = (uint32_t)(dob >> 32) & 0xffffu;
      const uint32_t p_lb_lo = (uint32_t)lb, p_lb_hi = (uint32_t)(lb >> 32) & 0xffffu;
      const uint32_t p_qs_lo = (uint32_t)(qstep - qhalf), p_qs_hi = (uint32_t)((uint64_t)(qstep - qhalf) >> 32);
      const uint32_t p_qw_lo = (uint32_t)qwrap, p_qw_hi = (uint32_t)((uint64_t)qwrap >> 32);
      const uint32_t p_ds_lo = (uint32_t)(dstep - dhalf), p_ds_hi = (uint32_t)((uint64_t)(dstep - dhalf) >> 32);
      const uint32_t p_dw_lo = (uint32_t)dwrap, p_dw_hi = (uint32_t)((uint64_t)dwrap >> 32);
      // last tile of a head -> first of the next
      const uint64_t ldw = (uint64_t)(p.lsd_tiles - nqt + 1 + qt0) * 2 * kPipeBM * 4;
      const uint32_t p_ldw = (uint32_t)ldw, p_ldw_hi = (uint32_t)(ldw >> 32);   // (high word: head_dim 256)
      (void)p_ldw_hi;
      const int p_qt0 = qt0, p_qs0 = q0, p_nitems = nitems;
      const int p_part = SPLIT ? __builtin_amdgcn_readfirstlane(nruns - 1) : 0;
      // dV and dK sums of this wave's 32 keys
      const uint64_t po = SPLIT ? (uint64_t)(uintptr_t)(p.kv_part + ((int64_t)slot * 4 + ws) * 64 * D) : 0;
      const uint32_t p_po_lo = (uint32_t)po, p_po_hi = (uint32_t)(po >> 32) & 0xffffu;
      const int p_kw0 = CAUSAL ? kw0 : -(1 << 30);
      constexpr bool F16 = std::is_same<T, half_t>::value;
      if constexpr (D == 128 && F16)
        asm volatile(FAL_BWDP_ASM_F16 : FAL_BWDP_OUTS : FAL_BWDP_INS : FAL_BWDP_CLOBBERS);
      if constexpr (D == 128 && !F16)
        asm volatile(FAL_BWDP_ASM_BF16 : FAL_BWDP_OUTS : FAL_BWDP_INS : FAL_BWDP_CLOBBERS);
      if constexpr (D == 256 && F16)
        asm volatile(FAL_BWDP256_ASM_F16 : FAL_BWDP256_OUTS : FAL_BWDP256_INS : FAL_BWDP256_CLOBBERS);
      if constexpr (D == 256 && !F16)
        asm volatile(FAL_BWDP256_ASM_BF16 : FAL_BWDP256_OUTS : FAL_BWDP256_INS : FAL_BWDP256_CLOBBERS);
    }
    if (part) return;
    if (AHEAD && tile_i == 0 && kt_b >= 0) load_kv(kt_b);
    // dV then dK*scale of this wave's keys: piece pc = db*4 + g4 of lane (hh, l32) holds
    // columns 8*pc + hh*4 .. +3 of key kw0 + l32, at which*kKvOPart + pc*kKvOStr + lane*8.
    // Written back row-wise: each 16-byte store instruction covers whole rows.
    {
      constexpr int RPI = 64 / CPR;            // rows per store instruction
      const char* wb = smem + ws * kKvOWave;
      const int cch = lane % CPR;
      // buffer resources over this wave's keys inside the sequence: stores past the end
      // are dropped (no branch, no 64-bit address per store)
      const int nkw = max(min(nk - kw0, 32), 0);
      const __amdgpu_buffer_rsrc_t rs[2] = {
          make_rsrc((T*)p.dv + (int64_t)b * p.dv_sb + (int64_t)hkv * p.dv_sh + (int64_t)(k_off + kw0) * p.dv_ss,
                    (uint32_t)((int64_t)nkw * p.dv_ss * 2)),
          make_rsrc((T*)p.dk + (int64_t)b * p.dk_sb + (int64_t)hkv * p.dk_sh + (int64_t)(k_off + kw0) * p.dk_ss,
                    (uint32_t)((int64_t)nkw * p.dk_ss * 2))};
      const int vo[2] = {((lane / CPR) * (int)p.dv_ss + cch * 8) * 2, ((lane / CPR) * (int)p.dk_ss + cch * 8) * 2};
      const int rstep[2] = {(int)p.dv_ss * 2 * RPI, (int)p.dk_ss * 2 * RPI};   // rows of an instruction, in bytes
#pragma unroll
      for (int which = 0; which < 2; ++which)
#pragma unroll
        for (int j0 = 0; j0 < 32 / RPI; j0 += 8) {
          u32x4 x[8];
#pragma unroll
          for (int jj = 0; jj < 8; ++jj) {
            const int r = (j0 + jj) * RPI + lane / CPR;
            const char* src = wb + which * kKvOPart + cch * kKvOStr;
            const uint2 lo = *reinterpret_cast<const uint2*>(src + r * 8);
            const uint2 hi = *reinterpret_cast<const uint2*>(src + (32 + r) * 8);
            x[jj] = nitems > 0 ? u32x4{lo.x, lo.y, hi.x, hi.y} : u32x4{0u, 0u, 0u, 0u};
          }
#pragma unroll
          for (int jj = 0; jj < 8; ++jj) buffer_store16(rs[which], vo[which] + (j0 + jj) * rstep[which], x[jj]);
        }
    }
  }
}

// Adds the runs of a split key tile (BwdParams::kv_run), in run order, and writes its dV and
// dK * scale.  One workgroup per (batch, KV head, key tile, 32 keys, dV or dK); a run's sums
// are blocks of 1 KB, block db*4 + g4 holding columns db*32 + g4*8 + hh*4 .. +3 of key l32 at
// (hh*32 + l32) * 16.
template <class T, int D, bool CAUSAL>
__global__ void __launch_bounds__(256)
bwd_kv_reduce_kernel(BwdParams p) {
  constexpr int CPR = D / 8, RPI = 256 / CPR;
  const int which = blockIdx.x & 1, w = (blockIdx.x >> 1) & 3;
  const int nkt = cdiv(p.Nk, kPipeBN);
  const int tile = blockIdx.x >> 3, kt = tile % nkt, bh = tile / nkt;
  int len, runs;
  const int nqt = cdiv(p.Nq, pipe_bm<D>());
  kv_runs_of((p.Hq / p.Hkv) * max(nqt - (CAUSAL ? kt * kPipeBN / pipe_bm<D>() : 0), 0), p.kv_run, &len, &runs);
  if (runs < 2) return;      // written by its workgroup
  const int b = bh / p.Hkv, hkv = bh % p.Hkv;
  const int cch = threadIdx.x % CPR, key0 = kt * kPipeBN + w * 32;
  T* out = which ? (T*)p.dk + (int64_t)b * p.dk_sb + (int64_t)hkv * p.dk_sh
                 : (T*)p.dv + (int64_t)b * p.dv_sb + (int64_t)hkv * p.dv_sh;
  const int64_t ss = which ? p.dk_ss : p.dv_ss;
  const float sc = which ? p.scale : 1.f;
  const float* part = p.kv_part + ((int64_t)tile * p.kv_runs * 4 + w) * 64 * D + which * 32 * D + cch * 256;
#pragma unroll
  for (int r0 = 0; r0 < 32; r0 += RPI) {
    const int r = r0 + threadIdx.x / CPR;
    f32x4 lo = f32x4{0.f, 0.f, 0.f, 0.f}, hi = lo;
    for (int i = 0; i < runs; ++i) {
      const float* x = part + (int64_t)i * 4 * 64 * D + r * 4;
      lo += *reinterpret_cast<const f32x4*>(x);
      hi += *reinterpret_cast<const f32x4*>(x + 128);
    }
    if (key0 + r < p.Nk) {
      vec8<T> h;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        h[e] = (T)(lo[e] * sc);
        h[4 + e] = (T)(hi[e] * sc);
      }
      st_u4(out + (int64_t)(key0 + r) * ss + cch * 8, __builtin_bit_cast(u32x4, h));
    }
  }
}

// --------------------------------------------------------------------------
// Query-outer dQ kernel of every head dim (the KV-outer
// kernel above then produces only dK/dV).  Same structure as the forward kernel: a workgroup owns
// 32*NW query rows of one query head, each wave 32 rows whose Q and dO slices stay
// in VGPRs as the B operands of S^T = K Q^T and dP^T = V dO^T; K/V tiles of BN keys
// are staged in swizzled LDS by direct buffer loads, double-buffered.  Per tile:
// P^T = exp2(S^T * scale*log2e - L*log2e), dS^T = P^T (dP^T - D), and
// dQ^T += K^T dS^T with dS^T taken straight from the accumulator as the B operand
// and K^T read transposed from the K tile.  dQ is written once, in fp16, scaled:
// no fp32 accumulator and no atomics.
// --------------------------------------------------------------------------
#ifndef FAL_BWD_DQ_PAIR
#define FAL_BWD_DQ_PAIR 1
#endif
// pipelined dQ loop's hand-off in LDS: D/8 blocks of 1 KB per wave, kDqOStr apart (row-wise
// reads of the epilogue spread over the banks)
constexpr int kDqOStr = 1040;
#ifndef FAL_BWD_DQ_WPE
#define FAL_BWD_DQ_WPE 2
#endif
template <class T, int D, int NW, int BN, bool CAUSAL, bool PIPE = false>
__global__ void __launch_bounds__(NW * 64)
__attribute__((amdgpu_waves_per_eu(PIPE ? 1 : FAL_BWD_DQ_WPE, PIPE ? 1 : 8)))
bwd_dq_kernel(BwdParams p) {
  using V8 = vec8<T>;
  using V4 = vec4<T>;
  using TL = SwizzledTile<D>;
  constexpr int BM = NW * 32;
  constexpr int KS = D / 16;
  constexpr int NKB = BN / 32;
  constexpr int DB = D / 32;
  constexpr int CPR = TL::CPR;
  constexpr int PART = BN * CPR * 8;
  constexpr int IPT = BN * CPR / (NW * 64);
  static_assert(BN * CPR % (NW * 64) == 0, "tile must split evenly over the waves");
  // PIPE (head_dim 128 and 256): the key-tile loop is the software-pipelined asm
  // block of fal_dq_pipe.inc at one wave per SIMD, with a ring of 4 K/V tiles
  static_assert(!PIPE || ((D == 128 || D == 256) && NW == 4 && BN * D == 8192),
                "the pipelined loop is written for these shapes");
  constexpr int kDqOWave = (D / 8) * kDqOStr, kPipeBM = pipe_bm<D>();
  constexpr int NRING = (PIPE ? 4 : 2) * 2 * PART;

  __shared__ __attribute__((aligned(1024))) T smem[PIPE && 2 * kDqOWave > NRING ? 2 * kDqOWave : NRING];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  int b, hq, qt_a, qt_b = -1, q_off, k_off, nq, nk, lsd0 = 0;
  if (p.cu_q) {
    // 1-D grid: (work item, KV head) groups dealt round-robin to the 8 XCDs in list
    // order, the query heads of a group back to back on one XCD (they read the same
    // K/V); the grid is padded to a multiple of 8 groups
    const int g = p.Hq / p.Hkv;
    const int k8 = blockIdx.x >> 3;
    const int grp = (k8 / g) * 8 + (blockIdx.x & 7);
    const int item = grp / p.Hkv;
    if (item >= p.n_qitems) return;
    const int2 wk = p.qwork[item];
    if (wk.x < 0) return;
    hq = (grp % p.Hkv) * g + k8 % g;
    b = 0;
    qt_a = wk.y;
    seg_bounds(p.cu_q, wk.x, p.total_q, q_off, nq);
    seg_bounds(p.cu_k, wk.x, p.total_k, k_off, nk);
    if (PIPE && p.lsd) lsd0 = p.lsd_seq[wk.x] * (BM / kPipeBM);
  } else {
    // heads of one KV head and the query tiles of a head are dealt to one XCD together
    const int total = gridDim.x;
    int id = blockIdx.x;
    if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    // causal: a workgroup takes query tiles t and nqt-1-t, so all do equal work
    const int nqt = cdiv(p.Nq, BM);
    const int nitems = (CAUSAL && FAL_BWD_DQ_PAIR) ? (nqt + 1) / 2 : nqt;
    const int g = p.Hq / p.Hkv;
    const int hg = id % g;
    int rest = id / g;
    const int t = rest % nitems;
    rest /= nitems;
    qt_a = CAUSAL ? (nqt - 1 - t) : t;
    if (CAUSAL && FAL_BWD_DQ_PAIR && t != nqt - 1 - t) qt_b = t;
    b = rest / p.Hkv;
    hq = (rest % p.Hkv) * g + hg;
    q_off = 0;
    k_off = 0;
    nq = p.Nq;
    nk = p.Nk;
  }
  const int hkv = hq / (p.Hq / p.Hkv);
  for (int pass = 0; pass < 2; ++pass) {
  const int qt = pass == 0 ? qt_a : qt_b;
  if (qt < 0) break;
  if (pass) __syncthreads();   // the previous tile's LDS readers are done
  const int m0 = qt * BM;
  if (m0 >= nq) continue;

  const T* qbase = (const T*)p.q + (int64_t)b * p.q_sb + (int64_t)hq * p.q_sh + (int64_t)q_off * p.q_ss;
  const T* dobase = (const T*)p.dout + (int64_t)b * p.do_sb + (int64_t)hq * p.do_sh + (int64_t)q_off * p.do_ss;
  const T* kbase = (const T*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh + (int64_t)k_off * p.k_ss;
  const T* vbase = (const T*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh + (int64_t)k_off * p.v_ss;
  const int64_t lrow = (int64_t)b * p.l_sb + (int64_t)hq * p.l_sh + (int64_t)q_off * p.l_ss;

  const int kend = CAUSAL ? min(nk, m0 + BM) : nk;
  const int ntiles = cdiv(kend, BN);
  const int nfull = CAUSAL ? min(nk / BN, (m0 + 1) / BN) : nk / BN;

  const int ws = __builtin_amdgcn_readfirstlane(w);
  int kvo[IPT], vvo[IPT];
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const int I = i * NW + ws;
    const int pch = I * 64 + lane;
    const int r = pch / CPR;
    const int cc = TL::logical_chunk(r, pch % CPR);
    kvo[i] = (int)(r * p.k_ss + cc * 8) * 2;   // from the tile's first row
    vvo[i] = (int)(r * p.v_ss + cc * 8) * 2;
  }
  if (PIPE && ntiles > 0) {
    // the pipelined loop's first two K/V tiles (rows past the end read as zeros): on their
    // way while the rows of Q, dO and O arrive.  Head_dim 256 also keeps fewer values alive
    // across the loop (no scratch left when causal, 48 bytes before): backward of 1 x 16 x
    // 1024 causal 110.6 -> 105.1 us, packed 16 x up to 2048, 16/4 heads 640 -> 618;
    // head_dim 128 level.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t rows = min(max((int64_t)nk - j * BN, (int64_t)0), (int64_t)BN);
      const __amdgpu_buffer_rsrc_t krs = make_rsrc(kbase + (int64_t)j * BN * p.k_ss, rows_bytes<D>(rows, p.k_ss));
      const __amdgpu_buffer_rsrc_t vrs = make_rsrc(vbase + (int64_t)j * BN * p.v_ss, rows_bytes<D>(rows, p.v_ss));
      T* slot = smem + j * 2 * PART + ws * 512;
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        buffer_to_lds16(krs, kvo[i], slot + i * NW * 512);
        buffer_to_lds16(vrs, vvo[i], slot + PART + i * NW * 512);
      }
    }
  }

  // Q and dO slices of this wave (B operands: n = query row, k = head dim), the row's
  // log-sum-exp (log2 domain) and D = rowsum(dO * O).  The two lanes of a row hold one
  // half of the head dim each.  D is also stored for the dK/dV kernel, which runs after
  // this one.
  const int row = m0 + w * 32 + l32;
  V8 qreg[KS], doreg[KS];
  float lrow2 = INFINITY, dpart = 0.f;
  if (row < nq) {
    const T* orow = (const T*)p.o + (int64_t)b * p.o_sb + (int64_t)hq * p.o_sh + (int64_t)(q_off + row) * p.o_ss;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      qreg[t] = ld8(qbase + (int64_t)row * p.q_ss + t * 16 + hh * 8);
      doreg[t] = ld8(dobase + (int64_t)row * p.do_ss + t * 16 + hh * 8);
      const V8 ov = ld8(orow + t * 16 + hh * 8);
      dpart = dot8(doreg[t], ov, dpart);
    }
    const float L = p.lse[lrow + (int64_t)row * p.l_ss];
    lrow2 = (L == -INFINITY) ? INFINITY : L * kLog2e;
  } else {
#pragma unroll
    for (int t = 0; t < KS; ++t) qreg[t] = doreg[t] = zero8<T>();
  }
  const float drow = pair_sum(dpart);
  if (hh == 0 && row < nq) p.delta[lrow + (int64_t)row * p.l_ss] = drow;
  const float c = p.scale_log2;
  if (p.lsd && hh == 0) {
    // tile-major copy for bwd_kv_pipe_kernel, kPipeBM rows per tile: -L*log2(e)/c, then -D.
    // Rows past the end (up to the tile boundary) and rows without keys get the value
    // whose exponent c * x is -inf, and -D = 0.
    const int nt = cdiv(nq, kPipeBM);
    if (row < nt * kPipeBM) {
      float* t = p.lsd + (((int64_t)b * p.Hq + hq) * p.lsd_tiles + lsd0 + row / kPipeBM) * 2 * kPipeBM + row % kPipeBM;
      const bool live = row < nq && lrow2 != INFINITY;
      t[0] = live ? -lrow2 / c : (c > 0.f ? -INFINITY : INFINITY);
      t[kPipeBM] = row < nq ? -drow : 0.f;
    }
  }

  int kaddr[KS];   // fragment (row l32, chunk 2t+hh) of 32-key block 0
#pragma unroll
  for (int t = 0; t < KS; ++t) kaddr[t] = TL::offset(l32, 2 * t + hh);
  int taddr[2][DB];   // transposed reads: rows hf*8 + hh*4 + i/4 of each 16-key step
  {
    const int i = lane & 15;
    const int rl = hh * 4 + (i >> 2);
    const int cl = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int db = 0; db < DB; ++db) taddr[hf][db] = TL::offset(hf * 8 + rl, db * 4 + cl) + 4 * (lane & 1);
  }

  if constexpr (PIPE) {
    // The whole key-tile loop: dQ^T += K^T dS^T of tile j-1, the gradient of tile j and
    // S^T, dP^T of tile j+1 overlap inside the wave; the masking of the diagonal and
    // last tiles is done inside.  dQ^T comes back through this wave's LDS blocks.
    typedef __attribute__((address_space(3))) T lds_t;
    const uint32_t lds0 = (uint32_t)(uintptr_t)((lds_t*)smem);
    uint32_t p_ka[KS], p_ta[2][DB];
#pragma unroll
    for (int t = 0; t < KS; ++t) p_ka[t] = lds0 + 2 * kaddr[t];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int db = 0; db < DB; ++db) p_ta[hf][db] = lds0 + 2 * taddr[hf][db];
    const uint32_t p_lbase = __builtin_amdgcn_readfirstlane(lds0 + ws * 64 * 16);
    const uint32_t p_olds = lds0 + ws * kDqOWave + lane * 16;
    const int p_row = CAUSAL ? row : 0x3fffffff;
    const int p_hh4 = hh * 4;
    const float p_nl = -lrow2, p_dl = drow;
    const float p_c = c, p_negc = c > 0.f ? -INFINITY : INFINITY;   // c * negc = -inf
    const int64_t rows_left = max((int64_t)nk - 2 * BN, (int64_t)0);   // from the third tile on
    const uint64_t ka0 = (uint64_t)(uintptr_t)(kbase + (int64_t)2 * BN * p.k_ss);
    const uint64_t va0 = (uint64_t)(uintptr_t)(vbase + (int64_t)2 * BN * p.v_ss);
    const uint32_t pk_rs[4] = {(uint32_t)ka0, (uint32_t)(ka0 >> 32) & 0xffffu,
                               (uint32_t)min(rows_left * p.k_ss * 2, (int64_t)0x7fffffff), 0x00020000u};
    const uint32_t pv_rs[4] = {(uint32_t)va0, (uint32_t)(va0 >> 32) & 0xffffu,
                               (uint32_t)min(rows_left * p.v_ss * 2, (int64_t)0x7fffffff), 0x00020000u};
    const uint32_t p_ktb = (uint32_t)(BN * p.k_ss * 2), p_vtb = (uint32_t)(BN * p.v_ss * 2);
    const uint32_t p_krb = (uint32_t)(p.k_ss * 2), p_vrb = (uint32_t)(p.v_ss * 2);
    // (head_dim 256) how far a tile's last row reaches past rows * stride
    const int p_kx = 2 * D - (int)p_krb, p_vx = 2 * D - (int)p_vrb;
    (void)p_kx, (void)p_vx;
    const int p_rows = (int)min(rows_left, (int64_t)0x7fffffff);
    // tiles of this wave: [0, jl]; causal waves stop at their diagonal tile, waves whose
    // rows are all past the end have none
    const int wrow0 = m0 + ws * 32;
    int jl = CAUSAL ? min(ntiles - 1, (wrow0 + 31) / BN) : ntiles - 1;
    if (wrow0 >= nq) jl = -1;
    const int p_jl = __builtin_amdgcn_readfirstlane(jl);
    const int p_jend = ntiles, p_nk = nk;
    const int p_wrow = CAUSAL ? wrow0 : 0x3fffffff;
    if (ntiles > 0) {
      constexpr bool F16 = std::is_same<T, half_t>::value;
      if constexpr (D == 128 && F16)
        asm volatile(FAL_DQP_ASM_F16 : FAL_DQP_OUTS : FAL_DQP_INS : FAL_DQP_CLOBBERS);
      if constexpr (D == 128 && !F16)
        asm volatile(FAL_DQP_ASM_BF16 : FAL_DQP_OUTS : FAL_DQP_INS : FAL_DQP_CLOBBERS);
      if constexpr (D == 256 && F16)
        asm volatile(FAL_DQP256_ASM_F16 : FAL_DQP256_OUTS : FAL_DQP256_INS : FAL_DQP256_CLOBBERS);
      if constexpr (D == 256 && !F16)
        asm volatile(FAL_DQP256_ASM_BF16 : FAL_DQP256_OUTS : FAL_DQP256_INS : FAL_DQP256_CLOBBERS);
    }
    {
      // dQ^T block g = db*4 + g4 of lane (hh, l32) holds columns 8g + hh*4 .. +3 of row
      // m0 + ws*32 + l32 at ws*kDqOWave + lane*16 + g*kDqOStr; written back row-wise,
      // each 16-byte store instruction covering whole rows
      constexpr int RPI = 64 / CPR;            // rows per store instruction
      const char* wb = (const char*)smem + ws * kDqOWave;
      const int cch = lane % CPR;
      // a buffer resource over this wave's rows inside the sequence: stores past the end
      // are dropped (no branch, no 64-bit address per store)
      const int wr0 = m0 + ws * 32;
      const __amdgpu_buffer_rsrc_t dqrs =
          make_rsrc((T*)p.dq + (int64_t)b * p.dq_sb + (int64_t)hq * p.dq_sh + (int64_t)(q_off + wr0) * p.dq_ss,
                    (uint32_t)((int64_t)max(min(nq - wr0, 32), 0) * p.dq_ss * 2));
      const int dvo = ((lane / CPR) * (int)p.dq_ss + cch * 8) * 2;
#pragma unroll
      for (int j0 = 0; j0 < 32 / RPI; j0 += 8) {
        f32x4 a0[8], a1[8];
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
          const int r = (j0 + jj) * RPI + lane / CPR;
          a0[jj] = a1[jj] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (ntiles > 0) {
            a0[jj] = *reinterpret_cast<const f32x4*>(wb + r * 16 + cch * kDqOStr);
            a1[jj] = *reinterpret_cast<const f32x4*>(wb + (32 + r) * 16 + cch * kDqOStr);
          }
        }
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
          V8 h;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            h[e] = (T)(a0[jj][e] * p.scale);
            h[4 + e] = (T)(a1[jj][e] * p.scale);
          }
          buffer_store16(dqrs, dvo + (j0 + jj) * RPI * (int)p.dq_ss * 2, __builtin_bit_cast(u32x4, h));
        }
      }
    }
    continue;
  }

  auto load_tile = [&](int tile, int buf) {
    const int n0 = tile * BN;
    T* kdst = smem + buf * 2 * PART;
    T* vdst = kdst + PART;
    const int64_t left = (int64_t)max(nk - n0, 0);
    const __amdgpu_buffer_rsrc_t krs =
        make_rsrc(kbase + (int64_t)n0 * p.k_ss, (uint32_t)min(left * p.k_ss * 2, (int64_t)0x7fffffff));
    const __amdgpu_buffer_rsrc_t vrs =
        make_rsrc(vbase + (int64_t)n0 * p.v_ss, (uint32_t)min(left * p.v_ss * 2, (int64_t)0x7fffffff));
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const int I = i * NW + ws;
      buffer_to_lds16(krs, kvo[i], kdst + I * 64 * 8);
      buffer_to_lds16(vrs, vvo[i], vdst + I * 64 * 8);
    }
  };

  f32x16 dqacc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) dqacc[i] = zero_f16();

  auto tile_body = [&](auto masked, int j, int buf) {
    constexpr bool MASK = decltype(masked)::value;
    const int n0 = j * BN;
    const T* ks = smem + buf * 2 * PART;
    const T* vs = ks + PART;
    // S^T = K Q^T and dP^T = V dO^T; fragments read one k-step ahead of their MFMAs
    f32x16 sacc[NKB], pacc[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) sacc[kb] = pacc[kb] = zero_f16();
    V8 kf[2][NKB], vf[2][NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      kf[0][kb] = ld8(ks + kaddr[0] + kb * 32 * CPR * 8);
      vf[0][kb] = ld8(vs + kaddr[0] + kb * 32 * CPR * 8);
    }
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      if (t + 1 < KS) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          kf[(t + 1) & 1][kb] = ld8(ks + kaddr[t + 1] + kb * 32 * CPR * 8);
          vf[(t + 1) & 1][kb] = ld8(vs + kaddr[t + 1] + kb * 32 * CPR * 8);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * NKB, 0);
      }
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        sacc[kb] = mfma32(kf[t & 1][kb], qreg[t], sacc[kb]);
        pacc[kb] = mfma32(vf[t & 1][kb], doreg[t], pacc[kb]);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * NKB, 0);
    }
    // P^T and dS^T; element i: key n0 + kb*32 + (i/4)*8 + hh*4 + i%4, query `row`
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float pv = fast_exp2(fmaf(sacc[kb][i], c, -lrow2));
        if (MASK) {
          const int key = n0 + kb * 32 + (i >> 2) * 8 + hh * 4 + (i & 3);
          if (key >= nk || (CAUSAL && key > row)) pv = 0.f;
        }
        pacc[kb][i] = pv * (pacc[kb][i] - drow);
      }
    // dQ^T += K^T dS^T
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const V8 sb = cvt8t<T>(pacc[kb], t2);
        const int kofs = (kb * 2 + t2) * 16 * CPR * 8;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const V4 lo = lds_tr(ks + taddr[0][db] + kofs);
          const V4 hi = lds_tr(ks + taddr[1][db] + kofs);
          dqacc[db] = mfma32(join8(lo, hi), sb, dqacc[db]);
        }
      }
  };
  auto step = [&](auto masked, int j, int buf) {
    wait_vmcnt0();
    __syncthreads();
    if (j + 1 < ntiles) load_tile(j + 1, buf ^ 1);
    tile_body(masked, j, buf);
  };

  if (ntiles > 0) load_tile(0, 0);
  int j = 0;
  for (; j + 1 < nfull; j += 2) {
    step(std::false_type{}, j, 0);
    step(std::false_type{}, j + 1, 1);
  }
  if (j < nfull) {
    step(std::false_type{}, j, 0);
    ++j;
  }
  const int wrow_hi = m0 + w * 32 + 31;
  for (; j < ntiles; ++j) {
    wait_vmcnt0();
    __syncthreads();
    if (j + 1 < ntiles) load_tile(j + 1, (j + 1) & 1);
    if (!CAUSAL || j * BN <= wrow_hi) tile_body(std::true_type{}, j, j & 1);
  }

  if (row < nq) {
    T* dqrow = (T*)p.dq + (int64_t)b * p.dq_sb + (int64_t)hq * p.dq_sh + (int64_t)(q_off + row) * p.dq_ss;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        V4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (T)(dqacc[db][g4 * 4 + e] * p.scale);
        *reinterpret_cast<V4*>(dqrow + db * 32 + g4 * 8 + hh * 4) = h;
      }
  }
  }
}

// --------------------------------------------------------------------------
// Launchers
// --------------------------------------------------------------------------
// head dims of bwd2_kernel (256 has the pipelined kernels only)
constexpr bool split_d(int d) { return d == 32 || d == 64 || d == 96 || d == 128; }

int bwd_block_n(int d) {
  return split_d(d) ? FAL_BWD2_NW * 16 : kPipeBN;
}

bool bwd_pipe(int d) { return d == 128 || d == 256; }
// Packed head_dim 256 has no other form (its fp32-atomic one took 2.5 to 3.7 times as long: 16
// sequences of up to 2048, 16/4 heads, causal 1909 -> 639 us, 4 of 300, 8/1 heads 556 -> 150).
// At head_dim 128 bwd2_kernel keeps two workgroups of 64 keys per CU, which hide each other's
// start and end; the pipelined kernel's one of 128 keys needs sequences of many items and a
// grid of several rounds.  us, bwd2_kernel -> this, 32/8 heads causal: 16 x 1024 697 -> 648,
// 32 x 512 497 -> 452, 16 of 64 to 2048 564 -> 553 (not causal 905 -> 862); but 32 of 16 to 512
// 214 -> 229, and 4 of 64 to 2048 (264 key tiles) 130 -> 135.
bool bwd_varlen_pipe(int d, int64_t num_seqs, int64_t total_k, int64_t heads_kv, int ncu) {
  return d == 256 || (d == 128 && total_k >= 512 * num_seqs && total_k / kPipeBN * heads_kv >= 3 * (int64_t)ncu);
}
int bwd_pipe_bm(int d) { return d == 256 ? pipe_bm<256>() : pipe_bm<128>(); }

// A dK/dV workgroup takes about 1.85 us per item and 8 us besides, so a grid smaller than the
// GPU (few KV heads, short sequences) ends with its longest workgroup while CUs idle.
// Cutting the key tiles' items into runs fills them; it costs the fp32 sums, written and
// read again (about 2.5 and 4 TB/s), and the launch that adds them, about 6 us.  Tried are
// 2 to 16 runs for the longest key tile, up to two workgroups per CU (longest first, so the
// longest is followed by the shortest); the best is taken if it saves a tenth.
// Backward us before -> after: 1 x 32/8 heads x 1024 x 128 causal 159 -> 86, x 2048 272 -> 163,
// 1 x 28/4 x 333 x 128 83 -> 43, 1 x 16/4 x 4096 x 128 causal 500 -> 292,
// 1 x 8/1 x 777 x 256 causal 371 -> 114.
size_t bwd_kv_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nk, int d, int causal, int ncu,
                   size_t avail, int* run, int* runs) {
  *run = *runs = 0;
  constexpr int kMaxTiles = 256;
  if (!bwd_pipe(d) || ncu <= 0 || Nq <= 0 || Nk <= 0) return 0;
  const int64_t bm = bwd_pipe_bm(d), nqt = (Nq + bm - 1) / bm, nkt = (Nk + kPipeBN - 1) / kPipeBN;
  const int64_t units = B * Hkv, G = Hq / Hkv, grid0 = units * (causal ? (nkt + 1) / 2 : nkt);
  if (grid0 >= ncu || nkt > kMaxTiles || G * nqt > (1 << 20)) return 0;
  auto items = [&](int64_t kt) { return (int)(G * std::max<int64_t>(nqt - (causal ? kt * kPipeBN / bm : 0), 0)); };
  int64_t longest = items(0);
  if (causal)
    for (int64_t kt = 0; kt < (nkt + 1) / 2; ++kt)
      longest = std::max<int64_t>(longest, items(kt) + (nkt - 1 - kt != kt ? items(nkt - 1 - kt) : 0));
  const double slot = (double)kPipeBN * d * 2 * sizeof(float);
  double best = 0.9 * (8 + 1.85 * longest);
  size_t used = 0;
  for (int r = 2; r <= 16 && r <= items(0); ++r) {
    const int c = (items(0) + r - 1) / r;
    int len, most;
    kv_runs_of(items(0), c, &len, &most);
    std::pair<int, int64_t> lens[kMaxTiles];      // (items, workgroups) of each key tile
    int64_t grid = 0, split = 0;
    for (int64_t kt = 0; kt < nkt; ++kt) {
      int n;
      kv_runs_of(items(kt), c, &len, &n);
      lens[kt] = {len, n * units};
      grid += n * units;
      if (n > 1) split += n * units;
    }
    if (grid > 2 * (int64_t)ncu || most * nkt * units * slot > (double)avail) break;
    std::sort(lens, lens + nkt, [](const auto& a, const auto& b) { return a.first > b.first; });
    // the first ncu workgroups in order, the rest (shortest on the longest) behind them
    int64_t span = lens[0].first, i = 0, j = nkt - 1, ni = lens[0].second, nj = lens[nkt - 1].second;
    for (int64_t second = grid - ncu; second > 0;) {
      const int64_t n = std::min({ni, nj, second});
      span = std::max<int64_t>(span, (int64_t)lens[i].first + lens[j].first);
      second -= n;
      if ((ni -= n) == 0 && i + 1 < nkt) ni = lens[++i].second;
      if ((nj -= n) == 0 && j > 0) nj = lens[--j].second;
    }
    const double us = (grid > ncu ? 16 : 8) + 1.85 * span + 6 + slot * split * (1 / 2.5e6 + 1 / 4e6);
    if (us < best) {
      best = us;
      *run = c;
      *runs = most;
      used = (size_t)(most * nkt * units * slot);
    }
  }
  return used;
}

template <class T, int D>
static hipError_t launch_bwd_t(const BwdParams& p, int causal, dim3 grid, hipStream_t st) {
  if constexpr (D == 128 || D == 256) {
    if (p.cu_q && p.lsd) {
      if (causal)
        hipLaunchKernelGGL((bwd_kv_pipe_kernel<T, D, true, kKvPacked>), grid, dim3(256), 0, st, p);
      else
        hipLaunchKernelGGL((bwd_kv_pipe_kernel<T, D, false, kKvPacked>), grid, dim3(256), 0, st, p);
      return hipGetLastError();
    }
    if (p.lsd) {
      const int nkt = cdiv(p.Nk, kPipeBN), tiles = nkt * p.B * p.Hkv;
      grid.x = p.kv_run ? (unsigned)(tiles * p.kv_runs) : (unsigned)((causal ? (nkt + 1) / 2 : nkt) * p.B * p.Hkv);
      if (causal && !p.kv_run)
        hipLaunchKernelGGL((bwd_kv_pipe_kernel<T, D, true, kKvWhole>), grid, dim3(256), 0, st, p);
      else if (causal)
        hipLaunchKernelGGL((bwd_kv_pipe_kernel<T, D, true, kKvSplit>), grid, dim3(256), 0, st, p);
      else if (!p.kv_run)
        hipLaunchKernelGGL((bwd_kv_pipe_kernel<T, D, false, kKvWhole>), grid, dim3(256), 0, st, p);
      else
        hipLaunchKernelGGL((bwd_kv_pipe_kernel<T, D, false, kKvSplit>), grid, dim3(256), 0, st, p);
      if (p.kv_run) {
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (causal)
          hipLaunchKernelGGL((bwd_kv_reduce_kernel<T, D, true>), dim3((unsigned)tiles * 8), dim3(256), 0, st, p);
        else
          hipLaunchKernelGGL((bwd_kv_reduce_kernel<T, D, false>), dim3((unsigned)tiles * 8), dim3(256), 0, st, p);
      }
      return hipGetLastError();
    }
  }
  if constexpr (split_d(D)) {
    // batched causal: one workgroup per pair of key tiles
    if (!p.cu_q && causal) grid.x = (unsigned)((p.n_ktiles + 1) / 2) * p.B * p.Hkv;
    if (causal)
      hipLaunchKernelGGL((bwd2_kernel<T, D, true>), grid, dim3(FAL_BWD2_NW * 64), 0, st, p);
    else
      hipLaunchKernelGGL((bwd2_kernel<T, D, false>), grid, dim3(FAL_BWD2_NW * 64), 0, st, p);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}
template <int D>
static hipError_t launch_bwd_d(const BwdParams& p, int causal, dim3 grid, hipStream_t st) {
  return p.bf16 ? launch_bwd_t<bf16_t, D>(p, causal, grid, st) : launch_bwd_t<half_t, D>(p, causal, grid, st);
}

#ifndef FAL_BWD_DQ_BN
#define FAL_BWD_DQ_BN 64
#endif
constexpr int kDqNW = 4;

int bwd_dq_block_m(int d) {
  (void)d;
  return kDqNW * 32;
}

template <class T, int D>
static hipError_t launch_bwd_dq_t(const BwdParams& p, int causal, dim3 grid, hipStream_t st) {
  if (!p.cu_q && causal && FAL_BWD_DQ_PAIR)
    grid.x = (unsigned)((cdiv(p.Nq, kDqNW * 32) + 1) / 2) * p.B * p.Hq;
  if constexpr (D == 128 || D == 256) {
    if (p.lsd) {
      constexpr int BN = 8192 / D;
      if (causal)
        hipLaunchKernelGGL((bwd_dq_kernel<T, D, kDqNW, BN, true, true>), grid, dim3(kDqNW * 64), 0, st, p);
      else
        hipLaunchKernelGGL((bwd_dq_kernel<T, D, kDqNW, BN, false, true>), grid, dim3(kDqNW * 64), 0, st, p);
      return hipGetLastError();
    }
  }
  if constexpr (split_d(D)) {
    if (causal)
      hipLaunchKernelGGL((bwd_dq_kernel<T, D, kDqNW, FAL_BWD_DQ_BN, true>), grid, dim3(kDqNW * 64), 0, st, p);
    else
      hipLaunchKernelGGL((bwd_dq_kernel<T, D, kDqNW, FAL_BWD_DQ_BN, false>), grid, dim3(kDqNW * 64), 0, st, p);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}

template <int D>
static hipError_t launch_bwd_dq_d(const BwdParams& p, int causal, dim3 grid, hipStream_t st) {
  return p.bf16 ? launch_bwd_dq_t<bf16_t, D>(p, causal, grid, st) : launch_bwd_dq_t<half_t, D>(p, causal, grid, st);
}

hipError_t launch_bwd_dq(const BwdParams& p, int d, int causal, dim3 grid, hipStream_t st) {
  switch (d) {
    case 32: return launch_bwd_dq_d<32>(p, causal, grid, st);
    case 64: return launch_bwd_dq_d<64>(p, causal, grid, st);
    case 96: return launch_bwd_dq_d<96>(p, causal, grid, st);
    case 128: return launch_bwd_dq_d<128>(p, causal, grid, st);
    case 256: return launch_bwd_dq_d<256>(p, causal, grid, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_bwd(const BwdParams& p, int d, int causal, dim3 grid, hipStream_t st) {
  switch (d) {
    case 32: return launch_bwd_d<32>(p, causal, grid, st);
    case 64: return launch_bwd_d<64>(p, causal, grid, st);
    case 96: return launch_bwd_d<96>(p, causal, grid, st);
    case 128: return launch_bwd_d<128>(p, causal, grid, st);
    case 256: return launch_bwd_d<256>(p, causal, grid, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fal
