// gfx950 multi-query ("chunk") attention with fused query RoPE: S >= 2 query
// tokens per sequence that share one K/V stream (chunked prefill, speculative
// verification).  Same operator semantics as the decode kernel
// (src/kernels/paged_kernel_v21.cuh:17-374 and kernel_v21.cuh:17-367 in the
// reference repository, which re-read K/V once per query token: grid.y = W*S,
// paged_kernel_v21.cuh:391); here each K/V row is read once per block of 16
// tokens.
//
//  * Workgroup = eight waves, two per SIMD, on one (sequence, 16-token block,
//    KV head) and a contiguous range of its visible keys.  Wave w owns tokens
//    2w and 2w+1: two 16-row query tiles (16 heads each), so a K/V stage read
//    from LDS feeds 32 query rows per wave and 256 per workgroup.  Groups of at
//    most eight tokens split the keys instead (KS wave sets, stream_range).
//  * K/V pages stream through an 8-stage LDS ring filled by direct-to-LDS loads
//    (global_load_lds_dwordx4, non-temporal): 32 keys x 256 B of K and of V per
//    stage, one eighth issued by each wave, seven stages ahead of the one
//    computed, completion tracked with vmcnt and one workgroup barrier per stage.
//  * Per stage and tile: S^T = K Q^T on 16x16x32 MFMA (8 per tile), online
//    softmax per query row, O^T += V^T P^T (8 MFMA per tile, 16 for fp16: see
//    p_operands); the K and V^T operands of a stage are read from LDS once per
//    wave and kept in registers for both tiles.
//  * MFMA / VALU overlap inside the wave: the two tiles (A = 0, B = 1) run half
//    a stage apart.  Each half-stage issues one tile's MFMAs (S of B and P V of
//    B's previous stage, or P V of A and S of A's next stage) while the other
//    tile's softmax runs on the VALU, so the two use disjoint registers and the
//    matrix core has work during the softmax; the second wave on the SIMD fills
//    what one wave's dependences leave idle.
//  * Rows are causal-masked per token (key l visible iff l <= locations[f,w,s]).
//  * The balanced split / LSE merge is the decode kernel's (equal key chunks per
//    workgroup, fp32 partial slots, dv_merge_chunk).
#include "dv_chunk.h"

namespace dv {
namespace chunk {

// Workgroup barrier that is also a compiler memory and scheduling barrier: no
// LDS access or MFMA moves across it.
__device__ inline void wg_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// swizzled 16-byte piece positions inside a 256-byte key row
__device__ inline int swz_k(int key, int piece) { return piece ^ (key & 15); }
__device__ inline int swz_v(int key, int piece) { return piece ^ ((key & 7) << 1); }

// Issue this wave's eighth of stage `st` (keys [kb0, kb0+32) of the range): key
// rows 4*wave .. 4*wave+3 of K and of V, lane -> (row lane/16, 16-byte piece).
template <int KVM, bool P2>
__device__ inline void issue_stage(const DecodeParams& p, const Range& r, const int* pages, uint32_t ring,
                                   int st, int kb0) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int pos = lane & 15;
    const uint32_t sbase = ring + (uint32_t)(st % kStages) * kStageBytes;
    const int kl = wv * 4 + (lane >> 4);
    const int gk = swz_k(kl, pos), gv = swz_v(kl, pos);
    const uint32_t koff = (uint32_t)(wv * 4) * 256;
    const unsigned char* ka;
    const unsigned char* va;
    if (KVM == kKvPaged && P2 && r.pages_ok && kb0 + kStep <= r.b) {
        // interior stage of a range whose pages are all valid: no visibility
        // test and no zero rows
        const uint32_t pos_l = (uint32_t)(r.off + kb0 + kl);
        const int pg = pages[(pos_l >> p.bs_shift) - r.lp0];
        const uint32_t rowidx = (((uint32_t)pg << p.bs_shift) + (pos_l & ((1u << p.bs_shift) - 1u))) *
                                    (uint32_t)p.Hkv + (uint32_t)r.hkv;
        const unsigned long long boff = (unsigned long long)rowidx << 8;
        ka = r.k + boff + gk * 16;
        va = r.v + boff + gv * 16;
    } else {
        const long long row = row_of<KVM, P2>(p, r, pages, kb0 + kl);
        ka = row >= 0 ? r.k + row + gk * 16 : zrow + gk * 16;
        va = row >= 0 ? r.v + row + gv * 16 : zrow + gv * 16;
    }
    dma16(ka, __builtin_amdgcn_readfirstlane(sbase + koff));
    dma16(va, __builtin_amdgcn_readfirstlane(sbase + kKvBytes + koff));
}

struct Tile {
    f32x4 o[8];
    float m, l;
    // -max(m, -FLT_MAX), the exponent offset of every stage: kept beside m and
    // updated only where m changes (sm_raise), not recomputed per stage
    float nm;
};

// Query tiles of this wave's tokens tok0 .. tok0 + ntile - 1 of group gr for
// view f, staged through LDS (the K/V ring is idle between view ranges): raw
// q rows arrive by direct-to-LDS loads, each lane rotates whole (d, d + R/2)
// pairs in place (src/rope.cuh:18-51 and :67-114: first R/2 cos/sin entries of
// the token's full-width row, or its half-width varlen row; separately rounded
// fp32 products and sum, rounded to the storage type; dims >= R untouched),
// then lane (g, n) reads Q[n][c*32 + g*8 + 0..7] of every tile.  Wave-private
// LDS region: 8 KiB.  A row's 16-byte pieces are XOR-swizzled by the head, like
// the K rows: the rotation and the operand reads touch the same piece of 16 rows
// at once, which unswizzled rows (256 B apart) serialised 16-fold on one group of
// banks -- 4.5-6 us of every piece for the eight waves together, 1.6-2.5 with the swizzle.
// Key split: the KS waves of the same tokens share one region, each staging and
// rotating the heads [kg * 16 / KS, + 16 / KS); read_q_tiles follows a barrier.
template <int DT, int QM, int RM, int KS>
__device__ inline void stage_q_tiles(const DecodeParams& p, unsigned char* qreg, float* csreg, const Grp& gr,
                                     int tok0, int ntile, int kg, int f, int hkv) {
#pragma clang fp contract(off)
    using raw = typename Tr<DT>::raw;
    const int lane = opaque_tid() & 63;
    const uint32_t qbase = lds_addr(qreg);
    const int half = p.R >> 1;
    // every load is issued before the first is waited for: cos/sin of both tiles
    // on clamped, in-bounds indices (a branch around a load waits for it at once)
    float cv[kTiles], sv[kTiles];
    const bool rot = QM != kQPre && half > 0;
    if (rot && ntile > 0) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            const long long row = (long long)f * tok_axis<RM>(p) + gr.lin + tok0 + (t < ntile ? t : 0);
            const long long co = (QM == kQRotHalf ? row * half : row * p.R) + (lane < half ? lane : 0);
            cv[t] = p.cosv[co];
            sv[t] = p.sinv[co];
        }
    }
    for (int t = 0; t < ntile; ++t) {
#pragma unroll
        for (int i4 = 0; i4 < 4 / KS; ++i4) {
            const int i = kg * (4 / KS) + i4;
            const int hn = i * 4 + (lane >> 4);
            const int h = hkv * kGqa + hn;
            const raw* q = reinterpret_cast<const raw*>(p.q) + q_row<QM, RM>(p, gr, tok0 + t, h, f);
            dma16(q + ((lane & 15) ^ hn) * 8, __builtin_amdgcn_readfirstlane(qbase + (uint32_t)(t * 4096 + i * 1024)));
        }
    }
    if (rot && ntile > 0) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            csreg[t * 128 + lane] = cv[t];
            csreg[t * 128 + 64 + lane] = sv[t];
        }
    }
    wait_vmcnt<0>();
    compiler_fence();
    if (rot) {
        constexpr int kLanes = 4 * KS;  // lanes per head
        const int hn = kg * (kGqa / KS) + lane / kLanes, q = lane % kLanes;
        for (int t = 0; t < ntile; ++t) {
            raw* x = reinterpret_cast<raw*>(qreg + t * 4096 + hn * 256);
            auto at = [&](int e) { return x + ((e ^ (hn << 3)) & 127); };  // element e of the row
            const float* cs = csreg + t * 128;
            const float* sn = cs + 64;
            if ((half & 7) == 0) {
                for (int j0 = q * 8; j0 < half; j0 += 8 * kLanes) {
                    u32x4* pa4 = reinterpret_cast<u32x4*>(at(j0));
                    u32x4* pb4 = reinterpret_cast<u32x4*>(at(j0 + half));
                    const u32x4 a = *pa4, b = *pb4;
                    u32x4 ya, yb;
#pragma unroll
                    for (int e2 = 0; e2 < 4; ++e2) {
                        uint32_t wa = 0, wb = 0;
#pragma unroll
                        for (int hl = 0; hl < 2; ++hl) {
                            const int e = e2 * 2 + hl;
                            const float x1 = Tr<DT>::tof((raw)((a[e2] >> (16 * hl)) & 0xffffu));
                            const float x2 = Tr<DT>::tof((raw)((b[e2] >> (16 * hl)) & 0xffffu));
                            const float c = cs[j0 + e], s = sn[j0 + e];
                            const float a1 = x1 * c, b1 = x2 * s;
                            const float a2 = x2 * c, b2 = x1 * s;
                            wa |= (uint32_t)Tr<DT>::fromf(a1 - b1) << (16 * hl);
                            wb |= (uint32_t)Tr<DT>::fromf(a2 + b2) << (16 * hl);
                        }
                        ya[e2] = wa;
                        yb[e2] = wb;
                    }
                    *pa4 = ya;
                    *pb4 = yb;
                }
            } else {
                for (int j = q; j < half; j += kLanes) {
                    raw *xa = at(j), *xb = at(j + half);
                    const float x1 = Tr<DT>::tof(*xa), x2 = Tr<DT>::tof(*xb);
                    const float c = cs[j], s = sn[j];
                    const float a1 = x1 * c, b1 = x2 * s;
                    const float a2 = x2 * c, b2 = x1 * s;
                    *xa = Tr<DT>::fromf(a1 - b1);
                    *xb = Tr<DT>::fromf(a2 + b2);
                }
            }
        }
        compiler_fence();
    }
}

__device__ inline void read_q_tiles(const unsigned char* qreg, int ntile, u32x4 (&qB)[kTiles][4]) {
    const int lane = opaque_tid() & 63;
    const int g = lane >> 4, n = lane & 15;
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
        if (t < ntile)
#pragma unroll
            for (int cc = 0; cc < 4; ++cc)
                qB[t][cc] = *reinterpret_cast<const u32x4*>(qreg + t * 4096 + n * 256 + (((cc * 4 + g) ^ n) << 4));
    compiler_fence();
}

// frag / view_vis: the views' tensors and visible key counts (dv_stream.h)

// K operand of one stage (A of S^T = K Q^T): lo[cc] holds key n, hi[cc] key
// 16 + n, dims cc*32 + g*8 .. +8 (lane (g, n)).  The K swizzle only flips
// address bits 6-7 of the row base, so slice cc is at kbase ^ (64 cc).
struct KOp {
    u32x4 lo[4], hi[4];
};

// V^T operand of one stage (A of O^T += V^T P^T), 16-dim slice cc: block lane
// sl -> key g*4 + sl/4 (and + 16), dims cc*16 + (sl%4)*4 (transposing reads);
// the V swizzle only flips address bits 5-7, so slice cc is at vbase ^ (32 cc).
struct VOp {
    u32x4 v[8];
};

__device__ inline void read_k(const unsigned char* kt, KOp& k) {
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, n = lane & 15;
    const uint32_t kbase = lds_addr(kt) + (uint32_t)(n * 256 + 16 * (g ^ (n & 3)) + 64 * (n >> 2));
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
        k.lo[cc] = lds_read16_at(kbase ^ (uint32_t)(64 * cc));
        k.hi[cc] = lds_read16_at((kbase ^ (uint32_t)(64 * cc)) + 16 * 256);
    }
}

__device__ inline void read_v(const unsigned char* vt, VOp& v) {
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, sl = lane & 15;
    const int k0 = g * 4 + (sl >> 2);
    const uint32_t vbase =
        lds_addr(vt) + (uint32_t)(k0 * 256 + 16 * ((sl & 3) >> 1) + (sl & 1) * 8 + 32 * (k0 & 7));
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) {
        const u32x2 a0 = lds_read_tr16_at(vbase ^ (uint32_t)(32 * cc));
        const u32x2 a1 = lds_read_tr16_at((vbase ^ (uint32_t)(32 * cc)) + 16 * 256);
        v.v[cc] = u32x4{a0[0], a0[1], a1[0], a1[1]};
    }
}

// Scores of one tile: s0 keys 0-15, s1 keys 16-31 (S^T, lane (g, n): keys
// g*4 + i of head n).
template <int DT>
__device__ inline void qk_tile(const KOp& k, const u32x4 (&q)[4], f32x4& s0, f32x4& s1) {
    s0 = f32x4{0.f, 0.f, 0.f, 0.f};
    s1 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
        s0 = Tr<DT>::mma(k.lo[cc], q[cc], s0);
        s1 = Tr<DT>::mma(k.hi[cc], q[cc], s1);
    }
}

// O^T += V^T P^T for one tile.
template <int DT>
__device__ inline void pv_tile(const VOp& v, const POperand& pB, Tile& t) {
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) t.o[cc] = Tr<DT>::mma(v.v[cc], pB.hi, t.o[cc]);
    if constexpr (DT == kF16) {
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) t.o[cc] = Tr<DT>::mma(v.v[cc], pB.lo, t.o[cc]);
    }
}

// Visibility of the 32 keys of the stage starting at kb0: the range end, and,
// when some page of the sub-range is missing, page validity (a scalar branch
// around a few instructions; the loop itself is not duplicated).
template <int KVM, bool P2, int KS>
__device__ inline uint32_t stage_mask(const DecodeParams& p, const Range& r, const int* pages, int sbnd, int kb0) {
    const int nin = sbnd - kb0;
    uint32_t m = nin >= 32 ? 0xffffffffu : ((1u << (KS > 1 && nin < 0 ? 0 : nin)) - 1u);  // KS > 1: stages past the end
    if (!r.pages_ok) {
        const int lane = threadIdx.x & 63;
        const bool kv_ok = row_of<KVM, P2>(p, r, pages, kb0 + (lane & 31)) >= 0;
        m &= (uint32_t)ballot(kv_ok && lane < 32);
    }
    return m;
}

// Scores of invisible keys set to -inf (mask bit k = key k; lane (g, n) holds
// keys g*4 + i and 16 + g*4 + i): a partially visible stage only, so full
// stages spend nothing on masks.
__device__ inline void mask_scores(f32x4& s0, f32x4& s1, uint32_t mask) {
    const int lane = threadIdx.x & 63;
    const uint32_t mg = mask >> ((lane >> 4) * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        s0[i] = ((mg >> i) & 1u) ? s0[i] : -DV_INF;
        s1[i] = ((mg >> (16 + i)) & 1u) ? s1[i] : -DV_INF;
    }
}

// Online softmax of two tiles over one 32-key stage, in two straight-line
// parts so that the MFMAs of the other tile group can be interleaved with it
// (a branch ends the scheduling region).  Scores of invisible keys are -inf
// already (mask_scores).  Part 1: base-2 exponents against the running max
// (lane (g, n) holds keys g*4 + i and 16 + g*4 + i of head n); returns the
// lane's largest, so the caller can ask whether some row exceeds its max by
// more than kMaxSlack or has no max yet -- then sm_raise (rare) raises the max
// to the rows' maximum, rescales the accumulators and recomputes the
// exponents.  Part 2 (sm_finish): the probabilities, the row sums and the P^T
// operands.  Same arithmetic as softmax32 + p_operands.
__device__ inline float sm_exponents(const Tile& t, const f32x4& s0, const f32x4& s1, float l2, float (&pr)[8]) {
    // a row with no max yet (m = -inf) subtracts -FLT_MAX instead (t.nm): a
    // visible key's exponent is then huge (the row takes sm_raise) and an
    // invisible key's stays -inf, where -inf - (-inf) would be NaN
    const float nm = t.nm;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        pr[i] = __builtin_fmaf(s0[i], l2, nm);
        pr[4 + i] = __builtin_fmaf(s1[i], l2, nm);
    }
    // shaped for three-operand maxima: max3(max3(0,1,2), max3(3,4,5), max(6,7)),
    // four instructions where a balanced pairwise tree compiled to five
    const float a = fmaxf(fmaxf(pr[0], pr[1]), pr[2]), b = fmaxf(fmaxf(pr[3], pr[4]), pr[5]);
    return fmaxf(fmaxf(a, b), fmaxf(pr[6], pr[7]));
}

__device__ inline void sm_raise(Tile& t, const f32x4& s0, const f32x4& s1, float l2, float (&pr)[8]) {
    float sc[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sc[i] = s0[i] * l2;
        sc[4 + i] = s1[i] * l2;
    }
    const float mx = rows4_max(
        fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7]))));
    if (ballot(mx > t.m + kMaxSlack)) {
        const float mnew = fmaxf(t.m, mx);
        const float alpha = mnew == -DV_INF ? 1.0f : __builtin_amdgcn_exp2f(t.m - mnew);
        t.l *= alpha;
#pragma unroll
        for (int c = 0; c < 8; ++c) t.o[c] *= alpha;
        t.m = mnew;
        t.nm = -fmaxf(mnew, -3.402823466e38f);
    }
    const float mm = t.m == -DV_INF ? 0.0f : t.m;  // p = 0 while the row has no visible key
#pragma unroll
    for (int i = 0; i < 8; ++i) pr[i] = sc[i] - mm;
}

template <int DT>
__device__ inline POperand sm_finish(Tile& t, float (&pr)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) pr[i] = __builtin_amdgcn_exp2f(pr[i]);
    return p_operands<DT>(pr, t.l);
}

// Register tie: the values are complete at this point in program order (the
// compiler may not move their computation past it, e.g. across a workgroup
// barrier into the next half-stage).  Only the words the P V MFMAs read are
// tied: bf16 has no residual operand, and tying its (zero) lo made the
// compiler rebuild and copy four zero registers every half-stage.
template <int DT>
__device__ inline void settle(POperand& a) {
    asm volatile("" : "+v"(a.hi));
    if constexpr (DT == kF16) asm volatile("" : "+v"(a.lo));
}

// Key split KS (1, 2 or 4): a row group of few tokens leaves waves without
// tokens, and the arithmetic of 16 tokens per stage, not the loads, bound calls
// of 2 .. 8 tokens.  So KS sets of kWaves / KS waves hold the same tokens and
// take every KS-th stage: wave set kg computes stages kg, kg + KS, ... and one
// step of the loop covers KS stages of the ring; the sets' tiles are combined
// at the end of a piece (combine_split).  Steps in flight: the ring's steps
// less one for KS = 1, every step of the ring for KS > 1.  32 sequences of
// 4608 keys, 8 KV heads, bf16, same call without the split -> with it: 4 tokens
// 194 -> 117 us (5.2 TB/s), 8 tokens 194 -> 131 us.
template <int KS> constexpr int lead() { return KS == 1 ? kAhead : kStages / KS; }

// Keys [sa, sbnd) of the current view for this wave's two tiles (A = tile 0,
// B = tile 1): the stage loop.  Ring slot i % kStages holds stage i.  Per
// stage i, in every wave:
//   H1(i): MFMA O_B += V(i-1) P_B(i-1) beside A's exponents; MFMA S_B(i) =
//          K(i) Q_B^T and read V(i) beside A's probabilities
//   own loads of stage i+1 landed; workgroup barrier
//   H2(i): read K(i+1); MFMA O_A += V(i) P_A(i) beside B's exponents; MFMA
//          S_A(i+1) = K(i+1) Q_A^T and the loads of stage i+kAhead beside B's
//          probabilities
// so each wave's instruction stream alternates MFMAs of one tile with the
// softmax of the other, and the two waves of a SIMD issue both at once.  The
// loads of H2(i) refill slots of step i (KS > 1) or i-1 only: the barrier of
// step i is reached by every wave with its reads of every stage <= i complete
// (K(i) is read in H2(i-1), the V reads of H1 are waited for before the barrier).  One
// K and one V^T operand set live in registers: K(i+1) is read after the MFMAs
// of K(i) are issued, V(i) after those of V(i-1).  A's accumulators are
// rescaled in H1 and written by MFMAs issued in H2 (and B's the other way
// round), so a softmax never touches registers an MFMA of the same half-stage
// writes; mfma_settle before each softmax covers the MFMA -> VALU dependence
// across the half-stage boundary.  Invisible keys get -inf scores only on a
// partially visible stage (a uniform branch between the interleaved regions).
template <int DT, int KVM, bool P2, int KS>
__device__ inline void stream_range(const DecodeParams& p, const Range& r, const int* pages, unsigned char* smem,
                                    int sa, int sbnd, int kg, const int (&vis_t)[kTiles],
                                    const u32x4 (&qB)[kTiles][4], Tile (&tl)[kTiles]) {
    constexpr int kLead = lead<KS>();
    constexpr int kDma = kDmaPerStage * KS;  // loads per wave and step
    const uint32_t ring = lds_addr(smem);
    const int nsteps = (sbnd - sa + KS * kStep - 1) / (KS * kStep);
    const float l2 = p.l2scale;
    // prologue: steps 0 .. kLead-1.  Past the end, KS = 1 issues rows of zeros; with a
    // key split such steps issue nothing (a view of 30 keys would pay for the
    // addresses of 12 stages and not 4: 2 tokens, 4 sequences, six such views, 8 KV
    // heads 112.5 -> 99.6 us; six of 150 keys 55 -> 50.5).
#pragma unroll
    for (int s = 0; s < kLead; ++s) {
        if (KS > 1 && s >= nsteps) break;
#pragma unroll
        for (int st = s * KS; st < (s + 1) * KS; ++st) issue_stage<KVM, P2>(p, r, pages, ring, st, sa + st * kStep);
    }
    if (KS == 1 || nsteps >= kLead) wait_vmcnt<kDma * (kLead - 1)>();  // own share of step 0 landed
    else wait_vmcnt<0>();
    wg_barrier();

    KOp kop;
    VOp vop;
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) vop.v[cc] = u32x4{0u, 0u, 0u, 0u};  // the first P V adds 0 * 0
    f32x4 sa0, sa1, sb0, sb1;
    POperand pa = {}, pb = {};
    read_k(smem + kg * kStageBytes, kop);
    qk_tile<DT>(kop, qB[0], sa0, sa1);

    for (int i = 0; i < nsteps; ++i) {
        const int st = i * KS + kg;  // this wave's stage of the step
        const int kb0 = sa + st * kStep;
        const unsigned char* slot = smem + (st % kStages) * kStageBytes;
        const uint32_t okm = stage_mask<KVM, P2, KS>(p, r, pages, sbnd, kb0);
        const uint32_t mka = okm & token_mask(vis_t[0], kb0), mkb = okm & token_mask(vis_t[1], kb0);
        float pr[8];
        // ---- H1(i)
        if (mka != 0xffffffffu) mask_scores(sa0, sa1, mka);
        mfma_settle(tl[0].o);
        pv_tile<DT>(vop, pb, tl[1]);  // zero at i = 0
        float lmx = sm_exponents(tl[0], sa0, sa1, l2, pr);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
        }
        if (ballot(lmx > kMaxSlack)) sm_raise(tl[0], sa0, sa1, l2, pr);
        qk_tile<DT>(kop, qB[1], sb0, sb1);
        read_v(slot + kKvBytes, vop);
        pa = sm_finish<DT>(tl[0], pr);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
        }
        settle<DT>(pa);
        lds_wait();
        // own share of step i + 1 landed (with a key split, fewer loads follow it near
        // the end)
        if (KS == 1 || i + kLead <= nsteps) wait_vmcnt<kDma * (kLead - 2)>();
        else wait_vmcnt<0>();
        wg_barrier();
        if (KS > 1 && i + kLead < nsteps) {
            // the loads of step i + kLead, into the slots of step i (free since the
            // barrier): at once, as no later step is in flight when KS = 4; one
            // stage at a time, the addresses of all do not fit the registers
#pragma unroll 1
            for (int q = (i + kLead) * KS; q < (i + kLead + 1) * KS; ++q)
                issue_stage<KVM, P2>(p, r, pages, ring, q, sa + q * kStep);
        }
        // ---- H2(i) (past the end, step i + 1 holds rows of zeros or what the slot
        // held before: K and S_A of the next stage need no branch, the last ones go
        // unused)
        read_k(smem + ((st + KS) % kStages) * kStageBytes, kop);
        if (mkb != 0xffffffffu) mask_scores(sb0, sb1, mkb);
        mfma_settle(tl[1].o);
        pv_tile<DT>(vop, pa, tl[0]);
        lmx = sm_exponents(tl[1], sb0, sb1, l2, pr);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
        }
        if (ballot(lmx > kMaxSlack)) sm_raise(tl[1], sb0, sb1, l2, pr);
        qk_tile<DT>(kop, qB[0], sa0, sa1);
        pb = sm_finish<DT>(tl[1], pr);
        // the loads of stage i + kAhead (into the slot of stage i - 1, free since
        // the barrier), their address arithmetic beside the MFMAs
        if constexpr (KS == 1) issue_stage<KVM, P2>(p, r, pages, ring, i + kLead, sa + (i + kLead) * kStep);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
        }
        settle<DT>(pb);
    }
    // P V of B's last stage
    mfma_settle(tl[1].o);
    pv_tile<DT>(vop, pb, tl[1]);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) mfma_settle(tl[t].o);
    wait_vmcnt<0>();  // the trailing zero-row stages land before the ring is reused
    __syncthreads();
}

// Key split: wave kg's tiles of the same tokens (kg = 0 .. KS - 1, waves
// kg * kWaves/KS + tp) combined into those of kg = 0, through the idle ring:
// lane by lane, O and the lane's row sum scaled to the common maximum (fp32).
template <int KS>
__device__ inline void combine_split(unsigned char* smem, int wv, int kg, int ntile, Tile (&tl)[kTiles]) {
    constexpr int kPairs = kWaves / KS;  // waves per key subset
    constexpr int kRec = 10 * 1024;      // per (wave, tile): 8 x 1 KiB of O, then m and l
    static_assert((kWaves - kPairs) * kTiles * kRec <= kRingBytes + kPageCap * 4, "LDS of the combination");
    const int lane = threadIdx.x & 63;
    auto rec = [&](int k, int t) {  // record of tile t of the wave with subset k >= 1 of these tokens
        return smem + (((k - 1) * kPairs + wv % kPairs) * kTiles + t) * kRec;
    };
    if (kg > 0) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            if (t >= ntile) continue;
            unsigned char* b = rec(kg, t);
#pragma unroll
            for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4*>(b + c * 1024 + lane * 16) = tl[t].o[c];
            float* ml = reinterpret_cast<float*>(b + 8 * 1024);
            ml[lane] = tl[t].m;
            ml[64 + lane] = tl[t].l;
        }
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            if (t >= ntile) continue;
            float mk[KS], M = tl[t].m;
#pragma unroll
            for (int k = 1; k < KS; ++k) {
                mk[k] = reinterpret_cast<const float*>(rec(k, t) + 8 * 1024)[lane];
                M = fmaxf(M, mk[k]);
            }
            // an empty subset (-inf) -> weight 0; with no maximum in any, all have
            // it, and what a NaN left in a subset's sums stays
            const float Mf = M == -DV_INF ? 0.0f : M;
            const float s0 = __builtin_amdgcn_exp2f(tl[t].m - Mf);
            tl[t].l *= s0;
#pragma unroll
            for (int c = 0; c < 8; ++c) tl[t].o[c] *= s0;
#pragma unroll
            for (int k = 1; k < KS; ++k) {
                const float sk = __builtin_amdgcn_exp2f(mk[k] - Mf);
                tl[t].l += sk * reinterpret_cast<const float*>(rec(k, t) + 8 * 1024)[64 + lane];
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    tl[t].o[c] += sk * *reinterpret_cast<const f32x4*>(rec(k, t) + c * 1024 + lane * 16);
            }
            tl[t].m = M;
        }
    }
    __syncthreads();  // the records are read before the ring is filled again
}

// One workgroup: keys [v0, v1) of row group rg for KV head hkv.
template <int DT, int QM, int KVM, bool P2, int RM, int KS>
__device__ void chunk_piece(const DecodeParams& p, unsigned char* smem, int* pages, int rg, int hkv, long long v0,
                            long long v1, bool final_out, int slot, long long row_keys) {
    const int wv = uniform((int)(threadIdx.x >> 6));
    Grp gr = group_of<RM>(p, rg);
    gr.w = uniform(gr.w);
    gr.s0 = uniform(gr.s0);
    gr.lin = uniform(gr.lin);
    gr.ntok = uniform(gr.ntok);
    const int w = gr.w;
    const int kg = KS == 1 ? 0 : wv / (kWaves / KS);                // this wave's key subset
    const int tok0 = (KS == 1 ? wv : wv % (kWaves / KS)) * kTiles;  // and first token of the group
    const int ntile = gr.ntok - tok0 < kTiles ? (gr.ntok - tok0 > 0 ? gr.ntok - tok0 : 0) : kTiles;

    Tile tl[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
#pragma unroll
        for (int c = 0; c < 8; ++c) tl[t].o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        tl[t].m = -DV_INF;
        tl[t].l = 0.0f;
        tl[t].nm = 3.402823466e38f;
    }

    long long P = 0, off = 0;
    for (int f = 0; f < p.F && P < v1; ++f) {
        // visible keys per tile (wave-uniform: the stage masks and their branches
        // stay scalar), and of this view for the block: the union over its tokens,
        // for a single view the row's keys, counted by the schedule
        int vis_t[kTiles];
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            const int last = gr.ntok - 1;  // >= 0: a group without tokens has no piece
            const int v = uniform(view_vis<KVM>(p, f, loc_of<RM>(p, f, gr, tok0 + t < last ? tok0 + t : last)));
            vis_t[t] = t < ntile ? v : 0;
        }
        const int vis_blk = p.F == 1 ? (int)row_keys : uniform(group_view_vis<KVM, RM>(p, f, gr));
        const long long a = v0 > P ? v0 : P;
        const long long bnd = v1 < P + vis_blk ? v1 : P + vis_blk;
        if (a < bnd) {
            const int la = (int)(a - P), lb = (int)(bnd - P);
            Range r;
            r.w = w;
            r.hkv = hkv;
            if (KVM == kKvPaged) {
                r.k = reinterpret_cast<const unsigned char*>(p.kc);
                r.v = reinterpret_cast<const unsigned char*>(p.vc);
                r.off = off;
                r.bstride = 0;
                r.L = 0;
            } else {
                const FragDesc& fd = frag<KVM>(p, f);
                r.k = reinterpret_cast<const unsigned char*>(fd.k);
                r.v = reinterpret_cast<const unsigned char*>(fd.v);
                r.off = 0;
                r.bstride = fd.bstride * w;
                r.L = fd.L;
            }
            u32x4 qB[kTiles][4] = {};
            // sub-ranges whose page ids fit the LDS page cache
            const int span = KVM == kKvPaged ? (p.bs_shift >= 0 ? (kPageCap - 2) << p.bs_shift : (kPageCap - 2) * p.bs)
                                             : (1 << 30);
            for (int sa = la; sa < lb; sa += span) {
                const int sbnd = sa + span < lb ? sa + span : lb;
                r.b = sbnd;
                int pg[kPageIt];
                uint32_t lpl = 0;
                r.lp0 = 0;
                if (KVM == kKvPaged) {
                    lpl = logical_page(p, off + sbnd - 1);
                    r.lp0 = logical_page(p, off + sa);
                    fetch_pages(p, p.bt + (long long)w * p.maxB, r.lp0, lpl, pg);
                }
                // the ring is idle here (previous range drained): stage the query tiles
                // in it, their round trip beside the page ids'
                unsigned char* qreg = smem + (KS == 1 ? wv : wv % (kWaves / KS)) * (kTiles * 4096);
                if (sa == la) {
                    stage_q_tiles<DT, QM, RM, KS>(
                        p, qreg, reinterpret_cast<float*>(smem + kWaves * kTiles * 4096 + wv * kTiles * 512), gr, tok0,
                        ntile, kg, f, hkv);
                    if (KS == 1) read_q_tiles(qreg, ntile, qB);
                }
                // every position and page of the sub-range is valid; the page ids are
                // written and the query tiles read (KS > 1: staged)
                bool ok = true;
                if (KVM == kKvPaged)
                    ok = store_pages(p, pages, r.lp0, lpl, pg) && position_in_range(off + sa) &&
                         position_in_range(off + sbnd - 1);
                r.pages_ok = __syncthreads_and(ok) != 0;
                if (KS > 1 && sa == la) {
                    read_q_tiles(qreg, ntile, qB);
                    __syncthreads();
                }
                stream_range<DT, KVM, P2, KS>(p, r, pages, smem, sa, sbnd, kg, vis_t, qB, tl);
            }
        }
        P += vis_blk;
        off += p.fl[f];
    }

    if constexpr (KS > 1) combine_split<KS>(smem, wv, kg, ntile, tl);

    // epilogue: per tile, normalise and write the output or a partial slot
    {
    const int lane = opaque_tid() & 63;
    const int g = lane >> 4, n = lane & 15;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        if (t >= ntile || kg > 0) continue;
        const float lt = rows4_sum(tl[t].l);
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        const int h = hkv * kGqa + n;
        if (final_out) {
            using raw = typename Tr<DT>::raw;
            raw* o = reinterpret_cast<raw*>(p.out) + out_row<RM>(p, gr, tok0 + t, h);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const u32x2 pk = {pack2<DT>(tl[t].o[c][0] * inv, tl[t].o[c][1] * inv),
                                  pack2<DT>(tl[t].o[c][2] * inv, tl[t].o[c][3] * inv)};
                *reinterpret_cast<u32x2*>(o + c * 16 + g * 4) = pk;
            }
        } else {
            const int tb = tok0 + t;  // token within the block
            store_partial<DT>(p.part + (long long)slot * p.slot_floats, kTokBlk * kGqa, tb * kGqa + n, g, tl[t].o,
                              inv, lt > 0.0f ? tl[t].m + log2f(lt) : -DV_INF);
        }
    }
    }
}

// P2: paged with a power-of-two block_size (shift and mask instead of a
// division in the stage loop's row addressing).  KS = 0 (varlen): the key split of
// each row group follows from its own tokens, four wave sets up to kFewTok tokens
// and none above (decodes beside prompt chunks, and the last tokens of a chunk).
template <int DT, int QM, int KVM, bool P2, int RM, int KS>
__global__ __launch_bounds__(kThreads) void dv_chunk(const DecodeParams p) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    // the ring starts at a 256-byte aligned LDS address (the XOR addressing of
    // the MFMA operands needs address bits 0-7 of every tile base clear)
    unsigned char* smem = smem_raw + ((256u - (lds_addr(smem_raw) & 255u)) & 255u);
    int* pages = reinterpret_cast<int*>(smem + kRingBytes);
    long long* s_scan = reinterpret_cast<long long*>(smem + kRingBytes + kPageCap * 4);  // kWaves entries
    long long* s_pref = s_scan + kWaves;
    const int NHG = p.Hkv;  // one KV head per workgroup

    if constexpr (KS > 0) {
        run_schedule(p, NHG, s_pref, s_scan, [&](int rg) { return group_visible<KVM, RM>(p, rg); },
                     [&](int rg, int hg, long long v0, long long v1, bool fin, int slot, long long rk) {
                         chunk_piece<DT, QM, KVM, P2, RM, KS>(p, smem, pages, uniform(rg), uniform(hg), uniform(v0),
                                                              uniform(v1), uniform((int)fin) != 0, uniform(slot),
                                                              uniform(rk));
                     });
    } else {
        // the schedule counts units, even for a group without the split, odd with it
        // (one unit more than its keys': both sides of a cut round down alike, so it
        // never makes a key); a split needs a positive scale (key_split)
        run_schedule<false, 1, kLongKeyCost>(
                     p, NHG, s_pref, s_scan,
                     [&](int rg) {
                         const long long v = group_visible<KVM, RM>(p, rg);
                         const bool split = p.l2scale > 0.0f && group_of<RM>(p, rg).ntok <= kFewTok &&
                                            v >= (long long)kSplitVarlenKeys * p.F;
                         return split ? v * kShortKeyCost + 1 : v * kLongKeyCost;
                     },
                     [&](int rg, int hg, long long v0, long long v1, bool fin, int slot, long long rk) {
                         if (uniform((int)rk & 1))
                             chunk_piece<DT, QM, KVM, P2, RM, 4>(p, smem, pages, uniform(rg), uniform(hg),
                                                                 uniform(v0 / kShortKeyCost),
                                                                 uniform(v1 / kShortKeyCost), uniform((int)fin) != 0,
                                                                 uniform(slot), uniform(rk / kShortKeyCost));
                         else
                             chunk_piece<DT, QM, KVM, P2, RM, 1>(p, smem, pages, uniform(rg), uniform(hg),
                                                                 uniform(v0 / kLongKeyCost),
                                                                 uniform(v1 / kLongKeyCost), uniform((int)fin) != 0,
                                                                 uniform(slot), uniform(rk / kLongKeyCost));
                     });
    }
}

size_t lds_bytes(int nrows) {
    return 256 + (size_t)kRingBytes + (size_t)kPageCap * 4 + (size_t)(kWaves + nrows + 1) * sizeof(long long);
}

// ---- varlen row groups ----------------------------------------------------------
//
// Token t of a varlen call belongs to the first sequence i with
// t < cu_seqlens_q[i + 1], or to sequence 0 when there is none (the decode
// path's rule, varlen_paged_kernel_v21.cuh:40-47).  With M_i the running
// maximum of cu_seqlens_q[1 .. i + 1], sequence i's tokens are therefore
// [max(0, M_{i-1}), min(T, M_i)) (M_{-1} = 0), and the tokens from M_{W-1} on
// form one more run, of sequence 0 -- also for tables that are not
// non-decreasing.  Each run is cut into groups of kTokBlk tokens.  One
// workgroup writes entry g = {first token, tokens, sequence, 0} for every
// group, and {0, 0, 0, 0} for the entries from the group count up to gmax
// (the host's bound T / kTokBlk + W + 1: a run of n tokens makes at most
// n / kTokBlk + 1 groups).
constexpr int kVgThreads = 1024;

__device__ inline int block_scan_excl(int v, int* s_part, bool is_max) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int ident = is_max ? INT_MIN : 0;
    int incl = v;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(incl, d, kWave);
        if (lane >= d) incl = is_max ? (o > incl ? o : incl) : incl + o;
    }
    if (lane == 63) s_part[wv] = incl;
    __syncthreads();
    int before = ident;
    for (int i = 0; i < wv; ++i) before = is_max ? (s_part[i] > before ? s_part[i] : before) : before + s_part[i];
    const int excl_lane = __shfl_up(incl, 1, kWave);
    const int mine = lane == 0 ? ident : excl_lane;
    __syncthreads();
    return is_max ? (mine > before ? mine : before) : before + mine;
}

__global__ __launch_bounds__(kVgThreads) void dv_varlen_groups(const int* cu, int W, int T, int gmax, int4* groups) {
    __shared__ int s_m[kVarlenChunkMaxW];       // M_i
    __shared__ int s_base[kVarlenChunkMaxW + 2];  // first group of run i (runs 0 .. W), then the total
    __shared__ int s_part[kVgThreads / kWave];
    const int tid = threadIdx.x;
    // running maximum of cu[1 .. W], each thread over a contiguous block of sequences
    const int per = (W + kVgThreads - 1) / kVgThreads;
    const int i0 = tid * per < W ? tid * per : W, i1 = i0 + per < W ? i0 + per : W;
    int mx = INT_MIN;
    for (int i = i0; i < i1; ++i) {
        const int c = cu[i + 1];
        mx = c > mx ? c : mx;
        s_m[i] = mx;
    }
    const int before = block_scan_excl(mx, s_part, true);
    for (int i = i0; i < i1; ++i) s_m[i] = s_m[i] > before ? s_m[i] : before;
    __syncthreads();
    // run i (i < W: sequence i; i == W: the tokens past M_{W-1}) = [a, b)
    auto run = [&](int i, int& a, int& b) {
        a = i == 0 ? 0 : (s_m[i - 1] > 0 ? s_m[i - 1] : 0);
        b = i == W ? T : (s_m[i] < T ? s_m[i] : T);
    };
    const int per1 = (W + 1 + kVgThreads - 1) / kVgThreads;
    const int j0 = tid * per1 < W + 1 ? tid * per1 : W + 1, j1 = j0 + per1 < W + 1 ? j0 + per1 : W + 1;
    int cnt = 0;
    for (int i = j0; i < j1; ++i) {
        int a, b;
        run(i, a, b);
        const int c = b > a ? (b - a + kTokBlk - 1) / kTokBlk : 0;
        s_base[i] = c;
        cnt += c;
    }
    int acc = block_scan_excl(cnt, s_part, false);
    for (int i = j0; i < j1; ++i) {
        const int c = s_base[i];
        s_base[i] = acc;
        acc += c;
    }
    if (tid == kVgThreads - 1) s_base[W + 1] = acc;
    __syncthreads();
    const int total = s_base[W + 1];
    for (int gi = tid; gi < gmax; gi += kVgThreads) {
        int4 e = {0, 0, 0, 0};
        if (gi < total) {
            // the last run whose first group is <= gi (it has groups: the next run's first is larger)
            int lo = 0, hi = W;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_base[mid] <= gi) lo = mid;
                else hi = mid - 1;
            }
            int a, b;
            run(lo, a, b);
            const int t0 = a + (gi - s_base[lo]) * kTokBlk;
            e.x = t0;
            e.y = b - t0 < kTokBlk ? b - t0 : kTokBlk;
            e.z = lo == W ? 0 : lo;
        }
        groups[gi] = e;
    }
}

template <int DT, int QM, int KVM, bool P2, int RM, int KS>
hipError_t launch1(DecodeParams p, int device, int cus, long long cap, hipStream_t stream) {
    static std::atomic<unsigned long long> attr_done{0};
    hipError_t ea = once_per_device(attr_done, device, [] {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(&dv_chunk<DT, QM, KVM, P2, RM, KS>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes(kMaxRows));
    });
    if (ea != hipSuccess) return ea;
    const size_t lds = lds_bytes(p.nrows);
    long long nwg = cus;  // one eight-wave workgroup per CU (LDS ring 96 KiB)
    if (nwg > cap) nwg = cap;
    p.nwg = nwg < 1 ? 1 : (int)nwg;
    hipLaunchKernelGGL((dv_chunk<DT, QM, KVM, P2, RM, KS>), dim3(p.nwg), dim3(kThreads), lds, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int ntb = max_group_tokens<RM>(p);
    hipLaunchKernelGGL((dv_merge_chunk<DT, RM>), dim3(p.nrows * p.Hkv * ntb), dim3(256), 0, stream, p, ntb);
    return hipGetLastError();
}

template <int DT, int QM, int KVM, int RM, bool P2>
hipError_t launch_split(const DecodeParams& p, int ks, int device, int cus, long long cap, hipStream_t stream) {
    if constexpr (RM == kRowVarlen) {
        return launch1<DT, QM, KVM, P2, RM, 0>(p, device, cus, cap, stream);
    } else {
        if (ks == 4) return launch1<DT, QM, KVM, P2, RM, 4>(p, device, cus, cap, stream);
        if (ks == 2) return launch1<DT, QM, KVM, P2, RM, 2>(p, device, cus, cap, stream);
        return launch1<DT, QM, KVM, P2, RM, 1>(p, device, cus, cap, stream);
    }
}

template <int DT, int QM, int KVM, int RM>
hipError_t launch(const DecodeParams& p, int ks, int device, int cus, long long cap, hipStream_t stream) {
    if constexpr (DT == kF32) {
        return launch_chunk32(QM, KVM, RM, p, device, cus, cap, stream);
    } else {
        if constexpr (KVM == kKvPaged)
            if (p.bs_shift >= 0) return launch_split<DT, QM, KVM, RM, true>(p, ks, device, cus, cap, stream);
        return launch_split<DT, QM, KVM, RM, false>(p, ks, device, cus, cap, stream);
    }
}

// Key split of a launch whose groups have at most ntok tokens: as many wave sets
// as hold two tokens per wave.  (Eight sets for two tokens would take a ring step
// of all eight stages, with nothing in flight beside it; two tokens run at 5.3
// TB/s with four.)  Faster than no split over the whole range: 2 / 4 / 8 tokens,
// bf16, one sequence of 3001 keys, 8 KV heads 29.7 / 30.8 / 32.7 -> 26.2 / 27.1 /
// 29.1 us; fp16, 32 x 4608 keys 224 / 223 / 234 -> 112 / 114 / 153; contiguous fp16,
// 16 x 4096 keys 119 / 120 / 122 -> 60 / 63 / 84; 64 x 60-100 keys, bf16 50.1 /
// 52.5 / 58.7 -> 45.1 / 47.0 / 51.6.  A split step with no visible key must leave no
// trace in the softmax, which -inf scores only do for a positive scale.  Short views
// gain nothing (each one's queries are staged for all sets, and a piece ends with the
// sets' combination), so a call is split from 48 keys per view on, as far as the host
// knows them (paged: what the block tables hold), and a contiguous one of 5 - 8
// tokens in several views from 128 on: without the split / with it, 8 KV heads, 6 x 30
// contiguous keys, 2 tokens 68 / 76 us, paged 96 / 99; 12 x 90 contiguous, 8 tokens 62
// / 67; 6 x 60 paged, 2 / 8 tokens 65 / 62, 70 / 62; 6 x 150 contiguous, 8 tokens 51 / 50.
int key_split(float l2scale, int ntok, long long keys, int F, bool contig) {
    if (!(l2scale > 0.0f) || ntok > 8) return 1;
    const int ks = ntok > kFewTok ? 2 : 4;
    const long long per_view = contig && ks == 2 && F > 1 ? kSplitContig2Keys : kSplitMinKeys;
    return keys < per_view * F ? 1 : ks;
}

}  // namespace chunk

namespace {
int chunk_cus(int device) { return device_cu_count(device); }

// Workspace of the chunk path for `groups` row groups: partial slots, merge
// directory, and (varlen) the group table.
struct ChunkWs {
    size_t part, dir, vgroups, total;
};

ChunkWs chunk_ws(long long groups, int Hkv, int device, bool varlen) {
    const long long rows = groups < kMaxRows ? groups : kMaxRows;
    const long long nseg = rows * Hkv;
    const long long slot_floats = (long long)chunk::kTokBlk * kGqa * (kHeadDim + 1);
    ChunkWs l;
    l.part = ((size_t)((chunk_cus(device) + nseg) * slot_floats * 4) + 255) & ~(size_t)255;
    l.dir = ((size_t)(nseg * 2 * 4) + 255) & ~(size_t)255;
    l.vgroups = varlen ? (size_t)groups * 16 : 0;
    l.total = l.part + l.dir + l.vgroups;
    return l;
}

long long varlen_gmax(int T, int W) { return (long long)T / chunk::kTokBlk + W + 1; }

// The chunk launches over `groups` row groups, kMaxRows at a time.
template <int RM>
hipError_t launch_groups(int dtype, int qmode, int kvmode, DecodeParams p, long long groups_total,
                         long long max_keys_per_group, int ks, const ChunkWs& l, void* workspace,
                         hipStream_t stream) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const int cus = chunk_cus(device);
    p.hpw = 1;
    p.slot_floats = chunk::kTokBlk * kGqa * (kHeadDim + 1);
    p.part = reinterpret_cast<float*>(workspace);
    p.dir = reinterpret_cast<int*>(reinterpret_cast<unsigned char*>(workspace) + l.part);
    // ks = 0: the schedule counts in cost units (dv_chunk)
    const int unit = ks == 0 ? chunk::kLongKeyCost : 1;
    p.piece_cost = unit * (ks <= 1 ? chunk::kPieceCost : chunk::kPieceCostSplit);
    const int min_keys = p.min_keys;
    p.min_keys *= unit;
    // odd workgroups (odd XCD of each pair) take shorter chunks, as in the decode
    // split; 30 per mille measured best on configuration 5
    static const int skew = env_per_mille("DVATTN_CHUNK_SKEW_PM", 30);
    p.skew_pm = skew;
    for (long long g0 = 0; g0 < groups_total; g0 += kMaxRows) {
        p.row_begin = (int)g0;
        p.nrows = (int)(groups_total - g0 < kMaxRows ? groups_total - g0 : kMaxRows);
        const long long cap = ((long long)p.nrows * p.Hkv * max_keys_per_group + min_keys - 1) / min_keys;
        if constexpr (RM == kRowVarlen) {
            if (dtype == kBF16 && qmode == kQRotHalf && kvmode == kKvPaged)
                e = chunk::launch<kBF16, kQRotHalf, kKvPaged, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kF16 && qmode == kQRotHalf && kvmode == kKvPaged)
                e = chunk::launch<kF16, kQRotHalf, kKvPaged, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kF32 && qmode == kQRotHalf && kvmode == kKvPaged)
                e = chunk::launch<kF32, kQRotHalf, kKvPaged, RM>(p, ks, device, cus, cap, stream);
            else
                e = hipErrorInvalidValue;
        } else {
            if (dtype == kBF16 && qmode == kQRotFull && kvmode == kKvPaged)
                e = chunk::launch<kBF16, kQRotFull, kKvPaged, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kF16 && qmode == kQRotFull && kvmode == kKvPaged)
                e = chunk::launch<kF16, kQRotFull, kKvPaged, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kBF16 && qmode == kQPre && kvmode == kKvContig)
                e = chunk::launch<kBF16, kQPre, kKvContig, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kF16 && qmode == kQPre && kvmode == kKvContig)
                e = chunk::launch<kF16, kQPre, kKvContig, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kF32 && qmode == kQRotFull && kvmode == kKvPaged)
                e = chunk::launch<kF32, kQRotFull, kKvPaged, RM>(p, ks, device, cus, cap, stream);
            else if (dtype == kF32 && qmode == kQPre && kvmode == kKvContig)
                e = chunk::launch<kF32, kQPre, kKvContig, RM>(p, ks, device, cus, cap, stream);
            else
                e = hipErrorInvalidValue;
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
}  // namespace

size_t chunk_workspace_bytes(int W, int S, int Hkv, int device) {
    if (W <= 0 || S <= 0 || Hkv <= 0) return 0;
    const long long groups = (long long)W * ((S + chunk::kTokBlk - 1) / chunk::kTokBlk);
    return chunk_ws(groups, Hkv, device, false).total;
}

hipError_t launch_chunk(int dtype, int qmode, int kvmode, const DecodeParams& base, long long max_keys_per_group,
                        void* workspace, size_t ws_bytes, hipStream_t stream) {
    if (base.W <= 0 || base.S <= 0 || base.Hkv <= 0) return hipSuccess;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const long long groups = (long long)base.W * ((base.S + chunk::kTokBlk - 1) / chunk::kTokBlk);
    const ChunkWs l = chunk_ws(groups, base.Hkv, device, false);
    if (ws_bytes < l.total) return hipErrorInvalidValue;
    const int ks = dtype == kF32 ? 1
                                 : chunk::key_split(base.l2scale, base.S, max_keys_per_group, base.F,
                                                    kvmode == kKvContig);
    return launch_groups<kRowWS>(dtype, qmode, kvmode, base, groups, max_keys_per_group, ks, l, workspace, stream);
}

size_t varlen_chunk_workspace_bytes(int T, int W, int Hkv, int device) {
    if (T <= 0 || W <= 0 || Hkv <= 0) return 0;
    return chunk_ws(varlen_gmax(T, W), Hkv, device, true).total;
}

hipError_t launch_varlen_chunk(int dtype, const DecodeParams& base, long long max_keys_per_group, void* workspace,
                               size_t ws_bytes, hipStream_t stream) {
    if (base.T <= 0 || base.W <= 0 || base.Hkv <= 0) return hipSuccess;
    if (base.W > kVarlenChunkMaxW) return hipErrorInvalidValue;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const long long gmax = varlen_gmax(base.T, base.W);
    const ChunkWs l = chunk_ws(gmax, base.Hkv, device, true);
    if (ws_bytes < l.total) return hipErrorInvalidValue;
    DecodeParams p = base;
    int4* groups = reinterpret_cast<int4*>(reinterpret_cast<unsigned char*>(workspace) + l.part + l.dir);
    p.vgroups = reinterpret_cast<const int*>(groups);
    hipLaunchKernelGGL(chunk::dv_varlen_groups, dim3(1), dim3(chunk::kVgThreads), 0, stream, base.cu_q, base.W,
                       base.T, (int)gmax, groups);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int ks = dtype == kF32 ? 1 : 0;
    return launch_groups<kRowVarlen>(dtype, kQRotHalf, kKvPaged, p, gmax, max_keys_per_group, ks, l, workspace,
                                     stream);
}

}  // namespace dv
