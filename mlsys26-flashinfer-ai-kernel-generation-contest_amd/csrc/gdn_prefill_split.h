// Column-split scan body (in the 4-wave scan and the segment kernel): 32 state rows per workgroup, each
// 16-row group's work of a chunk split over two waves.
#pragma once

#include <cstddef>

#include "gdn_prefill.h"

namespace gdn {

// A chunk in LDS (52 KB, double-buffered). K and Q as in ScanBuf; V row t (the workgroup's 32
// value columns, four 16-byte units), unit c at 4 t + (c ^ 2 (t / 8 % 2)); R is the record with
// the 16-byte units (row r, column half h) of each 16x16 block moved to 16 h + (r ^ 4 h) (T')
// or 16 h + r (P'), which keeps the operand reads free of bank conflicts (the T' rows of a
// tile fix bit 2 of r, the P' rows run over all 16).
struct SplitBuf {
    u32x4 K[kC * 16], Q[kC * 16], V[kC * 4], R[kRecBytes / 16];
};

// What the two waves (hc = 0, 1) of a row group hand each other, one 16-byte unit per lane.
struct SplitExch {
    u32x4 X[2][2][2][64];  // [row group][writer hc][tile]: partial X, later W hi / lo
    u32x4 O[2][2][2][64];  // partial S0 Q^T
    u32x4 Rr[2][2][64];    // R hi / lo of tokens 0 .. 31
    u32x4 U[2][64];        // U (bf16) of tokens 0 .. 31
};

// The bodies' LDS, in two parts that overlay the 64-row and 8-wave bodies' two chunk buffers
struct SplitLdsA {
    SplitBuf buf;
    SplitExch e;
};
struct SplitLdsB {
    SplitBuf buf;
    u32x4 ml[kMtUnits];  // chain steps: the low half of M^T (the high half is in buf)
};

// Wave (rg, hc) owns state rows v0 + 16 rg .. + 15, columns 64 hc .. + 63, and finishes the
// chunk's tokens 32 hc .. + 31; a fifth wave issues the copies. Per chunk (arithmetic and tile
// layouts of scan_body, gdn_prefill_scan.hip):
//   X and S0 Q^T over the wave's columns for all tokens; the other half's tokens go to the
//     other wave (barriers 1 and 2), which adds them to its own;
//   R and U of the wave's tokens; U of tokens 32 .. 63 also needs R of 0 .. 31 (barrier 2);
//   W of the wave's tokens to the other wave (barrier 3); S over the wave's columns, its own
//     tokens' terms before the barrier.
// A lone wave per SIMD runs its VALU, MFMA and LDS instructions one after the other (with the
// copies left out a 64-row body's chunk took 4.5k cycles: 1.6k MFMA, 1.4k VALU, 1.0k LDS, the
// rest latency and the barrier), so half the work per wave shortens the chunk, by less than half
// because of three more barriers and the exchanges: ~3.6k cycles. That needs twice the CUs.
// Whole prefills on MI355X against the 64-row bodies: 1 x 77 at 8 v-heads 13.75 -> 12.6 us, 1 x
// 300 at 32 19.95 -> 18.6, 1 x 1024 at 8 32.3 -> 29.6, 8 of 64 to 1024 at 8 39.7 -> 37.8. Two waves of this kind per SIMD (64 rows
// per workgroup) were slower than one 64-row body: 8 sequences of 64 to 1024 44 -> 51 us.
template <bool SEG, int INST, int OUTS>
__device__ __forceinline__ void split_body(const ScanArgs &p, const ScanJob &job, SplitLdsA &la_,
                                           SplitLdsB &lb_)
{
    SplitBuf &BA = la_.buf, &BB = lb_.buf;
    SplitExch &E = la_.e;
    constexpr bool kOut = OUTS == 1;
    const int grp = job.grp, wi = job.wi, n = job.n, tok0 = job.tok0, len = job.len,
              c0 = job.c0, kind = SEG ? job.kind : kJobFirst, cb = SEG ? job.cb : 0,
              q = SEG ? job.q : -1, steps = SEG ? job.steps : 0, last = SEG ? job.last : 0;
    const int g = grp % p.HQK, h = g * p.ratio + wi / 4, v0 = (wi % 4) * 32;
    // records exist only for chunk ids < header[0] (see the plan kernel's clamp)
    const int nck = min((len + kC - 1) / kC, max(p.header[0] - c0, 0));
    const int ce = min(SEG ? job.ce : 0x7fffffff, nck);

    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63,
              lr = l & 15, lg = l >> 4, rg = w & 1, hc = (w >> 1) & 1;
    const int v0w = v0 + 16 * rg;
    const SplitConsts sk = split_consts();
    auto split2 = [&](float a, float b, uint32_t &hi, uint32_t &lo) { split_bf16x2(a, b, hi, lo, sk); };

    const uint32_t kst2 = (uint32_t)p.k_st * 2, qst2 = (uint32_t)p.q_st * 2;
    const uint32_t vst2 = (uint32_t)p.v_st * 2, ost2 = (uint32_t)p.o_st * 2;
    const char *kbase = (const char *)(p.k + (int64_t)tok0 * p.k_st + g * p.k_sh);
    const char *qbase = (const char *)(p.q + (int64_t)tok0 * p.q_st + g * p.q_sh);
    const char *vbase = (const char *)(p.v + (int64_t)tok0 * p.v_st + h * p.v_sh + v0);
    char *obase = (char *)(p.out + (int64_t)tok0 * p.o_st + h * p.o_sh + v0w);
    const int64_t kstep = (int64_t)kC * p.k_st * 2, qstep = (int64_t)kC * p.q_st * 2;
    const int64_t vstep = (int64_t)kC * p.v_st * 2, ostep = (int64_t)kC * p.o_st * 2;
    const char *rbase = p.records + ((int64_t)c0 * p.HV + h) * kRecBytes;
    const int64_t rstep = (int64_t)p.HV * kRecBytes;
    auto rsrc = [&](const char *base, uint32_t range) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)range, 0x00020000);
    };

    // ---- the copy wave (see scan_body): 1 KB windows of K and Q (4 rows), V (16 rows) and the
    // record (two blocks; T' 0 .. 9, P' 10 .. 14, gates 15). Rows past a chunk's end read as
    // zero: they meet beta = 0 or the causal mask only.
    if (w == 4) {
        const int r = l >> 4, cs = l & 15;
        uint32_t rk = r * kst2, rq = r * qst2, sk4 = 16u * (cs ^ kswz(r)), sq4 = 16u * (cs ^ r),
                 rv = (l >> 2) * vst2 + 16u * ((l & 3) ^ (2 * (l >> 5)));
        const uint32_t hb = (l >> 4) & 1;
        const uint32_t rofT = 512u * (l >> 5) + 16u * (2 * ((l & 15) ^ (4 * hb)) + hb),
                       rofP = 512u * (l >> 5) + 16u * (2 * (l & 15) + hb), rofG = 16u * l;
        const uint32_t la = (uint32_t)(uintptr_t)(GDN_LDS char *)&BA,
                       lb = (uint32_t)(uintptr_t)(GDN_LDS char *)&BB;
        auto issue = [&](uint32_t buf, int c) {
            const uint32_t rows = min(kC, len - c * kC) - 1;
            const auto sk_ = rsrc(kbase + c * kstep, rows * kst2 + 256u), sr = rsrc(rbase + c * rstep, kRecBytes);
            asm volatile("" : "+v"(rk), "+v"(rq), "+v"(sk4), "+v"(sq4), "+v"(rv));
            auto copy = [&](__amdgpu_buffer_rsrc_t rs, uint32_t dst, uint32_t off, int soff) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (GDN_LDS void *)(uintptr_t)(buf + dst), 16, off, soff, 0, 0);
            };
#pragma unroll
            for (int b = 0; b < 16; ++b)
                copy(sk_, offsetof(SplitBuf, K) + 1024 * b, rk + 4 * b * kst2 + (sk4 ^ (16u * kswz(4 * b))), 0);
            if constexpr (OUTS != 2) {  // identity rows: V = 0
                const auto sv = rsrc(vbase + c * vstep, rows * vst2 + 64u);
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    copy(sv, offsetof(SplitBuf, V) + 1024 * b, rv + 16 * b * vst2, 0);
            }
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                if (!kOut && b >= 10 && b < 15)  // state maps read neither Q nor P'
                    continue;
                copy(sr, offsetof(SplitBuf, R) + 1024 * b, b < 10 ? rofT : b < 15 ? rofP : rofG, 1024 * b);
            }
            if constexpr (kOut) {
                const auto sq = rsrc(qbase + c * qstep, rows * qst2 + 256u);
#pragma unroll
                for (int b = 0; b < 16; ++b)
                    copy(sq, offsetof(SplitBuf, Q) + 1024 * b, rq + 4 * b * qst2 + (sq4 ^ (64u * (b & 3))), 0);
            }
        };
        if (ce > cb)
            issue(la, cb);
        for (int m = 0; m < 2 * steps; ++m)
            __builtin_amdgcn_s_barrier();
        for (int c = cb; c < ce; ++c) {
            dma_barrier();
            if (c + 1 < ce)
                issue((c - cb) & 1 ? la : lb, c + 1);
#pragma unroll
            for (int b = 0; b < 3; ++b)
                __builtin_amdgcn_s_barrier();
        }
        return;
    }

    // ---- LDS read offsets (bytes)
    const int c_ = lr & 3, r_ = lr >> 2;
    const int ta = 8 * (lr >> 2) + (lr & 3), tk = 8 * lg + r_;  // rows of the K and K^T reads
    uint32_t koffA[2], ktoff[2], qoff[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int s4 = 4 * (2 * hc + s);
        koffA[s] = 16u * (16 * ta + ((s4 + lg) ^ kswz(ta)));
        ktoff[s] = 256u * tk + 16u * ((s4 + c_) ^ kswz(tk));
        qoff[s] = 16u * (16 * lr + ((s4 + lg) ^ lr));
    }
    const uint32_t voff = 64u * (32 * hc + 8 * lg + r_) + 16u * ((2 * rg + (c_ >> 1)) ^ (2 * (lg & 1))) + 8u * (c_ & 1);
    // T' of tile 2 hc + j: rows 32 hc + 8 (lr / 4) + 4 j + lr % 4; k-step sp: columns 32 sp +
    // 8 lg .. + 7. The k-step sp = hc meets absent blocks, whose lanes read the record's zeros.
    const int bh = lg >> 1;
    uint32_t tdh[2], tdl[2], trm[2], pd[2], prm[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t u = 256u * (lg & 1) + 16u * (8 * ((lr >> 2) & 1) + (lr & 3)) + 64u * (j ^ (lg & 1));
        const int bi = 2 * hc + (lr >> 3), bj = 2 * hc + bh;
        tdh[j] = bj <= bi ? 512u * tri_blk(bi, bj) + u : kRecZero;
        tdl[j] = bj <= bi ? kRecTlo + 512u * tri_blk(bi, bj) + u : kRecZero;
        trm[j] = 512u * tri_blk(2 + (lr >> 3), bh) + u;
        const uint32_t up = kRecP + 256u * (lg & 1) + 16u * lr;
        pd[j] = bh <= j ? up + 512u * tri_blk(2 * hc + j, bj) : kRecZero;
        prm[j] = up + 512u * tri_blk(2 + j, bh);
    }
    const uint32_t gof = kRecGates + 32u * lg + 128u * hc, sgof = kRecGates + 512 + 4u * lr + 128u * hc;
    auto ld = [](const u32x4 *b, uint32_t off) { return *(const u32x4 *)((const char *)b + off); };
    auto ldf = [](const u32x4 *b, uint32_t off) { return *(const f32x4 *)((const char *)b + off); };

    // this lane's units of a slot in register-image order: S[t] at + 256 t
    auto seg_img = [&](const float *base, int qs) {
        return base + ((int64_t)qs * p.HV + h) * kSlotFloats + (((v0w >> 4) * 8 + 4 * hc) * 64 + l) * 4;
    };

    // A resumed segment with chain steps copies the first step's M^T (hi into BB, lo into its
    // own area) and loads R.
    const bool chain = SEG && steps > 0;
    static_assert(sizeof(SplitBuf) >= (kMtUnits + 2 * 512) * 16, "M^T hi and the exchanged state must fit");
    u32x4 *mh = (u32x4 *)&BB, *ml = lb_.ml;
    auto issue_m = [&](int qs) {
        const auto rs = rsrc((const char *)(p.seg_mt + ((int64_t)qs * p.HV + h) * kSlotFloats), 2 * kMtUnits * 16);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int b = w + 4 * i;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (GDN_LDS void *)&mh[64 * b], 16, 16u * l, 1024 * b, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (GDN_LDS void *)&ml[64 * b], 16, 16u * l,
                                                     1024 * b + kMtUnits * 16, 0, 0);
        }
    };
    f32x4 R[4];
    auto load_r = [&](int qs) {
        const float *rp = seg_img(p.seg_r, qs);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            R[t] = *(const f32x4 *)(rp + 256 * t);
    };
    if (chain) {
        issue_m(q);
        load_r(q);
    }
    // ---- state: S[2 s + hh] holds S[v0w + lr][64 hc + 32 s + 8 lg + 4 hh + i], i = 0..3
    f32x4 S[4];
    if (SEG && kind == kJobResume) {
        const float *ip = seg_img(p.seg_sin, q);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            S[t] = *(const f32x4 *)(ip + 256 * t);
    } else if (kind == kJobFirst && p.state) {
        const float *sp = p.state + n * p.st_sn + h * p.st_sh + (int64_t)(v0w + lr) * p.st_sv + 64 * hc + 8 * lg;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            S[t] = *(const f32x4 *)(sp + 32 * (t >> 1) + 4 * (t & 1));
    } else {
        const bool ident = SEG && kind == kJobIdent;  // row v0w + lr of the identity
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                S[t][i] = ident && 64 * hc + 32 * (t >> 1) + 8 * lg + 4 * (t & 1) + i == v0w + lr ? 1.f : 0.f;
    }

    // ---- chain steps of a resumed segment: S <- S M_m + R_m for the slots q .. q + steps - 1
    // (see scan_body; here each wave's output tiles are its own columns, and the other half of
    // its rows' state, split into bf16 hi + lo, comes from the other wave through LDS).
    if (chain) {
        u32x4 *sx = mh + kMtUnits + 512 * rg;
        for (int m = 0; m < steps; ++m) {
            u32x4 Bh[4], Bl[4];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                u32x4 bh4, bl4;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f32x4 x = S[2 * s + (e >> 1)];
                    uint32_t hi, lo;
                    split2(x[2 * (e & 1)], x[2 * (e & 1) + 1], hi, lo);
                    bh4[e] = hi;
                    bl4[e] = lo;
                }
                Bh[s] = bh4;
                Bl[s] = bl4;
                sx[256 * hc + 128 * s + l] = bh4;
                sx[256 * hc + 128 * s + 64 + l] = bl4;
            }
            dma_barrier();  // M_m^T and every wave's half of the state are in LDS, R_m in registers
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                Bh[2 + s] = sx[256 * (1 - hc) + 128 * s + l];
                Bl[2 + s] = sx[256 * (1 - hc) + 128 * s + 64 + l];
            }
            // k-steps in the order own, other: columns 64 hc + 32 s, then 64 (1 - hc) + 32 s
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int tg = 4 * hc + t, j = 32 * (tg >> 1) + 8 * (lr >> 2) + 4 * (tg & 1) + (lr & 3),
                          sw = kswz(j);
                f32x4 acc = R[t];
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const int kg = 2 * ((ks >> 1) ^ hc) + (ks & 1), u = 16 * j + ((4 * kg + lg) ^ sw);
                    const u32x4 ah = mh[u], al = ml[u];
                    acc = mfma_bf16(ah, Bh[ks], acc);
                    acc = mfma_bf16(ah, Bl[ks], acc);
                    acc = mfma_bf16(al, Bh[ks], acc);
                }
                S[t] = acc;
            }
            lds_barrier_inflight();  // every wave is done with M_m^T and the exchanged state
            if (m + 1 < steps) {
                issue_m(q + m + 1);
                load_r(q + m + 1);
            }
        }
    }

    auto chunk = [&](SplitBuf &B, int c) {
        const int lenc = min(kC, len - c * kC);
        const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
        auto kA = [&](int tt, int s) { return ld(B.K, koffA[s] + 256 * (32 * (tt >> 1) + 4 * (tt & 1))); };
        auto qA = [&](int tt, int s) { return ld(B.Q, qoff[s] + 4096 * tt); };

        // X and S0 Q^T over this wave's columns: the other wave's tokens first. S0 dies in its
        // split (residuals formed in its registers) and goes on as gammaC S0.
        const float gC = *(const float *)((const char *)B.R + kRecGates + 768);
        u32x4 ka[4][2], Sh[2], Sl[2];
        const int to = 2 * (1 - hc), tm = 2 * hc;  // the other's and this wave's first tile
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < 2; ++s)
                ka[i][s] = kA((i < 2 ? to : tm) + (i & 1), s);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f32x4 &x = S[2 * s + (e >> 1)];
                const float a = x[2 * (e & 1)], b = x[2 * (e & 1) + 1];
                float ga = gC * a, gb = gC * b;
                asm volatile("" : "+v"(ga), "+v"(gb));  // keeps the products from sinking to their use
                x[2 * (e & 1)] = ga;
                x[2 * (e & 1) + 1] = gb;
                uint32_t hi, lo;
                split2(a, b, hi, lo);
                Sh[s][e] = hi;
                Sl[s][e] = lo;
            }
        u32x2 vv[2];
        f32x4 gm[2];
        u32x4 qa[4][2];
        f32x4 X[4];
        // one tile per scheduling region, reads of what comes after barrier 1 between them
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            X[i] = z4;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                X[i] = mfma_bf16(ka[i][s], Sh[s], X[i]);
                X[i] = mfma_bf16(ka[i][s], Sl[s], X[i]);
                if constexpr (kOut)
                    qa[i][s] = qA((i < 2 ? to : tm) + (i & 1), s);
            }
            if (i < 2) {
                if constexpr (OUTS == 2)
                    vv[i] = u32x2{0u, 0u};
                else
                    vv[i] = lds_tr16((const char *)B.V + voff + 256 * i);
                gm[i] = ldf(B.R, gof + 16 * i);
            }
            if (i >= 2)
                E.X[rg][hc][i - 2][l] = __builtin_bit_cast(u32x4, X[i - 2]);
        }
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier_inflight();  // 1: partial X
        f32x4 Xo[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
            Xo[j] = __builtin_bit_cast(f32x4, E.X[rg][1 - hc][j][l]);
        f32x4 O[4];
        if constexpr (kOut) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                O[i] = mfma_bf16(Sh[0], qa[i][0], z4);
                O[i] = mfma_bf16(Sh[1], qa[i][1], O[i]);
            }
        }
        u32x4 td[2][2], tr[2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            td[j][0] = ld(B.R, tdh[j]);
            td[j][1] = ld(B.R, tdl[j]);
        }
        __builtin_amdgcn_sched_barrier(0);

        // R = V - gamma X of this wave's tokens, hi + lo
        u32x4 Rh, Rl;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const f32x4 x = X[2 + j] + Xo[j];
            const float r0 = fmaf(-gm[j][0], x[0], bf16lo(vv[j][0])), r1 = fmaf(-gm[j][1], x[1], bf16hi(vv[j][0])),
                        r2 = fmaf(-gm[j][2], x[2], bf16lo(vv[j][1])), r3 = fmaf(-gm[j][3], x[3], bf16hi(vv[j][1]));
            uint32_t h01, l01, h23, l23;
            split2(r0, r1, h01, l01);
            split2(r2, r3, h23, l23);
            Rh[2 * j] = h01; Rh[2 * j + 1] = h23;
            Rl[2 * j] = l01; Rl[2 * j + 1] = l23;
        }
        if (hc == 0) {
            E.Rr[rg][0][l] = Rh;
            E.Rr[rg][1][l] = Rl;
        }
        // U = T' R, this wave's k-step
        f32x4 U[2], dc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            U[j] = mfma_bf16(td[j][0], Rh, z4);
            U[j] = mfma_bf16(td[j][0], Rl, U[j]);
            U[j] = mfma_bf16(td[j][1], Rh, U[j]);
            dc[j] = ldf(B.R, gof + 256 + 16 * j);
        }
        if (hc == 1)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                tr[j][0] = ld(B.R, trm[j]);
                tr[j][1] = ld(B.R, trm[j] + kRecTlo);
            }
        float sg[2];
        u32x4 pa[2];
        if constexpr (kOut) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                E.O[rg][hc][j][l] = __builtin_bit_cast(u32x4, O[j]);
                sg[j] = *(const float *)((const char *)B.R + sgof + 64 * j);
                pa[j] = ld(B.R, pd[j]);
            }
        }
        u32x4 kt[4][2];
        auto ktRead = [&](int t, int sp) {
            const uint32_t o = ktoff[t >> 1] + 256 * (32 * sp) + 8 * (t & 1);
            const u32x2 k0 = lds_tr16((const char *)B.K + o), k1 = lds_tr16((const char *)B.K + o + 1024);
            return u32x4{k0[0], k0[1], k1[0], k1[1]};
        };
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier_inflight();  // 2: R of tokens 0 .. 31, partial S0 Q^T
        f32x4 Oo[2];
        if constexpr (kOut) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
                Oo[j] = __builtin_bit_cast(f32x4, E.O[rg][1 - hc][j][l]);
        }
        if (hc == 1) {
            const u32x4 r0h = E.Rr[rg][0][l], r0l = E.Rr[rg][1][l];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                U[j] = mfma_bf16(tr[j][0], r0h, U[j]);
                U[j] = mfma_bf16(tr[j][0], r0l, U[j]);
                U[j] = mfma_bf16(tr[j][1], r0h, U[j]);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
            kt[t][0] = ktRead(t, hc);
        // W = dec U (hi + lo), U (bf16)
        u32x4 Wh, Wl, Ub;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (kOut) {
                Ub[2 * j] = pack_bf16x2(U[j][0], U[j][1]);
                Ub[2 * j + 1] = pack_bf16x2(U[j][2], U[j][3]);
            }
            uint32_t h01, l01, h23, l23;
            split2(dc[j][0] * U[j][0], dc[j][1] * U[j][1], h01, l01);
            split2(dc[j][2] * U[j][2], dc[j][3] * U[j][3], h23, l23);
            Wh[2 * j] = h01; Wh[2 * j + 1] = h23;
            Wl[2 * j] = l01; Wl[2 * j + 1] = l23;
        }
        E.X[rg][hc][0][l] = Wh;
        E.X[rg][hc][1][l] = Wl;
        if (kOut && hc == 0)
            E.U[rg][l] = Ub;
        __builtin_amdgcn_sched_barrier(0);
        // S = gammaC S0 + W^T K, this wave's tokens; O = scale gamma S0 Q^T + U^T P'^T
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            S[t] = mfma_bf16(kt[t][0], Wh, S[t]);
            S[t] = mfma_bf16(kt[t][0], Wl, S[t]);
            kt[t][1] = ktRead(t, 1 - hc);
        }
        u32x4 pr[2];
        if constexpr (kOut) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                O[2 + j] = sg[j] * (O[2 + j] + Oo[j]);
                O[2 + j] = mfma_bf16(Ub, pa[j], O[2 + j]);
                if (hc == 1)
                    pr[j] = ld(B.R, prm[j]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier_inflight();  // 3: W, U of tokens 0 .. 31
        const u32x4 Woh = E.X[rg][1 - hc][0][l], Wol = E.X[rg][1 - hc][1][l];
        if constexpr (kOut) {
            if (hc == 1) {
                const u32x4 u0 = E.U[rg][l];
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    O[2 + j] = mfma_bf16(u0, pr[j], O[2 + j]);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            S[t] = mfma_bf16(kt[t][1], Woh, S[t]);
            S[t] = mfma_bf16(kt[t][1], Wol, S[t]);
        }
        if constexpr (kOut) {
            // lane (token 16 tt + lr) stores 4 values; rows past the chunk's end fall outside
            // the buffer range
            const auto orsrc = rsrc(obase + c * ostep, (uint32_t)lenc * ost2);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                __builtin_amdgcn_raw_buffer_store_b64(
                    u32x2{pack_bf16x2(O[2 + j][0], O[2 + j][1]), pack_bf16x2(O[2 + j][2], O[2 + j][3])},
                    orsrc, (int)((uint32_t)(16 * (tm + j) + lr) * ost2 + 8u * lg), 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    for (int c = cb; c < ce; c += 2) {
        lds_barrier_inflight();  // chunk c is in BA (the copy wave has waited for it)
        chunk(BA, c);
        if (c + 1 >= ce)
            break;
        lds_barrier_inflight();
        chunk(BB, c + 1);
    }

    if (SEG && kind == kJobResume && !last)
        return;
    if (SEG && kind == kJobIdent) {
        // This wave holds rows k = v0w .. + 15 of M_s for columns j = 64 hc .. + 63: k-chunks
        // cu0 and cu0 + 1 of those rows of M_s^T. Transposed through a per-wave LDS stage
        // (fp32, row j at 64 j bytes) in the M^T area, each unit split into bf16 hi and lo.
        float *stg = (float *)lb_.ml + 1024 * w;
        static_assert(sizeof(lb_.ml) >= 4 * 1024 * 4, "stage must fit");
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                stg[(32 * (t >> 1) + 8 * lg + 4 * (t & 1) + i) * 16 + lr] = S[t][i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        u32x4 *mt = (u32x4 *)(p.seg_mt + ((int64_t)q * p.HV + h) * kSlotFloats);
        const int cu0 = v0w >> 3;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int u = l + 64 * r, jl = u >> 1, c2 = u & 1, j = 64 * hc + jl;
            const f32x4 a = *(const f32x4 *)(stg + 16 * jl + 8 * c2);
            const f32x4 b = *(const f32x4 *)(stg + 16 * jl + 8 * c2 + 4);
            uint32_t h0, l0, h1, l1, h2, l2, h3, l3;
            split2(a[0], a[1], h0, l0);
            split2(a[2], a[3], h1, l1);
            split2(b[0], b[1], h2, l2);
            split2(b[2], b[3], h3, l3);
            const int un = 16 * j + ((cu0 + c2) ^ kswz(j));
            mt[un] = u32x4{h0, h1, h2, h3};
            mt[kMtUnits + un] = u32x4{l0, l1, l2, l3};
        }
        return;
    }
    if (SEG && (kind == kJobZero || (kind == kJobFirst && q >= 0))) {  // R_s or S_in(1)
        float *ip = (float *)seg_img(kind == kJobZero ? p.seg_r : p.seg_sin, q);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            *(f32x4 *)(ip + 256 * t) = S[t];
        return;
    }
    float *np = p.new_state + n * p.ns_sn + h * p.ns_sh + (int64_t)(v0w + lr) * p.ns_sv + 64 * hc + 8 * lg;
#pragma unroll
    for (int t = 0; t < 4; ++t)
        *(f32x4 *)(np + 32 * (t >> 1) + 4 * (t & 1)) = S[t];
}

}  // namespace gdn
