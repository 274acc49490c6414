// Prefill scan on 32x32 tiles: whole sequences, two workgroups per CU.
#include "gdn_prefill.h"

namespace gdn {

// One chunk in LDS, 16-byte units, 80 KB in all: two workgroups fit the 160 KB of a CU.
//   K, Q row t, k-chunk c (8 columns) and V row t, v-chunk c -> unit 16 t + (c ^ wswz(t))
//   record: the record's bytes with each 16x16 block's units (row r, column half h) moved
//           from 2 r + h to 16 h + r (T' hi, T' lo and the gates in T, P' in P)
// Only K is double-buffered: phase (a) of the next chunk needs it at once. V, T' and the
// gates are read before the chunk's second barrier and refilled after it; Q and P' are read
// after that barrier and refilled at the next chunk's first one.

// Swizzle of a row's units. Every read below is conflict-free under the b128 bank model of
// gdn_prefill.h (16 lanes of a 32-lane half with equal parity of lane bits 2, 3, 4): rows in
// either order (lr or vmap(lr)) meet 16 distinct units, rows that differ in bit 4 alone share
// one and never meet. The transposed reads take 64 contiguous bytes of four consecutive rows
// per cycle, which the two low row bits spread over all banks.
__device__ __forceinline__ int wswz(int t) { return ((t & 3) << 2) | ((t >> 2) & 3); }

// Row order of the MFMA tiles: bits 2 and 3 swapped. With A rows in this order a lane's 16
// results (C rows 8 (i / 4) + 4 (l / 32) + i % 4) are rows 16 (i / 8) + 8 (l / 32) + i % 8: two
// runs of eight, each the next MFMA's operand (k = 8 (l / 32) + j) as it stands.
__device__ __forceinline__ int vmap(int m)
{
    return (m & 19) | ((m & 4) << 1) | ((m & 8) >> 1);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The workgroup's 4 waves own 32 state rows each of one (sequence, v-head), all 128 columns
// and all 64 tokens of a chunk, and never exchange state. Per chunk and wave the arithmetic
// of scan_body (gdn_prefill_scan.hip):
//   X = K S0^T, R = V - gamma X, U = T' R, O = scale gamma Q S0^T + P' U,
//   S = gammaC S0 + (dec U)^T K, with S0, R, T' and dec U as bf16 hi + lo.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void
gdn_prefill_scanw_kernel(ScanArgs p)
{
    // (separate objects: the compiler then sees that a copy in flight to one does not alias
    // reads of another, and adds no wait for it)
    __shared__ u32x4 K0[kC * 16], K1[kC * 16], Q[kC * 16], V[kC * 16], T[704], P[320];
    ScanJob job;
    if (!scan_job<8, false>(p, job, blockIdx.x, p.header[p.njob_idx]))
        return;
    const int n = job.n, tok0 = job.tok0, len = job.len, c0 = job.c0;
    const int g = job.grp % p.HQK, h = g * p.ratio + job.wi;
    const int nck = min((len + kC - 1) / kC, max(p.header[0] - c0, 0));

    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63,
              lr = l & 31, hf = l >> 5, pl = l & 15, mh = (l >> 4) & 1;
    const int v0w = 32 * w, tv = vmap(lr);
    const SplitConsts sk = split_consts();

    // ---- copies: 1 KB windows of 64 units; window b of K / Q / V holds rows 4 b .. 4 b + 3.
    // A wave's windows are w + 4 i, so a lane's swizzle does not depend on i.
    const uint32_t kst2 = (uint32_t)p.k_st * 2, qst2 = (uint32_t)p.q_st * 2;
    const uint32_t vst2 = (uint32_t)p.v_st * 2, ost2 = (uint32_t)p.o_st * 2;
    const char *kbase = (const char *)(p.k + (int64_t)tok0 * p.k_st + g * p.k_sh);
    const char *qbase = (const char *)(p.q + (int64_t)tok0 * p.q_st + g * p.q_sh);
    const char *vbase = (const char *)(p.v + (int64_t)tok0 * p.v_st + h * p.v_sh);
    char *obase = (char *)(p.out + (int64_t)tok0 * p.o_st + h * p.o_sh + v0w);
    const int64_t kstep = (int64_t)kC * p.k_st * 2, qstep = (int64_t)kC * p.q_st * 2;
    const int64_t vstep = (int64_t)kC * p.v_st * 2, ostep = (int64_t)kC * p.o_st * 2;
    const char *rbase = p.records + ((int64_t)c0 * p.HV + h) * kRecBytes;
    const int64_t rstep = (int64_t)p.HV * kRecBytes;

    const uint32_t rowt = 4 * w + (l >> 4), cs16 = 16u * ((l & 15) ^ wswz(rowt));
    uint32_t kof = rowt * kst2 + cs16, qof = rowt * qst2 + cs16, vof = rowt * vst2 + cs16;
    uint32_t oof = lr * ost2 + 16 * hf, l16 = 16u * l;
    // record windows hold two blocks each
    const uint32_t rof = 512u * (l >> 5) + 16u * (2 * (l & 15) + ((l >> 4) & 1));

    auto rsrc = [&](const char *base, uint32_t range) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)range, 0x00020000);
    };
    // rows past a chunk's end read as zero: they meet beta = 0 or the causal mask only
    auto rows = [&](int c) { return (uint32_t)(min(kC, len - c * kC) - 1); };
    auto load16 = [&](__amdgpu_buffer_rsrc_t rs, u32x4 *dst, uint32_t off) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (GDN_LDS void *)dst, 16, off, 0, 0, 0);
    };
    // (of: the lane's offset in the wave's first window)
    auto copy_k = [&](u32x4 *K, __amdgpu_buffer_rsrc_t rs, uint32_t of, int i) {
        load16(rs, &K[64 * (w + 4 * i)], of + 16 * i * kst2);
    };
    auto copy_q = [&](__amdgpu_buffer_rsrc_t rs, uint32_t of, int i) {
        load16(rs, &Q[64 * (w + 4 * i)], of + 16 * i * qst2);
    };
    auto copy_v = [&](__amdgpu_buffer_rsrc_t rs, uint32_t of, int i) {
        load16(rs, &V[64 * (w + 4 * i)], of + 16 * i * vst2);
    };
    // record window b (T': 0 .. 9, P': 10 .. 14, gates: 15) to dst
    auto copy_r = [&](__amdgpu_buffer_rsrc_t rs, int b, u32x4 *dst, uint32_t off) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (GDN_LDS void *)dst, 16, off, 1024 * b, 0, 0);
    };
    // T' and the gates: three windows per wave, two for wave 3
    auto copy_t = [&](__amdgpu_buffer_rsrc_t rs, int i) {
        if (i < 2)
            copy_r(rs, w + 4 * i, &T[64 * (w + 4 * i)], rof);
        else if (w < 2)
            copy_r(rs, 8 + w, &T[64 * (8 + w)], rof);
        else if (w == 2)
            copy_r(rs, 15, &T[640], l16);
    };
    auto copy_p = [&](__amdgpu_buffer_rsrc_t rs) {
        copy_r(rs, 10 + w, &P[64 * w], rof);
        if (w == 3)
            copy_r(rs, 14, &P[256], rof);
    };

    // ---- LDS read offsets (bytes)
    const char *Vb = (const char *)V, *Qb = (const char *)Q, *Tb = (const char *)T,
               *Pb = (const char *)P;
    // K rows of (a) and Q rows of (e): k-step ks at offset ^ 32 ks
    uint32_t kA = 16u * (16 * tv + (hf ^ wswz(tv))), qA = 16u * (16 * lr + (hf ^ wswz(lr)));
    // transposed reads: four tokens 8 hf + 4 x .. + 3, columns 16 mh + 8 (pl & 1) + 4 (pl / 2 % 2)
    auto trow = [&](int x) { return 8 * hf + 4 * x + (pl >> 2); };
    uint32_t kT[2];  // columns + 32 kt at offset ^ 64 kt; V: columns 32 w
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        kT[x] = 256u * trow(x) + 16u * ((2 * mh + (pl & 1)) ^ wswz(trow(x))) + 8u * ((pl >> 1) & 1);
    }
    // T' / P' operand of tile tt, k-step ks: block (2 tt + lr / 16, ks). Rows of an absent
    // block read the record's zero bytes behind the gates (T') or are masked (P').
    const int hi16 = lr >> 4;
    constexpr uint32_t kG = 10240, kZero = kG + kRecZero - kRecGates;  // in T
    const uint32_t tl = 16u * (16 * hf + (tv & 15));
    uint32_t pof = 16u * (16 * hf + (lr & 15));
    uint32_t t0 = tl + 512u * hi16, t1 = tl + 512u * (3 + 3 * hi16);
    auto ld = [](const char *b, uint32_t off) { return *(const u32x4 *)(b + off); };
    auto tRead = [&](int tt, int ks, u32x4 &th, u32x4 &tlo) {
        const uint32_t o = tt == 0 ? t0 + 512 * ks : t1 + 512 * ks;
        if (ks == 2 * tt + 1) {
            th = ld(Tb, hi16 ? o : kZero);
            tlo = ld(Tb, hi16 ? o + kRecTlo : kZero);
        } else {
            th = ld(Tb, o);
            tlo = ld(Tb, o + kRecTlo);
        }
    };
    auto pRead = [&](int tt, int ks) {
        const uint32_t b = tt == 0 ? (hi16 ? 512 : 0) : (hi16 ? 3072 : 1536);
        u32x4 x = ld(Pb, pof + b + 512 * ks);
        if (ks == 2 * tt + 1)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                x[e] = hi16 ? x[e] : 0u;
        return x;
    };
    // gates: eight values of tokens 16 ks + 8 hf .. (area 0: gamma, 256: dec), and scale gamma
    // of token 32 tt + lr
    auto gLoad = [&](int ks, int area, f32x4 *dst) {
        const uint32_t o = kG + ((l16 >> 4) & 32) + area + 64 * ks;
        dst[0] = *(const f32x4 *)(Tb + o);
        dst[1] = *(const f32x4 *)(Tb + o + 16);
    };
    auto sgLoad = [&](int tt) {
        return *(const float *)(Tb + kG + 512 + ((l16 >> 2) & 124) + 128 * tt);
    };

    if (nck > 0) {
        const uint32_t r0 = rows(0);
        const auto rk = rsrc(kbase, r0 * kst2 + 256u), rv = rsrc(vbase, r0 * vst2 + 256u),
                   rr = rsrc(rbase, kRecBytes);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            copy_k(K0, rk, kof, i);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            copy_v(rv, vof, i);
#pragma unroll
        for (int i = 0; i < 3; ++i)
            copy_t(rr, i);
    }

    // ---- state: S[kt][8 s + j] holds S[v0w + tv][32 kt + 16 s + 8 hf + j]
    f32x16 S[4];
    if (p.state) {
        const float *sp = p.state + n * p.st_sn + h * p.st_sh + (int64_t)(v0w + tv) * p.st_sv + 8 * hf;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const f32x4 x = *(const f32x4 *)(sp + 32 * kt + 16 * (u >> 1) + 4 * (u & 1));
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    S[kt][4 * u + e] = x[e];
            }
    } else {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                S[kt][i] = 0.f;
    }

    // eight values 8 s .. 8 s + 7 of a tile as one MFMA operand, hi + lo
    auto split8 = [&](const float *x, u32x4 &hi, u32x4 &lo) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t hh, ll;
            split_bf16x2(x[2 * e], x[2 * e + 1], hh, ll, sk);
            hi[e] = hh;
            lo[e] = ll;
        }
    };
    constexpr f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                               0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // Operand reads run one region ahead of the MFMAs that consume them; the scheduling
    // barriers between regions keep them there (and bound the registers).
#define GDN_REGION() __builtin_amdgcn_sched_barrier(0)

    auto chunk = [&](const u32x4 *Kc, u32x4 *Kn, int c, bool more) {
        const char *Kb = (const char *)Kc;
        // re-derived per chunk: hoisted out of the loop, each k-step's offset would hold a
        // register of its own
        asm volatile("" : "+v"(kA), "+v"(qA), "+v"(kT[0]), "+v"(kT[1]), "+v"(kof), "+v"(qof), "+v"(vof),
                     "+v"(oof), "+v"(pof), "+v"(t0), "+v"(t1), "+v"(l16));
        const auto rq = rsrc(qbase + c * qstep, rows(c) * qst2 + 256u);
        const auto rr = rsrc(rbase + c * rstep, kRecBytes);
        // after the last chunk the next one's copies have empty ranges: they write zeros that
        // nothing reads, and every wait below counts the same operations
        const int cn = more ? c + 1 : c;
        const auto rk = rsrc(kbase + cn * kstep, more ? rows(cn) * kst2 + 256u : 0);

        // (a) X = K S0^T, S0 as hi + lo; S is scaled by gammaC as its split is taken (the
        // residuals are formed in S0's registers)
        f32x16 X[2];
        u32x4 Sh[8], Sl[2], Rh[4], Rl[4];
        u32x2 vv[8];
        u32x4 ka[2][2];
        const float gC = *(const float *)(Tb + kG + 768);
        auto kRead = [&](int ks, u32x4 *dst) {
            dst[0] = ld(Kb, kA ^ (32 * ks));
            dst[1] = ld(Kb, (kA ^ (32 * ks)) + 8192);
        };
        auto split_s = [&](int ks) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x[j] = S[ks >> 1][8 * (ks & 1) + j];
                S[ks >> 1][8 * (ks & 1) + j] = gC * x[j];
            }
            split8(x, Sh[ks], Sl[ks & 1]);
        };
        auto vRead = [&](int ks) {  // tokens 16 ks + 8 hf ..
            vv[2 * ks] = lds_tr16(Vb + (kT[0] ^ (64 * w)) + 4096 * ks);
            vv[2 * ks + 1] = lds_tr16(Vb + (kT[1] ^ (64 * w)) + 4096 * ks);
        };
        auto rForm = [&](int ks) {
            f32x4 gm[2];
            gLoad(ks, 0, gm);
            float r[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const u32x2 v2 = vv[2 * ks + (j >> 2)];
                const uint32_t vw = v2[(j >> 1) & 1];
                r[j] = fmaf(-gm[j >> 2][j & 3], X[ks >> 1][8 * (ks & 1) + j],
                            j & 1 ? bf16hi(vw) : bf16lo(vw));
            }
            split8(r, Rh[ks], Rl[ks]);
        };
        kRead(0, ka[0]);
        split_s(0);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            GDN_REGION();
            if (ks < 7) {
                kRead(ks + 1, ka[(ks + 1) & 1]);
                split_s(ks + 1);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    vRead(i);
            }
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
                X[tt] = mfma32(ka[ks & 1][tt], Sh[ks], ks == 0 ? zero16 : X[tt]);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
                X[tt] = mfma32(ka[ks & 1][tt], Sl[ks & 1], X[tt]);
            // Q and P' of this chunk, then K of the next
            if (ks < 4)
                copy_q(rq, qof, ks);
            else
                copy_k(Kn, rk, kof, ks - 4);
            if (ks == 3)
                copy_p(rr);
        }
        GDN_REGION();
        // (b) R = V - gamma X
        u32x4 tA[2][2];
        tRead(0, 0, tA[0][0], tA[0][1]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            rForm(ks);
        // (c) U = T' R
        f32x16 U[2];
#pragma unroll
        for (int it = 0; it < 6; ++it) {  // (tile, k-step) = (0, 0 .. 1), (1, 0 .. 3)
            const int tt = it >= 2, ks = tt ? it - 2 : it, cb = it & 1;
            GDN_REGION();
            if (it < 5)
                tRead(it >= 1, it >= 1 ? it - 1 : 1, tA[cb ^ 1][0], tA[cb ^ 1][1]);
            U[tt] = mfma32(tA[cb][0], Rh[ks], ks == 0 ? zero16 : U[tt]);
            U[tt] = mfma32(tA[cb][0], Rl[ks], U[tt]);
            U[tt] = mfma32(tA[cb][1], Rh[ks], U[tt]);
        }
        GDN_REGION();
        // (d) W = dec U (hi + lo) for the state update, U (bf16) for the readout
        u32x4 Wh[4], Wl[4], Ub[4];
        auto wForm = [&](int ks, const f32x4 *dec) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                Ub[ks][e] = pack_bf16x2(U[ks >> 1][8 * (ks & 1) + 2 * e], U[ks >> 1][8 * (ks & 1) + 2 * e + 1]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[j] = dec[j >> 2][j & 3] * U[ks >> 1][8 * (ks & 1) + j];
            split8(x, Wh[ks], Wl[ks]);
        };
        f32x4 dec[4][2];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            gLoad(ks, 256, dec[ks]);
        wForm(0, dec[0]);
        wForm(1, dec[1]);
        float sg[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
            sg[tt] = sgLoad(tt);

        // Second barrier: every wave is done with V, T' and the gates, and Q and P' are in
        // (the next chunk's four K copies, issued after them, stay in flight).
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0074);  // vmcnt(4) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const auto rv = rsrc(vbase + cn * vstep, more ? rows(cn) * vst2 + 256u : 0);
        const auto rn = rsrc(rbase + cn * rstep, more ? kRecBytes : 0);

        // (e) O^T = scale gamma S0 Q^T + U^T P'^T; lane (token 32 tt + lr) stores two runs of
        // eight values. Rows past the chunk's end fall outside the buffer range.
        const auto orsrc = rsrc(obase + c * ostep, (rows(c) + 1) * ost2);
        u32x4 qv[2][2];
        auto qRead = [&](int st) {  // k-steps 2 (st % 4), + 1 of tile st / 4
#pragma unroll
            for (int i = 0; i < 2; ++i)
                qv[st & 1][i] = ld(Qb, (qA ^ (64 * (st & 3) + 32 * i)) + 8192 * (st >> 2));
        };
        auto ktRead = [&](int kt, int ks) {
            const u32x2 k0 = lds_tr16(Kb + (kT[0] ^ (64 * kt)) + 4096 * ks),
                        k1 = lds_tr16(Kb + (kT[1] ^ (64 * kt)) + 4096 * ks);
            return u32x4{k0[0], k0[1], k1[0], k1[1]};
        };
        auto store_o = [&](int tt, const f32x16 &O) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = pack_bf16x2(O[8 * s + 2 * e], O[8 * s + 2 * e + 1]);
                __builtin_amdgcn_raw_buffer_store_b128(o, orsrc, (int)(oof + 32 * tt * ost2 + 32 * s),
                                                       0, 0);
            }
        };
        f32x16 O[2];
        u32x4 pv[4], kt[2][4];
        qRead(0);
#pragma unroll
        for (int st = 0; st < 8; ++st) {
            const int tt = st >> 2;
            GDN_REGION();
            if (st < 7)
                qRead(st + 1);
#pragma unroll
            for (int i = 0; i < 2; ++i)
                O[tt] = mfma32(Sh[2 * (st & 3) + i], qv[st & 1][i],
                               (st & 3) + i == 0 ? zero16 : O[tt]);
            // the next chunk's V, T' and gates, all before the first output store
            if (st < 4)
                copy_v(rv, vof, st);
            else if (st < 6)
                copy_t(rn, st - 4);
            if (st == 0 || st == 2)
                wForm(2 + (st >> 1), dec[2 + (st >> 1)]);
            if (st == 3 || st == 7)
#pragma unroll
                for (int ks = 0; ks < 2 + 2 * tt; ++ks)
                    pv[ks] = pRead(tt, ks);
            if (st == 4) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    O[0][i] *= sg[0];
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
                    O[0] = mfma32(Ub[ks], pv[ks], O[0]);
            }
        }
        GDN_REGION();
        copy_t(rn, 2);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            O[1][i] *= sg[1];
        store_o(0, O[0]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            kt[0][ks] = ktRead(0, ks);
        GDN_REGION();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            O[1] = mfma32(Ub[ks], pv[ks], O[1]);

        // (f) S = gammaC S0 + W^T K
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) {
            GDN_REGION();
            if (k4 < 3)
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    kt[(k4 + 1) & 1][ks] = ktRead(k4 + 1, ks);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                S[k4] = mfma32(kt[k4 & 1][ks], Wh[ks], S[k4]);
                S[k4] = mfma32(kt[k4 & 1][ks], Wl[ks], S[k4]);
            }
            if (k4 == 0)
                store_o(1, O[1]);
        }
        GDN_REGION();
    };

    // The first barrier of a chunk: K, V, T' and the gates are in, every wave is done with
    // the chunk before. After the first chunk exactly four younger operations, the previous
    // chunk's output stores, may stay in flight.
    auto chunk_barrier = [&](bool first) {
        asm volatile("" ::: "memory");
        if (first)
            __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
        else
            __builtin_amdgcn_s_waitcnt(0x0074);  // vmcnt(4) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    for (int c = 0; c < nck; c += 2) {
        chunk_barrier(c == 0);
        chunk(K0, K1, c, c + 1 < nck);
        if (c + 1 >= nck)
            break;
        chunk_barrier(false);
        chunk(K1, K0, c + 1, c + 2 < nck);
    }
#undef GDN_REGION
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no copy outlives the workgroup's LDS

    float *np = p.new_state + n * p.ns_sn + h * p.ns_sh + (int64_t)(v0w + tv) * p.ns_sv + 8 * hf;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *(f32x4 *)(np + 32 * kt + 16 * (u >> 1) + 4 * (u & 1)) =
                f32x4{S[kt][4 * u], S[kt][4 * u + 1], S[kt][4 * u + 2], S[kt][4 * u + 3]};
}

}  // namespace gdn
