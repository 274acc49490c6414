// Prefill host side: workspace layout and the launches behind gdn_prefill_launch
// (plan, prep, then one scan launch, or two over segment job tables).
#include "gdn_prefill.h"

#include <algorithm>
#include <cmath>

// ------------------------------------------------------------------------- host side
namespace {

constexpr int64_t kChunkH = 64;
constexpr int kZeroFillBlocks = 64;

int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

int64_t max_chunks(int64_t T, int64_t N) { return (T + kChunkH - 1) / kChunkH + N; }

// Segments per sequence at most (the default variant only; 1: none). Segments scan a sequence's
// parts side by side at the price of a second pass (its launch, state and first chunk: ~14 k
// cycles) and of state maps on more CUs, whose scan may be a slower one. The largest count is
// bounded by pass A's jobs, N HV (2 G - 3), at one workgroup per CU; G = 2 would scan its halves
// one after the other.
//
// One sequence of c chunks: the G with the smallest modelled time, both passes taking the
// planner's base(G) = (c + h (G - 1) (G - 2)) / (w + G - 1) chunks, against c chunks whole.
// Whole prefills, as many segments as pass A holds -> this rule: at 8 v-heads 1 x 4096 64.1 ->
// 51.1 us (9 segments; 5 59.4), 1 x 8192 90.5 -> 74.8 (9), 1 x 16384 131.3 -> 128.5 (9; 12 136.0);
// at 32 v-heads 1 x 800 33.9 -> 32.5 (whole), 1 x 1200 47.7 -> 42.1 (3), 1 x 1600 52.4 -> 48.8
// (3), 1 x 4096 90 (5; 3 is 4 % slower); at 48 1 x 8192 262 -> 235 and 1 x
// 16000 536 -> 440 (whole -> 4), at 64 1 x 12000 421 -> 390 (whole -> 3).
//
// More sequences: only the device knows their lengths. It weighs its plan against scanning every
// sequence whole (plan_jobs); what is decided here is whether it may cut, since a pass A without
// a job costs ~1.7 us. The most there is to gain is one sequence of all T tokens among empty
// ones, the most to lose that launch in a batch of equal lengths: segments where the first, as
// a share of its call, is at least kSegOdds times the second. Whole prefills, every sequence
// whole below a mean length -> this rule: 1980 + 20 tokens at 8 v-heads 59.8 -> 39.5 us, 2400 + 3
// of 20 70.2 -> 45.0, 6000 + 5 of 100 155.5 -> 90.8, 15000 + 9 of 200 380 -> 260, 3000 + 20 at
// 32 89.9 -> 72.4, 1500 + 300 at 16 49.2 -> 37.0; with nothing to cut 6 of 1000 at 8 40.0 ->
// 41.8, 2048 + 1100 at 32 69.1 -> 71.1, and 3 of 700 at 8, offered for what 2100 tokens in one
// sequence would gain, 28.9 -> 30.8. (8 of 64 to 1024 at 8 are not offered: 36.4.)
constexpr double kSegOdds = 3.75;
constexpr double kCallRest = 45.0;  // k cycles of a call besides its chunks (prep, starts)

// (cached: chunk times as if everything stayed in the cache; see prefill_launch)
int seg_count(int64_t T, int64_t N, int64_t HV, bool cached)
{
    // (the job planner runs one sequence per lane in the self-planned prep kernel)
    if (T <= 0 || N <= 0 || N > gdn::kSegSeqMax || N * HV * 3 > 256)
        return 1;
    const int64_t cmax = (T + kChunkH - 1) / kChunkH;  // no sequence has more chunks
    const double w = gdn::kSegFirstWeight, h = 0.5 * gdn::kSegChainChunks;
    const double whole = cmax * gdn::whole_chunk_cost(N * HV, cached ? 0.f : (float)(cmax * HV));
    // the planner cuts c chunks into at most G*(c) segments, its closed-form optimum (rising with
    // c; +1 for the device's float rounding): capacities sized for that are tight
    const int64_t gs = (int64_t)(1.0 - w + std::sqrt(w * w + w + (double)cmax / h)) + 1;
    int64_t G = 1;
    double best = whole;
    for (int64_t g = 3; g <= gdn::kSegMaxG && N * HV * (2 * g - 3) <= 256 && g <= cmax / gdn::kSegMinChunks; ++g) {
        if (N > 1 && g > gs)
            break;
        const double base = (cmax + h * (g - 1) * (g - 2)) / (w + g - 1);
        const double cost = base * (w * gdn::chunk_cost(HV * (2 * g - 3 + N - 1)) + gdn::chunk_cost(HV * (g - 1))) +
                            gdn::kSegPassCost;
        if (cost < best || N > 1) {
            best = cost;
            G = g;
        }
    }
    if (N > 1 && (whole - best) * (whole / N + kCallRest) < kSegOdds * gdn::kSegEmptyPass * (whole + kCallRest))
        return 1;
    return G >= 3 ? (int)G : 1;
}

struct Layout {
    int64_t nc;
    int64_t header, chunk_tok0, chunk_len, seq_rank, records, total;
    int G;                // segments per sequence at most (1: none)
    int64_t capA, capC;   // pass A / pass C job capacity
    int64_t jobs, seg_sin, seg_r, seg_mt;
};

Layout layout(int64_t T, int64_t N, int64_t HV, bool cached)
{
    Layout L;
    L.G = seg_count(T, N, HV, cached);
    L.capA = N * (2 * L.G - 3);
    L.capC = N * (L.G - 1);
    L.nc = max_chunks(T, N);
    int64_t o = 0;
    L.header = o;
    o += 64 * 4;
    L.chunk_tok0 = o;
    o += L.nc * 4;
    L.chunk_len = o;
    o += L.nc * 4;
    L.seq_rank = (o + 15) & ~int64_t(15);
    o = L.seq_rank + N * 16;
    L.records = align256(o);
    o = L.records + L.nc * HV * gdn::kRecBytes;
    L.jobs = L.seg_sin = L.seg_r = L.seg_mt = 0;
    if (L.G > 1) {
        const int64_t slot_bytes = N * (L.G - 1) * HV * gdn::kSlotFloats * 4;
        L.jobs = align256(o);
        o = L.jobs + (L.capA + L.capC) * gdn::kJobInts * 4;
        L.seg_sin = align256(o);
        L.seg_r = L.seg_sin + slot_bytes;
        L.seg_mt = L.seg_r + slot_bytes;
        o = L.seg_mt + slot_bytes;
    }
    L.total = o;
    return L;
}

bool aligned(const void *p, uintptr_t n) { return ((uintptr_t)p % n) == 0; }

// Compute units of the device that owns the stream (the current device when the
// stream is the null stream); 256 if the runtime cannot tell.
int num_cus(hipStream_t st)
{
    int dev = -1;
    if (st == nullptr || hipStreamGetDevice(st, &dev) != hipSuccess)
        if (hipGetDevice(&dev) != hipSuccess)
            return 256;
    static int cached[64] = {0};
    if (dev < 0 || dev >= 64)
        return 256;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

}  // namespace

extern "C" int64_t gdn_prefill_workspace_size(int32_t total_tokens, int32_t num_seqs,
                                              int32_t num_qk_heads, int32_t num_v_heads,
                                              int32_t head_size)
{
    gdn_begin_call();
    if (total_tokens < 0 || num_seqs < 0 || num_qk_heads <= 0 || num_v_heads <= 0 ||
        num_v_heads % num_qk_heads != 0 || head_size != 128)
        return gdn_set_error(GDN_EINVAL, "gdn_prefill_workspace_size: bad sizes T=%d N=%d "
                             "HQK=%d HV=%d D=%d", total_tokens, num_seqs, num_qk_heads,
                             num_v_heads, head_size);
    return layout(total_tokens, num_seqs, num_v_heads, false).total;
}

int64_t gdn::prefill_workspace_cached(int64_t T, int64_t N, int64_t HV)
{
    return layout(T, N, HV, true).total;
}

extern "C" int gdn_prefill_launch(const gdn_prefill_params *p, void *stream)
{
    return gdn::prefill_launch(p, stream, false);
}

int gdn::prefill_launch(const gdn_prefill_params *p, void *stream, bool cached)
{
    gdn_begin_call();
    if (!p || p->struct_size != (int32_t)sizeof(gdn_prefill_params))
        return gdn_set_error(GDN_EINVAL, "gdn_prefill: params NULL or struct_size mismatch");
    const int T = p->total_tokens, N = p->num_seqs, HQK = p->num_qk_heads,
              HV = p->num_v_heads, D = p->head_size;
    if (T < 0 || N < 0 || HQK <= 0 || HV <= 0 || HV % HQK != 0)
        return gdn_set_error(GDN_EINVAL, "gdn_prefill: bad sizes T=%d N=%d HQK=%d HV=%d", T, N,
                             HQK, HV);
    if (D != 128)
        return gdn_set_error(GDN_EINVAL, "gdn_prefill: head_size %d unsupported (128 only)", D);
    if (p->variant < 0 || p->variant > 2)
        return gdn_set_error(GDN_EINVAL, "gdn_prefill: variant %d unknown (0, 1, 2)", p->variant);
    if (!p->q || !p->k || !p->v || !p->A_log || !p->a || !p->dt_bias || !p->b ||
        !p->cu_seqlens || !p->output || !p->new_state)
        return gdn_set_error(GDN_EINVAL, "gdn_prefill: NULL tensor pointer");
    if (p->q_stride[2] != 1 || p->k_stride[2] != 1 || p->v_stride[2] != 1 ||
        p->output_stride[2] != 1 || p->new_state_stride[3] != 1 ||
        (p->state && p->state_stride[3] != 1))
        return gdn_set_error(GDN_ELAYOUT, "gdn_prefill: innermost stride must be 1");
    for (int i = 0; i < 2; ++i)
        if (p->q_stride[i] % 8 || p->k_stride[i] % 8 || p->output_stride[i] % 8)
            return gdn_set_error(GDN_ELAYOUT,
                                 "gdn_prefill: q/k/output strides must be multiples of 8");
    for (int i = 0; i < 2; ++i)
        if (p->v_stride[i] % 8)
            return gdn_set_error(GDN_ELAYOUT, "gdn_prefill: v strides must be multiples of 8");
    if (!aligned(p->q, 16) || !aligned(p->k, 16) || !aligned(p->v, 16) || !aligned(p->output, 16))
        return gdn_set_error(GDN_ELAYOUT, "gdn_prefill: q/k/v/output must be 16-byte aligned");
    for (int i = 0; i < 3; ++i)
        if (p->new_state_stride[i] % 4 || (p->state && p->state_stride[i] % 4))
            return gdn_set_error(GDN_ELAYOUT,
                                 "gdn_prefill: state strides must be multiples of 4");
    if (!aligned(p->new_state, 16) || (p->state && !aligned(p->state, 16)))
        return gdn_set_error(GDN_ELAYOUT, "gdn_prefill: state must be 16-byte aligned");
    // the kernels address a 64-token chunk with 32-bit byte offsets
    const int64_t kMaxStride = int64_t(1) << 24;
    for (int i = 0; i < 2; ++i)
        if (p->q_stride[i] >= kMaxStride || p->k_stride[i] >= kMaxStride ||
            p->v_stride[i] >= kMaxStride || p->output_stride[i] >= kMaxStride ||
            p->q_stride[i] < 0 || p->k_stride[i] < 0 || p->v_stride[i] < 0 ||
            p->output_stride[i] < 0)
            return gdn_set_error(GDN_ELAYOUT,
                                 "gdn_prefill: token / head strides must be in [0, 2^24)");
    const int64_t kMaxGateStride = int64_t(1) << 31;
    for (int i = 0; i < 2; ++i)
        if (p->a_stride[i] < 0 || p->a_stride[i] >= kMaxGateStride || p->b_stride[i] < 0 ||
            p->b_stride[i] >= kMaxGateStride)
            return gdn_set_error(GDN_ELAYOUT, "gdn_prefill: a / b strides must be in [0, 2^31)");
    if (p->A_log_stride < 0 || p->A_log_stride >= kMaxGateStride || p->dt_bias_stride < 0 ||
        p->dt_bias_stride >= kMaxGateStride)
        return gdn_set_error(GDN_ELAYOUT, "gdn_prefill: A_log / dt_bias strides must be in [0, 2^31)");
    const Layout L = layout(T, N, HV, cached);
    if (L.nc > 0x7fffffff)
        return gdn_set_error(GDN_EINVAL, "gdn_prefill: too many chunks");
    if (!p->workspace || p->workspace_bytes < L.total || !aligned(p->workspace, 256))
        return gdn_set_error(GDN_EWORKSPACE,
                             "gdn_prefill: workspace needs %lld bytes, 256-byte aligned "
                             "(got %lld at %p)", (long long)L.total,
                             (long long)p->workspace_bytes, p->workspace);
    if (p->state && (const void *)p->state == (const void *)p->new_state)
        for (int i = 0; i < 4; ++i)
            if (p->state_stride[i] != p->new_state_stride[i])
                return gdn_set_error(GDN_ELAYOUT,
                                     "gdn_prefill: in-place state needs identical strides");

    hipStream_t st = (hipStream_t)stream;
    char *ws = (char *)p->workspace;
    const int ratio = HV / HQK;
    const int HO = HV;  // max(HQK, HV) with HV a multiple of HQK

    gdn::PlanArgs pa;
    pa.cu = p->cu_seqlens;
    pa.cu64 = p->cu_seqlens_int64 ? 1 : 0;
    pa.N = N;
    pa.T = T;
    pa.HO = HO;
    pa.nc = (int)L.nc;
    pa.header = (int32_t *)(ws + L.header);
    pa.chunk_tok0 = (int32_t *)(ws + L.chunk_tok0);
    pa.chunk_len = (int32_t *)(ws + L.chunk_len);
    pa.seq_rank = (int32_t *)(ws + L.seq_rank);
    pa.out = (gdn::bf16_t *)p->output;
    pa.o_st = p->output_stride[0];
    pa.o_sh = p->output_stride[1];
    // segments only for the default variant (the tuning variants keep whole sequences)
    const int G = p->variant == 0 ? L.G : 1;
    // Whole sequences: 4 scan waves per workgroup (two workgroups per (sequence, v-head))
    // when there are at most 128 (sequence, v-head) pairs, else 8 (129 to 256 pairs: the
    // device picks, whole_dual below). Variants: 1 forces 4 waves, 2 forces 8.
    const bool nw4 = p->variant == 1 || (p->variant == 0 && (int64_t)N * HV <= gdn::kPairs4);
    pa.seg_G = G;
    pa.seg_capA = (int)L.capA;
    pa.jobs = G > 1 ? (int32_t *)(ws + L.jobs) : nullptr;
    // Up to 126 sequences the prep kernel plans for itself (one dependent launch fewer: the
    // plan kernel's 5 to 6 us sat on the critical path, mostly cu_seqlens load latency; 100
    // sequences of 1 to 130 at 32 v-heads 179.1 -> 176.8 us, 100 of 64 to 160 at 8 78.2 -> 74.2).
    const bool prep_runs = L.nc > 0 && T > 0;
    const bool self_plan = prep_runs && N >= 1 && N <= gdn::kSelfPlanMax;
    // Whole sequences, 129 to 256 (sequence, v-head) pairs: either width of the scan can be the
    // faster, depending on the longest sequence, which only the device knows: the self-planning
    // prep kernel chooses. Above 256 pairs the 8-wave scan alone (the 4-wave one rarely wins
    // there), or the wide one below.
    const bool whole_dual = G == 1 && p->variant == 0 && self_plan && N <= gdn::kSegSeqMax && (int64_t)N * HV > gdn::kPairs4 &&
                            (int64_t)N * HV <= 256;
    // With three (sequence, v-head) pairs per CU and more, of at most six chunks on average, a
    // pair's start and end (state and first chunk in, state out) weigh as much as its chunks:
    // the wide scan, whose two workgroups per CU cover one another's. Measured on MI355X, 8-wave
    // against wide scan, whole prefill: 100 sequences of 1 to 130 tokens at 32 v-heads 205 ->
    // 181 us, 64 of 128 162 -> 145, 40 of 64 to 200 108 -> 100, 24 of 1 to 100 56 -> 51, 100 of
    // 64 to 256 at 8 v-heads 97 -> 91. Fewer pairs gain nothing (20 of 300 to 500 at 32 v-heads
    // 114.5 -> 115.5, 16 of 64 to 1024 124 -> 128: two long jobs share a CU's time), nor do
    // longer sequences (32 of 512 209 -> 212, 64 of 1000 728 -> 743). A long sequence among the
    // short ones, which only the device knows of, makes the planner take the 8-wave scan after
    // all (choose_wide).
    const bool wide = G == 1 && p->variant == 0 && (int64_t)N * HV >= 3 * (int64_t)num_cus(st) &&
                      T <= 384 * (int64_t)N;
    pa.whole_cus = whole_dual ? num_cus(st) : 0;
    pa.wide_cus = wide ? num_cus(st) : 0;
    gdn_begin_launches();
    int rc = 0;
    if (!self_plan) {
        hipLaunchKernelGGL(gdn::gdn_prefill_plan_kernel, dim3(1 + kZeroFillBlocks), dim3(256),
                           0, st, pa);
        rc = gdn_check_launch("gdn_prefill_plan_kernel");
        if (rc)
            return rc;
    }

    if (prep_runs) {
        gdn::PrepArgs qa;
        qa.q = (const gdn::bf16_t *)p->q;
        qa.k = (const gdn::bf16_t *)p->k;
        qa.a = (const gdn::bf16_t *)p->a;
        qa.b = (const gdn::bf16_t *)p->b;
        qa.A_log = p->A_log;
        qa.dt_bias = p->dt_bias;
        qa.q_st = (int32_t)p->q_stride[0];
        qa.q_sh = (int32_t)p->q_stride[1];
        qa.k_st = (int32_t)p->k_stride[0];
        qa.k_sh = (int32_t)p->k_stride[1];
        qa.a_st = (int32_t)p->a_stride[0];
        qa.a_sh = (int32_t)p->a_stride[1];
        qa.b_st = (int32_t)p->b_stride[0];
        qa.b_sh = (int32_t)p->b_stride[1];
        qa.A_log_s = (int32_t)p->A_log_stride;
        qa.dt_s = (int32_t)p->dt_bias_stride;
        qa.header = pa.header;
        qa.chunk_tok0 = pa.chunk_tok0;
        qa.chunk_len = pa.chunk_len;
        qa.records = ws + L.records;
        qa.HQK = HQK;
        qa.HV = HV;
        qa.ratio = ratio;
        qa.scale = p->scale;
        qa.self_plan = self_plan ? 1 : 0;
        qa.plan = pa;
        // persistent: two workgroups per CU walk the (chunk, q/k head, v-head pair) units. While
        // single v-head units find a CU each, those, so that a unit's waves have a SIMD each
        // (MI355X, whole prefill: 1 x 300 at 32 v-heads 20.5 -> 20.1 us, 3 x 100 17.0 -> 16.6;
        // the prep kernel alone 7.4 -> 6.5, and 9.9 -> 10.8 where two of them share a CU).
        const int cus = num_cus(st), vh = ratio % 2 == 0 && L.nc * HV > cus ? 2 : 1;
        // One sequence scanned whole: every unit of q/k head g on the scan's XCD (1 x 77 at 4
        // q/k heads 14.7 -> 14.4 us, 1 x 700 29.2 -> 28.5).
        qa.gpad = N == 1 && G == 1 && HQK < 8 && 8 % HQK == 0 && L.nc * 8 * (ratio / vh) <= 2 * cus ? 8 : HQK;
        const int64_t units = L.nc * qa.gpad * (ratio / vh);
        const int64_t blocks = std::min<int64_t>(units, 2 * (int64_t)cus);
        if (blocks > 0x7fffffff)
            return gdn_set_error(GDN_EINVAL, "gdn_prefill: grid too large");
        if (vh == 2)
            hipLaunchKernelGGL(gdn::gdn_prefill_prep2_kernel, dim3((unsigned)blocks), dim3(512), 0,
                               st, qa);
        else
            hipLaunchKernelGGL(gdn::gdn_prefill_prep1_kernel, dim3((unsigned)blocks), dim3(256), 0,
                               st, qa);
        rc = gdn_check_launch("gdn_prefill_prep_kernel");
        if (rc)
            return rc;
    }

    if (N > 0) {
        gdn::ScanArgs sa;
        sa.q = (const gdn::bf16_t *)p->q;
        sa.k = (const gdn::bf16_t *)p->k;
        sa.v = (const gdn::bf16_t *)p->v;
        sa.state = p->state;
        sa.new_state = p->new_state;
        sa.out = (gdn::bf16_t *)p->output;
        sa.q_st = p->q_stride[0];
        sa.q_sh = p->q_stride[1];
        sa.k_st = p->k_stride[0];
        sa.k_sh = p->k_stride[1];
        sa.v_st = p->v_stride[0];
        sa.v_sh = p->v_stride[1];
        sa.o_st = p->output_stride[0];
        sa.o_sh = p->output_stride[1];
        sa.st_sn = p->state_stride[0];
        sa.st_sh = p->state_stride[1];
        sa.st_sv = p->state_stride[2];
        sa.ns_sn = p->new_state_stride[0];
        sa.ns_sh = p->new_state_stride[1];
        sa.ns_sv = p->new_state_stride[2];
        sa.header = pa.header;
        sa.seq_rank = pa.seq_rank;
        sa.records = ws + L.records;
        sa.HQK = HQK;
        sa.HV = HV;
        sa.ratio = ratio;
        sa.jobs = nullptr;
        sa.job_first = 0;
        sa.njob_idx = 0;
        sa.queue = pa.header + gdn::kQueueIdx;
        sa.seg_sin = G > 1 ? (float *)(ws + L.seg_sin) : nullptr;
        sa.seg_r = G > 1 ? (float *)(ws + L.seg_r) : nullptr;
        sa.seg_mt = G > 1 ? (float *)(ws + L.seg_mt) : nullptr;
        // 8 waves per workgroup = one (sequence, v-head) each, two waves per SIMD; with few
        // (sequence, v-head) pairs, 4 waves and two workgroups per pair (or four, where that still
        // fits one per CU: column-split bodies) spread the state rows over more CUs. (sequence or
        // job, q/k head) groups go to the XCDs in turn.
        const int64_t cus = num_cus(st);
        sa.split_groups = (int)(8 * (cus / (32 * (int64_t)ratio)));
        auto blocks_of = [&](int64_t groups, int tph) { return 8 * ((int64_t)tph * ratio) * ((groups + 7) / 8); };
        auto launch = [&](void (*kernel)(gdn::ScanArgs), int64_t units, int64_t blocks, int threads) {
            const int64_t ngroups = units * HQK;
            sa.ngroups = (int)ngroups;
            if (ngroups > 0x7fffffff || blocks > 0x7fffffff)
                return gdn_set_error(GDN_EINVAL, "gdn_prefill: grid too large");
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), 0, st, sa);
            return gdn_check_launch("gdn_prefill_scan_kernel");
        };
        // one pass over the segment jobs, as many as `units`: the grid holds every form that a
        // job count may call for
        auto pass = [&](int64_t units) {
            const int64_t groups = units * HQK, g4 = std::min<int64_t>(units, gdn::kPairs4 / HV) * HQK;
            return launch(gdn::gdn_prefill_scan_any_kernel<true>, units,
                          std::max({blocks_of(groups, 1), blocks_of(g4, 2),
                                    blocks_of(std::min<int64_t>(groups, sa.split_groups), 4)}), 512);
        };
        const int64_t groups = (int64_t)N * HQK;
        if (G > 1) {
            // pass A: segment 0 of every sequence and both state maps of the middle segments
            sa.jobs = pa.jobs;
            sa.job_first = 0;
            sa.njob_idx = 1;
            rc = pass(L.capA);
            if (rc)
                return rc;
            // pass C: outputs of segments 1 .. G - 1, each chaining its entering state first;
            // the last segment's final state is new_state
            sa.job_first = (int)L.capA;
            sa.njob_idx = 2;
            rc = pass(L.capC);
        } else if (whole_dual) {
            rc = launch(gdn::gdn_prefill_scan_any_kernel<false>, N, blocks_of(groups, 2), 512);
        } else if (wide) {
            sa.njob_idx = 6;
            rc = launch(gdn::gdn_prefill_scanw_kernel, N, blocks_of(groups, 1), 256);
            if (rc == 0) {
                sa.njob_idx = 5;  // one workgroup per CU, at least one per queue
                rc = launch(gdn::gdn_prefill_scan8q_kernel, N, 8 * std::max<int64_t>(cus / 8, 1), 512);
            }
        } else if (nw4) {
            rc = launch(gdn::gdn_prefill_scan4_kernel, N, blocks_of(groups, groups <= sa.split_groups ? 4 : 2), 320);
        } else {
            rc = launch(gdn::gdn_prefill_scan8_kernel, N, blocks_of(groups, 1), 512);
        }
        if (rc)
            return rc;
    }
    return GDN_OK;
}
