// qgemm_skinny.hip -- q_matrix x fp16 rows for 17 .. 128 rows: short prompts, prompt chunks, batches of 17 .. 128 sequences.
//
// Replaces, for these row counts, the reference's reconstruct_kernel + library Hgemm (cuda/q_gemm.cu:243-263: the whole fp16 [K, N]
// matrix written to HBM and read back for a product that needs K N / 2 bytes of weights).
//
// The product is bound by the weight stream (64 rows: 256 FLOP per weight byte, the chip's ridge is ~310), so the kernel is built like
// the decode kernels -- many small workgroups, every request far ahead of its use -- and not like a GEMM:
//   * workgroup = 4 waves = 128 columns x ALL rows x a slice of K (blockIdx.y = K split); wave w owns two 16-column tiles and streams
//     THEIR items (128 K-rows = one contiguous 64 b-dword run per tile) through a register ring NST deep, NST - 1 steps ahead;
//   * the activation rows of a K step (16 RB rows x 128 halfs) arrive by LDS-DMA (buffer form: counted by vmcnt like any load) into a
//     ring of NST stages, a wave's group scales (the make-time table of the fp16 values reconstruct() uses: 2 tiles x 4 chunks x 32
//     bytes) by one more copy beside them; the packed words are requested BEHIND the copies, so a wave that has its words has its share of
//     the copies; ONE workgroup barrier per step;
//   * per chunk of 32 K-rows a wave decodes its two tiles to fragments in registers (half(q - zero) * half(scale), reconstruct()'s
//     rounding) and multiplies them (W^T as the A operand: a lane owns four consecutive columns of a row) with every row fragment,
//     read once from LDS (swizzled, conflict-free): 8 RB v_mfma_f32_16x16x32_f16 per step and wave;
//   * split K: partial tiles leave in fragment order, a second launch adds them in split order and runs the epilogue (bias,
//     accumulate-into-c, the consumer's column order).
// What a step costs is a chain -- barrier, LDS reads, decode, matrix cores -- that only other waves hide, so registers and LDS are cut
// to three workgroups per CU (<= 64 rows).  Measured (whole calls, row pre-pass included), against two workgroups per CU with the scales
// unpacked by every workgroup, row blocks in pairs and the last split to arrive adding the partial tiles: 4096 x 4096 at 48 / 128 rows 28.5 ->
// 19.4 / 42.2 -> 28.8 us, 11008 x 4096 43.2 -> 32.6 / 62.1 -> 43.6 us, 4096 x 22016 38.9 -> 33.1 / 75.5 -> 50.2 us; at 17 rows, where the
// weights' own time is the larger part, 20.0 -> 17.7, 30.2 -> 28.1, 28.7 -> 28.5 us.
// Algorithmic bytes: packed weights + scales once, M K 2 of rows per 128-column group (L2), M N 2 out.
#include "qgemm_prefill.h"
#include "qgemm_skinny.h"
#include "errors.h"
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define SK_BN 128
#define SK_CT 2                                   // 16-column tiles per wave
#define SK_WAVES 4
#define SK_THREADS (SK_WAVES * 64)
#define SK_X_BYTES(RB) ((RB) * 16 * 256)          // one stage of rows: 16 RB rows x 128 halfs
#define SK_SC_BYTES(GPTQ) (SK_WAVES * 256 * ((GPTQ) ? 2 : 1))      // one stage of scales [wave][tile][chunk][16], (GPTQ) zero points behind a wave's
#define SK_NST(RB) ((RB) <= 3 ? 4 : (RB) <= 6 ? 3 : 2)             // stages = register-ring depth: requests run NST - 1 steps ahead
#define SK_LDS_BYTES(RB, GPTQ, chunks) (SK_NST(RB) * (SK_X_BYTES(RB) + SK_SC_BYTES(GPTQ)) + (((chunks) * 2 + 15) & ~15))

#define SK_MAX_JOBS 3        // matrices of one launch: q | k | v, gate | up multiply the same staged rows (GemvJob::rows_as_prev)
struct SkinnyJob { QMatDev m; f16* c; const u16* c_invperm; int ldc, c_mode; };
struct SkinnyArgs
{
    SkinnyJob job[SK_MAX_JOBS];
    int group0[SK_MAX_JOBS + 1];   // first column group (blockIdx.x) of every matrix
    const f16* a;           // [M, K] in packed K order, row stride K (stage_rows_kernel's output)
    int M;
    int ks;                 // K splits (gridDim.y)
    f32x4* part;            // ks > 1: [column group][split][wave][row block][tile][lane] partial accumulators
};

struct SkCtx
{
    const f16* a; const f16* sc[2]; const f16* zp[2];      // [1]: the second matrix of a pair (tile 1 is its tile then)
    const u16* cg[2];                             // chunk -> group maps [K / 32] (LDS)
    u8* x_st; u8* sc_st;                          // rings of stages
    int tile[SK_CT];
    u32 sc_row;                                   // per lane: first scale row (groups) of the tile whose scales it copies
    int lane, wv, last_chunk;
};

// a wave's scales of the chunks chunk0 .. chunk0 + 3 -> its part of `stage`: lane l < 16 copies 16 bytes, half l & 1 of the row of tile l >> 3,
// chunk (l >> 1) & 3; lanes 16 .. 31 (GPTQ) the zero points
template <bool GPTQ, bool PAIR>
DEV void sk_issue_scales(const SkCtx& x, int chunk0, u8* stage)
{
    const int l = x.lane & 15;
    const int ci = min(chunk0 + ((l >> 1) & 3), x.last_chunk);              // (chunks past the matrix are never multiplied in)
    const u32 off = (x.sc_row + (u32)x.cg[0][ci]) * 32u + (u32)(l & 1) * 16u;
    u8* const dst = stage + x.wv * (GPTQ ? 512 : 256);
    if constexpr (PAIR)
    {
        const u32 off1 = (x.sc_row + (u32)x.cg[1][ci]) * 32u + (u32)(l & 1) * 16u;
        if (x.lane < 8) dma_buf_to_lds16(x.sc[0], off, dst);
        if (x.lane >= 8 && x.lane < 16) dma_buf_to_lds16(x.sc[1], off1, dst);
        if constexpr (GPTQ)
        {
            if (x.lane >= 16 && x.lane < 24) dma_buf_to_lds16(x.zp[0], off, dst);
            if (x.lane >= 24 && x.lane < 32) dma_buf_to_lds16(x.zp[1], off1, dst);
        }
    }
    else
    {
        if (x.lane < 16) dma_buf_to_lds16(x.sc[0], off, dst);
        if constexpr (GPTQ) { if (x.lane >= 16 && x.lane < 32) dma_buf_to_lds16(x.zp[0], off, dst); }
    }
}

// rows of the K step at packed row k0: this wave's copies i hold rows 4 (4 i + w) .. + 3 (unit u of row r at slot u ^ (r & 15)); `nv` chunks
template <int RB>
DEV void sk_issue_rows(const SkCtx& x, const u32 (&voff)[RB], int k0, int nv, u8* stage)
{
    // (a partial item: units past it would lie past the row -- its last unit again instead)
    const u32 back = nv < 4 ? (u32)max(0, ((x.lane & 15) ^ (x.wv * 4 + (x.lane >> 4))) - (4 * nv - 1)) * 16u : 0u;
    #pragma unroll
    for (int i = 0; i < RB; i++)
        dma_buf_to_lds16_so(x.a, voff[i] - back, (u32)k0 * 2u, stage + (size_t)(i * SK_WAVES + x.wv) * 1024);
}

template <int BITS, bool GPTQ>
DEV f16x8 sk_decode(const LaneWords<BITS>& r, int q, f16 scale, f16 zero)
{
    ZC zc[4];
    #pragma unroll
    for (int i = 0; i < 4; i++) zc[i] = make_zc(GPTQ ? zero : (f16)(float)(1 << (BITS - 1)));
    f16x2 p[16];
    dequant_super<BITS>(r.w, zc, p);                                        // (the other chunks' work is dead code)
    const f16x2 s2 = h2_dup(scale);
    const f16x2 b0 = p[4 * q + 0] * s2, b1 = p[4 * q + 1] * s2, b2 = p[4 * q + 2] * s2, b3 = p[4 * q + 3] * s2;
    return (f16x8){b0.x, b0.y, b1.x, b1.y, b2.x, b2.y, b3.x, b3.y};
}

template <int BITS, bool GPTQ, int RB>
DEV void sk_multiply(const SkCtx& x, const LaneWords<BITS> (&r)[SK_CT], const u8* stage, const u8* sc_stage, int nv, f32x4 (&acc)[RB][SK_CT])
{
    // (the lane number made anew in every step: the addresses are a few operations, kept in registers they push others out)
    int lane = x.lane;
    pin_vector(lane);
    const int i16 = lane & 15, j4 = lane >> 4;
    const u8* const xr = stage + (size_t)i16 * 256;
    const f16* const sc = (const f16*)(sc_stage + x.wv * (GPTQ ? 512 : 256)) + i16;
    f16 s[SK_CT][4], z[SK_CT][4];
    #pragma unroll
    for (int ct = 0; ct < SK_CT; ct++)
        #pragma unroll
        for (int q = 0; q < 4; q++) { s[ct][q] = sc[(ct * 4 + q) * 16]; z[ct][q] = GPTQ ? sc[128 + (ct * 4 + q) * 16] : (f16)0.0f; }
    #pragma unroll
    for (int q = 0; q < 4; q++)
    {
        if (q < nv)
        {
            f16x8 wf[SK_CT], xf[RB];
            #pragma unroll
            for (int rb = 0; rb < RB; rb++) xf[rb] = *(const f16x8*)(xr + (((4 * q + j4) ^ i16) * 16) + rb * 4096);
            #pragma unroll
            for (int ct = 0; ct < SK_CT; ct++) wf[ct] = sk_decode<BITS, GPTQ>(r[ct], q, s[ct][q], z[ct][q]);
            #pragma unroll
            for (int rb = 0; rb < RB; rb++)
                #pragma unroll
                for (int ct = 0; ct < SK_CT; ct++) acc[rb][ct] = mfma_16x16x32_f16(wf[ct], xf[rb], acc[rb][ct]);
        }
    }
}

// F items of one section (from the split's first one on); the last holds nv_last chunks.  Every request is UNCONDITIONAL (past the end the
// last item again, never multiplied): a request under a branch makes the compiler's counted waits at the join as strict as the
// shorter path needs.
template <int BITS, bool GPTQ, int RB, bool PAIR>
DEV void sk_stream(const SkCtx& x, const u32 (&voff)[RB], const u32* base, const u32* base1, u32 tile_stride, int F, int k_base, int nv_last, f32x4 (&acc)[RB][SK_CT])
{
    constexpr int NST = SK_NST(RB);
    LaneWords<BITS> ring[NST][SK_CT];
    auto request = [&](int s, int slot)
    {
        const int sn = min(s, F - 1);
        sk_issue_rows<RB>(x, voff, k_base + sn * SUPER_ROWS, sn == F - 1 ? nv_last : 4, x.x_st + slot * SK_X_BYTES(RB));
        sk_issue_scales<GPTQ, PAIR>(x, (k_base >> 5) + 4 * sn, x.sc_st + slot * SK_SC_BYTES(GPTQ));
        asm volatile("" ::: "memory");
        #pragma unroll
        for (int ct = 0; ct < SK_CT; ct++)
            load_lane_words<BITS>((PAIR && ct ? base1 : base) + (size_t)x.tile[ct] * tile_stride + (size_t)sn * (64 * BITS), x.lane, ring[slot][ct]);
    };
    #pragma unroll
    for (int u = 0; u < NST - 1; u++) request(u, u);
    for (int s0 = 0; s0 < F; s0 += NST)
    {
        #pragma unroll
        for (int u = 0; u < NST; u++)
        {
            const int s = s0 + u;
            fence_load_use(ring[u][SK_CT - 1].w[BITS - 1]);             // this step's words are here, and with them its copies
            block_sync_lds();                                           // ... of every wave; everybody is done with the stage before
            request(s + NST - 1, (u + NST - 1) % NST);
            if (s < F) sk_multiply<BITS, GPTQ, RB>(x, ring[u], x.x_st + u * SK_X_BYTES(RB), x.sc_st + u * SK_SC_BYTES(GPTQ), s == F - 1 ? nv_last : 4, acc);
        }
    }
    wait_vmcnt_le<0>();                                     // (requests past the end of the run)
    block_sync_lds();                                       // the stages are free for the next section
}

// one contiguous stream of items per 16-column tile: a bit-width section (QRun, kernel arguments) or, for matrices with more sections
// than the argument block holds (n_runs = 0), a descriptor (QDesc, device memory); its last item may be partial
struct SkSegment { const u32* base; u32 tile_stride; int n_super, k_base, bits, nvl; };
DEV SkSegment sk_segment(const QMatDev& m, int i)
{
    SkSegment g;
    int in_tail; u32 base_word;
    if (m.n_runs > 0)
    {
        const QRun& r = m.runs[i];
        g.n_super = uniform((int)r.n_super); g.nvl = uniform((int)r.nvalid_last); in_tail = uniform((int)r.in_tail); base_word = uniform(r.base_word);
        g.tile_stride = uniform(r.tile_stride); g.k_base = uniform((int)r.k_base); g.bits = uniform((int)r.bits);
    }
    else
    {
        const QDesc* d = m.desc + i;
        g.n_super = uniform((int)d->n_super); g.nvl = uniform((int)d->nvalid_last); in_tail = uniform((int)d->in_tail); base_word = uniform(d->base_word);
        g.tile_stride = uniform(d->tile_stride); g.k_base = uniform((int)d->k_base); g.bits = uniform((int)d->bits);
    }
    g.base = (in_tail ? m.tail : m.qw) + base_word;
    return g;
}

DEV int sk_job(const SkinnyArgs& a, int group) { return (group >= a.group0[1] ? 1 : 0) + (group >= a.group0[2] ? 1 : 0); }

template <bool GPTQ, int RB>
KERNEL void __launch_bounds__(SK_THREADS, RB <= 4 ? 3 : 2) qgemm_skinny_kernel(const SkinnyArgs args)
{
    DYN_SMEM(smem);
    const int jb = sk_job(args, bid_x());
    const SkinnyJob& job = args.job[jb];
    const QMatDev& m = job.m;
    const int t = tid(), lane = lane_id(), wv = uniform(wave_id());
    const int KS = args.ks, z = bid_y();
    const int n0 = (bid_x() - args.group0[jb]) * SK_BN;
    const int n_tiles = m.N / TILE_N;

    SkCtx x;
    x.a = args.a; x.sc[0] = m.sc_tab; x.zp[0] = m.zp_tab; x.lane = lane; x.wv = wv; x.last_chunk = (m.K >> 5) - 1;
    x.x_st = smem; x.sc_st = smem + SK_NST(RB) * SK_X_BYTES(RB);
    #pragma unroll
    for (int ct = 0; ct < SK_CT; ct++) x.tile[ct] = min((n0 >> 4) + wv * SK_CT + ct, n_tiles - 1);      // partial last column group: computed, never stored
    x.sc_row = (u32)(((lane & 8) ? x.tile[1] : x.tile[0]) * m.G);
    u32 voff[RB];
    #pragma unroll
    for (int i = 0; i < RB; i++)
    {
        const int row = (i * SK_WAVES + wv) * 4 + (lane >> 4), u = (lane & 15) ^ (row & 15);
        voff[i] = (u32)(((size_t)min(row, args.M - 1) * m.K + u * 8) * 2);
    }
    // this split's items, counted over the sections in K order
    const int n_seg = m.n_runs > 0 ? m.n_runs : m.n_desc;
    int total = 0;
    for (int si = 0; si < n_seg; si++) total += sk_segment(m, si).n_super;
    const int it_lo = (int)((long long)total * z / KS), it_hi = (int)((long long)total * (z + 1) / KS);
    {
        u16* cg = (u16*)(smem + SK_NST(RB) * (SK_X_BYTES(RB) + SK_SC_BYTES(GPTQ)));
        for (int i = t; i < (m.K >> 5); i += SK_THREADS) cg[i] = m.chunk_group[i];
        x.cg[0] = cg;
        block_sync();
    }
    f32x4 acc[RB][SK_CT];
    #pragma unroll
    for (int rb = 0; rb < RB; rb++)
        #pragma unroll
        for (int ct = 0; ct < SK_CT; ct++) acc[rb][ct] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    int pos = 0;
    for (int si = 0; si < n_seg; si++)
    {
        const SkSegment sg = sk_segment(m, si);
        const int bits = GPTQ ? 4 : sg.bits;
        const int f0 = max(it_lo - pos, 0), f1 = min(it_hi - pos, sg.n_super);
        pos += sg.n_super;
        if (f1 <= f0) continue;
        const u32* base = sg.base + (size_t)f0 * (size_t)(64 * bits);
        const int k_base = sg.k_base + f0 * SUPER_ROWS, F = f1 - f0, nvl = f1 == sg.n_super ? sg.nvl : 4;
        switch (bits)
        {
            case 4: sk_stream<4, GPTQ, RB, false>(x, voff, base, base, sg.tile_stride, F, k_base, nvl, acc); break;
            case 8: if constexpr (!GPTQ) sk_stream<8, false, RB, false>(x, voff, base, base, sg.tile_stride, F, k_base, nvl, acc); break;
            case 6: if constexpr (!GPTQ) sk_stream<6, false, RB, false>(x, voff, base, base, sg.tile_stride, F, k_base, nvl, acc); break;
            case 5: if constexpr (!GPTQ) sk_stream<5, false, RB, false>(x, voff, base, base, sg.tile_stride, F, k_base, nvl, acc); break;
            case 3: if constexpr (!GPTQ) sk_stream<3, false, RB, false>(x, voff, base, base, sg.tile_stride, F, k_base, nvl, acc); break;
            default: if constexpr (!GPTQ) sk_stream<2, false, RB, false>(x, voff, base, base, sg.tile_stride, F, k_base, nvl, acc); break;
        }
    }

    if (KS > 1)
    {
        f32x4* const mine = args.part + ((((size_t)bid_x() * KS + z) * SK_WAVES + wv) * RB * SK_CT) * 64 + lane;
        #pragma unroll
        for (int rb = 0; rb < RB; rb++)
            #pragma unroll
            for (int ct = 0; ct < SK_CT; ct++) mine[(rb * SK_CT + ct) * 64] = acc[rb][ct];
        return;
    }
    // lane (i = l & 15, j = l >> 4) holds row i of the row block, columns 4 j .. 4 j + 3 of the tile
    #pragma unroll
    for (int ct = 0; ct < SK_CT; ct++)
    {
        const int n = n0 + (wv * SK_CT + ct) * 16 + 4 * (lane >> 4);
        if (n >= m.N) continue;
        #pragma unroll
        for (int rb = 0; rb < RB; rb++)
        {
            const int row = rb * 16 + (lane & 15);
            if (row < args.M) store_row4(job, row, n, acc[rb][ct]);
        }
    }
}

// K splits: one accumulator (four columns of one row) per thread, summed over the splits in order
template <int RB>
KERNEL void __launch_bounds__(256) sk_reduce_kernel(const SkinnyArgs args)
{
    constexpr int PER = SK_WAVES * RB * SK_CT * 64;          // accumulators of a column group
    const int grp = bid_x() / (PER / 256), u = (bid_x() - grp * (PER / 256)) * 256 + tid();
    const int jb = sk_job(args, grp);
    const SkinnyJob& job = args.job[jb];
    const int lane = u & 63, ct = (u >> 6) % SK_CT, rb = (u / (64 * SK_CT)) % RB, wv = u / (64 * SK_CT * RB);
    const int row = rb * 16 + (lane & 15), n = (grp - args.group0[jb]) * SK_BN + (wv * SK_CT + ct) * 16 + 4 * (lane >> 4);
    if (row >= args.M || n >= job.m.N) return;
    const f32x4* p = args.part + (size_t)grp * args.ks * PER + u;
    f32x4 acc = p[0];
    for (int z = 1; z < args.ks; z++) acc += p[(size_t)z * PER];
    store_row4(job, row, n, acc);
}

// ---- experts of a sparse block, 2 .. 64 rows (qgemm_skinny.h) ------------------------------------------------------------------------
// The same walk over every expert that has rows: workgroup = (expert, column group) x K split; the expert's rows are the set bits of a
// ballot over the rows' routing weights, so there is no list to make and nothing the host would have to know.  Pair form: wave w owns one
// tile of gate and the same tile of up, the epilogue writes act(gate) * up (fp32, one rounding) to the expert's slot rows in down's
// packed order.  Otherwise (down): partial tiles for the launch that adds splits and experts (modules.hip: moe_sum_slots_kernel).
// Bound by the weight stream (8 experts 4096 x 14336 at 3.5 bits, 16 rows: gate | up 101 us = 4.1 TB/s, down 54 us = 3.8 TB/s; the phased
// kernels over pairs and quadruples of experts 252 us + 26 us of row pre-passes).  Whole eight-layer steps, us, before -> now: 2 rows 1462 ->
// 1221, 4: 2009 -> 1448, 16: 2905 -> 1821, 33: 11097 -> 2505, 64: 20453 -> 2715; from 65 rows (3616, the ballot's end) qgemm_tile.hip.
template <bool GPTQ, int RB, bool PAIR>
KERNEL void __launch_bounds__(SK_THREADS, 3) qgemm_skinny_experts_kernel(const SkExpertReq args)
{
    DYN_SMEM(smem);
    constexpr int BM = 16 * RB, BN = PAIR ? 64 : SK_BN;
    const int t = tid(), lane = lane_id(), wv = uniform(wave_id());
    const int i16 = lane & 15, j4 = lane >> 4;
    const int e = bid_x() / args.groups, grp = bid_x() - e * args.groups, z = bid_y(), KS = args.ks;
    const u64 mask = wave_ballot(lane < args.M && as_u16(args.weights[(size_t)min(lane, args.M - 1) * args.n_experts + e]) != 0);
    const int cnt = __builtin_popcountll(mask);
    if (cnt == 0) return;
    auto global = [](const void* p) -> const void* { return global_ptr_of(uniform((u32)(u64)p), uniform((u32)((u64)p >> 32))); };
    const QMatDev* const m0 = args.table + (size_t)e * args.table_stride;
    const int K = uniform(m0->K), N = uniform(m0->N), n_runs = uniform(m0->n_runs);
    const int n_tiles = N / TILE_N, n0 = grp * BN;

    SkCtx x;
    x.a = args.a; x.lane = lane; x.wv = wv; x.last_chunk = (K >> 5) - 1;
    x.x_st = smem; x.sc_st = smem + SK_NST(RB) * SK_X_BYTES(RB);
    u8* const maps = smem + SK_NST(RB) * (SK_X_BYTES(RB) + SK_SC_BYTES(GPTQ));
    const int map_bytes = ((K >> 5) * 2 + 15) & ~15;
    const u32 *qw[2], *tail[2];
    #pragma unroll
    for (int mi = 0; mi < (PAIR ? 2 : 1); mi++)
    {
        const QMatDev* const m = m0 + mi;
        x.sc[mi] = (const f16*)global(m->sc_tab); x.zp[mi] = (const f16*)global(m->zp_tab);
        qw[mi] = (const u32*)global(m->qw); tail[mi] = (const u32*)global(m->tail);
        u16* const cg = (u16*)(maps + mi * map_bytes);
        const u16* const src = (const u16*)global(m->chunk_group);
        for (int i = t; i < (K >> 5); i += SK_THREADS) cg[i] = src[i];
        x.cg[mi] = cg;
    }
    if (!PAIR) { qw[1] = qw[0]; tail[1] = tail[0]; }
    #pragma unroll
    for (int ct = 0; ct < SK_CT; ct++) x.tile[ct] = min(PAIR ? grp * 4 + wv : grp * 8 + wv * SK_CT + ct, n_tiles - 1);      // (past the matrix: computed, never stored)
    const int G0 = uniform(m0->G), G1 = PAIR ? uniform(m0[1].G) : G0;
    x.sc_row = (u32)((lane & 8) ? x.tile[1] * G1 : x.tile[0] * G0);
    // the rows of this expert: bit r of the ballot = row r, its local number = the set bits below
    int* const list = (int*)(maps + 2 * map_bytes);
    if (wv == 0 && ((mask >> lane) & 1)) list[__builtin_popcountll(mask & (((u64)1 << lane) - 1))] = lane;
    block_sync();
    u32 voff[RB];
    #pragma unroll
    for (int i = 0; i < RB; i++)
    {
        const int row = (i * SK_WAVES + wv) * 4 + (lane >> 4), u = (lane & 15) ^ (row & 15);
        const int li = min(row, cnt - 1);                                   // (rows past the end: computed, never stored)
        voff[i] = (u32)(((size_t)(PAIR ? list[li] : e * BM + li) * K + u * 8) * 2);
    }
    f32x4 acc[RB][SK_CT];
    #pragma unroll
    for (int rb = 0; rb < RB; rb++)
        #pragma unroll
        for (int ct = 0; ct < SK_CT; ct++) acc[rb][ct] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    const int n_seg = n_runs > 0 ? n_runs : uniform(m0->n_desc);
    auto segment = [&](int i, u32& base_word, int& in_tail) -> SkSegment
    {
        SkSegment g;
        if (n_runs > 0)
        {
            const QRun& r = m0->runs[i];
            g.n_super = uniform((int)r.n_super); g.nvl = uniform((int)r.nvalid_last); in_tail = uniform((int)r.in_tail); base_word = uniform(r.base_word);
            g.tile_stride = uniform(r.tile_stride); g.k_base = uniform((int)r.k_base); g.bits = uniform((int)r.bits);
        }
        else
        {
            const QDesc* d = m0->desc + i;
            g.n_super = uniform((int)d->n_super); g.nvl = uniform((int)d->nvalid_last); in_tail = uniform((int)d->in_tail); base_word = uniform(d->base_word);
            g.tile_stride = uniform(d->tile_stride); g.k_base = uniform((int)d->k_base); g.bits = uniform((int)d->bits);
        }
        g.base = nullptr;
        return g;
    };
    int total = 0;
    u32 base_word; int in_tail;
    if (KS > 1) for (int si = 0; si < n_seg; si++) total += segment(si, base_word, in_tail).n_super;
    const int it_lo = KS > 1 ? (int)((long long)total * z / KS) : 0, it_hi = KS > 1 ? (int)((long long)total * (z + 1) / KS) : 0x7fffffff;
    int pos = 0;
    for (int si = 0; si < n_seg; si++)
    {
        const SkSegment sg = segment(si, base_word, in_tail);
        const int bits = GPTQ ? 4 : sg.bits;
        const int f0 = max(it_lo - pos, 0), f1 = min(it_hi - pos, sg.n_super);
        pos += sg.n_super;
        if (f1 <= f0) continue;
        const size_t at = (size_t)base_word + (size_t)f0 * (size_t)(64 * bits);
        const u32* const base = (in_tail ? tail[0] : qw[0]) + at;
        const u32* const base1 = (in_tail ? tail[1] : qw[1]) + at;
        const int k_base = sg.k_base + f0 * SUPER_ROWS, F = f1 - f0, nvl = f1 == sg.n_super ? sg.nvl : 4;
        switch (bits)
        {
            case 4: sk_stream<4, GPTQ, RB, PAIR>(x, voff, base, base1, sg.tile_stride, F, k_base, nvl, acc); break;
            case 8: if constexpr (!GPTQ) sk_stream<8, false, RB, PAIR>(x, voff, base, base1, sg.tile_stride, F, k_base, nvl, acc); break;
            case 6: if constexpr (!GPTQ) sk_stream<6, false, RB, PAIR>(x, voff, base, base1, sg.tile_stride, F, k_base, nvl, acc); break;
            case 5: if constexpr (!GPTQ) sk_stream<5, false, RB, PAIR>(x, voff, base, base1, sg.tile_stride, F, k_base, nvl, acc); break;
            case 3: if constexpr (!GPTQ) sk_stream<3, false, RB, PAIR>(x, voff, base, base1, sg.tile_stride, F, k_base, nvl, acc); break;
            default: if constexpr (!GPTQ) sk_stream<2, false, RB, PAIR>(x, voff, base, base1, sg.tile_stride, F, k_base, nvl, acc); break;
        }
    }

    if constexpr (!PAIR)
    {
        f32x4* const mine = args.part + ((((size_t)bid_x() * KS + z) * SK_WAVES + wv) * RB * SK_CT) * 64 + lane;
        #pragma unroll
        for (int rb = 0; rb < RB; rb++)
            #pragma unroll
            for (int ct = 0; ct < SK_CT; ct++) mine[(rb * SK_CT + ct) * 64] = acc[rb][ct];
        return;
    }
    const int n = (grp * 4 + wv) * 16 + 4 * j4;
    if (n >= N) return;
    const f16* const bias0 = (const f16*)global(m0->bias);
    const f16* const bias1 = (const f16*)global(m0[PAIR ? 1 : 0].bias);
    const u16* const invperm = (const u16*)global(args.invperms[e]);
    #pragma unroll
    for (int rb = 0; rb < RB; rb++)
    {
        if (rb * 16 + i16 >= cnt) continue;
        f16* const cp = args.c + (size_t)(e * BM + rb * 16 + i16) * N;
        f16x4 h;
        #pragma unroll
        for (int k = 0; k < 4; k++)
        {
            const float g = acc[rb][0][k] + (bias0 ? (float)bias0[n + k] : 0.0f), u = acc[rb][1][k] + (bias1 ? (float)bias1[n + k] : 0.0f);
            const float v = act_f32(g, args.act_gelu != 0) * u;
            h[k] = (f16)(v > 65504.0f ? 65504.0f : v < -65504.0f ? -65504.0f : v);
        }
        if (invperm)
        {
            #pragma unroll
            for (int k = 0; k < 4; k++) cp[invperm[n + k]] = h[k];
        }
        else *(f16x4*)(cp + n) = h;
    }
}

// ---- host ---------------------------------------------------------------------------------------------------------------------------

template <bool GPTQ, int RB>
static int sk_launch_rb(const SkinnyArgs& p, dim3 grid, size_t lds, void* stream)
{
    static bool attr[EXL2_MAX_DEVICES] = {false};
    if (exl2_first_on_device(attr))
        (void)hipFuncSetAttribute((const void*)qgemm_skinny_kernel<GPTQ, RB>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    LAUNCH((qgemm_skinny_kernel<GPTQ, RB>), grid, dim3(SK_THREADS), lds, stream, p);
    if (p.ks > 1) LAUNCH((sk_reduce_kernel<RB>), dim3(grid.x * (unsigned)(SK_WAVES * RB * SK_CT * 64 / 256)), dim3(256), 0, stream, p);
    return EXL2_OK;
}

// n (1 .. SK_MAX_JOBS) matrices over the SAME staged rows in one launch.  0 = launched, 1 = does not apply (the caller takes the generic
// kernel, one matrix at a time), < 0 = error
int qgemm_skinny_launch(const PrefillArgs* pas, int n, bool gptq, void* stream)
{
    if (n < 1 || n > SK_MAX_JOBS) return 1;
    const int M = pas[0].M, K = pas[0].m.K;
    if (M < 1 || M > 128) return 1;
    if ((size_t)128 * (size_t)K * 2 >= ((size_t)1 << 31)) return 1;               // the row copies address a 2 GB buffer window
    const int rb = (M + 15) / 16, RBT = rb <= 2 ? 2 : rb <= 4 ? rb : rb <= 6 ? 6 : 8;
    SkinnyArgs p;
    memset(&p, 0, sizeof(p));
    int groups = 0, min_items = 0x7fffffff;
    for (int i = 0; i < n; i++)
    {
        const QMatDev& m = pas[i].m;
        if (m.K != K || pas[i].M != M || pas[i].a != pas[0].a || !m.sc_tab || (gptq && !m.zp_tab)) return 1;
        int items = 0;
        for (int ri = 0; ri < m.n_runs; ri++) items += (int)m.runs[ri].n_super;
        if (m.n_runs <= 0) items = K >> 7;                                        // (descriptors live on the device: a lower bound)
        if (items < min_items) min_items = items;
        p.job[i].m = m;
        if (getenv("EXL2_SKINNY_FORCE_DESC")) p.job[i].m.n_runs = 0;      // tests: walk the descriptors (what a matrix with > MAX_RUNS sections takes)
        p.job[i].c = pas[i].c; p.job[i].ldc = pas[i].ldc; p.job[i].c_invperm = pas[i].c_invperm; p.job[i].c_mode = pas[i].c_mode;
        p.group0[i] = groups;
        groups += (m.N + SK_BN - 1) / SK_BN;
    }
    for (int i = n; i <= SK_MAX_JOBS; i++) p.group0[i] = i == n ? groups : 0x7fffffff;
    for (int i = n + 1; i <= SK_MAX_JOBS; i++) p.group0[i] = 0x7fffffff;
    const size_t lds = gptq ? (size_t)SK_LDS_BYTES(RBT, 1, K >> 5) : (size_t)SK_LDS_BYTES(RBT, 0, K >> 5);
    if (lds > 160 * 1024) return 1;
    // K splits: as many as fit the chip in one round (two workgroups per CU up to 32 rows, whatever fits from 33), 8 at most; >= 4 items per
    // split beyond four of them.  Whole calls over weights that come from memory, us (splits: time).  48 rows: 4096 x 4096 2: 24.9, 4: 19.6,
    // 8: 18.8; 11008 x 4096 2: 51.4, 4: 35.7, 8: 29.2; 4096 x 22016 2: 34.4, 4: 33.5, 8: 43.5 (two rounds); 2048 x 5632 2: 17.9, 4: 16.2, 8: 19.7
    // (two items each).  17 rows: 4096 x 11008 2: 23.3, 4: 21.2, 5: 22.6, 8: 23.2; 4096 x 32000 1: 34.7, 2: 33.0, 3: 34.9; 8192 x 28672 (8 / 4 bits)
    // 2: 55.7, 3: 57.1.  More splits are more bytes for the adding launch.
    const int per_cu = (int)((160 * 1024) / lds) < (RBT <= 4 ? 3 : 2) ? (int)((160 * 1024) / lds) : (RBT <= 4 ? 3 : 2);
    int ks = 256 * (RBT <= 2 ? 2 : per_cu) / groups;
    if (ks > 8) ks = 8;
    if (ks > 4 && ks > min_items / 4) ks = min_items / 4 > 4 ? min_items / 4 : 4;
    if (ks > min_items / 2) ks = min_items / 2;
    if (const char* e = getenv("EXL2_SKINNY_SPLITK")) { const int v = atoi(e); if (v >= 1) ks = v > 32 ? 32 : v; if (ks > min_items) ks = min_items; }
    if (ks < 1) ks = 1;
    p.a = pas[0].a; p.M = M; p.ks = ks;
    if (ks > 1)
    {
        p.part = (f32x4*)prefill_scratch_try((size_t)groups * ks * SK_WAVES * RBT * SK_CT * 64 * sizeof(f32x4), stream, 2);
        if (!p.part) p.ks = ks = 1;
    }
    const dim3 grid((unsigned)groups, (unsigned)ks, 1);
    if (getenv("EXL2_SKINNY_DEBUG")) fprintf(stderr, "[skinny] M %d K %d matrices %d RB %d grid %d x %d lds %zu items %d\n", M, K, n, RBT, groups, ks, lds, min_items);
    if (gptq)
        switch (RBT)
        {
            case 2: return sk_launch_rb<true, 2>(p, grid, lds, stream);
            case 3: return sk_launch_rb<true, 3>(p, grid, lds, stream);
            case 4: return sk_launch_rb<true, 4>(p, grid, lds, stream);
            case 6: return sk_launch_rb<true, 6>(p, grid, lds, stream);
            default: return sk_launch_rb<true, 8>(p, grid, lds, stream);
        }
    switch (RBT)
    {
        case 2: return sk_launch_rb<false, 2>(p, grid, lds, stream);
        case 3: return sk_launch_rb<false, 3>(p, grid, lds, stream);
        case 4: return sk_launch_rb<false, 4>(p, grid, lds, stream);
        case 6: return sk_launch_rb<false, 6>(p, grid, lds, stream);
        default: return sk_launch_rb<false, 8>(p, grid, lds, stream);
    }
}

template <bool GPTQ, int RB, bool PAIR>
static int sk_launch_experts(const SkExpertReq& p, size_t lds, void* stream)
{
    static bool attr[EXL2_MAX_DEVICES] = {false};
    if (exl2_first_on_device(attr))
        (void)hipFuncSetAttribute((const void*)qgemm_skinny_experts_kernel<GPTQ, RB, PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    LAUNCH((qgemm_skinny_experts_kernel<GPTQ, RB, PAIR>), dim3((unsigned)(p.n_experts * p.groups), (unsigned)p.ks), dim3(SK_THREADS), lds, stream, p);
    return EXL2_OK;
}

template <int RB>
static int sk_launch_experts_rb(const SkExpertReq& p, size_t lds, bool gptq, void* stream)
{
    if (gptq) return p.pair ? sk_launch_experts<true, RB, true>(p, lds, stream) : sk_launch_experts<true, RB, false>(p, lds, stream);
    return p.pair ? sk_launch_experts<false, RB, true>(p, lds, stream) : sk_launch_experts<false, RB, false>(p, lds, stream);
}

void qgemm_skinny_experts_plan(SkExpertReq& r, int N, int items)
{
    r.groups = (N + (r.pair ? 64 : SK_BN) - 1) / (r.pair ? 64 : SK_BN);
    // splits of down: about four workgroups per CU (at 16 rows an expert in eight has none), 8 at most, >= 4 items each
    int ks = r.pair ? 1 : 1024 / (r.groups * r.n_experts);
    if (ks > 8) ks = 8;
    if (ks > items / 4) ks = items / 4;
    if (const char* e = getenv("EXL2_SKINNY_EXPERT_KS")) { if (!r.pair) ks = atoi(e) < items ? atoi(e) : items; }
    r.ks = ks < 1 ? 1 : ks;
}

int qgemm_skinny_experts_launch(const SkExpertReq& r, int K, bool gptq, void* stream)
{
    const int rb = qgemm_skinny_experts_blocks(r.M);
    if (r.M < 1 || rb > 4) return 1;                         // (the ballot covers 64 rows)
    const int map_bytes = ((K >> 5) * 2 + 15) & ~15;
    const size_t lds = (size_t)SK_NST(rb) * (SK_X_BYTES(rb) + SK_SC_BYTES(gptq ? 1 : 0)) + 2 * (size_t)map_bytes + 64 * sizeof(int);
    if (lds > 160 * 1024 || (size_t)(r.pair ? r.M : r.n_experts * 16 * rb) * (size_t)K * 2 >= ((size_t)1 << 31)) return 1;
    switch (rb)
    {
        case 1:  return sk_launch_experts_rb<1>(r, lds, gptq, stream);
        case 2:  return sk_launch_experts_rb<2>(r, lds, gptq, stream);
        case 3:  return sk_launch_experts_rb<3>(r, lds, gptq, stream);
        default: return sk_launch_experts_rb<4>(r, lds, gptq, stream);
    }
}
