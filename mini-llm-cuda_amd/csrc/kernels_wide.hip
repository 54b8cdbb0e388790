// Decode of 6 to 64 sequences in one launch, every XCD of the MI355X a tensor-parallel rank (gfx950, wave64, fp32 weights, heads of 64).
//
// The split is that of kernels_ranks.hip: heads and FFN units over the XCDs, two exchanges of partial sums across them a layer and the rest
// inside one.  What differs is what is exchanged and who forms it.  There every workgroup gathers (value, tag) words of all rows and splits them
// into planes itself, which grows with the rows: at 16 it was 8 of 28 us a layer.  Here a value is split once, by the wave that produces it, and
// published as the planes of an MFMA operand (rows.h): a gather is the load of the next product's operand straight into registers, 6 bytes an
// element.  Planes carry no tags; the wave that has stored some waits for its stores and writes a flag word, and a wave that needs them
// polls the flags of exactly the pieces it reads.  What is small or goes across the XCDs (first phase, partial tiles) stays (value, tag) words:
// one way, no wait for the stores.
//
// Eight waves a workgroup, 32 workgroups an XCD, all waves alike: K of the first phase, gate / up and the LM head is dealt in chunks
// over the eight waves of a tile; output and down projection: four waves for tile r, four for a share of the tiles beyond the 32nd.  A layer:
//   first phase   planes of x -> q, k, v, gates                                                (words in the XCD)
//   mixing        a wave has 16 state rows of a (head, sequence), or a share of a pair's keys, or PLE columns    (planes in the XCD)
//   output proj.  partial tiles                                                                (words across the XCDs, same rank and wave)
//   residual      its columns: sum, planes of gain (.) h, sums of squares                        (planes in the XCD)
//   gate / up     -> planes of silu(gate) up                                                     (planes in the XCD)
//   down proj., residual                                                                       (as above)
// Weights, and the mixing's states, are issued one product ahead, behind the operand loads of the product before: loads return in order on this
// ISA, so a poll behind them would be answered late, and by the time of the next poll they have come.  The down projection's go out in front of the poll for
// gate / up, which waits for other workgroups anyway: behind its operands, in the waves that store nothing, a step took 1 to 3 % more (us, 6 / 16 / 48 / 64
// sequences: 253, 262, 430, 474 in front; 257, 265, 433, 488 behind).  (A ninth wave that brought them
// into the L2 instead met the others too late at the barriers: 480 us a step of 19 sequences, not 346; weights issued before the wait for
// other XCDs slow that exchange down, 5.1 us for 3.3.)  64 sequences: a workgroup has two tiles and half the tokens of a product over the whole
// width, which loads 240 KB and not 340.
//
// What bounds it: the chain of seven exchanges a layer, 1.1 to 1.4 us each inside the XCD and 3 across, and the instructions between them.  Time
// stamps, 19 sequences, a gated-delta-net layer 24 us: first phase 5.0 (of them operands and product 2.5), mixing 2.5, output projection 3.6,
// residual 3.5, gate / up 4.2, down projection 2.9, residual 2.8.  Measured, us per step (hybrid, fp32, d 768, 12 layers), row kernels and
// here: 17 sequences 443 and 312, 19 449 and 314, 33 529 and 407, 48 578 and 452, 64 610 and 512; k_decode_ranks at 16: 339 and 267.
//
// Why no buffer is overwritten while it is read: every workgroup owns tile r of the residual rows, and writes its flags behind the barriers of the
// phases before, that is after all its waves have read what those phases read.  A workgroup that writes x, q or the mixing output of the next layer, or h
// and the FFN units, has waited, itself or through the flags it waited for, for all tiles of the residual planes in between.  Across the
// XCDs wave u of rank r exchanges with wave u of rank r only, which has read the partial tiles before it stores its next ones.
//
// More than 8 heads: XCD X has head X and a share of the sequences of head 8 + X mod (heads - 8), whose weights all its sharers
// read (12 heads: 96 pairs of head and sequence an XCD for 64 sequences, not 128 on four of them and 64 on the others).
//
// The meeting at the start, bounded waits, the states' second place and what a redo finds are as in kernels_ranks.hip.
#include <string.h>

#include <algorithm>

#include "mlh_internal.h"
#include "rows_mul.h"
#include "wide_places.h"
#include "xcd_exchange.h"

#define WD_THREADS (WD_WAVES * 64)
#define WD_GRID (RK_XCDS * RK_PER)
#define WD_HD 64
#define WD_BR 16         // keys of a block: four loads of a wave each for K and V

struct WideArgs {
    StepArgs a;
    const LayerDev* layers;
    const unsigned char* ER;
    unsigned char* xw;            // exchange memory
    unsigned xwBytes, tagBase;
    int NL, steps, fs, rowsQ;     // fs: FFN units of an XCD; rowsQ: words per token of the first phase's region
    unsigned *abortFlag, *xcdCount;
    int abortAtStep;              // test hook: workgroup 0 gives up when it reaches this step (> 0)
    int otherAt;                  // floats from a sequence's gated-delta-net states to their second place
    unsigned long long sides;     // bit s: the states of sequence s are in the second place before the launch
    // What lies where: first phase, planes (mixing output, residual rows x and h, FFN units), partial sums of squares, partial tiles;
    // flags of the first phase, mixing, PLE, x, h, FFN units, partial tiles; behind all flags the candidates and the picks.
    // Words that are compared with tags lie where they do for every number of sequences: no stale data can pass for one.
    unsigned data, area, oMix, oX, oH, oU, oSX, oSH;     // data: of XCD 0, then of the others
    unsigned flags, oQ, fM, fE, fX, fH, fU, oXP, oHP, oAmax, oTok, oZero; // flags: bytes per XCD; oZero: a chunk of zeros
};

template <int MB> struct WideShared {
    f32x4 red[2][WD_WAVES][MB][64]; // partial sums: of tiles over the whole width, of the other two products
    f32x4 acc[WD_WAVES][16];        // attention: a wave's partial output, its largest score and sum
    float m[WD_WAVES], l[WD_WAVES];
    float ssq[WD_WAVES][64];        // sums of squares over a wave's columns
    int tok[64], pos[64], seq[64], ctl[4]; // ctl: leave, -, XCD, rank
};

// tiles of the first phase of a layer on an XCD with nh heads: their q, k, v (and gate) rows, the tile with its PLE gate rows, the tiles of all gate scalars
__device__ __forceinline__ int wd_tiles(LayerPtr L, int heads, int ple, int np, int nh, int& idxPle, int& idxG) {
    const bool gdn = L->kind != MLH_KIND_ATTENTION;
    int n = nh * (gdn ? 3 : np) * (WD_HD / 16);
    idxPle = n;
    if (ple > 0) n++;
    idxG = n;
    if (gdn) n += ((L->offGb + heads - 1) >> 4) - (L->offGa >> 4) + 1;
    return n;
}

template <int MB>
__global__ void __launch_bounds__(WD_THREADS, 2) k_decode_wide(WideArgs P) {
    constexpr int TS = MB == 4 ? 2 : 1, MW = MB / TS, N1 = (MB + 1) / 2; // a product over the whole width: TS tiles, MW blocks of tokens a workgroup
    extern __shared__ __align__(16) unsigned char lds[];
    WideShared<MB>& S = *reinterpret_cast<WideShared<MB>*>(lds);
    const StepArgs& a = P.a;
    const int n = a.nseq;
    if ((int)threadIdx.x < 64) {
        const int s = a.sidx[min((int)threadIdx.x, n - 1)];
        S.tok[threadIdx.x] = a.tok[min((int)threadIdx.x, n - 1)];
        S.seq[threadIdx.x] = s;
        S.pos[threadIdx.x] = a.pos[s];
        unsigned xcc, rank;
        const unsigned code = rk_meeting(P.xcdCount, xcc, rank);
        if (threadIdx.x == 0) {
            if (code) astu(P.abortFlag, code);
            S.ctl[0] = code ? 1 : 0;
            S.ctl[2] = (int)xcc;
            S.ctl[3] = (int)rank;
        }
    }
    lds_barrier();
    if (runi(S.ctl[0])) return;
    const int X = runi(S.ctl[2]), r = runi(S.ctl[3]), wave = runi((int)(threadIdx.x >> 6));
    int lane = threadIdx.x & 63, t16 = lane & 15, q = lane >> 4;
    const int d = a.dim, dt = d / 16, nch = d / 32, fs = P.fs, NL = P.NL, pleX = a.ple / RK_XCDS, npAttn = 3 + (a.gating ? 1 : 0);
    const unsigned own = P.data + (unsigned)X * P.area, ownF = (unsigned)X * P.flags; // the XCD's data and flags
    const rsrc_t W = __builtin_amdgcn_make_buffer_rsrc(P.xw, 0, P.xwBytes, 0x00027000);
    const LayerPtr layers = (LayerPtr)P.layers;
    const int stepRow = *a.stepCounter; // (advanced when everybody has read it)
    const int gw = r * RK_XCDS + X;
    // heads: X, and sequences [lo, hi) of a second one; pair p is head 0 of sequence p, then head 1 of sequence lo + p - n
    const int second = a.heads - RK_XCDS, nh = second > 0 ? 2 : 1;
    int head1 = X, lo = 0, hi = 0;
    if (second > 0) {
        const int j = X % second, sharers = (RK_XCDS - j + second - 1) / second, i = X / second;
        head1 = RK_XCDS + j; lo = n * i / sharers; hi = n * (i + 1) / sharers;
    }
    const int pairs = n + hi - lo, ko = nh * 2 + (a.ple > 0 ? 1 : 0);
    const int extra = dt - RK_PER, share = extra > 0 ? RK_PER / extra : 1; // of the tiles beyond the 32nd, each shared by as many workgroups
    int cnt, group, block0, slot2, blocks1, b1, part2, tile2, unitMb, unitTile, unitTok, g, lrow, c4;
    int fin; // the last MB waves: which block of which tile of a product over the whole width they finish
    bool on2, unit;
    unsigned unitAt;
    {
        group = r / TS; block0 = r % TS * MW;                       // tiles TS group .., blocks block0 ..
        fin = wave - (WD_WAVES - MB);
        cnt = wd_count(wave, nch);                                    // chunks wave, wave + 8, ... of a product over the whole width
        slot2 = wave >> 2; part2 = wave & 3;                        // output and down projection: tile r, or a share of the blocks of a later one; chunks part2, part2 + 4
        tile2 = slot2 ? min(RK_PER + r / share, dt - 1) : r;
        const int from1 = MB * (r % share) / share;
        blocks1 = extra > 0 ? MB * (r % share + 1) / share - from1 : 0; // the later tile's blocks: from1 .., formed in block places b1 ..
        b1 = min(from1, MB - N1);
        on2 = slot2 == 0 || blocks1 > 0;
        unit = wave < MB + blocks1;                                 // tile and block of tokens this wave finishes of those
        unitMb = wave < MB ? wave : unit ? from1 + wave - MB : 0;
        unitTile = wave < MB ? r : min(RK_PER + r / share, dt - 1);
        unitAt = (unsigned)(unitTile * MB + unitMb);
        g = wave * RK_PER + r;                                      // mixing units g and g + 256
    }
    auto place = [&]() __attribute__((always_inline)) {
        t16 = lane & 15; q = lane >> 4;
        lrow = q; c4 = t16 * 4;                                     // of a wave on rows of a head: row among four, column
        unitTok = unitMb * 16 + t16;
    };
    place();
    // What is made of the lane is formed again from here on, and not kept or moved across the phases.
    auto forget = [&]() __attribute__((always_inline)) {
        lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        place();
    };

    bool ok = true;
    auto give_up = [&](unsigned spins) { // bounded waits
        if (!ok) return true;
        if (spins > RK_SPIN || ((spins & 127) == 127 && aldu(P.abortFlag))) {
            ok = false;
            S.ctl[0] = 1;
            astu(P.abortFlag, 3u);
            return true;
        }
        return false;
    };
    auto stale = [](const u32x4& v, unsigned tag) { return (v.y ^ tag) | (v.w ^ tag); };
    auto word = [&](auto pol, unsigned off, unsigned base) __attribute__((always_inline)) { return __builtin_amdgcn_raw_buffer_load_b32(W, off, base, decltype(pol)::value); };
    auto wait1 = [&](auto pol, unsigned off, unsigned base, unsigned tag) __attribute__((always_inline)) {
        for (unsigned spins = 0;; spins++) {
            asm volatile("" ::: "memory");
            if (__all(word(pol, off, base) == tag) || give_up(spins)) break;
        }
        asm volatile("" ::: "memory");
    };
    constexpr std::integral_constant<int, LD_XCD> InXcd = {};
    // Behind the flags of what other workgroups have stored: nothing of it is taken from the compute unit's L1, whatever was loaded before.  (Values with tags
    // show what is old, planes and sums do not, and that a non-temporal load leaves no line behind is nothing the instruction set promises.  A launch takes what it took
    // without: 16 sequences 266 and 265 us a step, 32 326 and 328, 64 479 and 476.)
    auto past_l1 = [&]() __attribute__((always_inline)) { asm volatile("buffer_inv sc0" ::: "memory"); };
    auto flag = [&](auto pol, unsigned off, unsigned base, unsigned tag, bool mine) __attribute__((always_inline)) { // behind this wave's stores
        stores_landed();
        if (mine) __builtin_amdgcn_raw_buffer_store_b32(tag, W, off, base, decltype(pol)::value);
    };
    constexpr std::integral_constant<int, ST_XCD> ToXcd = {};
    auto loadF = [&](unsigned off, unsigned base) __attribute__((always_inline)) { return __uint_as_float(word(InXcd, off, base)); };
    auto loadF4 = [&](unsigned off, unsigned base) __attribute__((always_inline)) { return __builtin_bit_cast(f32x4, xget<LD_XCD>(W, off, base)); };
    auto store2 = [&](unsigned x, unsigned y, unsigned off, unsigned base) __attribute__((always_inline)) {
        const u32x2 v = {x, y};
        __builtin_amdgcn_raw_buffer_store_b64(v, W, off, base, ST_XCD);
    };
    // four neighbouring columns of a token: place `off` of plane 0 of a block, planes MB KB apart
    auto put4 = [&](const f32x4& v, unsigned off, unsigned base) __attribute__((always_inline)) {
        uint32_t x[3], y[3];
        p3_split2(v.x, v.y, x);
        p3_split2(v.z, v.w, y);
#pragma unroll
        for (int pl = 0; pl < 3; pl++) store2(x[pl], y[pl], off, base + pl * MB * 1024);
    };

    // ---- weights ----
    typedef RowsW<float> Wt;
    Wt w1[TS][WD_CA], w2[2];
    // (a wave with fewer chunks multiplies its own last operands once more, by zeros)
    const unsigned char* zeros = P.xw + P.oZero;
    auto chunk = [&](Wt& w, const void* m, size_t index, bool real) __attribute__((always_inline)) {
        w.load((real ? (const unsigned char*)m + index * 2048 : zeros) + (unsigned)lane * 16u);
    };
    auto issue1 = [&](int k, const void* m, int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WD_CA; i++) chunk(w1[k][i], m, (size_t)tile * nch + wave + WD_WAVES * i, i < cnt);
    };
    auto tilesA = [&](LayerPtr L) { int ip, ig; return wd_tiles(L, a.heads, a.ple, npAttn, nh, ip, ig); };
    auto tileA = [&](LayerPtr L, int k) { // a tile of this workgroup's in the first phase
        const int np = L->kind != MLH_KIND_ATTENTION ? 3 : npAttn;
        int idxPle, idxG;
        const int idx = min(group * TS + k, wd_tiles(L, a.heads, a.ple, npAttn, nh, idxPle, idxG) - 1);
        if (idx < idxPle) {
            const int hl = idx >= np * 4 ? 1 : 0, rem = idx - hl * (np * 4), p = rem >> 2;
            const int off = p == 0 ? 0 : p == 1 ? L->offK : p == 2 ? L->offV : L->offG;
            return ((off + (hl ? head1 : X) * WD_HD) >> 4) + (rem & 3);
        }
        if (idx < idxG) return (L->offPle + X * pleX) >> 4;
        return (L->offGa >> 4) + idx - idxG;
    };
    auto issueA = [&](LayerPtr L) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < TS; k++) issue1(k, L->WaR, tileA(L, k));
    };
    auto issue13 = [&](LayerPtr L) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < TS; k++) issue1(k, L->W13R, X * (fs / 8) + min(group * TS + k, fs / 8 - 1));
    };
    auto head_tile = [&](int round, int k) { return ((group * RK_XCDS + X) * TS + k) + round * WD_GRID; };
    auto issueO = [&](LayerPtr L) __attribute__((always_inline)) {
        const int total = ((int)L->ad + a.ple) / 32;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int c = part2 + 4 * i;
            const int gc = c < nh * 2 ? (c < 2 ? X : head1) * 2 + (c & 1) : ((int)L->ad + X * pleX) / 32;
            chunk(w2[i], L->WoR, (size_t)tile2 * total + gc, c < ko);
        }
    };
    auto issueW2 = [&](LayerPtr L) __attribute__((always_inline)) {
        const int k = fs / 32;
#pragma unroll
        for (int i = 0; i < 2; i++) chunk(w2[i], L->W2R, (size_t)tile2 * (RK_XCDS * k) + X * k + part2 + 4 * i, part2 + 4 * i < k);
    };

    // Where the flags lie that this lane reads (wide_places.h): of the pieces of residual planes, of the mixing output (a chunk's two units for 64
    // sequences, or the PLE columns' blocks) and of the FFN units.
    unsigned flag1, flagM[4], flagU;
    {
        flag1 = (unsigned)wd_flag1(lane, wave, cnt, MB, MW, block0) * 4u;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int c2 = wd_mix_chunk(part2, k, ko, nh, lo >= hi), hl = c2 >> 1;
            const bool ple = c2 >= nh * 2;
            flagM[2 * k] = ple ? P.fE + (unsigned)min(lane, MB - 1) * 4u : P.fM + (unsigned)wd_flagM(lane, c2, hl ? lo : 0, hl ? hi : n) * 4u;
            flagM[2 * k + 1] = flagM[2 * k] + (ple ? 0u : 256u);
        }
        flagU = (unsigned)wd_flagU(lane, part2, fs / 32, MB) * 4u;
        asm volatile("" : "+v"(flag1), "+v"(flagM[0]), "+v"(flagM[1]), "+v"(flagM[2]), "+v"(flagM[3]), "+v"(flagU));
    }

    // ---- products ----
    constexpr int NA = MW <= 2 ? WD_CA : 2; // chunks whose operands are in registers or on their way
    auto operand = [&](auto& v, int kb, int b0, unsigned planes) __attribute__((always_inline)) { // blocks b0 ..
        constexpr int N = sizeof(v[0][0]) / sizeof(u32x4);
        const unsigned base = own + planes + (unsigned)(kb * 3 * MB + b0) * 1024u;
#pragma unroll
        for (int pl = 0; pl < 3; pl++)
#pragma unroll
            for (int mb = 0; mb < N; mb++) v[0][pl][mb] = xget<LD_XCD>(W, (unsigned)lane * 16u + (unsigned)(pl * MB + mb) * 1024u, base);
    };
    auto times = [&](const Wt& w, const auto& v, auto& acc) __attribute__((always_inline)) {
        constexpr int N = sizeof(acc) / sizeof(f32x4);
        Wt x = w;
        asm volatile("" : "+v"(x.raw[0]), "+v"(x.raw[1])); // split here, not behind the loads
        x.template mul<N>(v, acc);
    };
    // This wave's chunks of residual planes times w1 -> the partial sums of the tiles' eight waves; beside them the sums of squares over its columns.
    auto product1 = [&](int buf, unsigned planes, unsigned ssq, bool first, unsigned flags, unsigned tag, auto&& behind) __attribute__((always_inline)) {
        if (first) { wait1(InXcd, flag1, ownF + flags, tag); past_l1(); }
        float s[2 * WD_CA];
#pragma unroll
        for (int k = 0; k < WD_CA; k++) {
            const unsigned at = own + ssq + (unsigned)wd_chunk(wave, k, cnt) * 512u + (unsigned)block0 * 64u;
            s[2 * k] = loadF((unsigned)min(lane, MW * 16 - 1) * 4u, at);
            s[2 * k + 1] = loadF((unsigned)min(lane, MW * 16 - 1) * 4u, at + 256u);
        }
        u32x4 av[NA][1][3][MW] = {};
#pragma unroll
        for (int k = 0; k < NA; k++) operand(av[k], wd_chunk(wave, k, cnt), block0, planes);
        f32x4 acc[TS][MW];
#pragma unroll
        for (int t = 0; t < TS; t++)
#pragma unroll
            for (int mb = 0; mb < MW; mb++) acc[t][mb] = (f32x4)(0.f);
#pragma unroll
        for (int k = 0; k < WD_CA; k++) {
#pragma unroll
            for (int t = 0; t < TS; t++) times(w1[t][k], av[k % NA], acc[t]);
            __builtin_amdgcn_sched_barrier(0);
            if (k + NA < WD_CA) operand(av[k % NA], wd_chunk(wave, k + NA, cnt), block0, planes);
            if (k == 0) { // (the last operands are on their way)
                asm volatile("" ::: "memory");
                behind();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < WD_CA; k++) sum += k < cnt ? s[2 * k] + s[2 * k + 1] : 0.f;
        S.ssq[wave][lane] = sum;
#pragma unroll
        for (int t = 0; t < TS; t++)
#pragma unroll
            for (int mb = 0; mb < MW; mb++) S.red[buf][wave][t * MW + mb][lane] = acc[t][mb];
    };
    auto finish1 = [&](int buf) __attribute__((always_inline)) { // block fin % MW of tile fin / MW, normalised (fin >= 0)
        f32x4 t[WD_WAVES];
        float s[WD_WAVES];
#pragma unroll
        for (int k = 0; k < WD_WAVES; k++) { t[k] = S.red[buf][k][fin][lane]; s[k] = S.ssq[k][fin % MW * 16 + t16]; }
        const float ss = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
        return (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) * (1.0f / sqrtf(ss / (float)d + 1e-8f));
    };
    // Chunks part2, part2 + 4 (< k) of `planes`, N blocks from b0 on -> the partial sums of the tile's four waves.
    auto product2 = [&](auto blocks, int b0, int k, unsigned planes, bool mixed, auto&& behind) __attribute__((always_inline)) {
        constexpr int N = decltype(blocks)::value;
        u32x4 av[2][1][3][N] = {};
#pragma unroll
        for (int i = 0; i < 2; i++) operand(av[i], wd_part(part2, i, k), b0, planes);
        asm volatile("" ::: "memory");
        behind();
        f32x4 acc[N];
#pragma unroll
        for (int mb = 0; mb < N; mb++) acc[mb] = (f32x4)(0.f);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int c = wd_part(part2, i, k);
            if (mixed) { // sequences of the second head that another XCD has
                const bool some = c >= 2 && c < nh * 2;
#pragma unroll
                for (int mb = 0; mb < N; mb++) {
                    const int m = (b0 + mb) * 16 + t16;
                    const bool in = !some || (m >= lo && m < hi);
#pragma unroll
                    for (int pl = 0; pl < 3; pl++) av[i][0][pl][mb] = in ? av[i][0][pl][mb] : (u32x4)(0u);
                }
            }
            times(w2[i], av[i], acc);
        }
#pragma unroll
        for (int mb = 0; mb < N; mb++) S.red[1][wave][mb][lane] = acc[mb];
    };
    auto project = [&](int k, unsigned planes, bool mixed, auto&& behind) __attribute__((always_inline)) {
        if (slot2 == 0) product2(std::integral_constant<int, MB>(), 0, k, planes, mixed, behind);
        else product2(std::integral_constant<int, N1>(), b1, k, planes, mixed, behind);
    };
    // partial tiles to the other XCDs (behind a barrier)
    auto publish2 = [&](unsigned to, unsigned tag) __attribute__((always_inline)) {
        if (!unit) return;
        f32x4 t[4];
#pragma unroll
        for (int k = 0; k < 4; k++) t[k] = S.red[1][(wave < MB ? 0 : 4) + k][wave < MB ? wave : unitMb - b1][lane];
        const f32x4 v = (t[0] + t[1]) + (t[2] + t[3]);
        xput<ST_CROSS>(W, (unsigned)lane * 16u, ownF + to + unitAt * 2048u, v.x, v.y, tag);
        xput<ST_CROSS>(W, (unsigned)lane * 16u, ownF + to + unitAt * 2048u + 1024u, v.z, v.w, tag);
    };
    // The residual elements of this wave's unit: columns 4 q .. 4 q + 3 of its tile, token unitTok.
    f32x4 resid = (f32x4)(0.f);
    auto publish_rows = [&](const f32x4& gain, unsigned planes, unsigned ssq, unsigned flags, unsigned tag) __attribute__((always_inline)) {
        float s = resid.x * resid.x;
        s = fmaf(resid.y, resid.y, s); s = fmaf(resid.z, resid.z, s); s = fmaf(resid.w, resid.w, s);
        put4(f32x4{gain.x * resid.x, gain.y * resid.y, gain.z * resid.z, gain.w * resid.w}, (unsigned)(q * 16 + t16) * 16u + (unsigned)(unitTile & 1) * 8u,
             own + planes + (unsigned)((unitTile >> 1) * 3 * MB + unitMb) * 1024u);
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (q == 0) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s), W, (unsigned)(unitTile * 64 + unitTok) * 4u, own + ssq, ST_XCD);
        flag(ToXcd, unitAt * 4u, ownF + flags, tag, lane == 0);
    };
    auto gain_of = [&](const float* p) { return *reinterpret_cast<const f32x4*>(p + unitTile * 16 + 4 * q); };
    auto residual = [&](unsigned partials, unsigned ptag, const f32x4& gain, unsigned planes, unsigned ssq, unsigned flags, unsigned tag) __attribute__((always_inline)) {
        if (!unit) return;
        u32x4 w[RK_XCDS][2];
        for (unsigned spins = 0;; spins++) {
            asm volatile("" ::: "memory");
            unsigned old = 0u;
#pragma unroll
            for (int x = 0; x < RK_XCDS; x++)
#pragma unroll
                for (int k = 0; k < 2; k++) w[x][k] = xget<LD_CROSS>(W, lane * 16, (unsigned)x * P.flags + partials + unitAt * 2048u + k * 1024u);
#pragma unroll
            for (int x = 0; x < RK_XCDS; x++) old |= stale(w[x][0], ptag) | stale(w[x][1], ptag);
            if (__all(old == 0u) || give_up(spins)) break;
        }
        f32x4 s = (f32x4)(0.f); // fixed order
#pragma unroll
        for (int x = 0; x < RK_XCDS; x++) s += f32x4{__uint_as_float(w[x][0].x), __uint_as_float(w[x][0].z), __uint_as_float(w[x][1].x), __uint_as_float(w[x][1].z)};
        resid += s;
        publish_rows(gain, planes, ssq, flags, tag);
    };

    // ---- token mixing ----
    auto pair_of = [&](int p, int& hl, int& tok) { hl = p >= n ? 1 : 0; tok = hl ? lo + p - n : p; };
    unsigned stateAt[2] = {0u, 0u}; // this lane's first state row of the wave's units, as read in the step
    auto states = [&](int step) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            int hl, tok;
            const int u = min(g + i * 256, pairs * 4 - 1);
            pair_of(u >> 2, hl, tok);
            const int seq = runi(S.seq[tok]);
            const bool other = ((P.sides >> seq & 1) != 0) == (step == 0);
            stateAt[i] = (unsigned)(((seq * a.gdnHeads + (hl ? head1 : X)) * WD_HD + (u & 3) * 16 + lrow * 4) * WD_HD + c4 + (other ? P.otherAt : 0));
        }
    };
    const int pw = (pairs + RK_PER - 1) / RK_PER, wp = pw > 2 ? 2 : pw > 1 ? 4 : 8; // attention: pairs of a workgroup, waves of a pair
    const int aPair = (wave / wp) * RK_PER + r, aSplit = wave % wp;
    const bool aOn = aPair < pairs;
    int aHl = 0, aTok = 0;
    if (aOn) pair_of(aPair, aHl, aTok);
    const int aSeq = runi(S.seq[aTok]), aHead = aHl ? head1 : X, pages = a.pageTable[aSeq * a.pagesPerSeq + min(lane, a.pagesPerSeq - 1)]; // lane i: page i

    issueA(layers + NL - 1);
    for (int step = 0; step < P.steps; step++) {
        const unsigned t0 = P.tagBase + (unsigned)(step * (NL + 1)) + 1u; // tag of the first layer
        lds_barrier(); // tokens and positions
        if (runi(S.ctl[0])) return;
        if (P.abortAtStep > 0 && step == P.abortAtStep && gw == 0) { ok = false; S.ctl[0] = 1; astu(P.abortFlag, 3u); }
        forget();
        if (step < 2) states(step);
        if (unit) { // the embedding (inference.cu:9-22)
            resid = *reinterpret_cast<const f32x4*>((const float*)a.E + (size_t)S.tok[unitTok] * d + unitTile * 16 + 4 * q);
            publish_rows(gain_of(layers[NL - 1].g1), P.oX, P.oSX, P.fX, t0);
        }
#pragma unroll 1
        for (int l = 0; l < NL; l++) {
            const LayerPtr L = layers + (NL - 1 - l); // file block 0 is the top (inference.cu:384-385)
            const unsigned lt = t0 + (unsigned)l;
            const bool gdn = L->kind != MLH_KIND_ATTENTION, last = l + 1 == NL;
            forget();
            const int nt = tilesA(L);
            // ---------------------------------------------------------------- first phase (inference.cu:388-465)
            f32x4 st[2][4] = {}; // state rows of the wave's two units of the mixing
            auto behind1 = [&]() __attribute__((always_inline)) {
                issueO(L);
                if (gdn)
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const float* p = L->S + stateAt[i];
#pragma unroll
                        for (int k = 0; k < 4; k++) st[i][k] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p + k * WD_HD));
                    }
            };
            if (group * TS < nt) product1(0, P.oX, P.oSX, true, P.fX, lt, behind1);
            else behind1();
            lds_barrier();
            if (fin >= 0 && group * TS + fin / MW < nt) {
                const f32x4 v = finish1(0);
                const int m = (block0 + fin % MW) * 16 + t16;
                if (m < n) {
                    const unsigned o = (unsigned)(m * P.rowsQ + (group * TS + fin / MW) * 16 + 4 * q) * 8u;
                    xput<ST_XCD>(W, o, ownF + P.oQ, v.x, v.y, lt);
                    xput<ST_XCD>(W, o + 16u, ownF + P.oQ, v.z, v.w, lt);
                }
            }
            // ---------------------------------------------------------------- token mixing
            forget();
            int idxPle, idxG;
            wd_tiles(L, a.heads, a.ple, npAttn, nh, idxPle, idxG);
            auto qget = [&](unsigned off, unsigned base) __attribute__((always_inline)) { return xget<LD_XCD>(W, off, base); };
            auto four = [&](const u32x4& x, const u32x4& y) { return f32x4{__uint_as_float(x.x), __uint_as_float(x.z), __uint_as_float(y.x), __uint_as_float(y.z)}; };
            if (gdn) {
                // state rows: u = S k; S <- alpha (S - beta u k^T) + beta v k^T; o = S q
                const int units = pairs * 4;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int u = g + i * 256;
                    if (u >= units) continue;
                    int hl, tok;
                    pair_of(u >> 2, hl, tok);
                    const int head = hl ? head1 : X;
                    const float ba = L->gdnBa[head], bb = L->gdnBb[head];
                    const unsigned row = ownF + P.oQ + (unsigned)(tok * P.rowsQ + hl * 3 * WD_HD) * 8u;
                    const unsigned grow = ownF + P.oQ + (unsigned)(tok * P.rowsQ + idxG * 16 + (L->offGa & 15) + head) * 8u, gstep = (unsigned)(L->offGb - L->offGa) * 8u;
                    u32x4 w[6];
                    u32x2 ga, gz;
                    for (unsigned spins = 0;; spins++) {
                        asm volatile("" ::: "memory");
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            w[k] = qget(c4 * 8 + k * 16, row);
                            w[2 + k] = qget(c4 * 8 + k * 16 + WD_HD * 8, row);
                            w[4 + k] = qget(lrow * 32 + k * 16 + 2 * WD_HD * 8, row + (u & 3) * 128);
                        }
                        ga = __builtin_amdgcn_raw_buffer_load_b64(W, 0u, grow, LD_XCD);
                        gz = __builtin_amdgcn_raw_buffer_load_b64(W, 0u, grow + gstep, LD_XCD);
                        unsigned old = (ga.y ^ lt) | (gz.y ^ lt);
#pragma unroll
                        for (int k = 0; k < 6; k++) old |= stale(w[k], lt);
                        if (__all(old == 0u) || give_up(spins)) break;
                    }
                    f32x4 qv = four(w[0], w[1]), kv = four(w[2], w[3]);
                    const f32x4 vv = four(w[4], w[5]);
                    const float za = __uint_as_float(ga.x) + ba, zb = __uint_as_float(gz.x) + bb;
                    float sq = 0.f, sk = 0.f;
#pragma unroll
                    for (int e = 0; e < 4; e++) { sq = fmaf(qv[e], qv[e], sq); sk = fmaf(kv[e], kv[e], sk); }
                    qv *= rsqrtf(pgroup_sum<16>(sq) + 1e-6f);
                    kv *= rsqrtf(pgroup_sum<16>(sk) + 1e-6f);
                    const float alpha = psigmoid(-za), beta = psigmoid(zb); // (exp(-softplus(z)) = sigmoid(-z))
                    f32x4 o;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        f32x4& s = st[i][k];
                        float x = s.x * kv.x;
                        x = fmaf(s.y, kv.y, x); x = fmaf(s.z, kv.z, x); x = fmaf(s.w, kv.w, x);
                        x = pgroup_sum<16>(x);
                        const float bu = beta * x, bv = beta * vv[k];
                        s.x = fmaf(alpha, s.x - bu * kv.x, bv * kv.x); s.y = fmaf(alpha, s.y - bu * kv.y, bv * kv.y);
                        s.z = fmaf(alpha, s.z - bu * kv.z, bv * kv.z); s.w = fmaf(alpha, s.w - bu * kv.w, bv * kv.w);
                        float y = s.x * qv.x;
                        y = fmaf(s.y, qv.y, y); y = fmaf(s.z, qv.z, y); y = fmaf(s.w, qv.w, y);
                        o[k] = pgroup_sum<16>(y);
                    }
                    if (t16 == 0)
                        put4(o, (unsigned)(lrow * 16 + (tok & 15)) * 16u + (unsigned)(u & 1) * 8u,
                             own + P.oMix + (unsigned)((hl * 2 + ((u & 3) >> 1)) * 3 * MB + (tok >> 4)) * 1024u);
                    flag(ToXcd, (unsigned)((hl * 4 + (u & 3)) * 64 + tok) * 4u, ownF + P.fM, lt, lane == 0);
                    if (ok) {
                        float* p = L->S + stateAt[i];
                        if (step == 0) p += P.sides >> runi(S.seq[tok]) & 1 ? -P.otherAt : P.otherAt; // to the place it was not read from
#pragma unroll
                        for (int k = 0; k < 4; k++) *reinterpret_cast<f32x4*>(p + k * WD_HD) = st[i][k];
                    }
                }
            } else {
                // key blocks s, s + wp, ... of a pair; split 0 adds this step's own row
                const int p = runi(S.pos[aTok]), nblk = (p + WD_BR - 1) / WD_BR;
                float m = -1.0e30f, lsum = 0.f; // of this lane's row group
                f32x4 acc = (f32x4)(0.f);
                if (aOn) {
                    auto key_base = [&](int j) { // row 0 of key block j
                        const int pg = j * WD_BR / MLH_KV_PAGE;
                        const int page = pg < 64 ? __builtin_amdgcn_readlane(pages, pg) : runi(a.pageTable[aSeq * a.pagesPerSeq + pg]);
                        return ((size_t)page * MLH_KV_PAGE + (j * WD_BR) % MLH_KV_PAGE) * d + aHead * WD_HD;
                    };
                    auto key_rows = [&](int j, f32x4 (&kv)[8]) __attribute__((always_inline)) { // (rows at and beyond p are not read: they may be written any time)
                        const size_t base = key_base(j);
                        const float *K = L->K + base, *V = L->V + base;
#pragma unroll
                        for (int it = 0; it < 4; it++) {
                            const unsigned o = (unsigned)(min(it * 4 + lrow, p - 1 - j * WD_BR) * d + c4);
                            kv[it] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(K + o));
                            kv[it + 4] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(V + o));
                        }
                    };
                    f32x4 kv[3][8] = {}; // three blocks of keys on their way: K, then V (none left: the last one again, from the cache)
                    if (aSplit < nblk)
#pragma unroll
                        for (int k = 0; k < 3; k++) key_rows(min(aSplit + k * wp, nblk - 1), kv[k]);
                    const f32x4 rot = *reinterpret_cast<const f32x4*>(a.rope + (size_t)p * WD_HD + c4);
                    f32x4 gq = (f32x4)(1.f), gk = (f32x4)(1.f);
                    if (a.qkNorm) {
                        gq = *reinterpret_cast<const f32x4*>(L->gq + aHead * WD_HD + c4);
                        gk = *reinterpret_cast<const f32x4*>(L->gk + aHead * WD_HD + c4);
                    }
                    const unsigned row = ownF + P.oQ + (unsigned)(aTok * P.rowsQ + aHl * npAttn * WD_HD) * 8u;
                    u32x4 w[6];
                    for (unsigned spins = 0;; spins++) {
                        asm volatile("" ::: "memory");
                        unsigned old = 0u;
#pragma unroll
                        for (int k = 0; k < 6; k++) w[k] = qget(c4 * 8 + (k & 1) * 16 + (k >> 1) * WD_HD * 8, row);
#pragma unroll
                        for (int k = 0; k < 6; k++) old |= stale(w[k], lt);
                        if (__all(old == 0u) || give_up(spins)) break;
                    }
                    auto norm_rope = [&](f32x4 v, const f32x4& gn) { // inference.cu:52-134
                        if (a.qkNorm) {
                            float ss = v.x * v.x;
                            ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
                            const float ri = rsqrtf(pgroup_sum<16>(ss) * (1.0f / WD_HD) + 1e-8f);
                            v.x = gn.x * (v.x * ri); v.y = gn.y * (v.y * ri); v.z = gn.z * (v.z * ri); v.w = gn.w * (v.w * ri);
                        }
                        return f32x4{rot.x * v.x - rot.y * v.y, rot.y * v.x + rot.x * v.y, rot.z * v.z - rot.w * v.w, rot.w * v.z + rot.z * v.w};
                    };
                    const f32x4 qv = norm_rope(four(w[0], w[1]), gq), kn = norm_rope(four(w[2], w[3]), gk), vn = four(w[4], w[5]);
                    auto dot = [&](const f32x4& k) {
                        float z = k.x * qv.x;
                        z = fmaf(k.y, qv.y, z); z = fmaf(k.z, qv.z, z); z = fmaf(k.w, qv.w, z);
                        return pgroup_sum<16>(z) * 0.125f; // 1 / sqrt(64)
                    };
                    const float sn = dot(kn);
                    if (aSplit == 0 && lrow == 0) {
                        m = sn; lsum = 1.f; acc = vn;
                        if (ok) {
                            const size_t o = key_base(p / WD_BR) + (size_t)(p % WD_BR) * d + c4;
                            *reinterpret_cast<f32x4*>(L->K + o) = kn;
                            *reinterpret_cast<f32x4*>(L->V + o) = vn;
                        }
                    }
                    auto keys = [&](int j, auto& kv) __attribute__((always_inline)) {
                        float sc[4];
#pragma unroll
                        for (int it = 0; it < 4; it++) {
                            sc[it] = dot(kv[it]);
                            sc[it] = j * WD_BR + it * 4 + lrow < p ? sc[it] : -1.0e30f;
                        }
                        const float mn = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), m), corr = expf(m - mn);
                        lsum *= corr;
                        acc *= corr;
#pragma unroll
                        for (int it = 0; it < 4; it++) {
                            const float e = j * WD_BR + it * 4 + lrow < p ? expf(sc[it] - mn) : 0.f;
                            lsum += e;
                            acc.x = fmaf(e, kv[it + 4].x, acc.x); acc.y = fmaf(e, kv[it + 4].y, acc.y);
                            acc.z = fmaf(e, kv[it + 4].z, acc.z); acc.w = fmaf(e, kv[it + 4].w, acc.w);
                        }
                        m = mn;
                    };
                    for (int j = aSplit; j < nblk; j += 3 * wp)
#pragma unroll
                        for (int k = 0; k < 3; k++) {
                            const int jk = j + k * wp;
                            if (jk < nblk) keys(jk, kv[k]);
                            __builtin_amdgcn_sched_barrier(0);
                            if (jk + 3 * wp < nblk) key_rows(jk + 3 * wp, kv[k]);
                            __builtin_amdgcn_sched_barrier(0);
                        }
#pragma unroll
                    for (int o = 16; o < 64; o <<= 1) { // the row groups of the wave
                        const float mo = __shfl_xor(m, o, 64), lo2 = __shfl_xor(lsum, o, 64);
                        f32x4 ao;
                        ao.x = __shfl_xor(acc.x, o, 64); ao.y = __shfl_xor(acc.y, o, 64); ao.z = __shfl_xor(acc.z, o, 64); ao.w = __shfl_xor(acc.w, o, 64);
                        const float mm = fmaxf(m, mo), ca = expf(m - mm), cb = expf(mo - mm);
                        lsum = lsum * ca + lo2 * cb;
                        acc = acc * ca + ao * cb;
                        m = mm;
                    }
                    if (lane < 16) S.acc[wave][lane] = acc;
                    if (lane == 0) { S.m[wave] = m; S.l[wave] = lsum; }
                }
                lds_barrier();
                if (aOn && aSplit == 0) { // the waves of the pair
                    float mm = -1.0e30f, den = 0.f;
                    f32x4 num = (f32x4)(0.f);
                    for (int k = 0; k < wp; k++) mm = fmaxf(mm, S.m[wave + k]);
                    for (int k = 0; k < wp; k++) {
                        const float c = expf(S.m[wave + k] - mm);
                        den = fmaf(c, S.l[wave + k], den);
                        num += S.acc[wave + k][t16] * c;
                    }
                    num *= 1.0f / den;
                    if (a.gating) { // inference.cu:241-250
                        const unsigned grow = ownF + P.oQ + (unsigned)(aTok * P.rowsQ + (aHl * npAttn + 3) * WD_HD) * 8u;
                        u32x4 w0, w1g;
                        for (unsigned spins = 0;; spins++) {
                            asm volatile("" ::: "memory");
                            w0 = qget(c4 * 8, grow); w1g = qget(c4 * 8 + 16, grow);
                            if (__all(xfresh(w0, lt) && xfresh(w1g, lt)) || give_up(spins)) break;
                        }
                        const f32x4 z = four(w0, w1g);
                        num.x *= psigmoid(z.x); num.y *= psigmoid(z.y); num.z *= psigmoid(z.z); num.w *= psigmoid(z.w);
                    }
                    if (lane < 16)
                        put4(num, (unsigned)((t16 & 3) * 16 + (aTok & 15)) * 16u + (unsigned)((t16 >> 2) & 1) * 8u + (unsigned)((t16 >> 3) * 3 * MB) * 1024u,
                             own + P.oMix + (unsigned)(aHl * 2 * 3 * MB + (aTok >> 4)) * 1024u);
                    flag(ToXcd, (unsigned)((aHl * 4 + (lane & 3)) * 64 + aTok) * 4u, ownF + P.fM, lt, lane < 4);
                }
            }
            forget();
            if (a.ple > 0 && g >= 256 - MB) { // block 255 - g of the tokens: e = silu(gate) * P[tok] in its chunk of the output projection, the other XCDs' columns zero
                const int j = 255 - g, tok = min(j * 16 + t16, n - 1), off = ((int)L->ad + X * pleX) % 32;
                u32x4 w[3];
#pragma unroll
                for (int half = 0; half < 2; half++) {
                    const int c = half * 16 + 4 * q - off; // of the XCD's columns
                    const bool in = c >= 0 && c < pleX;
                    const unsigned at = (unsigned)(tok * P.rowsQ + (in ? c : 0)) * 8u, base = ownF + P.oQ + (unsigned)(idxPle * 16 + ((L->offPle + X * pleX) & 15)) * 8u;
                    const f32x4 t = *reinterpret_cast<const f32x4*>((const float*)L->pleTable + (size_t)S.tok[tok] * a.ple + X * pleX + (in ? c : 0));
                    u32x4 x0, x1;
                    for (unsigned spins = 0;; spins++) {
                        asm volatile("" ::: "memory");
                        x0 = qget(at, base); x1 = qget(at + 16u, base);
                        if (__all(xfresh(x0, lt) && xfresh(x1, lt)) || give_up(spins)) break;
                    }
                    const f32x4 z = four(x0, x1);
                    const f32x4 e = in ? f32x4{psilu(z.x) * t.x, psilu(z.y) * t.y, psilu(z.z) * t.z, psilu(z.w) * t.w} : (f32x4)(0.f);
                    uint32_t x[3], y[3];
                    p3_split2(e.x, e.y, x);
                    p3_split2(e.z, e.w, y);
#pragma unroll
                    for (int pl = 0; pl < 3; pl++) { w[pl][2 * half] = x[pl]; w[pl][2 * half + 1] = y[pl]; }
                }
#pragma unroll
                for (int pl = 0; pl < 3; pl++)
                    __builtin_amdgcn_raw_buffer_store_b128(w[pl], W, lane * 16, own + P.oMix + (unsigned)((nh * 2 * 3 + pl) * MB + j) * 1024u, ST_XCD);
                flag(ToXcd, (unsigned)j * 4u, ownF + P.fE, lt, lane == 0);
            }
            // ---------------------------------------------------------------- output projection over the XCD's columns (inference.cu:582-610)
            forget();
            if (on2) {
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
                    const unsigned a0 = word(InXcd, flagM[0], ownF), a1 = word(InXcd, flagM[1], ownF), a2 = word(InXcd, flagM[2], ownF), a3 = word(InXcd, flagM[3], ownF);
                    if (__all(((a0 ^ lt) | (a1 ^ lt) | (a2 ^ lt) | (a3 ^ lt)) == 0) || give_up(spins)) break;
                }
                past_l1();
                project(ko, P.oMix, true, [&]() __attribute__((always_inline)) { issue13(L); });
            } else issue13(L);
            lds_barrier();
            forget();
            const f32x4 g2 = gain_of(L->g2);
            publish2(P.oHP, lt);
            residual(P.oHP, lt, g2, P.oH, P.oSH, P.fH, lt);
            issueW2(L); // in front of the poll: behind the product's operands its stores would wait for these
            // ---------------------------------------------------------------- gate / up of the XCD's FFN units (inference.cu:612-672)
            forget();
            if (group * TS < fs / 8) product1(0, P.oH, P.oSH, true, P.fH, lt, [&]() {});
            lds_barrier();
            if (fin >= 0) {
                const int tile = group * TS + fin / MW, block = block0 + fin % MW;
                if (tile < fs / 8) {
                    const f32x4 v = finish1(0);
                    uint32_t s[3];
                    p3_split2(psilu(v.x) * v.y, psilu(v.z) * v.w, s);
                    const int j = tile * 8 + 2 * q; // units j, j + 1
                    const unsigned o = (unsigned)(((j & 15) >> 2) * 16 + t16) * 16u + (unsigned)((j & 16) >> 1) + (unsigned)(j & 2) * 2u;
#pragma unroll
                    for (int pl = 0; pl < 3; pl++)
                        __builtin_amdgcn_raw_buffer_store_b32(s[pl], W, o, own + P.oU + (unsigned)(((tile >> 2) * 3 + pl) * MB + block) * 1024u, ST_XCD);
                    flag(ToXcd, (unsigned)(tile * MB + block) * 4u, ownF + P.fU, lt, lane == 0);
                }
            }
            // ---------------------------------------------------------------- down projection over the XCD's columns (inference.cu:675-699)
            forget();
            const LayerPtr Ln = layers + (last ? NL - 1 : NL - 2 - l);
            auto issue_next = [&]() __attribute__((always_inline)) { // (the LM head's first tile behind the last layer; one set of loads with selected addresses)
#pragma unroll
                for (int k = 0; k < TS; k++) issue1(k, last ? P.ER : (const unsigned char*)Ln->WaR, last ? min(head_tile(0, k), (a.vocab + 15) / 16 - 1) : tileA(Ln, k));
            };
            if (on2) {
                const int k = fs / 32;
                wait1(InXcd, flagU, ownF + P.fU, lt);
                past_l1();
                project(k, P.oU, false, issue_next);
            } else issue_next();
            lds_barrier();
            forget();
            const f32x4 g1 = gain_of(last ? a.gF : Ln->g1);
            publish2(P.oXP, lt);
            residual(P.oXP, lt, g1, P.oX, P.oSX, P.fX, lt + 1);
            if (runi(S.ctl[0])) return;
        }
        // -------------------------------------------------------------------- LM head (inference.cu:705-743)
        forget();
        const unsigned ht = t0 + (unsigned)NL;
        const int tiles = (a.vocab + 15) / 16;
        float best = -3.0e38f;
        int bi = 0x7fffffff;
        const int rounds = head_tile(0, 0) < tiles ? (tiles - head_tile(0, 0) + WD_GRID - 1) / WD_GRID : 0, tokHead = (block0 + max(fin, 0) % MW) * 16 + t16;
#pragma unroll 1
        for (int k = 0; k < rounds; k++) {
            product1(k & 1, P.oX, P.oSX, k == 0, P.fX, ht, [&]() {});
            if (k + 1 < rounds)
#pragma unroll
                for (int t = 0; t < TS; t++) issue1(t, P.ER, min(head_tile(k + 1, t), tiles - 1));
            lds_barrier();
            if (fin >= 0) {
                const f32x4 v = finish1(k & 1);
                const int m = tokHead, nn = head_tile(k, fin / MW) * 16 + 4 * q;
                if (m < n && nn < a.vocab) {
                    float* c = a.logits + (size_t)S.seq[m] * a.vocab + nn;
                    if ((a.vocab & 3) == 0) *reinterpret_cast<f32x4*>(c) = v;
                    else
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (nn + e < a.vocab) c[e] = v[e];
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (nn + e < a.vocab && v[e] > best) { best = v[e]; bi = nn + e; }
                }
            }
        }
        if (fin >= 0) { // the workgroup's candidates, lowest index on ties
#pragma unroll
            for (int o = 16; o < 64; o <<= 1) {
                const float ov = __shfl_xor(best, o, 64);
                const int oi = __shfl_xor(bi, o, 64);
                if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
            }
            if (q == 0 && tokHead < n) xput<ST_CROSS>(W, (unsigned)(tokHead * WD_GRID + (group * RK_XCDS + X) * TS + fin / MW) * 16u, P.oAmax, best, __int_as_float(bi), ht);
        }
        issueA(layers + NL - 1);
        // the pick: token slot s is decided by workgroup s out of a candidate per workgroup
        if (wave == 0) {
            if (gw < n) {
                u32x4 c[WD_GRID / 64];
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
                    bool all = true;
#pragma unroll
                    for (int k = 0; k < WD_GRID / 64; k++) c[k] = xget<LD_CROSS>(W, (unsigned)(k * 64 + lane) * 16u, P.oAmax + (unsigned)(gw * WD_GRID) * 16u);
#pragma unroll
                    for (int k = 0; k < WD_GRID / 64; k++) all = all && xfresh(c[k], ht);
                    if (__all(all) || give_up(spins)) break;
                }
                float v = -3.0e38f;
                int i = 0x7fffffff;
#pragma unroll
                for (int k = 0; k < WD_GRID / 64; k++) {
                    const float v2 = __uint_as_float(c[k].x);
                    const int i2 = (int)c[k].z;
                    if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
                }
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const float v2 = __shfl_xor(v, o, 64);
                    const int i2 = __shfl_xor(i, o, 64);
                    if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
                }
                if (i < 0 || i >= a.vocab) i = 0; // only reachable with non-finite logits
                if (lane == 0 && ok) {
                    xput<ST_CROSS>(W, (unsigned)gw * 16u, P.oTok, __int_as_float(i), 0.f, ht);
                    const int row = stepRow + step, seq = S.seq[gw];
                    if (row >= 0 && row < a.outCapacity) a.outIds[(size_t)row * a.nseq + gw] = i;
                    if (step + 1 == P.steps) {
                        a.nextTok[seq] = i;
                        ((int*)a.tok)[gw] = i;
                        a.pos[seq] = S.pos[gw] + 1;
                        if (gw == 0) *a.stepCounter = stepRow + P.steps;
                    }
                }
            }
            if (step + 1 < P.steps) {
                u32x4 c;
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
                    c = xget<LD_CROSS>(W, (unsigned)min(lane, n - 1) * 16u, P.oTok);
                    if (__all(xfresh(c, ht)) || give_up(spins)) break;
                }
                if (ok) { S.tok[lane] = (int)c.x; S.pos[lane] += 1; }
            }
        }
    }
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------
struct WidePlan { // how a launch of n sequences is laid out
    int rowsQ;
    size_t lds, words;
    unsigned data, area, oMix, oX, oH, oU, oSX, oSH;
    unsigned flags, oQ, fM, fE, fX, fH, fU, oXP, oHP, oAmax, oTok, oZero;
};

static int blocks_of(int n) { return (n + 15) / 16; }

// tiles of the first phase on an XCD, at most
static int first_tiles(const mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    const int nh = hp.attnHeads > RK_XCDS ? 2 : 1;
    int tiles = 0;
    for (const LayerDev& L : c->layers) {
        const bool gdn = L.kind != MLH_KIND_ATTENTION;
        int t = nh * (gdn || !hp.queryGating ? 3 : 4) * (hp.headDim / 16) + (hp.pleDim > 0 ? 1 : 0);
        if (gdn) t += (L.offGb + hp.gdnHeads - 1) / 16 - L.offGa / 16 + 1;
        tiles = std::max(tiles, t);
    }
    return tiles;
}

static bool wide_plan(const mlh_ctx* c, int n, WidePlan& p) {
    const mlh_hparams& hp = c->hp;
    const int mb = blocks_of(n), d = hp.dim, fs = hp.ffnDim / RK_XCDS, nh = hp.attnHeads > RK_XCDS ? 2 : 1;
    if (n > MLH_WIDE_MAX_SEQS) return false;
    p.rowsQ = first_tiles(c) * 16;
    p.lds = mb == 1 ? sizeof(WideShared<1>) : mb == 2 ? sizeof(WideShared<2>) : mb == 3 ? sizeof(WideShared<3>) : sizeof(WideShared<4>);
    p.lds = std::max(p.lds, (size_t)RK_LDS / 2 + 1024); // one workgroup per compute unit
    size_t at = 0;
    auto place = [&](size_t bytes) { const size_t o = at; at += (bytes + 255) / 256 * 256; return (unsigned)o; };
    const size_t flags = (size_t)d / 16 * (MLH_WIDE_MAX_SEQS / 16) * 4, few = (size_t)RK_PER * (MLH_WIDE_MAX_SEQS / 16) * 4, words = (size_t)d / 16 * (MLH_WIDE_MAX_SEQS / 16) * 2048;
    p.oQ = place((size_t)MLH_WIDE_MAX_SEQS * p.rowsQ * 8); p.fM = place(2 * 4 * 64 * 4); p.fE = place(MLH_WIDE_MAX_SEQS / 16 * 4); p.fX = place(flags); p.fH = place(flags);
    p.fU = place(few); p.oXP = place(words); p.oHP = place(words);
    p.flags = (unsigned)at;
    at *= RK_XCDS;
    p.oAmax = place((size_t)MLH_WIDE_MAX_SEQS * WD_GRID * 16);
    p.oTok = place((size_t)MLH_WIDE_MAX_SEQS * 16);
    p.oZero = place(2048);
    p.data = (unsigned)at;
    at = 0;
    const size_t planes = (size_t)mb * 16 * 6, ssq = (size_t)d / 16 * 256;
    p.oMix = place((nh * hp.headDim + 32) * planes);
    p.oX = place(d * planes); p.oH = place(d * planes); p.oU = place(fs * planes);
    p.oSX = place(ssq); p.oSH = place(ssq); 
    p.area = (unsigned)at;
    at = p.data + at * RK_XCDS;
    p.words = at;
    return true;
}

// Whether the kernel covers a model of these hyper-parameters on this device.
bool mlh_wide_model(const mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    if (c->numCUs != WD_GRID || hp.weightDtype == MLH_DTYPE_BF16 || hp.headDim != WD_HD) return false;
    if (hp.attnHeads < RK_XCDS || hp.attnHeads > 2 * RK_XCDS || hp.dim != hp.attnHeads * WD_HD) return false;
    for (const LayerDev& L : c->layers)
        if (L.kind != MLH_KIND_ATTENTION && (hp.gdnHeads != hp.attnHeads || hp.gdnDk != WD_HD || hp.gdnDv != WD_HD)) return false;
    // a wave's chunks of the width; a first-phase tile and a gate / up tile a workgroup; two tiles of the width a workgroup; two chunks of FFN units a wave
    if (hp.dim % 128 || hp.dim / 32 > WD_CA * WD_WAVES || hp.dim / 16 > 2 * RK_PER || hp.dim / 16 < RK_PER) return false;
    if (hp.ffnDim % (RK_XCDS * 32) || hp.ffnDim / RK_XCDS > 8 * RK_PER) return false;
    if (hp.pleDim > 0) {
        const int pleX = hp.pleDim / RK_XCDS;
        if (hp.pleDim % 32 || 16 % pleX) return false;
        for (const LayerDev& L : c->layers)
            if (L.offPle % 16) return false;
    }
    return first_tiles(c) <= RK_PER;
}

template <int MB>
static int wide_launch(mlh_ctx* c, const WideArgs* P, size_t lds) {
    const void* f = reinterpret_cast<const void*>(&k_decode_wide<MB>);
    if (!P) { // preparation
        MLH_CHECK(c, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, RK_LDS));
        int perCu = 0;
        MLH_CHECK(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, k_decode_wide<MB>, WD_THREADS, RK_LDS));
        return perCu < 1 ? 1 : 0;
    }
    hipLaunchKernelGGL((k_decode_wide<MB>), dim3(WD_GRID), dim3(WD_THREADS), lds, c->stream, *P);
    MLH_CHECK(c, hipGetLastError());
    return 0;
}
static int wide_launch(mlh_ctx* c, int mb, const WideArgs* P, size_t lds) {
    switch (mb) {
        case 1: return wide_launch<1>(c, P, lds);
        case 2: return wide_launch<2>(c, P, lds);
        case 3: return wide_launch<3>(c, P, lds);
        default: return wide_launch<4>(c, P, lds);
    }
}

// At finalize: how many sequences the kernel takes (none where the model or the device does not suit it), and its exchange memory.
int mlh_wide_prepare(mlh_ctx* c) {
    c->wideMax = 0;
    const int most = mlh_ranks_other_seqs(c); // (whose states have a second place)
    if (!mlh_wide_model(c) || !mlh_rows_applicable(c, 1)) return 0;
    size_t bytes = 0;
    WidePlan p;
    for (int n = 1; n <= most; n++) {
        if (!wide_plan(c, n, p)) return 0;
        bytes = std::max(bytes, p.words);
        if (const int rc = wide_launch(c, blocks_of(n), nullptr, 0)) return rc < 0 ? rc : 0;
    }
    if (bytes >= (size_t)1 << 31) return 0;
    if (bytes > c->wideBytes) {
        void* q = nullptr;
        if (hipMalloc(&q, bytes) != hipSuccess) { // no room: the row kernels
            (void)hipGetLastError();
            return 0;
        }
        c->allocs.push_back(q);
        c->wideBuf = q;
        c->wideBytes = bytes;
    }
    c->wideMax = most;
    return 0;
}

// `steps` decode steps of sequences 0 .. nseq - 1 in one launch (tags and the meeting: mlh_launch_ranks).
int mlh_launch_wide(mlh_ctx* c, int nseq, int steps, unsigned tagBase, int otherAt) {
    const mlh_hparams& hp = c->hp;
    WidePlan p;
    if (!wide_plan(c, nseq, p) || p.words > c->wideBytes) { c->err = "decode of many sequences: no plan"; return -1; }
    WideArgs P;
    mlh_fill_args(c, P.a, nseq, c->d_tok);
    P.layers = c->d_layers;
    P.ER = (const unsigned char*)c->ER;
    P.xw = (unsigned char*)c->wideBuf;
    P.xwBytes = (unsigned)c->wideBytes;
    P.tagBase = tagBase;
    P.NL = hp.transformers;
    P.steps = steps;
    P.fs = hp.ffnDim / RK_XCDS; P.rowsQ = p.rowsQ;
    P.abortFlag = c->d_sync + 64 * 20;
    P.xcdCount = c->d_sync + 64 * 23;
    P.data = p.data; P.area = p.area; P.oMix = p.oMix; P.oX = p.oX; P.oH = p.oH; P.oU = p.oU; P.oSX = p.oSX; P.oSH = p.oSH;
    P.flags = p.flags; P.oQ = p.oQ; P.fM = p.fM; P.fE = p.fE; P.fX = p.fX; P.fH = p.fH; P.fU = p.fU; P.oXP = p.oXP; P.oHP = p.oHP; P.oAmax = p.oAmax; P.oTok = p.oTok; P.oZero = p.oZero;
    P.otherAt = otherAt;
    P.sides = c->ranksSides;
    P.abortAtStep = c->injectAbortStep;
    c->injectAbortStep = 0;
    return wide_launch(c, blocks_of(nseq), &P, p.lds);
}
