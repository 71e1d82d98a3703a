// The prompt pass in large passes: hundreds to thousands of prompt positions through each layer at once
// (base2_stream.swift:74-91, 274-275 sends the whole prompt through each layer).  A pass holds `rows` rows, row
// r = slot n + (position - a) for S streams (slots) of n = b - a positions [a, b) each: whole prompts of several
// streams (a = 0), or part of one longer prompt (a a multiple of PCH).  Every number is the decode step's.
//   k_pgemm     a bank over all rows (base2.py:29-32): 64 x 64 output tiles of int8 MFMA over byte planes
//   k_kv_chunk  the pass's q, k, v of one head (base2.py:93) into the cache, and, for the pass's attention, the
//               byte planes of 64 positions in MFMA operand order
//   k_pattend   attention (base2.py:94-99) of 16 query positions a block, scores and value sums by MFMA
//   k_plight    the rows' lights (base2.py:24-27, 55-60); the Pythia machine's two gauges are k_py_rows'
// Why: in passes of 64 rows each launch (5-9 us, latency-bound) serves 64 rows, and the attention, one block a (head,
// row), reads a row's whole cache for one query.  Same box, a whole call: GPT-2, one 1000-word prompt 9.40 -> 2.13 ms;
// 19 prompts of 213 words and 17 words each 39.2 -> 12.3 ms; 64 prompts of 32 words and 128 words 85.8 -> 72.7 ms.
#include "sm_kernels.h"
#include <cstddef>
#include <type_traits>

typedef int v4p __attribute__((ext_vector_type(4)));
SMD v4p mfma_i8(v4p a, v4p b, v4p c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }

// A row between two kernels of the pass (qkv's, fc's hidden, the attention's output): its values' low 32 bits, and per
// strip of SW values the OR of their magnitudes.  Where that word is below 2^31 the 32 bits are the values; a strip
// past it is written whole as well.  Half the bytes of an int64 row, and its words give the row's water level
// (base2.py:24-27) before the row is read (at 4,028 rows the hidden row's light 42 -> 22 us, fc 85 -> 73).
struct PRow {
    int* x32; i64* x64; i64* orw;      // [rows][n], [rows][n] (only past 31 bits), [rows][n / SW]
};
constexpr int PSW = 32;                // a wave's strip of a bank's columns (the attention's: 64, a head)
SMD bool pnarrow(i64 o) { return (u64)o < ((u64)1 << 31); }
// the OR of a 64-bit value over the 16 lanes of a DPP row, in its lane 15
SMD i64 row_or64(i64 o) {
    o |= dpp64<0x111, 0xf, 0xf>(o, 0);
    o |= dpp64<0x112, 0xf, 0xf>(o, 0);
    o |= dpp64<0x114, 0xf, 0xf>(o, 0);
    o |= dpp64<0x118, 0xf, 0xf>(o, 0);
    return o;
}

// ---------------------------------------------------------------------------------------------------------
// The lights of a pass: eight rows a block, one wave each, so a row's reductions stay in its wave; a lane takes four
// consecutive values a time, the byte planes go through LDS (16-value chunks padded to 144 bytes, so that a wave's
// writes spread over the banks) and out as whole 128-byte lines of the MFMA A order.  The correction plane is written
// only for a row that holds a +32768 (its n32768 fact): k_pgemm reads it for those rows alone.  Bound by the row's read
// and the planes' write: 3072-wide rows 12.6 -> 8.8 us at 999 rows, 42 -> 22 us at 4,028 against one block a row, whose
// 16-byte pieces of eight rows' lines came from blocks on eight XCDs.
//   PRO_GAUGE: of the stream rows X (int64), with LS and its power factor in the row facts (base2.py:55-60)
//   PRO_EMBED: the words enter, R = wte[word] + wpe[pos] (base2.py:103), then PRO_GAUGE
//   PRO_TO16:  of rows x (PRow, strips of SW)                                                   (base2.py:24-27)
struct PLightArgs {
    int rows;
    const i64* X; PRow x;
    const i64* wte; const i64* wpe; const int* seq; int seq_stride; const int* rowmap; i64* Rw;
    signed char* planes; int* rowinfo;
    Tables tb;
};
template <int K, int PRO, int SW>
__global__ __launch_bounds__(512) void k_plight(PLightArgs a) {
    constexpr int NM = K / 256, NW = K / SW, CS = 144;
    static_assert(PRO == PRO_TO16 || K == 768, "a stream row is 768 wide");
    __shared__ __align__(16) unsigned char pl[2][K / 16 * CS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = blockIdx.x * 8 + wave;
    i64 v[NM][4];
    i64 orr = 0;
    bool narrow = false;
    if (r < a.rows) {
        if constexpr (PRO == PRO_TO16) {
#pragma unroll
            for (int m = 0; m < (NW + 63) / 64; m++)
                if (lane + 64 * m < NW) orr |= a.x.orw[(size_t)r * NW + lane + 64 * m];
            v4p w[NM];
#pragma unroll
            for (int m = 0; m < NM; m++) w[m] = *reinterpret_cast<const v4p*>(a.x.x32 + (size_t)r * K + 4 * lane + 256 * m);
            orr = wave_or64(orr);
            narrow = pnarrow(orr);
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int j = 0; j < 4; j++) v[m][j] = w[m][j];
            if (!narrow) {                                  // (rare) the strips past 31 bits, whole
#pragma unroll
                for (int m = 0; m < NM; m++) {
                    const int k = 4 * lane + 256 * m;
                    if (pnarrow(a.x.orw[(size_t)r * NW + k / SW])) continue;
#pragma unroll
                    for (int j = 0; j < 4; j++) v[m][j] = a.x.x64[(size_t)r * K + k + j];
                }
            }
        } else {
            typedef i64 v2 __attribute__((ext_vector_type(2)));
            if constexpr (PRO == PRO_EMBED) {
                const int pm = a.rowmap[r], q = pm & 0xFFFF;
                const i64 tok = a.seq[(size_t)(pm >> 16) * a.seq_stride + q];
#pragma unroll
                for (int m = 0; m < NM; m++)
#pragma unroll
                    for (int j = 0; j < 4; j += 2) {
                        const int k = 4 * lane + 256 * m + j;
                        const v2 t = *reinterpret_cast<const v2*>(a.wte + tok * 768 + k), e = *reinterpret_cast<const v2*>(a.wpe + (i64)q * 768 + k);
                        v[m][j] = wadd(t[0], e[0]); v[m][j + 1] = wadd(t[1], e[1]);
                        *reinterpret_cast<v2*>(a.Rw + (size_t)r * 768 + k) = v2{v[m][j], v[m][j + 1]};
                    }
            } else {
#pragma unroll
                for (int m = 0; m < NM; m++)
#pragma unroll
                    for (int j = 0; j < 4; j += 2) {
                        const v2 t = *reinterpret_cast<const v2*>(a.X + (size_t)r * K + 4 * lane + 256 * m + j);
                        v[m][j] = t[0]; v[m][j + 1] = t[1];
                    }
            }
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int j = 0; j < 4; j++) orr |= iabs64(v[m][j]);
            orr = wave_or64(orr);
            narrow = pnarrow(orr);
        }
        const int sh = water_shift(orr), s1h = sh > 0 ? sh - 1 : 0;
        int s1 = 0, sxh = 0, sxl = 0, n32 = 0;
        i64 s2 = 0;
#pragma unroll
        for (int m = 0; m < NM; m++) {
            unsigned ph = 0, pq = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // rshift(v, sh); a value below 2^31: (v >> (sh - 1)) + 1 >> 1, sh at most 16 there
                const int x = narrow ? (sh ? (((int)v[m][j] >> s1h) + 1) >> 1 : (int)v[m][j]) : (int)rsh(v[m][j], sh);
                if constexpr (PRO != PRO_TO16) { s1 += x; s2 += (i64)x * x; }
                const int c = x == 32768, xc = x - c, xh = xc >> 8, xl = (xc & 255) - 128;
                sxh += xh; sxl += xl; n32 += c;
                ph |= (unsigned)(xh & 255) << (8 * j);
                pq |= (unsigned)(xl & 255) << (8 * j);
            }
            const int k = 4 * lane + 256 * m, o = (k >> 4) * CS + wave * 16 + (k & 15);
            *reinterpret_cast<unsigned*>(&pl[0][o]) = ph;
            *reinterpret_cast<unsigned*>(&pl[1][o]) = pq;
        }
        sxh = wave_add32(sxh); sxl = wave_add32(sxl); n32 = wave_add32(n32);
        int* ri = a.rowinfo + (size_t)r * 8;
        const int ex = -16 + sh;
        if constexpr (PRO != PRO_TO16) {
            const i64 S1 = wave_add32(s1), S2 = ((i64)wave_add32((int)(s2 >> 16)) << 16) + wave_add32((int)(s2 & 0xFFFF));
            i64 e2;
            const i64 ls = gauge_ls_pow(S1, S2, ex, a.tb, e2);
            if (lane == 0) { ri[1] = (int)(u64)ls; ri[2] = (int)((u64)ls >> 32); ri[3] = (int)e2; }
        }
        if (lane == 0) { ri[0] = ex; ri[4] = sxh; ri[5] = sxl; ri[6] = n32; }
        if (n32) {                                          // (rare, uniform) the correction plane's row
#pragma unroll
            for (int m = 0; m < NM; m++) {
                const int k = 4 * lane + 256 * m;
                unsigned pc = 0;
#pragma unroll
                for (int j = 0; j < 4; j++) pc |= (unsigned)((int)rsh(v[m][j], sh) == 32768) << (8 * j);
                const size_t o = ((size_t)(r >> 4) * (K / 64) + (k >> 6)) * 3072 + 2048 + ((r & 15) + 16 * ((k & 63) >> 4)) * 16 + (k & 15);
                *reinterpret_cast<unsigned*>(a.planes + o) = pc;
            }
        }
    }
    __syncthreads();
    // out: unit u = chunk u / 8 (of 16 values), row u % 8
    const int t = blockIdx.x >> 1, r0 = (blockIdx.x & 1) * 8;
    v4p* dst = reinterpret_cast<v4p*>(a.planes) + (size_t)t * (K / 64) * 192;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int i = 0; i < K / 16 * 8 / 512 + (K / 16 * 8 % 512 != 0); i++) {
            const int u = threadIdx.x + 512 * i, c = u >> 3, rr = u & 7;
            if (c < K / 16) dst[(c >> 2) * 192 + p * 64 + r0 + rr + 16 * (c & 3)] = *reinterpret_cast<const v4p*>(&pl[p][c * CS + rr * 16]);
        }
}

// ---------------------------------------------------------------------------------------------------------
// One bank over a pass of rows.  Block: MT x NT tiles of 16 x 16 outputs, four waves (WM of them over the rows) of
// TM x TN tiles, three int32 accumulators a tile (HH, MID, LL of the pile identity in sm_batch.hip); a 64-k step's
// operands (1 KB a tile and plane) go through two LDS buffers, D steps ahead in registers.  All operands lie in memory
// in MFMA order, so every global load and LDS access is a whole wave's consecutive 1 KB.  Blocks are numbered so that
// each XCD (block index % 8) works on a contiguous run of row tiles.  KW = 2: two groups of such waves, each every
// second k step, whose sums meet in LDS (half the chain of a 3072-wide bank with few blocks).
// Bound by neither unit: at 999 / 4,028 rows fc keeps the matrix units 16 / 23 % busy, mproj 18 / 32 %, and the LDS units as
// much, with no bank conflicts; its waves wait 30 to 40 % of their cycles, mostly on memory and barriers.
// The machine's tiles are 64 x 64 (four waves of 32 x 32, 126 registers, four blocks a CU): at 999 / 4,028 rows fc
// takes 23.4 / 73 us and mproj 26.5 / 59 us with one group (0.7-1.3 POP/s of int8).  128 x 64 tiles measured 28.8 / 79 and 35.9 / 69
// us, 128 x 128 of eight waves 26.8 / 77 and 44.6 / 69, 128 x 128 of four waves 39 / 111 and 67 / 100 (fewer blocks to
// run beside each other's barriers and epilogues), four steps ahead in place of two 24.4 / 78 and 23.0 / 57.
struct PGemmArgs {
    int N, rows;
    const signed char* W; const int* csum; const int* we; const i64* bias;   // the plate (MfmaPlate)
    const signed char* planes; const int* rowinfo;                            // the rows' lights
    i64* Y;                       // EPI_PLAIN_ADD: [rows][N] the stream, added to; EPI_PILE: [rows][N] the piles
    PRow y;                       // the other epilogues: the rows written, strips of PSW
    Tables tb;
    int* err;                     // the Pythia machine: its rshift assert sets SM_ERR_RANGE here
};
template <int K, int EPI, int MT, int NT, int WM, int WN, int D, int KW = 1>
__global__ __launch_bounds__(64 * WM * WN * KW, 2) void k_pgemm(PGemmArgs a) {
    constexpr int KS = K / 64, CH = (MT + NT) * 2, NV = WM * WN, PER = CH / NV, TM = MT / WM, TN = NT / WN;
    constexpr bool GAUGED = EPI == EPI_GAUGED || EPI == EPI_GAUGED_EDGE, EDGE = EPI == EPI_GAUGED_EDGE || EPI == EPI_PLAIN_EDGE;
    constexpr bool PLAIN = EPI == EPI_PLAIN || EPI == EPI_PLAIN_EDGE || EPI == EPI_PLAIN_ADD;
    constexpr bool ROWS = GAUGED || EPI == EPI_PLAIN || EPI == EPI_PLAIN_EDGE;      // the outputs go to a PRow
    static_assert(CH % NV == 0 && KS % (D * KW) == 0 && D % 2 == 0, "whole chunks a wave, whole rounds of the ring");
    static_assert(!ROWS || TN * 16 % PSW == 0, "a wave's columns are whole strips");
    __shared__ v4p buf[2 * KW][CH][64];
    static_assert(KW == 1 || NV * TM * TN * 3 <= 2 * KW * CH, "the groups' accumulators meet in buf");
    __shared__ i64 rcC[16 * MT];             // a row's pile constant
    __shared__ int rcS[16 * MT], rcE[16 * MT], rcN[16 * MT];   // its power's row part and factor, n32768
    __shared__ int any32;
    const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) % NV, kg = (tid >> 6) / NV;
    const int ntiles = (a.N + 15) / 16, nb = (ntiles + NT - 1) / NT, mb = (a.rows + 16 * MT - 1) / (16 * MT), total = nb * mb;
    // block b of XCD b % 8: the (b / 8)-th of that XCD's run of `per` tiles
    const int per = (total + 7) / 8, id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (id >= total || (int)(blockIdx.x >> 3) >= per) return;
    const int m0 = id / nb * MT, n0 = id % nb * NT;                  // first row and column tile
    const int wm = (wave % WM) * TM, wn = (wave / WM) * TN;
    // chunk c of a step: c < 2 MT a light plane (row tile c / 2, plane c % 2), else a plate plane (a column tile past
    // the plate's last reads the last)
    const v4p* src[PER];
    static_assert(2 * MT % NV == 0, "a wave's chunk i is a light plane for NV i < 2 MT");
    auto step = [](int i) { return NV * i < 2 * MT ? 192 : 128; };    // 16-byte words from one k step to the next
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int c = wave + NV * i, d = c - 2 * MT;
        if (NV * i < 2 * MT) src[i] = reinterpret_cast<const v4p*>(a.planes) + ((size_t)(m0 + c / 2) * KS * 3 + c % 2) * 64 + lane;
        else src[i] = reinterpret_cast<const v4p*>(a.W) + ((size_t)min(n0 + d / 2, ntiles - 1) * KS * 2 + d % 2) * 64 + lane;
    }
    v4p r[D][PER];
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
        for (int i = 0; i < PER; i++) r[d][i] = src[i][(d * KW + kg) * step(i)];
    // the rows' facts (ex, LS lo, LS hi, e2, SXh, SXl, n32768; gauged lights carry LS and its power factor)
    if (tid == 0) any32 = 0;
    __syncthreads();
    if (tid < 16 * MT) {
        const int row = 16 * m0 + tid;
        i64 C = 0;
        int S = 0, E = 0, n32 = 0;
        if (row < a.rows) {
            const v4p f0 = *reinterpret_cast<const v4p*>(a.rowinfo + (size_t)row * 8);
            const v4p f1 = *reinterpret_cast<const v4p*>(a.rowinfo + (size_t)row * 8 + 4);
            C = 32768 * (i64)f1[0] + 128 * (i64)f1[1] + 16384 * (i64)K + 128 * (i64)f1[2];
            n32 = f1[2];
            if (GAUGED) {        // power(pile, (we + ex + 16) 65536 - LS) (base2.py:70): shift S - we, fine part the row's
                const i64 ls = (i64)(((u64)(unsigned)f0[2] << 32) | (unsigned)f0[1]);
                S = 16 - (int)(wsub(wmul((i64)f0[0] + 16, 65536), ls) >> 16);
                E = f0[3];
            } else {             // rshift(pile, -(we + ex + 16))
                S = -(f0[0] + 16);
            }
            if (n32) any32 = 1;
        }
        rcC[tid] = C; rcS[tid] = S; rcE[tid] = E; rcN[tid] = n32;
    }
    v4p acc[TM][TN][3];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j][0] = acc[i][j][1] = acc[i][j][2] = v4p{0, 0, 0, 0};
#pragma unroll 1
    for (int s0 = 0; s0 < KS / KW; s0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            v4p(*bs)[64] = buf[2 * kg + (d & 1)];
#pragma unroll
            for (int i = 0; i < PER; i++) bs[wave + NV * i][lane] = r[d][i];
            // D steps on (past the end the last step again: no branch around the loads)
            const int nx = min(s0 + d + D, KS / KW - 1) * KW + kg;
#pragma unroll
            for (int i = 0; i < PER; i++) r[d][i] = src[i][nx * step(i)];
            __syncthreads();
            v4p bh[TN], bl[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) {
                bh[j] = bs[2 * MT + 2 * (wn + j)][lane];
                bl[j] = bs[2 * MT + 2 * (wn + j) + 1][lane];
            }
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const v4p xh = bs[2 * (wm + i)][lane], xl = bs[2 * (wm + i) + 1][lane];
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    acc[i][j][0] = mfma_i8(xh, bh[j], acc[i][j][0]);
                    acc[i][j][1] = mfma_i8(xh, bl[j], acc[i][j][1]);
                    acc[i][j][2] = mfma_i8(xl, bl[j], acc[i][j][2]);
                    acc[i][j][1] = mfma_i8(xl, bh[j], acc[i][j][1]);
                }
            }
        }
    }
    if constexpr (KW > 1) {               // the second group's sums to the first
        __syncthreads();
        v4p* x = &buf[0][0][0] + wave * TM * TN * 3 * 64 + lane;
        if (kg > 0)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int k = 0; k < 3; k++) x[((i * TN + j) * 3 + k) * 64] = acc[i][j][k];
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int k = 0; k < 3; k++) acc[i][j][k] += x[((i * TN + j) * 3 + k) * 64];
    }
    // (rare) a light of +32768 among the block's rows, held as 32767: those rows' correction plane times the plate
    if (any32) {
        const v4p* A = reinterpret_cast<const v4p*>(a.planes) + ((size_t)(m0 + wm) * KS * 3 + 2) * 64 + lane;
        const v4p* B = reinterpret_cast<const v4p*>(a.W) + lane;
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const size_t o = ((size_t)min(n0 + wn + j, ntiles - 1) * KS + s) * 128;
                const v4p wh = B[o], wl = B[o + 64];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    v4p cc = {0, 0, 0, 0};
                    if (rcN[16 * (wm + i) + (lane & 15)]) cc = A[((size_t)i * KS + s) * 192];
                    acc[i][j][1] = mfma_i8(cc, wh, acc[i][j][1]);
                    acc[i][j][2] = mfma_i8(cc, wl, acc[i][j][2]);
                }
            }
    }
    // the epilogue: lane holds rows 4 (lane / 16) + q of each row tile, column lane % 16 of each column tile
    i64 ccol[TN], we[TN], bc[TN];
    const unsigned n = (unsigned)a.N;       // (columns past the last read zeros)
    const __amdgpu_buffer_rsrc_t rcs = buf_rsrc(a.csum, 8u * n), rwe = buf_rsrc(a.we, 4u * n), rbi = buf_rsrc(a.bias, 8u * n);
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const unsigned col = (unsigned)(16 * (n0 + wn + j) + (lane & 15));
        ccol[j] = 32768 * (i64)buf_load1(rcs, 8u * col) + 128 * (i64)buf_load1(rcs, 8u * col + 4u);
        we[j] = bc[j] = 0;
        if (EPI != EPI_PILE) { we[j] = buf_load1(rwe, 4u * col); bc[j] = buf_load8(rbi, 8u * col); }
    }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int lr = 16 * (wm + i) + 4 * (lane >> 4), row = 16 * m0 + lr;
        i64 y[TN][4];
        if constexpr (EPI == EPI_PLAIN_ADD) {      // bounded: a row past the last reads zeros
            const __amdgpu_buffer_rsrc_t ry = buf_rsrc(a.Y, (unsigned)a.rows * n * 8u);
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    y[j][q] = buf_load8(ry, ((unsigned)(row + q) * n + (unsigned)(16 * (n0 + wn + j) + (lane & 15))) * 8u);
        }
        i64 o[TN][4];
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const i64 pile = 65536 * (i64)acc[i][j][0][q] + 256 * (i64)acc[i][j][1][q] + acc[i][j][2][q] + rcC[lr + q] + ccol[j];
                o[j][q] = pile;
                if constexpr (EPI == EPI_PILE) continue;
                const bool live = row + q < a.rows;
                const i64 v = GAUGED ? (i64)((u64)pile * (u64)(unsigned)rcE[lr + q]) : pile;
                const i64 s = (i64)rcS[lr + q] - we[j];
                if (__ballot(live && (u64)(s - 1) >= 62) == 0) {
                    // the usual rounding right shift; |v| is below 2^60 (a pile below 2^42, a factor at most 2^17),
                    // so (v + 2^(s-1)) >> s is ((v >> (s-1)) + 1) >> 1
                    o[j][q] = ((v >> ((int)(s - 1) & 63)) + 1) >> 1;
                } else {
                    if (PLAIN && live && a.err && pyshift_fails(v, s)) atomicOr(a.err, SM_ERR_RANGE);
                    o[j][q] = rsh(v, s);
                }
                o[j][q] = wadd(o[j][q], bc[j]);
            }
        if constexpr (EDGE) {
            bool wide = false;
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) wide |= (u64)(o[j][q] + (1 << 30)) >= (1ull << 31);
            if (__ballot(wide) == 0) {
                // below 2^30 in magnitude: the edge (base2.py:78-83) in 32 bits, its product in 64
                int h[TN][4], ix[TN][4], sh[TN][4];
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        h[j][q] = (int)o[j][q];
                        ix[j][q] = ((h[j][q] + 8) >> 4) + 32768;
                        sh[j][q] = a.tb.PHI[min(max(ix[j][q], 0), 65535)];
                    }
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int share = ix[j][q] < 0 ? 0 : (ix[j][q] > 65535 ? 65536 : sh[j][q]);
                        o[j][q] = ((i64)h[j][q] * share + 32768) >> 16;
                    }
            } else {
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) o[j][q] = edge1(o[j][q], a.tb);
            }
        }
        if constexpr (ROWS) {
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int st = 0; st < TN / 2; st++) {            // the wave's strips, two column tiles each
                    i64 w = iabs64(o[2 * st][q]) | iabs64(o[2 * st + 1][q]);
                    const size_t at = (size_t)(row + q) * n + 16 * (n0 + wn + 2 * st) + (lane & 15);
                    bool wide = false;
                    if (__ballot(!pnarrow(w)) == 0) {        // (the strip's OR in 32 bits)
                        int w32 = (int)w;
                        w32 |= DPP(w32, 0x111, 0xf, 0xf); w32 |= DPP(w32, 0x112, 0xf, 0xf);
                        w32 |= DPP(w32, 0x114, 0xf, 0xf); w32 |= DPP(w32, 0x118, 0xf, 0xf);
                        w = w32;
                    } else {
                        w = row_or64(w);
                        wide = !pnarrow(__shfl(w, (lane & 48) | 15, 64));    // the row's strip holds a value past 31 bits
                    }
                    if (row + q < a.rows) {
                        if ((lane & 15) == 15) a.y.orw[(size_t)(row + q) * (n / PSW) + (n0 + wn) / 2 + st] = w;
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            a.y.x32[at + 16 * j] = (int)o[2 * st + j][q];
                            if (wide) a.y.x64[at + 16 * j] = o[2 * st + j][q];
                        }
                    }
                }
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const unsigned col = (unsigned)(16 * (n0 + wn + j) + (lane & 15));
                    if (row + q >= a.rows || col >= n) continue;
                    i64* to = a.Y + (size_t)(row + q) * n + col;
                    *to = EPI == EPI_PLAIN_ADD ? wadd(y[j][q], o[j][q]) : o[j][q];
                }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// The pass's attention operands, one chunk of PCH positions of one (slot, head) each, in MFMA order:
//   K  [4 position tiles][kh, kl'][64 lanes][16]: lane l position l % 16, dimensions 16 (l / 16) ..; a key k' (a
//      +32768 held as 32767) is 256 kh + kl' + 128
//   V  [4 dimension tiles][3 digits][64 lanes][16]: lane l dimension l % 16, byte 4 i + r the position
//      16 i + 4 (l / 16) + r (the order in which a lane holds its scores); v = d0 + 256 d1 + 65536 d2, each digit
//      a signed byte (of a value that three do not hold: its three lowest digits)
//   Q  [4 query tiles][qh, ql][64 lanes][16] and QO [qo]: lane l query l % 16; q = 256 (qh + qo) + ql, digits signed bytes
//      (qo: the 1 that a digit of 128 passes on)
// and per position ek, the +32768 mask km, eq, the sum of q; flag[0] bit 0: a value that three digits do not hold,
// bit 1: a mask is set, bit 2: a qo is, bit 3: a value that six digits do not hold; flag[1], flag[2]: the least and
// the largest ek; Pythia: vmax, the largest |v| of the positions of a wave that holds a value of bit 0 (else 0).
constexpr int PCH = 64;
struct PChunk {
    signed char K[4][2][1024];
    signed char V[4][3][1024];
    signed char Q[4][2][1024];
    i64 km[PCH];
    int ek[PCH], eq[PCH], sq[PCH], flag[PCH];        // flag[0 .. 2]
    signed char QO[4][1024];                         // these two written where flag[0] has bit 0 or bit 2
    i64 vmax[PCH];
};
// the four bytes of four words, by byte: d[k] holds byte k of t[0 .. 3]
SMD void byte_planes(const unsigned (&t)[4], unsigned (&d)[4]) {
    const unsigned l01 = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u), l23 = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u);
    const unsigned h01 = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u), h23 = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
    d[0] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
    d[1] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
    d[2] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
    d[3] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
}
// v without its three lowest signed digits, over 2^24 (modulo 2^40: v modulo 2^64 is those digits and 2^24 times it)
SMD i64 above3(i64 v) { return (i64)((u64)v + 0x808080u) >> 24; }
struct PAttArgs {
    AttArgs a;                    // the layer's cache, tables, error word
    PRow x;                       // the qkv rows (strips of PSW)
    PRow out;                     // the attention rows (strips of 64: a head)
    PChunk* ch;                   // [slot][head][nch]; k_kv_chunk without it only stores keys and values
    int n, pa, pb, nch, s0;       // rows a slot, its positions [pa, pb), chunks of [0, pb), the first slot's stream
};

// Block: one chunk of one (slot, head); wave w positions 4 w .. + 3, lane = dimension.  A chunk of this pass takes
// q, k, v from the qkv rows (base2.py:93: each through its own water level, which the rows' OR words give;
// pythia_base2.py:116-123: q and k turned first) and stores k and v; an earlier pass's chunk (all of it below pa)
// comes back from the cache.
template <int MODEL>
__global__ __launch_bounds__(1024) void k_kv_chunk(PAttArgs g) {
    const AttArgs& a = g.a;
    __shared__ __align__(16) PChunk ch;
    const int c = blockIdx.x, h = blockIdx.y, slot = blockIdx.z, st = g.s0 + slot;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ti = wave >> 2, gq = wave & 3;   // 16-position tile, group
    const size_t hrow = (size_t)st * 12 + h;
    const bool fresh = PCH * c >= g.pa;
    if (!fresh && !g.ch) return;                           // (the last layer: an earlier pass's chunk has nothing to do)
    auto at = [&](int part) { return MODEL == 1 ? h * 192 + part * 64 + lane : part * 768 + h * 64 + lane; };
    i64 q[4], k[4], v[4], oq[4], ok[4], ov[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int p = PCH * c + 4 * wave + j;
        q[j] = k[j] = v[j] = oq[j] = ok[j] = ov[j] = 0;
        if (fresh && p < g.pb) {
            const size_t r = (size_t)(slot * g.n + p - g.pa);
            const i64* w = g.x.orw + r * (2304 / PSW);
            const int* x = g.x.x32 + r * 2304;
            q[j] = x[at(0)]; k[j] = x[at(1)]; v[j] = x[at(2)];
            oq[j] = w[at(0) / PSW]; ok[j] = w[at(1) / PSW]; ov[j] = w[at(2) / PSW];
        }
    }
    if (threadIdx.x == 0) { ch.flag[0] = 0; ch.flag[1] = INT32_MAX; ch.flag[2] = INT32_MIN; }
    if (MODEL == 1 && threadIdx.x < PCH) ch.vmax[threadIdx.x] = 0;
    __syncthreads();
    // the OR of a head's two strips (lanes 0-31 hold the one's word, the others the other's), the same in every lane
    auto both = [](i64 o) -> i64 {
        const int lo = __builtin_amdgcn_readlane((int)o, 0) | __builtin_amdgcn_readlane((int)o, 63);
        const int hi = __builtin_amdgcn_readlane((int)(o >> 32), 0) | __builtin_amdgcn_readlane((int)(o >> 32), 63);
        return (i64)(((u64)(unsigned)hi << 32) | (unsigned)lo);
    };
    bool wide = false, masks = false, carry = false;
    int emin = INT32_MAX, emax = INT32_MIN;
    const int off = (lane >> 4) * 256 + (lane & 15);       // + 16 (position % 16): the byte in an operand tile
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = 4 * gq + j, pl = 4 * wave + j, p = PCH * c + pl;
        int q16 = 0, k16 = 0, ekv = -16, eqv = -16;
        u64 km = 0;
        if (fresh) {
            if (p < g.pb) {                                // (uniform)
                i64 aq = both(oq[j]), ak = both(ok[j]);
                if (!pnarrow(aq | ak | both(ov[j]))) {     // (rare) strips past 31 bits, whole
                    const i64* x = g.x.x64 + (size_t)(slot * g.n + p - g.pa) * 2304;
                    if (!pnarrow(oq[j])) q[j] = x[at(0)];
                    if (!pnarrow(ok[j])) k[j] = x[at(1)];
                    if (!pnarrow(ov[j])) v[j] = x[at(2)];
                }
                if constexpr (MODEL == 1) {
                    const int r = a.rot >> 1, src = lane < r ? lane + r : lane - r;
                    const i64 pq = __shfl(q[j], src, 64), pk = __shfl(k[j], src, 64);
                    if (lane < a.rot) {
                        if (iabs64(q[j]) >= ((i64)1 << 31) || iabs64(k[j]) >= ((i64)1 << 31)) atomicOr(a.err, SM_ERR_RANGE);
                        const int t = lane < r ? lane : lane - r;
                        const i64 cs = a.cosT[(size_t)p * r + t], sn = a.sinT[(size_t)p * r + t];
                        q[j] = turn1<0>(q[j], pq, lane < r, cs, sn, 0.0, 0.0);
                        k[j] = turn1<0>(k[j], pk, lane < r, cs, sn, 0.0, 0.0);
                    }
                    aq = wave_or64(iabs64(q[j])); ak = wave_or64(iabs64(k[j]));
                }
                const int shq = water_shift(aq), shk = water_shift(ak);
                q16 = (int)rsh(q[j], shq); k16 = (int)rsh(k[j], shk);
                eqv = -16 + shq; ekv = -16 + shk;
                const size_t slotp = hrow * a.ctx + p;
                key_store(a.K16 + slotp * 64, a.KM + slotp, k16, lane);
                if (lane == 0) a.EK[slotp] = ekv;
                v_store(a, hrow, p, lane, v[j]);
                km = __ballot(k16 == 32768);
                k16 = min(k16, 32767);
            }
        } else {                                           // (an earlier pass's position, below pb)
            const size_t slotp = hrow * a.ctx + p;
            k16 = a.K16[slotp * 64 + lane];
            km = (u64)a.KM[slotp];
            ekv = a.EK[slotp];
            v[j] = v_whole(a, hrow * a.ctx, p, lane);
        }
        wide |= (u64)v[j] + 0x808080u >= 0x1000000u;
        masks |= km != 0;
        emin = min(emin, ekv); emax = max(emax, ekv);
        // q in signed digits; a high digit of 128 as 127 + 1
        const int ql = (int)(signed char)q16, qh = (q16 - ql) >> 8, qo = qh == 128;
        carry |= qo != 0;
        ch.K[ti][0][off + 16 * i] = (signed char)(k16 >> 8);
        ch.K[ti][1][off + 16 * i] = (signed char)((k16 & 255) - 128);
        ch.Q[ti][0][off + 16 * i] = (signed char)(qh - qo);
        ch.Q[ti][1][off + 16 * i] = (signed char)ql;
        ch.QO[ti][off + 16 * i] = (signed char)qo;
        const int sq = wave_add32(q16);
        if (lane == 0) { ch.km[pl] = (i64)km; ch.ek[pl] = ekv; ch.eq[pl] = eqv; ch.sq[pl] = sq; }
    }
    // the values' digits: dimension tile lane / 16, lane' = lane % 16 + 16 gq, byte 4 ti + j
    unsigned t[4], dg[4];
#pragma unroll
    for (int r = 0; r < 4; r++) t[r] = (unsigned)v[r] + 0x808080u;
    byte_planes(t, dg);
    const int o = ((lane & 15) + 16 * gq) * 16 + 4 * ti;
#pragma unroll
    for (int k = 0; k < 3; k++) *reinterpret_cast<unsigned*>(&ch.V[lane >> 4][k][o]) = dg[k] ^ 0x80808080u;
    if (!g.ch) return;                                     // (uniform) the last layer: keys and values alone
    int fl = (__ballot(wide) ? 1 : 0) | (__ballot(masks) ? 2 : 0) | (__ballot(carry) ? 4 : 0);
    if (fl & 1) {                                          // (rare) values that three digits do not hold
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (__ballot((u64)v[j] + 0x808080808080u >= 0x1000000000000u)) fl |= 8;
            if (MODEL == 1) {
                const i64 m = wave_reduce64(iabs64(v[j]), OpMax());
                if (lane == 0) ch.vmax[4 * wave + j] = m;
            }
        }
    }
    if (lane == 0) {
        if (fl) atomicOr(&ch.flag[0], fl);
        atomicMin(&ch.flag[1], emin);
        atomicMax(&ch.flag[2], emax);
    }
    __syncthreads();
    static_assert(sizeof(PChunk) % 16 == 0 && offsetof(PChunk, QO) % 16 == 0, "copied as 16-byte words");
    const v4p* s = reinterpret_cast<const v4p*>(&ch);
    v4p* d = reinterpret_cast<v4p*>(g.ch + ((size_t)slot * 12 + h) * g.nch + c);
    const int words = (int)((ch.flag[0] & 5 ? sizeof(PChunk) : offsetof(PChunk, QO)) / 16);
    for (int i = threadIdx.x; i < words; i += 1024) d[i] = s[i];
}

// ---------------------------------------------------------------------------------------------------------
// Attention of 16 query positions of one (slot, head), base2.py:94-99 (pythia_base2.py:125-141).  Wave w takes the
// chunks w, w + NW, .. of the positions up to the tile's last, twice: once for the queries' maxima, then, from its last
// chunk back (whose 32-bit scores it still holds; the others' are formed again), for the arrivals against them and the value
// sums.  Scores: rows are positions and columns queries,
// so lane l holds query l % 16 at positions 16 i + 4 (l / 16) + r of a chunk; those 16 arrivals, split into digit
// bytes, are the B operand of the value product as they stand, with the chunk's V in the same order (PChunk).  An
// arrival, at most 2^24, is three signed digits and a 0/1 fourth, which most chunks lack; the products of equal
// weight share one int32 accumulator (at most 4 x 2^20 a chunk: callers keep positions below 16384, so none
// passes 2^31).  The waves' sums meet in LDS in 64 bits.
// A head with a value that three digits do not hold (past 2^23) takes the value sums two or three times: over the three
// lowest digits of every value, the next three and, with a value past 2^47, the rest, whose digits the waves form from
// the cache; a sum modulo 2^64 is the groups' sums at 2^0, 2^24 and 2^48.  Two of the four dimension tiles a pass over
// the chunks there: with four, the kernels spill 20 to 40 vector registers.  A whole call of one 1000-word prompt 2.53 ms
// with one head of every layer past 2^23, 3.31 with all, 5.76 with all past 2^33, against 2.13 without (15.2, 22.9 and 26.0
// with a wave walking each query's positions); 19 prompts of 213 words 4.70, 5.92 and 8.79 against 4.43.
// Bound by each wave's chain (keys, products, arrivals' table reads, values) at two waves a SIMD: 39 us at one
// stream's 999 positions, 48 at 19 of 212; with the scores in 64 bits throughout 56.5 and 81.
template <int MODEL>
SMD i64 patt_score(const AttArgs& a, i64 dot, i64 e) {      // e = eq + ek
    if constexpr (MODEL == 1) return rsh(wmul(dot, a.ehalf), wsub(16, wsub(wmul(e + 10, 65536), a.half) >> 16));
    else return rsh(dot, -(e + 7));
}
// over the total through its log (base2.py:99; Pythia: exact in 128 bits, pythia_base2.py:139, 90)
template <int MODEL>
SMD i64 patt_out(const AttArgs& a, i64 num, int zt, i64 lg, i64 hp, bool live) {
    const i64 F = wsub(0, wadd((i64)zt * 65536, lg));
    if constexpr (MODEL == 1) {
        const __int128 X = (__int128)num * hp;
        const i64 sft = 16 - (F >> 16);
        const __int128 r = sft >= 100 ? (__int128)0 : (X + ((__int128)1 << (sft - 1))) >> sft;
        if (live && (r > (__int128)INT64_MAX || r < (__int128)INT64_MIN)) atomicOr(a.err, SM_ERR_RANGE);
        return (i64)r;
    } else {
        return power_e(num, F, F & 0xFFFF, hp, a.tb);
    }
}
// the q of query ql, dimension d, back from its digits
SMD int pchunk_q(const PChunk* c, int tile, int ql, int d) {
    const int o = (d >> 4) * 256 + ql * 16 + (d & 15);
    return 256 * (c->Q[tile][0][o] + (c->flag[0] & 4 ? c->QO[tile][o] : 0)) + c->Q[tile][1][o];
}
template <int MODEL, int NW>
__global__ __launch_bounds__(64 * NW, 2) void k_pattend(PAttArgs g) {
    const AttArgs& a = g.a;
    __shared__ i64 mx_s[NW][16], z_s[NW][16];
    __shared__ i64 num_s[NW][16][64], vm_s[NW][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ql = lane & 15, pg = lane >> 4;
    const int h = blockIdx.y, slot = blockIdx.z;
    const int p0 = g.pa + 16 * (int)(gridDim.x - 1 - blockIdx.x);     // the longest tiles first
    const int plast = min(p0 + 15, g.pb - 1), nc = plast / PCH + 1, p = p0 + ql;
    const PChunk* ch = g.ch + ((size_t)slot * 12 + h) * g.nch;
    const PChunk* cq = ch + p0 / PCH;
    const int qt = (p0 % PCH) >> 4;
    const v4p qh = *reinterpret_cast<const v4p*>(&cq->Q[qt][0][16 * lane]), qll = *reinterpret_cast<const v4p*>(&cq->Q[qt][1][16 * lane]);
    const i64 eq = cq->eq[p0 % PCH + ql], sq128 = 128 * (i64)cq->sq[p0 % PCH + ql];
    const bool carry = cq->flag[0] & 4;
    int fl = 0, emn = INT32_MAX, emx = INT32_MIN;            // any chunk's flags, the keys' levels
    for (int c = lane; c < nc; c += 64) {
        fl |= ch[c].flag[0];
        emn = min(emn, ch[c].flag[1]); emx = max(emx, ch[c].flag[2]);
    }
    fl = (int)wave_or32((unsigned)fl);
    v4p qo = {0, 0, 0, 0};
    if (carry) qo = *reinterpret_cast<const v4p*>(&cq->QO[qt][16 * lane]);
    // the scores in 32 bits (GPT-2): with every shift s = -(eq + ek + 7) in 9..40, rshift(dot, s) is
    // ((dot >> 8) >> (s - 9)) + 1 >> 1, and dot >> 8 = 256 HH + MID + ((LL + 128 sum q) >> 8), below 2^30
    const int eql = (int)eq;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { emn = min(emn, __shfl_xor(emn, o, 64)); emx = max(emx, __shfl_xor(emx, o, 64)); }
    const bool ok32 = MODEL == 0 && !(fl & 2) && __ballot(eql + emx > -16 || eql + emn < -47) == 0;
    // arrivals' sum and digit products (below)
    v4p acc[4][6];
    i64 z = 0, vm = 0;
    // acc's products of equal weight as 64-bit sums: lane holds dimensions 16 d + 4 pg + r of query ql in [4 d + r]
    auto sum64 = [&](int d, int r) {
        u64 n = 0;
#pragma unroll
        for (int k = 5; k >= 0; k--) n = (n << 8) + (u64)(i64)acc[d][k][r];
        return (i64)n;
    };
    const __amdgpu_buffer_rsrc_t ra = buf_rsrc(a.tb.ARR, (unsigned)a.tb.alen * 4u);   // 0 past the table (base2.py:97)
    auto body = [&](auto fast, auto wide) {
        constexpr bool FAST = decltype(fast)::value, WIDE = decltype(wide)::value;
        constexpr int DN = WIDE ? 2 : 4;                     // dimension tiles a pass over the chunks
        typedef typename std::conditional<FAST, int, i64>::type S;
        constexpr S LOW = FAST ? (S)INT32_MIN : (S)INT64_MIN;
        S sc[16];
        // chunk c's 16 scores of this lane: positions 64 c + 16 i + 4 pg + r (past p: LOW)
        auto scores = [&](int c) {
            const PChunk* cc = ch + c;
            v4p kh[4], kl[4], ek[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                kh[i] = *reinterpret_cast<const v4p*>(&cc->K[i][0][16 * lane]);
                kl[i] = *reinterpret_cast<const v4p*>(&cc->K[i][1][16 * lane]);
                ek[i] = *reinterpret_cast<const v4p*>(&cc->ek[16 * i + 4 * pg]);
            }
            const int pc = p - PCH * c - 4 * pg;             // position 16 i + r is in for 16 i + r <= pc
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v4p hh = {0, 0, 0, 0}, mid = {0, 0, 0, 0}, ll = {0, 0, 0, 0};
                hh = mfma_i8(kh[i], qh, hh);
                mid = mfma_i8(kl[i], qh, mid);
                ll = mfma_i8(kl[i], qll, ll);
                mid = mfma_i8(kh[i], qll, mid);
                if (carry) {
                    hh = mfma_i8(kh[i], qo, hh);
                    mid = mfma_i8(kl[i], qo, mid);
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    S v;
                    if constexpr (FAST) {
                        const int t8 = (hh[r] << 8) + mid[r] + ((ll[r] + (int)sq128) >> 8);
                        v = ((t8 >> (-16 - eql - ek[i][r])) + 1) >> 1;      // s - 9 = -(eq + ek + 16)
                    } else {
                        i64 dot = 65536 * (i64)hh[r] + 256 * (i64)mid[r] + ll[r] + sq128;
                        if (fl & 2) {                        // (rare) keys holding a +32768: one more of q there
                            for (u64 m = (u64)ch[c].km[16 * i + 4 * pg + r]; m; m &= m - 1) dot += pchunk_q(cq, qt, ql, __builtin_ctzll(m));
                        }
                        v = patt_score<MODEL>(a, dot, eq + ek[i][r]);
                    }
                    sc[4 * i + r] = 16 * i + r <= pc ? v : LOW;
                }
            }
        };
        v4p vv[WIDE ? 1 : 4][3];
        auto vload = [&](int c, int d) {
#pragma unroll
            for (int k = 0; k < 3; k++) vv[WIDE ? 0 : d][k] = *reinterpret_cast<const v4p*>(&ch[c].V[d][k][16 * lane]);
        };
        // WIDE: digits 3 gr .. 3 gr + 2 of chunk c's values, dimension tile d, from the cached rows up to the tile's last
        // position (past it zeros)
        auto vform = [&](int c, int d, int gr) {
            // (the arguments that only this path needs, read here: as the kernel's own they are held in scalar registers
            // from its start, and the usual path's spill)
            typedef const __attribute__((address_space(4))) PAttArgs* arg_p;
            const arg_p ga = (arg_p)__builtin_amdgcn_kernarg_segment_ptr();
            const size_t hb = ((size_t)(ga->s0 + slot) * 12 + h) * ga->a.ctx;
            const unsigned n = (unsigned)plast + 1u;
            const __amdgpu_buffer_rsrc_t rv = buf_rsrc(ga->a.V + hb * 64, n * 256u), rw = buf_rsrc(ga->a.VW + hb, n * 4u),
                                         r8 = buf_rsrc(ga->a.V64 + hb * 64, n * 512u);
            int x[16], m[16], any = 0;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const unsigned s = (unsigned)(PCH * c + 16 * (i >> 2) + 4 * pg + (i & 3));
                x[i] = buf_load1(rv, (s * 64u + 16u * d + ql) * 4u);
                m[i] = buf_load1(rw, s * 4u);
            }
#pragma unroll
            for (int i = 0; i < 16; i++) any |= m[i];
            const bool whole = __ballot(any) != 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                unsigned t[4], dg[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    i64 v = x[4 * i + r];
                    if (whole) {                             // (uniform) rows held whole
                        const unsigned s = (unsigned)(PCH * c + 16 * i + 4 * pg + r);
                        const i64 y = buf_load8(r8, m[4 * i + r] ? (s * 64u + 16u * d + ql) * 8u : 0xFFFFFFF0u);
                        v = m[4 * i + r] ? y : v;
                    }
                    v = above3(v);
                    if (gr == 2) v = above3(v);
                    t[r] = (unsigned)v + 0x808080u;
                }
                byte_planes(t, dg);
#pragma unroll
                for (int k = 0; k < 3; k++) vv[0][k][i] = (int)(dg[k] ^ 0x80808080u);
            }
        };
        // the queries' maxima (base2.py:96): the wave's chunks, the four lane groups, then the waves
        S M = LOW;
        int c = wave;
        for (; c < nc; c += NW) {
            scores(c);
#pragma unroll
            for (int i = 0; i < 16; i++) M = sc[i] > M ? sc[i] : M;
        }
        c -= NW;                                             // the last chunk's scores are at hand
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) { const S x = __shfl_xor(M, o, 64); M = x > M ? x : M; }
        if constexpr (NW > 1) {
            if (lane < 16) mx_s[wave][lane] = M;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < NW; w++) { const S x = (S)mx_s[w][ql]; M = x > M ? x : M; }
        }
        // arrivals (base2.py:96-97), their sum, the value sums (base2.py:98): the wave's chunks, last to first
        const int clast = c, passes = !WIDE ? 1 : (fl & 8 ? 3 : 2) * (4 / DN);
#pragma unroll 1
        for (int ps = 0; ps < passes; ps++) {
            const int gr = WIDE ? ps / (4 / DN) : 0, d0 = WIDE ? ps % (4 / DN) * DN : 0;
            c = clast;
#pragma unroll
            for (int d = 0; d < DN; d++)
#pragma unroll
                for (int k = 0; k < 6; k++) acc[d][k] = v4p{0, 0, 0, 0};
            while (c >= 0) {
                if (!FAST) scores(c);                            // (64-bit scores kept over the loop would spill)
                const int pc = p - PCH * c - 4 * pg;
                unsigned t[16];
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    bool in = 16 * (i >> 2) + (i & 3) <= pc;
                    unsigned d;
                    if constexpr (FAST) {                        // (both below 2^30 in magnitude)
                        d = (unsigned)M - (unsigned)sc[i];   // (past p LOW: wraps, and is not in)
                        in = in && d < (unsigned)a.tb.alen;
                    } else {
                        const i64 dd = wsub(M, sc[i]);
                        in = in && (u64)dd < (u64)a.tb.alen;
                        d = (unsigned)dd;
                    }
                    t[i] = (unsigned)buf_load1(ra, in ? d * 4u : 0xFFFFFFF0u);
                }
                if constexpr (!WIDE) {
#pragma unroll
                    for (int d = 0; d < 4; d++) vload(c, d);
                }
                unsigned zs = 0;
                bool top = false;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    zs += t[i];                                  // at most 16 x 2^24
                    if (WIDE && MODEL == 1 && (ch[c].flag[0] & 1)) {     // (uniform) the largest |v| that an arrival weighs
                        const i64 x = ch[c].vmax[16 * (i >> 2) + 4 * pg + (i & 3)];
                        vm = t[i] && x > vm ? x : vm;
                    }
                    t[i] += 0x808080u;
                    top |= t[i] >> 24 != 0;
                }
                if (!WIDE || ps == 0) z += zs;
                v4p w0, w1, w2, w3;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const unsigned ti[4] = {t[4 * i], t[4 * i + 1], t[4 * i + 2], t[4 * i + 3]};
                    unsigned dg[4];
                    byte_planes(ti, dg);
                    w0[i] = (int)(dg[0] ^ 0x80808080u);
                    w1[i] = (int)(dg[1] ^ 0x80808080u);
                    w2[i] = (int)(dg[2] ^ 0x80808080u);
                    w3[i] = (int)dg[3];
                }
                const bool any_top = __ballot(top) != 0;
#pragma unroll
                for (int d = 0; d < DN; d++) {
                    if constexpr (WIDE) {
                        if (gr == 0) vload(c, d0 + d);
                        else vform(c, d0 + d, gr);
                    }
                    const v4p (&x)[3] = vv[WIDE ? 0 : d];
                    acc[d][0] = mfma_i8(x[0], w0, acc[d][0]);
                    acc[d][1] = mfma_i8(x[0], w1, acc[d][1]);
                    acc[d][2] = mfma_i8(x[0], w2, acc[d][2]);
                    acc[d][3] = mfma_i8(x[1], w2, acc[d][3]);
                    acc[d][4] = mfma_i8(x[2], w2, acc[d][4]);
                    acc[d][1] = mfma_i8(x[1], w0, acc[d][1]);
                    acc[d][2] = mfma_i8(x[1], w1, acc[d][2]);
                    acc[d][3] = mfma_i8(x[2], w1, acc[d][3]);
                    acc[d][2] = mfma_i8(x[2], w0, acc[d][2]);
                    if (any_top) {
                        acc[d][3] = mfma_i8(x[0], w3, acc[d][3]);
                        acc[d][4] = mfma_i8(x[1], w3, acc[d][4]);
                        acc[d][5] = mfma_i8(x[2], w3, acc[d][5]);
                    }
                }
                c -= NW;
                if (FAST && c >= 0) scores(c);
            }
            if constexpr (WIDE) {                                // the groups' sums so far, in the wave's LDS
#pragma unroll
                for (int i = 0; i < 4 * DN; i++) {
                    i64* n = &num_s[wave][4 * d0 + i][lane];
                    const i64 x = (i64)((u64)sum64(i >> 2, i & 3) << (24 * gr));
                    *n = gr ? wadd(*n, x) : x;
                }
            }
        }
    };
    // 64-bit sums; the waves meet in wave 0
    auto finish = [&](auto wide) {
        constexpr bool WIDE = decltype(wide)::value;
        i64 num[16];
#pragma unroll
        for (int i = 0; i < 16; i++) num[i] = WIDE ? num_s[wave][i][lane] : sum64(i >> 2, i & 3);
        z += __shfl_xor(z, 16, 64);
        z += __shfl_xor(z, 32, 64);
        if (WIDE && MODEL == 1)
#pragma unroll
            for (int o = 16; o < 64; o <<= 1) { const i64 x = __shfl_xor(vm, o, 64); vm = x > vm ? x : vm; }
        if constexpr (NW > 1) {
            if (wave > 0) {
                if (lane < 16) z_s[wave][lane] = z;
                if (WIDE && MODEL == 1 && lane < 16) vm_s[wave][lane] = vm;
                if (!WIDE)
#pragma unroll
                    for (int i = 0; i < 16; i++) num_s[wave][i][lane] = num[i];
            }
            __syncthreads();
            if (wave > 0) return;
#pragma unroll
            for (int w = 1; w < NW; w++) {
                z += z_s[w][ql];
                if (WIDE && MODEL == 1) { const i64 x = vm_s[w][ql]; vm = x > vm ? x : vm; }
#pragma unroll
                for (int i = 0; i < 16; i++) num[i] = wadd(num[i], num_s[w][i][lane]);
            }
        }
        const bool live = p < g.pb;
        // (pythia_base2.py:139; values that three digits hold stay below 2^61 whatever the arrivals)
        if (WIDE && MODEL == 1 && live && (double)vm * (double)z >= 4611686018427387904.0) atomicOr(a.err, SM_ERR_RANGE);
        int zt; i64 zm;
        log2_parts(z, zt, zm);
        const i64 lg = a.tb.LOG2[zm], hp = a.tb.HPOW[zm];
        i64 w = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            num[i] = patt_out<MODEL>(a, num[i], zt, lg, hp, live);
            w |= iabs64(num[i]);
        }
        w |= __shfl_xor(w, 16, 64);
        w |= __shfl_xor(w, 32, 64);
        if (!live) return;
        const size_t r = (size_t)(slot * g.n + p - g.pa), at = r * 768 + h * 64 + 4 * pg;
        if (pg == 0) g.out.orw[r * 12 + h] = w;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            *reinterpret_cast<v4p*>(g.out.x32 + at + 16 * d) = v4p{(int)num[4 * d], (int)num[4 * d + 1], (int)num[4 * d + 2], (int)num[4 * d + 3]};
            if (!pnarrow(w))
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) g.out.x64[at + 16 * d + r4] = num[4 * d + r4];
        }
    };
    if (__builtin_expect(fl & 1, 0)) {                        // (uniform over the block)
        body(Flag<false>{}, Flag<true>{});
        finish(Flag<true>{});
        return;
    }
    if (ok32) body(Flag<true>{}, Flag<false>{});
    else body(Flag<false>{}, Flag<false>{});
    finish(Flag<false>{});
}
