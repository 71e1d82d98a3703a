// The prompt pass in large passes: hundreds to thousands of prompt positions through each layer at once
// (base2_stream.swift:74-91, 274-275 sends the whole prompt through each layer).  A pass holds `rows` rows, row
// r = slot n + (position - a) for S streams (slots) of n = b - a positions [a, b) each: whole prompts of several
// streams (a = 0), or part of one longer prompt (a a multiple of PCH).  Every number is the decode step's.
//   k_pgemm     a bank over all rows (base2.py:29-32): 128 x 64 output tiles of int8 MFMA over byte planes
//   k_kv_chunk  the pass's q, k, v of one head (base2.py:93) into the cache, and, for the pass's attention, the
//               byte planes of 64 positions in MFMA operand order
//   k_pattend   attention (base2.py:94-99) of 16 query positions a block, scores and value sums by MFMA
// The lights between them are the row kernels' (k_light, k_py_rows), one block a row.
// Why: in passes of 64 rows each launch (5-9 us, latency-bound) serves 64 rows, and the attention, one block a (head,
// row), reads a row's whole cache for one query.  Same box, a whole call: GPT-2, one 1000-word prompt 9.42 -> 2.99 ms;
// 19 prompts of 213 words and 17 words each 39.1 -> 13.5 ms; 64 prompts of 32 words and 128 words 85.5 -> 73.4 ms.
#include "sm_kernels.h"

typedef int v4p __attribute__((ext_vector_type(4)));
SMD v4p mfma_i8(v4p a, v4p b, v4p c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }

// ---------------------------------------------------------------------------------------------------------
// One bank over a pass of prompt rows.  Block: 128 rows x 64 columns, four waves of 64 x 32 (4 x 2 MFMA tiles,
// three int32 accumulators each: HH, MID, LL of the pile identity in sm_batch.hip); each 64-k step's operands (16 KB
// of light planes, 8 KB of plate) go through two LDS buffers, one step ahead in registers.  All operands lie in
// memory in MFMA order, so every global load and LDS access is a whole wave's consecutive 1 KB.
// Blocks are numbered so that each XCD (block index % 8) works on a contiguous run of row tiles.
struct PGemmArgs {
    int N, rows;
    const signed char* W; const int* csum; const int* we; const i64* bias;   // the plate (MfmaPlate)
    const signed char* planes; const int* rowinfo;                            // the rows' lights
    i64* Y;                       // [rows][N]; EPI_PLAIN_ADD: the stream, added to
    Tables tb;
    int* err;                     // the Pythia machine: its rshift assert sets SM_ERR_RANGE here
};
constexpr int PBM = 8, PBN = 4;   // 16-row and 16-column tiles a block
template <int K, int EPI>
__global__ __launch_bounds__(256, 2) void k_pgemm(PGemmArgs a) {
    constexpr int KS = K / 64, CH = (PBM + PBN) * 2, PER = CH / 4;   // 1 KB chunks a k step, a wave
    __shared__ v4p buf[2][CH][64];
    __shared__ i64 rc[16 * PBM][3];          // a row's pile constant, its power's row part, its factor
    __shared__ int any32;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = a.N / (16 * PBN), mb = (a.rows + 16 * PBM - 1) / (16 * PBM), total = nb * mb;
    // block b of XCD b % 8: the (b / 8)-th of that XCD's run of `per` tiles
    const int per = (total + 7) / 8, id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (id >= total || (int)(blockIdx.x >> 3) >= per) return;
    const int m0 = id / nb * PBM, n0 = id % nb * PBN;                // first row and column tile
    const int wm = (wave & 1) * 4, wn = (wave >> 1) * 2;
    // chunk c of a step: c < 2 PBM a light plane (row tile c / 2, plane c % 2), else a plate plane
    const v4p* src[PER];
    int step[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int c = wave + 4 * i;
        if (c < 2 * PBM) {
            src[i] = reinterpret_cast<const v4p*>(a.planes) + ((size_t)(m0 + c / 2) * KS * 3 + c % 2) * 64 + lane;
            step[i] = 3 * 64;
        } else {
            const int d = c - 2 * PBM;
            src[i] = reinterpret_cast<const v4p*>(a.W) + ((size_t)(n0 + d / 2) * KS * 2 + d % 2) * 64 + lane;
            step[i] = 2 * 64;
        }
    }
    v4p r[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) r[i] = src[i][0];
    // the rows' facts (ex, LS lo, LS hi, e2, SXh, SXl, n32768; gauged lights carry LS and its power factor)
    if (tid == 0) any32 = 0;
    __syncthreads();
    if (tid < 16 * PBM) {
        const int row = 16 * m0 + tid;
        if (row < a.rows) {
            const v4p f0 = *reinterpret_cast<const v4p*>(a.rowinfo + (size_t)row * 8);
            const v4p f1 = *reinterpret_cast<const v4p*>(a.rowinfo + (size_t)row * 8 + 4);
            rc[tid][0] = 32768 * (i64)f1[0] + 128 * (i64)f1[1] + 16384 * (i64)K + 128 * (i64)f1[2];
            if (EPI == EPI_GAUGED || EPI == EPI_GAUGED_EDGE) {
                const i64 ls = (i64)(((u64)(unsigned)f0[2] << 32) | (unsigned)f0[1]);
                rc[tid][1] = wsub(wmul((i64)f0[0] + 16, 65536), ls) >> 16;
                rc[tid][2] = f0[3];
            } else {
                rc[tid][1] = (i64)f0[0] + 16;
                rc[tid][2] = 0;
            }
            if (f1[2]) any32 = 1;
        } else {
            rc[tid][0] = rc[tid][1] = rc[tid][2] = 0;
        }
    }
    v4p acc[4][2][3];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j][0] = acc[i][j][1] = acc[i][j][2] = v4p{0, 0, 0, 0};
#pragma unroll 2
    for (int s = 0; s < KS; s++) {
        v4p(*bs)[64] = buf[s & 1];
#pragma unroll
        for (int i = 0; i < PER; i++) bs[wave + 4 * i][lane] = r[i];
        // the next step (the last one re-reads itself: no branch around the loads)
        const int nx = s + 1 < KS ? s + 1 : s;
#pragma unroll
        for (int i = 0; i < PER; i++) r[i] = src[i][(size_t)nx * step[i]];
        __syncthreads();
        v4p bh[2], bl[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            bh[j] = bs[2 * PBM + 2 * (wn + j)][lane];
            bl[j] = bs[2 * PBM + 2 * (wn + j) + 1][lane];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const v4p xh = bs[2 * (wm + i)][lane], xl = bs[2 * (wm + i) + 1][lane];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                acc[i][j][0] = mfma_i8(xh, bh[j], acc[i][j][0]);
                acc[i][j][1] = mfma_i8(xh, bl[j], acc[i][j][1]);
                acc[i][j][2] = mfma_i8(xl, bl[j], acc[i][j][2]);
                acc[i][j][1] = mfma_i8(xl, bh[j], acc[i][j][1]);
            }
        }
    }
    // (rare) a light of +32768 among the block's rows, held as 32767: its correction plane times the plate
    if (any32) {
        const v4p* A = reinterpret_cast<const v4p*>(a.planes) + ((size_t)(m0 + wm) * KS * 3 + 2) * 64 + lane;
        const v4p* B = reinterpret_cast<const v4p*>(a.W) + (size_t)(n0 + wn) * KS * 2 * 64 + lane;
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const v4p wh = B[((size_t)j * KS + s) * 128], wl = B[((size_t)j * KS + s) * 128 + 64];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const v4p cc = A[((size_t)i * KS + s) * 192];
                    acc[i][j][1] = mfma_i8(cc, wh, acc[i][j][1]);
                    acc[i][j][2] = mfma_i8(cc, wl, acc[i][j][2]);
                }
            }
    }
    // the epilogue: lane holds rows 4 (lane / 16) + q of each row tile, column lane % 16 of each column tile
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = 16 * (n0 + wn + j) + (lane & 15);
        const i64 ccol = 32768 * (i64)a.csum[2 * col] + 128 * (i64)a.csum[2 * col + 1];
        const i64 we = a.we[col], bc = a.bias[col];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int lr = 16 * (wm + i) + 4 * (lane >> 4), row = 16 * m0 + lr;
            i64 y[4];
            if constexpr (EPI == EPI_PLAIN_ADD) {      // bounded: a row past the last reads zeros
                const __amdgpu_buffer_rsrc_t ry = buf_rsrc(a.Y, (unsigned)a.rows * (unsigned)a.N * 8u);
#pragma unroll
                for (int q = 0; q < 4; q++) y[q] = buf_load8(ry, (unsigned)((row + q) * a.N + col) * 8u);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const i64 pile = 65536 * (i64)acc[i][j][0][q] + 256 * (i64)acc[i][j][1][q] + acc[i][j][2][q] +
                                 rc[lr + q][0] + ccol;
                const bool live = row + q < a.rows;
                i64 v, s;
                if constexpr (EPI == EPI_GAUGED || EPI == EPI_GAUGED_EDGE) {
                    // power(pile, (we + ex + 16) 65536 - LS) (base2.py:70): the fine part is the row's
                    v = wmul(pile, rc[lr + q][2]);
                    s = 16 - we - rc[lr + q][1];
                } else {
                    v = pile;
                    s = -(we + rc[lr + q][1]);
                }
                i64 o;
                if (__ballot(live && (u64)(s - 1) >= 62) == 0) {      // the usual rounding right shift
                    const int s32 = (int)s & 63;
                    o = wadd(v, (i64)1 << ((s32 - 1) & 63)) >> s32;
                } else {
                    if ((EPI == EPI_PLAIN || EPI == EPI_PLAIN_EDGE || EPI == EPI_PLAIN_ADD) && live && a.err && pyshift_fails(v, s))
                        atomicOr(a.err, SM_ERR_RANGE);
                    o = rsh(v, s);
                }
                o = wadd(o, bc);
                if constexpr (EPI == EPI_GAUGED_EDGE || EPI == EPI_PLAIN_EDGE) o = edge1(o, a.tb);
                if constexpr (EPI == EPI_PLAIN_ADD) o = wadd(y[q], o);
                y[q] = o;
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (row + q < a.rows) a.Y[(size_t)(row + q) * a.N + col] = y[q];
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// The pass's attention operands, one chunk of PCH positions of one (slot, head) each, in MFMA order:
//   K  [4 position tiles][kh, kl'][64 lanes][16]: lane l position l % 16, dimensions 16 (l / 16) ..; a key k' (a
//      +32768 held as 32767) is 256 kh + kl' + 128
//   V  [4 dimension tiles][3 digits][64 lanes][16]: lane l dimension l % 16, byte 4 i + r the position
//      16 i + 4 (l / 16) + r (the order in which a lane holds its scores); v = d0 + 256 d1 + 65536 d2, each digit
//      a signed byte
//   Q  [4 query tiles][qh, ql, qo][64 lanes][16]: lane l query l % 16; q = 256 (qh + qo) + ql, digits signed bytes
//      (qo: the 1 that a digit of 128 passes on)
// and per position ek, the +32768 mask km, eq, the sum of q; flag bit 0: a value that three digits do not hold,
// bit 1: a mask is set, bit 2: a qo is.
constexpr int PCH = 64;
struct PChunk {
    signed char K[4][2][1024];
    signed char V[4][3][1024];
    signed char Q[4][3][1024];
    i64 km[PCH];
    int ek[PCH], eq[PCH], sq[PCH], flag[PCH];        // flag[0]
};
struct PAttArgs {
    AttArgs a;                    // the layer's cache, QKV rows, out, tables, error word
    PChunk* ch;                   // [slot][head][nch]
    int n, pa, pb, nch, s0;       // rows a slot, its positions [pa, pb), chunks of [0, pb), the first slot's stream
};

// Block: one chunk of one (slot, head); wave w positions 16 w .. + 15, lane = dimension.  A chunk of this pass takes
// q, k, v from the qkv rows (base2.py:93: each through its own water level; pythia_base2.py:116-123: q and k turned
// first) and stores k and v; an earlier pass's chunk (all of it below pa) comes back from the cache.
template <int MODEL>
__global__ __launch_bounds__(256) void k_kv_chunk(PAttArgs g) {
    const AttArgs& a = g.a;
    __shared__ __align__(16) PChunk ch;
    const int c = blockIdx.x, h = blockIdx.y, slot = blockIdx.z, st = g.s0 + slot;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t hrow = (size_t)st * 12 + h;
    const bool fresh = PCH * c >= g.pa;
    if (threadIdx.x == 0) ch.flag[0] = 0;
    auto at = [&](int part) { return MODEL == 1 ? h * 192 + part * 64 + lane : part * 768 + h * 64 + lane; };
    __syncthreads();
    bool wide = false, masks = false, carry = false;
    const int off = (lane >> 4) * 256 + (lane & 15);       // + 16 (position % 16): the byte in an operand tile
    // four positions at a time: their loads together, and their values' digits a dword
#pragma unroll 1
    for (int gq = 0; gq < 4; gq++) {
        i64 q[4], k[4], v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int p = PCH * c + 16 * wave + 4 * gq + j;
            q[j] = k[j] = v[j] = 0;
            if (fresh && p < g.pb) {
                const i64* row = a.QKV + (size_t)(slot * g.n + p - g.pa) * 2304;
                q[j] = row[at(0)]; k[j] = row[at(1)]; v[j] = row[at(2)];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = 4 * gq + j, pl = 16 * wave + i, p = PCH * c + pl;
            int q16 = 0, k16 = 0, ekv = -16, eqv = -16;
            u64 km = 0;
            if (fresh) {
                if (p < g.pb) {                            // (uniform)
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
                    }
                    const int shq = water_shift(wave_or64(iabs64(q[j]))), shk = water_shift(wave_or64(iabs64(k[j])));
                    q16 = (int)rsh(q[j], shq); k16 = (int)rsh(k[j], shk);
                    eqv = -16 + shq; ekv = -16 + shk;
                    const size_t slotp = hrow * a.ctx + p;
                    key_store(a.K16 + slotp * 64, a.KM + slotp, k16, lane);
                    if (lane == 0) a.EK[slotp] = ekv;
                    v_store(a, hrow, p, lane, v[j]);
                    km = __ballot(k16 == 32768);
                    k16 = min(k16, 32767);
                }
            } else {                                       // (an earlier pass's position, below pb)
                const size_t slotp = hrow * a.ctx + p;
                k16 = a.K16[slotp * 64 + lane];
                km = (u64)a.KM[slotp];
                ekv = a.EK[slotp];
                v[j] = v_whole(a, hrow * a.ctx, p, lane);
            }
            wide |= (u64)(v[j] + 0x808080) >= 0x1000000ull;
            masks |= km != 0;
            // q in signed digits; a high digit of 128 as 127 + 1
            const int ql = (int)(signed char)q16, qh = (q16 - ql) >> 8, qo = qh == 128;
            carry |= qo != 0;
            ch.K[wave][0][off + 16 * i] = (signed char)(k16 >> 8);
            ch.K[wave][1][off + 16 * i] = (signed char)((k16 & 255) - 128);
            ch.Q[wave][0][off + 16 * i] = (signed char)(qh - qo);
            ch.Q[wave][1][off + 16 * i] = (signed char)ql;
            ch.Q[wave][2][off + 16 * i] = (signed char)qo;
            const int sq = wave_add32(q16);
            if (lane == 0) { ch.km[pl] = (i64)km; ch.ek[pl] = ekv; ch.eq[pl] = eqv; ch.sq[pl] = sq; }
        }
        // the values' digits: dimension tile lane / 16, lane' = lane % 16 + 16 gq, byte 4 wave + j
        unsigned t[4];
#pragma unroll
        for (int r = 0; r < 4; r++) t[r] = (unsigned)((int)v[r] + 0x808080);
        const unsigned l01 = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u), l23 = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u);
        const unsigned h01 = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u), h23 = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
        const int o = ((lane & 15) + 16 * gq) * 16 + 4 * wave;
        *reinterpret_cast<unsigned*>(&ch.V[lane >> 4][0][o]) = __builtin_amdgcn_perm(l23, l01, 0x05040100u) ^ 0x80808080u;
        *reinterpret_cast<unsigned*>(&ch.V[lane >> 4][1][o]) = __builtin_amdgcn_perm(l23, l01, 0x07060302u) ^ 0x80808080u;
        *reinterpret_cast<unsigned*>(&ch.V[lane >> 4][2][o]) = __builtin_amdgcn_perm(h23, h01, 0x05040100u) ^ 0x80808080u;
    }
    const int fl = (__ballot(wide) ? 1 : 0) | (__ballot(masks) ? 2 : 0) | (__ballot(carry) ? 4 : 0);
    if (lane == 0 && fl) atomicOr(&ch.flag[0], fl);
    __syncthreads();
    static_assert(sizeof(PChunk) % 16 == 0, "copied as 16-byte words");
    const v4p* s = reinterpret_cast<const v4p*>(&ch);
    v4p* d = reinterpret_cast<v4p*>(g.ch + ((size_t)slot * 12 + h) * g.nch + c);
    for (int i = threadIdx.x; i < (int)(sizeof(PChunk) / 16); i += 256) d[i] = s[i];
}

// ---------------------------------------------------------------------------------------------------------
// Attention of 16 query positions of one (slot, head), base2.py:94-99 (pythia_base2.py:125-141).  Wave w takes the
// chunks w, w + NW, .. of the positions up to the tile's last, twice: once for the queries' maxima, then (scores
// formed again) for the arrivals against them and the value sums.  Scores: rows are positions and columns queries,
// so lane l holds query l % 16 at positions 16 i + 4 (l / 16) + r of a chunk; those 16 arrivals, split into digit
// bytes, are the B operand of the value product as they stand, with the chunk's V in the same order (PChunk).  An
// arrival, at most 2^24, is three signed digits and a 0/1 fourth, which most chunks lack; the products of equal
// weight share one int32 accumulator (at most 4 x 2^20 a chunk: callers keep positions below 16384, so none
// passes 2^31).  The waves' sums meet in LDS in 64 bits.
// A head with a value that three digits do not hold takes pattend_wide: a query at a time, one wave each.
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
    return 256 * (c->Q[tile][0][o] + c->Q[tile][2][o]) + c->Q[tile][1][o];
}
template <int MODEL>
SMD void pattend_wide(const PAttArgs& g, const PChunk* ch, int h, int slot, int p, int lane, int* q_s, int* w_s) {
    const AttArgs& a = g.a;
    const PChunk* cq = ch + p / PCH;
    const size_t hrow = (size_t)(g.s0 + slot) * 12 + h, hb = hrow * a.ctx;
    q_s[lane] = pchunk_q(cq, (p % PCH) >> 4, p & 15, lane);
    const i64 eq = cq->eq[p % PCH];
    auto score = [&](int s) -> i64 {                        // lane's position s <= p against q (LDS, the wave's own)
        const short* kr = a.K16 + (hb + s) * 64;
        const u64 km = (u64)a.KM[hb + s];
        i64 dot = 0;
        for (int d = 0; d < 64; d++) dot += (i64)q_s[d] * (kr[d] + (int)((km >> d) & 1));
        return patt_score<MODEL>(a, dot, eq + a.EK[hb + s]);
    };
    i64 mx = INT64_MIN;
    for (int s = lane; s <= p; s += 64) { const i64 v = score(s); mx = v > mx ? v : mx; }
    mx = wave_reduce64(mx, OpMax());
    i64 num = 0, z = 0, vm = 0;
    for (int b = 0; b <= p; b += 64) {
        const int w = b + lane <= p ? tab_arr(a.tb, wsub(mx, score(b + lane))) : 0;
        z += w;
        w_s[lane] = w;
        for (int s = 0; s < 64 && b + s <= p; s++) {
            const i64 ws = w_s[s], x = v_whole(a, hb, b + s, lane);
            num = wadd(num, wmul(ws, x));
            if (MODEL == 1 && ws) { const i64 ax = iabs64(x); vm = ax > vm ? ax : vm; }
        }
    }
    z = wave_reduce64(z, OpAdd());
    if (MODEL == 1 && (double)vm * (double)z >= 4611686018427387904.0) atomicOr(a.err, SM_ERR_RANGE);
    int zt; i64 zm;
    log2_parts(z, zt, zm);
    a.out[(size_t)(slot * g.n + p - g.pa) * 768 + h * 64 + lane] =
        patt_out<MODEL>(a, num, zt, a.tb.LOG2[zm], a.tb.HPOW[zm], true);
}

template <int MODEL, int NW>
__global__ __launch_bounds__(64 * NW, 2) void k_pattend(PAttArgs g) {
    const AttArgs& a = g.a;
    __shared__ i64 mx_s[NW][16], z_s[NW][16];
    __shared__ i64 num_s[NW > 1 ? NW - 1 : 1][NW > 1 ? 16 : 1][64];
    __shared__ __align__(16) int q_s[NW][64], w_s[NW][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ql = lane & 15, pg = lane >> 4;
    const int h = blockIdx.y, slot = blockIdx.z;
    const int p0 = g.pa + 16 * (int)(gridDim.x - 1 - blockIdx.x);     // the longest tiles first
    const int plast = min(p0 + 15, g.pb - 1), nc = plast / PCH + 1, p = p0 + ql;
    const PChunk* ch = g.ch + ((size_t)slot * 12 + h) * g.nch;
    int fl = 0;                                              // any chunk's flags
    for (int c = lane; c < nc; c += 64) fl |= ch[c].flag[0];
    fl = (int)wave_or32((unsigned)fl);
    if (fl & 1) {                                            // (uniform over the block)
        for (int i = wave; i < 16 && p0 + i < g.pb; i += NW)
            pattend_wide<MODEL>(g, ch, h, slot, p0 + i, lane, q_s[wave], w_s[wave]);
        return;
    }
    const PChunk* cq = ch + p0 / PCH;
    const int qt = (p0 % PCH) >> 4;
    const v4p qh = *reinterpret_cast<const v4p*>(&cq->Q[qt][0][16 * lane]), qll = *reinterpret_cast<const v4p*>(&cq->Q[qt][1][16 * lane]),
              qo = *reinterpret_cast<const v4p*>(&cq->Q[qt][2][16 * lane]);
    const bool carry = cq->flag[0] & 4;
    const i64 eq = cq->eq[p0 % PCH + ql], sq128 = 128 * (i64)cq->sq[p0 % PCH + ql];
    // a chunk's 16 scores of this lane: positions 64 c + 16 i + 4 pg + r (past p: INT64_MIN)
    auto scores = [&](int c, i64 (&sc)[16]) {
        const PChunk* cc = ch + c;
        v4p kh[4], kl[4], ek[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            kh[i] = *reinterpret_cast<const v4p*>(&cc->K[i][0][16 * lane]);
            kl[i] = *reinterpret_cast<const v4p*>(&cc->K[i][1][16 * lane]);
            ek[i] = *reinterpret_cast<const v4p*>(&cc->ek[16 * i + 4 * pg]);
        }
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
                i64 dot = 65536 * (i64)hh[r] + 256 * (i64)mid[r] + ll[r] + sq128;
                const int pl = 16 * i + 4 * pg + r, s = PCH * c + pl;
                if (fl & 2) {                                // (rare) keys holding a +32768: one more of q there
                    for (u64 m = (u64)cc->km[pl]; m; m &= m - 1) dot += pchunk_q(cq, qt, ql, __builtin_ctzll(m));
                }
                const i64 v = patt_score<MODEL>(a, dot, eq + ek[i][r]);
                sc[4 * i + r] = s <= p ? v : INT64_MIN;
            }
        }
    };
    i64 M = INT64_MIN;
    for (int c = wave; c < nc; c += NW) {
        i64 sc[16];
        scores(c, sc);
#pragma unroll
        for (int i = 0; i < 16; i++) M = sc[i] > M ? sc[i] : M;
    }
    // the queries' maxima (base2.py:96): the four lane groups, then the waves
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) { const i64 x = __shfl_xor(M, o, 64); M = x > M ? x : M; }
    if constexpr (NW > 1) {
        if (lane < 16) mx_s[wave][lane] = M;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; w++) M = mx_s[w][ql] > M ? mx_s[w][ql] : M;
    }
    // arrivals (base2.py:96-97), their sum, the value sums (base2.py:98)
    v4p acc[4][6];
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int k = 0; k < 6; k++) acc[d][k] = v4p{0, 0, 0, 0};
    i64 z = 0;
    const __amdgpu_buffer_rsrc_t ra = buf_rsrc(a.tb.ARR, (unsigned)a.tb.alen * 4u);   // 0 past the table (base2.py:97)
    for (int c = wave; c < nc; c += NW) {
        const PChunk* cc = ch + c;
        unsigned t[16];
        {
            i64 sc[16];
            scores(c, sc);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const i64 d = wsub(M, sc[i]);
                const bool in = PCH * c + 16 * (i >> 2) + 4 * pg + (i & 3) <= p && (u64)d < (u64)a.tb.alen;
                t[i] = (unsigned)buf_load1(ra, in ? (unsigned)d * 4u : 0xFFFFFFF0u);
            }
        }
        unsigned zs = 0;
        bool top = false;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            zs += t[i];                                      // at most 16 x 2^24
            t[i] += 0x808080u;
            top |= t[i] >> 24 != 0;
        }
        z += zs;
        v4p w0, w1, w2, w3;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned l01 = __builtin_amdgcn_perm(t[4 * i + 1], t[4 * i], 0x05010400u), l23 = __builtin_amdgcn_perm(t[4 * i + 3], t[4 * i + 2], 0x05010400u);
            const unsigned h01 = __builtin_amdgcn_perm(t[4 * i + 1], t[4 * i], 0x07030602u), h23 = __builtin_amdgcn_perm(t[4 * i + 3], t[4 * i + 2], 0x07030602u);
            w0[i] = (int)(__builtin_amdgcn_perm(l23, l01, 0x05040100u) ^ 0x80808080u);
            w1[i] = (int)(__builtin_amdgcn_perm(l23, l01, 0x07060302u) ^ 0x80808080u);
            w2[i] = (int)(__builtin_amdgcn_perm(h23, h01, 0x05040100u) ^ 0x80808080u);
            w3[i] = (int)__builtin_amdgcn_perm(h23, h01, 0x07060302u);
        }
        const bool any_top = __ballot(top) != 0;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const v4p v0 = *reinterpret_cast<const v4p*>(&cc->V[d][0][16 * lane]), v1 = *reinterpret_cast<const v4p*>(&cc->V[d][1][16 * lane]),
                      v2 = *reinterpret_cast<const v4p*>(&cc->V[d][2][16 * lane]);
            acc[d][0] = mfma_i8(v0, w0, acc[d][0]);
            acc[d][1] = mfma_i8(v0, w1, acc[d][1]);
            acc[d][2] = mfma_i8(v0, w2, acc[d][2]);
            acc[d][3] = mfma_i8(v1, w2, acc[d][3]);
            acc[d][4] = mfma_i8(v2, w2, acc[d][4]);
            acc[d][1] = mfma_i8(v1, w0, acc[d][1]);
            acc[d][2] = mfma_i8(v1, w1, acc[d][2]);
            acc[d][3] = mfma_i8(v2, w1, acc[d][3]);
            acc[d][2] = mfma_i8(v2, w0, acc[d][2]);
            if (any_top) {
                acc[d][3] = mfma_i8(v0, w3, acc[d][3]);
                acc[d][4] = mfma_i8(v1, w3, acc[d][4]);
                acc[d][5] = mfma_i8(v2, w3, acc[d][5]);
            }
        }
    }
    // 64-bit sums: lane holds dimensions 16 d + 4 pg + r of query ql; the waves meet in wave 0
    i64 num[16];
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            u64 n = 0;
#pragma unroll
            for (int k = 5; k >= 0; k--) n = (n << 8) + (u64)(i64)acc[d][k][r];
            num[4 * d + r] = (i64)n;
        }
    z += __shfl_xor(z, 16, 64);
    z += __shfl_xor(z, 32, 64);
    if constexpr (NW > 1) {
        if (wave > 0) {
            if (lane < 16) z_s[wave][lane] = z;
#pragma unroll
            for (int i = 0; i < 16; i++) num_s[wave - 1][i][lane] = num[i];
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 1; w < NW; w++) {
            z += z_s[w][ql];
#pragma unroll
            for (int i = 0; i < 16; i++) num[i] = wadd(num[i], num_s[w - 1][i][lane]);
        }
    }
    if (p >= g.pb) return;
    int zt; i64 zm;
    log2_parts(z, zt, zm);
    const i64 lg = a.tb.LOG2[zm], hp = a.tb.HPOW[zm];
    i64* o = a.out + (size_t)(slot * g.n + p - g.pa) * 768 + h * 64 + 4 * pg;
#pragma unroll
    for (int i = 0; i < 16; i++) o[16 * (i >> 2) + (i & 3)] = patt_out<MODEL>(a, num[i], zt, lg, hp, true);
}
