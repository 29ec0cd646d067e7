// Causal ALiBi attention at head width 4 (the spec's shape, ops.py:186-258): one workgroup per (sequence, head), T a
// multiple of 32 up to 256. The default kernels (k_atencao4m, k_atencao4m_back) use matrix cores, a wave per
// two stripes of 16 query rows; the layouts of jt_atencao_linhas have one or two query rows per thread, T / NR threads rounded up to whole
// waves of 64, where the threads without a row take part in the reductions with neutral values only.
//
// Forward: q, k, v of the head aligned to the head's largest exponent over the sequence with GA guard bits
// (a = rnd(m << GA, emx - e)); u_ij = rnd(q_i . k_j, -(eq + ek - 1 + 8)) - (i - j) << incl with
// incl = 8 - h // 8 (ops.py:208; H <= 64); ex = exp_int(max - u) >> 3; P = min((ex * (2^28 / sum ex) + 2^19) >> 20, 255) as uint8,
// stored transposed [j][i]; o_i = sum_j P_ij v_j (raw, exponent ev - 8).
// Backward: gP = dO . v^T shrunk to 15 bits by its causal maximum (or an upper bound in the LIMITE variant),
// s_i = rnd(sum_j P gP, 8), dS = P (gP - s) shrunk to DSB bits, then gq = dS k, gk = dS^T q, gv = P^T dO
// as raw outputs [M, 3D].
// Every product is a 24-bit one (mul24): aligned values |a| <= 128 << GA <= 2048 (GA <= 4), P <= 255, ex <= 4095,
// 2^28 / sum ex <= 2^16 (the row maximum alone adds 4095 to the sum), |gP'| <= 2^15, |gP' - s| < 2^17 (a row of P
// sums to at most 256 + T / 2), |dS| <= 2^12.
#include "jt_comum.h"

__device__ __forceinline__ int bloco_max(int v, int* red) {
    v = g_max<64>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    int r = SEM_TOPO;
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) r = max(r, red[i]);
    return r;
}

// Rows per thread (jt_atencao_linhas, jatai_cuda.cu:1091): with NR = 1 thread t owns query row t; with NR = 2 it
// owns rows t and T - 1 - t (t < T / 2), a short and a long causal row, so the threads' work is even. The backward
// assigns its columns (keys) the same way. -1: no row (a thread past the sequence).
template <int NR>
__device__ __forceinline__ int linha_de(int t, int k, int T) {
    if constexpr (NR == 1) return t < T ? t : -1;
    else return t < T / 2 ? (k == 0 ? t : T - 1 - t) : -1;
}

// aligned values of the thread's tokens for one head slice of 4 columns (jatai_cuda.cu:789-818 restated):
// al[t][d] = rnd(m << GA, emx - e) with emx the head's largest exponent over the sequence; eo = emx - GA
template <int NR>
__device__ __forceinline__ void alinha4(const int8_t* m, const int8_t* E, int ld, int col, int blk, int b0, int T, int GA, int* red,
                                        int (*al)[4], int& eo) {
    int e[NR], w[NR], tk[NR], emx = SEM_TOPO;
#pragma unroll
    for (int k = 0; k < NR; k++) {
        tk[k] = linha_de<NR>(threadIdx.x, k, T);
        e[k] = tk[k] >= 0 ? (int)E[(size_t)(b0 + tk[k]) * (ld / blk) + col / blk] : SEM_TOPO;
        w[k] = tk[k] >= 0 ? *reinterpret_cast<const int*>(m + (size_t)(b0 + tk[k]) * ld + col) : 0;
        emx = max(emx, e[k]);
    }
    emx = bloco_max(emx, red);
#pragma unroll
    for (int k = 0; k < NR; k++)
        if (tk[k] >= 0) {
#pragma unroll
            for (int d = 0; d < 4; d++) al[tk[k]][d] = rnd_d(((w[k] << (24 - 8 * d)) >> 24) << GA, emx - e[k]);
        }
    eo = emx - GA;
}

template <int TMAX, int NR>
__global__ void __launch_bounds__(TMAX) k_atencao4(const int8_t* __restrict__ qm, const int8_t* __restrict__ qE, int* __restrict__ Oacc,
                                                   int16_t* __restrict__ Oe, uint8_t* __restrict__ P, int T, int H, int D, int blk, int GA,
                                                   int kid) {
    __shared__ int qa[TMAX][4], ka[TMAX][4], va[TMAX][4];
    __shared__ int red[TMAX / 64];
    const int b = blockIdx.x / H, h = blockIdx.x % H, ld = 3 * D, b0 = b * T;
    int eq, ek, ev;
    alinha4<NR>(qm, qE, ld, h * 4, blk, b0, T, GA, red, qa, eq);
    alinha4<NR>(qm, qE, ld, D + h * 4, blk, b0, T, GA, red, ka, ek);
    alinha4<NR>(qm, qE, ld, 2 * D + h * 4, blk, b0, T, GA, red, va, ev);
    __syncthreads();
    const int su = -(eq + ek - 1 + 8), incl = 8 - h / 8;
    uint8_t* Pb = P + (size_t)blockIdx.x * T * T;
#pragma unroll 1
    for (int k = 0; k < NR; k++) {                                  // no barrier below: threads without a row leave
        const int i = linha_de<NR>(threadIdx.x, k, T), row = b0 + i;
        if (i < 0) continue;
        const int q0 = qa[i][0], q1 = qa[i][1], q2 = qa[i][2], q3 = qa[i][3];
        const long long idx = (long long)row * D + h * 4;
        auto sc = [&](int j) {
            const int s = mul24(q0, ka[j][0]) + mul24(q1, ka[j][1]) + mul24(q2, ka[j][2]) + mul24(q3, ka[j][3]);
            return rnd(s, su, kid, idx) - ((i - j) << incl);
        };
        int mx = U_MIN;
        for (int j = 0; j <= i; j++) mx = max(mx, sc(j));
        int soma = 0;
        for (int j = 0; j <= i; j++) soma += exp_dif(mx, sc(j)) >> 3;
        if (soma <= 0) { reporta(E_DIV, kid, idx, soma, mx); soma = 1; }
        const int inv = (1 << 28) / soma;
        int o[4] = {0, 0, 0, 0};
        for (int j = 0; j < T; j++) {
            int p = 0;
            if (j <= i) {
                const int ex = exp_dif(mx, sc(j)) >> 3;
                p = min((mul24(ex, inv) + (1 << 19)) >> 20, 255);
#pragma unroll
                for (int d = 0; d < 4; d++) o[d] += mul24(p, va[j][d]);
            }
            Pb[(size_t)j * T + i] = (uint8_t)p;
        }
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const size_t x = (size_t)row * D + h * 4 + d;
            if (o[d] >= LIM || o[d] <= -LIM) reporta(E_ACUM, kid, x, o[d], -3);
            Oacc[x] = o[d];
            Oe[x] = (int16_t)(ev - 8);
        }
    }
}

template <int TMAX, int LIMITE, int NR>
__global__ void __launch_bounds__(TMAX) k_atencao4_back(const int8_t* __restrict__ gom, const int8_t* __restrict__ goE,
                                                        const int8_t* __restrict__ qm, const int8_t* __restrict__ qE,
                                                        const uint8_t* __restrict__ P, int* __restrict__ Gacc, int16_t* __restrict__ Ge,
                                                        int T, int H, int D, int blk, int GA, int DSB, int kid) {
    __shared__ int goa[TMAX][4], qa[TMAX][4], ka[TMAX][4], va[TMAX][4], slin[TMAX];
    __shared__ int red[TMAX / 64];
    const int b = blockIdx.x / H, h = blockIdx.x % H, ld = 3 * D, b0 = b * T;
    const uint8_t* Pb = P + (size_t)blockIdx.x * T * T;
    int eq, ek, ev, ego;
    alinha4<NR>(gom, goE, D, h * 4, blk, b0, T, GA, red, goa, ego);
    alinha4<NR>(qm, qE, ld, h * 4, blk, b0, T, GA, red, qa, eq);
    alinha4<NR>(qm, qE, ld, D + h * 4, blk, b0, T, GA, red, ka, ek);
    alinha4<NR>(qm, qE, ld, 2 * D + h * 4, blk, b0, T, GA, red, va, ev);
    __syncthreads();
    // the thread's rows (-1: none); every thread stays for the barriers of the block reductions
    int lin[NR];
#pragma unroll
    for (int k = 0; k < NR; k++) lin[k] = linha_de<NR>(threadIdx.x, k, T);
    auto gp_ij = [&](int i, int j) {
        return mul24(goa[i][0], va[j][0]) + mul24(goa[i][1], va[j][1]) + mul24(goa[i][2], va[j][2]) + mul24(goa[i][3], va[j][3]);
    };
    // shift of gP: exact causal maximum, or max_i ||dO_i||_inf * max_j ||v_j||_1
    int mg = 0;
    if constexpr (LIMITE) {
        int b1 = 0, b2 = 0;
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const int i = lin[k];
            if (i < 0) continue;
            b1 = max(b1, max(max(abs(goa[i][0]), abs(goa[i][1])), max(abs(goa[i][2]), abs(goa[i][3]))));
            b2 = max(b2, abs(va[i][0]) + abs(va[i][1]) + abs(va[i][2]) + abs(va[i][3]));
        }
        mg = bloco_max(b1, red) * bloco_max(b2, red);
    } else {
#pragma unroll
        for (int k = 0; k < NR; k++)
            for (int j = 0; j <= lin[k]; j++) mg = max(mg, abs(gp_ij(lin[k], j)));
        mg = bloco_max(mg, red);
    }
    const int sh = max(bitlen(mg) - 15, 0), egp = ego + ev + sh;
    // s_i = rnd(sum_j P_ij gP'_ij, 8)
    int sl[NR], pm = 0, gm = 0;
#pragma unroll
    for (int k = 0; k < NR; k++) {
        const int i = lin[k];
        int s = 0;
        for (int j = 0; j <= i; j++) {
            const int p = Pb[(size_t)j * T + i], gp = rnd_d(gp_ij(i, j), sh);
            s += mul24(p, gp);
            if constexpr (LIMITE) { pm = max(pm, p); gm = max(gm, abs(gp)); }
        }
        if (s >= LIM || s <= -LIM) reporta(E_ACUM, kid, (long long)(b0 + i) * ld + h * 4, s, -4);
        sl[k] = rnd_d(s, 8);
        if (i >= 0) slin[i] = sl[k];
    }
    // shift of dS: exact maximum of |P (gP' - s)|, or max P * (max |gP'| + max |s|)
    int md = 0;
    if constexpr (LIMITE) {
        int sm = 0;
#pragma unroll
        for (int k = 0; k < NR; k++) sm = max(sm, lin[k] >= 0 ? abs(sl[k]) : 0);
        const int pmb = bloco_max(pm, red), gmb = bloco_max(gm, red), smb = bloco_max(sm, red);
        md = pmb * (gmb + smb);
    } else {
#pragma unroll
        for (int k = 0; k < NR; k++)
            for (int j = 0; j <= lin[k]; j++) md = max(md, abs(mul24((int)Pb[(size_t)j * T + lin[k]], rnd_d(gp_ij(lin[k], j), sh) - sl[k])));
        md = bloco_max(md, red);                                   // also publishes slin
    }
    const int sh2 = max(bitlen(md) - DSB, 0), eds = egp - 9 + sh2;
    // no barrier below: a thread without rows is done
#pragma unroll 1
    for (int k = 0; k < NR; k++) {
        const int i = lin[k];
        if (i < 0) continue;
        // row i: gq_i = sum_j dS_ij k_j
        int gq[4] = {0, 0, 0, 0};
        for (int j = 0; j <= i; j++) {
            const int ds = rnd_d(mul24((int)Pb[(size_t)j * T + i], rnd_d(gp_ij(i, j), sh) - sl[k]), sh2);
#pragma unroll
            for (int d = 0; d < 4; d++) gq[d] += mul24(ds, ka[j][d]);
        }
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const size_t o = (size_t)(b0 + i) * ld + h * 4 + d;
            if (gq[d] >= LIM || gq[d] <= -LIM) reporta(E_ACUM, kid, o, gq[d], -5);
            Gacc[o] = gq[d];
            Ge[o] = (int16_t)(eds + ek);
        }
        // column jj = i: gk_j = sum_{i >= j} dS_ij q_i, gv_j = sum_{i >= j} P_ij dO_i (row j of the stored P is contiguous)
        const int jj = i;
        const int v0 = va[jj][0], v1 = va[jj][1], v2 = va[jj][2], v3 = va[jj][3];
        const uint8_t* Pr = Pb + (size_t)jj * T;
        int gk[4] = {0, 0, 0, 0}, gv[4] = {0, 0, 0, 0};
        for (int ii = jj; ii < T; ii++) {
            const int p = Pr[ii];
            const int gp = mul24(goa[ii][0], v0) + mul24(goa[ii][1], v1) + mul24(goa[ii][2], v2) + mul24(goa[ii][3], v3);
            const int ds = rnd_d(mul24(p, rnd_d(gp, sh) - slin[ii]), sh2);
#pragma unroll
            for (int d = 0; d < 4; d++) { gk[d] += mul24(ds, qa[ii][d]); gv[d] += mul24(p, goa[ii][d]); }
        }
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const size_t o = (size_t)(b0 + jj) * ld + h * 4 + d;
            if (gk[d] >= LIM || gk[d] <= -LIM) reporta(E_ACUM, kid, o + D, gk[d], -5);
            if (gv[d] >= LIM || gv[d] <= -LIM) reporta(E_ACUM, kid, o + 2 * D, gv[d], -5);
            Gacc[o + D] = gk[d];
            Ge[o + D] = (int16_t)(eds + eq);
            Gacc[o + 2 * D] = gv[d];
            Ge[o + 2 * D] = (int16_t)(ego - 8);
        }
    }
}

// ---------------------------------------------------------------------------------------------- matrix cores
// The same arithmetic on f16 MFMA (16x16x16), one workgroup per (sequence, head), a wave per two stripes of 16 query
// rows (w and T / 16 - 1 - w, a short and a long one: T / 16 + 1 tiles in every wave), T <= TMAX. Aligned values |a| <= 2048 are exact in f16 and a product of 4 of them sums to at most 2^24: the
// fp32 scores are the exact integers. Only 4 of the 16 contraction slots of a score tile hold dimensions (lanes
// lg = 0; the A or B operand is 0 in the others), which costs nothing where the vector unit is the bound: the work
// that is left per pair is the softmax's or the dS chain's own.
//
// Forward: score tiles transposed (rows = keys 16 t + 4 lg + v, column = query 16 st + lr), so a lane's values all
// belong to one query: maxima and sums are in registers but for two exchanges across lg, and its four P are the B
// operand of O^T = V^T P^T as they stand. For a rounding shift su >= 3 a score is rounded and its ALiBi term
// subtracted by one FMA, s 2^-su + (1.5 2^23 - ((i - j) << incl)): the sum stays in [2^23, 2^24), where floats are
// spaced by 1 (|s| 2^-su <= 2^21, (i - j) << incl < 2^16), and the term is even (incl >= 1), so the addition's rounding
// to nearest even is the spec's of s 2^-su. The bits are u plus a constant, which the differences max - u drop.
// Backward: gP tiles with rows = queries 16 st + 4 lg + v, column = key 16 t + lr: four P of a lane are one 4-byte
// load, and dS, P are the B operands of gk^T = Q^T dS and gv^T = dO^T P as they stand. For gq^T = K^T dS^T a product
// with the identity transposes dS's tile (exact). dS (|dS| <= 2^DSB) is split as a 2^LB + b, |a|, |b| <= 2^(LB - 1) with
// LB = 7 (T <= 128, DSB 12) or 6 (T <= 256, DSB 11), so that each piece's sum over T terms stays within 2^24: exact in
// fp32. P <= 255 times |dO| <= 2048 over 32 rows stays within 2^24: gv moves to int32 every two tiles. dS and P
// tiles pass from the row waves to the column waves through LDS (12 bytes per lane and tile).
//
// Bound by the vector unit (585 instructions per wave of 16 rows forward and 1066 backward with a wave per stripe, over
// half of the kernels' time) and by the launch and the chain of barriers of one short workgroup per head. At 16
// sequences x 128 tokens and 64 heads of 4: forward 25 -> 16 us, backward 36 -> 24 against 8 lanes per query row (24-bit
// products, operands read from LDS per pair); at 13 x 256 tokens and 32 heads, against one row per thread, forward and
// backward with both quantizations 303 -> 75 us. A wave per stripe measured 15 and 25 us, and 28 before neighbouring
// heads shared an XCD; at most 64 registers in the backward (8 waves per SIMD) spilled 24 of them: 35 us. At 16 x 256 tokens
// and 64 heads 50 and 84 us, the vector unit half busy: 164 registers forward and 114 backward leave 3 and 4 waves per SIMD.
// One to three sequences of 96 tokens or fewer and 32 heads leave CUs idle either way; there 8 lanes per row had more waves
// on a head: backward 8.3-10.1 us with them, 8.7-9.9 here, forward 6.0-7.5 and 6.1-7.2.
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef short s2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
namespace at4 {
constexpr int PAD = 16;                                              // row padding: P bytes, transposed operands
constexpr float MG = 0x1.8p23f;                                      // 1.5 2^23
constexpr int MGB = 0x4b400000;
// LDS of a launch (bytes): exp table, P [T][T + PAD], two [T] x 4 f16 operands, one [4][T + PAD] f16
inline size_t lds_frente(int T) { return EXP_N * 2 + (size_t)T * (T + PAD) + 2 * 8 * (size_t)T + 8 * ((size_t)T + PAD); }
// dS (8) and P (4) of a lane per causal tile, two [T] x 4 and three [4][T + PAD] f16 operands
inline size_t lds_tras(int T) {
    const size_t n = T / 16;
    return n * (n + 1) / 2 * 64 * 12 + 2 * 8 * (size_t)T + 3 * 8 * ((size_t)T + PAD);
}
// head of workgroup g of n: the dispatcher deals workgroups to the 8 XCDs in turn, and 16 heads share the 64-byte lines of
// their operands and results (4 and 16 bytes a head and token): neighbouring heads go to one XCD's L2
__device__ __forceinline__ int cabeca(int g, int n) { return n % 8 == 0 ? (g & 7) * (n / 8) + (g >> 3) : g; }
__device__ __forceinline__ int max_lg(int v) { v = max(v, __shfl_xor(v, 16)); return max(v, __shfl_xor(v, 32)); }
__device__ __forceinline__ int soma_lg(int v) { v += __shfl_xor(v, 16); return v + __shfl_xor(v, 32); }
// workgroup maximum of a value >= 0 over n <= 8 waves; red is not in use by anyone. Wave w fills slots w, w + n, ...
__device__ __forceinline__ int grupo_max(int v, int (&red)[8], int n) {
    v = g_max<64>(v);
    if ((threadIdx.x & 63) == 0)
        for (int x = threadIdx.x >> 6; x < 8; x += n) red[x] = v;
    __syncthreads();
    return max(max(max(red[0], red[1]), max(red[2], red[3])), max(max(red[4], red[5]), max(red[6], red[7])));
}
// Eight wait states after the last MFMA of an accumulator whose use more than one path reaches: the compiler counts the
// states between an MFMA and a use of its result along one path only, and can leave too few on another. A use that a single
// path reaches (gv's drain below, behind a branch of its own) has the compiler's own wait. tests/test_codigo.py counts the
// states of every MFMA of the built library on every path.
__device__ __forceinline__ void pronto(f4_t& a) { asm volatile("s_nop 7" : "+v"(a)); }
// pieces of four dS: d = a 2^LB + b
template <int LB>
__device__ __forceinline__ void pedacos(const s2_t (&d)[2], h4_t& a, h4_t& b) {
    constexpr short M2 = 1 << (LB - 1);
#pragma unroll
    for (int k = 0; k < 2; k++) {                                    // 0x6600 + n (|n| < 512): the f16 1536 + n
        const s2_t t = d[k] + s2_t{M2, M2}, ta = (t >> LB) + s2_t{0x6600, 0x6600}, tb = (t & s2_t{2 * M2 - 1, 2 * M2 - 1}) | s2_t{0x6600, 0x6600};
        const h2_t ha = __builtin_bit_cast(h2_t, ta) - h2_t{1536, 1536}, hb = __builtin_bit_cast(h2_t, tb) - h2_t{1536 + M2, 1536 + M2};
        a[2 * k] = ha[0]; a[2 * k + 1] = ha[1];
        b[2 * k] = hb[0]; b[2 * k + 1] = hb[1];
    }
}
// four small integers (|v| <= 64: exact) as f16
__device__ __forceinline__ h4_t para_f16(const f4_t& v) {
    const auto x = __builtin_amdgcn_cvt_pkrtz(v[0], v[1]), y = __builtin_amdgcn_cvt_pkrtz(v[2], v[3]);
    return h4_t{(_Float16)x[0], (_Float16)x[1], (_Float16)y[0], (_Float16)y[1]};
}
// four bytes as f16: 0x6400 + p is the f16 1024 + p
__device__ __forceinline__ h4_t bytes_f16(unsigned p) {
    const h2_t x = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, p, 0x04010400u)) - h2_t{1024, 1024};
    const h2_t y = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, p, 0x04030402u)) - h2_t{1024, 1024};
    return h4_t{x[0], x[1], y[0], y[1]};
}
}  // namespace at4

// The head's slices q, k, v (f = 0, 1, 2) and, with DO, dO (f = 3), aligned at once by 2 T threads (the alignment of
// alinha4<1>): thread x < T takes token x of slices 0 and 2, thread T + t token t of slices 1 and 3, so all the loads,
// reductions and roundings run side by side. T is a multiple of 32, so the 32 lanes of a half wave share their slices
// and its maxima combine per half wave, into 8 slots a slice (all filled). a[k]: the thread's aligned values of slice
// f = par + 2 k (0 for a slice that is not there); guarda(f, t, h): their f16 values to LDS; entre() runs between the loads
// and the reduction. The caller's barrier publishes.
template <bool DO, class Guarda, class Entre>
__device__ __forceinline__ void alinha4f(const int8_t* __restrict__ gom, const int8_t* __restrict__ goE, const int8_t* __restrict__ qm,
                                         const int8_t* __restrict__ qE, int D, int h, int blk, int b0, int T, int GA, int (&red)[4][8],
                                         int (&a)[2][4], int& par, int (&eo)[4], Guarda&& guarda, Entre&& entre) {
    const int x = threadIdx.x, n = T / 32;
    par = x >= T;
    const int t = x - par * T;
    int e[2], w[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int f = par + 2 * k;
        const int8_t *m = DO && f == 3 ? gom : qm, *E = DO && f == 3 ? goE : qE;
        const int ld = DO && f == 3 ? D : 3 * D, col = (f == 3 ? 0 : f * D) + h * 4;
        e[k] = SEM_TOPO;
        w[k] = 0;
        if (DO || f < 3) {
            e[k] = (int)E[(size_t)(b0 + t) * (ld / blk) + col / blk];
            w[k] = *reinterpret_cast<const int*>(m + (size_t)(b0 + t) * ld + col);
        }
    }
    entre();
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int mx = g_max<32>(e[k]);
        if ((x & 31) == 0)
            for (int c = t >> 5; c < 8; c += n) red[par + 2 * k][c] = mx;
    }
    __syncthreads();
    int emx[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        emx[s] = max(max(max(red[s][0], red[s][1]), max(red[s][2], red[s][3])), max(max(red[s][4], red[s][5]), max(red[s][6], red[s][7])));
        eo[s] = emx[s] - GA;
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int f = par + 2 * k, r = par ? emx[1 + 2 * k] : emx[2 * k];
        h4_t v;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            a[k][d] = rnd_d(((w[k] << (24 - 8 * d)) >> 24) << GA, r - e[k]);
            v[d] = (_Float16)a[k][d];
        }
        if (DO || f < 3) guarda(f, t, v);
    }
}

template <int TMAX>
__global__ void __launch_bounds__(2 * TMAX) k_atencao4m(const int8_t* __restrict__ qm, const int8_t* __restrict__ qE, int* __restrict__ Oacc,
                                                        int16_t* __restrict__ Oe, uint8_t* __restrict__ P, int T, int H, int D, int blk,
                                                        int GA, int kid) {
    constexpr int NT = TMAX / 16;
    extern __shared__ __align__(16) char sm4[];
    __shared__ __align__(16) int red[4][8];
    const int PL = T + at4::PAD;
    auto texp = reinterpret_cast<unsigned short*>(sm4);
    auto pt = reinterpret_cast<uint8_t*>(sm4 + EXP_N * 2);           // P of the head, transposed ([j][i])
    auto qd = reinterpret_cast<h4_t*>(pt + (size_t)T * PL), kd = qd + T;
    auto vt = reinterpret_cast<_Float16*>(kd + T);
    const int bh = at4::cabeca(blockIdx.x, gridDim.x), b = bh / H, h = bh % H, b0 = b * T;
    int eo[4], al[2][4], par;
    alinha4f<false>(nullptr, nullptr, qm, qE, D, h, blk, b0, T, GA, red, al, par, eo,
                    [&](int f, int t, const h4_t& v) {
                        if (f < 2) qd[f * T + t] = v;                // q, then k
                        else
#pragma unroll
                            for (int d = 0; d < 4; d++) vt[d * PL + t] = v[d];
                    },
                    [&] { exp_tab_lds(texp); });
    const int eq = eo[0], ek = eo[1], ev = eo[2];
    __syncthreads();
    const int su = __builtin_amdgcn_readfirstlane(-(eq + ek - 1 + 8)), incl_ = 8 - h / 8;   // one per head
    const int nt = T / 16;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint8_t* Pb = P + (size_t)bh * T * T;
#pragma unroll 1
    for (int k = 0; k < 2; k++) {                                    // a short and a long stripe: nt + 1 tiles a wave
        const int st = k ? nt - 1 - wv : wv;
        // opaque per turn: what depends on them stays in it (kept across both, it takes 110 more registers)
        int lane = threadIdx.x & 63, incl = incl_;
        asm volatile("" : "+v"(lane), "+s"(incl));
        const int lr = lane & 15, lg = lane >> 4;
        const int i = 16 * st + lr, row = b0 + i;
        const long long idx = (long long)row * D + h * 4;
        const h4_t q4 = qd[i], qf = lg == 0 ? q4 : h4_t{};
        int u[NT][4], mx = U_MIN;
        if (su >= 3) {
            const float rs = __int_as_float((127 - min(su, 126)) << 23);  // 2^-su (below 2^-24 |s| any scale rounds to 0)
            const float c0 = at4::MG - (float)((i - 4 * lg) * (1 << incl)), pa = (float)(1 << incl);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if (t > st) continue;
                const f4_t s = __builtin_amdgcn_mfma_f32_16x16x16f16(kd[16 * t + lr], qf, f4_t{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    u[t][v] = __float_as_int(__builtin_fmaf(s[v], rs, c0 + (float)(16 * t + v) * pa));
                    if (t == st) u[t][v] = 4 * lg + v <= lr ? u[t][v] : U_MIN;
                    mx = max(mx, u[t][v]);
                }
            }
        } else {                                                          // small and left shifts (checked), causal pairs only
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if (t > st) continue;
                f4_t s = __builtin_amdgcn_mfma_f32_16x16x16f16(kd[16 * t + lr], qf, f4_t{0, 0, 0, 0}, 0, 0, 0);
                at4::pronto(s);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int j = 16 * t + 4 * lg + v;
                    u[t][v] = U_MIN;
                    if (j <= i) u[t][v] = rnd((int)s[v], su, kid, idx) - ((i - j) << incl);
                    mx = max(mx, u[t][v]);
                }
            }
        }
        mx = at4::max_lg(mx);
        int soma = 0;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (t > st) continue;
#pragma unroll
            for (int v = 0; v < 4; v++) { u[t][v] = exp_tab(texp, mx, u[t][v]); soma += u[t][v]; }   // a masked pair reads 0
        }
        soma = at4::soma_lg(soma);
        if (soma <= 0) {
            if (lg == 0) reporta(E_DIV, kid, idx, soma, mx);
            soma = 1;
        }
        // a row's sum is at least 4095 (its maximum contributes exp(0) >> 3), so 2^28 / sum < 2^20: div_exata's bound
        const int inv = soma > 256 ? div_exata(1 << 28, soma) : (1 << 28) / soma;
        f4_t o = {0, 0, 0, 0};                                           // O^T: row v = dimension v (the same for every lg)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (t > st) {                                                // above the diagonal: zeros
                if (t < nt) *reinterpret_cast<int*>(pt + (size_t)(16 * t + (lane >> 2)) * PL + 16 * st + 4 * (lane & 3)) = 0;
                continue;
            }
            h4_t p4;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int p = min((mul24(u[t][v], inv) + (1 << 19)) >> 20, 255);
                pt[(size_t)(16 * t + 4 * lg + v) * PL + i] = (uint8_t)p;
                p4[v] = (_Float16)(unsigned short)p;
            }
            o = __builtin_amdgcn_mfma_f32_16x16x16f16(*reinterpret_cast<const h4_t*>(vt + (lr & 3) * PL + 16 * t + 4 * lg), p4, o, 0, 0, 0);
        }
        at4::pronto(o);
        if (lg == 0) {
            const size_t x = (size_t)row * D + h * 4;
            int ov[4];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                ov[d] = (int)o[d];
                if (ov[d] >= LIM || ov[d] <= -LIM) reporta(E_ACUM, kid, x + d, ov[d], -3);
            }
            const int16_t e = (int16_t)(ev - 8);
            *reinterpret_cast<int4*>(Oacc + x) = make_int4(ov[0], ov[1], ov[2], ov[3]);
            *reinterpret_cast<short4*>(Oe + x) = make_short4(e, e, e, e);
        }
    }
    // the head's P, transposed in LDS, goes out as 16-byte pieces of whole rows: byte stores scattered over rows T
    // apart cost three times as much
    __syncthreads();
    for (int c = threadIdx.x; c < T * nt; c += blockDim.x) {
        const int r = c / nt, col = (c - r * nt) * 16;
        *reinterpret_cast<int4*>(Pb + (size_t)r * T + col) = *reinterpret_cast<const int4*>(pt + (size_t)r * PL + col);
    }
}

template <int TMAX, int LIMITE>
__global__ void __launch_bounds__(2 * TMAX) k_atencao4m_back(const int8_t* __restrict__ gom, const int8_t* __restrict__ goE,
                                                             const int8_t* __restrict__ qm, const int8_t* __restrict__ qE,
                                                             const uint8_t* __restrict__ P, int* __restrict__ Gacc, int16_t* __restrict__ Ge,
                                                             int T, int H, int D, int blk, int GA, int DSB, int kid) {
    constexpr int NT = TMAX / 16, LB = TMAX <= 128 ? 7 : 6;
    extern __shared__ __align__(16) char sm4[];
    __shared__ __align__(16) int red4[4][8];
    __shared__ __align__(16) int red[3][8];
    const int PL = T + at4::PAD, nt = T / 16, nw = nt / 2, ntri = nt * (nt + 1) / 2;
    auto dsm = reinterpret_cast<s2_t (*)[64][2]>(sm4);               // dS of tile st (st + 1) / 2 + t, per lane
    auto pm_ = reinterpret_cast<unsigned (*)[64]>(sm4 + (size_t)ntri * 512);
    auto gd = reinterpret_cast<h4_t*>(sm4 + (size_t)ntri * 768), vd = gd + T;
    auto kt = reinterpret_cast<_Float16*>(vd + T), qt = kt + 4 * PL, gt = qt + 4 * PL;
    const int bh = at4::cabeca(blockIdx.x, gridDim.x), b = bh / H, h = bh % H, ld = 3 * D, b0 = b * T;
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // this wave's rows: stripes wv and nt - 1 - wv, a short and a long one. Slot n <= wv: tile n of the short stripe, n = wv
    // its diagonal one; slot n > wv: tile n - wv - 1 of the long one, up to n = nt
    const int st2[2] = {wv, nt - 1 - wv};
    const uint8_t* Pb = P + (size_t)bh * T * T;
    unsigned pr[NT + 1];
    int eo[4], al[2][4], par;
    alinha4f<true>(gom, goE, qm, qE, D, h, blk, b0, T, GA, red4, al, par, eo,
                   [&](int f, int t, const h4_t& v) {
                       if (f >= 2) gd[(3 - f) * T + t] = v;          // dO, then v
                       if (f != 2)
#pragma unroll
                           for (int d = 0; d < 4; d++) (f == 0 ? qt : f == 1 ? kt : gt)[d * PL + t] = v[d];
                   },
                   [&] {
#pragma unroll
                       for (int n = 0; n <= NT; n++) {               // past the last slot: its tile again, unused
                           const int c = min(n, nt), k = c > wv, t = k ? c - wv - 1 : c;
                           pr[n] = *reinterpret_cast<const unsigned*>(Pb + (size_t)(16 * t + lr) * T + 16 * st2[k] + 4 * lg);
                       }
                   });
    const int eq = eo[0], ek = eo[1], ev = eo[2], ego = eo[3];
    __syncthreads();
    // f(n, the long stripe?, its values, its P) for every slot, and fim(k) after the last tile of stripe k
    int x[NT + 1][4];
    auto tiles = [&](auto f, auto fim) {
#pragma unroll
        for (int n = 0; n <= NT; n++) {
            if (n > nt) continue;
            f(n, n > wv, x[n], pr[n]);
            if (n == wv) fim(0);
        }
        fim(1);
    };
    // gP (float bits); the diagonal tiles' pairs past the diagonal get gP = P = 0
    h4_t gf[2];
#pragma unroll
    for (int k = 0; k < 2; k++) { const h4_t g4 = gd[16 * st2[k] + lr]; gf[k] = lg == 0 ? g4 : h4_t{}; }
    const int z = min(max(lr - 4 * lg, 0), 4);                       // rows before key lr of a diagonal tile
    const unsigned causal = z == 4 ? 0u : ~0u << (8 * z);
    float mgf = 0;
#pragma unroll
    for (int n = 0; n <= NT; n++) {
        if (n > nt) continue;
        const bool longa = n > wv, diag = n == wv || n == nt;
        const f4_t g = __builtin_amdgcn_mfma_f32_16x16x16f16(longa ? gf[1] : gf[0], vd[16 * (longa ? n - wv - 1 : n) + lr], f4_t{0, 0, 0, 0}, 0, 0, 0);
        const int zt = diag ? z : 0;
        pr[n] &= diag ? causal : ~0u;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float y = v < zt ? 0.0f : g[v];
            if constexpr (!LIMITE) mgf = fmaxf(mgf, fabsf(y));
            x[n][v] = __float_as_int(y);
        }
    }
    // shift of gP: exact causal maximum, or max_i ||dO_i||_inf * max_j ||v_j||_1
    int mg;
    if constexpr (LIMITE) {
        const int b1 = par ? max(max(abs(al[1][0]), abs(al[1][1])), max(abs(al[1][2]), abs(al[1][3]))) : 0;
        const int b2 = par ? 0 : abs(al[1][0]) + abs(al[1][1]) + abs(al[1][2]) + abs(al[1][3]);
        mg = at4::grupo_max(b1, red[0], nw) * at4::grupo_max(b2, red[1], nw);
    } else mg = at4::grupo_max((int)mgf, red[0], nw);
    const int sh = max(bitlen(mg) - 15, 0), egp = ego + ev + sh;
    // gP' = rnd(gP, sh): |gP| 2^-sh <= 2^15, so 1.5 2^23 + gP 2^-sh rounds to gP' in its low bits
    const float rs = __int_as_float((127 - sh) << 23);
    int s[4] = {0, 0, 0, 0}, sl[2][4], pm = 0, gm = 0, smx = 0;
    tiles([&](int, bool, int (&y)[4], unsigned p4) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            y[v] = __float_as_int(__builtin_fmaf(__int_as_float(y[v]), rs, at4::MG)) - at4::MGB;
            const int p = (p4 >> (8 * v)) & 255;
            s[v] += mul24(p, y[v]);
            if constexpr (LIMITE) { pm = max(pm, p); gm = max(gm, abs(y[v])); }
        }
    }, [&](int k) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int t = g_sum<16>(s[v]);
            if (lr == 0 && (t >= LIM || t <= -LIM)) reporta(E_ACUM, kid, (long long)(b0 + 16 * st2[k] + 4 * lg + v) * ld + h * 4, t, -4);
            sl[k][v] = rnd_d(t, 8);
            smx = max(smx, abs(sl[k][v]));
            s[v] = 0;
        }
    });
    // dS before its shrink; its shift from max |P (gP' - s)|, or max P * (max |gP'| + max |s|)
    int md = 0, mn = 0;
    tiles([&](int, bool k, int (&y)[4], unsigned p4) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            y[v] = mul24((int)((p4 >> (8 * v)) & 255), y[v] - (k ? sl[1][v] : sl[0][v]));
            if constexpr (!LIMITE) { md = max(md, y[v]); mn = min(mn, y[v]); }
        }
    }, [](int) {});
    if constexpr (LIMITE) {
        const int a = at4::grupo_max(pm, red[2], nw), c = at4::grupo_max(gm, red[0], nw);
        md = a * (c + at4::grupo_max(smx, red[1], nw));
    } else md = at4::grupo_max(max(md, -mn), red[1], nw);
    const int sh2 = max(bitlen(md) - DSB, 0), eds = egp - 9 + sh2;
    // rnd(d, sh2) in integers: floor((d + 2^(sh2 - 1) - 1 + bit sh2 of d) 2^-sh2) (d may pass 2^24)
    const int meio = sh2 ? (1 << (sh2 - 1)) - 1 : 0;
    const unsigned um = sh2 ? 1u : 0u;
    h4_t ident;
#pragma unroll
    for (int v = 0; v < 4; v++) ident[v] = (_Float16)(4 * lg + v == lr ? 1.0f : 0.0f);
    auto grava4 = [&](const int (&r)[4], int tok, int col, int e) {
        const size_t o = (size_t)(b0 + tok) * ld + col + h * 4;
#pragma unroll
        for (int d = 0; d < 4; d++)
            if (r[d] >= LIM || r[d] <= -LIM) reporta(E_ACUM, kid, o + d, r[d], -5);
        const int16_t ee = (int16_t)e;
        *reinterpret_cast<int4*>(Gacc + o) = make_int4(r[0], r[1], r[2], r[3]);
        *reinterpret_cast<short4*>(Ge + o) = make_short4(ee, ee, ee, ee);
    };
    auto junta = [](float a, float c) { return (int)((unsigned)(int)a * (1u << LB) + (unsigned)(int)c); };
    f4_t qa = {0, 0, 0, 0}, qb = {0, 0, 0, 0};
    tiles([&](int n, bool k, int (&y)[4], unsigned p4) {
        const int st = k ? st2[1] : st2[0], t = k ? n - wv - 1 : n, m = st * (st + 1) / 2 + t;
        int d[4];
#pragma unroll
        for (int v = 0; v < 4; v++) d[v] = (y[v] + meio + (int)__builtin_amdgcn_ubfe((unsigned)y[v], sh2, um)) >> sh2;
        const s2_t ds[2] = {s2_t{(short)d[0], (short)d[1]}, s2_t{(short)d[2], (short)d[3]}};
        dsm[m][lane][0] = ds[0];
        dsm[m][lane][1] = ds[1];
        pm_[m][lane] = p4;
        h4_t a, c;
        at4::pedacos<LB>(ds, a, c);
        const f4_t ta = __builtin_amdgcn_mfma_f32_16x16x16f16(a, ident, f4_t{0, 0, 0, 0}, 0, 0, 0);   // rows: keys
        const f4_t tc = __builtin_amdgcn_mfma_f32_16x16x16f16(c, ident, f4_t{0, 0, 0, 0}, 0, 0, 0);
        const h4_t k4 = *reinterpret_cast<const h4_t*>(kt + (lr & 3) * PL + 16 * t + 4 * lg);
        qa = __builtin_amdgcn_mfma_f32_16x16x16f16(k4, at4::para_f16(ta), qa, 0, 0, 0);
        qb = __builtin_amdgcn_mfma_f32_16x16x16f16(k4, at4::para_f16(tc), qb, 0, 0, 0);
    }, [&](int k) {
        at4::pronto(qa);
        at4::pronto(qb);
        if (lg == 0) {
            const int r[4] = {junta(qa[0], qb[0]), junta(qa[1], qb[1]), junta(qa[2], qb[2]), junta(qa[3], qb[3])};
            grava4(r, 16 * st2[k] + lr, 0, eds + ek);
        }
        qa = f4_t{0, 0, 0, 0};
        qb = f4_t{0, 0, 0, 0};
    });
    __syncthreads();                                                 // every dS and P tile of the head in LDS
    // columns: this wave takes key tiles wv and nt - 1 - wv, tile c with the stripes c .. nt - 1
#pragma unroll 1
    for (int k = 0; k < 2; k++) {
        const int c = k ? st2[1] : st2[0];
        f4_t ka = {0, 0, 0, 0}, kb = {0, 0, 0, 0}, va = {0, 0, 0, 0};
        int gv[4] = {0, 0, 0, 0};
        for (int r = c, n = 1; r < nt; r++, n++) {
            const int m = r * (r + 1) / 2 + c;
            const s2_t ds[2] = {dsm[m][lane][0], dsm[m][lane][1]};
            h4_t a, x4;
            at4::pedacos<LB>(ds, a, x4);
            const h4_t q4 = *reinterpret_cast<const h4_t*>(qt + (lr & 3) * PL + 16 * r + 4 * lg);
            const h4_t o4 = *reinterpret_cast<const h4_t*>(gt + (lr & 3) * PL + 16 * r + 4 * lg);
            ka = __builtin_amdgcn_mfma_f32_16x16x16f16(q4, a, ka, 0, 0, 0);
            kb = __builtin_amdgcn_mfma_f32_16x16x16f16(q4, x4, kb, 0, 0, 0);
            va = __builtin_amdgcn_mfma_f32_16x16x16f16(o4, at4::bytes_f16(pm_[m][lane]), va, 0, 0, 0);
            if (!(n & 1)) {                                              // two tiles' sum, exact, to int32
#pragma unroll
                for (int v = 0; v < 4; v++) gv[v] += (int)va[v];
                va = f4_t{0, 0, 0, 0};
            }
        }
        at4::pronto(ka);
        at4::pronto(kb);
        at4::pronto(va);
        if (lg == 0) {
            const int r[4] = {junta(ka[0], kb[0]), junta(ka[1], kb[1]), junta(ka[2], kb[2]), junta(ka[3], kb[3])};
            grava4(r, 16 * c + lr, D, eds + eq);
        } else if (lg == 1) {
            const int r[4] = {gv[0] + (int)va[0], gv[1] + (int)va[1], gv[2] + (int)va[2], gv[3] + (int)va[3]};
            grava4(r, 16 * c + lr, 2 * D, ego - 8);
        }
    }
}
