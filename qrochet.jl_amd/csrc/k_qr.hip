// Batched blocked Householder QR (complex FP64), used to precondition the
// one-sided Jacobi SVD:  X = Q1 R1,  R_{j-1}^H = Q_j R_j,  Jacobi on R_n^H (three
// passes by default).  The triangular factors grade the columns so that the
// Jacobi sweeps converge in fewer sweeps (the preconditioning of Drmac & Veselic,
// "New fast and accurate Jacobi SVD algorithm", SIAM J. Matrix Anal. Appl. 29
// (2008); on the matrices of a TEBD layer, 512 x 512, two passes take the rounds
// from ~1600 to ~900 per three layers and a third pass to ~775).
//
// Panels of QR_NB columns: one workgroup factors a panel (LAPACK zlarfg
// reflectors, H^H x = beta e1 with H = I - tau v v^H, real beta) and builds the
// compact-WY triangle T (Q_panel = I - V T V^H); Q_panel^H (factorisation) or Q_panel
// (forming Q·M) is applied to tiles of 16 columns.  Up to 1024 rows panels and tiles live in
// registers (k_qr_panel, k_qr_step, k_qr_form), taller ones go by column groups
// (k_qr_panel_tall, up to 4096 rows) or through memory (k_qr_panel_mem, k_qr_apply,
// k_qr_form_tall).
#include "qh_kernels.h"
#include "qh_complex.h"

namespace qh {

constexpr int QR_TC = 16;  // target columns per apply workgroup
typedef double qr_f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double2 shfl_xor2(double2 a, int off) {
    return make_double2(__shfl_xor(a.x, off, 64), __shfl_xor(a.y, off, 64));
}
// DPP moves of a double within 16-lane rows (register to register, no LDS round trip)
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
    // (mov_dpp: no old value to set first -- every lane has a source)
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
constexpr int DPP_XOR1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int DPP_ROW_BCAST = 0x150;  // + n: lane n of the row to the whole row
template <int C>
__device__ __forceinline__ double2 row_bcast(double2 a) {
    return make_double2(dpp_d<DPP_ROW_BCAST + C>(a.x), dpp_d<DPP_ROW_BCAST + C>(a.y));
}

// the value of lane `src` (the same lane for the whole wave) in every lane
__device__ __forceinline__ double bcast_d(double x, int src) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), src);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), src);
    return __hiloint2double(hi, lo);
}

// Cross-lane swaps of gfx950 (per dword of a double): permlane32 trades lanes 32..63
// of a with lanes 0..31 of b, permlane16 trades the odd 16-lane rows of a (lanes
// 16..31, 48..63) with the even rows of b (lanes 0..15, 32..47).  Afterwards a + b
// holds, in every lane, its own value plus the partner's (lane ^ 32, resp. ^ 16) of the
// half that the lane keeps: a's for the lower lanes, b's for the upper ones.
__device__ __forceinline__ void swap_lanes32(double& a, double& b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b),
                                                     false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b),
                                                     false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ void swap_lanes16(double& a, double& b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b),
                                                     false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b),
                                                     false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}
// halving step of block_sum16 with a lane swap: slot i (lower lanes) or i + half
// (upper lanes), summed over the lane and its partner, lands in v[i]
template <int OFF>
__device__ __forceinline__ double2 halve_swap(double2 lo, double2 hi) {
    if constexpr (OFF == 32) {
        swap_lanes32(lo.x, hi.x);
        swap_lanes32(lo.y, hi.y);
    } else {
        swap_lanes16(lo.x, hi.x);
        swap_lanes16(lo.y, hi.y);
    }
    return cadd(lo, hi);
}

// the sum over the four 16-lane rows of a wave, in every lane
__device__ __forceinline__ double2 sum_rows16(double2 a) {
    double2 b = a;
    swap_lanes32(a.x, b.x);
    swap_lanes32(a.y, b.y);
    a = b = cadd(a, b);
    swap_lanes16(a.x, b.x);
    swap_lanes16(a.y, b.y);
    return cadd(a, b);
}
constexpr int DPP_ROW_ROR = 0x120;  // + n: rotated by n lanes within the 16-lane row
template <int N>
__device__ __forceinline__ double2 row_ror(double2 a) {
    return make_double2(dpp_d<DPP_ROW_ROR + N>(a.x), dpp_d<DPP_ROW_ROR + N>(a.y));
}

// LDS written by one wave and read back by the same wave: the fences order the
// accesses across the wave's lanes, and no workgroup barrier is needed
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum over the workgroup (NW waves) of 16 complex values per thread, with one barrier.
// Each wave halves its values recursively: at the step with offset o a lane keeps the
// upper or the lower half (by lane bit o) and adds the partner's copy of that half (lane
// swaps for o = 32, 16; shuffles for o = 8, 4), so 16 values take 15 exchanges; lane l
// then holds value (l >> 2) & 15 summed over the
// lanes that agree with l in bits 0-1, which two plain steps add.  The wave's 16 sums go
// to sRed; after the barrier every lane adds the NW partials of value l & 15 in wave
// order, so all waves hold the same totals, value k in lanes k, k + 16, k + 32, k + 48.
// sRed is read after the barrier, so consecutive calls alternate two buffers: a fast
// wave's next writes then cannot overtake a slow wave's reads.
template <int NW>
__device__ __forceinline__ double2 block_sum16(double2 (&v)[16], double2* sRed /* NW*16 */) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double2 h8[8], h4[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) h8[i] = halve_swap<32>(v[i], v[i + 8]);
#pragma unroll
    for (int i = 0; i < 4; ++i) h4[i] = halve_swap<16>(h8[i], h8[i + 4]);
    double2 h2[2];
    {
        const bool up = (lane & 8) != 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const double2 send = up ? h4[i] : h4[i + 2];
            const double2 keep = up ? h4[i + 2] : h4[i];
            h2[i] = cadd(keep, shfl_xor2(send, 8));
        }
    }
    double2 s;
    {
        const bool up = (lane & 4) != 0;
        const double2 send = up ? h2[0] : h2[1];
        const double2 keep = up ? h2[1] : h2[0];
        s = cadd(keep, shfl_xor2(send, 4));
    }
    s = cadd(s, shfl_xor2(s, 2));
    s = cadd(s, shfl_xor2(s, 1));
    if ((lane & 3) == 0) sRed[wv * 16 + ((lane >> 2) & 15)] = s;
    __syncthreads();
    double2 t = sRed[lane & 15];
#pragma unroll
    for (int w = 1; w < NW; ++w) t = cadd(t, sRed[w * 16 + (lane & 15)]);
    return t;
}

// LAPACK zlarfg: H^H (alpha; x) = (beta; 0), H = I - tau v v^H, v = (1; x·scale), beta real
struct Reflector {
    double2 tau, scale;
    double beta, rbeta;  // (rbeta: 1 / beta, 0 where there is nothing to reflect)
};
__device__ __forceinline__ Reflector make_reflector(double2 alpha, double xnorm2) {
    Reflector h;
    h.tau = cz();
    h.scale = cz();
    h.beta = alpha.x;
    h.rbeta = 0.0;
    if (!(xnorm2 == 0.0 && alpha.y == 0.0)) {
        // (every column of a panel waits for these: refined reciprocals take half the
        // instructions of a square root and two divisions, and round as well: the same bits
        // in five workloads; mixed canonical form at chi = 200 8.04 -> 7.92 ms.  The limits keep
        // squares and estimates in range)
        const double n2 = cabs2(alpha) + xnorm2;
        double nrm, rn, rd;
        if (n2 > 1e-280 && n2 < 1e280) {
            const double r = rsqrt_refined(n2), n = n2 * r;
            nrm = fma(0.5 * r, fma(-n, n, n2), n);
            rn = fma(r, fma(-nrm, r, 1.0), r);
            const double m = fabs(alpha.x) + nrm;
            rd = rcp_refined(fma(m, m, alpha.y * alpha.y));
        } else {
            nrm = sqrt(n2);
            rn = 1.0 / nrm;
            const double m = fabs(alpha.x) + nrm;
            rd = 1.0 / fma(m, m, alpha.y * alpha.y);
        }
        const bool neg = alpha.x >= 0.0;
        h.beta = neg ? -nrm : nrm;
        h.rbeta = neg ? -rn : rn;
        h.tau = make_double2((h.beta - alpha.x) * h.rbeta, -alpha.y * h.rbeta);
        h.scale = make_double2((alpha.x - h.beta) * rd, -alpha.y * rd);  // 1 / (alpha - beta)
    }
    return h;
}

// The column step of a panel (column c, rows relative to the panel corner): one
// workgroup sum gives, over the rows below the diagonal with x = column c there,
// s_c = ||x||^2, s_k = x^H a_k (k > c) and s_k = v_k^H x (k < c); row c (alpha = a_c(c),
// a_k(c), v_k(c)) is published by its owner before that sum's barrier.  With the
// reflector v = (1; x·scale) the dots follow without a second sum:
// v^H a_k = a_k(c) + conj(scale)·s_k and v_k^H v = conj(v_k(c)) + scale·s_k.
struct PanelShared {
    double2 sRed[2][8 * QR_NB];  // wave partial sums (up to 8 waves), two alternating buffers
    double2 sRow[2][QR_NB];      // row c of the panel, two alternating buffers
    double2 sBc[8][QR_NB];       // per wave: the 16 dots, written by lanes 0..15 and read by all
    double2 sT[QR_NB][QR_NB + 1];
};

// the coefficient of slot k (held by lane k of every wave) for every lane: lanes 0..15 write
// the wave's own LDS row, which the wave then reads where it uses a dot (the next
// column's writes follow these reads in the wave's program order, after a barrier)
__device__ __forceinline__ const double2* panel_dots_publish(double2 dl, PanelShared& sh) {
    double2* bc = sh.sBc[threadIdx.x >> 6];
    if ((threadIdx.x & 63) < QR_NB) bc[threadIdx.x & 63] = dl;
    wave_lds_sync();
    return bc;
}

// slot k's coefficient from the unscaled sum `tot` and row c's entry `row`: for k > c
// the trailing update's conj(tau) v^H a_k, for k < c the dot v_k^H v that builds T,
// 0 for k = c
__device__ __forceinline__ double2 panel_coef(int k, int c, double2 tot, double2 row, const Reflector& h) {
    if (k > c) return cmul(cconj(h.tau), cadd(row, cmul(cconj(h.scale), tot)));
    if (k < c) return cadd(cconj(row), cmul(h.scale, tot));
    return cz();
}

// Column loop of a panel factorisation on a panel view P(c, r) (column c, row r
// relative to the panel corner) in global memory, NT threads.  Leaves R on and
// above the diagonal, the scaled reflectors below it, and the compact-WY triangle
// in sh.sT.  Thread tid owns rows r = tid + NT j for the whole panel, so the sums,
// the reflector's scaling and the trailing update touch only the thread's own rows;
// the only cross-thread data are the one sum per column and row c (PanelShared).
template <int NT, class Ref>
__device__ void qr_panel_columns(int rows, int nb, PanelShared& sh, Ref P) {
    constexpr int NW = NT / 64;
    const int tid = threadIdx.x;
    for (int c = 0; c < nb; ++c) {
        double2 sk[QR_NB];
#pragma unroll
        for (int k = 0; k < QR_NB; ++k) sk[k] = cz();
        for (int r = tid; r < rows; r += NT) {
            if (r <= c) continue;
            const double2 x = P(c, r);
            // all 16 loads issue before their first use (column min(k, nb - 1) is always
            // inside the panel; the values of k >= nb are discarded)
            double2 pk[QR_NB];
#pragma unroll
            for (int k = 0; k < QR_NB; ++k) pk[k] = P(min(k, nb - 1), r);
#pragma unroll
            for (int k = 0; k < QR_NB; ++k) {
                if (k < c) sk[k] = cfmac(pk[k], x, sk[k]);
                else if (k == c) sk[k].x += cabs2(x);
                else if (k < nb) sk[k] = cfmac(x, pk[k], sk[k]);
            }
        }
        if (tid == c) {
#pragma unroll
            for (int k = 0; k < QR_NB; ++k) sh.sRow[c & 1][k] = (k < nb && c < rows) ? P(k, c) : cz();
        }
        const double2 tot = block_sum16<NW>(sk, sh.sRed[c & 1]);
        const Reflector h = make_reflector(sh.sRow[c & 1][c], bcast_d(tot.x, c));
        const double2 dl = panel_coef(tid & 15, c, tot, sh.sRow[c & 1][tid & 15], h);
        const double2* dk = panel_dots_publish(dl, sh);
        if (tid == c && c < rows) P(c, c) = make_double2(h.beta, 0.0);
        if (tid < QR_NB) {
            const int i = tid;
            double2 val = cz();
            if (i < c) {
                double2 acc = cz();
#pragma unroll
                for (int l = 0; l < QR_NB; ++l)
                    if (l >= i && l < c) acc = cfma(sh.sT[i][l], dk[l], acc);
                const double2 tc = h.tau;
                val = make_double2(-(tc.x * acc.x - tc.y * acc.y), -(tc.x * acc.y + tc.y * acc.x));
            } else if (i == c) {
                val = h.tau;
            }
            sh.sT[i][c] = val;
        }
        // v below the diagonal (scaled in place) and the trailing update
        // a_k -= conj(tau) (v^H a_k) v on own rows
        double2 w[QR_NB];
#pragma unroll
        for (int k = 0; k < QR_NB; ++k) w[k] = (k > c && k < nb) ? dk[k] : cz();
        for (int r = tid; r < rows; r += NT) {
            if (r < c) continue;
            double2 vr = make_double2(1.0, 0.0);
            if (r > c) {
                vr = cmul(P(c, r), h.scale);
                P(c, r) = vr;
            }
            double2 pk[QR_NB];
#pragma unroll
            for (int k = 0; k < QR_NB; ++k) pk[k] = P(min(k, nb - 1), r);
#pragma unroll
            for (int k = 0; k < QR_NB; ++k)
                if (k > c && k < nb) P(k, r) = cfms(w[k], vr, pk[k]);
        }
    }
    __syncthreads();
}

// panel factorisation in place in global memory (any number of rows; the panel's
// 16 columns stay in L2 across the column loop)
template <int NT>
__device__ void qr_panel_global(const QrItem& it, int j0, PanelShared& sh) {
    const int tid = threadIdx.x;
    const int rows = it.m - j0;
    const int nb = min(QR_NB, it.n - j0);
    double2* base = it.a + j0 + (size_t)it.lda * j0;
    const size_t lda = it.lda;
    qr_panel_columns<NT>(rows, nb, sh, [&](int c, int r) -> double2& { return base[r + lda * c]; });
    __syncthreads();
    // explicit reflectors to v, zeros below the diagonal of R
    for (int e = tid; e < nb * rows; e += NT) {
        const int c = e / rows, r = e % rows;
        const size_t vi = (j0 + r) + (size_t)it.m * (j0 + c);
        double2& ar = base[r + lda * c];
        if (r < c) {
            it.v[vi] = cz();
        } else if (r == c) {
            it.v[vi] = make_double2(1.0, 0.0);
        } else {
            it.v[vi] = ar;
            ar = cz();
        }
    }
    double2* t = it.t + (size_t)(j0 / QR_NB) * QR_NB * QR_NB;
    for (int e = tid; e < QR_NB * QR_NB; e += NT) {
        const int i = e % QR_NB, j = e / QR_NB;
        t[i + QR_NB * j] = (i < nb && j < nb) ? sh.sT[i][j] : cz();
    }
}

// ---------------------------------------------------------------------------
// A column tile in registers (panels and tiles of up to 1024 rows)
// ---------------------------------------------------------------------------
// Sixteen columns of a matrix, in the operand layout of the matrix cores: the rows below
// r0 in blocks of 16, block b with wave b mod nw (its t = b / nw -th block); lane l holds
// column l % 16 and of each block the rows 4 q + l / 16, q < 4, in Y[t][q].  That is at once
// the B operand of a 16 × 16 × 4 step (rows as the contracted index), its result, and the A
// operand of a 4 × 4 × 4 step (columns as rows of A): a block reflector is applied and the
// panel factored without moving the tile, and the next panel's columns go from the one to
// the other without a trip through memory.
constexpr int QR_TILE_NT = 512;
struct TileShared {
    double2 part[8][QR_NB][QR_TC];   // per wave: its part of V^H Y
    double2 w[QR_NB][QR_TC + 1];
    double2 red[2][8][QR_NB];        // per wave: its part of a column's sums, two alternating buffers
    double2 row[QR_NB][QR_NB];       // row c of the panel as column c met it
    double2 tot[QR_NB][QR_NB];       // x^H a_k of column c
    double2 tau[QR_NB], scale[QR_NB];
    double2 dot[QR_NB][QR_NB + 1];   // v_i^H v_j, i < j
    double2 t[QR_NB][QR_NB + 1];
    double2 x[64];
};
// waves that factor a panel of nblk row blocks: a wave alone on its SIMD issues a vector
// instruction every 8 to 12 cycles, so two of them share the rows from the fifth block on
// (step of 256 rows: 30.5 us on eight waves, 33 on four; up to 64 rows four waves have a
// block each, and a sum over eight would only wait longer)
__device__ __forceinline__ int panel_waves(int nblk) { return nblk <= 4 ? 4 : 8; }

template <int NB>
__device__ __forceinline__ void tile_load(double2 (&Y)[NB][4], const double2* y, size_t ldy, int rows, int tc, int nw,
                                          int wv) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int b = wv + nw * t;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * b + 4 * q + lk;
            Y[t][q] = ld_or_zero(y, r + ldy * li, r < rows && li < tc);
        }
    }
}
// columns c0 .. of a unit matrix
template <int NB>
__device__ __forceinline__ void tile_unit(double2 (&Y)[NB][4], int c0, int tc, int nw, int wv) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            Y[t][q] = make_double2(li < tc && 16 * (wv + nw * t) + 4 * q + lk == c0 + li ? 1.0 : 0.0, 0.0);
}
template <int NB>
__device__ __forceinline__ void tile_store(const double2 (&Y)[NB][4], double2* y, size_t ldy, int rows, int tc, int nw,
                                           int wv) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int b = wv + nw * t;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * b + 4 * q + lk;
            if (r < rows && li < tc) gstore(y, r + ldy * li, Y[t][q]);
        }
    }
}

// Y <- (I - V T' V^H) Y for the tile's blocks b0 <= b, T' = T^H (adjoint) or T; v: the
// panel's reflectors from the tile's first row (ld ldv, nb of them, rows rows), all zero
// above block b0.  Three real products per complex one:
//   W = V^H Y: A[i][k] = V(row k, reflector i), B = Y's registers; the waves' parts meet in
//     LDS (one entry per thread adds them in wave order);
//   W2 = T' W: 16 × 16 × 16 by every wave for itself, so that its result registers are the
//     B operand of
//   Y -= V W2: A[i][k] = V(row i, reflector k).
template <int NB>
__device__ __forceinline__ void tile_apply(double2 (&Y)[NB][4], const double2* v, size_t ldv, int rows, int nb,
                                           const double2* tpan, int adjoint, int b0, int nw, int wv, TileShared& sh) {
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    double2 tv[4];  // T'(li, 4 k + lk)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int kk = 4 * k + lk;
        const double2 x = gload(tpan, adjoint ? kk + QR_NB * li : li + QR_NB * kk);
        tv[k] = adjoint ? cconj(x) : x;
    }
    const int nblk = (rows + 15) / 16;
    qr_f64x4 p = {0.0, 0.0, 0.0, 0.0}, q = p, s = p;
    auto vload = [&](double2 (&a)[4], int b) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = 16 * b + 4 * u + lk;
            a[u] = ld_or_zero(v, r + ldv * li, r < rows && li < nb);
        }
    };
    // (the next block's reflectors on their way; the taller tile has no registers for that)
    constexpr int BUF = NB <= 4 ? 2 : 1;
    double2 va[BUF][4];
    if (BUF == 2 && wv < nblk && wv >= b0) vload(va[0], wv);
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int b = wv + nw * t;
        if (b >= nblk) break;
        if (BUF == 2 && b + nw < nblk && b + nw >= b0) vload(va[(t + 1) % BUF], b + nw);
        if (b < b0) continue;
        if (BUF == 1) vload(va[0], b);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double2 a = va[t % BUF][u], y = Y[t][u];
            p = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, y.x, p, 0, 0, 0);
            q = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, y.y, q, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x - a.y, y.x + y.y, s, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)  // conj(a) b = (P + Q) + i (S - P + Q)
        sh.part[wv][lk + 4 * r][li] = make_double2(p[r] + q[r], s[r] - p[r] + q[r]);
    __syncthreads();
    for (int e = tid; e < QR_NB * QR_TC; e += 64 * nw) {
        double2 w = sh.part[0][e >> 4][e & 15];
        for (int k = 1; k < nw; ++k) w = cadd(w, sh.part[k][e >> 4][e & 15]);
        sh.w[e >> 4][e & 15] = w;
    }
    // the first block's reflectors for the last product, on their way during the barrier
    auto wload = [&](double2 (&a)[4], int b) {
        const int r = 16 * b + li;
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = ld_or_zero(v, r + ldv * (4 * k + lk), r < rows && 4 * k + lk < nb);
    };
    if (BUF == 2 && wv < nblk && wv >= b0) wload(va[0], wv);
    __syncthreads();
    p = q = s = qr_f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double2 w = sh.w[4 * k + lk][li];
        p = __builtin_amdgcn_mfma_f64_16x16x4f64(tv[k].x, w.x, p, 0, 0, 0);
        q = __builtin_amdgcn_mfma_f64_16x16x4f64(tv[k].y, w.y, q, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f64_16x16x4f64(tv[k].x + tv[k].y, w.x + w.y, s, 0, 0, 0);
    }
    double2 w2[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) w2[r] = make_double2(p[r] - q[r], s[r] - p[r] - q[r]);
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int b = wv + nw * t;
        if (b >= nblk) break;
        if (BUF == 2 && b + nw < nblk && b + nw >= b0) wload(va[(t + 1) % BUF], b + nw);
        if (b < b0) continue;
        if (BUF == 1) wload(va[0], b);
        p = q = s = qr_f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double2 a = va[t % BUF][k];
            p = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, w2[k].x, p, 0, 0, 0);
            q = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, w2[k].y, q, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x + a.y, w2[k].x + w2[k].y, s, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            Y[t][r] = csub(Y[t][r], make_double2(p[r] - q[r], s[r] - p[r] - q[r]));
    }
}

// T (sh.t) from the panel's rows, sums, scales and tau, by one wave: the dots
// v_k^H v_c = conj(s_k row_c(k)) + s_c conj(s_k tot_c(k)), then T of two neighbouring
// blocks of s columns from theirs, T12 = -T11 M12 T22, for s = 1, 2, 4, 8 (one entry per
// lane; 16 columns one after the other would be a chain twice as long, and inside the
// column loop it would hold up every column).
__device__ __forceinline__ void panel_t(TileShared& sh) {
    const int lane = threadIdx.x & 63;
    for (int e = lane; e < QR_NB * QR_NB; e += 64) {
        const int i = e / QR_NB, j = e % QR_NB;
        sh.t[i][j] = i == j ? sh.tau[i] : cz();
        const double2 si = sh.scale[i];
        sh.dot[i][j] = i < j ? cadd(cconj(cmul(si, sh.row[j][i])), cmul(sh.scale[j], cconj(cmul(si, sh.tot[j][i]))))
                             : cz();
    }
    wave_lds_sync();
#pragma unroll
    for (int s = 1; s < QR_NB; s *= 2) {
        const bool on = lane < 8 * s;  // QR_NB / (2 s) block pairs of s × s entries
        const int e = on ? lane : 0;
        const int p = e / (s * s), i = (e / s) % s, j = e % s;
        const int r0 = 2 * s * p, c0 = r0 + s;
        double2 x = cz();
#pragma unroll
        for (int l = 0; l < s; ++l) x = cfma(sh.dot[r0 + i][c0 + l], sh.t[c0 + l][c0 + j], x);
        if (on) sh.x[e] = x;
        wave_lds_sync();
        double2 t = cz();
#pragma unroll
        for (int l = 0; l < s; ++l) t = cfms(sh.t[r0 + i][r0 + l], sh.x[p * s * s + l * s + j], t);
        wave_lds_sync();
        if (on) sh.t[r0 + i][c0 + j] = t;
        wave_lds_sync();
    }
}

// Column C of the panel in Y, whose diagonal block is block D of the tile (D = 1: block 0
// holds rows above the panel).  With x = column C below the diagonal, one sum over the
// rows gives s_k = x^H a_k for every column k (s_C = ||x||^2); row C (alpha, a_k(C)) is
// published before that sum's barrier, so the reflector v = (1; x·scale) and every dot with
// it follow without a second sum: v^H a_k = a_k(C) + conj(scale) s_k.
// The sums on the matrix cores: a 4 × 4 × 4 step (four of them side by side) takes A = four
// rows of the sixteen columns and B = the real and imaginary part of x in two of its four
// columns, so two steps per four rows (real and imaginary part of the columns) give all
// sixteen complex sums already added over the lanes -- the vector unit needs 64 FMAs for
// the products and as many operations again to add 16 values over 64 lanes, at 12 cycles
// each for a wave that has its SIMD to itself.  x reaches the other columns' lanes by a
// broadcast within the 16-lane row.
// Factored columns stay unscaled; `scale` keeps the lane's column's factor (v = x·scale).
template <int C, int NB, int D>
__device__ __forceinline__ void panel_column(double2 (&Y)[NB][4], double2& scale, int nblk, int nb, int nw, int wv,
                                             TileShared& sh) {
    constexpr bool HOLD = NB <= 4;  // x kept for the update (else broadcast again)
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    auto xval = [&](int t, int u) {
        double2 x = row_bcast<C>(Y[t][u]);
        if (t == 0) {
            if (D == 1 && wv == 0) x = cz();
            if (wv == D && 4 * u + lk <= C) x = cz();
        }
        return x;
    };
    double2 xs[HOLD ? NB : 1][4];
    double d1[2] = {0.0, 0.0}, d2[2] = {0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        if (wv + nw * t >= nblk) break;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double2 x = xval(t, u);
            if (HOLD) xs[HOLD ? t : 0][u] = x;
            const double b = (lane & 1) ? x.y : x.x;
            d1[u & 1] = __builtin_amdgcn_mfma_f64_4x4x4f64(Y[t][u].x, b, d1[u & 1], 0, 0, 0);
            d2[u & 1] = __builtin_amdgcn_mfma_f64_4x4x4f64(Y[t][u].y, b, d2[u & 1], 0, 0, 0);
        }
    }
    // lane l: column 4 ((l % 16) / 4) + l / 16 against x's real (l % 4 = 0) or imaginary
    // part (1)
    const double e1 = d1[0] + d1[1], e2 = d2[0] + d2[1];
    const double o1 = dpp_d<DPP_XOR1>(e1), o2 = dpp_d<DPP_XOR1>(e2);
    if ((lane & 3) == 0) sh.red[C & 1][wv][4 * (li >> 2) + lk] = make_double2(e1 + o2, e2 - o1);
    if (wv == D && lk == C % 4) sh.row[C][li] = Y[0][C / 4];
    __syncthreads();
    const double2 row = sh.row[C][li];
    // the waves' parts, four to a 4 × 4 × 4 step with A = 1 (B: wave l / 16, column l % 16; the
    // sum lands in every row): two reads and four steps for eight waves instead of eight
    // reads and fourteen additions
    const double2 r0 = sh.red[C & 1][lk][li];
    double2 tot = make_double2(__builtin_amdgcn_mfma_f64_4x4x4f64(1.0, r0.x, 0.0, 0, 0, 0),
                               __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, r0.y, 0.0, 0, 0, 0));
    if (nw > 4) {
        const double2 r1 = sh.red[C & 1][4 + lk][li];
        tot = make_double2(__builtin_amdgcn_mfma_f64_4x4x4f64(1.0, r1.x, tot.x, 0, 0, 0),
                           __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, r1.y, tot.y, 0, 0, 0));
    }
    const Reflector h = make_reflector(row_bcast<C>(row), dpp_d<DPP_ROW_BCAST + C>(tot.x));
    if (wv == 0 && lk == 0) {  // (for T, once the panel is done)
        sh.tot[C][li] = tot;
        if (li == C) {
            sh.tau[C] = h.tau;
            sh.scale[C] = h.scale;
        }
    }
    if (li > C) {  // a_k -= conj(tau) (v^H a_k) v
        // (conj(tau scale) = -1 / beta)
        const double2 tr = cmul(cconj(h.tau), row);
        const double2 w = make_double2(fma(-h.rbeta, tot.x, tr.x), fma(-h.rbeta, tot.y, tr.y));
        const double2 ws = cmul(w, h.scale);
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            if (wv + nw * t >= nblk) break;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if constexpr (HOLD) Y[t][u] = cfms(ws, xs[t][u], Y[t][u]);
            }
        }
        if (wv == D && lk == C % 4) Y[0][C / 4] = csub(Y[0][C / 4], w);
        if constexpr (!HOLD) scale = ws;  // (used below, outside this branch)
    }
    if constexpr (!HOLD) {
        // broadcasts need every lane of the row: the factored columns update by zero
        const double2 ws = li > C ? scale : cz();
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            if (wv + nw * t >= nblk) break;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double2 x = xval(t, u);
                if (li > C) Y[t][u] = cfms(ws, x, Y[t][u]);
            }
        }
    }
    if (li == C) {
        scale = h.scale;
        if (wv == D && lk == C % 4) Y[0][C / 4] = make_double2(h.beta, 0.0);
    }
    if constexpr (C + 1 < QR_NB) {
        if (C + 1 < nb) panel_column<C + 1, NB, D>(Y, scale, nblk, nb, nw, wv, sh);
    }
}

// The panel at columns [j, j + nb) of the item, factored in the registers that hold it
// from row j - 16 D on; R back to a, the explicit reflectors to v, T to t.
template <int NB, int D>
__device__ __forceinline__ void panel_factor(double2 (&Y)[NB][4], const QrItem& it, int j, int nw, int wv,
                                             TileShared& sh) {
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int nb = min(QR_NB, it.n - j);
    const int rows = it.m - j + 16 * D, nblk = (rows + 15) / 16;
    if (wv == 0) {
        // (columns past the panel only: another wave may already have published row 0)
        for (int e = nb * QR_NB + lane; e < QR_NB * QR_NB; e += 64)
            sh.row[e >> 4][e & 15] = sh.tot[e >> 4][e & 15] = cz();
        if (lane < QR_NB) sh.tau[lane] = sh.scale[lane] = cz();
        wave_lds_sync();
    }
    double2 scale = cz();
    panel_column<0, NB, D>(Y, scale, nblk, nb, nw, wv, sh);
    const size_t lda = it.lda;
    double2* a = it.a + (j - 16 * D) + lda * j;
    double2* v = it.v + (j - 16 * D) + (size_t)it.m * j;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int b = wv + nw * t;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = 16 * b + 4 * u + lk, pr = r - 16 * D;  // pr: row of the panel
            if (r >= rows || li >= nb) continue;
            const bool upper = pr <= li;
            gstore(a, r + lda * li, upper ? Y[t][u] : cz());
            if (pr >= 0)
                gstore(v, r + (size_t)it.m * li,
                       upper ? make_double2(pr == li ? 1.0 : 0.0, 0.0) : cmul(Y[t][u], scale));
        }
    }
    if (wv == 0) {
        wave_lds_sync();
        panel_t(sh);
        double2* t = it.t + (size_t)(j / QR_NB) * QR_NB * QR_NB;
        for (int e = lane; e < QR_NB * QR_NB; e += 64) {
            const int i = e % QR_NB, k = e / QR_NB;
            gstore(t, e, (i < nb && k < nb) ? sh.t[i][k] : cz());
        }
    }
}

// Panel j of every item, one workgroup each.  What bounds it is the chain of 16 columns
// (sum, barrier, reflector, update: ~2900 cycles each at 256 rows), not the card: 65 panels
// of up to 256 rows took 29 us each with one row per thread and vector sums, 21.8 us with the sums
// on the matrix cores; refined reciprocals and the waves' parts added by 4 × 4 × 4 steps too: two
// panels to a launch, chi = 128, 22.9 -> 21.4 us.
template <int NB>
__global__ __launch_bounds__(QR_TILE_NT) __attribute__((amdgpu_waves_per_eu(2))) void k_qr_panel(
    const QrItem* __restrict__ items, int j) {
    __shared__ TileShared sh;
    const QrItem it = items[blockIdx.x];
    if (j >= it.n) return;
    const int wv = wave_index(), rows = it.m - j, nw = panel_waves((rows + 15) / 16);
    if (wv >= nw) return;  // (a barrier waits only for the waves still running)
    double2 Y[NB][4];
    tile_load<NB>(Y, it.a + j + (size_t)it.lda * j, it.lda, rows, min(QR_NB, it.n - j), nw, wv);
    panel_factor<NB, 0>(Y, it, j, nw, wv, sh);
}

// ---------------------------------------------------------------------------
// Panels of 1025 to 4096 rows: G columns at a time in registers
// ---------------------------------------------------------------------------
// One workgroup of 1024 threads, thread t with rows t + 1024 i, i < R, of the G columns that
// are being factored (R G = 16 entries, half of the 128 registers that 1024 threads leave each;
// with the sums and the next column's loads about 50 spill).  A column costs one sum over
// the workgroup as in panel_column.  When the G columns are done, one pass over the panel's
// other columns gives V^H a_k of the later ones and v_i^H V of the earlier ones (for T), and a
// second updates the later ones.  2048 rows: 16 columns in memory, every column read twice for
// each of the 16 steps, took 257 us a panel, now 104; what is left is the chain of 16 sums and the
// spilled registers.
constexpr int QR_TALL_NT = 1024, QR_TALL_NW = QR_TALL_NT / 64;
constexpr int QR_TALL_ROWS = 4096;
struct TallShared {
    double2 red[2][QR_TALL_NW][8];  // per wave: its part of a column's sums, two alternating buffers
    double2 row[2][8];              // row c of the group, likewise
    double2 part[QR_TALL_NW][64];   // per wave: its part of the passes' sums
    double2 w[64], z[64];
    double2 tau[QR_NB];
    double2 dot[QR_NB][QR_NB + 1];  // v_i^H v_j, i < j, within a group
    double2 t[QR_NB][QR_NB + 1];
};
// sums of G values per lane over the wave, value j to dst[j]
template <int G>
__device__ __forceinline__ void wave_sums(double2 (&s)[G], double2* dst) {
    const int lane = threadIdx.x & 63;
    double2 h[G / 2], q[G / 4];
#pragma unroll
    for (int j = 0; j < G / 2; ++j) h[j] = halve_swap<32>(s[j], s[j + G / 2]);
#pragma unroll
    for (int j = 0; j < G / 4; ++j) q[j] = halve_swap<16>(h[j], h[j + G / 4]);
    // lane l holds values (l / 32) G / 2 + (l / 16 mod 2) G / 4 + j summed over two lane bits;
    // the rest within the 16-lane row
#pragma unroll
    for (int j = 0; j < G / 4; ++j) {
        double2 a = cadd(q[j], row_ror<8>(q[j]));
        a = cadd(a, row_ror<4>(a));
        a = cadd(a, row_ror<2>(a));
        a = cadd(a, row_ror<1>(a));
        if ((lane & 15) == 0) dst[(lane >> 5) * (G / 2) + ((lane >> 4) & 1) * (G / 4) + j] = a;
    }
}

template <int R, int G>
__global__ __launch_bounds__(QR_TALL_NT) void k_qr_panel_tall(const QrItem* __restrict__ items, int j0) {
    __shared__ TallShared sh;
    const QrItem it = items[blockIdx.x];
    if (j0 >= it.n) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_index();
    const int rows = it.m - j0, nb = min(QR_NB, it.n - j0);
    const size_t lda = it.lda, ldv = it.m;
    double2* a = it.a + j0 + lda * j0;
    double2* v = it.v + j0 + ldv * j0;
    for (int e = tid; e < QR_NB * QR_NB; e += QR_TALL_NT) sh.t[e / QR_NB][e % QR_NB] = cz();
    for (int g0 = 0; g0 < nb; g0 += G) {
        double2 Y[R][G];
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const int r = tid + QR_TALL_NT * i;
                Y[i][k] = ld_or_zero(a, r + lda * (g0 + k), r < rows && g0 + k < nb);
            }
#pragma unroll
        for (int c = 0; c < G; ++c) {
            const int C = g0 + c;
            if (C < nb) {  // (the same for all threads)
                // rows above the diagonal's count as zero: they are thread 0 .. C's first
                double2 s[G];
#pragma unroll
                for (int k = 0; k < G; ++k) s[k] = cz();
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const double2 x = (i > 0 || tid > C) ? Y[i][c] : cz();
#pragma unroll
                    for (int k = 0; k < G; ++k) {
                        if (k == c) s[k].x += cabs2(x);
                        else s[k] = cfmac(x, Y[i][k], s[k]);
                    }
                }
                wave_sums<G>(s, sh.red[c & 1][wv]);
                if (tid == C) {
#pragma unroll
                    for (int k = 0; k < G; ++k) sh.row[c & 1][k] = Y[0][k];
                }
                __syncthreads();
                // lane l: value l mod G, waves l / G, l / G + 64 / G, ...
                const int k0 = lane % G;
                double2 tot = sh.red[c & 1][lane / G][k0];
                if (64 / G < QR_TALL_NW) tot = cadd(tot, sh.red[c & 1][lane / G + 64 / G][k0]);
                tot = cadd(tot, row_ror<8>(tot));
                if (G == 4) tot = cadd(tot, row_ror<4>(tot));
                tot = sum_rows16(tot);
                const double2 row = sh.row[c & 1][k0];
                const double2 alpha = make_double2(bcast_d(row.x, c), bcast_d(row.y, c));
                const Reflector h = make_reflector(alpha, bcast_d(tot.x, c));
                if (tid < c) sh.dot[g0 + tid][C] = cadd(cconj(row), cmul(h.scale, cconj(tot)));
                if (tid == c) sh.tau[C] = h.tau;
                // a_k -= conj(tau) (v^H a_k) v
                const double2 wl = cmul(cconj(h.tau), cadd(row, cmul(cconj(h.scale), tot)));
                const double2 wsl = cmul(wl, h.scale);
#pragma unroll
                for (int k = c + 1; k < G; ++k) {
                    const double2 ws = make_double2(bcast_d(wsl.x, k), bcast_d(wsl.y, k));
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        const double2 x = (i > 0 || tid > C) ? Y[i][c] : cz();
                        Y[i][k] = cfms(ws, x, Y[i][k]);
                    }
                    const double2 w = make_double2(bcast_d(wl.x, k), bcast_d(wl.y, k));
                    if (tid == C) Y[0][k] = csub(Y[0][k], w);
                }
#pragma unroll
                for (int i = 0; i < R; ++i)
                    if (i > 0 || tid > C) Y[i][c] = cmul(Y[i][c], h.scale);
                if (tid == C) Y[0][c] = make_double2(h.beta, 0.0);
            }
        }
        // R to a, explicit reflectors to v and to the registers
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const int r = tid + QR_TALL_NT * i, col = g0 + k;
                const bool upper = r <= col;
                const double2 vv = upper ? make_double2(r == col ? 1.0 : 0.0, 0.0) : Y[i][k];
                if (r < rows && col < nb) {
                    gstore(a, r + lda * col, upper ? Y[i][k] : cz());
                    gstore(v, r + ldv * col, vv);
                }
                Y[i][k] = col < nb ? vv : cz();
            }
        // the group's triangle of T by the first wave, lane i row i:
        // t_ic = -tau_c sum_l t_il (v_l^H v_c)
        if (wv == 0) {
            wave_lds_sync();
            double2 tr[G];
#pragma unroll
            for (int c = 0; c < G; ++c) {
                double2 acc = cz();
#pragma unroll
                for (int l = 0; l < c; ++l)
                    if (l >= lane && g0 + c < nb) acc = cfma(tr[l], sh.dot[g0 + l][g0 + c], acc);
                const double2 tau = g0 + c < nb ? sh.tau[g0 + c] : cz();
                const double2 p = cmul(tau, acc);
                tr[c] = lane == c ? tau : make_double2(-p.x, -p.y);
            }
            if (lane < G) {
#pragma unroll
                for (int c = 0; c < G; ++c)
                    if (c >= lane) sh.t[g0 + lane][g0 + c] = tr[c];
            }
        }
        // pass 1: entries [0, n2): V^H a_k of the later columns; [n2, n2 + g0): v_i^H V
        const int n2 = max(nb - g0 - G, 0), count = n2 + g0;
        auto column = [&](int e, double2 (&y)[R]) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int r = tid + QR_TALL_NT * i;
                y[i] = e < n2 ? ld_or_zero(a, r + lda * (g0 + G + e), r < rows)
                              : ld_or_zero(v, r + ldv * (e - n2), e < count && r < rows);
            }
        };
        double2 y[R], yn[R];
        column(0, y);
#pragma unroll 1
        for (int e = 0; e < count; ++e) {
            column(e + 1, yn);
            double2 s[G];
#pragma unroll
            for (int k = 0; k < G; ++k) {
                s[k] = cz();
#pragma unroll
                for (int i = 0; i < R; ++i) s[k] = cfmac(Y[i][k], y[i], s[k]);
            }
            wave_sums<G>(s, &sh.part[wv][e * G]);
#pragma unroll
            for (int i = 0; i < R; ++i) y[i] = yn[i];
        }
        __syncthreads();
        if (tid < count * G) {
            double2 w = sh.part[0][tid];
            for (int k = 1; k < QR_TALL_NW; ++k) w = cadd(w, sh.part[k][tid]);
            sh.w[tid] = w;
        }
        __syncthreads();
        if (tid < count * G) {
            const int e = tid / G, j = tid % G;
            double2 z = cz();
            if (e < n2) {  // T^H (V^H a_k)
                for (int l = 0; l <= j; ++l) z = cfmac(sh.t[g0 + l][g0 + j], sh.w[e * G + l], z);
            } else {  // (v_i^H V) T, the sums having V^H v_i
                for (int l = 0; l <= j; ++l) z = cfma(cconj(sh.w[e * G + l]), sh.t[g0 + l][g0 + j], z);
            }
            sh.z[tid] = z;
        }
        __syncthreads();
        // T's block above the group: -T (V_before^H V) T_group
        if (tid < g0 * G) {
            const int i = tid / G, j = tid % G;
            double2 t = cz();
            for (int l = i; l < g0; ++l) t = cfms(sh.t[i][l], sh.z[(n2 + l) * G + j], t);
            sh.t[i][g0 + j] = t;
        }
        // pass 2: a_k -= V z_k
        column(0, y);
#pragma unroll 1
        for (int e = 0; e < n2; ++e) {
            column(e + 1, yn);
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const double2 z = sh.z[e * G + k];
#pragma unroll
                for (int i = 0; i < R; ++i) y[i] = cfms(z, Y[i][k], y[i]);
            }
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int r = tid + QR_TALL_NT * i;
                if (r < rows) gstore(a, r + lda * (g0 + G + e), y[i]);
                y[i] = yn[i];
            }
        }
        __syncthreads();
    }
    double2* t = it.t + (size_t)(j0 / QR_NB) * QR_NB * QR_NB;
    for (int e = tid; e < QR_NB * QR_NB; e += QR_TALL_NT) gstore(t, e, sh.t[e % QR_NB][e / QR_NB]);
}

// panels of more rows, in place in global memory
__global__ __launch_bounds__(512) void k_qr_panel_mem(const QrItem* __restrict__ items, int j0) {
    __shared__ PanelShared sh;
    const QrItem it = items[blockIdx.x];
    if (j0 >= it.n) return;
    qr_panel_global<512>(it, j0, sh);
}

// Y[j0:, c0 : c0 + tc] <- (I - V T' V^H) Y[j0:, c0 : c0 + tc],  T' = T^H (adjoint) or T,
// V and T of the panel of nb reflectors at j0, on the matrix cores (v_mfma_f64_16x16x4,
// three real products per complex product), operands straight from memory into registers.
// Operand layouts of a 16x16x4 step: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16]; result register q of lane l is D[l / 16 + 4 q][l % 16].
//   W = V^H Y: A[i][k] = conj V(r + k, j0 + i), B[k][j] = Y(r + k, c0 + j), four rows a
//     step; wave wv takes steps wv, wv + NW, ..., loads of the next 8 steps in flight
//     while 8 are multiplied.  The waves' partial sums meet in LDS.
//   W2 = T' W on the vector ALUs (one entry per thread).
//   Y -= V W2 as (V W2)^T = W2^T V^T, so that a lane's results lie along one column
//     of Y: A[j][k] = W2(k, j), B[k][i] = V(r0 + i, j0 + k); one 16-row block per
//     step, wave wv takes blocks wv, wv + NW, ..., two at a time.
// (Eight waves: a matrix of 2048 columns has 128 tiles for 256 CUs; with four the update took
// 55 instead of 48 us and forming Q 4.5 instead of 3.9 ms.)
template <int NW>  // waves of the workgroup
struct ApplyMfmaShared {
    double2 sPart[NW][QR_NB][QR_TC];
    double2 sW[QR_NB][QR_TC + 1];
    double2 sW2[QR_NB][QR_TC + 1];
    double2 sT[QR_NB][QR_NB + 1];
};
template <int NW>
__device__ __forceinline__ void qr_apply_panel_mfma(const QrApplyItem& it, int c0, int tc, int j0, int nb,
                                                    int adjoint, ApplyMfmaShared<NW>& sh) {
    static_assert(QR_TC == QR_NB && QR_NB == 16, "tiles are 16 reflectors × 16 columns");
    constexpr int NT = 64 * NW;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int m = it.m;
    const size_t ldy = it.ldy;
    const double2* t = it.t + (size_t)(j0 / QR_NB) * QR_NB * QR_NB;
    for (int e = tid; e < QR_NB * QR_NB; e += NT) sh.sT[e % QR_NB][e / QR_NB] = gload(t, e);
    // ---- phase 1: W = V^H Y over rows j0 .. m - 1
    const int steps = (m - j0 + 3) / 4;
    const int mine = (steps - wv + NW - 1) / NW;  // this wave's steps: s = wv + NW t, t < mine
    const double2* vcol = it.v + (size_t)m * (j0 + li);
    const double2* ycol = it.y + ldy * (c0 + li);
    const bool vok = li < nb, yok = li < tc;
    constexpr int U = 8;
    double2 a0[U], b0[U], a1[U], b1[U];
    auto fetch = [&](int t0, double2 (&a)[U], double2 (&b)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = j0 + 4 * (wv + NW * (t0 + u)) + lk;
            const bool ok = t0 + u < mine && r < m;
            a[u] = ld_or_zero(vcol, r, ok && vok);
            b[u] = ld_or_zero(ycol, r, ok && yok);
        }
    };
    qr_f64x4 p = {0.0, 0.0, 0.0, 0.0}, q = p, s = p;
    auto mult = [&](const double2 (&a)[U], const double2 (&b)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            p = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].x, b[u].x, p, 0, 0, 0);
            q = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].y, b[u].y, q, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u].x - a[u].y, b[u].x + b[u].y, s, 0, 0, 0);
        }
    };
    fetch(0, a0, b0);
    for (int t0 = 0; t0 < mine; t0 += 2 * U) {
        fetch(t0 + U, a1, b1);
        mult(a0, b0);
        if (t0 + 2 * U < mine) fetch(t0 + 2 * U, a0, b0);
        mult(a1, b1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)  // conj(a) b = (P + Q) + i (S - P + Q)
        sh.sPart[wv][lk + 4 * r][li] = make_double2(p[r] + q[r], s[r] - p[r] + q[r]);
    __syncthreads();
    const int wa = (tid / QR_TC) % QR_NB, wc = tid % QR_TC;  // threads 0..255: one entry each
    if (tid < QR_NB * QR_TC) {
        double2 w = sh.sPart[0][wa][wc];
#pragma unroll
        for (int k = 1; k < NW; ++k) w = cadd(w, sh.sPart[k][wa][wc]);
        sh.sW[wa][wc] = w;
    }
    __syncthreads();
    // ---- phase 2: W2 = T' W
    if (tid < QR_NB * QR_TC) {
        double2 w2 = cz();
        for (int b = 0; b < QR_NB; ++b) {
            const double2 tab = adjoint ? cconj(sh.sT[b][wa]) : sh.sT[wa][b];
            w2 = cfma(tab, sh.sW[b][wc], w2);
        }
        sh.sW2[wa][wc] = w2;
    }
    __syncthreads();
    // ---- phase 3: Y -= V W2, 16-row blocks
    double2 wt[4];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) wt[k4] = sh.sW2[4 * k4 + lk][li];
    const int nblk = (m - j0 + 15) / 16;
    for (int blk0 = wv; blk0 < nblk; blk0 += 2 * NW) {
        double2 vv[2][4], yo[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int blk = blk0 + NW * h;
            const int row = j0 + 16 * blk + li;
            const bool rok = blk < nblk && row < m;
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4)
                vv[h][k4] = ld_or_zero(it.v, row + (size_t)m * (j0 + 4 * k4 + lk), rok && 4 * k4 + lk < nb);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                yo[h][r] = ld_or_zero(it.y, row + ldy * (c0 + lk + 4 * r), rok && lk + 4 * r < tc);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            qr_f64x4 dp = {0.0, 0.0, 0.0, 0.0}, dq = dp, ds = dp;
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) {
                const double2 a = wt[k4], b = vv[h][k4];
                dp = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, dp, 0, 0, 0);
                dq = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, dq, 0, 0, 0);
                ds = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x + a.y, b.x + b.y, ds, 0, 0, 0);
            }
            const int blk = blk0 + NW * h;
            const int row = j0 + 16 * blk + li;
            if (blk < nblk && row < m) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {  // a b = (P - Q) + i (S - P - Q)
                    const int c = lk + 4 * r;
                    if (c < tc)
                        gstore(it.y, row + ldy * (c0 + c),
                               csub(yo[h][r], make_double2(dp[r] - dq[r], ds[r] - dp[r] - dq[r])));
                }
            }
        }
    }
}

// one block reflector (panel j0) on one column tile per workgroup
__global__ __launch_bounds__(512) void k_qr_apply(const QrApplyItem* __restrict__ items, const int2* __restrict__ tiles,
                                                  int j0, int adjoint) {
    __shared__ ApplyMfmaShared<8> sh;
    const int2 tt = tiles[blockIdx.x];
    const QrApplyItem it = items[tt.x];
    const int nb = min(QR_NB, it.nrefl - j0);
    if (nb <= 0) return;
    const int c0 = (it.trailing ? j0 + nb : 0) + tt.y * QR_TC;
    const int tc = min(QR_TC, it.ncols - c0);
    if (tc <= 0) return;
    qr_apply_panel_mfma(it, c0, tc, j0, nb, adjoint, sh);
}

// Y <- Q Y with every block reflector of the factorisation, last panel first: the column
// tiles are independent, so one workgroup walks all panels of its tile, which stays in its
// registers from the first panel to the last (up to 1024 rows; taller ones in memory).
// A target that starts as a diagonal (eye) is still zero in a tile's columns until the panel
// that starts at or before the tile's last column.  (256 rows: 70 -> 31 us; 512 rows,
// layers of 256: 764 -> 553 us, there at the matrix cores' rate for its 24 multiply-adds.  The
// form for 513 to 1024 rows, 64 registers of tile more, spills 78.)
template <int NB>
__global__ __launch_bounds__(QR_TILE_NT) __attribute__((amdgpu_waves_per_eu(2))) void k_qr_form(
    const QrApplyItem* __restrict__ items, const int2* __restrict__ tiles) {
    __shared__ TileShared sh;
    const int2 tt = tiles[blockIdx.x];
    const QrApplyItem it = items[tt.x];
    const int c0 = tt.y * QR_TC;
    const int tc = min(QR_TC, it.ncols - c0);
    if (tc <= 0 || it.nrefl <= 0) return;
    const int wv = wave_index();
    double2 Y[NB][4];
    if (it.eye == 2) tile_unit<NB>(Y, c0, tc, 8, wv);
    else tile_load<NB>(Y, it.y + (size_t)it.ldy * c0, it.ldy, it.m, tc, 8, wv);
    const int last = it.eye ? min(it.nrefl - 1, c0 + tc - 1) : it.nrefl - 1;
    for (int j0 = (last / QR_NB) * QR_NB; j0 >= 0; j0 -= QR_NB)
        tile_apply<NB>(Y, it.v + (size_t)it.m * j0, it.m, it.m, min(QR_NB, it.nrefl - j0),
                       it.t + (size_t)(j0 / QR_NB) * QR_NB * QR_NB, 0, j0 / 16, 8, wv, sh);
    if (!it.trans) {
        tile_store<NB>(Y, it.y + (size_t)it.ldy * c0, it.ldy, it.m, tc, 8, wv);
        return;
    }
    // (a lane's column is a row of the result: 16 lanes write 16 neighbouring entries)
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * (wv + 8 * t) + 4 * q + lk;
            if (r >= it.m || li >= tc) continue;
            const int o = it.row_div > 0 ? r / it.row_div + (it.m / it.row_div) * (r % it.row_div) : r;
            gstore(it.y, c0 + li + (size_t)it.ldy * o, cconj(Y[t][q]));
        }
    }
}
__global__ __launch_bounds__(512) void k_qr_form_tall(const QrApplyItem* __restrict__ items,
                                                      const int2* __restrict__ tiles) {
    __shared__ ApplyMfmaShared<8> sh;
    const int2 tt = tiles[blockIdx.x];
    const QrApplyItem it = items[tt.x];
    const int c0 = tt.y * QR_TC;
    const int tc = min(QR_TC, it.ncols - c0);
    if (tc <= 0 || it.nrefl <= 0) return;
    const int last = it.eye ? min(it.nrefl - 1, c0 + tc - 1) : it.nrefl - 1;
    for (int j0 = (last / QR_NB) * QR_NB; j0 >= 0; j0 -= QR_NB) {
        qr_apply_panel_mfma(it, c0, tc, j0, min(QR_NB, it.nrefl - j0), 0, sh);
        __syncthreads();
    }
}

// Look-ahead step of the factorisation: workgroup i < count applies panel j0's block
// reflector to the next panel's columns of item i and then factors that panel; the
// others apply panel j0's block reflector to the trailing tiles beyond it.  The two
// parts touch disjoint columns and disjoint reflector storage, so they run in one
// launch and the panel's latency hides behind the trailing update.  It remains what a
// factorisation of up to 512 rows waits for: 43 -> 29 us a step (256 rows), of which 8 us
// apply the block reflector and 20 us are the columns.
template <int NB>
__global__ __launch_bounds__(QR_TILE_NT) __attribute__((amdgpu_waves_per_eu(2))) void k_qr_step(
    const QrItem* __restrict__ items, int count, const int2* __restrict__ tiles, int j0) {
    __shared__ TileShared sh;
    const int wv = wave_index();
    double2 Y[NB][4];
    if ((int)blockIdx.x < count) {
        const QrItem it = items[blockIdx.x];
        const int jn = j0 + QR_NB;
        if (jn >= it.n) return;
        const int rows = it.m - j0, nw = panel_waves((rows + 15) / 16);
        if (wv >= nw) return;
        tile_load<NB>(Y, it.a + j0 + (size_t)it.lda * jn, it.lda, rows, min(QR_NB, it.n - jn), nw, wv);
        tile_apply<NB>(Y, it.v + j0 + (size_t)it.m * j0, it.m, rows, QR_NB,
                       it.t + (size_t)(j0 / QR_NB) * QR_NB * QR_NB, 1, 0, nw, wv, sh);
        panel_factor<NB, 1>(Y, it, jn, nw, wv, sh);
        return;
    }
    const int2 tt = tiles[blockIdx.x - count];
    const QrItem it = items[tt.x];
    const int nb = min(QR_NB, it.n - j0);
    if (nb <= 0) return;
    const int c0 = j0 + nb + tt.y * QR_TC;
    const int tc = min(QR_TC, it.n - c0);
    if (tc <= 0) return;
    double2* y = it.a + j0 + (size_t)it.lda * c0;
    tile_load<NB>(Y, y, it.lda, it.m - j0, tc, 8, wv);
    tile_apply<NB>(Y, it.v + j0 + (size_t)it.m * j0, it.m, it.m - j0, nb,
                   it.t + (size_t)(j0 / QR_NB) * QR_NB * QR_NB, 1, 0, 8, wv, sh);
    tile_store<NB>(Y, y, it.lda, it.m - j0, tc, 8, wv);
}

// the form of a panel of `rows` rows (also in launch_qr_panel)
int qr_panel_form(int rows) {
    return rows <= QR_REG_ROWS ? 0 : rows <= 2 * QR_TALL_NT ? 1 : rows <= QR_TALL_ROWS ? 2 : 3;
}
void launch_qr_panel(const QrItem* d_items, int count, int j0, int rows, hipStream_t s) {
    if (count <= 0) return;
    switch (qr_panel_form(rows)) {
        case 0:
            if (rows <= 512) k_qr_panel<4><<<count, QR_TILE_NT, 0, s>>>(d_items, j0);
            else k_qr_panel<8><<<count, QR_TILE_NT, 0, s>>>(d_items, j0);
            break;
        case 1: k_qr_panel_tall<2, 8><<<count, QR_TALL_NT, 0, s>>>(d_items, j0); break;
        case 2: k_qr_panel_tall<4, 4><<<count, QR_TALL_NT, 0, s>>>(d_items, j0); break;
        default: k_qr_panel_mem<<<count, 512, 0, s>>>(d_items, j0);
    }
}
void launch_qr_apply(const QrApplyItem* d_items, const int2* d_tiles, int ntiles, int j0, int adjoint, hipStream_t s) {
    if (ntiles <= 0) return;
    k_qr_apply<<<ntiles, 512, 0, s>>>(d_items, d_tiles, j0, adjoint);
}
void launch_qr_form(const QrApplyItem* d_items, const int2* d_tiles, int ntiles, int rows, hipStream_t s) {
    if (ntiles <= 0) return;
    if (rows <= 512) k_qr_form<4><<<ntiles, QR_TILE_NT, 0, s>>>(d_items, d_tiles);
    else if (rows <= QR_REG_ROWS) k_qr_form<8><<<ntiles, QR_TILE_NT, 0, s>>>(d_items, d_tiles);
    else k_qr_form_tall<<<ntiles, 512, 0, s>>>(d_items, d_tiles);
}
void launch_qr_step(const QrItem* d_items, int count, const int2* d_tiles, int ntiles, int j0, int rows,
                    hipStream_t s) {
    if (count + ntiles <= 0) return;
    if (rows <= 512) k_qr_step<4><<<count + ntiles, QR_TILE_NT, 0, s>>>(d_items, count, d_tiles, j0);
    else k_qr_step<8><<<count + ntiles, QR_TILE_NT, 0, s>>>(d_items, count, d_tiles, j0);
}
int qr_tile_cols() { return QR_TC; }

// dst (n × n) = upper triangle of src (ld lds)^H, zeros above the diagonal of dst, for
// a batch (tile map: item, block of 256 entries)
__global__ void k_upper_h_batch(const UpperHItem* __restrict__ items, const int2* __restrict__ tiles) {
    const int2 tt = tiles[blockIdx.x];
    const UpperHItem it = items[tt.x];
    const size_t e = (size_t)tt.y * 256 + threadIdx.x;
    if (e >= (size_t)it.n * it.n) return;
    const int i = (int)(e % it.n), j = (int)(e / it.n);
    it.dst[e] = (i >= j) ? cconj(it.src[j + (size_t)it.lds * i]) : cz();
}
void launch_upper_h_batch(const UpperHItem* d_items, const int2* d_tiles, int ntiles, hipStream_t s) {
    if (ntiles <= 0) return;
    k_upper_h_batch<<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}

__global__ __launch_bounds__(256) void k_sign_eye(const SignEyeItem* __restrict__ items,
                                                  const int2* __restrict__ tiles) {
    const int2 tt = tiles[blockIdx.x];
    const SignEyeItem it = items[tt.x];
    const size_t e = (size_t)tt.y * 256 + threadIdx.x;
    if (e >= (size_t)it.rows * it.cols) return;
    const int i = (int)(e % it.rows), j = (int)(e / it.rows);
    double v = 0.0;
    if (i == j) v = it.r[j + (size_t)it.ldr * j].x < 0.0 ? -1.0 : 1.0;
    gstore(it.out, e, make_double2(v, 0.0));
}
void launch_sign_eye(const SignEyeItem* d_items, const int2* d_tiles, int ntiles, hipStream_t s) {
    if (ntiles > 0) k_sign_eye<<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}

// Column order by decreasing norm (the column pivoting of the first pass, taken from
// the initial norms): one 1024-thread workgroup per item, a wave per column for the
// norms, then a rank sort with one thread per column.  A NaN norm sorts last (the
// Jacobi reports the matrix as non-finite).
__global__ __launch_bounds__(1024) void k_pivot_order(const PivotItem* __restrict__ items) {
    __shared__ double sKey[PIVOT_MAXQ];
    const PivotItem it = items[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    for (int j = wv; j < it.q; j += 16) {
        const cplx* col = it.x + (size_t)it.p * j;
        double s = 0.0;
        for (int r = lane; r < it.p; r += 64) s += cabs2(col[r]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if (lane == 0) sKey[j] = (s == s) ? s : -1.0;
    }
    __syncthreads();
    for (int j = tid; j < it.q; j += 1024) {
        const double k = sKey[j];
        int rank = 0;
        for (int u = 0; u < it.q; ++u) {
            const double ku = sKey[u];
            rank += (ku > k || (ku == k && u < j)) ? 1 : 0;
        }
        it.perm[rank] = j;
        it.perm_inv[j] = rank;
    }
    if (tid == 0) *it.count = it.q;
}
void launch_pivot_order(const PivotItem* d_items, int count, hipStream_t s) {
    if (count > 0) k_pivot_order<<<count, 1024, 0, s>>>(d_items);
}

}  // namespace qh
