// Batched block one-sided (Hestenes) Jacobi SVD in complex FP64, and the
// finalisation kernels: singular values, sort, the `truncate!` rule
// (src/Ansatz/Chain.jl:404-417) and the write-back of the kept factors.
//
// One launch = one round of a round-robin (circle-method) tournament over the
// column blocks of every matrix in the batch.  A workgroup owns one block pair
// (I, J) of one matrix: it forms the Gram matrix G = X_IJ^H X_IJ (BC × BC) from
// HBM, and if any off-diagonal |g_ij| exceeds tol·sqrt(g_ii g_jj) it
// diagonalises G with a cyclic two-sided Jacobi in LDS (FP64) and applies the
// accumulated unitary Q to the columns of X and V:  X_IJ <- X_IJ Q,
// V_IJ <- V_IJ Q.  Convergence is judged on freshly computed inner products, so
// the singular values carry the accuracy of one-sided Jacobi (relative
// accuracy on each σ_j = ||X e_j||).
#include "qh_kernels.h"
#include "qh_complex.h"

typedef double f64x4 __attribute__((ext_vector_type(4)));

namespace qh {

// The tail criterion at the start of an item's own sweep s (after sweep w = s - 1): an
// item of at least JAC_TAIL_NB blocks, past the sorting sweeps, not before
// own[JAC_TAIL_MIN], whose sweep w rotated some but at most tail_switch per mille of its
// block pairs (own[w mod 5]; a sweep without a rotation converges the item in the plain
// loop).
constexpr int JAC_TAIL_NB = 8;
__device__ __forceinline__ bool tail_due(const JacItem& it, int s, int sort_sweeps, int tail_switch) {
    const int w = s - 1;
    if (tail_switch <= 0 || it.nb < JAC_TAIL_NB || w < sort_sweeps || s < it.own[JAC_TAIL_MIN]) return false;
    const long long pairs = (long long)(it.nb - 1) * (it.nb / 2);
    const long long cnt = it.own[w % 5];
    return cnt > 0 && 1000LL * cnt <= tail_switch * pairs;
}
// The round kernels' entry decision (ts: the item's tail state): whether the workgroup
// runs (the item is not waiting for the tail passes) and, at the start of the
// item's own sweep `own` (round % R == 0), the tail criterion on its previous sweeps
// (every workgroup of the item reads the same counts and takes the same decision;
// workgroup 0 records it, in the launch that records) and the rotation count of the next
// sweep cleared.
__device__ __forceinline__ int round_gate(const JacItem& it, int ts, int round, int own, int R, int pair, int sort_sweeps,
                                          int tail_switch, bool record) {
    int go = ts != 1;
    if (go && round % R == 0) {
        if (ts == 0 && tail_due(it, own, sort_sweeps, tail_switch)) {
            go = 0;
            if (pair == 0 && record) {
                *it.tail = 1;
                it.own[JAC_TAIL_AT] = own;
            }
        }
        if (go && pair == 0 && record) it.own[(own + 1) % 5] = 0;
    }
    return go;
}
// rr_pair(round + 1, k, nidx) from rr_pair(round, k, nidx)
__device__ __forceinline__ void rr_next(int k, int nidx, int& a, int& b) {
    const int m = nidx - 1;
    if (k == 0) {
        ++a;
    } else {
        a = (a + 1 == m) ? 0 : a + 1;
        b = (b + 1 == m) ? 0 : b + 1;
    }
}


// Rotation of the Hermitian 2×2 problem [[g_aa, g_ab], [conj(g_ab), g_bb]]:
// J = [[c, s e], [-s conj(e), c]] with e = g_ab/|g_ab| and t = s/c the smaller
// root of t^2 + 2 zeta t - 1 = 0, zeta = (g_bb - g_aa)/(2|g_ab|) (Rutishauser's
// formulation); naa / nbb are the new diagonal.  No rotation (s = 0) when the
// pair is already orthogonal, |g_ab|^2 <= tol2·g_aa·g_bb, or a column is below
// the deflation floor.
// With d = g_bb - g_aa and h = sqrt(d^2 + 4|g_ab|^2) (= 2|g_ab| sqrt(1 + zeta^2)):
// |t| = 2|g_ab| / (|d| + h) and c^2 = 1/(1 + t^2) = (|d| + h) / (2h).  The rotation
// is applied through c and se = s e = sign(d) (2c / (|d| + h)) g_ab, and the new
// diagonal through t|g_ab| = sign(d) 2|g_ab|^2 / (|d| + h), so neither |g_ab| nor e
// is formed: two square roots and two divisions, chain sqrt, divide, sqrt.
struct JRot {
    double c = 1.0, sx = 0.0, sy = 0.0, naa = 0.0, nbb = 0.0;  // se = (sx, sy)
};
__device__ __forceinline__ bool rotates(const JRot& j) { return j.sx != 0.0 || j.sy != 0.0; }
__device__ __forceinline__ bool needs_rotation(double gaa, double gbb, double2 gab, double tol2, double gfloor) {
    return gaa > gfloor && gbb > gfloor && cabs2(gab) > tol2 * gaa * gbb;
}
__device__ __forceinline__ JRot jacobi_rot(double gaa, double gbb, double2 gab, double tol2, double gfloor) {
    JRot r;
    r.naa = gaa;
    r.nbb = gbb;
    if (needs_rotation(gaa, gbb, gab, tol2, gfloor)) {
        const double g2 = cabs2(gab);
        const double d = gbb - gaa;
        const double h = sqrt(fma(d, d, 4.0 * g2));
        const double den = fabs(d) + h;
        const double rden = 1.0 / den;
        r.c = sqrt(den / (2.0 * h));
        const double sg = d >= 0.0 ? 2.0 : -2.0;
        const double f = sg * r.c * rden;
        r.sx = f * gab.x;
        r.sy = f * gab.y;
        const double tm = sg * g2 * rden;
        r.naa = gaa - tm;
        r.nbb = gbb + tm;
    }
    return r;
}
// (x_a, x_b) <- (x_a, x_b) J
// (one product and two FMAs per real output)
__device__ __forceinline__ void rot_cols(double2& xa, double2& xb, const JRot& j) {
    const double sx = j.sx, sy = j.sy;  // x_a' = c x_a - conj(se) x_b ; x_b' = se x_a + c x_b
    const double2 na = make_double2(fma(-sy, xb.y, fma(-sx, xb.x, j.c * xa.x)),
                                    fma(sy, xb.x, fma(-sx, xb.y, j.c * xa.y)));
    xb = make_double2(fma(-sy, xa.y, fma(sx, xa.x, j.c * xb.x)), fma(sy, xa.x, fma(sx, xa.y, j.c * xb.y)));
    xa = na;
}
// (y_a; y_b) <- J^H (y_a; y_b)
__device__ __forceinline__ void rot_rows(double2& ya, double2& yb, const JRot& j) {
    const double sx = j.sx, sy = j.sy;  // y_a' = c y_a - se y_b ; y_b' = conj(se) y_a + c y_b
    const double2 na = make_double2(fma(sy, yb.y, fma(-sx, yb.x, j.c * ya.x)),
                                    fma(-sy, yb.x, fma(-sx, yb.y, j.c * ya.y)));
    yb = make_double2(fma(sy, ya.y, fma(sx, ya.x, j.c * yb.x)), fma(-sy, ya.x, fma(sx, ya.y, j.c * yb.y)));
    ya = na;
}

// ---------------------------------------------------------------------------
// Block width 16 (the default): a block pair is 32 columns, a workgroup eight waves.
//
// The Gram matrix, the eigensolver and the update of a pair are device functions shared
// by two forms of a round with the same arithmetic in the same order (bit-identical
// results, so an item's values do not depend on the batch it is in):
//   fused   one launch a round, one workgroup per pair doing all three (k_jacobi_round16);
//   split   three launches (k_jacobi_gram16, k_jacobi_eig16, k_jacobi_update16), the Gram
//           and the update spread over row chunks, for pairs that are few or tall.
// What bounds a pair (512 rows): the Gram is 1152 matrix-core steps and the update 1536, at
// 64 cycles each 18 us of a CU's four matrix cores; the eigensolver is a chain of 31
// dependent rounds.  FP64 vector instructions of one wave issue every 12 cycles (4 with
// three waves on the SIMD), so the pair's work is laid over eight waves, two per SIMD, and
// the two workgroups of a CU overlap one's eigensolver with the other's products.
// Measured against four waves with V accumulated, per round: 32 matrices of 512 columns
// 114 -> 84 us, 15 of 180 columns 60 -> 41 us, 16 uneven chains of up to 256 columns 68 ->
// 42 us; one matrix of 2048 columns (split form; before, 64-column pairs) 540 -> 216 ms in all.
// A lone 180-column pair's 44 us: entry 1.1, Gram 3.5, its reduction 1.7, test 1.1,
// eigensolver 27 (cross rounds 14), order 0.8, update 6.4.
// ---------------------------------------------------------------------------
constexpr int J16_LP = 33;
constexpr int J16_NT = 512;
constexpr int J16_TALL = 512;  // Gram groups: 2 interleaved ones up to this height, else 512 rows each
__host__ __device__ inline int jac16_groups(int p) { return p <= J16_TALL ? 2 : (p + 511) / 512; }

// The sum of X_IJ^H X_IJ's three blocks G11, G12, G22 over one wave's rows, on the matrix
// cores (v_mfma_f64_16x16x4): a 16-column block is one tile, and one value per lane is the
// operand of X_I^H X_J from either side (A[i][k] = x_i at row k, B[k][j] = x_j at row k).
// Three real products per complex block: P = ar br, Q = ai bi, S = (ar - ai)(br + bi);
// Re = P + Q, Im = S - P + Q (the conjugate of A is in the signs).  Operands come straight
// from memory, the next step's loads in flight (a step is 576 cycles of its SIMD's matrix
// core, and two to four waves share the SIMD); nothing is staged, so the waves need no
// barrier.  Wave w of group gr takes the four-row steps 4 gr + w + 8 t (heights up to
// J16_TALL: two groups of four waves, neighbouring waves on neighbouring 64-byte pieces of
// each column), or the steps w + 4 t of rows [512 gr, 512 gr + 512).
struct Gram16 {
    f64x4 p[3], q[3], s[3];
};
__device__ __forceinline__ void jac16_gram(const JacItem& it, const int* sCol, int gr, int w, Gram16& g) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int p = it.p;
    const int c1 = sCol[li], c2 = sCol[16 + li];
    const double2* x1 = it.x + (size_t)p * max(c1, 0);
    const double2* x2 = it.x + (size_t)p * max(c2, 0);
    const bool tall = p > J16_TALL;
    const int first = tall ? 128 * gr + w : 4 * gr + w, stride = tall ? 4 : 8;
    const int end = tall ? min((p + 3) / 4, 128 * gr + 128) : (p + 3) / 4;
#pragma unroll
    for (int b = 0; b < 3; ++b) g.p[b] = g.q[b] = g.s[b] = f64x4{0.0, 0.0, 0.0, 0.0};
    auto fetch = [&](double2 (&x)[2], int s) {
        const int r = min(4 * s + lk, p - 1);
        x[0] = gload(x1, r);
        x[1] = gload(x2, r);
    };
    auto mult = [&](const double2 (&x)[2], int s) {
        // rows past the end and absent columns were read in range and count as zero
        const bool in = 4 * s + lk < p;
        const double2 a = (in && c1 >= 0) ? x[0] : cz(), b = (in && c2 >= 0) ? x[1] : cz();
        const double da = a.x - a.y, ea = a.x + a.y, db = b.x - b.y, eb = b.x + b.y;
        g.p[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, a.x, g.p[0], 0, 0, 0);
        g.q[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, a.y, g.q[0], 0, 0, 0);
        g.s[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(da, ea, g.s[0], 0, 0, 0);
        g.p[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, g.p[1], 0, 0, 0);
        g.q[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, g.q[1], 0, 0, 0);
        g.s[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(da, eb, g.s[1], 0, 0, 0);
        g.p[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.x, b.x, g.p[2], 0, 0, 0);
        g.q[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.y, b.y, g.q[2], 0, 0, 0);
        g.s[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(db, eb, g.s[2], 0, 0, 0);
    };
    const int n = first < end ? (end - first + stride - 1) / stride : 0;
    if (n == 0) return;
    // (no exit inside the loop: the accumulators would be held twice)
    double2 xa[2], xb[2];
    fetch(xa, first);
#pragma unroll 1
    for (int t = 0; t + 1 < n; t += 2) {
        fetch(xb, first + stride * (t + 1));
        __builtin_amdgcn_sched_barrier(0);
        mult(xa, first + stride * t);
        __builtin_amdgcn_sched_barrier(0);
        fetch(xa, first + stride * min(t + 2, n - 1));
        __builtin_amdgcn_sched_barrier(0);
        mult(xb, first + stride * (t + 1));
        __builtin_amdgcn_sched_barrier(0);
    }
    if (n & 1) mult(xa, first + stride * (n - 1));
}
// entry `q` of block b (0: G11, 1: G12, 2: G22) of the lane's result
__device__ __forceinline__ double2 gram16_entry(const Gram16& g, int b, int q) {
    return make_double2(g.p[b][q] + g.q[b][q], g.s[b][q] - g.p[b][q] + g.q[b][q]);
}

struct Jac16Shared {
    double2 g[2][32][J16_LP];  // G, and the buffer its rounds alternate with
    double2 q[32][J16_LP];
    int col[32], perm[32];
    int flag, more, go;
};

// entry e of the Gram's three blocks (256 each: G11, G12, G22) to its place in G
__device__ __forceinline__ void jac16_put(Jac16Shared& sh, int e, double2 v) {
    const int b = e >> 8, r = (e >> 4) & 15, c = e & 15;
    sh.g[0][b == 2 ? 16 + r : r][b == 0 ? c : 16 + c] = v;
}

// lane 0's value of each 16-lane row (DPP row_newbcast)
__device__ __forceinline__ double row_bcast0(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x150, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x150, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// jacobi_rot from two refined reciprocal square roots instead of two square roots and two
// divisions (half the instructions and less than half the dependent chain, which is what a
// round of the eigensolver waits for).  With r = 1/sqrt(d^2 + 4|g|^2), c^2 = (1 + |d| r)/2
// and k = 1/c: se = sign(d) g r k, t|g| = |g|^2 r k^2.  The error of r would leave c^2 + |s|^2 off 1
// by as much, and over hundreds of rotations V off a unitary by as many times that, so c takes
// up what s leaves (singular values of 128 columns 9e-16 instead of 1.8e-15 off, 2 % of a round).
__device__ __forceinline__ JRot jacobi_rot_fast(double gaa, double gbb, double2 gab, double tol2, double gfloor) {
    JRot j;
    j.naa = gaa;
    j.nbb = gbb;
    if (needs_rotation(gaa, gbb, gab, tol2, gfloor)) {
        const double g2 = cabs2(gab);
        const double d = gbb - gaa;
        const double h2 = fma(d, d, 4.0 * g2);
        double r;
        if (h2 > 1e-280 && h2 < 1e280) r = rsqrt_refined(h2);
        else r = 1.0 / sqrt(h2);
        const double c2 = fma(0.5 * fabs(d), r, 0.5);
        const double k = rsqrt_refined(c2);
        const double f = (d >= 0.0 ? r : -r) * k;
        j.sx = f * gab.x;
        j.sy = f * gab.y;
        const double c0 = c2 * k;
        j.c = fma(0.5 * k, fma(-j.sy, j.sy, fma(-j.sx, j.sx, fma(-c0, c0, 1.0))), c0);
        const double tm = f * k * g2;
        j.naa = gaa - tm;
        j.nbb = gbb + tm;
    }
    return j;
}

// A sweep all of whose rotations were below 1e-8 is the last one: convergence is quadratic, and
// what it leaves is tested on a fresh Gram anyway (24 columns: 193 -> 183 us without the sweep
// that found nothing).
constexpr double JAC16_LAST = 1e-16;  // squared

// From G (upper blocks in sh.g[0]) to the pair's unitary Q in
// sh.q: exact-Hermitian G, convergence test, one cyclic sweep of a two-sided Jacobi
// eigensolver, eigenpair order in the first sweeps.  Returns whether the pair rotates (the
// same for every thread).  Waves 0..3 own the 2 × 2 blocks of G at (row pair pb, column
// pair qb), waves 4..7 those of Q (rows 2 pb, 2 pb + 1), pb one per 16 lanes and qb rotated
// by pb so that the first of the 16 owns the diagonal block: every thread forms its column
// pair's rotation from the round's G, the row pair's is a broadcast from that lane.  G
// alternates between two buffers, so one barrier ends a round; Q's rows stay within a wave.
// cross: only the 16 × 16 pairs between the two blocks, in 16 rounds instead of 31.  The
// pairs inside a block meet in every round of a sweep; once the sorting sweeps are over
// they need a rotation once a sweep (in its first round), as in elementwise Jacobi.  (A
// model of the schedule: 180 columns 8 sweeps either way, 512 columns 7 either way, 64
// columns 7 instead of 6.)
__device__ __forceinline__ bool jac16_eig(const JacItem& it, Jac16Shared& sh, double fro2, int bi, int bj, int sort,
                                          bool cross, int max_inner, int mode, int own) {
    constexpr int BC = 32, B = 16;
    const int tid = threadIdx.x;
    const double tol2 = it.tol * it.tol;
    // columns at or below the rounding floor are frozen (treated as zero)
    const double gfloor = it.floor_rel2 * fro2;
    // G exactly Hermitian, so that every test below sees the same value for (i, j)
    for (int e = tid; e < BC * BC; e += J16_NT) {
        const int i = e / BC, j = e % BC;
        if (i > j) continue;
        if (i == j) sh.g[0][i][i].y = 0.0;
        else sh.g[0][j][i] = cconj(sh.g[0][i][j]);
        sh.q[i][j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
        if (i != j) sh.q[j][i] = cz();
    }
    if (tid == 0) sh.flag = 0;
    __syncthreads();
    bool bad = false;
    for (int e = tid; e < BC * BC; e += J16_NT) {
        const int i = e / BC, j = e % BC;
        if (i < j) bad = bad || needs_rotation(sh.g[0][i][i].x, sh.g[0][j][j].x, sh.g[0][i][j], tol2, gfloor);
    }
    if (bad) sh.flag = 1;
    __syncthreads();
    if (!sh.flag) return false;
    __syncthreads();  // (the flag is cleared below)

    // the eigensolver and the sort are a latency-bound chain; their waves get issue
    // priority over the co-resident workgroup's products
    __builtin_amdgcn_s_setprio(2);
    // A pair that rotates takes along what lies below the target, down to the Gram's rounding
    // noise (a sixteenth of it): the rotations cost nothing more, and the last ones leave
    // the vectors as orthogonal as their Gram can tell (a truncated 32 × 32 product 3e-15
    // instead of 7e-15 off).
    // one block pair per matrix: solve the block exactly; otherwise an approximate
    // diagonaliser suffices (the outer sweeps re-check every pair on fresh Grams)
    const int inner_cap = (it.nb == 2) ? 12 : max_inner;
    // (and a single pair has only its q columns, the first slots: q - 1 rounds)
    const int nx = it.nb == 2 ? max(2, it.q + (it.q & 1)) : BC, np = nx / 2;
    const bool gown = wave_index() < 4;
    const int li = tid & 15;
    const int pb = (tid & 255) >> 4, qb = li + pb < np ? li + pb : li + pb - np;
    const bool on = li < np && pb < np;
    double2 (*gA)[J16_LP] = sh.g[0];  // G at the start of the round
    double2 (*gB)[J16_LP] = sh.g[1];  // G after the round
    bool rotated = false;
#pragma unroll 1
    for (int sweep = 0; sweep < inner_cap; ++sweep) {
        if (tid == 0) sh.flag = sh.more = 0;
        __syncthreads();
        // the round's pairs, advanced from round to round without the modulo
        int ap, bp, aq, bq;
        if (cross) {
            ap = pb;
            bp = 16 + pb;
            aq = qb;
            bq = 16 + qb;
        } else {
            rr_pair(0, on ? pb : 0, nx, ap, bp);
            rr_pair(0, on ? qb : 0, nx, aq, bq);
        }
        const int rounds = cross ? 16 : nx - 1;
#pragma unroll 1
        for (int rnd = 0; rnd < rounds; ++rnd) {
            const double gaa = gA[aq][aq].x, gbb = gA[bq][bq].x;
            const double2 gab = gA[aq][bq];
            const JRot jq = jacobi_rot_fast(gaa, gbb, gab, tol2 * (1.0 / 256.0), gfloor);
            // (the block's reads after the rotation's: ahead of it they delay the three
            // that it waits for, 2.1k cycles a round instead of 1.95k)
            __builtin_amdgcn_sched_barrier(0);
            double2 m00, m01, m10, m11;
            if (gown) {
                m00 = gA[ap][aq]; m01 = gA[ap][bq]; m10 = gA[bp][aq]; m11 = gA[bp][bq];
            } else {
                m00 = sh.q[2 * pb][aq]; m01 = sh.q[2 * pb][bq];
                m10 = sh.q[2 * pb + 1][aq]; m11 = sh.q[2 * pb + 1][bq];
            }
            // columns: x_a' = c x_a - s conj(e) x_b ; x_b' = s e x_a + c x_b (without a
            // branch: c = 1, s = 0 where the pair does not rotate)
            rot_cols(m00, m01, jq);
            rot_cols(m10, m11, jq);
            if (gown) {
                JRot jp;  // the row pair's rotation: lane 0 of the 16 owns the diagonal block
                jp.c = row_bcast0(jq.c);
                jp.sx = row_bcast0(jq.sx);
                jp.sy = row_bcast0(jq.sy);
                rot_rows(m00, m10, jp);  // rows: y_a' = c y_a - s e y_b ; y_b' = s conj(e) y_a + c y_b
                rot_rows(m01, m11, jp);
                if (li == 0 && on) {
                    if (rotates(jq)) {  // the diagonal block becomes diag(λ_a, λ_b)
                        m00 = make_double2(jq.naa, 0.0);
                        m11 = make_double2(jq.nbb, 0.0);
                        m01 = cz();
                        m10 = cz();
                        if (needs_rotation(gaa, gbb, gab, tol2, gfloor)) sh.flag = 1;
                        if (needs_rotation(gaa, gbb, gab, JAC16_LAST, gfloor)) sh.more = 1;
                    }
                }
                if (on) {
                    gB[ap][aq] = m00; gB[ap][bq] = m01; gB[bp][aq] = m10; gB[bp][bq] = m11;
                }
            } else if (on) {
                sh.q[2 * pb][aq] = m00; sh.q[2 * pb][bq] = m01;
                sh.q[2 * pb + 1][aq] = m10; sh.q[2 * pb + 1][bq] = m11;
            }
            if (cross) {
                bp = 16 + ((bp + 1) & 15);
                bq = 16 + ((bq + 1) & 15);
            } else {
                rr_next(on ? pb : 0, nx, ap, bp);
                rr_next(on ? qb : 0, nx, aq, bq);
            }
            __syncthreads();
            double2 (*gt)[J16_LP] = gA;
            gA = gB;
            gB = gt;
        }
        const int any = sh.flag, more = sh.more;
        __syncthreads();
        if (!any) break;
        rotated = true;
        if (sweep == 0 && tid == 0) {  // counted only if a rotation happened
            atomicAdd(it.rot, 1);
            if (mode == JAC_ROUND) atomicAdd(&it.own[own % 5], 1);
        }
        if (!more) break;
    }

    // order eigenpairs: larger eigenvalues to the lower block (de Rijk-style sorting; valid
    // columns only, invalid positions keep e_j).  Used in the first sweeps only: afterwards
    // the plain cyclic ordering finishes with its usual quadratic convergence (sorting in a
    // parallel ordering can lock into a cycle).  A rank sort by ballots, four columns per
    // wave: the valid positions are taken in slot order (the block with the lower index
    // first) and position k of that order receives the column of the k-th largest
    // eigenvalue, ties kept in slot order.
    if (sort) {
        const int lane = tid & 63, wv = wave_index();
        const int lo = min(bi, bj), hi = max(bi, bj), first = (bi < bj) ? 0 : B;
        const int nlo = min(B, max(0, it.q - B * lo)), nhi = min(B, max(0, it.q - B * hi));
        auto order = [&](int u) {  // slot -> place in slot order, -1 if the column is absent
            const bool in_lo = (u < B) == (first == 0);
            const int k = u & (B - 1);
            return in_lo ? (k < nlo ? k : -1) : (k < nhi ? nlo + k : -1);
        };
        auto slot_of = [&](int o) { return o < nlo ? first + o : (B - first) + o - nlo; };
        auto key_of = [&](int u) {
            const double x = gA[u][u].x;  // the eigensolver's final G
            return (x == x) ? x : -INFINITY;  // a total order even with NaN
        };
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int i = 4 * wv + 2 * t + (lane >> 5), v = lane & 31;
            const int oi = order(i), ov = order(v);
            const double ki = key_of(i), kv = key_of(v);
            const unsigned long long m = __ballot(ov >= 0 && (kv > ki || (kv == ki && ov < oi)));
            const int rank = __popc((unsigned)(lane < 32 ? m : m >> 32));
            if (v == 0) sh.perm[oi >= 0 ? slot_of(rank) : i] = i;
        }
        __syncthreads();
        double2 k0 = sh.q[tid >> 5][sh.perm[tid & 31]], k1 = sh.q[16 + (tid >> 5)][sh.perm[tid & 31]];
        __syncthreads();
        sh.q[tid >> 5][tid & 31] = k0;
        sh.q[16 + (tid >> 5)][tid & 31] = k1;
        __syncthreads();
    } else if (!rotated) {
        return false;  // Q = I
    }
    __builtin_amdgcn_s_setprio(0);
    return true;
}

// X_IJ <- X_IJ Q (and V_IJ <- V_IJ Q where the item keeps V) for the 16-row tiles k = k0,
// k0 + step, ... < k1 of X (tiles [0, kx), kx = ceil(p / 16)) followed by V, one wave per
// tile, on the matrix cores: a tile times Q's two 16-column tiles, a complex product as
// three real ones: P1 = Xr Qr, P2 = Xi Qi, P3 = (Xr + Xi)(Qr + Qi); re = P1 - P2,
// im = P3 - P1 - P2.  Operand lanes: A[l % 16][l / 16], B[l / 16][l % 16]; result register
// q of lane l is D[l / 16 + 4 q][l % 16].  The wave reads and writes only its own rows, Q
// is read-only in LDS, so no barrier; each operand register takes its load for the next
// tile as soon as it is multiplied.  Loads are unconditional: a row past the end or an absent column reads an element in range --
// absent columns meet zero rows of Q (their positions keep e_j), rows past the end are not
// stored.
__device__ __forceinline__ void jac16_update(const JacItem& it, const int* sCol, const double2 (*sQ)[J16_LP], int k0,
                                             int step, int k1) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int p = it.p, kx = (p + 15) / 16;
    if (k0 >= k1) return;
    // the wave's columns, as element offsets per row count (X and V differ in it)
    int col[8];
#pragma unroll
    for (int st = 0; st < 8; ++st) col[st] = max(sCol[4 * st + lk], 0);
    const int gc0 = sCol[li], gc1 = sCol[16 + li];
    double2 x[8];
    auto row_of = [&](int k) {
        const bool isv = k >= kx;
        return min((isv ? k - kx : k) * 16 + li, (isv ? it.q : p) - 1);
    };
    auto load = [&](int st, int k) {
        const bool isv = k >= kx;
        return gload(isv ? it.v : it.x, (size_t)row_of(k) + (size_t)(isv ? it.q : p) * col[st]);
    };
#pragma unroll
    for (int st = 0; st < 8; ++st) x[st] = load(st, k0);
#pragma unroll 1
    for (int k = k0; k < k1; k += step) {
        const bool more = k + step < k1;
        f64x4 accP[2], accQ[2], accS[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) accP[b] = accQ[b] = accS[b] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int st = 0; st < 8; ++st) {
            // (each step's Q reads stay in their step: hoisted they take 64 registers)
            __builtin_amdgcn_sched_barrier(0);
            const double2 xa = x[st];
            if (more) x[st] = load(st, k + step);
            double2 qb[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) qb[b] = sQ[4 * st + lk][16 * b + li];
            const double xs = xa.x + xa.y;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const double qs = qb[b].x + qb[b].y;
                accP[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.x, qb[b].x, accP[b], 0, 0, 0);
                accQ[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.y, qb[b].y, accQ[b], 0, 0, 0);
                accS[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, qs, accS[b], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        const bool isv = k >= kx;
        double2* base = isv ? it.v : it.x;
        const int rows = isv ? it.q : p;
        const int r0 = (isv ? k - kx : k) * 16 + lk;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int gc = b ? gc1 : gc0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int grow = r0 + 4 * q;
                if (gc >= 0 && grow < rows)
                    gstore(base, grow + (size_t)rows * gc,
                           make_double2(accP[b][q] - accQ[b][q], accS[b][q] - accP[b][q] - accQ[b][q]));
            }
        }
    }
}
__device__ __forceinline__ int jac16_tiles(const JacItem& it) {
    return (it.p + 15) / 16 + (it.v ? (it.q + 15) / 16 : 0);
}

// the pair of a round (or, in JAC_PAIRS mode, the tile's explicit pair: bi | bj << 16)
struct Jac16Pair {
    int round, own, sort, bi, bj;
    bool cross, go;
};
// go: whether the pair runs (round_gate; record: this launch records its decisions)
__device__ __forceinline__ Jac16Pair jac16_pair(const JacItem& it, int2 tt, int round_arg, const int* round_base,
                                                int sort_sweeps, int mode, int tail_switch, bool record) {
    // the item's state, its loads issued together
    const int conv = *((volatile int*)it.conv), ts = *((volatile int*)it.tail);
    const int off = it.own[JAC_ROUND_OFF];
    const int base = round_base ? *round_base : 0;
    Jac16Pair r{-1, 0, 0, tt.y & 0xffff, tt.y >> 16, false, conv == 0};
    if (mode != JAC_PAIRS) {
        // the round of the tournament: an argument, or the sweep's first round kept in
        // device memory plus the argument (so that a captured sweep replays with
        // advancing rounds); eigenpair sorting during this matrix's own first sweeps
        // (independent of the batch)
        const int R = it.nb - 1;
        r.round = base + round_arg - off;
        r.own = r.round / R;
        r.sort = r.round < sort_sweeps * R;
        r.cross = !r.sort && r.round % R != 0;
        rr_pair(r.round % R, tt.y, it.nb, r.bi, r.bj);
        if (r.go) r.go = round_gate(it, ts, r.round, r.own, R, tt.y, sort_sweeps, tail_switch,
                                    record && threadIdx.x == 0);
    }
    return r;
}
__device__ __forceinline__ void jac16_cols(const JacItem& it, int bi, int bj, int* sCol) {
    const int tid = threadIdx.x;
    if (tid < 32) {
        const int c = (tid < 16) ? bi * 16 + tid : bj * 16 + (tid - 16);
        sCol[tid] = (c < it.q) ? c : -1;
    }
}

// the pair's Gram by the whole workgroup, both row groups, into sh.g[0]
__device__ __forceinline__ void jac16_gram_lds(const JacItem& it, Jac16Shared& sh) {
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_index();
    Gram16 g;
    jac16_gram(it, sh.col, wv >> 2, wv & 3, g);
    // the waves' blocks meet in LDS, a group's four at a time (in the storage of G and
    // Q), and are added in wave order
    double2* buf = &sh.g[0][0][0];
    static_assert(sizeof(sh.g) + sizeof(sh.q) >= 4 * 768 * sizeof(double2), "a group's blocks fit");
    double2 t0[2], t1[2];
    for (int gr = 0; gr < 2; ++gr) {
        if ((wv >> 2) == gr) {
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    buf[(wv & 3) * 768 + 256 * b + ((lane >> 4) + 4 * q) * 16 + (lane & 15)] =
                        gram16_entry(g, b, q);
        }
        __syncthreads();
        double2 (&t)[2] = gr ? t1 : t0;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + J16_NT * u;
            if (e < 768) {
                t[u] = buf[e];
#pragma unroll
                for (int w = 1; w < 4; ++w) t[u] = cadd(t[u], buf[768 * w + e]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = tid + J16_NT * u;
        if (e < 768) jac16_put(sh, e, cadd(t0[u], t1[u]));
    }
    __syncthreads();
}

// fused form (items of up to J16_TALL rows)
__global__ __launch_bounds__(J16_NT) __attribute__((amdgpu_waves_per_eu(4))) void k_jacobi_round16(
    const JacItem* __restrict__ items, const int2* __restrict__ tiles, int round_arg,
    const int* __restrict__ round_base, int sort_sweeps, int max_inner, int mode, int tail_switch) {
    __shared__ Jac16Shared sh;
    const int tid = threadIdx.x;
    const int2 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    const double fro2 = *it.fro2;
    const Jac16Pair pr = jac16_pair(it, tt, round_arg, round_base, sort_sweeps, mode, tail_switch, true);
    if (tid == 0) sh.go = pr.go;  // (one thread's decision for all)
    jac16_cols(it, pr.bi, pr.bj, sh.col);
    __syncthreads();
    if (!sh.go) return;
    jac16_gram_lds(it, sh);
    if (jac16_eig(it, sh, fro2, pr.bi, pr.bj, pr.sort, pr.cross, max_inner, mode, pr.own))
        jac16_update(it, sh.col, sh.q, wave_index(), 8, jac16_tiles(it));
}

// Matrices of one block pair (at most 32 columns) and up to J16_TALL rows, solved in one
// launch: the Gram is formed afresh after every update until it needs no rotation (the
// rounds would launch the same work again for every solve and read the outcome back).
// sweep: the batch's.  A solve is a sweep of such a matrix, and as many as the batch's limit
// allows are run: JAC16_SOLVES in a launch, the rest in the next ones (solves: this launch's
// share; with none left the item counts as still rotating).
__global__ __launch_bounds__(J16_NT) __attribute__((amdgpu_waves_per_eu(2))) void k_jacobi_single16(
    const JacItem* __restrict__ items, const int* __restrict__ list, int sweep, int sort_sweeps, int solves) {
    __shared__ Jac16Shared sh;
    const JacItem it = items[list[blockIdx.x]];
    if (*it.conv) return;
    if (solves <= 0) {
        if (threadIdx.x == 0) *it.rot = 1;
        return;
    }
    const double fro2 = *it.fro2;
    jac16_cols(it, 0, 1, sh.col);
    __syncthreads();
    for (int solve = 0; solve < solves; ++solve) {
        jac16_gram_lds(it, sh);
        if (!jac16_eig(it, sh, fro2, 0, 1, sweep + solve < sort_sweeps, false, 1, JAC_ROUND, 0)) {
            if (threadIdx.x == 0) *it.conv = 1;
            return;
        }
        jac16_update(it, sh.col, sh.q, wave_index(), 8, jac16_tiles(it));
        __syncthreads();  // (the next Gram reads every wave's rows, and G and Q are reused)
    }
}

// split form: the Gram of a tile's row group (map: tile, group, partial sum's slot), four
// waves adding in order; 3 × 256 values per slot
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_jacobi_gram16(
    const JacItem* __restrict__ items, const int2* __restrict__ tiles, const int4* __restrict__ map, int round_arg,
    const int* __restrict__ round_base, int sort_sweeps, int mode, int tail_switch, cplx* __restrict__ part) {
    __shared__ double2 sP[4][3][256];
    __shared__ int sCol[32];
    __shared__ int sGo;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_index();
    const int4 mp = map[blockIdx.x];
    const int2 tt = tiles[mp.x];
    const JacItem it = items[tt.x];
    // (the gate's decision is recorded by the eigensolver's launch)
    const Jac16Pair pr = jac16_pair(it, tt, round_arg, round_base, sort_sweeps, mode, tail_switch, false);
    if (tid == 0) sGo = pr.go;
    jac16_cols(it, pr.bi, pr.bj, sCol);
    __syncthreads();
    if (!sGo) return;
    Gram16 g;
    jac16_gram(it, sCol, mp.y, wv, g);
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) sP[wv][b][((lane >> 4) + 4 * q) * 16 + (lane & 15)] = gram16_entry(g, b, q);
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        double2 v = sP[0][b][tid];
#pragma unroll
        for (int w = 1; w < 4; ++w) v = cadd(v, sP[w][b][tid]);
        gstore(part, (size_t)mp.z * 768 + 256 * b + tid, v);
    }
}
// the eigensolver of every tile: slots info[tile].x .. + info[tile].y - 1 added in order; Q and
// a flag (rotates, bi, bj) for the update
__global__ __launch_bounds__(J16_NT) __attribute__((amdgpu_waves_per_eu(2))) void k_jacobi_eig16(
    const JacItem* __restrict__ items, const int2* __restrict__ tiles, const int2* __restrict__ info, int round_arg,
    const int* __restrict__ round_base, int sort_sweeps, int max_inner, int mode, int tail_switch,
    const cplx* __restrict__ part, cplx* __restrict__ qout, int4* __restrict__ hdr) {
    __shared__ Jac16Shared sh;
    const int tid = threadIdx.x;
    const int2 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    const double fro2 = *it.fro2;
    const Jac16Pair pr = jac16_pair(it, tt, round_arg, round_base, sort_sweeps, mode, tail_switch, true);
    if (tid == 0) {
        sh.go = pr.go;
        hdr[blockIdx.x] = make_int4(0, pr.bi, pr.bj, 0);
    }
    jac16_cols(it, pr.bi, pr.bj, sh.col);
    __syncthreads();
    if (!sh.go) return;
    const int2 in = info[blockIdx.x];
    for (int e = tid; e < 768; e += J16_NT) {
        const size_t at = (size_t)in.x * 768 + e;
        double2 v = gload(part, at);
        for (int k = 1; k < in.y; ++k) v = cadd(v, gload(part, at + (size_t)768 * k));
        jac16_put(sh, e, v);
    }
    __syncthreads();
    if (!jac16_eig(it, sh, fro2, pr.bi, pr.bj, pr.sort, pr.cross, max_inner, mode, pr.own)) return;
    for (int e = tid; e < 1024; e += J16_NT) gstore(qout, (size_t)blockIdx.x * 1024 + e, sh.q[e >> 5][e & 31]);
    if (tid == 0) hdr[blockIdx.x].x = 1;
}
// the update of a tile's row chunk (map: tile, first 16-row tile, end)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_jacobi_update16(
    const JacItem* __restrict__ items, const int2* __restrict__ tiles, const int4* __restrict__ map,
    const cplx* __restrict__ qin, const int4* __restrict__ hdr) {
    __shared__ double2 sQ[32][J16_LP];
    __shared__ int sCol[32];
    const int tid = threadIdx.x;
    const int4 mp = map[blockIdx.x];
    const int4 h = hdr[mp.x];
    if (h.x == 0) return;
    const JacItem it = items[tiles[mp.x].x];
    jac16_cols(it, h.y, h.z, sCol);
    for (int e = tid; e < 1024; e += 256) sQ[e >> 5][e & 31] = gload(qin, (size_t)mp.x * 1024 + e);
    __syncthreads();
    jac16_update(it, sCol, sQ, mp.y + wave_index(), 4, mp.z);
}

// ---------------------------------------------------------------------------
// Block width 8: 16-column pairs, four waves, on the vector ALUs.
// ---------------------------------------------------------------------------
// CHECK: the test of every (round, pair) of a sweep in one launch, without rotating (its
// own kernel, so that profiles and the round timings keep the rounds apart)
template <bool CHECK>
__global__ __launch_bounds__(256) void k_jacobi_round8(const JacItem* __restrict__ items,
                                                       const int2* __restrict__ tiles, int round_arg,
                                                       const int* __restrict__ round_base, int sort_sweeps,
                                                       int max_inner, int mode, int* __restrict__ flags,
                                                       const int* __restrict__ flag0, int tail_switch) {
    constexpr int BC = 16;
    constexpr int B = BC / 2;
    constexpr int LP = BC + 1;
    constexpr int CH = 32;
    constexpr int S = B / 8;     // Gram sub-tile per thread and block (8 × 8 threads per wave)
    constexpr int NP = BC / 2;   // rotations per inner round
    // the update stages 128-row × 8-column panels of X through the
    // same LDS as the Gram's 32-row chunks
    constexpr int RB = 128, IC = 8;
    constexpr int SX_ELEMS = (BC * (CH + 1) > IC * (RB + 1)) ? BC * (CH + 1) : IC * (RB + 1);
    __shared__ double2 sG[BC][LP];
    __shared__ double2 sQX[BC * LP + SX_ELEMS];
    double2 (*sQ)[LP] = reinterpret_cast<double2 (*)[LP]>(sQX);
    double2* sXraw = sQX + BC * LP;
    double2 (*sX)[CH + 1] = reinterpret_cast<double2 (*)[CH + 1]>(sXraw);
    __shared__ int sCol[BC];
    __shared__ int sPerm[BC];
    __shared__ int sSlot[BC], sOrd[BC];
    __shared__ double sKey[BC];
    __shared__ int sFlag;
    __shared__ int sGo;

    const int tid = threadIdx.x;
    const int2 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    if (*((volatile int*)it.conv)) return;
    const int R = it.nb - 1;
    const double tol2 = it.tol * it.tol;
    const double floor_rel2 = it.floor_rel2;
    int round, sort, bi, bj, own = 0;
    if (tid == 0) sGo = 1;
    if (mode == JAC_PAIRS) {
        // an explicit block pair (tile: item, bi | bj << 16), no sorting
        round = -1;
        sort = 0;
        bi = tt.y & 0xffff;
        bj = tt.y >> 16;
    } else if (CHECK) {
        // every (round, pair) of a sweep in one launch (tile: item, round · nb/2 + pair)
        const int np = it.nb / 2;
        round = tt.y / np;
        sort = 0;
        rr_pair(round, tt.y % np, it.nb, bi, bj);
    } else {
        // the round of the tournament: an argument, or the sweep's first round kept in
        // device memory plus the argument (so that a captured sweep replays with
        // advancing rounds); eigenpair sorting during this matrix's own first sweeps
        // (independent of the batch)
        round = (round_base ? *round_base + round_arg : round_arg) - it.own[JAC_ROUND_OFF];
        own = round / R;
        sort = round < sort_sweeps * R;
        rr_pair(round % R, tt.y, it.nb, bi, bj);
        // (the item's tail state may be set by its workgroup 0 during this launch;
        // counted per own sweep, the decision does not depend on the rest of the batch)
        if (tid == 0) sGo = round_gate(it, *((volatile int*)it.tail), round, own, R, tt.y, sort_sweeps, tail_switch, true);
    }
    if (tid < BC) {
        const int c = (tid < B) ? bi * B + tid : bj * B + (tid - B);
        sCol[tid] = (c < it.q) ? c : -1;
    }
    __syncthreads();
    if (!sGo) return;

    const int p = it.p;
    // columns at or below the rounding floor are frozen (treated as zero)
    const double gfloor = floor_rel2 * (*it.fro2);
    // ---------------- Gram matrix ----------------
    const int lane = tid & 63, wv = tid >> 6;
    const int ti = lane & 7, tj = lane >> 3;
    // G = [[G11, G12], [G12^H, G22]] over the two column blocks: only G11, G12 and
    // G22 are accumulated (3/4 of the products); G21 comes from G12 below
    double2 acc11[S][S], acc12[S][S], acc22[S][S];
#pragma unroll
    for (int a = 0; a < S; ++a)
#pragma unroll
        for (int b = 0; b < S; ++b) acc11[a][b] = acc12[a][b] = acc22[a][b] = cz();

    // chunk loads are software-pipelined: chunk k+1 is fetched into registers
    // while chunk k is reduced from LDS
    constexpr int LPT = BC * CH / 256;  // elements per thread per chunk
    double2 pre[LPT];
    auto fetch = [&](const double2* base, int rows, int row0) {
#pragma unroll
        for (int s2 = 0; s2 < LPT; ++s2) {
            const int e = tid + 256 * s2;
            const int c = e / CH, rr = e % CH;
            const int gc = sCol[c], grow = row0 + rr;
            pre[s2] = ld_or_zero(base, grow + (size_t)rows * gc, gc >= 0 && grow < rows);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int s2 = 0; s2 < LPT; ++s2) {
            const int e = tid + 256 * s2;
            sX[e / CH][e % CH] = pre[s2];
        }
    };
    {
        fetch(it.x, p, 0);
        for (int row0 = 0; row0 < p; row0 += CH) {
            stash();
            __syncthreads();
            if (row0 + CH < p) fetch(it.x, p, row0 + CH);
    #pragma unroll 2
            for (int rr = wv; rr < CH; rr += 4) {
                double2 x1i[S], x1j[S], x2i[S], x2j[S];
    #pragma unroll
                for (int a = 0; a < S; ++a) {
                    x1i[a] = sX[ti * S + a][rr];
                    x1j[a] = sX[tj * S + a][rr];
                    x2i[a] = sX[B + ti * S + a][rr];
                    x2j[a] = sX[B + tj * S + a][rr];
                }
    #pragma unroll
                for (int a = 0; a < S; ++a)
    #pragma unroll
                    for (int b = 0; b < S; ++b) {
                        acc11[a][b] = cfmac(x1i[a], x1j[b], acc11[a][b]);
                        acc12[a][b] = cfmac(x1i[a], x2j[b], acc12[a][b]);
                        acc22[a][b] = cfmac(x2i[a], x2j[b], acc22[a][b]);
                    }
            }
            __syncthreads();
        }
        for (int w = 0; w < 4; ++w) {
            if (wv == w) {
    #pragma unroll
                for (int a = 0; a < S; ++a)
    #pragma unroll
                    for (int b = 0; b < S; ++b) {
                        double2& g11 = sG[ti * S + a][tj * S + b];
                        double2& g12 = sG[ti * S + a][B + tj * S + b];
                        double2& g22 = sG[B + ti * S + a][B + tj * S + b];
                        g11 = (w == 0) ? acc11[a][b] : cadd(g11, acc11[a][b]);
                        g12 = (w == 0) ? acc12[a][b] : cadd(g12, acc12[a][b]);
                        g22 = (w == 0) ? acc22[a][b] : cadd(g22, acc22[a][b]);
                    }
            }
            __syncthreads();
        }
    }

    // make G exactly Hermitian so that every test below sees the same value for (i, j)
    for (int e = tid; e < BC * BC; e += 256) {
        const int i = e / BC, j = e % BC;
        if (i > j) sG[i][j] = cconj(sG[j][i]);
        else if (i == j) sG[i][i].y = 0.0;
    }
    __syncthreads();

    // ---------------- convergence test ----------------
    if (tid == 0) sFlag = 0;
    __syncthreads();
    for (int e = tid; e < BC * BC; e += 256) {
        const int i = e / BC, j = e % BC;
        if (i < j) {
            const double gii = sG[i][i].x, gjj = sG[j][j].x;
            const double2 g = sG[i][j];
            if (needs_rotation(gii, gjj, g, tol2, gfloor)) sFlag = 1;
        }
    }
    __syncthreads();
    if constexpr (CHECK) {  // the test's outcome only
        if (tid == 0) flags[flag0[tt.x] + tt.y] = sFlag;
        return;
    }
    if (!sFlag) return;

    // the eigensolver and the sort are a latency-bound chain; their waves get issue
    // priority over the co-resident workgroups' streaming Gram and update phases
    __builtin_amdgcn_s_setprio(2);

    // ---------------- EVD of G by cyclic Jacobi ----------------
    // A round applies NP disjoint rotations.  Thread (pb, qb) owns the 2×2 block of G
    // at (row pair pb, column pair qb) and the 2×2 block of Q at rows {2pb, 2pb+1} ×
    // column pair qb.  It derives both rotations from the round's starting G, forms
    // J_pb^H (G_blk J_qb) and Q_blk J_qb in registers and writes them back: G into the
    // other of two buffers (sG and the idle staging area, every entry every round), so
    // one barrier per round separates a round's reads from the next round's writes;
    // Q in place, since rows 2pb, 2pb+1 belong to the NP threads of one wave (whose
    // LDS operations execute in order).
    for (int e = tid; e < BC * BC; e += 256) {
        const int i = e / BC, j = e % BC;
        sQ[i][j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
    }
    __syncthreads();
    // one block pair per matrix: solve the block exactly; otherwise an approximate
    // diagonaliser suffices (the outer sweeps re-check every pair on fresh Grams)
    const int inner_cap = (it.nb == 2) ? 12 : max_inner;
    static_assert((NP * NP) % 64 == 0, "block owners must fill whole waves");
    const bool owner = tid < NP * NP;
    const int pb = tid / NP, qb = tid % NP;
    static_assert(SX_ELEMS >= BC * LP, "the staging area holds the second G buffer");
    double2 (*gA)[LP] = sG;                                       // G at the start of the round
    double2 (*gB)[LP] = reinterpret_cast<double2 (*)[LP]>(sXraw);  // G after the round
#pragma unroll 1
    for (int sweep = 0; sweep < inner_cap; ++sweep) {
        if (tid == 0) sFlag = 0;
        __syncthreads();
        // the round's pairs, advanced from round to round without the modulo
        int ap, bp, aq, bq;
        rr_pair(0, pb, BC, ap, bp);
        rr_pair(0, qb, BC, aq, bq);
#pragma unroll 1
        for (int rnd = 0; rnd < BC - 1; ++rnd) {
            if (owner) {
                // each lane solves its column pair; the row pair's rotation comes from
                // the lane of the same wave that owns diagonal block (pb, pb)
                const JRot jq = jacobi_rot(gA[aq][aq].x, gA[bq][bq].x, gA[aq][bq], tol2, gfloor);
                // (whole waves are owners or not, so every lane of the wave shuffles)
                const int src = (pb % (64 / NP)) * NP + pb;
                JRot jp;
                jp.c = __shfl(jq.c, src, 64);
                jp.sx = __shfl(jq.sx, src, 64);
                jp.sy = __shfl(jq.sy, src, 64);
                if (pb == qb) jp = jq;
                double2 g00 = gA[ap][aq], g01 = gA[ap][bq], g10 = gA[bp][aq], g11 = gA[bp][bq];
                if (rotates(jq)) {  // columns:  x_a' = c x_a - s conj(e) x_b ;  x_b' = s e x_a + c x_b
                    double2 q00 = sQ[2 * pb][aq], q01 = sQ[2 * pb][bq];
                    double2 q10 = sQ[2 * pb + 1][aq], q11 = sQ[2 * pb + 1][bq];
                    rot_cols(g00, g01, jq);
                    rot_cols(g10, g11, jq);
                    rot_cols(q00, q01, jq);
                    rot_cols(q10, q11, jq);
                    sQ[2 * pb][aq] = q00; sQ[2 * pb][bq] = q01; sQ[2 * pb + 1][aq] = q10; sQ[2 * pb + 1][bq] = q11;
                }
                if (rotates(jp)) {
                    if (pb == qb) {  // the diagonal block becomes diag(λ_a, λ_b)
                        g00 = make_double2(jp.naa, 0.0);
                        g11 = make_double2(jp.nbb, 0.0);
                        g01 = cz();
                        g10 = cz();
                    } else {  // rows:  y_a' = c y_a - s e y_b ;  y_b' = s conj(e) y_a + c y_b
                        rot_rows(g00, g10, jp);
                        rot_rows(g01, g11, jp);
                    }
                }
                gB[ap][aq] = g00; gB[ap][bq] = g01; gB[bp][aq] = g10; gB[bp][bq] = g11;
                if (pb == qb && rotates(jp)) sFlag = 1;
            }
            rr_next(pb, BC, ap, bp);
            rr_next(qb, BC, aq, bq);
            __syncthreads();
            double2 (*gt)[LP] = gA;
            gA = gB;
            gB = gt;
        }
        const int any = sFlag;
        __syncthreads();
        if (!any) break;
        if (sweep == 0 && tid == 0) {  // counted only if a rotation happened
            atomicAdd(it.rot, 1);
            if (mode == JAC_ROUND) atomicAdd(&it.own[own % 5], 1);
        }
    }

    // ---------------- order eigenpairs: larger eigenvalues to the lower block ----------------
    // (de Rijk-style sorting; valid columns only, invalid positions keep e_j).  Used in the
    // first sweeps only: afterwards the plain cyclic ordering finishes with its usual
    // quadratic convergence (sorting in a parallel ordering can lock into a cycle).
    if (sort) {
    // Rank sort, one thread per column: the valid positions are taken in slot order
    // (the block with the lower index first) and position k of that order receives
    // the column of the k-th largest eigenvalue, ties kept in slot order (a stable
    // descending sort).  Invalid positions keep e_j.
    {
        const int first = (bi < bj) ? 0 : B;
        if (tid < BC) {
            int o = -1;
            double key = 0.0;
            if (sCol[tid] >= 0) {
                const bool in_first = tid >= first && tid < first + B;
                int cnt = 0;
                if (!in_first)
                    for (int u = first; u < first + B; ++u) cnt += (sCol[u] >= 0) ? 1 : 0;
                for (int u = in_first ? first : B - first; u < tid; ++u) cnt += (sCol[u] >= 0) ? 1 : 0;
                o = cnt;
                sSlot[o] = tid;
                const double x = gA[tid][tid].x;  // the eigensolver's final G
                key = (x == x) ? x : -INFINITY;  // a total order even with NaN
            } else {
                sPerm[tid] = tid;
            }
            sOrd[tid] = o;
            sKey[tid] = key;
        }
        __syncthreads();
        if (tid < BC && sOrd[tid] >= 0) {
            const int o = sOrd[tid];
            const double key = sKey[tid];
            int rank = 0;
            for (int u = 0; u < BC; ++u) {
                const int ou = sOrd[u];
                const double ku = sKey[u];
                rank += (ou >= 0 && (ku > key || (ku == key && ou < o))) ? 1 : 0;
            }
            sPerm[sSlot[rank]] = tid;
        }
    }
    __syncthreads();
    for (int e = tid; e < BC * BC; e += 256) {
        const int i = e / BC, j = e % BC;
        sX[i][j] = sQ[i][sPerm[j]];
    }
    __syncthreads();
    for (int e = tid; e < BC * BC; e += 256) {
        const int i = e / BC, j = e % BC;
        sQ[i][j] = sX[i][j];
    }
    __syncthreads();
    }

    __builtin_amdgcn_s_setprio(0);

    // ---------------- X_IJ <- X_IJ Q ,  V_IJ <- V_IJ Q ----------------
    // Register-blocked on the vector ALUs in 128-row panels: thread (rg, cg)
    // accumulates rows rg + 32a (a < RA) × columns cg·JG + b (b < JG) of a panel, so
    // every LDS value feeds RA or JG complex FMAs; the panel's X is staged IC inner
    // columns at a time (prefetched into registers one stage ahead); the sum runs over
    // i = 0..BC-1 in order.
    constexpr int JG = BC / 8;      // output columns per thread
    constexpr int RA = RB / 32;     // output rows per thread
    constexpr int UPT = IC * RB / 256;
    double2 (*sU)[RB + 1] = reinterpret_cast<double2 (*)[RB + 1]>(sXraw);
    const int rg = tid & 31, cg = tid >> 5;
    double2 upre[UPT];
    auto ufetch = [&](const double2* base, int rows, int row0, int i0) {
#pragma unroll
        for (int s2 = 0; s2 < UPT; ++s2) {
            const int e = tid + 256 * s2;
            const int gc = sCol[i0 + e / RB], grow = row0 + e % RB;
            upre[s2] = ld_or_zero(base, grow + (size_t)rows * gc, gc >= 0 && grow < rows);
        }
    };
    auto ustash = [&]() {
#pragma unroll
        for (int s2 = 0; s2 < UPT; ++s2) {
            const int e = tid + 256 * s2;
            sU[e / RB][e % RB] = upre[s2];
        }
    };
#pragma unroll 1
    for (int mat = 0; mat < (it.v ? 2 : 1); ++mat) {
        double2* base = mat ? it.v : it.x;
        const int rows = mat ? it.q : p;
        ufetch(base, rows, 0, 0);
#pragma unroll 1
        for (int row0 = 0; row0 < rows; row0 += RB) {
            double2 o[RA][JG];
#pragma unroll
            for (int a = 0; a < RA; ++a)
#pragma unroll
                for (int b = 0; b < JG; ++b) o[a][b] = cz();
#pragma unroll 1
            for (int i0 = 0; i0 < BC; i0 += IC) {
                ustash();
                __syncthreads();
                if (i0 + IC < BC) ufetch(base, rows, row0, i0 + IC);
                else if (row0 + RB < rows) ufetch(base, rows, row0 + RB, 0);
#pragma unroll 2
                for (int i = 0; i < IC; ++i) {
                    double2 xv[RA], qv[JG];
#pragma unroll
                    for (int a = 0; a < RA; ++a) xv[a] = sU[i][rg + 32 * a];
#pragma unroll
                    for (int b = 0; b < JG; ++b) qv[b] = sQ[i0 + i][cg * JG + b];
#pragma unroll
                    for (int a = 0; a < RA; ++a)
#pragma unroll
                        for (int b = 0; b < JG; ++b) o[a][b] = cfma(xv[a], qv[b], o[a][b]);
                }
                __syncthreads();
            }
#pragma unroll
            for (int a = 0; a < RA; ++a) {
                const int grow = row0 + rg + 32 * a;
#pragma unroll
                for (int b = 0; b < JG; ++b) {
                    const int gc = sCol[cg * JG + b];
                    if (gc >= 0 && grow < rows) base[grow + (size_t)rows * gc] = o[a][b];
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Block width 32: a block pair is 64 columns.  Half as many rounds per sweep as block
// width 16, so each sweep streams X and V through HBM half as often; the price is a
// 64 × 64 eigenproblem per pair (63 inner rounds).  Eight waves; G and Q take 133 KB
// of LDS, so one workgroup per CU.
// ---------------------------------------------------------------------------
// Gram tiles of one wave group (16 × 16 tiles (ti, tj), ti <= tj, of the 4 × 4 grid):
// group 0 takes (0,0) (0,1) (0,2) (0,3) (1,1), group 1 (1,2) (1,3) (2,2) (2,3) (3,3)
template <int GRP>
__device__ __forceinline__ void gram64_step(const double2 (&x)[4], f64x4 (&P)[5], f64x4 (&Q)[5], f64x4 (&S)[5]) {
    constexpr int TI[2][5] = {{0, 0, 0, 0, 1}, {1, 1, 2, 2, 3}};
    constexpr int TJ[2][5] = {{0, 1, 2, 3, 1}, {2, 3, 2, 3, 3}};
#pragma unroll
    for (int t = 0; t < 5; ++t) {
        const double2 a = x[TI[GRP][t]], b = x[TJ[GRP][t]];
        // conj(a)·b by three real products: P = ar br, Q = ai bi, S = (ar - ai)(br + bi)
        P[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, P[t], 0, 0, 0);
        Q[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, Q[t], 0, 0, 0);
        S[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x - a.y, b.x + b.y, S[t], 0, 0, 0);
    }
}
template <int GRP>
__device__ __forceinline__ void gram64_store(double2 (*sG)[65], const f64x4 (&P)[5], const f64x4 (&Q)[5],
                                             const f64x4 (&S)[5], bool first, int lane) {
    constexpr int TI[2][5] = {{0, 0, 0, 0, 1}, {1, 1, 2, 2, 3}};
    constexpr int TJ[2][5] = {{0, 1, 2, 3, 1}, {2, 3, 2, 3, 3}};
#pragma unroll
    for (int t = 0; t < 5; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * TI[GRP][t] + (lane >> 4) + 4 * q, c = 16 * TJ[GRP][t] + (lane & 15);
            const double2 g = make_double2(P[t][q] + Q[t][q], S[t][q] - P[t][q] + Q[t][q]);
            sG[r][c] = first ? g : cadd(sG[r][c], g);
        }
}

__global__ __launch_bounds__(512) void k_jacobi_round64(const JacItem* __restrict__ items,
                                                        const int2* __restrict__ tiles, int round_arg,
                                                        const int* __restrict__ round_base, int sort_sweeps,
                                                        int max_inner, int mode, int tail_switch) {
    constexpr int BC = 64, B = 32, LP = BC + 1, CH = 32, NP = 32, NT = 512;
    __shared__ double2 sG[BC][LP];
    __shared__ double2 sQ[BC][LP];
    __shared__ int sCol[BC];
    __shared__ int sPerm[BC], sSlot[BC], sOrd[BC];
    __shared__ double sKey[BC];
    __shared__ int sFlag;
    __shared__ int sGo;
    // the Gram's 32-row chunks are staged in sQ's storage (Q is initialised afterwards)
    static_assert(BC * (CH + 1) <= BC * LP, "staging fits in sQ");
    double2 (*sX)[CH + 1] = reinterpret_cast<double2 (*)[CH + 1]>(&sQ[0][0]);

    const int tid = threadIdx.x;
    const int2 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    if (*((volatile int*)it.conv)) return;
    const int R = it.nb - 1;
    const double tol2 = it.tol * it.tol;
    // the modes of k_jacobi_round: a tournament round (with the item's round offset and
    // tail gate), or an explicit block pair of the tail passes (tile: item, bi | bj << 16)
    int round = -1, sort = 0, bi, bj, own = 0;
    if (tid == 0) sGo = 1;
    if (mode == JAC_PAIRS) {
        bi = tt.y & 0xffff;
        bj = tt.y >> 16;
    } else {
        round = (round_base ? *round_base + round_arg : round_arg) - it.own[JAC_ROUND_OFF];
        own = round / R;
        sort = round < sort_sweeps * R;
        rr_pair(round % R, tt.y, it.nb, bi, bj);
        if (tid == 0) sGo = round_gate(it, *((volatile int*)it.tail), round, own, R, tt.y, sort_sweeps, tail_switch, true);
    }
    if (tid < BC) {
        const int c = (tid < B) ? bi * B + tid : bj * B + (tid - B);
        sCol[tid] = (c < it.q) ? c : -1;
    }
    __syncthreads();
    if (!sGo) return;
    const int p = it.p;
    const double gfloor = it.floor_rel2 * (*it.fro2);
    const int lane = tid & 63, wv = tid >> 6;

    // ---------------- Gram matrix (upper 16 × 16 tiles) ----------------
    // Wave group grp = wv / 4 owns five tiles; wave wq = wv % 4 of the group takes rows
    // wq + 4t (t < 8) of each 32-row chunk, four per step; the four partial sums of a
    // tile are added in wave order.
    {
        const int grp = wv >> 2, wq = wv & 3;
        f64x4 P[5], Qa[5], S[5];
#pragma unroll
        for (int t = 0; t < 5; ++t) P[t] = Qa[t] = S[t] = f64x4{0.0, 0.0, 0.0, 0.0};
        constexpr int LPT = BC * CH / NT;
        double2 pre[LPT];
        auto fetch = [&](int row0) {
#pragma unroll
            for (int s2 = 0; s2 < LPT; ++s2) {
                const int e = tid + NT * s2;
                const int c = e / CH, rr = e % CH;
                const int gc = sCol[c], grow = row0 + rr;
                pre[s2] = ld_or_zero(it.x, grow + (size_t)p * gc, gc >= 0 && grow < p);
            }
        };
        fetch(0);
        for (int row0 = 0; row0 < p; row0 += CH) {
#pragma unroll
            for (int s2 = 0; s2 < LPT; ++s2) {
                const int e = tid + NT * s2;
                sX[e / CH][e % CH] = pre[s2];
            }
            __syncthreads();
            if (row0 + CH < p) fetch(row0 + CH);
#pragma unroll
            for (int s4 = 0; s4 < CH / 16; ++s4) {
                const int rr = wq + 4 * (4 * s4 + (lane >> 4));
                double2 x[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) x[t] = sX[16 * t + (lane & 15)][rr];
                if (grp == 0) gram64_step<0>(x, P, Qa, S);
                else gram64_step<1>(x, P, Qa, S);
            }
            __syncthreads();
        }
        for (int w = 0; w < 4; ++w) {
            if (wq == w) {
                if (grp == 0) gram64_store<0>(sG, P, Qa, S, w == 0, lane);
                else gram64_store<1>(sG, P, Qa, S, w == 0, lane);
            }
            __syncthreads();
        }
    }
    // make G exactly Hermitian (the lower tiles were not computed)
    for (int e = tid; e < BC * BC; e += NT) {
        const int i = e / BC, j = e % BC;
        if (i > j) sG[i][j] = cconj(sG[j][i]);
        else if (i == j) sG[i][i].y = 0.0;
    }
    __syncthreads();

    // ---------------- convergence test ----------------
    if (tid == 0) sFlag = 0;
    __syncthreads();
    for (int e = tid; e < BC * BC; e += NT) {
        const int i = e / BC, j = e % BC;
        if (i < j && needs_rotation(sG[i][i].x, sG[j][j].x, sG[i][j], tol2, gfloor)) sFlag = 1;
    }
    __syncthreads();
    if (!sFlag) return;

    __builtin_amdgcn_s_setprio(2);

    // ---------------- EVD of G by cyclic Jacobi ----------------
    // Thread (pb, qb), pb = tid / 32 < 16, owns the 2 × 2 blocks of G at (row pair pb,
    // column pair qb) and (row pair pb + 16, column pair qb), and the matching rows of
    // Q.  Both row rotations come by shuffle from the lanes of the same wave that own
    // the diagonal blocks.  G is updated in place: one barrier after the round's reads,
    // one after its writes; Q's rows belong to one wave each, so Q needs none.
    for (int e = tid; e < BC * BC; e += NT) {
        const int i = e / BC, j = e % BC;
        sQ[i][j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
    }
    __syncthreads();
    const int inner_cap = (it.nb == 2) ? 12 : max_inner;
    const int pb = tid / NP, qb = tid % NP;
    const int pb2 = pb + 16;
    const int srcA = (pb & 1) * 32 + pb, srcB = srcA + 16;
#pragma unroll 1
    for (int sweep = 0; sweep < inner_cap; ++sweep) {
        if (tid == 0) sFlag = 0;
        __syncthreads();
        int ap, bp, ap2, bp2, aq, bq;
        rr_pair(0, pb, BC, ap, bp);
        rr_pair(0, pb2, BC, ap2, bp2);
        rr_pair(0, qb, BC, aq, bq);
#pragma unroll 1
        for (int rnd = 0; rnd < BC - 1; ++rnd) {
            // the blocks' G and Q entries first, so that their reads overlap the rotation
            double2 a00 = sG[ap][aq], a01 = sG[ap][bq], a10 = sG[bp][aq], a11 = sG[bp][bq];
            double2 b00 = sG[ap2][aq], b01 = sG[ap2][bq], b10 = sG[bp2][aq], b11 = sG[bp2][bq];
            double2 qa[4] = {sQ[2 * pb][aq], sQ[2 * pb][bq], sQ[2 * pb + 1][aq], sQ[2 * pb + 1][bq]};
            double2 qb2[4] = {sQ[2 * pb2][aq], sQ[2 * pb2][bq], sQ[2 * pb2 + 1][aq], sQ[2 * pb2 + 1][bq]};
            const JRot jq = jacobi_rot(sG[aq][aq].x, sG[bq][bq].x, sG[aq][bq], tol2, gfloor);
            JRot jpA, jpB;
            jpA.c = __shfl(jq.c, srcA, 64);
            jpA.sx = __shfl(jq.sx, srcA, 64);
            jpA.sy = __shfl(jq.sy, srcA, 64);
            jpB.c = __shfl(jq.c, srcB, 64);
            jpB.sx = __shfl(jq.sx, srcB, 64);
            jpB.sy = __shfl(jq.sy, srcB, 64);
            if (pb == qb) jpA = jq;
            if (pb2 == qb) jpB = jq;
            __syncthreads();
            if (rotates(jq)) {
                rot_cols(a00, a01, jq);
                rot_cols(a10, a11, jq);
                rot_cols(b00, b01, jq);
                rot_cols(b10, b11, jq);
                rot_cols(qa[0], qa[1], jq);
                rot_cols(qa[2], qa[3], jq);
                rot_cols(qb2[0], qb2[1], jq);
                rot_cols(qb2[2], qb2[3], jq);
                sQ[2 * pb][aq] = qa[0]; sQ[2 * pb][bq] = qa[1]; sQ[2 * pb + 1][aq] = qa[2]; sQ[2 * pb + 1][bq] = qa[3];
                sQ[2 * pb2][aq] = qb2[0]; sQ[2 * pb2][bq] = qb2[1];
                sQ[2 * pb2 + 1][aq] = qb2[2]; sQ[2 * pb2 + 1][bq] = qb2[3];
            }
            if (rotates(jpA)) {
                if (pb == qb) {
                    a00 = make_double2(jpA.naa, 0.0);
                    a11 = make_double2(jpA.nbb, 0.0);
                    a01 = cz();
                    a10 = cz();
                } else {
                    rot_rows(a00, a10, jpA);
                    rot_rows(a01, a11, jpA);
                }
            }
            if (rotates(jpB)) {
                if (pb2 == qb) {
                    b00 = make_double2(jpB.naa, 0.0);
                    b11 = make_double2(jpB.nbb, 0.0);
                    b01 = cz();
                    b10 = cz();
                } else {
                    rot_rows(b00, b10, jpB);
                    rot_rows(b01, b11, jpB);
                }
            }
            sG[ap][aq] = a00; sG[ap][bq] = a01; sG[bp][aq] = a10; sG[bp][bq] = a11;
            sG[ap2][aq] = b00; sG[ap2][bq] = b01; sG[bp2][aq] = b10; sG[bp2][bq] = b11;
            if ((pb == qb && rotates(jpA)) || (pb2 == qb && rotates(jpB))) sFlag = 1;
            rr_next(pb, BC, ap, bp);
            rr_next(pb2, BC, ap2, bp2);
            rr_next(qb, BC, aq, bq);
            __syncthreads();
        }
        const int any = sFlag;
        __syncthreads();
        if (!any) break;
        if (sweep == 0 && tid == 0) {  // counted only if a rotation happened
            atomicAdd(it.rot, 1);
            if (mode == JAC_ROUND) atomicAdd(&it.own[own % 5], 1);
        }
    }

    // ---------------- order eigenpairs (first sweeps only; as for block width 16) ----------------
    if (sort) {
        const int first = (bi < bj) ? 0 : B;
        if (tid < BC) {
            int o = -1;
            double key = 0.0;
            if (sCol[tid] >= 0) {
                const bool in_first = tid >= first && tid < first + B;
                int cnt = 0;
                if (!in_first)
                    for (int u = first; u < first + B; ++u) cnt += (sCol[u] >= 0) ? 1 : 0;
                for (int u = in_first ? first : B - first; u < tid; ++u) cnt += (sCol[u] >= 0) ? 1 : 0;
                o = cnt;
                sSlot[o] = tid;
                const double x = sG[tid][tid].x;
                key = (x == x) ? x : -INFINITY;
            } else {
                sPerm[tid] = tid;
            }
            sOrd[tid] = o;
            sKey[tid] = key;
        }
        __syncthreads();
        if (tid < BC && sOrd[tid] >= 0) {
            const int o = sOrd[tid];
            const double key = sKey[tid];
            int rank = 0;
            for (int u = 0; u < BC; ++u) {
                const int ou = sOrd[u];
                const double ku = sKey[u];
                rank += (ou >= 0 && (ku > key || (ku == key && ou < o))) ? 1 : 0;
            }
            sPerm[sSlot[rank]] = tid;
        }
        __syncthreads();
        for (int e = tid; e < BC * BC; e += NT) {
            const int i = e / BC, j = e % BC;
            sG[i][j] = sQ[i][sPerm[j]];
        }
        __syncthreads();
        for (int e = tid; e < BC * BC; e += NT) {
            const int i = e / BC, j = e % BC;
            sQ[i][j] = sG[i][j];
        }
        __syncthreads();
    }

    __builtin_amdgcn_s_setprio(0);

    // ---------------- X_IJ <- X_IJ Q ,  V_IJ <- V_IJ Q  (matrix cores) ----------------
    // 128-row panels of X and then of V: wave wv owns panel rows [16 wv, 16 wv + 16)
    // times Q's four 16-column tiles; operands straight from HBM (each wave reads and
    // writes only its own rows), the next panel's sixteen loads issued before the
    // current panel's products (unconditional, in range: see the width-16 update);
    // three real products per complex tile: re = P1 - P2, im = P3 - P1 - P2.
    const int kx = (p + 127) / 128, kt = kx + (it.v ? (it.q + 127) / 128 : 0);
    auto panel_load = [&](double2 (&xall)[BC / 4], int k) {
        const bool isv = k >= kx;
        const double2* base = isv ? it.v : it.x;
        const int rows = isv ? it.q : p;
        const int rw = min((isv ? k - kx : k) * 128 + 16 * wv + (lane & 15), rows - 1);
#pragma unroll
        for (int st = 0; st < BC / 4; ++st) {
            const int c = sCol[4 * st + (lane >> 4)];
            xall[st] = gload(base, (size_t)rw + (size_t)rows * max(c, 0));
        }
    };
    auto panel_update = [&](const double2 (&xall)[BC / 4], int k) {
        f64x4 accP[4], accQ[4], accS[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) accP[b] = accQ[b] = accS[b] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int st = 0; st < BC / 4; ++st) {
            // keep each step's Q reads in their step (the loads stay in flight)
            __builtin_amdgcn_sched_barrier(0);
            const double2 xa = xall[st];
            const double xs = xa.x + xa.y;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const double2 qv = sQ[4 * st + (lane >> 4)][16 * b + (lane & 15)];
                accP[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.x, qv.x, accP[b], 0, 0, 0);
                accQ[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.y, qv.y, accQ[b], 0, 0, 0);
                accS[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, qv.x + qv.y, accS[b], 0, 0, 0);
            }
        }
        const bool isv = k >= kx;
        double2* base = isv ? it.v : it.x;
        const int rows = isv ? it.q : p;
        const int r0 = (isv ? k - kx : k) * 128 + 16 * wv + (lane >> 4);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int gc = sCol[16 * b + (lane & 15)];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int grow = r0 + 4 * q;
                if (gc >= 0 && grow < rows)
                    base[grow + (size_t)rows * gc] =
                        make_double2(accP[b][q] - accQ[b][q], accS[b][q] - accP[b][q] - accQ[b][q]);
            }
        }
    };
    double2 xa0[BC / 4], xa1[BC / 4];
    panel_load(xa0, 0);
#pragma unroll 1
    for (int k = 0; k < kt; k += 2) {
        if (k + 1 < kt) panel_load(xa1, k + 1);
        panel_update(xa0, k);
        if (k + 1 >= kt) break;
        if (k + 2 < kt) panel_load(xa0, k + 2);
        panel_update(xa1, k + 1);
    }
}

// one round, or one set of explicit pairs, at block width 16 in the form the batch runs in
static void launch_jacobi16(const JacItem* d_items, const int2* d_tiles, int ntiles, int round,
                            const int* round_base, int sort_sweeps, int max_inner, int mode, int tail_switch,
                            const Jac16Split* sp, hipStream_t s) {
    if (!sp) {
        k_jacobi_round16<<<ntiles, J16_NT, 0, s>>>(d_items, d_tiles, round, round_base, sort_sweeps, max_inner, mode,
                                                   tail_switch);
        return;
    }
    k_jacobi_gram16<<<sp->ngram, 256, 0, s>>>(d_items, d_tiles, sp->gram, round, round_base, sort_sweeps, mode,
                                              tail_switch, sp->part);
    k_jacobi_eig16<<<ntiles, J16_NT, 0, s>>>(d_items, d_tiles, sp->info, round, round_base, sort_sweeps, max_inner,
                                             mode, tail_switch, sp->part, sp->q, sp->hdr);
    k_jacobi_update16<<<sp->nupd, 256, 0, s>>>(d_items, d_tiles, sp->upd, sp->q, sp->hdr);
}
int jac16_gram_groups(int p) { return jac16_groups(p); }
void launch_jacobi_single(const JacItem* d_items, const int* d_list, int count, int sweep, int sort_sweeps,
                          int max_sweeps, hipStream_t s) {
    constexpr int JAC16_SOLVES = 20;
    if (count > 0)
        k_jacobi_single16<<<count, J16_NT, 0, s>>>(d_items, d_list, sweep, sort_sweeps,
                                                   min(JAC16_SOLVES, max_sweeps - JAC16_SOLVES * sweep));
}
void launch_jacobi_round(const JacItem* d_items, const int2* d_tiles, int ntiles, int round,
                         const int* round_base, int block, int sort_sweeps, int max_inner, int tail_switch,
                         const Jac16Split* sp, hipStream_t s) {
    if (ntiles <= 0) return;
    if (block == 8)
        k_jacobi_round8<false><<<ntiles, 256, 0, s>>>(d_items, d_tiles, round, round_base, sort_sweeps, max_inner,
                                                      JAC_ROUND, nullptr, nullptr, tail_switch);
    else if (block == 32)
        k_jacobi_round64<<<ntiles, 512, 0, s>>>(d_items, d_tiles, round, round_base, sort_sweeps, max_inner,
                                                JAC_ROUND, tail_switch);
    else
        launch_jacobi16(d_items, d_tiles, ntiles, round, round_base, sort_sweeps, max_inner, JAC_ROUND, tail_switch,
                        sp, s);
}
void launch_jacobi_check(const JacItem* d_items, const int2* d_tiles, int ntiles, int* d_flags, const int* d_flag0,
                         hipStream_t s) {
    if (ntiles <= 0) return;
    k_jacobi_round8<true><<<ntiles, 256, 0, s>>>(d_items, d_tiles, 0, nullptr, 0, 1, JAC_CHECK, d_flags, d_flag0, 0);
}
// Convergence test of whole items without rotating (block width 16 or 32): G = X^H X in
// 64 × 64 tiles of the upper triangle of 16-column blocks, one workgroup per tile, on the
// matrix cores (v_mfma_f64_16x16x4, three real products per complex block, as in the
// rounds' Gram); wave w holds the four 16 × 16 sub-tiles of row w of the tile, i.e. the
// 16-column block pairs (4·ti + w, 4·tj + b).  The column norms come from the same LDS
// chunks.  flags[first[item] + I·nb + J] is set to 1 where a column pair of the item's
// blocks I <= J (bsub = block / 16 sixteen-column blocks each) fails the rotation test
// (for I = J the pairs inside the block); the table starts at zero.  Rows are streamed in
// chunks of 16, the next chunk fetched while the current one is multiplied.
constexpr int JCT = 64, JCR = 16;
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_jacobi_check_tiles(const JacItem* __restrict__ items,
                                                            const int4* __restrict__ tiles, int* __restrict__ flags,
                                                            const int* __restrict__ first, int bsub) {
    __shared__ double2 sX[2 * JCT][JCR + 1];
    __shared__ double sN[2 * JCT];
    const int4 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int p = it.p, q = it.q;
    const int c0 = tt.y * JCT, c1 = tt.z * JCT;
    // thread tid stages rows e % JCR of column e / JCR, e = tid + 256 s (side I for the
    // columns below JCT, side J above)
    constexpr int LPT = 2 * JCT * JCR / 256;
    double2 pre[LPT];
    auto fetch = [&](int row0) {
#pragma unroll
        for (int s2 = 0; s2 < LPT; ++s2) {
            const int e = tid + 256 * s2;
            const int cl = e / JCR, r = row0 + e % JCR;
            const int col = (cl < JCT) ? c0 + cl : c1 + cl - JCT;
            pre[s2] = ld_or_zero(it.x, (size_t)min(r, p - 1) + (size_t)p * min(col, q - 1), r < p && col < q);
        }
    };
    f64x4 P[4], Q[4], S[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) P[b] = Q[b] = S[b] = f64x4{0.0, 0.0, 0.0, 0.0};
    double nrm = 0.0;  // thread tid < 2·JCT: |x|^2 of column tid of the tile pair
    fetch(0);
    for (int row0 = 0; row0 < p; row0 += JCR) {
#pragma unroll
        for (int s2 = 0; s2 < LPT; ++s2) {
            const int e = tid + 256 * s2;
            sX[e / JCR][e % JCR] = pre[s2];
        }
        __syncthreads();
        if (row0 + JCR < p) fetch(row0 + JCR);
        if (tid < 2 * JCT) {
#pragma unroll
            for (int r = 0; r < JCR; ++r) nrm += cabs2(sX[tid][r]);
        }
#pragma unroll
        for (int s4 = 0; s4 < JCR / 4; ++s4) {
            const int r = 4 * s4 + (lane >> 4);
            const double2 xa = sX[16 * wv + (lane & 15)][r];
            const double da = xa.x - xa.y;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const double2 xb = sX[JCT + 16 * b + (lane & 15)][r];
                P[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.x, xb.x, P[b], 0, 0, 0);
                Q[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa.y, xb.y, Q[b], 0, 0, 0);
                S[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(da, xb.x + xb.y, S[b], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    if (tid < 2 * JCT) sN[tid] = nrm;
    __syncthreads();
    const double tol2 = it.tol * it.tol;
    const double gfloor = it.floor_rel2 * (*it.fro2);
    const bool diag = tt.y == tt.z;
    const int n16 = it.nb * bsub;  // 16-column blocks of the item
    const int I = 4 * tt.y + wv;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int J = 4 * tt.z + b;
        if (I >= n16 || J >= n16 || (diag && b < wv)) continue;  // wave-uniform
        bool bad = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = (lane >> 4) + 4 * r, j = lane & 15;  // result register r of the lane
            if (diag && b == wv && i >= j) continue;
            const double2 g = make_double2(P[b][r] + Q[b][r], S[b][r] - P[b][r] + Q[b][r]);
            bad = bad || needs_rotation(sN[16 * wv + i], sN[JCT + 16 * b + j], g, tol2, gfloor);
        }
        const bool any = __ballot(bad) != 0;
        if (lane == 0 && any) flags[first[tt.x] + (I / bsub) * it.nb + J / bsub] = 1;
    }
}
void launch_jacobi_check_tiles(const JacItem* d_items, const int4* d_tiles, int ntiles, int* d_flags,
                               const int* d_first, int block, hipStream_t s) {
    if (ntiles <= 0) return;
    k_jacobi_check_tiles<<<ntiles, 256, 0, s>>>(d_items, d_tiles, d_flags, d_first, block / 16);
}
void launch_jacobi_pairs(const JacItem* d_items, const int2* d_tiles, int ntiles, int block, int max_inner,
                         const Jac16Split* sp, hipStream_t s) {
    if (ntiles <= 0) return;
    if (block == 32)
        k_jacobi_round64<<<ntiles, 512, 0, s>>>(d_items, d_tiles, 0, nullptr, 0, max_inner, JAC_PAIRS, 0);
    else if (block == 8)
        k_jacobi_round8<false><<<ntiles, 256, 0, s>>>(d_items, d_tiles, 0, nullptr, 0, max_inner, JAC_PAIRS, nullptr,
                                                      nullptr, 0);
    else
        launch_jacobi16(d_items, d_tiles, ntiles, 0, nullptr, 0, max_inner, JAC_PAIRS, 0, sp, s);
}

// ||X||_F^2 of every item, deterministic: each workgroup reduces one chunk into
// partial[tile]; a second pass adds an item's chunks in order.  The sum, and so the
// deflation floor, does not depend on scheduling.
__global__ __launch_bounds__(256) void k_frob2(const JacItem* __restrict__ items, const int2* __restrict__ tiles,
                                               double* __restrict__ partial) {
    __shared__ double sRed[4];
    const int2 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    const size_t total = (size_t)it.p * it.q;
    const size_t beg = (size_t)tt.y * FROB_CHUNK;
    const size_t end = beg + FROB_CHUNK < total ? beg + FROB_CHUNK : total;
    double s = 0.0;
    for (size_t e = beg + threadIdx.x; e < end; e += 256) s += cabs2(it.x[e]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sRed[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sRed[0] + sRed[1]) + (sRed[2] + sRed[3]);
}
// item i owns partial[first[i] .. first[i+1])
__global__ void k_frob2_sum(const JacItem* __restrict__ items, int count, const double* __restrict__ partial,
                            const int* __restrict__ first) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    double s = 0.0;
    for (int k = first[i]; k < first[i + 1]; ++k) s += partial[k];
    *items[i].fro2 = s;
    if (!isfinite(s)) *items[i].conv = -1;  // NaN / Inf input: never rotated, reported by the host
}
void launch_frob2(const JacItem* d_items, int count, const int2* d_tiles, int ntiles, double* partial,
                  const int* first, hipStream_t s) {
    if (count <= 0) return;
    if (ntiles > 0) k_frob2<<<ntiles, 256, 0, s>>>(d_items, d_tiles, partial);
    k_frob2_sum<<<(count + 255) / 256, 256, 0, s>>>(d_items, count, partial, first);
}

// V <- I (grid: items that keep V × columns)
__global__ void k_set_identity(const JacItem* __restrict__ items, const int2* __restrict__ tiles) {
    const int2 tt = tiles[blockIdx.x];
    const JacItem it = items[tt.x];
    const int col = tt.y;
    if (col >= it.q) return;
    for (int r = threadIdx.x; r < it.q; r += blockDim.x)
        it.v[r + (size_t)it.q * col] = make_double2(r == col ? 1.0 : 0.0, 0.0);
}
void launch_set_identity_items(const JacItem* d_items, const int2* d_tiles, int ntiles, hipStream_t s) {
    if (ntiles <= 0) return;
    k_set_identity<<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}

// After a window of rounds: an item with no rotation is converged.  remaining[0]
// receives the number of items still rotating, remaining[1] the number with
// non-finite entries.
__global__ void k_conv_update(const JacItem* __restrict__ items, int count, int* remaining, int* round_base,
                              int rounds, int first_round, int sort_sweeps, int tail_switch) {
    __shared__ int sRem, sBad, sTail;
    if (threadIdx.x == 0) sRem = sBad = sTail = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < count; i += blockDim.x) {
        const JacItem it = items[i];
        const int cv = *it.conv;
        // the window's rotation count and the tail state it ran under, for the host's
        // accounting (read back with `remaining`)
        remaining[4 + 2 * i] = *it.rot;
        remaining[4 + 2 * i + 1] = *it.tail;
        if (cv == 0) {
            // an item whose own sweep ends with the window takes the round kernel's tail
            // decision now, so that the next window does not start with it
            const int R = it.nb - 1, end = first_round + rounds - it.own[JAC_ROUND_OFF];
            if (*it.tail == 0 && *it.rot > 0 && end % R == 0 && tail_due(it, end / R, sort_sweeps, tail_switch)) {
                *it.tail = 1;
                it.own[JAC_TAIL_AT] = end / R;
            }
            if (*it.tail == 1) atomicAdd(&sTail, 1);  // waits for the tail passes
            else if (*it.rot == 0) *it.conv = 1;
            else atomicAdd(&sRem, 1);
        } else if (cv < 0) {
            atomicAdd(&sBad, 1);
        }
        *it.rot = 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        remaining[0] = sRem;
        remaining[1] = sBad;
        remaining[3] = sTail;
        if (round_base) *round_base += rounds;  // the next sweep's first round
    }
}
void launch_conv_update(const JacItem* d_items, int count, int* remaining, int* round_base, int rounds,
                        int first_round, int sort_sweeps, int tail_switch, hipStream_t s) {
    k_conv_update<<<1, 256, 0, s>>>(d_items, count, remaining, round_base, rounds, first_round, sort_sweeps,
                                    tail_switch);
}

// ---------------------------------------------------------------------------
// singular values: σ_j = ||X[:, j]||  (one wave per column)
// ---------------------------------------------------------------------------
__global__ void k_colnorms(const SelectItem* __restrict__ items, const int2* __restrict__ tiles) {
    const int2 tt = tiles[blockIdx.x];
    const SelectItem it = items[tt.x];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int col = tt.y * 4 + wv;
    if (col >= it.q) return;
    const double2* x = it.x + (size_t)it.p * col;
    double s = 0.0;
    for (int r = lane; r < it.p; r += 64) s += cabs2(x[r]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) it.sigma_sorted[col] = sqrt(s);
}

// sort descending, `truncate!` rule, renormalisation, discarded weight
constexpr int SELECT_MAXQ = 4096;
__global__ __launch_bounds__(1024) void k_select(const SelectItem* __restrict__ items) {
    __shared__ double sS[SELECT_MAXQ];
    __shared__ int sI[SELECT_MAXQ];
    __shared__ double sRed[32];
    __shared__ int sKept;
    const SelectItem it = items[blockIdx.x];
    const int tid = threadIdx.x, q = it.q;
    int n2 = 1;
    while (n2 < q) n2 <<= 1;
    for (int i = tid; i < n2; i += blockDim.x) {
        sS[i] = (i < q) ? it.sigma_sorted[i] : -1.0;
        sI[i] = (i < q) ? i : 0x7fffffff;
    }
    __syncthreads();
    for (int k = 2; k <= n2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < n2; i += blockDim.x) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const double si = sS[i], sj = sS[ixj];
                    const int ii = sI[i], ij = sI[ixj];
                    // "i before ixj" in descending order
                    const bool i_first = (si > sj) || (si == sj && ii < ij);
                    const bool desc = ((i & k) == 0);
                    if (desc != i_first) {
                        sS[i] = sj; sS[ixj] = si;
                        sI[i] = ij; sI[ixj] = ii;
                    }
                }
            }
            __syncthreads();
        }
    }
    if (tid == 0) {
        int lim = q;
        int kept = q;
        if (it.truncate) {
            if (it.maxdim >= 0 && it.maxdim < lim) lim = it.maxdim;
            kept = 0;
            while (kept < lim && fabs(sS[kept]) > it.threshold) ++kept;
        }
        sKept = kept;
    }
    __syncthreads();
    const int kept = sKept;
    // discarded weight and kept norm
    double dsc = 0.0, kn = 0.0;
    for (int i = tid; i < q; i += blockDim.x) {
        const double v = sS[i] * sS[i];
        if (i < kept) kn += v; else dsc += v;
    }
    for (int off = 32; off > 0; off >>= 1) {
        dsc += __shfl_xor(dsc, off, 64);
        kn += __shfl_xor(kn, off, 64);
    }
    const int lane = tid & 63, wv = tid >> 6;
    if (lane == 0) { sRed[wv] = dsc; sRed[16 + wv] = kn; }
    __syncthreads();
    if (tid == 0) {
        double a = 0.0, b = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) { a += sRed[w]; b += sRed[16 + w]; }
        sRed[0] = a; sRed[16] = b;
        *it.kept = kept;
        *it.discarded = sqrt(a);
    }
    __syncthreads();
    const double scale = (it.renormalize && sRed[16] > 0.0) ? 1.0 / sqrt(sRed[16]) : 1.0;
    for (int i = tid; i < q; i += blockDim.x) {
        it.sigma_sorted[i] = sS[i];
        it.perm[i] = sI[i];
        if (i < kept) it.lam_out[i] = sS[i] * scale;
    }
}

void launch_select_items(const SelectItem* d_items, const int2* d_norm_tiles, int n_norm_tiles, int count,
                         hipStream_t s) {
    if (n_norm_tiles > 0) k_colnorms<<<n_norm_tiles, 256, 0, s>>>(d_items, d_norm_tiles);
    if (count > 0) k_select<<<count, 1024, 0, s>>>(d_items);
}

// ---------------------------------------------------------------------------
// orthonormal completion of kept columns below the deflation floor
// ---------------------------------------------------------------------------
__device__ __forceinline__ double splitmix_unit(unsigned long long k) {
    k += 0x9e3779b97f4a7c15ull;
    k = (k ^ (k >> 30)) * 0xbf58476d1ce4e5b9ull;
    k = (k ^ (k >> 27)) * 0x94d049bb133111ebull;
    k ^= k >> 31;
    return (double)(k >> 11) * 0x1.0p-52 - 1.0;  // uniform in [-1, 1)
}

constexpr int COMPLETE_MAXQ = SELECT_MAXQ;
// The kept columns at or below the deflation floor (sorted positions [first, kept);
// σ sorted decreasing, so first = the number of kept σ² above the floor) are replaced
// by an orthonormal completion: deterministic pseudo-random starts, two passes of
// classical Gram-Schmidt against the columns above the floor (one workgroup per
// frozen column, all in parallel); the host then orthonormalises them among
// themselves by a Householder QR.  Sorted column i is x[:, perm[i]] / s_i with
// s_i = σ_i, or 1 where σ_i = 0.
__device__ __forceinline__ int complete_first(const CompleteItem& it, int kept, double floor2) {
    int lo = 0, hi = kept;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const double s = it.sigma_sorted[mid];
        if (s * s > floor2) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}
__device__ __forceinline__ const double2* complete_col(const CompleteItem& it, int i) {
    return it.x + (size_t)it.p * it.perm[i];
}
__device__ __forceinline__ double complete_inv(const CompleteItem& it, int i) {
    const double s = it.sigma_sorted[i];
    return s > 0.0 ? 1.0 / s : 1.0;
}
// sDot[i - i0] = <x_i, z> / s_i² for i in [i0, i1): a wave per column, four columns
// per wave in flight, lanes striding the rows
__device__ __forceinline__ void complete_dots(const CompleteItem& it, const double2* z, int i0, int i1,
                                              double2* sDot) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int i = i0 + wv; i < i1; i += 16) {
        double2 acc[4] = {cz(), cz(), cz(), cz()};
        const double2* cc[4];
        bool ok[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ok[u] = i + 4 * u < i1;
            cc[u] = complete_col(it, ok[u] ? i + 4 * u : i);
        }
        for (int r = lane; r < it.p; r += 64) {
            const double2 zr = z[r];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (ok[u]) acc[u] = cfmac(cc[u][r], zr, acc[u]);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                acc[u].x += __shfl_xor(acc[u].x, off, 64);
                acc[u].y += __shfl_xor(acc[u].y, off, 64);
            }
        if (lane == 0)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (ok[u]) {
                    const double w = complete_inv(it, i + 4 * u);
                    sDot[i + 4 * u - i0] = cscale(acc[u], w * w);
                }
    }
}
// z <- z - Σ_{i in [i0, i1)} sDot[i - i0] x_i, a thread per row
__device__ __forceinline__ void complete_update(const CompleteItem& it, double2* z, int i0, int i1,
                                                const double2* sDot) {
    for (int r = threadIdx.x; r < it.p; r += blockDim.x) {
        double2 v = z[r];
        int i = i0;
        for (; i + 4 <= i1; i += 4) {
            const double2 x0 = complete_col(it, i)[r], x1 = complete_col(it, i + 1)[r];
            const double2 x2 = complete_col(it, i + 2)[r], x3 = complete_col(it, i + 3)[r];
            v = csub(v, cmul(sDot[i - i0], x0));
            v = csub(v, cmul(sDot[i + 1 - i0], x1));
            v = csub(v, cmul(sDot[i + 2 - i0], x2));
            v = csub(v, cmul(sDot[i + 3 - i0], x3));
        }
        for (; i < i1; ++i) v = csub(v, cmul(sDot[i - i0], complete_col(it, i)[r]));
        z[r] = v;
    }
}

// phase 1, workgroup (item, j): a random start for frozen column j, orthogonalised
// twice against the columns above the floor
__global__ __launch_bounds__(256) void k_complete_project(const CompleteItem* __restrict__ items,
                                                          const int2* __restrict__ tiles) {
    __shared__ double2 sDot[COMPLETE_MAXQ];
    const int2 tt = tiles[blockIdx.x];
    const CompleteItem it = items[tt.x];
    const int j = tt.y;
    const int kept = *it.kept;
    if (j >= kept) return;
    const double floor2 = it.floor_rel2 * (*it.fro2);
    const double sj = it.sigma_sorted[j];
    if (sj * sj > floor2) return;
    const int first = complete_first(it, kept, floor2);
    double2* z = const_cast<double2*>(complete_col(it, j));
    // a deterministic pseudo-random start (the same for a matrix alone or in a batch)
    for (int r = threadIdx.x; r < it.p; r += 256) {
        const unsigned long long key = ((unsigned long long)j << 32) | (unsigned)r;
        z[r] = make_double2(splitmix_unit(2 * key), splitmix_unit(2 * key + 1));
    }
    __syncthreads();
    for (int pass = 0; pass < 2 && first > 0; ++pass) {
        complete_dots(it, z, 0, first, sDot);
        __syncthreads();
        complete_update(it, z, 0, first, sDot);
        __syncthreads();
    }
}

// per item: counts[2i] = first (the first frozen sorted position), counts[2i + 1] = kept
__global__ void k_complete_count(const CompleteItem* __restrict__ items, int count, int* __restrict__ counts) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const CompleteItem it = items[i];
    const int kept = *it.kept;
    counts[2 * i] = complete_first(it, kept, it.floor_rel2 * (*it.fro2));
    counts[2 * i + 1] = kept;
}

// frozen positions with σ below 1e-280 get σ = 0 and Λ = 0 (their completed columns are
// stored as unit vectors; the others as unit vectors times σ)
__global__ void k_complete_zero_tiny(const CompleteItem* __restrict__ items, const int* __restrict__ counts) {
    const CompleteItem it = items[blockIdx.x];
    for (int j = counts[2 * blockIdx.x] + threadIdx.x; j < counts[2 * blockIdx.x + 1]; j += blockDim.x)
        if (!(it.sigma_sorted[j] >= 1e-280)) {
            it.sigma_sorted[j] = 0.0;
            it.lam_out[j] = 0.0;
        }
}

void launch_complete_project(const CompleteItem* d_items, const int2* d_tiles, int ntiles, hipStream_t s) {
    if (ntiles > 0) k_complete_project<<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}
void launch_complete_count(const CompleteItem* d_items, int count, int* d_counts, hipStream_t s) {
    if (count > 0) k_complete_count<<<(count + 255) / 256, 256, 0, s>>>(d_items, count, d_counts);
}
void launch_complete_zero_tiny(const CompleteItem* d_items, const int* d_counts, int count, hipStream_t s) {
    if (count > 0) k_complete_zero_tiny<<<count, 256, 0, s>>>(d_items, d_counts);
}

__global__ __launch_bounds__(256) void k_scatter_cols(const ScatterItem* __restrict__ items,
                                                      const int2* __restrict__ tiles) {
    const int2 tt = tiles[blockIdx.x];
    const ScatterItem it = items[tt.x];
    const int j = tt.y;
    if (j >= *it.kept) return;
    const double sg = it.sigma_sorted[j];
    const double f = (it.mul_sigma && sg > 0.0) ? sg : 1.0;
    double2* dst = it.x + (size_t)it.p * it.perm[j];
    const double2* src = it.f + (size_t)it.ldf * j;
    for (int r = threadIdx.x; r < it.p; r += 256) dst[r] = cscale(src[r], f);
}
void launch_scatter_cols(const ScatterItem* d_items, const int2* d_tiles, int ntiles, hipStream_t s) {
    if (ntiles > 0) k_scatter_cols<<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}

// ---------------------------------------------------------------------------
// write-back of kept columns (32 × 32 tiles: j = output column, c = row of src)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_gather(const GatherItem* __restrict__ items, const int2* __restrict__ tiles) {
    __shared__ double2 sT[32][33];
    const int2 tt = tiles[blockIdx.x];
    const GatherItem g = items[tt.x];
    const int kept = *g.kept;
    const int rows_out = max(g.rows, g.zero_rows);
    const int ntc = (rows_out + 31) / 32;
    const int j0 = (tt.y / ntc) * 32, c0 = (tt.y % ntc) * 32;
    const bool fill = g.zero_rows > 0;
    if (j0 >= kept && !fill) return;
    const int tid = threadIdx.x;
    const int cc = tid & 31;
    for (int s = 0; s < 4; ++s) {
        const int jj = (tid >> 5) + 8 * s;
        const int j = j0 + jj, c = c0 + cc;
        double2 v = cz();
        if (j < kept && c < g.rows) {
            const int src_col = g.perm ? g.perm[j] : j;
            v = g.src[(g.row_src ? g.row_src[c] : c) + (size_t)g.ld_src * src_col];
            double f = 1.0;
            if (g.divide_sigma) {
                const double sg = g.sigma_sorted[j];
                f = sg > 0.0 ? 1.0 / sg : 1.0;  // σ = 0: the column holds its unit vector
            }
            if (g.rowscale) {
                const double w = g.rowscale[(c / g.rowscale_div) % g.rowscale_mod];
                f *= g.rowscale_atol >= 0.0 ? pinv_value(w, g.rowscale_atol) : w;
            }
            v = cscale(v, f);
        }
        if (!g.conj_transpose) {
            const size_t ldo = g.ld_out > 0 ? g.ld_out : g.rows;
            if (fill ? (j < g.max_cols && c < rows_out) : (j < kept && c < g.rows)) g.out[c + ldo * j] = v;
        } else {
            sT[jj][cc] = cconj(v);
        }
    }
    if (g.conj_transpose) {
        __syncthreads();
        for (int s = 0; s < 4; ++s) {
            const int c = c0 + (tid >> 5) + 8 * s;
            const int j = j0 + cc;
            if (j < kept && c < g.rows) g.out[j + (size_t)kept * c] = sT[cc][(tid >> 5) + 8 * s];
        }
    }
}
void launch_gather_items(const GatherItem* d_items, const int2* d_tiles, int ntiles, hipStream_t s) {
    if (ntiles <= 0) return;
    k_gather<<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}

}  // namespace qh
