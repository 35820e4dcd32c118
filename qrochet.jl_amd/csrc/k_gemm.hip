// Two-site contraction (θ build with fused gate, FP64 on the vector ALUs with LDS-staged
// tiles) and a batched complex FP64 GEMM on the matrix cores.
//
// θ[(l,a),(b,r)] = rs[l] cs[r] Σ_{o1,o2} G[a,b,o1,o2] Σ_m A_l[l,o1,m] λ[m] A_r[m,o2,r]
// (Qrochet `evolve_2site!`: contract!(tn, bond) then contract!(tn, gate inds),
//  src/Ansatz/Chain.jl:616,636, Vidal variant :669-685).  With the (l, o, r)
// device layout the product is a plain column-major GEMM (M = d·χl, K = χm,
// N = d·χr); a tile covers a range of l and r for *all* physical indices so the
// 4×4 gate mixes values a thread already holds.
#include "qh_kernels.h"
#include "qh_complex.h"

namespace qh {

// ---------------------------------------------------------------------------
// θ build
// ---------------------------------------------------------------------------
template <int D, int I>
__global__ __launch_bounds__(256) void k_theta_f64(const ThetaItem* __restrict__ items,
                                                   const int2* __restrict__ tiles) {
    constexpr int TL = 16 * I, TR = 16 * I, KC = 16;
    constexpr int BST = D * TR + 1;
    __shared__ double2 sA[KC][D * TL];
    __shared__ double2 sB[KC][BST];
    __shared__ double2 sG[D * D * D * D];

    const int tid = threadIdx.x;
    const int2 tt = tiles[blockIdx.x];
    const ThetaItem it = items[tt.x];
    const int l0 = (tt.y % it.tiles_l) * TL;
    const int r0 = (tt.y / it.tiles_l) * TR;
    const int chil = it.chil, chim = it.chim, chir = it.chir;
    const int lt = tid & 15, rt = tid >> 4;

    if (tid < D * D * D * D) sG[tid] = it.gate[tid];

    double2 acc[I][I][D][D];
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < I; ++j)
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int b = 0; b < D; ++b) acc[i][j][a][b] = cz();

    for (int m0 = 0; m0 < chim; m0 += KC) {
        for (int e = tid; e < KC * D * TL; e += 256) {
            const int l = e % TL, o = (e / TL) % D, kk = e / (TL * D);
            const int gl = l0 + l, gm = m0 + kk;
            double2 v = cz();
            if (gl < chil && gm < chim) {
                v = it.al[gl + (size_t)chil * (o + D * (size_t)gm)];
                if (it.lam) v = cscale(v, it.lam[gm]);
            }
            sA[kk][o * TL + l] = v;
        }
        for (int e = tid; e < KC * D * TR; e += 256) {
            const int kk = e % KC, o = (e / KC) % D, r = e / (KC * D);
            const int gr = r0 + r, gm = m0 + kk;
            double2 v = cz();
            if (gr < chir && gm < chim) v = it.ar[gm + (size_t)chim * (o + D * (size_t)gr)];
            sB[kk][o * TR + r] = v;
        }
        __syncthreads();
#pragma unroll 4
        for (int kk = 0; kk < KC; ++kk) {
            double2 av[I][D], bv[I][D];
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int o = 0; o < D; ++o) {
                    av[i][o] = sA[kk][o * TL + lt + 16 * i];
                    bv[i][o] = sB[kk][o * TR + rt + 16 * i];
                }
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int j = 0; j < I; ++j)
#pragma unroll
                    for (int a = 0; a < D; ++a)
#pragma unroll
                        for (int b = 0; b < D; ++b) acc[i][j][a][b] = cfma(av[i][a], bv[j][b], acc[i][j][a][b]);
        }
        __syncthreads();
    }

    const int m = D * chil, n = D * chir;
#pragma unroll
    for (int i = 0; i < I; ++i) {
        const int l = l0 + lt + 16 * i;
        if (l >= chil) continue;
        const double sl = it.rs ? it.rs[l] : 1.0;
#pragma unroll
        for (int j = 0; j < I; ++j) {
            const int r = r0 + rt + 16 * j;
            if (r >= chir) continue;
            const double sc = sl * (it.cs ? it.cs[r] : 1.0);
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int b = 0; b < D; ++b) {
                    double2 v = cz();
#pragma unroll
                    for (int o1 = 0; o1 < D; ++o1)
#pragma unroll
                        for (int o2 = 0; o2 < D; ++o2)
                            v = cfma(sG[a + D * b + D * D * (o1 + D * o2)], acc[i][j][o1][o2], v);
                    v = cscale(v, sc);
                    const size_t row = (size_t)l + (size_t)chil * a;
                    const size_t col = (size_t)b + (size_t)D * r;
                    if (!it.transposed)
                        it.x[row + (size_t)m * col] = v;
                    else
                        it.x[col + (size_t)n * row] = cconj(v);
                }
        }
    }
}

void launch_theta(const ThetaItem* d_items, const int2* d_tiles, int ntiles, int d, hipStream_t s) {
    if (ntiles <= 0) return;
    switch (d) {
        case 2: k_theta_f64<2, 2><<<ntiles, 256, 0, s>>>(d_items, d_tiles); break;
        case 3: k_theta_f64<3, 1><<<ntiles, 256, 0, s>>>(d_items, d_tiles); break;
        case 4: k_theta_f64<4, 1><<<ntiles, 256, 0, s>>>(d_items, d_tiles); break;
        default: break;
    }
}

int theta_tile_extent(int d) { return d == 2 ? 32 : 16; }

// ---------------------------------------------------------------------------
// batched GEMM  C = alpha op(A) diag(dk) op(B) (+ beta C), then row/col scales
// ---------------------------------------------------------------------------
// On the matrix cores (v_mfma_f64_16x16x4), four real products per complex one (the same
// error bound as scalar arithmetic), operands straight from memory into registers: a 16 × 16
// × 4 step of one wave is 4 × 64 cycles of matrix-core time for 2 KB of operands, so L1 and
// L2 keep up without LDS staging and no barrier stands between a load and its use; the
// loads of the next U steps are in flight while U are multiplied.
// A lane's operands are op(A)(m0 + l % 16, k + l / 16) and op(B)(k + l / 16, n0 + l % 16);
// the product is taken as D^T = op(B)^T op(A)^T, so result register q of lane l is
// C(m0 + l % 16, n0 + l / 16 + 4 q).
// KS = 4: the four waves of a workgroup share one (16 TI) × (16 TJ) tile and take every
// fourth K step each; their partial sums meet in LDS and are added in wave order.  A tile
// then has four waves' loads in flight whatever its size, which is what bounds the small
// products of a site sweep (90 × 180 × 90: 40 us with one 64 × 64 vector-ALU tile per
// workgroup, 7 us here), and no separate split-K launch is needed.
// KS = 1: each wave has its own tile, the workgroup's stacked along M.  For short contractions,
// 16 × 16 a wave; and, where the caller asks for it, for products with many rows, 32 × 32 a
// wave: a contraction of 64 leaves a wave of the split form four steps between its first loads
// and the sum in LDS, here 16 with the loads of four in flight (64 x 64 environments of a
// periodic chain, 4096 of them: 33 TFLOP/s split, 44 here).
// The summation order depends on the product's K alone (split from GEMM_KS_MIN on), never on
// the tile shape or the batch, but for those products with many rows.
typedef double f64x4 __attribute__((ext_vector_type(4)));

struct GemmOperand {  // element (i, k) at p[i·si + (k mod kin)·sk + (k / kin)·sk2]
    const double2* p;
    size_t si, sk, sk2;
    int kin;
};
__device__ __forceinline__ size_t gemm_koff(const GemmOperand& o, int k) {
    if (o.kin > 0) {
        const unsigned q = (unsigned)k / (unsigned)o.kin;
        return (size_t)(k - (int)q * o.kin) * o.sk + (size_t)q * o.sk2;
    }
    return (size_t)k * o.sk;
}

// PLAIN: no K scaling, and k_in (if any) a multiple of 4, so that a step's operands lie at an
// offset that is the same for all lanes, and a lane's part of the address never changes.  The loop
// is then loads and matrix instructions alone: four accumulators (ar br, ai bi, ai br, ar bi)
// whose signs -- conjugated operands -- come in at the end, and zeros past the end of K only in
// the last chunk.  (With the signs, the scaling and the zeros applied to every operand, a
// step of 1024 matrix-core cycles took 1650.)
template <int TI, int TJ, int KS, bool PLAIN>
__device__ __forceinline__ void gemm_tile_mfma(const GemmItem& g, int tile, double2* sP) {
    constexpr int U = (TI * TJ > 1) ? 2 : 4;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_index();
    const int li = lane & 15, lk = lane >> 4;
    constexpr int WM = KS == 1 ? 4 : 1;  // waves stacked along M
    constexpr int TM = 16 * TI * WM, TN = 16 * TJ;
    const int tiles_m = (g.m + TM - 1) / TM;
    const int m0 = (tile % tiles_m) * TM + (KS == 1 ? wv * 16 * TI : 0), n0 = (tile / tiles_m) * TN;

    const bool pa = op_plain(g.opa), pb = op_plain(g.opb);
    const GemmOperand A{g.a, pa ? 1 : (size_t)g.lda, pa ? (size_t)g.lda : 1, g.a_k2, g.k_in};
    const GemmOperand B{g.b, pb ? (size_t)g.ldb : 1, pb ? 1 : (size_t)g.ldb, g.b_k2, g.k_in};
    const bool ca = g.opa == GEMM_C || g.opa == GEMM_CONJ, cb = g.opb == GEMM_C || g.opb == GEMM_CONJ;
    // rows and columns past the end read the last one: their results are not stored
    size_t oa[TI], ob[TJ];
#pragma unroll
    for (int t = 0; t < TI; ++t) oa[t] = (size_t)min(m0 + 16 * t + li, g.m - 1) * A.si;
#pragma unroll
    for (int t = 0; t < TJ; ++t) ob[t] = (size_t)min(n0 + 16 * t + li, g.n - 1) * B.si;
    // the lane's part of the address of a whole step
    const double2 *la[TI], *lb[TJ];
#pragma unroll
    for (int t = 0; t < TI; ++t) la[t] = A.p + oa[t] + lk * A.sk;
#pragma unroll
    for (int t = 0; t < TJ; ++t) lb[t] = B.p + ob[t] + lk * B.sk;

    f64x4 acc[TJ][TI][4];  // sums of ar br, ai bi, ai br, ar bi
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[j][i][c] = f64x4{0.0, 0.0, 0.0, 0.0};

    const int steps = (g.k + 3) / 4;
    const int mine = KS == 1 ? steps : (steps - wv + KS - 1) / KS;  // steps wv, wv + KS, ...
    const int chunks = (mine + U - 1) / U;
    const bool dk_plain = g.dk_div == 1 && g.k + g.dk_off <= g.dk_mod;
    struct Frag {
        double2 a[U][TI], b[U][TJ];
        double f[U];
    };
    auto fetch = [&](Frag& r, int c) {
        if (PLAIN && (c + 1 < chunks || (g.k % 4 == 0 && mine % U == 0))) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = 4 * ((KS == 1 ? 0 : wv) + KS * (c * U + u));  // (the same for all lanes)
                const size_t ka = gemm_koff(A, k), kb = gemm_koff(B, k);
#pragma unroll
                for (int t = 0; t < TI; ++t) r.a[u][t] = gload(la[t], ka);
#pragma unroll
                for (int t = 0; t < TJ; ++t) r.b[u][t] = gload(lb[t], kb);
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // a step past the end multiplies zeros (both operands: no 0 · Inf)
            const int k = 4 * ((KS == 1 ? 0 : wv) + KS * (c * U + u)) + lk;
            const bool ok = c * U + u < mine && k < g.k;
            const int kc = ok ? k : 0;
            const size_t ka = gemm_koff(A, kc), kb = gemm_koff(B, kc);
#pragma unroll
            for (int t = 0; t < TI; ++t) r.a[u][t] = ld_or_zero(A.p, oa[t] + ka, ok);
#pragma unroll
            for (int t = 0; t < TJ; ++t) r.b[u][t] = ld_or_zero(B.p, ob[t] + kb, ok);
            if constexpr (!PLAIN) {
                r.f[u] = 1.0;
                if (g.dk)
                    r.f[u] = ((gconst_f64)g.dk)[dk_plain ? kc + g.dk_off : ((kc + g.dk_off) / g.dk_div) % g.dk_mod];
            }
        }
    };
    auto mult = [&](const Frag& r) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            double ar[TI], ai[TI];
#pragma unroll
            for (int t = 0; t < TI; ++t) {
                ar[t] = PLAIN ? r.a[u][t].x : r.a[u][t].x * r.f[u];
                ai[t] = PLAIN ? r.a[u][t].y : r.a[u][t].y * r.f[u];
            }
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                const double2 y = r.b[u][j];
#pragma unroll
                for (int i = 0; i < TI; ++i) {
                    f64x4(&c)[4] = acc[j][i];
                    c[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, ar[i], c[0], 0, 0, 0);
                    c[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(y.y, ai[i], c[1], 0, 0, 0);
                    c[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, ai[i], c[2], 0, 0, 0);
                    c[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(y.y, ar[i], c[3], 0, 0, 0);
                }
            }
        }
    };
    if (chunks > 0) {
        // (no exit inside the loop: the accumulators would be held twice)
        Frag f0, f1;
        fetch(f0, 0);
#pragma unroll 1
        for (int t = 0; t + 1 < chunks; t += 2) {
            fetch(f1, t + 1);
            mult(f0);
            if (t + 2 < chunks) fetch(f0, t + 2);
            mult(f1);
        }
        if (chunks & 1) mult(f0);
    }
    const double sa = ca ? -1.0 : 1.0, sb = cb ? -1.0 : 1.0, sab = -sa * sb;
    f64x4 re[TJ][TI], im[TJ][TI];
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                re[j][i][q] = fma(sab, acc[j][i][1][q], acc[j][i][0][q]);
                im[j][i][q] = fma(sa, acc[j][i][2][q], sb * acc[j][i][3][q]);
            }

    const bool use_beta = (g.beta.x != 0.0 || g.beta.y != 0.0);
    auto store = [&](int r, int c, double2 acc) {
        if (r >= g.m || c >= g.n) return;
        double2 v = cmul(g.alpha, acc);
        v = cscale(v, (g.rowscale ? g.rowscale[r] : 1.0) * (g.colscale ? g.colscale[c] : 1.0));
        const size_t at = r + (size_t)g.ldc * c;
        if (use_beta) v = cfma(g.beta, gload(g.add ? g.add : g.c, at), v);
        gstore(g.c, at, v);
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    store(m0 + 16 * i + li, n0 + 16 * j + lk + 4 * q, make_double2(re[j][i][q], im[j][i][q]));
    } else {
        constexpr int LD = TM + 1;
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sP[(wv * TN + 16 * j + lk + 4 * q) * LD + 16 * i + li] = make_double2(re[j][i][q], im[j][i][q]);
        __syncthreads();
#pragma unroll
        for (int e = tid; e < TM * TN; e += 256) {
            const int r = e % TM, c = e / TM;
            double2 v = sP[c * LD + r];
#pragma unroll
            for (int w = 1; w < KS; ++w) v = cadd(v, sP[(w * TN + c) * LD + r]);
            store(m0 + r, n0 + c, v);
        }
    }
}
template <int TI, int TJ>
constexpr int gemm_lds() { return 4 * 16 * TJ * (16 * TI + 1); }

// tile: workgroup tile of the item (gemm_tiles)
template <int T>  // 1: 16, 2: 32, or GEMM_TALL
__device__ __forceinline__ void gemm_tile(const GemmItem& g, int tile) {
    const bool plain = !g.dk && g.k_in % 4 == 0;
    if (g.k < GEMM_KS_MIN) {
        if (plain) gemm_tile_mfma<1, 1, 1, true>(g, tile, nullptr);
        else gemm_tile_mfma<1, 1, 1, false>(g, tile, nullptr);
    } else if constexpr (T == GEMM_TALL) {
        if (plain) gemm_tile_mfma<2, 2, 1, true>(g, tile, nullptr);
        else gemm_tile_mfma<2, 2, 1, false>(g, tile, nullptr);
    } else {
        __shared__ double2 sP[gemm_lds<T, T>()];
        if (plain) gemm_tile_mfma<T, T, 4, true>(g, tile, sP);
        else gemm_tile_mfma<T, T, 4, false>(g, tile, sP);
    }
}
template <int T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_f64(
    const GemmItem* __restrict__ items, const int2* __restrict__ tiles) {
    const int2 tt = tiles[blockIdx.x];
    const GemmItem g = items[tt.x];
    gemm_tile<T>(g, tt.y);
}
// a few products whose descriptors travel as a kernel argument (no descriptor upload)
template <int T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_f64_arg(const GemmArgs p) {
    int i = 0;
    while (i + 1 < p.count && (int)blockIdx.x >= p.first[i + 1]) ++i;
    gemm_tile<T>(p.item[i], (int)blockIdx.x - p.first[i]);
}

int gemm_tiles(const GemmItem& g, int tile) {
    const int tm = g.k < GEMM_KS_MIN ? 64 : tile, tn = g.k < GEMM_KS_MIN ? 16 : tile == GEMM_TALL ? 32 : tile;
    return ((g.m + tm - 1) / tm) * ((g.n + tn - 1) / tn);
}
void launch_gemm(const GemmItem* d_items, const int2* d_tiles, int ntiles, int tile, hipStream_t s) {
    if (ntiles <= 0) return;
    if (tile == GEMM_TALL) k_gemm_f64<GEMM_TALL><<<ntiles, 256, 0, s>>>(d_items, d_tiles);
    else if (tile == 32) k_gemm_f64<2><<<ntiles, 256, 0, s>>>(d_items, d_tiles);
    else k_gemm_f64<1><<<ntiles, 256, 0, s>>>(d_items, d_tiles);
}
void launch_gemm_args(GemmArgs& p, int tile, hipStream_t s) {
    p.first[0] = 0;
    for (int i = 0; i < p.count; ++i) p.first[i + 1] = p.first[i] + gemm_tiles(p.item[i], tile);
    const int ntiles = p.first[p.count];
    if (ntiles <= 0) return;
    if (tile == GEMM_TALL) k_gemm_f64_arg<GEMM_TALL><<<ntiles, 256, 0, s>>>(p);
    else if (tile == 32) k_gemm_f64_arg<2><<<ntiles, 256, 0, s>>>(p);
    else k_gemm_f64_arg<1><<<ntiles, 256, 0, s>>>(p);
}
int gemm_tile_choice(const GemmItem* items, int count, bool tall) {
    long long t32 = 0, talls = 0;
    for (int i = 0; tall && i < count; ++i) {
        tall = items[i].m >= GEMM_TALL_ROWS;
        talls += gemm_tiles(items[i], GEMM_TALL);
    }
    if (tall && talls >= GEMM_TILE32_MIN) return GEMM_TALL;
    for (int i = 0; i < count; ++i)
        if (items[i].k >= GEMM_KS_MIN) t32 += (long long)((items[i].m + 31) / 32) * ((items[i].n + 31) / 32);
    return t32 >= GEMM_TILE32_MIN ? 32 : 16;
}
void launch_gemm_arg(const GemmItem& g, hipStream_t s) {
    if (g.m <= 0 || g.n <= 0) return;
    GemmArgs p;
    p.count = 1;
    p.item[0] = g;
    if (p.item[0].dk_mod <= 0) p.item[0].dk_mod = 1;
    if (p.item[0].dk_div <= 0) p.item[0].dk_div = 1;
    launch_gemm_args(p, gemm_tile_choice(p.item, 1), s);
}

}  // namespace qh
