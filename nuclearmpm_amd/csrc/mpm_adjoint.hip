// Reverse-mode (adjoint) kernels of one MLS-MPM step (jelly, snow, liquid) for gfx950.
//
// Given the cotangent of the state after a step (x', v', F', C', Jp') these kernels produce the
// cotangent of the state before it (x, v, F, C, Jp) and of Young's modulus, per scene.  They run after
// the forward sort, P2G and grid kernels have been recomputed for the state before the step, and
// reuse that step's tiles, work items and P2G slots:
//
//   g2p_adjoint   one workgroup per P2G work item: per particle, the cotangents of the gathered
//                 velocity and affine matrix are scattered back to the 3^D nodes (exact fixed-point
//                 sums in LDS, as in P2G, stored per work item); the partial x and F cotangents
//                 that G2P itself contributes go to grad_in.  Snow and liquid first recompute the
//                 forward's F^ = (I' + dt C') F bit for bit and pass the cotangents of F' and Jp'
//                 back through the material update: snow's F' = U clamp(S) V^T (the backward pass
//                 of a function of the singular values) and Jp' = clamp(Jp det F^ / det F'),
//                 liquid's F'_00 = prod S
//   grid_adjoint  one workgroup per node tile: sums both slot sets (or, when the forward grid
//                 kernel kept the pre-update sums, reads those and sums the adjoint slots), recomputes grid_op
//                 (src/nclr.h:263-310) and maps the velocity cotangent to the cotangent of the
//                 pre-update {momentum, mass} (clamped components and sticky nodes pass nothing)
//   p2g_adjoint   per particle: gathers the grid cotangent through the P2G stencil and the fused
//                 affine matrix (src/nclr.h:104-165, 313-337), including the backward pass of the
//                 polar decomposition F = R S: for a cotangent Rbar of R, Fbar = 2 R Y with Y skew
//                 and S Y + Y S = skew(R^T Rbar); snow's hardening e = exp(10 (1 - Jp)) adds the
//                 Jp cotangent of mu = mu0 e and lambda = lambda0 e; completes grad_in and the
//                 per-particle dL/dE
//   e_sum         per scene, a fixed-order double sum of the dL/dE contributions
//
// The same restatement on the CPU in FP64 (the oracle's adjoint) is checked against central
// finite differences of the step.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mpm_device.hpp"

namespace nclr_dev {

// d det(A) / dA
NCLR_DI M<2> cofactor(const M<2>& a) {
    M<2> c;
    c.a[0][0] = a.a[1][1];
    c.a[0][1] = -a.a[1][0];
    c.a[1][0] = -a.a[0][1];
    c.a[1][1] = a.a[0][0];
    return c;
}

NCLR_DI M<3> cofactor(const M<3>& a) {
    M<3> c;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
            c.a[i][j] = a.a[i1][j1] * a.a[i2][j2] - a.a[i1][j2] * a.a[i2][j1];
        }
    return c;
}

// Fbar += d<Rbar, R(F)>/dF for the rotation factor R of the polar decomposition F = R S.
template <int D>
NCLR_DI void polar_backward(const M<D>& F, const M<D>& R, const M<D>& Rbar, M<D>& Fbar) {
    M<D> S, Mm;
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) {
            float s = 0.0f, m = 0.0f;
#pragma unroll
            for (int k = 0; k < D; ++k) {
                s += R.a[k][i] * F.a[k][j];
                m += R.a[k][i] * Rbar.a[k][j];
            }
            S.a[i][j] = s;
            Mm.a[i][j] = m;
        }
    M<D> Y;
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) Y.a[i][j] = 0.0f;
    if constexpr (D == 2) {
        const float y = 0.5f * (Mm.a[1][0] - Mm.a[0][1]) / (S.a[0][0] + S.a[1][1]);
        Y.a[1][0] = y;
        Y.a[0][1] = -y;
    } else {
        // skew(M) as a vector m: (tr(S) I - sym(S)) y = m
        const float mv[3] = {0.5f * (Mm.a[2][1] - Mm.a[1][2]), 0.5f * (Mm.a[0][2] - Mm.a[2][0]),
                             0.5f * (Mm.a[1][0] - Mm.a[0][1])};
        const float tr = S.a[0][0] + S.a[1][1] + S.a[2][2];
        M<3> Q;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) Q.a[i][j] = (i == j ? tr : 0.0f) - 0.5f * (S.a[i][j] + S.a[j][i]);
        const M<3> Qc = cofactor(Q);
        const float inv_det = 1.0f / det(Q);
        float y[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) y[i] = (Qc.a[0][i] * mv[0] + Qc.a[1][i] * mv[1] + Qc.a[2][i] * mv[2]) * inv_det;
        Y.a[2][1] = y[0];
        Y.a[1][2] = -y[0];
        Y.a[0][2] = y[1];
        Y.a[2][0] = -y[1];
        Y.a[1][0] = y[2];
        Y.a[0][1] = -y[2];
    }
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) {
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < D; ++k) s += R.a[i][k] * Y.a[k][j];
            Fbar.a[i][j] += 2.0f * s;
        }
}

// Fbar += the cotangent of A through A -> U f(S) V^T, f = the snow clamp of the signed singular
// values (src/nclr.h:241-245).  With P = U^T Gbar V: Q_ii = f'(s_i) P_ii and, for i != j,
// Q_ij = a_ij (P_ij + P_ji) / 2 + b_ij (P_ij - P_ji) / 2 with the divided differences
// a_ij = (f_i - f_j) / (s_i - s_j) (1 when both are inside the clamp, 0 when both are clamped to the
// same bound) and b_ij = (f_i + f_j) / (s_i + s_j); then Fbar += U Q V^T.
template <int D>
NCLR_DI void clamp_svd_backward(const M<D>& U, const float (&sig)[D], const M<D>& V, float lo, float hi,
                                const M<D>& Gbar, M<D>& Fbar) {
    float f[D];
    int side[D];  // -1: at or below lo, 1: at or above hi, 0: inside
#pragma unroll
    for (int i = 0; i < D; ++i) {
        side[i] = sig[i] <= lo ? -1 : (hi <= sig[i] ? 1 : 0);
        f[i] = side[i] < 0 ? lo : (side[i] > 0 ? hi : sig[i]);
    }
    M<D> GV, P;
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int j = 0; j < D; ++j) {
            float t = 0.0f;
#pragma unroll
            for (int b = 0; b < D; ++b) t += Gbar.a[a][b] * V.a[b][j];
            GV.a[a][j] = t;
        }
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) {
            float t = 0.0f;
#pragma unroll
            for (int a = 0; a < D; ++a) t += U.a[a][i] * GV.a[a][j];
            P.a[i][j] = t;
        }
    M<D> Q;
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (i == j) {
                Q.a[i][i] = side[i] == 0 ? P.a[i][i] : 0.0f;
                continue;
            }
            const float a = (side[i] == 0 && side[j] == 0) ? 1.0f
                            : (side[i] == side[j] ? 0.0f : (f[i] - f[j]) / (sig[i] - sig[j]));
            const float b = (f[i] + f[j]) / (sig[i] + sig[j]);
            Q.a[i][j] = 0.5f * (a * (P.a[i][j] + P.a[j][i]) + b * (P.a[i][j] - P.a[j][i]));
        }
    M<D> UQ;
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int j = 0; j < D; ++j) {
            float t = 0.0f;
#pragma unroll
            for (int i = 0; i < D; ++i) t += U.a[a][i] * Q.a[i][j];
            UQ.a[a][j] = t;
        }
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) {
            float t = 0.0f;
#pragma unroll
            for (int j = 0; j < D; ++j) t += UQ.a[a][j] * V.a[b][j];
            Fbar.a[a][b] += t;
        }
}

// Cotangents of F^ = (I' + dt C') F and of the old Jp from those of the material update's outputs
// (src/nclr.h:230-258): jelly F' = F^; snow F' = U clamp(S) V^T and Jp' = clamp(Jp det F^ / det F',
// 0.6, 20); liquid F' = diag<dim>(1) with F'_00 = J = prod S (|det F^| in 2D, det F^ in 3D).  The SVD
// is the forward's (same method and operation order).
template <int D, bool EXACT>
NCLR_DI void material_backward(int material, const M<D>& Fh, float Jp, const M<D>& Fbar_new, float Jbar_new,
                               M<D>& Fhbar, float& Jbar) {
    if (material == MPM_JELLY) {
        Fhbar = Fbar_new;
        Jbar = Jbar_new;
        return;
    }
    M<D> U, V;
    float sig[D];
    step_svd<EXACT ? kSvdExact : kSvdFast, D>(Fh, U, sig, V);
    if (material == MPM_SNOW) {
        const float lo = float(1.0 - 2.5e-2), hi = float(1.0 + 4.5e-3);
        M<D> US;
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) US.a[a][b] = U.a[a][b] * ((sig[b] < lo) ? lo : ((hi < sig[b]) ? hi : sig[b]));
        const M<D> Fn = matmul_bt<D>(US, V);
        const float old_J = det(Fh), new_J = det(Fn);
        const float r = Jp * old_J / new_J;
        const float rbar = (r > 0.6f && r < 20.0f) ? Jbar_new : 0.0f;
        Jbar = rbar * old_J / new_J;
        const M<D> cof_h = cofactor(Fh), cof_n = cofactor(Fn);
        const float c1 = rbar * Jp / new_J, c2 = rbar * Jp * old_J / (new_J * new_J);
        M<D> Gn;
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) {
                Fhbar.a[a][b] = c1 * cof_h.a[a][b];
                Gn.a[a][b] = Fbar_new.a[a][b] - c2 * cof_n.a[a][b];
            }
        clamp_svd_backward<D>(U, sig, V, lo, hi, Gn, Fhbar);
    } else {
        double J = 1.0;
#pragma unroll
        for (int d = 0; d < D; ++d) J *= double(sig[d]);
        const float sgn = float(J) * det(Fh) < 0.0f ? -1.0f : 1.0f;
        const M<D> cof = cofactor(Fh);
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) Fhbar.a[a][b] = Fbar_new.a[0][0] * sgn * cof.a[a][b];
        Jbar = Jbar_new;
    }
}

NCLR_DI float ldg(const float* __restrict__ g, int64_t gstride, int c, int64_t j) { return g[int64_t(c) * gstride + j]; }

// The stencil sums both particle adjoints take, over the 3^D nodes i of a particle with weights W_i and
// values g_i, in cell units around the middle node: u = off - 1, phi = fx - 1, and at every node the
// bracket b_i = k + B u (a polynomial in the node's offset, as the scattered and gathered affine velocities
// are):
//   m0_r = sum W_i g_ir      T_rc = sum W_i g_ir u_c      fxb_a = sum S_i dW_i / dfx_a
// with S_i = g_i . b_i (MASS: + cm g_i.w).  The weights are products over the axes, so the sums are nested
// per axis: about 20 multiply-adds a node where the sums node by node took 55 (3D).  emit(o, W_i, b_i)
// is called at every node.  These derivatives have no bitwise counterpart: fused multiply-adds, and
// the error against 64 bits is that of the sums node by node (gradients within 6e-7 of theirs).
// 3D: one plane of nine nodes' loads in flight (27 spill).  FMA_PLANE: the bracket moves to a plane by a
// multiply-add instead of selects; the form that leaves the caller's kernel without spills.  Both kernels are bound by VALU issue:
// 8 x 262,144 jelly particles, G2P adjoint 259 -> 187 us, P2G adjoint 342 -> 258 (60,007 snow
// particles 36.6 -> 29.6 and 27.4 -> 19.0).
template <int D, bool MASS, bool FMA_PLANE, typename Node, typename Emit>
NCLR_DI void adjoint_stencil(const float (&fx)[D], const M<D>& B, const float (&k)[D], float cm, const Node& node,
                             Emit emit, float (&m0)[D], M<D>& T, float (&fxb)[D]) {
    constexpr int L = D - 1;  // the innermost axis
    // the weights' derivatives are f, -2 f - 1 and f + 1 with f = fx - 1.5: their sum against S_0, S_1, S_2
    // is f ((S_0 - S_1) + (S_2 - S_1)) + (S_2 - S_1)
    float w[D][3], lo = 0.0f, hi = 0.0f;  // axis 0: S_0 - S_1 and S_2 - S_1 over the planes
#pragma unroll
    for (int a = 0; a < D; ++a) {
        bspline_weights(fx[a], w[a]);
        m0[a] = 0.0f;
        fxb[a] = 0.0f;
#pragma unroll
        for (int c = 0; c < D; ++c) T.a[a][c] = 0.0f;
    }
    auto dsum = [](float f, float s0, float s1, float s2) { return fmaf(f - 1.5f, (s0 - s1) + (s2 - s1), s2 - s1); };
    // one row of three nodes along the innermost axis: r0 = sum w g, r2 = sum w u g, rs = sum w S,
    // rd = sum dw S
    auto row = [&](int o0, int o1, const float (&b)[D], float wo, float (&r0)[D], float (&r2)[D], float& rs, float& rd) {
        float So[3];
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            int off[D];
            off[0] = o0;
            if constexpr (D == 3) off[1] = o1;
            off[L] = o;
            const float4 g = node(off);
            const float gr[3] = {g.x, g.y, g.z};
            float bi[D];
            float S = MASS ? g.w * cm : 0.0f;
#pragma unroll
            for (int r = 0; r < D; ++r) {
                bi[r] = o == 1 ? b[r] : (o == 0 ? b[r] - B.a[r][L] : b[r] + B.a[r][L]);
                S = !MASS && r == 0 ? gr[r] * bi[r] : fmaf(gr[r], bi[r], S);
                const float p = w[L][o] * gr[r];
                r0[r] = o == 0 ? p : r0[r] + p;
                if (o == 0) r2[r] = -p;
                if (o == 2) r2[r] = r2[r] + p;
            }
            rs = o == 0 ? w[L][o] * S : fmaf(w[L][o], S, rs);
            So[o] = S;
            emit(off, wo * w[L][o], bi);
        }
        rd = dsum(fx[L], So[0], So[1], So[2]);
    };
#pragma unroll(D == 3 ? 1 : 3)
    for (int o0 = 0; o0 < 3; ++o0) {
        const float w0 = pick3(w[0], o0);
        float b0[D], q0[D], q2[D], qs, qd;
#pragma unroll
        for (int r = 0; r < D; ++r) b0[r] = FMA_PLANE ? fmaf(B.a[r][0], float(o0 - 1), k[r])
                              : (o0 == 1 ? k[r] : (o0 == 0 ? k[r] - B.a[r][0] : k[r] + B.a[r][0]));
        if constexpr (D == 2) {
            row(o0, 0, b0, w0, q0, q2, qs, qd);
        } else {
            float q1[3], ro[3];
#pragma unroll
            for (int o1 = 0; o1 < 3; ++o1) {
                float b1[3], r0[3], r2[3], rs, rd;
#pragma unroll
                for (int r = 0; r < 3; ++r)
                    b1[r] = o1 == 1 ? b0[r] : (o1 == 0 ? b0[r] - B.a[r][1] : b0[r] + B.a[r][1]);
                row(o0, o1, b1, w0 * w[1][o1], r0, r2, rs, rd);
                ro[o1] = rs;
                const float w1 = w[1][o1];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    q0[r] = o1 == 0 ? w1 * r0[r] : fmaf(w1, r0[r], q0[r]);
                    if (o1 == 0) q1[r] = -q0[r];
                    if (o1 == 2) q1[r] = fmaf(w1, r0[r], q1[r]);
                    q2[r] = o1 == 0 ? w1 * r2[r] : fmaf(w1, r2[r], q2[r]);
                }
                qs = o1 == 0 ? w1 * rs : fmaf(w1, rs, qs);
                qd = o1 == 0 ? w1 * rd : fmaf(w1, rd, qd);
            }
#pragma unroll
            for (int r = 0; r < 3; ++r) T.a[r][1] = fmaf(w0, q1[r], T.a[r][1]);
            fxb[1] = fmaf(w0, dsum(fx[1], ro[0], ro[1], ro[2]), fxb[1]);
        }
#pragma unroll
        for (int r = 0; r < D; ++r) {
            const float wq = w0 * q0[r];
            m0[r] = m0[r] + wq;
            T.a[r][0] = T.a[r][0] + (o0 == 1 ? 0.0f : (o0 == 0 ? -wq : wq));
            T.a[r][L] = fmaf(w0, q2[r], T.a[r][L]);
        }
        lo += o0 == 0 ? qs : (o0 == 1 ? -qs : 0.0f);
        hi += o0 == 2 ? qs : (o0 == 1 ? -qs : 0.0f);
        fxb[L] = fmaf(w0, qd, fxb[L]);
    }
    fxb[0] = fmaf(fx[0] - 1.5f, lo + hi, hi);
}

// ---------------------------------------------------------------------------------------------
// G2P adjoint (src/nclr.h:167-258).  GENERAL: any material (the scene's, at run time); otherwise
// every scene is jelly.  A work item of TPB * PPT particles, PPT per thread.  At least two waves per
// SIMD (at most 256 VGPRs): measured 1.45x faster than one wave per SIMD; four (128 VGPRs) with one
// 3D particle per thread.
// ---------------------------------------------------------------------------------------------
template <int D, int PPT, int TPB, bool GENERAL, bool EXACT>
__global__ __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(D == 3 && PPT == 1 ? 4 : 2))) void k_g2p_adjoint(const float* __restrict__ st, const uint32_t* __restrict__ perm,
                                                     const uint32_t* __restrict__ item_offset, StepParams p,
                                                     const float4* __restrict__ gv, const float* __restrict__ gout,
                                                     float* __restrict__ gin, int64_t gstride,
                                                     float4* __restrict__ slots_b) {
    using TL = Tile<D>;
    using L = Layout<D>;
    constexpr int REG = TL::REGION;
    constexpr int K = D == 2 ? 9 : 27;
    __shared__ unsigned long long acc[D * REG];
    __shared__ uint32_t nonfinite[REG];
    constexpr int NW = TPB / 64;
    __shared__ float s_bound[NW][D];
    const uint32_t item = blockIdx.x;
    const WorkItem wi = work_item(p, item);  // loaded with the count below, used only if valid
    if (item >= item_offset[p.ntiles]) return;
    for (int r = threadIdx.x; r < D * REG; r += blockDim.x) acc[r] = 0ull;
    for (int r = threadIdx.x; r < REG; r += blockDim.x) nonfinite[r] = 0u;
    __syncthreads();
    const uint32_t tile = wi.tile;
    const SceneParams sp = p.scenes[p.nscenes == 1 ? 0 : scene_of_tile(p, tile)];
    int torg[D];
    tile_coords<D>(tile - sp.tile_base, sp.nt, torg);
#pragma unroll
    for (int a = 0; a < D; ++a) torg[a] *= TL::S;
    const uint32_t j0 = wi.j0, j1 = wi.j1;
    const float four_inv_dx = 4.0f * sp.inv_dx;

    // pass 1: cotangents of the gathered velocity (vb = v' + dt x') and affine matrix
    // (Cb = C' + dt F' F^T) and a bound of the scattered sums per channel
    bool valid[PPT], finite[PPT];
    int bases[PPT][D];
    float fxs[PPT][D], vb[PPT][D];
    M<D> Cb[PPT];
    float bound[D];
#pragma unroll
    for (int c = 0; c < D; ++c) bound[c] = 0.0f;
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const uint32_t j = j0 + uint32_t(k) * TPB + threadIdx.x;
        valid[k] = false;
        if (j >= j1) continue;
        const int64_t i = perm[j];
        float x[D];
        M<D> F;
#pragma unroll
        for (int a = 0; a < D; ++a) x[a] = ldf(st, p.stride, L::X + a, i);
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) F.a[a][b] = ldf(st, p.stride, L::F + a * D + b, i);
        int base[D];
        float fx[D], w[D][3];
        if (!stencil<D>(x, sp, base, fx, w)) continue;  // keyed into this tile, so never taken
        valid[k] = true;
        float wsum = 1.0f;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            bases[k][a] = base[a];
            fxs[k][a] = fx[a];
            vb[k][a] = ldg(gout, gstride, L::V + a, j) + sp.dt * ldg(gout, gstride, L::X + a, j);
            wsum *= fabsf(w[a][0]) + fabsf(w[a][1]) + fabsf(w[a][2]);
        }
        // Fb: cotangent of F^ = (I' + dt C') F
        M<D> Fb;
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) Fb.a[a][b] = ldg(gout, gstride, L::F + a * D + b, j);
        if constexpr (GENERAL) {
            // the forward's C' (k_g2p_sorted's operation order, so F^ is the forward's bit for bit)
            M<D> Cf;
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int b = 0; b < D; ++b) Cf.a[a][b] = 0.0f;
            const StencilRows<D> node(gv, base, sp.ntn, sp.node_tile_base);
#pragma unroll
            for (int o = 0; o < K; ++o) {
                int off[D];
                float dpos[D];
                offsets<D>(o, off);
#pragma unroll
                for (int a = 0; a < D; ++a) dpos[a] = float(off[a]) - fx[a];
                const float4 g = node(off);
                const float gvel[3] = {g.x, g.y, g.z};
                float weight = w[0][off[0]];
#pragma unroll
                for (int a = 1; a < D; ++a) weight = weight * w[a][off[a]];
#pragma unroll
                for (int a = 0; a < D; ++a) {
                    const float wv = four_inv_dx * (weight * gvel[a]);
#pragma unroll
                    for (int b = 0; b < D; ++b) Cf.a[a][b] = Cf.a[a][b] + wv * dpos[b];
                }
            }
            M<D> Mx;
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int b = 0; b < D; ++b) {
                    const float id1 = (a == b && (a < 2 || sp.identity_mode == 1)) ? 1.0f : 0.0f;
                    Mx.a[a][b] = id1 + sp.dt * Cf.a[a][b];
                }
            const M<D> Fh = matmul<D>(Mx, F);
            const float Jp = ldf(st, p.stride, L::JP, i);
            const M<D> Fbn = Fb;
            float Jb;
            material_backward<D, EXACT>(sp.material, Fh, Jp, Fbn, ldg(gout, gstride, L::JP, j), Fb, Jb);
            // F cotangent (I' + dt C')^T Fbar^ and the Jp cotangent of the G2P update
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int b = 0; b < D; ++b) {
                    float t = 0.0f;
#pragma unroll
                    for (int q = 0; q < D; ++q) t += Mx.a[q][a] * Fb.a[q][b];
                    gin[int64_t(L::F + a * D + b) * gstride + i] = t;
                }
            gin[int64_t(L::JP) * gstride + i] = Jb;
        }
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) {
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < D; ++q) s += Fb.a[a][q] * F.a[b][q];
                Cb[k].a[a][b] = ldg(gout, gstride, L::C + a * D + b, j) + sp.dt * s;
            }
#pragma unroll
        for (int a = 0; a < D; ++a) {
            float s = 0.0f;
#pragma unroll
            for (int b = 0; b < D; ++b) s += fabsf(Cb[k].a[a][b]);
            // |off - fx| is at most 1.5 on every axis, except in the half cell at the lower walls (stencil base 0,
            // fx from -0.5 to 0.5): up to 2.5 there, but beyond 1.5 only at the third node, whose weight is at
            // most an eighth of the axis's |weights|, so that no contribution exceeds the bound there either
            const float vc = fabsf(vb[k][a]), bc = wsum * (vc + 1.5f * four_inv_dx * s);
            // the unchecked deposits also need every bracket finite, which the weight is multiplied to
            finite[k] = (a == 0 || finite[k]) && bc < 3.0e38f && vc + 2.5f * four_inv_dx * s < 3.0e38f;
            if (bc < 3.0e38f) bound[a] = fmaxf(bound[a], bc);
        }
    }
#pragma unroll
    for (int c = 0; c < D; ++c) {
        float b = bound[c];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) b = fmaxf(b, __shfl_xor(b, off));
        bound[c] = b;
    }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int c = 0; c < D; ++c) s_bound[threadIdx.x >> 6][c] = bound[c];
    __syncthreads();
    float scale[D];
    double inv_scale[D];
#pragma unroll
    for (int c = 0; c < D; ++c) {
        float b = s_bound[0][c];
#pragma unroll
        for (int w = 1; w < NW; ++w) b = fmaxf(b, s_bound[w][c]);
        fixed_point_scale(b, scale[c], inv_scale[c]);
    }

    // pass 2: gather the updated grid (for the forward C and the weight derivatives), scatter the
    // quantised grid cotangent, write the partial x and F cotangents
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        if (!valid[k]) continue;
        const uint32_t j = j0 + uint32_t(k) * TPB + threadIdx.x;
        int rb = 0;
        M<D> Bm, Tm;
        float kb[D], m0[D], fxbar[D];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            rb = rb * TL::R + (bases[k][a] - torg[a]);
            kb[a] = vb[k][a];
#pragma unroll
            for (int b = 0; b < D; ++b) {
                Bm.a[a][b] = four_inv_dx * Cb[k].a[a][b];
                kb[a] = fmaf(-Bm.a[a][b], fxs[k][b] - 1.0f, kb[a]);
            }
        }
        const StencilRows<D> node(gv, bases[k], sp.ntn, sp.node_tile_base);
        // a particle whose bound is finite has every |contribution * scale| below 2^50 (up to the
        // rounding of the bracket, and the conversion holds to 2^51)
        if (finite[k]) {
            adjoint_stencil<D, false, !GENERAL>(
                fxs[k], Bm, kb, 0.0f, node,
                [&](const int (&off)[D], float weight, const float (&bi)[D]) {
                    int r = 0;
#pragma unroll
                    for (int a = 0; a < D; ++a) r = r * TL::R + off[a];
#pragma unroll
                    for (int a = 0; a < D; ++a)
                        atomicAdd(&acc[a * REG + rb + r], fixed_point(weight * bi[a], double(scale[a])));
                },
                m0, Tm, fxbar);
        } else {
            adjoint_stencil<D, false, !GENERAL>(
                fxs[k], Bm, kb, 0.0f, node,
                [&](const int (&off)[D], float weight, const float (&bi)[D]) {
                    int r = 0;
#pragma unroll
                    for (int a = 0; a < D; ++a) r = r * TL::R + off[a];
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        const float y = weight * bi[a] * scale[a];
                        if (fabsf(y) < kFixedLimit) atomicAdd(&acc[a * REG + rb + r], fixed_point(y));
                        else atomicOr(&nonfinite[rb + r], 1u << a);
                    }
                },
                m0, Tm, fxbar);
        }
        M<D> Cn;
#pragma unroll
        for (int b = 0; b < D; ++b)
#pragma unroll
            for (int a = 0; a < D; ++a) {
                fxbar[b] = fmaf(-Bm.a[a][b], m0[a], fxbar[b]);
                Cn.a[a][b] = four_inv_dx * fmaf(-m0[a], fxs[k][b] - 1.0f, Tm.a[a][b]);
            }
        const int64_t i = perm[j];
#pragma unroll
        for (int a = 0; a < D; ++a)
            gin[int64_t(L::X + a) * gstride + i] = ldg(gout, gstride, L::X + a, j) + sp.inv_dx * fxbar[a];
        if constexpr (!GENERAL) {
            // jelly: F' = (I' + dt C) F  =>  F cotangent (I' + dt C)^T F'; Jp is carried unchanged
#pragma unroll
            for (int a = 0; a < D; ++a)
#pragma unroll
                for (int b = 0; b < D; ++b) {
                    float s = 0.0f;
#pragma unroll
                    for (int q = 0; q < D; ++q) {
                        const float id1 = (q == a && (a < 2 || sp.identity_mode == 1)) ? 1.0f : 0.0f;
                        s += (id1 + sp.dt * Cn.a[q][a]) * ldg(gout, gstride, L::F + q * D + b, j);
                    }
                    gin[int64_t(L::F + a * D + b) * gstride + i] = s;
                }
            gin[int64_t(L::JP) * gstride + i] = ldg(gout, gstride, L::JP, j);
        }
    }
    __syncthreads();
    float4* dst = slots_b + int64_t(item) * REG;
    const float nan = __builtin_nanf("");
    for (int r = threadIdx.x; r < REG; r += blockDim.x) {
        float out[3] = {0.0f, 0.0f, 0.0f};
        const uint32_t bad = nonfinite[r];
#pragma unroll
        for (int c = 0; c < D; ++c)
            out[c] = (bad >> c) & 1u ? nan : fixed_point_value(acc[c * REG + r], inv_scale[c]);
        dst[r] = make_float4(out[0], out[1], out[2], 0.0f);
    }
}

// ---------------------------------------------------------------------------------------------
// grid adjoint (src/nclr.h:263-310)
// ---------------------------------------------------------------------------------------------
// A workgroup per node tile, a thread per node, as the forward grid kernels; LISTED: the node tiles come
// from the sort's list, otherwise every one has a workgroup.  TAPE: gpre holds the forward's pre-update
// sums and only the adjoint slots are summed; otherwise both slot sets are, the forward's in the
// forward grid kernel's order.  8 x 262,144 jelly particles 61.3 -> 36.0 us, 60,007 snow 12.0 -> 8.6.
template <int D, bool TAPE, bool LISTED>
__global__ __launch_bounds__(Tile<D>::NODES) void k_grid_adjoint(const float4* __restrict__ slots,
                                                                 const float4* __restrict__ slots_b,
                                                                 const float4* __restrict__ gpre,
                                                                 const uint32_t* __restrict__ item_offset, StepParams p,
                                                                 const GridTile<D>* __restrict__ tiles,
                                                                 const uint32_t* __restrict__ meta,
                                                                 float4* __restrict__ gbar) {
    using TL = Tile<D>;
    __shared__ SlotLists<D> s_lists;
    const GridThread<D> th;
    const uint32_t listed = LISTED ? meta[kMetaGridTiles] : p.node_tiles;
    uint32_t index;
    for (uint32_t i = 0; grid_tile_index(listed, i, index); ++i) {
        GridTile<D> tile;  // uniform over the workgroup
        if constexpr (LISTED) {
            tile = tiles[index];
        } else {
            tile.node_tile = int(index);
            tile.scene = p.nscenes == 1 ? 0 : scene_of_node_tile(p, index);
        }
        const uint32_t nt_idx = uint32_t(tile.node_tile);
        const SceneParams sp = p.scenes[tile.scene];
        if constexpr (!LISTED) {
            int nto[D];
            tile_coords<D>(nt_idx - sp.node_tile_base, sp.ntn, nto);
            int any = 0;
#pragma unroll
            for (int c = 0; c < (1 << D); ++c) {
                grid_tile_candidate<D>(sp, nto, c, item_offset, tile.first[c], tile.count[c]);
                any += tile.count[c];
            }
            if (any == 0) continue;  // no particle's stencil reaches this node tile
        }
        int n[D];
        th.node(nt_idx - sp.node_tile_base, sp.ntn, n);
        float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f), bv[8];
        float4 g = b, part[3] = {b, b, b}, av[TAPE ? 1 : 8];  // 2D: the forward's four partial sums
        if constexpr (TAPE) g = gpre[int64_t(nt_idx) * TL::NODES + th.l];
        // a position past the node's list adds +0.0, which leaves a sum that started at +0.0 unchanged
        visit_slots<D, D == 2 ? 4 : 1>(
            s_lists, tile.first, tile.count, th.cls, th.wave_classes,
            [&](int u, int64_t at) {
                bv[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if constexpr (!TAPE) av[u] = bv[u];
                if (at >= 0) {
                    bv[u] = slots_b[at + th.r];
                    if constexpr (!TAPE) av[u] = slots[at + th.r];
                }
            },
            [&](auto positions) {
#pragma unroll
                for (int u = 0; u < decltype(positions)::value; ++u) {
                    add4(b, bv[u]);
                    if constexpr (!TAPE) add4(D == 2 && (u & 3) ? part[(u & 3) - 1] : g, av[u]);
                }
            });
        if constexpr (D == 2 && !TAPE)
#pragma unroll
            for (int k = 0; k < 3; ++k) add4(g, part[k]);
        const float mom[3] = {g.x, g.y, g.z};
        const float vbar[3] = {b.x, b.y, b.z};
        const float m = g.w;
        // forward grid_op, remembering which components were clamped and whether the sticky
        // boundary zeroed the node
        float vel[D];
        bool clamped[D];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            vel[a] = mom[a];
            clamped[a] = false;
        }
        if (m > 0.0f) {
#pragma unroll
            for (int a = 0; a < D; ++a) vel[a] = vel[a] / m;
            vel[1] = vel[1] + sp.dt * sp.gravity;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                clamped[a] = vel[a] < -sp.allowed || sp.allowed < vel[a];
                vel[a] = (vel[a] < -sp.allowed) ? -sp.allowed : ((sp.allowed < vel[a]) ? sp.allowed : vel[a]);
            }
        }
        bool sticky = false;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            if ((n[a] < 3 && vel[a] < 0.0f) || (n[a] >= (sp.res + 1) - 3 && vel[a] > 0.0f)) {
#pragma unroll
                for (int q = 0; q < D; ++q) vel[q] = 0.0f;
                sticky = true;
            }
        }
        float out[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (m > 0.0f && !sticky) {
            const float inv_m2 = 1.0f / (m * m);
            float mb = 0.0f;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const float vtb = clamped[a] ? 0.0f : vbar[a];
                out[a] = vtb / m;
                mb -= vtb * mom[a] * inv_m2;
            }
            out[3] = mb;
        }
        gbar[int64_t(nt_idx) * TL::NODES + th.l] = make_float4(out[0], out[1], out[2], out[3]);
    }
}

// ---------------------------------------------------------------------------------------------
// P2G adjoint (src/nclr.h:104-165, 313-372) per sorted position j, XCD-local block order.  In 3D the
// forward P2G leaves the particle's polar factor in `rot` (36 bytes a particle; its exact SVD was a third of
// this kernel's instructions), and F and the factor are read again behind the stencil instead of
// held through it, which fits four waves per SIMD: 8 x 262,144 jelly particles 258 -> 180 us (296
// bytes a particle, 3.4 TB/s), P2G 214 -> 216 with the factor's stores; 60,007 snow 19.0 -> 13.
// ---------------------------------------------------------------------------------------------
template <int D, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_p2g_adjoint(const float* __restrict__ st, const uint32_t* __restrict__ pid,
                                                     const uint32_t* __restrict__ perm,
                                                     const uint32_t* __restrict__ keys, StepParams p,
                                                     const float4* __restrict__ gbar, const float* __restrict__ gout,
                                                     float* __restrict__ gin, int64_t gstride,
                                                     float* __restrict__ epart, const float* __restrict__ rot) {
    using L = Layout<D>;
    const int64_t j = int64_t(xcd_block()) * blockDim.x + threadIdx.x;
    if (j >= p.n) return;
    const int64_t i = perm[j];
    const int64_t s = p.stride;
    const SceneParams sp = p.scenes[p.nscenes == 1 ? 0 : scene_of_sorted(p, keys, j, pid[i])];
    float x[D], v[D];
    M<D> F, C;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        x[a] = ldf(st, s, L::X + a, i);
        v[a] = ldf(st, s, L::V + a, i);
    }
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) {
            F.a[a][b] = ldf(st, s, L::F + a * D + b, i);
            C.a[a][b] = ldf(st, s, L::C + a * D + b, i);
        }
    const float Jp = ldf(st, s, L::JP, i);
    const float mass = ldf(st, s, L::MASS, i);
    const float vol = ldf(st, s, L::VOL, i);
    int base[D];
    float fx[D], w[D][3];
    if (!stencil<D>(x, sp, base, fx, w)) {
        // outside the grid the forward step carries the particle through unchanged
        for (int c = 0; c < L::NG; ++c) gin[int64_t(c) * gstride + i] = ldg(gout, gstride, c, j);
        epart[j] = 0.0f;
        return;
    }
    // the forward's polar factor: in 3D P2G kept it (a third of this kernel's instructions were its SVD),
    // F - R in the accurate mode and R in the others; F - R is formed as the forward forms it
    M<D> A, FmR, R;
    if constexpr (D == 3) {
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) {
                const float q = rot[int64_t(a * D + b) * s + j];
                R.a[a][b] = MODE == kSvdAccurate ? F.a[a][b] - q : q;
                FmR.a[a][b] = MODE == kSvdAccurate ? q : F.a[a][b] - q;
            }
    } else {
        FmR = f_minus_rotation<MODE, D>(F, R);
    }
    A = fused_affine_from<D>(sp.material, F, FmR, C, Jp, mass, vol, sp);
    // the bracket m v + A dpos of P2G's contributions in cell units around the middle node
    M<D> Bm, Abar;
    float kb[D], m0[D], fxbar[D];
#pragma unroll
    for (int r = 0; r < D; ++r) {
        kb[r] = mass * v[r];
#pragma unroll
        for (int c = 0; c < D; ++c) {
            Bm.a[r][c] = A.a[r][c] * sp.dx;
            kb[r] = fmaf(-Bm.a[r][c], fx[c] - 1.0f, kb[r]);
        }
    }
    const StencilRows<D> node(gbar, base, sp.ntn, sp.node_tile_base);
    adjoint_stencil<D, true, false>(fx, Bm, kb, mass, node, [](const int (&)[D], float, const float (&)[D]) {}, m0, Abar, fxbar);
    if constexpr (D == 3) {  // F and R again (they would hold 18 registers through the stencil)
        const float* st2 = st;
        const float* rot2 = rot;
        asm volatile("" : "+s"(st2), "+s"(rot2));
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) {
                F.a[a][b] = ldf(st2, s, L::F + a * D + b, i);
                const float q = rot2[int64_t(a * D + b) * s + j];
                R.a[a][b] = MODE == kSvdAccurate ? F.a[a][b] - q : q;
            }
    }
    float vin[D];
#pragma unroll
    for (int r = 0; r < D; ++r) {
        vin[r] = mass * m0[r];
#pragma unroll
        for (int c = 0; c < D; ++c) {
            fxbar[c] = fmaf(-Bm.a[r][c], m0[r], fxbar[c]);
            Abar.a[r][c] = sp.dx * fmaf(-m0[r], fx[c] - 1.0f, Abar.a[r][c]);
        }
    }
    // A = -(dt V0) Dinv PF + m C  ->  G = dL/dPF
    const float Dinv = 4.0f * sp.inv_dx * sp.inv_dx;
    const float e = hardening(sp.material, Jp);
    const float mu = sp.mu0 * e, lambda = sp.lambda0 * e;
    M<D> G;
    float sG = 0.0f;
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) {
            G.a[a][b] = -(sp.dt * vol) * Dinv * Abar.a[a][b];
            sG += G.a[a][b];
        }
    // PF = 2 mu (F - R) F^T + lambda (J - 1) J on every entry
    const float J = det(F);
    M<D> Fbar, Rbar;
    float mubar = 0.0f;
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) {
            float gf = 0.0f, gtfr = 0.0f, fmrf = 0.0f;
#pragma unroll
            for (int q = 0; q < D; ++q) {
                gf += G.a[a][q] * F.a[q][b];
                gtfr += G.a[q][a] * (F.a[q][b] - R.a[q][b]);
                fmrf += (F.a[a][q] - R.a[a][q]) * F.a[b][q];
            }
            Fbar.a[a][b] = 2.0f * mu * (gf + gtfr);
            Rbar.a[a][b] = -2.0f * mu * gf;
            mubar += G.a[a][b] * 2.0f * fmrf;
        }
    polar_backward<D>(F, R, Rbar, Fbar);
    const M<D> cof = cofactor(F);
    const float Jbar = sG * lambda * (2.0f * J - 1.0f);
#pragma unroll
    for (int a = 0; a < D; ++a) {
        gin[int64_t(L::X + a) * gstride + i] += sp.inv_dx * fxbar[a];
        gin[int64_t(L::V + a) * gstride + i] = vin[a];
    }
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) {
            gin[int64_t(L::F + a * D + b) * gstride + i] += Fbar.a[a][b] + Jbar * cof.a[a][b];
            gin[int64_t(L::C + a * D + b) * gstride + i] = mass * Abar.a[a][b];
        }
    const float lambar = sG * (J - 1.0f) * J;
    // snow: mu = mu0 e, lambda = lambda0 e with e = exp(10 (1 - Jp)), de/dJp = -10 e
    if (sp.material == MPM_SNOW) gin[int64_t(L::JP) * gstride + i] += (mubar * sp.mu0 + lambar * sp.lambda0) * (-10.0f * e);
    epart[j] = e * (mubar * sp.dmu_dE + lambar * sp.dlambda_dE);
}

// grad_E[s] += the sum of epart over scene s's sorted particles, in a fixed order, in three
// kernels: the scene's sorted range [lo, hi) (scenes occupy consecutive keys; particles off their
// grid sort last), partial sums of consecutive chunks of kEChunk positions counted from lo (each a
// fixed tree), then the scene's chunks in order.  The partition depends only on the scene's own
// range, so a scene's dL/dE is the same alone and inside a batch.
//
// One launch of each sums several adjoint steps' contributions (ESteps: up to kESteps steps of a segment,
// each with its own sort), every step's sum added to grad_E in the order of the steps: the same bits as a
// sum after every step, without its launches (two of a 2D single scene's five per adjoint step,
// 7 of 33 us with 19,600 particles).
constexpr int kEChunk = 2048;

// Boundary t of the range table (scene t / 2's first sorted position for even t, one past its last
// for odd t): the first sorted position with keys[.] >= the boundary's key.  One wave per boundary
// searches 64-ary: the answer lies in [lo, hi] (keys[lo - 1] < key, and hi = n or keys[hi] >= key);
// each round the lanes probe 64 evenly spaced positions and the first probe at or above the key
// narrows the interval to one spacing, so 2^21 keys take four rounds of one load per lane.
__global__ __launch_bounds__(64) void k_scene_ranges(ESteps es, StepParams p, int64_t* __restrict__ range) {
    const int t = int(blockIdx.x), step = int(blockIdx.y);
    if (t >= 2 * p.nscenes) return;
    const uint32_t* keys = reinterpret_cast<const uint32_t*>(es.sort(step) + es.keys);
    range += int64_t(step) * 2 * p.nscenes;
    const int sc = t >> 1;
    const uint32_t key = (t & 1) == 0 ? p.scenes[sc].tile_base
                                      : (sc + 1 < p.nscenes ? p.scenes[sc + 1].tile_base : p.ntiles);
    const int lane = int(threadIdx.x);
    int64_t lo = 0, hi = p.n;
    while (hi - lo > 64) {
        const int64_t step = (hi - lo + 63) / 64;
        // probe q; lane 63's is at or past hi - 1, and probes at or past hi load nothing
        const int64_t q = lo + int64_t(lane + 1) * step - 1;
        const bool at_or_above = q >= hi || keys[q] >= key;
        const uint64_t ball = __ballot(at_or_above);
        if (ball == 0ull) {  // every probe below the key, lane 63's at hi - 1: the answer is hi
            lo = lo + 64 * step;
        } else {
            const int f = __ffsll((unsigned long long)ball) - 1;
            const int64_t qf = lo + int64_t(f + 1) * step - 1;
            const int64_t new_lo = f == 0 ? lo : lo + int64_t(f) * step;  // one past probe f - 1
            hi = qf < hi ? qf : hi;
            lo = new_lo;
        }
    }
    // at most 64 candidates [lo, hi): the first at or above the key, else hi
    const int64_t q = lo + lane;
    const uint64_t ball = __ballot(q < hi && keys[q] >= key);
    if (lane == 0) range[t] = ball == 0ull ? hi : lo + (__ffsll((unsigned long long)ball) - 1);
}

// Sum of part[0..256) by a fixed tree over threads t = 0 .. 255; the result is in part[0] (after the last
// barrier for every thread).
NCLR_DI void tree_sum_256(double* part, int t) {
    for (int off = 128; off > 0; off >>= 1) {
        __syncthreads();
        if (t < off) part[t] += part[t + off];
    }
    __syncthreads();
}

// Scene sc's sorted range in step `step`: from the range table, or with range == nullptr (a single
// scene) [0, meta[0]), the particles on the grid, which the sort places first.
NCLR_DI void scene_range(const ESteps& es, const int64_t* __restrict__ range, int step, int nscenes, int sc,
                         int64_t& lo, int64_t& hi) {
    if (range) {
        lo = range[2 * (int64_t(step) * nscenes + sc)];
        hi = range[2 * (int64_t(step) * nscenes + sc) + 1];
    } else {
        lo = 0;
        hi = reinterpret_cast<const uint32_t*>(es.sort(step) + es.meta)[0];
    }
}

// Grid (chunks, scenes, steps): chunk blockIdx.x -> partial[(step * scenes + scene) * chunks + chunk].
__global__ __launch_bounds__(256) void k_scene_e_partial(ESteps es, const int64_t* __restrict__ range, int chunks,
                                                         double* __restrict__ partial) {
    __shared__ double part[256];
    const int sc = int(blockIdx.y), nscenes = int(gridDim.y), step = int(blockIdx.z);
    const float* __restrict__ epart = es.epart + int64_t(step) * es.stride;
    int64_t s_lo, s_hi;
    scene_range(es, range, step, nscenes, sc, s_lo, s_hi);
    const int64_t lo = s_lo + int64_t(blockIdx.x) * kEChunk;
    const int64_t hi = min(s_hi, lo + int64_t(kEChunk));
    // the thread's elements j, j + 256, ... summed in that order, eight loads in flight
    double acc = 0.0;
    int64_t j = lo + threadIdx.x;
    for (; j + 7 * 256 < hi; j += 8 * 256) {
        float e[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) e[u] = epart[j + u * 256];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += double(e[u]);
    }
    for (; j < hi; j += 256) acc += double(epart[j]);
    part[threadIdx.x] = acc;
    tree_sum_256(part, int(threadIdx.x));
    if (threadIdx.x == 0) partial[(int64_t(step) * nscenes + sc) * chunks + blockIdx.x] = part[0];
}

// One workgroup per scene: the used chunks of every step, ceil((hi - lo) / kEChunk), in order; four
// steps at a time, 256 threads each, added in the order of the steps.
__global__ __launch_bounds__(1024) void k_scene_e_final(ESteps es, const double* __restrict__ partial,
                                                        const int64_t* __restrict__ range, int chunks, int steps,
                                                        double* __restrict__ grad_E) {
    __shared__ double part[4][256];
    const int sc = int(blockIdx.x), nscenes = int(gridDim.x);
    const int q = int(threadIdx.x) >> 8, t = int(threadIdx.x) & 255;
    double sum = 0.0;
    if (threadIdx.x == 0) sum = grad_E[sc];
    for (int s0 = 0; s0 < steps; s0 += 4) {
        const int step = s0 + q;
        double acc = 0.0;
        if (step < steps) {
            int64_t lo, hi;
            scene_range(es, range, step, nscenes, sc, lo, hi);
            const int used = int(min(int64_t(chunks), (hi - lo + kEChunk - 1) / kEChunk));
            for (int c = t; c < used; c += 256) acc += partial[(int64_t(step) * nscenes + sc) * chunks + c];
        }
        part[q][t] = acc;
        tree_sum_256(part[q], t);
        if (threadIdx.x == 0)
            for (int u = 0; u < 4 && s0 + u < steps; ++u) sum += part[u][0];
        __syncthreads();
    }
    if (threadIdx.x == 0) grad_E[sc] = sum;
}

}  // namespace nclr_dev

namespace nclr_host {

using namespace nclr_dev;

static inline unsigned blocks_of(int64_t n, int threads) { return unsigned((n + threads - 1) / threads); }

template <int D, int PPT, int TPB, bool GENERAL, bool EXACT>
static hipError_t g2p_adjoint_one(const LaunchArgs& a, const AdjointArgs& b) {
    // the forward's work items: TPB * PPT particles each
    const int64_t items = (a.p.n + TPB * PPT - 1) / (TPB * PPT) + a.p.ntiles;
    k_g2p_adjoint<D, PPT, TPB, GENERAL, EXACT><<<unsigned(items), TPB, 0, a.stream>>>(
        a.state_in, a.perm, a.item_offset, a.p, a.gv, b.grad_out, b.grad_in, b.gstride, b.slots_b);
    return hipGetLastError();
}

template <int D, int PPT, int TPB>
static hipError_t g2p_adjoint_material(const LaunchArgs& a, const AdjointArgs& b) {
    if (a.material == MPM_JELLY) return g2p_adjoint_one<D, PPT, TPB, false, true>(a, b);
    // 2D SVDs have one method; in 3D the forward's choice
    if (D == 2 || (a.svd_mode != 1)) return g2p_adjoint_one<D, PPT, TPB, true, true>(a, b);
    return g2p_adjoint_one<D, PPT, TPB, true, false>(a, b);
}

// 3D: one particle per thread (a workgroup of chunk threads), at most 128 VGPRs and four waves per
// SIMD, where two particles per thread need 144 and fit three.  2D: likewise when the particles
// fill fewer work items than the chip has CUs (half the latency of a work item), else 256
// threads and chunk / 256 particles each, as P2G.
template <int D>
static hipError_t g2p_adjoint_dispatch(const LaunchArgs& a, const AdjointArgs& b) {
    if constexpr (D == 2) {
        if (a.p.n >= int64_t(kFewItems) * a.p.chunk) {
            switch (a.p.chunk) {
                case 256: return g2p_adjoint_material<D, 1, 256>(a, b);
                case 1024: return g2p_adjoint_material<D, 4, 256>(a, b);
                default: return g2p_adjoint_material<D, 2, 256>(a, b);
            }
        }
    }
    switch (a.p.chunk) {
        case 256: return g2p_adjoint_material<D, 1, 256>(a, b);
        case 1024: return g2p_adjoint_material<D, 1, 1024>(a, b);
        default: return g2p_adjoint_material<D, 1, 512>(a, b);
    }
}

hipError_t launch_g2p_adjoint(const LaunchArgs& a, const AdjointArgs& b) {
    if (a.p.n == 0) return hipSuccess;
    return a.dim == 2 ? g2p_adjoint_dispatch<2>(a, b) : g2p_adjoint_dispatch<3>(a, b);
}

template <int D, bool LISTED>
static hipError_t grid_adjoint_one(const LaunchArgs& a, const AdjointArgs& b) {
    const unsigned blocks = grid_tile_blocks(a.p.node_tiles);
    const auto* tiles = static_cast<const GridTile<D>*>(a.grid_tiles);
    if (a.gpre)
        k_grid_adjoint<D, true, LISTED><<<blocks, Tile<D>::NODES, 0, a.stream>>>(
            a.slots, b.slots_b, a.gpre, a.item_offset, a.p, tiles, a.meta, b.gbar);
    else
        k_grid_adjoint<D, false, LISTED><<<blocks, Tile<D>::NODES, 0, a.stream>>>(
            a.slots, b.slots_b, a.gpre, a.item_offset, a.p, tiles, a.meta, b.gbar);
    return hipGetLastError();
}

hipError_t launch_grid_adjoint(const LaunchArgs& a, const AdjointArgs& b) {
    const unsigned tiles = a.p.node_tiles;
    if (tiles == 0 || a.p.n == 0) return hipSuccess;
    if (!grid_tiles_listed(a.dim, a.p)) return grid_adjoint_one<2, false>(a, b);
    return a.dim == 2 ? grid_adjoint_one<2, true>(a, b) : grid_adjoint_one<3, true>(a, b);
}

hipError_t launch_p2g_adjoint(const LaunchArgs& a, const AdjointArgs& b) {
    if (a.p.n > 0) {
        const unsigned blocks = xcd_grid(blocks_of(a.p.n, 256));
        auto launch = [&](auto kernel) {
            kernel<<<blocks, 256, 0, a.stream>>>(a.state_in, a.pid_in, a.perm, a.keys, a.p, b.gbar, b.grad_out, b.grad_in,
                                                 b.gstride, b.epart, a.rot);
        };
        if (a.dim == 2) launch(k_p2g_adjoint<2, kSvdExact>);
        else if (a.svd_mode == kSvdAccurate) launch(k_p2g_adjoint<3, kSvdAccurate>);
        else launch(k_p2g_adjoint<3, kSvdExact>);  // R from either method
    }
    return hipGetLastError();
}

hipError_t launch_e_sum(const StepParams& p, const ESteps& es, int steps, int64_t* erange, double* epartial, int echunks,
                        double* grad_E, hipStream_t s) {
    if (p.n == 0 || steps <= 0 || !grad_E) return hipSuccess;
    // one scene: its range is [0, meta[0]), no search needed
    const int64_t* range = p.nscenes == 1 ? nullptr : erange;
    if (range) k_scene_ranges<<<dim3(unsigned(2 * p.nscenes), unsigned(steps)), 64, 0, s>>>(es, p, erange);
    k_scene_e_partial<<<dim3(unsigned(echunks), unsigned(p.nscenes), unsigned(steps)), 256, 0, s>>>(es, range, echunks,
                                                                                                epartial);
    k_scene_e_final<<<unsigned(p.nscenes), 1024, 0, s>>>(es, epartial, range, echunks, steps, grad_E);
    return hipGetLastError();
}

int e_chunks(int64_t n) { return int(std::max<int64_t>(1, (n + kEChunk - 1) / kEChunk)); }

}  // namespace nclr_host
