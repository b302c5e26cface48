// The far field's Green's function at one mode of the half spectrum.
#pragma once
#include "fsd_internal.h"

// Mobility_WaveSpace_Green_kernel (Mobility.cu:315-479) on the half spectrum.
// Field order: Fx Fy Fz | C_xx C_xy C_xz C_yz C_yy C_yx C_zx C_zy.
__device__ inline void green_apply(const float4 tk, bool origin, const float2 v[11], float2 o[11])
{
#pragma unroll
    for (int c = 0; c < 11; ++c) o[c] = make_float2(0.f, 0.f);
    if (origin) return;
    const float k[3] = {tk.x, tk.y, tk.z};
    const float ksq = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
    const float kk = sqrtf(ksq);
    // couplet matrix rows (x, y, z)
    const float2 Cm[3][3] = {{v[3], v[4], v[5]}, {v[8], v[7], v[6]}, {v[9], v[10], make_float2(-(v[3].x + v[7].x), -(v[3].y + v[7].y))}};
    float2 kdF;
    kdF.x = (k[0] * v[0].x + k[1] * v[1].x + k[2] * v[2].x) / ksq;
    kdF.y = (k[0] * v[0].y + k[1] * v[1].y + k[2] * v[2].y) / ksq;
    float2 Cdk[3];
    for (int a = 0; a < 3; ++a) {
        Cdk[a].x = Cm[a][0].x * k[0] + Cm[a][1].x * k[1] + Cm[a][2].x * k[2];
        Cdk[a].y = Cm[a][0].y * k[0] + Cm[a][1].y * k[1] + Cm[a][2].y * k[2];
    }
    float2 kCk;
    kCk.x = (Cdk[0].x * k[0] + Cdk[1].x * k[1] + Cdk[2].x * k[2]) / ksq;
    kCk.y = (Cdk[0].y * k[0] + Cdk[1].y * k[1] + Cdk[2].y * k[2]) / ksq;
    const float sk = sinf(kk), ck = cosf(kk);
    const float j0 = sk / kk;
    const float jt = 3.0f * (sk - kk * ck) / (ksq * kk);
    const float Buf = tk.w * j0 * j0;
    const float Buc = -tk.w * j0 * jt;        // UC (imaginary coupling)
    const float Bdf = tk.w * j0 * jt;         // DF (imaginary coupling)
    const float q = (sk - kk * ck) / (ksq * kk);
    const float Bdc = tk.w * 9.0f * q * q;    // DC
    for (int a = 0; a < 3; ++a) {
        float2 ff = v[a];
        float2 u;
        u.x = (ff.x - k[a] * kdF.x) * Buf;
        u.y = (ff.y - k[a] * kdF.y) * Buf;
        // + i (Cdk_a - k_a kCk) Buc
        u.x += -(Cdk[a].y - k[a] * kCk.y) * Buc;
        u.y += (Cdk[a].x - k[a] * kCk.x) * Buc;
        o[a] = u;
    }
    // gradient slots in field order: (x,x) (x,y) (x,z) (y,z) (y,y) (y,x) (z,x) (z,y)
    const int sa[8] = {0, 0, 0, 1, 1, 1, 2, 2}, sc[8] = {0, 1, 2, 2, 1, 0, 0, 1};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int a = sa[s], c = sc[s];
        const float kk_ac = k[a] * k[c];
        float2 z;
        z.x = v[a].x * k[c] - kk_ac * kdF.x;
        z.y = v[a].y * k[c] - kk_ac * kdF.y;
        float2 d;
        d.x = -z.y * Bdf + (Cdk[a].x * k[c] - kk_ac * kCk.x) * Bdc;
        d.y = z.x * Bdf + (Cdk[a].y * k[c] - kk_ac * kCk.y) * Bdc;
        o[3 + s] = d;
    }
}

struct GreenGeom {
    int Nx, Ny, Nz;
    BoxF b;
    float xi, eta, twopi_k;
};

// v <- G v at mode (i, j, k).  The spread grid is real, so its spectrum at the conjugate mode is
// conj(v); modes with a Nyquist index get the Hermitian part of the two outputs
__device__ __forceinline__ void green_update(const GreenGeom &g, const float4 *gk, int i, int j, int k, float2 v[11])
{
    const int64_t id = ((int64_t)i * g.Ny + j) * (g.Nz / 2 + 1) + k;
    float2 o[11];
    green_apply(gk[id], id == 0, v, o);
    if (has_nyquist(i, j, k, g.Nx, g.Ny, g.Nz)) {
        const int ic = (g.Nx - i) % g.Nx, jc = (g.Ny - j) % g.Ny, kc = (g.Nz - k) % g.Nz;
        const float4 tkc = gridk_value(ic, jc, kc, g.Nx, g.Ny, g.Nz, g.b, g.xi, g.eta, g.twopi_k);
        float2 vc[11], oc[11];
#pragma unroll
        for (int c = 0; c < 11; ++c) vc[c] = make_float2(v[c].x, -v[c].y);
        green_apply(tkc, false, vc, oc);
#pragma unroll
        for (int c = 0; c < 11; ++c) o[c] = make_float2(0.5f * (o[c].x + oc[c].x), 0.5f * (o[c].y - oc[c].y));
    }
#pragma unroll
    for (int c = 0; c < 11; ++c) v[c] = o[c];
}
