// awp_staged.hpp -- the two-stage kernels' tile bodies with every line loaded
// once.  A wave loads its own row of each array and writes what its
// neighbours need to LDS; a few more loads a level, dealt out over the waves
// (Halo), bring the rows and columns around the tile.  The loads of the next
// level are issued before the current one's arithmetic, one barrier a level.
//
// In the forms without LDS each row of a stencil array is loaded by up to four
// waves and at up to five x offsets: 31 loads a point and level in the velocity
// kernel, 49 (mixed 41) in the stress kernel.  Here a wave has 10 (stress: 19
// FP32, 17 mixed) for its own points and 1.8 (2.5, 2.0) for the surroundings;
// at 1500x1000x300 FP32 170M and 287M wave loads a launch become 95M and 166M.
// us per step, velocity / stress, without -> with: 1500x1000x300 FP32 5200 /
// 11980 -> 4790 / 11490, mixed 5016 / 9130 -> 4604 / 8727; 517x389x149 FP32
// 370 / 842 -> 335 / 788, mixed 356 / 658 -> 325 / 615.  That is 5.0 TB/s for
// the stress kernel, the rate of bare streams in its mix of reads and writes.
// The vector cache waits for lines on their way in both forms, for fewer loads
// a larger part of the time (TCP_PENDING_STALL_CYCLES, velocity / stress: 59 /
// 63 % of the cycles without, 79 / 81 % with): the time is the memory's.
// 64 x 8 tiles, as 64 x 4 spill scalar registers (the halo loads of five items
// a wave) and 64 x 16 wait at longer barriers (16.29 / 16.38 / 16.63 ms per
// step with 8 / 4 / 16 rows).
// Statements and their order are those of velocity_tile_b / stress_tile_b.
#pragma once
#include "awp_kernels.hpp"

namespace awp {

// One load a level for the surroundings of a tile, the same array for the
// whole wave: from byte offset `off` of `base` to float `dst` of the level's
// planes (or of its media slot).  A lane without a point reads the level's
// first element and writes to the padding, so that neither needs a mask.
struct Halo {
    const G<char> *base;
    unsigned off;
    int dst;
    int kind;   // the same in the whole wave: 0 nothing; 1 a plane; 2, 3 media
};

struct Staged {
    static constexpr int TY = STAGED_TY;
    static constexpr int RW = TX + 4, RH = TY + 4, PL = RW * RH;   // columns -2 .. 65, rows -2 .. TY+1
    static constexpr int MW = TX + 1, MPL = MW * (TY + 1);         // media: columns 0 .. 64, rows -1 .. TY-1
    static constexpr int PAD = 2 * TX;                             // floats behind each set of planes and media slot
};

// the lane's point (i0 + col, j0 + r) of an array of eb-byte elements, to
// float dst, or its substitute (float pad) where it has none
__device__ __forceinline__ void halo_at(Halo &h, const Geo &g, const int i0, const int j0, const int col, const int r,
                                        const bool has, const int eb, const int dst, const int pad)
{
    const bool on = has && i0 + col <= g.nx + 2 && j0 + r <= g.ny + 2;   // two ghost layers around the grid
    h.off = on ? (unsigned)(g.base + (long long)(j0 + r) * g.sy + i0 + col) * (unsigned)eb : 0u;
    h.dst = on ? dst : pad;
}
// row item: row r of the tile's neighbourhood over the wave's columns
__device__ __forceinline__ void halo_row(Halo &h, const Geo &g, const int i0, const int j0, const int lane,
                                         const int r, const int plane, const int npl, const int eb)
{
    using S = Staged;
    halo_at(h, g, i0, j0, lane, r, true, eb, plane * S::PL + (r + 2) * S::RW + lane + 2, npl * S::PL + lane);
}
// column item: columns c0, c1, c2 of the tile's rows
__device__ __forceinline__ void halo_cols(Halo &h, const Geo &g, const int i0, const int j0, const int lane,
                                          const int c0, const int c1, const int c2, const int plane, const int npl)
{
    using S = Staged;
    const int r = lane / 3, q = lane - 3 * r;
    const int col = q == 0 ? c0 : q == 1 ? c1 : c2;
    halo_at(h, g, i0, j0, col, r, r < S::TY, 4, plane * S::PL + (r + 2) * S::RW + col + 2, npl * S::PL + lane);
}

template <class P>
__device__ __forceinline__ void velocity_tile_s(const Geo &g, const State &s0, const Coef &c, const int kc, const int bx,
                                       const int by, const int bz, const Hook &hook)
{
    using S = Staged;
    constexpr int TY = S::TY, RW = S::RW, PL = S::PL;
    enum { XX, XY, YY, XZ, YZ, DD, NPL };
    constexpr int SET = NPL * PL + S::PAD;
    __shared__ float lds[2 * SET];
    const GState s = as_global(s0);
    using M = typename P::M;
    constexpr int NS = (14 + TY - 1) / TY;
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int i0 = bx * TX + 1, j0 = by * TY + 1;
    const int i = i0 + lane, j = j0 + wv;
    const int kb = bz * kc + 1;
    const int ke = min(kb + kc - 1, g.nz);
    const bool act = i <= g.nx && j <= g.ny;
    const bool ldok = i <= g.nx + 2 && j <= g.ny + 2;   // two ghost layers around the grid
    Cursor32 p(g, g.base + (long long)kb * g.sz + (long long)j * g.sy + i);
    const unsigned sz4 = p.sz;
    const int lpos = (wv + 2) * RW + lane + 2;
    const G<M> *d1 = (const G<M> *)s.d1;
    const float c1 = c.c1, c2 = c.c2, dth = c.dth;
    const float fxy = act ? s.fx[i] * s.fy[j] : 0.0f;

    Halo hl[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        Halo &h = hl[t];
        const int q = wv + t * TY;
        h.kind = q < 12 ? 1 : q < 14 ? 3 : 0;
        h.base = (const G<char> *)(q <= 2 || q == 10 ? s.xy : q <= 5 ? s.yy : q <= 8 ? s.yz : q == 9 ? s.xx : s.xz);
        if (q < 9) {
            const int r = q == 0 || q == 6 ? -2 : q == 1 || q == 3 || q == 7 ? -1 : q == 5 ? TY + 1 : TY;
            halo_row(h, g, i0, j0, lane, r, q <= 2 ? XY : q <= 5 ? YY : YZ, NPL, 4);
        } else if (q < 12) {
            halo_cols(h, g, i0, j0, lane, q == 9 ? -2 : -1, q == 9 ? -1 : 64, q == 9 ? 64 : 65,
                          q == 9 ? XX : q == 10 ? XY : XZ, NPL);
        } else if (q == 12) {
            h.base = (const G<char> *)d1;
            halo_row(h, g, i0, j0, lane, -1, DD, NPL, (int)sizeof(M));
        } else {
            h.base = (const G<char> *)d1;
            const int r = lane - 1;
            halo_at(h, g, i0, j0, TX, r, r < TY, (int)sizeof(M), DD * PL + (r + 2) * RW + TX + 2, NPL * PL + lane);
        }
        // at level kb; a 2-byte array steps half as far
        h.off += (unsigned)kb * (h.kind == 3 && sizeof(M) == 2 ? sz4 / 2 : sz4);
    }
    auto load_halo = [&](const Halo &h) -> float {
        if (sizeof(M) == 2 && h.kind == 3)
            return __uint_as_float((unsigned)__builtin_bit_cast(unsigned short, (_Float16)*(const G<M> *)(h.base + h.off)));
        return *(const G<float> *)(h.base + h.off);
    };
    // a loaded value as the planes hold it
    auto halo_val = [&](const Halo &h, const float x, const float db) -> float {
        if (sizeof(M) == 2 && h.kind == 3)
            return mdec((M)__builtin_bit_cast(_Float16, (unsigned short)__float_as_uint(x)), db);
        return x;
    };
    auto mbar = [&](int k) -> float { return P::mixed ? s.mbar[mbar_idx(g, 0, k)] : 0.0f; };

    // z queues at the column, and the first level's own values
    float xz_m2 = 0.f, xz_m1 = 0.f, xz_0 = 0.f, xz_p1 = 0.f, yz_m2 = 0.f, yz_m1 = 0.f, yz_0 = 0.f, yz_p1 = 0.f;
    float zz_m1 = 0.f, zz_0 = 0.f, zz_p1 = 0.f, zz_p2 = 0.f;
    float dA_m = 1.f, dB_m = 1.f, dC_m = 1.f;
    float xx = 0.f, xy = 0.f, yy = 0.f, u0 = 0.f, v0 = 0.f, w0 = 0.f, hv[NS];
    M dr = (M)0.0f;
    if (ldok) {
        xz_m2 = p.ld(s.xz, 0, 0, -2); xz_m1 = p.ld(s.xz, 0, 0, -1); xz_0 = p.ld(s.xz); xz_p1 = p.ld(s.xz, 0, 0, 1);
        yz_m2 = p.ld(s.yz, 0, 0, -2); yz_m1 = p.ld(s.yz, 0, 0, -1); yz_0 = p.ld(s.yz); yz_p1 = p.ld(s.yz, 0, 0, 1);
        zz_m1 = p.ld(s.zz, 0, 0, -1); zz_0 = p.ld(s.zz); zz_p1 = p.ld(s.zz, 0, 0, 1);
        zz_p2 = p.template ldu<P::nt>(s.zz, 2);
        xx = p.ld(s.xx); xy = p.ld(s.xy); yy = p.ld(s.yy); dr = p.ld(d1);
    }
    if (act) {
        const float db = mbar(kb - 1);
        dA_m = mdec(p.ld(d1, 0, 0, -1), db); dB_m = mdec(p.ld(d1, 0, -1, -1), db); dC_m = mdec(p.ld(d1, 1, 0, -1), db);
        u0 = p.template ldn<P::nt>(s.u1); v0 = p.template ldn<P::nt>(s.v1); w0 = p.template ldn<P::nt>(s.w1);
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) hv[t] = hl[t].kind ? load_halo(hl[t]) : 0.0f;
    float mb = mbar(kb), fz = s.fz[kb];
    // a level's planes, from what was loaded for it
    auto put_planes = [&](const int k, const float d) {
        float *pl = lds + (k & 1) * SET;
        pl[XX * PL + lpos] = xx;
        pl[XY * PL + lpos] = xy;
        pl[YY * PL + lpos] = yy;
        pl[XZ * PL + lpos] = xz_0;
        pl[YZ * PL + lpos] = yz_0;
        pl[DD * PL + lpos] = d;
#pragma unroll
        for (int t = 0; t < NS; ++t)
            if (hl[t].kind) pl[hl[t].dst] = halo_val(hl[t], hv[t], mb);
    };
    for (int k = kb; k <= ke; ++k, p.up()) {
        const float dA = mdec(dr, mb);
        put_planes(k, dA);
        // the next level's loads
        const float xy_0 = xy, xx_0 = xx, yy_0 = yy;
        const float fzn = s.fz[min(k + 1, g.nz)];
        float xz_n = 0.f, yz_n = 0.f, zz_n = 0.f, un = 0.f, vn = 0.f, wn = 0.f;
        if (k < ke) {
            if (ldok) {
                xx = p.ld(s.xx, 0, 0, 1); xy = p.ld(s.xy, 0, 0, 1); yy = p.ld(s.yy, 0, 0, 1); dr = p.ld(d1, 0, 0, 1);
                xz_n = p.ld(s.xz, 0, 0, 2); yz_n = p.ld(s.yz, 0, 0, 2);
                zz_n = p.template ldu<P::nt>(s.zz, 3);
            }
            if (act) {
                un = p.template ldu<P::nt>(s.u1, 1); vn = p.template ldu<P::nt>(s.v1, 1);
                wn = p.template ldu<P::nt>(s.w1, 1);
            }
            mb = mbar(k + 1);
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                hl[t].off += hl[t].kind == 3 && sizeof(M) == 2 ? sz4 / 2 : sz4;
                if (hl[t].kind) hv[t] = load_halo(hl[t]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        const float *pl = lds + (k & 1) * SET;
        const float *pxx = pl + XX * PL + lpos, *pxy = pl + XY * PL + lpos, *pyy = pl + YY * PL + lpos;
        const float *pxz = pl + XZ * PL + lpos, *pyz = pl + YZ * PL + lpos, *pd = pl + DD * PL + lpos;
        const float dB = pd[-RW], dC = pd[1], dD = pd[1 - RW];
        const float xx_m1 = pxx[-1], xx_p1 = pxx[1], xx_m2 = pxx[-2];
        const float xy_jm1 = pxy[-RW], xy_jp1 = pxy[RW], xy_jm2 = pxy[-2 * RW];
        const float xy_ip1 = pxy[1], xy_ip2 = pxy[2], xy_im1 = pxy[-1];
        const float yy_jp1 = pyy[RW], yy_jp2 = pyy[2 * RW], yy_jm1 = pyy[-RW];
        const float xz_ip1 = pxz[1], xz_ip2 = pxz[2], xz_im1 = pxz[-1];
        const float yz_jm1 = pyz[-RW], yz_jp1 = pyz[RW], yz_jm2 = pyz[-2 * RW];
        if (act) {
            if (k == hook.k || k == hook.tk) hook_velocity(hook, i, j, k, dA, u0, v0, w0);
            float d, q, u, v, w;
            d = 0.25f * ((dA + dB) + (dA_m + dB_m));
            q = dth / d;
            u = u0 + q * (
                c1 * (xx_0 - xx_m1) + c2 * (xx_p1 - xx_m2) +
                c1 * (xy_0 - xy_jm1) + c2 * (xy_jp1 - xy_jm2) +
                c1 * (xz_0 - xz_m1) + c2 * (xz_p1 - xz_m2));
            d = 0.25f * ((dA + dC) + (dA_m + dC_m));
            q = dth / d;
            v = v0 + q * (
                c1 * (xy_ip1 - xy_0) + c2 * (xy_ip2 - xy_im1) +
                c1 * (yy_jp1 - yy_0) + c2 * (yy_jp2 - yy_jm1) +
                c1 * (yz_0 - yz_m1) + c2 * (yz_p1 - yz_m2));
            d = 0.25f * ((dA + dC) + (dB + dD));
            q = dth / d;
            w = w0 + q * (
                c1 * (xz_ip1 - xz_0) + c2 * (xz_ip2 - xz_im1) +
                c1 * (yz_0 - yz_jm1) + c2 * (yz_jp1 - yz_jm2) +
                c1 * (zz_p1 - zz_0) + c2 * (zz_p2 - zz_m1));
            const float D = fxy * fz;
            p.template stn<P::nt>(s.u1, u * D);
            p.template stn<P::nt>(s.v1, v * D);
            p.template stn<P::nt>(s.w1, w * D);
        }
        xz_m2 = xz_m1; xz_m1 = xz_0; xz_0 = xz_p1; xz_p1 = xz_n;
        yz_m2 = yz_m1; yz_m1 = yz_0; yz_0 = yz_p1; yz_p1 = yz_n;
        zz_m1 = zz_0; zz_0 = zz_p1; zz_p1 = zz_p2; zz_p2 = zz_n;
        dA_m = dA; dB_m = dB; dC_m = dC;
        fz = fzn;
        u0 = un; v0 = vn; w0 = wn;
    }
}

template <class P>
__device__ __forceinline__ void stress_tile_s(const Geo &g, const State &s0, const Coef &c, const int kc, const int bx,
                                     const int by, const int bz, const Hook &hook)
{
    using S = Staged;
    using F4 = float __attribute__((ext_vector_type(4)));
    constexpr int TY = S::TY, RW = S::RW, PL = S::PL, MW = S::MW, MPL = S::MPL;
    enum { U, V, W, NPL };
    constexpr int SET = NPL * PL + S::PAD, MSET = MPL + S::PAD / 4;
    __shared__ float lds[2 * SET];
    __shared__ F4 med[3 * MSET];
    const GState s = as_global(s0);
    using R = typename P::R;
    using M = typename P::M;
    using Q = typename P::Q;
    constexpr int NI = P::mixed ? 16 : 20, NS = (NI + TY - 1) / TY;
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int i0 = bx * TX + 1, j0 = by * TY + 1;
    const int i = i0 + lane, j = j0 + wv, seg = bx;
    const int kb = bz * kc + 1;
    const int ke = min(kb + kc - 1, g.nz);
    const bool row = j <= g.ny;                           // the wave's row lies in the grid
    const bool act = i <= g.nx && row;
    const bool ldok = i <= g.nx + 2 && j <= g.ny + 2;   // two ghost layers around the grid
    Cursor32 p(g, g.base + (long long)kb * g.sz + (long long)j * g.sy + i);
    const unsigned sz4 = p.sz;
    const int lpos = (wv + 2) * RW + lane + 2, mpos = (wv + 1) * MW + lane;
    const G<M> *lam = (const G<M> *)s.lam;
    const G<M> *mu = (const G<M> *)s.mu;
    const G<unsigned> *mlq = (const G<unsigned> *)s.mu;   // mixed: (mu, lam) pairs
    const G<Q> *qp = (const G<Q> *)s.qp;
    const G<Q> *qs = (const G<Q> *)s.qs;
    const G<unsigned> *qq = (const G<unsigned> *)s.qp;    // mixed: (qp, qs) pairs
    G<R> *const RR[6] = {(G<R> *)s.r1, (G<R> *)s.r2, (G<R> *)s.r3, (G<R> *)s.r4, (G<R> *)s.r5, (G<R> *)s.r6};
    G<float> *const SS[6] = {s.xx, s.yy, s.zz, s.xy, s.xz, s.yz};
    const float c1 = c.c1, c2 = c.c2, dth = c.dth, dt = c.dt, dh1 = c.dh1;
    const float fxy = act ? s.fx[i] * s.fy[j] : 0.0f;
    const int itxy = ((i & 1) * 2 + (j & 1)) * 2;
    const float t1e = c.tau1[itxy], t1o = c.tau1[itxy + 1];
    const float t2e = c.tau2[itxy], t2o = c.tau2[itxy + 1];

    Halo hl[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        Halo &h = hl[t];
        const int q = wv + t * TY;
        h.kind = 1;
        if (q < 9) {
            const int a = q == 0 || q == 2 || q == 5 ? V : q == 3 || q == 6 || q == 8 ? W : U;
            const int r = q == 0 ? -2 : q <= 3 ? -1 : q <= 6 ? TY : TY + 1;
            h.base = (const G<char> *)(a == U ? s.u1 : a == V ? s.v1 : s.w1);
            halo_row(h, g, i0, j0, lane, r, a, NPL, 4);
        } else if (q < 12) {
            h.base = (const G<char> *)(q == 9 ? s.u1 : q == 10 ? s.v1 : s.w1);
            halo_cols(h, g, i0, j0, lane, q == 9 ? -1 : -2, q == 9 ? 64 : -1, q == 9 ? 65 : 64, q - 9, NPL);
        } else {
            // media (4-byte elements in both modes): row -1, then column 64
            constexpr int NM = P::mixed ? 2 : 4;
            const int n = q - 12, a = n % NM, r = n < NM ? -1 : lane - 1, col = n < NM ? lane : TX;
            if constexpr (P::mixed)
                h.base = (const G<char> *)(a == 0 ? mlq : qq);
            else
                h.base = (const G<char> *)(a == 0 ? lam : a == 1 ? mu : a == 2 ? qp : qs);
            h.kind = q >= NI ? 0 : a == 0 ? 2 : 3;
            halo_at(h, g, i0, j0, col, r, r < TY, 4, 4 * ((r + 1) * MW + col) + (P::mixed ? 2 * a : a),
                    4 * MPL + 2 * lane);
        }
        h.off += (unsigned)(kb - 1) * sz4;
    }
    auto load_halo = [&](const Halo &h) -> float { return *(const G<float> *)(h.base + h.off); };
    // a media value of level k to its place: FP32 as it is, a mixed pair decoded
    auto put_media = [&](float *m, const float x, const float mb, const float lb, const bool first) {
        if constexpr (P::mixed) {
            const unsigned w = __float_as_uint(x);
            m[0] = first ? mdec(h_hi(w), lb) : q_lo(w);
            m[1] = first ? mdec(h_lo(w), mb) : q_hi(w);
        } else {
            m[0] = x;
        }
    };
    auto put_halo = [&](const Halo &h, const float x, float *pl, F4 *ms, const float mb, const float lb) {
        if (h.kind == 1)
            pl[h.dst] = x;
        else if (h.kind)
            put_media((float *)ms + h.dst, x, mb, lb, h.kind == 2);
    };
    struct Med {
        float x, y, z, w;   // mixed: the two words in x, y
    };
    auto load_media = [&](const int dk) -> Med {
        Med m = {0.f, 0.f, 0.f, 0.f};
        if (!ldok) return m;
        if constexpr (P::mixed) {
            m.x = __uint_as_float(p.template ldu<P::ntm>(mlq, dk));
            m.y = __uint_as_float(p.template ldu<P::ntm>(qq, dk));
        } else {
            m.x = p.template ldu<P::ntm>(lam, dk); m.y = p.template ldu<P::ntm>(mu, dk);
            m.z = p.template ldu<P::ntm>(qp, dk); m.w = p.template ldu<P::ntm>(qs, dk);
        }
        return m;
    };
    auto media_of = [&](const Med &m, const float mb, const float lb) -> F4 {
        if constexpr (P::mixed) {
            const unsigned w = __float_as_uint(m.x), q = __float_as_uint(m.y);
            return F4{mdec(h_hi(w), lb), mdec(h_lo(w), mb), q_lo(q), q_hi(q)};
        } else {
            return F4{m.x, m.y, m.z, m.w};
        }
    };

    // z queues of the velocities at the column
    float u_m1 = 0.f, u_0 = 0.f, u_p1 = 0.f, u_p2 = 0.f, v_m1 = 0.f, v_0 = 0.f, v_p1 = 0.f, v_p2 = 0.f;
    float w_m2 = 0.f, w_m1 = 0.f, w_0 = 0.f, w_p1 = 0.f;
    R rr[6];
    float ss[6];
    if (ldok) {
        u_m1 = p.ld(s.u1, 0, 0, -1); u_0 = p.ld(s.u1); u_p1 = p.ld(s.u1, 0, 0, 1); u_p2 = p.ld(s.u1, 0, 0, 2);
        v_m1 = p.ld(s.v1, 0, 0, -1); v_0 = p.ld(s.v1); v_p1 = p.ld(s.v1, 0, 0, 1); v_p2 = p.ld(s.v1, 0, 0, 2);
        w_m2 = p.ld(s.w1, 0, 0, -2); w_m1 = p.ld(s.w1, 0, 0, -1); w_0 = p.ld(s.w1); w_p1 = p.ld(s.w1, 0, 0, 1);
    }
    const Med m_1 = load_media(-1);
    Med mn = load_media(0);
    float hv[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) hv[t] = hl[t].kind ? load_halo(hl[t]) : 0.0f;
    // (not needed for the LDS, which nothing has touched yet: it lines up the
    // waves after their start-up loads, mixed 400x300x150 382 us against 384
    // without it, FP32 and larger grids the same within 0.1 %)
    __syncthreads();
    int m0 = kb % 3, mp = (kb + 2) % 3;   // media slots of levels k and k-1
    float mb0 = 0.f, lb0 = 0.f;
    if constexpr (P::mixed) { mb0 = s.mbar[mbar_idx(g, 1, kb - 1)]; lb0 = s.mbar[mbar_idx(g, 2, kb - 1)]; }
    med[mp * MSET + mpos] = media_of(m_1, mb0, lb0);
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        if (hl[t].kind > 1) put_halo(hl[t], hv[t], lds, med + mp * MSET, mb0, lb0);
        hl[t].off += sz4;
        if (hl[t].kind) hv[t] = load_halo(hl[t]);
    }
    // r and the stresses dk levels up
    auto load_own = [&](const int dk) {
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            rr[n] = p.template ldu<P::ntr>(RR[n], dk);
            ss[n] = p.template ldu<P::nt>(SS[n], dk);
        }
    };
    if (act) load_own(0);
    // final xz/yz/zz of the two levels below (for the free-surface images)
    float xz_f1 = 0.f, xz_f2 = 0.f, yz_f1 = 0.f, yz_f2 = 0.f, zz_f1 = 0.f;
    long long slot = P::mixed ? rexp_idx(g, s.nseg, seg, min(j, g.ny), kb) : 0;
    const long long sstep = (long long)g.ny * s.nseg;
    unsigned long long ewn = 0;   // mixed: the next level's exponents
    if constexpr (P::mixed) {
        if (row) ewn = rexp_load(s.rexp, slot);
    }
    float fzn = s.fz[kb], mbn = 0.f, lbn = 0.f;
    if constexpr (P::mixed) { mbn = s.mbar[mbar_idx(g, 1, kb)]; lbn = s.mbar[mbar_idx(g, 2, kb)]; }

    // a level's planes and media, from what was loaded for it
    auto put_planes = [&](const int k, const int slot3, const float u, const float v, const float w) {
        float *pl = lds + (k & 1) * SET;
        pl[U * PL + lpos] = u;
        pl[V * PL + lpos] = v;
        pl[W * PL + lpos] = w;
        med[slot3 * MSET + mpos] = media_of(mn, mbn, lbn);
#pragma unroll
        for (int t = 0; t < NS; ++t) put_halo(hl[t], hv[t], pl, med + slot3 * MSET, mbn, lbn);
    };
    // Where the planes of a level are written.  Mixed: at the end of the level
    // before, ahead of its stores, and only then the loads of r and the
    // stresses: the wait for the planes' loads is then not one for those and
    // for the stores.  FP32: at the top of the level, with r and the stresses
    // loaded as soon as the level before has read its own -- these bytes, half
    // as many again as in mixed storage, need the longer way.  us per step of
    // the stress kernel, at the end / at the top: FP32 200x200x100 115 / 106,
    // 400x300x150 459 / 457, 800x600x200 2390 / 2373, mixed 100 / 103, 383 /
    // 408, 1846 / 1905.
    constexpr bool AHEAD = P::mixed;
    if constexpr (AHEAD) put_planes(kb, m0, u_0, v_0, w_0);

    for (int k = kb; k <= ke; ++k, p.up(), slot += sstep) {
        if constexpr (!AHEAD) put_planes(k, m0, u_0, v_0, w_0);
        // mixed: the row segment's exponents before this update
        const unsigned long long ew = ewn;
        const float fz = fzn;
        if constexpr (AHEAD) __syncthreads();
        // the next level's loads
        float un = 0.f, vn = 0.f, wn = 0.f;
        if (k < ke) {
            mn = load_media(1);
            fzn = s.fz[k + 1];
            if constexpr (P::mixed) {
                if (row) ewn = rexp_load(s.rexp, slot + sstep);
                mbn = s.mbar[mbar_idx(g, 1, k + 1)];
                lbn = s.mbar[mbar_idx(g, 2, k + 1)];
            }
            if (ldok) {
                un = p.ld(s.u1, 0, 0, 3);
                vn = p.ld(s.v1, 0, 0, 3);
                wn = p.ld(s.w1, 0, 0, 2);
            }
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                hl[t].off += sz4;
                if (hl[t].kind) hv[t] = load_halo(hl[t]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!AHEAD) __syncthreads();
        const float *pl = lds + (k & 1) * SET;
        if (k == g.nz - 1 && act) {
            // the images at nz+1 (the top chunk spans at least three levels,
            // so this level is met before any that reads them)
            float ut, vt, wt;
            fs_images<P>(g, s, i, j, [&](const auto *a, int di, int dj, int dk) { return p.ld(a, di, dj, dk + 1); }, ut, vt, wt);
            u_p2 = ut;
            v_p2 = vt;
            wn = wt;   // w_p1 at k = nz
            p.st(s.u1, ut, 0, 0, 2);
            p.st(s.v1, vt, 0, 0, 2);
            p.st(s.w1, wt, 0, 0, 2);
        }
        float r1 = 0.f, r2 = 0.f, r3 = 0.f, r4 = 0.f, r5 = 0.f, r6 = 0.f;
        float xx = 0.f, yy = 0.f, zz = 0.f, xy = 0.f, xz = 0.f, yz = 0.f;
        if (act) {
            // media of the 2x2 cell: A (i, j), B (i+1, j), C (i, j-1), D (i+1, j-1)
            const F4 *ms = med + m0 * MSET + mpos, *mm = med + mp * MSET + mpos;
            const F4 A = ms[0], B = ms[1], C = ms[-MW], D = ms[1 - MW];
            const F4 Am = mm[0], Bm = mm[1], Cm = mm[-MW], Dm = mm[1 - MW];
            float vxl = 8.0f / (A.x + B.x + C.x + D.x + Am.x + Bm.x + Cm.x + Dm.x);
            const float vxm = 8.0f / (A.y + B.y + C.y + D.y + Am.y + Bm.y + Cm.y + Dm.y);
            vxl = vxl + 2.0f * vxm;
            float vqpa = 0.125f * (A.z + B.z + C.z + D.z + Am.z + Bm.z + Cm.z + Dm.z);
            float vqsa = 0.125f * (A.w + B.w + C.w + D.w + Am.w + Bm.w + Cm.w + Dm.w);
            const float vx4 = 2.0f / (A.y + Am.y), vx5 = 2.0f / (A.y + C.y), vx6 = 2.0f / (A.y + B.y);
            float va4 = 0.5f * (A.w + Am.w), va5 = 0.5f * (A.w + C.w), va6 = 0.5f * (A.w + B.w);
            if constexpr (P::mixed) {
                vqpa = vqpa * s.ms.iqp;
                vqsa = vqsa * s.ms.iqs;
                va4 = va4 * s.ms.iqs;
                va5 = va5 * s.ms.iqs;
                va6 = va6 * s.ms.iqs;
            }
            const float vh2_r4 = -va4 * vx4 / 2.0f, vh2_r5 = -va5 * vx5 / 2.0f, vh2_r6 = -va6 * vx6 / 2.0f;

            const float *pu = pl + U * PL + lpos, *pv = pl + V * PL + lpos, *pw = pl + W * PL + lpos;
            const float vt1 = c1 * (pu[1] - u_0) + c2 * (pu[2] - pu[-1]);
            const float vt2 = c1 * (v_0 - pv[-RW]) + c2 * (pv[RW] - pv[-2 * RW]);
            const float vt3 = c1 * (w_0 - w_m1) + c2 * (w_p1 - w_m2);
            const float vt4 = c1 * (pu[RW] - u_0) + c2 * (pu[2 * RW] - pu[-RW]) +
                              c1 * (v_0 - pv[-1]) + c2 * (pv[1] - pv[-2]);
            const float vt5 = c1 * (u_p1 - u_0) + c2 * (u_p2 - u_m1) +
                              c1 * (w_0 - pw[-1]) + c2 * (pw[1] - pw[-2]);
            const float vt6 = c1 * (v_p1 - v_0) + c2 * (v_p2 - v_m1);
            const float vt7 = c1 * (pw[RW] - w_0) + c2 * (pw[2 * RW] - pw[-RW]);

            const bool odd = (((g.nz + 1) - k) & 1) != 0;
            const float vx1 = odd ? t1o : t1e;
            const float vx2 = odd ? t2o : t2e;
            const float vh1 = -vxm * vqsa;
            const float vtmp = vxl * (vt1 + vt2 + vt3);
            const float va1 = -vqpa * vxl * dh1 * (vt1 + vt2 + vt3) / 2.0f;

            if constexpr (P::mixed) {
                r1 = r_decode(rr[0], rexp_of(ew, 0)); r2 = r_decode(rr[1], rexp_of(ew, 1));
                r3 = r_decode(rr[2], rexp_of(ew, 2)); r4 = r_decode(rr[3], rexp_of(ew, 3));
                r5 = r_decode(rr[4], rexp_of(ew, 4)); r6 = r_decode(rr[5], rexp_of(ew, 5));
            } else {
                r1 = rr[0]; r2 = rr[1]; r3 = rr[2]; r4 = rr[3]; r5 = rr[4]; r6 = rr[5];
            }
            xx = ss[0]; yy = ss[1]; zz = ss[2]; xy = ss[3]; xz = ss[4]; yz = ss[5];

            xx = xx + dth * (vtmp - 2.0f * vxm * (vt2 + vt3)) + dt * r1;
            yy = yy + dth * (vtmp - 2.0f * vxm * (vt1 + vt3)) + dt * r2;
            zz = zz + dth * (vtmp - 2.0f * vxm * (vt1 + vt2)) + dt * r3;
            xy = xy + vx4 * dth * vt4 + dt * r4;
            xz = xz + vx5 * dth * vt5 + dt * r5;
            yz = yz + vx6 * (dth * vt6 + dth * vt7) + dt * r6;

            r1 = (vx2 * r1 - vh1 * (vt2 + vt3) * dh1 + va1) * vx1;
            r2 = (vx2 * r2 - vh1 * (vt1 + vt3) * dh1 + va1) * vx1;
            r3 = (vx2 * r3 - vh1 * (vt1 + vt2) * dh1 + va1) * vx1;
            r4 = (vx2 * r4 + vh2_r4 * dh1 * vt4) * vx1;
            r5 = (vx2 * r5 + vh2_r5 * dh1 * vt5) * vx1;
            r6 = (vx2 * r6 + vh2_r6 * dh1 * (vt6 + vt7)) * vx1;

            xx = xx + dt * r1;
            yy = yy + dt * r2;
            zz = zz + dt * r3;
            xy = xy + dt * r4;
            xz = xz + dt * r5;
            yz = yz + dt * r6;

            const float Ds = fxy * fz;
            xx = xx * Ds; yy = yy * Ds; zz = zz * Ds;
            xz = xz * Ds; yz = yz * Ds; xy = xy * Ds;
            if (!AHEAD && k < ke) load_own(1);
        }
        const int mq = m0 == 2 ? 0 : m0 + 1;
        if constexpr (AHEAD) {
            __builtin_amdgcn_sched_barrier(0);
            if (k < ke) {
                put_planes(k + 1, mq, u_p1, v_p1, w_p1);
                if (act) load_own(1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // the new memory variables enter this step's stresses in FP32 and
        // are rounded to the storage format once, on the store
        if constexpr (P::mixed) {
            if (row) {
                const float rv[6] = {r1, r2, r3, r4, r5, r6};
                const unsigned long long en = row_exponents6(rv, act, ew);
#pragma unroll
                for (int q = 0; q < 6; ++q)
                    if (act) p.template stn<P::ntr>(RR[q], (R)r_encode(rv[q], rexp_of(en, q)));
                if (lane == 0) nt_st<P::nt>((G<unsigned long long> *)s.rexp + slot, en);
            }
        } else if (act) {
            p.template stn<P::ntr>(RR[0], (R)r1); p.template stn<P::ntr>(RR[1], (R)r2);
            p.template stn<P::ntr>(RR[2], (R)r3); p.template stn<P::ntr>(RR[3], (R)r4);
            p.template stn<P::ntr>(RR[4], (R)r5); p.template stn<P::ntr>(RR[5], (R)r6);
        }
        if (act) {
            p.template stn<P::nt>(s.xx, xx); p.template stn<P::nt>(s.yy, yy); p.template stn<P::nt>(s.xy, xy);
            if (k == g.nz) {
                // fstr: images above the surface, xz = yz = 0 on it
                p.st(s.zz, zz);
                p.st(s.zz, -zz, 0, 0, 1);
                p.st(s.zz, -zz_f1, 0, 0, 2);
                p.st(s.xz, 0.0f);
                p.st(s.yz, 0.0f);
                p.st(s.xz, -xz_f1, 0, 0, 1);
                p.st(s.xz, -xz_f2, 0, 0, 2);
                p.st(s.yz, -yz_f1, 0, 0, 1);
                p.st(s.yz, -yz_f2, 0, 0, 2);
                hook_stress(hook, s, i, j, [&](const auto *a, int dk) { return p.ld(a, 0, 0, dk); },
                            [&](auto *a, float v, int dk) { p.st(a, v, 0, 0, dk); });
            } else {
                p.template stn<P::nt>(s.zz, zz); p.template stn<P::nt>(s.xz, xz); p.template stn<P::nt>(s.yz, yz);
            }
        }
        xz_f2 = xz_f1; xz_f1 = xz;
        yz_f2 = yz_f1; yz_f1 = yz;
        zz_f1 = zz;
        u_m1 = u_0; u_0 = u_p1; u_p1 = u_p2; u_p2 = un;
        v_m1 = v_0; v_0 = v_p1; v_p1 = v_p2; v_p2 = vn;
        w_m2 = w_m1; w_m1 = w_0; w_0 = w_p1; w_p1 = wn;
        mp = m0;
        m0 = mq;
    }
}

}  // namespace awp
