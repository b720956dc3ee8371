// awp_sweep.hpp -- the fused step's tile body for FP32 storage on 64 x 11
// tiles, every line loaded once (see awp_fused.hip for the sweep itself).
//
// Waves 0..10 are the tile's rows, 11..14 the two rows below and above it and
// 15 the two columns left and right, as in step_tile.  At level m every wave
// loads its own row of the old stresses, density and velocities and writes
// what neighbours need to LDS planes; the five waves without a stress row
// bring the rows and columns around (items).  After the level's one barrier
// each thread computes its new velocity from the planes and its z queues and
// writes it to a ring of three velocity planes; the tile's rows then compute
// the stress of level m - 2, whose in-plane velocity neighbours the ring holds
// and whose z neighbours are the thread's own.  Statements and their order
// are those of step_tile.
//
// step_tile loads each row of a stencil array by up to four waves at up to five
// offsets, 52 loads a point, 389M wave loads a launch at 1500x1000x300; neither
// deeper prefetch nor less traffic from memory (regions of tiles that fit the
// L2s) changed its time.  Here a row takes 20 loads and an item wave 5 more,
// 223M a launch.  (The vector cache waits for lines on their way 67 % of the
// cycles there, 71 % here.)  A CU holds one block of 16 waves in step with each
// other, so what counts next is that a level has one wait: all loads of the
// next level are issued after the barrier, and waited for together before the
// level's stores, which no wait then includes
// (waiting at the top of the next level, behind the stores: 20.2 ms per step;
// stores of the stresses alone behind the wait: 15.1).  FP32, ms per step
// before -> after, against two-stage staged: 517x389x149 1.29 -> 1.10 (1.13),
// 800x600x200 3.74 -> 3.19 (3.43), 1500x1000x300 16.8 -> 14.64 (16.29), which
// is 4.3 TB/s of the 140 B a point.
#pragma once
#include "awp_kernels.hpp"

namespace awp {

struct Sweep {
    using F4 = float __attribute__((ext_vector_type(4)));
    static constexpr int TY = 11, NW = TY + 5;
    static constexpr int RW = TX + 4, RP = RW * (TY + 4);   // ring planes: columns -2 .. 65, rows -2 .. TY+1
    static constexpr int SW = TX + 8, SP = SW * (TY + 8);   // stress planes: columns -4 .. 67, rows -4 .. TY+3
    static constexpr int MW = TX + 1, MP = MW * (TY + 1);   // media: columns 0 .. 64, rows -1 .. TY-1
    static constexpr int PAD = TX;                          // floats for the lanes without a point
    enum { XX, XY, YY, XZ, YZ, DD, NPL };
    static constexpr int SET = NPL * SP + PAD, MSET = 4 * MP + PAD;   // floats
    // media (three levels), stress planes (two), ring (three of u, v, w), and
    // of each row thread the old xx, yy, xy of two levels
    static constexpr int OWN = TX * TY, FLOATS = 3 * MSET + 2 * SET + 9 * RP + 6 * OWN;
    static_assert(MSET % 4 == 0 && FLOATS * 4 <= 160 * 1024, "LDS of a CU");
    static constexpr int ITEMS = 5;   // per wave
};

// the values of loads are here from this point on
__device__ __forceinline__ void arrived(float &a, float &b, float &c, float &d, float &e, float &f)
{
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f));
}

// MAIN: the waves of the tile's rows.  Both forms pass the same barriers, one
// a level.  a, b rebased by rb elements (step_tile).
template <bool MAIN>
__device__ __forceinline__ void sweep_rows(const Geo &g, const GState &a, const GState &b, const Coef &c, const int kc,
                                           const int bx, const int by, const int bz, const long long rb, const int wv,
                                           float *lds)
{
    using S = Sweep;
    using F4 = S::F4;
    constexpr int TY = S::TY, RW = S::RW, RP = S::RP, SW = S::SW, SP = S::SP, MW = S::MW;
    float *const med = lds, *const planes = lds + 3 * S::MSET, *const ring = planes + 2 * S::SET;
    float *const own = ring + 9 * RP + wv * TX + threadIdx.x;   // MAIN
    const int lane = threadIdx.x;
    const int i0 = bx * TX + 1, j0 = by * TY + 1;
    const int kb = bz * kc + 1;
    const int ke = min(kb + kc - 1, g.nz);
    const int m0 = kb - 2, mtop = min(ke + 2, g.nz);

    // the thread's point: column and row relative to the tile
    int col = lane, row = wv;   // (MAIN: the same row in the whole wave)
    bool active = true;
    if (!MAIN) {
        if (wv < TY + 4) {
            row = wv - TY < 2 ? wv - TY - 2 : wv - 2;
        } else {
            const int q = lane & 3;
            col = q < 2 ? q - 2 : TX - 2 + q;
            row = lane >> 2;
            active = lane < 4 * TY;
        }
    }
    const int i = i0 + col, j = j0 + row;
    const bool dom = active && i >= 1 && i <= g.nx && j >= 1 && j <= g.ny;
    const bool has = active && i <= g.nx + 2 && j <= g.ny + 2;   // two ghost layers around the grid
    const unsigned ob = (unsigned)((g.base + (long long)j * g.sy + i - rb) * 4);
    const unsigned sz4 = (unsigned)(g.sz * 4);
    const int spos = (row + 4) * SW + col + 4, rpos = (row + 2) * RW + col + 2, mpos = 4 * ((row + 1) * MW + col);
    const float c1 = c.c1, c2 = c.c2, dth = c.dth, dt = c.dt, dh1 = c.dh1;
    const float fxy = dom ? a.fx[i] * a.fy[j] : 0.0f;
    const bool iodd = (i & 1) != 0;
    const G<float> *d1 = (const G<float> *)a.d1;
    const G<float> *ME[4] = {(const G<float> *)a.lam, (const G<float> *)a.mu, (const G<float> *)a.qp,
                             (const G<float> *)a.qs};
    G<float> *const RR[6] = {(G<float> *)a.r1, (G<float> *)a.r2, (G<float> *)a.r3,
                             (G<float> *)a.r4, (G<float> *)a.r5, (G<float> *)a.r6};

    // items: rows and columns around the tile, one array for the whole wave;
    // a lane without a point reads (1, 1) and writes to the padding
    const G<float> *hb[S::ITEMS];
    unsigned ho[S::ITEMS];
    int hd[S::ITEMS], hk[S::ITEMS];   // hk: 1 a stress plane, 2 media, 0 nothing
    float hv[S::ITEMS];
    if constexpr (!MAIN) {
#pragma unroll
        for (int t = 0; t < S::ITEMS; ++t) {
            const int q = wv - TY + 5 * t;
            int x = lane, y = 0, dst = 0;
            bool on = true;
            hk[t] = q < 16 ? 1 : q < 24 ? 2 : 0;
            if (q < 16) {
                const int p = q < 10 ? (q < 3 ? S::XY : q < 6 ? S::YY : q < 9 ? S::YZ : S::DD)
                                     : q == 10 ? S::XX : q == 11 ? S::XY : q == 12 ? S::XZ : q == 13 ? S::YY
                                     : q == 14 ? S::YZ : S::DD;
                hb[t] = p == S::XX ? a.xx : p == S::XY ? a.xy : p == S::YY ? a.yy : p == S::XZ ? a.xz
                        : p == S::YZ ? a.yz : d1;
                if (q < 10) {
                    y = q == 0 || q == 6 ? -4 : q == 1 || q == 3 || q == 7 || q == 9 ? -3 : q == 5 ? TY + 3 : TY + 2;
                } else if (lane < 3 * TY) {
                    // the tile rows' columns beyond those of wave 15
                    const int e = lane % 3;
                    y = lane / 3;
                    x = q == 10 ? (e == 0 ? -4 : e == 1 ? -3 : 66) : (e == 0 ? -3 : 65 + e);
                    on = q <= 12;
                    if (q == 15) {   // density: column 66 of rows -1 .., column 64 of row -3
                        on = lane <= TY + 1;
                        x = lane <= TY ? 66 : 64;
                        y = lane <= TY ? lane - 1 : -3;
                    }
                } else {
                    // columns -2, -1, 64, 65 of rows -2, -1, TY, TY+1
                    const int e = lane - 3 * TY;
                    on = e < 16;
                    x = (e & 3) < 2 ? (e & 3) - 2 : TX - 2 + (e & 3);
                    y = (e >> 2) < 2 ? (e >> 2) - 2 : TY - 2 + (e >> 2);
                }
                dst = p * SP + (y + 4) * SW + x + 4;
            } else {
                // media: row -1, then column 64
                const int n = (q - 16) & 3;
                hb[t] = n == 0 ? ME[0] : n == 1 ? ME[1] : n == 2 ? ME[2] : ME[3];
                x = q < 20 ? lane : TX;
                y = q < 20 ? -1 : lane - 1;
                on = q < 24 && y < TY;
                dst = 4 * ((y + 1) * MW + x) + n;
            }
            on = on && i0 + x >= -1 && i0 + x <= g.nx + 2 && j0 + y >= -1 && j0 + y <= g.ny + 2;
            ho[t] = (unsigned)((g.base + (on ? (long long)(j0 + y) * g.sy + i0 + x : g.sy + 1) - rb) * 4);
            hd[t] = on ? dst : (q < 16 ? S::NPL * SP : 4 * S::MP) + lane;
            hv[t] = 0.0f;
            if (hk[t] == 1) hv[t] = gl(hb[t], ho[t] + (unsigned)m0 * sz4);
        }
    }

    // z queues at the thread's point (levels below -1 are zero), values of m0
    float xz_m2 = 0.f, xz_m1 = 0.f, xz_0 = 0.f, xz_p1 = 0.f, yz_m2 = 0.f, yz_m1 = 0.f, yz_0 = 0.f, yz_p1 = 0.f;
    float zz_m2 = 0.f, zz_m1 = 0.f, zz_0 = 0.f, zz_p1 = 0.f, zz_p2 = 0.f;
    float dA_m = 0.f, dB_m = 0.f, dC_m = 0.f;
    float xx = 0.f, xy = 0.f, yy = 0.f, dr = 0.f, u0 = 0.f, v0 = 0.f, w0 = 0.f;
    if (has) {
        const unsigned o = ob + (unsigned)m0 * sz4;
        if (m0 >= 1) {
            xz_m2 = gl(a.xz, o - 2 * sz4); yz_m2 = gl(a.yz, o - 2 * sz4); zz_m2 = gl(a.zz, o - 2 * sz4);
        }
        if (m0 >= 0) {
            xz_m1 = gl(a.xz, o - sz4); yz_m1 = gl(a.yz, o - sz4); zz_m1 = gl(a.zz, o - sz4);
        }
        xz_0 = gl(a.xz, o); yz_0 = gl(a.yz, o); zz_0 = gl(a.zz, o);
        xz_p1 = gl(a.xz, o + sz4); yz_p1 = gl(a.yz, o + sz4); zz_p1 = gl(a.zz, o + sz4);
        zz_p2 = gl(a.zz, o + 2 * sz4);
        xx = gl(a.xx, o); xy = gl(a.xy, o); yy = gl(a.yy, o); dr = gl(d1, o);
    }
    if (dom) {
        const unsigned o = ob + (unsigned)m0 * sz4;
        if (m0 >= 0) {
            const unsigned om = o - sz4;
            dA_m = gl(d1, om); dB_m = gl(d1, om - (unsigned)(g.sy * 4)); dC_m = gl(d1, om, 4);
        }
        u0 = gl(a.u1, o); v0 = gl(a.v1, o); w0 = gl(a.w1, o);
    }
    float fz = a.fz[max(m0, 0)], fz_1 = 0.f, fz_2 = 0.f;
    float w_4 = 0.f;                    // the new w four levels below
    F4 mn = {0.f, 0.f, 0.f, 0.f};
    float rr[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int r0 = (m0 + 3) % 3;              // ring slot of level m
    int ms = (kb + 2) % 3, mp = 0;      // media slots of levels s and s - 1 (from level kb - 1 on)

    // the planes and media (slot `mslot`) of level m, from what was loaded for it
    auto put = [&](const int m, const int mslot) {
        float *const pl = planes + (m & 1) * S::SET;
        const bool lvl = m <= g.nz;
        if (lvl && active) {
            pl[S::XX * SP + spos] = xx;
            pl[S::XY * SP + spos] = xy;
            pl[S::YY * SP + spos] = yy;
            pl[S::XZ * SP + spos] = xz_0;
            pl[S::YZ * SP + spos] = yz_0;
            pl[S::DD * SP + spos] = dr;
        }
        if constexpr (MAIN) {
            if (m > kb) *(F4 *)(med + mslot * S::MSET + mpos) = mn;
        } else {
#pragma unroll
            for (int t = 0; t < S::ITEMS; ++t) {
                if (hk[t] == 1) {
                    if (lvl) pl[hd[t]] = hv[t];
                } else if (hk[t] == 2 && m > kb) {
                    med[mslot * S::MSET + hd[t]] = hv[t];
                }
            }
        }
    };
    put(m0, ms);

    for (int m = m0; m <= ke + 2; ++m) {
        float *const pl = planes + (m & 1) * S::SET;
        const bool lvl = m <= g.nz;
        __syncthreads();
        // ---- loads for the next level ---------------------------------------
        const bool more = m < mtop;
        const unsigned o = ob + (unsigned)m * sz4, o1 = o + sz4;
        const float fzn = a.fz[min(m + 1, g.nz)];
        float xzn = 0.f, yzn = 0.f, zzn = 0.f, up = 0.f, vp = 0.f, wp = 0.f;
        if (more && has) {
            xx = gl(a.xx, o1);
            xy = gl(a.xy, o1);
            yy = gl(a.yy, o1);
            dr = gl(d1, o1);
            xzn = gl(a.xz, o1 + sz4);
            yzn = gl(a.yz, o1 + sz4);
            zzn = gl(a.zz, o1 + 2 * sz4);
        }
        if (more && dom) {
            up = gl(a.u1, o1);
            vp = gl(a.v1, o1);
            wp = gl(a.w1, o1);
        }
        float rn[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if constexpr (MAIN) {
            if (m >= kb && m <= ke + 1 && has) {
                const unsigned ob1 = o - sz4;
                mn = F4{gl(ME[0], ob1), gl(ME[1], ob1), gl(ME[2], ob1), gl(ME[3], ob1)};
                if (m > kb && dom) {
#pragma unroll
                    for (int n = 0; n < 6; ++n) rn[n] = gln(RR[n], ob1);
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < S::ITEMS; ++t) {
                if (hk[t] == 1) {
                    if (more) hv[t] = gl(hb[t], ho[t] + (unsigned)(m + 1) * sz4);
                } else if (hk[t] == 2 && m >= kb && m <= ke + 1) {
                    hv[t] = gl(hb[t], ho[t] + (unsigned)(m - 1) * sz4);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- velocity of level m (operator.f:92-244) -------------------------
        float un = 0.f, vn = 0.f, wn = 0.f;
        if (dom && lvl) {
            const float *px = pl + S::XX * SP + spos, *pxy = pl + S::XY * SP + spos, *pyy = pl + S::YY * SP + spos;
            const float *pxz = pl + S::XZ * SP + spos, *pyz = pl + S::YZ * SP + spos, *pd = pl + S::DD * SP + spos;
            const float dA = pd[0], dB = pd[-SW], dC = pd[1], dD = pd[1 - SW];
            if (m >= 1) {
                float d, q, u, v, w;
                d = 0.25f * ((dA + dB) + (dA_m + dB_m));
                q = dth / d;
                u = u0 + q * (
                    c1 * (px[0] - px[-1]) + c2 * (px[1] - px[-2]) +
                    c1 * (pxy[0] - pxy[-SW]) + c2 * (pxy[SW] - pxy[-2 * SW]) +
                    c1 * (xz_0 - xz_m1) + c2 * (xz_p1 - xz_m2));
                d = 0.25f * ((dA + dC) + (dA_m + dC_m));
                q = dth / d;
                v = v0 + q * (
                    c1 * (pxy[1] - pxy[0]) + c2 * (pxy[2] - pxy[-1]) +
                    c1 * (pyy[SW] - pyy[0]) + c2 * (pyy[2 * SW] - pyy[-SW]) +
                    c1 * (yz_0 - yz_m1) + c2 * (yz_p1 - yz_m2));
                d = 0.25f * ((dA + dC) + (dB + dD));
                q = dth / d;
                w = w0 + q * (
                    c1 * (pxz[1] - xz_0) + c2 * (pxz[2] - pxz[-1]) +
                    c1 * (yz_0 - pyz[-SW]) + c2 * (pyz[SW] - pyz[-2 * SW]) +
                    c1 * (zz_p1 - zz_0) + c2 * (zz_p2 - zz_m1));
                const float D = fxy * fz;       // addcrjvel, cerjan.f:292-328
                un = u * D;
                vn = v * D;
                wn = w * D;
            }
            dA_m = dA; dB_m = dB; dC_m = dC;
        }
        // the z queues move up
        const float old_xz = xz_m2, old_yz = yz_m2, old_zz = zz_m2;
        xz_m2 = xz_m1; xz_m1 = xz_0; xz_0 = xz_p1;
        yz_m2 = yz_m1; yz_m1 = yz_0; yz_0 = yz_p1;
        zz_m2 = zz_m1; zz_m1 = zz_0; zz_0 = zz_p1; zz_p1 = zz_p2;
        float *const slot = ring + r0 * 3 * RP + rpos;
        // own column: the velocities of level m - 3 leave the ring
        float u_3 = 0.f, v_3 = 0.f, w_3 = 0.f;
        if (MAIN && m > kb) {
            u_3 = slot[0];
            v_3 = slot[RP];
            w_3 = slot[2 * RP];
        }
        if (lvl && active) {
            slot[0] = un;
            slot[RP] = vn;
            slot[2 * RP] = wn;
        }
        if constexpr (MAIN) {
            if (m == g.nz + 1 && dom) {
                // free-surface velocity images fvelxy / fvelz (operator.f:246-306)
                // from the level-nz plane (and w at nz-1)
                const float *pu = ring + (r0 == 0 ? 2 : r0 - 1) * 3 * RP + rpos, *pv = pu + RP, *pw = pv + RP;
                const float w0s = pw[0], u0s = pu[0], v0s = pv[0];
                const float ut = u0s - (w0s - pw[-1]);
                const float vt = v0s - (pw[RW] - w0s);
                const float ut_ip1 = (i < g.nx) ? (pu[1] - (pw[1] - w0s)) : 0.0f;
                const float vt_jm1 = (j > 1) ? (pv[-RW] - (w0s - pw[-RW])) : 0.0f;
                const float xl = 1.0f / gl(ME[0], o - sz4), xm = 2.0f / gl(ME[1], o - sz4);
                const float xl2m = xm + xl;
                const float wt = ring[(r0 == 2 ? 0 : r0 + 1) * 3 * RP + rpos + 2 * RP] - (xl / xl2m) * (
                    (ut_ip1 - ut) +
                    (pu[1] - u0s) +
                    (vt - vt_jm1) +
                    (v0s - pv[-RW]));
                un = ut;
                vn = vt;
                wn = wt;
                slot[0] = un;   // (its own position alone)
                slot[RP] = vn;
                slot[2 * RP] = wn;
                gsn(b.u1, o, un);
                gsn(b.v1, o, vn);
                gsn(b.w1, o, wn);
            }
        }
        const int s = m - 2;
        const int msn = m > kb ? (ms == 2 ? 0 : ms + 1) : ms;
        const unsigned os = o - 2 * sz4;
        float r1 = 0.f, r2 = 0.f, r3 = 0.f, r4 = 0.f, r5 = 0.f, r6 = 0.f;
        float sxx = 0.f, syy = 0.f, szz = 0.f, sxy = 0.f, sxz = 0.f, syz = 0.f;
        if constexpr (MAIN) {
            // ---- stress of level s (viscoop.f:49-191) ------------------------
            if (s >= kb && dom) {
                const F4 *ma = (const F4 *)(med + ms * S::MSET + mpos), *mb = (const F4 *)(med + mp * S::MSET + mpos);
                const F4 A = ma[0], B = ma[1], C = ma[-MW], D = ma[1 - MW];
                const F4 Am = mb[0], Bm = mb[1], Cm = mb[-MW], Dm = mb[1 - MW];
                float vxl = 8.0f / (A.x + B.x + C.x + D.x + Am.x + Bm.x + Cm.x + Dm.x);
                const float vxm = 8.0f / (A.y + B.y + C.y + D.y + Am.y + Bm.y + Cm.y + Dm.y);
                vxl = vxl + 2.0f * vxm;
                const float vqpa = 0.125f * (A.z + B.z + C.z + D.z + Am.z + Bm.z + Cm.z + Dm.z);
                const float vqsa = 0.125f * (A.w + B.w + C.w + D.w + Am.w + Bm.w + Cm.w + Dm.w);
                const float vx4 = 2.0f / (A.y + Am.y), vx5 = 2.0f / (A.y + C.y), vx6 = 2.0f / (A.y + B.y);
                const float va4 = 0.5f * (A.w + Am.w), va5 = 0.5f * (A.w + C.w), va6 = 0.5f * (A.w + B.w);
                const float vh2_r4 = -va4 * vx4 / 2.0f, vh2_r5 = -va5 * vx5 / 2.0f, vh2_r6 = -va6 * vx6 / 2.0f;
                __builtin_amdgcn_sched_barrier(0);

                const float *pu = ring + (r0 == 2 ? 0 : r0 + 1) * 3 * RP + rpos, *pv = pu + RP, *pw = pv + RP;
                const float *qu = ring + (r0 == 0 ? 2 : r0 - 1) * 3 * RP + rpos;   // level s + 1
                const float uc = pu[0], vc = pv[0], wc = pw[0], u_1 = qu[0], v_1 = qu[RP], w_1 = qu[2 * RP];
                const float vt1 = c1 * (pu[1] - uc) + c2 * (pu[2] - pu[-1]);
                const float vt2 = c1 * (vc - pv[-RW]) + c2 * (pv[RW] - pv[-2 * RW]);
                const float vt3 = c1 * (wc - w_3) + c2 * (w_1 - w_4);
                const float vt4 = c1 * (pu[RW] - uc) + c2 * (pu[2 * RW] - pu[-RW]) +
                                  c1 * (vc - pv[-1]) + c2 * (pv[1] - pv[-2]);
                const float vt5 = c1 * (u_1 - uc) + c2 * (un - u_3) +
                                  c1 * (wc - pw[-1]) + c2 * (pw[1] - pw[-2]);
                const float vt6 = c1 * (v_1 - vc) + c2 * (vn - v_3);
                const float vt7 = c1 * (pw[RW] - wc) + c2 * (pw[2 * RW] - pw[-RW]);

                const int it = (j & 1) * 2 + ((g.nz + 1 - s) & 1);   // the wave's
                const float vx1 = iodd ? c.tau1[4 + it] : c.tau1[it];
                const float vx2 = iodd ? c.tau2[4 + it] : c.tau2[it];
                const float vh1 = -vxm * vqsa;
                const float vtmp = vxl * (vt1 + vt2 + vt3);
                const float va1 = -vqpa * vxl * dh1 * (vt1 + vt2 + vt3) / 2.0f;

                r1 = rr[0]; r2 = rr[1]; r3 = rr[2]; r4 = rr[3]; r5 = rr[4]; r6 = rr[5];
                const float *po = own + (m & 1) * 3 * S::OWN;
                sxx = po[0]; syy = po[S::OWN]; szz = old_zz; sxy = po[2 * S::OWN]; sxz = old_xz; syz = old_yz;

                sxx = sxx + dth * (vtmp - 2.0f * vxm * (vt2 + vt3)) + dt * r1;
                syy = syy + dth * (vtmp - 2.0f * vxm * (vt1 + vt3)) + dt * r2;
                szz = szz + dth * (vtmp - 2.0f * vxm * (vt1 + vt2)) + dt * r3;
                sxy = sxy + vx4 * dth * vt4 + dt * r4;
                sxz = sxz + vx5 * dth * vt5 + dt * r5;
                syz = syz + vx6 * (dth * vt6 + dth * vt7) + dt * r6;

                r1 = (vx2 * r1 - vh1 * (vt2 + vt3) * dh1 + va1) * vx1;
                r2 = (vx2 * r2 - vh1 * (vt1 + vt3) * dh1 + va1) * vx1;
                r3 = (vx2 * r3 - vh1 * (vt1 + vt2) * dh1 + va1) * vx1;
                r4 = (vx2 * r4 + vh2_r4 * dh1 * vt4) * vx1;
                r5 = (vx2 * r5 + vh2_r5 * dh1 * vt5) * vx1;
                r6 = (vx2 * r6 + vh2_r6 * dh1 * (vt6 + vt7)) * vx1;

                sxx = sxx + dt * r1;
                syy = syy + dt * r2;
                szz = szz + dt * r3;
                sxy = sxy + dt * r4;
                sxz = sxz + dt * r5;
                syz = syz + dt * r6;

                const float Ds = fxy * fz_2;       // addcrjstr, cerjan.f:249-290
                sxx = sxx * Ds; syy = syy * Ds; szz = szz * Ds;
                sxz = sxz * Ds; syz = syz * Ds; sxy = sxy * Ds;
            }
            w_4 = w_3;
            float *po = own + (m & 1) * 3 * S::OWN;
            po[0] = pl[S::XX * SP + spos];
            po[S::OWN] = pl[S::YY * SP + spos];
            po[2 * S::OWN] = pl[S::XY * SP + spos];
            fz_2 = fz_1; fz_1 = fz;
        }
        // The level's one wait for loads: everything the next level takes
        // arrives here, ahead of this level's stores, so that no wait is one
        // for stores on their way.
        __builtin_amdgcn_sched_barrier(0);
        xz_p1 = xzn; yz_p1 = yzn; zz_p2 = zzn;
        u0 = up; v0 = vp; w0 = wp;
        if (m < ke + 2) put(m + 1, msn);
        if constexpr (MAIN) {
#pragma unroll
            for (int n = 0; n < 6; ++n) rr[n] = rn[n];
        }
        arrived(xz_p1, yz_p1, zz_p2, u0, v0, w0);
        if (MAIN) arrived(rr[0], rr[1], rr[2], rr[3], rr[4], rr[5]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MAIN) {
            if (m >= kb && m <= ke && dom) {
                gsn(b.u1, o, un);
                gsn(b.v1, o, vn);
                gsn(b.w1, o, wn);
            }
            if (s >= kb && dom) {
                gsn(RR[0], os, r1); gsn(RR[1], os, r2); gsn(RR[2], os, r3);
                gsn(RR[3], os, r4); gsn(RR[4], os, r5); gsn(RR[5], os, r6);
                gsn(b.xx, os, sxx); gsn(b.yy, os, syy); gsn(b.xy, os, sxy);
                if (s == g.nz) {
                    // fstr (operator.f:575-612): images above the surface, xz = yz = 0 on it
                    const unsigned q1 = os + sz4, q2 = q1 + sz4;
                    gsn(b.zz, os, szz);
                    gsn(b.zz, q1, -szz);
                    gsn(b.zz, q2, -gl(b.zz, os - sz4));
                    gsn(b.xz, os, 0.0f);
                    gsn(b.yz, os, 0.0f);
                    gsn(b.xz, q1, -gl(b.xz, os - sz4));
                    gsn(b.xz, q2, -gl(b.xz, os - 2 * sz4));
                    gsn(b.yz, q1, -gl(b.yz, os - sz4));
                    gsn(b.yz, q2, -gl(b.yz, os - 2 * sz4));
                } else {
                    gsn(b.zz, os, szz); gsn(b.xz, os, sxz); gsn(b.yz, os, syz);
                }
            }
        }
        if (m > kb) {
            mp = ms;
            ms = msn;
        }
        r0 = r0 == 2 ? 0 : r0 + 1;
        fz = fzn;
    }
}

// one column tile (bx, by, z chunk bz) of one run: the whole block calls it
__device__ __forceinline__ void sweep_tile(const Geo &g, const GState &a, const GState &b, const Coef &c, const int kc,
                                           const int bx, const int by, const int bz, const long long rb, float *lds)
{
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
    if (wv < Sweep::TY)
        sweep_rows<true>(g, a, b, c, kc, bx, by, bz, rb, wv, lds);
    else
        sweep_rows<false>(g, a, b, c, kc, bx, by, bz, rb, wv, lds);
}

}  // namespace awp
