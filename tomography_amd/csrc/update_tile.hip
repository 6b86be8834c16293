// update_tile.hip — the register-tile update kernel: one launch advances every
// tile of every simulation by one time block (replaces H_field_update +
// E_field_update + calculate_JandM's sampling, FDTD_GPU.cu:231-434).
//
// A workgroup of NW waves holds 64 columns times NW * R rows, R rows per wave,
// one column per lane, in registers; it requests them all at once, advances
// them up to 15 steps and stores the cells it owns.  A step invalidates one
// lane and one row at each edge of the tile that is not the grid's edge, so
// tiles overlap by twice the block's steps.  Waves couple through LDS: each
// publishes its bottom and top Ez rows, advances what needs no neighbour (H of
// all rows but the top one, E of the rows between), meets the others at the
// step's only barrier and finishes its two edge rows.  The Hx of the row below
// a wave is advanced by both waves, so H needs no exchange.
//
// Against the row sweeps (kernels.hip) no row waits for a memory round trip or
// for the stage before it, no register moves from stage to stage, and a wave
// takes the stage its cells need: the bare vacuum one (9 VALU instructions a
// row; 92% of a 256 mm domain is vacuum), with material coefficients in
// registers, or with the CPML recursions of its columns and rows.  All of them
// round as the row sweeps do, so every form gives the same bits.
//
// What bounds it: per launch dispatch (5 us) and the tiles' loads and stores
// (one step of 64 simulations of 512^2 costs 143 us, each further one 7: 3.5 TB/s
// of field traffic that little compute overlaps), per step one tile's own
// instruction issue and the LDS exchange.  So the tallest tiles whose state fits
// the 128 VGPRs of four waves per SIMD without spilling: 16 rows of vacuum, 8
// with one axis' CPML psi or with material coefficients, 4 with both (a corner
// row in material costs 3 times a vacuum one).  Spilled prologues cost more than
// shorter tiles (16 rows at the strips: 169 -> 270 us).  Reference-compatible
// mode, with its incident field and 64-bit kappa, spills 11 VGPRs all the same.
#include "device.h"
#include "fold.h"
#include "kernels.h"

namespace tomo {
namespace {

constexpr int kLane = 64;

// Lane shifts on the VALU (DPP wave_shl:1 / wave_shr:1), folded by the compiler
// into the subtraction that uses them: next(v)[i] = v[i+1], prev(v)[i] = v[i-1],
// 0 past the edge lane (a ghost lane, or a lane whose result is masked).
__device__ __forceinline__ float next_lane(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xF, 0xF, true));
}
__device__ __forceinline__ float prev_lane(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xF, 0xF, true));
}

__device__ __forceinline__ float read_lane(float v, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}

// a / k for a divisor whose reciprocal r = 1 / (double)k is known: the product in
// 64 bits is within 2^-52 of the quotient, which (a ratio of two 24-bit
// numbers) lies at least 2^-49 from any point where rounding to 32 bits turns,
// so this is the division's own result (but for ties among denormal results) in
// three instructions instead of eleven.
__device__ __forceinline__ float div_known(float a, double r) { return (float)((double)a * r); }

// Buffer views of one array: the address of an access is base + a per-lane byte
// offset + a wave-uniform one, so a tile's rows share one lane offset and step
// in scalar registers, and the hardware drops the lanes whose offset lies past
// the array (kOff): loads return 0 and stores do nothing, with no branch or
// execution mask.  Arrays are smaller than 2 GiB.
typedef __amdgpu_buffer_rsrc_t Buffer;
constexpr unsigned kOff = 0x80000000u;
__device__ __forceinline__ Buffer buffer_of(const void* base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ float ld(Buffer b, unsigned lane_off, int off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, lane_off, off, 0));
}
__device__ __forceinline__ void st(Buffer b, unsigned lane_off, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), b, lane_off, off, 0);
}

// Barrier over the LDS traffic alone: the sample and field stores in flight are
// not waited for.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// CPML coefficients of a row or a lane: the recursion's a and b and k = 1/kappa
// (in 64 bits for reference-compatible mode, which divides by kappa).  Off the
// strips a = b = 0 and k = 1, so that strip cells and others take the same
// instructions; the reference's stage tells them apart by k = 0.
template <bool REF>
struct Profile {
    float a, b, k;
};
template <>
struct Profile<true> {
    float a, b;
    double k;
};

template <bool REF, int NW>
struct TileLds {
    float4 coef[TOMO_MAX_MAT * 2];        // filled when a wave of the tile holds material
    Profile<REF> row_e[NW * kTileRowsTall], row_h[NW * kTileRowsTall + 1];  // of E row yl + i and of H row yl - 1 + i
    float ez[2][NW][2][kLane];            // per step parity: each wave's bottom and top Ez row
};

// CPML profile entry of E node v (1..n-1) and of H node v (0..n-1) of a line of
// n cells, -1 off the strips.
__device__ __forceinline__ int strip_e(int v, int n, int nc) {
    return (v >= 1 && v <= nc) ? nc - v : ((v >= n - nc && v <= n - 1) ? v - n + nc : -1);
}
__device__ __forceinline__ int strip_h(int v, int n, int nc) {
    return (v >= 0 && v < nc) ? nc - 1 - v : ((v >= n - nc && v < n) ? v - n + nc : -1);
}
template <bool REF>
__device__ __forceinline__ Profile<REF> profile(const float* k, const float* ik, const float* a, const float* b, int i) {
    Profile<REF> p{0.f, 0.f, REF ? 0.f : 1.f};
    if (i >= 0) {
        p.a = a[i];
        p.b = b[i];
        if constexpr (REF) p.k = 1.0 / (double)k[i];
        else p.k = ik[i];
    }
    return p;
}
template <bool REF>
__device__ __forceinline__ Profile<REF> profile_e(const DevSim* __restrict__ S, int i) {
    return profile<REF>(S->ke, S->ike, S->ae, S->be, i);
}
template <bool REF>
__device__ __forceinline__ Profile<REF> profile_h(const DevSim* __restrict__ S, int i) {
    return profile<REF>(S->km, S->ikm, S->am, S->bm, i);
}

// Wave-uniform value that the compiler may not fold into values computed
// outside a loop: row conditions then cost a scalar compare where they are
// used and hold no scalar register across the step loop.
__device__ __forceinline__ int opaque(int v) {
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
    return v;
}

// One wave's share of a tile: R rows [yb, yb + R) of 64 columns [xl, xl + 64),
// advanced nst steps.  XS / YS: the lanes / rows reach a CPML strip or the PEC
// edge; MAT: some cell is not vacuum; SRC: the source cell is one of the wave's
// and may lie in material.
template <int MODE, int R, int NW, bool XS, bool YS, bool MAT, bool SRC>
__device__ __forceinline__ void tile_wave(const RegTile& tile, const DevSim* __restrict__ Sp, TileLds<MODE == TOMO_MODE_REF_COMPAT, NW>& lds,
                                          int par, int step0, int k0, int nst, int wv, int lane, bool tables, bool frows) {
    constexpr bool REF = MODE == TOMO_MODE_REF_COMPAT;
    const int nx = Sp->nx, ny = Sp->ny, nc = Sp->nc, pitch = Sp->pitch, ps = Sp->ps;
    const int x = tile.xl + lane, yb = tile.yl + wv * R;
    const int w2 = 2 * nc;
    // x-strip columns of the lane in the psi arrays
    const int je = (x >= 1 && x <= nc) ? x - 1 : ((x >= nx - nc && x <= nx - 1) ? nc + x - (nx - nc) : -1);
    const int jh = x < nc ? x : ((x >= nx - nc && x < nx) ? nc + x - (nx - nc) : -1);
    // psi rows of the y strips: E node rows 1..nc and ny-nc..ny-1, H rows 0..nc-1
    // and ny-nc..ny-1 (no wave reaches both: they are 4 rows apart, ny >= 2 nc + 4,
    // and tiles of 8-row waves hold 64 rows from an end of the grid or clear of
    // the strips, so that with nc <= 31 the gap falls between two waves)
    const bool hi = yb + R > ny - nc;
    auto row_e = [&](int y) { return (unsigned)(hi ? y - (ny - nc) : y - 1) < (unsigned)nc; };
    auto row_h = [&](int y) { return (unsigned)(hi ? y - (ny - nc) : y) < (unsigned)nc; };
    const int re0 = hi ? 2 * nc - ny : -1, rh0 = hi ? 2 * nc - ny : 0;
    const Buffer F = buffer_of(Sp->fbase, (size_t)ps * 24), Q = buffer_of(Sp->xbase, (size_t)Sp->xs * 16),
                 Y = buffer_of(Sp->ybase, (size_t)Sp->ys * 16), Jb = buffer_of(Sp->jbase, (size_t)Sp->js * 8);
    const unsigned vx = (unsigned)x * 4u;
    const unsigned ve = XS && je >= 0 ? (unsigned)je * 4u : kOff, vh = XS && jh >= 0 ? (unsigned)jh * 4u : kOff;
    const int row4 = pitch * 4, plane = ps * 4;  // bytes
    kcint* span = (kcint*)Sp->span;
    // lane offset of row y's Jp (compact: one run per row over the dispersive span)
    auto jp_off = [&](int y) {
        const int lo = span[3 * y], hi = span[3 * y + 1], off = span[3 * y + 2];
        return x >= lo && x < hi ? (unsigned)(off - lo + x) * 4u : kOff;
    };

    // ---- the whole tile is requested at once: no row waits for another
    float ez[R], hx[R], hy[R], jp[MAT ? R : 1], phx[XS ? R : 1], pex[XS ? R : 1], phy[YS ? R : 1], pey[YS ? R : 1];
    int mat[MAT ? R : 1];
    float hxb, phyb = 0.f;  // Hx (and its psi) of the row below the wave, which it advances beside its own
    if constexpr (MAT) {
        const Buffer M = buffer_of(Sp->mat, (size_t)(ny + 1) * pitch);
#pragma unroll
        for (int i = 0; i < R; ++i) mat[i] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(M, (unsigned)x, (yb + i) * pitch, 0);
    }
    {
        const int o = par * plane + yb * row4;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            ez[i] = ld(F, vx, o + i * row4);
            hx[i] = ld(F, vx, o + i * row4 + 2 * plane);
            hy[i] = ld(F, vx, o + i * row4 + 4 * plane);
        }
        hxb = ld(F, yb > 0 ? vx : kOff, o - (yb > 0 ? row4 : 0) + 2 * plane);
    }
    if constexpr (MAT) {
#pragma unroll
        for (int i = 0; i < R; ++i) jp[i] = ld(Jb, jp_off(yb + i), par * Sp->js * 4);
    }
    if constexpr (XS) {
        const int o = (par * Sp->xs + yb * w2) * 4;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            pex[i] = ld(Q, ve, o + i * w2 * 4);
            phx[i] = ld(Q, vh, o + i * w2 * 4 + Sp->xs * 8);
        }
    }
    if constexpr (YS) {
        const int oe = (par * Sp->ys + re0 * pitch) * 4, oh = ((par + 2) * Sp->ys + rh0 * pitch) * 4;
        // (rows off the strips: the lane offset drops them, the row offset is the array's start)
        auto psi = [&](bool in, int o, int y) { return ld(Y, in ? vx : kOff, in ? o + y * row4 : 0); };
#pragma unroll
        for (int i = 0; i < R; ++i) {
            pey[i] = psi(row_e(yb + i), oe, yb + i);
            phy[i] = psi(row_h(yb + i), oh, yb + i);
        }
        phyb = psi(row_h(yb - 1), oh, yb - 1);
    }
    // the tile's tables, while those loads are on their way
    if (tables) {
        if (tile.matmask) {
            float* lcf = (float*)lds.coef;
            for (int i = threadIdx.x; i < Sp->nmat * TOMO_NCOEF; i += NW * kLane) lcf[i] = Sp->coef[i];
        }
        if (frows) {
            for (int i = threadIdx.x; i <= NW * R; i += NW * kLane) {
                if (i < NW * R) lds.row_e[i] = profile_e<REF>(Sp, strip_e(tile.yl + i, ny, nc));
                lds.row_h[i] = profile_h<REF>(Sp, strip_h(tile.yl - 1 + i, ny, nc));
            }
        }
        lds_barrier();
    }
    const float chx = Sp->chx, chy = Sp->chy, dxf = Sp->dxf, dyf = Sp->dyf, chx_d = Sp->chx_d, chy_d = Sp->chy_d;
    const float cb0 = Sp->coef[1];  // vacuum curl coefficient (the vacuum Ez coefficient is exactly 1)
    const bool clamp = REF && !(Sp->flags & TOMO_FLAG_NO_NAN_CLAMP);
    // the CPU form has no Jp: an infinite Ez must not make one (a mask keeps the
    // stage one basic block; a branch cost the drop-in objective 1%)
    const unsigned debye = Sp->flags & TOMO_FLAG_CPU_COEFS ? 0u : ~0u;
    const bool ex_ok = !XS || (x >= 1 && x < nx);
    const bool bot = YS && yb == 0, top = YS && yb + R - 1 == ny;  // PEC rows: the wave's first, its last
    Profile<REF> Le, Lh;
    if constexpr (XS) {
        Le = profile_e<REF>(Sp, strip_e(x, nx, nc));
        Lh = profile_h<REF>(Sp, strip_h(x, nx, nc));
    }
    float4 qa[MAT ? R : 1], qb[MAT ? R : 1];
    float f0[MAT && REF ? R : 1];  // the incident field half a step back: each step's new one is the next step's old
    auto delay = [&](int i) {
        const float X = Sp->inc_abs_origin ? (float)x : (float)(x - nx / 2);
        const float Y = Sp->inc_abs_origin ? (float)(yb + i) : (float)(yb + i - ny / 2);
        return Sp->inc_c - Sp->inc_ay * Y - Sp->inc_ax * X;
    };
    if constexpr (MAT) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            qa[i] = lds.coef[2 * mat[i]];
            qb[i] = lds.coef[2 * mat[i] + 1];
            if constexpr (REF) {
                const float a0 = (((float)step0 - 0.5f) * Sp->inc_dt + delay(i)) * Sp->inc_itau;
                f0[i] = expf(-a0 * a0);
            }
        }
    }

    // ---- contour samples: face rows / columns hold H and Ez, their outer neighbours Ez
    const int D = Sp->D, P = Sp->P, K = Sp->srows, cx_hi = Sp->cx_hi, cy_lo = Sp->cy_lo;
    const bool own = x >= tile.x0 && x < tile.xe;
    const Buffer Z = buffer_of(Sp->samp, (size_t)3 * K * P * 4);
    // rows of the wave that the tile owns: [ra, rb)
    const int ra = max(tile.y0 - yb, 0), rb = min(tile.y1 - yb, R);
    // bits of the owned rows that are face rows and their outer neighbours (lo:
    // the bottom leg's), and of the rows in the x legs' range
    const unsigned mine = rb > ra ? ((1u << rb) - 1u) & ~((1u << ra) - 1u) : 0u;
    auto bit = [&](int y) { return (unsigned)(y - yb) < (unsigned)R ? 1u << (y - yb) : 0u; };
    const int m_face = mine & (bit(D) | bit(ny - D - 1)), m_out = mine & (bit(D + 1) | bit(ny - D));
    int m_x = 0;
    auto has_col = [&](int c) { return c >= tile.x0 && c < tile.xe; };
    if (has_col(D) || has_col(D + 1) || has_col(nx - D - 1) || has_col(nx - D)) {
        const int a = min(max(cy_lo - yb, 0), R), z = min(max(ny - D - yb, 0), R);
        m_x = z > a ? mine & ((1u << z) - 1u) & ~((1u << a) - 1u) : 0;
    }
    // lane offsets of the samples: plane 0 (H) or, for the outer neighbours, plane 2 (their Ez)
    const bool y_lane = own && x >= D + 1 && x <= cx_hi;
    const bool x_face = x == D || x == nx - D - 1;
    const bool x_lane = own && (x_face || x == D + 1 || x == nx - D), x_hi = x >= nx - D - 1;
    const int kp4 = K * P * 4, x_dir = x_hi ? 4 : -4;
    const unsigned zx0 = x_lane ? (unsigned)((x_hi ? Sp->L1 - cy_lo + yb : Sp->L3 + ny - D - 1 - yb) * 4 + (x_face ? 0 : 2 * kp4)) : kOff;
    const unsigned zx1 = x_lane && x_face ? zx0 + (unsigned)kp4 : kOff;
    const int L2 = Sp->L2;
    auto sample = [&](int k) {
        const int o = (k >= K ? k - K : k) * P * 4, f = opaque(m_face), g = opaque(m_out), xr = opaque(m_x);
        if (f | g) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (!((f | g) >> i & 1)) continue;  // wave-uniform
                const unsigned z = !y_lane ? kOff : (unsigned)(2 * (yb + i) < ny ? x - D - 1 : L2 + cx_hi - x) * 4u;
                if (f >> i & 1) {
                    st(Z, z, o, hx[i]);
                    st(Z, z, o + kp4, ez[i]);
                } else {
                    st(Z, z, o + 2 * kp4, ez[i]);
                }
            }
        }
        if (xr) {
            unsigned z0 = zx0, z1 = zx1;
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (xr >> i & 1) {  // wave-uniform
                    st(Z, z0, o, x_face ? hy[i] : ez[i]);
                    st(Z, z1, o, ez[i]);
                }
                z0 += x_dir;
                z1 += x_dir;
            }
        }
    };

    // ---- source
    const int isrc = Sp->sy - yb;  // row of the source, if it is one of the wave's
    const bool wsrc = !REF && isrc >= 0 && isrc < R && Sp->sx >= tile.xl && Sp->sx < tile.xl + kLane;
    const bool lsrc = x == Sp->sx;
    const bool extra = wsrc || (m_face | m_out | m_x) != 0;  // a step has more to do than the update
    float sw = 0.f;  // lane t: the waveform of the block's step t
    if (wsrc && lane < nst) sw = ((gcfloat*)Sp->srcw)[step0 + lane];

    // H half-step of one row, in place; the psi of the strips advance with it.
    // Columns x = nx and the row y = ny have no H nodes: their Ez and the Ez
    // beyond them are 0 (next_lane past lane 63, ez_up above the top row), so
    // their H and psi, loaded as 0, stay 0 without a mask.
    auto h_step = [&](float ez_c, float ez_up, float& hx_, float* hy_, float* phx_, float* phy_, const Profile<REF> W) {
        const float dEy = ez_up - ez_c;
        float hxn, tx = dEy;
        if constexpr (REF) {
            hxn = hx_ - chx * dEy;
            if constexpr (YS) {
                const float u = chx * dEy;
                const float q = hx_ - div_known(u, W.k);
                *phy_ = W.b * *phy_ + W.a * dEy;
                hxn = W.k != 0.0 ? q - chx_d * *phy_ : hxn;
            }
        } else {
            if constexpr (YS) {
                *phy_ = W.b * *phy_ + W.a * dEy;
                tx = dEy * W.k + dyf * *phy_;
            }
            hxn = hx_ - chx * tx;
        }
        hx_ = hxn;
        if (!hy_) return;
        const float dEx = next_lane(ez_c) - ez_c;
        float hyn, ty = dEx;
        if constexpr (REF) {
            hyn = *hy_ + chy * dEx;
            if constexpr (XS) {
                const float u = chy * dEx;
                const float q = *hy_ + div_known(u, Lh.k);
                *phx_ = Lh.b * *phx_ + Lh.a * dEx;
                hyn = jh >= 0 ? q + chy_d * *phx_ : hyn;
            }
        } else {
            if constexpr (XS) {
                *phx_ = Lh.b * *phx_ + Lh.a * dEx;
                ty = dEx * Lh.k + dxf * *phx_;
            }
            hyn = *hy_ + chy * ty;
        }
        *hy_ = hyn;
    };
    // E half-step of row i given its new H and the new Hx of the row below;
    // `edge`: a PEC row.
    auto e_step = [&](int i, float hx_dn, int n, float s, const Profile<REF> W, bool edge) {
        const float dHy = hy[i] - prev_lane(hy[i]);
        const float dHx = hx[i] - hx_dn;
        const bool eok = ex_ok && !(YS && edge);
        const float e0 = ez[i];
        float4 A = make_float4(1.f, cb0, 0.f, 0.f), B = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (MAT) {
            A = qa[i];
            B = qb[i];
        }
        float en;
        if constexpr (REF) {
            if constexpr (MAT) {
                const float a1 = (((float)n + 0.5f) * Sp->inc_dt + delay(i)) * Sp->inc_itau;
                const float f1 = expf(-a1 * a1), fo = f0[i];
                f0[i] = f1;
                en = A.x * e0 + A.y * dHy - A.y * dHx + A.z * f1 + A.w * fo - B.x * jp[i];
                const float jn = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, B.y * jp[i] + B.z * (en - e0 + f1 - fo)) & debye);
                jp[i] = (XS || YS) ? (eok ? jn : 0.f) : jn;
            } else {
                const float u = A.y * dHy;
                const float v = e0 + u;
                en = v - A.y * dHx;
            }
            if constexpr (XS || YS) {
                const float uy = A.y * dHy, ux = A.y * dHx;
                if constexpr (XS) {
                    pex[i] = edge ? pex[i] : Le.b * pex[i] + Le.a * dHy;
                    float b = A.x * e0 + div_known(uy, Le.k);
                    b = b - div_known(ux, Le.k);
                    b = b + A.y * dxf * pex[i];
                    en = je >= 0 ? b : en;
                }
                if constexpr (YS) {
                    pey[i] = ex_ok ? W.b * pey[i] + W.a * dHx : pey[i];
                    float b = A.x * e0 + div_known(uy, W.k);
                    b = b - div_known(ux, W.k);
                    b = b - A.y * dyf * pey[i];
                    en = W.k != 0.0 ? b : en;
                }
            }
        } else {
            float cy = dHy, cx = dHx;
            if constexpr (XS) {
                pex[i] = Le.b * pex[i] + Le.a * dHy;
                cy = dHy * Le.k + dxf * pex[i];
            }
            if constexpr (YS) {
                pey[i] = W.b * pey[i] + W.a * dHx;
                cx = dHx * W.k + dyf * pey[i];
            }
            if constexpr (MAT) {
                en = A.x * e0 + A.y * cy - A.y * cx - B.x * jp[i];
                if constexpr (SRC) {
                    if (i == opaque(isrc)) en = lsrc ? en + s : en;
                }
                // (a PEC node: Ez stays 0, and so does Jp)
                if constexpr (XS || YS) en = eok ? en : 0.f;
                jp[i] = B.y * jp[i] + B.z * (en - e0);
            } else {
                // the material expression with Ez coefficient 1 and no Jp: the same roundings
                const float u = cb0 * cy;
                const float v = e0 + u;
                en = v - cb0 * cx;
                if constexpr (XS || YS) en = eok ? en : 0.f;
            }
        }
        if constexpr (REF && (XS || YS)) en = eok ? en : 0.f;
        ez[i] = en;
    };
    const Profile<REF>* we = lds.row_e + wv * R;      // E row i
    const Profile<REF>* wh = lds.row_h + wv * R + 1;  // H row i
    // Physical mode holds its rows' profiles in registers for the whole block:
    // read from LDS in each step, they were 12 to 24 waits on the way of a wave
    // with one other to hide behind (256^2 2.65 -> 2.36 ms per evaluation, 64 of
    // 512^2 88.0 -> 85.2).  The reference's, with 64-bit kappa, do not fit.
    constexpr bool HELD = YS && !REF;
    Profile<REF> he[HELD ? R : 1], hh[HELD ? R + 1 : 1];
    if constexpr (HELD) {
#pragma unroll
        for (int i = 0; i < R; ++i) he[i] = we[i];
#pragma unroll
        for (int i = 0; i <= R; ++i) hh[i] = wh[i - 1];
    }
    auto E = [&](int i) {
        if constexpr (HELD) return he[i];
        else return YS ? we[i] : Profile<REF>{};
    };
    auto H = [&](int i) {
        if constexpr (HELD) return hh[i + 1];
        else return YS ? wh[i] : Profile<REF>{};
    };
    auto hs = [&](int i, float up) {
        h_step(ez[i], up, hx[i], &hy[i], XS ? &phx[XS ? i : 0] : nullptr, YS ? &phy[YS ? i : 0] : nullptr, H(i));
    };

    // The reference's NaN clamp: NaN rows are looked for in pairs of values, and
    // the values replaced only where one was found (a compare and a select per
    // value cost a third of the reference's vacuum stage).
    auto clamp_nan = [&](bool bad, auto fix) {
        if (clamp && __builtin_amdgcn_ballot_w64(bad)) fix();
    };
    auto no_nan = [](float& v) { v = __builtin_isnan(v) ? 0.f : v; };

    const int wu = min(wv + 1, NW - 1), wd = max(wv - 1, 0);
    for (int t = 0; t < nst; ++t) {
        const int n = step0 + t, b = t & 1;
        const float s = SRC ? read_lane(sw, t) : 0.f;
        lds.ez[b][wv][0][lane] = ez[0];
        lds.ez[b][wv][1][lane] = ez[R - 1];
        // what needs no neighbour covers the exchange: H of all rows but the top
        // one before the barrier, E of the rows in between while the reads return
#pragma unroll
        for (int i = 0; i + 1 < R; ++i) hs(i, ez[i + 1]);
        if constexpr (REF) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i + 1 < R; ++i) bad |= __builtin_isunordered(hx[i], hy[i]);
            clamp_nan(bad, [&] {
#pragma unroll
                for (int i = 0; i + 1 < R; ++i) {
                    no_nan(hx[i]);
                    no_nan(hy[i]);
                }
            });
        }
        const float ez0 = ez[0];
#pragma unroll
        for (int i = 1; i + 1 < R; ++i) e_step(i, hx[i - 1], n, s, E(i), false);
        lds_barrier();
        float ez_up = lds.ez[b][wu][0][lane], ez_dn = lds.ez[b][wd][1][lane];
        if constexpr (YS) {
            ez_up = top ? 0.f : ez_up;
            ez_dn = bot ? 0.f : ez_dn;
        }
        h_step(ez_dn, ez0, hxb, nullptr, nullptr, &phyb, H(-1));
        hs(R - 1, ez_up);
        if constexpr (REF)
            clamp_nan(__builtin_isunordered(hx[R - 1], hy[R - 1]) || __builtin_isnan(hxb), [&] {
                no_nan(hx[R - 1]);
                no_nan(hy[R - 1]);
                no_nan(hxb);
            });
        e_step(0, hxb, n, s, E(0), bot);
        e_step(R - 1, hx[R - 2], n, s, E(R - 1), top);
        if constexpr (REF) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < R; i += 2) bad |= __builtin_isunordered(ez[i], ez[i + 1]);
            clamp_nan(bad, [&] {
#pragma unroll
                for (int i = 0; i < R; ++i) no_nan(ez[i]);
            });
        }
        if (extra) {
            if constexpr (!MAT && !REF) {
                // a source in vacuum: Jp does not see it, so it can be added to the finished row
                if (wsrc) {
                    const int is = opaque(isrc);
                    const float sv = read_lane(sw, t);
#pragma unroll
                    for (int i = 0; i < R; ++i)
                        if (i == is) ez[i] = lsrc ? ez[i] + sv : ez[i];
                }
            }
            sample(k0 + t);
        }
    }

    // ---- owned cells to the other buffer
    const int keep = opaque(mine);
    const unsigned wx = own ? vx : kOff, we4 = own ? ve : kOff, wh4 = own ? vh : kOff;
    const int po = opaque(par ^ 1), yo = opaque(yb);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        if (!(keep >> i & 1)) continue;  // wave-uniform
        const int y = yo + i, o = po * plane + y * row4;
        st(F, wx, o, ez[i]);
        st(F, wx, o + 2 * plane, hx[i]);
        st(F, wx, o + 4 * plane, hy[i]);
        if constexpr (MAT) st(Jb, own ? jp_off(y) : kOff, po * Sp->js * 4, jp[i]);
        if constexpr (XS) {
            const int q = (po * Sp->xs + y * w2) * 4;
            st(Q, we4, q, pex[i]);
            st(Q, wh4, q + Sp->xs * 8, phx[i]);
        }
        if constexpr (YS) {
            if (row_e(y)) st(Y, wx, (po * Sp->ys + (y + re0) * pitch) * 4, pey[i]);
            if (row_h(y)) st(Y, wx, ((po + 2) * Sp->ys + (y + rh0) * pitch) * 4, phy[i]);
        }
    }
}

// Bring the lines of a lone simulation's description that a tile reads, and its
// launch item, into the scalar cache while the tile itself is on its way (they
// are found through it: without this, three round trips before the first load
// of the state; 0.2 us a launch, 363^2 6.62 -> 6.52 ms per evaluation).
__device__ __forceinline__ void warm(const DevSim* __restrict__ lone, const LaunchItem* __restrict__ items) {
    if (!lone) return;
    constexpr int a = (int)(offsetof(DevSim, coef) + 63) / 64, b = (int)offsetof(DevSim, chx) / 64,
                  c = (int)offsetof(DevSim, inc_abs_origin) / 64;
    const kcint* q = (const kcint*)lone;
    int v[a + 1 + c - b + 1];
#pragma unroll
    for (int i = 0; i <= a; ++i) v[i] = q[16 * i];
#pragma unroll
    for (int i = b; i <= c; ++i) v[a + 1 + i - b] = q[16 * i];
    const int w = ((const kcint*)items)[0];
#pragma unroll
    for (int i = 0; i < a + 1 + c - b + 1; ++i) asm volatile("" ::"s"(v[i]));
    asm volatile("" ::"s"(w));
}

// Workgroups of a launch, after the tiles', that fold the previous epoch's
// samples: bx blocks of contour points x bz groups of fpb frequencies per item.
// The tiles of this launch write other sample rows (LaunchItem::samp0).  A fold
// is bound by its launch and the latency of its loads; beside the tiles it
// costs one simulation nothing that can be measured.
constexpr int kFoldFreqs = 8;
struct FoldShare {
    const LaunchItem* items;
    int blocks, bx, bz, fpb;
};

// Workgroups are dealt to the eight XCDs round-robin: XCD g walks the g-th
// contiguous eighth of the tile list, so that tiles that share halo rows and
// columns share an L2 (64 simulations of 512^2: 640 -> 237 MB read per launch,
// 203 -> 193 us; 4 x 401^2 20.2 -> 17.5 us).
// Aligned, so that a change to one instance does not move the others: the same
// instructions 2 KiB further on were 1.3% slower (mixed requests of 362 to 1448,
// 51.5 -> 52.2 us a launch).
template <int MODE, int NW>
__global__ __launch_bounds__(NW* kLane) __attribute__((amdgpu_waves_per_eu(4), aligned(4096))) void k_rtile(
    const RegTile* __restrict__ tiles, int ntiles, const LaunchItem* __restrict__ items, const DevSim* __restrict__ sims, int ordinal,
    int tsteps, const DevSim* __restrict__ lone, FoldShare fold) {
    __shared__ union {
        TileLds<MODE == TOMO_MODE_REF_COMPAT, NW> tile;
        struct { float2 wJ[kFoldFreqs * 64], wM[kFoldFreqs * 64]; } fold;
    } u;
    TileLds<MODE == TOMO_MODE_REF_COMPAT, NW>& lds = u.tile;
    const int tblocks = gridDim.x - fold.blocks;
    if ((int)blockIdx.x >= tblocks) {
        const int b = blockIdx.x - tblocks, z = b / fold.bx, item = z / fold.bz;
        const LaunchItem it = fold.items[item];
        const DevSim* S = sims + it.sim;
        const int fb = (z - item * fold.bz) * fold.fpb, nf = min(S->nfreq, fb + fold.fpb) - fb;
        const int nk = min(it.nsteps, S->chunk), p = (b - z * fold.bx) * (NW * kLane) + threadIdx.x;
        if (nk <= 0 || nf <= 0) return;
        if (fold.fpb == 1) fold_fp32<1>(S, it, nk, fb, nf, p, u.fold.wJ, u.fold.wM);
        else fold_fp32<kFoldFreqs>(S, it, nk, fb, nf, p, u.fold.wJ, u.fold.wM);
        return;
    }
    const int ti = (blockIdx.x & 7) * (tblocks >> 3) + (blockIdx.x >> 3);
    if (ti >= ntiles) return;
    const RegTile tile = tiles[ti];
    if constexpr (MODE == TOMO_MODE_PHYSICAL) warm(lone, items);
    if (tile.item < 0) return;  // an unused place of an XCD's share
    const LaunchItem it = items[tile.item];
    const DevSim* Sp = sims + tile.sim;
    const int nst = min(tsteps, it.nsteps - ordinal * tsteps);
    if (nst <= 0) return;  // uniform over the workgroup
    const int lane = threadIdx.x & (kLane - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kLane);
    const int par = it.parity0 ^ (ordinal & 1), step0 = it.step0 + ordinal * tsteps, k0 = it.samp0 + ordinal * tsteps;
    const int nx = Sp->nx, ny = Sp->ny, nc = Sp->nc;
    const int rows = tile.rows, yb = tile.yl + wv * rows;
    const bool mat = (tile.matmask >> wv) & 1;
    const bool xs = tile.xl <= nc || tile.xl + kLane > nx - nc;  // lanes reach a strip or an edge
    const bool tys = tile.yl <= nc + 1 || tile.yl + NW * rows > ny - nc;
    // rows reach a strip or an edge (the row below the wave is advanced too)
    const bool ys = yb <= nc + 1 || yb + rows > ny - nc;
    const bool tsrc = MODE == TOMO_MODE_PHYSICAL && Sp->sy >= tile.yl && Sp->sy < tile.yl + NW * rows &&
                      Sp->sx >= tile.xl && Sp->sx < tile.xl + kLane;
    const bool src = tsrc && mat && Sp->sy >= yb && Sp->sy < yb + rows;
    // row profiles: also where the source lies in material, whose wave takes the general stage
    const bool frows = tys || (tsrc && tile.matmask);
    const bool tables = tile.matmask || frows;
#define TW(R, XS, YS, MAT, SRC) \
    tile_wave<MODE, R, NW, XS, YS, MAT, SRC>(tile, Sp, lds, par, step0, k0, nst, wv, lane, tables, frows)
    if (rows == kTileRowsTall) {
        TW(kTileRowsTall, false, false, false, false);
        return;
    }
    if (rows == kTileRowsClean) {  // at the strips of one axis at most, material clear of them
        constexpr int R = kTileRowsClean;
        if constexpr (MODE == TOMO_MODE_PHYSICAL) {  // (reference-mode material takes 4-row tiles)
            if (mat) {
                TW(R, false, false, true, false);
                return;
            }
        }
        if (xs) TW(R, true, false, false, false);
        else if (ys) TW(R, false, true, false, false);
        else TW(R, false, false, false, false);
        return;
    }
    constexpr int R = kTileRowsEdge;
    if (src) TW(R, true, true, true, true);
    else if (mat) {
        if (xs) {
            if (ys) TW(R, true, true, true, false);
            else TW(R, true, false, true, false);
        } else if (ys) TW(R, false, true, true, false);
        else TW(R, false, false, true, false);
    } else if (xs) {
        if (ys) TW(R, true, true, false, false);
        else TW(R, true, false, false, false);
    } else if (ys) TW(R, false, true, false, false);
    else TW(R, false, false, false, false);
#undef TW
}

}  // namespace

hipError_t launch_rtile(int mode, int waves, const RegTile* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                        int ordinal, int tsteps, const DevSim* lone, const FoldRun& f, hipStream_t st) {
    if (ntiles <= 0) return hipErrorInvalidValue;
    FoldShare fold{};
    if (f.n > 0) {
        const int wg = waves * kLane;
        fold.items = f.items;
        fold.bx = (f.max_p + wg - 1) / wg;
        // fewer than about one block per CU: spread the frequencies too (as launch_fold)
        fold.fpb = (f.max_p + 255) / 256 * f.n < 256 ? 1 : kFoldFreqs;
        fold.bz = (f.max_f + fold.fpb - 1) / fold.fpb;
        fold.blocks = fold.bx * fold.bz * f.n;
    }
    dim3 g((ntiles + 7) / 8 * 8 + fold.blocks), b(waves * kLane);
#define TT(MM, WW)                                                                                        \
    if (mode == MM && waves == WW) {                                                                      \
        TIMED_LAUNCH((k_rtile<MM, WW>), g, b, 0, st, tiles, ntiles, items, sims, ordinal, tsteps, lone, fold);  \
        return hipGetLastError();                                                                         \
    }
    TT(TOMO_MODE_PHYSICAL, 8) TT(TOMO_MODE_PHYSICAL, 16) TT(TOMO_MODE_REF_COMPAT, 8)
#undef TT
    return hipErrorInvalidValue;
}

}  // namespace tomo
