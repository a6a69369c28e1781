// og_pair.hip -- LJ + zero-dipole cell-pair kernel, excluded-pair (excess)
// and bond terms, fixed-point gradient reduction and energy reductions.
//
// Pair kernel (reference: kernel_pairwise_ljzd + cal_pair, cuda_setup.cu:487-675;
// CPU: SubBox::calc_energy_pairwise, SubBox.cpp:956-1125).  It evaluates the
// same pairs as the reference -- every unmasked atom pair of every listed
// cell pair closer than the cutoff -- but schedules them for a wave64:
//
// * one wave per cell1 (the last cells of a large system: two waves, each
//   with half of the cell's records); its 8 atoms ("i") sit in scalar registers;
// * filter: the wave reads its cell pairs 8 at a time (lane = 8*pair + j) and
//   keeps the cell2 atoms ("rows") within the cutoff of the cell1 bounding
//   box, appending them (shifted to the pair's periodic image) to a per-wave
//   LDS queue.  About half of the rows of a 13 A list survive at 12 A;
// * rows: every 64 queued rows are one pass with lane = row, looping over
//   the 8 i atoms.  The row's j-gradient stays in its lane (no cross-lane
//   reduction) and is added once as 64-bit fixed point; each lane keeps 24
//   partial i-gradients, reduced over the wave once per cell1.
//
// FP32 pair math as the reference, fixed-point atomics (order-independent,
// so every run gives the same bits), energies summed per lane in FP64 and
// reduced per cell in a fixed order.
#include "og_terms.h"

#define OG_CHARGE_COEFF 332.06378f   // CelesteObject.cpp:36
#define OG_QCAP 128                  // per-wave row queue (two passes of 64)
#define OG_LJ_LDS_ENTRIES(FORM) ((FORM) == 2 ? 256 : 512)  // LJ table entries (whole leading rows, 4 KB) in LDS

typedef float og_f4 __attribute__((ext_vector_type(4)));
typedef float og_f2 __attribute__((ext_vector_type(2)));

// Pair forms (the FORM template argument): 0 = LJ + zero-dipole at alpha 0,
// 1 = LJ + zero-dipole at alpha > 0 (cal_pair, cuda_setup.cu:487-521),
// 2 = hydrophobicity-scale LJ + Debye-Hueckel (cal_pair_hps_dh,
// cuda_setup.cu:1273-1332), 3 / 4 = LJ + zero-quadrupole, -octupole or
// -hexadecapole at alpha 0 / > 0 (the reference's host forms,
// ZeroMultipoleSum.cpp:347-442).  The LJ table entry is {A6, A12} for forms 0 and
// 1 and {A6, A12, HPS switch distance, HPS lambda} for form 2.
template <int FORM> struct og_ljt { typedef og_f2 type; };
template <> struct og_ljt<2> { typedef og_f4 type; };

// erfc(x) for x >= 0 from Abramowitz & Stegun 7.1.26 (|abs error| <= 1.5e-7),
// sharing exp(-x^2) with the force term.
__device__ __forceinline__ float og_erfc_as(float x, float expmx2) {
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, x, 1.0f));
    float       p = fmaf(t, 1.061405429f, -1.453152027f);
    p             = fmaf(t, p, 1.421413741f);
    p             = fmaf(t, p, -0.284496736f);
    p             = fmaf(t, p, 0.254829592f);
    return p * t * expmx2;
}

__device__ __forceinline__ float og_rlane(float v, int k) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// a uniform value kept in a vector register: an FP32 add, multiply or fma
// with a scalar-register operand issues at half the rate of one without
// (4.2-4.5 cycles per wave against 2.2 measured on gfx950)
__device__ __forceinline__ float og_vgpr(float v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <int CTRL> __device__ __forceinline__ float og_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Cell1 data held by the wave, the same in every lane: atom coordinates and
// charge * 332.06378 (vector registers, see og_vgpr), LJ row offsets (type *
// n_types, the same in the global table and in the block's LDS copy of its
// leading rows; scalar) and the bounding box.
struct og_cell1 {
    float    x[OG_NAC], y[OG_NAC], z[OG_NAC], q[OG_NAC];
    unsigned row[OG_NAC];
    float    lo[3], hi[3];
};

// Sums of a row over the cell1 atoms, in atom order: j-gradient (before its
// sign), LJ and electrostatic energy, virial.
struct og_chain {
    float x, y, z, e, q, v;
};

// j-gradient of the last pass, not yet added: its fixed-point atomics are
// issued after the next pass has read its rows, so they complete while that
// pass computes.  (A vector-memory wait counts stores and atomics too, so an
// atomic issued just before a load that is waited on stalls the wave until
// the memory-side add has completed.)
struct og_jpend {
    float x, y, z;
    int   a;
    bool  live;
};

// Fixed-point add of a lane's gradient (x, y, z) at grid slot a (the
// j-gradient enters with a minus sign).  Zero contributions are skipped.
__device__ __forceinline__ void og_add_fx3(OG_GLOBAL(long long) *FX, int cap, int a, double sx, double sy,
                                           double sz) {
    const size_t    stride = OG_FX_CAP(cap);
    const long long vx = og_fx_fast(sx), vy = og_fx_fast(sy), vz = og_fx_fast(sz);
    if (vx != 0) og_atomic_add_fx_g(FX + a, vx);
    if (vy != 0) og_atomic_add_fx_g(FX + stride + a, vy);
    if (vz != 0) og_atomic_add_fx_g(FX + 2 * stride + a, vz);
}

// j-gradient of a row at 2^19 units: (x, y) packed into one 64-bit atomic, z
// into one 32-bit atomic.  The memory-side atomics cost per request and per
// byte, so two per row instead of three (z of a slot pair in one 64-bit word,
// added for two neighbouring rows at once, took 133 us at 99,200 atoms against
// 127 for this; x, y and z as three 32-bit words 145).  The (x, y) word is
// built in 32-bit halves and the words are addressed as a uniform base plus a
// 32-bit byte offset (no 64-bit index arithmetic).  Called by the whole wave.
__device__ __forceinline__ void og_flush_j(OG_GLOBAL(char) *FXJ, OG_GLOBAL(char) *FXZ, og_jpend &p) {
    if (p.live) {
        const unsigned f  = (unsigned)og_fx_slot(p.a);
        const int      fx = (int)__builtin_rintf(-p.x * 524288.0f);  // |x| < 4096: exact scaling, half-even rounding
        const int      fy = (int)__builtin_rintf(-p.y * 524288.0f);
        const int      fz = (int)__builtin_rintf(-p.z * 524288.0f);
        // the 64-bit sum x + y * 2^32 of sign-extended fields
        const unsigned xlo = (unsigned)fx, xhi = (unsigned)(fy + (fx >> 31));
        if (xlo | xhi)
            __hip_atomic_fetch_add((OG_GLOBAL(unsigned long long) *)(FXJ + (f << 3)), ((unsigned long long)xhi << 32) | xlo,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (fz)
            __hip_atomic_fetch_add((OG_GLOBAL(int) *)(FXZ + (f << 2)), fz, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    p.live = false;
}

// One pass over up to 64 queued rows (lane = row; lanes >= cnt idle).
// m8: the row's excluded pairs (bit i set = skip atom i).  LJ_LDS: the
// cell1's types are rows of the block's LDS copy of the LJ table.  The
// i-gradients are added to fi, or (COEF, a team wave) each pair's gradient
// coefficient is left in fi[i] for the wave that sums atom i.
template <int FORM, bool ENERGY, bool LJ_LDS, bool COEF>
__device__ __forceinline__ void og_rows(const og_dev_sys &s, const og_cell1 &c, const og_f4 pj, const unsigned tj,
                                        const unsigned m8, const typename og_ljt<FORM>::type *__restrict__ ljl,
                                        const OG_GLOBAL(typename og_ljt<FORM>::type) *__restrict__ LJP,
                                        float (&fi)[COEF ? OG_NAC : 3 * OG_NAC], int &npair, og_chain &ch) {
    const float rc2 = s.cutoff2;
    const float zcore = og_vgpr(s.zcore), bcoeff = og_vgpr(s.bcoeff), fcoeff = og_vgpr(s.fcoeff);
    const float alpha = s.alpha, piewald = s.piewald;
    const float hps_eps = s.hps_eps, kappa = s.dh_kappa;
    const float zmc = s.zm_core, ze0 = s.zm_c[0], ze1 = s.zm_c[1], ze2 = s.zm_c[2], ze3 = s.zm_c[3];
    const float zg0 = s.zm_pg[0], zg1 = s.zm_pg[1], zg2 = s.zm_pg[2], zg3 = s.zm_pg[3];
    const bool  dh_fix_on = s.dh_grad_fix != 0;
    float fjx = 0.0f, fjy = 0.0f, fjz = 0.0f, fe = 0.0f, fq = 0.0f, fv = 0.0f;
    float px = pj.x, py = pj.y, pz = pj.z, pw = pj.w;
    // the row's LJ pairs {A6, A12} load together, ahead of their use
    typename og_ljt<FORM>::type ljv[OG_NAC];
#pragma unroll
    for (int i = 0; i < OG_NAC; i++) ljv[i] = LJ_LDS ? ljl[c.row[i] + tj] : LJP[c.row[i] + tj];
    // the tables hold {6 A6, 12 A12}; a caller's table in the reference's {A6, A12} is scaled here
    if (s.lj_unscaled) {
#pragma unroll
        for (int i = 0; i < OG_NAC; i++) {
            ljv[i].x *= 6.0f;
            ljv[i].y *= 12.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < OG_NAC; i++) {
        const float dx = c.x[i] - px;
        const float dy = c.y[i] - py;
        const float dz = c.z[i] - pz;
        const float r2 = dx * dx + dy * dy + dz * dz;
        const bool  in = r2 < rc2, unmasked = !((m8 >> i) & 1u);
        const bool  ok = in && unmasked;
        // the pair count on the scalar unit: each ballot is its compare's lane mask as it stands
        if constexpr (ENERGY)
            npair += __builtin_popcountll(__builtin_amdgcn_ballot_w64(in) & __builtin_amdgcn_ballot_w64(unmasked));
        const typename og_ljt<FORM>::type lj = ljv[i];  // {6 A6, 12 A12(, HPS switch, HPS lambda)}
        // ZSEL (energy steps, forms 0, 1, 3, 4): a pair that is not evaluated
        // gets 1/r = 0 and charge product 0, which zero its gradient and both
        // energies (one select instead of three); the HPS form's short-range
        // constant needs the selects
        constexpr bool ZSEL = ENERGY && FORM != 2;
        const float rinv  = ZSEL && !ok ? 0.0f : __builtin_amdgcn_rsqf(r2);
        const float r2inv = rinv * rinv;
        const float r6inv = r2inv * r2inv * r2inv;
        // r^2 times the LJ gradient coefficient, 6 A6 r^-6 - 12 A12 r^-12, and (energy steps) the LJ energy
        const float lji   = fmaf(-lj.y, r6inv, lj.x);
        const float ljf   = r6inv * lji;
        const float cc    = ZSEL && !ok ? 0.0f : c.q[i] * pw;
        float       g, eel, elj = 0.0f;
        // LJ energy: forms 0, 1, 3, 4 keep -12 times it, r^-6 (6 A6 + lji) = r^-6 (12 A6 - 12 A12 r^-6), and the
        // cell's sum is scaled once (two fewer instructions per pair slot); the HPS form keeps the energy itself
        if constexpr (ENERGY) {
            if constexpr (FORM == 2) elj = r6inv * fmaf(lj.y * (1.0f / 12.0f), r6inv, lj.x * (-1.0f / 6.0f));
            else elj = r6inv * (lj.x + lji);
        }
        if constexpr (FORM == 0) {
            eel = cc * (rinv - zcore + bcoeff * r2);
            g   = r2inv * ljf - cc * (rinv * r2inv - fcoeff);
        } else if constexpr (FORM == 2) {
            // HPS: beyond the pair's switch distance lambda * LJ, inside it LJ + (1 - lambda) eps;
            // Debye-Hueckel: cc (charges x 332.06378 / eps_r) exp(-kappa r) / r, gradient coefficient
            // -E (1/r + kappa) as the reference (times 1/r with the gradient fix)
            const float r   = r2 * rinv;
            const bool  far = r > lj.z;
            const float sc  = far ? lj.w : 1.0f;
            elj             = fmaf(elj, sc, far ? 0.0f : (1.0f - lj.w) * hps_eps);
            eel             = cc * rinv * __expf(-r * kappa);
            g = sc * r2inv * ljf - eel * (rinv + kappa) * (dh_fix_on ? rinv : 1.0f);
        } else if constexpr (FORM == 3 || FORM == 4) {
            // zero-quadrupole/-octupole/-hexadecapole: the order's polynomials in r^2 by Horner's rule
            const float pe = r2 * fmaf(r2, fmaf(r2, fmaf(r2, ze3, ze2), ze1), ze0);
            const float pg = fmaf(r2, fmaf(r2, fmaf(r2, zg3, zg2), zg1), zg0);
            if constexpr (FORM == 3) {
                eel = cc * (rinv - zmc - pe);
                g   = r2inv * ljf - cc * (rinv * r2inv + pg);
            } else {
                const float r   = r2 * rinv;
                const float ar  = alpha * r;
                const float ex  = __expf(-ar * ar);
                const float erc = og_erfc_as(ar, ex);
                eel = cc * (rinv * erc - zmc - pe);
                g   = r2inv * ljf - cc * (erc * rinv * r2inv + piewald * ex * r2inv + pg);
            }
        } else {
            const float r   = r2 * rinv;
            const float ar  = alpha * r;
            const float ex  = __expf(-ar * ar);
            const float erc = og_erfc_as(ar, ex);
            eel = cc * (rinv * erc - zcore + bcoeff * r2);
            g   = r2inv * ljf - cc * (erc * rinv * r2inv + piewald * ex * r2inv - fcoeff);
        }
        // lanes without a pair (masked, out of range, idle) contribute exact zeros
        if (!ZSEL) g = ok ? g : 0.0f;
        fjx               = fmaf(g, dx, fjx);
        fjy               = fmaf(g, dy, fjy);
        fjz               = fmaf(g, dz, fjz);
        if constexpr (COEF) {
            fi[i] = g;
        } else {
            fi[3 * i]     = fmaf(g, dx, fi[3 * i]);
            fi[3 * i + 1] = fmaf(g, dy, fi[3 * i + 1]);
            fi[3 * i + 2] = fmaf(g, dz, fi[3 * i + 2]);
        }
        if (ENERGY) {
            fe += ZSEL || ok ? elj : 0.0f;
            fq += ZSEL || ok ? eel : 0.0f;
            fv = fmaf(g, r2, fv);
        }
        // finish atom i here: without this the compiler defers the
        // accumulations and keeps all 8 atoms' distances live
        if constexpr (COEF)
            asm volatile("" : "+v"(fjx), "+v"(fjy), "+v"(fjz), "+v"(fi[i]), "+v"(px), "+v"(py), "+v"(pz), "+v"(pw));
        else
            asm volatile("" : "+v"(fjx), "+v"(fjy), "+v"(fjz), "+v"(fi[3 * i]), "+v"(fi[3 * i + 1]),
                         "+v"(fi[3 * i + 2]), "+v"(px), "+v"(py), "+v"(pz), "+v"(pw));
        if constexpr (ENERGY) asm volatile("" : "+v"(fe), "+v"(fq), "+v"(fv));
    }
    ch = og_chain{fjx, fjy, fjz, fe, fq, fv};
}

// range check of a pass's j-gradients; fmaxf drops NaN, the sum keeps it
__device__ __forceinline__ void og_range(const og_chain &ch, float &vmax, float &vsum) {
    vmax = fmaxf(vmax, fmaxf(fabsf(ch.x), fmaxf(fabsf(ch.y), fabsf(ch.z))));
    vsum += ch.x + ch.y + ch.z;
}

// Pass over queue entries [q0, q0 + cnt) (q0 a multiple of 64): reads the
// rows, adds the previous pass's j-gradient, then evaluates the rows.
template <int FORM, bool ENERGY, bool LJ_LDS>
__device__ __forceinline__ void og_pass(const og_dev_sys &s, const og_cell1 &c, const og_f4 *qp, const int2 *qa,
                                        const int q0, const int cnt, const typename og_ljt<FORM>::type *ljl,
                                        const OG_GLOBAL(typename og_ljt<FORM>::type) *__restrict__ LJP,
                                        OG_GLOBAL(char) *FXJ, OG_GLOBAL(char) *FXZ, float (&fi)[3 * OG_NAC],
                                        int &npair, float &vmax, float &vsum, double &ev, double &ee, double &vir,
                                        og_jpend &pend) {
    const int  lane = threadIdx.x & 63;
    const int  slot = (q0 & (OG_QCAP - 1)) + lane;
    const bool live = lane < cnt;
    og_f4      pj   = qp[slot];
    const int2 ax   = qa[slot];
    unsigned   m8 = (unsigned)ax.y >> 24, tj = (unsigned)ax.y & 0xffffffu;
    // idle lanes (stale queue slots): finite coordinates, LJ column 0, every pair masked
    if (cnt < 64) {
        if (!live) pj = og_f4{0.0f, 0.0f, 0.0f, 0.0f};
        m8 = live ? m8 : 0xffu;
        tj = live ? tj : 0u;
    }
    // every outstanding load of the filter is complete before the atomics go
    // out, so nothing in the pass waits on the vector-memory counter
    // (s_waitcnt vmcnt(0); expcnt and lgkmcnt left at their maxima)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    og_flush_j(FXJ, FXZ, pend);
    og_chain ch;
    og_rows<FORM, ENERGY, LJ_LDS, false>(s, c, pj, tj, m8, ljl, LJP, fi, npair, ch);
    og_range(ch, vmax, vsum);
    pend = og_jpend{ch.x, ch.y, ch.z, ax.x, live};
    if (ENERGY) {
        ev += (double)ch.e;
        ee += (double)ch.q;
        vir += (double)ch.v;
    }
}

// What the filter reads: grid-order atoms and types, cell-pair records.
struct og_list {
    const OG_GLOBAL(char) *X, *TY, *CP, *CM;
};
// Cell-pair record of a lane (lane = 8 * record + j atom): cell2 | image << 24
// and the j atom's mask byte.
struct og_rec {
    unsigned cp, m8;
};
// The group of eight records at base.  Uniform base plus a lane offset that is
// constant but for the last group, where lanes past the end read its last record.
__device__ __forceinline__ og_rec og_load_rec(const og_list &L, const int base, const int p1) {
    const int lane = threadIdx.x & 63;
    const int b = min(base, p1 - 1), r = p1 - b;
    unsigned  k = (unsigned)lane >> 3;
    if (r < OG_NAC) k = min(k, (unsigned)(r - 1));
    og_rec t;
    t.cp = *(const OG_GLOBAL(unsigned) *)(L.CP + 4 * (size_t)b + 4u * k);
    t.m8 = *((const OG_GLOBAL(unsigned char) *)(L.CM + 8 * (size_t)b) + (8u * k + (unsigned)(lane & 7)));
    return t;
}
struct og_jatom {
    og_f4    p;
    unsigned ty;
};
__device__ __forceinline__ og_jatom og_load_atom(const og_list &L, const unsigned cp) {
    const unsigned off = ((cp << 7) & 0x7fffffffu) | ((threadIdx.x & 7u) << 4);  // 16 bytes per slot
    og_jatom       t;
    t.p  = *(const OG_GLOBAL(og_f4) *)(L.X + off);
    t.ty = *(const OG_GLOBAL(unsigned) *)(L.TY + (off >> 2));
    return t;
}
// Filter of one group: shifts the lanes' atoms to their pairs' periodic images
// and returns the mask of the lanes to keep (within the cutoff of the cell1
// box and not masked against all its atoms).  A row without a number for its
// distance is kept, so its pairs flag the evaluation.
__device__ __forceinline__ uint64_t og_keep(const float (&lo)[3], const float (&hi)[3], const float rcb2,
                                            const og_f4 *__restrict__ shift, const unsigned cp, const unsigned m8,
                                            og_f4 &p) {
    if (__builtin_amdgcn_ballot_w64(cp > 0xffffffu)) {  // a periodic image among the group's pairs
        const og_f4 sh = shift[(cp >> 24) & 63u];
        p.x += sh.x;
        p.y += sh.y;
        p.z += sh.z;
    }
    const float gx = p.x - __builtin_amdgcn_fmed3f(p.x, lo[0], hi[0]);
    const float gy = p.y - __builtin_amdgcn_fmed3f(p.y, lo[1], hi[1]);
    const float gz = p.z - __builtin_amdgcn_fmed3f(p.z, lo[2], hi[2]);
    return __builtin_amdgcn_ballot_w64(!(fmaf(gz, gz, fmaf(gx, gx, gy * gy)) >= rcb2)) &
           __builtin_amdgcn_ballot_w64(m8 != 0xffu);
}
// The cell1's atoms and box from the lanes' atoms p and types ty (lane & 7).
template <int FORM>
__device__ __forceinline__ void og_set_cell1(const og_dev_sys &s, const og_f4 p, const int ty, og_cell1 &c) {
    // charge x 332.06378 (x 1/eps_r under Debye-Hueckel)
    const float qc = FORM == 2 ? p.w * OG_CHARGE_COEFF * s.dh_diel_inv : p.w * OG_CHARGE_COEFF;
#pragma unroll
    for (int i = 0; i < OG_NAC; i++) {
        c.x[i]   = og_rlane(p.x, i);
        c.y[i]   = og_rlane(p.y, i);
        c.z[i]   = og_rlane(p.z, i);
        c.q[i]   = og_rlane(qc, i);
        c.row[i] = (unsigned)__builtin_amdgcn_readlane(ty, i) * (unsigned)s.n_types;
    }
    // bounding box: minima and maxima over the eight lanes
    float lo[3] = {p.x, p.y, p.z}, hi[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        lo[k]   = fminf(lo[k], og_dpp<0xB1>(lo[k]));
        hi[k]   = fmaxf(hi[k], og_dpp<0xB1>(hi[k]));
        lo[k]   = fminf(lo[k], og_dpp<0x4E>(lo[k]));
        hi[k]   = fmaxf(hi[k], og_dpp<0x4E>(hi[k]));
        c.lo[k] = fminf(lo[k], og_dpp<0x141>(lo[k]));
        c.hi[k] = og_rlane(fmaxf(hi[k], og_dpp<0x141>(hi[k])), 0);  // one scalar operand per instruction
    }
}

// What a work unit starts from.
struct og_unit {
    int   c1, p0, p1;  // its cell and records (scalar)
    og_f4 p;           // the cell's atom of the lane (lane & 7)
    int   ty;
    bool  run, energy;
};
// Work unit u of a system with n cells: cells 0 .. n-m-1 whole, then the last
// m cells as two units each (first and second half of their records).  run is
// false past the last unit, for a frozen system and after a list overflow.  It
// is the one field that two waves of a launch may read differently, as units
// that run flag an overlap (OG_F_NAN) meanwhile.
// The list head, the cell's atoms and the counters are read together (a unit
// is a chain of memory round trips of about a microsecond each: block map,
// system record, these, the records, their atoms); only a unit of the split
// tail, whose cell follows from the cell count, reads its own again.
__device__ __forceinline__ og_unit og_unit_start(const og_dev_sys &s, const int u) {
    const int jl = threadIdx.x & 7;
    og_unit   t;
    t.c1 = min(u, s.head_cells - 1);
    int             a = s.cp_head[t.c1], b = s.cp_head[t.c1 + 1];
    const OG_GLOBAL(og_f4) *X  = (const OG_GLOBAL(og_f4) *)s.gxyzq;
    const OG_GLOBAL(int) *TY   = (const OG_GLOBAL(int) *)s.gtype;
    t.p  = X[t.c1 * OG_NAC + jl];
    t.ty = TY[t.c1 * OG_NAC + jl];
    const og_dev_counters &c = *s.cnt;
    const int              n = c.n_cells, m = og_pair_split_cells(s.pair_split, n);
    // keeps these loads ahead of the branches on the counters
    asm volatile("" ::"v"(t.p.x), "v"(t.ty), "s"(a), "s"(b));
    t.run    = !og_frozen_c(c) && !(c.flags & OG_F_CP_OVERFLOW) && u < n + m;
    t.energy = og_energy_step_c(s, c);
    if (u >= n - m && u < n + m) {  // whatever run is: which cell a unit is must not hang on the flags
        const int half = (u - (n - m)) & 1;
        t.c1 = n - m + ((u - (n - m)) >> 1);
        a    = s.cp_head[t.c1], b = s.cp_head[t.c1 + 1];
        t.p  = X[t.c1 * OG_NAC + jl];
        t.ty = TY[t.c1 * OG_NAC + jl];
        const int mid = a + ((b - a + 1) >> 1);
        if (half == 0) b = mid;
        else a = mid;
    }
    // scalar bounds: the record loop counts and addresses on the scalar unit
    t.c1 = __builtin_amdgcn_readfirstlane(t.c1);
    t.p0 = __builtin_amdgcn_readfirstlane(a);
    t.p1 = __builtin_amdgcn_readfirstlane(b);
    return t;
}

// Halves of two registers exchanged and added: lanes of the lower half (of
// 64, or of each 32) get a summed over both halves, lanes of the upper half b.
__device__ __forceinline__ float og_fold32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float og_fold16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// the same over the halves of each 16 lanes (upper: the lane's bit 3)
__device__ __forceinline__ float og_fold8(float a, float b, bool upper) {
    const float keep = upper ? b : a, send = upper ? a : b;
    return keep + og_dpp<0x128>(send);
}
// Sum over the wave, in the order of a butterfly over 1, 2, 4, 8, 16, 32.
template <int CTRL> __device__ __forceinline__ double og_dpp_add64(double v) {
    return v + __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                                __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double og_wave_sum64(double v) {
    v = og_dpp_add64<0xB1>(v);
    v = og_dpp_add64<0x4E>(v);
    v = og_dpp_add64<0x141>(v);  // the quads of a half row hold equal sums: mirroring is the exchange over 4
    v = og_dpp_add64<0x128>(v);
    double r[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        r[k] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 16 * k),
                                __builtin_amdgcn_readlane(__double2loint(v), 16 * k));
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// One energy of the cell (per-lane partial sums v, scaled) into its accumulator slot.
__device__ __forceinline__ void og_cell_energy(const og_dev_sys &s, const int c1, const int term, double v,
                                               const double scale) {
    v = og_wave_sum64(v);
    if ((threadIdx.x & 63) == 0)
        og_atomic_add_fx_g((OG_GLOBAL(long long) *)s.e_acc + (c1 % OG_EACC_SLOTS) * OG_EACC_STRIDE + term,
                           og_to_fixed(v * scale));
}

// One cell1 (one wave), its cell-pair records [p0, p1) (all of them, or
// half of them for a split cell).  ENERGY = false on steps whose energies
// are not logged: forces and the pair count only.  LJ_LDS: the cell1's LJ rows are in
// the block's LDS copy ljl of the table's leading rows.
template <int FORM, bool ENERGY, bool LJ_LDS>
__device__ __forceinline__ void og_pair_cell(const og_dev_sys &s, const og_unit &un, const og_f4 *__restrict__ shift,
                                             const typename og_ljt<FORM>::type *__restrict__ ljl, og_f4 *qp,
                                             int2 *qa) {
    const int c1 = un.c1, p0 = un.p0, p1 = un.p1;
    const int lane = threadIdx.x & 63;
    const int jl   = lane & 7;

    typedef typename og_ljt<FORM>::type ljt;
    const OG_GLOBAL(char) *__restrict__ X = (const OG_GLOBAL(char) *)s.gxyzq;
    const OG_GLOBAL(char) *__restrict__ TY = (const OG_GLOBAL(char) *)s.gtype;
    const OG_GLOBAL(ljt) *__restrict__ LJP =
        (const OG_GLOBAL(ljt) *)(FORM == 2 ? (const void *)s.lj_hps : (const void *)s.lj_pair);
    OG_GLOBAL(long long) *__restrict__ FX      = (OG_GLOBAL(long long) *)s.fx;
    const int cap = s.cap_atom_array;
    // j-side words of the gradient: packed (x, y) and z, per slot
    OG_GLOBAL(char) *FXJ = (OG_GLOBAL(char) *)(FX + OG_FX_XY(cap));
    OG_GLOBAL(char) *FXZ = (OG_GLOBAL(char) *)(FX + OG_FX_Z(cap));
    // keep-test radius: the cutoff plus 10 ppm, so float rounding of the box
    // distance can never drop a row that holds an in-range pair
    const float rcb2 = s.cutoff2 * 1.00001f;

    const og_list L{X, TY, (const OG_GLOBAL(char) *)s.cp_c2, (const OG_GLOBAL(char) *)s.cp_mask};
    // the first groups' records load with the cell1 atoms
    og_rec rec{0u, 0xffu}, rec1{0u, 0xffu};
    if (p0 < p1) {
        rec  = og_load_rec(L, p0, p1);
        rec1 = og_load_rec(L, p0 + OG_NAC, p1);
    }

    og_cell1 c;
    og_set_cell1<FORM>(s, un.p, un.ty, c);

    float  fi[3 * OG_NAC];
#pragma unroll
    for (int k = 0; k < 3 * OG_NAC; k++) fi[k] = 0.0f;
    double ev = 0.0, ee = 0.0, vir = 0.0;  // ev: -12 x the LJ energy except under HPS (scaled at the end)
    int    npair = 0;                    // in-cutoff unmasked pairs of this cell1 (wave-uniform)
    float  vmax = 0.0f, vsum = 0.0f;     // j-gradient range check
    int    qn = 0, qd = 0;               // rows queued / rows evaluated (wave-uniform)
    og_jpend pend{0.0f, 0.0f, 0.0f, 0, false};

    // Two groups in flight: the next group's atoms and the records after them
    // load while this group is filtered (and its full pass evaluated).
    og_jatom at{og_f4{0.0f, 0.0f, 0.0f, 0.0f}, 0u};
    if (p0 < p1) at = og_load_atom(L, rec.cp);
    for (int base = p0; base < p1; base += OG_NAC) {
        const og_jatom at1  = og_load_atom(L, rec1.cp);
        const og_rec   rec2 = og_load_rec(L, base + 2 * OG_NAC, p1);
        unsigned       m8   = rec.m8;
        if (p1 - base < OG_NAC) m8 = (lane >> 3) < p1 - base ? m8 : 0xffu;  // lanes past the last record
        const uint64_t ub = og_keep(c.lo, c.hi, rcb2, shift, rec.cp, m8, at.p);
        if (__builtin_amdgcn_inverse_ballot_w64(ub)) {
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(ub >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)ub, 0u));
            const int slot = (qn + rank) & (OG_QCAP - 1);
            const int a2   = (int)(rec.cp & 0xffffffu) * OG_NAC + jl;
            qp[slot]       = at.p;
            qa[slot]       = make_int2(a2, (int)(at.ty | (m8 << 24)));
        }
        qn += __builtin_popcountll(ub);
        if (qn - qd >= 64) {
            og_pass<FORM, ENERGY, LJ_LDS>(s, c, qp, qa, qd, 64, ljl, LJP, FXJ, FXZ, fi, npair, vmax, vsum, ev, ee, vir, pend);
            qd += 64;
        }
        rec  = rec1;
        rec1 = rec2;
        at   = at1;
    }
    if (qn > qd)
        og_pass<FORM, ENERGY, LJ_LDS>(s, c, qp, qa, qd, qn - qd, ljl, LJP, FXJ, FXZ, fi, npair, vmax, vsum, ev, ee, vir, pend);
    og_flush_j(FXJ, FXZ, pend);

    // i-gradients: reduce-scatter the 24 partial sums over the wave.  After
    // the folds over 32, 16 and 8 lane L holds atom L>>3's (x, y, z) summed over 8
    // lanes; an 8-lane butterfly completes the sum.
    float h12[12], h6[6], h3[3];
#pragma unroll
    for (int k = 0; k < 12; k++) h12[k] = og_fold32(fi[k], fi[12 + k]);
#pragma unroll
    for (int k = 0; k < 6; k++) h6[k] = og_fold16(h12[k], h12[6 + k]);
#pragma unroll
    for (int k = 0; k < 3; k++) h3[k] = og_dpp_sum8(og_fold8(h6[k], h6[3 + k], lane & 8));
    if (!(vmax <= OG_FXJ_ROW_LIMIT) || !(fabsf(vsum) < INFINITY)) atomicOr(&s.cnt->flags, OG_F_NAN);
    if (jl == 0) {
        const int a1 = c1 * OG_NAC + (lane >> 3);
        if (!(fabsf(h3[0]) + fabsf(h3[1]) + fabsf(h3[2]) <= (float)OG_FX_LIMIT)) atomicOr(&s.cnt->flags, OG_F_NAN);
        og_add_fx3(FX, cap, og_fx_slot(a1), (double)h3[0], (double)h3[1], (double)h3[2]);
    }
    if (!ENERGY) return;
    og_cell_energy(s, c1, OG_EACC_VDW, ev, FORM == 2 ? 1.0 : -1.0 / 12.0);
    og_cell_energy(s, c1, OG_EACC_ELE, ee, 1.0);
    og_cell_energy(s, c1, OG_EACC_VIR, vir, 1.0);
    if (lane == 0)
        og_atomic_add_fx_g((OG_GLOBAL(long long) *)s.e_acc + (c1 % OG_EACC_SLOTS) * OG_EACC_STRIDE + OG_EACC_PAIRS,
                           (long long)npair);
}

// The block's table of image shifts and its LDS copy of the leading rows of
// the LJ table (as many whole rows as fit in OG_LJ_LDS_ENTRIES; the engine
// numbers types by frequency, so for water the oxygen and hydrogen rows
// against every type); returns the rows held.  Every thread of the block.
template <int FORM, int THREADS>
__device__ __forceinline__ int og_pair_tables(const og_dev_sys &s, og_f4 *shift, typename og_ljt<FORM>::type *ljl) {
    typedef typename og_ljt<FORM>::type ljt;
    const int nt   = s.n_types;
    const int rows = min(nt, OG_LJ_LDS_ENTRIES(FORM) / nt);
    if (threadIdx.x < 64) {
        // image bits of MiniCell::add_cell_pair (MiniCell.cpp:1174-1187): neg bit -> -L, pos bit -> +L
        const unsigned img = threadIdx.x;
        const float    L0 = s.L[0], L1 = s.L[1], L2 = s.L[2];
        shift[img] = og_f4{(img & 1u) ? -L0 : ((img & 2u) ? L0 : 0.0f), (img & 4u) ? -L1 : ((img & 8u) ? L1 : 0.0f),
                           (img & 16u) ? -L2 : ((img & 32u) ? L2 : 0.0f), 0.0f};
    }
    const ljt *tab = (const ljt *)(FORM == 2 ? (const void *)s.lj_hps : (const void *)s.lj_pair);
    for (int k = threadIdx.x; k < rows * nt; k += THREADS) ljl[k] = tab[k];
    return rows;
}

// WAVES waves (one work unit each: a cell, or half of one of the last
// cells) per block.  The block size is a launch shape the autotuner chooses
// (results do not depend on it).  Five waves per SIMD: the kernel needs 99
// vector registers when left free (four waves), and holding it to 96 costs a
// few spills and gains 5% at 450,000 atoms (400 to 380 us with energies; the
// same at 99,200); the HPS form would spill more.
template <int FORM, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, FORM == 2 ? 4 : 5) k_pair(const og_dev_sys *__restrict__ S,
                                                                       const int2 *__restrict__ map) {
    typedef typename og_ljt<FORM>::type ljt;
    __shared__ og_f4 shift[64];              // image code -> shift of cell2
    __shared__ ljt   ljl[OG_LJ_LDS_ENTRIES(FORM)];
    __shared__ og_f4 qpos[WAVES][OG_QCAP];  // row queue: shifted x, y, z, charge
    __shared__ int2  qaux[WAVES][OG_QCAP];  // grid slot, LJ column | mask byte << 24
    const int2        bm = map ? map[blockIdx.x] : make_int2(0, (int)blockIdx.x);
    const og_dev_sys &s  = S[bm.x];
    const int         w  = threadIdx.x >> 6;
    const og_unit     un = og_unit_start(s, __builtin_amdgcn_readfirstlane(bm.y * WAVES + w));
    const int rows = og_pair_tables<FORM, 64 * WAVES>(s, shift, ljl);
    __syncthreads();
    if (!un.run) return;
    // a cell1 whose types are all in the block's LDS rows reads LJ pairs from LDS, otherwise from the global table
    if (un.energy) {
        if (__all(un.ty < rows)) og_pair_cell<FORM, true, true>(s, un, shift, ljl, qpos[w], qaux[w]);
        else og_pair_cell<FORM, true, false>(s, un, shift, ljl, qpos[w], qaux[w]);
    } else {
        if (__all(un.ty < rows)) og_pair_cell<FORM, false, true>(s, un, shift, ljl, qpos[w], qaux[w]);
        else og_pair_cell<FORM, false, false>(s, un, shift, ljl, qpos[w], qaux[w]);
    }
}

// ------------------------------------------------------ team of waves --
// The same work unit by a team of four waves (one block), for launches that do
// not fill the chip: a lone wave issues one VALU instruction per 8 cycles and
// waits out every load, and takes about 24 us for a unit (6,000 atoms: 784
// units on 1,024 SIMDs).
//  * filter: the waves take the groups of eight records in turn and queue
//    their rows at the positions the one-wave filter would give them (ballot
//    counts exchanged through LDS);
//  * rows: the waves evaluate four passes at a time, one each: the j-gradients go
//    out, the pairs' gradient coefficients and the rows' energies to LDS;
//  * i side: wave w then sums atoms 2 w and 2 w + 1 over those passes in pass
//    order, waves 0 to 2 one energy each.
// Every sum is taken over the same values in the same order as by one wave,
// so the results are the same bits.  (Dividing the atoms instead, each wave
// continuing the rows' sums of the one before it a pass behind, measured
// 24.4 us at 6,000 atoms against 25.6 for one wave: too many steps.)
// Kernel time, a wave per unit / a team: 3,000 atoms 23.7 / 18.2 us, 6,000
// 25.0 / 21.9.  What is left: four to six dependent memory round trips before
// the first pass (about 4 us), and per four passes one of 2,400 cycles and a
// sum of 1,300.
#define OG_TEAM 4                                  // waves
#define OG_TEAM_NI (OG_NAC / OG_TEAM)              // cell1 atoms per wave on the i side
#define OG_TEAM_NG 2                               // groups per wave and batch
#define OG_TEAM_G (OG_TEAM_NG * OG_TEAM)           // groups per batch (64 candidate rows each)
struct og_team {
    og_f4 qp[OG_TEAM_G * 64 + 64];                 // queue: one batch and a remainder
    int2  qa[OG_TEAM_G * 64 + 64];
    float coef[OG_TEAM][OG_NAC][64];               // by pass: gradient coefficients of the row's pairs
    float en[OG_TEAM][3][64];                      // by pass: the rows' LJ and electrostatic energy and virial
    int   cnt[2][OG_TEAM_G];                       // rows kept by each group of a batch, by batch parity
    int   run;                                     // the block's unit runs
    og_f4 shift[64];
};

// LDS written by the block's waves is visible after it (no wait for memory)
__device__ __forceinline__ void og_lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int FORM, bool ENERGY, bool LJ_LDS>
__device__ __forceinline__ void og_team_cell(const og_dev_sys &s, const og_unit &un, const int w, og_team &T,
                                             const typename og_ljt<FORM>::type *__restrict__ ljl) {
    typedef typename og_ljt<FORM>::type ljt;
    constexpr int NI = OG_TEAM_NI, NG = OG_TEAM_NG, G = OG_TEAM_G;
    const int     c1 = un.c1, p0 = un.p0, p1 = un.p1;
    const int     lane = threadIdx.x & 63, jl = lane & 7, i0 = w * NI;
    const OG_GLOBAL(ljt) *__restrict__ LJP =
        (const OG_GLOBAL(ljt) *)(FORM == 2 ? (const void *)s.lj_hps : (const void *)s.lj_pair);
    const og_list L{(const OG_GLOBAL(char) *)s.gxyzq, (const OG_GLOBAL(char) *)s.gtype,
                    (const OG_GLOBAL(char) *)s.cp_c2, (const OG_GLOBAL(char) *)s.cp_mask};
    OG_GLOBAL(long long) *FX = (OG_GLOBAL(long long) *)s.fx;
    const int   cap  = s.cap_atom_array;
    OG_GLOBAL(char) *FXJ = (OG_GLOBAL(char) *)(FX + OG_FX_XY(cap));
    OG_GLOBAL(char) *FXZ = (OG_GLOBAL(char) *)(FX + OG_FX_Z(cap));
    const float rcb2 = s.cutoff2 * 1.00001f;

    // this wave's groups of the first batch, and the records of the second
    og_rec   rec[NG], rec1[NG];
    og_jatom at[NG];
    if (p0 < p1) {
#pragma unroll
        for (int j = 0; j < NG; j++) {
            rec[j]  = og_load_rec(L, p0 + OG_NAC * (j * OG_TEAM + w), p1);
            rec1[j] = og_load_rec(L, p0 + OG_NAC * (G + j * OG_TEAM + w), p1);
        }
#pragma unroll
        for (int j = 0; j < NG; j++) at[j] = og_load_atom(L, rec[j].cp);
    }
    og_cell1 c;
    og_set_cell1<FORM>(s, un.p, un.ty, c);
    float xi[NI], yi[NI], zi[NI];  // the atoms this wave sums
#pragma unroll
    for (int i = 0; i < NI; i++) {
        xi[i] = og_vgpr(og_rlane(un.p.x, i0 + i));
        yi[i] = og_vgpr(og_rlane(un.p.y, i0 + i));
        zi[i] = og_vgpr(og_rlane(un.p.z, i0 + i));
    }

    float fi[3 * NI];
#pragma unroll
    for (int k = 0; k < 3 * NI; k++) fi[k] = 0.0f;
    double en = 0.0;  // waves 0, 1, 2: -12 x the LJ energy (except under HPS), electrostatic energy, virial
    int    npair = 0, qn = 0, parity = 0;
    float  vmax = 0.0f, vsum = 0.0f;
    for (int base = p0;;) {
        if (base < p1) {
            uint64_t ub[NG];
#pragma unroll
            for (int j = 0; j < NG; j++) {
                const int left = p1 - (base + OG_NAC * (j * OG_TEAM + w));  // records from the group's first to the end
                if (left < OG_NAC) rec[j].m8 = (lane >> 3) < left ? rec[j].m8 : 0xffu;
                ub[j] = og_keep(c.lo, c.hi, rcb2, T.shift, rec[j].cp, rec[j].m8, at[j].p);
                if (lane == 0) T.cnt[parity][j * OG_TEAM + w] = __builtin_popcountll(ub[j]);
            }
            og_lds_barrier();
            // running counts of the batch's groups (lanes 0 .. G - 1): row shifts by 1, 2, 4 lanes
            static_assert(G == 8, "one row of lanes, three shifts");
            int sum = T.cnt[parity][lane & (G - 1)];
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x111, 0xf, 0xf, true);
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x112, 0xf, 0xf, true);
            sum += __builtin_amdgcn_update_dpp(0, sum, 0x114, 0xf, 0xf, true);
#pragma unroll
            for (int j = 0; j < NG; j++) {
                const int at0 = qn + __builtin_amdgcn_readlane(sum, j * OG_TEAM + w) - __builtin_popcountll(ub[j]);
                if (__builtin_amdgcn_inverse_ballot_w64(ub[j])) {
                    const int slot = at0 + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(ub[j] >> 32),
                                                                          __builtin_amdgcn_mbcnt_lo((unsigned)ub[j], 0u));
                    T.qp[slot] = at[j].p;
                    T.qa[slot] = make_int2((int)(rec[j].cp & 0xffffffu) * OG_NAC + jl, (int)(at[j].ty | (rec[j].m8 << 24)));
                }
            }
            qn += __builtin_amdgcn_readlane(sum, G - 1);
            base += G * OG_NAC;
            parity ^= 1;
            // the next batch's atoms and the records after them load while this batch's passes run
#pragma unroll
            for (int j = 0; j < NG; j++) {
                rec[j]  = rec1[j];
                at[j]   = og_load_atom(L, rec[j].cp);
                rec1[j] = og_load_rec(L, base + OG_NAC * (G + j * OG_TEAM + w), p1);
            }
        }
        // a pass per wave at a time: wave w evaluates pass q + w, then sums its atoms over the passes in order
        const bool last = base >= p1;
        const int  np   = last ? (qn + 63) >> 6 : qn >> 6;
        for (int q = 0; q < np; q += OG_TEAM) {
            og_lds_barrier();  // the queue is written, the last passes' coefficients are read
            const int p = q + w;
            if (p < np) {
                const int  cnt  = min(qn - 64 * p, 64);
                const bool live = lane < cnt;
                og_f4      pj   = T.qp[64 * p + lane];
                const int2 ax   = T.qa[64 * p + lane];
                unsigned   m8 = (unsigned)ax.y >> 24, tj = (unsigned)ax.y & 0xffffffu;
                if (cnt < 64) {  // idle lanes: finite coordinates, LJ column 0, every pair masked
                    if (!live) pj = og_f4{0.0f, 0.0f, 0.0f, 0.0f};
                    m8 = live ? m8 : 0xffu;
                    tj = live ? tj : 0u;
                }
                float    g[OG_NAC];
                og_chain ch;
                og_rows<FORM, ENERGY, LJ_LDS, true>(s, c, pj, tj, m8, ljl, LJP, g, npair, ch);
#pragma unroll
                for (int i = 0; i < OG_NAC; i++) T.coef[w][i][lane] = g[i];
                if (ENERGY) T.en[w][0][lane] = ch.e, T.en[w][1][lane] = ch.q, T.en[w][2][lane] = ch.v;
                og_range(ch, vmax, vsum);
                og_jpend pend{ch.x, ch.y, ch.z, ax.x, live};
                og_flush_j(FXJ, FXZ, pend);
            }
            og_lds_barrier();
            // the passes' rows and coefficients load together; a pass past the last adds coefficient 0
            og_f4 pj[OG_TEAM];
            float g[OG_TEAM][NI];
#pragma unroll
            for (int k = 0; k < OG_TEAM; k++) {
                const bool in = lane < qn - 64 * (q + k) && q + k < np;
                pj[k] = T.qp[64 * min(q + k, np - 1) + lane];
                if (!in) pj[k] = og_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const float v = T.coef[k][i0 + i][lane];
                    g[k][i]       = in ? v : 0.0f;
                }
            }
#pragma unroll
            for (int k = 0; k < OG_TEAM; k++)
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    fi[3 * i]     = fmaf(g[k][i], xi[i] - pj[k].x, fi[3 * i]);
                    fi[3 * i + 1] = fmaf(g[k][i], yi[i] - pj[k].y, fi[3 * i + 1]);
                    fi[3 * i + 2] = fmaf(g[k][i], zi[i] - pj[k].z, fi[3 * i + 2]);
                }
            if (ENERGY && w < 3) {
                float e[OG_TEAM];
#pragma unroll
                for (int k = 0; k < OG_TEAM; k++) e[k] = T.en[k][w][lane];
#pragma unroll
                for (int k = 0; k < OG_TEAM; k++) en += q + k < np ? (double)e[k] : 0.0;
            }
        }
        if (last) break;
        // the rows short of a pass lead the next batch's queue (its rows are written after another barrier)
        const int rem = qn - 64 * np;
        if (np > 0) {
            og_lds_barrier();
            if (w == 0 && lane < rem) {
                const og_f4 mp = T.qp[64 * np + lane];
                const int2  ma = T.qa[64 * np + lane];
                T.qp[lane]     = mp;
                T.qa[lane]     = ma;
            }
        }
        qn = rem;
    }
    // i-gradients: sums over the wave in the order of the one-wave reduction, lanes 0-31 and 32-63 an atom each
    static_assert(NI == 2, "two atoms per wave");
    float h3[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        float v = og_fold32(fi[k], fi[3 + k]);
        v       = og_fold16(v, v);
        h3[k]   = og_dpp_sum8(v + og_dpp<0x128>(v));
    }
    if (!(vmax <= OG_FXJ_ROW_LIMIT) || !(fabsf(vsum) < INFINITY)) atomicOr(&s.cnt->flags, OG_F_NAN);
    if ((lane & 31) == 0) {
        const int a1 = c1 * OG_NAC + i0 + (lane >> 5);
        if (!(fabsf(h3[0]) + fabsf(h3[1]) + fabsf(h3[2]) <= (float)OG_FX_LIMIT)) atomicOr(&s.cnt->flags, OG_F_NAN);
        og_add_fx3(FX, cap, og_fx_slot(a1), (double)h3[0], (double)h3[1], (double)h3[2]);
    }
    if (!ENERGY) return;
    if (w < 3) og_cell_energy(s, c1, OG_EACC_VDW + w, en, w == 0 && FORM != 2 ? -1.0 / 12.0 : 1.0);
    if (lane == 0)
        og_atomic_add_fx_g((OG_GLOBAL(long long) *)s.e_acc + (c1 % OG_EACC_SLOTS) * OG_EACC_STRIDE + OG_EACC_PAIRS,
                           (long long)npair);
}

// One work unit per block; the map lists units (one per block).
template <int FORM>
__global__ void __launch_bounds__(64 * OG_TEAM) k_pair_team(const og_dev_sys *__restrict__ S,
                                                           const int2 *__restrict__ map) {
    typedef typename og_ljt<FORM>::type ljt;
    __shared__ og_team T;
    __shared__ ljt     ljl[OG_LJ_LDS_ENTRIES(FORM)];
    const int2        bm = map ? map[blockIdx.x] : make_int2(0, (int)blockIdx.x);
    const og_dev_sys &s  = S[bm.x];
    const og_unit     un = og_unit_start(s, bm.y);
    const int rows = og_pair_tables<FORM, 64 * OG_TEAM>(s, T.shift, ljl);
    // One wave decides for the block: if another block flags an overlap between two waves' reads of the
    // flags, waves that left would leave queue entries unwritten that the others go on to read.
    if (threadIdx.x == 0) T.run = un.run;
    og_lds_barrier();
    if (!__builtin_amdgcn_readfirstlane(T.run)) return;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (un.energy) {
        if (__all(un.ty < rows)) og_team_cell<FORM, true, true>(s, un, w, T, ljl);
        else og_team_cell<FORM, true, false>(s, un, w, T, ljl);
    } else {
        if (__all(un.ty < rows)) og_team_cell<FORM, false, true>(s, un, w, T, ljl);
        else og_team_cell<FORM, false, false>(s, un, w, T, ljl);
    }
}

// Per atom: fixed-point pair gradient -> FP64 "work" with the atom's
// excluded-pair and bond terms (og_atom_work).
__global__ void __launch_bounds__(OG_THREADS) k_forces_to_work(const og_dev_sys *__restrict__ S,
                                                               const int2 *__restrict__ map) {
    const int2        bm = map[blockIdx.x];
    const og_dev_sys &s  = S[bm.x];
    if (og_frozen(s)) return;
    const int i    = bm.y * OG_THREADS + threadIdx.x;
    double    e_ex = 0.0, e_b = 0.0;
    if (i < s.n_atoms) og_atom_work(s, i, e_ex, e_b);
    if (!og_energy_step(s)) return;
    __shared__ double sh[2 * (OG_THREADS / 64)];
    og_add_misc_energies(s, bm.y, e_ex, e_b, sh);
}

// Energies of a call point's evaluation from the fixed-point accumulators
// (an MD step takes them in k_step_close).
__global__ void __launch_bounds__(64) k_energy_reduce(const og_dev_sys *__restrict__ S,
                                                      const int2 *__restrict__ map) {
    const og_dev_sys &s = S[map[blockIdx.x].x];
    if (og_frozen(s) || !og_energy_step(s)) return;
    __shared__ long long sh[16 * OG_EACC_STRIDE];
    og_take_pair_energies<64>(s, sh);
}

// A single-point evaluation of one system.  Its requests (energies, and a
// grid rebuild) go into the counters in the rebuild's first kernel, or without
// one in k_point_begin; the last kernel is k_forces_to_work with its outcome
// sent to pinned host memory: the gradient when work is given, and from the
// last block the counters and the energies.  One wait for the stream then
// delivers what took six copies with a wait each (4,230 atoms: 208 us per
// call, then 116; launches of their own for the requests and the reduction
// were 7 and 5 us of it).
__global__ void k_point_begin(og_dev_counters *c) { og_request_point(c, 0); }
__global__ void __launch_bounds__(OG_THREADS) k_point_end(const og_dev_sys *__restrict__ S,
                                                          og_point_out *__restrict__ out,
                                                          double *__restrict__ work) {
    const og_dev_sys &s      = S[0];
    const bool        run    = !og_frozen(s);
    const bool        energy = run && og_energy_step(s);
    const int         i0     = blockIdx.x * OG_THREADS, i = i0 + threadIdx.x;
    double            e_ex = 0.0, e_b = 0.0, w[3] = {0.0, 0.0, 0.0};
    if (i < s.n_atoms) {
        if (run) {
            og_atom_work_calc(s, i, w, e_ex, e_b);
            og_atom_work_store(s, i, w);
        } else {  // a system that stands still returns the gradient it has
            for (int k = 0; k < 3; k++) w[k] = s.work[3 * i + k];
        }
    }
    if (work) {  // whole lines to the host
        __shared__ double wl[3 * OG_THREADS];
        for (int k = 0; k < 3; k++) wl[3 * threadIdx.x + k] = w[k];
        __syncthreads();
        const int n = 3 * min(OG_THREADS, s.n_atoms - i0);
        for (int k = threadIdx.x; k < n; k += OG_THREADS) work[3 * (size_t)i0 + k] = wl[k];
    }
    if (energy) {
        __shared__ double sh[2 * (OG_THREADS / 64)];
        og_add_misc_energies(s, blockIdx.x, e_ex, e_b, sh);
    }
    if (!og_last_block(&s.sync->all, gridDim.x)) return;
    if (energy) {
        __shared__ long long sh[16 * OG_EACC_STRIDE];
        og_take_pair_energies<OG_THREADS>(s, sh);
    }
    if (threadIdx.x < OG_E_NTERMS) out->energy[threadIdx.x] = s.energy[threadIdx.x];
    if (threadIdx.x) return;
    s.cnt->rebuild_now  = 0;
    s.cnt->force_energy = 0;
    out->cnt            = *s.cnt;
}

// ------------------------------------------------------------- launchers --
template <int FORM>
static void og_launch_pair_form(const og_launch &a, int waves) {
    switch (waves) {
    case 1: hipLaunchKernelGGL((k_pair<FORM, 1>), dim3(a.n_blocks), dim3(64), 0, a.stream, a.sys, a.map); break;
    case 2: hipLaunchKernelGGL((k_pair<FORM, 2>), dim3(a.n_blocks), dim3(128), 0, a.stream, a.sys, a.map); break;
    case 8: hipLaunchKernelGGL((k_pair<FORM, 8>), dim3(a.n_blocks), dim3(512), 0, a.stream, a.sys, a.map); break;
    default: hipLaunchKernelGGL((k_pair<FORM, 4>), dim3(a.n_blocks), dim3(256), 0, a.stream, a.sys, a.map); break;
    }
}

void og_launch_pair(const og_launch &a, int form, int waves) {
    switch (form) {
    case OG_FORM_HPS_DH: og_launch_pair_form<2>(a, waves); break;
    case OG_FORM_ZM: og_launch_pair_form<3>(a, waves); break;
    case OG_FORM_ZM_ALPHA: og_launch_pair_form<4>(a, waves); break;
    case OG_FORM_ZD_ALPHA: og_launch_pair_form<1>(a, waves); break;
    default: og_launch_pair_form<0>(a, waves); break;
    }
}

template <int FORM>
static void og_launch_team_form(const og_launch &a) {
    hipLaunchKernelGGL((k_pair_team<FORM>), dim3(a.n_blocks), dim3(64 * OG_TEAM), 0, a.stream, a.sys, a.map);
}
void og_launch_pair_team(const og_launch &a, int form) {
    switch (form) {
    case OG_FORM_HPS_DH: og_launch_team_form<2>(a); break;
    case OG_FORM_ZM: og_launch_team_form<3>(a); break;
    case OG_FORM_ZM_ALPHA: og_launch_team_form<4>(a); break;
    case OG_FORM_ZD_ALPHA: og_launch_team_form<1>(a); break;
    default: og_launch_team_form<0>(a); break;
    }
}
void og_launch_forces_to_work(const og_launch &a) {
    hipLaunchKernelGGL(k_forces_to_work, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, a.map);
}
void og_launch_energy_reduce(const og_launch &a) {
    hipLaunchKernelGGL(k_energy_reduce, dim3(a.n_blocks), dim3(64), 0, a.stream, a.sys, a.map);
}
void og_launch_point_begin(og_dev_counters *cnt, hipStream_t st) {
    hipLaunchKernelGGL(k_point_begin, dim3(1), dim3(1), 0, st, cnt);
}
void og_launch_point_end(const og_launch &a, og_point_out *out, double *work) {
    hipLaunchKernelGGL(k_point_end, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, out, work);
}
