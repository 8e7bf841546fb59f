// plain_device.hpp -- the per-atom pieces of the FP64 form, shared by the
// kernels of the single calls (plain.hip) and of the whole step
// (plain_step.hip), so that both give the same bits.
#pragma once

#include "dsmc_device.hpp"
#include "plain.hpp"

namespace dsmc {

// Pair (offsets in the cell) and acceptance uniform of trial tr of a cell of n
// atoms (collisions.cu:400-425).
__device__ __forceinline__ void plain_trial(const CollideParams &cp, uint32_t stream, uint32_t cell,
                                            uint32_t step, int tr, int n, int &i, int &j, double &u_acc)
{
    i = 0; j = 1;
    if (cp.pair_mode == 0) {
        const U32x4 o = draw(cp.seed, stream, cell, step, (uint32_t)tr, kPurposeCollide, 0);
        i = (int)uint_below(o.x, (uint32_t)n);
        j = (int)uint_below(o.y, (uint32_t)(n - 1));
        j += (j >= i);
        u_acc = u01(o.z, o.w);
    } else {
        if (n > 2) {
            i = 0; j = 0;
            for (uint32_t k = 0; k < 64 && i == j; ++k) {
                const U32x4 o = draw(cp.seed, stream, cell, step, (uint32_t)tr, kPurposeCollide, 16 + k);
                i = (int)floor(u01(o.x, o.y) * (n - 1));
                j = (int)floor(u01(o.z, o.w) * (n - 1));
            }
            if (i == j) { i = 0; j = 1; }
        }
        const U32x4 o = draw(cp.seed, stream, cell, step, (uint32_t)tr, kPurposeCollide, 1);
        u_acc = u01(o.x, o.y);
    }
}

// Trials of a cell of n atoms (collisions.cu:318-322; the reference pair mode
// keeps the truncation of Mc * lambda).
__device__ __forceinline__ int plain_trials(const TrapDev &t, const CollideParams &cp, int n, double smax,
                                            double &lambda)
{
    const double Mc = 0.5 * (n - 1) * n;
    const double X = Mc * t.alpha * cp.lpc * cp.dt * smax / t.cell_vol;
    lambda = ceil(X) / Mc;
    return cp.pair_mode ? (int)(Mc * lambda) : (int)ceil(X);
}

// The pair's velocities after an accepted trial (collisions.cu:426-436).
__device__ __forceinline__ void plain_scatter(const TrapDev &t, const CollideParams &cp, uint32_t cell,
                                              uint32_t step, int tr, double magVrel, D3 &va, D3 &vb)
{
    const double cx = 0.5 * (va.x + vb.x), cy = 0.5 * (va.y + vb.y), cz = 0.5 * (va.z + vb.z);
    double nx, ny, nz;
    sphere_point(cp.seed, t.stream, cell, step, (uint32_t)tr, kPurposeCollide, 2, nx, ny, nz);
    const double wx = magVrel * nx, wy = magVrel * ny, wz = magVrel * nz;
    va = D3{ cx - 0.5 * wx, cy - 0.5 * wy, cz - 0.5 * wz };
    vb = D3{ cx + 0.5 * wx, cy + 0.5 * wy, cz + 0.5 * wz };
}

// Spinor components (psiUp re, im, psiDn re, im).
struct Spinor { double ur, ui, dr, di; };

// evolveWavefunction (wavefunction.cu:11-73) over one motion step.
__device__ __forceinline__ void plain_spin(const TrapDev &t, const SpinParams &sp, const D3 &p, const D3 &v,
                                           const D3 &a, Spinor &s)
{
    double hx = 0.0, hy = 0.0, hz = 0.0;
    if (sp.interp) {  // half-kicked velocity of the coming Verlet step
        hx = v.x + (0.5 * a.x) * sp.dt;
        hy = v.y + (0.5 * a.y) * sp.dt;
        hz = v.z + (0.5 * a.z) * sp.dt;
    }
    for (int m = 0; m < sp.substeps; ++m) {
        double x = p.x, y = p.y, z = p.z;
        if (sp.interp) {
            const double tau = (m + 0.5) * sp.dt_spin;
            x = p.x + hx * tau; y = p.y + hy * tau; z = p.z + hz * tau;
        }
        D3 Bn;
        const double B = field_dir(t, x, y, z, Bn);
        const double theta = 0.5 * sp.gs * kMuB * B * sp.dt_spin / kHbar;
        const double sn = sin(theta), cs = cos(theta);
        const double nur = s.ur * cs + (Bn.x * s.di - Bn.y * s.dr + Bn.z * s.ui) * sn;
        const double nui = s.ui * cs + ((-Bn.x) * s.dr - Bn.y * s.di - Bn.z * s.ur) * sn;
        const double ndr = s.dr * cs + (Bn.x * s.ui + Bn.y * s.ur - Bn.z * s.di) * sn;
        const double ndi = s.di * cs + ((-Bn.x) * s.ur + Bn.y * s.ui + Bn.z * s.dr) * sn;
        s.ur = nur; s.ui = nui; s.dr = ndr; s.di = ndi;
    }
}

// normalise (wavefunction.cu:279-299).
__device__ __forceinline__ void plain_normalise(Spinor &s)
{
    const double N = sqrt(s.ur * s.ur + s.ui * s.ui + s.dr * s.dr + s.di * s.di);
    s.ur = s.ur / N; s.ui = s.ui / N; s.dr = s.dr / N; s.di = s.di / N;
}

// moveAtoms (moveAtoms.cu:23-91): velocity Verlet; a: the acceleration at p,
// then at the new position.
__device__ __forceinline__ void plain_verlet(const TrapDev &t, double dt, bool up, D3 &p, D3 &v, D3 &a)
{
    v.x = v.x + (0.5 * a.x) * dt; v.y = v.y + (0.5 * a.y) * dt; v.z = v.z + (0.5 * a.z) * dt;
    p.x = p.x + v.x * dt; p.y = p.y + v.y * dt; p.z = p.z + v.z * dt;
    if (t.periodic) {
        p.x = wrap_periodic(p.x, t.hw[0]); p.y = wrap_periodic(p.y, t.hw[1]); p.z = wrap_periodic(p.z, t.hw[2]);
    }
    a = accel(t, p.x, p.y, p.z, up);
    v.x = v.x + (0.5 * a.x) * dt; v.y = v.y + (0.5 * a.y) * dt; v.z = v.z + (0.5 * a.z) * dt;
}

// evaporationTag (evaporation.cu:68-106) plus the energy cut; E: the atom's
// energy.
__device__ __forceinline__ bool plain_lost(const TrapDev &t, double mass, bool spin_loss, double e_cut,
                                           const D3 &p, const D3 &v, const Spinor &s, double &E)
{
    E = 0.5 * mass * (v.x * v.x + v.y * v.y + v.z * v.z) + potential_energy(t, p.x, p.y, p.z);
    bool lost = false;
    if (spin_loss) {
        D3 Bn;
        (void)field_dir(t, p.x, p.y, p.z, Bn);
        const double proj = 2. * Bn.x * (s.ur * s.dr + s.ui * s.di) + 2. * Bn.y * (s.ur * s.di - s.ui * s.dr) +
                            2. * Bn.z * (s.ur * s.ur + s.ui * s.ui - 0.5);
        lost = proj < 0.0;
    }
    if (e_cut > 0.0) lost = lost || E > e_cut;
    return lost;
}

// ---------------------------------------------------------------------------
// Majorana spin-flip model (wavefunction.cu:75-237): local populations before
// the motion substeps of a collision step, flips and decoherence after them.
// Populations are kept per atom label (the reference indexes them by atomID).
// ---------------------------------------------------------------------------
// projectLocalPopulations (wavefunction.cu:156-173): populations of the
// spinor in the spin-up and spin-down states of the local field axis.
__device__ __forceinline__ void local_pops(const TrapDev &t, const D3 &p, const Spinor &s, double &pu, double &pd)
{
    D3 Bn;
    (void)field_dir(t, p.x, p.y, p.z, Bn);
    const double re = s.ur * s.dr + s.ui * s.di, im = s.ui * s.dr - s.ur * s.di;
    const double w = 0.5 - s.ur * s.ur - s.ui * s.ui;
    pu = 0.5 + Bn.x * re - Bn.y * im - Bn.z * w;
    pd = 0.5 - Bn.x * re + Bn.y * im + Bn.z * w;
}

// flipAtoms (wavefunction.cu:99-154): an atom changes spin state with the
// probability that its population moved into the other state since the
// populations (opu, opd) were taken, if its kinetic energy can pay the
// potential step 2 mu |B| (gs muB |B| for the reference's mu); the speed then
// absorbs the step along the old direction.  The uniform is Philox (label,
// step, 0, purpose 3).  Returns whether it flipped.
__device__ __forceinline__ bool plain_flip(const TrapDev &t, const FlipParams &fp, uint32_t id, double opu,
                                           double opd, const D3 &p, const Spinor &s, D3 &v, bool &up)
{
    double npu, npd;
    local_pops(t, p, s, npu, npd);
    D3 Bn;
    const double magB = field_dir(t, p.x, p.y, p.z, Bn);
    double Pflip, dEp;
    if (up) {
        Pflip = (npd - opd) / opu;
        dEp = fp.gap * magB;
    } else {
        Pflip = (npu - opu) / opd;
        dEp = (-1.0 * fp.gap) * magB;
    }
    const double Ek = 0.5 * fp.mass * (v.x * v.x + v.y * v.y + v.z * v.z);
    const U32x4 o = draw(fp.seed, t.stream, id, fp.step, 0u, kPurposeFlip, 0u);
    if (!(Pflip > u01(o.x, o.y) && Ek + dEp > 0.0)) return false;
    up = !up;
    const double magVel = sqrt(v.x * v.x + v.y * v.y + v.z * v.z);
    const double speed = sqrt(2.0 * (Ek + dEp) / fp.mass);
    if (magVel > 0.0) v = D3{ speed * (v.x / magVel), speed * (v.y / magVel), speed * (v.z / magVel) };
    else v = D3{ 0.0, 0.0, speed };   // no direction to keep: along +z
    return true;
}

// calculateTau (wavefunction.cu:206-219) with getAcc (:221-237), the spin-up
// acceleration: the decoherence time from the position- and velocity-limited
// times of an atom that the field gradient separates.
__device__ __forceinline__ double decoherence_tau(const TrapDev &t, double sigma, double mass,
                                                  double x, double y, double z)
{
    const D3 a = accel(t, x, y, z, true);
    const double relAccel = 2.0 * sqrt(a.x * a.x + a.y * a.y + a.z * a.z);
    const double tauPos = 1.163 * sqrt(sigma / relAccel);
    const double tauVel = sqrt(2. / kPiRef) * kHbar / (mass * sigma * relAccel);
    return pow(1 / (tauPos * tauPos * tauPos) + 1 / (tauVel * tauVel * tauVel), -1. / 3.);
}

// exponentialDecay (wavefunction.cu:175-204): psi <- P+ psi + e P- psi with
// P+- = (1 +- B.sigma) / 2 and e = exp(-dt / tau), written out per component.
__device__ __forceinline__ void plain_decay(const TrapDev &t, const DecayParams &dp, const D3 &p, Spinor &s)
{
    D3 Bn;
    (void)field_dir(t, p.x, p.y, p.z, Bn);
    const double tau = decoherence_tau(t, dp.sigma, dp.mass, p.x, p.y, p.z);
    const double om = 1. - exp(-dp.dt / tau);
    const double op = 1. + exp(-dp.dt / tau);
    const Spinor q = s;
    s.ur = 0.5 * ((Bn.x * q.dr + Bn.y * q.di + Bn.z * q.ur) * om + q.ur * op);
    s.ui = 0.5 * ((Bn.x * q.di - Bn.y * q.dr + Bn.z * q.ui) * om + q.ui * op);
    s.dr = 0.5 * ((Bn.x * q.ur - Bn.y * q.ui - Bn.z * q.dr) * om + q.dr * op);
    s.di = 0.5 * ((Bn.x * q.ui + Bn.y * q.ur - Bn.z * q.di) * om + q.di * op);
}

}  // namespace dsmc
