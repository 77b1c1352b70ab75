// Forces behind the pair kernel: the slot-ordered pair sums added to the atoms,
// and the terms of fixed particles (exceptions, harmonic bonds and angles).
#pragma once

#include "nlist.h"

namespace ommhip {

enum TermKind : int { TERM_NONE = 0, TERM_EXCEPTION = 1, TERM_BOND = 2, TERM_ANGLE = 3 };

// One term: its kind and its particles' places in the tile's atom list, and its
// parameters (qq, sigma, epsilon; length, k; theta0, k).
struct Term {
    double p[3];
    int kind_atoms;  // kind << 24 | third << 16 | second << 8 | first
    int pad;
};

// The terms, in tiles of TERM_THREADS places and at most TERM_THREADS distinct
// atoms of one system.  A tile's wave holds terms of one kind.
constexpr int TERM_THREADS = 256;
struct TermTiles {
    int ntiles = 0;
    DevBuf<Term> terms;   // [ntiles][TERM_THREADS]
    DevBuf<int> atoms;    // [ntiles][TERM_THREADS], -1 padded
    DevBuf<int> sys;      // [ntiles]
    DevBuf<double> c6;    // LJPME: exception particles' C6, by place (else empty)
    // Host side: the terms as laid out, and the place of each exception.
    std::vector<Term> host;
    std::vector<int> place;

    // Global particle indices; theta0 and k of angle a are ap[2a], ap[2a + 1]
    // (bonds likewise).  set_exceptions, called next, gives the exceptions their
    // parameters and takes the terms to the device.
    void build(const std::vector<int>& e1, const std::vector<int>& e2, const std::vector<int>& b1,
               const std::vector<int>& b2, const std::vector<double>& bp, const std::vector<int>& a1,
               const std::vector<int>& a2, const std::vector<int>& a3, const std::vector<double>& ap,
               const std::vector<int>& atom_sys, hipStream_t s);
    void set_exceptions(const std::vector<double>& qq, const std::vector<double>& sig, const std::vector<double>& eps,
                        const std::vector<double>& c6_by_exception, hipStream_t s);
};

struct TermParams {
    int use_pbc = 0;         // exceptions: minimum image
    int screened = 0;        // exceptions: the reciprocal space's erf correction
    double alpha = 0.0, lj_alpha = 0.0;
};

// slots: add nl's slot-ordered pair sums into the forces and clear them;
// order_a/order_b (nullable, nl.nslots ints each) then receive the slot order.
// terms (nullable): evaluate them, energies (nullable) to E_EXCEPT, E_BOND and
// E_ANGLE of each system's E_SLOTS block.
void launch_fold(bool mixed, const NlistDev& nl, bool slots, const TermTiles* terms, const TermParams& prm,
                 const double* charge, const double* pos, const SysInfo* sys_dev, long long* force_fx, double* force_d,
                 long long* energy_fx, double* energy_d, unsigned* status, hipStream_t s, int* order_a = nullptr,
                 int* order_b = nullptr);

}  // namespace ommhip
