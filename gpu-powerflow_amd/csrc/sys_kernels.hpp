// Launchers of the one-workgroup-per-system kernels (sys_kernels.hip; plan:
// sys_plan.hpp).  Arrays are scenario-interleaved (x[i * Bp + b]); a launch
// covers the B real scenarios only.
#pragma once

#include "kernels.hpp"
#include "sys_plan.hpp"

namespace cupf::kern {

struct SysDevice {
    int n = 0, nnz = 0;
    int fac = 0, scratch = 0;
    int blob_quads = 0;               // int4s of the blob
    int num_levels = 0;
    int o_level = 0, o_slice = 0, o_task = 0, o_rows = 0, o_gptr = 0, o_gsrc = 0, o_perm = 0;
    const int4* blob = nullptr;
    const unsigned short* adds = nullptr;
    const int* slot_pos = nullptr;    // [nnz]
    const int* gate = nullptr;        // see LuDevice::gate
};

// Network tables of the fused Newton step.
struct SysNet {
    const int4* ydst = nullptr;             // [nnzY] factor elements of an entry's J11, J21, J12, J22 (-1: none)
    const int* yrow = nullptr;              // [nnzY] Ybus row
};

constexpr size_t kSysLdsMax = 159 * 1024;
// LDS bytes of the factor / solve kernels and of the fused Newton step
// (n_bus > 0) for front elements of `elem` bytes.
size_t sys_lds_bytes(const SysPlan& p, int elem, int n_bus);
// Elements of one scenario's stored factors (factors, then the pivots'
// reciprocals).
inline size_t sys_store_elems(const SysPlan& p) { return size_t(p.fac) + size_t(p.n); }
// Raises the kernels' LDS limits; once per process and device, before a launch
// that is captured.
void sys_prepare();

// Factors A [nnz][Bp] of scenarios 0..B-1 into store [B][sys_store_elems].
template <typename T>
void sys_factor(const SysDevice& d, const double* A, int B, int Bp, T* store, double pivot_eps,
                int static_piv, int* sing, size_t lds, hipStream_t s);
// x = A^-1 rhs (or A^-T rhs) from the stored factors.
template <typename T, typename TX>
void sys_solve(const SysDevice& d, const T* store, const double* rhs, int B, int Bp, TX* x,
               bool transpose, size_t lds, hipStream_t s);

// Newton loop on the state V / Va / Vm, one workgroup per scenario.  A launch
//  first:  evaluates the residual norms and starts the control word
//          (nr_control's layout); with seed it takes Va, Vm from V before;
//  steps:  then up to `steps` Newton steps (Jacobian, factors, solve,
//          `refine` FP64 refinement solves where the control word asks for
//          them, voltage update, residual norms, control word); more than one
//          only with one scenario.  A launch on a stopped word does nothing.
//  finish: one step on an unstopped or limit-stopped word without the
//          evaluation that follows it.
// normF[b], bmax[0] and ctl are left as the batched kernels leave them; sync2
// is two zeroed words of scratch that the launch leaves zeroed.
struct SysNewton {
    bool first = false, seed = false, finish = false, tolerant = false;
    int steps = 0, refine = 0, limit = 0;
    double tol = 0.0, refine_below = 0.0;
};
template <typename T>
void sys_newton(const SysDevice& d, const NrDevice& nr, const SysNet& net, const SysNewton& o,
                const double2* S, double2* V, double* Va, double* Vm, double* normF, double* bmax,
                int* ctl, unsigned long long* sync2, int B, int Bp, double pivot_eps,
                int static_piv, int* sing, size_t lds, hipStream_t s);

}  // namespace cupf::kern
