// line1d.h -- arguments and launchers of the 1-D kernels that run whole RK4 steps (line1d.hip).
#pragma once
#include "mgd_internal.h"

namespace mgd {

constexpr int kLineSteps = 4;                 // most time steps of one launch
constexpr int kLineStages = 4 * kLineSteps;

// Forward stages of whole RK4 steps from the state at `in`: stages 1, 2, .. in order, the last
// one of the launch the last of a step unless no state follows it.
struct LineForward {
  const double* in;
  double* out;                   // the state after the last stage, or null
  int nstages;                   // 1 .. kLineStages
  double dt;
  const double* control;         // actuator forcing of the first stage; the next ones na apart
  long control_stride;           // .. and instances this far
  int na;
  const Source* src;
  const double* src_amp;         // amplitudes of the first stage; the next ones nsrc apart
  long src_inst_stride;
  int nsrc;
  double* keep[kLineStages];     // where the stage's output goes, or null
  double* keep2[kLineSteps];     // second place of a step's last output, or null
  double* jpartial;              // [inst][slot][cost-patch point] functional terms, or null
  int npts, nslots, slot;        // slot: of the first stage
  int ip_cost, ip_act;
};

// Adjoint stages of whole RK4 steps, backwards: stages 4, 3, 2, 1 of step t1, then of t1 - 1 ..
struct LineAdjoint {
  const double* in;
  double* out;
  int nstages;                   // a multiple of 4, at most kLineStages
  int t1;
  double dt;
  const double* q[kLineStages];  // the forward state of each stage, in the order of use
  double* grad;                  // gradient entries of the first stage here (the later ones na
  long grad_stride;              // before each other), or null
  int na;
  double* spartial;              // [inst][slot][actuator point] sensitivity terms, or null
  int npts, nslots, slot;        // slot: of the first stage here; the later ones count down
  int ip_cost, ip_act;
};

// Time steps that one launch takes on this grid (1 .. kLineSteps).
int line_steps(const Geo& g);
void launch_line_forward(const Geo& g, const Patches* P, const LineForward& a, hipStream_t st);
void launch_line_adjoint(const Geo& g, const Patches* P, const LineAdjoint& a, hipStream_t st);

}  // namespace mgd
