// Host-side objects of the learned warm start: relaxation sample buffers and
// the network (device parameters, optimiser state, BF16 inference fragments).
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "../../include/ecogen_amd.h"
#include "ecg_mlp.hpp"

struct ecg_samples {
  float* buf = nullptr;                 // cap * SAMPLE_FLOATS on the device
  unsigned long long* seen = nullptr;   // device counter of candidate cells
  long long cap = 0;
  int stride = 1;                       // of the current attachment
  long long base = 0;                   // records held before the current attachment
  long long uploaded = -1;              // record count set by ecg_samples_upload (-1: from the counter)
  int attached = 0;                     // solver contexts writing into it (ecg_attach_samples)
};

struct ecg_mlp {
  float* prm = nullptr;       // FP32 master parameters (MLP_NPARAM)
  float* adam_m = nullptr;
  float* adam_v = nullptr;
  float* grad = nullptr;      // reduced gradient
  float* act = nullptr;       // activations of a batch segment, act_ld chunks wide
  int act_ld = 0;
  double* loss_acc = nullptr; // per-epoch loss sums (loss_cap of them) and a batch's running sum
  int loss_cap = 0;
  uint2* frag = nullptr;      // BF16 A fragments (MLP_NFRAG * 64)
  float* bias = nullptr;      // FP32 biases (MLP_NBIAS)
  long long adam_t = 0;
  hipStream_t stream = nullptr;
  mutable int attached = 0;   // solver contexts whose step kernels read frag / bias (ecg_set_warm_start)
};

// Attachment counts: an attached object is not freed, and the network's
// parameters are rewritten only after the device has finished the work queued
// by the contexts that read them.
inline void mlp_attach(const ecg_mlp* m) { m->attached++; }
inline void mlp_detach(const ecg_mlp* m) { m->attached--; }
inline void samples_attach(ecg_samples* s) { s->attached++; }
inline void samples_detach(ecg_samples* s) { s->attached--; }

namespace ecg {
int api_fail(int code, const std::string& msg);
// Number of records a sample buffer holds (synchronises the device).
long long samples_count(ecg_samples* s);
}  // namespace ecg
