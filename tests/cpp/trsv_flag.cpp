// Sets the time-out flag that a preconditioner's transposed upper solve leaves
// for the host, as a wait that ran out of time does, so that a test can see who
// reports it. Built by __graft_entry__.build() for tests/test_gpu_timeout.py.
#include "device.hpp"

struct la_prec_s {  // as in capi.cpp
  std::unique_ptr<laamd::Prec> p;
};

// 0: the transposed plan does not exist yet
extern "C" int flag_transposed_timeout(la_prec_s *P) {
  laamd::TrsvPlan *T = P->p->upper->transposed.get();
  if (!T || !T->err_host) return 0;
  *T->err_host = 1;
  return 1;
}
