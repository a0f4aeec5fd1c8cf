// The FP64 integrator's Thomas solve on the host, for test_thomas.py.
#include "sc_thomas.h"

extern "C" {

// Solves `rows` rows in place (rows[2 * i], rows[2 * i + 1]: diagonal and
// right-hand side); with `fast` 1, whether the shared quotients served.
int thomas(int fast, int n, double *rows, const double *off) {
  double2 *row = reinterpret_cast<double2 *>(rows);
  return fast ? sc::thomas_chain<true>(n, row, off) : sc::thomas_chain<false>(n, row, off);
}

int frictions(double gpar, double gperp) { return sc::shared_frictions(gpar, gperp); }

}  // extern "C"
