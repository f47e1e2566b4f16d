// The device code of libqrdm_amd.so as one translation unit: the kernels of
// panel.hip combine stages defined in kernels.hip (one launch runs several
// steps of a DM iteration); regpanel.hip holds the column-by-column panel,
// mixed.hip adds the reduced-precision trailing update, learned.hip the
// (tau, delta) network, trailing.hip the DM loop's trailing update merged into
// one pass over C per step, batched.hip the persistent many-matrix kernel,
// wide.hip the DM steps wider than 64 columns.
#include "kernels.hip"
#include "panel.hip"
#include "regpanel.hip"
#include "mixed.hip"
#include "learned.hip"
#include "trailing.hip"
#include "batched.hip"
#include "wide.hip"
