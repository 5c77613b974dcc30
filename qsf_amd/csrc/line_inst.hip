// line_inst.hip — instantiations of the line kernel for one precision and one group of lengths
// (QSF_PREC as in axis_pass_inst.hip; QSF_GROUP: 0 = 2^k, 1 = 3*2^k, 2 = 5*2^k).
#include "line_impl.hpp"

#if !defined(QSF_PREC) || !defined(QSF_GROUP)
#error "QSF_PREC and QSF_GROUP must be defined"
#endif

#if QSF_GROUP == 0
#define QSF_GROUP_SIZES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)
#elif QSF_GROUP == 1
#define QSF_GROUP_SIZES(X) X(12) X(24) X(48) X(96) X(192) X(384) X(768) X(1536) X(3072)
#else
#define QSF_GROUP_SIZES(X) X(10) X(20) X(40) X(80) X(160) X(320) X(640) X(1280) X(2560)
#endif

namespace qsf {
#if QSF_PREC == 1
#define QSF_INST(NN) template int launch_line_size<float, NN, false>(const LineParams&, int, hipStream_t);
#elif QSF_PREC == 2
#define QSF_INST(NN) template int launch_line_size<double, NN, true>(const LineParams&, int, hipStream_t);
#else
#define QSF_INST(NN) template int launch_line_size<double, NN, false>(const LineParams&, int, hipStream_t);
#endif
QSF_GROUP_SIZES(QSF_INST)
#undef QSF_INST
}  // namespace qsf
