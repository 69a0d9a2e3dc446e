// The layer kernels in complex128 (a translation unit of their own: they compile in parallel).
#include "iqs_layer.hpp"

template int iqsl::do_layer<double>(const iqsl::LayerArgs&, iqsl::LayerShape*);
