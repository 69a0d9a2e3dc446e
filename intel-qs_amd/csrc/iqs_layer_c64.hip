// The layer kernels in complex64 (a translation unit of their own: they compile in parallel).
#include "iqs_layer.hpp"

template int iqsl::do_layer<float>(const iqsl::LayerArgs&, iqsl::LayerShape*);
