// The merge kernel of the split-KV launches as a module of its own: see ae_combine.h.
#define AE_LAYOUT 1
#include "ae_hip.h"
#include "ae_config.h"
#include "ae_device.h"
#include "ae_functors.h"
#include "ae_combine.h"
