// awq_decode_plan<31> and its launch (awq_decode_flat.h).
#include "awq_decode_device.h"
#include "awq_decode_flat.h"

MPS_AWQ_FLAT_UNIT(31)
