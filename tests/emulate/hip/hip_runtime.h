// Stands in for the HIP runtime's header where kernels are compiled for the CPU.
#include "../wave_emu.h"
