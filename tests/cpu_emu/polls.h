// The limit of a wait, chosen by a test for each launch of the one-launch sweeps.
#pragma once
#include <stdint.h>
extern "C" uint32_t flemu_polls();
