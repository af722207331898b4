// csrc/stream_slots.hpp on the CPU, for tests/test_stream_slots.py.
#include "../../dnatok_amd/csrc/stream_slots.hpp"

extern "C" void *slots_create() { return new dnatok::StreamSlots(); }

extern "C" void slots_destroy(void *h) { delete (dnatok::StreamSlots *)h; }

extern "C" int slots_of(void *h, void *stream, unsigned long long capture) { return ((dnatok::StreamSlots *)h)->of(stream, capture); }

extern "C" int slots_streams() { return dnatok::StreamSlots::kStreams; }

extern "C" int slots_captures() { return dnatok::StreamSlots::kCaptures; }
