// Transfers through the pinned ring against a runtime whose events can fail.
//   transfer_check <up|down|stage> <record|sync|none> <call that fails> <MB>
// Exit 0: a transfer that succeeds has moved every byte; one that fails says so, has
// nothing in flight that could still touch the caller's memory or the ring, never
// filled a slot whose copy was still to run, and the next transfer works.
#include "fake_hip.h"

#include "../../wurstrenderer_amd/csrc/wr_transfer.h"

#include <cstdio>
#include <string>

int main(int argc, char **argv) {
    if (argc != 5) return 64;
    const bool stage = std::string(argv[1]) == "stage", up = stage || std::string(argv[1]) == "up";
    const std::string what = argv[2];
    const size_t bytes = (size_t(std::atoi(argv[4])) << 20) + 12345;
    std::vector<char> host(bytes), device(bytes, 0);
    for (size_t i = 0; i < bytes; i++) host[i] = char(i * 2654435761u >> 13);
    if (!up) std::swap(host, device);
    wr::TransferRing ring;
    hipStream_t st = reinterpret_cast<hipStream_t>(&ring);
    auto once = [&] {
        const size_t half = bytes / 3;
        if (stage) {
            wr::TransferRing::Lease lease;  // given back, with its copies done, when the lambda returns
            return ring.stage(&lease, st, device.data(), {{host.data(), half}, {host.data() + half, bytes - half}});
        }
        return up ? ring.upload(0, st, device.data(), {{host.data(), half}, {host.data() + half, bytes - half}})
                  : ring.download(0, st, {{host.data(), device.data(), half}, {host.data() + half, device.data() + half, bytes - half}});
    };
    (what == "record" ? fake::record_fails_at : fake::sync_fails_at) = what == "none" ? -1 : std::atoi(argv[3]);
    const hipError_t e = once();
    // (the wait of a lease has nobody to tell, and falls back on the stream's)
    const bool failed = what != "none" && !(stage && what == "sync") && (what == "record" ? fake::records : fake::syncs) > std::atoi(argv[3]);
    if (failed != (e != hipSuccess)) return std::puts("the error is not reported"), 1;
    if (fake::pending()) return std::puts("work is still in flight"), 2;
    // bytes that arrived are the right ones (a slot filled too early sends another chunk's)
    const std::vector<char> &from = up ? host : device, &to = up ? device : host;
    for (size_t i = 0; i < bytes; i++)
        if (to[i] != from[i] && (!failed || to[i] != 0)) return std::printf("wrong byte %zu\n", i), 3;
    fake::record_fails_at = fake::sync_fails_at = -1;
    if (once() != hipSuccess || fake::pending() || device != host) return std::puts("the next transfer fails"), 4;
    return 0;
}
