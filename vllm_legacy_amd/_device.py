"""The current stream's handle and the device of a launch, as cheaply as torch gives them."""
import torch

# 0.2 us; by way of a Stream object 3.  (Not a documented name of torch: without it the documented way serves.)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_handle(device) -> int:
    """The handle of the current stream of `device`, in any form torch.cuda.current_stream takes."""
    if _raw_stream is not None and isinstance(device, torch.device) and device.index is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


class _Stay:

    def __enter__(self):
        return None

    def __exit__(self, *what):
        return False


_STAY = _Stay()


def on_device(device):
    """A launch's device for the block: torch.cuda.device, which takes 2 us, only where it is another one."""
    return _STAY if device.index == torch.cuda.current_device() else torch.cuda.device(device)
