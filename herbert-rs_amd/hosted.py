"""Small arrays from the host to the GPU without waiting for it."""
import torch


def send(values, device):
    """A tensor on `device` with the numbers of a NumPy array. To a GPU they go through pinned memory of their own, in the
    order of the current stream: the host neither waits for what the stream holds nor needs the array afterwards. (A
    copy from ordinary memory waits for all of it: between two steps that left the GPU idle while the host prepared
    the second.) The pinned memory goes back to torch's pool of it, which hands it out again once the copy has run."""
    if torch.device(device).type != "cuda":
        return torch.from_numpy(values.copy()).to(device)
    staged = torch.empty(values.shape, dtype=torch.from_numpy(values[:0]).dtype, pin_memory=True)
    staged.numpy()[...] = values
    return staged.to(device, non_blocking=True)
